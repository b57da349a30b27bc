"""Calls on a context whose scratch memory holds NaN from an earlier call: padding that a kernel
leaves unwritten must not reach a result.  Ragged lengths, where there is padding."""
import numpy as np
import pytest

from localfold_amd import synthetic as S
from oracle import ops
from tests import helpers as H

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def stale():
    """A context of its own, and a call that fills its scratch memory with NaN: triangle attention
    over a NaN pair tensor of 384 residues writes every q, k, v, gate, output and bias value."""
    import torch
    from localfold_amd import capi, device as D
    ctx = D.Context(0)
    w = S.config3_attention_weights(128, 4, 3)
    dw = D.DeviceWeights(ctx.device)
    ws = D.attention_weights_af2(dw, w["attention"], w["pairBias"])
    z = torch.full((384, 384, 128), float("nan"), device=ctx.device)
    m = torch.ones(384, 384, device=ctx.device)

    def poison():
        D.attention(ctx, z, m, ws, 4, False, capi.LF_BIAS_NORMALIZED_INPUT)
        torch.cuda.synchronize()
        return ctx
    yield poison
    ctx.close()


@pytest.mark.parametrize("n", [1, 59, 130, 301])
@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("source", ["separate", "input", "logits"])
@pytest.mark.parametrize("heads", [4, 8])
def test_attention_pair_bias(stale, n, swap, source, heads):
    """Heads of 32 and 16; the last key masked, so the last 16 keys hold unmasked and masked ones
    and some past the end."""
    import torch
    from localfold_amd import capi, device as D
    rng = np.random.default_rng(n + heads)
    w = S.config3_attention_weights(128, heads, n)
    att = w["attention"]
    pn = {"layerNormScale": att["queryNormScale"], "layerNormOffset": att["queryNormOffset"],
          "projectionWeight": w["pairBias"]["projectionWeight"]}
    b = n if source == "input" else 3
    act = rng.standard_normal((b, n, 128)).astype(np.float32)
    pair = act if source == "input" else rng.standard_normal((n, n, 128)).astype(np.float32)
    logits = rng.standard_normal((heads, n, n)).astype(np.float32)
    mask = np.ones((b, n), np.float32)
    mask[:, n - 1] = 0
    mask[::2, ::5] = 0
    mask[:, 0] = 1

    ctx = stale()
    dw = D.DeviceWeights(ctx.device)
    ws = D.attention_weights_af2(dw, att, pn)
    dev = lambda x: torch.as_tensor(np.ascontiguousarray(x)).to(ctx.device)
    mode = {"separate": capi.LF_BIAS_SEPARATE, "input": capi.LF_BIAS_NORMALIZED_INPUT,
            "logits": capi.LF_BIAS_LOGITS}[source]
    out = D.attention(ctx, dev(act), dev(mask), ws, heads, False, mode, dev(pair) if source == "separate" else None,
                      swap_bias=swap, bias_logits=dev(logits) if source == "logits" else None)
    out = out.cpu().numpy()
    assert np.isfinite(out).all()

    if source == "logits":
        pb = {"source": "logits", "logits": logits.transpose(0, 2, 1) if swap else logits}
    else:   # the input's bias is that of a separate tensor with the input's norm
        pb = dict(pn, source="separate", activations=pair.transpose(1, 0, 2) if swap else pair)
    rows = [0, b // 2, b - 1]
    ref = ops.attention_af2(act, mask, att, heads, False, pb, batch_rows=rows)
    H.assert_close(out[rows], ref, label=f"{source} {n} swap={swap} heads={heads}")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("direction", ["outgoing", "incoming"])
def test_triangle_multiplication(stale, dtype, direction):
    import torch
    from localfold_amd import device as D
    n = 59
    inp = S.deterministic_triangle_input(n, 128, 128, 11)
    ctx = stale()
    dw = D.DeviceWeights(ctx.device)
    ws = D.tri_mult_weights(dw, inp["weights"])
    z = torch.as_tensor(inp["z"]).to(ctx.device).to(getattr(torch, dtype))
    out = D.tri_mult(ctx, z, torch.as_tensor(inp["mask"]).to(ctx.device), ws, direction)
    ref = ops.tri_mult_af2(z.float().cpu().numpy(), inp["mask"], inp["weights"], direction)
    H.assert_close(out.float().cpu().numpy(), ref, max_abs=H.MAX_ABS + float(np.abs(ref).max()) * 2.0 ** -8,
                   label=f"{dtype} {direction}")


@pytest.mark.parametrize("s,n,co", [(5, 21, 32), (13, 21, 16)])
def test_outer_product_mean(stale, s, n, co):
    import torch
    from localfold_amd import device as D
    w = S.synthetic_block_weights(c_m=64, c_z=128, c_outer=co, heads_msa=2, heads_pair=4, tri_hidden=32,
                                  msa_hidden=64, pair_hidden=64, seed=s)["outerProductMean"]
    act = S.synthetic_activations(s, n, 64, 128, seed=n)
    ctx = stale()
    dw = D.DeviceWeights(ctx.device)
    ws = D.opm_weights(dw, w)
    dev = lambda x: torch.as_tensor(np.ascontiguousarray(x)).to(ctx.device)
    out = D.outer_product_mean(ctx, dev(act["msa"]), dev(act["msaMask"]), ws, co, 128)
    H.assert_close(out.cpu().numpy(), ops.outer_product_mean_af2(act["msa"], act["msaMask"], w), label=f"opm {s}x{n}")
