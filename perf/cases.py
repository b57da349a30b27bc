"""The calls whose time this framework is judged by: the single layers of the AF2 Evoformer and
AF3 Pairformer over the protein lengths, MSA depths, storage types and weight codecs they are
used with, and two whole blocks.

A protein's length and an MSA's depth are what they happen to be, so most lengths here are not
multiples of a tile; the round ones (384, 512) are the crops and buckets that models are
trained and served at.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs, weights and masks on the GPU
    run(state)          one pass through localfold_amd.device
    work(case)          bytes and operations that the pass cannot do without
    tolerance(case)     how far two correct implementations at this precision may be apart
    exact(case, seed)   the same outputs in float64 with plain torch
"""
import math

import numpy as np
import torch

from localfold_amd import capi, synthetic
from localfold_amd import device as D

C_Z, C_M, C_E, C_S = 128, 256, 64, 384          # pair, MSA, extra-MSA and single channels
HEADS_PAIR, HEADS_MSA, HEADS_SINGLE, DIM_SINGLE = 4, 8, 16, 24
C_OUTER, FACTOR = 32, 4                         # outer product width, transition widening
DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
ACT_BYTES = {"f32": 4, "f16": 2, "bf16": 2}
WEIGHT_BITS = {"float32": 32.0, "float16": 16.0, "int8": 8.25, "int5": 6.0}
EPS, OPM_EPS = 1e-5, 1e-3


def listed():
    return [
        # a short protein (59 residues, the length of the reference's fixtures), full precision
        {"name": "tri_mult_59", "kind": "tri_mult", "n": 59, "dtype": "f32", "weights": "float32", "dialect": "af2",
         "tail": 0},
        # the headline workload: an AF2 training crop, int5 weights per output channel, padded tail
        {"name": "tri_mult_384", "kind": "tri_mult", "n": 384, "dtype": "bf16", "weights": "int5", "dialect": "af2",
         "tail": 16},
        # a long protein (825 residues, the length the reference quotes its kernels at)
        {"name": "tri_mult_825", "kind": "tri_mult", "n": 825, "dtype": "f32", "weights": "int8", "dialect": "af2",
         "tail": 0},
        # triangle attention at a serving bucket with 5% padding, fp16
        {"name": "tri_att_512", "kind": "tri_att", "n": 512, "dtype": "f16", "weights": "float16", "tail": 26},
        # triangle attention at an unpadded ordinary length, the full-precision residual stream
        {"name": "tri_att_301", "kind": "tri_att", "n": 301, "dtype": "f32", "weights": "int8", "tail": 0},
        # MSA row attention with pair bias: the AF2 crop at full MSA depth
        {"name": "msa_row_384", "kind": "msa_row", "n": 384, "s": 512, "dtype": "f32", "weights": "int8"},
        # MSA column attention at an ordinary length with 508 clusters (AF2's max_msa_clusters less templates)
        {"name": "msa_col_259", "kind": "msa_col", "n": 259, "s": 508, "dtype": "bf16", "weights": "int8"},
        # outer product mean of the same kind of MSA
        {"name": "opm_301", "kind": "opm", "n": 301, "s": 508, "c_m": C_M, "dtype": "f32", "weights": "int8"},
        # the MSA transition, the largest dense layer of the AF2 block
        {"name": "transition_384", "kind": "transition", "n": 384, "s": 512, "c": C_M, "act": "relu",
         "dtype": "f32", "weights": "int8"},
        # the extra-MSA stack's global column attention at AF2's 1024 extra sequences
        {"name": "global_col_384", "kind": "global_col", "n": 384, "s": 1024, "dtype": "bf16", "weights": "int8"},
        # a whole Evoformer block: a mid-size protein with a shallow MSA
        {"name": "evoformer_203", "kind": "evoformer", "n": 203, "s": 126, "dtype": "f32", "weights": "int8"},
        # a whole Pairformer block: int5 weights, a bucket with padded tokens
        {"name": "pairformer_512", "kind": "pairformer", "n": 512, "dtype": "bf16", "weights": "int5", "tail": 19},
    ]


def draw(rng):
    def log_int(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["tri_mult", "tri_att", "msa_row", "msa_col", "opm", "transition", "global_col", "evoformer",
                       "pairformer"])
    top = {"tri_mult": 825, "tri_att": 512, "msa_row": 384, "msa_col": 384, "opm": 384, "transition": 384,
           "global_col": 384, "evoformer": 203, "pairformer": 400}[kind]
    c = {"kind": kind, "n": log_int(40, top), "dtype": rng.choice(["f32", "f32", "bf16", "f16"]),
         "weights": rng.choice(["float32", "float16", "int8", "int8", "int5"])}
    if kind in ("tri_mult", "tri_att", "pairformer"):
        c["tail"] = rng.choice([0, 0, rng.randint(1, max(1, c["n"] // 16))])
    if kind == "tri_mult":
        c["dialect"] = rng.choice(["af2", "af3"])
    if kind in ("msa_row", "msa_col"):
        c["s"] = log_int(16, 512)
    if kind == "evoformer":   # a single sequence (no MSA) up to a shallow MSA
        c["s"] = rng.choice([1, log_int(8, 126), log_int(8, 126)])
    if kind == "opm":
        c["c_m"] = rng.choice([C_M, C_E])
        c["s"] = log_int(16, 512 if c["c_m"] == C_M else 1024)
    if kind == "transition":
        c["act"] = rng.choice(["relu", "swiglu"])
        c["c"] = rng.choice([C_M, C_Z]) if c["act"] == "relu" else C_Z
        c["s"] = log_int(16, 512) if c["c"] == C_M else c["n"]
    if kind == "global_col":
        c["s"] = log_int(64, 1024)
    return c


# ---- weights: float32 masters, the stored records and (for exact) their values -----------------

class Masters:
    """Random-init layers, N(0, 1/fan_in), LayerNorms near identity, named as the layers' inputs."""

    def __init__(self, seed):
        self.rng = np.random.default_rng(seed)

    def lin(self, i, o, transposed=False):
        w = (self.rng.standard_normal((i, o), dtype=np.float32) / np.float32(math.sqrt(i)))
        return np.ascontiguousarray(w.T) if transposed else w

    def vec(self, n, spread, centre=0.0):
        return self.rng.uniform(centre - spread, centre + spread, n).astype(np.float32)

    def tri_af2(self, c=C_Z):
        w = {"layerNormInWeight": self.vec(c, 0.2, 1), "layerNormInBias": self.vec(c, 0.1),
             "layerNormOutWeight": self.vec(c, 0.2, 1), "layerNormOutBias": self.vec(c, 0.1)}
        for name, centre in (("AP", 0), ("AG", 1), ("BP", 0), ("BG", 1), ("Z", 0), ("G", 1)):
            w[f"linear{name}Weight"] = self.lin(c, c, True)
            w[f"linear{name}Bias"] = self.vec(c, 0.03, centre)
        return w

    def tri_af3(self, c=C_Z):
        return {"leftNormInputScale": self.vec(c, 0.2, 1), "leftNormInputOffset": self.vec(c, 0.1),
                "projection": self.lin(c, 2 * c), "gate": self.lin(c, 2 * c),
                "centerNormScale": self.vec(c, 0.2, 1), "centerNormOffset": self.vec(c, 0.1),
                "outputProjection": self.lin(c, c), "gatingLinear": self.lin(c, c)}

    def att_af2(self, c, heads, bias=None):
        a = {"queryNormScale": self.vec(c, 0.2, 1), "queryNormOffset": self.vec(c, 0.1)}
        for name in ("query", "key", "value", "gating", "output"):
            a[name + "Weight"] = self.lin(c, c)
        a["gatingBias"], a["outputBias"] = self.vec(c, 0.1, 1), self.vec(c, 0.05)
        w = {"heads": heads, "attention": a}
        if bias == "pair":
            w["pairBias"] = {"layerNormScale": self.vec(C_Z, 0.2, 1), "layerNormOffset": self.vec(C_Z, 0.1),
                             "projectionWeight": self.lin(C_Z, heads)}
        elif bias == "input":
            w["pairBias"] = {"projectionWeight": self.lin(c, heads)}
        return w

    def grid(self, c=C_Z, heads=HEADS_PAIR):
        return {"heads": heads, "dimension": c // heads, "actNormScale": self.vec(c, 0.2, 1),
                "actNormOffset": self.vec(c, 0.1), "pairBiasProjection": self.lin(c, heads),
                "qProjection": self.lin(c, c, True), "kProjection": self.lin(c, c, True),
                "vProjection": self.lin(c, c), "gatingQuery": self.lin(c, c, True),
                "outputProjection": self.lin(c, c)}

    def global_col(self, c=C_E, heads=HEADS_MSA):
        d = c // heads
        return {"heads": heads, "attention": {
            "queryNormScale": self.vec(c, 0.2, 1), "queryNormOffset": self.vec(c, 0.1),
            "queryWeight": self.lin(c, c), "keyWeight": self.lin(c, d), "valueWeight": self.lin(c, d),
            "gatingWeight": self.lin(c, c), "gatingBias": self.vec(c, 0.1, 1),
            "outputWeight": self.lin(c, c), "outputBias": self.vec(c, 0.05)}}

    def relu(self, c):
        h = FACTOR * c
        return {"layerNormScale": self.vec(c, 0.2, 1), "layerNormOffset": self.vec(c, 0.1),
                "firstWeight": self.lin(c, h), "firstBias": self.vec(h, 0.1),
                "secondWeight": self.lin(h, c), "secondBias": self.vec(c, 0.05)}

    def swiglu(self, c):
        return {"inputLayerNormScale": self.vec(c, 0.2, 1), "inputLayerNormOffset": self.vec(c, 0.1),
                "transition1": self.lin(c, 2 * FACTOR * c), "transition2": self.lin(FACTOR * c, c)}

    def opm(self, c):
        return {"layerNormScale": self.vec(c, 0.2, 1), "layerNormOffset": self.vec(c, 0.1),
                "leftWeight": self.lin(c, C_OUTER), "leftBias": self.vec(C_OUTER, 0.1),
                "rightWeight": self.lin(c, C_OUTER), "rightBias": self.vec(C_OUTER, 0.1),
                "outputWeight": self.lin(C_OUTER * C_OUTER, C_Z), "outputBias": self.vec(C_Z, 0.05)}

    def evoformer(self):
        return {"msaRowAttention": self.att_af2(C_M, HEADS_MSA, "pair"),
                "msaColumnAttention": self.att_af2(C_M, HEADS_MSA),
                "msaTransition": self.relu(C_M), "outerProductMean": self.opm(C_M),
                "triangleMultiplicationOutgoing": self.tri_af2(), "triangleMultiplicationIncoming": self.tri_af2(),
                "triangleAttentionStarting": self.att_af2(C_Z, HEADS_PAIR, "input"),
                "triangleAttentionEnding": self.att_af2(C_Z, HEADS_PAIR, "input"),
                "pairTransition": self.relu(C_Z)}

    def pairformer(self):
        w = {"triangleMultiplicationOutgoing": self.tri_af3(), "triangleMultiplicationIncoming": self.tri_af3(),
             "pairAttention1": self.grid(), "pairAttention2": self.grid(), "pairTransition": self.swiglu(C_Z),
             "singlePairLogitsNormScale": self.vec(C_Z, 0.2, 1), "singlePairLogitsNormOffset": self.vec(C_Z, 0.1),
             "singlePairLogitsProjection": self.lin(C_Z, HEADS_SINGLE), "singleTransition": self.swiglu(C_S)}
        hw = HEADS_SINGLE * DIM_SINGLE
        w["singleAttention"] = {"heads": HEADS_SINGLE, "dimension": DIM_SINGLE,
                                "layerNormScale": self.vec(C_S, 0.2, 1), "layerNormOffset": self.vec(C_S, 0.1),
                                "qProjection": self.lin(C_S, hw), "qBias": self.vec(hw, 0.1),
                                "kProjection": self.lin(C_S, hw), "vProjection": self.lin(C_S, hw),
                                "gatingQuery": self.lin(C_S, hw), "outputProjection": self.lin(hw, C_S)}
        return w


def layers(case, seed):
    """The case's layers as stored records: a tuple of weight dictionaries."""
    m, kind = Masters(1000 + seed), case["kind"]
    if kind == "tri_mult":
        ws = (m.tri_af2(), m.tri_af2()) if case["dialect"] == "af2" else (m.tri_af3(), m.tri_af3())
        if case["weights"] == "int5" and case["dialect"] == "af2":   # tables per output channel
            return tuple(synthetic.quantise_records(w, synthetic.TRI_MATS, "int5", True, 0) for w in ws)
    else:
        ws = {"tri_att": lambda: (m.att_af2(C_Z, HEADS_PAIR, "input"), m.att_af2(C_Z, HEADS_PAIR, "input")),
              "msa_row": lambda: (m.att_af2(C_M, HEADS_MSA, "pair"),),
              "msa_col": lambda: (m.att_af2(C_M, HEADS_MSA),),
              "opm": lambda: (m.opm(case["c_m"]),),
              "transition": lambda: (m.relu(case["c"]) if case["act"] == "relu" else m.swiglu(case["c"]),),
              "global_col": lambda: (m.global_col(),),
              "evoformer": lambda: (m.evoformer(),),
              "pairformer": lambda: (m.pairformer(),)}[kind]()
    fmt = case["weights"]
    if fmt == "float32":
        return ws
    return tuple(synthetic.quantise_tree(w, fmt, {"int8": 64, "int5": 32}.get(fmt)) for w in ws)


def values(w):
    """The float64 values on the GPU that a stored weight dictionary stands for."""
    if not isinstance(w, dict):
        return torch.as_tensor(np.asarray(w, np.float64)).cuda() if isinstance(w, np.ndarray) else w
    if "dtype" not in w or "shape" not in w:
        return {k: values(v) for k, v in w.items()}
    shape = tuple(w["shape"])
    if w["dtype"] in ("float32", "float16"):
        return values(np.asarray(w["data"], np.float64).reshape(shape))
    count = int(np.prod(shape))
    if w["dtype"] == "int8":
        codes = np.asarray(w["data"]).view(np.int8).reshape(-1)[:count].astype(np.float64)
    else:
        bits = np.unpackbits(np.asarray(w["data"]).view(np.uint8), bitorder="little")[:5 * count]
        codes = bits.reshape(count, 5).astype(np.float64) @ (1 << np.arange(5))
    at = np.arange(count)
    if "channel_axis" in w:
        at = np.unravel_index(at, shape)[w["channel_axis"]]
    else:
        at = at // w["block"]
    got = codes * np.asarray(w["scales"], np.float64)[at]
    if w.get("zeros") is not None:
        got = got + np.asarray(w["zeros"], np.float64)[at]
    return values(got.reshape(shape))


# ---- inputs --------------------------------------------------------------------------------

def tensors(case, seed):
    """Activations (N(0, 1) in the case's storage type) and float32 masks."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt, kind, n, s = DTYPES[case["dtype"]], case["kind"], case["n"], case.get("s")

    def act(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).to(dt)

    t = {}
    if kind in ("tri_mult", "tri_att", "pairformer", "evoformer", "msa_row", "opm"):
        t["pair"] = act(n, n, C_Z)
    if kind in ("tri_mult", "tri_att", "pairformer", "evoformer"):
        keep = (torch.arange(n, device="cuda") < n - case.get("tail", 0)).float()   # padded residues last
        t["pair_mask"] = keep[:, None] * keep[None, :]
        t["seq_mask"] = keep
    if kind == "pairformer":
        t["single"] = act(n, C_S)
    if kind in ("msa_row", "msa_col", "evoformer"):
        t["msa"], t["msa_mask"] = act(s, n, C_M), torch.ones(s, n, device="cuda")
    if kind == "opm":
        t["msa"] = act(s, n, case["c_m"])
    if kind == "global_col":
        t["msa"] = act(s, n, C_E)
    if kind in ("opm", "global_col"):   # a fifth of the MSA positions are gaps without features
        t["msa_mask"] = (torch.rand(s, n, device="cuda", generator=gen) > 0.2).float()
    if kind == "transition":
        t["x"] = act(s, n, case["c"])
    return t


_context = None


def prepare(case, seed):
    global _context
    if _context is None:
        _context = D.Context(0)
    ws, kind = layers(case, seed), case["kind"]
    dw = D.DeviceWeights(_context.device)
    dialect = capi.LF_AF3 if case.get("dialect") == "af3" else capi.LF_AF2
    swiglu = capi.LF_TRANSITION_SWIGLU if case.get("act") == "swiglu" else capi.LF_TRANSITION_RELU
    build = {"tri_mult": lambda w: D.tri_mult_weights(dw, w, dialect),
             "tri_att": lambda w: D.attention_weights_af2(dw, w["attention"], w["pairBias"]),
             "msa_row": lambda w: D.attention_weights_af2(dw, w["attention"], w["pairBias"]),
             "msa_col": lambda w: D.attention_weights_af2(dw, w["attention"]),
             "opm": lambda w: D.opm_weights(dw, w),
             "transition": lambda w: D.transition_weights(dw, w, swiglu),
             "global_col": lambda w: D.global_attention_weights(dw, w["attention"]),
             "evoformer": lambda w: D.evoformer_weights(dw, w),
             "pairformer": lambda w: D.pairformer_weights(dw, w)}[kind]
    return dict(tensors(case, seed), case=case, ctx=_context, names=ws[0], dialect=dialect, swiglu=swiglu,
                weights=[build(w) for w in ws])


def run(state):
    ctx, kind, ws = state["ctx"], state["case"]["kind"], state["weights"]
    if kind == "tri_mult":
        z1 = D.tri_mult(ctx, state["pair"], state["pair_mask"], ws[0], "outgoing", state["dialect"], accumulate=True)
        z2 = D.tri_mult(ctx, z1, state["pair_mask"], ws[1], "incoming", state["dialect"], accumulate=True)
        return z1, z2
    if kind == "tri_att":
        z1 = D.attention(ctx, state["pair"], state["pair_mask"], ws[0], HEADS_PAIR, False,
                         capi.LF_BIAS_NORMALIZED_INPUT, accumulate=True)
        z2 = D.attention(ctx, z1, state["pair_mask"], ws[1], HEADS_PAIR, True, capi.LF_BIAS_NORMALIZED_INPUT,
                         accumulate=True)
        return z1, z2
    if kind == "msa_row":
        return D.attention(ctx, state["msa"], state["msa_mask"], ws[0], HEADS_MSA, False, capi.LF_BIAS_SEPARATE,
                           pair=state["pair"], accumulate=True)
    if kind == "msa_col":
        return D.attention(ctx, state["msa"], state["msa_mask"], ws[0], HEADS_MSA, True, accumulate=True)
    if kind == "opm":
        return D.outer_product_mean(ctx, state["msa"], state["msa_mask"], ws[0], C_OUTER, C_Z, pair=state["pair"],
                                    accumulate=True)
    if kind == "transition":
        return D.transition(ctx, state["x"], ws[0], FACTOR * state["case"]["c"], state["swiglu"], accumulate=True,
                            fast_variance=state["swiglu"] == capi.LF_TRANSITION_SWIGLU)
    if kind == "global_col":
        return D.global_column_attention(ctx, state["msa"], state["msa_mask"], ws[0], HEADS_MSA, accumulate=True)
    # the blocks work in place; the caller keeps its embeddings, as between recycles
    pair = state["pair"].clone()
    if kind == "evoformer":
        msa = state["msa"].clone()
        D.evoformer_block(ctx, msa, pair, state["msa_mask"], state["pair_mask"], ws[0], state["names"])
        return msa, pair
    single = state["single"].clone()
    D.pairformer_block(ctx, pair, single, state["pair_mask"], state["seq_mask"], ws[0])
    return pair, single


# ---- what a pass cannot do without ------------------------------------------------------------

def work(case):
    """Each input read once, each output written once; the multiply-adds of the layers' products."""
    n, s, a = case["n"], case.get("s", 0), ACT_BYTES[case["dtype"]]
    wb = WEIGHT_BITS[case["weights"]] / 8
    p = n * n

    def tri():
        return 2 * p * C_Z * C_Z * 6 + 2 * n ** 3 * C_Z, 6 * C_Z * C_Z

    def att(rows, queries, c, hw, heads=0, bias_rows=0, cb=0):
        return (2 * rows * c * hw * 5 + 4 * rows * queries * hw + 2 * bias_rows * cb * heads, 5 * c * hw + cb * heads)

    def mlp(rows, c, swiglu):
        k = 3 if swiglu else 2
        return 2 * rows * c * FACTOR * c * k, k * c * FACTOR * c

    def opm(c):
        return (4 * s * n * c * C_OUTER + 2 * s * p * C_OUTER ** 2 + 2 * p * C_OUTER ** 2 * C_Z,
                2 * c * C_OUTER + C_OUTER ** 2 * C_Z)

    kind = case["kind"]
    if kind == "tri_mult":
        parts, rd, wr = [tri(), tri()], p * C_Z * a + p * 4, 2 * p * C_Z * a
    elif kind == "tri_att":
        parts = [att(p, n, C_Z, C_Z, HEADS_PAIR, p, C_Z)] * 2
        rd, wr = p * C_Z * a + p * 4, 2 * p * C_Z * a
    elif kind == "msa_row":
        parts = [att(s * n, n, C_M, C_M, HEADS_MSA, p, C_Z)]
        rd, wr = s * n * (C_M * a + 4) + p * C_Z * a, s * n * C_M * a
    elif kind == "msa_col":
        parts, rd, wr = [att(s * n, s, C_M, C_M)], s * n * (C_M * a + 4), s * n * C_M * a
    elif kind == "opm":
        parts, rd, wr = [opm(case["c_m"])], s * n * (case["c_m"] * a + 4) + p * C_Z * a, p * C_Z * a
    elif kind == "transition":
        parts = [mlp(s * n, case["c"], case["act"] == "swiglu")]
        rd, wr = s * n * case["c"] * a, s * n * case["c"] * a
    elif kind == "global_col":
        d = C_E // HEADS_MSA
        parts = [(2 * s * n * C_E * (2 * C_E + 2 * d) + 2 * n * C_E * C_E + 4 * s * n * C_E, C_E * (3 * C_E + 2 * d))]
        rd, wr = s * n * (C_E * a + 4), s * n * C_E * a
    elif kind == "evoformer":
        parts = [att(s * n, n, C_M, C_M, HEADS_MSA, p, C_Z), att(s * n, s, C_M, C_M), mlp(s * n, C_M, False), opm(C_M),
                 tri(), tri(), att(p, n, C_Z, C_Z, HEADS_PAIR, p, C_Z), att(p, n, C_Z, C_Z, HEADS_PAIR, p, C_Z),
                 mlp(p, C_Z, False)]
        rd, wr = s * n * (C_M * a + 4) + p * (C_Z * a + 4), s * n * C_M * a + p * C_Z * a
    else:
        parts = [tri(), tri(), att(p, n, C_Z, C_Z, HEADS_PAIR, p, C_Z), att(p, n, C_Z, C_Z, HEADS_PAIR, p, C_Z),
                 mlp(p, C_Z, True), att(n, n, C_S, HEADS_SINGLE * DIM_SINGLE, HEADS_SINGLE, p, C_Z),
                 mlp(n, C_S, True)]
        rd, wr = p * (C_Z * a + 4) + n * (C_S * a + 4), p * C_Z * a + n * C_S * a
    return {"bytes": float(rd + wr + sum(w for _, w in parts) * wb), "flops": float(sum(f for f, _ in parts))}


# Products take f16 operands and sum in f32 whatever the storage.  Four times the relative error
# against float64 that f32 storage shows per kind; f16 and bf16 storage add their roundings, one
# per layer that is stored (2^-12 and 2^-9 relative at most, a third of that in the mean square).
TOLERANCE = {"tri_mult": 2.2e-3, "tri_att": 6e-4, "msa_row": 4e-4, "msa_col": 1e-3, "opm": 2e-4, "transition": 1e-3,
             "global_col": 1e-3, "evoformer": 3.3e-3, "pairformer": 4e-3}
STORAGE = {"f32": 0.0, "f16": 1e-3, "bf16": 7e-3}


def tolerance(case):
    stored = 2 if case["kind"] in ("evoformer", "pairformer") else 1
    return {"rel": TOLERANCE[case["kind"]] + stored * STORAGE[case["dtype"]]}


# ---- the same in float64 ------------------------------------------------------------------------

def ln(x, scale, offset):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * scale + offset


def tri_exact(z, mask, w, incoming):
    if "projection" in w:
        x = ln(z, w["leftNormInputScale"], w["leftNormInputOffset"])
        ab = (x @ w["projection"]) * torch.sigmoid(x @ w["gate"]) * mask[..., None]
        a, b = ab[..., 0::2], ab[..., 1::2]
    else:
        x = ln(z, w["layerNormInWeight"], w["layerNormInBias"])
        a, b = ((x @ w[f"linear{t}PWeight"].T + w[f"linear{t}PBias"]) * mask[..., None]
                * torch.sigmoid(x @ w[f"linear{t}GWeight"].T + w[f"linear{t}GBias"]) for t in "AB")
    # outgoing x_ij = sum_k a_ik b_jk, incoming x_ij = sum_k b_ki a_kj
    a, b = a.permute(2, 0, 1).contiguous(), b.permute(2, 0, 1).contiguous()
    t = torch.matmul(b.transpose(1, 2).contiguous(), a) if incoming else torch.matmul(a, b.transpose(1, 2).contiguous())
    t = t.permute(1, 2, 0)
    if "projection" in w:
        return (ln(t, w["centerNormScale"], w["centerNormOffset"]) @ w["outputProjection"]) * torch.sigmoid(
            x @ w["gatingLinear"])
    t = ln(t, w["layerNormOutWeight"], w["layerNormOutBias"]) @ w["linearZWeight"].T + w["linearZBias"]
    return t * torch.sigmoid(x @ w["linearGWeight"].T + w["linearGBias"])


def softmax_rows(q, k, v, bias, mask, heads):
    """q, k, v [B, Q, H*d], bias [H, Q, Q] or None, mask [B, Q]: softmax(q k / sqrt(d) + bias) v, by rows."""
    rows, n, hw = q.shape
    d, step = hw // heads, max(1, int(2 ** 27 // (heads * n * n)))
    out = torch.empty_like(v)

    def split(t):
        return t.reshape(t.shape[0], n, heads, d).transpose(1, 2).contiguous()

    for r in range(0, rows, step):
        at = slice(r, r + step)
        x = torch.matmul(split(q[at]) / math.sqrt(d), split(k[at]).transpose(2, 3).contiguous())
        if bias is not None:
            x += bias
        x += 1e9 * (mask[at, None, None, :] - 1)
        out[at] = torch.matmul(torch.softmax(x.clamp_(-1e8, 1e8), -1), split(v[at])).transpose(1, 2).reshape(-1, n, hw)
    return out


def att_exact(act, mask, w, transpose=False, pair=None):
    a, heads = w["attention"], w["heads"]
    if transpose:
        act, mask = act.transpose(0, 1), mask.T
    x = ln(act, a["queryNormScale"], a["queryNormOffset"])
    bias = None
    if "pairBias" in w:
        b = w["pairBias"]
        src = ln(pair, b["layerNormScale"], b["layerNormOffset"]) if "layerNormScale" in b else x
        bias = (src @ b["projectionWeight"]).permute(2, 0, 1)
    o = softmax_rows(x @ a["queryWeight"], x @ a["keyWeight"], x @ a["valueWeight"], bias, mask, heads)
    o = (o * torch.sigmoid(x @ a["gatingWeight"] + a["gatingBias"])) @ a["outputWeight"] + a["outputBias"]
    return o.transpose(0, 1) if transpose else o


def grid_exact(pair, mask, w, transpose):
    x = ln(pair, w["actNormScale"], w["actNormOffset"])
    bias = (x @ w["pairBiasProjection"]).permute(2, 0, 1)
    if transpose:
        x, mask = x.transpose(0, 1), mask.T
    o = softmax_rows(x @ w["qProjection"].T, x @ w["kProjection"].T, x @ w["vProjection"], bias, mask, w["heads"])
    o = (o * torch.sigmoid(x @ w["gatingQuery"].T)) @ w["outputProjection"]
    return o.transpose(0, 1) if transpose else o


def mlp_exact(x, w):
    if "transition1" in w:
        h = ln(x, w["inputLayerNormScale"], w["inputLayerNormOffset"]) @ w["transition1"]
        gate, value = h.chunk(2, -1)
        return (torch.nn.functional.silu(gate) * value) @ w["transition2"]
    h = ln(x, w["layerNormScale"], w["layerNormOffset"]) @ w["firstWeight"] + w["firstBias"]
    return torch.relu(h) @ w["secondWeight"] + w["secondBias"]


def opm_exact(msa, mask, w):
    s, n, _ = msa.shape
    x = ln(msa, w["layerNormScale"], w["layerNormOffset"])
    left = (x @ w["leftWeight"] + w["leftBias"]) * mask[..., None]
    right = (x @ w["rightWeight"] + w["rightBias"]) * mask[..., None]
    outer = left.reshape(s, -1).T.contiguous() @ right.reshape(s, -1)          # [(i, a), (j, b)]
    outer = outer.reshape(n, C_OUTER, n, C_OUTER).transpose(1, 2).reshape(n, n, C_OUTER ** 2)
    return (outer @ w["outputWeight"] + w["outputBias"]) / (OPM_EPS + mask.T.contiguous() @ mask)[..., None]


def global_exact(msa, mask, w):
    a, heads = w["attention"], w["heads"]
    s, n, c = msa.shape
    d = c // heads
    x = ln(msa, a["queryNormScale"], a["queryNormOffset"])
    q = (x * mask[..., None]).sum(0) / (1e-10 + mask.sum(0))[:, None] @ a["queryWeight"] / math.sqrt(d)
    logits = torch.matmul((x @ a["keyWeight"]).transpose(0, 1), q.reshape(n, heads, d).transpose(1, 2).contiguous())
    logits = torch.where(mask.T[..., None] > 0, logits, torch.full_like(logits, -1e9))    # [n, s, h]
    o = torch.matmul(torch.softmax(logits, 1).transpose(1, 2).contiguous(), (x @ a["valueWeight"]).transpose(0, 1))
    gate = torch.sigmoid(x @ a["gatingWeight"] + a["gatingBias"])
    return (gate * o.reshape(1, n, heads * d)) @ a["outputWeight"] + a["outputBias"]


def single_exact(single, pair, mask, w):
    a = w["singleAttention"]
    bias = (ln(pair, w["singlePairLogitsNormScale"], w["singlePairLogitsNormOffset"])
            @ w["singlePairLogitsProjection"]).permute(2, 0, 1)
    x = ln(single, a["layerNormScale"], a["layerNormOffset"])
    o = softmax_rows((x @ a["qProjection"] + a["qBias"])[None], (x @ a["kProjection"])[None],
                     (x @ a["vProjection"])[None], bias, mask[None], a["heads"])[0]
    return (o * torch.sigmoid(x @ a["gatingQuery"])) @ a["outputProjection"]


def exact(case, seed):
    t = {k: v.double() for k, v in tensors(case, seed).items()}
    ws, kind = [values(w) for w in layers(case, seed)], case["kind"]
    if kind in ("tri_mult", "tri_att"):
        z, mask, out = t["pair"], t["pair_mask"], []
        for i in (0, 1):
            z = z + (tri_exact(z, mask, ws[i], i == 1) if kind == "tri_mult" else att_exact(z, mask, ws[i], i == 1))
            out.append(z)
        return tuple(out)
    w = ws[0]
    if kind in ("msa_row", "msa_col"):
        return t["msa"] + att_exact(t["msa"], t["msa_mask"], w, kind == "msa_col", t.get("pair"))
    if kind == "opm":
        return t["pair"] + opm_exact(t["msa"], t["msa_mask"], w)
    if kind == "transition":
        return t["x"] + mlp_exact(t["x"], w)
    if kind == "global_col":
        return t["msa"] + global_exact(t["msa"], t["msa_mask"], w)
    pair, pair_mask = t["pair"], t["pair_mask"]
    if kind == "evoformer":
        msa, msa_mask = t["msa"], t["msa_mask"]
        msa = msa + att_exact(msa, msa_mask, w["msaRowAttention"], False, pair)
        msa = msa + att_exact(msa, msa_mask, w["msaColumnAttention"], True)
        msa = msa + mlp_exact(msa, w["msaTransition"])
        pair = pair + opm_exact(msa, msa_mask, w["outerProductMean"])
        pair = pair + tri_exact(pair, pair_mask, w["triangleMultiplicationOutgoing"], False)
        pair = pair + tri_exact(pair, pair_mask, w["triangleMultiplicationIncoming"], True)
        pair = pair + att_exact(pair, pair_mask, w["triangleAttentionStarting"], False)
        pair = pair + att_exact(pair, pair_mask, w["triangleAttentionEnding"], True)
        return msa, pair + mlp_exact(pair, w["pairTransition"])
    pair = pair + tri_exact(pair, pair_mask, w["triangleMultiplicationOutgoing"], False)
    pair = pair + tri_exact(pair, pair_mask, w["triangleMultiplicationIncoming"], True)
    pair = pair + grid_exact(pair, pair_mask, w["pairAttention1"], False)
    pair = pair + grid_exact(pair, pair_mask, w["pairAttention2"], True)
    pair = pair + mlp_exact(pair, w["pairTransition"])
    single = t["single"] + single_exact(t["single"], pair, t["seq_mask"], w)
    return pair, single + mlp_exact(single, w["singleTransition"])
