// Fused transition for c in {128, 256}: out = [x +] act(LN(x) W1 + b1) W2 + b2 in one kernel;
// the hidden activation never leaves registers, so no hidden buffer (and no row chunking) is
// needed.  Semantics as the two-kernel path in lf_transition.hip: ReLU (AF2,
// webgpu/kernels/transition.js:745-766, 1080-1085) or swish(h_gate) * h_value (AF3 SwiGLU,
// cpu/af3/trunk/pairformer.js:180-201).
//
// A wave owns RT 16-row tiles, a block four waves.  A wave LayerNorms its rows into f16 MFMA
// fragments (lane: row lane%16, channels 32j + 8*(lane/16) .. +7) that stay in registers.  The
// hidden dimension streams through two LDS buffers in chunks of 32 units, packed so that a
// fragment is 1 KB in lane order.
//   GEMM1, weights as the A operand: the lane gets H[row][16t + 4g + i] (g = lane/16, i < 4) of
//          the chunk's two 16-unit tiles t, starting from b1; then ReLU or swish-gating.
//   GEMM2: those 8 values are the lane's B fragment as they stand: MFMA k index 8g + e stands
//          for hidden unit 4g + e (e < 4) or 16 + 4g + e - 4 (e >= 4) of the chunk, and the
//          packed W2^T rows hold the hidden units in that order.
//   Output: the lane holds out[row][16ct + 4g + i], started at b2; the residual is added and
//          four channels stored as one vector at the end.
// The next chunk is copied straight to the other buffer during the current chunk's products.
//
// What bounds it: the matrix pipes, and the vector instructions and waits that they do not overlap
// with.  Counters at 196608 rows of 256, f32, hidden 1024: matrix pipes busy 36% of the time (197 k of
// 543 k cycles), 2.2 vector instructions to a product.  Copies that skip the registers leave room for
// two blocks of 128 rows a CU, whose LayerNorm, store and product phases interleave; against one block
// of 8 waves, weights staged through registers and the activation in f32, 262144 rows of 256 in bf16
// went from 332 to 274 us (1.0 PFLOP/s), 512 x 384 rows of 256 in f32 from 337 to 258 us (on another
// card 326 to 247), 512 x 512 of 128 with SwiGLU in bf16 from 163 to 142 us.  Eight waves sharing a
// buffer (305), 64 rows a wave (350), three or four buffers and wider read-ahead (275 to 280) were no
// better.
#include <algorithm>
#include <cmath>

#include "lf_gemm.h"
#include "lf_ops.h"

namespace lf {

constexpr int MLP_WAVES = 4, MLP_NT = 64 * MLP_WAVES, MLP_HC = 32;

typedef float f8 __attribute__((ext_vector_type(8)));

template <int C, int NG>
struct MlpShape {
  static constexpr int KS = C / 32, CT = C / 16;
  static constexpr int F1 = KS * NG * 2, NF = F1 + CT;         // 1 KB fragments of a chunk: W1^T, all
  static constexpr int CE = 512 * NF;                          // packed halves per chunk
  static_assert(NF % MLP_WAVES == 0 && F1 % 4 == 0 && CT % 4 == 0, "fragments must divide over the waves and groups");
};

struct MlpParams {
  const void* x;
  void* out;
  int accumulate, rows, H, fast_var;
  float eps;
  const _Float16* w;   // packed chunks (mlp_pack_kernel)
  const float *ln_s, *ln_o, *b1g, *b1v, *b2;
};

// GEMM2's k order within a chunk: position q = 8g + e holds hidden unit 4g + e (e < 4) or
// 16 + 4g + e - 4 (e >= 4); q_of is the inverse, the position of hidden unit hl (its 4-aligned
// groups stay together: q_of(4a + i) = q_of(4a) + i).
__host__ __device__ constexpr int mlp_q_of(int hl) {
  return hl < 16 ? 8 * (hl >> 2) + (hl & 3) : 8 * ((hl - 16) >> 2) + 4 + (hl & 3);
}

// Packed weights, chunk s of 32 hidden units: the A fragments in the order and lane layout the
// kernel reads them, 512 halves each (lane l's 8 halves at 8l), so that a wave's read is 1 KB in
// lane order (no padding, no bank conflicts) and a chunk is copied to LDS as it stands.  First
// W1^T: k-step j of tile ht of group grp (gate, value) is fragment (j*NG + grp)*2 + ht, its lane
// (r16, g4) holding hidden unit 32s + 16ht + r16, inputs 32j + 8g4 + e; then W2^T: tile ct, its
// lane holding output 16ct + r16, positions 8g4 + e of GEMM2's k order.
// Decoding from f32/f16/bf16/int8/int5 happens here, on the device, one thread per run of 8 stored
// weights (wrun_fetch / wrun_decode): W1 runs are 8 inputs of one hidden unit (a 16-byte store) or
// 8 hidden units of one input (8 lanes); W2 runs 8 hidden units of one output (two 4-wide pieces
// of the k order) or 8 outputs of one hidden unit (8 lanes).
__global__ __launch_bounds__(256) void mlp_pack_kernel(WView w1g, WView w1v, WView w2, int C, int H, int NG,
                                                       _Float16* dst) {
  const long long ce = (long long)(NG * MLP_HC + MLP_HC) * C, w1e = (long long)NG * MLP_HC * C;
  const bool k1 = w1g.run != WRUN_N, k2 = w2.run != WRUN_N;
  const long long r1 = (long long)NG * H * C / 8, total = r1 + (long long)H * C / 8;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long long)gridDim.x * 256) {
    if (i < r1) {   // W1: (hidden unit u of group grp, input c)
      const int grp = (int)(i / ((long long)H * C / 8)), j = (int)(i - (long long)grp * H * C / 8);
      const int u = k1 ? j / (C / 8) : 8 * (j / C), c = k1 ? 8 * (j % (C / 8)) : j % C;
      const WView& w = grp ? w1v : w1g;
      const h8 h = wrun_decode(w, wrun_fetch(w, c, u, 1.f), c, u, 1.f);
      const int ht = (u % MLP_HC) >> 4, lane = ((c % 32) >> 3) * 16 + (u & 15);
      _Float16* base = dst + (long long)(u / MLP_HC) * ce + (((c / 32) * NG + grp) * 2 + ht) * 512 + lane * 8 + (c & 7);
      if (k1) {
        *reinterpret_cast<h8*>(base) = h;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) base[8 * e] = h[e];
      }
    } else {        // W2: (hidden unit u, output c)
      const int j = (int)(i - r1);
      const int c = k2 ? j / (H / 8) : 8 * (j % (C / 8)), u = k2 ? 8 * (j % (H / 8)) : j / (C / 8);
      const h8 h = wrun_decode(w2, wrun_fetch(w2, u, c, 1.f), u, c, 1.f);
      const int q = mlp_q_of(u % MLP_HC);
      _Float16* base = dst + (long long)(u / MLP_HC) * ce + w1e + (c >> 4) * 512 + ((q >> 3) * 16 + (c & 15)) * 8 + (q & 7);
      if (k2) {   // hidden units u..u+3 and u+4..u+7 sit 8 apart in the k order: the next 16 lanes
        *reinterpret_cast<h4*>(base) = __builtin_shufflevector(h, h, 0, 1, 2, 3);
        *reinterpret_cast<h4*>(base + 128) = __builtin_shufflevector(h, h, 4, 5, 6, 7);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) base[8 * e] = h[e];
      }
    }
  }
}

template <int ACT, int C, int NG, int RT>
__global__ __launch_bounds__(MLP_NT, 2) void mlp_kernel(MlpParams p) {
  using S = MlpShape<C, NG>;
  constexpr int KS = S::KS, CT = S::CT, NF = S::NF, F1 = S::F1, PER = NF / MLP_WAVES;
  // separate objects: reads of one buffer are then known not to wait for copies into the other
  __shared__ __attribute__((aligned(16))) _Float16 W0[S::CE], W1[S::CE];
  __shared__ __attribute__((aligned(16))) float B0[64], B1[64];   // b1 of the chunk: gate, then value
  __shared__ __attribute__((aligned(16))) float Gs[3 * C];        // LN scale, offset, b2
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, g4 = lane >> 4;
  const int nch = p.H / MLP_HC;
  const long long row_base = ((long long)blockIdx.x * MLP_WAVES + wave) * (16 * RT);

  // chunk s straight to an LDS buffer, PER fragments a wave
  const _Float16* wsrc = p.w + wave * (PER * 512) + lane * 8;
  const float* bsrc = (NG == 2 && lane >= 32 ? p.b1v : p.b1g) + (lane & 31);
  auto issue = [&](int s, _Float16* W, float* B) __attribute__((always_inline)) {
#if __HIP_DEVICE_COMPILE__   // a target builtin: the host pass, which only emits the launch stub, lacks it
#pragma unroll
    for (int k = 0; k < PER; ++k)
      __builtin_amdgcn_global_load_lds(wsrc + (size_t)s * S::CE + k * 512, W + (wave * PER + k) * 512, 16, 0, 0);
    if (wave == 0 && p.b1g) __builtin_amdgcn_global_load_lds(bsrc + s * MLP_HC, B, 4, 0, 0);
#endif
  };
  issue(0, W0, B0);
  if (!p.b1g && tid < 64) B0[tid] = B1[tid] = 0.f;
  stage_vec(Gs, p.ln_s, C, 1.f, C, tid, MLP_NT);
  stage_vec(Gs + C, p.ln_o, C, 0.f, C, tid, MLP_NT);
  stage_vec(Gs + 2 * C, p.b2, C, 0.f, C, tid, MLP_NT);
  __syncthreads();
  h8 xf[RT][KS];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const long long row = std::min(row_base + rt * 16 + r16, (long long)p.rows - 1);
    FragTile<ACT, KS> xt;
    frag_load_row(xt, p.x, (size_t)row, C, lane);
    frag_ln_raw1(xt, xf[rt], C, Gs, Gs + C, p.eps, p.fast_var, lane);
    __builtin_amdgcn_sched_barrier(0);   // one raw tile live at a time
  }

  f4 acc[RT][CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const f4 b = *reinterpret_cast<const f4*>(Gs + 2 * C + ct * 16 + 4 * g4);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[rt][ct] = b;
  }

  auto chunk = [&](int s, const _Float16* W, const float* B, _Float16* Wn, float* Bn) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();   // chunk s in LDS for every wave; every wave done with the other buffer
    issue(min(s + 1, nch - 1), Wn, Bn);
    const _Float16* cur = W + lane * 8;
    const float* Bc = B + 4 * g4;
    h8 fr[2][4];
#pragma unroll
    for (int t = 0; t < 4; ++t) fr[0][t] = *reinterpret_cast<const h8*>(cur + t * 512);
    // GEMM1: hacc[grp][rt][ht] = H^T tile (hidden 32s + 16ht + 4g4 + i, row r16)
    f4 hacc[NG][RT][2];
#pragma unroll
    for (int grp = 0; grp < NG; ++grp)
#pragma unroll
      for (int ht = 0; ht < 2; ++ht) {
        const f4 b = *reinterpret_cast<const f4*>(Bc + grp * 32 + ht * 16);
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) hacc[grp][rt][ht] = b;
      }
    h8 hb[RT];
#pragma unroll
    for (int f = 0; f < NF; f += 4) {
      // the next group of fragments is read while this group's products run
      if (f + 4 < NF) {
#pragma unroll
        for (int t = 0; t < 4; ++t) fr[(f / 4 + 1) & 1][t] = *reinterpret_cast<const h8*>(cur + (f + 4 + t) * 512);
      }
      if (f == F1) {
        // activation -> GEMM2 B fragments (k order: hidden 4g4 + i, then 16 + 4g4 + i)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          f8 v;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            v[e] = hacc[0][rt][e >> 2][e & 3];
            if constexpr (NG == 2) v[e] *= sigmoidf_(v[e]) * hacc[NG - 1][rt][e >> 2][e & 3];
          }
          hb[rt] = __builtin_convertvector(v, h8);
          if constexpr (NG == 1) hb[rt] = __builtin_elementwise_max(hb[rt], (h8)(_Float16)0.f);   // rounding keeps the sign
        }
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const h8 w = fr[(f / 4) & 1][t];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
          if (f < F1) {
            const int q = f + t, j = q / (2 * NG), grp = q / 2 % NG, ht = q & 1;
            hacc[grp][rt][ht] = mfma16(w, xf[rt][j], hacc[grp][rt][ht]);
          } else {
            const int ct = f + t - F1;
            acc[rt][ct] = mfma16(w, hb[rt], acc[rt][ct]);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  for (int s = 0;;) {
    chunk(s, W0, B0, W1, B1);
    if (++s == nch) break;
    chunk(s, W1, B1, W0, B0);
    if (++s == nch) break;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the last copy, which nothing reads

  // residual and store: lane -> row r16 of tile rt, channels 16ct + 4g4 .. +3
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const long long row = row_base + rt * 16 + r16;
    if (row >= p.rows) continue;
#pragma unroll
    for (int c4 = 0; c4 < CT; c4 += 4) {   // four tiles' residual in flight at a time
      float r[4][4];
      for (int t = 0; t < 4; ++t)
        for (int i = 0; i < 4; ++i) r[t][i] = 0.f;
      if (p.accumulate) {
#pragma unroll
        for (int t = 0; t < 4; ++t) ld4v<ACT>(p.x, (size_t)row * C + (c4 + t) * 16 + 4 * g4, r[t]);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const f4 a = acc[rt][c4 + t];
        const float v[4] = {a[0] + r[t][0], a[1] + r[t][1], a[2] + r[t][2], a[3] + r[t][3]};
        st4v<ACT>(p.out, (size_t)row * C + (c4 + t) * 16 + 4 * g4, v);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

bool mlp_supported(int C, int H, bool swiglu) {
  return H % MLP_HC == 0 && (C == 128 || (C == 256 && !swiglu));
}

size_t mlp_packed_bytes(int C, int H, bool swiglu) {
  return (size_t)(H / MLP_HC) * (size_t)((swiglu ? 2 : 1) * MLP_HC + MLP_HC) * C * sizeof(_Float16);
}

template <int ACT, int C, int NG>
static void launch_mlp(lf_context* ctx, const MlpParams& mp) {
  // Rows a wave: 32 read a weight fragment from LDS once for two products, but need two blocks of
  // 128 rows on every CU; below that 16 leave fewer CUs idle.  Measured 16 against 32: 8192 rows of
  // 256, bf16 34 / 43 us, 25578 of 256, f32 50 / 55, 41209 of 128 with SwiGLU, f32 34 / 40; 65536 of
  // 128, bf16 30.5 / 28.5, 196608 of 256, f32 290 / 258.
  const int rt = mp.rows >= 2LL * ctx->num_cus * 32 * MLP_WAVES ? 2 : 1;
  const dim3 grid((unsigned)((mp.rows + 16 * rt * MLP_WAVES - 1) / (16 * rt * MLP_WAVES)));
  auto k = rt == 2 ? mlp_kernel<ACT, C, NG, 2> : mlp_kernel<ACT, C, NG, 1>;
  hipLaunchKernelGGL(k, grid, dim3(MLP_NT), 0, ctx->stream, mp);
}

template <int ACT>
static void launch_mlp(lf_context* ctx, const MlpParams& mp, int C, bool swiglu) {
  if (C == 256) launch_mlp<ACT, 256, 1>(ctx, mp);
  else if (swiglu) launch_mlp<ACT, 128, 2>(ctx, mp);
  else launch_mlp<ACT, 128, 1>(ctx, mp);
}

int transition_fused(lf_context* ctx, const lf_transition_args& a, const WView* views, void* packed) {
  const int C = a.channels, H = a.hidden;
  const bool swiglu = a.kind == LF_TRANSITION_SWIGLU;
  const int NG = swiglu ? 2 : 1;
  const lf_transition_weights& w = *a.w;
  {
    LaunchScope ls(ctx, "transition.pack");
    const long long runs = (long long)(NG + 1) * H * C / 8;
    const long long blocks = std::min<long long>((runs + 255) / 256, 8192);
    hipLaunchKernelGGL(mlp_pack_kernel, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, views[0],
                       swiglu ? views[1] : views[0], views[NG], C, H, NG, static_cast<_Float16*>(packed));
  }
  LF_TRY(check_hip(hipGetLastError(), "transition pack launch"));
  MlpParams mp{};
  mp.x = a.act;
  mp.out = a.out;
  mp.accumulate = a.accumulate;
  mp.rows = a.rows;
  mp.H = H;
  mp.fast_var = a.fast_variance;
  mp.eps = a.epsilon;
  mp.w = static_cast<const _Float16*>(packed);
  mp.ln_s = w.norm_scale;
  mp.ln_o = w.norm_offset;
  mp.b1g = w.b1;
  mp.b1v = swiglu && w.b1 ? w.b1 + H : nullptr;
  mp.b2 = w.b2;
  {
    LaunchScope ls(ctx, "transition.fused");
    if (a.act_dtype == LF_F32) launch_mlp<DT_F32>(ctx, mp, C, swiglu);
    else if (a.act_dtype == LF_F16) launch_mlp<DT_F16>(ctx, mp, C, swiglu);
    else launch_mlp<DT_BF16>(ctx, mp, C, swiglu);
  }
  return check_hip(hipGetLastError(), "transition fused launch");
}

}  // namespace lf
