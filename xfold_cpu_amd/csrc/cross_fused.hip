// CrossAttention.forward (xfold/nn/diffusion_transformer.py:304-350) at the atom attention's widths:
// bf16 compute, 128 channels everywhere, 4 heads of 32, at most 128 keys per subset. Three
// launches instead of the composed path's thirteen:
//   cross_project  both adaptive LayerNorms and the four projections: rows of x_q give q (bf16) and
//                  the gating Linear's output (fp32), rows of x_k give k and v^T;
//   cross_attend   one wavefront per head and 16 queries: S^T = K Q^T over all keys in registers, the
//                  pair logits and the reference's positive 1e9 (a masked query on a masked key) added
//                  in fp32, softmax, O^T = V^T P^T, times sigmoid(gate);
//   cross_output   transition2(o) * sigmoid(adaptive_zero_cond(cond)), stored or accumulated.
// Rows and weights are rowstep.h's (a wavefront owns 16 rows, weights resident in LDS). scale and
// shift stay in registers (fp32), as does the gate between its sigmoid and the product.
//
// What bounded the composed path was its launches (13 for ~4 us of floor) and, in them, the
// logits' detour through an fp32 [subsets][4][32][128] buffer read back one float at a time.
// 192 subsets of 32 queries and 128 keys: 127 us of kernels before, 40 now; 1100 subsets 125.
#include <algorithm>
#include <cstring>
#include <string>

#include "common.h"
#include "kernels.h"
#include "rowstep.h"

namespace xfh {

namespace {

using rowstep::C;
constexpr int HEADS = 4, HD = 32;
constexpr int MAXK = 128;              // keys per subset (one register tile of scores)

struct Side {
  const void *x, *cond;                // [subsets * rows][128]
  const float *cond_w, *cond_b;        // LayerNorm of the condition
  const bf16 *w_scale, *w_shift;       // [128][128]
  const float *b_scale;
  const bf16 *w0, *w1;                 // q, gating / k, v
  const float *b0;                     // q bias
  int rows, steps;                     // rows per subset; 16-row steps in all
};
struct ProjectArgs {
  Side side[2];                        // queries, keys
  float cond_eps[2], x_eps[2];
  int q_wgs;                           // workgroups of the query side
  int kpad;                            // keys per subset in k and vt (a multiple of 32)
  bf16 *q, *k, *vt;                    // [subsets*nq][128]; [subsets][kpad][128]; [subsets][128][kpad]
  float *gate;                         // [subsets*nq][128]
};

// One wavefront per 16 rows at a time; the next step's rows are loaded while this one is
// computed. The key side's steps cover kpad rows of a subset, those from nk on as zeros.
// 192 subsets: 20 us for both sides (the norms and projections it replaces took 69).
template <typename TIN>
__global__ __launch_bounds__(512, 1) void cross_project_kernel(ProjectArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 w_scale[C * C], w_shift[C * C], w0[C * C], w1[C * C];
  __shared__ __attribute__((aligned(16))) float cw[C], cb[C], bs[C], b0[C];
  const bool keys = int(blockIdx.x) >= a.q_wgs;
  const Side &sd = a.side[keys ? 1 : 0];
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wg = keys ? int(blockIdx.x) - a.q_wgs : int(blockIdx.x);
  const int wgs = keys ? int(gridDim.x) - a.q_wgs : a.q_wgs;
  const int waves = wgs * 8;
  const float cond_eps = a.cond_eps[keys ? 1 : 0], x_eps = a.x_eps[keys ? 1 : 0];
  const TIN *x = static_cast<const TIN *>(sd.x), *cond = static_cast<const TIN *>(sd.cond);
  const int per = keys ? a.kpad : 0;     // key side: rows of a subset in the outputs
  // Source row of this lane in step st (clamped), and whether it exists.
  auto row_of = [&](int st, bool &in) -> int64_t {
    const int64_t row = int64_t(st) * 16 + r;
    if (!keys) {
      in = row < int64_t(sd.rows);       // (queries: rows holds subsets * nq)
      return in ? row : sd.rows - 1;
    }
    const int64_t subset = row / per;
    const int key = int(row - subset * per);
    in = key < sd.rows;
    return subset * sd.rows + (in ? key : sd.rows - 1);
  };
  struct Rows {
    rowstep::Raw4<TIN> c[8], x[8];       // K-layout condition, O-layout x
  };
  auto fetch = [&](int st, Rows &rw) {
    bool in;
    const int64_t row = row_of(st, in);
    rowstep::load_k<TIN>(cond + row * C, rw.c);
    rowstep::load_o<TIN>(x + row * C, rw.x);
  };
  int st = wg * 8 + int(threadIdx.x >> 6);
  Rows cur;
  if (st < sd.steps) fetch(st, cur);                // in flight while the weights are stored
  {
    rowstep::WeightStage<C, 512> s0, s1, s2, s3;
    s0.load([&](int r) { return sd.w_scale + r * C; }, false);
    s1.load([&](int r) { return sd.w_shift + r * C; }, false);
    s2.load([&](int r) { return sd.w0 + r * C; }, true);
    s3.load([&](int r) { return sd.w1 + r * C; }, true);
    rowstep::LnStage ln, bias;
    ln.load(sd.cond_w, sd.cond_b);
    bias.load(sd.b_scale, sd.b0);
    s0.store(w_scale);
    s1.store(w_shift);
    s2.store(w0);
    s3.store(w1);
    ln.store(cw, cb);
    bias.store(bs, b0);
    if (threadIdx.x < C) {               // LnStage's default weight is one, a bias's is zero
      if (!sd.b_scale) bs[threadIdx.x] = 0.f;
      if (!sd.b0) b0[threadIdx.x] = 0.f;
    }
  }
  __syncthreads();
  for (; st < sd.steps; st += waves) {
    Rows next;
    if (st + waves < sd.steps) fetch(st + waves, next);
    bf16x8 op[4];
    {
      float v[32];
      rowstep::k_to_float(cur.c, v);
      rowstep::ln_k(v, cw, cb, cond_eps, op);
    }
    float y[8][4];
    {
      float v[32];
      rowstep::k_to_float(cur.x, v);     // v[4 t + e]: channel 16 t + 4 g + e
      float mean, rstd;
      rowstep::ln_stats(v, x_eps, mean, rstd);
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        f32x4 sc = {0.f, 0.f, 0.f, 0.f}, sh = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          sc = mfma16(rowstep::weight_frag(w_scale, t, ks), op[ks], sc);
          sh = mfma16(rowstep::weight_frag(w_shift, t, ks), op[ks], sh);
        }
        const f32x4 b = *reinterpret_cast<const f32x4 *>(bs + 16 * t + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) y[t][e] = sigmoidf_(sc[e] + b[e]) * ((v[4 * t + e] - mean) * rstd) + sh[e];
      }
    }
    rowstep::o_to_operand(y, op);
    bool in;
    const int64_t row = row_of(st, in);
    if (!keys) {
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        f32x4 q = {0.f, 0.f, 0.f, 0.f}, gt = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
          q = mfma16(rowstep::weight_frag(w0, t, ks), op[ks], q);
          gt = mfma16(rowstep::weight_frag(w1, t, ks), op[ks], gt);
        }
        const f32x4 b = *reinterpret_cast<const f32x4 *>(b0 + 16 * t + 4 * g);
        if (in) {
          const float o[4] = {q[0] + b[0], q[1] + b[1], q[2] + b[2], q[3] + b[3]};
          rowstep::store4f<bf16>(a.q + row * C + 16 * t + 4 * g, o);
          *reinterpret_cast<f32x4 *>(a.gate + row * C + 16 * t + 4 * g) = gt;
        }
      }
    } else {
      const int64_t out_row = int64_t(st) * 16, subset = out_row / per;
      const int key0 = int(out_row - subset * per);          // a multiple of 16 below kpad
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        f32x4 k = {0.f, 0.f, 0.f, 0.f}, v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) k = mfma16(rowstep::weight_frag(w0, t, ks), op[ks], k);
        rowstep::gemm_n(w1, t, op, v);                       // 4 keys 4 g .. + 3 of channel 16 t + r
        const float ko[4] = {in ? k[0] : 0.f, in ? k[1] : 0.f, in ? k[2] : 0.f, in ? k[3] : 0.f};
        rowstep::store4f<bf16>(a.k + (out_row + r) * C + 16 * t + 4 * g, ko);
        float vo[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) vo[e] = key0 + 4 * g + e < sd.rows ? v[e] : 0.f;
        // Keys 4 g + e (even 16-key tile) or 16 + 4 g + e (odd) of a run of 32 sit at 8 g + e or
        // 8 g + 4 + e: the k order of a lane's P^T fragment.
        rowstep::store4f<bf16>(a.vt + (subset * C + 16 * t + r) * per + (key0 & ~31) + 8 * g + ((key0 >> 2) & 4), vo);
      }
    }
    cur = next;
  }
}

struct AttendArgs {
  const bf16 *q, *k, *vt;
  const float *gate;
  const void *logits;                    // element (b, h, q, key) at the strides ls, or null
  int64_t ls[4];
  const void *mask_q, *mask_k;           // [subsets][nq], [subsets][nk]
  int mask_q_dtype, mask_k_dtype;
  int nq, nk, kpad, qtiles;              // qtiles: query tiles per subset
  float scale;                           // key_dim^-0.5
  bf16 *o;                               // [subsets*nq][128]
};

// Workgroup = (subset, 16 queries), wavefront = head. Every operand is
// read straight from memory into its MFMA lanes: the whole problem of a wavefront is 8 K and 8 V
// fragments per 128 keys. 192 subsets with the heads of the logits innermost: 13 us (42 for the bias
// pass and the general kernel before).
// How a wavefront reads its logits: one by one; four consecutive keys at a time; or all four
// heads of a (query, key) at a time into LDS, for views with the heads innermost (a projection
// for several layers): lane after lane takes the next key, where the direct reads touch a cache
// line per lane (1100 subsets: 68 us direct).
enum class Logits { One, Keys, Heads };
template <typename TL, Logits MODE>
__global__ __launch_bounds__(256, 2) void cross_attend_kernel(AttendArgs a) {
  const int lane = threadIdx.x & 63, h = threadIdx.x >> 6, col = lane & 15, g = lane >> 4;
  const int64_t b = int(blockIdx.x) / a.qtiles;
  const int q0 = (int(blockIdx.x) - int(b) * a.qtiles) * 16;
  constexpr int KT = MAXK / 16;          // key tiles
  const int tiles = a.kpad / 16;
  const int qc = min(q0 + col, a.nq - 1);
  const bf16x8 qf = *reinterpret_cast<const bf16x8 *>(a.q + (b * a.nq + qc) * C + h * HD + g * 8);
  const bool masked_q = load_any(a.mask_q, a.mask_q_dtype, b * a.nq + qc) == 0.f;
  // Bit k of the words: key k is masked (wavefront ballots, so the tile loop has no mask loads).
  uint64_t masked_k[2];
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const int key = 64 * w + lane;
    masked_k[w] = __ballot(key < a.nk && load_any(a.mask_k, a.mask_k_dtype, b * a.nk + min(key, a.nk - 1)) == 0.f);
  }
  constexpr int PITCH = MAXK + 8;
  __shared__ __attribute__((aligned(16))) TL tile[MODE == Logits::Heads ? HEADS * 16 * PITCH : 1];
  if constexpr (MODE == Logits::Heads) {
    struct alignas(4 * sizeof(TL)) Four { TL v[4]; };
#pragma unroll
    for (int i = threadIdx.x; i < 16 * MAXK; i += 256) {
      const int qi = i / MAXK, key = i % MAXK;
      const int64_t at = b * a.ls[0] + min(q0 + qi, a.nq - 1) * a.ls[2] + min(key, a.nk - 1) * a.ls[3];
      const Four f = *reinterpret_cast<const Four *>(static_cast<const TL *>(a.logits) + at);
#pragma unroll
      for (int hh = 0; hh < HEADS; ++hh) tile[(hh * 16 + qi) * PITCH + key] = f.v[hh];
    }
    __syncthreads();
  }
  // Every logit of the wavefront is in flight before the first product.
  TL raw[KT][4];
  const TL *row = static_cast<const TL *>(a.logits) + b * a.ls[0] + h * a.ls[1] + qc * a.ls[2];
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    const int key0 = kt * 16 + 4 * g;
    if (!a.logits || kt >= tiles) {                  // (uniform)
#pragma unroll
      for (int e = 0; e < 4; ++e) raw[kt][e] = TL(0.f);
    } else if (MODE == Logits::Heads) {
      __builtin_memcpy(raw[kt], __builtin_assume_aligned(tile + (h * 16 + col) * PITCH + key0, 4 * sizeof(TL)),
                       4 * sizeof(TL));
    } else if (MODE == Logits::Keys && key0 + 4 <= a.nk) {
      __builtin_memcpy(raw[kt], __builtin_assume_aligned(row + key0, 4 * sizeof(TL)), 4 * sizeof(TL));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) raw[kt][e] = row[min(key0 + e, a.nk - 1) * a.ls[3]];
    }
  }
  f32x4 s[KT];
  float mx = -INFINITY;
  const float qscale = a.scale * kLog2e;
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) {
    s[kt] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (kt >= tiles) continue;           // (uniform)
    const bf16x8 kf = *reinterpret_cast<const bf16x8 *>(a.k + (b * a.kpad + kt * 16 + col) * C + h * HD + g * 8);
    const int key0 = kt * 16 + 4 * g;
    const f32x4 acc = mfma16(kf, qf, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool both = masked_q && ((masked_k[kt / 4] >> ((key0 + e) & 63)) & 1);
      const float bias = to_f32(raw[kt][e]) + (both ? 1e9f : 0.f);
      s[kt][e] = key0 + e < a.nk ? acc[e] * qscale + bias * kLog2e : -INFINITY;
      mx = fmaxf(mx, s[kt][e]);
    }
  }
  float sum = 0.f;
  f32x4 o[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
#pragma unroll
  for (int c = 0; c < KT / 2; ++c) {
    if (2 * c >= tiles) continue;
    bf16x8 vf[2];
#pragma unroll
    for (int d = 0; d < 2; ++d)
      vf[d] = *reinterpret_cast<const bf16x8 *>(a.vt + (b * C + h * HD + 16 * d + col) * a.kpad + 32 * c + 8 * g);
    bf16x8 pf;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float p0 = exp2f(s[2 * c][e] - mx), p1 = exp2f(s[2 * c + 1][e] - mx);
      sum += p0 + p1;
      pf[e] = bf16(p0);
      pf[4 + e] = bf16(p1);
    }
#pragma unroll
    for (int d = 0; d < 2; ++d) o[d] = mfma16(vf[d], pf, o[d]);
  }
  float l = sum + __shfl_xor(sum, 16, 64);
  l += __shfl_xor(l, 32, 64);
  const int q = q0 + col;
  if (q >= a.nq) return;
  const float inv = 1.0f / l;
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const int64_t at = (b * a.nq + q) * C + h * HD + 16 * d + 4 * g;
    const f32x4 gt = *reinterpret_cast<const f32x4 *>(a.gate + at);
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = sigmoidf_(gt[e]) * static_cast<float>(bf16(o[d][e] * inv));
    rowstep::store4f<bf16>(a.o + at, v);
  }
}

struct OutputArgs {
  const bf16 *o;
  const void *cond;
  const bf16 *w_zero, *w_out;
  const float *b_zero;
  void *out;
  int accumulate, rows;
};

// 16 rows per wavefront, both weights resident: 6.7 us at 192 subsets (the two GEMMs took 14.6).
template <typename TIN, typename TOUT>
__global__ __launch_bounds__(512, 1) void cross_output_kernel(OutputArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 w_zero[C * C], w_out[C * C];
  __shared__ __attribute__((aligned(16))) float bz[C], unused[C];
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int steps = (a.rows + 15) / 16, waves = int(gridDim.x) * 8;
  struct Rows {
    rowstep::Raw4<TIN> c[8];
    bf16x8 o[4];
  };
  auto fetch = [&](int st, Rows &rw) {
    const int64_t row = int64_t(st) * 16 + r, rc = row < a.rows ? row : a.rows - 1;
    rowstep::load_k<TIN>(static_cast<const TIN *>(a.cond) + rc * C, rw.c);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) rw.o[ks] = *reinterpret_cast<const bf16x8 *>(a.o + rc * C + 32 * ks + 8 * g);
  };
  int st = int(blockIdx.x) * 8 + int(threadIdx.x >> 6);
  Rows cur;
  if (st < steps) fetch(st, cur);                   // in flight while the weights are stored
  {
    rowstep::WeightStage<C, 512> s0, s1;
    rowstep::LnStage b;
    s0.load([&](int r) { return a.w_zero + r * C; }, false);
    s1.load([&](int r) { return a.w_out + r * C; }, false);
    b.load(a.b_zero, nullptr);
    s0.store(w_zero);
    s1.store(w_out);
    b.store(bz, unused);
    if (threadIdx.x < C && !a.b_zero) bz[threadIdx.x] = 0.f;
  }
  __syncthreads();
  for (; st < steps; st += waves) {
    Rows next;
    if (st + waves < steps) fetch(st + waves, next);
    const int64_t row = int64_t(st) * 16 + r, rc = row < a.rows ? row : a.rows - 1;
    bf16x8 co[4];
    float v[32];
    rowstep::k_to_float(cur.c, v);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int j = 0; j < 8; ++j) co[ks][j] = bf16(v[8 * ks + j]);
    TOUT *dst = static_cast<TOUT *>(a.out) + rc * C + 4 * g;
#pragma unroll 1                                     // (unrolled, every fragment is hoisted out of the row loop: spills)
    for (int t = 0; t < 8; ++t) {
      f32x4 z = {0.f, 0.f, 0.f, 0.f}, u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        z = mfma16(rowstep::weight_frag(w_zero, t, ks), co[ks], z);
        u = mfma16(rowstep::weight_frag(w_out, t, ks), cur.o[ks], u);
      }
      const f32x4 b = *reinterpret_cast<const f32x4 *>(bz + 16 * t + 4 * g);
      float res[4] = {0.f, 0.f, 0.f, 0.f}, w[4];
      if (a.accumulate) rowstep::load4f<TOUT>(dst + 16 * t, res);
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = res[e] + u[e] * sigmoidf_(z[e] + b[e]);
      if (row < a.rows) rowstep::store4f<TOUT>(dst + 16 * t, w);
    }
    cur = next;
  }
}

struct CrossPlan {
  bf16 *q, *k, *vt, *o;
  float *gate;
};
int64_t cross_carve(Carver &cv, CrossPlan &p, int64_t subsets, int64_t nq, int64_t nk) {
  const int64_t kpad = align_up(nk, 32);
  p.q = static_cast<bf16 *>(cv.take(subsets * nq * C * 2));
  p.k = static_cast<bf16 *>(cv.take(subsets * kpad * C * 2));
  p.vt = static_cast<bf16 *>(cv.take(subsets * kpad * C * 2));
  p.o = static_cast<bf16 *>(cv.take(subsets * nq * C * 2));
  p.gate = static_cast<float *>(cv.take(subsets * nq * C * 4));
  return cv.used;
}

bool mask_ok(int d) { return d == XFH_F32 || d == XFH_BF16 || d == XFH_BOOL; }
bool float_ok(int d) { return d == XFH_F32 || d == XFH_BF16; }
bool aligned16(const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace
}  // namespace xfh

using namespace xfh;

extern "C" {

int64_t xfh_cross_attention_workspace_size(int64_t subsets, int64_t nq, int64_t nk) {
  if (subsets < 0 || nq < 0 || nk < 0) return -1;
  Carver cv(nullptr, 0);
  CrossPlan p;
  return cross_carve(cv, p, subsets, nq, nk) + 256;
}

int xfh_cross_attention(const void *x_q, const void *x_k, const void *cond_q, const void *cond_k, int x_dtype,
                        const void *mask_q, int mask_q_dtype, const void *mask_k, int mask_k_dtype,
                        const void *logits, int logit_dtype, const int64_t *logit_strides, int64_t subsets, int64_t nq,
                        int64_t nk, const XfhCrossWeights *weights, const float *eps, float scale, void *out,
                        int out_dtype, int accumulate, void *workspace, int64_t workspace_bytes, void *stream) {
  XFH_REQUIRE(subsets >= 0 && nq >= 0 && nk >= 0, "cross_attention: bad size");
  XFH_REQUIRE(nk >= 1 && nk <= MAXK, "cross_attention: 1..128 keys per subset");
  XFH_REQUIRE(float_ok(x_dtype) && float_ok(out_dtype), "cross_attention: dtypes must be f32/bf16");
  XFH_REQUIRE(mask_ok(mask_q_dtype) && mask_ok(mask_k_dtype), "cross_attention: bad mask dtype");
  XFH_REQUIRE(!logits || (float_ok(logit_dtype) && logit_strides), "cross_attention: logits must be f32/bf16 with strides");
  if (subsets * nq == 0) return XFH_OK;
  const int64_t kpad = align_up(nk, 32);
  XFH_REQUIRE(subsets * nq < (int64_t(1) << 31) && subsets * kpad < (int64_t(1) << 31),
              "cross_attention: rows must fit in 32 bits");
  XFH_REQUIRE(x_q && x_k && cond_q && cond_k && mask_q && mask_k && weights && eps && out, "cross_attention: null tensor");
  XFH_REQUIRE(aligned16(x_q) && aligned16(x_k) && aligned16(cond_q) && aligned16(cond_k) && aligned16(out),
              "cross_attention: rows must be 16-byte aligned");
  Carver cv(workspace, workspace_bytes);
  CrossPlan p;
  const int64_t need = cross_carve(cv, p, subsets, nq, nk);
  if (!workspace || need > workspace_bytes)
    return fail(XFH_EWORKSPACE, "cross_attention: workspace too small (need " + std::to_string(need) + " bytes)");
  hipStream_t s = as_stream(stream);
  int cus = 0;
  XFH_TRY(device_cu_count(&cus));
  const XfhCrossWeights &w = *weights;
  auto b16 = [](const void *v) { return static_cast<const bf16 *>(v); };
  ProjectArgs pa;
  pa.side[0] = Side{x_q, cond_q, w.q_cond_w, w.q_cond_b, b16(w.q_scale), b16(w.q_shift), w.q_scale_b, b16(w.q),
                    b16(w.gating), w.q_b, int(subsets * nq), int(ceil_div(subsets * nq, int64_t(16)))};
  pa.side[1] = Side{x_k, cond_k, w.k_cond_w, w.k_cond_b, b16(w.k_scale), b16(w.k_shift), w.k_scale_b, b16(w.k),
                    b16(w.v), nullptr, int(nk), int(subsets * kpad / 16)};
  pa.cond_eps[0] = eps[0]; pa.x_eps[0] = eps[1]; pa.cond_eps[1] = eps[2]; pa.x_eps[1] = eps[3];
  pa.kpad = int(kpad);
  pa.q = p.q; pa.k = p.k; pa.vt = p.vt; pa.gate = p.gate;
  // One workgroup per CU in all, split by the sides' steps.
  const int64_t steps = pa.side[0].steps + int64_t(pa.side[1].steps);
  const int64_t wgs = std::max<int64_t>(2, balanced_grid(steps, 8, cus));
  const int64_t q_wgs = std::min(wgs - 1, std::max<int64_t>(1, (wgs * pa.side[0].steps + steps / 2) / steps));
  pa.q_wgs = int(q_wgs);
  {
    KernelTimer timer("cross_project", s, 0.0, true);
    if (x_dtype == XFH_BF16) timer.launch(cross_project_kernel<bf16>, dim3(unsigned(wgs)), dim3(512), 0, pa);
    else timer.launch(cross_project_kernel<float>, dim3(unsigned(wgs)), dim3(512), 0, pa);
    XFH_TRY(check_launch("cross_project"));
  }
  AttendArgs aa;
  std::memset(&aa, 0, sizeof(aa));
  aa.q = p.q; aa.k = p.k; aa.vt = p.vt; aa.gate = p.gate; aa.o = p.o;
  aa.logits = logits;
  if (logits) for (int i = 0; i < 4; ++i) aa.ls[i] = logit_strides[i];
  aa.mask_q = mask_q; aa.mask_q_dtype = mask_q_dtype; aa.mask_k = mask_k; aa.mask_k_dtype = mask_k_dtype;
  aa.nq = int(nq); aa.nk = int(nk); aa.kpad = int(kpad); aa.qtiles = int(ceil_div(nq, int64_t(16)));
  aa.scale = scale;
  const int64_t grid = subsets * aa.qtiles;
  XFH_REQUIRE(grid < (int64_t(1) << 31), "cross_attention: too many subsets");
  {
    // Four keys or four heads in one load where every group of four is aligned.
    const int64_t el = logit_dtype == XFH_F32 ? 4 : 2;
    const bool four = logits && aa.ls[0] % 4 == 0 && aa.ls[2] % 4 == 0 && reinterpret_cast<uintptr_t>(logits) % (4 * el) == 0;
    const Logits mode = four && aa.ls[3] == 1 && aa.ls[1] % 4 == 0 ? Logits::Keys
                        : four && aa.ls[1] == 1 && aa.ls[3] % 4 == 0 ? Logits::Heads
                                                                     : Logits::One;
    KernelTimer timer("cross_attend", s, 0.0, true);
    const dim3 grid3{unsigned(grid)};
    auto go = [&](auto tl) {
      using TL = decltype(tl);
      if (mode == Logits::Keys) timer.launch(cross_attend_kernel<TL, Logits::Keys>, grid3, dim3(256), 0, aa);
      else if (mode == Logits::Heads) timer.launch(cross_attend_kernel<TL, Logits::Heads>, grid3, dim3(256), 0, aa);
      else timer.launch(cross_attend_kernel<TL, Logits::One>, grid3, dim3(256), 0, aa);
    };
    if (logits && logit_dtype == XFH_F32) go(0.0f);
    else go(bf16(0.0f));
    XFH_TRY(check_launch("cross_attend"));
  }
  OutputArgs oa{p.o, cond_q, b16(w.zero), b16(w.output), w.zero_b, out, accumulate, int(subsets * nq)};
  KernelTimer timer("cross_output", s, 0.0, true);
  const dim3 og(unsigned(balanced_grid(ceil_div(subsets * nq, int64_t(16)), 8, cus)));
  if (x_dtype == XFH_BF16 && out_dtype == XFH_BF16) timer.launch(cross_output_kernel<bf16, bf16>, og, dim3(512), 0, oa);
  else if (x_dtype == XFH_BF16) timer.launch(cross_output_kernel<bf16, float>, og, dim3(512), 0, oa);
  else if (out_dtype == XFH_BF16) timer.launch(cross_output_kernel<float, bf16>, og, dim3(512), 0, oa);
  else timer.launch(cross_output_kernel<float, float>, og, dim3(512), 0, oa);
  return check_launch("cross_output");
}

}  // extern "C"
