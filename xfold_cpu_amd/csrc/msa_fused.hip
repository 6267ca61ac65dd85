// Row kernels of the MSA stack at 64 MSA channels (bf16 compute; rowstep.h layouts, weights resident in
// LDS, a wavefront per unit of rows, the next unit's rows in flight):
//   msa_project  LayerNorm(msa) and one [64][64] projection, written channel by channel along the
//                sequences (OuterProductMean's masked left/right operands and its mask) or along
//                the keys (MSAAttention's values), where a GEMM over that axis reads them;
//   msa_output   MSAAttention's tail: the averages back to row order, times sigmoid(gating), the output
//                projection, msa += update.
// Both are bound by HBM: the rows once in, the result once out. They replace LayerNorm -> GEMM ->
// transposing kernel chains (us at 512 x 256: OuterProductMean's operands 41 -> 11, the values 56 -> 11,
// gather, gate and output projection 49 -> 13).
#include <algorithm>

#include "common.h"
#include "kernels.h"
#include "rowstep.h"

namespace xfh {

namespace {

using namespace rowstep;
constexpr int CM = 64, KS = CM / 32, NT = CM / 16;

// Unit u = (line, 32 positions t0 ..): rows line * line_rows + t * t_rows of the MSA for t < t_len and
// line < lines, zeros up to t_pad and lines_pad. Row m of row tile rt is position t0 + 8 (m / 4) +
// 4 rt + m % 4, so the lane that holds channel c of rows 4 g .. + 3 in both tiles has 8 consecutive
// positions: one 16-byte store (as in trimul_project).
template <typename TIN>
__global__ __launch_bounds__(512, 2) void msa_project_kernel(MsaProjectArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 w[CM * CM];
  __shared__ __attribute__((aligned(16))) float lnw[CM], lnb[CM];
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  const int per_line = a.t_pad / 32, units = a.lines_pad * per_line, waves = int(gridDim.x) * 8;
  const TIN *x = static_cast<const TIN *>(a.x);
  struct Unit {
    Raw4<TIN> z[2][NT];
    float mask[2];
  };
  auto fetch = [&](int u, Unit &un) {
    const int line = u / per_line, t0 = (u - line * per_line) * 32;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      const int t = t0 + 8 * (m >> 2) + 4 * rt + (m & 3);
      const bool in = t < a.t_len && line < a.lines;
      const int64_t row = in ? line * a.line_rows + t * a.t_rows : 0;
      load_k<TIN>(x + row * CM, un.z[rt]);
      un.mask[rt] = !in ? 0.f : a.mask ? load_any(a.mask, a.mask_dtype, row) : 1.f;
    }
  };
  int u = int(blockIdx.x) * 8 + int(threadIdx.x >> 6);
  Unit cur;
  if (u < units) fetch(u, cur);                     // in flight while the weights are stored
  {
    WeightStage<CM, 512, CM> s;
    LnStageOf<CM> sl;
    s.load([&](int r) { return a.w + r * CM; }, false);
    sl.load(a.ln_w, a.ln_b);
    s.store(w);
    sl.store(lnw, lnb);
  }
  __syncthreads();
  for (; u < units; u += waves) {
    Unit next;
    if (u + waves < units) fetch(u + waves, next);
    const int line = u / per_line, t0 = (u - line * per_line) * 32;
    bf16x8 xa[2][KS];
    float mk[8];                                    // mask of positions t0 + 8 g + 0..7
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
      float v[CM / 4];
      k_to_float(cur.z[rt], v);
      ln_k(v, lnw, lnb, a.eps, xa[rt]);
#pragma unroll
      for (int e = 0; e < 4; ++e) mk[4 * rt + e] = __shfl(cur.mask[rt], 4 * g + e, 64);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4 acc[2];
#pragma unroll
      for (int rt = 0; rt < 2; ++rt) {
        acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
        gemm_n(w, t, xa[rt], acc[rt]);
      }
      bf16x8 o;
#pragma unroll
      for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        // (a position without a row has mask 0 but row 0's product, which may be infinite)
        for (int e = 0; e < 4; ++e)
          o[4 * rt + e] = t0 + 8 * g + 4 * rt + e < a.t_len && line < a.lines ? bf16(acc[rt][e] * mk[4 * rt + e]) : bf16(0.0f);
      const int p = 16 * t + m;
      bf16 *dst = p < a.split ? a.out0 + p * a.ch_stride : a.out1 + (p - a.split) * a.ch_stride;
      *reinterpret_cast<bf16x8 *>(dst + line * a.line_stride + t0 + 8 * g) = o;
    }
    if (a.mask_out && m == 0) {                     // lane (0, g): the mask of its 8 positions
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = bf16(mk[e]);
      *reinterpret_cast<bf16x8 *>(a.mask_out + int64_t(line) * a.t_pad + t0 + 8 * g) = o;
    }
    cur = next;
  }
}

// Step = residue q, sequences s0 .. s0 + 15. The averages of a channel are contiguous along the
// sequences: 16-byte loads are MFMA A fragments, and identity B fragments turn them to row
// order (as trimul_output reads the contraction's result).
template <typename TIN, typename TOUT>
__global__ __launch_bounds__(512, 2) void msa_output_kernel(MsaOutputArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 w_gate[CM * CM], w_out[CM * CM];
  __shared__ __attribute__((aligned(16))) float lnw[CM], lnb[CM];
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int blocks = a.rows_pad / 16, steps = a.n * blocks, waves = int(gridDim.x) * 8;
  const TIN *x = static_cast<const TIN *>(a.x);
  TOUT *out = static_cast<TOUT *>(a.out);
  constexpr bool kBf16 = sizeof(TIN) == 2 && sizeof(TOUT) == 2;
  const bool res_from_x = kBf16 && a.accumulate && a.x == a.out;
  const bool res_load = a.accumulate && !res_from_x;
  const int dv_log2 = __builtin_ctz(a.dv);           // (dv divides 64)
  bf16x8 id[2];
  identity_frags(id);
  struct Rows {
    Raw4<TIN> z[NT];
    bf16x8 c[KS];
  };
  auto row_of = [&](int st, int &s) -> int64_t {
    const int q = st / blocks;
    s = (st - q * blocks) * 16 + r;
    return int64_t(s < a.rows ? s : a.rows - 1) * a.n + q;
  };
  auto fetch = [&](int st, Rows &rw) {
    int s;
    load_k<TIN>(x + row_of(st, s) * CM, rw.z);
    const int q = st / blocks, s0 = (st - q * blocks) * 16;
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      const int p = 16 * (k + KS * (g >> 1)) + r, h = p >> dv_log2, c = p - h * a.dv;
      rw.c[k] = *reinterpret_cast<const bf16x8 *>(a.avg_t + ((int64_t(h) * a.n + q) * a.dv + c) * a.rows_pad + s0 + 8 * (g & 1));
    }
  };
  int st = int(blockIdx.x) * 8 + int(threadIdx.x >> 6);
  Rows cur;
  if (st < steps) fetch(st, cur);                   // in flight while the weights are stored
  {
    WeightStage<CM, 512, CM> sg, so;
    LnStageOf<CM> sl;
    sg.load([&](int row) { return a.w_gating + row * CM; }, false);
    so.load([&](int row) { return a.w_out + row * CM; }, true);
    sl.load(a.ln_w, a.ln_b);
    sg.store(w_gate);
    so.store(w_out);
    sl.store(lnw, lnb);
  }
  __syncthreads();
  for (; st < steps; st += waves) {
    Rows next;
    if (st + waves < steps) fetch(st + waves, next);
    bf16x8 op[KS];
    {
      float v[CM / 4];
      k_to_float(cur.z, v);
      ln_k(v, lnw, lnb, a.eps, op);
    }
    f32x4 acc[NT], avg[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    gemm_t(w_gate, op, acc);
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      avg[k] = mfma16(cur.c[k], id[0], f32x4{0.f, 0.f, 0.f, 0.f});
      avg[k + KS] = mfma16(cur.c[k], id[1], f32x4{0.f, 0.f, 0.f, 0.f});
    }
    if (moved_nonfinite(avg)) {                      // a bad sequence leaves the 15 others of its step alone
      const int q = st / blocks, s0 = (st - q * blocks) * 16;
      int p0 = 4 * g;
      asm volatile("" : "+v"(p0));                   // (keeps the 16 offsets in here: 60 registers)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int p = 16 * t + p0 + e, h = p >> dv_log2, c = p - h * a.dv;
          avg[t][e] = static_cast<float>(a.avg_t[((int64_t(h) * a.n + q) * a.dv + c) * a.rows_pad + s0 + r]);
        }
    }
    float y[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) y[t][e] = sigmoidf_(acc[t][e]) * avg[t][e];
    o_to_operand(y, op);
    f32x4 res[NT];
    if (res_from_x) {
      if constexpr (kBf16) {
        bf16x8 zk[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            zk[ks][e] = cur.z[2 * ks].v[e];
            zk[ks][4 + e] = cur.z[2 * ks + 1].v[e];
          }
        k_to_o(id, zk, res);
      }
    } else {
#pragma unroll
      for (int t = 0; t < NT; ++t) res[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    gemm_t(w_out, op, res);                         // the accumulators start from the residual
    int s;
    const int64_t row = row_of(st, s);
    if (s < a.rows) {
      TOUT *dst = out + row * CM + 4 * g;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        float o[4] = {res[t][0], res[t][1], res[t][2], res[t][3]};
        if (res_load) {
          float old[4];
          load4f<TOUT>(dst + 16 * t, old);
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] += old[e];
        }
        store4f<TOUT>(dst + 16 * t, o);
      }
    }
    cur = next;
  }
}

}  // namespace

int msa_project(const MsaProjectArgs &a, int x_dtype, hipStream_t s) {
  const int64_t units = int64_t(a.lines_pad) * (a.t_pad / 32);
  if (units == 0) return XFH_OK;
  if (a.t_pad % 32 || units >= (int64_t(1) << 31)) return fail(XFH_EUNSUPPORTED, "msa_project: problem too large");
  int cus = 0;
  XFH_TRY(device_cu_count(&cus));
  const dim3 grid(unsigned(balanced_grid(units, 8, 2 * cus)));
  KernelTimer timer("msa_project", s, 0.0, true);
  if (x_dtype == XFH_BF16) timer.launch(msa_project_kernel<bf16>, grid, dim3(512), 0, a);
  else timer.launch(msa_project_kernel<float>, grid, dim3(512), 0, a);
  return check_launch("msa_project");
}

int msa_output(const MsaOutputArgs &a, int x_dtype, int out_dtype, hipStream_t s) {
  const int64_t steps = int64_t(a.n) * (a.rows_pad / 16);
  if (steps == 0) return XFH_OK;
  if (a.rows_pad % 16 || steps >= (int64_t(1) << 31)) return fail(XFH_EUNSUPPORTED, "msa_output: problem too large");
  int cus = 0;
  XFH_TRY(device_cu_count(&cus));
  const dim3 grid(unsigned(balanced_grid(steps, 8, 2 * cus)));
  KernelTimer timer("msa_output", s, 0.0, true);
  if (x_dtype == XFH_BF16 && out_dtype == XFH_BF16) timer.launch(msa_output_kernel<bf16, bf16>, grid, dim3(512), 0, a);
  else if (x_dtype == XFH_BF16) timer.launch(msa_output_kernel<bf16, float>, grid, dim3(512), 0, a);
  else if (out_dtype == XFH_BF16) timer.launch(msa_output_kernel<float, bf16>, grid, dim3(512), 0, a);
  else timer.launch(msa_output_kernel<float, float>, grid, dim3(512), 0, a);
  return check_launch("msa_output");
}

}  // namespace xfh
