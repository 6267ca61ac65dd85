// Transition at 64 channels (bf16 compute): the template stack's pair transition (128 hidden features) and
// the MSA stack's (256), xfold/nn/primitives.py:33-37: LN(x) -> silu(x Wg) * (x Wv) -> transition2 -> x += update.
//
// The whole weight set fits in LDS (48 or 96 KB), so unlike the 128-channel kernel
// (transition_fused.hip) nothing streams: a wavefront takes 32 rows at a time (rowstep.h
// layouts, two sets of 16 that share every weight fragment), the next rows in flight, and no
// barrier after the weights are in. The hidden features never leave the registers: transition1's
// rows are permuted on their way into LDS so that a lane's gate and value results are the
// k-operand of transition2. The bound is HBM (a row is read and written once); the composed path
// (LayerNorm, GLU GEMM, GEMM) moved 5 and 9 times the bytes through its normed rows and hidden features.
// us per call, before -> now: 512 x 256 rows, f = 256 54 -> 26; 300 x 300 rows, f = 128 39 -> 17.5.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "rowstep.h"

namespace xfh {

namespace {

using namespace rowstep;
constexpr int CW = 64;                 // channels
constexpr int KS1 = CW / 32, NT = CW / 16;

// INPLACE (bf16 x updated in place): the accumulators start from x itself.
template <typename TIN, typename TOUT, int F, bool INPLACE>
__global__ __launch_bounds__(512, 1) void transition_rows_kernel(TransitionArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 w1[2 * F * CW];
  __shared__ __attribute__((aligned(16))) bf16 w2[CW * F];
  __shared__ __attribute__((aligned(16))) float lnw[CW], lnb[CW];
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const TIN *x = static_cast<const TIN *>(a.x);
  TOUT *out = static_cast<TOUT *>(a.out);
  const int64_t steps = (a.rows + 31) / 32, waves = int64_t(gridDim.x) * 8;
  struct Rows {
    Raw4<TIN> z[2][2 * KS1];
  };
  auto fetch = [&](int64_t st, Rows &rw) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t row = st * 32 + 16 * i + r;
      load_k<TIN>(x + (row < a.rows ? row : a.rows - 1) * CW, rw.z[i]);
    }
  };
  int64_t st = int64_t(blockIdx.x) * 8 + (threadIdx.x >> 6);
  Rows cur;
  if (st < steps) fetch(st, cur);                   // in flight while the weights are stored
  {
    // Row 64 c + 16 t + m of the LDS copy: chunk c of 32 hidden features, tile t (0, 1 gate, 2, 3
    // value), whose row m is feature 8 (m / 4) + 4 (t % 2) + m % 4 of the chunk.
    WeightStage<2 * F, 512, CW> s1;
    WeightStage<CW, 512, F> s2;
    LnStageOf<CW> sl;
    s1.load([&](int n) {
      const int c = n >> 6, t = (n >> 4) & 3, m = n & 15, f = 8 * (m >> 2) + 4 * (t & 1) + (m & 3);
      return a.w1 + (64 * c + 32 * (f >> 4) + (t < 2 ? 0 : 16) + (f & 15)) * CW;
    }, false);
    s2.load([&](int n) { return a.w2 + n * F; }, false);
    sl.load(a.ln_w, a.ln_b);
    s1.store(w1);
    s2.store(w2);
    sl.store(lnw, lnb);
  }
  __syncthreads();
  bf16x8 id[2];
  identity_frags(id);
  for (; st < steps; st += waves) {
    Rows next;
    if (st + waves < steps) fetch(st + waves, next);
    bf16x8 xop[2][KS1];
    f32x4 acc[2][NT];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float v[CW / 4];
      k_to_float(cur.z[i], v);
      ln_k(v, lnw, lnb, a.eps, xop[i]);
      if constexpr (INPLACE) {
        bf16x8 zk[KS1];
#pragma unroll
        for (int ks = 0; ks < KS1; ++ks)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            zk[ks][e] = cur.z[i][2 * ks].v[e];
            zk[ks][4 + e] = cur.z[i][2 * ks + 1].v[e];
          }
        k_to_o(id, zk, acc[i]);
      } else {
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
#pragma unroll 1                                    // (unrolled, the fragments are hoisted out of the row loop)
    for (int c = 0; c < F / 32; ++c) {
      f32x4 h[2][4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int i = 0; i < 2; ++i) h[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS1; ++ks) {
          const bf16x8 wf = weight_frag<CW>(w1, 4 * c + t, ks);
#pragma unroll
          for (int i = 0; i < 2; ++i) h[i][t] = mfma16(wf, xop[i][ks], h[i][t]);
        }
      }
      bf16x8 hop[2];                                // lane g: hidden features 8 g .. 8 g + 7
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          hop[i][e] = bf16(siluf_(h[i][0][e]) * h[i][2][e]);
          hop[i][4 + e] = bf16(siluf_(h[i][1][e]) * h[i][3][e]);
        }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const bf16x8 wf = weight_frag<F>(w2, t, c);
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i][t] = mfma16(wf, hop[i], acc[i][t]);
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t row = st * 32 + 16 * i + r;
      if (row < a.rows) {
        TOUT *dst = out + row * CW + 4 * g;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          float o[4] = {acc[i][t][0], acc[i][t][1], acc[i][t][2], acc[i][t][3]};
          if (!INPLACE && a.accumulate) {
            float old[4];
            load4f<TOUT>(dst + 16 * t, old);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] += old[e];
          }
          store4f<TOUT>(dst + 16 * t, o);
        }
      }
    }
    cur = next;
  }
}

template <int F> int launch(const TransitionArgs &a, int x_dtype, int out_dtype, hipStream_t s) {
  int cus = 0;
  XFH_TRY(device_cu_count(&cus));
  const dim3 grid(unsigned(balanced_grid(ceil_div(a.rows, int64_t(32)), 8, cus)));
  KernelTimer timer("transition_rows", s, 0.0, true);
  const bool in_place = a.accumulate && a.out == a.x;
  if (x_dtype == XFH_BF16 && out_dtype == XFH_BF16 && in_place)
    timer.launch(transition_rows_kernel<bf16, bf16, F, true>, grid, dim3(512), 0, a);
  else if (x_dtype == XFH_BF16 && out_dtype == XFH_BF16)
    timer.launch(transition_rows_kernel<bf16, bf16, F, false>, grid, dim3(512), 0, a);
  else if (x_dtype == XFH_BF16)
    timer.launch(transition_rows_kernel<bf16, float, F, false>, grid, dim3(512), 0, a);
  else if (out_dtype == XFH_F32)
    timer.launch(transition_rows_kernel<float, float, F, false>, grid, dim3(512), 0, a);
  else
    timer.launch(transition_rows_kernel<float, bf16, F, false>, grid, dim3(512), 0, a);
  return check_launch("transition_rows");
}

}  // namespace

int transition_rows(const TransitionArgs &a, int f, int x_dtype, int out_dtype, hipStream_t s) {
  if (a.rows == 0) return XFH_OK;
  return f == 128 ? launch<128>(a, x_dtype, out_dtype, s) : launch<256>(a, x_dtype, out_dtype, s);
}

}  // namespace xfh
