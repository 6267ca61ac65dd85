// Vector epilogue of the GEMM kernels (gemm_ring.hip, gemm_direct.h, gemm.hip): a lane holds four
// consecutive output columns of a row, so bias, auxiliary operand, accumulation and the store are
// 8 (bf16) or 16 (fp32) bytes.
#pragma once

#include "common.h"
#include "kernels.h"

namespace xfh {
namespace {

template <typename TO> struct Vec4;
template <> struct Vec4<bf16> {
  __device__ static void load(const bf16 *p, float (&v)[4]) {
    const bf16x4 x = *reinterpret_cast<const bf16x4 *>(p);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = static_cast<float>(x[e]);
  }
  __device__ static void store(bf16 *p, const float (&v)[4]) {
    bf16x4 x;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = bf16(v[e]);
    *reinterpret_cast<bf16x4 *>(p) = x;
  }
};
template <> struct Vec4<float> {
  __device__ static void load(const float *p, float (&v)[4]) {
    const float4 x = *reinterpret_cast<const float4 *>(p);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
  }
  __device__ static void store(float *p, const float (&v)[4]) {
    *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
  }
};

template <int EPI> __device__ __forceinline__ float epilogue(float acc, float c, float aux) {
  if constexpr (EPI == XFH_EPI_MUL_SIGMOID_AUX) return acc * sigmoidf_(aux);
  else if constexpr (EPI == XFH_EPI_SIGMOID_MUL_AUX) return sigmoidf_(acc) * aux;
  else if constexpr (EPI == XFH_EPI_ACCUMULATE) return c + acc;
  else if constexpr (EPI == XFH_EPI_MUL_SIGMOID_AUX_ACCUMULATE) return c + acc * sigmoidf_(aux);
  else return acc;
}

// Stores one wavefront's 64 x (16 NT) sub-tile (rows mw + 16 y + col, columns nw + 16 x +
// 4 grp + e) through epilogue EPI. The epilogue kind is a template parameter and the row
// quantities (row divisor, auxiliary row) are taken once per row: a runtime switch per
// element made this code ~10x larger than the main loop, and its instruction-cache misses
// cost ~10 us per launch whatever the grid. DIV divides by the row divisor; else its
// reciprocal, taken once per row, multiplies (one fp32 rounding more, on bf16 products).
template <int EPI, typename TO, int NT, bool DIV = false, int MT>
__device__ __forceinline__ void store_tile(const GemmArgs &p, const f32x4 (&acc)[NT][MT], int64_t batch, int mw,
                                           int nw, int col, int grp) {
  constexpr bool READS_C = EPI == XFH_EPI_ACCUMULATE || EPI == XFH_EPI_MUL_SIGMOID_AUX_ACCUMULATE;
  constexpr bool AUX = EPI == XFH_EPI_MUL_SIGMOID_AUX || EPI == XFH_EPI_SIGMOID_MUL_AUX ||
                       EPI == XFH_EPI_MUL_SIGMOID_AUX_ACCUMULATE;
  TO *C = static_cast<TO *>(p.C) + batch * p.sC;
  auto scaled = [](float v, float r) { return DIV ? v / r : v * r; };
  int m[MT];
  float rs[MT];
  const TO *arow[MT];
#pragma unroll
  for (int y = 0; y < MT; ++y) {
    m[y] = mw + y * 16 + col;
    rs[y] = 1.0f;
    if (p.row_div && m[y] < p.M) rs[y] = DIV ? p.row_div_eps + p.row_div[m[y]] : 1.0f / (p.row_div_eps + p.row_div[m[y]]);
    arow[y] = nullptr;
    if constexpr (AUX) {
      const int ar = p.aux_rows > 0 ? m[y] % int(p.aux_rows) : m[y];
      arow[y] = static_cast<const TO *>(p.aux) + batch * p.sAux + int64_t(ar) * p.ldaux;
    }
  }
  if (p.pair_blk == 0 && mw + 16 * MT <= p.M && nw + 16 * NT <= p.N) {
    // Interior sub-tile (every tile of the usual shapes): straight-line code, no per-element
    // bounds, row-major addresses.
#pragma unroll
    for (int x = 0; x < NT; ++x) {
      const int n = nw + x * 16 + grp * 4;
      float bias[4] = {0.f, 0.f, 0.f, 0.f};
      if (p.bias)
#pragma unroll
        for (int e = 0; e < 4; ++e) bias[e] = p.bias[batch * p.sBias + n + e];
#pragma unroll
      for (int y = 0; y < MT; ++y) {
        TO *c = C + int64_t(m[y]) * p.ldc + n;
        float cv[4] = {0.f, 0.f, 0.f, 0.f}, av[4] = {0.f, 0.f, 0.f, 0.f}, out[4];
        if constexpr (READS_C) Vec4<TO>::load(c, cv);
        if constexpr (AUX) Vec4<TO>::load(arow[y] + n, av);
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = epilogue<EPI>(scaled(acc[x][y][e] + bias[e], rs[y]), cv[e], av[e]);
        Vec4<TO>::store(c, out);
      }
    }
    return;
  }
#pragma unroll
  for (int x = 0; x < NT; ++x) {
    const int n = nw + x * 16 + grp * 4;
    if (n >= p.N) continue;
    const bool full = n + 4 <= p.N;
    float bias[4] = {0.f, 0.f, 0.f, 0.f};
    if (p.bias)
#pragma unroll
      for (int e = 0; e < 4; ++e) bias[e] = n + e < p.N ? p.bias[batch * p.sBias + n + e] : 0.f;
#pragma unroll
    for (int y = 0; y < MT; ++y) {
      if (m[y] >= p.M) continue;
      TO *c = c_element(p, C, m[y], n);
      float cv[4] = {0.f, 0.f, 0.f, 0.f}, av[4] = {0.f, 0.f, 0.f, 0.f}, out[4];
      if (full) {
        if constexpr (READS_C) Vec4<TO>::load(c, cv);
        if constexpr (AUX) Vec4<TO>::load(arow[y] + n, av);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (n + e >= p.N) continue;
          if constexpr (READS_C) cv[e] = to_f32(c[e]);
          if constexpr (AUX) av[e] = to_f32(arow[y][n + e]);
        }
      }
      // (acc + bias) * 1.0f is exact, so rows without a divisor keep acc + bias.
#pragma unroll
      for (int e = 0; e < 4; ++e) out[e] = epilogue<EPI>(scaled(acc[x][y][e] + bias[e], rs[y]), cv[e], av[e]);
      if (full) {
        Vec4<TO>::store(c, out);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < p.N) c[e] = from_f32<TO>(out[e]);
      }
    }
  }
}

// The runtime switch over the epilogue kinds, once per sub-tile. DIV: products with a row divisor
// (OuterProductMean's, stored or accumulated) divide.
template <bool DIV, typename TO, int NT, int MT>
__device__ __forceinline__ void store_any(const GemmArgs &p, const f32x4 (&acc)[NT][MT], int64_t batch, int mw, int nw,
                                          int col, int grp) {
  if constexpr (DIV) {
    if (p.row_div && p.epi == XFH_EPI_STORE)
      return store_tile<XFH_EPI_STORE, TO, NT, true>(p, acc, batch, mw, nw, col, grp);
    if (p.row_div && p.epi == XFH_EPI_ACCUMULATE)
      return store_tile<XFH_EPI_ACCUMULATE, TO, NT, true>(p, acc, batch, mw, nw, col, grp);
  }
  switch (p.epi) {
    case XFH_EPI_MUL_SIGMOID_AUX: store_tile<XFH_EPI_MUL_SIGMOID_AUX, TO, NT>(p, acc, batch, mw, nw, col, grp); break;
    case XFH_EPI_SIGMOID_MUL_AUX: store_tile<XFH_EPI_SIGMOID_MUL_AUX, TO, NT>(p, acc, batch, mw, nw, col, grp); break;
    case XFH_EPI_ACCUMULATE: store_tile<XFH_EPI_ACCUMULATE, TO, NT>(p, acc, batch, mw, nw, col, grp); break;
    case XFH_EPI_MUL_SIGMOID_AUX_ACCUMULATE:
      store_tile<XFH_EPI_MUL_SIGMOID_AUX_ACCUMULATE, TO, NT>(p, acc, batch, mw, nw, col, grp);
      break;
    default: store_tile<XFH_EPI_STORE, TO, NT>(p, acc, batch, mw, nw, col, grp);
  }
}

// Whether C (and aux) take four consecutive columns in one aligned access of `ob`-byte elements.
inline bool vector_output(const GemmArgs &p, int ob) {
  auto al = [](const void *ptr, int bytes) { return reinterpret_cast<uintptr_t>(ptr) % bytes == 0; };
  if (p.pair_blk && (p.pair_blk % 4 || !al(p.C, 4 * ob) || p.sC % 4)) return false;
  return p.aux_rows <= INT32_MAX && p.ldc % 4 == 0 && p.sC % 4 == 0 && al(p.C, 4 * ob) &&
         (!p.aux || (p.ldaux % 4 == 0 && p.sAux % 4 == 0 && al(p.aux, 4 * ob)));
}

}  // namespace
}  // namespace xfh
