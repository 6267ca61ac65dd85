// bf16 "NT" GEMM for outputs too small to fill the chip with gemm_ring's tiles (included by
// gemm_ring.hip, whose epilogues it uses): C[b][m][n] = epilogue(sum_k A[b][m][k] B[b][n][k]).
//
// A workgroup owns a 16 TM x 16 TN output tile and its KW wavefronts split the sum over k: wavefront w
// takes the 32-deep k-substeps w, w + KW, .. Fragments go global -> registers (a lane's 16 bytes
// of a row are its MFMA operand), U substeps ahead, with no LDS and no barrier in the loop; the
// partial tiles are added through LDS in wavefront order and every wavefront finishes a share of
// the tile. What bounds such a launch is the latency of its serial k-loop: gemm_ring's 64-column
// tile gives 12 workgroups on a [96][768] output and walks k = 1536 in 24 barrier-separated steps;
// here it is 72 workgroups and 3 rounds of loads per wavefront.
#pragma once

namespace xfh {
namespace {

template <int TM_, int TN_, int KW_, int U_> struct Direct {
  static constexpr int TM = TM_, TN = TN_, KW = KW_, U = U_;
  static constexpr int BM = 16 * TM, BN = 16 * TN;
  static constexpr int TILES = TM * TN;                   // MFMA tiles of the output tile
  static_assert(TN % 2 == 0, "GLU pairs two 16-column tiles");
};

template <typename T> __device__ __forceinline__ typename Frag<T>::type direct_frag(const T *p);
template <> __device__ __forceinline__ bf16x8 direct_frag<bf16>(const bf16 *p) { return *reinterpret_cast<const bf16x8 *>(p); }
template <> __device__ __forceinline__ f32x8 direct_frag<float>(const float *p) {
  f32x8 f;
  const float4 lo = reinterpret_cast<const float4 *>(p)[0], hi = reinterpret_cast<const float4 *>(p)[1];
  f.v[0] = lo.x; f.v[1] = lo.y; f.v[2] = lo.z; f.v[3] = lo.w;
  f.v[4] = hi.x; f.v[5] = hi.y; f.v[6] = hi.z; f.v[7] = hi.w;
  return f;
}

template <typename T, typename TO, bool GLU, class G, bool ATTN>
__global__ __launch_bounds__(64 * G::KW) void gemm_direct_kernel(GemmArgs p) {
  constexpr int TM = G::TM, TN = G::TN, KW = G::KW, U = G::U, TILES = G::TILES;
  __shared__ __attribute__((aligned(16))) f32x4 part[KW][TILES][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int m0 = blockIdx.y * G::BM, n0 = blockIdx.x * G::BN;
  const int64_t batch = blockIdx.z;
  // Rows past M or N read the last row (their results are never stored).
  const T *a[TM], *b[TN];
#pragma unroll
  for (int y = 0; y < TM; ++y) {
    const int m = m0 + 16 * y + col;
    a[y] = static_cast<const T *>(p.A) + batch * p.sA + int64_t(m < p.M ? m : p.M - 1) * p.lda + grp * 8;
  }
#pragma unroll
  for (int x = 0; x < TN; ++x) {
    const int n = n0 + 16 * x + col;
    b[x] = static_cast<const T *>(p.B) + batch * p.sB + int64_t(n < p.N ? n : p.N - 1) * p.ldb + grp * 8;
  }
  f32x4 acc[TN][TM];
#pragma unroll
  for (int x = 0; x < TN; ++x)
#pragma unroll
    for (int y = 0; y < TM; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = p.K / 32;
  struct Frags {
    typename Frag<T>::type a[U][TM], b[U][TN];
  };
  auto load = [&](Frags &f, int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u * KW;
      if (s >= steps) break;                              // (uniform over the wavefront)
#pragma unroll
      for (int y = 0; y < TM; ++y) f.a[u][y] = direct_frag<T>(a[y] + s * 32);
#pragma unroll
      for (int x = 0; x < TN; ++x) f.b[u][x] = direct_frag<T>(b[x] + s * 32);
    }
  };
  auto multiply = [&](const Frags &f, int s0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s0 + u * KW >= steps) break;
      mfma_tiles(f.b[u], f.a[u], acc);
    }
  };
  Frags f0, f1;
  load(f0, wave);
  for (int s = wave; s < steps; s += 2 * U * KW) {
    load(f1, s + U * KW);
    multiply(f0, s);
    load(f0, s + 2 * U * KW);
    multiply(f1, s + U * KW);
  }
#pragma unroll
  for (int x = 0; x < TN; ++x)
#pragma unroll
    for (int y = 0; y < TM; ++y) part[wave][x * TM + y][lane] = acc[x][y];
  __syncthreads();
  auto total = [&](int tile) {
    f32x4 v = part[0][tile][lane];
#pragma unroll
    for (int w = 1; w < KW; ++w) v += part[w][tile][lane];
    return v;
  };
  if constexpr (GLU) {
    TO *C = static_cast<TO *>(p.C) + batch * p.sC;
    for (int i = wave; i < TILES / 2; i += KW) {          // gate tile x, value tile x + 1
      const int x = 2 * (i / TM), y = i % TM;
      const f32x4 g = total(x * TM + y), v = total((x + 1) * TM + y);
      const int m = m0 + 16 * y + col, f = n0 / 2 + 8 * x + grp * 4;
      if (m >= p.M) continue;
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = siluf_(g[e]) * v[e];
      TO *dst = C + int64_t(m) * p.ldc + f;
      if (f + 4 <= p.glu_f) {
        Vec4<TO>::store(dst, o);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (f + e < p.glu_f) dst[e] = from_f32<TO>(o[e]);
      }
    }
  } else {
    for (int i = wave; i < TILES; i += KW) {
      const int x = i / TM, y = i % TM;
      const f32x4 t[1][1] = {{total(i)}};
      const int mw = m0 + 16 * y, nw = n0 + 16 * x;
      if constexpr (ATTN) {
        store_attn<1, 1>(p, t, mw, nw, col, grp);
      } else {
        store_any<sizeof(T) == 4, TO>(p, t, batch, mw, nw, col, grp);
      }
    }
  }
}

template <class G>
int launch_direct(const GemmArgs &p, int64_t batch, int out_dtype, bool glu, hipStream_t s, KernelTimer &timer) {
  const dim3 grid(unsigned(ceil_div(p.N, G::BN)), unsigned(ceil_div(p.M, G::BM)), unsigned(batch));
  const dim3 block(64 * G::KW);
  const bool b16 = out_dtype == XFH_BF16;
  if (glu) {
    if (b16) timer.launch(gemm_direct_kernel<bf16, bf16, true, G, false>, grid, block, 0, p);
    else timer.launch(gemm_direct_kernel<bf16, float, true, G, false>, grid, block, 0, p);
  } else if (p.attn.q) {
    if (!b16) return fail(XFH_EUNSUPPORTED, "gemm_direct: the attention layouts are bf16");
    timer.launch(gemm_direct_kernel<bf16, bf16, false, G, true>, grid, block, 0, p);
  } else {
    if (b16) timer.launch(gemm_direct_kernel<bf16, bf16, false, G, false>, grid, block, 0, p);
    else timer.launch(gemm_direct_kernel<bf16, float, false, G, false>, grid, block, 0, p);
  }
  return check_launch("gemm_direct");
}

template <class G> int launch_direct_f32(const GemmArgs &p, int64_t batch, bool glu, hipStream_t s, KernelTimer &timer) {
  const dim3 grid(unsigned(ceil_div(p.N, G::BN)), unsigned(ceil_div(p.M, G::BM)), unsigned(batch));
  const dim3 block(64 * G::KW);
  if (glu) timer.launch(gemm_direct_kernel<float, float, true, G, false>, grid, block, 0, p);
  else timer.launch(gemm_direct_kernel<float, float, false, G, false>, grid, block, 0, p);
  return check_launch("gemm_direct_f32");
}

}  // namespace
}  // namespace xfh
