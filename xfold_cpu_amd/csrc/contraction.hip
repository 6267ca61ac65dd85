// Per-channel triangle contraction: out[k][i][j] = sum_t L[k][i][t] * R[k][j][t]
// (bf16 operands, fp32 accumulation, bf16 result), the N x N x N product at the centre
// of xfold/nn/triangle_multiplication.py:96 for both directions (the operand layouts are
// prepared by trimul_project).
//
// Operands: L, R in the blocked operand layout (kernels.h): 16 rows x 32 t of one channel
// are one contiguous 1 KB block, ld = contraction_ld(n), zeros for t in [n, ld) so that the
// last k-step needs no bounds. The result goes to the blocked result layout: 16 pair
// positions' channels contiguous.
//
// Tiling: the output tile is picked by n (pick_tile): 192 x 384 to 64 x 64, one to four workgroups
// per CU, each wavefront owning 96 x 96, 64 x 64 or 32 x 32 (MFMA 16x16x32 tiles). Per k-step of 32
// both operand tiles go global -> LDS with global_load_lds_dwordx4 (no registers) into a ring
// of 3 or 4 slots, so the loads of the next 1 or 2
// steps are in flight while step s is multiplied; one barrier per step. Rows
// are 64 B in LDS with the 16-byte slots XOR-swizzled (slot c of row r holds chunk
// c ^ ((r >> 2) & 3)), so the 16 rows of an MFMA operand read hit distinct bank groups.
// The MFMA takes R rows as its A operand so that a lane ends up with four consecutive j
// of one i and writes them as one 8-byte store. Channels are numbered so that each XCD
// works through a contiguous run of tiles: the workgroups in flight on an XCD cover a few
// consecutive channels, whose k-slices share 128-byte lines and DRAM pages.
#include <algorithm>

#include "common.h"
#include "kernels.h"

namespace xfh {

namespace {

constexpr int TK = 32;                  // k-step
typedef __attribute__((address_space(1))) void global_void;
typedef __attribute__((address_space(3))) void lds_void;

template <int N> __device__ __forceinline__ void wait_vmcnt() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Waits until at most `younger` k-steps of this wavefront's loads (P each) are in flight.
template <int P, int MAXY> __device__ __forceinline__ void wait_younger(int younger) {
  if constexpr (MAXY == 0) {
    wait_vmcnt<0>();
  } else {
    if (younger >= MAXY) wait_vmcnt<MAXY * P>();
    else wait_younger<P, MAXY - 1>(younger);
  }
}

// TBI x TBJ output tiles (rows i of L, rows j of R) of WI x WJ wavefronts, each owning
// NI x NJ MFMA tiles; SLOTS ring stages, WGS workgroups per CU.
template <int NI_, int NJ_, int WI_, int WJ_, int SLOTS_, int WGS_> struct Tiling {
  static constexpr int NI = NI_, NJ = NJ_, WI = WI_, WJ = WJ_, W = WI_ * WJ_, SLOTS = SLOTS_, WGS = WGS_;
  static constexpr int TBI = 16 * NI * WI, TBJ = 16 * NJ * WJ;
  static constexpr int RBI = TBI / 16, RBJ = TBJ / 16;   // 16-row (1 KB) blocks per operand tile
  static constexpr int PIECES = RBI + RBJ;               // 1 KB direct loads per k-step
  static constexpr int PMAX = (PIECES + W - 1) / W;      // per wavefront (the first PIECES % W one more)
  static constexpr int SLOT_ELEMS = (TBI + TBJ) * TK;
  static_assert(SLOTS * SLOT_ELEMS * 2 * WGS <= 160 * 1024, "LDS budget");
  static_assert(NJ % 2 == 0, "R fragments are read in pairs");
};
using TileWide = Tiling<6, 6, 2, 4, 4, 1>;     // 192 x 384, one workgroup of 8 wavefronts per CU
using TileSquare = Tiling<6, 6, 2, 2, 3, 2>;   // 192 x 192, two of 4
using TileHalf = Tiling<4, 4, 2, 4, 3, 2>;     // 128 x 256, two of 8
using TileSmall = Tiling<2, 2, 2, 2, 4, 4>;    // 64 x 64, four of 4

template <class T>
__global__ __launch_bounds__(64 * T::W, T::WGS) void contraction_kernel(ContractionArgs a) {
  constexpr int TBI = T::TBI, TBJ = T::TBJ, WJ = T::WJ, W = T::W, SLOTS = T::SLOTS, NI = T::NI, NJ = T::NJ;
  constexpr int RBI = T::RBI, PIECES = T::PIECES, PMAX = T::PMAX, SLOT_ELEMS = T::SLOT_ELEMS;
  __shared__ __attribute__((aligned(16))) bf16 lds[SLOTS * SLOT_ELEMS];
  const int n = a.n, ld = a.ld;
  const int tiles_i = (n + TBI - 1) / TBI, tiles_j = (n + TBJ - 1) / TBJ;
  const int64_t per_channel = int64_t(tiles_i) * tiles_j;
  const int64_t total = per_channel * a.channels;
  const int64_t per_xcd = (total + 7) / 8;
  const int64_t logical = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
  if (logical >= total) return;
  const int64_t ch = logical / per_channel;
  const int tile = int(logical % per_channel);
  const int i0 = (tile / tiles_j) * TBI, j0 = (tile % tiles_j) * TBJ;

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wi = wave / WJ, wj = wave % WJ, col = lane & 15, grp = lane >> 4;
  // k-step s of row g of channel ch at op_offset(n, c, ch, g, 0) + s * step_stride.
  const int64_t step_stride = op_step_stride(n, a.channels);

  // Piece p of a k-step (wavefront w loads p = w, w + W, ...): L row block p (p < RBI) or R
  // row block p - RBI, 16 rows each (one 1 KB block); lane -> row 16 (block) + lane / 4, LDS
  // slot lane % 4 holding chunk (lane % 4) ^ ((lane >> 4) & 3). Rows beyond n read row n-1
  // (their results are never stored).
  const int chunk = (lane & 3) ^ ((lane >> 4) & 3);
  const bool full = wave < PIECES - (PMAX - 1) * W;  // this wavefront loads PMAX pieces
  const bf16 *src[PMAX];
#pragma unroll
  for (int j = 0; j < PMAX; ++j) {
    const int p = wave + W * j < PIECES ? wave + W * j : PIECES - 1;
    const bool lp = p < RBI;
    const int g = (lp ? i0 + p * 16 : j0 + (p - RBI) * 16) + (lane >> 2);
    src[j] = (lp ? a.left : a.right) + op_offset(n, a.channels, int(ch), g < n ? g : n - 1, 0) + chunk * 8;
  }
  auto issue = [&](int step, int slot) {
#pragma unroll
    for (int j = 0; j < PMAX; ++j) {
      const int p = wave + W * j;
      if (p >= PIECES) continue;
      bf16 *dst = lds + slot * SLOT_ELEMS + p * 16 * TK;   // L blocks, then R blocks
      __builtin_amdgcn_global_load_lds((global_void *)(src[j] + step * step_stride), (lds_void *)dst, 16, 0, 0);
    }
  };

  // Fragment offsets: row r of an operand tile, k-chunk grp, lives at r*TK + slot*8 with
  // slot = grp ^ ((r >> 2) & 3); for r = base + col with base a multiple of 16 that is
  // grp ^ ((col >> 2) & 3).
  const int frag = col * TK + ((grp ^ ((col >> 2) & 3)) * 8);

  f32x4 acc[NJ][NI];   // [jt][it]: rows j (A operand = R), cols i (B operand = L)
#pragma unroll
  for (int x = 0; x < NJ; ++x)
#pragma unroll
    for (int y = 0; y < NI; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int steps = ld / TK;
#pragma unroll
  for (int s = 0; s < SLOTS - 1; ++s)
    if (s < steps) issue(s, s);
  for (int s = 0; s < steps; ++s) {
    // This wavefront's loads of step s have landed (those of the younger steps, up to
    // SLOTS - 2 of them, may still fly), then every wavefront's have, and every wavefront
    // is done with step s-1.
    const int younger = steps - 1 - s < SLOTS - 2 ? steps - 1 - s : SLOTS - 2;
    if (full) wait_younger<PMAX, SLOTS - 2>(younger);
    else wait_younger<PMAX - 1, SLOTS - 2>(younger);
    ring_barrier();
    if (s + SLOTS - 1 < steps) issue(s + SLOTS - 1, (s + SLOTS - 1) % SLOTS);
    const bf16 *tl = lds + (s % SLOTS) * SLOT_ELEMS, *tr = tl + TBI * TK;
    // All L fragments and the first two R fragments, then each pair of R fragments is read
    // while the previous pair's MFMAs run (scheduling barriers keep the compiler from
    // sinking the reads next to their use).
    bf16x8 fl[NI], fr[NJ];
#pragma unroll
    for (int y = 0; y < NI; ++y)
      fl[y] = *reinterpret_cast<const bf16x8 *>(tl + (wi * NI + y) * 16 * TK + frag);
#pragma unroll
    for (int x = 0; x < 2; ++x) fr[x] = *reinterpret_cast<const bf16x8 *>(tr + (wj * NJ + x) * 16 * TK + frag);
#pragma unroll
    for (int xp = 0; xp < NJ / 2; ++xp) {
      __builtin_amdgcn_sched_barrier(0);
      if (xp + 1 < NJ / 2) {
#pragma unroll
        for (int x = 2 * xp + 2; x < 2 * xp + 4; ++x)
          fr[x] = *reinterpret_cast<const bf16x8 *>(tr + (wj * NJ + x) * 16 * TK + frag);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 2 * xp; x < 2 * xp + 2; ++x)
#pragma unroll
        for (int y = 0; y < NI; ++y) acc[x][y] = mfma16(fr[x], fl[y], acc[x][y]);
    }
  }

  // acc[x][y][e] = out[i = i0 + (wi NI + y) 16 + col][j = j0 + (wj NJ + x) 16 + 4 grp + e]. A row
  // of the result layout is a whole number of 16-position blocks, so the 4 positions of a
  // lane are one 8-byte store whatever n is; the columns of the last block from n on are
  // written too (finite, never read as results), the tile's columns beyond it are not.
  bf16 *out = a.out + ch * 16 + grp * 4;
  const int blocks = int(res_row_blocks(n));
#pragma unroll
  for (int y = 0; y < NI; ++y) {
    const int i = i0 + (wi * NI + y) * 16 + col;
    if (i >= n) continue;
#pragma unroll
    for (int x = 0; x < NJ; ++x) {
      const int jb = j0 / 16 + wj * NJ + x;
      if (jb >= blocks) continue;
      bf16x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = bf16(acc[x][y][e]);
      *reinterpret_cast<bf16x4 *>(out + (int64_t(i) * blocks + jb) * res_block_stride(a.channels)) = v;
    }
  }
}

template <class T> int launch(const ContractionArgs &a, hipStream_t s) {
  const int64_t total = ceil_div(a.n, T::TBI) * ceil_div(a.n, T::TBJ) * a.channels;
  const int64_t grid = ceil_div(total, 8) * 8;
  KernelTimer timer("trimul_contract", s, 2.0 * double(a.channels) * a.n * a.n * a.n, true);
  timer.launch(contraction_kernel<T>, dim3(grid), dim3(64 * T::W), 0, a);
  return check_launch("contraction");
}

// Tile of an n x n product: the one with the least (rounds of workgroups) x (time of a round's
// k-step). A last round that is partly empty counts half of what it leaves idle: its
// workgroups have less company for the L2. The k-step weights are measured (us; all tiles
// give the same bits): Wide 1.6; Square 1.44-1.6, above n = 1152 as fast as Wide or faster per
// round; Half 1.4-1.57 up to n = 768 and 1.75-1.9 above (half again the operand bytes per MFMA);
// Small 0.45 up to n = 384, 0.65-0.75 above. In us per launch, the tile taken against Wide up to n = 1024, Square above: n = 72
// 4.3 (Small) / 6.7, 128 5.4 (Small) / 9.4, 256 13.0 (Small) / 18.0, 420 42.5 (Half) / 75.0, 509 49.8 (Half)
// / 81.4, 576 81.8 (Square) / 89.9, 640 120.5 (Half) / 128.2, 900 307 (Square) / 331, 1100 470 (Wide) / 500; Wide
// stays at 384 and 768 (26.1, 155). A tile's time jumps where its edge divides n: on either side, Wide / Square /
// Half / Small, n = 383 26.3 / 29.8 / 33.5 / 33.8, 385 70.4 / 47.8 / 40.9 / 42.6, 767 153 / 160 / 196 / 325, 769 262 / 234 /
// 247 / 359, 1151 492 / 527 / 582 / 927, 1153 714 / 637 / 639 / 997: the pick is the fastest or within noise of it at
// each. It is 5% off at n = 700 (Wide 138, Square 132). With 64 channels, whose rounds are half as many, the
// same weights serve: right at 300, 385 to 600 and 769 up, 8-12% off Square at 352 (17.1 / 15.7), 383, 700 (68.4 / 61.1)
// and 767.
enum class Tile { Wide, Square, Half, Small };
template <class T> double tile_cost(int64_t n, int64_t channels, int cus, double step_us) {
  const int64_t wgs = ceil_div(n, T::TBI) * ceil_div(n, T::TBJ) * channels, slots = int64_t(cus) * T::WGS;
  return step_us * 0.5 * (double(ceil_div(wgs, slots)) + std::max(1.0, double(wgs) / double(slots)));
}
Tile pick_tile(int64_t n, int64_t channels, int cus) {
  const double cost[4] = {tile_cost<TileWide>(n, channels, cus, 1.6),
                          tile_cost<TileSquare>(n, channels, cus, n <= 1152 ? 1.62 : 1.5),
                          tile_cost<TileHalf>(n, channels, cus, n <= 768 ? 1.45 : 1.85),
                          tile_cost<TileSmall>(n, channels, cus, n <= 384 ? 0.45 : 0.75)};
  int best = 0;
  for (int t = 1; t < 4; ++t)
    if (cost[t] < cost[best]) best = t;
  return Tile(best);
}

}  // namespace

int64_t contraction_ld(int64_t n) { return align_up(n, TK); }
int64_t contraction_operand_elems(int64_t n, int64_t channels) {
  return (contraction_ld(n) / TK) * op_step_stride(n, int(channels));
}
int64_t contraction_result_elems(int64_t n, int64_t channels) {
  return n * res_row_blocks(n) * res_block_stride(int(channels));
}

int contraction(const ContractionArgs &a, hipStream_t s) {
  if (a.n == 0 || a.channels == 0) return XFH_OK;
  if (a.ld != contraction_ld(a.n)) return fail(XFH_EINVAL, "contraction: operand rows must be padded to 32");
  int cus = 0;
  XFH_TRY(device_cu_count(&cus));
  switch (pick_tile(a.n, a.channels, cus)) {
    case Tile::Wide: return launch<TileWide>(a, s);
    case Tile::Square: return launch<TileSquare>(a, s);
    case Tile::Half: return launch<TileHalf>(a, s);
    default: return launch<TileSmall>(a, s);
  }
}

}  // namespace xfh
