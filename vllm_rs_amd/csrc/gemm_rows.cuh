// gemm_rows.cuh — 16-bit GEMM of prompt steps on ROW-MAJOR weights: out[m, n] = epilogue( sum_k x[row(m), k] * w[n, k] ), f32 accumulation.
//
// Bound: what a CU can pull past L2, and how well that overlaps with the matrix work.  LDS-DMA alone (no LDS reads, no MFMAs) delivers ~28 B
// per clock and CU on full 128-byte lines and ~21 on half lines where the panels come from past L2, whatever the depth of the ring or the row
// stride (panels that stay in L2: 58..60, on either); a 128 x 128 tile needs 32 KiB per 512 clocks of MFMAs.  So: whole lines per request
// (a DMA instruction fetches 8 rows x 128 bytes), the largest tiles the problem has enough of, and the DMA instructions spread between the MFMAs —
// issued in one run they stall the wave in front of its LDS reads.  Measured (2048 x 2048 outputs, K = 8192, 256 tiles of 128 x 128): 87 us
// with the requests in one run, 74 spread; without the MFMAs 67, and 47 with the weights in L2: requests and MFMAs do not overlap as well as they could.
//
// Tile: WM x WN waves, 64 x 64 outputs each (16 accumulator tiles of v_mfma_f32_16x16x32: weights = A, rows of x = B, so a lane holds 4
// consecutive columns of one row).  K in steps of 64, ascending, one accumulation chain per output: the result of a row does not depend
// on the tile, the row's place in it or the rows beside it, and is bit-equal to any other kernel that walks K in steps of 32 on this
// instruction.
// LDS ring of S stages; a stage holds 4 (WM + WN) blocks of 16 rows x 64 k (2 KiB): row r of a block at r * 128 bytes, its 16-byte chunk c in
// slot c ^ (r & 7), which spreads a fragment read's lanes over all banks.  At the top of step ks the stages ks and ks + 1 have landed
// and the first half of ks is in registers; the step reads its second half, runs the first half's MFMAs, reads the first half of ks + 1,
// runs the second half's, requests stage ks + S - 1 into the buffer of ks - 1 (every wave is past its reads: the barrier at the end of
// ks - 1) and waits until stage ks + 2 is complete before the barrier.
#pragma once
#include "common.cuh"

#define GR_MAX_SEG 3

struct GemmRowsArgs {
  const void* x = nullptr;  // [rows, x_ld]
  int x_ld = 0;
  const int* x_row = nullptr;  // row of x for output row m (-1: no row, nothing is stored); null: m
  const void* w[GR_MAX_SEG] = {};  // [n[s], K] each: the segments of one launch (q | k | v), or gate and up of a pair (PAIR)
  int n[GR_MAX_SEG] = {};
  int nseg = 1;
  int M = 0, K = 0;  // K % 64 == 0
  int MT = 0, NT = 0;  // tiles along m, and along n over all segments
  // grouped rows: tile row t (BM rows) multiplies with w[0] + tile_group[t] * w_group_stride (elements); -1: an empty tile row
  const int* tile_group = nullptr;
  int64_t w_group_stride = 0;
  int64_t x_batch_stride = 0, w_batch_stride = 0;  // elements between the operands of two products of a batch (grid y)
};

// a row's 4 x 4 columns of four accumulator tiles, held by the lanes r16, r16 + 16, r16 + 32, r16 + 48 -> lane q holds tile q's 16 columns
// (register pair c = columns 4 c .. 4 c + 3 of that tile)
__device__ __forceinline__ void gr_gather_columns(u32x2 (&v)[4]) {
#pragma unroll
  for (int e = 0; e < 2; e++) {
    auto a = __builtin_amdgcn_permlane32_swap(v[0][e], v[2][e], false, false);
    auto b = __builtin_amdgcn_permlane32_swap(v[1][e], v[3][e], false, false);
    auto c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
    auto d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
    v[0][e] = c[0], v[1][e] = c[1], v[2][e] = d[0], v[3][e] = d[1];
  }
}
// the same for two tiles (32 columns of a row): lane q holds columns 8 q .. 8 q + 7
__device__ __forceinline__ void gr_gather_columns(u32x2 (&v)[2]) {
#pragma unroll
  for (int e = 0; e < 2; e++) {
    auto a = __builtin_amdgcn_permlane32_swap(v[0][e], v[1][e], false, false);
    auto c = __builtin_amdgcn_permlane16_swap(a[0], a[1], false, false);
    v[0][e] = c[0], v[1][e] = c[1];
  }
}

static inline size_t gemm_rows_lds_bytes(int wm, int wn, int s) { return (size_t)s * 4 * (wm + wn) * 2048; }

// EPI::store(m, seg, n0, q4, acc): the wave's 64 columns n0 .. n0 + 63 (of segment seg) of output row m; the lane holds columns n0 + 16 j + 4 q4 ..
// + 3 in acc[j].  Called by all lanes (lanes beyond the matrix with m = -1), so that a lane may trade columns with its row's other three.
// PAIR: w[0] and w[1] (gate, up; neither grouped nor batched) interleaved in blocks of 16 virtual columns, n[0] = virtual columns.
template <class DT, int WM, int WN, int S, bool SPREAD, bool PAIR, class EPI>
__global__ __launch_bounds__(64 * WM * WN + (SPREAD ? 0 : 64)) void gemm_rows_kernel(const GemmRowsArgs a, const EPI epi) {
#ifdef __HIP_DEVICE_COMPILE__
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int NW = WM * WN, XB = 4 * WM, NB = 4 * (WM + WN), PER = NB / NW, D = 2 * PER, STG = NB * 2048, PEND = (S - 3) * D;
  static_assert(NB % NW == 0 && XB % NW == 0 && S >= 3 && (!PAIR || NW % 2 == 0), "block split");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM, r16 = lane & 15, q4 = lane >> 4;
  // tile: the ids of one XCD (id mod 8) take a contiguous run of an order that walks 8 tile rows before the next tile column, so the
  // workgroups of an XCD share their operands' panels in its L2
  int mt, nt;
  {
    const int nwg = (int)gridDim.x, bid = (int)blockIdx.x, q = nwg >> 3, r = nwg & 7, xcd = bid & 7;
    const int lin = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (bid >> 3);
    constexpr int GM = 8;
    const int per = GM * a.NT, grp = lin / per, rem = lin - grp * per, first = grp * GM, gsz = min(a.MT - first, GM);
    mt = first + rem % gsz;
    nt = rem / gsz;
  }
  int group = 0;
  if (a.tile_group) {
    group = __builtin_amdgcn_readfirstlane(a.tile_group[mt]);
    if (group < 0) return;
  }
  // segment of the tile column (whole tiles per segment)
  int seg = 0, N = a.n[0];
  const uint16_t* w = static_cast<const uint16_t*>(a.w[0]);
  if (!PAIR) {
    if (a.nseg > 1 && nt >= (N + 64 * WN - 1) / (64 * WN)) nt -= (N + 64 * WN - 1) / (64 * WN), seg = 1, N = a.n[1], w = static_cast<const uint16_t*>(a.w[1]);
    if (seg == 1 && a.nseg > 2 && nt >= (N + 64 * WN - 1) / (64 * WN)) nt -= (N + 64 * WN - 1) / (64 * WN), seg = 2, N = a.n[2], w = static_cast<const uint16_t*>(a.w[2]);
  } else if (wave & 1) {
    w = static_cast<const uint16_t*>(a.w[1]);  // (virtual block f: tensor f & 1; a wave requests the blocks wave + i * NW, all of one parity)
  }
  const int m0 = mt * 64 * WM, n0 = nt * 64 * WN, K = a.K, KT = K >> 6;
  const uint16_t* const x = static_cast<const uint16_t*>(a.x) + (int64_t)blockIdx.y * a.x_batch_stride;
  w += (int64_t)group * a.w_group_stride + (int64_t)blockIdx.y * a.w_batch_stride;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, 0x7FFFFFF0, 0x00020000u);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w), 0, 0x7FFFFFF0, 0x00020000u);
  // DMA sources: lane p fetches row p >> 3 (and 8 + (p >> 3) with the second instruction of a block), the chunk that slot p & 7 holds
  uint32_t vo[PER][2];
  {
    const int sr = lane >> 3, sc = (lane & 7) ^ (lane >> 3);
#pragma unroll
    for (int i = 0; i < PER; i++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int b = wave + i * NW;
        int row;
        uint32_t ld;
        if (i * NW < XB) {
          row = min(m0 + b * 16 + h * 8 + sr, a.M - 1);
          if (a.x_row) row = max(a.x_row[row], 0);
          ld = (uint32_t)a.x_ld;
        } else if (PAIR) {
          row = min(((n0 >> 4) + b - XB) / 2 * 16 + h * 8 + sr, (N >> 1) - 1);
          ld = (uint32_t)K;
        } else {
          row = min(n0 + (b - XB) * 16 + h * 8 + sr, N - 1);
          ld = (uint32_t)K;
        }
        vo[i][h] = ((uint32_t)row * ld + (uint32_t)sc * 8u) * 2u;
      }
  }
  if constexpr (!SPREAD) {
    // One wave more, which computes nothing: it touches a line of K step ks + 8 for its share of the panels that the workgroups of an XCD
    // have in common (8 tile rows x 4 tile columns at a time: a quarter of this tile's rows of x, an eighth of its columns of w), so that
    // the ring's requests find them in L2.  With two stages in flight the ring alone does not cover the way to memory (2048 x 8192, K =
    // 2048, weights not in any cache: 94 -> 82 us); the 128 x 128 tile's three stages do, and gain nothing.
    if (wave == NW) {
      constexpr int XL = 16 * WM, WL = 8 * WN;
      static_assert(XL + WL <= 64, "a lane a line");
      const bool isx = lane < XL;
      const int xr = min(m0 + (nt & 3) * XL + lane, a.M - 1), wrow = (mt & 7) * WL + (lane - XL);
      int nr = min(n0 + wrow, N - 1);
      const uint16_t* wp = w;
      if (PAIR) {  // (this wave's w is the gate tensor's)
        const uint16_t* const up = static_cast<const uint16_t*>(a.w[1]);
        nr = min((n0 >> 1) + (wrow >> 1), (N >> 1) - 1);
        if (wrow & 1) wp = up;
      }
      const int xi = isx && a.x_row ? max(a.x_row[xr], 0) : xr;
      const uint16_t* const p = isx ? x + (int64_t)xi * a.x_ld : wp + (int64_t)nr * K;
      const bool live = lane < XL + WL;
      uint32_t v[8] = {}, seen = 0;
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (live) v[u] = *reinterpret_cast<const uint32_t*>(p + min(u, KT - 1) * 64);
      __builtin_amdgcn_s_barrier();
      for (int ks = 0; ks < KT; ks += 8) {
#pragma unroll
        for (int u = 0; u < 8; u++) {
          if (ks + u >= KT) break;  // (one barrier a step, as the other waves)
          seen ^= v[u];
          if (live) v[u] = *reinterpret_cast<const uint32_t*>(p + min(ks + u + 8, KT - 1) * 64);
          __builtin_amdgcn_sched_barrier(0);
          __builtin_amdgcn_s_barrier();
        }
      }
#pragma unroll
      for (int u = 0; u < 8; u++) seen ^= v[u];
      asm volatile("" ::"v"(seen));
      return;
    }
  }
  typedef __attribute__((address_space(3))) void* lds_ptr;
  auto request = [&](int ks, int e) {  // the e-th of the wave's D instructions for stage ks (beyond K: the last step again, never read)
    const uint32_t so = (uint32_t)min(ks, KT - 1) * 128u;
    const int i = e >> 1, h = e & 1;
    unsigned char* const d = smem + (ks % S) * STG + (wave + i * NW) * 2048 + h * 1024;
    if (i * NW < XB) __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr)d, 16, vo[i][h], so, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr)d, 16, vo[i][h], so, 0, 0);
  };
  const int c0 = r16 * 128 + (q4 ^ (r16 & 7)) * 16, c1 = r16 * 128 + ((4 + q4) ^ (r16 & 7)) * 16;
  const unsigned char* const xb = smem + wm * 4 * 2048;
  const unsigned char* const wb = smem + (XB + wn * 4) * 2048;
  s16x8 xa[2][4], wa[2][4];
  auto read = [&](int half, int ks) {  // k half `half` of step ks
    const int o = (ks % S) * STG + (half ? c1 : c0);
#pragma unroll
    for (int j = 0; j < 4; j++) wa[half][j] = *reinterpret_cast<const s16x8*>(wb + o + j * 2048);
#pragma unroll
    for (int i = 0; i < 4; i++) xa[half][i] = *reinterpret_cast<const s16x8*>(xb + o + i * 2048);
  };
  f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = vra_zero_acc();
  auto mma = [&](int half, int ks) {  // 16 MFMAs, with the instructions of that half of stage ks + S - 1 between them
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if constexpr (SPREAD) {
#pragma unroll
        for (int e = half * PER + PER * i / 4; e < half * PER + PER * (i + 1) / 4; e++) request(ks + S - 1, e);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; j++) DT::mfma(acc[i][j], wa[half][j], xa[half][i]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int s = 0; s < S - 1; s++)
#pragma unroll
    for (int e = 0; e < D; e++) request(s, e);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PEND) : "memory");
  __builtin_amdgcn_s_barrier();
  read(0, 0);
  for (int ks = 0; ks < KT; ks++) {
    if constexpr (!SPREAD) {
#pragma unroll
      for (int e = 0; e < D; e++) request(ks + S - 1, e);
    }
    read(1, ks);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    mma(0, ks);
    read(0, ks + 1);
    __builtin_amdgcn_sched_barrier(0);
    mma(1, ks);
    __builtin_amdgcn_s_setprio(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PEND) : "memory");
    __builtin_amdgcn_s_barrier();
  }
  // (the requests beyond K still write LDS: they end before the workgroup does)
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  VRA_MFMA_DRAIN();
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int m = m0 + wm * 64 + i * 16 + r16;
    if (m >= a.M || (a.x_row && a.x_row[m] < 0)) m = -1;
    epi.store(m, seg, n0 + wn * 64, N, q4, acc[i]);
  }
#endif
}

// Tile for a product of M rows x ncols[0..nseg) columns x `batch`: workgroups run in rounds of one per CU, a round of a tile takes (us per 64
// of K, measured with all CUs at work) 0.55 at 64 x 128, 0.62 at 128 x 128, 1.10 at 128 x 256.  -> WM * 16 + WN; *us: the time per 64 of K
static inline int gemm_rows_tile(long M, const int* ncols, int nseg, long batch, double* us = nullptr) {
  const struct { int wm, wn; double us; } t[3] = {{2, 4, 1.10}, {2, 2, 0.62}, {1, 2, 0.55}};
  int best = 0;
  double cost = 0.0;
  for (const auto& c : t) {
    long cols = 0;
    for (int s = 0; s < nseg; s++) cols += (ncols[s] + 64 * c.wn - 1) / (64 * c.wn);
    const long tiles = (M + 64 * c.wm - 1) / (64 * c.wm) * cols * batch;
    const double v = (double)((tiles + 255) / 256) * c.us;
    if (!best || v < cost) best = c.wm * 16 + c.wn, cost = v;
  }
  if (us) *us = cost;
  return best;
}
static inline bool gemm_rows_has_tile(int tile) { return tile == 2 * 16 + 4 || tile == 2 * 16 + 2 || tile == 16 + 2; }
// fills the tile counts and launches
template <class DT, int WM, int WN, int S, bool SPREAD, bool PAIR, class EPI>
static void gemm_rows_launch_t(GemmRowsArgs a, const EPI& epi, int batch, hipStream_t st) {
  a.MT = (a.M + 64 * WM - 1) / (64 * WM);
  a.NT = 0;
  for (int s = 0; s < a.nseg; s++) a.NT += (a.n[s] + 64 * WN - 1) / (64 * WN);
  static uint64_t attr_devs = 0;  // function attributes belong to the device current at the call
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (!((attr_devs >> (dev & 63)) & 1)) {
    void (*const k)(GemmRowsArgs, EPI) = gemm_rows_kernel<DT, WM, WN, S, SPREAD, PAIR, EPI>;
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr_devs |= (uint64_t)1 << (dev & 63);
  }
  gemm_rows_kernel<DT, WM, WN, S, SPREAD, PAIR, EPI>
      <<<dim3((unsigned)(a.MT * a.NT), (unsigned)batch), dim3(64 * WM * WN + (SPREAD ? 0 : 64)), gemm_rows_lds_bytes(WM, WN, S), st>>>(a, epi);
}
template <class DT, bool PAIR, class EPI>
static void gemm_rows_launch(const GemmRowsArgs& a, const EPI& epi, int tile, int batch, hipStream_t st) {
  if (tile == 2 * 16 + 4) gemm_rows_launch_t<DT, 2, 4, 3, false, PAIR>(a, epi, batch, st);
  else if (tile == 2 * 16 + 2) gemm_rows_launch_t<DT, 2, 2, 4, true, PAIR>(a, epi, batch, st);
  else gemm_rows_launch_t<DT, 1, 2, 4, true, PAIR>(a, epi, batch, st);
}
