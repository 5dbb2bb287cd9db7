// gemm_rows.cuh — 16-bit GEMM of prompt steps on ROW-MAJOR weights: out[m, n] = epilogue( sum_k x[row(m), k] * w[n, k] ), f32 accumulation.
//
// Bound: 256 x 256 outputs a workgroup, the chip's power — the loop runs 2240 clocks a K step of 64 (its MFMAs are 2048), at a clock that
// settles at 1.3..1.5 GHz (matrix instructions alone: 1.9); smaller tiles, what a CU gets past L2: 28..35 B per clock where lines come from
// memory, whatever the number of buffers, the cache policy or a wave that touches lines ahead (requests in flight a CU are limited, and
// a line that another CU has asked for costs as long).  A 128 x 128 tile needs 32 KiB per 512 clocks of MFMAs, 256 x 256 64 KiB per 2048.
//
// Two groups of four waves (a wave of each on every SIMD) run one barrier apart: while one group's MFMAs run, the other reads its operands of the
// next phase from LDS and requests tiles.  A phase is a K step of 64 — with 256 x 256 and 192 x 256 outputs two of them a step, the upper and the lower rows of every wave —
//   { LDS reads | requests | vmcnt: the next phase's tiles have landed, lgkmcnt: this phase's reads are done | barrier | MFMAs | barrier }
// and requests go to the buffer that the phase before read: both groups' reads ended ahead of a barrier that the requesting wave has passed.
// Fragments come from LDS only, so the MFMAs need no wait states between them (10 % of a group's phase).  Against one group in step with itself
// (128 x 256: 8 waves and one touching lines; 128 x 128: 4 waves), us: 2048 x 8192, K = 2048: 84 -> 63 (256 x 256; 128 x 256 78); 2048 x 2048 x 2048
// 25.5 -> 23.5 (128 x 128); 2048 x 2048, K = 8192: 82 -> 76; 2120 rows x 2048, K = 2048 / 5632: 35.9 -> 30.7 / 84.5 -> 78.6 (128 x 256).
//
// Weights = A, rows of x = B of v_mfma_f32_16x16x32, so a lane holds 4 consecutive columns of one row.  K ascending, one accumulation chain per
// output: the result of a row does not depend on the tile, the row's place in it or the rows beside it, and is bit-equal to any other kernel
// that walks K in steps of 32 on this instruction.
// LDS: blocks of 16 rows x 64 k (2 KiB): row r of a block at r * 128 bytes, its 16-byte chunk c in slot c ^ (r & 7), which spreads a fragment
// read's lanes over all banks; a request (LDS-DMA) fetches 8 rows x 128 bytes, whole lines.
#pragma once
#include <algorithm>
#include <type_traits>

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
  int chunk = 0;  // grouped rows: tile columns of a unit (gemm_rows_launch_t)
  int mixed = 0;  // gemm_rows_mixed_kernel: tile columns of 256 x 256
  // grouped rows (on tiles of 64 and 128 rows): tile row t (BM rows) multiplies with w[0] + tile_group[t] * w_group_stride (elements); -1: an empty tile row
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

// waves of a tile: two groups of four (rows 0 .. BM/2 - 1 and the others), CW of them side by side with 64 columns each
template <int BM, int BN, bool DEEP>
struct GrTile {
  static constexpr int H = BM * BN > 128 * 256 ? 2 : 1;                 // phases of a K step (the upper, the lower rows of a wave)
  static constexpr int KP = DEEP ? 2 : 1;                                     // K steps of a phase
  static constexpr int S = H == 2 ? 2 : (BM == 128 && BN == 128 ? 4 : 3);  // LDS buffers (of a phase's K steps)
  static constexpr int CW = BN / 64, RW = 4 / CW;
  static constexpr int NX = BM / 32 / RW / H;  // 16-row blocks of a wave in a phase
  static constexpr int XB = BM / 16, WB = BN / 16, STG = (XB + WB) * 2048;
  static constexpr int EX = BM / 64, EW = BN / 64;  // a wave's DMA instructions (8 rows of 128 bytes) a K step
};

// place of workgroup bid of nwg in an order whose contiguous runs go to one XCD (ids mod 8) each, and a place's tile of MT x NT: about 8 tile rows, in equal
// groups, before the next tile column
__device__ __forceinline__ int gr_xcd_run(int bid, int nwg) {
  const int q = nwg >> 3, r = nwg & 7, xcd = bid & 7;
  return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (bid >> 3);
}
__device__ __forceinline__ void gr_tile_of(int lin, int MT, int NT, int& mt, int& nt) {
  const int groups = max((MT + 4) >> 3, 1), GM = (MT + groups - 1) / groups;
  const int per = GM * NT, grp = lin / per, rem = lin - grp * per, first = grp * GM, gsz = min(MT - first, GM);
  mt = first + rem % gsz;
  nt = rem / gsz;
}

// EPI::in_form(n0, N, q4, f): f(form, columns): a constant that store takes as its template argument, and what it reads of the lane's columns: what is the same for
// all rows is decided and loaded once.
// EPI::store(m, row, columns, seg, n0, N, q4, acc): the wave's 64 columns n0 .. n0 + 63 (of segment seg) of output row m; the lane holds columns n0 + 16 j + 4 q4 ..
// + 3 in acc[j].  Called by all lanes (lanes beyond the matrix with m = -1), so that a lane may trade columns with its row's other three.
// row: EPI::row(m), taken ahead of the loop (rows beyond the matrix: of its last).
// PAIR: w[0] and w[1] (gate, up; neither grouped nor batched) interleaved in blocks of 16 virtual columns, n[0] = virtual columns.
// tile (mt, nt) of segment seg (w, N columns)
template <class DT, int BM, int BN, bool DEEP, bool PAIR, class EPI>
__device__ __forceinline__ void gemm_rows_tile_product(const GemmRowsArgs& a, const EPI& epi, int mt, int nt, int seg, int N, const uint16_t* w, int group) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  using T = GrTile<BM, BN, DEEP>;
  constexpr int H = T::H, KP = T::KP, S = T::S, NX = T::NX, STG = T::STG, EX = T::EX, EW = T::EW, D = EX + EW;
  static_assert(EW == 4 || EW == 2, "a wave has 64 columns");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wg = wave >> 2, cw = (wave & 3) % T::CW, rw = (wave & 3) / T::CW, r16 = lane & 15, q4 = lane >> 4;
  const int m0 = mt * BM, n0 = nt * BN, K = a.K, KT = K >> 6;
  const uint16_t* const x = static_cast<const uint16_t*>(a.x) + (int64_t)blockIdx.y * a.x_batch_stride;
  w += (int64_t)group * a.w_group_stride + (int64_t)blockIdx.y * a.w_batch_stride;
  // (PAIR: virtual block f is of tensor f & 1.  A wave requests the blocks 2 wave and 2 wave + 1 of a 256-column tile, block wave of a 128-column one)
  const uint16_t* const wlo = PAIR && EW == 2 && (wave & 1) ? static_cast<const uint16_t*>(a.w[1]) : w;
  const uint16_t* const whi = PAIR && EW == 4 ? static_cast<const uint16_t*>(a.w[1]) : wlo;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, 0x7FFFFFF0, 0x00020000u);
  const __amdgpu_buffer_rsrc_t rlo = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(wlo), 0, 0x7FFFFFF0, 0x00020000u);
  const __amdgpu_buffer_rsrc_t rhi = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(whi), 0, 0x7FFFFFF0, 0x00020000u);
  // DMA sources: lane p fetches row p >> 3 of an instruction's eight, the chunk that slot p & 7 holds
  const int sr = lane >> 3, sc = (lane & 7) ^ sr;
  // instruction e of this wave: eight rows from this one on.  Two phases, of 256 rows: e = 0, 1 upper, 2, 3 lower rows of a group; of 192 rows, a group's
  // upper and lower 48: waves 0-3 two of the upper rows' instructions and one of the lower ones', waves 4-7 the other way about
  auto upper = [&](int e) { return EX == 4 ? e < 2 : e == 0 || (e == 1 && wave < 4); };
  auto xrow8 = [&](int e) {
    if (H == 1) return (wave * EX + e) * 8;
    if (EX == 4) return (wave < 4 ? wave : wave + 4) * 16 + (e >> 1) * 64 + (e & 1) * 8;
    const int i = wave < 4 ? (upper(e) ? wave * 2 + e : 8 + wave) : (upper(e) ? 4 + wave : (wave - 4) * 2 + e - 1);  // of the twelve of its half
    return i / 6 * 96 + i % 6 * 8 + (upper(e) ? 0 : 48);
  };
  uint32_t vx[EX], vw[EW];
#pragma unroll
  for (int e = 0; e < EX; e++) {
    int row = min(m0 + xrow8(e) + sr, a.M - 1);
    if (a.x_row) row = max(a.x_row[row], 0);
    vx[e] = ((uint32_t)row * (uint32_t)a.x_ld + (uint32_t)sc * 8u) * 2u;
  }
#pragma unroll
  for (int e = 0; e < EW; e++) {
    const int r8 = (wave * EW + e) * 8;  // (of a pair: block r8 / 16, half of the virtual columns' row in its tensor)
    const int row = PAIR ? min((((n0 + r8) >> 4) >> 1) * 16 + (r8 & 15) + sr, (N >> 1) - 1) : min(n0 + r8 + sr, N - 1);
    vw[e] = ((uint32_t)row * (uint32_t)K + (uint32_t)sc * 8u) * 2u;
  }
  typedef __attribute__((address_space(3))) void* lds_ptr;
  // requests of K step ks (beyond K: the last step again, never read) into the buffer at byte `o`
  auto stage_x = [&](int o, int ks, int e0, int e1) {
    const uint32_t so = (uint32_t)min(ks, KT - 1) * 128u;
#pragma unroll
    for (int e = e0; e < e1; e++) __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr)(smem + o + xrow8(e) * 128), 16, vx[e], so, 0, 0);
  };
  auto stage_half = [&](int o, int ks, bool up) {  // the upper or the lower rows
#pragma unroll
    for (int e = 0; e < EX; e++)
      if (upper(e) == up) stage_x(o, ks, e, e + 1);
  };
  auto stage_w = [&](int o, int ks) {
    const uint32_t so = (uint32_t)min(ks, KT - 1) * 128u;
#pragma unroll
    for (int e = 0; e < EW; e++) {
      unsigned char* const d = smem + o + T::XB * 2048 + (wave * EW + e) * 1024;
      if (e < EW / 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(rlo, (lds_ptr)d, 16, vw[e], so, 0, 0);
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(rhi, (lds_ptr)d, 16, vw[e], so, 0, 0);
    }
  };
  const int row0 = wg * (BM / 2) + rw * (BM / 2 / T::RW);  // the wave's first row in the tile
  const int c0 = r16 * 128 + (q4 ^ (r16 & 7)) * 16, c1 = c0 ^ 64;
  const unsigned char* const xb = smem + row0 * 128;
  const unsigned char* const wb = smem + T::XB * 2048 + cw * 4 * 2048;
  s16x8 xa[KP * NX][2], wa[KP * 4][2];
  auto read_x = [&](int o, int h, int k = 0) {
#pragma unroll
    for (int i = 0; i < NX; i++) {
      xa[k * NX + i][0] = *reinterpret_cast<const s16x8*>(xb + o + c0 + (h * NX + i) * 2048);
      xa[k * NX + i][1] = *reinterpret_cast<const s16x8*>(xb + o + c1 + (h * NX + i) * 2048);
    }
  };
  auto read_w = [&](int o, int k = 0) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      wa[k * 4 + j][0] = *reinterpret_cast<const s16x8*>(wb + o + c0 + j * 2048);
      wa[k * 4 + j][1] = *reinterpret_cast<const s16x8*>(wb + o + c1 + j * 2048);
    }
  };
  f32x4 acc[H * NX][4];
  typename EPI::Row erow[H * NX];  // what the epilogue reads of its rows: asked for ahead of the loop, whose first requests come behind it
#pragma unroll
  for (int i = 0; i < H * NX; i++) {
    erow[i] = epi.row(min(m0 + row0 + i * 16 + r16, a.M - 1));
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = vra_zero_acc();
  }
  // (a wave's 64 columns, a phase's rows: nothing of them in the matrix, no MFMAs)
  const bool in = n0 + cw * 64 < N && m0 + row0 < a.M, in1 = H == 2 && n0 + cw * 64 < N && m0 + row0 + NX * 16 < a.M;
  auto compute = [&](auto HH, int steps) {  // steps: of the phase's KP those that are within K
    constexpr int h = decltype(HH)::value;
    // the next phase's requests have landed (those of the last S - 2 steps, with two phases of the last step, may be on their way), this phase's reads are done
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(H == 2 ? D : (S - 2) * KP * D) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (h ? in1 : in) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int k = 0; k < KP; k++) {
        if (k && k >= steps) break;
#pragma unroll
        for (int kc = 0; kc < 2; kc++)
#pragma unroll
          for (int i = 0; i < NX; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) DT::mfma_ready(acc[h * NX + i][j], wa[k * 4 + j][kc], xa[k * NX + i][kc]);
      }
      __builtin_amdgcn_s_setprio(0);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
  };
  // The compiler asks for the epilogue's arguments ahead of the loop.  A scalar load on its way into it turns the loop's counted waits for LDS reads into waits for all of
  // them (the two kinds of load share a counter and return out of order): 2048 x 8192, K = 2048, f32 results 62.3 us without one, 64.4 with.  So they land first.
  auto no_scalar_loads = [] {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  if constexpr (H == 2) {
    stage_half(0, 0, true);
    stage_w(0, 0);
    stage_half(0, 0, false);
    stage_half(STG, 1, true);
    stage_w(STG, 1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(D) : "memory");
    __builtin_amdgcn_s_barrier();
    if (wg == 1) __builtin_amdgcn_s_barrier();  // the second group runs one barrier behind the first
    auto step = [&](auto B, int ks) {
      constexpr int o = decltype(B)::value * STG;
      read_w(o);
      __builtin_amdgcn_sched_barrier(0);
      read_x(o, 0);
      stage_half(STG - o, ks + 1, false);
      compute(C0{}, 1);
      read_x(o, 1);
      stage_half(o, ks + 2, true);
      stage_w(o, ks + 2);
      compute(C1{}, 1);
    };
    no_scalar_loads();
    for (int ks = 0; ks < KT; ks += 2) {
      step(C0{}, ks);
      step(C1{}, ks + 1);
    }
  } else {
#pragma unroll
    for (int s = 0; s < (S - 1) * KP; s++) stage_x(s * STG, s, 0, EX), stage_w(s * STG, s);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * KP * D) : "memory");
    __builtin_amdgcn_s_barrier();
    if (wg == 1) __builtin_amdgcn_s_barrier();
    no_scalar_loads();
    int o = 0, p = (S - 1) * KP * STG;  // buffers of this phase and of the one before it
    for (int ks = 0; ks < KT; ks += KP) {
#pragma unroll
      for (int k = 0; k < KP; k++) read_w(o + k * STG, k), read_x(o + k * STG, 0, k);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < KP; k++) {
        stage_x(p + k * STG, ks + (S - 1) * KP + k, 0, EX);
        stage_w(p + k * STG, ks + (S - 1) * KP + k);
      }
      compute(C0{}, KT - ks);
      p = o;
      o = o == (S - 1) * KP * STG ? 0 : o + KP * STG;
    }
  }
  if (wg == 0) __builtin_amdgcn_s_barrier();
  // (the requests beyond K still write LDS: they end before the workgroup does)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  VRA_MFMA_DRAIN();
  epi.in_form(n0 + cw * 64, N, q4, [&](auto F, const auto& columns) {
#pragma unroll
    for (int i = 0; i < H * NX; i++) {
      int m = m0 + row0 + i * 16 + r16;
      if (m >= a.M || (a.x_row && a.x_row[m] < 0)) m = -1;
      epi.template store<decltype(F)::value>(m, erow[i], columns, seg, n0 + cw * 64, N, q4, acc[i]);
    }
  });
}

template <class DT, int BM, int BN, bool DEEP, bool PAIR, class EPI>
__global__ __launch_bounds__(512, 2) void gemm_rows_kernel(const GemmRowsArgs a, const EPI epi) {
#ifdef __HIP_DEVICE_COMPILE__
  // tile: the ids of one XCD (id mod 8) take a contiguous run of an order that walks about 8 tile rows before the next tile column, so the
  // workgroups of an XCD share their operands' panels in its L2; the tile rows in equal groups (the weights come by once a group: with 8 + 1 tile
  // rows of 64, 557 rows x 14336, K = 4096 99 us, with 9 77.5).  Grouped rows: the empty tile rows are the last ones, so the XCDs take units of two tile
  // rows (an expert's, more often than not) in turn, two rows to a column (16 experts of 188 rows, 2048 columns, 40 tile rows with 8 empty
  // ones: in runs two XCDs idle and the others work two rounds, K = 2048 / 1024 77.7 / 45.9 us; so 50.8 / 27.0)
  int mt, nt, group = 0;
  if (GrTile<BM, BN, DEEP>::H == 1 && a.tile_group) {
    const int size = 2 * a.chunk, i = (int)blockIdx.x >> 3, unit = ((int)blockIdx.x & 7) + 8 * (i / size), rem = i % size;
    const int per = (a.NT + a.chunk - 1) / a.chunk;  // units of a pair of tile rows
    mt = unit / per * 2 + (rem & 1), nt = unit % per * a.chunk + (rem >> 1);
    if (nt >= a.NT) return;
    if (mt >= a.MT) return;
    group = __builtin_amdgcn_readfirstlane(a.tile_group[mt]);
    if (group < 0) return;
  } else {
    gr_tile_of(gr_xcd_run((int)blockIdx.x, (int)gridDim.x), a.MT, a.NT, mt, nt);
  }
  // segment of the tile column (whole tiles per segment)
  int seg = 0, N = a.n[0];
  const uint16_t* w = static_cast<const uint16_t*>(a.w[0]);
  if (!PAIR) {
    if (a.nseg > 1 && nt >= (N + BN - 1) / BN) nt -= (N + BN - 1) / BN, seg = 1, N = a.n[1], w = static_cast<const uint16_t*>(a.w[1]);
    if (seg == 1 && a.nseg > 2 && nt >= (N + BN - 1) / BN) nt -= (N + BN - 1) / BN, seg = 2, N = a.n[2], w = static_cast<const uint16_t*>(a.w[2]);
  }
  gemm_rows_tile_product<DT, BM, BN, DEEP, PAIR>(a, epi, mt, nt, seg, N, w, group);
#endif
}

// One segment on two tiles: 256 x 256 for the first `mixed` tile columns of the whole 256-row blocks, 128 x 256 for the columns behind them and the rows
// below.  256 x 256 is the faster tile for the work it does, but its rounds are long: what is left of the last one idles.  2120 x (5632 gate + 5632 up),
// K = 2048: 8.3 x 44 of the large tile are 1.5 rounds, 16.6 x 44 of the small one 2.9; 256 of the one and 236 of the other are a round each.
// us, the best single tile / so (weights from memory): that pair 105 / 97, K = 4096 185 / 167; 3300 x 12288, K = 2048 156 / 143; 8192 x 3072 120 / 93; 6500 x 8192, K = 4096 367 / 342; over the
// 46 products of 1021..8192 rows, 3072..28672 columns that the rule takes 1.004..1.28 times as fast, 1.06 on average
template <class DT, bool PAIR, class EPI>
__global__ __launch_bounds__(512, 2) void gemm_rows_mixed_kernel(const GemmRowsArgs a, const EPI epi) {
#ifdef __HIP_DEVICE_COMPILE__
  const int N = a.n[0], fa = a.M >> 8, ca = a.mixed, large = fa * ca;
  const uint16_t* const w = static_cast<const uint16_t*>(a.w[0]);
  int bid = (int)blockIdx.x, mt, nt;
  if (bid < large) {
    gr_tile_of(gr_xcd_run(bid, large), fa, ca, mt, nt);
    gemm_rows_tile_product<DT, 256, 256, false, PAIR>(a, epi, mt, nt, 0, N, w, 0);
    return;
  }
  const int MT = (a.M + 127) >> 7, right = MT * (a.NT - ca), lin = gr_xcd_run(bid - large, (int)gridDim.x - large);
  if (lin < right) {
    gr_tile_of(lin, MT, a.NT - ca, mt, nt);
    nt += ca;
  } else {
    gr_tile_of(lin - right, MT - 2 * fa, ca, mt, nt);
    mt += 2 * fa;
  }
  gemm_rows_tile_product<DT, 128, 256, false, PAIR>(a, epi, mt, nt, 0, N, w, 0);
#endif
}

// Tile for a product of M rows x ncols[0..nseg) columns x `batch`: the least time by this model (us; 3079 shapes of 33..6000 rows, 1024..28672 columns,
// K = 512..18944, weights from memory: within 6..12 % rms, and the tile it picks 0.05 % behind the best on average, 7 % at most; every third of the
// shapes in profiles/gemm_rows_tile_times.txt): workgroups run in rounds of `slots`; a launch costs t0, a round `round` (first requests, outputs) and `full` for
// 64 of K, the last round between `one` (a few workgroups; `half`: every CU with one of its two) and `full`.  64 x 128 has two forms (gemm_rows_launch).
// With weights from the last-level cache 64 x 128 on two workgroups a CU is as fast as 128 x 128; from memory it is not: 192 rows x 14336, K = 4096 57 / 40 us, 700 x
// 4096, K = 2048 27 / 20.  192 x 128 is for what is a little more than one round of 128 x 128 and leaves much of one of 128 x 256 idle; us without / with it: 2120
// rows x 2048, K = 2048 31.7 / 26.5, K = 5632 67.2 / 56.2; 700 x 8192, K = 2048 35.1 / 30.5; 1280 x 4096, K = 14336 163 / 135.  192 x 256 does the same between
// 128 x 256 and 256 x 256: 1500 x 8192, K = 2048 57.2 / 48.8; 2120 x 4096, K = 4096 86.1 / 71.6; 2560 x 4096, K = 14336 272 / 235.
// rows: only tiles of that many (0: any).  -> rows / 64 * 16 + columns / 64; *us: the time
static inline int gemm_rows_tile(long M, const int* ncols, int nseg, long batch, int K, int rows = 0, double* us = nullptr) {
  const struct { int bm, bn, slots; double t0, round, one, half, full; } t[7] = {{256, 256, 256, 1.3, 9.2, 0.91, 0, 1.30}, {192, 256, 256, 1.0, 8.1, 0.72, 0, 1.00},
      {128, 256, 256, 0.5, 5.4, 0.70, 0, 0.81}, {192, 128, 256, 0.5, 5.0, 0.55, 0, 0.64}, {128, 128, 256, 1.3, 3.5, 0.41, 0, 0.51},
      {64, 128, 512, 3.2, 1.7, 0.34, 0.58, 0.66}, {64, 128, 256, 3.6, 0.0, 0.36, 0, 0.40}};
  int best = 0;
  double cost = 0.0;
  for (const auto& c : t) {
    if ((rows && c.bm != rows) || (c.bm * c.bn > 128 * 256 && K % 128)) continue;
    long cols = 0;
    for (int s = 0; s < nseg; s++) cols += (ncols[s] + c.bn - 1) / c.bn;
    const long tiles = (M + c.bm - 1) / c.bm * cols * batch, full = tiles / c.slots, rem = tiles % c.slots;
    if (c.bm == 64 && (tiles <= 256) != (c.slots == 256)) continue;
    double last = rem ? c.one + (c.full - c.one) * rem / c.slots : 0.0;
    if (c.slots == 512 && rem) last = rem <= 256 ? c.one : c.half + (c.full - c.half) * (rem - 256) / 256;  // (the second workgroup of a CU)
    const double v = c.t0 + (full + (rem ? 1 : 0)) * c.round + K / 64 * (full * c.full + last);
    if (!best || v < cost) best = c.bm / 64 * 16 + c.bn / 64, cost = v;
  }
  if (us) *us = cost;
  return best;
}
// ... for one segment that may be on two tiles (gemm_rows_mixed_kernel): the choice above, or 0x44 with the columns of 256 x 256 in the bits from 8 on.  The CUs
// that the last round of large tiles leaves free start on small ones; taken where the same model says 4 % or more.
static inline int gemm_rows_tiles(long M, int N, int K) {
  double us = 0.0;
  const int one = gemm_rows_tile(M, &N, 1, 1, K, 0, &us);
  const long fa = M / 256, MT = (M + 127) / 128, NT = (N + 255) / 256, KT = K / 64;
  if (K % 128 || fa == 0 || MT * NT <= 256) return one;
  const double large = 9.2 + KT * 1.30, small = 5.4 + KT * 0.81;
  int best = one;
  us *= 0.96;
  for (long ca = 1; ca <= NT; ca++) {
    const long rounds = (fa * ca + 255) / 256, early = (rounds * 256 - fa * ca) * (long)(large / small);
    const long rest = std::max(0L, MT * (NT - ca) + (MT - 2 * fa) * ca - early), full = rest / 256, rem = rest % 256;
    const double v = 1.3 + rounds * large + full * small + (rem ? 5.4 + KT * (0.70 + 0.11 * rem / 256) : 0.0);
    if (v < us) best = 0x44 | (int)ca << 8, us = v;
  }
  return best;
}
static inline bool gemm_rows_has_tile(int tile, int K) { return ((tile == 4 * 16 + 4 || tile == 3 * 16 + 4) && K % 128 == 0) || tile == 2 * 16 + 4 || tile == 3 * 16 + 2 || tile == 2 * 16 + 2 || tile == 16 + 2; }
// (columns of 256 x 256 in the bits from 8 on, a product of M rows and N columns)
static inline bool gemm_rows_has_tiles(int tile, int M, int N, int K) { return (tile & 0xff) == 0x44 && tile >> 8 > 0 && K % 128 == 0 && M >= 256 && (tile >> 8) * 256 < N + 256; }
// fills the tile counts and launches
template <class DT, int BM, int BN, bool DEEP, bool PAIR, class EPI>
static void gemm_rows_launch_t(GemmRowsArgs a, const EPI& epi, int batch, hipStream_t st) {
  a.MT = (a.M + BM - 1) / BM;
  a.NT = 0;
  for (int s = 0; s < a.nseg; s++) a.NT += (a.n[s] + BN - 1) / BN;
  static uint64_t attr_devs = 0;  // function attributes belong to the device current at the call
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (!((attr_devs >> (dev & 63)) & 1)) {
    void (*const k)(GemmRowsArgs, EPI) = gemm_rows_kernel<DT, BM, BN, DEEP, PAIR, EPI>;
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr_devs |= (uint64_t)1 << (dev & 63);
  }
  using T = GrTile<BM, BN, DEEP>;
  unsigned grid = (unsigned)(a.MT * a.NT);
  if (a.tile_group) {
    // Units of two tile rows x `chunk` columns, dealt to the eight XCDs in turn: all columns where there are pairs enough for four an XCD, otherwise as many
    // parts of equal size as make up for it, or an odd number of them, which go round the XCDs.  4 experts x 20 rows, 4096 columns, K = 4096, two tile rows
    // a unit with all columns / so 59.8 / 26.5 us (in runs 30.2); 8 x 260, 768 columns, K = 2048 27.5 / 17.9 (18.4); with 64 units instead of 32 19.0
    const int pairs = (a.MT + 1) / 2;
    int parts = std::min((32 + pairs - 1) / pairs, a.NT);
    do a.chunk = (a.NT + parts - 1) / parts;
    while (a.NT % a.chunk && (a.NT + a.chunk - 1) / a.chunk % 2 == 0 && ++parts);
    const int units = pairs * ((a.NT + a.chunk - 1) / a.chunk);
    grid = (unsigned)((units + 7) / 8 * 8 * 2 * a.chunk);
  }
  gemm_rows_kernel<DT, BM, BN, DEEP, PAIR, EPI><<<dim3(grid, (unsigned)batch), dim3(512), (size_t)T::S * T::KP * T::STG, st>>>(a, epi);
}
template <class DT, bool PAIR, class EPI>
static void gemm_rows_launch_mixed(GemmRowsArgs a, const EPI& epi, int columns, hipStream_t st) {
  a.mixed = columns;
  a.NT = (a.n[0] + 255) / 256;
  void (*const k)(GemmRowsArgs, EPI) = gemm_rows_mixed_kernel<DT, PAIR, EPI>;
  static uint64_t attr_devs = 0;  // (as above)
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (!((__atomic_load_n(&attr_devs, __ATOMIC_RELAXED) >> (dev & 63)) & 1)) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    __atomic_fetch_or(&attr_devs, (uint64_t)1 << (dev & 63), __ATOMIC_RELAXED);
  }
  using A = GrTile<256, 256, false>;
  using B = GrTile<128, 256, false>;
  const int fa = a.M / 256, MT = (a.M + 127) / 128;
  const unsigned grid = (unsigned)(fa * columns + MT * (a.NT - columns) + (MT - 2 * fa) * columns);
  k<<<grid, 512, (size_t)std::max(A::S * A::STG, B::S * B::STG), st>>>(a, epi);
}
// 64 x 128: two K steps a phase and twice the LDS where every workgroup has a CU to itself, otherwise two workgroups a CU.  (A phase of one step is two
// waits for LDS around 8 MFMAs a wave: 64 rows x 4096, K = 14336, 32 workgroups 79.7 us, six buffers 73.2, so 69.6; with the waves in step 94.4.)
template <class DT, bool PAIR, class EPI>
static void gemm_rows_launch(const GemmRowsArgs& a, const EPI& epi, int tile, int batch, hipStream_t st) {
  if constexpr (EPI::mixes)
    if (tile >> 8) return gemm_rows_launch_mixed<DT, PAIR>(a, epi, tile >> 8, st);
  if (tile == 4 * 16 + 4) return gemm_rows_launch_t<DT, 256, 256, false, PAIR>(a, epi, batch, st);
  if (tile == 3 * 16 + 4) return gemm_rows_launch_t<DT, 192, 256, false, PAIR>(a, epi, batch, st);
  if (tile == 2 * 16 + 4) return gemm_rows_launch_t<DT, 128, 256, false, PAIR>(a, epi, batch, st);
  if (tile == 3 * 16 + 2) return gemm_rows_launch_t<DT, 192, 128, false, PAIR>(a, epi, batch, st);
  if (tile == 2 * 16 + 2) return gemm_rows_launch_t<DT, 128, 128, false, PAIR>(a, epi, batch, st);
  long cols = 0;
  for (int s = 0; s < a.nseg; s++) cols += (a.n[s] + 127) / 128;
  if ((a.M + 63) / 64 * cols * batch <= 256) gemm_rows_launch_t<DT, 64, 128, true, PAIR>(a, epi, batch, st);
  else gemm_rows_launch_t<DT, 64, 128, false, PAIR>(a, epi, batch, st);
}
