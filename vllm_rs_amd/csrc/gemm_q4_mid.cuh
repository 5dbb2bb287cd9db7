// gemm_q4_mid.cuh — "kernel M": int4 GEMM for 64 rows up (short and middle prompts), every row of a block of up to 160 in one workgroup.
//
// What bounds a short prompt's int4 product is not memory (the codes of a gate/up pair of 4096 x 14336 take 13 us) but the instructions beside the
// MFMAs: converting the codes, scaling the group sums, LDS reads, requests; and the kernels of 32- or 64-row tiles convert every code once per row
// block.  Here a workgroup owns 128 virtual columns (64 gate + 64 up of a pair) and ALL rows of the block, 32 MB of them (MB 2..5): 8 waves as 4
// (columns, two n-blocks each) x 2 (rows, MB m-tiles each), so a code is converted twice for up to 160 rows, and a k-tile's 8 MB MFMAs of a wave are
// 2 MB independent chains.  x, codes and scales of a k-tile of 128 travel by LDS-DMA through a ring of three stages; the 16-byte chunks of an x row
// lie at slot chunk ^ (row mod 16), so the fragment reads meet no bank twice.
// The two row halves (a wave of each on every SIMD) run one barrier apart: while one multiplies, the other scales its last group sums into acc and
// prepares its next tile.  A lone wave issues an instruction every five cycles or so, so the two phases are of about 130 instructions each; the
// conversions of a tile's later fragments lie between the MFMAs of its earlier ones.  Codes, scales and row sums are fetched by the first half
// alone: it asks for them a phase earlier and so two and a half phases ahead.
// us a launch with its row sums, both halves in step / so: gate/up of 4096 x 14336, 64 rows 37.6 / 34.6, 150 rows 57.7 / 54.8, 320 rows 104 / 97; down
// of 18944 x 3584, 150 rows 46.7 / 43.7, 700 rows 218 / 186; AWQ 62.3 / 61.5, 113 / 112, 49.3 / 47.9, 237 / 219.  Where a
// workgroup has few k-tiles the shift by a barrier shows: 300 rows, 2048 columns, K = 5632 AWQ 29.3 / 30.1, 192 x 4608, K = 3584 20.8 / 21.6; all else within 2 %.
// Against kernel D or W: gate/up of 4096 x 14336 behind its norm, 150 rows 91 / 53; AWQ, 3584 x 18944, 320 rows 190 / 147.
//
// The zero points come off per k-tile, acc += s (acc_g - (C + z) Sx): acc never holds more than the result's own size.  (Taken off once behind the
// k loop, x of mean 0.5 left the float32 sums of K = 14336 ten times as far from the 64-bit result.)  Symmetric codes have one z: a row's group sums
// start from -(C + 8) Sx as the C operand of the first MFMAs, four products for all columns; AWQ, and only it, takes (C + z) Sx off
// a column at a time.  The row sums Sx (xsum_rows_kernel, or the norm's launch) and the zero points travel with the ring.  That costs 3..5 % of a
// launch with symmetric codes and 10 % with AWQ against one product behind the loop.
//
// Few columns leave the chip idle: K is then split over gridDim.z, with the exchange of kernel D (slabs written through, a flag line a slice;
// only the last slice, whose workgroups start last, waits, and adds the slabs in slice order).
#pragma once
#include "gemm_q4_big.cuh"  // GemmDArgs

#define GM_THREADS 512
static inline size_t gemm_q4_mid_lds_bytes(int mb) { return (size_t)3 * (32 * mb * 256 + 8 * 1024 + 4 * 256 + 32 * mb * 4); }

template <class DT, bool DUAL, bool AWQ, int MB>
__global__ __launch_bounds__(GM_THREADS) void gemm_q4_mid_kernel(const GemmDArgs a) {
#ifdef __HIP_DEVICE_COMPILE__
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  constexpr int NB = 2, ROWS = 32 * MB, XB = ROWS * 256, WB = 8 * 1024, SB = 4 * 256, STG = XB + WB + SB + ROWS * 4, PER = MB + 4;
  constexpr uint32_t RSRC3 = 0x00020000u;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nn = lane & 15, oct = lane >> 4, wn = wave & 3, wm = wave >> 2;
  const int K = a.K, M = a.M, KT = K >> 7;
  const bool grouped = a.group_size > 0 && a.group_size < K;
  const int gsh = grouped ? 31 - __builtin_clz(a.group_size) : 31;
  const int m0 = (int)blockIdx.y * ROWS;

  // ---- the wave's two n-blocks: DUAL, block nb0 of gate and of up; else blocks nb0, nb0 + 1 of one tensor (segments are whole 64 columns)
  const void* wt[2] = {a.w0, DUAL ? a.w1 : a.w0};
  const void* sct[2] = {a.sc0, DUAL ? a.sc1 : a.sc0};
  const uint32_t* qzt[2] = {a.qz0, DUAL ? a.qz1 : a.qz0};
  const void* biast[2] = {a.bias0, a.bias1};
  void* outp = a.out;
  int N = a.N, out_ld = a.out_ld, nb0;
  if (DUAL) {
    nb0 = (int)blockIdx.x * 4 + wn;
  } else {
    nb0 = (int)blockIdx.x * 8 + wn * 2;
    if (a.nseg > 1) {
      const int s = (a.nseg > 2 && nb0 >= a.xseg[1].blk_start) ? 1 : (nb0 >= a.xseg[0].blk_start ? 0 : -1);
      if (s >= 0) {
        const GemvSeg& sg = a.xseg[s];
        wt[0] = wt[1] = sg.w, sct[0] = sct[1] = sg.scales, qzt[0] = qzt[1] = sg.qzeros, biast[0] = sg.bias, outp = sg.out, N = sg.n, out_ld = sg.out_ld;
        nb0 -= sg.blk_start;
      }
    }
  }
  bool ok[NB];
  int nbc[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int nb = nb0 + (DUAL ? 0 : b);
    ok[b] = nb * 16 < N;
    nbc[b] = ok[b] ? nb : 0;  // (a missing block streams block 0; its results are never stored)
  }
  // this workgroup's k-tiles: all of them, or slice blockIdx.z of a.splitk
  const int SK = a.splitk > 1 ? a.splitk : 1, zi = (int)blockIdx.z;
  const int kt0 = (int)((long)KT * zi / SK), kt1 = (int)((long)KT * (zi + 1) / SK);

  // ---- DMA sources.  Every wave fetches MB KiB of x (4 rows each).  The first row half's waves (wm = 0) alone also fetch, for their pair of columns, the
  // codes of both blocks, one copy of the blocks' scales (lanes 0..15) and zero points (lanes 16..19; the rest fetch the same again) and 8 MB row
  // sums: MB + 4 requests a k-tile (PER) against MB
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.x), 0, 0x7FFFFFF0, RSRC3);
  const __amdgpu_buffer_rsrc_t rw0 = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(wt[0]), 0, 0x7FFFFFF0, RSRC3);
  const __amdgpu_buffer_rsrc_t rw1 = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(wt[1]), 0, 0x7FFFFFF0, RSRC3);
  uint32_t vo_x[MB];
#pragma unroll
  for (int i = 0; i < MB; i++) {
    const int row = (wave * MB + i) * 4 + oct;
    vo_x[i] = ((uint32_t)min(m0 + row, M - 1) * (uint32_t)a.x_ld + (uint32_t)(nn ^ (row & 15)) * 8u) * 2u;  // rows >= M alias row M - 1 (never stored)
  }
  const uint32_t vo_w = (uint32_t)lane * 16u, so_w0 = (uint32_t)nbc[0] * (uint32_t)KT, so_w1 = (uint32_t)nbc[1] * (uint32_t)KT;
  typedef const __attribute__((address_space(1))) void* glb_ptr;
  typedef __attribute__((address_space(3))) void* lds_ptr;
  const int second = (lane & 16) ? (lane >> 1) & 1 : (lane >> 3) & 1;  // (the lane's block of the two)
  const bool zero_lane = AWQ && (lane & 16);
  const unsigned char *z0 = reinterpret_cast<const unsigned char*>(qzt[0]), *z1 = reinterpret_cast<const unsigned char*>(qzt[1]);
  const unsigned char *s0 = static_cast<const unsigned char*>(sct[0]), *s1 = static_cast<const unsigned char*>(sct[1]);
  asm("" : "+s"(z0), "+s"(z1), "+s"(s0), "+s"(s1));  // (in scalar registers: selected under a lane's index, they would be fetched by vector loads)
  const unsigned char* const sc_src = zero_lane ? (second ? z1 : z0) + ((second ? nbc[1] : nbc[0]) * 2 + (lane & 1)) * 4
                                                : (second ? s1 : s0) + ((second ? nbc[1] : nbc[0]) * 32 + (lane & 7) * 4);
  const uint32_t sc_ld = zero_lane ? (uint32_t)N / 2 : (uint32_t)N * 2;  // bytes between two groups
  const int srow = wn * 8 * MB;  // row sums of the rows srow + lane, lane < 8 MB
  const float* const sum_src = a.xsum + (size_t)min(m0 + srow + lane, M - 1) * KT;
  // requests of k-tile kt (beyond the last: the last again, never read) into the stage at byte `o`
  auto request = [&](int o, int kt) {
    unsigned char* const d = smem + o;
    kt = min(kt, kt1 - 1);
#pragma unroll
    for (int i = 0; i < MB; i++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr)(d + (wave * MB + i) * 1024), 16, vo_x[i], (uint32_t)kt * 256u, 0, 0);
    if (wm) return;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rw0, (lds_ptr)(d + XB + 2 * wn * 1024), 16, vo_w, (so_w0 + (uint32_t)kt) * 1024u, 0, 2);  // nt
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rw1, (lds_ptr)(d + XB + (2 * wn + 1) * 1024), 16, vo_w, (so_w1 + (uint32_t)kt) * 1024u, 0, 2);
    const int grp = grouped ? (kt * 128) >> gsh : 0;
    __builtin_amdgcn_global_load_lds((glb_ptr)(sc_src + (size_t)grp * sc_ld), (lds_ptr)(d + XB + WB + wn * 256), 4, 0, 0);
    if (lane < 8 * MB) __builtin_amdgcn_global_load_lds((glb_ptr)(sum_src + kt), (lds_ptr)(d + XB + WB + SB + srow * 4), 4, 0, 0);
  };

  f32x4 acc[NB][MB], ag[NB][MB];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int t = 0; t < MB; t++) acc[b][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const unsigned char* const xl = smem + (wm * MB * 16 + nn) * 256;
  const unsigned char* const wl = smem + XB + 2 * wn * 1024 + lane * 16;
  const unsigned char* const scl = smem + XB + WB + wn * 256;
  const unsigned char* const sml = smem + XB + WB + SB + (wm * MB * 16 + nn) * 4;
  u32x4 xf[4][MB];
  u32x4 wq[NB];
  s16x8 af[2][NB];
  u32x2 scc[NB];
  uint32_t zc[NB];
  float sxc[MB];
  f32x4 zx[MB];  // symmetric codes: the zero points' part of a row's group sums, the same for every column
  auto read_x = [&](int o, int j) {
#pragma unroll
    for (int t = 0; t < MB; t++) xf[j][t] = *reinterpret_cast<const u32x4*>(xl + o + (((j * 4 + oct) ^ nn) * 16) + t * 4096);
  };
  // a k-tile's group sums, scaled, into acc
  auto fix = [&]() {
    VRA_MFMA_DRAIN();
#pragma unroll
    for (int b = 0; b < NB; b++) {
      float s4[4], z4[4];
      unpack_scale4<DT>(scc[b], zc[b], oct * 4, s4, z4);
#pragma unroll
      for (int t = 0; t < MB; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[b][t][r] = fmaf(s4[r], AWQ ? fmaf(-z4[r], sxc[t], ag[b][t][r]) : ag[b][t][r], acc[b][t][r]);
    }
  };
  // the vector half of k-tile kt: codes, scales, zero points and row sums from LDS; the sums of tile kt - 1 into acc meanwhile; conversions
  auto prepare = [&](int o, bool first) {
    u32x2 scw[NB];
    uint32_t zw[NB];
    float sx[MB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
      wq[b] = *reinterpret_cast<const u32x4*>(wl + o + b * 1024);
      scw[b] = *reinterpret_cast<const u32x2*>(scl + o + b * 32 + oct * 8);
      if (AWQ) zw[b] = *reinterpret_cast<const uint32_t*>(scl + o + 64 + b * 8 + (oct >> 1) * 4);
    }
#pragma unroll
    for (int t = 0; t < MB; t++) sx[t] = *reinterpret_cast<const float*>(sml + o + t * 64);
    read_x(o, 0);
    read_x(o, 1);
    __builtin_amdgcn_sched_barrier(0);
    if (!first) fix();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < NB; b++) {
      scc[b] = scw[b], zc[b] = AWQ ? zw[b] : 0;
      af[0][b] = magic_word<DT>(wq[b][0]);
    }
#pragma unroll
    for (int t = 0; t < MB; t++) {
      sxc[t] = sx[t];
      const float z = AWQ ? 0.f : -(Magic<DT>::bias + 8.f) * sx[t];
      zx[t] = f32x4{z, z, z, z};
      asm volatile("" : "+v"(zx[t]));
    }
#pragma unroll
    for (int b = 0; b < NB; b++) asm volatile("" : "+v"(af[0][b]));
  };
  auto multiply = [&](int o) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (j < 2) read_x(o, j + 2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < MB; t++)
#pragma unroll
        for (int b = 0; b < NB; b++) {
          const s16x8 xv = __builtin_bit_cast(s16x8, xf[j][t]);
          if (j == 0 && AWQ) DT::mfma0(ag[b][t], af[0][b], xv);
          else if (j == 0) DT::mfma_from(ag[b][t], af[0][b], xv, zx[t]);
          else if (t == 0) DT::mfma(ag[b][t], af[j & 1][b], xv);
          else DT::mfma_ready(ag[b][t], af[j & 1][b], xv);
          if (j < 3 && t == 1) af[(j + 1) & 1][b] = magic_word<DT>(wq[b][j + 1]);
        }
    }
    __builtin_amdgcn_s_setprio(0);
  };
  auto barrier = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  request(0, kt0);
  request(STG, kt0 + 1);
  if (wm == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER) : "memory");
  else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MB) : "memory");
  barrier();
  if (wm == 1) barrier();  // the second group runs one barrier behind the first
  int o = 0, q = 2 * STG;  // stages of this k-tile and of the one after the next
  for (int kt = kt0; kt < kt1; kt++) {
    prepare(o, kt == kt0);
    if (wm == 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    barrier();
    request(q, kt + 2);
    multiply(o);
    if (wm == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER) : "memory");
    barrier();
    o = o == 2 * STG ? 0 : o + STG;
    q = q == 2 * STG ? 0 : q + STG;
  }
  if (wm == 0) barrier();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the requests beyond the last tile still write LDS)
  fix();

  // ---- split K: kernel D's exchange
  if (SK > 1) {
    const int tile = (int)(blockIdx.y * gridDim.x + blockIdx.x), ntiles = (int)(gridDim.x * gridDim.y);
    const __amdgpu_buffer_rsrc_t srs = __builtin_amdgcn_make_buffer_rsrc(a.slabs, 0, 0x7FFFFFF0, RSRC3);
    auto slab_off = [&](int z, int b, int mt) { return (uint32_t)((((z * ntiles + tile) * NB + b) * MB + mt) * GM_THREADS + tid) * 16u; };
    uint32_t* fl = a.counters + (size_t)tile * SK * 16;
    if (zi != SK - 1) {
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int mt = 0; mt < MB; mt++) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[b][mt]), srs, slab_off(zi, b, mt), 0, 16);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // write-through stores: acknowledged by memory
      __syncthreads();
      if (tid == 0) __hip_atomic_store(fl + zi * 16, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    if (tid < SK - 1) {
      const uint64_t c0 = __builtin_readcyclecounter();
      while (__hip_atomic_load(fl + tid * 16, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) {
        __builtin_amdgcn_s_sleep(1);
        if (__builtin_readcyclecounter() - c0 > (1ull << 31)) {  // never hang the device on a lost slice
          __hip_atomic_store(a.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
      }
      __hip_atomic_store(fl + tid * 16, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    // a slab's 2 MB loads a lane are requested one slab ahead of their sum; slice order
    u32x4 p[2][NB][MB];
    auto fetch = [&](int z, u32x4 (&d)[NB][MB]) {
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int mt = 0; mt < MB; mt++) d[b][mt] = __builtin_amdgcn_raw_buffer_load_b128(srs, slab_off(z, b, mt), 0, 16);
    };
    auto add = [&](const u32x4 (&d)[NB][MB]) {
#pragma unroll
      for (int b = 0; b < NB; b++)
#pragma unroll
        for (int mt = 0; mt < MB; mt++) acc[b][mt] += __builtin_bit_cast(f32x4, d[b][mt]);
    };
    fetch(0, p[0]);
    for (int z = 0; z < SK - 1; z += 2) {
      fetch(min(z + 1, SK - 2), p[1]);
      __builtin_amdgcn_sched_barrier(0);
      add(p[0]);
      fetch(min(z + 2, SK - 2), p[0]);
      __builtin_amdgcn_sched_barrier(0);
      if (z + 1 < SK - 1) add(p[1]);
    }
  }

  // ---- epilogue: column oct * 4 + r of the block, row nn of the m-tile
#pragma unroll
  for (int b = 0; b < (DUAL ? 1 : NB); b++) {
    if (!ok[b]) continue;
    const int n = nbc[b] * 16 + oct * 4;
    auto four = [&](const void* p, size_t at, float (&f)[4]) {
      const u32x2 v = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(p) + at);
      f[0] = DT::to_f32((uint16_t)(v[0] & 0xffffu)), f[1] = DT::to_f32((uint16_t)(v[0] >> 16));
      f[2] = DT::to_f32((uint16_t)(v[1] & 0xffffu)), f[3] = DT::to_f32((uint16_t)(v[1] >> 16));
    };
    float bs[4] = {0.f, 0.f, 0.f, 0.f}, bs2[4] = {0.f, 0.f, 0.f, 0.f};
    if (biast[0]) four(biast[0], n, bs);
    if (DUAL && biast[1]) four(biast[1], n, bs2);
#pragma unroll
    for (int mt = 0; mt < MB; mt++) {
      const int m = m0 + wm * (MB * 16) + mt * 16 + nn;
      if (m >= M) continue;
      float v[4], rs[4];
#pragma unroll
      for (int r = 0; r < 4; r++) {
        float t = rnd_dt<DT>(acc[b][mt][r]);
        if (biast[0]) t = rnd_dt<DT>(t + bs[r]);
        if (DUAL) {
          float u = rnd_dt<DT>(acc[1][mt][r]);
          if (biast[1]) u = rnd_dt<DT>(u + bs2[r]);
          t = rnd_dt<DT>(t / (1.0f + expf(-t))) * u;
        }
        v[r] = t;
      }
      if (a.residual) {
        four(a.residual, (size_t)m * a.res_ld + n, rs);
#pragma unroll
        for (int r = 0; r < 4; r++) v[r] = rnd_dt<DT>(v[r]) + rs[r];
      }
      if (a.out_f32) {
        const f32x4 o = {rnd_dt<DT>(v[0]), rnd_dt<DT>(v[1]), rnd_dt<DT>(v[2]), rnd_dt<DT>(v[3])};
        *reinterpret_cast<f32x4*>(static_cast<float*>(outp) + (size_t)m * out_ld + n) = o;
      } else {
        const u32x2 o = {DT::pack2(v[0], v[1]), DT::pack2(v[2], v[3])};
        *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(outp) + (size_t)m * out_ld + n) = o;
      }
    }
  }
#endif
}
