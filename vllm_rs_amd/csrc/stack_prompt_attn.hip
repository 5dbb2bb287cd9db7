// stack_prompt_attn.hip — softmax attention of prompt steps with 64- and 128-channel heads (vra_stack_attention sends them here), gfx950.
//
// A workgroup: 64 query rows of one head, 16 a wave, over key tiles of 64 aligned to absolute positions:
//   S^T = K . Q^T    A operand = key rows (ds_read_b128), B = the wave's query rows, kept in registers;
//   O^T += V^T . P^T  A operand = the value tile read transposed (ds_read_b64_tr_b16), B = the lane's own weights, split into a bf16 head and a
//                    bf16 tail (p = hi + lo to 2^-17), so that the weights stay f32 in effect.
// Bound: the score arithmetic (VALU).  Per score: product and cap constants folded into one factor, hardware exponential (base 2),
// reciprocal, one multiply-add, maximum, exponential, sum, the hi / lo split; visibility is compared only in tiles that a row does not see whole.
// K and V tiles come from the paged cache straight into LDS (16 bytes a lane, no registers, no transposition by hand), one tile ahead of the
// arithmetic, two buffers of 32 KiB: two workgroups a CU cover each other's chains.  Before, every wave fetched its own key fragments and the
// tile's values went through registers, 32 keys between two barriers: 2048 tokens, 16 heads of 128, soft cap: 195 us; now 73.
//
// A row's running reference moves only when a score exceeds it by more than 8 (weights then stay below e^8, sums are f32): a decision of the row
// alone.  Tiles without a visible key change nothing.  So a row's result does not depend on the rows it shares a wave with, on the portion its
// token came in or on the pages.
#include "stack_common.cuh"
#include "stack_launch.h"

namespace {

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t* lds_s16x4_ptr;
typedef __attribute__((address_space(3))) void* lds_void_ptr;
typedef __attribute__((address_space(1))) const void* glb_void_ptr;

// chunk c (16 bytes) of row r of a tile lies at place c ^ swz(r): the 16 rows that a key fragment touches at one chunk lie in 16 different bank
// groups (rows of 256 bytes; of 128 bytes: two rows share the banks, and the row's low bit picks its half), and a transposed read's
// row groups spread as well
template <int RC>
__device__ __forceinline__ int tile_swz(int r) {
  return RC == 16 ? ((r & 7) << 1) | ((r >> 3) & 1) : (r >> 1) & 7;
}

template <int DC, int VT, bool CAP>
__global__ __launch_bounds__(256, 2) void stk_attn_prompt_kernel(StkAttnArgs a, int nblk, int pair) {
  constexpr int KT = 64, KC = 4 * DC, VC = 2 * VT, KROWB = KC * 16, VROWB = VC * 16, KB = KT * KROWB, TILEB = KB + KT * VROWB;
  constexpr float LOG2E = 1.4426950408889634f;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  __shared__ long long wmax[4], wmin[4];
  const int b = blockIdx.y, H = a.H;
  // the heads of a key/value head run on one XCD (ids mod 8); row blocks from the end of the portion first, as they see the most keys — when all
  // workgroups are on the chip at once (two a CU), the second half of the ids takes them from the start, so that a CU gets a long and a short one
  const int hi = (int)blockIdx.x % H, h = H % 8 == 0 ? (hi & 7) * (H >> 3) + (hi >> 3) : hi;
  int blk = (int)blockIdx.x / H;
  if (!pair || blk < (nblk + 1) / 2) blk = nblk - 1 - blk;
  else blk = blk - (nblk + 1) / 2;
  const int g = h / (H / a.G);
  const int q0 = a.cu_q[b], q1 = a.cu_q[b + 1], t0 = q0 + blk * 64;
  if (t0 >= q1) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), rq = lane & 15, oct = lane >> 4;
  const int tq = t0 + wave * 16 + rq;
  const bool qv = tq < q1;
  const int64_t pq = qv ? a.positions[tq] : -1;
  s16x8 qf[DC];
  {
    const uint16_t* q = (const uint16_t*)a.q + (size_t)(qv ? tq : q0) * a.ldq + (size_t)h * (DC * 32) + oct * 8;
#pragma unroll
    for (int c = 0; c < DC; c++) {
      const u32x4 v = *(const u32x4*)(q + c * 32);
      qf[c] = __builtin_bit_cast(s16x8, qv ? v : u32x4{0u, 0u, 0u, 0u});
    }
  }
  float temp = 1.f;
  if (a.temp_every > 0 && a.temp_coef != 0.f) temp = 1.f + a.temp_coef * logf((float)(((pq < 0 ? 0 : pq) + 1) / a.temp_every) + 1.f);
  const float sc = a.scale * temp * (a.head_scale ? a.head_scale[h] : 1.f);
  // scores in units of log2(e): x = f1 * s, or with a cap  cap - 2 cap / (1 + e^(2 s sc / cap))
  const float f1 = CAP ? sc * (2.f / a.softcap) * LOG2E : sc * LOG2E, cap2 = a.softcap * LOG2E;
  int64_t key_lo64 = a.chunk > 0 && pq >= 0 ? pq / a.chunk * a.chunk : 0;
  if (a.window > 0 && pq >= 0) key_lo64 = max(key_lo64, pq - a.window + 1);
  // the wave's rows: the keys any of them sees, and the ones all of them see
  int64_t pmax = pq, pmin = pq >= 0 ? pq : INT64_MAX, lmin = pq >= 0 ? key_lo64 : INT64_MAX, lmax = pq >= 0 ? key_lo64 : 0;
  for (int o = 32; o > 0; o >>= 1) {
    pmax = max(pmax, (int64_t)__shfl_xor((long long)pmax, o, 64));
    pmin = min(pmin, (int64_t)__shfl_xor((long long)pmin, o, 64));
    lmin = min(lmin, (int64_t)__shfl_xor((long long)lmin, o, 64));
    lmax = max(lmax, (int64_t)__shfl_xor((long long)lmax, o, 64));
  }
  if (lane == 0) wmax[wave] = pmax, wmin[wave] = lmin;
  __syncthreads();
  const int64_t gmax = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3])), gmin = min(min(wmin[0], wmin[1]), min(wmin[2], wmin[3]));
  const int kt_begin = gmin == INT64_MAX ? 0 : __builtin_amdgcn_readfirstlane((int)(gmin / KT) * KT);
  const int n_keys = __builtin_amdgcn_readfirstlane((int)min((int64_t)a.context_lens[b], gmax + 1));
  const int wave_end = __builtin_amdgcn_readfirstlane((int)min((int64_t)n_keys, pmax + 1));
  const int wave_lo = __builtin_amdgcn_readfirstlane(lmin == INT64_MAX ? 0 : (int)lmin);
  const int whole_lo = __builtin_amdgcn_readfirstlane((int)lmax), whole_end = __builtin_amdgcn_readfirstlane(pmin == INT64_MAX ? 0 : (int)min((int64_t)n_keys, pmin + 1));
  const int key_lo = (int)key_lo64, key_end = (int)min((int64_t)n_keys, pq + 1);
  const int k_ld = a.k_ld ? a.k_ld : a.G * DC * 32, v_ld = a.v_ld ? a.v_ld : a.G * VT * 16;
  const uint16_t* const kc = (const uint16_t*)a.kc + g * (DC * 32);
  const uint16_t* const vc = (const uint16_t*)a.vc + g * (VT * 16);
  const uint32_t* const bt = a.block_tables + (size_t)b * a.max_blocks;
  // The page size is a multiple of 64: a tile lies in one page.  Its first slot is a scalar, read from the block table one tile ahead of the
  // requests that use it.  Rows beyond the last key repeat it (their weights are 0).
  auto page_slot = [&](int k0) -> int64_t { return k0 < n_keys ? (int64_t)bt[k0 / a.BS] * a.BS + k0 % a.BS : 0; };
  auto request_tile = [&](int buf, int k0, int64_t slot0) {
    const int last = n_keys - 1 - k0;
#pragma unroll
    for (int k = 0; k < KC / 4; k++) {  // KT * KC chunks, 64 a request, 4 waves
      const int idx = k * 4 + wave, p = idx * 64 + lane, row = p / KC, c = (p % KC) ^ tile_swz<KC>(row);
      __builtin_amdgcn_global_load_lds((glb_void_ptr)(kc + (slot0 + min(row, last)) * k_ld + c * 8), (lds_void_ptr)(smem + buf * TILEB + idx * 1024), 16, 0, 0);
    }
#pragma unroll
    for (int k = 0; k < VC / 4; k++) {
      const int idx = k * 4 + wave, p = idx * 64 + lane, row = p / VC, c = (p % VC) ^ tile_swz<VC>(row);
      __builtin_amdgcn_global_load_lds((glb_void_ptr)(vc + (slot0 + min(row, last)) * v_ld + c * 8), (lds_void_ptr)(smem + buf * TILEB + KB + idx * 1024), 16, 0, 0);
    }
  };
  // LDS addresses of this lane inside a tile: key 16 u + rq, channels oct * 8 ..;  value rows 16 u + oct * 4 + rq / 4, 8 bytes of channels (rq & 3) * 4 ..
  const int ksw = tile_swz<KC>(rq), vrow = oct * 4 + (rq >> 2), vsw = tile_swz<VC>(vrow);
  f32x4 acc[VT];
#pragma unroll
  for (int t = 0; t < VT; t++) acc[t] = vra_zero_acc();
  float m = -INFINITY, l = 0.f;
  if (a.sink) m = a.sink[h] * LOG2E, l = oct == 0 ? 1.f : 0.f;  // (the four lanes of a row add their sums at the end: the sink counts once)
  if (kt_begin < n_keys) request_tile(0, kt_begin, page_slot(kt_begin));
  int64_t slot_next = page_slot(kt_begin + KT);
  int buf = 0;
  for (int kt0 = kt_begin; kt0 < n_keys; kt0 += KT, buf ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's part of the tile has arrived ...
    __syncthreads();                                  // ... and so has every wave's; nobody reads the other buffer any more
    if (kt0 + KT < n_keys) {
      request_tile(buf ^ 1, kt0 + KT, slot_next);
      slot_next = page_slot(kt0 + 2 * KT);
    }
    if (kt0 >= wave_end || kt0 + KT <= wave_lo) continue;  // (wave-uniform: nothing of this tile is visible to the wave's rows)
    const unsigned char* const kt = smem + buf * TILEB;
    const unsigned char* const vt = kt + KB;
    f32x4 s[4];
#pragma unroll
    for (int u = 0; u < 4; u++) s[u] = vra_zero_acc();
    s16x8 kf[2][4];
#pragma unroll
    for (int u = 0; u < 4; u++) kf[0][u] = *(const s16x8*)(kt + (u * 16 + rq) * KROWB + (oct ^ ksw) * 16);
#pragma unroll
    for (int c = 0; c < DC; c++) {
      if (c + 1 < DC)
#pragma unroll
        for (int u = 0; u < 4; u++) kf[(c + 1) & 1][u] = *(const s16x8*)(kt + (u * 16 + rq) * KROWB + (((c + 1) * 4 + oct) ^ ksw) * 16);
#pragma unroll
      for (int u = 0; u < 4; u++) BF16::mfma(s[u], kf[c & 1][u], qf[c]);
    }
    VRA_MFMA_DRAIN();
    const bool whole = kt0 >= whole_lo && kt0 + KT <= whole_end;  // (wave-uniform: every row sees every key of the tile)
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
      float z = s[i >> 2][i & 3] * f1;
      if (CAP) z = cap2 - 2.f * cap2 * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(__builtin_amdgcn_fmed3f(z, -43.f, 43.f)));
      x[i] = z;
    }
    if (!whole) {
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int key = kt0 + (i >> 2) * 16 + oct * 4 + (i & 3);
        x[i] = key < key_end && key >= key_lo ? x[i] : -INFINITY;
      }
    }
    float tmax = x[0];
#pragma unroll
    for (int i = 1; i < 16; i++) tmax = fmaxf(tmax, x[i]);
    tmax = vra_xor32_max(vra_xor16_max(tmax));
    const bool move = tmax > m + 8.f * LOG2E;  // (m = -inf: every finite score moves it; a row without a visible key so far: tmax = -inf, no move)
    if (__any(move)) {
      const float corr = move ? (m > -INFINITY ? __builtin_amdgcn_exp2f(m - tmax) : 0.f) : 1.f;
      m = move ? tmax : m;
      l *= corr;
#pragma unroll
      for (int t = 0; t < VT; t++) acc[t][0] *= corr, acc[t][1] *= corr, acc[t][2] *= corr, acc[t][3] *= corr;
    }
    float psum = 0.f;
    const float mr = m > -INFINITY ? m : 0.f;  // (a row without a visible key so far: its scores are -inf, its weights 0)
#pragma unroll
    for (int i = 0; i < 16; i++) {
      x[i] = __builtin_amdgcn_exp2f(x[i] - mr);
      psum += x[i];
    }
    l += psum;
    u32x4 ph[2], pl[2];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float a0 = x[2 * e], a1 = x[2 * e + 1];
      const uint32_t w = BF16::pack2(a0, a1);
      ph[e >> 2][e & 3] = w;
      pl[e >> 2][e & 3] = BF16::pack2(a0 - __uint_as_float(w << 16), a1 - __uint_as_float(w & 0xffff0000u));
    }
    auto vread = [&](int half, int t) {
      const unsigned char* const p = vt + (half * 32 + vrow) * VROWB + ((2 * t + ((rq & 3) >> 1)) ^ vsw) * 16 + (rq & 1) * 8;
      const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p));
      const s16x4_t up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_ptr)(p + 16 * VROWB));
      return __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    s16x8 vf[2][2];
    vf[0][0] = vread(0, 0), vf[0][1] = vread(0, 1);
#pragma unroll
    for (int i = 0; i < VT; i++) {  // pairs of channel tiles, first half of the keys, then the second
      const int half = i / (VT / 2), t = i % (VT / 2) * 2, n = i + 1, u = i & 1;
      if (n < VT) vf[u ^ 1][0] = vread(n / (VT / 2), n % (VT / 2) * 2), vf[u ^ 1][1] = vread(n / (VT / 2), n % (VT / 2) * 2 + 1);
      BF16::mfma(acc[t], vf[u][0], __builtin_bit_cast(s16x8, ph[half]));
      BF16::mfma(acc[t + 1], vf[u][1], __builtin_bit_cast(s16x8, ph[half]));
      BF16::mfma(acc[t], vf[u][0], __builtin_bit_cast(s16x8, pl[half]));
      BF16::mfma(acc[t + 1], vf[u][1], __builtin_bit_cast(s16x8, pl[half]));
    }
    VRA_MFMA_DRAIN();
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (!qv) return;
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (a.gate) inv *= sigmoidf_(a.gate[(size_t)tq * a.gate_ld + h]);
  uint16_t* const out = (uint16_t*)a.out + ((size_t)tq * H + h) * (VT * 16) + oct * 4;
#pragma unroll
  for (int t = 0; t < VT; t++) {
    uint2 v;
    v.x = BF16::pack2(acc[t][0] * inv, acc[t][1] * inv);
    v.y = BF16::pack2(acc[t][2] * inv, acc[t][3] * inv);
    *(uint2*)(out + t * 16) = v;
  }
}

}  // namespace

// heads of exactly 64 or 128 channels (keys and values), pages of whole 64-key tiles, rows on 16 bytes; other shapes stay with the general kernel
bool vra_stack_prompt_attention(const StkAttnArgs& a, int dtype, int64_t stream) {
  if (dtype != VRA_BF16 || !a.cu_q || a.maps != 1 || (a.dim != 64 && a.dim != 128) || (a.vdim != 64 && a.vdim != 128) || a.BS % 64 != 0) return false;
  if (a.ldq % 8 || a.k_ld % 8 || a.v_ld % 8 || (uintptr_t)a.q % 16 || (uintptr_t)a.kc % 16 || (uintptr_t)a.vc % 16 || (uintptr_t)a.out % 8) return false;
  const int nblk = (a.max_q + 63) / 64;
  if ((int64_t)nblk * a.H > 0x7fffffff || a.B > 65535) return false;
  const dim3 grid((unsigned)(nblk * a.H), (unsigned)a.B);
  const int pair = (int64_t)nblk * a.H * a.B <= 512;
  const size_t lds = (size_t)2 * 64 * (a.dim + a.vdim) * 2;
  hipStream_t st = as_stream(stream);
  auto go = [&](auto kernel) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    launch_checked("stack attention (prompt)", [&] { kernel<<<grid, 256, lds, st>>>(a, nblk, pair); });
  };
  const bool cap = a.softcap > 0.f;
  if (a.dim == 64 && a.vdim == 64) cap ? go(stk_attn_prompt_kernel<2, 4, true>) : go(stk_attn_prompt_kernel<2, 4, false>);
  else if (a.dim == 64) cap ? go(stk_attn_prompt_kernel<2, 8, true>) : go(stk_attn_prompt_kernel<2, 8, false>);
  else if (a.vdim == 64) cap ? go(stk_attn_prompt_kernel<4, 4, true>) : go(stk_attn_prompt_kernel<4, 4, false>);
  else cap ? go(stk_attn_prompt_kernel<4, 8, true>) : go(stk_attn_prompt_kernel<4, 8, false>);
  return true;
}
