// stack_prompt_attn.hip — softmax attention of prompt steps with 64- and 128-channel heads (vra_stack_attention sends them here), gfx950.
//
// A workgroup: 64 query rows of one head, over key tiles of 64 aligned to absolute positions; eight waves, 16 rows and 32 keys of every tile each,
// the two halves of the keys joined at the end:
//   S^T = K . Q^T    A operand = key rows (ds_read_b128), B = the wave's query rows, kept in registers;
//   O^T += V^T . P^T  A operand = the value tile read transposed (ds_read_b64_tr_b16), B = the lane's own weights, split into a bf16 head and a
//                    bf16 tail (p = hi + lo to 2^-17), so that the weights stay f32 in effect.
// Bound: the score arithmetic (VALU, about 60 % of the cycles).  Per score: product and cap constants folded into one factor, hardware exponential (base
// 2), reciprocal, minimum, multiply-add, exponential, sum, the hi / lo split; visibility is compared only in half tiles that a row does not see whole, and
// lanes compare their maxima only when one of them would move its row's reference.
// K and V tiles come from the paged cache straight into LDS (16 bytes a lane, no registers, no transposition by hand), one tile ahead of the
// arithmetic, two buffers of 32 KiB: two workgroups a CU cover each other's chains.  2048 tokens, 16 heads of 128, soft cap: 195 us with key fragments
// fetched by every wave and values through registers; 73 with four waves of 64 keys (two waves a SIMD, and one once a short row block has ended), the page
// looked up by a vector load and the compiler's transposed reads, either of which waited for the next tile's requests; 57 without all three; 53
// with the shorter arithmetic.  1500 tokens: 52, now 38.
//
// A row's running reference moves only when a score exceeds it by more than 8 (weights then stay below e^8, sums are f32): a decision of the row
// alone.  Half tiles without a visible key change nothing.  So a row's result does not depend on the rows it shares a wave with, on the portion its
// token came in or on the pages.
#include "stack_common.cuh"
#include "stack_launch.h"

namespace {

typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void* lds_void_ptr;
typedef __attribute__((address_space(1))) const void* glb_void_ptr;
typedef const __attribute__((address_space(4))) uint32_t* const_u32_ptr;

// chunk c (16 bytes) of row r of a tile lies at place c ^ swz(r): the 16 rows that a key fragment touches at one chunk lie in 16 different bank
// groups (rows of 256 bytes; of 128 bytes: two rows share the banks, and the row's low bit picks its half), and a transposed read's
// row groups spread as well
template <int RC>
__device__ __forceinline__ int tile_swz(int r) {
  return RC == 16 ? ((r & 7) << 1) | ((r >> 3) & 1) : (r >> 1) & 7;
}

// four channel tiles of 32 keys, transposed, and their wait: the compiler's own reads of this form would first wait for every request in flight, that is
// for the next tile
template <int LO, int UP>
__device__ __forceinline__ void value_tiles(s16x4_t (&lo)[4], s16x4_t (&up)[4], const uint32_t (&at)[4]) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8 offset:%12\n\tds_read_b64_tr_b16 %1, %8 offset:%13\n\t"
      "ds_read_b64_tr_b16 %2, %9 offset:%12\n\tds_read_b64_tr_b16 %3, %9 offset:%13\n\t"
      "ds_read_b64_tr_b16 %4, %10 offset:%12\n\tds_read_b64_tr_b16 %5, %10 offset:%13\n\t"
      "ds_read_b64_tr_b16 %6, %11 offset:%12\n\tds_read_b64_tr_b16 %7, %11 offset:%13\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(lo[0]), "=&v"(up[0]), "=&v"(lo[1]), "=&v"(up[1]), "=&v"(lo[2]), "=&v"(up[2]), "=&v"(lo[3]), "=&v"(up[3])
      : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "n"(LO), "n"(UP)
      : "memory");
}

template <int DC, int VT, bool CAP>
__global__ __launch_bounds__(512, 4) void stk_attn_prompt_kernel(StkAttnArgs a, int nblk, int pair) {
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
  const int tid = threadIdx.x, lane = tid & 63, wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave8 & 3, hh = wave8 >> 2, rq = lane & 15, oct = lane >> 4;
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
  if (lane == 0 && hh == 0) wmax[wave] = pmax, wmin[wave] = lmin;
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
  // The page size is a multiple of 64: a tile lies in one page, whose number is a scalar load one tile ahead of the requests that use it (as a vector load
  // its wait takes in the tile's requests as well).  Rows beyond the last key repeat it (their weights are 0).
  const const_u32_ptr bt = (const_u32_ptr)(uintptr_t)(a.block_tables + (size_t)b * a.max_blocks);
  int page = kt_begin / a.BS, in_page = kt_begin % a.BS;
  auto page_slot = [&]() -> int64_t {
    const int64_t at = (int64_t)bt[page] * a.BS + in_page;
    in_page += KT;
    if (in_page == a.BS) in_page = 0, page++;
    return at;
  };
  // this lane's rows and chunks of a request (KT * KC chunks, 64 a request, 8 waves), and its byte offsets in a tile of 64 keys
  uint32_t koff[KC / 8], voff[VC / 8];
  auto krow = [&](int k) { return ((k * 8 + wave8) * 64 + lane) / KC; };
  auto vrow_of = [&](int k) { return ((k * 8 + wave8) * 64 + lane) / VC; };
  auto kat = [&](int k, int row) { return (uint32_t)(row * k_ld + (lane % KC ^ tile_swz<KC>(krow(k))) * 8) * 2; };
  auto vat = [&](int k, int row) { return (uint32_t)(row * v_ld + (lane % VC ^ tile_swz<VC>(vrow_of(k))) * 8) * 2; };
#pragma unroll
  for (int k = 0; k < KC / 8; k++) koff[k] = kat(k, krow(k));
#pragma unroll
  for (int k = 0; k < VC / 8; k++) voff[k] = vat(k, vrow_of(k));
  auto request_tile = [&](int buf, int k0, int64_t slot0) __attribute__((always_inline)) {
    const int last = n_keys - 1 - k0;
    const unsigned char* const ks = (const unsigned char*)(kc + slot0 * k_ld);
    const unsigned char* const vs = (const unsigned char*)(vc + slot0 * v_ld);
    uint32_t ko[KC / 8], vo[VC / 8];
#pragma unroll
    for (int k = 0; k < KC / 8; k++) ko[k] = koff[k];
#pragma unroll
    for (int k = 0; k < VC / 8; k++) vo[k] = voff[k];
    if (last < KT - 1) {
#pragma unroll
      for (int k = 0; k < KC / 8; k++) ko[k] = kat(k, min(krow(k), last));
#pragma unroll
      for (int k = 0; k < VC / 8; k++) vo[k] = vat(k, min(vrow_of(k), last));
    }
#pragma unroll
    for (int k = 0; k < KC / 8; k++)
      __builtin_amdgcn_global_load_lds((glb_void_ptr)(ks + ko[k]), (lds_void_ptr)(smem + buf * TILEB + (k * 8 + wave8) * 1024), 16, 0, 0);
#pragma unroll
    for (int k = 0; k < VC / 8; k++)
      __builtin_amdgcn_global_load_lds((glb_void_ptr)(vs + vo[k]), (lds_void_ptr)(smem + buf * TILEB + KB + (k * 8 + wave8) * 1024), 16, 0, 0);
  };
  // LDS addresses of this lane inside a tile: key 16 u + rq, channels oct * 8 ..;  value rows 16 u + oct * 4 + rq / 4, 8 bytes of channels (rq & 3) * 4 ..
  const int ksw = tile_swz<KC>(rq), vrow = oct * 4 + (rq >> 2), vsw = tile_swz<VC>(vrow);
  const uint32_t smem0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  f32x4 acc[VT];
#pragma unroll
  for (int t = 0; t < VT; t++) acc[t] = vra_zero_acc();
  float m = -INFINITY, l = 0.f;
  if (a.sink && hh == 0) m = a.sink[h] * LOG2E, l = oct == 0 ? 1.f : 0.f;  // (the four lanes of a row add their sums at the end: the sink counts once)
  int64_t slot_next = 0;
  if (kt_begin < n_keys) request_tile(0, kt_begin, page_slot());
  if (kt_begin + KT < n_keys) slot_next = page_slot();
  int buf = 0;
  for (int kt0 = kt_begin; kt0 < n_keys; kt0 += KT, buf ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's part of the tile has arrived ...
    __syncthreads();                                  // ... and so has every wave's; nobody reads the other buffer any more
    if (kt0 + KT < n_keys) {
      request_tile(buf ^ 1, kt0 + KT, slot_next);
      if (kt0 + 2 * KT < n_keys) slot_next = page_slot();
    }
    const int k0 = kt0 + hh * 32;
    if (k0 >= wave_end || k0 + 32 <= wave_lo) continue;  // (wave-uniform: none of the wave's keys of this tile is visible to its rows)
    const unsigned char* const kt = smem + buf * TILEB + hh * 32 * KROWB;
    const uint32_t vt = smem0 + buf * TILEB + (hh * 32 + vrow) * VROWB + (rq & 1) * 8;  // (KB behind it)
    f32x4 s[2];
#pragma unroll
    for (int u = 0; u < 2; u++) s[u] = vra_zero_acc();
    s16x8 kf[2][2];
#pragma unroll
    for (int u = 0; u < 2; u++) kf[0][u] = *(const s16x8*)(kt + (u * 16 + rq) * KROWB + (oct ^ ksw) * 16);
#pragma unroll
    for (int c = 0; c < DC; c++) {
      if (c + 1 < DC)
#pragma unroll
        for (int u = 0; u < 2; u++) kf[(c + 1) & 1][u] = *(const s16x8*)(kt + (u * 16 + rq) * KROWB + (((c + 1) * 4 + oct) ^ ksw) * 16);
#pragma unroll
      for (int u = 0; u < 2; u++) BF16::mfma(s[u], kf[c & 1][u], qf[c]);
    }
    VRA_MFMA_DRAIN();
    const bool whole = k0 >= whole_lo && k0 + 32 <= whole_end;  // (wave-uniform: every row sees every one of these keys)
    // the scores; under a cap what the exponential leaves of them, 1 / (1 + e^..), from 1 (lowest) to 0, infinite where a key is not visible: the
    // weight is one multiply-add and one exponential from there, and the least of them, compared as whole numbers, is the largest score
    constexpr float HIDDEN = CAP ? INFINITY : -INFINITY;
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      x[i] = s[i >> 2][i & 3] * f1;
      if (CAP) x[i] = __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x[i]));
    }
    if (!whole) {
#pragma unroll
      for (int i = 0; i < 8; i++) {
        const int key = k0 + (i >> 2) * 16 + oct * 4 + (i & 3);
        x[i] = key < key_end && key >= key_lo ? x[i] : HIDDEN;
      }
    }
    float tmax = x[0];
    if (CAP) {
      uint32_t least = __float_as_uint(x[0]);
#pragma unroll
      for (int i = 1; i < 8; i++) least = min(least, __float_as_uint(x[i]));
      tmax = fmaf(-2.f * cap2, __uint_as_float(least), cap2);
    } else {
#pragma unroll
      for (int i = 1; i < 8; i++) tmax = fmaxf(tmax, x[i]);
    }
    if (__any(tmax > m + 8.f * LOG2E)) {  // (m = -inf: every finite score moves it; no visible key so far: tmax = -inf, no move)
      tmax = vra_xor32_max(vra_xor16_max(tmax));
      const bool move = tmax > m + 8.f * LOG2E;
      const float corr = move ? (m > -INFINITY ? __builtin_amdgcn_exp2f(m - tmax) : 0.f) : 1.f;
      m = move ? tmax : m;
      l *= corr;
#pragma unroll
      for (int t = 0; t < VT; t++) acc[t][0] *= corr, acc[t][1] *= corr, acc[t][2] *= corr, acc[t][3] *= corr;
    }
    float psum = 0.f;
    const float mr = m > -INFINITY ? m : 0.f;  // (a row without a visible key so far: its scores are -inf, its weights 0)
    const float top = cap2 - mr;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      x[i] = __builtin_amdgcn_exp2f(CAP ? fmaf(-2.f * cap2, x[i], top) : x[i] - mr);
      psum += x[i];
    }
    l += psum;
    u32x4 ph, pl;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float a0 = x[2 * e], a1 = x[2 * e + 1];
      const uint32_t w = BF16::pack2(a0, a1);
      ph[e] = w;
      pl[e] = BF16::pack2(a0 - __uint_as_float(w << 16), a1 - __uint_as_float(w & 0xffff0000u));
    }
#pragma unroll
    for (int t = 0; t < VT; t += 4) {
      s16x4_t lo[4], up[4];
      uint32_t at[4];
#pragma unroll
      for (int i = 0; i < 4; i++) at[i] = vt + (((2 * (t + i) + ((rq & 3) >> 1)) ^ vsw) * 16);
      value_tiles<KB, KB + 16 * VROWB>(lo, up, at);
      s16x8 vf[4];
#pragma unroll
      for (int i = 0; i < 4; i++) vf[i] = __builtin_shufflevector(lo[i], up[i], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
      for (int i = 0; i < 4; i++) BF16::mfma(acc[t + i], vf[i], __builtin_bit_cast(s16x8, ph));
#pragma unroll
      for (int i = 0; i < 4; i++) BF16::mfma(acc[t + i], vf[i], __builtin_bit_cast(s16x8, pl));
    }
    VRA_MFMA_DRAIN();
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  // the two halves of the keys: each wave gives away half of its channel tiles and finishes the other half with its partner's
  constexpr int HV = VT / 2;
  f32x4* const px = (f32x4*)smem;                 // [8 waves][HV][64]
  float* const pml = (float*)(smem + 8 * HV * 1024);  // [8 waves][2][16]
  __syncthreads();  // (the tiles have been read)
#pragma unroll
  for (int t = 0; t < HV; t++) px[(wave8 * HV + t) * 64 + lane] = hh ? acc[t] : acc[t + HV];
  if (lane < 16) pml[wave8 * 32 + lane] = m, pml[wave8 * 32 + 16 + lane] = l;
  __syncthreads();
  if (!qv) return;
  const int other = wave8 ^ 4;
  const float mo = pml[other * 32 + rq], lo = pml[other * 32 + 16 + rq], mm = fmaxf(m, mo);
  const float c = m > -INFINITY ? __builtin_amdgcn_exp2f(m - mm) : 0.f, co = mo > -INFINITY ? __builtin_amdgcn_exp2f(mo - mm) : 0.f;
  l = l * c + lo * co;
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (a.gate) inv *= sigmoidf_(a.gate[(size_t)tq * a.gate_ld + h]);
  uint16_t* const out = (uint16_t*)a.out + ((size_t)tq * H + h) * (VT * 16) + hh * (HV * 16) + oct * 4;
#pragma unroll
  for (int t = 0; t < HV; t++) {
    const f32x4 mine = hh ? acc[t + HV] : acc[t], po = px[(other * HV + t) * 64 + lane];
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; e++) y[e] = (mine[e] * c + po[e] * co) * inv;
    uint2 v;
    v.x = BF16::pack2(y[0], y[1]);
    v.y = BF16::pack2(y[2], y[3]);
    *(uint2*)(out + t * 16) = v;
  }
}

}  // namespace

// heads of exactly 64 or 128 channels (keys and values), pages of whole 64-key tiles, rows on 16 bytes; other shapes stay with the general kernel
bool vra_stack_prompt_attention(const StkAttnArgs& a, int dtype, int64_t stream) {
  if (dtype != VRA_BF16 || !a.cu_q || a.maps != 1 || (a.dim != 64 && a.dim != 128) || (a.vdim != 64 && a.vdim != 128) || a.BS % 64 != 0) return false;
  if (a.k_ld > 1 << 24 || a.v_ld > 1 << 24) return false;  // (byte offsets inside a tile in 32 bits)
  if (a.ldq % 8 || a.k_ld % 8 || a.v_ld % 8 || (uintptr_t)a.q % 16 || (uintptr_t)a.kc % 16 || (uintptr_t)a.vc % 16 || (uintptr_t)a.out % 8) return false;
  const int nblk = (a.max_q + 63) / 64;
  if ((int64_t)nblk * a.H > 0x7fffffff || a.B > 65535) return false;
  const dim3 grid((unsigned)(nblk * a.H), (unsigned)a.B);
  const int pair = (int64_t)nblk * a.H * a.B <= 512;
  const size_t lds = (size_t)2 * 64 * (a.dim + a.vdim) * 2;
  hipStream_t st = as_stream(stream);
  auto go = [&](auto kernel) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    launch_checked("stack attention (prompt)", [&] { kernel<<<grid, 512, lds, st>>>(a, nblk, pair); });
  };
  const bool cap = a.softcap > 0.f;
  if (a.dim == 64 && a.vdim == 64) cap ? go(stk_attn_prompt_kernel<2, 4, true>) : go(stk_attn_prompt_kernel<2, 4, false>);
  else if (a.dim == 64) cap ? go(stk_attn_prompt_kernel<2, 8, true>) : go(stk_attn_prompt_kernel<2, 8, false>);
  else if (a.vdim == 64) cap ? go(stk_attn_prompt_kernel<4, 4, true>) : go(stk_attn_prompt_kernel<4, 4, false>);
  else cap ? go(stk_attn_prompt_kernel<4, 8, true>) : go(stk_attn_prompt_kernel<4, 8, false>);
  return true;
}
