// stack_decode_attn.hip — softmax attention of decode steps over bf16 key/value heads (vra_stack_attention sends them here), gfx950.
//
// A workgroup: one sequence, one key/value head with all its query heads, one part of the context; the last part of a (sequence, key/value head) to
// finish adds the parts up, in their order, in the same launch.
//   scores  S^T = K . Q^T on the matrix cores: key rows go from the cache straight into the A operand (64 bytes a row and load), the query heads
//           are the columns (bf16 values with f32 sums: the products are exact, the query's temperature and the scale come after the sum);
//   values  f32 weights times values on the VALU: a lane holds 8 channels of some of the tile's keys, for every head.  The weights stay f32.
// What bounds it: the chain position -> block table -> rows -> sums -> exchange, so a wave has all rows of its 16 keys in flight at once, and parts
// are short (128 keys, a tile a wave) until a context has more parts than STK_DEC_PARTS.  The one-head kernel in stack_ops.hip, which reads every
// key row a lane (16 bytes from each of 64 cache lines a load) and the rows again for every query head of a key/value head, took 19.4 us for 8
// sequences of up to 700 tokens, 16 heads over 4 of 128 channels; this one 11.1.  It still serves float32 models, head sizes off 8 channels, callers
// without scratch memory and more than 8 query heads a key/value head.
//
// Parts begin at the first visible key's place in steps of 64 and their length follows from the number of visible keys: the order of a row's sums depends
// on its own context alone.
#include <algorithm>

#include "stack_common.cuh"
#include "stack_launch.h"

namespace {

// R: query heads of a key/value head, rounded up; DC: chunks of 32 key channels; OC: octets of value channels, rounded up
constexpr int group_waves(int R, int OC) { return R * OC > 128 ? 4 : 8; }  // (their sums meet in 32 KB of LDS)
template <int R, int DC, int OC>
__global__ __launch_bounds__(64 * group_waves(R, OC)) void stk_attn_decode_group_kernel(StkAttnArgs a) {
  constexpr int NW = group_waves(R, OC), NT = 64 * NW, KPL = OC / 4, VD = OC * 8, E = (R * VD + NT - 1) / NT;  // KPL: keys of a tile whose values a lane takes
  __shared__ __attribute__((aligned(16))) float ps[NW][R][16];
  __shared__ __attribute__((aligned(16))) float os[NW][R][VD];
  __shared__ float ms[NW][R], ls[NW][R], pm[R][STK_DEC_PARTS], pl[R][STK_DEC_PARTS];
  __shared__ int last_here;
  const int part = blockIdx.x, g = blockIdx.y, b = blockIdx.z, HR = a.H / a.G;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), rq = lane & 15, oct = lane >> 4;
  const uint32_t* bt = a.block_tables + (size_t)b * a.max_blocks;
  // the page of the first tile's keys as it is when nothing is masked and the parts are short, asked for beside the position
  const int guess = min((part * 128 + wave * 16 + rq) / a.BS, a.max_blocks - 1);
  const uint32_t guessed = bt[guess];
  const int64_t p = a.positions[b];
  const int n_keys = max(0, (int)min((int64_t)a.context_lens[b], p + 1));
  int key_lo = a.chunk > 0 ? (int)(p / a.chunk * a.chunk) : 0;
  if (a.window > 0) key_lo = max(key_lo, (int)(p - a.window + 1));
  const int lo = key_lo / 64 * 64, span = max(n_keys - lo, 0);
  const int len = max(1, (span + 128 * a.splits - 1) / (128 * a.splits)) * 128, parts = max(1, (span + len - 1) / len);
  if (part >= parts) return;
  const int k0 = lo + part * len, k1 = min(n_keys, k0 + len);
  const int dim = a.dim, vdim = a.vdim, kld = a.G * dim, vld = a.G * vdim;
  const u32x4 zero4 = {0u, 0u, 0u, 0u};
  const bool hv = rq < HR;
  s16x8 qf[DC];
  {
    const uint16_t* q = (const uint16_t*)a.q + (size_t)b * a.ldq + (size_t)(g * HR + (hv ? rq : 0)) * dim;
#pragma unroll
    for (int c = 0; c < DC; c++) {
      const int ch = c * 32 + oct * 8;
      const bool in = hv && ch < dim;
      const u32x4 v = *(const u32x4*)(q + (in ? ch : 0));
      qf[c] = __builtin_bit_cast(s16x8, in ? v : zero4);
    }
  }
  const float temp = (a.temp_every <= 0 || a.temp_coef == 0.f) ? 1.f : 1.f + a.temp_coef * logf((float)((p + 1) / a.temp_every) + 1.f);
  const float hscale = a.head_scale ? a.scale * a.head_scale[g * HR + (hv ? rq : 0)] : a.scale;
  const uint16_t* kc = (const uint16_t*)a.kc + (size_t)g * dim;
  const uint16_t* vc = (const uint16_t*)a.vc + (size_t)g * vdim;
  const int co = lane & (OC - 1), kg = lane / OC;
  const bool cv = co * 8 < vdim;
  float m = -INFINITY, l = 0.f, acc[R][8];
#pragma unroll
  for (int r = 0; r < R; r++)
#pragma unroll
    for (int i = 0; i < 8; i++) acc[r][i] = 0.f;
  for (int kt = k0 + wave * 16; kt < k1; kt += 16 * NW) {
    const int kk = min(kt + rq, k1 - 1), page = kk / a.BS;  // keys beyond the part: its last key, weight 0
    const int slot = (int)(page == guess ? guessed : bt[page]) * a.BS + kk % a.BS;
    u32x4 kf[DC], vf[KPL];
    const uint16_t* row = kc + (size_t)slot * kld;
#pragma unroll
    for (int c = 0; c < DC; c++) {
      const int ch = c * 32 + oct * 8;
      kf[c] = *(const u32x4*)(row + (ch < dim ? ch : 0));
    }
#pragma unroll
    for (int u = 0; u < KPL; u++) vf[u] = *(const u32x4*)(vc + (size_t)__shfl(slot, kg * KPL + u, 64) * vld + (cv ? co * 8 : 0));
    f32x4 s = vra_zero_acc();
#pragma unroll
    for (int c = 0; c < DC; c++) BF16::mfma(s, __builtin_bit_cast(s16x8, c * 32 + oct * 8 < dim ? kf[c] : zero4), qf[c]);
    VRA_MFMA_DRAIN();
    float x[4], tmax = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int key = kt + oct * 4 + j;
      float v = s[j] * temp * hscale;
      if (a.softcap > 0.f) v = a.softcap * tanhf(v / a.softcap);
      x[j] = key < k1 && key >= key_lo ? v : -INFINITY;
      tmax = fmaxf(tmax, x[j]);
    }
    tmax = vra_xor32_max(vra_xor16_max(tmax));
    const float mn = fmaxf(m, tmax), corr = m > -INFINITY ? expf(m - mn) : 0.f;
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      x[j] = x[j] > -INFINITY ? expf(x[j] - mn) : 0.f;
      sum += x[j];
    }
    l = l * corr + sum, m = mn;
    if (rq < R) *(float4*)&ps[wave][rq][oct * 4] = make_float4(x[0], x[1], x[2], x[3]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int r = 0; r < R; r++) {
      const float c = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(corr), r));
#pragma unroll
      for (int i = 0; i < 8; i++) acc[r][i] *= c;
    }
#pragma unroll
    for (int u = 0; u < KPL; u++) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 4; i++) v[2 * i] = __uint_as_float(vf[u][i] << 16), v[2 * i + 1] = __uint_as_float(vf[u][i] & 0xffff0000u);
#pragma unroll
      for (int r = 0; r < R; r++) {
        const float w = ps[wave][r][kg * KPL + u];
#pragma unroll
        for (int i = 0; i < 8; i++) acc[r][i] = fmaf(w, v[i], acc[r][i]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  l = vra_xor32_sum(vra_xor16_sum(l));
  if (oct == 0 && rq < R) ms[wave][rq] = m, ls[wave][rq] = l;
#pragma unroll
  for (int r = 0; r < R; r++) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      float v = acc[r][i];
      if (OC <= 8) v += __shfl_xor(v, 8, 64);
      if (OC <= 16) v = vra_xor16_sum(v);
      v = vra_xor32_sum(v);
      acc[r][i] = v;
    }
    if (lane < OC) {
      *(float4*)&os[wave][r][lane * 8] = make_float4(acc[r][0], acc[r][1], acc[r][2], acc[r][3]);
      *(float4*)&os[wave][r][lane * 8 + 4] = make_float4(acc[r][4], acc[r][5], acc[r][6], acc[r][7]);
    }
  }
  __syncthreads();
  // the waves' sums in wave order
  float o[E];
#pragma unroll
  for (int e = 0; e < E; e++) {
    const int r = min((tid + e * NT) / VD, R - 1), c = (tid + e * NT) % VD;
    float M = ms[0][r], v = 0.f;
#pragma unroll
    for (int w = 1; w < NW; w++) M = fmaxf(M, ms[w][r]);
#pragma unroll
    for (int w = 0; w < NW; w++) v += os[w][r][c] * (ms[w][r] > -INFINITY ? expf(ms[w][r] - M) : 0.f);
    o[e] = v;
  }
  float M = -INFINITY, L = 0.f;
  if (tid < R) {
#pragma unroll
    for (int w = 0; w < NW; w++) M = fmaxf(M, ms[w][tid]);
#pragma unroll
    for (int w = 0; w < NW; w++) L += ms[w][tid] > -INFINITY ? ls[w][tid] * expf(ms[w][tid] - M) : 0.f;
  }
  const size_t bg = (size_t)b * a.G + g;
  float* rows = a.scratch + bg * a.splits * R * VD;                                             // [part][R][VD]
  float* ml = a.scratch + (size_t)gridDim.z * a.G * a.splits * R * VD + bg * a.splits * R * 2;  // [part][R][2]
  float v[E][8];
  auto fetch = [&](int s0) {  // (parts beyond the last: its rows again, weight 0)
#pragma unroll
    for (int u = 0; u < 8; u++)
#pragma unroll
      for (int e = 0; e < E; e++)
        v[e][u] = __hip_atomic_load(rows + (size_t)min(s0 + u, parts - 1) * R * VD + min(tid + e * NT, R * VD - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if (parts > 1) {
#pragma unroll
    for (int e = 0; e < E; e++)
      if (tid + e * NT < R * VD) __hip_atomic_store(rows + (size_t)part * R * VD + tid + e * NT, o[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (tid < R) {
      __hip_atomic_store(ml + (part * R + tid) * 2, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(ml + (part * R + tid) * 2 + 1, L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // write-through stores: acknowledged by memory
    __syncthreads();
    if (tid == 0) last_here = __hip_atomic_fetch_add(a.arrived + bg, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(parts - 1);
    __syncthreads();
    if (!last_here) return;
    if (tid == 0) __hip_atomic_store(a.arrived + bg, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // all parts' maxima and sums and the first eight's rows are requested at once, past the caches of this XCD
    static_assert(R * STK_DEC_PARTS <= NT, "a part's maximum and sum a thread");
    float mi = 0.f, li = 0.f;
    if (tid < parts * R) {
      mi = __hip_atomic_load(ml + tid * 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      li = __hip_atomic_load(ml + tid * 2 + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    fetch(0);
    if (tid < parts * R) pm[tid % R][tid / R] = mi, pl[tid % R][tid / R] = li;
  } else {
    if (tid < R) pm[tid][0] = M, pl[tid][0] = L;
#pragma unroll
    for (int e = 0; e < E; e++)
#pragma unroll
      for (int u = 0; u < 8; u++) v[e][u] = o[e];
  }
  __syncthreads();
  // a head's weights of its parts: wave w takes heads w, w + NW, ..; a lane a part (at most 32: both halves of the wave hold the same)
  for (int r = wave; r < HR; r += NW) {
    const int i = lane & 31;
    const float mi = i < parts ? pm[r][i] : -INFINITY, li = i < parts ? pl[r][i] : 0.f;
    const float sink = a.sink ? a.sink[g * HR + r] : -INFINITY;
    float top = mi;
    top = fmaxf(top, dpp_f32<0xB1>(top));
    top = fmaxf(top, dpp_f32<0x4E>(top));
    top = fmaxf(top, dpp_f32<0x141>(top));
    top = fmaxf(top, dpp_f32<0x140>(top));
    top = fmaxf(vra_xor16_max(top), sink);
    const float w = mi > -INFINITY ? expf(mi - top) : 0.f;
    float total = w * li;
    total += dpp_f32<0xB1>(total);
    total += dpp_f32<0x4E>(total);
    total += dpp_f32<0x141>(total);
    total += dpp_f32<0x140>(total);
    total = vra_xor16_sum(total) + (a.sink ? expf(sink - top) : 0.f);
    const float f = total > 0.f ? (a.gate ? sigmoidf_(a.gate[(size_t)b * a.gate_ld + g * HR + r]) : 1.f) / total : 0.f;
    if (lane < STK_DEC_PARTS) pm[r][lane] = w;
    if (lane == 0) pl[r][0] = f;
  }
  __syncthreads();
  float t[E];
#pragma unroll
  for (int e = 0; e < E; e++) t[e] = 0.f;
  for (int s0 = 0; s0 < parts; s0 += 8) {
    if (s0 > 0) fetch(s0);
#pragma unroll
    for (int e = 0; e < E; e++) {
      const int r = min((tid + e * NT) / VD, HR - 1);
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (s0 + u < parts) t[e] = fmaf(pm[r][s0 + u], v[e][u], t[e]);
    }
  }
  uint16_t* out = (uint16_t*)a.out + ((size_t)b * a.H + (size_t)g * HR) * vdim;
#pragma unroll
  for (int e = 0; e < E; e++) {
    const int r = (tid + e * NT) / VD, c = (tid + e * NT) % VD;
    if (r < HR && c < vdim) out[(size_t)r * vdim + c] = BF16::from_f32(t[e] * pl[r][0]);
  }
}

int group_width(int n) { return n <= 1 ? 1 : n <= 2 ? 2 : n <= 4 ? 4 : 8; }
int value_width(int dim, int vdim) { return std::max(dim, vdim) <= 64 ? 64 : std::max(dim, vdim) <= 128 ? 128 : 256; }
bool group_shape(int heads, int kv_heads, int dim, int vdim) {
  return kv_heads > 0 && heads / kv_heads <= 8 && dim % 8 == 0 && vdim % 8 == 0 && dim <= 256 && vdim <= 256;
}

}  // namespace

// parts of a context's keys: no more than its 128-key tiles, the workspace's memory (256 MB) and STK_DEC_PARTS
int vra_stack_decode_parts(int max_len, int max_seqs, int heads, int kv_heads, int dim, int vdim, int dtype) {
  if (dtype != VRA_BF16 || !group_shape(heads, kv_heads, dim, vdim)) return 0;
  int s = std::min(STK_DEC_PARTS, (std::max(max_len, 1) + 127) / 128);
  while (s > 1 && vra_stack_decode_scratch(s, max_seqs, heads, kv_heads, dim, vdim) > (size_t)256 << 20) s--;
  return s;
}
size_t vra_stack_decode_scratch(int parts, int max_seqs, int heads, int kv_heads, int dim, int vdim) {
  return (size_t)max_seqs * kv_heads * parts * group_width(heads / kv_heads) * (value_width(dim, vdim) + 2) * sizeof(float);
}

bool vra_stack_decode_group(const StkAttnArgs& a, int dtype, int64_t stream) {
  auto al16 = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  if (dtype != VRA_BF16 || a.maps != 1 || a.cu_q || !a.arrived || !a.scratch || a.splits < 1 || a.splits > STK_DEC_PARTS || a.B > 65535 || a.G > 65535) return false;
  if (a.k_ld || a.v_ld) return false;  // (cache rows apart: no model's heads have them)
  if (!group_shape(a.H, a.G, a.dim, a.vdim) || a.ldq % 8 || !al16(a.q) || !al16(a.kc) || !al16(a.vc)) return false;
  if (vra_stack_decode_scratch(a.splits, a.B, a.H, a.G, a.dim, a.vdim) > a.scratch_bytes) return false;
  const dim3 grid(std::min<int64_t>(a.splits, ((int64_t)a.max_blocks * a.BS + 127) / 128), a.G, a.B);
  const int R = group_width(a.H / a.G), w = value_width(a.dim, a.vdim);
  hipStream_t st = as_stream(stream);
#define STK_GRP(RV, DCV, OCV) launch_checked("stack attention (decode, heads together)", [&] { stk_attn_decode_group_kernel<RV, DCV, OCV><<<grid, 64 * group_waves(RV, OCV), 0, st>>>(a); })
#define STK_GRPR(DCV, OCV)            \
  do {                                \
    if (R == 1) STK_GRP(1, DCV, OCV); \
    else if (R == 2) STK_GRP(2, DCV, OCV); \
    else if (R == 4) STK_GRP(4, DCV, OCV); \
    else STK_GRP(8, DCV, OCV);        \
  } while (0)
  if (w == 64) STK_GRPR(2, 8);
  else if (w == 128) STK_GRPR(4, 16);
  else STK_GRPR(8, 32);
#undef STK_GRPR
#undef STK_GRP
  return true;
}

// the decode form as a model calls it: scratch for `splits` parts, and B * G arrival counters that are zero and are left zero
extern "C" void vra_stack_op_attention_decode(const void* q, int32_t ldq, void* out, const void* kc, const void* vc, const int64_t* positions,
                                              const uint32_t* block_tables, const uint32_t* context_lens, int32_t B, int32_t H, int32_t G, int32_t dim,
                                              int32_t vdim, int32_t BS, int32_t max_blocks, float scale, float softcap, float temp_coef, int32_t temp_every,
                                              int32_t chunk, int32_t window, const float* sink, const float* head_scale, const float* gate, int32_t gate_ld,
                                              float* scratch, int64_t scratch_bytes, int32_t splits, uint32_t* arrived, int32_t dtype, int64_t stream) {
  StkAttnArgs a;
  a.q = q, a.ldq = ldq, a.out = out, a.kc = kc, a.vc = vc, a.positions = positions, a.block_tables = block_tables, a.context_lens = context_lens;
  a.B = B, a.T = B, a.H = H, a.G = G, a.dim = dim, a.vdim = vdim, a.BS = BS, a.max_blocks = max_blocks, a.scale = scale, a.softcap = softcap;
  a.temp_coef = temp_coef, a.temp_every = temp_every, a.chunk = chunk, a.window = window, a.sink = sink, a.head_scale = head_scale, a.gate = gate;
  a.gate_ld = gate_ld, a.scratch = scratch, a.scratch_bytes = (size_t)scratch_bytes, a.splits = splits, a.arrived = arrived;
  vra_stack_attention(a, dtype, stream);
}
