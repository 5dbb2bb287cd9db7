// stack_ops.hip — operators of config-driven layer stacks (host/stack_model.cpp; every operator is specified in stack_launch.h), gfx950.
//
// What is kept in f32 whatever the storage type: positions and angles, norms, router logits and weights, attention scores and
// softmax weights (the value product included: p stays f32, v is widened), the residual stream and every sum into it.
// Matrix products: bf16 operands on v_mfma_f32_16x16x32_bf16 with f32 accumulation, or f32 operands on FMA (VRA_F32: no reduced
// matrix mode anywhere).  Every reduction has an order that depends on the shapes of the model alone — never on the number of rows
// of a step, on a row's place in the batch or on the pages it uses — so a token's result does not depend on how its prompt was cut.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "gemm_rows.cuh"
#include "stack_common.cuh"
#include "stack_launch.h"

namespace {

// a wave's sum by DPP and permlane swaps: a VALU operation per step where a shuffle is an LDS round trip
__device__ __forceinline__ float wave_total(float v) { return vra_xor32_sum(vra_xor16_sum(row16_sum(v))); }

__device__ __forceinline__ float gelu_tanh_(float z) { return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z))); }
__device__ __forceinline__ float gelu_erf_(float z) { return 0.5f * z * (1.f + erff(z * 0.7071067811865476f)); }
// the finished value of a plain product: element-wise activation (epi 2), soft cap
__device__ __forceinline__ float plain_value(const StkGemmArgs& g, float v) {
  if (g.epi == 2) {
    if (g.act == 3) v = gelu_erf_(v);
    else if (g.act == 4) v = v > 0.f ? v * v : 0.f;
    else if (g.act == 5) v = tanhf(v);
    else v = expf(-expf(v));
  }
  if (g.softcap > 0.f) v = g.softcap * tanhf(v / g.softcap);
  return v;
}
// act 0: min(g, L) * sigmoid(act_alpha * min(g, L)) * (clamp(u, +-L) + 1);  act 1: gelu_tanh(g) * u;  act 2: silu(g) * u
__device__ __forceinline__ float gated_pair(float g, float u, float limit, float act_alpha, int act = 0) {
  if (act == 1) return gelu_tanh_(g) * u;
  if (act == 2) return g * sigmoidf_(g) * u;
  if (limit > 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
  }
  return g * sigmoidf_(act_alpha * g) * (u + 1.f);
}

// ------------------------------------------------------------------------------------------------ embedding + positions
// A thread takes both entries of an angle: lanes that alternate between sine and cosine would each wait for the other's.
// N angles at a time: one load and one store for all of them where rows are whole fours of columns (N = 2: 8 bytes of bf16, 16 of f32), and the rows of a long prompt
// (DEPTH) asked for ahead of the first sine.  2048 rows of 2048: 16.0 us one angle after the other, now 12.6; 1500 rows 13.5, 8.9.
template <typename T, int N, int DEPTH>
__global__ __launch_bounds__(256) void stk_embed_sinpos_kernel(const uint32_t* ids, const int64_t* pos, const T* embed, const float* inv_freq, float* x,
                                                               int W, int V) {
  typedef T tvec __attribute__((ext_vector_type(2 * N)));
  typedef float fvec __attribute__((ext_vector_type(N)));
  typedef float ovec __attribute__((ext_vector_type(2 * N)));
  const int t = blockIdx.x;
  uint32_t id = ids[t];
  if (id >= (uint32_t)V) id = 0;
  const float p = (float)pos[t];
  const T* const er = embed + (size_t)id * W;
  float* const xr = x + (size_t)t * W;
  // (few rows: a row's angles over the grid's second dimension, as a thread's sines and cosines one after the other are most of the launch.  8 rows of 2048: 3.4 us, one
  // workgroup a row 6.5)
  const int first = (blockIdx.y * 256 + threadIdx.x) * N, step = 256 * gridDim.y * N, angles = (W + 1) / 2;
  for (int i0 = first; i0 < angles; i0 += step * DEPTH) {
    if constexpr (N == 1) {
      float sn = 0.f, cs = 0.f;
      if (inv_freq) sincosf(p * inv_freq[i0], &sn, &cs);
      xr[2 * i0] = El<T>::ld(er + 2 * i0) + sn;
      if (2 * i0 + 1 < W) xr[2 * i0 + 1] = El<T>::ld(er + 2 * i0 + 1) + cs;
    } else {
      tvec e[DEPTH];
      fvec f[DEPTH];
#pragma unroll
      for (int d = 0; d < DEPTH; d++) {
        const int i = min(i0 + d * step, angles - N);
        e[d] = *(const tvec*)(er + 2 * i);
        f[d] = inv_freq ? *(const fvec*)(inv_freq + i) : (fvec)(0.f);
      }
#pragma unroll
      for (int d = 0; d < DEPTH; d++) {
        const int i = i0 + d * step;
        ovec o;
#pragma unroll
        for (int n = 0; n < N; n++) {
          float sn = 0.f, cs = 0.f;
          if (inv_freq) sincosf(p * f[d][n], &sn, &cs);
          const T pair[2] = {e[d][2 * n], e[d][2 * n + 1]};
          o[2 * n] = El<T>::ld(pair) + sn, o[2 * n + 1] = El<T>::ld(pair + 1) + cs;
        }
        if (i < angles) *(ovec*)(xr + 2 * i) = o;
      }
    }
  }
}

// a fold over the wave's lanes in wave_sum's order, without LDS: after the exchange at distance 8 the values of 16 lanes repeat every 8, so a rotation by 4
// is the exchange at distance 4, and so on
template <class F>
__device__ __forceinline__ float wave_fold(float v, F f) {
  auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  v = f(v, vra_dpp_f<0x128>(v));  // row_ror:8, 4, 2, 1
  v = f(v, vra_dpp_f<0x124>(v));
  v = f(v, vra_dpp_f<0x122>(v));
  return f(v, vra_dpp_f<0x121>(v));
}

// ------------------------------------------------------------------------------------------------ grouped RMS norm (+ router)
// (ROUTER a template parameter and 8 waves a SIMD: a norm that carries the router's registers, or a router with the 74 it would take, leaves room for 6
// waves, and 2048 rows are two rounds of workgroups.  2048 rows, us: norm of 2048 7.6 -> 6.8, of 2051 12.4 -> 9.5; with eight router
// outputs 21.1 -> 19.1, of 1001 17.6 -> 13.3.  The picks by a wave and not by one thread, five outputs of a wave and not four in a round: 1500 rows of
// 2048, 16 outputs and a gate 22.0 -> 15.2; 64 outputs, eight picks 76.6 -> 21.7; 160 outputs 163 -> 74.  A wave's outputs of a round
// counted ahead of the loop over the row, not tested in it: 8 rows of 12288, eight outputs 20.2 -> 15.6.  PARTS a template parameter too, and a row without
// parts asked for ahead of its weights: 1500 rows of 2048 5.64 -> 5.33, the other way about 5.43)
// The final norm takes the last layer's parts and the chosen rows in the same launch (x_out null, rows): behind a sum over all rows and a gather, two launches, 2048 rows of
// 2048, one wanted 20.7 us, so 4.9; a decode step of 8 rows 6.5, 3.9.
template <typename T, bool ROUTER, bool PARTS>
__global__ __launch_bounds__(256, 8) void stk_group_norm_kernel(StkNormArgs a) {
  extern __shared__ float lds[];
  float* xs = lds;                      // [W] the row, then the normalised row
  float* rs = lds + a.W;                // [groups] 1 / rms
  float* zs = rs + a.groups;            // [n_router + gate_row]
  const int t = blockIdx.x, W = a.W, gs = W / a.groups, ts = a.rows ? (int)a.rows[t] : t;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float* x = a.x + (size_t)ts * W;
  T* h = (T*)a.h + (size_t)t * W;
  auto sums = [&] {
    __syncthreads();
    for (int g = wave; g < a.groups; g += 4) {
      float s = 0.f;
      for (int c = lane; c < gs; c += 64) {
        const float v = xs[g * gs + c];
        s = fmaf(v, v, s);
      }
      s = wave_total(s);
      if (lane == 0) rs[g] = 1.f / sqrtf(s / (float)gs + a.eps);
    }
    __syncthreads();
  };
  const float gt = PARTS && a.gate_in ? a.gate_in[ts] : 1.f;
  const bool quads = W % 4 == 0 && gs % 4 == 0 && (((uintptr_t)a.x | (uintptr_t)a.x_out | (uintptr_t)a.o | (uintptr_t)a.p1 | (uintptr_t)a.p2 | (uintptr_t)a.w) % 16) == 0;
  if (quads) {
    // (four values a load where rows and groups allow it, two loads of every part of the row ahead of the first sum: its parts arrive in one round trip
    // instead of one a part, and the row stays in registers: 8 rows of 2048: 6.6 us, now 4.0; 1500 rows of 2048 with two experts' and a shared
    // expert's parts, with the router 29.4, now 22.5)
    constexpr int R = 2;
    f32x4 keep[R], wt[R];
    auto load = [&](int c0, f32x4 (&v)[R]) {  // (values beyond the row: the last ones again, not kept)
      f32x4 s[R], s1[R], s2[R], s3[R];
      int c[R];
#pragma unroll
      for (int n = 0; n < R; n++) c[n] = min(c0 + n * 1024, W - 4);
      auto read = [&](const float* p, f32x4 (&d)[R]) {
#pragma unroll
        for (int n = 0; n < R; n++) d[n] = *(const f32x4*)(p + c[n]);
      };
      auto add = [&](const f32x4 (&d)[R]) {
#pragma unroll
        for (int n = 0; n < R; n++) s[n] += d[n];
      };
      read(x, v);
      const float* const p1 = a.p1 + (size_t)ts * a.n1 * W;
      read(a.o + (size_t)ts * W, s);
      if (a.n1 > 0) read(p1, s1);
      if (a.n1 > 1) read(p1 + W, s2);
      if (a.p2) read(a.p2 + (size_t)ts * W, s3);
      if (a.n1 > 0) add(s1);
      if (a.n1 > 1) add(s2);
      for (int j = 2; j < a.n1; j++) {
        read(p1 + (size_t)j * W, s1);
        add(s1);
      }
      if (a.p2) {
#pragma unroll
        for (int n = 0; n < R; n++) s[n] += gt * s3[n];
      }
#pragma unroll
      for (int n = 0; n < R; n++) v[n] += a.mult * s[n];
#pragma unroll
      for (int n = 0; n < R; n++)
        if (c0 + n * 1024 < W) {
          *(f32x4*)(xs + c0 + n * 1024) = v[n];
          if (a.x_out) *(f32x4*)(a.x_out + (size_t)ts * W + c0 + n * 1024) = v[n];
        }
    };
    auto put = [&](int c, f32x4 v, f32x4 w) {
      const f32x4 y = v * rs[c / gs] * w;
      if (ROUTER) *(f32x4*)(xs + c) = y;
#pragma unroll
      for (int e = 0; e < 4; e++) El<T>::st(h + c + e, y[e]);
    };
    if constexpr (PARTS) {
      for (int c = threadIdx.x * 4 + R * 1024; c < W; c += R * 1024) {
        f32x4 v[R];
        load(c, v);  // (ahead of what stays in registers)
      }
      load(threadIdx.x * 4, keep);
#pragma unroll
      for (int n = 0; n < R; n++) {
        const int c = threadIdx.x * 4 + n * 1024;
        if (c < W) wt[n] = *(const f32x4*)(a.w + c);
      }
    } else {  // (the row alone: its weights with it)
#pragma unroll
      for (int n = 0; n < R; n++) {
        const int c = threadIdx.x * 4 + n * 1024;
        if (c < W) keep[n] = *(const f32x4*)(x + c), wt[n] = *(const f32x4*)(a.w + c);
      }
#pragma unroll
      for (int n = 0; n < R; n++) {
        const int c = threadIdx.x * 4 + n * 1024;
        if (c < W) *(f32x4*)(xs + c) = keep[n];
      }
      for (int c = threadIdx.x * 4 + R * 1024; c < W; c += 1024) *(f32x4*)(xs + c) = *(const f32x4*)(x + c);
    }
    sums();
#pragma unroll
    for (int n = 0; n < R; n++) {
      const int c = threadIdx.x * 4 + n * 1024;
      if (c < W) put(c, keep[n], wt[n]);
    }
    for (int c = threadIdx.x * 4 + R * 1024; c < W; c += 1024) put(c, *(const f32x4*)(xs + c), *(const f32x4*)(a.w + c));
  } else {
    if constexpr (PARTS) {
      for (int c = threadIdx.x; c < W; c += 256) {
        float s = a.o[(size_t)ts * W + c];
        for (int j = 0; j < a.n1; j++) s += a.p1[((size_t)ts * a.n1 + j) * W + c];
        if (a.p2) s += gt * a.p2[(size_t)ts * W + c];
        const float v = x[c] + a.mult * s;
        if (a.x_out) a.x_out[(size_t)ts * W + c] = v;
        xs[c] = v;
      }
    } else {
      for (int c = threadIdx.x; c < W; c += 256) xs[c] = x[c];
    }
    sums();
    for (int c = threadIdx.x; c < W; c += 256) {
      const float v = xs[c] * rs[c / gs] * a.w[c];
      if (ROUTER) xs[c] = v;
      El<T>::st(h + c, v);
    }
  }
  if constexpr (!ROUTER) return;
  __syncthreads();
  const int nz = a.n_router + (a.gate_row ? 1 : 0);
  const T* rw = (const T*)a.router_w;
  if (sizeof(T) == 2 && W % 8 == 0 && ((uintptr_t)rw % 16) == 0) {  // 8 weights a load; the lane's partial sums keep one order for a given W
    auto dots = [&](auto N, int e0) {  // N outputs of a wave side by side: their weights are under way together, the row is read once
      constexpr int Q = decltype(N)::value;
      float s[Q] = {};
      for (int c = lane * 8; c < W; c += 64 * 8) {
        u32x4 v[Q];
#pragma unroll
        for (int q = 0; q < Q; q++) v[q] = *(const u32x4*)((const uint16_t*)rw + (size_t)(e0 + q * 4) * W + c);
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; i++) f[i] = xs[c + i];
#pragma unroll
        for (int q = 0; q < Q; q++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            s[q] = fmaf(f[2 * i], __uint_as_float(v[q][i] << 16), s[q]);
            s[q] = fmaf(f[2 * i + 1], __uint_as_float(v[q][i] & 0xffff0000u), s[q]);
          }
      }
#pragma unroll
      for (int q = 0; q < Q; q++) {
        s[q] = wave_fold(s[q], [](float p, float r) { return p + r; });
        if (lane == 0) zs[e0 + q * 4] = s[q];
      }
    };
    for (int e0 = wave; e0 < nz; e0 += 20) {
      switch (min((nz - e0 + 3) / 4, 5)) {
        case 1: dots(std::integral_constant<int, 1>{}, e0); break;
        case 2: dots(std::integral_constant<int, 2>{}, e0); break;
        case 3: dots(std::integral_constant<int, 3>{}, e0); break;
        case 4: dots(std::integral_constant<int, 4>{}, e0); break;
        default: dots(std::integral_constant<int, 5>{}, e0);
      }
    }
  } else {
    for (int e = wave; e < nz; e += 4) {
      float s = 0.f;
      for (int c = lane; c < W; c += 64) s = fmaf(xs[c], El<T>::ld(rw + (size_t)e * W + c), s);
      s = wave_sum(s);
      if (lane == 0) zs[e] = s;
    }
  }
  __syncthreads();
  if (a.gate_row && threadIdx.x == 255) a.gate_out[t] = sigmoidf_(zs[a.n_router]);
  if (wave != 0) return;
  if (a.n_router <= 4096) {  // the picks, by one wave: the largest of what is left, the first of equal ones; a NaN counts only where it comes first
    constexpr int NONE = 0x7fffffff;
    auto least = [&](int v) -> int {
      if (a.n_router <= 64) return __builtin_ctzll(__ballot(v != NONE));  // (a lane's value is its number)
      return __float_as_int(wave_fold(__int_as_float(v), [](float p, float r) { return __int_as_float(min(__float_as_int(p), __float_as_int(r))); }));
    };
    uint64_t taken = 0;  // bit i: output lane + 64 i
    for (int j = 0; j < a.top; j++) {
      int first = NONE, at = NONE;
      float m = -INFINITY;
      for (int e = lane, i = 0; e < a.n_router; e += 64, i++) {
        if (taken >> i & 1) continue;
        const float z = zs[e];
        first = min(first, e);
        if (z > m || (at == NONE && z == m)) m = z, at = e;
      }
      int best = least(first);
      float bz = zs[best];
      if (!__builtin_isnan(bz)) {
        bz = wave_fold(m, [](float p, float r) { return fmaxf(p, r); });
        best = least(m == bz ? at : NONE);
        bz = zs[best];
      }
      if (lane == (best & 63)) taken |= 1ull << (best >> 6);
      if (lane == 0) a.pair_expert[(size_t)t * a.top + j] = best, a.pair_weight[(size_t)t * a.top + j] = sigmoidf_(bz);
    }
    return;
  }
  // (more outputs: by one thread from LDS; the row is not needed any more, its place holds the marks)
  if (threadIdx.x == 0) {
    int* taken = (int*)xs;
    const bool marks = a.n_router <= W;  // (more outputs than channels: look the earlier picks up)
    if (marks)
      for (int e = 0; e < a.n_router; e++) taken[e] = 0;
    for (int j = 0; j < a.top; j++) {
      int best = -1;
      float bz = -INFINITY;
      for (int e = 0; e < a.n_router; e++) {
        bool skip = marks && taken[e];
        if (!marks)
          for (int q = 0; q < j; q++) skip = skip || a.pair_expert[(size_t)t * a.top + q] == e;
        if (!skip && (best < 0 || zs[e] > bz)) best = e, bz = zs[e];
      }
      if (marks) taken[best] = 1;
      a.pair_expert[(size_t)t * a.top + j] = best;
      a.pair_weight[(size_t)t * a.top + j] = sigmoidf_(bz);
    }
  }
}

// ------------------------------------------------------------------------------------------------ MoE rows sorted by expert
__global__ __launch_bounds__(1024) void stk_moe_sort_kernel(const int* pair_expert, const float* pair_weight, int P, int top, int n_groups, int granule,
                                                            int max_rows, int* row_token, float* row_scale, int* row_pair, int* tile_group) {
  extern __shared__ int sl[];
  int* counts = sl;
  int* offs = sl + n_groups;
  int* cursor = offs + n_groups;
  const int tid = threadIdx.x;
  for (int e = tid; e < n_groups; e += 1024) counts[e] = 0, cursor[e] = 0;
  for (int r = tid; r < max_rows; r += 1024) row_token[r] = -1, row_pair[r] = -1, row_scale[r] = 0.f;
  for (int t = tid; t < max_rows / granule; t += 1024) tile_group[t] = -1;
  __syncthreads();
  for (int p = tid; p < P; p += 1024) {
    const int e = pair_expert[p];
    if (e >= 0 && e < n_groups) atomicAdd(&counts[e], 1);
  }
  __syncthreads();
  if (tid == 0) {
    int off = 0;
    for (int e = 0; e < n_groups; e++) {
      offs[e] = off;
      const int nt = (counts[e] + granule - 1) / granule;
      for (int t = 0; t < nt; t++) tile_group[off / granule + t] = e;
      off += nt * granule;
    }
  }
  __syncthreads();
  for (int p = tid; p < P; p += 1024) {
    const int e = pair_expert[p];
    if (e < 0 || e >= n_groups) continue;
    const int r = offs[e] + atomicAdd(&cursor[e], 1);
    row_token[r] = p / top;
    row_scale[r] = pair_weight[p];
    row_pair[r] = p;
  }
}

// the rows of a mixture's first product, times their weights (bound: HBM, one read and one write of the pairs' rows): 1500 tokens, two experts
// each, width 2048: 6 us; scaled inside the product, that took 192 us where an unscaled one of its size took 111
__global__ __launch_bounds__(256) void stk_scale_rows_kernel(const uint16_t* a, int W, const int* row_token, const float* row_scale, uint16_t* out) {
  const int r = blockIdx.x, t = row_token[r];
  if (t < 0) return;
  const float s = row_scale[r];
  for (int c = threadIdx.x * 8; c < W; c += 256 * 8) {
    float f[8];
    unpack8<BF16>(*(const u32x4*)(a + (size_t)t * W + c), f);
#pragma unroll
    for (int e = 0; e < 8; e++) f[e] *= s;
    *(u32x4*)(out + (size_t)r * W + c) = pack8<BF16>(f);
  }
}

// ------------------------------------------------------------------------------------------------ GEMM, f32 FMA (any shape)
// 256 threads: 16 (m) x 16 (n) threads, RM rows x 4 columns each; K in steps of 16 through LDS; k ascending: one fixed order.  For rows off
// 16 bytes (f32; bf16 where the matrix form does not take the product).
template <typename T, int RM>
__global__ __launch_bounds__(256) void stk_gemm_simple_kernel(StkGemmArgs g) {
  constexpr int TM = 16 * RM;
  __shared__ float As[16][TM + 1];
  __shared__ float Ws[16][65];
  __shared__ int a_idx[TM];
  __shared__ float a_sc[TM];
  const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4;
  const int m0 = blockIdx.x * TM, n0 = blockIdx.y * 64;
  int group = 0;
  if (g.tile_group) {
    group = g.tile_group[blockIdx.x];
    if (group < 0) return;
  }
  const T* A = (const T*)g.a + (int64_t)blockIdx.z * g.a_batch_stride;
  const T* Wt = (const T*)g.w + (int64_t)group * g.w_group_stride + (int64_t)blockIdx.z * g.w_batch_stride;
  const int64_t ob = (int64_t)blockIdx.z * g.out_batch_stride;
  if (tid < TM) {
    const int r = m0 + tid;
    int idx = r < g.M ? (g.a_row ? g.a_row[r] : r) : -1;
    a_idx[tid] = idx;
    a_sc[tid] = g.a_scale && idx >= 0 ? g.a_scale[r] : 1.f;
  }
  __syncthreads();
  float acc[RM][4];
  for (int i = 0; i < RM; i++)
    for (int j = 0; j < 4; j++) acc[i][j] = 0.f;
  for (int k0 = 0; k0 < g.K; k0 += 16) {
    for (int i = tid; i < TM * 16; i += 256) {
      const int r = i >> 4, kk = i & 15, idx = a_idx[r];
      float v = 0.f;
      if (idx >= 0 && k0 + kk < g.K) {
        v = El<T>::ld(A + (int64_t)idx * g.lda + k0 + kk);
        if (g.a_scale) v = El<T>::rnd(v * a_sc[r]);
      }
      As[kk][r] = v;
    }
    for (int i = tid; i < 64 * 16; i += 256) {
      const int n = i >> 4, kk = i & 15;
      Ws[kk][n] = (n0 + n < g.N && k0 + kk < g.K) ? El<T>::ld(Wt + (int64_t)(n0 + n) * g.K + k0 + kk) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; kk++) {
      float av[RM], wv[4];
      for (int i = 0; i < RM; i++) av[i] = As[kk][ty * RM + i];
      for (int j = 0; j < 4; j++) wv[j] = Ws[kk][tx * 4 + j];
      for (int i = 0; i < RM; i++)
        for (int j = 0; j < 4; j++) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
    }
    __syncthreads();
  }
  for (int i = 0; i < RM; i++) {
    const int r = m0 + ty * RM + i;
    if (r >= g.M || a_idx[ty * RM + i] < 0) continue;
    const int orow = g.out_row ? g.out_row[r] : r;
    if (orow < 0) continue;
    for (int j = 0; j < 4; j++) {
      const int n = n0 + tx * 4 + j;
      if (n >= g.N) continue;
      const float v = plain_value(g, acc[i][j] * g.alpha + (g.bias ? g.bias[(int64_t)blockIdx.z * g.bias_batch_stride + n] : 0.f));
      if (g.out_f32) ((float*)g.out)[ob + (int64_t)orow * g.ldo + n] = v;
      else El<T>::st((T*)g.out + ob + (int64_t)orow * g.ldo + n, v);
    }
  }
}

// ------------------------------------------------------------------------------------------------ GEMM, f32 MFMA (16-byte rows)
// A wave is a workgroup and owns MT x NT tiles of 16 x 16 of v_mfma_f32_16x16x4_f32 (weights = A, rows = B: a lane ends with 4 consecutive columns of
// one row).  That instruction adds its four products one after the other, each fused: the bits of the chain above, k ascending.  Lane (r, q) loads 16
// bytes of its row a block of 16 k, P blocks ahead, into registers: no LDS, no barrier; lane swaps, which run under the matrix instructions, then put
// k = 4 s + q where step s reads it.
// Bound: the loads' addresses (16 rows of 64 bytes each, 64 clocks a load for a CU), about half the matrix units' 157 TFLOP/s; few rows, the chain of
// a lone wave.  us, the form above -> this, launch included: 2 rows, 2048 x 2048 198 -> 20, K = 8192 805 -> 61, 32000 columns 326 -> 56;
// 342 rows, 8192 x 2048 479 -> 174; 2048 rows, 1486 -> 915.
template <int MT, int NT, int P, bool SCALED>
__global__ __launch_bounds__(64) void stk_gemm_f32_kernel(StkGemmArgs g) {
  const int lane = threadIdx.x, r16 = lane & 15, q4 = lane >> 4;
  const int m0 = (int)blockIdx.x * 16 * MT, n0 = (int)blockIdx.y * 16 * NT;
  int group = 0;
  if (g.tile_group) {
    group = g.tile_group[m0 / g.granule];
    if (group < 0) return;
  }
  const float* const A = (const float*)g.a + (int64_t)blockIdx.z * g.a_batch_stride;
  const float* const Wt = (const float*)g.w + (int64_t)group * g.w_group_stride + (int64_t)blockIdx.z * g.w_batch_stride;
  const float *xp[MT], *wp[NT];
  float sc[MT];
  int orow[MT];  // -1: nothing to store
#pragma unroll
  for (int i = 0; i < MT; i++) {
    const int row = m0 + i * 16 + r16, idx = row < g.M ? (g.a_row ? g.a_row[row] : row) : -1;
    xp[i] = A + (int64_t)max(idx, 0) * g.lda + q4 * 4;
    sc[i] = SCALED && idx >= 0 ? g.a_scale[row] : 1.f;
    orow[i] = idx < 0 ? -1 : (g.out_row ? g.out_row[row] : row);
  }
#pragma unroll
  for (int j = 0; j < NT; j++) wp[j] = Wt + (int64_t)min(n0 + j * 16 + r16, g.N - 1) * g.K + q4 * 4;
  f32x4 x[P][MT], w[P][NT];
  auto fetch = [&](int off, int u) {
#pragma unroll
    for (int i = 0; i < MT; i++) x[u][i] = *(const f32x4*)(xp[i] + off * 16);
#pragma unroll
    for (int j = 0; j < NT; j++) w[u][j] = *(const f32x4*)(wp[j] + off * 16);
  };
  auto turn = [](f32x4& v) {  // value s of lane (r, q): from value q of lane (r, s)
    float v0 = v[0], v1 = v[1], v2 = v[2], v3 = v[3];
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %2\n\tv_permlane32_swap_b32 %1, %3\n\ts_nop 1\n\t"
                 "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3" : "+v"(v0), "+v"(v1), "+v"(v2), "+v"(v3));
    v = f32x4{v0, v1, v2, v3};
  };
  auto turn_x = [&](int u) {
#pragma unroll
    for (int i = 0; i < MT; i++) {
      if (SCALED) x[u][i] *= sc[i];
      turn(x[u][i]);
    }
  };
  auto turn_w = [&](int u) {
#pragma unroll
    for (int j = 0; j < NT; j++) turn(w[u][j]);
  };
  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int u, int s) {
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++)
        asm volatile("v_mfma_f32_16x16x4_f32 %0, %1, %2, %0" : "+v"(acc[i][j]) : "v"(w[u][j][s]), "v"(x[u][i][s]));
  };
  const int KF = g.K >> 4;  // whole blocks
  int left = KF;
  if (KF >= 2 * P) {
#pragma unroll
    for (int u = 0; u < P; u++) fetch(u, u);
    turn_x(0), turn_w(0);
    asm volatile("s_nop 1");
    do {
#pragma unroll
      for (int u = 0; u < P; u++) {
        step(u, 0);
        turn_x((u + 1) % P);
        step(u, 1);
        turn_w((u + 1) % P);
        step(u, 2);
        step(u, 3);
        fetch(P + u, u);
      }
#pragma unroll
      for (int i = 0; i < MT; i++) xp[i] += P * 16;
#pragma unroll
      for (int j = 0; j < NT; j++) wp[j] += P * 16;
      left -= P;
    } while (left >= 2 * P);
  } else {
#pragma unroll
    for (int u = 0; u < P; u++)
      if (u < KF) fetch(u, u);
    if (KF) turn_x(0), turn_w(0);
  }
#pragma unroll
  for (int u = 0; u < 2 * P; u++) {
    if (u < left) {
      asm volatile("s_nop 1");
#pragma unroll
      for (int s = 0; s < 4; s++) step(u % P, s);
      if (u < P && u + P < left) fetch(P + u, u);
      if (u + 1 < left) turn_x((u + 1) % P), turn_w((u + 1) % P);
    }
  }
  if (g.K & 15) {  // (K % 4 == 0: a lane's four values are inside or beyond K together; zeros add nothing)
    const bool in = KF * 16 + q4 * 4 < g.K;
#pragma unroll
    for (int i = 0; i < MT; i++) x[0][i] = in ? *(const f32x4*)(xp[i] + left * 16) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NT; j++) w[0][j] = in ? *(const f32x4*)(wp[j] + left * 16) : f32x4{0.f, 0.f, 0.f, 0.f};
    turn_x(0), turn_w(0);
    asm volatile("s_nop 1");
#pragma unroll
    for (int s = 0; s < 4; s++) step(0, s);
  }
  VRA_MFMA_DRAIN();
  const int64_t ob = (int64_t)blockIdx.z * g.out_batch_stride;
#pragma unroll
  for (int i = 0; i < MT; i++) {
    if (orow[i] < 0) continue;
    float* const o = (float*)g.out + ob + (int64_t)orow[i] * g.ldo;
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int n = n0 + j * 16 + q4 * 4 + e;
        if (n < g.N) o[n] = plain_value(g, acc[i][j][e] * g.alpha + (g.bias ? g.bias[(int64_t)blockIdx.z * g.bias_batch_stride + n] : 0.f));
      }
  }
}

// ------------------------------------------------------------------------------------------------ GEMM, bf16 MFMA (K % 8 == 0)
// A wave owns MT x NT tiles of 16 x 16; both operands come straight from global memory in the instruction's operand order (lane =
// (row rq = lane & 15, k octet oct = lane >> 4): 16 bytes of one row per lane and K-step of 32), the weights as the A operand and the
// activations as B, so a lane ends up with 4 consecutive output columns of ONE activation row.  K ascending in steps of 32.
// POST: the plain epilogue also applies an activation or a soft cap
template <int MT, int NT, int WM, int WN, bool SCALED, bool POST = false>
__global__ __launch_bounds__(64 * WM * WN) void stk_gemm_mfma_kernel(StkGemmArgs g) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave % WM, wn = wave / WM, rq = lane & 15, oct = lane >> 4;
  int group = 0;
  if (g.tile_group) {
    group = g.tile_group[blockIdx.x];
    if (group < 0) return;
  }
  const uint16_t* A = (const uint16_t*)g.a + (int64_t)blockIdx.z * g.a_batch_stride;
  const uint16_t* Wt = (const uint16_t*)g.w + (int64_t)group * g.w_group_stride + (int64_t)blockIdx.z * g.w_batch_stride;
  const int64_t ob = (int64_t)blockIdx.z * g.out_batch_stride;
  const int m_base = blockIdx.x * (16 * MT * WM) + wm * 16 * MT;
  const int n_base = blockIdx.y * (16 * NT * WN) + wn * 16 * NT;
  const uint16_t* ap[MT];
  const uint16_t* wp[NT];
  bool av[MT], wv[NT];
  float asc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    const int r = m_base + mt * 16 + rq;
    const int idx = r < g.M ? (g.a_row ? g.a_row[r] : r) : -1;
    av[mt] = idx >= 0;
    ap[mt] = A + (int64_t)(idx >= 0 ? idx : 0) * g.lda;
    asc[mt] = SCALED && idx >= 0 ? g.a_scale[r] : 1.f;
  }
#pragma unroll
  for (int nt = 0; nt < NT; nt++) {
    const int n = n_base + nt * 16 + rq;
    wv[nt] = n < g.N;
    wp[nt] = Wt + (int64_t)(n < g.N ? n : 0) * g.K;
  }
  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int nt = 0; nt < NT; nt++) acc[mt][nt] = vra_zero_acc();
  const u32x4 zero4 = {0u, 0u, 0u, 0u};
  // the fragments of K-step k + 1 are requested before the MFMAs of step k run
  u32x4 af[MT], wf[NT], afn[MT], wfn[NT];
  auto request = [&](int k0, u32x4* ao, u32x4* wo) {
    const int k = k0 + oct * 8;
    const bool kin = k < g.K;
    const int kc = kin ? k : 0;
  #pragma unroll
  for (int mt = 0; mt < MT; mt++) {
      u32x4 v = *(const u32x4*)(ap[mt] + kc);
      if (SCALED) {
        const float s = asc[mt];
        for (int i = 0; i < 4; i++) {
          const float lo = __uint_as_float(v[i] << 16) * s, hi = __uint_as_float(v[i] & 0xffff0000u) * s;
          v[i] = BF16::pack2(lo, hi);
        }
      }
      ao[mt] = (av[mt] && kin) ? v : zero4;
    }
  #pragma unroll
  for (int nt = 0; nt < NT; nt++) {
      const u32x4 v = *(const u32x4*)(wp[nt] + kc);
      wo[nt] = (wv[nt] && kin) ? v : zero4;
    }
  };
  request(0, afn, wfn);
  for (int k0 = 0; k0 < g.K; k0 += 32) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++) af[mt] = afn[mt];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) wf[nt] = wfn[nt];
    request(k0 + 32, afn, wfn);  // (beyond K: loads from offset 0, counted as zeros)
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++) BF16::mfma(acc[mt][nt], __builtin_bit_cast(s16x8, wf[nt]), __builtin_bit_cast(s16x8, af[mt]));
  }
  VRA_MFMA_DRAIN();
  // lane: activation row rq of tile mt, output columns oct * 4 + j of tile nt
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    const int r = m_base + mt * 16 + rq;
    if (r >= g.M || !av[mt]) continue;
    const int orow = g.out_row ? g.out_row[r] : r;
    if (orow < 0) continue;
    if (g.epi == 1) {
#pragma unroll
      for (int nt = 0; nt + 1 < NT; nt += 2)
        for (int j = 0; j < 4; j++) {
          const int n = (n_base + nt * 16) / 2 + oct * 4 + j;
          if (n >= g.N / 2) continue;
          const float y = gated_pair(acc[mt][nt][j], acc[mt][nt + 1][j], g.limit, g.act_alpha, g.act);
          if (g.out_f32) ((float*)g.out)[ob + (int64_t)orow * g.ldo + n] = y;
          else ((uint16_t*)g.out)[ob + (int64_t)orow * g.ldo + n] = BF16::from_f32(y);
        }
    } else {
#pragma unroll
      for (int nt = 0; nt < NT; nt++)
        for (int j = 0; j < 4; j++) {
          const int n = n_base + nt * 16 + oct * 4 + j;
          if (n >= g.N) continue;
          float v = acc[mt][nt][j] * g.alpha + (g.bias ? g.bias[(int64_t)blockIdx.z * g.bias_batch_stride + n] : 0.f);
          if (POST) v = plain_value(g, v);
          if (g.out_f32) ((float*)g.out)[ob + (int64_t)orow * g.ldo + n] = v;
          else ((uint16_t*)g.out)[ob + (int64_t)orow * g.ldo + n] = BF16::from_f32(v);
        }
    }
  }
}

// where a bf16 product with cache columns (StkGemmArgs::kv_slot) stores column n of its row (null: nowhere)
__device__ __forceinline__ uint16_t* kv_place(uint16_t* row, int64_t slot, void* kc, void* vc, int from, int k, int N, int n) {
  if (n < from) return row + n;
  if (slot < 0) return nullptr;
  return n < from + k ? (uint16_t*)kc + slot * k + (n - from) : (uint16_t*)vc + slot * (N - from - k) + (n - from - k);
}

// Steps of up to 32 rows (decoding): the weights are the whole traffic, and what bounds it is the CUs that pull at them.  A
// workgroup takes 16 * NT output columns and its 8 waves take an eighth of K each (whole K-steps of 32, ascending inside a wave); the partial
// tiles meet in LDS and are summed in wave order.  One fixed order for a given K — another one than the large-M kernel's single chain, so the
// two agree to rounding, not to the bit.
// MORE: cache columns or a second output, whose places the plain form does not ask for (with both in one kernel its loop had fewer loads in flight: see STK_SMALL).
template <bool SCALED, bool POST, int NT, bool MORE = false>
__global__ __launch_bounds__(512) void stk_gemm_mfma_small_kernel(StkGemmArgs g) {
  constexpr int BN = 16 * NT, NW = 8;
  __shared__ float part[NW][16 * BN];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, rq = lane & 15, oct = lane >> 4;
  int group = 0;
  if (g.tile_group) {
    group = g.tile_group[blockIdx.x];
    if (group < 0) return;
  }
  const uint16_t* A = (const uint16_t*)g.a + (int64_t)blockIdx.z * g.a_batch_stride;
  const uint16_t* Wt = (const uint16_t*)g.w + (int64_t)group * g.w_group_stride + (int64_t)blockIdx.z * g.w_batch_stride;
  const int64_t ob = (int64_t)blockIdx.z * g.out_batch_stride;
  const int m_base = blockIdx.x * 16, n_base = blockIdx.y * BN;
  const int r = m_base + rq;
  const int idx = r < g.M ? (g.a_row ? g.a_row[r] : r) : -1;
  const uint16_t* ap = A + (int64_t)(idx >= 0 ? idx : 0) * g.lda;
  const float asc = SCALED && idx >= 0 ? g.a_scale[r] : 1.f;
  const uint16_t* wp[NT];
  bool wv[NT];
#pragma unroll
  for (int nt = 0; nt < NT; nt++) {
    const int n = n_base + nt * 16 + rq;
    wv[nt] = n < g.N;
    wp[nt] = Wt + (int64_t)(n < g.N ? n : 0) * g.K;
  }
  const int ksteps = (g.K + 31) / 32, per = (ksteps + NW - 1) / NW;
  const int k_lo = wave * per * 32, k_hi = min(g.K, (wave + 1) * per * 32);
  f32x4 acc[NT];
#pragma unroll
  for (int nt = 0; nt < NT; nt++) acc[nt] = vra_zero_acc();
  const u32x4 zero4 = {0u, 0u, 0u, 0u};
  // four K-steps per round: their 16-byte requests are in flight together, then the MFMAs (steps beyond the wave's range load from offset 0 and
  // count as zeros: same order of the sum, no branch between the MFMAs).  Eight at a time, the next round ahead of the MFMAs, or 16 waves
  // are slower at every size (2048 columns, K = 8192: 15.0 us; 16.5, 15.8 and 15.3).
  for (int k0 = k_lo; k0 < k_hi; k0 += 4 * 32) {
    u32x4 af[4], wf[4][NT];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int k = k0 + u * 32 + oct * 8;
      const bool kin = k < k_hi;
      const int kc = kin ? k : 0;
      u32x4 a4 = *(const u32x4*)(ap + kc);
      if (SCALED) {
        for (int i = 0; i < 4; i++) a4[i] = BF16::pack2(__uint_as_float(a4[i] << 16) * asc, __uint_as_float(a4[i] & 0xffff0000u) * asc);
      }
      af[u] = (idx >= 0 && kin) ? a4 : zero4;
#pragma unroll
      for (int nt = 0; nt < NT; nt++) {
        const u32x4 v = *(const u32x4*)(wp[nt] + kc);
        wf[u][nt] = (wv[nt] && kin) ? v : zero4;
      }
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int nt = 0; nt < NT; nt++) BF16::mfma(acc[nt], __builtin_bit_cast(s16x8, wf[u][nt]), __builtin_bit_cast(s16x8, af[u]));
  }
  VRA_MFMA_DRAIN();
#pragma unroll
  for (int nt = 0; nt < NT; nt++)
#pragma unroll
    for (int j = 0; j < 4; j++) part[wave][rq * BN + nt * 16 + oct * 4 + j] = acc[nt][j];
  __syncthreads();
  const int e = threadIdx.x, m = e / BN, c = e % BN;  // one output element per thread
  if (e >= 16 * BN) return;
  const int row = m_base + m;
  if (row >= g.M) return;
  const int ridx = g.a_row ? g.a_row[row] : row;
  if (ridx < 0) return;
  const int orow = g.out_row ? g.out_row[row] : row;
  if (orow < 0) return;
  auto total = [&](int col) {
    float s = part[0][m * BN + col];
#pragma unroll
    for (int w = 1; w < NW; w++) s += part[w][m * BN + col];
    return s;
  };
  if (NT == 2 && g.epi == 1) {
    if (c >= 16) return;
    const int n = n_base / 2 + c;
    if (n >= g.N / 2) return;
    const float y = gated_pair(total(c), total(16 + c), g.limit, g.act_alpha, g.act);
    if (g.out_f32) ((float*)g.out)[ob + (int64_t)orow * g.ldo + n] = y;
    else ((uint16_t*)g.out)[ob + (int64_t)orow * g.ldo + n] = BF16::from_f32(y);
  } else {
    const int n = n_base + c;
    if (n >= g.N) return;
    float v = total(c) * g.alpha + (g.bias ? g.bias[(int64_t)blockIdx.z * g.bias_batch_stride + n] : 0.f);
    if (POST) v = plain_value(g, v);
    if (MORE && !POST && g.kv_slot) {
      if (uint16_t* const p = kv_place((uint16_t*)g.out + (int64_t)row * g.ldo, n < g.kv_from ? 0 : g.kv_slot[row], g.kv_kc, g.kv_vc, g.kv_from, g.kv_k, g.N, n)) *p = BF16::from_f32(v);
    } else if (g.out_f32) {
      if (MORE && g.mirror) g.mirror[(int64_t)orow * g.ldo + n] = v;
      ((float*)g.out)[ob + (int64_t)orow * g.ldo + n] = v;
    } else ((uint16_t*)g.out)[ob + (int64_t)orow * g.ldo + n] = BF16::from_f32(v);
  }
}

// Products of up to 8 rows over columns that sixteen a workgroup would leave on half of the chip or less: eight a workgroup, with the sums of the kernel
// above to the bit.  A load's sixteen weight rows are the eight columns at an even K-step and at the odd one behind it, its sixteen activation rows the same
// two steps of the eight rows: every lane loads, whole 128-byte lines, and half as many of either.  The first eight rows and columns of a tile
// count: the even step as loaded, the odd one with the halves of the lanes' rows of sixteen traded.  What bounds it is what a CU pulls past L2 and the latency
// of its rounds.  8 rows, us, sixteen columns / eight: 2048 columns, K = 2048 6.7 / 5.6, 5632 11.8 / 8.6, 8192 14.8 / 10.4 (one row 11.8 / 8.4); 1024
// columns, K = 8192 14.4 / 9.9.  Beyond one workgroup a CU it gives nothing: 3072 columns, K = 2048 6.9 / 6.9; 4096, K = 4096 9.5 / 10.0, 14336 25.4 / 29.4.
template <bool POST, bool MORE = false>
__global__ __launch_bounds__(512) void stk_gemm_mfma_eight_kernel(StkGemmArgs g) {
  constexpr int NW = 8, U = 2;  // steps of 64 a round, the next round's loads ahead of this one's MFMAs (without: 12.8 us at 2048 x 8192)
  __shared__ float part[NW][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c8 = lane & 7, odd = (lane >> 3) & 1, oct = lane >> 4;
  const uint16_t* A = (const uint16_t*)g.a + (int64_t)blockIdx.z * g.a_batch_stride;
  const uint16_t* Wt = (const uint16_t*)g.w + (int64_t)blockIdx.z * g.w_batch_stride;
  const int n_base = blockIdx.y * 8;
  const int idx = c8 < g.M ? (g.a_row ? g.a_row[c8] : c8) : -1;
  const bool wv = n_base + c8 < g.N;
  const uint16_t* ap = A + (int64_t)(idx >= 0 ? idx : 0) * g.lda;
  const uint16_t* wp = Wt + (int64_t)(wv ? n_base + c8 : 0) * g.K;
  const int ksteps = (g.K + 31) / 32, per = (ksteps + NW - 1) / NW;
  const int k_lo = wave * per * 32, k_hi = min(g.K, (wave + 1) * per * 32);
  f32x4 acc = vra_zero_acc();
  auto traded = [](u32x4 v) {
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = __builtin_amdgcn_mov_dpp((int)v[i], 0x128, 0xf, 0xf, true);  // row_ror:8
    return __builtin_bit_cast(s16x8, v);
  };
  const u32x4 zero4 = {0u, 0u, 0u, 0u};
  u32x4 af[2][U], wf[2][U];
  auto ask = [&](int b, int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = k0 + u * 64 + odd * 32 + oct * 8, kc = k < k_hi ? k : 0;
      wf[b][u] = *(const u32x4*)(wp + kc);
      af[b][u] = *(const u32x4*)(ap + kc);
    }
  };
  auto use = [&](int b, int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const bool kin = k0 + u * 64 + odd * 32 + oct * 8 < k_hi;
      const u32x4 w4 = wv && kin ? wf[b][u] : zero4, a4 = idx >= 0 && kin ? af[b][u] : zero4;
      BF16::mfma(acc, __builtin_bit_cast(s16x8, w4), __builtin_bit_cast(s16x8, a4));
      BF16::mfma(acc, traded(w4), traded(a4));
    }
  };
  if (k_lo < k_hi) ask(0, k_lo);
  for (int k0 = k_lo; k0 < k_hi; k0 += U * 128) {
    if (k0 + U * 64 < k_hi) ask(1, k0 + U * 64);
    use(0, k0);
    if (k0 + U * 64 >= k_hi) break;
    if (k0 + U * 128 < k_hi) ask(0, k0 + U * 128);
    use(1, k0 + U * 64);
  }
  VRA_MFMA_DRAIN();
  // lane: activation row lane % 16, columns oct * 4 + j
  if (oct < 2 && !odd)
#pragma unroll
    for (int j = 0; j < 4; j++) part[wave][c8 * 8 + oct * 4 + j] = acc[j];
  __syncthreads();
  const int e = threadIdx.x, row = e >> 3, n = n_base + (e & 7);  // one output element per thread
  if (e >= 64 || row >= g.M || n >= g.N) return;
  if (g.a_row && g.a_row[row] < 0) return;
  const int orow = g.out_row ? g.out_row[row] : row;
  if (orow < 0) return;
  float v = part[0][e];
#pragma unroll
  for (int w = 1; w < NW; w++) v += part[w][e];
  v = v * g.alpha + (g.bias ? g.bias[(int64_t)blockIdx.z * g.bias_batch_stride + n] : 0.f);
  if (POST) v = plain_value(g, v);
  const int64_t at = (int64_t)blockIdx.z * g.out_batch_stride + (int64_t)orow * g.ldo + n;
  if (MORE && !POST && g.kv_slot) {
    if (uint16_t* const p = kv_place((uint16_t*)g.out + (int64_t)row * g.ldo, n < g.kv_from ? 0 : g.kv_slot[row], g.kv_kc, g.kv_vc, g.kv_from, g.kv_k, g.N, n)) *p = BF16::from_f32(v);
  } else if (g.out_f32) {
    if (MORE && g.mirror) g.mirror[(int64_t)orow * g.ldo + n] = v;
    ((float*)g.out)[at] = v;
  } else ((uint16_t*)g.out)[at] = BF16::from_f32(v);
}

// Epilogue of gemm_rows_kernel for these products: alpha, bias, FN, row scatter.  FN as a template parameter: with all functions in one epilogue
// the kernel is 28 000 instructions long and a launch pays ~12 us for fetching what it jumps over (2048 x 2048 x 2048: 37 us, 24 so).
// vec: rows of the output start on 16 bytes, a lane stores whole 16-byte pieces (bf16: after trading columns with its row's other
// three lanes).
enum StkFn { FN_NONE, FN_KV, FN_PAIR_CLAMPED, FN_PAIR_GELU, FN_PAIR_SILU, FN_GELU, FN_RELU2, FN_TANH, FN_EXPEXP, FN_SOFTCAP };
// the epilogues that gemm_rows_mixed_kernel is built with: q | k | v, o, up, down and the clamped pairs, whose prompts were measured on it.  The others were not measured
// there; they have the single tiles
static constexpr bool stk_mixes(int fn) { return fn == FN_NONE || fn == FN_KV || fn == FN_PAIR_CLAMPED; }
template <int FN>
struct StkRowsEpi {
  void* out;
  const int* out_row;
  const float* bias;
  int64_t out_batch_stride, bias_batch_stride;
  float alpha, limit, act_alpha, softcap;
  int ldo, out_f32, vec, form;
  const int64_t* kv_slot;  // FN_KV
  void *kc, *vc;
  int kv_from, kv_k;
  static constexpr bool pair = FN == FN_PAIR_CLAMPED || FN == FN_PAIR_GELU || FN == FN_PAIR_SILU;
  __device__ __forceinline__ float fn(float v) const {
    if (FN == FN_GELU) return gelu_erf_(v);
    if (FN == FN_RELU2) return v > 0.f ? v * v : 0.f;
    if (FN == FN_TANH) return tanhf(v);
    if (FN == FN_EXPEXP) return expf(-expf(v));
    if (FN == FN_SOFTCAP) return softcap * tanhf(v / softcap);
    return v;
  }
  static constexpr bool mixes = stk_mixes(FN);  // (with gemm_rows_mixed_kernel)
  struct None {};
  typedef std::conditional_t<FN == FN_KV, int64_t, None> Row;
  __device__ __forceinline__ Row row(int m) const {
    if constexpr (FN == FN_KV) return kv_slot[m];
    else return {};
  }
  // form: rows as they lie, no bias, whole 16-byte pieces, bf16 (1) or f32 (2); everything else (0).  (Clamped pairs of 3300 x 14336, K = 4096, the tests at each of a wave's
  // blocks of 16 rows / once: 297 / 293 us.)  The lane's 16 bias values are loaded once for all its rows (2048 x 8192, K = 2048, us, at each block / once: f32 60.9 / 59.9, bf16 57.7 /
  // 55.5; 4096 x 3072, K = 1024, exp(-exp) 41.5 / 39.1)
  struct Bias {
    float b[4][4];
  };
  template <class F>
  __device__ __forceinline__ void in_form(int n0, int N, int q4, const F& f) const {
    if (form == 2) f(std::integral_constant<int, 2>{}, None{});
    else if (form == 1) f(std::integral_constant<int, 1>{}, None{});
    else if constexpr (pair) f(std::integral_constant<int, 0>{}, None{});
    else {
      Bias c = {};
      if (bias) {
        const float* const b = bias + (int64_t)blockIdx.y * bias_batch_stride;
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int e = 0; e < 4; e++) c.b[j][e] = b[min(n0 + j * 16 + q4 * 4 + e, N - 1)];
      }
      f(std::integral_constant<int, 0>{}, c);
    }
  }
  template <int FORM, class COLUMNS>
  __device__ __forceinline__ void store(int m, const Row& slot, const COLUMNS& columns, int, int n0, int N, int q4, const f32x4 (&acc)[4]) const {
    constexpr int NJ = pair ? 2 : 4;  // blocks of 16 output columns
    const int orow = m < 0 ? -1 : (FORM == 0 && out_row ? out_row[m] : m);
    const int64_t ob = (int64_t)blockIdx.y * out_batch_stride + (int64_t)max(orow, 0) * ldo;
    float* const of = (float*)out + ob;
    uint16_t* const oh = (uint16_t*)out + ob;
    const int no = pair ? n0 / 2 : n0, lim = pair ? N / 2 : N;
    float y[NJ][4];
    if constexpr (pair) {
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) y[j][e] = gated_pair(acc[2 * j][e], acc[2 * j + 1][e], limit, act_alpha, FN == FN_PAIR_GELU ? 1 : (FN == FN_PAIR_SILU ? 2 : 0));
    } else {
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          float b = 0.f;  // (added without a bias, too: -0 becomes 0)
          if constexpr (FORM == 0) b = columns.b[j][e];
          y[j][e] = acc[j][e] * alpha + b;
        }
#pragma unroll
      for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) y[j][e] = fn(y[j][e]);
    }
    if (FORM == 1 || (FORM == 0 && vec && !out_f32)) {
      u32x2 v[NJ];
#pragma unroll
      for (int j = 0; j < NJ; j++) v[j] = u32x2{BF16::pack2(y[j][0], y[j][1]), BF16::pack2(y[j][2], y[j][3])};
      gr_gather_columns(v);
#pragma unroll
      for (int h = 0; h < NJ / 2; h++) {
        const int n = no + q4 * (NJ * 4) + h * 8;
        uint16_t* p = orow >= 0 && n < lim ? oh + n : nullptr;
        if constexpr (FN == FN_KV)
          if (p) p = kv_place(oh, slot, kc, vc, kv_from, kv_k, N, n);  // (whole pieces: the launcher's condition)
        if (p) *(u32x4*)p = u32x4{v[2 * h][0], v[2 * h][1], v[2 * h + 1][0], v[2 * h + 1][1]};
      }
      return;
    }
    if (FORM == 2 || (FORM == 0 && vec && out_f32 && lim % 4 == 0)) {
      // The stores of the sixteen rows before are through ahead of these: waves that run ahead of each other write too many rows at a time (2048 x 8192, K = 512 / 2048
      // 27.8 / 62.3 us without the wait, 25.2 / 60.2 so; with a bias 4096 x 8192, K = 2048 117.4 / 114.9)
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        if (orow >= 0 && no + j * 16 + q4 * 4 < lim) *(f32x4*)(of + no + j * 16 + q4 * 4) = f32x4{y[j][0], y[j][1], y[j][2], y[j][3]};
        __builtin_amdgcn_sched_barrier(0);
      }
      return;
    }
    if (orow < 0) return;
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      const int n = no + j * 16 + q4 * 4;
      if (vec && n + 4 <= lim) {
        *(f32x4*)(of + n) = f32x4{y[j][0], y[j][1], y[j][2], y[j][3]};
        continue;
      }
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (n + e < lim) {
          if (out_f32) of[n + e] = y[j][e];
          else oh[n + e] = BF16::from_f32(y[j][e]);
        }
    }
  }
};

// ------------------------------------------------------------------------------------------------ activations
template <typename T>
__global__ __launch_bounds__(256) void stk_gated_act_kernel(const float* gu, T* out, int F, float limit, float act_alpha, int act) {
  const int m = blockIdx.x;
  const int Fp = (F + 15) / 16 * 16;
  for (int f = threadIdx.x; f < F; f += 256) {
    const int b = f >> 4, i = f & 15;
    const float gv = gu[(size_t)m * 2 * Fp + (2 * b) * 16 + i], uv = gu[(size_t)m * 2 * Fp + (2 * b + 1) * 16 + i];
    El<T>::st(out + (size_t)m * Fp + f, gated_pair(gv, uv, limit, act_alpha, act));
  }
  for (int f = F + threadIdx.x; f < Fp; f += 256) El<T>::st(out + (size_t)m * Fp + f, 0.f);
}

#define STK_PN_THREADS 1024
// one workgroup of 1024 threads per token (bound: HBM, z read and the activation written once): 8 values a thread stay in registers between the
// sums and the output — two loads of four where rows start on 16 bytes — and the three sums meet behind one barrier.  2048 tokens x 8192: 35 us
// with single values and a pair of barriers per sum, now 21
template <typename T, int N>
__global__ __launch_bounds__(STK_PN_THREADS) void stk_polynorm_kernel(const float* z, T* out, const float* coef, int F, float eps) {
  typedef float vec __attribute__((ext_vector_type(N)));
  constexpr int R = 8 / N, STEP = STK_PN_THREADS * N;
  __shared__ float red[3][STK_PN_THREADS / 64];
  const int m = blockIdx.x;
  const float* zr = z + (size_t)m * F;
  const float ca = coef[0], cb = coef[1], cc = coef[2], ce = coef[3];
  vec keep[R];
  float s1 = 0.f, s2 = 0.f, s3 = 0.f;
  auto add = [&](vec x) {
#pragma unroll
    for (int e = 0; e < N; e++) {
      const float v = x[e], v2 = v * v, v3 = v2 * v;
      s1 = fmaf(v, v, s1), s2 = fmaf(v2, v2, s2), s3 = fmaf(v3, v3, s3);
    }
  };
#pragma unroll
  for (int n = 0; n < R; n++) {
    const int f = threadIdx.x * N + n * STEP;
    keep[n] = f < F ? *(const vec*)(zr + f) : (vec)(0.f);
  }
#pragma unroll
  for (int n = 0; n < R; n++) add(keep[n]);
  for (int f = threadIdx.x * N + R * STEP; f < F; f += STEP) add(*(const vec*)(zr + f));
  s1 = wave_total(s1), s2 = wave_total(s2), s3 = wave_total(s3);
  if ((threadIdx.x & 63) == 0) red[0][threadIdx.x >> 6] = s1, red[1][threadIdx.x >> 6] = s2, red[2][threadIdx.x >> 6] = s3;
  __syncthreads();
  s1 = s2 = s3 = 0.f;
  for (int w = 0; w < STK_PN_THREADS / 64; w++) s1 += red[0][w], s2 += red[1][w], s3 += red[2][w];
  const float r1 = 1.f / sqrtf(s1 / (float)F + eps), r2 = 1.f / sqrtf(s2 / (float)F + eps), r3 = 1.f / sqrtf(s3 / (float)F + eps);
  auto put = [&](int f, vec x) {
    float y[N];
#pragma unroll
    for (int e = 0; e < N; e++) {
      const float v = x[e], v2 = v * v, v3 = v2 * v;
      y[e] = ca * (v * r1) + cb * (v2 * r2) + cc * (v3 * r3) + ce;
    }
    T* const o = out + (size_t)m * F + f;
    if constexpr (N == 4 && sizeof(T) == 2) {
      *(u32x2*)o = u32x2{BF16::pack2(y[0], y[1]), BF16::pack2(y[2], y[3])};
    } else if constexpr (N == 4) {
      *(f32x4*)o = f32x4{y[0], y[1], y[2], y[3]};
    } else {
      El<T>::st(o, y[0]);
    }
  };
#pragma unroll
  for (int n = 0; n < R; n++) {
    const int f = threadIdx.x * N + n * STEP;
    if (f < F) put(f, keep[n]);
  }
  for (int f = threadIdx.x * N + R * STEP; f < F; f += STEP) put(f, *(const vec*)(zr + f));
}

__global__ __launch_bounds__(256) void stk_residual_combine_kernel(float* x, const float* o, const float* p1, int n1, const float* p2, const float* gate,
                                                                   float mult, int W, int quads) {
  const int t = blockIdx.x;
  const float gt = gate ? gate[t] : 1.f;
  auto row = [&](auto width) {
    constexpr int N = decltype(width)::value;
    typedef float vec __attribute__((ext_vector_type(N)));
    for (int c = threadIdx.x * N; c < W; c += 256 * N) {
      vec s = 0.f;
      if (o) s = *(const vec*)(o + (size_t)t * W + c);
      for (int j = 0; j < n1; j++) s += *(const vec*)(p1 + ((size_t)t * n1 + j) * W + c);
      if (p2) s += gt * *(const vec*)(p2 + (size_t)t * W + c);
      *(vec*)(x + (size_t)t * W + c) += mult * s;
    }
  };
  if (quads) row(std::integral_constant<int, 4>{});
  else row(std::integral_constant<int, 1>{});
}

__global__ __launch_bounds__(256) void stk_gather_rows_kernel(const float* src, const uint32_t* rows, float* dst, int W) {
  const int r = blockIdx.x;
  const float* s = src + (size_t)rows[r] * W;
  for (int c = threadIdx.x; c < W; c += 256) dst[(size_t)r * W + c] = s[c];
}

// ------------------------------------------------------------------------------------------------ paged KV cache
template <typename T>
__global__ __launch_bounds__(256) void stk_kv_store_kernel(const T* k, const T* v, int ld, T* kc, T* vc, const int64_t* slots, int kdim, int vdim) {
  const int t = blockIdx.x;
  const int64_t s = slots[t];
  if (s < 0) return;
  for (int c = threadIdx.x; c < kdim; c += 256) kc[s * kdim + c] = k[(size_t)t * ld + c];
  for (int c = threadIdx.x; c < vdim; c += 256) vc[s * vdim + c] = v[(size_t)t * ld + c];
}

__device__ __forceinline__ float q_temperature(int64_t p, float coef, int every) {
  if (every <= 0 || coef == 0.f) return 1.f;
  return 1.f + coef * logf((float)((p + 1) / every) + 1.f);
}
__device__ __forceinline__ float cap_score(float s, float softcap) { return softcap > 0.f ? softcap * tanhf(s / softcap) : s; }
// the same through the hardware exponential (f32 arithmetic, ~2^-21 relative in the exponential; |error| of the capped score below
// 2^-22 * softcap): the bf16 kernel's choice, where 16 library calls per lane and key tile would cost more than its matrix products
__device__ __forceinline__ float cap_score_fast(float s, float softcap) {
  if (!(softcap > 0.f)) return s;
  const float x = fminf(fmaxf(s / softcap, -15.f), 15.f);
  return softcap * (1.f - 2.f / (1.f + __expf(2.f * x)));
}

// Portions of prompts (and whatever else shares their step): 16 query rows of one head per workgroup, 4 per wave; key tiles of KT
// tokens staged once in LDS (f32) for all 16 rows; lane = key for the scores, lane = value channel for the weighted sum.
// Tiles start at key 0 of the sequence and a row's running maximum / sum go tile by tile: the order does not depend on the portion.
// MAPS 2: the differential form of StkAttnArgs (a query row and a key row hold two maps; both weigh the same staged values).
#define STK_QT 16
template <typename T, int KT, int NR, int MAPS>
__global__ __launch_bounds__(256) void stk_attn_prefill_kernel(StkAttnArgs a) {
  extern __shared__ float lds[];
  const int dim = a.dim, vdim = a.vdim, dm = MAPS * dim, kld = dm + 1;
  float* qs = lds;                      // [16][dm]  q * temp
  float* ks = qs + STK_QT * dm;         // [KT][dm + 1]
  float* vs = ks + KT * kld;            // [KT][vdim]
  float* ps = vs + KT * vdim;           // [MAPS][16][KT]
  const int b = blockIdx.y, h = blockIdx.z, g = h / (a.H / a.G);
  const int q0 = a.cu_q[b], q1 = a.cu_q[b + 1];
  const int t0 = q0 + blockIdx.x * STK_QT;
  if (t0 >= q1) return;
  const int nq = min(STK_QT, q1 - t0);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const T* q = (const T*)a.q;
  for (int i = tid; i < STK_QT * dm; i += 256) {
    const int r = i / dm, d = i % dm;
    float v = 0.f;
    if (r < nq) v = El<T>::ld(q + (size_t)(t0 + r) * a.ldq + h * dm + d) * q_temperature(a.positions[t0 + r], a.temp_coef, a.temp_every);
    qs[i] = v;
  }
  int64_t pq[4], plo[4];
  int64_t pmax = -1, lo_min = INT64_MAX;
  auto block_start = [&](int64_t p) {  // first key a query at p may see
    const int64_t lo = a.chunk > 0 ? p / a.chunk * a.chunk : (int64_t)0;
    return a.window > 0 ? max(lo, p - a.window + 1) : lo;
  };
  for (int i = 0; i < 4; i++) {
    const int r = wave * 4 + i;
    pq[i] = r < nq ? a.positions[t0 + r] : -1;
    plo[i] = pq[i] >= 0 ? block_start(pq[i]) : 0;
  }
  for (int r = 0; r < nq; r++) pmax = max(pmax, a.positions[t0 + r]), lo_min = min(lo_min, block_start(a.positions[t0 + r]));
  const int n_keys = (int)min((int64_t)a.context_lens[b], pmax + 1);
  const int kt_begin = (int)(lo_min / KT) * KT;  // (tiles stay aligned to absolute positions)
  float m[MAPS][4], l[MAPS][4], acc[MAPS][4][NR];
  for (int mp = 0; mp < MAPS; mp++)
    for (int i = 0; i < 4; i++) {
      m[mp][i] = -INFINITY, l[mp][i] = 0.f;
      if (a.sink) m[mp][i] = a.sink[h], l[mp][i] = 1.f;  // the sink: one more term exp(sink - m) of the denominator, present from the start
      for (int r = 0; r < NR; r++) acc[mp][i][r] = 0.f;
    }
  const T* kc = (const T*)a.kc;
  const T* vc = (const T*)a.vc;
  const uint32_t* bt = a.block_tables + (size_t)b * a.max_blocks;
  const int kdim = a.k_ld ? a.k_ld : a.G * dm, vd_all = a.v_ld ? a.v_ld : a.G * vdim;
  const float hscale = a.head_scale ? a.scale * a.head_scale[h] : a.scale;
  for (int kt0 = kt_begin; kt0 < n_keys; kt0 += KT) {
    __syncthreads();
    for (int i = tid; i < KT * dm; i += 256) {
      const int j = i / dm, d = i % dm, key = kt0 + j;
      float v = 0.f;
      if (key < n_keys) {
        const int64_t slot = (int64_t)bt[key / a.BS] * a.BS + key % a.BS;
        v = El<T>::ld(kc + slot * kdim + g * dm + d);
      }
      ks[j * kld + d] = v;
    }
    for (int i = tid; i < KT * vdim; i += 256) {
      const int j = i / vdim, d = i % vdim, key = kt0 + j;
      float v = 0.f;
      if (key < n_keys) {
        const int64_t slot = (int64_t)bt[key / a.BS] * a.BS + key % a.BS;
        v = El<T>::ld(vc + slot * vd_all + g * vdim + d);
      }
      vs[i] = v;
    }
    __syncthreads();
    for (int mp = 0; mp < MAPS; mp++)
      for (int i = 0; i < 4; i++) {
        const int r = wave * 4 + i;
        float s = -INFINITY;
        if (lane < KT && pq[i] >= 0 && kt0 + lane <= pq[i] && kt0 + lane >= plo[i] && kt0 + lane < n_keys) {
          float d0 = 0.f;
          for (int d = 0; d < dim; d++) d0 = fmaf(qs[r * dm + mp * dim + d], ks[lane * kld + mp * dim + d], d0);
          s = cap_score(d0 * hscale, a.softcap);
        }
        const float mn = fmaxf(m[mp][i], wave_max(s));
        float p = 0.f, corr = 1.f;
        if (mn > -INFINITY) {
          p = s > -INFINITY ? expf(s - mn) : 0.f;
          corr = m[mp][i] > -INFINITY ? expf(m[mp][i] - mn) : 0.f;
        }
        l[mp][i] = l[mp][i] * corr + wave_sum(p);
        m[mp][i] = mn;
        for (int rr = 0; rr < NR; rr++) acc[mp][i][rr] *= corr;
        if (lane < KT) ps[(mp * STK_QT + r) * KT + lane] = p;
      }
    __syncthreads();
    for (int rr = 0; rr < NR; rr++) {
      const int d = lane + 64 * rr;
      if (d >= vdim) break;
#pragma unroll 4
      for (int j = 0; j < KT; j++) {
        const float v = vs[j * vdim + d];
        for (int mp = 0; mp < MAPS; mp++)
          for (int i = 0; i < 4; i++) acc[mp][i][rr] = fmaf(ps[(mp * STK_QT + wave * 4 + i) * KT + j], v, acc[mp][i][rr]);
      }
    }
  }
  T* out = (T*)a.out;
  for (int i = 0; i < 4; i++) {
    const int r = wave * 4 + i;
    if (r >= nq) continue;
    if constexpr (MAPS == 2) {
      const float i1 = l[0][i] > 0.f ? 1.f / l[0][i] : 0.f, i2 = l[MAPS - 1][i] > 0.f ? a.diff_lambda / l[MAPS - 1][i] : 0.f;
      float o[NR], q2 = 0.f;
      for (int rr = 0; rr < NR; rr++) {
        o[rr] = lane + 64 * rr < vdim ? acc[0][i][rr] * i1 - acc[MAPS - 1][i][rr] * i2 : 0.f;
        q2 = fmaf(o[rr], o[rr], q2);
      }
      const float f = a.diff_scale / sqrtf(wave_sum(q2) / (float)vdim + a.diff_eps);
      for (int rr = 0; rr < NR; rr++)
        if (lane + 64 * rr < vdim) El<T>::st(out + (size_t)(t0 + r) * a.H * vdim + h * vdim + lane + 64 * rr, o[rr] * f);
      continue;
    }
    float inv = l[0][i] > 0.f ? 1.f / l[0][i] : 0.f;
    if (a.gate) inv *= sigmoidf_(a.gate[(size_t)(t0 + r) * a.gate_ld + h]);
    for (int rr = 0; rr < NR; rr++) {
      const int d = lane + 64 * rr;
      if (d < vdim) El<T>::st(out + (size_t)(t0 + r) * a.H * vdim + h * vdim + d, acc[0][i][rr] * inv);
    }
  }
}

// bf16 models, key size a multiple of 8 and value size a multiple of 16: the same operator on the matrix cores.
// A workgroup of 4 waves owns 64 query rows of one head (16 per wave) and walks the keys in tiles of 32 from key 0.
//   S^T = K . Q^T   A operand = K rows straight from the cache (lane = (key rq, channel octet oct)), B = Q fragments kept in registers;
//                   the lane ends up with query row rq and keys oct * 4 + j of both 16-key halves: 8 scores, all in f32 — temperature,
//                   scale, soft cap, mask, running maximum (two xor shuffles join the 4 lanes of a row) and exponentials;
//   O^T += V^T . P^T  A operand = the V tile, transposed once per workgroup into LDS with the keys in the order the lanes hold their
//                   scores (position = oct * 8 + half * 4 + j), B = the lane's own 8 weights.  The weights stay f32 in effect: each is
//                   split into a bf16 head and a bf16 tail (p = hi + lo to 2^-17) and the product runs twice.
// Every sum goes tile by tile from key 0 with a fixed lane pattern: the result of a row does not depend on the portion it came in.
// MAPS 2: the differential form of StkAttnArgs.  Four more waves own the second map of the same 64 rows (their registers are those of the plain
// kernel), all eight share the transposed V tile; at the end the second map's rows travel through LDS to the first map's waves, which
// combine, norm and store.
template <int DC, int VT, int MAPS>
__global__ __launch_bounds__(256 * MAPS, MAPS == 2 && DC <= 2 ? 4 : 1) void stk_attn_prefill_mfma_kernel(StkAttnArgs a) {
  constexpr int KT = 32, VLD = KT + 8;  // LDS row of a value channel: 32 positions + 8 (rows stay 16-byte aligned, lanes spread over banks)
  constexpr int NT = 256 * MAPS, XT = VT < 4 ? VT : 4;  // threads; channel tiles handed over at a time (MAPS 2: 4 waves x 64 lanes x 16 bytes each)
  constexpr int VT_BYTES = VT * 16 * VLD * 2, X_BYTES = MAPS == 2 ? XT * 4096 : 0;
  __shared__ __attribute__((aligned(16))) unsigned char smem[VT_BYTES > X_BYTES ? VT_BYTES : X_BYTES];
  uint16_t* vt = (uint16_t*)smem;
  const int dim = a.dim, vdim = a.vdim, dm = MAPS * dim;
  const int b = blockIdx.y, h = blockIdx.z, g = h / (a.H / a.G);
  const int q0 = a.cu_q[b], q1 = a.cu_q[b + 1];
  // the last row blocks of a portion see the most keys: they are dispatched first, so that no long block is left to run alone at the end
  const int t0 = q0 + ((int)gridDim.x - 1 - (int)blockIdx.x) * 64;
  if (t0 >= q1) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, rq = lane & 15, oct = lane >> 4;
  const int mp = MAPS == 2 ? wave >> 2 : 0;  // this wave's map
  const int tq = t0 + (wave & 3) * 16 + rq;  // this lane's query row
  const bool qv = tq < q1;
  const int64_t pq = qv ? a.positions[tq] : -1;
  const uint16_t* q = (const uint16_t*)a.q;
  const u32x4 zero4 = {0u, 0u, 0u, 0u};
  u32x4 qf[DC];
  for (int c = 0; c < DC; c++) {
    const int ch = c * 32 + oct * 8;
    const bool ok = qv && ch < dim;
    const u32x4 v = *(const u32x4*)(q + (size_t)(ok ? tq : q0) * a.ldq + h * dm + mp * dim + (ok ? ch : 0));
    qf[c] = ok ? v : zero4;
  }
  const float sc = a.scale * q_temperature(pq < 0 ? 0 : pq, a.temp_coef, a.temp_every) * (a.head_scale ? a.head_scale[h] : 1.f);
  // keys this workgroup needs: up to the largest position of its rows
  int64_t pmax = pq;
  for (int o = 32; o > 0; o >>= 1) pmax = max(pmax, (int64_t)__shfl_xor((long long)pmax, o, 64));
  // block mask: this row sees the keys from key_lo on; the workgroup's tiles start at the tile of its smallest key_lo
  int64_t key_lo = a.chunk > 0 && pq >= 0 ? pq / a.chunk * a.chunk : 0;
  if (a.window > 0 && pq >= 0) key_lo = max(key_lo, pq - a.window + 1);
  int64_t lmin = pq >= 0 ? key_lo : INT64_MAX;
  for (int o = 32; o > 0; o >>= 1) lmin = min(lmin, (int64_t)__shfl_xor((long long)lmin, o, 64));
  __shared__ long long wmax[4 * MAPS], wmin[4 * MAPS];  // (the waves of the second map own the same rows)
  if (lane == 0) wmax[wave] = pmax, wmin[wave] = lmin;
  __syncthreads();
  const int64_t gmax = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
  const int64_t gmin = min(min(wmin[0], wmin[1]), min(wmin[2], wmin[3]));
  const int kt_begin = gmin == INT64_MAX ? 0 : (int)(gmin / 32) * 32;
  const int n_keys = (int)min((int64_t)a.context_lens[b], gmax + 1);
  const int n_keys_wave = (int)min((int64_t)n_keys, pmax + 1);
  const uint16_t* kc = (const uint16_t*)a.kc;
  const uint16_t* vc = (const uint16_t*)a.vc;
  const uint32_t* bt = a.block_tables + (size_t)b * a.max_blocks;
  const int kdim = a.k_ld ? a.k_ld : a.G * dm, vd_all = a.v_ld ? a.v_ld : a.G * vdim;
  f32x4 acc[VT];
  for (int t = 0; t < VT; t++) acc[t] = vra_zero_acc();
  float m = -INFINITY, l = 0.f;
  if (a.sink) m = a.sink[h], l = oct == 0 ? 1.f : 0.f;  // (the four lanes of a row add their sums at the end: the sink counts once)
  const bool capped = a.softcap > 0.f;
  const float two_inv_cap = capped ? 2.f / a.softcap : 0.f, two_cap = 2.f * a.softcap;
  const int key_end = (int)min((int64_t)n_keys, pq + 1);  // this row sees the keys below key_end
  // The K fragments and this thread's share of the V tile are requested one tile ahead, so that their way from memory runs beside the
  // current tile's arithmetic.  V item = (key, 8 channels): NV per thread.
  // V item = (pair of neighbouring keys, 8 channels): NV per thread, two 16-byte requests each
  constexpr int NV = (KT / 2 * VT * 2 + NT - 1) / NT;
  u32x4 kfn[2][DC], vgn[NV][2];
  // The page size is a multiple of 32 (the launcher sends other sizes to the FMA kernel), so a 32-key tile lies in ONE page: its first
  // slot is a scalar, read from the block table one tile ahead of the requests that use it — no request of a tile waits behind a
  // block-table read (vector loads return in order: a per-key read would also wait for everything issued before it).
  auto page_slot = [&](int kt0) -> int64_t {  // first cache slot of the tile that starts at key kt0 (uniform)
    const int t = __builtin_amdgcn_readfirstlane(kt0);
    return t < n_keys ? (int64_t)bt[t / a.BS] * a.BS + t % a.BS : 0;
  };
  auto request_tile = [&](int kt0, int64_t slot0) {
    auto slot_of = [&](int key) { return slot0 + (key - kt0); };
    for (int u = 0; u < 2; u++) {
      const int key = kt0 + u * 16 + rq;
      const bool kv = key < n_keys;
      const int64_t slot = kv ? slot_of(key) : 0;
      const uint16_t* kr = kc + slot * kdim + g * dm + mp * dim;
      for (int c = 0; c < DC; c++) {
        const int ch = c * 32 + oct * 8;
        const bool ok = kv && ch < dim;
        const u32x4 kf = *(const u32x4*)(kr + (ok ? ch : 0));
        kfn[u][c] = ok ? kf : zero4;
      }
    }
    for (int n = 0; n < NV; n++) {
      const int i = tid + n * NT;
      const int kp = i / (VT * 2), c8 = (i % (VT * 2)) * 8;
      for (int e = 0; e < 2; e++) {
        const int key = kt0 + kp * 2 + e;
        const bool ok = i < KT / 2 * VT * 2 && key < n_keys && c8 < vdim;
        const int64_t slot = ok ? slot_of(key) : 0;
        const u32x4 v = *(const u32x4*)(vc + slot * vd_all + g * vdim + (ok ? c8 : 0));
        vgn[n][e] = ok ? v : zero4;
      }
    }
  };
  request_tile(kt_begin, page_slot(kt_begin));
  int64_t slot_next = page_slot(kt_begin + KT);
  for (int kt0 = kt_begin; kt0 < n_keys; kt0 += KT) {
    u32x4 kfc[2][DC], vgc[NV][2];
    for (int u = 0; u < 2; u++)
      for (int c = 0; c < DC; c++) kfc[u][c] = kfn[u][c];
    for (int n = 0; n < NV; n++) vgc[n][0] = vgn[n][0], vgc[n][1] = vgn[n][1];
    __syncthreads();
    // V tile -> LDS, transposed, the keys in the order the lanes hold their scores: keys 2 kp and 2 kp + 1 are neighbours there too,
    // so one 32-bit store carries both for a channel
    for (int n = 0; n < NV; n++) {
      const int i = tid + n * NT;
      if (i >= KT / 2 * VT * 2) break;
      const int kl = (i / (VT * 2)) * 2, c8 = (i % (VT * 2)) * 8;
      const int pos = ((kl & 15) >> 2) * 8 + (kl >> 4) * 4 + (kl & 3);  // even
      uint32_t* row = (uint32_t*)vt;
      for (int e = 0; e < 4; e++) {
        const uint32_t lo0 = vgc[n][0][e] & 0xffffu, hi0 = vgc[n][0][e] >> 16, lo1 = vgc[n][1][e] & 0xffffu, hi1 = vgc[n][1][e] >> 16;
        row[((c8 + 2 * e) * VLD + pos) >> 1] = lo0 | (lo1 << 16);
        row[((c8 + 2 * e + 1) * VLD + pos) >> 1] = hi0 | (hi1 << 16);
      }
    }
    __syncthreads();
    if (kt0 + KT < n_keys) {
      request_tile(kt0 + KT, slot_next);
      slot_next = page_slot(kt0 + 2 * KT);
    }
    if (kt0 >= n_keys_wave) continue;  // (wave-uniform: nothing of this tile is visible to the wave's rows)
    // scores of the two 16-key halves
    f32x4 s[2];
    s[0] = vra_zero_acc();
    s[1] = vra_zero_acc();
    for (int c = 0; c < DC; c++) {  // (the two halves' chains alternate: an MFMA never waits for the one issued just before it)
      BF16::mfma(s[0], __builtin_bit_cast(s16x8, kfc[0][c]), __builtin_bit_cast(s16x8, qf[c]));
      BF16::mfma(s[1], __builtin_bit_cast(s16x8, kfc[1][c]), __builtin_bit_cast(s16x8, qf[c]));
    }
    VRA_MFMA_DRAIN();
    float sv[8];
    float tmax = -INFINITY;
    for (int u = 0; u < 2; u++)
      for (int j = 0; j < 4; j++) {
        const int key = kt0 + u * 16 + oct * 4 + j;
        float x = s[u][j] * sc;
        if (capped) {  // softcap * tanh(x / softcap) = softcap - 2 softcap / (1 + e^(2 x / softcap)), hardware exponential and reciprocal
          const float y = fminf(fmaxf(x * two_inv_cap, -30.f), 30.f);
          x = a.softcap - two_cap * __builtin_amdgcn_rcpf(1.f + __expf(y));
        }
        x = key < key_end && key >= key_lo ? x : -INFINITY;
        sv[u * 4 + j] = x;
        tmax = fmaxf(tmax, x);
      }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float mn = fmaxf(m, tmax);
    float corr = 1.f, psum = 0.f, pv[8];
    for (int i = 0; i < 8; i++) pv[i] = 0.f;
    if (mn > -INFINITY) {
      corr = m > -INFINITY ? __expf(m - mn) : 0.f;
      for (int i = 0; i < 8; i++) {
        pv[i] = sv[i] > -INFINITY ? __expf(sv[i] - mn) : 0.f;
        psum += pv[i];
      }
    }
    l = l * corr + psum;
    m = mn;
    u32x4 phi, plo;
    for (int e = 0; e < 4; e++) {
      const float a0 = pv[2 * e], a1 = pv[2 * e + 1];
      const uint32_t hi = BF16::pack2(a0, a1);
      phi[e] = hi;
      plo[e] = BF16::pack2(a0 - __uint_as_float(hi << 16), a1 - __uint_as_float(hi & 0xffff0000u));
    }
    for (int t = 0; t < VT; t++) {
      acc[t][0] *= corr, acc[t][1] *= corr, acc[t][2] *= corr, acc[t][3] *= corr;
    }
    // heads of four channel tiles first, then their tails: the two MFMAs into one accumulator are four instructions apart, and only four V
    // fragments are held at a time (fully unrolled: every accumulator keeps its registers, no indexed register moves next to an MFMA)
    constexpr int VG = 4;
#pragma unroll
    for (int t0_ = 0; t0_ < VT; t0_ += VG) {
      u32x4 vf[VG];
#pragma unroll
      for (int t = 0; t < VG; t++) vf[t] = *(const u32x4*)(vt + ((t0_ + t) * 16 + rq) * VLD + oct * 8);
#pragma unroll
      for (int t = 0; t < VG; t++) BF16::mfma(acc[t0_ + t], __builtin_bit_cast(s16x8, vf[t]), __builtin_bit_cast(s16x8, phi));
#pragma unroll
      for (int t = 0; t < VG; t++) BF16::mfma(acc[t0_ + t], __builtin_bit_cast(s16x8, vf[t]), __builtin_bit_cast(s16x8, plo));
    }
    VRA_MFMA_DRAIN();
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if constexpr (MAPS == 2) {  // (channels beyond vdim hold zeros: their V columns were staged as zeros)
    const float inv = l > 0.f ? (mp == 0 ? 1.f : a.diff_lambda) / l : 0.f;
    float* ex = (float*)smem;
    float q2 = 0.f;
#pragma unroll
    for (int x0 = 0; x0 < VT; x0 += XT) {
      __syncthreads();
      if (mp == 1)
#pragma unroll
        for (int t = 0; t < XT; t++) *(f32x4*)(ex + ((t * 4 + (wave & 3)) * 64 + lane) * 4) = acc[x0 + t] * inv;
      __syncthreads();
      if (mp == 0)
#pragma unroll
        for (int t = 0; t < XT; t++) {
          const f32x4 o2 = *(const f32x4*)(ex + ((t * 4 + wave) * 64 + lane) * 4);
#pragma unroll
          for (int j = 0; j < 4; j++) {
            const float o = acc[x0 + t][j] * inv - o2[j];
            acc[x0 + t][j] = o;
            q2 = fmaf(o, o, q2);
          }
        }
    }
    q2 += __shfl_xor(q2, 16, 64);
    q2 += __shfl_xor(q2, 32, 64);
    if (mp == 1 || !qv) return;
    const float f = a.diff_scale / sqrtf(q2 / (float)vdim + a.diff_eps);
    uint16_t* out = (uint16_t*)a.out + (size_t)tq * a.H * vdim + h * vdim;
#pragma unroll
    for (int t = 0; t < VT; t++) {
      const int c = t * 16 + oct * 4;  // (vdim is a multiple of 16: a lane's four channels are in or out together)
      uint2 p;
      p.x = BF16::pack2(acc[t][0] * f, acc[t][1] * f), p.y = BF16::pack2(acc[t][2] * f, acc[t][3] * f);
      if (c < vdim) *(uint2*)(out + c) = p;
    }
    return;
  }
  if (!qv) return;
  float inv = l > 0.f ? 1.f / l : 0.f;
  if (a.gate) inv *= sigmoidf_(a.gate[(size_t)tq * a.gate_ld + h]);
  uint16_t* out = (uint16_t*)a.out + (size_t)tq * a.H * vdim + h * vdim;
  for (int t = 0; t < VT; t++)
    for (int j = 0; j < 4; j++) {
      const int c = t * 16 + oct * 4 + j;
      if (c < vdim) out[c] = BF16::from_f32(acc[t][j] * inv);
    }
}

// One decoded token per sequence, for what stack_decode_attn.hip does not take: a workgroup per (sequence, query head); its 8 waves take the 64-key tiles of the context in turn,
// read K rows straight from the cache (lane = key, 16 bytes a load where the row allows) and V rows channel-wise (lane = channel), and
// meet once in LDS.  The order of the sums depends on the context length alone.
// MAPS 2: the differential form of StkAttnArgs (both maps' scores of a key, then one pass over the values for both);
// with scratch the key tiles are spread over gridDim.z workgroups and stk_attn_decode_join_kernel adds their parts.
#define STK_DW 8
template <typename T>
__device__ __forceinline__ float stk_dot_row(const float* qs, const T* kr, int dim) {
  float d0 = 0.f;
  for (int d = 0; d < dim; d++) d0 = fmaf(qs[d], El<T>::ld(kr + d), d0);
  return d0;
}
template <>
__device__ __forceinline__ float stk_dot_row<uint16_t>(const float* qs, const uint16_t* kr, int dim) {
  float d0 = 0.f;
  if (dim % 8 == 0 && ((uintptr_t)kr % 16) == 0) {
    for (int d = 0; d < dim; d += 8) {
      const u32x4 v = *(const u32x4*)(kr + d);
      for (int e = 0; e < 4; e++) {
        d0 = fmaf(qs[d + 2 * e], __uint_as_float(v[e] << 16), d0);
        d0 = fmaf(qs[d + 2 * e + 1], __uint_as_float(v[e] & 0xffff0000u), d0);
      }
    }
    return d0;
  }
  for (int d = 0; d < dim; d++) d0 = fmaf(qs[d], BF16::to_f32(kr[d]), d0);
  return d0;
}
template <typename T, int NR, int MAPS>
__global__ __launch_bounds__(64 * STK_DW) void stk_attn_decode_kernel(StkAttnArgs a) {
  extern __shared__ float lds[];
  const int dim = a.dim, vdim = a.vdim, dm = MAPS * dim;
  float* qs = lds;                     // [dm]
  float* ps = qs + dm;                 // [MAPS][waves][64]
  float* ms = ps + MAPS * STK_DW * 64;   // [MAPS][waves] max, [MAPS][waves] sum
  float* os = ms + MAPS * 2 * STK_DW;    // [MAPS][waves][vdim]
  int* ss = (int*)(os + MAPS * STK_DW * vdim);  // [waves][64] cache slot of each key of the wave's current tile
  const int b = blockIdx.x, h = blockIdx.y, g = h / (a.H / a.G);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t p = a.positions[b];
  const int n_keys = (int)min((int64_t)a.context_lens[b], p + 1);
  const T* q = (const T*)a.q + (size_t)b * a.ldq + h * dm;
  const float temp = q_temperature(p, a.temp_coef, a.temp_every);
  for (int d = tid; d < dm; d += 64 * STK_DW) qs[d] = El<T>::ld(q + d) * temp;
  __syncthreads();
  const T* kc = (const T*)a.kc;
  const T* vc = (const T*)a.vc;
  const uint32_t* bt = a.block_tables + (size_t)b * a.max_blocks;
  const int kdim = a.k_ld ? a.k_ld : a.G * dm, vd_all = a.v_ld ? a.v_ld : a.G * vdim;
  float m[MAPS], l[MAPS], acc[MAPS][NR], vacc[MAPS][8];
#pragma unroll
  for (int mp = 0; mp < MAPS; mp++) {
    m[mp] = -INFINITY, l[mp] = 0.f;
    for (int i = 0; i < NR; i++) acc[mp][i] = 0.f;
    for (int i = 0; i < 8; i++) vacc[mp][i] = 0.f;
  }
  if (a.sink && wave == 0) m[0] = a.sink[h], l[0] = 1.f;
  // 16-bit values in whole octets: the value phase reads 16 bytes a lane (oc = channel octets rounded up to a power of two)
  const bool vec = sizeof(T) == 2 && vdim % 8 == 0 && vd_all % 8 == 0 && ((uintptr_t)vc % 16) == 0;
  int oc = 1;
  while (oc * 8 < vdim) oc <<= 1;
  const int co = lane & (oc - 1), kg = lane / oc, kpar = 64 / oc;
  // block mask: the keys from key_lo on; tiles stay aligned to absolute positions (the first one may begin below key_lo: those keys
  // count with weight 0)
  int key_lo = a.chunk > 0 ? (int)(p / a.chunk * a.chunk) : 0;
  if (a.window > 0) key_lo = max(key_lo, (int)(p - a.window + 1));
  const float hscale = a.head_scale ? a.scale * a.head_scale[h] : a.scale;
  for (int kt0 = key_lo / 64 * 64 + (wave * (int)gridDim.z + (int)blockIdx.z) * 64; kt0 < n_keys; kt0 += STK_DW * (int)gridDim.z * 64) {
    const int key = kt0 + lane;
    float s[MAPS], corr[MAPS];
    for (int mp = 0; mp < MAPS; mp++) s[mp] = -INFINITY;
    if (key < n_keys) {
      const int64_t slot = (int64_t)bt[key / a.BS] * a.BS + key % a.BS;
      ss[wave * 64 + lane] = (int)slot;
      if (key >= key_lo)
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) s[mp] = cap_score(stk_dot_row<T>(qs + mp * dim, kc + slot * kdim + g * dm + mp * dim, dim) * hscale, a.softcap);
    }
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
      const float mn = fmaxf(m[mp], wave_max(s[mp]));  // (the tile's first key exists: mn is finite)
      const float pj = s[mp] > -INFINITY ? expf(s[mp] - mn) : 0.f;
      corr[mp] = m[mp] > -INFINITY ? expf(m[mp] - mn) : 0.f;
      l[mp] = l[mp] * corr[mp] + wave_sum(pj);
      m[mp] = mn;
      ps[(mp * STK_DW + wave) * 64 + lane] = pj;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int nj = min(64, n_keys - kt0);
    if (vec) {
      // lane = (key group kg, channel octet co): one 16-byte load covers 8 channels of one key, 64 / OC keys are in flight per step;
      // the groups' partial sums meet after the last tile
#pragma unroll
      for (int mp = 0; mp < MAPS; mp++)
        for (int i = 0; i < 8; i++) vacc[mp][i] *= corr[mp];
      // four keys of a group per step, their rows requested together (the slots come from LDS, where the score phase left them, so no
      // request waits for a block-table read); keys beyond the tile count with weight 0
      for (int j = kg; j < nj && co * 8 < vdim; j += 4 * kpar) {
        u32x4 v[4];
        float pw[MAPS][4];
        for (int u = 0; u < 4; u++) {
          const int ju = j + u * kpar;
          const bool in = ju < nj;
          const int64_t sl = ss[wave * 64 + (in ? ju : j)];
          v[u] = *(const u32x4*)((const uint16_t*)vc + sl * vd_all + g * vdim + co * 8);
#pragma unroll
          for (int mp = 0; mp < MAPS; mp++) pw[mp][u] = in ? ps[(mp * STK_DW + wave) * 64 + ju] : 0.f;
        }
        for (int u = 0; u < 4; u++)
#pragma unroll
          for (int mp = 0; mp < MAPS; mp++)
            for (int i = 0; i < 4; i++) {
              vacc[mp][2 * i] = fmaf(pw[mp][u], __uint_as_float(v[u][i] << 16), vacc[mp][2 * i]);
              vacc[mp][2 * i + 1] = fmaf(pw[mp][u], __uint_as_float(v[u][i] & 0xffff0000u), vacc[mp][2 * i + 1]);
            }
      }
    } else {
      for (int rr = 0; rr < NR; rr++) {
        const int d = lane + 64 * rr;
        if (d >= vdim) break;
        float o[MAPS];
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) o[mp] = acc[mp][rr] * corr[mp];
        for (int j = 0; j < nj; j++) {
          const float v = El<T>::ld(vc + (int64_t)ss[wave * 64 + j] * vd_all + g * vdim + d);
#pragma unroll
          for (int mp = 0; mp < MAPS; mp++) o[mp] = fmaf(ps[(mp * STK_DW + wave) * 64 + j], v, o[mp]);
        }
#pragma unroll
        for (int mp = 0; mp < MAPS; mp++) acc[mp][rr] = o[mp];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int mp = 0; mp < MAPS; mp++) {
    float* ow = os + (mp * STK_DW + wave) * vdim;
    if (vec) {
      for (int o = oc; o < 64; o <<= 1)
        for (int i = 0; i < 8; i++) vacc[mp][i] += __shfl_xor(vacc[mp][i], o, 64);
      if (lane < oc && co * 8 < vdim)
        for (int i = 0; i < 8; i++) ow[co * 8 + i] = vacc[mp][i];
    } else {
      for (int rr = 0; rr < NR; rr++) {
        const int d = lane + 64 * rr;
        if (d < vdim) ow[d] = acc[mp][rr];
      }
    }
    if (lane == 0) ms[mp * 2 * STK_DW + wave] = m[mp], ms[mp * 2 * STK_DW + STK_DW + wave] = l[mp];
  }
  __syncthreads();
  T* out = (T*)a.out + (size_t)b * a.H * vdim + h * vdim;
  const float og = a.gate ? sigmoidf_(a.gate[(size_t)b * a.gate_ld + h]) : 1.f;
  if (MAPS == 2 && a.splits > 1) {  // this part's sums relative to its own maximum: [B, S, H, MAPS, vdim], then (maximum, sum) [B, S, H, MAPS, 2]
    const size_t row = (((size_t)b * gridDim.z + blockIdx.z) * a.H + h) * MAPS;
    float* ml = a.scratch + (size_t)gridDim.x * gridDim.z * a.H * MAPS * vdim;
#pragma unroll
    for (int mp = 0; mp < MAPS; mp++) {
      const float *mm = ms + mp * 2 * STK_DW, *ow = os + mp * STK_DW * vdim;
      float M = mm[0], L = 0.f;
      for (int w = 1; w < STK_DW; w++) M = fmaxf(M, mm[w]);
      float cw[STK_DW];
      for (int w = 0; w < STK_DW; w++) {
        cw[w] = mm[w] > -INFINITY ? expf(mm[w] - M) : 0.f;
        L += mm[STK_DW + w] * cw[w];
      }
      for (int d = tid; d < vdim; d += 64 * STK_DW) {
        float o = 0.f;
        for (int w = 0; w < STK_DW; w++) o += ow[w * vdim + d] * cw[w];
        a.scratch[(row + mp) * vdim + d] = o;
      }
      if (tid == 0) ml[(row + mp) * 2] = M, ml[(row + mp) * 2 + 1] = L;
    }
    return;
  }
  auto joined = [&](int mp, int d) {  // the waves' partial sums of channel d, in wave order
    const float *mm = ms + mp * 2 * STK_DW, *ow = os + mp * STK_DW * vdim;
    float M = mm[0];
    for (int w = 1; w < STK_DW; w++) M = fmaxf(M, mm[w]);
    float L = 0.f, o = 0.f;
    for (int w = 0; w < STK_DW; w++) {
      const float c = mm[w] > -INFINITY ? expf(mm[w] - M) : 0.f;
      L += mm[STK_DW + w] * c;
      o += ow[w * vdim + d] * c;
    }
    return L > 0.f ? o / L : 0.f;
  };
  if constexpr (MAPS == 2) {  // (vdim <= 512: a channel a thread)
    const float o = tid < vdim ? joined(0, tid) - a.diff_lambda * joined(1, tid) : 0.f;
    const float q2 = wave_sum(o * o);
    if (lane == 0) qs[wave] = q2;  // (ps and qs are free: every wave has passed the barrier)
    __syncthreads();
    float t2 = qs[0];
    for (int w = 1; w < STK_DW; w++) t2 += qs[w];
    if (tid < vdim) El<T>::st(out + tid, o * (a.diff_scale / sqrtf(t2 / (float)vdim + a.diff_eps)));
    return;
  }
  for (int d = tid; d < vdim; d += 64 * STK_DW) El<T>::st(out + d, joined(0, d) * og);
}

// the parts of a differential decode added up in order, the two maps combined, normed and stored: a workgroup per (sequence, head)
template <typename T>
__global__ __launch_bounds__(128) void stk_attn_decode_join_kernel(StkAttnArgs a) {
  __shared__ float ws[2][64], red[2];
  const int b = blockIdx.x, h = blockIdx.y, S = a.splits, vdim = a.vdim, tid = threadIdx.x, lane = tid & 63, mp = tid >> 6;
  const float* ml = a.scratch + (size_t)gridDim.x * S * a.H * 2 * vdim;
  {  // wave mp: the weights of map mp's parts, lane = part
    const bool in = lane < S;
    const size_t at = ((((size_t)b * S + (in ? lane : 0)) * a.H + h) * 2 + mp) * 2;
    const float m = in ? ml[at] : -INFINITY, l = in ? ml[at + 1] : 0.f;
    const float M = wave_max(m), w = m > -INFINITY ? expf(m - M) : 0.f;
    const float L = wave_sum(w * l);
    ws[mp][lane] = L > 0.f ? w * (mp ? a.diff_lambda : 1.f) / L : 0.f;
  }
  __syncthreads();
  float o[4], q2 = 0.f;
#pragma unroll
  for (int i = 0; i < 4; i++) {  // (vdim <= 512)
    const int c = tid + i * 128;
    o[i] = 0.f;
    if (c >= vdim) continue;
    float o1 = 0.f, o2 = 0.f;
    for (int s = 0; s < S; s++) {
      const float* p = a.scratch + (((size_t)b * S + s) * a.H + h) * 2 * vdim + c;
      o1 = fmaf(ws[0][s], p[0], o1), o2 = fmaf(ws[1][s], p[vdim], o2);
    }
    o[i] = o1 - o2;
    q2 = fmaf(o[i], o[i], q2);
  }
  q2 = wave_sum(q2);
  if (lane == 0) red[mp] = q2;
  __syncthreads();
  const float f = a.diff_scale / sqrtf((red[0] + red[1]) / (float)vdim + a.diff_eps);
  T* out = (T*)a.out + ((size_t)b * a.H + h) * vdim;
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (tid + i * 128 < vdim) El<T>::st(out + tid + i * 128, o[i] * f);
}

}  // namespace

// ================================================================================================ launchers
#define STK_DIFF_PARTS 512  // (sequence, head, part) workgroups a decode step aims at
int vra_stack_diff_splits(int max_len, int B, int heads) { return max_len > 512 ? std::min(8, std::max(1, STK_DIFF_PARTS / std::max(B * heads, 1))) : 1; }
size_t vra_stack_diff_scratch(int max_len, int max_seqs, int heads, int vdim) {  // (more than one part: B * heads * parts <= STK_DIFF_PARTS)
  return vra_stack_diff_splits(max_len, 1, heads) > 1 ? (size_t)STK_DIFF_PARTS * 2 * (vdim + 2) * sizeof(float) : 0;
}

// (128-row tiles: a tile row costs the same however few of its rows hold pairs — from 96 rows an expert on they are full enough)
int vra_stack_gemm_granule(int rows, int groups, bool tiles128) {
  if (groups > 0 && tiles128 && rows / groups >= 96) return 128;
  return groups > 0 && rows / groups >= 128 ? 64 : 16;
}
int32_t vra_stack_op_expert_rows(int32_t pairs, int32_t experts, int32_t tiles128) {
  const int g = vra_stack_gemm_granule(pairs, experts, tiles128 != 0);
  return (pairs + experts * (g - 1) + g - 1) / g * g;
}
void vra_stack_scale_rows(const void* a, int W, const int* row_token, const float* row_scale, void* out, int rows, int64_t stream) {
  VRA_CHECK_ARG(a && row_token && row_scale && out && rows > 0 && W > 0 && W % 8 == 0, "stack scale rows: null pointer or bad shape");
  launch_checked("stack scale rows", [&] { stk_scale_rows_kernel<<<rows, 256, 0, as_stream(stream)>>>((const uint16_t*)a, W, row_token, row_scale, (uint16_t*)out); });
}

// Steps of more than 32 rows on gemm_rows_kernel: whole 64-steps of K, and operands whose byte offsets stay within 31 bits (a gathered
// operand must say how many rows it has)
static int rows_fn(const StkGemmArgs& g) {
  if (g.epi == 1) return g.act == 1 ? FN_PAIR_GELU : (g.act == 2 ? FN_PAIR_SILU : FN_PAIR_CLAMPED);
  if (g.epi == 2) return g.act == 3 ? FN_GELU : (g.act == 4 ? FN_RELU2 : (g.act == 5 ? FN_TANH : FN_EXPEXP));
  return g.softcap > 0.f ? FN_SOFTCAP : (g.kv_slot ? FN_KV : FN_NONE);
}
static bool rows_kernel_takes(const StkGemmArgs& g) {
  if (g.epi == 2 && g.softcap > 0.f) return false;  // (both at once: nobody asks for it)
  const int64_t rows = g.a_row ? g.a_rows : g.M;
  return g.K % 64 == 0 && rows > 0 && rows * g.lda * 2 < 0x7FFF0000ll && (int64_t)g.N * g.K * 2 < 0x7FFF0000ll && g.batch <= 65535;
}

// Columns a workgroup takes of a product of up to 32 rows.  32 read x half as often, but while 16 fit one round of the CUs they leave CUs idle (8 rows:
// 2048 columns, K = 2048 / 8192: 7.3 / 22.9 us, with 16 columns 5.5 / 14.6; 17 rows, 2048 columns: 8.3 / 24.9, 6.2 / 17.3).  Beyond that round 16
// lose (17 rows, 3072 columns, K = 8192: 25.4, with 16 columns 31.1; 16 rows, 6144 columns, K = 4096: 16.7, 19.2) or change little (8 rows, 8000
// columns, K = 512 / 4096: 5.3 / 17.9, 5.6 / 16.2).  A gated pair needs both its blocks.
int32_t vra_stack_op_gemm_few_columns(int32_t M, int32_t N, int32_t batch, int32_t pair) {
  const int64_t wide = (int64_t)((M + 15) / 16) * ((N + 31) / 32) * batch;
  return pair || wide > 128 ? 32 : 16;
}

// Cache columns of a product: in its epilogue where a kernel that has one takes it (in 16-byte pieces: no piece crosses from q to k or k to v), otherwise a copy
// behind it.  The copy moves little (2048 rows: 8 MB) but is a launch: 5.1 us a layer of a 2048-token prompt, 3.0 and the gap before it of a decode step.
// Whole steps, 16 + 4 + 4 heads of 128, width 2048, with the copy / so: 4 layers, 2048 tokens 1196 / 1184 us, eight decoded tokens 320 / 306.  A row's slot is
// read ahead of the product's loop: behind it, where every row waits for its own, the prompt's gain was lost.
static void gemm_any(const StkGemmArgs& g, int dtype, int64_t stream);
bool vra_stack_gemm_mirrors(const StkGemmArgs& g, int dtype) {
  return dtype == VRA_BF16 && g.M <= 32 && g.out_f32 && g.batch == 1 && g.epi != 1 && !g.tile_group && g.K % 8 == 0 && g.lda % 8 == 0 && (uintptr_t)g.a % 16 == 0 &&
         (uintptr_t)g.w % 16 == 0;
}
void vra_stack_gemm(const StkGemmArgs& g, int dtype, int64_t stream) {
  if (!g.kv_slot) return gemm_any(g, dtype, stream);
  const int kd = g.kv_k, vd = g.N - g.kv_from - g.kv_k;
  VRA_CHECK_ARG(g.kv_kc && g.kv_vc && g.kv_from > 0 && kd > 0 && vd > 0, "stack gemm: cache columns without a cache, or beyond the product's");
  VRA_CHECK_ARG(g.batch == 1 && g.epi == 0 && g.softcap <= 0.f && !g.tile_group && !g.a_row && !g.out_row && !g.a_scale && (!g.out_f32 || dtype == VRA_F32),
                "stack gemm: cache columns come with a plain product in the cache's type");
  auto al16 = [](const void* p) { return (uintptr_t)p % 16 == 0; };
  const bool fused = dtype == VRA_BF16 && g.K % 64 == 0 && g.lda % 8 == 0 && al16(g.a) && al16(g.w) && al16(g.out) && g.ldo % 8 == 0 && al16(g.kv_kc) && al16(g.kv_vc) &&
                     g.kv_from % 8 == 0 && kd % 8 == 0 && vd % 8 == 0 && (g.M <= 32 || (g.N > 128 && rows_kernel_takes(g)));
  if (fused) return gemm_any(g, dtype, stream);
  StkGemmArgs p = g;
  p.kv_slot = nullptr;
  gemm_any(p, dtype, stream);
  const int es = dtype == VRA_F32 ? 4 : 2;
  vra_stack_kv_store((const char*)g.out + (size_t)g.kv_from * es, (const char*)g.out + (size_t)(g.kv_from + kd) * es, g.ldo, g.kv_kc, g.kv_vc, g.kv_slot, g.M, kd, vd, dtype, stream);
}
static void gemm_any(const StkGemmArgs& g, int dtype, int64_t stream) {
  VRA_CHECK_ARG(g.a && g.w && g.out && g.M > 0 && g.N > 0 && g.K > 0, "stack gemm: null pointer or empty shape");
  VRA_CHECK_ARG(dtype == VRA_BF16 || dtype == VRA_F32, "stack gemm: dtype must be bf16 or f32");
  VRA_CHECK_ARG(!g.tile_group || g.granule == 16 || g.granule == 64 || g.granule == 128, "stack gemm: granule must be 16, 64 or 128");
  VRA_CHECK_ARG(!g.mirror || vra_stack_gemm_mirrors(g, dtype), "stack gemm: a second output goes with plain f32 products of up to 32 rows");
  VRA_CHECK_ARG(g.batch >= 1 && (g.batch == 1 || !g.tile_group), "stack gemm: a batched product has no row groups");
  hipStream_t st = as_stream(stream);
  const int nb = g.batch;
  // (few columns over a long K, the first stage of a low-rank projection: the 64-row tiles would leave most of the chip idle)
  const bool narrow = dtype == VRA_BF16 && !g.tile_group && !g.a_scale && nb == 1 && g.N <= 128 && g.K >= 1024 && g.M <= 8192;
  const bool big = g.tile_group ? g.granule >= 64 : g.M > 32 && !narrow;
  const bool mfma = dtype == VRA_BF16 && g.K % 8 == 0 && g.lda % 8 == 0 && ((uintptr_t)g.a % 16 == 0) && ((uintptr_t)g.w % 16 == 0) &&
                    (g.w_group_stride % 8 == 0) && (g.a_batch_stride % 8 == 0) && (g.w_batch_stride % 8 == 0);
  VRA_CHECK_ARG(g.epi >= 0 && g.epi <= 2 && (g.epi != 2 || (g.act >= 3 && g.act <= 6)) && (g.softcap <= 0.f || g.epi != 1), "stack gemm: unknown epilogue");
  const bool post = g.epi == 2 || g.softcap > 0.f;
  VRA_CHECK_ARG(!post || !g.a_scale, "stack gemm: scaled rows and an element-wise epilogue do not come together");
  VRA_CHECK_ARG(g.epi != 1 || (mfma && g.N % 32 == 0), "stack gemm: the gated epilogue needs the bf16 MFMA path and whole gate / up blocks");
  if (mfma) {
    const bool rows = big && !g.a_scale && rows_kernel_takes(g);
    const int fn = rows_fn(g);
    const bool mixes = nb == 1 && !g.tile_group && stk_mixes(fn);
    VRA_CHECK_ARG(!g.tile || (rows && ((gemm_rows_has_tile(g.tile, g.K) && (!g.tile_group || g.granule == (g.tile >> 4) * 64)) || (mixes && gemm_rows_has_tiles(g.tile, g.M, g.N, g.K)))),
                  "stack gemm: no such tile for this product");
    if (rows) {
      GemmRowsArgs r;
      r.x = g.a, r.x_ld = g.lda, r.x_row = g.a_row, r.w[0] = g.w, r.n[0] = g.N, r.M = g.M, r.K = g.K;
      r.tile_group = g.tile_group, r.w_group_stride = g.w_group_stride, r.x_batch_stride = g.a_batch_stride, r.w_batch_stride = g.w_batch_stride;
      const int tile = g.tile ? g.tile : mixes ? gemm_rows_tiles(g.M, r.n[0], g.K) : gemm_rows_tile(g.tile_group && g.likely_rows > 0 ? g.likely_rows : g.M, r.n, 1, nb, g.K, g.tile_group ? g.granule : 0);  // (a tile row is one granule)
      auto go = [&](auto fn) {
        const int per = g.out_f32 ? 4 : 8;  // elements of 16 bytes
        const bool vec = (uintptr_t)g.out % 16 == 0 && g.ldo % per == 0 && g.out_batch_stride % per == 0 && (g.out_f32 || (g.epi == 1 ? g.N % 32 : g.N % 8) == 0);
        const int form = !vec || g.out_row || g.bias ? 0 : (!g.out_f32 ? 1 : ((g.epi == 1 ? g.N / 2 : g.N) % 4 == 0 ? 2 : 0));
        StkRowsEpi<decltype(fn)::value> e{g.out, g.out_row, g.bias, g.out_batch_stride, g.bias_batch_stride, g.alpha, g.limit, g.act_alpha, g.softcap, g.ldo, g.out_f32, vec ? 1 : 0, form,
                                             g.kv_slot, g.kv_kc, g.kv_vc, g.kv_from, g.kv_k};
        launch_checked("stack gemm", [&] { gemm_rows_launch<BF16, false>(r, e, tile, nb, st); });
      };
      switch (fn) {
        case FN_PAIR_CLAMPED: go(std::integral_constant<int, FN_PAIR_CLAMPED>{}); break;
        case FN_PAIR_GELU: go(std::integral_constant<int, FN_PAIR_GELU>{}); break;
        case FN_PAIR_SILU: go(std::integral_constant<int, FN_PAIR_SILU>{}); break;
        case FN_GELU: go(std::integral_constant<int, FN_GELU>{}); break;
        case FN_RELU2: go(std::integral_constant<int, FN_RELU2>{}); break;
        case FN_TANH: go(std::integral_constant<int, FN_TANH>{}); break;
        case FN_EXPEXP: go(std::integral_constant<int, FN_EXPEXP>{}); break;
        case FN_SOFTCAP: go(std::integral_constant<int, FN_SOFTCAP>{}); break;
        case FN_KV: go(std::integral_constant<int, FN_KV>{}); break;
        default: go(std::integral_constant<int, FN_NONE>{}); break;
      }
    } else if (big) {
      dim3 grid((g.M + 63) / 64, (g.N + 127) / 128, nb);
      VRA_CHECK_ARG(!g.tile_group || g.granule == 64, "stack gemm: granules of 128 rows need an unscaled product with K a multiple of 64 and a known row count");
      if (g.a_scale) launch_checked("stack gemm", [&] { stk_gemm_mfma_kernel<2, 4, 2, 2, true><<<grid, 256, 0, st>>>(g); });
      else if (post) launch_checked("stack gemm", [&] { stk_gemm_mfma_kernel<2, 4, 2, 2, false, true><<<grid, 256, 0, st>>>(g); });
      else launch_checked("stack gemm", [&] { stk_gemm_mfma_kernel<2, 4, 2, 2, false><<<grid, 256, 0, st>>>(g); });
    } else {
      const bool wide = vra_stack_op_gemm_few_columns(g.M, g.N, nb, g.epi == 1) == 32, more = g.kv_slot || g.mirror;
#define STK_SMALL(NTV)                                                                                                                 \
  do {                                                                                                                               \
    dim3 grid((g.M + 15) / 16, (g.N + 16 * NTV - 1) / (16 * NTV), nb);                                                               \
    if (g.a_scale) launch_checked("stack gemm", [&] { stk_gemm_mfma_small_kernel<true, false, NTV><<<grid, 512, 0, st>>>(g); });     \
    else if (post && more) launch_checked("stack gemm", [&] { stk_gemm_mfma_small_kernel<false, true, NTV, true><<<grid, 512, 0, st>>>(g); }); \
    else if (post) launch_checked("stack gemm", [&] { stk_gemm_mfma_small_kernel<false, true, NTV><<<grid, 512, 0, st>>>(g); });     \
    else if (more) launch_checked("stack gemm", [&] { stk_gemm_mfma_small_kernel<false, false, NTV, true><<<grid, 512, 0, st>>>(g); }); \
    else launch_checked("stack gemm", [&] { stk_gemm_mfma_small_kernel<false, false, NTV><<<grid, 512, 0, st>>>(g); });              \
  } while (0)
      if (!wide && g.M <= 8 && (int64_t)((g.N + 7) / 8) * nb <= 256 && !g.a_scale && !g.tile_group) {
        dim3 grid(1, (g.N + 7) / 8, nb);
        if (post && more) launch_checked("stack gemm", [&] { stk_gemm_mfma_eight_kernel<true, true><<<grid, 512, 0, st>>>(g); });
        else if (post) launch_checked("stack gemm", [&] { stk_gemm_mfma_eight_kernel<true><<<grid, 512, 0, st>>>(g); });
        else if (more) launch_checked("stack gemm", [&] { stk_gemm_mfma_eight_kernel<false, true><<<grid, 512, 0, st>>>(g); });
        else launch_checked("stack gemm", [&] { stk_gemm_mfma_eight_kernel<false><<<grid, 512, 0, st>>>(g); });
      } else if (wide) STK_SMALL(2);
      else STK_SMALL(1);
#undef STK_SMALL
    }
    return;
  }
  VRA_CHECK_ARG(!g.tile, "stack gemm: no such tile for this product");
  VRA_CHECK_ARG(!g.tile_group || g.granule != 128, "stack gemm: granules of 128 rows are for bf16 products on the matrix cores");
  if (dtype == VRA_F32 && g.K % 4 == 0 && g.lda % 4 == 0 && (uintptr_t)g.a % 16 == 0 && (uintptr_t)g.w % 16 == 0 && g.w_group_stride % 4 == 0 && g.a_batch_stride % 4 == 0 &&
      g.w_batch_stride % 4 == 0) {
    // The tile with the least time a block of 16 k: 64 clocks for each load of the waves of a CU, a lone wave's 240, 400 or 700 at the least.  us of
    // 16 x 16, 32 x 16, 32 x 32 tiles: 64 rows, 2048 x 2048: 21.6, 29.0, 46.0; 128 rows, 3072 x 2048: 50.2, 39.0, 47.9; 342 rows, 8192 x 2048: 313, 264, 175
    auto waves = [&](int rows, int cols) { return ((int64_t)(g.M + rows - 1) / rows * ((g.N + cols - 1) / cols) * nb + 255) / 256; };
    const int64_t t11 = std::max<int64_t>(waves(16, 16) * 128, 240), t21 = std::max<int64_t>(waves(32, 16) * 192, 400), t22 = std::max<int64_t>(waves(32, 32) * 256, 700);
    const bool whole = !g.tile_group || g.granule >= 64;  // (row tiles of 32 lie in one group)
    auto go = [&](auto scaled) {
      constexpr bool S = decltype(scaled)::value;
      if (whole && t22 <= std::min(t11, t21)) stk_gemm_f32_kernel<2, 2, 8, S><<<dim3((g.M + 31) / 32, (g.N + 31) / 32, nb), 64, 0, st>>>(g);
      else if (whole && t21 < t11) stk_gemm_f32_kernel<2, 1, 8, S><<<dim3((g.M + 31) / 32, (g.N + 15) / 16, nb), 64, 0, st>>>(g);
      else stk_gemm_f32_kernel<1, 1, 12, S><<<dim3((g.M + 15) / 16, (g.N + 15) / 16, nb), 64, 0, st>>>(g);
    };
    launch_checked("stack gemm", [&] { g.a_scale ? go(std::true_type{}) : go(std::false_type{}); });
    return;
  }
  if (big) {
    dim3 grid((g.M + 63) / 64, (g.N + 63) / 64, nb);
    if (dtype == VRA_F32) launch_checked("stack gemm", [&] { stk_gemm_simple_kernel<float, 4><<<grid, 256, 0, st>>>(g); });
    else launch_checked("stack gemm", [&] { stk_gemm_simple_kernel<uint16_t, 4><<<grid, 256, 0, st>>>(g); });
  } else {
    dim3 grid((g.M + 15) / 16, (g.N + 63) / 64, nb);
    if (dtype == VRA_F32) launch_checked("stack gemm", [&] { stk_gemm_simple_kernel<float, 1><<<grid, 256, 0, st>>>(g); });
    else launch_checked("stack gemm", [&] { stk_gemm_simple_kernel<uint16_t, 1><<<grid, 256, 0, st>>>(g); });
  }
}

void vra_stack_embed_sinpos(const uint32_t* ids, const int64_t* positions, const void* embed, const float* inv_freq, float* x, int T, int W, int V,
                            int dtype, int64_t stream) {
  VRA_CHECK_ARG(ids && positions && embed && x && T > 0 && W > 0, "stack embed: null pointer or empty shape");
  const dim3 grid(T, std::max(1, std::min((W / 2 + 255) / 256, 256 / T)));
  // Two by two from 256 rows of more than 512 columns on, and from 1024 rows of 256 or 512: up to 512 columns a thread has one angle at most, and two by two leaves half of the
  // workgroup idle, which pays only where whole waves are left and the rows are many (512 columns, 300 rows 2.05 / 2.13, 1024 2.64 / 2.39, 8192 8.17 / 7.33; 384 columns, 512 rows
  // 2.12 / 2.24, 8192 6.99 / 7.09; 64 columns, 8192 rows 3.99 / 4.51).  us a launch, one angle / two by two (bf16): 2048 columns, 16 rows 1.98 / 2.05, 64 2.09 / 2.12, 128 2.62 / 2.22, 160 3.54 / 2.34, 255
  // 3.67 / 2.47, 512 4.08 / 2.81; 4096 columns, 32 rows 2.07 / 2.12, 64 2.66 / 2.22, 160 5.68 / 3.17.  What decides is whether a thread would take a second angle
  // (256 * grid.y < W / 2): the line could lie lower, at 65 rows of 2048
  const bool quads = W % 4 == 0 && (((uintptr_t)embed | (uintptr_t)inv_freq | (uintptr_t)x) % 16) == 0;
  const bool two = quads && T >= 256 && (W > 512 || (T >= 1024 && W % 256 == 0));
  auto go = [&](auto one) {
    typedef decltype(one) E;
    hipStream_t st = as_stream(stream);
    launch_checked("stack embed", [&] {
      if (!two) stk_embed_sinpos_kernel<E, 1, 1><<<grid, 256, 0, st>>>(ids, positions, (const E*)embed, inv_freq, x, W, V);
      else stk_embed_sinpos_kernel<E, 2, 2><<<grid, 256, 0, st>>>(ids, positions, (const E*)embed, inv_freq, x, W, V);
    });
  };
  if (dtype == VRA_F32) go(float{});
  else go(uint16_t{});
}

void vra_stack_group_norm(const StkNormArgs& a, int dtype, int64_t stream) {
  VRA_CHECK_ARG(a.x && a.w && a.h && a.T > 0 && a.W > 0, "stack norm: null pointer or empty shape");
  VRA_CHECK_ARG(a.groups >= 1 && a.W % a.groups == 0, "stack norm: the width must split into equal groups");
  VRA_CHECK_ARG(!a.o || ((a.x_out == a.x || !a.x_out) && (a.n1 == 0 || a.p1)), "stack norm: parts of the row without a place for the sum");
  VRA_CHECK_ARG(!a.rows || !a.x_out, "stack norm: chosen rows keep no sum");
  VRA_CHECK_ARG(!a.router_w || (a.pair_expert && a.pair_weight && a.top >= 1 && a.top <= a.n_router && (!a.gate_row || a.gate_out)), "stack norm: router outputs");
  const size_t lds = ((size_t)a.W + a.groups + a.n_router + 2) * sizeof(float);
  VRA_CHECK_ARG(lds <= 64 * 1024, "stack norm: row does not fit LDS");
  launch_checked("stack norm", [&] {
    auto go = [&](auto router, auto parts) {
      constexpr bool RT = decltype(router)::value, PA = decltype(parts)::value;
      if (dtype == VRA_F32) stk_group_norm_kernel<float, RT, PA><<<a.T, 256, lds, as_stream(stream)>>>(a);
      else stk_group_norm_kernel<uint16_t, RT, PA><<<a.T, 256, lds, as_stream(stream)>>>(a);
    };
    if (a.router_w) a.o ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
    else a.o ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
  });
}

void vra_stack_moe_sort(const int* pair_expert, const float* pair_weight, int P, int top, int n_groups, int granule, int max_rows, int* row_token,
                        float* row_scale, int* row_pair, int* tile_group, int64_t stream) {
  VRA_CHECK_ARG(pair_expert && pair_weight && row_token && row_scale && row_pair && tile_group && P > 0 && top > 0, "stack moe sort: null pointer");
  VRA_CHECK_ARG((granule == 16 || granule == 64 || granule == 128) && max_rows % granule == 0 && max_rows >= P + n_groups * (granule - 1), "stack moe sort: row space too small");
  const size_t lds = (size_t)n_groups * 3 * sizeof(int);
  VRA_CHECK_ARG(lds <= 48 * 1024, "stack moe sort: too many experts");
  launch_checked("stack moe sort", [&] {
    stk_moe_sort_kernel<<<1, 1024, lds, as_stream(stream)>>>(pair_expert, pair_weight, P, top, n_groups, granule, max_rows, row_token, row_scale, row_pair, tile_group);
  });
}

void vra_stack_gated_act(const float* gu, void* out, int M, int F, float limit, float act_alpha, int dtype, int64_t stream, int act) {
  VRA_CHECK_ARG(gu && out && M > 0 && F > 0, "stack gated act: null pointer or empty shape");
  if (dtype == VRA_F32) launch_checked("stack gated act", [&] { stk_gated_act_kernel<float><<<M, 256, 0, as_stream(stream)>>>(gu, (float*)out, F, limit, act_alpha, act); });
  else launch_checked("stack gated act", [&] { stk_gated_act_kernel<uint16_t><<<M, 256, 0, as_stream(stream)>>>(gu, (uint16_t*)out, F, limit, act_alpha, act); });
}

void vra_stack_polynorm(const float* z, void* out, const float* coef, int M, int F, float eps, int dtype, int64_t stream) {
  VRA_CHECK_ARG(z && out && coef && M > 0 && F > 0, "stack polynorm: null pointer or empty shape");
  const bool quads = F % 4 == 0 && (((uintptr_t)z | (uintptr_t)out) % 16) == 0;
  launch_checked("stack polynorm", [&] {
    if (dtype == VRA_F32) {
      if (quads) stk_polynorm_kernel<float, 4><<<M, STK_PN_THREADS, 0, as_stream(stream)>>>(z, (float*)out, coef, F, eps);
      else stk_polynorm_kernel<float, 1><<<M, STK_PN_THREADS, 0, as_stream(stream)>>>(z, (float*)out, coef, F, eps);
    } else {
      if (quads) stk_polynorm_kernel<uint16_t, 4><<<M, STK_PN_THREADS, 0, as_stream(stream)>>>(z, (uint16_t*)out, coef, F, eps);
      else stk_polynorm_kernel<uint16_t, 1><<<M, STK_PN_THREADS, 0, as_stream(stream)>>>(z, (uint16_t*)out, coef, F, eps);
    }
  });
}

void vra_stack_residual_combine(float* x, const float* o, const float* p1, int n1, const float* p2, const float* gate, float mult, int T, int W,
                                int64_t stream) {
  VRA_CHECK_ARG(x && T > 0 && W > 0 && (n1 == 0 || p1), "stack combine: null pointer or empty shape");
  const int quads = W % 4 == 0 && (((uintptr_t)x | (uintptr_t)o | (uintptr_t)p1 | (uintptr_t)p2) % 16) == 0;
  launch_checked("stack combine", [&] { stk_residual_combine_kernel<<<T, 256, 0, as_stream(stream)>>>(x, o, p1, n1, p2, gate, mult, W, quads); });
}

void vra_stack_gather_rows_f32(const float* src, const uint32_t* rows, float* dst, int n, int W, int64_t stream) {
  VRA_CHECK_ARG(src && rows && dst && n > 0 && W > 0, "stack gather: null pointer or empty shape");
  launch_checked("stack gather", [&] { stk_gather_rows_kernel<<<n, 256, 0, as_stream(stream)>>>(src, rows, dst, W); });
}

void vra_stack_kv_store(const void* k, const void* v, int ld, void* kc, void* vc, const int64_t* slots, int T, int kdim, int vdim, int dtype,
                        int64_t stream) {
  VRA_CHECK_ARG(k && v && kc && vc && slots && T > 0, "stack kv store: null pointer or empty shape");
  if (dtype == VRA_F32)
    launch_checked("stack kv store", [&] { stk_kv_store_kernel<float><<<T, 256, 0, as_stream(stream)>>>((const float*)k, (const float*)v, ld, (float*)kc, (float*)vc, slots, kdim, vdim); });
  else
    launch_checked("stack kv store", [&] {
      stk_kv_store_kernel<uint16_t><<<T, 256, 0, as_stream(stream)>>>((const uint16_t*)k, (const uint16_t*)v, ld, (uint16_t*)kc, (uint16_t*)vc, slots, kdim, vdim);
    });
}

void vra_stack_attention(const StkAttnArgs& a, int dtype, int64_t stream) {
  VRA_CHECK_ARG(a.q && a.out && a.kc && a.vc && a.positions && a.block_tables && a.context_lens, "stack attention: null pointer");
  VRA_CHECK_ARG(a.B > 0 && a.H > 0 && a.G > 0 && a.H % a.G == 0 && a.dim > 0 && a.vdim > 0 && a.vdim <= 512 && a.BS > 0 && a.max_blocks > 0,
                "stack attention: heads must be a multiple of kv heads, value size at most 512");
  VRA_CHECK_ARG(a.maps == 1 || (a.maps == 2 && !a.sink && !a.gate && !a.head_scale && a.chunk <= 0 && a.window <= 0 && a.softcap <= 0.f && a.temp_every <= 0),
                "stack attention: the differential form has two maps and no sink, gate, head scale, mask, cap or temperature");
  const bool two = a.maps == 2;
  const size_t dm = (size_t)a.maps * a.dim;
  hipStream_t st = as_stream(stream);
  if (!a.cu_q) {
    if (!two && a.arrived ? vra_stack_decode_group(a, dtype, stream) : !two && vra_stack_latent_decode(a, dtype, stream)) return;
    const size_t lds = (std::max<size_t>(dm, STK_DW) + (a.maps + 1) * STK_DW * 64 + a.maps * (2 * STK_DW + STK_DW * (size_t)a.vdim)) * sizeof(float);
    VRA_CHECK_ARG(lds <= 64 * 1024, "stack attention: head does not fit LDS");
    StkAttnArgs k = a;
    if (!two || !k.scratch || k.splits < 1) k.splits = 1;
    VRA_CHECK_ARG(k.splits <= 64 && (k.splits == 1 || (size_t)a.B * k.splits * a.H * 2 * (a.vdim + 2) * sizeof(float) <= a.scratch_bytes),
                  "stack attention: at most 64 parts, and their scratch");
    dim3 grid(a.B, a.H, k.splits);
#define STK_DEC(TT, NRV)                                                                              \
  launch_checked("stack attention (decode)", [&] {                                                    \
    if (two) stk_attn_decode_kernel<TT, NRV, 2><<<grid, 64 * STK_DW, lds, st>>>(k);                   \
    else stk_attn_decode_kernel<TT, NRV, 1><<<grid, 64 * STK_DW, lds, st>>>(k);                       \
  })
    if (dtype == VRA_F32) {
      if (a.vdim <= 256) STK_DEC(float, 4);
      else STK_DEC(float, 8);
    } else {
      if (a.vdim <= 256) STK_DEC(uint16_t, 4);
      else STK_DEC(uint16_t, 8);
    }
#undef STK_DEC
    if (k.splits > 1)
      launch_checked("stack attention (join)", [&] {
        if (dtype == VRA_F32) stk_attn_decode_join_kernel<float><<<dim3(a.B, a.H), 128, 0, st>>>(k);
        else stk_attn_decode_join_kernel<uint16_t><<<dim3(a.B, a.H), 128, 0, st>>>(k);
      });
    return;
  }
  if (!two && vra_stack_latent_prefill(a, dtype, stream)) return;
  if (vra_stack_prompt_attention(a, dtype, stream)) return;
  if (dtype == VRA_BF16 && a.dim % 8 == 0 && a.vdim % 16 == 0 && a.dim <= 256 && a.vdim <= 256 && a.ldq % 8 == 0 && ((uintptr_t)a.q % 16 == 0) && a.BS % 32 == 0 &&
      a.k_ld % 8 == 0 && a.v_ld % 8 == 0 && ((uintptr_t)a.vc % 16 == 0)) {
    dim3 grid((a.max_q + 63) / 64, a.B, a.H);
#define STK_PFMN(DCV, VTV, MV) launch_checked("stack attention (prefill, mfma)", [&] { stk_attn_prefill_mfma_kernel<DCV, VTV, MV><<<grid, 256 * MV, 0, st>>>(a); })
#define STK_PFM(DCV, VTV) STK_PFMN(DCV, VTV, 1)
    if (two) {
      if (a.dim <= 64 && a.vdim <= 64) STK_PFMN(2, 4, 2);
      else if (a.dim <= 64 && a.vdim <= 128) STK_PFMN(2, 8, 2);
      else if (a.dim <= 128 && a.vdim <= 128) STK_PFMN(4, 8, 2);
      else if (a.dim <= 128) STK_PFMN(4, 16, 2);
      else STK_PFMN(8, 16, 2);
    } else if (a.dim <= 64 && a.vdim <= 64) STK_PFM(2, 4);
    else if (a.dim <= 128 && a.vdim <= 128) STK_PFM(4, 8);
    else if (a.vdim <= 192) STK_PFM(8, 12);  // (a latent cache's rows: 192 value channels do not pay for 256)
    else STK_PFM(8, 16);
#undef STK_PFM
#undef STK_PFMN
    return;
  }
  auto need = [&](int kt) { return ((size_t)STK_QT * dm + (size_t)kt * (dm + 1) + (size_t)kt * a.vdim + (size_t)a.maps * STK_QT * kt) * sizeof(float); };
  dim3 grid((a.max_q + STK_QT - 1) / STK_QT, a.B, a.H);
  const int kt = need(64) <= 64 * 1024 ? 64 : (need(32) <= 64 * 1024 ? 32 : 16);
  const size_t lds = need(kt);
  VRA_CHECK_ARG(lds <= 160 * 1024, "stack attention: head does not fit LDS");
#define STK_PFM2(TT, KTV, NRV, MV)                                                                                                                \
  do {                                                                                                                                            \
    if (lds > 64 * 1024) (void)hipFuncSetAttribute((const void*)stk_attn_prefill_kernel<TT, KTV, NRV, MV>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024); \
    launch_checked("stack attention (prefill)", [&] { stk_attn_prefill_kernel<TT, KTV, NRV, MV><<<grid, 256, lds, st>>>(a); });                     \
  } while (0)
#define STK_PFN(TT, KTV, NRV)              \
  do {                                     \
    if (two) STK_PFM2(TT, KTV, NRV, 2);    \
    else STK_PFM2(TT, KTV, NRV, 1);        \
  } while (0)
#define STK_PF(TT, KTV)                      \
  do {                                       \
    if (a.vdim <= 256) STK_PFN(TT, KTV, 4);  \
    else STK_PFN(TT, KTV, 8);                \
  } while (0)
  if (dtype == VRA_F32) {
    if (kt == 64) STK_PF(float, 64);
    else if (kt == 32) STK_PF(float, 32);
    else STK_PF(float, 16);
  } else {
    if (kt == 64) STK_PF(uint16_t, 64);
    else if (kt == 32) STK_PF(uint16_t, 32);
    else STK_PF(uint16_t, 16);
  }
#undef STK_PF
#undef STK_PFN
#undef STK_PFM2
}

// ================================================================================================ C entry points (one operator each)
extern "C" void vra_stack_op_embed_sinpos(const uint32_t* ids, const int64_t* positions, const void* embed, const float* inv_freq, float* x, int32_t T,
                                          int32_t W, int32_t V, int32_t dtype, int64_t stream) {
  vra_stack_embed_sinpos(ids, positions, embed, inv_freq, x, T, W, V, dtype, stream);
}
extern "C" void vra_stack_op_group_norm(const float* x, const float* w, void* h, int32_t T, int32_t W, int32_t groups, float eps, const void* router_w,
                                        int32_t n_router, int32_t top, int32_t gate_row, int32_t* pair_expert, float* pair_weight, float* gate_out,
                                        int32_t dtype, int64_t stream) {
  StkNormArgs a;
  a.x = x, a.w = w, a.h = h, a.T = T, a.W = W, a.groups = groups, a.eps = eps;
  a.router_w = router_w, a.n_router = n_router, a.top = top, a.gate_row = gate_row;
  a.pair_expert = pair_expert, a.pair_weight = pair_weight, a.gate_out = gate_out;
  vra_stack_group_norm(a, dtype, stream);
}
extern "C" void vra_stack_op_gemm(const void* a, int32_t lda, const void* w, int64_t w_group_stride, void* out, int32_t ldo, int32_t out_f32, int32_t M,
                                  int32_t N, int32_t K, float alpha, const int32_t* tile_group, int32_t granule, const int32_t* a_row,
                                  const float* a_scale, const int32_t* out_row, int32_t epi, float limit, int32_t dtype, int64_t stream) {
  VRA_CHECK_ARG(!tile_group || granule == 16 || granule == 64, "stack gemm: granule must be 16 or 64");
  StkGemmArgs g;
  g.a = a, g.lda = lda, g.w = w, g.w_group_stride = w_group_stride, g.out = out, g.ldo = ldo, g.out_f32 = out_f32, g.M = M, g.N = N, g.K = K;
  g.alpha = alpha, g.tile_group = tile_group, g.granule = granule, g.a_row = a_row, g.a_scale = a_scale, g.out_row = out_row, g.epi = epi, g.limit = limit;
  vra_stack_gemm(g, dtype, stream);
}
extern "C" void vra_stack_op_gemm_kv(const void* a, int32_t lda, const void* w, void* out, int32_t ldo, void* kc, void* vc, const int64_t* slots, int32_t M, int32_t N, int32_t K,
                                     int32_t kv_from, int32_t kv_k, int32_t dtype, int64_t stream) {
  vra_stack_op_gemm_kv_tile(0, a, lda, w, out, ldo, kc, vc, slots, M, N, K, kv_from, kv_k, dtype, stream);
}
extern "C" void vra_stack_op_gemm_kv_tile(int32_t tile, const void* a, int32_t lda, const void* w, void* out, int32_t ldo, void* kc, void* vc, const int64_t* slots, int32_t M,
                                          int32_t N, int32_t K, int32_t kv_from, int32_t kv_k, int32_t dtype, int64_t stream) {
  VRA_CHECK_ARG(slots, "stack gemm: cache columns without slots");
  StkGemmArgs g;
  g.a = a, g.lda = lda, g.w = w, g.out = out, g.ldo = ldo, g.M = M, g.N = N, g.K = K, g.tile = tile;
  g.kv_slot = slots, g.kv_kc = kc, g.kv_vc = vc, g.kv_from = kv_from, g.kv_k = kv_k;
  vra_stack_gemm(g, dtype, stream);
}
extern "C" void vra_stack_op_gemm_tile(int32_t tile, const void* a, int32_t lda, const void* w, int64_t w_group_stride, void* out, int32_t ldo, int32_t out_f32,
                                       int32_t M, int32_t N, int32_t K, const int32_t* tile_group, const int32_t* a_row, int32_t a_rows,
                                       const int32_t* out_row, int32_t epi, float limit, int64_t stream) {
  VRA_CHECK_ARG(tile != 0, "stack gemm: no such tile for this product");
  StkGemmArgs g;
  g.a = a, g.lda = lda, g.w = w, g.w_group_stride = w_group_stride, g.out = out, g.ldo = ldo, g.out_f32 = out_f32, g.M = M, g.N = N, g.K = K;
  g.tile_group = tile_group, g.granule = (tile >> 4) * 64, g.a_row = a_row, g.a_rows = a_rows, g.out_row = out_row, g.epi = epi, g.limit = limit, g.tile = tile;
  vra_stack_gemm(g, VRA_BF16, stream);
}
extern "C" void vra_stack_op_moe_sort(const int32_t* pair_expert, const float* pair_weight, int32_t P, int32_t top, int32_t n_groups, int32_t granule,
                                      int32_t max_rows, int32_t* row_token, float* row_scale, int32_t* row_pair, int32_t* tile_group, int64_t stream) {
  VRA_CHECK_ARG(granule == 16 || granule == 64, "stack moe sort: granule must be 16 or 64");
  vra_stack_moe_sort(pair_expert, pair_weight, P, top, n_groups, granule, max_rows, row_token, row_scale, row_pair, tile_group, stream);
}
extern "C" void vra_stack_op_gated_act(const float* gu, void* out, int32_t M, int32_t F, float limit, float act_alpha, int32_t dtype, int64_t stream) {
  vra_stack_gated_act(gu, out, M, F, limit, act_alpha, dtype, stream, 0);
}
extern "C" void vra_stack_op_polynorm(const float* z, void* out, const float* coef, int32_t M, int32_t F, float eps, int32_t dtype, int64_t stream) {
  vra_stack_polynorm(z, out, coef, M, F, eps, dtype, stream);
}
extern "C" void vra_stack_op_residual_combine(float* x, const float* o, const float* p1, int32_t n1, const float* p2, const float* gate, float mult,
                                              int32_t T, int32_t W, int64_t stream) {
  vra_stack_residual_combine(x, o, p1, n1, p2, gate, mult, T, W, stream);
}
extern "C" void vra_stack_op_kv_store(const void* k, const void* v, int32_t ld, void* kc, void* vc, const int64_t* slots, int32_t T, int32_t kdim,
                                      int32_t vdim, int32_t dtype, int64_t stream) {
  vra_stack_kv_store(k, v, ld, kc, vc, slots, T, kdim, vdim, dtype, stream);
}
extern "C" void vra_stack_op_attention(const void* q, int32_t ldq, void* out, const void* kc, const void* vc, const int64_t* positions,
                                       const uint32_t* block_tables, const uint32_t* context_lens, const uint32_t* cu_q, int32_t B, int32_t T,
                                       int32_t max_q, int32_t H, int32_t G, int32_t dim, int32_t vdim, int32_t BS, int32_t max_blocks, float scale,
                                       float softcap, float temp_coef, int32_t temp_every, int32_t dtype, int64_t stream) {
  StkAttnArgs a;
  a.q = q, a.ldq = ldq, a.out = out, a.kc = kc, a.vc = vc, a.positions = positions, a.block_tables = block_tables, a.context_lens = context_lens;
  a.cu_q = cu_q, a.B = B, a.T = T, a.max_q = max_q, a.H = H, a.G = G, a.dim = dim, a.vdim = vdim, a.BS = BS, a.max_blocks = max_blocks;
  a.scale = scale, a.softcap = softcap, a.temp_coef = temp_coef, a.temp_every = temp_every;
  vra_stack_attention(a, dtype, stream);
}
// the matrix product with row groups and the element-wise epilogues: activation (epi 2), bias, soft cap
extern "C" void vra_stack_op_gemm_post(const void* a, int32_t lda, const void* w, int64_t w_group_stride, void* out, int32_t ldo, int32_t out_f32, int32_t M,
                                       int32_t N, int32_t K, float alpha, const float* bias, const int32_t* tile_group, int32_t granule, const int32_t* a_row,
                                       const int32_t* out_row, int32_t epi, int32_t act, float softcap, int32_t dtype, int64_t stream) {
  VRA_CHECK_ARG(!tile_group || granule == 16 || granule == 64, "stack gemm: granule must be 16 or 64");
  StkGemmArgs g;
  g.a = a, g.lda = lda, g.w = w, g.w_group_stride = w_group_stride, g.out = out, g.ldo = ldo, g.out_f32 = out_f32, g.M = M, g.N = N, g.K = K;
  g.alpha = alpha, g.bias = bias, g.tile_group = tile_group, g.granule = granule, g.a_row = a_row, g.out_row = out_row, g.epi = epi, g.act = act;
  g.softcap = softcap;
  vra_stack_gemm(g, dtype, stream);
}
// two maps per head over the same values, combined and normed (decode form: with scratch the key range in `splits` parts)
extern "C" void vra_stack_op_attention_differential(const void* q, int32_t ldq, void* out, const void* kc, const void* vc, const int64_t* positions,
                                                    const uint32_t* block_tables, const uint32_t* context_lens, const uint32_t* cu_q, int32_t B, int32_t T,
                                                    int32_t max_q, int32_t H, int32_t G, int32_t dim, int32_t vdim, int32_t BS, int32_t max_blocks,
                                                    float scale, float lambda, float eps, float out_scale, float* scratch, int64_t scratch_bytes,
                                                    int32_t splits, int32_t dtype, int64_t stream) {
  StkAttnArgs a;
  a.q = q, a.ldq = ldq, a.out = out, a.kc = kc, a.vc = vc, a.positions = positions, a.block_tables = block_tables, a.context_lens = context_lens;
  a.cu_q = cu_q, a.B = B, a.T = T, a.max_q = max_q, a.H = H, a.G = G, a.dim = dim, a.vdim = vdim, a.BS = BS, a.max_blocks = max_blocks;
  a.scale = scale, a.maps = 2, a.diff_lambda = lambda, a.diff_eps = eps, a.diff_scale = out_scale;
  a.scratch = scratch, a.scratch_bytes = (size_t)scratch_bytes, a.splits = splits;
  vra_stack_attention(a, dtype, stream);
}
