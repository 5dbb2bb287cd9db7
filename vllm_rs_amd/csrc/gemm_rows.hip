// gemm_rows.hip — the row-major prompt GEMM (gemm_rows.cuh) for unquantised decoder layers: q | k | v in one launch, o / down with the residual
// added, gate / up with SiLU * mul (the reference's dense Linear and MLP, src/models/layers/mlp.rs:451-469).
#include "gemm_rows_launch.h"

#include <algorithm>

namespace {

// the roundings of the other dense kernels: rnd(sum), + bias rounded, SiLU rounded, + residual rounded; f32 output: the rounded value
template <class DT, bool DUAL>
struct DenseRowsEpi {
  GemmRowsOut o[GR_MAX_SEG];
  const uint16_t* bias_up;
  const uint16_t* residual;
  int res_ld, out_f32;
  static constexpr bool mixes = true;  // (with gemm_rows_mixed_kernel)
  struct Row {};
  __device__ __forceinline__ Row row(int) const { return {}; }
  template <class F>
  __device__ __forceinline__ void in_form(int, int, int, const F& f) const {
    f(std::integral_constant<int, 0>{}, Row{});
  }
  template <int>
  __device__ __forceinline__ void store(int m, const Row&, const Row&, int seg, int n0, int N, int q4, const f32x4 (&acc)[4]) const {
    constexpr int NJ = DUAL ? 2 : 4;
    const GemmRowsOut* const s = seg == 0 ? &o[0] : (seg == 1 ? &o[1] : &o[2]);
    const int no = DUAL ? n0 / 2 : n0, lim = DUAL ? N / 2 : N;
    const uint16_t* const b = static_cast<const uint16_t*>(s->bias);
    float y[NJ][4];
#pragma unroll
    for (int j = 0; j < NJ; j++) {
      float bs[4] = {0.f, 0.f, 0.f, 0.f}, bu[4] = {0.f, 0.f, 0.f, 0.f};
      const int n = min(no + j * 16 + q4 * 4, lim - 4);
      if (b) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(b + n);
        bs[0] = DT::to_f32((uint16_t)(v[0] & 0xffffu)), bs[1] = DT::to_f32((uint16_t)(v[0] >> 16));
        bs[2] = DT::to_f32((uint16_t)(v[1] & 0xffffu)), bs[3] = DT::to_f32((uint16_t)(v[1] >> 16));
      }
      if (DUAL && bias_up) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(bias_up + n);
        bu[0] = DT::to_f32((uint16_t)(v[0] & 0xffffu)), bu[1] = DT::to_f32((uint16_t)(v[0] >> 16));
        bu[2] = DT::to_f32((uint16_t)(v[1] & 0xffffu)), bu[3] = DT::to_f32((uint16_t)(v[1] >> 16));
      }
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float t = rnd_dt<DT>(acc[DUAL ? 2 * j : j][e]);
        if (b) t = rnd_dt<DT>(t + bs[e]);
        if (DUAL) {
          float u = rnd_dt<DT>(acc[2 * j + 1][e]);
          if (bias_up) u = rnd_dt<DT>(u + bu[e]);
          t = rnd_dt<DT>(t / (1.0f + expf(-t))) * u;
        }
        y[j][e] = t;
      }
    }
    if (out_f32) {
      if (m < 0) return;
      float* const of = static_cast<float*>(s->out) + (size_t)m * s->ld;
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        const int n = no + j * 16 + q4 * 4;
        if (n < lim) *reinterpret_cast<f32x4*>(of + n) = f32x4{rnd_dt<DT>(y[j][0]), rnd_dt<DT>(y[j][1]), rnd_dt<DT>(y[j][2]), rnd_dt<DT>(y[j][3])};
      }
      return;
    }
    u32x2 v[NJ];
#pragma unroll
    for (int j = 0; j < NJ; j++) v[j] = u32x2{DT::pack2(y[j][0], y[j][1]), DT::pack2(y[j][2], y[j][3])};
    gr_gather_columns(v);  // whole 16-byte pieces of a row
    if (m < 0) return;
    uint16_t* const oh = static_cast<uint16_t*>(s->out) + (size_t)m * s->ld;
#pragma unroll
    for (int h = 0; h < NJ / 2; h++) {
      const int n = no + q4 * (NJ * 4) + h * 8;
      if (n >= lim) continue;
      u32x4 p = {v[2 * h][0], v[2 * h][1], v[2 * h + 1][0], v[2 * h + 1][1]};
      if (residual) {
        float f[8], r[8];
        unpack8<DT>(p, f);
        unpack8<DT>(*reinterpret_cast<const u32x4*>(residual + (size_t)m * res_ld + n), r);
#pragma unroll
        for (int e = 0; e < 8; e++) f[e] += r[e];
        p = pack8<DT>(f);
      }
      *reinterpret_cast<u32x4*>(oh + n) = p;
    }
  }
};

}  // namespace

// x rows and every tensor within 31-bit byte offsets, whole 64-steps of K, 16-byte pieces in all rows
bool vra_gemm_rows_takes(const GemmRowsCall& c) {
  if (c.M <= 32 || c.K % 64 || (int64_t)c.M * c.x_ld * 2 >= 0x7FFF0000ll || c.x_ld % 8 || (uintptr_t)c.x % 16) return false;
  for (int s = 0; s < c.nseg; s++)
    if ((int64_t)c.n[s] * c.K * 2 >= 0x7FFF0000ll || c.n[s] % 16 || (uintptr_t)c.w[s] % 16 || (uintptr_t)c.bias[s] % 8) return false;
  for (int s = 0; s < (c.dual ? 1 : c.nseg); s++)
    if ((uintptr_t)c.out[s] % 16 || c.out_ld[s] % 8) return false;
  if (c.residual && ((uintptr_t)c.residual % 16 || c.res_ld % 8 || c.out_f32)) return false;
  return true;
}
// then time against time: gemm_rows_tile's here, kernel B at 250 TFLOP/s on whole 64-row blocks behind ~10 us of exchange
// between its K slices
bool vra_gemm_rows_fits(const GemmRowsCall& c) {
  if (!vra_gemm_rows_takes(c)) return false;
  int n[GR_MAX_SEG] = {};
  double b_us = 0.0;
  for (int s = 0; s < c.nseg; s++) n[s] = c.n[s], b_us += 10.0 + 2.0 * ((c.M + 63) / 64 * 64) * (double)c.n[s] * c.K / 250e6;
  if (c.dual) n[0] = 2 * c.n[0];
  double us = 0.0;
  (void)gemm_rows_tile(c.M, n, c.dual ? 1 : c.nseg, 1, c.K, 0, &us);
  return us < b_us;
}

void vra_launch_gemm_rows(const GemmRowsCall& c, int dtype, int64_t stream) {
  GemmRowsArgs a;
  a.x = c.x, a.x_ld = c.x_ld, a.M = c.M, a.K = c.K;
  a.nseg = c.dual ? 1 : c.nseg;
  for (int s = 0; s < c.nseg; s++) a.w[s] = c.w[s], a.n[s] = c.n[s];
  if (c.dual) a.n[0] = 2 * c.n[0];
  const int tile = c.tile ? c.tile : (a.nseg == 1 ? gemm_rows_tiles(c.M, a.n[0], c.K) : gemm_rows_tile(c.M, a.n, a.nseg, 1, c.K));
  auto go = [&](auto dt, auto dual) {
    DenseRowsEpi<decltype(dt), decltype(dual)::value> e = {};
    for (int s = 0; s < a.nseg; s++) e.o[s] = GemmRowsOut{c.out[s], c.bias[s], c.out_ld[s]};
    e.bias_up = c.dual ? static_cast<const uint16_t*>(c.bias[1]) : nullptr;
    e.residual = static_cast<const uint16_t*>(c.residual), e.res_ld = c.res_ld, e.out_f32 = c.out_f32;
    gemm_rows_launch<decltype(dt), decltype(dual)::value>(a, e, tile, 1, reinterpret_cast<hipStream_t>(stream));
  };
  if (dtype == VRA_BF16) c.dual ? go(BF16{}, std::true_type{}) : go(BF16{}, std::false_type{});
  else c.dual ? go(F16{}, std::true_type{}) : go(F16{}, std::false_type{});
}

extern "C" void vra_dense_gemm_tile(int32_t tile, const void* x, const void* const* w, const void* const* bias, const int32_t* n, int32_t nseg,
                                    int32_t pair, const void* residual, void* const* out, int32_t out_f32, int32_t m, int32_t k, int32_t dtype,
                                    int64_t stream) {
  VRA_CHECK_ARG(x && w && bias && n && out && m > 0 && k > 0 && (pair ? nseg == 2 && n[0] == n[1] : nseg >= 1 && nseg <= GR_MAX_SEG), "dense gemm tile: null pointer or bad segments");
  VRA_CHECK_ARG((dtype == VRA_BF16 || dtype == VRA_F16) && (gemm_rows_has_tile(tile, k) || gemm_rows_has_tiles(tile, m, pair ? 2 * n[0] : (nseg == 1 ? n[0] : 0), k)) && !(pair && residual), "dense gemm tile: no such form");
  GemmRowsCall r;
  r.x = x, r.x_ld = k, r.M = m, r.K = k, r.nseg = nseg, r.dual = pair != 0, r.tile = tile, r.out_f32 = out_f32, r.residual = residual, r.res_ld = n[0];
  for (int s = 0; s < nseg; s++) {
    VRA_CHECK_ARG(w[s] && n[s] > 0 && (out[s] || (pair && s)), "dense gemm tile: null pointer or bad segments");
    r.w[s] = w[s], r.n[s] = n[s], r.bias[s] = bias[s], r.out[s] = out[s], r.out_ld[s] = n[s];
  }
  VRA_CHECK_ARG(vra_gemm_rows_takes(r), "dense gemm tile: a shape or an alignment that these tiles do not take");
  vra_launch_gemm_rows(r, dtype, stream);
}

extern "C" int32_t vra_dense_gemm_tiles_choice(int32_t m, int32_t n, int32_t k) { return m > 0 && n > 0 && k > 0 ? gemm_rows_tiles(m, n, k) : 0; }
extern "C" int32_t vra_dense_gemm_tile_choice(int32_t m, const int32_t* n, int32_t nseg, int32_t k) {
  return m > 0 && n && nseg >= 1 && nseg <= GR_MAX_SEG && k > 0 ? gemm_rows_tile(m, n, nseg, 1, k) : 0;
}
