// gemm_q4_mid.hip — kernel M (gemm_q4_mid.cuh): which launches take it, and the launch (the reference's int4 linear layers,
// src/models/layers/linear.rs; its prompts go through the Marlin kernel, src/models/layers/others.rs).
#include <algorithm>
#include <type_traits>

#include "gemm_launch.h"
#include "gemm_q4_mid.cuh"
#include "scratch.h"

static const size_t kXsum = (size_t)16 << 20;  // the end of the slab region holds the row sums
static const int kLds = 160 * 1024;

static int mid_cus() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 256;
  static int cus[64] = {};
  if (dev < 64 && cus[dev]) return cus[dev];
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
  if (dev < 64) cus[dev] = n;
  return n;
}

int vra_gemm_q4_mid_plan(bool dual, int M, int cols, int K, int group_size, const GemmDArgs* segs, bool awq, bool summed, double* us) {
  if (M < 64 || K % 128 || cols % 16) return 0;
  if (group_size > 0 && group_size < K && (group_size < 128 || (group_size & (group_size - 1)))) return 0;
  if (segs && segs->nseg > 1) {  // a wave's columns must not straddle tensors
    if (dual || segs->residual || segs->N % 64) return 0;
    for (int i = 0; i + 1 < segs->nseg; i++)
      if (segs->xseg[i].n % 64) return 0;
  }
  if (!vra_gemm_q4_big_xsum_table(M, K)) return 0;
  const int cus = mid_cus(), KT = K >> 7, gx = dual ? (cols + 63) / 64 : (cols + 127) / 128;
  const int rb = (M + 159) / 160, mb = std::max(2, (M + 32 * rb - 1) / (32 * rb));
  const long tiles = (long)gx * ((M + 32 * mb - 1) / (32 * mb));
  const bool split = vra_scratch_slabs() && vra_scratch_counters();
  int best = 0;
  for (int S = 1; S <= 16; S *= 2) {
    if (S > 1 && (!split || KT < 2 * S || tiles * S > cus)) break;  // the whole grid is resident: the owners find their slices running
    if (S > 1 && ((size_t)S * tiles * 2 * mb * GM_THREADS * 16 > vra_scratch_slab_bytes() - kXsum || (size_t)tiles * S * 16 > vra_scratch_counter_count())) break;
    // Fitted to the Llama-3-8B and Qwen2-7B shapes at 64..760 rows (us): a launch 3 and 5.5 a round of workgroups; a k-tile as in `tile`, symmetric
    // codes and AWQ (which unpacks its zero points and takes them off a column at a time): gate/up of 4096 x 14336, one round of 224 workgroups: 33 / 39 /
    // 46 / 53 at MB 2..5; down of 18944 x 3584, 256 rows in 4 slices: 65 (with the row halves a barrier apart symmetric codes take 5 % less: the
    // lines to the other kernels stayed where they were); a slab of the exchange 0.43 per 32 rows beyond the first; two
    // workgroups of MB 2 share a CU, 13 % faster than one after the other; 4 for the row sums where no norm's launch leaves them
    static const double tile[2][6] = {{0, 0, 0.76, 0.93, 1.17, 1.44}, {0, 0, 0.82, 1.00, 1.28, 1.57}};
    const double rounds = (double)((tiles * S + cus - 1) / cus), q = rounds * (mb == 2 && rounds > 1 ? 0.87 : 1.0);
    const double t = 3.0 + 5.5 * rounds + q * ((KT + S - 1) / S) * tile[awq][mb] + (S > 1 ? 0.43 * (mb - 1) * (S - 1) : 0.0) + (summed ? 0.0 : 4.0);
    if (!best || t < *us) best = mb | (S << 8), *us = t;
  }
  return best;
}

template <class DT, bool DUAL, bool AWQ, int MB>
static void launch_t(const GemmDArgs& a, dim3 grid, hipStream_t st) {
  static uint64_t seen = 0;  // per device: function attributes belong to the device current at the call
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (!((__atomic_load_n(&seen, __ATOMIC_RELAXED) >> (dev & 63)) & 1)) {
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_q4_mid_kernel<DT, DUAL, AWQ, MB>), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    __atomic_fetch_or(&seen, 1ull << (dev & 63), __ATOMIC_RELAXED);
  }
  gemm_q4_mid_kernel<DT, DUAL, AWQ, MB><<<grid, GM_THREADS, gemm_q4_mid_lds_bytes(MB), st>>>(a);
}
template <class DT, bool DUAL>
static void launch_mb(const GemmDArgs& a, bool awq, int mb, dim3 grid, hipStream_t st) {
  auto go = [&](auto m) {
    constexpr int MB = decltype(m)::value;
    awq ? launch_t<DT, DUAL, true, MB>(a, grid, st) : launch_t<DT, DUAL, false, MB>(a, grid, st);
  };
  if (mb == 2) go(std::integral_constant<int, 2>{});
  else if (mb == 3) go(std::integral_constant<int, 3>{});
  else if (mb == 4) go(std::integral_constant<int, 4>{});
  else go(std::integral_constant<int, 5>{});
}

void vra_launch_gemm_q4_mid(GemmDArgs a, bool dual, bool awq, int plan, int dtype, int64_t stream) {
  const int mb = plan & 0xff, sk = plan >> 8;
  const int cols = a.nseg > 1 ? a.xseg[a.nseg - 2].blk_start * 16 + a.xseg[a.nseg - 2].n : a.N;
  const dim3 grid(dual ? (cols + 63) / 64 : (cols + 127) / 128, (a.M + 32 * mb - 1) / (32 * mb), sk);
  a.splitk = sk;
  if (sk > 1) {
    a.slabs = vra_scratch_slabs(), a.counters = vra_scratch_counters(), a.err = vra_scratch_error_word();
    if (!a.slabs || !a.counters) {
      vra_set_error("gemm_q4_mid: split-K scratch unavailable");
      return;
    }
  }
  hipStream_t st = as_stream(stream);
  if (dtype == VRA_BF16) dual ? launch_mb<BF16, true>(a, awq, mb, grid, st) : launch_mb<BF16, false>(a, awq, mb, grid, st);
  else dual ? launch_mb<F16, true>(a, awq, mb, grid, st) : launch_mb<F16, false>(a, awq, mb, grid, st);
}
