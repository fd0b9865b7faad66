// Weight-streaming GEMM for decode batches (up to 64 input rows):  y[m, n] = bf16( sum_k x[m, k] * w[n, k] ).
//
// The weights are read once, in whole cache lines: a load instruction covers 4 weight rows x 256
// contiguous bytes (16 lanes x 16 bytes per row), never a fraction of a line that another
// instruction would have to find in a cache again.  That is the layout a matrix-vector kernel
// streams in, not the one the matrix cores want (there a lane feeds 8 consecutive k of ITS OWN row,
// 16 different rows per instruction), so every chunk takes one trip through a wave-private piece of
// LDS: written row-major as it arrives, read back as v_mfma_f32_16x16x32_bf16 A fragments.  Rows
// are padded by 16 bytes, which puts the 16 rows of a fragment read on 16 different bank groups.
// No workgroup barrier is involved: the LDS unit executes a wave's instructions in order.
//
// A workgroup (4 waves, one per SIMD, so each has the whole register budget) owns a band of up to
// 32 weight rows -- the number of rows is chosen so that every CU gets the same share -- and its
// waves walk K in 128-element chunks, in turn or, where that measured faster, a slice of K each
// (stream_band).  Each wave keeps 4 chunks of weights (32 KiB) in flight in registers, 128 KiB per CU.
// The input rows come from L2 straight into B-fragment layout.  The waves' partial sums meet in LDS and
// are added in a fixed order.
//
// Two projections that read the same layer input can share one launch (the band index selects the
// projection), and a projection whose weight holds [up; gate] rows can take the band as row PAIRS
// and store bf16(bf16(silu(g)) * u) instead of u and g.  The fused q/k/v projection of a decode step
// can rotate q and k and put k and v into the cache on its way out (what lr_rope_kv_write does).
#include "stream_band.h"

namespace {

template <int MT, int UNITS, bool W8, bool XL, int UROWS, bool DEEP, bool X8>
__global__ __launch_bounds__(NWV * 64, MT == 16 ? 2 : 0) void k_stream_gemm(const Proj p0, const Proj p1, const int M) {
  extern __shared__ __attribute__((aligned(16))) u16 sg_smem[];
  const bool second = (int)blockIdx.x >= p0.nwg;
  const Proj p = second ? p1 : p0;
  stream_band<MT, UNITS, W8, XL, false, RESID_NONE, NWV, UROWS, DEEP, X8>(p, M, second ? (int)blockIdx.x - p0.nwg : (int)blockIdx.x, sg_smem);
}

template <int MT, int UNITS, bool W8 = false, bool XL = (MT >= XLDS_MIN_MT), int UROWS = 16, bool X8 = (MT == 16 && !XL && !W8), bool DEEP = (MT == 16)>
static int launch_units(Proj& a, Proj& b, int M, hipStream_t s) {
  const size_t na = stream_band_norm_bytes(a, M), nb = stream_band_norm_bytes(b, M), lds = stream_band_lds_bytes<MT, UNITS, W8, XL>() + (na > nb ? na : nb);
  static std::atomic<unsigned long long> lds_raised{0};
  if (!lr_raise_lds_limit(reinterpret_cast<const void*>(&k_stream_gemm<MT, UNITS, W8, XL, UROWS, DEEP, X8>), lds, lds_raised)) return LR_E_LAUNCH;
  k_stream_gemm<MT, UNITS, W8, XL, UROWS, DEEP, X8><<<dim3((unsigned)(a.nwg + b.nwg)), dim3(NWV * 64), lds, s>>>(a, b, M);
  return LR_OK;
}

template <int MT>
static int launch(Proj& a, Proj& b, int M, int units, hipStream_t s) {
  if (MT == 16 && M >= XLDS_M16_FROM)  // the 16-row band with its inputs read in whole lines
    return units == 2 ? launch_units<MT, 2, false, true>(a, b, M, s) : launch_units<MT, 1, false, true>(a, b, M, s);
  // bands of at most 8 weight rows load half a unit (8 input rows, 2048 x 2048: 4.83 -> 4.10 us; with 9 to 16 input rows,
  // 1280 x 8192, nothing moves: 10.0 / 10.1)
  if (MT == 16 && units == 1 && a.rpw <= 8 && b.rpw <= 8) return launch_units<16, 1, false, false, 8>(a, b, M, s);
  return units == 2 ? launch_units<MT, 2>(a, b, M, s) : launch_units<MT, 1>(a, b, M, s);
}

template <bool X8>
static int launch_fp8(Proj& a, Proj& b, int M, int units, hipStream_t s) {
  if (units == 2) return launch_units<16, 2, true, false, 16, X8>(a, b, M, s);
  if (a.rpw <= 8 && b.rpw <= 8) return launch_units<16, 1, true, false, 8, X8>(a, b, M, s);
  return launch_units<16, 1, true, false, 16, X8>(a, b, M, s);
}

// one 16-row unit per workgroup when every CU still gets a band that way; row pairs always take two units
static int pick_units_and_plan(Proj* pr, int n_proj, int M, int ncu) {
  bool any_pair = false, all_thin = true;
  for (int i = 0; i < n_proj; ++i) {
    any_pair = any_pair || pr[i].pair_off != 0;
    if (pr[i].N > 16 * ncu) all_thin = false;
  }
  const int units = (any_pair || !all_thin) ? 2 : 1;
  for (int i = 0; i < n_proj; ++i) plan(pr[i], M, pr[i].pair_off ? 16 : 16 * units, ncu);
  return units;
}

}  // namespace

extern "C" int lr_linear_multi(const lr_projection_t* proj, int n_proj, int M, lr_stream_t stream) {
  return lr_linear_multi_normed(proj, nullptr, n_proj, M, stream);
}

extern "C" int lr_linear_multi_normed(const lr_projection_t* proj, const lr_row_norm_t* norms, int n_proj, int M, lr_stream_t stream) {
  if (proj == nullptr) return LR_E_NULL;
  if (n_proj < 1 || n_proj > 2 || M < 1) return LR_E_SHAPE;
  if (M > 64) return LR_E_UNSUPPORTED;
  Proj pr[2] = {};
  for (int i = 0; i < n_proj; ++i) {
    int rc = sb_fill_projection(proj[i], pr[i]);
    if (rc == LR_OK && norms) rc = sb_fill_norm(norms + i, pr[i]);
    if (rc != LR_OK) return rc;
    if (pr[i].norm_sums && M > LR_ROW_NORM_MAX_ROWS) return LR_E_UNSUPPORTED;
  }
  const int ncu = lr_num_cus();
  if (ncu < 1) return LR_E_LAUNCH;
  const int units = pick_units_and_plan(pr, n_proj, M, ncu);
  for (int i = 0; i < n_proj; ++i)
    if (pr[i].fold_sums && pr[i].nwg < M) return LR_E_UNSUPPORTED;   // (a row per workgroup)
  hipStream_t s = (hipStream_t)stream;
  const int rc = M <= 16 ? launch<16>(pr[0], pr[1], M, units, s)
                 : (M <= 32 ? launch<32>(pr[0], pr[1], M, units, s) : launch<64>(pr[0], pr[1], M, units, s));
  return rc != LR_OK ? rc : lr_launch_status();
}

namespace {

template <int MT, int UNITS, bool XL>
__global__ __launch_bounds__(NWV * 64, MT == 16 ? 2 : 0) void k_stream_residual(const Proj p, const int M, const BandResidual rs) {
  extern __shared__ __attribute__((aligned(16))) u16 sg_smem[];
  stream_band<MT, UNITS, false, XL, false, RESID_TANH, NWV, 16, MT == 16, MT == 16 && !XL>(p, M, blockIdx.x, sg_smem, nullptr, 1, rs);
}

template <int MT, int UNITS, bool XL>
int launch_residual_units(const Proj& p, int M, const BandResidual& rs, hipStream_t s) {
  constexpr size_t lds = stream_band_lds_bytes<MT, UNITS, false, XL>();
  static std::atomic<unsigned long long> raised{0};
  if (!lr_raise_lds_limit(reinterpret_cast<const void*>(&k_stream_residual<MT, UNITS, XL>), lds, raised)) return LR_E_LAUNCH;
  k_stream_residual<MT, UNITS, XL><<<dim3((unsigned)p.nwg), dim3(NWV * 64), lds, s>>>(p, M, rs);
  return lr_launch_status();
}
template <int MT, bool XL>
int launch_residual(const Proj& p, int M, int units, const BandResidual& rs, hipStream_t s) {
  return units == 2 ? launch_residual_units<MT, 2, XL>(p, M, rs, s) : launch_residual_units<MT, 1, XL>(p, M, rs, s);
}

}  // namespace

extern "C" int lr_linear_residual_tanh(const void* x, int64_t ldx, const void* w, int M, int N, int K, float* resid, const void* expert_out,
                                       const float* expert_weights, int top, const void* alpha, const void* gain, const void* bias,
                                       void* x_compute, lr_stream_t stream) {
  LR_REQUIRE_PTR(resid);
  LR_REQUIRE_PTR(gain);
  LR_REQUIRE_PTR(bias);
  LR_REQUIRE_PTR(x_compute);
  LR_OPTIONAL_PTR(expert_out);
  if (alpha == nullptr || (expert_out && expert_weights == nullptr)) return LR_E_NULL;
  if (M < 1 || (expert_out && top <= 0)) return LR_E_SHAPE;
  if (M > 64) return LR_E_UNSUPPORTED;
  const lr_projection_t q = {x, ldx, w, x_compute, N, N, K, LR_EPI_NONE, nullptr};
  Proj pr[1] = {};
  const int rc = sb_fill_projection(q, pr[0]);
  if (rc != LR_OK) return rc;
  const int ncu = lr_num_cus();
  if (ncu < 1) return LR_E_LAUNCH;
  const int units = pick_units_and_plan(pr, 1, M, ncu);
  const BandResidual rs = {resid, (u16*)x_compute, (const u16*)alpha, (const u16*)gain, (const u16*)bias, (const u16*)expert_out,
                           expert_weights, top};
  hipStream_t s = (hipStream_t)stream;
  if (M > 32) return launch_residual<64, true>(pr[0], M, units, rs, s);
  if (M > 16) return launch_residual<32, true>(pr[0], M, units, rs, s);
  return M >= XLDS_M16_FROM ? launch_residual<16, true>(pr[0], M, units, rs, s) : launch_residual<16, false>(pr[0], M, units, rs, s);
}

// ---- a post-norm sublayer's output projection with the residual update and what its norm needs (lr_linear_residual_rms)
//
// Such a norm is a launch between a projection into the residual and the next one out of it.  Here the band that owns a column adds
// to the residual there, and leaves the column with its gain and its share of the rows' sums of squares: the projections that follow
// divide their results (has_norm), and the next sublayer's residual update divides what it reads.  Up to 16 rows, like those.
// Bound: HBM, as the bands without; a launch of 5 us less per sublayer, some of it given back by bands that add the parts first.
// Decode steps, us, before / now: Lasivik 8B 8 rows at 1792 tokens 3693 / 3474, 3 rows 3522 / 3297, 16 rows 4129 / 3985; 1B 3 rows 888 / 819,
// 8 rows 1001 / 941, 16 rows 1080 / 1043 (in part by the bands' slices of K, see stream_band).
namespace {

struct Range {
  const void* p;
  size_t bytes;
  bool meets(const Range& r) const {
    const uintptr_t a = (uintptr_t)p, b = (uintptr_t)r.p;
    return r.p != nullptr && a < b + r.bytes && b < a + bytes;
  }
};

// (Bands of 32 columns with their inputs through LDS: one workgroup per CU, which is all that a grid of up to 8192 columns has.  Held to the
// registers of two they kept six in memory: 9 rows of 8192 x 8192 and the 16384 x 8192 behind 74.3 us, now 72.3.)
template <int UNITS, bool XL, int UROWS>
__global__ __launch_bounds__(NWV * 64, XL && UNITS == 2 ? 1 : 2) void k_stream_rms(const Proj p, const int M, const BandResidual rs) {
  extern __shared__ __attribute__((aligned(16))) u16 sg_smem[];
  stream_band<16, UNITS, false, XL, false, RESID_RMS, NWV, UROWS, true, !XL>(p, M, blockIdx.x, sg_smem, nullptr, 1, rs);
}

template <int UNITS, bool XL, int UROWS = 16>
int launch_rms(const Proj& p, int M, const BandResidual& rs, hipStream_t s) {
  const size_t lds = stream_band_lds_bytes<16, UNITS, false, XL>() + stream_band_norm_bytes(p, M);
  static std::atomic<unsigned long long> raised{0};
  if (!lr_raise_lds_limit(reinterpret_cast<const void*>(&k_stream_rms<UNITS, XL, UROWS>), lds, raised)) return LR_E_LAUNCH;
  k_stream_rms<UNITS, XL, UROWS><<<dim3((unsigned)p.nwg), dim3(NWV * 64), lds, s>>>(p, M, rs);
  return lr_launch_status();
}

}  // namespace

extern "C" int lr_linear_residual_rms_sums(int N) {
  const int ncu = lr_num_cus();
  if (N <= 0 || ncu < 1) return 0;
  Proj p{};
  p.N = N;
  pick_units_and_plan(&p, 1, 16, ncu);
  return p.nwg <= LR_ROW_NORM_MAX ? p.nwg : 0;
}

extern "C" int lr_linear_residual_rms(const void* x, int64_t ldx, const void* w, int M, int N, int K, float* resid, float scale,
                                      const lr_row_norm_t* before, const void* gain_before, const void* gain, float gain_offset,
                                      void* x_compute, float* sums, lr_stream_t stream) {
  LR_REQUIRE_PTR(resid);
  LR_REQUIRE_PTR(gain);
  LR_REQUIRE_PTR(x_compute);
  LR_OPTIONAL_PTR(gain_before);
  if (sums == nullptr || (before && (before->sums == nullptr || gain_before == nullptr))) return LR_E_NULL;
  if (before && (before->dim != N || before->fold_sums)) return LR_E_SHAPE;
  if (M < 1) return LR_E_SHAPE;
  const lr_projection_t q = {x, ldx, w, x_compute, N, N, K, LR_EPI_NONE, nullptr};
  Proj p{};
  int rc = sb_fill_projection(q, p);
  if (rc != LR_OK) return rc;
  if (M > LR_ROW_NORM_MAX_ROWS || (int64_t)M * N * 4 >= 0x7fffffff) return LR_E_UNSUPPORTED;
  // Every band reads all of x and of the parts before while others write theirs of the results.
  const int parts = lr_linear_residual_rms_sums(N);
  const Range out[3] = {{resid, (size_t)M * N * 4}, {x_compute, (size_t)M * N * 2}, {sums, (size_t)M * (parts ? parts : 1) * 4}};
  const Range in[4] = {{x, ((size_t)(M - 1) * ldx + K) * 2}, {gain, (size_t)N * 2}, {before ? before->sums : nullptr, before ? (size_t)M * before->count * 4 : 0},
                       {before ? gain_before : nullptr, (size_t)N * 2}};
  for (int i = 0; i < 3; ++i) {
    for (int j = 0; j < i; ++j)
      if (out[i].meets(out[j])) return LR_E_SHAPE;
    for (const Range& r : in)
      if (out[i].meets(r)) return LR_E_SHAPE;
  }
  if (parts == 0) return LR_E_UNSUPPORTED;
  if (before) {
    lr_row_norm_t of_input = *before;
    of_input.dim = K;   // (checked against N above: the sums are the residual's)
    rc = sb_fill_norm(&of_input, p);
    if (rc != LR_OK) return rc;
    p.norm_dim = N;
  }
  const int units = pick_units_and_plan(&p, 1, M, lr_num_cus());
  BandResidual rs{};
  rs.x = resid; rs.xc = (u16*)x_compute; rs.gain = (const u16*)gain; rs.scale = scale; rs.offset = gain_offset;
  rs.before = before ? (const u16*)gain_before : nullptr; rs.squares = sums;
  hipStream_t s = (hipStream_t)stream;
  if (M >= XLDS_M16_FROM) return units == 2 ? launch_rms<2, true>(p, M, rs, s) : launch_rms<1, true>(p, M, rs, s);
  if (units == 2) return launch_rms<2, false>(p, M, rs, s);
  return p.rpw <= 8 ? launch_rms<1, false, 8>(p, M, rs, s) : launch_rms<1, false>(p, M, rs, s);
}

// ---- a layer's output projections with the residual updates and what the next norms need of the rows (lr_linear_resid)
//
// A norm between two projections is a launch that moves next to nothing and waits for everything.  Here the workgroup that
// owns a band of columns forms both products of it, so it can update the residual there; it leaves the rows with their gains
// and its share of their sums of squares, and the next projections divide their results by the rows' root mean squares
// (stream_band: has_norm).  Bound: HBM, like the bands it replaces, whose two workgroups of four waves per CU become one of
// eight: chunks of the first weight, then of the second, are dealt round the waves.  Measured, us per launch under a
// profiler (70B rank shard, 8 rows): 8192 x (1024 | 3584) 17.0 -> 17.9 and q/k/v 8.6 -> 9.1, e4m3 11.8 -> 12.7 and 7.9 -> 9.0,
// for a norm launch of 4.8; a step, us: 70B rank shard, 8 rows 4617 -> 4403, e4m3 5 rows 3450 -> 3257; 8B 16 rows 3576 -> 3560;
// 8B parallel blocks, 6 rows 3220 -> 3114.
// Not for 17 rows and more (the 32-row band fills the register file with four waves), nor where the norm stands between a
// block's attention and its MLP: up/gate then has several bands per CU, each of which would add all the parts (12 rows of 8B
// desync blocks 3755 -> 3772), and rounding the rows once instead of twice moves near-ties of two-row batches.
namespace {

constexpr int RN_WAVES = 8;

template <int UNITS, bool W8, bool XL, int UROWS, bool X8>
__global__ __launch_bounds__(RN_WAVES * 64) void k_stream_resid(const Proj p, const int M, const ResidNorm rn) {
  extern __shared__ __attribute__((aligned(16))) u16 sg_smem[];
  stream_band<16, UNITS, W8, XL, false, RESID_NONE, RN_WAVES, UROWS, !(XL && UNITS == 2), X8, RN_WAVES, true>(p, M, blockIdx.x, sg_smem, nullptr, 1, BandResidual{}, rn);
}

template <int UNITS, bool W8, bool XL, int UROWS, bool X8>
int launch_resid_as(const Proj& p, int M, const ResidNorm& rn, hipStream_t s) {
  constexpr size_t lds = stream_band_lds_bytes<16, UNITS, W8, XL, RN_WAVES>();
  static std::atomic<unsigned long long> raised{0};
  if (!lr_raise_lds_limit(reinterpret_cast<const void*>(&k_stream_resid<UNITS, W8, XL, UROWS, X8>), lds, raised)) return LR_E_LAUNCH;
  k_stream_resid<UNITS, W8, XL, UROWS, X8><<<dim3((unsigned)p.nwg), dim3(RN_WAVES * 64), lds, s>>>(p, M, rn);
  return lr_launch_status();
}
template <int UNITS, int UROWS>
int launch_resid_rows(const Proj& p, int M, const ResidNorm& rn, hipStream_t s) {
  if (p.scales) return M <= 8 ? launch_resid_as<UNITS, true, false, UROWS, true>(p, M, rn, s) : launch_resid_as<UNITS, true, false, UROWS, false>(p, M, rn, s);
  return M >= XLDS_M16_FROM ? launch_resid_as<UNITS, false, true, UROWS, false>(p, M, rn, s) : launch_resid_as<UNITS, false, false, UROWS, true>(p, M, rn, s);
}
// bands of the columns: every CU the same number of rows
void plan_resid(int D, int ncu, int& rows, int& bands) {
  const int rounds = (D + 32 * ncu - 1) / (32 * ncu);
  rows = (D + ncu * rounds - 1) / (ncu * rounds);
  bands = (D + rows - 1) / rows;
}

}  // namespace

extern "C" int lr_linear_resid_sums(int D) {
  const int ncu = lr_num_cus();
  if (D <= 0 || ncu < 1) return 0;
  int rows, bands;
  plan_resid(D, ncu, rows, bands);
  return bands;
}

extern "C" int lr_linear_resid(const lr_linear_resid_t* d, int M, lr_stream_t stream) {
  if (d == nullptr) return LR_E_NULL;
  LR_REQUIRE_PTR(d->resid_in);
  LR_REQUIRE_PTR(d->resid_out);
  LR_REQUIRE_PTR(d->gain2);
  LR_REQUIRE_PTR(d->out2);
  const bool joint = d->joint != 0;
  if (d->sums2 == nullptr) return LR_E_NULL;
  if (!joint) {
    LR_REQUIRE_PTR(d->gain1);
    LR_REQUIRE_PTR(d->out1);
    if (d->sums1 == nullptr) return LR_E_NULL;
  }
  if (M < 1) return LR_E_SHAPE;
  if (M > LR_ROW_NORM_MAX_ROWS) return LR_E_UNSUPPORTED;
  const bool w8 = d->scales1 != nullptr;
  Proj pr[2] = {};
  for (int i = 0; i < 2; ++i) {
    int rc;
    if (w8) {
      const lr_projection_fp8_t q = {i ? d->x2 : d->x1, i ? d->ldx2 : d->ldx1, i ? d->w2 : d->w1, i ? d->scales2 : d->scales1, d->resid_out, d->D,
                                     d->D, i ? d->K2 : d->K1, LR_EPI_NONE, nullptr};
      rc = sb_fill_projection_fp8(q, pr[i]);
    } else {
      const lr_projection_t q = {i ? d->x2 : d->x1, i ? d->ldx2 : d->ldx1, i ? d->w2 : d->w1, d->resid_out, d->D, d->D, i ? d->K2 : d->K1,
                                 LR_EPI_NONE, nullptr};
      rc = sb_fill_projection(q, pr[i]);
    }
    if (rc != LR_OK) return rc;
  }
  if ((int64_t)M * d->D * 2 >= 0x7fffffff) return LR_E_UNSUPPORTED;
  const int ncu = lr_num_cus();
  if (ncu < 1) return LR_E_LAUNCH;
  plan_resid(d->D, ncu, pr[0].rpw, pr[0].nwg);
  const ResidNorm rn = {pr[1].x, pr[1].w, pr[1].scales, pr[1].ldx, pr[1].K, (const u16*)d->resid_in, (u16*)d->resid_out,
                        (const u16*)(joint ? d->gain2 : d->gain1), (const u16*)d->gain2, (u16*)d->out1, (u16*)d->out2,
                        d->sums1, d->sums2, joint};
  hipStream_t s = (hipStream_t)stream;
  if (pr[0].rpw > 16) return launch_resid_rows<2, 16>(pr[0], M, rn, s);
  return pr[0].rpw > 8 ? launch_resid_rows<1, 16>(pr[0], M, rn, s) : launch_resid_rows<1, 8>(pr[0], M, rn, s);
}

#ifdef LR_BAND_PROFILE
// Profile builds only (not declared in the public header): following launches of this file's kernels record, per
// wave, the six wall-clock stamps of stream_band.h into `device_buffer` (NULL switches it off).  Returns the
// bytes the buffer must hold for the first `workgroups` workgroups of a launch (the others record nothing), or a
// negative error code.
extern "C" long long lr_band_profile(void* device_buffer, int workgroups) {
  if (workgroups < 0) return LR_E_SHAPE;
  unsigned long long* ptr = (unsigned long long*)device_buffer;
  const unsigned wgs = (unsigned)workgroups;
  if (hipMemcpyToSymbol(HIP_SYMBOL(g_band_prof), &ptr, sizeof(ptr)) != hipSuccess ||
      hipMemcpyToSymbol(HIP_SYMBOL(g_band_prof_wgs), &wgs, sizeof(wgs)) != hipSuccess)
    return LR_E_LAUNCH;
  return band_prof_bytes(wgs);
}
#endif

// lr_linear_fp8_multi (gemv_fp8.hip) for 3 to 16 input rows: the same bands with e4m3 weights.
namespace lr_detail {
int stream_fp8_multi(const lr_projection_fp8_t* proj, const lr_row_norm_t* norms, int n_proj, int M, lr_stream_t stream) {
  if (M < 1 || M > 16) return LR_E_UNSUPPORTED;
  Proj pr[2] = {};
  for (int i = 0; i < n_proj; ++i) {
    int rc = sb_fill_projection_fp8(proj[i], pr[i]);
    if (rc == LR_OK && norms) rc = sb_fill_norm(norms + i, pr[i]);
    if (rc != LR_OK) return rc;
  }
  const int ncu = lr_num_cus();
  if (ncu < 1) return LR_E_LAUNCH;
  const int units = pick_units_and_plan(pr, n_proj, M, ncu);
  for (int i = 0; i < n_proj; ++i)
    if (pr[i].fold_sums && pr[i].nwg < M) return LR_E_UNSUPPORTED;   // (a row per workgroup)
  hipStream_t s = (hipStream_t)stream;
  const int rc = M <= 8 ? launch_fp8<true>(pr[0], pr[1], M, units, s) : launch_fp8<false>(pr[0], pr[1], M, units, s);
  return rc != LR_OK ? rc : lr_launch_status();
}
}  // namespace lr_detail
