// The band of the weight-streaming matrix-core kernel as a device function, and what its callers share on the host
// (stream_gemm.hip launches bands only; decode_pair.hip runs decode-attention items beside them).
#pragma once
#include "lr_common.h"

namespace {


constexpr int KC = 128;        // k elements per chunk
constexpr int NWV = 4;         // waves per workgroup
constexpr int SETS = 4;        // weight chunks in flight per wave
constexpr int LROW = KC + 8;   // LDS row length in elements (272 bytes)
constexpr int OOB = (int)0x80000000;  // a buffer offset beyond every resource: the load returns zero, untouched memory
// Input rows from which a band reads the inputs in whole cache lines (through LDS) rather than in fragment layout:
// always with the 32- and 64-row bands; the 16-row band has both forms and the launcher picks by the row count
// (70B rank shard, ms per step, fragment layout / whole lines: 4 rows 4.99 / 5.12, 8 rows 5.14 / 5.19, 16 rows
// 6.26 / 6.00; 8B, 16 rows: 4.00 / 3.78)
constexpr int XLDS_MIN_MT = 32;       // band heights that always read their inputs in whole lines
constexpr int XLDS_M16_FROM = 9;      // input rows from which the 16-row band does too
static_assert(XLDS_M16_FROM <= 9, "the fragment layout of a bf16 band holds 8 input rows (X8)");
constexpr int AUX_WEIGHTS = 2;        // weights: non-temporal (every line is used exactly once)

#ifdef LR_BAND_PROFILE
// Profile builds only: when set (lr_band_profile, stream_gemm.hip), every wave of every band records 100 MHz
// wall-clock stamps at six points -- 0 entry, 1 first requests made, 2 first chunk in LDS, 3 end of the K loop,
// 4 partial sums exchanged (second barrier), 5 end -- at band_prof_at(workgroup, wave, point).
constexpr int BAND_PROF_WAVES = 8;  // of the widest workgroups; narrower ones leave the rest as it was
__host__ __device__ constexpr size_t band_prof_at(unsigned workgroup, int wave, int point) {
  return ((size_t)workgroup * BAND_PROF_WAVES + wave) * 8 + point;
}
constexpr long long band_prof_bytes(unsigned workgroups) { return (long long)(band_prof_at(workgroups, 0, 0) * sizeof(unsigned long long)); }
static __device__ unsigned long long* g_band_prof;
static __device__ unsigned g_band_prof_wgs;  // workgroups the buffer has room for; the others record nothing
#define LR_BAND_STAMP(k)                                                \
  static_assert(NW <= BAND_PROF_WAVES, "a workgroup's stamps are its own"); \
  if (g_band_prof && blockIdx.x < g_band_prof_wgs && lane == 0) g_band_prof[band_prof_at(blockIdx.x, wave, k)] = wall_clock64();
#else
#define LR_BAND_STAMP(k)
#endif

struct Proj {
  const u16* x;
  const u16* w;
  u16* y;
  int64_t ldx, ldy;
  int N, K;      // weight rows, row length
  int rpw;       // rows (row pairs if pair_off) per workgroup
  int pair_off;  // 0, or the distance from an up row to its gate row (= outputs)
  int nwg;       // workgroups of this projection
  int in_turn;   // how a band's four waves share K, see band_in_turn
  const u16* scales;  // weight-only e4m3 weights (the W8 kernels): one bf16 scale per weight row; else nullptr
  // RoPE + KV-cache epilogue of a fused q/k/v projection (rope_table == nullptr: none)
  const u16* rope_table;
  const int32_t* pos;
  u16 *k_cache, *v_cache;
  int32_t* err;
  int Hq, Hkv, hd, Smax, block_size;
  // the input rows still have to be divided by their root mean square (norm_sums == nullptr: they do not): a row's sum of
  // squares is the sum of its norm_count values, [M][norm_count]
  const float* norm_sums;
  int norm_count, norm_dim;
  float norm_eps;
  // the parts of another norm's sums of squares, [M][fold_count], which this launch adds to [M] sums for a later one
  const float* fold_sums;
  float* fold_total;
  int fold_count;
};
// log2 of the distance between a wave's chunks of K in a bf16 band of four waves: 0 a slice each, 2 in turn.  A matter of K alone, measured: see
// stream_band
inline int band_in_turn(int K) { return (K % 2048 == 0 ? K % 16384 == 0 : K > 1024 && (K <= 3072 || (K >= 12288 && K % 1024 != 0))) ? 2 : 0; }
__host__ __device__ constexpr int norm_pitch(int count) { return (count + 255) & ~255; }   // LDS row of parts: whole requests

// What a layer's output projections leave for the next layer's input projections instead of their sums (stream_band, RN):
// a = x w^T, and behind it with a second pair m = x2 w2^T; r1 = resid + a, r2 = r1 + m; out1 = r1 * gain1,
// out2 = r2 * gain2 and the sums of squares of the band's columns of r1 and r2.
struct ResidNorm {
  const u16 *x2, *w2;
  const u16* scales2;
  int64_t ldx2;
  int K2;
  const u16* rin;          // [M, N]
  u16* rout;
  const u16 *gain1, *gain2;
  u16 *out1, *out2;        // [M, N]
  float *sums1, *sums2;    // [M][bands]
  int joint;               // r2 = resid + (m + a), and nothing is kept of r1
};

// the low (HI == false) or high two e4m3 values of a dword as a packed bf16 pair (exact)
template <bool HI>
__device__ __forceinline__ u32 sb_fp8_pair(u32 v) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(u32, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, HI));
}

template <int MT, int UNITS, bool W8 = false, bool XL = (MT >= XLDS_MIN_MT), int NW = NWV>
constexpr size_t stream_band_lds_bytes() {
  constexpr int LRW = (W8 ? 2 * KC : KC) + 8;
  return (size_t)NW * (UNITS * 16 * LRW + (XL ? MT * LRW : 0)) * sizeof(u16);
}
// and behind that, where the input's rows come with sums of squares: the sums, in whole requests, a factor per row, and a row
// of the sums that are added for a later launch
static inline size_t stream_band_norm_bytes(const Proj& p, int M) {
  const int parts = (p.norm_count == 1 ? 256 : M * norm_pitch(p.norm_count)) + (p.fold_sums ? norm_pitch(p.fold_count) : 0);
  return p.norm_sums ? (size_t)(parts + 64) * sizeof(float) : 0;
}
// One wave instruction: 64 x 16 bytes to LDS at `lds` + 16 * lane; what lies beyond `bytes` reads as zero.
__device__ __forceinline__ void band_dma16(const void* base, int bytes, int voff, u32 lds) {
  typedef int i32x4_t __attribute__((ext_vector_type(4)));
  i32x4_t r;
  r.x = (int)(u32)(unsigned long long)base;
  r.y = (int)(u32)((unsigned long long)base >> 32) & 0xffff;
  r.z = bytes;
  r.w = 0x00020000;
  asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"{m0}"(lds), "v"(voff), "s"(r) : "memory");
}

// One band of one projection, by the 256 lanes of a workgroup.  `sg_smem`: stream_band_lds_bytes<MT, UNITS>() bytes of LDS.
// W8: the weights are e4m3 bytes with one bf16 scale per row (p.scales): a load instruction still covers 4 rows x
// 256 bytes, now 256 elements of K, which are expanded to bf16 (exactly: e4m3 is a subset of bf16) on their way
// into the LDS piece; the sum is rounded to bf16, multiplied by the row's scale and rounded again, as
// F.linear(x, w.to(bf16)) * scales does, before the epilogue sees it.
// RESID: nothing is stored to y.  TANH: the sums, and a token's experts' weighted rows if there are any, are added to the fp32 residual,
// whose scaled tanh (lr_residual_tanh) goes out as the next layer's input.  RMS: they are added to the scaled fp32 residual, which is
// brought up to date first where it lacks the norm of the sublayer before (lr_linear_residual_rms).
struct BandResidual {
  float* x;                              // [M, N]
  u16* xc;                               // [M, N]
  const u16 *alpha, *gain, *bias, *eo;   // eo [M * top, N] or nullptr
  const float* ew;                       // [M, top]
  int top;
  // RMS: x <- scale * x + sums, x divided by its rows' root mean square and times offset + before ahead of that if before != nullptr (the
  // rows' sums of squares are the projection's norm_sums); xc = x times offset + gain, squares [M][bands] its rows' sums of squares
  float scale, offset;
  const u16* before;
  float* squares;
};
enum { RESID_NONE, RESID_TANH, RESID_RMS };
// KW: waves that share a band's K, all of them or 1: then every wave has a band of its own (`band_` counts groups of NWV).
// DEEP: the inputs are requested as far ahead as the weights.  Loads come back in the order of their requests, so a wait
// for inputs that were asked for one chunk ago is a wait for nearly all the weights asked for before them; with both in
// one order a wait leaves the younger chunks in flight.  (16-row bands; at 32 rows the registers for it cost more.)
// X8: at most 8 input rows.  Fragment columns 8 to 15 would be empty, so their lanes carry the next 32 elements of K of
// rows 0 to 7, and every second fragment is the previous load rotated by 8 lanes: half as many input loads (which were a
// third of a bf16 band's requests and half of an e4m3 band's) and half their registers.
// UROWS: weight rows of a unit that are loaded, 8 where no band has more: a load of absent rows takes its time too.
// The three together, us, 8 rows: 1280 x 8192 9.43 -> 7.41, 4096 x 4096 9.37 -> 8.64, 10240 x 4096 19.25 -> 18.50, up/gate
// 7168 x 8192 22.4 -> 21.9, 8192 x (1024 | 3584) 16.9 -> 16.3; 16 rows (DEEP alone) 4096 x 14336 25.1 -> 23.8; e4m3, 5 rows:
// 1280 x 8192 7.80 -> 6.32, 8192 x (1024 | 3584) 11.9 -> 10.8, up/gate 14.2 -> 13.6.  The sums keep their order.
// GATHER: input row m is row rows[m] / xdiv of x, output row m is row rows[m] of y (`rows`: M of them, in LDS).
template <int MT, int UNITS, bool W8 = false, bool XL = (MT >= XLDS_MIN_MT), bool GATHER = false, int RESID = RESID_NONE, int KW = NWV,
          int UROWS = 16, bool DEEP = true, bool X8 = false, int NW = NWV, bool RN = false>
__device__ __forceinline__ void stream_band(const Proj& p, const int M, const int band_, u16* sg_smem,
                                            const int32_t* rows = nullptr, const int xdiv = 1, const BandResidual rs = {},
                                            const ResidNorm& rn = {}) {
  static_assert(!W8 || MT == 16, "the e4m3 path is built for up to 16 input rows");
  const bool has_norm = MT == 16 && KW == NW && !GATHER && RESID != RESID_TANH && !RN && p.norm_sums != nullptr;
  constexpr int KCW = W8 ? 256 : 128;  // k elements per chunk
  constexpr int LRW = KCW + 8;         // LDS row length in elements
  constexpr int WB = W8 ? 1 : 2;       // bytes per weight
  // weight chunks in flight per wave: the e4m3 variant has twice the A fragments and input registers per chunk
  // and gives up two of its four sets for a second workgroup per CU (with half the input registers, X8, four sets would
  // fit: up/gate of 5 rows 13.3 -> 15.0 us), except where a band is 8 rows (1280 x 8192: 6.9 us with two, 6.3 with four;
  // a bf16 band of 8 rows with eight sets: 8.1, with four 7.4)
  constexpr int NS = W8 && UROWS == 16 ? 2 : SETS;
  constexpr int XS = DEEP ? NS : 2;
  constexpr int MTILES = MT / 16, KS = KCW / 32, NLD = UNITS * UROWS / 4;
  static_assert(!X8 || (MT == 16 && !XL), "one tile of inputs in fragment layout");
  static_assert(UROWS == 16 || (UROWS == 8 && UNITS == 1), "a unit is loaded whole or by half");
  constexpr int NV = UNITS * MTILES * 4;  // accumulator registers per lane
  // XL: the inputs too are loaded in whole lines (4 rows x 256 bytes per instruction) and take the trip through
  // LDS into B-fragment layout: L2 serves whole-line reads 1.5 times as fast as the 16 rows x 64 bytes a
  // fragment-layout load touches, and at 64 rows the input bytes are twice the weight bytes.
  constexpr bool XLDS = XL;
  static_assert(!(XL && W8), "the e4m3 band reads its inputs in fragment layout");
  constexpr int WPIECE = UNITS * 16 * LRW, XPIECE = XLDS ? MT * LRW : 0;  // elements per wave
  // sg_smem: [NWV][WPIECE + XPIECE]
  static_assert(sizeof(float) * (RN ? 2 : 1) * NV * 64 <= sizeof(u16) * WPIECE, "the partial sums reuse the wave's weight piece");

  const u16* const xg = p.x;
  const u16* const wg_ = p.w;
  u16* const yg = p.y;
  const int64_t ldx = p.ldx, ldy = p.ldy;
  const int N = p.N, K = p.K, rpw = p.rpw;
  const int pair_off = p.pair_off;
  const u16* const rope_table = p.rope_table;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, l4 = lane >> 4;
  const int la = lane & (UROWS - 1);  // the band row of a lane's A fragment (beyond UROWS the first rows again: unused sums)
  static_assert(KW == NW || (KW == 1 && !W8 && !XL), "");
  static_assert(!RN || (KW == NW && MT == 16 && !GATHER && !RESID), "");
  const int band = KW == 1 ? band_ * NW + wave : band_;
  const int kwave = KW == 1 ? 0 : wave;
  LR_BAND_STAMP(0)
  const int n_out = pair_off ? pair_off : N;         // output columns
  const int n0 = band * rpw;                          // first row (pair) of the band
  const int nrows = n_out - n0 < rpw ? n_out - n0 : rpw;

  // ---- lane constants of the weight loads: instruction i covers band rows 4 i .. 4 i + 3 (in pair mode
  //      unit 0 holds the up rows, unit 1 the gate rows of the same pairs)
  const __amdgpu_buffer_rsrc_t wres =
      __builtin_amdgcn_make_buffer_rsrc(
          const_cast<unsigned char*>(reinterpret_cast<const unsigned char*>(wg_) + (int64_t)n0 * K * WB), 0, 0x7fffffff,
          0x00020000);
  const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(xg), 0, 0x7fffffff, 0x00020000);
  int woff[NLD];
#pragma unroll
  for (int i = 0; i < NLD; ++i) {
    const int r = 4 * i + l4;  // row inside the LDS piece
    int rr = r, extra = 0;
    if (pair_off && r >= 16) { rr = r - 16; extra = pair_off; }
    woff[i] = rr < nrows ? (int)((int64_t)(extra + rr) * K * WB + l16 * 16) : OOB;
  }
  // fragment layout: tile mt, k-step ks <- input row 16 mt + lane % 16, elements 32 ks + 8 (lane / 16) ..;
  // whole-line layout: instruction i <- input rows 4 i + lane / 16, elements 8 (lane % 16) ..
  int xoff[XLDS ? MT / 4 : MTILES];
  if (XLDS) {
#pragma unroll
    for (int i = 0; i < MT / 4; ++i) {
      const int m = 4 * i + l4;
      const int xm = GATHER ? (m < M ? rows[m] / xdiv : 0) : m;
      xoff[i] = m < M ? (int)((xm * ldx + l16 * 8) * 2) : OOB;
    }
  } else {
#pragma unroll
    for (int mt = 0; mt < MTILES; ++mt) {
      const int m = mt * 16 + (X8 ? l16 & 7 : l16);
      const int xm = GATHER ? (m < M ? rows[m] / xdiv : 0) : m;
      xoff[mt] = m < M ? (int)((xm * ldx + (X8 ? (l16 >> 3) * 32 : 0) + l4 * 8) * 2) : OOB;
    }
  }
  // k-step ks of input tile mt as a B fragment
  auto xfrag = [&](const u32x4_t (&r)[MTILES][X8 ? KS / 2 : KS], int mt, int ks) {
    if constexpr (X8) {
      u32x4_t v = r[0][ks / 2];
      if (ks & 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __builtin_amdgcn_update_dpp(v[e], v[e], 0x128, 0xf, 0xf, false);  // row_ror:8
      return __builtin_bit_cast(bf16x8_t, v);
    } else {
      return __builtin_bit_cast(bf16x8_t, r[mt][ks]);
    }
  };
  // OOB where v >= n, else 0: no branch, and a scalar stays one
  auto beyond = [](int v, int n) { return ~(v - n) & OOB; };
  // (RN) the first pair's chunks of K come first, then the second's; a lane's offsets within each matrix, its rows' in scalars
  const int nck1 = (K + KCW - 1) / KCW;
  int wv1 = 0, wv2 = 0, xoff2[XLDS ? MT / 4 : MTILES];
  if constexpr (RN) {
    wv1 = l4 * K * WB + l16 * 16;
    wv2 = l4 * rn.K2 * WB + l16 * 16;
#pragma unroll
    for (int i = 0; i < (XLDS ? MT / 4 : MTILES); ++i) {
      const int m = XLDS ? 4 * i + l4 : (X8 ? l16 & 7 : l16);
      xoff2[i] = m < M ? (int)((m * rn.ldx2 + (XLDS ? l16 * 8 : (X8 ? (l16 >> 3) * 32 : 0) + l4 * 8)) * 2) : OOB;
    }
  }
  u16* const my = sg_smem + wave * (WPIECE + XPIECE);
  u16* const myx = my + WPIECE;

  u32x4_t wr[NS][NLD];
  u32x4_t xr[XS][MTILES][X8 ? KS / 2 : KS];
  f32x4_t acc[UNITS][MTILES];
#pragma unroll
  for (int u = 0; u < UNITS; ++u)
#pragma unroll
    for (int mt = 0; mt < MTILES; ++mt) acc[u][mt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // Which chunk of K is the wave's ci-th: the waves' chunks in turn, g = ci KW + wave, or a slice of K per wave, one chunk behind the
  // other.  All workgroups walk K from the same end: over rows that lie a multiple of 4 KiB apart the four waves' 1 KiB in turn are the same
  // quarter of the DRAM's interleaving all over the grid, and places a slice apart are not.  Slices of whole 4 KiB begin at four
  // different quarters and wrap around (8192 columns: 20.7 us for 7168 rows, 24.8 without).  us, 8 input rows, in turn / in slices, one library:
  // 128256 x 2048 92.2 / 84.8, 16384 x 2048 15.3 / 14.1, 128256 x 4096 199 / 156, 6144 x 4096 11.7 / 11.0, 8192 x 8192 31.1 / 23.8, 16032 x 8192 55.9 /
  // 42.2, 4096 x 14336 21.4 / 20.3, 8192 x 20480 55.2 / 51.4.
  // Other widths gain less by slices or lose by them, and are in turn where they measured slower so (2048 to 16384 rows, 8 to 32 input rows, time in
  // slices over that in turn): 1024 0.92 to 1.01; 1536 to 3072 1.02 to 1.11; 3584 to 9216 0.95 to 1.04, as long on average; 11008 0.93 to 0.97;
  // 12800 1.01 to 1.06; 15360 0.97 to 1.01; 22016 1.08 to 1.20 (8192 rows, 8 input rows, 80.9 / 68.0 us); but 17920 0.95 to 1.00.  In turn, too:
  // multiples of 32 KiB (13312 x 16384 76.7 / 69.6, 2304 x 16384 16.8 / 15.6, 2048 x 32768 30.5 / 29.7; 8192 x 32768 88.5 / 96.2), the two
  // matrices of RN, where a wave that wraps around would mix them (8192 x (1024 | 3584) 19.6 / 18.4 without), and e4m3, where a row's chunk is half
  // as long (5 input rows: 1280 x 8192 6.40 / 6.33, 28672 x 4096 22.5 / 22.9, 6144 x 4096 7.82 / 7.86, 16 rows 10.11 / 9.73; but 16032 x 8192 22.9 /
  // 28.5, 128256 x 4096 82.2 / 92.3).
  // What lies beyond K or the wave's last chunk reads as zero (no branch around a load: the number of loads in flight is fixed, so
  // the waits between chunks are exact).  The order of a sum is a matter of K alone, not of how the rows are cut into bands.
  const int nck = nck1 + (RN ? (rn.K2 + KCW - 1) / KCW : 0);
  constexpr bool SLICES = !RN && !W8;
  // (selects and shifts: a branch here is 0.1 us of a launch, 4 to 8 % of the smallest)
  static_assert(KW == 1 || KW == 4 || (KW == 8 && !SLICES), "");
  const int turn = !SLICES ? (KW == 8 ? 3 : KW == 4 ? 2 : 0) : KW == 1 ? 0 : p.in_turn;   // log2 of the distance between a wave's chunks
  const int kper = (nck + KW - 1) / KW, kfirst = kwave * (turn ? 1 : kper), kend = min(nck, turn ? nck : kfirst + kper);
  const int nch = max(kend - kfirst + (1 << turn) - 1, 0) >> turn;  // chunks of this wave
  constexpr int CHUNKS_4K = 4096 / (KCW * WB), QUARTER = CHUNKS_4K / 4;
  const int kturn = SLICES ? (kwave * QUARTER % CHUNKS_4K) & -(int)((turn == 0) & (kper % CHUNKS_4K == 0) & (nch == kper)) : 0;
  auto chunk_at = [&](int ci) {
    if (!SLICES) return ci * KW + kfirst;
    const int c = ci + kturn, g = kfirst + ((c - (c < nch ? 0 : nch)) << turn);
    return ci < nch ? g : nck;
  };
  auto issue_w = [&](int ci, u32x4_t (&dst)[NLD]) {
    if constexpr (RN) {
      const int g = chunk_at(ci);
      const bool second = g >= nck1;
      const int k0 = (second ? g - nck1 : g) * KCW, Kx = second ? rn.K2 : K;
      const __amdgpu_buffer_rsrc_t res = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<unsigned char*>(reinterpret_cast<const unsigned char*>(second ? rn.w2 : wg_) + (int64_t)n0 * Kx * WB), 0, 0x7fffffff,
          0x00020000);
      const int at = (second ? wv2 : wv1) | beyond(k0 + l16 * (16 / WB), Kx);
#pragma unroll
      for (int i = 0; i < NLD; ++i)
        dst[i] = __builtin_amdgcn_raw_buffer_load_b128(res, at | beyond(4 * i + l4, nrows), (k0 + 4 * i * Kx) * WB, AUX_WEIGHTS);
      return;
    }
    const int k0 = chunk_at(ci) * KCW;
    const bool kok = k0 + l16 * (16 / WB) < K;
#pragma unroll
    for (int i = 0; i < NLD; ++i)
      dst[i] = __builtin_amdgcn_raw_buffer_load_b128(wres, (kok && woff[i] != OOB) ? woff[i] : OOB, k0 * WB, AUX_WEIGHTS);
  };
  auto issue_x = [&](int ci, u32x4_t (&dst)[MTILES][X8 ? KS / 2 : KS]) {
    if constexpr (RN) {
      const int g = chunk_at(ci);
      const bool second = g >= nck1;
      const int k0 = (second ? g - nck1 : g) * KCW, Kx = second ? rn.K2 : K;
      const __amdgpu_buffer_rsrc_t res =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(second ? rn.x2 : xg), 0, 0x7fffffff, 0x00020000);
      constexpr int NX = XLDS ? MT / 4 : (X8 ? KS / 2 : KS);
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        const int at = XLDS ? l16 * 8 : (X8 ? (2 * j + (l16 >> 3)) * 32 : j * 32) + l4 * 8;   // the lane's first k in the chunk
        const int off = second ? xoff2[XLDS ? j : 0] : xoff[XLDS ? j : 0];
        dst[XLDS ? j / KS : 0][XLDS ? j % KS : j] = __builtin_amdgcn_raw_buffer_load_b128(
            res, off | beyond(k0 + at, Kx), (k0 + (XLDS ? 0 : (X8 ? 2 : 1) * j * 32)) * 2, 0);
      }
      return;
    }
    const int k0 = chunk_at(ci) * KCW;
    if constexpr (XLDS) {
      const bool kok = k0 + l16 * 8 < K;
#pragma unroll
      for (int i = 0; i < MT / 4; ++i)
        dst[i / KS][i % KS] =
            __builtin_amdgcn_raw_buffer_load_b128(xres, (kok && xoff[i] != OOB) ? xoff[i] : OOB, k0 * 2, 0);
    } else if constexpr (X8) {
#pragma unroll
      for (int j = 0; j < KS / 2; ++j)
        dst[0][j] = __builtin_amdgcn_raw_buffer_load_b128(
            xres, (k0 + (2 * j + (l16 >> 3)) * 32 + l4 * 8 < K && xoff[0] != OOB) ? xoff[0] : OOB, (k0 + 2 * j * 32) * 2, 0);
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const bool kok = k0 + ks * 32 + l4 * 8 < K;
#pragma unroll
        for (int mt = 0; mt < MTILES; ++mt)
          dst[mt][ks] = __builtin_amdgcn_raw_buffer_load_b128(xres, (kok && xoff[mt] != OOB) ? xoff[mt] : OOB,
                                                             (k0 + ks * 32) * 2, 0);
      }
    }
  };

  // (the fences keep the requests in this order: the wait for chunk 0 counts the requests made after it, and the
  // scheduler, left alone, asks for chunk 0 last -- the loop then waited for all but the last 8 requests at the top
  // of every round of NS chunks)
  // The parts of the sums of squares of rows wave, wave + NW, ... go to LDS ahead of everything else, and while the first
  // weights are on their way the wave adds them.  Whole sums (norm_count 1) need one request.
  const int npitch = norm_pitch(p.norm_count);
  float* const nsum = reinterpret_cast<float*>(sg_smem + NW * (WPIECE + XPIECE));
  float* const nscale = nsum + (p.norm_count == 1 ? 256 : M * npitch);
  const bool folds = has_norm && p.fold_sums != nullptr && band < M && wave == NW - 1;   // the other norm's row `band`
  float* const nfold = nscale + 64;
  if (has_norm) {
    const u32 at = __builtin_amdgcn_readfirstlane((u32)(uintptr_t)(__attribute__((address_space(3))) float*)nsum);
    if (p.norm_count == 1) {
      if (wave == 0) band_dma16(p.norm_sums, M * 4, lane * 16, at);
    } else {
      for (int m = wave; m < M; m += NW)
        for (int o = 0; o < npitch; o += 256)
          band_dma16(p.norm_sums + m * p.norm_count, p.norm_count * 4, (o + lane * 4) * 4, at + (m * npitch + o) * 4);
    }
    if (folds) {
      const u32 fat = __builtin_amdgcn_readfirstlane((u32)(uintptr_t)(__attribute__((address_space(3))) float*)nfold);
      for (int o = 0; o < norm_pitch(p.fold_count); o += 256)
        band_dma16(p.fold_sums + band * p.fold_count, p.fold_count * 4, (o + lane * 4) * 4, fat + o * 4);
    }
  }
  // the residual and the gains of the lane's output
  u16 r_in = 0, ga1 = 0, ga2 = 0, sc1 = 0, sc2 = 0;
  constexpr int ROWS_RN = 16 * UNITS;
  static_assert(!RN || ROWS_RN * MT <= NW * 64, "an output per lane");
  const int rn_r = tid % ROWS_RN, rn_m = tid / ROWS_RN;
  const bool rn_ok = RN && rn_r < nrows && rn_m < M;
  if constexpr (RN) {
    // (no branch around a load: see above)
    const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(rn.rin), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t r1 = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(rn.gain1), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t r2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(rn.gain2), 0, 0x7fffffff, 0x00020000);
    r_in = __builtin_amdgcn_raw_buffer_load_b16(rr, rn_ok ? (rn_m * N + n0 + rn_r) * 2 : OOB, 0, 0);
    ga1 = __builtin_amdgcn_raw_buffer_load_b16(r1, rn_ok ? (n0 + rn_r) * 2 : OOB, 0, 0);
    ga2 = __builtin_amdgcn_raw_buffer_load_b16(r2, rn_ok ? (n0 + rn_r) * 2 : OOB, 0, 0);
    if constexpr (W8) {
      const __amdgpu_buffer_rsrc_t s1 = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(p.scales), 0, 0x7fffffff, 0x00020000);
      const __amdgpu_buffer_rsrc_t s2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(rn.scales2), 0, 0x7fffffff, 0x00020000);
      sc1 = __builtin_amdgcn_raw_buffer_load_b16(s1, rn_ok ? (n0 + rn_r) * 2 : OOB, 0, 0);
      sc2 = __builtin_amdgcn_raw_buffer_load_b16(s2, rn_ok ? (n0 + rn_r) * 2 : OOB, 0, 0);
    }
    asm volatile("" ::: "memory");
  }
  // (RMS) the lane's outputs' residuals and gains
  constexpr int RMS_ROWS = 16 * UNITS;
  static_assert(RESID != RESID_RMS || (MT == 16 && KW == NWV && NW == NWV), "UNITS outputs per lane");
  u32 rms_x[UNITS];
  u16 rms_before[UNITS], rms_gain[UNITS];
  if constexpr (RESID == RESID_RMS) {
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(rs.x, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(rs.before), 0, rs.before ? N * 2 : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(rs.gain), 0, N * 2, 0x00020000);
#pragma unroll
    for (int i = 0; i < UNITS; ++i) {
      const int o = tid + i * NW * 64, r = o % RMS_ROWS, m = o / RMS_ROWS;
      const bool ok = r < nrows && m < M;
      rms_x[i] = __builtin_amdgcn_raw_buffer_load_b32(rx, ok ? (m * N + n0 + r) * 4 : OOB, 0, 0);
      rms_before[i] = __builtin_amdgcn_raw_buffer_load_b16(rb, ok ? (n0 + r) * 2 : OOB, 0, 0);
      rms_gain[i] = __builtin_amdgcn_raw_buffer_load_b16(rg, ok ? (n0 + r) * 2 : OOB, 0, 0);
    }
    asm volatile("" ::: "memory");
  }
  f32x4_t acc1[UNITS][MTILES];   // (RN) the first pair's sums, once the wave has its last chunk of it
  bool in_first = true;
  issue_x(0, xr[0]);
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    if (DEEP && s) issue_x(s, xr[s]);
    asm volatile("" ::: "memory");
    issue_w(s, wr[s]);
  }
  asm volatile("" ::: "memory");
  if (has_norm) {
    constexpr int YOUNGER = NS * NLD + (DEEP ? NS : 1) * (XLDS ? MT / 4 : MTILES * (X8 ? KS / 2 : KS));   // requests since
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER < 63 ? YOUNGER : 63) : "memory");
    auto part = [&](const float* row, int pitch) {   // (zeros beyond the count)
      float v = 0.0f;
      for (int o = 0; o < pitch; o += 256) {
        const float4 q = *reinterpret_cast<const float4*>(row + o + lane * 4);
        v += (q.x + q.y) + (q.z + q.w);
      }
      return v;
    };
    if (p.norm_count == 1) {
      if (wave == 0 && lane < M) nscale[lane] = rsqrtf(nsum[lane] / (float)p.norm_dim + p.norm_eps);
    } else {
      constexpr int R = MT / NW;   // rows of a wave, their sums side by side
      float v[R];
#pragma unroll
      for (int i = 0; i < R; ++i) v[i] = part(nsum + (wave + i * NW < M ? wave + i * NW : 0) * npitch, npitch);
#pragma unroll
      for (int i = 0; i < R; ++i) v[i] = wave_sum(v[i]);
#pragma unroll
      for (int i = 0; i < R; ++i)
        if (lane == 0 && wave + i * NW < M) nscale[wave + i * NW] = rsqrtf(v[i] / (float)p.norm_dim + p.norm_eps);
    }
    if (folds) {
      const float v = wave_sum(part(nfold, norm_pitch(p.fold_count)));
      if (lane == 0) p.fold_total[band] = v;
    }
    asm volatile("" ::: "memory");
  }
  LR_BAND_STAMP(1)
  for (int c0 = 0; c0 < nch; c0 += NS) {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int ci = c0 + s;
      if constexpr (RN) {
        if (in_first && chunk_at(ci) >= nck1) {
          in_first = false;
#pragma unroll
          for (int u = 0; u < UNITS; ++u)
#pragma unroll
            for (int mt = 0; mt < MTILES; ++mt) {
              acc1[u][mt] = acc[u][mt];
              acc[u][mt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            }
        }
      }
      if (!DEEP) issue_x(ci + 1, xr[(s + 1) % XS]);
      // ---- this chunk's weights: registers -> LDS (row-major) -> A fragments
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        if constexpr (W8) {
          u32x4_t lo, hi;
          lo[0] = sb_fp8_pair<false>(wr[s][i][0]); lo[1] = sb_fp8_pair<true>(wr[s][i][0]);
          lo[2] = sb_fp8_pair<false>(wr[s][i][1]); lo[3] = sb_fp8_pair<true>(wr[s][i][1]);
          hi[0] = sb_fp8_pair<false>(wr[s][i][2]); hi[1] = sb_fp8_pair<true>(wr[s][i][2]);
          hi[2] = sb_fp8_pair<false>(wr[s][i][3]); hi[3] = sb_fp8_pair<true>(wr[s][i][3]);
          *reinterpret_cast<u32x4_t*>(my + (4 * i + l4) * LRW + l16 * 16) = lo;
          *reinterpret_cast<u32x4_t*>(my + (4 * i + l4) * LRW + l16 * 16 + 8) = hi;
        } else {
          *reinterpret_cast<u32x4_t*>(my + (4 * i + l4) * LRW + l16 * 8) = wr[s][i];
        }
      }
      asm volatile("" ::: "memory");
#ifdef LR_BAND_PROFILE
      if (ci == 0) { LR_BAND_STAMP(2) }
#endif
      if constexpr (W8) {
        // 256 elements of K per chunk: the A fragments are taken in two halves to keep them at 32 registers
        issue_w(ci + NS, wr[s]);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          bf16x8_t ah[UNITS][KS / 2];
#pragma unroll
          for (int u = 0; u < UNITS; ++u)
#pragma unroll
            for (int k2 = 0; k2 < KS / 2; ++k2)
              ah[u][k2] =
                  *reinterpret_cast<const bf16x8_t*>(my + (16 * u + la) * LRW + (h * (KS / 2) + k2) * 32 + l4 * 8);
#pragma unroll
          for (int k2 = 0; k2 < KS / 2; ++k2)
#pragma unroll
            for (int mt = 0; mt < MTILES; ++mt) {
              const bf16x8_t bx = xfrag(xr[s % XS], mt, h * (KS / 2) + k2);
#pragma unroll
              for (int u = 0; u < UNITS; ++u)
                acc[u][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[u][k2], bx, acc[u][mt], 0, 0, 0);
            }
        }
        asm volatile("" ::: "memory");
        if (DEEP) issue_x(ci + NS, xr[s % XS]);
        continue;
      }
      bf16x8_t af[UNITS][KS];
#pragma unroll
      for (int u = 0; u < UNITS; ++u)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          af[u][ks] = *reinterpret_cast<const bf16x8_t*>(my + (16 * u + la) * LRW + ks * 32 + l4 * 8);
      asm volatile("" ::: "memory");
      issue_w(ci + NS, wr[s]);
      if (XLDS) {
#pragma unroll
        for (int i = 0; i < MT / 4; ++i)
          *reinterpret_cast<u32x4_t*>(myx + (4 * i + l4) * LRW + l16 * 8) = xr[s % XS][i / KS][i % KS];
        asm volatile("" ::: "memory");
        if (DEEP) issue_x(ci + NS, xr[s % XS]);
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int mt = 0; mt < MTILES; ++mt) {
          bf16x8_t bx;
          if (XLDS) bx = *reinterpret_cast<const bf16x8_t*>(myx + (16 * mt + l16) * LRW + ks * 32 + l4 * 8);
          else bx = xfrag(xr[s % XS], mt, ks);
#pragma unroll
          for (int u = 0; u < UNITS; ++u)
            acc[u][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[u][ks], bx, acc[u][mt], 0, 0, 0);
        }
      if (XLDS) asm volatile("" ::: "memory");
      else if (DEEP) issue_x(ci + NS, xr[s % XS]);
    }
  }

  LR_BAND_STAMP(3)
  if constexpr (RN) {
    if (in_first) {
#pragma unroll
      for (int u = 0; u < UNITS; ++u)
#pragma unroll
        for (int mt = 0; mt < MTILES; ++mt) {
          acc1[u][mt] = acc[u][mt];
          acc[u][mt] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
  }
  // ---- the waves' partial sums meet in LDS (accumulator element e of tile (u, mt): band row
  //      16 u + 4 (lane / 16) + e, input row 16 mt + lane % 16) and are added in wave order
  __syncthreads();
  float* const red = reinterpret_cast<float*>(sg_smem);
  constexpr int WSTRIDE = (WPIECE + XPIECE) / 2;  // floats per wave piece
#pragma unroll
  for (int u = 0; u < UNITS; ++u)
#pragma unroll
    for (int mt = 0; mt < MTILES; ++mt)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        red[wave * WSTRIDE + ((u * MTILES + mt) * 4 + e) * 64 + lane] = acc[u][mt][e];
        if constexpr (RN) red[wave * WSTRIDE + NV * 64 + ((u * MTILES + mt) * 4 + e) * 64 + lane] = acc1[u][mt][e];
      }
  __syncthreads();
  // a sum, or that of the input's normed rows
  auto normed = [&](float v, int m) { return has_norm ? v * nscale[m] : v; };
  LR_BAND_STAMP(4)
  if constexpr (RN) {
    float a = 0.0f, m2 = 0.0f;
    const int ln = ((rn_r & 15) >> 2) * 16 + (rn_m & 15), e = rn_r & 3, u = rn_r >> 4;
#pragma unroll
    for (int wv = 0; wv < NW; ++wv) {
      a += red[wv * WSTRIDE + NV * 64 + (u * 4 + e) * 64 + ln];
      m2 += red[wv * WSTRIDE + (u * 4 + e) * 64 + ln];
    }
    a = round_bf(a);
    m2 = round_bf(m2);
    const int n = n0 + rn_r;
    if constexpr (W8) {
      a = round_bf(a * bf_to_f(sc1));
      m2 = round_bf(m2 * bf_to_f(sc2));
    }
    const float r1 = round_bf(bf_to_f(r_in) + a), r2 = rn.joint ? round_bf(bf_to_f(r_in) + round_bf(m2 + a)) : round_bf(r1 + m2);
    float s1 = rn_ok ? r1 * r1 : 0.0f, s2 = rn_ok ? r2 * r2 : 0.0f;
    s1 = row_sum(s1);
    s2 = row_sum(s2);
    if (ROWS_RN == 32) {
      s1 += __shfl_xor(s1, 16, LR_WAVE);
      s2 += __shfl_xor(s2, 16, LR_WAVE);
    }
    if (rn_ok) {
      const int64_t at = (int64_t)rn_m * N + n;
      rn.rout[at] = f_to_bf(r2);
      if (!rn.joint) rn.out1[at] = f_to_bf(r1 * bf_to_f(ga1));
      rn.out2[at] = f_to_bf(r2 * bf_to_f(ga2));
      if (rn_r == 0) {
        if (!rn.joint) rn.sums1[rn_m * p.nwg + band] = s1;
        rn.sums2[rn_m * p.nwg + band] = s2;
      }
    }
    LR_BAND_STAMP(5)
    return;
  }
  if constexpr (RESID == RESID_RMS) {
#pragma unroll
    for (int i = 0; i < UNITS; ++i) {
      const int o = tid + i * NW * 64, r = o % RMS_ROWS, m = o / RMS_ROWS;
      const int ln = ((r & 15) >> 2) * 16 + m, e = r & 3, u = r >> 4;
      const bool ok = r < nrows && m < M;
      float s0 = 0.0f, v = __builtin_bit_cast(float, rms_x[i]);
#pragma unroll
      for (int wv = 0; wv < NW; ++wv) s0 += red[wv * WSTRIDE + (u * 4 + e) * 64 + ln];
      if (rs.before) v = normed(v, m) * (rs.offset + bf_to_f(rms_before[i]));
      v = ok ? fmaf(rs.scale, v, s0) : 0.0f;
      float sq = row_sum(v * v);
      if (UNITS == 2) sq += __shfl_xor(sq, 16, LR_WAVE);
      if (ok) {
        rs.x[(int64_t)m * N + n0 + r] = v;
        rs.xc[(int64_t)m * N + n0 + r] = f_to_bf(v * (rs.offset + bf_to_f(rms_gain[i])));
        if (r == 0) rs.squares[m * p.nwg + band] = sq;
      }
    }
    LR_BAND_STAMP(5)
    return;
  }
  const int rows_out = pair_off ? 16 : 16 * UNITS;
  if (rope_table != nullptr) {
    // The fused q/k/v projection of a decode step (one token per sequence: input row m is sequence m):
    // what lr_rope_kv_write would do to the stored row, done here on the (even, odd) output pairs.  A
    // position outside the cache or the table: the plain projection is stored, the error word is set.
    const Proj& pp = p;
    const int hd = pp.hd, nq = pp.Hq * hd, nkv = pp.Hkv * hd;
    const int ps = pp.pos[0];
    const bool in_range = ps >= 0 && ps < pp.Smax && ps < pp.block_size;
    if (!in_range && pp.err && band == 0 && tid == 0) *pp.err = LR_DEV_POS_RANGE;
    for (int o = tid; o < (rows_out / 2) * MT; o += NW * 64) {
      const int r = 2 * (o % (rows_out / 2)), m = o / (rows_out / 2);
      if (r >= nrows || m >= M) continue;
      const int mt = m >> 4, ln = ((r & 15) >> 2) * 16 + (m & 15), e = r & 3, u = r >> 4;
      float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
      for (int wv = 0; wv < NW; ++wv) {
        s0 += red[wv * WSTRIDE + ((u * MTILES + mt) * 4 + e) * 64 + ln];
        s1 += red[wv * WSTRIDE + ((u * MTILES + mt) * 4 + e + 1) * 64 + ln];
      }
      const int n = n0 + r;
      float x0 = round_bf(normed(s0, m)), x1 = round_bf(normed(s1, m));
      if constexpr (W8) {
        x0 = round_bf(x0 * bf_to_f(pp.scales[n]));
        x1 = round_bf(x1 * bf_to_f(pp.scales[n + 1]));
      }
      u32 plain = pack_bf2(x0, x1), out = plain;
      if (in_range) {
        const int sect = n < nq ? 0 : (n < nq + nkv ? 1 : 2);
        const int cc = n - (sect == 0 ? 0 : (sect == 1 ? nq : nq + nkv));
        const int h = cc / hd, d = cc - h * hd;
        if (sect < 2) {
#pragma clang fp contract(off)
          const u32 cs = *reinterpret_cast<const u32*>(rope_table + (int64_t)ps * hd + d);
          const float c = bf_lo(cs), sn = bf_hi(cs);
          const float a = x0 * c, b = x1 * sn, dd = x1 * c, ee = x0 * sn;
          out = pack_bf2(a - b, dd + ee);
        }
        if (sect == 0) plain = out;  // q is rotated in place; k and v stay as projected, the cache gets them
        if (sect == 1) *reinterpret_cast<u32*>(pp.k_cache + (((int64_t)m * pp.Hkv + h) * pp.Smax + ps) * hd + d) = out;
        if (sect == 2) *reinterpret_cast<u32*>(pp.v_cache + (((int64_t)m * pp.Hkv + h) * pp.Smax + ps) * hd + d) = plain;
      }
      *reinterpret_cast<u32*>(yg + (int64_t)m * ldy + n) = plain;
    }
    LR_BAND_STAMP(5)
    return;
  }
  for (int o = KW == 1 ? lane : tid; o < rows_out * MT; o += KW * 64) {
    const int r = o % rows_out, m = o / rows_out;
    if (r >= nrows || m >= M) continue;
    const int mt = m >> 4, ln = ((r & 15) >> 2) * 16 + (m & 15), e = r & 3, u = r >> 4;
    const int ym = GATHER ? rows[m] : m;
    float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
    for (int wv = 0; wv < KW; ++wv) s0 += red[(KW == 1 ? wave : wv) * WSTRIDE + ((u * MTILES + mt) * 4 + e) * 64 + ln];
    if constexpr (RESID == RESID_TANH) {
      const int n = n0 + r;
      const int64_t at = (int64_t)m * N + n;
      float v = rs.x[at] + s0;
      if (rs.eo) {
        float t = 0.0f;
#pragma unroll 4
        for (int k = 0; k < rs.top; ++k) t = fmaf(rs.ew[m * rs.top + k], bf_to_f(rs.eo[((int64_t)m * rs.top + k) * N + n]), t);
        v += t;
      }
      rs.x[at] = v;
      rs.xc[at] = f_to_bf(fmaf(tanhf(bf_to_f(rs.alpha[0]) * v), bf_to_f(rs.gain[n]), bf_to_f(rs.bias[n])));
    } else if (pair_off) {
      if (UNITS == 2) {
#pragma unroll
        for (int wv = 0; wv < KW; ++wv) s1 += red[(KW == 1 ? wave : wv) * WSTRIDE + ((MTILES + mt) * 4 + e) * 64 + ln];
      }
      float u_ = round_bf(normed(s0, m)), g_ = round_bf(normed(s1, m));
      if constexpr (W8) {
        u_ = round_bf(u_ * bf_to_f(p.scales[n0 + r]));
        g_ = round_bf(g_ * bf_to_f(p.scales[pair_off + n0 + r]));
      }
      yg[(int64_t)ym * ldy + n0 + r] = f_to_bf(swiglu_bf(u_, g_));
    } else if constexpr (W8) {
      yg[(int64_t)ym * ldy + n0 + r] = f_to_bf(round_bf(normed(s0, m)) * bf_to_f(p.scales[n0 + r]));
    } else {
      yg[(int64_t)ym * ldy + n0 + r] = f_to_bf(normed(s0, m));
    }
  }
  LR_BAND_STAMP(5)
}

// Rows per workgroup: the rows are spread evenly over whole rounds of the CUs, at most `cap` per
// workgroup; with few weight rows and many input rows a band is not made thinner than `floor_rows`
// (every band re-reads all input rows from L2).
static void plan(Proj& p, int M, int cap, int ncu) {
  // (the RoPE epilogue works on output pairs: bands of an even number of rows)
  const int items = p.pair_off ? p.pair_off : p.N;
  const int rounds = (items + ncu * cap - 1) / (ncu * cap);
  int rpw = (items + ncu * rounds - 1) / (ncu * rounds);
  const int floor_rows = M > 32 ? 16 : (M > 16 ? 8 : 4);
  if (rpw < floor_rows) rpw = floor_rows;
  if (p.rope_table) rpw = (rpw + 1) & ~1;
  if (rpw > cap) rpw = cap;
  p.rpw = rpw;
  p.nwg = (items + rpw - 1) / rpw;
}

// the sums of squares that come with a projection's input
static int sb_fill_norm(const lr_row_norm_t* q, Proj& p) {
  if (q == nullptr || q->sums == nullptr) return LR_OK;
  LR_REQUIRE_PTR(q->sums);
  if (q->count <= 0 || q->dim != p.K) return LR_E_SHAPE;
  if (q->count > LR_ROW_NORM_MAX) return LR_E_UNSUPPORTED;
  p.norm_sums = q->sums;
  p.norm_count = q->count;
  p.norm_dim = q->dim;
  p.norm_eps = q->eps;
  if (q->fold_sums) {
    LR_REQUIRE_PTR(q->fold_sums);
    if (q->fold_total == nullptr) return LR_E_NULL;
    if (q->fold_count <= 0) return LR_E_SHAPE;
    if (q->fold_count > LR_ROW_NORM_MAX) return LR_E_UNSUPPORTED;
    p.fold_sums = q->fold_sums;
    p.fold_total = q->fold_total;
    p.fold_count = q->fold_count;
  }
  return LR_OK;
}

// lr_projection_t -> Proj (validated; rpw / nwg are set by plan())
static int sb_fill_projection(const lr_projection_t& q, Proj& p) {
  LR_REQUIRE_PTR(q.x);
  LR_REQUIRE_PTR(q.w);
  LR_REQUIRE_PTR(q.y);
  if (q.N <= 0 || q.K <= 0 || q.ldx < q.K) return LR_E_SHAPE;
  if (q.epilogue != LR_EPI_NONE && q.epilogue != LR_EPI_SWIGLU && q.epilogue != LR_EPI_ROPE_KV) return LR_E_SHAPE;
  const bool pair = q.epilogue == LR_EPI_SWIGLU;
  if (pair && q.N % 2) return LR_E_SHAPE;
  if (q.ldy < (pair ? q.N / 2 : q.N)) return LR_E_SHAPE;
  if (q.K % 8 || q.ldx % 8) return LR_E_ALIGN;
  // offsets inside a band and inside the input rows are 32-bit
  if ((int64_t)64 * q.ldx * 2 >= 0x7fffffff || ((int64_t)(pair ? q.N / 2 : 0) + 64) * q.K * 2 >= 0x7fffffff)
    return LR_E_UNSUPPORTED;
  p = Proj{};
  p.x = (const u16*)q.x; p.w = (const u16*)q.w; p.y = (u16*)q.y;
  p.ldx = q.ldx; p.ldy = q.ldy; p.N = q.N; p.K = q.K;
  p.in_turn = band_in_turn(q.K);
  p.pair_off = pair ? q.N / 2 : 0;
  if (q.epilogue == LR_EPI_ROPE_KV) {
    const lr_rope_kv_t* r = q.rope;
    if (r == nullptr || r->pos == nullptr) return LR_E_NULL;
    LR_REQUIRE_PTR(r->table);
    LR_REQUIRE_PTR(r->k_cache);
    LR_REQUIRE_PTR(r->v_cache);
    if (r->n_head <= 0 || r->n_kv_head <= 0 || r->head_dim <= 0 || r->smax <= 0 || r->block_size <= 0 ||
        (int64_t)(r->n_head + 2 * r->n_kv_head) * r->head_dim != q.N || q.ldy % 2)
      return LR_E_SHAPE;
    if (r->head_dim % 8) return LR_E_ALIGN;
    p.rope_table = (const u16*)r->table; p.pos = r->pos; p.k_cache = (u16*)r->k_cache; p.v_cache = (u16*)r->v_cache;
    p.err = r->err; p.Hq = r->n_head; p.Hkv = r->n_kv_head; p.hd = r->head_dim; p.Smax = r->smax;
    p.block_size = r->block_size;
  }
  return LR_OK;
}

// lr_projection_fp8_t -> Proj for the e4m3 bands (W8 = true)
static int sb_fill_projection_fp8(const lr_projection_fp8_t& q, Proj& p) {
  if (q.scales == nullptr) return LR_E_NULL;
  if (lr_misaligned(q.w8)) return LR_E_ALIGN;
  if (q.K % 16) return LR_E_ALIGN;
  // the bf16 projection's checks, with the weight pointer standing in (its rows are half as long: every
  // 32-bit offset limit holds a fortiori)
  const lr_projection_t as_bf16 = {q.x, q.ldx, q.w8, q.y, q.ldy, q.N, q.K, q.epilogue, q.rope};
  const int rc = sb_fill_projection(as_bf16, p);
  if (rc != LR_OK) return rc;
  p.scales = (const u16*)q.scales;
  return LR_OK;
}

}  // namespace
