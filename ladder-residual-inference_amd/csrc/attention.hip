// Attention over the contiguous [B, Hkv, Smax, hd] KV cache.
//
// Decode (one query per sequence): the valid keys 0..pos are cut into `nsplit` contiguous chunks;
// one workgroup per (chunk, kv head, sequence) serves ALL q heads of that kv head, so K and V are
// read from HBM once per GQA group.  Scores, softmax and P.V stay in fp32 (P is never rounded),
// chunk results carry their own (max, sum) and a second tiny kernel merges them in chunk order.
// Only slots <= pos are touched: with the reference's boolean mask the other slots get weight
// exp(-inf) = 0, so this is the same function of the cache.
//
// Prefill (S >= 16 queries per sequence): flash-style causal attention on the matrix cores in the
// transposed form (k_attn_prefill_mfma below: a query is a lane, four waves share K / V^T tiles in
// LDS, P enters the second product as bf16 hi + lo so the fp32 softmax weights survive).  Shorter
// inputs (1 < S < 16) use the older lane-per-query kernel (k_attn_prefill: running max / sum /
// output in registers, K/V tiles of 32 keys broadcast from LDS as fp32).  Both: exact fp32
// softmax semantics, one rounding of the output.
#include "lr_common.h"
#include "attn_decode_item.h"
#include <atomic>

// ------------------------------------------------------------------------------------ decode
extern "C" size_t lr_attn_decode_scratch_bytes(int B, int Hq, int hd, int Smax) {
  if (B <= 0 || Hq <= 0 || hd <= 0 || Smax <= 0) return 0;
  return (size_t)B * Hq * attn_nsplit_cap(Smax) * (hd + 2) * sizeof(float);
}

template <int HD, int G, int GROUPS>
__global__ __launch_bounds__(256) void k_attn_decode_partial(const u16* __restrict__ q, int64_t ldq,
                                                             const u16* __restrict__ kc, const u16* __restrict__ vc,
                                                             const int32_t* __restrict__ pos_ptr,
                                                             float* __restrict__ o_part, float* __restrict__ ml_part,
                                                             int Hkv, int Smax, int nsplit, int chunk_max) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  attn_partial_item<HD, G, GROUPS>(q, ldq, kc, vc, pos_ptr, o_part, ml_part, Hkv, Smax, nsplit, chunk_max, blockIdx.x,
                           blockIdx.y, blockIdx.z, smem);
}

template <int HD, int G, int GROUPS>
static int launch_decode_as(const u16* q, int64_t ldq, const u16* kc, const u16* vc, const int32_t* pos, u16* y,
                            int64_t ldy, int B, int Hkv, int Smax, int nsplit, int chunk_max, float* scratch, hipStream_t s) {
  const int Hq = Hkv * G;
  float* o_part = scratch;
  float* ml_part = scratch + (size_t)B * Hq * nsplit * HD;
  const size_t lds = (size_t)attn_item_lds_floats<HD, G>(chunk_max) * sizeof(float);
  static std::atomic<unsigned long long> lds_raised{0};
  if (!lr_raise_lds_limit(reinterpret_cast<const void*>(&k_attn_decode_partial<HD, G, GROUPS>), lds, lds_raised)) return LR_E_LAUNCH;
  k_attn_decode_partial<HD, G, GROUPS><<<dim3(nsplit, Hkv, B), dim3(256), lds, s>>>(q, ldq, kc, vc, pos, o_part, ml_part, Hkv,
                                                                                    Smax, nsplit, chunk_max);
  launch_attn_combine<HD>(o_part, ml_part, y, ldy, Hq, B, nsplit, s);
  return lr_launch_status();
}
template <int HD, int G>
static int launch_decode(const u16* q, int64_t ldq, const u16* kc, const u16* vc, const int32_t* pos, u16* y,
                         int64_t ldy, int B, int Hkv, int Smax, float* scratch, hipStream_t s) {
  const int nsplit = attn_pick_nsplit(B, Hkv, Smax);
  const int chunk_max = ((Smax + nsplit - 1) / nsplit + 3) & ~3;
  return attn_two_groups(chunk_max) ? launch_decode_as<HD, G, 2>(q, ldq, kc, vc, pos, y, ldy, B, Hkv, Smax, nsplit, chunk_max, scratch, s)
                                    : launch_decode_as<HD, G, 4>(q, ldq, kc, vc, pos, y, ldy, B, Hkv, Smax, nsplit, chunk_max, scratch, s);
}

extern "C" int lr_attn_decode(const void* q, int64_t ldq, const void* k_cache, const void* v_cache,
                              const int32_t* pos, void* y, int64_t ldy, int B, int Hq, int Hkv, int hd, int Smax,
                              void* scratch, size_t scratch_bytes, lr_stream_t stream) {
  LR_REQUIRE_PTR(q);
  LR_REQUIRE_PTR(k_cache);
  LR_REQUIRE_PTR(v_cache);
  LR_REQUIRE_PTR(y);
  LR_REQUIRE_PTR(scratch);
  if (pos == nullptr) return LR_E_NULL;
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || hd <= 0 || Smax <= 0 || Hq % Hkv) return LR_E_SHAPE;
  if ((int64_t)Smax * hd * 2 >= 0x7fffffff) return LR_E_UNSUPPORTED;  // the rows of one (sequence, head) are addressed with 32-bit offsets
  if (ldq < (int64_t)Hq * hd || ldy < (int64_t)Hq * hd || B > 65535) return LR_E_SHAPE;
  if (ldq % 8 || ldy % 8) return LR_E_ALIGN;
  if (scratch_bytes < lr_attn_decode_scratch_bytes(B, Hq, hd, Smax)) return LR_E_SHAPE;
  const int G = Hq / Hkv;
  hipStream_t s = (hipStream_t)stream;
#define LR_DEC(HDV, GV)                                                                                           \
  if (hd == HDV && G == GV)                                                                                       \
    return launch_decode<HDV, GV>((const u16*)q, ldq, (const u16*)k_cache, (const u16*)v_cache, pos, (u16*)y, ldy, \
                                  B, Hkv, Smax, (float*)scratch, s);
  LR_DEC(128, 1) LR_DEC(128, 2) LR_DEC(128, 4) LR_DEC(128, 8) LR_DEC(128, 16)
  LR_DEC(64, 1) LR_DEC(64, 2) LR_DEC(64, 4) LR_DEC(64, 8)
#undef LR_DEC
  return LR_E_UNSUPPORTED;
}

// ------------------------------------------------------------------------------------ decode, allocation-free
// lr_attn_decode for callers that cannot allocate or carry a workspace: the split-KV partial
// results live in a fixed device array of this library instead of caller memory.  `scratch` below
// is, in host code, only a stand-in for the device symbol: the address kernels may use is looked
// up once per device with hipGetSymbolAddress (every device holds its own copy of the array at
// its own address) and kept in g_static_scratch; host code never passes `scratch` itself.
constexpr size_t LR_STATIC_SCRATCH_BYTES = LR_ATTN_DECODE_STATIC_MAX_BYTES;
static __device__ __align__(256) unsigned char scratch[LR_STATIC_SCRATCH_BYTES];
static std::atomic<float*> g_static_scratch[LR_MAX_DEVICES];

// device address of `scratch` on the current device (looked up on the first call per device)
static int static_scratch(float** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= LR_MAX_DEVICES) return LR_E_LAUNCH;
  float* p = g_static_scratch[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    void* sym = nullptr;
    if (hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch)) != hipSuccess || sym == nullptr) {
      (void)hipGetLastError();
      return LR_E_LAUNCH;
    }
    p = reinterpret_cast<float*>(sym);
    g_static_scratch[dev].store(p, std::memory_order_release);  // concurrent first calls store the same address
  }
  *out = p;
  return LR_OK;
}

extern "C" int lr_attn_decode_static(const void* q, int64_t ldq, const void* k_cache, const void* v_cache,
                                     const int32_t* pos, void* y, int64_t ldy, int B, int Hq, int Hkv, int hd,
                                     int Smax, lr_stream_t stream) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || hd <= 0 || Smax <= 0) return LR_E_SHAPE;
  const size_t need = lr_attn_decode_scratch_bytes(B, Hq, hd, Smax);
  if (need > LR_STATIC_SCRATCH_BYTES) return LR_E_TOO_LARGE;
  float* ws = nullptr;
  const int rc = static_scratch(&ws);
  if (rc != LR_OK) return rc;
  return lr_attn_decode(q, ldq, k_cache, v_cache, pos, y, ldy, B, Hq, Hkv, hd, Smax, ws, need, stream);
}

// ------------------------------------------------------------------------------------ prefill
template <int HD>
__global__ __launch_bounds__(64) void k_attn_prefill(const u16* __restrict__ q, int64_t ldq,
                                                     const u16* __restrict__ kc, const u16* __restrict__ vc,
                                                     const int32_t* __restrict__ pos, u16* __restrict__ y, int64_t ldy,
                                                     int S, int Hq, int Hkv, int Smax) {
  constexpr int TK = 32;
  __shared__ __attribute__((aligned(16))) float ks[TK * HD];
  __shared__ __attribute__((aligned(16))) float vs[TK * HD];
  const int lane = threadIdx.x;
  const int h = blockIdx.y, b = blockIdx.z;
  const int kvh = h / (Hq / Hkv);
  const int s = blockIdx.x * 64 + lane;
  const bool valid = s < S;
  int p = valid ? pos[s] : -1;
  p = p >= Smax ? Smax - 1 : p;
  int kmax = p;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const int t = __shfl_xor(kmax, o, LR_WAVE);
    kmax = t > kmax ? t : kmax;
  }
  const int nkeys = kmax + 1;

  float qf[HD];
  {
    const u16* qrow = q + ((int64_t)b * S + (valid ? s : 0)) * ldq + h * HD;
#pragma unroll
    for (int c = 0; c < HD; c += 8) unpack8(ld16(qrow + c), &qf[c]);
  }
  float o[HD];
#pragma unroll
  for (int d = 0; d < HD; ++d) o[d] = 0.0f;
  float m = -INFINITY, l = 0.0f;
  const float scale = rsqrtf((float)HD);
  const u16* kbase = kc + ((int64_t)b * Hkv + kvh) * Smax * HD;
  const u16* vbase = vc + ((int64_t)b * Hkv + kvh) * Smax * HD;

  for (int t0 = 0; t0 < nkeys; t0 += TK) {
    // stage TK keys and values as fp32: TK * HD / 8 chunks of 8 elements over 64 lanes
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TK * HD / 8 / 64; ++i) {
      const int c = lane + i * 64;
      const int key = t0 + c / (HD / 8), d = (c % (HD / 8)) * 8;
      float kf[8], vf[8];
      if (key < nkeys) {
        unpack8(ld16(kbase + (int64_t)key * HD + d), kf);
        unpack8(ld16(vbase + (int64_t)key * HD + d), vf);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) kf[j] = vf[j] = 0.0f;
      }
      float4* kd = reinterpret_cast<float4*>(&ks[(c / (HD / 8)) * HD + d]);
      float4* vd = reinterpret_cast<float4*>(&vs[(c / (HD / 8)) * HD + d]);
      kd[0] = make_float4(kf[0], kf[1], kf[2], kf[3]);
      kd[1] = make_float4(kf[4], kf[5], kf[6], kf[7]);
      vd[0] = make_float4(vf[0], vf[1], vf[2], vf[3]);
      vd[1] = make_float4(vf[4], vf[5], vf[6], vf[7]);
    }
    __syncthreads();

    float sc[TK];
    float tmax = -INFINITY;
#pragma unroll
    for (int j = 0; j < TK; ++j) {
      float a = 0.0f;
#pragma unroll
      for (int d = 0; d < HD; d += 4) {
        const float4 kk = *reinterpret_cast<const float4*>(&ks[j * HD + d]);
        a = fmaf(qf[d], kk.x, a);
        a = fmaf(qf[d + 1], kk.y, a);
        a = fmaf(qf[d + 2], kk.z, a);
        a = fmaf(qf[d + 3], kk.w, a);
      }
      sc[j] = (t0 + j <= p) ? a * scale : -INFINITY;
      tmax = fmaxf(tmax, sc[j]);
    }
    const float mn = fmaxf(m, tmax);
    if (mn != -INFINITY) {  // this lane sees at least one key so far
      const float corr = expf(m - mn);  // m == -inf -> 0
      l *= corr;
#pragma unroll
      for (int d = 0; d < HD; ++d) o[d] *= corr;
#pragma unroll
      for (int j = 0; j < TK; ++j) {
        const float pj = expf(sc[j] - mn);  // masked -> 0
        l += pj;
#pragma unroll
        for (int d = 0; d < HD; d += 4) {
          const float4 vv = *reinterpret_cast<const float4*>(&vs[j * HD + d]);
          o[d] = fmaf(pj, vv.x, o[d]);
          o[d + 1] = fmaf(pj, vv.y, o[d + 1]);
          o[d + 2] = fmaf(pj, vv.z, o[d + 2]);
          o[d + 3] = fmaf(pj, vv.w, o[d + 3]);
        }
      }
      m = mn;
    }
  }
  if (valid) {
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    u16* yrow = y + ((int64_t)b * S + s) * ldy + h * HD;
#pragma unroll
    for (int c = 0; c < HD; c += 8) {
      float t[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) t[j] = o[c + j] * inv;
      st16(yrow + c, pack8(t));
    }
  }
}

// ----------------------------------------------------------------------- prefill on the matrix cores
// Flash-style causal attention in the TRANSPOSED form, so that everything per query sits in one lane:
//   S^T[key][q]  = sum_d K[key][d] Q[q][d]          (A = K tile from LDS, B = Q from registers)
//   O^T[d][q]   += sum_key V^T[d][key] P^T[key][q]  (A = V^T tile from LDS, B = P^T from the S^T registers)
// with v_mfma_f32_32x32x16_bf16.  An accumulator column is a query (lane % 32), so row maxima, sums and
// the rescaling factor are per-lane scalars; the 16 S^T values a lane holds for its query are exactly,
// in order, the B operand of the two PV k-steps (the key order of a k-step is free as long as the V^T
// operand uses the same one), so P never moves between lanes.  P enters the bf16 MFMA as hi + lo
// (p = bf16(p) + bf16(p - bf16(p))), which keeps the fp32 softmax weights to ~2^-17: the result matches
// the fp32 "math" attention of the eager reference (utils.py:247-258) to rounding of the final bf16.
// A workgroup is 4 waves = NWH heads of one kv head x NWQ tiles of 32 queries sharing the K / V tiles.
// e^x through the hardware exp2 (1 ulp in fp32: far below the bf16 rounding of the output), with the score scale
// folded into its argument; the library expf costs ~15 VALU instructions, and this kernel is VALU-bound next to
// its MFMAs
// max(a, b) as the median of {a, b, +inf}: one instruction (fmaxf makes the compiler canonicalise both operands
// first, an instruction each, when they come out of a matrix-core product).  Not for NaN operands.
// (No inline assembler here: the compiler does not count the wait states between a matrix-core instruction and
// an assembler statement that reads its result, and the statement then reads the registers too early.)
__device__ __forceinline__ float max_med3(float a, float b) { return __builtin_amdgcn_fmed3f(a, b, INFINITY); }
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }
constexpr float PREFILL_TAU2 = 8.0f;  // log2 of the largest softmax weight before the reference point moves

struct WindowKeys {
  int window, n_keys, ld, dk, dv;
  float scale;
};

// Keys come 64 at a time, K and V as they lie, by loads straight into LDS (a row of HD elements is 16-byte pieces; which piece lands
// where is XOR-ed with the key, see key_swizzle and value_swizzle, so that the fragment reads below meet no bank twice), one portion
// ahead of the products: one barrier per 64 keys.  V^T fragments are read across the rows (ds_read_b64_tr_b16).
// KSP 2: a grid that leaves CUs without a second workgroup has eight waves in a workgroup, the second four the second 32 keys of every portion
// for the same queries; their results are merged at the end.  From 512 keys on, where that pays for the merge (us, four waves / eight: 32 heads
// of 128, 512 tokens 17.5 / 17.3, 777 23.3 / 22.4; 16 heads, 1500 tokens, window of 1024 30.7 / 28.1, of 128 10.9 / 11.7).  Keys, as far as
// the host knows them: those of the call itself or of its window.  (A portion of 32 to 256 tokens at position 3000 would be 10 to 15 %
// faster with eight waves, 32 tokens of 32 heads 72 / 62, but at position 0, where it is 6.5 / 8.2, looks the same to the host.)
// KEYS 32: 32 at a time and with fewer registers, so that three workgroups share a CU where the grid has as many (64 / 32: 32 heads, 8 kv heads of
// 128, 8 x 2048 tokens 401 / 397, 4 x 777 44.2 / 41.8, 4 x 1024 62.5 / 63.1, 4 x 1300 93.0 / 96.5; 2 x 1500 of window 128 27.2 / 25.0),
// and for the 33 to 96 queries of two heads to a workgroup, whose first 32 have no use for the second 32 keys (28 heads, 14 kv heads, 64 tokens
// 7.5 / 6.9).
// PREFILL_EACH: a portion's 32-key tiles one after the other, with a reference point each: up to 128 queries of heads of 128, which have KEYS 32's
// results so, and a barrier per 64 keys (KEYS 32 / so: 32 heads, 8 kv heads, 64 tokens 7.28 / 7.07, 100 8.21 / 8.17, 128 9.21 / 8.74, 4 x 32 tokens
// at position 3000 102 / 92.  Both tiles at a time would be 7.66, 8.37 and 74 us at 100, 128 and 4 x 32, in other last bits: a whole model's outputs,
// 80 layers later, are 1 to 2 % of their norm apart by that, no nearer to 64 bits).
// PREFILL_HALF: a last portion of up to 32 keys is computed as such (us without / with: 32 heads, 8 kv heads of 64, 32 tokens 5.32 / 4.64, 100 tokens
// 6.42 / 5.70; of 128, 300 tokens 12.9 / 12.1), and narrow windows have few others (1500 tokens, window of 128 11.1 / 10.1).  Heads of 64: up to 128
// keys, the loop is slower beside a second copy of its body (32 tokens at position 3000 47.5 / 51.0).
// Heads of 64 keep to the 128 registers that let four workgroups share a CU (40 heads, 20 kv heads, 3000 tokens, window of 128: three to a CU
// 22.6 us, four 19.0).
// Bound: matrix instructions 48 % of a SIMD's cycles, vector instructions 46 % (exponentials at a quarter of the rate, splitting P), which hardly
// run at the same time, in another wave or between the matrix instructions of the same one (written so, it took as long).  No bank
// conflicts.  Before (32 keys in one LDS buffer through registers, V transposed on its way in, two barriers) / now, us: 32 heads of 128,
// 8 kv heads: 8 x 2048 tokens 460 / 396 (598 / 694 TFLOP/s of products), 4 x 1300 112 / 96, 2 x 1000 50.8 / 35.9, 777 28.4 / 22.4, 300 14.0 / 12.1,
// 100 8.2 / 8.2, 32 6.3 / 6.4, 16 5.6 / 5.7; of 64: 4 x 1024 59.9 / 40.1, 512 15.1 / 11.8, 100 6.3 / 5.8, 32 4.8 / 4.7.
typedef int i32x4_t __attribute__((ext_vector_type(4)));
constexpr int PREFILL_PARTS_FROM = 512, PREFILL_HALF_TO = 128;   // keys that are seen, see above
enum { PREFILL_WHOLE, PREFILL_HALF, PREFILL_EACH };
template <int HD, int KSP, int KEYS>
struct PrefillLds {
  static constexpr int TILE = KEYS * HD * 2, STAGE = 2 * TILE;   // a portion's keys or values; both
  static constexpr int MERGE = KSP == 2 ? 4 * (HD / 2 + 2) * 64 * 4 : 0;
  static constexpr int KMAX = 2 * STAGE > MERGE ? 2 * STAGE : MERGE, BYTES = KMAX + 32;   // (KMAX: an int of each of up to eight waves)
};
// the place among a row's pieces is the piece's number XOR this: 16 lanes reading one piece of 16 consecutive keys, and 16 reading four
// neighbouring pieces (32 dimensions) of four keys, touch every bank once
template <int HD>
__device__ __forceinline__ int key_swizzle(int key) { return HD == 128 ? key & 15 : (key >> 1) & 7; }
template <int HD>
__device__ __forceinline__ int value_swizzle(int key) { return HD == 128 ? (key & 3) << 2 : ((key >> 1) & 1) << 2; }

// WIN (lr_window_attention): a sliding window, the score scale as an argument, and the kv heads' keys and values side by
// side as rows of a matrix, in the order lr_latent_window gives them; head sizes up to HD.
template <int HD, int NWH, int KSP, int KEYS, int HALF, bool WIN>
__global__ __launch_bounds__(256 * KSP, HD == 64 ? 4 : KEYS == 32 ? 3 : 2) void k_attn_prefill_mfma(const u16* __restrict__ q, int64_t ldq,
                                                                    const u16* __restrict__ kc, const u16* __restrict__ vc,
                                                                    const int32_t* __restrict__ pos, u16* __restrict__ y,
                                                                    int64_t ldy, int S, int Hq, int Hkv, int Smax,
                                                                    const WindowKeys w = {}) {
  constexpr int NWQ = 4 / NWH;            // query tiles per workgroup
  constexpr int KS = HD / 16;             // k-steps of the score product
  constexpr int DT = HD / 32;             // 32-row tiles of O^T
  using L = PrefillLds<HD, KSP, KEYS>;
  constexpr int NS = KEYS / 32 / KSP;             // 32-key tiles of a portion that a wave takes
  constexpr int NW = 4 * KSP, RB = HD * 2, PIECES = RB / 16;
  constexpr int RPL = 1024 / RB, LOADS = KEYS / RPL / NW;   // rows per load instruction, a wave's loads of K or V per portion
  extern __shared__ __attribute__((aligned(1024))) unsigned char prefill_lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), part = KSP == 2 ? wave >> 2 : 0, w4 = wave & 3;
  const int col = lane & 31, half = lane >> 5;
  const int G = Hq / Hkv;
  const int hgroups = G / NWH;                       // workgroups per kv head along heads
  // Which (query block, head group, sequence) this workgroup takes.  The grid is one-dimensional and workgroup i
  // runs on XCD i % 8, each with an L2 of its own: XCD k takes the k-th eighth of the work in its logical order, so
  // that the workgroups that share the K / V rows of one (sequence, kv head) -- the query blocks, neighbours in that
  // order -- meet in one L2.  Inside, the query blocks go from the last (the longest history) to the first.
  const int gx = (S + 32 * NWQ - 1) / (32 * NWQ), gy = Hq / NWH;
  int bx, by, b;
  {
    const int n = gridDim.x, xcd = blockIdx.x % 8, idx = blockIdx.x / 8, columns = n / gx;
    int column;   // a head group of a sequence
    if (columns % 8 == 0) {
      column = xcd * (columns / 8) + idx % (columns / 8);   // (all columns' longest first: 8 x 2048 tokens 414 us -> 399)
      bx = gx - 1 - idx / (columns / 8);
    } else {
      const int wg = xcd * (n / 8) + (xcd < n % 8 ? xcd : n % 8) + idx;
      column = wg / gx;
      bx = gx - 1 - wg % gx;
    }
    by = column % gy;
    b = column / gy;
  }
  const int kvh = by / hgroups;
  const int head = kvh * G + (by % hgroups) * NWH + (w4 % NWH);
  const int s = (bx * NWQ + w4 / NWH) * 32 + col;  // this lane's query
  const bool valid = s < S;
  int p = valid ? pos[s] : -1;
  if constexpr (WIN) {
    if (valid) p -= lr_window_base(pos[0], w.window, w.n_keys, Smax);   // this query's row among the keys
    p = p >= w.n_keys ? w.n_keys - 1 : p;
  } else {
    p = p >= Smax ? Smax - 1 : p;
  }
  // the last and the first key of this wave's queries (lanes without one do not count), and
  // the keys needed by anybody in the workgroup
  int kmax = p, pmin = valid ? p : 0x7fffffff;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const int t = __shfl_xor(kmax, o, LR_WAVE), u = __shfl_xor(pmin, o, LR_WAVE);
    kmax = t > kmax ? t : kmax;
    pmin = u < pmin ? u : pmin;
  }
  const int pmax = __builtin_amdgcn_readfirstlane(kmax);
  pmin = __builtin_amdgcn_readfirstlane(pmin);
  if constexpr (NWQ > 1) {   // (else all waves have the same queries)
    int* const s_kmax = reinterpret_cast<int*>(prefill_lds + L::KMAX);
    if (lane == 0) s_kmax[wave] = kmax;
    __syncthreads();
    kmax = max(max(s_kmax[0], s_kmax[1]), max(s_kmax[2], s_kmax[3]));
  }
  const int nkeys = __builtin_amdgcn_readfirstlane(kmax + 1);
  // (WIN) the first portion anybody in the workgroup sees
  int t_first = 0;
  if constexpr (WIN) {
    int lo = 0x7fffffff;
#pragma unroll
    for (int t = 0; t < NWQ; ++t) {
      const int s_lo = (bx * NWQ + t) * 32;   // positions are consecutive: a query tile's first query is its smallest
      if (s_lo < S) lo = min(lo, pos[s_lo] - lr_window_base(pos[0], w.window, w.n_keys, Smax));
    }
    lo = lo - w.window + 1;
    t_first = __builtin_amdgcn_readfirstlane(lo > 0 ? lo & ~31 : 0);
  }

  // Q as B operands: k-step ks_ holds elements 16 ks_ + 8 half .. + 8 of this lane's query
  u32x4_t qb[KS];
  {
    const int dq = WIN ? w.dk : HD;
    const u16* qrow = q + ((int64_t)b * S + (valid ? s : 0)) * ldq + head * dq;
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const uint4 t = valid && 16 * i + 8 * half < dq ? ld16(qrow + 16 * i + 8 * half) : make_uint4(0, 0, 0, 0);
      qb[i] = u32x4_t{t.x, t.y, t.z, t.w};
    }
    // (waited for here: inside the loop the compiler's wait for them would be one for the next portion)
#pragma unroll
    for (int i = 0; i < KS; ++i) asm volatile("" : "+v"(qb[i]));
  }
  f32x16_t o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[d][v] = 0.0f;
  float m = -INFINITY, l = 0.0f;  // m: reference point in raw score units; l: this lane's half of the row sum
  const float c2 = (WIN ? w.scale : rsqrtf((float)HD)) * 1.4426950408889634f;  // e^(x / sqrt(HD)) = 2^(x c2)
  const float tau_raw = PREFILL_TAU2 / c2;
  const int krow = WIN ? w.ld : HD;   // elements from key to key
  const u16* kbase = WIN ? kc + (int64_t)b * w.n_keys * w.ld + kvh * w.dk : kc + ((int64_t)b * Hkv + kvh) * Smax * HD;
  const u16* vbase = WIN ? vc + (int64_t)b * w.n_keys * w.ld + kvh * w.dv : vc + ((int64_t)b * Hkv + kvh) * Smax * HD;

  // Loads: instruction i of a wave covers rows (i NW + wave) RPL .. of a portion, a lane the piece that belongs to its place.  (A key
  // beyond the needed ones, or a piece beyond the head's, is asked for outside the resource and comes as zeros.)
  constexpr int OUT = (int)0x80000000;
  const int lrow = lane / PIECES, place = lane % PIECES;
  const int kpiece = place ^ key_swizzle<HD>(wave * RPL + lrow), vpiece = place ^ value_swizzle<HD>(lrow);
  static_assert(NW * RPL % 16 == 0 && RPL % 4 == 0, "a lane's piece is the same for all of a wave's loads");
  const int kvoff = !WIN || kpiece * 8 < w.dk ? lrow * krow * 2 + kpiece * 16 : OUT;
  const int vvoff = !WIN || vpiece * 8 < w.dv ? lrow * krow * 2 + vpiece * 16 : OUT;
  auto resource = [](const u16* at) {
    return i32x4_t{(int)(u32)(unsigned long long)at, (int)(u32)((unsigned long long)at >> 32) & 0xffff, 0x7fffffff, 0x00020000};
  };
  const i32x4_t kres = resource(kbase), vres = resource(vbase);
  const u32 lds0 = __builtin_amdgcn_readfirstlane((u32)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)prefill_lds);
  auto load16 = [](const i32x4_t& res, int voff, int soff, u32 lds) {
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"{m0}"(lds), "v"(voff), "s"(res), "s"(soff) : "memory");
  };
  auto stage = [&](int t0, int buf) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int first = (i * NW + wave) * RPL;
      const bool ok = t0 + first + lrow < nkeys;
      const int soff = t0 + first < nkeys ? (t0 + first) * krow * 2 : 0;
      const u32 at = lds0 + buf * L::STAGE + (i * NW + wave) * 1024;
      load16(kres, ok ? kvoff : OUT, soff, at);
      load16(vres, ok ? vvoff : OUT, soff, at + L::TILE);
    }
  };
  // where this lane reads: the K fragments of key `col` of its tile (k-step i: XOR 32 i), and 4 dimensions of key (lane % 16) / 4
  // of the four keys whose values 16 lanes exchange (32-row tile d of O^T: see below)
  const int kat = (part * 32 + col) * RB + ((half ^ key_swizzle<HD>(col)) * 16);
  const int vkey = (lane & 15) >> 2;
  int vat[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) {
    const int piece = 4 * d + ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
    vat[d] = L::TILE + (part * 32 + 4 * half + vkey) * RB + (piece ^ value_swizzle<HD>(vkey)) * 16 + (lane & 1) * 8;
  }
  if (t_first < nkeys) stage(t_first, 0);
  int buf = 0;
  // N 32-key tiles of the portion at t0, from its tile `first` on, for this wave's queries
  auto tiles = [&](auto N_, const int t0, const int buf, const int first) {
    constexpr int N = decltype(N_)::value;
    const int tk = t0 + (part + first) * 32;
    if (tk > pmax || (WIN && tk + 32 * N - 1 <= pmin - w.window)) return;   // nothing here for them
    const unsigned char* const at = prefill_lds + buf * L::STAGE + first * 32 * RB;
    // ---- S^T tiles: rows = keys, columns = queries
    f32x16_t sacc[N];
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
      for (int v = 0; v < 16; ++v) sacc[n][v] = 0.0f;
    u32x4_t ka[KS][N];   // (all on their way before the first product)
#pragma unroll
    for (int i = 0; i < KS; ++i)
#pragma unroll
      for (int n = 0; n < N; ++n) ka[i][n] = *reinterpret_cast<const u32x4_t*>(at + (kat ^ (32 * i)) + n * 32 * RB);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < KS; ++i)
#pragma unroll
      for (int n = 0; n < N; ++n)
        sacc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, ka[i][n]), __builtin_bit_cast(bf16x8_t, qb[i]),
                                                          sacc[n], 0, 0, 0);
    // element v of tile n is key tk + 32 n + (v / 4) * 8 + half * 4 + v % 4 for query `col`; only a portion that reaches past the
    // smallest position of the wave's queries has anything to mask
    if (tk + 32 * N - 1 > pmin || (WIN && tk <= pmax - w.window)) {
#pragma unroll
      for (int n = 0; n < N; ++n)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int key = tk + 32 * n + (v / 4) * 8 + half * 4 + (v % 4);
          sacc[n][v] = key <= p && (!WIN || key > p - w.window) ? sacc[n][v] : -INFINITY;
        }
    }
    float tmax = max_med3(sacc[0][0], sacc[0][1]);
#pragma unroll
    for (int v = 2; v < 16 * N; ++v) tmax = max_med3(tmax, sacc[v / 16][v % 16]);
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, LR_WAVE));
    // The reference point m of the exponentials follows the running maximum lazily: it moves only when a portion's
    // maximum exceeds it by more than PREFILL_TAU2 / c2, so the weights stay below 2^PREFILL_TAU2 (harmless in fp32,
    // and hi + lo keeps their relative precision) and the accumulators are rescaled on few portions instead of on
    // most (with 32 queries per wave, some running maximum moves in the majority of them).
    const bool grow = tmax > m + tau_raw;  // m = -inf: any finite maximum
    const float mn = grow ? tmax : m;
    const float corr = grow ? exp2_hw((m - mn) * c2) : 1.0f;  // m = -inf -> 0
    const float nmc = mn == -INFINITY ? 0.0f : -mn * c2;     // nothing seen yet: every score is -inf, weight 0
    m = mn;
    l *= corr;
    if (__any(grow)) {
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[d][v] *= corr;
    }
#pragma unroll
    for (int n = 0; n < N; ++n) {
      u32x4_t phi[2], plo[2];
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float a0 = exp2_hw(fmaf(sacc[n][8 * h2 + 2 * j], c2, nmc));  // masked -> 0
          const float a1 = exp2_hw(fmaf(sacc[n][8 * h2 + 2 * j + 1], c2, nmc));
          l += a0 + a1;
          const u32 hi = pack_bf2(a0, a1);
          phi[h2][j] = hi;
          plo[h2][j] = pack_bf2(a0 - __uint_as_float(hi << 16), a1 - __uint_as_float(hi & 0xffff0000u));
        }
      // ---- O^T += V^T P^T ; k-step h2 covers keys 16 h2 + {0..3, 8..11} + 4 half of the tile, in the order of sacc
      // (consecutive matrix instructions go to different accumulators: one that adds to the result of the instruction
      // right before it has to wait for that result)
#pragma unroll
      for (int h2 = 0; h2 < 2; ++h2) {
        bf16x8_t va[DT];
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          // 16 lanes read 4 keys of 16 dimensions, a lane 4 of one key, and receive the 4 keys of one dimension each
          const unsigned char* const v0 = at + vat[d] + (n * 32 + 16 * h2) * RB;
          const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(v0));
          const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(v0 + 8 * RB));
          va[d] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
#pragma unroll
        for (int d = 0; d < DT; ++d)
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[d], __builtin_bit_cast(bf16x8_t, phi[h2]), o[d], 0, 0, 0);
#pragma unroll
        for (int d = 0; d < DT; ++d)
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[d], __builtin_bit_cast(bf16x8_t, plo[h2]), o[d], 0, 0, 0);
      }
    }
  };
  // (that portion has arrived, for all waves, and nobody reads the one before any more)
  auto arrived = [] { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  constexpr int LAST = HALF == PREFILL_HALF ? 32 : 0;
  int t0 = t_first;
  for (; t0 + LAST < nkeys; t0 += KEYS, buf ^= 1) {
    arrived();
    if (t0 + KEYS < nkeys) stage(t0 + KEYS, buf ^ 1);
    if constexpr (HALF == PREFILL_EACH) {
#pragma unroll 1
      for (int first = 0; first < NS && t0 + 32 * first < nkeys; ++first) tiles(std::integral_constant<int, 1>{}, t0, buf, first);
    } else {
      tiles(std::integral_constant<int, NS>{}, t0, buf, 0);
    }
  }
  if (HALF == PREFILL_HALF && t0 < nkeys) {   // at most 32 keys are left
    arrived();
    tiles(std::integral_constant<int, 1>{}, t0, buf, 0);
  }
  if constexpr (KSP == 2) {
    // the second four waves' results to the first four, which saw the other keys of the same queries
    __syncthreads();
    float* const mine = reinterpret_cast<float*>(prefill_lds) + w4 * (HD / 2 + 2) * 64 + lane;
    if (part) {
#pragma unroll
      for (int d = 0; d < DT; ++d)
#pragma unroll
        for (int v = 0; v < 16; ++v) mine[(d * 16 + v) * 64] = o[d][v];
      mine[(HD / 2) * 64] = m;
      mine[(HD / 2 + 1) * 64] = l;
    }
    __syncthreads();
    if (part) return;
    const float m1 = mine[(HD / 2) * 64], mn = fmaxf(m, m1);
    const float f0 = m == -INFINITY ? 0.0f : exp2_hw((m - mn) * c2), f1 = m1 == -INFINITY ? 0.0f : exp2_hw((m1 - mn) * c2);
    l = l * f0 + mine[(HD / 2 + 1) * 64] * f1;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[d][v] = fmaf(o[d][v], f0, mine[(d * 16 + v) * 64] * f1);
  }
  l += __shfl_xor(l, 32, LR_WAVE);
  if (valid) {
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    const int dy = WIN ? w.dv : HD;
    u16* yrow = y + ((int64_t)b * S + s) * ldy + head * dy;
    // element v of tile d: dimension d * 32 + (v / 4) * 8 + half * 4 + v % 4
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        uint2 w2;
        w2.x = pack_bf2(o[d][4 * g4] * inv, o[d][4 * g4 + 1] * inv);
        w2.y = pack_bf2(o[d][4 * g4 + 2] * inv, o[d][4 * g4 + 3] * inv);
        if (!WIN || d * 32 + g4 * 8 < dy) *reinterpret_cast<uint2*>(yrow + d * 32 + g4 * 8 + half * 4) = w2;
      }
  }
}

template <int HD, int NWH, int KSP, int KEYS, int HALF, bool WIN>
static int launch_prefill_as(unsigned workgroups, const u16* q, int64_t ldq, const u16* kc, const u16* vc, const int32_t* pos, u16* y, int64_t ldy,
                             int S, int Hq, int Hkv, int Smax, const WindowKeys& w, hipStream_t s) {
  constexpr size_t lds = PrefillLds<HD, KSP, KEYS>::BYTES;
  static std::atomic<unsigned long long> raised{0};
  if (!lr_raise_lds_limit(reinterpret_cast<const void*>(&k_attn_prefill_mfma<HD, NWH, KSP, KEYS, HALF, WIN>), lds, raised)) return LR_E_LAUNCH;
  k_attn_prefill_mfma<HD, NWH, KSP, KEYS, HALF, WIN><<<dim3(workgroups), dim3(256 * KSP), lds, s>>>(q, ldq, kc, vc, pos, y, ldy, S, Hq, Hkv, Smax, w);
  return lr_launch_status();
}
template <int HD, int NWH, bool WIN>
static int launch_prefill_heads(const u16* q, int64_t ldq, const u16* kc, const u16* vc, const int32_t* pos, u16* y, int64_t ldy, int B, int S,
                                int Hq, int Hkv, int Smax, const WindowKeys& w, hipStream_t s) {
  constexpr int queries = 32 * (4 / NWH);
  const int64_t n = (int64_t)((S + queries - 1) / queries) * (Hq / NWH) * B;
  const int cus = lr_num_cus();
  const int seen = WIN && w.window < S ? w.window : S;   // keys (at least: how long the history ahead of the queries is only the device knows)
  auto run = &launch_prefill_as<HD, NWH, 1, 64, PREFILL_HALF, WIN>;
  if constexpr (HD == 128) {
    if (n > 2 * cus || (NWH == 2 && S > 32 && S <= 96)) run = &launch_prefill_as<HD, NWH, 1, 32, PREFILL_WHOLE, WIN>;
    else if (S <= 128) run = &launch_prefill_as<HD, NWH, 1, 64, PREFILL_EACH, WIN>;
  } else {
    if (seen > PREFILL_HALF_TO) run = &launch_prefill_as<HD, NWH, 1, 64, PREFILL_WHOLE, WIN>;
  }
  if (n <= cus && seen >= PREFILL_PARTS_FROM) run = &launch_prefill_as<HD, NWH, 2, 64, PREFILL_WHOLE, WIN>;
  return run((unsigned)n, q, ldq, kc, vc, pos, y, ldy, S, Hq, Hkv, Smax, w, s);
}
// NWH heads of a kv head in a workgroup: as many of four as divide its share
template <int HD, bool WIN>
static int launch_prefill_mfma(const u16* q, int64_t ldq, const u16* kc, const u16* vc, const int32_t* pos, u16* y, int64_t ldy, int B, int S,
                               int Hq, int Hkv, int Smax, const WindowKeys& w, hipStream_t s) {
  const int G = Hq / Hkv;
  if (G % 4 == 0) return launch_prefill_heads<HD, 4, WIN>(q, ldq, kc, vc, pos, y, ldy, B, S, Hq, Hkv, Smax, w, s);
  if (G % 2 == 0) return launch_prefill_heads<HD, 2, WIN>(q, ldq, kc, vc, pos, y, ldy, B, S, Hq, Hkv, Smax, w, s);
  return launch_prefill_heads<HD, 1, WIN>(q, ldq, kc, vc, pos, y, ldy, B, S, Hq, Hkv, Smax, w, s);
}

extern "C" int lr_attn_prefill(const void* q, int64_t ldq, const void* k_cache, const void* v_cache,
                               const int32_t* pos, void* y, int64_t ldy, int B, int S, int Hq, int Hkv, int hd,
                               int Smax, lr_stream_t stream) {
  LR_REQUIRE_PTR(q);
  LR_REQUIRE_PTR(k_cache);
  LR_REQUIRE_PTR(v_cache);
  LR_REQUIRE_PTR(y);
  if (pos == nullptr) return LR_E_NULL;
  if (B <= 0 || S <= 0 || Hq <= 0 || Hkv <= 0 || hd <= 0 || Smax <= 0 || Hq % Hkv) return LR_E_SHAPE;
  if (ldq < (int64_t)Hq * hd || ldy < (int64_t)Hq * hd || B > 65535 || Hq > 65535) return LR_E_SHAPE;
  if (ldq % 8 || ldy % 8) return LR_E_ALIGN;
  const dim3 grid((S + 63) / 64, Hq, B);
  hipStream_t s = (hipStream_t)stream;
  if (S >= 16 && Hq <= 65535 * 4) {  // matrix-core kernel; the lane-per-query kernel below serves short inputs
    // (its staging addresses the rows of one (sequence, kv head) with 32-bit byte offsets)
    if ((hd == 128 || hd == 64) && (int64_t)Smax * hd * 2 >= 0x7fffffff) return LR_E_UNSUPPORTED;
    // (and its grid is one-dimensional, at most (S / 32) * Hq * B workgroups of 256 lanes: 2^32 lanes is the limit)
    if ((hd == 128 || hd == 64) && (int64_t)((S + 31) / 32) * Hq * B >= (1 << 24)) return LR_E_UNSUPPORTED;
    if (hd == 128)
      return launch_prefill_mfma<128, false>((const u16*)q, ldq, (const u16*)k_cache, (const u16*)v_cache, pos, (u16*)y, ldy,
                                             B, S, Hq, Hkv, Smax, {}, s);
    if (hd == 64)
      return launch_prefill_mfma<64, false>((const u16*)q, ldq, (const u16*)k_cache, (const u16*)v_cache, pos, (u16*)y, ldy, B,
                                            S, Hq, Hkv, Smax, {}, s);
  }
  if (hd == 128)
    k_attn_prefill<128><<<grid, dim3(64), 0, s>>>((const u16*)q, ldq, (const u16*)k_cache, (const u16*)v_cache, pos,
                                                  (u16*)y, ldy, S, Hq, Hkv, Smax);
  else if (hd == 64)
    k_attn_prefill<64><<<grid, dim3(64), 0, s>>>((const u16*)q, ldq, (const u16*)k_cache, (const u16*)v_cache, pos,
                                                 (u16*)y, ldy, S, Hq, Hkv, Smax);
  else
    return LR_E_UNSUPPORTED;
  return lr_launch_status();
}

// lr_window_attention on the matrix cores (bf16; head sizes up to 128 and multiples of 8, all strides multiples of 8).
namespace lr_detail {
int window_attention_mfma(const lr_window_attention_t* d, lr_stream_t stream) {
  const int hd = d->dk > d->dv ? d->dk : d->dv;
  if (d->dtype != LR_BF16 || hd > 128 || d->dk % 8 || d->dv % 8 || d->ldq % 8 || d->ldk % 8 || d->ldy % 8 ||
      lr_misaligned(d->q) || lr_misaligned(d->k) || lr_misaligned(d->v) || lr_misaligned(d->y) || !(d->scale > 0.0f))
    return LR_E_UNSUPPORTED;
  if ((int64_t)(d->n_keys + 64) * d->ldk * 2 >= 0x7fffffff || (int64_t)((d->S + 31) / 32) * d->H * d->B >= (1 << 24))
    return LR_E_UNSUPPORTED;
  const WindowKeys w = {d->window, d->n_keys, (int)d->ldk, d->dk, d->dv, d->scale};
  const int G = d->kv_heads > 0 ? d->kv_heads : d->H;
  auto run = hd <= 64 ? &launch_prefill_mfma<64, true> : &launch_prefill_mfma<128, true>;
  return run((const u16*)d->q, d->ldq, (const u16*)d->k, (const u16*)d->v, d->pos, (u16*)d->y, d->ldy, d->B, d->S, d->H, G, d->Smax, w,
             (hipStream_t)stream);
}
}  // namespace lr_detail
