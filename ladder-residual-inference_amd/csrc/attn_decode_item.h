#pragma once
#include "lr_common.h"
#include <type_traits>

// ---- how the valid keys are cut into chunks (one workgroup item per chunk, kv head and sequence).
//      A chunk never exceeds ATT_CHUNK keys: the item then requests all of its K and V rows at once.
constexpr int ATT_CHUNK = 256;
constexpr int ATT_NCU = 256;  // CUs of the MI355X
typedef short i16x4_t __attribute__((ext_vector_type(4)));

static inline int attn_nsplit_cap(int Smax) {
  const int by_len = (Smax + ATT_CHUNK - 1) / ATT_CHUNK;
  return by_len > 64 ? by_len : 64;
}

static inline int attn_pick_nsplit(int B, int Hkv, int Smax) {
  const int cap = attn_nsplit_cap(Smax);
  int n = (512 + B * Hkv - 1) / (B * Hkv);   // aim at >= 512 workgroups
  const int by_work = (Smax + 63) / 64;      // but at least ~64 keys per chunk at full length
  if (n > by_work) n = by_work;
  const int by_len = (Smax + ATT_CHUNK - 1) / ATT_CHUNK;
  if (n < by_len) n = by_len;
  if (n < 1) n = 1;
  if (n > cap) n = cap;
  // With more items than CUs the slowest CU sets the time: among the neighbouring chunk counts take the one
  // whose items fill whole rounds of the 256 CUs best (64 sequences: 12 chunks = 768 items instead of 9 = 576).
  // (beyond four rounds the gain is smaller than the cost of more chunks to merge)
  if ((int64_t)n * B * Hkv >= ATT_NCU && (int64_t)n * B * Hkv < 4 * ATT_NCU) {
    int best = n;
    int64_t best_num = 0, best_den = 1;  // padded / real items of the best candidate
    const int lo = n - 3 > by_len ? n - 3 : by_len, hi = n + 3 < cap ? n + 3 : cap;
    for (int c = lo < 1 ? 1 : lo; c <= hi; ++c) {
      const int64_t items = (int64_t)c * B * Hkv, padded = (items + ATT_NCU - 1) / ATT_NCU * ATT_NCU;
      if (best_num == 0 || padded * best_den < best_num * items) { best = c; best_num = padded; best_den = items; }
    }
    n = best;
  }
  return n;
}

// LDS row length of the score buffer: whole 16-key tiles, plus 4 so that the 16 heads a tile's scores are
// written for do not share a bank
__host__ __device__ constexpr int attn_sc_ld(int chunk_max) { return ((chunk_max + 15) & ~15) + 4; }
// and of the softmax weights', in bf16 elements: whole 64-key groups, plus 16 bytes for the same reason
__host__ __device__ constexpr int attn_p_ld(int chunk_max) { return ((chunk_max + 63) & ~63) + 8; }

// What other XCDs are to see or have written: past this XCD's L2 (bit 0 sc0, bit 4 sc1 of a raw buffer operation).
constexpr int ATT_AUX_COHERENT = 17;

// One (split, kv head, sequence) item of the split-KV decode attention, by 256 lanes (4 waves): scores,
// softmax statistics and the un-normalised P.V of keys [k0, k1) (at most 64 GROUPS <= ATT_CHUNK) for all G q heads of
// the kv head.  `smem`: attn_item_lds_floats<HD, G>(chunk_max) floats of LDS.  (A kv head with more q heads than
// an instantiation takes can be served as kv_share groups of G: every head's result is the same either way.)
//
// Bound: memory latency and the instructions behind it.  Every K and V row of the chunk is requested before anything else
// -- whole rows, 1 KiB contiguous per wave instruction, up to 32 KiB per wave in flight, buffer loads whose offset lies
// outside the buffer for what is not wanted (a branch per load makes the compiler wait for everything in flight in the
// middle of the sequence) -- so the item costs one memory round trip.  Scores run on the matrix cores: a 16-key tile of K
// takes a trip through a wave-private piece of LDS (written row-major as loaded, read back as v_mfma_f32_16x16x32_bf16 A
// fragments, rows padded by 16 bytes), the q heads are the B operand (loaded straight into fragment layout, heads beyond G
// are zero columns).  P.V too: V lies in LDS as it came, 64 keys at a time, and is read transposed
// (ds_read_b64_tr_b16) as A fragments, a wave multiplies HD / 4 of the dimensions by all keys, and a softmax weight enters as
// three bf16 summands, which hold all 24 bits of it: the products are those of fp32 weights.
// (P.V on the vector units, lanes owning 8 dimensions of one key in four and the four waves' sums met in LDS, was a thousand
// vector instructions one behind the other, at 4 to 8 cycles each: 6.7 us from the last row's arrival to the stored result for 8
// heads of 65 keys beside a weight stream, now 2.5 us.  64 sequences of the 70B rank shard, ms per step: 7.45 -> 7.05.  The
// chunk results' error against 64 bits is 1.6e-7 of their norm, as it was.)
template <int HD, int G>
__host__ __device__ constexpr int attn_item_lds_floats(int chunk_max) {
  return 32 * (HD + 8) + G * attn_sc_ld(chunk_max) + (3 * G * attn_p_ld(chunk_max) + 1) / 2 + 2 * G + 4;
}
// GROUPS of 64 keys that an item's registers hold: two, or ATT_CHUNK / 64
static inline bool attn_two_groups(int chunk_max) { return chunk_max <= 128; }

// THROUGH: the results are written through to the memory side (sc0 sc1), where attn_merge_wave reads them.
template <int HD, int G, int GROUPS, bool THROUGH = false>
__device__ __forceinline__ void attn_partial_item(const u16* __restrict__ q, int64_t ldq, const u16* __restrict__ kc,
                                                  const u16* __restrict__ vc, const int32_t* __restrict__ pos_ptr,
                                                  float* __restrict__ o_part, float* __restrict__ ml_part, int Hkv,
                                                  int Smax, int nsplit, int chunk_max, int split, int kvh, int b,
                                                  float* __restrict__ smem, int kv_share = 1) {
  static_assert(G <= 16, "the q heads of a kv head are the 16 columns of one matrix-core tile");
  static_assert(GROUPS * 64 <= ATT_CHUNK, "");
  constexpr int LPK = HD / 8;    // lanes that share one key row (8 elements each)
  constexpr int KPW = 64 / LPK;  // keys per wave instruction
  constexpr int NI = 16 / KPW;   // instructions per 16-key tile
  constexpr int KS = HD / 32;    // matrix-core k-steps per row
  constexpr int LROW = HD + 8;   // LDS row length of the K and V pieces, in elements
  constexpr int DT = HD / 64;    // 16-dimension tiles of a wave
  u16* const piece = reinterpret_cast<u16*>(smem);  // [4 waves][16][LROW] of K (during the scores), then [64][LROW] of V
  float* const sc = smem + 32 * LROW;               // [G][ldsc]
  const int ldsc = attn_sc_ld(chunk_max), ldp = attn_p_ld(chunk_max);
  float* const s_m = sc + G * ldsc;                 // [G]
  float* const s_l = s_m + G;                       // [G]
  u16* const sp = reinterpret_cast<u16*>(s_l + G + (4 - 2 * G % 4) % 4);  // [3][G][ldp] the weights' summands

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int Hq = Hkv * G;
  int nkeys = pos_ptr[0] + 1;
  nkeys = nkeys < 0 ? 0 : (nkeys > Smax ? Smax : nkeys);
  const int chunk = (nkeys + nsplit - 1) / nsplit;
  const int k0 = split * chunk;
  const int k1 = k0 + chunk < nkeys ? k0 + chunk : nkeys;
  const int n = k1 - k0;  // <= chunk_max <= 64 GROUPS by construction

  float* o_out = o_part + (((int64_t)b * Hq + kvh * G) * nsplit + split) * HD;  // + g * nsplit * HD
  float* ml_out = ml_part + (((int64_t)b * Hq + kvh * G) * nsplit + split) * 2;  // + g * nsplit * 2
  const __amdgpu_buffer_rsrc_t ores = __builtin_amdgcn_make_buffer_rsrc(o_out, 0, ((G - 1) * nsplit + 1) * HD * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t mres = __builtin_amdgcn_make_buffer_rsrc(ml_out, 0, ((G - 1) * nsplit + 1) * 8, 0x00020000);
  // four consecutive outputs of head g; a head's statistics
  auto put = [&](int g, int d, const f32x4_t& v) {
    const int at = g * nsplit * HD + d;
    if constexpr (THROUGH) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v), ores, at * 4, 0, ATT_AUX_COHERENT);
    else *reinterpret_cast<f32x4_t*>(o_out + at) = v;
  };
  auto put_ml = [&](int g, float m, float l) {
    const f32x2_t v = {m, l};
    if constexpr (THROUGH) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, v), mres, g * nsplit * 8, 0, ATT_AUX_COHERENT);
    else *reinterpret_cast<f32x2_t*>(ml_out + g * nsplit * 2) = v;
  };
  if (n <= 0) {
    for (int i = tid * 4; i < G * HD; i += 1024) put(i / HD, i % HD, f32x4_t{0.0f, 0.0f, 0.0f, 0.0f});
    if (tid < G) put_ml(tid, -INFINITY, 0.0f);
    return;
  }

  const int kl = lane / LPK, dl = (lane % LPK) * 8;
  // kv_share > 1: `Hkv` and `kvh` count groups of G q heads, kv_share of them on one head of the cache
  const u16* kbase = kc + ((int64_t)b * (Hkv / kv_share) + kvh / kv_share) * Smax * HD;
  const u16* vbase = vc + ((int64_t)b * (Hkv / kv_share) + kvh / kv_share) * Smax * HD;
  const float scale = rsqrtf((float)HD);
  // wave w owns the 16-key tiles w, w + 4, ...; instruction i of a tile covers keys i * KPW .. + KPW
  // q as B fragments: column = head lane % 16, k-step ks holds elements ks * 32 + (lane / 16) * 8 .. + 8
  const int l16 = lane & 15, l4 = lane >> 4;
  u32x4_t kr[GROUPS][NI], vr[GROUPS][NI];
  bf16x8_t qf[KS];
  {
    constexpr int OOB_ = (int)0x80000000;
    const __amdgpu_buffer_rsrc_t kres = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(kbase), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t vres = __builtin_amdgcn_make_buffer_rsrc(const_cast<u16*>(vbase), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t qres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<u16*>(q + (int64_t)b * ldq + (int64_t)kvh * G * HD), 0, 0x7fffffff, 0x00020000);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      qf[ks] = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(qres, l16 < G ? (l16 * HD + ks * 32 + l4 * 8) * 2 : OOB_, 0, 0));
    // (non-temporal: a row is read once per step, and what it would push out of the L2 are the inputs of the projection beside it --
    // unless two groups of heads share it.  70B rank shard, us per step: 64 rows 6826 -> 6744, 8 rows 4383 -> 4331, 8B 16 rows 3469 -> 3442)
    auto load = [&](auto AUX) {
      int off[GROUPS][NI];
#pragma unroll
      for (int j = 0; j < GROUPS; ++j)
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int key = k0 + (j * 4 + wave) * 16 + i * KPW + kl;
          off[j][i] = key < k1 ? (key * HD + dl) * 2 : OOB_;
          kr[j][i] = __builtin_amdgcn_raw_buffer_load_b128(kres, off[j][i], 0, decltype(AUX)::value);
        }
#pragma unroll
      for (int j = 0; j < GROUPS; ++j)
#pragma unroll
        for (int i = 0; i < NI; ++i) vr[j][i] = __builtin_amdgcn_raw_buffer_load_b128(vres, off[j][i], 0, decltype(AUX)::value);
    };
    if (kv_share == 1) load(std::integral_constant<int, 2>{});
    else load(std::integral_constant<int, 0>{});
  }

  // ---- scores: S[key][head] = sum_d K[key][d] q[head][d] on the matrix cores
  {
    u16* my = piece + wave * 16 * LROW;
#pragma unroll
    for (int j = 0; j < GROUPS; ++j) {
      const int t16 = (j * 4 + wave) * 16;  // first key of the tile, relative to k0
      if (t16 < n) {  // uniform
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < NI; ++i) *reinterpret_cast<u32x4_t*>(my + (i * KPW + kl) * LROW + dl) = kr[j][i];
        asm volatile("" ::: "memory");
        f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const bf16x8_t af = *reinterpret_cast<const bf16x8_t*>(my + l16 * LROW + ks * 32 + l4 * 8);
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, qf[ks], acc, 0, 0, 0);
        }
        asm volatile("" ::: "memory");
        // accumulator element e: key t16 + 4 (lane / 16) + e, head lane % 16 (keys beyond n: never read)
        if (l16 < G)
          *reinterpret_cast<float4*>(sc + l16 * ldsc + t16 + 4 * l4) =
              make_float4(acc[0] * scale, acc[1] * scale, acc[2] * scale, acc[3] * scale);
      }
    }
  }
  __syncthreads();
  auto store_v = [&](int j) {
#pragma unroll
    for (int i = 0; i < NI; ++i) *reinterpret_cast<u32x4_t*>(piece + (wave * 16 + i * KPW + kl) * LROW + dl) = vr[j][i];
  };
  store_v(0);

  // ---- softmax statistics per head; the weights exp(s - max) as sums of three bf16 numbers, zero from key n on
  for (int g = wave; g < G; g += 4) {
    float v[GROUPS], m = -INFINITY, l = 0.0f;
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
      v[t] = t * 64 + lane < n ? sc[g * ldsc + t * 64 + lane] : -INFINITY;
      m = fmaxf(m, v[t]);
    }
    m = wave_max(m);
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
      if (t * 64 < n) {  // uniform
        const float p = t * 64 + lane < n ? expf(v[t] - m) : 0.0f;
        l += p;
        const float p0 = round_bf(p), p1 = round_bf(p - p0);
        u16* const at = sp + g * ldp + t * 64 + lane;
        at[0] = f_to_bf(p0);
        at[G * ldp] = f_to_bf(p1);
        at[2 * G * ldp] = f_to_bf(p - p0 - p1);
      }
    }
    l = wave_sum(l);
    if (lane == 0) { s_m[g] = m; s_l[g] = l; }
  }
  __syncthreads();

  // ---- P.V: O^T[dim][head] = sum_key V[key][dim] p[head][key]; a wave has DT tiles of 16 dimensions.  Three sums, of the
  // weights' leading parts in even and in odd steps and of what is left of them: few roundings at the size of the result, short chains.
  f32x4_t acc[DT][3];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int c = 0; c < 3; ++c) acc[d][c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  const int ph = l16 < G ? l16 : 0;   // (the columns beyond G are not stored)
#pragma unroll
  for (int j = 0; j < GROUPS; ++j) {
    if (j * 64 < n) {  // uniform
      if (j > 0) {
        __syncthreads();
        store_v(j);
        __syncthreads();
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        bf16x8_t pf[3];
#pragma unroll
        for (int w = 0; w < 3; ++w) pf[w] = *reinterpret_cast<const bf16x8_t*>(sp + (w * G + ph) * ldp + j * 64 + ks * 32 + l4 * 8);
#pragma unroll
        for (int d = 0; d < DT; ++d) {
          // 16 lanes read 4 rows of 16 dimensions, a lane 4 of one row, and receive the 4 keys of one dimension each
          const u16* const at = piece + (ks * 32 + l4 * 8 + (l16 >> 2)) * LROW + wave * (HD / 4) + d * 16 + (l16 & 3) * 4;
          const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(at));
          const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(at + 4 * LROW));
          const bf16x8_t vf = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
          for (int w = 2; w >= 0; --w) {
            f32x4_t& to = acc[d][w ? 2 : ks];
            to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[w], to, 0, 0, 0);
          }
        }
      }
    }
  }
  if (l16 < G) {
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      f32x4_t o = acc[d][1];
#pragma unroll
      for (int e = 0; e < 4; ++e)   // the small ones first (an infinite V: its weight's parts may be zero or negative)
        o[e] = acc[d][0][e] + (fabsf(acc[d][2][e]) < INFINITY ? o[e] + acc[d][2][e] : o[e]);
      put(l16, wave * (HD / 4) + d * 16 + l4 * 4, o);
    }
  }
  if (tid < G) put_ml(tid, s_m[tid], s_l[tid]);
}

// ---- merge of the chunk results: y = sum_s w_s o_s with w_s = exp(m_s - max) / sum_s' exp(m_s' - max) l_s'
template <int HD>
__global__ __launch_bounds__(HD) void k_attn_decode_combine(const float* __restrict__ o_part,
                                                            const float* __restrict__ ml_part, u16* __restrict__ y,
                                                            int64_t ldy, int Hq, int nsplit) {
  const int h = blockIdx.x, b = blockIdx.y, d = threadIdx.x;
  const float* ml = ml_part + ((int64_t)b * Hq + h) * nsplit * 2;
  const float* op = o_part + ((int64_t)b * Hq + h) * nsplit * HD;
  // branch-free loops, unrolled: the loads of eight splits are in flight together instead of one
  // dependent round trip per split
  float M = -INFINITY;
#pragma unroll 8
  for (int s = 0; s < nsplit; ++s) M = fmaxf(M, ml[2 * s]);
  float L = 0.0f, o = 0.0f;
#pragma unroll 8
  for (int s = 0; s < nsplit; ++s) {
    const float m = ml[2 * s];
    const float wgt = m == -INFINITY ? 0.0f : expf(m - M);  // an empty split carries (-inf, 0, 0)
    L = fmaf(wgt, ml[2 * s + 1], L);
    o = fmaf(wgt, op[(int64_t)s * HD + d], o);
  }
  y[(int64_t)b * ldy + h * HD + d] = f_to_bf(L > 0.0f ? o / L : 0.0f);
}

// The same for up to 32 * NB <= 64 splits.  The merge is a chain of memory round trips and little else, so here all of
// it is requested before anything is waited for: lane s of a wave asks for (max, sum) of split s, every lane for
// its element of every partial result (no branch around a load: a split beyond the last reads the last one again
// and gets weight zero).  The weights exp(m_s - max) are formed by the 64 lanes at once and handed round through
// v_readlane: one round trip, where the loop above makes two per eight splits and a scalar load per split.  The
// sums run over the splits in ascending order with the same operations: the results are the same bits.
template <int HD, int NB>
__global__ __launch_bounds__(HD) void k_attn_decode_combine_once(const float* __restrict__ o_part,
                                                                 const float* __restrict__ ml_part,
                                                                 u16* __restrict__ y, int64_t ldy, int Hq, int nsplit) {
  constexpr int NS = 32 * NB;
  const int h = blockIdx.x, b = blockIdx.y, d = threadIdx.x, lane = d & 63;
  const float* ml = ml_part + ((int64_t)b * Hq + h) * nsplit * 2;
  const float* op = o_part + ((int64_t)b * Hq + h) * nsplit * HD;
  const int sl = lane < nsplit ? lane : nsplit - 1;
  const float2 mlv = *reinterpret_cast<const float2*>(ml + 2 * sl);
  float ov[NS];
#pragma unroll
  for (int j = 0; j < NS; ++j) ov[j] = op[(int64_t)(j < nsplit ? j : nsplit - 1) * HD + d];
  const float M = wave_max(mlv.x);  // (lanes beyond the last split repeat it: the maximum is the same)
  const float w_lane = (lane >= nsplit || mlv.x == -INFINITY) ? 0.0f : expf(mlv.x - M);  // an empty split: (-inf, 0, 0)
  float L = 0.0f, o = 0.0f;
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const float wgt = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w_lane), j));
    const float lj = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mlv.y), j));
    if (j < nsplit) {  // uniform (a sum must not see the -0.0 + 0.0 of a padded split)
      L = fmaf(wgt, lj, L);
      o = fmaf(wgt, ov[j], o);
    }
  }
  y[(int64_t)b * ldy + h * HD + d] = f_to_bf(L > 0.0f ? o / L : 0.0f);
}

// The same inside the launch of the items, by waves of workgroups that stand behind them in the grid.  An item counts its
// kv head's chunks up when the memory side has acknowledged its results (attn_item_done), and a wave reads them from there
// (sc0 sc1): 64 outputs, all of up to 64 chunks' in one round trip.
//
// A wave waits for the chunks, an item for nobody.  Workgroups are dealt to the XCDs in turn and every XCD starts its own in
// order: a wave that runs has seen the items of its XCD start, those of another may still stand behind a projection's workgroups there,
// or behind the waiting waves of a second grid whose items stand behind this one's.  So a wave that has looked ATT_MERGE_LOOKS times
// (about a millisecond, where 20 us are usual) hands its part over and ends; the item that stores the last chunk merges what was handed over.  One
// word decides which of the two it is, whatever the order: bits 0 to 7 chunks stored, 8 to 15 parts merged, 16 to 31 parts handed
// over.  A wave that sets its bit sees in the same operation whether all chunks are there -- then the last item has gone by, and
// the part is still its own; the last item sees in its own the bits set before it.  Whoever merges a kv head's last part sets the word to zero: nobody
// looks at it any more.
constexpr int ATT_MERGE_MAX = 64;   // chunks
constexpr int ATT_TICKET = 32;      // words from one kv head's to the next: 128 bytes
constexpr u32 ATT_MERGE_LOOKS = 512;
// the other words of a kv head's: [1] n > 0: n - 1 looks instead; [2] parts handed over so far
__device__ __forceinline__ u32 attn_look(u32* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// one lane adds; the value before, in every lane
__device__ __forceinline__ u32 attn_count(u32* p, u32 n) {
  u32 was = 0;
  if ((threadIdx.x & 63) == 0) was = __hip_atomic_fetch_add(p, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return __builtin_amdgcn_readfirstlane(was);
}

// `part`: which 64 of the outputs [B][Hq * HD].  A merge in a launch of its own is 4.7 us per block
// and step; here it ends before the weight stream does (70B rank shard, 8 rows: chunks stored at 6 us of 23, merged at 20).
// What did not do: all of a head's outputs by whoever stores its last chunk (131 KB of 32 chunks through one CU beside its part of the
// stream: the launch 2.5 us longer); tickets in one cache line, polled without a pause (the polls queue before the items' counts: e4m3,
// 5 rows, the whole stream 12 -> 17 us).
template <int HD>
__device__ __forceinline__ void attn_merge_part(const float* __restrict__ o_part, const float* __restrict__ ml_part, u16* __restrict__ y, int64_t ldy,
                                                int Hq, int nsplit, int part) {
  const int lane = threadIdx.x & 63;
  const int head = part / (HD / 64), b = head / Hq, h = head - b * Hq, d = part % (HD / 64) * 64 + lane;   // (head: of all sequences)
  const __amdgpu_buffer_rsrc_t ores = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(o_part + (int64_t)head * nsplit * HD), 0, nsplit * HD * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t mres = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(ml_part + (int64_t)head * nsplit * 2), 0, nsplit * 8, 0x00020000);
  // (a chunk beyond the last lies outside the resource and reads as zero)
  const u32x2_t mlv = __builtin_amdgcn_raw_buffer_load_b64(mres, lane * 8, 0, ATT_AUX_COHERENT);
  constexpr int NB = 32;
  float ov[NB], o = 0.0f, L = 0.0f, w_lane = 0.0f, l_lane = 0.0f;
  for (int s0 = 0; s0 < nsplit; s0 += NB) {
#pragma unroll
    for (int j = 0; j < NB; ++j) ov[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ores, ((s0 + j) * HD + d) * 4, 0, ATT_AUX_COHERENT));
    if (s0 == 0) {
      const float ms = lane < nsplit ? __uint_as_float(mlv.x) : -INFINITY;
      l_lane = __uint_as_float(mlv.y);
      const float M = wave_max(ms);
      w_lane = ms == -INFINITY ? 0.0f : expf(ms - M);  // an empty chunk: (-inf, 0, 0)
    }
#pragma unroll
    for (int j = 0; j < NB; ++j)
      if (s0 + j < nsplit) {  // uniform
        const float wgt = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w_lane), s0 + j));
        L = fmaf(wgt, __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(l_lane), s0 + j)), L);
        o = fmaf(wgt, ov[j], o);
      }
  }
  y[(int64_t)b * ldy + h * HD + d] = f_to_bf(L > 0.0f ? o / L : 0.0f);
}
template <int HD, int G>
__device__ __forceinline__ void attn_merged(u32* ticket, u32 parts) {
  if ((attn_count(ticket, parts << 8) >> 8 & 255) + parts == G * (HD / 64) && (threadIdx.x & 63) == 0)
    __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <int HD, int G>
__device__ __forceinline__ void attn_merge_wave(const float* __restrict__ o_part, const float* __restrict__ ml_part, u32* tickets, u16* __restrict__ y,
                                                int64_t ldy, int Hkv, int nsplit, int part) {
  constexpr int PARTS = G * (HD / 64);
  static_assert(PARTS <= 16 && ATT_MERGE_MAX < 256, "fields of a ticket");
  u32* const ticket = tickets + part / PARTS * ATT_TICKET;
  const u32 limit = attn_look(ticket + 1), looks = limit ? limit - 1 : ATT_MERGE_LOOKS;
  u32 seen = attn_look(ticket);
  for (u32 i = 0; (seen & 255) < (u32)nsplit && i < looks; ++i) {
    __builtin_amdgcn_s_sleep(40);
    seen = attn_look(ticket);
  }
  if ((seen & 255) < (u32)nsplit) {
    if ((threadIdx.x & 63) == 0) seen = __hip_atomic_fetch_or(ticket, 1u << (16 + part % PARTS), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((__builtin_amdgcn_readfirstlane(seen) & 255) < (u32)nsplit) {
      attn_count(ticket + 2, 1);
      return;
    }
  }
  asm volatile("" ::: "memory");
  attn_merge_part<HD>(o_part, ml_part, y, ldy, Hkv * G, nsplit, part);
  attn_merged<HD, G>(ticket, 1);
}
// The end of an item of kv head `group` of all sequences'.
template <int HD, int G>
__device__ __forceinline__ void attn_item_done(const float* __restrict__ o_part, const float* __restrict__ ml_part, u32* tickets, u16* __restrict__ y,
                                               int64_t ldy, int Hkv, int nsplit, int group) {
  constexpr int PARTS = G * (HD / 64);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x >= 64) return;
  u32* const ticket = tickets + group * ATT_TICKET;
  const u32 was = attn_count(ticket, 1), handed = was >> 16;
  if ((was & 255) + 1 < (u32)nsplit || handed == 0) return;
  asm volatile("" ::: "memory");
  for (int i = 0; i < PARTS; ++i)
    if (handed >> i & 1) attn_merge_part<HD>(o_part, ml_part, y, ldy, Hkv * G, nsplit, group * PARTS + i);
  attn_merged<HD, G>(ticket, __builtin_popcount(handed));
}

template <int HD>
static inline void launch_attn_combine(const float* o_part, const float* ml_part, u16* y, int64_t ldy, int Hq, int B,
                                       int nsplit, hipStream_t s) {
  if (nsplit <= 32) k_attn_decode_combine_once<HD, 1><<<dim3(Hq, B), dim3(HD), 0, s>>>(o_part, ml_part, y, ldy, Hq, nsplit);
  else if (nsplit <= 64) k_attn_decode_combine_once<HD, 2><<<dim3(Hq, B), dim3(HD), 0, s>>>(o_part, ml_part, y, ldy, Hq, nsplit);
  else k_attn_decode_combine<HD><<<dim3(Hq, B), dim3(HD), 0, s>>>(o_part, ml_part, y, ldy, Hq, nsplit);
}

// ---- the items, and the waves that merge them, as the workgroups of a grid that holds a projection too (decode_pair.hip, gemm.hip)
struct AttnItems {
  const u16* q;
  int64_t ldq;
  const u16* kc;
  const u16* vc;
  const int32_t* pos;
  float* o_part;
  float* ml_part;
  int Hkv, Smax, nsplit, chunk_max;  // Hkv: groups of G q heads (kv_share of them per head of the cache)
  int kv_share;
  int n_items;  // nsplit * Hkv * B workgroups
  // with tickets: the chunks are merged into y by workgroups of their own
  u32* tickets;  // [B * Hkv * ATT_TICKET], zero
  u16* y;
  int64_t ldy;
  int merge_waves, waves_per_wg;  // of 64 outputs; of them in a workgroup

  int mergers() const { return tickets ? (merge_waves + waves_per_wg - 1) / waves_per_wg : 0; }
};
// item `wg` of n_items; merging workgroup `wg` of mergers(), behind all items in the grid
template <int HD, int G, int GROUPS, bool MERGE>
__device__ __forceinline__ void attn_item(const AttnItems& a, int wg, float* smem) {
  const int split = wg % a.nsplit, rest = wg / a.nsplit;
  attn_partial_item<HD, G, GROUPS, MERGE>(a.q, a.ldq, a.kc, a.vc, a.pos, a.o_part, a.ml_part, a.Hkv, a.Smax, a.nsplit,
                                          a.chunk_max, split, rest % a.Hkv, rest / a.Hkv, smem, a.kv_share);
  if constexpr (MERGE) attn_item_done<HD, G>(a.o_part, a.ml_part, a.tickets, a.y, a.ldy, a.Hkv, a.nsplit, rest);
}
template <int HD, int G>
__device__ __forceinline__ void attn_merge(const AttnItems& a, int wg) {
  const int wave = threadIdx.x >> 6, m = wg * a.waves_per_wg + wave;
  if (wave < a.waves_per_wg && m < a.merge_waves)
    attn_merge_wave<HD, G>(a.o_part, a.ml_part, a.tickets, a.y, a.ldy, a.Hkv, a.nsplit, __builtin_amdgcn_readfirstlane(m));
}
// Checks lr_attn_decode's arguments and fills `a`; G: q heads of an item.
static inline int attn_fill_items(const void* q, int64_t ldq, const void* k_cache, const void* v_cache, const int32_t* pos, void* y, int64_t ldy,
                                  int B, int Hq, int Hkv, int hd, int Smax, void* scratch, size_t scratch_bytes, void* tickets, AttnItems& a,
                                  int& G) {
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
  if (((uintptr_t)tickets & 3) != 0) return LR_E_ALIGN;
  a = AttnItems{};
  G = Hq / Hkv;
  a.kv_share = 1;
  a.q = (const u16*)q; a.ldq = ldq; a.kc = (const u16*)k_cache; a.vc = (const u16*)v_cache; a.pos = pos;
  a.Smax = Smax;
  a.nsplit = attn_pick_nsplit(B, Hkv, Smax);  // the chunks of lr_attn_decode
  if (G == 16) {
    // 16 q heads per kv head need the whole register file (one workgroup per CU): two groups of 8 instead
    G = 8;
    a.kv_share = 2;
  }
  a.Hkv = Hkv * a.kv_share;
  a.chunk_max = ((Smax + a.nsplit - 1) / a.nsplit + 3) & ~3;
  a.o_part = (float*)scratch;
  a.ml_part = a.o_part + (size_t)B * Hq * a.nsplit * hd;
  if ((int64_t)a.nsplit * a.Hkv * B > 0x3fffffff) return LR_E_UNSUPPORTED;
  a.n_items = a.nsplit * a.Hkv * B;
  a.y = (u16*)y; a.ldy = ldy;
  a.tickets = a.nsplit <= ATT_MERGE_MAX ? (u32*)tickets : nullptr;   // (more chunks: a launch of their own)
  if (!((hd == 128 || hd == 64) && (G == 1 || G == 2 || G == 4 || G == 8))) return LR_E_UNSUPPORTED;
  a.merge_waves = B * Hq * (hd / 64);
  a.waves_per_wg = a.merge_waves > 2 * ATT_NCU ? 4 : a.merge_waves > ATT_NCU ? 2 : 1;   // (spread over the CUs, whose parts of a projection are to end together)
  return LR_OK;
}
