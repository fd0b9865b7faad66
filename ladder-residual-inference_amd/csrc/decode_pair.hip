// Decode attention and one weight-streaming projection in ONE launch.
//
// In a ladder block the MLP's input does not contain the block's own attention output, so the
// attention over the KV cache and the up/gate projection of the same block are independent.  The
// attention of a decode step is a latency chain (a few hundred workgroups that each wait for one
// memory round trip and then do a little arithmetic); the projection is pure streaming.  Launched
// one after the other, the chip idles through the first and the second cannot start; launched as
// one grid -- the first workgroups are attention items, the rest are bands of the projection --
// two workgroups share a CU and the attention disappears behind the weight stream.
//
// Both halves are the device functions their own kernels use (attn_partial_item, stream_band), so
// the results are bit-identical to lr_attn_decode followed by lr_linear_multi.  With a ticket per kv head
// the chunks are merged here too, by workgroups at the end of the grid (attn_merge_wave), also beside the
// weight stream; without, in a launch of their own.
//
// lr_attn_decode_beside_fp8: the same grid with the e4m3 variant of the band (weight-only quantised models,
// 2 to 16 rows).
#include "attn_decode_item.h"
#include "stream_band.h"

namespace {

constexpr int PAIR_MT = 16, PAIR_UNITS = 2;

// X8: at most 8 input rows in fragment layout, requested as far ahead as the weights (see stream_band)
// GROUPS: keys of an attention item, in 64s (see attn_partial_item)
template <int HD, int G, bool W8, bool XL, int GROUPS, bool X8, bool MERGE>
__global__ __launch_bounds__(256, XL ? 0 : 2) void k_attn_beside_band(const AttnItems a, const Proj p, const int M) {
  extern __shared__ __attribute__((aligned(16))) unsigned char pair_smem[];
  const int wg = blockIdx.x;
  if (wg < a.n_items) {
    attn_item<HD, G, GROUPS, MERGE>(a, wg, reinterpret_cast<float*>(pair_smem));
  } else if (MERGE && wg >= a.n_items + p.nwg) {
    attn_merge<HD, G>(a, wg - a.n_items - p.nwg);
  } else {
    stream_band<PAIR_MT, PAIR_UNITS, W8, XL, false, RESID_NONE, NWV, 16, X8, X8>(p, M, wg - a.n_items, reinterpret_cast<u16*>(pair_smem));
  }
}

template <int HD, int G, bool W8, bool XL, int GROUPS, bool X8, bool MERGE>
static int launch_pair_merge(const AttnItems& a, const Proj& p, int M, int B, hipStream_t s) {
  const size_t lds_att = (size_t)attn_item_lds_floats<HD, G>(a.chunk_max) * sizeof(float);
  const size_t lds_band = stream_band_lds_bytes<PAIR_MT, PAIR_UNITS, W8, XL>() + stream_band_norm_bytes(p, M);
  const size_t lds = lds_att > lds_band ? lds_att : lds_band;
  static std::atomic<unsigned long long> lds_raised{0};
  if (!lr_raise_lds_limit(reinterpret_cast<const void*>(&k_attn_beside_band<HD, G, W8, XL, GROUPS, X8, MERGE>), lds, lds_raised)) return LR_E_LAUNCH;
  k_attn_beside_band<HD, G, W8, XL, GROUPS, X8, MERGE><<<dim3((unsigned)(a.n_items + p.nwg + a.mergers())), dim3(256), lds, s>>>(a, p, M);
  if (!MERGE) launch_attn_combine<HD>(a.o_part, a.ml_part, a.y, a.ldy, a.Hkv * G, B, a.nsplit, s);
  return lr_launch_status();
}
template <int HD, int G, bool W8, bool XL, int GROUPS, bool X8 = !W8 && !XL>
static int launch_pair_as(const AttnItems& a, const Proj& p, int M, int B, hipStream_t s) {
  return a.tickets ? launch_pair_merge<HD, G, W8, XL, GROUPS, X8, true>(a, p, M, B, s)
                   : launch_pair_merge<HD, G, W8, XL, GROUPS, X8, false>(a, p, M, B, s);
}

// (the band's inputs in whole lines or in fragment layout: the choice lr_linear_multi makes for the same rows)
template <int HD, int G, bool W8>
static int launch_pair(const AttnItems& a, const Proj& p, int M, int B, hipStream_t s) {
  const bool two = attn_two_groups(a.chunk_max);
  if (!W8 && M >= XLDS_M16_FROM)
    return two ? launch_pair_as<HD, G, false, true, 2>(a, p, M, B, s)
               : launch_pair_as<HD, G, false, true, 4>(a, p, M, B, s);
  if (W8 && M <= 8)
    return two ? launch_pair_as<HD, G, W8, false, 2, true>(a, p, M, B, s)
               : launch_pair_as<HD, G, W8, false, 4, true>(a, p, M, B, s);
  return two ? launch_pair_as<HD, G, W8, false, 2>(a, p, M, B, s)
             : launch_pair_as<HD, G, W8, false, 4>(a, p, M, B, s);
}

// shared body of the two entry points; `fill` turns the caller's projection into a Proj
template <bool W8, class Projection, class Fill>
static int beside(const void* q, int64_t ldq, const void* k_cache, const void* v_cache, const int32_t* pos, void* y,
                  int64_t ldy, int B, int Hq, int Hkv, int hd, int Smax, void* scratch, size_t scratch_bytes,
                  const Projection* proj, const lr_row_norm_t* norm, void* tickets, int M, int m_min, lr_stream_t stream,
                  Fill fill) {
  AttnItems a;
  int G;
  const int arc = attn_fill_items(q, ldq, k_cache, v_cache, pos, y, ldy, B, Hq, Hkv, hd, Smax, scratch, scratch_bytes, tickets, a, G);
  if (arc != LR_OK && arc != LR_E_UNSUPPORTED) return arc;
  if (proj == nullptr) return LR_E_NULL;
  if (M < 1) return LR_E_SHAPE;
  if (arc != LR_OK) return arc;
  // the projection must not touch the cache the attention reads, and only the 16-row band shares a CU
  if (proj->epilogue == LR_EPI_ROPE_KV || M > PAIR_MT || M < m_min) return LR_E_UNSUPPORTED;
  Proj p;
  int rc = fill(*proj, p);
  if (rc == LR_OK) rc = sb_fill_norm(norm, p);
  if (rc != LR_OK) return rc;
  const int ncu = lr_num_cus();
  if (ncu < 1) return LR_E_LAUNCH;
  plan(p, M, p.pair_off ? 16 : 16 * PAIR_UNITS, ncu);
  if (p.fold_sums && p.nwg < M) return LR_E_UNSUPPORTED;   // (a row per workgroup)
  hipStream_t s = (hipStream_t)stream;
#define LR_PAIR(HDV, GV) \
  if (hd == HDV && G == GV) return launch_pair<HDV, GV, W8>(a, p, M, B, s);
  LR_PAIR(128, 1) LR_PAIR(128, 2) LR_PAIR(128, 4) LR_PAIR(128, 8)
  LR_PAIR(64, 1) LR_PAIR(64, 2) LR_PAIR(64, 4) LR_PAIR(64, 8)
#undef LR_PAIR
  return LR_E_UNSUPPORTED;
}

}  // namespace

extern "C" int lr_attn_decode_beside_merged(const void* q, int64_t ldq, const void* k_cache, const void* v_cache,
                                            const int32_t* pos, void* y, int64_t ldy, int B, int Hq, int Hkv, int hd,
                                            int Smax, void* scratch, size_t scratch_bytes, const lr_projection_t* proj,
                                            const lr_row_norm_t* norm, void* tickets, int M, lr_stream_t stream) {
  return beside<false>(q, ldq, k_cache, v_cache, pos, y, ldy, B, Hq, Hkv, hd, Smax, scratch, scratch_bytes, proj, norm, tickets, M, 1,
                       stream, sb_fill_projection);
}

extern "C" int lr_attn_decode_beside_normed(const void* q, int64_t ldq, const void* k_cache, const void* v_cache,
                                            const int32_t* pos, void* y, int64_t ldy, int B, int Hq, int Hkv, int hd,
                                            int Smax, void* scratch, size_t scratch_bytes, const lr_projection_t* proj,
                                            const lr_row_norm_t* norm, int M, lr_stream_t stream) {
  return lr_attn_decode_beside_merged(q, ldq, k_cache, v_cache, pos, y, ldy, B, Hq, Hkv, hd, Smax, scratch, scratch_bytes, proj,
                                      norm, nullptr, M, stream);
}

extern "C" int lr_attn_decode_beside(const void* q, int64_t ldq, const void* k_cache, const void* v_cache,
                                     const int32_t* pos, void* y, int64_t ldy, int B, int Hq, int Hkv, int hd,
                                     int Smax, void* scratch, size_t scratch_bytes, const lr_projection_t* proj,
                                     int M, lr_stream_t stream) {
  return lr_attn_decode_beside_merged(q, ldq, k_cache, v_cache, pos, y, ldy, B, Hq, Hkv, hd, Smax, scratch, scratch_bytes, proj,
                                      nullptr, nullptr, M, stream);
}

// (for one row lr_linear_fp8_multi uses the matrix-vector kernel, which has no band to put beside the attention)
extern "C" int lr_attn_decode_beside_fp8_merged(const void* q, int64_t ldq, const void* k_cache, const void* v_cache,
                                                const int32_t* pos, void* y, int64_t ldy, int B, int Hq, int Hkv, int hd,
                                                int Smax, void* scratch, size_t scratch_bytes,
                                                const lr_projection_fp8_t* proj, const lr_row_norm_t* norm, void* tickets,
                                                int M, lr_stream_t stream) {
  return beside<true>(q, ldq, k_cache, v_cache, pos, y, ldy, B, Hq, Hkv, hd, Smax, scratch, scratch_bytes, proj, norm, tickets, M,
                      LR_FP8_GEMV_MAX_M + 1, stream, sb_fill_projection_fp8);
}

extern "C" int lr_attn_decode_beside_fp8_normed(const void* q, int64_t ldq, const void* k_cache, const void* v_cache,
                                                const int32_t* pos, void* y, int64_t ldy, int B, int Hq, int Hkv, int hd,
                                                int Smax, void* scratch, size_t scratch_bytes,
                                                const lr_projection_fp8_t* proj, const lr_row_norm_t* norm, int M,
                                                lr_stream_t stream) {
  return lr_attn_decode_beside_fp8_merged(q, ldq, k_cache, v_cache, pos, y, ldy, B, Hq, Hkv, hd, Smax, scratch, scratch_bytes, proj,
                                          norm, nullptr, M, stream);
}

extern "C" int lr_attn_decode_beside_fp8(const void* q, int64_t ldq, const void* k_cache, const void* v_cache,
                                         const int32_t* pos, void* y, int64_t ldy, int B, int Hq, int Hkv, int hd,
                                         int Smax, void* scratch, size_t scratch_bytes,
                                         const lr_projection_fp8_t* proj, int M, lr_stream_t stream) {
  return lr_attn_decode_beside_fp8_merged(q, ldq, k_cache, v_cache, pos, y, ldy, B, Hq, Hkv, hd, Smax, scratch, scratch_bytes, proj,
                                          nullptr, nullptr, M, stream);
}
