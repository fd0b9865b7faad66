// One ladder block of a prompt, from the residual stream and the block before's outputs to its own (lr_ladder_block).
//
// What bounds a short prompt is not one of its kernels: nine launches per block, each with a ramp, a drain and, at 128 rows,
// half of the chip idle, and as many trips from the interpreter (15 us each: 1.25 ms of the 1.40 ms that 16 blocks of the 1B
// model took).  Here a block is one call and four to eight launches: the norms add the partial sums of the outputs that
// come in, q/k/v and up/gate share a grid where that is the faster way (lr_detail::gemm_inputs), and so do wo and w2, whose
// partial sums stay for the next block's norms (lr_detail::gemm_outputs).  us per prompt, replayed from a graph, in one grid /
// q/k/v and up/gate apart / wo and w2 apart: 1B, 64 tokens 900 / 1081 / 1000, 128 tokens 1064 / 1159 / 1130, 256 tokens 1332 /
// 1452 / 1525; 8B, 128 tokens 4568 / 4731 / 4788.  Of the tiles and pieces tried for them, the costs picked the best or one
// within 2 %.
#include "lr_common.h"

namespace lr_detail {   // gemm.hip
int gemm_inputs(const void* x0, const void* wqkv, void* qkv, int S, const lr_rope_kv_t* rope, const void* x1, const void* w1, void* act,
                int I, int M, int K, size_t sums_bytes, hipStream_t s);
int gemm_pieces(const void* x, int64_t ldx, const void* w, int M, int N, int K, void* sums, size_t sums_bytes, int* pieces, hipStream_t s);
bool gemm_outputs_pay(int M, int N, int K0, int K1, size_t sums_bytes);
int gemm_outputs(const void* x0, const void* w0, int K0, void* sums0, int* pieces0, const void* x1, const void* w1, int K1, void* sums1, int* pieces1,
                 int M, int N, size_t sums_bytes, hipStream_t s);
}

extern "C" int lr_ladder_block(lr_ladder_block_t* d, lr_stream_t stream) {
  if (d == nullptr || d->rope.pos == nullptr) return LR_E_NULL;
  LR_REQUIRE_PTR(d->x);
  LR_REQUIRE_PTR(d->xn);
  LR_REQUIRE_PTR(d->xn2);
  LR_REQUIRE_PTR(d->qkv);
  LR_REQUIRE_PTR(d->y);
  LR_REQUIRE_PTR(d->act);
  LR_REQUIRE_PTR(d->h);
  LR_REQUIRE_PTR(d->a);
  LR_REQUIRE_PTR(d->m);
  LR_REQUIRE_PTR(d->gain1);
  LR_REQUIRE_PTR(d->gain2);
  LR_REQUIRE_PTR(d->wqkv);
  LR_REQUIRE_PTR(d->wo);
  LR_REQUIRE_PTR(d->w1);
  LR_REQUIRE_PTR(d->w2);
  LR_REQUIRE_PTR(d->rope.table);
  LR_REQUIRE_PTR(d->rope.k_cache);
  LR_REQUIRE_PTR(d->rope.v_cache);
  LR_OPTIONAL_PTR(d->sums_a);
  LR_OPTIONAL_PTR(d->sums_m);
  const int Hq = d->rope.n_head, Hkv = d->rope.n_kv_head, hd = d->rope.head_dim, D = d->dim, I = d->ffn, S = d->S;
  if (d->B <= 0 || S <= 0 || D <= 0 || I <= 0 || Hq <= 0 || Hkv <= 0 || hd <= 0 || d->rope.smax <= 0 || d->rope.block_size <= 0 || Hq % Hkv)
    return LR_E_SHAPE;
  const int64_t rows64 = (int64_t)d->B * S, nqkv64 = (int64_t)(Hq + 2 * (int64_t)Hkv) * hd;
  if (rows64 > 0x7fffffff || nqkv64 > 0x7fffffff || I > 0x3fffffff) return LR_E_SHAPE;
  if (rows64 < 5) return LR_E_UNSUPPORTED;   // (the activation is the second projection's there)
  if (D % 8 || I % 8 || hd % 8) return LR_E_ALIGN;
  if ((d->a_pieces > 0 || d->m_pieces > 0) && (d->sums_a == nullptr || d->sums_m == nullptr)) return LR_E_NULL;
  for (const int n : {d->a_pieces, d->m_pieces})   // (as many as there is room for)
    if (n > 0 && d->sums_bytes / sizeof(float) / (unsigned)D / (unsigned)n < (size_t)rows64) return LR_E_SHAPE;
  const int rows = (int)rows64, nqkv = (int)nqkv64, Dq = Hq * hd;
  const bool sums = d->sums_a != nullptr && d->sums_m != nullptr;
  const size_t bytes = sums ? d->sums_bytes : 0;
  void* const sa = sums ? d->sums_a : nullptr;
  void* const sm = sums ? d->sums_m : nullptr;
  hipStream_t s = (hipStream_t)stream;

  const void* in_a = d->a_pieces < 0 ? nullptr : (d->a_pieces ? sa : d->a);
  const void* in_m = d->m_pieces < 0 ? nullptr : (d->m_pieces ? sm : d->m);
  int rc = lr_ladder_norms_pieces(d->x, in_a, d->a_pieces > 0 ? d->a_pieces : 0, in_m, d->m_pieces > 0 ? d->m_pieces : 0, d->gain1, d->gain2,
                                  d->x, d->xn, d->xn2, rows, D, d->eps, stream);
  if (rc != LR_OK) return rc;

  const bool keep = sums && !d->finish;
  int out_a = 0, out_m = 0;
  auto attention = [&] {
    return lr_attn_prefill(d->qkv, nqkv, d->rope.k_cache, d->rope.v_cache, d->rope.pos, d->y, Dq, d->B, S, Hq, Hkv, hd, d->rope.smax, stream);
  };
  auto inputs_mlp = [&] {
    return lr_linear_swiglu_out_scratch(d->xn2, D, d->w1, d->act, I, rows, 2 * I, D, d->h, (size_t)rows * 2 * I * sizeof(u16), sm, bytes, stream);
  };
  auto output = [&](const void* x, int K, const void* w, void* y, void* part, int* pieces) {
    const int r = keep ? lr_detail::gemm_pieces(x, K, w, rows, D, K, part, bytes, pieces, s) : LR_E_UNSUPPORTED;
    return r != LR_E_UNSUPPORTED ? r : lr_linear_scratch(x, K, w, y, D, rows, D, K, part, bytes, stream);
  };
  rc = sums ? lr_detail::gemm_inputs(d->xn, d->wqkv, d->qkv, S, &d->rope, d->xn2, d->w1, d->act, I, rows, D, bytes, s) : LR_E_UNSUPPORTED;
  const bool both = rc == LR_OK;
  if (rc == LR_E_UNSUPPORTED) rc = lr_linear_rope_kv_scratch(d->xn, D, d->wqkv, d->qkv, nqkv, rows, D, S, &d->rope, sa, bytes, stream);
  if (rc == LR_OK) rc = attention();
  // wo and w2 in a grid where that is faster; else each behind what it reads
  const bool may_two = keep && lr_detail::gemm_outputs_pay(rows, D, Dq, I, bytes);
  if (rc == LR_OK && !may_two) rc = output(d->y, Dq, d->wo, d->a, sa, &out_a);
  if (rc == LR_OK && !both) rc = inputs_mlp();
  if (rc == LR_OK)
    rc = may_two ? lr_detail::gemm_outputs(d->y, d->wo, Dq, sa, &out_a, d->act, d->w2, I, sm, &out_m, rows, D, bytes, s)
                 : output(d->act, I, d->w2, d->m, sm, &out_m);
  if (rc != LR_OK) return rc;
  d->a_pieces = out_a;
  d->m_pieces = out_m;
  return LR_OK;
}
