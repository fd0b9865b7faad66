// Matrix-core bf16 GEMMs for prefill, decode batches above 64 rows, and from 33 rows on where there is memory for partial sums
// (from 17 in the grids that a decode step's blocks share, lr_attn_decode_beside_product and lr_linear_pieces_two):
//   y[m, n] = bf16( sum_k x[m, k] * w[n, k] ),  fp32 accumulation.
// k_gemm_dma (below) is the one that matters; k_gemm here serves an input that is activated on its way in, and rows longer
// than the 2 GiB offsets of k_gemm_dma's requests reach.
//
// k_gemm: v_mfma_f32_32x32x16_bf16, workgroup tile 128 x 128 x 64, four waves in a 2 x 2 arrangement, each wave owning a 64 x 64
// block = 2 x 2 MFMA tiles (64 accumulator VGPRs).  Both operands are K-contiguous in memory, so
// the same staging path serves them: 128-bit global loads -> registers -> LDS rows padded by 16
// bytes (stride 144 B keeps ds_read_b128 of 16 consecutive rows on distinct banks) -> 128-bit LDS
// reads that deliver exactly the 8 consecutive k an MFMA lane feeds.  LDS is double-buffered and
// the global loads of tile t+1 are in flight while tile t is multiplied.
#include "attn_decode_item.h"
#include "lr_common.h"
#include <type_traits>

int lr_gemv_dispatch(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K,
                     int act_swiglu, int gemv_cfg, hipStream_t s);

namespace lr_detail {
int swiglu_rows(const void* h, int64_t ldh, void* out, int64_t ldo, int rows, int I, lr_stream_t stream);   // elementwise.hip
}

constexpr int BM = 128, BN = 128, BK = 64, LDT = BK + 8;  // LDT: padded LDS row length in elements

template <bool SWIGLU>
__device__ __forceinline__ uint4 load_x_chunk(const u16* __restrict__ x, int64_t ldx, int M, int K, int m, int k) {
  if (m >= M || k >= K) return make_uint4(0, 0, 0, 0);
  if (SWIGLU) {
    float u[8], g[8], o[8];
    unpack8(ld16(x + (int64_t)m * ldx + k), u);
    unpack8(ld16(x + (int64_t)m * ldx + K + k), g);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = swiglu_bf(u[j], g[j]);
    return pack8(o);
  }
  return ld16(x + (int64_t)m * ldx + k);
}

__device__ __forceinline__ uint4 load_w_chunk(const u16* __restrict__ w, int N, int K, int n, int k) {
  if (n >= N || k >= K) return make_uint4(0, 0, 0, 0);
  return ld16(w + (int64_t)n * K + k);
}

template <bool SWIGLU>
__global__ __launch_bounds__(256) void k_gemm(const u16* __restrict__ x, int64_t ldx, const u16* __restrict__ w,
                                              u16* __restrict__ y, int64_t ldy, int M, int N, int K) {
  __shared__ __attribute__((aligned(16))) u16 xs[2][BM * LDT];
  __shared__ __attribute__((aligned(16))) u16 ws[2][BN * LDT];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;

  // staging assignment: 1024 16-byte chunks per operand tile, 4 per thread
  int srow[4], scol[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int id = tid + i * 256;
    srow[i] = id >> 3;
    scol[i] = (id & 7) * 8;
  }

  f32x16_t acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;

  uint4 xr[4], wr[4];
  const int nk = (K + BK - 1) / BK;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    xr[i] = load_x_chunk<SWIGLU>(x, ldx, M, K, m0 + srow[i], scol[i]);
    wr[i] = load_w_chunk(w, N, K, n0 + srow[i], scol[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    st16(&xs[0][srow[i] * LDT + scol[i]], xr[i]);
    st16(&ws[0][srow[i] * LDT + scol[i]], wr[i]);
  }
  __syncthreads();

  const int arow = lane & 31, akq = (lane >> 5) * 8;
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) {
      const int k0 = (kt + 1) * BK;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        xr[i] = load_x_chunk<SWIGLU>(x, ldx, M, K, m0 + srow[i], k0 + scol[i]);
        wr[i] = load_w_chunk(w, N, K, n0 + srow[i], k0 + scol[i]);
      }
    }
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
      bf16x8_t af[2], bfr[2];
#pragma unroll
      for (int a = 0; a < 2; ++a)
        af[a] = *reinterpret_cast<const bf16x8_t*>(&xs[cur][(wm * 64 + a * 32 + arow) * LDT + kk + akq]);
#pragma unroll
      for (int b = 0; b < 2; ++b)
        bfr[b] = *reinterpret_cast<const bf16x8_t*>(&ws[cur][(wn * 64 + b * 32 + arow) * LDT + kk + akq]);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[a], bfr[b], acc[a][b], 0, 0, 0);
    }
    if (kt + 1 < nk) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        st16(&xs[cur ^ 1][srow[i] * LDT + scol[i]], xr[i]);
        st16(&ws[cur ^ 1][srow[i] * LDT + scol[i]], wr[i]);
      }
    }
    __syncthreads();
  }

  // accumulator element v of a 32x32 tile: row = (v / 4) * 8 + (lane / 32) * 4 + v % 4, col = lane % 32
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int n = n0 + wn * 64 + b * 32 + (lane & 31);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = m0 + wm * 64 + a * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
        if (m < M && n < N) y[(int64_t)m * ldy + n] = f_to_bf(acc[a][b][v]);
      }
    }
}

// ---------------------------------------------------------------------------------------------
// The GEMM of prompts and of decode batches above 32.  A workgroup of four waves (2 x 2) multiplies a tile of 32 A input
// rows x 128 BH weight rows: 160 to 256 rows in steps of 32, or 128, by 256; 64, 128, 160 or 192 by 128 (gemm_plan picks).  Bound: the matrix cores, at the
// clock the chip's power allows, from a few hundred rows on (16384 x 4096 x 14336, one counter run: 1302 us = 1.48 PFLOP/s,
// matrix cores busy 79 % of the cycles at 1.78 GHz); the weights' HBM traffic below.
//
// Operands go from memory to LDS directly (buffer_load ... lds, 16 bytes per lane, 8 rows x 64 k per instruction): no
// registers, no LDS write instructions.  An instruction fills 1 KiB of LDS in lane order, so rows cannot be padded; the
// sixteen-byte groups of a row are exchanged instead (group g of row r lies at g ^ (r & 7)), by the address a lane loads
// from and again by the address a fragment is read at: conflict-free for the 16-row fragments of
// v_mfma_f32_16x16x32_bf16.
//
// What a tile of fewer rows costs is what a CU draws, about 65 GB/s while part of it comes from HBM (from L2 alone 127): (m + n) * 128 bytes per k-tile, 1.0 us at 256 x 256 where the
// matrix cores need 1.1 to 1.2, 0.5 at 128 x 128 where they need 0.3.  So tiles from 160 rows on are as good per row as the largest, and rows
// that are no multiple of 256 want them: 777 rows are four tiles of 224 (measured below, at GEMM_TILES).
//
// A k-tile is 64 elements; its operand rows come in two halves each (A: input rows, B: weight rows; the first half of the input
// rows has a group of 16 per wave more where A is odd) and the tile's four
// quarter products follow one another in four phases, (A0 B0) (A0 B1) (A1 B1) (A1 B0).  Every phase reads ONE half from
// LDS into registers for a later phase and requests the half of two k-tiles ahead into the LDS slot that the phase before
// it emptied: a request has seven phases to land, a slot is read in exactly one phase, and one barrier per phase orders
// both.  The reads and requests stand between the matrix instructions, one at a time, and every request is made whatever
// the tile (a k-tile past the end is a resource of no records: zeros, no traffic), so the waits are exact.  (They count the
// youngest requests: memory operations that a compiler put between them, a spill's, would make them wait for more, not less.
// There are none in any instance's loop.)  The next
// k-tile's A0 and B0 take the registers that A0 and B1 leave, so B0 and B1 change registers from one k-tile to the next:
// the loop walks two.
//
// Before (128 x 128 wave tiles of v_mfma_f32_32x32x16_bf16, operands staged through registers and padded LDS rows):
// 16384 rows x (N x K), us before / now: 6144 x 4096 646 / 560, 4096 x 4096 428 / 381, 28672 x 4096 with SwiGLU 3112 /
// 2755, 4096 x 14336 1462 / 1281 (from machine to machine 2750 - 2870 and 1275 - 1315).  The same loop on 32x32x16
// instructions took 1337 us for the last: twice the accumulator traffic per product, at a power-limited clock.  The matrix
// instruction is assembler text because its accumulator has to be one register block in and out: left to the compiler,
// 180 accumulator moves per two k-tiles (1.15 PFLOP/s).
//
// A ring of three k-tiles, for up to 64 rows and, as a tile of its own (GEMM_LONG), 128 x 128 of up to 128: what bounds these is the
// weights' way from HBM, and a CU has at most some 48 KiB of requests on their way whoever waits for them, so a ring of two, of
// which a k-tile and a half are, asks for too little; four are no faster (7168 x 8192, 64 rows, four pieces: two 31.0 us, three 27.4,
// four 27.6).  And all workgroups walk K from the same end, over rows that lie a multiple of 4 KiB apart: at any time they ask for
// one place of the DRAM's interleaving.  With a long ring column tile nt begins at k-tile GEMM_TURN * nt and goes round (a stream of such
// operands without products, 128 rows, 7168 x 8192: ring of two 33.3 us, turned 30.9, ring of four 27.2, turned 23.3).  Not with several row
// tiles, which share the rows and the weights in L2 while they go in step.  us, ring of two / now: 48 rows, 28672 x 4096 (pairs) 48.8 / 39.9,
// 16384 x 11008 78.2 / 64.9, 16032 x 8192 56.6 / 48.9; 112 rows, 28672 x 4096 (pairs) 55.5 / 52.5, 10240 x 8192 45.2 / 43.9.
// Steps of so and so many k-tiles meet the interleaving's own period where rows are an odd multiple of 1 KiB: there, from 4096 columns on, a tile
// begins where the fraction of nt times the golden ratio lies in K (48 rows, steps of five / so: 16384 x 6656 47.1 / 42.2, ring of two 42.6; 6656 x
// 6656 24.6 / 23.8, 8192 x 22016 81.0 / 70.6; 5120 x 13824 32.6 / 32.7, 6656 x 17920 49.7 / 50.5).  Of 81 products of other
// widths, 48 and 112 rows, it takes 0.94 to 1.04 of the steps' time, as long on average, and 26624 x 16384 (pairs), 112 rows, 204 us for 170.
// ---------------------------------------------------------------------------------------------
constexpr int GEMM_RING = 3, GEMM_TURN = 5;
constexpr unsigned GEMM_TURN_GOLDEN = 2654435761u;   // 2^32 / golden ratio, the prime next to it
struct GemmRope {   // the projection is the fused q/k/v projection of a prefill: see lr_linear_rope_kv
  const u16* table;
  const int32_t* pos;
  u16 *k_cache, *v_cache;
  int32_t* err;
  int S, Hq, Hkv, hd, Smax, block_size;
};
// The rows of a tile are entries of a list, tile (matrix, first entry, entries) as a device table says: input row
// entry / xdiv, output row entry, weights of one of several matrices that lie `wstride` elements apart.
struct GemmGroup {
  const int32_t* tiles;    // [][3]
  const int32_t* ntiles;
  const int32_t* entries;
  int xdiv;
  int64_t wstride;
  int64_t xrows;           // rows of x
};
// Tiles [0, full) are computed whole; each of the `rem` tiles after them is cut along K into `splits` pieces, whose fp32
// sums go to `part` in the order a wave holds them (k_gemm_sum adds them in order and finishes the tile), or, in ROWS mode
// (full == 0, N % 4 == 0), to part [splits][M][N] for a launch that needs whole rows anyway.
struct GemmSplit {
  float* part;
  int full, rem, splits;
  const u16* scales;   // of e4m3 weights, one per weight row
};
enum { GEMM_PLAIN, GEMM_PAIR, GEMM_ROPE, GEMM_ROWS };   // ROWS: every tile is cut, the pieces stay, see GemmSplit; PAIR: w holds [up; gate] rows, N counts pairs, output silu(gate) * up

template <int A, int BH, int R = 2, bool W8 = false>
struct GemmTile {
  static constexpr int KT = W8 ? 128 : 64;               // k elements of a k-tile: 128 bytes of a weight row
  static constexpr int NA = KT / 64;                     // 64-element parts of its input rows
  static constexpr int TM = 32 * A, TN = 128 * BH;
  static constexpr int A0 = (A + 1) / 2, A1 = A / 2;     // 16-row groups of a wave in either half of the input rows
  static constexpr int NB = 2 * BH;                      // DMA instructions of a wave for half a k-tile of weights (of input rows: A0, A1)
  static constexpr int HB = 8192 * BH;                   // its bytes
  static constexpr int ABYTES = 4096 * A * NA;           // and those of a k-tile of input rows
  static constexpr int SLOT = ABYTES + 2 * HB;           // a k-tile
  static constexpr int RING = R * SLOT;
  static constexpr int EPITCH = 64 * BH + 8;             // row pitch of a wave's output piece (plain), in elements
  static constexpr int EBYTES = 4 * 16 * A * EPITCH * 2;
  static constexpr int LDS = RING > EBYTES ? RING : EBYTES;
  // tile row at which 16-row group g of the waves `wm` begins
  static __device__ __forceinline__ int group_row(int g, int wm) { return g < A0 ? wm * 16 * A0 + g * 16 : 32 * A0 + wm * 16 * A1 + (g - A0) * 16; }
};

// workgroups of a tile that share a CU (LDS and registers: 160 KB, 256 registers per lane)
constexpr int GEMM_PER_CU(int A, int BH) { return A * BH <= 5 ? 2 : 1; }

typedef int i32x4_t __attribute__((ext_vector_type(4)));
// One wave instruction: 64 x 16 bytes from memory to LDS at `lds` + 16 * lane.  M0, which holds `lds`, is an operand: the
// compiler writes it and knows that it did.  (s_nop: the wait state between that and its use; the scalar operands come from
// scalar instructions.)
template <bool NT>
__device__ __forceinline__ void dma16(const i32x4_t& rsrc, int voff, int soff, u32 lds) {
  if (NT)
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"{m0}"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
  else
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"{m0}"(lds), "v"(voff), "s"(rsrc), "s"(soff) : "memory");
}
// the low (HI == false) or high two e4m3 values of a dword as a packed bf16 pair (exact)
template <bool HI>
__device__ __forceinline__ u32 gemm_fp8_pair(u32 v) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(u32, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, HI));
}
template <int N>
__device__ __forceinline__ void wait_requests_and_lds() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// Which of `n` tiles workgroup `id` of `count` takes: an XCD (id % 8) has a contiguous run of them.
__device__ __forceinline__ int xcd_run(int id, int n) {
  const int xcd = id & 7, base = n >> 3, rem = n & 7;
  return xcd * base + (xcd < rem ? xcd : rem) + (id >> 3);
}
// Tile number -> (row tile, column tile): bands of up to four row tiles, a band's columns one after the other, so that the
// workgroups an XCD runs at the same time share operand rows in its L2.
__device__ __forceinline__ void gemm_tile_at(int t, int tm, int tn, int& mt, int& nt) {
  const int band = t / (4 * tn), r = t - band * 4 * tn;
  const int h = tm - band * 4 < 4 ? tm - band * 4 : 4;
  nt = r / h;
  mt = band * 4 + r - nt * h;
}

// Eight columns of an output row, from column n on.
__device__ __forceinline__ void gemm_put(u16* __restrict__ y, int64_t ldy, int N, int m, int n, const uint4& v) {
  if ((ldy & 7) == 0 && n + 7 < N) {
    st16(y + (int64_t)m * ldy + n, v);
  } else {
    const u32 q[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (n + e < N) y[(int64_t)m * ldy + n + e] = (u16)(q[e >> 1] >> ((e & 1) * 16));
  }
}
// The section (q, k, v), head and dimension of column n.
__device__ __forceinline__ void gemm_rope_at(const GemmRope& rp, int n, int& sect, int& hh, int& dd) {
  const int nq = rp.Hq * rp.hd, nkv = rp.Hkv * rp.hd;
  sect = n < nq ? 0 : (n < nq + nkv ? 1 : 2);
  const int cc = n - (sect == 0 ? 0 : (sect == 1 ? nq : nq + nkv));
  hh = cc / rp.hd;
  dd = cc - hh * rp.hd;
}
// What k_rope_kv_write would do to eight columns of sequence b's row at position ps, with their table entries tv; what is stored.
__device__ __forceinline__ uint4 gemm_rope(const GemmRope& rp, int sect, int hh, int dd, int b, int ps, const uint4& v, const uint4& tv) {
  const uint4 r = sect < 2 ? rope8(v, tv) : v;
  if (sect == 0) return r;
  st16((sect == 1 ? rp.k_cache : rp.v_cache) + (((int64_t)b * rp.Hkv + hh) * rp.Smax + ps) * rp.hd + dd, r);
  return v;
}

// The outputs of a wave's part of a tile.  The products are W-tile x X-tile^T: a lane of
// acc[a][b] holds four consecutive columns 4 (lane / 16) .. of row lane % 16; b < 2 BH are columns of the tile's first half
// of weight rows, the others of its second.  Stored from there an instruction would touch 32 bytes in each of 16 rows: they
// take one trip through LDS (`eb`, a piece of the wave's own) and leave as whole rows.
template <int A, int BH, int MODE>
__device__ __forceinline__ void gemm_store(const f32x4_t (&acc)[A][4 * BH], u16* eb, int wm, int wn, int m0, int n0, u16* __restrict__ y,
                                           int64_t ldy, int M, int N, const GemmRope& rp, const int32_t* entry) {
  int lane = threadIdx.x & 63;   // (laundered: the addresses below are not formed before the k loop and kept through it)
  asm volatile("" : "+v"(lane));
  constexpr bool P = MODE == GEMM_PAIR;
  constexpr int HC = 32 * BH;                        // a wave's columns in one half
  constexpr int EP = (P ? HC : 2 * HC) + 8;
#pragma unroll
  for (int a = 0; a < A; ++a) {
    const int ml = a * 16 + (lane & 15);
#pragma unroll
    for (int b = 0; b < (P ? 2 * BH : 4 * BH); ++b) {
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = P ? swiglu_bf(round_bf(acc[a][b][e]), round_bf(acc[a][b + 2 * BH][e])) : acc[a][b][e];
      *reinterpret_cast<uint2*>(&eb[ml * EP + b * 16 + (lane >> 4) * 4]) = make_uint2(pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3]));
    }
    __builtin_amdgcn_sched_barrier(0);   // (not all accumulators out of their half of the register file at once)
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // a wave reads back only what it wrote itself
  constexpr int LPR = HC / 8, RPI = 64 / LPR;         // lanes per row, rows per instruction
  const int cl = (lane % LPR) * 8;
  auto row_of = [&](int ml) { return m0 + GemmTile<A, BH>::group_row(ml >> 4, wm) + (ml & 15); };
  auto store_row = [&](int m, int n, const uint4& v) {
    if (m >= M) return;
    gemm_put(y, ldy, N, entry != nullptr ? entry[m] : m, n, v);
  };
#pragma unroll
  for (int hb = 0; hb < (P ? 1 : 2); ++hb) {
    const int n = n0 + hb * 64 * BH + wn * HC + cl;
    if constexpr (MODE == GEMM_ROPE) {
      // What k_rope_kv_write would do to the stored rows.  The lane's eight columns lie in one head of one section
      // (head_dim % 8 == 0).  Positions of several rows first, then their table entries, then the arithmetic: two memory
      // round trips per RB rows (row by row the position and the entry it selects are a chain of two loads per row, and
      // the output pass of a tile took three times as long).
      constexpr int RI = A * 16 / RPI, RB = RI <= 8 ? RI : RI % 8 == 0 ? 8 : RI / 2;   // (10, 12 and 14 in two halves)
      static_assert(RI % RB == 0 && RB <= 8, "");
      int sect, hh, dd;
      gemm_rope_at(rp, n, sect, hh, dd);
      for (int i0 = 0; i0 < RI; i0 += RB) {
        int ps[RB], bb[RB];
#pragma unroll
        for (int i = 0; i < RB; ++i) {
          const int m = row_of((i0 + i) * RPI + lane / LPR);
          bb[i] = m / rp.S;
          ps[i] = (m < M && n < N) ? rp.pos[m - bb[i] * rp.S] : -1;  // (N % 8 == 0 and ldy % 8 == 0: the columns are whole)
        }
        uint4 tv[RB];
        bool ok[RB];
#pragma unroll
        for (int i = 0; i < RB; ++i) {
          ok[i] = ps[i] >= 0 && ps[i] < rp.Smax && ps[i] < rp.block_size;
          tv[i] = (ok[i] && sect < 2) ? ld16(rp.table + (int64_t)ps[i] * rp.hd + dd) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < RB; ++i) {
          const int ml = (i0 + i) * RPI + lane / LPR, m = row_of(ml);
          uint4 v = *reinterpret_cast<const uint4*>(&eb[ml * EP + hb * HC + cl]);
          if (ok[i]) {
            v = gemm_rope(rp, sect, hh, dd, bb[i], ps[i], v, tv[i]);
          } else if (m < M && n == 0 && rp.err) {
            *rp.err = LR_DEV_POS_RANGE;
          }
          store_row(m, n, v);
        }
      }
    } else {
#pragma unroll 4
      for (int r0 = 0; r0 < A * 16; r0 += RPI) {
        const int ml = r0 + lane / LPR;
        store_row(row_of(ml), n, *reinterpret_cast<const uint4*>(&eb[ml * EP + hb * HC + cl]));
      }
    }
  }
}

// KTAIL: K is not a multiple of the 64-element k-tile, so the last one needs a per-lane range check.  NT: weights are loaded
// non-temporally.
// W8: e4m3 weights with a bf16 scale per row, K % 128 == 0.  A k-tile is 128 elements: as many bytes of a weight row as of 64 in bf16 and
// two parts of the input rows.  A lane takes sixteen consecutive k of its row in one LDS read, expands them on their way into the
// matrix instructions (exactly: e4m3 is a subset of bf16) and multiplies them by the input's same sixteen, eight and eight; the sums are
// scaled as they are, in fp32, before anything else sees them.  The ring holds two k-tiles, 64 KiB, so that two workgroups share a CU.
// Bound: what a CU draws, of which the input rows are half (58 GB/s: 0.55 us per k-tile), below HBM's rate.  us, 64 rows, in passes of 16
// through the bands / here: 14336 x 4096 pairs 160 / 26.2, 8B decode step 10154 / 3505; 70B rank shard 14067 / 4843, 17 rows 6298 / 4120.
template <int A, int BH, bool KTAIL, int MODE, bool GROUP, bool NT, int R = 2, bool W8 = false>
__device__ __forceinline__ void gemm_tile(const int block, const int blocks, const u16* __restrict__ x, int64_t ldx, const u16* __restrict__ w,
                                          u16* __restrict__ y, int64_t ldy, int M, int N, int K, int tm, int tn, const GemmRope& rp,
                                          const GemmSplit& sp, const GemmGroup& gp) {
  using T = GemmTile<A, BH, R, W8>;
  static_assert(!W8 || (!KTAIL && !GROUP), "");
  // Where k-tile t lies in LDS: of a ring of two by its parity, a constant; else a slot is input rows and weight rows together, at
  // an offset that goes round with the loop.
  constexpr bool LONG = R > 2 || W8;
  constexpr int KT = T::KT, NA = T::NA, KS = KT / 32, WB = W8 ? 1 : 2;   // (KS: k-steps; WB: bytes per weight)
  constexpr int A0 = T::A0, A1 = T::A1, HB = T::HB, NB = T::NB, BOFF = LONG ? T::ABYTES : 2 * T::ABYTES;
  constexpr int APAR = LONG ? 0 : T::ABYTES, BPAR = LONG ? 0 : 2 * HB;
  extern __shared__ __attribute__((aligned(1024))) u16 gsm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  int mt, nt, piece = -1, kt0 = 0, nk = (K + KT - 1) / KT;
  int32_t* const entry = reinterpret_cast<int32_t*>(gsm + T::LDS / 2);   // (GROUP) the tile's entries
  if constexpr (GROUP) {
    const int tiles = gp.ntiles[0] * tn;   // (of the grid's: there may be fewer, and each XCD has its share of those there are)
    if (block >= tiles) return;
    const int id = xcd_run(block, tiles);   // a row tile's column tiles one after the other
    mt = id / tn;
    nt = id - mt * tn;
    const int32_t* tile = gp.tiles + 3 * mt;
    w += tile[0] * gp.wstride;
    M = tile[2];
    if (tid < T::TM) entry[tid] = gp.entries[tile[1] + (tid < M ? tid : 0)];
    mt = 0;
    __syncthreads();
  } else {
    int t = block;
    if (t < sp.full) {
      t = xcd_run(t, sp.full);
    } else {
      const int q = xcd_run(t - sp.full, sp.rem * sp.splits), split = q / sp.rem;
      t = sp.full + q - split * sp.rem;
      piece = (t - sp.full) * sp.splits + split;
      const int pairs = (nk + 1) / 2, p0 = (int)((int64_t)pairs * split / sp.splits), p1 = (int)((int64_t)pairs * (split + 1) / sp.splits);
      kt0 = 2 * p0;
      nk = (nk < 2 * p1 ? nk : 2 * p1) - kt0;
    }
    gemm_tile_at(t, tm, tn, mt, nt);
  }
  const int m0 = mt * T::TM, n0 = nt * (MODE == GEMM_PAIR ? T::TN / 2 : T::TN);

  // Requests.  Instruction i of a wave's share of a half covers the half's rows (wave * n + i) * 8 + lane / 8, a lane 16
  // bytes of one.  Operand rows are read through buffer resources that hold the tile's rows and no more; a row beyond M or N
  // has an offset outside the resource and reads as zero.
  const u16* const xb = x + (int64_t)m0 * ldx + kt0 * KT;
  const u16* const wb = reinterpret_cast<const u16*>(reinterpret_cast<const char*>(w) + ((int64_t)n0 * K + kt0 * KT) * WB);
  constexpr int OUT = (int)0x80000000;
  const int klen = K - kt0 * KT;
  const int chunk = ((lane & 7) ^ (lane >> 3)) * 8;      // (row % 8 == lane / 8)
  int xo[2][A0], wo[2][NB];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int i = 0; i < (h ? A1 : A0); ++i) {
      const int r = h * 32 * A0 + (wave * (h ? A1 : A0) + i) * 8 + (lane >> 3);
      const int row = GROUP ? entry[r] / gp.xdiv : r;
      xo[h][i] = m0 + r < M ? (int)((int64_t)row * ldx * 2) + chunk * 2 : OUT;
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int r = (wave * NB + i) * 8 + (lane >> 3);
      if (MODE == GEMM_PAIR) wo[h][i] = n0 + r < N ? (int)((int64_t)(h * N + r) * K * WB) + chunk * 2 : OUT;   // (half 0 up, half 1 gate)
      else wo[h][i] = n0 + h * 64 * BH + r < N ? (int)((int64_t)(h * 64 * BH + r) * K * WB) + chunk * 2 : OUT;
    }
  }
  const u32 lds0 = __builtin_amdgcn_readfirstlane((u32)(uintptr_t)(__attribute__((address_space(3))) u16*)gsm);
  const int64_t xlast = GROUP ? gp.xrows - 1 : (M - m0 < T::TM ? M - m0 : T::TM) - 1;
  const int64_t wlast = MODE == GEMM_PAIR ? N + (int64_t)(N - n0 < T::TN / 2 ? N - n0 : T::TN / 2) - 1 : (N - n0 < T::TN ? N - n0 : T::TN) - 1;
  const int xbytes = (int)((xlast * ldx + klen) * 2), wbytes = (int)((wlast * K + klen) * WB);   // (below 2 GiB: gemm_reaches)
  // the k-tile that is multiplied first
  const bool golden = !W8 && K % 1024 == 512 && K >= 4096;
  const int turn = !LONG ? 0 : golden ? (int)__umulhi((unsigned)nt * GEMM_TURN_GOLDEN, (unsigned)nk) : (int)((unsigned)(nt * GEMM_TURN) % (unsigned)nk);
  auto request = [&](auto ONCE, const u16* base, int bytes, int voff, int t, int per, int part, u32 lds) {   // (per: bytes of a row in a k-tile)
    const bool in = t < nk;
    if (LONG) t = t + turn < nk ? t + turn : t + turn - nk;
    i32x4_t r;
    r.x = (int)(u32)(unsigned long long)base;
    r.y = (int)(u32)((unsigned long long)base >> 32) & 0xffff;
    r.z = in ? bytes : 0;
    r.w = 0x00020000;
    if (KTAIL) voff = t * 64 + chunk < klen ? voff : OUT;
    dma16<decltype(ONCE)::value>(r, voff, in ? t * per + part * 128 : 0, lds);
  };
  auto dma_a = [&](int t, int par, int slot, int h, int e) {   // part e % NA of the wave's e / NA-th rows
    const int i = e / NA, part = e % NA;
    request(std::false_type{}, xb, xbytes, xo[h][i], t, 2 * KT, part,
            lds0 + slot + par * APAR + part * 4096 * A + h * 4096 * A0 + (wave * (h ? A1 : A0) + i) * 1024);
  };
  auto dma_b = [&](int t, int par, int slot, int h, int i) {
    request(std::bool_constant<NT>{}, wb, wbytes, wo[h][i], t, 128, 0, lds0 + slot + BOFF + par * BPAR + h * HB + (wave * NB + i) * 1024);
  };

  f32x4_t acc[A][4 * BH];
#pragma unroll
  for (int a = 0; a < A; ++a)
#pragma unroll
    for (int b = 0; b < 4 * BH; ++b)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[a][b][v] = 0.0f;
  bf16x8_t af[2][A0][KS], bf[2][2 * BH][KS];
  u32x4_t raw[2 * BH][2];   // (W8) half a k-tile's weights as they are: sixteen consecutive k of a lane's row, twice
  const char* const smb = reinterpret_cast<const char*>(gsm);
  int fa[2][2], fb[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int c = ((4 * ks + (lane >> 4)) ^ (lane & 7)) * 16;
    const int ca = W8 ? ((2 * (lane >> 4) + ks) ^ (lane & 7)) * 16 : c;   // (W8: the k of the lane's weights, eight and eight)
    fa[0][ks] = (wm * 16 * A0 + (lane & 15)) * 128 + ca;
    fa[1][ks] = (wm * 16 * A1 + (lane & 15)) * 128 + ca;
    fb[ks] = (wn * 32 * BH + (lane & 15)) * 128 + c + BOFF;
  }
  auto read_a = [&](int par, int slot, int h, int t, int ks) {
    af[h][t][ks] = *reinterpret_cast<const bf16x8_t*>(smb + (fa[h][ks & 1] + slot) + par * APAR + (ks >> 1) * 4096 * A + h * 4096 * A0 + t * 2048);
  };
  auto read_b = [&](int set, int par, int slot, int h, int t, int ks) {   // (W8: ks half the k-steps)
    const char* const at = smb + (fb[ks] + slot) + par * BPAR + h * HB + t * 2048;
    if constexpr (W8) raw[t][ks] = *reinterpret_cast<const u32x4_t*>(at);
    else bf[set][t][ks] = *reinterpret_cast<const bf16x8_t*>(at);
  };
  auto expand = [&](int half) {   // what read_b has read, as bf16 (exactly)
#pragma unroll
    for (int t = 0; t < 2 * BH; ++t)
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const u32 lo = raw[t][ks >> 1][2 * (ks & 1)], hi = raw[t][ks >> 1][2 * (ks & 1) + 1];
        const u32x4_t v = {gemm_fp8_pair<false>(lo), gemm_fp8_pair<true>(lo), gemm_fp8_pair<false>(hi), gemm_fp8_pair<true>(hi)};
        if constexpr (W8) bf[half][t][ks] = __builtin_bit_cast(bf16x8_t, v);
      }
  };
  auto barrier = [&] {
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  constexpr int QA0 = NA * A0, QA1 = NA * A1, QA = QA0 + QA1, AHEAD = (R - 2) * (QA + 2 * NB);   // requests of a wave; those beyond two k-tiles'
  // the scales of the lane's columns, ahead of the requests that are counted
  float scale[2 * BH * 2][4];
  if constexpr (W8) {
#pragma unroll
    for (int b = 0; b < 4 * BH; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int half = b / (2 * BH), c = n0 + (MODE == GEMM_PAIR ? 0 : half * 64 * BH) + wn * 32 * BH + b % (2 * BH) * 16 + (lane >> 4) * 4 + e;
        scale[b][e] = bf_to_f(sp.scales[c < N ? c + (MODE == GEMM_PAIR ? half * N : 0) : 0]);
      }
    asm volatile("" ::: "memory");
  }
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int par = t & 1, slot = LONG ? t * T::SLOT : 0;
#pragma unroll
    for (int i = 0; i < QA0; ++i) dma_a(t, par, slot, 0, i);
#pragma unroll
    for (int i = 0; i < NB; ++i) dma_b(t, par, slot, 0, i);
#pragma unroll
    for (int i = 0; i < NB; ++i) dma_b(t, par, slot, 1, i);
#pragma unroll
    for (int i = 0; i < QA1; ++i) dma_a(t, par, slot, 1, i);
  }
  wait_requests_and_lds<AHEAD + QA0 + 2 * QA1 + 3 * NB>();
  barrier();
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
    for (int t = 0; t < A0; ++t) read_a(0, 0, 0, t, ks);
#pragma unroll
    for (int t = 0; t < 2 * BH; ++t)
      if (ks < 2) read_b(0, 0, 0, 0, t, ks);
  }
  wait_requests_and_lds<AHEAD + QA0 + 2 * QA1 + 3 * NB>();
  barrier();
#pragma unroll
  for (int i = 0; i < QA0; ++i) dma_a(R, 0, 0, 0, i);

  // Phase P of k-tile t (even: PAR 0).  Reads B1 of this tile, A1 of this tile, A0 of the next, B0 of the next; requests
  // B0, B1, A1 of tile t + R and A0 of tile t + 1 + R.  `here`, `next`: the slots of this tile and the next.
  auto phase = [&](auto PAR_, auto P_, int t, int here, int next) {
    constexpr int PAR = decltype(PAR_)::value, P = decltype(P_)::value;
    constexpr int ah = P >> 1, bh = (P == 1 || P == 2), set = W8 ? bh : bh ^ PAR;
    // requests younger than the slot read here: those of the six phases since
    wait_requests_and_lds<AHEAD + (P == 0 ? 2 * QA + 2 * NB : P == 1 ? QA + QA0 + 3 * NB : P == 2 ? QA + 4 * NB : QA + QA1 + 3 * NB)>();
    barrier();
    constexpr int AH = ah ? A1 : A0, J = 2 * KS * AH * BH, RD = P == 1 ? KS * A1 : P == 2 ? KS * A0 : 4 * BH, RQ = P == 2 ? QA1 : P == 3 ? QA0 : NB;
    if constexpr (W8 && P < 2) {
      expand(P);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int tb = j % (2 * BH), ta = j / (2 * BH) % AH, ks = j / (2 * AH * BH);
      if constexpr (W8)   // (behind vector instructions that write its operand: the compiler sees to the wait states)
        acc[ah * A0 + ta][bh * 2 * BH + tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[set][tb][ks], af[ah][ta][ks], acc[ah * A0 + ta][bh * 2 * BH + tb], 0, 0, 0);
      else
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+a"(acc[ah * A0 + ta][bh * 2 * BH + tb])
                     : "v"(bf[set][tb][ks]), "v"(af[ah][ta][ks]));
      if (j < J / 2) {
#pragma unroll
        for (int e = j * RD / (J / 2); e < (j + 1) * RD / (J / 2); ++e) {
          if (P == 0) read_b(1 ^ PAR, PAR, here, 1, e % (2 * BH), e / (2 * BH));
          if (P == 1) read_a(PAR, here, 1, e % A1, e / A1);
          if (P == 2) read_a(PAR ^ 1, next, 0, e % A0, e / A0);
          if (P == 3) read_b(1 ^ PAR, PAR ^ 1, next, 0, e % (2 * BH), e / (2 * BH));
        }
      } else {
#pragma unroll
        for (int e = (j - J / 2) * RQ / (J / 2); e < (j + 1 - J / 2) * RQ / (J / 2); ++e) {
          if (P == 0) dma_b(t + R, PAR, here, 0, e);
          if (P == 1) dma_b(t + R, PAR, here, 1, e);
          if (P == 2) dma_a(t + R, PAR, here, 1, e);
          if (P == 3) dma_a(t + 1 + R, PAR ^ 1, next, 0, e);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  {
    std::integral_constant<int, 0> c0;
    std::integral_constant<int, 1> c1;
    std::integral_constant<int, 2> c2;
    std::integral_constant<int, 3> c3;
    int s0 = 0;
    auto after = [](int slot) { return !LONG ? 0 : slot + T::SLOT < T::RING ? slot + T::SLOT : 0; };
    for (int t = 0; t < nk; t += 2) {   // (an odd number of k-tiles ends with one of zeros)
      const int s1 = after(s0), s2 = after(s1);
      phase(c0, c0, t, s0, s1);
      phase(c0, c1, t, s0, s1);
      phase(c0, c2, t, s0, s1);
      phase(c0, c3, t, s0, s1);
      phase(c1, c0, t + 1, s1, s2);
      phase(c1, c1, t + 1, s1, s2);
      phase(c1, c2, t + 1, s1, s2);
      phase(c1, c3, t + 1, s1, s2);
      s0 = s2;
    }
  }
  // the last matrix instructions' results can be read (they are assembler text: the wait states are ours), nothing is on its
  // way into LDS, nobody still reads it
  asm volatile("s_nop 15\n\ts_nop 15\n\ts_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if constexpr (W8)
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
      for (int b = 0; b < 4 * BH; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[a][b][e] *= scale[b][e];
  if constexpr (!GROUP) {
    if constexpr (MODE == GEMM_ROWS) {
      float* const p = sp.part + (int64_t)(piece % sp.splits) * M * N;
#pragma unroll
      for (int a = 0; a < A; ++a) {
        const int m = m0 + T::group_row(a, wm) + (lane & 15);
#pragma unroll
        for (int b = 0; b < 4 * BH; ++b) {
          const int n = n0 + b / (2 * BH) * 64 * BH + wn * 32 * BH + b % (2 * BH) * 16 + (lane >> 4) * 4;
          if (m < M && n < N) *reinterpret_cast<f32x4_t*>(p + (int64_t)m * N + n) = acc[a][b];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      return;
    } else if (piece >= 0) {
      float* p = sp.part + (int64_t)piece * (T::TM * T::TN) + (int64_t)wave * (4 * A * BH * 256) + lane * 4;
#pragma unroll
      for (int a = 0; a < A; ++a) {
#pragma unroll
        for (int b = 0; b < 4 * BH; ++b) *reinterpret_cast<f32x4_t*>(p + (a * 4 * BH + b) * 256) = acc[a][b];
        __builtin_amdgcn_sched_barrier(0);
      }
      return;
    }
  }
  if constexpr (MODE != GEMM_ROWS) gemm_store<A, BH, MODE>(acc, gsm + wave * (T::EBYTES / 8), wm, wn, m0, n0, y, ldy, M, N, rp, GROUP ? entry : nullptr);
}

template <int A, int BH, bool KTAIL, int MODE, bool GROUP, bool NT = false, int R = 2, bool W8 = false>
__global__ __launch_bounds__(256, R > 2 && A > 2 ? 1 : GEMM_PER_CU(A, BH)) void k_gemm_dma(const u16* __restrict__ x, int64_t ldx, const u16* __restrict__ w,
                                                                        u16* __restrict__ y, int64_t ldy, int M, int N, int K, int tm, int tn,
                                                                        const GemmRope rp, const GemmSplit sp, const GemmGroup gp) {
  gemm_tile<A, BH, KTAIL, MODE, GROUP, NT, R, W8>(blockIdx.x, gridDim.x, x, ldx, w, y, ldy, M, N, K, tm, tn, rp, sp, gp);
}

// Two products of as many rows in one grid, the first `n0` workgroups the first's.  A short prompt's products each leave most
// of the chip idle or end with a ramp and a drain of their own; in a ladder block q/k/v and up/gate have their inputs at the
// same time, and so have, behind the attention, wo and w2.
struct GemmProduct {
  const u16* x;
  int64_t ldx;
  const u16* w;
  u16* y;
  int64_t ldy;
  int M, N, K, tm, tn;
  GemmSplit sp;
};
template <int A, int BH, int MODE0, int MODE1, bool NT, int R, bool W8>
__global__ __launch_bounds__(256, R > 2 && A > 2 ? 1 : GEMM_PER_CU(A, BH)) void k_gemm_two(const GemmProduct a, const GemmProduct b, const int n0, const GemmRope rp) {
  const bool second = (int)blockIdx.x >= n0;
  if constexpr (MODE0 == MODE1) {
    const GemmProduct p = second ? b : a;
    gemm_tile<A, BH, false, MODE0, false, NT, R, W8>(blockIdx.x - (second ? n0 : 0), 0, p.x, p.ldx, p.w, p.y, p.ldy, p.M, p.N, p.K, p.tm, p.tn, rp, p.sp, GemmGroup{});
  } else if (second) {
    gemm_tile<A, BH, false, MODE1, false, NT, R, W8>(blockIdx.x - n0, 0, b.x, b.ldx, b.w, b.y, b.ldy, b.M, b.N, b.K, b.tm, b.tn, GemmRope{}, b.sp, GemmGroup{});
  } else {
    gemm_tile<A, BH, false, MODE0, false, NT, R, W8>(blockIdx.x, 0, a.x, a.ldx, a.w, a.y, a.ldy, a.M, a.N, a.K, a.tm, a.tn, rp, a.sp, GemmGroup{});
  }
}

// The attention of a decode step of 17 to 64 sequences and the block's up/gate product, which do not depend on each other in a ladder
// or a parallel block, in one grid: an attention item (attn_decode_item.h) for every CU, the product's tiles, the other items, the
// waves that merge them.  Bound: HBM; apart, the attention's items leave the memory idle between their rows' arrival and the next
// item's request, and the product's workgroups at their ramp and drain.  us per step of the 70B rank shard at 64 rows: the two chains of
// a block on two branches of the graph 7125, in this grid 6825 (all items behind the tiles 6935, all in front 7059; the plan's three
// pieces of K, with four 7340), of it per block 38 here, where the product alone takes 28 and the attention alone 16 and 4.
// An item for every CU, and of more than two rounds one round more, so that a round is left for the CUs whose tiles are done (70B rank
// shard, 2048 tokens, 64 rows, 768 items: 256 in front 6523 us per step, 512 6296, all 6282; 40 rows, 520 items: 256 5856, 512 5892).
__device__ __forceinline__ int attn_items_in_front(int items) {
  return items < ATT_NCU ? items : items <= 2 * ATT_NCU ? ATT_NCU : items - ATT_NCU < 2 * ATT_NCU ? items - ATT_NCU : 2 * ATT_NCU;
}
template <int HD, int G, int GROUPS, bool W8>
__global__ __launch_bounds__(256, 2) void k_attn_beside_gemm(const AttnItems a, const GemmProduct p, const int n_gemm) {
  extern __shared__ __attribute__((aligned(1024))) u16 gsm[];
  const int first = attn_items_in_front(a.n_items), tile = (int)blockIdx.x - first, wg = tile < 0 ? (int)blockIdx.x : (int)blockIdx.x - n_gemm;
  if (tile >= 0 && tile < n_gemm)
    gemm_tile<2, 1, false, GEMM_PAIR, false, true, W8 ? 2 : GEMM_RING, W8>(tile, 0, p.x, p.ldx, p.w, p.y, p.ldy, p.M, p.N, p.K, p.tm, p.tn, GemmRope{}, p.sp, GemmGroup{});
  else if (wg < a.n_items)
    attn_item<HD, G, GROUPS, true>(a, wg, reinterpret_cast<float*>(gsm));
  else
    attn_merge<HD, G>(a, wg - a.n_items);
}

// The cut tiles: a workgroup adds the pieces of 16 rows of a wave's part of one and finishes them.  Bound: memory, mostly the
// last-level cache, since the pieces were just written; of small products the round trips: so a wave takes a quarter of the
// columns, up to eight pieces' loads in flight together, summed in order, and a lane finishes eight columns of one row.  (A
// wave for all columns and four pieces at a time, us: q/k/v of the 70B rank shard at 64 rows, 16 pieces, 7.1 -> 4.9, up/gate 4.7 -> 4.9.)
template <int A, int BH, int MODE>
__global__ __launch_bounds__(256) void k_gemm_sum(u16* __restrict__ y, int64_t ldy, int M, int N, int tm, int tn, const GemmRope rp, const GemmSplit sp) {
  using T = GemmTile<A, BH>;
  constexpr bool P = MODE == GEMM_PAIR;
  constexpr int HC = 32 * BH, EP = (P ? HC : 2 * HC) + 8;
  __shared__ __attribute__((aligned(16))) u16 eb[16 * EP];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int part = blockIdx.x & 3, wm = part >> 1, wn = part & 1;
  const int rt = blockIdx.x / (4 * A), g = blockIdx.x / 4 - rt * A;
  int mt, nt;
  gemm_tile_at(sp.full + rt, tm, tn, mt, nt);
  const int m0 = mt * T::TM + T::group_row(g, wm), n0 = nt * (P ? T::TN / 2 : T::TN) + wn * HC;
  if (m0 >= M) return;   // uniform
  constexpr int C = 4 * BH, STEP = T::TM * T::TN, UNITS = P ? 2 * BH : C;   // a unit: sixteen columns, or as many pairs
  const float* const p = sp.part + (int64_t)rt * sp.splits * STEP + ((int64_t)part * A + g) * (C * 256) + lane * 4;
  for (int u = wave; u < UNITS; u += 4) {
    constexpr int NF = P ? 2 : 1, NP = 8;
    f32x4_t acc[NF], v[NP][NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = *reinterpret_cast<const f32x4_t*>(p + (u + f * 2 * BH) * 256);
    for (int s = 1; s < sp.splits; s += NP) {
#pragma unroll
      for (int i = 0; i < NP; ++i)
#pragma unroll
        for (int f = 0; f < NF; ++f)
          v[i][f] = *reinterpret_cast<const f32x4_t*>(p + (int64_t)(s + i < sp.splits ? s + i : 0) * STEP + (u + f * 2 * BH) * 256);
#pragma unroll
      for (int i = 0; i < NP; ++i)
        if (s + i < sp.splits) {
#pragma unroll
          for (int f = 0; f < NF; ++f) acc[f] += v[i][f];
        }
    }
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = P ? swiglu_bf(round_bf(acc[0][e]), round_bf(acc[NF - 1][e])) : acc[0][e];
    *reinterpret_cast<uint2*>(&eb[(lane & 15) * EP + u * 16 + (lane >> 4) * 4]) = make_uint2(pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3]));
  }
  __syncthreads();
  constexpr int LPR = HC / 8, LANES = 16 * LPR * (P ? 1 : 2);   // of a row's half
  static_assert(LANES <= 256, "");
  if (tid >= LANES) return;
  const int hb = tid / (16 * LPR), r = tid / LPR % 16, cl = tid % LPR * 8;
  const int m = m0 + r, n = n0 + hb * 64 * BH + cl;
  if (m >= M) return;
  uint4 v = *reinterpret_cast<const uint4*>(&eb[r * EP + hb * HC + cl]);
  if constexpr (MODE == GEMM_ROPE) {
    int sect, hh, dd;
    gemm_rope_at(rp, n, sect, hh, dd);
    const int b = m / rp.S, ps = rp.pos[m - b * rp.S];
    if (n < N && ps >= 0 && ps < rp.Smax && ps < rp.block_size)
      v = gemm_rope(rp, sect, hh, dd, b, ps, v, sect < 2 ? ld16(rp.table + (int64_t)ps * rp.hd + dd) : make_uint4(0, 0, 0, 0));
    else if (n == 0 && rp.err)
      *rp.err = LR_DEV_POS_RANGE;
  }
  gemm_put(y, ldy, N, m, n, v);
}

// ---- which tile, and which tiles are cut along K
struct GemmPlan {
  int tile;        // index into GEMM_TILES; -1: no tile serves the shape
  int full, rem, splits;
  float us;        // what it should take
};
// A round of workgroups takes k * (ktile + busy * slope), `busy` the workgroups per CU: the more CUs are at work, the lower
// the clock and the more of them ask the L2s.  Two to a CU take `pair` per k-tile.  A single row tile reads every weight from
// HBM itself, which is `cold` (`pair_cold`) in their place; with two row tiles GEMM_TWO of the way to it is left, with more
// none (128 x 128, two to a CU: 1.25 | 0.93 | 0.87 us per k-tile).  `fixed` is the ramp and drain of a round, `store` what the
// outputs of a whole tile per CU add to it; weights and outputs need their time from and to HBM whatever the tiles.  Pieces
// cost a launch, their trip through memory and the round trips of whoever adds them.
// The costs are fitted to 1296 products, 33 to 16384 rows of the 37 weights of the model families, with 64 MiB for pieces, 6.5 and
// none (2700 choices, of each the tiles and pieces that could be near the best, weights from HBM).  What the plan takes is 0.8 % above
// the best of them on average and 22 % at worst; with the costs of the fit before (219 products of up to 3002 rows, 90 of more) 1.2 and
// 25 %, with those before that 2.2 and 38 %.  Some products in us, N x K, with the first costs / the second / now | the best there is:
//   128 rows,  2048 x  2048  12.4 / 10.4 / 10.4 | 10.1         200 rows,  8192 x   512   6.0 /  7.2 /  6.0 |  6.0
//   128 rows,  3072 x  2048  17.2 / 13.3 / 13.3 | 13.0         900 rows,  2048 x    16   4.2 /  5.1 /  4.2 |  4.2
//   128 rows,  4096 x 14336  38.3 / 32.8 / 32.8 | 32.8        1501 rows,  7168 x  8192 153.9 / 168.2 / 153.9 | 153.9 (pairs)
//   128 rows, 28672 x  4096  65.8 / 54.8 / 54.8 | 54.8 (pairs)  2100 rows, 4608 x 4096  79.2 / 82.3 / 79.2 | 77.2
// Tiles of 160, 192 and 224 rows came later; their costs are fitted to 1457 products of 131 to 4096 rows of 31 weights, with 64 MiB for pieces
// and none, the first four tiles' as they were.  160 x 128 is cut into eight pieces at most: of a single row tile more were the slower choice
// (131 to 160 rows: 1280 x 8192 15.5 -> 16.5 us, 2048 x 5120 16.2 -> 17.9).  The products take 4.7 % less on average, 12 of 2898 choices
// more than 2 % more (777 rows, 2048 x 8192 36.8 -> 40.7, 2200 rows, 6144 x 2048 49.4 -> 53.0, 4096 rows, 6144 x 4096 without memory 158 -> 167,
// else less than 5 %; costs that spare these lose as much elsewhere), and the plan is 0.8 % above the best choice.  us, with four tiles / now:
//   300 rows, 28672 x 4096 100.3 / 74.0 (pairs)   450 rows,  7168 x 8192  69.4 / 58.7 (pairs)   777 rows, 28672 x 4096 197.2 / 176.9 (pairs)
//   777 rows,  6144 x 4096  55.7 / 44.1           777 rows,  4096 x 14336 94.7 / 89.4          1501 rows,  7168 x 8192 162.5 / 138.4 (pairs)
//  1100 rows,  4096 x 4096  52.1 / 41.0          9205 rows,  2048 x 8192 278.1 / 227.4 (no memory)
// Up to 128 rows they would hold rows that are not there, and K of no whole k-tiles is left to the first four: neither is looked at.
// Where the first four lose most: 129 rows, 16032 x 8192 65.9 / 78.8 / 77.1 | 65.9; 5000 rows, 2048 x 5120 95.5 / 95.5 / 109.6 | 95.5; 192 rows,
// 3072 x 2048 17.1 in all three | 14.0; 1100 rows, 8192 x 512 19.9 in all three | 16.4.
struct GemmTileCost {
  int a, bh, per_cu, pieces;   // (pieces: at most)
  float ktile, slope, cold, pair, pair_cold, fixed, store;
};
constexpr int GEMM_NTILES = 10, GEMM_TILES_ANY = 4;   // the first four take any K and any number of rows, see gemm_plan
constexpr int GEMM_ROWS64 = 3, GEMM_LONG = 9;
constexpr GemmTileCost GEMM_TILES[GEMM_NTILES] = {{8, 2, 1, 16, 1.2f, 0.0f, 0.0f, 0.0f, 0.0f, 4.35f, 4.43f},
                                                  {4, 2, 1, 16, 0.684f, 0.108f, 0.552f, 0.0f, 0.0f, 2.85f, 1.47f},
                                                  {4, 1, 2, 16, 0.504f, 0.0f, 0.262f, 0.874f, 1.25f, 3.18f, 0.166f},
                                                  {2, 1, 2, 16, 0.302f, 0.201f, 0.284f, 0.737f, 1.19f, 3.24f, 0.0f},
                                                  {7, 2, 1, 16, 1.098f, 0.0394f, 0.0f, 0.0f, 0.0f, 6.28f, 2.11f},
                                                  {6, 2, 1, 16, 0.953f, 0.0412f, 0.119f, 0.0f, 0.0f, 6.24f, 1.61f},
                                                  {5, 2, 1, 16, 0.668f, 0.2935f, 0.581f, 0.0f, 0.0f, 3.12f, 5.41f},
                                                  {5, 1, 2, 8, 0.553f, 0.0159f, 0.173f, 1.103f, 4.77f, 3.88f, 0.0077f},
                                                  {6, 1, 1, 16, 0.617f, 0.0f, 0.0944f, 0.0f, 0.0f, 4.28f, 0.0f},
                                                  {4, 1, 1, 16, 0.56f, 0.0508f, 0.08f, 0.0f, 0.0f, 5.0f, 0.101f}};
// The long rings' costs are fitted to 25 weights of the model families: 17 to 64 rows (92 products; what the plan takes is 0.6 % above the
// best of the pieces, 6 % at worst; with the ring of two's costs 1.7 and 17 %).  128 x 128's of 65 to 128 rows are fitted to 201 products of
// 72 weights, each against the best of the other tiles: with CUs to spare it is the slower one (8192 x 15360, 112 rows: 192 workgroups 66.6 us, 256 of
// the ring of two 56.9; 20480 x 5120 (pairs) 62.5 / 54.1, 6144 x 17920 64.3 / 56.0), which costs that fell with them did not see.
constexpr GemmTileCost GEMM_FEW_COST = {2, 1, 2, 16, 0.353f, 0.201f, 0.281f, 0.737f, 1.19f, 3.17f, 0.0f};
constexpr GemmTileCost GEMM_FEW8_COST = {2, 1, 2, 16, 0.547f, 0.201f, 0.242f, 0.8f, 1.405f, 1.78f, 0.0f};   // (64 products of 17 weights: 0.7 % above the best pieces)
// The same over rows a power of two apart, where all row distances meet the same channels and the tiles that do not turn are the slower ones (us, they /
// this one: 13312 x 16384 (pairs) 66 rows 115 / 90, 112 rows 117 / 98, 12288 x 4096 66 rows 29.4 / 27.5): fitted to 66 products beside 64 x 128
// and 128 x 128, 0.7 % above the best, 6 % at worst.
constexpr GemmTileCost GEMM_LONG_COST = {4, 1, 1, 16, 0.407f, 0.0508f, 0.206f, 0.0f, 0.0f, 5.0f, 0.101f};
static const GemmTileCost& gemm_cost(int tile, int M, int K) {
  if (tile == GEMM_LONG && (K & (K - 1)) == 0) return GEMM_LONG_COST;
  return tile == GEMM_ROWS64 && M <= 64 ? GEMM_FEW_COST : GEMM_TILES[tile];
}
// whether a tile serves the product
static bool gemm_takes(int tile, int M, int K) {
  if (tile < GEMM_TILES_ANY) return true;
  if (tile == GEMM_LONG) return M > 64 && M <= 128 && K % 64 == 0;
  return M > 128 && K % 64 == 0;
}
// and the two input projections of a block in one grid (K % 64 == 0): q/k/v beside up/gate of 1B, 128 rows, ring of two 29.5 us, of three 28.2,
// which the whole prompt of 128 tokens, 1050 us, does not show beyond the 1.5 % that two runs of it differ by.  Its output projections, cut so
// that every CU has a workgroup, are 64 x 128 there in 17.0 us and would be 18.0 with the long ring: they keep the first four.
static bool gemm_shares(int tile, int M, int K) { return (tile < GEMM_TILES_ANY || tile == GEMM_LONG) && gemm_takes(tile, M, K); }
constexpr size_t GEMM_SCRATCH = (size_t)64 << 20;   // pieces of one round of the largest tiles
constexpr int GEMM_SCRATCH_FROM = 33;               // rows from which a projection that has memory for pieces is one of this file's
// and from which the two grids of a decode step are, that hold a product beside the attention or another product: below, the
// bands of 16 rows leave room for the attention; those of 32 do not, and read their inputs at half the rate (us per step, up/gate, wo
// and w2 in bands / in these grids, q/k/v in bands: 70B rank shard, 17 rows 6565 / 5240, 32 rows 7020 / 5780; 8B, 17 rows 4190 / 3680,
// 32 rows 4530 / 3780; 1B, 24 rows at 1900 tokens 1371 / 1101)
constexpr int GEMM_BESIDE_FROM = 17;

constexpr float GEMM_WEIGHT_BYTES_US = 5.73e6f, GEMM_OUTPUT_BYTES_US = 6.98e6f, GEMM_SUM_US = 4.92f, GEMM_TRIP_US = 0.267f, GEMM_PIECE_BYTES_US = 3.83e6f,
                GEMM_TWO = 0.157f, GEMM_NORM_PIECE_US = 0.15f;

// `workgroups` of k k-tiles each, at the same time
static float gemm_round_us(const GemmTileCost& t, int M, int cus, int workgroups, int k) {
  const float busy = (float)workgroups / cus;
  const int TM = 32 * t.a;
  const float own = M <= TM ? 1.0f : M <= 2 * TM ? GEMM_TWO : 0.0f;   // how much a weight is one row tile's own
  return k * (busy > 1.0f ? t.pair + (t.pair_cold - t.pair) * own : t.ktile + busy * (t.slope + (t.cold - t.slope) * own));
}
// N outputs per row, of as many weight rows or twice as many
static float gemm_bytes_us(int M, int N, int K, int mode) {
  return (mode == GEMM_PAIR ? 2.0f : 1.0f) * N * K * 2 / GEMM_WEIGHT_BYTES_US + (float)M * N * 2 / GEMM_OUTPUT_BYTES_US;
}
// What more pieces cost whoever adds them, beside their bytes: a step for every four, as the norms take them.  (k_gemm_sum takes eight at a
// time; measured again with it, 1740 products are nearest their best with these steps and 4.92 us: 1.1 % above it from 129 rows on; steps of
// eight, of one or none, 3.5 to 5.3 us and other rates: 1.1 to 2.6 %.)
static int gemm_trips(int pieces) { return (pieces + 2) / 4; }
static float gemm_store_us(const GemmTileCost& t, int64_t tiles, int cus, int mode) {
  return t.store * (mode == GEMM_PAIR ? 0.5f : 1.0f) * tiles / cus;
}
static int gemm_cus() {
  const int cus = lr_num_cus();
  return cus > 0 ? cus : 256;
}

// the best of tile c's ways to compute a product of nk k-tiles, if it is better than `best`
static void gemm_consider(const GemmTileCost& t, int c, int M, int N, int nk, int mode, float bytes_us, size_t scratch, GemmPlan& best) {
  const int cus = gemm_cus(), TM = 32 * t.a, TN = (mode == GEMM_PAIR ? 64 : 128) * t.bh, slots = cus * t.per_cu;
  const int64_t tiles = (int64_t)((M + TM - 1) / TM) * ((N + TN - 1) / TN), rounds = tiles / slots;
  if (tiles > 0x3fffffff) return;
  const int left = (int)(tiles - rounds * slots);
  auto round_us = [&](int workgroups, int k) { return gemm_round_us(t, M, cus, workgroups, k); };
  auto consider = [&](float us, float more, int whole, int cut, int pieces) {
    us = (us > bytes_us ? us : bytes_us) + more + gemm_store_us(t, whole, cus, mode);
    if (best.tile < 0 || us < best.us) best = GemmPlan{c, whole, cut, pieces, us};
  };
  const float whole = rounds * round_us(slots, nk), fixed = (rounds + (left ? 1 : 0)) * t.fixed;
  consider(whole + (left ? round_us(left, nk) : 0.0f), fixed, (int)tiles, 0, 1);
  for (int s = 2; left && s <= t.pieces && 4 * s <= nk && left * s <= slots; ++s) {
    const size_t bytes = (size_t)left * s * (32 * t.a) * (128 * t.bh) * sizeof(float);
    if (bytes > scratch) break;
    consider(whole + round_us(left * s, (nk + s - 1) / s), fixed + GEMM_SUM_US + gemm_trips(s) * GEMM_TRIP_US + bytes / GEMM_PIECE_BYTES_US,
             (int)tiles - left, left, s);
  }
}
static GemmPlan gemm_plan(int M, int N, int K, int mode, size_t scratch) {
  GemmPlan best{-1, 0, 0, 1, 0.0f};
  if (M > 0x7fffffff - 256 || N > 0x7fffffff - 256 || K > 0x7fffffff - 256) return best;   // (row, column and k of the last tile are ints)
  const float bytes_us = gemm_bytes_us(M, N, K, mode);
  for (int c = 0; c < GEMM_NTILES; ++c)
    if (gemm_takes(c, M, K)) gemm_consider(gemm_cost(c, M, K), c, M, N, (K + 63) / 64, mode, bytes_us, scratch, best);
  return best;
}
// The same for e4m3 weights (K % 128 == 0): tiles of 64 x 128, k-tiles of 128.
static GemmPlan gemm_plan8(int M, int N, int K, int mode, size_t scratch) {
  GemmPlan best{-1, 0, 0, 1, 0.0f};
  if (M < GEMM_BESIDE_FROM || M > 64 || K % 128 || N > 0x7fffffff - 256) return best;
  gemm_consider(GEMM_FEW8_COST, GEMM_ROWS64, M, N, K / 128, mode, gemm_bytes_us(M, N, K / 2, mode), scratch, best);
  return best;
}

template <int A, int BH, bool KTAIL, int MODE, bool NT = false, int R = 2, bool W8 = false>
static int gemm_run_as(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K, const GemmRope& rp,
                       const GemmPlan& p, void* scratch, hipStream_t s, const void* scales = nullptr) {
  using T = GemmTile<A, BH, R, W8>;
  static std::atomic<unsigned long long> raised{0};
  if (!lr_raise_lds_limit(reinterpret_cast<const void*>(&k_gemm_dma<A, BH, KTAIL, MODE, false, NT, R, W8>), T::LDS, raised)) return LR_E_LAUNCH;
  const int gn = MODE == GEMM_PAIR ? T::TN / 2 : T::TN, tm = (M + T::TM - 1) / T::TM, tn = (N + gn - 1) / gn;
  const GemmSplit sp{(float*)scratch, p.full, p.rem, p.splits, (const u16*)scales};
  k_gemm_dma<A, BH, KTAIL, MODE, false, NT, R, W8><<<dim3((unsigned)(p.full + p.rem * p.splits)), dim3(256), T::LDS, s>>>(
      (const u16*)x, ldx, (const u16*)w, (u16*)y, ldy, M, N, K, tm, tn, rp, sp, GemmGroup{});
  if constexpr (MODE != GEMM_ROWS)
    if (p.rem) k_gemm_sum<A, BH, MODE><<<dim3((unsigned)(p.rem * A * 4)), dim3(256), 0, s>>>((u16*)y, ldy, M, N, tm, tn, rp, sp);
  return lr_launch_status();
}
template <int A, int BH, bool KTAIL, bool NT = false, int R = 2>
static int gemm_run_mode(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K, int mode, const GemmRope& rp,
                         const GemmPlan& p, void* scratch, hipStream_t s) {
  if (mode == GEMM_PAIR) return gemm_run_as<A, BH, KTAIL, GEMM_PAIR, NT, R>(x, ldx, w, y, ldy, M, N, K, rp, p, scratch, s);
  if (mode == GEMM_ROPE) return gemm_run_as<A, BH, KTAIL, GEMM_ROPE, NT, R>(x, ldx, w, y, ldy, M, N, K, rp, p, scratch, s);
  if (mode == GEMM_ROWS) return gemm_run_as<A, BH, KTAIL, GEMM_ROWS, NT, R>(x, ldx, w, y, ldy, M, N, K, rp, p, scratch, s);
  return gemm_run_as<A, BH, KTAIL, GEMM_PLAIN, NT, R>(x, ldx, w, y, ldy, M, N, K, rp, p, scratch, s);
}
static int gemm_run(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K, int mode, const GemmRope& rp,
                    const GemmPlan& p, void* scratch, hipStream_t s) {
  const bool kt = K % 64 != 0;
  if (p.tile == 0)
    return kt ? gemm_run_mode<8, 2, true>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s)
              : gemm_run_mode<8, 2, false>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
  if (p.tile == 1)
    return kt ? gemm_run_mode<4, 2, true>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s)
              : gemm_run_mode<4, 2, false>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
  if (p.tile == 2)
    return kt ? gemm_run_mode<4, 1, true>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s)
              : gemm_run_mode<4, 1, false>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
  if (p.tile == 4) return gemm_run_mode<7, 2, false>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
  if (p.tile == 5) return gemm_run_mode<6, 2, false>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
  if (p.tile == 6) return gemm_run_mode<5, 2, false>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
  if (p.tile == 7) return gemm_run_mode<5, 1, false>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
  if (p.tile == 8) return gemm_run_mode<6, 1, false>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
  if (p.tile == GEMM_LONG) return gemm_run_mode<4, 1, false, false, GEMM_RING>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
  if (M <= 64)   // every weight is used once: non-temporal (28672 x 4096 at 64 rows 50.0 -> 46.7 us, 16032 x 8192 61.9 -> 57.5)
    return kt ? gemm_run_mode<2, 1, true, true, GEMM_RING>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s)
              : gemm_run_mode<2, 1, false, true, GEMM_RING>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
  return kt ? gemm_run_mode<2, 1, true>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s)
            : gemm_run_mode<2, 1, false>(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
}
// whether a tile's rows lie within the 2 GiB that an offset of a request reaches (N: pairs in PAIR mode)
static bool gemm_reaches(int64_t ldx, int N, int K, int mode) {
  return 256 * ldx * 2 < 0x7fffffff && ((mode == GEMM_PAIR ? (int64_t)N : 0) + 256) * K * 2 < 0x7fffffff;
}
static int gemm(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K, int mode, const GemmRope& rp, void* scratch,
                size_t scratch_bytes, hipStream_t s) {
  if (!gemm_reaches(ldx, N, K, mode)) return LR_E_UNSUPPORTED;
  const GemmPlan p = gemm_plan(M, N, K, mode, scratch == nullptr || lr_misaligned(scratch) ? 0 : scratch_bytes);
  if (p.tile < 0) return LR_E_UNSUPPORTED;
  return gemm_run(x, ldx, w, y, ldy, M, N, K, mode, rp, p, scratch, s);
}

// ---- two products of one grid, and products whose partial sums stay
static GemmProduct gemm_product(int tile, int mode, const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K) {
  const GemmTileCost& t = GEMM_TILES[tile];
  const int TM = 32 * t.a, TN = (mode == GEMM_PAIR ? 64 : 128) * t.bh;
  GemmProduct p = {(const u16*)x, ldx, (const u16*)w, (u16*)y, ldy, M, N, K, (M + TM - 1) / TM, (N + TN - 1) / TN, GemmSplit{}};
  p.sp.full = p.tm * p.tn;
  p.sp.splits = 1;
  return p;
}
template <int A, int BH, int MODE0, int MODE1, bool NT, int R = 2, bool W8 = false>
static int gemm_two_as(const GemmProduct& a, const GemmProduct& b, const GemmRope& rp, hipStream_t s) {
  using T = GemmTile<A, BH, R, W8>;
  static std::atomic<unsigned long long> raised{0};
  if (!lr_raise_lds_limit(reinterpret_cast<const void*>(&k_gemm_two<A, BH, MODE0, MODE1, NT, R, W8>), T::LDS, raised)) return LR_E_LAUNCH;
  const int n0 = a.sp.full + a.sp.rem * a.sp.splits, n1 = b.sp.full + b.sp.rem * b.sp.splits;
  k_gemm_two<A, BH, MODE0, MODE1, NT, R, W8><<<dim3((unsigned)(n0 + n1)), dim3(256), T::LDS, s>>>(a, b, n0, rp);
  return lr_launch_status();
}
template <int MODE0, int MODE1>
static int gemm_two(int tile, const GemmProduct& a, const GemmProduct& b, const GemmRope& rp, hipStream_t s) {
  if (tile == 0) return gemm_two_as<8, 2, MODE0, MODE1, false>(a, b, rp, s);
  if (tile == 1) return gemm_two_as<4, 2, MODE0, MODE1, false>(a, b, rp, s);
  if (tile == 2) return gemm_two_as<4, 1, MODE0, MODE1, false>(a, b, rp, s);
  if (tile == GEMM_LONG) return gemm_two_as<4, 1, MODE0, MODE1, false, GEMM_RING>(a, b, rp, s);
  return a.M <= 64 ? gemm_two_as<2, 1, MODE0, MODE1, true, GEMM_RING>(a, b, rp, s) : gemm_two_as<2, 1, MODE0, MODE1, false>(a, b, rp, s);
}

namespace lr_detail {
// The q/k/v projection of x0 (rotated and cached on its way out) and the up/gate projection of x1 (activated), M rows, in one
// launch where that should take less than the two (the plan's costs decide); LR_E_UNSUPPORTED, nothing launched, otherwise.
int gemm_inputs(const void* x0, const void* wqkv, void* qkv, int S, const lr_rope_kv_t* rope, const void* x1, const void* w1, void* act,
                int I, int M, int K, size_t sums_bytes, hipStream_t s) {
  const int N = (rope->n_head + 2 * rope->n_kv_head) * rope->head_dim, cus = gemm_cus(), nk = (K + 63) / 64;
  if (K % 64 || !gemm_reaches(K, N, K, GEMM_ROPE) || !gemm_reaches(K, I, K, GEMM_PAIR)) return LR_E_UNSUPPORTED;
  const GemmPlan p0 = gemm_plan(M, N, K, GEMM_ROPE, sums_bytes), p1 = gemm_plan(M, I, K, GEMM_PAIR, sums_bytes);
  if (p0.tile < 0 || p1.tile < 0) return LR_E_UNSUPPORTED;
  const float bytes_us = gemm_bytes_us(M, N, K, GEMM_ROPE) + gemm_bytes_us(M, I, K, GEMM_PAIR);
  float best_us = p0.us + p1.us;
  int best = -1;
  for (int c = 0; c < GEMM_NTILES; ++c) {
    if (!gemm_shares(c, M, K)) continue;
    const GemmTileCost& t = gemm_cost(c, M, K);
    const int TM = 32 * t.a, slots = cus * t.per_cu;
    const int64_t tm = (M - 1) / TM + 1, tiles0 = tm * ((N - 1) / (128 * t.bh) + 1), tiles1 = tm * ((I - 1) / (64 * t.bh) + 1), tiles = tiles0 + tiles1;
    // (of several rounds only the last one leaves room, and q/k/v goes cold before the attention reads it: 8 x 2048 tokens of
    // the 8B model, in one grid 185.4 ms, apart 183.2)
    if (tiles > slots) continue;
    float us = gemm_round_us(t, M, cus, (int)tiles, nk);
    us = (us > bytes_us ? us : bytes_us) + t.fixed + gemm_store_us(t, tiles0, cus, GEMM_ROPE) + gemm_store_us(t, tiles1, cus, GEMM_PAIR);
    if (us < best_us) {
      best_us = us;
      best = c;
    }
  }
  if (best < 0) return LR_E_UNSUPPORTED;
  const GemmRope rp{(const u16*)rope->table, rope->pos, (u16*)rope->k_cache, (u16*)rope->v_cache, rope->err, S, rope->n_head,
                    rope->n_kv_head, rope->head_dim, rope->smax, rope->block_size};
  return gemm_two<GEMM_ROPE, GEMM_PAIR>(best, gemm_product(best, GEMM_ROPE, x0, K, wqkv, qkv, N, M, N, K),
                                        gemm_product(best, GEMM_PAIR, x1, K, w1, act, I, M, I, K), rp, s);
}

template <int HD, int G, int GROUPS, bool W8>
static int attn_beside_gemm(const AttnItems& a, const GemmProduct& p, hipStream_t s) {
  using T = GemmTile<2, 1, W8 ? 2 : GEMM_RING, W8>;
  const size_t att = (size_t)attn_item_lds_floats<HD, G>(a.chunk_max) * sizeof(float), lds = att > T::LDS ? att : T::LDS;
  static std::atomic<unsigned long long> raised{0};
  if (!lr_raise_lds_limit(reinterpret_cast<const void*>(&k_attn_beside_gemm<HD, G, GROUPS, W8>), lds, raised)) return LR_E_LAUNCH;
  const int n = p.sp.full + p.sp.rem * p.sp.splits;
  k_attn_beside_gemm<HD, G, GROUPS, W8><<<dim3((unsigned)(n + a.n_items + a.mergers())), dim3(256), lds, s>>>(a, p, n);
  if (p.sp.rem)
    k_gemm_sum<2, 1, GEMM_PAIR><<<dim3((unsigned)(p.sp.rem * 2 * 4)), dim3(256), 0, s>>>(p.y, p.ldy, p.M, p.N, p.tm, p.tn, GemmRope{}, p.sp);
  return lr_launch_status();
}
// lr_attn_decode_beside_product, arguments checked; LR_E_UNSUPPORTED, nothing launched, where the product is none of 64-row tiles.
// scales: of e4m3 weights.
template <bool W8>
int gemm_beside_attention(const AttnItems& a, int hd, int G, const void* x, int64_t ldx, const void* w, const void* scales, void* y, int64_t ldy,
                          int M, int I, int K, void* sums, size_t sums_bytes, hipStream_t s) {
  if (M < GEMM_BESIDE_FROM || M > 64 || K % (W8 ? 128 : 64) || !gemm_reaches(ldx, I, K, GEMM_PAIR)) return LR_E_UNSUPPORTED;
  auto planned = [&](size_t bytes) { return W8 ? gemm_plan8(M, I, K, GEMM_PAIR, bytes) : gemm_plan(M, I, K, GEMM_PAIR, bytes); };
  GemmPlan plan = planned(sums_bytes);
  // Of two numbers of pieces that take a product alone as long the smaller: what it leaves is the attention's (70B rank shard, 17 to 24 rows,
  // three pieces or four, a product alone 30.9 us: 24 layers 1629 to 1677 and 1662 to 1711 us).
  for (const float best = plan.us; plan.tile == GEMM_ROWS64 && plan.rem;) {
    const GemmPlan fewer = planned((size_t)plan.rem * plan.splits * GemmTile<2, 1>::TM * GemmTile<2, 1>::TN * sizeof(float) - 1);
    if (fewer.tile != GEMM_ROWS64 || fewer.us > 1.003f * best) break;
    plan = fewer;
  }
  if (plan.tile != GEMM_ROWS64) return LR_E_UNSUPPORTED;
  GemmProduct p = gemm_product(GEMM_ROWS64, GEMM_PAIR, x, ldx, w, y, ldy, M, I, K);
  p.sp = GemmSplit{(float*)sums, plan.full, plan.rem, plan.splits, (const u16*)scales};
  const bool two = attn_two_groups(a.chunk_max);
#define LR_PRODUCT(HDV, GV) \
  if (hd == HDV && G == GV) return two ? attn_beside_gemm<HDV, GV, 2, W8>(a, p, s) : attn_beside_gemm<HDV, GV, 4, W8>(a, p, s);
  LR_PRODUCT(128, 1) LR_PRODUCT(128, 2) LR_PRODUCT(128, 4) LR_PRODUCT(128, 8)
  LR_PRODUCT(64, 1) LR_PRODUCT(64, 2) LR_PRODUCT(64, 4) LR_PRODUCT(64, 8)
#undef LR_PRODUCT
  return LR_E_UNSUPPORTED;
}

// x w^T as partial sums [pieces][M][N] in `sums`; LR_E_UNSUPPORTED, nothing launched, where a product of this shape has whole tiles
int gemm_pieces(const void* x, int64_t ldx, const void* w, int M, int N, int K, void* sums, size_t sums_bytes, int* pieces, hipStream_t s) {
  if (M < GEMM_SCRATCH_FROM || sums == nullptr || lr_misaligned(sums) || N % 4 || !gemm_reaches(ldx, N, K, GEMM_PLAIN)) return LR_E_UNSUPPORTED;
  const GemmPlan p = gemm_plan(M, N, K, GEMM_PLAIN, sums_bytes);
  if (p.tile < 0 || p.full || !p.rem) return LR_E_UNSUPPORTED;
  *pieces = p.splits;   // (less memory than the plan's own pieces, which have their tiles' absent rows and columns)
  return gemm_run(x, ldx, w, nullptr, 0, M, N, K, GEMM_ROWS, GemmRope{}, p, sums, s);
}

// Two such products of N columns each in one launch, pieces of about the same length, where that should take less than the two.
// (GEMM_NORM_PIECE_US: the norms add a row per workgroup, slower than k_gemm_sum.  With it 128 rows of the 1B model keep eight pieces in tiles of 64
// rows, a prompt 1059 us; ten in tiles of 128, 1063.)
struct GemmOutputs {
  int tile, s0, s1;   // tile -1: the two are faster
};
template <bool W8 = false>
static GemmOutputs outputs_plan(int M, int N, int K0, int K1, size_t sums_bytes) {
  constexpr int KT = W8 ? 128 : 64;
  GemmOutputs best{-1, 1, 1};
  if (N % 4 || K0 % KT || K1 % KT || !gemm_reaches(K0, N, K0, GEMM_PLAIN) || !gemm_reaches(K1, N, K1, GEMM_PLAIN)) return best;
  auto planned = [&](int K) { return W8 ? gemm_plan8(M, N, K, GEMM_PLAIN, sums_bytes) : gemm_plan(M, N, K, GEMM_PLAIN, sums_bytes); };
  const GemmPlan p0 = planned(K0), p1 = planned(K1);
  if (p0.tile < 0 || p1.tile < 0) return best;
  const float bytes_us = gemm_bytes_us(M, N, W8 ? K0 / 2 : K0, GEMM_ROWS) + gemm_bytes_us(M, N, W8 ? K1 / 2 : K1, GEMM_ROWS);
  auto alone = [](const GemmPlan& p) { return p.us - (p.rem && !p.full ? GEMM_SUM_US : 0.0f); };   // (its sum would be the norms' too)
  float best_us = W8 ? 1e30f : alone(p0) + alone(p1);   // (e4m3: there is no other way to leave pieces)
  const int cus = gemm_cus(), pairs0 = (K0 / KT + 1) / 2, pairs1 = (K1 / KT + 1) / 2;
  const size_t row = (size_t)M * N * sizeof(float);
  for (int c = W8 ? GEMM_ROWS64 : 0; c < GEMM_TILES_ANY; ++c) {
    const GemmTileCost& t = W8 ? GEMM_FEW8_COST : gemm_cost(c, M, K0);
    const int TM = 32 * t.a, TN = 128 * t.bh, slots = cus * t.per_cu;
    const int64_t tiles = (int64_t)((M + TM - 1) / TM) * ((N + TN - 1) / TN);
    for (int s0 = 1; s0 <= 16 && 2 * s0 <= pairs0 + 1 && row * s0 <= sums_bytes; ++s0)
      for (int s1 = 1; s1 <= 16 && 2 * s1 <= pairs1 + 1 && row * s1 <= sums_bytes && tiles * (s0 + s1) <= slots; ++s1) {
        const int k0 = 2 * ((pairs0 + s0 - 1) / s0), k1 = 2 * ((pairs1 + s1 - 1) / s1);
        float us = gemm_round_us(t, M, cus, (int)tiles * (s0 + s1), k0 > k1 ? k0 : k1);
        us = (us > bytes_us ? us : bytes_us) + t.fixed + (gemm_trips(s0) + gemm_trips(s1)) * GEMM_TRIP_US + row * (s0 + s1) / GEMM_PIECE_BYTES_US + (s0 + s1) * GEMM_NORM_PIECE_US;
        if (us < best_us) {
          best_us = us;
          best = GemmOutputs{c, s0, s1};
        }
      }
  }
  return best;
}
// Bytes for either of the two with which the plan is that of all the memory it could ask for; 0: two launches.
template <bool W8>
static size_t outputs_bytes(int M, int N, int K0, int K1) {
  const GemmOutputs p = M < GEMM_BESIDE_FROM ? GemmOutputs{-1, 1, 1} : outputs_plan<W8>(M, N, K0, K1, GEMM_SCRATCH);
  return p.tile < 0 ? 0 : (size_t)M * N * sizeof(float) * (p.s0 > p.s1 ? p.s0 : p.s1);
}
bool gemm_outputs_pay(int M, int N, int K0, int K1, size_t sums_bytes) {
  return M >= GEMM_SCRATCH_FROM && outputs_plan<>(M, N, K0, K1, sums_bytes).tile >= 0;
}
int gemm_outputs(const void* x0, const void* w0, int K0, void* sums0, int* pieces0, const void* x1, const void* w1, int K1, void* sums1, int* pieces1,
                 int M, int N, size_t sums_bytes, hipStream_t s) {
  if (lr_misaligned(sums0) || lr_misaligned(sums1)) return LR_E_ALIGN;
  if (M < GEMM_BESIDE_FROM) return LR_E_UNSUPPORTED;
  const GemmOutputs p = outputs_plan<>(M, N, K0, K1, sums_bytes);
  if (p.tile < 0) return LR_E_UNSUPPORTED;
  GemmProduct a = gemm_product(p.tile, GEMM_ROWS, x0, K0, w0, nullptr, 0, M, N, K0), b = gemm_product(p.tile, GEMM_ROWS, x1, K1, w1, nullptr, 0, M, N, K1);
  a.sp = GemmSplit{(float*)sums0, 0, a.sp.full, p.s0};
  b.sp = GemmSplit{(float*)sums1, 0, b.sp.full, p.s1};
  *pieces0 = p.s0;
  *pieces1 = p.s1;
  return gemm_two<GEMM_ROWS, GEMM_ROWS>(p.tile, a, b, GemmRope{}, s);
}
// The same of e4m3 weights; there is no other way to leave their pieces.
static int gemm_outputs8(const void* x0, const void* w0, const void* scales0, int K0, void* sums0, int* pieces0, const void* x1, const void* w1,
                         const void* scales1, int K1, void* sums1, int* pieces1, int M, int N, size_t sums_bytes, hipStream_t s) {
  if (lr_misaligned(sums0) || lr_misaligned(sums1)) return LR_E_ALIGN;
  const GemmOutputs p = outputs_plan<true>(M, N, K0, K1, sums_bytes);
  if (p.tile < 0) return LR_E_UNSUPPORTED;
  GemmProduct a = gemm_product(GEMM_ROWS64, GEMM_ROWS, x0, K0, w0, nullptr, 0, M, N, K0), b = gemm_product(GEMM_ROWS64, GEMM_ROWS, x1, K1, w1, nullptr, 0, M, N, K1);
  a.sp = GemmSplit{(float*)sums0, 0, a.sp.full, p.s0, (const u16*)scales0};
  b.sp = GemmSplit{(float*)sums1, 0, b.sp.full, p.s1, (const u16*)scales1};
  *pieces0 = p.s0;
  *pieces1 = p.s1;
  return gemm_two_as<2, 1, GEMM_ROWS, GEMM_ROWS, true, 2, true>(a, b, GemmRope{}, s);
}
}  // namespace lr_detail

// Grouped products (lr_moe): rows of several matrices' tiles, see GemmGroup; pair_off != 0: GEMM_PAIR (N counts pairs).
// tile_rows: the height the tile table was made for (grouped_rows): 128 or 160 (K % 64 == 0) with 128 columns, the latter's pairs with
// 256 where that leaves no half of a tile without columns, or 256 x 256.
static int grouped_pairs_bh(int tile_rows, int I) { return tile_rows == 128 || (tile_rows == 160 && (I + 63) / 64 % 2) ? 1 : 2; }
// what one of the two takes whose row tiles are `tiles` of `rows` rows of an expert
static float grouped_us(int a, int bh, float tiles, int rows, int N, int K, int mode) {
  const GemmTileCost* t = nullptr;
  for (const GemmTileCost& c : GEMM_TILES)
    if (t == nullptr && c.a == a && c.bh == bh) t = &c;
  const int cus = gemm_cus(), gn = (mode == GEMM_PAIR ? 64 : 128) * bh, nk = (K + 63) / 64;
  const float workgroups = tiles * ((N + gn - 1) / gn), slots = (float)cus * t->per_cu, rounds = floorf(workgroups / slots), left = workgroups - rounds * slots;
  float us = rounds * (gemm_round_us(*t, rows, cus, (int)slots, nk) + t->fixed);
  if (left > 0.0f) us += gemm_round_us(*t, rows, cus, (int)left, nk) + t->fixed;
  return us + t->store * (mode == GEMM_PAIR ? 0.5f : 1.0f) * workgroups / cus;
}
namespace lr_detail {
// Height of the tiles for n rows of `experts` that are taken: what the costs of GEMM_TILES give both products, an expert ending in half a
// tile on average.  The factors are fitted to 47 mixtures of 8 to 64 experts, 500 to 16384 tokens, even and skewed choices, where the
// height taken is then 1.1 % above the best (13 % at worst; without them 2.2 and 17 %; 256 wherever an expert has as many rows and 128
// below, as it was, 6.7 and 29 %).  us of the whole mixture, before / now (the empty tiles' place included, see gemm_tile): 32 experts,
// 6 chosen, 384 x 4096: 500 tokens 145 / 111, 2500 309 / 198, 3002 316 / 258, 6000 512 / 421, 8192 582 / 582; 16 experts, 4 chosen, 448 x 2048:
// 1000 63 / 53, 5000 181 / 141, 16384 477 / 438.
int grouped_rows(int64_t n, int experts, int I, int D) {
  const float rows = (float)n / experts;
  auto us = [&](int h) {
    const float tiles = (float)n / h + 0.5f * experts;
    const int r = rows < 1.0f ? 1 : (int)rows, a = h / 32;
    return grouped_us(a, grouped_pairs_bh(h, I), tiles, r, I, D, GEMM_PAIR) + grouped_us(a, h == 256 ? 2 : 1, tiles, r, D, I, GEMM_PLAIN);
  };
  const float u128 = 1.1f * us(128), u160 = I % 64 || D % 64 ? 1e30f : 0.95f * us(160), u256 = us(256);
  return u160 < u128 && u160 < u256 ? 160 : u128 < u256 ? 128 : 256;
}
template <int A, int BH, bool KTAIL, int MODE>
static int gemm_grouped_as(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int N, int K, const GemmGroup& gp, int max_tiles,
                           hipStream_t s) {
  using T = GemmTile<A, BH>;
  constexpr size_t lds = T::LDS + T::TM * sizeof(int32_t);
  static std::atomic<unsigned long long> raised{0};
  if (!lr_raise_lds_limit(reinterpret_cast<const void*>(&k_gemm_dma<A, BH, KTAIL, MODE, true>), lds, raised)) return LR_E_LAUNCH;
  const int gn = MODE == GEMM_PAIR ? T::TN / 2 : T::TN, tn = (N + gn - 1) / gn;
  k_gemm_dma<A, BH, KTAIL, MODE, true><<<dim3((unsigned)(max_tiles * tn)), dim3(256), lds, s>>>(
      (const u16*)x, ldx, (const u16*)w, (u16*)y, ldy, T::TM, N, K, max_tiles, tn, GemmRope{}, GemmSplit{}, gp);
  return lr_launch_status();
}
int gemm_grouped(const void* x, int64_t ldx, int64_t xrows, const void* w, void* y, int64_t ldy, int N, int K, int pair_off, int64_t wstride,
                 const int32_t* tiles, const int32_t* ntiles, const int32_t* entries, int xdiv, int max_tiles, int tile_rows, hipStream_t s) {
  if (xrows * ldx * 2 >= 0x7fffffff || ((int64_t)pair_off + 256) * K * 2 >= 0x7fffffff) return LR_E_UNSUPPORTED;
  const GemmGroup gp = {tiles, ntiles, entries, xdiv, wstride, xrows};
  const bool kt = K % 64 != 0;
  if (tile_rows == 160) {
    if (kt) return LR_E_UNSUPPORTED;
    if (!pair_off) return gemm_grouped_as<5, 1, false, GEMM_PLAIN>(x, ldx, w, y, ldy, N, K, gp, max_tiles, s);
    return grouped_pairs_bh(tile_rows, N) == 1 ? gemm_grouped_as<5, 1, false, GEMM_PAIR>(x, ldx, w, y, ldy, N, K, gp, max_tiles, s)
                                               : gemm_grouped_as<5, 2, false, GEMM_PAIR>(x, ldx, w, y, ldy, N, K, gp, max_tiles, s);
  }
  if (tile_rows == 128) {
    if (pair_off)
      return kt ? gemm_grouped_as<4, 1, true, GEMM_PAIR>(x, ldx, w, y, ldy, N, K, gp, max_tiles, s)
                : gemm_grouped_as<4, 1, false, GEMM_PAIR>(x, ldx, w, y, ldy, N, K, gp, max_tiles, s);
    return kt ? gemm_grouped_as<4, 1, true, GEMM_PLAIN>(x, ldx, w, y, ldy, N, K, gp, max_tiles, s)
              : gemm_grouped_as<4, 1, false, GEMM_PLAIN>(x, ldx, w, y, ldy, N, K, gp, max_tiles, s);
  }
  if (pair_off)
    return kt ? gemm_grouped_as<8, 2, true, GEMM_PAIR>(x, ldx, w, y, ldy, N, K, gp, max_tiles, s)
              : gemm_grouped_as<8, 2, false, GEMM_PAIR>(x, ldx, w, y, ldy, N, K, gp, max_tiles, s);
  return kt ? gemm_grouped_as<8, 2, true, GEMM_PLAIN>(x, ldx, w, y, ldy, N, K, gp, max_tiles, s)
            : gemm_grouped_as<8, 2, false, GEMM_PLAIN>(x, ldx, w, y, ldy, N, K, gp, max_tiles, s);
}
}  // namespace lr_detail

static int linear_rows(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K, int act_swiglu, int gemv_cfg,
                       void* scratch, size_t scratch_bytes, hipStream_t s) {
  LR_REQUIRE_PTR(x);
  LR_REQUIRE_PTR(w);
  LR_REQUIRE_PTR(y);
  if (M <= 0 || N <= 0 || K <= 0) return LR_E_SHAPE;
  if (ldx < (act_swiglu ? 2 : 1) * (int64_t)K || ldy < N) return LR_E_SHAPE;
  if (K % 8 || ldx % 8) return LR_E_ALIGN;
  if (M <= 4 || ((act_swiglu || gemv_cfg) && M <= 8))
    return lr_gemv_dispatch(x, ldx, w, y, ldy, M, N, K, act_swiglu, gemv_cfg, s);
  if (!act_swiglu && M <= 64 && !(M >= GEMM_SCRATCH_FROM && scratch && gemm_reaches(ldx, N, K, GEMM_PLAIN))) {
    // decode batches: the weight-streaming matrix-core kernel (stream_gemm.hip); shapes it declines fall through
    lr_projection_t pr;
    pr.x = x; pr.ldx = ldx; pr.w = w; pr.y = y; pr.ldy = ldy; pr.N = N; pr.K = K; pr.epilogue = LR_EPI_NONE; pr.rope = nullptr;
    const int rc = lr_linear_multi(&pr, 1, M, s);
    if (rc != LR_E_UNSUPPORTED) return rc;
  }
  if (!act_swiglu) {
    const int rc = gemm(x, ldx, w, y, ldy, M, N, K, GEMM_PLAIN, GemmRope{}, scratch, scratch_bytes, s);
    if (rc != LR_E_UNSUPPORTED) return rc;
  }
  const dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
  if (grid.y > 65535) return LR_E_UNSUPPORTED;
  if (act_swiglu)
    k_gemm<true><<<grid, dim3(256), 0, s>>>((const u16*)x, ldx, (const u16*)w, (u16*)y, ldy, M, N, K);
  else
    k_gemm<false><<<grid, dim3(256), 0, s>>>((const u16*)x, ldx, (const u16*)w, (u16*)y, ldy, M, N, K);
  return lr_launch_status();
}

extern "C" int lr_linear_tuned(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K,
                               int act_swiglu, int gemv_cfg, lr_stream_t stream) {
  return linear_rows(x, ldx, w, y, ldy, M, N, K, act_swiglu, gemv_cfg, nullptr, 0, (hipStream_t)stream);
}

extern "C" int lr_linear(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K,
                         int act_swiglu, lr_stream_t stream) {
  return linear_rows(x, ldx, w, y, ldy, M, N, K, act_swiglu, 0, nullptr, 0, (hipStream_t)stream);
}

extern "C" size_t lr_linear_scratch_bytes(int M) { return M >= GEMM_SCRATCH_FROM ? GEMM_SCRATCH : 0; }

extern "C" int lr_linear_plan(int M, int N, int K, int pair, size_t scratch_bytes, lr_linear_plan_t* plan) {
  if (plan == nullptr) return LR_E_NULL;
  if (M <= 0 || N <= 0 || K <= 0 || (pair && N % 2)) return LR_E_SHAPE;
  if (K % 8) return LR_E_ALIGN;
  const GemmPlan p = gemm_plan(M, pair ? N / 2 : N, K, pair ? GEMM_PAIR : GEMM_PLAIN, scratch_bytes);
  if (p.tile < 0) return LR_E_UNSUPPORTED;
  plan->tile_rows = 32 * GEMM_TILES[p.tile].a;
  plan->tile_cols = 128 * GEMM_TILES[p.tile].bh;
  plan->whole = p.full;
  plan->cut = p.rem;
  plan->pieces = p.splits;
  plan->sums_bytes = p.rem ? (size_t)p.rem * p.splits * plan->tile_rows * plan->tile_cols * sizeof(float) : 0;
  return LR_OK;
}

extern "C" float lr_linear_plan_us(int M, int N, int K, int pair, size_t scratch_bytes) {
  if (M <= 0 || N <= 0 || K <= 0 || (pair && N % 2) || K % 8) return 0.0f;
  const GemmPlan p = gemm_plan(M, pair ? N / 2 : N, K, pair ? GEMM_PAIR : GEMM_PLAIN, scratch_bytes);
  return p.tile < 0 ? 0.0f : p.us;
}

extern "C" int lr_linear_scratch(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K, void* scratch,
                                 size_t scratch_bytes, lr_stream_t stream) {
  LR_OPTIONAL_PTR(scratch);
  return linear_rows(x, ldx, w, y, ldy, M, N, K, 0, 0, scratch, scratch_bytes, (hipStream_t)stream);
}

extern "C" int lr_linear_pieces(const void* x, int64_t ldx, const void* w, int M, int N, int K, void* sums, size_t sums_bytes, int32_t* pieces,
                                lr_stream_t stream) {
  LR_REQUIRE_PTR(x);
  LR_REQUIRE_PTR(w);
  LR_REQUIRE_PTR(sums);
  if (pieces == nullptr) return LR_E_NULL;
  if (M <= 0 || N <= 0 || K <= 0 || ldx < K) return LR_E_SHAPE;
  if (K % 8 || ldx % 8) return LR_E_ALIGN;
  return lr_detail::gemm_pieces(x, ldx, w, M, N, K, sums, sums_bytes, pieces, (hipStream_t)stream);
}

// The fused q/k/v projection of M = B * S rows (S tokens per sequence, row b * S + s at position pos[s]) finished as
// lr_rope_kv_write would finish it, in the GEMM's output pass; decode batches without scratch (and rows out of the requests'
// reach) in the two calls.
extern "C" int lr_linear_rope_kv_scratch(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int K, int S,
                                         const lr_rope_kv_t* rope, void* scratch, size_t scratch_bytes, lr_stream_t stream) {
  LR_REQUIRE_PTR(x);
  LR_REQUIRE_PTR(w);
  LR_REQUIRE_PTR(y);
  LR_OPTIONAL_PTR(scratch);
  if (rope == nullptr || rope->pos == nullptr) return LR_E_NULL;
  LR_REQUIRE_PTR(rope->table);
  LR_REQUIRE_PTR(rope->k_cache);
  LR_REQUIRE_PTR(rope->v_cache);
  if (M <= 0 || K <= 0 || S <= 0 || M % S) return LR_E_SHAPE;
  if (rope->n_head <= 0 || rope->n_kv_head <= 0 || rope->head_dim <= 0 || rope->smax <= 0 || rope->block_size <= 0)
    return LR_E_SHAPE;
  const int64_t n64 = (int64_t)(rope->n_head + 2 * rope->n_kv_head) * rope->head_dim;
  if (n64 > 0x7fffffff || ldx < K || ldy < n64) return LR_E_SHAPE;
  if (K % 8 || ldx % 8 || ldy % 8 || rope->head_dim % 8) return LR_E_ALIGN;
  const int N = (int)n64;
  hipStream_t s = (hipStream_t)stream;
  if (M > 64 || (M >= GEMM_SCRATCH_FROM && scratch)) {
    const GemmRope rp{(const u16*)rope->table, rope->pos, (u16*)rope->k_cache, (u16*)rope->v_cache, rope->err, S, rope->n_head,
                      rope->n_kv_head, rope->head_dim, rope->smax, rope->block_size};
    const int rc = gemm(x, ldx, w, y, ldy, M, N, K, GEMM_ROPE, rp, scratch, scratch_bytes, s);
    if (rc != LR_E_UNSUPPORTED) return rc;
  }
  const int rc = linear_rows(x, ldx, w, y, ldy, M, N, K, 0, 0, scratch, scratch_bytes, s);
  if (rc != LR_OK) return rc;
  return lr_rope_kv_write(y, ldy, rope->table, 0, rope->pos, rope->k_cache, rope->v_cache, M / S, S, rope->n_head,
                          rope->n_kv_head, rope->head_dim, rope->smax, rope->block_size, rope->err, stream);
}

extern "C" int lr_linear_rope_kv(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int K, int S,
                                 const lr_rope_kv_t* rope, lr_stream_t stream) {
  return lr_linear_rope_kv_scratch(x, ldx, w, y, ldy, M, K, S, rope, nullptr, 0, stream);
}

// y[M, I] = bf16( bf16(silu(g)) * u ) for [u | g] = x w^T with w = [up; gate] rows (N = 2 I): the MLP's first
// projection with the activation applied on the way out (utils.py:145-148 without the [M, 2 I] tensor).
extern "C" int lr_linear_swiglu_out_scratch(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K,
                                            void* scratch, size_t scratch_bytes, void* sums, size_t sums_bytes, lr_stream_t stream) {
  LR_REQUIRE_PTR(x);
  LR_REQUIRE_PTR(w);
  LR_REQUIRE_PTR(y);
  LR_OPTIONAL_PTR(sums);
  if (M <= 0 || N <= 0 || K <= 0 || N % 2 || ldx < K || ldy < N / 2) return LR_E_SHAPE;
  if (K % 8 || ldx % 8) return LR_E_ALIGN;
  const int I = N / 2;
  const bool product = M <= 64 && M >= GEMM_SCRATCH_FROM && sums && gemm_reaches(ldx, I, K, GEMM_PAIR);   // of a decode batch
  if (M <= 64 && !product) {
    lr_projection_t pr;
    pr.x = x; pr.ldx = ldx; pr.w = w; pr.y = y; pr.ldy = ldy; pr.N = N; pr.K = K; pr.epilogue = LR_EPI_SWIGLU; pr.rope = nullptr;
    const int rc = lr_linear_multi(&pr, 1, M, stream);
    if (rc != LR_E_UNSUPPORTED) return rc;
  }
  // (a caller of other than large problems brings `scratch` [M, N]; used where the weights are out of the requests' reach)
  const bool large = M >= 512 && I >= 128 && (int64_t)((M + 255) / 256) * ((I + 127) / 128) >= 192 && gemm_reaches(ldx, I, K, GEMM_PAIR);
  if (!large && !product) {
    LR_REQUIRE_PTR(scratch);
    if (scratch_bytes < (size_t)M * N * sizeof(u16) || M > 65535 * 64) return LR_E_SHAPE;
    if (I % 8 || ldy % 8) return LR_E_ALIGN;
  }
  int rc = gemm(x, ldx, w, y, ldy, M, I, K, GEMM_PAIR, GemmRope{}, sums, sums_bytes, (hipStream_t)stream);
  if (rc != LR_E_UNSUPPORTED || scratch == nullptr || scratch_bytes < (size_t)M * N * sizeof(u16)) return rc;
  rc = linear_rows(x, ldx, w, scratch, N, M, N, K, 0, 0, nullptr, 0, (hipStream_t)stream);
  if (rc != LR_OK) return rc;
  return lr_detail::swiglu_rows(scratch, N, y, ldy, M, I, stream);
}

extern "C" int lr_linear_swiglu_out(const void* x, int64_t ldx, const void* w, void* y, int64_t ldy, int M, int N, int K,
                                    void* scratch, size_t scratch_bytes, lr_stream_t stream) {
  return lr_linear_swiglu_out_scratch(x, ldx, w, y, ldy, M, N, K, scratch, scratch_bytes, nullptr, 0, stream);
}

static int beside_product(const void* q, int64_t ldq, const void* k_cache, const void* v_cache, const int32_t* pos, void* y, int64_t ldy, int B,
                          int Hq, int Hkv, int hd, int Smax, void* scratch, size_t scratch_bytes, void* tickets, const void* x, int64_t ldx,
                          const void* w, const void* scales, void* act, int64_t ld_act, int M, int N, int K, void* sums, size_t sums_bytes,
                          lr_stream_t stream) {
  AttnItems a;
  int G;
  const int rc = attn_fill_items(q, ldq, k_cache, v_cache, pos, y, ldy, B, Hq, Hkv, hd, Smax, scratch, scratch_bytes, tickets, a, G);
  if (rc != LR_OK && rc != LR_E_UNSUPPORTED) return rc;
  LR_REQUIRE_PTR(x);
  LR_REQUIRE_PTR(w);
  LR_REQUIRE_PTR(act);
  LR_OPTIONAL_PTR(sums);
  if (tickets == nullptr) return LR_E_NULL;
  if (M <= 0 || N <= 0 || K <= 0 || N % 2 || ldx < K || ld_act < N / 2) return LR_E_SHAPE;
  if (K % 8 || ldx % 8) return LR_E_ALIGN;
  if (rc != LR_OK || a.tickets == nullptr) return LR_E_UNSUPPORTED;
  auto run = scales ? &lr_detail::gemm_beside_attention<true> : &lr_detail::gemm_beside_attention<false>;
  return run(a, hd, G, x, ldx, w, scales, act, ld_act, M, N / 2, K, sums, sums ? sums_bytes : 0, (hipStream_t)stream);
}

extern "C" int lr_attn_decode_beside_product(const void* q, int64_t ldq, const void* k_cache, const void* v_cache, const int32_t* pos, void* y,
                                             int64_t ldy, int B, int Hq, int Hkv, int hd, int Smax, void* scratch, size_t scratch_bytes,
                                             void* tickets, const void* x, int64_t ldx, const void* w, void* act, int64_t ld_act, int M, int N,
                                             int K, void* sums, size_t sums_bytes, lr_stream_t stream) {
  return beside_product(q, ldq, k_cache, v_cache, pos, y, ldy, B, Hq, Hkv, hd, Smax, scratch, scratch_bytes, tickets, x, ldx, w, nullptr, act,
                        ld_act, M, N, K, sums, sums_bytes, stream);
}

extern "C" int lr_attn_decode_beside_product_fp8(const void* q, int64_t ldq, const void* k_cache, const void* v_cache, const int32_t* pos, void* y,
                                                 int64_t ldy, int B, int Hq, int Hkv, int hd, int Smax, void* scratch, size_t scratch_bytes,
                                                 void* tickets, const void* x, int64_t ldx, const void* w8, const void* scales, void* act,
                                                 int64_t ld_act, int M, int N, int K, void* sums, size_t sums_bytes, lr_stream_t stream) {
  if (scales == nullptr) return LR_E_NULL;
  return beside_product(q, ldq, k_cache, v_cache, pos, y, ldy, B, Hq, Hkv, hd, Smax, scratch, scratch_bytes, tickets, x, ldx, w8, scales, act,
                        ld_act, M, N, K, sums, sums_bytes, stream);
}

extern "C" size_t lr_linear_fp8_product_bytes(int M, int N, int K, int pair) {
  if (M <= 0 || N <= 0 || K <= 0 || (pair && N % 2)) return 0;
  const GemmPlan p = gemm_plan8(M, pair ? N / 2 : N, K, pair ? GEMM_PAIR : GEMM_PLAIN, GEMM_SCRATCH);
  return p.tile < 0 ? 0 : (size_t)p.rem * (p.rem ? p.splits : 0) * GemmTile<2, 1>::TM * GemmTile<2, 1>::TN * sizeof(float);
}

extern "C" int lr_linear_fp8_product(const void* x, int64_t ldx, const void* w8, const void* scales, void* y, int64_t ldy, int M, int N, int K,
                                     const lr_rope_kv_t* rope, void* sums, size_t sums_bytes, lr_stream_t stream) {
  LR_REQUIRE_PTR(x);
  LR_REQUIRE_PTR(w8);
  LR_REQUIRE_PTR(y);
  LR_OPTIONAL_PTR(sums);
  if (scales == nullptr) return LR_E_NULL;
  if (M <= 0 || N <= 0 || K <= 0 || ldx < K || ldy < N) return LR_E_SHAPE;
  if (K % 16 || ldx % 8) return LR_E_ALIGN;
  GemmRope rp{};
  if (rope) {
    if (rope->pos == nullptr) return LR_E_NULL;
    LR_REQUIRE_PTR(rope->table);
    LR_REQUIRE_PTR(rope->k_cache);
    LR_REQUIRE_PTR(rope->v_cache);
    if (rope->n_head <= 0 || rope->n_kv_head <= 0 || rope->head_dim <= 0 || rope->smax <= 0 || rope->block_size <= 0 ||
        (int64_t)(rope->n_head + 2 * (int64_t)rope->n_kv_head) * rope->head_dim != N)
      return LR_E_SHAPE;
    if (ldy % 8 || rope->head_dim % 8) return LR_E_ALIGN;
    rp = GemmRope{(const u16*)rope->table, rope->pos, (u16*)rope->k_cache, (u16*)rope->v_cache, rope->err, 1, rope->n_head,
                  rope->n_kv_head, rope->head_dim, rope->smax, rope->block_size};
  }
  if (!gemm_reaches(ldx, N, K, GEMM_PLAIN)) return LR_E_UNSUPPORTED;
  const int mode = rope ? GEMM_ROPE : GEMM_PLAIN;
  const GemmPlan p = gemm_plan8(M, N, K, mode, sums ? sums_bytes : 0);
  if (p.tile < 0) return LR_E_UNSUPPORTED;
  hipStream_t s = (hipStream_t)stream;
  return rope ? gemm_run_as<2, 1, false, GEMM_ROPE, true, 2, true>(x, ldx, w8, y, ldy, M, N, K, rp, p, sums, s, scales)
              : gemm_run_as<2, 1, false, GEMM_PLAIN, true, 2, true>(x, ldx, w8, y, ldy, M, N, K, rp, p, sums, s, scales);
}

extern "C" size_t lr_linear_fp8_pieces_two_bytes(int M, int N, int K0, int K1) {
  return M <= 0 || N <= 0 || K0 <= 0 || K1 <= 0 ? 0 : lr_detail::outputs_bytes<true>(M, N, K0, K1);
}

extern "C" int lr_linear_fp8_pieces_two(const void* x0, const void* w0, const void* scales0, int K0, void* sums0, int32_t* pieces0, const void* x1,
                                        const void* w1, const void* scales1, int K1, void* sums1, int32_t* pieces1, int M, int N,
                                        size_t sums_bytes, lr_stream_t stream) {
  LR_REQUIRE_PTR(x0);
  LR_REQUIRE_PTR(w0);
  LR_REQUIRE_PTR(sums0);
  LR_REQUIRE_PTR(x1);
  LR_REQUIRE_PTR(w1);
  LR_REQUIRE_PTR(sums1);
  if (scales0 == nullptr || scales1 == nullptr || pieces0 == nullptr || pieces1 == nullptr) return LR_E_NULL;
  if (M <= 0 || N <= 0 || K0 <= 0 || K1 <= 0) return LR_E_SHAPE;
  if (K0 % 16 || K1 % 16) return LR_E_ALIGN;
  const uintptr_t s0 = (uintptr_t)sums0, s1 = (uintptr_t)sums1;
  if ((s0 > s1 ? s0 - s1 : s1 - s0) < sums_bytes) return LR_E_SHAPE;   // (both are written at the same time)
  return lr_detail::gemm_outputs8(x0, w0, scales0, K0, sums0, pieces0, x1, w1, scales1, K1, sums1, pieces1, M, N, sums_bytes, (hipStream_t)stream);
}

extern "C" size_t lr_linear_pieces_two_bytes(int M, int N, int K0, int K1) {
  return M <= 0 || N <= 0 || K0 <= 0 || K1 <= 0 || K0 % 8 || K1 % 8 ? 0 : lr_detail::outputs_bytes<false>(M, N, K0, K1);
}

extern "C" int lr_linear_pieces_two(const void* x0, const void* w0, int K0, void* sums0, int32_t* pieces0, const void* x1, const void* w1, int K1,
                                    void* sums1, int32_t* pieces1, int M, int N, size_t sums_bytes, lr_stream_t stream) {
  LR_REQUIRE_PTR(x0);
  LR_REQUIRE_PTR(w0);
  LR_REQUIRE_PTR(sums0);
  LR_REQUIRE_PTR(x1);
  LR_REQUIRE_PTR(w1);
  LR_REQUIRE_PTR(sums1);
  if (pieces0 == nullptr || pieces1 == nullptr) return LR_E_NULL;
  if (M <= 0 || N <= 0 || K0 <= 0 || K1 <= 0) return LR_E_SHAPE;
  if (K0 % 8 || K1 % 8) return LR_E_ALIGN;
  const uintptr_t s0 = (uintptr_t)sums0, s1 = (uintptr_t)sums1;
  if ((s0 > s1 ? s0 - s1 : s1 - s0) < sums_bytes) return LR_E_SHAPE;   // (both are written at the same time)
  return lr_detail::gemm_outputs(x0, w0, K0, sums0, pieces0, x1, w1, K1, sums1, pieces1, M, N, sums_bytes, (hipStream_t)stream);
}
