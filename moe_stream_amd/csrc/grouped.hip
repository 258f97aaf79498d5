// Multi-token (prefill / batched) expert block for gfx950: the T*k routed
// (token, slot) pairs are grouped by slot and every group runs as a dense
// bf16 MFMA contraction against that slot's 4-bit weights.
//
//   group_pairs_kernel : counting sort of the pairs by slot reference, one
//                        workgroup; emits perm (sorted row -> pair) and the
//                        list of 64-row tiles {ref, first row, rows}
//   grouped_mm (gate/up): per (tile, NB features): H = act(X Wg^T, X Wu^T)
//   grouped_mm (down)   : per (tile, NB outputs):  Yp[pair] = score * H Wd^T
//   combine_pairs      : y[t] = sum over ranks r of Yp[t*k + r] (rank order)
//
// Dequantisation rides on the MFMA.  A word of eight 4-bit codes becomes a
// B fragment of bf16 values 128+q (exact, one v_and_or_b32 per pair), each
// 64-input quant group accumulates into a fresh accumulator, and
//   out += S * acc + (B - 128*S) * rowsum(X over the group),
// the factorised group form of kernels.py:141-145, with exact products and
// fp32 accumulation.  The second term is added every 4 groups, so the 128 offset
// cancels there and is not carried through the row (relative rms error of the sums
// against 64 bits, fp32 emulation: 1.8e-6 at 768, 2,048 and 2,880 inputs of mean
// zero, 4e-6 to 5e-6 of mean one; with the whole row's term added at once 2.9e-6,
// 4.3e-6 and 5.1e-6, and 3e-5 to 4e-5).  The 8 inputs of one MFMA lane are permuted
// identically in A and B (x_pairs order), which leaves every dot product unchanged.
//
// Every output row is one dot product per feature, computed by exactly one
// tile with a fixed accumulation order, so results do not depend on how the
// pairs were grouped or on the order of pairs inside a group.
//
// Reference: the batched gather_qmm calls with rhs_indices = slot per
// (token, rank) (engine_v3.py:588-598, engine_120b.py:132-143) and the
// score-weighted sum over ranks (engine_v3.py:600, engine_120b.py:145).
#include <algorithm>
#include <type_traits>

#include "launchers.h"

namespace moe {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mfma16x16x32(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0,
                                                 0);
}

constexpr int kTileM = 64;
// Wide items (twice the features) from this many of them on: four rounds of the
// 512 resident workgroups.  Below it the last round and the longest items decide,
// and narrow items are faster; past it the wide item's halved token-row reads win.
// A block with the line at 1,024 / 2,048 / never: gpt-oss 29 tokens (wide from 1,024
// on) 180 / 176 / 177 us, 60 tokens 260 / 252 / 254, 128 tokens 373 / 368 / 362;
// Qwen3 1,024 tokens 216 / 220 / 222, 2,048 tokens 340 / 354 / 364, 4,096 tokens
// 622 / 622 / 690.
constexpr int kWideItems = 2048;

// ---------------------------------------------------------------------------
// grouping: one workgroup of 1024 threads; hist[] in dynamic LDS spans every
// valid slot reference, key = ref + n_records in [0, n_slots + n_records).
// ---------------------------------------------------------------------------
// Inclusive scans on DPP (no LDS round trips): within each 16-lane row
// (row_shr 1, 2, 4, 8; lanes without a source add 0), and across the wave
// (then row 0's total into row 1 and row 2's into row 3 by row_bcast:15, rows
// 0-1's total into rows 2-3 by row_bcast:31).
__device__ __forceinline__ int row16_incl_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  return v;
}
__device__ __forceinline__ int wave_incl_scan(int v) {
  v = row16_incl_scan(v);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

__device__ __forceinline__ void group_pairs_body(
    const int32_t *__restrict__ refs, int n_pairs, int n_slots, int n_records, int D,
    int32_t *__restrict__ perm, int4 *__restrict__ tiles, int32_t *__restrict__ n_tiles,
    float *__restrict__ yp) {
  extern __shared__ int hist[];
  // tiles are listed by size class, largest first (classes 4..1: a tile of
  // r rows is class ceil(r / 16)), so the longest work items start first
  __shared__ int wsum[5][16];   // per wave: pairs, class-1..4 tiles
  __shared__ int wpre[5][16];   // exclusive prefixes over the waves
  __shared__ int cbase[4];      // first tile of each class (class 4 first)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nkeys = n_slots + n_records;
  for (int i = tid; i < nkeys; i += 1024) hist[i] = 0;
  __syncthreads();
  for (int p = tid; p < n_pairs; p += 1024) {
    const int key = refs[p] + n_records;
    if (key >= 0 && key < nkeys) {
      atomicAdd(&hist[key], 1);
    } else {   // out-of-range reference: flagged, contributes zero
      flag_error();
      for (int n = 0; n < D; ++n) yp[(int64_t)p * D + n] = 0.f;
    }
  }
  __syncthreads();
  // per-thread contiguous key chunk: pair and per-class tile totals, then
  // block scans
  const int chunk = (nkeys + 1023) / 1024;
  const int k0 = min(tid * chunk, nkeys), k1 = min(k0 + chunk, nkeys);
  auto tile_class = [](int rows) { return (rows + 15) >> 4; };   // 1..4
  int st[5] = {0, 0, 0, 0, 0};   // pairs, then tiles of classes 1..4
  for (int i = k0; i < k1; ++i) {
    const int c = hist[i];
    const int cl = c % kTileM ? tile_class(c % kTileM) : 0;
    st[0] += c;
    st[1] += cl == 1;
    st[2] += cl == 2;
    st[3] += cl == 3;
    st[4] += c / kTileM + (cl == 4);
  }
  int it[5];
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    it[q] = wave_incl_scan(st[q]);
    if (lane == 63) wsum[q][wave] = it[q];
  }
  __syncthreads();
  if (wave == 0) {   // the 16 waves' prefixes: one quantity per 16-lane row
    const int row = lane >> 4, w = lane & 15;
    __shared__ int ctot[8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int q = h * 4 + row;   // quantities 0-3, then 4
      const int v = q < 5 ? wsum[q][w] : 0;
      const int sc = row16_incl_scan(v);
      if (q < 5) wpre[q][w] = sc - v;
      if (w == 15) ctot[q] = sc;   // the quantity's total
    }
    if (lane == 0) {   // class bases, class 4 first
      const int c1 = ctot[1], c2 = ctot[2], c3 = ctot[3], c4 = ctot[4];
      cbase[3] = 0;
      cbase[2] = c4;
      cbase[1] = c4 + c3;
      cbase[0] = c4 + c3 + c2;
      *n_tiles = c4 + c3 + c2 + c1;
    }
  }
  __syncthreads();
  int bp = wpre[0][wave] + it[0] - st[0], bt[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) bt[q] = cbase[q] + wpre[q + 1][wave] + it[q + 1] - st[q + 1];
  for (int i = k0; i < k1; ++i) {
    const int c = hist[i];
    hist[i] = bp;   // becomes the scatter cursor of key i
    for (int m = 0; m < c; m += kTileM) {
      const int rows = min(kTileM, c - m), q = tile_class(rows) - 1;   // bt index
      int t = 0;
#pragma unroll
      for (int qq = 0; qq < 4; ++qq)   // (registers, not a dynamic index)
        if (qq == q) t = bt[qq]++;
      tiles[t] = make_int4(i - n_records, bp + m, rows, 0);
    }
    bp += c;
  }
  __syncthreads();
  for (int p = tid; p < n_pairs; p += 1024) {
    const int key = refs[p] + n_records;
    if (key >= 0 && key < nkeys) perm[atomicAdd(&hist[key], 1)] = p;
  }
}

__global__ __launch_bounds__(1024) void group_pairs_kernel(
    const int32_t *__restrict__ refs, int n_pairs, int n_slots, int n_records, int D,
    int32_t *__restrict__ perm, int4 *__restrict__ tiles, int32_t *__restrict__ n_tiles,
    float *__restrict__ yp) {
  group_pairs_body(refs, n_pairs, n_slots, n_records, D, perm, tiles, n_tiles, yp);
}

// Row sums: fp32, a row's groups padded to a multiple of 4 (16-byte rows).
__host__ __device__ constexpr int rs_pitch(int K) { return (K / 64 + 3) / 4 * 4; }

// ---------------------------------------------------------------------------
// The A operand's rows in x_pairs order (each 8-input piece p holds inputs
// (0,4), (1,5), (2,6), (3,7) pairwise, the order of the B fragments) and their
// 64-input row sums, once per call: one thread per piece, the 8 pieces of a
// group in 8 consecutive lanes (rs: [rows][rs_pitch(K)] fp32).
// ---------------------------------------------------------------------------
// piece i of `rows` rows of K inputs (32-bit index arithmetic: the host
// passes at most 2^30 pieces at a time)
__device__ __forceinline__ void prep_piece(int i, const uint16_t *__restrict__ src, int64_t rows,
                                           int K, uint16_t *__restrict__ dst,
                                           float *__restrict__ rs) {
  const int ppr = K / 8;
  const bool ok = i < (int)(rows * ppr);
  const int r = ok ? i / ppr : 0;
  const int pc = ok ? i - r * ppr : 0;
  const uint4 v = ok ? load16(reinterpret_cast<const uint4 *>(src + (int64_t)r * K + pc * 8))
                     : make_uint4(0, 0, 0, 0);
  const uint32_t in[4] = {v.x, v.y, v.z, v.w};
  uint32_t out[4];
  x_pairs(in, out);
  float sm = 0.f;
#pragma unroll
  for (int m = 0; m < 4; ++m) sm += bf16_to_f32(in[m] & 0xffffu) + bf16_to_f32(in[m] >> 16);
  sm = group_sum<8>(sm);
  if (ok) {
    *reinterpret_cast<uint4 *>(dst + (int64_t)r * K + pc * 8) = make_uint4(out[0], out[1], out[2], out[3]);
    if ((pc & 7) == 0) rs[(int64_t)r * rs_pitch(K) + pc / 8] = sm;
  }
}

__global__ __launch_bounds__(256) void grouped_prep_kernel(const uint16_t *__restrict__ src,
                                                           int64_t rows, int K,
                                                           uint16_t *__restrict__ dst,
                                                           float *__restrict__ rs) {
  prep_piece(blockIdx.x * 256 + threadIdx.x, src, rows, K, dst, rs);
}

// The grouping (workgroup 0) and the token rows' prep (the other workgroups)
// in one launch: they are independent, so the prep runs beside the grouping.
__global__ __launch_bounds__(1024) void group_prep_kernel(
    const int32_t *__restrict__ refs, int n_pairs, int n_slots, int n_records, int D,
    int32_t *__restrict__ perm, int4 *__restrict__ tiles, int32_t *__restrict__ n_tiles,
    float *__restrict__ yp, const uint16_t *__restrict__ x, int64_t T, uint16_t *__restrict__ xq,
    float *__restrict__ rsx) {
  if (blockIdx.x == 0)
    group_pairs_body(refs, n_pairs, n_slots, n_records, D, perm, tiles, n_tiles, yp);
  else
    prep_piece((blockIdx.x - 1) * 1024 + threadIdx.x, x, T, D, xq, rsx);
}

// ---------------------------------------------------------------------------
// One work item of the grouped contraction: the rows of one tile (A, up to
// 64 rows of KIN bf16 inputs, already in x_pairs order) against NPROJ
// projections' 4-bit weights for 64 * CB consecutive output features, on 4
// waves.  Wave w owns CB 16-feature column blocks of every projection for all
// M 16-row blocks the tile fills (a template parameter: no branches around
// the MFMAs).
//
//  * A: one quad (4 quant groups of 64 inputs) of the tile's rows in LDS, in
//    two buffers, one barrier per quad: while a quad is computed the next
//    one's pieces are loaded into registers half a quad at a time and written
//    to the other buffer.  Piece p of row r of a group sits at
//    r * 8 + (p ^ (r & 7)): the 8 lanes that copy a row and the 16 rows of a
//    fragment read both fall on distinct banks.
//  * B: each wave loads its own rows' codes (64 bytes of a row by 4 lanes) a
//    quad ahead into registers and turns them into fragments through an LDS
//    region of its own, half a quad at a time and without a barrier: chunk c of
//    row r at c ^ (r >> 2), so the 32 lanes of an 8-byte fragment read fall on
//    distinct banks.  (Loaded in fragment order, 16 rows per 16 lanes, each
//    8-byte piece costs a cache access of its own.)
//  * Each group accumulates into a fresh 16x16 block (2 MFMAs over the bf16
//    128+q codes), folded into the output by S.
//  * The scale and bias rows come 16 groups at a time (32 bytes of a row), a chunk
//    ahead through registers into a region of the wave's own, the row sums are in
//    LDS for the whole item.
//  * The bias term sum_g rowsum[g] * (B[g] - 128 S[g]): per quad and block one
//    fp32 MFMA of K = 4 groups from zero, added behind the quad's folds.  (The fp32
//    MFMA takes two of the bf16 ones' time, an eighth of a quad's; bf16 ones over
//    the sums in three parts are cheaper but have no exact B - 128 S to work on.)
//
// Measured (whole block against the kernels before these: 64-row tiles with codes
// and rows staged a quad at a time behind two barriers, narrow items only, cold
// weights; results bit for bit the same): Qwen3 4,096 tokens 704 -> 596 us, 512
// tokens 145 -> 142, gpt-oss 700 tokens 743 -> 608, 29 tokens 211 -> 173; 8 and 16 Qwen3
// tokens through 48 layers 2.34 -> 2.37 and 2.73 -> 2.79 ms.
//
// What sets the shape: per group a wave's M x N blocks (N = CB * NPROJ) take
// 32 M N matrix-core cycles (8 M N more for the bias term), 64 M LDS cycles (a
// 16-row fragment is 2 KB, the CU's LDS serves four SIMDs at 128 B/cycle) and
// 4 * (14 N + 5 M N) VALU cycles (decode of 2 N code words, fold, bias term).  At
// M = 4 the LDS reads alone exceed the MFMAs for N < 2; at N = 4 they are half of
// them and the VALU work is level.
// Rows past the tile compute garbage from a copy of a real row, which no
// output row depends on (MFMA rows are independent) and nothing stores;
// features past the matrix likewise (their addresses are clamped).
// ---------------------------------------------------------------------------
constexpr int kCodeBytes = 4096;   // a wave's code region: 4 blocks of 16 rows x 64 bytes

template <int KIN>
struct GDim {
  static constexpr int NG = KIN / 64;             // quant groups along the inputs
  static constexpr int NQ = (NG + 3) / 4;         // quads
  static constexpr int NGL = NG - 4 * (NQ - 1);   // groups of the last quad
  // scales and biases in LDS: 16 groups (a chunk, 32 bytes of a row) at a time
  static constexpr int NCH = (NQ + 3) / 4;        // chunks
  // row sums in LDS: the 16 rows of a fragment on distinct banks (pitch 4 x odd)
  static constexpr int RP = rs_pitch(KIN), RSP = RP % 8 ? RP : RP + 4;
  static_assert(KIN % 64 == 0, "whole quant groups");
};

constexpr int kMmWaves = 4, kMmThreads = 64 * kMmWaves;

typedef u32x4_t u32x4_a4_t __attribute__((aligned(4)));
__device__ __forceinline__ uint32_t gload2(const void *p) {
  return *(const __attribute__((address_space(1))) uint16_t *)(p);
}

// Chunk ci of a row of NG bf16 values: halfwords 8 ci .. + 7, zero past NG.  The
// load never leaves the row's dwords (a window across the row's end is read 8
// halfwords before it and shifted) and is dword-aligned: a 16-byte load at an odd
// halfword takes several times as long.
template <int NG>
__device__ __forceinline__ uint4 row_chunk(const char *row, int ci) {
  if (NG % 8 == 0) return gload16(row + 16 * ci);
  if (NG < 8) {
    uint32_t h[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = i < NG ? gload2(row + 2 * (i < NG ? i : 0)) : 0u;
    return make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16),
                      h[6] | (h[7] << 16));
  }
  constexpr int SH = 8 - NG % 8;   // of the window across the end
  const int b = 8 * ci;
  const char *p = row + min(b, NG - 8) * 2;
  const uint32_t odd = NG % 2 ? (uint32_t)(uintptr_t)p & 2u : 0u;   // (even: rows of dwords)
  const char *p4 = p - odd;
  const u32x4_t f = *(const __attribute__((address_space(1))) u32x4_a4_t *)(p4);
  const uint32_t l = NG % 2 ? (uint32_t)gload4i(p4 + (odd ? 16 : 12)) : 0u;
  const uint32_t x[5] = {f.x, f.y, f.z, f.w, l};
  uint32_t w[8] = {0, 0, 0, 0, 0, 0, 0, 0}, t[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = odd ? (x[i] >> 16) | (x[i + 1] << 16) : x[i];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    t[i] = SH % 2 ? (w[i + SH / 2] >> 16) | (w[i + SH / 2 + 1] << 16) : w[i + SH / 2];
  return b > NG - 8 ? make_uint4(t[0], t[1], t[2], t[3]) : make_uint4(w[0], w[1], w[2], w[3]);
}

// Keeps the value's computation here in program order (emits nothing).
template <class T>
__device__ __forceinline__ void pin(T &v) {
  asm volatile("" : "+v"(v));
}

// The sum of a row's 64 activations, 8 in x_pairs order in each of 8 consecutive
// lanes (the lane of the first 8 has it).  Two orders of equal depth: each geometry
// keeps the one that its results have always been computed with, prep_piece's where
// d_ff is no multiple of 128 (there a kernel of its own took the sums).
template <int F>
__device__ __forceinline__ float h_row_sum(uint4 v) {
  auto lo = [](uint32_t w) { return bf16_to_f32(w & 0xffffu); };
  auto hi = [](uint32_t w) { return bf16_to_f32(w >> 16); };
  const float a = (lo(v.x) + lo(v.y)) + (lo(v.z) + lo(v.w));
  const float b0 = hi(v.x) + hi(v.y), b1 = hi(v.z) + hi(v.w);
  if (F % 128) return group_sum<8>((a + b0) + b1);
  // 16 features as a balanced tree, then the four of them in order
  float s = a + (b0 + b1);
  s += dpp_f<kDppQuadXor1>(s);
  const float t = dpp_f<kDppQuadXor2>(s);   // (first lane: the second sum, ...)
  return ((s + t) + dpp_f<kDppHalfMirror>(t)) + dpp_f<kDppHalfMirror>(s);
}

struct GLds {
  uint4 *a;                    // two buffers of [groups][row * 8 + (piece ^ (row & 7))]
  char *b;                     // [4 waves][N blocks][16 rows][64 bytes], swizzled
  char *s;                     // [4 waves][S, B][N blocks][16 rows][32 bytes]: a chunk
  float *rs;                   // [64 rows][RSP]: the tile rows' sums
  float *pb;                   // [4 waves][4 blocks][16]: the projection biases
  int *rperm;                  // down: the tile rows' pair ids [64] ...
  float *rsc;                  // ... and their scores [64]
};

// pair / k by the multiplier ceil(2^32 / k), exact for pairs below 2^24 and
// k <= 32; k == 1 has no such multiplier and takes the pair itself (no branch:
// the rows' loads hang on this)
struct TokenOf {
  uint32_t mul, one;
  __device__ __forceinline__ int operator()(int pair) const {
    return (int)(__umulhi((uint32_t)pair, mul) + ((uint32_t)pair & one));
  }
};
static TokenOf token_of(int k) {
  if (k == 1) return {0u, ~0u};
  return {(uint32_t)((((uint64_t)1 << 32) + k - 1) / k), 0u};
}

template <int M, int CB, int D, int F, bool PBIAS, bool GU>
__device__ __forceinline__ void grouped_item(
    const PoolArgs &pa, const uint16_t *__restrict__ aq, const float *__restrict__ ars,
    TokenOf tok, const int32_t *__restrict__ perm, int ref, int r0, int rows, int nb0,
    uint16_t *__restrict__ h_out, float *__restrict__ rs_out,
    const float *__restrict__ scores, float *__restrict__ yp, int act, float alpha, float limit,
    const GLds &L) {
  constexpr int KIN = GU ? D : F, NOUT = GU ? F : D, NPROJ = GU ? 2 : 1;
  using I = GDim<KIN>;
  constexpr int NG = I::NG, NQ = I::NQ, NGL = I::NGL;
  constexpr int NP = PBIAS ? 4 : 3, NB = 16 * CB * kMmWaves, RB = KIN / 2;
  constexpr int ROWS = 16 * M;
  // A in LDS: whole quads of 32 rows, or half quads of 64; R quads wait in
  // registers
  constexpr bool QA = M <= 2;
  constexpr int AROWS = QA ? 32 : 64, AG = QA ? 4 : 2, R = M == 1 ? 2 : 1;
  constexpr int SPG = AROWS * 8 / kMmThreads;   // A pieces per thread and group
  // (opaque here and at the epilogue: what hangs on it is computed there, not held
  // in registers across the items or the quads)
  int tid = threadIdx.x;
  pin(tid);
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, kq = lane >> 4;
  // (named, not arrays: a pointer picked from an array by a lane's index goes
  // through memory)
  constexpr int PF = GU ? PROJ_GATE : PROJ_DOWN, PL = GU ? PROJ_UP : PROJ_DOWN;
  const char *const w0 = resolve(pa, comp_index(PF, PART_W, NP), ref);
  const char *const w1 = resolve(pa, comp_index(PL, PART_W, NP), ref);
  const char *const s0 = resolve(pa, comp_index(PF, PART_S, NP), ref);
  const char *const s1 = resolve(pa, comp_index(PL, PART_S, NP), ref);
  const char *const o0 = resolve(pa, comp_index(PF, PART_B, NP), ref);
  const char *const o1 = resolve(pa, comp_index(PL, PART_B, NP), ref);
  constexpr int N = CB * NPROJ;                        // blocks of a wave
  constexpr int NG0 = NQ > 1 ? 4 : NGL;                // groups of the first quad
  // the row indices first: everything else of the tile's rows hangs on them
  auto row_index = [&](int r) { return gload4i(perm + r0 + min(r, rows - 1)); };
  int pr_st[SPG], pr_rs = 0, pr_ep = 0;
#pragma unroll
  for (int j = 0; j < SPG; ++j) pr_st[j] = GU ? row_index((tid >> 3) + 32 * j) : 0;
  if (GU) pr_rs = row_index(tid >> 2);
  if (!GU) pr_ep = row_index(lane);
  // codes of half a quad: lane l of a wave loads 16-byte chunk l & 3 of row l >>
  // 2 of each of its blocks
  const int bch = (lane & 3) * 16;
  // first feature of column block cb (a block past the matrix: its last one)
  auto block_f = [&](int cb) { return (uint32_t)min(nb0 + (wave * CB + cb) * 16, NOUT - 16); };
  // (offsets per lane: as scalars they are spilled, 8 tokens through 12 layers 557 us
  // against 548)
  uint32_t boff[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) boff[cb] = (block_f(cb) + (lane >> 2)) * RB;
  uint4 breg[R][2][N];   // codes to come
  auto load_b = [&](int q, int hf, int rs) {
    // (chunks past the row, in a last partial quad: its last one, unused)
    const int o = q * 128 + hf * 64;
    const uint32_t c = RB % 64 == 0 || o + 64 <= RB ? (uint32_t)(o + bch)
                                                    : (uint32_t)min(o + bch, RB - 16);
#pragma unroll
    for (int n = 0; n < N; ++n)
      breg[rs][hf][n] = gload16((n % NPROJ ? w1 : w0) + (boff[n / NPROJ] + c));
  };
  char *const bl = L.b + wave * kCodeBytes;
  const uint32_t bwr = (uint32_t)((lane >> 2) * 64 + (((lane & 3) ^ (lane >> 4)) << 4));
  // (a wave's own region: its LDS accesses are in order, the fences keep the
  // compiler from moving one lane's reads across another's writes)
  auto store_b = [&](int hf, int rs) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int n = 0; n < N; ++n) *reinterpret_cast<uint4 *>(bl + n * 1024 + bwr) = breg[rs][hf][n];
    asm volatile("" ::: "memory");
  };
  // this lane's 16 codes of a group: row col of block n, bytes 8 kq .. + 7
  const uint32_t brd = (uint32_t)(col * 64 + (((kq >> 1) ^ (col >> 2)) << 4) + (kq & 1) * 8);
  auto read_b = [&](int gi, int n) {
    return *reinterpret_cast<const uint2 *>(bl + n * 1024 + (brd ^ ((gi & 1) << 5)));
  };
  // the wave's scale and bias rows a chunk at a time, as 16-byte pieces, SPT per lane
  // and array: piece h = lane & 1 of row (lane >> 1) & 15 of block 2 t + (lane >> 5);
  // in LDS at h ^ (row >> 3), so the 16 rows of an 8-byte read fall on distinct banks
  constexpr int SPT = N / 2;
  char *const sl = L.s + wave * (N * 1024);
  auto load_s = [&](int ch, const char *b0, const char *b1, uint4 (&v)[SPT]) {
    int ln = lane;
    pin(ln);   // (the addresses are computed here each time)
    const uint32_t row = (uint32_t)((ln >> 1) & 15) * (NG * 2);
    // (pieces past the row: its last one, unused)
    const int pc = min(2 * ch + (ln & 1), (NG - 1) / 8);
#pragma unroll
    for (int t = 0; t < SPT; ++t) {   // (block 2 t + 1: the other projection's, or the next)
      const char *p0 = b0 + block_f(NPROJ > 1 ? t : 2 * t) * (NG * 2);
      const char *p1 = b1 + block_f(NPROJ > 1 ? t : 2 * t + 1) * (NG * 2);
      v[t] = row_chunk<NG>((ln & 32 ? p1 : p0) + row, pc);
    }
  };
  const uint32_t swr = (uint32_t)((lane >> 1) * 32 + (((lane & 1) ^ ((lane >> 4) & 1)) << 4));
  auto store_s = [&](int arr, const uint4 (&v)[SPT]) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int t = 0; t < SPT; ++t)
      *reinterpret_cast<uint4 *>(sl + arr * (N * 512) + t * 1024 + swr) = v[t];
    asm volatile("" ::: "memory");
  };
  // a row's 4 values (groups) of quad q
  const uint32_t srd = (uint32_t)(col * 32 + ((col >> 3) << 4));
  auto read_s = [&](int arr, int q, int n) {
    return *reinterpret_cast<const uint2 *>(sl + (arr * N + n) * 512 + (srd ^ ((q & 3) << 3)));
  };
  // A: this thread's pieces of the rows (tid >> 3) + 32 j, half a quad at a time
  const uint16_t *asrc[SPG];
  uint32_t adst[SPG];
  uint4 areg[R][AG][SPG];
  // groups g0 .. g0 + AG - 1 of a quad, as many as its ng
  auto load_a = [&](int q, int g0, int ng, int rs) {
#pragma unroll
    for (int i = 0; i < AG; ++i)
      if (g0 + i < ng)
#pragma unroll
        for (int j = 0; j < SPG; ++j) areg[rs][i][j] = gload16(asrc[j] + (q * 4 + g0 + i) * 64);
  };
  auto store_a = [&](int buf, int g0, int ng, int rs) {
#pragma unroll
    for (int i = 0; i < AG; ++i)
      if (g0 + i < ng)
#pragma unroll
        for (int j = 0; j < SPG; ++j)
          L.a[(buf * AG + i) * (AROWS * 8) + adst[j]] = areg[rs][i][j];
  };
  // the first scales, biases and codes, the row sums and the first A rows on their way
  uint4 sv[SPT], bv[SPT];
  load_s(0, s0, s1, sv);
  load_s(0, o0, o1, bv);
  uint32_t pbv = 0;   // the projection bias of feature col of block kq
  if (PBIAS) {
    const char *const q0 = resolve(pa, comp_index(PF, PART_BIAS, NP), ref);
    const char *const q1 = resolve(pa, comp_index(PL, PART_BIAS, NP), ref);
    const int n = min(kq, N - 1);
    const uint32_t f = (uint32_t)min(nb0 + (wave * CB + n / NPROJ) * 16, NOUT - 16) + col;
    pbv = gload2((NPROJ > 1 && (n & 1) ? q1 : q0) + 2 * f);
  }
  load_b(0, 0, 0);
  if (NG0 > 2) load_b(0, 1, 0);
  constexpr int RPP = I::RP / 4, RSJ = (RPP + 3) / 4;   // 16-byte pieces of a row, per thread
  uint4 rsv[RSJ];
  {
    const int64_t row = GU ? tok(pr_rs) : r0 + min(tid >> 2, rows - 1);
    const float *src = ars + row * I::RP;
#pragma unroll
    for (int i = 0; i < RSJ; ++i) rsv[i] = gload16(src + 4 * min((tid & 3) + 4 * i, RPP - 1));
  }
#pragma unroll
  for (int j = 0; j < SPG; ++j) {
    const int r = (tid >> 3) + 32 * j, p = tid & 7;
    const int64_t arow = GU ? tok(pr_st[j]) : r0 + min(r, rows - 1);
    asrc[j] = aq + arow * KIN + p * 8;
    adst[j] = (uint32_t)(r * 8 + (p ^ (r & 7)));
  }
  load_a(0, 0, NG0, 0);
  f32x4_t acc[M][CB][NPROJ];
#pragma unroll
  for (int rb = 0; rb < M; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int j = 0; j < NPROJ; ++j) acc[rb][cb][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  if (!GU && wave == 0) {
    L.rperm[lane] = pr_ep;
    L.rsc[lane] = gload4f(scores + pr_ep);
  }
  store_s(0, sv);
  store_s(1, bv);
  if (PBIAS) L.pb[wave * 64 + lane] = bf16_to_f32(pbv);
#pragma unroll
  for (int i = 0; i < RSJ; ++i) {
    const int p = (tid & 3) + 4 * i;
    uint4 v = rsv[i];
    if (NG % 4 && p == RPP - 1)   // (the pad meets a zero factor: it must be finite)
      v = make_uint4(v.x, NG % 4 > 1 ? v.y : 0u, NG % 4 > 2 ? v.z : 0u, 0u);
    if (p < RPP) *reinterpret_cast<uint4 *>(L.rs + (tid >> 2) * I::RSP + 4 * p) = v;
  }
  store_a(0, 0, NG0, 0);
  store_b(0, 0);
  // quads 1 .. R on their way (of the A rows whole quads only)
#pragma unroll
  for (int q = 1; q <= R; ++q)
    if (q < NQ) {
      if (QA) load_a(q, 0, q < NQ - 1 ? 4 : NGL, q % R);
      load_b(q, 0, q % R);
      if (R > 1 && q < R) load_b(q, 1, q % R);
    }
  __syncthreads();
  // The quads as a software pipeline of steps, one per (group, block n of the
  // wave's N): a step issues its 2 M MFMAs into fresh blocks, and between them
  // the VALU work of its neighbours: ahead of each first MFMA the fold of the
  // step before out of the block it overwrites (4 instructions, that MFMA's own
  // 16 cycles), behind the second ones the decode of the step after.  The order
  // is pinned: left to itself the compiler puts each fold right behind its
  // MFMAs and waits for them.
  uint4 a0[M], a1[M];     // the group's A fragments (inputs 0-31 and 32-63 of the lane order)
  uint32_t bf[2][8];      // a step's B fragments: both halves
  uint2 creg[2];          // codes of the steps after
  f32x4_t c[M];           // its blocks
  float S[2];
  uint2 scur[N];          // the quad's scales
  int ard[2];             // LDS index of this lane's two pieces in row block 0
  ard[0] = col * 8 + ((2 * kq) ^ (col & 7));
  ard[1] = col * 8 + ((2 * kq + 1) ^ (col & 7));
#pragma unroll
  for (int rb = 0; rb < M; ++rb) {
    a0[rb] = L.a[rb * 128 + ard[0]];
    a1[rb] = L.a[rb * 128 + ard[1]];
    c[rb] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  }
  S[1] = 0.f;
#pragma unroll
  for (int n = 0; n < N; ++n) scur[n] = read_s(0, 0, n);
  // The bias term of a quad, sum over its groups of rowsum * (B - 128 S): one fp32
  // MFMA of K = 4 groups per block (A: row col, group kq; B: feature col, group kq)
  // from zero, added behind the quad's folds, in the first group of the next quad:
  // there the 128 offset of the codes cancels before it is carried any further.
  float ra[M], C[N];
  uint2 bcur[2];          // bias values to come
  constexpr int BZ = M <= 2 ? M : 1;
  f32x4_t bz[BZ];
#pragma unroll
  for (int rb = 0; rb < M; ++rb) ra[rb] = 0.f;
#pragma unroll
  for (int n = 0; n < N; ++n) C[n] = 0.f;
  // halfword kq of 4 as an fp32 value
  const uint32_t hsel = 0x01000c0cu + (uint32_t)kq * 0x02020000u;
  auto pick = [&](uint2 v) { return __uint_as_float(__builtin_amdgcn_perm(v.y, v.x, hsel)); };
  const float *const rsl = L.rs + col * I::RSP + kq;
  auto bias_block = [&](int rb, int n) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(ra[rb], C[n], (f32x4_t){0.f, 0.f, 0.f, 0.f}, 0, 0,
                                                0);
  };
  auto factor = [&](int n) { return fmaf(-128.f, pick(scur[n]), pick(bcur[n & 1])); };
  auto add_block = [&](f32x4_t &o, const f32x4_t &v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] += v[e];
    pin(o);
  };
  // fragment word m of 8, 4 of each code word, as pairs of bf16 128+q (one
  // v_and_or_b32 after the shift: its constants in registers, one of them scalar.
  // Not bfi_mask(), see there)
  uint32_t kmask = 0x000f000fu, kexp = 0x43004300u;
  asm volatile("" : "+s"(kmask));
  pin(kexp);
  auto decode = [&](uint2 cw, int m) {
    return (((m < 4 ? cw.x : cw.y) >> (4 * (m & 3))) & kmask) | kexp;
  };
  creg[0] = read_b(0, 0);
  creg[1] = read_b(1 / N, 1 % N);
#pragma unroll
  for (int m = 0; m < 8; ++m) bf[0][m] = decode(creg[0], m);
  // One quad of ng groups (constants, as is everything but q; par: its parity;
  // first: known to be quad 0, behind which there is no bias term to add: in the
  // rolled loop quad 0 adds zeros): steps s = gi * N + n, the step registers
  // alternating by s.  Two steps before the end of each half, when the last of its
  // codes are read, the next half's go from registers to the wave's own LDS and the
  // loads of the same half R quads on are issued into the registers (ng_next,
  // ng_second, ng_load: groups of quads q + 1, q + R and q + 1 + R, 0: none).  The A
  // rows of the next quad go along with M <= 2, else half a quad ahead.  The barrier
  // is one step before the quad's (half's) end, so that the last step can read the
  // next fragments.
  auto quad = [&](int q, int par, int ng, int ng_next, int ng_second, int ng_load, bool first) {
    const int ns = ng * N, rs = (par + 1) % R;
    // the next chunk's scales and biases: the LDS of a chunk's scales is free from
    // its quad 3 on, of its biases from that quad's second group on
    const bool chunk = q / 4 + 1 < I::NCH;
    if ((q & 3) == 2 && chunk) load_s(q / 4 + 1, s0, s1, sv);
    if ((q & 3) == 3 && chunk) {
      store_s(0, sv);
      load_s(q / 4 + 1, o0, o1, sv);
    }
    if (!QA && ng > 2) load_a(q, 2, ng, 0);
    // a step; G0: of the quad's first group
    auto step = [&](int st, auto G0) {
      constexpr bool g0 = decltype(G0)::value;
      const int gi = g0 ? 0 : st / N, n = st % N, j = n % NPROJ, cb = n / NPROJ;
      const int cur = st & 1, prv = cur ^ 1;
      // the block folded here: the step before's
      const int pn = (n + N - 1) % N, pj = pn % NPROJ, pcb = pn / NPROJ;
      const bool dec = st + 1 < ns || ng_next > 0;   // there is a step after
      const bool last = st + 1 == ns;
      const bool half_end = last || (!QA && st == 2 * N - 1);
      // the bias term of the quad before, block n; added in the step after where
      // there are registers to hold it
      const bool bias = g0 && !first, pend = BZ == M && !first && st > 0 && st <= N;
      if (last && (q & 3) == 3 && chunk) store_s(1, sv);
      const int nbuf = QA ? par ^ 1 : last ? 0 : 1;   // the A buffer after this one
      if (!QA && st == (ng > 2 ? 2 * N : 0) && ng_next > 0) load_a(q + 1, 0, ng_next, 0);
      if (!QA && half_end && (!last || ng_next > 0))
        store_a(nbuf, last ? 0 : 2, last ? ng_next : ng, 0);
      // codes: the second half's when the last of the first are read ...
      if (ng > 2 && st + 2 == 2 * N) {
        store_b(1, par % R);
        if (ng_second > 2) load_b(q + R, 1, par % R);
      }
      // ... and the next quad's
      if (st + 2 == ns && ng_next > 0) {
        if (QA) store_a(par ^ 1, 0, ng_next, rs);
        store_b(0, rs);
        if (ng_load > 0) {
          if (QA) load_a(q + 1 + R, 0, ng_load, rs);
          load_b(q + 1 + R, 0, rs);
        }
      }
      if (half_end && (!last || ng_next > 0)) __syncthreads();
      // codes of the step after next
      if (st + 2 < ns)
        creg[cur] = read_b((st + 2) / N, (st + 2) % N);
      else if (ng_next > 0)
        creg[cur] = read_b((st + 2 - ns) / N, (st + 2 - ns) % N);
      // A fragments of the next group, on a group's last step
      const bool nxa = n == N - 1 && dec;
      const int ag = half_end ? nbuf * AG : QA ? par * AG + gi + 1 : gi + 1;
      const uint4 *an = L.a + ag * (AROWS * 8);
      const uint32_t h = gi < 2 ? scur[n].x : scur[n].y;
      S[cur] = __uint_as_float((gi & 1) ? (h & 0xffff0000u) : (h << 16));
      if (last && ng_next > 0)
#pragma unroll
        for (int i = 0; i < N; ++i)
          scur[i] = read_s(0, q + 1, i);
      const uint4 fb0 = make_uint4(bf[cur][0], bf[cur][1], bf[cur][2], bf[cur][3]);
      const uint4 fb1 = make_uint4(bf[cur][4], bf[cur][5], bf[cur][6], bf[cur][7]);
      uint2 cw = creg[prv];
      if (dec) pin(cw.x), pin(cw.y);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int rb = 0; rb < M; ++rb) {
        f32x4_t &o = acc[rb][pcb][pj];
        if (pend) add_block(o, bz[rb % BZ]);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] += S[prv] * c[rb][e];
        pin(o);
        c[rb] = mfma16x16x32(a0[rb], fb0, (f32x4_t){0.f, 0.f, 0.f, 0.f});
        pin(c[rb]);
        if (nxa) a0[rb] = an[rb * 128 + ard[0]];
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int rb = 0; rb < M; ++rb) {
        if constexpr (g0) if (bias) {
          bz[rb % BZ] = bias_block(rb, n);
          pin(bz[rb % BZ]);
        }
        c[rb] = mfma16x16x32(a1[rb], fb1, c[rb]);
        pin(c[rb]);
        if (nxa) a1[rb] = an[rb * 128 + ard[1]];
        if (dec)
#pragma unroll
          for (int m = 8 * rb / M; m < 8 * (rb + 1) / M; ++m)
            bf[prv][m] = decode(cw, m), pin(bf[prv][m]);
        if constexpr (g0) if (bias && BZ < M) add_block(acc[rb][cb][j], bz[0]);
        __builtin_amdgcn_sched_barrier(0);
      }
      // this quad's factors, two steps behind the reads of their biases (one step
      // of one row block is shorter than an LDS read: 8 tokens through 48 layers
      // 2.38 ms with one step and the row sums read in a quad's last, 2.37 so)
      if (st >= 2 && st < N + 2) C[st - 2] = factor(st - 2);
      if constexpr (g0) {
        bcur[st & 1] = read_s(1, q, st);
        if (st == N - 1)
#pragma unroll
          for (int rb = 0; rb < M; ++rb) ra[rb] = rsl[rb * 16 * I::RSP + 4 * q];
      }
    };
    // (two loops, each small enough to be unrolled)
#pragma unroll
    for (int st = 0; st < N; ++st) step(st, std::true_type());
#pragma unroll
    for (int st = N; st < 4 * N; ++st)
      if (st < ns) step(st, std::false_type());
  };
  // the quads whose loads are whole quads (in pairs where the registers
  // alternate), then the rest
  constexpr int QR = R == 2 || QA ? 2 : 1, QP = NQ > R + 2 ? (NQ - R - 2) / QR * QR : 0;
#pragma unroll 1
  for (int q = 0; q < QP; q += QR) {
    quad(q, 0, 4, 4, 4, 4, false);
    if (QR == 2) quad(q + 1, 1, 4, 4, 4, 4, false);
  }
#pragma unroll
  for (int q = QP; q < NQ; ++q) {
    auto groups = [](int i) { return i < NQ - 1 ? 4 : i == NQ - 1 ? NGL : 0; };
    quad(q, q & 1, groups(q), groups(q + 1), groups(q + R), groups(q + 1 + R), q == 0);
  }
  {   // the last step's fold and the last quad's bias term
    if (NGL == 1) {   // (too short for its last two factors)
      C[N - 2] = factor(N - 2);
      C[N - 1] = factor(N - 1);
    }
    constexpr int last = (NGL * N - 1) & 1, lc = (N - 1) / NPROJ, lj = (N - 1) % NPROJ;
#pragma unroll
    for (int rb = 0; rb < M; ++rb) {
      if (NGL == 1 && NQ > 1 && BZ == M) add_block(acc[rb][lc][lj], bz[rb % BZ]);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[rb][lc][lj][e] += S[last] * c[rb][e];
    }
#pragma unroll
    for (int rb = 0; rb < M; ++rb)
#pragma unroll
      for (int n = 0; n < N; ++n) {
        const f32x4_t b = bias_block(rb, n);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[rb][n / NPROJ][n % NPROJ][e] += b[e];
      }
  }

  int tid_e = tid;
  pin(tid_e);
  float pb[CB][NPROJ];
#pragma unroll
  for (int n = 0; n < N; ++n)
    pb[n / NPROJ][n % NPROJ] = PBIAS ? L.pb[wave * 64 + n * 16 + (tid_e & 15)] : 0.f;
  if (GU) {
    // the activations go through LDS (the A buffers, free once every wave is
    // past the last quad) and out as whole rows, 16 bytes per lane, in x_pairs
    // order (feature f of an 8-feature piece at 2 * (f % 4) + f / 4) with the
    // sums of their bf16 values over each 64-feature group, the down kernel's
    // input.  Staged element npl of row r at npl ^ 16 * ((r >> 2) & 3) (the 4
    // rows of one store fall on distinct banks).
    static_assert(NB % 64 == 0 && F % 64 == 0, "whole groups of h");
    __syncthreads();
    uint16_t *tile = reinterpret_cast<uint16_t *>(L.a);
    auto swz = [](int r) { return ((r >> 2) & 3) << 4; };
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
      const int nl = (wave * CB + cb) * 16 + col;
      const int npl = (nl & ~7) + ((nl & 3) << 1) + ((nl >> 2) & 1);
#pragma unroll
      for (int rb = 0; rb < M; ++rb)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int rr = rb * 16 + 4 * kq + e;
          const float hv = apply_act(act, acc[rb][cb][0][e] + pb[cb][0],
                                     acc[rb][cb][NPROJ - 1][e] + pb[cb][NPROJ - 1], alpha, limit);
          tile[rr * NB + (npl ^ swz(rr))] = (uint16_t)f32_to_bf16(hv);
        }
    }
    __syncthreads();
    constexpr int CPR = NB / 8;                       // 16-byte pieces per row
#pragma unroll 1
    for (int it = 0; it < (ROWS * CPR + kMmThreads - 1) / kMmThreads; ++it) {
      const int i = tid_e + kMmThreads * it;
      if (i >= ROWS * CPR) break;   // (whole waves)
      const int r = i / CPR, c = i % CPR, f = nb0 + c * 8;
      const uint4 v = *reinterpret_cast<const uint4 *>(tile + r * NB + ((c * 8) ^ swz(r)));
      const float sm = h_row_sum<F>(v);
      if (r < rows && f < F) {
        *reinterpret_cast<uint4 *>(h_out + (int64_t)(r0 + r) * F + f) = v;
        if ((c & 7) == 0) rs_out[(int64_t)(r0 + r) * rs_pitch(F) + f / 64] = sm;
      }
    }
  } else {
    // each row scaled by its score, through LDS (the A buffers) and out as whole
    // rows, 16 bytes per lane, 32 rows at a time.  Staged element nl of row r at
    // nl ^ 16 * ((r >> 2) & 3).
    float *tile = reinterpret_cast<float *>(L.a);
    constexpr int CPR = NB / 4;   // 16-byte pieces per row
    static_assert(32 * NB * 4 <= 4 * kTileM * 8 * 16, "32 rows in the A buffers");
#pragma unroll
    for (int r2 = 0; r2 < M; r2 += 2) {
      __syncthreads();
#pragma unroll
      for (int rb = r2; rb < (r2 + 2 < M ? r2 + 2 : M); ++rb)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int rr = rb * 16 + 4 * kq + e;
          const float sc = L.rsc[rr];
#pragma unroll
          for (int cb = 0; cb < CB; ++cb)
            tile[(rr - r2 * 16) * NB + (((wave * CB + cb) * 16 + col) ^ (kq << 4))] =
                sc * (acc[rb][cb][0][e] + pb[cb][0]);
        }
      __syncthreads();
#pragma unroll 4
      for (int it = 0; it < 32 * CPR / kMmThreads; ++it) {
        const int i = tid_e + kMmThreads * it;
        const int r = i / CPR, cc = (i % CPR) * 4, rr = r2 * 16 + r;
        if (rr < rows && (D % NB == 0 || nb0 + cc < D))
          *reinterpret_cast<uint4 *>(yp + (int64_t)L.rperm[rr] * D + nb0 + cc) =
              *reinterpret_cast<const uint4 *>(tile + r * NB + (cc ^ (((r >> 2) & 3) << 4)));
      }
    }
  }
}

// Items of a call: (tile, feature block).  From kXcdTiles tiles on the items
// of one tile go to workgroups of one XCD (workgroup i runs on XCD i % 8), so
// the tile's rows are read from HBM once and from that XCD's L2 by the other
// items, and a hot expert's codes once per XCD.  With fewer tiles that leaves some
// XCDs with a tile more than others; the items are dealt in order.  A block by XCD
// from 64 tiles on / from 128 / never: Qwen3 32 tokens (75 tiles) 70.2 / 69.1 / 68.4
// us, 64 tokens (99) 85.8 / 83.8 / 83.7, gpt-oss 60 tokens (73) 252 / 245 / 248;
// Qwen3 2,048 tokens (319) 354 / 350 / 358, 4,096 tokens (572) 622 / 626 / 640.
constexpr int kXcdTiles = 128;

template <int CB, int D, int F, bool PBIAS, bool GU>
__device__ __forceinline__ void grouped_items(
    const PoolArgs &pa, const uint16_t *aq, const float *ars, TokenOf tok,
    const int32_t *perm, const int4 *tiles, int n_tiles, uint16_t *h_out, float *rs_out,
    const float *scores, float *yp, int act, float alpha, float limit, const GLds &L) {
  constexpr int NOUT = GU ? F : D, NB = 16 * CB * kMmWaves, NBK = (NOUT + NB - 1) / NB;
  constexpr int NP = PBIAS ? 4 : 3, NPROJ = GU ? 2 : 1;
  const bool by_xcd = n_tiles >= kXcdTiles;
  const int n_items = (by_xcd ? (n_tiles + 7) / 8 * 8 : n_tiles) * NBK;
  for (int item = blockIdx.x; item < n_items; item += gridDim.x) {
    const int j = item >> 3;
    const int tile = by_xcd ? (j / NBK) * 8 + (item & 7) : item / NBK;
    const int nb0 = (by_xcd ? j % NBK : item % NBK) * NB;
    if (tile >= n_tiles) continue;
    const int4 tl = tiles[tile];
    const int ref = tl.x, r0 = tl.y, rows = tl.z;
    bool bad = false;
#pragma unroll
    for (int p = 0; p < NPROJ; ++p) {
      const int proj = GU ? (p == 0 ? PROJ_GATE : PROJ_UP) : PROJ_DOWN;
      bad = bad || resolve(pa, comp_index(proj, PART_W, NP), ref) == nullptr;
    }
    if (bad) {   // uniform over the workgroup
      if (threadIdx.x == 0) flag_error();
      continue;
    }
    const int nmb = (rows + 15) >> 4;
#define MOE_GITEM(M)                                                                          \
  grouped_item<M, CB, D, F, PBIAS, GU>(pa, aq, ars, tok, perm, ref, r0, rows, nb0, h_out, \
                                       rs_out, scores, yp, act, alpha, limit, L)
    if (nmb == 1) MOE_GITEM(1);
    else if (nmb == 2) MOE_GITEM(2);
    else if (nmb == 3) MOE_GITEM(3);
    else MOE_GITEM(4);
#undef MOE_GITEM
    __syncthreads();   // the LDS of this item is read before the next item stages
  }
}

// CBW column blocks per wave and projection when the call has at least
// kWideItems such items, CBN otherwise
template <int D, int F, bool PBIAS, int CBW, int CBN, bool GU>
__global__ __launch_bounds__(kMmThreads) __attribute__((amdgpu_waves_per_eu(2))) void
grouped_mm_kernel(PoolArgs pa, const uint16_t *__restrict__ aq, const float *__restrict__ ars,
                  TokenOf tok, const int32_t *__restrict__ perm,
                  const int4 *__restrict__ tiles, const int32_t *__restrict__ n_tiles,
                  uint16_t *__restrict__ h_out, float *__restrict__ rs_out,
                  const float *__restrict__ scores, float *__restrict__ yp, int act, float alpha,
                  float limit) {
  constexpr int NOUT = GU ? F : D, NBW = 16 * CBW * kMmWaves;
  constexpr int NW = CBW * (GU ? 2 : 1);
  __shared__ uint4 a_l[4 * kTileM * 8];
  static_assert(NW <= 4, "code region");
  __shared__ uint4 b_l[kMmWaves * kCodeBytes / 16];
  __shared__ uint4 s_l[kMmWaves * NW * 64];
  __shared__ uint4 rs_l[kTileM * GDim<GU ? D : F>::RSP / 4];
  __shared__ float pb_l[PBIAS ? kMmThreads : 1];
  __shared__ int rp_l[GU ? 1 : kTileM];
  __shared__ float rc_l[GU ? 1 : kTileM];
  const GLds L{a_l, reinterpret_cast<char *>(b_l), reinterpret_cast<char *>(s_l),
               reinterpret_cast<float *>(rs_l), pb_l, rp_l, rc_l};
  const int nt = *n_tiles;
  if (nt * ((NOUT + NBW - 1) / NBW) >= kWideItems)
    grouped_items<CBW, D, F, PBIAS, GU>(pa, aq, ars, tok, perm, tiles, nt, h_out, rs_out,
                                        scores, yp, act, alpha, limit, L);
  else
    grouped_items<CBN, D, F, PBIAS, GU>(pa, aq, ars, tok, perm, tiles, nt, h_out, rs_out,
                                        scores, yp, act, alpha, limit, L);
}

// y[t, :] = sum over ranks r (ascending) of Yp[t*k + r, :]; 4 outputs/thread
__global__ __launch_bounds__(256) void combine_pairs_kernel(
    const float *__restrict__ yp, int T, int k, int D, uint16_t *__restrict__ out,
    float *__restrict__ out32) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= (int64_t)T * D) return;
  const int64_t t = i / D, n = i % D;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int r = 0; r < k; ++r) {
    const float4 v = *reinterpret_cast<const float4 *>(yp + (t * k + r) * D + n);
    s.x += v.x;
    s.y += v.y;
    s.z += v.z;
    s.w += v.w;
  }
  if (out) {
    const uint32_t lo = f32_to_bf16(s.x) | (f32_to_bf16(s.y) << 16);
    const uint32_t hi = f32_to_bf16(s.z) | (f32_to_bf16(s.w) << 16);
    *reinterpret_cast<uint2 *>(out + i) = make_uint2(lo, hi);
  }
  if (out32) *reinterpret_cast<float4 *>(out32 + i) = s;
}

// ---------------------------------------------------------------------------
template <int D, int F, bool PB, int CBW, int CBN>
static void launch_gg(dim3 g, hipStream_t s, const PoolArgs &pa, const uint16_t *xq,
                      const float *rsx, int k, const int32_t *perm, const int4 *tiles,
                      const int32_t *nt, uint16_t *h, float *rsh, int act, float alpha,
                      float limit) {
  hipLaunchKernelGGL((grouped_mm_kernel<D, F, PB, CBW, CBN, true>), g, dim3(kMmThreads), 0, s, pa,
                     xq, rsx, token_of(k), perm, tiles, nt, h, rsh, nullptr, nullptr, act, alpha,
                     limit);
}
template <int D, int F, bool PB, int CBW, int CBN>
static void launch_gd(dim3 g, hipStream_t s, const PoolArgs &pa, const uint16_t *hq,
                      const float *rsh, const float *sc, const int32_t *perm,
                      const int4 *tiles, const int32_t *nt, float *yp) {
  hipLaunchKernelGGL((grouped_mm_kernel<D, F, PB, CBW, CBN, false>), g, dim3(kMmThreads), 0, s,
                     pa, hq, rsh, token_of(1), perm, tiles, nt, nullptr, nullptr, sc, yp, 0, 0.f, 0.f);
}

// column blocks per wave (many items, few items) of gate/up and of down
#define MOE_GROUPED_GEOM(D, F, PB)                                                         \
  {D, F, PB, 64, 128, &launch_gg<D, F, PB, 2, 1>, &launch_gd<D, F, PB, 4, 2>}
static const GroupedLaunch kGroupedTable[] = {
    MOE_GROUPED_GEOM(2048, 768, false),   // Qwen3-30B-A3B
    MOE_GROUPED_GEOM(2048, 768, true),
    MOE_GROUPED_GEOM(2880, 2880, true),   // gpt-oss-120b
    MOE_GROUPED_GEOM(2880, 2880, false),
    MOE_GROUPED_GEOM(256, 128, false),    // small test geometry
    MOE_GROUPED_GEOM(256, 128, true),
};

const GroupedLaunch *find_grouped(int d_model, int d_ff, int has_bias) {
  for (const auto &e : kGroupedTable)
    if (e.d_model == d_model && e.d_ff == d_ff && e.has_bias == (has_bias != 0)) return &e;
  return nullptr;
}

GroupedWs grouped_ws(int64_t T, int k, int D, int F) {
  auto al = [](size_t v) { return (v + 255) & ~(size_t)255; };
  const int64_t P = T * k;
  GroupedWs w;
  w.max_tiles = P + P / kTileM + 1;
  size_t o = 0;
  w.off_perm = o; o += al((size_t)P * 4);
  w.off_tiles = o; o += al((size_t)w.max_tiles * 16);
  w.off_ntiles = o; o += al(4);
  w.off_yp = o; o += al((size_t)P * D * 4);
  w.off_xq = o; o += al((size_t)T * D * 2);
  w.off_rsx = o; o += al((size_t)T * rs_pitch(D) * 4);
  w.off_hq = o; o += al((size_t)P * F * 2);
  w.off_rsh = o; o += al((size_t)P * rs_pitch(F) * 4);
  w.total = o;
  return w;
}

// (in launches of at most 2^30 pieces, so the kernel's indices fit 32 bits)
static void launch_prep(const uint16_t *src, int64_t rows, int K, uint16_t *dst, float *rs,
                        hipStream_t s) {
  const int64_t chunk = ((int64_t)1 << 30) / (K / 8);
  for (int64_t r0 = 0; r0 < rows; r0 += chunk) {
    const int64_t nr = std::min(chunk, rows - r0);
    const int64_t n = nr * (K / 8);
    hipLaunchKernelGGL(grouped_prep_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                       src + r0 * K, nr, K, dst + r0 * K, rs + r0 * rs_pitch(K));
  }
}

void launch_grouped(const GroupedLaunch *G, const PoolArgs &pa, const int32_t *refs,
                    const float *scores, const uint16_t *x, int T, int k, uint16_t *out,
                    float *out32, char *ws, int act, float alpha, float limit,
                    hipStream_t s) {
  const int D = G->d_model, F = G->d_ff, P = T * k;
  const GroupedWs w = grouped_ws(T, k, D, F);
  int32_t *perm = reinterpret_cast<int32_t *>(ws + w.off_perm);
  int4 *tiles = reinterpret_cast<int4 *>(ws + w.off_tiles);
  int32_t *ntiles = reinterpret_cast<int32_t *>(ws + w.off_ntiles);
  float *yp = reinterpret_cast<float *>(ws + w.off_yp);
  uint16_t *xq = reinterpret_cast<uint16_t *>(ws + w.off_xq);
  float *rsx = reinterpret_cast<float *>(ws + w.off_rsx);
  uint16_t *hq = reinterpret_cast<uint16_t *>(ws + w.off_hq);
  float *rsh = reinterpret_cast<float *>(ws + w.off_rsh);
  const int nkeys = pa.n_slots + pa.n_records;
  const int64_t xpieces = (int64_t)T * (D / 8);
  if (xpieces < ((int64_t)1 << 30)) {   // grouping and x prep in one launch
    hipLaunchKernelGGL(group_prep_kernel, dim3((unsigned)(1 + (xpieces + 1023) / 1024)), dim3(1024),
                       (size_t)nkeys * 4, s, refs, P, pa.n_slots, pa.n_records, D, perm, tiles,
                       ntiles, yp, x, (int64_t)T, xq, rsx);
  } else {
    hipLaunchKernelGGL(group_pairs_kernel, dim3(1), dim3(1024), (size_t)nkeys * 4, s, refs, P,
                       pa.n_slots, pa.n_records, D, perm, tiles, ntiles, yp);
    launch_prep(x, T, D, xq, rsx, s);
  }
  // (at most one partial tile per slot reference in use)
  const int64_t max_tiles = std::min<int64_t>(P, nkeys) + P / kTileM;
  auto grid = [&](int nout, int nb) {
    const int64_t items = (max_tiles + 7) / 8 * 8 * ((nout + nb - 1) / nb);
    return dim3((unsigned)std::min<int64_t>(items, kGroupedMaxWGs));
  };
  G->gate_up(grid(F, G->nb_up), s, pa, xq, rsx, k, perm, tiles, ntiles, hq, rsh, act, alpha, limit);
  G->down(grid(D, G->nb_down), s, pa, hq, rsh, scores, perm, tiles, ntiles, yp);
  const int64_t n4 = (int64_t)T * D / 4;
  hipLaunchKernelGGL(combine_pairs_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0,
                     s, yp, T, k, D, out, out32);
}

}  // namespace moe
