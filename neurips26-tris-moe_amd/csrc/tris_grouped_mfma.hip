// Grouped compact3 expert GEMM on MFMA for decode-sized segments, reading
// dense (predecoded) split bitmaps.
//
// Arithmetic.  Every non-salient weight is the reference's exact fp16 value
// w[n,k] = s1 * fp16(C_j[k] * R_j[n,g]) with j = d if the split bit is set,
// else nd, and s1 = +-1 from qweight1 (TriSMoE_cuda_kernel.cu:665-774); the
// products are formed with packed fp16 multiplies (round to nearest even, as
// __hmul) on column factors staged negated (P_j = fp16(-C_j * R_j) = -fp16(C_j * R_j)
// exactly); the split bits pick P_d or P_nd and the sign bits flip it (mf_row_b).
// Salient columns (a few per cent, w = fp16(+-fp16(C0*R0) +- fp16(C1*R1))) are zero in
// that operand and get MFMA steps of their own.  Products with the activations are
// exact in fp32 and accumulate in fp32, as in the reference's tensor-core
// kernel (TriSMoE_cuda_kernel.cu:4889-5093).
//
// Operand layout of the decode kernel (v_mfma_f32_16x16x32_f16): A rows are up to 16 rows
// of one segment (a sub-tile of its row tile); lane group kg (lanes 16kg..16kg+15) supplies the 8 columns kg + 4i and
// kg + 4i + 16 (i < 4) of each 32-column packed row.  Activations and the column factors are
// staged in LDS in the same permuted column order, so each lane reads its 8
// values with one 16-byte LDS load.
//
// Work decomposition of the decode kernel: workgroup = 4 wavefronts = a run of 64-output
// tiles x one row tile (up to 4, 16, 32 or 64 rows of one segment) x one projection (blockIdx.z;
// two units of 4 wavefronts take two projections side by side).  The workgroup stages the rows' activations and the column factors of a 512-column
// chunk in LDS once; wavefront w then owns outputs [16w, 16w+16) of each tile over the whole
// chunk, two tiles at a time, while its weight words of the next two are in flight, so no
// partial sums cross wavefronts.  Salient columns are zero in that pass; afterwards each lane
// builds the exact salient weights of its column, and one or two more MFMA steps multiply the
// activations gathered at the salient columns by them, into the same fp32 accumulator.
// Requires each 64-column K tile to lie in a single group (the reference's UniformK64Groups
// case) and rank % 64 == 0.
//
// What bounds the decode kernel.  At decode sizes a launch is short (10 to 30 us), and three
// things share it: the operand build (VALU issue, see mf_row_b); the way to the first tile, a
// chain of dependent scalar and vector loads and some 700 instructions which every wavefront
// runs; and fetching the instructions, since a launch starts with a cold instruction cache.  So
// the kernel asks for its scalars and row indices at once, keeps the K loop rolled, and hides
// the sizes and the lane index from the compiler per row tile, which otherwise computes
// every address of the rare paths ahead of the loop.  T = 16 gate/up launch at the Mixtral shape
// 31.5 -> 27.7 us, T = 64 42.3 -> 36.3 us (32-row tiles: 32.3); OLMoE T = 16 gate/up 17.6 -> 12.7, down
// 16.3 -> 11.9 us; A3B T = 1024 gate/up 67 -> 49, down 113 -> 79 us (64-row tiles and even runs: 39 and 58).
#include <type_traits>

#include "tris_common.h"

namespace tris {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMfWaves = 4;
constexpr int kMfThreads = kMfWaves * kWave;
constexpr int kMfRows = 16;         // segment rows per workgroup tile
constexpr int kMfChunk = 512;       // K columns staged per pass
constexpr int kMfSalWin = 32;             // salient columns per MFMA pass
constexpr int kMfSalStride = kMfSalWin + 8;

struct MfmaProj {
  const uint16_t* hidden;     // [batch, rank], or [hidden_rows, rank] read through row_index
  uint16_t* out;              // [batch, N]
  const int32_t* decoded;     // [num_segments, nblk, 128]
  tris_compact3_payload p;
  const int64_t* row_index;   // null, or [batch]: segment row r reads hidden row row_index[r]
  int hidden_rows;            // row_index's range, or with partials the rows of each slice
  // null, or [slices][hidden_rows][rank] fp32 split-K partial sums of the backbone that produced the activations:
  // hidden row r is then fp16(the slices' sum, added in slice order) and `hidden` is not read (rank <= kMfChunk)
  const float* partials;
  int slices;
};

struct MfmaArgs {
  MfmaProj proj[2];
  const int32_t* expert_ids;
  const int32_t* segment_offsets;
  int num_segments;
  int batch;              // routed rows
  int decoded_by_expert;  // 0: decoded holds one slot per segment; 1: one per expert id (every expert decoded)
  // One token's combine in the launch (two units, proj[1] == proj[0]; null: none): the token's two routed rows are
  // row tiles 0 and 1, one a unit, and unit 0 writes dt(fp16(out_r0 * w_r0) + fp16(out_r1 * w_r1)) to comb_out.
  uint16_t* comb_out;
  const int32_t* comb_inv;  // inverse_perm [2]: the row of each pick
  const uint16_t* comb_w;   // fp16 routing weights [2], by pick
  int comb_bf16;            // comb_out is bf16 (else fp16)
};

// Position of column k (0..31) of a packed row in the staged order: lane group k % 4, elements 2 i and 2 i + 1 of it
// columns k % 4 + 4 i and 16 past that, so that a packed pair of weights takes its bits from the two halves of a word.
__device__ __forceinline__ int mf_perm32(int k) { return 8 * (k & 3) + 2 * ((k >> 2) & 3) + (k >> 4); }

// Nibbles 2i, 2i+1 (byte i) of eight fp4 values -> two fp16 (low nibble -> low half).
__device__ __forceinline__ f16x2 fp4x2_to_f16x2(uint32_t nib, int byte_sel) {
  switch (byte_sel) {
    case 0: return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(nib, 1.0f, 0);
    case 1: return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(nib, 1.0f, 1);
    case 2: return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(nib, 1.0f, 2);
    default: return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(nib, 1.0f, 3);
  }
}

__device__ __forceinline__ f16x2 u32_as_f16x2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
__device__ __forceinline__ uint32_t f16x2_as_u32(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }

// Same mapping as the in-kernel-decode GEMM (tris_grouped.hip), plus the segment's expert id, loaded
// in the same round trip as the segment lengths.
__device__ inline bool mf_map_row_tile(const int32_t* __restrict__ seg, const int32_t* __restrict__ expert_ids,
                                       int nseg, int tile, int row_tile, int* s_out, int* row0_out, int* rc_out,
                                       int* e_out) {
  const int lane = static_cast<int>(__lane_id());
  int base = 0;
  for (int c = 0; c < nseg; c += kWave) {
    const int i = c + lane;
    const int ic = i < nseg ? i : nseg - 1;
    const int lo = seg[ic];
    const int hi = seg[ic + 1];
    const int ex = expert_ids[ic];
    int t = 0;
    if (i < nseg) {
      const int len = hi - lo;
      t = len > 0 ? (len + row_tile - 1) / row_tile : 0;
    }
    const int incl = wave_incl_sum_i32(t);
    const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
    if (tile < base + total) {  // wave-uniform
      const uint64_t hit = __ballot(i < nseg && tile < base + incl);
      const int L = __builtin_amdgcn_readfirstlane(__ffsll(static_cast<unsigned long long>(hit)) - 1);
      const int local = tile - base - __builtin_amdgcn_readlane(incl - t, L);
      const int row0 = __builtin_amdgcn_readlane(lo, L) + local * row_tile;
      const int end = __builtin_amdgcn_readlane(hi, L);
      *s_out = c + L;
      *row0_out = row0;
      *rc_out = (end - row0) < row_tile ? (end - row0) : row_tile;
      *e_out = __builtin_amdgcn_readlane(ex, L);
      return true;
    }
    base += total;
  }
  return false;
}

// Row tiles of the segments (tiles of <= row_tile rows), scanned once: with at most 64 segments the
// scan stays in registers and mapping a row tile costs no memory access.
struct MfSegScan {
  int lo, hi, ex;  // this lane's segment (lane < nseg): row range and expert id
  int t, incl;     // its row tiles, inclusive prefix over lanes
  int total;       // row tiles of all segments (the same in every lane)
};

__device__ inline MfSegScan mf_scan_segments(const int32_t* __restrict__ seg, const int32_t* __restrict__ expert_ids,
                                             int nseg, int row_tile) {
  const int lane = static_cast<int>(__lane_id());
  MfSegScan r;
  r.total = 0;
  for (int c = 0; c < nseg; c += kWave) {
    const int i = c + lane;
    const int ic = i < nseg ? i : nseg - 1;
    const int lo = seg[ic];
    const int hi = seg[ic + 1];
    const int ex = expert_ids[ic];
    int t = 0;
    if (i < nseg) t = hi > lo ? (hi - lo + row_tile - 1) / row_tile : 0;
    const int incl = wave_incl_sum_i32(t);
    if (c == 0) {
      r.lo = lo;
      r.hi = hi;
      r.ex = ex;
      r.t = t;
      r.incl = incl;
    }
    r.total += __builtin_amdgcn_readlane(incl, kWave - 1);
  }
  return r;
}

// Row tile `tile` (< sc.total) -> segment, first row, row count and expert id.
__device__ inline void mf_map_scanned(const MfSegScan& sc, const int32_t* __restrict__ seg,
                                      const int32_t* __restrict__ expert_ids, int nseg, int tile, int row_tile,
                                      int* s_out, int* row0_out, int* rc_out, int* e_out) {
  if (nseg <= kWave) {
    const int lane = static_cast<int>(__lane_id());
    const uint64_t hit = __ballot(lane < nseg && tile < sc.incl);
    const int L = __builtin_amdgcn_readfirstlane(__ffsll(static_cast<unsigned long long>(hit)) - 1);
    const int local = tile - __builtin_amdgcn_readlane(sc.incl - sc.t, L);
    const int row0 = __builtin_amdgcn_readlane(sc.lo, L) + local * row_tile;
    const int end = __builtin_amdgcn_readlane(sc.hi, L);
    *s_out = L;
    *row0_out = row0;
    *rc_out = (end - row0) < row_tile ? (end - row0) : row_tile;
    *e_out = __builtin_amdgcn_readlane(sc.ex, L);
    return;
  }
  mf_map_row_tile(seg, expert_ids, nseg, tile, row_tile, s_out, row0_out, rc_out, e_out);
}

constexpr int kMfPR = kMfChunk / 32;         // packed rows per chunk
constexpr int kMfTiles = kMfChunk / kTileK;  // 64-column K tiles per chunk
constexpr int kMfQ1Stride = kTileOut + 1;    // words per staged qweight1 row (odd, so per-lane row reads spread over banks)
constexpr int kMfMaxGroups = 8;              // the 64 columns x G row-scale block is staged whole
// One output tile's weight words in LDS: qweight1 [kMfPR][kMfQ1Stride], split words [kMfPR][64],
// row_pack3 [64][kMfMaxGroups][2] (32-bit words; every piece 16-byte aligned).
constexpr int kMfTbQ1 = 0;
constexpr int kMfTbGw = kMfPR * kMfQ1Stride;
constexpr int kMfTbRs = kMfTbGw + kMfPR * kTileOut;
constexpr int kMfTbWords = kMfTbRs + kTileOut * kMfMaxGroups * 2;
static_assert(kMfTbGw % 4 == 0 && kMfTbRs % 4 == 0, "tile buffer pieces must be 16-byte aligned");
constexpr int kMfCus = 256;  // MI355X compute units
// Mean rows a segment from which the decode kernel takes 32-row tiles (64 in the compact layout): a segment's weights are
// then built once where two 16-row tiles would build them twice, but the taller instances hold more LDS and registers.
// Tall against 16-row tiles, segments of random length, us: 8 of N = 14336, rank 512, pair: mean 11 28.3 / 27.6, 13 30.5 /
// 31.3, 16 30.4 / 36.2, 24 31.7 / 44.8; 128 of N = 2048, rank 256, pair: 11 37.9 / 37.8, 13 38.1 / 42.4, 16 39.0 / 46.6.
// (One or two tiles a workgroup gain later: 64 of N = 1024, rank 256, one projection 11.3 / 9.5 at 12 and 12.9 / 11.9 at
// 24.)  With single-word loads: 8 of N = 8194, rank 512, pair: 12 22.7 / 20.9, 14 24.8 / 25.5, 17 24.5 / 27.4.
constexpr int kMfTallMinRows = 12;
constexpr int kMfTallMinRowsSingle = 17;
// Decode kernel: row-scale groups and salient slots per chunk its LDS holds; the compact variant (at most 4
// groups and 64 salient columns per expert, a rank of at most 256) stages half the columns.
constexpr int mf_groups_cap(bool compact) { return compact ? 4 : kMfMaxGroups; }
constexpr int mf_sal_slots(bool compact) { return compact ? 64 : kMfChunk; }
constexpr int mf_chunk(bool compact) { return compact ? kMfChunk / 2 : kMfChunk; }  // K columns staged
constexpr int mf_xstride(bool compact) { return mf_chunk(compact) + 8; }  // fp16 elements per staged row (pad breaks bank aliasing)
// per wavefront and tile: a zero word, the qweight1 and split words of 16 columns and their row-scale block
constexpr int mf_wave_alloc_bytes(bool compact) {
  return (4 + 2 * (mf_chunk(compact) / 32) * 16 + 16 * mf_groups_cap(compact) * 2) * 4;
}
constexpr int kMfRuns = kMfRows * (kMfChunk / 8) / kMfThreads;  // activation runs per thread of a unit

constexpr int kMfExchBytes = kMfThreads * 4 * 4;  // SwiGLU: the up unit's accumulators of a tile for the gate unit

// Bump allocation of 16-byte aligned pieces (byte offsets into dynamic LDS).
__host__ __device__ inline int mf_take(int* o, int b) {
  const int at = *o;
  *o += (b + 15) & ~15;
  return at;
}

// Static LDS of the decode kernel with `units` units and `rows` staged activation rows (as declared there).
constexpr int mf_static_lds_bytes(int units, int rows, bool compact) {
  return units * (rows * mf_xstride(compact) * 2 + mf_chunk(compact) * (2 + 2) + mf_sal_slots(compact) * (4 + 2 + 4) + 48 +
                  (mf_chunk(compact) / kTileK) * 8 +
                  2 * kMfWaves * mf_wave_alloc_bytes(compact)) +
         (units == 2 ? 2 * (rows > kMfRows ? rows / kMfRows : 1) * kMfExchBytes : 16);
}

struct MfChunk {       // a unit's staged chunk
  uint16_t* xs;        // [rows][mf_xstride] activations, staged column order; the column past the chunk is zero (decode)
  uint16_t* cds;       // -C_d, staged column order (0 for salient columns); decode: -C_nd follows
  uint16_t* cns;       // weight-stationary: -C_nd (0 for salient columns)
  // Weight-stationary kernel (natural column order):
  uint32_t* col_sal;   // C0 | C1 << 16, natural order
  uint16_t* sal_col;   // chunk column of the chunk's q-th salient column
  // Decode kernel, per salient slot q (slots past the chunk's salient count, up to the next multiple of
  // kMfSalWin, read as zero weights and zero activations):
  uint32_t* sal_w;     // bits 0-4: (column - 15) mod 32, the right rotation that puts the column's qweight1 bit
                       // at bit 15; bits 8-15: byte offset of its group's R0 | R1 in a column's row-scale block;
                       // bits 16-31: byte offset of its packed row in a wavefront's weight words
  uint16_t* sal_xo;    // byte offset of its activation in a staged row (the zero column for padding slots)
  uint32_t* sal_cp;    // C0 | C1 << 16 with both signs flipped (decode), or as stored (weight-stationary)
  uint16_t* sal_xi;    // weight-stationary: its position in the staged column order
  int32_t* meta;       // weight-stationary: [t < 8] group of K tile t (-1: none); [8] first salient index; [9] end
  uint2* goff;         // decode: per K tile, where a column's R_d | R_nd word lies in a tile's words: byte offset, and a
                       // mask of the lane's column offset (a K tile without a group reads the zero word: 0, 0)
};
struct MfTileBuf {     // one output tile's weight words
  uint32_t* q1;        // [kMfPR][kMfQ1Stride] qweight1 words of the tile's 64 columns
  uint32_t* gw;        // [kMfPR][64] predecoded split words
  uint32_t* rs;        // [64][G][2] row_pack3: R0 | R1 << 16, R_d | R_nd << 16
};

// Decode kernel: each wavefront loads only the weight words of its own 16 output columns of a tile, so no other
// wavefront waits for them: into registers (MfWaveRegs) while the tiles before are computed, then into its own LDS
// words.  Per tile: a zero word (read for K tiles without a group); packed rows 2 t and 2 t + 1 of a column together,
// qweight1 and split word each; the row-scale block [16 columns][G][R0 | R1, R_d | R_nd].
constexpr int kMfWCols = 16;
constexpr int kMfWw = 4;                            // word offset of the weight words (the zero word is word 0)
template <bool kCompact>
struct MfWaveWords {
  static constexpr int kPR = mf_chunk(kCompact) / 32;            // packed rows
  static constexpr int kRs = kMfWw + 2 * kPR * kMfWCols;         // word offset of the row scales
  static constexpr int kRsLane = kMfWCols * mf_groups_cap(kCompact) * 2 / kWave;  // row-scale words a lane loads
  static constexpr int kAlloc = kRs + kRsLane * kWave;
  static_assert(kRsLane * kWave == kMfWCols * mf_groups_cap(kCompact) * 2 && (kRsLane == 2 || kRsLane == 4),
                "one 8- or 16-byte row-scale load a lane");
  static_assert(kAlloc * 4 == mf_wave_alloc_bytes(kCompact) && kRs % 4 == 0, "LDS accounting");
};
template <bool kCompact>
struct MfWaveRegs {    // a tile's words in flight: lane l holds columns 4 (l % 4) .. + 3 of packed row l / 4, and
  uint32_t q[4], g[4], rs[MfWaveWords<kCompact>::kRsLane];  // row-scale words kRsLane l .. of the 16 columns' run
};
constexpr uint32_t kMfOob = 0x80000000u;  // a byte offset past every buffer (each is below 2 GiB): reads 0, drops stores

// Byte offset of 8 activation columns [c, c + 8) of segment row row0 + r (r < rc), or `oob` (an offset
// past the buffer: the load reads zeros) for rows outside the tile, columns past the rank and gathered
// rows whose index lies outside [0, hidden_rows).  With a row index the buffer resource covers all of
// hidden; without, it starts at row row0.  r is wave-uniform, so the index load is one scalar load.
__device__ __forceinline__ uint32_t mf_hidden_voff(const MfmaProj& pa, int row0, int r, int rc, int c, int rank,
                                                   uint32_t oob) {
  if (r >= rc || c >= rank) return oob;
  int64_t src = r;
  if (pa.row_index != nullptr) {
    src = pa.row_index[row0 + r];
    if (src < 0 || src >= pa.hidden_rows) return oob;
  }
  return static_cast<uint32_t>(src * rank + c) * 2u;
}

// The activation buffer resource of rows [row0, row0 + rc) and its size (the offset that reads zeros).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t mf_hidden_rsrc(const MfmaProj& pa, int row0, int rc, int rank,
                                                                 uint32_t* bytes) {
  if (pa.row_index != nullptr) {
    *bytes = static_cast<uint32_t>(pa.hidden_rows) * rank * 2u;
    return make_rsrc(pa.hidden, *bytes);
  }
  *bytes = static_cast<uint32_t>(rc) * rank * 2u;
  return make_rsrc(pa.hidden + static_cast<int64_t>(row0) * rank, *bytes);
}
// Raw buffer loads: voffset at or past the buffer size returns 0 without a memory access.
__device__ __forceinline__ uint32_t bload32(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
}
__device__ __forceinline__ uint64_t bload64(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
  return static_cast<uint64_t>(v[0]) | (static_cast<uint64_t>(v[1]) << 32);
}
__device__ __forceinline__ uint4 bload128(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
  return make_uint4(v[0], v[1], v[2], v[3]);
}
// Buffer loads straight into LDS (the weight-stationary kernel): lane l's 4 (16) bytes land at dst + 4l (16l); dst is
// wave-uniform.
__device__ __forceinline__ void dma32(__amdgpu_buffer_rsrc_t r, void* dst, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 4, voff, soff, 0, 0);
}
__device__ __forceinline__ void dma128(__amdgpu_buffer_rsrc_t r, void* dst, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voff, soff, 0, 0);
}

// Weight-stationary kernel: register-staged column loads of a unit's chunk, held between issue and write.
struct MfRegs {
  uint64_t cpv[2];    // col_pack3 of columns kc + utid, kc + utid + 256
  uint32_t cmt[2];    // their salient words
  int q2t[2];         // their packed rows' salient prefix
  int sbase0;         // salient prefix at the chunk's first packed row
  int32_t mv;         // metadata word (see mf_chunk_issue)
};

// Issue the register loads of the columns of chunk [kc, kc + 512) of one projection of expert e.  utid is the thread's
// index within its unit.  Every load is issued unconditionally (a branch around a load makes the compiler wait for it
// at the join); invalid lanes get an offset past their buffer, which reads 0, or a clamped index.
__device__ __forceinline__ void mf_chunk_issue(const MfmaProj& pa, int e, int kc, int utid, MfRegs& R) {
  const tris_compact3_payload& p = pa.p;
  const int rank = p.rank;
  const int packed_rows = rank / 32;  // rank % 64 == 0
  const int pr0 = kc / 32;
  const int npr = (packed_rows - pr0) < kMfPR ? (packed_rows - pr0) : kMfPR;
  const uint32_t col_bytes = static_cast<uint32_t>(rank) * 8u;
  const __amdgpu_buffer_rsrc_t r_col = make_rsrc(p.col_pack3 + static_cast<int64_t>(e) * rank, col_bytes);
  gmem_i32* cmap_e = as_gmem(p.c_map + static_cast<int64_t>(e) * packed_rows);
  gmem_i32* q2p_e = as_gmem(p.qweight2_sparse_prefix + static_cast<int64_t>(e) * (packed_rows + 1));
  gmem_i32* gidx_e = as_gmem(p.g_idx + static_cast<int64_t>(e) * rank);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int k = kc + utid + h * kMfThreads;
    const bool kv = k < rank;
    const int pr = kv ? (k >> 5) : 0;
    R.cpv[h] = bload64(r_col, kv ? static_cast<uint32_t>(k) * 8u : col_bytes, 0u);
    R.cmt[h] = static_cast<uint32_t>(cmap_e[pr]);
    R.q2t[h] = q2p_e[pr];
  }
  R.sbase0 = q2p_e[pr0];
  // metadata: utid 64..71 -> group of K tile utid - 64; 72 / 73 -> salient prefix at the chunk's
  // start / end
  gmem_i32* mp = q2p_e + pr0;
  if (utid >= 64 && utid < 72) {
    const int kt = kc + (utid - 64) * kTileK;
    mp = gidx_e + (kt < rank ? kt : rank - 1);
  } else if (utid == 73) {
    mp = q2p_e + pr0 + npr;
  }
  R.mv = *mp;
}

// Decode kernel: the columns of a unit's chunk, two neighbours a thread (2 utid and 2 utid + 1 of the chunk: one packed
// row and, with uniform groups, one group), held between issue and write.
struct MfColRegs {
  uint4 cp;      // their col_pack3 entries
  uint32_t cm;   // their packed row's salient word
  int q2t;       // its salient prefix
  int g;         // their group (g_idx)
  int sbase0;    // salient prefix at the chunk's first packed row (the same in every lane)
  int send;      // salient prefix at the chunk's end (the same in every lane)
};
template <bool kCompact>
__device__ __forceinline__ void mf_cols_issue(const MfmaProj& pa, int e, int kc, int utid, MfColRegs& R) {
  const tris_compact3_payload& p = pa.p;
  const int rank = p.rank;
  const int packed_rows = rank / 32;  // rank % 64 == 0
  const int end = kc + mf_chunk(kCompact) < rank ? kc + mf_chunk(kCompact) : rank;
  const __amdgpu_buffer_rsrc_t r_col =
      make_rsrc(p.col_pack3 + static_cast<int64_t>(e) * rank, static_cast<uint32_t>(rank) * 8u);
  const __amdgpu_buffer_rsrc_t r_cm =
      make_rsrc(p.c_map + static_cast<int64_t>(e) * packed_rows, static_cast<uint32_t>(packed_rows) * 4u);
  const __amdgpu_buffer_rsrc_t r_pre = make_rsrc(p.qweight2_sparse_prefix + static_cast<int64_t>(e) * (packed_rows + 1),
                                                 static_cast<uint32_t>(packed_rows + 1) * 4u);
  const __amdgpu_buffer_rsrc_t r_g = make_rsrc(p.g_idx + static_cast<int64_t>(e) * rank, static_cast<uint32_t>(rank) * 4u);
  // columns past the rank read zeros (zero factors, not salient)
  const uint32_t k = static_cast<uint32_t>(kc + 2 * utid);
  R.cp = bload128(r_col, k * 8u, 0u);
  R.cm = bload32(r_cm, (k >> 5) * 4u, 0u);
  R.q2t = static_cast<int>(bload32(r_pre, (k >> 5) * 4u, 0u));
  R.g = static_cast<int>(bload32(r_g, k * 4u, 0u));
  R.sbase0 = static_cast<int>(bload32(r_pre, static_cast<uint32_t>(kc / 32) * 4u, 0u));
  R.send = static_cast<int>(bload32(r_pre, static_cast<uint32_t>(end / 32) * 4u, 0u));
}

// Writes the columns to LDS (waits for their loads): the factors of the main pass, staged negated (-C * R rounds to
// exactly -fp16(C * R), so a set qweight1 bit is the selectors' sign bit) and zero for salient columns, whatever their
// selector bits; the salient slots; the K tiles' row-scale offsets; the zero columns of the rc staged rows.  sal_cap:
// the slots staged (a payload whose prefix counts disagree with its salient map writes no slot past them).
template <bool kCompact, bool kByTile = false>
__device__ __forceinline__ void mf_cols_write(const MfmaProj& pa, int rc, int kc, int utid, const MfChunk& ch,
                                              const MfColRegs& R, int sal_cap) {
  constexpr int kChunk = mf_chunk(kCompact);
  const int rank = pa.p.rank;
  const int G = pa.p.num_groups;
  const int j = 2 * utid;
  const int pos = (j & ~31) + mf_perm32(j & 31);  // the second column's is pos + 8
  // the column's place in the row-scale block: its group, or (kByTile: the block holds a pair per K tile) its K tile
  const bool gv = kByTile || (R.g >= 0 && R.g < G);
  const int place = kByTile ? j >> 6 : (gv ? R.g : 0);
  const int bit = j & 31;
  const uint32_t sal = kc + j < rank ? (R.cm >> bit) & 3u : 0u;
  const uint32_t cdn[2] = {R.cp.y ^ 0x80008000u, R.cp.w ^ 0x80008000u};  // C_d | C_nd << 16
  if (j < kChunk) {  // wave-uniform
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const uint32_t v = (sal >> h) & 1u ? 0u : cdn[h];
      ch.cds[pos + 8 * h] = static_cast<uint16_t>(v);
      ch.cds[kChunk + pos + 8 * h] = static_cast<uint16_t>(v >> 16);
    }
    // (a column that is not salient writes the spare slot sal_cap, so that no load is put off into a branch and waited
    // for there, with every load issued after it)
    int q = R.q2t - R.sbase0 + __popc(R.cm & ((1u << bit) - 1u));
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // the column's group as the main pass takes it (uniform 64-column groups); an invalid group gives
      // zero factors, as a K tile without a group does
      const bool is = ((sal >> h) & 1u) != 0u;
      const int at = is && q >= 0 && q < sal_cap ? q : sal_cap;
      ch.sal_w[at] = (static_cast<uint32_t>((j >> 6) * kMfWCols * 16 + ((j >> 5) & 1) * 8) << 16) |
                     (static_cast<uint32_t>(place * 8) << 8) | (static_cast<uint32_t>(bit + h - 15) & 31u);
      ch.sal_xo[at] = static_cast<uint16_t>((pos + 8 * h) * 2);
      ch.sal_cp[at] = (gv ? (h ? R.cp.z : R.cp.x) : 0u) ^ 0x80008000u;
      q += is ? 1 : 0;
    }
    if ((utid & 31) == 0) {  // the first column of K tile utid / 32
      ch.goff[utid >> 5] = kc + j < rank && gv ? make_uint2(static_cast<uint32_t>(MfWaveWords<kCompact>::kRs * 4 + place * 8 + 4), ~0u)
                                               : make_uint2(0u, 0u);
    }
  }
  if (utid < kMfSalWin) {
    // padding slots up to the last window's end read the zero activation column with zero factors
    const int nsal = R.send - R.sbase0;
    const int q = nsal + utid;
    if (q >= 0 && q < sal_cap && q < ((nsal + kMfSalWin - 1) & ~(kMfSalWin - 1))) {
      ch.sal_w[q] = 0u;
      ch.sal_xo[q] = static_cast<uint16_t>(kChunk * 2);
      ch.sal_cp[q] = 0x80008000u;
    }
  }
  // the zero column (and its neighbour, so that row 0 holds an aligned zero word)
  if (utid < rc) *reinterpret_cast<uint32_t*>(&ch.xs[utid * mf_xstride(kCompact) + kChunk]) = 0u;
}

// Activation rows of a unit's chunk, 8 columns a lane: a wavefront's load h takes kRpl rows (one of 512 columns, two of
// 256), and the four wavefronts neighbouring ones.
template <int kRows, bool kCompact>
struct MfRowRegs {
  static constexpr int kRpl = kMfChunk / mf_chunk(kCompact);  // rows a load
  static constexpr int kRuns = (kRows + 4 * kRpl - 1) / (4 * kRpl);
  uint4 xv[kRuns];
};

// Issue the loads of the row tile's rows: lane tok0 + r of roff holds the byte offset of row r in r_hid, or kMfOob (rows
// past the tile, index entries that name no hidden row: they read zeros, as columns past the rank do).
template <int kRows, bool kCompact>
__device__ __forceinline__ void mf_rows_issue(__amdgpu_buffer_rsrc_t r_hid, int rank, int kc, int wave, int lane,
                                              uint32_t roff, int tok0, MfRowRegs<kRows, kCompact>& R) {
  constexpr int kRpl = MfRowRegs<kRows, kCompact>::kRpl;
  const int c = kc + (lane % (kWave / kRpl)) * 8;
  const uint32_t col = c < rank ? static_cast<uint32_t>(c) * 2u : kMfOob;
#pragma unroll
  for (int h = 0; h < MfRowRegs<kRows, kCompact>::kRuns; ++h) {
    const int at = tok0 + kRpl * (4 * h + wave);  // wave-uniform
    uint32_t ro = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(roff), at & (kWave - 1)));
    if constexpr (kRpl == 2) {
      const uint32_t r1 = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(roff), (at + 1) & (kWave - 1)));
      ro = lane < kWave / 2 ? ro : r1;
    }
    R.xv[h] = bload128(r_hid, __builtin_elementwise_add_sat(ro, col), 0u);
  }
}

// Writes the loaded rows to LDS in the staged order.
template <int kRows, bool kCompact>
__device__ __forceinline__ void mf_rows_write(const MfRowRegs<kRows, kCompact>& R, int rc, int wave, int lane,
                                              uint16_t* xs) {
  constexpr int kRpl = MfRowRegs<kRows, kCompact>::kRpl;
  const int c = (lane % (kWave / kRpl)) * 8;  // run start within the chunk
  uint16_t* const dst = xs + (c & ~31) + 2 * ((c >> 2) & 3) + ((c >> 4) & 1);
#pragma unroll
  for (int h = 0; h < MfRowRegs<kRows, kCompact>::kRuns; ++h) {
    const int r0 = kRpl * (4 * h + wave);  // wave-uniform
    if (r0 < rc) {
      const int r = kRpl == 2 ? r0 + lane / (kWave / kRpl) : r0;
      const uint32_t w[4] = {R.xv[h].x, R.xv[h].y, R.xv[h].z, R.xv[h].w};
      if (kRpl == 1 || r < rc) {
#pragma unroll
        for (int x = 0; x < 8; ++x) {  // column c + x
          dst[r * mf_xstride(kCompact) + 8 * (x & 3) + 2 * (x >> 2)] = static_cast<uint16_t>(w[x >> 1] >> (16 * (x & 1)));
        }
      }
    }
  }
}

// Weight-stationary kernel: write the register-staged columns to LDS in natural order (waits for those loads).  Salient
// columns get zero C_d / C_nd, so the main pass gives them zero weights whatever their selector bits.
__device__ __forceinline__ void mf_chunk_write(const MfmaProj& pa, int kc, int utid, const MfChunk& ch,
                                               const MfRegs& R) {
  const tris_compact3_payload& p = pa.p;
  const int rank = p.rank;
  const int G = p.num_groups;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int j = utid + h * kMfThreads;
    const int k = kc + j;
    const int bit = k & 31;
    const uint32_t cm = R.cmt[h];
    const bool sal = k < rank && ((cm >> bit) & 1u);
    // staged negated (-C * R rounds to exactly -fp16(C * R)), so a set qweight1 bit is the selectors' sign bit
    ch.cds[j] = sal ? static_cast<uint16_t>(0) : static_cast<uint16_t>((R.cpv[h] >> 32) ^ 0x8000u);
    ch.cns[j] = sal ? static_cast<uint16_t>(0) : static_cast<uint16_t>((R.cpv[h] >> 48) ^ 0x8000u);
    ch.col_sal[j] = static_cast<uint32_t>(R.cpv[h]);
    if (sal) {
      const int q = R.q2t[h] - R.sbase0 + __popc(cm & ((1u << bit) - 1u));
      ch.sal_col[q] = static_cast<uint16_t>(j);
      ch.sal_xi[q] = static_cast<uint16_t>((j & ~31) + mf_perm32(j & 31));
      ch.sal_cp[q] = static_cast<uint32_t>(R.cpv[h]);
    }
  }
  if (utid >= 64 && utid < 72) {
    const bool tv = kc + (utid - 64) * kTileK < rank && R.mv >= 0 && R.mv < G;
    ch.meta[utid - 64] = tv ? R.mv : -1;
  } else if (utid >= 72 && utid < 74) {
    ch.meta[8 + (utid - 72)] = R.mv;
  }
}

// Activation rows [row0, row0 + rc) of the one chunk (rank <= kMfChunk) from the split-K partial sums of the backbone
// that produced them: fp16 of the slices' sum added in slice order, the bits the backbone's own reduction
// (backbone_reduce_at) writes.  Thread utid of the unit takes columns 2 utid and 2 utid + 1 of each row, with
// kMfPartialBatch slices' loads in flight.
constexpr int kMfPartialBatch = 16;
template <bool kCompact>
__device__ __forceinline__ void mf_partials_stage(const MfmaProj& pa, int row0, int rc, int utid, const MfChunk& ch) {
  const int rank = pa.p.rank;
  const int c = 2 * utid;
  const int slices = pa.slices;
  const int prow = pa.hidden_rows;
  const uint32_t bytes = static_cast<uint32_t>(slices) * static_cast<uint32_t>(prow) * rank * 4u;
  const __amdgpu_buffer_rsrc_t r = make_rsrc(pa.partials, bytes);
  const int pos0 = (c & ~31) + mf_perm32(c & 31);
  const int pos1 = ((c + 1) & ~31) + mf_perm32((c + 1) & 31);
  for (int i = 0; i < rc; ++i) {  // uniform
    float a0 = 0.0f, a1 = 0.0f;
    for (int s0 = 0; s0 < slices; s0 += kMfPartialBatch) {
      uint64_t v[kMfPartialBatch];
#pragma unroll
      for (int j = 0; j < kMfPartialBatch; ++j) {
        const bool ok = s0 + j < slices && c < rank;
        v[j] = bload64(r, ok ? static_cast<uint32_t>(((s0 + j) * prow + row0 + i) * rank + c) * 4u : bytes, 0u);
      }
#pragma unroll
      for (int j = 0; j < kMfPartialBatch; ++j) {
        if (s0 + j < slices) {
          a0 += __uint_as_float(static_cast<uint32_t>(v[j]));
          a1 += __uint_as_float(static_cast<uint32_t>(v[j] >> 32));
        }
      }
    }
    if (c < rank) {
      ch.xs[i * mf_xstride(kCompact) + pos0] = f2h_bits(a0);
      ch.xs[i * mf_xstride(kCompact) + pos1] = f2h_bits(a1);
    }
  }
}

// LDS copies of one output tile's weight words for chunk kc: qweight1 and split words (wave w of the
// unit copies packed rows w, w + 4, ...) and the 64 x G row-scale block.  Wave-uniform conditions
// only; the caller waits (s_waitcnt) before reading.
__device__ __forceinline__ void mf_tile_issue(const MfmaProj& pa, int s, int e, int kc, int ob, int utid,
                                              const MfTileBuf& tb) {
  const tris_compact3_payload& p = pa.p;
  const int N = p.outfeatures;
  const int rank = p.rank;
  const int G = p.num_groups;
  const int wave = __builtin_amdgcn_readfirstlane(utid / kWave);  // wave-uniform
  const int lane = utid % kWave;
  const int packed_rows = rank / 32;
  const int nob = ceil_div(N, kTileOut);
  const int nblk = (packed_rows / 2) * nob;
  const int pr0 = kc / 32;
  const int npr = (packed_rows - pr0) < kMfPR ? (packed_rows - pr0) : kMfPR;
  const int n0 = ob * kTileOut;
  const uint32_t q1_bytes = static_cast<uint32_t>(packed_rows) * N * 4u;
  const __amdgpu_buffer_rsrc_t r_q1 = make_rsrc(p.qweight1 + static_cast<int64_t>(e) * packed_rows * N, q1_bytes);
  const __amdgpu_buffer_rsrc_t r_dec =
      make_rsrc(pa.decoded + static_cast<int64_t>(s) * nblk * kGrWords, static_cast<uint32_t>(nblk) * kGrWords * 4u);
  const int n = n0 + lane;
  const uint32_t v_q1 = n < N ? static_cast<uint32_t>(n) * 4u : q1_bytes;
#pragma unroll
  for (int jj = 0; jj < kMfPR / kMfWaves; ++jj) {
    const int j = wave + kMfWaves * jj;
    if (j < npr) {
      const uint32_t pr = static_cast<uint32_t>(pr0 + j);
      dma32(r_q1, tb.q1 + j * kMfQ1Stride, v_q1, pr * N * 4u);
      dma32(r_dec, tb.gw + j * kTileOut, static_cast<uint32_t>(lane) * 4u,
            ((((pr >> 1) * nob) + ob) * kGrWords + (pr & 1u) * kTileOut) * 4u);
    }
  }
  // row_pack3[e][n0 .. n0 + 63][0 .. G - 1] is one contiguous block; columns >= N read 0
  const __amdgpu_buffer_rsrc_t r_rs =
      make_rsrc(p.row_pack3 + (static_cast<int64_t>(e) * N + n0) * G, static_cast<uint32_t>(N - n0) * G * 8u);
  const int kb = ceil_div(kTileOut * G * 8, 1024);  // <= 4 KiB (G <= kMfMaxGroups)
  for (int b = wave; b < kb; b += kMfWaves) {
    dma128(r_rs, reinterpret_cast<unsigned char*>(tb.rs) + b * 1024, static_cast<uint32_t>(b * 1024 + lane * 16), 0u);
  }
}

// Where a wavefront's words of output tile 0 lie for chunk kc: expert e's tensors (wave-uniform; the tile's own
// columns are added to the bases) and the lane's byte offsets.
struct MfWaveSrc {
  const uint32_t* q1;    // qweight1[e] [packed rows][N]
  const uint32_t* dec;   // the segment's predecoded blocks [packed rows / 2][tiles][128]
  const uint32_t* rs;    // row_pack3[e], the wavefront's columns of tile 0
  uint32_t q1_bytes, dec_bytes;
  int rs_cols;           // columns from the wavefront's first to the expert's last
  uint32_t v_q1, v_dec;  // lane l: packed row kc / 32 + l / 4, columns 16 wave + 4 (l % 4) ..
};
template <bool kCompact>
__device__ __forceinline__ MfWaveSrc mf_wave_src(const MfmaProj& pa, int s, int e, int kc, int wave, int lane) {
  const tris_compact3_payload& p = pa.p;
  const int N = p.outfeatures;
  const int packed_rows = p.rank / 32;
  const int nob = ceil_div(N, kTileOut);
  const int nblk = (packed_rows / 2) * nob;
  const uint32_t pr = static_cast<uint32_t>(kc / 32 + lane / 4);
  const uint32_t c = static_cast<uint32_t>(kMfWCols * wave + 4 * (lane % 4));
  MfWaveSrc w;
  w.q1 = reinterpret_cast<const uint32_t*>(p.qweight1) + static_cast<int64_t>(e) * packed_rows * N;
  w.dec = reinterpret_cast<const uint32_t*>(pa.decoded) + static_cast<int64_t>(s) * nblk * kGrWords;
  w.rs = reinterpret_cast<const uint32_t*>(p.row_pack3) +
         (static_cast<int64_t>(e) * N + kMfWCols * wave) * (2 * p.num_groups);
  w.q1_bytes = static_cast<uint32_t>(packed_rows) * N * 4u;
  w.dec_bytes = static_cast<uint32_t>(nblk) * kGrWords * 4u;
  w.rs_cols = N - kMfWCols * wave;
  // packed rows past the rank (or past the staged chunk's) read nothing
  const bool rv = static_cast<int>(pr) < packed_rows && lane / 4 < MfWaveWords<kCompact>::kPR;
  w.v_q1 = rv ? (pr * N + c) * 4u : kMfOob;
  w.v_dec = rv ? ((pr >> 1) * nob * kGrWords + (pr & 1u) * kTileOut + c) * 4u : kMfOob;
  return w;
}

// kWords consecutive words at byte offset voff: one load, or with kSingle one a word (a load that straddles the buffer's
// end, for column counts that are no multiple of 4, must still return the words inside it).
template <int kWords, bool kSingle>
__device__ __forceinline__ void bload_words(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t* dst) {
  if constexpr (kSingle) {
#pragma unroll
    for (int i = 0; i < kWords; ++i) dst[i] = bload32(r, voff + 4u * i, 0u);
  } else if constexpr (kWords == 4) {
    const uint4 v = bload128(r, voff, 0u);
    dst[0] = v.x, dst[1] = v.y, dst[2] = v.z, dst[3] = v.w;
  } else {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, 0u, 0);
    dst[0] = v[0], dst[1] = v[1];
  }
}

// Issues the wavefront's loads of its 16 columns of output tile ob: one 16-byte load a lane for the packed rows'
// qweight1 words, one for their split words, one for the row scales (16 / 16 / 8 or 16 bytes; kSingle: a word at a time).
// An offset past its buffer reads zeros, and what lies inside it but past the groups or column N (the next row's words,
// the next tile's block) only feeds scales that are not read or output columns that are not stored.  valid = false (a prefetch with no tile to fetch, wave-uniform)
// empties the buffers, so every load reads zeros without a memory access: a workgroup does not fetch the tile after
// its run, which another workgroup reads (likely through another XCD's L2).
template <bool kCompact, bool kSingle>
__device__ __forceinline__ void mf_wave_words_issue(const MfWaveSrc& w, int ob, MfWaveRegs<kCompact>& r, bool valid) {
  const uint32_t col = static_cast<uint32_t>(ob) * kTileOut;
  const __amdgpu_buffer_rsrc_t r_q1 = make_rsrc(w.q1 + col, valid ? w.q1_bytes - col * 4u : 0u);
  const __amdgpu_buffer_rsrc_t r_dec =
      make_rsrc(w.dec + static_cast<uint32_t>(ob) * kGrWords, valid ? w.dec_bytes - static_cast<uint32_t>(ob) * kGrWords * 4u : 0u);
  bload_words<4, kSingle>(r_q1, w.v_q1, r.q);
  bload_words<4, kSingle>(r_dec, w.v_dec, r.g);
}
template <bool kCompact, bool kSingle>
__device__ __forceinline__ void mf_wave_tile_issue(const MfWaveSrc& w, int G, int ob, int lane,
                                                   MfWaveRegs<kCompact>& r, bool valid = true) {
  constexpr int kRsLane = MfWaveWords<kCompact>::kRsLane;
  const uint32_t col = static_cast<uint32_t>(ob) * kTileOut;
  mf_wave_words_issue<kCompact, kSingle>(w, ob, r, valid);
  const int ncols = valid ? w.rs_cols - static_cast<int>(col) : 0;  // the wavefront's columns to the expert's last
  const __amdgpu_buffer_rsrc_t r_rs = make_rsrc(w.rs + (ncols > 0 ? static_cast<int64_t>(col) * 2 * G : 0),
                                                ncols > 0 ? static_cast<uint32_t>(ncols) * G * 8u : 0u);
  bload_words<kRsLane, kSingle>(r_rs, static_cast<uint32_t>(lane * kRsLane) * 4u, r.rs);
}

// Writes the loaded words to the wavefront's LDS words wb of that tile (this waits for the loads).
template <bool kCompact>
__device__ __forceinline__ void mf_wave_tile_write(const MfWaveRegs<kCompact>& r, int lane, uint32_t* wb) {
  constexpr int kRsLane = MfWaveWords<kCompact>::kRsLane;
  const int row = lane / 4;
  uint32_t* dst = wb + kMfWw + ((row >> 1) * kMfWCols + 4 * (lane % 4)) * 4 + (row & 1) * 2;
  if (!kCompact || row < MfWaveWords<kCompact>::kPR) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2*>(dst + 4 * i) = make_uint2(r.q[i], r.g[i]);
  }
  if constexpr (kRsLane == 4) {
    *reinterpret_cast<uint4*>(wb + MfWaveWords<kCompact>::kRs + lane * 4) = make_uint4(r.rs[0], r.rs[1], r.rs[2], r.rs[3]);
  } else {
    *reinterpret_cast<uint2*>(wb + MfWaveWords<kCompact>::kRs + lane * 2) = make_uint2(r.rs[0], r.rs[1]);
  }
}

// Exact B operand of the lane's column for packed row j: the 8 weights k = kg + 4 i and kg + 4 i + 16 (i < 4).  Per pair
// a 16-bit mask of the two split bits (shifted to each half's top bit, then an arithmetic shift) picks fp16(-C_d * R_d)
// or fp16(-C_nd * R_nd), and the two qweight1 bits, at each half's bit 0, times 0x8000 are added to the halves: the sum
// mod 2^16 flips the sign where the bit is set, to +fp16(C * R).  left = 3 - kg; right = kg.
// Bound by VALU issue.  Picking the terms by fp4 selectors (two v_cvt_scalef32_pk_f16_fp4, a product and a
// fused multiply-add a pair) took 148 cycles a packed row with three wavefronts a SIMD, this form 132.
__device__ __forceinline__ f16x8 mf_row_b(uint32_t qw, uint32_t gw, const uint4& cdv, const uint4& cnv, uint32_t rs2,
                                          uint32_t left, uint32_t right) {
  const f16x2 r = u32_as_f16x2(rs2);
  const f16x2 rd2 = __builtin_shufflevector(r, r, 0, 0);  // (operand selects of the packed products)
  const f16x2 rn2 = __builtin_shufflevector(r, r, 1, 1);
  const uint32_t cd[4] = {cdv.x, cdv.y, cdv.z, cdv.w};
  const uint32_t cn[4] = {cnv.x, cnv.y, cnv.z, cnv.w};
  const uint32_t g = gw << left;
  const uint32_t q = qw >> right;
  uint32_t b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t pd = f16x2_as_u32(u32_as_f16x2(cd[i]) * rd2);
    const uint32_t pn = f16x2_as_u32(u32_as_f16x2(cn[i]) * rn2);
    uint32_t m, w;
    asm("v_pk_ashrrev_i16 %0, 15, %1 op_sel_hi:[0,1]" : "=v"(m) : "v"(g << (12 - 4 * i)));
    w = ((pd ^ pn) & m) ^ pn;
    asm("v_pk_mad_u16 %0, %1, %2, %0" : "+v"(w) : "v"(q >> (4 * i)), "s"(0x80008000u));
    b[i] = w;
  }
  return __builtin_bit_cast(f16x8, make_uint4(b[0], b[1], b[2], b[3]));
}

// Bit m of b (m < 8) to bit 4m.
__device__ __forceinline__ uint32_t spread8(uint32_t b) {
  b = (b | (b << 12)) & 0x000F000Fu;
  b = (b | (b << 6)) & 0x03030303u;
  return (b | (b << 3)) & 0x11111111u;
}

// mf_row_b for the natural column order: the lane's 8 weights are k = 8 kg + m (m < 8), so the A operand is 16
// contiguous bytes of an activation row.  The selector bits of those columns are byte kg of the packed words,
// spread to one nibble each.
__device__ __forceinline__ f16x8 mf_row_b_nat(uint32_t qw, uint32_t gw, const uint4& cdv, const uint4& cnv,
                                              uint32_t rs2, int kg) {
  const f16x2 r = u32_as_f16x2(rs2);
  const f16x2 rd2 = __builtin_shufflevector(r, r, 0, 0);  // (operand selects of the packed products)
  const f16x2 rn2 = __builtin_shufflevector(r, r, 1, 1);
  const uint32_t cd[4] = {cdv.x, cdv.y, cdv.z, cdv.w};
  const uint32_t cn[4] = {cnv.x, cnv.y, cnv.z, cnv.w};
  const uint32_t q4 = spread8(__builtin_amdgcn_ubfe(qw, 8u * kg, 8u));
  const uint32_t g4 = spread8(__builtin_amdgcn_ubfe(gw, 8u * kg, 8u));
  const uint32_t sd = (g4 << 1) | (q4 << 3);  // d term: fp4 +-1.0, else +-0; bit 3 = qweight1 (negated factors)
  const uint32_t sn = sd ^ 0x22222222u;                        // nd term: the others
  uint32_t b[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f16x2 pd = u32_as_f16x2(cd[i]) * rd2;
    const f16x2 pn = u32_as_f16x2(cn[i]) * rn2;
    const f16x2 tn = fp4x2_to_f16x2(sn, i) * pn;
    b[i] = f16x2_as_u32(__builtin_elementwise_fma(fp4x2_to_f16x2(sd, i), pd, tn));
  }
  return __builtin_bit_cast(f16x8, make_uint4(b[0], b[1], b[2], b[3]));
}

// Salient window [w0, w0 + wn) of the chunk (wn <= kMfSalWin): lane group kg writes the exact fp16 weights
// w = fp16(+-fp16(C0 * R0) +- fp16(C1 * R1)) of column tc for window slots kg, kg + 4, ... into its wave's
// ws row i16 (every slot, zero past wn, with no per-slot branch so the LDS reads overlap).  q2w holds the
// lane's qweight2_sparse words of rows q2b and q2b + 1 (a window spans at most two).
__device__ __forceinline__ void mf_salient_weights(const MfChunk& ch, const MfTileBuf& tb, const uint32_t* r01t,
                                                   int tc, int kg, int wave, int i16, int sbase0, int w0, int wn,
                                                   int q2b, const uint32_t q2w[2], uint16_t (*ws)[16][kMfSalStride]) {
  uint16_t wv[kMfSalWin / 4];
#pragma unroll
  for (int u = 0; u < kMfSalWin / 4; ++u) {
    const int q = 4 * u + kg;
    const bool qv = q < wn;
    const int c = ch.sal_col[w0 + (qv ? q : 0)];  // chunk column
    const uint32_t w1 = tb.q1[(c >> 5) * kMfQ1Stride + tc];
    const uint32_t rr = r01t[(c >> 6) * kTileOut + tc];
    const uint32_t cp = ch.col_sal[c];
    const int sidx = sbase0 + w0 + q;  // qweight2_sparse index
    const uint32_t q2 = ((sidx >> 5) - q2b) == 0 ? q2w[0] : q2w[1];
    // sign bits: positive where the qweight1 / qweight2 bit is set
    const uint32_t neg = ((~(w1 >> (c & 31)) & 1u) << 15) | ((~(q2 >> (sidx & 31)) & 1u) << 31);
    const f16x2 t = __builtin_bit_cast(f16x2, f16x2_as_u32(u32_as_f16x2(cp) * u32_as_f16x2(rr)) ^ neg);
    const _Float16 w = t[0] + t[1];
    wv[u] = qv ? __builtin_bit_cast(uint16_t, w) : static_cast<uint16_t>(0);
  }
#pragma unroll
  for (int u = 0; u < kMfSalWin / 4; ++u) ws[wave][i16][4 * u + kg] = wv[u];
}

// Both MFMA operands of the salient window starting at slot w0, built in registers: lane (i16, kg) takes window
// slots 8 kg .. 8 kg + 7.  bv[b] holds the exact fp16 weights of its column of tile b, w = fp16(+-fp16(C0 * R0) +-
// fp16(C1 * R1)) (both products in one packed multiply), and av[m] its activation row xr[m] at those slots'
// columns.  The staged slot words carry every column-dependent offset, so a slot costs three LDS reads (its
// qweight1 word, its group's R0 | R1, its activation) and no masking: padding slots read zero factors and the
// zero activation column.  q1_lane / rs_lane: the byte offsets of the lane's column in the wavefront's qweight1
// words and in its row-scale block (of wb); q2w: the lane's qweight2_sparse words of rows (sbase0 + w0) / 32 and the next
// (a window spans at most two), q2off = (sbase0 + w0) % 32 + 8 kg the bit of slot 0 in q2w[0] | q2w[1] << 32.
template <int kNs, int kRt, bool kCompact>
__device__ __forceinline__ void mf_salient_operands(const MfChunk& ch, const uint32_t* wb,
                                                    const uint16_t* const (&xr)[kRt], uint32_t q1_lane,
                                                    uint32_t rs_lane, int kg, int w0, int q2off,
                                                    const uint32_t (&q2w)[kNs][2], f16x8 (&av)[kRt],
                                                    f16x8 (&bv)[kNs]) {
  constexpr int kStride = MfWaveWords<kCompact>::kAlloc;
  const int s0 = w0 + 8 * kg;  // a multiple of 8: the slot vectors are 16-byte aligned
  const uint4 swa = *reinterpret_cast<const uint4*>(&ch.sal_w[s0]);
  const uint4 swb = *reinterpret_cast<const uint4*>(&ch.sal_w[s0 + 4]);
  const uint4 xov = *reinterpret_cast<const uint4*>(&ch.sal_xo[s0]);
  const uint32_t sw[8] = {swa.x, swa.y, swa.z, swa.w, swb.x, swb.y, swb.z, swb.w};
  const uint32_t xo[4] = {xov.x, xov.y, xov.z, xov.w};
  uint32_t w1v[kNs][8], rrv[kNs][8], a16[kRt][8];
#pragma unroll
  for (int u = 0; u < 8; ++u) {  // every read issued before any is used
#pragma unroll
    for (int b = 0; b < kNs; ++b) {
      const unsigned char* q1b = reinterpret_cast<const unsigned char*>(wb + b * kStride + kMfWw) + q1_lane;
      const unsigned char* rsb = reinterpret_cast<const unsigned char*>(wb + b * kStride + MfWaveWords<kCompact>::kRs) + rs_lane;
      w1v[b][u] = *reinterpret_cast<const uint32_t*>(q1b + (sw[u] >> 16));
      rrv[b][u] = *reinterpret_cast<const uint32_t*>(rsb + ((sw[u] >> 8) & 0xFFu));
    }
#pragma unroll
    for (int m = 0; m < kRt; ++m) {
      const unsigned char* xb = reinterpret_cast<const unsigned char*>(xr[m]);
      a16[m][u] = *reinterpret_cast<const uint16_t*>(xb + ((xo[u / 2] >> (16 * (u & 1))) & 0xFFFFu));
    }
  }
  const uint4 cpa = *reinterpret_cast<const uint4*>(&ch.sal_cp[s0]);
  const uint4 cpb = *reinterpret_cast<const uint4*>(&ch.sal_cp[s0 + 4]);
  const uint32_t cp[8] = {cpa.x, cpa.y, cpa.z, cpa.w, cpb.x, cpb.y, cpb.z, cpb.w};
#pragma unroll
  for (int b = 0; b < kNs; ++b) {
    // qweight2_sparse bits of the 8 slots: bit u of q2lo
    const uint32_t q2lo = static_cast<uint32_t>(((static_cast<uint64_t>(q2w[b][1]) << 32) | q2w[b][0]) >> q2off);
    uint32_t t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      // staged factors have both signs flipped; flip back where the qweight1 (bit 15) / qweight2 (bit 31) bit is
      // set (the positive weights)
      const uint32_t rot = __builtin_amdgcn_alignbit(w1v[b][u], w1v[b][u], sw[u]);  // column's bit at bit 15
      const uint32_t pos = (rot & 0x8000u) | ((q2lo << (31 - u)) & 0x80000000u);
      t[u] = f16x2_as_u32(u32_as_f16x2(cp[u]) * u32_as_f16x2(rrv[b][u])) ^ pos;
    }
    uint32_t wb[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t lo = __builtin_amdgcn_perm(t[2 * i + 1], t[2 * i], 0x05040100u);  // the C0 R0 terms
      const uint32_t hi = __builtin_amdgcn_perm(t[2 * i + 1], t[2 * i], 0x07060302u);  // the C1 R1 terms
      wb[i] = f16x2_as_u32(u32_as_f16x2(lo) + u32_as_f16x2(hi));
    }
    bv[b] = __builtin_bit_cast(f16x8, make_uint4(wb[0], wb[1], wb[2], wb[3]));
  }
#pragma unroll
  for (int m = 0; m < kRt; ++m) {
    uint32_t ab[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ab[i] = a16[m][2 * i] | (a16[m][2 * i + 1] << 16);
    av[m] = __builtin_bit_cast(f16x8, make_uint4(ab[0], ab[1], ab[2], ab[3]));
  }
}

// A staged chunk's first salient index and its salient count, in scalar registers, the count held to the slots staged.
struct MfChunkMeta {
  int sbase0, num_sal;
};
__device__ __forceinline__ MfChunkMeta mf_chunk_meta(const MfColRegs& R, int sal_cap) {
  MfChunkMeta r;
  r.sbase0 = __builtin_amdgcn_readfirstlane(R.sbase0);
  const int n = __builtin_amdgcn_readfirstlane(R.send) - r.sbase0;
  r.num_sal = n < 0 ? 0 : (n < sal_cap ? n : sal_cap);
  return r;
}

// The lane's qweight2_sparse words of the chunk's first salient window (a window of kMfSalWin salient columns spans at
// most two qweight2_sparse rows), for output column n.  Issued before the next tiles' loads, so that waiting for them does
// not wait for those.  q2: the expert's qweight2_sparse [q2rows][N].
__device__ __forceinline__ void mf_q2_issue(const uint32_t* q2, int q2rows, int N, int n, const MfChunkMeta& cm,
                                            uint32_t (&q2w)[2]) {
  const uint32_t v_q2 = n < N ? static_cast<uint32_t>(n) * 4u : kMfOob;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    // a row past the last: an empty resource
    const int row = (cm.sbase0 >> 5) + h;
    const bool rv = cm.num_sal > 0 && row < q2rows;
    const __amdgpu_buffer_rsrc_t r_q2 = make_rsrc(q2 + (rv ? static_cast<int64_t>(row) * N : 0),
                                                  rv ? static_cast<uint32_t>(N) * 4u : 0u);
    q2w[h] = bload32(r_q2, v_q2, 0u);
  }
}

// kNs output tiles over one staged chunk: adds rows 16 m + 4 kg + v, column n[b] of x . W^T to acc[b][m].  Every
// activation and column-factor read from LDS feeds all kNs tiles and every weight built all kRt row sub-tiles.
// xr[m]: the staged activation row this lane's A operand of sub-tile m reads.
//
// The K loop stays rolled, two packed rows (a K tile) an iteration.  A launch starts with a cold instruction cache, and
// its workgroups share few passes over the code: unrolled over the chunk, a pass was about 8 KB of instructions a tile
// and the first one of each wavefront took 20000 cycles against 8400 for the next (T = 16 gate/up; timestamps
// in the kernel), the difference being instruction fetch.
template <int kNs, int kRt, bool kCompact>
__device__ __forceinline__ void mf_compute(const uint32_t* q2, int q2rows, int N, int rank, int G, int kc,
                                           const int (&n)[kNs], const uint16_t* const (&xr)[kRt], int lane,
                                           const MfChunk& ch, const MfChunkMeta& cm, const uint32_t* wb,
                                           const uint32_t (&q2w0)[kNs][2], f32x4 (&acc)[kNs][kRt]) {
  const int i16 = lane % 16;   // MFMA column within the wave's 16 outputs / A row
  const int kg = lane / 16;    // MFMA k group: columns k = kg (mod 4) of every packed row
  constexpr int kStride = MfWaveWords<kCompact>::kAlloc;
  constexpr int kTiles = mf_chunk(kCompact) / kTileK;
  const int nt = (rank - kc) / kTileK < kTiles ? (rank - kc) / kTileK : kTiles;  // K tiles (rank % 64 == 0)

  // ---- MFMA over the chunk's packed rows (salient columns have zero factors here).  Each packed row's LDS reads
  // are issued as soon as the same row of the K tile before is computed.
  // the lane's column in the wavefront's row-scale block [16 columns][G][R0 | R1, R_d | R_nd]
  const uint32_t rs_lane = static_cast<uint32_t>(i16 * G * 8);
  const uint32_t* wp = wb + kMfWw + i16 * 4;
  const uint16_t* cp = ch.cds + 8 * kg;  // C_nd follows C_d
  const uint16_t* xp[kRt];
#pragma unroll
  for (int m = 0; m < kRt; ++m) xp[m] = xr[m] + 8 * kg;
  struct Row {
    uint2 w[kNs];
    uint4 av[kRt], cd, cn;
  };
  auto load_row = [&](int h) {
    Row r;
#pragma unroll
    for (int b = 0; b < kNs; ++b) r.w[b] = *reinterpret_cast<const uint2*>(wp + b * kStride + 2 * h);
#pragma unroll
    for (int m = 0; m < kRt; ++m) r.av[m] = *reinterpret_cast<const uint4*>(xp[m] + 32 * h);
    r.cd = *reinterpret_cast<const uint4*>(cp + 32 * h);
    r.cn = *reinterpret_cast<const uint4*>(cp + mf_chunk(kCompact) + 32 * h);
    return r;
  };
  auto row_mfma = [&](const Row& r, const uint32_t (&rs2)[kNs]) {
#pragma unroll
    for (int b = 0; b < kNs; ++b) {
      const f16x8 bv = mf_row_b(r.w[b].x, r.w[b].y, r.cd, r.cn, rs2[b], static_cast<uint32_t>(3 - kg), static_cast<uint32_t>(kg));
#pragma unroll
      for (int m = 0; m < kRt; ++m) {
        acc[b][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, r.av[m]), bv, acc[b][m], 0, 0, 0);
      }
    }
  };
  // R_d | R_nd << 16 of a K tile's group for this lane's columns
  auto load_rs = [&](uint2 go, uint32_t (&rs2)[kNs]) {
    const uint32_t off = (rs_lane & go.y) + go.x;
#pragma unroll
    for (int b = 0; b < kNs; ++b) {
      rs2[b] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const unsigned char*>(wb + b * kStride) + off);
    }
  };
  uint32_t rs2[kNs];
  load_rs(ch.goff[0], rs2);
  uint2 go = ch.goff[nt > 1 ? 1 : 0];
  Row r0 = load_row(0), r1 = load_row(1);
#pragma unroll 1
  for (int t = 0; t < nt; ++t) {
    const int step = t + 1 < nt ? 1 : 0;  // the last iteration reads its own K tile again (not used)
    wp += step * 2 * kMfWCols * 2;
    cp += step * kTileK;
#pragma unroll
    for (int m = 0; m < kRt; ++m) xp[m] += step * kTileK;
    uint32_t rn[kNs];
    load_rs(go, rn);
    go = ch.goff[t + 2 < nt ? t + 2 : nt - 1];
    row_mfma(r0, rs2);
    r0 = load_row(0);
    row_mfma(r1, rs2);
    r1 = load_row(1);
#pragma unroll
    for (int b = 0; b < kNs; ++b) rs2[b] = rn[b];
  }

  // ---- salient columns, kMfSalWin at a time: both operands in registers (mf_salient_operands).
  // The first window uses the words loaded with the tile; later windows load their own.
  const int sbase0 = cm.sbase0;
  const int num_sal = cm.num_sal;
  auto window = [&](int w0, const uint32_t (&q2w)[kNs][2]) {
    f16x8 av[kRt], bv[kNs];
    mf_salient_operands<kNs, kRt, kCompact>(ch, wb, xr, static_cast<uint32_t>(i16 * 16), rs_lane, kg, w0,
                                  ((sbase0 + w0) & 31) + 8 * kg, q2w, av, bv);
#pragma unroll
    for (int b = 0; b < kNs; ++b) {
#pragma unroll
      for (int m = 0; m < kRt; ++m) acc[b][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av[m], bv[b], acc[b][m], 0, 0, 0);
    }
  };
  if (num_sal > 0) {
    const __amdgpu_buffer_rsrc_t r_q2 = make_rsrc(q2, static_cast<uint32_t>(q2rows) * N * 4u);
    uint32_t q2w[kNs][2];
#pragma unroll
    for (int b = 0; b < kNs; ++b) {
      q2w[b][0] = q2w0[b][0];
      q2w[b][1] = q2w0[b][1];
    }
#pragma unroll 1
    for (int w0 = 0;;) {
      window(w0, q2w);
      w0 += kMfSalWin;
      if (w0 >= num_sal) break;
      const int q2b = (sbase0 + w0) >> 5;  // qweight2_sparse row of the window's first salient column
#pragma unroll
      for (int b = 0; b < kNs; ++b) {
        const uint32_t v_q2 = n[b] < N ? static_cast<uint32_t>(n[b]) * 4u : kMfOob;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const bool rv = q2b + h < q2rows;
          q2w[b][h] = bload32(r_q2, rv ? v_q2 : kMfOob, static_cast<uint32_t>(rv ? q2b + h : 0) * N * 4u);
        }
      }
    }
  }
}

// Workgroup = kUnits units of 4 wavefronts.  The grid is sized to what the GPU holds at once, and the
// workgroups share the (row tile, output tile) pairs evenly, row-tile major (a row tile is up to kRows rows of one
// segment): as long as there are enough workgroups, each row tile's output tiles are split into runs, else all pairs are,
// and a run may go on in the next row tile.
// kUnits == 1: one projection (blockIdx.z picks it when two are given, unfused).
// kUnits == 2: unit 0 computes the gate and unit 1 the up projection of the same tiles, side by side;
// the output is fp16(silu(g) * u).
// Along a run the units compute two output tiles at a time (mf_compute) while the next two tiles' weight words are
// in flight to registers.  kSingle: weight words loaded one at a time (column counts that are no multiple of 4, misaligned
// tensors).  kChunks: more than one 512-column chunk (rank > 512), staged in turn for each two tiles, with nothing in
// flight meanwhile.  Both ran one tile a pass, word by word and restaged for every tile: SwiGLU launch of 8 segments of 33
// rows, N = 8194, rank 512: 85.8 -> 49.4 us; 4 segments of 33, N = 2048, rank 576: 22.6 -> 16.4.
// Wavefronts a SIMD each instance is held to: what its LDS lets reside anyway (one unit: three workgroups a CU, with 32
// staged rows of 512 columns two).
constexpr int mf_waves(int units, int rows, bool compact) {
  return units == 2 ? 2 : (rows > kMfRows && !compact ? 2 : 3);
}

// a / b for b > 0 (wave-uniform).  Below 2^22 a reciprocal estimate corrected by one (the general 32-bit division is some
// 20 dependent instructions, and every wavefront does some of these before its first load).
__device__ __forceinline__ uint32_t mf_div(uint32_t a, uint32_t b) {
  if (a >= (1u << 22)) return a / b;  // uniform
  int q = static_cast<int>(static_cast<float>(a) * __builtin_amdgcn_rcpf(static_cast<float>(b)));
  const int r = static_cast<int>(a) - q * static_cast<int>(b);
  q += r >= static_cast<int>(b) ? 1 : 0;
  q -= r < 0 ? 1 : 0;
  return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(q));
}

template <int kUnits, int kRows, bool kCompact, bool kSingle, bool kChunks>
__global__ __launch_bounds__(kUnits * kMfThreads)
__attribute__((amdgpu_waves_per_eu(mf_waves(kUnits, kRows, kCompact), 8)))
void grouped_mfma_kernel(MfmaArgs a) {
  using WW = MfWaveWords<kCompact>;
  constexpr int kSal = mf_sal_slots(kCompact);
  constexpr int kRowTile = kRows > kMfRows ? kRows : kMfRows;  // rows of a row tile (the 4-row instances have no more)
  const int unit = kUnits == 2 ? __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kMfThreads) : 0;
  const int which = kUnits == 2 ? unit : static_cast<int>(blockIdx.z);
  const MfmaProj& pa = a.proj[which];
  const tris_compact3_payload& p = pa.p;
  // the launch's scalars and pointers, all asked for at once (left alone, the compiler loads each where it is first
  // used, and the workgroup waits for one scalar load after another before its first weight load)
  const int num_experts = p.num_experts;
  const int64_t* const row_index = pa.row_index;
  asm volatile("" ::"s"(p.outfeatures), "s"(num_experts), "s"(p.rank), "s"(p.num_groups), "s"(row_index), "s"(pa.hidden), "s"(pa.out),
               "s"(pa.decoded), "s"(p.qweight1), "s"(p.qweight2_sparse), "s"(p.qweight2_sparse_prefix), "s"(p.c_map),
               "s"(p.g_idx), "s"(p.col_pack3), "s"(p.row_pack3), "s"(pa.hidden_rows), "s"(p.qweight2_sparse_rows),
               "s"(a.segment_offsets), "s"(a.expert_ids), "s"(a.num_segments), "s"(a.batch), "s"(a.decoded_by_expert),
               "s"(a.comb_out));
  const int nob = ceil_div(p.outfeatures, kTileOut);
  // with at most 64 routed rows, every row's index in the segments' round trip (lane i: row i)
  const int lane = static_cast<int>(threadIdx.x) % kWave;
  // (without one, any readable words)
  const int64_t* const any_index = row_index != nullptr ? row_index : reinterpret_cast<const int64_t*>(p.col_pack3);
  const int64_t early = any_index[row_index != nullptr ? (lane < a.batch ? lane : a.batch - 1) : 0];
  const MfSegScan sc = mf_scan_segments(a.segment_offsets, a.expert_ids, a.num_segments, kRowTile);
  const int R = __builtin_amdgcn_readfirstlane(sc.total);
  if (R == 0) return;  // no rows
  // the one-token combine: the two units take row tiles 0 and 1 of the same output tiles, so the workgroups share
  // out output tiles only
  const bool comb = kUnits == 2 && a.comb_out != nullptr;
  const int Rm = comb ? 1 : R;
  const int W = static_cast<int>(gridDim.x);
  const int w = static_cast<int>(blockIdx.x);
  // The workgroup's (row tile, output tile) pairs [t_lo, t_hi), row-tile major.  As long as there are enough workgroups,
  // workgroup w is the (w / Rm)-th of row tile w % Rm (its activations and column data stay with few XCDs); that
  // tile's workgroups split its output tiles into runs, and those past its output tiles, the last of the grid, are idle.
  // With fewer than three workgroups a row tile the runs would differ by half or more; where they are long (8 output
  // tiles and up) all pairs are split evenly instead, and a run may go on in the next row tile, which it stages too
  // (A3B T = 1024, 257 row tiles on 768 workgroups: down 64 -> 58 us; the gate/up launch's runs of five: 39 -> 40 us).
  uint32_t t_lo, t_hi;
  const uint32_t total = static_cast<uint32_t>(Rm) * nob;
  if (Rm * 3 <= W || (Rm <= W && total < 8u * W)) {
    const uint32_t per = mf_div(W, Rm);
    const uint32_t sub = mf_div(w, Rm);
    const uint32_t rt = w - sub * Rm;
    uint32_t cnt = per + (rt < W - per * Rm ? 1u : 0u);
    cnt = cnt < static_cast<uint32_t>(nob) ? cnt : nob;
    if (sub >= cnt) return;
    const uint32_t run = mf_div(nob, cnt), more = nob - run * cnt;  // the first `more` runs have one output tile more
    t_lo = rt * nob + sub * run + (sub < more ? sub : more);
    t_hi = t_lo + run + (sub < more ? 1u : 0u);
  } else {
    const uint32_t run = mf_div(total, W), more = total - run * W;
    t_lo = w * run + (static_cast<uint32_t>(w) < more ? w : more);
    t_hi = t_lo + run + (static_cast<uint32_t>(w) < more ? 1u : 0u);
    if (t_hi <= t_lo) return;
  }
  // the combine's weights by row (w_row[inverse_perm[s]] = w[s]); a route that is not one token on two experts,
  // one row each, gets zero outputs (before any barrier, the same in both units)
  uint16_t wr0 = 0, wr1 = 0;
  if (comb) {
    const int inv0 = a.comb_inv[0], inv1 = a.comb_inv[1];
    bool ok = R == 2 && ((inv0 == 0 && inv1 == 1) || (inv0 == 1 && inv1 == 0));
    for (int t = 0; t < 2 && ok; ++t) {
      int cs = 0, cr0 = 0, crc = 0, ce = -1;
      mf_map_scanned(sc, a.segment_offsets, a.expert_ids, a.num_segments, t, kRowTile, &cs, &cr0, &crc, &ce);
      ce = __builtin_amdgcn_readfirstlane(ce);
      ok = __builtin_amdgcn_readfirstlane(crc) == 1 && ce >= 0 && ce < num_experts;
    }
    if (!ok) {
      if (unit == 0) {
        const int t0 = static_cast<int>(threadIdx.x) % kMfThreads;
        for (int n = t_lo * kTileOut + t0; n < static_cast<int>(t_hi) * kTileOut && n < p.outfeatures; n += kMfThreads) a.comb_out[n] = 0;
      }
      return;
    }
    wr0 = a.comb_w[inv0 == 0 ? 0 : 1];
    wr1 = a.comb_w[inv0 == 0 ? 1 : 0];
  }
  uint16_t* out = kUnits == 2 ? a.proj[0].out : pa.out;
  __shared__ __attribute__((aligned(16))) uint16_t mf_xs[kUnits][kRows * mf_xstride(kCompact)];
  __shared__ __attribute__((aligned(16))) uint16_t mf_cds[kUnits][2 * mf_chunk(kCompact)];  // C_d, then C_nd
  __shared__ __attribute__((aligned(16))) uint2 mf_goff[kUnits][mf_chunk(kCompact) / kTileK];
  __shared__ __attribute__((aligned(16))) uint32_t mf_salw[kUnits][kSal + 4];  // (one spare slot)
  __shared__ __attribute__((aligned(16))) uint16_t mf_salxo[kUnits][kSal + 8];
  __shared__ __attribute__((aligned(16))) uint32_t mf_salcp[kUnits][kSal + 4];
  __shared__ __attribute__((aligned(16))) float mf_exch[kUnits == 2 ? kMfThreads * 4 * 2 * (kRowTile / kMfRows) : 4];
  MfChunk ch;
  ch.xs = &mf_xs[unit][0];
  ch.cds = &mf_cds[unit][0];
  ch.cns = &mf_cds[unit][mf_chunk(kCompact)];
  ch.goff = &mf_goff[unit][0];
  ch.col_sal = nullptr;
  ch.sal_col = nullptr;
  ch.sal_xi = nullptr;
  ch.sal_w = &mf_salw[unit][0];
  ch.sal_xo = &mf_salxo[unit][0];
  ch.sal_cp = &mf_salcp[unit][0];
  ch.meta = nullptr;
  // each wavefront's words of the two tiles it computes together
  __shared__ __attribute__((aligned(16))) uint32_t mf_wb[kUnits * kMfWaves][2][WW::kAlloc];
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) % kMfThreads / kWave);
  uint32_t* const wb = &mf_wb[unit * kMfWaves + wave][0][0];
  if (lane < 2) wb[lane * WW::kAlloc] = 0u;  // the zero words (the first row tile's barrier orders these writes)
  float* exch = mf_exch;

  for (uint32_t t = t_lo; t < t_hi;) {
  const int rt_i = static_cast<int>(mf_div(t, nob));
  // the lane index and sizes of this row tile: opaque, so that the many addresses and conditions made of them are not
  // computed ahead of the loop and held across it (most launches run it once, and the held registers spill)
  int ln = lane, N = p.outfeatures, rank = p.rank, G = p.num_groups, nseg = a.num_segments;
  int ob_begin = static_cast<int>(t - static_cast<uint32_t>(rt_i) * nob), ob_end = ob_begin + static_cast<int>(t_hi - t);
  ob_end = ob_end < nob ? ob_end : nob;
  const bool first = t == t_lo;
  t += ob_end - ob_begin;
  asm volatile("" : "+v"(ln), "+s"(N), "+s"(rank), "+s"(G), "+s"(nseg), "+s"(ob_begin), "+s"(ob_end));
  const int utid = wave * kWave + ln;
  const int i16 = ln % 16;
  const int kg = ln / 16;
  const int rt = comb ? unit : rt_i;  // the combine's units: row tiles 0 and 1
  int s = 0, row0 = 0, rc = 0, e = -1;
  mf_map_scanned(sc, a.segment_offsets, a.expert_ids, nseg, rt, kRowTile, &s, &row0, &rc, &e);
  s = __builtin_amdgcn_readfirstlane(s);  // the mapping is the same in every lane
  row0 = __builtin_amdgcn_readfirstlane(row0);
  rc = __builtin_amdgcn_readfirstlane(rc);
  e = __builtin_amdgcn_readfirstlane(e);
  const int ds = a.decoded_by_expert ? e : s;  // the decoded bitmaps' slot
  // activations from partial sums: only the 4-row instances carry that staging (the host sends at most 4 rows),
  // so the others keep no register for it across their tile loop
  const bool part = kRows == 4 && !kChunks && pa.partials != nullptr;
  if (e < 0 || e >= num_experts) {  // rows routed to no expert: zero output
    if (unit == 0) {
      const int span = (ob_end - ob_begin) * kTileOut;
      for (int idx = utid; idx < rc * span; idx += kMfThreads) {
        const int n = ob_begin * kTileOut + idx % span;
        if (n < N) out[static_cast<int64_t>(row0 + idx / span) * N + n] = 0;
      }
    }
    continue;
  }
  if (!first) __syncthreads();  // the previous row tile's LDS readers are done
  const MfWaveSrc src = mf_wave_src<kCompact>(pa, ds, e, 0, wave, ln);
  const uint32_t* q2 = reinterpret_cast<const uint32_t*>(p.qweight2_sparse) +
                       static_cast<int64_t>(e) * p.qweight2_sparse_rows * N;
  const int q2rows = p.qweight2_sparse_rows;
  MfWaveRegs<kCompact> wr[2];  // the next two tiles' words in flight
  int64_t entry = early;
  int tok0 = row0;
  if (row_index == nullptr) {
    entry = ln;
    tok0 = 0;
  } else if (a.batch > kWave) {  // more rows than lanes: this row tile's own
    entry = row_index[row0 + (ln < rc ? ln : rc - 1)];
    tok0 = 0;
  }
  const int hidden_rows = row_index != nullptr ? pa.hidden_rows : rc;
  const uint32_t roff = entry >= 0 && entry < hidden_rows && static_cast<uint32_t>(ln - tok0) < static_cast<uint32_t>(rc)
                            ? static_cast<uint32_t>(entry) * static_cast<uint32_t>(rank) * 2u : kMfOob;
  const __amdgpu_buffer_rsrc_t r_hid =
      make_rsrc(pa.hidden + (row_index != nullptr ? 0 : static_cast<int64_t>(row0) * rank),
                part ? 0u : static_cast<uint32_t>(hidden_rows) * rank * 2u);
  MfChunkMeta cm;
  {  // chunk 0 and the first tiles' weights
    MfColRegs cols;
    MfRowRegs<kRows, kCompact> rows;
    mf_cols_issue<kCompact>(pa, e, 0, utid, cols);
    mf_rows_issue<kRows, kCompact>(r_hid, rank, 0, wave, ln, roff, tok0, rows);
    mf_wave_tile_issue<kCompact, kSingle>(src, G, ob_begin, ln, wr[0]);
    const bool two = !(kSingle || kChunks) || ob_begin + 1 < ob_end;  // uniform
    if (two) mf_wave_tile_issue<kCompact, kSingle>(src, G, ob_begin + 1, ln, wr[1], ob_begin + 1 < ob_end);
    mf_cols_write<kCompact>(pa, rc, 0, utid, ch, cols, kSal);
    if (!part) mf_rows_write<kRows, kCompact>(rows, rc, wave, ln, ch.xs);
    if (part) mf_partials_stage<kCompact>(pa, row0, rc, utid, ch);  // one chunk (host-checked)
    cm = mf_chunk_meta(cols, kSal);
    mf_wave_tile_write<kCompact>(wr[0], ln, wb);
    if (two) mf_wave_tile_write<kCompact>(wr[1], ln, wb + WW::kAlloc);
    __syncthreads();
  }
  // The outputs of rows 16 m .. of tile ob, from their accumulators.  Stores go through a buffer resource over the
  // tile's rows from its first column: rows past rc have an offset past it and are dropped, so every lane issues all
  // four; only the expert's last tile can have columns past N.
  uint16_t* const out0 = out + static_cast<int64_t>(row0) * N;
  auto store = [&](int ob, int m, const f32x4& acc, const float* ex) {
    const int n = ob * kTileOut + 16 * wave + i16;
    if (kUnits == 2 && comb) {
      // row 0 of each unit's tile (one row a tile): the combine of the token's two rows at column n, the products
      // rounded to fp16 (the asm keeps them from being fused into the sum) and added in fp32 (two terms: the
      // pick order does not matter), rounded once to the output dtype
      if (kg == 0 && n < N) {
        const float up0 = ex[utid * 4];
        uint16_t p0 = hmul_bits(f2h_bits(acc[0]), wr0);
        uint16_t p1 = hmul_bits(f2h_bits(up0), wr1);
        asm volatile("" : "+v"(p0), "+v"(p1));
        const float y = h2f(p0) + h2f(p1);
        a.comb_out[n] = a.comb_bf16 ? f32_to_bf16_rne(y) : f2h_bits(y);
      }
      return;
    }
    f32x4 up = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (kUnits == 2) up = *reinterpret_cast<const f32x4*>(&ex[utid * 4]);
    const uint32_t bytes = (static_cast<uint32_t>(rc) * N - ob * kTileOut) * 2u;
    const __amdgpu_buffer_rsrc_t r_out = make_rsrc(out0 + ob * kTileOut, bytes);
    const int r0 = 16 * m + 4 * kg;  // the lane's rows r0 .. r0 + 3
    // Where a lane without an output stores: past the buffer.  The launcher keeps the 32- and 64-row tiles' outputs below
    // 2 GiB; a 16-row tile's can be larger, and kMfOob inside them.  (The size in a register made the 64-row instance spill.)
    const uint32_t drop = kRows > kMfRows ? kMfOob : bytes;
    const uint32_t vo = n < N ? static_cast<uint32_t>(r0 * N + 16 * wave + i16) * 2u : drop;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      // two units: g and u rounded to fp16 as the two outputs would be.  One unit: no output scale or bias here, the
      // host sends none (launch_grouped_mfma rejects payloads with them)
      const uint16_t y = kUnits == 2 ? swiglu_bits(f2h_bits(acc[v]), f2h_bits(up[v])) : f2h_bits(acc[v]);
      __builtin_amdgcn_raw_buffer_store_b16(y, r_out, r0 + v < rc && (kRows > kMfRows || n < N) ? vo + static_cast<uint32_t>(v * N) * 2u : drop,
                                            0u, 0);
    }
  };
  // kNs output tiles from `ob`, whose words are in wb, kRt 16-row sub-tiles; with one chunk the next tiles' words are
  // loaded to registers meanwhile and written to wb after the last read of this pass (one wavefront's LDS operations
  // stay in order).
  auto tiles = [&](auto ns, auto nrt, int ob) {
    constexpr int kNs = decltype(ns)::value;
    constexpr int kRt = decltype(nrt)::value;
    f32x4 acc[kNs][kRt];
    int n[kNs];
    uint32_t q2w[kNs][2];
    // A operand rows of this lane: rows past rc feed output rows that are not stored, so they read row 0 (the same
    // LDS words as lane 0's rows: broadcast reads instead of bank conflicts; T = 16 gate/up launch 33.2 -> 32.5 us)
    const uint16_t* xr[kRt];
#pragma unroll
    for (int m = 0; m < kRt; ++m) xr[m] = ch.xs + (16 * m + i16 < rc ? 16 * m + i16 : 0) * mf_xstride(kCompact);
#pragma unroll
    for (int b = 0; b < kNs; ++b) {
#pragma unroll
      for (int m = 0; m < kRt; ++m) acc[b][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      n[b] = (ob + b) * kTileOut + 16 * wave + i16;
    }
    if constexpr (!kChunks) {
#pragma unroll
      for (int b = 0; b < kNs; ++b) mf_q2_issue(q2, q2rows, N, n[b], cm, q2w[b]);
      // the next tiles' words, if any (uniform; the one-unit 64-row instance always loads and writes two tiles, of zeros
      // at the end: at its register limit the branch spills, and A3B's 64-row segments took 10 to 25% longer)
      const bool more = (kUnits == 1 && kRows == 64) || ob + kNs < ob_end;
      if (more) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          mf_wave_tile_issue<kCompact, kSingle>(src, G, ob + kNs + b, ln, wr[b], ob + kNs + b < ob_end);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the pass they overlap
      mf_compute<kNs, kRt, kCompact>(q2, q2rows, N, rank, G, 0, n, xr, ln, ch, cm, wb, q2w, acc);
      __builtin_amdgcn_sched_barrier(0);
      if (more) {
        // the words pass between lanes: the last pass's reads come before these writes, and the next pass's after
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int b = 0; b < 2; ++b) mf_wave_tile_write<kCompact>(wr[b], ln, wb + b * WW::kAlloc);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    } else {
      // (the next chunk's loads in flight during this one's pass made every launch 2 to 10% longer: spilled registers and
      // more instructions to fetch)
      for (int kc = 0; kc < rank; kc += kMfChunk) {
        if (ob > ob_begin || kc > 0) {
          __syncthreads();  // the previous chunk's readers are done
          MfColRegs cols;
          MfRowRegs<kRows, kCompact> rows;
          mf_cols_issue<kCompact>(pa, e, kc, utid, cols);
          mf_rows_issue<kRows, kCompact>(r_hid, rank, kc, wave, ln, roff, tok0, rows);
          const MfWaveSrc at = mf_wave_src<kCompact>(pa, ds, e, kc, wave, ln);
#pragma unroll
          for (int b = 0; b < kNs; ++b) mf_wave_tile_issue<kCompact, kSingle>(at, G, ob + b, ln, wr[b]);
          mf_cols_write<kCompact>(pa, rc, kc, utid, ch, cols, kSal);
          mf_rows_write<kRows, kCompact>(rows, rc, wave, ln, ch.xs);
          cm = mf_chunk_meta(cols, kSal);
#pragma unroll
          for (int b = 0; b < kNs; ++b) mf_wave_tile_write<kCompact>(wr[b], ln, wb + b * WW::kAlloc);
          __syncthreads();
        }
#pragma unroll
        for (int b = 0; b < kNs; ++b) mf_q2_issue(q2, q2rows, N, n[b], cm, q2w[b]);
        mf_compute<kNs, kRt, kCompact>(q2, q2rows, N, rank, G, kc, n, xr, ln, ch, cm, wb, q2w, acc);
      }
    }
    if (kUnits == 2) {
      if (unit == 1) {
#pragma unroll
        for (int b = 0; b < kNs; ++b) {
#pragma unroll
          for (int m = 0; m < kRt; ++m) *reinterpret_cast<f32x4*>(&exch[((b * kRt + m) * kMfThreads + utid) * 4]) = acc[b][m];
        }
      }
      __syncthreads();
      if (unit == 0) {
#pragma unroll
        for (int b = 0; b < kNs; ++b) {
#pragma unroll
          for (int m = 0; m < kRt; ++m) store(ob + b, m, acc[b][m], exch + (b * kRt + m) * kMfThreads * 4);
        }
      }
      __syncthreads();  // exch is rewritten by the next tiles
    } else {
#pragma unroll
      for (int b = 0; b < kNs; ++b) {
#pragma unroll
        for (int m = 0; m < kRt; ++m) store(ob + b, m, acc[b][m], exch);
      }
    }
  };
  // the run's output tiles, two at a time, with as many row sub-tiles as the row tile's rows need
  auto run = [&](auto nrt) {
    for (int ob = ob_begin; ob < ob_end;) {
      if (ob + 1 < ob_end) {
        tiles(std::integral_constant<int, 2>{}, nrt, ob);
        ob += 2;
      } else {
        tiles(std::integral_constant<int, 1>{}, nrt, ob);
        ob += 1;
      }
    }
  };
  if (kRows <= 16 || rc <= 16) {  // uniform
    run(std::integral_constant<int, 1>{});
  } else if constexpr (kRows > 16) {
    if (kRows <= 32 || rc <= 32) {
      run(std::integral_constant<int, 2>{});
    } else if constexpr (kRows > 32) {
      run(std::integral_constant<int, 4>{});
    }
  }
  }  // row tiles
}

// ----------------------------------------------------------------------------------------------------
// Non-expert linears: one matrix over the full input width (thousands of columns, a row-scale group each 128), any
// batch, up to three of them on one input.  A workgroup takes one 64-output tile, kRows rows and a run of 512-column
// chunks (blockIdx.y = row tile x slice), stages each chunk as the decode kernel does, and leaves fp32 partial sums
// [slice][batch][N]; linear_finish_kernel adds the slices in order, then the addend, scale and bias.  Slices are taken
// until the launch fills the GPU; where the tiles alone do, there is one, and the workgroup writes the outputs itself.  The row scales are staged per K tile (the decode kernel's per group would not fit), and
// whether every K tile of a chunk lies in one group is found on the way: a chunk where one does not (or with an
// infinite activation, or a row scale that is not finite) builds its operands column by column from memory instead
// (lin_exact_row), so no launch waits for the host to look at g_idx.  Bound by the loads of each column's scales: a
// matrix of 4096 x 4096 with a shuffled g_idx takes 65 us at 16 rows and 406 at 256 (the exact kernel 697 and 873, one
// output column's weights at a time in every wavefront 340 and 3003; with a uniform g_idx 45 and 87).
// Q, K and V of 2048 x 2048 at 16 rows: 10.0 us, the finish 3.4 and the bitmaps 9.5, against 504 us of the exact VALU
// kernel (two launches) and seven host round trips to read g_idx.
struct LinProj {
  tris_compact3_payload p;
  const int32_t* decoded;  // [packed rows / 2][tiles][128]
  float* part;             // [slices][batch][N] (null with one slice)
  const float* addend;     // [batch][N] or null
  uint16_t* out;           // [batch][N]
};
struct LinArgs {
  LinProj proj[TRIS_MAX_LINEARS];
  const uint16_t* x;         // [batch][rank]
  const uint16_t* in_scale;  // [rank] or null
  int batch, slices, chunks;
};

// A sum's output, as the exact kernel ends: fp16((v + addend) * scale + bias).
__device__ __forceinline__ void lin_store(const LinProj& lp, int64_t at, float v, float scale, float bias) {
  if (lp.addend != nullptr) v += lp.addend[at];
  if (lp.p.has_output_scale) v = v * scale;
  if (lp.p.has_bias) v = v + bias;
  lp.out[at] = f2h_bits(v);
}

// B operand of packed row pr, column n, straight from memory: the lane's 8 weights in mf_row_b's order, each with its own
// column's group and salient columns in place (chunks with split K tiles, infinities or scales that are not finite).
// q1, gw: the column's qweight1 and split words of the row.
__device__ __forceinline__ f16x8 lin_exact_row(const tris_compact3_payload& p, int pr, int n, int kg, uint32_t q1,
                                               uint32_t gw) {
  const int N = p.outfeatures, G = p.num_groups;
  const uint32_t cm = static_cast<uint32_t>(p.c_map[pr]);
  const int64_t* const row = p.row_pack3 + static_cast<int64_t>(n) * G;
  int g[8];
  uint64_t cp[8], rp[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {  // element i: column kg + 4 (i / 2) + 16 (i % 2) of the packed row
    const int k = 32 * pr + kg + 4 * (i >> 1) + 16 * (i & 1);
    g[i] = p.g_idx[k];
    cp[i] = static_cast<uint64_t>(p.col_pack3[k]);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const bool gv = g[i] >= 0 && g[i] < G;
    const uint64_t v = static_cast<uint64_t>(row[gv ? g[i] : 0]);
    rp[i] = gv ? v : 0ull;
  }
  uint32_t w[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int bit = kg + 4 * (i >> 1) + 16 * (i & 1);
    const auto prod = [&](int h) {
      return hmul_bits(static_cast<uint16_t>(cp[i] >> (16 * h)), static_cast<uint16_t>(rp[i] >> (16 * h)));
    };
    const uint16_t neg1 = (q1 >> bit) & 1u ? 0u : 0x8000u;
    uint16_t v = ((gw >> bit) & 1u ? prod(2) : prod(3)) ^ neg1;
    if ((cm >> bit) & 1u) {
      const int idx = p.qweight2_sparse_prefix[pr] + __popc(cm & ((1u << bit) - 1u));
      const int r2 = idx >> 5;
      const uint32_t q2 = r2 >= 0 && r2 < p.qweight2_sparse_rows
                              ? static_cast<uint32_t>(p.qweight2_sparse[static_cast<int64_t>(r2) * N + n]) : 0u;
      const uint16_t neg2 = (q2 >> (idx & 31)) & 1u ? 0u : 0x8000u;
      v = hadd_bits(prod(0) ^ neg1, prod(1) ^ neg2);
    }
    w[i] = v;
  }
  return __builtin_bit_cast(f16x8, make_uint4(w[0] | (w[1] << 16), w[2] | (w[3] << 16), w[4] | (w[5] << 16),
                                              w[6] | (w[7] << 16)));
}

template <int kRows, bool kSingle>
__global__ __launch_bounds__(kMfThreads) __attribute__((amdgpu_waves_per_eu(3, 8))) void linear_mfma_kernel(LinArgs a) {
  constexpr int kRt = kRows / kMfRows;
  const LinProj& lp = a.proj[blockIdx.z];
  const tris_compact3_payload& p = lp.p;
  const int N = p.outfeatures, rank = p.rank, G = p.num_groups;
  const int ob = static_cast<int>(blockIdx.x);
  if (ob * kTileOut >= N) return;  // uniform, before any barrier
  const int sl = static_cast<int>(blockIdx.y) % a.slices;
  const int row0 = static_cast<int>(blockIdx.y) / a.slices * kRows;
  const int rc = a.batch - row0 < kRows ? a.batch - row0 : kRows;
  const int c_lo = static_cast<int>(static_cast<int64_t>(sl) * a.chunks / a.slices);
  const int c_hi = static_cast<int>(static_cast<int64_t>(sl + 1) * a.chunks / a.slices);
  __shared__ __attribute__((aligned(16))) uint16_t xs[kRows * mf_xstride(false)];
  __shared__ __attribute__((aligned(16))) uint16_t cds[2 * kMfChunk];
  __shared__ __attribute__((aligned(16))) uint2 goff[kMfTiles];
  __shared__ __attribute__((aligned(16))) uint32_t salw[kMfChunk + 4];
  __shared__ __attribute__((aligned(16))) uint16_t salxo[kMfChunk + 8];
  __shared__ __attribute__((aligned(16))) uint32_t salcp[kMfChunk + 4];
  __shared__ __attribute__((aligned(16))) uint32_t wbuf[kMfWaves][MfWaveWords<false>::kAlloc];
  MfChunk ch{};
  ch.xs = xs;
  ch.cds = cds;
  ch.goff = goff;
  ch.sal_w = salw;
  ch.sal_xo = salxo;
  ch.sal_cp = salcp;
  const int utid = static_cast<int>(threadIdx.x);
  const int wave = __builtin_amdgcn_readfirstlane(utid / kWave);
  const int lane = utid % kWave;
  const int i16 = lane % 16, kg = lane / 16;
  uint32_t* const wb = wbuf[wave];
  MfmaProj pa{};
  pa.decoded = lp.decoded;
  pa.p = p;
  const uint32_t roff = lane < rc ? static_cast<uint32_t>(lane) * static_cast<uint32_t>(rank) * 2u : kMfOob;
  const __amdgpu_buffer_rsrc_t r_x =
      make_rsrc(a.x + static_cast<int64_t>(row0) * rank, static_cast<uint32_t>(rc) * rank * 2u);
  const __amdgpu_buffer_rsrc_t r_sc = make_rsrc(a.in_scale, a.in_scale != nullptr ? static_cast<uint32_t>(rank) * 2u : 0u);
  const __amdgpu_buffer_rsrc_t r_g = make_rsrc(p.g_idx, static_cast<uint32_t>(rank) * 4u);
  const int n0w = ob * kTileOut + kMfWCols * wave;  // the wavefront's first column
  const __amdgpu_buffer_rsrc_t r_rs = make_rsrc(p.row_pack3 + (n0w < N ? static_cast<int64_t>(n0w) * G : 0),
                                                n0w < N ? static_cast<uint32_t>(N - n0w) * G * 8u : 0u);
  const uint32_t* q2 = reinterpret_cast<const uint32_t*>(p.qweight2_sparse);
  const uint16_t* xr[kRt];
#pragma unroll
  for (int m = 0; m < kRt; ++m) xr[m] = xs + (16 * m + i16 < rc ? 16 * m + i16 : 0) * mf_xstride(false);
  const int n[1] = {n0w + i16};
  f32x4 acc[1][kRt];
#pragma unroll
  for (int m = 0; m < kRt; ++m) acc[0][m] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  for (int c = c_lo; c < c_hi; ++c) {
    const int kc = c * kMfChunk;
    if (c > c_lo) __syncthreads();  // the previous chunk's readers are done
    MfColRegs cols;
    MfRowRegs<kRows, false> rows;
    MfWaveRegs<false> wr;
    int gt[2];  // the groups of K tiles lane / 16 and lane / 16 + 4
#pragma unroll
    for (int h = 0; h < 2; ++h) gt[h] = static_cast<int>(bload32(r_g, static_cast<uint32_t>(kc + (kg + 4 * h) * kTileK) * 4u, 0u));
    const uint64_t gp = bload64(r_g, static_cast<uint32_t>(kc + 2 * utid) * 4u, 0u);  // of the thread's two columns
    mf_cols_issue<false>(pa, 0, kc, utid, cols);
    mf_rows_issue<kRows, false>(r_x, rank, kc, wave, lane, roff, 0, rows);
    mf_wave_words_issue<false, kSingle>(mf_wave_src<false>(pa, 0, 0, kc, wave, lane), ob, wr, true);
    uint64_t rp[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      rp[h] = bload64(r_rs, gt[h] >= 0 && gt[h] < G ? static_cast<uint32_t>(i16 * G + gt[h]) * 8u : kMfOob, 0u);
    }
    const int first = __shfl(static_cast<int>(gp), lane & 32);  // the group of the K tile's first column
    const bool split = kc + 2 * utid < rank && (static_cast<int>(gp) != first || static_cast<int>(gp >> 32) != first);
    if (a.in_scale != nullptr) {
      const uint4 sc = bload128(r_sc, static_cast<uint32_t>(kc + lane * 8) * 2u, 0u);
      const uint32_t sv[4] = {sc.x, sc.y, sc.z, sc.w};
#pragma unroll
      for (int h = 0; h < MfRowRegs<kRows, false>::kRuns; ++h) {
        uint32_t v[4] = {rows.xv[h].x, rows.xv[h].y, rows.xv[h].z, rows.xv[h].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = f16x2_as_u32(u32_as_f16x2(v[i]) * u32_as_f16x2(sv[i]));
        rows.xv[h] = make_uint4(v[0], v[1], v[2], v[3]);
      }
    }
    mf_cols_write<false, true>(pa, rc, kc, utid, ch, cols, kMfChunk);
    mf_rows_write<kRows, false>(rows, rc, wave, lane, xs);
    // an infinite activation: the GEMM multiplies a salient column by its zero factors first (inf * 0), so the chunk walks
    // its columns.  |v| + 0x83FF (modulo 2^16) is 0xFFFF for an infinity alone; a NaN gives NaN either way.
    u16x2 top = {0, 0};
#pragma unroll
    for (int h = 0; h < MfRowRegs<kRows, false>::kRuns; ++h) {
      const uint32_t v[4] = {rows.xv[h].x, rows.xv[h].y, rows.xv[h].z, rows.xv[h].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const u16x2 m = __builtin_bit_cast(u16x2, v[i] & 0x7FFF7FFFu) + u16x2{0x83FF, 0x83FF};
        top = __builtin_elementwise_max(top, m);
      }
    }
    const bool infinite = top[0] == 0xFFFF || top[1] == 0xFFFF;
    // a row scale that is not finite: where no column picks it (R_d without a split column, R0 and R1 without a salient
    // one) it must not count, but the GEMM multiplies it by the zero factors of salient columns and padding slots
    u16x2 expo = {0, 0};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      expo = __builtin_elementwise_max(expo, __builtin_bit_cast(u16x2, static_cast<uint32_t>(rp[h]) & 0x7C007C00u));
      expo = __builtin_elementwise_max(expo, __builtin_bit_cast(u16x2, static_cast<uint32_t>(rp[h] >> 32) & 0x7C007C00u));
    }
    const bool unbounded = expo[0] == 0x7C00 || expo[1] == 0x7C00;
    const MfChunkMeta cm = mf_chunk_meta(cols, kMfChunk);
    {
      const int row = lane / 4;
      uint32_t* dst = wb + kMfWw + ((row >> 1) * kMfWCols + 4 * (lane % 4)) * 4 + (row & 1) * 2;
#pragma unroll
      for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2*>(dst + 4 * i) = make_uint2(wr.q[i], wr.g[i]);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        *reinterpret_cast<uint2*>(wb + MfWaveWords<false>::kRs + (i16 * kMfMaxGroups + kg + 4 * h) * 2) =
            make_uint2(static_cast<uint32_t>(rp[h]), static_cast<uint32_t>(rp[h] >> 32));
      }
    }
    if (!__syncthreads_or(split || infinite || unbounded ? 1 : 0)) {
      uint32_t q2w[1][2];
      mf_q2_issue(q2, p.qweight2_sparse_rows, N, n[0], cm, q2w[0]);
      mf_compute<1, kRt, false>(q2, p.qweight2_sparse_rows, N, rank, kMfMaxGroups, kc, n, xr, lane, ch, cm, wb, q2w, acc);
    } else {  // uniform over the workgroup
      const int npr = (rank - kc < kMfChunk ? rank - kc : kMfChunk) / 32;
      const int nc = n[0] < N ? n[0] : N - 1;  // (columns past N are not stored)
#pragma unroll 1
      for (int j = 0; j < npr; ++j) {
        const uint2 w = *reinterpret_cast<const uint2*>(wb + kMfWw + ((j >> 1) * kMfWCols + i16) * 4 + 2 * (j & 1));
        const f16x8 bv = lin_exact_row(p, kc / 32 + j, nc, kg, w.x, w.y);
#pragma unroll
        for (int m = 0; m < kRt; ++m) {
          const f16x8 av = __builtin_bit_cast(f16x8, *reinterpret_cast<const uint4*>(xr[m] + 32 * j + 8 * kg));
          acc[0][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bv, acc[0][m], 0, 0, 0);
        }
      }
    }
  }
  const bool whole = a.slices == 1;  // the workgroup has the whole sums: no partial sums, no finishing launch
  float* const part = whole ? nullptr : lp.part + (static_cast<int64_t>(sl) * a.batch + row0) * N;
  const float scale = whole && p.has_output_scale && n[0] < N ? h2f(p.output_scale[n[0]]) : 1.0f;
  const float bias = whole && p.has_bias && n[0] < N ? h2f(p.bias[n[0]]) : 0.0f;
#pragma unroll
  for (int m = 0; m < kRt; ++m) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = 16 * m + 4 * kg + v;
      if (r >= rc || n[0] >= N) continue;
      if (whole) {
        lin_store(lp, static_cast<int64_t>(row0 + r) * N + n[0], acc[0][m][v], scale, bias);
      } else {
        part[static_cast<int64_t>(r) * N + n[0]] = acc[0][m][v];
      }
    }
  }
}

// The outputs from the slices' sums, added in order (more than one slice).
__global__ __launch_bounds__(256) void linear_finish_kernel(LinArgs a) {
  const LinProj& lp = a.proj[blockIdx.z];
  const tris_compact3_payload& p = lp.p;
  const int N = p.outfeatures;
  const int n = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  if (n >= N) return;
  const float scale = p.has_output_scale ? h2f(p.output_scale[n]) : 1.0f;
  const float bias = p.has_bias ? h2f(p.bias[n]) : 0.0f;
  for (int b = static_cast<int>(blockIdx.y); b < a.batch; b += static_cast<int>(gridDim.y)) {
    const int64_t at = static_cast<int64_t>(b) * N + n;
    const int64_t step = static_cast<int64_t>(a.batch) * N;
    float v = 0.0f;
#pragma unroll 4
    for (int s = 0; s < a.slices; ++s) v += lp.part[s * step + at];
    lin_store(lp, at, v, scale, bias);
  }
}

// ----------------------------------------------------------------------------------------------------
// Weight-stationary variant for long segments (prefill).  A work item is (active segment, kSub 64-column
// output tiles): the unit copies the tiles' weight words, builds the exact B operands of its columns over the
// whole K (rank <= 512: 16 packed rows, 4 registers each per tile, plus at most two 32-column salient windows)
// once, and streams the segment's 16-row activation tiles through them: per row tile and output tile 16 + 1
// or 2 MFMAs per wavefront, with the next row tile's loads in flight meanwhile (two activation buffers).
// Each A-operand read from LDS feeds kSub MFMAs: one 16 x 16 x 32 MFMA per kilobyte read would need 256 B
// of LDS reads per clock on a CU (4 SIMDs), twice what the LDS delivers.  kUnits == 2 runs the gate and up
// projections of the same item side by side and writes fp16(silu(g) * u).
constexpr int kWsSalWindows = 2;  // salient columns per item <= 64
#ifndef TRIS_WS_SUB
#define TRIS_WS_SUB 2
#endif
constexpr int kWsSub = TRIS_WS_SUB;  // output tiles per item (2: one activation read feeds two MFMAs)
#ifndef TRIS_WS_XSTRIDE
#define TRIS_WS_XSTRIDE 528
#endif
constexpr int kWsXStride = TRIS_WS_XSTRIDE;  // fp16 elements per staged activation row (kMfChunk + zero column + pad)
static_assert(kWsXStride > kMfChunk && kWsXStride % 8 == 0, "staged rows need the zero column and 16-byte runs");
#ifndef TRIS_WS_READ_AHEAD
#define TRIS_WS_READ_AHEAD 4
#endif
constexpr int kWsReadAhead = TRIS_WS_READ_AHEAD;  // A-operand LDS reads in flight ahead of the MFMAs
#ifndef TRIS_WS_XDEPTH
#define TRIS_WS_XDEPTH 1
#endif
constexpr int kWsXDepth = TRIS_WS_XDEPTH;  // row tiles of activations in flight in registers (1 or 2)
static_assert(kWsXDepth == 1 || kWsXDepth == 2, "activation prefetch depth is 1 or 2");

struct MfWsLayout {  // per unit, byte offsets into dynamic LDS
  int xs[2], cds, cns, col_sal, sal_col, sal_xi, sal_cp, meta, r01t, ws, bytes;
};

__host__ __device__ inline MfWsLayout mf_ws_layout() {
  MfWsLayout L;
  int o = 0;
  L.xs[0] = mf_take(&o, kMfRows * kWsXStride * 2);
  L.xs[1] = mf_take(&o, kMfRows * kWsXStride * 2);
  L.cds = mf_take(&o, kMfChunk * 2);
  L.cns = mf_take(&o, kMfChunk * 2);
  L.col_sal = mf_take(&o, kMfChunk * 4);
  L.sal_col = mf_take(&o, kMfChunk * 2);
  L.sal_xi = mf_take(&o, kMfChunk * 2);
  L.sal_cp = mf_take(&o, kMfChunk * 4);
  L.meta = mf_take(&o, 16 * 4);
  L.r01t = mf_take(&o, kMfTiles * kTileOut * 4);
  L.ws = mf_take(&o, kMfWaves * 16 * kMfSalStride * 2);
  L.bytes = o;
  return L;
}

__host__ __device__ inline int mf_ws_lds_bytes(int units, int sub) {
  return units * mf_ws_layout().bytes + (units == 2 ? sub * kMfExchBytes : 0);
}

// Activation rows [row0, row0 + rc) of the chunk: register loads (issued early) and the permuted LDS write.
struct WsX {
  uint4 xv[kMfRuns];
};

__device__ __forceinline__ void ws_x_issue(const MfmaProj& pa, int row0, int rc, int utid, WsX& X) {
  const int rank = pa.p.rank;
  const int wave = utid / kWave;
  const int lane = utid % kWave;
  uint32_t hid_bytes;
  const __amdgpu_buffer_rsrc_t r_hid = mf_hidden_rsrc(pa, row0, rc, rank, &hid_bytes);
#pragma unroll
  for (int h = 0; h < kMfRuns; ++h) {
    const int r = 4 * h + wave;
    X.xv[h] = bload128(r_hid, mf_hidden_voff(pa, row0, r, rc, lane * 8, rank, hid_bytes), 0u);
  }
}

// The same for materialised rows (no row_index): r_seg covers the segment's rows, rel0 is row0's row within
// it; rows past the segment read zeros through the resource's size, so no per-row test is needed.
__device__ __forceinline__ void ws_x_issue_seg(__amdgpu_buffer_rsrc_t r_seg, int rel0, int rank, int utid, WsX& X) {
  const int wave = utid / kWave;
  const int lane = utid % kWave;
  const uint32_t base = (static_cast<uint32_t>(rel0 + wave) * rank + lane * 8) * 2u;
#pragma unroll
  for (int h = 0; h < kMfRuns; ++h) X.xv[h] = bload128(r_seg, base + static_cast<uint32_t>(4 * h * rank) * 2u, 0u);
}

// Writes every staged row in natural column order (rows >= rc get the zeros their loads returned): one
// 16-byte LDS write per run, a wave's 64 runs one contiguous kilobyte.
__device__ __forceinline__ void ws_x_write(int utid, uint16_t* xs, const WsX& X) {
  const int wave = utid / kWave;
  const int lane = utid % kWave;
#pragma unroll
  for (int h = 0; h < kMfRuns; ++h) {
    const int r = 4 * h + wave;
    *reinterpret_cast<uint4*>(&xs[r * kWsXStride + lane * 8]) = X.xv[h];
  }
}

// Work split: item (segment a, kSub output tiles from tile kSub * i) costs t_a + kWsBuildCost row tiles (t_a:
// the segment's row tiles; building the B operands costs about kWsBuildCost of them).  Items are ordered
// segment-major, each item's build first and then its row tiles, and the workgroup of virtual index v takes
// the row tiles whose cost position lies in [v * total / W, (v + 1) * total / W), building the B operands of
// every item it touches: an item split between two workgroups is built twice, and every workgroup gets the
// same cost to within one item's build.  Each lane works out the item and row range of its segment, so no
// item list exists anywhere.  Virtual indices are XCD-major: the hardware places workgroup w on XCD w % 8, and each
// XCD gets a contiguous share of the items, so its L2 holds the activations of about one segment instead
// of every XCD streaming every segment.
constexpr int kWsBuildCost = 2;
constexpr int kXcds = 8;  // MI355X: 8 XCDs (32 CUs and one L2 each)

__device__ __forceinline__ int xcd_major_index(int w, int W) {
  const int x = w % kXcds;
  const int q = W / kXcds;
  const int r = W % kXcds;
  return x * q + (x < r ? x : r) + w / kXcds;
}

// kSub output tiles per item: wavefront w computes columns 16 w + (0..15) of each, so one activation read
// from LDS feeds kSub MFMAs (B operands: 16 packed rows x kSub x 4 registers).  Activations are staged in
// natural column order (a plain copy) and the B operands built for it (mf_row_b_nat).
template <int kUnits, int kSub>
__global__ __launch_bounds__(kUnits * kMfThreads) __attribute__((amdgpu_waves_per_eu(2, 8))) void grouped_mfma_ws_kernel(
    MfmaArgs a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char mf_lds[];
  __shared__ __attribute__((aligned(16))) uint32_t ws_tb[kUnits][kSub][kMfTbWords];
  const int unit = kUnits == 2 ? __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kMfThreads) : 0;
  const int utid = static_cast<int>(threadIdx.x) % kMfThreads;
  const MfmaProj& pa = a.proj[kUnits == 2 ? unit : blockIdx.z];
  const tris_compact3_payload& p = pa.p;
  const int N = p.outfeatures;
  const int G = p.num_groups;
  const int nob = ceil_div(N, kTileOut);
  const int nit = ceil_div(nob, kSub);  // items per segment
  const int npr = p.rank / 32;          // <= kMfPR: rank <= kMfChunk (host-checked)
  const int wave = __builtin_amdgcn_readfirstlane(utid / kWave);
  const int lane = utid % kWave;
  const int i16 = lane % 16;
  const int kg = lane / 16;
  const int tc = 16 * wave + i16;
  uint16_t* out = kUnits == 2 ? a.proj[0].out : pa.out;

  // segments (<= 64, host-checked): lane i holds segment i
  const MfSegScan sc = mf_scan_segments(a.segment_offsets, a.expert_ids, a.num_segments, kMfRows);
  const bool act = static_cast<int>(__lane_id()) < a.num_segments && sc.t > 0;
  const int u = act ? sc.t + kWsBuildCost : 0;
  int incl = u;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const int v = __shfl_up(incl, d);
    if (static_cast<int>(__lane_id()) >= d) incl += v;
  }
  const int64_t total = static_cast<int64_t>(nit) * __shfl(incl, kWave - 1);
  const int64_t W = gridDim.x;
  const int64_t vw = xcd_major_index(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
  const int64_t lo_w = vw * total / W;
  const int64_t hi_w = (vw + 1) * total / W;
  const int64_t base = static_cast<int64_t>(nit) * (incl - u);
  // this workgroup's cost range relative to the segment's first item, clamped to the segment's cost; item it
  // covers [it * u, (it + 1) * u), its row tile r sits at it * u + kWsBuildCost + r
  int d0 = 0, d1 = 0, it_lo = 0, it_hi = 0;
  if (act) {
    const int64_t seg_cost = static_cast<int64_t>(nit) * u;
    const int64_t e0 = lo_w - base, e1 = hi_w - base;
    d0 = static_cast<int>(e0 < 0 ? 0 : (e0 > seg_cost ? seg_cost : e0));
    d1 = static_cast<int>(e1 < 0 ? 0 : (e1 > seg_cost ? seg_cost : e1));
    it_lo = d0 / u;  // first item with a row tile at or past d0
    it_hi = d1 > kWsBuildCost ? (d1 - kWsBuildCost + u - 1) / u : 0;  // first item whose row tiles start at or past d1
    it_hi = it_hi < nit ? it_hi : nit;
  }
  uint64_t todo = __ballot(act && it_hi > it_lo);

  const MfWsLayout L = mf_ws_layout();
  unsigned char* lbase = mf_lds + unit * L.bytes;
  MfChunk ch;
  ch.xs = nullptr;
  ch.cds = reinterpret_cast<uint16_t*>(lbase + L.cds);
  ch.cns = reinterpret_cast<uint16_t*>(lbase + L.cns);
  ch.col_sal = reinterpret_cast<uint32_t*>(lbase + L.col_sal);
  ch.sal_col = reinterpret_cast<uint16_t*>(lbase + L.sal_col);
  ch.sal_xi = reinterpret_cast<uint16_t*>(lbase + L.sal_xi);
  ch.sal_cp = reinterpret_cast<uint32_t*>(lbase + L.sal_cp);
  ch.sal_w = nullptr;
  ch.sal_xo = nullptr;
  ch.goff = nullptr;
  ch.meta = reinterpret_cast<int32_t*>(lbase + L.meta);
  uint16_t* const xsb0 = reinterpret_cast<uint16_t*>(lbase + L.xs[0]);
  uint16_t* const xsb1 = reinterpret_cast<uint16_t*>(lbase + L.xs[1]);
  // column kMfChunk of every staged row stays zero (the activation writes cover columns 0 .. 511): the salient
  // gather's padding slots read it
  if (utid < 2 * kMfRows) (utid < kMfRows ? xsb0 : xsb1)[(utid % kMfRows) * kWsXStride + kMfChunk] = 0;
  uint32_t* r01t = reinterpret_cast<uint32_t*>(lbase + L.r01t);
  auto ws = reinterpret_cast<uint16_t (*)[16][kMfSalStride]>(lbase + L.ws);
  float* exch = reinterpret_cast<float*>(mf_lds + kUnits * L.bytes);
  MfTileBuf tb[kSub];
#pragma unroll
  for (int b = 0; b < kSub; ++b) {
    tb[b].q1 = &ws_tb[unit][b][kMfTbQ1];
    tb[b].gw = &ws_tb[unit][b][kMfTbGw];
    tb[b].rs = &ws_tb[unit][b][kMfTbRs];
  }
  while (todo != 0) {
    const int s = __ffsll(static_cast<unsigned long long>(todo)) - 1;  // wave-uniform
    todo &= todo - 1;
    const int seg_lo = __builtin_amdgcn_readfirstlane(__shfl(sc.lo, s));
    const int seg_hi = __builtin_amdgcn_readfirstlane(__shfl(sc.hi, s));
    const int e = __builtin_amdgcn_readfirstlane(__shfl(sc.ex, s));
    const int it0 = __builtin_amdgcn_readfirstlane(__shfl(it_lo, s));
    const int it1 = __builtin_amdgcn_readfirstlane(__shfl(it_hi, s));
    const int sd0 = __builtin_amdgcn_readfirstlane(__shfl(d0, s));
    const int sd1 = __builtin_amdgcn_readfirstlane(__shfl(d1, s));
    const int rows = seg_hi - seg_lo;
    const int nrt = ceil_div(rows, kMfRows);
    const int cu = nrt + kWsBuildCost;
    const bool dead = e < 0 || e >= p.num_experts;  // rows routed to no expert: zero output
    for (int it = it0; it < it1; ++it) {
      // this workgroup's row tiles of the item (never empty: see it_lo, it_hi)
      const int r_lo = max(0, min(nrt, sd0 - it * cu - kWsBuildCost));
      const int r_hi = max(0, min(nrt, sd1 - it * cu - kWsBuildCost));
      const int ob = it * kSub;
      if (dead) {
        if (unit == 0) {
          const int n_lo = ob * kTileOut;
          const int n_hi = ((ob + kSub) * kTileOut) < N ? (ob + kSub) * kTileOut : N;
          const int span = n_hi - n_lo;
          const int row_lo = seg_lo + r_lo * kMfRows;
          const int nrow = min(seg_hi, seg_lo + r_hi * kMfRows) - row_lo;
          for (int idx = utid; idx < nrow * span; idx += kMfThreads) {
            out[static_cast<int64_t>(row_lo + idx / span) * N + n_lo + idx % span] = 0;
          }
        }
        continue;
      }
      __syncthreads();  // the previous item's LDS readers are done
#pragma unroll
      for (int b = 0; b < kSub; ++b) {
        if (ob + b < nob) mf_tile_issue(pa, a.decoded_by_expert ? e : s, e, 0, ob + b, utid, tb[b]);  // uniform
      }
      if (it == it0) {  // the segment's column data
        MfRegs regs;
        mf_chunk_issue(pa, e, 0, utid, regs);
        mf_chunk_write(pa, 0, utid, ch, regs);
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      int n[kSub];
      bool nv[kSub];
#pragma unroll
      for (int b = 0; b < kSub; ++b) {
        n[b] = (ob + b) * kTileOut + tc;
        nv[b] = n[b] < N;
      }
      const int sbase0 = __builtin_amdgcn_readfirstlane(ch.meta[8]);
      const int num_sal = __builtin_amdgcn_readfirstlane(ch.meta[9]) - sbase0;
      uint32_t q2w[kSub][kWsSalWindows + 1];  // qweight2_sparse words of the rows the windows span
      {
        const int q2rows = p.qweight2_sparse_rows;
        const uint32_t q2_bytes = static_cast<uint32_t>(q2rows) * N * 4u;
        const __amdgpu_buffer_rsrc_t r_q2 =
            make_rsrc(p.qweight2_sparse + static_cast<int64_t>(e) * q2rows * N, q2_bytes);
#pragma unroll
        for (int b = 0; b < kSub; ++b) {
          const uint32_t v_q2 = nv[b] ? static_cast<uint32_t>(n[b]) * 4u : q2_bytes;
#pragma unroll
          for (int h = 0; h <= kWsSalWindows; ++h) {
            const int row = (sbase0 >> 5) + h;
            const bool rv = num_sal > 0 && row < q2rows;
            q2w[b][h] = bload32(r_q2, rv ? v_q2 : q2_bytes, static_cast<uint32_t>(rv ? row : 0) * N * 4u);
          }
        }
      }
      // materialised rows: one buffer resource over the segment's activations and one over its outputs (rows
      // past the segment read zeros and drop their stores through the resources' sizes)
      const bool seg_rows = pa.row_index == nullptr;
      const __amdgpu_buffer_rsrc_t r_seg =
          make_rsrc(pa.hidden + static_cast<int64_t>(seg_lo) * p.rank, static_cast<uint32_t>(rows) * p.rank * 2u);
      const uint32_t out_bytes = static_cast<uint32_t>(rows) * N * 2u;
      const __amdgpu_buffer_rsrc_t r_out = make_rsrc(out + static_cast<int64_t>(seg_lo) * N, out_bytes);
      uint32_t ocol[kSub];  // byte offset of the lane's column in row 4 kg of the row tile, or past the outputs
#pragma unroll
      for (int b = 0; b < kSub; ++b) ocol[b] = nv[b] ? static_cast<uint32_t>(4 * kg * N + n[b]) * 2u : 0x80000000u;
      auto x_issue = [&](int rt, WsX& X) {
        const int r0 = seg_lo + rt * kMfRows;
        if (seg_rows) {
          ws_x_issue_seg(r_seg, rt * kMfRows, p.rank, utid, X);
        } else {
          ws_x_issue(pa, r0, min(seg_hi - r0, kMfRows), utid, X);
        }
      };
      // the first two row tiles' activations, in flight while the B operands are built; row tile rt's
      // registers are X[rt % 2], reloaded with row tile rt + 2 once staged
      WsX X0, X1;
      x_issue(r_lo, X0);
      if (kWsXDepth == 2 && r_lo + 1 < r_hi) x_issue(r_lo + 1, X1);

      // columns of the salient activations of each window, two 16-bit offsets a word, in the A operand's slot
      // order (padding slots point at the zero column kMfChunk)
      uint32_t soff[kWsSalWindows][4];
#pragma unroll
      for (int win = 0; win < kWsSalWindows; ++win) {
        const int w0 = win * kMfSalWin;
        const int wn = (num_sal - w0) < kMfSalWin ? (num_sal - w0) : kMfSalWin;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int q0 = 8 * kg + 2 * i;
          uint32_t lo = kMfChunk, hi = kMfChunk;
          if (q0 < wn) {
            const int c = ch.sal_col[w0 + q0];
            lo = static_cast<uint32_t>(c);
          }
          if (q0 + 1 < wn) {
            const int c = ch.sal_col[w0 + q0 + 1];
            hi = static_cast<uint32_t>(c);
          }
          soff[win][i] = lo | (hi << 16);
        }
      }
      // ---- B operands over the whole K, per output tile: the packed rows, then the salient windows (the
      // row scales R0 | R1 << 16 go through r01t, rewritten per tile)
      f16x8 bmain[kSub][kMfPR];
      f16x8 bsal[kSub][kWsSalWindows];
#pragma unroll
      for (int b = 0; b < kSub; ++b) {
#pragma unroll
        for (int t = 0; t < kMfTiles; ++t) {
          const int g = __builtin_amdgcn_readfirstlane(ch.meta[t]);
          const int gi = (tc * G + (g >= 0 ? g : 0)) * 2;
          const uint32_t rdn = g >= 0 ? tb[b].rs[gi + 1] : 0u;
          if ((t & 3) == kg) r01t[t * kTileOut + tc] = g >= 0 ? tb[b].rs[gi] : 0u;
#pragma unroll
          for (int jj = 0; jj < 2; ++jj) {
            const int j = 2 * t + jj;
            bmain[b][j] = f16x8{};
            if (j < npr) {  // uniform
              const int kl = j * 32 + 8 * kg;
              bmain[b][j] = mf_row_b_nat(tb[b].q1[j * kMfQ1Stride + tc], tb[b].gw[j * kTileOut + tc],
                                         *reinterpret_cast<const uint4*>(&ch.cds[kl]),
                                         *reinterpret_cast<const uint4*>(&ch.cns[kl]), rdn, kg);
            }
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();  // r01t written
#pragma unroll
        for (int win = 0; win < kWsSalWindows; ++win) {
          const int w0 = win * kMfSalWin;
          const int wn = (num_sal - w0) < kMfSalWin ? (num_sal - w0) : kMfSalWin;
          bsal[b][win] = f16x8{};
          if (wn > 0) {  // uniform
            const int q2b = (sbase0 + w0) >> 5;
            const uint32_t q2pair[2] = {q2w[b][win], q2w[b][win + 1]};
            mf_salient_weights(ch, tb[b], r01t, tc, kg, wave, i16, sbase0, w0, wn, q2b, q2pair, ws);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
            bsal[b][win] = __builtin_bit_cast(f16x8, *reinterpret_cast<const uint4*>(&ws[wave][i16][8 * kg]));
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();  // ws (and, after the last window, r01t) are rewritten next
          }
        }
      }

      // ---- the segment's row tiles through the stationary B operands
      auto row_tile = [&](int rt, uint16_t* xs, WsX& X) {
        ws_x_write(utid, xs, X);
        __syncthreads();  // staged rows visible; the previous row tile's exch reads are done
        if (rt + kWsXDepth < r_hi) x_issue(rt + kWsXDepth, X);  // depth 1: X0 is the only register set
        const uint16_t* xr = xs + i16 * kWsXStride;
        f32x4 acc[kSub];
#pragma unroll
        for (int b = 0; b < kSub; ++b) acc[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        // activations at the salient columns of window win (their A operand)
        auto sal_gather = [&](int win) {
          uint32_t ap[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t lo = xr[soff[win][i] & 0xFFFFu];
            const uint32_t hi = xr[soff[win][i] >> 16];
            ap[i] = lo | (hi << 16);
          }
          return __builtin_bit_cast(f16x8, make_uint4(ap[0], ap[1], ap[2], ap[3]));
        };
        auto row_mfma = [&](int j) {
          const f16x8 av = __builtin_bit_cast(f16x8, *reinterpret_cast<const uint4*>(&xr[j * 32 + 8 * kg]));
#pragma unroll
          for (int b = 0; b < kSub; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bmain[b][j], acc[b], 0, 0, 0);
        };
        // window 0 always runs (zero weights and the zero column when the chunk has no salient column), so it
        // joins the main block: its gathers are issued first and its MFMA comes last
        const f16x8 as0 = sal_gather(0);
        if (npr == kMfPR) {  // rank 512: no branch between the MFMAs, so the LDS reads run ahead of them
#pragma unroll
          for (int j = 0; j < kMfPR; ++j) row_mfma(j);
#pragma unroll
          for (int b = 0; b < kSub; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as0, bsal[b][0], acc[b], 0, 0, 0);
          // schedule: kWsReadAhead A reads, then one MFMA group per further read
          __builtin_amdgcn_sched_group_barrier(0x100, kWsReadAhead, 0);
#pragma unroll
          for (int j = kWsReadAhead; j < kMfPR; ++j) {
            __builtin_amdgcn_sched_group_barrier(0x008, kSub, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          }
          __builtin_amdgcn_sched_group_barrier(0x008, (kWsReadAhead + 1) * kSub, 0);
        } else {
#pragma unroll
          for (int j = 0; j < kMfPR; ++j) {
            if (j < npr) row_mfma(j);  // uniform
          }
#pragma unroll
          for (int b = 0; b < kSub; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(as0, bsal[b][0], acc[b], 0, 0, 0);
        }
#pragma unroll
        for (int win = 1; win < kWsSalWindows; ++win) {
          if (win * kMfSalWin < num_sal) {  // uniform
            const f16x8 av = sal_gather(win);
#pragma unroll
            for (int b = 0; b < kSub; ++b) acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(av, bsal[b][win], acc[b], 0, 0, 0);
          }
        }
        if (kUnits == 2) {
          if (unit == 1) {
#pragma unroll
            for (int b = 0; b < kSub; ++b) *reinterpret_cast<f32x4*>(&exch[(b * kMfThreads + utid) * 4]) = acc[b];
          }
          __syncthreads();
          if (unit == 0) {
#pragma unroll
            for (int b = 0; b < kSub; ++b) {
              const f32x4 up = *reinterpret_cast<const f32x4*>(&exch[(b * kMfThreads + utid) * 4]);
#pragma unroll
              for (int v = 0; v < 4; ++v) {
                __builtin_amdgcn_raw_buffer_store_b16(swiglu_bits(f2h_bits(acc[b][v]), f2h_bits(up[v])), r_out,
                                                      ocol[b] + static_cast<uint32_t>(rt * kMfRows + v) * N * 2u, 0u, 0);
              }
            }
          }
        } else {
#pragma unroll
          for (int b = 0; b < kSub; ++b) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              __builtin_amdgcn_raw_buffer_store_b16(f2h_bits(acc[b][v]), r_out,
                                                    ocol[b] + static_cast<uint32_t>(rt * kMfRows + v) * N * 2u, 0u, 0);
            }
          }
        }
      };
      // two activation buffers in alternation (distinct objects per call site)
      for (int rt = r_lo; rt < r_hi; rt += 2) {
        row_tile(rt, xsb0, X0);
        if (rt + 1 < r_hi) row_tile(rt + 1, xsb1, kWsXDepth == 2 ? X1 : X0);
      }
    }
  }
}

int check_payload(const tris_compact3_payload* p, bool need_gr, const char* who);
int predecode_linears(const tris_gr_predecode_job* jobs, int num_jobs, const int32_t* expert0, void* stream,
                      const char* who);

static bool allow_mfma_lds(const void* kernel, int bytes) {
  // dynamic LDS granted so far per kernel (the weight-stationary kernel's two instantiations)
  static const void* kernels[2] = {reinterpret_cast<const void*>(&grouped_mfma_ws_kernel<1, kWsSub>),
                                   reinterpret_cast<const void*>(&grouped_mfma_ws_kernel<2, kWsSub>)};
  static int granted[2] = {0, 0};
  int which = 0;
  while (which < 1 && kernels[which] != kernel) ++which;
  if (bytes <= granted[which]) return true;
  // Raising the dynamic LDS limit is not a stream operation, so it is safe while a caller captures a graph.
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  granted[which] = bytes;
  return true;
}

// Weight-stationary launch (long segments, one 512-column chunk, <= 64 salient columns per expert):
// workgroups as the GPU holds at once (the occupancy the compiled kernel allows with this LDS), no more
// than the items.
static int launch_grouped_mfma_ws(const MfmaArgs& args, int units, int nproj, int max_n, int batch,
                                  hipStream_t s, const char* who) {
  const int lds = mf_ws_lds_bytes(units, kWsSub);
  const int lds_total = lds + units * kWsSub * kMfTbWords * 4;
  TRIS_REQUIRE(lds_total <= 160 * 1024, "%s: LDS request %d exceeds a CU", who, lds_total);
  const void* kernel = units == 2 ? reinterpret_cast<const void*>(&grouped_mfma_ws_kernel<2, kWsSub>)
                                  : reinterpret_cast<const void*>(&grouped_mfma_ws_kernel<1, kWsSub>);
  TRIS_REQUIRE(allow_mfma_lds(kernel, lds), "%s: %s", who, "cannot raise the kernel's dynamic LDS limit");
  static int per_cu[2] = {0, 0};  // resident workgroups per CU, per kernel (queried once)
  int& wgs_per_cu = per_cu[units - 1];
  if (wgs_per_cu == 0) {
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, units * kMfThreads, lds) != hipSuccess) {
      (void)hipGetLastError();
      nb = 1;
    }
    wgs_per_cu = nb > 0 ? nb : 1;
  }
  int wgs = (kMfCus * wgs_per_cu) / nproj;
  // an upper bound of the work's cost in row tiles (each segment's last row tile may be partial, and every
  // item has its build): workgroups past it would find no row tile
  const int64_t items = static_cast<int64_t>(args.num_segments) * ceil_div(ceil_div(max_n, kTileOut), kWsSub);
  const int64_t cost = static_cast<int64_t>(ceil_div(ceil_div(max_n, kTileOut), kWsSub)) *
                           (ceil_div(batch, kMfRows) + args.num_segments) +
                       items * kWsBuildCost;
  if (cost < wgs) wgs = static_cast<int>(cost);
  const dim3 grid(wgs > 0 ? wgs : 1, 1, nproj);
  if (units == 2) {
    hipLaunchKernelGGL((grouped_mfma_ws_kernel<2, kWsSub>), grid, dim3(2 * kMfThreads), lds, s, args);
  } else {
    hipLaunchKernelGGL((grouped_mfma_ws_kernel<1, kWsSub>), grid, dim3(kMfThreads), lds, s, args);
  }
  return check_launch(who);
}

// The decode kernel may load a projection's weight words 16 bytes at a time: 16-byte aligned tensors and a column
// count that is a multiple of 4, so that no load straddles a row's or the tensor's end.
static bool mf_wide(const MfmaProj& p) {
  const auto al = [](const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; };
  return p.p.outfeatures % 4 == 0 && al(p.p.qweight1) && al(p.p.row_pack3) && al(p.decoded);
}

// Workgroups of a decode launch: as many as the GPU holds at once (LDS and the kernel's registers, mf_waves, bound them),
// shared by the projections of an unfused pair.
static int mf_workgroups(int units, int rows, bool compact, int nproj) {
  int per_cu = (160 * 1024) / mf_static_lds_bytes(units, rows, compact);
  const int by_regs = units == 1 ? mf_waves(units, rows, compact) : 1;
  per_cu = per_cu < by_regs ? per_cu : by_regs;
  return kMfCus * (per_cu > 0 ? per_cu : 1) / nproj;
}

// The sizes of a predecoded launch that pick its kernel (of a pair: the larger of the two).
struct MfShape {
  int rank, n, groups, q2rows;
  bool single;    // weight words one at a time (mf_wide does not hold)
  bool swiglu;    // the pair side by side (two units)
  bool gathered;  // rows read through row_index
  int nproj;      // projections of one unit each
};

// The compact LDS layout: a chunk of 256 columns (rank <= 256), at most 4 row-scale groups and 64 salient columns per
// expert.  The 64-row tiles fit in it three workgroups a CU.
static bool mf_compact(const MfShape& h) {
  return !h.single && h.groups <= mf_groups_cap(true) && h.q2rows * kMfSalWin <= mf_sal_slots(true) &&
         h.rank <= kMfChunk / 2;
}

// Whether a launch goes weight-stationary.  Below 64 rows a segment on average none does; from 120 rows on (500 in the
// compact layout) every one does (Mixtral's gate/up + down, decode against weight-stationary: 130 rows 153 / 149 us, 150
// rows 167 / 155; OLMoE's 500 rows 240 / 243).  Between them neither kernel is always the faster one: weight-stationary
// takes from 0.70 (64 segments of 65 rows, N = 512, rank 512, SwiGLU: 28 against 39 us) to 1.6 times the decode kernel's
// time (8 of 65, N = 2048, one projection: 21 against 13).  It pays for each item a workgroup touches (building its
// operands) and little for the rows, the decode kernel for each pair of a 32- or 64-row tile and an output tile, and both
// wait for the workgroup with the most of them.  So their times are estimated, us = constant + cost x that workgroup's
// count, the part of a cost proportional to the rank apart, fitted over 769 launches of 1 to 64 segments, N 512 to 14336,
// ranks 64 to 512 (90 with gathered rows).  The kernel picked there is at most 3% slower than the weight-stationary one,
// 20 to 25% faster in the mean, and 0.3 to 0.7% slower in the mean than always the better one.  Single-word launches,
// which the fit does not cover, go weight-stationary from 64 rows.
constexpr int kWsMinRows = 64;
constexpr int kWsAlwaysRows = 120;
constexpr int kWsAlwaysRowsCompact = 500;
struct MfCost {
  float ws, build, build_k, row, row_k;  // weight-stationary: constant, an item, 16 rows of one (_k: times rank / 512)
  float dec, tile, tile_k;               // decode: constant, a pair of a row tile and an output tile
};
constexpr MfCost kMfCost[3][2] = {
    // one unit                                                    SwiGLU
    {{10.4f, 2.1f, 4.5f, 1.65f, 0.45f, 6.0f, 0.8f, 2.6f}, {7.7f, 5.9f, 5.2f, 1.46f, 0.41f, 6.9f, 1.3f, 2.8f}},
    {{7.6f, 6.0f, 5.7f, 0.73f, 0.82f, 7.2f, 2.0f, 4.0f}, {8.0f, 6.3f, 6.0f, 1.08f, 0.79f, 7.0f, 2.2f, 2.9f}},  // compact
    {{7.7f, -0.4f, 12.9f, 2.67f, -0.72f, 6.0f, 0.8f, 2.6f}, {5.6f, -2.9f, 18.8f, 3.45f, -1.46f, 6.9f, 1.3f, 2.8f}},  // gathered
};

static bool mf_weight_stationary(const MfShape& h, int64_t batch, int segments) {
  if (segments < 1 || segments > kWave || batch < int64_t{kWsMinRows} * segments) return false;
  // one chunk, the salient windows it holds, and 32-bit byte offsets over the whole batch
  if (h.rank > kMfChunk || h.q2rows > kWsSalWindows || batch * h.n * 2 >= (int64_t{1} << 31) ||
      batch * kMfChunk * 2 >= (int64_t{1} << 31)) {
    return false;
  }
  if (h.single) return true;
  const bool compact = mf_compact(h);
  if (batch >= int64_t{compact ? kWsAlwaysRowsCompact : kWsAlwaysRows} * segments) return true;
  if (compact && h.gathered) return false;  // gathering costs the weight-stationary kernel more than its rows save
  const MfCost& c = kMfCost[compact ? 1 : h.gathered ? 2 : 0][h.swiglu ? 1 : 0];
  const float f = static_cast<float>(h.rank) / 512.0f;
  const int nob = ceil_div(h.n, kTileOut);
  const int64_t mean = (batch + segments - 1) / segments;
  // weight-stationary: `items` shared by W workgroups in equal parts, p / q items each: the unluckiest starts (q - 1) / q
  // into one
  const int64_t items = static_cast<int64_t>(segments) * ceil_div(nob, kWsSub);
  const int64_t row_tiles = (mean + kMfRows - 1) / kMfRows;
  const int64_t cost = items * (row_tiles + kWsBuildCost);
  int64_t w = h.swiglu ? kMfCus : 2 * kMfCus / h.nproj;
  w = cost < w ? cost : w;
  int64_t p = items, q = w;
  for (int64_t x = p, y = q;;) {  // by their greatest common divisor
    const int64_t m = x % y;
    if (m == 0) {
      p /= y;
      q /= y;
      break;
    }
    x = y;
    y = m;
  }
  const float visits = static_cast<float>((p + 2 * q - 2) / q);
  const float rows = static_cast<float>(row_tiles) * static_cast<float>(items) / static_cast<float>(w);
  const float ws = c.ws + visits * (c.build + c.build_k * f) + rows * (c.row + c.row_k * f);
  // decode: the longest run, as the kernel splits them
  const int tile = compact ? 64 : 32;
  const int64_t rt = segments * ((mean + tile - 1) / tile);
  const int64_t pairs = rt * nob;
  const int64_t wd = mf_workgroups(h.swiglu ? 2 : 1, tile, compact, h.nproj);
  int64_t run;
  if (rt * 3 <= wd || (rt <= wd && pairs < 8 * wd)) {
    const int64_t per = wd / rt < nob ? wd / rt : nob;
    run = (nob + per - 1) / per;
  } else {
    run = (pairs + wd - 1) / wd;
  }
  const float dec = c.dec + static_cast<float>(run) * (c.tile + c.tile_k * f);
  return dec * 1.08f >= ws;  // (the estimates' own error)
}

int launch_grouped_mfma(const uint16_t* hidden_a, const uint16_t* hidden_b, int batch, const int32_t* expert_ids,
                        const int32_t* segment_offsets, int num_segments, const int32_t* decoded_a,
                        const int32_t* decoded_b, const tris_compact3_payload* pa, const tris_compact3_payload* pb,
                        uint16_t* out_a, uint16_t* out_b, bool swiglu, void* stream, const char* who,
                        const int64_t* row_index, int hidden_rows, bool decoded_by_expert, const float* partials,
                        int slices, uint16_t* comb_out, const int32_t* comb_inv, const uint16_t* comb_w,
                        bool comb_bf16) {
  TRIS_REQUIRE(batch >= 0 && num_segments >= 0, "%s: negative batch or segment count", who);
  TRIS_REQUIRE(row_index == nullptr || hidden_rows >= 0, "%s: negative hidden row count", who);
  int rc = check_payload(pa, false, who);
  if (rc) return rc;
  if (pb) {
    rc = check_payload(pb, false, who);
    if (rc) return rc;
  }
  TRIS_REQUIRE(!swiglu || pb != nullptr, "%s: the fused SwiGLU needs two projections", who);
  TRIS_REQUIRE(!pa->has_output_scale && !pa->has_bias && (!pb || (!pb->has_output_scale && !pb->has_bias)),
               "%s: the MFMA GEMM applies no output scale or bias", who);
  if (batch == 0 || num_segments == 0) return TRIS_OK;
  TRIS_REQUIRE((hidden_a || partials) && out_a && expert_ids && segment_offsets && decoded_a, "%s: null pointer", who);
  if (comb_out != nullptr) {
    // one token routed to two experts: two rows, two segments, one projection
    TRIS_REQUIRE(pb == nullptr && !swiglu && row_index == nullptr && comb_inv && comb_w,
                 "%s: the one-token combine takes one projection and the route's picks", who);
    TRIS_REQUIRE(batch == 2 && num_segments == 2, "%s: the one-token combine takes 2 rows in 2 segments", who);
  }
  if (partials != nullptr) {
    // one projection, one chunk, every slice's rows addressed by 32-bit buffer offsets
    TRIS_REQUIRE(pb == nullptr && !swiglu && row_index == nullptr, "%s: partial sums feed one projection", who);
    TRIS_REQUIRE(pa->rank <= kMfChunk, "%s: partial sums need rank <= %d (one chunk)", who, kMfChunk);
    TRIS_REQUIRE(slices >= 1 && hidden_rows >= batch, "%s: bad partial-sum shape", who);
    TRIS_REQUIRE(batch <= 4, "%s: partial sums take at most 4 rows (%d given)", who, batch);
    TRIS_REQUIRE(static_cast<int64_t>(slices) * hidden_rows * pa->rank * 4 < (int64_t{1} << 31),
                 "%s: partial sums exceed the 2 GiB limit", who);
  }
  TRIS_REQUIRE(!pb || (hidden_b && decoded_b && (swiglu || out_b)), "%s: null pointer (second projection)", who);
  int max_n = 0;
  for (int i = 0; i < (pb ? 2 : 1); ++i) {
    const tris_compact3_payload* p = i ? pb : pa;
    TRIS_REQUIRE(p->num_experts > 0 && p->rank > 0 && p->outfeatures > 0, "%s: empty payload", who);
    max_n = p->outfeatures > max_n ? p->outfeatures : max_n;
  }
  TRIS_REQUIRE(!swiglu || (pa->outfeatures == pb->outfeatures && pa->num_experts == pb->num_experts &&
                           pa->rank == pb->rank),
               "%s: gate and up projections differ in shape", who);
  if (row_index != nullptr) {
    // gathered rows: one 32-bit buffer offset spans every hidden row
    const int64_t bytes = static_cast<int64_t>(hidden_rows) * (pb && pb->rank > pa->rank ? pb->rank : pa->rank) * 2;
    TRIS_REQUIRE(bytes < (int64_t{1} << 31), "%s: %d hidden rows exceed the 2 GiB activation limit", who,
                 hidden_rows);
  }
  MfmaArgs args{};
  args.proj[0] = MfmaProj{hidden_a, out_a, decoded_a, *pa, row_index, hidden_rows, partials, slices};
  if (pb) args.proj[1] = MfmaProj{hidden_b, out_b, decoded_b, *pb, row_index, hidden_rows};
  args.expert_ids = expert_ids;
  args.segment_offsets = segment_offsets;
  args.num_segments = num_segments;
  args.batch = batch;
  args.decoded_by_expert = decoded_by_expert ? 1 : 0;
  if (comb_out != nullptr) {  // both units run the one projection, on row tiles 0 and 1
    args.proj[1] = args.proj[0];
    args.comb_out = comb_out;
    args.comb_inv = comb_inv;
    args.comb_w = comb_w;
    args.comb_bf16 = comb_bf16 ? 1 : 0;
  }
  const int units = (swiglu || comb_out != nullptr) ? 2 : 1;
  const int nproj = (pb && !swiglu) ? 2 : 1;
  hipStream_t s = static_cast<hipStream_t>(stream);
  MfShape shape{pa->rank, max_n, pa->num_groups, pa->qweight2_sparse_rows, !mf_wide(args.proj[0]), swiglu,
                row_index != nullptr, nproj};
  if (pb) {
    shape.rank = pb->rank > shape.rank ? pb->rank : shape.rank;
    shape.groups = pb->num_groups > shape.groups ? pb->num_groups : shape.groups;
    shape.q2rows = pb->qweight2_sparse_rows > shape.q2rows ? pb->qweight2_sparse_rows : shape.q2rows;
    shape.single = shape.single || !mf_wide(args.proj[1]);
  }
  const bool chunks = shape.rank > kMfChunk;  // more than one 512-column chunk
  const bool single = shape.single;
  const bool compact = mf_compact(shape);
  // long segments: keep each output tile's weights in registers and stream the segment's rows through them
  if (partials == nullptr && comb_out == nullptr && mf_weight_stationary(shape, batch, num_segments)) {
    return launch_grouped_mfma_ws(args, units, nproj, max_n, batch, s, who);
  }
  // Staged activation rows: a row tile has at most min(row tile, batch).  From kMfTallMinRows rows a segment on average,
  // row tiles of 32 rows (64 at rank <= 256, where they take half the LDS): a segment then rarely needs two, and its
  // weights are built once, not once every 16 rows.
  const int64_t tall_min = single ? kMfTallMinRowsSingle : kMfTallMinRows;
  const bool tall = !chunks && partials == nullptr && static_cast<int64_t>(batch) >= tall_min * num_segments &&
                    static_cast<int64_t>(max_n) * (compact ? 64 : 32) * 2 < (int64_t{1} << 31);
  const int rows = batch <= 4 ? 4 : (!tall ? kMfRows : (compact ? 64 : 32));
  const int lds_total = mf_static_lds_bytes(units, rows, compact);
  TRIS_REQUIRE(lds_total <= 160 * 1024, "%s: LDS request %d exceeds a CU", who, lds_total);
  int wgs = mf_workgroups(units, rows, compact, nproj);
  // no more than the (row tile, output tile) pairs there can be: row tiles <= batch / row tile + min(segments, batch)
  const int64_t pairs = (static_cast<int64_t>(batch) / (rows > kMfRows ? rows : kMfRows) +
                         (num_segments < batch ? num_segments : batch)) * ceil_div(max_n, kTileOut);
  if (pairs < wgs) wgs = static_cast<int>(pairs);
  if (comb_out != nullptr && ceil_div(max_n, kTileOut) < wgs) wgs = ceil_div(max_n, kTileOut);  // output tiles only
  const dim3 grid(wgs > 0 ? wgs : 1, 1, nproj);
  const dim3 block(units * kMfThreads);
#define TRIS_MF_LAUNCH(ROWS, C, S, M)                                                                        \
  do {                                                                                                       \
    if (units == 2) hipLaunchKernelGGL((grouped_mfma_kernel<2, ROWS, C, S, M>), grid, block, 0, s, args);    \
    else hipLaunchKernelGGL((grouped_mfma_kernel<1, ROWS, C, S, M>), grid, block, 0, s, args);               \
  } while (0)
  if (chunks) {
    if (rows == 4 && single) TRIS_MF_LAUNCH(4, false, true, true);
    else if (rows == 4) TRIS_MF_LAUNCH(4, false, false, true);
    else if (single) TRIS_MF_LAUNCH(kMfRows, false, true, true);
    else TRIS_MF_LAUNCH(kMfRows, false, false, true);
  } else if (single) {
    if (rows == 4) TRIS_MF_LAUNCH(4, false, true, false);
    else if (rows == 32) TRIS_MF_LAUNCH(32, false, true, false);
    else TRIS_MF_LAUNCH(kMfRows, false, true, false);
  } else if (compact) {
    if (rows == 4) TRIS_MF_LAUNCH(4, true, false, false);
    else if (rows == 64) TRIS_MF_LAUNCH(64, true, false, false);
    else TRIS_MF_LAUNCH(kMfRows, true, false, false);
  } else {
    if (rows == 4) TRIS_MF_LAUNCH(4, false, false, false);
    else if (rows == 32) TRIS_MF_LAUNCH(32, false, false, false);
    else TRIS_MF_LAUNCH(kMfRows, false, false, false);
  }
#undef TRIS_MF_LAUNCH
  return check_launch(who);
}

// Slices of a linear's K: chunks are split until one matrix's launch has about three workgroups a CU (whatever the number
// of matrices, so that each gives the same bits alone and beside others of its width).  With more than one slice there
// are fewer than 1536 (tile, slice) pairs of at most 32 x 64 sums, so the partial sums stay below 12 MiB a matrix however
// long the batch.
static int lin_slices(int batch, int rank, int max_n) {
  const int chunks = ceil_div(rank, kMfChunk);
  const int64_t tiles = static_cast<int64_t>(ceil_div(max_n, kTileOut)) * ceil_div(batch, batch <= kMfRows ? kMfRows : 32);
  const int64_t want = tiles > 0 ? (3 * kMfCus + tiles - 1) / tiles : 1;
  return static_cast<int>(want < chunks ? want : chunks);
}

static int64_t lin_decoded_words(int rank, int n) {
  return static_cast<int64_t>((rank / 32 + 1) / 2) * ceil_div(n, kTileOut) * kGrWords;
}

int64_t linear_mfma_workspace(int batch, int rank, const int32_t* outfeatures, int count) {
  int max_n = 0;
  int64_t words = 0, sums = 0;
  for (int i = 0; i < count; ++i) {
    max_n = outfeatures[i] > max_n ? outfeatures[i] : max_n;
    words += lin_decoded_words(rank, outfeatures[i]);
    sums += static_cast<int64_t>(batch) * outfeatures[i];
  }
  const int slices = lin_slices(batch, rank, max_n);
  return 4 * (words + (slices > 1 ? sums * slices : 0));
}

// The matrix sizes linear_mfma_kernel takes: whole 64-column K tiles, every 32-bit buffer offset below 2 GiB.
static bool lin_fits(const tris_compact3_payload* p) {
  const int64_t limit = int64_t{1} << 31;
  const int64_t n = p->outfeatures;
  return p->rank > 0 && p->rank % kTileK == 0 && n > 0 && p->num_groups > 0 &&
         static_cast<int64_t>(p->rank / 32) * n * 4 < limit && int64_t{p->qweight2_sparse_rows} * n * 4 < limit &&
         n * p->num_groups * 8 < limit && lin_decoded_words(p->rank, p->outfeatures) * 4 < limit &&
         int64_t{32} * p->rank * 2 < limit && int64_t{p->rank} * 8 < limit;
}

// Entry 0 of an expert list: the matrix itself.
__device__ int32_t lin_expert0[4];

int launch_linear_mfma(const uint16_t* input, int batch, const tris_compact3_payload* payloads, int count,
                       const uint16_t* input_scale, const float* addend, uint16_t* const* outs, void* workspace,
                       int64_t workspace_bytes, void* stream, const char* who) {
  TRIS_REQUIRE(batch >= 0 && count >= 1 && count <= TRIS_MAX_LINEARS && payloads && outs, "%s: bad arguments", who);
  LinArgs args{};
  int max_n = 0;
  int32_t widths[TRIS_MAX_LINEARS];
  bool wide = true;
  for (int i = 0; i < count; ++i) {
    const tris_compact3_payload* p = payloads + i;
    int rc = check_payload(p, true, who);
    if (rc) return rc;
    TRIS_REQUIRE(p->num_experts == 1 && p->q_gmap_gr_offsets != nullptr,
                 "%s: a non-expert payload holds one block-GR matrix", who);
    TRIS_REQUIRE(p->rank == payloads[0].rank, "%s: the matrices' ranks differ", who);
    TRIS_REQUIRE(lin_fits(p), "%s: rank must be a multiple of %d and the tensors below 2 GiB", who, kTileK);
    widths[i] = p->outfeatures;
    max_n = p->outfeatures > max_n ? p->outfeatures : max_n;
  }
  if (batch == 0) return TRIS_OK;
  TRIS_REQUIRE(input && workspace, "%s: null pointer", who);
  TRIS_REQUIRE(reinterpret_cast<uintptr_t>(input) % 16 == 0 && reinterpret_cast<uintptr_t>(input_scale) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(workspace) % 16 == 0,
               "%s: input, input_scale and workspace must be 16-byte aligned", who);
  const int rank = payloads[0].rank;
  TRIS_REQUIRE(workspace_bytes >= linear_mfma_workspace(batch, rank, widths, count), "%s: workspace too small", who);
  void* ids = nullptr;
  TRIS_REQUIRE(hipGetSymbolAddress(&ids, HIP_SYMBOL(lin_expert0)) == hipSuccess, "%s: no expert list", who);
  args.x = input;
  args.in_scale = input_scale;
  args.batch = batch;
  args.chunks = ceil_div(rank, kMfChunk);
  args.slices = lin_slices(batch, rank, max_n);
  int32_t* words = static_cast<int32_t*>(workspace);
  tris_gr_predecode_job jobs[TRIS_MAX_LINEARS];
  for (int i = 0; i < count; ++i) {
    const tris_compact3_payload& p = payloads[i];
    TRIS_REQUIRE(outs[i], "%s: null pointer", who);
    args.proj[i].p = p;
    args.proj[i].decoded = words;
    args.proj[i].out = outs[i];
    args.proj[i].addend = i == 0 ? addend : nullptr;
    jobs[i] = tris_gr_predecode_job{words, p.q_gmap_gr_words, p.q_gmap_gr_offsets, p.q_gmap_gr_meta, 1,
                                    p.gr_words_stride, rank / 32, p.outfeatures};
    words += lin_decoded_words(rank, p.outfeatures);
    const MfmaProj probe{nullptr, nullptr, args.proj[i].decoded, p, nullptr, 0, nullptr, 0};
    wide = wide && mf_wide(probe);
  }
  float* sums = reinterpret_cast<float*>(words);
  for (int i = 0; i < count && args.slices > 1; ++i) {
    args.proj[i].part = sums;
    sums += static_cast<int64_t>(args.slices) * batch * widths[i];
  }
  int rc = predecode_linears(jobs, count, static_cast<const int32_t*>(ids), stream, who);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int rows = batch <= kMfRows ? kMfRows : 32;
  // grid.y is limited to 65535: longer batches go in several launches of whole row tiles (with more than one slice there
  // are fewer than 1536 (tile, slice) pairs, so one launch)
  const int per = args.slices > 1 ? batch : 65535 * rows;
  for (int b0 = 0; b0 < batch; b0 += per) {
    LinArgs part = args;
    part.x = input + static_cast<int64_t>(b0) * rank;
    part.batch = batch - b0 < per ? batch - b0 : per;
    for (int i = 0; i < count; ++i) {
      part.proj[i].out = args.proj[i].out + static_cast<int64_t>(b0) * widths[i];
      if (args.proj[i].addend != nullptr) part.proj[i].addend = args.proj[i].addend + static_cast<int64_t>(b0) * widths[i];
    }
    const dim3 grid(ceil_div(max_n, kTileOut), ceil_div(part.batch, rows) * args.slices, count);
    if (rows == kMfRows) {
      if (wide) hipLaunchKernelGGL((linear_mfma_kernel<kMfRows, false>), grid, dim3(kMfThreads), 0, s, part);
      else hipLaunchKernelGGL((linear_mfma_kernel<kMfRows, true>), grid, dim3(kMfThreads), 0, s, part);
    } else {
      if (wide) hipLaunchKernelGGL((linear_mfma_kernel<32, false>), grid, dim3(kMfThreads), 0, s, part);
      else hipLaunchKernelGGL((linear_mfma_kernel<32, true>), grid, dim3(kMfThreads), 0, s, part);
    }
    if (args.slices == 1) continue;
    const int ty = part.batch < 4096 ? part.batch : 4096;
    hipLaunchKernelGGL(linear_finish_kernel, dim3(ceil_div(max_n, 256), ty, count), dim3(256), 0, s, part);
  }
  return check_launch(who);
}

// True when the MFMA kernel can run this payload: uniform 64-column groups (so
// a 64-column K tile has one row scale) and a rank that is a whole number of
// 64-column tiles, with 16-byte aligned activations (8-column loads).
bool grouped_mfma_supported(const tris_compact3_payload* p, const uint16_t* hidden) {
  if (p == nullptr || !p->use_uniform_k64_groups || p->rank <= 0 || p->rank % kTileK != 0 ||
      p->num_groups < 1 || p->num_groups > kMfMaxGroups || reinterpret_cast<uintptr_t>(hidden) % 16 != 0) {
    return false;
  }
  // the kernel addresses each expert's tensors with 32-bit buffer offsets
  const int64_t limit = int64_t{1} << 31;
  const int64_t packed_rows = (p->rank + 31) / 32;
  const int64_t n = p->outfeatures;
  return packed_rows * n * 4 < limit && int64_t{p->qweight2_sparse_rows} * n * 4 < limit &&
         n * p->num_groups * 8 < limit && int64_t{kMfRows} * p->rank * 2 < limit &&
         ((packed_rows + 1) / 2) * ((n + kTileOut - 1) / kTileOut) * kGrWords * 4 < limit;
}

}  // namespace tris

extern "C" int tris_grouped_predecoded_weight_stationary(int32_t rank, int32_t outfeatures, int32_t num_groups,
                                                         int32_t qweight2_sparse_rows, int32_t wide,
                                                         int32_t projections, int32_t swiglu, int32_t gathered,
                                                         int64_t rows, int32_t segments) {
  if (rank < 1 || outfeatures < 1 || rows < 0 || rows > INT32_MAX || projections < 1 || projections > 2 || (swiglu && projections != 2)) return 0;
  const tris::MfShape h{rank, outfeatures, num_groups, qweight2_sparse_rows, wide == 0, swiglu != 0, gathered != 0,
                        swiglu ? 1 : projections};
  return tris::mf_weight_stationary(h, rows, segments) ? 1 : 0;
}

extern "C" int64_t tris_compact3_linears_workspace_bytes(int32_t batch, int32_t rank, const int32_t* outfeatures,
                                                         int32_t count) {
  if (batch < 0 || rank <= 0 || count < 1 || count > TRIS_MAX_LINEARS || outfeatures == nullptr) return 0;
  return tris::linear_mfma_workspace(batch, rank, outfeatures, count);
}

extern "C" int tris_compact3_linears_forward(const uint16_t* input, int32_t batch, const tris_compact3_payload* payloads,
                                             int32_t count, const uint16_t* input_scale, const float* addend,
                                             uint16_t* const* outputs, void* workspace, int64_t workspace_bytes,
                                             void* stream) {
  return tris::launch_linear_mfma(input, batch, payloads, count, input_scale, addend, outputs, workspace,
                                  workspace_bytes, stream, "tris_compact3_linears_forward");
}
