// MFMA tile primitives for gfx950 shared by the chunk kernels.
//
// All block-level products have the "NT" form C[M x N] += A[M x K] * B[N x K]^T with both
// operands K-contiguous in LDS, which is the native operand layout of the 32x32 MFMA
// instructions: lane = (row r = lane & 31, k-group kg = lane >> 5) holds VEC consecutive
// k-elements of row r.  bf16 uses v_mfma_f32_32x32x16_bf16 (8 elements per lane), fp32 uses
// four v_mfma_f32_32x32x2_f32 per 8-wide k-step (4 elements per lane).
//
// Accumulator fragment (floatx16) of one 32x32 tile: element e of lane l is
//   row = 8 * (e / 4) + 4 * (l >> 5) + (e % 4),  col = l & 31.
// Four consecutive e share a column and cover four consecutive rows, so a fragment can be
// written transposed ([col][row]) with 4-element vector stores.
#pragma once

#include "lnx_common.h"

#define LNX_C 64  // chunk length (tokens)

template <typename T> struct Mma;

template <> struct Mma<bf16_t> {
  static constexpr int KS = 16;   // k per step
  static constexpr int VEC = 8;   // elements per lane per step == elements per 16-byte vector
  static constexpr int PAD = 8;   // LDS row padding (elements) = 16 bytes
  typedef bf16x8 Frag;
  typedef bf16x4 Quad;
  static __device__ __forceinline__ Frag load(const bf16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }
  static __device__ __forceinline__ void mma(floatx16& c, const Frag& a, const Frag& b) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
  // Operand fragment whose contraction index runs along the ROWS of a row-major LDS tile:
  // lane (r = lane & 31, kg = lane >> 5) gets tile[k0 + 8 kg + 0..7][c0 + r].  Two
  // ds_read_b64_tr_b16: inside a 16-lane group, result element j of lane L is element (L % 4) of
  // what lane 4 j + L / 4 addressed, so source lane s = 4 j + q points at row j, columns 4 q .. 4 q + 3.
  static __device__ __forceinline__ Frag load_t(const bf16_t* tile, int ld, int k0, int c0, int lane) {
    typedef short short4_ __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) short4_ lds_short4;
    const int s = lane & 15, grp = lane >> 4;
    const bf16_t* p = tile + (k0 + 8 * (grp >> 1) + (s >> 2)) * ld + c0 + 16 * (grp & 1) + 4 * (s & 3);
    const short4_ lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p));
    const short4_ hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p + 4 * ld));
    typedef short short8_ __attribute__((ext_vector_type(8)));
    const short8_ v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(Frag, v);
  }

  // ---- chaining products through registers ----
  // A 32x32 accumulator fragment can be the B operand of the next product without a trip through LDS when the
  // contraction runs over the fragment's rows: lane (n = lane & 31, kg = lane >> 5) holds, as elements 8 h .. 8 h + 7
  // of the fragment (h = 0, 1), the rows  16 h + 4 kg + (0..3)  and  16 h + 8 + 4 kg + (0..3)  of column n.  The MFMA
  // only needs both operands to agree on which contraction index sits in which slot, so the A operand is loaded in
  // that same order ("chain order") with two 8-byte reads instead of one 16-byte read.
  static __device__ __forceinline__ Frag from_acc(const floatx16& c, int h) {
    typedef unsigned uint4_ __attribute__((ext_vector_type(4)));
    typedef unsigned uint2_ __attribute__((ext_vector_type(2)));
    const uint2_ lo = __builtin_bit_cast(uint2_, pack_bf16x4(floatx4{c[8 * h], c[8 * h + 1], c[8 * h + 2], c[8 * h + 3]}));
    const uint2_ hi = __builtin_bit_cast(uint2_, pack_bf16x4(floatx4{c[8 * h + 4], c[8 * h + 5], c[8 * h + 6], c[8 * h + 7]}));
    return __builtin_bit_cast(Frag, (uint4_{lo[0], lo[1], hi[0], hi[1]}));
  }
  // A operand in chain order from a [rows][k] tile: p points at (this lane's row, first k of the 16-wide step)
  static __device__ __forceinline__ Frag load_chain(const bf16_t* p, int lane) {
    const bf16_t* q = p + 4 * (lane >> 5);
    const bf16x4 lo = *reinterpret_cast<const bf16x4*>(q), hi = *reinterpret_cast<const bf16x4*>(q + 8);
    Frag v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return v;
  }
  // A operand in chain order from a row-major [k][rows] tile (contraction along the tile's rows), like load_t
  static __device__ __forceinline__ Frag load_t_chain(const bf16_t* tile, int ld, int k0, int c0, int lane) {
    typedef short short4_ __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) short4_ lds_short4;
    const int s = lane & 15, grp = lane >> 4;
    const bf16_t* p = tile + (k0 + 4 * (grp >> 1) + (s >> 2)) * ld + c0 + 16 * (grp & 1) + 4 * (s & 3);
    const short4_ lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p));
    const short4_ hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p + 8 * ld));
    typedef short short8_ __attribute__((ext_vector_type(8)));
    const short8_ v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(Frag, v);
  }
  // Four consecutive rows of this lane's column of a row-major tile, i.e. elements 4 q .. 4 q + 3 of an accumulator
  // fragment's position: tile[r0 + 8 q + 4 (lane >> 5) + (0..3)][c0 + (lane & 31)], one transposing read.
  static __device__ __forceinline__ bf16x4 load_acc_rows_raw(const bf16_t* tile, int ld, int r0, int q, int c0, int lane) {
    typedef short short4_ __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) short4_ lds_short4;
    const int s = lane & 15, grp = lane >> 4;
    const bf16_t* p = tile + (r0 + 8 * q + 4 * (grp >> 1) + (s >> 2)) * ld + c0 + 16 * (grp & 1) + 4 * (s & 3);
    return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p)));
  }
  static __device__ __forceinline__ floatx4 load_acc_rows(const bf16_t* tile, int ld, int r0, int q, int c0, int lane) {
    typedef short short4_ __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) short4_ lds_short4;
    const int s = lane & 15, grp = lane >> 4;
    const bf16_t* p = tile + (r0 + 8 * q + 4 * (grp >> 1) + (s >> 2)) * ld + c0 + 16 * (grp & 1) + 4 * (s & 3);
    const short4_ x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p));
    const bf16x4 y = __builtin_bit_cast(bf16x4, x);
    floatx4 r = {(float)y[0], (float)y[1], (float)y[2], (float)y[3]};
    return r;
  }
};

// 16 x 16 x 32 products of bf16 operands, for waves that own 16 columns.  Lane: l16 = lane & 15, g = lane >> 4.  The product adds
// its eight contraction slots of group 0 first, then those of groups 1, 2, 3 -- the order in which two 32 x 32 x 16 products
// add theirs -- so with group g holding what (step g >> 1, half g & 1) holds there, both give the same bits, and 16- and
// 32-column strips can be exchanged freely.  In the order that chained products use ("chain order") group g holds the indices
// grp(g) + 0 .. 3 and grp(g) + 8 .. 11 of a step of 32, grp(g) = 16 (g >> 1) + 4 (g & 1); in natural order 8 g .. 8 g + 7.
// Accumulators that become operands: tile i of a column of tiles covers the rows  row0(i) + grp(g) + r  (element r of group
// g), row0(i) = 32 (i >> 1) + 8 (i & 1), so tiles 2 s and 2 s + 1 in registers are the operand of step s in chain order.
struct Mma16 {
  typedef bf16x8 Frag;
  typedef short short4_ __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) short4_ lds_short4;
  static __device__ __forceinline__ void mma(floatx4& c, const Frag& a, const Frag& b) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ Frag join(bf16x4 lo, bf16x4 hi) {
    typedef unsigned uint4_ __attribute__((ext_vector_type(4)));
    typedef unsigned uint2_ __attribute__((ext_vector_type(2)));
    const uint2_ a = __builtin_bit_cast(uint2_, lo), b = __builtin_bit_cast(uint2_, hi);
    return __builtin_bit_cast(Frag, (uint4_{a[0], a[1], b[0], b[1]}));
  }
  static __device__ __forceinline__ int row0(int i) { return 32 * (i >> 1) + 8 * (i & 1); }
  static __device__ __forceinline__ int grp(int lane) { return 16 * ((lane >> 5) & 1) + 4 * ((lane >> 4) & 1); }
  static __device__ __forceinline__ int row(int lane) { return 16 * ((lane >> 3) & 1) + (lane & 7); }  // of operand row l16 in such a tile
  static __device__ __forceinline__ Frag from_acc(floatx4 lo, floatx4 hi) { return join(pack_bf16x4(lo), pack_bf16x4(hi)); }
  // Tiles whose rows are operands ([rows][k], k along the row) lie in LDS in one of two column orders.  Plain: an operand is
  // two 8-byte reads.  CHAIN: inside each block of 32 columns, position 8 g + j holds column grp(g) + j (j < 4) or
  // grp(g) + 4 + j, so an operand is one ds_read_b128 per step, and an aligned vector of eight columns is written in two
  // halves.  Measured per KB of the CU's LDS: ds_read_b128 3.9 cycles where rows are 32 bytes off a multiple of 64 (288, 160)
  // and 6.6 at 272 or 144; two ds_read_b64 5.4; the ds_read2_b64 that hipcc makes of them 12 - 16 (hence the volatile reads);
  // writes 7.5 - 13 in one piece, 9 - 16 in two.  A wave can have 15 reads in flight, so a wave whose chain waits for its reads
  // wants CHAIN; where the movers' writes are what a chunk waits for, plain is the better one.
  template <bool CHAIN> static __device__ __forceinline__ int pos(int c) {  // of the vector at column c, c % 8 == 0
    return CHAIN ? (c & ~31) + ((c >> 4) & 1) * 16 + ((c >> 3) & 1) * 4 : c;
  }
  template <bool CHAIN> static __device__ __forceinline__ void put(bf16_t* p, bf16x8 v) {  // p: the row at pos(c)
    if (CHAIN) {
      *reinterpret_cast<bf16x4*>(p) = bf16x4{v[0], v[1], v[2], v[3]};
      *reinterpret_cast<bf16x4*>(p + 8) = bf16x4{v[4], v[5], v[6], v[7]};
    } else {
      *reinterpret_cast<bf16x8*>(p) = v;
    }
  }
  // operand rows in chain order: p points at (this lane's row, first column of the step)
  template <bool CHAIN> static __device__ __forceinline__ Frag load(const bf16_t* p, int lane) {
    if (CHAIN) return *reinterpret_cast<const bf16x8*>(p + 8 * (lane >> 4));
    typedef float float2_ __attribute__((ext_vector_type(2)));
    typedef const volatile __attribute__((address_space(3))) float2_ lds_float2;
    lds_float2* q = (lds_float2*)(p + grp(lane));
    const float2_ lo = q[0], hi = q[2];
    return join(__builtin_bit_cast(bf16x4, lo), __builtin_bit_cast(bf16x4, hi));
  }
  // operand from the columns of tile ci of such a tile (contraction along the tile's rows from k0)
  template <bool CHAIN, bool NATURAL = false> static __device__ __forceinline__ Frag load_cols(const bf16_t* tile, int ld, int k0, int ci, int lane) {
    const int s = lane & 15;
    const bf16_t* p = tile + (k0 + (NATURAL ? 8 * (lane >> 4) : grp(lane)) + (s >> 2)) * ld + 32 * (ci >> 1) +
                      (CHAIN ? 4 * (ci & 1) + 8 * (s & 3) : 8 * (ci & 1) + 16 * ((s >> 1) & 1) + 4 * (s & 1));
    return join(__builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p))),
                __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p + (NATURAL ? 4 : 8) * ld))));
  }
  // four consecutive rows from r0 of column c0 + l16 of a row-major tile (r0 may differ between groups of 16 lanes): one transposing read
  static __device__ __forceinline__ bf16x4 rows4(const bf16_t* tile, int ld, int r0, int c0, int lane) {
    const int s = lane & 15;
    const bf16_t* p = tile + (r0 + (s >> 2)) * ld + c0 + 4 * (s & 3);
    return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p)));
  }
  // operand in natural order from a plain row-major [k][columns] tile, columns c0 + l16
  static __device__ __forceinline__ Frag load_t(const bf16_t* tile, int ld, int k0, int c0, int lane) {
    return join(rows4(tile, ld, k0 + 8 * (lane >> 4), c0, lane), rows4(tile, ld, k0 + 8 * (lane >> 4) + 4, c0, lane));
  }
};

template <> struct Mma<float> {
  static constexpr int KS = 8;
  static constexpr int VEC = 4;
  static constexpr int PAD = 4;
  typedef floatx4 Frag;
  typedef floatx4 Quad;
  static __device__ __forceinline__ Frag load(const float* p) { return *reinterpret_cast<const floatx4*>(p); }
  static __device__ __forceinline__ void mma(floatx16& c, const Frag& a, const Frag& b) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
  }
  // fp32: one element per MFMA, so the transposed-source fragment is four conflict-free scalar reads
  static __device__ __forceinline__ Frag load_t(const float* tile, int ld, int k0, int c0, int lane) {
    const float* p = tile + (k0 + 4 * (lane >> 5)) * ld + c0 + (lane & 31);
    Frag v = {p[0], p[ld], p[2 * ld], p[3 * ld]};
    return v;
  }
};

template <int MT, int NT>
__device__ __forceinline__ void frag_zero(floatx16 (&acc)[MT][NT]) {
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
}

// acc[i][j] += A[32 i .. , :K] * B[32 j .. , :K]^T ; A, B point at this wave's first rows.
template <typename T, int MT, int NT>
__device__ __forceinline__ void mma_nt(floatx16 (&acc)[MT][NT], const T* A, int lda, const T* B, int ldb, int K,
                                       int lane) {
  typedef Mma<T> M;
  const int r = lane & 31, ko = (lane >> 5) * M::VEC;
  const T* ap = A + r * lda + ko;
  const T* bp = B + r * ldb + ko;
  for (int k0 = 0; k0 < K; k0 += M::KS) {
    typename M::Frag a[MT], b[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) a[i] = M::load(ap + i * 32 * lda + k0);
#pragma unroll
    for (int j = 0; j < NT; ++j) b[j] = M::load(bp + j * 32 * ldb + k0);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) M::mma(acc[i][j], a[i], b[j]);
  }
}

// General form: TA / TB say that the operand is given as a row-major [K][rows] tile (contraction
// index along the tile's rows; A / B then point at the tile's first used column) instead of the
// native [rows][K] layout.
template <typename T, int MT, int NT, bool TA, bool TB>
__device__ __forceinline__ void mma_x(floatx16 (&acc)[MT][NT], const T* A, int lda, const T* B, int ldb, int K,
                                      int lane) {
  typedef Mma<T> M;
  const int r = lane & 31, ko = (lane >> 5) * M::VEC;
  for (int k0 = 0; k0 < K; k0 += M::KS) {
    typename M::Frag a[MT], b[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
      a[i] = TA ? M::load_t(A, lda, k0, 32 * i, lane) : M::load(A + (r + 32 * i) * lda + ko + k0);
#pragma unroll
    for (int j = 0; j < NT; ++j)
      b[j] = TB ? M::load_t(B, ldb, k0, 32 * j, lane) : M::load(B + (r + 32 * j) * ldb + ko + k0);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) M::mma(acc[i][j], a[i], b[j]);
  }
}

// ---------------------------------------------------------------------------------------
// Loads that go straight to LDS (global_load_lds_dwordx4): one wave instruction fetches 16 bytes per lane from per-lane
// global addresses and writes them to 1 KB of consecutive LDS, lane l at `dst` + 16 l; no registers hold the data, so
// whole slabs can be in flight behind the one being multiplied.  The LDS layout of a tile is therefore unpadded; which
// 16-byte granule a lane fetches is free, so the granules of a row are permuted by an XOR of the row index instead
// (SwzTile) -- rows that an access pattern reads together land in different banks.  The compiler does not know that
// these instructions write LDS or count towards vmcnt: the callers wait with dma_wait<N>() (all but the N youngest of
// this wave's memory instructions have completed; the counter retires in order) and a workgroup barrier before reading.
// ---------------------------------------------------------------------------------------
typedef __attribute__((address_space(3))) char lds_char_t;
__device__ __forceinline__ unsigned lds_byte_addr(const void* p) { return (unsigned)(uintptr_t)(lds_char_t*)p; }
__device__ __forceinline__ void dma16(const void* src, unsigned dst) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(__builtin_amdgcn_readfirstlane(dst)) : "memory", "m0");
}
// The same with four bytes per lane: 256 consecutive bytes of LDS
__device__ __forceinline__ void dma4(const void* src, unsigned dst) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(__builtin_amdgcn_readfirstlane(dst)) : "memory", "m0");
}
template <int N> __device__ __forceinline__ void dma_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// A [ROWS][COLS] bf16 tile in LDS without padding, COLS * 2 bytes per row, granule g (16 bytes) of row r at granule
// position g ^ x(r).  x is chosen so that both ways of reading the tile touch every bank once per access:
//   a row read (16 lanes = 16 consecutive rows, one granule each) needs 16 rows on 16 different 16-byte slots of the
//   256 bytes of bank space, a transposing read (half a wave = 4 consecutive rows r0 % 4 == 0 times 4 aligned granules)
//   needs the 4 rows on different 64-byte quarters:
//   256-byte rows: x = 4 (r % 4) + r / 4 % 4;  128-byte rows: x = 4 (r / 2 % 2) + r / 4 % 4;  64-byte rows: x = r / 4 % 4.
// Tiles of 256- or 128-byte rows that are only read through transposing reads (ROW_READS = false) drop the second
// term: fewer address instructions.
template <int ROWS, int COLS, bool ROW_READS = true> struct SwzTile {
  typedef bf16_t T;
  typedef Mma<bf16_t> M;
  typedef short short4_ __attribute__((ext_vector_type(4)));
  typedef short short8_ __attribute__((ext_vector_type(8)));
  typedef __attribute__((address_space(3))) short4_ lds_short4;
  static constexpr int G = COLS / 8, BYTES = ROWS * COLS * 2, NINSTR = BYTES / 1024;
  static_assert(G == 16 || G == 8 || G == 4, "rows of 256, 128 or 64 bytes");
  static __device__ __forceinline__ int x(int r) {
    const int lo = ROW_READS || G == 4 ? (r >> 2) & 3 : 0;
    return G == 16 ? ((r & 3) << 2) | lo : G == 8 ? (((r >> 1) & 1) << 2) | lo : lo;
  }
  // element offset of (row r, column c)
  static __device__ __forceinline__ int at(int r, int c) { return r * COLS + ((((c >> 3) ^ x(r)) << 3) | (c & 7)); }
  // instruction j of the tile's load: the row and the column of the granule this lane fetches
  static __device__ __forceinline__ void src(int j, int lane, int& r, int& c) {
    const int p = 64 * j + lane;
    r = p / G;
    c = ((p % G) ^ x(r)) << 3;
  }
  // the four consecutive rows r0 .. r0 + 3 (r0 % 4 == 0) of column c0 + (this lane's column): one transposing read
  static __device__ __forceinline__ short4_ tr4(const T* tile, int r0, int c0, int lane) {
    const int s = lane & 15;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(tile + at(r0 + (s >> 2), c0 + 4 * (s & 3))));
  }
  // Mma::load_t on the swizzled tile: contraction index along the tile's rows k0 .. k0 + 15, columns c0 .. c0 + 31
  static __device__ __forceinline__ typename M::Frag load_t(const T* tile, int k0, int c0, int lane) {
    const int grp = lane >> 4;
    const short4_ lo = tr4(tile, k0 + 8 * (grp >> 1), c0 + 16 * (grp & 1), lane);
    const short4_ hi = tr4(tile, k0 + 8 * (grp >> 1) + 4, c0 + 16 * (grp & 1), lane);
    const short8_ v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(typename M::Frag, v);
  }
  // Mma::load on the swizzled tile: eight consecutive elements of row r from column c (c % 8 == 0)
  static __device__ __forceinline__ typename M::Frag load(const T* tile, int r, int c) {
    return *reinterpret_cast<const typename M::Frag*>(tile + at(r, c));
  }
};

__device__ __forceinline__ int frag_row(int e, int lane) { return 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3); }
__device__ __forceinline__ int frag_col(int lane) { return lane & 31; }

// dst[row][col] = acc (row-major tile with leading dimension ld); dst points at the tile origin.
template <typename T, int MT, int NT>
__device__ __forceinline__ void frag_store(const floatx16 (&acc)[MT][NT], T* dst, int64_t ld, int lane,
                                           int row_limit = 1 << 30) {
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = 32 * i + frag_row(e, lane);
        if (row < row_limit) dst[row * ld + 32 * j + frag_col(lane)] = from_f32<T>(acc[i][j][e]);
      }
}

// dst[col][row] = acc: transposed store, four consecutive rows per vector.
template <typename T, int MT, int NT>
__device__ __forceinline__ void frag_store_t(const floatx16 (&acc)[MT][NT], T* dst, int64_t ld, int lane) {
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = 32 * i + 8 * q + 4 * (lane >> 5);
        const int col = 32 * j + frag_col(lane);
        floatx4 x = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        store4(dst + col * ld + row, x);
      }
}

// ---------------------------------------------------------------------------------------
// global <-> LDS staging of [rows x cols] tiles by a 256-thread block
// ---------------------------------------------------------------------------------------

template <typename T> struct Vec16 {
  static constexpr int N = 16 / sizeof(T);
  typedef typename Mma<T>::Frag V;
};

template <typename T>
__device__ __forceinline__ typename Vec16<T>::V vec_zero() {
  typename Vec16<T>::V z;
#pragma unroll
  for (int e = 0; e < Vec16<T>::N; ++e) z[e] = (T)0.f;
  return z;
}

// A [ROWS x COLS] tile held in registers between its global loads and its LDS stores, so that a
// kernel can issue the loads of all tiles of a phase before it waits for any of them.
// Rows >= valid read as zero (valid <= 0: the whole tile).  COLS % VEC == 0.
// The loads are buffer loads through a descriptor that covers exactly the valid rows: the hardware's range check
// returns zeros past the end, the per-thread offsets do not depend on the chunk (no address arithmetic in vector
// registers per load), and no load sits behind a branch or a select -- either would keep the compiler from
// counting the loads in flight exactly, and it would then make the next tile store wait for (nearly) all of
// them, younger prefetches included.
template <typename T, int ROWS, int COLS, int THREADS = 256> struct TileRegs {
  static constexpr int N = Vec16<T>::N, VPR = COLS / N, TOTAL = ROWS * VPR, IT = (TOTAL + THREADS - 1) / THREADS;
  typename Vec16<T>::V x[IT];
  __device__ __forceinline__ void load(const T* src, int64_t stride, int valid, int tid) {
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    const int bytes = valid > 0 ? (int)(valid * stride * (int64_t)sizeof(T)) : 0;
    // raw buffer (no stride, no swizzle) of `bytes` bytes; 0x00020000: 32-bit data format, as untyped loads need
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(src), 0, bytes, 0x00020000);
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int idx = tid + THREADS * it, r = idx / VPR, c = (idx - r * VPR) * N;
      const u32x4 raw = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)((r * stride + c) * (int64_t)sizeof(T)), 0, 0);
      x[it] = __builtin_bit_cast(typename Vec16<T>::V, raw);
    }
  }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int it = 0; it < IT; ++it) x[it] = vec_zero<T>();
  }
  __device__ __forceinline__ typename Vec16<T>::V get(int it, int) const { return x[it]; }
  __device__ __forceinline__ void store(T* dst, int ld, int tid) const {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int idx = tid + THREADS * it, r = idx / VPR, c = (idx - r * VPR) * N;
      if (idx < TOTAL) *reinterpret_cast<typename Vec16<T>::V*>(dst + r * ld + c) = x[it];
    }
  }
};

// A lower-triangular [64 x 64] 2-byte tile travels packed: of its 512 eight-element vectors (row r, columns 8 c .. 8 c + 7)
// only the 288 with 8 c <= r can hold a non-zero.  Rows come in groups of eight; group g has g + 1 vectors per row and starts
// at packed index 4 g (g + 1); a slot of the workspace keeps its 64 x 64 elements and uses the first 288 x 16 bytes.
constexpr int LNX_TRI_VECS = 288;
__device__ __forceinline__ void tri_vec_pos(int idx, int& r, int& c) {  // idx < LNX_TRI_VECS
  int g = 0;
#pragma unroll
  for (int h = 1; h < 8; ++h) g += (4 * h * (h + 1) <= idx) ? 1 : 0;
  const int o = idx - 4 * g * (g + 1);  // < 64
  // o / (g + 1) without an integer division: (o + 0.5) / (g + 1) is at least 1/16 away from every integer
  const int q = (int)(((float)o + 0.5f) * __builtin_amdgcn_rcpf((float)(g + 1)));
  r = 8 * g + q;
  c = o - q * (g + 1);
}
// The vectors above the diagonal (8 c > r) in turn, idx < 512 - LNX_TRI_VECS: group g of eight rows has 7 - g of them per row.
__device__ __forceinline__ void upper_vec_pos(int idx, int& r, int& c) {
  int g = 0;
  while (56 * (g + 1) - 4 * (g + 1) * g <= idx) ++g;  // vectors of the groups before g + 1
  const int o = idx - (56 * g - 4 * g * (g - 1)), per = 7 - g;
  r = 8 * g + o / per;
  c = g + 1 + (o - (o / per) * per);
}
// The packed tile in the registers of 256 or 512 threads (vector tid, with 256 also vector 256 + tid for tid < 32) between its global
// loads and its LDS stores (columns in the order CHAIN of Mma16), like TileRegs; the LDS tile's upper part is zeroed once by the caller and never written.
template <typename T, bool CHAIN, int THREADS = 256> struct TriRegs {
  static_assert(sizeof(T) == 2, "packed triangles are a 2-byte format");
  static constexpr bool TWO = THREADS < LNX_TRI_VECS;
  typename Vec16<T>::V x[2];
  int o0, o1;  // LDS element offsets of this thread's two vectors for a leading dimension fixed at init
  bool first, second;
  __device__ __forceinline__ void init(int ld, int tid) {
    int r, c;
    first = TWO || tid < LNX_TRI_VECS;
    tri_vec_pos(first ? tid : LNX_TRI_VECS - 1, r, c);
    o0 = r * ld + Mma16::pos<CHAIN>(8 * c);
    second = TWO && tid < LNX_TRI_VECS - 256;
    if (!TWO) return;
    tri_vec_pos(second ? 256 + tid : LNX_TRI_VECS - 1, r, c);
    o1 = r * ld + Mma16::pos<CHAIN>(8 * c);
  }
  __device__ __forceinline__ void load(const T* src, int tid) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(src), 0, LNX_TRI_VECS * 16, 0x00020000);
    // threads without a (second) vector read past the end: the range check returns zeros, nothing sits behind a branch
    x[0] = __builtin_bit_cast(typename Vec16<T>::V, __builtin_amdgcn_raw_buffer_load_b128(rsrc, 16 * tid, 0, 0));
    if (TWO) x[1] = __builtin_bit_cast(typename Vec16<T>::V, __builtin_amdgcn_raw_buffer_load_b128(rsrc, 16 * (256 + tid), 0, 0));
  }
  __device__ __forceinline__ void store(T* dst) const {
    if (first) Mma16::put<CHAIN>(dst + o0, x[0]);
    if (TWO && second) Mma16::put<CHAIN>(dst + o1, x[1]);
  }
};

// One-shot form (load, then store) for a single tile.
template <typename T, int ROWS, int COLS>
__device__ __forceinline__ void stage_tile(T* dst, int ld, const T* src, int64_t stride, int valid, int tid) {
  TileRegs<T, ROWS, COLS> t;
  t.load(src, stride, valid, tid);
  t.store(dst, ld, tid);
}

// LDS tile [ROWS][COLS] (leading dimension ld) -> global, 16-byte vectors, rows < valid only.
// FULL: every row is written and the tile is a whole number of 256-thread passes, so the loads
// and stores are unconditional and issued as two batches.
template <typename T, int ROWS, int COLS, bool FULL = false, int THREADS = 256>
__device__ __forceinline__ void unstage_tile(T* dst, int64_t stride, const T* src, int ld, int valid, int tid) {
  typedef typename Vec16<T>::V V;
  constexpr int N = Vec16<T>::N, VPR = COLS / N, TOTAL = ROWS * VPR, IT = (TOTAL + THREADS - 1) / THREADS;
  if constexpr (FULL) {
    static_assert(TOTAL % THREADS == 0, "whole passes only");
    V x[IT];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int idx = tid + THREADS * it, r = idx / VPR, c = (idx - r * VPR) * N;
      x[it] = *reinterpret_cast<const V*>(src + r * ld + c);
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int idx = tid + THREADS * it, r = idx / VPR, c = (idx - r * VPR) * N;
      *reinterpret_cast<V*>(dst + r * stride + c) = x[it];
    }
  } else {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int idx = tid + THREADS * it, r = idx / VPR, c = (idx - r * VPR) * N;
      if (idx < TOTAL && r < valid) *reinterpret_cast<V*>(dst + r * stride + c) = *reinterpret_cast<const V*>(src + r * ld + c);
    }
  }
}

// The same through a buffer descriptor that covers rows < valid only: the hardware drops the stores past the end, so
// no store sits behind a branch and a loop that also prefetches can count its memory instructions exactly.
template <typename T, int ROWS, int COLS>
__device__ __forceinline__ void unstage_tile_checked(T* dst, int64_t stride, const T* src, int ld, int valid, int tid) {
  typedef typename Vec16<T>::V V;
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  constexpr int N = Vec16<T>::N, VPR = COLS / N, TOTAL = ROWS * VPR, IT = TOTAL / 256;
  static_assert(TOTAL % 256 == 0, "whole passes only");
  const int bytes = valid > 0 ? (int)(valid * stride * (int64_t)sizeof(T)) : 0;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(dst, 0, bytes, 0x00020000);
  V x[IT];
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int idx = tid + 256 * it, r = idx / VPR, c = (idx - r * VPR) * N;
    x[it] = *reinterpret_cast<const V*>(src + r * ld + c);
  }
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int idx = tid + 256 * it, r = idx / VPR, c = (idx - r * VPR) * N;
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x[it]), rsrc, (int)((r * stride + c) * (int64_t)sizeof(T)), 0, 0);
  }
}

// A bf16 LDS tile written out as fp32 rows (same range check): the direct-solve forward scan stages its outputs in
// bf16 -- the precision the reference returns them in for bf16 inputs -- and widens them here when the caller asked
// for fp32 outputs.
template <int ROWS, int COLS>
__device__ __forceinline__ void unstage_tile_checked_widen(float* dst, int64_t stride, const bf16_t* src, int ld, int valid, int tid) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  constexpr int VPR = COLS / 8, TOTAL = ROWS * VPR, IT = TOTAL / 256;
  static_assert(TOTAL % 256 == 0, "whole passes only");
  const int bytes = valid > 0 ? (int)(valid * stride * (int64_t)sizeof(float)) : 0;
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(dst, 0, bytes, 0x00020000);
  bf16x8 x[IT];
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int idx = tid + 256 * it, r = idx / VPR, c = (idx - r * VPR) * 8;
    x[it] = *reinterpret_cast<const bf16x8*>(src + r * ld + c);
  }
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int idx = tid + 256 * it, r = idx / VPR, c = (idx - r * VPR) * 8;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const floatx4 y = {(float)x[it][4 * h], (float)x[it][4 * h + 1], (float)x[it][4 * h + 2], (float)x[it][4 * h + 3]};
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, y), rsrc, (int)((r * stride + c + 4 * h) * (int64_t)sizeof(float)), 0, 0);
    }
  }
}

// Sums f(e) * acc[i][0][e] over the 32 lanes that share rows, for all 16*MT rows of a wave's
// fragments at once, by a transpose-reduce (31 shuffles per 32 values instead of 160), then adds
// the row totals into rows[] (LDS) with one atomic per row and wave.  Callers zero rows[] and have at most two waves
// per row, so the result does not depend on the order of arrival (0 + a + b = 0 + b + a in floating point).
template <int MT>
__device__ __forceinline__ void rows_reduce_add(float (&v)[16 * MT], int row0, int lane, float* rows) {
  // after the step with mask m, v[t] (t < n/2) holds the partial for value index t + (lane & m ? n/2 : 0)
  static_assert(MT == 1 || MT == 2, "one or two row tiles");
  constexpr int NV = 16 * MT;
  int n = NV;
  // reduce value count down to 1 using lane bits 4,3,2,1 (and 0 when NV == 32); remaining lane bits by plain xor-adds
  constexpr int STEPS = (MT == 2) ? 5 : 4;
  int masks[5] = {16, 8, 4, 2, 1};
#pragma unroll
  for (int s_ = 0; s_ < STEPS; ++s_) {
    const int m = masks[s_];
    const int half = NV >> (s_ + 1);
    const bool hi = (lane & m) != 0;
#pragma unroll
    for (int t = 0; t < half; ++t) {
      const float a = v[t], b = v[t + half];
      const float send = hi ? a : b, keep = hi ? b : a;
      v[t] = keep + __shfl_xor(send, m, LNX_WAVE);
    }
  }
  (void)n;
  float total = v[0];
  if (MT == 1) total += __shfl_xor(total, 1, LNX_WAVE);  // 16 values: lane bit 0 still unreduced
  // value index owned by this lane: bits (4,3,2,1[,0]) of the lane select the halves kept
  int idx = 0;
#pragma unroll
  for (int s_ = 0; s_ < STEPS; ++s_) idx |= ((lane & masks[s_]) ? (NV >> (s_ + 1)) : 0);
  const int i = idx >> 4, e = idx & 15;
  if (MT == 2 || (lane & 1) == 0) atomicAdd(&rows[row0 + 32 * i + frag_row(e, lane)], total);
}

// ---------------------------------------------------------------------------------------
// 16x16 fp32 products on v_mfma_f32_16x16x4_f32, operands row-major in LDS
//   returns C[i][j] = sum_k A[i][k] * B[k][j];  fragment: c[e] is row 4*(lane>>4)+e, col lane&15
// ---------------------------------------------------------------------------------------
__device__ __forceinline__ floatx4 mm16_f32(const float* A, int lda, const float* B, int ldb, int K, int lane) {
  floatx4 c = {0.f, 0.f, 0.f, 0.f};
  const int i = lane & 15, kq = lane >> 4;
  for (int k0 = 0; k0 < K; k0 += 4) {
    const float a = A[i * lda + k0 + kq];
    const float b = B[(k0 + kq) * ldb + i];
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  return c;
}

__device__ __forceinline__ void mm16_store(float* dst, int ld, floatx4 c, int lane, float sign) {
#pragma unroll
  for (int e = 0; e < 4; ++e) dst[(4 * (lane >> 4) + e) * ld + (lane & 15)] = sign * c[e];
}

#define LNX_LDA 68  // leading dimension of the fp32 64x64 matrices in LDS

// In-LDS inverse of the unit lower-triangular matrix I + A: `M` holds A (strictly lower, zeros on and above the diagonal of the 16x16 diagonal
// blocks, 64x64, fp32, leading dimension LNX_LDA) and receives Tm = (I + A)^-1.  Called by the 256 threads of a workgroup.  Wave `solver` takes
// the four diagonal blocks by forward substitution, sixteen lanes each, a lane a column of the inverse; then two levels of block merges
//   [[L0, 0], [B, L1]]^-1 = [[L0^-1, 0], [-L1^-1 B L0^-1, L1^-1]]
// on v_mfma_f32_16x16x4_f32: a product's result fragment (rows 4 g + r, column l16) is the right operand of the next as it is, with the
// contraction index of step r being 4 g + r in both (a left operand is then one 16-byte read), so a merge needs no scratch and no barrier of its
// own.
// A chunk's inverse is a serial chain that other workgroups of the CU have to cover: with every wave solving a block and the merges' products
// through LDS it took seven barriers and 730 instructions of forward substitution instead of 180 (B4 H16 T8192 d128 kda_prepare 374 -> 361 us,
// RWKV-7's chunk kernels 994 -> 975 of 2095).
__device__ __forceinline__ void tri_inverse_64(float* M, int tid, int solver = 0) {
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  if (wave == solver) {
    float* D = M + 16 * g * (LNX_LDA + 1);
    float d[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) d[i] = (i == l16) ? 1.f : 0.f;
#pragma unroll
    for (int m4 = 0; m4 < 4; ++m4) {  // by columns of A: what a solved row takes off the later ones
      floatx4 a[16];
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (i > 4 * m4) a[i] = load4(D + i * LNX_LDA + 4 * m4);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          if (i > 4 * m4 + u) d[i] -= a[i][u] * d[4 * m4 + u];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) D[i * LNX_LDA + l16] = d[i];
  }
  lds_barrier();
  auto rows = [&](int i0, int k0) { return load4(M + (i0 + l16) * LNX_LDA + k0 + 4 * g); };
  auto add = [&](floatx4& c, floatx4 a, floatx4 b) {
#pragma unroll
    for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
  };
  auto cols = [&](int k0, int j0) {
    const float* p = M + (k0 + 4 * g) * LNX_LDA + j0 + l16;
    return floatx4{p[0], p[LNX_LDA], p[2 * LNX_LDA], p[3 * LNX_LDA]};
  };
  auto put = [&](floatx4 c, int i0, int j0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) M[(i0 + 4 * g + r) * LNX_LDA + j0 + l16] = -c[r];
  };
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  if (wave < 2) {  // blocks (1, 0) and (3, 2) of the 16x16 grid
    const int b = 32 * wave;
    floatx4 x = zero, y = zero;
    add(x, rows(b + 16, b), cols(b, b));
    add(y, rows(b + 16, b + 16), x);
    put(y, b + 16, b);
  }
  lds_barrier();
  const int bi = wave >> 1, bj = wave & 1;  // block (2 + bi, bj); both triangular factors have one block of zeros
  floatx4 y = zero;
#pragma unroll
  for (int r = 0; r < 2; ++r)
    if (r <= bi) {
      floatx4 x = zero;
#pragma unroll
      for (int k = 0; k < 2; ++k)
        if (k >= bj) add(x, rows(32 + 16 * r, 16 * k), cols(16 * k, 16 * bj));
      add(y, rows(32 + 16 * bi, 32 + 16 * r), x);
    }
  lds_barrier();  // the block of A has been read
  put(y, 32 + 16 * bi, 16 * bj);
  lds_barrier();
}

// The same with the sums grouped another way: Tm of the calls without a per-channel gate.  Neither is the more exact one.  This one's bits are those
// that these calls' results have had, which shows only where a sequence grows to the end of fp32's range (keys longer than one, no gate) and the
// last bits decide which values are infinite.  They are so by measurement: -ffast-math lets the compiler regroup the substitution, and it does
// (held to the order written here, fp32 results have other last bits).  Price: chunk_prepare2 43 instead of 41 us on one prompt of 65536 tokens and
// 4 heads, none at B8 H16 T4096.  In place; A's upper triangle
// within the 32x32 diagonal blocks must hold zeros, `sX` is a [32][36] scratch that is first written behind the first barrier.  Four waves solve a
// diagonal block each (16 lanes a block), the merges' products go through the scratch.
__device__ __forceinline__ void tri_inverse_64_rows(float* M, float* sX, int tid) {
  const int wave = tid >> 6, lane = tid & 63;
  if (lane < 16) {
    const int r0 = 16 * wave, c = lane;
    float d[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float s = (i == c) ? 1.f : 0.f;
#pragma unroll
      for (int m = 0; m < i; ++m) s -= M[(r0 + i) * LNX_LDA + r0 + m] * d[m];
      d[i] = s;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) M[(r0 + i) * LNX_LDA + r0 + c] = d[i];
  }
  lds_barrier();
  // blocks (1,0) and (3,2) of the 16x16 grid, one per wave 0/1
  float* sXw = sX + (wave & 1) * 16 * 36;
  const int b = 32 * (wave & 1);
  if (wave < 2) mm16_store(sXw, 36, mm16_f32(M + (b + 16) * LNX_LDA + b, LNX_LDA, M + b * LNX_LDA + b, LNX_LDA, 16, lane), lane, 1.f);
  lds_barrier();
  if (wave < 2) mm16_store(M + (b + 16) * LNX_LDA + b, LNX_LDA, mm16_f32(M + (b + 16) * LNX_LDA + b + 16, LNX_LDA, sXw, 36, 16, lane), lane, -1.f);
  lds_barrier();
  // the 32x32 lower-left block, one 16x16 output per wave
  const int bi = 16 * (wave >> 1), bj = 16 * (wave & 1);
  mm16_store(sX + bi * 36 + bj, 36, mm16_f32(M + (32 + bi) * LNX_LDA, LNX_LDA, M + bj, LNX_LDA, 32, lane), lane, 1.f);
  lds_barrier();
  mm16_store(M + (32 + bi) * LNX_LDA + bj, LNX_LDA, mm16_f32(M + (32 + bi) * LNX_LDA + 32, LNX_LDA, sX + bj, 36, 32, lane), lane, -1.f);
  lds_barrier();
}

