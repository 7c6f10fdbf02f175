// RWKV-7's diagonal-plus-low-rank delta rule over chunks of 64 tokens, for heads of 64 x 64 (RWKV-7's own size), in fp32.
//
// The token-by-token scan (dplr.hip) is one dependent step of some 270 wave instructions per token on the one or two waves
// that a (batch, head) row has.  Over a chunk the recurrence is a linear map of the state, so everything but a 64 x 64
// product per chunk can be done for all chunks at once, on the matrix cores (v_mfma_f32_16x16x4_f32: fp32 operands and
// accumulation; with v and dO in bf16 three bf16 products that add up to the same: no operand is rounded to less).
//
// Per chunk, w = e^gk, E_ts = product of w over the tokens after s up to and with t, per channel; e_t = E from the chunk's start, r_s = E
// to its end, and t- the token before t (a token's own decay comes after its a):
//   Aab = stril(<a_t E_t-s, b_s>)  Aak = stril(<a_t E_t-s, k_s>)  Pqb, Pqk = tril(<q_t E_ts, b_s / k_s>)
//   Tm = (I - Aab)^-1     u = Tm (a e_t- h + Aak v)     o = q e_t h + Pqb u + Pqk v     h' = e_C h + (b r)^T u + (k r)^T v
// and with W = Tm (a e_t-), U0 = Tm Aak v:
//   o = X h + Y,  X = q e + Pqb W,  Y = Pqb U0 + Pqk v          h' = M h + N,  M = e_C + (b r)^T W,  N = (b r)^T U0 + (k r)^T v
// Backward: D = gradient of the state leaving the chunk, R = X^T dO; the gradient of the state entering it is M^T D + R, and
//   dU = Tm^T (Pqb^T dO + b r D)      dv = Pqk^T dO + k r D + Aak^T dU
//   dPqb = tril(dO u^T)  dPqk = tril(dO v^T)  dAab = stril(dU u^T)  dAak = stril(dU v^T), and from these the vectors' gradients;
//   dgk_t = <D, h'>_c + sum_{t' >= t} (q dq + a da - b db - k dk)_t' - (a da)_t   (how each decay depends on gk).
//
// Decays are products and never differences of rounded sums: a float sum of gates over 64 tokens is rounded to its own size, which costs
// the decays of later tokens 4e-7 of their value inside RWKV-7's range and all of it behind a large negative gate (a caller without
// cu_seqlens ends a document inside a row that way).  A block of 16 tokens is a row of 16 lanes; it has P_t, the decay from before the
// block's first token to token t, and S_s, that of the tokens after s.  A pair in two blocks has E = P_t (whole blocks between) S_s:
// factors of the path from s to t, so any decay down to 0 (gk = -inf) gives what the token kernels give.  A pair inside a block has
// E = P_t / P_s.  P and S come from sums in fixed point, which are exact; a block whose P leave 2^+-60 (RWKV-7's decays are above
// exp(-0.607), 2^-14 over a block) multiplies its decays up as floats and takes its 120 pairs one by one (a uniform branch per wave, DIRECT
// below: B8 H16 T4096 forward and backward 2.2 ms without such blocks, 6.2 ms where all are).
//
// Sums that carry the recent tokens' large terms take the far ones first, and a sum of two products is added up from two chains: what
// comes second on one chain would be rounded at the size of the whole, 64 times.  Errors against fp64, relative 2-norms, one row of 512
// tokens with RWKV-7's decays (behind a reset of any size the same), in brackets the token kernels: o 1.2e-7 (1.0), h 0.7e-7 (0.6), dq,
// dk, dv 1.2e-7 (0.9), da, db 1.8, 1.7e-7 (1.3), dgk 2.4e-7 (1.2), dh0 1.1e-7 (0.8); with gates a hundredth of that o 2.5e-7 (4.7),
// gradients 2.3 - 4.1e-7 (4.7 - 7.4): there the token kernels round the state at every token.
//
// Kernels, each a workgroup per chunk but for the two sequential passes: the launch functions name them with their times.
#include "lnx_common.h"
#include "chunk_common.h"

namespace {

constexpr int C = 64, D = 64;       // tokens of a chunk, channels of a head
constexpr int LD = LNX_LDA;         // leading dimension of the fp32 tiles in LDS: 68 floats, rows 4 banks apart
constexpr int TS = C * LD;          // floats of a tile in LDS
constexpr int TG = C * D;           // floats of a tile in the workspace
constexpr int RANGE = 60;           // products of decays of a block's first tokens lie within 2^+-RANGE, or the block is DIRECT

// A tile in the workspace is sixteen blocks of 16 x 16, block row by block row, and a block lies as a wave holds it, four elements of a row
// per lane: lane 16 g + l16 has row l16, columns 4 g ... to 4 g + 3.  Every kernel reads and writes the tiles that way, consecutive lanes
// side by side.  With rows of 64 floats an instruction took 64 bytes of 16 rows, and such a one passes the CU's address path a lane a
// cycle, 15.8 bytes instead of 61 (measured, data in L2).  B8 H16 T4096 forward and backward 1937 -> 1870 us (the scans 110 -> 89 and 101 -> 89,
// dplr_out 112 -> 97), B1 H16 T16384 1228 -> 1143 (179 -> 135, 158 -> 142).
__device__ __forceinline__ int block_at(int row, int col) { return (4 * row + col) * 256 + 4 * (threadIdx.x & 63); }

struct ChunkParams {
  const void *q, *k, *v, *a, *b;
  const float* gk;
  const void* d_o;
  void* o;
  void *dq, *dk, *dv, *da, *db;
  float* dgk;
  float *M, *X, *hT;         // kept for the backward pass: [rows][KN] tiles, hT [rows][KN + 1] (states transposed: [dv][dk])
  float *s1, *s2, *s3, *s4;  // of a window of chunks, [rows][nw] tiles.  forward: N^T, Y; backward: D^T, R^T, u, dU
  int T, N, n0, nw;          // tokens, chunks of a row, the window [n0, n0 + nw)
  int KN, k0;                // the kept tensors hold chunks [k0, k0 + KN) of every row: all, or without a backward pass the window
  float scale;
};

struct Slot {
  int64_t row;
  int n, len;         // chunk and its tokens
  int64_t tok, kept, win, st;  // first token; tile index in the kept tensors, in the window's and in hT
};
__device__ __forceinline__ Slot slot_of(const ChunkParams& p) {
  Slot s;
  s.row = blockIdx.x / p.nw;
  s.n = p.n0 + (int)(blockIdx.x - s.row * p.nw);
  s.len = min(C, p.T - s.n * C);
  s.tok = s.row * p.T + (int64_t)s.n * C;
  s.kept = s.row * p.KN + s.n - p.k0;
  s.win = blockIdx.x;
  s.st = s.row * (p.KN + 1) + s.n - p.k0;
  return s;
}

// e^x with the rounding of x log2(e) carried along, 0 for -inf and whatever underflows.  The correction is that of a clamped x: of x
// near the lowest float or -inf its own would be inf - inf.
__device__ __forceinline__ float exp_f(float x) {
  float t = x * 1.44269504f;
  const float y = fmaxf(x, -128.f);
  float ty = y * 1.44269504f;
  asm volatile("" : "+v"(t), "+v"(ty));  // -ffast-math must not see that the next line is a rounding error
  const float e = __builtin_fmaf(y, 1.44269504f, -ty) + y * 1.92596299e-8f;
  return __builtin_amdgcn_exp2f(t) * (1.f + 0.69314718f * e);
}
__device__ __forceinline__ float rcp_f(float x) {  // one Newton step on the instruction's estimate
  const float r = __builtin_amdgcn_rcpf(x);
  return __builtin_fmaf(__builtin_fmaf(-x, r, 1.f), r, r);
}
__device__ __forceinline__ floatx4 rcp4(floatx4 x) { return floatx4{rcp_f(x[0]), rcp_f(x[1]), rcp_f(x[2]), rcp_f(x[3])}; }

// ---- products of 16 x 16 tiles ------------------------------------------------------------------------------------
// Result fragment: r-th element = row i0 + 4 g + r, column j0 + l16 (g = lane / 16, l16 = lane % 16).  The contraction
// index of step r inside a block of 16 is 4 g + r in both operands, so an operand stored with the contraction along its
// rows (ROW) is read as one 16-byte vector per block, the other way round as four single reads of 16 consecutive columns;
// with rows 68 floats apart both touch every bank once.  A result fragment is itself an operand whose contraction index is the
// result's row -- with the result's column as its row or its column --, and so are four consecutive elements of a row per lane.
template <bool ROW> __device__ __forceinline__ floatx4 frag(const float* t, int i, int k) {
  if (ROW) return load4(t + i * LD + k);
  return floatx4{t[k * LD + i], t[(k + 1) * LD + i], t[(k + 2) * LD + i], t[(k + 3) * LD + i]};
}
__device__ __forceinline__ void mfma4(floatx4& c, floatx4 a, floatx4 b) {
#pragma unroll
  for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
}
__device__ __forceinline__ floatx4 zero4() { return floatx4{0.f, 0.f, 0.f, 0.f}; }
// c[i] += a_i b_i over a block of 16 of the contraction, N sums in turn so that no product waits for the one before it
template <int N, typename F, typename G> __device__ __forceinline__ void mfma4_each(floatx4* const (&c)[N], F&& a, G&& b) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int i = 0; i < N; ++i) *c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a(i)[r], b(i)[r], *c[i], 0, 0, 0);
}
// ... the block summed from zero: for the pairs' sums over channels, where one chain of 64 additions rounds the outputs by 1.5e-7 at RWKV-7's
// decays and four chains of 16 by 1.1e-7 (all else exact).  In dplr_grad it took 750 -> 771 us, for dq 1.62 -> 1.15e-7,
// dk 1.65 -> 1.19, da 2.2 -> 1.8, db 2.1 -> 1.7, dgk 2.7 -> 2.4.
template <int N, typename F, typename G> __device__ __forceinline__ void mfma_block(floatx4* const (&c)[N], F&& a, G&& b) {
  floatx4 t[N];
  floatx4* pt[N];
#pragma unroll
  for (int i = 0; i < N; ++i) t[i] = zero4(), pt[i] = &t[i];
  mfma4_each<N>(pt, a, b);
#pragma unroll
  for (int i = 0; i < N; ++i) *c[i] += t[i];
}

// Four waves, each with a block of 16 tokens (of rows of the state tiles); the lane's token is t, its channels in block cb
// are 16 cb + 4 g + 0..3.  Sums over earlier tokens make blocks 0 .. j work, sums over later ones j .. 3: the workgroups that
// share a CU (256 apart at the start) take the blocks in opposite order.
struct Lane {
  int j, l16, g, t;
  __device__ __forceinline__ Lane() {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    j = (blockIdx.x >> 8) & 1 ? 3 - wave : wave;
    l16 = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    t = 16 * j + l16;
  }
};

// Blocks 0 .. j, 3 .. j, and those without j, as constants: the accumulators stay where they are when a wave leaves early (a branch
// around each block's products made the compiler copy them, 1000 moves among 850 products)
template <int B> struct Int {
  static constexpr int value = B;
};
template <typename F> __device__ __forceinline__ void upto(int j, F&& f) {
  f(Int<0>{});
  if (j == 0) return;
  f(Int<1>{});
  if (j == 1) return;
  f(Int<2>{});
  if (j == 2) return;
  f(Int<3>{});
}
template <typename F> __device__ __forceinline__ void downto(int j, F&& f) {
  f(Int<3>{});
  if (j == 3) return;
  f(Int<2>{});
  if (j == 2) return;
  f(Int<1>{});
  if (j == 1) return;
  f(Int<0>{});
}
template <typename F> __device__ __forceinline__ void before(int j, F&& f) {
  if (j == 0) return;
  f(Int<0>{});
  if (j == 1) return;
  f(Int<1>{});
  if (j == 2) return;
  f(Int<2>{});
}
template <typename F> __device__ __forceinline__ void after(int j, F&& f) {
  if (j == 3) return;
  f(Int<3>{});
  if (j == 2) return;
  f(Int<2>{});
  if (j == 1) return;
  f(Int<1>{});
}

// Four consecutive elements as loaded
template <typename T> struct Raw4;
template <> struct Raw4<bf16_t> {
  bf16x4 x;
  __device__ __forceinline__ void load(const bf16_t* p) { x = *reinterpret_cast<const bf16x4*>(p); }
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int o) { x = __builtin_bit_cast(bf16x4, __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0)); }
  __device__ __forceinline__ floatx4 get() const { return floatx4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]}; }
};
template <> struct Raw4<float> {
  floatx4 x;
  __device__ __forceinline__ void load(const float* p) { x = load4(p); }
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, int o) { x = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0)); }
  __device__ __forceinline__ floatx4 get() const { return x; }
};
// This lane's share of a row of 64: of a tile, or of the token's row of a caller's tensor, zeros past the chunk's end.  Those go through a buffer
// descriptor that ends there: as a choice at every use of a row the zeros were one VALU instruction in ten of dplr_grad and cost it its spilled
// registers (B8 H16 T4096 forward and backward 2138 -> 2094 us).
template <typename T> struct Row {
  Raw4<T> x[4];
  __device__ __forceinline__ void load_tile(const float* tile, int row) {  // block row of a tile in the workspace
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) x[cb].load(tile + block_at(row, cb));
  }
  __device__ __forceinline__ void load(const void* base, int64_t at) {  // at: element of the lane's first channel
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) x[cb].load(static_cast<const T*>(base) + at + 16 * cb);
  }
  __device__ __forceinline__ void load(const void* base, const Slot& s, const Lane& w) {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(static_cast<const T*>(base) + s.tok * D), 0, s.len * D * (int)sizeof(T), 0x00020000);
    const int o = (w.t * D + 4 * w.g) * (int)sizeof(T);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) x[cb].load(rsrc, o + 16 * cb * (int)sizeof(T));
  }
  __device__ __forceinline__ floatx4 operator[](int cb) const { return x[cb].get(); }
};
// What was read, not what it was converted to, is what a kernel short of registers keeps from here on
template <typename T> __device__ __forceinline__ void keep_as_read(Row<T>& r) {
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) asm volatile("" : "+v"(r.x[cb].x));
}
// ... into its row of a tile
template <typename F> __device__ __forceinline__ void put_row(float* tile, const Lane& w, F&& value) {
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) store4(tile + w.t * LD + 16 * cb + 4 * w.g, value(cb));
}

// ---- products with a tensor as the caller gave it ------------------------------------------------------------------
// v and dO in bf16 are exact in one part, and an fp32 operand is the sum of three (its top eight bits, the next eight, the last eight: all
// differences are exact), so a block of 16 of the contraction is two bf16 products of 16 cycles, {last, next} {x, x} and {top, 0} {x, x},
// instead of four fp32 ones of 32, and no operand is rounded.  The small parts come first, so that c meets the large sum once (the other way round
// h's error 0.76e-7 of its 2-norm instead of 0.53; four fp32 products 0.69).  B8 H16 T4096: dplr_prepare 486 -> 437, dplr_u 486 -> 443 us, and with dPqk in dplr_grad 733 -> 724.  Where neither operand is given, six products of parts cost what they save: an operand takes 22
// instructions to split, dplr_grad's pairs so 733 us, dAak alone 750.
// An operand below 2^-110 loses those of its bits that lie under the smallest bf16 number, 2^-133.
//
// Whatever an infinite operand reaches is NaN by parts: inf - inf where it is the one split, inf times the empty half of `top` where it is the
// given one.  A workgroup that finds a NaN among its sums begins again with FULL products, fp32 ones, which leave infinite what the fp32
// kernels do (B8 H16 T4096 forward and backward 1895 -> 1905 us, of that dplr_prepare 434 -> 443).
template <typename T, bool FULL> struct Parts {
  floatx4 x;
  __device__ __forceinline__ explicit Parts(floatx4 y) : x(y) {}
};
template <> struct Parts<bf16_t, false> {
  typedef unsigned uint4_ __attribute__((ext_vector_type(4)));
  uint4_ top, rest;
  __device__ __forceinline__ explicit Parts(floatx4 x) {
    const floatx4 y = x - high(x), z = y - high(y);
    top = uint4_{pack(x[0], x[1]), pack(x[2], x[3]), 0, 0};
    rest = uint4_{pack(z[0], z[1]), pack(z[2], z[3]), pack(y[0], y[1]), pack(y[2], y[3])};
  }
  static __device__ __forceinline__ floatx4 high(floatx4 x) { return __builtin_bit_cast(floatx4, __builtin_bit_cast(uint4_, x) & 0xffff0000u); }
  static __device__ __forceinline__ unsigned pack(float a, float b) { return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302); }
};
template <typename T> __device__ __forceinline__ void mfma_parts(floatx4& c, const Parts<T, true>& a, const Raw4<T>& b) { mfma4(c, a.x, b.get()); }
template <typename T> __device__ __forceinline__ void mfma_parts(floatx4& c, const Raw4<T>& a, const Parts<T, true>& b) { mfma4(c, a.get(), b.x); }
__device__ __forceinline__ void mfma_parts(floatx4& c, const Parts<bf16_t, false>& a, const Raw4<bf16_t>& b) {
  const bf16x8 x = Mma16::join(b.x, b.x);
  Mma16::mma(c, __builtin_bit_cast(bf16x8, a.rest), x);
  Mma16::mma(c, __builtin_bit_cast(bf16x8, a.top), x);
}
__device__ __forceinline__ void mfma_parts(floatx4& c, const Raw4<bf16_t>& a, const Parts<bf16_t, false>& b) {
  const bf16x8 x = Mma16::join(a.x, a.x);
  Mma16::mma(c, x, __builtin_bit_cast(bf16x8, b.rest));
  Mma16::mma(c, x, __builtin_bit_cast(bf16x8, b.top));
}
// NaN in any lane's sums
template <typename... S> __device__ __forceinline__ bool any_nan(const S&... sums) {
  bool x = false;
  auto look = [&](const floatx4(&c)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) x |= __builtin_isunordered(c[i][0], c[i][1]) | __builtin_isunordered(c[i][2], c[i][3]);
  };
  (look(sums), ...);
  return __ballot(x) != 0;
}
// ... of the workgroup's waves: four words of LDS between the two, and a barrier
__device__ __forceinline__ void put_flag(float* flags, bool x) { flags[threadIdx.x >> 6] = x ? 1.f : 0.f; }
__device__ __forceinline__ bool any_flag(const float* flags) {
  const floatx4 f = load4(flags);
  return __builtin_amdgcn_readfirstlane(f[0] + f[1] + f[2] + f[3] != 0.f);
}
// Tiles of such a tensor in LDS, rows as given: bf16 rows 80 elements apart, which touch every bank once in both directions, and a wave's
// sixteen where its rows of an fp32 tile begin (before a barrier they are the wave's alone)
constexpr int LDG = 80;
static_assert(16 * LDG * sizeof(bf16_t) <= 16 * LD * sizeof(float), "a wave's rows");
__device__ __forceinline__ int given_at(int row) { return (row >> 4) * (16 * LD * 2) + (row & 15) * LDG; }
__device__ __forceinline__ void put_given(float* tile, const Lane& w, const Row<float>& x) {
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) store4(tile + w.t * LD + 16 * cb + 4 * w.g, x[cb]);
}
__device__ __forceinline__ void put_given(float* tile, const Lane& w, const Row<bf16_t>& x) {
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16_t*>(tile) + given_at(w.t) + 16 * cb + 4 * w.g) = x.x[cb].x;
}
// Elements k .. k + 3 of row i; rows k .. k + 3 (of one block) of column c0 + l16
template <typename T> __device__ __forceinline__ Raw4<T> given_row(const float* tile, int i, int k) {
  Raw4<T> r;
  if constexpr (sizeof(T) == 2) r.x = *reinterpret_cast<const bf16x4*>(reinterpret_cast<const bf16_t*>(tile) + given_at(i) + k);
  else r.x = frag<true>(tile, i, k);
  return r;
}
template <typename T> __device__ __forceinline__ Raw4<T> given_col(const float* tile, int c0, int k, const Lane& w) {
  Raw4<T> r;
  if constexpr (sizeof(T) == 2) r.x = Mma16::rows4(reinterpret_cast<const bf16_t*>(tile) + given_at(k), LDG, 0, c0, threadIdx.x);
  else r.x = frag<false>(tile, c0 + w.l16, k);
  return r;
}

// A result whose columns are the wave's tokens (column l16, rows 16 nb + 4 g ..) into rows = tokens
__device__ __forceinline__ void put_cols(float* tile, const Lane& w, const floatx4 (&c)[4]) {
  put_row(tile, w, [&](int cb) { return c[cb]; });
}
// A result whose rows are the wave's tokens (rows 4 g .., column 16 nb + l16) into rows = columns
__device__ __forceinline__ void put_rows(float* tile, const Lane& w, const floatx4 (&c)[4]) {
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) store4(tile + (16 * nb + w.l16) * LD + 16 * w.j + 4 * w.g, c[nb]);
}
__device__ __forceinline__ void clear(floatx4 (&c)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c[i] = zero4();
}

// ---- decays --------------------------------------------------------------------------------------------------
// of another lane in the row of 16 (CTRL: a DPP control), 1 where there is none
template <int CTRL> __device__ __forceinline__ floatx4 neighbour(floatx4 x) {
  floatx4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = __int_as_float(__builtin_amdgcn_update_dpp(0x3f800000, __float_as_int(x[e]), CTRL, 0xF, 0xF, false));
  return r;
}
__device__ __forceinline__ floatx4 token_before(floatx4 x) { return neighbour<0x111>(x); }
__device__ __forceinline__ floatx4 token_after(floatx4 x) { return neighbour<0x101>(x); }
// Products over the row of 16 lanes up to and with the lane's own, and from it on
__device__ __forceinline__ floatx4 product_upto(floatx4 x) {  // row_shr 1, 2, 4, 8
  x *= neighbour<0x111>(x);
  x *= neighbour<0x112>(x);
  x *= neighbour<0x114>(x);
  return x * neighbour<0x118>(x);
}
__device__ __forceinline__ floatx4 product_from(floatx4 x) {  // row_shl
  x *= neighbour<0x101>(x);
  x *= neighbour<0x102>(x);
  x *= neighbour<0x104>(x);
  return x * neighbour<0x108>(x);
}

constexpr int LDS_TILES = 4;
constexpr int SX = 15 * 64;  // dplr_grad's sums that cross waves; the flags of the others
constexpr unsigned LDS_BYTES = (LDS_TILES * TS + 5 * 64 + SX) * sizeof(float);
static_assert(LDS_BYTES <= 80 * 1024, "two workgroups per CU");
struct Lds {
  float *base, *total, *one;  // total: [4][64], decays of the whole blocks; one: 64 ones
  float* sx;                  // SX floats
  __device__ __forceinline__ Lds(char* smem) {
    base = reinterpret_cast<float*>(smem);
    total = base + LDS_TILES * TS, one = total + 256, sx = one + 64;
  }
  __device__ __forceinline__ float* tile(int i) const { return base + i * TS; }
  // Decays of the whole blocks between two, e < l: blocks 1 and 2 are the only ones that can lie between others.  One of the two is a
  // constant; `at`: channel.  No branch: a block that is not in between reads ones.
  template <int E> __device__ __forceinline__ floatx4 from(int l, int at) const { return between4(E, l, at, E < 1, E < 2); }
  template <int L> __device__ __forceinline__ floatx4 to(int e, int at) const { return between4(e, L, at, L > 1, L > 2); }
  template <int E> __device__ __forceinline__ float from1(int l, int at) const { return between1(E, l, at, E < 1, E < 2); }
  template <int L> __device__ __forceinline__ float to1(int e, int at) const { return between1(e, L, at, L > 1, L > 2); }
  __device__ __forceinline__ const float* if_between(int e, int m, int l) const { return e < m && m < l ? total + 64 * m : one; }
  __device__ __forceinline__ floatx4 between4(int e, int l, int at, bool m1, bool m2) const {
    floatx4 x = {1.f, 1.f, 1.f, 1.f};
    if (m1) x = load4(if_between(e, 1, l) + at);
    if (m2) x *= load4(if_between(e, 2, l) + at);
    return x;
  }
  __device__ __forceinline__ float between1(int e, int l, int at, bool m1, bool m2) const {
    float x = 1.f;
    if (m1) x = if_between(e, 1, l)[at];
    if (m2) x *= if_between(e, 2, l)[at];
    return x;
  }
  // Decays from the chunk's start to block j, and from its end to the chunk's
  __device__ __forceinline__ floatx4 start_to(int j, int at) const { return load4((j > 0 ? total : one) + at) * load4(if_between(0, 1, j) + at) * load4(if_between(0, 2, j) + at); }
  __device__ __forceinline__ floatx4 end_from(int j, int at) const { return load4(if_between(j, 1, 3) + at) * load4(if_between(j, 2, 3) + at) * load4((j < 3 ? total + 192 : one) + at); }
  __device__ __forceinline__ float start_to1(int j, int c) const { return (j > 0 ? total : one)[c] * if_between(0, 1, j)[c] * if_between(0, 2, j)[c]; }
  __device__ __forceinline__ float end_from1(int j, int c) const { return if_between(j, 1, 3)[c] * if_between(j, 2, 3)[c] * (j < 3 ? total + 192 : one)[c]; }
  // ... from the end of each block, of one channel, and of the whole chunk
  __device__ __forceinline__ void ends(int c, float (&r)[4], float& chunk) const {
    r[3] = 1.f, r[2] = total[192 + c], r[1] = r[2] * total[128 + c], r[0] = r[1] * total[64 + c], chunk = r[0] * total[c];
  }
};

// The gates of the lane's block.  Sums of gates in fixed point (2^-24 in units of log 2) are exact: P and S carry the rounding of one
// exponential each, whatever the sums' sizes.  A gate or a sum that the format does not hold, or NaN, makes the block DIRECT.
constexpr int ONE = 1 << 24;
__device__ __forceinline__ int fixed_gate(float g, bool& ok) {
  const float c = 1.44269504f * ONE;
  float t = g * c;
  asm volatile("" : "+v"(t));  // -ffast-math must not see that the next line is a rounding error
  const float e = __builtin_fmaf(g, 1.92596299e-8f * ONE, __builtin_fmaf(g, c, -t));
  ok = fabsf(t) <= 7.f * ONE;  // sixteen of them stay below 2^31
  return ok ? (int)__builtin_rintf(t + e) : 0;
}
__device__ __forceinline__ float exp2_fixed(int x) { return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f((float)(x & (ONE - 1)) * (1.f / ONE)), x >> 24); }
template <int CTRL> __device__ __forceinline__ int dpp_of(int x) { return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xF, 0xF, true); }
struct Gates {
  int sum[4][4];  // from the block's first token up to and with the lane's
  bool direct;
  __device__ __forceinline__ explicit Gates(const Row<float>& gk) {
    bool fits = true;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const floatx4 g = gk[cb];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bool ok;
        int x = fixed_gate(g[e], ok);
        fits = fits && ok;
        x += dpp_of<0x111>(x), x += dpp_of<0x112>(x), x += dpp_of<0x114>(x), x += dpp_of<0x118>(x);  // row_shr 1, 2, 4, 8
        fits = fits && abs(x) <= RANGE * ONE;
        sum[cb][e] = x;
      }
    }
    direct = __ballot(!fits) != 0;
  }
  __device__ __forceinline__ floatx4 upto(int cb) const {  // P
    floatx4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = exp2_fixed(sum[cb][e]);
    return r;
  }
  __device__ __forceinline__ floatx4 behind(int cb) const {  // S
    floatx4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = exp2_fixed(dpp_of<0x15F>(sum[cb][e]) - sum[cb][e]);  // row_newbcast:15
    return r;
  }
};
// The decays of a DIRECT block's tokens, one by one
__device__ __forceinline__ void token_decays(const ChunkParams& p, const Slot& s, const Lane& w, floatx4 (&x)[4]) {
  Row<float> gk;
  gk.load(p.gk, s, w);
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const floatx4 g = gk[cb];
    x[cb] = floatx4{exp_f(g[0]), exp_f(g[1]), exp_f(g[2]), exp_f(g[3])};
  }
}
struct Decay {
  floatx4 p[4], s[4];
  __device__ __forceinline__ Decay(const Gates& g, const ChunkParams& c, const Slot& sl, const Lane& w) {
    if (!g.direct) {
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) p[cb] = g.upto(cb), s[cb] = g.behind(cb);
    } else {
      floatx4 x[4];
      token_decays(c, sl, w, x);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) p[cb] = product_upto(x[cb]), s[cb] = product_from(token_after(x[cb]));
    }
  }
};
// The whole block's, for the other waves (visible after a barrier)
__device__ __forceinline__ void put_total(const Lds& L, const Lane& w, int cb, floatx4 p) {
  if (w.l16 == 15) store4(L.total + 64 * w.j + 16 * cb + 4 * w.g, p);
}

// The lane's row of q, k, a, b and its gates
template <typename T> struct Own {
  Row<T> q, k, a, b;
  Row<float> gk;
  __device__ __forceinline__ void load(const ChunkParams& p, const Slot& s, const Lane& w) { load_gates(p, s, w), load_rows(p, s, w); }
  __device__ __forceinline__ void load_gates(const ChunkParams& p, const Slot& s, const Lane& w) { gk.load(p.gk, s, w); }
  __device__ __forceinline__ void load_rows(const ChunkParams& p, const Slot& s, const Lane& w) {
    q.load(p.q, s, w);
    a.load(p.a, s, w);
    b.load(p.b, s, w);
    k.load(p.k, s, w);
  }
};

// DIRECT block: its pairs one by one.  The lane has four pairs, of tokens l16 and 4 g + r; BY_T: l16 is the later one.  The vectors come
// from memory, the decays w from the wave's rows of `own`.
struct Pairs {
  floatx4 ab, ak, qb, qk;
};
template <typename T, bool BY_T> __device__ __forceinline__ Pairs direct_pairs(const ChunkParams& p, const Slot& sl, const Lane& w, const float* own) {
  auto row = [&](const void* base, int i, int c) {
    Raw4<T> x;
    const bool ok = 16 * w.j + i < sl.len;
    x.load(static_cast<const T*>(base) + (ok ? (sl.tok + 16 * w.j + i) * D + c : 0));
    return ok ? x.get() : zero4();
  };
  auto dot = [](floatx4 x, floatx4 y) { return x[0] * y[0] + x[1] * y[1] + x[2] * y[2] + x[3] * y[3]; };
  Pairs m{zero4(), zero4(), zero4(), zero4()};
#pragma unroll 1
  for (int c = 0; c < D; c += 4) {
    floatx4 e[4], el[4];  // E of the later token and of the one before it
#pragma unroll
    for (int r = 0; r < 4; ++r) e[r] = el[r] = floatx4{1.f, 1.f, 1.f, 1.f};
#pragma unroll 1
    for (int i = 1; i < 16; ++i) {
      const floatx4 x = load4(own + (16 * w.j + i) * LD + c);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = BY_T ? w.l16 : 4 * w.g + r, s = BY_T ? 4 * w.g + r : w.l16;
#pragma unroll
        for (int n = 0; n < 4; ++n) {
          e[r][n] *= i > s && i <= t ? x[n] : 1.f;
          el[r][n] *= i > s && i < t ? x[n] : 1.f;
        }
      }
    }
    const floatx4 f1 = row(BY_T ? p.a : p.b, w.l16, c), f2 = row(BY_T ? p.q : p.k, w.l16, c);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int o = 4 * w.g + r;
      const floatx4 h1 = row(BY_T ? p.b : p.a, o, c), h2 = row(BY_T ? p.k : p.q, o, c);
      const floatx4 a = BY_T ? f1 : h1, q = p.scale * (BY_T ? f2 : h2), b = BY_T ? h1 : f1, k = BY_T ? h2 : f2;
      const int t = BY_T ? w.l16 : o, s = BY_T ? o : w.l16;
      if (s < t) m.ab[r] += dot(a * el[r], b), m.ak[r] += dot(a * el[r], k);
      if (s <= t) m.qb[r] += dot(q * e[r], b), m.qk[r] += dot(q * e[r], k);
    }
  }
  return m;
}

// A block of a lower-triangular pair matrix M[t][s] on the diagonal.  BY_T: rows s, columns t, else rows t, columns s.  Entries above the
// diagonal (STRICT: on it, too) are cleared.
template <bool BY_T, bool STRICT> __device__ __forceinline__ void mask(floatx4& m, const Lane& w) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = 4 * w.g + r, t = BY_T ? w.l16 : row, s = BY_T ? row : w.l16;
    m[r] = (STRICT ? s >= t : s > t) ? 0.f : m[r];
  }
}
// The wave's rows of a lower-triangular matrix: what lies before block j, the block itself, zeros
template <typename F> __device__ __forceinline__ void put_tri(float* tile, const Lane& w, const floatx4 (&x)[3], floatx4 d, F&& value) {
#pragma unroll
  for (int sb = 0; sb < 4; ++sb) {
    floatx4 y = sb == w.j ? d : zero4();
    if (sb < 3) y = sb < w.j ? x[sb < 3 ? sb : 0] : y;
    store4(tile + w.t * LD + 16 * sb + 4 * w.g, value(y));
  }
}

// ---- forward: M, X, N^T, Y of a chunk ------------------------------------------------------------------------
template <typename T, bool FULL> __device__ __forceinline__ bool prepare_chunk(const ChunkParams& p, const Lds& L) {
  const Slot s = slot_of(p);
  const Lane w;
  const int l16 = w.l16, g = w.g, g4 = 4 * w.g;
  float *tb = L.tile(0), *tk = L.tile(1), *ta = L.tile(2), *tx = L.tile(3);
  Own<T> x;
  x.load(p, s, w);
  Row<T> v;
  v.load(p.v, s, w);
  floatx4 fq[4], fa[4];                // q P, a P of the token before
  floatx4 ab[3], ak[3], qb[3], qk[3];  // pairs with tokens of earlier blocks, by t
  Pairs m{zero4(), zero4(), zero4(), zero4()};  // and of the lane's own
#pragma unroll
  for (int i = 0; i < 3; ++i) ab[i] = ak[i] = qb[i] = qk[i] = zero4();
  {
    const Gates gates(x.gk);
    const Decay e(gates, p, s, w);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) put_total(L, w, cb, e.p[cb]);
    if (threadIdx.x < 64) L.one[threadIdx.x] = 1.f;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) fq[cb] = p.scale * x.q[cb] * e.p[cb], fa[cb] = x.a[cb] * token_before(e.p[cb]);
    if (!gates.direct) {
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        const floatx4 r = rcp4(e.p[cb]), b = x.b[cb] * r, k = x.k[cb] * r;
        mfma_block<4>({&m.ab, &m.ak, &m.qb, &m.qk}, [&](int i) { return i & 1 ? k : b; }, [&](int i) { return i & 2 ? fq[cb] : fa[cb]; });
      }
      mask<true, true>(m.ab, w), mask<true, true>(m.ak, w), mask<true, false>(m.qb, w), mask<true, false>(m.qk, w);
    } else {
      floatx4 decays[4];
      token_decays(p, s, w, decays);
      put_cols(tx, w, decays);
      __builtin_amdgcn_wave_barrier();
      m = direct_pairs<T, true>(p, s, w, tx);
      __builtin_amdgcn_wave_barrier();
    }
    put_row(tb, w, [&](int cb) { return x.b[cb] * e.s[cb]; });
    put_row(tk, w, [&](int cb) { return x.k[cb] * e.s[cb]; });
    put_given(tx, w, v);
  }
  lds_barrier();
  before(w.j, [&](auto sb_) {
    constexpr int sb = decltype(sb_)::value;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const floatx4 rb = frag<true>(tb, 16 * sb + l16, 16 * kb + g4), rk = frag<true>(tk, 16 * sb + l16, 16 * kb + g4), gap = L.from<sb>(w.j, 16 * kb + g4);
      const floatx4 ra = fa[kb] * gap, rq = fq[kb] * gap;
      mfma_block<4>({&ab[sb], &ak[sb], &qb[sb], &qk[sb]}, [&](int i) { return i & 1 ? rk : rb; }, [&](int i) { return i & 2 ? rq : ra; });
    }
  });
  floatx4 xx[4];  // q e, then X^T: rows = channels, columns = tokens
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const floatx4 st = L.start_to(w.j, 16 * cb + g4);
    xx[cb] = fq[cb] * st;
    store4(ta + w.t * LD + 16 * cb + g4, fa[cb] * st);  // a e of the token before
  }
  float end[4], chunk;  // decays of channel w.t from the end of each block
  L.ends(w.t, end, chunk);
  floatx4 nt[4], z[4], y[4];  // N (rows i, columns n), Aak v (rows t, columns n), Y^T (rows n, columns t)
  clear(nt), clear(z), clear(y);
  auto new_sums = [&](auto full) {
#pragma unroll
    for (int sb = 0; sb < 4; ++sb) {
      const Parts<T, decltype(full)::value> kf(frag<false>(tk, 16 * w.j + l16, 16 * sb + g4) * end[sb]);
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) mfma_parts(nt[nb], kf, given_col<T>(tx, 16 * nb, 16 * sb + g4, w));
    }
  };
  // Where a channel's decay over the last block is below 2^-24, N is the sum of a few tokens: the matrix instruction cuts a sum of bf16 products off
  // where it rounds one of fp32 ones, and with so few terms no rounding of a longer sum outweighs that.  h's error, 1e-7 of its 2-norm, by parts and
  // in fp32: RWKV-7's decays (2^-14 and above) 0.53 and 0.69, three times those 0.47 and 0.50, four 0.46 and 0.45, six 0.46 and 0.41, ten 0.48
  // and 0.37.  Parts' sums apart, added at the end: 0.59 .. 0.54.
  bool full = FULL;
  if constexpr (!FULL) {
    full = __ballot(end[2] < 0x1p-24f) != 0;
    if (!full) new_sums(std::false_type{});
  }
  if (full) new_sums(std::true_type{});
  before(w.j, [&](auto sb_) {
    constexpr int sb = decltype(sb_)::value;
    const Parts<T, FULL> a(ak[sb]), q(qk[sb]);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const Raw4<T> vf = given_col<T>(tx, 16 * nb, 16 * sb + g4, w);
      mfma_parts(z[nb], a, vf);
      mfma_parts(y[nb], vf, q);
    }
  });
  {
    const Parts<T, FULL> a(m.ak), q(m.qk);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const Raw4<T> vf = given_col<T>(tx, 16 * nb, 16 * w.j + g4, w);
      mfma_parts(z[nb], a, vf);
      mfma_parts(y[nb], vf, q);
    }
  }
  lds_barrier();
  put_tri(tx, w, ab, m.ab, [](floatx4 y_) { return -y_; });
  put_rows(tk, w, z);
  lds_barrier();
  tri_inverse_64(tx, threadIdx.x);
  {
    floatx4 W[4], u[4];
    clear(W), clear(u);
    upto(w.j, [&](auto sb_) {
      constexpr int sb = decltype(sb_)::value;
      const floatx4 tf = frag<true>(tx, w.t, 16 * sb + g4);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        mfma4(W[cb], tf, frag<false>(ta, 16 * cb + l16, 16 * sb + g4));
        mfma4(u[cb], tf, frag<true>(tk, 16 * cb + l16, 16 * sb + g4));
      }
    });
    lds_barrier();
    put_rows(ta, w, W);
    put_rows(tk, w, u);
  }
  lds_barrier();
  floatx4 mm[4];  // M[i][c]: rows c, columns i
  floatx4 ntu[4], xw[4], yu[4];  // what W and U0 add to N, X and Y
  clear(mm), clear(ntu), clear(xw), clear(yu);
#pragma unroll
  for (int sb = 0; sb < 4; ++sb) {
    const floatx4 bf = frag<false>(tb, 16 * w.j + l16, 16 * sb + g4) * end[sb];
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const floatx4 wf = frag<true>(ta, 16 * cb + l16, 16 * sb + g4), uf = frag<true>(tk, 16 * cb + l16, 16 * sb + g4);
      mfma4(mm[cb], wf, bf);
      mfma4(ntu[cb], bf, uf);
    }
  }
  before(w.j, [&](auto sb_) {
    constexpr int sb = decltype(sb_)::value;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      mfma4(xw[cb], frag<true>(ta, 16 * cb + l16, 16 * sb + g4), qb[sb]);
      mfma4(yu[cb], frag<true>(tk, 16 * cb + l16, 16 * sb + g4), qb[sb]);
    }
  });
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    mfma4(xw[cb], frag<true>(ta, 16 * cb + l16, 16 * w.j + g4), m.qb);
    mfma4(yu[cb], frag<true>(tk, 16 * cb + l16, 16 * w.j + g4), m.qb);
    floatx4 r = mm[cb];
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (16 * cb + g4 + e == w.t) r[e] += chunk;
    const int at = block_at(w.j, cb);
    store4(p.M + s.kept * TG + at, r);
    store4(p.X + s.kept * TG + at, xx[cb] + xw[cb]);
    y[cb] += yu[cb], nt[cb] += ntu[cb];
    store4(p.s2 + s.win * TG + at, y[cb]);
    store4(p.s1 + s.win * TG + block_at(cb, w.j), nt[cb]);
  }
  if constexpr (!FULL) {  // (what z had, N has in the whole column)
    put_flag(L.sx, any_nan(nt, y));
    lds_barrier();
    return !any_flag(L.sx);
  }
  return true;
}
template <typename T>
__global__ __launch_bounds__(256, 2) void dplr_prepare_kernel(ChunkParams p) {
  extern __shared__ __align__(16) char smem[];
  const Lds L(smem);
  if (!prepare_chunk<T, sizeof(T) == 4>(p, L)) prepare_chunk<T, true>(p, L);
}

// ---- the sequential pass: h <- M h + N (forward), D <- M^T D + R (backward) ------------------------------------
// One workgroup per row and 16 of the 64 value columns; wave w forms 16 rows of the new state, sixteen products of 32 cycles, from its
// rows of M, which come straight into its registers three chunks ahead, and the old state, which the waves exchange
// through LDS (transposed), one LDS barrier per chunk.  A whole chain on one wave per 16 columns took four times the products and
// M through LDS: 1.85 us per chunk.  In reverse a wave's rows of M^T are columns of M: its blocks of M are turned through LDS of its own,
// a chunk ahead (read from memory as columns, four rows at a time, the pass took 101 us instead of 89 at B8 H16 T4096).
struct ScanParams {
  const float* M;    // kept tiles [rows][KN]
  const float* add;  // window tiles: N^T or R^T
  float* st;         // the state entering (forward: kept [rows][KN + 1]) or the gradient leaving (backward: window) each chunk, transposed
  const float* s_in; // [dk][dv] per row, or NULL
  float* s_out;      // [dk][dv] per row, or NULL
  int64_t rows;
  int KN, at, nw;    // the window is chunks [at, at + nw) of the kept tensors
};

constexpr int LDT = 20;  // rows of 16 floats on their way through LDS: both ways touch every bank once

template <bool BWD>
__global__ __launch_bounds__(256) void dplr_chunk_scan_kernel(ScanParams p) {
  __shared__ __align__(16) float buf[2][16 * LD], own_[BWD ? 4 : 1][BWD ? 64 * LDT : 4];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  int64_t row;
  int part;
  if (!xcd_slot_part(p.rows, 4, row, part)) return;  // the four parts read the same M: one XCD
  const int col = 16 * part + l16, r0 = 16 * wave + 4 * g;  // this lane's column and its first row of the state
  const float* Mrow = p.M + (row * p.KN + p.at) * TG + (BWD ? block_at(0, wave) : block_at(wave, 0));
  const float* Arow = p.add + row * p.nw * TG + block_at(part, wave);
  float* Srow = p.st + (BWD ? row * p.nw : row * (p.KN + 1) + p.at) * TG + block_at(part, wave);
  float* own = own_[BWD ? wave : 0];
  auto chunk = [&](int i) { return (int64_t)(BWD ? p.nw - 1 - i : i); };
  floatx4 h;
#pragma unroll
  for (int r = 0; r < 4; ++r) h[r] = p.s_in ? p.s_in[row * TG + (r0 + r) * D + col] : 0.f;
  struct Ahead {
    floatx4 m[4], a;
  } x0, x1, x2, x3;
  auto fetch = [&](Ahead& x, int i) {
    const float* M = Mrow + chunk(min(i, p.nw - 1)) * TG;
#pragma unroll
    for (int b = 0; b < 4; ++b) x.m[b] = load4(M + (BWD ? 4 * 256 : 256) * b);
    x.a = load4(Arow + chunk(min(i, p.nw - 1)) * TG);
  };
  floatx4 m[4];  // backward: the rows of M^T of the chunk at hand
  auto turn = [&](const Ahead& x) {
#pragma unroll
    for (int b = 0; b < 4; ++b) store4(own + (16 * b + l16) * LDT + 4 * g, x.m[b]);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e) m[b][e] = own[(16 * b + 4 * g + e) * LDT + l16];
    __builtin_amdgcn_wave_barrier();
  };
  auto step = [&](Ahead& x, const Ahead& next, Ahead& free, int i) {  // next: chunk i + 1; free: the set that chunk i - 1 has used
    lds_barrier();
    const float* cur = buf[i & 1] + l16 * LD + 4 * g;
    floatx4 f[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) f[b] = load4(cur + 16 * b);
    fetch(free, i + 3);
    store4(Srow + chunk(i) * TG, h);
    floatx4 y0 = zero4(), y1 = zero4();
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        y0 = __builtin_amdgcn_mfma_f32_16x16x4f32((BWD ? m[2 * b] : x.m[2 * b])[r], f[2 * b][r], y0, 0, 0, 0);
        y1 = __builtin_amdgcn_mfma_f32_16x16x4f32((BWD ? m[2 * b + 1] : x.m[2 * b + 1])[r], f[2 * b + 1][r], y1, 0, 0, 0);
      }
    if (BWD) turn(next);
    h = (y0 + y1) + x.a;
    store4(buf[(i + 1) & 1] + l16 * LD + r0, h);
  };
  fetch(x0, 0);
  fetch(x1, 1);
  fetch(x2, 2);
  store4(buf[0] + l16 * LD + r0, h);
  if (BWD) turn(x0);
  int i = 0;
  for (; i + 4 <= p.nw; i += 4) {  // no way out in between: with one the compiler waited for the loads in flight here
    step(x0, x1, x3, i);
    step(x1, x2, x0, i + 1);
    step(x2, x3, x1, i + 2);
    step(x3, x0, x2, i + 3);
  }
  if (i < p.nw) step(x0, x1, x3, i);
  if (i + 1 < p.nw) step(x1, x2, x0, i + 1);
  if (i + 2 < p.nw) step(x2, x3, x1, i + 2);
  if (!BWD && p.at + p.nw == p.KN) store4(Srow + (int64_t)p.nw * TG, h);
  if (p.s_out) {
#pragma unroll
    for (int r = 0; r < 4; ++r) p.s_out[row * TG + (r0 + r) * D + col] = h[r];
  }
}

template <typename T> __device__ __forceinline__ void store_row4(void* base, int64_t at, floatx4 x) { store4(static_cast<T*>(base) + at, x); }

// ---- outputs: o = X h + Y ------------------------------------------------------------------------------------
// Bound by its 48 KB of reads per chunk: operands straight from memory in fragment order (each wave: 16 tokens), no LDS.
template <typename T>
__global__ __launch_bounds__(256) void dplr_out_kernel(ChunkParams p) {
  const Slot s = slot_of(p);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4, t = 16 * wave + l16;
  const float* X = p.X + s.kept * TG + block_at(wave, 0);
  const float* Y = p.s2 + s.win * TG + block_at(wave, 0);
  const float* h = p.hT + s.st * TG + block_at(0, 0);
  if (16 * wave >= s.len) return;
  floatx4 x[4], y[4], acc[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) x[b] = load4(X + 256 * b), y[b] = load4(Y + 256 * b), acc[b] = zero4();
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) mfma4(acc[nb], load4(h + (4 * nb + kb) * 256), x[kb]);
  if (t < s.len) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) store_row4<T>(p.o, (s.tok + t) * D + 16 * nb + 4 * g, acc[nb] + y[nb]);
  }
}

// ---- backward: R^T = (X^T dO)^T ------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void dplr_r_kernel(ChunkParams p) {
  __shared__ __align__(16) float tX[TS], tO[TS];
  const Slot s = slot_of(p);
  const Lane w;
  const int l16 = w.l16, g4 = 4 * w.g;
  Row<float> x;
  Row<T> d;
  x.load_tile(p.X + s.kept * TG, w.j);
  d.load(p.d_o, s, w);
  put_row(tX, w, [&](int cb) { return x[cb]; });
  put_given(tO, w, d);
  lds_barrier();
  floatx4 acc[4];
  auto sums = [&](auto full) {
    clear(acc);
#pragma unroll
    for (int kb = 3; kb >= 0; --kb) {  // the chunk's first tokens, whose share is the largest, last
      const Parts<T, decltype(full)::value> a(frag<false>(tX, w.t, 16 * kb + g4));
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) mfma_parts(acc[nb], a, given_col<T>(tO, 16 * nb, 16 * kb + g4, w));
    }
  };
  sums(std::bool_constant<sizeof(T) == 4>{});
  if (sizeof(T) == 2 && any_nan(acc)) sums(std::true_type{});
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) store4(p.s2 + s.win * TG + block_at(nb, w.j), acc[nb]);
}

// ---- backward: u, dU and dv of a chunk -----------------------------------------------------------------------
// The pair matrices and the inverse are formed again: keeping the pairs would move 128 KB per chunk through memory, and the inverse alone (10 KB of
// 48 more to hold between the passes) gave 1.4 % of forward and backward, 0.4 % with fp32 tensors.
template <typename T, bool FULL> __device__ __forceinline__ bool u_chunk(const ChunkParams& p, const Lds& L) {
  const Slot s = slot_of(p);
  const Lane w;
  const int l16 = w.l16, g4 = 4 * w.g;
  float *tb = L.tile(0), *tk = L.tile(1), *ta = L.tile(2), *tx = L.tile(3);
  Own<T> x;
  x.load(p, s, w);
  Row<T> v, d_o;
  v.load(p.v, s, w);
  d_o.load(p.d_o, s, w);
  Row<float> h0, dC;
  h0.load_tile(p.hT + s.st * TG, w.j);
  dC.load_tile(p.s1 + s.win * TG, w.j);
  floatx4 fa[4], fb[4], fk[4];  // the lane's row: a P of the token before, b S, k S
  floatx4 ab[3], akT[3];        // Aab, Aak by t, with earlier blocks
  floatx4 ak[3], qb[3], qk[3];  // Aak, Pqb, Pqk by s, with later blocks (of block i + 1)
  floatx4 abd = zero4(), akTd = zero4(), akd = zero4(), qbd = zero4(), qkd = zero4();  // the lane's own block
#pragma unroll
  for (int i = 0; i < 3; ++i) ab[i] = akT[i] = ak[i] = qb[i] = qk[i] = zero4();
  {
    const Gates gates(x.gk);
    const Decay e(gates, p, s, w);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) put_total(L, w, cb, e.p[cb]);
    if (threadIdx.x < 64) L.one[threadIdx.x] = 1.f;
    floatx4 fq[4];
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
      fq[cb] = p.scale * x.q[cb] * e.p[cb], fa[cb] = x.a[cb] * token_before(e.p[cb]), fb[cb] = x.b[cb] * e.s[cb], fk[cb] = x.k[cb] * e.s[cb];
    if (!gates.direct) {
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        const floatx4 r = rcp4(e.p[cb]), b = x.b[cb] * r, k = x.k[cb] * r;
        mfma_block<5>({&abd, &akTd, &akd, &qbd, &qkd}, [&](int i) { return i == 0 ? b : i == 1 ? k : i == 2 ? fa[cb] : fq[cb]; },
                      [&](int i) { return i < 2 ? fa[cb] : i == 3 ? b : k; });
      }
      mask<true, true>(abd, w), mask<true, true>(akTd, w), mask<false, true>(akd, w), mask<false, false>(qbd, w), mask<false, false>(qkd, w);
    } else {
      floatx4 decays[4];
      token_decays(p, s, w, decays);
      put_cols(tx, w, decays);
      __builtin_amdgcn_wave_barrier();
      const Pairs byt = direct_pairs<T, true>(p, s, w, tx), bys = direct_pairs<T, false>(p, s, w, tx);
      abd = byt.ab, akTd = byt.ak, akd = bys.ak, qbd = bys.qb, qkd = bys.qk;
      __builtin_amdgcn_wave_barrier();
    }
    put_cols(ta, w, fa), put_cols(tb, w, fb), put_cols(tk, w, fk), put_cols(tx, w, fq);
  }
  lds_barrier();
  before(w.j, [&](auto b_) {
    constexpr int b = decltype(b_)::value;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const floatx4 rb = frag<true>(tb, 16 * b + l16, 16 * kb + g4), rk = frag<true>(tk, 16 * b + l16, 16 * kb + g4), ra = fa[kb] * L.from<b>(w.j, 16 * kb + g4);
      mfma_block<2>({&ab[b], &akT[b]}, [&](int i) { return i ? rk : rb; }, [&](int) { return ra; });
    }
  });
  after(w.j, [&](auto b_) {
    constexpr int b = decltype(b_)::value;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const floatx4 ra = frag<true>(ta, 16 * b + l16, 16 * kb + g4), rq = frag<true>(tx, 16 * b + l16, 16 * kb + g4), gap = L.to<b>(w.j, 16 * kb + g4);
      const floatx4 rk = fk[kb] * gap, rb = fb[kb] * gap;
      mfma_block<3>({&ak[b - 1], &qb[b - 1], &qk[b - 1]}, [&](int i) { return i ? rq : ra; }, [&](int i) { return i == 1 ? rb : rk; });
    }
  });
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {  // from here on relative to the chunk's start and end
    const floatx4 en = L.end_from(w.j, 16 * cb + g4);
    fa[cb] *= L.start_to(w.j, 16 * cb + g4), fb[cb] *= en, fk[cb] *= en;
  }
  lds_barrier();
  float *th = ta, *tO = tb, *tD = tk, *tv = tx;
  put_given(tv, w, v);
  put_given(tO, w, d_o);
  put_row(th, w, [&](int cb) { return h0[cb]; });  // [value column][channel]
  put_row(tD, w, [&](int cb) { return dC[cb]; });
  lds_barrier();
  floatx4 z[4], y[4], dv[4];  // a h + Aak v, b r D + Pqb^T dO (rows t, columns n), dv (rows n, columns t)
  clear(z), clear(y), clear(dv);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const floatx4 hf = frag<true>(th, 16 * nb + l16, 16 * kb + g4), df = frag<true>(tD, 16 * nb + l16, 16 * kb + g4);
      mfma4(z[nb], fa[kb], hf);
      mfma4(y[nb], fb[kb], df);
      mfma4(dv[nb], df, fk[kb]);
    }
  // The sums go on from fp32 to bf16 matrix instructions.  hipcc's wait states for a change of kind on one accumulator have been too few once
  // (16x16x16 into 16x16x32, both bf16, lost elements), so whatever the schedule none of the first kind's results, of eight passes, is under way
  // behind these 32 states.  Sums of their own for the two kinds cost 150 spills (no difference in time measured with the states).
  if constexpr (sizeof(T) == 2 && !FULL)
    asm volatile("s_nop 15\n\ts_nop 15"
                 : "+v"(z[0]), "+v"(z[1]), "+v"(z[2]), "+v"(z[3]), "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3]), "+v"(dv[0]), "+v"(dv[1]), "+v"(dv[2]), "+v"(dv[3]));
  before(w.j, [&](auto b_) {
    constexpr int b = decltype(b_)::value;
    const Parts<T, FULL> a(akT[b]);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) mfma_parts(z[nb], a, given_col<T>(tv, 16 * nb, 16 * b + g4, w));
  });
  after(w.j, [&](auto b_) {
    constexpr int b = decltype(b_)::value;
    const Parts<T, FULL> pb(qb[b - 1]), pk(qk[b - 1]);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const Raw4<T> of = given_col<T>(tO, 16 * nb, 16 * b + g4, w);
      mfma_parts(y[nb], pb, of);
      mfma_parts(dv[nb], of, pk);
    }
  });
  {
    const Parts<T, FULL> a(akTd), pb(qbd), pk(qkd);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const Raw4<T> of = given_col<T>(tO, 16 * nb, 16 * w.j + g4, w);
      mfma_parts(z[nb], a, given_col<T>(tv, 16 * nb, 16 * w.j + g4, w));
      mfma_parts(y[nb], pb, of);
      mfma_parts(dv[nb], of, pk);
    }
  }
  if constexpr (!FULL) put_flag(L.sx, any_nan(z, y, dv));
  lds_barrier();
  if constexpr (!FULL)
    if (any_flag(L.sx)) return false;
  float *Tm = tx, *tz = ta, *ty = tk, *tdu = tb;
  put_tri(Tm, w, ab, abd, [](floatx4 x_) { return -x_; });
  put_rows(tz, w, z);
  put_rows(ty, w, y);
  lds_barrier();
  tri_inverse_64(Tm, threadIdx.x);
  floatx4 u[4], du[4];  // rows n, columns t
  clear(u), clear(du);
  upto(w.j, [&](auto b_) {
    constexpr int b = decltype(b_)::value;
    const floatx4 tf = frag<true>(Tm, w.t, 16 * b + g4);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) mfma4(u[nb], frag<true>(tz, 16 * nb + l16, 16 * b + g4), tf);
  });
  downto(w.j, [&](auto b_) {
    constexpr int b = decltype(b_)::value;
    const floatx4 tf = frag<false>(Tm, w.t, 16 * b + g4);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) mfma4(du[nb], frag<true>(ty, 16 * nb + l16, 16 * b + g4), tf);
  });
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    store4(p.s3 + s.win * TG + block_at(w.j, nb), u[nb]);
    store4(p.s4 + s.win * TG + block_at(w.j, nb), du[nb]);
  }
  put_cols(tdu, w, du);
  lds_barrier();
  floatx4 dva[4];  // Aak^T dU
  clear(dva);
  after(w.j, [&](auto b_) {
    constexpr int b = decltype(b_)::value;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) mfma4(dva[nb], frag<false>(tdu, 16 * nb + l16, 16 * b + g4), ak[b - 1]);
  });
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) mfma4(dva[nb], frag<false>(tdu, 16 * nb + l16, 16 * w.j + g4), akd);
  if (w.t < s.len) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) store_row4<T>(p.dv, (s.tok + w.t) * D + 16 * nb + g4, dv[nb] + dva[nb]);
  }
  return true;
}
template <typename T>
__global__ __launch_bounds__(256, 2) void dplr_u_kernel(ChunkParams p) {
  extern __shared__ __align__(16) char smem[];
  const Lds L(smem);
  if (!u_chunk<T, sizeof(T) == 4>(p, L)) u_chunk<T, true>(p, L);
}

// ---- backward: dq, dk, da, db, dgk of a chunk ----------------------------------------------------------------
// DIRECT block: what the pairs of the block add to the gradients of the lane's token, four channels from ch.  The matrices lie in LDS rows
// of the wave ([t][s]); E of consecutive partners is a running product of decays, which are formed again from the gates.
template <typename T> struct DirectRows {
  const ChunkParams& p;
  const Slot& sl;
  const Lane& w;
  __device__ __forceinline__ floatx4 operator()(const void* base, int i, int ch) const {
    Raw4<T> x;
    const bool ok = 16 * w.j + i < sl.len;
    x.load(static_cast<const T*>(base) + (ok ? (sl.tok + 16 * w.j + i) * D + ch : 0));
    return ok ? x.get() : zero4();
  }
  __device__ __forceinline__ floatx4 decay(int i, int ch) const {
    const bool ok = 16 * w.j + i < sl.len;
    const floatx4 g = load4(p.gk + (ok ? (sl.tok + 16 * w.j + i) * D + ch : 0));
    return ok ? floatx4{exp_f(g[0]), exp_f(g[1]), exp_f(g[2]), exp_f(g[3])} : floatx4{1.f, 1.f, 1.f, 1.f};
  }
};
// of earlier tokens to dq and da (a token's own b and k apart); m: the lane's row with dPqb, dPqk, dAab, dAak at columns 0, 16, 32, 48
template <typename T> __device__ __forceinline__ void direct_sinks(const DirectRows<T>& row, const float* m, int ch, floatx4& dq, floatx4& da) {
  const int t = row.w.l16;
  floatx4 e = {1.f, 1.f, 1.f, 1.f}, el = e;
#pragma unroll 1
  for (int s = 15; s >= 0; --s) {
    const floatx4 b = row(row.p.b, s, ch), k = row(row.p.k, s, ch), x = row.decay(s, ch);
    if (s <= t) {
      dq += e * (m[s] * b + m[16 + s] * k);
      e *= x;
    }
    if (s < t) {
      da += el * (m[32 + s] * b + m[48 + s] * k);
      el *= x;
    }
  }
}
// of later tokens to db and dk; m: the lane's column of the block's matrices, which lie at columns 0, 16, 32, 48
template <typename T> __device__ __forceinline__ void direct_sources(const DirectRows<T>& row, const float* m, int ch, floatx4& db, floatx4& dk) {
  const int s = row.w.l16;
  floatx4 e = {1.f, 1.f, 1.f, 1.f}, el = e;
#pragma unroll 1
  for (int t = 0; t < 16; ++t) {
    const floatx4 q = row.p.scale * row(row.p.q, t, ch), a = row(row.p.a, t, ch), x = row.decay(t, ch);
    const float* mt = m + t * LD;
    if (t > s) {
      e *= x;
      db += el * a * mt[32], dk += el * a * mt[48];
      el *= x;
    }
    if (t >= s) db += e * q * mt[0], dk += e * q * mt[16];
  }
}

// Over the tokens of the lane's block, from its own on (inclusive) / before its own: each step is one addition with a DPP operand
template <int CTRL> __device__ __forceinline__ floatx4 dpp_add(floatx4 x) {
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x[e]), CTRL, 0xF, 0xF, true));
  return x;
}
__device__ __forceinline__ floatx4 sum_from(floatx4 x) { return dpp_add<0x108>(dpp_add<0x104>(dpp_add<0x102>(dpp_add<0x101>(x)))); }  // row_shl 1, 2, 4, 8
__device__ __forceinline__ floatx4 sum_upto(floatx4 x) { return dpp_add<0x118>(dpp_add<0x114>(dpp_add<0x112>(dpp_add<0x111>(x)))); }  // row_shr
__device__ __forceinline__ floatx4 sum_block(floatx4 x) { return dpp_add<0x128>(dpp_add<0x124>(dpp_add<0x122>(dpp_add<0x121>(x)))); }  // row_ror

// Of another lane in the row of 16, 0 where there is none
template <int CTRL> __device__ __forceinline__ floatx4 dpp_move(floatx4 x) {
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = __int_as_float(dpp_of<CTRL>(__float_as_int(x[e])));
  return x;
}
// Of two rows whose difference sums up to 0 over the block, the difference from the lane on: from lane 8 on that sum, below minus what lies
// before, half as many terms (without bank masks, which keep the additions from taking a DPP operand: 760 us against 750)
__device__ __forceinline__ floatx4 to_middle(floatx4 x) {
  const floatx4 from = dpp_add<0x104>(dpp_add<0x102>(dpp_add<0x101>(x)));                   // right in lanes 8 to 15
  const floatx4 upto = dpp_move<0x111>(dpp_add<0x114>(dpp_add<0x112>(dpp_add<0x111>(x))));  // right in lanes 0 to 7
  return threadIdx.x & 8 ? from : -upto;
}

// dgk_t is what flows through the decay of token t: pairs of a source (b or k of a token before t, the state entering) and a sink (q of t or
// later, a of a later token, the state's gradient).  The formula at the top takes it from sums over the rest of the chunk, where a pair
// behind t is added at its sink and taken away at its source, and their roundings stay: what does not flow through t is left out here.
//   in t's block   sinks from t on of sources in earlier blocks, sources before t of sinks in later ones: nothing to take away
//   past the block sinks in later blocks of sources in earlier ones: a later block adds up its sinks before each earlier block's sources are
//                  added (`over`), the state's gradient takes sources block by block (`out_of`) and the state entering as <D, e_C h> (`through`)
//   pairs inside   both, over the half of the block that has fewer of them (to_middle).  A q with its own token's b and k passes no decay: dPqb
//                  and dPqk lose their diagonals, which go to dq, db and dk by themselves.
// dgk's error against fp64, 1e-7 of its 2-norm, with RWKV-7's decays, a hundredth of those, ten times those: 5.7, 4.4, 26 with sums over the
// block and <D, h'> less what does not pass, 4.6, 4.3, 5.0 (21 in the last chunk under a state's gradient) with the diagonals apart, 3.3,
// 3.6, 4.1 with `over` and `out_of`, 2.7, 3.6, 3.1 with to_middle, 2.4, 3.5, 2.9 as it is (mfma_block); dplr_grad 725, 714, 735, 750, 771 us.
template <typename T>
__global__ __launch_bounds__(256, 2) void dplr_grad_kernel(ChunkParams p) {
  extern __shared__ __align__(16) char smem[];
  const Lds L(smem);
  const Slot s = slot_of(p);
  const Lane w;
  const int l16 = w.l16, g4 = 4 * w.g;
  float *t0 = L.tile(0), *t1 = L.tile(1), *t2 = L.tile(2), *t3 = L.tile(3);
  float* through = L.sx;                             // [4][64] per channel: parts of <D, h>
  float* over = L.sx + 256;                          // [6][64]: row l (l - 1) / 2 + m has what flows into block l from before block m
  float* out_of = L.sx + 640;                        // [3][64]: from block j to D
  float *same_b = L.sx + 832, *same_k = L.sx + 896;  // [64]: the diagonals of dPqb and dPqk
  const int64_t at = (s.tok + w.t) * D + g4, wt = s.win * TG;
  const bool ok = w.t < s.len;
  Own<T> x;
  Row<T> v, d_o;
  Row<float> u, du;
  {
    Row<float> h0, dC;
    dC.load_tile(p.s1 + wt, w.j);
    x.load_gates(p, s, w);
    v.load(p.v, s, w);
    d_o.load(p.d_o, s, w);
    u.load_tile(p.s3 + wt, w.j);
    du.load_tile(p.s4 + wt, w.j);
    h0.load_tile(p.hT + s.st * TG, w.j);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {  // the wave's sixteen value columns
      const floatx4 y = sum_block(dC[cb] * h0[cb]);
      if (l16 == 0) store4(through + 64 * w.j + 16 * cb + g4, y);
    }
    put_given(t0, w, v);
    put_row(t2, w, [&](int cb) { return u[cb]; });
    put_row(t1, w, [&](int cb) { return h0[cb]; });  // states: [value column][channel]
    put_row(t3, w, [&](int cb) { return dC[cb]; });
  }
  Gates gates(x.gk);
  if (!gates.direct) {
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) put_total(L, w, cb, gates.upto(cb));
  } else {
    floatx4 y[4];
    token_decays(p, s, w, y);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) put_total(L, w, cb, product_upto(y[cb]));
  }
  if (threadIdx.x < 64) L.one[threadIdx.x] = 1.f;
  lds_barrier();
  floatx4 pb[3], pk[3], nb_[3], nk[3];          // dPqb, dPqk, dAab, dAak by t, with earlier blocks
  Pairs m{zero4(), zero4(), zero4(), zero4()};  // of the lane's own block
#pragma unroll
  for (int i = 0; i < 3; ++i) pb[i] = pk[i] = nb_[i] = nk[i] = zero4();
  auto pair_sums = [&](floatx4& qb, floatx4& qk, floatx4& ab, floatx4& ak, int row) {
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const floatx4 fu = frag<true>(t2, row, 16 * kb + g4), fo = d_o[kb], fd = du[kb];
      const Raw4<T> fv = given_row<T>(t0, row, 16 * kb + g4);
      if constexpr (sizeof(T) == 4) {
        mfma_block<4>({&qb, &qk, &ab, &ak}, [&](int i) { return i & 1 ? fv.x : fu; }, [&](int i) { return i & 2 ? fd : fo; });
      } else {  // dPqk's operands are both as given: one product for two blocks
        mfma_block<3>({&qb, &ab, &ak}, [&](int i) { return i == 2 ? fv.get() : fu; }, [&](int i) { return i ? fd : fo; });
        if (kb & 1) Mma16::mma(qk, Mma16::join(given_row<T>(t0, row, 16 * kb - 16 + g4).x, fv.x), Mma16::join(d_o.x[kb - (kb & 1)].x, d_o.x[kb].x));
      }
    }
  };
  before(w.j, [&](auto sb_) {
    constexpr int sb = decltype(sb_)::value;
    pair_sums(pb[sb], pk[sb], nb_[sb], nk[sb], 16 * sb + l16);
  });
  floatx4 dq[4], da[4];  // rows = channels, columns = tokens
  clear(dq), clear(da);
  float st[4];  // decays from the chunk's start to the lane's block, channels 16 cb + l16
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) st[cb] = L.start_to1(w.j, 16 * cb + l16);
  pair_sums(m.qb, m.qk, m.ab, m.ak, w.t);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const floatx4 fo = d_o[kb], fd = du[kb];
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const floatx4 hf = frag<false>(t1, 16 * cb + l16, 16 * kb + g4) * st[cb];
      mfma4(dq[cb], hf, fo);
      mfma4(da[cb], hf, fd);
    }
  }
  x.load_rows(p, s, w);  // not before: the registers are full up to here
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (g4 + r == l16) same_b[w.t] = m.qb[r], same_k[w.t] = m.qk[r];  // read by this wave alone, behind barriers
  mask<true, true>(m.qb, w), mask<true, true>(m.qk, w), mask<true, true>(m.ab, w), mask<true, true>(m.ak, w);
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) asm volatile("" : "+v"(gates.sum[cb][0]), "+v"(gates.sum[cb][1]), "+v"(gates.sum[cb][2]), "+v"(gates.sum[cb][3]));
  const Decay e(gates, p, s, w);  // formed here, not kept from the totals on: the registers are full in between
  lds_barrier();
  put_row(t0, w, [&](int cb) { return x.b[cb] * e.s[cb]; });
  put_row(t2, w, [&](int cb) { return x.k[cb] * e.s[cb]; });
  keep_as_read(x.b), keep_as_read(x.k);
  lds_barrier();
  before(w.j, [&](auto sb_) {
    constexpr int sb = decltype(sb_)::value;
    keep_as_read(x.q), keep_as_read(x.a);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const floatx4 y = sum_block(p.scale * x.q[cb] * e.p[cb] * dq[cb] + x.a[cb] * token_before(e.p[cb]) * da[cb]);
      if (l16 == 0) store4(over + 64 * (w.j * (w.j - 1) / 2 + sb) + 16 * cb + g4, y);
    }
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const float gap = L.from1<sb>(w.j, 16 * cb + l16);
      const floatx4 bf = frag<false>(t0, 16 * cb + l16, 16 * sb + g4) * gap, kf = frag<false>(t2, 16 * cb + l16, 16 * sb + g4) * gap;
      mfma4(dq[cb], bf, pb[sb]);
      mfma4(da[cb], bf, nb_[sb]);
      mfma4(dq[cb], kf, pk[sb]);
      mfma4(da[cb], kf, nk[sb]);
    }
  });
  float rt[4];  // 1 / decays of the whole block, channels 16 cb + l16: turns S of the block into 1 / P
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) rt[cb] = rcp_f(L.total[64 * w.j + 16 * cb + l16]);
  if (gates.direct) {
    float* own = t1 + w.t * LD;  // the state was last read before a barrier
    store4(own + g4, m.qb), store4(own + 16 + g4, m.qk), store4(own + 32 + g4, m.ab), store4(own + 48 + g4, m.ak);
    __builtin_amdgcn_wave_barrier();
  }
  const DirectRows<T> rows{p, s, w};
  floatx4 flow[4];  // dgk so far: of the q from the lane's token on and the a behind it
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const floatx4 pl = token_before(e.p[cb]), q = p.scale * x.q[cb];
    floatx4 dqo = zero4(), dao = zero4();  // of the block's own pairs
    if (!gates.direct) {
      const floatx4 bf = frag<false>(t0, 16 * cb + l16, 16 * w.j + g4) * rt[cb], kf = frag<false>(t2, 16 * cb + l16, 16 * w.j + g4) * rt[cb];
      mfma4(dqo, bf, m.qb);
      mfma4(dao, bf, m.ab);
      mfma4(dqo, kf, m.qk);
      mfma4(dao, kf, m.ak);
      dqo *= e.p[cb], dao *= pl;
    } else {
      direct_sinks<T>(rows, t1 + w.t * LD, 16 * cb + g4, dqo, dao);
    }
    dq[cb] *= e.p[cb], da[cb] *= pl;
    flow[cb] = sum_from(q * dq[cb] + dpp_move<0x101>(x.a[cb] * da[cb])) + (to_middle(q * dqo + x.a[cb] * dao) - x.a[cb] * dao);  // row_shl:1
    dq[cb] += dqo + (same_b[w.t] * x.b[cb] + same_k[w.t] * x.k[cb]), da[cb] += dao;
    if (ok) {
      store4(p.dgk + at + 16 * cb, flow[cb]);  // read back at the end
      store_row4<T>(p.dq, at + 16 * cb, dq[cb] * p.scale);
      store_row4<T>(p.da, at + 16 * cb, da[cb]);
    }
  }
  keep_as_read(x.b), keep_as_read(x.k), keep_as_read(x.q), keep_as_read(x.a);
  u.load_tile(p.s3 + wt, w.j), v.load(p.v, s, w);  // again, ahead of their use: in between the registers are full
  lds_barrier();
  // db, dk, relative to the end of the lane's block: the matrices with the contraction along t, first those of q, then those of a
  floatx4 db[4], dk[4], own[4];  // own: b db + k dk of the block's own pairs
  clear(db), clear(dk), clear(own);
  auto same = [](floatx4 y) { return y; };
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    if (half) lds_barrier();
    put_tri(t1, w, half ? nb_ : pb, half ? m.ab : m.qb, same), put_tri(t2, w, half ? nk : pk, half ? m.ak : m.qk, same);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) store4(t0 + w.t * LD + 16 * cb + g4, half ? x.a[cb] * token_before(e.p[cb]) : p.scale * x.q[cb] * e.p[cb]);
    lds_barrier();
    if (!half) {
      float en[4];
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) en[cb] = L.end_from1(w.j, 16 * cb + l16);
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const floatx4 fu = u[kb], fv = v[kb];
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
          const floatx4 df = frag<false>(t3, 16 * cb + l16, 16 * kb + g4) * en[cb];
          mfma4(db[cb], df, fu);
          mfma4(dk[cb], df, fv);
        }
      }
    }
    if (!half && w.j < 3) {
      keep_as_read(x.b), keep_as_read(x.k);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        const floatx4 y = sum_block((x.b[cb] * db[cb] + x.k[cb] * dk[cb]) * e.s[cb]);
        if (l16 == 0) store4(out_of + 64 * w.j + 16 * cb + g4, y);
      }
      keep_as_read(x.b), keep_as_read(x.k);
    }
    floatx4 dbh[4], dkh[4];  // apart from the other half's sums
    clear(dbh), clear(dkh);
    after(w.j, [&](auto tb_) {
      constexpr int tb = decltype(tb_)::value;
      const floatx4 mb = frag<false>(t1, w.t, 16 * tb + g4), mk = frag<false>(t2, w.t, 16 * tb + g4);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        const floatx4 xf = frag<false>(t0, 16 * cb + l16, 16 * tb + g4) * L.to1<tb>(w.j, 16 * cb + l16);
        mfma4(dbh[cb], xf, mb);
        mfma4(dkh[cb], xf, mk);
      }
    });
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) db[cb] += dbh[cb], dk[cb] += dkh[cb];
    if (!gates.direct) {
      const floatx4 mb = frag<false>(t1, w.t, 16 * w.j + g4), mk = frag<false>(t2, w.t, 16 * w.j + g4);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        const floatx4 xf = frag<false>(t0, 16 * cb + l16, 16 * w.j + g4) * rt[cb];
        floatx4 ob = zero4(), ok_ = zero4();
        mfma4(ob, xf, mb);
        mfma4(ok_, xf, mk);
        db[cb] += ob, dk[cb] += ok_;
        own[cb] += x.b[cb] * ob + x.k[cb] * ok_;
      }
    }
  }
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) db[cb] *= e.s[cb], dk[cb] *= e.s[cb], own[cb] *= e.s[cb];
  Row<float> fl;
  fl.load(p.dgk, ok ? at : 0);
  x.q.load(p.q, s, w);
  lds_barrier();
  if (gates.direct) {
    float* mine = t1 + w.t * LD;
    store4(mine + g4, m.qb), store4(mine + 16 + g4, m.qk), store4(mine + 32 + g4, m.ab), store4(mine + 48 + g4, m.ak);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      floatx4 ob = zero4(), ok_ = zero4();
      direct_sources<T>(rows, t1 + 16 * w.j * LD + l16, 16 * cb + g4, ob, ok_);
      db[cb] += ob, dk[cb] += ok_;
      own[cb] = x.b[cb] * ob + x.k[cb] * ok_;
    }
  }
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const floatx4 source = x.b[cb] * db[cb] + x.k[cb] * dk[cb] - own[cb], out = sum_upto(source);  // of later blocks' sinks
    flow[cb] = fl[cb] + (dpp_move<0x111>(out) - to_middle(own[cb]));  // row_shr:1
    const floatx4 q = p.scale * x.q[cb];
    db[cb] += same_b[w.t] * q, dk[cb] += same_k[w.t] * q;
    if (ok) {
      store_row4<T>(p.db, at + 16 * cb, db[cb]);
      store_row4<T>(p.dk, at + 16 * cb, dk[cb]);
    }
  }
  lds_barrier();
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const int c = 16 * cb + g4;
    floatx4 pass = (load4(through + c) + load4(through + 64 + c)) + (load4(through + 128 + c) + load4(through + 192 + c));
    pass *= load4(L.total + c) * load4(L.total + 64 + c) * (load4(L.total + 128 + c) * load4(L.total + 192 + c));
    for (int l = 3; l > w.j; --l) pass += load4(over + 64 * (l * (l - 1) / 2 + w.j) + c);
    for (int j = 0; j < w.j; ++j) pass += load4(out_of + 64 * j + c);
    if (ok) store4(p.dgk + at + 16 * cb, flow[cb] + pass);
  }
}

int64_t tiles(int64_t rows, int64_t n) { return rows * n * TG * (int64_t)sizeof(float); }

// Chunks of a window: the tensors that only live between the kernels of a call take at most 1 GiB (and a window at least
// eight chunks), whatever the sequence length.
int window(int64_t rows, int N, int per_chunk) {
  const int64_t w = (1ll << 30) / tiles(rows, per_chunk);
  return (int)(w < 8 ? (N < 8 ? N : 8) : w < N ? w : N);
}

int check_common(const lnx_dplr_args* a) {
  if (!a) return lnx_set_error(LNX_ERR_NULL, "args is NULL");
  if (!lnx_dplr_chunk_fits(a->B, a->H, a->T, a->dk, a->dv))
    return lnx_set_error(LNX_ERR_SHAPE, "dplr chunk kernels do not take B=%d H=%d T=%d dk=%d dv=%d", a->B, a->H, a->T, a->dk, a->dv);
  if ((a->dtype != LNX_F32 && a->dtype != LNX_BF16) || a->o_dtype != a->dtype) return lnx_set_error(LNX_ERR_DTYPE, "dplr chunk kernels: dtype %d, o_dtype %d", a->dtype, a->o_dtype);
  if (!a->q || !a->k || !a->v || !a->a || !a->b || !a->gk) return lnx_set_error(LNX_ERR_NULL, "q, k, v, a, b and gk are required");
  const void* ps[6] = {a->q, a->k, a->v, a->a, a->b, a->gk};
  for (const void* x : ps)
    if (reinterpret_cast<uintptr_t>(x) % 16) return lnx_set_error(LNX_ERR_SHAPE, "dplr chunk kernels: tensors must be 16-byte aligned");
  return LNX_OK;
}

ChunkParams params(const lnx_dplr_args* a) {
  ChunkParams p{};
  p.q = a->q, p.k = a->k, p.v = a->v, p.a = a->a, p.b = a->b, p.gk = a->gk, p.o = a->o;
  p.T = a->T, p.N = (a->T + C - 1) / C, p.scale = a->scale;
  return p;
}
void set_kept(ChunkParams& p, float* kept, int64_t rows, int k0, int KN) {
  const int64_t n = rows * KN * TG;
  p.M = kept, p.X = p.M + n, p.hT = p.X + n;
  p.k0 = k0, p.KN = KN;
}
constexpr int64_t kept_tiles(int64_t n) { return 3 * n + 1; }  // of a row that keeps n chunks

template <typename K> int lds_limit(K* k) { return lnx_lds_limit(reinterpret_cast<const void*>(k), LDS_BYTES); }

// B8 H16 T4096 bf16 (8192 chunks), us: dplr_prepare 447, dplr_chunk_scan 90, dplr_out 93 (48 KB of reads and 8 of writes per chunk: 5.0 TB/s)
template <typename T> int forward(const lnx_dplr_args* a, ChunkParams p, float* kept, float* scratch, hipStream_t st) {
  const int64_t rows = (int64_t)a->B * a->H;
  if (int rc = lds_limit(dplr_prepare_kernel<T>)) return rc;
  const int W = window(rows, p.N, kept ? 2 : 5);
  p.s1 = scratch, p.s2 = scratch + rows * W * TG;
  for (int n0 = 0; n0 < p.N; n0 += W) {
    p.n0 = n0, p.nw = p.N - n0 < W ? p.N - n0 : W;
    if (kept) set_kept(p, kept, rows, 0, p.N);
    else set_kept(p, scratch + 2 * rows * W * TG, rows, n0, p.nw);
    const unsigned grid = (unsigned)(rows * p.nw);
    lnx_profile_mark("dplr_prepare", st);
    hipLaunchKernelGGL(dplr_prepare_kernel<T>, dim3(grid), dim3(256), LDS_BYTES, st, p);
    lnx_profile_mark("dplr_chunk_scan", st);
    const ScanParams sp{p.M, p.s1, p.hT, n0 ? a->final_state : a->initial_state, a->final_state, rows, p.KN, n0 - p.k0, p.nw};
    hipLaunchKernelGGL(dplr_chunk_scan_kernel<false>, dim3(lnx_xcd_grid(rows, 4)), dim3(256), 0, st, sp);
    lnx_profile_mark("dplr_out", st);
    hipLaunchKernelGGL(dplr_out_kernel<T>, dim3(grid), dim3(256), 0, st, p);
  }
  return LNX_OK;
}

// Same shape: dplr_r 53, dplr_chunk_scan_bwd 88, dplr_u 441, dplr_grad 709 (two workgroups per CU leave 256 registers, and what a
// token needs between the pair sums and the last products is more: rows stay as they were read, and three are loaded twice)
template <typename T> int backward(const lnx_dplr_chunk_grads* g, const lnx_dplr_args* a, ChunkParams p, float* kept, float* scratch, hipStream_t st) {
  const int64_t rows = (int64_t)a->B * a->H;
  set_kept(p, kept, rows, 0, p.N);
  if (int rc = lds_limit(dplr_u_kernel<T>)) return rc;
  if (int rc = lds_limit(dplr_grad_kernel<T>)) return rc;
  const int W = window(rows, p.N, 4);
  const int64_t n = rows * W * TG;
  float* carry = scratch;  // the state's gradient between windows
  p.s1 = carry + rows * TG, p.s2 = p.s1 + n, p.s3 = p.s2 + n, p.s4 = p.s3 + n;
  p.d_o = g->d_o;
  p.dq = g->dq, p.dk = g->dk, p.dv = g->dv, p.da = g->da, p.db = g->db, p.dgk = g->dgk;
  const int nwin = (p.N + W - 1) / W;
  for (int i = nwin - 1; i >= 0; --i) {
    p.n0 = i * W, p.nw = p.N - p.n0 < W ? p.N - p.n0 : W;
    const unsigned grid = (unsigned)(rows * p.nw);
    lnx_profile_mark("dplr_r", st);
    hipLaunchKernelGGL(dplr_r_kernel<T>, dim3(grid), dim3(256), 0, st, p);
    lnx_profile_mark("dplr_chunk_scan_bwd", st);
    const ScanParams sp{p.M, p.s2, p.s1, i == nwin - 1 ? g->d_final_state : carry, i ? carry : g->d_initial_state, rows, p.KN, p.n0, p.nw};
    hipLaunchKernelGGL(dplr_chunk_scan_kernel<true>, dim3(lnx_xcd_grid(rows, 4)), dim3(256), 0, st, sp);
    lnx_profile_mark("dplr_u", st);
    hipLaunchKernelGGL(dplr_u_kernel<T>, dim3(grid), dim3(256), LDS_BYTES, st, p);
    lnx_profile_mark("dplr_grad", st);
    hipLaunchKernelGGL(dplr_grad_kernel<T>, dim3(grid), dim3(256), LDS_BYTES, st, p);
  }
  return LNX_OK;
}

int finish(int rc, hipStream_t st) {
  lnx_profile_mark(nullptr, st);
  if (rc != LNX_OK) return rc;
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? LNX_OK : lnx_set_error(LNX_ERR_LAUNCH, "dplr chunk kernel launch: %s", hipGetErrorString(e));
}

}  // namespace

extern "C" int lnx_dplr_chunk_fits(int32_t B, int32_t H, int32_t T, int32_t dk, int32_t dv) {
  return B > 0 && H > 0 && dk == D && dv == D && T >= 16 && (int64_t)B * H * ((T + C - 1) / C) < (1ll << 31);
}

extern "C" uint64_t lnx_dplr_chunk_bytes(int32_t B, int32_t H, int32_t T, int32_t what) {
  if (B <= 0 || H <= 0 || T <= 0) return 0;
  const int64_t rows = (int64_t)B * H;
  const int N = (T + C - 1) / C;
  switch (what) {
    case LNX_DPLR_KEPT: return (uint64_t)tiles(rows, kept_tiles(N));
    case LNX_DPLR_ONLY_SCRATCH: return (uint64_t)tiles(rows, 2 * (int64_t)window(rows, N, 5) + kept_tiles(window(rows, N, 5)));
    case LNX_DPLR_FWD_SCRATCH: return (uint64_t)tiles(rows, 2 * (int64_t)window(rows, N, 2));
    case LNX_DPLR_BWD_SCRATCH: return (uint64_t)tiles(rows, 4 * (int64_t)window(rows, N, 4) + 1);
    default: return 0;
  }
}

extern "C" int lnx_dplr_chunk_fwd(const lnx_dplr_args* a, void* kept, void* scratch, void* hip_stream) {
  if (int rc = check_common(a)) return rc;
  if (!a->o || !a->final_state || !scratch) return lnx_set_error(LNX_ERR_NULL, "o, final_state and the scratch area are required");
  hipStream_t st = static_cast<hipStream_t>(hip_stream);
  const ChunkParams p = params(a);
  float *kp = static_cast<float*>(kept), *sc = static_cast<float*>(scratch);
  return finish(a->dtype == LNX_BF16 ? forward<bf16_t>(a, p, kp, sc, st) : forward<float>(a, p, kp, sc, st), st);
}

extern "C" int lnx_dplr_chunk_bwd(const lnx_dplr_args* a, const lnx_dplr_chunk_grads* g, void* kept, void* scratch, void* hip_stream) {
  if (int rc = check_common(a)) return rc;
  if (!g || !g->d_o || !g->dq || !g->dk || !g->dv || !g->da || !g->db || !g->dgk || !kept || !scratch)
    return lnx_set_error(LNX_ERR_NULL, "d_o, the six token gradients and the two work areas are required");
  hipStream_t st = static_cast<hipStream_t>(hip_stream);
  const ChunkParams p = params(a);
  float *kp = static_cast<float*>(kept), *sc = static_cast<float*>(scratch);
  return finish(a->dtype == LNX_BF16 ? backward<bf16_t>(g, a, p, kp, sc, st) : backward<float>(g, a, p, kp, sc, st), st);
}
