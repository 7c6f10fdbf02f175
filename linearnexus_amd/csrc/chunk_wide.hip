// The two sequential passes of the direct-solve split (chunk_direct.hip has the algebra) for 2-byte inputs with dk = 256 and no / a
// scalar gate (the head shape of the Gated DeltaNet presets):
//
//   forward   Y = K S    R = diag(beta) (V - diag(e^G) Y)    D = Tm R    O = scale diag(e^G) (Q S) + Pm D
//             S' = e^{G_C} S + (diag(e^{G_C - G}) K)^T D
//   reverse   dD = Pm^T dO + diag(e^{G_C - G}) K dS'    dR = Tm^T dD    dv = diag(beta) dR    dY = -diag(beta e^G) dR
//             dS = e^{G_C} dS' + (scale diag(e^G) Q)^T dO + K^T dY
//
// What bounds them: with dk = 256 a chunk's K and Q rows are 64 KB, which every workgroup of a (state, head) loads again for
// its slab of value columns.  So a slab is as wide as the registers allow: a compute wave owns 16 NC value
// columns, whose [256 x 16 NC] part of the state stays in accumulators for the whole sequence and is the operand of the next
// products as it stands (a column of tiles as Mma16 describes, in natural order); only K, Q, Tm and Pm come from LDS.  The state also
// leaves from there: an operand fragment is 16 bytes of a row of the saved tensor.  Four mover waves hold the next chunk
// in registers.  Per chunk:
//   B1   tiles of chunk n in LDS               compute: everything but the last product     movers: loads of the next chunk
//   B2   its K is left                         compute: the last product    movers: results -> global, the other tiles -> LDS
//   B3                                         compute: state -> global     movers: K -> LDS
// Slabs of 32 and 64 columns are taken where a chunk's chain is what a call waits for.  Their compute waves leave registers and LDS for more:
// the movers hold two chunks, so that rows which the op normalises are converted ahead of B2 without waiting for memory, and K has two tiles
// and no barrier of its own (AHEAD):
//   B1   compute: everything but the last product     movers: loads of chunk n + 2; of chunk n + 1 Q (in reverse behind B2) and K converted, K -> LDS
//   B2   compute: the last product, state -> global   movers: results -> global, the other tiles -> LDS
// With one chunk held and converted where it is stored, between the barriers, 4 heads dv 256 of 8192 tokens took 418 us forward only and 849
// with gradients, more than the WY split's kernels (360 and 769, the normalisation ahead of them); so 331 and 743.  The movers' loads and
// conversions in turn, a tile at a time, and Q's conversion behind B2 in reverse are 366 -> 349 and 368 -> 326 us of the scans.
// Measured at B8 H8 T4096 dv512 (128-column slabs, 256 workgroups): forward 498 - 510 us, reverse 448 - 459 us by box, 7.9 and 7.1 us a chunk, of which
// 185 KB through the CU's memory path (64 KB of state per chunk and slab leave for the backward kernels) are most.  The WY split's
// passes, which read W and U instead of Tm and V, took 521 and 435 us behind 205 us of preparation (now 68) and 221 us of normalisation
// outside the kernels (now none), and before two more kernels of 804 and 289 us (now one of 788 - 795): the step 2478 -> 1830 us.
// State stores among the products of the first phase instead of
// behind the last barrier: 551 -> 587 and 464 -> 521 us (a wave whose store waits for a slot multiplies nothing).

#include <type_traits>

#include "chunk_common.h"

namespace {

using T = bf16_t;
typedef Mma16 S16;
typedef S16::Frag Frag;
constexpr int DK = 256, KT = DK / 16, NK = DK / 32;
template <typename X> __device__ __forceinline__ X* at(char* ws, uint64_t off) { return reinterpret_cast<X*>(ws + off); }

// Natural order: group g of a step of 32 holds the contraction indices 8 g .. 8 g + 7 (the sums of two 32 x 32 x 16 products from
// row-major operands).  Tile i of a column of accumulator tiles covers the rows  row0(i) + grp + r, so tiles 2 s and 2 s + 1 are
// the operand of step s.  The rows of LDS tiles lie such that a tile's sixteen rows are consecutive.
__device__ __forceinline__ int row0(int i) { return 32 * (i >> 1) + 4 * (i & 1); }
__device__ __forceinline__ int grp(int lane) { return 8 * ((lane >> 4) & 3); }
__device__ __forceinline__ int row_of(int lane) { return 8 * ((lane >> 2) & 3) + (lane & 3); }
__device__ __forceinline__ int place(int r) { return (r & 32) + 16 * ((r >> 2) & 1) + 4 * ((r >> 3) & 3) + (r & 3); }
// operand rows of tile i, step ks
__device__ __forceinline__ Frag load_rows(const T* tile, int ld, int i, int ks, int lane) {
  return *reinterpret_cast<const bf16x8*>(tile + (16 * i + (lane & 15)) * ld + 32 * ks + 8 * (lane >> 4));
}
// operand from the columns of tile ci, contraction along rows 32 s ..
__device__ __forceinline__ Frag load_cols(const T* tile, int ld, int s, int ci, int lane) {
  const int q = lane & 15;
  const T* p = tile + (32 * s + 4 * (lane >> 4) + (q >> 2)) * ld + 32 * (ci >> 1) + 8 * (q & 3) + 4 * (ci & 1);
  return S16::join(__builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((S16::lds_short4*)(p))),
                   __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((S16::lds_short4*)(p + 16 * ld))));
}
template <int NC, int NCW> struct WideL {
  static constexpr int BV = 16 * NC * NCW, LDK = DK + 16, LDC = LNX_C + 16, LDV = BV + 8, LDT = LNX_C + 8;
  static constexpr int kRow = 64 * LDK, kC = 64 * LDC, kV = 64 * LDV, kT = BV * LDT;
  static constexpr bool AHEAD = NC == 1;  // the movers hold two chunks, and LDS two K tiles
  static constexpr int NK2 = AHEAD ? 2 : 1;
  // K [NK2] | Q | Tm | Pm | V (reverse: dO) | O (reverse: dv) on its way out | D^T (reverse: dR^T) on its way out | scalars
  static constexpr size_t bytes = sizeof(T) * ((NK2 + 1) * kRow + 2 * kC + 2 * kV + kT) + sizeof(float) * 272;
  static constexpr int threads = 64 * NCW + 256;
  static_assert(bytes <= 160 * 1024, "LDS");
};
struct Sc {
  enum { R = 0, Q = 64, BETA = 128, GAM = 192, DEC = 256 };  // e^{G_C - G}, scale e^G, beta, beta e^G, e^{G_C}
};

// Tm or Pm, lower-triangular and packed in the workspace, between its loads and its LDS stores: 288 vectors for 256 threads, rows at
// their places.  The vectors above the diagonal are zeroed once ...
struct PlacedTri {
  bf16x8 x[2];
  int o[2];
  bool second;
  __device__ __forceinline__ void init(int ld, int tid) {
    second = tid < LNX_TRI_VECS - 256;
    int r, c;
    tri_vec_pos(tid, r, c);
    o[0] = place(r) * ld + 8 * c;
    tri_vec_pos(second ? 256 + tid : 0, r, c);
    o[1] = place(r) * ld + 8 * c;
  }
  __device__ __forceinline__ void load(const T* src, int tid) {  // threads without a second vector read past the end: zeros
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(src), 0, LNX_TRI_VECS * 16, 0x00020000);
#pragma unroll
    for (int u = 0; u < 2; ++u) x[u] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rsrc, 16 * (256 * u + tid), 0, 0));
  }
  __device__ __forceinline__ void store(T* dst) const {
    *reinterpret_cast<bf16x8*>(dst + o[0]) = x[0];
    if (second) *reinterpret_cast<bf16x8*>(dst + o[1]) = x[1];
  }
};
// ... of both, one behind the other
__device__ __forceinline__ void zero_upper(T* tiles, int ld, int stride, int tid) {
  if (tid >= 512 - LNX_TRI_VECS) return;
  int r, c;
  upper_vec_pos(tid, r, c);
#pragma unroll
  for (int t = 0; t < 2; ++t) *reinterpret_cast<bf16x8*>(tiles + t * stride + place(r) * ld + 8 * c) = vec_zero<T>();
}
// Row factors of a [64][DK] tile (1 / (|x| + eps) where the op normalises), and the tile's rows times them.  A thread's vectors lie in eight
// rows: it loads their factors, or where two chunks in flight leave the memory counter no room for that (LANES) that of row `lane`, and takes
// the wave's two rows of every eight out of the lanes (128-column slabs, forward only, 202 us with the loads, 206 so).
template <bool LANES> struct RowFactors {
  static constexpr int IT = 64 * DK / 8 / 256;
  float f[LANES ? 1 : IT];
  __device__ __forceinline__ void load(const float* src, int tid) {
#pragma unroll
    for (int it = 0; it < (LANES ? 1 : IT); ++it) f[it] = src[LANES ? tid & 63 : (tid + 256 * it) / (DK / 8)];
  }
  __device__ __forceinline__ float of(int it, int tid) const {
    if constexpr (!LANES) return f[it];
    const int r = 2 * __builtin_amdgcn_readfirstlane(tid >> 6) + 8 * it, x = __float_as_int(f[0]);
    const int lo = __builtin_amdgcn_readlane(x, r), hi = __builtin_amdgcn_readlane(x, r + 1);
    return __int_as_float(tid & 32 ? hi : lo);
  }
};
template <bool LANES> __device__ __forceinline__ void scale_rows(TileRegs<T, 64, DK>& R, const RowFactors<LANES>& F, int tid) {
#pragma unroll
  for (int it = 0; it < TileRegs<T, 64, DK>::IT; ++it) {
    const float f = F.of(it, tid);
#pragma unroll
    for (int e = 0; e < 8; ++e) R.x[it][e] = (bf16_t)((float)R.x[it][e] * f);
  }
}
__device__ __forceinline__ void store_rows(const TileRegs<T, 64, DK>& R, T* dst, int ld, int tid) {
#pragma unroll
  for (int it = 0; it < TileRegs<T, 64, DK>::IT; ++it) {
    const int idx = tid + 256 * it, r = idx / (DK / 8), c = (idx - r * (DK / 8)) * 8;
    *reinterpret_cast<bf16x8*>(dst + place(r) * ld + c) = R.x[it];
  }
}
// What the movers read per chunk besides the row and value tiles
template <int GATE> struct Scalars {
  float g = 0.f, gl = 0.f, b = 0.f;
  __device__ __forceinline__ void load(const DirectParams& p, int64_t slot, int64_t tbase, int len, int mt) {
    const int t = mt & 63;
    if (GATE == LNX_GATE_SCALAR) {
      const float* G = at<const float>(p.ws, p.off.G) + slot * 64;
      g = G[t];
      gl = G[63];
    }
    b = p.beta[tbase + (int64_t)min(t, len - 1) * p.geom.ts];
    if (t >= len) b = 0.f;
  }
  __device__ __forceinline__ void put(float* sc, float scale, int mt) const {  // by the first 64 movers
    if (mt >= 64) return;
    const float eg = (GATE == LNX_GATE_SCALAR) ? __expf(g) : 1.f;
    sc[Sc::R + mt] = (GATE == LNX_GATE_SCALAR) ? __expf(fminf(gl - g, 0.f)) : 1.f;
    sc[Sc::Q + mt] = scale * eg;
    sc[Sc::BETA + mt] = b;
    sc[Sc::GAM + mt] = b * eg;
    if (mt == 0) sc[Sc::DEC] = (GATE == LNX_GATE_SCALAR) ? __expf(gl) : 1.f;
  }
};

struct Chain {
  int sidx, row, seq, v0, c0, c1;
  SeqSpan span;
};
template <int BV> __device__ __forceinline__ bool chain_of(const DirectParams& p, Chain& c) {
  int64_t chain;
  int slab;
  if (!xcd_slot_part((int64_t)(p.geom.tab ? p.geom.nseq : p.geom.rows / p.geom.H) * p.geom.H, p.dv / BV, chain, slab)) return false;
  scan_state(p.geom, (int)chain, c.sidx, c.row, c.seq);
  c.v0 = slab * BV;
  seq_chunks(p.geom, c.seq, c.c0, c.c1);
  c.span = seq_span(p.geom, c.seq, c.c0);
  return true;
}

// The strip's state: column l16 of column tile c, rows by tiles.
template <int NC> struct Strip {
  floatx4 x[NC][KT];
  __device__ __forceinline__ void load(const float* src, int dv, int lane) {  // src at the strip's first column, or NULL
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int ci = 0; ci < KT; ++ci)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[c][ci][e] = 0.f;
    if (!src) return;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int ci = 0; ci < KT; ++ci)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[c][ci][e] = src[(int64_t)(row0(ci) + grp(lane) + e) * dv + 16 * c + (lane & 15)];
    // the loads complete here: left pending into the loop, every iteration would count them down again
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int ci = 0; ci < KT; ++ci)
#pragma unroll
        for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(x[c][ci][e]));
  }
  __device__ __forceinline__ void identity(int first, int lane) {  // of the columns from `first` on, the strip's first one
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int ci = 0; ci < KT; ++ci)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[c][ci][e] = row0(ci) + grp(lane) + e == first + 16 * c + (lane & 15) ? 1.f : 0.f;
  }
  __device__ __forceinline__ void store(float* dst, int dv, int lane) const {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int ci = 0; ci < KT; ++ci)
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[(int64_t)(row0(ci) + grp(lane) + e) * dv + 16 * c + (lane & 15)] = x[c][ci][e];
  }
  // What is formed of the state is formed again behind this: operands kept from one product for the next were 64 registers, which went to
  // scratch memory
  __device__ __forceinline__ void settle() {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int ci = 0; ci < KT; ++ci) asm volatile("" : "+v"(x[c][ci]));
  }
  __device__ __forceinline__ Frag operand(int c, int ks) const { return S16::from_acc(x[c][2 * ks], x[c][2 * ks + 1]); }
  __device__ __forceinline__ void save(T* dst, int lane) const {  // [value column][dk] of the strip
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) *reinterpret_cast<bf16x8*>(dst + (16 * c + (lane & 15)) * DK + 32 * ks + 8 * (lane >> 4)) = operand(c, ks);
  }
  // LDS reads go out two groups of products ahead (R rows of operands at a time) where a wave has two column tiles: left to the compiler they went
  // out in front of the products that take them, 7950 cycles a chunk until D and O are there, 5900 so (2430 of products).  B8 H8 T4096 dv = 512
  // forward scan 506 -> 452 us (5.1 TB/s of what HBM carries a chunk), nothing saved 375 -> 317.  With one column tile the compiler's order is as
  // fast in reverse and 1 % faster forward.
  static constexpr bool PIPED = NC == 2;
  // x = f x + tile^T b: rows of the tile (tokens) contracted
  template <bool SCALED> __device__ __forceinline__ void add(const T* tile, int ld, const Frag (&b)[NC][2], int lane, float f = 1.f) {
    if constexpr (!PIPED) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int ci = 0; ci < KT; ++ci)
          if (SCALED) x[c][ci] *= f;
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int ci = 0; ci < KT; ++ci) {
          const Frag a = load_cols(tile, ld, s, ci, lane);
#pragma unroll
          for (int c = 0; c < NC; ++c) S16::mma(x[c][ci], a, b[c][s]);
        }
    } else {
      constexpr int NG = 2 * KT / 4;
      Frag a[3][4];
      auto load = [&](int g) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 4; ++j) a[g % 3][j] = load_cols(tile, ld, 4 * g / KT, (4 * g) % KT + j, lane);
      };
      load(0), load(1);
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if (g + 2 < NG) load(g + 2);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            floatx4& y = x[c][(4 * g) % KT + j];
            if (SCALED && 4 * g < KT) y *= f;
            S16::mma(y, a[g % 3][j], b[c][4 * g / KT]);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  // y[c][i] += rows of tile i0 + i (tokens) times x, or the other way round (COLS: columns = tokens)
  template <int NI, bool COLS> __device__ __forceinline__ void rows_times(floatx4 (&y)[NC][NI], const T* tile, int ld, int i0, int lane) const {
    constexpr int AHEAD = PIPED ? (NI == 4 ? 2 : 3) : 0;
    Frag a[AHEAD + 1][NI];
    auto load = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NI; ++i) a[ks % (AHEAD + 1)][i] = load_rows(tile, ld, i0 + i, ks, lane);
    };
#pragma unroll
    for (int ks = 0; ks < AHEAD; ++ks) load(ks);
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      if (PIPED && ks + AHEAD < NK) load(ks + AHEAD);
      Frag b[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) b[c] = operand(c, ks);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if (!PIPED) a[0][i] = load_rows(tile, ld, i0 + i, ks, lane);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          if (COLS) S16::mma(y[c][i], b[c], a[ks % (AHEAD + 1)][i]);
          else S16::mma(y[c][i], a[ks % (AHEAD + 1)][i], b[c]);
        }
      }
      if (PIPED) __builtin_amdgcn_sched_barrier(0);
    }
  }
};

// D (dR) of a column tile as operands, transposed to LDS: 16 bytes are eight tokens of a value column
__device__ __forceinline__ void put_t(T* sT, int ld, int col, const Frag (&b)[2], int lane) {
#pragma unroll
  for (int s = 0; s < 2; ++s) *reinterpret_cast<bf16x8*>(sT + (col + (lane & 15)) * ld + 32 * s + grp(lane)) = b[s];
}

template <int GATE, int NC, int NCW, typename OT>
__global__ __launch_bounds__((WideL<NC, NCW>::threads)) void wide_scan_fwd_kernel(DirectParams p) {
  typedef WideL<NC, NCW> L;
  constexpr bool OUT = !std::is_void<OT>::value;  // void: final states alone (forward only): no Q, no Pm, nothing saved
  constexpr int BV = L::BV, LDK = L::LDK, LDC = L::LDC, LDV = L::LDV, LDT = L::LDT;
  extern __shared__ __align__(16) char smem[];
  T* sK = reinterpret_cast<T*>(smem);
  T* sQ = sK + L::NK2 * L::kRow;
  T* sTm = sQ + L::kRow;
  T* sP = sTm + L::kC;
  T* sV = sP + L::kC;
  T* sO = sV + L::kV;
  T* sDT = sO + L::kV;
  float* sc = reinterpret_cast<float*>(sDT + L::kT);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  Chain ch;
  if (!chain_of<BV>(p, ch)) return;
  auto k_tile = [&](int n) { return sK + (L::AHEAD ? (n & 1) * L::kRow : 0); };
  const int N = p.geom.N, c0 = ch.c0, c1 = ch.c1, v0 = ch.v0;
  const int64_t tso = (int64_t)p.geom.ts * p.dv;

  if (wave >= NCW) {
    // ---------------- movers ----------------
    const int mt = tid - 64 * NCW;
    struct Chunk {
      TileRegs<T, 64, DK> K, Q;
      TileRegs<T, 64, BV> V;
      PlacedTri Tm, P;
      RowFactors<L::AHEAD> fk, fq;
      Scalars<GATE> sc;
    };
    Chunk a, b;
    a.Tm.init(LDC, mt), a.P.init(LDC, mt), b.Tm.init(LDC, mt), b.P.init(LDC, mt);
    zero_upper(sTm, LDC, L::kC, mt);
    const int64_t tsk = (int64_t)p.geom.ts * DK, tsv = (int64_t)p.geom.ts * p.vcols;
    // part 0: Q, 1: K, 2: the rest; < 0: everything.  Unconditional, as the commits: a load behind a branch cannot be counted
    auto fetch = [&](Chunk& R, int n, int part = -1) __attribute__((always_inline)) {
      n = min(n, c1 - 1);
      const int64_t slot = (int64_t)ch.row * N + n;
      int tok0, len;
      chunk_span(ch.span, n, tok0, len);
      const int64_t tbase = tok_index(p.geom, ch.row, tok0);
      if (OUT && (part < 0 || part == 0)) {
        R.Q.load(p.q + tbase * DK, tsk, len, mt);
        R.fq.load(at<const float>(p.ws, p.off.Nq) + slot * 64, mt);
      }
      if (part < 0 || part == 2) {
        R.V.load(p.v + tbase * p.vcols + v0, tsv, (v0 < p.vcols) ? len : 0, mt);  // columns v does not hold read as zero
        R.Tm.load(at<const T>(p.ws, p.off.Tm) + slot * 64 * 64, mt);
        if (OUT) R.P.load(at<const T>(p.ws, p.off.P) + slot * 64 * 64, mt);
        R.sc.load(p, slot, tbase, len, mt);
      }
      if (part < 0 || part == 1) {
        R.K.load(p.k + tbase * DK, tsk, len, mt);
        R.fk.load(at<const float>(p.ws, p.off.Nk) + slot * 64, mt);
      }
    };
    auto normalise = [&](Chunk& R, int part = -1) __attribute__((always_inline)) {
      if (OUT && p.l2norm && part != 1) scale_rows(R.Q, R.fq, mt);
      if (p.l2norm && part != 0) scale_rows(R.K, R.fk, mt);
    };
    auto commit = [&](const Chunk& R) __attribute__((always_inline)) {
      if constexpr (OUT) store_rows(R.Q, sQ, LDK, mt);
      R.V.store(sV, LDV, mt);
      R.Tm.store(sTm);
      if constexpr (OUT) R.P.store(sP);
      R.sc.put(sc, p.scale, mt);
    };
    auto commit_k = [&](const Chunk& R, int n) __attribute__((always_inline)) { store_rows(R.K, k_tile(n), LDK, mt); };
    // cur, whose chunk n is in LDS, takes chunk n + 2, a tile at a time between the conversions of nxt, which holds chunk n + 1 since the step
    // before.  Without AHEAD the same registers take chunk n + 1.
    auto step = [&](Chunk& cur, Chunk& nxt, int n) __attribute__((always_inline)) {
      if constexpr (L::AHEAD) {
        fetch(cur, n + 2, 2);
        __builtin_amdgcn_sched_barrier(0);
        normalise(nxt, 0);
        __builtin_amdgcn_sched_barrier(0);
        fetch(cur, n + 2, 0);
        __builtin_amdgcn_sched_barrier(0);
        normalise(nxt, 1);
        commit_k(nxt, n + 1);
        __builtin_amdgcn_sched_barrier(0);
        fetch(cur, n + 2, 1);
      } else {
        fetch(cur, n + 1);
      }
      lds_barrier();  // B2
      const int64_t slot = (int64_t)ch.row * N + n;
      int tok0, len;
      chunk_span(ch.span, n, tok0, len);
      if (std::is_same<OT, T>::value && p.o)
        unstage_tile_checked<T, 64, BV>(reinterpret_cast<T*>(p.o) + tok_index(p.geom, ch.row, tok0) * p.dv + v0, tso, sO, LDV, len, mt);
      if (OUT && p.save) unstage_tile<T, BV, 64, true>(at<T>(p.ws, p.off.D) + slot * p.dv * 64 + (int64_t)v0 * 64, 64, sDT, LDT, BV, mt);
      if (!L::AHEAD) normalise(nxt, 0);
      commit(nxt);
      if (!L::AHEAD) {
        lds_barrier();  // B3
        normalise(nxt, 1);
        commit_k(nxt, n + 1);
      }
      lds_barrier();  // B1 of the next chunk
    };
    if (c0 < c1) {
      fetch(a, c0);
      if (L::AHEAD) fetch(b, c0 + 1);
      normalise(a);
      commit(a);
      commit_k(a, c0);
    }
    lds_barrier();  // B1 of the first chunk
    if constexpr (L::AHEAD) {
      for (int n = c0; n < c1;) {  // ways out lead out of the loop: they do not join the count of loads in flight
        step(a, b, n);
        if (++n >= c1) break;
        step(b, a, n++);
      }
    } else {
      for (int n = c0; n < c1; ++n) step(a, a, n);
    }
    return;
  }

  // ---------------- compute waves: wave w owns value columns [16 NC w, 16 NC (w + 1)) of the slab ----------------
  const int vs = 16 * NC * wave;
  Strip<NC> S;
  if (!OUT && p.ident) S.identity(v0 + vs - p.vcols, lane);
  else S.load(p.s0 ? p.s0 + (int64_t)ch.sidx * DK * p.dv + v0 + vs : nullptr, p.dv, lane);
  auto save = [&](int n) {
    if (OUT && p.save) S.save(at<T>(p.ws, p.off.SnT) + ((int64_t)ch.row * N + n) * p.dv * DK + (int64_t)(v0 + vs) * DK, fresh(tid & 63));
  };
  if (c0 < c1) save(c0);
  lds_barrier();  // B1 of the first chunk
  for (int n = c0; n < c1; ++n) {
    const int lane = fresh(tid & 63), g8 = grp(lane);
    // ---- Y = K S: rows = tokens ----
    floatx4 y[NC][4];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) y[c][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    S.template rows_times<4, false>(y, k_tile(n), LDK, 0, lane);
    __builtin_amdgcn_sched_barrier(0);
    // ---- R = beta V - beta e^G Y, in place of Y ----
    Frag br[NC][2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 2 * s; i < 2 * s + 2; ++i) {
        const floatx4 bt = load4(sc + Sc::BETA + row0(i) + g8), gm = load4(sc + Sc::GAM + row0(i) + g8);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const bf16x4 u = S16::rows4(sV, LDV, row0(i) + g8, vs + 16 * c, lane);
          y[c][i] = bt * floatx4{(float)u[0], (float)u[1], (float)u[2], (float)u[3]} - gm * y[c][i];
        }
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) br[c][s] = S16::from_acc(y[c][2 * s], y[c][2 * s + 1]);
    }
    // ---- D = Tm R (Tm is lower-triangular: the first 32 tokens take the first step only) ----
    Frag bd[NC][2], bu[NC][2];  // D, and D with its rows scaled by e^{G_C - G}, as operands
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x4 d0[NC], u0[NC];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int i = 2 * s + h;
        floatx4 d[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) d[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k <= s; ++k) {
          const Frag f = load_rows(sTm, LDC, i, k, lane);
#pragma unroll
          for (int c = 0; c < NC; ++c) S16::mma(d[c], f, br[c][k]);
        }
        const floatx4 r = load4(sc + Sc::R + row0(i) + g8);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const bf16x4 x = pack_bf16x4(d[c]), u = pack_bf16x4(d[c] * r);
          if (h == 0) d0[c] = x, u0[c] = u;
          else bd[c][s] = S16::join(d0[c], x), bu[c][s] = S16::join(u0[c], u);
        }
      }
    }
#pragma unroll
    for (int c = 0; c < (OUT ? NC : 0); ++c) put_t(sDT, LDT, vs + 16 * c, bd[c], lane);
    __builtin_amdgcn_sched_barrier(0);
    // ---- O^T = scale e^G (Q S)^T + D^T Pm^T: columns = tokens, 32 of them at a time ----
#pragma unroll
    for (int h = 0; h < (OUT ? 2 : 0); ++h) {
      const int lane = fresh(tid & 63);
      floatx4 o[NC][2];
#pragma unroll
      for (int c = 0; c < NC; ++c) o[c][0] = o[c][1] = floatx4{0.f, 0.f, 0.f, 0.f};
      if (S.PIPED) S.settle();
      S.template rows_times<2, true>(o, sQ, LDK, 2 * h, lane);
      int tok0, len;
      chunk_span(ch.span, n, tok0, len);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int t = row0(2 * h + i) + row_of(lane);
        const float f = sc[Sc::Q + t];
#pragma unroll
        for (int c = 0; c < NC; ++c) o[c][i] *= f;
#pragma unroll
        for (int k = 0; k <= h; ++k) {  // Pm is lower-triangular, too
          const Frag f = load_rows(sP, LDC, 2 * h + i, k, lane);
#pragma unroll
          for (int c = 0; c < NC; ++c) S16::mma(o[c][i], bd[c][k], f);
        }
        if constexpr (std::is_same<OT, T>::value) {
#pragma unroll
          for (int c = 0; c < NC; ++c) store4(sO + t * LDV + vs + 16 * c + 4 * (lane >> 4), o[c][i]);
        } else if constexpr (OUT) {
          if (p.o && t < len) {
#pragma unroll
            for (int c = 0; c < NC; ++c)
              store4(reinterpret_cast<float*>(p.o) + (tok_index(p.geom, ch.row, tok0) + (int64_t)t * p.geom.ts) * p.dv + v0 + vs + 16 * c + 4 * (lane >> 4), o[c][i]);
          }
        }
      }
    }
    const float dec = sc[Sc::DEC];
    lds_barrier();  // B2
    S.template add<GATE == LNX_GATE_SCALAR>(k_tile(n), LDK, bu, fresh(tid & 63), dec);
    if (!L::AHEAD) lds_barrier();  // B3
    if (n + 1 < c1) save(n + 1);
    lds_barrier();  // B1 of the next chunk
  }
  S.store(p.sT_out.at(ch.sidx, (int64_t)DK * p.dv) + v0 + vs, p.dv, fresh(tid & 63));
}

template <int GATE, int NC, int NCW>
__global__ __launch_bounds__((WideL<NC, NCW>::threads)) void wide_scan_bwd_kernel(DirectParams p) {
  typedef WideL<NC, NCW> L;
  constexpr int BV = L::BV, LDK = L::LDK, LDC = L::LDC, LDV = L::LDV, LDT = L::LDT;
  extern __shared__ __align__(16) char smem[];
  T* sK = reinterpret_cast<T*>(smem);
  T* sQ = sK + L::NK2 * L::kRow;
  T* sTm = sQ + L::kRow;
  T* sP = sTm + L::kC;
  T* sdO = sP + L::kC;
  T* sdV = sdO + L::kV;
  T* sdRT = sdV + L::kV;
  float* sc = reinterpret_cast<float*>(sdRT + L::kT);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  Chain ch;
  if (!chain_of<BV>(p, ch)) return;
  auto k_tile = [&](int n) { return sK + (L::AHEAD ? (n & 1) * L::kRow : 0); };
  const int N = p.geom.N, c0 = ch.c0, c1 = ch.c1, v0 = ch.v0;

  if (wave >= NCW) {
    // ---------------- movers ----------------
    const int mt = tid - 64 * NCW;
    struct Chunk {
      TileRegs<T, 64, DK> K, Q;
      TileRegs<T, 64, BV> dO;
      PlacedTri Tm, P;
      RowFactors<L::AHEAD> fk, fq;
      Scalars<GATE> sc;
    };
    Chunk a, b;
    a.Tm.init(LDC, mt), a.P.init(LDC, mt), b.Tm.init(LDC, mt), b.P.init(LDC, mt);
    zero_upper(sTm, LDC, L::kC, mt);
    const int64_t tsk = (int64_t)p.geom.ts * DK, tsv = (int64_t)p.geom.ts * p.dv;
    auto fetch = [&](Chunk& R, int n, int part = -1) __attribute__((always_inline)) {  // part 0: Q, 1: K, 2: the rest; < 0: everything
      n = max(n, c0);
      const int64_t slot = (int64_t)ch.row * N + n;
      int tok0, len;
      chunk_span(ch.span, n, tok0, len);
      const int64_t tbase = tok_index(p.geom, ch.row, tok0);
      if (part < 0 || part == 2) {
        R.dO.load(p.d_o + tbase * p.dv + v0, tsv, len, mt);
        R.P.load(at<const T>(p.ws, p.off.P) + slot * 64 * 64, mt);
        R.Tm.load(at<const T>(p.ws, p.off.Tm) + slot * 64 * 64, mt);
        R.sc.load(p, slot, tbase, len, mt);
      }
      if (part < 0 || part == 0) {
        R.Q.load(p.q + tbase * DK, tsk, len, mt);
        R.fq.load(at<const float>(p.ws, p.off.Nq) + slot * 64, mt);
      }
      if (part < 0 || part == 1) {
        R.K.load(p.k + tbase * DK, tsk, len, mt);
        R.fk.load(at<const float>(p.ws, p.off.Nk) + slot * 64, mt);
      }
    };
    auto normalise = [&](Chunk& R, int part = -1) __attribute__((always_inline)) {
      if (p.l2norm && part != 1) scale_rows(R.Q, R.fq, mt);
      if (p.l2norm && part != 0) scale_rows(R.K, R.fk, mt);
    };
    auto commit = [&](const Chunk& R) __attribute__((always_inline)) {
      R.dO.store(sdO, LDV, mt);
      R.P.store(sP);
      R.Tm.store(sTm);
      R.sc.put(sc, p.scale, mt);
      store_rows(R.Q, sQ, LDK, mt);
    };
    auto step = [&](Chunk& cur, Chunk& nxt, int n) __attribute__((always_inline)) {  // as in the forward pass
      if constexpr (L::AHEAD) {
        fetch(cur, n - 2, 2);
        fetch(cur, n - 2, 0);
        __builtin_amdgcn_sched_barrier(0);
        normalise(nxt, 1);
        store_rows(nxt.K, k_tile(n - 1), LDK, mt);
        __builtin_amdgcn_sched_barrier(0);
        fetch(cur, n - 2, 1);
      } else {
        fetch(cur, n - 1);
      }
      lds_barrier();  // B2
      int tok0, len;
      chunk_span(ch.span, n, tok0, len);
      unstage_tile<T, BV, 64, true>(at<T>(p.ws, p.off.dD) + ((int64_t)ch.row * N + n) * p.dv * 64 + (int64_t)v0 * 64, 64, sdRT, LDT, BV, mt);
      unstage_tile_checked<T, 64, BV>(p.dv_out + tok_index(p.geom, ch.row, tok0) * p.dv + v0, tsv, sdV, LDV, len, mt);
      normalise(nxt, 0);
      commit(nxt);
      if (!L::AHEAD) {
        lds_barrier();  // B3
        normalise(nxt, 1);
        store_rows(nxt.K, sK, LDK, mt);
      }
      lds_barrier();  // B1 of the next chunk
    };
    if (c0 < c1) {
      fetch(a, c1 - 1);
      if (L::AHEAD) fetch(b, c1 - 2);
      normalise(a);
      commit(a);
      store_rows(a.K, k_tile(c1 - 1), LDK, mt);
    }
    lds_barrier();  // B1 of the first chunk
    if constexpr (L::AHEAD) {
      for (int n = c1 - 1; n >= c0;) {
        step(a, b, n);
        if (--n < c0) break;
        step(b, a, n--);
      }
    } else {
      for (int n = c1 - 1; n >= c0; --n) step(a, a, n);
    }
    return;
  }

  // ---------------- compute waves ----------------
  const int vs = 16 * NC * wave;
  Strip<NC> dS;
  dS.load(p.d_sT ? p.d_sT + (int64_t)ch.sidx * DK * p.dv + v0 + vs : nullptr, p.dv, lane);
  auto save = [&](int n) { dS.save(at<T>(p.ws, p.off.dSn) + ((int64_t)ch.row * N + n) * p.dv * DK + (int64_t)(v0 + vs) * DK, fresh(tid & 63)); };
  if (c0 < c1) save(c1 - 1);
  lds_barrier();  // B1 of the first chunk
  for (int n = c1 - 1; n >= c0; --n) {
    const int lane = fresh(tid & 63), g8 = grp(lane);
    // ---- Z = K dS' ----
    floatx4 z[NC][4];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) z[c][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    dS.template rows_times<4, false>(z, k_tile(n), LDK, 0, lane);
    // ---- dO as an operand, and its rows times scale e^G ----
    Frag fo[NC][2], foq[NC][2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const floatx4 f0 = load4(sc + Sc::Q + 32 * s + g8), f1 = load4(sc + Sc::Q + 32 * s + g8 + 4);
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const Frag x = S16::load_t(sdO, LDV, 32 * s, vs + 16 * c, lane);
        fo[c][s] = x;
        foq[c][s] = S16::from_acc(f0 * floatx4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]},
                                  f1 * floatx4{(float)x[4], (float)x[5], (float)x[6], (float)x[7]});
      }
    }
    // ---- dD = Pm^T dO + e^{G_C - G} Z; Pm^T is upper-triangular ----
    Frag bd[NC][2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      floatx4 d[NC][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int i = 2 * s + h;
        const floatx4 r = load4(sc + Sc::R + row0(i) + g8);
#pragma unroll
        for (int c = 0; c < NC; ++c) d[c][h] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = s; k < 2; ++k) {
          const Frag f = load_cols(sP, LDC, k, i, lane);
#pragma unroll
          for (int c = 0; c < NC; ++c) S16::mma(d[c][h], f, fo[c][k]);
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) d[c][h] += r * z[c][i];
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) bd[c][s] = S16::from_acc(d[c][0], d[c][1]);
    }
    // ---- dR = Tm^T dD (rows = tokens), and once more with the operands exchanged (columns = tokens), the orientation that dv leaves in;
    //      Tm^T is upper-triangular ----
    Frag by[NC][2];  // dY
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      floatx4 x[NC][2], gm[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int i = 2 * s + h;
        floatx4 w[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) x[c][h] = w[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = s; k < 2; ++k) {
          const Frag f = load_cols(sTm, LDC, k, i, lane);
#pragma unroll
          for (int c = 0; c < NC; ++c) S16::mma(x[c][h], f, bd[c][k]), S16::mma(w[c], bd[c][k], f);
        }
        gm[h] = load4(sc + Sc::GAM + row0(i) + g8);
        const int t = row0(i) + row_of(lane);
        const float bt = sc[Sc::BETA + t];
#pragma unroll
        for (int c = 0; c < NC; ++c) store4(sdV + t * LDV + vs + 16 * c + 4 * (lane >> 4), w[c] * bt);
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        *reinterpret_cast<bf16x8*>(sdRT + (vs + 16 * c + (lane & 15)) * LDT + 32 * s + g8) = S16::from_acc(x[c][0], x[c][1]);
        by[c][s] = S16::from_acc(-gm[0] * x[c][0], -gm[1] * x[c][1]);
      }
    }
    // ---- dS <- e^{G_C} dS' + (scale e^G Q)^T dO ----
    dS.template add<GATE == LNX_GATE_SCALAR>(sQ, LDK, foq, lane, sc[Sc::DEC]);
    lds_barrier();  // B2
    // ---- dS += K^T dY ----
    dS.template add<false>(k_tile(n), LDK, by, lane);
    if (!L::AHEAD) lds_barrier();  // B3
    if (n > c0) save(n - 1);
    lds_barrier();  // B1 of the next chunk
  }
  if (p.ds0) dS.store(p.ds0 + (int64_t)ch.sidx * DK * p.dv + v0 + vs, p.dv, fresh(tid & 63));
}

// Width of the slabs: the cheapest by rounds of 256 workgroups times the time of a chunk, which grows less than the width
// because every workgroup loads the chunk's K and Q (relative times).  One round, us a chunk, few workgroups .. all 256:
//   32 columns   forward 2.8 .. 3.3 (nothing saved 2.6 .. 2.8)   reverse 2.6 .. 3.2
//   64           3.5 .. 4.9 (2.9 .. 3.7)                         3.1 .. 5.2
//   128          6.9 .. 7.2 (5.5)                                6.1 .. 6.5     (at dv = 512 with LDS reads ahead 7.9 -> 7.1 (5.8 -> 5.0) forward)
// Up to 256 workgroups of 128 columns the choice is the fastest, also for forms that save nothing: T4096 dv128, forward / reverse, 64 heads
// 209 / 203 us with 32 columns, 263 / 263 with 64; 96 heads 385 / 380 and 275 / 281; 128 heads 311 / 331 with 64 and 461 / 414 with 128; 160 heads
// 545 / 545 and 476 / 431.  Beyond, where 128 columns take two rounds and 64 three, 64 would be faster by up to 15 % (T1024, 320 heads
// 233 / 243 against 267 / 262; 448 heads 314 / 321 against 294 / 286).
int slab_width(const DirectParams& p, int nstate) {
  if (p.slab == 32 || p.slab == 64) return p.slab;
  const int64_t chains = (int64_t)nstate * p.geom.H;
  auto cost = [&](int bv, double us) { return p.dv % bv ? 1e30 : us * (double)((chains * (p.dv / bv) + 255) / 256); };
  const double c128 = cost(128, 4.2), c64 = cost(64, 2.9), c32 = cost(32, 2.5);
  return c128 <= c64 && c128 <= c32 ? 128 : c64 <= c32 ? 64 : 32;
}

template <typename K> int launch(K k, size_t bytes, int bv, int threads, const char* name, const DirectParams& p, int nstate, hipStream_t st) {
  if (const int rc = lnx_lds_limit(reinterpret_cast<const void*>(k), bytes); rc != LNX_OK) return rc;
  lnx_profile_mark(name, st);
  hipLaunchKernelGGL(k, dim3(lnx_xcd_grid((int64_t)nstate * p.geom.H, p.dv / bv)), dim3(threads), bytes, st, p);
  return LNX_OK;
}
template <int GATE, int NC, int NCW> int launch_width(bool bwd, const DirectParams& p, int nstate, hipStream_t st) {
  typedef WideL<NC, NCW> L;
  if (bwd) return launch(wide_scan_bwd_kernel<GATE, NC, NCW>, L::bytes, L::BV, L::threads, "bwd_scan", p, nstate, st);
  if (!p.o && !p.save) return launch(wide_scan_fwd_kernel<GATE, NC, NCW, void>, L::bytes, L::BV, L::threads, "chunk_scan", p, nstate, st);
  if (p.o_dtype == LNX_BF16) return launch(wide_scan_fwd_kernel<GATE, NC, NCW, bf16_t>, L::bytes, L::BV, L::threads, "chunk_scan", p, nstate, st);
  return launch(wide_scan_fwd_kernel<GATE, NC, NCW, float>, L::bytes, L::BV, L::threads, "chunk_scan", p, nstate, st);
}
template <int GATE> int launch_gate(bool bwd, const DirectParams& p, int nstate, hipStream_t st) {
  switch (slab_width(p, nstate)) {
    case 128: return launch_width<GATE, 2, 4>(bwd, p, nstate, st);
    case 64: return launch_width<GATE, 1, 4>(bwd, p, nstate, st);
    default: return launch_width<GATE, 1, 2>(bwd, p, nstate, st);
  }
}

}  // namespace

int lnx_wide_scan(bool backward, const DirectParams& p, int nstate, hipStream_t st) {
  return p.gate == LNX_GATE_SCALAR ? launch_gate<LNX_GATE_SCALAR>(backward, p, nstate, st) : launch_gate<LNX_GATE_NONE>(backward, p, nstate, st);
}
