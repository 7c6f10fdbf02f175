// The two sequential passes of the WY-split chunk kernels for 2-byte inputs with dk = 256 and no / a scalar gate (the head shape of
// the Gated DeltaNet presets).  Same products and roundings as chunk_scan (chunk_fwd.hip) and bwd_scan (chunk_bwd.hip), which serve
// the other shapes.  The forward sums have their order, too; in reverse Q^T dO is added before W^T dD, as bwd_scan does up to dk = 128 --
// its 64-column slabs of dk = 256 added W^T dD first, because Q shared a tile with K -- so that gradients differ from that form's by the
// rounding of one sum (1.2e-4 of the 2-norm in bf16):
//
//   forward   D = U - W S       O = scale diag(e^G) (Q S) + Pm D       S' = e^{G_C} S + (diag(e^{G_C - G}) K)^T D
//   reverse   dD = Pm^T dO + diag(e^{G_C - G}) K dS'                   dS = e^{G_C} dS' + (scale diag(e^G) Q)^T dO - W^T dD
//
// What bounds them: with dk = 256 a chunk's K, Q and W rows are 96 KB, which every workgroup of a (state, head) loads again for
// its slab of value columns, and LDS holds them once.  So a slab is as wide as the registers allow: a compute wave owns 16 NC value
// columns, whose [256 x 16 NC] part of the state stays in accumulators for the whole sequence and is the operand of the next
// products as it stands (a column of tiles as Mma16 describes, in natural order); only K, Q, W and Pm come from LDS.  The state also
// leaves from there: an operand fragment is 16 bytes of a row of the saved tensor.  Four mover waves hold the next chunk
// in registers.  Per chunk:
//   B1   tiles of chunk n in LDS               compute: everything but the last product     movers: loads of the next chunk
//   B2   its K (forward) / W (reverse) is left   compute: the last product    movers: results -> global, the other tiles -> LDS
//   B3                                         compute: state -> global     movers: the last tile -> LDS
// Measured at B8 H8 T4096 dv512 (128-column slabs, 256 workgroups): forward 750 -> 551 us, reverse 658 -> 464 us against the
// passes with 64-column slabs.  A chunk takes 7 - 8.6 us there, of which 216 KB through the CU's memory path are most: 64 KB of
// state per chunk and slab leave for the backward kernels.  State stores among the products of the first phase instead of
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
// a fetched tile to LDS, its rows at their places
template <int COLS> __device__ __forceinline__ void store_placed(const TileRegs<T, 64, COLS>& R, T* dst, int ld, int tid) {
  typedef TileRegs<T, 64, COLS> Tile;
#pragma unroll
  for (int it = 0; it < Tile::IT; ++it) {
    const int idx = tid + 256 * it, r = idx / Tile::VPR, c = (idx - r * Tile::VPR) * Tile::N;
    *reinterpret_cast<bf16x8*>(dst + place(r) * ld + c) = R.x[it];
  }
}

template <int NC, int NCW> struct WideL {
  static constexpr int BV = 16 * NC * NCW, LDK = DK + 16, LDC = LNX_C + 16, LDV = BV + 8;
  static constexpr int kRow = 64 * LDK, kC = 64 * LDC, kV = 64 * LDV;
  // K | Q | W | Pm | U, replaced by D (reverse: dO) | O on its way out (reverse: dD) | scalars
  static constexpr size_t bytes = sizeof(T) * (3 * kRow + kC + 2 * kV) + sizeof(float) * 192;
  static constexpr int threads = 64 * NCW + 256;
  static_assert(bytes <= 160 * 1024, "LDS");
};
struct Sc {
  enum { R = 0, Q = 64, DEC = 128 };  // e^{G_C - G}, scale e^G, e^{G_C}
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

// the gate's scalars of a chunk, by 64 threads
template <int GATE> __device__ __forceinline__ void put_scalars(float* sc, float g, float gl, float scale, int t) {
  sc[Sc::R + t] = (GATE == LNX_GATE_SCALAR) ? __expf(fminf(gl - g, 0.f)) : 1.f;
  sc[Sc::Q + t] = (GATE == LNX_GATE_SCALAR) ? scale * __expf(g) : scale;
  if (t == 0) sc[Sc::DEC] = (GATE == LNX_GATE_SCALAR) ? __expf(gl) : 1.f;
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
        for (int e = 0; e < 4; ++e) x[c][ci][e] = src ? src[(int64_t)(row0(ci) + grp(lane) + e) * dv + 16 * c + (lane & 15)] : 0.f;
    // the loads complete here: left pending into the loop, every iteration would count them down again
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int ci = 0; ci < KT; ++ci)
#pragma unroll
        for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(x[c][ci][e]));
  }
  __device__ __forceinline__ void store(float* dst, int dv, int lane) const {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int ci = 0; ci < KT; ++ci)
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[(int64_t)(row0(ci) + grp(lane) + e) * dv + 16 * c + (lane & 15)] = x[c][ci][e];
  }
  __device__ __forceinline__ Frag operand(int c, int ks) const { return S16::from_acc(x[c][2 * ks], x[c][2 * ks + 1]); }
  __device__ __forceinline__ void save(T* dst, int lane) const {  // [value column][dk] of the strip
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) *reinterpret_cast<bf16x8*>(dst + (16 * c + (lane & 15)) * DK + 32 * ks + 8 * (lane >> 4)) = operand(c, ks);
  }
  __device__ __forceinline__ void scale(float f) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int ci = 0; ci < KT; ++ci) x[c][ci] *= f;
  }
  // x += tile^T b: rows of the tile (tokens) contracted
  __device__ __forceinline__ void add(const T* tile, int ld, const Frag (&b)[NC][2], int lane) {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int ci = 0; ci < KT; ++ci) {
        const Frag f = load_cols(tile, ld, s, ci, lane);
#pragma unroll
        for (int c = 0; c < NC; ++c) S16::mma(x[c][ci], f, b[c][s]);
      }
  }
};

template <int GATE, int NC, int NCW, typename OT>
__global__ __launch_bounds__((WideL<NC, NCW>::threads)) void wide_scan_fwd_kernel(DirectParams p) {
  typedef WideL<NC, NCW> L;
  constexpr int BV = L::BV, LDK = L::LDK, LDC = L::LDC, LDV = L::LDV;
  extern __shared__ __align__(16) char smem[];
  T* sK = reinterpret_cast<T*>(smem);
  T* sQ = sK + L::kRow;
  T* sW = sQ + L::kRow;
  T* sP = sW + L::kRow;
  T* sU = sP + L::kC;
  T* sO = sU + L::kV;
  float* sc = reinterpret_cast<float*>(sO + L::kV);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  Chain ch;
  if (!chain_of<BV>(p, ch)) return;
  const int N = p.geom.N, c0 = ch.c0, c1 = ch.c1, v0 = ch.v0;
  const int64_t tso = (int64_t)p.geom.ts * p.dv;

  if (wave >= NCW) {
    // ---------------- movers ----------------
    const int mt = tid - 64 * NCW;
    TileRegs<T, 64, DK> rK, rQ, rW;
    TileRegs<T, 64, BV> rU;
    TileRegs<T, 64, 64> rP;
    float g = 0.f, gl = 0.f;
    const int64_t tsk = (int64_t)p.geom.ts * DK;
    auto fetch = [&](int n) {
      const int64_t slot = (int64_t)ch.row * N + n;
      int tok0, len;
      chunk_span(ch.span, n, tok0, len);
      const int64_t tbase = tok_index(p.geom, ch.row, tok0);
      rW.load(at<const T>(p.ws, p.off.W) + slot * 64 * DK, DK, 64, mt);
      rQ.load(p.q + tbase * DK, tsk, len, mt);
      rU.load(at<const T>(p.ws, p.off.U) + slot * 64 * p.dv + v0, p.dv, 64, mt);
      rP.load(at<const T>(p.ws, p.off.P) + slot * 64 * 64, 64, 64, mt);
      if (GATE == LNX_GATE_SCALAR) {
        const float* G = at<const float>(p.ws, p.off.G) + slot * 64;
        g = G[mt & 63];
        gl = G[63];
      }
      rK.load(p.k + tbase * DK, tsk, len, mt);
    };
    auto commit = [&]() {
      store_placed<DK>(rW, sW, LDK, mt);
      store_placed<DK>(rQ, sQ, LDK, mt);
      rU.store(sU, LDV, mt);
      store_placed<64>(rP, sP, LDC, mt);
    };
    auto commit_k = [&]() {  // the scalars with it: the last product's decay is read until here
      store_placed<DK>(rK, sK, LDK, mt);
      if (mt < 64) put_scalars<GATE>(sc, g, gl, p.scale, mt);
    };
    if (c0 < c1) {
      fetch(c0);
      commit();
      commit_k();
    }
    lds_barrier();  // B1 of the first chunk
    for (int n = c0; n < c1; ++n) {
      fetch(min(n + 1, c1 - 1));  // unconditional, as the commits: a load behind a branch cannot be counted
      lds_barrier();  // B2
      const int64_t slot = (int64_t)ch.row * N + n;
      int tok0, len;
      chunk_span(ch.span, n, tok0, len);
      if (std::is_same<OT, T>::value && p.o)
        unstage_tile_checked<T, 64, BV>(reinterpret_cast<T*>(p.o) + tok_index(p.geom, ch.row, tok0) * p.dv + v0, tso, sO, LDV, len, mt);
      if (p.save) unstage_tile<T, 64, BV, true>(at<T>(p.ws, p.off.D) + slot * 64 * p.dv + v0, p.dv, sU, LDV, 64, mt);
      commit();  // U over D: every thread writes the vectors that it has just read
      lds_barrier();  // B3
      commit_k();
      lds_barrier();  // B1 of the next chunk
    }
    return;
  }

  // ---------------- compute waves: wave w owns value columns [16 NC w, 16 NC (w + 1)) of the slab ----------------
  const int vs = 16 * NC * wave;
  Strip<NC> S;
  S.load(p.s0 ? p.s0 + (int64_t)ch.sidx * DK * p.dv + v0 + vs : nullptr, p.dv, lane);
  auto save = [&](int n) {
    if (p.save) S.save(at<T>(p.ws, p.off.SnT) + ((int64_t)ch.row * N + n) * p.dv * DK + (int64_t)(v0 + vs) * DK, fresh(tid & 63));
  };
  if (c0 < c1) save(c0);
  lds_barrier();  // B1 of the first chunk
  for (int n = c0; n < c1; ++n) {
    const int lane = fresh(tid & 63), l16 = lane & 15, g8 = grp(lane);
    // ---- D = U - W S: rows = tokens ----
    floatx4 y[NC][4];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) y[c][i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      Frag b[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) b[c] = S.operand(c, ks);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const Frag a = load_rows(sW, LDK, i, ks, lane);
#pragma unroll
        for (int c = 0; c < NC; ++c) S16::mma(y[c][i], a, b[c]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    Frag bd[NC][2], bu[NC][2];  // D, and D with its rows scaled by e^{G_C - G}, as operands
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      floatx4 d[4], e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bf16x4 u = S16::rows4(sU, LDV, row0(i) + g8, vs + 16 * c, lane);
        d[i] = floatx4{(float)u[0], (float)u[1], (float)u[2], (float)u[3]} - y[c][i];
        e[i] = d[i] * load4(sc + Sc::R + row0(i) + g8);
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) bd[c][s] = S16::from_acc(d[2 * s], d[2 * s + 1]), bu[c][s] = S16::from_acc(e[2 * s], e[2 * s + 1]);
#pragma unroll
      for (int s = 0; s < 2; ++s)  // D replaces U
#pragma unroll
        for (int r = 0; r < 8; ++r) sU[(32 * s + g8 + r) * LDV + vs + 16 * c + l16] = bd[c][s][r];
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- O^T = scale e^G (Q S)^T + D^T Pm^T: columns = tokens, 32 of them at a time ----
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int lane = fresh(tid & 63);
      floatx4 o[NC][2];
#pragma unroll
      for (int c = 0; c < NC; ++c) o[c][0] = o[c][1] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) {
        Frag b[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) b[c] = S.operand(c, ks);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const Frag q = load_rows(sQ, LDK, 2 * h + i, ks, lane);
#pragma unroll
          for (int c = 0; c < NC; ++c) S16::mma(o[c][i], b[c], q);
        }
      }
      int tok0, len;
      chunk_span(ch.span, n, tok0, len);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int t = row0(2 * h + i) + row_of(lane);
        const float f = sc[Sc::Q + t];
#pragma unroll
        for (int c = 0; c < NC; ++c) o[c][i] *= f;
#pragma unroll
        for (int k = 0; k <= h; ++k) {  // Pm is lower-triangular: the first 32 tokens take the first step only
          const Frag f = load_rows(sP, LDC, 2 * h + i, k, lane);
#pragma unroll
          for (int c = 0; c < NC; ++c) S16::mma(o[c][i], bd[c][k], f);
        }
        if constexpr (std::is_same<OT, T>::value) {
#pragma unroll
          for (int c = 0; c < NC; ++c) store4(sO + t * LDV + vs + 16 * c + 4 * (lane >> 4), o[c][i]);
        } else if (p.o && t < len) {
#pragma unroll
          for (int c = 0; c < NC; ++c)
            store4(reinterpret_cast<float*>(p.o) + (tok_index(p.geom, ch.row, tok0) + (int64_t)t * p.geom.ts) * p.dv + v0 + vs + 16 * c + 4 * (lane >> 4), o[c][i]);
        }
      }
    }
    const float dec = sc[Sc::DEC];
    lds_barrier();  // B2
    if (GATE == LNX_GATE_SCALAR) S.scale(dec);
    S.add(sK, LDK, bu, fresh(tid & 63));
    lds_barrier();  // B3
    if (n + 1 < c1) save(n + 1);
    lds_barrier();  // B1 of the next chunk
  }
  S.store(p.sT_out.at(ch.sidx, (int64_t)DK * p.dv) + v0 + vs, p.dv, fresh(tid & 63));
}

template <int GATE, int NC, int NCW>
__global__ __launch_bounds__((WideL<NC, NCW>::threads)) void wide_scan_bwd_kernel(DirectParams p) {
  typedef WideL<NC, NCW> L;
  constexpr int BV = L::BV, LDK = L::LDK, LDC = L::LDC, LDV = L::LDV;
  extern __shared__ __align__(16) char smem[];
  T* sK = reinterpret_cast<T*>(smem);
  T* sQ = sK + L::kRow;
  T* sW = sQ + L::kRow;
  T* sP = sW + L::kRow;
  T* sdO = sP + L::kC;
  T* sdD = sdO + L::kV;
  float* sc = reinterpret_cast<float*>(sdD + L::kV);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  Chain ch;
  if (!chain_of<BV>(p, ch)) return;
  const int N = p.geom.N, c0 = ch.c0, c1 = ch.c1, v0 = ch.v0;

  if (wave >= NCW) {
    // ---------------- movers ----------------
    const int mt = tid - 64 * NCW;
    TileRegs<T, 64, DK> rK, rQ, rW;
    TileRegs<T, 64, BV> rdO;
    TileRegs<T, 64, 64> rP;
    float g = 0.f, gl = 0.f;
    const int64_t tsk = (int64_t)p.geom.ts * DK, tsv = (int64_t)p.geom.ts * p.dv;
    auto fetch = [&](int n) {
      const int64_t slot = (int64_t)ch.row * N + n;
      int tok0, len;
      chunk_span(ch.span, n, tok0, len);
      const int64_t tbase = tok_index(p.geom, ch.row, tok0);
      rK.load(p.k + tbase * DK, tsk, len, mt);
      rdO.load(p.d_o + tbase * p.dv + v0, tsv, len, mt);
      rP.load(at<const T>(p.ws, p.off.P) + slot * 64 * 64, 64, 64, mt);
      rQ.load(p.q + tbase * DK, tsk, len, mt);
      if (GATE == LNX_GATE_SCALAR) {
        const float* G = at<const float>(p.ws, p.off.G) + slot * 64;
        g = G[mt & 63];
        gl = G[63];
      }
      rW.load(at<const T>(p.ws, p.off.W) + slot * 64 * DK, DK, 64, mt);
    };
    auto commit = [&]() {
      store_placed<DK>(rK, sK, LDK, mt);
      rdO.store(sdO, LDV, mt);
      store_placed<64>(rP, sP, LDC, mt);
      store_placed<DK>(rQ, sQ, LDK, mt);
      if (mt < 64) put_scalars<GATE>(sc, g, gl, p.scale, mt);
    };
    if (c0 < c1) {
      fetch(c1 - 1);
      commit();
      store_placed<DK>(rW, sW, LDK, mt);
    }
    lds_barrier();  // B1 of the first chunk
    for (int n = c1 - 1; n >= c0; --n) {
      fetch(max(n - 1, c0));
      lds_barrier();  // B2
      unstage_tile<T, 64, BV, true>(at<T>(p.ws, p.off.dD) + ((int64_t)ch.row * N + n) * 64 * p.dv + v0, p.dv, sdD, LDV, 64, mt);
      commit();
      lds_barrier();  // B3
      store_placed<DK>(rW, sW, LDK, mt);
      lds_barrier();  // B1 of the next chunk
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
    const int lane = fresh(tid & 63), l16 = lane & 15, g8 = grp(lane);
    // ---- Z = K dS' ----
    floatx4 z[NC][4];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) z[c][i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      Frag b[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) b[c] = dS.operand(c, ks);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const Frag a = load_rows(sK, LDK, i, ks, lane);
#pragma unroll
        for (int c = 0; c < NC; ++c) S16::mma(z[c][i], a, b[c]);
      }
    }
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
    Frag bd[NC][2];  // -dD
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
      for (int c = 0; c < NC; ++c) {
        const Frag x = S16::from_acc(d[c][0], d[c][1]);
#pragma unroll
        for (int r = 0; r < 8; ++r) sdD[(32 * s + g8 + r) * LDV + vs + 16 * c + l16] = x[r];
        bd[c][s] = S16::from_acc(-d[c][0], -d[c][1]);
      }
    }
    // ---- dS <- e^{G_C} dS' + (scale e^G Q)^T dO ----
    if (GATE == LNX_GATE_SCALAR) dS.scale(sc[Sc::DEC]);
    dS.add(sQ, LDK, foq, lane);
    lds_barrier();  // B2
    // ---- dS -= W^T dD ----
    dS.add(sW, LDK, bd, lane);
    lds_barrier();  // B3
    if (n > c0) save(n - 1);
    lds_barrier();  // B1 of the next chunk
  }
  if (p.ds0) dS.store(p.ds0 + (int64_t)ch.sidx * DK * p.dv + v0 + vs, p.dv, fresh(tid & 63));
}

// Width of the slabs: the cheapest by rounds of 256 workgroups times the time of a chunk, which grows less than the width
// because every workgroup loads the chunk's K, Q and W (relative times; at one round of workgroups 8.6 us with 128 columns).
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
