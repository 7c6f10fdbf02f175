// Chunked delta-rule forward and backward for 2-byte inputs with no / a scalar gate, in the
// "direct solve" split (dk = 256: the scans are those of chunk_wide.hip): the only per-chunk tensors that cross kernels are Tm = (I + A)^-1, Pm = scale tril(E * Q K^T)
// and the cumulative gate G from the chunk-parallel prepare kernel, the states entering the chunks and D (forward scan
// -> chunk-local backward) and the state gradients leaving them and dR (reverse scan -> chunk-local backward).  W, U,
// dD, dW of the WY form are never materialised: with S the state entering a chunk,
//
//   Y = K S          R = diag(beta) (V - diag(e^G) Y)      D = Tm R                     (forward substitution applied
//   O = scale diag(e^G) (Q S) + Pm D                                                     to the chunk's right-hand
//   S' = e^{G_C} S + (diag(e^{G_C - G}) K)^T D                                           side, gated_deltanet.py:450-477)
//
// and in reverse, with dS' the gradient of the state leaving the chunk,
//
//   dD = Pm^T dO + diag(e^{G_C - G}) K dS'     dR = Tm^T dD     dY = -diag(beta e^G) dR
//   dS = e^{G_C} dS' + (scale diag(e^G) Q)^T dO + K^T dY
//
// which is the algorithm of linearnexus/modules/linear_attn/gated_deltanet.py:444-523 (delta_net.py:296-330 without
// a gate) and its hand-derived adjoint (the reference's gradients come from JAX autodiff).  Three kernels:
//
//   scan_fwd   (one workgroup per (state, slab of dv), sequential over chunks)   O, the entering states, S_T
//   scan_bwd   (same grid, reverse)                                              the leaving state gradients, dS_0
//   bwd_chunk  (one workgroup per chunk, all in parallel)                         dq, dk, dbeta, dg from q, k, v, dO, the
//              two saved states and D, dR as the scans left them (dv leaves the reverse scan)
//
// Both scans split their waves into one compute wave per 16 value columns of the slab (matrix work on the tiles in LDS, the fp32 state in MFMA
// accumulators for the whole sequence) and four or eight mover waves (global loads two chunks ahead into registers, the next chunk's tiles into
// LDS, LDS -> global copies of results as whole rows), scan_fwd's narrow form into output waves as well; all five input tiles are
// double-buffered in LDS, so one or two LDS-only barriers per chunk suffice.  bwd_chunk brings its slabs in with loads that go straight to LDS (mma_tiles.h).

#include <type_traits>

#include "chunk_common.h"

namespace {

using T = bf16_t;
typedef Mma<T> M;
typedef Mma16 S16;
template <typename X> __device__ __forceinline__ X* at(char* ws, uint64_t off) { return reinterpret_cast<X*>(ws + off); }

// dst[l16][grp ..] = accumulator tile in Mma16's order of rows (transposed store: this lane's column, four consecutive rows, 8 bytes)
__device__ __forceinline__ void store_t(const floatx4& a, T* dst, int ld, int lane) {
  store4(dst + (lane & 15) * ld + S16::grp(lane), a);
}

// dst[col][row0 + ...] = fragment (transposed store, four consecutive rows per 8-byte vector)
__device__ __forceinline__ void store_frag_t(const floatx16& a, T* dst, int ld, int lane) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const floatx4 x = {a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
    store4(dst + (lane & 31) * ld + 8 * q + 4 * (lane >> 5), x);
  }
}

// Zeroes the vectors above the diagonal of `ntile` consecutive [64][ld] tiles of `stride` elements, columns in the order CHAIN; 256 threads
// or more.
template <bool CHAIN> __device__ __forceinline__ void zero_upper_triangles(T* tiles, int ntile, int stride, int ld, int tid) {
  if (tid >= 512 - LNX_TRI_VECS) return;
  int r, c;
  upper_vec_pos(tid, r, c);
  for (int t = 0; t < ntile; ++t) S16::put<CHAIN>(tiles + t * stride + r * ld + S16::pos<CHAIN>(8 * c), vec_zero<T>());
}

// A row's elements times its factor, rounded back
__device__ __forceinline__ typename Vec16<T>::V scaled(typename Vec16<T>::V x, float f) {
#pragma unroll
  for (int e = 0; e < Vec16<T>::N; ++e) x[e] = (bf16_t)((float)x[e] * f);
  return x;
}

// Per-token scalars of one chunk in LDS, written by the movers when they commit a chunk
struct Scal {
  enum { BETA = 0, GAM = 64, R = 128, DEC = 192, SIZE = 256, NK = 256, FQ = 320, SIZE_FACTORS = 384 };  // beta, beta e^G, e^{G_C - G}, e^{G_C}, factors of the K and Q rows
};
template <int GATE> __device__ __forceinline__ void put_scalars(float* sc, int t, float b, float g, float gc) {
  const float gam = (GATE == LNX_GATE_SCALAR) ? __expf(g) : 1.f;
  sc[Scal::BETA + t] = b;
  sc[Scal::GAM + t] = b * gam;
  sc[Scal::R + t] = (GATE == LNX_GATE_SCALAR) ? __expf(fminf(gc - g, 0.f)) : 1.f;
  if (t == 0) sc[Scal::DEC] = (GATE == LNX_GATE_SCALAR) ? __expf(gc) : 1.f;
}

// ---------------------------------------------------------------------------------------
// scan_fwd.  A compute wave owns a 16-column strip of the value slab: its [dk x 16] part of the state stays in MFMA
// accumulators for the whole sequence, and the chain  S -> Y = K S -> R -> D = Tm R -> S'  never leaves the wave's
// registers -- two accumulator tiles are the B operand of the next product as they are (Mma16::from_acc), only the A
// operands (K, Q, Tm, Pm rows) come from LDS.  Strips of 16 columns put a slab's chain on twice as many SIMDs as strips of 32, which counts
// where there are fewer workgroups than CUs: B2 H16 T2007 d128 (32 chunks in a row, 128 workgroups) 66 -> 57 us forward and 74 -> 60 us
// in reverse, one prompt of 1000 tokens 34 -> 29 us.  With 256 workgroups of 64-column slabs, bound by what the movers carry, it changes
// nothing: B8 H16 T4096 184 and 200 us before and after.  The bits are those of 32-column strips (Mma16).  What is left of a chunk's
// 1.5 us in the short calls: a SIMD takes 1 KB of LDS reads in about 16 cycles, and a strip reads 60 KB of operands whatever its
// width.  The movers convert K and Q rows, 2.5 VALU instructions an element: with eight waves of them instead of four 57 -> 52 us and
// 29 -> 27 us; in reverse the third wave of each SIMD leaves too few registers (59 -> 59 - 68 us), it keeps four.
// All five input tiles are double-buffered, so the movers write chunk n + 1 while chunk n is being read.  64-column slabs with outputs:
//   B1    buffers of chunk n complete           compute: S^T -> LDS (saved states), Y, Q S, R, D (-> LDS, transposed), O -> LDS
//                                               movers:  loads of chunk n + 2; chunk n + 1 -> the other buffers
//   Bmid  O, S^T and D^T are in LDS             compute: state update        movers: O, S^T, D^T -> global
// 32-column slabs, where the chain of one chunk is what a call waits for: O hangs on S and D but nothing on O, so it has waves of its own, a
// chunk behind, and one barrier per chunk is enough:
//   B1    K, V, Tm of chunk n, Q, Pm of n - 1   compute: Y, R, D, state update; S^T and D^T -> LDS [n mod 2]
//                                               output:  O of chunk n - 1 from S^T and D^T as the compute wave has them in registers -> global;
//                                                        behind it the per-token scalars of chunk n + 2
//                                               movers:  S^T, D^T of n - 1 -> global; loads and writes as above, Q and Pm of the chunk before
// A chunk of one prompt of 1000 tokens: 1.43 us with everything in the compute waves (Y and Q S 0.5, R and D 0.2, the rest of O 0.2, update 0.3,
// movers 0.7 between B1 and Bmid), 1.23 so (compute 1.0, movers 1.15, output 0.8); the call 33.3 -> 32.1 us, the scan of B2 H16 T2007 53 -> 48.
// Output waves beside two barriers: 35.4 us, the movers' 0.85 us then stood between B1 and Bmid alone.  One barrier with the row factors from
// memory, five small loads a mover: 33.0; every mover in the same order: 33.0, all of them load, convert and write at the same time, so half
// write a tile ahead of the next loads and half behind them.  The same bits in all.
// Final states alone (OUT false, the first pass over a segmented prompt): no Q, no Pm, no O, one barrier: 16 segments of 4 heads, 64 chunks
// each, 111 -> 73 us.
// ---------------------------------------------------------------------------------------
template <int DK, int BVW, bool OUT> struct FScanL {
  // 32-column slabs are taken where the chip has room for more workgroups, so what counts there is the time of a chunk's
  // chain: operand tiles in chain order, rows 32 bytes off a multiple of 64 (Mma16).  64-column slabs are bound by what the
  // movers carry.
  static constexpr bool CHAIN = BVW == 32;
  static constexpr int BV = BVW, PAD = M::PAD, OPAD = CHAIN ? 16 : 8, LDK = DK + OPAD, LDC = LNX_C + OPAD, LDV = BV + PAD, NCW = BV / 16, MT = CHAIN && DK == 128 ? 512 : 256;
  static constexpr int LDS = DK + PAD, LDD = LNX_C + PAD;  // of the tiles on their way out: states, D or dR
  static constexpr int kK = 64 * LDK, kST = BV * LDS, kV = 64 * LDV, kC = 64 * LDC;
  static constexpr int kDT = BV * LDD;
  static constexpr int NOW = OUT && CHAIN ? NCW : 0;  // output waves, one per strip
  static constexpr int NST = NOW ? 2 : 1;             // buffers of S^T and D^T
  static constexpr int NSC = NOW ? 4 : 2;             // ... of scalars
  static constexpr int SCS = NOW ? Scal::SIZE_FACTORS : Scal::SIZE;
  // [2] x (K, Q, V, Tm, Pm) | O, unless output waves store it | S^T [NST] | D^T [NST] | scalars [2]; without outputs [2] x (K, V, Tm) | scalars [2]
  static constexpr size_t bytes = sizeof(T) * (OUT ? 2 * (2 * kK + kV + 2 * kC) + (NOW ? 0 : kV) + NST * (kST + kDT) : 2 * (kK + kV + kC)) + sizeof(float) * NSC * SCS;
  static constexpr int threads = 64 * (NCW + NOW) + MT;
};

template <int DK, int GATE, int BVW, typename OT>
__global__ __launch_bounds__((FScanL<DK, BVW, !std::is_void<OT>::value>::threads)) void scan_fwd_kernel(DirectParams p) {
  constexpr bool OUT = !std::is_void<OT>::value;  // void: final states alone (forward only)
  typedef FScanL<DK, BVW, OUT> L;
  constexpr int LDK = L::LDK, LDC = L::LDC, BV = L::BV, LDV = L::LDV, NCW = L::NCW, LDS = L::LDS, LDD = L::LDD;
  constexpr bool CHAIN = L::CHAIN;
  constexpr int MT = L::MT;  // mover threads
  constexpr int NOW = L::NOW;
  constexpr int KT = DK / 16;  // row tiles of the state strip
  static_assert(DK == 64 || DK == 128, "dk = 64 or 128");
  extern __shared__ __align__(16) char smem[];
  T* sK = reinterpret_cast<T*>(smem);  // [2][64][LDK]
  T* sQ = sK + 2 * L::kK;
  T* sV = sQ + (OUT ? 2 * L::kK : 0);  // [2][64][LDV]
  T* sTm = sV + 2 * L::kV;             // [2][64][LDC]
  T* sP = sTm + 2 * L::kC;
  T* sO = sP + 2 * L::kC;              // bf16 outputs on their way out [64][LDV]
  T* sST = sO + (NOW ? 0 : L::kV);                 // entering state, transposed [v][dk], for the output waves and on its way to the workspace
  T* sDT = sST + L::NST * L::kST;      // D^T [v][token], likewise
  float* sSc = reinterpret_cast<float*>(OUT ? sDT + L::NST * L::kDT : sP);  // [2][L::SCS]

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int N = p.geom.N;
  int sidx, row, seq;
  int64_t chain;
  int slab;
  if (!xcd_slot_part((int64_t)(p.geom.tab ? p.geom.nseq : p.geom.rows / p.geom.H) * p.geom.H, p.dv / BV, chain, slab)) return;
  scan_state(p.geom, (int)chain, sidx, row, seq);
  const int v0 = slab * BV;
  int c0, c1;
  seq_chunks(p.geom, seq, c0, c1);
  const SeqSpan span = seq_span(p.geom, seq, c0);
  const int64_t tsk = (int64_t)p.geom.ts * DK, tsv = (int64_t)p.geom.ts * p.vcols, tso = (int64_t)p.geom.ts * p.dv;

  if (wave >= NCW + NOW) {
    // ---------------- movers ----------------
    const int mt = tid - 64 * (NCW + NOW);
    typedef TileRegs<T, 64, DK, MT> RowTile;
    typedef TileRegs<T, 64, BV, MT> ValTile;
    struct Tiles {
      RowTile K, Q;
      ValTile V;
      TriRegs<T, CHAIN, MT> Tm, P;  // lower-triangular tiles, packed in the workspace
      float g, gc, b;  // per-token scalars of token mt % 64
      float fq[RowTile::IT], nk[RowTile::IT];  // factors of the token each of this thread's Q / K vectors belongs to
      float bv[ValTile::IT];  // beta of the token each of its V vectors belongs to
      int len;
    };
    Tiles ta, tb;
    ta.g = ta.gc = ta.b = tb.g = tb.gc = tb.b = 0.f;
    ta.Tm.init(LDC, mt), ta.P.init(LDC, mt), tb.Tm.init(LDC, mt), tb.P.init(LDC, mt);
    zero_upper_triangles<CHAIN>(sTm, OUT ? 4 : 2, L::kC, LDC, mt);  // both buffers of Tm and Pm: the packed tiles never write there
    ta.len = tb.len = 0;
#pragma unroll
    for (int it = 0; it < RowTile::IT; ++it) ta.fq[it] = tb.fq[it] = ta.nk[it] = tb.nk[it] = 0.f;
#pragma unroll
    for (int it = 0; it < ValTile::IT; ++it) ta.bv[it] = tb.bv[it] = 0.f;
    // part 0: K, 1: Q, 2: the rest; < 0: everything.  With output waves Q and Pm are those of the chunk before (part 1).
    auto fetch = [&](Tiles& R, int n, int part = -1) __attribute__((always_inline)) {
      if (NOW && part == 1) {
        const int64_t slot = (int64_t)row * N + n - 1;
        int tok0, len;
        chunk_span(span, n - 1, tok0, len);
        R.Q.load(p.q + tok_index(p.geom, row, tok0) * DK, tsk, len, mt);
        R.P.load(at<const T>(p.ws, p.off.P) + slot * 64 * 64, mt);
        return;
      }
      const int64_t slot = (int64_t)row * N + n;
      int tok0;
      chunk_span(span, n, tok0, R.len);
      const int64_t tbase = tok_index(p.geom, row, tok0);
      if (part < 0 || part == 0) R.K.load(p.k + tbase * DK, tsk, R.len, mt);
      if (OUT && (part < 0 || part == 1)) R.Q.load(p.q + tbase * DK, tsk, R.len, mt);
      if (part == 0 || part == 1) return;
      R.V.load(p.v + tbase * p.vcols + v0, tsv, (v0 < p.vcols) ? R.len : 0, mt);  // columns v does not hold read as zero
      R.Tm.load(at<const T>(p.ws, p.off.Tm) + slot * 64 * 64, mt);
      if (OUT && !NOW) R.P.load(at<const T>(p.ws, p.off.P) + slot * 64 * 64, mt);
      if (NOW) return;
      // every thread loads the scalars of token mt % 64 (no load behind a branch); tokens past the end are masked below
      const int t = mt & 63;
      if (GATE == LNX_GATE_SCALAR) {
        const float* G = at<const float>(p.ws, p.off.G) + slot * 64;
        R.g = G[t];
        R.gc = G[63];
      }
#pragma unroll
      for (int it = 0; it < RowTile::IT; ++it) {
        if (OUT) R.fq[it] = at<const float>(p.ws, p.off.Fq)[slot * 64 + (mt + MT * it) / RowTile::VPR];
        R.nk[it] = at<const float>(p.ws, p.off.Nk)[slot * 64 + (mt + MT * it) / RowTile::VPR];
      }
      R.b = p.beta[tbase + (int64_t)min(t, R.len - 1) * p.geom.ts];
#pragma unroll
      for (int it = 0; it < ValTile::IT; ++it)
        R.bv[it] = p.beta[tbase + (int64_t)min(min((mt + MT * it) / ValTile::VPR, 63), R.len - 1) * p.geom.ts];
    };
    // K rows normalised (their own bits where nothing is to be normalised), Q rows normalised and scaled by scale e^{G_i}
    auto commit = [&](const Tiles& R, int n, int part = -1) __attribute__((always_inline)) {
      const int pb = (n - c0) & 1;
      const float* sc = sSc + ((n - c0) & (L::NSC - 1)) * L::SCS;               // NOW: the factors come from the output waves
      const float* scq = sSc + ((n - 1 - c0) & (L::NSC - 1)) * L::SCS + Scal::FQ;
#pragma unroll
      for (int it = 0; it < RowTile::IT; ++it) {
        const int idx = mt + MT * it, r = idx / RowTile::VPR, c = (idx - r * RowTile::VPR) * RowTile::N;
        if (part < 0 || part == 0)
          S16::put<CHAIN>(sK + pb * L::kK + r * LDK + S16::pos<CHAIN>(c), p.l2norm ? scaled(R.K.x[it], NOW ? sc[Scal::NK + r] : R.nk[it]) : R.K.x[it]);
        if (OUT && (part < 0 || part == 1))
          S16::put<CHAIN>(sQ + (NOW ? pb ^ 1 : pb) * L::kK + r * LDK + S16::pos<CHAIN>(c), scaled(R.Q.x[it], NOW ? scq[r] : R.fq[it]));
      }
      if (NOW && part == 1) R.P.store(sP + (pb ^ 1) * L::kC);
      if (part == 0 || part == 1) return;
      {  // V rows scaled by beta_i: R = beta V - (beta e^G) Y
        T* dst = sV + pb * L::kV;
#pragma unroll
        for (int it = 0; it < ValTile::IT; ++it) {
          const int idx = mt + MT * it, r = idx / ValTile::VPR, c = (idx - r * ValTile::VPR) * ValTile::N;
          typename Vec16<T>::V x = R.V.x[it];
          const float bt = NOW ? sc[Scal::BETA + min(r, 63)] : R.bv[it];
#pragma unroll
          for (int e = 0; e < ValTile::N; ++e) x[e] = (bf16_t)((float)x[e] * bt);
          if (idx < ValTile::TOTAL) *reinterpret_cast<typename Vec16<T>::V*>(dst + r * LDV + c) = x;
        }
      }
      R.Tm.store(sTm + pb * L::kC);
      if (OUT && !NOW) R.P.store(sP + pb * L::kC);
      if (!NOW && mt < 64) put_scalars<GATE>(sSc + pb * L::SCS, mt, mt < R.len ? R.b : 0.f, R.g, R.gc);
    };
    // cur: the register set that held chunk n (in LDS since the last step) and now takes chunk n + 2; nxt: chunk n + 1.
    // `steady` (a std::bool_constant): chunks n + 1 and n + 2 exist, so nothing below sits behind a branch -- behind a
    // conditional fetch the compiler cannot count the younger loads in flight and would wait for all of them.
    // The loads are admitted at the rate the memory path takes them, and a wave that has a load waiting for a slot
    // issues nothing else: so the tile writes of chunk n + 1 sit between the loads of chunk n + 2, a tile at a time, and
    // go out while the loads before them drain (issued one after the other: forward scan 237 -> 216 us).
    // with 512 movers: O and D are 256 vectors each, one half of the movers takes each
    const bool lower = MT == 256 || mt < 256, upper = MT == 256 || mt >= 256;
    auto out_o = [&](int n) {
      int tok0, len;
      chunk_span(span, n, tok0, len);
      if constexpr (OUT && !NOW)
        if (p.o && lower) {
          const int ot = mt & 255;
          if constexpr (std::is_same<OT, float>::value)
            unstage_tile_checked_widen<64, BV>(reinterpret_cast<float*>(p.o) + tok_index(p.geom, row, tok0) * p.dv + v0, tso, sO, LDV, len, ot);
          else
            unstage_tile_checked<bf16_t, 64, BV>(reinterpret_cast<bf16_t*>(p.o) + tok_index(p.geom, row, tok0) * p.dv + v0, tso, sO, LDV, len, ot);
        }
    };
    auto out_state = [&](int n) {
      if constexpr (OUT)
        if (p.save) {
          const int64_t slot = (int64_t)row * N + n;
          unstage_tile<T, BV, DK, true, MT>(at<T>(p.ws, p.off.SnT) + slot * p.dv * DK + (int64_t)v0 * DK, DK, sST + (NOW ? ((n - c0) & 1) * L::kST : 0), LDS, BV, mt);
          if (upper) unstage_tile<T, BV, 64, true>(at<T>(p.ws, p.off.D) + slot * p.dv * 64 + (int64_t)v0 * 64, 64, sDT + (NOW ? ((n - c0) & 1) * L::kDT : 0), LDD, BV, mt & 255);
        }
    };
    auto step = [&](Tiles& cur, const Tiles& nxt, int n, auto steady, auto write_first) __attribute__((always_inline)) {
      constexpr bool STEADY = decltype(steady)::value, WRITE_FIRST = decltype(write_first)::value;
      auto carry = [&](int part) __attribute__((always_inline)) {
        const int lag = NOW && part == 1;
        if (WRITE_FIRST && (STEADY || n + 1 - lag < c1)) commit(nxt, n + 1, part);
        if (WRITE_FIRST) __builtin_amdgcn_sched_barrier(0);
        if (STEADY || n + 2 - lag < c1) fetch(cur, n + 2, part);
        if (!WRITE_FIRST && (STEADY || n + 1 - lag < c1)) commit(nxt, n + 1, part);
        if (STEADY) __builtin_amdgcn_sched_barrier(0);
      };
      if (NOW && n > c0) out_state(n - 1);
      if constexpr (OUT && !NOW && !STEADY) {  // the last chunks: every request before the first wait (8 chunks, 264 slabs: 163 -> 161 us a pass)
        if (n + 2 < c1) fetch(cur, n + 2);
        if (n + 1 < c1) commit(nxt, n + 1);
      } else {
        carry(0);
        if (OUT) carry(1);
        carry(2);
      }
      if constexpr (OUT && !NOW) {
        lds_barrier();  // Bmid
        out_o(n);
        out_state(n);
      }
      lds_barrier();  // B1 of the next chunk
    };
    // the register sets and the LDS double buffers alternate by position in the sequence (chunk c0: set a, buffer 0)
    if constexpr (NOW || !OUT) {
      if (c0 < c1) {
        fetch(ta, c0, 0), fetch(ta, c0, 2);
        if (NOW) lds_barrier();  // the first chunks' scalars are there
        commit(ta, c0, 0), commit(ta, c0, 2);
        if (OUT) fetch(tb, c0 + 1, 1);
      }
      if (c0 + 1 < c1) fetch(tb, c0 + 1, 0), fetch(tb, c0 + 1, 2);
    } else {
      if (c0 < c1) {
        fetch(ta, c0);
        commit(ta, c0);
      }
      if (c0 + 1 < c1) fetch(tb, c0 + 1);
    }
    lds_barrier();  // B1 of the first chunk
    auto run = [&](auto write_first) __attribute__((always_inline)) {
      int n = c0;
      for (; n + 3 < c1; n += 2) {  // chunks n + 2 and n + 3 exist
        step(ta, tb, n, std::true_type{}, write_first);
        step(tb, ta, n + 1, std::true_type{}, write_first);
      }
      for (; n < c1; n += 2) {
        step(ta, tb, n, std::false_type{}, write_first);
        if (n + 1 < c1) step(tb, ta, n + 1, std::false_type{}, write_first);
      }
    };
    // each SIMD has a wave of either order
    if (NOW && MT == 512 && mt >= 256) run(std::true_type{});
    else run(std::false_type{});
    if (NOW && c0 < c1) out_state(c1 - 1);
    return;
  }

  const int vs = 16 * (wave < NCW ? wave : wave - NCW);
  const int l16 = lane & 15, lr = S16::row(lane), g4 = S16::grp(lane);
  constexpr int NK = DK / 32;  // 32-wide steps over dk
  if constexpr (NOW > 0)
    if (wave >= NCW) {
      // ---------------- output waves: O^T = (Q~ S)^T + D^T Pm^T of a strip, lane = token ----------------
      // S^T and D^T as the compute wave stored them are the operands that it has in registers.
      auto acc_rows = [&](const T* tile, int ld, int ks) {
        const T* r = tile + (vs + l16) * ld + 32 * ks + g4;
        return S16::join(*reinterpret_cast<const bf16x4*>(r), *reinterpret_cast<const bf16x4*>(r + 8));
      };
      // They bring the scalars, too, the same from every output wave: those of chunk n + 3 go to LDS and those of chunk n + 4 are requested behind
      // the outputs of chunk n.  No load behind a branch: past the end the last chunk's come again.  Nor may the barrier that every wave waits at
      // stand behind a load just requested or a store: beta's choice waits until it is used, and the stores are range-checked instead of
      // branched around, so that the scalars are waited for by count (before: calls that exceed the 256 MiB cache, 16384 tokens forward only,
      // 32 heads 443 us, without a gate 450; so 398 and 378; without output waves 410 and 374).
      float b_ = 0.f, g_ = 0.f, gc_ = 0.f, nk_ = 0.f, fq_ = 0.f;  // beta, G, G_C, the factors of the K and Q rows
      int len_ = 0;                                               // past the end beta is 0
      auto fetch_scalars = [&](int n) {
        n = min(n, c1 - 1);
        const int64_t slot = (int64_t)row * N + n;
        int tok0;
        chunk_span(span, n, tok0, len_);
        b_ = p.beta[tok_index(p.geom, row, tok0) + (int64_t)min(lane, len_ - 1) * p.geom.ts];
        if (GATE == LNX_GATE_SCALAR) {
          const float* G = at<const float>(p.ws, p.off.G) + slot * 64;
          g_ = G[lane], gc_ = G[63];
        }
        nk_ = at<const float>(p.ws, p.off.Nk)[slot * 64 + lane];
        fq_ = at<const float>(p.ws, p.off.Fq)[slot * 64 + lane];
      };
      auto commit_scalars = [&](int n) {
        float* sc = sSc + ((n - c0) & (L::NSC - 1)) * L::SCS;
        put_scalars<GATE>(sc, lane, lane < len_ ? b_ : 0.f, g_, gc_);
        sc[Scal::NK + lane] = nk_, sc[Scal::FQ + lane] = fq_;
      };
      if (c0 < c1) {
        fetch_scalars(c0), commit_scalars(c0);
        fetch_scalars(c0 + 1), commit_scalars(c0 + 1);
        fetch_scalars(c0 + 2);
        lds_barrier();
      }
      lds_barrier();  // B1 of the first chunk
      if (c0 < c1) {
        commit_scalars(c0 + 2);
        fetch_scalars(c0 + 3);
      }
      int off[4];  // of the lane's pieces of O
#pragma unroll
      for (int i = 0; i < 4; ++i) off[i] = (int)(((16 * i + l16) * tso + vs + 4 * (lane >> 4)) * (int64_t)sizeof(OT));
      for (int n = c0; n < c1; ++n) {
        lds_barrier();  // B1 of the next chunk, or the end of the last
        const int pb = (n - c0) & 1;
        const T* sQc = sQ + pb * L::kK;
        const T* sPc = sP + pb * L::kC;
        int tok0, len;
        chunk_span(span, n, tok0, len);
        floatx4 o[4];
        S16::Frag fq[2][4], pm[6];
        auto load_q = [&](int ks) {
#pragma unroll
          for (int i = 0; i < 4; ++i) fq[ks & 1][i] = S16::load<CHAIN>(sQc + (16 * i + l16) * LDK + 32 * ks, lane);
        };
        S16::Frag b[NK];
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) b[ks] = acc_rows(sST + pb * L::kST, LDS, ks);
        load_q(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) {
          if (ks + 1 < NK) {
            load_q(ks + 1);
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) pm[i] = S16::load<CHAIN>(sPc + (16 * i + l16) * LDC, lane);
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) S16::mma(o[i], b[ks], fq[ks & 1][i]);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 2; i < 4; ++i) pm[i + 2] = S16::load<CHAIN>(sPc + (16 * i + l16) * LDC + 32, lane);
        const S16::Frag bd0 = acc_rows(sDT + pb * L::kDT, LDD, 0), bd1 = acc_rows(sDT + pb * L::kDT, LDD, 1);
#pragma unroll
        for (int i = 0; i < 4; ++i) S16::mma(o[i], bd0, pm[i]);
        S16::mma(o[2], bd1, pm[4]);
        S16::mma(o[3], bd1, pm[5]);
        const __amdgpu_buffer_rsrc_t rsrc =
            __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<OT*>(p.o) + tok_index(p.geom, row, tok0) * p.dv + v0, 0, (int)(len * tso * (int64_t)sizeof(OT)), 0x00020000);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bf16x4 x = pack_bf16x4(o[i]);
          if constexpr (std::is_same<OT, float>::value) {  // fp32 outputs are rounded as the others and widened
            typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
            const floatx4 y = {(float)x[0], (float)x[1], (float)x[2], (float)x[3]};
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, y), rsrc, off[i], 0, 0);
          } else {
            typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), rsrc, off[i], 0, 0);
          }
        }
        commit_scalars(n + 3);
        fetch_scalars(n + 4);
      }
      return;
    }

  // ---------------- compute waves: wave w owns value columns [16 w, 16 w + 16) of the slab ----------------
  floatx4 S[KT];
#pragma unroll
  for (int ci = 0; ci < KT; ++ci) S[ci] = floatx4{0.f, 0.f, 0.f, 0.f};
  if (!OUT && p.ident) {
    const int r = v0 + vs + l16 - p.vcols;
#pragma unroll
    for (int ci = 0; ci < KT; ++ci)
#pragma unroll
      for (int e = 0; e < 4; ++e) S[ci][e] = S16::row0(ci) + g4 + e == r ? 1.f : 0.f;
  } else if (p.s0) {
    const float* s0 = p.s0 + (int64_t)sidx * DK * p.dv + v0 + vs + l16;
#pragma unroll
    for (int ci = 0; ci < KT; ++ci)
#pragma unroll
      for (int e = 0; e < 4; ++e) S[ci][e] = s0[(int64_t)(S16::row0(ci) + g4 + e) * p.dv];
    // the loads complete here: left pending into the loop, every iteration would count them down again
#pragma unroll
    for (int ci = 0; ci < KT; ++ci)
#pragma unroll
      for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(S[ci][e]));
  }
  auto store_state = [&](int n) {
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) store_t(S[ci], sST + (NOW ? ((n - c0) & 1) * L::kST : 0) + vs * LDS + S16::row0(ci), LDS, lane);
  };
  if (NOW && c0 < c1) lds_barrier();
  lds_barrier();  // B1 of the first chunk
  // Every LDS read is issued well ahead of the product that consumes it (A fragments two steps ahead, the next
  // phase's first fragments and scalars during the current phase's last steps): a compute wave has nothing else to cover
  // the LDS latency with.  The scheduling fences pin that order.
  if constexpr (NOW || !OUT) {
    for (int n = c0; n < c1; ++n) {
      const int pb = (n - c0) & 1;
      const T* sKc = sK + pb * L::kK;
      const T* sVc = sV + pb * L::kV;
      const T* sTc = sTm + pb * L::kC;
      const float* sc = sSc + ((n - c0) & (L::NSC - 1)) * L::SCS;
      // ---- Y = K S (lane = value column) ----
      floatx4 y[4], d[4], sv[4];
      S16::Frag fa[NK][4], tm[6];  // K rows; Tm as below
      bf16x4 vr[4];
      auto load_k = [&](int ks) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fa[ks][i] = S16::load<CHAIN>(sKc + (S16::row0(i) + lr) * LDK + 32 * ks, lane);
      };
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = d[i] = floatx4{0.f, 0.f, 0.f, 0.f};
      load_k(0), load_k(1);
      if (NK > 2) load_k(NK > 2 ? 2 : 0);
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) {
        const S16::Frag b = S16::from_acc(S[2 * ks], S[2 * ks + 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) S16::mma(y[i], fa[ks][i], b);
        if (ks == 0 && NK > 2) load_k(NK > 2 ? 3 : 0);
        if (ks == (NK > 2 ? 1 : 0)) {
#pragma unroll
          for (int i = 0; i < 4; ++i) vr[i] = S16::rows4(sVc, LDV, S16::row0(i) + g4, vs, lane);
#pragma unroll
          for (int i = 0; i < 4; ++i) sv[i] = load4(sc + Scal::GAM + S16::row0(i) + g4);
        }
        if (ks == (NK > 2 ? 2 : 1)) {
#pragma unroll
          for (int i = 0; i < 4; ++i) tm[i] = S16::load<CHAIN>(sTc + (S16::row0(i) + lr) * LDC, lane);
#pragma unroll
          for (int i = 2; i < 4; ++i) tm[i + 2] = S16::load<CHAIN>(sTc + (S16::row0(i) + lr) * LDC + 32, lane);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      // ---- R = beta V - (beta e^G) Y, in place of Y; D = Tm R ----
      auto form_r = [&](int i) {
#pragma unroll
        for (int u = 0; u < 4; ++u) y[i][u] = (float)vr[i][u] - sv[i][u] * y[i][u];
      };
      form_r(0), form_r(1);
      const S16::Frag br0 = S16::from_acc(y[0], y[1]);
#pragma unroll
      for (int i = 0; i < 4; ++i) S16::mma(d[i], tm[i], br0);
      form_r(2), form_r(3);
      const S16::Frag br1 = S16::from_acc(y[2], y[3]);
      __builtin_amdgcn_sched_barrier(0);
      S16::mma(d[2], tm[4], br1);
      S16::mma(d[3], tm[5], br1);
      if (NOW) store_state(n);  // read behind the next barrier: it fills the wait for D
#pragma unroll
      for (int i = 0; i < 4; ++i) sv[i] = load4(sc + Scal::R + S16::row0(i) + g4);  // e^{G_C - G} for the state update
      const float dec = (GATE == LNX_GATE_SCALAR) ? sc[Scal::DEC] : 1.f;
      S16::Frag fu[2][KT];  // K^T fragments of the state update, [step][row tile of the state]
      constexpr int AHEAD = KT < 6 ? KT : 6;
#pragma unroll
      for (int ci = 0; ci < AHEAD; ++ci) fu[0][ci] = S16::load_cols<CHAIN>(sKc, LDK, 0, ci, lane);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (OUT) {
#pragma unroll
        for (int i = 0; i < 4; ++i) store_t(d[i], sDT + pb * L::kDT + vs * LDD + S16::row0(i), LDD, lane);
      }
      const S16::Frag bu0 = S16::from_acc(d[0] * sv[0], d[1] * sv[1]), bu1 = S16::from_acc(d[2] * sv[2], d[3] * sv[3]);
      if (GATE == LNX_GATE_SCALAR) {
#pragma unroll
        for (int ci = 0; ci < KT; ++ci) S[ci] *= dec;
      }
      __builtin_amdgcn_sched_barrier(0);
      // ---- S <- e^{G_C} S + K^T (e^{G_C - G} D) ----
#pragma unroll
      for (int ci = AHEAD; ci < KT; ++ci) fu[0][ci] = S16::load_cols<CHAIN>(sKc, LDK, 0, ci, lane);
#pragma unroll
      for (int ci = 0; ci < 4; ++ci) fu[1][ci] = S16::load_cols<CHAIN>(sKc, LDK, 32, ci, lane);
#pragma unroll
      for (int ci = 0; ci < 4; ++ci) S16::mma(S[ci], fu[0][ci], bu0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ci = 4; ci < KT; ++ci) fu[1][ci] = S16::load_cols<CHAIN>(sKc, LDK, 32, ci, lane);
#pragma unroll
      for (int ci = 4; ci < KT; ++ci) S16::mma(S[ci], fu[0][ci], bu0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ci = 0; ci < KT; ++ci) S16::mma(S[ci], fu[1][ci], bu1);
      lds_barrier();  // B1 of the next chunk
    }
  } else {
  for (int n = c0; n < c1; ++n) {
    const int pb = (n - c0) & 1;
    const T* sKc = sK + pb * L::kK;
    const T* sQc = sQ + pb * L::kK;
    const T* sVc = sV + pb * L::kV;
    const T* sTc = sTm + pb * L::kC;
    const T* sPc = sP + pb * L::kC;
    const float* sc = sSc + pb * L::SCS;
    if (p.save) store_state(n);
    // ---- Y = K S (lane = value column) and (Q~ S)^T (lane = token): the state fragments are the shared operand ----
    floatx4 y[4], o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    S16::Frag fa[2][4], fb[2][4];  // [step mod 2][token tile]
    bf16x4 vr[4];                  // beta V at this lane's accumulator positions
    floatx4 sv[4];                 // per-row scalars at this lane's accumulator positions: beta e^G, later e^{G_C - G}
    S16::Frag tm[6], pm[6];        // [token tile, step]: (0,0) (1,0) (2,0) (3,0) (2,1) (3,1): Tm and Pm are lower-triangular
#pragma unroll
    for (int i = 0; i < 4; ++i) fa[0][i] = S16::load<CHAIN>(sKc + (S16::row0(i) + lr) * LDK, lane);
#pragma unroll
    for (int i = 0; i < 4; ++i) fb[0][i] = S16::load<CHAIN>(sQc + (16 * i + l16) * LDK, lane);
    // at most 16 LDS reads are in flight (the wave's counter ends at 15): K of the next step goes out ahead of this step's
    // products, Q behind them
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      const S16::Frag b = S16::from_acc(S[2 * ks], S[2 * ks + 1]);
      if (ks + 1 < NK) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fa[(ks + 1) & 1][i] = S16::load<CHAIN>(sKc + (S16::row0(i) + lr) * LDK + 32 * (ks + 1), lane);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) vr[i] = S16::rows4(sVc, LDV, S16::row0(i) + g4, vs, lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) sv[i] = load4(sc + Scal::GAM + S16::row0(i) + g4);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) S16::mma(y[i], fa[ks & 1][i], b);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; ++i) S16::mma(o[i], b, fb[ks & 1][i]);
      if (ks + 1 < NK) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fb[(ks + 1) & 1][i] = S16::load<CHAIN>(sQc + (16 * i + l16) * LDK + 32 * (ks + 1), lane);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) tm[i] = S16::load<CHAIN>(sTc + (S16::row0(i) + lr) * LDC, lane);
#pragma unroll
        for (int i = 2; i < 4; ++i) tm[i + 2] = S16::load<CHAIN>(sTc + (S16::row0(i) + lr) * LDC + 32, lane);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- R = beta V - (beta e^G) Y, in place of Y; D = Tm R: the first half of the rows takes the first 32 tokens only ----
    auto form_r = [&](int i) {
#pragma unroll
      for (int u = 0; u < 4; ++u) y[i][u] = (float)vr[i][u] - sv[i][u] * y[i][u];
    };
    floatx4 d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    form_r(0), form_r(1);
    const S16::Frag br0 = S16::from_acc(y[0], y[1]);
#pragma unroll
    for (int i = 0; i < 4; ++i) S16::mma(d[i], tm[i], br0);
    form_r(2), form_r(3);
    const S16::Frag br1 = S16::from_acc(y[2], y[3]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) pm[i] = S16::load<CHAIN>(sPc + (16 * i + l16) * LDC, lane);
    S16::mma(d[2], tm[4], br1);
    S16::mma(d[3], tm[5], br1);
#pragma unroll
    for (int i = 0; i < 4; ++i) sv[i] = load4(sc + Scal::R + S16::row0(i) + g4);  // e^{G_C - G} for the state update
    const float dec = (GATE == LNX_GATE_SCALAR) ? sc[Scal::DEC] : 1.f;
    __builtin_amdgcn_sched_barrier(0);
    // ---- O^T = (Q~ S)^T + D^T Pm^T ----
    const S16::Frag bd0 = S16::from_acc(d[0], d[1]);
#pragma unroll
    for (int i = 2; i < 4; ++i) pm[i + 2] = S16::load<CHAIN>(sPc + (16 * i + l16) * LDC + 32, lane);
#pragma unroll
    for (int i = 0; i < 4; ++i) S16::mma(o[i], bd0, pm[i]);
    S16::Frag fu[2][KT];  // K^T fragments of the state update, [step][row tile of the state]
#pragma unroll
    for (int ci = 0; ci < 4; ++ci) fu[0][ci] = S16::load_cols<CHAIN>(sKc, LDK, 0, ci, lane);
#pragma unroll
    for (int i = 0; i < 4; ++i) store_t(d[i], sDT + vs * LDD + S16::row0(i), LDD, lane);  // also when nothing is saved: a branch here would split the schedule
    const S16::Frag bd1 = S16::from_acc(d[2], d[3]);
    S16::mma(o[2], bd1, pm[4]);
    S16::mma(o[3], bd1, pm[5]);
    // the state update's operand while the last products finish: D rows scaled by e^{G_C - G}
    const S16::Frag bu0 = S16::from_acc(d[0] * sv[0], d[1] * sv[1]), bu1 = S16::from_acc(d[2] * sv[2], d[3] * sv[3]);
    if (GATE == LNX_GATE_SCALAR) {
#pragma unroll
      for (int ci = 0; ci < KT; ++ci) S[ci] *= dec;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) store4(sO + (16 * i + l16) * LDV + vs + 4 * (lane >> 4), o[i]);  // [token][value column]
    lds_barrier();  // Bmid
    // ---- S <- e^{G_C} S + K^T (e^{G_C - G} D) ----
#pragma unroll
    for (int ci = 4; ci < KT; ++ci) fu[0][ci] = S16::load_cols<CHAIN>(sKc, LDK, 0, ci, lane);
#pragma unroll
    for (int ci = 0; ci < 4; ++ci) S16::mma(S[ci], fu[0][ci], bu0);
#pragma unroll
    for (int ci = 0; ci < 4; ++ci) fu[1][ci] = S16::load_cols<CHAIN>(sKc, LDK, 32, ci, lane);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ci = 4; ci < KT; ++ci) S16::mma(S[ci], fu[0][ci], bu0);
#pragma unroll
    for (int ci = 4; ci < KT; ++ci) fu[1][ci] = S16::load_cols<CHAIN>(sKc, LDK, 32, ci, lane);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) S16::mma(S[ci], fu[1][ci], bu1);
    lds_barrier();  // B1 of the next chunk
  }
  }
  float* out = p.sT_out.at(sidx, (int64_t)DK * p.dv) + v0 + vs + l16;
#pragma unroll
  for (int ci = 0; ci < KT; ++ci)
#pragma unroll
    for (int e = 0; e < 4; ++e) out[(int64_t)(S16::row0(ci) + g4 + e) * p.dv] = S[ci][e];
}

template <int DK, int GATE, typename OT>
int launch_scan_fwd(const DirectParams& p, int nstate, hipStream_t st) {
  constexpr bool OUT = !std::is_void<OT>::value;
  // 32-column slabs (two compute waves) when 64-column ones would occupy at most half of the chip
  const bool narrow = lnx_narrow_slabs((int64_t)nstate * p.geom.H * (p.dv / 64), p.slab);
  auto k = narrow ? scan_fwd_kernel<DK, GATE, 32, OT> : scan_fwd_kernel<DK, GATE, 64, OT>;
  const size_t b = narrow ? FScanL<DK, 32, OUT>::bytes : FScanL<DK, 64, OUT>::bytes;
  const int bv = narrow ? 32 : 64, threads = narrow ? FScanL<DK, 32, OUT>::threads : FScanL<DK, 64, OUT>::threads;
  if (const int rc = lnx_lds_limit((const void*)k, b); rc != LNX_OK) return rc;
  lnx_profile_mark("chunk_scan", st);
  hipLaunchKernelGGL(k, dim3(lnx_xcd_grid((int64_t)nstate * p.geom.H, p.dv / bv)), dim3(threads), b, st, p);
  lnx_profile_mark(nullptr, st);
  return LNX_OK;
}

// ---------------------------------------------------------------------------------------
// scan_bwd: the reverse pass, same organisation as scan_fwd.  A compute wave owns a 16-column strip of dS (the
// gradient of the state leaving the chunk); the chain  dS' -> Z = K dS' -> dD -> dR = Tm^T dD -> dY -> dS  stays in
// its registers.  Needs no forward state: only K, Q, dO, Tm, Pm and the per-token scalars.
//   B1    buffers of chunk n complete           compute: dS'^T -> LDS (saved), Z, Pm^T dO, dD, dR (-> LDS, transposed),
//                                                        dv = beta dR -> LDS, dY
//                                               movers:  loads of chunk n - 2; chunk n - 1 -> the other buffers
//   Bmid  dS'^T, dR^T and dv are in LDS         compute: dS update          movers: dS'^T, dR^T -> workspace, dv out
// ---------------------------------------------------------------------------------------
template <int DK, int BVW> struct BScanL {
  // 32-column slabs are taken where the chip has room for more workgroups, so what counts there is the time of a chunk's
  // chain: operand tiles in chain order, rows 32 bytes off a multiple of 64 (Mma16).  64-column slabs are bound by what the
  // movers carry.
  static constexpr bool CHAIN = BVW == 32;
  static constexpr int BV = BVW, PAD = M::PAD, OPAD = CHAIN ? 16 : 8, LDK = DK + OPAD, LDC = LNX_C + OPAD, LDV = BV + PAD, NCW = BV / 16, MT = 256;
  static constexpr int LDS = DK + PAD, LDD = LNX_C + PAD;  // of the tiles on their way out: states, D or dR
  static constexpr int kK = 64 * LDK, kST = BV * LDS, kV = 64 * LDV, kC = 64 * LDC;
  static constexpr int kDT = BV * LDD;
  // [2] x (K, scaled Q, dO, Tm, Pm) | dS'^T | dR^T | dv | scalars [2]
  static constexpr size_t bytes = sizeof(T) * (2 * (2 * kK + kV + 2 * kC) + kST + kDT + kV) + sizeof(float) * 2 * Scal::SIZE;
  static constexpr int threads = 64 * NCW + MT;
};

template <int DK, int GATE, int BVW>
__global__ __launch_bounds__((BScanL<DK, BVW>::threads)) void scan_bwd_kernel(DirectParams p) {
  typedef BScanL<DK, BVW> L;
  constexpr int LDK = L::LDK, LDC = L::LDC, BV = L::BV, LDV = L::LDV, NCW = L::NCW, LDS = L::LDS, LDD = L::LDD;
  constexpr bool CHAIN = L::CHAIN;
  constexpr int MT = L::MT;  // mover threads
  constexpr int KT = DK / 16;
  extern __shared__ __align__(16) char smem[];
  T* sK = reinterpret_cast<T*>(smem);  // [2][64][LDK]
  T* sQ = sK + 2 * L::kK;              // rows scaled by scale e^G
  T* sdO = sQ + 2 * L::kK;             // [2][64][LDV]
  T* sTm = sdO + 2 * L::kV;
  T* sP = sTm + 2 * L::kC;
  T* sdST = sP + 2 * L::kC;            // dS'^T [v][dk] on its way to the workspace
  T* sdRT = sdST + L::kST;             // dR^T [v][token] on its way to the workspace
  T* sdV = sdRT + L::kDT;              // dv = beta dR [token][v] on its way out
  float* sSc = reinterpret_cast<float*>(sdV + L::kV);

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int N = p.geom.N;
  int sidx, row, seq;
  int64_t chain;
  int slab;
  if (!xcd_slot_part((int64_t)(p.geom.tab ? p.geom.nseq : p.geom.rows / p.geom.H) * p.geom.H, p.dv / BV, chain, slab)) return;
  scan_state(p.geom, (int)chain, sidx, row, seq);
  const int v0 = slab * BV;
  int c0, c1;
  seq_chunks(p.geom, seq, c0, c1);
  const SeqSpan span = seq_span(p.geom, seq, c0);
  const int64_t tsk = (int64_t)p.geom.ts * DK, tsv = (int64_t)p.geom.ts * p.dv;

  if (wave >= NCW) {
    // ---------------- movers ----------------
    const int mt = tid - 64 * NCW;
    typedef TileRegs<T, 64, DK, MT> RowTile;
    struct Tiles {
      RowTile K, Q;
      TileRegs<T, 64, BV, MT> dO;
      TriRegs<T, CHAIN, MT> Tm, P;  // lower-triangular tiles, packed in the workspace
      float g, gc, b;  // per-token scalars of token mt % 64
      float fq[RowTile::IT], nk[RowTile::IT];  // factors of the token each of this thread's Q / K vectors belongs to
      int len;
    };
    Tiles ta, tb;
    ta.g = ta.gc = ta.b = tb.g = tb.gc = tb.b = 0.f;
    ta.Tm.init(LDC, mt), ta.P.init(LDC, mt), tb.Tm.init(LDC, mt), tb.P.init(LDC, mt);
    zero_upper_triangles<CHAIN>(sTm, 4, L::kC, LDC, mt);  // both buffers of Tm and Pm: the packed tiles never write there
    ta.len = tb.len = 0;
#pragma unroll
    for (int it = 0; it < RowTile::IT; ++it) ta.fq[it] = tb.fq[it] = ta.nk[it] = tb.nk[it] = 0.f;
    auto fetch = [&](Tiles& R, int n, int part = -1) {  // part 0: K, 1: Q, 2: the rest; < 0: everything
      const int64_t slot = (int64_t)row * N + n;
      int tok0;
      chunk_span(span, n, tok0, R.len);
      const int64_t tbase = tok_index(p.geom, row, tok0);
      if (part < 0 || part == 0) R.K.load(p.k + tbase * DK, tsk, R.len, mt);
      if (part < 0 || part == 1) R.Q.load(p.q + tbase * DK, tsk, R.len, mt);
      if (part == 0 || part == 1) return;
      R.dO.load(p.d_o + tbase * p.dv + v0, tsv, R.len, mt);
      R.Tm.load(at<const T>(p.ws, p.off.Tm) + slot * 64 * 64, mt);
      R.P.load(at<const T>(p.ws, p.off.P) + slot * 64 * 64, mt);
      const int t = mt & 63;
      if (GATE == LNX_GATE_SCALAR) {
        const float* G = at<const float>(p.ws, p.off.G) + slot * 64;
        R.g = G[t];
        R.gc = G[63];
      }
#pragma unroll
      for (int it = 0; it < RowTile::IT; ++it) {
        R.fq[it] = at<const float>(p.ws, p.off.Fq)[slot * 64 + (mt + MT * it) / RowTile::VPR];
        R.nk[it] = at<const float>(p.ws, p.off.Nk)[slot * 64 + (mt + MT * it) / RowTile::VPR];
      }
      R.b = p.beta[tbase + (int64_t)min(t, R.len - 1) * p.geom.ts];
    };
    // K rows normalised (their own bits where nothing is to be normalised), Q rows normalised and scaled by scale e^{G_i}
    auto commit = [&](const Tiles& R, int pb, int part = -1) {
#pragma unroll
      for (int it = 0; it < RowTile::IT; ++it) {
        const int idx = mt + MT * it, r = idx / RowTile::VPR, c = (idx - r * RowTile::VPR) * RowTile::N;
        if (part < 0 || part == 0)
          S16::put<CHAIN>(sK + pb * L::kK + r * LDK + S16::pos<CHAIN>(c), p.l2norm ? scaled(R.K.x[it], R.nk[it]) : R.K.x[it]);
        if (part < 0 || part == 1)
          S16::put<CHAIN>(sQ + pb * L::kK + r * LDK + S16::pos<CHAIN>(c), scaled(R.Q.x[it], R.fq[it]));
      }
      if (part == 0 || part == 1) return;
      R.dO.store(sdO + pb * L::kV, LDV, mt);
      R.Tm.store(sTm + pb * L::kC);
      R.P.store(sP + pb * L::kC);
      if (mt < 64) {
        float* sc = sSc + pb * Scal::SIZE;
        const float gam = (GATE == LNX_GATE_SCALAR) ? __expf(R.g) : 1.f;
        const float bt = (mt < R.len) ? R.b : 0.f;
        sc[Scal::BETA + mt] = bt;
        sc[Scal::GAM + mt] = bt * gam;  // dY = -(beta e^G) dR
        sc[Scal::R + mt] = (GATE == LNX_GATE_SCALAR) ? __expf(fminf(R.gc - R.g, 0.f)) : 1.f;
        if (mt == 0) sc[Scal::DEC] = (GATE == LNX_GATE_SCALAR) ? __expf(R.gc) : 1.f;
      }
    };
    // cur: the register set that held chunk n and now takes chunk n - 2; nxt: chunk n - 1 (see scan_fwd)
    auto step = [&](Tiles& cur, const Tiles& nxt, int n, auto steady) {
      constexpr bool STEADY = decltype(steady)::value;
      const int pbn = (c1 - n) & 1;  // position of chunk n - 1 from the end: c1 - 1 - (n - 1)
      if constexpr (STEADY) {  // tile writes between the loads, a tile at a time (see scan_fwd)
#pragma unroll
        for (int part = 0; part < 3; ++part) {
          fetch(cur, n - 2, part);
          commit(nxt, pbn, part);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        if (n - 2 >= c0) fetch(cur, n - 2);
        if (n - 1 >= c0) commit(nxt, pbn);
      }
      lds_barrier();  // Bmid
      const int64_t slot = (int64_t)row * N + n;
      unstage_tile<T, BV, DK, true, MT>(at<T>(p.ws, p.off.dSn) + slot * p.dv * DK + (int64_t)v0 * DK, DK, sdST, LDS, BV, mt);
      unstage_tile<T, BV, 64, true>(at<T>(p.ws, p.off.dD) + slot * p.dv * 64 + (int64_t)v0 * 64, 64, sdRT, LDD, BV, mt);
      int tok0, len;
      chunk_span(span, n, tok0, len);
      unstage_tile_checked<T, 64, BV>(p.dv_out + tok_index(p.geom, row, tok0) * p.dv + v0, tsv, sdV, LDV, len, mt);
      lds_barrier();  // B1 of the next chunk
    };
    if (c0 < c1) {
      fetch(ta, c1 - 1);
      commit(ta, 0);
    }
    if (c1 - 2 >= c0) fetch(tb, c1 - 2);
    lds_barrier();  // B1 of the first chunk
    int n = c1 - 1;
    for (; n - 3 >= c0; n -= 2) {  // chunks n - 2 and n - 3 exist
      step(ta, tb, n, std::true_type{});
      step(tb, ta, n - 1, std::true_type{});
    }
    for (; n >= c0; n -= 2) {
      step(ta, tb, n, std::false_type{});
      if (n - 1 >= c0) step(tb, ta, n - 1, std::false_type{});
    }
    return;
  }

  // ---------------- compute waves ----------------
  const int vs = 16 * wave;
  const int l16 = lane & 15, lr = S16::row(lane), g4 = S16::grp(lane);
  floatx4 dS[KT];
#pragma unroll
  for (int ci = 0; ci < KT; ++ci) dS[ci] = floatx4{0.f, 0.f, 0.f, 0.f};
  if (p.d_sT) {
    const float* src = p.d_sT + (int64_t)sidx * DK * p.dv + v0 + vs + l16;
#pragma unroll
    for (int ci = 0; ci < KT; ++ci)
#pragma unroll
      for (int e = 0; e < 4; ++e) dS[ci][e] = src[(int64_t)(S16::row0(ci) + g4 + e) * p.dv];
#pragma unroll
    for (int ci = 0; ci < KT; ++ci)
#pragma unroll
      for (int e = 0; e < 4; ++e) asm volatile("" : "+v"(dS[ci][e]));  // complete here, as in scan_fwd
  }
  lds_barrier();  // B1 of the first chunk
  // LDS reads are issued ahead of the products that consume them, as in scan_fwd.  The products that do not depend on
  // the incoming dS' (Pm^T dO, Q~^T dO) fill the gaps of the chain  dS' -> Z -> dD -> dR -> dY -> dS.
  constexpr int NK = DK / 32;
  for (int n = c1 - 1; n >= c0; --n) {
    const int pb = (c1 - 1 - n) & 1;
    const T* sKc = sK + pb * L::kK;
    const T* sQc = sQ + pb * L::kK;
    const T* sOc = sdO + pb * L::kV;
    const T* sTc = sTm + pb * L::kC;
    const T* sPc = sP + pb * L::kC;
    const float* sc = sSc + pb * Scal::SIZE;
    S16::Frag fa[2][4];  // K rows, [step mod 2][token tile]
    S16::Frag ft[6];     // Pm^T, then Tm^T: [token tile, step] (0,1) (1,1) (2,1) (3,1) (0,0) (1,0): upper-triangular
    S16::Frag fo[2];     // dO
    floatx4 sv[4];       // per-row scalars at this lane's accumulator positions: e^{G_C - G}, later beta e^G
    auto load_tri = [&](const T* tile, auto natural) {
      constexpr bool NATURAL = decltype(natural)::value;
#pragma unroll
      for (int i = 0; i < 4; ++i) ft[i] = S16::load_cols<CHAIN, NATURAL>(tile, LDC, 32, i, lane);
#pragma unroll
      for (int i = 0; i < 2; ++i) ft[i + 4] = S16::load_cols<CHAIN, NATURAL>(tile, LDC, 0, i, lane);
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) fa[0][i] = S16::load<CHAIN>(sKc + (S16::row0(i) + lr) * LDK, lane);
#pragma unroll
    for (int s_ = 0; s_ < 2; ++s_) fo[s_] = S16::load_t(sOc, LDV, 32 * s_, vs, lane);
    // the state gradient as the B operand of Z = K dS'; its accumulators are then free to take the next dS
    S16::Frag bs[NK];
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) bs[ks] = S16::from_acc(dS[2 * ks], dS[2 * ks + 1]);
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) store_t(dS[ci], sdST + vs * LDS + S16::row0(ci), LDS, lane);
    const float dec = (GATE == LNX_GATE_SCALAR) ? sc[Scal::DEC] : 1.f;
    // ---- Z = K dS' and the chunk-local part Pm^T dO ----
    floatx4 z[4], dd[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) z[i] = dd[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      if (ks + 1 < NK) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fa[(ks + 1) & 1][i] = S16::load<CHAIN>(sKc + (S16::row0(i) + lr) * LDK + 32 * (ks + 1), lane);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) sv[i] = load4(sc + Scal::R + S16::row0(i) + g4);
      }
      if (ks == 0) load_tri(sPc, std::true_type{});
#pragma unroll
      for (int i = 0; i < 4; ++i) S16::mma(z[i], fa[ks & 1][i], bs[ks]);
      if (ks == NK - 1) {
#pragma unroll
        for (int i = 0; i < 2; ++i) S16::mma(dd[i], ft[i + 4], fo[0]);
#pragma unroll
        for (int i = 0; i < 4; ++i) S16::mma(dd[i], ft[i], fo[1]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- dS <- e^{G_C} dS' + (scale e^G Q)^T dO fills the wait for Z; Tm^T is fetched behind it ----
    S16::Frag fq[2][KT];
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) fq[0][ci] = S16::load_cols<CHAIN, true>(sQc, LDK, 0, ci, lane);
    load_tri(sTc, std::false_type{});
    if (GATE == LNX_GATE_SCALAR) {
#pragma unroll
      for (int ci = 0; ci < KT; ++ci) dS[ci] *= dec;
    }
    // ---- dD = Pm^T dO + e^{G_C - G} Z ----
#pragma unroll
    for (int i = 0; i < 4; ++i) dd[i] += sv[i] * z[i];
    S16::Frag bd0 = S16::from_acc(dd[0], dd[1]), bd1 = S16::from_acc(dd[2], dd[3]);
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) S16::mma(dS[ci], fq[0][ci], fo[0]);
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) fq[1][ci] = S16::load_cols<CHAIN, true>(sQc, LDK, 32, ci, lane);
#pragma unroll
    for (int i = 0; i < 4; ++i) sv[i] = load4(sc + Scal::GAM + S16::row0(i) + g4);
    __builtin_amdgcn_sched_barrier(0);
    // ---- dR = Tm^T dD (lane = value column, in z) and once more with the operands exchanged (lane = token, in dd), which
    //      is the orientation dv = beta dR leaves in ----
#pragma unroll
    for (int i = 0; i < 4; ++i) z[i] = dd[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 2; ++i) S16::mma(z[i], ft[i + 4], bd0);
#pragma unroll
    for (int i = 0; i < 2; ++i) S16::mma(dd[i], bd0, ft[i + 4]);
#pragma unroll
    for (int i = 0; i < 4; ++i) S16::mma(z[i], ft[i], bd1);
#pragma unroll
    for (int i = 0; i < 4; ++i) S16::mma(dd[i], bd1, ft[i]);
    S16::Frag fu[2][KT];  // K^T fragments of the dS update
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) fu[0][ci] = S16::load_cols<CHAIN>(sKc, LDK, 0, ci, lane);
    float bl[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) bl[i] = sc[Scal::BETA + S16::row0(i) + lr];
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) S16::mma(dS[ci], fq[1][ci], fo[1]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) store_t(z[i], sdRT + vs * LDD + S16::row0(i), LDD, lane);
    // dY = -beta e^G dR
    bd0 = S16::from_acc(-sv[0] * z[0], -sv[1] * z[1]);
    bd1 = S16::from_acc(-sv[2] * z[2], -sv[3] * z[3]);
    // dv = beta dR: tile dd[i] holds tokens 16 i .. (one per lane) x the strip's value columns
#pragma unroll
    for (int i = 0; i < 4; ++i) store4(sdV + (S16::row0(i) + lr) * LDV + vs + 4 * (lane >> 4), dd[i] * bl[i]);
    lds_barrier();  // Bmid
    // ---- dS += K^T dY ----
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) fu[1][ci] = S16::load_cols<CHAIN>(sKc, LDK, 32, ci, lane);
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) S16::mma(dS[ci], fu[0][ci], bd0);
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) S16::mma(dS[ci], fu[1][ci], bd1);
    lds_barrier();  // B1 of the next chunk
  }
  if (p.ds0) {
    float* out = p.ds0 + (int64_t)sidx * DK * p.dv + v0 + vs + l16;
#pragma unroll
    for (int ci = 0; ci < KT; ++ci)
#pragma unroll
      for (int e = 0; e < 4; ++e) out[(int64_t)(S16::row0(ci) + g4 + e) * p.dv] = dS[ci][e];
  }
}

template <int DK, int GATE>
int launch_scan_bwd(const DirectParams& p, int nstate, hipStream_t st) {
  const bool narrow = lnx_narrow_slabs((int64_t)nstate * p.geom.H * (p.dv / 64), p.slab);
  auto k = narrow ? scan_bwd_kernel<DK, GATE, 32> : scan_bwd_kernel<DK, GATE, 64>;
  const size_t b = narrow ? BScanL<DK, 32>::bytes : BScanL<DK, 64>::bytes;
  const int bv = narrow ? 32 : 64, threads = narrow ? BScanL<DK, 32>::threads : BScanL<DK, 64>::threads;
  if (const int rc = lnx_lds_limit((const void*)k, b); rc != LNX_OK) return rc;
  lnx_profile_mark("bwd_scan", st);
  hipLaunchKernelGGL(k, dim3(lnx_xcd_grid((int64_t)nstate * p.geom.H, p.dv / bv)), dim3(threads), b, st, p);
  return LNX_OK;
}

// ---------------------------------------------------------------------------------------
// bwd_chunk: the chunk-local gradients, one workgroup per chunk, all chunks in parallel.  Reads q, k, v, dO of the
// chunk, the states S (entering) and dS' (leaving) and D, dR from the two scans; writes dq, dk, dbeta, dg (dv left
// the reverse scan).  A loop over 32-column slabs of the value dimension accumulates every product that contracts
// over value columns; the slabs arrive in two LDS buffers through loads that bypass the registers, two slabs ahead:
//   dQa = dO S^T     dK1 = dR S^T     dK2 = D dS'^T     dPm = dO D^T     dAm = dR D^T     <dR_t, v_t>     <dS', S>
// then an epilogue over the chunk's tokens:
//   dPe = scale tril(E * dPm)          dXa = -tril(E * dAm, -1)          dXe = diag(beta) dXa
//   dq  = scale e^G dQa + dPe K
//   row = dXa K - e^G dK1              m_t = <k_t, row_t>                 dbeta = <dR, v> + m
//   dk  = beta row + e^{G_C - G} dK2 + dPe^T Q + dXe^T K
//   dG  = <q, dq> - <k, dk> + 2 beta m;   dG_C += sum_t e^{G_C - G_t} <k_t, dK2_t> + e^{G_C} <dS', S>;   dg = reverse cumsum(dG)
// Wave (wi, wj) owns the token-row tile wi and the key-column tiles NKT wj .. of the [64 x dk] accumulators and the
// (wi, wj) tile of the [64 x 64] ones.  The epilogue's tiles that are only read through transposing LDS loads get a row
// stride of 64 bytes mod 256, which spreads the four rows that half a wave reads over all banks.
// Measured per workgroup at B8 H16 T4096 d128 (wall clock of wave 0, 2 workgroups per CU): 4.3 us until the first slab
// is there, 6.2 us for the loop, 2.1 us staging K, Q and the four small tiles, 1.8 us for the epilogue's products and
// 3.4 us until dq, dk have left -- memory latency at every step; the kernel moves 4.9 TB/s.
// dk = 256: 896 KB a chunk at dv = 512, most of it the two states; B8 H8 T4096 788 - 795 us, 4.8 TB/s.
// ---------------------------------------------------------------------------------------
template <int DK> struct BChunkL {
  // dk = 256: eight waves, one workgroup per CU -- the [64 x dk] accumulators of four would take 192 registers, the slabs of two
  // workgroups more LDS than there is -- and a third slab buffer, for nobody else's loads are in flight while this workgroup multiplies
  static constexpr int NW = DK == 256 ? 8 : 4, THREADS = 64 * NW, NBUF = DK == 256 ? 3 : 2;
  static constexpr int SV = 32;
  static constexpr int SC = DK < 128 ? DK : 128, NH = DK / SC;  // a state slab is NH tiles of SC columns
  typedef SwzTile<64, SV> TokT;            // dO, V slabs [64][SV], read by rows
  typedef SwzTile<SV, 64, false> TrT;      // D^T, dR^T slabs [SV][64], transposing reads only
  typedef SwzTile<SV, SC, false> StT;      // S^T, dS'^T slabs [SV][SC], transposing reads only
  static constexpr int LDKT = DK + 32;     // the epilogue's K, Q tiles [64][DK], transposing reads
  static constexpr int LDC = 64 + 8;       // dPe, dPe^T, dXa, dXe^T [64][64], read by rows
  static constexpr int LDK = DK + 8;       // staging tile for dq, dk [64][DK]
  static constexpr int kC = 64 * LDC, kRow = 64 * LDKT, kSt = 64 * LDK;
  // one slab of the loop: dO | V | D^T | dR^T | S^T | dS'^T, unpadded; NBUF of them, filled by LDS-direct loads in turn
  static constexpr int oV = TokT::BYTES, oDT = 2 * TokT::BYTES, odRT = oDT + TrT::BYTES, oSn = odRT + TrT::BYTES, odSn = oSn + NH * StT::BYTES;
  static constexpr int slab_bytes = odSn + NH * StT::BYTES;
  static constexpr size_t loop_bytes = NBUF * slab_bytes;
  // the staging tiles of dq and dk: over dPe and dPe^T, over dXa and dXe^T; dk = 256: dq over all four, dk's behind the Q tile
  static constexpr bool OVER2 = DK <= 128;
  static constexpr size_t epi_bytes = sizeof(T) * (2 * kRow + 4 * kC + (OVER2 ? 0 : kSt));
  static_assert(kSt <= (OVER2 ? 2 : 4) * kC, "the staging tile overlays the small tiles");
  // The gate gradient's row dots <q_t, dq_t> - <k_t, dk_t> from the accumulators, before anything is rounded (what one pair of tokens gives
  // to both cancels along the chunk): dg is 4.0e-3 off instead of 6.5e-3.  dk <= 128 takes them from the staged rows, which its
  // emit reads anyway: 7.0e-3.  The accumulators would halve that, too, but move the sums over all tokens that callers form of dg (A_log's and
  // dt_bias' gradients, whose terms nearly cancel) by up to 3 %, as much as they are off: a change of results, left.
  static constexpr bool DOTS = DK == 256;
  static constexpr int nfloat = 64 * 10;
  static constexpr size_t bytes = sizeof(float) * nfloat + (epi_bytes > loop_bytes ? epi_bytes : loop_bytes);
  static_assert(bytes <= (NW == 4 ? 80 : 160) * 1024, "two workgroups of four waves per CU, one of eight");
};

template <int DK, int GATE>
__global__ __launch_bounds__(BChunkL<DK>::THREADS, 2) void bwd_chunk_kernel(DirectParams p) {
  typedef BChunkL<DK> L;
  constexpr int SV = L::SV, LDKT = L::LDKT, LDC = L::LDC, LDK = L::LDK, NW = L::NW, THREADS = L::THREADS, NBUF = L::NBUF, SC = L::SC, NH = L::NH;
  typedef typename L::TokT TokT;
  typedef typename L::TrT TrT;
  typedef typename L::StT StT;
  constexpr int NKT = DK / (16 * NW);  // key-column tiles per wave
  constexpr int NPA = 8 / NW;          // of dPm's and dAm's eight tiles: one of each per wave, or one of either
  constexpr int TPT = THREADS / 64;    // threads per token where rows are summed
  extern __shared__ __align__(16) char smem[];
  float* sG = reinterpret_cast<float*>(smem);
  float* sBeta = sG + 64;
  float* sRdv = sBeta + 64;   // <dR_t, v_t>
  float* sM = sRdv + 64;      // [2]: m_t is the sum of the two
  float* sdG = sM + 128;      // [2]: <q_t, dq_t> - <k_t, dk_t> is the sum of the two
  float* sMisc = sdG + 128;    // [8 + wave] = the wave's share of sum_t r_t <k_t, dK2_t>, [16 + wave] = of <dS', S>
  float* sNq = sMisc + 64;    // normalisation factors of the q and k rows (1 when the inputs come normalised)
  float* sNk = sNq + 64;
  T* tiles = reinterpret_cast<T*>(smem + sizeof(float) * L::nfloat);
  char* sSlab = reinterpret_cast<char*>(tiles);  // [2][slab_bytes]
  // epilogue
  T* sPe = tiles;             // [i][j]
  T* sPeT = sPe + L::kC;      // [j][i]
  T* sXa = sPeT + L::kC;      // [i][j]
  T* sXeT = sXa + L::kC;      // [j][i]
  T* sK = sXeT + L::kC;       // [token][dk]
  T* sQ = sK + L::kRow;
  T* sSt = tiles;             // staging for dq and dk, once the four small tiles are dead
  T* sSt2 = L::OVER2 ? sXa : sQ + L::kRow;

  const int tid = threadIdx.x, wave = NW == 4 ? tid >> 6 : __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int N = p.geom.N;
  const int64_t slot = blockIdx.x;
  const int row = (int)(slot / N), n = (int)(slot % N);
  int tok0, len;
  chunk_span(p.geom, n, tok0, len);
  if (len <= 0) return;
  const int64_t tbase = tok_index(p.geom, row, tok0);
  const int64_t ts = p.geom.ts, tsk = ts * DK, tsv = ts * p.dv;
  const int wi = wave / (NW / 2), wj = wave % (NW / 2);
  const int fr = lane & 31, kg8 = 8 * (lane >> 5);
  // the wave's tiles of dPm (all waves, or those of wj < 2) and dAm: token-row tile wi, columns 32 jt ..
  const int jt = wj & 1;
  const bool has_p = NPA == 2 || wj < 2, has_a = NPA == 2 || wj >= 2;

  TileRegs<T, 64, DK, THREADS> rK, rQ;  // the epilogue's tiles, requested during the last slab
  floatx16 aPA[NPA][1][1], aQ[1][NKT], aK1[1][NKT], aK2[1][NKT];
  auto& aP = aPA[0];
  auto& aA = aPA[NPA - 1];
  frag_zero(aP);
  frag_zero(aA);
  frag_zero(aQ);
  frag_zero(aK1);
  frag_zero(aK2);
  float ss = 0.f, rdv = 0.f;
  auto token_sum = [](float x) {  // over the TPT threads of a token
    x = quad_sum(x);
    return TPT == 8 ? x + __shfl_xor(x, 4, LNX_WAVE) : x;
  };
  auto waves_sum = [](const float* x) {
    const float lo = (x[0] + x[1]) + (x[2] + x[3]);
    return NW == 8 ? lo + ((x[4] + x[5]) + (x[6] + x[7])) : lo;
  };
  // the small loads go straight to LDS, ahead of the slabs: nothing waits for them before the first slab is requested
  if (wave == 0) dma4(p.beta + tbase + (int64_t)min(lane, len - 1) * ts, lds_byte_addr(sBeta));  // (past the end k and q are zero)
  if (GATE == LNX_GATE_SCALAR && wave == 1) dma4(at<const float>(p.ws, p.off.G) + slot * 64 + lane, lds_byte_addr(sG));
  if (wave == 2) dma4(at<const float>(p.ws, p.off.Nq) + slot * 64 + lane, lds_byte_addr(sNq));
  if (wave == 3) dma4(at<const float>(p.ws, p.off.Nk) + slot * 64 + lane, lds_byte_addr(sNk));
  if (tid < 64) {
    if (GATE == LNX_GATE_NONE) sG[tid] = 0.f;
    sM[tid] = sM[64 + tid] = sdG[tid] = sdG[64 + tid] = 0.f;
    sMisc[tid] = 0.f;
  }
  // ---- the slab loads: one-KB instructions, PER_WAVE of them per wave and slab, straight into LDS buffer `b` ----
  // Token rows past the chunk's end fetch the chunk's last row instead of zeros: whatever they hold only reaches rows of
  // dq, dk, dbeta, dg that are not stored (q, k and beta of those rows are zero).
  const unsigned slab0 = lds_byte_addr(sSlab);
  const T* gSn = at<const T>(p.ws, p.off.SnT) + slot * p.dv * DK;
  const T* gdSn = at<const T>(p.ws, p.off.dSn) + slot * p.dv * DK;
  const T* gDT = at<const T>(p.ws, p.off.D) + slot * p.dv * 64;
  const T* gdRT = at<const T>(p.ws, p.off.dD) + slot * p.dv * 64;
  const T* gdO = p.d_o + tbase * p.dv;
  const T* gV = p.v + tbase * p.dv;
  auto issue = [&](int v0, int b) {
    const unsigned dst = slab0 + b * L::slab_bytes;
    int r, c;
    // wave w: instructions w, w + NW, ... of the states; of the four small tiles one each, or with eight waves one of two
#pragma unroll
    for (int u = 0; u < NH * StT::NINSTR / NW; ++u) {
      const int i = wave + NW * u, h = i / StT::NINSTR, j = i % StT::NINSTR;
      StT::src(j, lane, r, c);
      dma16(gSn + (int64_t)(v0 + r) * DK + SC * h + c, dst + L::oSn + 1024 * i);
      dma16(gdSn + (int64_t)(v0 + r) * DK + SC * h + c, dst + L::odSn + 1024 * i);
    }
    const int j = wave & 3;
    if (NW == 4 || wave < 4) {
      TokT::src(j, lane, r, c);
      r = min(r, len - 1);
      dma16(gdO + (int64_t)r * tsv + v0 + c, dst + 1024 * j);
      dma16(gV + (int64_t)r * tsv + v0 + c, dst + L::oV + 1024 * j);
    }
    if (NW == 4 || wave >= 4) {
      TrT::src(j, lane, r, c);
      dma16(gDT + (int64_t)(v0 + r) * 64 + c, dst + L::oDT + 1024 * j);
      dma16(gdRT + (int64_t)(v0 + r) * 64 + c, dst + L::odRT + 1024 * j);
    }
  };
  constexpr int PER_WAVE = 2 * NH * StT::NINSTR / NW + 16 / NW;  // loads per wave and slab
  static_assert(NH * StT::NINSTR % NW == 0 && TokT::NINSTR == 4 && TrT::NINSTR == 4, "the same count for every wave");
#pragma unroll
  for (int u = 0; u < NBUF; ++u)
    if (u * SV < p.dv) issue(u * SV, u);
  int b = 0;
#pragma unroll 1
  for (int v0 = 0; v0 < p.dv; v0 += SV, b = b + 1 == NBUF ? 0 : b + 1) {
    // this slab has landed: all but this wave's loads of the slabs behind it, then every wave's
    if (NBUF > 2 && v0 + 2 * SV < p.dv) dma_wait<2 * PER_WAVE>();
    else if (v0 + SV < p.dv) dma_wait<PER_WAVE>();
    else dma_wait<0>();
    lds_barrier();
    const T* sdO = reinterpret_cast<const T*>(sSlab + b * L::slab_bytes);
    const T* sV = reinterpret_cast<const T*>(sSlab + b * L::slab_bytes + L::oV);
    const T* sDT = reinterpret_cast<const T*>(sSlab + b * L::slab_bytes + L::oDT);
    const T* sdRT = reinterpret_cast<const T*>(sSlab + b * L::slab_bytes + L::odRT);
    const T* sSn = reinterpret_cast<const T*>(sSlab + b * L::slab_bytes + L::oSn);
    const T* sdSn = reinterpret_cast<const T*>(sSlab + b * L::slab_bytes + L::odSn);
    static_assert(SV == 32, "two 16-wide steps per slab");
    if (v0 + SV >= p.dv) {  // last slab: the epilogue's K and Q tiles (a slab earlier gains nothing)
      rK.load(p.k + tbase * DK, tsk, len, tid);
      rQ.load(p.q + tbase * DK, tsk, len, tid);
    }
#pragma unroll
    for (int k0 = 0; k0 < SV; k0 += 16) {
      const M::Frag fdO = TokT::load(sdO, 32 * wi + fr, k0 + kg8);
      const M::Frag fdR = TrT::load_t(sdRT, k0, 32 * wi, lane);
      const M::Frag fDi = TrT::load_t(sDT, k0, 32 * wi, lane);
      const M::Frag fDj = TrT::load_t(sDT, k0, 32 * jt, lane);
      if (has_p) M::mma(aP[0][0], fdO, fDj);
      if (has_a) M::mma(aA[0][0], fdR, fDj);
#pragma unroll
      for (int c = 0; c < NKT; ++c) {
        const int col = 32 * (NKT * wj + c), st = NH == 1 ? 0 : (col / SC) * (StT::BYTES / 2);
        const M::Frag fS = StT::load_t(sSn + st, k0, NH == 1 ? col : col % SC, lane);
        const M::Frag fdS = StT::load_t(sdSn + st, k0, NH == 1 ? col : col % SC, lane);
        M::mma(aQ[0][c], fdO, fS);
        M::mma(aK1[0][c], fdR, fS);
        M::mma(aK2[0][c], fDi, fdS);
      }
    }
    {  // <dR_t, v_t> over this slab: thread = (token tid / TPT, SV / TPT value columns)
      typedef bf16_t VecV __attribute__((ext_vector_type(SV / TPT)));
      const int t = tid / TPT, c0 = (SV / TPT) * (tid % TPT);
      const VecV vv = *reinterpret_cast<const VecV*>(sV + TokT::at(t, c0));
#pragma unroll
      for (int e = 0; e < SV / TPT; ++e) rdv += (float)vv[e] * (float)sdRT[TrT::at(c0 + e, t)];
    }
    if (GATE == LNX_GATE_SCALAR) {  // <dS', S> over this slab: the two tiles share one layout, so granule by granule
#pragma unroll
      for (int u = 0; u < NH * StT::BYTES / 16 / THREADS; ++u) {
        const M::Frag a = *reinterpret_cast<const M::Frag*>(sSn + 8 * (tid + THREADS * u));
        const M::Frag b2 = *reinterpret_cast<const M::Frag*>(sdSn + 8 * (tid + THREADS * u));
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += (float)a[e] * (float)b2[e];
      }
    }
    if (v0 + NBUF * SV < p.dv) {  // this buffer takes the slab NBUF ahead, once every wave has read it
      lds_barrier();
      issue(v0 + NBUF * SV, b);
    }
  }
  rdv = token_sum(rdv);
  if (tid % TPT == 0) sRdv[tid / TPT] = rdv;
  if (GATE == LNX_GATE_SCALAR) {
    ss = wave_sum(ss);
    if (lane == 0) sMisc[16 + wave] = ss;  // one slot per wave, added in a fixed order below
  }
  lds_barrier();  // slab tiles are dead from here on

  // ---- epilogue ----
  {  // K and Q rows, normalised
    typedef TileRegs<T, 64, DK, THREADS> RowTile;
#pragma unroll
    for (int it = 0; it < RowTile::IT; ++it) {
      const int idx = tid + THREADS * it, r = idx / RowTile::VPR, c = (idx - r * RowTile::VPR) * RowTile::N;
      const float fk = sNk[r], fq = sNq[r];
      typename Vec16<T>::V x = rK.x[it], y = rQ.x[it];
#pragma unroll
      for (int e = 0; e < RowTile::N; ++e) x[e] = (bf16_t)((float)x[e] * fk), y[e] = (bf16_t)((float)y[e] * fq);
      *reinterpret_cast<typename Vec16<T>::V*>(sK + r * LDKT + c) = x;
      *reinterpret_cast<typename Vec16<T>::V*>(sQ + r * LDKT + c) = y;
    }
  }
  // The cumulative gate and beta of this lane's sixteen accumulator rows (four runs of four), as vectors and once: read one
  // by one between the tile stores below, each read would wait out its own round trip to LDS (the stores might alias it).
  floatx4 gi[4], bi[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i0 = 32 * wi + 8 * q + 4 * (lane >> 5);
    gi[q] = load4(sG + i0);
    bi[q] = load4(sBeta + i0);
  }
  const float gC = sG[63];
  {
    float dec[16];
    const int j = 32 * jt + frag_col(lane);
    const float gj = sG[j];
#pragma unroll
    for (int e = 0; e < 16; ++e) dec[e] = (GATE == LNX_GATE_NONE) ? 1.f : __expf(fminf(gi[e >> 2][e & 3] - gj, 0.f));
    if (has_p) {
      floatx16 pe[1][1];
#pragma unroll
      for (int e = 0; e < 16; ++e) pe[0][0][e] = (32 * wi + frag_row(e, lane) >= j) ? p.scale * dec[e] * aP[0][0][e] : 0.f;
      frag_store<T, 1, 1>(pe, sPe + 32 * wi * LDC + 32 * jt, LDC, lane);
      frag_store_t<T, 1, 1>(pe, sPeT + 32 * jt * LDC + 32 * wi, LDC, lane);
    }
    if (has_a) {
#pragma unroll
      for (int e = 0; e < 16; ++e) aA[0][0][e] = (32 * wi + frag_row(e, lane) > j) ? -dec[e] * aA[0][0][e] : 0.f;  // dXa
      frag_store<T, 1, 1>(aA, sXa + 32 * wi * LDC + 32 * jt, LDC, lane);
#pragma unroll
      for (int e = 0; e < 16; ++e) aA[0][0][e] *= bi[e >> 2][e & 3];  // dXe
      frag_store_t<T, 1, 1>(aA, sXeT + 32 * jt * LDC + 32 * wi, LDC, lane);
    }
  }
  lds_barrier();
  // dq = scale e^G dQa + dPe K;   row = dXa K - e^G dK1 (in aK1)
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const float gm = (GATE == LNX_GATE_NONE) ? 1.f : __expf(gi[e >> 2][e & 3]);
#pragma unroll
    for (int c = 0; c < NKT; ++c) {
      aQ[0][c][e] *= p.scale * gm;
      aK1[0][c][e] *= -gm;
    }
  }
#pragma unroll
  for (int k0 = 0; k0 < 64; k0 += 16) {
    const M::Frag fPe = M::load(sPe + (32 * wi + fr) * LDC + k0 + kg8);
    const M::Frag fXa = M::load(sXa + (32 * wi + fr) * LDC + k0 + kg8);
#pragma unroll
    for (int c = 0; c < NKT; ++c) {
      const M::Frag fK = M::load_t(sK, LDKT, k0, 32 * (NKT * wj + c), lane);
      M::mma(aQ[0][c], fPe, fK);
      M::mma(aK1[0][c], fXa, fK);
    }
  }
  // m_t = <k_t, row_t>;  chunk-end gate term sum_t r_t <k_t, dK2_t>;  dk <- beta row + r dK2 (in aK2)
  {
    float mv[16], tot = 0.f;
    floatx4 kq[NKT][4];  // K at this lane's accumulator positions, one transposing read per run of four rows
#pragma unroll
    for (int c = 0; c < NKT; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q) kq[c][q] = M::load_acc_rows(sK, LDKT, 32 * wi, q, 32 * (NKT * wj + c), lane);
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float rr = (GATE == LNX_GATE_NONE) ? 1.f : __expf(fminf(gC - gi[e >> 2][e & 3], 0.f));
      const float bt = bi[e >> 2][e & 3];
      mv[e] = 0.f;
#pragma unroll
      for (int c = 0; c < NKT; ++c) {
        const float kk = kq[c][e >> 2][e & 3];
        mv[e] += kk * aK1[0][c][e];
        aK2[0][c][e] *= rr;
        tot += kk * aK2[0][c][e];
        aK2[0][c][e] += bt * aK1[0][c][e];
      }
    }
    rows_reduce_add<1>(mv, 32 * wi, lane, sM + 64 * (wj >> 1));  // two waves (wj even, odd) add to a zeroed entry: order-independent
    if (GATE == LNX_GATE_SCALAR) {
      tot = wave_sum(tot);
      if (lane == 0) sMisc[8 + wave] = tot;
    }
  }
  // dk += dPe^T Q + dXe^T K
#pragma unroll
  for (int k0 = 0; k0 < 64; k0 += 16) {
    const M::Frag fPt = M::load(sPeT + (32 * wi + fr) * LDC + k0 + kg8);
    const M::Frag fXt = M::load(sXeT + (32 * wi + fr) * LDC + k0 + kg8);
#pragma unroll
    for (int c = 0; c < NKT; ++c) {
      M::mma(aK2[0][c], fPt, M::load_t(sQ, LDKT, k0, 32 * (NKT * wj + c), lane));
      M::mma(aK2[0][c], fXt, M::load_t(sK, LDKT, k0, 32 * (NKT * wj + c), lane));
    }
  }
  if constexpr (GATE == LNX_GATE_SCALAR && L::DOTS) {
    float x[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e] = 0.f;
#pragma unroll
    for (int c = 0; c < NKT; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const floatx4 k4 = M::load_acc_rows(sK, LDKT, 32 * wi, q, 32 * (NKT * wj + c), lane);
        const floatx4 q4 = M::load_acc_rows(sQ, LDKT, 32 * wi, q, 32 * (NKT * wj + c), lane);
#pragma unroll
        for (int u = 0; u < 4; ++u) x[4 * q + u] += q4[u] * aQ[0][c][4 * q + u] - k4[u] * aK2[0][c][4 * q + u];
      }
    rows_reduce_add<1>(x, 32 * wi, lane, sdG + 64 * (wj >> 1));
  }
  lds_barrier();  // the four small tiles are dead; sM, sdG and sMisc are complete
  // dq and dk through their staging tiles.  Thread = (token tid / TPT, the 8-column groups tid % TPT, tid % TPT + TPT, ...): the
  // row dots <q_t, dq_t> and <k_t, dk_t> carry the gradients through the normalisation,
  //   d/dx of x / (|x| + eps) applied to dy:  dy / (|x| + eps) - y <y, dy> / |x|.
  const int tr = tid / TPT, tq = 8 * (tid % TPT);
  float dgp = 0.f;
  auto emit = [&](const T* sSt, const T* sIn, float fac, T* out, float sign) {
    float cf = 0.f;
    if (!L::DOTS || p.l2norm) {
      float dot = 0.f;
#pragma unroll
      for (int u = 0; u < DK; u += 8 * TPT) {
        const M::Frag a = M::load(sSt + tr * LDK + tq + u), b = M::load(sIn + tr * LDKT + tq + u);
#pragma unroll
        for (int e = 0; e < 8; ++e) dot += (float)a[e] * (float)b[e];
      }
      dot = token_sum(dot);
      dgp += sign * dot;
      const float nrm = 1.f / fac - LNX_L2_EPS;
      cf = (p.l2norm && nrm > 0.f) ? dot / nrm : 0.f;
    }
    if (tr < len) {
#pragma unroll
      for (int u = 0; u < DK; u += 8 * TPT) {
        M::Frag a = M::load(sSt + tr * LDK + tq + u);
        const M::Frag b = M::load(sIn + tr * LDKT + tq + u);
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = (bf16_t)(fac * (float)a[e] - cf * (float)b[e]);
        *reinterpret_cast<M::Frag*>(out + tbase * DK + (int64_t)tr * tsk + tq + u) = a;
      }
    }
  };
  frag_store<T, 1, NKT>(aQ, sSt + 32 * wi * LDK + 32 * NKT * wj, LDK, lane);
  frag_store<T, 1, NKT>(aK2, sSt2 + 32 * wi * LDK + 32 * NKT * wj, LDK, lane);
  lds_barrier();
  emit(sSt, sQ, sNq[tr], p.dq, 1.f);
  emit(sSt2, sK, sNk[tr], p.dk, -1.f);
  if (GATE == LNX_GATE_SCALAR && !L::DOTS) {
    if (tid % TPT == 0) sdG[tr] = dgp;
    lds_barrier();
  }
  if (wave == 0) {
    const int t = lane;
    if (t < len) p.dbeta[tbase + t * ts] = sRdv[t] + (sM[t] + sM[64 + t]);
    if (GATE == LNX_GATE_SCALAR) {  // dg = reverse cumulative sum of dG over the chunk
      float d = (L::DOTS ? sdG[t] + sdG[64 + t] : sdG[t]) + 2.f * sBeta[t] * (sM[t] + sM[64 + t]);
      if (t == 63) d += waves_sum(sMisc + 8) + __expf(gC) * waves_sum(sMisc + 16);
#pragma unroll
      for (int s_ = 1; s_ < 64; s_ <<= 1) {
        const float y = __shfl_down(d, s_, LNX_WAVE);
        if (t + s_ < 64) d += y;
      }
      if (t < len) p.dg[tbase + t * ts] = d;
    }
  }
}

template <int DK, int GATE>
int launch_bwd_chunk(const DirectParams& p, hipStream_t st) {
  auto k = bwd_chunk_kernel<DK, GATE>;
  const size_t b = BChunkL<DK>::bytes;
  if (const int rc = lnx_lds_limit((const void*)k, b); rc != LNX_OK) return rc;
  lnx_profile_mark("bwd_chunk", st);
  hipLaunchKernelGGL(k, dim3((unsigned)((int64_t)p.geom.rows * p.geom.N)), dim3(BChunkL<DK>::THREADS), b, st, p);
  lnx_profile_mark(nullptr, st);
  return LNX_OK;
}

template <int DK, int GATE>
int launch_bwd(const DirectParams& p, int nstate, hipStream_t st) {
  int rc;
  if constexpr (DK == 256) rc = lnx_wide_scan(true, p, nstate, st);
  else rc = launch_scan_bwd<DK, GATE>(p, nstate, st);
  if (rc != LNX_OK) return rc;
  return launch_bwd_chunk<DK, GATE>(p, st);
}

}  // namespace

namespace {
template <typename OT>
int scan_fwd_by_shape(const DirectParams& p, int dk, int gate, int nstate, hipStream_t st) {
  if (dk == 128)
    return gate == LNX_GATE_SCALAR ? launch_scan_fwd<128, LNX_GATE_SCALAR, OT>(p, nstate, st) : launch_scan_fwd<128, LNX_GATE_NONE, OT>(p, nstate, st);
  return gate == LNX_GATE_SCALAR ? launch_scan_fwd<64, LNX_GATE_SCALAR, OT>(p, nstate, st) : launch_scan_fwd<64, LNX_GATE_NONE, OT>(p, nstate, st);
}
}  // namespace

int lnx_direct_scan_fwd(const DirectParams& p, int dk, int gate, int nstate, hipStream_t st) {
  if (dk == 256) {
    const int rc = lnx_wide_scan(false, p, nstate, st);
    lnx_profile_mark(nullptr, st);
    return rc;
  }
  if (!p.o && !p.save) return scan_fwd_by_shape<void>(p, dk, gate, nstate, st);
  return p.o_dtype == LNX_F32 ? scan_fwd_by_shape<float>(p, dk, gate, nstate, st) : scan_fwd_by_shape<bf16_t>(p, dk, gate, nstate, st);
}

namespace {
template <int DK> int bwd_by_gate(const DirectParams& p, int gate, int nstate, hipStream_t st) {
  return gate == LNX_GATE_SCALAR ? launch_bwd<DK, LNX_GATE_SCALAR>(p, nstate, st) : launch_bwd<DK, LNX_GATE_NONE>(p, nstate, st);
}
}  // namespace

int lnx_direct_bwd(const DirectParams& p, int dk, int gate, int nstate, hipStream_t st) {
  return dk == 256 ? bwd_by_gate<256>(p, gate, nstate, st) : dk == 128 ? bwd_by_gate<128>(p, gate, nstate, st) : bwd_by_gate<64>(p, gate, nstate, st);
}
