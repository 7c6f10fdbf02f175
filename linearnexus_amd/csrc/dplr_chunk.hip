// RWKV-7's diagonal-plus-low-rank delta rule over chunks of 64 tokens, for heads of 64 x 64 (RWKV-7's own size), in fp32.
//
// The token-by-token scan (dplr.hip) is one dependent step of some 270 wave instructions per token on the one or two waves
// that a (batch, head) row has.  Over a chunk the recurrence is a linear map of the state, so everything but a 64 x 64
// product per chunk can be done for all chunks at once, on the matrix cores (v_mfma_f32_16x16x4_f32: fp32 operands and
// accumulation, nothing is rounded below the token kernels' precision).
//
// Per chunk, G = cumulative gk, Gp the same before the token's own decay, E_ts = exp(G_t - G_s) per channel:
//   Aab = stril(<a_t e^Gp_t, b_s e^-G_s>)  Aak = stril(<a_t e^Gp_t, k_s e^-G_s>)  Pqb, Pqk = tril(<q_t e^G_t, b_s / k_s e^-G_s>)
//   Tm = (I - Aab)^-1     u = Tm (a e^Gp h + Aak v)     o = q e^G h + Pqb u + Pqk v     h' = e^G_C h + (b e^(G_C-G))^T u + (k e^(G_C-G))^T v
// and with W = Tm (a e^Gp), U0 = Tm Aak v:
//   o = X h + Y,  X = q e^G + Pqb W,  Y = Pqb U0 + Pqk v          h' = M h + N,  M = e^G_C + Bg^T W,  N = Bg^T U0 + Kg^T v
// Backward: D = gradient of the state leaving the chunk, R = X^T dO; the gradient of the state entering it is M^T D + R, and
//   dU = Tm^T (Pqb^T dO + Bg D)      dv = Pqk^T dO + Kg D + Aak^T dU
//   dPqb = tril(dO u^T)  dPqk = tril(dO v^T)  dAab = stril(dU u^T)  dAak = stril(dU v^T), and from these the vectors' gradients;
//   dgk_t = <D, h'>_c + sum_{t' >= t} (q dq + a da - b db - k dk)_t' - (a da)_t   (how each exponential depends on G).
//
// The factors e^(G_t - G_s) <= 1 are split as e^(G_t - m) e^(m - G_s) around the middle m of the chunk's range of G, one m
// per channel.  RWKV-7's decays are above exp(-0.607) per token, so |G - m| <= 20 and both factors are harmless; a chunk in
// which any channel's range exceeds LNX_DPLR_RANGE evaluates its pairs one by one from the difference instead (a uniform
// branch per chunk: exact for any decay, and some 20 us per workgroup slower).
//
// Kernels, each a workgroup per chunk but for the two sequential passes.  Measured at B8 H16 T4096 bf16 (8192 chunks):
// see the table at the launch functions.
#include "lnx_common.h"
#include "chunk_common.h"

namespace {

constexpr int C = 64, D = 64;       // tokens of a chunk, channels of a head
constexpr int LD = LNX_LDA;         // leading dimension of the fp32 tiles in LDS: 68 floats, rows 4 banks apart
constexpr int TS = C * LD;          // floats of a tile in LDS
constexpr int TG = C * D;           // floats of a tile in the workspace
constexpr float RANGE = 80.f;       // widest range of G that the split around its middle may span: e^40 e^-40 in each factor

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

// e^x with the rounding of x log2(e) carried along: the factors' exponents reach 40, where the plain product's rounding is
// already 2e-6 of the result.
__device__ __forceinline__ float exp_f(float x) {
  float t = x * 1.44269504f;
  asm volatile("" : "+v"(t));  // -ffast-math must not see that the next line is a rounding error
  const float e = __builtin_fmaf(x, 1.44269504f, -t) + x * 1.92596299e-8f;
  return __builtin_amdgcn_exp2f(t) * (1.f + 0.69314718f * e);
}

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

// Blocks 0 .. j, or 3 .. j, as constants: the accumulators stay where they are when a wave leaves early (a branch around each
// block's products made the compiler copy them, 1000 moves among 850 products)
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

// Four consecutive elements as loaded
template <typename T> struct Raw4;
template <> struct Raw4<bf16_t> {
  bf16x4 x;
  __device__ __forceinline__ void load(const bf16_t* p) { x = *reinterpret_cast<const bf16x4*>(p); }
  __device__ __forceinline__ floatx4 get() const { return floatx4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]}; }
};
template <> struct Raw4<float> {
  floatx4 x;
  __device__ __forceinline__ void load(const float* p) { x = load4(p); }
  __device__ __forceinline__ floatx4 get() const { return x; }
};
// This lane's share of a row of 64, zeros where there is no such token (no load behind a branch: `base` is readable anyway)
template <typename T> struct Row {
  Raw4<T> x[4];
  bool ok;
  __device__ __forceinline__ void load(const void* base, int64_t at, bool ok_ = true) {  // at: element of the lane's first channel
    ok = ok_;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) x[cb].load(static_cast<const T*>(base) + (ok ? at + 16 * cb : 0));
  }
  __device__ __forceinline__ floatx4 operator[](int cb) const { return ok ? x[cb].get() : zero4(); }
};
// ... into its row of a tile
template <typename F> __device__ __forceinline__ void put_row(float* tile, const Lane& w, F&& value) {
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) store4(tile + w.t * LD + 16 * cb + 4 * w.g, value(cb));
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
struct Gates {      // arrays of 64 floats in LDS
  float *em, *ec, *eC, *gm;  // e^m, e^(G_C - m), e^G_C, m
  int* wide;                 // some channel's range is too wide for the split: pairs one by one, em = ec = 1
};

// Gt: gk of the chunk on entry ([t][c], visible after the first barrier), its cumulative sum on return; scr: 768 floats
__device__ __forceinline__ void cumulate(float* Gt, float* scr, const Gates& s) {
  const int tid = threadIdx.x, c = tid & 63, seg = tid >> 6;
  lds_barrier();
  float v[16], sum = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = (sum += Gt[(16 * seg + i) * LD + c]);
  scr[64 * seg + c] = sum;
  lds_barrier();
  float pre = 0.f;
  for (int j = 0; j < seg; ++j) pre += scr[64 * j + c];
  float mx = 0.f, mn = 0.f;  // the token before the chunk has G = 0
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float x = pre + v[i];
    Gt[(16 * seg + i) * LD + c] = x;
    mx = fmaxf(mx, x), mn = fminf(mn, x);
  }
  scr[256 + 64 * seg + c] = mx;
  scr[512 + 64 * seg + c] = mn;
  lds_barrier();
  if (seg == 0) {
#pragma unroll
    for (int j = 1; j < 4; ++j) mx = fmaxf(mx, scr[256 + 64 * j + c]), mn = fminf(mn, scr[512 + 64 * j + c]);
    const bool wide = __ballot(!(mx - mn <= RANGE)) != 0;
    const float m = 0.5f * (mx + mn), last = Gt[(C - 1) * LD + c];
    s.gm[c] = m;
    s.em[c] = wide ? 1.f : exp_f(m);
    s.ec[c] = wide ? 1.f : exp_f(last - m);
    s.eC[c] = exp_f(last);
    if (c == 0) *s.wide = wide;
  }
  lds_barrier();
}

__device__ __forceinline__ floatx4 rcp4(floatx4 x) {  // of e^x, |x| <= RANGE / 2
  return floatx4{__builtin_amdgcn_rcpf(x[0]), __builtin_amdgcn_rcpf(x[1]), __builtin_amdgcn_rcpf(x[2]), __builtin_amdgcn_rcpf(x[3])};
}
__device__ __forceinline__ floatx4 exp4(floatx4 x) { return floatx4{exp_f(x[0]), exp_f(x[1]), exp_f(x[2]), exp_f(x[3])}; }

// The lane's row of q, k, a, b and of the cumulative gate
template <typename T> struct Own {
  Row<T> q, k, a, b;
  floatx4 G[4];
  __device__ __forceinline__ void load(const ChunkParams& p, const Slot& s, const Lane& w, float* Gt) {
    const bool ok = w.t < s.len;
    const int64_t at = (s.tok + w.t) * D + 4 * w.g;
    Row<float> g;
    g.load(p.gk, at, ok);
    q.load(p.q, at, ok);
    a.load(p.a, at, ok);
    b.load(p.b, at, ok);
    k.load(p.k, at, ok);
    put_row(Gt, w, [&](int cb) { return g[cb]; });
  }
  __device__ __forceinline__ void gates(const float* Gt, const Lane& w) {  // Gt: the cumulative sums
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      G[cb] = load4(Gt + w.t * LD + 16 * cb + 4 * w.g);
    }
  }
};
// e^(G - m), e^(Gp - m) and e^(m - G), or e^G, e^Gp and e^(G_C - G) in a wide chunk, of the lane's channels
struct Decay {
  floatx4 q[4], a[4], b[4];
  __device__ __forceinline__ Decay(const floatx4 (&G)[4], const floatx4 (&Gp)[4], const float* last, const Gates& s, const Lane& w, bool wide) {
    if (!wide) {
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        const floatx4 m = load4(s.gm + 16 * cb + 4 * w.g);
        q[cb] = exp4(G[cb] - m), a[cb] = exp4(Gp[cb] - m), b[cb] = rcp4(q[cb]);
      }
    } else {
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) q[cb] = exp4(G[cb]), a[cb] = exp4(Gp[cb]), b[cb] = exp4(load4(last + 16 * cb + 4 * w.g) - G[cb]);
    }
  }
};
__device__ __forceinline__ void gates_before(floatx4 (&Gp)[4], const float* Gt, const Lane& w) {  // of the token before the lane's
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const floatx4 x = load4(Gt + max(w.t - 1, 0) * LD + 16 * cb + 4 * w.g);
#pragma unroll
    for (int e = 0; e < 4; ++e) Gp[cb][e] = w.t ? x[e] : 0.f;
  }
}

// Wide chunk: the pair (t, s) of Aab, Aak, Pqb, Pqk from the difference of the gates, the vectors from memory
struct Pair {
  float ab, ak, qb, qk;
};
template <typename T> __device__ __forceinline__ Pair wide_pair(const ChunkParams& p, int64_t tok, int len, const float* Gt, int t, int s) {
  Pair r{0.f, 0.f, 0.f, 0.f};
  if (s > t || t >= len) return r;
  const T *q = static_cast<const T*>(p.q) + (tok + t) * D, *a = static_cast<const T*>(p.a) + (tok + t) * D;
  const T *b = static_cast<const T*>(p.b) + (tok + s) * D, *k = static_cast<const T*>(p.k) + (tok + s) * D;
  for (int c = 0; c < D; ++c) {
    const float G = Gt[s * LD + c], eq = p.scale * to_f32(q[c]) * exp_f(Gt[t * LD + c] - G), vb = to_f32(b[c]), vk = to_f32(k[c]);
    r.qb += eq * vb;
    r.qk += eq * vk;
    if (s < t) {
      const float ea = to_f32(a[c]) * exp_f(Gt[(t - 1) * LD + c] - G);
      r.ab += ea * vb;
      r.ak += ea * vk;
    }
  }
  return r;
}

// What `pair(o, x)` gives of the lane's pairs with tokens o = 16 b + 4 g + r, through the lane's own places of N tiles
template <int N, typename F> __device__ __forceinline__ void wide_pairs(floatx4 (*const (&m)[N])[4], float* const (&tile)[N], const Lane& w, F&& pair) {
#pragma unroll 1
  for (int e = 0; e < 16; ++e) {
    const int o = 16 * (e >> 2) + 4 * w.g + (e & 3);
    float x[N];
    pair(o, x);
#pragma unroll
    for (int i = 0; i < N; ++i) tile[i][w.t * LD + o] = x[i];
  }
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int b = 0; b < 4; ++b) (*m[i])[b] = load4(tile[i] + w.t * LD + 16 * b + 4 * w.g);
}

// Blocks of a lower-triangular pair matrix M[t][s].  `ByT`: tile sb <= j holds rows s, columns t = the wave's tokens; ByS: tile
// tb >= j rows t, columns s = the wave's tokens.  Entries above the diagonal (STRICT: on it, too) are cleared.
template <bool BY_T, bool STRICT> __device__ __forceinline__ void mask(floatx4 (&m)[4], const Lane& w) {
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const bool diagonal = b == w.j;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 4 * w.g + r, t = BY_T ? w.l16 : row, s = BY_T ? row : w.l16;
      m[b][r] = (diagonal && (STRICT ? s >= t : s > t)) ? 0.f : m[b][r];
    }
  }
}

constexpr int LDS_TILES = 4;
constexpr unsigned LDS_BYTES = (LDS_TILES * TS + 4 * 64 + 4 + 32 * 36) * sizeof(float);
static_assert(LDS_BYTES <= 80 * 1024, "two workgroups per CU");
struct Lds {
  float* base;
  Gates gate;
  float* sx;  // 32 x 36 floats
  __device__ __forceinline__ Lds(char* smem) {
    base = reinterpret_cast<float*>(smem);
    float* x = base + LDS_TILES * TS;
    gate = Gates{x, x + 64, x + 128, x + 192, reinterpret_cast<int*>(x + 256)};
    sx = x + 260;
  }
  __device__ __forceinline__ float* tile(int i) const { return base + i * TS; }
};

// ---- forward: M, X, N^T, Y of a chunk ------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256, 2) void dplr_prepare_kernel(ChunkParams p) {
  extern __shared__ __align__(16) char smem[];
  const Lds L(smem);
  const Slot s = slot_of(p);
  const Lane w;
  const int l16 = w.l16, g = w.g, g4 = 4 * w.g;
  float *tb = L.tile(0), *tk = L.tile(1), *ta = L.tile(2), *tx = L.tile(3);
  Own<T> x;
  x.load(p, s, w, tx);
  Row<T> v;
  v.load(p.v, (s.tok + w.t) * D + g4, w.t < s.len);
  cumulate(tx, L.sx, L.gate);
  x.gates(tx, w);
  const bool wide = *L.gate.wide;
  floatx4 xx[4];  // q with its factor, then X^T: rows = channels, columns = tokens
  floatx4 ab[4], ak[4], qb[4], qk[4];
  clear(ab), clear(ak), clear(qb), clear(qk);
  {
    floatx4 fa[4], fb[4], fk[4];
    {
      floatx4 Gp[4];
      gates_before(Gp, tx, w);
      const Decay e(x.G, Gp, tx + (C - 1) * LD, L.gate, w, wide);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) xx[cb] = p.scale * x.q[cb] * e.q[cb], fa[cb] = x.a[cb] * e.a[cb], fb[cb] = x.b[cb] * e.b[cb], fk[cb] = x.k[cb] * e.b[cb];
    }
    if (wide) {
      wide_pairs<2>({&ab, &ak}, {tb, tk}, w, [&](int o, float* r) { const Pair y = wide_pair<T>(p, s.tok, s.len, tx, w.t, o); r[0] = y.ab, r[1] = y.ak; });
      wide_pairs<2>({&qb, &qk}, {tb, tk}, w, [&](int o, float* r) { const Pair y = wide_pair<T>(p, s.tok, s.len, tx, w.t, o); r[0] = y.qb, r[1] = y.qk; });
    }
    put_cols(ta, w, fa), put_cols(tb, w, fb), put_cols(tk, w, fk);
    lds_barrier();
    if (!wide) {
      upto(w.j, [&](auto sb_) {
        constexpr int sb = decltype(sb_)::value;
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          const floatx4 rb = frag<true>(tb, 16 * sb + l16, 16 * kb + g4), rk = frag<true>(tk, 16 * sb + l16, 16 * kb + g4);
#pragma unroll
          for (int r = 0; r < 4; ++r) {  // four accumulators in turn: no product waits for the one before it
            ab[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(rb[r], fa[kb][r], ab[sb], 0, 0, 0);
            ak[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(rk[r], fa[kb][r], ak[sb], 0, 0, 0);
            qb[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(rb[r], xx[kb][r], qb[sb], 0, 0, 0);
            qk[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(rk[r], xx[kb][r], qk[sb], 0, 0, 0);
          }
        }
      });
      mask<true, true>(ab, w), mask<true, true>(ak, w), mask<true, false>(qb, w), mask<true, false>(qk, w);
    }
  }
  lds_barrier();  // the gates have been read
  put_row(tx, w, [&](int cb) { return v[cb]; });
  lds_barrier();
  floatx4 nt[4], z[4], y[4];  // N (rows i, columns n), Aak v (rows t, columns n), Y^T (rows n, columns t)
  clear(nt), clear(z), clear(y);
#pragma unroll
  for (int sb = 0; sb < 4; ++sb) {
    const floatx4 kf = frag<false>(tk, 16 * w.j + l16, 16 * sb + g4);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) mfma4(nt[nb], kf, frag<false>(tx, 16 * nb + l16, 16 * sb + g4));
  }
  upto(w.j, [&](auto sb_) {
    constexpr int sb = decltype(sb_)::value;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const floatx4 vf = frag<false>(tx, 16 * nb + l16, 16 * sb + g4);
      mfma4(z[nb], ak[sb], vf);
      mfma4(y[nb], vf, qk[sb]);
    }
  });
  lds_barrier();
#pragma unroll
  for (int sb = 0; sb < 4; ++sb) store4(tx + w.t * LD + 16 * sb + g4, sb <= w.j ? -ab[sb] : zero4());
  put_rows(tk, w, z);
  lds_barrier();
  tri_inverse_64<true>(tx, tx, L.sx, threadIdx.x);
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
  floatx4 m[4];  // M[i][c]: rows c, columns i
  clear(m);
#pragma unroll
  for (int sb = 0; sb < 4; ++sb) {
    const floatx4 bf = frag<false>(tb, 16 * w.j + l16, 16 * sb + g4);
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const floatx4 wf = frag<true>(ta, 16 * cb + l16, 16 * sb + g4), uf = frag<true>(tk, 16 * cb + l16, 16 * sb + g4);
      mfma4(m[cb], wf, bf);
      mfma4(nt[cb], bf, uf);
    }
  }
  upto(w.j, [&](auto sb_) {
    constexpr int sb = decltype(sb_)::value;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      mfma4(xx[cb], frag<true>(ta, 16 * cb + l16, 16 * sb + g4), qb[sb]);
      mfma4(y[cb], frag<true>(tk, 16 * cb + l16, 16 * sb + g4), qb[sb]);
    }
  });
  const float eci = L.gate.ec[w.t], eCi = L.gate.eC[w.t];
  const floatx4 ec4 = load4(L.gate.ec + 16 * w.j + g4);
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const floatx4 em = load4(L.gate.em + 16 * cb + g4);
    floatx4 r = m[cb] * em * eci;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (16 * cb + g4 + e == w.t) r[e] += eCi;
    const int at = w.t * D + 16 * cb + g4;
    store4(p.M + s.kept * TG + at, r);
    store4(p.X + s.kept * TG + at, xx[cb] * em);
    store4(p.s2 + s.win * TG + at, y[cb]);
    store4(p.s1 + s.win * TG + (16 * cb + l16) * D + 16 * w.j + g4, nt[cb] * ec4);
  }
}

// ---- the sequential pass: h <- M h + N (forward), D <- M^T D + R (backward) ------------------------------------
// One workgroup per row and 16 of the 64 value columns; wave w forms 16 rows of the new state, sixteen products of 32 cycles, from its
// rows of M, which come straight into its registers three chunks ahead, and the old state, which the waves exchange
// through LDS (transposed), one LDS barrier per chunk.  A whole chain on one wave per 16 columns took four times the products and
// M through LDS: 1.85 us per chunk.
struct ScanParams {
  const float* M;    // kept tiles [rows][KN]
  const float* add;  // window tiles: N^T or R^T
  float* st;         // the state entering (forward: kept [rows][KN + 1]) or the gradient leaving (backward: window) each chunk, transposed
  const float* s_in; // [dk][dv] per row, or NULL
  float* s_out;      // [dk][dv] per row, or NULL
  int64_t rows;
  int KN, at, nw;    // the window is chunks [at, at + nw) of the kept tensors
};

template <bool BWD>
__global__ __launch_bounds__(256) void dplr_chunk_scan_kernel(ScanParams p) {
  __shared__ __align__(16) float buf[2][16 * LD];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  int64_t row;
  int part;
  if (!xcd_slot_part(p.rows, 4, row, part)) return;  // the four parts read the same M: one XCD
  const int col = 16 * part + l16, r0 = 16 * wave + 4 * g;  // this lane's column and its first row of the state
  const float* Mrow = p.M + (row * p.KN + p.at) * TG + (BWD ? 4 * g * D + 16 * wave + l16 : (16 * wave + l16) * D + 4 * g);
  const float* Arow = p.add + row * p.nw * TG + col * D + r0;
  float* Srow = p.st + (BWD ? row * p.nw : row * (p.KN + 1) + p.at) * TG + col * D + r0;
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
    for (int b = 0; b < 4; ++b) {
      if (BWD) x.m[b] = floatx4{M[16 * b * D], M[(16 * b + 1) * D], M[(16 * b + 2) * D], M[(16 * b + 3) * D]};
      else x.m[b] = load4(M + 16 * b);
    }
    x.a = load4(Arow + chunk(min(i, p.nw - 1)) * TG);
  };
  auto step = [&](Ahead& x, Ahead& next, int i) {  // next: the set that chunk i - 1 has used
    lds_barrier();
    const float* cur = buf[i & 1] + l16 * LD + 4 * g;
    floatx4 f[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) f[b] = load4(cur + 16 * b);
    fetch(next, i + 3);
    store4(Srow + chunk(i) * TG, h);
    floatx4 y0 = x.a, y1 = zero4();
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        y0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.m[2 * b][r], f[2 * b][r], y0, 0, 0, 0);
        y1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x.m[2 * b + 1][r], f[2 * b + 1][r], y1, 0, 0, 0);
      }
    h = y0 + y1;
    store4(buf[(i + 1) & 1] + l16 * LD + r0, h);
  };
  fetch(x0, 0);
  fetch(x1, 1);
  fetch(x2, 2);
  store4(buf[0] + l16 * LD + r0, h);
  for (int i = 0; i < p.nw; i += 4) {
    step(x0, x3, i);
    if (i + 1 >= p.nw) break;
    step(x1, x0, i + 1);
    if (i + 2 >= p.nw) break;
    step(x2, x1, i + 2);
    if (i + 3 >= p.nw) break;
    step(x3, x2, i + 3);
  }
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
  const float* X = p.X + s.kept * TG + t * D + 4 * g;
  const float* Y = p.s2 + s.win * TG + t * D + 4 * g;
  const float* h = p.hT + s.st * TG + l16 * D + 4 * g;
  if (16 * wave >= s.len) return;
  floatx4 x[4], acc[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) x[b] = load4(X + 16 * b), acc[b] = load4(Y + 16 * b);
#pragma unroll
  for (int nb = 0; nb < 4; ++nb)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) mfma4(acc[nb], load4(h + 16 * nb * D + 16 * kb), x[kb]);
  if (t < s.len) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) store_row4<T>(p.o, (s.tok + t) * D + 16 * nb + 4 * g, acc[nb]);
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
  x.load(p.X, s.kept * TG + w.t * D + g4);
  d.load(p.d_o, (s.tok + w.t) * D + g4, w.t < s.len);
  put_row(tX, w, [&](int cb) { return x[cb]; });
  put_row(tO, w, [&](int cb) { return d[cb]; });
  lds_barrier();
  floatx4 acc[4];
  clear(acc);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const floatx4 a = frag<false>(tX, w.t, 16 * kb + g4);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) mfma4(acc[nb], a, frag<false>(tO, 16 * nb + l16, 16 * kb + g4));
  }
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) store4(p.s2 + s.win * TG + (16 * nb + l16) * D + 16 * w.j + g4, acc[nb]);
}

// ---- backward: u, dU and dv of a chunk -----------------------------------------------------------------------
// The pair matrices and the inverse are formed again: keeping them would move 128 KB per chunk through memory.
template <typename T>
__global__ __launch_bounds__(256, 2) void dplr_u_kernel(ChunkParams p) {
  extern __shared__ __align__(16) char smem[];
  const Lds L(smem);
  const Slot s = slot_of(p);
  const Lane w;
  const int l16 = w.l16, g4 = 4 * w.g;
  float *tb = L.tile(0), *tk = L.tile(1), *ta = L.tile(2), *tx = L.tile(3);
  Own<T> x;
  x.load(p, s, w, tx);
  Row<T> v, d_o;
  v.load(p.v, (s.tok + w.t) * D + g4, w.t < s.len);
  d_o.load(p.d_o, (s.tok + w.t) * D + g4, w.t < s.len);
  Row<float> h0, dC;
  h0.load(p.hT, s.st * TG + w.t * D + g4);
  dC.load(p.s1, s.win * TG + w.t * D + g4);
  cumulate(tx, L.sx, L.gate);
  x.gates(tx, w);
  const bool wide = *L.gate.wide;
  floatx4 fa[4], fb[4], fk[4];  // the lane's row with its factors
  floatx4 ab[4], akT[4];        // Aab, Aak by t
  floatx4 ak[4], qb[4], qk[4];  // Aak, Pqb, Pqk by s
  clear(ab), clear(akT), clear(ak), clear(qb), clear(qk);
  {
    floatx4 fq[4];
    {
      floatx4 Gp[4];
      gates_before(Gp, tx, w);
      const Decay e(x.G, Gp, tx + (C - 1) * LD, L.gate, w, wide);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) fq[cb] = p.scale * x.q[cb] * e.q[cb], fa[cb] = x.a[cb] * e.a[cb], fb[cb] = x.b[cb] * e.b[cb], fk[cb] = x.k[cb] * e.b[cb];
    }
    if (!wide) {
      put_cols(ta, w, fa), put_cols(tb, w, fb), put_cols(tk, w, fk);
      lds_barrier();  // the gates have been read
      put_cols(tx, w, fq);
      lds_barrier();
    }
  }
  if (!wide) {
    upto(w.j, [&](auto b_) {
      constexpr int b = decltype(b_)::value;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const floatx4 rb = frag<true>(tb, 16 * b + l16, 16 * kb + g4), rk = frag<true>(tk, 16 * b + l16, 16 * kb + g4);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          ab[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(rb[r], fa[kb][r], ab[b], 0, 0, 0);
          akT[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(rk[r], fa[kb][r], akT[b], 0, 0, 0);
        }
      }
    });
    downto(w.j, [&](auto b_) {
      constexpr int b = decltype(b_)::value;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const floatx4 ra = frag<true>(ta, 16 * b + l16, 16 * kb + g4), rq = frag<true>(tx, 16 * b + l16, 16 * kb + g4);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          ak[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[r], fk[kb][r], ak[b], 0, 0, 0);
          qb[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(rq[r], fb[kb][r], qb[b], 0, 0, 0);
          qk[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(rq[r], fk[kb][r], qk[b], 0, 0, 0);
        }
      }
    });
    mask<true, true>(ab, w), mask<true, true>(akT, w), mask<false, true>(ak, w), mask<false, false>(qb, w), mask<false, false>(qk, w);
  } else {
    wide_pairs<2>({&ab, &akT}, {tb, tk}, w, [&](int o, float* r) { const Pair y = wide_pair<T>(p, s.tok, s.len, tx, w.t, o); r[0] = y.ab, r[1] = y.ak; });
    wide_pairs<3>({&ak, &qb, &qk}, {tb, tk, ta}, w, [&](int o, float* r) { const Pair y = wide_pair<T>(p, s.tok, s.len, tx, o, w.t); r[0] = y.ak, r[1] = y.qb, r[2] = y.qk; });
  }
  lds_barrier();
  float *th = ta, *tO = tb, *tD = tk, *tv = tx;
  put_row(tv, w, [&](int cb) { return v[cb]; });
  put_row(tO, w, [&](int cb) { return d_o[cb]; });
  put_row(th, w, [&](int cb) { return h0[cb] * load4(L.gate.em + 16 * cb + g4); });  // e^m h, [value column][channel]
  put_row(tD, w, [&](int cb) { return dC[cb] * load4(L.gate.ec + 16 * cb + g4); });  // e^(G_C - m) D, [value column][channel]
  lds_barrier();
  floatx4 z[4], y[4], dv[4];  // a h + Aak v, Bg D + Pqb^T dO (rows t, columns n), dv (rows n, columns t)
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
  upto(w.j, [&](auto b_) {
    constexpr int b = decltype(b_)::value;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) mfma4(z[nb], akT[b], frag<false>(tv, 16 * nb + l16, 16 * b + g4));
  });
  downto(w.j, [&](auto b_) {
    constexpr int b = decltype(b_)::value;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
      const floatx4 of = frag<false>(tO, 16 * nb + l16, 16 * b + g4);
      mfma4(y[nb], qb[b], of);
      mfma4(dv[nb], of, qk[b]);
    }
  });
  lds_barrier();
  float *Tm = tx, *tz = ta, *ty = tk, *tdu = tb;
#pragma unroll
  for (int sb = 0; sb < 4; ++sb) store4(Tm + w.t * LD + 16 * sb + g4, sb <= w.j ? -ab[sb] : zero4());
  put_rows(tz, w, z);
  put_rows(ty, w, y);
  lds_barrier();
  tri_inverse_64<true>(Tm, Tm, L.sx, threadIdx.x);
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
  const int64_t wt = s.win * TG + w.t * D + g4;
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    store4(p.s3 + wt + 16 * nb, u[nb]);
    store4(p.s4 + wt + 16 * nb, du[nb]);
  }
  put_cols(tdu, w, du);
  lds_barrier();
  downto(w.j, [&](auto b_) {
    constexpr int b = decltype(b_)::value;
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) mfma4(dv[nb], frag<false>(tdu, 16 * nb + l16, 16 * b + g4), ak[b]);
  });
  if (w.t < s.len) {
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) store_row4<T>(p.dv, (s.tok + w.t) * D + 16 * nb + g4, dv[nb]);
  }
}

// ---- backward: dq, dk, da, db, dgk of a chunk ----------------------------------------------------------------
// Wide chunk: what the matrices Mb, Mk (which pair b and k with q: LAG 0, or with a, whose decay lags by its own token: LAG 1) add to
// the gradients of the lane's token: d1 (q or a), db, dk, four channels from ch.
template <typename T, int LAG>
__device__ __forceinline__ void wide_grads(const ChunkParams& p, int64_t tok, int len, const float* Mb, const float* Mk, const float* Gt, int t, int ch,
                                                     floatx4& d1, floatx4& db, floatx4& dk) {
  auto row = [&](const void* base, int i) { Raw4<T> x; x.load(static_cast<const T*>(base) + (tok + min(i, len - 1)) * D + ch); return i < len ? x.get() : zero4(); };
  auto gate = [&](int i) { return i < 0 ? zero4() : load4(Gt + i * LD + ch); };
  const floatx4 G = gate(t), Gl = gate(t - LAG);
  for (int i = 0; i <= t - LAG; ++i) d1 += exp4(Gl - gate(i)) * (Mb[t * LD + i] * row(p.b, i) + Mk[t * LD + i] * row(p.k, i));
  for (int i = t + LAG; i < C; ++i) {
    const floatx4 e = exp4(gate(i - LAG) - G) * (LAG ? row(p.a, i) : p.scale * row(p.q, i));
    db += e * Mb[i * LD + t];
    dk += e * Mk[i * LD + t];
  }
}

template <typename T>
__global__ __launch_bounds__(256, 2) void dplr_grad_kernel(ChunkParams p) {
  extern __shared__ __align__(16) char smem[];
  const Lds L(smem);
  const Slot s = slot_of(p);
  const Lane w;
  const int tid = threadIdx.x, l16 = w.l16, g4 = 4 * w.g;
  float *t0 = L.tile(0), *t1 = L.tile(1), *t2 = L.tile(2), *t3 = L.tile(3);
  float* red = L.sx + 768;  // [4][64]: partial sums of <D, h'> per channel
  const int64_t at = (s.tok + w.t) * D + g4, wt = s.win * TG + w.t * D + g4, ht = s.st * TG + w.t * D + g4;
  const bool ok = w.t < s.len;
  Own<T> x;
  Row<T> v, d_o;
  Row<float> u, du;
  {
    Row<float> hC, dC;
    hC.load(p.hT, ht + TG);
    dC.load(p.s1, wt);
    x.load(p, s, w, t3);
    v.load(p.v, at, ok);
    d_o.load(p.d_o, at, ok);
    u.load(p.s3, wt);
    du.load(p.s4, wt);
    put_row(t0, w, [&](int cb) { return dC[cb] * hC[cb]; });
  }
  cumulate(t3, L.sx, L.gate);
  x.gates(t3, w);
  {
    const int c = tid & 63, seg = tid >> 6;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) sum += t0[(16 * seg + i) * LD + c];
    red[64 * seg + c] = sum;
  }
  const bool wide = *L.gate.wide;
  float* edge = L.sx;  // G of the blocks' last tokens
  edge[tid] = t3[(16 * (tid >> 6) + 15) * LD + (tid & 63)];
  lds_barrier();
  put_row(t0, w, [&](int cb) { return v[cb]; });
  put_row(t2, w, [&](int cb) { return u[cb]; });
  lds_barrier();
  floatx4 pb[4], pk[4], nb_[4], nk[4];  // dPqb, dPqk, dAab, dAak by t
  clear(pb), clear(pk), clear(nb_), clear(nk);
  upto(w.j, [&](auto sb_) {
    constexpr int sb = decltype(sb_)::value;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const floatx4 fu = frag<true>(t2, 16 * sb + l16, 16 * kb + g4), fv = frag<true>(t0, 16 * sb + l16, 16 * kb + g4);
      const floatx4 fo = d_o[kb], fd = du[kb];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pb[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(fu[r], fo[r], pb[sb], 0, 0, 0);
        pk[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(fv[r], fo[r], pk[sb], 0, 0, 0);
        nb_[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(fu[r], fd[r], nb_[sb], 0, 0, 0);
        nk[sb] = __builtin_amdgcn_mfma_f32_16x16x4f32(fv[r], fd[r], nk[sb], 0, 0, 0);
      }
    }
  });
  mask<true, false>(pb, w), mask<true, false>(pk, w), mask<true, true>(nb_, w), mask<true, true>(nk, w);
  {
    Row<float> h0, dC;
    h0.load(p.hT, ht);
    dC.load(p.s1, wt);
    // t1 and t3 are free since the gates were read
    put_row(t1, w, [&](int cb) { return h0[cb] * load4(L.gate.em + 16 * cb + g4); });
    put_row(t3, w, [&](int cb) { return dC[cb] * load4(L.gate.ec + 16 * cb + g4); });
  }
  lds_barrier();
  floatx4 dq[4], da[4], db[4], dk[4];  // rows = channels, columns = tokens
  clear(dq), clear(da), clear(db), clear(dk);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const floatx4 fo = d_o[kb], fd = du[kb], fu = u[kb], fv = v[kb];
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      const floatx4 hf = frag<false>(t1, 16 * cb + l16, 16 * kb + g4), df = frag<false>(t3, 16 * cb + l16, 16 * kb + g4);
      mfma4(dq[cb], hf, fo);
      mfma4(da[cb], hf, fd);
      mfma4(db[cb], df, fu);
      mfma4(dk[cb], df, fv);
    }
  }
  floatx4 Gp[4];  // from the lane before
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    const floatx4 G = load4(edge + 64 * max(w.j - 1, 0) + 16 * cb + g4);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float prev = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x.G[cb][e]), 0x111, 0xF, 0xF, true));  // row_shr:1
      Gp[cb][e] = l16 ? prev : w.j ? G[e] : 0.f;
    }
  }
  const Decay e(x.G, Gp, edge + 192, L.gate, w, wide);
  auto put_tri = [&](float* tile, const floatx4 (&m)[4]) {  // [t][s]
#pragma unroll
    for (int sb = 0; sb < 4; ++sb)
      if (sb <= w.j) store4(tile + w.t * LD + 16 * sb + g4, m[sb]);
  };
  floatx4 xs[4], as[4];  // q dq + a da - b db - k dk and a da
  if (!wide) {
    put_row(t0, w, [&](int cb) { return x.b[cb] * e.b[cb]; });
    put_row(t2, w, [&](int cb) { return x.k[cb] * e.b[cb]; });  // v and u were last read before a barrier
    lds_barrier();
    upto(w.j, [&](auto sb_) {
      constexpr int sb = decltype(sb_)::value;
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        const floatx4 bf = frag<false>(t0, 16 * cb + l16, 16 * sb + g4), kf = frag<false>(t2, 16 * cb + l16, 16 * sb + g4);
        mfma4(dq[cb], bf, pb[sb]);
        mfma4(da[cb], bf, nb_[sb]);
        mfma4(dq[cb], kf, pk[sb]);
        mfma4(da[cb], kf, nk[sb]);
      }
    });
    lds_barrier();
    // db, dk: the matrices with the contraction along t, first those of q, then those of a
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if (half) lds_barrier();
      put_tri(t1, half ? nb_ : pb), put_tri(t2, half ? nk : pk);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        if (half) store4(t0 + w.t * LD + 16 * cb + g4, x.a[cb] * e.a[cb]);
        else store4(t0 + w.t * LD + 16 * cb + g4, p.scale * x.q[cb] * e.q[cb]);
      }
      lds_barrier();
      downto(w.j, [&](auto tb_) {
        constexpr int tb = decltype(tb_)::value;
        const floatx4 mb = frag<false>(t1, w.t, 16 * tb + g4), mk = frag<false>(t2, w.t, 16 * tb + g4);
#pragma unroll
        for (int cb = 0; cb < 4; ++cb) {
          const floatx4 xf = frag<false>(t0, 16 * cb + l16, 16 * tb + g4);
          mfma4(db[cb], xf, mb);
          mfma4(dk[cb], xf, mk);
        }
      });
    }
  }
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) dq[cb] *= e.q[cb], da[cb] *= e.a[cb], db[cb] *= e.b[cb], dk[cb] *= e.b[cb];
  if (wide) {
    put_tri(t0, pb), put_tri(t2, pk);
    lds_barrier();
    put_cols(t1, w, x.G);
    lds_barrier();
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) wide_grads<T, 0>(p, s.tok, s.len, t0, t2, t1, w.t, 16 * cb + g4, dq[cb], db[cb], dk[cb]);
    lds_barrier();
    put_tri(t0, nb_), put_tri(t2, nk);
    lds_barrier();
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) wide_grads<T, 1>(p, s.tok, s.len, t0, t2, t1, w.t, 16 * cb + g4, da[cb], db[cb], dk[cb]);
  }
#pragma unroll
  for (int cb = 0; cb < 4; ++cb) {
    as[cb] = x.a[cb] * da[cb];
    xs[cb] = p.scale * x.q[cb] * dq[cb] + as[cb] - x.b[cb] * db[cb] - x.k[cb] * dk[cb];
  }
  if (ok) {
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      store_row4<T>(p.dq, at + 16 * cb, dq[cb] * p.scale);
      store_row4<T>(p.da, at + 16 * cb, da[cb]);
      store_row4<T>(p.db, at + 16 * cb, db[cb]);
      store_row4<T>(p.dk, at + 16 * cb, dk[cb]);
    }
  }
  float *tx = t3, *tas = wide ? t1 : t0, *scr = L.sx;  // tas: read by nobody since the last barrier but in the products above
  lds_barrier();
  put_cols(tx, w, xs);
  put_cols(tas, w, as);
  lds_barrier();
  {
    const int c = tid & 63, seg = tid >> 6;
    float val[16], sum = 0.f;
#pragma unroll
    for (int i = 15; i >= 0; --i) val[i] = (sum += tx[(16 * seg + i) * LD + c]);
    scr[64 * seg + c] = sum;
    lds_barrier();
    float after = 0.f;
    for (int j = seg + 1; j < 4; ++j) after += scr[64 * j + c];
#pragma unroll
    for (int j = 0; j < 4; ++j) after += red[64 * j + c];
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (16 * seg + i < s.len) p.dgk[(s.tok + 16 * seg + i) * D + c] = val[i] + after - tas[(16 * seg + i) * LD + c];
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
