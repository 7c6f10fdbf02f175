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
#include "mma_tiles.h"

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

// Eight consecutive elements as loaded
template <typename T> struct Raw8;
template <> struct Raw8<bf16_t> {
  bf16x8 x;
  __device__ __forceinline__ void load(const bf16_t* p, bool ok) {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = (bf16_t)0.f;
    if (ok) x = *reinterpret_cast<const bf16x8*>(p);
  }
  __device__ __forceinline__ float get(int i) const { return (float)x[i]; }
};
template <> struct Raw8<float> {
  floatx4 x[2];
  __device__ __forceinline__ void load(const float* p, bool ok) {
    x[0] = x[1] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (ok) x[0] = load4(p), x[1] = load4(p + 4);
  }
  __device__ __forceinline__ float get(int i) const { return x[i >> 2][i & 3]; }
};

__device__ __forceinline__ void put8(float* p, const float (&v)[8]) {
  store4(p, floatx4{v[0], v[1], v[2], v[3]});
  store4(p + 4, floatx4{v[4], v[5], v[6], v[7]});
}
template <typename R> __device__ __forceinline__ void put8(float* p, const R& r) {
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = r.get(i);
  put8(p, v);
}

// ---- products of 16 x 16 tiles, operands in LDS --------------------------------------------------------------
// Result fragment: r-th element = row i0 + 4 g + r, column j0 + l16 (g = lane / 16, l16 = lane % 16).  The contraction
// index of step r inside a block of 16 is 4 g + r in both operands, so an operand stored with the contraction along its
// rows (ROW) is read as one 16-byte vector per block, the other way round as four single reads of 16 consecutive columns;
// with rows 68 floats apart both touch every bank once.
template <bool ROW> __device__ __forceinline__ floatx4 frag(const float* t, int i, int k) {
  if (ROW) return load4(t + i * LD + k);
  return floatx4{t[k * LD + i], t[(k + 1) * LD + i], t[(k + 2) * LD + i], t[(k + 3) * LD + i]};
}
__device__ __forceinline__ void mfma4(floatx4& c, floatx4 a, floatx4 b) {
#pragma unroll
  for (int r = 0; r < 4; ++r) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r], b[r], c, 0, 0, 0);
}
// c += A[rows i0..][k] B[k][columns j0..] over the blocks kb0 <= kb < kb1 of 16
template <bool AR, bool BR>
__device__ __forceinline__ void mm(floatx4& c, const float* A, int i0, const float* B, int j0, int kb0, int kb1, int l16, int g) {
  for (int kb = kb0; kb < kb1; ++kb) mfma4(c, frag<AR>(A, i0 + l16, 16 * kb + 4 * g), frag<BR>(B, j0 + l16, 16 * kb + 4 * g));
}
// the same for two column tiles over one range
template <bool AR, bool BR>
__device__ __forceinline__ void mm2(floatx4 (&c)[2], const float* A, int i0, const float* B, int j0, int j1, int kb0, int kb1, int l16, int g) {
  for (int kb = kb0; kb < kb1; ++kb) {
    const floatx4 a = frag<AR>(A, i0 + l16, 16 * kb + 4 * g);
    const floatx4 b0 = frag<BR>(B, j0 + l16, 16 * kb + 4 * g), b1 = frag<BR>(B, j1 + l16, 16 * kb + 4 * g);
    mfma4(c[0], a, b0);
    mfma4(c[1], a, b1);
  }
}
template <bool AR, bool BR>
__device__ __forceinline__ void mm2_full(floatx4 (&c)[2], const float* A, int i0, const float* B, int j0, int j1, int l16, int g) {
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const floatx4 a = frag<AR>(A, i0 + l16, 16 * kb + 4 * g);
    const floatx4 b0 = frag<BR>(B, j0 + l16, 16 * kb + 4 * g), b1 = frag<BR>(B, j1 + l16, 16 * kb + 4 * g);
    mfma4(c[0], a, b0);
    mfma4(c[1], a, b1);
  }
}
__device__ __forceinline__ void put_frag(float* t, int i0, int j0, floatx4 c, int l16, int g) {  // [row][column]
#pragma unroll
  for (int r = 0; r < 4; ++r) t[(i0 + 4 * g + r) * LD + j0 + l16] = c[r];
}
__device__ __forceinline__ floatx4 zero4() { return floatx4{0.f, 0.f, 0.f, 0.f}; }

// Eight waves on the 4 x 4 tiles of a 64 x 64 result, two tiles each.  `row`: the wave's row block for results whose
// contraction is cut by the row (waves w and w + 4, which share a SIMD, take complementary ones), columns c0, c1; `rowT`,
// t0, t1: the same for results whose contraction is cut by the column.
struct Role {
  int wave, lane, l16, g, row, c0, c1, rowT, t0, t1;
  __device__ __forceinline__ Role() {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = threadIdx.x & 63;
    l16 = lane & 15, g = lane >> 4;
    row = 16 * (wave < 4 ? wave : 7 - wave);
    c0 = wave < 4 ? 0 : 32, c1 = c0 + 16;
    rowT = 16 * (wave & 3);
    t0 = wave < 4 ? 0 : 16, t1 = 48 - t0;
  }
};

// ---- decays --------------------------------------------------------------------------------------------------
struct Gates {      // arrays of 64 floats in LDS
  float *em, *ec, *eC, *gm;  // e^m, e^(G_C - m), e^G_C, m
  int* wide;                 // some channel's range is too wide for the split: pairs one by one, em = ec = 1
};

// Gt: gk of the chunk on entry ([t][c], visible after the first barrier), its cumulative sum on return; scr: 1536 floats
__device__ __forceinline__ void cumulate(float* Gt, float* scr, const Gates& s) {
  const int tid = threadIdx.x, c = tid & 63, seg = tid >> 6;
  lds_barrier();
  float v[8], sum = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (sum += Gt[(8 * seg + i) * LD + c]);
  scr[64 * seg + c] = sum;
  lds_barrier();
  float pre = 0.f;
  for (int j = 0; j < seg; ++j) pre += scr[64 * j + c];
  float mx = 0.f, mn = 0.f;  // the token before the chunk has G = 0
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float x = pre + v[i];
    Gt[(8 * seg + i) * LD + c] = x;
    mx = fmaxf(mx, x), mn = fminf(mn, x);
  }
  scr[512 + 64 * seg + c] = mx;
  scr[1024 + 64 * seg + c] = mn;
  lds_barrier();
  if (seg == 0) {
#pragma unroll
    for (int j = 1; j < 8; ++j) mx = fmaxf(mx, scr[512 + 64 * j + c]), mn = fminf(mn, scr[1024 + 64 * j + c]);
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

// The chunk's vectors with their factors (q also times scale) -- plain where the chunk is wide
template <typename T> struct Vectors {
  Raw8<T> q, k, a, b;
  Raw8<float> g;
  __device__ __forceinline__ void load(const ChunkParams& p, const Slot& s) {
    const int t = threadIdx.x >> 3, c = (threadIdx.x & 7) * 8;
    const bool ok = t < s.len;
    const int64_t at = (s.tok + t) * D + c;
    g.load(p.gk + at, ok);
    q.load(static_cast<const T*>(p.q) + at, ok);
    a.load(static_cast<const T*>(p.a) + at, ok);
    b.load(static_cast<const T*>(p.b) + at, ok);
    k.load(static_cast<const T*>(p.k) + at, ok);
  }
  __device__ __forceinline__ void store(float* tq, float* ta, float* tb, float* tk, const float* Gt, const Gates& s, float scale) const {
    const int t = threadIdx.x >> 3, c = (threadIdx.x & 7) * 8, at = t * LD + c;
    float vq[8], va[8], vb[8], vk[8];
    if (*s.wide) {
#pragma unroll
      for (int i = 0; i < 8; ++i) vq[i] = scale * q.get(i), va[i] = a.get(i), vb[i] = b.get(i), vk[i] = k.get(i);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float m = s.gm[c + i], G = Gt[at + i], Gp = t ? Gt[at - LD + i] : 0.f;
        const float eb = exp_f(m - G);
        vq[i] = scale * q.get(i) * exp_f(G - m);
        va[i] = a.get(i) * exp_f(Gp - m);
        vb[i] = b.get(i) * eb;
        vk[i] = k.get(i) * eb;
      }
    }
    put8(tq + at, vq);
    put8(ta + at, va);
    put8(tb + at, vb);
    put8(tk + at, vk);
  }
};

// Wide chunk: the tiles' plain vectors become q e^G, a e^Gp, b e^(G_C - G), k e^(G_C - G) (no factor of either sign left over)
__device__ __forceinline__ void rescale_wide(float* tq, float* ta, float* tb, float* tk, const float* Gt) {
  const int t = threadIdx.x >> 3, c = (threadIdx.x & 7) * 8, at = t * LD + c;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float G = Gt[at + i], Gp = t ? Gt[at - LD + i] : 0.f, eb = exp_f(Gt[(C - 1) * LD + c + i] - G);
    tq[at + i] *= exp_f(G);
    ta[at + i] *= exp_f(Gp);
    tb[at + i] *= eb;
    tk[at + i] *= eb;
  }
}

// -Aab, Pqb, Pqk, Aak into their tiles, zeros above the diagonal.  The tiles of a wide chunk hold the plain vectors.
__device__ __forceinline__ void pair_matrices(const float* tq, const float* ta, const float* tb, const float* tk, const float* Gt, bool wide, const Role& w,
                                              float* nAab, float* Pqb, float* Pqk, float* Aak) {
  if (!wide) {
    floatx4 ab[2], ak[2], qb[2], qk[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) ab[j] = ak[j] = qb[j] = qk[j] = zero4();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = j ? w.c1 : w.c0;
      if (col > w.row) continue;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const int k = 16 * kb + 4 * w.g;
        const floatx4 fa = frag<true>(ta, w.row + w.l16, k), fq = frag<true>(tq, w.row + w.l16, k);
        const floatx4 fb = frag<true>(tb, col + w.l16, k), fk = frag<true>(tk, col + w.l16, k);
#pragma unroll
        for (int r = 0; r < 4; ++r) {  // four accumulators in turn: no product waits for the one before it
          ab[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[r], fb[r], ab[j], 0, 0, 0);
          ak[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[r], fk[r], ak[j], 0, 0, 0);
          qb[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fq[r], fb[r], qb[j], 0, 0, 0);
          qk[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fq[r], fk[r], qk[j], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = (j ? w.c1 : w.c0) + w.l16;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = w.row + 4 * w.g + r;
        nAab[t * LD + col] = col < t ? -ab[j][r] : 0.f;
        Aak[t * LD + col] = col < t ? ak[j][r] : 0.f;
        Pqb[t * LD + col] = col <= t ? qb[j][r] : 0.f;
        Pqk[t * LD + col] = col <= t ? qk[j][r] : 0.f;
      }
    }
    return;
  }
  const int t = threadIdx.x >> 3;
  for (int s = threadIdx.x & 7; s < C; s += 8) {
    float ab = 0.f, ak = 0.f, qb = 0.f, qk = 0.f;
    if (s <= t) {
      for (int c = 0; c < D; ++c) {
        const float G = Gt[s * LD + c], eq = exp_f(Gt[t * LD + c] - G);
        qb += tq[t * LD + c] * eq * tb[s * LD + c];
        qk += tq[t * LD + c] * eq * tk[s * LD + c];
        if (s < t) {
          const float ea = exp_f(Gt[(t - 1) * LD + c] - G);
          ab += ta[t * LD + c] * ea * tb[s * LD + c];
          ak += ta[t * LD + c] * ea * tk[s * LD + c];
        }
      }
    }
    nAab[t * LD + s] = -ab;
    Aak[t * LD + s] = ak;
    Pqb[t * LD + s] = qb;
    Pqk[t * LD + s] = qk;
  }
}

constexpr int LDS_TILES = 9;
constexpr unsigned LDS_BYTES = (LDS_TILES * TS + 4 * 64 + 4 + 32 * 36) * sizeof(float);
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
__global__ __launch_bounds__(512) void dplr_prepare_kernel(ChunkParams p) {
  extern __shared__ __align__(16) char smem[];
  const Lds L(smem);
  const Slot s = slot_of(p);
  const Role w;
  float *tq = L.tile(0), *ta = L.tile(1), *tb = L.tile(2), *tk = L.tile(3), *Tm = L.tile(4), *Pqb = L.tile(5), *Pqk = L.tile(6), *Aak = L.tile(7), *tv = L.tile(8);
  const int t = threadIdx.x >> 3, c8 = (threadIdx.x & 7) * 8;
  Vectors<T> x;
  x.load(p, s);
  Raw8<T> v;
  v.load(static_cast<const T*>(p.v) + (s.tok + t) * D + c8, t < s.len);
  put8(tv + t * LD + c8, x.g);  // G until the pairs are done
  cumulate(tv, Pqb, L.gate);
  x.store(tq, ta, tb, tk, tv, L.gate, p.scale);
  lds_barrier();
  const bool wide = *L.gate.wide;
  pair_matrices(tq, ta, tb, tk, tv, wide, w, Tm, Pqb, Pqk, Aak);
  lds_barrier();
  if (wide) {
    rescale_wide(tq, ta, tb, tk, tv);
    lds_barrier();
  }
  put8(tv + t * LD + c8, v);
  lds_barrier();
  floatx4 z[2] = {zero4(), zero4()};
  mm2<true, false>(z, Aak, w.row, tv, w.c0, w.c1, 0, w.row / 16 + 1, w.l16, w.g);  // Aak v
  tri_inverse_64<true, 512>(Tm, Tm, L.sx, threadIdx.x);
  put_frag(Aak, w.row, w.c0, z[0], w.l16, w.g);  // every wave has passed a barrier since its last read of Aak
  put_frag(Aak, w.row, w.c1, z[1], w.l16, w.g);
  lds_barrier();
  floatx4 W[2] = {zero4(), zero4()}, u[2] = {zero4(), zero4()};
  mm2<true, false>(W, Tm, w.row, ta, w.c0, w.c1, 0, w.row / 16 + 1, w.l16, w.g);
  mm2<true, false>(u, Tm, w.row, Aak, w.c0, w.c1, 0, w.row / 16 + 1, w.l16, w.g);
  lds_barrier();
  float *tW = ta, *tU = Aak;
  put_frag(tW, w.row, w.c0, W[0], w.l16, w.g);
  put_frag(tW, w.row, w.c1, W[1], w.l16, w.g);
  put_frag(tU, w.row, w.c0, u[0], w.l16, w.g);
  put_frag(tU, w.row, w.c1, u[1], w.l16, w.g);
  lds_barrier();
  // Results as [column][4 consecutive rows]: 16-byte stores
  const int i0 = w.rowT, ch = i0 + 4 * w.g;  // this lane's four channels (of M's columns, X's columns, N^T's columns, Y's)
  {
    floatx4 m[2] = {zero4(), zero4()}, nt[2] = {zero4(), zero4()};
    mm2_full<false, false>(m, tW, i0, tb, w.t0, w.t1, w.l16, w.g);    // M[i][c] at rows c, columns i
    mm2_full<false, false>(nt, tb, i0, tU, w.t0, w.t1, w.l16, w.g);   // N[i][n] at rows i, columns n
    mm2_full<false, false>(nt, tk, i0, tv, w.t0, w.t1, w.l16, w.g);
    const floatx4 em = load4(L.gate.em + ch), ec4 = load4(L.gate.ec + ch);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = (j ? w.t1 : w.t0) + w.l16;
      floatx4 r = m[j] * em * L.gate.ec[col];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (ch + e == col) r[e] += L.gate.eC[col];
      store4(p.M + s.kept * TG + col * D + ch, r);
      store4(p.s1 + s.win * TG + col * D + ch, nt[j] * ec4);
    }
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = j ? w.t1 : w.t0, tt = col + w.l16;  // this lane's token
    floatx4 xx = zero4(), y = zero4();
    mm<false, true>(xx, tW, i0, Pqb, col, 0, col / 16 + 1, w.l16, w.g);
    mm<false, true>(y, tU, i0, Pqb, col, 0, col / 16 + 1, w.l16, w.g);
    mm<false, true>(y, tv, i0, Pqk, col, 0, col / 16 + 1, w.l16, w.g);
    store4(p.X + s.kept * TG + tt * D + ch, (xx + load4(tq + tt * LD + ch)) * load4(L.gate.em + ch));
    store4(p.s2 + s.win * TG + tt * D + ch, y);
  }
}

// ---- the sequential pass: h <- M h + N (forward), D <- M^T D + R (backward) ------------------------------------
// One workgroup per row; wave w owns 16 of the 64 value columns, whose part of the state stays in four accumulator
// fragments: an accumulator fragment is the B operand of the next product as it stands (its rows 16 b + 4 g + r are the
// contraction indices that step r of block b wants in lane group g), so the state never leaves the wave.  M arrives
// through registers two chunks ahead and one LDS tile ahead; one LDS barrier per chunk.  64 products of 32 cycles on the
// chain of a chunk, 0.9 us.
struct ScanParams {
  const float* M;    // kept tiles [rows][KN]
  const float* add;  // window tiles: N^T or R^T
  float* st;         // the state entering (forward: kept [rows][KN + 1]) or the gradient leaving (backward: window) each chunk, transposed
  const float* s_in; // [dk][dv] per row, or NULL
  float* s_out;      // [dk][dv] per row, or NULL
  int KN, at, nw;    // the window is chunks [at, at + nw) of the kept tensors
};

template <bool BWD>
__global__ __launch_bounds__(256) void dplr_chunk_scan_kernel(ScanParams p) {
  __shared__ __align__(16) float buf[2][TS];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int64_t row = blockIdx.x;
  const int col = 16 * wave + l16;
  const float* Mrow = p.M + (row * p.KN + p.at) * TG;
  const float* Arow = p.add + row * p.nw * TG + col * D + 4 * g;
  float* Srow = p.st + (BWD ? row * p.nw : row * (p.KN + 1) + p.at) * TG + col * D + 4 * g;
  auto chunk = [&](int i) { return (int64_t)(BWD ? p.nw - 1 - i : i); };
  floatx4 h[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) h[b][r] = p.s_in ? p.s_in[row * TG + (16 * b + 4 * g + r) * D + col] : 0.f;
  struct Ahead {
    floatx4 m[4], a[4];
  } r0, r1;
  const int lr = tid >> 2, lc = (tid & 3) * 4;  // this thread's row of M and its first column in each quarter
  auto fetch = [&](Ahead& x, int i) {
    const int64_t n = chunk(min(i, p.nw - 1));
#pragma unroll
    for (int q = 0; q < 4; ++q) x.m[q] = load4(Mrow + n * TG + lr * D + 16 * q + lc);
#pragma unroll
    for (int q = 0; q < 4; ++q) x.a[q] = load4(Arow + n * TG + 16 * q);
  };
  auto stage = [&](const Ahead& x, float* dst) {
#pragma unroll
    for (int q = 0; q < 4; ++q) store4(dst + lr * LD + 16 * q + lc, x.m[q]);
  };
  auto step = [&](const Ahead& x, const float* M, int i) {
    floatx4 y[4];
    float* out = Srow + chunk(i) * TG;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      store4(out + 16 * b, h[b]);
      y[b] = x.a[b];
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {  // contraction block
      floatx4 f[4];
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) f[ib] = frag<!BWD>(M, 16 * ib + l16, 16 * b + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) y[ib] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[ib][r], h[b][r], y[ib], 0, 0, 0);
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) h[b] = y[b];
  };
  fetch(r0, 0);
  fetch(r1, 1);
  stage(r0, buf[0]);
  for (int i = 0; i < p.nw; i += 2) {
    lds_barrier();
    step(r0, buf[0], i);
    stage(r1, buf[1]);
    fetch(r0, i + 2);
    if (i + 1 >= p.nw) break;
    lds_barrier();
    step(r1, buf[1], i + 1);
    stage(r0, buf[0]);
    fetch(r1, i + 3);
  }
  if (!BWD && p.at + p.nw == p.KN) {
#pragma unroll
    for (int b = 0; b < 4; ++b) store4(Srow + (int64_t)p.nw * TG + 16 * b, h[b]);
  }
  if (p.s_out) {
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) p.s_out[row * TG + (16 * b + 4 * g + r) * D + col] = h[b][r];
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
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int t = (threadIdx.x >> 3) + 32 * h, c = (threadIdx.x & 7) * 8;
    Raw8<float> x;
    Raw8<T> d;
    x.load(p.X + s.kept * TG + t * D + c, true);
    d.load(static_cast<const T*>(p.d_o) + (s.tok + t) * D + c, t < s.len);
    put8(tX + t * LD + c, x);
    put8(tO + t * LD + c, d);
  }
  lds_barrier();
  floatx4 acc[4] = {zero4(), zero4(), zero4(), zero4()};
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const floatx4 a = frag<false>(tX, 16 * wave + l16, 16 * kb + 4 * g);
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) mfma4(acc[nb], a, frag<false>(tO, 16 * nb + l16, 16 * kb + 4 * g));
  }
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) store4(p.s2 + s.win * TG + (16 * nb + l16) * D + 16 * wave + 4 * g, acc[nb]);
}

// ---- backward: u, dU and dv of a chunk -----------------------------------------------------------------------
// The pair matrices and the inverse are formed again: keeping them would move 128 KB per chunk through memory.
template <typename T>
__global__ __launch_bounds__(512) void dplr_u_kernel(ChunkParams p) {
  extern __shared__ __align__(16) char smem[];
  const Lds L(smem);
  const Slot s = slot_of(p);
  const Role w;
  float *tq = L.tile(0), *ta = L.tile(1), *tb = L.tile(2), *tk = L.tile(3), *Tm = L.tile(4), *Pqb = L.tile(5), *Pqk = L.tile(6), *Aak = L.tile(7), *tv = L.tile(8);
  const int t = threadIdx.x >> 3, c8 = (threadIdx.x & 7) * 8, at = t * LD + c8;
  Vectors<T> x;
  x.load(p, s);
  Raw8<T> v, d_o;
  v.load(static_cast<const T*>(p.v) + (s.tok + t) * D + c8, t < s.len);
  d_o.load(static_cast<const T*>(p.d_o) + (s.tok + t) * D + c8, t < s.len);
  Raw8<float> h0, dC;
  h0.load(p.hT + s.st * TG + t * D + c8, true);
  dC.load(p.s1 + s.win * TG + t * D + c8, true);
  put8(tv + at, x.g);
  cumulate(tv, Pqb, L.gate);
  x.store(tq, ta, tb, tk, tv, L.gate, p.scale);
  lds_barrier();
  const bool wide = *L.gate.wide;
  pair_matrices(tq, ta, tb, tk, tv, wide, w, Tm, Pqb, Pqk, Aak);
  lds_barrier();
  if (wide) {
    rescale_wide(tq, ta, tb, tk, tv);
    lds_barrier();
  }
  put8(tv + at, v);
  {
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = h0.get(i) * L.gate.em[c8 + i];
    put8(tq + at, y);  // e^m h, [value column][channel]; q is not needed any more
  }
  lds_barrier();
  floatx4 z[2] = {zero4(), zero4()};
  mm2_full<true, true>(z, ta, w.row, tq, w.c0, w.c1, w.l16, w.g);                   // a h
  mm2<true, false>(z, Aak, w.row, tv, w.c0, w.c1, 0, w.row / 16 + 1, w.l16, w.g);   // + Aak v
  tri_inverse_64<true, 512>(Tm, Tm, L.sx, threadIdx.x);
  put_frag(ta, w.row, w.c0, z[0], w.l16, w.g);
  put_frag(ta, w.row, w.c1, z[1], w.l16, w.g);
  put8(tv + at, d_o);
  {
    float y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = dC.get(i) * L.gate.ec[c8 + i];
    put8(tq + at, y);  // e^(G_C - m) D, [value column][channel]
  }
  lds_barrier();
  // u = Tm z: rows = value columns, columns = tokens
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = j ? w.t1 : w.t0;
    floatx4 u = zero4();
    mm<false, true>(u, ta, w.rowT, Tm, col, 0, col / 16 + 1, w.l16, w.g);
    store4(p.s3 + s.win * TG + (col + w.l16) * D + w.rowT + 4 * w.g, u);
  }
  floatx4 y[2] = {zero4(), zero4()};
  mm2_full<true, true>(y, tb, w.row, tq, w.c0, w.c1, w.l16, w.g);                        // Bg D
  mm2<false, false>(y, Pqb, w.row, tv, w.c0, w.c1, w.row / 16, 4, w.l16, w.g);           // + Pqb^T dO
  floatx4 dv[2] = {zero4(), zero4()};
#pragma unroll
  for (int j = 0; j < 2; ++j) {  // rows = value columns, columns = tokens
    const int col = j ? w.t1 : w.t0;
    mm<true, true>(dv[j], tq, w.rowT, tk, col, 0, 4, w.l16, w.g);                        // Kg D
    mm<false, false>(dv[j], tv, w.rowT, Pqk, col, col / 16, 4, w.l16, w.g);              // + Pqk^T dO
  }
  lds_barrier();
  put_frag(ta, w.row, w.c0, y[0], w.l16, w.g);
  put_frag(ta, w.row, w.c1, y[1], w.l16, w.g);
  lds_barrier();
  floatx4 du[2] = {zero4(), zero4()};
  mm2<false, false>(du, Tm, w.row, ta, w.c0, w.c1, w.row / 16, 4, w.l16, w.g);
  put_frag(tb, w.row, w.c0, du[0], w.l16, w.g);  // b was last read before two barriers
  put_frag(tb, w.row, w.c1, du[1], w.l16, w.g);
  lds_barrier();
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = j ? w.t1 : w.t0, tt = col + w.l16;
    mm<false, false>(dv[j], tb, w.rowT, Aak, col, col / 16, 4, w.l16, w.g);              // + Aak^T dU
    if (tt < s.len) store_row4<T>(p.dv, (s.tok + tt) * D + w.rowT + 4 * w.g, dv[j]);
  }
  store4(p.s4 + s.win * TG + t * D + c8, load4(tb + at));
  store4(p.s4 + s.win * TG + t * D + c8 + 4, load4(tb + at + 4));
}

// ---- backward: dq, dk, da, db, dgk of a chunk ----------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(512) void dplr_grad_kernel(ChunkParams p) {
  extern __shared__ __align__(16) char smem[];
  const Lds L(smem);
  const Slot s = slot_of(p);
  const Role w;
  const int tid = threadIdx.x, t = tid >> 3, c8 = (tid & 7) * 8, at = t * LD + c8;
  float *Gt = L.tile(8), *prod = L.tile(6);
  float* red = L.sx;  // [8][64]: partial sums of <D, h'> per channel
  Vectors<T> x;
  x.load(p, s);
  {
    Raw8<T> v, d_o;
    Raw8<float> u, du, h0, dC, hC;
    v.load(static_cast<const T*>(p.v) + (s.tok + t) * D + c8, t < s.len);
    d_o.load(static_cast<const T*>(p.d_o) + (s.tok + t) * D + c8, t < s.len);
    const int64_t wt = s.win * TG + t * D + c8, ht = s.st * TG + t * D + c8;
    u.load(p.s3 + wt, true);
    du.load(p.s4 + wt, true);
    h0.load(p.hT + ht, true);
    hC.load(p.hT + ht + TG, true);
    dC.load(p.s1 + wt, true);
    put8(Gt + at, x.g);
    cumulate(Gt, L.tile(7), L.gate);
    put8(L.tile(0) + at, v);
    put8(L.tile(1) + at, d_o);
    put8(L.tile(2) + at, u);
    put8(L.tile(3) + at, du);
    float y[8], z[8], r[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      y[i] = h0.get(i) * L.gate.em[c8 + i];
      z[i] = dC.get(i) * L.gate.ec[c8 + i];
      r[i] = dC.get(i) * hC.get(i);
    }
    put8(L.tile(4) + at, y);
    put8(L.tile(5) + at, z);
    put8(prod + at, r);
  }
  lds_barrier();
  const float *tv = L.tile(0), *tO = L.tile(1), *tu = L.tile(2), *tdu = L.tile(3), *th = L.tile(4), *tD = L.tile(5);
  {
    const int c = tid & 63, seg = tid >> 6;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) sum += prod[(8 * seg + i) * LD + c];
    red[64 * seg + c] = sum;
  }
  floatx4 pb[2], pk[2], ab[2], ak[2];  // dPqb, dPqk, dAab, dAak
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    pb[j] = pk[j] = ab[j] = ak[j] = zero4();
    const int col = j ? w.c1 : w.c0;
    if (col > w.row) continue;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const int k = 16 * kb + 4 * w.g;
      const floatx4 fo = frag<true>(tO, w.row + w.l16, k), fd = frag<true>(tdu, w.row + w.l16, k);
      const floatx4 fu = frag<true>(tu, col + w.l16, k), fv = frag<true>(tv, col + w.l16, k);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        pb[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fo[r], fu[r], pb[j], 0, 0, 0);
        pk[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fo[r], fv[r], pk[j], 0, 0, 0);
        ab[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fd[r], fu[r], ab[j], 0, 0, 0);
        ak[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fd[r], fv[r], ak[j], 0, 0, 0);
      }
    }
  }
  // rows = channels, columns = tokens from here on
  floatx4 dq[2] = {zero4(), zero4()}, da[2] = {zero4(), zero4()}, db[2] = {zero4(), zero4()}, dk[2] = {zero4(), zero4()};
  mm2_full<false, true>(dq, th, w.rowT, tO, w.t0, w.t1, w.l16, w.g);
  mm2_full<false, true>(da, th, w.rowT, tdu, w.t0, w.t1, w.l16, w.g);
  mm2_full<false, true>(db, tD, w.rowT, tu, w.t0, w.t1, w.l16, w.g);
  mm2_full<false, true>(dk, tD, w.rowT, tv, w.t0, w.t1, w.l16, w.g);
  lds_barrier();
  float *Mb = L.tile(0), *Mk = L.tile(1), *Nb = L.tile(2), *Nk = L.tile(3), *tq = L.tile(4), *ta = L.tile(5), *tb = L.tile(6), *tk = L.tile(7);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = (j ? w.c1 : w.c0) + w.l16;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tt = w.row + 4 * w.g + r, o = tt * LD + col;
      Mb[o] = col <= tt ? pb[j][r] : 0.f;
      Mk[o] = col <= tt ? pk[j][r] : 0.f;
      Nb[o] = col < tt ? ab[j][r] : 0.f;
      Nk[o] = col < tt ? ak[j][r] : 0.f;
    }
  }
  x.store(tq, ta, tb, tk, Gt, L.gate, p.scale);
  lds_barrier();
  const bool wide = *L.gate.wide;
  const int ch = w.rowT + 4 * w.g;
  floatx4 xs[2], as[2];  // q dq + a da - b db - k dk and a da
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int col = j ? w.t1 : w.t0, tt = col + w.l16, cb = col / 16;
    if (!wide) {
      mm<false, true>(dq[j], tb, w.rowT, Mb, col, 0, cb + 1, w.l16, w.g);
      mm<false, true>(dq[j], tk, w.rowT, Mk, col, 0, cb + 1, w.l16, w.g);
      mm<false, true>(da[j], tb, w.rowT, Nb, col, 0, cb + 1, w.l16, w.g);
      mm<false, true>(da[j], tk, w.rowT, Nk, col, 0, cb + 1, w.l16, w.g);
      mm<false, false>(db[j], tq, w.rowT, Mb, col, cb, 4, w.l16, w.g);
      mm<false, false>(db[j], ta, w.rowT, Nb, col, cb, 4, w.l16, w.g);
      mm<false, false>(dk[j], tq, w.rowT, Mk, col, cb, 4, w.l16, w.g);
      mm<false, false>(dk[j], ta, w.rowT, Nk, col, cb, 4, w.l16, w.g);
    }
    const floatx4 G = load4(Gt + tt * LD + ch), Gp = tt ? load4(Gt + (tt - 1) * LD + ch) : zero4(), gl = load4(Gt + (C - 1) * LD + ch);
    const floatx4 q4 = load4(tq + tt * LD + ch), a4 = load4(ta + tt * LD + ch), b4 = load4(tb + tt * LD + ch), k4 = load4(tk + tt * LD + ch);
    if (!wide) {
      const floatx4 m = load4(L.gate.gm + ch);
      as[j] = a4 * da[j];
      xs[j] = q4 * dq[j] + as[j] - b4 * db[j] - k4 * dk[j];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float eb = exp_f(m[e] - G[e]);
        dq[j][e] *= exp_f(G[e] - m[e]);
        da[j][e] *= exp_f(Gp[e] - m[e]);
        db[j][e] *= eb;
        dk[j][e] *= eb;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = ch + e;
        const float eb = exp_f(gl[e] - G[e]);
        float rq = exp_f(G[e]) * dq[j][e], ra = exp_f(Gp[e]) * da[j][e], rb = eb * db[j][e], rk = eb * dk[j][e];
        for (int i = 0; i <= tt; ++i) {
          const float eq = exp_f(G[e] - Gt[i * LD + c]);
          rq += eq * (Mb[tt * LD + i] * tb[i * LD + c] + Mk[tt * LD + i] * tk[i * LD + c]);
          if (i < tt) ra += exp_f(Gp[e] - Gt[i * LD + c]) * (Nb[tt * LD + i] * tb[i * LD + c] + Nk[tt * LD + i] * tk[i * LD + c]);
        }
        for (int i = tt; i < C; ++i) {
          const float eq = exp_f(Gt[i * LD + c] - G[e]) * tq[i * LD + c];
          rb += eq * Mb[i * LD + tt];
          rk += eq * Mk[i * LD + tt];
          if (i > tt) {
            const float ea = exp_f(Gt[(i - 1) * LD + c] - G[e]) * ta[i * LD + c];
            rb += ea * Nb[i * LD + tt];
            rk += ea * Nk[i * LD + tt];
          }
        }
        dq[j][e] = rq, da[j][e] = ra, db[j][e] = rb, dk[j][e] = rk;
      }
      as[j] = a4 * da[j];
      xs[j] = q4 * dq[j] + as[j] - b4 * db[j] - k4 * dk[j];
    }
    if (tt < s.len) {
      const int64_t o = (s.tok + tt) * D + ch;
      store_row4<T>(p.dq, o, dq[j] * p.scale);
      store_row4<T>(p.da, o, da[j]);
      store_row4<T>(p.db, o, db[j]);
      store_row4<T>(p.dk, o, dk[j]);
    }
  }
  lds_barrier();
  float *tx = L.tile(0), *tas = L.tile(1), *scr = L.tile(2);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int tt = (j ? w.t1 : w.t0) + w.l16;
    store4(tx + tt * LD + ch, xs[j]);
    store4(tas + tt * LD + ch, as[j]);
  }
  lds_barrier();
  {
    const int c = tid & 63, seg = tid >> 6;
    float v[8], sum = 0.f;
#pragma unroll
    for (int i = 7; i >= 0; --i) v[i] = (sum += tx[(8 * seg + i) * LD + c]);
    scr[64 * seg + c] = sum;
    lds_barrier();
    float after = 0.f;
    for (int j = seg + 1; j < 8; ++j) after += scr[64 * j + c];
#pragma unroll
    for (int j = 0; j < 8; ++j) after += red[64 * j + c];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (8 * seg + i < s.len) p.dgk[(s.tok + 8 * seg + i) * D + c] = v[i] + after - tas[(8 * seg + i) * LD + c];
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

template <typename K> int lds_limit(K* k) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_BYTES);
  return e == hipSuccess ? LNX_OK : lnx_set_error(LNX_ERR_LAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(e));
}

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
    hipLaunchKernelGGL(dplr_prepare_kernel<T>, dim3(grid), dim3(512), LDS_BYTES, st, p);
    lnx_profile_mark("dplr_chunk_scan", st);
    const ScanParams sp{p.M, p.s1, p.hT, n0 ? a->final_state : a->initial_state, a->final_state, p.KN, n0 - p.k0, p.nw};
    hipLaunchKernelGGL(dplr_chunk_scan_kernel<false>, dim3((unsigned)rows), dim3(256), 0, st, sp);
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
    const ScanParams sp{p.M, p.s2, p.s1, i == nwin - 1 ? g->d_final_state : carry, i ? carry : g->d_initial_state, p.KN, p.n0, p.nw};
    hipLaunchKernelGGL(dplr_chunk_scan_kernel<true>, dim3((unsigned)rows), dim3(256), 0, st, sp);
    lnx_profile_mark("dplr_u", st);
    hipLaunchKernelGGL(dplr_u_kernel<T>, dim3(grid), dim3(512), LDS_BYTES, st, p);
    lnx_profile_mark("dplr_grad", st);
    hipLaunchKernelGGL(dplr_grad_kernel<T>, dim3(grid), dim3(512), LDS_BYTES, st, p);
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
