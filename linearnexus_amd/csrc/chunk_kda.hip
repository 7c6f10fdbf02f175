// Chunk-local gradients of the per-channel gate (KDA) for 2-byte inputs with dk <= 128: one kernel between the reverse scan and the
// caller's tensors.  The scans (chunk_fwd.hip, chunk_bwd.hip) leave D, the states S entering the chunks, dD and the state gradients dS'
// leaving them; with G the cumulative gate of the chunk (fp32, per channel), E_ij = e^{G_i - G_j} and r_t = e^{G_C - G_t},
//
//   dR  = Tm^T dD          dv = beta dR                 dPm = scale tril(dO D^T)       dXa = -tril(dR D^T, -1)
//   dq  = scale e^G (dO S^T) + sum_j dPm_tj E_tj k_j
//   row = sum_j dXa_tj E_tj k_j - e^G (dR S^T)          m_t = <k_t, row_t>             dbeta = <dR, v> + m
//   dk  = beta row + r (D dS'^T) + sum_i dPm_it E_it q_i + sum_i beta_i dXa_it E_it k_i
//   dG  = q dq - k dk + 2 beta k row  per channel;      dG_C += sum_t r_t k_t (D dS'^T)_t + e^{G_C} <dS', S>;   dg = reverse cumsum(dG)
//
// the adjoint of linearnexus/modules/linear_attn/kda.py:569-648 in the form of chunk_direct.hip: neither dW = -dD S^T nor W, U and the
// forward pass's X are needed, nor partial sums of dk and dG in memory between two kernels.
//
// One workgroup per chunk, four waves per 64 channels.  A loop over 32-column slabs of the value dimension (LDS-direct loads, NBUF slabs
// in flight) forms dR and accumulates what contracts over value columns on 16x16x32 products: wave w of a team owns the 16 channels
// 16 w .. of its 64 and all tokens, so that an accumulator element is at the place where pair_levels wants its channel and token:
// lane (c = lane % 16, kq = lane / 16) holds the tokens 16 t + 4 kq + e of channel c, and everything between the loop and the
// tiles on their way out happens in registers.  The four pair sums share their factors (pair_sums).
//@@MEASURED@@

#include "chunk_common.h"
#include "reduce_rows.h"

namespace {

using T = bf16_t;
typedef Mma16 S16;
typedef S16::Frag Frag;
template <typename X> __device__ __forceinline__ X* at(char* ws, uint64_t off) { return reinterpret_cast<X*>(ws + off); }
constexpr float LOG2E = 1.4426950408889634f;
constexpr int LDX = LNX_C + 8, LDF = 64 + 4;  // bf16 and fp32 [64][64] tiles

// The four tokens 16 t + 4 kq + e of column c0 + l16 of a bf16 [64][LDX] tile: one transposing read
__device__ __forceinline__ bf16x4 column4(const T* tile, int t, int c0, int lane) { return S16::rows4(tile, LDX, 16 * t + 4 * (lane >> 4), c0, lane); }
// A operands of the 16x16x16 products from such a tile: block (ti, t), lane = (row l16, k-slots 4 kq + e); transposed: (column l16, rows)
__device__ __forceinline__ bf16x4 block_rows(const T* X, int ti, int t, int lane) {
  return *reinterpret_cast<const bf16x4*>(X + (16 * ti + (lane & 15)) * LDX + 16 * t + 4 * (lane >> 4));
}
__device__ __forceinline__ bf16x4 block_cols(const T* X, int ti, int t, int lane) { return column4(X, ti, 16 * t, lane); }

// pair_levels (chunk_common.h) for two matrices at once.  Per level every token has one factor, and P and A share it and the column
// tokens' operand F k:
//   rp[i] += sum_{j < i} P_ij E_ij k_j     ra[i] += sum_{j < i} A_ij E_ij k_j     co[j] += sum_{i > j} E_ij (P_ij q_i + A_ij (beta k)_i)
// Lane, index 4 t + e and levels as there; g = G log2(e).  P and A: bf16 [64][LDX].
struct PairSums {
  float rp[16], ra[16], co[16];
  // Everything so far is computed here: arithmetic may pass a scheduling barrier, loads may not, and what had been loaded for sums that were
  // put off went to scratch memory.
  __device__ __forceinline__ void settle() {
#pragma unroll
    for (int x = 0; x < 16; ++x) asm volatile("" : "+v"(rp[x]), "+v"(ra[x]), "+v"(co[x]));
  }
};
template <int H>
__device__ __forceinline__ void sums_cross(PairSums& s, const float (&g)[16], const float (&dec)[16], const bf16x4 (&k4)[4], const bf16x4 (&q4)[4],
                                           const float* __restrict__ beta, const T* __restrict__ P, const T* __restrict__ A, const float* __restrict__ G, int c, int lane_) {
  const int lane = fresh(lane_);  // the matrices' blocks are read where they are used
  const float m0 = LOG2E * G[H * LDF + c], m1 = H == 32 ? m0 : LOG2E * G[48 * LDF + c];
  float F[16];
  bf16x4 B[4], Bk[4];  // a column block's F k; a row block's F q and F beta k
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const bool up = ((16 * t) & H) != 0;
    const float ref = (H == 32 || t < 2) ? m0 : m1;
    // one exponential per four tokens, the others by the single-step decays: away from the reference the factors shrink
    if (up) {
      F[4 * t] = __builtin_amdgcn_exp2f(fminf(g[4 * t] - ref, 0.f));
#pragma unroll
      for (int e = 1; e < 4; ++e) F[4 * t + e] = F[4 * t + e - 1] * dec[4 * t + e];
    } else {
      F[4 * t + 3] = __builtin_amdgcn_exp2f(fminf(ref - g[4 * t + 3], 0.f));
#pragma unroll
      for (int e = 2; e >= 0; --e) F[4 * t + e] = F[4 * t + e + 1] * dec[4 * t + e + 1];
    }
    floatx4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = F[4 * t + e] * (float)(up ? q4[t][e] : k4[t][e]);
    B[t] = pack_bf16x4(v);
    if (up) {
      const floatx4 bt = load4(beta + 16 * t + 4 * (lane >> 4));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = F[4 * t + e] * (bt[e] * (float)k4[t][e]);
      Bk[t] = pack_bf16x4(v);
    }
  }
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ti = 1; ti < 4; ++ti) {
    if (H == 32 ? ti < 2 : !(ti & 1)) continue;
    floatx4 xp = zero, xa = zero;
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (H == 32 ? t < 2 : t == ti - 1) {
        xp = mfma16_bf16(block_rows(P, ti, t, lane), B[t], xp);
        xa = mfma16_bf16(block_rows(A, ti, t, lane), B[t], xa);
      }
#pragma unroll
    for (int e = 0; e < 4; ++e) s.rp[4 * ti + e] += F[4 * ti + e] * xp[e], s.ra[4 * ti + e] += F[4 * ti + e] * xa[e];
  }
#pragma unroll
  for (int tj = 0; tj < 3; ++tj) {
    if (H == 32 ? tj >= 2 : (tj & 1)) continue;
    floatx4 x = zero;
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (H == 32 ? t >= 2 : t == tj + 1) {
        x = mfma16_bf16(block_cols(P, t, tj, lane), B[t], x);
        x = mfma16_bf16(block_cols(A, t, tj, lane), Bk[t], x);
      }
#pragma unroll
    for (int e = 0; e < 4; ++e) s.co[4 * tj + e] += F[4 * tj + e] * x[e];
  }
}

// Levels 8, 4, 2, 1 of the diagonal 16x16 block t
__device__ __forceinline__ void sums_diag(PairSums& s, const float (&g)[16], const float (&dec)[16], const bf16x4 (&kb)[4], const bf16x4 (&qb)[4],
                                          const float* __restrict__ beta, const T* __restrict__ P, const T* __restrict__ A, const float* __restrict__ G, int c, int t, int lane_) {
  const int lane = fresh(lane_);
  typedef unsigned uint2_ __attribute__((ext_vector_type(2)));
  const int l16 = lane & 15, kq = lane >> 4;
  const uint2_ pr = __builtin_bit_cast(uint2_, block_rows(P, t, t, lane)), pc = __builtin_bit_cast(uint2_, block_cols(P, t, t, lane));
  const uint2_ ar = __builtin_bit_cast(uint2_, block_rows(A, t, t, lane)), ac = __builtin_bit_cast(uint2_, block_cols(A, t, t, lane));
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  const float d1 = dec[4 * t + 1], d2 = dec[4 * t + 2], d3 = dec[4 * t + 3];
  const floatx4 k4 = {(float)kb[t][0], (float)kb[t][1], (float)kb[t][2], (float)kb[t][3]}, q4 = {(float)qb[t][0], (float)qb[t][1], (float)qb[t][2], (float)qb[t][3]};
  const floatx4 b4 = load4(beta + 16 * t + 4 * kq) * k4;
#pragma unroll
  for (int H = 8; H >= 1; H >>= 1) {
    floatx4 fu, fl;  // the factor of each token in its role at this level (row token: fu, column token: fl), 0 in the other
    if (H >= 4) {  // all four tokens share the role and the reference: one exponential, the rest by the single-step decays
      const bool up = H == 8 ? (kq & 2) != 0 : (kq & 1) != 0;
      const float ref = LOG2E * G[(16 * t + (H == 8 ? 8 : 8 * (kq >> 1) + 4)) * LDF + c];
      const float f = __builtin_amdgcn_exp2f(fminf(up ? g[4 * t] - ref : ref - g[4 * t + 3], 0.f));
      floatx4 F;
      F[0] = up ? f : f * d3 * d2 * d1;
      F[1] = up ? f * d1 : f * d3 * d2;
      F[2] = up ? F[1] * d2 : f * d3;
      F[3] = up ? F[2] * d3 : f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        fu[e] = up ? F[e] : 0.f;
        fl[e] = up ? 0.f : F[e];
      }
    } else if (H == 2) {  // reference: token 2 of the four
      fl = floatx4{d1 * d2, d2, 0.f, 0.f};
      fu = floatx4{0.f, 0.f, 1.f, d3};
    } else {  // references: tokens 1 and 3
      fl = floatx4{d1, 0.f, d3, 0.f};
      fu = floatx4{0.f, 1.f, 0.f, 1.f};
    }
    // k-slots (0, 1) and (2, 3) each share a 2-token segment, so the masks act on whole dwords of the packed operand
    uint2_ mk;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const bool on = H == 8 ? true : H == 4 ? (l16 >> 3) == (kq >> 1) : H == 2 ? (l16 >> 2) == kq : (l16 >> 1) == 2 * kq + w;
      mk[w] = on ? 0xffffffffu : 0u;
    }
    const bf16x4 B = pack_bf16x4(fl * k4);
    const floatx4 rp = mfma16_bf16(__builtin_bit_cast(bf16x4, pr & mk), B, zero), ra = mfma16_bf16(__builtin_bit_cast(bf16x4, ar & mk), B, zero);
    floatx4 x = mfma16_bf16(__builtin_bit_cast(bf16x4, pc & mk), pack_bf16x4(fu * q4), zero);
    x = mfma16_bf16(__builtin_bit_cast(bf16x4, ac & mk), pack_bf16x4(fu * b4), x);
#pragma unroll
    for (int e = 0; e < 4; ++e) s.rp[4 * t + e] += fu[e] * rp[e], s.ra[4 * t + e] += fu[e] * ra[e], s.co[4 * t + e] += fl[e] * x[e];
  }
}

// Adds to what s holds; the diagonal's part of P (E = 1) is the caller's.
__device__ __forceinline__ void pair_sums(PairSums& s, const float (&g)[16], const bf16x4 (&k4)[4], const bf16x4 (&q4)[4], const float* __restrict__ beta,
                                          const T* __restrict__ P, const T* __restrict__ A, const float* __restrict__ G, int c, int lane) {
  float dec[16];  // single-step decays exp(G_tok - G_{tok-1}) inside each group of four (the first entry of a group is unused)
#pragma unroll
  for (int x = 0; x < 16; ++x) dec[x] = (x & 3) ? __builtin_amdgcn_exp2f(fminf(g[x] - g[x - 1], 0.f)) : 1.f;
  // one part at a time: interleaving them multiplies the live factors
  s.settle();
  sums_cross<32>(s, g, dec, k4, q4, beta, P, A, G, c, lane);
  s.settle();
  sums_cross<16>(s, g, dec, k4, q4, beta, P, A, G, c, lane);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    s.settle();
    sums_diag(s, g, dec, k4, q4, beta, P, A, G, c, t, lane);
  }
  s.settle();
}

template <int DK> struct KdaL {
  static constexpr int NT = DK / 64, THREADS = 256 * NT, NW = 4 * NT, SV = 32;  // teams of four waves
  static constexpr int NBUF = NT == 2 ? 3 : 2;  // one workgroup per CU, or two
  typedef SwzTile<64, SV> TokT;         // dO, D, dD, V slabs, and dR
  typedef SwzTile<SV, DK, false> StT;   // S^T, dS'^T slabs, transposing reads only
  static constexpr int oD = TokT::BYTES, odD = 2 * oD, oV = 3 * oD, oS = 4 * oD, odS = oS + StT::BYTES, slab_bytes = odS + StT::BYTES;
  static constexpr int tile = 64 * LDX * 2, ftile = 64 * LDF * 4;
  static constexpr int odR = NBUF * slab_bytes, oTm = odR + TokT::BYTES;
  static constexpr size_t loop_bytes = oTm + tile;
  // epilogue: dPm, dXa | per team G (fp32), K, Q, dq and dk on their way out (then dg, fp32)
  static constexpr int team_bytes = ftile + 4 * tile;
  static constexpr size_t epi_bytes = 2 * tile + NT * team_bytes;
  static_assert(ftile <= 2 * tile, "dg leaves over dq and dk");
  static constexpr int nfloat = 64 * (6 + NW);
  static constexpr size_t bytes = sizeof(float) * nfloat + (epi_bytes > loop_bytes ? epi_bytes : loop_bytes);
  static_assert(bytes <= (NT == 2 ? 160 : 80) * 1024, "LDS");
};

template <int DK, bool GRAW>
__global__ __launch_bounds__(KdaL<DK>::THREADS, 2) void kda_bwd_chunk_kernel(KdaBwdParams p) {
  typedef KdaL<DK> L;
  constexpr int NT = L::NT, THREADS = L::THREADS, NW = L::NW, NBUF = L::NBUF, SV = L::SV;
  typedef typename L::TokT TokT;
  typedef typename L::StT StT;
  extern __shared__ __align__(16) char smem[];
  float* sBeta = reinterpret_cast<float*>(smem);
  float* sDiag = sBeta + 64;      // scale dPm_tt
  float* sRdv = sDiag + 64;       // [2] <dR_t, v_t> over the even and the odd slabs
  float* sNq = sRdv + 128;        // normalisation factors of the q and k rows (1 when the inputs come normalised)
  float* sNk = sNq + 64;
  float* sM = sNk + 64;           // [wave] the wave's share of m_t
  char* region = smem + sizeof(float) * L::nfloat;
  T* sdR = reinterpret_cast<T*>(region + L::odR);
  T* sTm = reinterpret_cast<T*>(region + L::oTm);  // Tm^T

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, kq = lane >> 4;
  const int team = wave >> 2, w4 = wave & 3;
  const int N = p.geom.N;
  const int64_t slot = blockIdx.x;
  const int row = (int)(slot / N), n = (int)(slot % N);
  int tok0, len;
  chunk_span(p.geom, n, tok0, len);
  // fused gate activation: this chunk's row of the parameter-gradient partial sums, columns of this head
  auto gate_part = [&](int which) {
    const int64_t gD = (int64_t)p.geom.H * DK;
    return p.gpart + (which * (p.gprows + LNX_SUM_SLICES) + (int64_t)(row / p.geom.H) * N + n) * gD + (row % p.geom.H) * DK;
  };
  if (len <= 0) {  // an unused slot of a packed batch: its partial sums are zero
    if constexpr (GRAW)
      for (int c = tid; c < DK; c += THREADS) gate_part(0)[c] = gate_part(1)[c] = 0.f;
    return;
  }
  const int64_t tbase = tok_index(p.geom, row, tok0);
  const int64_t ts = p.geom.ts, tsk = ts * DK, tsv = ts * p.dv;
  // the head's gate scale, fetched here: a load behind the epilogue's stores would wait for every one of them
  float gna = 0.f;
  if constexpr (GRAW) gna = -__expf(p.gA[row % p.geom.H]);

  if (tid < 64) {
    sBeta[tid] = (tid < len) ? p.beta[tbase + tid * ts] : 0.f;
    sRdv[tid] = sRdv[64 + tid] = 0.f;
    sNq[tid] = p.l2norm ? at<const float>(p.ws, p.off.Nq)[slot * 64 + tid] : 1.f;
    sNk[tid] = p.l2norm ? at<const float>(p.ws, p.off.Nk)[slot * 64 + tid] : 1.f;
  }
  if (NT == 1 || team == 0) stage_tile<T, 64, 64>(sTm, LDX, at<const T>(p.ws, p.off.TmT) + slot * 64 * 64, 64, 64, tid);
  __builtin_amdgcn_s_waitcnt(0);  // the small loads are behind us: this wave's vmcnt now counts slab loads and the stores of dv

  // ---- the slab loads: one-KB instructions, PER_WAVE of them per wave and slab.  Token rows past the chunk's end fetch the chunk's last
  // row instead of zeros: they only reach rows that are not stored and products with rows of q and k that are zero.
  const unsigned slab0 = lds_byte_addr(region);
  const T* gdO = p.d_o + tbase * p.dv;
  const T* gV = p.v + tbase * p.dv;
  const T* gD = at<const T>(p.ws, p.off.D) + slot * 64 * p.dv;
  const T* gdD = at<const T>(p.ws, p.off.dD) + slot * 64 * p.dv;
  const T* gS = at<const T>(p.ws, p.off.SnT) + slot * p.dv * DK;
  const T* gdS = at<const T>(p.ws, p.off.dSn) + slot * p.dv * DK;
  auto issue = [&](int s) {
    const int v0 = SV * s;
    const unsigned dst = slab0 + (s % NBUF) * L::slab_bytes;
    int r, c;
    StT::src(wave, lane, r, c);
    dma16(gS + (int64_t)(v0 + r) * DK + c, dst + L::oS + 1024 * wave);
    dma16(gdS + (int64_t)(v0 + r) * DK + c, dst + L::odS + 1024 * wave);
    TokT::src(w4, lane, r, c);
    const int64_t rc = (int64_t)min(r, len - 1) * tsv + v0 + c, rw = (int64_t)r * p.dv + v0 + c;
    if (NT == 1 || team == 0) {
      dma16(gdO + rc, dst + 1024 * w4);
      dma16(gD + rw, dst + L::oD + 1024 * w4);
    }
    if (NT == 1 || team == 1) {
      dma16(gdD + rw, dst + L::odD + 1024 * w4);
      dma16(gV + rc, dst + L::oV + 1024 * w4);
    }
  };
  constexpr int PER_WAVE = NT == 1 ? 6 : 4;
  static_assert(StT::NINSTR == NW && TokT::NINSTR == 4, "the same count for every wave");
  const int nslab = p.dv / SV;  // two or more
#pragma unroll
  for (int s = 0; s < NBUF; ++s)
    if (s < nslab) issue(s);

  const int ch = 64 * team + 16 * w4;  // the wave's first channel
  floatx4 aQ[4], aK1[4], aK2[4], aP[4], aA[4];  // dO S^T, dR S^T, D dS'^T: [token tile]; row tile w4 of dO D^T (team 0) and dR D^T (last team)
#pragma unroll
  for (int i = 0; i < 4; ++i) aQ[i] = aK1[i] = aK2[i] = aP[i] = aA[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  const bool has_p = team == 0, has_a = team == NT - 1;
  float ss = 0.f, rdv = 0.f;
  TileRegs<T, 64, 64> rK, rQ;  // the epilogue's tiles of this team's channels, requested during the last slab
  TileRegs<float, 64, 64> rG;
  const int tt = tid & 255;
#pragma unroll 1
  for (int s = 0; s < nslab; ++s) {
    // this slab has landed: all but this wave's loads of the slabs behind it, then every wave's
    if (NBUF == 3 && s == 0 && nslab > 2) dma_wait<2 * PER_WAVE>();
    else if (s + 1 < nslab) dma_wait<PER_WAVE>();
    else dma_wait<0>();
    lds_barrier();  // and every wave is done with the slab before, whose buffer takes the next one but one
    if (NBUF == 3 && s > 0 && s + 2 < nslab) issue(s + 2);
    if (s + 1 == nslab) {
      rK.load(p.k + tbase * DK + 64 * team, tsk, len, tt);
      rQ.load(p.q + tbase * DK + 64 * team, tsk, len, tt);
      rG.load(at<const float>(p.ws, p.off.G) + slot * 64 * DK + 64 * team, DK, 64, tt);
    }
    const char* slab = region + (s % NBUF) * L::slab_bytes;
    const T* tdO = reinterpret_cast<const T*>(slab);
    const T* tD = reinterpret_cast<const T*>(slab + L::oD);
    const T* tdD = reinterpret_cast<const T*>(slab + L::odD);
    const T* tV = reinterpret_cast<const T*>(slab + L::oV);
    const T* tS = reinterpret_cast<const T*>(slab + L::oS);
    const T* tdS = reinterpret_cast<const T*>(slab + L::odS);
    // ---- dR = Tm^T dD, transposed products: lane = token 16 w4 + l16, four value columns; Tm^T is upper-triangular ----
#pragma unroll
    for (int u = 0; u < 2 / NT; ++u) {
      const int vt = NT == 1 ? u : team;
      floatx4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if (k == 0 && w4 >= 2) continue;
        const Frag fa = S16::join(__builtin_bit_cast(bf16x4, TokT::tr4(tdD, 32 * k + 8 * kq, 16 * vt, lane)),
                                  __builtin_bit_cast(bf16x4, TokT::tr4(tdD, 32 * k + 8 * kq + 4, 16 * vt, lane)));
        S16::mma(x, fa, *reinterpret_cast<const Frag*>(sTm + (16 * w4 + l16) * LDX + 32 * k + 8 * kq));
      }
      store4(sdR + TokT::at(16 * w4 + l16, 16 * vt + 4 * kq), x);
    }
    // ---- what does not need dR ----
    Frag fD[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) fD[i] = TokT::load(tD, 16 * i + l16, 8 * kq);
    const Frag fS = S16::join(__builtin_bit_cast(bf16x4, StT::tr4(tS, 8 * kq, ch, lane)), __builtin_bit_cast(bf16x4, StT::tr4(tS, 8 * kq + 4, ch, lane)));
    const Frag fdS = S16::join(__builtin_bit_cast(bf16x4, StT::tr4(tdS, 8 * kq, ch, lane)), __builtin_bit_cast(bf16x4, StT::tr4(tdS, 8 * kq + 4, ch, lane)));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Frag f = TokT::load(tdO, 16 * i + l16, 8 * kq);
      S16::mma(aQ[i], f, fS);
      S16::mma(aK2[i], fD[i], fdS);
      if (has_p && i == w4) {
#pragma unroll
        for (int j = 0; j <= i; ++j) S16::mma(aP[j], f, fD[j]);
      }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) ss += (float)fS[e] * (float)fdS[e];  // <dS', S> of channel ch + l16
    lds_barrier();  // dR is there
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Frag f = TokT::load(sdR, 16 * i + l16, 8 * kq);
      S16::mma(aK1[i], f, fS);
      if (has_a && i == w4) {
#pragma unroll
        for (int j = 0; j <= i; ++j) S16::mma(aA[j], f, fD[j]);
      }
    }
    if (NT == 1 || team == (s & 1)) {  // <dR_t, v_t> and dv = beta dR: thread = (token tt / 4, eight value columns); the teams take turns
      const int t = tt >> 2, c0 = 8 * (tt & 3);
      Frag x = TokT::load(sdR, t, c0);
      const Frag vv = TokT::load(tV, t, c0);
      const float bt = sBeta[t];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        rdv += (float)x[e] * (float)vv[e];
        x[e] = (bf16_t)((float)x[e] * bt);
      }
      if (t < len) *reinterpret_cast<Frag*>(p.dv_out + tbase * p.dv + (int64_t)t * tsv + SV * s + c0) = x;
    }
    if (NBUF == 2 && s + 2 < nslab) {  // this buffer takes the slab after the next, once every wave has read it
      lds_barrier();
      issue(s + 2);
    }
  }
  rdv = quad_sum(rdv);
  if ((lane & 3) == 0) sRdv[64 * team + (tt >> 2)] = rdv;
  lds_barrier();  // slab tiles are dead from here on

  // ---- epilogue ----
  T* sP = reinterpret_cast<T*>(region);
  T* sA = sP + 64 * LDX;
  char* mine = region + 2 * L::tile + team * L::team_bytes;
  float* sG = reinterpret_cast<float*>(mine);
  T* sK = reinterpret_cast<T*>(mine + L::ftile);
  T* sQ = sK + 64 * LDX;
  T* sdQ = sQ + 64 * LDX;
  T* sdK = sdQ + 64 * LDX;
  float* sOut = reinterpret_cast<float*>(sdQ);  // dg, once dq and dk have left
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j <= w4) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * w4 + 4 * kq + e, col = 16 * j + l16;
        if (has_p) {
          const float x = p.scale * aP[j][e];
          sP[i * LDX + col] = (bf16_t)(i > col ? x : 0.f);
          if (i == col) sDiag[i] = x;
        }
        if (has_a) sA[i * LDX + col] = (bf16_t)(i > col ? -aA[j][e] : 0.f);
      }
    }
  {
    typedef TileRegs<T, 64, 64> RowTile;
#pragma unroll
    for (int it = 0; it < RowTile::IT; ++it) {
      const int idx = tt + 256 * it, r = idx / RowTile::VPR, c = (idx - r * RowTile::VPR) * RowTile::N;
      Frag x = rK.x[it], y = rQ.x[it];
      if (p.l2norm) {
        const float fk = sNk[r], fq = sNq[r];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = (bf16_t)((float)x[e] * fk), y[e] = (bf16_t)((float)y[e] * fq);
      }
      *reinterpret_cast<Frag*>(sK + r * LDX + c) = x;
      *reinterpret_cast<Frag*>(sQ + r * LDX + c) = y;
    }
    rG.store(sG, LDF, tt);
  }
  lds_barrier();
  const int c = 16 * w4 + l16;  // this lane's channel of the team's 64
  float dG[16];
  {
    float g[16], tot = 0.f;
    bf16x4 k4[4], q4[4];
    PairSums s;
    const float gC = LOG2E * sG[63 * LDF + c];
    // what the loop left, and the diagonal of dPm; rp becomes dq, ra row, co dk without beta row
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      k4[t] = column4(sK, t, 16 * w4, lane), q4[t] = column4(sQ, t, 16 * w4, lane);
      const floatx4 d4 = load4(sDiag + 16 * t + 4 * kq);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int x = 4 * t + e;
        g[x] = LOG2E * sG[(16 * t + 4 * kq + e) * LDF + c];
        const float eg = __builtin_amdgcn_exp2f(g[x]), k2 = __builtin_amdgcn_exp2f(fminf(gC - g[x], 0.f)) * aK2[t][e], kv = (float)k4[t][e];
        s.rp[x] = p.scale * eg * aQ[t][e] + d4[e] * kv;
        s.ra[x] = -eg * aK1[t][e];
        s.co[x] = k2 + d4[e] * (float)q4[t][e];
        tot += kv * k2;
      }
    }
    pair_sums(s, g, k4, q4, sBeta, sP, sA, sG, c, lane);
    float mv[16];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const floatx4 bt = load4(sBeta + 16 * t + 4 * kq);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int x = 4 * t + e, tok = 16 * t + 4 * kq + e;
        const float kv = (float)k4[t][e], dk = bt[e] * s.ra[x] + s.co[x];
        mv[x] = kv * s.ra[x];
        dG[x] = (float)q4[t][e] * s.rp[x] - kv * dk + 2.f * bt[e] * mv[x];
        sdQ[tok * LDX + c] = (bf16_t)s.rp[x];
        sdK[tok * LDX + c] = (bf16_t)dk;
      }
    }
    tot = xor32_sum(xor16_sum(tot + __builtin_amdgcn_exp2f(gC) * ss));  // over the tokens (ss: over its value columns) of this channel
    if (kq == 3) dG[15] += tot;
    // m_t over the wave's sixteen channels: sixteen values over sixteen lanes, halving the values with each exchange
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1) {
      const bool hi = (l16 & m) != 0;
#pragma unroll
      for (int x = 0; x < m; ++x) {
        const float send = hi ? mv[x] : mv[x + m], keep = hi ? mv[x + m] : mv[x];
        mv[x] = keep + __shfl_xor(send, m, LNX_WAVE);
      }
    }
    sM[64 * wave + 16 * (l16 >> 2) + 4 * kq + (l16 & 3)] = mv[0];  // lane l16 ends with value l16 = 4 t + e
  }
  // ---- dg: reverse cumulative sum over the chunk's tokens of this channel ----
  {
    float after = 0.f;  // what later blocks of sixteen tokens add
#pragma unroll
    for (int t = 3; t >= 0; --t) {
#pragma unroll
      for (int e = 2; e >= 0; --e) dG[4 * t + e] += dG[4 * t + e + 1];
      const float own = dG[4 * t];
      const float y1 = __shfl_down(own, 16, LNX_WAVE), y2 = __shfl_down(own, 32, LNX_WAVE), y3 = __shfl_down(own, 48, LNX_WAVE);
      float add = after;
      if (kq < 3) add += y1;
      if (kq < 2) add += y2;
      if (kq < 1) add += y3;
#pragma unroll
      for (int e = 0; e < 4; ++e) dG[4 * t + e] += add;
      after = __shfl(dG[4 * t], l16, LNX_WAVE);  // the block's first token holds the sum of everything from it on
    }
  }
  lds_barrier();  // dq, dk and the shares of m are in LDS
  // ---- dq, dk out: thread = (token, the 8-channel groups tq, tq + TPT, ...); the row dots carry them through the normalisation,
  //      d/dx of x / (|x| + eps) applied to dy:  dy / (|x| + eps) - y <y, dy> / |x| ----
  {
    constexpr int TPT = THREADS / 64;
    const int tr = tid / TPT, tq = tid % TPT;
    auto emit = [&](int from, int own, const float* fac, T* out) {  // tiles `from` (gradient) and `own` (the row) of a team's 64-channel block
      auto rows = [&](int tile, int u) {
        return *reinterpret_cast<const Frag*>(region + 2 * L::tile + (u >> 3) * L::team_bytes + L::ftile + tile * L::tile + (tr * LDX + 8 * (u & 7)) * 2);
      };
      const float f = fac[tr];
      float cf = 0.f;
      if (p.l2norm) {
        float dot = 0.f;
#pragma unroll
        for (int u = 0; u < DK / 8; u += TPT) {
          const Frag a = rows(from, tq + u), b = rows(own, tq + u);
#pragma unroll
          for (int e = 0; e < 8; ++e) dot += (float)a[e] * (float)b[e];
        }
        dot = quad_sum(dot);
        if (TPT == 8) dot += __shfl_xor(dot, 4, LNX_WAVE);
        const float nrm = 1.f / f - LNX_L2_EPS;
        cf = nrm > 0.f ? dot / nrm : 0.f;
      }
      if (tr < len) {
#pragma unroll
        for (int u = 0; u < DK / 8; u += TPT) {
          Frag a = rows(from, tq + u);
          if (p.l2norm) {
            const Frag b = rows(own, tq + u);
#pragma unroll
            for (int e = 0; e < 8; ++e) a[e] = (bf16_t)(f * (float)a[e] - cf * (float)b[e]);
          }
          *reinterpret_cast<Frag*>(out + tbase * DK + (int64_t)tr * tsk + 8 * (tq + u)) = a;
        }
      }
    };
    emit(2, 1, sNq, p.dq);
    emit(3, 0, sNk, p.dk);
  }
  if (tid < 64 && tid < len) {
    float m = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) m += sM[64 * w + tid];
    p.dbeta[tbase + tid * ts] = sRdv[tid] + (NT == 2 ? sRdv[64 + tid] : 0.f) + m;
  }
  lds_barrier();  // dq and dk have left
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) sOut[(16 * t + 4 * kq + e) * LDF + c] = dG[4 * t + e];
  lds_barrier();
  // dg leaves by rows: thread = (row tt / 16 + 16 it, four channels), 16-byte accesses.  With the gate activated inside the op,
  // g = -e^{A_log} softplus(x), x = raw + bias (kda.py:153-165), the gradient goes on to the raw projection as bwd_wy2 (chunk_bwd.hip)
  // explains: the activated gate is the difference of two rows of the cumulative gate, its derivative 1 - e^{-softplus}; x itself
  // is read again only where the threshold is so low that it does not follow from softplus(x) (gband).
  if constexpr (!GRAW) {
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int idx = tt + 256 * it, r = idx >> 4, c4 = (idx & 15) * 4;
      if (r < len) store4(p.dg + (tbase + (int64_t)r * ts) * DK + 64 * team + c4, load4(sOut + r * LDF + c4));
    }
  } else {
    const int c4 = (tt & 15) * 4, r0 = tt >> 4;
    const float na = gna, inv_na = 1.f / na;
    floatx4 sb = {0.f, 0.f, 0.f, 0.f}, sa = sb;
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int r = r0 + 16 * it;
      const floatx4 dgv = load4(sOut + r * LDF + c4);
      floatx4 gv = load4(sG + r * LDF + c4);
      if (r > 0) gv = gv - load4(sG + (r - 1) * LDF + c4);
      floatx4 xv = {0.f, 0.f, 0.f, 0.f};  // x = raw + bias, fetched where it is used: the unusual case may wait
      if (p.gband) {
        if (p.gbias) xv = load4(p.gbias + (row % p.geom.H) * DK + 64 * team + c4);
        const bf16x4 rq = *reinterpret_cast<const bf16x4*>(p.graw + (tbase + (int64_t)min(r, len - 1) * ts) * DK + 64 * team + c4);
#pragma unroll
        for (int e = 0; e < 4; ++e) xv[e] += (float)rq[e];
      }
      floatx4 dr;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float sp = gv[e] * inv_na;
        const bool lin = p.gband ? xv[e] > p.gthr : sp > p.gthr;
        const float ds = lin ? 1.f : 1.f - __expf(-sp);
        dr[e] = r < len ? dgv[e] * na * ds : 0.f;
        sb[e] += dr[e];
        sa[e] += r < len ? dgv[e] * gv[e] : 0.f;
      }
      if (r < len) store4(p.dgraw + (tbase + (int64_t)r * ts) * DK + 64 * team + c4, dr);
    }
    float* sPart = reinterpret_cast<float*>(sK);  // [2][16 row groups][64]: the K and Q tiles are dead
    store4(sPart + r0 * 64 + c4, sb);
    store4(sPart + 1024 + r0 * 64 + c4, sa);
    lds_barrier();
    if (tt < 128) {  // the sixteen row groups in a fixed order
      const float* src = sPart + (tt >> 6) * 1024 + (tt & 63);
      float t = 0.f;
#pragma unroll
      for (int q = 0; q < 16; ++q) t += src[64 * q];
      gate_part(tt >> 6)[64 * team + (tt & 63)] = t;
    }
  }
}

template <int DK>
int launch(const KdaBwdParams& p, hipStream_t st) {
  auto k = p.graw ? kda_bwd_chunk_kernel<DK, true> : kda_bwd_chunk_kernel<DK, false>;
  const size_t b = KdaL<DK>::bytes;
  if (const int rc = lnx_lds_limit((const void*)k, b); rc != LNX_OK) return rc;
  lnx_profile_mark("bwd_chunk", st);
  hipLaunchKernelGGL(k, dim3((unsigned)((int64_t)p.geom.rows * p.geom.N)), dim3(KdaL<DK>::THREADS), b, st, p);
  lnx_profile_mark(nullptr, st);
  return LNX_OK;
}

}  // namespace

int lnx_kda_bwd_chunk(const KdaBwdParams& p, int dk, hipStream_t st) { return dk == 128 ? launch<128>(p, st) : launch<64>(p, st); }
