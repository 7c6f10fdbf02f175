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
// One workgroup of four waves per chunk, two of them per CU: what one loads, the other covers with the pair sums, which take about as
// long on the VALU as the loads on the memory path.  A loop over 32-column slabs of the value dimension (LDS-direct loads, two slabs in
// flight) forms dR and accumulates what contracts over value columns on 16x16x32 products: wave w owns the channels 64 s + 16 w .. of every
// set s of 64 and all tokens, so that an accumulator element is at the place where pair_levels wants its channel and token:
// lane (c = lane % 16, kq = lane / 16) holds the tokens 16 t + 4 kq + e of channel c, and everything between the loop and the
// tiles on their way out happens in registers.  The four pair sums share their factors (pair_sums).
// Measured at B4 H16 T8192 d128 (8192 chunks): 461 - 472 us by box for 280 KB a chunk, 5 TB/s, and two thirds of the time on vector instructions (the
// normalisation adds about 20 us to it and kda_prepare together, the gate's activation 65); bwd_dqk and bwd_wy2, which passed dW, a partial dk
// and an fp32 partial gradient of the gate through memory, 402 + 497 us behind and before 217 us of normalisation outside.  The cumulative gate
// is summed up again from the gate: 461 -> 470 us here, 25 less where the prepare kernel wrote it.  With eight waves and one workgroup per CU
// 650 us: of 20.6 us a chunk 8.5 were pair sums with nothing in flight.

#include "chunk_common.h"
#include "reduce_rows.h"

namespace {

using T = bf16_t;
typedef Mma16 S16;
typedef S16::Frag Frag;
template <typename X> __device__ __forceinline__ X* at(char* ws, uint64_t off) { return reinterpret_cast<X*>(ws + off); }
constexpr int LDX = LNX_C + 8;  // dPm, dXa: bf16 [64][64] tiles

// A operands of the 16x16x16 products from such a tile: block (ti, t), lane = (row l16, k-slots 4 kq + e); transposed: (column l16, rows)
__device__ __forceinline__ bf16x4 block_rows(const T* X, int ti, int t, int lane) {
  return *reinterpret_cast<const bf16x4*>(X + (16 * ti + (lane & 15)) * LDX + 16 * t + 4 * (lane >> 4));
}
__device__ __forceinline__ bf16x4 block_cols(const T* X, int ti, int t, int lane) { return S16::rows4(X, LDX, 16 * ti + 4 * (lane >> 4), 16 * t, lane); }

// pair_levels (chunk_common.h) for two matrices at once.  Per level every token has one factor, and P and A share it and the column
// tokens' operand F k:
//   rp[i] += sum_{j < i} P_ij E_ij k_j     ra[i] += sum_{j < i} A_ij E_ij k_j     co[j] += sum_{i > j} E_ij (P_ij q_i + A_ij (beta k)_i)
// Lane, index 4 t + e and levels as there; g = G, whose reference tokens are values of the other lane groups of the channel.
// P and A: bf16 [64][LDX].
// the value of lane group 0, and of group 2, in every group; of the odd group of a pair, in both
__device__ __forceinline__ float of_group0(float x) {
  const unsigned u = __float_as_uint(x), v = __builtin_amdgcn_permlane32_swap(u, u, false, false)[0];
  return __uint_as_float(__builtin_amdgcn_permlane16_swap(v, v, false, false)[0]);
}
__device__ __forceinline__ float of_group2(float x) {
  const unsigned u = __float_as_uint(x), v = __builtin_amdgcn_permlane32_swap(u, u, false, false)[1];
  return __uint_as_float(__builtin_amdgcn_permlane16_swap(v, v, false, false)[0]);
}
__device__ __forceinline__ float of_odd_group(float x) {
  const unsigned u = __float_as_uint(x);
  return __uint_as_float(__builtin_amdgcn_permlane16_swap(u, u, false, false)[1]);
}
// Everything these depend on is computed here: arithmetic may pass a scheduling barrier, loads may not, and what had been loaded for sums
// that were put off went to scratch memory.
__device__ __forceinline__ void settle16(float (&x)[16]) {
#pragma unroll
  for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(x[i]));
}
struct PairSums {
  float rp[16], ra[16], co[16];
  __device__ __forceinline__ void settle() { settle16(rp), settle16(ra), settle16(co); }
};
template <int H>
__device__ __forceinline__ void sums_cross(PairSums& s, const float (&g)[16], const float (&dec)[16], const bf16x4 (&k4)[4], const bf16x4 (&q4)[4],
                                           const float* __restrict__ beta, const T* __restrict__ P, const T* __restrict__ A, int lane_) {
  const int lane = fresh(lane_);  // the matrices' blocks are read where they are used
  const float m0 = of_group0(g[H / 4]), m1 = H == 32 ? m0 : of_group0(g[12]);  // G of token H, and of token 48
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
                                          const float* __restrict__ beta, const T* __restrict__ P, const T* __restrict__ A, int t, int lane_) {
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
      const float ref = H == 8 ? of_group2(g[4 * t]) : of_odd_group(g[4 * t]);  // G of token 16 t + 8, or of the half block's fifth
      const float f = __builtin_amdgcn_exp2f(fminf(up ? g[4 * t] - ref : ref - g[4 * t + 3], 0.f));
      fu[0] = up ? f : 0.f, fu[1] = fu[0] * d1, fu[2] = fu[1] * d2, fu[3] = fu[2] * d3;
      fl[3] = up ? 0.f : f, fl[2] = fl[3] * d3, fl[1] = fl[2] * d2, fl[0] = fl[1] * d1;
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
                                          const T* __restrict__ P, const T* __restrict__ A, int lane) {
  float dec[16];  // single-step decays exp(G_tok - G_{tok-1}) inside each group of four (the first entry of a group is unused)
#pragma unroll
  for (int x = 0; x < 16; ++x) dec[x] = (x & 3) ? __builtin_amdgcn_exp2f(fminf(g[x] - g[x - 1], 0.f)) : 1.f;
  // one part at a time: interleaving them multiplies the live factors
  s.settle();
  sums_cross<32>(s, g, dec, k4, q4, beta, P, A, lane);
  s.settle();
  sums_cross<16>(s, g, dec, k4, q4, beta, P, A, lane);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    s.settle();
    sums_diag(s, g, dec, k4, q4, beta, P, A, t, lane);
  }
  s.settle();
}

// One step of sixteen sums over sixteen lanes: of 2 M values a lane keeps M, adding what its partner sends
template <int M> __device__ __forceinline__ void exchange(float (&v)[16], int l16) {
  const bool hi = (l16 & M) != 0;
#pragma unroll
  for (int x = 0; x < M; ++x) {
    const float lo = v[x], up = v[x + M];
    v[x] = (hi ? up : lo) + __shfl_xor(hi ? lo : up, M, LNX_WAVE);
  }
}

template <int DK> struct KdaL {
  static constexpr int NS = DK / 64, SV = 32, NBUF = 2;  // sets of 64 channels
  typedef SwzTile<64, SV> TokT;         // dO, D, dD, V slabs, and dR
  typedef SwzTile<SV, DK, false> StT;   // S^T, dS'^T slabs, transposing reads only
  typedef SwzTile<64, 64> TmT;          // Tm^T, read by rows
  typedef SwzTile<64, DK> RowT;         // K and Q rows; dq and dk on their way out
  static constexpr int oD = TokT::BYTES, odD = 2 * oD, oV = 3 * oD, oS = 4 * oD, odS = oS + StT::BYTES, slab_bytes = odS + StT::BYTES;
  static constexpr int odR = NBUF * slab_bytes, oTm = odR + TokT::BYTES, loop_bytes = oTm + TmT::BYTES;
  // epilogue: K | Q (then dq | dk, then the gate's gradient) | dPm | dXa | diagonal of dPm, <dR, v>, factors of the normalisation [2], shares of
  // m, <q, dq>, <k, dk> [3][set, wave]
  static constexpr int tile = 64 * LDX * 2, oP = 2 * RowT::BYTES, oF = oP + 2 * tile, epi_bytes = oF + 4 * 64 * (4 + 12 * NS);
  // the gate's gradient, fp32 [64][LDF] per set: the last set's over K and Q, the one before it waits behind everything else
  static constexpr int LDF = 64 + 4, oG0 = epi_bytes, all_bytes = epi_bytes + (NS - 1) * 64 * LDF * 4;
  // a gate activated inside the op: its partial sums [set][which][wave][64], behind the gradient, which other waves still read when they are
  // stored -- at dk = 64 its last rows lie over dPm
  static constexpr int grad = 64 * LDF * 4, oPart = oP > grad ? oP : grad;
  static_assert(NS <= 2 && oPart % 16 == 0 && grad <= oPart && oPart + NS * 2 * 4 * 64 * 4 <= oF, "gradient and partial sums leave over the tiles, side by side");
  static constexpr size_t bytes = sizeof(float) * 192 + (all_bytes > loop_bytes ? all_bytes : loop_bytes);
  static_assert(bytes <= 80 * 1024, "two workgroups per CU");
};

template <int DK, bool GRAW>
__global__ __launch_bounds__(256, 2) void kda_bwd_chunk_kernel(KdaBwdParams p) {
  typedef KdaL<DK> L;
  constexpr int NS = L::NS, SV = L::SV;
  typedef typename L::TokT TokT;
  typedef typename L::StT StT;
  typedef typename L::TmT TmT;
  typedef typename L::RowT RowT;
  extern __shared__ __align__(16) char smem[];
  float* sBeta = reinterpret_cast<float*>(smem);
  float* sNq = sBeta + 64;        // normalisation factors of the q and k rows
  float* sNk = sNq + 64;
  char* region = smem + sizeof(float) * 192;
  T* sdR = reinterpret_cast<T*>(region + L::odR);
  T* sTm = reinterpret_cast<T*>(region + L::oTm);  // Tm^T

  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, kq = lane >> 4;
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
      for (int c = tid; c < DK; c += 256) gate_part(0)[c] = gate_part(1)[c] = 0.f;
    return;
  }
  const int64_t tbase = tok_index(p.geom, row, tok0);
  const int64_t ts = p.geom.ts, tsk = ts * DK, tsv = ts * p.dv;
  // the head's gate scale, fetched here: a load behind the epilogue's stores would wait for every one of them
  float gna = 0.f;
  if constexpr (GRAW) gna = -__expf(p.gA[row % p.geom.H]);

  // ---- the slab loads: one-KB instructions, PER_WAVE of them per wave and slab.  Token rows past the chunk's end fetch the chunk's last
  // row instead of zeros: they only reach rows that are not stored and products with rows of q and k that are zero.  The small loads go the
  // same way ahead of them.
  const unsigned slab0 = lds_byte_addr(region);
  if (wave == 0) dma4(p.beta + tbase + (int64_t)min(lane, len - 1) * ts, lds_byte_addr(sBeta));
  if (p.l2norm) {
    if (wave == 1) dma4(at<const float>(p.ws, p.off.Nq) + slot * 64 + lane, lds_byte_addr(sNq));
    if (wave == 2) dma4(at<const float>(p.ws, p.off.Nk) + slot * 64 + lane, lds_byte_addr(sNk));
  }
#pragma unroll
  for (int u = 0; u < TmT::NINSTR / 4; ++u) {
    int r, c;
    TmT::src(wave + 4 * u, lane, r, c);
    dma16(at<const T>(p.ws, p.off.TmT) + slot * 64 * 64 + r * 64 + c, slab0 + L::oTm + 1024 * (wave + 4 * u));
  }
  const T* gdO = p.d_o + tbase * p.dv;
  const T* gV = p.v + tbase * p.dv;
  const T* gD = at<const T>(p.ws, p.off.D) + slot * 64 * p.dv;
  const T* gdD = at<const T>(p.ws, p.off.dD) + slot * 64 * p.dv;
  const T* gS = at<const T>(p.ws, p.off.SnT) + slot * p.dv * DK;
  const T* gdS = at<const T>(p.ws, p.off.dSn) + slot * p.dv * DK;
  auto issue = [&](int s) {
    const int v0 = SV * s;
    const unsigned dst = slab0 + (s & 1) * L::slab_bytes;
    int r, c;
#pragma unroll
    for (int u = 0; u < StT::NINSTR / 4; ++u) {
      StT::src(wave + 4 * u, lane, r, c);
      dma16(gS + (int64_t)(v0 + r) * DK + c, dst + L::oS + 1024 * (wave + 4 * u));
      dma16(gdS + (int64_t)(v0 + r) * DK + c, dst + L::odS + 1024 * (wave + 4 * u));
    }
    TokT::src(wave, lane, r, c);
    const int64_t rc = (int64_t)min(r, len - 1) * tsv + v0 + c, rw = (int64_t)r * p.dv + v0 + c;
    dma16(gdO + rc, dst + 1024 * wave);
    dma16(gD + rw, dst + L::oD + 1024 * wave);
    dma16(gdD + rw, dst + L::odD + 1024 * wave);
    dma16(gV + rc, dst + L::oV + 1024 * wave);
  };
  constexpr int PER_WAVE = StT::NINSTR / 2 + 4;
  static_assert(StT::NINSTR % 4 == 0 && TokT::NINSTR == 4 && TmT::NINSTR % 4 == 0, "the same count for every wave");
  const int nslab = p.dv / SV;  // two or more
  issue(0);
  issue(1);

  floatx4 aQ[NS][4], aK1[NS][4], aK2[NS][4], aP[4], aA[4];  // dO S^T, dR S^T, D dS'^T: [set][token tile]; row tile `wave` of dO D^T and dR D^T
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    aP[i] = aA[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NS; ++u) aQ[u][i] = aK1[u][i] = aK2[u][i] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  float ss[NS] = {}, rdv = 0.f;
#pragma unroll 1
  for (int s = 0; s < nslab; ++s) {
    // this slab has landed: all but this wave's loads of the next one, then every wave's
    if (s + 1 < nslab) dma_wait<PER_WAVE>();
    else dma_wait<0>();
    lds_barrier();
    const char* slab = region + (s & 1) * L::slab_bytes;
    const T* tdO = reinterpret_cast<const T*>(slab);
    const T* tD = reinterpret_cast<const T*>(slab + L::oD);
    const T* tdD = reinterpret_cast<const T*>(slab + L::odD);
    const T* tV = reinterpret_cast<const T*>(slab + L::oV);
    const T* tS = reinterpret_cast<const T*>(slab + L::oS);
    const T* tdS = reinterpret_cast<const T*>(slab + L::odS);
    // ---- dR = Tm^T dD, transposed products: lane = token 16 wave + l16, four value columns; Tm^T is upper-triangular ----
#pragma unroll
    for (int vt = 0; vt < 2; ++vt) {
      floatx4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if (k == 0 && wave >= 2) continue;
        const Frag fa = S16::join(__builtin_bit_cast(bf16x4, TokT::tr4(tdD, 32 * k + 8 * kq, 16 * vt, lane)),
                                  __builtin_bit_cast(bf16x4, TokT::tr4(tdD, 32 * k + 8 * kq + 4, 16 * vt, lane)));
        S16::mma(x, fa, TmT::load(sTm, 16 * wave + l16, 32 * k + 8 * kq));
      }
      store4(sdR + TokT::at(16 * wave + l16, 16 * vt + 4 * kq), x);
    }
    // ---- what does not need dR ----
    Frag fD[4], fS[NS], fdS[NS];
#pragma unroll
    for (int i = 0; i < 4; ++i) fD[i] = TokT::load(tD, 16 * i + l16, 8 * kq);
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      const int ch = 64 * u + 16 * wave;
      fS[u] = S16::join(__builtin_bit_cast(bf16x4, StT::tr4(tS, 8 * kq, ch, lane)), __builtin_bit_cast(bf16x4, StT::tr4(tS, 8 * kq + 4, ch, lane)));
      fdS[u] = S16::join(__builtin_bit_cast(bf16x4, StT::tr4(tdS, 8 * kq, ch, lane)), __builtin_bit_cast(bf16x4, StT::tr4(tdS, 8 * kq + 4, ch, lane)));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Frag f = TokT::load(tdO, 16 * i + l16, 8 * kq);
#pragma unroll
      for (int u = 0; u < NS; ++u) S16::mma(aQ[u][i], f, fS[u]), S16::mma(aK2[u][i], fD[i], fdS[u]);
      if (i == wave) {
#pragma unroll
        for (int j = 0; j <= i; ++j) S16::mma(aP[j], f, fD[j]);
      }
    }
#pragma unroll
    for (int u = 0; u < NS; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) ss[u] += (float)fS[u][e] * (float)fdS[u][e];  // <dS', S> of channel 64 u + 16 wave + l16
    lds_barrier();  // dR is there
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Frag f = TokT::load(sdR, 16 * i + l16, 8 * kq);
#pragma unroll
      for (int u = 0; u < NS; ++u) S16::mma(aK1[u][i], f, fS[u]);
      if (i == wave) {
#pragma unroll
        for (int j = 0; j <= i; ++j) S16::mma(aA[j], f, fD[j]);
      }
    }
    {  // <dR_t, v_t> and dv = beta dR: thread = (token tid / 4, eight value columns)
      const int t = tid >> 2, c0 = 8 * (tid & 3);
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
    if (s + 2 < nslab) {  // this buffer takes the slab after the next, once every wave has read it
      lds_barrier();
      issue(s + 2);
    }
  }
  lds_barrier();  // slab tiles are dead from here on

  // ---- epilogue ----
  T* sK = reinterpret_cast<T*>(region);
  T* sQ = reinterpret_cast<T*>(region + RowT::BYTES);
  T* sP = reinterpret_cast<T*>(region + L::oP);
  T* sA = sP + 64 * LDX;
  float* sDiag = reinterpret_cast<float*>(region + L::oF);  // scale dPm_tt
  float* sRdv = sDiag + 64;
  float* sC = sRdv + 64;   // [2] <q, dq> / |q|, <k, dk> / |k|
  float* sM = sC + 128;    // [3][set, wave]
#pragma unroll
  for (int u = 0; u < RowT::NINSTR / 4; ++u) {
    int r, c;
    RowT::src(wave + 4 * u, lane, r, c);
    r = min(r, len - 1);
    dma16(p.k + (tbase + (int64_t)r * ts) * DK + c, slab0 + 1024 * (wave + 4 * u));
    dma16(p.q + (tbase + (int64_t)r * ts) * DK + c, slab0 + RowT::BYTES + 1024 * (wave + 4 * u));
  }
  constexpr float LOG2E = 1.44269504f;
  float G[NS][16];  // the gate of this lane's channels and tokens, later its cumulative sum in units of log 2: it is read by exponentials alone
#pragma unroll
  for (int u = 0; u < NS; ++u)
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const int r = min(16 * (x >> 2) + 4 * kq + (x & 3), len - 1);
      const int64_t o = (tbase + (int64_t)r * ts) * DK + 64 * u + 16 * wave + l16;
      if constexpr (GRAW) G[u][x] = (float)p.graw[o];
      else G[u][x] = p.g[o];
    }
  rdv = quad_sum(rdv);
  if ((tid & 3) == 0) sRdv[tid >> 2] = rdv;
  if (tid < 64 && (!p.l2norm || tid >= len)) sNq[tid] = sNk[tid] = tid < len ? 1.f : 0.f;  // rows past the chunk's end are zero by their factor
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (j <= wave) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 16 * wave + 4 * kq + e, col = 16 * j + l16;
        const float x = p.scale * aP[j][e];
        sP[i * LDX + col] = (bf16_t)(i > col ? x : 0.f);
        sA[i * LDX + col] = (bf16_t)(i > col ? -aA[j][e] : 0.f);
        if (i == col) sDiag[i] = x;
      }
    }
  dma_wait<0>();
  lds_barrier();
#pragma unroll
  for (int u = 0; u < NS; ++u) {
    float gb = 0.f;
    if constexpr (GRAW) gb = p.gbias ? p.gbias[(row % p.geom.H) * DK + 64 * u + 16 * wave + l16] : 0.f;
    float before = 0.f;  // what the blocks of sixteen tokens before add
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int x = 4 * t + e;
        if constexpr (GRAW) G[u][x] = gna * lnx_softplus_thr(G[u][x] + gb, p.gthr);
        G[u][x] *= LOG2E;
        G[u][x] = 16 * t + 4 * kq + e < len ? G[u][x] : 0.f;
        if (e) G[u][x] += G[u][x - (e ? 1 : 0)];
      }
      // as the reverse sum of its gradient below
      const unsigned own = __float_as_uint(G[u][4 * t + 3]);
      const auto p16 = __builtin_amdgcn_permlane16_swap(own, own, false, false);
      const unsigned pair = __float_as_uint(__uint_as_float(p16[0]) + __uint_as_float(p16[1]));
      const auto p32 = __builtin_amdgcn_permlane32_swap(pair, pair, false, false);
      const float add = before + (((kq & 1) ? __uint_as_float(p16[0]) : 0.f) + ((kq & 2) ? __uint_as_float(p32[0]) : 0.f));
#pragma unroll
      for (int e = 0; e < 4; ++e) G[u][4 * t + e] += add;
      before += __uint_as_float(p32[0]) + __uint_as_float(p32[1]);
    }
    settle16(G[u]);
  }
  float dq[NS][16], dk[NS][16], dG[16];
  // K and Q at this lane's channel and tokens, normalised (rounded as the op rounds the normalised rows), zero past the chunk's end
  auto rows = [&](int u, bf16x4 (&k4)[4], bf16x4 (&q4)[4]) {
    const int lane = fresh(tid & 63);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const bf16x4 k = __builtin_bit_cast(bf16x4, RowT::tr4(sK, 16 * t + 4 * kq, 64 * u + 16 * wave, lane));
      const bf16x4 q = __builtin_bit_cast(bf16x4, RowT::tr4(sQ, 16 * t + 4 * kq, 64 * u + 16 * wave, lane));
      const floatx4 fk = load4(sNk + 16 * t + 4 * kq), fq = load4(sNq + 16 * t + 4 * kq);
      floatx4 kf, qf;
#pragma unroll
      for (int e = 0; e < 4; ++e) kf[e] = (float)k[e] * fk[e], qf[e] = (float)q[e] * fq[e];
      k4[t] = pack_bf16x4(kf), q4[t] = pack_bf16x4(qf);
    }
  };
  // Sums over the wave's sixteen channels of a set; lane l16 ends with value l16
  auto channel_sum = [&](float (&v)[16], int which, int u) {
    exchange<8>(v, l16), exchange<4>(v, l16), exchange<2>(v, l16), exchange<1>(v, l16);
    sM[64 * (4 * (NS * which + u) + wave) + 16 * (l16 >> 2) + 4 * kq + (l16 & 3)] = v[0];
  };
#pragma unroll
  for (int u = 0; u < NS; ++u) {
    const int lane = fresh(tid & 63);
    bf16x4 k4[4], q4[4];
    rows(u, k4, q4);
    PairSums s;
    float tot = 0.f;
    const float gC = __shfl(G[u][15], 48 + l16, LNX_WAVE);
    // what the loop left, and the diagonal of dPm; rp becomes dq, ra row, co dk without beta row
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const floatx4 d4 = load4(sDiag + 16 * t + 4 * kq);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int x = 4 * t + e;
        const float eg = __builtin_amdgcn_exp2f(G[u][x]), k2 = __builtin_amdgcn_exp2f(fminf(gC - G[u][x], 0.f)) * aK2[u][t][e], kv = (float)k4[t][e];
        s.rp[x] = p.scale * eg * aQ[u][t][e] + d4[e] * kv;
        s.ra[x] = -eg * aK1[u][t][e];
        s.co[x] = k2 + d4[e] * (float)q4[t][e];
        tot += kv * k2;
      }
    }
    pair_sums(s, G[u], k4, q4, sBeta, sP, sA, lane);
    float mv[16];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const floatx4 bt = load4(sBeta + 16 * t + 4 * kq);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int x = 4 * t + e;
        const float kv = (float)k4[t][e];
        mv[x] = kv * s.ra[x];
        dq[u][x] = s.rp[x];
        dk[u][x] = bt[e] * s.ra[x] + s.co[x];
        dG[x] = (float)q4[t][e] * dq[u][x] - kv * dk[u][x] + 2.f * bt[e] * mv[x];
      }
    }
    settle16(dq[u]), settle16(dk[u]), settle16(dG);
    channel_sum(mv, 0, u);
    if (p.l2norm) {
#pragma unroll
      for (int x = 0; x < 16; ++x) mv[x] = (float)q4[x >> 2][x & 3] * dq[u][x];
      channel_sum(mv, 1, u);
#pragma unroll
      for (int x = 0; x < 16; ++x) mv[x] = (float)k4[x >> 2][x & 3] * dk[u][x];
      channel_sum(mv, 2, u);
    }
    tot = xor32_sum(xor16_sum(tot + __builtin_amdgcn_exp2f(gC) * ss[u]));  // over the tokens (ss: over its value columns) of this channel
    if (kq == 3) dG[15] += tot;
    // dg: reverse cumulative sum over the chunk's tokens of this channel
    float after = 0.f;  // what later blocks of sixteen tokens add
#pragma unroll
    for (int t = 3; t >= 0; --t) {
#pragma unroll
      for (int e = 2; e >= 0; --e) dG[4 * t + e] += dG[4 * t + e + 1];
      // the four lane groups' totals on the VALU (xor16_sum in lnx_common.h): a group adds its odd neighbour's and the upper pair's
      const unsigned own = __float_as_uint(dG[4 * t]);
      const auto p16 = __builtin_amdgcn_permlane16_swap(own, own, false, false);
      const unsigned pair = __float_as_uint(__uint_as_float(p16[0]) + __uint_as_float(p16[1]));
      const auto p32 = __builtin_amdgcn_permlane32_swap(pair, pair, false, false);
      const float add = after + ((kq & 1) ? 0.f : __uint_as_float(p16[1])) + ((kq & 2) ? 0.f : __uint_as_float(p32[1]));
#pragma unroll
      for (int e = 0; e < 4; ++e) dG[4 * t + e] += add;
      after += __uint_as_float(p32[0]) + __uint_as_float(p32[1]);
    }
    settle16(dG);
    if (u + 1 < NS) {
      float* sG0 = reinterpret_cast<float*>(region + L::oG0);
#pragma unroll
      for (int x = 0; x < 16; ++x) sG0[(16 * (x >> 2) + 4 * kq + (x & 3)) * L::LDF + 16 * wave + l16] = dG[x];
    }
    settle16(dq[u]), settle16(dk[u]), settle16(dG);  // one set at a time
  }
  lds_barrier();  // the shares are there; dPm and dXa are dead, a wave's channels of K and Q are its own
  auto shares = [&](int which, int t) {
    float x = 0.f;
#pragma unroll
    for (int w = 0; w < 4 * NS; ++w) x += sM[64 * (4 * NS * which + w) + t];
    return x;
  };
  if (tid < 64) {
    if (tid < len) p.dbeta[tbase + tid * ts] = sRdv[tid] + shares(0, tid);
  } else if (p.l2norm && tid < 192) {  // through the normalisation: d/dx of x / (|x| + eps) applied to dy is dy / (|x| + eps) - y <y, dy> / |x|
    const int t = tid & 63, w = (tid >> 6) - 1;
    const float nrm = 1.f / (w ? sNk : sNq)[t] - LNX_L2_EPS;
    sC[64 * w + t] = nrm > 0.f ? shares(1 + w, t) / nrm : 0.f;
  }
  if (p.l2norm) {
    lds_barrier();
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      bf16x4 k4[4], q4[4];
      rows(u, k4, q4);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const floatx4 fq = load4(sNq + 16 * t + 4 * kq), fk = load4(sNk + 16 * t + 4 * kq), cq = load4(sC + 16 * t + 4 * kq), ck = load4(sC + 64 + 16 * t + 4 * kq);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          dq[u][4 * t + e] = fq[e] * dq[u][4 * t + e] - cq[e] * (float)q4[t][e];
          dk[u][4 * t + e] = fk[e] * dk[u][4 * t + e] - ck[e] * (float)k4[t][e];
        }
      }
    }
  }
  // ---- dq, dk out over the K and Q tiles, by rows ----
#pragma unroll
  for (int u = 0; u < NS; ++u)
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const int o = RowT::at(16 * (x >> 2) + 4 * kq + (x & 3), 64 * u + 16 * wave + l16);
      sK[o] = (bf16_t)dk[u][x];
      sQ[o] = (bf16_t)dq[u][x];
    }
  lds_barrier();
#pragma unroll
  for (int u = 0; u < 64 * DK / 8 / 256; ++u) {
    const int idx = tid + 256 * u, r = idx / (DK / 8), c = 8 * (idx % (DK / 8));
    if (r < len) {
      *reinterpret_cast<Frag*>(p.dq + tbase * DK + (int64_t)r * tsk + c) = RowT::load(sQ, r, c);
      *reinterpret_cast<Frag*>(p.dk + tbase * DK + (int64_t)r * tsk + c) = RowT::load(sK, r, c);
    }
  }
  lds_barrier();  // dq and dk have left
  // ---- dg, or the raw projection's gradient, by rows ----
  // With the gate activated inside the op, g = -e^{A_log} softplus(x), x = raw + bias (kda.py:153-165), the gradient goes on to the raw
  // projection: dg g for A_log, -e^{A_log} sigmoid(x) dg (softplus' derivative is 1 beyond the threshold) for it and the bias.  The projection
  // is read again here, by rows: as the difference of two rows of the cumulative gate, in the registers of the loop above, the activated gate
  // cost shuffles and 21 spilled registers (B4 H16 T8192 d128: 643 us, so 544; 470 without the activation).
  float* sOut = reinterpret_cast<float*>(region);
#pragma unroll
  for (int x = 0; x < 16; ++x) sOut[(16 * (x >> 2) + 4 * kq + (x & 3)) * L::LDF + 16 * wave + l16] = dG[x];
  lds_barrier();
  float* sPart = reinterpret_cast<float*>(region + L::oPart);  // GRAW: [set][which][wave][64]
#pragma unroll
  for (int u = 0; u < NS; ++u) {
    const float* src = u + 1 < NS ? reinterpret_cast<const float*>(region + L::oG0) : sOut;
    const int c = 4 * (tid & 15);  // the thread's channels of the set, in all its rows
    bf16x4 raw[4];
    floatx4 gb = {0.f, 0.f, 0.f, 0.f}, sb = gb, sa = gb;
    if constexpr (GRAW) {
#pragma unroll
      for (int it = 0; it < 4; ++it) raw[it] = *reinterpret_cast<const bf16x4*>(p.graw + (tbase + (int64_t)min((tid >> 4) + 16 * it, len - 1) * ts) * DK + 64 * u + c);
      if (p.gbias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) gb[e] = p.gbias[(row % p.geom.H) * DK + 64 * u + c + e];
      }
    }
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      const int r = (tid >> 4) + 16 * it;
      const int64_t o = (tbase + (int64_t)r * ts) * DK + 64 * u + c;
      floatx4 d = load4(src + r * L::LDF + c);
      if constexpr (GRAW) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = (float)raw[it][e] + gb[e], ex = __expf(-fabsf(x)), q = 1.f + ex;
          const bool lin = x > p.gthr;
          const float sp = lin ? x : fmaxf(x, 0.f) + __logf(q), ds = lin ? 1.f : __fdividef(x > 0.f ? 1.f : ex, q);
          const float dr = r < len ? d[e] * gna : 0.f;
          sa[e] += dr * sp;
          d[e] = dr * ds;
          sb[e] += d[e];
        }
        if (r < len) store4(p.dgraw + o, d);
      } else if (r < len) {
        store4(p.dg + o, d);
      }
    }
    if constexpr (GRAW) {
#pragma unroll
      for (int e = 0; e < 4; ++e) sb[e] = xor32_sum(xor16_sum(sb[e])), sa[e] = xor32_sum(xor16_sum(sa[e]));
      if (lane < 16) store4(sPart + (2 * u * 4 + wave) * 64 + c, sb), store4(sPart + ((2 * u + 1) * 4 + wave) * 64 + c, sa);
    }
  }
  if constexpr (GRAW) {
    lds_barrier();
    if (tid < 2 * DK) {
      const int which = tid / DK, c = tid % DK;
      const float* x = sPart + (2 * (c >> 6) + which) * 256 + (c & 63);
      gate_part(which)[c] = (x[0] + x[64]) + (x[128] + x[192]);
    }
  }
}

// ---------------------------------------------------------------------------------------
// kda_scan_fwd: the forward pass over the chunks of one (state, 32-column slab of dv) where there are few of them and the
// chain of a chunk is what a call waits for:  D = U - W S,  S <- diag(e^{G_C}) S + Kr^T D,  O = Qg S + P D.  chunk_scan
// (chunk_fwd.hip) takes the chain through LDS between every two products, three barriers a chunk; here, as in scan_fwd
// (chunk_direct.hip), a compute wave owns sixteen value columns, their part of the state stays in accumulators and is, like
// D, an operand as it stands, and O has waves of its own a chunk behind.  What prepare leaves is an operand as it is, so no
// wave converts anything: four waves request the tiles straight into LDS, four others take the states and D away.
// One chunk: dk = 128 1.80 -> 1.38 us, dk = 64 1.99 -> 1.12 us.  Fetching lines ahead into the L2 by the idle savers (three
// chunks ahead, for the full chip) made it slower: a prompt of four heads 192 -> 197 us, a saving scan 378 -> 408.
//   B1    W, Kr, U of chunk n,   compute: D, state update; S^T and D^T -> LDS [n mod 2]   loads:  W, Kr, U of n + 1, Qg, P of n
//         Qg, P of n - 1         output:  O of chunk n - 1; e^{G_C} of n + 1              savers: S, D of n - 1 -> workspace
// ---------------------------------------------------------------------------------------
template <int DK> struct KdaScanL {
  typedef SwzTile<64, DK> RowT;  // W, Kr, Qg
  typedef SwzTile<64, 32> ValT;  // U
  typedef SwzTile<64, 64> TriT;  // P
  typedef SwzTile<32, DK> StT;   // S^T
  typedef SwzTile<32, 64> DtT;   // D^T
  static constexpr int oKr = RowT::BYTES, oU = 2 * RowT::BYTES, first = oU + ValT::BYTES;  // W | Kr | U
  static constexpr int oP = RowT::BYTES, second = oP + TriT::BYTES;                        // Qg | P
  static constexpr int oSecond = 2 * first, oS = oSecond + 2 * second, oD = oS + 2 * StT::BYTES, oE = oD + 2 * DtT::BYTES;
  static constexpr size_t bytes = oE + 2 * DK * sizeof(float);
  static_assert(bytes <= 160 * 1024, "LDS");
  static constexpr int threads = 64 * 12;
};

template <int DK>
__global__ __launch_bounds__((KdaScanL<DK>::threads)) void kda_scan_fwd_kernel(DirectParams p) {
  typedef KdaScanL<DK> L;
  typedef typename L::RowT RowT;
  typedef typename L::ValT ValT;
  typedef typename L::TriT TriT;
  typedef typename L::StT StT;
  typedef typename L::DtT DtT;
  constexpr int KT = DK / 16, NK = DK / 32;
  extern __shared__ __align__(16) char smem[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l16 = lane & 15, kq = lane >> 4;
  const int N = p.geom.N;
  int64_t chain;
  int slab, sidx, row, seq, c0, c1;
  if (!xcd_slot_part((int64_t)(p.geom.tab ? p.geom.nseq : p.geom.rows / p.geom.H) * p.geom.H, p.dv / 32, chain, slab)) return;
  scan_state(p.geom, (int)chain, sidx, row, seq);
  seq_chunks(p.geom, seq, c0, c1);
  const SeqSpan span = seq_span(p.geom, seq, c0);
  const int v0 = 32 * slab, vs = 16 * (wave & 1);
  auto first = [&](int n) { return smem + ((n - c0) & 1) * L::first; };
  auto second = [&](int n) { return smem + L::oSecond + ((n - c0) & 1) * L::second; };
  auto state_t = [&](int n) { return reinterpret_cast<T*>(smem + L::oS + ((n - c0) & 1) * StT::BYTES); };
  auto d_t = [&](int n) { return reinterpret_cast<T*>(smem + L::oD + ((n - c0) & 1) * DtT::BYTES); };
  auto decay = [&](int n) { return reinterpret_cast<float*>(smem + L::oE) + ((n - c0) & 1) * DK; };

  if (wave >= 8) {  // ---------------- savers ----------------
    const int t = tid - 512;
    auto save = [&](int n) {
      const int64_t slot = (int64_t)row * N + n;
      const T* st = state_t(n);
      const T* dt = d_t(n);
      T* S = at<T>(p.ws, p.off.SnT) + slot * p.dv * DK + (int64_t)v0 * DK;
      T* D = at<T>(p.ws, p.off.D) + slot * 64 * p.dv + v0;
#pragma unroll
      for (int u = 0; u < 32 * DK / 8 / 256; ++u) {
        const int i = t + 256 * u, r = i / (DK / 8), c = 8 * (i % (DK / 8));
        *reinterpret_cast<Frag*>(S + r * DK + c) = StT::load(st, r, c);
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {  // four value columns of a token: rows of D^T
        const int b = 2 * (wave & 3) + u, v = 4 * (kq + 4 * (b & 1)), tok = 16 * (b >> 1);
        *reinterpret_cast<bf16x4*>(D + (int64_t)(tok + l16) * p.dv + v) = __builtin_bit_cast(bf16x4, DtT::tr4(dt, v, tok, lane));
      }
    };
    lds_barrier();
    for (int n = c0; n < c1; ++n) {
      if (p.save && n > c0) save(n - 1);
      lds_barrier();
    }
    if (p.save && c0 < c1) save(c1 - 1);
    return;
  }
  if (wave >= 4) {  // ---------------- loads ----------------
    const int w = wave - 4;
    auto rows = [&](uint64_t off, int64_t slot, char* dst) {
#pragma unroll
      for (int u = 0; u < RowT::NINSTR / 4; ++u) {
        int r, c;
        RowT::src(w + 4 * u, lane, r, c);
        dma16(at<const T>(p.ws, off) + slot * 64 * DK + r * DK + c, lds_byte_addr(dst) + 1024 * (w + 4 * u));
      }
    };
    auto load_first = [&](int n) {
      const int64_t slot = (int64_t)row * N + n;
      char* dst = first(n);
      rows(p.off.W, slot, dst);
      rows(p.off.Kr, slot, dst + L::oKr);
      int r, c;
      ValT::src(w, lane, r, c);
      dma16(at<const T>(p.ws, p.off.U) + slot * 64 * p.dv + (int64_t)r * p.dv + v0 + c, lds_byte_addr(dst) + L::oU + 1024 * w);
    };
    auto load_second = [&](int n) {
      const int64_t slot = (int64_t)row * N + n;
      char* dst = second(n);
      rows(p.off.Qg, slot, dst);
#pragma unroll
      for (int u = 0; u < TriT::NINSTR / 4; ++u) {
        int r, c;
        TriT::src(w + 4 * u, lane, r, c);
        dma16(at<const T>(p.ws, p.off.P) + slot * 64 * 64 + r * 64 + c, lds_byte_addr(dst) + L::oP + 1024 * (w + 4 * u));
      }
    };
    static_assert(ValT::NINSTR == 4 && RowT::NINSTR % 4 == 0 && TriT::NINSTR % 4 == 0, "the same count for every wave");
    if (c0 < c1) load_first(c0);
    dma_wait<0>();
    lds_barrier();
    for (int n = c0; n < c1; ++n) {
      if (n + 1 < c1) load_first(n + 1);
      if (p.o) load_second(n);
      dma_wait<0>();
      lds_barrier();
    }
    return;
  }
  if (wave >= 2) {  // ---------------- output waves: O^T of a strip, lane = token ----------------
    const int ch = DK == 128 ? 64 * (wave & 1) + lane : lane;
    float g = 0.f;
    auto fetch = [&](int n) { g = at<const float>(p.ws, p.off.G)[((int64_t)row * N + min(n, c1 - 1)) * DK + ch]; };
    auto commit = [&](int n) { decay(n)[ch] = __expf(g); };
    if (c0 < c1) {
      fetch(c0), commit(c0);
      fetch(c0 + 1);
    }
    lds_barrier();
    for (int n = c0; n < c1; ++n) {
      commit(n + 1);
      fetch(n + 2);
      lds_barrier();  // chunk n + 1, or the end of the last
      if (!p.o) continue;
      const T* tQ = reinterpret_cast<const T*>(second(n));
      const T* tP = reinterpret_cast<const T*>(second(n) + L::oP);
      int tok0, len;
      chunk_span(span, n, tok0, len);
      floatx4 o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) {
        const Frag b = StT::load(state_t(n), vs + l16, 32 * ks + 8 * kq);
#pragma unroll
        for (int i = 0; i < 4; ++i) S16::mma(o[i], b, RowT::load(tQ, 16 * i + l16, 32 * ks + 8 * kq));
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const Frag b = DtT::load(d_t(n), vs + l16, 32 * s + 8 * kq);
#pragma unroll
        for (int i = 2 * s; i < 4; ++i) S16::mma(o[i], b, TriT::load(tP, 16 * i + l16, 32 * s + 8 * kq));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 16 * i + l16;
        const int64_t e = (tok_index(p.geom, row, tok0) + (int64_t)t * p.geom.ts) * p.dv + v0 + vs + 4 * kq;
        if (t < len) {
          if (p.o_dtype == LNX_F32) store4(reinterpret_cast<float*>(p.o) + e, o[i]);
          else store4(reinterpret_cast<T*>(p.o) + e, o[i]);
        }
      }
    }
    return;
  }

  // ---------------- compute waves: value columns v0 + vs .. + 15, rows of tile i: row0(i) + 8 kq + e ----------------
  auto row0 = [](int i) { return 32 * (i >> 1) + 4 * (i & 1); };
  const int lr = 8 * ((lane >> 2) & 3) + (lane & 3);  // operand row l16 of such a tile
  floatx4 S[KT];
#pragma unroll
  for (int ci = 0; ci < KT; ++ci)
#pragma unroll
    for (int e = 0; e < 4; ++e) S[ci][e] = p.ident && row0(ci) + 8 * kq + e == v0 + vs + l16 - p.vcols ? 1.f : 0.f;
  if (!p.ident && p.s0) {
    const float* s0 = p.s0 + (int64_t)sidx * DK * p.dv + v0 + vs + l16;
#pragma unroll
    for (int ci = 0; ci < KT; ++ci)
#pragma unroll
      for (int e = 0; e < 4; ++e) S[ci][e] = s0[(int64_t)(row0(ci) + 8 * kq + e) * p.dv];
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) asm volatile("" : "+v"(S[ci]));
  }
  const bool keep = p.o || p.save;
  lds_barrier();
  for (int n = c0; n < c1; ++n) {
    const T* tW = reinterpret_cast<const T*>(first(n));
    const T* tK = reinterpret_cast<const T*>(first(n) + L::oKr);
    const T* tU = reinterpret_cast<const T*>(first(n) + L::oU);
    const float* eg = decay(n);
    floatx4 y[4];
    Frag fa[NK][4], b[NK], bd[2], fu[2][KT];
    bf16x4 u4[4];
    auto load_w = [&](int ks) {
#pragma unroll
      for (int i = 0; i < 4; ++i) fa[ks][i] = RowT::load(tW, row0(i) + lr, 32 * ks + 8 * kq);
    };
    // channels of state tile ci, tokens 32 s + 8 kq ..
    auto load_k = [&](int s, int ci) {
      const int q = lane & 15, c = 32 * (ci >> 1) + 4 * (ci & 1) + 8 * (q & 3), r = 32 * s + 8 * kq + (q >> 2);
      return S16::join(__builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((S16::lds_short4*)(tK + RowT::at(r, c)))),
                       __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((S16::lds_short4*)(tK + RowT::at(r + 4, c)))));
    };
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    load_w(0), load_w(1);
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      b[ks] = S16::from_acc(S[2 * ks], S[2 * ks + 1]);
      if (ks + 2 < NK) {
        load_w(ks + 2);
      } else if (ks + 2 == NK) {
#pragma unroll
        for (int i = 0; i < 4; ++i) u4[i] = __builtin_bit_cast(bf16x4, ValT::tr4(tU, row0(i) + 8 * kq, vs, lane));
      } else {
#pragma unroll
        for (int ci = 0; ci < KT / 2; ++ci) fu[0][ci] = load_k(0, ci);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; ++i) S16::mma(y[i], fa[ks][i], b[ks]);
    }
    if (keep) {  // read behind the next barrier
#pragma unroll
      for (int ks = 0; ks < NK; ++ks) *reinterpret_cast<Frag*>(state_t(n) + StT::at(vs + l16, 32 * ks + 8 * kq)) = b[ks];
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 2 * s; i < 2 * s + 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) y[i][e] = (float)u4[i][e] - y[i][e];
      bd[s] = S16::from_acc(y[2 * s], y[2 * s + 1]);
    }
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) S[ci] *= load4(eg + row0(ci) + 8 * kq);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ci = KT / 2; ci < KT; ++ci) fu[0][ci] = load_k(0, ci);
#pragma unroll
    for (int ci = 0; ci < KT / 2; ++ci) S16::mma(S[ci], fu[0][ci], bd[0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) fu[1][ci] = load_k(1, ci);
#pragma unroll
    for (int ci = KT / 2; ci < KT; ++ci) S16::mma(S[ci], fu[0][ci], bd[0]);
    if (keep) {
#pragma unroll
      for (int s = 0; s < 2; ++s) *reinterpret_cast<Frag*>(d_t(n) + DtT::at(vs + l16, 32 * s + 8 * kq)) = bd[s];
    }
#pragma unroll
    for (int ci = 0; ci < KT; ++ci) S16::mma(S[ci], fu[1][ci], bd[1]);
    lds_barrier();
  }
  float* out = p.sT_out.at(sidx, (int64_t)DK * p.dv) + v0 + vs + l16;
#pragma unroll
  for (int ci = 0; ci < KT; ++ci)
#pragma unroll
    for (int e = 0; e < 4; ++e) out[(int64_t)(row0(ci) + 8 * kq + e) * p.dv] = S[ci][e];
}

template <int DK>
int launch_scan(const DirectParams& p, int nstate, hipStream_t st) {
  auto k = kda_scan_fwd_kernel<DK>;
  const size_t b = KdaScanL<DK>::bytes;
  if (const int rc = lnx_lds_limit((const void*)k, b); rc != LNX_OK) return rc;
  lnx_profile_mark("chunk_scan", st);
  hipLaunchKernelGGL(k, dim3(lnx_xcd_grid((int64_t)nstate * p.geom.H, p.dv / 32)), dim3(KdaScanL<DK>::threads), b, st, p);
  lnx_profile_mark(nullptr, st);
  return LNX_OK;
}

template <int DK>
int launch(const KdaBwdParams& p, hipStream_t st) {
  auto k = p.graw ? kda_bwd_chunk_kernel<DK, true> : kda_bwd_chunk_kernel<DK, false>;
  const size_t b = KdaL<DK>::bytes;
  if (const int rc = lnx_lds_limit((const void*)k, b); rc != LNX_OK) return rc;
  lnx_profile_mark("bwd_chunk", st);
  hipLaunchKernelGGL(k, dim3((unsigned)((int64_t)p.geom.rows * p.geom.N)), dim3(256), b, st, p);
  lnx_profile_mark(nullptr, st);
  return LNX_OK;
}

}  // namespace

int lnx_kda_bwd_chunk(const KdaBwdParams& p, int dk, hipStream_t st) { return dk == 128 ? launch<128>(p, st) : launch<64>(p, st); }

int lnx_kda_scan_fwd(const DirectParams& p, int dk, int nstate, hipStream_t st) { return dk == 128 ? launch_scan<128>(p, nstate, st) : launch_scan<64>(p, nstate, st); }
