// Gated DeltaNet's gate and learning-rate activations and their gradient
// (linearnexus/modules/linear_attn/gated_deltanet.py:804-815):
//   g[r, h]    = -exp(A_log[h]) * softplus(a[r, h] + dt_bias[h])        fp32 log-decay per token and head
//   beta[r, h] = beta_scale * sigmoid(b[r, h])                          beta_scale = 2 with allow_neg_eigval, else 1
// a and b are the [rows, H] outputs of the block's a_proj / b_proj in the activation dtype; g and beta leave in fp32,
// the type the scan kernels read.  Two megabytes at the benchmark shapes, so what bounds both directions is the memory
// round trips of a wave and not the bytes: every lane works on an element of its own (a workgroup takes 256 / H whole rows
// at a time), in the backward on at least four.  B2 T2007 H16: forward 45 -> 3.6 us, backward 56 + 22 (four launches for the
// sums) -> 8 + 4.5 us against a thread per (head, 64 rows), which left 240 of 256 lanes idle and walked 64 dependent rows.
// The backward keeps the per-head sums for d_A_log and d_dt_bias in registers, adds them over the workgroup in LDS,
// leaves one partial row per workgroup in a caller-owned workspace, and one more launch adds the rows (no atomics,
// deterministic).
#include "lnx_common.h"

namespace {

constexpr int BWD_BLOCKS = 512;  // most workgroups of the backward along the rows: partial rows that one wave per sum adds in one round

struct GdnGateParams {
  const void* a; const void* b; const float* A_log; const float* dt_bias;
  float* g; float* beta;
  const float* d_g; const float* d_beta; void* d_a; void* d_b; float* part;  // part: [2][nblocks][H]
  int64_t rows; int H, per; float beta_scale;                               // per: rows of a backward workgroup
};

// log(1 + e^x) in the overflow-free form max(x, 0) + log1p(e^-|x|) (what jax.nn.softplus evaluates)
__device__ __forceinline__ float softplus_f(float x) { return fmaxf(x, 0.f) + log1pf(__expf(-fabsf(x))); }
__device__ __forceinline__ float sigmoid_f(float x) { return 1.f / (1.f + __expf(-x)); }

// thread = element
template <typename T>
__global__ __launch_bounds__(256) void gdn_gate_fwd_kernel(GdnGateParams p) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= p.rows * p.H) return;
  const int h = (int)(i % p.H);
  const float x = to_f32(static_cast<const T*>(p.a)[i]) + (p.dt_bias ? p.dt_bias[h] : 0.f);
  p.g[i] = -__expf(p.A_log[h]) * softplus_f(x);
  if (p.b) p.beta[i] = p.beta_scale * sigmoid_f(to_f32(static_cast<const T*>(p.b)[i]));
}

// Heads in blocks of 256 (blockIdx.x); a workgroup covers `per` rows of its heads, G = 256 / heads of them at a time
template <typename T>
__global__ __launch_bounds__(256) void gdn_gate_bwd_kernel(GdnGateParams p) {
  __shared__ float red[2][256];
  const int h0 = blockIdx.x * 256, nh = min(256, p.H - h0), G = 256 / nh;
  const int rg = threadIdx.x / nh, h = h0 + threadIdx.x - rg * nh;
  float sb = 0.f, sa = 0.f;
  if (rg < G) {
    const int64_t r0 = (int64_t)blockIdx.y * p.per, r1 = min(r0 + p.per, p.rows);
    const float na = -__expf(p.A_log[h]), bias = p.dt_bias ? p.dt_bias[h] : 0.f;
    const T* a = static_cast<const T*>(p.a);
    const T* b = static_cast<const T*>(p.b);
    T* da = static_cast<T*>(p.d_a);
    T* db = static_cast<T*>(p.d_b);
#pragma unroll 4
    for (int64_t r = r0 + rg; r < r1; r += G) {
      const int64_t i = r * p.H + h;
      const float x = to_f32(a[i]) + bias, dg = p.d_g ? p.d_g[i] : 0.f;
      const float dx = dg * na * sigmoid_f(x);  // softplus' = sigmoid
      sa += dg * na * softplus_f(x);            // d g / d A_log = g
      sb += dx;
      da[i] = from_f32<T>(dx);
      if (b) {
        const float s = sigmoid_f(to_f32(b[i]));
        db[i] = from_f32<T>((p.d_beta ? p.d_beta[i] : 0.f) * p.beta_scale * s * (1.f - s));
      }
    }
  }
  if (!p.part) return;
  red[0][threadIdx.x] = sb;
  red[1][threadIdx.x] = sa;
  __syncthreads();
  if (rg == 0) {
    for (int q = 1; q < G; ++q) sb += red[0][q * nh + threadIdx.x], sa += red[1][q * nh + threadIdx.x];
    p.part[(int64_t)blockIdx.y * p.H + h] = sb;
    p.part[((int64_t)gridDim.y + blockIdx.y) * p.H + h] = sa;
  }
}

// The partial rows added up: one wavefront per (head, sum)
__global__ __launch_bounds__(64) void gdn_gate_sum_kernel(const float* part, int n, int H, float* d_bias, float* d_A) {
  float* out = blockIdx.y ? d_A : d_bias;
  if (!out) return;
  part += (int64_t)blockIdx.y * n * H + blockIdx.x;
  float t = 0.f;
#pragma unroll 8
  for (int r = threadIdx.x; r < n; r += 64) t += part[(int64_t)r * H];
  t = wave_sum(t);
  if (threadIdx.x == 0) out[blockIdx.x] = t;
}

__global__ void zero_heads_kernel(float* a, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0.f;
}

int check(int64_t rows, int H, int dtype) {
  if (rows < 0 || H <= 0) return lnx_set_error(LNX_ERR_SHAPE, "gdn_gate: rows=%lld H=%d", (long long)rows, H);
  if (dtype != LNX_F32 && dtype != LNX_BF16) return lnx_set_error(LNX_ERR_DTYPE, "gdn_gate: dtype %d", dtype);
  return LNX_OK;
}

// Rows of a backward workgroup: four per lane, more only where that would leave over BWD_BLOCKS partial rows
int64_t bwd_rows(int64_t rows, int H) {
  const int G = 256 / (H < 256 ? H : 256);
  const int64_t need = (rows + BWD_BLOCKS - 1) / BWD_BLOCKS;
  return need > 4 * G ? (need + G - 1) / G * G : 4 * G;
}

}  // namespace

extern "C" int lnx_gdn_gate_fwd(const void* a, const void* b, const float* A_log, const float* dt_bias, float* g, float* beta,
                                int64_t rows, int32_t H, float beta_scale, int32_t dtype, void* hip_stream) {
  if (int rc = check(rows, H, dtype)) return rc;
  if (rows == 0) return LNX_OK;
  if (!a || !A_log || !g || (b && !beta)) return lnx_set_error(LNX_ERR_NULL, "gdn_gate_fwd: a, A_log and g are required (beta with b)");
  hipStream_t st = static_cast<hipStream_t>(hip_stream);
  GdnGateParams p{a, b, A_log, dt_bias, g, beta, nullptr, nullptr, nullptr, nullptr, nullptr, rows, H, 0, beta_scale};
  dim3 grid((unsigned)((rows * H + 255) / 256));
  lnx_profile_mark("gdn_gate_fwd", st);
  if (dtype == LNX_BF16) gdn_gate_fwd_kernel<bf16_t><<<grid, 256, 0, st>>>(p);
  else gdn_gate_fwd_kernel<float><<<grid, 256, 0, st>>>(p);
  lnx_profile_mark(nullptr, st);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? LNX_OK : lnx_set_error(LNX_ERR_LAUNCH, "gdn_gate_fwd: %s", hipGetErrorString(e));
}

extern "C" uint64_t lnx_gdn_gate_bwd_workspace_bytes(int64_t rows, int32_t H) {
  if (rows <= 0 || H <= 0) return 0;
  const int64_t per = bwd_rows(rows, H);
  return 2 * (uint64_t)((rows + per - 1) / per) * H * sizeof(float);
}

extern "C" int lnx_gdn_gate_bwd(const void* a, const void* b, const float* A_log, const float* dt_bias, const float* d_g,
                                const float* d_beta, void* d_a, void* d_b, float* d_A_log, float* d_dt_bias, int64_t rows,
                                int32_t H, float beta_scale, int32_t dtype, void* workspace, uint64_t workspace_bytes,
                                void* hip_stream) {
  if (int rc = check(rows, H, dtype)) return rc;
  if (!A_log) return lnx_set_error(LNX_ERR_NULL, "gdn_gate_bwd: A_log is required");
  if (rows > 0 && (!a || !d_a || (b && !d_b))) return lnx_set_error(LNX_ERR_NULL, "gdn_gate_bwd: a and d_a are required (d_b with b)");
  hipStream_t st = static_cast<hipStream_t>(hip_stream);
  const bool sums = d_A_log || d_dt_bias;
  float* part = nullptr;
  if (sums && rows > 0) {
    const uint64_t need = lnx_gdn_gate_bwd_workspace_bytes(rows, H);
    if (!workspace || workspace_bytes < need)
      return lnx_set_error(LNX_ERR_WORKSPACE, "gdn_gate_bwd: parameter gradients need a workspace of %llu bytes", (unsigned long long)need);
    part = static_cast<float*>(workspace);
  }
  lnx_profile_mark("gdn_gate_bwd", st);
  if (rows > 0) {
    const int64_t per = bwd_rows(rows, H);
    const int nblk = (int)((rows + per - 1) / per);
    GdnGateParams p{a, b, A_log, dt_bias, nullptr, nullptr, d_g, d_beta, d_a, d_b, part, rows, H, (int)per, beta_scale};
    dim3 grid((H + 255) / 256, nblk);
    if (dtype == LNX_BF16) gdn_gate_bwd_kernel<bf16_t><<<grid, 256, 0, st>>>(p);
    else gdn_gate_bwd_kernel<float><<<grid, 256, 0, st>>>(p);
    if (sums) gdn_gate_sum_kernel<<<dim3(H, 2), 64, 0, st>>>(part, nblk, H, d_dt_bias, d_A_log);
  } else if (sums) {  // no rows: the sums are zero
    if (d_dt_bias) zero_heads_kernel<<<(H + 255) / 256, 256, 0, st>>>(d_dt_bias, H);
    if (d_A_log) zero_heads_kernel<<<(H + 255) / 256, 256, 0, st>>>(d_A_log, H);
  }
  lnx_profile_mark(nullptr, st);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? LNX_OK : lnx_set_error(LNX_ERR_LAUNCH, "gdn_gate_bwd: %s", hipGetErrorString(e));
}
