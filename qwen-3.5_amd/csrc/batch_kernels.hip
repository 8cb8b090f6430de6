// Kernels of the batched decode step that the single-sequence kernels do not cover: the
// per-sequence token selection + embedding into the residual rows, the residual add and RMSNorm
// between two projections of the multi-row matvec, and the per-sequence greedy argmax over the logits rows (the reference's tie order), which advances
// each sequence's position and history.
#include "q35_internal.h"

#include <algorithm>
#include <climits>

namespace q35 {
namespace {

constexpr int kBT = 256;

// Row b: the prompt id at pos[b] while pos[b] < plen[b], else the row's last argmax; its
// dequantised embedding row goes to the residual row h[b] (fixed point).
__global__ __launch_bounds__(kBT) void batch_embed_kernel(const int8_t* q, const float* s, int D,
                                                         const int32_t* token, const int32_t* prompt, int ldp,
                                                         const int32_t* plen, const int32_t* pos, fx_t* h) {
  const int b = blockIdx.y;
  const int p = pos[b];
  const int tok = p < plen[b] ? prompt[(int64_t)b * ldp + p] : token[b];
  const int8_t* qr = q + (int64_t)tok * D;
  const float* sr = s + (int64_t)tok * (D / 64);
  for (int k = blockIdx.x * kBT + threadIdx.x; k < D; k += gridDim.x * kBT)
    h[(int64_t)b * D + k] = to_fx((float)qr[k] * sr[k >> 6]);
}

// f32 residual rows for the batched step on the matrix cores: row b's embedding (as above) into
// h[b] and its sum of squares into ss[b] (the first RMSNorm's statistic); every block also
// clears its share of zero_ptr[0 .. zero_n) (accumulators the step adds into).
__global__ __launch_bounds__(kBT) void batch_embed_f32_kernel(const int8_t* q, const float* s, int D,
                                                             const int32_t* token, const int32_t* prompt, int ldp,
                                                             const int32_t* plen, const int32_t* pos, float* h, fx_t* ss,
                                                             fx_t* zero_ptr, int64_t zero_n, uint32_t* err) {
  __shared__ float sh[4];
  for (int64_t i = (int64_t)blockIdx.x * kBT + threadIdx.x; i < zero_n; i += (int64_t)gridDim.x * kBT) zero_ptr[i] = 0;
  const int b = blockIdx.x;
  const int p = pos[b];
  const int tok = p < plen[b] ? prompt[(int64_t)b * ldp + p] : token[b];
  const int8_t* qr = q + (int64_t)tok * D;
  const float* sr = s + (int64_t)tok * (D / 64);
  float acc = 0.f;
  for (int k = threadIdx.x; k < D; k += kBT) {
    const float e = (float)qr[k] * sr[k >> 6];
    h[(int64_t)b * D + k] = e;
    acc += e * e;
  }
  acc = block_sum256(acc, sh);
  if (threadIdx.x == 0) {
    if (!fx_addable(acc)) __hip_atomic_fetch_or((Q35_GLOBAL uint32_t*)err, kWsErrRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    ss[b] = fx_addable(acc) ? to_fx(acc) : 0;
  }
}

typedef int i32x2 __attribute__((ext_vector_type(2)));
// x from lane (l + N) mod 16 of the 16-lane row, and the sum over a wave, of doubles (as row_ror and
// wave_sum)
template <int N>
Q35_DEV double row_ror64(double x) {
  const i32x2 u = __builtin_bit_cast(i32x2, x);
  return __builtin_bit_cast(double, i32x2{__builtin_amdgcn_update_dpp(0, u[0], 0x120 + N, 0xf, 0xf, false),
                                          __builtin_amdgcn_update_dpp(0, u[1], 0x120 + N, 0xf, 0xf, false)});
}
Q35_DEV double row_lane64(double x, int l) {
  const i32x2 u = __builtin_bit_cast(i32x2, x);
  return __builtin_bit_cast(double, i32x2{__builtin_amdgcn_readlane(u[0], l), __builtin_amdgcn_readlane(u[1], l)});
}
Q35_DEV double wave_sum64(double v) {
  v += row_ror64<8>(v);
  v += row_ror64<4>(v);
  v += row_ror64<2>(v);
  v += row_ror64<1>(v);
  return (row_lane64(v, 0) + row_lane64(v, 16)) + (row_lane64(v, 32) + row_lane64(v, 48));
}

// Between two projections of the batched step: row m of h gets the residual projection's K splits
// (part_0 + part_1 + ..., then h; NS of them, 0: none, -1: n, in groups of 16), and y the RMSNorm of the
// new row, y = h * rsqrt(mean(h^2) + eps) * (1 + w).  The sums are 64-bit, as those of the step's
// other launch sequence (fixed point) are.  A row whose sum of squares is not finite or reaches 2^31
// raises kWsErrRange.
// A block is a row, a thread 4 columns, so all loads of the row are one memory round trip, which with
// the launch is what the kernel takes (16 rows of 2048, 12 / 8 splits: 4.7 / 4.5 us; with 256 threads and
// f32 sums 5.0, the step at 16 rows 1635 -> 1613 us).
constexpr int kRowMaxK = 4096;
template <int NS>
__global__ __launch_bounds__(kRowMaxK / 4) void rms_step_kernel(float* h, int K, const float* w, float eps, float* y,
                                                                const float* part, int n, uint32_t* err) {
  constexpr int G = NS > 0 ? NS : 16;
  __shared__ double sh[kRowMaxK / 256];
  const int tid = threadIdx.x, k = min(4 * tid, K - 4);  // (threads past the row repeat its end)
  const bool in = 4 * tid < K;
  float* hr = h + (int64_t)blockIdx.x * K + k;
  q35_f32x4 v = *(const Q35_GLOBAL q35_f32x4*)hr;
  const q35_f32x4 wv = *(const Q35_GLOBAL q35_f32x4*)(w + k);
  if (NS != 0) {
    const float* pr = part + (int64_t)blockIdx.x * K + k;
    const int64_t stride = (int64_t)gridDim.x * K;
    double t[4] = {0, 0, 0, 0};
    for (int s0 = 0; s0 < (NS > 0 ? 1 : n); s0 += G) {
      q35_f32x4 p[G];
#pragma unroll
      for (int u = 0; u < G; ++u)
        p[u] = *(const Q35_GLOBAL q35_f32x4*)(pr + (NS > 0 ? u : min(s0 + u, n - 1)) * stride);
#pragma unroll
      for (int u = 0; u < G; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) t[j] += (NS > 0 || s0 + u < n) ? (double)p[u][j] : 0;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (float)(t[j] + v[j]);
    if (in) *(Q35_GLOBAL q35_f32x4*)hr = v;
  }
  double ss = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) ss += (double)v[j] * (double)v[j];
  ss = wave_sum64(in ? ss : 0);
  if ((tid & 63) == 0) sh[tid >> 6] = ss;
  __syncthreads();
  ss = 0;
  for (int i = 0; i < (int)blockDim.x >> 6; ++i) ss += sh[i];
  const float sf = (float)ss;
  if (tid == 0 && !fx_addable(sf))
    __hip_atomic_fetch_or((Q35_GLOBAL uint32_t*)err, kWsErrRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const float r = rsqrt_f(sf * rcp_f((float)K) + eps);
  if (in) {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (v[j] * r) * (1.0f + wv[j]);
    *(Q35_GLOBAL q35_f32x4*)(y + (int64_t)blockIdx.x * K + k) = v;
  }
}

Q35_DEV void block_argmax256(float& v, int& i, float* shv, int* shi, const ArgOrder& o) {
  wave_argmax(v, i, o);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) { shv[wid] = v; shi[wid] = i; }
  __syncthreads();
  v = shv[0]; i = shi[0];
#pragma unroll
  for (int w = 1; w < 4; ++w)
    if (argmax_better(shv[w], shi[w], v, i, o)) { v = shv[w]; i = shi[w]; }
}

// Block (b, g) reduces values [g*span, (g+1)*span) of logits row b to one partial.
__global__ __launch_bounds__(kBT) void batch_argmax_part_kernel(const float* logits, int V, int G, int span,
                                                               float* pv, int32_t* pi, const ArgOrder ord) {
  __shared__ float shv[4];
  __shared__ int shi[4];
  const int b = blockIdx.x / G, g = blockIdx.x % G;
  const float* row = logits + (int64_t)b * V;
  const int lo = g * span, hi = min(V, lo + span);
  float v = -INFINITY;
  int ix = INT_MAX;
  for (int i = lo + threadIdx.x; i < hi; i += kBT) {
    const float x = row[i];
    if (argmax_better(x, i, v, ix, ord)) { v = x; ix = i; }
  }
  block_argmax256(v, ix, shv, shi, ord);
  if (threadIdx.x == 0) {
    pv[blockIdx.x] = v;
    pi[blockIdx.x] = ix;
  }
}

// Block b: the row's argmax from its G partials -> token[b], hist[b][pos[b]], pos[b] + 1.
__global__ __launch_bounds__(kBT) void batch_argmax_final_kernel(const float* pv, const int32_t* pi, int G,
                                                                int32_t* token, int32_t* pos, int32_t* hist, int ldh,
                                                                const ArgOrder ord) {
  __shared__ float shv[4];
  __shared__ int shi[4];
  const int b = blockIdx.x;
  float v = -INFINITY;
  int ix = INT_MAX;
  for (int g = threadIdx.x; g < G; g += kBT)
    if (argmax_better(pv[b * G + g], pi[b * G + g], v, ix, ord)) { v = pv[b * G + g]; ix = pi[b * G + g]; }
  block_argmax256(v, ix, shv, shi, ord);
  if (threadIdx.x == 0) {
    const int tok = ix == INT_MAX ? 0 : ix;
    const int p = pos[b];
    token[b] = tok;
    hist[(int64_t)b * ldh + p] = tok;
    pos[b] = p + 1;
  }
}

}  // namespace

int batch_embed_f32_launch(const int8_t* q, const float* s, int D, const int32_t* token, const int32_t* prompt, int ldp,
                           const int32_t* plen, const int32_t* pos, float* h, fx_t* ss, fx_t* zero_ptr, int64_t zero_n,
                           uint32_t* err, int B, hipStream_t st) {
  hipLaunchKernelGGL(batch_embed_f32_kernel, dim3(B), dim3(kBT), 0, st, q, s, D, token, prompt, ldp, plen, pos, h, ss,
                     zero_ptr, zero_n, err);
  Q35_HIP_TRY(hipGetLastError());
  return Q35_OK;
}

int batch_embed_launch(const int8_t* q, const float* s, int D, const int32_t* token, const int32_t* prompt, int ldp,
                       const int32_t* plen, const int32_t* pos, fx_t* h, int B, hipStream_t st) {
  const int gx = std::min((D + kBT - 1) / kBT, 8);
  hipLaunchKernelGGL(batch_embed_kernel, dim3(gx, B), dim3(kBT), 0, st, q, s, D, token, prompt, ldp, plen, pos, h);
  Q35_HIP_TRY(hipGetLastError());
  return Q35_OK;
}

int rms_step_launch(float* h, int M, int K, const float* w, float eps, float* y, const float* part, int nsplit,
                    uint32_t* err, hipStream_t st) {
  if (M < 1 || K < 4 || K % 4 || K > kRowMaxK || nsplit < 0 || (nsplit > 0 && !part))
    return fail(Q35_E_SHAPE, "rms_step: rows of up to 4096 columns, a multiple of 4");
  using Fn = void (*)(float*, int, const float*, float, float*, const float*, int, uint32_t*);
  static constexpr Fn fn[] = {rms_step_kernel<0>,  rms_step_kernel<1>,  rms_step_kernel<2>,  rms_step_kernel<3>,
                              rms_step_kernel<4>,  rms_step_kernel<5>,  rms_step_kernel<6>,  rms_step_kernel<7>,
                              rms_step_kernel<8>,  rms_step_kernel<9>,  rms_step_kernel<10>, rms_step_kernel<11>,
                              rms_step_kernel<12>, rms_step_kernel<13>, rms_step_kernel<14>, rms_step_kernel<15>,
                              rms_step_kernel<16>, rms_step_kernel<-1>};
  hipLaunchKernelGGL(fn[std::min(nsplit, 17)], dim3(M), dim3((K / 4 + 63) / 64 * 64), 0, st, h, K, w, eps, y, part, nsplit,
                     err);
  Q35_HIP_TRY(hipGetLastError());
  return Q35_OK;
}

int batch_argmax_groups(int V) { return std::max(1, std::min(64, (V + 4095) / 4096)); }

int batch_argmax_launch(const float* logits, int V, int B, float* pv, int32_t* pi, int32_t* token, int32_t* pos,
                        int32_t* hist, int ldh, hipStream_t st) {
  const int G = batch_argmax_groups(V), span = (V + G - 1) / G;
  const ArgOrder ord = make_arg_order(V);
  hipLaunchKernelGGL(batch_argmax_part_kernel, dim3(B * G), dim3(kBT), 0, st, logits, V, G, span, pv, pi, ord);
  Q35_HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL(batch_argmax_final_kernel, dim3(B), dim3(kBT), 0, st, pv, pi, G, token, pos, hist, ldh, ord);
  Q35_HIP_TRY(hipGetLastError());
  return Q35_OK;
}

}  // namespace q35
