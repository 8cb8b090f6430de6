// Gated GQA attention for one decode token (text_modules.rs:842-944): per-head q/k RMSNorm
// (1+w), partial RoPE on the first rot dims (rotate_half, :739-774), K/V append at the
// current position, softmax(q K^T / sqrt(d)) V over the cache with GQA (q head h reads kv
// head h / (nh/nkv), repeat_kv :776-792) and the sigmoid output gate (:936).
//
// Split-T ("flash decoding") in two kernels:
//  * chunk kernel, block (b, kv head g, chunk c) over `chunk` cached tokens for the rep = nh/nkv
//    query heads of g, so each K/V row is read once for all of them.  Wave w takes 4 tokens of every
//    16, one per 16-lane row; lane j of a row owns dims 4 j + 64 i (i < 4) of its token, so a score is
//    16 multiply-adds and 4 row rotations for 4 tokens at once (with a whole wave on one token the
//    64-lane sums were most of the kernel's vector work).  The next 4 tokens' rows are requested
//    before the current ones are computed.  Each 16-lane row keeps its own online softmax (running
//    max, sum and P.V per head in registers); rows and waves are combined at the end.  A block whose
//    chunk is the only one writes the gated output; otherwise it publishes (max, sum, o[rep][256]).
//    Bound: the K/V stream.  16 rows over 8192-token caches at mixed positions (335 MB, both kernels):
//    91.2 -> 63.0 us, 5.3 TB/s.
//  * merge kernel, block (b, query head h, 64-dim slice): chunk weights 2^(m_c - M) in LDS (the
//    maxima are kept in log2 units), 4 threads per dim each summing a quarter of the chunks (16
//    loads in flight), then the gate.
// The grids cover tmax, so a captured graph stays valid as the position advances; blocks past
// the current length exit at once.  A position outside [0, tmax) is reported through the
// workspace's error word and its row is left untouched.
#include "q35_internal.h"

namespace q35 {

namespace {

constexpr int kThreads = 256;
constexpr int kNW = kThreads / 64;
constexpr int kHd = 256;
constexpr int kMaxRep = 4;
constexpr int kMinChunk = 16;
constexpr int kMaxChunk = 512;     // tokens per block
constexpr int kMaxChunks = 1024;   // chunks per (b, kv head): the merge keeps their weights in LDS
constexpr int kMaxTokens = 262144; // longest cache
constexpr int kStep = 4 * kNW;         // tokens per block iteration

struct AttnArgs {
  AttnCall c;
  float scale;
  int32_t chunk, nchunk;
  uint32_t* counters;  // counters[kWsErrWord]: the sticky error word
  float* part_ml;      // [B*nkv][nchunk][2][kMaxRep]
  float* part_o;       // [B*nkv][nchunk][kMaxRep][hd]
};

Q35_DEV float4 ld4(const float* f, const fx_t* x, size_t i) {
  if (x) return make_float4(from_fx(x[i]), from_fx(x[i + 1]), from_fx(x[i + 2]), from_fx(x[i + 3]));
  return *reinterpret_cast<const float4*>(f + i);
}
Q35_DEV float ld1(const float* f, const fx_t* x, size_t i) { return x ? from_fx(x[i]) : f[i]; }

// a summed over lanes l and l ^ 32 in the lower half, b in the upper half (v_permlane32_swap)
Q35_DEV float add_swap32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// a summed over lanes l and l ^ 16 in even 16-lane rows, b in odd rows (v_permlane16_swap)
Q35_DEV float add_swap16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

Q35_DEV bool pos_ok(const AttnArgs& A, int b, int* pos) {
  *pos = A.c.pos[b];
  return *pos >= 0 && *pos < A.c.tmax;
}

__global__ __launch_bounds__(kThreads, 2) void attn_chunk_kernel(const AttnArgs A) {
  const AttnCall& a = A.c;
  __shared__ __align__(16) float qn[kMaxRep][kHd];
  __shared__ __align__(16) float kn[kHd];
  __shared__ __align__(16) float vn[kHd];
  __shared__ float rtmp[kMaxRep + 1][kHd];
  __shared__ __align__(16) float wo[kNW][kMaxRep][kHd];
  __shared__ float wm[kNW][kMaxRep], wl[kNW][kMaxRep];

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int c = blockIdx.x % A.nchunk;
  const int g = (blockIdx.x / A.nchunk) % a.nkv;
  const int b = blockIdx.x / (A.nchunk * a.nkv);
  const int rep = a.nh / a.nkv;
  int pos;
  if (!pos_ok(A, b, &pos)) {  // no cache row or rotary row exists for it: report, touch nothing
    if (tid == 0 && c == 0 && g == 0) ws_raise(A.counters, kWsErrPos);
    return;
  }
  const int T = pos + 1;
  const int nact = (T + A.chunk - 1) / A.chunk;
  if (c >= nact) return;
  const int t0 = c * A.chunk;
  const int len = min(A.chunk, T - t0);
  const bool has_new = (c == nact - 1);
  const size_t cache_off = (((size_t)b * a.nkv + g) * a.tmax) * kHd;
  const float* Kc = a.kc + cache_off;
  const float* Vc = a.vc + cache_off;
  // iteration it: the lane's token t0 + 16 it + 4 wid + tg; tokens at or past pos (the new one) are
  // not read (rows clamped into the cache, masked when used).  Two register buffers, so the
  // iteration loop is unrolled by two.
  const int j = lane & 15, tg = lane >> 4;
  const int nit = (len + kStep - 1) / kStep;
  q35_f32x4 k0b[4], v0b[4], k1b[4], v1b[4];
  auto load_it = [&](int it, q35_f32x4 (&kb)[4], q35_f32x4 (&vb)[4]) {
    const int t = max(0, min(t0 + kStep * it + 4 * wid + tg, pos - 1));
    const float* kr = Kc + (size_t)t * kHd + 4 * j;
    const float* vr = Vc + (size_t)t * kHd + 4 * j;
#pragma unroll
    for (int i = 0; i < 4; ++i) kb[i] = __builtin_nontemporal_load((const Q35_GLOBAL q35_f32x4*)(kr + 64 * i));
#pragma unroll
    for (int i = 0; i < 4; ++i) vb[i] = __builtin_nontemporal_load((const Q35_GLOBAL q35_f32x4*)(vr + 64 * i));
  };
  load_it(0, k0b, v0b);

  // q heads (wave w -> head g*rep + w), plus k/v of the new token in the chunk holding it
  for (int w = wid; w < rep + (has_new ? 2 : 0); w += kNW) {
    const int d = 4 * lane;
    if (w < rep) {
      const int hq = g * rep + w;
      const float4 v = ld4(a.qg, a.qg_f, (size_t)b * a.ld_qg + (size_t)hq * 2 * kHd + d);
      const float r = rsqrt_f(wave_sum(v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w) / (float)kHd + a.eps);
      qn[w][d + 0] = (v.x * r) * (1.0f + a.qnw[d + 0]);
      qn[w][d + 1] = (v.y * r) * (1.0f + a.qnw[d + 1]);
      qn[w][d + 2] = (v.z * r) * (1.0f + a.qnw[d + 2]);
      qn[w][d + 3] = (v.w * r) * (1.0f + a.qnw[d + 3]);
    } else if (w == rep) {
      const float4 v = ld4(a.k, a.k_f, (size_t)b * a.ld_kv + (size_t)g * kHd + d);
      const float r = rsqrt_f(wave_sum(v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w) / (float)kHd + a.eps);
      kn[d + 0] = (v.x * r) * (1.0f + a.knw[d + 0]);
      kn[d + 1] = (v.y * r) * (1.0f + a.knw[d + 1]);
      kn[d + 2] = (v.z * r) * (1.0f + a.knw[d + 2]);
      kn[d + 3] = (v.w * r) * (1.0f + a.knw[d + 3]);
    } else {
      *reinterpret_cast<float4*>(&vn[d]) = ld4(a.v, a.v_f, (size_t)b * a.ld_kv + (size_t)g * kHd + d);
    }
  }
  __syncthreads();
  // RoPE on dims [0, rot): x' = x*cos + rotate_half(x)*sin (computed into rtmp, then copied)
  const int half = a.rot / 2;
  const float* cs = a.rcos + (size_t)pos * a.rot;
  const float* sn = a.rsin + (size_t)pos * a.rot;
  const int nrot_heads = rep + (has_new ? 1 : 0);
  for (int e = tid; e < nrot_heads * a.rot; e += kThreads) {
    const int hh = e / a.rot, i = e % a.rot;
    const float* src = (hh < rep) ? qn[hh] : kn;
    const float rh = (i < half) ? -src[i + half] : src[i - half];
    rtmp[hh][i] = src[i] * cs[i] + rh * sn[i];
  }
  __syncthreads();
  for (int e = tid; e < nrot_heads * a.rot; e += kThreads) {
    const int hh = e / a.rot, i = e % a.rot;
    if (hh < rep) qn[hh][i] = rtmp[hh][i];
    else kn[i] = rtmp[hh][i];
  }
  __syncthreads();
  if (has_new) {  // append (post-RoPE k, raw v) at row `pos`
    a.kc[cache_off + (size_t)pos * kHd + tid] = kn[tid];
    a.vc[cache_off + (size_t)pos * kHd + tid] = vn[tid];
  }

  q35_f32x4 q4[kMaxRep][4];
#pragma unroll
  for (int h = 0; h < kMaxRep; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i) q4[h][i] = *(const q35_f32x4*)&qn[min(h, rep - 1)][4 * j + 64 * i];
  // online softmax per head and 16-lane row: running max m, sum l, and acc = sum p v (the lane's dims)
  float m[kMaxRep], l[kMaxRep];
  q35_f32x4 acc[kMaxRep][4];
#pragma unroll
  for (int h = 0; h < kMaxRep; ++h) {
    m[h] = -INFINITY;
    l[h] = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[h][i] = q35_f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // Scores are kept in log2 units (scale * log2 e folded in) so that every exponential is one
  // hardware exp2; a head's sums are rescaled only when a token of the wave raises a maximum.
  const float sl2 = A.scale * 1.44269504088896341f;
  auto compute = [&](int it, q35_f32x4 (&kb)[4], q35_f32x4 (&vb)[4]) {
    const int t = t0 + kStep * it + 4 * wid + tg;
    if (has_new && kStep * it + 4 * wid + 4 > pos - t0) {  // (uniform) the new token may be among these
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const q35_f32x4 kx = *(const q35_f32x4*)&kn[4 * j + 64 * i], vx = *(const q35_f32x4*)&vn[4 * j + 64 * i];
        kb[i] = t == pos ? kx : kb[i];
        vb[i] = t == pos ? vx : vb[i];
      }
    }
    const bool in = t < t0 + len;
#pragma unroll
    for (int h = 0; h < kMaxRep; ++h) {
      if (h >= rep) break;
      q35_f32x4 d = q4[h][0] * kb[0];
#pragma unroll
      for (int i = 1; i < 4; ++i) d += q4[h][i] * kb[i];
      float s = (d[0] + d[1]) + (d[2] + d[3]);
      s += row_ror<8>(s);
      s += row_ror<4>(s);
      s += row_ror<2>(s);
      s += row_ror<1>(s);
      s = in ? s * sl2 : -INFINITY;
      const float mn = fmaxf(m[h], s);
      if (__ballot(mn > m[h])) {
        const float al = m[h] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[h] - mn);
        l[h] *= al;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[h][i] *= al;
        m[h] = mn;
      }
      const float p = s == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(s - mn);
      l[h] += p;
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[h][i] += p * vb[i];
    }
  };
  // the next iteration's rows are requested before the current ones are computed
  for (int it = 0; it < nit; it += 2) {
    if (it + 1 < nit) load_it(it + 1, k1b, v1b);
    compute(it, k0b, v0b);
    if (it + 1 >= nit) break;
    if (it + 2 < nit) load_it(it + 2, k0b, v0b);
    compute(it + 1, k1b, v1b);
  }
  // the wave's 4 rows: a common maximum, then the lane swaps add the rows and leave row tg with head
  // tg (swap by 32 lanes pairs heads h and h + 2, by 16 lanes heads 0 and 1 of what is left)
  float mw[kMaxRep], lw[kMaxRep];
#pragma unroll
  for (int h = 0; h < kMaxRep; ++h) {
    float M = fmaxf(m[h], __shfl_xor(m[h], 16));
    M = fmaxf(M, __shfl_xor(M, 32));
    const float f = m[h] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[h] - M);
    float L = l[h] * f;
    L += __shfl_xor(L, 16);
    L += __shfl_xor(L, 32);
    mw[h] = M;
    lw[h] = L;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[h][i] *= f;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    q35_f32x4 r;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x0 = add_swap32(acc[0][i][e], acc[2][i][e]), x1 = add_swap32(acc[1][i][e], acc[3][i][e]);
      r[e] = add_swap16(x0, x1);
    }
    *(q35_f32x4*)&wo[wid][tg][4 * j + 64 * i] = r;
  }
  if (lane == 0) {
#pragma unroll
    for (int h = 0; h < kMaxRep; ++h) { wm[wid][h] = mw[h]; wl[wid][h] = lw[h]; }
  }
  __syncthreads();
  const int grpi = b * a.nkv + g;
  float* pml = A.part_ml + ((size_t)grpi * A.nchunk + c) * 2 * kMaxRep;
  float* po = A.part_o + ((size_t)grpi * A.nchunk + c) * kMaxRep * kHd;
#pragma unroll
  for (int h = 0; h < kMaxRep; ++h) {
    if (h >= rep) break;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kNW; ++w) M = fmaxf(M, wm[w][h]);
    float L = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < kNW; ++w) {
      const float e = (wm[w][h] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f(wm[w][h] - M);
      L += wl[w][h] * e;
      o += wo[w][h][tid] * e;
    }
    if (nact == 1) {  // the only chunk: finish here
      const int hq = g * rep + h;
      const float gv = ld1(a.qg, a.qg_f, (size_t)b * a.ld_qg + (size_t)hq * 2 * kHd + kHd + tid);
      a.out[(size_t)b * a.ld_out + (size_t)hq * kHd + tid] = (o / L) * sigmoid_f(gv);
    } else {
      po[h * kHd + tid] = o;
      if (tid == 0) { pml[h] = M; pml[kMaxRep + h] = L; }
    }
  }
}

// Block (b, query head hq, 64-dim slice ds): merges the chunk partials of that slice.
__global__ __launch_bounds__(kThreads) void attn_merge_kernel(const AttnArgs A) {
  const AttnCall& a = A.c;
  __shared__ float wts[kMaxChunks];
  __shared__ float red[kNW][64];
  __shared__ float shm[kNW], shl[kNW];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int nds = kHd / 64;
  const int ds = blockIdx.x % nds;
  const int hq = (blockIdx.x / nds) % a.nh;
  const int b = blockIdx.x / (nds * a.nh);
  const int rep = a.nh / a.nkv, g = hq / rep, hr = hq % rep;
  int pos;
  if (!pos_ok(A, b, &pos)) return;  // reported by the chunk kernel
  const int nact = (pos + A.chunk) / A.chunk;
  if (nact <= 1) return;  // the chunk kernel wrote the output
  const int grpi = b * a.nkv + g;
  const float* ml = A.part_ml + (size_t)grpi * A.nchunk * 2 * kMaxRep;
  const float* og = A.part_o + (size_t)grpi * A.nchunk * kMaxRep * kHd;
  // chunk maxima -> M, weights w_c = exp(m_c - M) (LDS) and L = sum l_c w_c
  float mx = -INFINITY;
  for (int cc = tid; cc < nact; cc += kThreads) mx = fmaxf(mx, ml[(size_t)cc * 2 * kMaxRep + hr]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if (lane == 0) shm[wid] = mx;
  __syncthreads();
  const float M = fmaxf(fmaxf(shm[0], shm[1]), fmaxf(shm[2], shm[3]));
  float ls = 0.f;
  for (int cc = tid; cc < nact; cc += kThreads) {
    const float w = __builtin_amdgcn_exp2f(ml[(size_t)cc * 2 * kMaxRep + hr] - M);  // maxima in log2 units
    wts[cc] = w;
    ls += ml[(size_t)cc * 2 * kMaxRep + kMaxRep + hr] * w;
  }
  ls = wave_sum(ls);
  if (lane == 0) shl[wid] = ls;
  __syncthreads();
  const float L = (shl[0] + shl[1]) + (shl[2] + shl[3]);
  // thread (part = wid, dim = lane): chunks part, part + 4, ... , 16 loads in flight
  const int d = ds * 64 + lane;
  const float* src = og + (size_t)hr * kHd + d;
  float o = 0.f;
  for (int c0 = wid; c0 < nact; c0 += kNW * 16) {
    float v[16], w[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int cc = min(c0 + kNW * j, nact - 1);  // clamped; masked below
      v[j] = src[(size_t)cc * kMaxRep * kHd];
      w[j] = wts[cc];
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) o += (c0 + kNW * j < nact) ? v[j] * w[j] : 0.f;
  }
  red[wid][lane] = o;
  __syncthreads();
  if (tid < 64) {
    const float s = (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
    const float gv = ld1(a.qg, a.qg_f, (size_t)b * a.ld_qg + (size_t)hq * 2 * kHd + kHd + d);
    a.out[(size_t)b * a.ld_out + (size_t)hq * kHd + d] = (s / L) * sigmoid_f(gv);
  }
}

// Tokens per chunk: about 512 chunk blocks over the (b, kv head, tmax) work, 16 .. 512 tokens: two
// blocks fit a CU, and a block's start (norms, rotary, first rows) is paid once per chunk (the 335 MB
// case above with at most 64 / 128 / 256 / 512 tokens: 86 / 78 / 70.5 / 63 us).
int pick_chunk(int32_t B, int32_t nkv, int32_t tmax) {
  const long long work = (long long)B * nkv * tmax;
  long long ch = (work + 511) / 512;
  ch = (ch + kMinChunk - 1) / kMinChunk * kMinChunk;
  if (ch < kMinChunk) ch = kMinChunk;
  if (ch > kMaxChunk) ch = kMaxChunk;
  return (int)ch;
}

struct AttnLayout {
  int chunk, nchunk;
  size_t cnt_bytes, ml_bytes, o_bytes;
};

AttnLayout attn_layout(int32_t B, int32_t nkv, int32_t hd, int32_t tmax) {
  AttnLayout L;
  L.chunk = pick_chunk(B, nkv, tmax);
  L.nchunk = (tmax + L.chunk - 1) / L.chunk;
  const size_t groups = (size_t)B * nkv;
  L.cnt_bytes = kCounterBytes;
  L.ml_bytes = (groups * L.nchunk * 2 * kMaxRep * 4 + 255) & ~(size_t)255;
  L.o_bytes = (groups * L.nchunk * kMaxRep * (size_t)hd * 4 + 255) & ~(size_t)255;
  return L;
}

}  // namespace

size_t attn_ws_bytes(int32_t B, int32_t nh, int32_t nkv, int32_t hd, int32_t tmax) {
  (void)nh;
  AttnLayout L = attn_layout(B, nkv, hd, tmax);
  return L.cnt_bytes + L.ml_bytes + L.o_bytes;
}

int attn_launch(const AttnCall& c, void* ws, size_t ws_bytes, hipStream_t st) {
  if (!ws || ws_bytes < kCounterBytes) return fail(Q35_E_WS, "attention: workspace too small");
  return attn_launch_split(c, ws_counters(ws), ws_scratch(ws), ws_bytes - kCounterBytes, st);
}

int attn_launch_split(const AttnCall& c, uint32_t* counters, char* scratch, size_t scratch_bytes, hipStream_t st) {
  if ((!c.qg && !c.qg_f) || (!c.k && !c.k_f) || (!c.v && !c.v_f) || !c.qnw || !c.knw || !c.rcos || !c.rsin || !c.kc || !c.vc || !c.pos || !c.out)
    return fail(Q35_E_ARG, "attention: null pointer");
  if (c.hd != kHd) return fail(Q35_E_SHAPE, "attention: head_dim must be 256");
  if (c.nkv < 1 || c.nh % c.nkv != 0 || c.nh / c.nkv > kMaxRep)
    return fail(Q35_E_SHAPE, "attention: heads must be a multiple of kv heads, ratio <= 4");
  if (c.rot <= 0 || c.rot > c.hd || (c.rot % 2) != 0) return fail(Q35_E_SHAPE, "attention: bad rotary dim");
  if (c.B < 1 || c.tmax < 1) return fail(Q35_E_SHAPE, "attention: B and tmax must be >= 1");
  if ((size_t)c.B * c.nkv * c.tmax * c.hd > (size_t)1 << 40) return fail(Q35_E_SHAPE, "attention: cache too large");
  AttnLayout L = attn_layout(c.B, c.nkv, c.hd, c.tmax);
  if (!counters || !scratch || scratch_bytes < L.ml_bytes + L.o_bytes) return fail(Q35_E_WS, "attention: workspace too small");
  if (c.tmax > kMaxTokens || L.nchunk > kMaxChunks) return fail(Q35_E_SHAPE, "attention: tmax too large for one merge");
  AttnArgs A;
  A.c = c;
  A.scale = (float)(1.0 / sqrt((double)c.hd));
  A.chunk = L.chunk; A.nchunk = L.nchunk;
  A.counters = counters;
  A.part_ml = reinterpret_cast<float*>(scratch);
  A.part_o = reinterpret_cast<float*>(scratch + L.ml_bytes);
  hipLaunchKernelGGL(attn_chunk_kernel, dim3(c.B * c.nkv * L.nchunk), dim3(kThreads), 0, st, A);
  Q35_HIP_TRY(hipGetLastError());
  if (L.nchunk > 1) {
    hipLaunchKernelGGL(attn_merge_kernel, dim3(c.B * c.nh * (kHd / 64)), dim3(kThreads), 0, st, A);
    Q35_HIP_TRY(hipGetLastError());
  }
  return Q35_OK;
}

}  // namespace q35
