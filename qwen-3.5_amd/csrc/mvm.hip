// Multi-row Q8F matvec (2..32 rows) on the bf16 matrix cores for the reference's projection
// layouts (KN and its tile-major form): the layer calls of a batch of sequences and
// multi-row q8_gemv (text_modules.rs:497-508, :855-893, :1003-1005; kernels.rs:53-92).
//
// What bounds it: the weight stream (each weight is read once for all rows).  The
// one-row kernel's vector-ALU form multiplies every weight by every row, re-reads the weights
// for each 8 rows and adds every column of every row with a 64-bit atomic; at 24 rows the MLP
// spent 193 us on 38 MB of weights.  Here the products go to v_mfma_f32_16x16x32_bf16 and the
// K splits leave plain f32 partials that a second kernel adds in split order.  Measured, 2B layer
// calls: MLP at 24 rows 192.6 -> 31.8 us, DeltaNet at 9 rows 85.6 -> 27.8, the projections around the
// attention of 16 rows 104 -> 24, q8_gemv 2048 x 6144 at 8 rows 35.0 -> 8.6.
//
// Arithmetic (f32 products): the int8 weight is exact in bf16; its block scale multiplies the input,
// y = x * s (f32), and y is carried whole, as three bf16 values (8 bits each): q * y is exact before
// the f32 accumulation, whatever the range of the row.  The small values' products have an
// accumulator of their own, added at the end (the matrix instruction's own additions do not always
// round to nearest), so a single product comes out as the rounded f32 product.
//
// Split: a wave owns one 64-column block x NS * 32 rows of K and issues all of its loads (a dword
// of 4 columns per row and lane; its x rows; its scales) before the first use, so the launch's
// whole weight range is in flight at once.  Lane (g, c) = (lane / 16, lane % 16) takes columns
// 4 c .. 4 c + 3 of rows 8 g + j, j < 8, of a 32-row step: A operand nt holds column 4 c + nt,
// which needs one v_perm per pair of rows, and no transposition of the stored layout.  The NW
// waves of a block split K and add their results through LDS.
#include "q35_internal.h"

#include <algorithm>

namespace q35 {
namespace {

typedef q35_f32x4 f4;
typedef q35_b8 b8;

constexpr int kAuxRows = 128;  // K rows per gate-projection block
constexpr int kAuxLd = 132;    // its padded f32 x row in LDS

enum { LAY_KN = 0, LAY_SO = 1 };  // KN / tile-major, or the batched decoder's stream-order records
struct MvmSegArg {
  const int8_t* q;
  const float* s;
  int32_t ldq, lds;   // bytes / scales per row of K
  int32_t tiled, cb0; // cb0: first column block of the segment in the launch
};
struct MvmArgs {
  MvmSegArg seg[kMvmMaxSeg];
  int32_t nseg, K, M, ncb, nsplit, naux;
  const float* x; int32_t ldx;
  const float* z; int32_t ldz; const float* pw; float eps;  // gated RMSNorm over 128-wide heads
  float* part;                                              // [nsplit][M][64 ncb]
  const float* aux_wb; const float* aux_wa; int32_t aux_nh; float* aux_part;  // [naux][M][2 nh]
};

Q35_DEV f4 ld4(const float* p) { return *(const Q35_GLOBAL f4*)p; }

// bf16 operand of column byte NT of the 8 rows d[0..7].
template <int NT>
Q35_DEV b8 col8(const uint32_t (&d)[8]) {
  q35_u32x4 r;
#pragma unroll
  for (int j = 0; j < 4; ++j) r[j] = bf_pair(s8_of<NT>(d[2 * j]), s8_of<NT>(d[2 * j + 1]));
  return __builtin_bit_cast(b8, r);
}

// Gate projection (in_proj_b | in_proj_a, f32 [K][nh] each, kernels.rs:174-247): block ab sums
// rows [128 ab, 128 ab + 128) of x . W for every row m; mvm_reduce adds the blocks in order and
// applies the activations.
template <int MT, int NW>
Q35_DEV void mvm_aux(const MvmArgs& a, int ab, float* xs) {
  constexpr int T = 64 * NW, RG = T / 32, RPG = kAuxRows / RG;  // row groups, rows of each
  const int t = threadIdx.x, k0 = ab * kAuxRows, klen = min(kAuxRows, a.K - k0);
  const int o = t & 31, rg = t >> 5, nh = a.aux_nh, no = 2 * nh;
  const float* W = o < nh ? a.aux_wb : a.aux_wa;
  const int oc = o < nh ? o : min(o - nh, nh - 1);
  float w[RPG];
#pragma unroll
  for (int i = 0; i < RPG; ++i) {
    const int r = rg * RPG + i;
    w[i] = ldg(W + (size_t)(k0 + min(r, klen - 1)) * nh + oc);
    if (r >= klen || o >= no) w[i] = 0.f;
  }
  for (int i = t; i < a.M * (kAuxRows / 4); i += T) {
    const int m = i / (kAuxRows / 4), k = (i % (kAuxRows / 4)) * 4;
    f4 v = f4{0.f, 0.f, 0.f, 0.f};
    if (k < klen) v = ld4(a.x + (size_t)m * a.ldx + k0 + k);
    *(f4*)(xs + m * kAuxLd + k) = v;
  }
  __syncthreads();
  float acc[16 * MT];
#pragma unroll
  for (int m = 0; m < 16 * MT; ++m) {
    acc[m] = 0.f;
    const float* xr = xs + min(m, a.M - 1) * kAuxLd + rg * RPG;
#pragma unroll
    for (int i = 0; i < RPG; ++i) acc[m] += xr[i] * w[i];
  }
  __syncthreads();  // the row groups' sums replace the x rows
#pragma unroll
  for (int m = 0; m < 16 * MT; ++m) xs[(rg * 16 * MT + m) * 33 + o] = acc[m];
  __syncthreads();
  for (int i = t; i < a.M * 32; i += T) {
    const int m = i >> 5, oo = i & 31;
    float v = 0.f;
#pragma unroll
    for (int r = 0; r < RG; ++r) v += xs[(r * 16 * MT + m) * 33 + oo];
    if (oo < no) a.aux_part[((size_t)ab * a.M + m) * no + oo] = v;
  }
}

template <int MT, int NS, int NW, bool GATED, int LAY>
__global__ __launch_bounds__(64 * NW) void mvm_kernel(const MvmArgs a) {
  constexpr int RW = 32 * NS;               // K rows per wave
  constexpr int LD = 68;                    // padded row of the reduction buffer
  constexpr int RED = NW * 16 * MT * LD;
  constexpr int AUX = (16 * MT * kAuxLd) > (2 * NW * 16 * MT * 33) ? 16 * MT * kAuxLd : 2 * NW * 16 * MT * 33;
  __shared__ __align__(16) float red[RED > AUX ? RED : AUX];
  __shared__ __align__(16) float scs[NW][RW];
  if ((int)blockIdx.x < a.naux) {
    mvm_aux<MT, NW>(a, (int)blockIdx.x, red);
    return;
  }
  // column blocks of one K split are neighbours on one XCD (blocks are dealt round-robin over
  // the 8 XCDs): they share the 128-byte lines of the row-major weights and scales
  const int nmain = a.ncb * a.nsplit, bid = (int)blockIdx.x - a.naux;
  const int q8 = nmain >> 3, r8 = nmain & 7, xcd = bid & 7;
  const int L = xcd * q8 + min(xcd, r8) + (bid >> 3);
  const int split = L / a.ncb, cb = L - split * a.ncb;
  MvmSegArg sg = a.seg[0];
#pragma unroll
  for (int i = 1; i < kMvmMaxSeg; ++i)
    if (i < a.nseg && cb >= a.seg[i].cb0) sg = a.seg[i];
  const int lcb = cb - sg.cb0;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 4, c = lane & 15;
  const int k0 = (split * NW + w) * RW;
  // tile-major: tile lcb / 4 starts at row (lcb / 4) * K of a 256-column matrix.  Stream order: per
  // 32-row step 2 KB, the lane's operands of column tiles 0, 1 at 16 lane and of 2, 3 at 1024 + 16
  // lane (column 16 nt + c there); scales [cb][K].
  const size_t trow = sg.tiled ? (size_t)(lcb >> 2) * a.K : 0;
  const int8_t* wb = LAY == LAY_SO ? sg.q + (size_t)lcb * a.K * 64 + 16 * lane
                                   : sg.q + trow * sg.ldq + (sg.tiled ? lcb & 3 : lcb) * 64 + 4 * c;
  const float* sb = LAY == LAY_SO ? sg.s + (size_t)lcb * a.K : sg.s + trow * sg.lds + (sg.tiled ? lcb & 3 : lcb);
  const int lds = LAY == LAY_SO ? 1 : sg.lds;

  // every load of the wave, issued in the order of use; rows past K repeat its last 8 (their y
  // is set to zero)
  float sv[(RW + 63) / 64];
#pragma unroll
  for (int i = 0; i < (RW + 63) / 64; ++i) sv[i] = ldg(sb + (size_t)min(k0 + 64 * i + lane, a.K - 1) * lds);
  f4 xv[NS][MT][2], zv[GATED ? NS : 1][MT][2], pv[GATED ? NS : 1][2];
  int kk[NS];
#pragma unroll
  for (int st = 0; st < NS; ++st) {
    kk[st] = min(k0 + 32 * st + 8 * g, a.K - 8);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const size_t m = (size_t)min(16 * mt + c, a.M - 1);  // rows past M repeat row M - 1 (never stored)
      xv[st][mt][0] = ld4(a.x + m * a.ldx + kk[st]);
      xv[st][mt][1] = ld4(a.x + m * a.ldx + kk[st] + 4);
      if constexpr (GATED) {
        zv[st][mt][0] = ld4(a.z + m * a.ldz + kk[st]);
        zv[st][mt][1] = ld4(a.z + m * a.ldz + kk[st] + 4);
      }
    }
    if constexpr (GATED) {
      pv[st][0] = ld4(a.pw + (kk[st] & 127));
      pv[st][1] = ld4(a.pw + (kk[st] & 127) + 4);
    }
  }
  uint32_t wv[NS][8];
#pragma unroll
  for (int st = 0; st < NS; ++st) {
    if constexpr (LAY == LAY_SO) {
      const int8_t* p = wb + (size_t)min(k0 + 32 * st, a.K - 32) * 64;
      const q35_u32x4 w0 = ldg16v_nt(p), w1 = ldg16v_nt(p + 1024);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        wv[st][j] = w0[j];
        wv[st][4 + j] = w1[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j)  // (64 bytes of a line: its other half belongs to the next column block,
                                   // so no non-temporal hint: 36.4 -> 33.6 us for the MLP at 24 rows)
        wv[st][j] = ldg((const uint32_t*)(wb + (size_t)(kk[st] + j) * sg.ldq));
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // (the scheduler would sink the loads to their uses)

  // the wave's scales through its own LDS rows (no other wave reads them)
#pragma unroll
  for (int i = 0; i < (RW + 63) / 64; ++i)
    if (RW % 64 == 0 || 64 * i + lane < RW) scs[w][64 * i + lane] = sv[i];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();

  if constexpr (GATED) {
    // RMSNormGated (text_modules.rs:91-100); the wave's 128 rows are one head
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      float ss = 0.f;
#pragma unroll
      for (int st = 0; st < NS; ++st)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j) ss += xv[st][mt][h][j] * xv[st][mt][h][j];
      ss += __shfl_xor(ss, 16);
      ss += __shfl_xor(ss, 32);
      const float r = rsqrt_f(ss * (1.0f / 128.0f) + a.eps);
#pragma unroll
      for (int st = 0; st < NS; ++st)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            xv[st][mt][h][j] = (pv[st][h][j] * (xv[st][mt][h][j] * r)) * silu_f(zv[st][mt][h][j]);
    }
  }

  // y = x * s in place
#pragma unroll
  for (int st = 0; st < NS; ++st) {
    const bool in = k0 + 32 * st < a.K;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f4 s4 = *(const f4*)&scs[w][32 * st + 8 * g + 4 * h];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int j = 0; j < 4; ++j) xv[st][mt][h][j] = in ? xv[st][mt][h][j] * s4[j] : 0.f;
    }
  }

  f4 acc[4][MT], accs[4][MT];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = accs[nt][mt] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int st = 0; st < NS; ++st) {
    b8 b[3][MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      uint32_t p[3][4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        split3(xv[st][mt][j >> 1][2 * (j & 1)], xv[st][mt][j >> 1][2 * (j & 1) + 1], p[2][j], p[1][j], p[0][j]);
#pragma unroll
      for (int q = 0; q < 3; ++q) b[q][mt] = __builtin_bit_cast(b8, q35_u32x4{p[q][0], p[q][1], p[q][2], p[q][3]});
    }
    b8 aw[4];
    if constexpr (LAY == LAY_SO) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) aw[nt] = s8_from(wv[st][2 * nt] ^ 0x80808080u, wv[st][2 * nt + 1] ^ 0x80808080u);  // (bytes q + 128)
    } else {
      aw[0] = col8<0>(wv[st]);
      aw[1] = col8<1>(wv[st]);
      aw[2] = col8<2>(wv[st]);
      aw[3] = col8<3>(wv[st]);
    }
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        accs[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aw[nt], b[0][mt], accs[nt][mt], 0, 0, 0);
        acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aw[nt], b[2][mt], acc[nt][mt], 0, 0, 0);
      }
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        accs[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aw[nt], b[1][mt], accs[nt][mt], 0, 0, 0);
  }
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] += accs[nt][mt];

  // lane holds column 16 g + 4 r + nt (stream order: 16 nt + 4 g + r) of row 16 mt + c in
  // acc[nt][mt][r]; the waves' sums meet in LDS and are added in wave order
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float* rr = &red[(w * 16 * MT + 16 * mt + c) * LD];
      if constexpr (LAY == LAY_SO) *(f4*)(rr + 16 * r + 4 * g) = acc[r][mt];
      else *(f4*)(rr + 16 * g + 4 * r) = f4{acc[0][mt][r], acc[1][mt][r], acc[2][mt][r], acc[3][mt][r]};
    }
  __syncthreads();
  const int ldp = 64 * a.ncb;
#pragma unroll
  for (int i = 0; i < 16 * MT * 16 / (64 * NW); ++i) {
    const int m = (tid >> 4) + 4 * NW * i, col = (tid & 15) * 4;
    f4 v = *(const f4*)&red[m * LD + col];
#pragma unroll
    for (int q = 1; q < NW; ++q) v += *(const f4*)&red[(q * 16 * MT + m) * LD + col];
    if (m < a.M) *(f4*)(a.part + ((size_t)split * a.M + m) * ldp + 64 * cb + col) = v;
  }
}

// Adds the K splits in split order, in 64 bits (the one-row path's sums are 64-bit fixed point).  A
// partial that is not finite or whose magnitude reaches 2^31 is dropped and raises kWsErrRange, the
// contract of those sums.  clear: zeros are left in the partials' place.  G splits are loaded at a time.
template <int G>
Q35_DEV f4 sum_splits(float* p, int nsplit, size_t stride, bool clear, bool& bad) {
  double t[4] = {0, 0, 0, 0};
  for (int s = 0; s < nsplit; s += G) {
    f4 v[G];
#pragma unroll
    for (int u = 0; u < G; ++u) v[u] = ld4(p + (size_t)min(s + u, nsplit - 1) * stride);
#pragma unroll
    for (int u = 0; u < G; ++u)
      if (s + u < nsplit) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const bool ok = fx_addable(v[u][j]);
          bad = bad || !ok;
          t[j] += ok ? (double)v[u][j] : 0;
        }
        if (clear) *(Q35_GLOBAL f4*)(p + (size_t)(s + u) * stride) = f4{0.f, 0.f, 0.f, 0.f};
      }
  }
  return f4{(float)t[0], (float)t[1], (float)t[2], (float)t[3]};
}

struct RedArgs {
  float* part; int32_t nsplit, M, N;  // partials [nsplit][M][N]
  float* y; int32_t ldy;
  int32_t swiglu;  // y[m][j] = up * silu(gate), gate columns [0, N/2), up [N/2, N)
  int32_t clear;   // the partials are zero again afterwards
  const float* aux; int32_t naux, nh; const float* alog; const float* dtb; float* bg;  // gates [M][2 nh]
  uint32_t* err;
};

// One float4 of outputs per thread; the last block's threads finish the gates.
template <int G>
__global__ __launch_bounds__(256) void mvm_reduce_kernel(const RedArgs a) {
  const int nq = (a.swiglu ? a.N / 2 : a.N) / 4;
  const int64_t nout = (int64_t)a.M * nq;
  const size_t stride = (size_t)a.M * a.N;
  bool bad = false;
  if (a.naux && blockIdx.x == gridDim.x - 1) {
    // beta = sigmoid(b); g = -exp(A_log) * softplus(a + dt_bias) (kernels.rs:228-244)
    const int no = 2 * a.nh;
    for (int i = threadIdx.x; i < a.M * no; i += 256) {
      const int m = i / no, o = i - m * no, h = o < a.nh ? o : o - a.nh;
      double vs = 0;
      for (int s = 0; s < a.naux; s += 8) {
        float t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] = ldg(a.aux + ((size_t)min(s + u, a.naux - 1) * a.M + m) * no + o);
#pragma unroll
        for (int u = 0; u < 8; ++u) vs += s + u < a.naux ? (double)t[u] : 0;
      }
      float v = (float)vs;
      if (!fx_addable(v)) {
        bad = true;
        v = 0.f;
      }
      if (o < a.nh) {
        v = sigmoid_f(v);
      } else {
        const float xg = v + ldg(a.dtb + h);
        const float pre = logf(expf(xg) + 1.0f);
        v = -expf(ldg(a.alog + h)) * (pre > 20.0f ? xg : pre);
      }
      stg(a.bg + (size_t)m * no + o, v);
    }
  } else {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < nout) {
      const int m = (int)(i / nq), j = (int)(i - (int64_t)m * nq) * 4;
      float* p = a.part + (size_t)m * a.N + j;
      f4 v = sum_splits<G>(p, a.nsplit, stride, a.clear, bad);
      if (a.swiglu) {
        const f4 up = sum_splits<G>(p + a.N / 2, a.nsplit, stride, a.clear, bad);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = up[r] * silu_f(v[r]);
      }
      *(f4*)(a.y + (size_t)m * a.ldy + j) = v;
    }
  }
  if (bad)
    __hip_atomic_fetch_or((Q35_GLOBAL uint32_t*)a.err, kWsErrRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct MvmPlan { int ns, nw, nsplit; };

// Rows of K per wave (64 or 128) and waves per block (2 or 4): the most rows per block that still
// give 384 blocks, one and a half per CU, so that few partials are written while every CU streams.  (A
// number and not the device's: the plan fixes the partials' size and a call's bits.)
MvmPlan mvm_plan(int ncb, int K, bool gated) {
  const int cand[3][2] = {{4, 4}, {4, 2}, {2, 2}};
  MvmPlan p{4, 2, 1};
  for (const auto& t : cand) {
    if (gated && t[0] != 4) break;  // a wave covers whole 128-wide heads
    p.ns = t[0];
    p.nw = t[1];
    const int kb = 32 * p.ns * p.nw;
    p.nsplit = (K + kb - 1) / kb;
    if ((int64_t)ncb * p.nsplit >= 384) break;
  }
  return p;
}

template <int MT, bool GATED, int LAY>
const void* mvm_fn(const MvmPlan& p) {
  if (p.ns == 4 && p.nw == 4) return (const void*)mvm_kernel<MT, 4, 4, GATED, LAY>;
  if (p.ns == 4) return (const void*)mvm_kernel<MT, 4, 2, GATED, LAY>;
  if constexpr (!GATED) return (const void*)mvm_kernel<MT, 2, 2, false, LAY>;
  return nullptr;
}
template <int LAY>
const void* mvm_pick(const MvmPlan& p, int M, bool gated) {
  if (M <= 16) return gated ? mvm_fn<1, true, LAY>(p) : mvm_fn<1, false, LAY>(p);
  return gated ? mvm_fn<2, true, LAY>(p) : mvm_fn<2, false, LAY>(p);
}

}  // namespace

size_t mvm_part_floats(int32_t M, int32_t K, int32_t N, bool gated) {
  return (size_t)mvm_plan(N / 64, K, gated).nsplit * std::min(M, kMvmRows) * N;
}
size_t mvm_aux_floats(int32_t M, int32_t K, int32_t nh) {
  return (size_t)((K + kAuxRows - 1) / kAuxRows) * std::min(M, kMvmRows) * 2 * nh;
}
bool mvm_ok(const float* x, int32_t ldx, int32_t K) {
  return K >= 64 && K % 32 == 0 && ldx % 4 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
}

int mvm_launch(const MvmCall& c, hipStream_t st) {
  if (c.M < 1 || c.M > kMvmRows || c.nseg < 1 || c.nseg > kMvmMaxSeg) return fail(Q35_E_SHAPE, "mvm: bad rows or segments");
  if (!mvm_ok(c.x, c.ldx, c.K)) return fail(Q35_E_ALIGN, "mvm: K % 32 and 16-byte aligned rows required");
  if ((!c.y && !c.nsplit_out) || !c.part || !c.err) return fail(Q35_E_ARG, "mvm: null pointer");
  const bool gated = c.z != nullptr;
  if (gated && (!c.pw || c.K % 128 || c.ldz % 4 || (reinterpret_cast<uintptr_t>(c.z) & 15) ||
                (reinterpret_cast<uintptr_t>(c.pw) & 15)))
    return fail(Q35_E_ALIGN, "mvm: gated rows");
  MvmArgs a{};
  int ncb = 0;
  for (int i = 0; i < c.nseg; ++i) {
    const MvmSeg& s = c.seg[i];
    if (!s.q || !s.s || s.N < 64 || s.N % 64) return fail(Q35_E_SHAPE, "mvm: N must be a positive multiple of 64");
    a.seg[i] = MvmSegArg{s.q, s.s, s.tiled ? 256 : s.N, s.tiled ? 4 : s.N / 64, s.tiled, ncb};
    ncb += s.N / 64;
  }
  const MvmPlan p = mvm_plan(ncb, c.K, gated);
  if ((size_t)p.nsplit * c.M * 64 * ncb > c.part_floats) return fail(Q35_E_WS, "mvm: workspace too small");
  a.nseg = c.nseg; a.K = c.K; a.M = c.M; a.ncb = ncb; a.nsplit = p.nsplit;
  a.x = c.x; a.ldx = c.ldx; a.z = c.z; a.ldz = c.ldz; a.pw = c.pw; a.eps = c.eps;
  a.part = c.part;
  RedArgs r{};
  if (c.aux_nh > 0) {
    if (2 * c.aux_nh > 32 || !c.aux_wb || !c.aux_wa || !c.aux_part || !c.bg) return fail(Q35_E_ARG, "mvm: gate projection");
    a.naux = (c.K + kAuxRows - 1) / kAuxRows;
    a.aux_wb = c.aux_wb; a.aux_wa = c.aux_wa; a.aux_nh = c.aux_nh; a.aux_part = c.aux_part;
    r.aux = c.aux_part; r.naux = a.naux; r.nh = c.aux_nh; r.alog = c.a_log; r.dtb = c.dt_bias; r.bg = c.bg;
  }
  const void* k = c.stream_order ? mvm_pick<LAY_SO>(p, c.M, gated) : mvm_pick<LAY_KN>(p, c.M, gated);
  void* params[] = {&a};
  Q35_HIP_TRY(hipLaunchKernel(k, dim3((unsigned)(a.naux + ncb * p.nsplit)), dim3(64 * p.nw), params, 0, st));
  Q35_HIP_TRY(hipGetLastError());
  if (c.nsplit_out) {
    *c.nsplit_out = p.nsplit;
    return Q35_OK;
  }
  r.part = c.part; r.nsplit = p.nsplit; r.M = c.M; r.N = 64 * ncb; r.y = c.y; r.ldy = c.ldy;
  r.swiglu = c.swiglu; r.clear = c.clear; r.err = c.err;
  const int64_t nout = (int64_t)c.M * (c.swiglu ? r.N / 2 : r.N) / 4;
  const auto red = p.nsplit <= 2 ? mvm_reduce_kernel<2> : (p.nsplit <= 4 ? mvm_reduce_kernel<4> : mvm_reduce_kernel<8>);
  hipLaunchKernelGGL(red, dim3((unsigned)((nout + 255) / 256 + (r.naux ? 1 : 0))), dim3(256), 0, st, r);
  Q35_HIP_TRY(hipGetLastError());
  return Q35_OK;
}

}  // namespace q35
