// A decode step of the depth-1 kernel memory with the plain sum (gfx950): at
// most eight tokens per sequence continuing a carried state.
//
// ts_memory_step runs everything between the projections for one (batch,
// head) in one workgroup: input RoPE and L2 norm, W1, RMSNorm, threshold,
// feature map and feature RoPE of keys and queries, the residual xn + s W2 h,
// the recurrence on the fp32 state, the (normalized) read and the output gate
// (block.py:595-618, engine.py:117-158, 426-544, kernel_features.py:73-135,
// block.py:721-722).  Bound: latency.  Every load (weights, state, rows) is
// issued up front, so a step waits for memory once; RoPE phases are formed
// from the position (a host value, or a device counter under graph replay).
// B8 H8 d = m = 64, one token: replaces two feature launches (4.8 us each),
// the token-by-token scan (10.4 us), the read with the gate's own launches
// (9.5 us) and four launches of the phases; it takes 9.1 us, and a captured
// step 29 us against 53 us.
//
// ts_skinny_linear is the projection around it, y = x [Wa; Wb]^T for at most
// 64 rows (bf16): 16 outputs per workgroup, the contraction split over its
// four waves, so 2048 outputs keep 128 workgroups busy and two weights need
// neither two launches nor a concatenated copy.

#include "ts_common.h"
#include "thetascan_hip.h"

#include <string.h>

namespace ts {

constexpr int kStepT = 8;

struct MemStepP {
  int H, T, d, m, in_rot, feat_rot, kind, normalize, gate, param_bf16, has_init;
  float gain, s, eps;
  ts_strided q, k, v, g, y;
  const void* w1;     // [H][m][d] of the rows' dtype
  const void* w2;     // [H][d][m]
  const void* tau;    // [H] parameters' dtype or null
  const void* gbias;  // [H*d] parameters' dtype or null
  const float* inv_in;    // [in_rot / 2] inverse frequencies
  const float* inv_feat;  // [feat_rot / 2]
  const int64_t* pos_dev;
  int64_t pos;
  const float* init;  // [B*H][m][d + normalize] or null
  float* fin;
};

__device__ __forceinline__ float step_param(const void* p, int bf, int i) {
  return bf ? tof(((const bf16*)p)[i]) : ((const float*)p)[i];
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// NE consecutive elements of a weight row as raw 16-byte vectors.
template <typename E, int NE>
struct WRow {
  static constexpr int NV = NE * (int)sizeof(E) / 16;
  uint4 r[NV];
  __device__ __forceinline__ void load(const E* p) {
#pragma unroll
    for (int i = 0; i < NV; ++i) r[i] = ((const uint4*)p)[i];
  }
  __device__ __forceinline__ float dot(const float* x) const {
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      Vec16<E> v;
      v.raw = r[i];
#pragma unroll
      for (int e = 0; e < Vec16<E>::N; ++e) acc = fmaf(tof(v.e[e]), x[i * Vec16<E>::N + e], acc);
    }
    return acc;
  }
};

// DP, MP: head width and feature count padded to 64 or 128 (DP <= MP).
template <typename E, int DP, int MP>
__global__ __launch_bounds__(256) void memory_step_kernel(MemStepP p) {
  constexpr int NG = 256 / DP;    // row groups of the state
  constexpr int RPT = MP / NG;    // state rows per thread
  constexpr int W1N = DP / 4, W2N = MP / 4;
  __shared__ float xs[2 * kStepT][DP];   // normalized keys (0..7), queries (8..15)
  __shared__ float fs[2 * kStepT][MP];   // W1 xn, then the rotated features
  __shared__ float hs[kStepT][MP];       // the queries' features before the rotation
  __shared__ float vs[kStepT][DP], gs[kStepT][DP], rs[kStepT][DP];
  __shared__ float red[2][NG][DP], dred[2][4];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int bh = blockIdx.x, b = bh / p.H, h = bh - b * p.H;
  const int T = p.T, d = p.d, m = p.m;
  const int cols = d + p.normalize;

  // ---- every load of the step, in flight together
  WRow<E, W1N> w1r[MP / 64];
  WRow<E, W2N> w2r[DP / 64];
  const int part = tid & 3, row0 = tid >> 2;
#pragma unroll
  for (int i = 0; i < MP / 64; ++i) {
    const int row = row0 + 64 * i;
    if (row < m && part * W1N < d) w1r[i].load((const E*)p.w1 + ((int64_t)h * m + row) * d + part * W1N);
  }
#pragma unroll
  for (int i = 0; i < DP / 64; ++i) {
    const int row = row0 + 64 * i;
    if (row < d && part * W2N < m) w2r[i].load((const E*)p.w2 + ((int64_t)h * d + row) * m + part * W2N);
  }
  const int j = tid % DP, rg = tid / DP;
  float S[RPT], D = 0.f;
  const size_t state = (size_t)bh * m * cols;
#pragma unroll
  for (int r = 0; r < RPT; ++r) {
    const int i = rg * RPT + r;
    S[r] = p.has_init && i < m && j < d ? p.init[state + (size_t)i * cols + j] : 0.f;
  }
  if (p.normalize && p.has_init && tid < m) D = p.init[state + (size_t)tid * cols + d];
  auto at = [&](const ts_strided& s, int t) { return (const E*)s.ptr + (int64_t)b * s.sb + (int64_t)h * s.sh + t * s.st; };
  const float tau = p.tau ? step_param(p.tau, p.param_bf16, h) : 0.f;
  const int64_t pos = p.pos_dev ? *p.pos_dev : p.pos;
  for (int e = tid; e < T * d; e += 256) {
    const int t = e / d, c = e - t * d;
    vs[t][c] = tof(at(p.v, t)[c]);
    if (p.gate) gs[t][c] = tof(at(p.g, t)[c]) + (p.gbias ? step_param(p.gbias, p.param_bf16, h * d + c) : 0.f);
  }
  // ---- keys and queries: a wave per row, a pair (2 lane, 2 lane + 1) per lane
  for (int r = w; r < 2 * T; r += 4) {
    const int t = r < T ? r : r - T;
    const E* src = at(r < T ? p.k : p.q, t);
    float a = 0.f, c = 0.f;
    if (2 * lane < d) {
      a = tof(src[2 * lane]);
      c = tof(src[2 * lane + 1]);
      if (2 * lane < p.in_rot) {
        const float ang = (float)(pos + t) * p.inv_in[lane];
        const float cs = cosf(ang), sn = sinf(ang);
        const float a0 = a;
        a = a0 * cs - c * sn;
        c = a0 * sn + c * cs;
      }
    }
    const float inv = 1.0f / fmaxf(sqrtf(wave_sum(a * a + c * c)), p.eps);
    const int slot = r < T ? t : kStepT + t;
    if (2 * lane < DP) {
      xs[slot][2 * lane] = 2 * lane < d ? a * inv : 0.f;
      xs[slot][2 * lane + 1] = 2 * lane < d ? c * inv : 0.f;
    }
  }
  __syncthreads();
  // ---- W1 xn: four lanes per feature row
  for (int r = 0; r < 2 * T; ++r) {
    const int slot = r < T ? r : kStepT + r - T;
#pragma unroll
    for (int i = 0; i < MP / 64; ++i) {
      const int row = row0 + 64 * i;
      float a = row < m && part * W1N < d ? w1r[i].dot(&xs[slot][part * W1N]) : 0.f;
      a += __shfl_xor(a, 1, 64);
      a += __shfl_xor(a, 2, 64);
      if (part == 0) fs[slot][row] = a;
    }
  }
  __syncthreads();
  // ---- RMSNorm, threshold, map, feature RoPE: a wave per row
  for (int r = w; r < 2 * T; r += 4) {
    const int t = r < T ? r : r - T;
    const int slot = r < T ? t : kStepT + t;
    float* f = fs[slot];
    float a = 0.f, c = 0.f;
    const bool on = 2 * lane < m;
    if (on) {
      a = f[2 * lane];
      c = f[2 * lane + 1];
    }
    const float rinv = rsqrtf(wave_sum(a * a + c * c) / (float)m + p.eps);
    if (p.kind == TS_FEAT_RELU2) {
      a = fmaxf(a * rinv - tau, 0.f);
      c = fmaxf(c * rinv - tau, 0.f);
      a = on ? a * a : 0.f;
      c = on ? c * c : 0.f;
      const float mass = wave_sum(a + c);
      const bool ok = mass > p.eps;
      a = ok ? a / mass : 1.0f / (float)m;
      c = ok ? c / mass : 1.0f / (float)m;
    } else {
      a = on ? p.gain * (a * rinv - tau) : -INFINITY;
      c = on ? p.gain * (c * rinv - tau) : -INFINITY;
      const float mx = wave_max(fmaxf(a, c));
      a = on ? expf(a - mx) : 0.f;
      c = on ? expf(c - mx) : 0.f;
      const float inv = 1.0f / wave_sum(a + c);
      a *= inv;
      c *= inv;
    }
    if (on) {
      if (r >= T) {
        hs[t][2 * lane] = a;
        hs[t][2 * lane + 1] = c;
      }
      if (2 * lane < p.feat_rot) {
        const float ang = (float)(pos + t) * p.inv_feat[lane];
        const float cs = cosf(ang), sn = sinf(ang);
        const float a0 = a;
        a = a0 * cs - c * sn;
        c = a0 * sn + c * cs;
      }
      f[2 * lane] = a;
      f[2 * lane + 1] = c;
    } else if (2 * lane < MP) {
      f[2 * lane] = f[2 * lane + 1] = 0.f;
      if (r >= T) hs[t][2 * lane] = hs[t][2 * lane + 1] = 0.f;
    }
  }
  __syncthreads();
  // ---- residual xn + s W2 h of the queries
  for (int t = 0; t < T; ++t) {
#pragma unroll
    for (int i = 0; i < DP / 64; ++i) {
      const int row = row0 + 64 * i;
      float a = row < d && part * W2N < m ? w2r[i].dot(&hs[t][part * W2N]) : 0.f;
      a += __shfl_xor(a, 1, 64);
      a += __shfl_xor(a, 2, 64);
      if (part == 0) rs[t][row] = xs[kStepT + t][row] + p.s * a;
    }
  }
  // ---- the recurrence and the read.  A group's state rows are all features
  // or all padding (m is the padded width or a multiple of its rows a group);
  // the padding's weights are zeros, and stay so against an infinite value
  // only if it does not reach them.
  const bool on = j < d && rg * RPT < m;
  for (int t = 0; t < T; ++t) {
    const int buf = t & 1;
    const float vj = on ? vs[t][j] : 0.f;
    float num = 0.f;
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int i = rg * RPT + r;
      S[r] = fmaf(fs[t][i], vj, S[r]);
      num = fmaf(fs[kStepT + t][i], S[r], num);
    }
    red[buf][rg][j] = num;
    if (p.normalize) {
      float md = 0.f;
      if (tid < m) {
        D += fs[t][tid];
        md = fs[kStepT + t][tid] * D;
      }
      md = wave_sum(md);
      if (lane == 0) dred[buf][w] = md;
    }
    // a thread still reading buffer `buf` of token t has passed this barrier
    // before any thread writes it again (token t + 2)
    __syncthreads();
    if (tid < d) {
      float o = 0.f;
#pragma unroll
      for (int i = 0; i < NG; ++i) o += red[buf][i][tid];
      float sc = p.s;
      if (p.normalize) sc /= dred[buf][0] + dred[buf][1] + dred[buf][2] + dred[buf][3] + p.eps;
      float y = rs[t][tid] + sc * o;
      if (p.gate) {
        const float x = gs[t][tid];
        y *= x / (1.0f + expf(-x));
      }
      ((E*)p.y.ptr)[(int64_t)b * p.y.sb + (int64_t)h * p.y.sh + (int64_t)t * p.y.st + tid] = cvt<E>(y);
    }
  }
  if (p.fin) {
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const int i = rg * RPT + r;
      if (i < m && j < d) p.fin[state + (size_t)i * cols + j] = S[r];
    }
    if (p.normalize && tid < m) p.fin[state + (size_t)tid * cols + d] = D;
  }
}

// y[n][o] = sum_k x[n][k] W[o][k], W = [Wa; Wb] (Wb may be absent): 16 outputs
// and 16 rows per workgroup, the contraction split over the four waves in
// blocks of 32; lanes of group g hold k = 32 blk + 8g .. +7 of both operands.
struct SkinnyP {
  int n, k, na, nb;
  int64_t x_st, y_st;
  const bf16* x;
  const bf16* wa;
  const bf16* wb;
  bf16* y;
};

__global__ __launch_bounds__(256) void skinny_linear_kernel(SkinnyP p) {
  constexpr int U = 4;  // blocks in flight per wave
  __shared__ floatx4 part[4][64];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 4, l16 = lane & 15;
  const int o0 = blockIdx.x * 16, n0 = blockIdx.y * 16;
  const int o = o0 + l16;  // a workgroup's outputs belong to one weight (na % 16 == 0)
  const bf16* wr = (o < p.na ? p.wa + (int64_t)o * p.k : p.wb + (int64_t)(o - p.na) * p.k) + 8 * g;
  const bool live = n0 + l16 < p.n;
  const bf16* xr = p.x + (int64_t)(live ? n0 + l16 : 0) * p.x_st + 8 * g;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  const int nblk = p.k / 32;
  for (int blk0 = w; blk0 < nblk; blk0 += 4 * U) {
    uint4 a[U], x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int blk = blk0 + 4 * u;
      if (blk < nblk) {
        a[u] = *(const uint4*)(wr + 32 * blk);
        x[u] = *(const uint4*)(xr + 32 * blk);
      } else {
        a[u] = x[u] = make_uint4(0u, 0u, 0u, 0u);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      acc = mma32(__builtin_bit_cast(bf16x8, a[u]), __builtin_bit_cast(bf16x8, x[u]), acc);
  }
  part[w][lane] = acc;
  __syncthreads();
  if (w == 0 && live) {
    floatx4 v = part[0][lane];
#pragma unroll
    for (int i = 1; i < 4; ++i) {
      const floatx4 u = part[i][lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += u[e];
    }
    // rows of the accumulator are outputs o0 + 4g + i, columns the rows of x
    LdsIO<bf16>::st4(p.y + (int64_t)(n0 + l16) * p.y_st + o0 + 4 * g, v[0], v[1], v[2], v[3]);
  }
}

}  // namespace ts

namespace {

using ts::fail;

int finish(const char* what) {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TS_OK : fail(TS_ERR_RUNTIME, "%s: launch failed: %s", what, hipGetErrorString(e));
}

template <typename E>
void launch_step(int d, int m, int bh, hipStream_t stream, const ts::MemStepP& p) {
  if (d <= 64) {
    if (m <= 64) hipLaunchKernelGGL((ts::memory_step_kernel<E, 64, 64>), dim3(bh), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((ts::memory_step_kernel<E, 64, 128>), dim3(bh), dim3(256), 0, stream, p);
  } else {
    hipLaunchKernelGGL((ts::memory_step_kernel<E, 128, 128>), dim3(bh), dim3(256), 0, stream, p);
  }
}

}  // namespace

extern "C" {

int ts_memory_step(const ts_memory_step_desc* d, const ts_memory_step_io* io, hipStream_t stream) {
  if (!d || !io) return fail(TS_ERR_VALUE, "memory step: null arguments");
  if (d->B < 1 || d->H < 1) return fail(TS_ERR_VALUE, "memory step: bad shape");
  if (d->T < 1 || d->T > ts::kStepT)
    return fail(TS_ERR_NOT_IMPLEMENTED, "memory step: %d tokens (1 .. %d)", d->T, ts::kStepT);
  if (d->dtype != TS_BF16 && d->dtype != TS_F32) return fail(TS_ERR_VALUE, "memory step: unknown dtype");
  if (d->param_dtype != TS_BF16 && d->param_dtype != TS_F32) return fail(TS_ERR_VALUE, "memory step: unknown dtype");
  if (d->kind != TS_FEAT_RELU2 && d->kind != TS_FEAT_SOFTMAX) return fail(TS_ERR_VALUE, "memory step: unknown map");
  for (int v : {d->d, d->m})
    if (v != 16 && v != 32 && v != 64 && v != 128)
      return fail(TS_ERR_NOT_IMPLEMENTED, "memory step: widths d %d, m %d (16, 32, 64 or 128)", d->d, d->m);
  if (d->m < d->d)  // a memory has at least as many features as head channels
    return fail(TS_ERR_NOT_IMPLEMENTED, "memory step: %d features below the head width %d", d->m, d->d);
  if (d->in_rot < 0 || d->in_rot > d->d || d->in_rot % 2 || d->feat_rot < 0 || d->feat_rot > d->m || d->feat_rot % 2)
    return fail(TS_ERR_VALUE, "memory step: rotated widths %d, %d", d->in_rot, d->feat_rot);
  if ((d->in_rot && !io->inv_in) || (d->feat_rot && !io->inv_feat))
    return fail(TS_ERR_VALUE, "memory step: missing inverse frequencies");
  if (!io->q.ptr || !io->k.ptr || !io->v.ptr || !io->y.ptr || !io->w1 || !io->w2 || (d->gate && !io->g.ptr))
    return fail(TS_ERR_VALUE, "memory step: missing tensors");
  if (((uintptr_t)io->w1 | (uintptr_t)io->w2) & 15u) return fail(TS_ERR_VALUE, "memory step: weights must be 16-byte aligned");
  ts::MemStepP p;
  memset(&p, 0, sizeof(p));
  p.H = d->H; p.T = d->T; p.d = d->d; p.m = d->m; p.in_rot = d->in_rot; p.feat_rot = d->feat_rot; p.kind = d->kind;
  p.normalize = d->normalize ? 1 : 0; p.gate = d->gate ? 1 : 0; p.param_bf16 = d->param_dtype == TS_BF16;
  p.has_init = io->init_state ? 1 : 0;
  p.gain = d->gain; p.s = d->resid_scale; p.eps = d->eps;
  p.q = io->q; p.k = io->k; p.v = io->v; p.g = io->g; p.y = io->y;
  p.w1 = io->w1; p.w2 = io->w2; p.tau = io->tau; p.gbias = io->gbias;
  p.inv_in = io->inv_in; p.inv_feat = io->inv_feat; p.pos_dev = io->position; p.pos = d->position;
  p.init = io->init_state; p.fin = io->final_state;
  if (d->dtype == TS_BF16) launch_step<ts::bf16>(d->d, d->m, d->B * d->H, stream, p);
  else launch_step<float>(d->d, d->m, d->B * d->H, stream, p);
  return finish("memory step");
}

int ts_skinny_linear(const void* x, int32_t n, int32_t k, int64_t x_stride, const void* wa, int32_t na, const void* wb,
                     int32_t nb, void* y, int64_t y_stride, hipStream_t stream) {
  if (n < 1 || n > 64 || k < 32 || k % 32 || na < 16 || na % 16 || nb < 0 || nb % 16)
    return fail(TS_ERR_NOT_IMPLEMENTED, "skinny linear: %d rows of %d into %d + %d outputs", n, k, na, nb);
  if (!x || !wa || !y || (nb && !wb)) return fail(TS_ERR_VALUE, "skinny linear: missing tensors");
  if (((uintptr_t)x | (uintptr_t)wa | (uintptr_t)wb) & 15u || ((uintptr_t)y & 7u) || x_stride % 8 || y_stride % 4)
    return fail(TS_ERR_VALUE, "skinny linear: rows must be 16-byte aligned");
  const ts::SkinnyP p = {n, k, na, nb, x_stride, y_stride, (const ts::bf16*)x, (const ts::bf16*)wa, (const ts::bf16*)wb,
                         (ts::bf16*)y};
  hipLaunchKernelGGL(ts::skinny_linear_kernel, dim3((na + nb) / 16, (n + 15) / 16), dim3(256), 0, stream, p);
  return finish("skinny linear");
}

}  // extern "C"
