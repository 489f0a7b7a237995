// The reads of a temporal bank in one pass (gfx950): every view's normalized
// read, the bank's blend and the output gate,
//   y = (sum_j c_j (r_j + s num_j / (mass_j + eps))) * silu(g + g_bias)
// (engine.py:440-442, 526-528; block.py:683-722; gates.py:34-40), and its
// backward.  The sums stay in fp32 from the bf16 numerators to the one
// rounding of y; the separate chain rounded every view's read and the blend.
//
// Bound: HBM.  A fast bank of two rates (three views) reads 3 num, 1 resid
// and 1 gate row of d elements per token and writes one; one launch replaces
// three reads, the blend, the gate's SiLU and product and a transposing copy
// (backward: the gate's products, the blend's and three reads' backward and
// the sums of the residual gradients).

#include "ts_common.h"
#include "thetascan_hip.h"

#include <string.h>

namespace ts {

struct BankReadP {
  int B, H, T, d, n, nres, normalize, gate, tiles;
  float s, eps;
  ts_strided num[TS_BANK_MAX], mass[TS_BANK_MAX], resid[TS_BANK_MAX], g, y, dy;
  ts_strided dnum[TS_BANK_MAX], dmass[TS_BANK_MAX], dresid[TS_BANK_MAX], dg;
  const float* coef;   // [n][H]
  const float* gbias;  // [H][d] or null
  float* dcoef_part;   // [B * tiles][n][H]
  float* dgb_part;     // [B * tiles][H * d] or null
};

// A row (one token of one head) is CPR 16-byte chunks in CPR consecutive
// lanes, as in the single-view read kernels; a block covers kPasses *
// (256 / CPR) consecutive tokens of one (b, h), kFlight passes at a time with
// all their loads issued before any arithmetic.  B8 T4096 H8 d64, three
// views and the gate: forward 55 us (201 MB, 3.6 TB/s; the separate launches
// took about 150 us), backward 127 us (369 MB; about 300 us).
constexpr int kBankPasses = 4;
constexpr int kBankFlight = 2;

template <int CPR>
__host__ __device__ constexpr int bank_rows() { return kBankPasses * (256 / CPR); }

template <typename T>
__device__ __forceinline__ T* bank_at(const ts_strided& s, int b, int h) {
  return (T*)s.ptr + (int64_t)b * s.sb + (int64_t)h * s.sh;
}
template <typename E, int N>
__device__ __forceinline__ void bank_unpack(const uint4& raw, float* out) {
  Vec16<E> v;
  v.raw = raw;
#pragma unroll
  for (int e = 0; e < N; ++e) out[e] = tof(v.e[e]);
}
template <typename E, int N>
__device__ __forceinline__ uint4 bank_pack(const float* in) {
  Vec16<E> v;
#pragma unroll
  for (int e = 0; e < N; ++e) v.e[e] = cvt<E>(in[e]);
  return v.raw;
}
__device__ __forceinline__ float bank_sigmoid(float x) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x));
}

template <typename E, int CPR, int NV>
__global__ __launch_bounds__(256) void bank_read_fwd_kernel(BankReadP p) {
  constexpr int N = Vec16<E>::N;
  constexpr int RP = 256 / CPR;
  const int bh = blockIdx.y, b = bh / p.H, h = bh - b * p.H;
  const int c = ((int)threadIdx.x % CPR) * N;
  const bool colok = c < p.d;
  float coef[NV], gb[N];
#pragma unroll
  for (int j = 0; j < NV; ++j) coef[j] = j < p.n ? p.coef[j * p.H + h] : 0.0f;
#pragma unroll
  for (int e = 0; e < N; ++e) gb[e] = p.gbias && colok ? p.gbias[h * p.d + c + e] : 0.0f;
#pragma unroll
  for (int pass = 0; pass < kBankPasses; pass += kBankFlight) {
    uint4 rn[kBankFlight][NV], rr[kBankFlight][NV], rg[kBankFlight];
    float ms[kBankFlight][NV];
#pragma unroll
    for (int i = 0; i < kBankFlight; ++i) {
      const int64_t t = (int64_t)blockIdx.x * bank_rows<CPR>() + (pass + i) * RP + (int)threadIdx.x / CPR;
      if (t < p.T && colok) {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          if (j < p.n) {
            rn[i][j] = *(const uint4*)(bank_at<const E>(p.num[j], b, h) + t * p.num[j].st + c);
            if (p.normalize) ms[i][j] = bank_at<const float>(p.mass[j], b, h)[t * p.mass[j].st];
            if (j < p.nres) rr[i][j] = *(const uint4*)(bank_at<const E>(p.resid[j], b, h) + t * p.resid[j].st + c);
          }
        }
        if (p.gate) rg[i] = *(const uint4*)(bank_at<const E>(p.g, b, h) + t * p.g.st + c);
      }
    }
#pragma unroll
    for (int i = 0; i < kBankFlight; ++i) {
      const int64_t t = (int64_t)blockIdx.x * bank_rows<CPR>() + (pass + i) * RP + (int)threadIdx.x / CPR;
      if (t >= p.T || !colok) continue;
      float acc[N], rv[N];
#pragma unroll
      for (int e = 0; e < N; ++e) acc[e] = 0.0f;
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        if (j < p.n) {
          float nv[N];
          bank_unpack<E, N>(rn[i][j], nv);
          if (j < p.nres) bank_unpack<E, N>(rr[i][j], rv);
          const float sc = p.normalize ? p.s * __builtin_amdgcn_rcpf(ms[i][j] + p.eps) : p.s;
#pragma unroll
          for (int e = 0; e < N; ++e) acc[e] += coef[j] * (rv[e] + sc * nv[e]);
        }
      }
      if (p.gate) {
        float gv[N];
        bank_unpack<E, N>(rg[i], gv);
#pragma unroll
        for (int e = 0; e < N; ++e) {
          const float x = gv[e] + gb[e];
          acc[e] *= x * bank_sigmoid(x);
        }
      }
      *(uint4*)(bank_at<E>(p.y, b, h) + t * p.y.st + c) = bank_pack<E, N>(acc);
    }
  }
}

// Backward.  Per token and view: dnum_j = c_j s/(mass_j+eps) dpre,
// dmass_j = -s c_j (dpre . num_j) / (mass_j+eps)^2 (a butterfly over the
// row's lanes), dresid = c_j dpre (one shared residual: its sum over j),
// dg = dy y_pre silu'(x) with dpre = dy silu(x).  dL/dc_j and the gate-bias
// gradient leave each block as one partial per (view, head) and per column,
// summed over the block in a fixed order.
template <typename E, int CPR, int NV>
__global__ __launch_bounds__(256) void bank_read_bwd_kernel(BankReadP p) {
  constexpr int N = Vec16<E>::N;
  constexpr int RP = 256 / CPR;
  __shared__ float red[256 * N];
  __shared__ float redc[4][NV];
  const int bh = blockIdx.y, b = bh / p.H, h = bh - b * p.H;
  const int tid = threadIdx.x;
  const int c = (tid % CPR) * N;
  const bool colok = c < p.d;
  float coef[NV], dc[NV], gb[N], colsum[N], csum = 0.0f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    coef[j] = j < p.n ? p.coef[j * p.H + h] : 0.0f;
    csum += coef[j];
    dc[j] = 0.0f;
  }
#pragma unroll
  for (int e = 0; e < N; ++e) {
    gb[e] = p.gbias && colok ? p.gbias[h * p.d + c + e] : 0.0f;
    colsum[e] = 0.0f;
  }
#pragma unroll
  for (int pass = 0; pass < kBankPasses; pass += kBankFlight) {
    uint4 rn[kBankFlight][NV], rr[kBankFlight][NV], rg[kBankFlight], rd[kBankFlight];
    float ms[kBankFlight][NV];
#pragma unroll
    for (int i = 0; i < kBankFlight; ++i) {
      const int64_t t = (int64_t)blockIdx.x * bank_rows<CPR>() + (pass + i) * RP + tid / CPR;
      if (t < p.T) {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          if (j < p.n) {
            if (p.normalize) ms[i][j] = bank_at<const float>(p.mass[j], b, h)[t * p.mass[j].st];
            if (colok) {
              rn[i][j] = *(const uint4*)(bank_at<const E>(p.num[j], b, h) + t * p.num[j].st + c);
              if (j < p.nres) rr[i][j] = *(const uint4*)(bank_at<const E>(p.resid[j], b, h) + t * p.resid[j].st + c);
            }
          }
        }
        if (colok) {
          rd[i] = *(const uint4*)(bank_at<const E>(p.dy, b, h) + t * p.dy.st + c);
          if (p.gate) rg[i] = *(const uint4*)(bank_at<const E>(p.g, b, h) + t * p.g.st + c);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kBankFlight; ++i) {
      const int64_t t = (int64_t)blockIdx.x * bank_rows<CPR>() + (pass + i) * RP + tid / CPR;
      const bool live = t < p.T && colok;  // dead rows and columns join the row butterfly with zeros
      float dpre[N], ypre[N], rv[N];
#pragma unroll
      for (int e = 0; e < N; ++e) dpre[e] = ypre[e] = rv[e] = 0.0f;
      if (live) bank_unpack<E, N>(rd[i], dpre);
      float gv[N];
      if (p.gate && live) {
        bank_unpack<E, N>(rg[i], gv);
        // y before the gate
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          if (j < p.n) {
            float nv[N];
            bank_unpack<E, N>(rn[i][j], nv);
            if (j < p.nres) bank_unpack<E, N>(rr[i][j], rv);
            const float sc = p.normalize ? p.s * __builtin_amdgcn_rcpf(ms[i][j] + p.eps) : p.s;
#pragma unroll
            for (int e = 0; e < N; ++e) ypre[e] += coef[j] * (rv[e] + sc * nv[e]);
          }
        }
        float o_dg[N];
#pragma unroll
        for (int e = 0; e < N; ++e) {
          const float x = gv[e] + gb[e];
          const float sg = bank_sigmoid(x);
          o_dg[e] = dpre[e] * ypre[e] * (sg * (1.0f + x * (1.0f - sg)));
          colsum[e] += o_dg[e];
          dpre[e] *= x * sg;
        }
        *(uint4*)(bank_at<E>(p.dg, b, h) + t * p.dg.st + c) = bank_pack<E, N>(o_dg);
      }
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        if (j < p.n) {
          const float inv = p.normalize ? __builtin_amdgcn_rcpf((t < p.T ? ms[i][j] : 1.0f) + p.eps) : 1.0f;
          const float sc = p.s * inv;
          float dot = 0.0f, rdot = 0.0f;
          if (live) {
            float nv[N], o[N];
            bank_unpack<E, N>(rn[i][j], nv);
            if (j < p.nres) bank_unpack<E, N>(rr[i][j], rv);
#pragma unroll
            for (int e = 0; e < N; ++e) {
              dot += dpre[e] * nv[e];
              rdot += dpre[e] * rv[e];
              o[e] = coef[j] * sc * dpre[e];
            }
            *(uint4*)(bank_at<E>(p.dnum[j], b, h) + t * p.dnum[j].st + c) = bank_pack<E, N>(o);
            if (j < p.nres && p.dresid[j].ptr) {
              const float cr = p.nres == 1 ? csum : coef[j];
#pragma unroll
              for (int e = 0; e < N; ++e) o[e] = cr * dpre[e];
              *(uint4*)(bank_at<E>(p.dresid[j], b, h) + t * p.dresid[j].st + c) = bank_pack<E, N>(o);
            }
          }
          dc[j] += rdot + sc * dot;
          if (p.normalize) {
#pragma unroll
            for (int o = 1; o < CPR; o <<= 1) dot += __shfl_xor(dot, o, 64);
            if (t < p.T && tid % CPR == 0)
              bank_at<float>(p.dmass[j], b, h)[t * p.dmass[j].st] = -p.s * coef[j] * dot * inv * inv;
          }
        }
      }
    }
  }
  const int64_t slot = (int64_t)b * gridDim.x + blockIdx.x;
  if (p.dcoef_part) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      float v = dc[j];
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
      if ((tid & 63) == 0) redc[tid >> 6][j] = v;
    }
    __syncthreads();
    if (tid < NV && tid < p.n)
      p.dcoef_part[(slot * p.n + tid) * p.H + h] = redc[0][tid] + redc[1][tid] + redc[2][tid] + redc[3][tid];
  }
  if (p.dgb_part) {
#pragma unroll
    for (int e = 0; e < N; ++e) red[tid * N + e] = colsum[e];
    __syncthreads();
    // one output column per thread (the host checks d <= 256)
    if (tid < p.d) {
      const int chunk = tid / N, e = tid - chunk * N;
      float v = 0.0f;
      for (int l = 0; l < RP; ++l) v += red[(l * CPR + chunk) * N + e];
      p.dgb_part[slot * (p.H * p.d) + h * p.d + tid] = v;
    }
  }
}

// A fast bank's parameters in one launch each way (block.py:647-695): thread h
// forms every branch's log retention -softplus(-alpha_raw), rounded through
// the parameter's and the streams' dtypes as the tensor expression is, and the
// blend coefficients (1 - sum eta, eta_1 ..), eta through tanh when asked.
// Latency only: a few dozen numbers, which as tensor expressions took about
// twenty launches forward and as many backward.
struct BankParamsP {
  int n, H, tanh_eta, pbf, xbf;    // pbf / xbf: the parameters / the streams are bf16
  const void* alpha;               // [n][H]
  const void* eta;                 // [n][H]
  float* la[TS_BANK_MAX];          // [H] each
  float* coef;                     // [n + 1][H]
  const float* dla[TS_BANK_MAX];   // [H] each or null
  const float* dcoef;              // [n + 1][H] or null
  void* dalpha;                    // parameters' dtype
  void* deta;
};

__device__ __forceinline__ float bank_param(const void* p, int bf, int i) {
  return bf ? tof(((const bf16*)p)[i]) : ((const float*)p)[i];
}
__device__ __forceinline__ float bank_round(float x, int bf) { return bf ? tof((bf16)x) : x; }
__device__ __forceinline__ float bank_eta(const BankParamsP& p, int i) {
  const float e = bank_param(p.eta, p.pbf, i);
  return p.tanh_eta ? bank_round(tanhf(e), p.pbf) : e;
}

__global__ void bank_params_fwd_kernel(BankParamsP p) {
  for (int h = threadIdx.x; h < p.H; h += blockDim.x) {
    float sum = 0.0f;
    for (int j = 0; j < p.n; ++j) {
      const float x = -bank_param(p.alpha, p.pbf, j * p.H + h);
      const float sp = x > 20.0f ? x : log1pf(expf(x));
      p.la[j][h] = bank_round(-bank_round(sp, p.pbf), p.xbf);
      const float e = bank_eta(p, j * p.H + h);
      p.coef[(j + 1) * p.H + h] = e;
      sum += e;
    }
    p.coef[h] = 1.0f - sum;
  }
}

__global__ void bank_params_bwd_kernel(BankParamsP p) {
  for (int h = threadIdx.x; h < p.H; h += blockDim.x)
    for (int j = 0; j < p.n; ++j) {
      const int i = j * p.H + h;
      const float x = -bank_param(p.alpha, p.pbf, i);
      // d(-softplus(-a)) / da = sigmoid(-a)
      const float da = p.dla[j] ? p.dla[j][h] * (x > 20.0f ? 1.0f : 1.0f / (1.0f + expf(-x))) : 0.0f;
      float de = p.dcoef ? p.dcoef[(j + 1) * p.H + h] - p.dcoef[h] : 0.0f;
      if (p.tanh_eta) {
        const float e = bank_eta(p, i);
        de *= 1.0f - e * e;
      }
      if (p.pbf) {
        ((bf16*)p.dalpha)[i] = (bf16)da;
        ((bf16*)p.deta)[i] = (bf16)de;
      } else {
        ((float*)p.dalpha)[i] = da;
        ((float*)p.deta)[i] = de;
      }
    }
}

}  // namespace ts

namespace {

using ts::fail;

int fill_params(const ts_bank_params_desc* d, const void* alpha, const void* eta, ts::BankParamsP* p) {
  if (!d || !alpha || !eta) return fail(TS_ERR_VALUE, "bank params: missing descriptor or parameters");
  if (d->n < 1 || d->n >= TS_BANK_MAX || d->H < 1) return fail(TS_ERR_VALUE, "bank params: %d branches of %d heads", d->n, d->H);
  for (int t : {d->param_dtype, d->stream_dtype})
    if (t != TS_BF16 && t != TS_F32) return fail(TS_ERR_VALUE, "bank params: unknown dtype");
  memset(p, 0, sizeof(*p));
  p->n = d->n; p->H = d->H; p->tanh_eta = d->tanh_eta;
  p->pbf = d->param_dtype == TS_BF16; p->xbf = d->stream_dtype == TS_BF16;
  p->alpha = alpha; p->eta = eta;
  return TS_OK;
}

int params_done() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TS_OK : fail(TS_ERR_RUNTIME, "bank params: launch failed: %s", hipGetErrorString(e));
}

int chunks_p2(const ts_bank_read_desc* d) {
  const int chunks = d->d / (d->dtype == TS_BF16 ? 8 : 4);
  int p2 = 2;
  while (p2 < chunks) p2 <<= 1;
  return p2;
}

int check(const ts_bank_read_desc* d) {
  if (!d) return fail(TS_ERR_VALUE, "bank read: null descriptor");
  if (d->B < 1 || d->H < 1 || d->T < 0 || d->d < 1) return fail(TS_ERR_VALUE, "bank read: bad shape");
  if (d->n_views < 1 || d->n_views > TS_BANK_MAX)
    return fail(TS_ERR_VALUE, "bank read: %d views (1 .. %d)", d->n_views, TS_BANK_MAX);
  if (d->n_resid != 1 && d->n_resid != d->n_views)
    return fail(TS_ERR_VALUE, "bank read: one residual, or one per view (got %d)", d->n_resid);
  if (d->dtype != TS_BF16 && d->dtype != TS_F32) return fail(TS_ERR_VALUE, "bank read: unknown dtype");
  const int vec = d->dtype == TS_BF16 ? 8 : 4;
  if (d->d % vec) return fail(TS_ERR_VALUE, "bank read: width %d is not a multiple of 16 bytes", d->d);
  if (d->d > 32 * vec) return fail(TS_ERR_NOT_IMPLEMENTED, "bank read: width %d is too wide", d->d);
  if ((int64_t)d->B * d->H > 65535) return fail(TS_ERR_NOT_IMPLEMENTED, "bank read: B*H above 65535");
  return TS_OK;
}

int tiles_of(const ts_bank_read_desc* d) {
  const int rows = ts::kBankPasses * (256 / chunks_p2(d));
  return (d->T + rows - 1) / rows;
}

int check_rows(const char* name, const ts_strided& s, int vec) {
  if (!s.ptr) return fail(TS_ERR_VALUE, "bank read: missing %s", name);
  if (((uintptr_t)s.ptr & 15u) || s.st % vec || s.sh % vec || s.sb % vec)
    return fail(TS_ERR_VALUE, "bank read: rows of %s must be 16-byte aligned", name);
  return TS_OK;
}

template <typename E, int CPR, int NV>
void launch(bool bwd, dim3 grid, hipStream_t stream, const ts::BankReadP& p) {
  if (bwd) hipLaunchKernelGGL((ts::bank_read_bwd_kernel<E, CPR, NV>), grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((ts::bank_read_fwd_kernel<E, CPR, NV>), grid, dim3(256), 0, stream, p);
}
template <typename E, int CPR>
void dispatch_n(bool bwd, dim3 grid, hipStream_t stream, const ts::BankReadP& p) {
  if (p.n <= 2) launch<E, CPR, 2>(bwd, grid, stream, p);
  else if (p.n == 3) launch<E, CPR, 3>(bwd, grid, stream, p);
  else launch<E, CPR, TS_BANK_MAX>(bwd, grid, stream, p);
}
template <typename E>
void dispatch(int cpr, bool bwd, dim3 grid, hipStream_t stream, const ts::BankReadP& p) {
  switch (cpr) {
    case 2: dispatch_n<E, 2>(bwd, grid, stream, p); break;
    case 4: dispatch_n<E, 4>(bwd, grid, stream, p); break;
    case 8: dispatch_n<E, 8>(bwd, grid, stream, p); break;
    case 16: dispatch_n<E, 16>(bwd, grid, stream, p); break;
    default: dispatch_n<E, 32>(bwd, grid, stream, p); break;
  }
}

int fill(const ts_bank_read_desc* d, const ts_bank_read_io* io, ts::BankReadP* p) {
  int rc = check(d);
  if (rc) return rc;
  if (!io || !io->coef) return fail(TS_ERR_VALUE, "bank read: missing io or coefficients");
  const int vec = d->dtype == TS_BF16 ? 8 : 4;
  memset(p, 0, sizeof(*p));
  p->B = d->B; p->H = d->H; p->T = d->T; p->d = d->d; p->n = d->n_views; p->nres = d->n_resid;
  p->normalize = d->normalize; p->gate = d->gate; p->s = d->scale; p->eps = d->eps; p->tiles = tiles_of(d);
  p->coef = io->coef; p->gbias = io->gbias;
  for (int j = 0; j < d->n_views; ++j) {
    p->num[j] = io->num[j];
    if ((rc = check_rows("num", p->num[j], vec))) return rc;
    if (d->normalize) {
      p->mass[j] = io->mass[j];
      if (!p->mass[j].ptr) return fail(TS_ERR_VALUE, "bank read: missing mass %d", j);
    }
    if (j < d->n_resid) {
      p->resid[j] = io->resid[j];
      if ((rc = check_rows("resid", p->resid[j], vec))) return rc;
    }
  }
  if (d->gate) {
    p->g = io->g;
    if ((rc = check_rows("gate", p->g, vec))) return rc;
  }
  return TS_OK;
}

int run(const ts_bank_read_desc* d, bool bwd, hipStream_t stream, const ts::BankReadP& p) {
  if (d->T == 0) return TS_OK;
  const dim3 grid((unsigned)p.tiles, (unsigned)(d->B * d->H));
  if (d->dtype == TS_BF16) dispatch<ts::bf16>(chunks_p2(d), bwd, grid, stream, p);
  else dispatch<float>(chunks_p2(d), bwd, grid, stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "bank read: launch failed: %s", hipGetErrorString(e));
  return TS_OK;
}

}  // namespace

extern "C" {

int ts_bank_read_fwd(const ts_bank_read_desc* d, const ts_bank_read_io* io, ts_strided y, hipStream_t stream) {
  ts::BankReadP p;
  int rc = fill(d, io, &p);
  if (rc) return rc;
  p.y = y;
  if ((rc = check_rows("y", p.y, d->dtype == TS_BF16 ? 8 : 4))) return rc;
  return run(d, false, stream, p);
}

int ts_bank_read_parts(const ts_bank_read_desc* d, int32_t* parts) {
  int rc = check(d);
  if (rc) return rc;
  if (parts) *parts = d->B * tiles_of(d);
  return TS_OK;
}

int ts_bank_read_bwd(const ts_bank_read_desc* d, const ts_bank_read_io* io, const ts_bank_read_grads* g,
                     hipStream_t stream) {
  ts::BankReadP p;
  int rc = fill(d, io, &p);
  if (rc) return rc;
  if (!g) return fail(TS_ERR_VALUE, "bank read: missing gradients");
  const int vec = d->dtype == TS_BF16 ? 8 : 4;
  p.dy = g->dy;
  if ((rc = check_rows("dy", p.dy, vec))) return rc;
  for (int j = 0; j < d->n_views; ++j) {
    p.dnum[j] = g->dnum[j];
    if ((rc = check_rows("dnum", p.dnum[j], vec))) return rc;
    if (d->normalize) {
      p.dmass[j] = g->dmass[j];
      if (!p.dmass[j].ptr) return fail(TS_ERR_VALUE, "bank read: missing dmass %d", j);
    }
    if (j < d->n_resid) {
      p.dresid[j] = g->dresid[j];
      if (p.dresid[j].ptr && (rc = check_rows("dresid", p.dresid[j], vec))) return rc;
    }
  }
  if (d->gate) {
    p.dg = g->dg;
    if ((rc = check_rows("dg", p.dg, vec))) return rc;
    if (g->dgb_part && d->d > 256) return fail(TS_ERR_NOT_IMPLEMENTED, "bank read: gate bias width %d", d->d);
    p.dgb_part = g->dgb_part;
  }
  p.dcoef_part = g->dcoef_part;
  return run(d, true, stream, p);
}

int ts_bank_params_fwd(const ts_bank_params_desc* d, const void* alpha, const void* eta, float* const* log_alpha,
                       float* coef, hipStream_t stream) {
  ts::BankParamsP p;
  int rc = fill_params(d, alpha, eta, &p);
  if (rc) return rc;
  if (!log_alpha || !coef) return fail(TS_ERR_VALUE, "bank params: missing outputs");
  for (int j = 0; j < d->n; ++j)
    if (!(p.la[j] = log_alpha[j])) return fail(TS_ERR_VALUE, "bank params: missing log retention %d", j);
  p.coef = coef;
  hipLaunchKernelGGL(ts::bank_params_fwd_kernel, dim3(1), dim3(64), 0, stream, p);
  return params_done();
}

int ts_bank_params_bwd(const ts_bank_params_desc* d, const void* alpha, const void* eta, const float* const* dlog_alpha,
                       const float* dcoef, void* dalpha, void* deta, hipStream_t stream) {
  ts::BankParamsP p;
  int rc = fill_params(d, alpha, eta, &p);
  if (rc) return rc;
  if (!dlog_alpha || !dalpha || !deta) return fail(TS_ERR_VALUE, "bank params: missing gradients");
  for (int j = 0; j < d->n; ++j) p.dla[j] = dlog_alpha[j];
  p.dcoef = dcoef; p.dalpha = dalpha; p.deta = deta;
  hipLaunchKernelGGL(ts::bank_params_bwd_kernel, dim3(1), dim3(64), 0, stream, p);
  return params_done();
}

}  // extern "C"
