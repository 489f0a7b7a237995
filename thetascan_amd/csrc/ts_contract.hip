// Token contractions for gfx950: out[g] = sum_n a[g, n, :]^T b[g, n, :] in fp32
// for token-major tiles a [G, N, p] and b [G, N, q] (p, q multiples of 16).
// These are the weight gradients of the GN fast network (dW1 = da^T x,
// dW2 = lam^T dz + ...), formed from per-token tiles written by the GN backward
// kernels.
//
// Workgroup (slice s, group g, block z of a sum: at most 128 x 128 of its
// output) contracts tokens [s * span, (s + 1) * span) in
// 64-token tiles: both tiles are staged in LDS (rows fetched with 16-byte
// loads one tile ahead), and wave w accumulates the 16 x 16 output blocks of
// rows 16 * (w + 4 j) with MFMAs whose token-axis operands come from the
// transposing LDS read (the same fragments as the feature backward's weight
// gradients).  Every slice writes an fp32 partial [p, q]; ts_sum_slots or the
// finish kernel adds the partials in slice order, so the result does not
// depend on timing.
//
// One call takes several sums over the same tokens (ts_contract_sums), each of
// up to two products added in the accumulators, and forms outputs from them: a
// backward's contractions take two launches, where one contraction, its
// reduction and the adds and casts after it were a dozen.  Bound by reading
// the tiles: the sums of a training step with one write and two read stages
// (B8 H8 T2048 d64 m128) read 400 MB in 86 us (4.7 TB/s).

#include "ts_common.h"
#include "ts_tokens.h"
#include "thetascan_hip.h"

#include <string.h>

namespace ts {

struct ContractTerm {
  const void* a;
  const void* b;
  int64_t a_sg, a_sn, b_sg, b_sn;  // element strides: group, token
};
struct ContractSum {
  int p, q, pw, qw, qc;  // widths, block widths, blocks along q
  int z0;                // this sum's first block
  int nterms;
  ContractTerm t[TS_CONTRACT_TERMS];
  float* parts;          // [S][G][p][q]
};
struct ContractP {
  int G, N, span, nsums;
  ContractSum sums[TS_CONTRACT_SUMS];
};

// a / b tile rows fetched one tile ahead (16-byte vectors, rows past the
// slice's end load as zero).
template <typename E>
struct ContractTile {
  static constexpr int VEC = 16 / (int)sizeof(E);
  static constexpr int SLOTS = (TT * 128 / VEC + 255) / 256;
  uint4 r[SLOTS];
  __device__ __forceinline__ void fetch(const E* base, int64_t sn, int width, int n0, int n1, int tid) {
    const int per_row = width / VEC;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      const int idx = tid + i * 256;
      const int row = idx / per_row;
      r[i] = make_uint4(0u, 0u, 0u, 0u);
      if (idx < TT * per_row && n0 + row < n1)
        r[i] = *(const uint4*)(base + (int64_t)(n0 + row) * sn + (idx - row * per_row) * VEC);
    }
  }
  __device__ __forceinline__ void store(E* dst, int pitch, int width, int tid) const {
    const int per_row = width / VEC;
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      const int idx = tid + i * 256;
      if (idx < TT * per_row) {
        const int row = idx / per_row;
        *(uint4*)(dst + row * pitch + (idx - row * per_row) * VEC) = r[i];
      }
    }
  }
};

template <typename E>
__global__ __launch_bounds__(256) void contract_kernel(ContractP P) {
  typedef TokFrag<E> TF;
  constexpr int VEC = 16 / (int)sizeof(E);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l16 = lane & 15, g4 = lane >> 4;
  const int s = blockIdx.x, grp = blockIdx.y;
  int is = 0;
  while (is + 1 < P.nsums && (int)blockIdx.z >= P.sums[is + 1].z0) ++is;
  const ContractSum& C = P.sums[is];
  const int blk = blockIdx.z - C.z0;
  const int p0 = blk / C.qc * C.pw, q0 = blk % C.qc * C.qw;
  const int pn = min(C.pw, C.p - p0), qn = min(C.qw, C.q - q0);
  const int pitch_a = pn + VEC, pitch_b = qn + VEC;
  extern __shared__ __align__(16) unsigned char smem[];
  E* As = (E*)smem;
  E* Bs = As + TT * pitch_a;
  const int n0 = s * P.span;
  const int n1 = min(n0 + P.span, P.N);
  const int npb = pn / 16, nqb = qn / 16;

  floatx4 acc[2][8];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int qb = 0; qb < 8; ++qb) acc[j][qb] = floatx4{0.f, 0.f, 0.f, 0.f};

  ContractTile<E> la, lb;
  const int tiles = n1 > n0 ? (n1 - n0 + TT - 1) / TT : 0;
  auto fetch = [&](int i) {  // tile i of the terms' tiles, one term after the other
    const ContractTerm& t = C.t[i >= tiles];
    const int t0 = n0 + (i >= tiles ? i - tiles : i) * TT;
    la.fetch((const E*)t.a + grp * t.a_sg + p0, t.a_sn, pn, t0, n1, tid);
    lb.fetch((const E*)t.b + grp * t.b_sg + q0, t.b_sn, qn, t0, n1, tid);
  };
  const int total = tiles * C.nterms;
  if (total > 0) fetch(0);
  for (int i = 0; i < total; ++i) {
    __syncthreads();  // the previous tile is no longer read
    la.store(As, pitch_a, pn, tid);
    lb.store(Bs, pitch_b, qn, tid);
    if (i + 1 < total) fetch(i + 1);
    __syncthreads();
#pragma unroll
    for (int kp = 0; kp < 2; ++kp) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int pb = w + 4 * j;
        if (pb >= npb) break;
        const auto fa = TF::get(As, pitch_a, pb * 16, kp, lane);
#pragma unroll
        for (int qb = 0; qb < 8; ++qb) {
          if (qb >= nqb) break;
          acc[j][qb] = mma32(fa, TF::get(Bs, pitch_b, qb * 16, kp, lane), acc[j][qb]);
        }
      }
    }
  }
  // acc[j][qb] lane (l16, g4) holds rows pb*16 + 4*g4 + i, column qb*16 + l16
  float* out = C.parts + (((size_t)s * P.G + grp) * C.p + p0) * (size_t)C.q + q0;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int pb = w + 4 * j;
    if (pb >= npb) break;
#pragma unroll
    for (int qb = 0; qb < 8; ++qb) {
      if (qb >= nqb) break;
#pragma unroll
      for (int i = 0; i < 4; ++i) out[(size_t)(pb * 16 + 4 * g4 + i) * C.q + qb * 16 + l16] = acc[j][qb][i];
    }
  }
}

struct ContractOut {
  void* out;
  const void* w;          // nullptr: no scaled sum
  const float* parts;     // [S][n]
  const float* w_parts;
  int64_t n;
  int blocks;             // of 256 threads, four elements each
  float scale;
};
struct ContractOutP {
  int S, nouts, out_bf16, w_bf16;
  ContractOut o[TS_CONTRACT_SUMS];
};

// out = sum_s parts[s] + scale * w * sum_s w_parts[s], in fp32, rounded once.
__global__ __launch_bounds__(256) void contract_finish_kernel(ContractOutP P) {
  int blk = blockIdx.x, io = 0;
  while (io + 1 < P.nouts && blk >= P.o[io].blocks) blk -= P.o[io++].blocks;
  const ContractOut& o = P.o[io];
  const int64_t e = ((int64_t)blk * 256 + threadIdx.x) * 4;
  if (e >= o.n) return;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 16
  for (int s = 0; s < P.S; ++s) acc += *(const floatx4*)(o.parts + s * o.n + e);
  if (o.w) {
    floatx4 wa = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 16
    for (int s = 0; s < P.S; ++s) wa += *(const floatx4*)(o.w_parts + s * o.n + e);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float w = P.w_bf16 ? tof(((const bf16*)o.w)[e + i]) : ((const float*)o.w)[e + i];
      acc[i] += o.scale * w * wa[i];
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (P.out_bf16)
      ((bf16*)o.out)[e + i] = (bf16)acc[i];
    else
      ((float*)o.out)[e + i] = acc[i];
  }
}

}  // namespace ts

namespace {

using ts::fail;

struct ContractPlan {
  int S, span;
  size_t lds, parts_bytes;
};

int plan_contract(const ts_contract_desc* d, ContractPlan* P) {
  if (!d) return fail(TS_ERR_VALUE, "contract: null descriptor");
  if (d->G < 1 || d->N < 0 || d->p < 16 || d->q < 16) return fail(TS_ERR_VALUE, "contract: bad shape");
  if (d->p % 16 || d->q % 16 || d->p > 128 || d->q > 128)
    return fail(TS_ERR_NOT_IMPLEMENTED, "contract: widths %d x %d must be multiples of 16 up to 128", d->p, d->q);
  if (d->dtype != TS_BF16 && d->dtype != TS_F32) return fail(TS_ERR_VALUE, "contract: unknown dtype");
  // slices: about two workgroups per CU (256 CUs), at least two tiles each
  const int tiles = (d->N + ts::TT - 1) / ts::TT;
  int S = 1;
  while ((long)S * 2 * d->G <= 512 && tiles >= 4 * S) S *= 2;
  const int tiles_per = (tiles + S - 1) / S;
  P->span = tiles_per * ts::TT;
  P->S = tiles > 0 ? (tiles + tiles_per - 1) / tiles_per : 1;
  const int es = d->dtype == TS_BF16 ? 2 : 4;
  const int vec = 16 / es;
  P->lds = (size_t)ts::TT * (d->p + vec + d->q + vec) * es;
  P->parts_bytes = (size_t)P->S * d->G * d->p * d->q * sizeof(float);
  return TS_OK;
}

struct SumsPlan {
  int S, span, nz;
  int pw[TS_CONTRACT_SUMS], qw[TS_CONTRACT_SUMS], qc[TS_CONTRACT_SUMS], z0[TS_CONTRACT_SUMS];
  size_t off[TS_CONTRACT_SUMS], lds, bytes;
};

int plan_sums(const ts_contract_sums_desc* d, SumsPlan* P) {
  if (!d) return fail(TS_ERR_VALUE, "contract sums: null descriptor");
  if (d->G < 1 || d->N < 0 || d->nsums < 1 || d->nsums > TS_CONTRACT_SUMS)
    return fail(TS_ERR_VALUE, "contract sums: bad shape");
  if (d->dtype != TS_BF16 && d->dtype != TS_F32) return fail(TS_ERR_VALUE, "contract sums: unknown dtype");
  const int es = d->dtype == TS_BF16 ? 2 : 4, vec = 16 / es;
  P->nz = 0;
  P->lds = 0;
  for (int i = 0; i < d->nsums; ++i) {
    const int p = d->p[i], q = d->q[i];
    if (p < 16 || q < 16 || p % 16 || q % 16 || p > 512 || q > 512)
      return fail(TS_ERR_NOT_IMPLEMENTED, "contract sums: widths %d x %d must be multiples of 16 up to 512", p, q);
    // equal blocks of at most 128 columns
    const int pc = (p + 127) / 128, qc = (q + 127) / 128;
    P->pw[i] = (p / 16 + pc - 1) / pc * 16;
    P->qw[i] = (q / 16 + qc - 1) / qc * 16;
    const int pb = (p + P->pw[i] - 1) / P->pw[i];
    P->qc[i] = (q + P->qw[i] - 1) / P->qw[i];
    P->z0[i] = P->nz;
    P->nz += pb * P->qc[i];
    const size_t lds = (size_t)ts::TT * (P->pw[i] + vec + P->qw[i] + vec) * es;
    if (lds > P->lds) P->lds = lds;
  }
  // slices: about four workgroups per CU over all sums, at least two tiles each
  const int tiles = (d->N + ts::TT - 1) / ts::TT;
  int S = 1;
  while ((long)S * 2 * d->G * P->nz <= 1024 && tiles >= 4 * S) S *= 2;
  const int per = (tiles + S - 1) / S;
  P->span = per * ts::TT;
  P->S = tiles > 0 ? (tiles + per - 1) / per : 1;
  P->bytes = 0;
  for (int i = 0; i < d->nsums; ++i) {
    P->off[i] = P->bytes;
    P->bytes += (size_t)P->S * d->G * d->p[i] * d->q[i] * sizeof(float);
  }
  return TS_OK;
}

}  // namespace

extern "C" {

int ts_contract_sums_workspace_bytes(const ts_contract_sums_desc* d, size_t* bytes) {
  SumsPlan P;
  int rc = plan_sums(d, &P);
  if (rc) return rc;
  if (bytes) *bytes = P.bytes;
  return TS_OK;
}

int ts_contract_sums(const ts_contract_sums_desc* d, const ts_contract_term* terms, const ts_contract_out* outs,
                     int32_t nouts, int32_t out_dtype, void* workspace, size_t ws_bytes, hipStream_t stream) {
  SumsPlan P;
  int rc = plan_sums(d, &P);
  if (rc) return rc;
  if (!terms || !outs || nouts < 1 || nouts > TS_CONTRACT_SUMS) return fail(TS_ERR_VALUE, "contract sums: missing tensors");
  if (out_dtype != TS_BF16 && out_dtype != TS_F32) return fail(TS_ERR_VALUE, "contract sums: unknown output dtype");
  if (!workspace || ws_bytes < P.bytes || ((uintptr_t)workspace & 15u))
    return fail(TS_ERR_VALUE, "contract sums: workspace needs %zu bytes, 16-byte aligned", P.bytes);
  const int vec = d->dtype == TS_BF16 ? 8 : 4;
  ts::ContractP p;
  memset(&p, 0, sizeof(p));
  p.G = d->G; p.N = d->N; p.span = P.span; p.nsums = d->nsums;
  const ts_contract_term* t = terms;
  for (int i = 0; i < d->nsums; ++i) {
    ts::ContractSum& c = p.sums[i];
    if (d->nterms[i] < 1 || d->nterms[i] > TS_CONTRACT_TERMS) return fail(TS_ERR_VALUE, "contract sums: bad term count");
    c.p = d->p[i]; c.q = d->q[i]; c.pw = P.pw[i]; c.qw = P.qw[i]; c.qc = P.qc[i]; c.z0 = P.z0[i];
    c.nterms = d->nterms[i];
    c.parts = (float*)((char*)workspace + P.off[i]);
    for (int j = 0; j < c.nterms; ++j, ++t) {
      if ((!t->a || !t->b) && d->N > 0) return fail(TS_ERR_VALUE, "contract sums: missing tensors");
      if (((uintptr_t)t->a & 15u) || ((uintptr_t)t->b & 15u) || t->a_sn % vec || t->b_sn % vec || t->a_sg % vec ||
          t->b_sg % vec)
        return fail(TS_ERR_VALUE, "contract sums: rows must be 16-byte aligned");
      c.t[j] = ts::ContractTerm{t->a, t->b, t->a_sg, t->a_sn, t->b_sg, t->b_sn};
    }
  }
  ts::ContractOutP o;
  memset(&o, 0, sizeof(o));
  o.S = P.S; o.nouts = nouts; o.out_bf16 = out_dtype == TS_BF16; o.w_bf16 = d->dtype == TS_BF16;
  int blocks = 0;
  for (int i = 0; i < nouts; ++i) {
    const ts_contract_out& u = outs[i];
    if (!u.out || u.sum < 0 || u.sum >= d->nsums) return fail(TS_ERR_VALUE, "contract sums: bad output");
    o.o[i].out = u.out;
    o.o[i].parts = p.sums[u.sum].parts;
    o.o[i].n = (int64_t)d->G * d->p[u.sum] * d->q[u.sum];
    if (u.w) {
      if (u.w_sum < 0 || u.w_sum >= d->nsums || d->p[u.w_sum] != d->p[u.sum] || d->q[u.w_sum] != d->q[u.sum])
        return fail(TS_ERR_VALUE, "contract sums: the scaled sum has another shape");
      o.o[i].w = u.w;
      o.o[i].w_parts = p.sums[u.w_sum].parts;
      o.o[i].scale = u.scale;
    }
    o.o[i].blocks = (int)((o.o[i].n + 1023) / 1024);
    blocks += o.o[i].blocks;
  }
  if (d->G > 65535 || P.nz > 65535) return fail(TS_ERR_NOT_IMPLEMENTED, "contract sums: grid too large");
  auto fn = d->dtype == TS_BF16 ? ts::contract_kernel<ts::bf16> : ts::contract_kernel<float>;
  if (P.lds > 65536) {
    hipError_t e = ts::ensure_lds_limit((const void*)fn, (int)P.lds);
    if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "contract sums: LDS request failed: %s", hipGetErrorString(e));
  }
  hipLaunchKernelGGL(fn, dim3((unsigned)P.S, (unsigned)d->G, (unsigned)P.nz), dim3(256), P.lds, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "contract sums: launch failed: %s", hipGetErrorString(e));
  hipLaunchKernelGGL(ts::contract_finish_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, o);
  e = hipGetLastError();
  if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "contract sums: finish launch failed: %s", hipGetErrorString(e));
  return TS_OK;
}

int ts_contract_workspace_bytes(const ts_contract_desc* d, size_t* bytes) {
  ContractPlan P;
  int rc = plan_contract(d, &P);
  if (rc) return rc;
  if (bytes) *bytes = P.parts_bytes;
  return TS_OK;
}

int ts_contract_tokens(const ts_contract_desc* d, const void* a, int64_t a_sg, int64_t a_sn, const void* b,
                       int64_t b_sg, int64_t b_sn, float* out, void* workspace, size_t ws_bytes, hipStream_t stream) {
  ContractPlan P;
  int rc = plan_contract(d, &P);
  if (rc) return rc;
  if (!a || !b || !out) return fail(TS_ERR_VALUE, "contract: missing tensors");
  const int vec = d->dtype == TS_BF16 ? 8 : 4;
  if (((uintptr_t)a & 15u) || ((uintptr_t)b & 15u) || a_sn % vec || b_sn % vec || a_sg % vec || b_sg % vec)
    return fail(TS_ERR_VALUE, "contract: rows must be 16-byte aligned");
  if (!workspace || ws_bytes < P.parts_bytes)
    return fail(TS_ERR_VALUE, "contract: workspace needs %zu bytes", P.parts_bytes);
  ts::ContractP p;
  memset(&p, 0, sizeof(p));
  p.G = d->G; p.N = d->N; p.span = P.span; p.nsums = 1;
  ts::ContractSum& c = p.sums[0];
  c.p = c.pw = d->p; c.q = c.qw = d->q; c.qc = 1; c.nterms = 1;
  c.t[0] = ts::ContractTerm{a, b, a_sg, a_sn, b_sg, b_sn};
  c.parts = (float*)workspace;
  const dim3 grid((unsigned)P.S, (unsigned)d->G);
  const void* fn = d->dtype == TS_BF16 ? (const void*)ts::contract_kernel<ts::bf16> : (const void*)ts::contract_kernel<float>;
  if (P.lds > 65536) {
    hipError_t e = ts::ensure_lds_limit(fn, (int)P.lds);
    if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "contract: LDS request failed: %s", hipGetErrorString(e));
  }
  if (d->dtype == TS_BF16)
    hipLaunchKernelGGL(ts::contract_kernel<ts::bf16>, grid, dim3(256), P.lds, stream, p);
  else
    hipLaunchKernelGGL(ts::contract_kernel<float>, grid, dim3(256), P.lds, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "contract: launch failed: %s", hipGetErrorString(e));
  return ts_sum_slots(c.parts, P.S, nullptr, 0, (int64_t)d->G * d->p * d->q, out, TS_F32, 1.0f, stream);
}

}  // extern "C"
