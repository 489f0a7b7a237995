// Gradient of a causal scan with respect to a static per-head retention
// (gfx950).
//
// A scan with static retention alpha = exp(log_alpha[h]),
//   o_t = sum_{i<=t} alpha^(t-i) (q_t . k_i) v_i   (+ the key-mass column),
// has the exact derivative
//   dL/dlog_alpha = sum_t sum_{i<=t} (t-i) alpha^(t-i) (q_t . k_i) (dO_t . v_i + dm_t),
// where dm is the gradient of the mass column (v_i = 1; dm enters as two
// bf16 columns hi + lo against two unit columns).  This is the
// retention gradient the reference's autograd forms through the chunk
// backend's tile weights (scan_chunk.py:102-155, 246-339).  Written as
// sum_t t dL_t with dL_t = q_t . dq_t - k_t . dk_t, it is a small difference
// of terms about T / (1 - alpha) times larger, which bf16 scans cannot
// resolve; this kernel sums the pair terms themselves instead.
//
// A workgroup walks one segment of seg_tiles 64-token tiles of one (b, h).
// The [dk][values] states split into 16x16 blocks: wave w owns key block
// w % NKB for every S-th value block (S waves a key block, so that narrow keys
// too run eight waves; the last value block of a call with a mass column holds
// that column).  Per tile:
//   * pairs inside the tile: the ten causal 16x16 blocks of S = Q K^T, each
//     formed once by one wave on MFMA, times G = D V^T (summed over the values
//     by its MFMAs), with the weights d alpha^d, d = t - i >= 0;
//   * pairs with i in earlier tiles of the segment: with the states
//     M = sum_{i<t0} alpha^(t0-1-i) k_i v_i^T and M' = sum (t0-1-i) alpha^(..) k_i v_i^T
//     and the tile's query sums A = sum_t (tau+1) alpha^(tau+1) q_t dO_t^T,
//     B = sum_t alpha^(tau+1) q_t dO_t^T (tau = t - t0), they are
//     <M, A> + <M', B>: all four are fp32 MFMA accumulators of one layout, so
//     the products are element by element in registers.
// The weighted keys and queries enter the MFMAs as bf16 pairs hi + lo,
// hi = bf16(x), lo = bf16(x - hi), against the exact bf16 values and
// gradients: every product then carries about 16 bits, as the fp32 sums need.
// The kernel is bound by vector and matrix issue (per key and value block and
// tile 16 MFMAs and 40 vector instructions, and 290 a key block for the
// weighted pairs: vector units 52 %, MFMA 26 % busy), so every wave has a block
// and no work is repeated.  An
// earlier split by value blocks (five of eight waves busy at 64 values with a
// mass column, the query products formed against split copies of the states)
// took 163 us where this takes 97 us: B8 H8 T4096, dk 128, dv 64 + mass.
// Pairs across segments need the state entering the segment, which is not
// known here; each segment therefore also leaves its own forward summaries
// M_s, M'_s and the query-side sums A_s, B_s with n = t - segment start in the
// place of tau (summed from the tiles' A and B), and a combine
// kernel adds <M_in, A_s> + <M'_in, B_s> with M_in, M'_in the prefix of the
// summaries (M'_in composes as alpha^L (M'_in + L M_in) + M'_s).

#include "ts_common.h"
#include "ts_scan_impl.h"
#include "thetascan_hip.h"

#include <string.h>

namespace ts {

struct RetP {
  int B, H, T, dk, dv, nvr, has_mass, seg_tiles, nseg, vw;  // nvr: real value blocks; vw: padded width
  ts_strided q, k, v, dout, dm;
  uint32_t q_rec, k_rec, v_rec, o_rec, dm_rec;
  const float* log_alpha;
  float* part;  // [BH][nseg]
  float* sums;  // [BH][nseg][4][dk][vw]: M, M', A, B
};

// LDS of one workgroup: the four bf16 tiles, then fp32 weight tables.
struct RetLayout {
  int qp, vp;
  int qs, ks, vs, ds;  // element offsets (bf16)
  int fbase;           // float offset of the tables
  int bytes;
};
// table offsets (floats from fbase)
constexpr int kTabD = 0;      // [128] at 64 + d: d alpha^d for d >= 0, 0 for d < 0
constexpr int kTabRA = 128;   // [64] (tau+1) alpha^(tau+1)
constexpr int kTabRB = 192;   // [64] alpha^(tau+1)
constexpr int kTabPow = 256;  // [68] alpha^d, d = 0..64
constexpr int kTabWM = 324;   // [64] this tile's alpha^(len-1-tok), 0 past len
constexpr int kTabWMp = 388;  // [64] (len-1-tok) alpha^(len-1-tok)
constexpr int kTabRed = 452;  // [8]
constexpr int kTabFloats = 460;

__host__ __device__ constexpr RetLayout ret_layout(int DK, int vw) {
  RetLayout L{};
  L.qp = DK + 8;
  L.vp = vw + 8;
  L.qs = 0;
  L.ks = L.qs + C * L.qp;
  L.vs = L.ks + C * L.qp;
  L.ds = L.vs + C * L.vp;
  const int e_end = L.ds + C * L.vp;
  const int e_bytes = (e_end * 2 + 15) / 16 * 16;
  L.fbase = e_bytes / 4;
  L.bytes = e_bytes + kTabFloats * 4;
  return L;
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));

// Two floats rounded to bf16 (RNE) in one dword, a in the low half.
__device__ __forceinline__ uint32_t pk2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{a, b}, bf16x2));
}

// x = hi + lo to about 16 bits for eight values: hi = bf16(x), lo = bf16(x - hi).
__device__ __forceinline__ void split8(const float (&x)[8], bf16x8& hi, bf16x8& lo) {
  uint32_t h[4], l[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    h[j] = pk2(x[2 * j], x[2 * j + 1]);
    l[j] = pk2(x[2 * j] - __uint_as_float(h[j] << 16), x[2 * j + 1] - __uint_as_float(h[j] & 0xffff0000u));
  }
  hi = __builtin_bit_cast(bf16x8, make_uint4(h[0], h[1], h[2], h[3]));
  lo = __builtin_bit_cast(bf16x8, make_uint4(l[0], l[1], l[2], l[3]));
}

// bf16 element e of a fragment as float
__device__ __forceinline__ float elt(bf16x8 v, int e) { return tof(v[e]); }

// The eight tokens of a col8 fragment x (kp, lane group g) times a table's
// weights, as hi + lo.
__device__ __forceinline__ void weigh8(bf16x8 x, const float* t, int kp, int g, bf16x8& hi, bf16x8& lo) {
  const floatx4 a = *(const floatx4*)(t + 32 * kp + 4 * g);
  const floatx4 b = *(const floatx4*)(t + 32 * kp + 16 + 4 * g);
  float y[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    y[i] = elt(x, i) * a[i];
    y[4 + i] = elt(x, 4 + i) * b[i];
  }
  split8(y, hi, lo);
}

// (query block, key block) pairs of the causal tile, key block <= query block
__constant__ int kPairs[10][2] = {{0, 0}, {1, 0}, {1, 1}, {2, 0}, {2, 1}, {2, 2}, {3, 0}, {3, 1}, {3, 2}, {3, 3}};

// Waves that share a key block: as many as keep a workgroup at eight waves.
constexpr int ret_share(int dk) { return 128 / dk; }

template <int DK, int NVB>
__global__ __launch_bounds__(64 * (DK / 16) * ret_share(DK)) void retention_grad_kernel(RetP p) {
  typedef bf16 E;
  typedef Tok<E> TK;
  constexpr int NK32 = DK / 32;
  constexpr bool KTAIL = (DK % 32) != 0;
  constexpr int NKB = DK / 16;
  constexpr int QC = DK / 8;  // 16-byte chunks per key row
  constexpr int S = ret_share(DK), nwave = NKB * S, bd = 64 * nwave;
  constexpr int NQ = (C * QC + bd - 1) / bd;                // chunks of a query or key tile per thread
  constexpr int NW = NVB * S, vw = NW * 16;                 // value blocks (the host rounds up; the rest are zeros)
  constexpr int NV = (C * 2 * NW + bd - 1) / bd;            // chunks of a value or gradient tile per thread
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4,
            l16 = lane & 15;
  const int kb = w % NKB, vs = w / NKB;  // this wave's blocks: keys kb, values vs, vs + S, ..
  const int seg = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int bh = b * p.H + h;
  constexpr RetLayout L = ret_layout(DK, vw);
  extern __shared__ __align__(16) unsigned char smem[];
  E* base = (E*)smem;
  E* Qs = base + L.qs;
  E* Ks = base + L.ks;
  E* Vs = base + L.vs;
  E* Ds = base + L.ds;
  float* tab = (float*)smem + L.fbase;

  const float la = p.log_alpha[h];
  for (int i = tid; i < 128; i += bd) {
    const int d = i - 64;
    tab[kTabD + i] = d >= 0 ? (float)d * expf(la * (float)d) : 0.f;
  }
  for (int i = tid; i < 65; i += bd) tab[kTabPow + i] = expf(la * (float)i);
  for (int i = tid; i < 64; i += bd) {
    const float a = expf(la * (float)(i + 1));
    tab[kTabRA + i] = (float)(i + 1) * a;
    tab[kTabRB + i] = a;
  }

  const int nchunks = (p.T + C - 1) / C;
  const int c0 = seg * p.seg_tiles;
  const int c1 = min(c0 + p.seg_tiles, nchunks);
  const int q_st = (int)p.q.st * 2, k_st = (int)p.k.st * 2, v_st = (int)p.v.st * 2, o_st = (int)p.dout.st * 2;
  const rsrc_t q_rs = make_rsrc(bh_base(p.q, b, h, 2), p.q_rec);
  const rsrc_t k_rs = make_rsrc(bh_base(p.k, b, h, 2), p.k_rec);
  const rsrc_t v_rs = make_rsrc(bh_base(p.v, b, h, 2), p.v_rec);
  const rsrc_t o_rs = make_rsrc(bh_base(p.dout, b, h, 2), p.o_rec);
  const rsrc_t dm_rs = make_rsrc(bh_base(p.dm, b, h, 4), p.dm_rec);
  const int vr = p.nvr * 16;  // real (padded) value columns; the mass block follows

  // the states and the segment's query sums, rows (keys) kb*16 + 4g + i,
  // column (value) (vs + n S)*16 + l16
  floatx4 M[NVB], Mp[NVB], A[NVB], Bq[NVB];
#pragma unroll
  for (int n = 0; n < NVB; ++n) M[n] = Mp[n] = A[n] = Bq[n] = floatx4{0.f, 0.f, 0.f, 0.f};
  float acc = 0.f;

  // tile c's loads go to registers while tile c - 1 is computed
  uint4 rq[NQ], rk[NQ], rv[NV], rd[NV];
  float rdm[NV];
  auto fetch = [&](int c) {
    const int t0 = c * C;
#pragma unroll
    for (int r = 0; r < NQ; ++r) {
      const int idx = tid + r * bd;
      const int row = idx / QC, col = (idx % QC) * 8;
      const bool on = idx < C * QC;
      rq[r] = bld16(q_rs, on ? (uint32_t)((t0 + row) * q_st + col * 2) : kOOB);
      rk[r] = bld16(k_rs, on ? (uint32_t)((t0 + row) * k_st + col * 2) : kOOB);
    }
#pragma unroll
    for (int r = 0; r < NV; ++r) {
      const int idx = tid + r * bd;
      const int row = idx / (2 * NW), col = (idx % (2 * NW)) * 8;
      const bool in = idx < C * 2 * NW, on = in && col < p.dv;
      rv[r] = bld16(v_rs, on ? (uint32_t)((t0 + row) * v_st + col * 2) : kOOB);
      rd[r] = bld16(o_rs, on ? (uint32_t)((t0 + row) * o_st + col * 2) : kOOB);
      const bool mass = in && col == vr && p.has_mass && t0 + row < p.T;
      rdm[r] = bldf(dm_rs, mass ? (uint32_t)((t0 + row) * (int)p.dm.st * 4) : kOOB);
    }
  };
  if (c0 < c1) fetch(c0);

  for (int c = c0; c < c1; ++c) {
    const int t0 = c * C;
    const int len = min(C, p.T - t0);
    __syncthreads();  // the previous tile's operands and tables are consumed
    {
#pragma unroll
      for (int r = 0; r < NQ; ++r) {
        const int idx = tid + r * bd;
        if (idx < C * QC) {
          const int row = idx / QC, col = (idx % QC) * 8;
          *(uint4*)(Qs + row * L.qp + col) = rq[r];
          *(uint4*)(Ks + row * L.qp + col) = rk[r];
        }
      }
#pragma unroll
      for (int r = 0; r < NV; ++r) {
        const int idx = tid + r * bd;
        const int row = idx / (2 * NW), col = (idx % (2 * NW)) * 8;
        if (idx < C * 2 * NW) {
          uint4 vv = rv[r], dd = rd[r];
          if (col == vr && p.has_mass) {
            // two unit V columns against dm as bf16 hi + lo
            const bool valid = t0 + row < p.T;
            const uint32_t one = valid ? 0x3f803f80u : 0u;  // bf16 1.0 twice
            const uint32_t dh = pk2(rdm[r], 0.f);
            const float hi = __uint_as_float(dh << 16);
            vv = make_uint4(one, 0u, 0u, 0u);
            dd = make_uint4(pk2(hi, rdm[r] - hi), 0u, 0u, 0u);
          }
          *(uint4*)(Vs + row * L.vp + col) = vv;
          *(uint4*)(Ds + row * L.vp + col) = dd;
        }
      }
      // this tile's weights
      if (tid < 64) {
        const int tok = tid, d = len - 1 - tok;
        const float pw = d >= 0 ? tab[kTabPow + max(d, 0)] : 0.f;
        tab[kTabWM + tok] = pw;
        tab[kTabWMp + tok] = (float)d * pw;
      }
    }
    __syncthreads();
    if (c + 1 < c1) fetch(c + 1);

    // ---- pairs inside the tile: each score block once, against D V^T
    for (int pi = w; pi < 10; pi += nwave) {
      const int tb = kPairs[pi][0], ib = kPairs[pi][1];
      floatx4 sc = {0.f, 0.f, 0.f, 0.f}, gg = sc;
#pragma unroll
      for (int j = 0; j < NK32; ++j)
        sc = mma32(frow8<E>(Qs, L.qp, tb * 16 + l16, j, g), frow8<E>(Ks, L.qp, ib * 16 + l16, j, g), sc);
      if (KTAIL) sc = mma16(frow4<E>(Qs, L.qp, tb * 16 + l16, NK32, g), frow4<E>(Ks, L.qp, ib * 16 + l16, NK32, g), sc);
#pragma unroll
      for (int j = 0; j < NW / 2; ++j)
        gg = mma32(frow8<E>(Ds, L.vp, tb * 16 + l16, j, g), frow8<E>(Vs, L.vp, ib * 16 + l16, j, g), gg);
      if (NW & 1)
        gg = mma16(frow4<E>(Ds, L.vp, tb * 16 + l16, NW / 2, g), frow4<E>(Vs, L.vp, ib * 16 + l16, NW / 2, g), gg);
      // rows (queries) tb*16 + 4g + i, columns (keys) ib*16 + l16; d = t - i
      const float* dt = tab + kTabD + 64 + (tb - ib) * 16 + 4 * g - l16;
#pragma unroll
      for (int i = 0; i < 4; ++i) acc += dt[i] * sc[i] * gg[i];
    }

    // ---- this tile's query sums against the states of the earlier tiles, and
    // into the segment's (their weights start at the segment: off tokens back)
    {
      bf16x8 ah[2], al[2], bh8[2], bl8[2];
#pragma unroll
      for (int kp = 0; kp < 2; ++kp) {
        const bf16x8 q8 = TK::col8(Qs, L.qp, kb * 16, kp, lane);
        weigh8(q8, tab + kTabRA, kp, g, ah[kp], al[kp]);
        weigh8(q8, tab + kTabRB, kp, g, bh8[kp], bl8[kp]);
      }
      const float off = (float)((c - c0) * C), aoff = expf(la * off), aoff1 = aoff * off;
#pragma unroll
      for (int n = 0; n < NVB; ++n) {
        const int vb = vs + n * S;
        floatx4 at = {0.f, 0.f, 0.f, 0.f}, bt = at;
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
          const bf16x8 d8 = TK::col8(Ds + vb * 16, L.vp, 0, kp, lane);
          at = mma32(ah[kp], d8, at);
          at = mma32(al[kp], d8, at);
          bt = mma32(bh8[kp], d8, bt);
          bt = mma32(bl8[kp], d8, bt);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc += M[n][i] * at[i] + Mp[n][i] * bt[i];
          A[n][i] += aoff * at[i] + aoff1 * bt[i];
          Bq[n][i] += aoff * bt[i];
        }
      }
    }
    // ---- states after this tile (relative to its last token)
    {
      bf16x8 mh[2], ml[2], mph[2], mpl[2];
#pragma unroll
      for (int kp = 0; kp < 2; ++kp) {
        const bf16x8 k8 = TK::col8(Ks, L.qp, kb * 16, kp, lane);
        weigh8(k8, tab + kTabWM, kp, g, mh[kp], ml[kp]);
        weigh8(k8, tab + kTabWMp, kp, g, mph[kp], mpl[kp]);
      }
      const float dec = tab[kTabPow + len], dec1 = dec * (float)len;
#pragma unroll
      for (int n = 0; n < NVB; ++n) {
        const int vb = vs + n * S;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          Mp[n][i] = dec * Mp[n][i] + dec1 * M[n][i];
          M[n][i] *= dec;
        }
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
          const bf16x8 v8 = TK::col8(Vs + vb * 16, L.vp, 0, kp, lane);
          M[n] = mma32(mh[kp], v8, M[n]);
          M[n] = mma32(ml[kp], v8, M[n]);
          Mp[n] = mma32(mph[kp], v8, Mp[n]);
          Mp[n] = mma32(mpl[kp], v8, Mp[n]);
        }
      }
    }
  }

  // ---- this segment's pair sum and summaries
  float* red = tab + kTabRed;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) acc += __shfl_xor(acc, o, 64);
  if (lane == 0) red[w] = acc;
  __syncthreads();
  if (tid == 0) {
    float s = 0.f;
    for (int i = 0; i < nwave; ++i) s += red[i];
    p.part[(size_t)bh * p.nseg + seg] = s;
  }
  // the first segment has no state before it, the last no segment after it
  const size_t nel = (size_t)p.dk * vw;
  float* out = p.sums + ((size_t)bh * p.nseg + seg) * 4 * nel;
#pragma unroll
  for (int n = 0; n < NVB; ++n)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const size_t e = (size_t)(kb * 16 + 4 * g + i) * vw + (vs + n * S) * 16 + l16;
      if (seg + 1 < p.nseg) {
        out[e] = M[n][i];
        out[nel + e] = Mp[n][i];
      }
      if (seg > 0) {
        out[2 * nel + e] = A[n][i];
        out[3 * nel + e] = Bq[n][i];
      }
    }
}

__global__ void retention_zero_kernel(float* out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = 0.f;
}

// Cross-segment pairs: <M_in, A_s> + <M'_in, B_s> with the running prefix of
// the segment summaries.  Block (x, bh) takes elements x*256 .. +255 of the
// [dk][vw] states and writes its partial sum; the finish kernel adds the
// partials and the segments' own pair sums -> out[b][h].
__global__ __launch_bounds__(256) void retention_combine_kernel(RetP p, float* partials) {
  const int bh = blockIdx.y;
  const int h = bh % p.H;
  const float la = p.log_alpha[h];
  const size_t nel = (size_t)p.dk * p.vw;
  const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int seg_len = p.seg_tiles * C;
  float acc = 0.f;
  if (e < nel) {
    float m = 0.f, mp = 0.f;
    // every segment but the last is whole
    const float aL = expf(la * (float)seg_len);
#pragma unroll 4
    for (int s = 1; s < p.nseg; ++s) {
      const float* base = p.sums + ((size_t)bh * p.nseg + s - 1) * 4 * nel + e;
      mp = aL * (mp + (float)seg_len * m) + base[nel];
      m = aL * m + base[0];
      acc += m * base[6 * nel] + mp * base[7 * nel];
    }
  }
  __shared__ float red[4];
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) acc += __shfl_xor(acc, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) partials[(size_t)bh * gridDim.x + blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

__global__ __launch_bounds__(64) void retention_finish_kernel(RetP p, const float* partials, int nparts, float* out) {
  const int bh = blockIdx.x;
  float s = 0.f;
  for (int i = threadIdx.x; i < nparts; i += 64) s += partials[(size_t)bh * nparts + i];
  for (int i = threadIdx.x; i < p.nseg; i += 64) s += p.part[(size_t)bh * p.nseg + i];
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) s += __shfl_xor(s, o, 64);
  if (threadIdx.x == 0) out[bh] = s;
}

}  // namespace ts

namespace {

using ts::fail;

typedef void (*RetFn)(ts::RetP);

// Value blocks of a kernel with room for nw: 4, 5 (64 values and a mass
// column) or 8, in whole multiples of the waves that share a key block.
int ret_blocks(int dk, int nw) {
  const int S = ts::ret_share(dk), n = nw <= 4 ? 4 : nw <= 5 ? 5 : 8;
  return (n + S - 1) / S * S;
}

template <int DK>
RetFn pick_ret_dk(int nw) {
  constexpr int S = ts::ret_share(DK);
  return nw <= (4 + S - 1) / S * S   ? ts::retention_grad_kernel<DK, (4 + S - 1) / S>
         : nw <= (5 + S - 1) / S * S ? ts::retention_grad_kernel<DK, (5 + S - 1) / S>
                                     : ts::retention_grad_kernel<DK, 8 / S>;
}

RetFn pick_ret(int dk, int nw) {
  switch (dk) {
    case 16: return pick_ret_dk<16>(nw);
    case 32: return pick_ret_dk<32>(nw);
    case 48: return pick_ret_dk<48>(nw);
    case 64: return pick_ret_dk<64>(nw);
    case 80: return pick_ret_dk<80>(nw);
    case 96: return pick_ret_dk<96>(nw);
    case 112: return pick_ret_dk<112>(nw);
    case 128: return pick_ret_dk<128>(nw);
  }
  return nullptr;
}

struct RetPlan {
  int dkp, nvr, vw, nw, waves, seg_tiles, nseg;
  int ncomb;  // combine blocks per (b, h): 256 state elements each
  size_t part_bytes, sums_bytes, comb_bytes;
};

int ret_plan(const ts_retention_desc* d, RetPlan* P) {
  if (!d) return fail(TS_ERR_VALUE, "retention grad: null descriptor");
  if (d->B < 1 || d->H < 1 || d->T < 0 || d->dk < 1 || d->dv < 1)
    return fail(TS_ERR_VALUE, "retention grad: bad shape");
  if (d->dtype != TS_BF16) return fail(TS_ERR_NOT_IMPLEMENTED, "retention grad: bf16 streams only");
  if (d->dk > 128 || d->dk % 16 || d->dv % 8)
    return fail(TS_ERR_NOT_IMPLEMENTED,
                "retention grad: dk a multiple of 16 up to 128, dv a multiple of 8 (split wider keys)");
  P->dkp = d->dk;
  P->nvr = (d->dv + 15) / 16;
  P->nw = P->nvr + (d->has_mass ? 1 : 0);
  if (P->nw > 8) return fail(TS_ERR_NOT_IMPLEMENTED, "retention grad: at most 8 value blocks per call (split wider values)");
  P->nw = ret_blocks(d->dk, P->nw);
  P->vw = P->nw * 16;
  P->waves = d->dk / 16 * ts::ret_share(d->dk);
  if (ts::ret_layout(P->dkp, P->vw).bytes > ts::kLdsPerCU)
    return fail(TS_ERR_NOT_IMPLEMENTED, "retention grad: tiles of dk=%d and %d value columns exceed LDS (split the values)",
                P->dkp, P->vw);
  const int tiles = (d->T + ts::C - 1) / ts::C;
  int st = d->seg_tiles;
  if (st <= 0) {
    // at most 256 workgroups, one per CU, since more and shorter segments cost
    // more in summaries than they hide (B8 H8 T4096, dk 128, 64 values + mass:
    // 97 us against 117 us at 512; dk 32: 70 against 77); 512 for 16 keys,
    // whose summaries are small and several of whose workgroups share a CU
    // (56 us against 61 us).  Segments of at least two tiles.
    const long most = d->dk <= 16 ? 512 : 256;
    st = 2;
    while (st < tiles && (long)d->B * d->H * ((tiles + st - 1) / st) > most) st *= 2;
  }
  P->seg_tiles = st;
  P->nseg = tiles > 0 ? (tiles + st - 1) / st : 0;
  P->part_bytes = (size_t)d->B * d->H * P->nseg * sizeof(float);
  P->sums_bytes = (size_t)d->B * d->H * P->nseg * 4 * (size_t)P->dkp * P->vw * sizeof(float);
  P->ncomb = (P->dkp * P->vw + 255) / 256;
  P->comb_bytes = (size_t)d->B * d->H * P->ncomb * sizeof(float);
  return TS_OK;
}

// workspace: [part | pad to 256 | sums | pad to 256 | combine partials]
size_t ws_bytes(const RetPlan& P) {
  return (P.part_bytes + 255) / 256 * 256 + (P.sums_bytes + 255) / 256 * 256 + P.comb_bytes;
}

// Bytes spanned by one (batch, head) slice of a [.., T, width] stream (the
// range of its buffer loads), or an error if the rows the kernel addresses --
// up to T rounded up to whole tiles, plus one tile -- could not be reached with
// 31-bit offsets (the tile offsets are computed in 32-bit integers).
int span_bytes(const char* name, const ts_strided& s, int T, int width, int es, uint32_t* out) {
  *out = 0;
  if (!s.ptr || T == 0) return TS_OK;
  if (s.st < 0) return fail(TS_ERR_VALUE, "retention grad: negative time stride of %s", name);
  const int64_t rows = ((int64_t)T + ts::C - 1) / ts::C * ts::C + ts::C;
  const int64_t reach = rows * s.st * es + (int64_t)width * es;
  if (reach >= ((int64_t)1 << 31))
    return fail(TS_ERR_NOT_IMPLEMENTED, "retention grad: one (batch, head) slice of %s spans more than 2 GiB", name);
  *out = (uint32_t)(((int64_t)(T - 1) * s.st + width) * es);
  return TS_OK;
}

}  // namespace

extern "C" {

int ts_retention_workspace_bytes(const ts_retention_desc* d, size_t* bytes) {
  RetPlan P;
  int rc = ret_plan(d, &P);
  if (rc) return rc;
  if (bytes) *bytes = ws_bytes(P);
  return TS_OK;
}

int ts_retention_grad(const ts_retention_desc* d, const ts_retention_io* io, float* out, void* workspace,
                      size_t workspace_bytes, hipStream_t stream) {
  RetPlan P;
  int rc = ret_plan(d, &P);
  if (rc) return rc;
  if (!io || !out || !io->log_alpha || !io->q.ptr || !io->k.ptr || !io->v.ptr || !io->dout.ptr)
    return fail(TS_ERR_VALUE, "retention grad: missing tensors");
  if (d->has_mass && !io->dmass.ptr) return fail(TS_ERR_VALUE, "retention grad: missing dmass");
  for (const ts_strided* s : {&io->q, &io->k, &io->v, &io->dout})
    if (((uintptr_t)s->ptr & 15u) || s->st % 8 || s->sh % 8 || s->sb % 8)
      return fail(TS_ERR_VALUE, "retention grad: streams need 16-byte aligned rows");
  // every slice must be addressable with 31-bit offsets (checked before any launch)
  uint32_t rec[5];
  if ((rc = span_bytes("q", io->q, d->T, d->dk, 2, &rec[0])) || (rc = span_bytes("k", io->k, d->T, d->dk, 2, &rec[1])) ||
      (rc = span_bytes("v", io->v, d->T, d->dv, 2, &rec[2])) ||
      (rc = span_bytes("dout", io->dout, d->T, d->dv, 2, &rec[3])) ||
      (rc = span_bytes("dmass", io->dmass, d->T, 1, 4, &rec[4])))
    return rc;
  const size_t need = ws_bytes(P);
  if (!workspace || workspace_bytes < need || ((uintptr_t)workspace & 15u))
    return fail(TS_ERR_VALUE, "retention grad: workspace needs %zu bytes, 16-byte aligned", need);
  const int bh = d->B * d->H;
  if (d->T == 0) {
    hipLaunchKernelGGL(ts::retention_zero_kernel, dim3((bh + 255) / 256), dim3(256), 0, stream, out, bh);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? TS_OK : fail(TS_ERR_RUNTIME, "retention grad: launch failed: %s", hipGetErrorString(e));
  }
  ts::RetP p;
  memset(&p, 0, sizeof(p));
  p.B = d->B; p.H = d->H; p.T = d->T; p.dk = P.dkp; p.dv = d->dv; p.nvr = P.nvr; p.has_mass = d->has_mass;
  p.seg_tiles = P.seg_tiles; p.nseg = P.nseg; p.vw = P.vw;
  p.q = io->q; p.k = io->k; p.v = io->v; p.dout = io->dout; p.dm = io->dmass;
  p.q_rec = rec[0]; p.k_rec = rec[1]; p.v_rec = rec[2]; p.o_rec = rec[3]; p.dm_rec = rec[4];
  p.log_alpha = io->log_alpha;
  p.part = (float*)workspace;
  p.sums = (float*)((char*)workspace + (P.part_bytes + 255) / 256 * 256);
  RetFn fn = pick_ret(P.dkp, P.nw);
  if (!fn) return fail(TS_ERR_NOT_IMPLEMENTED, "retention grad: no kernel for dk=%d", P.dkp);
  const ts::RetLayout L = ts::ret_layout(P.dkp, P.vw);
  if (L.bytes > 65536) {
    hipError_t e = ts::ensure_lds_limit((const void*)fn, L.bytes);
    if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "retention grad: LDS request failed: %s", hipGetErrorString(e));
  }
  hipLaunchKernelGGL(fn, dim3(P.nseg, d->H, d->B), dim3(64 * P.waves), (size_t)L.bytes, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "retention grad: launch failed: %s", hipGetErrorString(e));
  float* comb = (float*)((char*)p.sums + (P.sums_bytes + 255) / 256 * 256);
  hipLaunchKernelGGL(ts::retention_combine_kernel, dim3(P.ncomb, bh), dim3(256), 0, stream, p, comb);
  e = hipGetLastError();
  if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "retention grad: combine launch failed: %s", hipGetErrorString(e));
  hipLaunchKernelGGL(ts::retention_finish_kernel, dim3(bh), dim3(64), 0, stream, p, (const float*)comb, P.ncomb, out);
  e = hipGetLastError();
  if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "retention grad: finish launch failed: %s", hipGetErrorString(e));
  return TS_OK;
}

}  // extern "C"
