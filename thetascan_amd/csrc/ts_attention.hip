// Causal softmax attention, forward only (gfx950): the hybrid language
// model's softmax layers where nothing is recorded for a backward.
//
//   out[b, h, t] = sum_{s <= t} softmax_s(scale q_t . k_s) v_s
//
// bf16 [B,H,T,64] queries against [B,Hkv,T,64] keys and values (head h reads
// head h / (H / Hkv)), fp32 scores, softmax and sums; the probabilities enter
// the second product in bf16, as the operands of every MFMA here do.
//
// A workgroup owns 128 queries of a head, a wave 32 of them (two 16-query
// blocks, so each key and value fragment read from LDS feeds two MFMAs), and
// walks the keys up to its diagonal in tiles of 64: S^T = K Q^T leaves a lane
// with one query's scores (16 per block and tile), so the running maximum and
// sum are per-lane scalars with two lane swaps per tile, and the scores are
// the B operand of O^T += V^T P^T without leaving registers (V^T by the
// transposing LDS read).  Two LDS buffers: one barrier per tile, the next
// tile's rows in flight meanwhile.  Bound by the exponentials' and the
// scores' vector arithmetic (about 1.2 k cycles a tile of 32 x 64, against
// 0.5 k of MFMA).  The longest query tiles start first, so that what remains
// at the end of the launch is short.  B16 H8 (4 key/value heads) T1024:
// 36 us, against 88 us of the library's fused attention.

#include "ts_common.h"
#include "ts_tokens.h"
#include "thetascan_hip.h"

#include <string.h>

namespace ts {

struct AttnP {
  int H, rep, T;
  float scale2;  // scale * log2(e)
  ts_strided q, k, v, out;
};

constexpr int kAttnQ = 128;           // queries per workgroup
constexpr int kAttnPitch = 64 + 8;    // LDS pitch of a key or value row

__global__ __launch_bounds__(256, 3) void causal_attention_kernel(AttnP p) {
  typedef bf16 E;
  typedef LdsIO<E> IO;
  typedef TokFrag<E> TF;
  __shared__ __align__(16) E ks[2][TT * kAttnPitch];
  __shared__ __align__(16) E vs[2][TT * kAttnPitch];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l16 = lane & 15, g = lane >> 4;
  const int b = blockIdx.x / p.H, h = blockIdx.x % p.H;
  const int q0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * kAttnQ;
  const int qw = q0 + w * 32;  // this wave's first query
  const E* kb = (const E*)p.k.ptr + b * p.k.sb + (h / p.rep) * p.k.sh;
  const E* vb = (const E*)p.v.ptr + b * p.v.sb + (h / p.rep) * p.v.sh;

  // two rows' 16-byte vectors per thread of each tile; rows past T are zero
  const int lr = tid >> 3, lc = (tid & 7) * 8;
  uint4 kr[2], vr[2];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int t = k0 + lr + 32 * i;
      kr[i] = vr[i] = make_uint4(0u, 0u, 0u, 0u);
      if (t < p.T) {
        kr[i] = *(const uint4*)(kb + (int64_t)t * p.k.st + lc);
        vr[i] = *(const uint4*)(vb + (int64_t)t * p.v.st + lc);
      }
    }
  };
  fetch(0);

  // the queries as B operands (a query past T repeats the last one, unstored)
  bf16x8 qf[2][2];
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const E* qrow = (const E*)p.q.ptr + b * p.q.sb + h * p.q.sh + (int64_t)min(qw + 16 * n + l16, p.T - 1) * p.q.st;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) qf[n][kk] = __builtin_bit_cast(bf16x8, *(const uint4*)(qrow + 32 * kk + 8 * g));
  }
  floatx4 o[2][4];
  float mx[2], sum[2];
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    mx[n] = -INFINITY;
    sum[n] = 0.f;
#pragma unroll
    for (int db = 0; db < 4; ++db) o[n][db] = floatx4{0.f, 0.f, 0.f, 0.f};
  }

  const int tiles = (min(q0 + kAttnQ, p.T) + TT - 1) / TT;
  for (int it = 0; it < tiles; ++it) {
    const int k0 = it * TT, buf = it & 1;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      *(uint4*)(ks[buf] + (lr + 32 * i) * kAttnPitch + lc) = kr[i];
      *(uint4*)(vs[buf] + (lr + 32 * i) * kAttnPitch + lc) = vr[i];
    }
    if (it + 1 < tiles) fetch(k0 + TT);
    // this tile is staged; the other buffer, read in the last round, is free
    // once every wave has passed here, and is written only after it
    __syncthreads();
    if (k0 > qw + 31) continue;  // wave-uniform: the tile is past this wave's diagonal
    floatx4 s[2][4];
#pragma unroll
    for (int kf = 0; kf < 4; ++kf) {
      const E* krow = ks[buf] + (kf * 16 + l16) * kAttnPitch + 8 * g;
      const auto k_lo = IO::ld8(krow), k_hi = IO::ld8(krow + 32);
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        s[n][kf] = mma32(k_lo, qf[n][0], floatx4{0.f, 0.f, 0.f, 0.f});
        s[n][kf] = mma32(k_hi, qf[n][1], s[n][kf]);
      }
    }
    if (k0 + TT - 1 > qw) {  // wave-uniform: the diagonal crosses the tile
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const int last = qw + 16 * n + l16 - k0;  // last key of the tile this query sees
#pragma unroll
        for (int kf = 0; kf < 4; ++kf)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (kf * 16 + 4 * g + i > last) s[n][kf][i] = -INFINITY;
      }
    }
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      float m = s[n][0][0];
#pragma unroll
      for (int kf = 0; kf < 4; ++kf)
#pragma unroll
        for (int i = 0; i < 4; ++i) m = fmaxf(m, s[n][kf][i]);
      // (key 0 is seen by every query: the maximum is finite from the first tile on)
      m = fmaxf(mx[n], max_g(m));
      const float fac = __builtin_amdgcn_exp2f((mx[n] - m) * p.scale2);
      const float c = m * p.scale2;
      mx[n] = m;
      float part = 0.f;
#pragma unroll
      for (int kf = 0; kf < 4; ++kf)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[n][kf][i] = __builtin_amdgcn_exp2f(fmaf(s[n][kf][i], p.scale2, -c));
          part += s[n][kf][i];
        }
      sum[n] = fmaf(sum[n], fac, part);  // this lane's keys; the lanes are added at the end
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) o[n][db][i] *= fac;
    }
#pragma unroll
    for (int kp = 0; kp < 2; ++kp) {
      const auto p0 = IO::from_acc(s[0][2 * kp], s[0][2 * kp + 1]);
      const auto p1 = IO::from_acc(s[1][2 * kp], s[1][2 * kp + 1]);
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const auto vt = TF::get(vs[buf], kAttnPitch, db * 16, kp, lane);
        o[0][db] = mma32(vt, p0, o[0][db]);
        o[1][db] = mma32(vt, p1, o[1][db]);
      }
    }
  }
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    const int t = qw + 16 * n + l16;
    const float inv = 1.0f / sum_g(sum[n]);
    if (t < p.T) {
      E* orow = (E*)p.out.ptr + b * p.out.sb + h * p.out.sh + (int64_t)t * p.out.st + 4 * g;
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        const float r[4] = {o[n][db][0] * inv, o[n][db][1] * inv, o[n][db][2] * inv, o[n][db][3] * inv};
        st4f<E>(orow + db * 16, r);
      }
    }
  }
}

}  // namespace ts

namespace {

using ts::fail;

// Rows (feature axis contiguous) of 16-byte alignment at every stride.
bool attn_rows(const ts_strided& s) {
  return s.ptr && ((uintptr_t)s.ptr & 15u) == 0 && s.sb % 8 == 0 && s.sh % 8 == 0 && s.st % 8 == 0;
}

}  // namespace

extern "C" {

int ts_causal_attention_fwd(const ts_attention_desc* d, ts_strided q, ts_strided k, ts_strided v, ts_strided out,
                            hipStream_t stream) {
  if (!d || d->B < 1 || d->H < 1 || d->Hkv < 1 || d->H % d->Hkv || d->T < 0 || !(d->scale > 0.f))
    return fail(TS_ERR_VALUE, "attention: bad shape");
  if (d->dtype != TS_BF16 || d->d != 64) return fail(TS_ERR_NOT_IMPLEMENTED, "attention: bf16 heads of 64 only");
  if (d->T == 0) return TS_OK;
  if (!attn_rows(q) || !attn_rows(k) || !attn_rows(v) || !attn_rows(out))
    return fail(TS_ERR_VALUE, "attention: rows must be 16-byte aligned");
  const int64_t heads = (int64_t)d->B * d->H, tiles = ((int64_t)d->T + ts::kAttnQ - 1) / ts::kAttnQ;
  if (heads > 0x7fffffff || tiles > 65535) return fail(TS_ERR_NOT_IMPLEMENTED, "attention: grid too large");
  ts::AttnP p;
  memset(&p, 0, sizeof(p));
  p.H = d->H; p.rep = d->H / d->Hkv; p.T = d->T;
  p.scale2 = d->scale * 1.44269504088896340736f;
  p.q = q; p.k = k; p.v = v; p.out = out;
  hipLaunchKernelGGL(ts::causal_attention_kernel, dim3((unsigned)heads, (unsigned)tiles), dim3(256), 0, stream, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "attention: launch failed: %s", hipGetErrorString(e));
  return TS_OK;
}

}  // extern "C"
