// Backward scans of several retentions of one q, k, v in two passes (gfx950).
//
// For views r with static retentions alpha_r (1: the plain sum), upstream
// gradients dO_r [T][dv] and, with a key mass, dm_r [T]:
//   dq_t = sum_r sum_{i<=t} alpha_r^(t-i) (dO_r,t . v_i + dm_r,t) k_i
//   dk_i = sum_r sum_{t>=i} alpha_r^(t-i) (dO_r,t . v_i + dm_r,t) q_t
//   dv_i = sum_r sum_{t>=i} alpha_r^(t-i) (q_t . k_i) dO_r,t
// (the gradients autograd forms through scan_chunk.py:246-339).  Each sum over
// views stays in the accumulators: one causal pass for dq, one anti-causal
// pass for dk and dv, results rounded once to bf16.  As scans of one view
// each, three views took nine scans that stored and re-read fp32 partial
// gradients of the width of q (B8 H8 T4096: 402 MB per pass at 384 features).
//
// Work: one workgroup of four waves per (segment, batch*head, 64-column slice
// of the m features); wave w owns query block w and value block w of its slice
// (ts_scan.hip describes the tile).  Both passes have dO / v as 64-wide keys
// and the features as values, so every view's state is [64][64] for any m.
//   dq:     queries dO_r (per view), keys v, values k[slice]; the scores of all
//           views are weighted and summed in fp32, go to bf16 as hi + lo and
//           feed one contraction with the values.
//   dk, dv: queries v, keys dO_r (per view), values q[slice]; dv takes the same
//           states transposed (ds_read_b64_tr_b16) and the scores q . k of this
//           slice's features, whose partial dv the slices leave in fp32 for
//           one sum (m <= 64: the only slice writes dv itself).
// The key mass enters as the rank-1 ext pair of ts_scan.hip: dq's queries
// carry dm_r against a ones column of the keys, dk's keys dm_r against a ones
// column of the queries, with the state row u_r = sum of the weighted values.
//
// Bound: at m = 64 the tile's dependency chain (LDS reads and MFMAs between
// two barriers, two workgroups per CU), above that the matrix and LDS work of
// the slices (dO and v are re-read from L2).  B8 H8 T4096, three views with
// mass, both passes with their summaries: m = 64 231 us (per-view scans: about
// 620 us with the conversions of the fp32 gradients); m = 384 1.10 ms with the
// sum of the dv partials (about 2.9 ms).

#include "ts_common.h"
#include "ts_scan_impl.h"
#include "thetascan_hip.h"

#include <string.h>

namespace ts {

struct VbwdP {
  ScanP s;  // B, H, T, nchunks, seg_chunks, nseg, nsum, reverse
  int m, dv, nsl, mass, has_b;
  const float* log_alpha[TS_MAX_VIEWS];
  ts_strided dout[TS_MAX_VIEWS], dm[TS_MAX_VIEWS];  // per view: queries (dq) or keys (dk, dv)
  ts_strided v;                                     // keys (dq) or queries (dk, dv)
  ts_strided val;                                   // values: k (dq) or q (dk, dv)
  ts_strided kf;                                    // dk, dv: the features k, scored against q for dv
  ts_strided out, outb;                             // dq or dk; dv
  uint32_t o_rec[TS_MAX_VIEWS], dm_rec[TS_MAX_VIEWS], v_rec, val_rec, kf_rec, out_rec, outb_rec;
  float* part;     // dv partials [nsl][B*H][T][dv] fp32 (nsl > 1), else null
  float* seg;      // [view][lane][nseg][kNelem], lane = slice * B*H + bh
  float* segdec;   // [view][lane][nseg]
  size_t seg_vstride, dec_vstride;
};

constexpr int kD = 64;                  // padded width of dO and v
constexpr int kNelem = kD * 64 + 64;    // S [key][64 values], u [64]
constexpr int kTabPitch = 128;

// LDS (bf16 pitch 72): key tiles [nk][64][72], values [64][72], state copies
// [NV][64][72] (main); fp32: alpha^d [NV][68], the masked powers
// [NV][4][128] (ts_scan_views.hip), u [NV][64], key ext [NV][64].
struct VbwdLayout {
  int pitch, tile, vs, st, fbase, bytes;
};
__host__ __device__ constexpr VbwdLayout vbwd_layout(int NV, bool per_view_keys, bool main_kernel) {
  VbwdLayout L{};
  L.pitch = kD + 8;
  L.tile = C * L.pitch;
  const int nk = per_view_keys ? NV : 1;
  L.vs = nk * L.tile;
  L.st = L.vs + L.tile;
  const int e_bytes = (L.st + (main_kernel ? NV * L.tile : 0)) * 2;
  L.fbase = e_bytes / 4;
  L.bytes = e_bytes + NV * (68 + 4 * kTabPitch + 64 + 64) * 4;
  return L;
}

// f(d0 .. d0 + 3) of one view's masked powers: alpha^d for 0 <= d <= 64, else 0
__device__ __forceinline__ floatx4 vbwd_window(const float* pwx, int d0) {
  const int j = d0 + 64;
  const int sft = j & 3;
  return *(const floatx4*)(pwx + sft * kTabPitch + (j - sft));
}

// One [64 x 64] bf16 tile in registers (two 16-byte vectors per thread).
struct VTile {
  uint4 r[2];
  __device__ __forceinline__ void fetch(const ScanP& p, rsrc_t data, int t0, int st_b, int width, int tid) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + i * 256, row = idx >> 3, c0 = (idx & 7) * 8;
      r[i] = bld16(data, c0 < width ? row_off(p, t0, row, st_b) + (uint32_t)(c0 * 2) : kOOB);
    }
  }
  __device__ __forceinline__ void store(bf16* dst, int pitch, int tid) const {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = tid + i * 256;
      *(uint4*)(dst + (idx >> 3) * pitch + (idx & 7) * 8) = r[i];
    }
  }
};

// KV false: the dq pass; true: the dk, dv pass (reverse).
template <int NV, bool KV, bool MAIN>
__global__ __launch_bounds__(256, 2) void views_bwd_kernel(VbwdP vp) {
  typedef bf16 E;
  typedef bf16x8 F8;
  typedef LdsIO<E> IO;
  typedef Tok<E> TK;
  constexpr int NK = KV ? NV : 1;   // key tiles
  constexpr int NQ = KV ? 1 : NV;   // query fragments
  const ScanP& p = vp.s;
  const bool mass = vp.mass != 0;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4;
  const int l16 = lane & 15;
  const int seg = blockIdx.x;
  const int bh = blockIdx.y;
  const int b = bh / p.H;
  const int h = bh - b * p.H;
  const int col0 = blockIdx.z * 64;
  const int vcols = min(64, vp.m - col0);
  const size_t ln = (size_t)blockIdx.z * gridDim.y + bh;

  constexpr VbwdLayout L = vbwd_layout(NV, KV, MAIN);
  constexpr int P = L.pitch;
  extern __shared__ __align__(16) unsigned char smem[];
  E* Ks = (E*)smem;
  E* Vs = Ks + L.vs;
  E* st_base = Ks + L.st;
  float* s_pw = (float*)smem + L.fbase;     // [NV][68]
  float* s_pwx = s_pw + NV * 68;            // [NV][4][kTabPitch]
  float* s_u = s_pwx + NV * 4 * kTabPitch;  // [NV][64]
  float* s_ke = s_u + NV * 64;              // [NV][64]

  const rsrc_t v_rs = make_rsrc(bh_base(vp.v, b, h, 2), vp.v_rec);
  const rsrc_t val_rs = make_rsrc((const char*)bh_base(vp.val, b, h, 2) + col0 * 2, vp.val_rec - (uint32_t)(col0 * 2));
  const int v_st_b = (int)vp.v.st * 2, val_st_b = (int)vp.val.st * 2;

  float la[NV];
#pragma unroll
  for (int r = 0; r < NV; ++r) la[r] = vp.log_alpha[r] ? vp.log_alpha[r][h] : 0.0f;
  if (w == 0) {
#pragma unroll
    for (int r = 0; r < NV; ++r) {
      s_pw[r * 68 + lane] = expf(la[r] * (float)lane);
      if (lane == 0) s_pw[r * 68 + 64] = expf(la[r] * 64.0f);
    }
  }
  for (int e = tid; e < NV * 4 * kTabPitch; e += 256) {
    const int r = e / (4 * kTabPitch), rem = e - r * 4 * kTabPitch;
    const int sft = rem / kTabPitch, j = rem - sft * kTabPitch;
    const int d = j + sft - 64;
    float a = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) a = r == i ? la[i] : a;
    s_pwx[e] = d >= 0 && d <= 64 ? expf(a * (float)d) : 0.0f;
  }

  // ---- states: S[r][kb] rows key kb*16+4g+i, column value w*16+l16; u of that block
  floatx4 S[NV][4], us[NV];
#pragma unroll
  for (int r = 0; r < NV; ++r) {
    us[r] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) S[r][kb] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  const int c_begin = seg * p.seg_chunks;
  const int c_end = min(c_begin + p.seg_chunks, p.nchunks);
  bool state_zero = true;
  if (MAIN && seg > 0) {
    state_zero = false;
#pragma unroll
    for (int r = 0; r < NV; ++r) {
      const float* src = vp.seg + r * vp.seg_vstride + (ln * p.nseg + seg) * (size_t)kNelem;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) S[r][kb][i] = src[(kb * 16 + 4 * g + i) * 64 + w * 16 + l16];
      const float u = src[kD * 64 + w * 16 + l16];
      us[r] = floatx4{u, u, u, u};
    }
  }
  auto publish = [&]() {
#pragma unroll
    for (int r = 0; r < NV; ++r) {
      E* st = st_base + r * L.tile;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
        IO::st4(st + (w * 16 + l16) * P + kb * 16 + 4 * g, S[r][kb][0], S[r][kb][1], S[r][kb][2], S[r][kb][3]);
      if (mass && g == 0) s_u[r * 64 + w * 16 + l16] = us[r][0];
    }
  };

  // ---- tile loading (registers one tile ahead, then LDS)
  VTile ldk[NK], ldv;
  float ke_r = 0.0f;  // wave r < NV: this lane's key ext of view r (KV)
  auto fetch = [&](int t0) {
    if constexpr (KV) {
#pragma unroll
      for (int r = 0; r < NV; ++r)
        ldk[r].fetch(p, make_rsrc(bh_base(vp.dout[r], b, h, 2), vp.o_rec[r]), t0, (int)vp.dout[r].st * 2, vp.dv, tid);
      if (mass) {
#pragma unroll
        for (int r = 0; r < NV; ++r)
          if (w == r)
            ke_r = bldf(make_rsrc(bh_base(vp.dm[r], b, h, 4), vp.dm_rec[r]), row_off(p, t0, lane, (int)vp.dm[r].st * 4));
      }
    } else {
      ldk[0].fetch(p, v_rs, t0, v_st_b, vp.dv, tid);
    }
    ldv.fetch(p, val_rs, t0, val_st_b, vcols, tid);
  };

  // ---- queries of this wave's block: dO_r (dq) or v and the features k (dk, dv)
  F8 qr[NQ][2], qk[2];
  float qe[NQ];
  auto qfrag = [&](rsrc_t rs, uint32_t ro, int width, F8* dst) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int c0 = 32 * j + 4 * g, c1 = c0 + 16;
      const bf16x4 lo = __builtin_bit_cast(bf16x4, bld8(rs, c0 < width ? ro + (uint32_t)(c0 * 2) : kOOB));
      const bf16x4 hi = __builtin_bit_cast(bf16x4, bld8(rs, c1 < width ? ro + (uint32_t)(c1 * 2) : kOOB));
      dst[j] = IO::cat(lo, hi);
    }
  };
  auto qload = [&](int t0) {
    const int row = w * 16 + l16;
    if constexpr (KV) {
      qfrag(v_rs, row_off(p, t0, row, v_st_b), vp.dv, qr[0]);
      qe[0] = t0 + row < p.T ? 1.0f : 0.0f;
      if (vp.has_b)
        qfrag(make_rsrc((const char*)bh_base(vp.kf, b, h, 2) + col0 * 2, vp.kf_rec - (uint32_t)(col0 * 2)),
              row_off(p, t0, row, (int)vp.kf.st * 2), vcols, qk);
    } else {
#pragma unroll
      for (int r = 0; r < NV; ++r) {
        qfrag(make_rsrc(bh_base(vp.dout[r], b, h, 2), vp.o_rec[r]), row_off(p, t0, row, (int)vp.dout[r].st * 2), vp.dv,
              qr[r]);
        qe[r] = mass ? bldf(make_rsrc(bh_base(vp.dm[r], b, h, 4), vp.dm_rec[r]),
                            row_off(p, t0, row, (int)vp.dm[r].st * 4)) : 0.0f;
      }
    }
  };
  F8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (E)1.0f;

  fetch(c_begin * C);
  if (MAIN) qload(c_begin * C);

  for (int c = c_begin; c < c_end; ++c) {
    const int t0 = c * C;
    const int len = min(C, p.T - t0);
    __syncthreads();  // the previous tile's K, V, state copies and ext rows are no longer read
#pragma unroll
    for (int r = 0; r < NK; ++r) ldk[r].store(Ks + r * L.tile, P, tid);
    ldv.store(Vs, P, tid);
    if (KV && mass && w < NV) s_ke[w * 64 + lane] = ke_r;
    if (c + 1 < c_end) fetch(t0 + C);
    if (MAIN && !state_zero) publish();
    __syncthreads();

    if constexpr (MAIN) {
      const int query = w * 16 + l16;
      // ---- weighted causal scores of this query block, summed over the views
      floatx4 ps[4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        ps[kb] = floatx4{0.f, 0.f, 0.f, 0.f};
        if (kb > w) continue;
        const int krow = kb * 16 + l16;
#pragma unroll
        for (int r = 0; r < NV; ++r) {
          const E* K = Ks + (KV ? r * L.tile : 0);
          floatx4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int j = 0; j < 2; ++j) sc = mma32(frow8<E>(K, P, krow, j, g), qr[KV ? 0 : r][j], sc);
          // key kb*16+4g+i sits query - key before the query: weight element 3 - i
          const floatx4 wv = vbwd_window(s_pwx + r * 4 * kTabPitch, query - kb * 16 - 4 * g - 3);
          if (mass) {
            if constexpr (KV) {
              const floatx4 kev = *(const floatx4*)(s_ke + r * 64 + kb * 16 + 4 * g);
#pragma unroll
              for (int i = 0; i < 4; ++i) sc[i] += qe[0] * kev[i];
            } else {
#pragma unroll
              for (int i = 0; i < 4; ++i) sc[i] += qe[r];
            }
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) ps[kb][i] += sc[i] * wv[3 - i];
        }
        // keys past the query are left out, not only weighted by zero: a score
        // that is not finite stays with the queries that see its key
        if (kb == w) {
#pragma unroll
          for (int i = 0; i < 4; ++i) ps[kb][i] = 4 * g + i <= l16 ? ps[kb][i] : 0.0f;
        }
      }
      // the summed score enters the contraction as hi + lo (one view's score
      // is rounded once; a sum of them would lose more to the same rounding)
      F8 p0 = IO::from_acc(ps[0], ps[1]), p1 = IO::from_acc(ps[2], ps[3]), p0l, p1l;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        p0l[e] = bf16_rest(ps[e >> 2][e & 3], p0[e]);
        p1l[e] = bf16_rest(ps[2 + (e >> 2)][e & 3], p1[e]);
      }
      const uint32_t ro = row_off(p, t0, query, (int)vp.out.st * 2);
      const rsrc_t out_rs =
          make_rsrc((const char*)bh_base(vp.out, b, h, 2) + col0 * 2, vp.out_rec - (uint32_t)(col0 * 2));
#pragma unroll
      for (int vb = 0; vb < 4; ++vb) {
        floatx4 acc = {0.f, 0.f, 0.f, 0.f};
        if (!state_zero) {
#pragma unroll
          for (int r = 0; r < NV; ++r) {
            const E* st = st_base + r * L.tile;
            floatx4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 2; ++j) t = mma32(frow8<E>(st, P, vb * 16 + l16, j, g), qr[KV ? 0 : r][j], t);
            const float cw = s_pw[r * 68 + query + 1];
            if (mass) {
              const floatx4 u4 = *(const floatx4*)(s_u + r * 64 + vb * 16 + 4 * g);
#pragma unroll
              for (int i = 0; i < 4; ++i) t[i] += qe[KV ? 0 : r] * u4[i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] += cw * t[i];
          }
        }
        const F8 v0 = TK::col8(Vs, P, vb * 16, 0, lane);
        acc = mma32(v0, p0, acc);
        acc = mma32(v0, p0l, acc);
        if (w >= 2) {
          const F8 v1 = TK::col8(Vs, P, vb * 16, 1, lane);
          acc = mma32(v1, p1, acc);
          acc = mma32(v1, p1l, acc);
        }
        const int ocol = vb * 16 + 4 * g;
        bf16x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = (E)acc[i];
        bst8(out_rs, ocol < vcols ? ro + (uint32_t)(ocol * 2) : kOOB, __builtin_bit_cast(uint2, o));
      }

      if constexpr (KV) {
        if (vp.has_b) {
          // ---- dv: scores q . k of this slice, every view's weights, values dO_r
          floatx4 sb[4], ob[4];
#pragma unroll
          for (int kb = 0; kb < 4; ++kb) {
            sb[kb] = floatx4{0.f, 0.f, 0.f, 0.f};
            ob[kb] = floatx4{0.f, 0.f, 0.f, 0.f};
            if (kb > w) continue;
#pragma unroll
            for (int j = 0; j < 2; ++j) sb[kb] = mma32(frow8<E>(Vs, P, kb * 16 + l16, j, g), qk[j], sb[kb]);
            if (kb == w) {
#pragma unroll
              for (int i = 0; i < 4; ++i) sb[kb][i] = 4 * g + i <= l16 ? sb[kb][i] : 0.0f;
            }
          }
#pragma unroll
          for (int r = 0; r < NV; ++r) {
            const E* K = Ks + r * L.tile;
            const E* st = st_base + r * L.tile;
            floatx4 pr[4];
#pragma unroll
            for (int kb = 0; kb < 4; ++kb) {
              const floatx4 wv = vbwd_window(s_pwx + r * 4 * kTabPitch, query - kb * 16 - 4 * g - 3);
#pragma unroll
              for (int i = 0; i < 4; ++i) pr[kb][i] = sb[kb][i] * wv[3 - i];
            }
            const F8 b0 = IO::from_acc(pr[0], pr[1]), b1 = IO::from_acc(pr[2], pr[3]);
            const float cw = s_pw[r * 68 + query + 1];
#pragma unroll
            for (int vb = 0; vb < 4; ++vb) {
              if (!state_zero) {
                floatx4 t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 2; ++j) t = mma32(TK::col8(st, P, vb * 16, j, lane), qk[j], t);
#pragma unroll
                for (int i = 0; i < 4; ++i) ob[vb][i] += cw * t[i];
              }
              ob[vb] = mma32(TK::col8(K, P, vb * 16, 0, lane), b0, ob[vb]);
              if (w >= 2) ob[vb] = mma32(TK::col8(K, P, vb * 16, 1, lane), b1, ob[vb]);
            }
          }
          if (vp.part) {
            const rsrc_t pr_rs = make_rsrc(vp.part + ln * (size_t)p.T * vp.dv, (uint32_t)((size_t)p.T * vp.dv * 4));
            const uint32_t po = row_off(p, t0, query, vp.dv * 4);
#pragma unroll
            for (int vb = 0; vb < 4; ++vb) {
              const int ocol = vb * 16 + 4 * g;
              bst16(pr_rs, ocol < vp.dv ? po + (uint32_t)(ocol * 4) : kOOB, __builtin_bit_cast(uint4, ob[vb]));
            }
          } else {
            const rsrc_t ob_rs = make_rsrc(bh_base(vp.outb, b, h, 2), vp.outb_rec);
            const uint32_t rb = row_off(p, t0, query, (int)vp.outb.st * 2);
#pragma unroll
            for (int vb = 0; vb < 4; ++vb) {
              const int ocol = vb * 16 + 4 * g;
              bf16x4 o;
#pragma unroll
              for (int i = 0; i < 4; ++i) o[i] = (E)ob[vb][i];
              bst8(ob_rs, ocol < vp.dv ? rb + (uint32_t)(ocol * 2) : kOOB, __builtin_bit_cast(uint2, o));
            }
          }
        }
      }
      if (c + 1 < c_end) qload(t0 + C);
    }

    // ---- state updates: S_r = alpha_r^len S_r + K_r^T diag(w_r) V (value block w)
    F8 av[2];
#pragma unroll
    for (int kp = 0; kp < 2; ++kp) av[kp] = TK::col8(Vs, P, w * 16, kp, lane);
#pragma unroll
    for (int r = 0; r < NV; ++r) {
      __builtin_amdgcn_sched_barrier(0);  // keep each view's loads with its MFMAs (register pressure)
      const E* K = Ks + (KV ? r * L.tile : 0);
      const float cdec = s_pw[r * 68 + len];
      F8 avw[2];
#pragma unroll
      for (int kp = 0; kp < 2; ++kp) {
        // keys 32kp+4g+e and 32kp+16+4g+e sit len-1-key before the tile's end
        const int c0 = len - 1 - 32 * kp - 4 * g;
        const floatx4 lo = vbwd_window(s_pwx + r * 4 * kTabPitch, c0 - 3);
        const floatx4 hi = vbwd_window(s_pwx + r * 4 * kTabPitch, c0 - 16 - 3);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          avw[kp][e] = (E)(tof(av[kp][e]) * lo[3 - e]);
          avw[kp][4 + e] = (E)(tof(av[kp][4 + e]) * hi[3 - e]);
        }
      }
      if (!(MAIN && state_zero)) {
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) S[r][kb][i] *= cdec;
#pragma unroll
        for (int i = 0; i < 4; ++i) us[r][i] *= cdec;
      }
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) S[r][kb] = mma32(TK::col8(K, P, kb * 16, kp, lane), avw[kp], S[r][kb]);
      if (mass) {
#pragma unroll
        for (int kp = 0; kp < 2; ++kp)
          us[r] = mma32(KV ? bcast8<E>(s_ke + r * 64, 32 * kp, g) : ones, avw[kp], us[r]);
      }
    }
    state_zero = false;
  }

  if constexpr (!MAIN) {
#pragma unroll
    for (int r = 0; r < NV; ++r) {
      float* dst = vp.seg + r * vp.seg_vstride + (ln * p.nseg + seg) * (size_t)kNelem;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[(kb * 16 + 4 * g + i) * 64 + w * 16 + l16] = S[r][kb][i];
      if (g == 0) dst[kD * 64 + w * 16 + l16] = us[r][0];
      if (tid == 0) {
        float lg = 0.0f;
        for (int c = c_begin; c < c_end; ++c) lg += la[r] * (float)min(C, p.T - c * C);
        vp.segdec[r * vp.dec_vstride + ln * p.nseg + seg] = lg;
      }
    }
  }
}

// Exclusive scan of every view's segment summaries (y: slice and batch*head, z: view).
__global__ void views_bwd_prefix_kernel(float* seg, const float* segdec, int nseg, int nsum, size_t seg_vstride,
                                        size_t dec_vstride) {
  const int e0 = (blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (e0 >= kNelem) return;
  const size_t ln = blockIdx.y;
  segment_prefix4(seg + blockIdx.z * seg_vstride + ln * nseg * kNelem + e0,
                  segdec + blockIdx.z * dec_vstride + ln * nseg, nseg, nsum, kNelem, make_float4(0.f, 0.f, 0.f, 0.f));
}

}  // namespace ts

namespace {

using ts::fail;

struct Plan {
  int nchunks, seg_chunks, nseg, nsum, nsl, lanes;
  size_t seg_vstride, dec_vstride, seg_bytes, part_bytes, bytes;
};

int make_plan(const ts_views_bwd_desc* d, Plan* P) {
  if (!d) return fail(TS_ERR_VALUE, "views bwd: null descriptor");
  if (d->B < 1 || d->H < 1 || d->T < 0) return fail(TS_ERR_VALUE, "views bwd: bad shape");
  if (d->n_views < 2 || d->n_views > TS_MAX_VIEWS)
    return fail(TS_ERR_NOT_IMPLEMENTED, "views bwd: %d views (2 .. %d)", d->n_views, TS_MAX_VIEWS);
  if (d->dtype != TS_BF16) return fail(TS_ERR_NOT_IMPLEMENTED, "views bwd: bf16 streams only");
  if (d->m < 8 || d->m > 512 || d->m % 8 || d->dv < 8 || d->dv > 64 || d->dv % 8)
    return fail(TS_ERR_NOT_IMPLEMENTED, "views bwd: widths m %d (8..512) and dv %d (8..64), multiples of 8", d->m, d->dv);
  if (d->seg_chunks < 0) return fail(TS_ERR_VALUE, "views bwd: seg_chunks must be >= 0");
  if ((int64_t)d->T * d->dv * 4 >= ((int64_t)1 << 31))
    return fail(TS_ERR_NOT_IMPLEMENTED, "views bwd: one (batch, head) slice spans more than 2 GiB");
  if ((int64_t)d->B * d->H * ((d->m + 63) / 64) > 65535)
    return fail(TS_ERR_NOT_IMPLEMENTED, "views bwd: too many (batch, head) slices");
  P->nchunks = (d->T + ts::C - 1) / ts::C;
  P->nsl = (d->m + 63) / 64;
  P->lanes = d->B * d->H * P->nsl;
  // segments of the time axis up to two workgroups per CU (what registers
  // and LDS keep resident)
  int sc = d->seg_chunks;
  if (sc == 0) {
    int want = 512 / P->lanes;
    if (want < 1) want = 1;
    sc = (P->nchunks + want - 1) / want;
    if (sc < 1) sc = 1;
  }
  P->seg_chunks = sc;
  P->nseg = P->nchunks > 0 ? (P->nchunks + sc - 1) / sc : 0;
  P->nsum = P->nseg > 0 ? P->nseg - 1 : 0;
  P->seg_vstride = (size_t)P->lanes * P->nseg * ts::kNelem;
  P->dec_vstride = (size_t)P->lanes * P->nseg;
  P->seg_bytes = P->nsum > 0 ? d->n_views * (P->seg_vstride + P->dec_vstride) * sizeof(float) : 0;
  P->seg_bytes = (P->seg_bytes + 255) / 256 * 256;
  P->part_bytes = P->nsl > 1 ? (size_t)P->lanes * d->T * d->dv * sizeof(float) : 0;
  P->bytes = P->seg_bytes + P->part_bytes;
  return TS_OK;
}

typedef void (*Fn)(ts::VbwdP);

template <bool KV>
Fn pick(int nv, bool main_kernel) {
  if (nv == 2) return main_kernel ? ts::views_bwd_kernel<2, KV, true> : ts::views_bwd_kernel<2, KV, false>;
  return main_kernel ? ts::views_bwd_kernel<3, KV, true> : ts::views_bwd_kernel<3, KV, false>;
}

int launch(Fn fn, dim3 grid, int lds, hipStream_t stream, const ts::VbwdP& p) {
  if (lds > 65536) {
    hipError_t e = ts::ensure_lds_limit((const void*)fn, lds);
    if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "views bwd: LDS request failed: %s", hipGetErrorString(e));
  }
  hipLaunchKernelGGL(fn, grid, dim3(256), lds, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "views bwd: launch failed: %s", hipGetErrorString(e));
  return TS_OK;
}

int rows_of(const char* name, const ts_strided& s, int T, int width, int esize, int align, uint32_t* rec) {
  if (!s.ptr) return fail(TS_ERR_VALUE, "views bwd: missing %s", name);
  const int unit = align / esize > 0 ? align / esize : 1;
  if (((uintptr_t)s.ptr & (uintptr_t)(align - 1)) || s.st % unit || s.sh % unit || s.sb % unit)
    return fail(TS_ERR_VALUE, "views bwd: rows of %s must be %d-byte aligned", name, align);
  if (s.st < 0) return fail(TS_ERR_VALUE, "views bwd: negative time stride of %s", name);
  const int64_t reach = ((int64_t)T + 2 * ts::C) * s.st * esize + (int64_t)width * esize;
  if (reach >= ((int64_t)1 << 31))
    return fail(TS_ERR_NOT_IMPLEMENTED, "views bwd: one (batch, head) slice of %s spans more than 2 GiB", name);
  *rec = (uint32_t)(((int64_t)(T > 0 ? T - 1 : 0) * s.st + width) * esize);
  return TS_OK;
}

template <bool KV>
int pass(const ts_views_bwd_desc* d, const Plan& P, ts::VbwdP& vp, hipStream_t stream) {
  int rc;
  const int bh = d->B * d->H;
  vp.s.reverse = KV ? 1 : 0;
  if (P.nsum > 0) {
    if ((rc = launch(pick<KV>(d->n_views, false), dim3(P.nsum, bh, P.nsl), ts::vbwd_layout(d->n_views, KV, false).bytes,
                     stream, vp)))
      return rc;
    hipLaunchKernelGGL(ts::views_bwd_prefix_kernel, dim3((ts::kNelem / 4 + 255) / 256, P.lanes, d->n_views), dim3(256),
                       0, stream, vp.seg, vp.segdec, P.nseg, P.nsum, P.seg_vstride, P.dec_vstride);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "views bwd: prefix launch failed: %s", hipGetErrorString(e));
  }
  return launch(pick<KV>(d->n_views, true), dim3(P.nseg, bh, P.nsl), ts::vbwd_layout(d->n_views, KV, true).bytes, stream,
                vp);
}

}  // namespace

extern "C" {

int ts_views_bwd_workspace_bytes(const ts_views_bwd_desc* d, size_t* bytes) {
  Plan P;
  int rc = make_plan(d, &P);
  if (rc) return rc;
  if (bytes) *bytes = P.bytes;
  return TS_OK;
}

int ts_views_bwd(const ts_views_bwd_desc* d, const ts_views_bwd_io* io, void* workspace, size_t ws_bytes,
                 hipStream_t stream) {
  Plan P;
  int rc = make_plan(d, &P);
  if (rc) return rc;
  if (!io) return fail(TS_ERR_VALUE, "views bwd: null io");
  if (!io->dq.ptr && !io->dk.ptr && !io->dv) return fail(TS_ERR_VALUE, "views bwd: no gradient wanted");
  if ((io->dk.ptr != nullptr) != (io->dv != nullptr))
    return fail(TS_ERR_NOT_IMPLEMENTED, "views bwd: dk and dv come from one pass (both or neither)");
  if (d->T == 0) return TS_OK;
  if (P.bytes > 0 && (!workspace || ws_bytes < P.bytes || ((uintptr_t)workspace & 15u)))
    return fail(TS_ERR_VALUE, "views bwd: workspace missing, misaligned or too small (%zu < %zu bytes)", ws_bytes, P.bytes);
  if (io->dv && ((uintptr_t)io->dv & 15u)) return fail(TS_ERR_VALUE, "views bwd: dv is not 16-byte aligned");

  ts::VbwdP vp;
  memset(&vp, 0, sizeof(vp));
  ts::ScanP& p = vp.s;
  p.B = d->B; p.H = d->H; p.T = d->T;
  p.nchunks = P.nchunks; p.seg_chunks = P.seg_chunks; p.nseg = P.nseg; p.nsum = P.nsum;
  vp.m = d->m; vp.dv = d->dv; vp.nsl = P.nsl; vp.mass = d->mass ? 1 : 0;
  for (int r = 0; r < d->n_views; ++r) {
    vp.log_alpha[r] = io->log_alpha[r];
    vp.dout[r] = io->dout[r];
    if ((rc = rows_of("dout", vp.dout[r], d->T, d->dv, 2, 16, &vp.o_rec[r]))) return rc;
    if (d->mass) {
      vp.dm[r] = io->dmass[r];
      if ((rc = rows_of("dmass", vp.dm[r], d->T, 1, 4, 4, &vp.dm_rec[r]))) return rc;
    }
  }
  vp.v = io->v;
  if ((rc = rows_of("v", vp.v, d->T, d->dv, 2, 16, &vp.v_rec))) return rc;
  ts_strided q = io->q, k = io->k;
  uint32_t q_rec = 0, k_rec = 0;
  if ((rc = rows_of("k", k, d->T, d->m, 2, 16, &k_rec))) return rc;
  if (io->dk.ptr && (rc = rows_of("q", q, d->T, d->m, 2, 16, &q_rec))) return rc;
  vp.seg_vstride = P.seg_vstride;
  vp.dec_vstride = P.dec_vstride;
  if (P.nsum > 0) {
    vp.seg = (float*)workspace;
    vp.segdec = vp.seg + (size_t)d->n_views * P.seg_vstride;
  }
  if (io->dq.ptr) {
    vp.val = k; vp.val_rec = k_rec;
    vp.out = io->dq;
    if ((rc = rows_of("dq", vp.out, d->T, d->m, 2, 8, &vp.out_rec))) return rc;
    if ((rc = pass<false>(d, P, vp, stream))) return rc;
  }
  if (io->dk.ptr) {
    vp.val = q; vp.val_rec = q_rec;
    vp.kf = k; vp.kf_rec = k_rec;
    vp.out = io->dk;
    if ((rc = rows_of("dk", vp.out, d->T, d->m, 2, 8, &vp.out_rec))) return rc;
    vp.has_b = 1;
    const size_t n = (size_t)d->B * d->H * d->T * d->dv;
    if (P.nsl > 1) {
      vp.part = (float*)((char*)workspace + P.seg_bytes);
    } else {
      vp.outb.ptr = io->dv;
      vp.outb.sb = (int64_t)d->H * d->T * d->dv; vp.outb.sh = (int64_t)d->T * d->dv; vp.outb.st = d->dv;
      vp.outb_rec = (uint32_t)((size_t)d->T * d->dv * 2);
    }
    if ((rc = pass<true>(d, P, vp, stream))) return rc;
    if (P.nsl > 1) {
      const ts::SlotSum job = {vp.part, P.nsl, nullptr, 0, (int64_t)n, io->dv, TS_BF16, 1.0f};
      if ((rc = ts::sum_slots_batch(&job, 1, stream))) return rc;
    }
  }
  return TS_OK;
}

}  // extern "C"
