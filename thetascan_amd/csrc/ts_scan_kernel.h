// The one-view scan kernel (summary and main pass) and its LDS layout,
// instantiated for key widths up to 128 in ts_scan.hip and for 192, 256 and
// 384 in ts_scan_wide.hip.  The passes are described in ts_scan.hip.
#pragma once

#include "ts_common.h"
#include "ts_scan_impl.h"
#include "thetascan_hip.h"

namespace ts {

// LDS carve-up (elements of E unless noted), shared with the host.
struct ScanLayout {
  int kp, vp;        // row pitches of K / V / state tiles
  int stage;         // elements per stage: K [C][kp], V [C][vp]
  int stages;
  int st;            // state copy [dvp][kp] (MAIN), `nst` buffers
  int nst;
  int fbase;         // float offset (in floats, from the byte end of the E part)
  int bytes;
};

// K and V tiles are double-buffered in LDS where two stages fit beside the
// state copies: bf16 keys up to 128 wide.  One stage keeps the next tile in
// registers instead (two barriers per tile).
__host__ __device__ constexpr int scan_stages(int esize, int DK) { return esize == 2 && DK <= 128 ? 2 : 1; }

// Float region after the E tiles (per stage: ke[C], ve[C]; then per state
// copy u[dvp] and D[DK]; pw[68], lloc[4][C]).
__host__ __device__ inline ScanLayout scan_layout_n(int esize, int DK, int dvp, int nst) {
  const int vec = 16 / esize;
  ScanLayout L{};
  L.kp = DK + vec;
  L.vp = dvp + vec;
  L.stage = C * L.kp + C * L.vp;
  L.stages = scan_stages(esize, DK);
  L.nst = nst;
  L.st = dvp * L.kp;
  const int e_elems = L.stages * L.stage + L.nst * L.st;
  const int e_bytes = (e_elems * esize + 15) / 16 * 16;
  L.fbase = e_bytes / 4;
  const int floats = L.stages * 2 * C + L.nst * (dvp + DK) + 68 + 4 * C;
  L.bytes = e_bytes + floats * 4;
  return L;
}

// The main kernel double-buffers the published state (one barrier per tile)
// unless that leaves a CU room for only one workgroup while a single copy
// (one more barrier per tile) fits two: at 128-wide keys and 64 value
// columns the two copies take 92 KB, one copy 75 KB of the CU's 160 KB.
__host__ __device__ inline ScanLayout scan_layout(int esize, int DK, int dvp, bool main_kernel) {
  if (!main_kernel) return scan_layout_n(esize, DK, dvp, 0);
  ScanLayout L = scan_layout_n(esize, DK, dvp, scan_stages(esize, DK));
  if (L.nst == 2 && 2 * L.bytes > kLdsPerCU) {
    const ScanLayout L1 = scan_layout_n(esize, DK, dvp, 1);
    if (2 * L1.bytes <= kLdsPerCU) L = L1;
  }
  return L;
}

// MODE selects what the kernel supports, so a call carries no code for what
// it does not use.  Bits: kStatic (static [H] retention), kKeyExt (the
// key-side ext column pair q_ext, k_ext), kValExt (the value-side ext column
// v_ext, out_ext), kF32Out (fp32 outputs, stored or accumulated); kGeneral
// alone reads every retention, ext column and output mode at run time.  The
// host picks an instantiated mode that covers the call, else kGeneral.
constexpr int kPlain = 0, kStatic = 1, kKeyExt = 2, kValExt = 4, kF32Out = 8, kGeneral = 16;

template <typename E, int DK, int NVW, bool MAIN, int MODE>
__global__ __launch_bounds__(256, DK == 192 || DK == 256 ? 2 : 1) void scan_kernel(ScanP p) {
  typedef typename Frag<E>::f8 F8;
  typedef typename Frag<E>::f4 F4;
  typedef LdsIO<E> IO;
  typedef Tok<E> TK;
  constexpr int ES = (int)sizeof(E);
  constexpr int VEC = 16 / ES;
  constexpr int NK32 = DK / 32;
  constexpr bool KTAIL = (DK % 32) != 0;
  constexpr int NKB = DK / 16;
  constexpr int NKO = (NKB + 3) / 4;         // key blocks of D owned per wave
  constexpr int STAGES = scan_stages(ES, DK);
  constexpr int SLOTS_K = (C * DK / VEC + 255) / 256;
  constexpr int SLOTS_V = (C * 64 * NVW / VEC + 255) / 256;

  constexpr bool GEN = MODE == kGeneral;
  constexpr bool M_KX = (MODE & kKeyExt) != 0, M_VX = (MODE & kValExt) != 0;
  const int ret = GEN ? p.ret : ((MODE & kStatic) ? TS_RET_STATIC : TS_RET_NONE);
  const int q_ext = GEN || M_KX ? p.q_ext : TS_EXT_NONE;
  const int k_ext = GEN || M_KX ? p.k_ext : TS_EXT_NONE;
  const int v_ext = GEN || M_VX ? p.v_ext : TS_EXT_NONE;
  // key-side rank-1 term (kKeyExt: the host guarantees both columns)
  const bool kx = M_KX || (GEN && q_ext != TS_EXT_NONE && k_ext != TS_EXT_NONE);
  const bool vx = (M_VX || (GEN && v_ext != TS_EXT_NONE)) && blockIdx.z == 0;
  const int out_mode = GEN || (MODE & kF32Out) ? p.out_mode : TS_OUT_STORE;
  const bool has_oe = (GEN || M_VX) && p.oe.ptr != nullptr;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = tid >> 6;
  const int g = lane >> 4;
  const int l16 = lane & 15;
  const int seg = blockIdx.x;
  const int bh = blockIdx.y;
  const int b = bh / p.H;
  const int h = bh - b * p.H;
  // value slice of this workgroup: padded columns col0 .. col0 + vs, of which
  // dvz are real.  Slices of one (segment, b, h) share the q / k tiles through
  // L2; the value-side ext column belongs to slice 0.
  const int col0 = blockIdx.z * p.vs;
  const int vs = p.vs;
  const int dvz = min(p.vs, p.dv - col0);
  const int nvb = vs >> 4;
  const int sgn = p.reverse ? -1 : 1;
  const int wave_first = __builtin_amdgcn_readfirstlane(tid & ~63);

  // ---- LDS carve-up
  const ScanLayout L = scan_layout(ES, DK, vs, MAIN);
  extern __shared__ __align__(16) unsigned char smem[];
  E* ebase = (E*)smem;
  E* st_base = ebase + STAGES * L.stage;
  float* fb = (float*)smem + L.fbase;
  float* s_ext = fb;                              // [stage][ke C | ve C]
  float* s_u = s_ext + STAGES * 2 * C;            // [nst][vs]
  float* s_d = s_u + L.nst * vs;                  // [nst][DK]
  float* s_pw = s_d + L.nst * DK;                 // alpha^d, d = 0..64 (static)
  float* my_lloc = s_pw + 68 + w * C;             // per-wave tile log-decay (stream)

  // ---- per-(b, h) addressing
  const int64_t bh_q = (int64_t)b * p.q.sb + (int64_t)h * p.q.sh;
  const int64_t bh_k = (int64_t)b * p.k.sb + (int64_t)h * p.k.sh;
  const int64_t bh_v = (int64_t)b * p.v.sb + (int64_t)h * p.v.sh + col0;
  const int q_st_b = (int)p.q.st * ES;
  const int k_st_b = (int)p.k.st * ES;
  const int v_st_b = (int)p.v.st * ES;
  const int dec_st_b = (int)p.decay.st * 4;
  auto k_rsrc = [&]() { return make_rsrc((const E*)p.k.ptr + bh_k, p.k_rec); };
  auto v_rsrc = [&]() { return make_rsrc((const E*)p.v.ptr + bh_v, p.v_rec - (uint32_t)(col0 * ES)); };
  auto q_rsrc = [&]() { return make_rsrc((const E*)p.q.ptr + bh_q, p.q_rec); };

  // a(s), the decay applied when stepping into logical position s: a reversed
  // scan steps from physical s+1 down to s and uses the decay of the physical
  // successor (logical s = 0 has none).
  auto decay_of = [&](int t0) -> float {
    const int s = t0 + lane;
    const int src = p.reverse ? p.T - s : s;
    const uint32_t off = (s < p.T && src < p.T) ? (uint32_t)(src * dec_st_b) : kOOB;
    return bldf(make_rsrc(bh_base(p.decay, b, h, 4), p.dec_rec), off);
  };
  // ext value of token t0 + row for an ext column (ones or fp32 array)
  auto ext_of = [&](int mode, const ts_strided& e, uint32_t rec, int t0, int row) -> float {
    if (mode == TS_EXT_ONES) return t0 + row < p.T ? 1.0f : 0.0f;
    return bldf(make_rsrc(bh_base(e, b, h, 4), rec), row_off(p, t0, row, (int)e.st * 4));
  };

  // ---- state: value blocks vb = w + 4r owned by this wave
  floatx4 S[NVW][NKB];
  floatx4 us[NVW];   // u for the owned value blocks (every row the same)
  floatx4 dst_[NKO]; // D for the owned key blocks kb = w + 4r (every row the same)
#pragma unroll
  for (int r = 0; r < NVW; ++r) {
    us[r] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) S[r][kb] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int r = 0; r < NKO; ++r) dst_[r] = floatx4{0.f, 0.f, 0.f, 0.f};

  const float la = ret == TS_RET_STATIC ? p.log_alpha[h] : 0.0f;
  if (ret == TS_RET_STATIC && w == 0) {
    s_pw[lane] = expf(la * (float)lane);
    if (lane == 0) s_pw[64] = expf(la * 64.0f);
  }

  const int c_begin = seg * p.seg_chunks;
  const int c_end = min(c_begin + p.seg_chunks, p.nchunks);
  float seg_log = 0.0f;
  bool state_zero = true;

  // publish the state entering a tile (bf16 / fp32 copy, u, D) into buffer `bi`
  auto publish = [&](int bi) {
    E* st = st_base + bi * L.st;
#pragma unroll
    for (int r = 0; r < NVW; ++r) {
      const int vb = w + 4 * r;
      if (vb < nvb) {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
          IO::st4(st + (vb * 16 + l16) * L.kp + kb * 16 + 4 * g, S[r][kb][0], S[r][kb][1], S[r][kb][2], S[r][kb][3]);
        if (kx && g == 0) s_u[bi * vs + vb * 16 + l16] = us[r][0];
      }
    }
    if (vx && g == 0) {
#pragma unroll
      for (int r = 0; r < NKO; ++r) {
        const int kb = w + 4 * r;
        if (kb < NKB) s_d[bi * DK + kb * 16 + l16] = dst_[r][0];
      }
    }
  };

  if (MAIN && (seg > 0 || p.has_init)) {
    state_zero = false;
    const float* src = p.seg + ((size_t)bh * p.nseg + seg) * (size_t)p.nelem;
#pragma unroll
    for (int r = 0; r < NVW; ++r) {
      const int vb = w + 4 * r;
      if (vb < nvb) {
        float u;
        if (p.states_t) {
          // the swapped scan's state [value][key] is this scan's [key][value],
          // and its value-side ext state D (sum of its keys times its ext
          // value) is this scan's key-side ext row u
          const int c = col0 + vb * 16 + l16;
          const float* row = src + (size_t)c * DK;
#pragma unroll
          for (int kb = 0; kb < NKB; ++kb) {
            const floatx4 v4 = *(const floatx4*)(row + kb * 16 + 4 * g);
            S[r][kb] = v4;
          }
          u = src[DK * DK + DK + c];
        } else {
#pragma unroll
          for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) S[r][kb][i] = src[(kb * 16 + 4 * g + i) * p.dvp + col0 + vb * 16 + l16];
          u = src[DK * p.dvp + col0 + vb * 16 + l16];
        }
        us[r] = floatx4{u, u, u, u};
      }
    }
#pragma unroll
    for (int r = 0; r < NKO; ++r) {
      const int kb = w + 4 * r;
      if (kb < NKB) {
        const float d = src[DK * p.dvp + p.dvp + kb * 16 + l16];
        dst_[r] = floatx4{d, d, d, d};
      }
    }
  }

  // ---- tile loading
  const int nk_vec = C * (DK / VEC);
  const int nv_vec = C * (vs / VEC);
  TileLoader<E, SLOTS_K> ldk;
  TileLoader<E, SLOTS_V> ldv;
  ldk.setup(p, DK / VEC, p.dk, L.kp, k_st_b, tid);
  ldv.setup(p, vs / VEC, dvz, L.vp, v_st_b, tid);
  float ext_r = 0.0f;  // this thread's ke (wave 0) / ve (wave 1) of the fetched tile
  auto fetch = [&](int t0) {
    ldk.fetch(k_rsrc(), t0, sgn, k_st_b, wave_first, nk_vec);
    ldv.fetch(v_rsrc(), t0, sgn, v_st_b, wave_first, nv_vec);
    if (w == 0 && kx) ext_r = ext_of(k_ext, p.ke, p.ke_rec, t0, lane);
    if (w == 1 && vx) ext_r = ext_of(v_ext, p.ve, p.ve_rec, t0, lane);
  };
  auto store = [&](int stg) {
    E* base = ebase + stg * L.stage;
    ldk.store(base, wave_first, nk_vec);
    ldv.store(base + C * L.kp, wave_first, nv_vec);
    if (w < 2) s_ext[stg * 2 * C + w * C + lane] = ext_r;
  };

  // ---- queries of this wave's block (registers)
  F8 qr[NK32 > 0 ? NK32 : 1];
  F4 qt;
  float qe = 0.0f;
  auto qload = [&](int t0) {
    const int row = w * 16 + l16;
    const uint32_t ro = row_off(p, t0, row, q_st_b);
    auto part = [&](int c) -> F4 {
      const uint32_t off = c < p.dk ? ro + (uint32_t)(c * ES) : kOOB;
      if constexpr (ES == 2) {
        return __builtin_bit_cast(F4, bld8(q_rsrc(), off));
      } else {
        return __builtin_bit_cast(F4, bld16(q_rsrc(), off));
      }
    };
#pragma unroll
    for (int j = 0; j < NK32; ++j) qr[j] = IO::cat(part(32 * j + 4 * g), part(32 * j + 16 + 4 * g));
    if (KTAIL) qt = part(32 * NK32 + 4 * g);
    if (kx) qe = ext_of(q_ext, p.qe, p.qe_rec, t0, row);
  };

  // ---- output addressing
  const int osz = out_mode == TS_OUT_STORE ? ES : 4;
  const void* out_base = (const char*)bh_base(p.out, b, h, osz) + col0 * osz;
  const uint32_t out_rec = p.out_rec - (uint32_t)(col0 * osz);
  const int out_st_b = (int)p.out.st * osz;
  const int oe_st_b = (int)p.oe.st * 4;

  // ---- prologue
  float dcur = 0.0f, dnext = 0.0f;
  fetch(c_begin * C);
  if (ret == TS_RET_STREAM) dnext = decay_of(c_begin * C);
  if constexpr (STAGES == 2) {
    store(c_begin & 1);
    if (c_begin + 1 < c_end) fetch((c_begin + 1) * C);
  }
  if (MAIN) {
    qload(c_begin * C);
    if (!state_zero) publish(c_begin & (L.nst - 1));
  }
  if constexpr (STAGES == 2) __syncthreads();

  for (int c = c_begin; c < c_end; ++c) {
    const int t0 = c * C;
    const int len = min(C, p.T - t0);
    const E* Ks;
    const float* ext_s;
    if constexpr (STAGES == 2) {
      if (c + 1 < c_end) store((c + 1) & 1);
      if (c + 2 < c_end) fetch(t0 + 2 * C);
      Ks = ebase + (c & 1) * L.stage;
      ext_s = s_ext + (c & 1) * 2 * C;
    } else {
      // the previous tile is no longer read (the main pass has waited for that
      // before it published this tile's state)
      if (!MAIN && c > c_begin) __syncthreads();
      store(0);
      if (c + 1 < c_end) fetch(t0 + C);  // in flight during this tile
      __syncthreads();
      Ks = ebase;
      ext_s = s_ext;
    }
    if (ret == TS_RET_STREAM) {
      dcur = dnext;
      if (c + 1 < c_end) dnext = decay_of(t0 + C);
    }
    const E* Vs = Ks + C * L.kp;
    const float* ke_s = ext_s;
    const float* ve_s = ext_s + C;

    // ---- retention of this tile (per wave)
    float tile_log = 0.0f;
    if (ret == TS_RET_STATIC) {
      tile_log = la * (float)len;
    } else if (ret == TS_RET_STREAM) {
      float x = dcur;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        float y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
      }
      my_lloc[lane] = x;
      tile_log = __shfl(x, len - 1, 64);
    }
    seg_log += tile_log;

    if constexpr (MAIN) {
      const int query = w * 16 + l16;
      const float lq = ret == TS_RET_STREAM ? my_lloc[query] : 0.0f;
      const float cw = ret == TS_RET_STATIC ? s_pw[query + 1] : (ret == TS_RET_STREAM ? expf(lq) : 1.0f);
      // ---- causal scores of this query block: sc[kb] = D[key][query], kb <= w
      floatx4 sc[4];
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        sc[kb] = floatx4{0.f, 0.f, 0.f, 0.f};
        if (kb > w) continue;
        const int krow = kb * 16 + l16;
#pragma unroll
        for (int j = 0; j < NK32; ++j) sc[kb] = mma32(frow8<E>(Ks, L.kp, krow, j, g), qr[j], sc[kb]);
        if (KTAIL) sc[kb] = mma16(frow4<E>(Ks, L.kp, krow, NK32, g), qt, sc[kb]);
        floatx4 lk;
        if (ret == TS_RET_STREAM) lk = *(const floatx4*)(my_lloc + kb * 16 + 4 * g);
        floatx4 kev;
        if (kx) kev = *(const floatx4*)(ke_s + kb * 16 + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = kb * 16 + 4 * g + i;
          float s = sc[kb][i];
          if (kx) s += qe * kev[i];
          float wt = 1.0f;
          if (ret == TS_RET_STATIC) wt = s_pw[max(query - key, 0)];
          else if (ret == TS_RET_STREAM) wt = expf(fminf(lq - lk[i], 0.0f));
          sc[kb][i] = (kb < w || key <= query) ? s * wt : 0.0f;
        }
      }
      const F8 p0 = IO::from_acc(sc[0], sc[1]);
      const F8 p1 = IO::from_acc(sc[2], sc[3]);
      // a wide key's score sums more products than one 128-wide block's and is
      // rounded once: its bf16 remainder goes through the same contraction,
      // so the score loses nothing against the sum of rounded block scores
      constexpr bool LO = ES == 2 && DK > 128;
      F8 p0lo, p1lo;
      if constexpr (LO) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          p0lo[e] = bf16_rest(sc[e >> 2][e & 3], p0[e]);
          p1lo[e] = bf16_rest(sc[2 + (e >> 2)][e & 3], p1[e]);
        }
      }
      const E* st = st_base + (c & (L.nst - 1)) * L.st;
      const float* u_in = s_u + (c & (L.nst - 1)) * vs;
      const float* d_in = s_d + (c & (L.nst - 1)) * DK;

      // ---- outputs O^T[v][query] = cw (S^T Q^T)[v] + (V^T P^T)[v], every value block
      const uint32_t ro = row_off(p, t0, query, out_st_b);
      const rsrc_t out_rs = make_rsrc(out_base, out_rec);
#pragma unroll
      for (int vb = 0; vb < 4 * NVW; ++vb) {
        if (vb >= nvb) break;
        floatx4 acc = {0.f, 0.f, 0.f, 0.f};
        if (!state_zero) {
          const int vrow = vb * 16 + l16;
#pragma unroll
          for (int j = 0; j < NK32; ++j) acc = mma32(frow8<E>(st, L.kp, vrow, j, g), qr[j], acc);
          if (KTAIL) acc = mma16(frow4<E>(st, L.kp, vrow, NK32, g), qt, acc);
          if (kx) {
            const floatx4 u4 = *(const floatx4*)(u_in + vb * 16 + 4 * g);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] += qe * u4[i];
          }
          if (ret != TS_RET_NONE) {
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] *= cw;
          }
        }
        const F8 v0 = TK::col8(Vs, L.vp, vb * 16, 0, lane);
        acc = mma32(v0, p0, acc);
        if constexpr (LO) acc = mma32(v0, p0lo, acc);
        if (w >= 2) {
          const F8 v1 = TK::col8(Vs, L.vp, vb * 16, 1, lane);
          acc = mma32(v1, p1, acc);
          if constexpr (LO) acc = mma32(v1, p1lo, acc);
        }

        const int ocol = vb * 16 + 4 * g;
        const uint32_t ooff = ocol < dvz ? ro + (uint32_t)(ocol * osz) : kOOB;
        if (out_mode == TS_OUT_STORE) {
          if constexpr (ES == 2) {
            bf16x4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = (bf16)acc[i];
            bst8(out_rs, ooff, __builtin_bit_cast(uint2, o));
          } else {
            bst16(out_rs, ooff, __builtin_bit_cast(uint4, acc));
          }
        } else {
          floatx4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = p.out_scale * acc[i];
          if (out_mode == TS_OUT_ACCUM_F32) {
            const floatx4 prev = __builtin_bit_cast(floatx4, bld16(out_rs, ooff));
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] += prev[i];
          }
          bst16(out_rs, ooff, __builtin_bit_cast(uint4, o));
        }
      }

      // ---- value-side ext column: out_ext = cw <q, D> + sum_keys P ve
      if (vx) {
        floatx4 oacc = {0.f, 0.f, 0.f, 0.f};
        if (!state_zero) {
#pragma unroll
          for (int j = 0; j < NK32; ++j) oacc = mma32(bcast8<E>(d_in, 32 * j, g), qr[j], oacc);
          if (KTAIL) oacc = mma16(bcast4<E>(d_in, 32 * NK32, g), qt, oacc);
#pragma unroll
          for (int i = 0; i < 4; ++i) oacc[i] *= cw;
        }
        oacc = mma32(bcast8<E>(ve_s, 0, g), p0, oacc);
        if (w >= 2) oacc = mma32(bcast8<E>(ve_s, 32, g), p1, oacc);
        if constexpr (LO) {
          oacc = mma32(bcast8<E>(ve_s, 0, g), p0lo, oacc);
          if (w >= 2) oacc = mma32(bcast8<E>(ve_s, 32, g), p1lo, oacc);
        }
        if (has_oe && g == 0) {
          float val = oacc[0];
          if (out_mode != TS_OUT_STORE) val *= p.out_scale;
          const uint32_t eo = row_off(p, t0, query, oe_st_b);
          const rsrc_t oe_rs = make_rsrc(bh_base(p.oe, b, h, 4), p.oe_rec);
          if (out_mode == TS_OUT_ACCUM_F32) val += bldf(oe_rs, eo);
          bstf(oe_rs, eo, val);
        }
      }
      if (c + 1 < c_end) qload(t0 + C);  // next tile's queries of this block
    }

    // ---- state update: S = decay(tile) * S + K^T diag(wk) V (owned value blocks)
    const float cdec = ret == TS_RET_STATIC ? s_pw[len] : (ret == TS_RET_STREAM ? expf(tile_log) : 1.0f);
    floatx4 wk4[2][2];  // per-key weights of this lane's keys {32kp+4g+i, 32kp+16+4g+i}
#pragma unroll
    for (int kp = 0; kp < 2; ++kp)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = 32 * kp + 16 * hf + 4 * g + i;
          float wk = 1.0f;
          if (ret == TS_RET_STATIC) wk = key < len ? s_pw[len - 1 - key] : 0.0f;
          else if (ret == TS_RET_STREAM) wk = key < len ? expf(tile_log - my_lloc[key]) : 0.0f;
          wk4[kp][hf][i] = wk;
        }
#pragma unroll
    for (int r = 0; r < NVW; ++r) {
      const int vb = w + 4 * r;
      if (vb >= nvb) break;
      F8 avw[2];
#pragma unroll
      for (int kp = 0; kp < 2; ++kp) {
        avw[kp] = TK::col8(Vs, L.vp, vb * 16, kp, lane);
        if (ret != TS_RET_NONE) {
#pragma unroll
          for (int e = 0; e < 8; ++e) avw[kp][e] = cvt<E>(tof(avw[kp][e]) * wk4[kp][e >> 2][e & 3]);
        }
      }
      if (ret != TS_RET_NONE && !(MAIN && state_zero)) {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) S[r][kb][i] *= cdec;
#pragma unroll
        for (int i = 0; i < 4; ++i) us[r][i] *= cdec;
      }
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) S[r][kb] = mma32(TK::col8(Ks, L.kp, kb * 16, kp, lane), avw[kp], S[r][kb]);
      if (kx) {
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) us[r] = mma32(bcast8<E>(ke_s, 32 * kp, g), avw[kp], us[r]);
      }
    }
    if (vx) {
      // D = decay * D + K^T (wk ve): a broadcast (wk ve) row against K columns
#pragma unroll
      for (int r = 0; r < NKO; ++r) {
        const int kb = w + 4 * r;
        if (kb >= NKB) break;
        if (ret != TS_RET_NONE) {
#pragma unroll
          for (int i = 0; i < 4; ++i) dst_[r][i] *= cdec;
        }
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
          F8 a;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int key = 32 * kp + (e < 4 ? 4 * g + e : 12 + 4 * g + e);
            a[e] = cvt<E>(ve_s[key] * wk4[kp][e >> 2][e & 3]);
          }
          dst_[r] = mma32(a, TK::col8(Ks, L.kp, kb * 16, kp, lane), dst_[r]);
        }
      }
    }
    state_zero = false;
    if constexpr (MAIN) {
      if (c + 1 < c_end) {
        if (STAGES == 1 || L.nst == 1) __syncthreads();  // single state copy: readers of this tile are done
        publish((c + 1) & (L.nst - 1));
      }
    }
    if constexpr (STAGES == 2) __syncthreads();
  }

  if constexpr (!MAIN) {
    float* dst = p.seg + ((size_t)bh * p.nseg + seg) * (size_t)p.nelem;
#pragma unroll
    for (int r = 0; r < NVW; ++r) {
      const int vb = w + 4 * r;
      if (vb < nvb) {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) dst[(kb * 16 + 4 * g + i) * p.dvp + col0 + vb * 16 + l16] = S[r][kb][i];
        if (g == 0) dst[DK * p.dvp + col0 + vb * 16 + l16] = us[r][0];
      }
    }
    if (g == 0 && blockIdx.z == 0) {
#pragma unroll
      for (int r = 0; r < NKO; ++r) {
        const int kb = w + 4 * r;
        if (kb < NKB) dst[DK * p.dvp + p.dvp + kb * 16 + l16] = dst_[r][0];
      }
    }
    if (tid == 0 && blockIdx.z == 0) p.segdec[(size_t)bh * p.nseg + seg] = seg_log;
  }
}

// The bf16 scan kernel of 192, 256 or 384 wide keys (ts_scan_wide.hip).
typedef void (*ScanFn)(ScanP);
ScanFn pick_wide_scan(int dkp, bool main_kernel, int mode);

}  // namespace ts
