// GN write payloads and read stages: the C entry points and their checks
// (the kernels are in ts_gn_kernels.h).

#include "ts_gn_kernels.h"

#include <string.h>

namespace {

using ts::fail;

bool gn_is_wide(const ts_gn_desc* d);

int check_gn(const ts_gn_desc* d) {
  if (!d) return fail(TS_ERR_VALUE, "gn: null descriptor");
  if (d->B < 1 || d->H < 1 || d->T < 0) return fail(TS_ERR_VALUE, "gn: bad shape");
  if (d->dtype != TS_BF16 && d->dtype != TS_F32) return fail(TS_ERR_VALUE, "gn: unknown dtype");
  if (d->d != 16 && d->d != 32 && d->d != 64 && d->d != 128)
    return fail(TS_ERR_NOT_IMPLEMENTED, "gn: head width %d (16, 32, 64 or 128)", d->d);
  if (d->m < 16 || d->m % 16 || (d->m > 128 && d->m != 192 && d->m != 256 && !gn_is_wide(d)))
    return fail(TS_ERR_NOT_IMPLEMENTED,
                "gn: hidden width %d (a multiple of 16 up to 128, 192 or 256; 384 in bf16 at head widths 32, 64)", d->m);
  if (d->H > 65535 || d->B > 65535) return fail(TS_ERR_NOT_IMPLEMENTED, "gn: grid too large");
  if (d->act != TS_GN_RELU2 && d->act != TS_GN_TANH && d->act != TS_GN_SILU)
    return fail(TS_ERR_VALUE, "gn: unknown nonlinearity %d", d->act);
  if (!(d->damping > 0.f)) return fail(TS_ERR_VALUE, "gn: damping must be > 0");
  return TS_OK;
}

// A group's rows stay below the 32-bit offsets of their buffer resource: the
// rows that there are from the first, or, backwards, all 64 from the last.
bool gn_stream_ok(const ts_strided& s, int T, int vec) {
  if (!s.ptr) return true;
  if (((uintptr_t)s.ptr & 15u) || s.sb % vec || s.sh % vec || s.st % vec) return false;
  if (T <= 1) return true;
  const int rows = s.st < 0 || T > ts::TT ? ts::TT : T;
  const int64_t most = (int64_t)(ts::kGnRowsEnd / (16u / vec) - 512u) / (rows - 1);
  return -most <= s.st && s.st <= most;
}

// (one row has no stride)
ts::Str gn_str(const ts_strided& s, int T) {
  return ts::Str{const_cast<void*>(s.ptr), s.sb, s.sh, T > 1 ? (int)s.st : 0};
}

// Hidden widths the chunked kernels take (bf16, head widths 32 and 64).
bool gn_is_wide(const ts_gn_desc* d) {
  return d->dtype == TS_BF16 && (d->d == 32 || d->d == 64) && (d->m == 192 || d->m == 384);
}

int gn_lds_bytes(const ts_gn_desc* d, bool fwd) {
  const int es = d->dtype == TS_BF16 ? 2 : 4;
  const ts::GnLayout full = ts::gn_layout(es, d->d, d->m, fwd, true);
  const bool wl = full.end * es <= ts::kGnLdsMax;
  return ts::gn_layout(es, d->d, d->m, fwd, wl).end * es;
}

int gn_read_lds_bytes(const ts_gn_desc* d, bool fwd) {
  const int es = d->dtype == TS_BF16 ? 2 : 4;
  const ts::GnLayout full = ts::gn_read_layout(es, d->d, d->m, fwd, true);
  const bool wl = full.end * es <= ts::kGnLdsMax;
  return ts::gn_read_layout(es, d->d, d->m, fwd, wl).end * es;
}

// Groups of 64 tokens per workgroup: enough workgroups to fill 256 CUs.
int gn_groups(const ts_gn_desc* d) {
  const int ngroups = (d->T + ts::TT - 1) / ts::TT;
  const int64_t slices = (int64_t)d->B * d->H;
  int per = 1;
  while (per < ngroups && slices * ((ngroups + 2 * per - 1) / (2 * per)) >= 512) per *= 2;
  return per;
}

void gn_fill(const ts_gn_desc* d, ts::GnP& p) {
  memset(&p, 0, sizeof(p));
  p.B = d->B; p.H = d->H; p.T = d->T;
  p.groups = gn_groups(d);
  p.has_tau = d->has_tau;
  p.s = d->s; p.inv_L = d->inv_depth; p.eps = d->eps; p.damp = d->damping;
  p.inv_m = 1.0f / (float)d->m;
}

int gn_launch(const ts_gn_desc* d, const ts::GnP& p, bool fwd, hipStream_t stream) {
  const bool wide = gn_is_wide(d);
  const ts::GnKernel k = (d->act == TS_GN_TANH   ? ts::gn_tanh_kernel
                          : d->act == TS_GN_SILU ? ts::gn_silu_kernel
                                                 : ts::gn_relu2_kernel)(d->dtype == TS_BF16, wide, fwd, d->d, d->m);
  if (!k) return fail(TS_ERR_NOT_IMPLEMENTED, "gn: no kernel for d=%d m=%d", d->d, d->m);
  const int lds = wide ? ts::gn_wide_layout(d->d, d->m, 1).end * 2 : gn_lds_bytes(d, fwd);
  if (lds > ts::kGnLdsMax) return fail(TS_ERR_NOT_IMPLEMENTED, "gn: tile of %d bytes exceeds LDS", lds);
  if (lds > 65536) {
    hipError_t e = ts::ensure_lds_limit((const void*)k, lds);
    if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "gn: LDS request failed: %s", hipGetErrorString(e));
  }
  const int ngroups = (d->T + ts::TT - 1) / ts::TT;
  const dim3 grid((unsigned)((ngroups + p.groups - 1) / p.groups), (unsigned)d->H, (unsigned)d->B);
  hipLaunchKernelGGL(k, grid, dim3(256), lds, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "gn: launch failed: %s", hipGetErrorString(e));
  return TS_OK;
}

int check_gn_read(const ts_gn_read_desc* r, ts_gn_desc* d) {
  if (!r) return fail(TS_ERR_VALUE, "gn read: null descriptor");
  if (r->corr < 0 || r->corr > 2) return fail(TS_ERR_VALUE, "gn read: corr must be 0, 1 or 2");
  memset(d, 0, sizeof(*d));
  d->B = r->B; d->H = r->H; d->T = r->T; d->d = r->d; d->m = r->m; d->dtype = r->dtype; d->has_tau = r->has_tau;
  d->s = r->s; d->inv_depth = 1.f; d->eps = r->eps; d->act = r->act;
  d->damping = 1.f;  // the read stage has no Jacobi diagonal
  return check_gn(d);
}

void gn_read_fill(const ts_gn_read_desc* r, const ts_gn_desc* d, ts::GnReadP& p, const ts_strided& mass) {
  memset(&p, 0, sizeof(p));
  p.B = r->B; p.H = r->H; p.T = r->T;
  p.groups = gn_groups(d);
  p.has_tau = r->has_tau; p.corr = r->corr; p.want_resid = r->want_resid;
  p.s = r->s; p.eps = r->eps; p.inv_m = 1.0f / (float)r->m;
  p.mass = (const float*)mass.ptr;
  p.msb = mass.sb; p.msh = mass.sh; p.mst = mass.st;
}

int gn_read_launch(const ts_gn_desc* d, const ts::GnReadP& p, bool fwd, hipStream_t stream) {
  const bool wide = gn_is_wide(d);
  const ts::GnReadKernel k = (d->act == TS_GN_TANH   ? ts::gn_read_tanh_kernel
                              : d->act == TS_GN_SILU ? ts::gn_read_silu_kernel
                                                     : ts::gn_read_relu2_kernel)(d->dtype == TS_BF16, wide, fwd, d->d, d->m);
  if (!k) return fail(TS_ERR_NOT_IMPLEMENTED, "gn read: no kernel for d=%d m=%d", d->d, d->m);
  const int lds = wide ? ts::gn_wide_layout(d->d, d->m, p.want_resid ? (fwd ? 1 : 2) : 0).end * 2
                       : gn_read_lds_bytes(d, fwd);
  if (lds > ts::kGnLdsMax) return fail(TS_ERR_NOT_IMPLEMENTED, "gn read: tile of %d bytes exceeds LDS", lds);
  if (lds > 65536) {
    hipError_t e = ts::ensure_lds_limit((const void*)k, lds);
    if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "gn read: LDS request failed: %s", hipGetErrorString(e));
  }
  const int ngroups = (d->T + ts::TT - 1) / ts::TT;
  const dim3 grid((unsigned)((ngroups + p.groups - 1) / p.groups), (unsigned)d->H, (unsigned)d->B);
  hipLaunchKernelGGL(k, grid, dim3(256), lds, stream, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TS_ERR_RUNTIME, "gn read: launch failed: %s", hipGetErrorString(e));
  return TS_OK;
}

}  // namespace

extern "C" {

int ts_gn_write_fwd(const ts_gn_desc* d, const ts_gn_io* io, hipStream_t stream) {
  int rc = check_gn(d);
  if (rc) return rc;
  if (!io || !io->x.ptr || !io->v.ptr || !io->w1 || !io->w2 || !io->w2t || !io->h.ptr || !io->lam.ptr || !io->g.ptr)
    return fail(TS_ERR_VALUE, "gn: missing tensors");
  if (d->has_tau && !io->tau) return fail(TS_ERR_VALUE, "gn: missing tau");
  const int vec = d->dtype == TS_BF16 ? 8 : 4;
  for (const ts_strided* s : {&io->x, &io->v, &io->h, &io->lam, &io->g})
    if (!gn_stream_ok(*s, d->T, vec)) return fail(TS_ERR_VALUE, "gn: streams need 16-byte aligned rows (64 of them under 4 GiB)");
  if (d->T == 0) return TS_OK;
  ts::GnP p;
  gn_fill(d, p);
  p.x = gn_str(io->x, d->T); p.v = gn_str(io->v, d->T);
  p.h = gn_str(io->h, d->T); p.lam = gn_str(io->lam, d->T); p.g = gn_str(io->g, d->T);
  p.w1 = io->w1; p.w2 = io->w2; p.w2t = io->w2t; p.tau = io->tau;
  return gn_launch(d, p, true, stream);
}

int ts_gn_write_bwd(const ts_gn_desc* d, const ts_gn_bwd_io* io, hipStream_t stream) {
  int rc = check_gn(d);
  if (rc) return rc;
  if (!io || !io->x.ptr || !io->v.ptr || !io->w1 || !io->w2 || !io->w1t || !io->w2t || !io->dx.ptr || !io->dv.ptr ||
      !io->tiles_m || !io->tiles_d)
    return fail(TS_ERR_VALUE, "gn bwd: missing tensors");
  if (d->has_tau && !io->tau) return fail(TS_ERR_VALUE, "gn bwd: missing tau");
  const int vec = d->dtype == TS_BF16 ? 8 : 4;
  for (const ts_strided* s : {&io->x, &io->v, &io->dh, &io->dlam, &io->dg, &io->dx_in, &io->dx, &io->dv})
    if (!gn_stream_ok(*s, d->T, vec)) return fail(TS_ERR_VALUE, "gn bwd: streams need 16-byte aligned rows (64 of them under 4 GiB)");
  if (d->T == 0) return TS_OK;
  ts::GnP p;
  gn_fill(d, p);
  p.x = gn_str(io->x, d->T); p.v = gn_str(io->v, d->T);
  p.dh = gn_str(io->dh, d->T); p.dlam = gn_str(io->dlam, d->T); p.dg = gn_str(io->dg, d->T); p.dxin = gn_str(io->dx_in, d->T);
  p.dx = gn_str(io->dx, d->T); p.dv = gn_str(io->dv, d->T);
  p.w1 = io->w1; p.w2 = io->w2; p.w1t = io->w1t; p.w2t = io->w2t; p.tau = io->tau;
  p.tm = io->tiles_m; p.td = io->tiles_d;
  return gn_launch(d, p, false, stream);
}


int ts_gn_read_fwd(const ts_gn_read_desc* r, const ts_gn_read_io* io, hipStream_t stream) {
  ts_gn_desc d;
  int rc = check_gn_read(r, &d);
  if (rc) return rc;
  if (!io || !io->q.ptr || !io->w1 || !io->h.ptr) return fail(TS_ERR_VALUE, "gn read: missing tensors");
  if (r->want_resid && (!io->w2 || !io->resid.ptr)) return fail(TS_ERR_VALUE, "gn read: missing W2 or resid");
  if (r->corr && !io->num.ptr) return fail(TS_ERR_VALUE, "gn read: missing num");
  if (r->corr == 2 && !io->mass.ptr) return fail(TS_ERR_VALUE, "gn read: missing mass");
  if (r->has_tau && !io->tau) return fail(TS_ERR_VALUE, "gn read: missing tau");
  const int vec = r->dtype == TS_BF16 ? 8 : 4;
  for (const ts_strided* s : {&io->q, &io->num, &io->h, &io->resid})
    if (!gn_stream_ok(*s, r->T, vec)) return fail(TS_ERR_VALUE, "gn read: streams need 16-byte aligned rows (64 of them under 4 GiB)");
  if (r->T == 0) return TS_OK;
  ts::GnReadP p;
  gn_read_fill(r, &d, p, io->mass);
  p.q = gn_str(io->q, r->T); p.num = gn_str(io->num, r->T); p.h = gn_str(io->h, r->T); p.resid = gn_str(io->resid, r->T);
  p.w1 = io->w1; p.w2 = io->w2; p.tau = io->tau;
  return gn_read_launch(&d, p, true, stream);
}

int ts_gn_read_bwd(const ts_gn_read_desc* r, const ts_gn_read_bwd_io* io, hipStream_t stream) {
  ts_gn_desc d;
  int rc = check_gn_read(r, &d);
  if (rc) return rc;
  if (!io || !io->q.ptr || !io->w1 || !io->w1t || !io->dq.ptr || !io->tiles_m || !io->tiles_d)
    return fail(TS_ERR_VALUE, "gn read bwd: missing tensors");
  if (r->want_resid && !io->w2t) return fail(TS_ERR_VALUE, "gn read bwd: missing W2^T");
  if (r->corr && (!io->num.ptr || !io->dnum.ptr)) return fail(TS_ERR_VALUE, "gn read bwd: missing num");
  if (r->corr == 2 && (!io->mass.ptr || !io->dmass)) return fail(TS_ERR_VALUE, "gn read bwd: missing mass");
  if (r->has_tau && !io->tau) return fail(TS_ERR_VALUE, "gn read bwd: missing tau");
  const int vec = r->dtype == TS_BF16 ? 8 : 4;
  for (const ts_strided* s : {&io->q, &io->num, &io->dh, &io->dresid, &io->dq, &io->dnum})
    if (!gn_stream_ok(*s, r->T, vec)) return fail(TS_ERR_VALUE, "gn read bwd: streams need 16-byte aligned rows (64 of them under 4 GiB)");
  if (r->T == 0) return TS_OK;
  ts::GnReadP p;
  gn_read_fill(r, &d, p, io->mass);
  p.q = gn_str(io->q, r->T); p.num = gn_str(io->num, r->T);
  p.dh = gn_str(io->dh, r->T); if (r->want_resid) p.dresid = gn_str(io->dresid, r->T); p.dq = gn_str(io->dq, r->T); p.dnum = gn_str(io->dnum, r->T);
  p.dmass = io->dmass;
  p.w1 = io->w1; p.w1t = io->w1t; p.w2t = io->w2t; p.tau = io->tau;
  p.tm = io->tiles_m; p.td = io->tiles_d;
  return gn_read_launch(&d, p, false, stream);
}

}  // extern "C"
