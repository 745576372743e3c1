// crm_glue.hip -- the GCM-side code around crm() on the device (include/crm_glue.h):
// crm_input from the physics state, the surface-flux bypass, the tendencies and radiation
// conversions after the call, and check_energy_chng.  Level sums run in the reference's level
// order and floating-point contraction is off, so every result is the reference's expression
// evaluated in the reference's order.
//
// These kernels only move memory.  Their arrays are (pcols, rows): a row is a level, or a
// radiation column of a level.  A wave takes 64 columns of a row, so its accesses are contiguous,
// and every row is a wave of its own; with one thread per column looping over the rows, 4096
// columns were 64 waves on 1024 SIMDs (k_gcm_input 640 us, k_gcm_tend 690 us at 4096 x 60 levels
// x 16 radiation columns).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/crm_glue.h"
#include "crm_engine.hpp"
#include "crm_index.hpp"

#pragma clang fp contract(off)

namespace {

// physconst (cime/src/share/util/shr_const_mod.F90:22,47,53,54)
constexpr double GRAVIT = 9.80616, CPAIR = 1.00464e3, LATVAP = 2.501e6, LATICE = 3.337e5;
// the literal 0.61 of crm_physics.F90:1092 is a default (4-byte) real
constexpr double C061 = (double)0.61f;

struct Cols {
  int pcols;
  __device__ size_t at(int i, int k) const { return (size_t)i + (size_t)pcols * k; }
};

// Rows of 64 columns: a workgroup covers 64 columns of RPB rows at a time; rows beyond the
// grid's are reached by striding.
constexpr int COLS = 64, RPB = 4;
__device__ __forceinline__ Strided my_rows(long rows) {
  return {(long)blockIdx.y * RPB + threadIdx.y, (long)gridDim.y * RPB, rows};
}
__device__ __forceinline__ int my_column() { return (int)(blockIdx.x * COLS + threadIdx.x); }

// crm_physics.F90:1005-1010, 1050-1125.  Rows 0..pver are the levels (interfaces), the others the
// radiation columns of the CRM levels.
__global__ void __launch_bounds__(COLS* RPB) k_gcm_input(int ncol, int pcols, int pver, int crm_nz, int nrad,
                                                         crm_gcm_state_view st, crm_gcm_surface_view sf,
                                                         const double* angle, crm_input_view in, crm_rad_view rad) {
  const int i = my_column();
  if (i >= ncol) return;
  const Cols L{pcols};
  auto W = [](const double* p) { return const_cast<double*>(p); };
  for (Strided row = my_rows(pver + 1 + (long)nrad * crm_nz); row.more(); row.next()) {
    if (row.at > pver) {
      // Q dp -> heating rate on the CRM levels (CRM level m sits on GCM level pver-1-m)
      const long mr = row.at - pver - 1;
      const int m = level_of(mr, nrad);
      const double dp = st.pdel[L.at(i, pver - 1 - m)];
      double* qrad = W(rad.qrad);
      const size_t o = (size_t)i + (size_t)pcols * mr;
      qrad[o] = qrad[o] / dp;
      continue;
    }
    const int k = (int)row.at;
    const size_t o = L.at(i, k);
    W(in.zint)[o] = st.zi[o];
    W(in.pint)[o] = st.pint[o];
    if (k == pver) continue;
    const double ca = cos(angle[i]), sa = sin(angle[i]);
    W(in.zmid)[o] = st.zm[o];
    W(in.tl)[o] = st.t[o];
    W(in.ql)[o] = st.qv[o];
    W(in.qccl)[o] = st.qcl[o];
    W(in.qiil)[o] = st.qci[o];
    W(in.pmid)[o] = st.pmid[o];
    W(in.pdel)[o] = st.pdel[o];
    W(in.ul)[o] = st.u[o] * ca + st.v[o] * sa;
    W(in.vl)[o] = st.v[o] * ca - st.u[o] * sa;
    if (k < pver - 1) continue;
    // the surface, with the lowest level
    W(in.ps)[i] = st.ps[i];
    W(in.phis)[i] = st.phis[i];
    W(in.ocnfrac)[i] = sf.ocnfrac[i];
    W(in.tau00)[i] = sqrt(sf.wsx[i] * sf.wsx[i] + sf.wsy[i] * sf.wsy[i]);
    W(in.bflxls)[i] = sf.shf[i] / CPAIR + C061 * st.t[o] * sf.lhf[i] / LATVAP;
    W(in.fluxu00)[i] = sf.wsx[i];
    W(in.fluxv00)[i] = sf.wsy[i];
    W(in.fluxt00)[i] = sf.shf[i] / CPAIR;
    W(in.fluxq00)[i] = sf.lhf[i] / LATVAP;
    W(in.wndls)[i] = sqrt(st.u[o] * st.u[o] + st.v[o] * st.v[o]);
  }
}

// crm_physics.F90:1690-1703 (rpdel = 1/pdel)
__global__ void __launch_bounds__(COLS* RPB) k_flux_bypass(int ncol, int pcols, int pver, const double* pdel,
                                                           const double* shf, const double* cflx, double* ps_,
                                                           double* pq) {
  const int i = my_column();
  if (i >= ncol) return;
  for (Strided k = my_rows(pver); k.more(); k.next()) {
    const size_t o = (size_t)i + (size_t)pcols * k.at;
    if (k.at < pver - 1) {
      ps_[o] = 0.;
      pq[o] = 0.;
    } else {
      const double g_dp = GRAVIT * (1. / pdel[o]);
      ps_[o] = g_dp * shf[i];
      pq[o] = g_dp * cflx[i];
    }
  }
}

// A sum over the levels of a column in level order, its terms made by all waves of a workgroup:
// TILE levels at a time, the waves leave their terms in LDS and then wave q adds quantity q's to
// its sum, lane = column.
constexpr int SUM_WAVES = 8, TILE = 16;

// crm_physics.F90:1158-1169, 1203-1209, 1310-1330.  The first blocks (of the x dimension) convert
// qrad back to Q dp, a row per wave; the last nsum take 64 columns each with their radiative flux.
__global__ void __launch_bounds__(COLS* SUM_WAVES) k_gcm_tend(int ncol, int pcols, int pver, int crm_nz, int nrad,
                                                              int nsum, const double* pdel, crm_output_view out,
                                                              crm_rad_view rad, double* qrs, double* qrl, double* pts,
                                                              double* pqv, double* pqcl, double* pqci,
                                                              double* sp_rad_flux) {
  const Cols L{pcols};
  const int lane = threadIdx.x, wave = threadIdx.y;
  const int nq = (int)gridDim.x - nsum;
  if ((int)blockIdx.x < nq) {
    // heating rate -> Q dp on the CRM levels (CRM level m sits on GCM level pver-1-m)
    double* qrad = const_cast<double*>(rad.qrad);
    for (long i = lane; i < ncol; i += COLS)
      for (Strided mr{(long)blockIdx.x * SUM_WAVES + wave, (long)nq * SUM_WAVES, (long)nrad * crm_nz}; mr.more();
           mr.next()) {
        const double dp = pdel[L.at((int)i, pver - 1 - level_of(mr.at, nrad))];
        const size_t o = (size_t)i + (size_t)pcols * mr.at;
        qrad[o] = qrad[o] * dp;
      }
    return;
  }
  __shared__ double term[TILE][COLS];
  const int i = ((int)blockIdx.x - nq) * COLS + lane;
  const bool ok = i < ncol;
  const int ntop = pver - crm_nz + 2;
  double f = 0.0;
  for (int k0 = 0; k0 < pver; k0 += TILE) {
    for (int j = wave; j < TILE; j += SUM_WAVES) {
      const int k = k0 + j;
      if (!ok || k >= pver) continue;
      const size_t o = L.at(i, k);
      const double dp = pdel[o], s_ = qrs[o] / dp, l_ = qrl[o] / dp;
      qrs[o] = s_;
      qrl[o] = l_;
      pqv[o] = out.qltend[o];
      pqcl[o] = out.qcltend[o];
      pqci[o] = out.qiltend[o];
      // radiative heating above the CRM and in its top two levels
      pts[o] = k < ntop ? s_ + l_ : out.sltend[o];
      term[j][lane] = (s_ + l_) * dp / GRAVIT;
    }
    __syncthreads();
    if (wave == 0 && ok)
      for (int j = 0; j < TILE && k0 + j < pver; j++) f = f + term[j][lane];
    __syncthreads();
  }
  if (wave == 0 && ok) {
    sp_rad_flux[i] = f;
    out.precc[i] = out.precc[i] + out.precl[i];
    out.precsc[i] = out.precsc[i] + out.precsl[i];
    out.precl[i] = 0.;
    out.precsl[i] = 0.;
  }
}

// check_energy.F90:358-561 with no rain or snow constituents (wr = ws = 0)
__global__ void __launch_bounds__(COLS* SUM_WAVES) k_check_energy(
    int ncol, int pcols, int pver, crm_gcm_state_view st, double ztodt, const double* flx_vap, const double* flx_cnd,
    const double* flx_ice, const double* flx_sen, double* te_cur, double* tw_cur, double* te_tnd_c, double* tw_tnd_c,
    double* te_rer, double* tw_rer) {
  const int lane = threadIdx.x, wave = threadIdx.y;
  const int i = (int)blockIdx.x * COLS + lane;
  const bool ok = i < ncol;
  const Cols L{pcols};
  // ke, se, wv, wl, wi: wave q adds quantity q
  __shared__ double term[5][TILE][COLS], sums[5][COLS];
  double acc = 0.;
  for (int k0 = 0; k0 < pver; k0 += TILE) {
    for (int j = wave; j < TILE; j += SUM_WAVES) {
      const int k = k0 + j;
      if (!ok || k >= pver) continue;
      const size_t o = L.at(i, k);
      const double u = st.u[o], v = st.v[o], dp = st.pdel[o];
      term[0][j][lane] = 0.5 * (u * u + v * v) * dp / GRAVIT;
      term[1][j][lane] = st.t[o] * CPAIR * dp / GRAVIT;
      term[2][j][lane] = st.qv[o] * dp / GRAVIT;
      term[3][j][lane] = st.qcl[o] * dp / GRAVIT;
      term[4][j][lane] = st.qci[o] * dp / GRAVIT;
    }
    __syncthreads();
    if (wave < 5 && ok)
      for (int j = 0; j < TILE && k0 + j < pver; j++) acc = acc + term[wave][j][lane];
    __syncthreads();
  }
  if (wave < 5) sums[wave][lane] = acc;
  __syncthreads();
  if (wave > 0 || !ok) return;
  const double wr = 0., ws = 0.;
  const double ke = sums[0][lane], se = sums[1][lane] + st.phis[i] * st.ps[i] / GRAVIT;
  const double wv = sums[2][lane], wl = sums[3][lane], wi = sums[4][lane];
  const double te = se + ke + (LATVAP + LATICE) * wv + LATICE * (wl + wr);
  const double tw = wv + wl + wi + wr + ws;
  const double te_tnd = flx_vap[i] * (LATVAP + LATICE) - (flx_cnd[i] - flx_ice[i]) * 1000. * LATICE + flx_sen[i];
  const double tw_tnd = flx_vap[i] - flx_cnd[i] * 1000.;
  te_tnd_c[i] = te_tnd_c[i] + te_tnd;
  tw_tnd_c[i] = tw_tnd_c[i] + tw_tnd;
  const double te_xpd = te_cur[i] + te_tnd * ztodt;
  const double tw_xpd = tw_cur[i] + tw_tnd * ztodt;
  te_rer[i] = (te_xpd - te) / te_cur[i];
  tw_rer[i] = tw_cur[i] > 0. ? (tw_xpd - tw) / tw_cur[i] : 0.;
  te_cur[i] = te;
  tw_cur[i] = tw;
}

int col_blocks(int ncol) { return (ncol + COLS - 1) / COLS; }
// grid of a row kernel over 64-column blocks and rows
dim3 row_grid(int ncol, long rows) {
  return dim3((unsigned)col_blocks(ncol), (unsigned)std::min<long>((rows + RPB - 1) / RPB, 65535));
}
const dim3 ROW_BLOCK(COLS, RPB), SUM_BLOCK(COLS, SUM_WAVES);

int finish(const crm_hip_ctx* ctx) {
  if (hipGetLastError() != hipSuccess) return CRM_ERR_DEVICE;
  return hipStreamSynchronize(crm_ctx_stream(ctx)) == hipSuccess ? CRM_OK : CRM_ERR_DEVICE;
}

// rrtmg/radiation.F90:1584-1636: a row is a radiation column of a level
__global__ void __launch_bounds__(COLS* RPB) k_rad_columns(int ncol, int pcols, int pver, int crm_nz, int nrad,
                                                           crm_gcm_state_view st, crm_gcm_cloud_view cl,
                                                           crm_rad_view rad, crm_rad_column_view out) {
  const int i = my_column();
  if (i >= ncol) return;
  for (Strided row = my_rows((long)nrad * pver); row.more(); row.next()) {
    const int k = level_of(row.at, nrad), r = (int)(row.at - (long)k * nrad);
    const size_t g = (size_t)i + (size_t)pcols * k;    // (pcols,pver)
    const size_t o = (size_t)i + (size_t)pcols * row.at;  // (pcols,nrad,pver)
    const int m = pver - 1 - k;  // CRM level on GCM level k
    if (m >= crm_nz) {  // above the CRM: the GCM column's values
      out.t[o] = st.t[g];
      out.qv[o] = st.qv[g];
      out.qc[o] = st.qcl[g];
      out.qi[o] = st.qci[g];
      out.cld[o] = cl.cld[g];
      out.fice[o] = cl.fice[g];
      out.cicewp[o] = cl.cicewp[g];
      out.cliqwp[o] = cl.cliqwp[g];
      continue;
    }
    const size_t a = (size_t)i + (size_t)pcols * (r + (size_t)nrad * m);  // (pcols,nrad,crm_nz)
    const double cld = rad.cld[a], qc = rad.qc[a], qi = rad.qi[a];
    out.cld[o] = cld;
    if (cld > 0) {
      const double qtot = qc + qi;
      out.fice[o] = qi / qtot;
      out.cicewp[o] = qi * st.pdel[g] / GRAVIT / fmax(0.01, cld);
      out.cliqwp[o] = qc * st.pdel[g] / GRAVIT / fmax(0.01, cld);
    } else {
      out.fice[o] = 0.0;
      out.cicewp[o] = 0.0;
      out.cliqwp[o] = 0.0;
    }
    out.qi[o] = qi;
    out.qc[o] = qc;
    out.qv[o] = fmax(1.e-9, rad.qv[a]);
    out.t[o] = rad.temperature[a];
  }
}

// radiation.F90:2393-2398
__global__ void __launch_bounds__(COLS* RPB) k_rad_qrad(int ncol, int pcols, long rows, const double* qrs,
                                                        const double* qrl, double* qrad) {
  const int i = my_column();
  if (i >= ncol) return;
  for (Strided row = my_rows(rows); row.more(); row.next()) {
    const size_t o = (size_t)i + (size_t)pcols * row.at;
    qrad[o] = qrs[o] + qrl[o];
  }
}

bool dims_ok(int ncol, int pcols, int pver) { return ncol >= 0 && pcols >= ncol && pver >= 1; }

}  // namespace

extern "C" {

int crm_hip_gcm_input(crm_hip_ctx* ctx, int ncol, int pcols, int pver, int crm_nz, int nrad,
                      const crm_gcm_state_view* state, const crm_gcm_surface_view* srf, const double* crm_angle,
                      const crm_input_view* in, const crm_rad_view* rad) {
  if (!ctx || !state || !srf || !crm_angle || !in || !rad || !dims_ok(ncol, pcols, pver) || crm_nz < 2 ||
      crm_nz > pver || nrad < 1)
    return CRM_ERR_ARG;
  if (ncol == 0) return CRM_OK;
  if (hipSetDevice(crm_ctx_device(ctx)) != hipSuccess) return CRM_ERR_DEVICE;
  k_gcm_input<<<row_grid(ncol, pver + 1 + (long)nrad * crm_nz), ROW_BLOCK, 0, crm_ctx_stream(ctx)>>>(
      ncol, pcols, pver, crm_nz, nrad, *state, *srf, crm_angle, *in, *rad);
  return finish(ctx);
}

int crm_hip_gcm_flux_bypass(crm_hip_ctx* ctx, int ncol, int pcols, int pver, const double* pdel,
                            const double* shf, const double* cflx_vap, double* ptend_s, double* ptend_qv) {
  if (!ctx || !pdel || !shf || !cflx_vap || !ptend_s || !ptend_qv || !dims_ok(ncol, pcols, pver))
    return CRM_ERR_ARG;
  if (ncol == 0) return CRM_OK;
  if (hipSetDevice(crm_ctx_device(ctx)) != hipSuccess) return CRM_ERR_DEVICE;
  k_flux_bypass<<<row_grid(ncol, pver), ROW_BLOCK, 0, crm_ctx_stream(ctx)>>>(ncol, pcols, pver, pdel, shf, cflx_vap,
                                                                             ptend_s, ptend_qv);
  return finish(ctx);
}

int crm_hip_gcm_tend(crm_hip_ctx* ctx, int ncol, int pcols, int pver, int crm_nz, int nrad, const double* pdel,
                     crm_output_view* out, const crm_rad_view* rad, double* qrs, double* qrl, double* ptend_s,
                     double* ptend_qv, double* ptend_qcl, double* ptend_qci, double* sp_rad_flux) {
  if (!ctx || !pdel || !out || !rad || !qrs || !qrl || !ptend_s || !ptend_qv || !ptend_qcl || !ptend_qci ||
      !sp_rad_flux || !dims_ok(ncol, pcols, pver) || crm_nz < 2 || crm_nz > pver || nrad < 1)
    return CRM_ERR_ARG;
  if (ncol == 0) return CRM_OK;
  if (hipSetDevice(crm_ctx_device(ctx)) != hipSuccess) return CRM_ERR_DEVICE;
  const int nsum = col_blocks(ncol), nq = (int)std::min<long>(((long)nrad * crm_nz + SUM_WAVES - 1) / SUM_WAVES, 4096);
  k_gcm_tend<<<dim3((unsigned)(nq + nsum)), SUM_BLOCK, 0, crm_ctx_stream(ctx)>>>(
      ncol, pcols, pver, crm_nz, nrad, nsum, pdel, *out, *rad, qrs, qrl, ptend_s, ptend_qv, ptend_qcl, ptend_qci,
      sp_rad_flux);
  return finish(ctx);
}

int crm_hip_check_energy_chng(crm_hip_ctx* ctx, int ncol, int pcols, int pver, const crm_gcm_state_view* state,
                              double ztodt, const double* flx_vap, const double* flx_cnd, const double* flx_ice,
                              const double* flx_sen, double* te_cur, double* tw_cur, double* te_tnd,
                              double* tw_tnd, double* te_rer, double* tw_rer) {
  if (!ctx || !state || !flx_vap || !flx_cnd || !flx_ice || !flx_sen || !te_cur || !tw_cur || !te_tnd ||
      !tw_tnd || !te_rer || !tw_rer || !dims_ok(ncol, pcols, pver))
    return CRM_ERR_ARG;
  if (ncol == 0) return CRM_OK;
  if (hipSetDevice(crm_ctx_device(ctx)) != hipSuccess) return CRM_ERR_DEVICE;
  k_check_energy<<<dim3((unsigned)col_blocks(ncol)), SUM_BLOCK, 0, crm_ctx_stream(ctx)>>>(ncol, pcols, pver, *state, ztodt, flx_vap,
                                                                    flx_cnd, flx_ice, flx_sen, te_cur, tw_cur,
                                                                    te_tnd, tw_tnd, te_rer, tw_rer);
  return finish(ctx);
}

int crm_hip_rad_columns(crm_hip_ctx* ctx, int ncol, int pcols, int pver, int crm_nz, int nrad,
                        const crm_gcm_state_view* state, const crm_gcm_cloud_view* cloud, const crm_rad_view* rad,
                        const crm_rad_column_view* cols) {
  if (!ctx || !state || !cloud || !rad || !cols || !dims_ok(ncol, pcols, pver) || crm_nz < 2 || crm_nz > pver ||
      nrad < 1)
    return CRM_ERR_ARG;
  if (ncol == 0) return CRM_OK;
  if (hipSetDevice(crm_ctx_device(ctx)) != hipSuccess) return CRM_ERR_DEVICE;
  k_rad_columns<<<row_grid(ncol, (long)nrad * pver), ROW_BLOCK, 0, crm_ctx_stream(ctx)>>>(
      ncol, pcols, pver, crm_nz, nrad, *state, *cloud, *rad, *cols);
  return finish(ctx);
}

int crm_hip_rad_qrad(crm_hip_ctx* ctx, int ncol, int pcols, int nrad, int crm_nz, const double* qrs_crm,
                     const double* qrl_crm, const crm_rad_view* rad) {
  if (!ctx || !qrs_crm || !qrl_crm || !rad || !rad->qrad || ncol < 0 || pcols < ncol || nrad < 1 || crm_nz < 1)
    return CRM_ERR_ARG;
  if (ncol == 0) return CRM_OK;
  if (hipSetDevice(crm_ctx_device(ctx)) != hipSuccess) return CRM_ERR_DEVICE;
  k_rad_qrad<<<row_grid(ncol, (long)nrad * crm_nz), ROW_BLOCK, 0, crm_ctx_stream(ctx)>>>(
      ncol, pcols, (long)nrad * crm_nz, qrs_crm, qrl_crm, const_cast<double*>(rad->qrad));
  return finish(ctx);
}

}  // extern "C"
