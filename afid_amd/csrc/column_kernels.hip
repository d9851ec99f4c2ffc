// column_kernels.hip -- explicit terms, implicit Crank-Nicolson solves in the
// wall-normal direction, corrections, on the chunk-interleaved column layout.
//
// Reference routines restated (AFiD 1.1):
//   ExplicitTermsVX.F90:42-104, ExplicitTermsVY.F90:40-100,
//   ExplicitTermsVZ.F90:41-104, ExplicitTermsTemp.F90:37-95,
//   ImplicitAndUpdateVX.F90:33-77, ImplicitAndUpdateVY.F90:36-74,
//   ImplicitAndUpdateVZ.F90:35-71, ImplicitAndUpdateTemp.F90:34-73,
//   SolveImpEqnUpdate_X.F90, _YZ.F90, _Temp.F90 (dgttrf/dgttrs replaced by a
//   pivot-free LU applied with a 16-lane affine scan),
//   CalcLocalDivergence.F90:27-41, CorrectVelocity.F90:28-45,
//   CorrectPressure.F90:32-52.
// The order of floating-point operations inside each stencil follows the
// reference expressions (parenthesisation kept), so per-routine results match
// the reference to rounding.
#include <algorithm>
#include <type_traits>

#include "afid_internal.h"
#include "kernels.h"

namespace afid {

struct Nb {
  int64_t C, CJM, CIM;   // the column and its neighbours at j-1 and i-1
};

__device__ __forceinline__ Nb make_nb(int j, int i, const Geom &g) {
  return {col_off(j, i, g), col_off(wrapm(j - 1, g.nym), i, g), col_off(j, wrapm(i - 1, g.nzm), g)};
}

// ---------------------------------------------------------------- RHS assembly
// ImplicitAndUpdateVX.F90:47-60 (unscaled rhs; the x-solve applies ackl_b)
__device__ __forceinline__ double rhs_vx(double q, double ru, const double *vx, const double *pr,
                                         const Nb &n, int s, int skm, int skp, const double *kc,
                                         int ldx, const StepScalars &c) {
  double dxxvx = vx[n.C + skp] * kc[KC_AP3CK * ldx + s] + vx[n.C + s] * kc[KC_AC3CK * ldx + s] +
                 vx[n.C + skm] * kc[KC_AM3CK * ldx + s];
  double udx3 = c.al * kc[KC_UDX3C * ldx + s];
  double dxp = (pr[n.C + s] - pr[n.C + skm]) * udx3;
  double r = c.use_ru ? c.ro * ru : 0.0;
  return (c.ga * q + r + c.alre * dxxvx - dxp) * c.dt;
}
// ImplicitAndUpdateVY.F90:52-68
__device__ __forceinline__ double rhs_vy(double q, double ru, const double *vy, const double *pr,
                                         const Nb &n, int s, int skmm, int skpp, const double *kc,
                                         int ldx, const StepScalars &c) {
  double dxxvy = vy[n.C + skpp] * kc[KC_AP3SK * ldx + s] + vy[n.C + s] * kc[KC_AC3SK * ldx + s] +
                 vy[n.C + skmm] * kc[KC_AM3SK * ldx + s];
  double dyp = (pr[n.C + s] - pr[n.CJM + s]) * c.udy_al;
  double r = c.use_ru ? c.ro * ru : 0.0;
  return (c.ga * q + r + c.alre * dxxvy - dyp) * c.dt;
}
// ImplicitAndUpdateVZ.F90:48-64
__device__ __forceinline__ double rhs_vz(double q, double ru, const double *vz, const double *pr,
                                         const Nb &n, int s, int skmm, int skpp, const double *kc,
                                         int ldx, const StepScalars &c) {
  double dxxvz = vz[n.C + skpp] * kc[KC_AP3SK * ldx + s] + vz[n.C + s] * kc[KC_AC3SK * ldx + s] +
                 vz[n.C + skmm] * kc[KC_AM3SK * ldx + s];
  double dzp = (pr[n.C + s] - pr[n.CIM + s]) * c.dz * c.al;
  double r = c.use_ru ? c.ro * ru : 0.0;
  return (c.ga * q + r + c.alre * dxxvz - dzp) * c.dt;
}
// ImplicitAndUpdateTemp.F90:41-54
__device__ __forceinline__ double rhs_temp(double q, double ru, const double *T, const Nb &n, int s,
                                           int skm, int skp, const double *kc, int ldx,
                                           const StepScalars &c) {
  double dxxt = T[n.C + skp] * kc[KC_AP3CK * ldx + s] + T[n.C + s] * kc[KC_AC3CK * ldx + s] +
                T[n.C + skm] * kc[KC_AM3CK * ldx + s];
  double r = c.use_ru ? c.ro * ru : 0.0;
  return (c.ga * q + r + c.alpec * dxxt) * c.dt;
}

// ---------------------------------------------------------------- lane scan solve
// (L U) x = b for one column held as 16 chunks: lane p owns points k = p*L + t
// (t < L) of an n-point system.  Forward  y_k = b_k - l_k y_{k-1}, backward x_k = y_k rinv_k - e_k x_{k+1}:
// each is an affine recurrence, evaluated per chunk from a zero carry and
// fixed up with the true carry from a Kogge-Stone scan of the chunk maps
// (A = product of -l or -e over the chunk, B = local end value).  The forward
// fix-up is folded into the backward sweep; the backward fix-up is returned
// as cin so that the caller folds it into its write-out: x = b[t] + H_t*cin.

__device__ __forceinline__ double scan_up(double A, double B, int p) {
#pragma unroll
  for (int off = 1; off < P; off <<= 1) {
    double A2 = __shfl_up(A, off, P), B2 = __shfl_up(B, off, P);
    if (p >= off) {
      B = A * B2 + B;
      A = A * A2;
    }
  }
  double cin = __shfl_up(B, 1, P);
  return p == 0 ? 0.0 : cin;
}
__device__ __forceinline__ double scan_down(double A, double B, int p) {
#pragma unroll
  for (int off = 1; off < P; off <<= 1) {
    double A2 = __shfl_down(A, off, P), B2 = __shfl_down(B, off, P);
    if (p + off < P) {
      B = A * B2 + B;
      A = A * A2;
    }
  }
  double cin = __shfl_down(B, 1, P);
  return p == P - 1 ? 0.0 : cin;
}

// ---------------------------------------------------------------- load/store helpers
// Byte-offset loads and stores against a uniform base pointer (32-bit offsets
// while a field fits in 4 GiB).
template <typename OffT>
__device__ __forceinline__ double ldf(const double *base, OffT boff) {
  return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(base) + boff);
}

// What goes past the caches (non-temporal), by how the cell's sixteen arrays
// compare with the 256 MiB cache behind the L2s:
// CM_STREAM: the stencil pass's b', pr and histories, the column solve's new
// fields and the correction's inputs, which no later access of the same pass
// reads (2-3 % of each pass's time at 384x768x768, whose arrays are far larger
// than the caches); the histories' loads as well (3 % less fetched, 1 % faster).
// CM_HIST: the histories alone, which leaves the cache to the other arrays.
// CM_KEEP: nothing; the cell lives in the cache.
// FP32 histories are always ordinary: a tile row of 16 positions is half a
// 128-byte line, whose other half the neighbouring tile writes, and the halves
// merge in the L2 only when the stores are ordinary (streamed loads: 4 % slower).
// Steps with CM_STREAM, CM_HIST and CM_KEEP: 64x128x128 (10 MiB a field) 450, 426
// and 394 us; 96x128x128 (14 MiB) 576, 536, 492; 117x135x150 (20 MiB) 826, 769,
// 832; 96x192x192 (31.5 MiB) 1080, 1078, 1080; 128x256x256 (72 MiB) 2240, 2247,
// 2270; 192x384x384 6.79, 6.87, 6.94 ms.
// Steps that fold CalcMaxCFL into the last correction follow the same rule: 64x128x128
// 494 us with that correction's inputs streamed, 469 without.
enum CacheMode { CM_STREAM = 0, CM_HIST, CM_KEEP };
static int cache_mode(const Geom &g) {
  const uint64_t field = (uint64_t)g.ncol * g.ldx * sizeof(double);
  return field < (16u << 20) ? CM_KEEP : (field < (32u << 20) ? CM_HIST : CM_STREAM);
}
template <bool NT, typename OffT>
__device__ __forceinline__ void stf(double *base, OffT boff, double v) {
  double *p = reinterpret_cast<double *>(reinterpret_cast<char *>(base) + boff);
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}
// History arrays (rux..rutemp): FP64, or FP32 in the mixed-precision mode (H32),
// where element e sits at byte 4e, half the FP64 byte offset.
template <bool H32, bool NT, typename OffT>
__device__ __forceinline__ void sth(double *base, OffT boff, double v) {
  if constexpr (H32) *reinterpret_cast<float *>(reinterpret_cast<char *>(base) + (boff >> 1)) = (float)v;
  else stf<NT>(base, boff, v);
}
template <bool H32, bool NT, typename OffT>
__device__ __forceinline__ double ldh(const double *base, OffT boff) {
  if constexpr (H32) return (double)*reinterpret_cast<const float *>(reinterpret_cast<const char *>(base) + (boff >> 1));
  const double *p = reinterpret_cast<const double *>(reinterpret_cast<const char *>(base) + boff);
  return NT ? __builtin_nontemporal_load(p) : *p;
}

// ---------------------------------------------------------------- substep update
// The explicit terms, right-hand sides and wall-normal solves of one substep
// in two passes.  Each system is solved for the new value directly:
// A q_new = b + A q_old, with A the unit-diagonal normalised matrix, which
// equals q_old + A^-1 b of SolveImpEqnUpdate_* and spares re-reading q_old.
// k_stencil_rhs: the explicit terms and right-hand sides of all four fields
// (ExplicitTerms*, ImplicitAndUpdate* RHS loops), the history update, and
// b' = ackl_b*rhs + A q_old, where A is the unit-diagonal normalised system of
// SolveImpEqnUpdate_*; identity rows store q_old (+ rhs(1) = the stale row for
// vx).  A block holds ST_GC = 16 neighbouring y columns, all at the same
// ST_SP = 16 stored positions (one 128-byte line of each column; a wave covers
// four columns), and marches through zplanes consecutive z planes: each thread
// keeps its position's values of planes i-1, i and i+1 in registers, so the z
// neighbours cost no loads.  Each thread publishes the plane values its y
// neighbours need in LDS (double-buffered by plane, one barrier per plane), so
// only the group's two edge columns read a y neighbour from memory.  A column
// holds ldx = 16 L stored positions, so its L tiles are all full.  Blocks are
// ordered position-range fastest, then y group, then z range (XCD-remapped),
// so the k+-1 lines a tile reads belong to tiles running on the same XCD at
// the same time.  A plane's loads issue in one batch before any value is
// used; the history rows outside the reference loops (k = 1 and nx for
// vx/temp, nx for vy/vz), which nothing reads, are kept at 0.  Histories that no later substep reads (keep_ru = 0: RK3
// substep 3, since the next step's substep 1 has ro = 0) are not stored.
// CORR (substeps 2 and 3 of a whole step): the fields still hold the previous
// substep's u* and pr, and dph its pressure increment.  The pass corrects every
// value as it reads it, by the operations of k_correct, so the results are the
// same bit for bit, and the corrected velocities never go to memory: seven words
// a point fewer than the two passes apart (u* and dph read, pr read and written,
// against 9 words of k_correct and 5 of the reads here).  dph needs the rows
// k-2..k+1 of the own column, carried for three planes, and k-1..k+1 of the two
// neighbour columns, through LDS as the fields.  pr is read by neighbouring blocks
// while this one would write it, hence the second array.  209 VGPRs leave two
// waves per SIMD where the plain pass has three.  The three stencil and two more
// correction passes of a step took 25.8 ms at 384x768x768 (18.5 + 7.3) and take
// 22.1, 3.45 at 192x384x384 and take 2.94; the whole step 56.4 -> 52.4 and
// 7.33 -> 6.76 ms, mixed 17.85 -> 16.65 at 256x512x512, 469 -> 449 us at
// 64x128x128, 193 -> 187 at 32x64x64, where two launches fewer are the gain.
// k_column_solve: a wave owns four columns (16 chunk lanes each) and solves the
// four systems in registers: A q_new = b', with the factor rows staged in LDS.
// The new velocities u* (before the pressure correction) go to (ux, uy, uz):
// the fields themselves, in place (each lane rewrites only positions of its
// own column, and reads vz at k = 1 before writing it), or, where the
// correction must see u* apart from the corrected fields, the b buffers over
// b' itself.  The new temperature is final and goes to its field.  The vz
// increment at k=1, q_new - q_old, becomes the new stale row and the
// temperature's rhs(1).
constexpr int ZM_MAX = 32;             // most z planes per block unless afid_tune chose another limit
constexpr int SY_WG = 256;             // threads per block of the stencil and correction passes
constexpr int ST_SP = 16;              // stored positions per column tile (one 128-byte line)
constexpr int ST_GC = SY_WG / ST_SP;   // y columns per block, four per wave
// Coefficient rows staged in LDS by k_stencil_rhs: eight per-k metric rows,
// then scale, dl, du of the x, y/z and temperature systems, then (CORR) the
// correction's.
enum StencilCoef {
  SC_UDX3C = 0, SC_UDX3M, SC_AMC, SC_ACC, SC_APC, SC_AMS, SC_ACS, SC_APS,
  SC_XSC, SC_XDL, SC_XDU, SC_YSC, SC_YDL, SC_YDU, SC_TSC, SC_TDL, SC_TDU, SC_N,
  // rows of the correction: udx3c at k-1 and k+1, amphk/acphk/apphk at k and k-1
  SC_UM = SC_N, SC_UP, SC_PAM, SC_PAC, SC_PAP, SC_QAM, SC_QAC, SC_QAP, SC_NC
};
__device__ __forceinline__ int kc_row_of(int r) {
  const int rows[8] = {KC_UDX3C, KC_UDX3M, KC_AM3CK, KC_AC3CK, KC_AP3CK, KC_AM3SK, KC_AC3SK, KC_AP3SK};
  return rows[r];
}
__device__ __forceinline__ int fac_row_of(int q) { return q == 0 ? FR_SCALE : (q == 1 ? FR_DL : FR_DU); }

// The centre-column values of one plane at a thread's position (k-1, k, k+1).
struct Plane {
  double vxm, vxc, vxp, vym, vyc, vyp, vzm, vzc, vzp, tm, tc, tp, prm, prc;
};
template <typename OffT>
__device__ __forceinline__ Plane load_plane(const double *__restrict__ vx, const double *__restrict__ vy,
                                            const double *__restrict__ vz, const double *__restrict__ T,
                                            const double *__restrict__ pr, OffT C, OffT smb, OffT sb, OffT spb) {
  Plane q;
  q.vxm = ldf(vx, C + smb); q.vxc = ldf(vx, C + sb); q.vxp = ldf(vx, C + spb);
  q.vym = ldf(vy, C + smb); q.vyc = ldf(vy, C + sb); q.vyp = ldf(vy, C + spb);
  q.vzm = ldf(vz, C + smb); q.vzc = ldf(vz, C + sb); q.vzp = ldf(vz, C + spb);
  q.tm = ldf(T, C + smb); q.tc = ldf(T, C + sb); q.tp = ldf(T, C + spb);
  q.prm = ldf(pr, C + smb); q.prc = ldf(pr, C + sb);
  return q;
}

// Plane values a wave publishes for its y neighbours (the k-1 value of vy and
// the k+1 value of vx are those at the neighbour's own position s).
enum { SV_VX = 0, SV_VY, SV_VYM, SV_VZ, SV_T, SV_VXP, SV_PR, SV_VZIP, SV_N, SV_DM = SV_N, SV_DC, SV_DP, SV_NC };
static constexpr size_t stencil_lds(bool corr) {
  return sizeof(double) * (corr ? SC_NC * ST_SP + 2 * SV_NC * SY_WG : SC_N * ST_SP + 2 * SV_N * SY_WG);
}

// CorrectVelocity.F90:28-45 and CorrectPressure.F90:32-52 at a point: u* (dd the
// difference of dph across it) and pr (dph of the point and its six neighbours).
// Which products are fused is written out, so that every pass rounds alike.
__device__ __forceinline__ double corr(double u, double dd, double f) { return __builtin_fma(-dd, f, u); }
__device__ __forceinline__ double corr_pr(double pr, double d, double dkm, double dkp, double djm, double djp,
                                          double dim, double dip, double be, double dzq, double dyq, double am,
                                          double ac, double ap) {
  const double z = dip - 2.0 * d + dim, y = djp - 2.0 * d + djm;
  const double x = __builtin_fma(dkm, am, __builtin_fma(d, ac, dkp * ap));
  return __builtin_fma(-be, __builtin_fma(z, dzq, y * dyq) + x, pr + d);
}

// One rounding of a b + c, and a b - c d with the second product rounded first.
template <typename E = double>
__device__ __forceinline__ E fma_(E a, E b, E c) {
  if constexpr (std::is_same<E, float>::value) return __builtin_fmaf(a, b, c);
  else return __builtin_fma(a, b, c);
}
template <typename E>
__device__ __forceinline__ E pdiff(E a, E b, E c, E d) { return fma_<E>(a, b, -(c * d)); }

// DEV: the substep scalars come from the device step state (a.ds) rather
// than from the argument block; two instantiations keep each one's scalar
// loads unconditional.
template <typename OffT, bool USE_RU, bool DEV, bool H32, bool CORR, int CM>
__global__ void __launch_bounds__(SY_WG)
    k_stencil_rhs(FusedArgs a, const double *__restrict__ vx, const double *__restrict__ vy,
                  const double *__restrict__ vz, const double *__restrict__ T, const double *__restrict__ pr,
                  double *__restrict__ rux, double *__restrict__ ruy, double *__restrict__ ruz,
                  double *__restrict__ rut, double *__restrict__ bx, double *__restrict__ by,
                  double *__restrict__ bz, double *__restrict__ bt, double *__restrict__ stalep,
                  const double *__restrict__ kc, const double *__restrict__ facp,
                  const double *__restrict__ dph, double *__restrict__ pro) {
  extern __shared__ double sh[];
  constexpr int NC = CORR ? SC_NC : SC_N, NV = CORR ? SV_NC : SV_N;
  double *cf = sh;                    // [NC][ST_SP] coefficient rows of the block's positions
  double *xv = sh + NC * ST_SP;       // [2][NV][SY_WG] published plane values
  const Geom g = a.g;
  const int L = g.L, ldx = g.ldx, nx = g.nx, nxm = g.nxm;
  const int nq = (ldx + ST_SP - 1) / ST_SP;
  const int ngr = (g.nym + ST_GC - 1) / ST_GC;
  const int zplanes = a.zm;
  const int nib = (g.nzm + zplanes - 1) / zplanes;
  const int64_t tile = xcd_block<64>((int64_t)nib * ngr * nq);
  if (tile < 0) return;
  const int q = (int)(tile % nq);
  const int64_t rest = tile / nq;
  const int gr = (int)(rest % ngr), ib = (int)(rest / ngr);
  if (DEV && coh_int(&a.ds->halted)) return;
  const StepScalars c = DEV ? coh_scalars(&a.ds->sc[a.ns - 1]) : a.sc;
  const bool keep_ru = a.keep_ru != 0;
  for (int idx = threadIdx.x; idx < SC_N * ST_SP; idx += SY_WG) {
    const int r = idx / ST_SP, sl = min(q * ST_SP + idx - r * ST_SP, ldx - 1);
    const int src = r < SC_XSC ? kc_row_of(r) * ldx : (((r - SC_XSC) / 3) * FR_N + fac_row_of((r - SC_XSC) % 3)) * ldx;
    cf[idx] = (r < SC_XSC ? kc : facp)[src + sl];
  }
  if constexpr (CORR) {
    for (int idx = threadIdx.x; idx < (SC_NC - SC_N) * ST_SP; idx += SY_WG) {
      const int r = SC_N + idx / ST_SP, sl = min(q * ST_SP + idx % ST_SP, ldx - 1);
      const int kk = k_of_pos(sl, L);
      const int sm = kk >= 1 ? pos_of_k(kk - 1, L) : sl, sp = kk + 1 < nx ? pos_of_k(kk + 1, L) : sl;
      const int rows[8] = {KC_UDX3C, KC_UDX3C, KC_AMPHK, KC_ACPHK, KC_APPHK, KC_AMPHK, KC_ACPHK, KC_APPHK};
      cf[SC_N * ST_SP + idx] = kc[rows[r - SC_N] * ldx + (r == SC_UP ? sp : (r == SC_UM || r >= SC_QAM ? sm : sl))];
    }
  }
  __syncthreads();
  const int lane = (int)threadIdx.x & (ST_SP - 1);        // position within the tile
  const int w = (int)threadIdx.x / ST_SP;                  // column within the group
  const int ncols = min(ST_GC, g.nym - gr * ST_GC);        // columns of this group
  const bool colok = w < ncols;
  const int jc = colok ? gr * ST_GC + w : g.nym - 1;       // idle threads read a valid column, store nothing
  const int sraw = q * ST_SP + lane;
  const int s = min(sraw, ldx - 1);
  const int k = k_of_pos(s, L);
  // Every stored position of a column is written, the padding (k >= nx) as
  // zeros: a 128-byte line written in part costs the memory system about as
  // much again as a whole one (1.6 ms of 8.6 per launch at 384x768x768).
  const bool stv = colok && sraw < ldx;
  const bool pad = k >= nx;
  const bool jp_in = w + 1 < ncols, jm_in = w > 0;        // neighbour column in this block
  const int jm = wrapm(jc - 1, g.nym), jp = wrapp(jc + 1, g.nym);
  const OffT cb = (OffT)ldx * sizeof(double);
  auto colb = [&](int jj, int ii) { return ((OffT)ii * (OffT)g.nym + (OffT)jj) * cb; };
  const OffT sb = (OffT)s * sizeof(double);
  const OffT smb = (OffT)(k >= 1 ? pos_of_k(k - 1, L) : s) * sizeof(double);
  const OffT spb = (OffT)(k + 1 < nx ? pos_of_k(k + 1, L) : s) * sizeof(double);
  const bool inx = k >= 1 && k <= nx - 2;
  const bool iny = k <= nxm - 1;
  auto cfv = [&](int r) { return cf[r * ST_SP + lane]; };
  const double udx3c = cfv(SC_UDX3C), udx3m = cfv(SC_UDX3M);
  const double amc = cfv(SC_AMC), acc = cfv(SC_ACC), apc = cfv(SC_APC);
  const double ams = cfv(SC_AMS), acs = cfv(SC_ACS), aps = cfv(SC_APS);
  const int i0 = ib * zplanes, i1 = min(i0 + zplanes, g.nzm);
  Plane cur = load_plane<OffT>(vx, vy, vz, T, pr, colb(jc, i0), smb, sb, spb);
  const int ib0 = wrapm(i0 - 1, g.nzm);
  const OffT CP = colb(jc, ib0);
  // CORR: the fields hold u* and the pressure before the correction, and each
  // value is corrected as it enters.  dph at k-2, k-1, k, k+1 (mm, m, c, p) of
  // the plane (d), of the plane before (e) and of the y neighbours (a: j-1, b: j+1).
  const OffT smmb = CORR ? (OffT)(k >= 2 && k < nx ? pos_of_k(k - 2, L) : (k >= 1 ? pos_of_k(k - 1, L) : s)) * sizeof(double) : 0;
  const bool okm = k - 1 <= nxm - 1, okp = k + 1 <= nxm - 1;
  const bool dtop = k >= nxm - 1;
  double fm = 0.0, f0 = 0.0, fp = 0.0, fy = 0.0, fz = 0.0, be = 0.0, pzq = 0.0, pyq = 0.0;
  double dmm = 0.0, dm = 0.0, dc = 0.0, dp = 0.0, em = 0.0, ec = 0.0;
  double am = 0.0, ac = 0.0, ap = 0.0, ae = 0.0, bm = 0.0, bc = 0.0, bee = 0.0;
  const int jmm = wrapm(jm - 1, g.nym);
  auto prk = [&](double v, double d, double dkm, double dkp, double djm, double djp, double dim, double dip) {
    return corr_pr(v, d, dkm, dtop ? d : dkp, djm, djp, dim, dip, be, pzq, pyq, cfv(SC_PAM), cfv(SC_PAC), cfv(SC_PAP));
  };
  if constexpr (CORR) {
    const StepScalars pc = DEV ? coh_scalars(&a.ds->sc[a.ns - 2]) : a.psc;
    const double adt = pc.al * pc.dt;
    fm = adt * cfv(SC_UM);
    f0 = adt * udx3c;
    fp = adt * cfv(SC_UP);
    fy = adt * pc.dy;
    fz = adt * pc.dz;
    be = pc.al * pc.beta;
    pzq = pc.dzq;
    pyq = pc.dyq;
    const OffT C = colb(jc, i0), A = colb(jm, i0), B = colb(jp, i0);
    dmm = ldf(dph, C + smmb); dm = ldf(dph, C + smb); dc = ldf(dph, C + sb); dp = ldf(dph, C + spb);
    am = ldf(dph, A + smb); ac = ldf(dph, A + sb); ap = ldf(dph, A + spb);
    bm = ldf(dph, B + smb); bc = ldf(dph, B + sb);
    em = ldf(dph, CP + smb); ec = ldf(dph, CP + sb);
    ae = ldf(dph, colb(jm, ib0) + sb); bee = ldf(dph, colb(jp, ib0) + sb);
  }
  double vxim = ldf(vx, CP + sb), vximp = ldf(vx, CP + spb), vyim = ldf(vy, CP + sb);
  double vzim = ldf(vz, CP + sb), tim = ldf(T, CP + sb), prim = ldf(pr, CP + sb);
  double vyjpim = ldf(vy, colb(jp, ib0) + sb);
  if constexpr (CORR) {
    const double ep = ldf(dph, CP + spb), e2 = ldf(dph, colb(jc, wrapm(ib0 - 1, g.nzm)) + sb);
    if (okm) {
      cur.vxm = corr(cur.vxm, dm - dmm, fm);
      cur.vym = corr(cur.vym, dm - am, fy);
      cur.vzm = corr(cur.vzm, dm - em, fz);
    }
    if (iny) {
      cur.vxc = corr(cur.vxc, dc - dm, f0);
      cur.vyc = corr(cur.vyc, dc - ac, fy);
      cur.vzc = corr(cur.vzc, dc - ec, fz);
      vxim = corr(vxim, ec - em, f0);
      vyim = corr(vyim, ec - ae, fy);
      vzim = corr(vzim, ec - e2, fz);
      prim = prk(prim, ec, em, ep, ae, bee, e2, dc);
      vyjpim = corr(vyjpim, bee - ec, fy);
    }
    if (okp) {
      cur.vxp = corr(cur.vxp, dp - dc, fp);
      cur.vyp = corr(cur.vyp, dp - ap, fy);
      cur.vzp = corr(cur.vzp, dp - ep, fz);
      vximp = corr(vximp, ep - ec, fp);
    }
  }
  const int tid = (int)threadIdx.x;
  int par = 0;
  for (int ic = i0; ic < i1; ic++) {
    const int ip = wrapp(ic + 1, g.nzm);
    const OffT C = colb(jc, ic), CJM = colb(jm, ic), CJP = colb(jp, ic);
    Plane nxt = load_plane<OffT>(vx, vy, vz, T, pr, colb(jc, ip), smb, sb, spb);
    double nmm = 0.0, nm = 0.0, nc = 0.0, np = 0.0, anm = 0.0, anc = 0.0, anp = 0.0, bnm = 0.0, bnc = 0.0, a2 = 0.0;
    if constexpr (CORR) {
      const OffT N = colb(jc, ip);
      nmm = ldf(dph, N + smmb); nm = ldf(dph, N + smb); nc = ldf(dph, N + sb); np = ldf(dph, N + spb);
      if (!jp_in) {
        const OffT NB = colb(jp, ip);
        bnm = ldf(dph, NB + smb); bnc = ldf(dph, NB + sb);
      }
      if (!jm_in) {
        const OffT NA = colb(jm, ip);
        anm = ldf(dph, NA + smb); anc = ldf(dph, NA + sb); anp = ldf(dph, NA + spb);
        a2 = ldf(dph, colb(jmm, ic) + sb);
      }
    }
    double vxjp = 0.0, vyjp = 0.0, vyjpm = 0.0, vzjp = 0.0, tjp = 0.0;
    double vxjm = 0.0, vxjmp = 0.0, vyjm = 0.0, vzjm = 0.0, tjm = 0.0, prjm = 0.0, vzjmip = 0.0;
    if (!jp_in) {
      vxjp = ldf(vx, CJP + sb); vyjp = ldf(vy, CJP + sb); vyjpm = ldf(vy, CJP + smb);
      vzjp = ldf(vz, CJP + sb); tjp = ldf(T, CJP + sb);
    }
    if (!jm_in) {
      vxjm = ldf(vx, CJM + sb); vxjmp = ldf(vx, CJM + spb); vyjm = ldf(vy, CJM + sb);
      vzjm = ldf(vz, CJM + sb); tjm = ldf(T, CJM + sb); prjm = ldf(pr, CJM + sb);
      vzjmip = ldf(vz, colb(jm, ip) + sb);
    }
    const double rxo = USE_RU ? ldh<H32, CM != CM_KEEP>(rux, C + sb) : 0.0, ryo = USE_RU ? ldh<H32, CM != CM_KEEP>(ruy, C + sb) : 0.0;
    const double rzo = USE_RU ? ldh<H32, CM != CM_KEEP>(ruz, C + sb) : 0.0, rto = USE_RU ? ldh<H32, CM != CM_KEEP>(rut, C + sb) : 0.0;
    const double st0 = q == 0 ? coh_dbl(stalep + (int64_t)ic * g.nym + jc) : 0.0;   // k = 0 lies in row 0
    const double stale0 = k == 0 ? st0 : 0.0;
    double *buf = xv + par * (NV * SY_WG);
    if constexpr (CORR) {
      if (okm) {
        cur.prm = corr_pr(cur.prm, dm, dmm, dc, am, bm, em, nm, be, pzq, pyq, cfv(SC_QAM), cfv(SC_QAC), cfv(SC_QAP));
        nxt.vxm = corr(nxt.vxm, nm - nmm, fm);
        nxt.vzm = corr(nxt.vzm, nm - dm, fz);
      }
      if (iny) {
        cur.prc = prk(cur.prc, dc, dm, dp, ac, bc, ec, nc);
        nxt.vxc = corr(nxt.vxc, nc - nm, f0);
        nxt.vzc = corr(nxt.vzc, nc - dc, fz);
      }
      if (okp) {
        nxt.vxp = corr(nxt.vxp, np - nc, fp);
        nxt.vzp = corr(nxt.vzp, np - dp, fz);
      }
      buf[SV_DM * SY_WG + tid] = nm;
      buf[SV_DC * SY_WG + tid] = nc;
      buf[SV_DP * SY_WG + tid] = np;
    }
    buf[SV_VX * SY_WG + tid] = cur.vxc;
    buf[SV_VY * SY_WG + tid] = cur.vyc;
    buf[SV_VYM * SY_WG + tid] = cur.vym;
    buf[SV_VZ * SY_WG + tid] = cur.vzc;
    buf[SV_T * SY_WG + tid] = cur.tc;
    buf[SV_VXP * SY_WG + tid] = cur.vxp;
    buf[SV_PR * SY_WG + tid] = cur.prc;
    buf[SV_VZIP * SY_WG + tid] = nxt.vzc;
    __syncthreads();
    if (jp_in) {
      const int o = tid + ST_SP;
      vxjp = buf[SV_VX * SY_WG + o]; vyjp = buf[SV_VY * SY_WG + o]; vyjpm = buf[SV_VYM * SY_WG + o];
      vzjp = buf[SV_VZ * SY_WG + o]; tjp = buf[SV_T * SY_WG + o];
    }
    if (jm_in) {
      const int o = tid - ST_SP;
      vxjm = buf[SV_VX * SY_WG + o]; vxjmp = buf[SV_VXP * SY_WG + o]; vyjm = buf[SV_VY * SY_WG + o];
      vzjm = buf[SV_VZ * SY_WG + o]; tjm = buf[SV_T * SY_WG + o]; prjm = buf[SV_PR * SY_WG + o];
      vzjmip = buf[SV_VZIP * SY_WG + o];
    }
    if constexpr (CORR) {
      if (jp_in) {
        const int o = tid + ST_SP;
        bnm = buf[SV_DM * SY_WG + o]; bnc = buf[SV_DC * SY_WG + o];
      } else {
        if (okm) vyjpm = corr(vyjpm, bm - dm, fy);
        if (iny) {
          vxjp = corr(vxjp, bc - bm, f0);
          vyjp = corr(vyjp, bc - dc, fy);
          vzjp = corr(vzjp, bc - bee, fz);
        }
      }
      if (jm_in) {
        const int o = tid - ST_SP;
        anm = buf[SV_DM * SY_WG + o]; anc = buf[SV_DC * SY_WG + o]; anp = buf[SV_DP * SY_WG + o];
      } else {
        if (okp) vxjmp = corr(vxjmp, ap - ac, fp);
        if (iny) {
          vxjm = corr(vxjm, ac - am, f0);
          vyjm = corr(vyjm, ac - a2, fy);
          vzjm = corr(vzjm, ac - ae, fz);
          prjm = prk(prjm, ac, am, ap, a2, dc, ae, anc);
          vzjmip = corr(vzjmip, anc - ac, fz);
        }
      }
      if (okm) nxt.vym = corr(nxt.vym, nm - anm, fy);
      if (iny) nxt.vyc = corr(nxt.vyc, nc - anc, fy);
      if (okp) nxt.vyp = corr(nxt.vyp, np - anp, fy);
    }
    par ^= 1;
    const double vxm = cur.vxm, vxc = cur.vxc, vxp = cur.vxp, vym = cur.vym, vyc = cur.vyc, vyp = cur.vyp;
    const double vzm = cur.vzm, vzc = cur.vzc, vzp = cur.vzp, tm = cur.tm, tc = cur.tc, tp = cur.tp;
    const double prm = cur.prm, prc = cur.prc;
    const double vxip = nxt.vxc, vyip = nxt.vyc, vzip = nxt.vzc, vzipm = nxt.vzm, tip = nxt.tc;
    if (CORR && stv) {
      stf<CM == CM_STREAM>(pro, C + sb, prc);
      if (k == 0) stalep[(int64_t)ic * g.nym + jc] = vzc;   // the column solve reads it there, then writes the row
    }
    if (stv) {
// Which products are fused is written out, here as in the correction: left to
// the compiler, an instance may fuse another product of a sum than its siblings,
// and a cell's result would hang on the route that its steps take.
#pragma clang fp contract(off)
      // The explicit terms in E: FP64, or FP32 in the mixed-precision mode (their
      // inputs rounded from the FP64 fields); the right-hand sides, b' and the
      // solves stay FP64.  With E = double the expressions are the FP64 ones.
      using E = typename std::conditional<H32, float, double>::type;
      const E Evxm = vxm, Evxc = vxc, Evxp = vxp, Evym = vym, Evyc = vyc, Evyp = vyp;
      const E Evzm = vzm, Evzc = vzc, Evzp = vzp, Etm = tm, Etc = tc, Etp = tp;
      const E Evxip = vxip, Evyip = vyip, Evzip = vzip, Evzipm = vzipm, Etip = tip;
      const E Evxim = vxim, Evximp = vximp, Evyim = vyim, Evzim = vzim, Etim = tim;
      const E Evxjp = vxjp, Evyjp = vyjp, Evyjpm = vyjpm, Evzjp = vzjp, Etjp = tjp, Evyjpim = vyjpim;
      const E Evxjm = vxjm, Evxjmp = vxjmp, Evyjm = vyjm, Evzjm = vzjm, Etjm = tjm, Evzjmip = vzjmip;
      const E Eudz4 = c.udz4, Eudy4 = c.udy4, Eudx3c = udx3c, Eudx3m = udx3m;
      const E Eudzq_re = c.udzq_re, Eudyq_re = c.udyq_re, Eudzq_pe = c.udzq_pe, Eudyq_pe = c.udyq_pe;
      // ---- vx (ExplicitTermsVX.F90:55-101, ImplicitAndUpdateVX.F90:47-60)
      {
        const E hxz = pdiff<E>(Evzip + Evzipm, Evxip + Evxc, Evzc + Evzm, Evxc + Evxim);   // times udz4
        const E hxy = pdiff<E>(Evyjp + Evyjpm, Evxjp + Evxc, Evyc + Evym, Evxc + Evxjm);   // times udy4
        const E aa = Evxp + Evxc, bb = Evxc + Evxm;
        const E hxx = pdiff<E>(aa, aa, bb, bb) * Eudx3c;                                   // times 0.25
        const E dzzvx = fma_<E>((E)-2.0, Evxc, Evxim) + Evxip, dyyvx = fma_<E>((E)-2.0, Evxc, Evxjm) + Evxjp;
        const E hx = fma_<E>(hxz, Eudz4, fma_<E>(hxx, (E)0.25, hxy * Eudy4));
        const double q = fma_<E>(dzzvx, Eudzq_re, fma_<E>(dyyvx, Eudyq_re, -hx)) + Etc;
        const double dxxvx = fma_(vxm, amc, fma_(vxc, acc, vxp * apc));
        const double rq = USE_RU ? fma_(c.ro, rxo, c.ga * q) : fma_(c.ga, q, 0.0);
        const double rhs = fma_(-(c.al * udx3c), prc - prm, fma_(c.alre, dxxvx, rq)) * c.dt;
        const double vin = fma_(rhs, cfv(SC_XSC), fma_(cfv(SC_XDU), vxp, fma_(cfv(SC_XDL), vxm, vxc)));
        double vbd = stale0 + vxc;
        if (keep_ru) sth<H32, CM != CM_KEEP>(rux, C + sb, pad ? 0.0 : (inx ? q : 0.0));
        stf<CM == CM_STREAM>(bx, C + sb, pad ? 0.0 : (inx ? vin : vbd));
      }
      // ---- vy (ExplicitTermsVY.F90:52-98, ImplicitAndUpdateVY.F90:52-68); kmv/kpv clamps
      {
        const double vymm = k == 0 ? vyc : vym, vypp = k == nxm - 1 ? vyc : vyp;
        const E Evymm = vymm, Evypp = vypp;
        const E hyx = pdiff<E>(Evxp + Evxjmp, Evypp + Evyc, Evxc + Evxjm, Evyc + Evymm) * Eudx3m;   // times 0.25
        const E yp = Evyjp + Evyc, ym = Evyjm + Evyc;
        const E hyy = pdiff<E>(yp, yp, ym, ym);                                                     // times udy4
        const E hyz = pdiff<E>(Evyip + Evyc, Evzip + Evzjmip, Evyc + Evyim, Evzc + Evzjm);          // times udz4
        const E dyyvy = fma_<E>((E)-2.0, Evyc, Evyjp) + Evyjm, dzzvy = fma_<E>((E)-2.0, Evyc, Evyip) + Evyim;
        const E hy = fma_<E>(hyz, Eudz4, fma_<E>(hyy, Eudy4, hyx * (E)0.25));
        const double h = fma_<E>(dzzvy, Eudzq_re, fma_<E>(dyyvy, Eudyq_re, -hy));
        const double dxxvy = fma_(vymm, ams, fma_(vyc, acs, vypp * aps));
        const double rq = USE_RU ? fma_(c.ro, ryo, c.ga * h) : fma_(c.ga, h, 0.0);
        const double rhs = fma_(-(prc - prjm), c.udy_al, fma_(c.alre, dxxvy, rq)) * c.dt;
        const double vin = fma_(rhs, cfv(SC_YSC), fma_(cfv(SC_YDU), vyp, fma_(cfv(SC_YDL), vym, vyc)));
        if (keep_ru) sth<H32, CM != CM_KEEP>(ruy, C + sb, pad ? 0.0 : (iny ? h : 0.0));
        stf<CM == CM_STREAM>(by, C + sb, pad ? 0.0 : vin);   // row nx-1 is outside the nxm system and never read
      }
      // ---- vz (ExplicitTermsVZ.F90:56-101, ImplicitAndUpdateVZ.F90:48-64)
      {
        const double vzmm = k == 0 ? vzc : vzm, vzpp = k == nxm - 1 ? vzc : vzp;
        const E Evzmm = vzmm, Evzpp = vzpp;
        const E zp = Evzip + Evzc, zm = Evzim + Evzc;
        const E hzz = pdiff<E>(zp, zp, zm, zm);                                                     // times udz4
        const E hzy = pdiff<E>(Evyjp + Evyjpim, Evzjp + Evzc, Evyc + Evyim, Evzc + Evzjm);          // times udy4
        const E hzx = pdiff<E>(Evxp + Evximp, Evzpp + Evzc, Evxc + Evxim, Evzc + Evzmm) * Eudx3m;   // times 0.25
        const E dzzvz = fma_<E>((E)-2.0, Evzc, Evzip) + Evzim, dyyvz = fma_<E>((E)-2.0, Evzc, Evzjp) + Evzjm;
        const E hz = fma_<E>(hzz, Eudz4, fma_<E>(hzx, (E)0.25, hzy * Eudy4));
        const double h = fma_<E>(dzzvz, Eudzq_re, fma_<E>(dyyvz, Eudyq_re, -hz));
        const double dxxvz = fma_(vzmm, ams, fma_(vzc, acs, vzpp * aps));
        const double rq = USE_RU ? fma_(c.ro, rzo, c.ga * h) : fma_(c.ga, h, 0.0);
        const double rhs = fma_(-((prc - prim) * c.dz), c.al, fma_(c.alre, dxxvz, rq)) * c.dt;
        const double vin = fma_(rhs, cfv(SC_YSC), fma_(cfv(SC_YDU), vzp, fma_(cfv(SC_YDL), vzm, vzc)));
        if (keep_ru) sth<H32, CM != CM_KEEP>(ruz, C + sb, pad ? 0.0 : (iny ? h : 0.0));
        stf<CM == CM_STREAM>(bz, C + sb, pad ? 0.0 : vin);
      }
      // ---- temperature (ExplicitTermsTemp.F90:52-93, ImplicitAndUpdateTemp.F90:41-54)
      {
        const E htz = pdiff<E>(Evzipm + Evzip, Etip + Etc, Evzm + Evzc, Etc + Etim);           // times udz4
        const E hty = pdiff<E>(Evyjp + Evyjpm, Etjp + Etc, Evyc + Evym, Etc + Etjm);           // times udy4
        const E htx = pdiff<E>(Evxp + Evxc, Etp + Etc, Evxc + Evxm, Etc + Etm) * Eudx3c;       // times 0.25
        const E dzzt = fma_<E>((E)-2.0, Etc, Etip) + Etim, dyyt = fma_<E>((E)-2.0, Etc, Etjp) + Etjm;
        const E ht = fma_<E>(htz, Eudz4, fma_<E>(htx, (E)0.25, hty * Eudy4));
        const double h = fma_<E>(dzzt, Eudzq_pe, fma_<E>(dyyt, Eudyq_pe, -ht));
        const double dxxt = fma_(tm, amc, fma_(tc, acc, tp * apc));
        const double rq = USE_RU ? fma_(c.ro, rto, c.ga * h) : fma_(c.ga, h, 0.0);
        const double rhs = fma_(c.alpec, dxxt, rq) * c.dt;
        const double vin = fma_(rhs, cfv(SC_TSC), fma_(cfv(SC_TDU), tp, fma_(cfv(SC_TDL), tm, tc)));
        if (keep_ru) sth<H32, CM != CM_KEEP>(rut, C + sb, pad ? 0.0 : (inx ? h : 0.0));
        stf<CM == CM_STREAM>(bt, C + sb, pad ? 0.0 : (inx ? vin : tc));   // row 1 gets the vz increment added by the solve pass
      }
    }
    vxim = vxc; vximp = vxp; vyim = vyc; vzim = vzc; tim = tc; prim = prc;
    vyjpim = vyjp;
    cur = nxt;
    em = dm; ec = dc; ae = ac; bee = bc;
    dmm = nmm; dm = nm; dc = nc; dp = np;
    am = anm; ac = anc; ap = anp; bm = bnm; bc = bnc;
  }
}

// Lane p's chunk of one column's b' into registers (zeros past cnt).  The
// loads are unconditional (slot index clamped into the column's L rows) so
// that all LM of them issue back to back; the select discards the extras.
template <int LM, typename OffT>
__device__ __forceinline__ void load_chunk(double (&b)[LM], const double *__restrict__ src, OffT C, int cnt,
                                           int L, int p) {
#pragma unroll
  for (int t = 0; t < LM; t++) {
    const double v = ldf(src, C + (OffT)(min(t, L - 1) * P + p) * sizeof(double));
    b[t] = t < cnt ? v : 0.0;
  }
}

// Solves the chunk held in b in place; returns cin, with the solution
// x = b + H cin.  `rows` holds the system's factor rows L, RINV, E, G, H
// (row r at rows + r*ldx), staged in LDS by the caller.
enum { RW_L = 0, RW_RINV, RW_E, RW_G, RW_H, RW_N };
template <int LM>
__device__ __forceinline__ double solve_chunk(double (&b)[LM], const double *rows, int ldx, int cnt, int p) {
  const double *fl = rows + RW_L * ldx, *fr = rows + RW_RINV * ldx, *fe = rows + RW_E * ldx;
  const double *fg = rows + RW_G * ldx, *fh = rows + RW_H * ldx;
  double acc = 0.0;
#pragma unroll
  for (int t = 0; t < LM; t++) {
    if (t < cnt) {
      acc = b[t] - fl[t * P + p] * acc;
      b[t] = acc;
    }
  }
  const double cin = scan_up(cnt > 0 ? fg[(cnt - 1) * P + p] : 1.0, cnt > 0 ? acc : 0.0, p);
  acc = 0.0;
#pragma unroll
  for (int t = LM - 1; t >= 0; t--) {
    if (t < cnt) {
      const int s = t * P + p;
      const double y = b[t] + fg[s] * cin;
      acc = y * fr[s] - fe[s] * acc;
      b[t] = acc;
    }
  }
  return scan_down(cnt > 0 ? fh[p] : 1.0, cnt > 0 ? acc : 0.0, p);
}

constexpr int SOLVE_WG = 512;                 // 8 waves, 32 columns per block
constexpr int SOLVE_COLS = SOLVE_WG / P;

// LDS bytes of k_column_solve: rows L..H of the three systems.
static size_t solve_lds(const Geom &g) { return sizeof(double) * SYS_N * RW_N * (size_t)g.ldx; }

template <int LM, typename OffT, bool NT>
__global__ void __launch_bounds__(SOLVE_WG)
    k_column_solve(FusedArgs a, const double *vz, const double *bx, const double *by, const double *bz,
                   const double *__restrict__ bt, double *ox, double *oy, double *oz, double *__restrict__ tn,
                   double *__restrict__ stalep, const double *__restrict__ facp) {
  extern __shared__ double rows[];   // [SYS_N][RW_N][ldx]
  const Geom g = a.g;
  const int64_t blk = xcd_block<0>((g.ncol + SOLVE_COLS - 1) / SOLVE_COLS);
  if (blk < 0 || (a.ds && coh_int(&a.ds->halted))) return;
  const int L = g.L, ldx = g.ldx, nx = g.nx, nxm = g.nxm;
  // the factor rows are the same for every column: stage them once per block
  for (int idx = threadIdx.x; idx < SYS_N * RW_N * ldx; idx += SOLVE_WG) {
    const int sr = idx / ldx, s = idx - sr * ldx;
    const int sys = sr / RW_N, r = sr - sys * RW_N;
    rows[idx] = facp[(sys * FR_N + FR_L + r) * ldx + s];
  }
  __syncthreads();
  const int p = threadIdx.x % P;
  const int64_t col = blk * SOLVE_COLS + threadIdx.x / P;
  const bool live = col < g.ncol;
  const int64_t colc = live ? col : 0;
  const OffT C = (OffT)colc * (OffT)g.ldx * sizeof(double);
  const int k0 = p * L;
  const int cntx = live ? max(0, min(L, nx - k0)) : 0;
  const int cntm = live ? max(0, min(L, nxm - k0)) : 0;
  const double *rX = rows + (SYS_X * RW_N) * ldx, *rY = rows + (SYS_YZ * RW_N) * ldx,
               *rT = rows + (SYS_T * RW_N) * ldx;
  // Row nx-1 of vy and vz is outside the nxm systems and keeps the field's
  // value; it is stored again with the rest, so that every 128-byte line of a
  // column is written whole (one broadcast load per column).
  const OffT Ctop = C + (OffT)pos_of_k(nx - 1, L) * sizeof(double);
  const double vytop = ldf(a.f.vy, Ctop), vztop = ldf(vz, Ctop);
  double b[LM];
  load_chunk<LM, OffT>(b, bx, C, cntx, L, p);
  {  // vx
    const double *fh = rX + RW_H * ldx;
    const double cin = solve_chunk<LM>(b, rX, ldx, cntx, p);
    if (live)
#pragma unroll
      for (int t = 0; t < LM; t++)
        if (t < L) {   // slots of k >= nx (t >= cntx) are written 0
          const int k = k0 + t, s = t * P + p;
          stf<NT>(ox, C + (OffT)s * sizeof(double), (k >= 1 && k <= nx - 2) ? b[t] + fh[s] * cin : 0.0);
        }
  }
  load_chunk<LM, OffT>(b, by, C, cntm, L, p);
  {  // vy
    const double *fh = rY + RW_H * ldx;
    const double cin = solve_chunk<LM>(b, rY, ldx, cntm, p);
    if (live)
#pragma unroll
      for (int t = 0; t < LM; t++)
        if (t < L) {
          const int k = k0 + t, s = t * P + p;
          stf<NT>(oy, C + (OffT)s * sizeof(double), k == nx - 1 ? vytop : (k < nxm ? b[t] + fh[s] * cin : 0.0));
        }
  }
  load_chunk<LM, OffT>(b, bz, C, cntm, L, p);
  // vz at k = 0 (slot 0) before the substep: the corrected one from the stale
  // row where the stencil pass corrected the fields
  const double vz0 = (live && p == 0) ? (a.dph ? stalep[colc] : ldf(vz, C)) : 0.0;
  double dvz0 = 0.0;
  {  // vz
    const double *fh = rY + RW_H * ldx;
    const double cin = solve_chunk<LM>(b, rY, ldx, cntm, p);
    dvz0 = b[0] + fh[p] * cin - vz0;   // used from lane p = 0 (k = 0) only
    if (live)
#pragma unroll
      for (int t = 0; t < LM; t++)
        if (t < L) {
          const int k = k0 + t, s = t * P + p;
          stf<NT>(oz, C + (OffT)s * sizeof(double), k == nx - 1 ? vztop : (k < nxm ? b[t] + fh[s] * cin : 0.0));
        }
  }
  dvz0 = __shfl(dvz0, 0, P);
  load_chunk<LM, OffT>(b, bt, C, cntx, L, p);
  if (live && p == 0) {
    stalep[colc] = dvz0;
    b[0] += dvz0;   // temperature row 1: rhs(1) = vz increment (lane 0 holds k = 0)
  }
  {  // temperature
    const double *fh = rT + RW_H * ldx;
    const double cin = solve_chunk<LM>(b, rT, ldx, cntx, p);
    if (live)
#pragma unroll
      for (int t = 0; t < LM; t++)
        if (t < L) {
          const int k = k0 + t, s = t * P + p;
          double y = b[t] + fh[s] * cin;
          y = k == 0 ? a.sc.tempbp : y;
          y = k == nx - 1 ? a.sc.temptp : y;
          stf<NT>(tn, C + (OffT)s * sizeof(double), k < nx ? y : 0.0);
        }
  }
}

// ---------------------------------------------------------------- per-routine kernels
// One thread per stored point, in the order of memory.  A point's row and lane
// of the interleaved layout give its k and the positions of k-1 and k+1 without
// a division; the two that are left are of 32 bits (a cell of 2^32 points would
// not fit the GPU).  The blocks keep the order in which they are dealt to the
// XCDs: with a contiguous range of columns per XCD, or with blocks of one row of
// sixteen columns, the right-hand sides took 99 us and the divergence 82 at
// 128x256x256, against 86 and 65 (88 and 66 with 64-bit divisions).
struct PointIdx {
  int col, j, i, s, k, skm, skp;   // skm, skp: positions of k-1 and k+1 (s itself at the ends of the column)
  bool live;
};
__device__ __forceinline__ PointIdx point_idx(const Geom &g) {
  PointIdx q;
  const uint32_t n = (uint32_t)g.ncol * (uint32_t)g.ldx;
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  q.live = gid < n;
  const uint32_t e = q.live ? (uint32_t)gid : 0u, col = e / (uint32_t)g.ldx;
  const int L = g.L;
  q.col = (int)col;
  q.s = (int)(e - col * (uint32_t)g.ldx);
  q.i = (int)(col / (uint32_t)g.nym);
  q.j = q.col - q.i * g.nym;
  const int row = q.s / P, lane = q.s % P;
  q.k = lane * L + row;
  q.skm = row > 0 ? q.s - P : (lane > 0 ? (L - 1) * P + lane - 1 : q.s);
  q.skp = row < L - 1 ? q.s + P : (lane < P - 1 ? lane + 1 : q.s);
  return q;
}

// The routines' results and histories, read once by a later routine: past the
// caches where the cell's fields are far larger than those (NT), which leaves
// them to the fields that neighbours share.  A template argument: the compiler
// folds a choice at run time into one ordinary access.
template <bool NT>
__device__ __forceinline__ double ld_stream(const double *p) {
  return NT ? __builtin_nontemporal_load(p) : *p;
}
template <bool NT>
__device__ __forceinline__ void st_stream(double *p, double v) {
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// ExplicitTerms*: one term (W: 0 vx, 1 vy, 2 vz, 3 temp) in the block shape of
// k_stencil_rhs, sixteen columns at sixteen positions marching through zplanes
// planes.  A point needs 13 to 18 values of four fields, most of them its y and z
// neighbours'; taken one point to a thread, their loads bound the pass at the rate
// of the caches.  Here the z neighbours are carried in registers and the y
// neighbours come through LDS, which leaves six to ten loads.  The four terms
// (vx, vy, vz, temp) took 126, 109, 107, 128 us at 128x256x256 and take 121,
// 80, 58, 104; 20, 16, 15, 18 and 20, 13, 13, 15 at 64x128x128.
// GC columns to a block: sixteen, or four or eight where nym holds no more, since
// the columns left over would be idle lanes.  The four terms together at nzm = 512,
// nxm = 128: nym = 2 17 us one point to a thread, 39 with sixteen columns, 21 with
// four; nym = 8 36, 40 and (eight) 27; nym = 16 67 and 42.
// Published per plane: the term's own field, then what the other columns need of
// the transporting ones.
constexpr int EX_N = 5;
template <int W, bool NT, int GC>
__global__ void __launch_bounds__(GC * ST_SP) k_explicit(RoutineArgs a, int zplanes) {
  __shared__ double xv[2][EX_N][GC * ST_SP];
  const Geom g = a.g;
  const int L = g.L, ldx = g.ldx, nq = ldx / ST_SP;
  const int ngr = (g.nym + GC - 1) / GC, nib = (g.nzm + zplanes - 1) / zplanes;
  const int64_t tile = xcd_block<64>((int64_t)nib * ngr * nq);
  if (tile < 0) return;
  const int q = (int)(tile % nq);
  const int64_t rest = tile / nq;
  const int gr = (int)(rest % ngr), ib = (int)(rest / ngr);
  const int tid = (int)threadIdx.x, w = tid / ST_SP;
  const int ncols = min(GC, g.nym - gr * GC);
  const bool colok = w < ncols;
  const int jc = colok ? gr * GC + w : g.nym - 1;   // idle threads read a valid column, store nothing
  const bool jp_in = w + 1 < ncols, jm_in = w > 0;
  const int jm = wrapm(jc - 1, g.nym), jp = wrapp(jc + 1, g.nym);
  const int s = q * ST_SP + tid % ST_SP, k = k_of_pos(s, L);
  const int sm = k >= 1 ? pos_of_k(k - 1, L) : s, sp = k + 1 < g.nx ? pos_of_k(k + 1, L) : s;
  // rows of the loops: vx, temp k = 1..nx-2; vy, vz k = 0..nxm-1, whose kmv/kpv stay inside
  const bool live = colok && (W == 0 || W == 3 ? k >= 1 && k <= g.nx - 2 : k <= g.nxm - 1);
  const int smm = k == 0 ? s : sm, spp = k == g.nxm - 1 ? s : sp;
  const StepScalars &c = a.sc;
  const double udx = a.kc[(W == 0 || W == 3 ? KC_UDX3C : KC_UDX3M) * ldx + s];
  const double *__restrict__ vx = a.f.vx, *__restrict__ vy = a.f.vy, *__restrict__ vz = a.f.vz;
  const double *__restrict__ f = W == 0 ? vx : (W == 1 ? vy : (W == 2 ? vz : a.f.temp));   // the term's own field
  double *__restrict__ out = a.out;
  const double udzq = W == 3 ? c.udzq_pe : c.udzq_re, udyq = W == 3 ? c.udyq_pe : c.udyq_re;
  const int i0 = ib * zplanes, i1 = min(i0 + zplanes, g.nzm);
  int64_t C = col_off(jc, i0, g);
  const int64_t CM = col_off(jc, wrapm(i0 - 1, g.nzm), g);
  double fim = f[CM + s], fc = f[C + s];
  // vx, vy, temp: vz at k (and k-1) of the plane; vz: vx at k+1 and k, vy and vy of j+1 of the plane before
  double zc = W != 2 ? vz[C + s] : 0.0, zm = W == 0 || W == 3 ? vz[C + sm] : 0.0;
  double xpi = 0.0, xci = 0.0, yci = 0.0, yjpi = 0.0;
  if constexpr (W == 2) {
    xpi = vx[CM + sp];
    xci = vx[CM + s];
    yci = vy[CM + s];
    yjpi = vy[col_off(jp, wrapm(i0 - 1, g.nzm), g) + s];
  }
  int par = 0;
  for (int ic = i0; ic < i1; ic++) {
    const int ip = wrapp(ic + 1, g.nzm);
    const int64_t CIP = col_off(jc, ip, g), CJM = col_off(jm, ic, g), CJP = col_off(jp, ic, g);
    const double fip = f[CIP + s];
    const double fm = f[C + (W == 0 || W == 3 ? sm : smm)], fp = f[C + (W == 0 || W == 3 ? sp : spp)];
    const double zip = W != 2 ? vz[CIP + s] : 0.0, zipm = W == 0 || W == 3 ? vz[CIP + sm] : 0.0;
    const double yc = W != 1 ? vy[C + s] : 0.0, ym = W == 0 || W == 3 ? vy[C + sm] : 0.0;
    const double xc = W != 0 ? vx[C + s] : 0.0, xp = W != 0 ? vx[C + sp] : 0.0, xm = W == 3 ? vx[C + sm] : 0.0;
    const double tc = W == 0 ? a.f.temp[C + s] : 0.0;
    double fjm = 0.0, fjp = 0.0, yjp = 0.0, yjpm = 0.0, xjm = 0.0, xjmp = 0.0, zjm = 0.0, zjmip = 0.0;
    if (!jp_in) {
      fjp = f[CJP + s];
      if (W != 1) yjp = vy[CJP + s];
      if (W == 0 || W == 3) yjpm = vy[CJP + sm];
    }
    if (!jm_in) {
      fjm = f[CJM + s];
      if (W == 1) {
        xjm = vx[CJM + s];
        xjmp = vx[CJM + sp];
        zjm = vz[CJM + s];
        zjmip = vz[col_off(jm, ip, g) + s];
      }
    }
    double (*buf)[GC * ST_SP] = xv[par];
    buf[0][tid] = fc;
    if (W != 1) buf[1][tid] = yc;
    if (W == 0 || W == 3) buf[2][tid] = ym;
    if (W == 1) {
      buf[1][tid] = xc;
      buf[2][tid] = xp;
      buf[3][tid] = zc;
      buf[4][tid] = zip;
    }
    __syncthreads();
    if (jp_in) {
      const int o = tid + ST_SP;
      fjp = buf[0][o];
      if (W != 1) yjp = buf[1][o];
      if (W == 0 || W == 3) yjpm = buf[2][o];
    }
    if (jm_in) {
      const int o = tid - ST_SP;
      fjm = buf[0][o];
      if (W == 1) {
        xjm = buf[1][o];
        xjmp = buf[2][o];
        zjm = buf[3][o];
        zjmip = buf[4][o];
      }
    }
    par ^= 1;
    const double dzz = (fim - 2.0 * fc + fip) * udzq, dyy = (fjm - 2.0 * fc + fjp) * udyq;
    double hx, hy, hz, v;
    if constexpr (W == 0) {   // ExplicitTermsVX.F90:55-101
      hz = (((zip + zipm) * (fip + fc)) - ((zc + zm) * (fc + fim))) * c.udz4;
      hy = (((yjp + yjpm) * (fjp + fc)) - ((yc + ym) * (fc + fjm))) * c.udy4;
      const double p = fp + fc, m = fc + fm;
      hx = (p * p - m * m) * udx * 0.25;
      v = -(hx + hy + hz) + dyy + dzz + tc;
    } else if constexpr (W == 1) {   // ExplicitTermsVY.F90:52-98
      hx = ((xp + xjmp) * (fp + fc) - (xc + xjm) * (fc + fm)) * udx * 0.25;
      const double p = fjp + fc, m = fjm + fc;
      hy = (p * p - m * m) * c.udy4;
      hz = ((fip + fc) * (zip + zjmip) - (fc + fim) * (zc + zjm)) * c.udz4;
      v = -(hx + hy + hz) + dyy + dzz;
    } else if constexpr (W == 2) {   // ExplicitTermsVZ.F90:56-101
      const double p = fip + fc, m = fim + fc;
      hz = (p * p - m * m) * c.udz4;
      hy = ((yjp + yjpi) * (fjp + fc) - (yc + yci) * (fc + fjm)) * c.udy4;
      hx = ((xp + xpi) * (fp + fc) - (xc + xci) * (fc + fm)) * udx * 0.25;
      v = -(hx + hy + hz) + dyy + dzz;
    } else {   // ExplicitTermsTemp.F90:52-93
      hz = ((zipm + zip) * (fip + fc) - (zm + zc) * (fc + fim)) * c.udz4;
      hy = ((yjp + yjpm) * (fjp + fc) - (yc + ym) * (fc + fjm)) * c.udy4;
      hx = ((xp + xc) * (fp + fc) - (xc + xm) * (fc + fm)) * udx * 0.25;
      v = -(hx + hy + hz) + dyy + dzz;
    }
    if (live) st_stream<NT>(&out[C + s], v);
    fim = fc; fc = fip;
    zc = zip; zm = zipm;
    xpi = xp; xci = xc; yci = yc; yjpi = yjp;
    C = CIP;
  }
}

// ImplicitAndUpdate* RHS loops: rhs (unscaled) and history ru = explicit term.
template <bool NT>
__global__ void __launch_bounds__(256) k_rhs(RoutineArgs a, int which) {
  const Geom g = a.g;
  const PointIdx q = point_idx(g);
  if (!q.live) return;
  const Nb n = make_nb(q.j, q.i, g);
  const int k = q.k, s = q.s, ldx = g.ldx;
  const double *kc = a.kc;
  const int64_t o = n.C + s;
  if (which == 0 || which == 3) {
    if (k < 1 || k > g.nx - 2) return;
    double qv = ld_stream<NT>(&a.expl[o]);
    double ru = a.sc.use_ru ? ld_stream<NT>(&a.ru[o]) : 0.0;
    const double r = which == 0 ? rhs_vx(qv, ru, a.f.vx, a.f.pr, n, s, q.skm, q.skp, kc, ldx, a.sc)
                                : rhs_temp(qv, ru, a.f.temp, n, s, q.skm, q.skp, kc, ldx, a.sc);
    st_stream<NT>(&a.ru[o], qv);
    st_stream<NT>(&a.rhs[o], r);
  } else {
    if (k > g.nxm - 1) return;
    const int skmm = k == 0 ? s : q.skm, skpp = k == g.nxm - 1 ? s : q.skp;
    double qv = ld_stream<NT>(&a.expl[o]);
    double ru = a.sc.use_ru ? ld_stream<NT>(&a.ru[o]) : 0.0;
    const double r = which == 1 ? rhs_vy(qv, ru, a.f.vy, a.f.pr, n, s, skmm, skpp, kc, ldx, a.sc)
                                : rhs_vz(qv, ru, a.f.vz, a.f.pr, n, s, skmm, skpp, kc, ldx, a.sc);
    st_stream<NT>(&a.ru[o], qv);
    st_stream<NT>(&a.rhs[o], r);
  }
}

// SolveImpEqnUpdate_{X,YZ,Temp}: scale rhs rows, solve in place (rhs receives
// the increments, as dgttrs overwrites B), add to the field, apply the
// ImplicitAndUpdate* boundary rows.  which: 0 vx, 1 vy, 2 vz, 3 temp.  The
// column solve's shape: a lane's chunk of the right-hand side and of the field
// in registers, loaded in one batch, the factor rows in LDS, every stored line
// written whole (rows outside the system and padding as they were).  Walked
// row by row through LDS it took 109 us a routine at 128x256x256, now 64.
template <int LM>
__global__ void __launch_bounds__(SOLVE_WG) k_solve_update(SolveArgs a, int which) {
  extern __shared__ double rows[];   // [FR_SCALE..FR_H][ldx]
  const Geom g = a.g;
  const int64_t blk = xcd_block<0>((g.ncol + SOLVE_COLS - 1) / SOLVE_COLS);
  if (blk < 0) return;
  const int L = g.L, ldx = g.ldx, nx = g.nx, nxm = g.nxm;
  for (int idx = threadIdx.x; idx < (FR_H + 1) * ldx; idx += SOLVE_WG) rows[idx] = a.fac[idx];
  __syncthreads();
  const int p = threadIdx.x % P;
  const int64_t col = blk * SOLVE_COLS + threadIdx.x / P;
  const bool live = col < g.ncol;
  const int64_t C = (live ? col : 0) * g.ldx;
  const bool yz = which == 1 || which == 2;
  const int nsys = yz ? nxm : nx;
  const int k0 = p * L;
  const int cnt = live ? max(0, min(L, nsys - k0)) : 0;
  double q[LM], b[LM];
#pragma unroll
  for (int t = 0; t < LM; t++) b[t] = a.rhs[C + min(t, L - 1) * P + p];
#pragma unroll
  for (int t = 0; t < LM; t++) q[t] = a.q[C + min(t, L - 1) * P + p];
  const double st0 = p == 0 && !yz ? a.stale[live ? col : 0] : 0.0;
#pragma unroll
  for (int t = 0; t < LM; t++) {
    const int k = k0 + t;
    if (t >= cnt) b[t] = 0.0;
    else if (yz || (k >= 1 && k <= nx - 2)) b[t] = b[t] * rows[FR_SCALE * ldx + t * P + p];
    else if (k == 0) b[t] = st0;   // else rhs(nx): identity row, never written by the reference routines
  }
  const double *sys = rows + FR_L * ldx, *fh = rows + FR_H * ldx;
  const double cin = solve_chunk<LM>(b, sys, ldx, cnt, p);
  if (!live) return;
#pragma unroll
  for (int t = 0; t < LM; t++) {
    if (t < L) {
      const int k = k0 + t, s = t * P + p;
      const double x = b[t] + fh[s] * cin;
      const double r = t < cnt && (yz || k <= nx - 2) ? x : a.rhs[C + s];   // few lanes read again
      double v = q[t];
      if (t < cnt) {
        if (yz || (k >= 1 && k <= nx - 2)) v = v + x;
        if (which == 0 && (k == 0 || k == nx - 1)) v = 0.0;
        if (which == 3 && k == 0) v = a.tempbp;
        if (which == 3 && k == nx - 1) v = a.temptp;
        if (yz && k == 0) a.stale[col] = x;
      }
      a.rhs[C + s] = r;
      a.q[C + s] = v;
    }
  }
}

// CalcLocalDivergence.F90:27-41 -> dph (k = 0..nxm-1)
__global__ void __launch_bounds__(256) k_divergence(RoutineArgs a) {
  const Geom g = a.g;
  const PointIdx q = point_idx(g);
  if (!q.live || q.k > g.nxm - 1) return;
  const int64_t C = col_off(q.j, q.i, g), CJP = col_off(wrapp(q.j + 1, g.nym), q.i, g),
                CIP = col_off(q.j, wrapp(q.i + 1, g.nzm), g);
  const int s = q.s;
  const double usdtal = 1.0 / (a.sc.dt * a.sc.al);
  double dqcap = (a.f.vz[CIP + s] - a.f.vz[C + s]) * a.sc.dz + (a.f.vy[CJP + s] - a.f.vy[C + s]) * a.sc.dy +
                 (a.f.vx[C + q.skp] - a.f.vx[C + s]) * a.kc[KC_UDX3M * g.ldx + s];
  a.out[C + s] = dqcap * usdtal;
}

// CorrectVelocity.F90:28-45 and CorrectPressure.F90:32-52 from dph (= dphhalo).
// which: 1 velocity, 2 pressure, 3 both (the substep path).  The velocities
// are read from (ux, uy, uz) and written to (vx, vy, vz): the u* buffers of
// the substep path, or the fields themselves (in place) for the per-routine
// entries and the refinement sweep.  The block shape is that of
// k_stencil_rhs: ST_GC neighbouring y columns at the same ST_SP stored
// positions, marching through zplanes z planes with dph of planes i-1, i, i+1
// in registers; each thread publishes its plane-i dph in LDS for its y
// neighbours (double-buffered, one barrier per plane), so only the group's
// edge columns load a y neighbour.
//
// CFL = true (the last correction of a device step, not in place) also
// reduces CalcMaxCFL.F90:26-41 over the corrected velocities into
// a.cflbits (the bits of a non-negative double, so an integer atomic max is
// the floating-point max).  The corrected value of each neighbour a point
// needs (vx at k+1, vy at j+1, vz at i+1) is recomputed from u* and dph by
// the same fused multiply-add that stores it, so the maximum equals that of
// k_red_cfl over the stored fields bit for bit.
constexpr int CZ_ROWS = 6;   // udx3c, amphk, acphk, apphk, udx3m, udx3c at k+1
template <bool CFL, bool NT>
__global__ void __launch_bounds__(SY_WG) k_correct(CorrectArgs a, int which, int zplanes) {
  extern __shared__ double sh[];
  double *cr = sh;                    // [CZ_ROWS][ST_SP]
  double *xv = sh + CZ_ROWS * ST_SP;  // [2][2][SY_WG] published dph (and u*_y) of plane i
  const Geom g = a.g;
  const int L = g.L, ldx = g.ldx, nxm = g.nxm;
  const int nq = (ldx + ST_SP - 1) / ST_SP;
  const int ngr = (g.nym + ST_GC - 1) / ST_GC;
  const int nib = (g.nzm + zplanes - 1) / zplanes;
  const int64_t tile = xcd_block<0>((int64_t)nib * ngr * nq);
  if (tile < 0 || (a.ds && coh_int(&a.ds->halted))) return;
  const int q = (int)(tile % nq);
  const int64_t rest = tile / nq;
  const int gr = (int)(rest % ngr), ib = (int)(rest / ngr);
  const StepScalars c = a.ds ? coh_scalars(&a.ds->sc[a.ns - 1]) : a.sc;
  for (int idx = threadIdx.x; idx < CZ_ROWS * ST_SP; idx += SY_WG) {
    const int r = idx / ST_SP, sl = min(q * ST_SP + idx - r * ST_SP, ldx - 1);
    int sp = sl;
    if (r == 5) {   // the position of k+1 (k+1 <= nx-1 holds for every stored k < nx-1)
      const int kk = k_of_pos(sl, L);
      sp = kk + 1 < g.nx ? pos_of_k(kk + 1, L) : sl;
    }
    const int src = r == 0 || r == 5 ? KC_UDX3C
                    : (r == 1 ? KC_AMPHK : (r == 2 ? KC_ACPHK : (r == 3 ? KC_APPHK : KC_UDX3M)));
    cr[idx] = a.kc[src * ldx + sp];
  }
  __syncthreads();
  const int lane = (int)threadIdx.x & (ST_SP - 1);   // position within the tile
  const int w = (int)threadIdx.x / ST_SP;             // column within the group
  const int ncols = min(ST_GC, g.nym - gr * ST_GC);
  const bool colok = w < ncols;
  const int jc = colok ? gr * ST_GC + w : g.nym - 1;
  const int sraw = q * ST_SP + lane;
  const int s = min(sraw, ldx - 1);
  const int k = k_of_pos(s, L);
  const bool live = colok && sraw < ldx && k <= nxm - 1;
  // Positions k >= nxm (the wall row of vx, where u* is 0, row nx-1 of the
  // other fields, and the padding) keep what u* and pr hold there; they are
  // stored too, so that every 128-byte line of a column is written whole.
  const bool stv = colok && sraw < ldx;
  const bool jp_in = w + 1 < ncols, jm_in = w > 0;
  const int jm = wrapm(jc - 1, g.nym), jp = wrapp(jc + 1, g.nym);
  const int skm = (k == 0 || k > nxm - 1) ? s : pos_of_k(k - 1, L);
  const int skp = (k >= nxm - 1) ? s : pos_of_k(k + 1, L);
  const int sx1 = k + 1 < g.nx ? pos_of_k(k + 1, L) : s;   // vx at k+1 (the wall row for k = nxm-1)
  const double *__restrict__ dph = a.dph;
  const double *ux = a.ux, *uy = a.uy, *uz = a.uz;
  double *qx = a.vx, *qy = a.vy, *qz = a.vz, *__restrict__ qp = a.pr;
  const double usukm = c.al * c.dt * cr[lane];   // row r of cr at cr[r * ST_SP + lane]
  const double udy = c.al * c.dt * c.dy, udz = c.al * c.dt * c.dz;
  const double be = c.al * c.beta;
  const double amm = cr[ST_SP + lane], acc = cr[2 * ST_SP + lane], app = cr[3 * ST_SP + lane];
  const double u3m = cr[4 * ST_SP + lane], usukp = c.al * c.dt * cr[5 * ST_SP + lane];
  const int i0 = ib * zplanes, i1 = min(i0 + zplanes, g.nzm);
  double dim_ = dph[col_off(jc, wrapm(i0 - 1, g.nzm), g) + s];
  double d = dph[col_off(jc, i0, g) + s];
  double uzc = CFL ? uz[col_off(jc, i0, g) + s] : 0.0;   // u*_z of the current plane, carried
  const int tid = (int)threadIdx.x;
  int par = 0;
  double cflm = 0.0;
  for (int ic = i0; ic < i1; ic++) {
    const int64_t C = col_off(jc, ic, g);
    const int64_t CIP = col_off(jc, wrapp(ic + 1, g.nzm), g);
    const double dip = dph[CIP + s];
    const double dkm = dph[C + skm], dkp = dph[C + skp];
    double djm = 0.0, djp = 0.0;
    if (!jm_in) djm = dph[col_off(jm, ic, g) + s];
    if (!jp_in) djp = dph[col_off(jp, ic, g) + s];
    double vxo = 0.0, vyo = 0.0, vzo = 0.0, pro = 0.0;
    double uxk1 = 0.0, uyjp = 0.0, uzip = 0.0;
    if (which & 1) {   // read here only (streamed: 2 % less fetched, 2 % faster)
      vxo = ld_stream<NT>(&ux[C + s]);
      vyo = ld_stream<NT>(&uy[C + s]);
      vzo = CFL ? uzc : ld_stream<NT>(&uz[C + s]);
    }
    if (CFL) {
      uxk1 = ux[C + sx1];
      uzip = uz[CIP + s];
      if (!jp_in) uyjp = uy[col_off(jp, ic, g) + s];
    }
    if (which & 2) pro = ld_stream<NT>(&qp[C + s]);
    double *buf = xv + par * (2 * SY_WG);
    buf[tid] = d;
    if (CFL) buf[SY_WG + tid] = vyo;
    __syncthreads();
    if (jm_in) djm = buf[tid - ST_SP];
    if (jp_in) djp = buf[tid + ST_SP];
    if (CFL && jp_in) uyjp = buf[SY_WG + tid + ST_SP];
    par ^= 1;
    if (stv) {
      if (which & 1) {
        const double nvx = corr(vxo, d - dkm, usukm);
        const double nvy = corr(vyo, d - djm, udy);
        const double nvz = corr(vzo, d - dim_, udz);
        qx[C + s] = live ? nvx : vxo;
        qy[C + s] = live ? nvy : vyo;
        qz[C + s] = live ? nvz : vzo;
        if (CFL && live) {
          const double nvxk1 = k + 1 <= nxm - 1 ? corr(uxk1, dkp - d, usukp) : uxk1;
          const double nvyjp = corr(uyjp, djp - d, udy);
          const double nvzip = corr(uzip, dip - d, udz);
          const double qcf = (fabs((nvz + nvzip) * 0.5 * c.dz) + fabs((nvy + nvyjp) * 0.5 * c.dy) +
                              fabs((nvx + nvxk1) * 0.5 * u3m));
          cflm = fmax(cflm, qcf);
        }
      }
      if (which & 2)
        qp[C + s] = live ? corr_pr(pro, d, dkm, dkp, djm, djp, dim_, dip, be, c.dzq, c.dyq, amm, acc, app) : pro;
    }
    dim_ = d;
    d = dip;
    uzc = uzip;
  }
  if (CFL) {   // one atomic per block
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) cflm = fmax(cflm, __shfl_xor(cflm, off, 64));
    __syncthreads();   // every wave is past its last read of xv
    if ((threadIdx.x & 63) == 0) xv[threadIdx.x >> 6] = cflm;
    __syncthreads();
    if (threadIdx.x == 0) {
      double m = xv[0];
      for (int q = 1; q < SY_WG / 64; q++) m = fmax(m, xv[q]);
      atomicMax(a.cflbits, (unsigned long long)__double_as_longlong(m));
    }
  }
}

// ---------------------------------------------------------------- launchers
#define AFID_LM_LIST(X) X(2) X(4) X(8) X(12) X(16) X(25) X(32) X(48) X(64) X(80)

static int pick_lm(int L) {
  const int lms[] = {2, 4, 8, 12, 16, 25, 32, 48, 64, 80};
  for (int v : lms)
    if (L <= v) return v;
  return -1;
}

hipError_t column_configure_lds(size_t bytes) {
  hipError_t e = hipSuccess;
#define SETB(V)                                                                                          \
  SETC1(V, uint32_t, true) SETC1(V, uint32_t, false) SETC1(V, uint64_t, true)
#define SETC1(V, O, NT)                                                                                  \
  e = hipFuncSetAttribute((const void *)k_column_solve<V, O, NT>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                          (int)bytes);                                                                   \
  if (e != hipSuccess) return e;
  AFID_LM_LIST(SETB)
#undef SETC1
#undef SETB
  return hipSuccess;
}

// z planes per block of the stencil and correction passes, whose blocks march
// serially through their planes.  A large cell takes ZM_MAX planes (each run's
// first planes are read twice); a small one shorter runs, since 32 planes leave
// it with fewer blocks than the GPU holds at once and its time is that of one
// block's march: at 32x64x64 24 blocks took 61 us (stencil) and 35 us
// (correction), two planes 14 and 10; 64x128x128 73 and 37, now 49 and 24;
// 128x256x256 294 and 143, now 279 and 139.  The rule takes the run with the
// least (waves of resident blocks) x (planes + RUN_IN), RUN_IN standing for a
// run's start-up; one plane only was slower everywhere (66.8 us against 49 at
// 64x128x128).  `resident` is what the registers let 256 CUs hold.
constexpr int RUN_IN = 2;
constexpr int STENCIL_RESIDENT = 3 * 256, STENCIL_CORR_RESIDENT = 2 * 256;
constexpr int CORRECT_RESIDENT = 7 * 256, EXPLICIT_RESIDENT = 7 * 256;
static int march_planes(const Geom &g, int resident, int most) {
  const int64_t strips = (int64_t)((g.nym + ST_GC - 1) / ST_GC) * ((g.ldx + ST_SP - 1) / ST_SP);
  int best = std::min(2, g.nzm);
  int64_t least = INT64_MAX;
  for (int zm = best; zm <= std::min(most, g.nzm); zm++) {
    const int64_t blocks = strips * ((g.nzm + zm - 1) / zm);
    const int64_t cost = (blocks + resident - 1) / resident * (zm + RUN_IN);
    if (cost <= least) {   // of equals the longer run, which re-reads less
      least = cost;
      best = zm;
    }
  }
  return best;
}
int stencil_planes(const Geom &g, bool corrects, int zm) {
  return march_planes(g, corrects ? STENCIL_CORR_RESIDENT : STENCIL_RESIDENT, zm > 0 ? zm : ZM_MAX);
}
hipError_t launch_stencil_rhs(const FusedArgs &args, hipStream_t st) {
  FusedArgs a = args;
  const int64_t n = a.g.ncol * a.g.ldx;
  a.zm = stencil_planes(a.g, a.dph != nullptr, a.zm);
  const int zplanes = a.zm;
  const int64_t ntile = (int64_t)((a.g.nzm + zplanes - 1) / zplanes) * ((a.g.nym + ST_GC - 1) / ST_GC) *
                        ((a.g.ldx + ST_SP - 1) / ST_SP);
  const dim3 grid((unsigned)(((ntile + 7) / 8) * 8));
  const size_t shm = stencil_lds(a.dph != nullptr);
  const bool small = (uint64_t)n * sizeof(double) < (1ull << 32);
  const bool ru = a.sc.use_ru != 0, dev = a.ds != nullptr, h32 = a.h32 != 0;
  const int cm = small ? cache_mode(a.g) : CM_STREAM;
#define SR1(O, R, D, H, K, M)                                                                            \
  if (std::is_same<O, uint32_t>::value == small && R == ru && D == dev && H == h32 && K == (a.dph != nullptr) && M == cm) { \
    hipLaunchKernelGGL((k_stencil_rhs<O, R, D, H, K, M>), grid, dim3(SY_WG), shm, st, a, a.f.vx, a.f.vy, \
                       a.f.vz, a.f.temp, a.f.pr, a.rux, a.ruy, a.ruz, a.rut, a.bx, a.by, a.bz, a.bt, a.stale, \
                       a.kc, a.fac, a.dph, a.pr_out);                                                  \
    return hipGetLastError();                                                                          \
  }
#define SR2(O, R, K, M) \
  SR1(O, R, true, false, K, M) SR1(O, R, false, false, K, M) SR1(O, R, true, true, K, M) SR1(O, R, false, true, K, M)
#define SR(O, M) SR2(O, true, false, M) SR2(O, false, false, M)
  SR(uint32_t, CM_STREAM) SR(uint32_t, CM_HIST) SR(uint32_t, CM_KEEP) SR(uint64_t, CM_STREAM)
  SR2(uint32_t, true, true, CM_STREAM) SR2(uint32_t, true, true, CM_HIST) SR2(uint32_t, true, true, CM_KEEP)
#undef SR
#undef SR2
#undef SR1
  return hipErrorInvalidValue;
}

hipError_t launch_column_solve(const FusedArgs &a, hipStream_t st) {
  const bool small = (uint64_t)a.g.ncol * a.g.ldx * sizeof(double) < (1ull << 32);
  const int64_t nblk = (a.g.ncol + SOLVE_COLS - 1) / SOLVE_COLS;
  const dim3 grid((unsigned)(((nblk + 7) / 8) * 8));
  const size_t shm = solve_lds(a.g);
  switch (pick_lm(a.g.L)) {
#define GO(V, O, NT)                                                                                   \
  hipLaunchKernelGGL((k_column_solve<V, O, NT>), grid, dim3(SOLVE_WG), shm, st, a, a.f.vz, a.bx, a.by, \
                     a.bz, a.bt, a.ux, a.uy, a.uz, a.tn, a.stale, a.fac);
#define CASE(V)                                                                                        \
  case V:                                                                                              \
    if (!small) GO(V, uint64_t, true)                                                                  \
    else if (cache_mode(a.g) == CM_STREAM) GO(V, uint32_t, true)                                       \
    else GO(V, uint32_t, false)                                                                        \
    return hipGetLastError();
    AFID_LM_LIST(CASE)
#undef CASE
#undef GO
    default: break;
  }
  return hipErrorInvalidValue;
}

hipError_t launch_solve_update(const SolveArgs &a, int which, hipStream_t st) {
  const int64_t nblk = (a.g.ncol + SOLVE_COLS - 1) / SOLVE_COLS;
  const dim3 grid((unsigned)(((nblk + 7) / 8) * 8));
  const size_t shm = sizeof(double) * (FR_H + 1) * (size_t)a.g.ldx;   // at most 60 KiB
  switch (pick_lm(a.g.L)) {
#define CASE(V)                                                                                   \
  case V: hipLaunchKernelGGL(k_solve_update<V>, grid, dim3(SOLVE_WG), shm, st, a, which); break;
    AFID_LM_LIST(CASE)
#undef CASE
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

static dim3 point_grid(const Geom &g) {
  return dim3((unsigned)((g.ncol * g.ldx + 255) / 256));
}

// Fields from 32 MiB stream: the eight or so of a routine's cycle then outgrow the
// 256 MiB cache.  A substep by routines took 1480 us without and 1383 with it at
// 128x256x256 (72 MiB a field), 905 and 866 at 159x192x192 (45), as long with
// either at 117x135x150 (20), 238 and 245 at 64x128x128 (10).
static bool streams(const Geom &g) { return cache_mode(g) == CM_STREAM; }
hipError_t launch_explicit(const RoutineArgs &a, int which, hipStream_t st) {
  const int zplanes = march_planes(a.g, EXPLICIT_RESIDENT, ZM_MAX);
  const int gc = a.g.nym <= 4 ? 4 : (a.g.nym <= 8 ? 8 : ST_GC);
  const int64_t ntile = (int64_t)((a.g.nzm + zplanes - 1) / zplanes) * ((a.g.nym + gc - 1) / gc) * (a.g.ldx / ST_SP);
  const dim3 grid((unsigned)(((ntile + 7) / 8) * 8));
  const bool nt = streams(a.g);
#define GO(W, NT, GC)                                                                        \
  if (which == W && nt == NT && gc == GC) {                                                  \
    hipLaunchKernelGGL((k_explicit<W, NT, GC>), grid, dim3(GC * ST_SP), 0, st, a, zplanes);  \
    return hipGetLastError();                                                                \
  }
#define GOW(NT, GC) GO(0, NT, GC) GO(1, NT, GC) GO(2, NT, GC) GO(3, NT, GC)
  GOW(false, ST_GC) GOW(true, ST_GC) GOW(false, 8) GOW(true, 8) GOW(false, 4) GOW(true, 4)
#undef GOW
#undef GO
  return hipErrorInvalidValue;
}
hipError_t launch_rhs(const RoutineArgs &a, int which, hipStream_t st) {
  if (streams(a.g)) hipLaunchKernelGGL(k_rhs<true>, point_grid(a.g), dim3(256), 0, st, a, which);
  else hipLaunchKernelGGL(k_rhs<false>, point_grid(a.g), dim3(256), 0, st, a, which);
  return hipGetLastError();
}
hipError_t launch_divergence(const RoutineArgs &a, hipStream_t st) {
  hipLaunchKernelGGL(k_divergence, point_grid(a.g), dim3(256), 0, st, a);
  return hipGetLastError();
}
hipError_t launch_correct(const CorrectArgs &a, int which, hipStream_t st) {
  const int zplanes = march_planes(a.g, CORRECT_RESIDENT, ZM_MAX);
  const int64_t nt = (int64_t)((a.g.nzm + zplanes - 1) / zplanes) * ((a.g.nym + ST_GC - 1) / ST_GC) *
                     ((a.g.ldx + ST_SP - 1) / ST_SP);
  const size_t shm = sizeof(double) * (CZ_ROWS * ST_SP + 2 * 2 * SY_WG);
  const dim3 grid((unsigned)(((nt + 7) / 8) * 8));
  const bool stream = cache_mode(a.g) == CM_STREAM;
  if (a.cflbits && (which != 3 || a.ux == a.vx)) return hipErrorInvalidValue;   // the fold needs u* apart from the fields
  if (a.cflbits && stream) hipLaunchKernelGGL((k_correct<true, true>), grid, dim3(SY_WG), shm, st, a, which, zplanes);
  else if (a.cflbits) hipLaunchKernelGGL((k_correct<true, false>), grid, dim3(SY_WG), shm, st, a, which, zplanes);
  else if (stream) hipLaunchKernelGGL((k_correct<false, true>), grid, dim3(SY_WG), shm, st, a, which, zplanes);
  else hipLaunchKernelGGL((k_correct<false, false>), grid, dim3(SY_WG), shm, st, a, which, zplanes);
  return hipGetLastError();
}

// LDS per block: SC_NC*ST_SP + 2*SV_NC*SY_WG doubles (correcting stencil pass), SYS_N*RW_N*16*L (column
// solve), 6*16*L (per-routine solve); L <= 80 keeps all within gfx950's 160 KiB.
int max_supported_L() { return 80; }
size_t column_lds_need(const Geom &g) {
  size_t b = std::max(stencil_lds(true), solve_lds(g));
  return b;
}

}  // namespace afid
