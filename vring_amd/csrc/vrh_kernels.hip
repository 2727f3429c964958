// vrh_kernels.hip -- gfx950 kernels of the vring RK3 substep.
//
// All kernels read and write HBM-resident fields in the reference's Fortran
// layout (theta fastest), so 64-lane wavefronts always span contiguous theta
// rows and every global access is coalesced.  TW is the work type (double in
// the FP64 path, float in the mixed path); the state q, the predictor dq,
// phi and p are always double.
#include <hip/hip_runtime.h>
#include <rocblas/rocblas.h>

#include <cmath>
#include <mutex>

#include "vrh_internal.h"

namespace {

template <typename T> __device__ __forceinline__ T ldg(const T *p) { return __builtin_nontemporal_load(p); }

// The block's logical (x, y, z) coordinates of a 2-D or 3-D grid in the
// order of xcd_tile, x fastest: tiles adjacent in x (whose halo rows
// overlap) share an L2.
__device__ __forceinline__ void xcd_block(int &bx, int &by, int &bz) {
  const long nx = gridDim.x, ny = gridDim.y, nb = nx * ny * (long)gridDim.z;
  const long l = xcd_tile((long)blockIdx.x + nx * ((long)blockIdx.y + ny * (long)blockIdx.z), nb);
  bx = (int)(l % nx);
  const long r = l / nx;
  by = (int)(r % ny);
  bz = (int)(r / ny);
}

// Inlet time profile (gen_tools_swirl.F90:159-175): smooth ramp to 1 over
// 0.1n, hold until n, ramp down (n = 2).
__device__ __host__ inline double profile_fn(double t) {
  const double n = 2.0, t1 = (double)0.1f * n;
  double u = 0.0;
  if (t > 0.0 && t < t1) { double x = t / t1; u = 3.0 * (x * x) - 2.0 * (x * x * x); }
  if (t > t1 && t < n) u = 1.0;
  if (t > n && t < n + t1) { double x = (n + t1 - t) / t1; u = 3.0 * (x * x) - 2.0 * (x * x * x); }
  if (t > n + t1) u = 0.0;
  return u;
}

// Per-step scalars (loop.F90:53; momentum_terms_swirl.F90:192-212, 261-283):
// advance ntime by dt, then for each substep the inlet increment
// c3s = (profile(t+dt) - profile(t)) alpha and the mass-correction factor
// cor = c3s * inlet_area / (sum qc^2 da + 1e-15).
__global__ void k_scalars(double *sc, double dt, double a1, double a2, double a3, double inlet_area,
                          double cor_red, int advance, double t_set) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  const double t = advance ? dt + sc[0] : t_set;
  sc[0] = t;
  const double u0 = profile_fn(t), u1 = profile_fn(t + dt);
  const double al[3] = {a1, a2, a3};
  for (int q = 0; q < 3; q++) {
    const double c3s = (u1 - u0) * al[q];
    sc[1 + q] = c3s;
    sc[4 + q] = (c3s * inlet_area - 0.0) / (cor_red + (double)1.e-15f);
  }
}

// ---------------------------------------------------------------------------
// Explicit part: hdnl1-3 (momentum_terms_swirl.F90:15-174) fused with the
// explicit right-hand sides of step (step.F90:32-165) and the periodic theta
// solves solqi/tripij (step.F90:212-263, 487-534).
// A block owns whole theta rows (NTP >= nt lanes) of RJ consecutive r rows
// and marches up a chunk of z planes.  The planes k-1, k, k+1 of q1, q2, q3
// (rows j0-1 .. j0+RJ) sit in a 3-slot LDS ring, so every stencil operand
// comes from LDS; the next plane is prefetched into registers while the
// current one is computed.  The theta systems (constant coefficients
// (-acc, 1+2acc, -acc) per r row) are solved by parallel cyclic reduction
// on LDS-resident lines.  Row coefficients, reduction ratios and the depth
// of each row's reduction come from host tables (explicit_tables).  The inlet planes q1s, q2s, q3s are zero
// (momentum_terms_swirl.F90:216-223).
// ---------------------------------------------------------------------------

// z second differences on the axial mesh (ZMet, vrh_set_axial_mesh): at a
// cell centre (q1, q2, p, the first two pressure-gradient components) with
// the one-sided form through the wall value 0 in the inlet cell, and at a
// face (q3, the third component)
template <typename T> __device__ __forceinline__ T zd2c(const ZMet &z, int k, T fm1, T f0, T fp1) {
  if (k == 1) return (fp1 - f0) * (T)z.w2 - (f0 - (T)0) * (T)z.ws;
  return (fp1 - f0) * (T)z.cp[k] - (f0 - fm1) * (T)z.cm[k];
}
template <typename T> __device__ __forceinline__ T zd2f(const ZMet &z, int k, T fm1, T f0, T fp1) {
  return (fp1 - f0) * (T)z.fp[k] - (f0 - fm1) * (T)z.fm[k];
}

template <typename TW, typename TC, bool ZS>
__global__ __launch_bounds__(512, sizeof(TC) == 4 ? 4 : 3) void k_explicit_march(VGrid g, const double *__restrict__ rowc, const double *__restrict__ pcrt, VRK rk, ZMet zm, int kchunk,
                                                  const double *__restrict__ q1, const double *__restrict__ q2,
                                                  const double *__restrict__ q3, const double *__restrict__ prg1,
                                                  const double *__restrict__ prg2, const double *__restrict__ prg3,
                                                  TW *__restrict__ ru1, TW *__restrict__ ru2, TW *__restrict__ ru3,
                                                  TW *__restrict__ r1, TW *__restrict__ r2, TW *__restrict__ r3) {
  extern __shared__ unsigned char smem_raw[];
  const int NTP = blockDim.x, RJ = blockDim.y, ti = threadIdx.x, tj = threadIdx.y;
  const int NTH = NTP * RJ, tid = tj * NTP + ti;
  const int nt = g.nt, nr = g.nr, nz = g.nz;
  const long sj = g.sj, sk = g.sk;
  int bx, by, bz;
  xcd_block(bx, by, bz);  // r blocks of one z chunk (sharing halo rows) on one XCD
  const int j0 = 1 + bx * RJ;
  const int kb = 1 + by * kchunk, ke = min(kb + kchunk - 1, nz);
  const int LRW = RJ + 2, PL = LRW * NTP;
  double *pcr = reinterpret_cast<double *>(smem_raw);             // [RJ][kPcrRow]
  TC *cfs = reinterpret_cast<TC *>(pcr + RJ * kPcrRow);           // [RJ][kRowCoefs]
  TC *ring = cfs + RJ * kRowCoefs;                                // [3 slots][3 arrays][LRW][NTP]
  TC *fb = ring + 9 * PL;                                         // [2][3][RJ][NTP]
  const int j = j0 + tj;
  const bool cell = (ti < nt) && (j <= nr);
  const int jc = (j <= nr) ? j : nr;
  // this row's coefficients, and its reduction ratios, depth and last factors
  if (ti < kRowCoefs) cfs[tj * kRowCoefs + ti] = (TC)rowc[(size_t)jc * kRowCoefs + ti];
  for (int q = ti; q < kPcrRow; q += NTP) pcr[tj * kPcrRow + q] = pcrt[(size_t)jc * kPcrStride + q];
  // plane fetch: element e = tid + l*NTH of the (LRW x NTP) tile, three arrays
  constexpr int NL = 3;
  long goff[NL];
  int lidx[NL];
  bool lval[NL];
#pragma unroll
  for (int l = 0; l < NL; l++) {
    const int e = tid + l * NTH;
    const int r = e / NTP, cc = e - r * NTP;
    const int jj = j0 - 1 + r;
    lidx[l] = (e < PL) ? e : -1;
    lval[l] = (e < PL) && cc < nt && jj <= nr + 2;
    goff[l] = lval[l] ? (long)cc + (long)jj * sj : 0;
  }
  TC pre[3][NL];
  // unconditional loads (masked after) so that a plane's loads issue together
  auto fetch = [&](int kk) {
#pragma unroll
    for (int l = 0; l < NL; l++) {
      const long o = goff[l] + (long)kk * sk;
      const double a1 = q1[o], a2 = q2[o], a3 = q3[o];
      pre[0][l] = lval[l] ? (TC)a1 : (TC)0;
      pre[1][l] = lval[l] ? (TC)a2 : (TC)0;
      pre[2][l] = lval[l] ? (TC)a3 : (TC)0;
    }
  };
  auto stash = [&](int slot) {
#pragma unroll
    for (int l = 0; l < NL; l++)
      if (lidx[l] >= 0) {
        ring[(slot * 3 + 0) * PL + lidx[l]] = pre[0][l];
        ring[(slot * 3 + 1) * PL + lidx[l]] = pre[1][l];
        ring[(slot * 3 + 2) * PL + lidx[l]] = pre[2][l];
      }
  };
  int sM = (kb - 1) % 3, s0 = kb % 3, sP = (kb + 1) % 3;
  fetch(kb - 1); stash(sM);
  fetch(kb); stash(s0);
  fetch(kb + 1);
  // per-row coefficients
  const TC ga = (TC)rk.g, ro = (TC)rk.r, al = (TC)rk.a, dt = (TC)g.dt, aRe = (TC)(rk.a / g.Re);
  const TC dx3 = (TC)g.dx3, dx3q = (TC)g.dx3q;
  const TC *cf = cfs + tj * kRowCoefs;  // per-row metric coefficients (LDS, broadcast reads)
#define h1d11 cf[0]
#define h1d22d cf[1]
#define h1d22n cf[2]
#define h1dare cf[3]
#define h2d11 cf[4]
#define h2d22p cf[5]
#define h2d22m cf[6]
#define h2dare cf[7]
#define s1t11 cf[8]
#define s1t2n cf[9]
#define s1t2s cf[10]
#define s1t2c cf[11]
#define s2t11 cf[12]
#define s2t2p cf[13]
#define s2t2c cf[14]
#define s2t2m cf[15]
#define s3t2n cf[16]
#define s3t2s cf[17]
#define irmn cf[18]
#define irm cf[19]
#define irmm cf[20]
  const int ci = ti, cip = (ti + 1 >= nt) ? 0 : ti + 1, cim = (ti == 0) ? nt - 1 : ti - 1;
  const int rw = tj + 1, rm1 = (jc == 1) ? rw : rw - 1;   // LDS rows of j and jm
  // ru and prg of the next plane stream in while this one is computed
  // (clamped in-bounds addresses for lanes and planes that do not use them)
  const int tic = min(ti, nt - 1);
  TC n_ru[3], n_pg[3];
  // rho = 0 (the first substep): the previous RHS is not needed
  const bool use_ru = rk.r != 0.0;
  auto load_rp = [&](int kk) {
    const int kc = min(kk, ke);
    const long oo = (long)tic + (long)jc * sj + (long)kc * sk;
    const long pp = (long)tic + (long)nt * ((long)(jc - 1) + (long)nr * (long)(kc - 1));
    if (use_ru) { n_ru[0] = ru1[oo]; n_ru[1] = ru2[oo]; n_ru[2] = ru3[oo]; }
    else { n_ru[0] = (TC)0; n_ru[1] = (TC)0; n_ru[2] = (TC)0; }
    n_pg[0] = prg1[pp]; n_pg[1] = prg2[pp]; n_pg[2] = prg3[pp];
  };
  // FP32: one plane ahead; FP64 (register budget): this plane, issued with
  // the ring fetch
  constexpr bool kAhead = sizeof(TC) == 4;
  if (kAhead) load_rp(kb);
  for (int k = kb; k <= ke; k++) {
    stash(sP);
    TC c_ru1 = n_ru[0], c_ru2 = n_ru[1], c_ru3 = n_ru[2];
    TC c_pg1 = n_pg[0], c_pg2 = n_pg[1], c_pg3 = n_pg[2];
    __syncthreads();
    fetch(k + 2);
    if (kAhead) {
      load_rp(k + 1);
    } else {
      load_rp(k);
      c_ru1 = n_ru[0]; c_ru2 = n_ru[1]; c_ru3 = n_ru[2];
      c_pg1 = n_pg[0]; c_pg2 = n_pg[1]; c_pg3 = n_pg[2];
    }
    TC v1 = (TC)0, v2 = (TC)0, v3 = (TC)0;
    const long o = (long)ti + (long)j * sj + (long)k * sk;
    constexpr bool zs = ZS;  // axial mesh: per-plane metric (a separate instantiation)
    const TC zmk = zs ? (TC)zm.m3[k] : dx3, zck = zs ? (TC)zm.c3[k] : dx3;
    if (cell) {
      const TC *A1m = ring + (sM * 3 + 0) * PL, *A1 = ring + (s0 * 3 + 0) * PL, *A1p = ring + (sP * 3 + 0) * PL;
      const TC *A2m = ring + (sM * 3 + 1) * PL, *A2 = ring + (s0 * 3 + 1) * PL, *A2p = ring + (sP * 3 + 1) * PL;
      const TC *A3m = ring + (sM * 3 + 2) * PL, *A3 = ring + (s0 * 3 + 2) * PL, *A3p = ring + (sP * 3 + 2) * PL;
#define L(A, row, col) A[(row) * NTP + (col)]
      const TC q1c = L(A1, rw, ci), q1ip = L(A1, rw, cip), q1im = L(A1, rw, cim);
      const TC q1n = L(A1, rw + 1, ci), q1jm = L(A1, rm1, ci), q1s = L(A1, rw - 1, ci), q1ips = L(A1, rw - 1, cip);
      const TC q1kp = L(A1p, rw, ci), q1km = L(A1m, rw, ci), q1ipkm = L(A1m, rw, cip);
      const TC q2c = L(A2, rw, ci), q2n = L(A2, rw + 1, ci), q2imn = L(A2, rw + 1, cim), q2im = L(A2, rw, cim);
      const TC q2ip = L(A2, rw, cip), q2s = L(A2, rw - 1, ci), q2kp = L(A2p, rw, ci), q2km = L(A2m, rw, ci);
      const TC q2nkm = L(A2m, rw + 1, ci);
      const TC q3c = L(A3, rw, ci), q3kp = L(A3p, rw, ci), q3imkp = L(A3p, rw, cim), q3im = L(A3, rw, cim);
      const TC q3ip = L(A3, rw, cip), q3s = L(A3, rw - 1, ci), q3skp = L(A3p, rw - 1, ci), q3n = L(A3, rw + 1, ci);
      const TC q3jm = L(A3, rm1, ci), q3km = L(A3m, rw, ci);
#undef L
      // ---- q1 at (theta_c, r_m, z_m) ----
      {
        TC qnn = q1ip + q1c, qss = q1im + q1c;
        TC h11 = (qnn * qnn - qss * qss) * h1d11;
        qnn = (q2n + q2imn) * (q1n + q1c);
        qss = (q1c + q1jm) * (q2c + q2im);
        TC h12d = (qnn - qss) * h1d22d;
        qnn = (q1ip + q1c) * (q2n + q2c);
        qss = (q1c + q1im) * (q2imn + q2im);
        TC h12n = (qnn + qss) * h1d22n;
        qnn = (TC)0.25 * (q3kp + q3imkp) * (q1kp + q1c);
        qss = (k == 1) ? (TC)0 : (TC)0.25 * (q3c + q3im) * (q1c + q1km);
        TC h13 = (qnn - qss) * zmk;
        qnn = q2n + q2c;
        qss = q2imn + q2im;
        TC d1q2 = (qnn - qss) * h1dare;
        TC H1 = d1q2 - (h11 + (h12d + h12n) + h13);
        TC d11 = (q1ip - (TC)2 * q1c + q1im) * s1t11;
        TC d33 = zs ? zd2c<TC>(zm, k, q1km, q1c, q1kp)
                    : (k == 1) ? (TC)(4.0 / 3.0) * (q1kp - (TC)3 * q1c) * dx3q : (q1kp - (TC)2 * q1c + q1km) * dx3q;
        TC qn2 = (q1n * irmn - q1c * irm) * s1t2n;
        TC qs2 = (q1c * irm - q1jm * irmm) * s1t2s;
        TC d22 = (qn2 - qs2) * s1t2c;
        v1 = (ga * H1 + ro * c_ru1 - al * c_pg1 + aRe * (d11 + d33 + d22)) * dt;
        ru1[o] = H1;
      }
      // ---- q2 at (theta_m, r_c, z_m), j >= 2 ----
      if (j >= 2) {
        TC qnn = (q1ip + q1ips) * (q2ip + q2c);
        TC qss = (q1c + q1s) * (q2c + q2im);
        TC h21 = (qnn - qss) * h2d11;
        qnn = q2n + q2c;
        qss = q2c + q2s;
        TC h22 = qnn * qnn * h2d22p - qss * qss * h2d22m;
        qnn = (TC)0.5 * (q1c + q1ip);
        qss = (TC)0.5 * (q1s + q1ips);
        TC h11n = (TC)0.25 * (qnn + qss) * (qnn + qss);
        qnn = (TC)0.25 * (q3kp + q3skp) * (q2kp + q2c);
        qss = (k == 1) ? (TC)0 : (TC)0.25 * (q3c + q3s) * (q2c + q2km);
        TC h23 = (qnn - qss) * zmk;
        qnn = q1ip + q1ips;
        qss = q1c + q1s;
        TC d1q1 = -((qnn - qss) * h2dare);
        TC H2 = d1q1 - (h21 + h22 + h23 - h11n);
        TC d11 = (q2ip - (TC)2 * q2c + q2im) * s2t11;
        TC d33 = zs ? zd2c<TC>(zm, k, q2km, q2c, q2kp)
                    : (k == 1) ? (TC)(4.0 / 3.0) * (q2kp - (TC)3 * q2c) * dx3q : (q2kp - (TC)2 * q2c + q2km) * dx3q;
        TC d22 = q2n * s2t2p - q2c * s2t2c + q2s * s2t2m;
        v2 = (ga * H2 + ro * c_ru2 - al * c_pg2 + aRe * (d11 + d33 + d22)) * dt;
        ru2[o] = H2;
      }
      // ---- q3 at (theta_m, r_m, z_c), k >= 2 ----
      if (k >= 2) {
        TC qnn = (q3n + q3c) * (q2n + q2nkm);
        TC qss = (q3jm + q3c) * (q2c + q2km);
        TC h32 = (qnn - qss) * h1d22d;
        qnn = (q3c + q3ip) * (q1ip + q1ipkm);
        qss = (q3im + q3c) * (q1c + q1km);
        TC h31 = (qnn - qss) * h1d11;
        qnn = (TC)0.25 * (q3c + q3kp) * (q3c + q3kp);
        qss = (TC)0.25 * (q3c + q3km) * (q3c + q3km);
        TC h33 = (qnn - qss) * zck;
        TC H3 = -(h31 + h32 + h33);
        TC d11 = (q3ip - (TC)2 * q3c + q3im) * s1t11;
        TC d33 = zs ? zd2f<TC>(zm, k, q3km, q3c, q3kp) : (q3kp - (TC)2 * q3c + q3km) * dx3q;
        TC qn2 = (q3n - q3c) * s3t2n;
        TC qs2 = (q3c - q3jm) * s3t2s;
        TC d22 = qn2 - qs2;
        v3 = (ga * H3 + ro * c_ru3 - al * c_pg3 + aRe * (d11 + d33 + d22)) * dt;
        ru3[o] = H3;
      }
    }
    // ---- periodic theta solves by PCR (ping-pong buffers: one barrier per level) ----
    const long S3 = 3L * RJ * NTP;
    TC *f1 = fb + tj * NTP, *f2 = f1 + RJ * NTP, *f3 = f2 + RJ * NTP;
    f1[ti] = v1; f2[ti] = v2; f3[ti] = v3;
    __syncthreads();
    int sm = 1 % nt;
    const double *pr = pcr + tj * kPcrRow;
    const int mylev = (int)pr[2];
    int blev = 0;  // the block's deepest row (its barriers)
    for (int r = 0; r < RJ; r++) blev = max(blev, (int)pcr[r * kPcrRow + 2]);
    for (int lvl = 0; lvl < blev; ++lvl) {
      const TC al1 = (TC)pr[kPcrHead + 2 * lvl], al2 = (TC)pr[kPcrHead + 2 * lvl + 1];
      TC n1 = v1, n2 = v2, n3 = v3;
      if (ti < nt && lvl < mylev) {
        int imv = ti - sm; if (imv < 0) imv += nt;
        int ipv = ti + sm; if (ipv >= nt) ipv -= nt;
        n1 = v1 + al1 * (f1[imv] + f1[ipv]);
        n2 = v2 + al2 * (f2[imv] + f2[ipv]);
        n3 = v3 + al1 * (f3[imv] + f3[ipv]);
      }
      sm = (2 * sm) % nt;
      const long flip = (lvl & 1) ? -S3 : S3;
      f1 += flip; f2 += flip; f3 += flip;
      f1[ti] = n1; f2[ti] = n2; f3[ti] = n3;
      v1 = n1; v2 = n2; v3 = n3;
      __syncthreads();
    }
    if (cell) {
      const TC d1 = (TC)pr[0], d2 = (TC)pr[1];
      r1[o] = v1 * d1;
      if (j >= 2) r2[o] = v2 * d2;
      if (k >= 2) r3[o] = v3 * d1;
    }
    sM = s0; s0 = sP; sP = (sP == 2) ? 0 : sP + 1;
    __syncthreads();
  }
#undef h1d11
#undef h1d22d
#undef h1d22n
#undef h1dare
#undef h2d11
#undef h2d22p
#undef h2d22m
#undef h2dare
#undef s1t11
#undef s1t2n
#undef s1t2s
#undef s1t2c
#undef s2t11
#undef s2t2p
#undef s2t2c
#undef s2t2m
#undef s3t2n
#undef s3t2s
#undef irmn
#undef irm
#undef irmm
}

// The explicit kernel with one wavefront per r row (nθ <= 64 CPL): each
// lane computes the cells θ = lane + 64 c, and the periodic θ solves run by
// PCR inside the wavefront (LDS exchange ordered by wave-local fences, no
// block barrier per level), which leaves two block barriers per z plane for
// the plane ring.  Same arithmetic as k_explicit_march.
template <typename TW, typename TC, int CPL, int RJT, int WPE, bool ZS>
__global__ __launch_bounds__(64 * RJT, WPE) void k_explicit_wave(VGrid g, const double *__restrict__ rowc, const double *__restrict__ pcrt, VRK rk, ZMet zm, int nlev, int kchunk,
                                                  const double *__restrict__ q1, const double *__restrict__ q2,
                                                  const double *__restrict__ q3, const double *__restrict__ prg1,
                                                  const double *__restrict__ prg2, const double *__restrict__ prg3,
                                                  TW *__restrict__ ru1, TW *__restrict__ ru2, TW *__restrict__ ru3,
                                                  TW *__restrict__ r1, TW *__restrict__ r2, TW *__restrict__ r3) {
  extern __shared__ unsigned char smem_raw[];
  // one wave per r row; lane holds theta cells lane + 64 c, c < CPL
  constexpr int NTP = 64 * CPL, RJ = RJT;
  const int lane = threadIdx.x, tj = threadIdx.y;
  const int NTH = 64 * RJ, tid = tj * 64 + lane;
  const int nt = g.nt, nr = g.nr, nz = g.nz;
  const long sj = g.sj, sk = g.sk;
  int bx, by, bz;
  xcd_block(bx, by, bz);  // r blocks of one z chunk (sharing halo rows) on one XCD
  const int j0 = 1 + bx * RJ;
  const int kb = 1 + by * kchunk, ke = min(kb + kchunk - 1, nz);
  const int LRW = RJ + 2, PL = LRW * NTP;
  const int prow = kPcrHead + 2 * nlev;
  double *pcr = reinterpret_cast<double *>(smem_raw);             // [RJ][prow]
  TC *cfs = reinterpret_cast<TC *>(pcr + RJ * prow);              // [RJ][kRowCoefs]
  TC *ring = cfs + RJ * kRowCoefs;                                // [3 slots][3 arrays][LRW][NTP]
  TC *fb = ring + 9 * PL;                                         // [2][3][RJ][NTP]
  const int j = j0 + tj;
  const int jc = (j <= nr) ? j : nr;
  // this row's coefficients, and its reduction ratios, depth and last factors
  if (lane < kRowCoefs) cfs[tj * kRowCoefs + lane] = (TC)rowc[(size_t)jc * kRowCoefs + lane];
  for (int q = lane; q < prow; q += 64) pcr[tj * prow + q] = pcrt[(size_t)jc * kPcrStride + q];
  // plane fetch: element e = tid + l*NTH of the (LRW x NTP) tile, three arrays
  constexpr int NL = (CPL * (RJT + 2) + RJT - 1) / RJT;  // ceil((RJ + 2) NTP / (64 RJ))
  long goff[NL];
  int lidx[NL];
  bool lval[NL];
#pragma unroll
  for (int l = 0; l < NL; l++) {
    const int e = tid + l * NTH;
    const int r = e / NTP, cc = e - r * NTP;
    const int jj = j0 - 1 + r;
    lidx[l] = (e < PL) ? e : -1;
    lval[l] = (e < PL) && cc < nt && jj <= nr + 2;
    goff[l] = lval[l] ? (long)cc + (long)jj * sj : 0;
  }
  TC pre[3][NL];
  // unconditional loads (masked after) so that a plane's loads issue together
  auto fetch = [&](int kk) {
#pragma unroll
    for (int l = 0; l < NL; l++) {
      const long o = goff[l] + (long)kk * sk;
      const double a1 = q1[o], a2 = q2[o], a3 = q3[o];
      pre[0][l] = lval[l] ? (TC)a1 : (TC)0;
      pre[1][l] = lval[l] ? (TC)a2 : (TC)0;
      pre[2][l] = lval[l] ? (TC)a3 : (TC)0;
    }
  };
  auto stash = [&](int slot) {
#pragma unroll
    for (int l = 0; l < NL; l++)
      if (lidx[l] >= 0) {
        ring[(slot * 3 + 0) * PL + lidx[l]] = pre[0][l];
        ring[(slot * 3 + 1) * PL + lidx[l]] = pre[1][l];
        ring[(slot * 3 + 2) * PL + lidx[l]] = pre[2][l];
      }
  };
  int sM = (kb - 1) % 3, s0 = kb % 3, sP = (kb + 1) % 3;
  fetch(kb - 1); stash(sM);
  fetch(kb); stash(s0);
  fetch(kb + 1);
  // per-row coefficients
  const TC ga = (TC)rk.g, ro = (TC)rk.r, al = (TC)rk.a, dt = (TC)g.dt, aRe = (TC)(rk.a / g.Re);
  const TC dx3 = (TC)g.dx3, dx3q = (TC)g.dx3q;
  const TC *cf = cfs + tj * kRowCoefs;  // per-row metric coefficients (LDS, broadcast reads)
#define h1d11 cf[0]
#define h1d22d cf[1]
#define h1d22n cf[2]
#define h1dare cf[3]
#define h2d11 cf[4]
#define h2d22p cf[5]
#define h2d22m cf[6]
#define h2dare cf[7]
#define s1t11 cf[8]
#define s1t2n cf[9]
#define s1t2s cf[10]
#define s1t2c cf[11]
#define s2t11 cf[12]
#define s2t2p cf[13]
#define s2t2c cf[14]
#define s2t2m cf[15]
#define s3t2n cf[16]
#define s3t2s cf[17]
#define irmn cf[18]
#define irm cf[19]
#define irmm cf[20]
  const int rw = tj + 1, rm1 = (jc == 1) ? rw : rw - 1;   // LDS rows of j and jm
  // ru and prg of the next plane stream in while this one is computed
  // (clamped in-bounds addresses for lanes and planes that do not use them)
  TC n_ru[CPL][3], n_pg[CPL][3];
  // rho = 0 (the first substep): the previous RHS is not needed
  const bool use_ru = rk.r != 0.0;
  auto load_rp = [&](int kk) {
    const int kc = min(kk, ke);
#pragma unroll
    for (int cc = 0; cc < CPL; cc++) {
      const int tic = min(lane + 64 * cc, nt - 1);
      const long oo = (long)tic + (long)jc * sj + (long)kc * sk;
      const long pp = (long)tic + (long)nt * ((long)(jc - 1) + (long)nr * (long)(kc - 1));
      if (use_ru) { n_ru[cc][0] = ru1[oo]; n_ru[cc][1] = ru2[oo]; n_ru[cc][2] = ru3[oo]; }
      else { n_ru[cc][0] = (TC)0; n_ru[cc][1] = (TC)0; n_ru[cc][2] = (TC)0; }
      n_pg[cc][0] = prg1[pp]; n_pg[cc][1] = prg2[pp]; n_pg[cc][2] = prg3[pp];
    }
  };
  auto wave_sync = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  load_rp(kb);
  for (int k = kb; k <= ke; k++) {
    stash(sP);
    TC cru[CPL][3], cpg[CPL][3];
#pragma unroll
    for (int cc = 0; cc < CPL; cc++)
#pragma unroll
      for (int q = 0; q < 3; q++) { cru[cc][q] = n_ru[cc][q]; cpg[cc][q] = n_pg[cc][q]; }
    __syncthreads();
    fetch(k + 2);
    load_rp(k + 1);
    TC w1[CPL], w2[CPL], w3[CPL];
#pragma unroll
    for (int cc = 0; cc < CPL; cc++) {
      const int ti = lane + 64 * cc;
      const int ci = ti, cip = (ti + 1 >= nt) ? 0 : ti + 1, cim = (ti == 0) ? nt - 1 : ti - 1;
      const bool cell = (ti < nt) && (j <= nr);
      const TC c_ru1 = cru[cc][0], c_ru2 = cru[cc][1], c_ru3 = cru[cc][2];
      const TC c_pg1 = cpg[cc][0], c_pg2 = cpg[cc][1], c_pg3 = cpg[cc][2];
      TC v1 = (TC)0, v2 = (TC)0, v3 = (TC)0;
      constexpr bool zs = ZS;  // axial mesh: per-plane metric (a separate instantiation)
      const TC zmk = zs ? (TC)zm.m3[k] : dx3, zck = zs ? (TC)zm.c3[k] : dx3;
      const long o = (long)ti + (long)j * sj + (long)k * sk;
      if (cell) {
      const TC *A1m = ring + (sM * 3 + 0) * PL, *A1 = ring + (s0 * 3 + 0) * PL, *A1p = ring + (sP * 3 + 0) * PL;
      const TC *A2m = ring + (sM * 3 + 1) * PL, *A2 = ring + (s0 * 3 + 1) * PL, *A2p = ring + (sP * 3 + 1) * PL;
      const TC *A3m = ring + (sM * 3 + 2) * PL, *A3 = ring + (s0 * 3 + 2) * PL, *A3p = ring + (sP * 3 + 2) * PL;
#define L(A, row, col) A[(row) * NTP + (col)]
      const TC q1c = L(A1, rw, ci), q1ip = L(A1, rw, cip), q1im = L(A1, rw, cim);
      const TC q1n = L(A1, rw + 1, ci), q1jm = L(A1, rm1, ci), q1s = L(A1, rw - 1, ci), q1ips = L(A1, rw - 1, cip);
      const TC q1kp = L(A1p, rw, ci), q1km = L(A1m, rw, ci), q1ipkm = L(A1m, rw, cip);
      const TC q2c = L(A2, rw, ci), q2n = L(A2, rw + 1, ci), q2imn = L(A2, rw + 1, cim), q2im = L(A2, rw, cim);
      const TC q2ip = L(A2, rw, cip), q2s = L(A2, rw - 1, ci), q2kp = L(A2p, rw, ci), q2km = L(A2m, rw, ci);
      const TC q2nkm = L(A2m, rw + 1, ci);
      const TC q3c = L(A3, rw, ci), q3kp = L(A3p, rw, ci), q3imkp = L(A3p, rw, cim), q3im = L(A3, rw, cim);
      const TC q3ip = L(A3, rw, cip), q3s = L(A3, rw - 1, ci), q3skp = L(A3p, rw - 1, ci), q3n = L(A3, rw + 1, ci);
      const TC q3jm = L(A3, rm1, ci), q3km = L(A3m, rw, ci);
#undef L
      // ---- q1 at (theta_c, r_m, z_m) ----
      {
        TC qnn = q1ip + q1c, qss = q1im + q1c;
        TC h11 = (qnn * qnn - qss * qss) * h1d11;
        qnn = (q2n + q2imn) * (q1n + q1c);
        qss = (q1c + q1jm) * (q2c + q2im);
        TC h12d = (qnn - qss) * h1d22d;
        qnn = (q1ip + q1c) * (q2n + q2c);
        qss = (q1c + q1im) * (q2imn + q2im);
        TC h12n = (qnn + qss) * h1d22n;
        qnn = (TC)0.25 * (q3kp + q3imkp) * (q1kp + q1c);
        qss = (k == 1) ? (TC)0 : (TC)0.25 * (q3c + q3im) * (q1c + q1km);
        TC h13 = (qnn - qss) * zmk;
        qnn = q2n + q2c;
        qss = q2imn + q2im;
        TC d1q2 = (qnn - qss) * h1dare;
        TC H1 = d1q2 - (h11 + (h12d + h12n) + h13);
        TC d11 = (q1ip - (TC)2 * q1c + q1im) * s1t11;
        TC d33 = zs ? zd2c<TC>(zm, k, q1km, q1c, q1kp)
                    : (k == 1) ? (TC)(4.0 / 3.0) * (q1kp - (TC)3 * q1c) * dx3q : (q1kp - (TC)2 * q1c + q1km) * dx3q;
        TC qn2 = (q1n * irmn - q1c * irm) * s1t2n;
        TC qs2 = (q1c * irm - q1jm * irmm) * s1t2s;
        TC d22 = (qn2 - qs2) * s1t2c;
        v1 = (ga * H1 + ro * c_ru1 - al * c_pg1 + aRe * (d11 + d33 + d22)) * dt;
        ru1[o] = H1;
      }
      // ---- q2 at (theta_m, r_c, z_m), j >= 2 ----
      if (j >= 2) {
        TC qnn = (q1ip + q1ips) * (q2ip + q2c);
        TC qss = (q1c + q1s) * (q2c + q2im);
        TC h21 = (qnn - qss) * h2d11;
        qnn = q2n + q2c;
        qss = q2c + q2s;
        TC h22 = qnn * qnn * h2d22p - qss * qss * h2d22m;
        qnn = (TC)0.5 * (q1c + q1ip);
        qss = (TC)0.5 * (q1s + q1ips);
        TC h11n = (TC)0.25 * (qnn + qss) * (qnn + qss);
        qnn = (TC)0.25 * (q3kp + q3skp) * (q2kp + q2c);
        qss = (k == 1) ? (TC)0 : (TC)0.25 * (q3c + q3s) * (q2c + q2km);
        TC h23 = (qnn - qss) * zmk;
        qnn = q1ip + q1ips;
        qss = q1c + q1s;
        TC d1q1 = -((qnn - qss) * h2dare);
        TC H2 = d1q1 - (h21 + h22 + h23 - h11n);
        TC d11 = (q2ip - (TC)2 * q2c + q2im) * s2t11;
        TC d33 = zs ? zd2c<TC>(zm, k, q2km, q2c, q2kp)
                    : (k == 1) ? (TC)(4.0 / 3.0) * (q2kp - (TC)3 * q2c) * dx3q : (q2kp - (TC)2 * q2c + q2km) * dx3q;
        TC d22 = q2n * s2t2p - q2c * s2t2c + q2s * s2t2m;
        v2 = (ga * H2 + ro * c_ru2 - al * c_pg2 + aRe * (d11 + d33 + d22)) * dt;
        ru2[o] = H2;
      }
      // ---- q3 at (theta_m, r_m, z_c), k >= 2 ----
      if (k >= 2) {
        TC qnn = (q3n + q3c) * (q2n + q2nkm);
        TC qss = (q3jm + q3c) * (q2c + q2km);
        TC h32 = (qnn - qss) * h1d22d;
        qnn = (q3c + q3ip) * (q1ip + q1ipkm);
        qss = (q3im + q3c) * (q1c + q1km);
        TC h31 = (qnn - qss) * h1d11;
        qnn = (TC)0.25 * (q3c + q3kp) * (q3c + q3kp);
        qss = (TC)0.25 * (q3c + q3km) * (q3c + q3km);
        TC h33 = (qnn - qss) * zck;
        TC H3 = -(h31 + h32 + h33);
        TC d11 = (q3ip - (TC)2 * q3c + q3im) * s1t11;
        TC d33 = zs ? zd2f<TC>(zm, k, q3km, q3c, q3kp) : (q3kp - (TC)2 * q3c + q3km) * dx3q;
        TC qn2 = (q3n - q3c) * s3t2n;
        TC qs2 = (q3c - q3jm) * s3t2s;
        TC d22 = qn2 - qs2;
        v3 = (ga * H3 + ro * c_ru3 - al * c_pg3 + aRe * (d11 + d33 + d22)) * dt;
        ru3[o] = H3;
      }
          }
      w1[cc] = v1; w2[cc] = v2; w3[cc] = v3;
    }
    // ---- periodic theta solves by PCR within the wavefront ----
    const long S3 = 3L * RJ * NTP;
    TC *f1 = fb + tj * NTP, *f2 = f1 + RJ * NTP, *f3 = f2 + RJ * NTP;
#pragma unroll
    for (int cc = 0; cc < CPL; cc++) {
      const int ti = lane + 64 * cc;
      f1[ti] = w1[cc]; f2[ti] = w2[cc]; f3[ti] = w3[cc];
    }
    wave_sync();
    int sm = 1 % nt;
    const double *pr = pcr + tj * prow;
    const int mylev = __builtin_amdgcn_readfirstlane((int)pr[2]);
    for (int lvl = 0; lvl < mylev; ++lvl) {
      const TC al1 = (TC)pr[kPcrHead + 2 * lvl], al2 = (TC)pr[kPcrHead + 2 * lvl + 1];
      TC n1[CPL], n2[CPL], n3[CPL];
#pragma unroll
      for (int cc = 0; cc < CPL; cc++) {
        const int ti = lane + 64 * cc;
        n1[cc] = w1[cc]; n2[cc] = w2[cc]; n3[cc] = w3[cc];
        if (ti < nt) {
          int imv = ti - sm; if (imv < 0) imv += nt;
          int ipv = ti + sm; if (ipv >= nt) ipv -= nt;
          n1[cc] = w1[cc] + al1 * (f1[imv] + f1[ipv]);
          n2[cc] = w2[cc] + al2 * (f2[imv] + f2[ipv]);
          n3[cc] = w3[cc] + al1 * (f3[imv] + f3[ipv]);
        }
      }
      sm = (2 * sm) % nt;
      const long flip = (lvl & 1) ? -S3 : S3;
      f1 += flip; f2 += flip; f3 += flip;
#pragma unroll
      for (int cc = 0; cc < CPL; cc++) {
        const int ti = lane + 64 * cc;
        f1[ti] = n1[cc]; f2[ti] = n2[cc]; f3[ti] = n3[cc];
        w1[cc] = n1[cc]; w2[cc] = n2[cc]; w3[cc] = n3[cc];
      }
      wave_sync();
    }
    const TC d1 = (TC)pr[0], d2 = (TC)pr[1];
#pragma unroll
    for (int cc = 0; cc < CPL; cc++) {
      const int ti = lane + 64 * cc;
      if (ti < nt && j <= nr) {
        const long o = (long)ti + (long)j * sj + (long)k * sk;
        r1[o] = w1[cc] * d1;
        if (j >= 2) r2[o] = w2[cc] * d2;
        if (k >= 2) r3[o] = w3[cc] * d1;
      }
    }
    sM = s0; s0 = sP; sP = (sP == 2) ? 0 : sP + 1;
    __syncthreads();
  }
#undef h1d11
#undef h1d22d
#undef h1d22n
#undef h1dare
#undef h2d11
#undef h2d22p
#undef h2d22m
#undef h2dare
#undef s1t11
#undef s1t2n
#undef s1t2s
#undef s1t2c
#undef s2t11
#undef s2t2p
#undef s2t2c
#undef s2t2m
#undef s3t2n
#undef s3t2s
#undef irmn
#undef irm
#undef irmm
}

// Variant with one z plane per block (no z marching): every stencil operand
// is read through L1/L2.  Fewer registers and LDS than the marching form;
// the autotuner picks whichever is faster for the precision and grid.
// ROWW = 32, 64: rows of that many lanes, solved within the wavefront (no
// block barrier); 0: rows of several wavefronts.  The divisions by rm and by the
// last diagonal keep a quotient's accuracy (quot below): up to 1 % of the time (rows
// of 32 lanes, four waves a SIMD: 15.0 -> 16.0 us at 32x64x128, 64x96x256 45.9).
template <typename TW, typename TC, bool ZS, int ROWW>
__global__ __launch_bounds__(512, ROWW == 32 ? 4 : 1) void k_explicit_cell(VGrid g, const double *__restrict__ rowc,
                                                   const double *__restrict__ pcrt, VRK rk, ZMet zm,
                                                   const double *__restrict__ q1, const double *__restrict__ q2,
                                                   const double *__restrict__ q3, const double *__restrict__ prg1,
                                                   const double *__restrict__ prg2, const double *__restrict__ prg3,
                                                   TW *__restrict__ ru1, TW *__restrict__ ru2, TW *__restrict__ ru3,
                                                   TW *__restrict__ r1, TW *__restrict__ r2, TW *__restrict__ r3) {
  extern __shared__ unsigned char smem_raw[];
  const int NTP = blockDim.x, RJ = blockDim.y, ti = threadIdx.x, tj = threadIdx.y;
  const int i = ti + 1;
  int bx, by, bz;
  xcd_block(bx, by, bz);  // r blocks of one plane (sharing halo rows) on one XCD
  const int j = bx * RJ + tj + 1;
  const int k = by + 1;
  const bool cell = (i <= g.nt) && (j <= g.nr);
  // the row's tables; a row of whole wavefronts is uniform in each of them
  int jc = min(j, g.nr);
  if (ROWW != 32) jc = __builtin_amdgcn_readfirstlane(jc);
  // x / d from the rounded inverse of d, with one correction by the remainder
  // (Markstein): the quotient's own rounding in all but a few cases, where the
  // bare product has the inverse's on top
  auto quot = [](TC x, TC inv, TC d) {
    auto fma_t = [](TC a, TC b, TC c) {
      if constexpr (sizeof(TC) == 4) return __builtin_fmaf(a, b, c); else return __builtin_fma(a, b, c);
    };
    const TC q = x * inv;
    return fma_t(fma_t(-q, d, x), inv, q);
  };
  const double *cf = rowc + (size_t)jc * kRowCoefs, *pr = pcrt + (size_t)jc * kPcrStride;
  TC v1 = (TC)0, v2 = (TC)0, v3 = (TC)0;
  if (cell) {
  const int ip = (i == g.nt) ? 1 : i + 1, im = (i == 1) ? g.nt : i - 1;
  const int jm = (j == 1) ? 1 : j - 1;
  const long o = hidx(g, i, j, k);
  const long dip = ip - i, dim = im - i, sj = g.sj, sk = g.sk, djm = (long)(jm - j) * sj;
  const TC ga = (TC)rk.g, ro = (TC)rk.r, al = (TC)rk.a, dt = (TC)g.dt, aRe = (TC)(rk.a / g.Re);
  const bool use_ru = rk.r != 0.0;  // rho = 0 (the first substep): the previous RHS is not needed
  const TC dx3 = (TC)g.dx3, dx3q = (TC)g.dx3q;
  constexpr bool zs = ZS;  // axial mesh: per-plane metric (a separate instantiation)
  const TC zmk = zs ? (TC)zm.m3[k] : dx3, zck = zs ? (TC)zm.c3[k] : dx3;
  const long pc = cidx(g, i, j, k);
#define Q1(d) ((TC)q1[o + (d)])
#define Q2(d) ((TC)q2[o + (d)])
#define Q3(d) ((TC)q3[o + (d)])
  // ---- q1 at (theta_c, r_m, z_m) ----
  {
    TC qnn = Q1(dip) + Q1(0), qss = Q1(dim) + Q1(0);
    TC h11 = (qnn * qnn - qss * qss) * (TC)cf[0];
    qnn = (Q2(sj) + Q2(dim + sj)) * (Q1(sj) + Q1(0));
    qss = (Q1(0) + Q1(djm)) * (Q2(0) + Q2(dim));
    TC h12d = (qnn - qss) * (TC)cf[1];
    qnn = (Q1(dip) + Q1(0)) * (Q2(sj) + Q2(0));
    qss = (Q1(0) + Q1(dim)) * (Q2(dim + sj) + Q2(dim));
    TC h12n = (qnn + qss) * (TC)cf[2];
    qnn = (TC)0.25 * (Q3(sk) + Q3(dim + sk)) * (Q1(sk) + Q1(0));
    qss = (k == 1) ? (TC)0 : (TC)0.25 * (Q3(0) + Q3(dim)) * (Q1(0) + Q1(-sk));
    TC h13 = (qnn - qss) * zmk;
    qnn = Q2(sj) + Q2(0);
    qss = Q2(dim + sj) + Q2(dim);
    TC d1q2 = (qnn - qss) * (TC)cf[3];
    TC H1 = d1q2 - (h11 + (h12d + h12n) + h13);
    TC d11 = (Q1(dip) - (TC)2 * Q1(0) + Q1(dim)) * (TC)cf[8];
    TC d33 = zs ? zd2c<TC>(zm, k, Q1(-sk), Q1(0), Q1(sk))
                : (k == 1) ? (TC)(4.0 / 3.0) * (Q1(sk) - (TC)3 * Q1(0)) * dx3q
                           : (Q1(sk) - (TC)2 * Q1(0) + Q1(-sk)) * dx3q;
    const TC w0 = quot(Q1(0), (TC)cf[19], (TC)cf[22]);
    TC qn2 = (quot(Q1(sj), (TC)cf[18], (TC)cf[21]) - w0) * (TC)cf[9];
    TC qs2 = (w0 - quot(Q1(djm), (TC)cf[20], (TC)cf[23])) * (TC)cf[10];
    TC d22 = (qn2 - qs2) * (TC)cf[11];
    v1 = (ga * H1 + ro * (use_ru ? ru1[o] : (TC)0) - al * prg1[pc] + aRe * (d11 + d33 + d22)) * dt;
    ru1[o] = H1;
  }
  // ---- q2 at (theta_m, r_c, z_m), j >= 2 ----
  if (j >= 2) {
    TC qnn = (Q1(dip) + Q1(dip - sj)) * (Q2(dip) + Q2(0));
    TC qss = (Q1(0) + Q1(-sj)) * (Q2(0) + Q2(dim));
    TC h21 = (qnn - qss) * (TC)cf[4];
    qnn = Q2(sj) + Q2(0);
    qss = Q2(0) + Q2(-sj);
    TC h22 = qnn * qnn * (TC)cf[5] - qss * qss * (TC)cf[6];
    qnn = (TC)0.5 * (Q1(0) + Q1(dip));
    qss = (TC)0.5 * (Q1(-sj) + Q1(dip - sj));
    TC h11n = (TC)0.25 * (qnn + qss) * (qnn + qss);
    qnn = (TC)0.25 * (Q3(sk) + Q3(sk - sj)) * (Q2(sk) + Q2(0));
    qss = (k == 1) ? (TC)0 : (TC)0.25 * (Q3(0) + Q3(-sj)) * (Q2(0) + Q2(-sk));
    TC h23 = (qnn - qss) * zmk;
    qnn = Q1(dip) + Q1(dip - sj);
    qss = Q1(0) + Q1(-sj);
    TC d1q1 = -((qnn - qss) * (TC)cf[7]);
    TC H2 = d1q1 - (h21 + h22 + h23 - h11n);
    TC d11 = (Q2(dip) - (TC)2 * Q2(0) + Q2(dim)) * (TC)cf[12];
    TC d33 = zs ? zd2c<TC>(zm, k, Q2(-sk), Q2(0), Q2(sk))
                : (k == 1) ? (TC)(4.0 / 3.0) * (Q2(sk) - (TC)3 * Q2(0)) * dx3q
                           : (Q2(sk) - (TC)2 * Q2(0) + Q2(-sk)) * dx3q;
    TC d22 = Q2(sj) * (TC)cf[13] - Q2(0) * (TC)cf[14] + Q2(-sj) * (TC)cf[15];
    v2 = (ga * H2 + ro * (use_ru ? ru2[o] : (TC)0) - al * prg2[pc] + aRe * (d11 + d33 + d22)) * dt;
    ru2[o] = H2;
  }
  // ---- q3 at (theta_m, r_m, z_c), k >= 2 ----
  if (k >= 2) {
    TC qnn = (Q3(sj) + Q3(0)) * (Q2(sj) + Q2(sj - sk));
    TC qss = (Q3(djm) + Q3(0)) * (Q2(0) + Q2(-sk));
    TC h32 = (qnn - qss) * (TC)cf[1];
    qnn = (Q3(0) + Q3(dip)) * (Q1(dip) + Q1(dip - sk));
    qss = (Q3(dim) + Q3(0)) * (Q1(0) + Q1(-sk));
    TC h31 = (qnn - qss) * (TC)cf[0];
    qnn = (TC)0.25 * (Q3(0) + Q3(sk)) * (Q3(0) + Q3(sk));
    qss = (TC)0.25 * (Q3(0) + Q3(-sk)) * (Q3(0) + Q3(-sk));
    TC h33 = (qnn - qss) * zck;
    TC H3 = -(h31 + h32 + h33);
    TC d11 = (Q3(dip) - (TC)2 * Q3(0) + Q3(dim)) * (TC)cf[8];
    TC d33 = zs ? zd2f<TC>(zm, k, Q3(-sk), Q3(0), Q3(sk)) : (Q3(sk) - (TC)2 * Q3(0) + Q3(-sk)) * dx3q;
    TC qn2 = (Q3(sj) - Q3(0)) * (TC)cf[16];
    TC qs2 = (Q3(0) - Q3(djm)) * (TC)cf[17];
    TC d22 = qn2 - qs2;
    v3 = (ga * H3 + ro * (use_ru ? ru3[o] : (TC)0) - al * prg3[pc] + aRe * (d11 + d33 + d22)) * dt;
    ru3[o] = H3;
  }
#undef Q1
#undef Q2
#undef Q3
  }
  // ---- periodic theta solves of the three components (solqi/tripij,
  // step.F90:212-263, 487-534): constant coefficients (-acc, 1+2acc, -acc)
  // per line, parallel cyclic reduction on the LDS-resident lines ----
  TC *f1 = reinterpret_cast<TC *>(smem_raw) + (size_t)tj * NTP;
  TC *f2 = f1 + (size_t)RJ * NTP;
  TC *f3 = f2 + (size_t)RJ * NTP;
  f1[ti] = v1; f2[ti] = v2; f3[ti] = v3;
  const int N = g.nt, mylev = (int)pr[2];
  int blev = mylev;  // the depth that the lanes which meet at the syncs share
  if (ROWW == 0) {
    for (int r = 0; r < RJ; r++) blev = max(blev, (int)pcrt[(size_t)min(bx * RJ + r + 1, g.nr) * kPcrStride + 2]);
  } else if (ROWW == 32) {
    blev = max(mylev, __shfl_xor(mylev, 32));
  }
  auto sync = [&]() {
    if (ROWW == 0) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  };
  sync();
  // ping-pong buffers: one sync per reduction level
  const long S3 = 3L * RJ * NTP;
  int sm = 1 % N;
  for (int lvl = 0; lvl < blev; ++lvl) {
    TC n1 = v1, n2 = v2, n3 = v3;
    if (ti < N && lvl < mylev) {
      const TC al1 = (TC)pr[kPcrHead + 2 * lvl], al2 = (TC)pr[kPcrHead + 2 * lvl + 1];
      int imv = ti - sm; if (imv < 0) imv += N;
      int ipv = ti + sm; if (ipv >= N) ipv -= N;
      n1 = v1 + al1 * (f1[imv] + f1[ipv]);
      n2 = v2 + al2 * (f2[imv] + f2[ipv]);
      n3 = v3 + al1 * (f3[imv] + f3[ipv]);
    }
    sm = (2 * sm) % N;
    const long flip = (lvl & 1) ? -S3 : S3;
    f1 += flip; f2 += flip; f3 += flip;
    f1[ti] = n1; f2[ti] = n2; f3[ti] = n3;
    v1 = n1; v2 = n2; v3 = n3;
    sync();
  }
  if (!cell) return;
  const TC d1 = (TC)pr[0], d2 = (TC)pr[1], b1 = (TC)pr[kPcrRow], b2 = (TC)pr[kPcrRow + 1];
  const long o = hidx(g, i, j, k);
  r1[o] = quot(v1, d1, b1);
  if (j >= 2) r2[o] = quot(v2, d2, b2);
  if (k >= 2) r3[o] = quot(v3, d1, b1);
}

// ---------------------------------------------------------------------------
// Poisson solve (poisson_solve.F90:140-179) in five passes: divergence +
// theta FFT, z DCT-II, radial Thomas, z DCT-III, inverse theta FFT.
// ---------------------------------------------------------------------------

// complex multiply (x + iy)(c + is)
template <typename T> __device__ __forceinline__ void cmul(T &x, T &y, T c, T s) {
  const T t = x * c - y * s;
  y = x * s + y * c;
  x = t;
}
// in-register DFT of R = 2, 4 or 8 points, v_s = sum_r v_r e^{i sign 2 pi r s / R}
template <typename T> __device__ __forceinline__ void dft2(T &ar, T &ai, T &br, T &bi) {
  const T tr = ar - br, ti = ai - bi;
  ar = ar + br; ai = ai + bi;
  br = tr; bi = ti;
}
template <typename T> __device__ __forceinline__ void dft4(T *vr, T *vi, int st, T sign) {
  // inputs at 0, st, 2 st, 3 st
  T t0r = vr[0], t0i = vi[0], t1r = vr[2 * st], t1i = vi[2 * st];
  dft2(t0r, t0i, t1r, t1i);  // t0 = v0 + v2, t1 = v0 - v2
  T t2r = vr[st], t2i = vi[st], t3r = vr[3 * st], t3i = vi[3 * st];
  dft2(t2r, t2i, t3r, t3i);  // t2 = v1 + v3, t3 = v1 - v3
  // t3 *= (i sign)
  const T u = t3r;
  t3r = -sign * t3i;
  t3i = sign * u;
  vr[0] = t0r + t2r; vi[0] = t0i + t2i;
  vr[2 * st] = t0r - t2r; vi[2 * st] = t0i - t2i;
  vr[st] = t1r + t3r; vi[st] = t1i + t3i;
  vr[3 * st] = t1r - t3r; vi[3 * st] = t1i - t3i;
}
template <typename T> __device__ __forceinline__ void dft8(T *vr, T *vi, T sign) {
  // even points 0,2,4,6 and odd points 1,3,5,7: two 4-point DFTs in place
  dft4(vr, vi, 2, sign);
  dft4(vr + 1, vi + 1, 2, sign);
  const T h = (T)0.70710678118654752440;
  // odd outputs s = 0..3 sit at 1,3,5,7: multiply by w8^s
  cmul(vr[3], vi[3], h, sign * h);
  { const T u = vr[5]; vr[5] = -sign * vi[5]; vi[5] = sign * u; }
  cmul(vr[7], vi[7], -h, sign * h);
  T er[4] = {vr[0], vr[2], vr[4], vr[6]}, ei[4] = {vi[0], vi[2], vi[4], vi[6]};
  T orr[4] = {vr[1], vr[3], vr[5], vr[7]}, oi[4] = {vi[1], vi[3], vi[5], vi[7]};
  for (int q = 0; q < 4; q++) {
    vr[q] = er[q] + orr[q]; vi[q] = ei[q] + oi[q];
    vr[q + 4] = er[q] - orr[q]; vi[q + 4] = ei[q] - oi[q];
  }
}

// radix of pass with `bits` bits still to do: 8 while the rest stays a
// multiple of 3, else 4 (2 for a lone bit)
__host__ __device__ constexpr int fft_pass_bits(int bits) {
  if (bits % 3 == 0) return 3;
  return bits == 1 ? 1 : 2;
}
__host__ inline int fft_min_radix(int logn) {
  int bits = logn, m = 8;
  while (bits > 0) { const int lr = fft_pass_bits(bits); m = m < (1 << lr) ? m : (1 << lr); bits -= lr; }
  return m;
}

// butterflies each thread holds across the barrier of an FFT pass (one: the
// register budget keeps five or more waves per SIMD in both precisions)
template <typename T> constexpr int fft_qt() { return 1; }

// One radix-2^LR pass of the Stockham autosort FFT (ls bits already done):
// every butterfly reads its R inputs at stride n/R, applies the twiddles,
// and after the barrier writes the in-register DFT at stride 2^ls.  The
// length and pass (logn, ls) come either from template arguments (CL > 0:
// logn = CL, ls = CS; the LDS offsets r << lg then fold into immediates) or
// from the run-time arguments (CL = 0).
template <typename T, int LR, int QT, int CL = 0, int CS = 0>
__device__ __forceinline__ void fft_pass(T *re, T *im, int nfft, int logn_rt, int sstr, int ls_rt, const T *twr,
                                         const T *twi, T sign, int tid, int nth) {
  constexpr int R = 1 << LR;
  const int logn = CL > 0 ? CL : logn_rt, ls = CL > 0 ? CS : ls_rt;
  const int nh = 1 << (logn - 1), lg = logn - LR;
  const int tasks = nfft << lg;
  T vr[QT][R], vi[QT][R];
#pragma unroll
  for (int q = 0; q < QT; q++) {
    const int t = tid + q * nth;
    if (t < tasks) {
      const int f = t >> lg, j = t & ((1 << lg) - 1), k = j & ((1 << ls) - 1);
      const T *br = re + f * sstr, *bi = im + f * sstr;
#pragma unroll
      for (int r = 0; r < R; r++) {
        T x = br[j + (r << lg)], y = bi[j + (r << lg)];
        if (r > 0 && k > 0) {
          const int idx = (r * k) << (logn - ls - LR);
          T c, sn;
          if (idx < nh) { c = twr[idx]; sn = twi[idx]; }
          else { c = -twr[idx - nh]; sn = -twi[idx - nh]; }
          cmul(x, y, c, sign * sn);
        }
        vr[q][r] = x; vi[q][r] = y;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < QT; q++) {
    const int t = tid + q * nth;
    if (t < tasks) {
      const int f = t >> lg, j = t & ((1 << lg) - 1), k = j & ((1 << ls) - 1);
      if (LR == 3) dft8(vr[q], vi[q], sign);
      else if (LR == 2) dft4(vr[q], vi[q], 1, sign);
      else dft2(vr[q][0], vi[q][0], vr[q][1], vi[q][1]);
      const int d = ((j >> ls) << (ls + LR)) + k;
      T *br = re + f * sstr, *bi = im + f * sstr;
#pragma unroll
      for (int r = 0; r < R; r++) { br[d + (r << ls)] = vr[q][r]; bi[d + (r << ls)] = vi[q][r]; }
    }
  }
  __syncthreads();
}

// the passes of a transform of compile-time length 2^CL from pass CS on
template <typename T, int QT, int CL, int CS>
__device__ __forceinline__ void lds_fft_c(T *re, T *im, int nfft, int sstr, const T *twr, const T *twi, T sign,
                                          int tid, int nth) {
  if constexpr (CS < CL) {
    constexpr int LR = fft_pass_bits(CL - CS);
    fft_pass<T, LR, QT, CL, CS>(re, im, nfft, CL, sstr, CS, twr, twi, sign, tid, nth);
    lds_fft_c<T, QT, CL, CS + LR>(re, im, nfft, sstr, twr, twi, sign, tid, nth);
  }
}

// In-place Stockham autosort FFT of nfft sequences of length n = 2^logn in
// LDS (re, im; sequence f starts at f * sstr), natural order in and out,
// radix-8/4/2 passes with the DFT in
// registers.  Twiddles w_p = (twr[p], sign twi[p]), p < n/2, from LDS (the
// upper half by symmetry).  Each thread holds at most fft_qt<T>() butterflies
// of a pass across the barrier that separates the reads from the writes; the
// caller keeps nfft n / (min radix) <= fft_qt<T>() nth.
template <typename T>
__device__ __forceinline__ void lds_fft(T *re, T *im, int nfft, int logn, int sstr, const T *twr, const T *twi, T sign,
                                        int tid, int nth) {
  constexpr int QT = fft_qt<T>();
  // the lengths of the workloads' theta and z transforms: passes with
  // compile-time geometry
  switch (logn) {
    case 5: lds_fft_c<T, QT, 5, 0>(re, im, nfft, sstr, twr, twi, sign, tid, nth); return;
    case 6: lds_fft_c<T, QT, 6, 0>(re, im, nfft, sstr, twr, twi, sign, tid, nth); return;
    case 7: lds_fft_c<T, QT, 7, 0>(re, im, nfft, sstr, twr, twi, sign, tid, nth); return;
    case 8: lds_fft_c<T, QT, 8, 0>(re, im, nfft, sstr, twr, twi, sign, tid, nth); return;
    case 9: lds_fft_c<T, QT, 9, 0>(re, im, nfft, sstr, twr, twi, sign, tid, nth); return;
    case 10: lds_fft_c<T, QT, 10, 0>(re, im, nfft, sstr, twr, twi, sign, tid, nth); return;
    default: break;
  }
  int ls = 0;
  while (ls < logn) {
    const int lr = fft_pass_bits(logn - ls);
    if (lr == 3) fft_pass<T, 3, QT>(re, im, nfft, logn, sstr, ls, twr, twi, sign, tid, nth);
    else if (lr == 2) fft_pass<T, 2, QT>(re, im, nfft, logn, sstr, ls, twr, twi, sign, tid, nth);
    else fft_pass<T, 1, QT>(re, im, nfft, logn, sstr, ls, twr, twi, sign, tid, nth);
    ls += lr;
  }
}

// byte offset rounded up to 16
__host__ __device__ constexpr size_t al16(size_t b) { return (b + 15) & ~(size_t)15; }

// divq (divergence.F90:31-41) + fft_ptf_multi packing
// (fastfouriertransform.F90:39-43) for LB theta lines per block, ntheta a
// power of two: two real lines per complex FFT in LDS (other ntheta: k_divdft).
// In mixed mode the packed positions 0..4 (m = 0,1,2) are also produced in
// double from the double divergence into S64 (layout (5, nr, nz)).
template <typename TW, bool SPLIT>
__global__ __launch_bounds__(256) void k_divfft(VGrid g, VCoef c, ZMet zm, double inv_adt, const double *__restrict__ dq1,
                                                const double *__restrict__ dq2, const double *__restrict__ dq3,
                                                const double *__restrict__ ext, TW *__restrict__ S,
                                                double *__restrict__ S64, const double *__restrict__ twr,
                                                const double *__restrict__ twi, int LB, int logn) {
  extern __shared__ unsigned char smem_raw[];
  const int N = g.nt, tid = threadIdx.x, nth = blockDim.x;
  const long nlines = (long)g.nr * g.nz;
  const long l0 = (long)blockIdx.x * LB;
  // LDS: re, im ((LB/2)*N TW each) | [tw (2N double), part (10 LB double)] |
  // twl (N TW) | jk (2 LB int) | 1/rm, dx2/dmr (LB double each).  The FP64
  // low modes of the mixed path are summed in registers.
  TW *re = reinterpret_cast<TW *>(smem_raw);
  TW *im = re + (size_t)(LB / 2) * N;
  size_t off = al16(sizeof(TW) * LB * N);
  double *tw = reinterpret_cast<double *>(smem_raw + off);     // cos (N) then sin (N), S64 only
  double *part = tw + 2 * (size_t)N;                           // (line, coefficient, 2 waves), S64 only
  if (S64) off = al16(off + sizeof(double) * (2 * (size_t)N + 10 * (size_t)LB));
  TW *twl = reinterpret_cast<TW *>(smem_raw + off);            // FFT twiddles: N/2 cos, N/2 sin
  off = al16(off + sizeof(TW) * N);
  int *jk = reinterpret_cast<int *>(smem_raw + off);           // (j, k) of each line
  // 1/rm(j) and dx2/dmr(j) of each line: divq's theta and r differences
  // (divergence.F90:38-39) share the 1/rm factor, so a cell needs no division
  double *lirm = reinterpret_cast<double *>(smem_raw + al16(off + sizeof(int) * 2 * LB));
  double *lcx2 = lirm + LB;
  if (tid < LB) {  // lines past the end are clamped to the last line (never stored)
    const long l = min(l0 + tid, nlines - 1);
    const int j = (int)(l % g.nr) + 1;
    jk[2 * tid] = j;
    jk[2 * tid + 1] = (int)(l / g.nr) + 1;
    lirm[tid] = 1.0 / c.rm[j];
    lcx2[tid] = g.dx2 / c.dmr[j];
  }
  for (int q = tid; q < N / 2; q += nth) { twl[q] = (TW)twr[q]; twl[N / 2 + q] = (TW)twi[q]; }
  if (S64)
    for (int q = tid; q < N; q += nth) { tw[q] = twr[q]; tw[N + q] = twi[q]; }
  __syncthreads();
  // TPL threads per line: thread tl of line lpt takes the angles tl,
  // tl + TPL, ... (consecutive lanes read consecutive angles), so its FP64
  // low-mode sums (mixed path) stay within one line
  const int TPL = nth / LB, lpt = tid / TPL, tl = tid - lpt * TPL;
  const int NU = (N + TPL - 1) / TPL;
  const bool lvalid = l0 + lpt < nlines;
  // partial sums of the FP64 low modes: with SPLIT a thread keeps those of its
  // even and odd angles apart (see launch_poisson)
  double sm[SPLIT ? 2 : 1][5] = {};
  auto put = [&](int ii, int u, double val) {
    const int pos = (lpt >> 1) * N + ii;
    if (lpt & 1) im[pos] = (TW)val; else re[pos] = (TW)val;
    if (S64) {  // cos and sin sums of wavenumbers 0, 1, 2
      int q2 = 2 * ii;
      if (q2 >= N) q2 -= N;
      double *s = sm[SPLIT ? u & 1 : 0];
      s[0] += val;
      s[1] += val * tw[ii];
      s[2] += val * tw[N + ii];
      s[3] += val * tw[q2];
      s[4] += val * tw[N + q2];
    }
  };
  const int jl = jk[2 * lpt], kl = jk[2 * lpt + 1];
  if (ext) {
    for (int u = 0; u < NU; ++u) {
      const int ii = tl + TPL * u;
      if (ii < N) put(ii, u, lvalid ? ext[cidx(g, ii + 1, jl, kl)] : 0.0);
    }
  } else {
    // the loads of U angles are all issued before the first is used;
    // indices are clamped to valid cells, so the loads are unconditional
    constexpr int U = 4;
    const double rmv = lirm[lpt], rdv = lcx2[lpt];
    const double zkv = zm.m3 ? zm.m3[kl] : g.dx3;  // dx3, or the axial mesh's 1/width of plane kl
    const long ob = hidx(g, 1, jl, kl);
    for (int ub = 0; ub < NU; ub += U) {
      double a1[U], b1[U], a2[U], b2[U], a3[U], b3[U];
      #pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = min(tl + TPL * (ub + u), N - 1) + 1;
        const long o = ob + (i - 1);
        a1[u] = dq1[o];
        b1[u] = dq1[o + ((i == N) ? 1 - N : 1)];
        a2[u] = dq2[o];
        b2[u] = dq2[o + g.sj];
        a3[u] = dq3[o];
        b3[u] = dq3[o + g.sk];
      }
      __builtin_amdgcn_sched_barrier(0);
      #pragma unroll
      for (int u = 0; u < U; ++u) {
        const int ii = tl + TPL * (ub + u);
        if (ii < N) {
          const double rhs = divq_rhs(b1[u] - a1[u], g.dx1 * g.axsym, b2[u] - a2[u], rdv, rmv, b3[u] - a3[u], zkv, inv_adt);
          put(ii, u, lvalid ? rhs : 0.0);  // ub is a multiple of U: u has the parity of ub + u
        }
      }
    }
  }
  if (S64) {
    // the line's TPL lanes: a fixed butterfly within each wave (deterministic
    // order), then one partial per wave into LDS
    const int grp = TPL < 64 ? TPL : 64;
    if (SPLIT)
#pragma unroll
      for (int w = 0; w < 5; w++) sm[0][w] += sm[SPLIT ? 1 : 0][w];
    for (int o = grp >> 1; o > 0; o >>= 1)
#pragma unroll
      for (int w = 0; w < 5; w++) sm[0][w] += __shfl_xor(sm[0][w], o, grp);
    if ((tl & (grp - 1)) == 0) {
      double *pp = part + (size_t)lpt * 10 + tl / grp;
#pragma unroll
      for (int w = 0; w < 5; w++) pp[2 * w] = sm[0][w];
    }
  }
  __syncthreads();
  lds_fft(re, im, LB / 2, logn, N, twl, twl + N / 2, (TW)-1, tid, nth);
  // a power-of-two N scales exactly, so x * (1/N) is x / N bit for bit
  // without a double division per element
  const double inv_n = 1.0 / N;
  for (int e = tid; e < LB * N; e += nth) {
    const int lp = e >> logn, pos = e - lp * N;
    const long l = l0 + lp;
    if (l >= nlines) continue;
    const int k = (pos + 1) >> 1;  // wavenumber of this packed position
    double Fr, Fi;
    const int q = lp >> 1, kr = (N - k) & (N - 1);
    const double zr = re[q * N + k], zi = im[q * N + k], wr = re[q * N + kr], wi = im[q * N + kr];
    if ((lp & 1) == 0) { Fr = 0.5 * (zr + wr); Fi = 0.5 * (zi - wi); }
    else { Fr = 0.5 * (zi + wi); Fi = -0.5 * (zr - wr); }
    const double num = (pos == 0) ? Fr : (pos & 1) ? 2.0 * Fr : -2.0 * Fi;
    S[(size_t)pos + (size_t)N * l] = (TW)(num * inv_n);
  }
  if (S64) {
    // FP64 modes m = 0, 1, 2 (t(1), t(2k), t(2k+1) packing) from the wave
    // partials, summed in wave order
    const int nw = TPL > 64 ? TPL / 64 : 1;
    for (int e = tid; e < LB * 5; e += nth) {
      const int lp = e / 5, c5 = e - lp * 5;
      const long l = l0 + lp;
      if (l >= nlines || c5 >= N) continue;
      double acc = part[(size_t)e * 2];
      for (int w = 1; w < nw; ++w) acc += part[(size_t)e * 2 + w];
      S64[(size_t)c5 + 5 * l] = (c5 == 0) ? acc / N : 2.0 * acc / N;
    }
  }
}

// z DCT-II (REDFT10, then /(2nz): fastfouriertransform.F90:299-332) of TL
// lines per block, nz a power of two (other nz: k_zdense); lines are contiguous in memory (line stride 1, position
// stride nl).  Makhoul's reordering turns each pair of real lines into one
// complex FFT of length nz.  dir=+1 forward, -1 inverse (REDFT01).
// FP32: at most 64 VGPRs, so that two 1024-lane blocks share a CU, one
// loading while the other transforms (us forward/inverse, without and with:
// 256x512x1024 758/749, 482/456; 128x256x512 54/49, 50/48).
template <typename TW>
__device__ __forceinline__ void dctz_block(unsigned blk, unsigned nblk, TW *__restrict__ S, long nl, int n, int logn, int TL,
                                           int logtl, int dir, const double *__restrict__ twr,
                                           const double *__restrict__ twi, const double *__restrict__ er,
                                           const double *__restrict__ ei) {
  extern __shared__ unsigned char smem_raw[];
  TW *re = reinterpret_cast<TW *>(smem_raw);
  // sequences at stride n + 1 in LDS: the line-to-sequence transposes
  // below touch consecutive sequences from consecutive lanes, which would
  // all hit one bank at stride n
  const int sn = n + 1;
  TW *im = re + (size_t)(TL / 2) * sn;
  TW *twl = im + (size_t)(TL / 2) * sn;  // n/2 cos, n/2 sin
  // Makhoul post/pre-twiddles e^{i pi k/2n}: in FP32 an LDS copy (n cos,
  // n sin) spares the per-element global loads; FP64 reads them from global
  // memory (the LDS would cost the tile lines)
  constexpr bool lds_tw = sizeof(TW) == 4;
  TW *etw = twl + n;
  auto ecos = [&](int k) { return lds_tw ? etw[k] : (TW)er[k]; };
  auto esin = [&](int k) { return lds_tw ? etw[n + k] : (TW)ei[k]; };
  const int tid = threadIdx.x, nth = blockDim.x;
  const long l0 = xcd_tile(blk, nblk) * TL;
  for (int q = tid; q < n / 2; q += nth) { twl[q] = (TW)twr[q]; twl[n / 2 + q] = (TW)twi[q]; }
  if (lds_tw)
    for (int q = tid; q < n; q += nth) { etw[q] = (TW)er[q]; etw[n + q] = (TW)ei[q]; }
  // Element u of a thread is line lp = tid mod TL (consecutive lanes,
  // consecutive lines) at position kz0 + u dk, dk = nth / TL (a multiple
  // of 8, so every position of a thread has the parity of kz0).  The
  // launch keeps TL n <= 16 nth; lanes with kz0 >= n (TL n < nth) only
  // help with the LDS phases.  Lines past nl load the last line and are
  // zeroed (forward) or not stored.
  constexpr int PF = 16;
  const int tot = TL * n, lp = tid & (TL - 1), kz0 = tid >> logtl, dk = nth >> logtl;
  const int nu = min(PF, (tot + nth - 1) / nth);
  const bool lin = l0 + lp < nl;
  TW v[PF];
  {
    const int kc = min(kz0, n - 1);
    const TW *src = S + min(l0 + lp, nl - 1) + nl * kc;
    const long step = nl * dk, last = (long)((n - 1 - kc) / dk) * step;
#pragma unroll
    for (int u = 0; u < PF; ++u)
      if (u < nu) v[u] = src[min(u * step, last)];
  }
  __syncthreads();  // twiddle tables
  // Makhoul order of position kz: kz/2 for even kz, n-1-kz/2 for odd kz,
  // for the thread's positions pm0 + u dpm.  Forward: the lines go into
  // the pair's complex sequence in Makhoul order (and come out in natural
  // order); inverse: in natural order (and out in Makhoul order).
  TW *const dpair = ((lp & 1) ? im : re) + (lp >> 1) * sn;
  const int pm0 = (kz0 & 1) ? n - 1 - (kz0 >> 1) : (kz0 >> 1);
  const int dpm = (kz0 & 1) ? -(dk >> 1) : (dk >> 1);
  const int pi0 = dir > 0 ? pm0 : kz0, dpi = dir > 0 ? dpm : dk;
#pragma unroll
  for (int u = 0; u < PF; ++u)
    if (u < nu && kz0 + u * dk < n) dpair[pi0 + u * dpi] = lin ? v[u] : (TW)0;
  __syncthreads();
  if (dir < 0) {
    // in place, one (k, n-k) pair per task (k = 0..n/2, Y[n] = 0):
    // W[k] = e^{i pi k/2n} ((Ya[k] + Yb[n-k]) + i (Yb[k] - Ya[n-k]))
    const int ltq = logtl - 1, TQ = TL >> 1, nh = n >> 1, tq = TQ * (nh + 1);
    for (int e = tid; e < tq; e += nth) {
      const int q = e & (TQ - 1), k = e >> ltq, kn = (n - k) & (n - 1);
      TW *rq = re + q * sn, *iq = im + q * sn;
      const TW a0 = rq[k], b0 = iq[k];
      const TW an = k > 0 ? rq[kn] : (TW)0, bn = k > 0 ? iq[kn] : (TW)0;
      {
        const TW uu = a0 + bn, w = b0 - an, c = ecos(k), sv = esin(k);
        rq[k] = uu * c - w * sv;
        iq[k] = uu * sv + w * c;
      }
      if (k > 0 && k < nh) {
        const TW uu = an + b0, w = bn - a0, c = ecos(kn), sv = esin(kn);
        rq[kn] = uu * c - w * sv;
        iq[kn] = uu * sv + w * c;
      }
    }
    __syncthreads();
  }
  lds_fft(re, im, TL / 2, logn, sn, twl, twl + n / 2, (TW)(dir > 0 ? -1 : 1), tid, nth);
  const TW inv_n = (TW)1 / (TW)n;  // exact: n is a power of two
  if (kz0 < n && lin) {
    TW *dst = S + (l0 + lp) + nl * kz0;
    const long step = nl * dk;
    const TW *zq = re + (lp >> 1) * sn, *zi = im + (lp >> 1) * sn;
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int kz = kz0 + u * dk;
      if (u < nu && kz < n) {
        TW outv;
        if (dir > 0) {
          const int kr = (n - kz) & (n - 1);
          const TW zr = zq[kz], zim = zi[kz], wr = zq[kr], wi = zi[kr];
          TW vr, vi;
          if ((lp & 1) == 0) { vr = (TW)0.5 * (zr + wr); vi = (TW)0.5 * (zim - wi); }
          else { vr = (TW)0.5 * (zim + wi); vi = (TW)(-0.5) * (zr - wr); }
          outv = (vr * ecos(kz) + vi * esin(kz)) * inv_n;  // Re(e^{-i pi k/2n} V)/n
        } else {
          outv = dpair[pm0 + u * dpm];
        }
        dst[u * step] = outv;
      }
    }
  }
}

struct DctzTab { const double *twr, *twi, *er, *ei; };
template <typename TW> struct DctzLines {
  TW *S;
  long nl;
  int TL, logtl;
  unsigned nb;  // blocks
};
template <typename TW>
__global__ __launch_bounds__(1024, sizeof(TW) == 4 ? 8 : 1) void k_dctz(DctzLines<TW> a, DctzTab t, int n, int logn, int dir) {
  dctz_block<TW>(blockIdx.x, a.nb, a.S, a.nl, n, logn, a.TL, a.logtl, dir, t.twr, t.twi, t.er, t.ei);
}
// the mixed path's FP64 low modes (first blocks) and its FP32 lines
__global__ __launch_bounds__(1024) void k_dctz2(DctzLines<double> a, DctzLines<float> b, DctzTab t, int n, int logn, int dir) {
  if (blockIdx.x < a.nb) dctz_block<double>(blockIdx.x, a.nb, a.S, a.nl, n, logn, a.TL, a.logtl, dir, t.twr, t.twi, t.er, t.ei);
  else dctz_block<float>(blockIdx.x - a.nb, b.nb, b.S, b.nl, n, logn, b.TL, b.logtl, dir, t.twr, t.twi, t.er, t.ei);
}

// Radial tridiagonal solves of every (mode, kz) system (solve_radial,
// poisson_solve.F90:270-323) with precomputed inverse pivots ib; lanes over
// the packed mode index (contiguous), P waves of M rows each.
// FP32: at most 64 VGPRs, so that two 1024-lane blocks share a CU.
template <typename T, int M>
__device__ __forceinline__ void radial_block(unsigned blk, T (&sh_v)[16][64], T (&sh_p)[16][64], T *__restrict__ S,
                                             const T *__restrict__ ib, long nm, long nlines, int nr,
                                             const T *__restrict__ aab, const T *__restrict__ ccb) {
#pragma clang fp contract(off)
  // Every fused operation is written out, so that all kernels and segment
  // lengths with this body round alike: the mixed path's forms are compared bit
  // for bit, and a last bit of an FP32 line reaches the whole field.  (The
  // carry G joins the last row of a segment with one rounding and the others
  // with two: the results have always had these bits.)
  auto fma_t = [](T x, T y, T z) {
    if constexpr (sizeof(T) == 4) return __builtin_fmaf(x, y, z); else return __builtin_fma(x, y, z);
  };
  const int lane = threadIdx.x & 63;
  const int s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int P = blockDim.x >> 6;
  const long L = (long)blk * 64 + lane;
  const bool act = L < nlines;
  const long Lc = act ? L : nlines - 1;  // addresses stay in bounds; results of !act lanes are dropped
  const long pos = Lc % nm, kz = Lc / nm;
  const long base = pos + nm * (long)nr * kz;
  const int p0 = s * M, len = min(M, nr - p0);
  // all loads of the segment go out before the first use; positions past
  // the line end clamp to its last row and are masked (uniform selects)
  T x[M], w[M];
#pragma unroll
  for (int t = 0; t < M; ++t) {
    const long ad = base + nm * min(p0 + t, nr - 1);
    w[t] = ib[ad];
    x[t] = S[ad];
  }
  __builtin_amdgcn_sched_barrier(0);
  T gp = (T)0, Pacc = (T)1;
#pragma unroll
  for (int t = 0; t < M; ++t) {
    const int p = p0 + t, pc = min(p, nr - 1);
    const bool in = t < len;
    const T ibv = w[t];
    const T B = -aab[pc + 1] * ibv * (T)(p > 0);
    const T v = fma_t(ibv, x[t], B * gp);
    x[t] = in ? v : (T)0;
    gp = in ? v : gp;
    Pacc = in ? Pacc * B : Pacc;
  }
  sh_v[s][lane] = gp;
  sh_p[s][lane] = Pacc;
  __syncthreads();
  T G = (T)0;
  for (int s2 = 0; s2 < s; ++s2) G = fma_t(sh_p[s2][lane], G, sh_v[s2][lane]);
  __syncthreads();
  T Pr = (T)1;
#pragma unroll
  for (int t = 0; t < M; ++t) {
    const int p = p0 + t, pc = min(p, nr - 1);
    const bool in = t < len;
    Pr = in ? Pr * (-aab[pc + 1] * w[t] * (T)(p > 0)) : Pr;
    x[t] = !in ? x[t] : t < M - 1 ? x[t] + Pr * G : fma_t(Pr, G, x[t]);
  }
  T xp = (T)0, Qacc = (T)1;
#pragma unroll
  for (int t = M - 1; t >= 0; --t) {
    const int p = p0 + t, pc = min(p, nr - 1);
    const bool in = t < len;
    const T C = ccb[pc + 1] * w[t] * (T)(p < nr - 1);
    const T v = fma_t(-C, xp, x[t]);
    x[t] = in ? v : x[t];
    xp = in ? v : xp;
    Qacc = in ? Qacc * -C : Qacc;
  }
  sh_v[s][lane] = xp;
  sh_p[s][lane] = Qacc;
  __syncthreads();
  T X = (T)0;
  for (int s2 = P - 1; s2 > s; --s2) X = fma_t(sh_p[s2][lane], X, sh_v[s2][lane]);
  if (!act) return;
  T Qr = (T)1;
#pragma unroll
  for (int t = M - 1; t >= 0; --t) {
    if (t < len) {
      const int p = p0 + t;
      Qr *= -ccb[p + 1] * w[t] * (T)(p < nr - 1);
      S[base + nm * p] = fma_t(Qr, X, x[t]);
    }
  }
}

template <typename T> struct RadialLines {
  T *S;
  const T *ib, *aab, *ccb;
  long nm, nlines;
};
template <typename T, int M>
__global__ __launch_bounds__(1024, sizeof(T) == 4 ? 8 : 1) void k_radial(RadialLines<T> a, int nr) {
  __shared__ T sh_v[16][64];
  __shared__ T sh_p[16][64];
  radial_block<T, M>(blockIdx.x, sh_v, sh_p, a.S, a.ib, a.nm, a.nlines, nr, a.aab, a.ccb);
}
// the mixed path's FP64 low modes (first blocks) and its FP32 lines, up to 256
// rows
__global__ __launch_bounds__(1024) void k_radial2(RadialLines<double> a, RadialLines<float> b, int nr) {
  __shared__ double sh_v[16][64];
  __shared__ double sh_p[16][64];
  const unsigned na = (unsigned)((a.nlines + 63) / 64);
  if (blockIdx.x < na)
    radial_block<double, 16>(blockIdx.x, sh_v, sh_p, a.S, a.ib, a.nm, a.nlines, nr, a.aab, a.ccb);
  else
    radial_block<float, 16>(blockIdx.x - na, reinterpret_cast<float(&)[16][64]>(sh_v),
                           reinterpret_cast<float(&)[16][64]>(sh_p), b.S, b.ib, b.nm, b.nlines, nr, b.aab, b.ccb);
}

// fft_ftp_multi (fastfouriertransform.F90:74-82) + copy into dph
// (poisson_solve.F90:29) + dph(nzc)=dph(nz) (divergence.F90:93-99).
template <typename TW>
__global__ __launch_bounds__(256) void k_ifft(VGrid g, const TW *__restrict__ S, const double *__restrict__ S64,
                                              double *__restrict__ phi_out, double *__restrict__ dph,
                                              const double *__restrict__ twr, const double *__restrict__ twi, int LB,
                                              int logn) {
  extern __shared__ unsigned char smem_raw[];
  const int N = g.nt, tid = threadIdx.x, nth = blockDim.x;
  const long nlines = (long)g.nr * g.nz;
  const long l0 = (long)blockIdx.x * LB;
  TW *re = reinterpret_cast<TW *>(smem_raw);
  TW *im = re + (size_t)(LB / 2) * N;
  TW *tb = im + (size_t)(LB / 2) * N;  // packed input, LB*N
  TW *twl = tb + (size_t)LB * N;       // N/2 cos, N/2 sin
  const size_t ojk = al16(sizeof(TW) * ((size_t)2 * LB * N + N));
  int *jk = reinterpret_cast<int *>(smem_raw + ojk);
  // mixed path: the FP64 low modes of the block's lines and an FP64 cos/sin
  // table (N each) staged in LDS for the merge
  double *s64l = reinterpret_cast<double *>(smem_raw + al16(ojk + sizeof(int) * 2 * LB));
  double *tw64 = s64l + 5 * (size_t)LB;
  if (tid < LB) {
    const long l = l0 + tid;
    jk[2 * tid] = (int)(l % g.nr) + 1;
    jk[2 * tid + 1] = (int)(l / g.nr) + 1;
  }
  for (int q = tid; q < N / 2; q += nth) { twl[q] = (TW)twr[q]; twl[N / 2 + q] = (TW)twi[q]; }
  if (S64) {
    for (int q = tid; q < N; q += nth) { tw64[q] = twr[q]; tw64[N + q] = twi[q]; }
    for (int e = tid; e < 5 * LB; e += nth) s64l[e] = S64[5 * min(l0 + e / 5, nlines - 1) + e % 5];
  }
  {
    // batches of U elements: all loads (line clamped, then masked) go out
    // before the first is used
    constexpr int U = 8;
    const int tot = LB * N;
    for (int eb = tid; eb < tot; eb += U * nth) {
      TW v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = min(eb + u * nth, tot - 1);
        const int lp = e >> logn, pos = e - lp * N;
        v[u] = S[(size_t)pos + (size_t)N * min(l0 + lp, nlines - 1)];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = eb + u * nth;
        if (e < tot) {
          const int lp = e >> logn, pos = e - lp * N;
          tb[e] = (l0 + lp < nlines && !(S64 && pos < 5)) ? v[u] : (TW)0;
        }
      }
    }
  }
  __syncthreads();
  {
    // Z[k] = Fa[k] + i Fb[k], Fa[k] = (t(2k-1) - i t(2k))/2, Hermitian extension
    for (int e = tid; e < (LB / 2) * N; e += nth) {
      const int q = e >> logn, k = e - q * N;
      double ar, ai, br, bi;
      auto coef = [&](const TW *t, int kk, double &cr, double &ci) {
        if (kk == 0) { cr = t[0]; ci = 0.0; return; }
        int kh = kk <= N / 2 ? kk : N - kk;
        double a = t[2 * kh - 1];
        double b = (2 * kh < N) ? t[2 * kh] : 0.0;
        cr = 0.5 * a;
        ci = (kk <= N / 2) ? -0.5 * b : 0.5 * b;
        if (2 * kh == N) ci = 0.0;
      };
      coef(tb + (2 * q) * N, k, ar, ai);
      coef(tb + (2 * q + 1) * N, k, br, bi);
      const int slot = q * N + k;
      re[slot] = (TW)(ar - bi);
      im[slot] = (TW)(ai + br);
    }
    __syncthreads();
    lds_fft(re, im, LB / 2, logn, N, twl, twl + N / 2, (TW)1, tid, nth);
  }
  {
    // N divides the block (N <= 256 = nth): every element of a thread has the same theta
    // index ii, so the low-mode twiddles of the merge are loaded once
    const int ii = tid & (N - 1), lstep = nth >> logn;
    double cw1 = 0.0, sw1 = 0.0, cw2 = 0.0, sw2 = 0.0;
    if (S64) {
      int ph2 = 2 * ii;
      if (ph2 >= N) ph2 -= N;
      cw1 = tw64[ii]; sw1 = tw64[N + ii];
      if (3 < N) { cw2 = tw64[ph2]; sw2 = tw64[N + ph2]; }
    }
    for (int lp = tid >> logn; lp < LB; lp += lstep) {
      const long l = l0 + lp;
      if (l >= nlines) break;
      const int q = lp >> 1;
      double v = (lp & 1) ? (double)im[q * N + ii] : (double)re[q * N + ii];
      if (S64) {
        const double *t = s64l + 5 * lp;
        v += t[0];
        {
          const double a = t[1], b = (2 < N) ? t[2] : 0.0;
          if (2 == N) v += 0.5 * a * cw1;
          else v += a * cw1 + b * sw1;
        }
        if (3 < N) {
          const double a = t[3], b = (4 < N) ? t[4] : 0.0;
          if (4 == N) v += 0.5 * a * cw2;
          else v += a * cw2 + b * sw2;
        }
      }
      const int j = jk[2 * lp], k = jk[2 * lp + 1];
      if (phi_out) phi_out[cidx(g, ii + 1, j, k)] = v;
      if (dph) {
        dph[hidx(g, ii + 1, j, k)] = v;
        if (k == g.nz) dph[hidx(g, ii + 1, j, g.nzc)] = v;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// upsol (divergence.F90:69-236) fused with uppres (divergence.F90:239-480).
// A block owns a W (theta) x R (r) column tile and marches up a chunk of z
// planes.  The planes k-2..k+1 of dph live in a 4-slot LDS ring (with two
// theta columns and two r rows of halo on the low side, one on the high
// side), so each dph value is fetched from HBM about once; the gradient
// components qcap are recomputed from the ring where the reference stores
// them.  Everything that depends on the thread's r row only (metric ratios,
// reciprocals of rm) is hoisted out of the z loop; a wavefront of a 64-wide
// tile has one row and holds these in scalar registers, which leaves room for
// a fourth wave per SIMD (64x128x256: 64.5 -> 60 us).  Bound by memory: 15
// arrays, 5.2 TB/s at 128x256x512.
// ---------------------------------------------------------------------------
template <int W, int R, bool ZS>
__global__ __launch_bounds__(W * R, W == 64 ? 4 : 3) void k_project(VGrid g, VCoef c, ZMet zm, double adt, double be,
                                                    int kchunk, int xcd, const double *__restrict__ dph,
                                                    const double *__restrict__ dq1,
                                                    const double *__restrict__ dq2, const double *__restrict__ dq3,
                                                    double *__restrict__ q1, double *__restrict__ q2,
                                                    double *__restrict__ q3, double *__restrict__ prg1,
                                                    double *__restrict__ prg2, double *__restrict__ prg3,
                                                    double *__restrict__ pres, int *__restrict__ flag) {
  constexpr int LC = W + 3, LR = R + 3, NE = LR * LC, NT = W * R;
  constexpr int NL = (NE + NT - 1) / NT;
  __shared__ double ring[4][LR][LC + 1];
  // a wavefront has one r row (W = 64): its coefficients sit in scalar registers
  const int tx = threadIdx.x, ty = W == 64 ? __builtin_amdgcn_readfirstlane(threadIdx.y) : threadIdx.y, tid = ty * W + tx;
  auto uni = [](double v) {
    if (W != 64) return v;
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)), __builtin_amdgcn_readfirstlane(__double2loint(v)));
  };
  const int nt = g.nt, nr = g.nr, nz = g.nz, nrc = g.nrc, nzc = g.nzc;
  const long sj = g.sj, sk = g.sk;
  int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
  if (xcd) xcd_block(bx, by, bz);
  const int i0 = bx * W;  // 0-based theta of the tile's first column
  const int j0 = by * R;  // rows 0..nrc (row 0 only takes the inlet copy of q3)
  const int kb = 1 + bz * kchunk;
  const int ke = min(kb + kchunk - 1, nzc);
  // ring fill: element e = tid + l*NT of the (LR x LC) plane tile
  long goff[NL];
  int lrow[NL], lcol[NL];
  bool lval[NL];
#pragma unroll
  for (int l = 0; l < NL; l++) {
    const int e = tid + l * NT;
    const int r = e / LC, cc = e - r * LC;
    const int jj = j0 - 2 + r;
    int ii = i0 - 2 + cc;
    ii %= nt;
    if (ii < 0) ii += nt;
    lrow[l] = r; lcol[l] = cc;
    lval[l] = (e < NE) && jj >= 0 && jj <= nr + 2;
    goff[l] = lval[l] ? (long)ii + (long)jj * sj : 0;
  }
  double pre[NL];
  // unconditional loads from in-bounds (clamped) addresses, masked after:
  // the loads of one plane issue together
  auto fetch = [&](int kk) {
    const long kc = (long)min(max(kk, 0), nz + 2) * sk;
    const bool kin = kk >= 0 && kk <= nz + 2;
#pragma unroll
    for (int l = 0; l < NL; l++) {
      const double v = dph[goff[l] + kc];
      pre[l] = (lval[l] && kin) ? v : 0.0;
    }
  };
  auto stash = [&](int kk) {
#pragma unroll
    for (int l = 0; l < NL; l++)
      if (tid + l * NT < NE) ring[kk & 3][lrow[l]][lcol[l]] = pre[l];
  };
  fetch(kb - 2); stash(kb - 2);
  fetch(kb - 1); stash(kb - 1);
  fetch(kb); stash(kb);
  fetch(kb + 1);
  // the thread's cell column
  const int i = i0 + tx + 1, j = j0 + ty;
  const bool act = (i <= nt) && (j <= nrc);
  const int jr = (j <= nrc) ? j : nrc;           // clamped row for coefficient loads
  const int jq = (jr >= 1 && jr <= nr) ? jr : 1;  // rows of the uppres coefficients
  const int djp = (jq == nr) ? 0 : 1, djm = (jq == 1) ? 0 : -1;
  // radial gradient rc dx2 / dcr (divergence.F90:132, 327)
  const double a1 = uni(adt * g.dx1 / c.rm[jq]), a2 = uni(adt * c.rc[jr] * g.dx2 / c.dcr[jr]), a3 = adt * g.dx3;
  const double irm = uni(1.0 / c.rm[jq]), irmp = uni(1.0 / c.rm[jq + djp]), irmm = uni(1.0 / c.rm[jq + djm]);
  const double irmn = uni(1.0 / c.rm[jq + 1]);
  const double s1t11 = c.s1t11[jq], s1t2n = c.s1t2n[jq], s1t2s = c.s1t2s[jq], s1t2c = c.s1t2c[jq];
  const double s2t11 = c.s2t11[jq], s2t2p = c.s2t2p[jq], s2t2m = c.s2t2m[jq];
  const double s3t2n = c.s3t2n[jq], s3t2s = c.s3t2s[jq];
  const int jqp = min(jq + 1, nrc), jqm = max(jq - 1, 1);
  const double rcj = uni(c.rc[jq] / c.dcr[jq]), rcp = uni(c.rc[jqp] / c.dcr[jqp]), rcm = uni(c.rc[jqm] / c.dcr[jqm]);
  const double dx1 = g.dx1, dx2 = g.dx2, dx3 = g.dx3, dx3q = g.dx3q, slip = g.slip;
  const int cx = tx + 2, cy = ty + 2;
  // the streamed operands of the next plane are loaded while this one is computed
  const bool rowu = act && j >= 1 && j <= nr;
  double n_dq1 = 0.0, n_dq2 = 0.0, n_dq3 = 0.0, n_pres = 0.0;
  double n_p1 = 0.0, n_p2 = 0.0, n_p3 = 0.0;
  // operands of cell (i, j, kk); lanes, rows and planes where a value is not
  // used read a clamped in-bounds address instead of branching, so that the
  // seven loads issue together
  const int ic = min(i, nt), jc1 = min(max(j, 1), nr);
  auto load_cell = [&](int kk) {
    const int kc = min(kk, ke), kp = min(max(kc, 1), nz);
    const long oo = (long)(ic - 1) + (long)min(j, nrc) * sj + (long)kc * sk;
    const long pp = (long)(ic - 1) + (long)nt * ((long)(jc1 - 1) + (long)nr * (long)(kp - 1));
    n_dq3 = dq3[oo];
    n_dq1 = dq1[oo];
    n_dq2 = dq2[oo];
    n_p1 = prg1[pp];
    n_p2 = prg2[pp];
    n_p3 = prg3[pp];
    n_pres = pres[oo];
  };
  load_cell(kb);
  // the plane's axial metric terms, read one plane ahead as well
  struct ZM { double c3, c3p, c3m, cp, cm, fp, fm; };
  auto load_zm = [&](int k) { return ZM{zm.c3[k], zm.c3[k + 1], zm.c3[k - 1], zm.cp[k], zm.cm[k], zm.fp[k], zm.fm[k]}; };
  ZM z{};
  if (ZS) z = load_zm(kb);
  for (int k = kb; k <= ke; k++) {
    const ZM zk = z;
    stash(k + 1);
    const double c_dq1 = n_dq1, c_dq2 = n_dq2, c_dq3 = n_dq3, c_pres = n_pres;
    const double c_p1 = n_p1, c_p2 = n_p2, c_p3 = n_p3;
    __syncthreads();
    fetch(k + 2);
    load_cell(k + 1);
    if (ZS) z = load_zm(min(k + 1, ke));
    if (act) {
      const double(*P0)[LC + 1] = ring[k & 3];
      const double(*Pm)[LC + 1] = ring[(k - 1) & 3];
      const double(*Pp)[LC + 1] = ring[(k + 1) & 3];
      const double(*Pm2)[LC + 1] = ring[(k - 2) & 3];
      // kmv quirk of uppres: km = 1 at k = 1 and km = nz at k = nz
      const double(*Pkm)[LC + 1] = (k == 1 || k == nz) ? P0 : Pm;
      const long o = (long)(i - 1) + (long)j * sj + (long)k * sk;
      const double p0 = P0[cy][cx];
      // axial mesh: the z gradient at faces k, k+1, k-1 and the z-gradient
      // factor of upsol; the uniform mesh keeps dx3
      constexpr bool zs = ZS;  // axial mesh (a separate instantiation)
      const double zc0 = zs ? zk.c3 : dx3, zcp = zs ? zk.c3p : dx3, zcm = zs ? zk.c3m : dx3;
      const double a3k = zs ? adt * zc0 : a3;
      // ---- upsol ----
      if (j >= 1 && j <= nr) {
        const double v = c_dq1 - a1 * (p0 - P0[cy][cx - 1]);
        q1[o] = v;
        if (j == nr) q1[o + sj] = slip * v;
      }
      if (j >= 2 && j <= nr) q2[o] = c_dq2 - a2 * (p0 - P0[cy - 1][cx]);
      if (j == 1 || j == nrc) q2[o] = 0.0;
      if (k == 1) q3[o] = c_dq3;
      if (k >= 2 && j >= 1 && j <= nr) {
        const double v = c_dq3 - a3k * (p0 - Pm[cy][cx]);
        q3[o] = v;
        if (j == nr) q3[o + sj] = slip * v;
      }
      if (k <= nz && j >= 1 && j <= nr) {
        const long pc = (long)(i - 1) + (long)nt * ((long)(j - 1) + (long)nr * (long)(k - 1));
        // theta component: qcap = (dph(i) - dph(i-1)) dx1 / rm
        {
          const double qc0 = (p0 - P0[cy][cx - 1]) * dx1 * irm;
          const double qip = (P0[cy][cx + 1] - p0) * dx1 * irm;
          const double qim = (P0[cy][cx - 1] - P0[cy][cx - 2]) * dx1 * irm;
          const double qkp = (Pp[cy][cx] - Pp[cy][cx - 1]) * dx1 * irm;
          const double qkm = (Pkm[cy][cx] - Pkm[cy][cx - 1]) * dx1 * irm;
          const double qjp = (P0[cy + djp][cx] - P0[cy + djp][cx - 1]) * dx1 * irmp;
          const double qjm = (P0[cy + djm][cx] - P0[cy + djm][cx - 1]) * dx1 * irmm;
          const double d11 = (qip - 2.0 * qc0 + qim) * s1t11;
          const double d33 = zs ? (qkp - qc0) * zk.cp - (qc0 - qkm) * zk.cm : (qkp - 2.0 * qc0 + qkm) * dx3q;
          const double qnn = qjp * irmn - qc0 * irm;
          const double qss = qc0 * irm - qjm * irmm;
          const double d22 = (qnn * s1t2n - qss * s1t2s) * s1t2c;
          prg1[pc] = c_p1 + qc0 - be * (d11 + d33 + d22);
        }
        // r component: qcap = (dph(j) - dph(j-1)) dx2 rc, zero at j = 1 and nrc
        if (j >= 2) {
          const double qc0 = (p0 - P0[cy - 1][cx]) * dx2 * rcj;
          const double qip = (P0[cy][cx + 1] - P0[cy - 1][cx + 1]) * dx2 * rcj;
          const double qim = (P0[cy][cx - 1] - P0[cy - 1][cx - 1]) * dx2 * rcj;
          const double qkp = (Pp[cy][cx] - Pp[cy - 1][cx]) * dx2 * rcj;
          const double qkm = (Pkm[cy][cx] - Pkm[cy - 1][cx]) * dx2 * rcj;
          const double qjp = (j + 1 < nrc) ? (P0[cy + 1][cx] - p0) * dx2 * rcp : 0.0;
          const double qjm = (j - 1 > 1) ? (P0[cy - 1][cx] - P0[cy - 2][cx]) * dx2 * rcm : 0.0;
          const double d11 = (qip - 2.0 * qc0 + qim) * s2t11;
          const double d33 = zs ? (qkp - qc0) * zk.cp - (qc0 - qkm) * zk.cm : (qkp - 2.0 * qc0 + qkm) * dx3q;
          const double d22 = (qjp - qc0) * s2t2p - (qc0 - qjm) * s2t2m;
          prg2[pc] = c_p2 + qc0 - be * (d11 + d22 + d33);
        }
        // z component: qcap = (dph(k) - dph(k-1)) dx3, zero at k = 1
        {
          const double qkp = (Pp[cy][cx] - p0) * zcp;
          if (qkp != qkp) atomicOr(flag, 1);  // "Flow field crash" (divergence.F90:396-399)
          if (k >= 2) {
            const double qc0 = (p0 - Pm[cy][cx]) * zc0;
            const double qip = (P0[cy][cx + 1] - Pm[cy][cx + 1]) * zc0;
            const double qim = (P0[cy][cx - 1] - Pm[cy][cx - 1]) * zc0;
            const double qkm = (k - 1 > 1) ? (Pm[cy][cx] - Pm2[cy][cx]) * zcm : 0.0;
            const double qjp = (P0[cy + djp][cx] - Pm[cy + djp][cx]) * zc0;
            const double qjm = (P0[cy + djm][cx] - Pm[cy + djm][cx]) * zc0;
            const double d11 = (qip - 2.0 * qc0 + qim) * s1t11;
            const double d33 = zs ? (qkp - qc0) * zk.fp - (qc0 - qkm) * zk.fm : (qkp - 2.0 * qc0 + qkm) * dx3q;
            const double d22 = (qjp - qc0) * s3t2n - (qc0 - qjm) * s3t2s;
            prg3[pc] = c_p3 + qc0 - be * (d11 + d22 + d33);
          }
        }
        {
          const double d11 = (P0[cy][cx + 1] + P0[cy][cx - 1] - 2.0 * p0) * s1t11;
          const double d22 = (P0[cy + djp][cx] - p0) * s3t2n - (p0 - P0[cy + djm][cx]) * s3t2s;
          const double d33 = zs ? (Pp[cy][cx] - p0) * zk.cp - (p0 - Pkm[cy][cx]) * zk.cm
                                : (Pp[cy][cx] + Pkm[cy][cx] - 2.0 * p0) * dx3q;
          pres[o] = c_pres + p0 - be * (d11 + d22 + d33);
        }
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Vortex-core statistics of analysis (run.F90:238-388) as a device
// reduction: per cell the azimuthal vorticity (dvdz - dwdr) and the swirl
// q1m of the cell centre; inside the window 0.1 < z/L < 0.9,
// 0.05 < r/R < 0.8, j != 1: their maxima and the sums of z w^2 r, w^2 r,
// w^2 r, w^2 (w = vorticity where > 0, then swirl where > 0) times dx1 dx2
// dx3.  Per-block partials [block][10], summed in a fixed order.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_analysis(VGrid g, double rmax, double zmax, const double *__restrict__ rmv,
                                                  const double *__restrict__ zpos,
                                                  const double *__restrict__ q1, const double *__restrict__ q2,
                                                  const double *__restrict__ q3, double *__restrict__ part) {
  const long ncell = (long)g.nt * g.nr * g.nz;
  const double dz = zmax / g.nz, w = g.dx1 * g.dx2 * g.dx3;
  double v[10] = {-10000.0, -10000.0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (long c = (long)blockIdx.x * 256 + threadIdx.x; c < ncell; c += (long)gridDim.x * 256) {
    const int ith = (int)(c % g.nt) + 1;
    const long rest = c / g.nt;
    const int ir = (int)(rest % g.nr) + 1, iz = (int)(rest / g.nr) + 1;
    // msh%rm, msh%zm: the radial and axial meshes (uniform or set)
    const double rm = rmv[ir], zm = zpos ? zpos[iz] : (iz - 0.5) * dz;
    if (!(zm < 0.90 * zmax && zm > 0.10 * zmax && rm < 0.80 * rmax && rm > rmax * 0.05 && ir != 1)) continue;
    const int ithp1 = ith == g.nt ? 1 : ith + 1;
    const double q1m = g.nt > 1 ? 0.5 * (q1[hidx(g, ith, ir, iz)] + q1[hidx(g, ithp1, ir, iz)]) : q1[hidx(g, ith, ir, iz)];
    const double rp = rmv[ir + 1], rmm = rmv[ir - 1];
    const double dwdr = 0.5 * ((q3[hidx(g, ith, ir + 1, iz)] + q3[hidx(g, ith, ir + 1, iz + 1)]) -
                               (q3[hidx(g, ith, ir - 1, iz)] + q3[hidx(g, ith, ir - 1, iz + 1)])) / (rp - rmm);
    const double zp = zpos ? zpos[iz + 1] : (iz + 0.5) * dz, zmm = zpos ? zpos[iz - 1] : (iz - 1.5) * dz;
    const double dvdz = 0.5 * ((q2[hidx(g, ith, ir, iz + 1)] / rm + q2[hidx(g, ith, ir + 1, iz + 1)] / rp) -
                               (q2[hidx(g, ith, ir + 1, iz - 1)] / rp + q2[hidx(g, ith, ir, iz - 1)] / rm)) / (zp - zmm);
    const double vort = +(dvdz - dwdr), swrl = q1m;
    v[0] = fmax(vort, v[0]);
    v[1] = fmax(swrl, v[1]);
    if (vort > 0.0) {
      v[2] += zm * vort * vort * rm * w;
      v[3] += vort * vort * rm * w;
      v[4] += vort * vort * rm * w;
      v[5] += vort * vort * w;
    }
    if (swrl > 0.0) {
      v[6] += zm * swrl * swrl * rm * w;
      v[7] += swrl * swrl * rm * w;
      v[8] += swrl * swrl * rm * w;
      v[9] += swrl * swrl * w;
    }
  }
  __shared__ double red[10][4];
  for (int q = 0; q < 10; q++) {
    double x = v[q];
    for (int o = 32; o > 0; o >>= 1) {
      const double y = __shfl_xor(x, o);
      x = (q < 2) ? fmax(x, y) : x + y;
    }
    if ((threadIdx.x & 63) == 0) red[q][threadIdx.x >> 6] = x;
  }
  __syncthreads();
  if (threadIdx.x < 10) {
    const int q = threadIdx.x;
    const double a = red[q][0], b = red[q][1], cc = red[q][2], d = red[q][3];
    part[(long)blockIdx.x * 10 + q] = (q < 2) ? fmax(fmax(a, b), fmax(cc, d)) : ((a + b) + (cc + d));
  }
}
__global__ void k_analysis_sum(const double *__restrict__ part, int nblk, double *__restrict__ out) {
  const int q = threadIdx.x;
  if (q >= 10) return;
  double x = (q < 2) ? -10000.0 : 0.0;
  for (int b = 0; b < nblk; b++) x = (q < 2) ? fmax(x, part[(long)b * 10 + q]) : x + part[(long)b * 10 + q];
  out[q] = x;
}

}  // namespace

// ===========================================================================
// launchers
// ===========================================================================
#define CHECK_LAUNCH() (void)hipGetLastError()

void launch_scalars(vrh_t *h) {
  hipLaunchKernelGGL(k_scalars, dim3(1), dim3(64), 0, h->stream, h->d_sc, h->dt, h->rk[1].a, h->rk[2].a,
                     h->rk[3].a, h->inlet_area, h->cor_red, 1, 0.0);
}
// the same scalars for the step that has reached time t (no advance)
void launch_scalars_at(vrh_t *h, double t) {
  hipLaunchKernelGGL(k_scalars, dim3(1), dim3(64), 0, h->stream, h->d_sc, h->dt, h->rk[1].a, h->rk[2].a,
                     h->rk[3].a, h->inlet_area, h->cor_red, 0, t);
}

template <typename TW> void launch_explicit(vrh_t *h, int irk) {
  // compute type of the stencils: the work type (FP32 in the mixed path)
  using TC = TW;
  const VGrid &g = h->g;
  const int ntp = (g.nt + 63) / 64 * 64;  // lanes of a theta row
  const int nlev = h->theta_levels[irk];
  const double *rowc = h->d_rowc, *pcrt = h->pcrt(irk);
  // The default form (the tuner times all four).  us at the chunk lengths below,
  // plane, marching, wave (2), wave (3):
  //   FP64   32x64x128: 16, 34, 29, 32; 64x96x256: 53, 70, 62, 127; 64x400x64: 57, 83, 74, 134
  //          96x64x256: 58, 59, 64, 50; 100x96x200: 74, 73, 74, 63; 128x256x512: 642, 453, 436, 387
  //          129x128x128: 91, 106, 106, 107; 144x96x160: 92, 92, 92, 108; 192x40x600: 186, 146, 145, 184
  //          200x96x160: 140, 132, 132, 435; 256x64x128: 71, 71, 71, 221; 256x128x256: 328, 264, 264, 857
  //   mixed  32x64x128: 14.7, 21, 17, 17; 64x128x256: 53, 52, 43, 43; 64x400x64: 41, 47, 39, 39
  //          100x96x200: 60, 60, 72, 46; 128x256x512: 514, 341, 391, 321
  //          129x128x128: 71, 89, 58, 58; 192x40x600: 149, 138, 103, 103
  //          200x96x160: 109, 97, 100, 101; 256x128x256: 270, 182, 219, 219
  // so rows of up to 64 lanes take the plane form in FP64 and the wave form in
  // mixed, up to 128 the wave form, beyond the marching form, or in mixed up to
  // 192 the wave form (four rows of 192 lanes).  Two sizes miss their best: FP64
  // rows just beyond 128 (129x128x128), where the line cannot be drawn by the
  // row's width alone, and narrow mixed rows, whose default leaves the plane form
  // out: its contraction of q3's terms and its quotients round differently from
  // the others', which agree bit for bit.
  const bool f64 = sizeof(TW) == 8;
  const int var = h->explicit_variant >= 0 ? h->explicit_variant
                  : g.nt <= 64             ? (f64 ? 0 : 2)
                  : g.nt <= 128            ? 3
                  : g.nt <= 192            ? (f64 ? 1 : 2)
                                           : 1;
  KTimer kt(h, KT_EXPLICIT);
#define EXPL_ARGS                                                                                                    \
  h->f.q1, h->f.q2, h->f.q3, h->f.prg1, h->f.prg2, h->f.prg3, (TW *)h->f.ru1, (TW *)h->f.ru2, (TW *)h->f.ru3,        \
      (TW *)h->f.r1, (TW *)h->f.r2, (TW *)h->f.r3
  if (var == 0) {
    // one z plane per block
    const int roww = g.nt <= 32 ? 32 : g.nt <= 64 ? 64 : 0, rl = roww ? roww : ntp;
    const int rj = rl <= 128 ? 256 / rl : 1;
    dim3 blk(rl, rj), grd((g.nr + rj - 1) / rj, g.nz);
    const size_t sh = sizeof(TC) * 6 * (size_t)rj * rl;
    const bool zs = h->zmet.m3 != nullptr;
    auto kern = roww == 32   ? (zs ? k_explicit_cell<TW, TC, true, 32> : k_explicit_cell<TW, TC, false, 32>)
                : roww == 64 ? (zs ? k_explicit_cell<TW, TC, true, 64> : k_explicit_cell<TW, TC, false, 64>)
                             : (zs ? k_explicit_cell<TW, TC, true, 0> : k_explicit_cell<TW, TC, false, 0>);
    hipLaunchKernelGGL(kern, grd, blk, sh, h->stream, g, rowc, pcrt, h->rk[irk], h->zmet, EXPL_ARGS);
    return;
  }
  // Planes per block: each block first loads three planes of its rows, so
  // long chunks, as far as they leave four blocks per CU (us at 4, 8, 16, 32
  // planes: mixed 33x96x200 31, 34, 44, 78; 128x96x256 65, 61, 76, 123;
  // 128x256x512 310, 299, 295, 332; 256x512x1024 2939, 2642, 2483, 2428).
  auto chunk = [&](int rows) {
    const long rb = (g.nr + rows - 1) / rows;
    int kc = 32;
    while (kc > 4 && rb * ((g.nz + kc - 1) / kc) < 1024) kc /= 2;
    return kc;
  };
  // z marching: rows per block for 512 threads within 64 KB of LDS
  auto lds = [&](int rj, int prow) {
    return sizeof(double) * (size_t)rj * prow +
           sizeof(TC) * ((size_t)rj * kRowCoefs + (size_t)9 * (rj + 2) * ntp + (size_t)6 * rj * ntp);
  };
  // the wave form's ratio table holds this substep's levels only
  auto lds_w = [&](int rw) { return lds(rw, kPcrHead + 2 * nlev); };
  if (var == 2 || var == 3) {
    // one wavefront per r row.  Form 2: the most rows (<= 8) whose LDS fits
    // 64 KB.  Form 3: among the instantiated row counts, the one that keeps
    // the most waves resident on a CU within the device's LDS per block and
    // per CU (ties: more rows, less r-halo re-read).  Shapes without an
    // instantiation fall back to the marching form.  WPE: waves per SIMD the
    // LDS allows (register budget).
    const int cpl = ntp / 64;
    int rw = 8;
    size_t lim = 65536;
    if (var == 2) {
      while (rw > 1 && lds(rw, kPcrRow) > lim) rw--;
    } else {
      lim = (size_t)h->lds_block;
      const int cand1[] = {8, 6}, cand2[] = {6, 4, 2}, cand3[] = {4, 2}, cand4[] = {2};
      const int *cd = cpl == 1 ? cand1 : cpl == 2 ? cand2 : cpl == 3 ? cand3 : cand4;
      const int ncd = cpl == 1 ? 2 : cpl == 2 ? 3 : cpl == 3 ? 2 : 1;
      int best = 0;
      rw = 0;
      for (int i = 0; i < ncd; i++) {
        const size_t L = lds_w(cd[i]);
        if (L > lim) continue;
        const int waves = cd[i] * (int)((size_t)h->lds_cu / L);
        if (waves > best) { best = waves; rw = cd[i]; }
      }
      if (rw == 0) rw = 1;
    }
    const int kchunk = chunk(rw);
    dim3 grd((g.nr + rw - 1) / rw, (g.nz + kchunk - 1) / kchunk);
    bool done = rw > 1 && (var == 2 ? lds(rw, kPcrRow) : lds_w(rw)) <= lim;
#define EXPL_WAVE(C, R, W)                                                                                            \
  hipLaunchKernelGGL((h->zmet.m3 ? k_explicit_wave<TW, TC, C, R, W, true> : k_explicit_wave<TW, TC, C, R, W, false>), \
                     grd, dim3(64, R), lds_w(R), h->stream, g, rowc, pcrt, h->rk[irk], h->zmet, nlev, kchunk, EXPL_ARGS)
    if (done) {
      if (cpl == 1 && rw == 8) EXPL_WAVE(1, 8, 4);
      else if (cpl == 1 && rw == 6) EXPL_WAVE(1, 6, 3);
      else if (cpl == 2 && rw == 6) EXPL_WAVE(2, 6, 3);
      else if (cpl == 2 && rw == 4) EXPL_WAVE(2, 4, 2);
      else if (cpl == 2 && rw == 2) EXPL_WAVE(2, 2, 2);
      else if (cpl == 3 && rw == 4) EXPL_WAVE(3, 4, 2);
      else if (cpl == 3 && rw == 2) EXPL_WAVE(3, 2, 2);
      else if (cpl == 4 && rw == 2) EXPL_WAVE(4, 2, 2);
      else done = false;
    }
#undef EXPL_WAVE
    if (done) return;
  }
  int rj = 512 / ntp;
  if (rj < 1) rj = 1;
  while (rj > 1 && lds(rj, kPcrRow) > 65536) rj--;
  const int kchunk = chunk(rj);
  dim3 blk(ntp, rj), grd((g.nr + rj - 1) / rj, (g.nz + kchunk - 1) / kchunk);
  auto kern = h->zmet.m3 ? k_explicit_march<TW, TC, true> : k_explicit_march<TW, TC, false>;
  hipLaunchKernelGGL(kern, grd, blk, lds(rj, kPcrRow), h->stream, g, rowc, pcrt, h->rk[irk], h->zmet, kchunk, EXPL_ARGS);
#undef EXPL_ARGS
}

// Blocks of the explicit kernel's one-wave-per-row form and tuned z-DCT
// tiles may take more than 64 KB of LDS where the device allows it (gfx950:
// 160 KB per CU).  Those instantiations opt in once per handle; if the
// runtime refuses, they keep the 64 KB limit.
void lds_optin(vrh_t *h) {
  int dev = 0, lb = 0, lc = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&lb, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
      hipDeviceGetAttribute(&lc, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) != hipSuccess)
    return;
  if (lc < lb) lc = lb;
  bool ok = true;
  if (lb > 65536) {
    const void *fns[] = {
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 1, 8, 4, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 1, 6, 3, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 2, 6, 3, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 2, 4, 2, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 2, 2, 2, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 3, 4, 2, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 3, 2, 2, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 4, 2, 2, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 1, 8, 4, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 1, 6, 3, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 2, 6, 3, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 2, 4, 2, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 2, 2, 2, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 3, 4, 2, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 3, 2, 2, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 4, 2, 2, false>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 1, 8, 4, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 1, 6, 3, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 2, 6, 3, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 2, 4, 2, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 2, 2, 2, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 3, 4, 2, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 3, 2, 2, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<double, double, 4, 2, 2, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 1, 8, 4, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 1, 6, 3, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 2, 6, 3, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 2, 4, 2, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 2, 2, 2, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 3, 4, 2, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 3, 2, 2, true>),
        reinterpret_cast<const void *>(&k_explicit_wave<float, float, 4, 2, 2, true>),
        reinterpret_cast<const void *>(&k_dctz<float>),
        reinterpret_cast<const void *>(&k_dctz<double>),
        reinterpret_cast<const void *>(&k_dctz2)};
    for (const void *f : fns)
      ok = ok && hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lb) == hipSuccess;
  }
  (void)hipGetLastError();
  if (lb > 65536) ok = ok && dense_lds_optin(lb);
  (void)hipGetLastError();
  if (ok) { h->lds_block = lb; h->lds_cu = lc; }
}

static int ilog2(int n) { int l = 0; while ((1 << l) < n) ++l; return l; }

// rows per wave of the radial solves: 16 keeps the segment's rhs and pivots
// in registers (a 1024-lane block allows 128 VGPRs) up to nr = 256; 32 beyond
// (P <= 16)
static int radial_rows(const VGrid &g) { return g.nr <= 256 ? 16 : 32; }
// the radial base coefficients in the solve's type (float copies rounded as
// the device conversion)
static RadialLines<double> radial_lines(vrh_t *h, double *S, const double *ib, long nm) {
  return {S, ib, h->d_aab, h->d_ccb, nm, nm * h->g.nz};
}
static RadialLines<float> radial_lines(vrh_t *h, float *S, const float *ib, long nm) {
  return {S, ib, h->d_aabf, h->d_ccbf, nm, nm * h->g.nz};
}
template <typename T>
static void radial_launch(vrh_t *h, T *S, const T *ib, long nm, hipStream_t st) {
  const VGrid &g = h->g;
  const int M = radial_rows(g), P = (g.nr + M - 1) / M;
  const RadialLines<T> a = radial_lines(h, S, ib, nm);
  dim3 blk(64 * P), grd((unsigned)((a.nlines + 63) / 64));
  KTimer kt(h, KT_RADIAL);
  if (M == 16) hipLaunchKernelGGL((k_radial<T, 16>), grd, blk, 0, st, a, g.nr);
  else hipLaunchKernelGGL((k_radial<T, 32>), grd, blk, 0, st, a, g.nr);
}
static void radial_launch2(vrh_t *h, double *S64, const double *ib64, float *S, const float *ib) {
  const VGrid &g = h->g;
  const int P = (g.nr + 15) / 16;
  const RadialLines<double> a = radial_lines(h, S64, ib64, 5);
  const RadialLines<float> b = radial_lines(h, S, ib, g.nt);
  dim3 blk(64 * P), grd((unsigned)((a.nlines + 63) / 64 + (b.nlines + 63) / 64));
  hipLaunchKernelGGL(k_radial2, grd, blk, 0, h->stream, a, b, g.nr);
}

// z transform of the mixed path's pressure solve on an axial mesh (FP64 path:
// launch_zdense): every spectral line (the nl lines of one z position are
// contiguous, so the array is a column-major nl x nz matrix) times a dense
// nz x nz matrix, out of place.
// Forward: out(:, q) = sum_k in(:, k) Vinv(q, k); inverse: out(:, k) =
// sum_q in(:, q) V(k, q).  The row-major matrices read column-major are
// their transposes, the right operand of both products.
// A failed call is reported through the step's error (mode_rc).
static void zgemm_status(vrh_t *h, rocblas_status st) {
  if (st != rocblas_status_success && !h->mode_rc) {
    h->mode_rc = -3;
    h->err = "rocBLAS z transform failed (status " + std::to_string((int)st) + ")";
  }
}
static void zgemm(vrh_t *h, hipStream_t st, const float *in, float *out, long nl, int dir) {
  const int nz = h->g.nz;
  const float one = 1.f, zero = 0.f;
  rocblas_handle b = (rocblas_handle)h->blas;
  zgemm_status(h, rocblas_set_stream(b, st));
  zgemm_status(h, rocblas_sgemm(b, rocblas_operation_none, rocblas_operation_none, (rocblas_int)nl, nz, nz, &one,
                                in, (rocblas_int)nl, h->d_zvf + (dir > 0 ? 0 : (size_t)nz * nz), nz, &zero, out,
                                (rocblas_int)nl));
  zgemm_status(h, rocblas_set_stream(b, h->stream));
}
static void zgemm(vrh_t *h, hipStream_t st, const double *in, double *out, long nl, int dir) {
  const int nz = h->g.nz;
  const double one = 1.0, zero = 0.0;
  rocblas_handle b = (rocblas_handle)h->blas;
  zgemm_status(h, rocblas_set_stream(b, st));
  zgemm_status(h, rocblas_dgemm(b, rocblas_operation_none, rocblas_operation_none, (rocblas_int)nl, nz, nz, &one,
                                in, (rocblas_int)nl, h->d_zv + (dir > 0 ? 0 : (size_t)nz * nz), nz, &zero, out,
                                (rocblas_int)nl));
  zgemm_status(h, rocblas_set_stream(b, h->stream));
}

// Spectral array (position fastest, then r, then z) <-> the Helmholtz
// handle's slots (slot, z, r), for positions pos0..N-1: 64 x 64 tiles of
// (position, r) through LDS, one z plane per blockIdx.z.
template <typename TW>
__global__ __launch_bounds__(256) void k_hz_gather(const TW *__restrict__ S, double *__restrict__ f, int N, int nr,
                                                   int nz, int pos0) {
  __shared__ double t[64][65];
  const int p0 = pos0 + blockIdx.x * 64, j0 = blockIdx.y * 64, k = blockIdx.z;
  const int np = N - pos0;
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    const int pp = e & 63, jj = e >> 6;
    const int pos = p0 + pp, j = j0 + jj;
    t[jj][pp] = (pos < N && j < nr) ? (double)S[(size_t)pos + (size_t)N * ((size_t)j + (size_t)nr * k)] : 0.0;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    const int jj = e & 63, pp = e >> 6;
    const int b = p0 + pp - pos0, j = j0 + jj;
    if (b < np && j < nr) f[((size_t)b * nz + k) * nr + j] = t[jj][pp];
  }
}
template <typename TW>
__global__ __launch_bounds__(256) void k_hz_scatter(const double *__restrict__ x, TW *__restrict__ S, int N, int nr,
                                                    int nz, int pos0) {
  __shared__ double t[64][65];
  const int p0 = pos0 + blockIdx.x * 64, j0 = blockIdx.y * 64, k = blockIdx.z;
  const int np = N - pos0;
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    const int jj = e & 63, pp = e >> 6;
    const int b = p0 + pp - pos0, j = j0 + jj;
    t[pp][jj] = (b < np && j < nr) ? x[((size_t)b * nz + k) * nr + j] : 0.0;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 64 * 64; e += 256) {
    const int pp = e & 63, jj = e >> 6;
    const int pos = p0 + pp, j = j0 + jj;
    if (pos < N && j < nr) S[(size_t)pos + (size_t)N * ((size_t)j + (size_t)nr * k)] = (TW)t[pp][jj];
  }
}

// shape of a cosine transform by FFT: a power of two of lines per block, data
// + twiddles within 64 KB of LDS (a tuned width may take the device's larger
// per-block LDS: 32 FP32 lines read whole 128-byte rows of the strided
// layout), one FFT butterfly per thread with up to 1024 threads
struct DctzShape { int tl, nth; size_t sh; };
template <typename T> static DctzShape dctz_shape(vrh_t *h, int want) {
  const int nz = h->g.nz, lz = ilog2(nz);
  const size_t es = sizeof(T), lim = want > 0 ? (size_t)h->lds_block : 65536;
  const int tmax = want > 0 ? 32 : 16;
  int tl = 2;
  while (tl * 2 <= tmax && (size_t)(tl * 2) * (nz + 1) * es + (size_t)(es == 4 ? 3 : 1) * nz * es <= lim &&
         (tl * 2 / 2) * nz / fft_min_radix(lz) <= 1024)
    tl *= 2;
  if (want > 0) while (tl > 2 && tl > want) tl /= 2;
  const int b = (tl / 2) * nz / fft_min_radix(lz), nth = b > 512 ? 1024 : b > 256 ? 512 : 256;
  // tile lines, FFT twiddles, and in FP32 the Makhoul twiddles
  return {tl, nth, es * ((size_t)tl * (nz + 1) + (size_t)(es == 4 ? 3 : 1) * nz)};
}
template <typename T> static DctzLines<T> dctz_lines(const DctzShape &p, T *S, long nl) {
  return {S, nl, p.tl, ilog2(p.tl), (unsigned)((nl + p.tl - 1) / p.tl)};
}

// One z transform of the pressure solve, in place on nl lines: the cosine
// transform by FFT (nz a power of two) or as a dense product, or on an axial
// mesh the product with its eigenvectors.
template <typename T> static void z_transform(vrh_t *h, hipStream_t st, T *S, long nl, int dir, int want) {
  const int nz = h->g.nz, lz = ilog2(nz);
  if (h->zmet.m3 || (nz & (nz - 1)) != 0) { launch_zdense<T>(h, st, S, nl, dir); return; }
  const DctzShape p = dctz_shape<T>(h, want);
  const DctzLines<T> a = dctz_lines(p, S, nl);
  hipLaunchKernelGGL(k_dctz<T>, dim3(a.nb), dim3(p.nth), p.sh, st, a, DctzTab{h->d_twz, h->d_twz + nz, h->d_ez, h->d_ez + nz},
                     nz, lz, dir);
}
// that of the mixed path's FP64 low modes and FP32 lines in one launch
static void z_transform2(vrh_t *h, double *S64, long nl64, float *S, long nl, int dir) {
  const int nz = h->g.nz, lz = ilog2(nz);
  if ((nz & (nz - 1)) != 0) { launch_zdense2(h, S64, nl64, S, nl, dir); return; }
  const DctzShape p = dctz_shape<double>(h, 0), q = dctz_shape<float>(h, h->dct_lines);
  const DctzLines<double> a = dctz_lines(p, S64, nl64);
  const DctzLines<float> b = dctz_lines(q, S, nl);
  hipLaunchKernelGGL(k_dctz2, dim3(a.nb + b.nb), dim3(std::max(p.nth, q.nth)), std::max(p.sh, q.sh), h->stream, a, b,
                     DctzTab{h->d_twz, h->d_twz + nz, h->d_ez, h->d_ez + nz}, nz, lz, dir);
}

template <typename TW> void launch_poisson(vrh_t *h, int irk, const double *ext_rhs, double *phi_out) {
  const VGrid &g = h->g;
  const int N = g.nt, logn = ilog2(N), nz = g.nz;
  const bool pow2 = (N & (N - 1)) == 0;
  const long nlines = (long)g.nr * nz, nl = (long)N * g.nr, nl64 = 5L * g.nr;
  TW *S = (TW *)h->f.S;
  double *S64 = (h->prec == VRH_MIXED) ? h->f.S64 : nullptr;
  const double adt = h->rk[irk].a * h->dt;
  // Lines per block: 16, or 8 of 256 angles (butterflies per thread of the LDS
  // FFT: (LB/2) N / rmin <= qt 256).  us forward/inverse with 4, 8, 16 lines:
  // mixed 128x256x512 289/124, 179/84, 150/68; FP64 255/124, 162/84, 144/79;
  // with 2, 4, 8 of mixed 256x512x1024 2310/1080, 1348/710, 1089/536.
  int LB = h->fft_lines > 0 ? h->fft_lines : 16;
  while (LB > 2 && (LB / 2) * N / fft_min_radix(logn) > 256 * fft_qt<TW>()) LB /= 2;
  // The low modes' sums run over 256 / LB lanes; the default keeps the order of
  // N / 4 lanes (of 1024 / N lines), two of whose sums a lane then holds
  // apart, so that the mixed path's results do not depend on LB.
  const bool split = S64 && h->fft_lines <= 0 && 2 * (256 / LB) == N / 4;
  const dim3 fgrd((unsigned)((nlines + LB - 1) / LB));
  {
    KTimer kt(h, KT_DIVFFT);
    if (pow2) {
      size_t sh = al16(sizeof(TW) * LB * N);
      if (S64) sh = al16(sh + sizeof(double) * (2 * (size_t)N + 10 * (size_t)LB));
      sh = al16(al16(sh + sizeof(TW) * N) + sizeof(int) * 2 * LB) + sizeof(double) * 2 * LB;
      hipLaunchKernelGGL((split ? k_divfft<TW, true> : k_divfft<TW, false>), fgrd, dim3(256), sh, h->stream, g, h->coef, h->zmet, 1.0 / adt, h->f.dq1,
                         h->f.dq2, h->f.dq3, ext_rhs, S, S64, h->d_twt, h->d_twt + N, LB, logn);
    } else {
      launch_divdft<TW>(h, 1.0 / adt, ext_rhs, S, S64);
    }
  }
  // The FP64 low-mode chain (mixed precision) reads only what the forward
  // theta transform wrote to S64 and feeds only the inverse one: it runs on
  // a side stream, forked and joined between them, beside the FP32
  // transforms.  With the kernel timer on, or inside an ensemble graph, it
  // stays in order on the handle's stream.
  // On grids of up to 14 MB a component (FP32) and 256 rows the two chains
  // share launches instead: three kernels instead of six with a fork and a
  // join, whose gaps took 14 us of a substep.  us a step, side by side ->
  // shared: 32x64x128 307 -> 267, 33x96x200 524 -> 477, 64x96x256 551 -> 521,
  // 100x128x200 1245 -> 1205, 64x128x400 1459 -> 1435, 64x192x256 even; the
  // FP32 lines then run with the FP64 kernel's registers, and 128x192x256
  // (25 MB) took 1642 instead of 1625.  A chosen width of the z
  // transforms is that of the FP32 lines in either form (tuned steps: 290 -> 256
  // at 32x64x128, 550 -> 518 at 64x96x256).  The kernel timer's entries are those
  // of the kernels alone.
  const bool pair = S64 && !h->kt_on && !h->zmet.m3 && radial_rows(g) == 16 && 4 * g.ncomp <= 14L << 20;
  const bool par = S64 && !pair && !h->kt_on && !h->serial_sweeps;
  hipStream_t s64 = par ? h->side[0] : h->stream;
  const int ie = (irk >= 1 && irk <= 3) ? irk : 0;
  if (par) {
    (void)hipEventRecord(h->poi_ev[ie][0], h->stream);
    (void)hipStreamWaitEvent(s64, h->poi_ev[ie][0], 0);
  }
  if (S64 && h->zmet.m3) {
    zgemm(h, s64, S64, h->S2_64, nl64, 1);
    radial_launch<double>(h, h->S2_64, h->f.ib64, 5, s64);
    zgemm(h, s64, h->S2_64, S64, nl64, -1);
  } else if (S64 && !pair) {
    z_transform<double>(h, s64, S64, nl64, 1, 0);
    radial_launch<double>(h, S64, h->f.ib64, 5, s64);
    z_transform<double>(h, s64, S64, nl64, -1, 0);
  }
  // per-mode iterative solve of the positions >= hz_pos0: stage their
  // right-hand sides before the direct path overwrites them
  const dim3 hzg((unsigned)((N - h->hz_pos0 + 63) / 64), (unsigned)((g.nr + 63) / 64), (unsigned)nz);
  if (h->hz)
    hipLaunchKernelGGL(k_hz_gather<TW>, hzg, dim3(256), 0, h->stream, S, hz_step_input(h->hz), N, g.nr, nz,
                       h->hz_pos0);
  bool done = false;
  if constexpr (sizeof(TW) == 4) {
    if (h->zmet.m3) {  // mixed path on an axial mesh: library GEMMs, out of place
      TW *S2 = (TW *)h->S2;
      { KTimer kt(h, KT_DCT_FWD); zgemm(h, h->stream, S, S2, nl, 1); }
      radial_launch<TW>(h, S2, (const TW *)h->f.ib, N, h->stream);
      { KTimer kt(h, KT_DCT_INV); zgemm(h, h->stream, S2, S, nl, -1); }
      done = true;
    } else if (pair) {
      z_transform2(h, S64, nl64, S, nl, 1);
      radial_launch2(h, S64, h->f.ib64, S, (const TW *)h->f.ib);
      z_transform2(h, S64, nl64, S, nl, -1);
      done = true;
    }
  }
  if (!done) {
    { KTimer kt(h, KT_DCT_FWD); z_transform<TW>(h, h->stream, S, nl, 1, h->dct_lines); }
    radial_launch<TW>(h, S, (const TW *)h->f.ib, N, h->stream);
    { KTimer kt(h, KT_DCT_INV); z_transform<TW>(h, h->stream, S, nl, -1, h->dct_lines); }
  }
  if (par) {
    (void)hipEventRecord(h->poi_ev[ie][1], s64);
    (void)hipStreamWaitEvent(h->stream, h->poi_ev[ie][1], 0);
  }
  if (h->hz) {
    if (!h->mode_rc) {
      const int rc = hz_step_solve(h->hz, h->stream, h->hz_method, h->hz_tol, h->hz_maxit, &h->hz_iters);
      if (rc) { h->mode_rc = rc; h->err = hz_error(h->hz); }
    }
    h->hz_solves++;
    hipLaunchKernelGGL(k_hz_scatter<TW>, hzg, dim3(256), 0, h->stream, hz_step_output(h->hz), S, N, g.nr, nz,
                       h->hz_pos0);
  }
  double *dph = ext_rhs ? nullptr : h->f.dph;
  KTimer kti(h, KT_IFFT);
  if (!pow2) { launch_idft<TW>(h, S, S64, phi_out, dph); return; }
  size_t sh3 = al16(sizeof(TW) * ((size_t)2 * LB * N + N)) + sizeof(int) * 2 * LB;
  if (S64) sh3 = al16(sh3) + sizeof(double) * (5 * (size_t)LB + 2 * (size_t)N);
  hipLaunchKernelGGL(k_ifft<TW>, fgrd, dim3(256), sh3, h->stream, g, S, S64, phi_out, dph, h->d_twt, h->d_twt + N, LB,
                     logn);
}

template <typename TW> void launch_project(vrh_t *h, int irk) {
  const VGrid &g = h->g;
  const double adt = h->rk[irk].a * h->dt;
  const double be = 0.5 * (h->rk[irk].a * h->dt) / h->Re;
  // Planes per block: 8 (a block re-reads three planes of phi, 2 % of its
  // bytes; its waves' first loads are exposed once per chunk), 4 up to 20 MB
  // a component, where 8 leave too few blocks.  us at 8 and 4 planes:
  // 32x64x128 18.4, 16.0; 64x128x256 60.0, 58.1 (tanh mesh 69, 63);
  // 129x128x128 79.6, 77.5; 200x96x160 92.1, 94.7; 128x192x256 149.1, 150.8;
  // 128x256x512 388, 406.
  // Tiles of 32 x 8 where they idle fewer lanes, up to 32 and from 65 to 96
  // angles: 64 x 4 against 32 x 8 take 18.8 and 16.0 at 32x64x128, 48.4 and
  // 44.4 at 96x64x256, but 73 and 82 at 129x128x128 and 65 and 72 at 100x96x200.
  const int W = g.nt <= 32 || (g.nt > 64 && g.nt <= 96) ? 32 : 64, R = 256 / W;
  const int kchunk = (long)sizeof(double) * g.ncomp <= (20L << 20) ? 4 : 8;
  // Neighbouring tiles on one XCD where rows are not whole 64-byte pieces, so
  // that the pieces two tiles share are joined in one L2: 77.5 -> 72.1 us at
  // 129x128x128, 65.2 -> 62.3 at 100x96x200, 225 -> 213 at 255x128x256.  Whole
  // pieces are better spread over all XCDs: 66.4 against 69.9 at 144x96x160.
  const int xcd = g.nt % 8 != 0;
  dim3 blk(W, R), grd((g.nt + W - 1) / W, (g.nrc + 1 + R - 1) / R, (g.nzc + kchunk - 1) / kchunk);
  KTimer kt(h, KT_PROJECT);
  auto kern = W == 64 ? (h->zmet.m3 ? k_project<64, 4, true> : k_project<64, 4, false>)
                      : (h->zmet.m3 ? k_project<32, 8, true> : k_project<32, 8, false>);
  hipLaunchKernelGGL(kern, grd, blk, 0, h->stream, g, h->coef, h->zmet, adt, be, kchunk, xcd, h->f.dph, h->f.dq1,
                     h->f.dq2, h->f.dq3, h->f.q1, h->f.q2, h->f.q3, h->f.prg1, h->f.prg2,
                     h->f.prg3, h->f.pres, h->f.flag);
}

void launch_analysis(vrh_t *h, double *part, int nblk, double *out) {
  hipLaunchKernelGGL(k_analysis, dim3(nblk), dim3(256), 0, h->stream, h->g, h->rmax, h->zmax, h->coef.rm, h->zmet.zpos, h->f.q1,
                     h->f.q2, h->f.q3, part);
  hipLaunchKernelGGL(k_analysis_sum, dim3(1), dim3(64), 0, h->stream, part, nblk, out);
}

// Block partials of the allocation-free analysis (vrh_analysis_noalloc):
// a file-scope device array, one copy per GPU, held until the process
// ends.  Host code never passes the array's name to a kernel (on the host
// it is only a stand-in for the symbol): each device's address is taken
// once, with that device current, by analysis_scratch_init, and used from
// then on.  Every block of k_analysis writes all ten of its partials, so
// the array needs no clearing between calls.
static __device__ __align__(256) double scratch[(size_t)kAnalysisBlocks * 10];
namespace {
std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices] = {};
}  // namespace

int analysis_scratch_init(int dev) {
  if (dev < 0 || dev >= kMaxDevices) return -1;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev]) return 0;
  void *p = nullptr;
  if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return -1;
  g_scratch_ptr[dev] = static_cast<double *>(p);
  return 0;
}

double *analysis_scratch(int dev) {
  if (dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  return g_scratch_ptr[dev];
}

#define INST(TW)                                                   \
  template void launch_explicit<TW>(vrh_t *, int);                 \
  template void launch_poisson<TW>(vrh_t *, int, const double *, double *); \
  template void launch_project<TW>(vrh_t *, int);
INST(double)
INST(float)
