// vrh_lines.hip -- the implicit r and z sweeps of the substep, and hdnbc's
// outlet rows, which only the q3 z sweep reads.
#include <hip/hip_runtime.h>

#include "vrh_internal.h"

namespace {

// ---------------------------------------------------------------------------
// hdnbc: outlet convective condition and mass correction, one thread per
// (theta, r) outlet point (momentum_terms_swirl.F90:225-291).  zm3n: the
// outlet cell's z difference dx3/dmz(nz) on an axial mesh, dx3 on the uniform
// one.
// ---------------------------------------------------------------------------
struct HdnbcArgs {
  VGrid g;
  const double *qc;
  double zm3n, gam, rom, cor;
  const double *cor_dev;  // the mass correction read from the device, or null
  const double *q3;
  double *csort, *dq3no, *corr3n;
};
__device__ __forceinline__ void hdnbc_point(const HdnbcArgs &a, int i, int j) {  // i = 1..nt, j = 1..nrc
#pragma clang fp contract(off)
  const VGrid &g = a.g;
  const double cor = a.cor_dev ? *a.cor_dev : a.cor;
  const long p = (long)(i - 1) + (long)g.nt * j;
  const double qn = a.q3[hidx(g, i, j, g.nzc)], qm = a.q3[hidx(g, i, j, g.nz)];
  double cs = a.csort[p];
  if (j <= g.nr && qn > 0.0) cs = (double)0.6f * qn;
  a.csort[p] = cs;
  const double tconv = -(cs * a.zm3n) * (qn - qm);
  const double c3n = __builtin_fma(a.rom, a.dq3no[p], a.gam * tconv) * g.dt;
  a.dq3no[p] = tconv;
  a.corr3n[p] = __builtin_fma(a.qc[j], cor, c3n);
}
__global__ __launch_bounds__(64) void k_hdnbc(HdnbcArgs a) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x + 1;
  if (i <= a.g.nt) hdnbc_point(a, i, blockIdx.y + 1);
}

// ---------------------------------------------------------------------------
// Partitioned Thomas solve of the r and z sweeps (solqj/solqk with
// solve_lap_par/solve_lap_thom, step.F90:266-485; tripar.F90:11-145).
// A block owns 64 lines (one per lane, consecutive theta -> coalesced) and P
// waves; wave s owns positions [s*M, s*M+M) of every line and keeps them in
// registers.  The two linear recurrences of the Thomas algorithm are closed
// across segments with precomputed carry products (one LDS exchange each).
// ---------------------------------------------------------------------------
// what a sweep does with its right-hand sides and its solution: solved in
// place; the z sweeps of q1 and q3 (dq = q + x); the r sweep of q2 (dq2)
enum SweepKind { SK_PLACE = 0, SK_Z = 1, SK_R2 = 2 };
struct LineArgs {
  LineCoef lc;
  int nlines, M;
  bool along_z;                // lines along z (position stride sk), else along r
  int j0;                      // first r index of z lines
  bool zero_ends;              // right-hand sides 0 at both ends (q1, q2 z sweeps and the q2 r sweep)
  bool q3_ends;                // inlet and outlet values at the ends (q3 z sweep)
  const double *q;             // state component (SK_Z, SK_R2)
  double *dq;                  // predictor output (SK_Z, SK_R2)
  void *r;                     // qrhs of the component (TW)
};
struct SweepArgs {
  VGrid g;
  double slip;
  const double *corr3n;        // outlet row of the q3 z sweep
  double c3s;                  // inlet row value of the q3 z sweep (uniform in theta)
  const double *c3s_dev;       // same value read from the device (captured steps), or null
  int jlim;                    // inlet rows: j <= jlim
};

// Lines blk * 64 + lane of a sweep by waves 0..P-1 (further waves of the
// block only meet the barriers).
template <typename TW, int M, int KIND>
__device__ __forceinline__ void line_solve(const SweepArgs &sa, const LineArgs &a, int blk, TW (&sh_a)[16][64]) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const VGrid &g = sa.g;
  const int n = a.lc.n, P = a.lc.P;
  if (s >= P) {
    __syncthreads();
    __syncthreads();
    __syncthreads();
    return;
  }
  const int L = blk * 64 + lane;
  const bool act = L < a.nlines;
  const int Lc = act ? L : a.nlines - 1;  // addresses stay in bounds; results of !act lanes are dropped
  const int p0 = s * M;
  const int len = min(M, n - p0);
  TW *rr = reinterpret_cast<TW *>(a.r);
  // the coefficients in the work type (the mixed path's float copies)
  auto cw = [](const double *d, const float *f) {
    if constexpr (sizeof(TW) == 4) { (void)d; return f; } else { (void)f; return d; }
  };
  const TW *cA = cw(a.lc.A, a.lc.Af), *cB = cw(a.lc.B, a.lc.Bf), *cC = cw(a.lc.C, a.lc.Cf);
  const TW *cPk = cw(a.lc.Pk, a.lc.Pkf), *cQk = cw(a.lc.Qk, a.lc.Qkf);
  const TW *cPs = cw(a.lc.Pseg, a.lc.Psegf), *cQs = cw(a.lc.Qseg, a.lc.Qsegf);
  auto fma_ = [](TW x, TW y, TW z) {
    if constexpr (sizeof(TW) == 4) return __builtin_fmaf(x, y, z); else return __builtin_fma(x, y, z);
  };
  // line -> (i, second index)
  const int l2 = Lc / g.nt, i = Lc - l2 * g.nt + 1;
  const int jz = l2 + a.j0;
  const long base = a.along_z ? hidx(g, i, jz, 1) : hidx(g, i, 1, l2 + 1);  // address of position 0
  const long step = a.along_z ? g.sk : g.sj;
  // every load of the segment is issued before the first use (positions
  // beyond the line clamp to its last one and are masked afterwards)
  TW x[M];
#pragma unroll
  for (int t = 0; t < M; ++t) x[t] = rr[base + step * min(p0 + t, n - 1)];
  TW first = (TW)0, rlast = (TW)0;
  if (KIND == SK_Z && a.q3_ends) {
    rlast = (TW)sa.corr3n[(long)(i - 1) + (long)g.nt * jz];
    first = (jz <= sa.jlim) ? (TW)(sa.c3s_dev ? *sa.c3s_dev : sa.c3s) : (TW)0;
  }
  const bool ends = a.zero_ends || a.q3_ends;
  __builtin_amdgcn_sched_barrier(0);
  TW gp = (TW)0;
#pragma unroll
  for (int t = 0; t < M; ++t) {
    const int p = p0 + t;
    TW rv = x[t];
    if (ends && p == 0) rv = first;
    if (ends && p == n - 1) rv = rlast;
    const TW v = fma_(cA[p], rv, cB[p] * gp);
    const bool in = t < len;
    x[t] = in ? v : (TW)0;
    gp = in ? v : gp;
  }
  sh_a[s][lane] = gp;
  __syncthreads();
  TW G = (TW)0;
  for (int s2 = 0; s2 < s; ++s2) G = fma_(cPs[s2], G, sh_a[s2][lane]);
  __syncthreads();
  TW xp = (TW)0;
#pragma unroll
  for (int t = M - 1; t >= 0; --t) {
    const int p = p0 + t;
    const TW v = fma_(-cC[p], xp, fma_(cPk[p], G, x[t]));
    const bool in = t < len;
    x[t] = in ? v : x[t];
    xp = in ? v : xp;
  }
  sh_a[s][lane] = xp;
  __syncthreads();
  TW X = (TW)0;
  for (int s2 = P - 1; s2 > s; --s2) X = fma_(cQs[s2], X, sh_a[s2][lane]);
#pragma unroll
  for (int t = 0; t < M; ++t) x[t] = fma_(cQk[p0 + t], X, x[t]);
  if (KIND == SK_PLACE) {
    if (!act) return;
#pragma unroll
    for (int t = 0; t < M; ++t)
      if (t < len) rr[base + step * (p0 + t)] = x[t];
  } else {
    auto put = [&](int t, double qv) {
      const int p = p0 + t;
      const long ad = base + step * p;
      if (KIND == SK_R2) {
        // dq2 = x + q2 for j = 1..nr; dq2(nrc) = 0 (step.F90:330-333, 183-187)
        a.dq[ad] = (p == n - 1) ? 0.0 : (double)x[t] + qv;
      } else {
        // dq = q + x for k = 1..nzc; slip row at nrc (step.F90:84-88, 133-138)
        const double d = qv + (double)x[t];
        a.dq[ad] = d;
        if (jz == g.nr) a.dq[ad + g.sj] = sa.slip * d;
      }
    };
    // in chunks of 8 positions whose q loads go out together before their stores
    constexpr int CH = 8;
#pragma unroll
    for (int c0 = 0; c0 < M; c0 += CH) {
      double qv[CH];
#pragma unroll
      for (int u = 0; u < CH; ++u)
        qv[u] = (c0 + u < M) ? a.q[base + step * min(p0 + c0 + u, n - 1)] : 0.0;
      __builtin_amdgcn_sched_barrier(0);
      if (act) {
#pragma unroll
        for (int u = 0; u < CH; ++u)
          if (c0 + u < M && c0 + u < len) put(c0 + u, qv[u]);
      }
    }
  }
}

template <typename TW, int M, int KIND>
__global__ __attribute__((amdgpu_flat_work_group_size(64, 1024), amdgpu_waves_per_eu(1, 4))) void k_line(SweepArgs sa,
                                                                                                       LineArgs a) {
  __shared__ TW sh_a[16][64];
  line_solve<TW, M, KIND>(sa, a, (int)blockIdx.x, sh_a);
}

// Three sweeps in one launch: blocks [0, b1) take a[0], [b1, b2) a[1], [b2, b3)
// a[2], the rest hdnbc's outlet points (first launch only).  PHASE 0: the z
// sweep of q2 and the r sweeps of q1 and q3; PHASE 1: the z sweeps of q1 and
// q3 and the r sweep of q2.  MR, MZ: the segments of the r and z sweeps.
// The grid is one block per 64 lines of any of the three, so short sweeps
// fill the chip together without a fork and a join of streams; all blocks
// have the waves of the longest line.
struct SweepGroup {
  SweepArgs s;
  LineArgs a[3];
  int b1, b2, b3;
  HdnbcArgs hd;
};
template <typename TW, int PHASE, int MR, int MZ>
__global__ __attribute__((amdgpu_flat_work_group_size(64, 1024), amdgpu_waves_per_eu(1, 4))) void k_sweeps(SweepGroup w) {
  __shared__ TW sh[16][64];
  const int b = (int)blockIdx.x;
  if (PHASE == 0) {
    if (b < w.b1) {
      line_solve<TW, MZ, SK_PLACE>(w.s, w.a[0], b, sh);
    } else if (b < w.b3) {
      line_solve<TW, MR, SK_PLACE>(w.s, w.a[b < w.b2 ? 1 : 2], b - (b < w.b2 ? w.b1 : w.b2), sh);
    } else {
      const VGrid &g = w.s.g;
      const int e = (b - w.b3) * (int)blockDim.x + (int)threadIdx.x, j = e / g.nt;
      if (j < g.nrc) hdnbc_point(w.hd, e - j * g.nt + 1, j + 1);
    }
  } else {
    if (b < w.b2) line_solve<TW, MZ, SK_Z>(w.s, w.a[b < w.b1 ? 0 : 1], b < w.b1 ? b : b - w.b1, sh);
    else line_solve<TW, MR, SK_R2>(w.s, w.a[2], b - w.b2, sh);
  }
}

HdnbcArgs hdnbc_args(vrh_t *h, int irk, double cor, const double *cor_dev) {
  const VGrid &g = h->g;
  return HdnbcArgs{g, h->coef.qc, h->zmesh[2].empty() ? g.dx3 : g.dx3 / h->zmesh[2][g.nz], h->rk[irk].g, h->rk[irk].r,
                   cor, cor_dev, h->f.q3, h->f.csort, h->f.dq3no, h->f.corr3n};
}
void hdnbc_on(vrh_t *h, int irk, double cor, const double *cor_dev, hipStream_t st) {
  dim3 blk(64), grd((h->nt + 63) / 64, h->nrc);
  KTimer kt(h, KT_HDNBC);
  hipLaunchKernelGGL(k_hdnbc, grd, blk, 0, st, hdnbc_args(h, irk, cor, cor_dev));
}

template <typename TW, int KIND> void line_launch(vrh_t *h, const SweepArgs &s, const LineArgs &a, hipStream_t st) {
  dim3 blk(64 * a.lc.P), grd((unsigned)((a.nlines + 63) / 64));
  KTimer kt(h, a.along_z ? KT_LINE_Z : KT_LINE_R);
  switch (a.M) {
    case 16: hipLaunchKernelGGL((k_line<TW, 16, KIND>), grd, blk, 0, st, s, a); break;
    case 24: hipLaunchKernelGGL((k_line<TW, 24, KIND>), grd, blk, 0, st, s, a); break;
    case 32: hipLaunchKernelGGL((k_line<TW, 32, KIND>), grd, blk, 0, st, s, a); break;
    case 40: hipLaunchKernelGGL((k_line<TW, 40, KIND>), grd, blk, 0, st, s, a); break;
    case 48: hipLaunchKernelGGL((k_line<TW, 48, KIND>), grd, blk, 0, st, s, a); break;
    case 72: hipLaunchKernelGGL((k_line<TW, 72, KIND>), grd, blk, 0, st, s, a); break;
    default: hipLaunchKernelGGL((k_line<TW, 64, KIND>), grd, blk, 0, st, s, a); break;
  }
}

// The segments that the grouped kernels are built for.  40 (z lines of 385 to
// 400 and 513 to 520 points) only in FP32: in FP64 the grouped kernel spills
// and the single sweeps are faster (600 us a step grouped, 525 alone at
// 24x48x512; FP32 at 32x64x512 takes 547 and 593).
template <typename TW> bool group_has(int mr, int mz) {
  return (mr == 16 || mr == 24) && (mz == 16 || mz == 24 || (mz == 40 && sizeof(TW) == 4));
}
template <typename TW, int PHASE> void group_launch(vrh_t *h, SweepGroup &w, int mr, int mz, bool hdnbc) {
  const VGrid &g = h->g;
  int P = 1;
  for (const LineArgs &a : w.a) P = a.lc.P > P ? a.lc.P : P;
  auto nb = [](const LineArgs &a) { return (a.nlines + 63) / 64; };
  w.b1 = nb(w.a[0]);
  w.b2 = w.b1 + nb(w.a[1]);
  w.b3 = w.b2 + nb(w.a[2]);
  const int hb = hdnbc ? (g.nt * g.nrc + 64 * P - 1) / (64 * P) : 0;
  const dim3 grd((unsigned)(w.b3 + hb)), blk(64 * P);
  auto go = [&](auto *kern) { hipLaunchKernelGGL(kern, grd, blk, 0, h->stream, w); };
  if (mr == 16 && mz == 16) go(k_sweeps<TW, PHASE, 16, 16>);
  else if (mr == 16 && mz == 24) go(k_sweeps<TW, PHASE, 16, 24>);
  else if (mr == 24 && mz == 16) go(k_sweeps<TW, PHASE, 24, 16>);
  else if (mr == 24 && mz == 24) go(k_sweeps<TW, PHASE, 24, 24>);
  else if constexpr (sizeof(TW) == 4) {
    if (mr == 16) go(k_sweeps<TW, PHASE, 16, 40>);
    else go(k_sweeps<TW, PHASE, 24, 40>);
  }
}

}  // namespace

template <typename TW> void launch_hdnbc(vrh_t *h, int irk, double cor, const double *cor_dev) {
  hdnbc_on(h, irk, cor, cor_dev, h->stream);
}

template <typename TW> void launch_sweeps(vrh_t *h, int irk, double c3s, const double *c3s_dev, bool hdnbc,
                                          double cor, const double *cor_dev) {
  const VGrid &g = h->g;
  const SweepArgs s{g, h->slip, h->f.corr3n, c3s, c3s_dev, h->jlim};
  const int nt = g.nt;
  auto line = [&](int sw, bool along_z, int nlines, int j0, bool zero_ends, bool q3_ends, const double *q, double *dq,
                  void *r) {
    return LineArgs{h->lc[irk][sw], nlines, h->Msw[sw], along_z, j0, zero_ends, q3_ends, q, dq, r};
  };
  // q1: r then z (step.F90:75-78); q3: r then z (step.F90:124-127); q2: z then r (step.F90:171-177)
  const LineArgs r1 = line(SW_R1, false, nt * g.nz, 0, false, false, nullptr, nullptr, h->f.r1),
                 z1 = line(SW_Z1, true, nt * g.nr, 1, true, false, h->f.q1, h->f.dq1, h->f.r1),
                 r3 = line(SW_R3, false, nt * g.nz, 0, false, false, nullptr, nullptr, h->f.r3),
                 z3 = line(SW_Z3, true, nt * g.nr, 1, false, true, h->f.q3, h->f.dq3, h->f.r3),
                 z2 = line(SW_Z2, true, nt * (g.nr - 1), 2, true, false, nullptr, nullptr, h->f.r2),
                 r2 = line(SW_R2, false, nt * g.nzc, 0, true, false, h->f.q2, h->f.dq2, h->f.r2);
  const int mr = h->Msw[SW_R1], mr2 = h->Msw[SW_R2], mz = h->Msw[SW_Z1];
  // Grouped while a component of the work arrays is at most 14 MB, where the
  // step is a chain of short kernels and six launches with a fork and a join
  // of two streams cost more than their work: a whole step takes, alone ->
  // grouped, 351 -> 286 us at 32x64x128 FP64, 623 -> 549 at 33x96x200 mixed,
  // 668 -> 643 at 64x96x256 FP64, 725 -> 712 at 64x128x256 mixed, 1102 -> 1085
  // at 128x128x192 mixed.  Beyond it the single sweeps' fewer registers (7
  // waves a SIMD against 4) win: 1021 -> 1052 at 96x96x200 FP64 (15 MB), 1183
  // -> 1224 at 129x128x128 FP64; 128x192x256 is even in both precisions.
  // The kernel timer's entries are those of the kernels alone.
  if (!h->kt_on && (long)sizeof(TW) * g.ncomp <= (14L << 20) && h->Msw[SW_R3] == mr && h->Msw[SW_Z2] == mz && h->Msw[SW_Z3] == mz &&
      group_has<TW>(mr, mz) && group_has<TW>(mr2, mz)) {
    SweepGroup w{s, {z2, r1, r3}, 0, 0, 0, hdnbc_args(h, irk, cor, cor_dev)};
    SweepGroup v{s, {z1, z3, r2}, 0, 0, 0, w.hd};
    group_launch<TW, 0>(h, w, mr, mz, hdnbc);
    group_launch<TW, 1>(h, v, mr2, mz, false);
    return;
  }
  // The three components' chains are independent: q3 and q2 run on the
  // side streams, forked from and joined back into the handle's stream
  // (captured steps record the fork as graph branches).  With the kernel
  // timer on, and inside an ensemble graph (whose members already run side
  // by side), all run in order on the handle's stream.
  const bool par = !h->kt_on && !h->serial_sweeps;
  hipStream_t s1 = par ? h->side[0] : h->stream, s2 = par ? h->side[1] : h->stream;
  const int ie = (irk >= 1 && irk <= 3) ? irk : 0;
  if (par) {
    (void)hipEventRecord(h->fork_ev[ie], h->stream);
    (void)hipStreamWaitEvent(s1, h->fork_ev[ie], 0);
    (void)hipStreamWaitEvent(s2, h->fork_ev[ie], 0);
  }
  line_launch<TW, SK_PLACE>(h, s, r1, h->stream);
  line_launch<TW, SK_Z>(h, s, z1, h->stream);
  // In a whole step the outlet rows of hdnbc (csort, dq3no, corr3n: read
  // only by the q3 z sweep; computed from q3, which the explicit kernel
  // leaves alone) head this chain, off the critical path.
  if (hdnbc) hdnbc_on(h, irk, cor, cor_dev, s1);
  line_launch<TW, SK_PLACE>(h, s, r3, s1);
  line_launch<TW, SK_Z>(h, s, z3, s1);
  line_launch<TW, SK_PLACE>(h, s, z2, s2);
  line_launch<TW, SK_R2>(h, s, r2, s2);
  if (par) {
    (void)hipEventRecord(h->join_ev[ie][0], s1);
    (void)hipEventRecord(h->join_ev[ie][1], s2);
    (void)hipStreamWaitEvent(h->stream, h->join_ev[ie][0], 0);
    (void)hipStreamWaitEvent(h->stream, h->join_ev[ie][1], 0);
  }
}

#define INST(TW)                                                        \
  template void launch_hdnbc<TW>(vrh_t *, int, double, const double *); \
  template void launch_sweeps<TW>(vrh_t *, int, double, const double *, bool, double, const double *);
INST(double)
INST(float)
