// vrh_dense.hip -- the pressure solve's transforms as dense sums: the z cosine
// and the theta transforms of lengths that are no power of two, and the FP64
// z eigen-transforms of an axial mesh.
//
// All but the inverse theta transform run on the FP64 matrix cores.
// v_mfma_f64_16x16x4: lane l holds A(l % 16, l / 16), B(l / 16, l % 16) and
// D(4 v + l / 16, l % 16), v = 0..3, and every element of D is the chain of
// fused multiply-adds over ascending k, so a product equals the plain
// sequential sum bit for bit.  The sums keep the definition's order (no
// folding by parity) because of that: the mixed path's FP32 roundings spread a
// change in the last bit of any input over the whole field.  The matrices
// are packed in the order in which the lanes read them, so that a wave's A
// operand is one contiguous 512-byte load from L2.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "vrh_internal.h"

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

// Column steps of A whose loads are in flight at once: a wave loads the next
// group while the matrix cores work on this one (8 steps are 512 cycles of
// them).  With it and 32 lines per block a z transform of 64x128x256 takes
// 34 us (55 before; rocBLAS dgemm 37; 15 at the FP64 matrix rate) and the
// forward theta transform of 129x128x128 38 (61 before).  The packed matrices
// are padded to whole groups.
constexpr int kGrp = 8;

// ---------------------------------------------------------------------------
// z transforms, in place.  A block holds TN = 16 NT lines (consecutive in
// memory) whole in LDS as x[row][line]; every wave forms 16-row tiles of the
// result from them and stores straight to global memory, divided by `div`.
// Rows past the end of the K range meet zero columns of A; they are clamped
// to the line's last row, so nothing outside the line enters.  33x96x200:
// 18 us a transform, where a direct sum with a cosine per term took 460.
// ---------------------------------------------------------------------------
template <typename TW, int NT>
__device__ __forceinline__ void zdense_block(unsigned blk, double *x, TW *__restrict__ S, long nl, int n, const DenseMat &m,
                                             double div) {
  constexpr int TN = 16 * NT, NTH = 512, RS = NTH / TN;  // RS rows per pass of the block
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long l0 = (long)blk * TN;
  {
    const int c = tid % TN, r0 = tid / TN;
    const TW *src = S + min(l0 + c, nl - 1);
    constexpr int U = 8;
    for (int rb = r0; rb < n; rb += U * RS) {
      TW v[U];
#pragma unroll
      for (int u = 0; u < U; u++) v[u] = src[nl * min(rb + u * RS, n - 1)];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; u++)
        if (rb + u * RS < n) x[(rb + u * RS) * TN + c] = (double)v[u];
    }
  }
  __syncthreads();
  const int kq = lane >> 4, c = lane & 15;
  for (int t = wave; t < m.mt; t += NTH / 64) {
    d4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) acc[j] = d4{0.0, 0.0, 0.0, 0.0};
    const double *ap = m.a + (size_t)t * m.ks * 64 + lane;
    double cur[kGrp], nxt[kGrp];
#pragma unroll
    for (int s = 0; s < kGrp; s++) cur[s] = ap[s * 64];
    for (int s0 = 0; s0 < m.ks; s0 += kGrp) {
      const double *np = ap + min(s0 + kGrp, m.ks - kGrp) * 64;
#pragma unroll
      for (int s = 0; s < kGrp; s++) nxt[s] = np[s * 64];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < kGrp; s++) {
        const int row = min(4 * (s0 + s) + kq, n - 1);
#pragma unroll
        for (int j = 0; j < NT; j++)
          acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(cur[s], x[row * TN + j * 16 + c], acc[j], 0, 0, 0);
      }
#pragma unroll
      for (int s = 0; s < kGrp; s++) cur[s] = nxt[s];
    }
#pragma unroll
    for (int j = 0; j < NT; j++) {
      const long l = l0 + j * 16 + c;
      if (l >= nl) continue;
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int q = t * 16 + 4 * v + kq;
        if (q < n) S[l + nl * q] = (TW)(acc[j][v] / div);
      }
    }
  }
}

template <typename TW, int NT>
__global__ __launch_bounds__(512) void k_zdense(TW *__restrict__ S, long nl, int n, DenseMat m, double div) {
  extern __shared__ double x[];
  zdense_block<TW, NT>(blockIdx.x, x, S, nl, n, m, div);
}
// the mixed path's FP64 low modes (first na blocks) and its FP32 lines
template <int NT>
__global__ __launch_bounds__(512) void k_zdense2(double *__restrict__ S64, long nl64, unsigned na, float *__restrict__ S,
                                                 long nl, int n, DenseMat m, double div) {
  extern __shared__ double x[];
  if (blockIdx.x < na) zdense_block<double, 1>(blockIdx.x, x, S64, nl64, n, m, div);
  else zdense_block<float, NT>(blockIdx.x - na, x, S, nl, n, m, div);
}

// ---------------------------------------------------------------------------
// divq (divergence.F90:31-41) and fft_ptf_multi's packing
// (fastfouriertransform.F90:39-43) for ntheta no power of two: t(1) = F0/N,
// t(2k) = 2 Re Fk/N, t(2k+1) = -2 Im Fk/N.  32 lines per block in LDS as
// x[line][theta] (odd stride: the 16 lines of an operand read hit different
// banks), the rows of A in the packed order; the 16 x 16 tiles of the result
// (two halves of the lines for each 16 rows) are dealt to eight waves.
// 129x128x128: 38 us, 374 with the sums on the vector units from L1 (20 at
// the copy rate).  The mixed path's FP64 low modes
// (positions 0..4) are summed over virtual lanes ii mod 128, then by halves
// within 64 and over the two groups of 64.
// ---------------------------------------------------------------------------
constexpr int kThLines = 32, kThThreads = 16 * kThLines, kThWaves = kThThreads / 64;

template <typename TW>
__global__ __launch_bounds__(kThThreads) void k_divdft(VGrid g, VCoef c, ZMet zm, double inv_adt, const double *__restrict__ dq1,
                                                const double *__restrict__ dq2, const double *__restrict__ dq3,
                                                const double *__restrict__ ext, TW *__restrict__ S,
                                                double *__restrict__ S64, const double *__restrict__ tw, DenseMat m) {
  extern __shared__ double x[];
  const int N = g.nt, ldn = N | 1, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long nlines = (long)g.nr * g.nz, l0 = (long)blockIdx.x * kThLines;
  // 16 lanes per line, all lines at once
  const int lp = tid >> 4, tl = tid & 15;
  const long l = l0 + lp, lc = min(l, nlines - 1);
  {
    const int j = (int)(lc % g.nr) + 1, k = (int)(lc / g.nr) + 1;
    if (ext) {
      for (int ii = tl; ii < N; ii += 16) x[lp * ldn + ii] = ext[cidx(g, ii + 1, j, k)];
    } else {
      const double rmv = 1.0 / c.rm[j], rdv = g.dx2 / c.dmr[j];
      const double zkv = zm.m3 ? zm.m3[k] : g.dx3;  // dx3, or the axial mesh's 1/width of plane k
      const long ob = hidx(g, 1, j, k);
      constexpr int U = 4;
      for (int ub = tl; ub < N; ub += 16 * U) {
        double a1[U], b1[U], a2[U], b2[U], a3[U], b3[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int i = min(ub + 16 * u, N - 1);
          const long p = ob + i;
          a1[u] = dq1[p];
          b1[u] = dq1[p + (i == N - 1 ? 1 - N : 1)];
          a2[u] = dq2[p];
          b2[u] = dq2[p + g.sj];
          a3[u] = dq3[p];
          b3[u] = dq3[p + g.sk];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (ub + 16 * u < N)
            x[lp * ldn + ub + 16 * u] = divq_rhs(b1[u] - a1[u], g.dx1 * g.axsym, b2[u] - a2[u], rdv, rmv,
                                                 b3[u] - a3[u], zkv, inv_adt);
      }
    }
  }
  __syncthreads();
  if (S64) {
    double acc[5];
#pragma unroll
    for (int half = 0; half < 2; half++) {
      double s[4][5];  // virtual lanes tl + 16 q of this group of 64
#pragma unroll
      for (int q = 0; q < 4; q++) {
#pragma unroll
        for (int w = 0; w < 5; w++) s[q][w] = 0.0;
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const int ii = 64 * half + tl + 16 * q + 128 * u;
          if (ii < N) {
            const double val = x[lp * ldn + ii];
            int q2 = 2 * ii;
            if (q2 >= N) q2 -= N;
            s[q][0] += val;
            s[q][1] += val * tw[ii];
            s[q][2] += val * tw[N + ii];
            s[q][3] += val * tw[q2];
            s[q][4] += val * tw[N + q2];
          }
        }
      }
#pragma unroll
      for (int w = 0; w < 5; w++) {
        double v = (s[0][w] + s[2][w]) + (s[1][w] + s[3][w]);
        for (int o = 8; o > 0; o >>= 1) v += __shfl_xor(v, o, 16);
        acc[w] = half == 0 ? v : acc[w] + v;
      }
    }
    if (tl == 0 && l < nlines) {
#pragma unroll
      for (int w = 0; w < 5; w++)
        if (w < N) S64[(size_t)w + 5 * l] = (w == 0) ? acc[w] / N : 2.0 * acc[w] / N;
    }
  }
  constexpr int TPW = 4;  // N < 256: at most 2 x 16 tiles on eight waves
  d4 acc[TPW];
  const int kq = lane >> 4;
#pragma unroll
  for (int u = 0; u < TPW; u++) {
    acc[u] = d4{0.0, 0.0, 0.0, 0.0};
    const int t = wave + kThWaves * u;  // rows t / 2, lines of half t % 2
    if (t >= 2 * m.mt) continue;
    const double *ap = m.a + (size_t)(t >> 1) * m.ks * 64 + lane;
    const double *xl = x + ((t & 1) * 16 + (lane & 15)) * ldn;
    double cur[kGrp], nxt[kGrp];
#pragma unroll
    for (int s = 0; s < kGrp; s++) cur[s] = ap[s * 64];
    for (int s0 = 0; s0 < m.ks; s0 += kGrp) {
      const double *np = ap + min(s0 + kGrp, m.ks - kGrp) * 64;
#pragma unroll
      for (int s = 0; s < kGrp; s++) nxt[s] = np[s * 64];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < kGrp; s++)
        acc[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(cur[s], xl[min(4 * (s0 + s) + kq, N - 1)], acc[u], 0, 0, 0);
#pragma unroll
      for (int s = 0; s < kGrp; s++) cur[s] = nxt[s];
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < TPW; u++) {
    const int t = wave + kThWaves * u;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int pos = (t >> 1) * 16 + 4 * v + kq;
      if (pos < N)
        x[((t & 1) * 16 + (lane & 15)) * ldn + pos] = (pos == 0 ? acc[u][v] : 2.0 * acc[u][v]) / N;
    }
  }
  __syncthreads();
  if (l >= nlines) return;
  for (int pos = tl; pos < N; pos += 16) S[(size_t)pos + (size_t)N * l] = (TW)x[lp * ldn + pos];
}

// ---------------------------------------------------------------------------
// fft_ftp_multi (fastfouriertransform.F90:74-82), the copy into dph
// (poisson_solve.F90:29) and dph(nzc) = dph(nz) (divergence.F90:93-99) for
// ntheta no power of two, mixed path.  One lane per line (64 lines per block in LDS, odd
// stride), kIdT angles per wave at a time: a coefficient pair read from LDS
// serves kIdT angles, and the cosines and sines, the same for all lanes, come
// as scalar loads from a table in their order of use.  A term is
// v + (a cos + b sin): three FP64 instructions, whose rate (10 us at
// 129x128x128) and the latency of the loads bound the kernel: 45 us there, 248
// with a thread per angle and line and its table reads from L1.
// The low modes of the mixed path are added last, from S64.
// ---------------------------------------------------------------------------
// v + (a c + b s) with the inner sum fused the one way, whatever the code around it
__device__ __forceinline__ double id_term(double v, double a, double c, double b, double s) {
#pragma clang fp contract(off)
  return v + __builtin_fma(a, c, b * s);
}

constexpr int kIdLines = 64, kIdT = 4, kIdWaves = 16;

__global__ __launch_bounds__(64 * kIdWaves) void k_idft(VGrid g, const float *__restrict__ S,
                                                        const double *__restrict__ S64, double *__restrict__ phi_out,
                                                        double *__restrict__ dph, const double *__restrict__ tab) {
  extern __shared__ double x[];
  const int N = g.nt, ldn = N | 1, nk = N / 2, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long nlines = (long)g.nr * g.nz, l0 = (long)blockIdx.x * kIdLines;
  const int nln = (int)min((long)kIdLines, nlines - l0), tot = nln * N;
  constexpr int NTH = 64 * kIdWaves;
  {
    // the block's lines are contiguous in S; (line, position) advances by NTH
    const float *src = S + (size_t)N * l0;
    const int dl = NTH / N, dp = NTH - dl * N;
    constexpr int U = 8;
    int lp = tid / N, pos = tid - lp * N;
    for (int eb = tid; eb < tot; eb += U * NTH) {
      float v[U];
#pragma unroll
      for (int u = 0; u < U; u++) v[u] = src[min(eb + u * NTH, tot - 1)];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; u++) {
        if (eb + u * NTH < tot) x[lp * ldn + pos] = (S64 && pos < 5) ? 0.0 : (double)v[u];
        lp += dl;
        pos += dp;
        if (pos >= N) { pos -= N; lp++; }
      }
    }
  }
  __syncthreads();
  const double *t = x + min(lane, nln - 1) * ldn;
  const int ntile = (N + kIdT - 1) / kIdT;
  constexpr int TPW = 4;  // N < 256: at most 64 tiles on sixteen waves
  double v[TPW][kIdT];
#pragma unroll
  for (int q = 0; q < TPW; q++) {
    const int tile = wave + kIdWaves * q;
    if (tile >= ntile) continue;
    const double *tt = tab + (size_t)tile * nk * 2 * kIdT;
    const double v0 = t[0];
#pragma unroll
    for (int i = 0; i < kIdT; i++) v[q][i] = v0;
    for (int kk = 1; 2 * kk < N; ++kk) {
      const double a = t[2 * kk - 1], b = t[2 * kk];
      const double *w = tt + (size_t)(kk - 1) * 2 * kIdT;
#pragma unroll
      for (int i = 0; i < kIdT; i++) v[q][i] = id_term(v[q][i], a, w[i], b, w[kIdT + i]);
    }
    if (2 * nk == N) {
      const double a = t[N - 1];
      const double *w = tt + (size_t)(nk - 1) * 2 * kIdT;
#pragma unroll
      for (int i = 0; i < kIdT; i++) v[q][i] += 0.5 * a * w[i];
    }
    if (S64) {
      const double *s = S64 + 5 * min(l0 + lane, nlines - 1);
      const double s0 = s[0];
#pragma unroll
      for (int i = 0; i < kIdT; i++) v[q][i] += s0;
#pragma unroll
      for (int kk = 1; kk <= 2; ++kk) {
        if (2 * kk - 1 >= N) break;
        const double a = s[2 * kk - 1], b = (2 * kk < N) ? s[2 * kk] : 0.0;
        const double *w = tt + (size_t)(kk - 1) * 2 * kIdT;
#pragma unroll
        for (int i = 0; i < kIdT; i++) v[q][i] = id_term(v[q][i], a, w[i], b, w[kIdT + i]);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < TPW; q++) {
    const int tile = wave + kIdWaves * q;
    if (tile >= ntile || lane >= nln) continue;
#pragma unroll
    for (int i = 0; i < kIdT; i++)
      if (tile * kIdT + i < N) x[lane * ldn + tile * kIdT + i] = v[q][i];
  }
  __syncthreads();
  // a wave per line
  for (int lp = wave; lp < nln; lp += kIdWaves) {
    const long l = l0 + lp;
    const int j = (int)(l % g.nr) + 1, k = (int)(l / g.nr) + 1;
    for (int ii = lane; ii < N; ii += 64) {
      const double y = x[lp * ldn + ii];
      if (phi_out) phi_out[cidx(g, ii + 1, j, k)] = y;
      if (dph) {
        dph[hidx(g, ii + 1, j, k)] = y;
        if (k == g.nz) dph[hidx(g, ii + 1, j, g.nzc)] = y;
      }
    }
  }
}

// The same for the FP64 path, as a product with the matrix of the cosines and
// sines on the matrix cores: tiles and lines as in k_divdft.  129x128x128:
// 30 us, 45 with the vector units above (whose order of terms the mixed
// path's results hold to); 8 at the FP64 matrix rate, 7 at the copy rate.
// Four partial sums a tile keep the products from waiting for each other and
// the chains of roundings shorter than the vector units'.
__global__ __launch_bounds__(kThThreads) void k_idft64(VGrid g, const double *__restrict__ S, double *__restrict__ phi_out,
                                                       double *__restrict__ dph, DenseMat m) {
  extern __shared__ double x[];
  const int N = g.nt, ldn = N | 1, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long nlines = (long)g.nr * g.nz, l0 = (long)blockIdx.x * kThLines;
  const int nln = (int)min((long)kThLines, nlines - l0), tot = nln * N;
  {
    // the block's lines are contiguous in S; (line, position) advances by kThThreads
    const double *src = S + (size_t)N * l0;
    const int dl = kThThreads / N, dp = kThThreads - dl * N;
    constexpr int U = 8;
    int lp = tid / N, pos = tid - lp * N;
    for (int eb = tid; eb < tot; eb += U * kThThreads) {
      double v[U];
#pragma unroll
      for (int u = 0; u < U; u++) v[u] = src[min(eb + u * kThThreads, tot - 1)];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < U; u++) {
        if (eb + u * kThThreads < tot) x[lp * ldn + pos] = v[u];
        lp += dl;
        pos += dp;
        if (pos >= N) { pos -= N; lp++; }
      }
    }
    // lines past the last one: zeros
    for (int e = tot + tid; e < kThLines * N; e += kThThreads) x[(e / N) * ldn + e % N] = 0.0;
  }
  __syncthreads();
  constexpr int TPW = 4;  // N < 256: at most 2 x 16 tiles on eight waves
  d4 acc[TPW];
  const int kq = lane >> 4;
#pragma unroll
  for (int u = 0; u < TPW; u++) {
    d4 part[4];
#pragma unroll
    for (int q = 0; q < 4; q++) part[q] = d4{0.0, 0.0, 0.0, 0.0};
    const int t = wave + kThWaves * u;  // angles of tile t / 2, lines of half t % 2
    if (t >= 2 * m.mt) continue;
    const double *ap = m.a + (size_t)(t >> 1) * m.ks * 64 + lane;
    const double *xl = x + ((t & 1) * 16 + (lane & 15)) * ldn;
    double cur[kGrp], nxt[kGrp];
#pragma unroll
    for (int s = 0; s < kGrp; s++) cur[s] = ap[s * 64];
    for (int s0 = 0; s0 < m.ks; s0 += kGrp) {
      const double *np = ap + min(s0 + kGrp, m.ks - kGrp) * 64;
#pragma unroll
      for (int s = 0; s < kGrp; s++) nxt[s] = np[s * 64];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < kGrp; s++)
        part[s & 3] = __builtin_amdgcn_mfma_f64_16x16x4f64(cur[s], xl[min(4 * (s0 + s) + kq, N - 1)], part[s & 3], 0, 0, 0);
#pragma unroll
      for (int s = 0; s < kGrp; s++) cur[s] = nxt[s];
    }
    acc[u] = (part[0] + part[1]) + (part[2] + part[3]);
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < TPW; u++) {
    const int t = wave + kThWaves * u;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int i = (t >> 1) * 16 + 4 * v + kq;
      if (i < N) x[((t & 1) * 16 + (lane & 15)) * ldn + i] = acc[u][v];
    }
  }
  __syncthreads();
  // a wave per line
  for (int lp = wave; lp < nln; lp += kThWaves) {
    const long l = l0 + lp;
    const int j = (int)(l % g.nr) + 1, k = (int)(l / g.nr) + 1;
    for (int ii = lane; ii < N; ii += 64) {
      const double y = x[lp * ldn + ii];
      if (phi_out) phi_out[cidx(g, ii + 1, j, k)] = y;
      if (dph) {
        dph[hidx(g, ii + 1, j, k)] = y;
        if (k == g.nz) dph[hidx(g, ii + 1, j, g.nzc)] = y;
      }
    }
  }
}

// the z cosine matrices of n points, packed: forward rows q, columns k, entry
// cos(pi (k + 1/2) q / n); inverse rows k, columns q, twice that (1 for q = 0).
// The angle is not reduced first: the entries are those of the sums written
// out as in the definition, which the oracle evaluates too (beyond 1000
// points they are off by up to 7e-13, and reduced ones gave results 2e-11
// from the oracle's).
__global__ void k_pack_cos(double *__restrict__ fwd, double *__restrict__ inv, int n, int mt, int ks) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long)mt * ks * 64) return;
  const int l = (int)(e & 63), s = (int)((e >> 6) % ks), t = (int)((e >> 6) / ks);
  const int r = t * 16 + (l & 15), k = s * 4 + (l >> 4);
  const bool in = r < n && k < n;
  fwd[e] = in ? cos(M_PI * (k + 0.5) * r / n) : 0.0;
  inv[e] = !in ? 0.0 : k == 0 ? 1.0 : 2.0 * cos(M_PI * k * (r + 0.5) / n);
}

// steps of four columns, in whole groups
int dense_steps(int cols) { return ((cols + 3) / 4 + kGrp - 1) / kGrp * kGrp; }

// appends the rows x cols matrix f(r, k) in MFMA order (16-row tiles, steps
// of four columns, zeros outside) and returns its shape with the offset in `at`
template <typename F> DenseMat pack_dense(std::vector<double> &out, size_t &at, int rows, int cols, F f) {
  DenseMat m{nullptr, (rows + 15) / 16, dense_steps(cols)};
  at = out.size();
  out.resize(at + (size_t)m.mt * m.ks * 64, 0.0);
  for (int t = 0; t < m.mt; t++)
    for (int s = 0; s < m.ks; s++)
      for (int l = 0; l < 64; l++) {
        const int r = t * 16 + l % 16, k = s * 4 + l / 16;
        if (r < rows && k < cols) out[at + ((size_t)t * m.ks + s) * 64 + l] = f(r, k);
      }
  return m;
}

// device copy of `pk` in *dev
int upload_pack(vrh_t *h, double **dev, const std::vector<double> &pk) {
  double *nd = nullptr;
  if (hipMalloc((void **)&nd, pk.size() * sizeof(double)) != hipSuccess ||
      hipMemcpyAsync(nd, pk.data(), pk.size() * sizeof(double), hipMemcpyHostToDevice, h->stream) != hipSuccess ||
      hipStreamSynchronize(h->stream) != hipSuccess) {
    (void)hipGetLastError();
    if (nd) (void)hipFree(nd);
    h->err = "transform matrices: device allocation or copy failed";
    return -3;
  }
  *dev = nd;
  return 0;
}

}  // namespace

// Transform matrices of a grid's lengths that are no power of two (made at
// vrh_create).
int dense_create(vrh_t *h) {
  const int n = h->nz, N = h->nt;
  int rc;
  if ((n & (n - 1)) != 0) {
    DenseMat m{nullptr, (n + 15) / 16, dense_steps(n)};
    const size_t sz = (size_t)m.mt * m.ks * 64;
    if (hipMalloc((void **)&h->d_zcos, 2 * sz * sizeof(double)) != hipSuccess) {
      (void)hipGetLastError();
      h->err = "transform matrices: device allocation failed";
      return -3;
    }
    hipLaunchKernelGGL(k_pack_cos, dim3((unsigned)((sz + 255) / 256)), dim3(256), 0, h->stream, h->d_zcos,
                       h->d_zcos + sz, n, m.mt, m.ks);
    for (int q = 0; q < 2; q++) { h->zdct[q] = m; h->zdct[q].a = h->d_zcos + q * sz; }
  }
  if ((N & (N - 1)) != 0) {
    std::vector<double> cs(N), sn(N), pk;
    for (int q = 0; q < N; q++) { cs[q] = cos(2.0 * M_PI * q / N); sn[q] = sin(2.0 * M_PI * q / N); }
    size_t at;
    h->tdft = pack_dense(pk, at, N, N, [&](int pos, int i) {
      const int k = (pos + 1) / 2, ph = (int)(((long)k * i) % N);
      return pos == 0 || (pos & 1) ? cs[ph] : sn[ph];
    });
    if (h->prec != VRH_MIXED) {
      // inverse: row i, columns as the packed positions
      size_t ai;
      h->itdft = pack_dense(pk, ai, N, N, [&](int i, int pos) {
        const int k = (pos + 1) / 2, ph = (int)(((long)k * i) % N);
        return pos == 0 ? 1.0 : !(pos & 1) ? sn[ph] : 2 * k == N ? 0.5 * cs[ph] : cs[ph];
      });
      if ((rc = upload_pack(h, &h->d_tdft, pk))) return rc;
      h->tdft.a = h->d_tdft + at;
      h->itdft.a = h->d_tdft + ai;
      return 0;
    }
    // inverse: (cos, sin) of wavenumber kk at kIdT angles, tile by tile
    const size_t ti = pk.size();
    const int nk = N / 2;
    for (int tile = 0; tile * kIdT < N; tile++)
      for (int kk = 1; kk <= nk; kk++)
        for (int f = 0; f < 2; f++)
          for (int i = 0; i < kIdT; i++) {
            const int ii = tile * kIdT + i;
            pk.push_back(ii < N ? (f ? sn : cs)[((long)ii * kk) % N] : 0.0);
          }
    if ((rc = upload_pack(h, &h->d_tdft, pk))) return rc;
    h->tdft.a = h->d_tdft + at;
    h->idft_tab = h->d_tdft + ti;
  }
  return 0;
}

// V^-1 and V (row-major nz x nz) of an axial mesh, FP64 path, packed into a
// new array *dev: m[0] forward, m[1] inverse
int dense_axial(vrh_t *h, const std::vector<double> &vi, const std::vector<double> &vf, double **dev, DenseMat m[2]) {
  std::vector<double> pk;
  size_t at[2];
  const int n = h->nz;
  m[0] = pack_dense(pk, at[0], n, n, [&](int r, int k) { return vi[(size_t)r * n + k]; });
  m[1] = pack_dense(pk, at[1], n, n, [&](int r, int k) { return vf[(size_t)r * n + k]; });
  const int rc = upload_pack(h, dev, pk);
  for (int q = 0; q < 2 && !rc; q++) m[q].a = *dev + at[q];
  return rc;
}

// Tiles of 16 lines of a block: two, where a matrix entry read from L2 feeds two
// products; one where two would leave CUs without a block, take more LDS than
// lets two blocks share a CU (n > 320) or more than the device granted.
static int zdense_tiles(const vrh_t *h, long nl) {
  return nl >= 32 * 256 && h->nz <= 320 && sizeof(double) * 32 * (size_t)h->nz <= (size_t)h->lds_block ? 2 : 1;
}

// In-place z transform of nl lines.
template <typename TW> void launch_zdense(vrh_t *h, hipStream_t st, TW *S, long nl, int dir) {
  const bool axial = h->zmet.m3 != nullptr;
  const DenseMat &m = (axial ? h->zeig : h->zdct)[dir > 0 ? 0 : 1];
  const int n = h->nz, nt = zdense_tiles(h, nl);
  const double div = dir > 0 && !axial ? (double)n : 1.0;
  const dim3 grd((unsigned)((nl + 16 * nt - 1) / (16 * nt))), blk(512);
  const size_t sh = sizeof(double) * 16 * nt * (size_t)n;
  if (nt == 2) hipLaunchKernelGGL((k_zdense<TW, 2>), grd, blk, sh, st, S, nl, n, m, div);
  else hipLaunchKernelGGL((k_zdense<TW, 1>), grd, blk, sh, st, S, nl, n, m, div);
}

// cosine transforms of the mixed path's low modes and of its FP32 lines
void launch_zdense2(vrh_t *h, double *S64, long nl64, float *S, long nl, int dir) {
  const DenseMat &m = h->zdct[dir > 0 ? 0 : 1];
  const int n = h->nz, nt = zdense_tiles(h, nl);
  const double div = dir > 0 ? (double)n : 1.0;
  const unsigned na = (unsigned)((nl64 + 15) / 16), nb = (unsigned)((nl + 16 * nt - 1) / (16 * nt));
  const size_t sh = sizeof(double) * 16 * nt * (size_t)n;
  if (nt == 2) hipLaunchKernelGGL(k_zdense2<2>, dim3(na + nb), dim3(512), sh, h->stream, S64, nl64, na, S, nl, n, m, div);
  else hipLaunchKernelGGL(k_zdense2<1>, dim3(na + nb), dim3(512), sh, h->stream, S64, nl64, na, S, nl, n, m, div);
}

template <typename TW>
void launch_divdft(vrh_t *h, double inv_adt, const double *ext, TW *S, double *S64) {
  const VGrid &g = h->g;
  const long nlines = (long)g.nr * g.nz;
  hipLaunchKernelGGL(k_divdft<TW>, dim3((unsigned)((nlines + kThLines - 1) / kThLines)), dim3(kThThreads),
                     sizeof(double) * kThLines * (g.nt | 1), h->stream, g, h->coef, h->zmet, inv_adt, h->f.dq1, h->f.dq2,
                     h->f.dq3, ext, S, S64, h->d_twt, h->tdft);
}
template <typename TW>
void launch_idft(vrh_t *h, const TW *S, const double *S64, double *phi_out, double *dph) {
  const VGrid &g = h->g;
  const long nlines = (long)g.nr * g.nz;
  if constexpr (sizeof(TW) == 8)
    hipLaunchKernelGGL(k_idft64, dim3((unsigned)((nlines + kThLines - 1) / kThLines)), dim3(kThThreads),
                       sizeof(double) * kThLines * (g.nt | 1), h->stream, g, S, phi_out, dph, h->itdft);
  else
    hipLaunchKernelGGL(k_idft, dim3((unsigned)((nlines + kIdLines - 1) / kIdLines)), dim3(64 * kIdWaves),
                       sizeof(double) * kIdLines * (g.nt | 1), h->stream, g, S, S64, phi_out, dph, h->idft_tab);
}

// LDS that a grid's dense kernels need beyond the default limit, and their opt-in
size_t dense_lds_need(int nt, int nz) {
  const size_t z = (nz & (nz - 1)) ? sizeof(double) * 16 * (size_t)nz : 0;
  const size_t t = (nt & (nt - 1)) ? sizeof(double) * kIdLines * (size_t)(nt | 1) : 0;
  return z > t ? z : t;
}
bool dense_lds_optin(int bytes) {
  const void *fns[] = {reinterpret_cast<const void *>(&k_zdense<double, 1>), reinterpret_cast<const void *>(&k_zdense<double, 2>),
                       reinterpret_cast<const void *>(&k_zdense<float, 1>), reinterpret_cast<const void *>(&k_zdense<float, 2>),
                       reinterpret_cast<const void *>(&k_zdense2<1>), reinterpret_cast<const void *>(&k_zdense2<2>),
                       reinterpret_cast<const void *>(&k_divdft<double>), reinterpret_cast<const void *>(&k_divdft<float>),
                       reinterpret_cast<const void *>(&k_idft64), reinterpret_cast<const void *>(&k_idft)};
  for (const void *f : fns)
    if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return false;
  return true;
}

#define INST(TW)                                                                    \
  template void launch_zdense<TW>(vrh_t *, hipStream_t, TW *, long, int);           \
  template void launch_divdft<TW>(vrh_t *, double, const double *, TW *, double *); \
  template void launch_idft<TW>(vrh_t *, const TW *, const double *, double *, double *);
INST(double)
INST(float)
