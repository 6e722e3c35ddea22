// Reference-structured ("staged") path: one kernel per step of
// solver::calcResidual (src/solver.cpp:366-445), FR operators applied to all
// elements' columns by their non-zeros (dense where a row has too many),
// pointwise kernels over
// [point][element] and a face kernel over every face flux point.  It is the
// drop-in that mirrors the reference call for call; the fused path
// (fhip_fused.hip) is the fast one.
#include "fhip_internal.hpp"

#include <algorithm>
#include <cstdio>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

namespace fhip {

#define HIPCHK(x)                                                                     \
  do {                                                                                \
    hipError_t e_ = (x);                                                              \
    if (e_ != hipSuccess) throw std::runtime_error(std::string("HIP: ") + hipGetErrorString(e_)); \
  } while (0)

static inline unsigned blocks_for(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// ---------------------------------------------------------------------------
// Dense operator product C[m][n] = A[m][k] B[k][n] (+ C when beta).  A is a
// small FR operator read through uniform (scalar) loads; each thread owns one
// column j of B/C, keeps up to KC entries of it in registers and sweeps the
// rows of A.  Columns are contiguous in memory, so every load and store is
// coalesced.  k > KC is done in chunks, accumulating into C.
template <int KC>
__global__ __launch_bounds__(256) void k_opgemm(int m, long long n, int k, const double* __restrict__ A,
                                                 const double* __restrict__ B, double* __restrict__ C, int beta) {
  long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  for (int l0 = 0; l0 < k; l0 += KC) {
    int kc = min(KC, k - l0);
    double b[KC];
#pragma unroll
    for (int l = 0; l < KC; l++) b[l] = (l < kc) ? B[(long long)(l0 + l) * n + j] : 0.0;
    bool acc = beta || l0 > 0;
    for (int i = 0; i < m; i++) {
      const double* a = A + (long long)i * k + l0;
      double s = 0.0;
#pragma unroll
      for (int l = 0; l < KC; l++)
        if (l < kc) s += a[l] * b[l];
      double* cp = C + (long long)i * n + j;
      *cp = acc ? s + *cp : s;
    }
  }
}

static void opgemm(Ctx& c, const char* name, int m, int k, const double* A, const double* B, double* C, bool beta) {
  long long n = (long long)c.z.E * c.z.N;
  Launch L(c, name);
  if (k <= 16) hipLaunchKernelGGL(k_opgemm<16>, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, m, n, k, A, B, C, beta ? 1 : 0);
  else if (k <= 32) hipLaunchKernelGGL(k_opgemm<32>, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, m, n, k, A, B, C, beta ? 1 : 0);
  else hipLaunchKernelGGL(k_opgemm<64>, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, m, n, k, A, B, C, beta ? 1 : 0);
  HIPCHK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// The same product by the operator's non-zeros: C[i][n] = sum_g sum_q w B[idx]
// (+ C when beta), the entries in ascending order within each group and the
// groups added in turn, i.e. the dense sums without their zero terms.  On
// quads and hexes a row of 16 to 216 entries has at most P+1 non-zeros (2 per
// direction in the corrections), so the dense product is bound by multiplying
// zeros and this one by memory: it reads each operand row through the L2
// (every row serves up to 2D(P+1) outputs) and writes C once.  A wave takes 64
// columns and kRowsPerWave rows: with one thread per column over all rows a
// mesh of 18^3 P3 hexes launches 114 blocks on 256 CUs.  The row is uniform
// over the wave, so entries come through scalar loads.  Measured on 18^3 P3
// hexes (29,160 columns): the products of one Navier-Stokes residual took 5.99
// ms dense (17 launches) and took 0.148 ms this way (7 launches).  Two further
// forms save an array's way through memory: the result subtracted from another
// array (from; the flux jump), and a second operator's product added to it (q2
// entries per row of idx2, w2 over B2; the divergence's correction).
constexpr int kRowsPerWave = 8;
template <int Q>
__global__ __launch_bounds__(256) void k_oprows(int m, long long n, int groups, const int* __restrict__ idx,
                                                 const double* __restrict__ w, const double* __restrict__ B,
                                                 long long strideB, double* __restrict__ C, long long strideC,
                                                 int beta, const double* __restrict__ from, int q2,
                                                 const int* __restrict__ idx2, const double* __restrict__ w2,
                                                 const double* __restrict__ B2) {
  const long long j = (long long)blockIdx.x * 64 + (threadIdx.x & 63);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (j >= n) return;
  B += blockIdx.z * strideB + j;
  C += blockIdx.z * strideC + j;
  const int i0 = (blockIdx.y * 4 + wave) * kRowsPerWave;
#pragma unroll 2
  for (int r = 0; r < kRowsPerWave; r++) {
    const int i = i0 + r;
    if (i >= m) return;
    double tot = 0.0;
    for (int g = 0; g < groups; g++) {
      const int* ix = idx + ((long long)i * groups + g) * Q;
      const double* wt = w + ((long long)i * groups + g) * Q;
      double s = 0.0;
#pragma unroll
      for (int q = 0; q < Q; q++) s += wt[q] * B[ix[q] * n];
      tot = g ? s + tot : s;
    }
    if (q2) {
      double s = 0.0;
#pragma unroll 2
      for (int q = 0; q < q2; q++) s += w2[(long long)i * q2 + q] * B2[idx2[(long long)i * q2 + q] * n + j];
      tot = s + tot;
    }
    double* cp = C + i * n;
    *cp = from ? from[i * n + j] - tot : (beta ? tot + *cp : tot);
  }
}

// Largest number of entries per group kept as rows: P+1 = 11 at the highest
// order on quads and hexes.  An operator with wider rows (one the caller built
// on other bases) is a dense product and stays one.
constexpr int kMaxRowEntries = 12;

// op: m rows of `groups` partial sums over `blocks` of k entries each, row(i, g, b) the
// k entries of one, which belong to operand rows (g * blocks + b) * k + 0..k-1.  Its
// tables go to the end of mem, at the offsets left in their pointers.
template <class F>
static void build_rows(RowOp& op, std::vector<char>& mem, int m, int groups, int blocks, int k, F&& row) {
  std::vector<int> idx, n((size_t)m * groups, 0);  // the non-zeros' operand rows, their number
  std::vector<double> w;
  int q = 1;
  for (int i = 0, r = 0; i < m; i++)
    for (int g = 0; g < groups; g++, r++) {
      for (int b = 0; b < blocks; b++) {
        const double* a = row(i, g, b);
        each_nonzero(a, k, [&](int l) {
          idx.push_back((g * blocks + b) * k + l);
          w.push_back(a[l]);
          n[r]++;
          return true;
        });
      }
      q = std::max(q, n[r]);
      if (q > kMaxRowEntries) return;
    }
  if (q > 6) q = kMaxRowEntries;
  op.m = m;
  op.groups = groups;
  op.q = q;
  const size_t rows = n.size() * q, at = (mem.size() + 15) / 16 * 16;
  mem.resize(at + rows * (sizeof(double) + sizeof(int)));
  op.w = reinterpret_cast<double*>(at);
  op.idx = reinterpret_cast<int*>(at + rows * sizeof(double));
  double* const tw = reinterpret_cast<double*>(mem.data() + at);
  int* const ti = reinterpret_cast<int*>(tw + rows);
  size_t from = 0;
  for (size_t r = 0; r < n.size(); r++) {
    for (int p = 0; p < q; p++) {
      // padding repeats the row's own first operand with weight zero
      const bool in = p < n[r];
      ti[r * q + p] = in ? idx[from + p] : (n[r] ? idx[from] : (int)(r % groups) * blocks * k);
      tw[r * q + p] = in ? w[from + p] : 0.0;
    }
    from += n[r];
  }
}

// (One allocation and one copy for all of them: with two of each per operator, 16 in
// all, the context of an 8x8 mesh took 0.53 ms to set up instead of 0.39.)
void staged_setup(Ctx& c, const fhip_desc* d) {
  const int D = c.z.D, S = c.z.S, F = c.z.F;
  std::vector<char> mem;
  build_rows(c.r_sf, mem, F, 1, 1, S, [&](int i, int, int) { return d->opp_spts_to_fpts + (size_t)i * S; });
  build_rows(c.r_div, mem, S, D, 1, S, [&](int i, int g, int) { return d->opp_grad_spts + ((size_t)g * S + i) * S; });
  build_rows(c.r_efn, mem, F, 1, D, S, [&](int i, int, int b) { return d->opp_extrapolate_fn + ((size_t)b * F + i) * S; });
  build_rows(c.r_corr, mem, S, 1, 1, F, [&](int i, int, int) { return d->opp_correction + (size_t)i * F; });
  if (c.prm.viscous) {
    build_rows(c.r_grad, mem, D * S, 1, 1, S, [&](int i, int, int) { return d->opp_grad_spts + (size_t)i * S; });
    build_rows(c.r_corru, mem, D * S, 1, 1, F, [&](int i, int, int) { return d->opp_correct_u + (size_t)i * F; });
  }
  if (mem.empty()) return;
  HIPCHK(hipMalloc(&c.row_mem, mem.size()));
  HIPCHK(hipMemcpy(c.row_mem, mem.data(), mem.size(), hipMemcpyHostToDevice));
  for (RowOp* op : {&c.r_sf, &c.r_grad, &c.r_corru, &c.r_efn, &c.r_div, &c.r_corr}) {
    if (!op->q) continue;
    op->w = reinterpret_cast<double*>(static_cast<char*>(c.row_mem) + reinterpret_cast<size_t>(op->w));
    op->idx = reinterpret_cast<int*>(static_cast<char*>(c.row_mem) + reinterpret_cast<size_t>(op->idx));
  }
}

void staged_release(Ctx& c) {
  if (c.row_mem) (void)hipFree(c.row_mem);
  c.row_mem = nullptr;
}

// op applied to `count` operands strideB apart, into outputs strideC apart.
static void oprows(Ctx& c, const char* name, const RowOp& op, const double* B, double* C, bool beta, int count = 1,
                   long long strideB = 0, long long strideC = 0, const double* from = nullptr,
                   const RowOp* op2 = nullptr, const double* B2 = nullptr) {
  const long long n = (long long)c.z.E * c.z.N;
  const dim3 grid(blocks_for(n, 64), blocks_for(op.m, 4 * kRowsPerWave), count);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, c.stream, op.m, n, op.groups, op.idx, op.w, B, strideB, C, strideC,
                       beta ? 1 : 0, from, op2 ? op2->q : 0, op2 ? op2->idx : nullptr, op2 ? op2->w : nullptr, B2);
  };
  Launch L(c, name);
  switch (op.q) {
    case 1: go(k_oprows<1>); break;
    case 2: go(k_oprows<2>); break;
    case 3: go(k_oprows<3>); break;
    case 4: go(k_oprows<4>); break;
    case 5: go(k_oprows<5>); break;
    case 6: go(k_oprows<6>); break;
    default: go(k_oprows<kMaxRowEntries>); break;
  }
  HIPCHK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// calcInviscidFlux_spts (src/solver.cpp:707-736): one thread per (spt, ele); the
// transform follows with the viscous flux.
template <int D>
__global__ __launch_bounds__(256) void k_inviscid_spts(long long nPts, long long SE, const double* __restrict__ U,
                                                        double* __restrict__ Fs, double gamma) {
  constexpr int N = D + 2;
  long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nPts) return;
  double u[N], F[D][N];
#pragma unroll
  for (int k = 0; k < N; k++) u[k] = U[p * N + k];
  inviscid_flux<D, double>(u, F, gamma);
#pragma unroll
  for (int d = 0; d < D; d++)
#pragma unroll
    for (int k = 0; k < N; k++) Fs[(d * SE + p) * N + k] = F[d][k];
}

// ---------------------------------------------------------------------------
// Inviscid face pass (face::calcInviscidFlux, src/face.cpp:163-208; right
// side src/intFace.cpp:147-161): one thread per face flux point.
template <int D>
__global__ __launch_bounds__(256) void k_face_inviscid(int nFF, const int* __restrict__ ptL, const int* __restrict__ ptR,
                                                        const int* __restrict__ bcs, const double* __restrict__ Uf,
                                                        const double* __restrict__ nrm, const double* __restrict__ dA,
                                                        double* __restrict__ Fn, double* __restrict__ faceFn,
                                                        double* __restrict__ waveSp, double* __restrict__ dUc,
                                                        Phys ph) {
  constexpr int N = D + 2;
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nFF) return;
  int pl = ptL[t], pr = ptR[t], bc = bcs[t];
  double UL[N], UR[N], n[D], fn[N];
#pragma unroll
  for (int k = 0; k < N; k++) UL[k] = Uf[(long long)pl * N + k];
#pragma unroll
  for (int d = 0; d < D; d++) n[d] = nrm[(long long)pl * D + d];
  if (pr < 0) apply_bc<D, double>(bc, UL, n, UR, ph);
  else {
#pragma unroll
    for (int k = 0; k < N; k++) UR[k] = Uf[(long long)pr * N + k];
  }
  if (pr < 0 || ph.riemann_type == 0) waveSp[pl] = rusanov<D, double>(UL, UR, n, fn, ph.gamma);
  else {
    if constexpr (D == 2) roe2d<double>(UL, UR, n, fn, ph.gamma);
  }
  // (viscous runs: the viscous face pass, which follows, adds to faceFn and
  // writes Fn)
  if (ph.viscous) {
#pragma unroll
    for (int k = 0; k < N; k++) faceFn[(long long)t * N + k] = fn[k];
    double pf = (pr < 0) ? 0.0 : ldg_pen<D, double>(n, ph.pen_fact);
#pragma unroll
    for (int k = 0; k < N; k++) {
      double uc = (pr < 0) ? 0.5 * (UL[k] + UR[k]) : 0.5 * (UL[k] + UR[k]) - pf * (UL[k] - UR[k]);
      dUc[(long long)pl * N + k] = uc - UL[k];
      if (pr >= 0) dUc[(long long)pr * N + k] = uc - UR[k];
    }
    return;
  }
  double dAL = dA[pl];
#pragma unroll
  for (int k = 0; k < N; k++) Fn[(long long)pl * N + k] = fn[k] * dAL;
  if (pr >= 0) {
    double dAR = dA[pr];
#pragma unroll
    for (int k = 0; k < N; k++) Fn[(long long)pr * N + k] = -fn[k] * dAR;
  }
}

// correctGradU physical transform (src/solver.cpp:1105-1136).
template <int D>
__global__ __launch_bounds__(256) void k_grad_transform(long long nPts, long long SE, double* __restrict__ dU,
                                                         const double* __restrict__ JG, const double* __restrict__ detj) {
  constexpr int N = D + 2;
  long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nPts) return;
  double inv = 1. / detj[p];
  double G[D][D];
#pragma unroll
  for (int r = 0; r < D; r++)
#pragma unroll
    for (int x = 0; x < D; x++) G[r][x] = JG[(r * SE + p) * D + x];
#pragma unroll
  for (int k = 0; k < N; k++) {
    double r[D];
#pragma unroll
    for (int d = 0; d < D; d++) r[d] = dU[(d * SE + p) * N + k];
#pragma unroll
    for (int x = 0; x < D; x++) {
      double acc = r[0] * G[0][x] + r[1] * G[1][x];
      if constexpr (D == 3) acc += r[2] * G[2][x];
      dU[(x * SE + p) * N + k] = inv * acc;
    }
  }
}

// calcViscousFlux_spts (src/solver.cpp:777-811).
template <int D>
__global__ __launch_bounds__(256) void k_viscous_spts(long long nPts, long long SE, const double* __restrict__ U,
                                                       const double* __restrict__ dU, const double* __restrict__ JG,
                                                       double* __restrict__ Fs, Phys ph) {
  constexpr int N = D + 2;
  long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nPts) return;
  double u[N], g[D][N], Fv[D][N];
#pragma unroll
  for (int k = 0; k < N; k++) u[k] = U[p * N + k];
#pragma unroll
  for (int d = 0; d < D; d++)
#pragma unroll
    for (int k = 0; k < N; k++) g[d][k] = dU[(d * SE + p) * N + k];
  viscous_flux<D, double>(u, g, Fv, ph);
#pragma unroll
  for (int d = 0; d < D; d++)
#pragma unroll
    for (int k = 0; k < N; k++) Fv[d][k] += Fs[(d * SE + p) * N + k];
#pragma unroll
  for (int d1 = 0; d1 < D; d1++)
#pragma unroll
    for (int k = 0; k < N; k++) {
      double acc = 0.;
#pragma unroll
      for (int d2 = 0; d2 < D; d2++) acc += JG[(d1 * SE + p) * D + d2] * Fv[d2][k];
      Fs[(d1 * SE + p) * N + k] = acc;
    }
}

// All pointwise work between the operators in one kernel, for operators of rows
// with at most 6 entries (2 in the gradient's correction): gradient, its
// correction (opp_correctU) and physical transform (viscous runs), inviscid and
// viscous flux, transformed flux; the sums are those of k_oprows, k_grad_transform,
// k_inviscid_spts and k_viscous_spts, in their order.  Those kernels moved the
// gradient and the flux of every point through memory seven times.
//
// A wave takes one solution point of 64 elements, as 64 * N contiguous columns for
// the operators and for every load and store of fields, and as 64 points for the
// physics, with its part of LDS between the two: a thread per point that reads and
// writes its fields itself touches a 40-byte stride with each access, which took
// as long as the bytes again.  18^3 P3 hexes: 132 us in five kernels, now 50 us.
template <int D, int Q, bool VISC>
__global__ __launch_bounds__(256) void k_point_flux(int S, int E, const int* __restrict__ gi,
                                                     const double* __restrict__ gw, const int* __restrict__ ci,
                                                     const double* __restrict__ cw, const double* __restrict__ U,
                                                     const double* __restrict__ dUc, const double* __restrict__ JG,
                                                     const double* __restrict__ detj, double* __restrict__ dU,
                                                     double* __restrict__ Fs, Phys ph) {
  constexpr int N = D + 2, C = 64 * N;
  __shared__ double lds[4][(D + 1) * C];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = blockIdx.y * 4 + wave, e0 = blockIdx.x * 64;
  const int ne = s < S ? min(64, E - e0) : 0, nc = ne * N;  // elements and columns of this wave
  const long long n = (long long)E * N, j0 = (long long)e0 * N, SE = (long long)S * E;
  double* const su = lds[wave];      // [64][N] U
  double* const sv = su + C;         // [D][64][N] gradient, then flux
#pragma unroll
  for (int t = 0; t < N; t++) {
    const int c = t * 64 + lane;
    if (c < nc) {
      const double* const u = U + j0 + c;
      su[c] = u[s * n];
      if constexpr (VISC) {
        const double* const uc = dUc + j0 + c;
#pragma unroll
        for (int d = 0; d < D; d++) {
          const int i = d * S + s;
          double g = 0.0, a = 0.0;
#pragma unroll
          for (int q = 0; q < Q; q++) g += gw[i * Q + q] * u[gi[i * Q + q] * n];
#pragma unroll
          for (int q = 0; q < 2; q++) a += cw[i * 2 + q] * uc[ci[i * 2 + q] * n];
          sv[d * C + c] = a + g;
        }
      }
    }
  }
  const long long p = (long long)s * E + e0 + lane;
  double G[D][D];
  if (lane < ne) {
#pragma unroll
    for (int r = 0; r < D; r++)
#pragma unroll
      for (int x = 0; x < D; x++) G[r][x] = JG[(r * SE + p) * D + x];
  }
  __syncthreads();
  double g[D][N];
  if constexpr (VISC) {
    if (lane < ne) {
      const double inv = 1. / detj[p];
#pragma unroll
      for (int k = 0; k < N; k++) {
        double r[D];
#pragma unroll
        for (int d = 0; d < D; d++) r[d] = sv[d * C + lane * N + k];
#pragma unroll
        for (int x = 0; x < D; x++) {
          double acc = r[0] * G[0][x] + r[1] * G[1][x];
          if constexpr (D == 3) acc += r[2] * G[2][x];
          g[x][k] = inv * acc;
          sv[x * C + lane * N + k] = g[x][k];
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int t = 0; t < N; t++) {
        const int c = t * 64 + lane;
        if (c < nc) dU[((long long)d * S + s) * n + j0 + c] = sv[d * C + c];
      }
    __syncthreads();
  }
  if (lane < ne) {
    double u[N], F[D][N];
#pragma unroll
    for (int k = 0; k < N; k++) u[k] = su[lane * N + k];
    inviscid_flux<D, double>(u, F, ph.gamma);
    if constexpr (VISC) {
      double Fv[D][N];
      viscous_flux<D, double>(u, g, Fv, ph);
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int k = 0; k < N; k++) F[d][k] = Fv[d][k] + F[d][k];
    }
#pragma unroll
    for (int d1 = 0; d1 < D; d1++)
#pragma unroll
      for (int k = 0; k < N; k++) {
        double acc = 0.;
#pragma unroll
        for (int d2 = 0; d2 < D; d2++) acc += G[d1][d2] * F[d2][k];
        sv[d1 * C + lane * N + k] = acc;
      }
  }
  __syncthreads();
#pragma unroll
  for (int d = 0; d < D; d++)
#pragma unroll
    for (int t = 0; t < N; t++) {
      const int c = t * 64 + lane;
      if (c < nc) Fs[((long long)d * S + s) * n + j0 + c] = sv[d * C + c];
    }
}

// Viscous face pass (face::calcViscousFlux, src/face.cpp:210-311).
template <int D>
__global__ __launch_bounds__(256) void k_face_viscous(int nFF, const int* __restrict__ ptL, const int* __restrict__ ptR,
                                                       const int* __restrict__ bcs, const double* __restrict__ Uf,
                                                       const double* __restrict__ dUf, long long FE,
                                                       const double* __restrict__ nrm, const double* __restrict__ dA,
                                                       double* __restrict__ Fn, const double* __restrict__ faceFn,
                                                       Phys ph) {
  constexpr int N = D + 2;
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nFF) return;
  int pl = ptL[t], pr = ptR[t], bc = bcs[t];
  double UL[N], UR[N], n[D], gL[D][N], gR[D][N], fn[N];
#pragma unroll
  for (int k = 0; k < N; k++) UL[k] = Uf[(long long)pl * N + k];
#pragma unroll
  for (int d = 0; d < D; d++) n[d] = nrm[(long long)pl * D + d];
#pragma unroll
  for (int d = 0; d < D; d++)
#pragma unroll
    for (int k = 0; k < N; k++) gL[d][k] = dUf[(d * FE + pl) * N + k];
  int bnd = 0;
  if (pr < 0) {
    apply_bc<D, double>(bc, UL, n, UR, ph);
    bnd = (bc == 10) ? 2 : 1;
    if (bnd == 2) {
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int k = 0; k < N; k++) gR[d][k] = gL[d][k];
      adiabatic_grad<D, double>(UL, UR, gR, ph.gamma);
    } else {
#pragma unroll
      for (int d = 0; d < D; d++)
#pragma unroll
        for (int k = 0; k < N; k++) gR[d][k] = 0.;
    }
  } else {
#pragma unroll
    for (int k = 0; k < N; k++) UR[k] = Uf[(long long)pr * N + k];
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int k = 0; k < N; k++) gR[d][k] = dUf[(d * FE + pr) * N + k];
  }
#pragma unroll
  for (int k = 0; k < N; k++) fn[k] = faceFn[(long long)t * N + k];
  ldg_flux<D, double>(bnd, UL, UR, gL, gR, n, fn, ph);
  double dAL = dA[pl];
#pragma unroll
  for (int k = 0; k < N; k++) Fn[(long long)pl * N + k] = fn[k] * dAL;
  if (pr >= 0) {
    double dAR = dA[pr];
#pragma unroll
    for (int k = 0; k < N; k++) Fn[(long long)pr * N + k] = -fn[k] * dAR;
  }
}

__global__ void k_sub(long long n, const double* __restrict__ a, double* __restrict__ b) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = a[i] - b[i];
}

__global__ void k_copy(long long n, double* __restrict__ dst, const double* __restrict__ src) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// timeStepA / timeStepB (src/solver.cpp:470-536); dt from device memory.  A thread
// per value: one per point, each access at a stride of 40 bytes, took 24 us on
// 18^3 P3 hexes where this takes 11 us.
template <int N>
__global__ __launch_bounds__(256) void k_time_step(long long n, unsigned E, int modeB, double rk,
                                                    double* __restrict__ U, const double* __restrict__ U0,
                                                    const double* __restrict__ divF, const double* __restrict__ src,
                                                    const double* __restrict__ detj, const double* __restrict__ dtp,
                                                    const double* __restrict__ eleDt, int local) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const long long p = i / N;
  const double dt = local ? eleDt[p % E] : *dtp;
  const double dj = detj[p];
  const double r = src ? (divF[i] + src[i]) : divF[i];
  if (modeB) U[i] -= rk * r / dj * dt;
  else U[i] = U0[i] - rk * r / dj * dt;
}

// calcWaveSpFpts for every element (src/ele.cpp:1097-1124).  waveSp is
// stored [fpt][ele].
template <int D>
__global__ void k_wave_speed(long long nPts, const double* __restrict__ Uf, const double* __restrict__ nrm,
                             double* __restrict__ waveSp, double gamma) {
  constexpr int N = D + 2;
  long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nPts) return;
  const double* U = Uf + p * N;
  double rho = U[0], u = U[1] / rho, v = U[2] / rho, w = 0;
  if constexpr (D == 3) w = U[3] / rho;
  double rhoVSq = rho * (u * u + v * v + w * w);
  double pr = (gamma - 1) * (U[D + 1] - 0.5 * rhoVSq);
  double vN = u * nrm[p * D] + v * nrm[p * D + 1];
  if constexpr (D == 3) vN += w * nrm[p * D + 2];
  double csq = smax(gamma * pr / rho, 0.0);
  waveSp[p] = (fabs(vN - 0.) + sqrt(csq));
}

// ele::calcDt for every element (src/ele.cpp:1127-1146) and a per-block
// minimum; a second kernel folds the block minima into *dtp.
__global__ __launch_bounds__(256) void k_ele_dt(int E, int S, int F, int Ff, const double* __restrict__ detj,
                                                 const double* __restrict__ ws, const double* __restrict__ wf,
                                                 const double* __restrict__ waveSp, const double* __restrict__ dA,
                                                 double cflfac, double* __restrict__ eleDt, double* __restrict__ part) {
  __shared__ double red[256];
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  double dt = INFINITY;
  if (e < E) {
    double vol = 0;
    for (int s = 0; s < S; s++) vol += detj[(long long)s * E + e] * ws[s];
    double iw = 0;
    for (int f = 0; f < F; f++) iw += waveSp[(long long)f * E + e] * wf[f % Ff] * dA[(long long)f * E + e];
    dt = cflfac * 2 * vol / iw;
    eleDt[e] = dt;
  }
  red[threadIdx.x] = dt;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] = fmin(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void k_min_final(int n, const double* __restrict__ part, double* __restrict__ out) {
  __shared__ double red[256];
  double v = INFINITY;
  for (int i = threadIdx.x; i < n; i += blockDim.x) v = fmin(v, part[i]);
  red[threadIdx.x] = v;
  __syncthreads();
  for (int s = blockDim.x / 2; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] = fmin(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

// Residual norm (ele::getNormResidual, src/ele.cpp:1922-1945): partial sums
// [block][N].  A block takes 256 elements and every gridDim.y-th solution point,
// a thread one element and all its fields at once.  (A thread per element over
// all points, one pass per field, left most of the chip idle, with each wave
// using 8 bytes of the 40 that it read: 264 us on 9261 P4 hexes, now
// 25 us and 5 us for the final sum.)
constexpr int kResFields = 5;
__device__ __forceinline__ double res_join(int type, double a, double b) { return type == 3 ? fmax(a, b) : a + b; }
__device__ __forceinline__ void res_block(int N, int type, double* r, double* out) {
  __shared__ double red[4][kResFields];
#pragma unroll
  for (int k = 0; k < kResFields; k++) {
    if (k >= N) break;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) r[k] = res_join(type, r[k], __shfl_xor(r[k], o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][k] = r[k];
  }
  __syncthreads();
  if ((int)threadIdx.x < N) {
    double v = red[0][threadIdx.x];
    for (int w = 1; w < 4; w++) v = res_join(type, v, red[w][threadIdx.x]);
    out[threadIdx.x] = v;
  }
}
__global__ __launch_bounds__(256) void k_res_norm(int E, int S, int N, int type, const double* __restrict__ divF,
                                                   const double* __restrict__ detj, const double* __restrict__ ws,
                                                   double* __restrict__ part) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  double r[kResFields] = {};
  if (e < E) {
    for (int s = blockIdx.y; s < S; s += gridDim.y) {
      const long long p = (long long)s * E + e;
      const double* v = divF + p * N;
      const double w = ws[s], dj = type == 1 ? 1. : detj[p];
#pragma unroll
      for (int k = 0; k < kResFields; k++) {
        if (k >= N) break;
        if (type == 1) r[k] += fabs(v[k]) * w;
        else if (type == 2) r[k] += v[k] * v[k] / dj * w;
        else r[k] = fmax(fabs(v[k]) / dj, r[k]);
      }
    }
  }
  res_block(N, type, r, part + ((long long)blockIdx.y * gridDim.x + blockIdx.x) * N);
}

// The norm from the partial sums, one block.
__global__ __launch_bounds__(256) void k_res_final(int rows, int N, int type, const double* __restrict__ part,
                                                    double* __restrict__ out) {
  double r[kResFields] = {};
  for (int b = threadIdx.x; b < rows; b += blockDim.x) {
#pragma unroll
    for (int k = 0; k < kResFields; k++) {
      if (k >= N) break;
      r[k] = res_join(type, r[k], part[(long long)b * N + k]);
    }
  }
  __shared__ double fin[kResFields];
  res_block(N, type, r, fin);
  __syncthreads();
  if ((int)threadIdx.x < N) out[threadIdx.x] = type == 2 ? sqrt(fin[threadIdx.x]) : fin[threadIdx.x];
}

// NaN / non-positive density or pressure scan.
template <int D>
__global__ void k_check(long long nPts, const double* __restrict__ U, double gamma, int* flag) {
  constexpr int N = D + 2;
  long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= nPts) return;
  const double* u = U + p * N;
  double q = 0;
  for (int d = 0; d < D; d++) q += u[d + 1] * u[d + 1];
  double pr = (gamma - 1) * (u[D + 1] - 0.5 * q / u[0]);
  bool bad = !(u[0] > 0) || !(pr > 0);
  for (int k = 0; k < N; k++) bad = bad || !isfinite(u[k]);
  if (bad) atomicOr(flag, 1);
}

// ---------------------------------------------------------------------------

void op_apply(Ctx& c, const char* name, int m, int k, const double* A, const double* B, double* C, bool beta) {
  opgemm(c, name, m, k, A, B, C, beta);
}

// out may alias a
__global__ void k_sub_arr(long long n, double* out, const double* a, const double* __restrict__ b) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    double v = a[i];
    v -= b[i];
    out[i] = v;
  }
}

__global__ void k_add_arr(long long n, double* __restrict__ y, const double* __restrict__ x) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] += x[i];
}

void sub_array(Ctx& c, double* out, const double* a, const double* b, long long n) {
  Launch L(c, "pmg_sub");
  hipLaunchKernelGGL(k_sub_arr, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, out, a, b);
  HIPCHK(hipGetLastError());
}

void add_array(Ctx& c, double* y, const double* x, long long n) {
  Launch L(c, "pmg_add");
  hipLaunchKernelGGL(k_add_arr, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, y, x);
  HIPCHK(hipGetLastError());
}

void copy_array(Ctx& c, double* dst, const double* src, long long n) {
  Launch L(c, "copy");
  hipLaunchKernelGGL(k_copy, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, dst, src);
  HIPCHK(hipGetLastError());
}

void staged_extrapolate_u(Ctx& c) {
  if (c.r_sf.q) oprows(c, "oprows_extrapolate_u", c.r_sf, c.U, c.Uf, false);
  else opgemm(c, "opgemm_extrapolate_u", c.z.F, c.z.S, c.sf, c.U, c.Uf, false);
}

void staged_wave_speed(Ctx& c) {
  long long n = (long long)c.z.F * c.z.E;
  Launch L(c, "wave_speed");
  if (c.z.D == 2) hipLaunchKernelGGL(k_wave_speed<2>, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, c.Uf, c.norm, c.waveSp, c.ph.gamma);
  else hipLaunchKernelGGL(k_wave_speed<3>, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, c.Uf, c.norm, c.waveSp, c.ph.gamma);
  HIPCHK(hipGetLastError());
}

template <int D, bool VISC>
static void launch_point_flux(Ctx& c) {
  const dim3 grid(blocks_for(c.z.E, 64), blocks_for(c.z.S, 4));
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, c.stream, c.z.S, c.z.E, c.r_grad.idx, c.r_grad.w, c.r_corru.idx,
                       c.r_corru.w, c.U, c.dUc, c.jginv, c.detj, c.dU, c.Fs, c.ph);
  };
  Launch L(c, "point_flux");
  if constexpr (VISC) {
    switch (c.r_grad.q) {
      case 1: go(k_point_flux<D, 1, true>); break;
      case 2: go(k_point_flux<D, 2, true>); break;
      case 3: go(k_point_flux<D, 3, true>); break;
      case 4: go(k_point_flux<D, 4, true>); break;
      case 5: go(k_point_flux<D, 5, true>); break;
      default: go(k_point_flux<D, 6, true>); break;
    }
  } else {
    go(k_point_flux<D, 1, false>);
  }
  HIPCHK(hipGetLastError());
}
static void launch_point_flux(Ctx& c) {
  if (c.z.D == 2) c.prm.viscous ? launch_point_flux<2, true>(c) : launch_point_flux<2, false>(c);
  else c.prm.viscous ? launch_point_flux<3, true>(c) : launch_point_flux<3, false>(c);
}

void staged_residual(Ctx& c, int step) {
  const Sizes& z = c.z;
  const long long nS = z.nS(), nF = z.nF(), SE = (long long)z.S * z.E, FE = (long long)z.F * z.E;
  const bool visc = c.prm.viscous != 0;
  double* divF = c.divF + step * nS;
  unsigned gS = blocks_for(SE, 256), gFF = blocks_for(z.nFaceFpts, 256);

  // the pointwise kernels in one
  const bool points = c.r_grad.q <= 6 && (!visc || (c.r_grad.q > 0 && c.r_corru.q == 2));

  staged_extrapolate_u(c);
  if (points) {
  } else if (visc && c.r_grad.q) oprows(c, "oprows_grad_u", c.r_grad, c.U, c.dU, false);
  else if (visc)
    for (int d = 0; d < z.D; d++) opgemm(c, "opgemm_grad_u", z.S, z.S, c.grad + (long long)d * z.S * z.S, c.U, c.dU + d * nS, false);
  if (!points) {
    Launch L(c, "inviscid_spts");
    if (z.D == 2) hipLaunchKernelGGL(k_inviscid_spts<2>, dim3(gS), dim3(256), 0, c.stream, SE, SE, c.U, c.Fs, c.ph.gamma);
    else hipLaunchKernelGGL(k_inviscid_spts<3>, dim3(gS), dim3(256), 0, c.stream, SE, SE, c.U, c.Fs, c.ph.gamma);
    HIPCHK(hipGetLastError());
  }
  if (z.nFaceFpts > 0) {
    Launch L(c, "face_inviscid");
    if (z.D == 2) hipLaunchKernelGGL(k_face_inviscid<2>, dim3(gFF), dim3(256), 0, c.stream, z.nFaceFpts, c.ft.ptL, c.ft.ptR, c.ft.bc, c.Uf, c.norm, c.da, c.Fn, c.faceFn, c.waveSp, c.dUc, c.ph);
    else hipLaunchKernelGGL(k_face_inviscid<3>, dim3(gFF), dim3(256), 0, c.stream, z.nFaceFpts, c.ft.ptL, c.ft.ptR, c.ft.bc, c.Uf, c.norm, c.da, c.Fn, c.faceFn, c.waveSp, c.dUc, c.ph);
    HIPCHK(hipGetLastError());
  }
  if (points) launch_point_flux(c);
  if (visc) {
    if (points) {
    } else if (c.r_corru.q) oprows(c, "oprows_correct_grad_u", c.r_corru, c.dUc, c.dU, true);
    else for (int d = 0; d < z.D; d++) opgemm(c, "opgemm_correct_grad_u", z.S, z.F, c.corru + (long long)d * z.S * z.F, c.dUc, c.dU + d * nS, true);
    if (!points) {
      Launch L(c, "grad_transform");
      if (z.D == 2) hipLaunchKernelGGL(k_grad_transform<2>, dim3(gS), dim3(256), 0, c.stream, SE, SE, c.dU, c.jginv, c.detj);
      else hipLaunchKernelGGL(k_grad_transform<3>, dim3(gS), dim3(256), 0, c.stream, SE, SE, c.dU, c.jginv, c.detj);
      HIPCHK(hipGetLastError());
    }
    if (c.r_sf.q) oprows(c, "oprows_extrapolate_grad_u", c.r_sf, c.dU, c.dUf, false, z.D, nS, nF);
    else for (int d = 0; d < z.D; d++) opgemm(c, "opgemm_extrapolate_grad_u", z.F, z.S, c.sf, c.dU + d * nS, c.dUf + d * nF, false);
    if (!points) {
      Launch L(c, "viscous_spts");
      if (z.D == 2) hipLaunchKernelGGL(k_viscous_spts<2>, dim3(gS), dim3(256), 0, c.stream, SE, SE, c.U, c.dU, c.jginv, c.Fs, c.ph);
      else hipLaunchKernelGGL(k_viscous_spts<3>, dim3(gS), dim3(256), 0, c.stream, SE, SE, c.U, c.dU, c.jginv, c.Fs, c.ph);
      HIPCHK(hipGetLastError());
    }
    if (z.nFaceFpts > 0) {
      Launch L(c, "face_viscous");
      if (z.D == 2) hipLaunchKernelGGL(k_face_viscous<2>, dim3(gFF), dim3(256), 0, c.stream, z.nFaceFpts, c.ft.ptL, c.ft.ptR, c.ft.bc, c.Uf, c.dUf, FE, c.norm, c.da, c.Fn, c.faceFn, c.ph);
      else hipLaunchKernelGGL(k_face_viscous<3>, dim3(gFF), dim3(256), 0, c.stream, z.nFaceFpts, c.ft.ptL, c.ft.ptR, c.ft.bc, c.Uf, c.dUf, FE, c.norm, c.da, c.Fn, c.faceFn, c.ph);
      HIPCHK(hipGetLastError());
    }
  }
  // extrapolateNormalFlux (static grid), calcDivF_spts, correctDivFlux
  if (c.r_efn.q) oprows(c, "oprows_flux_jump", c.r_efn, c.Fs, c.disFn, false, 1, 0, 0, c.Fn);
  else for (int d = 0; d < z.D; d++) opgemm(c, "opgemm_extrapolate_fn", z.F, z.S, c.efn + (long long)d * z.F * z.S, c.Fs + d * nS, c.disFn, d > 0);
  const bool both = c.r_efn.q && c.r_div.q && c.r_corr.q;
  if (both) oprows(c, "oprows_div_f", c.r_div, c.Fs, divF, false, 1, 0, 0, nullptr, &c.r_corr, c.disFn);
  else if (c.r_div.q) oprows(c, "oprows_div_f", c.r_div, c.Fs, divF, false);
  else for (int d = 0; d < z.D; d++) opgemm(c, "opgemm_div_f", z.S, z.S, c.grad + (long long)d * z.S * z.S, c.Fs + d * nS, divF, d > 0);
  if (!c.r_efn.q) {
    Launch L(c, "sub_fn");
    hipLaunchKernelGGL(k_sub, dim3(blocks_for(nF, 256)), dim3(256), 0, c.stream, nF, c.Fn, c.disFn);
    HIPCHK(hipGetLastError());
  }
  if (both) return;
  if (c.r_corr.q) oprows(c, "oprows_correction", c.r_corr, c.disFn, divF, true);
  else opgemm(c, "opgemm_correction", z.S, z.F, c.corr, c.disFn, divF, true);
}

static void time_step(Ctx& c, const char* name, int modeB, double rk, int step, bool src) {
  const long long n = c.z.nS();
  Launch L(c, name);
  auto* kern = c.z.D == 2 ? k_time_step<4> : k_time_step<5>;
  hipLaunchKernelGGL(kern, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, (unsigned)c.z.E, modeB, rk, c.U, c.U0,
                     c.divF + step * n, src ? c.src : nullptr, c.detj, c.d_dt, c.eleDt, c.prm.dt_type == 2 ? 1 : 0);
  HIPCHK(hipGetLastError());
}

void staged_time_step_a(Ctx& c, int step, double rk, bool src) { time_step(c, "time_step_a", 0, rk, step, src); }

void staged_time_step_b(Ctx& c, int step, bool src) { time_step(c, "time_step_b", 1, c.prm.rk_b[step], step, src); }

static double cfl_limit(int order) {  // getCFLLimit, src/global.cpp:81-105
  static const double t[6] = {1.393, 0.464, 0.235, 0.1453, 0.100, 0.0736};
  if (order < 0 || order > 5) throw std::invalid_argument("CFL limit not available for this order!");
  return t[order];
}

void calc_dt(Ctx& c, bool refresh) {
  if (refresh) {
    staged_extrapolate_u(c);
    staged_wave_speed(c);
  }
  const Sizes& z = c.z;
  unsigned nb = blocks_for(z.E, 256);
  {
    Launch L(c, "ele_dt");
    hipLaunchKernelGGL(k_ele_dt, dim3(nb), dim3(256), 0, c.stream, z.E, z.S, z.F, z.Ff, c.detj, c.ws, c.wf, c.waveSp, c.da,
                       c.prm.cfl * cfl_limit(z.P), c.eleDt, c.partial);
    HIPCHK(hipGetLastError());
  }
  Launch L(c, "dt_min");
  hipLaunchKernelGGL(k_min_final, dim3(1), dim3(256), 0, c.stream, (int)nb, c.partial, c.d_dt);
  HIPCHK(hipGetLastError());
}

// Point groups of the norm's grid: at least kResBlocks blocks, two for each CU,
// where there are points for them.
static unsigned res_groups(const Sizes& z, unsigned nb) {
  return std::min<unsigned>(z.S, (kResBlocks + nb - 1) / nb);
}
// The norm into out[N] on the device: part holds the grid's rows of N.
static void launch_res_norm(Ctx& c, int type, double* part, double* out) {
  const Sizes& z = c.z;
  if (z.N > kResFields) throw std::invalid_argument("residual norm: too many fields");
  const unsigned nb = blocks_for(z.E, 256), ng = res_groups(z, nb);
  hipLaunchKernelGGL(k_res_norm, dim3(nb, ng), dim3(256), 0, c.stream, z.E, z.S, z.N, type, c.divF, c.detj, c.ws, part);
  HIPCHK(hipGetLastError());
  hipLaunchKernelGGL(k_res_final, dim3(1), dim3(256), 0, c.stream, (int)(nb * ng), z.N, type, part, out);
  HIPCHK(hipGetLastError());
}

void residual_norm(Ctx& c, int type, double* out) {
  double* fin = c.partial + (long long)blocks_for(c.z.E, 256) * res_groups(c.z, blocks_for(c.z.E, 256)) * c.z.N;
  launch_res_norm(c, type, c.partial, fin);
  HIPCHK(hipMemcpyAsync(out, fin, (size_t)c.z.N * sizeof(double), hipMemcpyDeviceToHost, c.stream));
  HIPCHK(hipStreamSynchronize(c.stream));
}

// ---------------------------------------------------------------------------
// Residual norm without allocation, for callers that cannot call hipMalloc.
// The per-block partial sums and the final N values live in `scratch`, a
// file-scope device array of kNoAllocScratch doubles that every GPU the
// library runs on holds until the process ends.  Host code never passes the
// array's name to a kernel (on the host it is a stand-in, not a device
// address): the device address of each GPU's copy is looked up once, with
// that GPU current, and kept in g_scratch_ptr.  Calls on one GPU share its
// copy, so calls that overlap on one GPU race; nothing in it has to start at
// zero (every value read was written earlier in the same call).
static __device__ __align__(256) double scratch[kNoAllocScratch];
static std::mutex g_scratch_mu;
static double* g_scratch_ptr[kNoAllocMaxDevices] = {};

double* noalloc_scratch(int device) {
  if (device < 0 || device >= kNoAllocMaxDevices) throw std::invalid_argument("device ordinal out of range");
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    int cur = -1;
    HIPCHK(hipGetDevice(&cur));
    if (cur != device) HIPCHK(hipSetDevice(device));
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != device) (void)hipSetDevice(cur);
    HIPCHK(e);
    g_scratch_ptr[device] = static_cast<double*>(p);
  }
  return g_scratch_ptr[device];
}

void residual_norm_noalloc(Ctx& c, int type, double* out) {
  const Sizes& z = c.z;
  const unsigned nb = blocks_for(z.E, 256);
  const long long need = ((long long)nb + 1) * z.N;
  if (need > kNoAllocScratch)
    throw std::length_error("fhip_residual_norm_noalloc: " + std::to_string(z.E) + " elements need " +
                            std::to_string(need) + " doubles of scratch, more than its maximum of " +
                            std::to_string(kNoAllocScratch) + " (at most " +
                            std::to_string((kNoAllocScratch / z.N - 1) * 256) + " elements)");
  double* part = noalloc_scratch(c.device);
  double* fin = part + kNoAllocScratch - z.N;
  launch_res_norm(c, type, part, fin);
  HIPCHK(hipMemcpyAsync(out, fin, (size_t)z.N * sizeof(double), hipMemcpyDeviceToHost, c.stream));
  HIPCHK(hipStreamSynchronize(c.stream));
}

int check_state(Ctx& c) {
  long long SE = (long long)c.z.S * c.z.E;
  int zero = 0, h = 0;
  HIPCHK(hipMemcpyAsync(c.flag, &zero, sizeof(int), hipMemcpyHostToDevice, c.stream));
  if (c.z.D == 2) hipLaunchKernelGGL(k_check<2>, dim3(blocks_for(SE, 256)), dim3(256), 0, c.stream, SE, c.U, c.ph.gamma, c.flag);
  else hipLaunchKernelGGL(k_check<3>, dim3(blocks_for(SE, 256)), dim3(256), 0, c.stream, SE, c.U, c.ph.gamma, c.flag);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpyAsync(&h, c.flag, sizeof(int), hipMemcpyDeviceToHost, c.stream));
  HIPCHK(hipStreamSynchronize(c.stream));
  return h;
}

}  // namespace fhip
