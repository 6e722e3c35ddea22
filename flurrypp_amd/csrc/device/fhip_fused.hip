// Fused tensor-product paths: FP64 ("fused") and mixed precision ("mixed").
//
// FlurryPP applies its FR operators as dense GEMMs (src/solver.cpp:556-1158),
// but on quads and hexes every operator row is non-zero only along one line
// of solution points: the Lagrange factors of the other directions are
// evaluated at their own nodes and are exactly 0 or 1.  These paths read the
// dense operators handed to fhip_create, keep only their non-zero entries
// (at most P+1 per row for extrapolation and gradient, one per face for the
// correction) and apply them inside fused kernels, so the sums are the dense
// products minus terms that are exactly zero.
//
// Data live element-major on the device ([ele][field][point]) so that a block
// of elements is one contiguous slab.  Per RK stage:
//   inviscid   stage      common flux of the element's own flux points, flux,
//                         divergence, correction, RK update, U at the faces
//   viscous    volume     common inviscid flux and LDG common U at the element's
//                         own flux points, corrected gradient, inviscid and
//                         viscous flux, divergence, this side's part of the LDG
//                         viscous flux, correction with all but the other
//                         side's part
//              rk         correction with the other sides' LDG parts, RK update,
//                         U at the faces of the next stage
//
// Every kernel is templated on R, the type of the face and volume
// intermediates and of the flux arithmetic: double for the FP64 path, float
// for the mixed path.  The solution, its RK stage copies, the metric terms,
// the wave speeds, dt and the residual array stay FP64 in both (the mixed
// path also keeps FP32 roundings of the geometry and of U for its kernels).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <map>
#include <mutex>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <stdexcept>
#include <type_traits>
#include <vector>

#include "fhip_internal.hpp"

namespace fhip {

#define FCHK(x)                                                                               \
  do {                                                                                        \
    hipError_t e_ = (x);                                                                      \
    if (e_ != hipSuccess) throw std::runtime_error(std::string("HIP: ") + hipGetErrorString(e_)); \
  } while (0)

static inline unsigned nblk(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

template <int D, int P>
struct Shape {
  static constexpr int P1 = P + 1;
  static constexpr int Ff = (D == 2) ? P1 : P1 * P1;
  static constexpr int S = (D == 2) ? P1 * P1 : P1 * P1 * P1;
  static constexpr int F = 2 * D * Ff;
  static constexpr int N = D + 2;
  static constexpr int NC = 2 * D;  // correction entries per solution point
};

// Element kernels take a runtime block of NT >= S threads holding EB = NT/S
// elements, with their LDS slabs in dynamic shared memory; the block size of
// each kernel is chosen per context (default 256, or by fused_autotune).
extern __shared__ __align__(16) unsigned char fhip_lds[];
constexpr int kMaxBlock = 512;
// Dynamic LDS that a block may take.  (The factors of the operators are up to 480
// bytes of static LDS more; a workgroup may have 160 KiB.)
constexpr size_t kMaxLds = 64 * 1024;
constexpr long long kStreamBytes = 64ll << 20;
// (kVolume: the stage kernel on inviscid runs; kFaceBnd: no kernel, the place in
// the block sizes' order remains)
enum { kExtrap = 0, kFaceInv = 1, kVolume = 2, kFaceBnd = 3, kRk = 4 };

// Sparse operator tables (device pointers into one allocation).  Indices of
// solution points are positions in the swizzled LDS layout (spt_lds below).
struct Tabs {
  const double* ext_w;  // [F][P1]    opp_spts_to_fpts entries (of the points in line)
  const int* efn_dir;   // [F]        the one direction d with opp_extrapolate_fn[d][f] != 0
  const double* efn_w;  // [F][P1]    opp_extrapolate_fn[efn_dir[f]] entries (same points)
  const int* grd_idx;   // [D][S][P1]
  const double* grd_w;  // [D][S][P1] opp_grad_spts entries
  const int* cor_idx;   // [S][NC]    flux points correcting solution point s
  const double* cor_w;  // [S][NC]    opp_correction entries
  const int* cu_idx;    // [D][S][2]  flux points with opp_correct_u[d][s][f] != 0
  const double* cu_w;   // [D][S][2]  their opp_correct_u entries
  // the same weights rounded to FP32 once, for the mixed path
  const float *ext_wf, *efn_wf, *grd_wf, *cor_wf, *cu_wf;
  // opp_grad_spts as one 1-D derivative matrix d1[i][m] (derivative of basis
  // m at point i) shared by every direction and line, FP64 and FP32; null
  // where the operator is not of that form (the fused paths then do not take
  // P3 hexes, whose FP64 volume kernel contracts with it on the matrix cores)
  const double* d1;
  const float* d1f;
  // operators of full tensor-product form (Ten below): their 1-D factors
  // [Ten::NW], FP64 and FP32, or null
  const double* w1;
  const float* w1f;
  // [F][(P1+3)/4] solution points feeding flux point f, one byte each (S <= 216)
  const unsigned* line;
};

// The 1-D contractions of FP64 P3 hexes along x and z run on the matrix
// cores (v_mfma_f64_4x4x4f64: four independent 4x4x4 products per wave).  One
// element per wave, lane L = solution point x + 4y + 16z.  The instruction
// takes A[i][k] of block b from lane 16k + 4b + i, B[k][j] from lane
// 16k + 4b + j, and returns D[i][j] = C[i][j] + sum_k A[i][k] B[k][j] in lane
// 16i + 4b + j (measured lane layout).  With b = y:
//   z: A = d1[L % 4][L / 16], B = the lane's own point: D is the z-derivative
//      at the lane's own point;
//   x: A = the point (x, z) = (L / 16, L % 4) of the lane's row y, B = the
//      same operator entry: D is the x-derivative at the lane's own point.
// C carries the terms added on the vector unit (the gradient's correction,
// the divergence's other directions).  y stays on the vector unit.
template <int D, int P, class R>
constexpr bool kMfma = D == 3 && P == 3 && sizeof(R) == 8;

__device__ __forceinline__ double mfma444(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float mfma444(float, float, float c) { return c; }  // never taken (kMfma)

// The mixed path's z contractions of P3 hexes on the matrix cores in BF16
// (v_mfma_f32_16x16x32_bf16, FP32 accumulation).  Both factors are split into
// BF16 pieces: x = p0 + p1 + p2 with p0 = bf16(x), p1 = bf16(x - p0),
// p2 = bf16(x - p0 - p1).  With 2 pieces (hi+lo) the product takes the terms
// d0 v0 + d0 v1 + d1 v0, with 3 also d0 v2 + d2 v0 + d1 v1 (the rest are
// below FP32 rounding).  One element per wave, lane L = point xy + 16 z
// (xy = L % 16).  The instruction takes A[i][k] from lane 16(k/8) + i, element
// k % 8, B[k][j] from lane 16(k/8) + j, element k % 8, and returns D[i][j] in
// lane 16(i/4) + j, register i % 4 (measured lane layout).  With j = xy, the
// rows i = 4z of A hold the pieces of d1[z][m] and the column xy of B the
// pieces of v(xy, m), m = 0..3, eight K slots per lane group g = L / 16:
//   2 pieces: g0: (d0 | d0) x (v0 | v1), g1: (d1 | 0) x (v0 | 0)
//   3 pieces: g0: (d0 | d0) x (v0 | v1), g1: (d1 | d0) x (v0 | v2),
//             g2: (d2 | d1) x (v0 | v1)
// so register 0 of each lane is the z contraction at the lane's own point.
__host__ __device__ constexpr int spt_lds(int D, int P1, int s);  // the slab position of point s (below)

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void bf16_pieces(float x, __bf16 p[3]) {
  p[0] = (__bf16)x;
  const float r1 = x - float(p[0]);
  p[1] = (__bf16)r1;
  p[2] = (__bf16)(r1 - float(p[1]));
}

// Which pieces lane group g puts in its two halves of eight K slots (-1: zero).
__device__ __forceinline__ void bf16_plan(int np, int g, int& da, int& db, int& va, int& vb) {
  da = db = va = vb = -1;
  if (g == 0) da = 0, db = 0, va = 0, vb = 1;
  if (g == 1) da = 1, db = (np == 3 ? 0 : -1), va = 0, vb = (np == 3 ? 2 : -1);
  if (g == 2 && np == 3) da = 2, db = 1, va = 0, vb = 1;
}

// A operand of lane L: the pieces of row z = (L % 16) / 4 of d1 for rows
// i = L % 16 with i % 4 == 0, else zero.
__device__ __forceinline__ bf16x8 bf16_opnd_a(const float* d1, int lane, int np) {
  bf16x8 a;
  for (int e = 0; e < 8; e++) a[e] = (__bf16)0.f;
  const int i = lane % 16, g = lane / 16;
  if (i % 4 != 0) return a;
  int da, db, va, vb;
  bf16_plan(np, g, da, db, va, vb);
  for (int m = 0; m < 4; m++) {
    __bf16 p[3];
    bf16_pieces(d1[(i / 4) * 4 + m], p);
    if (da >= 0) a[m] = p[da];
    if (db >= 0) a[4 + m] = p[db];
  }
  return a;
}

// The z contraction at the lane's own point plus c: v is this field's slab
// (swizzled LDS positions), column xy = lane % 16.
template <int D, int P1>
__device__ __forceinline__ float mfma_z_bf16(const float* v, int lane, bf16x8 a, float c, int np) {
  const int xy = lane % 16, g = lane / 16;
  int da, db, va, vb;
  bf16_plan(np, g, da, db, va, vb);
  bf16x8 bv;
  for (int e = 0; e < 8; e++) bv[e] = (__bf16)0.f;
  if (va >= 0) {
    for (int m = 0; m < 4; m++) {
      __bf16 p[3];
      bf16_pieces(v[spt_lds(D, P1, xy + 16 * m)], p);
      bv[m] = p[va];
      if (vb >= 0) bv[4 + m] = p[vb];
    }
  }
  const f32x4 cc = {c, 0.f, 0.f, 0.f};
  const f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bv, cc, 0, 0, 0);
  return d[0];
}

template <int D, int P, class R>
constexpr bool kBf16 = D == 3 && P == 3 && sizeof(R) == 4;


// Operator weights in the kernels' arithmetic type.
template <class R>
__device__ __forceinline__ const R* tw(const double* d, const float* f);
template <>
__device__ __forceinline__ const double* tw<double>(const double* d, const float*) { return d; }
template <>
__device__ __forceinline__ const float* tw<float>(const double*, const float* f) { return f; }

// Position of solution point s = i + P1*(j + P1*k) in an element's LDS slab.
// Hexes with an even P1: each (j,k) row is rotated by j+k and each k plane by
// k, so that the P1^2 points a face's flux points read at one depth fall into
// distinct LDS banks for all three face orientations (row-major order would
// give 4-way bank conflicts on the x and y faces at P=3).  With an odd P1 (rows
// of an odd number of doubles) and on quads, row-major order spreads the
// slab's reads over the banks at least as well (the rotation measured 48% of
// the P4 volume kernel's LDS cycles as bank conflicts).  A bijection on every
// plane.
__host__ __device__ constexpr int spt_lds(int D, int P1, int s) {
  if (D == 2 || P1 % 2 == 1) return s;
  const int i = s % P1, j = (s / P1) % P1, k = s / (P1 * P1);
  return (k * P1 + (j + k) % P1) * P1 + (i + k) % P1;
}

// The operators of a quad or hex by their 1-D factors: entry (point, m) sits on
// a line of the element, at a position that follows from the point's
// coordinates, and its weight is one of P1*P1 + 4*P1 numbers: the derivative
// matrix d1[i][m], the extrapolation to the low and high end l[side][m], the
// correction from the low and high end c[side][i].  A kernel keeps those in LDS
// and computes the positions.  Read from per-point tables instead (PtTab, FpTab:
// operators whose non-zeros have this pattern but other values) every use
// waits for two loads, the position and the weight, a chain through the caches
// in each phase; entries and their order are the same, so are the sums.
// Measured, tables -> factors: P4 channel 67x29, update and multigrid cycle 1005
// -> 941 us; 3-D vortex 23^3 P4 mixed, 4 steps 1841 -> 1711 us; Navier-Stokes
// Taylor-Green 37^3 P2, 4 steps 7.12 -> 6.91 ms, 48^3 P3 20.36 -> 20.15 ms.
template <int D, int P>
struct Ten {
  static constexpr int P1 = P + 1, NW = P1 * P1 + 4 * P1;
  static constexpr int L = P1 * P1, C = L + 2 * P1;  // offsets of l and c
  // slab position of the point at coordinates (i, j, k)
  __host__ __device__ static constexpr int pos(int i, int j, int k) {
    if (D == 2) return i + P1 * j;
    if (P1 % 2 == 1) return i + P1 * (j + P1 * k);
    int jk = j + k, ik = i + k;
    jk -= jk >= P1 ? P1 : 0;
    ik -= ik >= P1 ? P1 : 0;
    return (k * P1 + jk) * P1 + ik;
  }
  // Flux point f: the direction dn of its normal, whether it lies on the high
  // end, its coordinates in the other directions (getLocFpts,
  // src/points.cpp:67-162)
  struct Face {
    int dn, hi, c[3];
    __host__ __device__ explicit Face(int f) {
      c[0] = c[1] = c[2] = 0;
      if (D == 2) {
        const int face = f / P1, i = f - face * P1, a = face < 2 ? i : P - i;
        dn = (face & 1) ? 0 : 1;
        hi = face == 1 || face == 2;
        c[0] = dn == 0 ? 0 : a;
        c[1] = dn == 0 ? a : 0;
      } else {
        const int face = f / (P1 * P1), r = f - face * (P1 * P1), j = r / P1, i = r - j * P1;
        dn = face < 2 ? 2 : (face < 4 ? 0 : 1);
        hi = face & 1;
        const int a = (face == 1 || face == 3 || face == 4) ? P - i : i;
        c[0] = dn == 0 ? 0 : a;
        c[1] = dn == 0 ? a : (dn == 2 ? j : 0);
        c[2] = dn == 2 ? 0 : j;
      }
    }
    // the point of the flux point's line at depth m
    __host__ __device__ int at(int m) const {
      return pos(dn == 0 ? m : c[0], dn == 1 ? m : c[1], dn == 2 ? m : c[2]);
    }
  };
  struct Point {
    int c[3];
    __host__ __device__ explicit Point(int s) {
      c[0] = s % P1;
      c[1] = D == 2 ? s / P1 : (s / P1) % P1;
      c[2] = D == 2 ? 0 : s / (P1 * P1);
    }
    __host__ __device__ int line(int d, int m) const {
      return pos(d == 0 ? m : c[0], d == 1 ? m : c[1], d == 2 ? m : c[2]);
    }
  };
  // Face j's direction and end, and the flux point on it opposite a point
  __host__ __device__ static constexpr int face_dir(int j) { return D == 2 ? (j & 1 ? 0 : 1) : (j < 2 ? 2 : (j < 4 ? 0 : 1)); }
  __host__ __device__ static constexpr int face_hi(int j) { return D == 2 ? (j == 1 || j == 2) : (j & 1); }
  __host__ __device__ static int face_fpt(int j, const int* c) {
    if (D == 2) {
      const int a = j & 1 ? c[1] : c[0];
      return j * P1 + (j < 2 ? a : P - a);
    }
    const int a = j == 2 || j == 3 ? c[1] : c[0], b = j < 2 ? c[1] : c[2];
    return j * P1 * P1 + (j == 1 || j == 3 || j == 4 ? P - a : a) + P1 * b;
  }
  // the two faces normal to direction d, ascending
  __host__ __device__ static constexpr int dir_face(int d, int j) {
    return D == 2 ? (d == 0 ? 1 + 2 * j : 2 * j) : (d == 2 ? j : 2 * (d + 1) + j);
  }
};

// A solution point's operator entries.
template <int D, int P, class R>
struct PtTen {
  using T = Ten<D, P>;
  const R* w;
  typename T::Point p;
  __device__ PtTen(const struct Tabs&, const R* sW, int s) : w(sW), p(s) {}
  __device__ int grd_idx(int d, int m) const { return p.line(d, m); }
  __device__ R grd_w(int d, int m) const { return w[p.c[d] * T::P1 + m]; }
  __device__ int cor_idx(int j) const { return T::face_fpt(j, p.c); }
  __device__ R cor_w(int j) const { return w[T::C + T::face_hi(j) * T::P1 + p.c[T::face_dir(j)]]; }
  __device__ int cu_idx(int d, int j) const { return cor_idx(T::dir_face(d, j)); }
  __device__ R cu_w(int d, int j) const {
    const R c = cor_w(T::dir_face(d, j));
    return T::face_hi(T::dir_face(d, j)) ? c : -c;
  }
};
template <int D, int P, class R>
struct PtTab {
  static constexpr int P1 = P + 1, S = Shape<D, P>::S, NC = 2 * D;
  const Tabs& tb;
  int s;
  __device__ PtTab(const Tabs& t, const R*, int s_) : tb(t), s(s_) {}
  __device__ int grd_idx(int d, int m) const { return tb.grd_idx[(d * S + s) * P1 + m]; }
  __device__ R grd_w(int d, int m) const { return tw<R>(tb.grd_w, tb.grd_wf)[(d * S + s) * P1 + m]; }
  __device__ int cor_idx(int j) const { return tb.cor_idx[s * NC + j]; }
  __device__ R cor_w(int j) const { return tw<R>(tb.cor_w, tb.cor_wf)[s * NC + j]; }
  __device__ int cu_idx(int d, int j) const { return tb.cu_idx[(d * S + s) * 2 + j]; }
  __device__ R cu_w(int d, int j) const { return tw<R>(tb.cu_w, tb.cu_wf)[(d * S + s) * 2 + j]; }
};
// A flux point's operator entries: extrapolation weights (the sum over them,
// negated on a low end, is the normal flux's), normal direction.
template <int D, int P, class R>
struct FpTen {
  using T = Ten<D, P>;
  const R* w;
  int face;
  __device__ FpTen(const Tabs&, const R* sW, int fpt) : w(sW), face(fpt / Shape<D, P>::Ff) {}
  __device__ R ext_w(int m) const { return w[T::L + T::face_hi(face) * T::P1 + m]; }
  __device__ R efn_w(int m) const { return ext_w(m); }
  __device__ R efn_sign(R a) const { return T::face_hi(face) ? a : -a; }
  __device__ int dir() const { return T::face_dir(face); }
};
template <int D, int P, class R>
struct FpTab {
  static constexpr int P1 = P + 1;
  const Tabs& tb;
  int f;
  __device__ FpTab(const Tabs& t, const R*, int fpt) : tb(t), f(fpt) {}
  __device__ R ext_w(int m) const { return tw<R>(tb.ext_w, tb.ext_wf)[f * P1 + m]; }
  __device__ R efn_w(int m) const { return tw<R>(tb.efn_w, tb.efn_wf)[f * P1 + m]; }
  __device__ R efn_sign(R a) const { return a; }
  __device__ int dir() const { return tb.efn_dir[f]; }
};
template <int D, int P, class R, bool TEN>
using PtOp = std::conditional_t<TEN, PtTen<D, P, R>, PtTab<D, P, R>>;
template <int D, int P, class R, bool TEN>
using FpOp = std::conditional_t<TEN, FpTen<D, P, R>, FpTab<D, P, R>>;
// The 1-D factors into the block's LDS (a barrier follows before their use).
template <int D, int P, class R, bool TEN>
__device__ __forceinline__ void stage_factors(R* sW, const Tabs& tb) {
  if constexpr (TEN) {
    if (threadIdx.x < Ten<D, P>::NW) sW[threadIdx.x] = tw<R>(tb.w1, tb.w1f)[threadIdx.x];
  }
}

// The solution points of a flux point's line, by slab position in a byte each: a
// register or two, loaded with a kernel's first loads and kept for all its phases
// (computed, with the selects on the face's direction, they are some 100
// instructions).
template <int P1>
struct Packed {
  static constexpr int W = (P1 + 3) / 4;
  unsigned v[W];
  __device__ void load(const Tabs& tb, int f) {
#pragma unroll
    for (int j = 0; j < W; j++) v[j] = tb.line[f * W + j];
  }
  __device__ int operator[](int m) const { return (v[m / 4] >> (8 * (m % 4))) & 255; }
};
// Pointers to those points in an element's slab and their weights.  The fields of
// the slab are then at constant offsets, which LDS reads take for nothing: an
// address formed for each read (an add, often a multiply) and the weights read
// again for each field were a third of the viscous volume kernel's instructions.
template <int P1, class R>
struct LineOp {
  const R* q[P1];
  R w[P1];
  template <class At, class W>
  __device__ LineOp(const R* slab, const At& at, const W& weight) {
#pragma unroll
    for (int m = 0; m < P1; m++) q[m] = slab + at(m), w[m] = weight(m);
  }
  __device__ R operator()(int off) const {
    R a = 0;
#pragma unroll
    for (int m = 0; m < P1; m++) a += w[m] * q[m][off];
    return a;
  }
};

// Face and volume intermediates of one precision.
template <class R>
struct Work {
  R *divFe = nullptr, *Ufe = nullptr;
  // inviscid runs: U at the flux points of every second stage (a stage reads
  // one of Ufe, Ufe2 and writes the other; a call starts in Ufe)
  R* Ufe2 = nullptr;
  // viscous runs: each flux point's side of the LDG flux [ele][N][F] (divFe then
  // holds the divergence corrected with all but the other sides' parts)
  R* Bve = nullptr;
  R* Jne = nullptr;  // mixed path: the flux jump less the other side's part (divFe is then uncorrected)
  R* Rst = nullptr;  // mixed path: residual of each classical RK stage but the last
  // mixed path: U at the solution points rounded to FP32, the only form in
  // which the flux kernels read it; the RK stages inside a step keep their
  // states here and write the FP64 state only at the step's last stage
  R* Us = nullptr;
  // geometry in the kernels' arithmetic type: the FP64 arrays themselves, or
  // FP32 copies rounded once (the values the FP32 kernels would convert to)
  const R *JG = nullptr, *iJ = nullptr, *dA = nullptr, *nf = nullptr;
  void* geo_mem = nullptr;
  bool ready = false;
  void release() {
    void* ps[] = {divFe, Ufe, Bve, Jne, Rst, Us, geo_mem, Ufe2};
    for (void* p : ps)
      if (p) (void)hipFree(p);
    *this = Work<R>();
  }
};

// The kernels whose block sizes a run uses: FP64 0, mixed 1, mixed with 2 or 3 BF16
// pieces 2 or 3.
static int tune_form(const Ctx& c, bool mixed) { return mixed ? std::max(c.bf16, 1) : 0; }

struct FusedState {
  Tabs tb{};
  void* tab_mem = nullptr;
  // FP64 element-major state, metrics and wave speeds (both paths)
  double *Ue = nullptr, *Uacc = nullptr, *divF0e = nullptr, *JGe = nullptr, *detJe = nullptr,
         *iJe = nullptr, *norme = nullptr, *dAe = nullptr, *waveSpe = nullptr;
  // per element flux point, 4 * (partner flux point e*F + f) + side (0 left,
  // 1 right) or 4 * boundary slot + 2; the face's normal (the left element's)
  // at every element flux point; boundary codes by slot (behind fpart)
  int *fpart = nullptr, *bndBc = nullptr;
  double* nfe = nullptr;
  int nBnd = 0;
  // batching: boundary-state table, element -> mesh map, per-mesh dt and activity
  int nMesh = 1;
  std::vector<int> h_meshStart;
  double *bst = nullptr, *meshDt = nullptr, *meshRes = nullptr;
  double* dtAcc = nullptr;       // minimum of the blocks of the dt kernel that have finished (infinity between launches)
  unsigned* dtTicket = nullptr;  // their number (zero between launches), behind it
  double* vole = nullptr;        // element volumes, sum_s detJ w_s (calcDt's numerator)
  int *eleMesh = nullptr, *meshStart = nullptr, *active = nullptr;
  // P-multigrid source term (element-major copy of src_spts), used while use_src
  double* srce = nullptr;
  bool use_src = false;
  // the stage being formed reads its state from the stage copy Us (the
  // stages after the first of an RK step); otherwise from the state itself.
  // FP32 kernels always read the FP32 copy.
  bool read_stage = false;
  // inviscid runs: U at the flux points of the current state is in Ufe2.  A step of
  // an odd number of stages ends there (a copy back to Ufe took 2.4 of the 28.5 us
  // of a single-stage step of a channel 113x41 P3).
  bool flipped = false;
  // stream once-touched arrays past the caches: set when U alone (FP64,
  // element-major) exceeds kStreamBytes, i.e. a stage's arrays are many times
  // the 256 MiB infinity cache
  bool stream = false;
  // block size of each kernel (kExtrap..kRk), by tune_form()
  int nt[4][5] = {{256, 256, 256, 256, 256},
                  {256, 256, 256, 256, 256},
                  {256, 256, 256, 256, 256},
                  {256, 256, 256, 256, 256}};
  Work<double> w64;
  Work<float> w32;
  ~FusedState() {
    w64.release();
    w32.release();
    void* ps[] = {tab_mem, Ue,  Uacc,   divF0e,  JGe,     detJe,     iJe,    norme, dAe,      waveSpe, fpart,
                  nfe,     bst, meshDt, meshRes, eleMesh, meshStart, active, srce,  dtAcc,    vole};
    for (void* p : ps)
      if (p) (void)hipFree(p);
  }
  template <class R>
  Work<R>& work();
};
template <>
inline Work<double>& FusedState::work<double>() { return w64; }
template <>
inline Work<float>& FusedState::work<float>() { return w32; }

// ---------------------------------------------------------------------------
// Minimum over the block (a multiple of 64 threads), returned to every thread:
// across each wave by lane exchanges, then across the waves through red, one
// entry each.  min is exact, so the order of the comparisons does not matter.
__device__ __forceinline__ double block_min(double v, double* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o));
  __syncthreads();  // red may still be read by an earlier call
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  v = red[0];
  for (int w = 1; w < (int)(blockDim.x >> 6); w++) v = fmin(v, red[w]);
  return v;
}

// The minimum of `blocks` blocks' minima (thread 0 of each calls this) at out, put
// there by the block that finishes last, which also sets counter and accumulator
// back (0, infinity) for the next launch; a single block's minimum is the result at
// once.  Through atomics alone: a release here would write back what the kernel
// before left in the L2, which took longer than all else.  The minimum's own result
// is waited for, so it is in place before the block is counted, and the last
// block's exchange comes after all of them.
__device__ __forceinline__ void grid_min(double bmin, unsigned blocks, double* acc, unsigned* ticket, double* out) {
  if (blocks == 1) {
    *out = bmin;
    return;
  }
  const double before = __hip_atomic_fetch_min(acc, bmin, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0)" ::"v"(before) : "memory");
  const unsigned t = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (t != blocks - 1) return;
  *out = __hip_atomic_exchange(acc, double(INFINITY), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

#ifndef FHIP_FAMILY
// Layout conversions between FlurryPP's [pt][ele][k] and element-major
// [ele][k][pt]: both are the transpose of a matrix with one row per point,
// [P][E*K] <-> [E*K][P].  32x32 tiles through LDS so that reads and writes
// are both coalesced; tiles are numbered on a 1-D grid over all the arrays that
// a call converts at one place (Layouts): on a small mesh each launch is some 4
// us.  One each -> together: a step of the 8x8 P3 vortex 55 -> 49 us, update and
// cycle of the P4 channel 67x29 690 -> 652 us.
//
// The same launch puts the minimum of an array at one place (Least), in blocks after
// the tiles: the solver's dt after local time steps, whose elements' the stage
// kernel forms (a launch of its own per level would be some 4 us of a call's 600).
constexpr int kTile = 32, kMaxLayouts = 16, kMaxLeast = 8;
constexpr long long kLeastPerBlock = 4096;
struct LayoutJobs {
  int n = 0, nLeast = 0;
  unsigned tiles = 0, blocks = 0;  // blocks: tiles and the minima's blocks
  struct Job {
    long long R, C;  // in [R][C] -> out [C][R]
    const double* in;
    double* out;
    unsigned first;  // its first tile
  } job[kMaxLayouts];
  struct Least {
    long long n;
    const double* in;
    double *acc, *out;
    unsigned* ticket;
    unsigned first, blocks;  // its first block after the tiles, their number
  } least[kMaxLeast];
};
static __global__ __launch_bounds__(256) void k_transpose(LayoutJobs jobs) {
  __shared__ double t[kTile][kTile + 1];
  if (blockIdx.x >= jobs.tiles) {
    const unsigned b = blockIdx.x - jobs.tiles;
    int n = 0;
    while (n + 1 < jobs.nLeast && b >= jobs.least[n + 1].first) n++;
    const LayoutJobs::Least& lb = jobs.least[n];
    double v = INFINITY;
    for (long long i = (long long)(b - lb.first) * blockDim.x + threadIdx.x; i < lb.n; i += (long long)lb.blocks * blockDim.x)
      v = fmin(v, lb.in[i]);
    v = block_min(v, &t[0][0]);
    if (threadIdx.x == 0) grid_min(v, lb.blocks, lb.acc, lb.ticket, lb.out);
    return;
  }
  int n = 0;
  while (n + 1 < jobs.n && blockIdx.x >= jobs.job[n + 1].first) n++;
  const LayoutJobs::Job& jb = jobs.job[n];
  const long long R = jb.R, C = jb.C;
  const double* const __restrict__ in = jb.in;
  double* const __restrict__ out = jb.out;
  const unsigned tilesC = (unsigned)((C + kTile - 1) / kTile), tile = blockIdx.x - jb.first;
  const long long r0 = (long long)(tile / tilesC) * kTile, c0 = (long long)(tile % tilesC) * kTile;
  const int tx = threadIdx.x % kTile, ty = threadIdx.x / kTile;  // ty 0..7
#pragma unroll
  for (int j = 0; j < kTile; j += 8) {
    const long long r = r0 + ty + j, c = c0 + tx;
    if (r < R && c < C) t[ty + j][tx] = in[r * C + c];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kTile; j += 8) {
    const long long c = c0 + ty + j, r = r0 + tx;
    if (r < R && c < C) out[c * R + r] = t[tx][ty + j];
  }
}

// The conversions of one place of a call, launched together (go, or when full).
// They must not depend on each other.
struct Layouts {
  hipStream_t st;
  LayoutJobs jobs;
  explicit Layouts(hipStream_t s) : st(s) {}
  void least(long long n, const double* in, double* acc, unsigned* ticket, double* out) {
    if (jobs.nLeast == kMaxLeast) go();
    const unsigned blocks = (unsigned)((n + kLeastPerBlock - 1) / kLeastPerBlock);
    jobs.least[jobs.nLeast++] = LayoutJobs::Least{n, in, acc, out, ticket, jobs.blocks - jobs.tiles, blocks};
    jobs.blocks += blocks;
  }
  void add(long long R, long long C, const double* in, double* out) {
    if (R == 0 || C == 0) return;
    const long long tiles = ((R + kTile - 1) / kTile) * ((C + kTile - 1) / kTile);
    if (jobs.n == kMaxLayouts || jobs.blocks + tiles > 0x7fffffffll) go();
    jobs.job[jobs.n++] = LayoutJobs::Job{R, C, in, out, jobs.tiles};
    jobs.tiles += (unsigned)tiles;
    jobs.blocks += (unsigned)tiles;
  }
  // in [P][E][K] -> out [E][K][P]
  void to_em(int P, long long E, int K, const double* in, double* out) { add(P, E * K, in, out); }
  // in [E][K][P] -> out [P][E][K]
  void from_em(int P, long long E, int K, const double* in, double* out) { add(E * K, P, in, out); }
  void go() {
    if (jobs.blocks) {
      hipLaunchKernelGGL(k_transpose, dim3(jobs.blocks), dim3(256), 0, st, jobs);
      FCHK(hipGetLastError());
    }
    jobs = LayoutJobs();
  }
};
#endif  // FHIP_FAMILY

// ---------------------------------------------------------------------------
// U at the flux points from U at the solution points (opp_spts_to_fpts rows).
template <int D, int P, class R, bool TEN>
__global__ __launch_bounds__(kMaxBlock) void k_extrap(int E, const double* __restrict__ Ue, R* __restrict__ Ufe,
                                                       R* __restrict__ Us, Tabs tb) {
  using Sh = Shape<D, P>;
  constexpr int S = Sh::S, F = Sh::F, N = Sh::N, P1 = Sh::P1;
  __shared__ R sW[Ten<D, P>::NW];
  stage_factors<D, P, R, TEN>(sW, tb);
  const int EB = blockDim.x / S;
  R* const sU = reinterpret_cast<R*>(fhip_lds);
  const int e0 = blockIdx.x * EB, nb = min(EB, E - e0);
  const double* src = Ue + (long long)e0 * N * S;
  // all loads first (at most N per thread), then the stores
  R v[N];
#pragma unroll
  for (int u = 0; u < N; u++) {
    const int i = threadIdx.x + u * blockDim.x;
    if (i < nb * N * S) v[u] = R(src[i]);
  }
#pragma unroll
  for (int u = 0; u < N; u++) {
    const int i = threadIdx.x + u * blockDim.x;
    if (i < nb * N * S) {
      const int r = i / S, q = i - r * S;
      sU[r * S + spt_lds(D, P1, q)] = v[u];
      if (Us) Us[(long long)e0 * N * S + i] = v[u];
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < nb * F; i += blockDim.x) {
    int b = i / F, f = i - b * F;
    const FpOp<D, P, R, TEN> fp(tb, sW, f);
    Packed<P1> lp;
    lp.load(tb, f);
    const LineOp<P1, R> line(sU + b * N * S, [&](int m) { return lp[m]; }, [&](int m) { return fp.ext_w(m); });
    R* const o = Ufe + (long long)(e0 + b) * N * F + f;
#pragma unroll
    for (int k = 0; k < N; k++) o[k * F] = line(k * S);
  }
}

// Loads and stores of arrays a kernel touches once per launch.  On meshes
// whose arrays are far larger than the caches (NT) they stream past them
// (nontemporal); on smaller ones they stay plain, since there the next kernel
// of the stage finds them in L2 or the infinity cache (measured both ways).
// A kernel streams only where the rows it stores are whole 64-byte blocks
// (Runner::kEleRowsWhole).
template <bool NT, class T>
__device__ __forceinline__ T ld_s(const T* p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}
template <bool NT, class T>
__device__ __forceinline__ void st_s(T v, T* p) {
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}
// A product meant to be rounded on its own before a following add.
__device__ __forceinline__ double mul_rn(double a, double b) { return __dmul_rn(a, b); }
__device__ __forceinline__ float mul_rn(float a, float b) { return __fmul_rn(a, b); }

// ---------------------------------------------------------------------------
// Common inviscid flux at face flux points; pL/pR are ele*F+fpt.
// Boundary state of a face flux point: the packed code holds the BC number in
// its low 4 bits and (row of the boundary-state table + 1) above them.
template <int D, class R>
__device__ __forceinline__ void bc_state(int code, const R* UL, const R* n, R* UR, const Phys& ph,
                                         const double* __restrict__ bst) {
  const int bc = code & 15, row = (code >> 4) - 1;
  if (row < 0) {
    apply_bc<D, R>(bc, UL, n, UR, ph);
  } else {
    Phys q = ph;
    q.rho_bound = bst[row * 5 + 0];
    q.u_bound = bst[row * 5 + 1];
    q.v_bound = bst[row * 5 + 2];
    q.w_bound = bst[row * 5 + 3];
    q.p_bound = bst[row * 5 + 4];
    apply_bc<D, R>(bc, UL, n, UR, q);
  }
}

// The common inviscid flux fn of a point pair (left and right state, the left
// element's normal); true where the flux has a wave speed lam (Roe has none).
template <int D, class R>
__device__ __forceinline__ bool pair_flux(bool bnd, const R* UL, const R* UR, const R* n, R* fn, const Phys& ph,
                                          double& lam) {
  if constexpr (D == 2) {
    if (ph.riemann_type != 0 && !bnd) {
      roe2d<R>(UL, UR, n, fn, R(ph.gamma));
      return false;
    }
  }
  lam = double(rusanov<D, R>(UL, UR, n, fn, R(ph.gamma)));
  return true;
}

// ---------------------------------------------------------------------------
// Correction of the divergence (correctDivFlux), RK update (timeStepA/B
// folded into one pass per stage, FP64) and U at the flux points for the
// next stage.  mode: 0 first classical stage, 1 middle classical stage,
// 2 last classical stage, 3 single-stage forward Euler, 4 Jameson-form stage,
// 6 first Jameson-form stage; 5, 7 and 8 the residual alone (see rk_point).
// Classical stages combine into U0 - sum_j b_j r_j (dt / detJ) in timeStepB's
// order (src/solver.cpp:504-536): either through the FP64 accumulator Uacc, or
// (mixed path, Rst given) from the stored stage residuals, which FP32 holds
// exactly there since they are sums of FP32 values; both give the same bits.
struct RkB {
  double b[8];
};
// The RK update's inputs and outputs besides the flux jump and divF: the
// stage's mode and coefficients, dt (0 global, 1 per element, 2 per mesh),
// the FP64 state and its stage copies, batching and multigrid arrays.
template <class R>
struct RkArgs {
  int mode;
  double a, bcoef;
  const double* detJe;
  const double* dtp;
  const double* eleDt;
  int local;
  double* Ue;
  double* Uacc;
  double* divF0e;
  const int* eleMesh;
  const double* meshDt;
  const int* active;
  const double* srce;
  R* Rst;
  int stage;
  RkB bs;
  R* Us;
  int fin;
  R* Ufe;
  double* makeSrc;  // MK instances of the stage kernel: srce, to be written
};

// What the update of one solution point reads besides its flux jump and divF,
// loaded ahead of the phases that form those (rk_load), so that the loads are in
// flight meanwhile: a launch on a small mesh is a chain of such waits.
template <int D, class R>
struct RkIn {
  static constexpr int N = D + 2;
  double dj, dt;
  double u[N];    // U at the step's start (its U0; U itself in the first stage)
  double acc[N];  // RK accumulator; mode 7: the source that the residual is taken from
  double src[N];  // P-multigrid source
  R rs[3][N];     // mixed path, last stage: the residuals of the first three stages
  bool frozen;
};

template <int D, int P, class R, bool NT>
__device__ __forceinline__ RkIn<D, R> rk_load(int E, long long e, int s, const RkArgs<R>& ra) {
  using Sh = Shape<D, P>;
  constexpr int S = Sh::S, N = Sh::N;
  RkIn<D, R> in{};
  const int mode = ra.mode;
  const long long at = e * N * S + s;
  if (mode == 5 || mode == 7 || mode == 8) {
#pragma unroll
    for (int k = 0; k < N; k++) {
      if (mode == 7) in.acc[k] = ra.divF0e[at + k * S];
      if (mode == 8) in.src[k] = ra.srce[at + k * S];
    }
    return in;
  }
  in.dj = ld_s<NT>(&ra.detJe[e * S + s]);
  // (the state itself is the step's U0 until the last stage writes it)
#pragma unroll
  for (int k = 0; k < N; k++) in.u[k] = ld_s<NT>(&ra.Ue[at + k * S]);
  if (!ra.Rst && (mode == 1 || mode == 2)) {
#pragma unroll
    for (int k = 0; k < N; k++) in.acc[k] = ld_s<NT>(&ra.Uacc[at + k * S]);
  }
  if (ra.srce) {
#pragma unroll
    for (int k = 0; k < N; k++) in.src[k] = ra.srce[at + k * S];
  }
  if (sizeof(R) == 4 && ra.Rst && mode == 2) {
#pragma unroll
    for (int j = 0; j < 3; j++)
      if (j < ra.stage) {
#pragma unroll
        for (int k = 0; k < N; k++) in.rs[j][k] = ld_s<NT>(&ra.Rst[j * ((long long)E * N * S) + at + k * S]);
      }
  }
  in.dt = ra.local == 1 ? ra.eleDt[e] : (ra.local == 2 ? ra.meshDt[ra.eleMesh[e]] : *ra.dtp);
  in.frozen = ra.active && !ra.active[ra.eleMesh[e]];
  return in;
}

// correctDivFlux at a point of the block's element b, from the flux jump in sD:
// out[k] is the correction of field k plus dv[k].
template <int D, int P, class R, class Op>
__device__ __forceinline__ void correction(const R* sD, int b, const Op& po, const R* dv, R* out) {
  using Sh = Shape<D, P>;
  const LineOp<Sh::NC, R> line(sD + b * Sh::N * Sh::F, [&](int j) { return po.cor_idx(j); },
                               [&](int j) { return po.cor_w(j); });
#pragma unroll
  for (int k = 0; k < Sh::N; k++) out[k] = line(k * Sh::F) + dv[k];
}

// correctDivFlux and timeStepA/B at point s of the block's element b: dv holds
// its divF (one value per field), sD the flux jump at the block's flux points,
// and sU receives the new state (its previous contents are no longer read).
// The increment is coefficient * residual * (dt / detJ), one division per point.
// MK (a multigrid level's first smoothing stage): the source becomes itself less
// the residual that the stage forms, before it is used.
template <int D, int P, class R, bool NT, bool TEN, bool MK = false>
__device__ __forceinline__ void rk_point(int E, long long e, int b, int s, const R* dv, R* sU, const R* sD, const R* sW,
                                         const RkIn<D, R>& in, const RkArgs<R>& ra, const Tabs& tb) {
  using Sh = Shape<D, P>;
  constexpr int S = Sh::S, N = Sh::N, P1 = Sh::P1;
  const int mode = ra.mode;
  const PtOp<D, P, R, TEN> po(tb, sW, s);
  R res[N];
  correction<D, P, R>(sD, b, po, dv, res);
  const long long at = e * N * S + s;
  if (mode == 5 || mode == 7 || mode == 8) {
    // residual only (calcResidual(0) + correctDivFlux), no update: 5 into
    // divF_spts[0]; 7 subtracted in place from the array divF0e points to
    // (the P-multigrid source); 8 plus the source into divF_spts[0]
#pragma unroll
    for (int k = 0; k < N; k++) {
      const double r0 = double(res[k]);
      if (mode == 7) ra.divF0e[at + k * S] = in.acc[k] - r0;
      else st_s<NT>(mode == 8 ? r0 + in.src[k] : r0, &ra.divF0e[at + k * S]);
    }
    return;
  }
  const double q = in.dt / in.dj;
  R* const qu = sU + b * N * S + spt_lds(D, P1, s);
#pragma unroll
  for (int k = 0; k < N; k++) {
    const long long iu = at + k * S;
    const double r0 = double(res[k]);
    if (ra.divF0e) st_s<NT>(r0, &ra.divF0e[iu]);
    // P-multigrid source: divF_spts[step] + src_spts (src/solver.cpp:480,514)
    double src = in.src[k];
    if constexpr (MK) {
      src -= r0;
      ra.makeSrc[iu] = src;
    }
    const double r = ra.srce ? r0 + src : r0;
    const double u = in.u[k];
    double un;
    if (mode == 0) {
      if (ra.Rst) st_s<NT>(R(r), &ra.Rst[iu]);
      else st_s<NT>(u - ra.bcoef * r * q, &ra.Uacc[iu]);
      un = u - ra.a * r * q;
    } else if (mode == 1) {
      if (ra.Rst) st_s<NT>(R(r), &ra.Rst[ra.stage * ((long long)E * N * S) + iu]);
      else st_s<NT>(in.acc[k] - ra.bcoef * r * q, &ra.Uacc[iu]);
      un = u - ra.a * r * q;
    } else if (mode == 2) {
      double acc = in.acc[k];
      if (ra.Rst) {
        acc = u;
#pragma unroll
        for (int j = 0; j < 3; j++)
          if (j < ra.stage) acc = acc - ra.bs.b[j] * double(in.rs[j][k]) * q;
#pragma unroll
        for (int j = 3; j < 7; j++)  // constant indices: the arguments stay out of scratch
          if (j < ra.stage) acc = acc - ra.bs.b[j] * double(ld_s<NT>(&ra.Rst[j * ((long long)E * N * S) + iu])) * q;
      }
      un = acc - ra.bcoef * r * q;
    } else if (mode == 3) {
      un = u - ra.bcoef * r * q;
    } else {
      un = u - ra.a * r * q;
    }
    if (in.frozen) un = u;
    // the state is written at the step's last stage only (earlier stages
    // leave it at the step's start, its U0, and write the stage copy); the
    // FP32 copy is written at the last stage too (the flux kernels read U
    // only through it), the FP64 one is not (the next step's first stage
    // reads the state itself)
    if (ra.fin) st_s<NT>(un, &ra.Ue[iu]);
    if (sizeof(R) == 4 || !ra.fin) st_s<NT>(R(un), &ra.Us[iu]);
    qu[k * S] = R(un);
  }
}

// extrapolateU at flux point i of the block, from the states in sU.
template <int D, int P, class R, bool NT, bool TEN>
__device__ __forceinline__ void face_point(int i, int e0, const Packed<P + 1>& lp, const R* sU, const R* sW, R* Ufe,
                                           const Tabs& tb) {
  using Sh = Shape<D, P>;
  constexpr int S = Sh::S, F = Sh::F, N = Sh::N, P1 = Sh::P1;
  const int bb = i / F, f = i - bb * F;
  const FpOp<D, P, R, TEN> fp(tb, sW, f);
  const LineOp<P1, R> line(sU + bb * N * S, [&](int m) { return lp[m]; }, [&](int m) { return fp.ext_w(m); });
  R* const o = Ufe + (long long)(e0 + bb) * N * F + f;
#pragma unroll
  for (int k = 0; k < N; k++) st_s<NT>(line(k * S), &o[k * F]);
}

// Shapes whose volume kernel is held to 4 waves per SIMD (128 VGPRs): quads
// and the FP32 path (but its BF16 forms).  FP64 hexes need more registers and are held to 3.
template <int D, class R>
constexpr bool kHold = D == 2 || sizeof(R) == 4;

// The volume kernel's flux-point inputs and outputs.
template <class R>
struct VFace {
  const int* fpart;    // [E*F] 4 * partner flux point + side, or 4 * boundary slot + 2
  const R* Ufe;        // [E][N][F] U at the flux points
  const R* nfe;        // [E][D][F] the face's normal (its left element's)
  const R* dA;         // [E][F] face area factor
  R* Bve;              // [E][N][F] this side's part of the LDG flux . n (interior points)
  R* Jne;              // [E][N][F] kJumpOut: the flux jump, less the other side's part
  double* wave;        // wave speeds of the left and boundary points, or null: not read before they change again
  const int* bndBc;    // [nBnd] boundary code (number and state row) by slot
  const double* bst;   // boundary-state table
};

// calcDivF_spts at point s of the block's element b, from the transformed flux in
// sF: the sum over directions in order (matrix cores: y on the vector unit, then
// z and x added).
template <int D, int P, class R, int np, class Op>
__device__ __forceinline__ void divergence(const R* sF, int b, int s, int sw, int swx, R opv, bf16x8 abf, const Op& po,
                                           R* dv) {
  using Sh = Shape<D, P>;
  constexpr int S = Sh::S, N = Sh::N, P1 = Sh::P1;
  constexpr bool mf = kMfma<D, P, R>;
  const R* const f0 = sF + b * D * N * S;
#pragma unroll
  for (int d = 0; d < D; d++) {
    if (mf && d != 1) continue;
    if constexpr (np != 0) {
      if (d == 2) {
#pragma unroll
        for (int k = 0; k < N; k++)
          dv[k] = mfma_z_bf16<D, P1>(reinterpret_cast<const float*>(f0 + (2 * N + k) * S), s, abf, dv[k], np);
        continue;
      }
    }
    const LineOp<P1, R> line(f0 + d * N * S, [&](int m) { return po.grd_idx(d, m); },
                             [&](int m) { return po.grd_w(d, m); });
#pragma unroll
    for (int k = 0; k < N; k++) {
      const R a = line(k * S);
      dv[k] = (d == 0 || mf) ? a : a + dv[k];
    }
  }
  if (mf) {
    const R *const qz = f0 + 2 * N * S + sw, *const qx = f0 + swx;
#pragma unroll
    for (int k = 0; k < N; k++) {
      dv[k] = mfma444(opv, qz[k * S], dv[k]);
      dv[k] = mfma444(qx[k * S], opv, dv[k]);
    }
  }
}

// ---------------------------------------------------------------------------
// Stage kernel of inviscid runs: one launch per RK stage.  Each element forms
// the common flux at its own flux points from U there and across (the left
// element's order of arguments and normal on both sides, so that both form the
// same bits), the flux and its divergence, the correction and the RK update,
// and writes U at its flux points for the next stage into a second array
// (neighbours still read the first).
//
// What it replaces: a face kernel that wrote the common flux once per point
// pair and a volume kernel that read it back.  A stage is then one dependent
// launch instead of two, which is what bounds small meshes (about 4.6 us per
// launch in a captured graph), and on large ones the flux array's write and
// two reads go (5.8 kB per P3 hex and stage) for one more read of U at the
// flux points.  The common flux is evaluated on both sides of a pair; the
// boundary states' code is compiled into the BND instances only, which meshes
// without boundary faces do not take.
//
// Measured, two kernels -> one: 2-D vortex 32x32 P3, 20 RK44 steps 842 -> 683 us;
// 3-D vortex 17^3 P2, 10 steps 1351 -> 1132 us; 23^3 P4 mixed, 4 steps 2140 ->
// 1841 us; P4 channel 67x29, update and multigrid cycle 1142 -> 1005 us.  With
// the points apart, the update's inputs loaded early and one division per point
// (below): vortex 663 -> 587 us, channel 941 -> 678 us, 17^3 P2 1109 -> 903 us.
//
// Steady runs (local time steps, 2-D) also form the element's time step here,
// in the step's first stage: it needs only the element's own wave speeds.
template <class R>
struct StageFace {
  const int* fpart;    // [E*F] 4 * partner flux point + side, or 4 * boundary slot + 2
  const R* Ufe;        // [E][N][F] U at the flux points, this stage's
  const R* Fne;        // [E][N][F] kGiven: the common flux, at left and boundary points
  const R* nfe;        // [E][D][F] the face's normal (its left element's)
  const R* dA;         // [E][F] face area factor
  double* wave;        // wave speeds of the left and boundary points, or null: not read before they change again
  const int* bndBc;    // [nBnd] boundary code (number and state row) by slot
  const double* bst;   // boundary-state table
  // local time step formed here, or wf null: from the wave speeds left by the
  // stage before, or (MK) those of this stage where it forms them
  const double *wf, *wavein, *dAd, *vole;
  double cflfac;
  double* eleDt;
};

// Two forms.  Apart: a block's threads are the solution points' waves and then
// the flux points' (stage_threads), so that the two kinds of work of a phase run
// side by side: the common flux beside the flux at the points, the flux jump
// beside the divergence; the update's inputs (2-D) are loaded with the slab.  On
// a small mesh, where a CU holds a few waves, a launch takes as long as the
// instructions and waits of one wave, and this shortens them.  Together: a
// thread does a solution point and then ceil(F/S) flux points; more elements are
// in flight per register, which is what counts once the mesh fills the chip
// (kApartWaves below).
__host__ __device__ constexpr int up64(int n) { return (n + 63) / 64 * 64; }

//
// FORM: the usual one; kMakeSrc, a multigrid level's first smoothing stage (rk_point's
// MK); kGiven, a single-stage step whose common flux was formed with the wave speeds
// that its time step needs (k_wave_dt): it is read, once per pair, and U at the flux
// points is not, so the new one takes its place.  Formed again here a step of
// channels 200x150 P2 took 46.8 us (in two kernels 42.1), now 43.0; mixed 41.5 (34.6), 36.2.
enum { kUsual = 0, kMakeSrc = 1, kGiven = 2 };
template <int D, int P, class R, bool NT, bool BND, bool TEN, bool APART, int BF, int FORM>
__device__ __forceinline__ void stage_body(int E, int EB, const double* __restrict__ Ue, const R* __restrict__ Us,
                                           const R* __restrict__ JGe, const StageFace<R>& fc, const Tabs& tb,
                                           const Phys& ph, const RkArgs<R>& ra) {
  using Sh = Shape<D, P>;
  constexpr int S = Sh::S, F = Sh::F, N = Sh::N, P1 = Sh::P1;
  constexpr bool MK = FORM == kMakeSrc, GV = FORM == kGiven;
  // U, the transformed flux and the flux jump of the block's elements:
  // [EB*N*S] [EB*D*N*S] [EB*N*F]
  R* const sU = reinterpret_cast<R*>(fhip_lds);
  R* const sF = sU + EB * N * S;
  R* const sD = sF + EB * D * N * S;
  // [EB*F] each flux point's term of the local time step: in sD, which the flux
  // jump takes over later, or (MK) behind it
  double* const sT = reinterpret_cast<double*>(MK ? sD + EB * N * F : sD);
  __shared__ R sW[Ten<D, P>::NW];
  stage_factors<D, P, R, TEN>(sW, tb);
  const int e0 = blockIdx.x * EB, nb = min(EB, E - e0);
  const int b = threadIdx.x / S, s = threadIdx.x - b * S;
  const int sw = spt_lds(D, P1, s);
  const bool act = (int)threadIdx.x < nb * S;  // a solution point's thread
  const long long e = e0 + b;
  // the thread's flux points: fi(u) < nP (negative: none)
  constexpr int KF = APART ? 1 : (F + S - 1) / S;
  const int fb = APART ? up64(EB * S) : 0, nP = nb * F;
  auto fi = [&](int u) { return (int)threadIdx.x - fb + u * (int)blockDim.x; };
  auto flx = [&](int u) { return (!APART || fi(u) >= 0) && fi(u) < nP; };
  constexpr bool mf = kMfma<D, P, R>;
  constexpr int np = kBf16<D, P, R> ? BF : 0;
  bf16x8 abf = {};
  if constexpr (np != 0) abf = bf16_opnd_a(tw<float>(tb.d1, tb.d1f), s % 64, np);
  const int swx = mf ? spt_lds(D, P1, s / 16 + 4 * ((s / 4) % 4) + 16 * (s % 4)) : 0;
  const R opv = mf ? tw<R>(tb.d1, tb.d1f)[(s % 4) * P1 + s / 16] : R(0);
  const bool fold = D == 2 && fc.wf;
  // the flux points' side codes first: the partners' addresses come from them
  int cd[KF];
  Packed<P1> lp[KF];
#pragma unroll
  for (int u = 0; u < KF; u++) {
    cd[u] = flx(u) ? fc.fpart[(long long)e0 * F + fi(u)] : 0;
    lp[u].load(tb, flx(u) ? fi(u) % F : 0);
  }
  R vu[N];
#pragma unroll
  for (int u = 0; u < N; u++) {
    const int i = threadIdx.x + u * blockDim.x;
    if (i < nb * N * S)
      vu[u] = Us ? ld_s<NT>(&Us[(long long)e0 * N * S + i]) : R(ld_s<NT>(&Ue[(long long)e0 * N * S + i]));
  }
  R G[D][D] = {};
  RkIn<D, R> in{};
  if (act) {
#pragma unroll
    for (int r = 0; r < D; r++)
#pragma unroll
      for (int x = 0; x < D; x++) G[r][x] = JGe[((e * D + r) * D + x) * S + s];
    if constexpr (APART && D == 2) in = rk_load<D, P, R, NT>(E, e, s, ra);
  }
  R own[N], oth[N], n[D], dA = 0, fo[KF][N];
  // U at flux point u and across, its normal and dA
  auto load_face = [&](int u) {
    const int i = fi(u), bb = i / F, f = i - bb * F;
    const long long ob = (long long)(e0 + bb) * N * F + f;
    if constexpr (GV) {
      // the common flux, at the pair's left point
      dA = ld_s<NT>(&fc.dA[(long long)e0 * F + i]);
      long long pb = ob;
      if ((cd[u] & 3) == 1) {
        const int p = cd[u] >> 2, ep = p / F;
        pb = (long long)ep * N * F + (p - ep * F);
      }
#pragma unroll
      for (int k = 0; k < N; k++) fo[u][k] = fc.Fne[pb + k * F];
      return;
    }
#pragma unroll
    for (int k = 0; k < N; k++) own[k] = fc.Ufe[ob + k * F];
#pragma unroll
    for (int x = 0; x < D; x++) n[x] = ld_s<NT>(&fc.nfe[((long long)(e0 + bb) * D + x) * F + f]);
    dA = ld_s<NT>(&fc.dA[(long long)e0 * F + i]);
    long long pb = ob;
    if (!BND || (cd[u] & 3) != 2) {
      const int p = cd[u] >> 2, ep = p / F;
      pb = (long long)ep * N * F + (p - ep * F);
    }
#pragma unroll
    for (int k = 0; k < N; k++) oth[k] = fc.Ufe[pb + k * F];
    if (fold && (!MK || (cd[u] & 3) == 1))
      sT[i] = fc.wavein[(long long)e0 * F + i] * fc.wf[f % Sh::Ff] * fc.dAd[(long long)e0 * F + i];
  };
  // the common flux times this side's dA, negated on the right side
  auto common = [&](int u) {
    const int side = cd[u] & 3;
    if constexpr (GV) {
#pragma unroll
      for (int k = 0; k < N; k++) {
        const R v = mul_rn(fo[u][k], dA);
        fo[u][k] = side == 1 ? -v : v;
      }
      return;
    }
    if constexpr (BND) {
      if (side == 2) bc_state<D, R>(fc.bndBc[cd[u] >> 2], own, n, oth, ph, fc.bst);
    }
    const bool right = side == 1;
    R UL[N], UR[N], fn[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
      UL[k] = right ? oth[k] : own[k];
      UR[k] = right ? own[k] : oth[k];
    }
    double lam;
    const bool has_lam = pair_flux<D, R>(BND && side == 2, UL, UR, n, fn, ph, lam);
    if (has_lam && fc.wave && !right) st_s<NT>(lam, &fc.wave[(long long)e0 * F + fi(u)]);
    if (MK && fold && !right) {
      const long long i = (long long)e0 * F + fi(u);
      sT[fi(u)] = (has_lam ? lam : fc.wavein[i]) * fc.wf[fi(u) % Sh::Ff] * fc.dAd[i];
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
      const R v = mul_rn(fn[k], dA);
      fo[u][k] = right ? -v : v;
    }
  };
#pragma unroll
  for (int u = 0; u < KF; u++)
    if (flx(u)) {
      load_face(u);
      if constexpr (!APART) common(u);
    }
#pragma unroll
  for (int u = 0; u < N; u++) {
    const int i = threadIdx.x + u * blockDim.x;
    if (i < nb * N * S) {
      const int r = i / S, q = i - r * S;
      sU[r * S + spt_lds(D, P1, q)] = vu[u];
    }
  }
  __syncthreads();
  double dtl = 0;
  auto local_dt = [&] {
    double iw = 0;
    for (int g = 0; g < F; g++) iw += sT[b * F + g];
    dtl = fc.cflfac * 2 * fc.vole[e] / iw;
    if (s == 0) fc.eleDt[e] = dtl;
  };
  if (act) {
    if (!MK && fold) local_dt();
    // flux at the point, transformed to the reference element
    R u[N], Fl[D][N];
    const R* const qu = sU + b * N * S + sw;
#pragma unroll
    for (int k = 0; k < N; k++) u[k] = qu[k * S];
    inviscid_flux<D, R, true>(u, Fl, R(ph.gamma));
    R* const qf = sF + b * D * N * S + sw;
#pragma unroll
    for (int d1 = 0; d1 < D; d1++)
#pragma unroll
      for (int k = 0; k < N; k++) {
        R acc = 0;
#pragma unroll
        for (int d2 = 0; d2 < D; d2++) acc += G[d1][d2] * Fl[d2][k];
        qf[(d1 * N + k) * S] = acc;
      }
  }
  if constexpr (APART) {
    if (flx(0)) common(0);
  }
  __syncthreads();
  R dv[N];
  if (act) {
    // (without the registers for the update's inputs earlier)
    if constexpr (!(APART && D == 2)) in = rk_load<D, P, R, NT>(E, e, s, ra);
    if (MK && fold) local_dt();
    if (fold) in.dt = dtl;
    const PtOp<D, P, R, TEN> po(tb, sW, s);
    divergence<D, P, R, np>(sF, b, s, sw, swx, opv, abf, po, dv);
  }
#pragma unroll
  for (int u = 0; u < KF; u++)
    if (flx(u)) {
      // the flux jump: the common flux less the extrapolated normal flux (of
      // the sum over directions only the face's own normal direction is
      // non-zero)
      const int bb = fi(u) / F, f = fi(u) - bb * F;
      const FpOp<D, P, R, TEN> fp(tb, sW, f);
      const LineOp<P1, R> line(sF + (bb * D + fp.dir()) * N * S, [&](int m) { return lp[u][m]; },
                               [&](int m) { return fp.efn_w(m); });
      R* const o = sD + bb * N * F + f;
#pragma unroll
      for (int k = 0; k < N; k++) o[k * F] = fo[u][k] - fp.efn_sign(line(k * S));
    }
  __syncthreads();
  if (act) rk_point<D, P, R, NT, TEN, MK>(E, e, b, s, dv, sU, sD, sW, in, ra, tb);
  if (ra.mode == 5 || ra.mode == 7 || ra.mode == 8) return;  // uniform over the launch
  __syncthreads();
#pragma unroll
  for (int u = 0; u < KF; u++)
    if (flx(u)) face_point<D, P, R, NT, TEN>(fi(u), e0, lp[u], sU, sW, ra.Ufe, tb);
}

// Held as the viscous volume kernels: 4 waves per SIMD for quads and FP32, 3
// for FP64 hexes and the BF16 forms (which spill 41-78 VGPRs under 4: Taylor-Green
// 30^3 142.9 us, under 3 107.6).
template <int D, int P, class R, bool NT, bool BND, bool TEN, bool APART, int BF, int FORM>
__global__ __launch_bounds__(kMaxBlock) __attribute__((amdgpu_waves_per_eu(3))) void k_stage_w3(
    int E, int EB, const double* __restrict__ Ue, const R* __restrict__ Us, const R* __restrict__ JGe, StageFace<R> fc, Tabs tb,
    Phys ph, RkArgs<R> ra) {
  stage_body<D, P, R, NT, BND, TEN, APART, BF, FORM>(E, EB, Ue, Us, JGe, fc, tb, ph, ra);
}
template <int D, int P, class R, bool NT, bool BND, bool TEN, bool APART, int FORM>
__global__ __launch_bounds__(kMaxBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_stage_w4(
    int E, int EB, const double* __restrict__ Ue, const R* __restrict__ Us, const R* __restrict__ JGe, StageFace<R> fc, Tabs tb,
    Phys ph, RkArgs<R> ra) {
  stage_body<D, P, R, NT, BND, TEN, APART, 0, FORM>(E, EB, Ue, Us, JGe, fc, tb, ph, ra);
}

// ---------------------------------------------------------------------------
// The same value, as far as the compiler can tell another one: what is computed
// from it is not kept in registers from an earlier phase.
__device__ __forceinline__ int fresh(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// A value that is complete here: what is computed from it is not moved up among
// the sums that form it, which costs the registers of both.
template <class T>
__device__ __forceinline__ void pin(T& v) {
  asm volatile("" : "+v"(v));
}

// Where the correction with this side's part of the flux jump is applied.  FP64:
// here, so that the jump stays on chip.  FP32: by the RK kernel, together with
// the other side's part; split in two, the correction's roundings would differ
// by some 1e-8 of the state after a step, for 6% of the stage's traffic.
template <class R>
constexpr bool kJumpOut = sizeof(R) == 4;

// Whether the flux jump takes U's place in LDS (which has to be that large), not
// the transformed flux's, which would cost a barrier; P0 blocks, of many
// elements, would not fit the LDS limit.
template <int D, int P>
constexpr bool jump_over_u = P > 0;

// Threads that an element takes in the volume kernel.  One per solution point, which
// then take ceil(F/S) flux points each; at low orders, where that is 2 to 6, one per
// flux point instead, the solution points in the first of them: a round over flux
// points is most of the kernel's instructions, a mesh of this order fills few
// waves, and the rounds' values kept in registers spilled (P0 quads 243 of them).
// us a step with walls, in the three kernels before / one per solution point / now:
// quads 64^2 P0 116 / 194 / 80, 16^2 P1 92 / 106 / 78, 200^2 P2 320 / 331 / 232; hexes
// 24^3 P0 195 / 295 / 132, 12^3 P1 139 / 159 / 96, 48^3 P1 1690 / 1368 / 1078.
template <int D, int P>
constexpr int kVolThreads = P <= 1 || (D == 2 && P == 2) ? Shape<D, P>::F : Shape<D, P>::S;

// Volume kernel of viscous runs: all of a stage's residual but the other sides'
// parts of the LDG flux.  Solution points and then flux points in the same
// threads (kVolThreads an element), EB elements per block, element data in LDS.
//
// What a stage costs is its traffic, and most of that was intermediates: the
// common inviscid flux and the common U, written by a face kernel and read here
// and by the RK kernel, and the flux jump, written here and read there.  Both
// sides of a pair now form the common flux from U there and across (one read of
// U at the flux points; the own side is extrapolated again from the slab), and
// FP64 corrects the divergence with this side's part of the jump before it is
// written: 7.3 -> 4.6 GB per stage at 48^3 P3.  Sums that form a value are pinned
// before what uses them: otherwise both are live at once and the FP64 P3 kernel
// spills 136 registers.
// Measured, three kernels -> two: Navier-Stokes Taylor-Green 4 steps, 48^3 P3
// 20.07 -> 16.8 ms; 37^3 P2 6.89 -> 4.30 ms; 40^3 P3 mixed 7.93 -> 6.86 ms; 21^3
// P4 with monitor 1.43 -> 1.22 ms.
template <int D, int P, class R, bool NT, bool BND, bool TEN, int BF = 0>
__device__ __forceinline__ void volume_body(int E, const double* __restrict__ Ue, const R* __restrict__ Us,
                                            const R* __restrict__ JGe, const R* __restrict__ iJe,
                                            R* __restrict__ divFe, const VFace<R>& vf, const Tabs& tb, const Phys& ph) {
  using Sh = Shape<D, P>;
  constexpr int S = Sh::S, F = Sh::F, N = Sh::N, P1 = Sh::P1;
  const int EB = blockDim.x / kVolThreads<D, P>;
  // sU holds U until the flux has been formed, then the flux jump; sF holds, in
  // turn: dUc at the flux points, the physical gradient until it has been
  // extrapolated to the faces, then the transformed flux at the same indices as
  // the gradient.  [EB*N*SU] + [EB*N*max(F,D*S)]
  constexpr int SU = !kJumpOut<R> && jump_over_u<D, P> && F > S ? F : S;
  R* const sU = reinterpret_cast<R*>(fhip_lds);
  R* const sF = sU + EB * N * SU;
  R* const sD = jump_over_u<D, P> ? sU : sF;
  R* const sG = sF;
  R* const sC = sF;
  __shared__ R sW[Ten<D, P>::NW];
  stage_factors<D, P, R, TEN>(sW, tb);
  const int e0 = blockIdx.x * EB, nb = min(EB, E - e0);
  const int b = threadIdx.x / S, s = threadIdx.x - b * S;
  const int sw = spt_lds(D, P1, s);
  const bool act = b < nb;
  const long long e = e0 + b;
  // the thread's flux points: fi(u) < nP
  constexpr int KF = (F + kVolThreads<D, P> - 1) / kVolThreads<D, P>;
  const int nP = nb * F;
  auto fi = [&](int u) { return (int)threadIdx.x + u * (int)blockDim.x; };
  // matrix-core contractions: this lane's operator entry d1[s % 4][s / 16]
  // and the slab position of the point whose x and z are this lane's z and x
  constexpr bool mf = kMfma<D, P, R>;
  // mixed path, P3 hexes (BF = 2 or 3): z contractions in BF16 pieces on the
  // matrix cores
  constexpr int np = kBf16<D, P, R> ? BF : 0;
  bf16x8 abf;
  if constexpr (np != 0) abf = bf16_opnd_a(tw<float>(tb.d1, tb.d1f), s, np);
  const int swx = mf ? spt_lds(D, P1, s / 16 + 4 * ((s / 4) % 4) + 16 * (s % 4)) : 0;
  const R opv = mf ? tw<R>(tb.d1, tb.d1f)[(s % 4) * P1 + s / 16] : R(0);
  // every load is issued before the first LDS store, so that their latencies
  // overlap; the flux points' side codes first: the partners' addresses come
  // from them
  int cd[KF];
  Packed<P1> lp[KF];
#pragma unroll
  for (int u = 0; u < KF; u++) {
    cd[u] = fi(u) < nP ? vf.fpart[(long long)e0 * F + fi(u)] : 0;
    lp[u].load(tb, fi(u) < nP ? fi(u) % F : 0);
  }
  R vu[N];
  if (act) {
    const long long at = e * N * S + s;
    if (Us) {
#pragma unroll
      for (int k = 0; k < N; k++) vu[k] = ld_s<NT>(&Us[at + k * S]);
    } else {
#pragma unroll
      for (int k = 0; k < N; k++) vu[k] = R(ld_s<NT>(&Ue[at + k * S]));
    }
  }
  // U across and the normal
  R fn[KF][N], nv[KF][D];
#pragma unroll
  for (int u = 0; u < KF; u++)
    if (fi(u) < nP) {
      const int i = fi(u), bb = i / F, f = i - bb * F;
#pragma unroll
      for (int x = 0; x < D; x++) nv[u][x] = ld_s<NT>(&vf.nfe[((long long)(e0 + bb) * D + x) * F + f]);
      if (!BND || (cd[u] & 3) != 2) {
        const int p = cd[u] >> 2, ep = p / F;
        const long long pb = (long long)ep * N * F + (p - ep * F);
#pragma unroll
        for (int k = 0; k < N; k++) fn[u][k] = vf.Ufe[pb + k * F];
      }
    }
  // the point's metric terms
  R G[D][D] = {};
  auto load_G = [&] {
#pragma unroll
    for (int r = 0; r < D; r++)
#pragma unroll
      for (int x = 0; x < D; x++) G[r][x] = JGe[((e * D + r) * D + x) * S + s];
  };
  R inv = 0;
  if (act) {
    load_G();
    inv = iJe[e * S + s];
  }
  if (act) {
    R* const q = sU + b * N * S + sw;
#pragma unroll
    for (int k = 0; k < N; k++) q[k * S] = vu[k];
  }
  __syncthreads();
  // U at flux point u, of the block's element bb (the RK kernel's sums and bits)
  auto u_face = [&](int u, int bb, const FpOp<D, P, R, TEN>& fp, R* own) {
    const LineOp<P1, R> line(sU + bb * N * S, [&](int m) { return lp[u][m]; }, [&](int m) { return fp.ext_w(m); });
#pragma unroll
    for (int k = 0; k < N; k++) {
      own[k] = line(k * S);
      pin(own[k]);
    }
  };
  // the common inviscid flux (FP64: with the LDG penalty on the states, which
  // FP32 leaves in the two sides' parts), and the common U less U,
  // from U on both sides; the flux outward
#pragma unroll
  for (int u = 0; u < KF; u++)
    if (fi(u) < nP) {
      const int i = fresh(fi(u)), bb = i / F, f = i - bb * F, side = cd[u] & 3;
      const FpOp<D, P, R, TEN> fp(tb, sW, f);
      const bool right = side == 1, bnd = BND && side == 2;
      R own[N];
      u_face(u, bb, fp, own);
      if constexpr (BND) {
        if (bnd) bc_state<D, R>(vf.bndBc[cd[u] >> 2], own, nv[u], fn[u], ph, vf.bst);
      }
      double lam;
      bool has_lam;
      R pf = bnd ? R(0) : ldg_pen<D, R>(nv[u], R(ph.pen_fact));
      const R tn = bnd || kJumpOut<R> ? R(0) : ldg_tau<D, R>(nv[u], R(ph.tau));
      R* const qc = sC + bb * N * F + f;
      R fc[N];
      if constexpr (D == 3) {
        // from this side: its state first and the normal outward.  Rusanov's flux
        // from the other side is the same bits with the sign turned
        R no[D];
#pragma unroll
        for (int x = 0; x < D; x++) no[x] = right ? -nv[u][x] : nv[u][x];
        if (right) pf = -pf;
        has_lam = pair_flux<D, R>(bnd, own, fn[u], no, fc, ph, lam);
#pragma unroll
        for (int k = 0; k < N; k++) {
          const R du = own[k] - fn[u][k], mid = R(0.5) * (own[k] + fn[u][k]);
          qc[k * F] = (bnd ? mid : mid - pf * du) - own[k];
          if constexpr (!kJumpOut<R>) fc[k] += tn * du;
          fn[u][k] = fc[k];
        }
      } else {
        R UL[N], UR[N];
#pragma unroll
        for (int k = 0; k < N; k++) {
          UL[k] = right ? fn[u][k] : own[k];
          UR[k] = right ? own[k] : fn[u][k];
        }
        has_lam = pair_flux<D, R>(bnd, UL, UR, nv[u], fc, ph, lam);
#pragma unroll
        for (int k = 0; k < N; k++) {
          const R du = UL[k] - UR[k], mid = R(0.5) * (UL[k] + UR[k]);
          qc[k * F] = (bnd ? mid : mid - pf * du) - own[k];
          if constexpr (!kJumpOut<R>) fc[k] += tn * du;
          fn[u][k] = right ? -fc[k] : fc[k];
        }
      }
      if (has_lam && vf.wave && !right) st_s<NT>(lam, &vf.wave[(long long)e0 * F + i]);
#pragma unroll
      for (int k = 0; k < N; k++) pin(fn[u][k]);
    }
  __syncthreads();
  // phase 1: reference-space gradient (opp_grad_spts) plus correction
  // (opp_correctU), then the physical gradient (correctGradU transform,
  // src/solver.cpp:1105-1136), kept in LDS for phase 2 and the faces
  R gr[D][N];
  if (act) {
    const PtOp<D, P, R, TEN> po(tb, sW, fresh(s));
    const R *const qu = sU + b * N * S, *const qc = sC + b * N * F;
#pragma unroll
    for (int d = 0; d < D; d++) {
      // the other correction entries of the row are exactly zero
      const LineOp<2, R> cor(qc, [&](int j) { return po.cu_idx(d, j); }, [&](int j) { return po.cu_w(d, j); });
      if constexpr (np != 0) {
        if (d == 2) {
#pragma unroll
          for (int k = 0; k < N; k++)
            gr[d][k] = mfma_z_bf16<D, P1>(reinterpret_cast<const float*>(qu + k * S), s, abf, cor(k * F), np);
          continue;
        }
      }
      if (mf && d != 1) {  // compile-time: d and mf are constants here
        const R* const q = qu + (d == 2 ? sw : swx);
#pragma unroll
        for (int k = 0; k < N; k++)
          gr[d][k] = d == 2 ? mfma444(opv, q[k * S], cor(k * F)) : mfma444(q[k * S], opv, cor(k * F));
        continue;
      }
      const LineOp<P1, R> line(qu, [&](int m) { return po.grd_idx(d, m); }, [&](int m) { return po.grd_w(d, m); });
#pragma unroll
      for (int k = 0; k < N; k++) gr[d][k] = cor(k * F) + line(k * S);
    }
    // physical gradient, in place
#pragma unroll
    for (int k = 0; k < N; k++) {
      R acc[D];
#pragma unroll
      for (int x = 0; x < D; x++) {
        acc[x] = gr[0][k] * G[0][x] + gr[1][k] * G[1][x];
        if constexpr (D == 3) acc[x] += gr[2][k] * G[2][x];
      }
#pragma unroll
      for (int x = 0; x < D; x++) gr[x][k] = inv * acc[x];
    }
  }
  __syncthreads();  // sC is overwritten by the gradient below
  R* const qg = sG + b * D * N * S + sw;
  if (act) {
#pragma unroll
    for (int k = 0; k < N; k++)
#pragma unroll
      for (int x = 0; x < D; x++) qg[(x * N + k) * S] = gr[x][k];
  }
  __syncthreads();
  // physical gradient at the flux points (extrapolateGradU) and, with U there,
  // this side's viscous flux folded into its part of the LDG flux
  // (face::calcViscousFlux, src/face.cpp:216-293).  fn becomes the common flux,
  // as far as it is known on this side, times dA, outward: the other side's
  // part is added by the RK kernel.  Boundary points take the boundary state's
  // flux (boundFace::applyViscousBCs, src/boundFace.cpp:316-352).
  R bo[kJumpOut<R> ? KF : 1][N], dA = 0;
#pragma unroll
  for (int u = 0; u < KF; u++)
    if (fi(u) < nP) {
      const int i = fresh(fi(u)), bb = i / F, f = i - bb * F, side = cd[u] & 3;
      const FpOp<D, P, R, TEN> fp(tb, sW, f);
      dA = ld_s<NT>(&vf.dA[(long long)e0 * F + i]);
      R g[D][N];
      {
        const LineOp<P1, R> line(sG + bb * D * N * S, [&](int m) { return lp[u][m]; },
                                 [&](int m) { return fp.ext_w(m); });
#pragma unroll
        for (int x = 0; x < D; x++) {
#pragma unroll
          for (int k = 0; k < N; k++) {
            g[x][k] = line((x * N + k) * S);
            pin(g[x][k]);
          }
        }
      }
      R own[N], bv[N];
      u_face(u, bb, fp, own);
      if (BND && side == 2) {
        R UR[N], nF[N], d12[N];
        const int bc = vf.bndBc[cd[u] >> 2];
        bc_state<D, R>(bc, own, nv[u], UR, ph, vf.bst);
        const bool adiabatic = (bc & 15) == 10;
        if (adiabatic) adiabatic_grad<D, R>(own, UR, g, R(ph.gamma));
        ldg_side<D, R>(adiabatic ? UR : own, g, nv[u], nF, d12, ph);
#pragma unroll
        for (int k = 0; k < N; k++) bv[k] = 0;
        ldg_boundary<D, R>(own, UR, nF, nv[u], bv, ph);
      } else {
        if constexpr (kJumpOut<R>) {
#pragma unroll
          for (int k = 0; k < N; k++) bv[k] = 0;
          ldg_add_side<D, R>(side == 0, own, g, nv[u], bv, ph);
        } else {
          ldg_part<D, R>(side == 0, own, g, nv[u], bv, ph);
        }
        R* const o = vf.Bve + (long long)(e0 + bb) * N * F + f;
#pragma unroll
        for (int k = 0; k < N; k++) st_s<NT>(bv[k], &o[k * F]);
      }
#pragma unroll
      for (int k = 0; k < N; k++) {
        const R bs = side == 1 ? -bv[k] : bv[k];
        fn[u][k] = kJumpOut<R> ? mul_rn(fn[u][k], dA) : (fn[u][k] + bs) * dA;
        if constexpr (kJumpOut<R>) bo[u][k] = bs;
      }
    }
  // under the register hold, the metric terms again (from cache): keeping
  // them live across the face loop above costs more registers than it allows
  if constexpr (kHold<D, R>) {
    if (act) load_G();
  }
  // phase 2: flux at the point, transformed to the reference element.  It is
  // formed in registers and stored after a barrier, over the gradient slab,
  // which other threads may still be reading in the face loop; threads with
  // fewer face points go on here meanwhile.
  R Ft[D][N];
  if (act) {
    const R* const qs = sU + b * N * S + sw;
    R u[N];
#pragma unroll
    for (int k = 0; k < N; k++) u[k] = qs[k * S];
    R Fl[D][N];
    R g[D][N];
#pragma unroll
    for (int x = 0; x < D; x++)
#pragma unroll
      for (int k = 0; k < N; k++) g[x][k] = qg[(x * N + k) * S];
    R Fi[D][N];
    viscous_flux<D, R>(u, g, Fl, ph);
    inviscid_flux<D, R>(u, Fi, R(ph.gamma));
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
      for (int k = 0; k < N; k++) Fl[d][k] = Fl[d][k] + Fi[d][k];
#pragma unroll
    for (int d1 = 0; d1 < D; d1++)
#pragma unroll
      for (int k = 0; k < N; k++) {
        R acc = 0;
#pragma unroll
        for (int d2 = 0; d2 < D; d2++) acc += G[d1][d2] * Fl[d2][k];
        Ft[d1][k] = acc;
      }
  }
  __syncthreads();
  if (act) {
#pragma unroll
    for (int d1 = 0; d1 < D; d1++)
#pragma unroll
      for (int k = 0; k < N; k++) qg[(d1 * N + k) * S] = Ft[d1][k];
  }
  __syncthreads();
  R dv[N];
  if (act) {
    const PtOp<D, P, R, TEN> po(tb, sW, fresh(s));
    divergence<D, P, R, np>(sF, b, s, sw, swx, opv, abf, po, dv);
    if constexpr (kJumpOut<R>) {
#pragma unroll
      for (int k = 0; k < N; k++) st_s<NT>(dv[k], &divFe[e * N * S + s + k * S]);
    }
  }
  // faces: the flux jump, less the other side's part (extrapolateNormalFlux: of
  // the sum over directions only the face's own normal direction is non-zero)
#pragma unroll
  for (int u = 0; u < KF; u++)
    if (fi(u) < nP) {
      const int i = fresh(fi(u)), bb = i / F, f = i - bb * F;
      const FpOp<D, P, R, TEN> fp(tb, sW, f);
      const LineOp<P1, R> line(sF + (bb * D + fp.dir()) * N * S, [&](int m) { return lp[u][m]; },
                               [&](int m) { return fp.efn_w(m); });
      const R dJ = kJumpOut<R> ? (KF == 1 ? dA : vf.dA[(long long)e0 * F + i]) : R(0);
#pragma unroll
      for (int k = 0; k < N; k++) {
        const R a = fp.efn_sign(line(k * S));
        if constexpr (kJumpOut<R>) {
          const R j = bo[u][k] * dJ - a;
          st_s<NT>(fn[u][k] + j, &vf.Jne[((long long)(e0 + bb) * N + k) * F + f]);
          continue;
        }
        fn[u][k] -= a;
        if constexpr (jump_over_u<D, P>) sD[(bb * N + k) * F + f] = fn[u][k];
      }
    }
  if constexpr (kJumpOut<R>) return;
  if constexpr (!jump_over_u<D, P>) {
    __syncthreads();
#pragma unroll
    for (int u = 0; u < KF; u++)
      if (fi(u) < nP) {
        const int i = fresh(fi(u)), bb = i / F, f = i - bb * F;
#pragma unroll
        for (int k = 0; k < N; k++) sD[(bb * N + k) * F + f] = fn[u][k];
      }
  }
  __syncthreads();
  if (act) {
    const PtOp<D, P, R, TEN> po(tb, sW, fresh(s));
    correction<D, P, R>(sD, b, po, dv, dv);
#pragma unroll
    for (int k = 0; k < N; k++) st_s<NT>(dv[k], &divFe[e * N * S + s + k * S]);
  }
}

// The volume kernel held to 4 waves per SIMD (at most 128 VGPRs) for quads
// and the FP32 path, which fit there without spilling (holding the FP32
// viscous hex kernel to 5 or 6 waves spills 26 or 41 VGPRs and was measured
// 13-16% slower), and to 3 waves (168 VGPRs) for FP64 hexes and for the BF16 forms,
// whose pieces of a whole column and its accumulators are live at once: 153 VGPRs, under
// the 4-wave hold 21-29 spilled (Navier-Stokes Taylor-Green 24^3 84.1 us, under 3 67.8).
template <int D, int P, class R, bool NT, bool BND, bool TEN, int BF = 0>
__global__ __launch_bounds__(kMaxBlock) __attribute__((amdgpu_waves_per_eu(3))) void k_volume_w3(
    int E, const double* __restrict__ Ue, const R* __restrict__ Us, const R* __restrict__ JGe, const R* __restrict__ iJe,
    R* __restrict__ divFe, VFace<R> vf, Tabs tb, Phys ph) {
  volume_body<D, P, R, NT, BND, TEN, BF>(E, Ue, Us, JGe, iJe, divFe, vf, tb, ph);
}
template <int D, int P, class R, bool NT, bool BND, bool TEN>
__global__ __launch_bounds__(kMaxBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_volume_w4(
    int E, const double* __restrict__ Ue, const R* __restrict__ Us, const R* __restrict__ JGe, const R* __restrict__ iJe,
    R* __restrict__ divFe, VFace<R> vf, Tabs tb, Phys ph) {
  volume_body<D, P, R, NT, BND, TEN>(E, Ue, Us, JGe, iJe, divFe, vf, tb, ph);
}

// After the viscous volume kernel: correction of the divergence with the other
// sides' LDG parts (FP32: with the whole flux jump), RK update and U at the flux
// points.  With NT, the arrays this kernel reads or writes exactly once per launch
// go through nontemporal loads and stores (they stream past the caches).
template <int D, int P, class R, bool NT, bool TEN>
__global__ __launch_bounds__(kMaxBlock) void k_rk(int E, const R* __restrict__ divFe, RkArgs<R> ra, Tabs tb,
                                             const int* __restrict__ fpart, const R* __restrict__ dAe,
                                             const R* __restrict__ Bve, const R* __restrict__ Jne) {
  using Sh = Shape<D, P>;
  constexpr int S = Sh::S, F = Sh::F, N = Sh::N;
  const int EB = blockDim.x / S;
  R* const sU = reinterpret_cast<R*>(fhip_lds);  // [EB*N*S]
  R* const sD = sU + EB * N * S;                  // [EB*N*F] the flux jump (FP64: the other side's part of it)
  __shared__ R sW[Ten<D, P>::NW];
  stage_factors<D, P, R, TEN>(sW, tb);
  const int e0 = blockIdx.x * EB, nb = min(EB, E - e0);
  const int b = threadIdx.x / S, s = threadIdx.x - b * S;
  // The flux points' loads are unconditional (a boundary point reads its own
  // row where an interior point reads its partner's, and selects) and, for
  // the points a thread stages, issued before their LDS stores, so that their
  // latencies overlap.  A thread stages at most KF = ceil(F / S) points.
  constexpr int KF = (F + S - 1) / S;
  int cd[KF];
  Packed<P + 1> lp[KF];
#pragma unroll
  for (int u = 0; u < KF; u++) {
    const int i = threadIdx.x + u * blockDim.x;
    cd[u] = (i < nb * F) ? fpart[(long long)e0 * F + i] : 2;
    lp[u].load(tb, (i < nb * F) ? i % F : 0);
  }
#pragma unroll
  for (int u = 0; u < KF; u++) {
    const int i = threadIdx.x + u * blockDim.x;
    if (i >= nb * F) break;
    const int bb = i / F, f = i - bb * F;
    const int code = cd[u], side = code & 3;
    const R dA = dAe[(long long)e0 * F + i];
    const long long ob = (long long)(e0 + bb) * N * F + f;
    long long pb = ob;
    if (side != 2) {
      const long long p = code >> 2, ep = p / F;
      pb = ep * N * F + (p - ep * F);
    }
#pragma unroll
    for (int k = 0; k < N; k++) {
      const R bp = ld_s<NT>(&Bve[pb + k * F]);
      const R base = kJumpOut<R> ? ld_s<NT>(&Jne[ob + k * F]) : R(0);
      sD[(bb * N + k) * F + f] = side == 2 ? base : base + (side == 0 ? bp : -bp) * dA;
    }
  }
  __syncthreads();
  if (b < nb) {
    R dv[N];
#pragma unroll
    for (int k = 0; k < N; k++) dv[k] = ld_s<NT>(&divFe[((e0 + b) * (long long)N + k) * S + s]);
    const RkIn<D, R> in = rk_load<D, P, R, NT>(E, e0 + b, s, ra);
    rk_point<D, P, R, NT, TEN>(E, e0 + b, b, s, dv, sU, sD, sW, in, ra, tb);
  }
  if (ra.mode == 5 || ra.mode == 7 || ra.mode == 8) return;  // uniform over the launch
  __syncthreads();
#pragma unroll
  for (int u = 0; u < KF; u++) {
    const int i = threadIdx.x + u * blockDim.x;
    if (i < nb * F) face_point<D, P, R, NT, TEN>(i, e0, lp[u], sU, sW, ra.Ufe, tb);
  }
}


#ifndef FHIP_FAMILY
// P-multigrid transfers in element-major layout ([ele][field][point] rows of
// S values), the products the staged operator GEMM forms in FlurryPP's layout
// with the same sums (chunks of kc columns of the operator, added in turn).
// multiGrid::restrict_pmg (src/multigrid.cpp:315-345) and the start of
// compute_source_term (:381-398): the coarse level's U = R U_fine, its FAS
// source = R divF_fine (the residual of U is subtracted later) and sol = U.
static __global__ void k_restrict_em(long long rows, int Sc, int Sf, int kc, const double* __restrict__ R,
                              const double* __restrict__ Uf, const double* __restrict__ divFf,
                              double* __restrict__ Uc, double* __restrict__ srcc, double* __restrict__ solc) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= rows * Sc) return;
  const long long r = t / Sc;
  const int i = (int)(t - r * Sc);
  const double* a = R + (long long)i * Sf;
  const double* u = Uf + r * Sf;
  const double* d = divFf + r * Sf;
  double cu = 0, cd = 0;
  for (int l0 = 0; l0 < Sf; l0 += kc) {
    const int n = min(kc, Sf - l0);
    double su = 0, sd = 0;
    for (int l = 0; l < n; l++) {
      su += a[l0 + l] * u[l0 + l];
      sd += a[l0 + l] * d[l0 + l];
    }
    cu = l0 ? su + cu : su;
    cd = l0 ? sd + cd : sd;
  }
  Uc[t] = cu;
  solc[t] = cu;
  srcc[t] = cd;
}

// prolong_err (src/multigrid.cpp:347-364): U_up += P (U - sol) of the level
// below.
static __global__ void k_prolong_em(long long rows, int Su, int Sc, int kc, const double* __restrict__ Pm,
                             const double* __restrict__ Uc, const double* __restrict__ solc, double* __restrict__ Uu) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= rows * Su) return;
  const long long r = t / Su;
  const int i = (int)(t - r * Su);
  const double* a = Pm + (long long)i * Sc;
  const double* u = Uc + r * Sc;
  const double* o = solc + r * Sc;
  double c = Uu[t];
  for (int l0 = 0; l0 < Sc; l0 += kc) {
    const int n = min(kc, Sc - l0);
    double s = 0;
    for (int l = 0; l < n; l++) {
      double v = u[l0 + l];
      v -= o[l0 + l];
      s += a[l0 + l] * v;
    }
    c = s + c;
  }
  Uu[t] = c;
}

#endif  // FHIP_FAMILY

// The same transfers with the operator (transposed, so that the lanes of a
// wave read consecutive entries) and the rows of the block's EB elements staged in
// LDS, one output per thread, the sums in the same order as above; and, where Ufe
// is given, the level's new U at the flux points (and its FP32 copy), which the
// level's next residual or smoothing step starts from.  Used where an element's
// rows fit a block and all of it 64 KiB.
template <int D, int P, class R, bool TEN>
__device__ __forceinline__ void transfer_faces(int e0, int nb, const R* sX, const R* sW, R* Ufe, const Tabs& tb) {
  for (int i = threadIdx.x; i < nb * Shape<D, P>::F; i += blockDim.x) {
    Packed<P + 1> lp;
    lp.load(tb, i % Shape<D, P>::F);
    face_point<D, P, R, false, TEN>(i, e0, lp, sX, sW, Ufe, tb);
  }
}
template <int D, int P, class R, bool TEN>
__global__ __launch_bounds__(kMaxBlock) void k_restrict_lds(int ne, int EB, int Sf, int kc, const double* __restrict__ A,
                                                             const double* __restrict__ Uf,
                                                             const double* __restrict__ divFf, double* __restrict__ Uc,
                                                             double* __restrict__ srcc, double* __restrict__ solc,
                                                             R* __restrict__ Ufe, R* __restrict__ Us, Tabs tb) {
  using Sh = Shape<D, P>;
  constexpr int S = Sh::S, N = Sh::N, P1 = Sh::P1;
  const int e0 = blockIdx.x * EB, nb = min(EB, ne - e0), nr = EB * N, rows = nb * N;
  double* const sA = reinterpret_cast<double*>(fhip_lds);  // [Sf][S]
  double* const sU = sA + S * Sf;                           // [nr][Sf]
  double* const sV = sU + nr * Sf;                          // [nr][Sf]
  R* const sX = reinterpret_cast<R*>(sV + nr * Sf);         // [nr][S]
  __shared__ R sW[Ten<D, P>::NW];
  stage_factors<D, P, R, TEN>(sW, tb);
  const long long r0 = (long long)e0 * N;
  for (int j = threadIdx.x; j < S * Sf; j += blockDim.x) {
    const int i = j / Sf;
    sA[(j - i * Sf) * S + i] = A[j];
  }
  for (int j = threadIdx.x; j < rows * Sf; j += blockDim.x) {
    sU[j] = Uf[r0 * Sf + j];
    sV[j] = divFf[r0 * Sf + j];
  }
  __syncthreads();
  const int rr = threadIdx.x / S, i = threadIdx.x - rr * S;
  if (rr < rows) {
    const double* u = sU + rr * Sf;
    const double* d = sV + rr * Sf;
    double cu = 0, cd = 0;
    for (int l0 = 0; l0 < Sf; l0 += kc) {
      const int n = min(kc, Sf - l0);
      double su = 0, sd = 0;
      for (int l = 0; l < n; l++) {
        const double a = sA[(l0 + l) * S + i];
        su += a * u[l0 + l];
        sd += a * d[l0 + l];
      }
      cu = l0 ? su + cu : su;
      cd = l0 ? sd + cd : sd;
    }
    const long long t = r0 * S + threadIdx.x;
    Uc[t] = cu;
    solc[t] = cu;
    srcc[t] = cd;
    sX[rr * S + spt_lds(D, P1, i)] = R(cu);
    if (Us) Us[t] = R(cu);
  }
  __syncthreads();
  transfer_faces<D, P, R, TEN>(e0, nb, sX, sW, Ufe, tb);
}

template <int D, int P, class R, bool TEN>
__global__ __launch_bounds__(kMaxBlock) void k_prolong_lds(int ne, int EB, int Sc, int kc, const double* __restrict__ A,
                                                            const double* __restrict__ Uc,
                                                            const double* __restrict__ solc, double* __restrict__ Uu,
                                                            R* __restrict__ Ufe, R* __restrict__ Us, Tabs tb) {
  using Sh = Shape<D, P>;
  constexpr int S = Sh::S, N = Sh::N, P1 = Sh::P1;
  const int e0 = blockIdx.x * EB, nb = min(EB, ne - e0), nr = EB * N, rows = nb * N;
  double* const sA = reinterpret_cast<double*>(fhip_lds);  // [Sc][S]
  double* const sV = sA + S * Sc;                           // [nr][Sc]: U - sol
  R* const sX = reinterpret_cast<R*>(sV + nr * Sc);         // [nr][S]
  __shared__ R sW[Ten<D, P>::NW];
  stage_factors<D, P, R, TEN>(sW, tb);
  const long long r0 = (long long)e0 * N;
  for (int j = threadIdx.x; j < S * Sc; j += blockDim.x) {
    const int i = j / Sc;
    sA[(j - i * Sc) * S + i] = A[j];
  }
  for (int j = threadIdx.x; j < rows * Sc; j += blockDim.x) {
    double v = Uc[r0 * Sc + j];
    v -= solc[r0 * Sc + j];
    sV[j] = v;
  }
  __syncthreads();
  const int rr = threadIdx.x / S, i = threadIdx.x - rr * S;
  if (rr < rows) {
    const double* v = sV + rr * Sc;
    const long long t = r0 * S + threadIdx.x;
    double c = Uu[t];
    for (int l0 = 0; l0 < Sc; l0 += kc) {
      const int n = min(kc, Sc - l0);
      double s = 0;
      for (int l = 0; l < n; l++) s += sA[(l0 + l) * S + i] * v[l0 + l];
      c = s + c;
    }
    Uu[t] = c;
    if (Ufe) {
      sX[rr * S + spt_lds(D, P1, i)] = R(c);
      if (Us) Us[t] = R(c);
    }
  }
  if (!Ufe) return;  // uniform over the launch
  __syncthreads();
  transfer_faces<D, P, R, TEN>(e0, nb, sX, sW, Ufe, tb);
}

// Wave speeds from U at the flux points (ele::calcWaveSpFpts), element-major.
template <int D, int P, class R>
__global__ void k_wave_em(int E, const R* __restrict__ Ufe, const double* __restrict__ norme,
                          double* __restrict__ waveSpe, double gamma) {
  using Sh = Shape<D, P>;
  constexpr int F = Sh::F, N = Sh::N;
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)E * F) return;
  long long e = i / F, f = i - e * F;
  double U[N];
#pragma unroll
  for (int k = 0; k < N; k++) U[k] = double(Ufe[(e * N + k) * F + f]);
  double rho = U[0], u = U[1] / rho, v = U[2] / rho, w = 0;
  if constexpr (D == 3) w = U[3] / rho;
  double rhoVSq = rho * (u * u + v * v + w * w);
  double pr = (gamma - 1) * (U[D + 1] - 0.5 * rhoVSq);
  double vN = u * norme[(e * D + 0) * F + f] + v * norme[(e * D + 1) * F + f];
  if constexpr (D == 3) vN += w * norme[(e * D + 2) * F + f];
  double csq = smax(gamma * pr / rho, 0.0);
  waveSpe[i] = (fabs(vN - 0.) + sqrt(csq));
}

// The element volumes calcDt divides by, once per context (the geometry is
// fixed): the same sum as the reference's per call.
template <int D, int P>
__global__ __launch_bounds__(256) void k_ele_vol(int E, const double* __restrict__ detJe, const double* __restrict__ ws,
                                                  double* __restrict__ vole) {
  constexpr int S = Shape<D, P>::S;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= E) return;
  double vol = 0;
  for (int s = 0; s < S; s++) vol += detJe[(long long)e * S + s] * ws[s];
  vole[e] = vol;
}

// The dt kernel: lanes that sum one element's flux points, elements that a group of
// lanes has in flight, and blocks at most, each of which takes its turn at two atomics,
// some 20 ns.  (A thread per element, each read 8 F bytes from its neighbour's, on E/256
// blocks whose release wrote back the L2, took 8 to 52 us below.)  More lanes per
// element than these are more blocks; fewer, longer chains: as many as flux points up
// to 64, 16 for all, these, 8 for all: quads 86^2 P2 11.0, -, 8.6, 8.6 us, 64^2 P5 11.7,
// -, 7.2, 7.2; hexes 17^3 P2 11.4, 9.5, 9.5, 9.6, 20^3 P3 13.4, 10.3, 10.3, 10.0, 23^3 P4
// 20.2, 15.6, 15.6, 24.1, 48^3 P1 24.5, -, 16.3, 16.3.
//
// Meshes that need more than kDtSmall blocks of 256 threads take blocks of 1024:
// fewer turns, and on more than kDtBlocks more loads in flight.  256 / 1024 threads:
// quads 120^2 P2 (225 blocks) 11.0 / 8.9 us, 100^2 P3 (157) 9.1 / 8.5, 64^2 P5 (64) 7.3 /
// 8.8; hexes 23^3 P4 (191) 15.8 / 26, 20^3 P3 (125) 10.3 / 13.3.  30^3 P3 with lanes for 64
// flux points 42 / 22, in 1024 blocks of 256 threads 26; 400^2 P3 37 / 21.
template <int F>
constexpr int kDtLanes = F <= 4 ? 4 : (F <= 24 ? 8 : 16);
template <int D>
constexpr int kDtEles = D == 2 ? 2 : 4;
constexpr unsigned kDtBlocks = 256;
template <int D>
constexpr unsigned kDtSmall = D == 2 ? 128 : 256;

// ele::calcDt per element (element-major inputs) and, with a ticket counter, the
// minimum of all at out, the global dt (solver::calcDt, src/solver.cpp:447-468).
template <int D, int P, int NT>
__global__ __launch_bounds__(NT) void k_ele_dt_em(int E, const double* __restrict__ vole, const double* __restrict__ wf,
                                                    const double* __restrict__ waveSpe, const double* __restrict__ dAe,
                                                    double cflfac, double* __restrict__ eleDt, double* acc,
                                                    unsigned* ticket, double* __restrict__ out) {
  using Sh = Shape<D, P>;
  constexpr int F = Sh::F, Ff = Sh::Ff, G = kDtLanes<F>;
  __shared__ double red[NT / 64];
  const int l = threadIdx.x % G;
  double dt = INFINITY;
  constexpr int EB = NT / G, M = kDtEles<D>;
  for (int e0 = blockIdx.x * (EB * M); e0 < E; e0 += gridDim.x * (EB * M)) {  // uniform over the block
    double iw[M], vol[M];
#pragma unroll
    for (int u = 0; u < M; u++) {
      const int e = e0 + u * EB + threadIdx.x / G, ec = e < E ? e : E - 1;
      vol[u] = vole[ec];
      iw[u] = 0;
#pragma unroll
      for (int f0 = 0; f0 < F; f0 += G) {
        const int f = f0 + l;
        if (f < F) iw[u] += waveSpe[(long long)ec * F + f] * wf[f % Ff] * dAe[(long long)ec * F + f];
      }
    }
#pragma unroll
    for (int u = 0; u < M; u++) {
      const int e = e0 + u * EB + threadIdx.x / G;
#pragma unroll
      for (int o = G / 2; o > 0; o >>= 1) iw[u] += __shfl_xor(iw[u], o);
      const double v = cflfac * 2 * vol[u] / iw[u];
      if (e < E) {
        if (l == 0) eleDt[e] = v;
        dt = fmin(dt, v);
      }
    }
  }
  const double bmin = block_min(dt, red);
  if (!ticket) return;  // merged meshes: per-mesh minima of eleDt follow
  if (threadIdx.x == 0) grid_min(bmin, gridDim.x, acc, ticket, out);
}

// The common inviscid flux and its wave speeds at the left and boundary points, for
// the steps that need the speeds ahead of their stage kernel (face_first); right points
// keep their speeds (and, with Roe's flux, all but the boundary's).
template <int D, int P, class R>
__global__ __launch_bounds__(kMaxBlock) void k_pair_wave(int n, const int* __restrict__ fpart, const R* __restrict__ Ufe,
                                                    const R* __restrict__ nfe, const int* __restrict__ bndBc,
                                                    double* __restrict__ waveSpe, R* __restrict__ Fne, Phys ph,
                                                    const double* __restrict__ bst) {
  using Sh = Shape<D, P>;
  constexpr int F = Sh::F, N = Sh::N;
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int code = fpart[q], side = code & 3;
  if (side == 1) return;
  const int e = q / F, f = q - e * F;
  R UL[N], UR[N], nv[D], fn[N];
#pragma unroll
  for (int k = 0; k < N; k++) UL[k] = Ufe[((long long)e * N + k) * F + f];
#pragma unroll
  for (int d = 0; d < D; d++) nv[d] = nfe[((long long)e * D + d) * F + f];
  if (side == 2) {
    bc_state<D, R>(bndBc[code >> 2], UL, nv, UR, ph, bst);
  } else {
    const int p = code >> 2, ep = p / F, fp = p - ep * F;
#pragma unroll
    for (int k = 0; k < N; k++) UR[k] = Ufe[((long long)ep * N + k) * F + fp];
  }
  double lam;
  if (pair_flux<D, R>(side == 2, UL, UR, nv, fn, ph, lam)) waveSpe[q] = lam;
#pragma unroll
  for (int k = 0; k < N; k++) Fne[((long long)e * N + k) * F + f] = fn[k];
}

// The same and the elements' time steps from them in one pass, up to kWaveDtPoints
// flux points: one launch less, but in the dt kernel's blocks, which are too few for
// the gathers of a large mesh.  A step of quads in one / two launches: 64^2 P4 (82 k
// points) 23.7 / 26.5 us, 64^2 P5 (98 k) 28.4 / 29, 200^2 P3 (640 k) 62 / 57; hexes 6^3 P3 (21 k)
// 18.3 / 22.
constexpr long long kWaveDtPoints = 1 << 17;
template <int D>
constexpr int kWaveDtLanes = D == 2 ? 8 : 32;
template <int D, int P, class R, int NT>
__global__ __launch_bounds__(NT) void k_wave_dt(int E, const int* __restrict__ fpart, const R* __restrict__ Ufe,
                                                const R* __restrict__ nfe, const int* __restrict__ bndBc,
                                                const double* __restrict__ bst, Phys ph,
                                                const double* __restrict__ vole, const double* __restrict__ wf,
                                                double* waveSpe, R* __restrict__ Fne,
                                                const double* __restrict__ dAe, double cflfac,
                                                double* __restrict__ eleDt, double* acc, unsigned* ticket,
                                                double* __restrict__ out) {
  using Sh = Shape<D, P>;
  constexpr int F = Sh::F, Ff = Sh::Ff, N = Sh::N, G = kWaveDtLanes<D>, EB = NT / G;
  __shared__ double red[NT / 64];
  const int l = threadIdx.x % G;
  double dt = INFINITY;
  for (int e0 = blockIdx.x * EB; e0 < E; e0 += gridDim.x * EB) {  // uniform over the block
    const int e = e0 + threadIdx.x / G;
    double iw = 0;
#pragma unroll
    for (int f0 = 0; f0 < F; f0 += G) {
      const int f = f0 + l;
      if (f >= F || e >= E) continue;
      const long long q = (long long)e * F + f;
      const int code = fpart[q], side = code & 3;
      double lam = waveSpe[q];
      if (side != 1) {
        R UL[N], UR[N], n[D], fn[N];
#pragma unroll
        for (int k = 0; k < N; k++) UL[k] = Ufe[((long long)e * N + k) * F + f];
#pragma unroll
        for (int d = 0; d < D; d++) n[d] = nfe[((long long)e * D + d) * F + f];
        if (side == 2) {
          bc_state<D, R>(bndBc[code >> 2], UL, n, UR, ph, bst);
        } else {
          const int p = code >> 2, ep = p / F;
#pragma unroll
          for (int k = 0; k < N; k++) UR[k] = Ufe[((long long)ep * N + k) * F + (p - ep * F)];
        }
        if (pair_flux<D, R>(side == 2, UL, UR, n, fn, ph, lam)) waveSpe[q] = lam;
#pragma unroll
        for (int k = 0; k < N; k++) Fne[((long long)e * N + k) * F + f] = fn[k];
      }
      iw += lam * wf[f % Ff] * dAe[q];
    }
#pragma unroll
    for (int o = G / 2; o > 0; o >>= 1) iw += __shfl_xor(iw, o);
    if (e < E) {
      const double v = cflfac * 2 * vole[e] / iw;
      if (l == 0) eleDt[e] = v;
      dt = fmin(dt, v);
    }
  }
  const double bmin = block_min(dt, red);
  if (!ticket) return;
  if (threadIdx.x == 0) grid_min(bmin, gridDim.x, acc, ticket, out);
}

// Per-mesh minimum of the element time steps (batched contexts, dt_type 1).
static __global__ void k_mesh_dt_min(const int* __restrict__ start, const double* __restrict__ eleDt,
                              double* __restrict__ meshDt) {
  __shared__ double red[256];
  const int m = blockIdx.x;
  double v = INFINITY;
  for (int e = start[m] + threadIdx.x; e < start[m + 1]; e += blockDim.x) v = fmin(v, eleDt[e]);
  red[threadIdx.x] = v;
  __syncthreads();
  for (int st = blockDim.x / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st) red[threadIdx.x] = fmin(red[threadIdx.x], red[threadIdx.x + st]);
    __syncthreads();
  }
  if (threadIdx.x == 0) meshDt[m] = red[0];
}

#ifndef FHIP_FAMILY
// Per-mesh residual norm over divF_spts[0] (element-major), as
// ele::getNormResidual summed over the mesh's elements (src/ele.cpp:1922-1945).
static __global__ void k_mesh_res(int S, int N, int type, const int* __restrict__ start, const double* __restrict__ divF0e,
                           const double* __restrict__ detJe, const double* __restrict__ ws, double* __restrict__ out) {
  __shared__ double red[256];
  const int m = blockIdx.x;
  for (int k = 0; k < N; k++) {
    double r = 0;
    for (long long i = (long long)start[m] * S + threadIdx.x; i < (long long)start[m + 1] * S; i += blockDim.x) {
      long long e = i / S;
      int s = (int)(i - e * S);
      double v = divF0e[(e * N + k) * S + s], dj = detJe[i];
      if (type == 1) r += fabs(v) * ws[s];
      else if (type == 2) r += v * v / dj * ws[s];
      else r = fmax(r, fabs(v) / dj);
    }
    red[threadIdx.x] = r;
    __syncthreads();
    for (int st = blockDim.x / 2; st > 0; st >>= 1) {
      if (threadIdx.x < st)
        red[threadIdx.x] = (type == 3) ? fmax(red[threadIdx.x], red[threadIdx.x + st]) : red[threadIdx.x] + red[threadIdx.x + st];
      __syncthreads();
    }
    if (threadIdx.x == 0) out[(long long)m * N + k] = (type == 2) ? sqrt(red[0]) : red[0];
    __syncthreads();
  }
}

#endif  // FHIP_FAMILY

// ---------------------------------------------------------------------------
// Host side.

static FusedState& fs(Ctx& c) { return *reinterpret_cast<FusedState*>(c.fused); }

template <class T>
static T* dal(size_t n) {
  void* p = nullptr;
  FCHK(hipMalloc(&p, (n ? n : 1) * sizeof(T)));
  poison_fill(p, (n ? n : 1) * sizeof(T));
  return (T*)p;
}

#ifndef FHIP_FAMILY
// Extract the non-zero structure of the dense operators.  Returns false if an
// operator row has more non-zeros than the tensor-product structure allows.
// opp_grad_spts as one 1-D derivative matrix (Tabs::d1): true when every
// entry equals its tensor-product counterpart d1[coordinate of q along d]
// [coordinate of r along d] on q's d-line and is zero off it (the dense
// operator of a tensor-product element on one 1-D point set is: its factors
// in the other directions are exactly 0 or 1).
static bool build_d1(const Ctx& c, const fhip_desc* dsc, std::vector<double>& d1) {
  const int D = c.z.D, S = c.z.S, P1 = c.z.P + 1;
  d1.assign(P1 * P1, 0.);
  for (int i = 0; i < P1; i++)
    for (int m = 0; m < P1; m++) d1[i * P1 + m] = dsc->opp_grad_spts[(size_t)i * S + m];  // d = 0, line 0
  for (int dd = 0, step = 1; dd < D; dd++, step *= P1)
    for (int q = 0; q < S; q++) {
      const double* const row = dsc->opp_grad_spts + ((size_t)dd * S + q) * S;
      const int at = (q / step) % P1, line = q - at * step;  // the point's place on its line, the line's first point
      int on = 0;
      for (int m = 0; m < P1; m++) {
        const double v = row[line + m * step];
        if (!(v == d1[at * P1 + m])) return false;  // +0 == -0
        on += v != 0.;
      }
      if (count_nonzeros(row, S) != on) return false;
    }
  return true;
}

// The 1-D factors (Ten) of the dense operators, or false where an entry of one
// of them is not what the factors give.
template <int D, int P>
static bool build_ten(const Ctx& c, const fhip_desc* d, const std::vector<double>& d1, std::vector<double>& w,
                      std::vector<int>& line) {
  using T = Ten<D, P>;
  using Sh = Shape<D, P>;
  constexpr int S = Sh::S, F = Sh::F, P1 = Sh::P1;
  w.assign(T::NW, 0.);
  std::copy(d1.begin(), d1.end(), w.begin());
  std::vector<int> at((size_t)F * P1);
  // l and c from the first point of a face on each end of direction 0
  for (int j = 0; j < 2 * D; j++) {
    if (T::face_dir(j) != 0) continue;
    const int f = j * Sh::Ff, hi = T::face_hi(j);
    const typename T::Face face(f);
    for (int m = 0; m < P1; m++) {
      int cc[3] = {m, face.c[1], face.c[2]};
      const int q = cc[0] + P1 * (cc[1] + P1 * cc[2]);
      w[T::L + hi * P1 + m] = d->opp_spts_to_fpts[(size_t)f * S + q];
      w[T::C + hi * P1 + m] = d->opp_correction[(size_t)q * F + T::face_fpt(j, cc)];
    }
  }
  // every entry on a flux point's line as the factors give it, and no others
  long long nc = 0;  // of the corrections
  for (int f = 0; f < F; f++) {
    const typename T::Face face(f);
    const int j = f / Sh::Ff;
    if (face.dn != T::face_dir(j) || face.hi != T::face_hi(j)) return false;
    const double sg = face.hi ? 1. : -1.;
    int nl = 0;
    for (int m = 0; m < P1; m++) {
      at[(size_t)f * P1 + m] = face.at(m);
      int cc[3] = {face.c[0], face.c[1], face.c[2]};
      cc[face.dn] = m;
      if (T::face_fpt(j, cc) != f) return false;
      const size_t q = cc[0] + P1 * (cc[1] + P1 * cc[2]);
      const double l = w[T::L + face.hi * P1 + m], cr = w[T::C + face.hi * P1 + m];
      if (!(d->opp_spts_to_fpts[(size_t)f * S + q] == l && d->opp_correction[q * F + f] == cr &&
            d->opp_extrapolate_fn[((size_t)face.dn * F + f) * S + q] == l * sg))
        return false;
      if (c.prm.viscous && !(d->opp_correct_u[((size_t)face.dn * S + q) * F + f] == cr * sg)) return false;
      nl += l != 0.;
      nc += cr != 0.;
    }
    if (count_nonzeros(d->opp_spts_to_fpts + (size_t)f * S, S) != nl) return false;
    for (int x = 0; x < D; x++)
      if (count_nonzeros(d->opp_extrapolate_fn + ((size_t)x * F + f) * S, S) != (x == face.dn ? nl : 0)) return false;
  }
  if (count_nonzeros(d->opp_correction, (long long)S * F) != nc) return false;
  if (c.prm.viscous && count_nonzeros(d->opp_correct_u, (long long)D * S * F) != nc) return false;
  line = at;
  return true;
}

static bool build_ten(const Ctx& c, const fhip_desc* d, const std::vector<double>& d1, std::vector<double>& w,
                      std::vector<int>& line) {
  switch (c.z.D * 10 + c.z.P) {
    case 20: return build_ten<2, 0>(c, d, d1, w, line);
    case 21: return build_ten<2, 1>(c, d, d1, w, line);
    case 22: return build_ten<2, 2>(c, d, d1, w, line);
    case 23: return build_ten<2, 3>(c, d, d1, w, line);
    case 24: return build_ten<2, 4>(c, d, d1, w, line);
    case 25: return build_ten<2, 5>(c, d, d1, w, line);
    case 30: return build_ten<3, 0>(c, d, d1, w, line);
    case 31: return build_ten<3, 1>(c, d, d1, w, line);
    case 32: return build_ten<3, 2>(c, d, d1, w, line);
    case 33: return build_ten<3, 3>(c, d, d1, w, line);
    case 34: return build_ten<3, 4>(c, d, d1, w, line);
    default: return build_ten<3, 5>(c, d, d1, w, line);
  }
}

static bool build_tables(const Ctx& c, const fhip_desc* d, std::vector<char>& blob, size_t off[19]) {
  const int D = c.z.D, S = c.z.S, F = c.z.F, P1 = c.z.P + 1, NC = 2 * D;
  std::vector<int> ext_idx((size_t)F * P1, 0), efn_dir(F, 0), grd_idx((size_t)D * S * P1, 0),
      cor_idx((size_t)S * NC, 0), cu_idx((size_t)D * S * 2, 0);
  std::vector<double> ext_w((size_t)F * P1, 0.), efn_w((size_t)F * P1, 0.), grd_w((size_t)D * S * P1, 0.),
      cor_w((size_t)S * NC, 0.), cu_w((size_t)D * S * 2, 0.);
  for (int f = 0; f < F; f++) {
    // the face's normal direction: the only d with non-zero extrapolate_fn entries
    int dn = -1;
    for (int dd = 0; dd < D; dd++)
      if (count_nonzeros(d->opp_extrapolate_fn + ((size_t)dd * F + f) * S, S)) {
        if (dn >= 0) return false;
        dn = dd;
      }
    efn_dir[f] = dn < 0 ? 0 : dn;
    int n = 0;
    for (int q = 0; q < S; q++) {
      double v = d->opp_spts_to_fpts[(size_t)f * S + q];
      double w = dn < 0 ? 0. : d->opp_extrapolate_fn[((size_t)dn * F + f) * S + q];
      if (v == 0. && w == 0.) continue;
      if (n >= P1) return false;
      ext_idx[(size_t)f * P1 + n] = spt_lds(D, P1, q);
      ext_w[(size_t)f * P1 + n] = v;
      efn_w[(size_t)f * P1 + n] = w;
      n++;
    }
    for (int m = n; m < P1; m++) ext_idx[(size_t)f * P1 + m] = ext_idx[(size_t)f * P1];
  }
  for (int dd = 0; dd < D; dd++)
    for (int q0 = 0; q0 < S; q0++) {
      int n = 0;
      const double* const row = d->opp_grad_spts + ((size_t)dd * S + q0) * S;
      if (!each_nonzero(row, S, [&](int q) {
            if (n >= P1) return false;
            grd_idx[((size_t)dd * S + q0) * P1 + n] = spt_lds(D, P1, q);
            grd_w[((size_t)dd * S + q0) * P1 + n++] = row[q];
            return true;
          }))
        return false;
      for (int m = n; m < P1; m++) grd_idx[((size_t)dd * S + q0) * P1 + m] = spt_lds(D, P1, q0);
    }
  for (int q = 0; q < S; q++) {
    int n = 0;
    const double* const row = d->opp_correction + (size_t)q * F;
    if (!each_nonzero(row, F, [&](int f) {
          if (n >= NC) return false;
          cor_idx[(size_t)q * NC + n] = f;
          cor_w[(size_t)q * NC + n++] = row[f];
          return true;
        }))
      return false;
    if (c.prm.viscous)
      for (int dd = 0; dd < D; dd++) {
        int m = 0;
        const double* const ru = d->opp_correct_u + ((size_t)dd * S + q) * F;
        if (!each_nonzero(ru, F, [&](int f) {
              if (m >= 2) return false;
              cu_idx[((size_t)dd * S + q) * 2 + m] = f;
              cu_w[((size_t)dd * S + q) * 2 + m++] = ru[f];
              return true;
            }))
          return false;
      }
  }
  auto put = [&](const void* p, size_t bytes, size_t& o) {
    o = (blob.size() + 255) / 256 * 256;
    blob.resize(o + bytes);
    std::memcpy(blob.data() + o, p, bytes);
  };
  blob.clear();
  put(ext_w.data(), ext_w.size() * 8, off[1]);
  put(efn_dir.data(), efn_dir.size() * 4, off[2]);
  put(efn_w.data(), efn_w.size() * 8, off[3]);
  put(grd_idx.data(), grd_idx.size() * 4, off[4]);
  put(grd_w.data(), grd_w.size() * 8, off[5]);
  put(cor_idx.data(), cor_idx.size() * 4, off[6]);
  put(cor_w.data(), cor_w.size() * 8, off[7]);
  put(cu_idx.data(), cu_idx.size() * 4, off[8]);
  put(cu_w.data(), cu_w.size() * 8, off[9]);
  auto putf = [&](const std::vector<double>& v, size_t& o) {
    std::vector<float> f(v.begin(), v.end());
    put(f.data(), f.size() * 4, o);
  };
  putf(ext_w, off[10]);
  putf(efn_w, off[11]);
  putf(grd_w, off[12]);
  putf(cor_w, off[13]);
  putf(cu_w, off[14]);
  // the matrix-core path of FP64 P3 hexes needs the 1-D derivative matrix
  std::vector<double> d1;
  off[15] = off[16] = off[17] = off[18] = 0;
  std::vector<int> line = ext_idx;  // with the factors: by depth, zero weights included
  if (build_d1(c, d, d1)) {
    put(d1.data(), d1.size() * 8, off[15]);
    putf(d1, off[16]);
    std::vector<double> w;
    if (build_ten(c, d, d1, w, line)) {
      put(w.data(), w.size() * 8, off[17]);
      putf(w, off[18]);
    }
  } else if (D == 3 && P1 == 4) {
    return false;
  }
  const int W = (P1 + 3) / 4;
  std::vector<unsigned> packed((size_t)F * W, 0u);
  for (int f = 0; f < F; f++)
    for (int m = 0; m < P1; m++) packed[(size_t)f * W + m / 4] |= (unsigned)line[(size_t)f * P1 + m] << (8 * (m % 4));
  put(packed.data(), packed.size() * 4, off[0]);
  return true;
}

#endif  // FHIP_FAMILY

static __global__ void k_round_f32(long long n, const double* __restrict__ in, float* __restrict__ out) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    out[i] = float(in[i]);
}

// Geometry views of one precision (Work::JG .. nf).
static void set_geometry(Ctx& c, Work<double>& w) {
  FusedState& st = fs(c);
  w.JG = st.JGe;
  w.iJ = st.iJe;
  w.dA = st.dAe;
  w.nf = st.nfe;
}
static void set_geometry(Ctx& c, Work<float>& w) {
  FusedState& st = fs(c);
  const long long E = c.z.E, S = c.z.S, F = c.z.F, D = c.z.D;
  const long long n[4] = {E * D * D * S, E * S, E * F, E * D * F};
  const double* src[4] = {st.JGe, st.iJe, st.dAe, st.nfe};
  long long tot = 0;
  for (long long v : n) tot += (v + 63) / 64 * 64;
  float* m = dal<float>(tot);
  w.geo_mem = m;
  const float** dst[4] = {&w.JG, &w.iJ, &w.dA, &w.nf};
  for (int i = 0; i < 4; i++) {
    *dst[i] = m;
    hipLaunchKernelGGL(k_round_f32, dim3(1024), dim3(256), 0, c.stream, n[i], src[i], m);
    FCHK(hipGetLastError());
    m += (n[i] + 63) / 64 * 64;
  }
}

// A single-stage step with a CFL time step takes its dt from the wave speeds of
// the residual it is about to apply (solver::update), so they are formed, and on
// the refresh step replaced by the points' own, in launches of their own before it,
// with the common flux, which its stage kernel then reads (kGiven).
static bool face_first(const Ctx& c) { return !c.prm.viscous && c.z.nRK == 1 && c.prm.dt_type != 0; }
// Whether a step's first stage forms the elements' time steps itself.
static bool folds_dt(const Ctx& c) {
  return c.z.D == 2 && !c.prm.viscous && c.prm.dt_type == 2 && c.z.nRK > 1;
}

template <class R>
static void ensure_work(Ctx& c) {
  Work<R>& w = fs(c).work<R>();
  if (w.ready) return;
  const long long E = c.z.E, S = c.z.S, F = c.z.F, N = c.z.N;
  w.Ufe = dal<R>(E * N * F);
  if (!c.prm.viscous) w.Ufe2 = dal<R>(E * N * F);
  if (c.prm.viscous) {
    // inviscid runs keep divF and the discontinuous normal flux in the stage kernel
    w.divFe = dal<R>(E * N * S);
    w.Bve = dal<R>(E * N * F);
    if (kJumpOut<R>) w.Jne = dal<R>(E * N * F);
  }
  if (sizeof(R) == 4 && c.z.nRK > 1 && c.prm.time_type < 5) w.Rst = dal<R>((long long)(c.z.nRK - 1) * E * N * S);
  w.Us = dal<R>(E * N * S);
  set_geometry(c, w);
  w.ready = true;
}

#ifndef FHIP_FAMILY
// The face's normal, its left element's, at every element flux point (on the host
// it was the longest part of setting up a 23^3 P4 mesh: 30 of 230 ms).
static __global__ void k_face_normals(long long n, int F, int D, const int* __restrict__ fpart,
                                      const double* __restrict__ norme, double* __restrict__ nfe) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int code = fpart[q];
  const long long l = (code & 3) == 1 ? code >> 2 : q, e = q / F, f = q - e * F, eL = l / F, fL = l - eL * F;
  for (int x = 0; x < D; x++) nfe[(e * D + x) * F + f] = norme[(eL * D + x) * F + fL];
}

bool fused_setup(Ctx& c, const fhip_desc* d) {
  const Sizes& z = c.z;
  if (z.P < 0 || z.P > 5) return false;
  std::vector<char> blob;
  size_t off[19];
  if (!build_tables(c, d, blob, off)) return false;
  auto* st = new FusedState();
  c.fused = st;
  st->tab_mem = dal<char>(blob.size());
  FCHK(hipMemcpy(st->tab_mem, blob.data(), blob.size(), hipMemcpyHostToDevice));
  char* base = (char*)st->tab_mem;
  st->tb = Tabs{(const double*)(base + off[1]), (const int*)(base + off[2]),
                (const double*)(base + off[3]), (const int*)(base + off[4]),    (const double*)(base + off[5]),
                (const int*)(base + off[6]),    (const double*)(base + off[7]), (const int*)(base + off[8]),
                (const double*)(base + off[9]), (const float*)(base + off[10]), (const float*)(base + off[11]),
                (const float*)(base + off[12]), (const float*)(base + off[13]), (const float*)(base + off[14]),
                off[15] ? (const double*)(base + off[15]) : nullptr, off[16] ? (const float*)(base + off[16]) : nullptr,
                off[17] ? (const double*)(base + off[17]) : nullptr, off[18] ? (const float*)(base + off[18]) : nullptr,
                (const unsigned*)(base + off[0])};
  const long long E = z.E, S = z.S, F = z.F, N = z.N, D = z.D;
  st->stream = E * N * S * (long long)sizeof(double) > kStreamBytes;
  st->Ue = dal<double>(E * N * S);
  st->Uacc = dal<double>(E * N * S);
  st->divF0e = dal<double>(E * N * S);
  st->waveSpe = dal<double>(E * F);
  const double none[2] = {INFINITY, 0.0};  // no minimum yet, no block finished
  st->dtAcc = dal<double>(2);
  st->dtTicket = reinterpret_cast<unsigned*>(st->dtAcc + 1);
  FCHK(hipMemcpy(st->dtAcc, none, sizeof(none), hipMemcpyHostToDevice));
  st->JGe = dal<double>(E * D * D * S);
  st->detJe = dal<double>(E * S);
  st->iJe = dal<double>(E * S);
  st->norme = dal<double>(E * D * F);
  st->dAe = dal<double>(E * F);
  {
    std::vector<double> jg((size_t)E * D * D * S), dj((size_t)E * S), nr((size_t)E * D * F), da((size_t)E * F);
    for (long long r = 0; r < D; r++)
      for (long long s = 0; s < S; s++)
        for (long long e = 0; e < E; e++)
          for (long long x = 0; x < D; x++)
            jg[((e * D + r) * D + x) * S + s] = d->jginv_spts[((r * S + s) * E + e) * D + x];
    for (long long s = 0; s < S; s++)
      for (long long e = 0; e < E; e++) dj[e * S + s] = d->detjac_spts[s * E + e];
    for (long long f = 0; f < F; f++)
      for (long long e = 0; e < E; e++) {
        da[e * F + f] = d->da_fpts[f * E + e];
        for (long long x = 0; x < D; x++) nr[(e * D + x) * F + f] = d->norm_fpts[(f * E + e) * D + x];
      }
    FCHK(hipMemcpy(st->JGe, jg.data(), jg.size() * 8, hipMemcpyHostToDevice));
    FCHK(hipMemcpy(st->detJe, dj.data(), dj.size() * 8, hipMemcpyHostToDevice));
    for (double& v : dj) v = 1. / v;
    FCHK(hipMemcpy(st->iJe, dj.data(), dj.size() * 8, hipMemcpyHostToDevice));
    FCHK(hipMemcpy(st->norme, nr.data(), nr.size() * 8, hipMemcpyHostToDevice));
    FCHK(hipMemcpy(st->dAe, da.data(), da.size() * 8, hipMemcpyHostToDevice));
  }
  // batching: meshes, boundary-state table
  if (d->n_meshes > 1 || d->mesh_ele_start) {
    int nm = std::max(1, d->n_meshes);
    if (!d->mesh_ele_start) throw std::invalid_argument("n_meshes > 1 needs mesh_ele_start");
    st->h_meshStart.assign(d->mesh_ele_start, d->mesh_ele_start + nm + 1);
    if (st->h_meshStart[0] != 0 || st->h_meshStart[nm] != z.E) throw std::invalid_argument("mesh_ele_start must span [0, nEles]");
    std::vector<int> em(z.E);
    for (int m = 0; m < nm; m++) {
      if (st->h_meshStart[m + 1] <= st->h_meshStart[m]) throw std::invalid_argument("mesh_ele_start must increase");
      for (int e = st->h_meshStart[m]; e < st->h_meshStart[m + 1]; e++) em[e] = m;
    }
    st->nMesh = nm;
    st->eleMesh = dal<int>(z.E);
    st->meshStart = dal<int>(nm + 1);
    st->meshDt = dal<double>(nm);
    st->meshRes = dal<double>((size_t)nm * z.N);
    FCHK(hipMemcpy(st->eleMesh, em.data(), em.size() * 4, hipMemcpyHostToDevice));
    FCHK(hipMemcpy(st->meshStart, st->h_meshStart.data(), (nm + 1) * 4, hipMemcpyHostToDevice));
  } else {
    st->h_meshStart = {0, z.E};
  }
  if (d->n_bnd_states > 0) {
    if (!d->bnd_states || !d->face_bnd_state) throw std::invalid_argument("boundary-state table needs bnd_states and face_bnd_state");
    st->bst = dal<double>((size_t)d->n_bnd_states * 5);
    FCHK(hipMemcpy(st->bst, d->bnd_states, (size_t)d->n_bnd_states * 5 * 8, hipMemcpyHostToDevice));
  }
  {
    std::vector<int> pl(z.nFaceFpts), pr(z.nFaceFpts), bc(z.nFaceFpts);
    for (int t = 0; t < z.nFaceFpts; t++) {
      int a = c.h_ptL[t];  // fpt*E + ele
      pl[t] = (a % z.E) * z.F + a / z.E;
      int r = c.h_ptR[t];
      pr[t] = (r < 0) ? -1 : (r % z.E) * z.F + r / z.E;
      int row = -1;
      if (r < 0 && d->n_bnd_states > 0) {
        row = d->face_bnd_state[t / z.Ff];
        if (row < -1 || row >= d->n_bnd_states) throw std::invalid_argument("face_bnd_state out of range");
      }
      bc[t] = (r < 0) ? (d->face_bc[t / z.Ff] | ((row + 1) << 4)) : -1;
    }
    {
      // every element flux point must lie on exactly one face point pair;
      // its code: 4 * partner flux point + side, or 4 * boundary slot + 2, and
      // the face's normal
      if (E * F >= (1LL << 29)) throw std::invalid_argument("fused path: more than 2^29 element flux points");
      std::vector<int> part((size_t)E * F, -1), bb;
      for (int t = 0; t < z.nFaceFpts; t++) {
        if (part[pl[t]] != -1 || (pr[t] >= 0 && part[pr[t]] != -1)) {
          fused_release(c);
          return false;
        }
        if (pr[t] < 0) {
          part[pl[t]] = 4 * (int)bb.size() + 2;
          bb.push_back(bc[t]);
        } else {
          part[pl[t]] = 4 * pr[t];
          part[pr[t]] = 4 * pl[t] + 1;
        }
      }
      for (int q : part)
        if (q == -1) {
          fused_release(c);
          return false;
        }
      st->nBnd = (int)bb.size();
      part.insert(part.end(), bb.begin(), bb.end());
      st->fpart = dal<int>(part.size());
      st->bndBc = st->fpart + E * F;
      FCHK(hipMemcpy(st->fpart, part.data(), part.size() * 4, hipMemcpyHostToDevice));
      st->nfe = dal<double>(E * D * F);
      hipLaunchKernelGGL(k_face_normals, dim3(nblk(E * F, 256)), dim3(256), 0, c.stream, E * F, (int)F, (int)D,
                         st->fpart, st->norme, st->nfe);
      FCHK(hipGetLastError());
    }
  }
  return true;
}

void fused_mesh_residuals(Ctx& c, int type, double* out) {
  FusedState& st = fs(c);
  const int nm = st.nMesh;
  int* start = st.meshStart;
  double* res = st.meshRes;
  int* tmpStart = nullptr;
  double* tmpRes = nullptr;
  if (nm == 1) {  // single mesh: a two-entry range
    tmpStart = dal<int>(2);
    tmpRes = dal<double>(c.z.N);
    int h[2] = {0, c.z.E};
    FCHK(hipMemcpyAsync(tmpStart, h, 8, hipMemcpyHostToDevice, c.stream));
    start = tmpStart;
    res = tmpRes;
  }
  hipLaunchKernelGGL(k_mesh_res, dim3(nm), dim3(256), 0, c.stream, c.z.S, c.z.N, type, start, st.divF0e, st.detJe, c.ws, res);
  FCHK(hipGetLastError());
  FCHK(hipMemcpyAsync(out, res, (size_t)nm * c.z.N * 8, hipMemcpyDeviceToHost, c.stream));
  FCHK(hipStreamSynchronize(c.stream));
  if (tmpStart) (void)hipFree(tmpStart);
  if (tmpRes) (void)hipFree(tmpRes);
}

int fused_n_meshes(Ctx& c) { return fs(c).nMesh; }

void fused_set_active(Ctx& c, const int* active) {
  FusedState& st = fs(c);
  if (!st.active || !st.eleMesh) c.drop_graphs();  // captured steps hold null flag pointers
  if (!st.active) st.active = dal<int>(st.nMesh);
  if (!st.eleMesh) {  // single mesh: every element belongs to mesh 0
    std::vector<int> em(c.z.E, 0);
    st.eleMesh = dal<int>(c.z.E);
    FCHK(hipMemcpy(st.eleMesh, em.data(), em.size() * 4, hipMemcpyHostToDevice));
  }
  FCHK(hipMemcpyAsync(st.active, active, (size_t)st.nMesh * 4, hipMemcpyHostToDevice, c.stream));
  FCHK(hipStreamSynchronize(c.stream));
}

void fused_release(Ctx& c) {
  if (c.fused) delete reinterpret_cast<FusedState*>(c.fused);
  c.fused = nullptr;
}

#endif  // FHIP_FAMILY

// ---- per-order / per-precision dispatch ------------------------------------

static double cfl_limit_f(int order) {  // getCFLLimit, src/global.cpp:81-105
  static const double t[6] = {1.393, 0.464, 0.235, 0.1453, 0.100, 0.0736};
  if (order < 0 || order > 5) throw std::invalid_argument("CFL limit not available for this order!");
  return t[order];
}

template <int D, int P, class R>
struct Runner {
  using Sh = Shape<D, P>;
  static constexpr int S = Sh::S, F = Sh::F, N = Sh::N;
  static const char* nm(const char* f64, const char* f32) { return sizeof(R) == 8 ? f64 : f32; }
  // Streamed (nontemporal) stores pay only when the rows that a kernel stores are
  // whole 64-byte blocks, the memory's write granule: a partial block written
  // past the caches costs a read-modify-write.
  // The element kernels store rows of S or F values per field; a wave's
  // streamed store covers whole blocks only when those rows are whole blocks.
  static constexpr bool kEleRowsWhole = (S * sizeof(R)) % 64 == 0 && (F * sizeof(R)) % 64 == 0;
  static int& blk(Ctx& c, int k) { return fs(c).nt[tune_form(c, sizeof(R) == 4)][k]; }
  // Elements of a block of the stage kernel's form with solution and flux points
  // apart, within nt threads (one at least), and its threads: whole waves of
  // solution points, then whole waves of flux points
  static constexpr int stage_threads(int EB) { return up64(EB * S) + up64(EB * Sh::F); }
  static_assert(stage_threads(1) <= kMaxBlock);
  static int stage_eles(int nt) {
    int EB = 1;
    while (stage_threads(EB + 1) <= nt) EB++;
    return EB;
  }
  static constexpr size_t stage_lds(size_t EB) { return EB * N * (S + D * S + Sh::F) * sizeof(R); }
  // Which form of the stage kernel: apart while every wave of the launch can be
  // resident at once (256 CUs x 16 waves), together beyond.  Measured per stage,
  // apart / together, tuned sizes: quads P3 32^2 (512 waves) 5.9 / 6.6 us, 64^2
  // (2048) 7.2 / 7.6, 96^2 (4608) 12.5 / 11.5; P4 hexes 8^3 (2200) 10.4 / 10.6,
  // 12^3 (7425) 28.4 / 23.9; FP32 P3 hexes 8^3 (1280) 7.3 / 9.9, 12^3 (4320) 13.9 /
  // 13.3, 16^3 (10240) 23.2 / 19.5.  FP64 hexes of orders 1 to 3, whose
  // registers hold the other form to 3 waves per SIMD and whose blocks fill
  // their waves, gain further up: P2 20^3 (10125) 27.7 / 30.3, P3 16^3 (10240)
  // 26.4 / 28.9, P2 28^3 (27783) 64.2 / 62.2.  P0, whose solution points would take 4
  // or 6 rounds over flux points, stays apart at every size: quads 300x200 (4688)
  // 15.1 / 22.7, 600x500 (23438) 42 / 49, hexes 60^3 (23625) 57 / 70, with walls 60 / 84.
  static constexpr long long kApartWaves =
      P == 0 ? 1ll << 40 : (D == 3 && P <= 3 && sizeof(R) == 8 ? 12288 : 4096);
  static bool apart(const Ctx& c) { return (long long)c.z.E * (S + F) <= kApartWaves * 64; }
  // LDS bytes of an element kernel at block size nt (0 for the face kernel)
  static size_t lds(int k, int nt, bool visc) {
    const size_t EB = nt / S;
    if (k == kExtrap) return EB * N * S * sizeof(R);
    if (k == kVolume) return visc ? volume_lds(EB) : EB * N * (S + D * S + F) * sizeof(R);
    if (k == kRk) return EB * N * (S + F) * sizeof(R);
    return 0;
  }
  // (a viscous volume block holds nt / kVolThreads elements, which is never more)
  static constexpr size_t volume_lds(size_t EB) {
    return EB * N * ((!kJumpOut<R> && jump_over_u<D, P> && F > S ? F : S) + (F > D * S ? F : D * S)) * sizeof(R);
  }
  static bool valid(int k, int nt, bool visc) {
    if (nt < 64 || nt > kMaxBlock) return false;
    if (k == kFaceInv || k == kFaceBnd) return true;
    return nt >= S && lds(k, nt, visc) <= kMaxLds;
  }
  static void launch_extrap(Ctx& c, int nt) {
    FusedState& st = fs(c);
    Work<R>& w = st.work<R>();
    // the FP32 stage copy starts from the state; the FP64 one is first
    // written by a step's first stage (which reads the state itself)
    auto* kern = st.tb.w1 ? k_extrap<D, P, R, true> : k_extrap<D, P, R, false>;
    hipLaunchKernelGGL(kern, dim3(nblk(c.z.E, nt / S)), dim3(nt), lds(kExtrap, nt, false), c.stream, c.z.E, st.Ue, w.Ufe, sizeof(R) == 4 ? w.Us : nullptr, st.tb);
    st.flipped = false;
    FCHK(hipGetLastError());
  }
  // U at the flux points of the current state
  static R* cur_ufe(Ctx& c) { return fs(c).flipped ? fs(c).work<R>().Ufe2 : fs(c).work<R>().Ufe; }
  // viscous runs: the volume kernel.  Quads and FP32 are held to 4 waves per
  // SIMD (128 VGPRs); FP64 hexes and the BF16 forms, which spill under that hold, to 3 (168 VGPRs:
  // P3 without spills, where the unheld compiler would take 211 and leave 2
  // waves)
  template <bool NT, bool BND, bool TEN>
  static void launch_volume_t(Ctx& c, int nt, bool wave) {
    FusedState& st = fs(c);
    Work<R>& w = st.work<R>();
    const VFace<R> vf{st.fpart, w.Ufe, w.nf, w.dA, w.Bve, w.Jne, wave ? st.waveSpe : nullptr, st.bndBc, st.bst};
    const R* us = (sizeof(R) == 4 || st.read_stage) ? w.Us : nullptr;
    const int EB = nt / kVolThreads<D, P>;
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(nblk(c.z.E, EB)), dim3(nt), volume_lds(EB), c.stream, c.z.E, st.Ue, us,
                         w.JG, w.iJ, w.divFe, vf, st.tb, c.ph);
    };
    if constexpr (kBf16<D, P, R>) {
      if (c.bf16 == 2) go(k_volume_w3<D, P, R, NT, BND, TEN, 2>);
      else if (c.bf16 == 3) go(k_volume_w3<D, P, R, NT, BND, TEN, 3>);
      else go(k_volume_w4<D, P, R, NT, BND, TEN>);
    } else if constexpr (kHold<D, R>) {
      go(k_volume_w4<D, P, R, NT, BND, TEN>);
    } else {
      go(k_volume_w3<D, P, R, NT, BND, TEN>);
    }
    FCHK(hipGetLastError());
  }
  // inviscid runs: the stage kernel with the RK update ra
  template <bool NT, bool BND, bool TEN, bool APART, int FORM>
  static void launch_stage_t(Ctx& c, int nt, RkArgs<R> ra, bool fold) {
    FusedState& st = fs(c);
    Work<R>& w = st.work<R>();
    // wave speeds are read by the next step's dt and after the call: stages
    // that another stage follows leave them
    const bool wave = (ra.fin && FORM != kGiven) || ra.mode == 5 || ra.mode == 7 || ra.mode == 8;
    const StageFace<R> fc{st.fpart, cur_ufe(c), w.Ufe2, w.nf, w.dA, wave ? st.waveSpe : nullptr, st.bndBc,
                          st.bst, fold ? c.wf : nullptr, st.waveSpe, st.dAe, st.vole,
                          fold ? c.prm.cfl * cfl_limit_f(P) : 0., c.eleDt};
    ra.Ufe = FORM == kGiven || st.flipped ? w.Ufe : w.Ufe2;
    const R* us = (sizeof(R) == 4 || st.read_stage) ? w.Us : nullptr;
    int EB = APART ? stage_eles(nt) : nt / S;
    auto bytes = [&] { return stage_lds(EB) + (FORM == kMakeSrc ? EB * F * sizeof(double) : 0); };
    while (EB > 1 && bytes() > kMaxLds) EB--;
    const int threads = APART ? stage_threads(EB) : (EB == nt / S ? nt : EB * S);
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(nblk(c.z.E, EB)), dim3(threads), bytes(), c.stream, c.z.E, EB, st.Ue, us,
                         w.JG, fc, st.tb, c.ph, ra);
    };
    if constexpr (kBf16<D, P, R>) {
      if (c.bf16 == 2) go(k_stage_w3<D, P, R, NT, BND, TEN, APART, 2, FORM>);
      else if (c.bf16 == 3) go(k_stage_w3<D, P, R, NT, BND, TEN, APART, 3, FORM>);
      else go(k_stage_w4<D, P, R, NT, BND, TEN, APART, FORM>);
    } else if constexpr (kHold<D, R>) {
      go(k_stage_w4<D, P, R, NT, BND, TEN, APART, FORM>);
    } else {
      go(k_stage_w3<D, P, R, NT, BND, TEN, APART, 0, FORM>);
    }
    FCHK(hipGetLastError());
  }
  // (instances that stream exist only for the orders whose rows are whole)
  static void launch_volume(Ctx& c, int nt, bool wave) {
    const bool bnd = fs(c).nBnd > 0;
    if (!fs(c).tb.w1) return launch_volume_t<false, true, false>(c, nt, wave);
    if constexpr (kEleRowsWhole) {
      if (fs(c).stream) return bnd ? launch_volume_t<true, true, true>(c, nt, wave) : launch_volume_t<true, false, true>(c, nt, wave);
    }
    if (bnd) launch_volume_t<false, true, true>(c, nt, wave);
    else launch_volume_t<false, false, true>(c, nt, wave);
  }
  static void launch_stage(Ctx& c, int nt, const RkArgs<R>& ra, bool fold = false, bool given = false) {
    const bool bnd = fs(c).nBnd > 0;
    if (given) return launch_stage_f<kGiven, false>(c, nt, ra, fold);
    if constexpr (D == 2) {
      if (ra.makeSrc)
        return bnd ? launch_stage_f<kMakeSrc, true>(c, nt, ra, fold) : launch_stage_f<kMakeSrc, false>(c, nt, ra, fold);
    }
    bnd ? launch_stage_f<kUsual, true>(c, nt, ra, fold) : launch_stage_f<kUsual, false>(c, nt, ra, fold);
  }
  // (with the flux given there is no boundary state to form)
  template <int FORM, bool BND>
  static void launch_stage_f(Ctx& c, int nt, const RkArgs<R>& ra, bool fold) {
    // operators read from their tables: one instance for every mesh
    if (!fs(c).tb.w1) return launch_stage_t<false, FORM != kGiven, false, false, FORM>(c, nt, ra, fold);
    if constexpr (kEleRowsWhole && FORM != kMakeSrc) {
      if (fs(c).stream) return launch_stage_t<true, BND, true, false, FORM>(c, nt, ra, fold);
    }
    if (apart(c)) return launch_stage_t<false, BND, true, true, FORM>(c, nt, ra, fold);
    if constexpr (P > 0) launch_stage_t<false, BND, true, false, FORM>(c, nt, ra, fold);
  }
  static RkArgs<R> rk_args(Ctx& c, int mode, double a, double b, bool write0, int stage, bool make_src = false) {
    FusedState& st = fs(c);
    Work<R>& w = st.work<R>();
    RkB bs{};
    for (int j = 0; j < c.z.nRK && j < 8; j++) bs.b[j] = c.prm.rk_b[j];
    // residual modes 7 and 8: the source is the array written, or read
    double* d0 = mode == 7 ? st.srce : (write0 ? st.divF0e : nullptr);
    const double* src = mode == 8 ? st.srce : (st.use_src && mode != 7 ? st.srce : nullptr);
    return RkArgs<R>{mode, a, b, st.detJe, c.d_dt, c.eleDt,
                     c.prm.dt_type == 2 ? 1 : (c.prm.dt_type == 1 && st.nMesh > 1 ? 2 : 0), st.Ue,
                     st.Uacc,
                     d0, st.eleMesh, st.meshDt, st.active, src,
                     (w.Rst && !st.use_src) ? w.Rst : nullptr, stage, bs, w.Us,
                     (mode == 2 || mode == 3 || (mode == 4 && stage == c.z.nRK - 1)) ? 1 : 0, w.Ufe,
                     make_src ? st.srce : nullptr};
  }
  // the RK kernel of viscous runs; inviscid runs do its work at the end of
  // their stage kernel
  static void launch_rk(Ctx& c, int nt, int mode, double a, double b, bool write0, int stage = 0) {
    FusedState& st = fs(c);
    Work<R>& w = st.work<R>();
    auto* kern = st.tb.w1 ? k_rk<D, P, R, false, true> : k_rk<D, P, R, false, false>;
    if constexpr (kEleRowsWhole) {
      if (st.tb.w1 && st.stream) kern = k_rk<D, P, R, true, true>;
    }
    hipLaunchKernelGGL(kern, dim3(nblk(c.z.E, nt / S)), dim3(nt), lds(kRk, nt, false), c.stream, c.z.E, w.divFe,
                       rk_args(c, mode, a, b, write0, stage), st.tb, st.fpart, w.dA, w.Bve, w.Jne);
    FCHK(hipGetLastError());
  }
  static void extrap(Ctx& c) {
    Launch L(c, nm("fused_extrapolate", "mixed_extrapolate"));
    launch_extrap(c, blk(c, kExtrap));
  }
  // The transfers in LDS into this level (restriction: its elements [e0, e0 + ne)),
  // with U at its flux points (prolongation: if extrap).  False, and nothing
  // done, where they do not fit.
  static int transfer_eles() { return N * S <= kMaxBlock ? std::max(1, 256 / (N * S)) : 0; }
  static bool restrict_lds(Ctx& c, long long e0, long long ne, int Sf, int kc, const double* A, const double* Uf,
                           const double* divFf, double* solc) {
    FusedState& st = fs(c);
    Work<R>& w = st.work<R>();
    const int EB = transfer_eles(), nr = EB * N;
    const size_t bytes = ((size_t)S * Sf + 2 * (size_t)nr * Sf) * sizeof(double) + (size_t)nr * S * sizeof(R);
    if (!EB || bytes > kMaxLds) return false;
    auto* kern = st.tb.w1 ? k_restrict_lds<D, P, R, true> : k_restrict_lds<D, P, R, false>;
    const long long off = e0 * N * S;
    hipLaunchKernelGGL(kern, dim3(nblk(ne, EB)), dim3(nr * S), bytes, c.stream, (int)ne, EB, Sf, kc, A, Uf, divFf,
                       st.Ue + off, st.srce + off, solc + off, w.Ufe + e0 * N * F,
                       sizeof(R) == 4 ? w.Us + off : nullptr, st.tb);
    st.flipped = false;
    FCHK(hipGetLastError());
    return true;
  }
  static bool prolong_lds(Ctx& c, int Sc, int kc, const double* A, const double* Uc, const double* solc, bool extrap) {
    FusedState& st = fs(c);
    Work<R>& w = st.work<R>();
    const int EB = transfer_eles(), nr = EB * N;
    const size_t bytes = ((size_t)S * Sc + (size_t)nr * Sc) * sizeof(double) + (size_t)nr * S * sizeof(R);
    if (!EB || bytes > kMaxLds) return false;
    auto* kern = st.tb.w1 ? k_prolong_lds<D, P, R, true> : k_prolong_lds<D, P, R, false>;
    hipLaunchKernelGGL(kern, dim3(nblk(c.z.E, EB)), dim3(nr * S), bytes, c.stream, c.z.E, EB, Sc, kc, A, Uc, solc,
                       st.Ue, extrap ? w.Ufe : nullptr, sizeof(R) == 4 ? w.Us : nullptr, st.tb);
    if (extrap) st.flipped = false;
    FCHK(hipGetLastError());
    return true;
  }
  static void wave(Ctx& c) {
    FusedState& st = fs(c);
    long long n = (long long)c.z.E * Sh::F;
    Launch L(c, nm("fused_wave_speed", "mixed_wave_speed"));
    hipLaunchKernelGGL((k_wave_em<D, P, R>), dim3(nblk(n, 256)), dim3(256), 0, c.stream, c.z.E, cur_ufe(c), st.norme,
                       st.waveSpe, c.ph.gamma);
    FCHK(hipGetLastError());
  }
  // Threads and blocks of the dt kernels, which have `eles` elements in flight in a
  // block of 256 (blocks of merged meshes take no turns, so they are not limited).
  static std::pair<int, unsigned> dt_grid(Ctx& c, int eles, unsigned limit) {
    const unsigned small = nblk(c.z.E, eles);
    if (small <= limit || fs(c).nMesh > 1) return {256, small};
    return {1024, std::min(nblk(c.z.E, 4 * eles), kDtBlocks)};
  }
  static void dt(Ctx& c, double cflfac) {
    FusedState& st = fs(c);
    {
      // one mesh: the element kernel's last block forms the global minimum
      Launch L(c, nm("fused_ele_dt", "mixed_ele_dt"));
      const auto [nt, nb] = dt_grid(c, 256 / kDtLanes<F> * kDtEles<D>, kDtSmall<D>);
      auto* kern = nt == 1024 ? k_ele_dt_em<D, P, 1024> : k_ele_dt_em<D, P, 256>;
      hipLaunchKernelGGL(kern, dim3(nb), dim3(nt), 0, c.stream, c.z.E, st.vole, c.wf, st.waveSpe, st.dAe, cflfac,
                         c.eleDt, st.dtAcc, st.nMesh == 1 ? st.dtTicket : nullptr, c.d_dt);
      FCHK(hipGetLastError());
    }
    mesh_dt(c);
  }
  // The common flux (into Ufe2), its wave speeds and the time steps from them; refresh:
  // from the points' own speeds, which replace these.
  static void wave_dt(Ctx& c, double cflfac, bool refresh) {
    FusedState& st = fs(c);
    Work<R>& w = st.work<R>();
    const int n = c.z.E * F;
    if (n > kWaveDtPoints || refresh) {
      {
        Launch L(c, nm("fused_face_inviscid", "mixed_face_inviscid"));
        const int nt = blk(c, kFaceInv);
        hipLaunchKernelGGL((k_pair_wave<D, P, R>), dim3(nblk(n, nt)), dim3(nt), 0, c.stream, n, st.fpart, cur_ufe(c),
                           w.nf, st.bndBc, st.waveSpe, w.Ufe2, c.ph, st.bst);
        FCHK(hipGetLastError());
      }
      if (refresh) wave(c);
      return dt(c, cflfac);
    }
    {
      Launch L(c, nm("fused_wave_dt", "mixed_wave_dt"));
      const auto [nt, nb] = dt_grid(c, 256 / kWaveDtLanes<D>, kDtSmall<D>);
      auto* kern = nt == 1024 ? k_wave_dt<D, P, R, 1024> : k_wave_dt<D, P, R, 256>;
      hipLaunchKernelGGL(kern, dim3(nb), dim3(nt), 0, c.stream, c.z.E, st.fpart, cur_ufe(c), w.nf, st.bndBc, st.bst,
                         c.ph, st.vole, c.wf, st.waveSpe, w.Ufe2, st.dAe, cflfac, c.eleDt, st.dtAcc,
                         st.nMesh == 1 ? st.dtTicket : nullptr, c.d_dt);
      FCHK(hipGetLastError());
    }
    mesh_dt(c);
  }
  // merged meshes: per-mesh minima for a global CFL dt per mesh (a local CFL dt
  // uses the element values alone)
  static void mesh_dt(Ctx& c) {
    FusedState& st = fs(c);
    if (st.nMesh == 1 || c.prm.dt_type != 1) return;
    Launch L(c, nm("fused_dt_min", "mixed_dt_min"));
    hipLaunchKernelGGL(k_mesh_dt_min, dim3(st.nMesh), dim3(256), 0, c.stream, st.meshStart, c.eleDt, st.meshDt);
    FCHK(hipGetLastError());
  }
  // calcResidual up to what the RK update needs: the volume kernel of viscous
  // runs (wave: with the wave speeds, which stages that another stage follows
  // leave); nothing on inviscid ones, whose stage kernel runs in rk below
  static void residual(Ctx& c, bool wave) {
    if (!c.prm.viscous) return;
    Launch L(c, nm("fused_volume_viscous", "mixed_volume_viscous"));
    launch_volume(c, blk(c, kVolume), wave);
  }
  static void rk(Ctx& c, int mode, double a, double b, bool write0, int stage, bool make_src) {
    if (!c.prm.viscous) {
      Launch L(c, nm("fused_stage", "mixed_stage"));
      const bool update = mode != 5 && mode != 7 && mode != 8, given = update && face_first(c);
      launch_stage(c, blk(c, kVolume), rk_args(c, mode, a, b, write0, stage, make_src),
                   folds_dt(c) && (mode == 0 || mode == 6), given);
      if (update && !given) fs(c).flipped = !fs(c).flipped;
      return;
    }
    Launch L(c, nm("fused_rk_update", "mixed_rk_update"));
    launch_rk(c, blk(c, kRk), mode, a, b, write0, stage);
  }
  // Time every valid block size of every kernel on this context's data and
  // keep the fastest.  The RK kernel (and the stage kernel of inviscid runs,
  // which includes the update) runs in its middle-stage mode, which rewrites
  // U and the RK accumulator: both are saved and restored, as are the wave
  // speeds; block shapes never change results.
  static void tune(Ctx& c) {
    FusedState& st = fs(c);
    const bool visc = c.prm.viscous != 0;
    const long long nS = (long long)c.z.E * N * S, nW = (long long)c.z.E * F;
    double *bU = nullptr, *bA = nullptr, *bW = nullptr;
    FCHK(hipMalloc(&bU, nS * 8));
    FCHK(hipMalloc(&bA, nS * 8));
    FCHK(hipMalloc(&bW, nW * 8));
    FCHK(hipMemcpyAsync(bU, st.Ue, nS * 8, hipMemcpyDeviceToDevice, c.stream));
    FCHK(hipMemcpyAsync(bA, st.Uacc, nS * 8, hipMemcpyDeviceToDevice, c.stream));
    FCHK(hipMemcpyAsync(bW, st.waveSpe, nW * 8, hipMemcpyDeviceToDevice, c.stream));
    hipEvent_t e0, e1;
    FCHK(hipEventCreate(&e0));
    FCHK(hipEventCreate(&e1));
    // multiples of the 64-wide wavefront; element kernels hold floor(NT/S)
    // elements, so sizes between the powers of two pay off where S divides them
    const int cand[7] = {64, 128, 192, 256, 320, 384, 512};
    for (int k = kExtrap; k <= kRk; k++) {
      if (k == kFaceBnd || k == kFaceInv || (k == kRk && !visc)) continue;
      auto run = [&](int nt) {
        switch (k) {
          case kExtrap: launch_extrap(c, nt); break;
          case kVolume:
            if (visc) launch_volume(c, nt, false);
            else launch_stage(c, nt, rk_args(c, 1, 0.5, 1. / 3., false, 0));
            break;
          default: launch_rk(c, nt, 1, 0.5, 1. / 3., false);
        }
      };
      int best = blk(c, k);
      float bt = 1e30f;
      for (int nt : cand) {
        if (!valid(k, nt, visc)) continue;
        run(nt);
        FCHK(hipEventRecord(e0, c.stream));
        for (int r = 0; r < 3; r++) run(nt);
        FCHK(hipEventRecord(e1, c.stream));
        FCHK(hipEventSynchronize(e1));
        float ms = 0;
        FCHK(hipEventElapsedTime(&ms, e0, e1));
        if (ms < bt) bt = ms, best = nt;
      }
      blk(c, k) = best;
      run(best);  // leave this kernel's outputs for the next one's inputs
    }
    FCHK(hipMemcpyAsync(st.Ue, bU, nS * 8, hipMemcpyDeviceToDevice, c.stream));
    FCHK(hipMemcpyAsync(st.Uacc, bA, nS * 8, hipMemcpyDeviceToDevice, c.stream));
    FCHK(hipMemcpyAsync(st.waveSpe, bW, nW * 8, hipMemcpyDeviceToDevice, c.stream));
    FCHK(hipStreamSynchronize(c.stream));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(bU);
    (void)hipFree(bA);
    (void)hipFree(bW);
    launch_extrap(c, blk(c, kExtrap));  // U at the faces of the restored state
  }
  static bool check(Ctx& c, const int* nt) {
    const bool visc = c.prm.viscous != 0;
    for (int k = kExtrap; k <= kRk; k++)
      if (!valid(k, nt[k], visc)) return false;
    return true;
  }
  // Each block size brought within its kernel's limits: the default of 256
  // threads exceeds kMaxLds for the RK kernel and the viscous volume kernel
  // of P0 hexes (256 elements of 7 FP64 N-vectors per block)
  static void fit(Ctx& c) {
    const bool visc = c.prm.viscous != 0;
    for (int k = kExtrap; k <= kRk; k++)
      while (!valid(k, blk(c, k), visc) && blk(c, k) > 64) blk(c, k) -= 64;
  }
  static void ensure(Ctx& c) {
    ensure_work<R>(c);
    fit(c);
    FusedState& st = fs(c);
    if (!st.vole) {
      st.vole = dal<double>(c.z.E);
      hipLaunchKernelGGL((k_ele_vol<D, P>), dim3(nblk(c.z.E, 256)), dim3(256), 0, c.stream, c.z.E, st.detJe, c.ws,
                         st.vole);
      FCHK(hipGetLastError());
    }
  }
};

struct Ops {
  bool (*apart)(const Ctx&);
  void (*extrap)(Ctx&);
  void (*wave)(Ctx&);
  void (*dt)(Ctx&, double);
  void (*wave_dt)(Ctx&, double, bool);
  void (*residual)(Ctx&, bool);
  void (*rk)(Ctx&, int, double, double, bool, int, bool);
  void (*ensure)(Ctx&);
  void (*tune)(Ctx&);
  bool (*check)(Ctx&, const int*);
  void (*fit)(Ctx&);
  bool (*restrict_lds)(Ctx&, long long, long long, int, int, const double*, const double*, const double*, double*);
  bool (*prolong_lds)(Ctx&, int, int, const double*, const double*, const double*, bool);
};

template <int D, int P, class R>
static Ops ops_for() {
  using Rn = Runner<D, P, R>;
  return Ops{Rn::apart, Rn::extrap, Rn::wave, Rn::dt, Rn::wave_dt, Rn::residual, Rn::rk, Rn::ensure, Rn::tune, Rn::check, Rn::fit, Rn::restrict_lds, Rn::prolong_lds};
}

// The kernels of one dimension, precision and range of orders.  This file is
// compiled once for each (FHIP_FAMILY = 0 to 5, side by side: one after the
// other they take minutes) and once without for everything else.
Ops ops_2d_f64(int P), ops_2d_f32(int P), ops_3d_f64_low(int P), ops_3d_f64_high(int P), ops_3d_f32_low(int P),
    ops_3d_f32_high(int P);
#ifdef FHIP_FAMILY
template <int D, int P0, int P, class R>
static Ops ops_range(int p) {
  if constexpr (P > P0) {
    if (p < P) return ops_range<D, P0, P - 1, R>(p);
  }
  return ops_for<D, P, R>();
}
#if FHIP_FAMILY == 0
Ops ops_2d_f64(int P) { return ops_range<2, 0, 5, double>(P); }
#elif FHIP_FAMILY == 1
Ops ops_2d_f32(int P) { return ops_range<2, 0, 5, float>(P); }
#elif FHIP_FAMILY == 2
Ops ops_3d_f64_low(int P) { return ops_range<3, 0, 2, double>(P); }
#elif FHIP_FAMILY == 3
Ops ops_3d_f64_high(int P) { return ops_range<3, 3, 5, double>(P); }
#elif FHIP_FAMILY == 4
Ops ops_3d_f32_low(int P) { return ops_range<3, 0, 2, float>(P); }
#else
Ops ops_3d_f32_high(int P) { return ops_range<3, 3, 5, float>(P); }
#endif
#else

static Ops get_ops(const Ctx& c, bool mixed) {
  const int P = c.z.P;
  if (c.z.D == 2) return mixed ? ops_2d_f32(P) : ops_2d_f64(P);
  if (P < 3) return mixed ? ops_3d_f32_low(P) : ops_3d_f64_low(P);
  return mixed ? ops_3d_f32_high(P) : ops_3d_f64_high(P);
}

// Tuned block sizes, shared by the contexts of one process: keyed by (nDims, order,
// tune_form, viscous, log2 of the element count) and by what else decides which
// kernels run: the form of the stage kernel (inviscid runs; it changes within one
// log2 of the element count), operators from factors or tables.  The BF16 kernels
// are held to 3 waves per SIMD, under which a CU takes one block of 512 threads and
// no two: on Taylor-Green 48^3 512 threads are the mixed path's best size or close
// to it, and the BF16 forms' worst but ragged ones (stage 567 us, 410 with 128;
// Navier-Stokes volume 703 us, 505).
static std::mutex g_tune_mu;
static std::map<std::array<int, 7>, std::array<int, 5>> g_tuned;

void fused_autotune(Ctx& c, bool mixed, int* out) {
  FusedState& st = fs(c);
  Ops o = get_ops(c, mixed);
  const int m = tune_form(c, mixed);
  int lg = 0;
  for (long long e = c.z.E; e > 1; e >>= 1) lg++;
  const bool visc = c.prm.viscous != 0;
  const std::array<int, 7> key{c.z.D, c.z.P, m, visc, lg, !visc && o.apart(c), st.tb.w1 != nullptr};
  bool hit = false;
  {
    std::lock_guard<std::mutex> g(g_tune_mu);
    auto it = g_tuned.find(key);
    if (it != g_tuned.end()) {
      std::copy(it->second.begin(), it->second.end(), st.nt[m]);
      hit = true;
    }
  }
  if (!hit) {
    c.drop_graphs();
    fused_begin(c, mixed, false);  // reads U and the wave speeds; both are left as they were
    o.tune(c);
    std::array<int, 5> v;
    std::copy(st.nt[m], st.nt[m] + 5, v.begin());
    std::lock_guard<std::mutex> g(g_tune_mu);
    g_tuned[key] = v;
  }
  c.drop_graphs();
  if (out) std::copy(st.nt[m], st.nt[m] + 5, out);
}

void fused_set_blocks(Ctx& c, bool mixed, const int* nt) {
  Ops o = get_ops(c, mixed);
  if (!o.check(c, nt)) throw std::invalid_argument("block size not valid for this kernel and order");
  c.drop_graphs();
  std::copy(nt, nt + 5, fs(c).nt[tune_form(c, mixed)]);
}

void fused_get_blocks(Ctx& c, bool mixed, int* out) {
  get_ops(c, mixed).fit(c);
  const int* nt = fs(c).nt[tune_form(c, mixed)];
  std::copy(nt, nt + 5, out);
}

// What a call on the fused paths starts from, element-major.
static void add_begin(Ctx& c, bool mixed, bool src, Layouts& lay) {
  FusedState& st = fs(c);
  st.read_stage = st.flipped = false;
  const Sizes& z = c.z;
  get_ops(c, mixed).ensure(c);
  long long nS = (long long)z.E * z.N * z.S;
  lay.to_em(z.S, z.E, z.N, c.U, st.Ue);
  st.use_src = src;
  if (src) {
    if (!c.src) throw std::invalid_argument("no P-multigrid source term on this context");
    if (!st.srce) {
      c.drop_graphs();
      FCHK(hipMalloc(&st.srce, nS * sizeof(double)));
      poison_fill(st.srce, nS * sizeof(double));
    }
    lay.to_em(z.S, z.E, z.N, c.src, st.srce);
  }
  lay.to_em(z.F, z.E, 1, c.waveSp, st.waveSpe);
}

void fused_begin(Ctx& c, bool mixed, bool src) {
  Layouts lay(c.stream);
  add_begin(c, mixed, src, lay);
  lay.go();
  get_ops(c, mixed).extrap(c);
}

// P-multigrid cycle with every level kept element-major (the transfers above;
// a level's FlurryPP-layout arrays are written back by the caller at the end).
static int opgemm_chunk(int k) { return k <= 16 ? 16 : (k <= 32 ? 32 : 64); }

void fused_em_prepare(Ctx& c, bool mixed) {
  FusedState& st = fs(c);
  st.read_stage = st.flipped = false;
  get_ops(c, mixed).ensure(c);
  if (!st.srce) {
    c.drop_graphs();
    FCHK(hipMalloc(&st.srce, (size_t)c.z.E * c.z.N * c.z.S * sizeof(double)));
    poison_fill(st.srce, (size_t)c.z.E * c.z.N * c.z.S * sizeof(double));
  }
}

// The start of a cycle: fused_begin of the fine levels, and the coarse levels'
// wave speeds, of which the stage kernel rewrites only the entries of left and
// boundary flux points (the reference's calcWaveSp stores into the left element)
// and the time steps sum all.  All on one stream.
void fused_em_begin(Ctx* const* coarse, int nc, Ctx* const* fine, int nf, bool mixed) {
  Layouts lay(fine[0]->stream);
  for (int i = 0; i < nc; i++) {
    const Ctx& c = *coarse[i];
    lay.to_em(c.z.F, c.z.E, 1, c.waveSp, fs(*coarse[i]).waveSpe);
  }
  for (int i = 0; i < nf; i++) add_begin(*fine[i], mixed, false, lay);
  lay.go();
  for (int i = 0; i < nf; i++) get_ops(*fine[i], mixed).extrap(*fine[i]);
}

void fused_em_residual(Ctx& c, bool mixed, int how) {
  Ops o = get_ops(c, mixed);
  fs(c).use_src = false;
  o.residual(c, true);
  o.rk(c, how == 1 ? 7 : (how == 2 ? 8 : 5), 0., 0., true, 0, false);
}

// Whether a level's first smoothing step can take the residual that its source
// needs from its own first stage, which forms the same one: inviscid 2-D runs of
// several stages, where a time step that needs the wave speeds of that residual
// is formed in the stage too.  One launch of 11 per level on the way down:
// update and cycle of the P4 channel 67x29 630 -> 611 us.  (Instances of their own:
// as a switch in the stage kernel it cost every stage 0.5 of 7.2 us.)
bool fused_em_source_in_step(const Ctx& c) {
  return !c.prm.viscous && c.z.nRK > 1 && c.z.D == 2 && (c.prm.dt_type == 0 || c.prm.dt_type == 2);
}

void fused_em_set_src(Ctx& c, bool on) { fs(c).use_src = on; }

double* fused_em_array(Ctx& c, int which) {
  FusedState& st = fs(c);
  return which == 0 ? st.Ue : (which == 1 ? st.divF0e : st.srce);
}

// The solver's dt of a call whose steps formed the elements' in their stages: their
// minimum (solver::calcDt, src/solver.cpp:447-468).  Merged meshes have none.
static void add_dt(Ctx& c, Layouts& lay) {
  FusedState& st = fs(c);
  if (folds_dt(c) && st.nMesh == 1) lay.least(c.z.E, c.eleDt, st.dtAcc, st.dtTicket, c.d_dt);
}

static void add_end(Ctx& c, Layouts& lay) {
  FusedState& st = fs(c);
  st.use_src = false;
  const Sizes& z = c.z;
  lay.from_em(z.S, z.E, z.N, st.Ue, c.U);
  lay.from_em(z.S, z.E, z.N, st.divF0e, c.divF);
  lay.from_em(z.F, z.E, 1, st.waveSpe, c.waveSp);
}

// The end of a cycle on the element-major levels: U of the coarse levels (stepped:
// and their dt), U, divF_spts[0] and wave speeds of the fine ones, which took no step.
void fused_em_end(Ctx* const* coarse, int nc, Ctx* const* fine, int nf, bool stepped) {
  Layouts lay(fine[0]->stream);
  for (int i = 0; i < nc; i++) {
    Ctx& c = *coarse[i];
    fs(c).use_src = false;
    lay.from_em(c.z.S, c.z.E, c.z.N, fs(c).Ue, c.U);
    if (stepped) add_dt(c, lay);
  }
  for (int i = 0; i < nf; i++) add_end(*fine[i], lay);
  lay.go();
}

// Both leave U at the level's flux points current (prolongation: if extrap).
// Restriction and extrapolation, prolongation and extrapolation in one launch
// each, and a level's launches with them: update and cycle of the P4 channel
// 67x29 652 -> 630 us.
void pmg_restrict_em(Ctx& c, bool mixed, long long e0, long long ne, int Sf, const double* R, const double* Uf,
                     const double* divFf, double* solc) {
  FusedState& st = fs(c);
  if (e0 < 0 || ne < 0 || e0 + ne > c.z.E) throw std::invalid_argument("restriction rows out of range");
  if (ne == 0) return;
  const Ops o = get_ops(c, mixed);
  {
    Launch L(c, "pmg_restrict");
    if (o.restrict_lds(c, e0, ne, Sf, opgemm_chunk(Sf), R, Uf, divFf, solc)) return;
    const long long rows = ne * c.z.N, off = e0 * c.z.N * c.z.S;  // the first coarse element's rows
    hipLaunchKernelGGL(k_restrict_em, dim3(nblk(rows * c.z.S, 256)), dim3(256), 0, c.stream, rows, c.z.S, Sf,
                       opgemm_chunk(Sf), R, Uf, divFf, st.Ue + off, st.srce + off, solc + off);
    FCHK(hipGetLastError());
  }
  o.extrap(c);
}

void pmg_prolong_em(Ctx& up, bool mixed, int Sc, const double* Pm, const double* Uc, const double* solc, bool extrap) {
  FusedState& st = fs(up);
  const Ops o = get_ops(up, mixed);
  {
    Launch L(up, "pmg_prolong");
    if (o.prolong_lds(up, Sc, opgemm_chunk(Sc), Pm, Uc, solc, extrap)) return;
    const long long rows = (long long)up.z.E * up.z.N;
    hipLaunchKernelGGL(k_prolong_em, dim3(nblk(rows * up.z.S, 256)), dim3(256), 0, up.stream, rows, up.z.S, Sc,
                       opgemm_chunk(Sc), Pm, Uc, solc, st.Ue);
    FCHK(hipGetLastError());
  }
  if (extrap) o.extrap(up);
}

void fused_end(Ctx& c) {
  Layouts lay(c.stream);
  add_end(c, lay);
  add_dt(c, lay);
  lay.go();
}

// calcResidual(0) at the current state (src/solver.cpp:366-445) on a fused
// path: divF_spts[0] and the face wave speeds in FlurryPP's layouts.
void fused_residual(Ctx& c, bool mixed) {
  FusedState& st = fs(c);
  const Sizes& z = c.z;
  Ops o = get_ops(c, mixed);
  fused_begin(c, mixed, false);
  o.residual(c, true);
  o.rk(c, 5, 0., 0., true, 0, false);
  Layouts lay(c.stream);
  lay.from_em(z.S, z.E, z.N, st.divF0e, c.divF);
  lay.from_em(z.F, z.E, 1, st.waveSpe, c.waveSp);
  lay.go();
}

// One iteration of solver::update (src/solver.cpp:319-363) on a fused path.
void fused_rk_step(Ctx& c, bool refresh, bool mixed, bool keep, bool make_src) {
  Ops o = get_ops(c, mixed);
  FusedState& st = fs(c);
  const int nRK = c.z.nRK;
  const double* A = c.prm.rk_a;
  const double* B = c.prm.rk_b;
  const bool cfl = c.prm.dt_type != 0;
  const double cflfac = cfl ? c.prm.cfl * cfl_limit_f(c.z.P) : 0.;
  const bool jameson = c.prm.time_type >= 5;
  if (nRK == 1) {
    if (c.prm.viscous) o.residual(c, true);
    if (face_first(c)) {
      o.wave_dt(c, cflfac, refresh);
    } else if (cfl) {
      if (refresh) o.wave(c);
      o.dt(c, cflfac);
    }
    o.rk(c, jameson ? 4 : 3, A[1], B[0], keep, 0, false);
    return;
  }
  if (cfl) {
    if (refresh) o.wave(c);
    if (!folds_dt(c)) o.dt(c, cflfac);
  }
  for (int step = 0; step < nRK; step++) {
    st.read_stage = step > 0;
    o.residual(c, step == nRK - 1);
    // the Jameson form's first stage reads the state itself (the step's U0)
    int mode;
    if (jameson) mode = step == 0 ? 6 : 4;
    else mode = (step == 0) ? 0 : (step == nRK - 1 ? 2 : 1);
    o.rk(c, mode, A[step + 1], B[step], keep && step == 0, step, make_src && step == 0);
  }
  st.read_stage = false;
}

bool fused_flipped(const Ctx& c) { return ((const FusedState*)c.fused)->flipped; }
void fused_set_flipped(Ctx& c, bool flipped) { fs(c).flipped = flipped; }
bool fused_step_flips(const Ctx& c) { return !c.prm.viscous && (c.z.nRK & 1) && !face_first(c); }

#endif  // FHIP_FAMILY

}  // namespace fhip
