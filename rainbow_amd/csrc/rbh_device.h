// Device-side helpers for the rigid-body contact step: small vector and
// quaternion algebra, trilinear SDF lookups, proximal operators.
//
// Every routine is templated on the arithmetic type R (float for the product
// path, double for the FP64 parity build of the same kernels).  Expression
// order follows the reference formulas cited at each function, so the FP64
// instantiation reproduces the reference arithmetic up to FMA contraction.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace rbh {

template <typename R> struct alignas(4 * sizeof(R)) V4 { R x, y, z, w; };
template <typename R> struct V3 { R x, y, z; };

template <typename R> __device__ __forceinline__ V3<R> v3(R x, R y, R z) { return V3<R>{x, y, z}; }
template <typename R> __device__ __forceinline__ V3<R> xyz(const V4<R>& a) { return V3<R>{a.x, a.y, a.z}; }
template <typename R> __device__ __forceinline__ V3<R> operator+(V3<R> a, V3<R> b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
template <typename R> __device__ __forceinline__ V3<R> operator-(V3<R> a, V3<R> b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
template <typename R> __device__ __forceinline__ V3<R> operator*(R s, V3<R> a) { return {s * a.x, s * a.y, s * a.z}; }
template <typename R> __device__ __forceinline__ V3<R> operator-(V3<R> a) { return {-a.x, -a.y, -a.z}; }
template <typename R> __device__ __forceinline__ R dot(V3<R> a, V3<R> b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
template <typename R> __device__ __forceinline__ V3<R> cross(V3<R> a, V3<R> b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
template <typename R> __device__ __forceinline__ R norm(V3<R> a) { return sqrt(a.x * a.x + a.y * a.y + a.z * a.z); }

// ---------------------------------------------------------------- quaternions
// q = (s, x, y, z) stored in V4 as (x=s, y=qx, z=qy, w=qz).
template <typename R> struct Quat { R s, x, y, z; };

template <typename R> __device__ __forceinline__ Quat<R> quat(const V4<R>& a) { return Quat<R>{a.x, a.y, a.z, a.w}; }
template <typename R> __device__ __forceinline__ Quat<R> conj(Quat<R> q) { return Quat<R>{q.s, -q.x, -q.y, -q.z}; }

// quaternion.py:186-193 -- [a b - A.B, a B + b A + A x B]
template <typename R> __device__ __forceinline__ Quat<R> qprod(Quat<R> a, Quat<R> b) {
  R s = a.s * b.s - (a.x * b.x + a.y * b.y + a.z * b.z);
  R x = a.s * b.x + a.x * b.s + (a.y * b.z - a.z * b.y);
  R y = a.s * b.y + a.y * b.s + (a.z * b.x - a.x * b.z);
  R z = a.s * b.z + a.z * b.s + (a.x * b.y - a.y * b.x);
  return Quat<R>{s, x, y, z};
}

// quaternion.py:196-198 -- (q (0, r) q*)[1:]
template <typename R> __device__ __forceinline__ V3<R> qrotate(Quat<R> q, V3<R> r) {
  Quat<R> t = qprod(qprod(q, Quat<R>{R(0), r.x, r.y, r.z}), conj(q));
  return V3<R>{t.x, t.y, t.z};
}

// quaternion.py:201-250 -- rotate_array: prod_array(prod_array(q, (0,V)), conj(q))
template <typename R> __device__ __forceinline__ V3<R> qrotate_array(Quat<R> a, V3<R> v) {
  // inner = a (x) (0, v), written as prod_array(Qa, Qb) with Qb = (0, v)
  R i0 = a.s * R(0) - a.x * v.x - a.y * v.y - a.z * v.z;
  R i1 = a.s * v.x + a.x * R(0) + a.y * v.z - a.z * v.y;
  R i2 = a.s * v.y - a.x * v.z + a.y * R(0) + a.z * v.x;
  R i3 = a.s * v.z + a.x * v.y - a.y * v.x + a.z * R(0);
  Quat<R> b = conj(a);
  // outer = inner (x) b, prod_array(Qa_array, Qb)
  R o1 = i0 * b.x + i1 * b.s + i2 * b.z - i3 * b.y;
  R o2 = i0 * b.y - i1 * b.z + i2 * b.s + i3 * b.x;
  R o3 = i0 * b.z + i1 * b.y - i2 * b.x + i3 * b.s;
  return V3<R>{o1, o2, o3};
}

// quaternion.py:76-80
template <typename R> __device__ __forceinline__ Quat<R> qunit(Quat<R> q) {
  R l = sqrt(q.s * q.s + q.x * q.x + q.y * q.y + q.z * q.z);
  if (l > R(0)) return Quat<R>{q.s / l, q.x / l, q.y / l, q.z / l};
  return Quat<R>{R(1), R(0), R(0), R(0)};
}

// quaternion.py:108-129 (normalises first). Row-major 3x3.
template <typename R> __device__ __forceinline__ void qmatrix(Quat<R> Q, R M[9]) {
  Quat<R> q = qunit(Q);
  R s = q.s, x = q.x, y = q.y, z = q.z;
  M[0] = R(1) - R(2) * (y * y + z * z);
  M[4] = R(1) - R(2) * (x * x + z * z);
  M[8] = R(1) - R(2) * (y * y + x * x);
  M[3] = R(2) * (x * y + s * z);
  M[1] = R(2) * (x * y - s * z);
  M[6] = R(2) * (-s * y + x * z);
  M[2] = R(2) * (s * y + x * z);
  M[7] = R(2) * (z * y + s * x);
  M[5] = R(2) * (z * y - s * x);
}

// mass.py:395-452: W = R diag(B) R^T, packed symmetric (xx, yy, zz, xy, xz, yz).
template <typename R> __device__ __forceinline__ void rot_diag_rt(const R M[9], R b0, R b1, R b2, R W[6]) {
  W[0] = M[0] * M[0] * b0 + M[1] * M[1] * b1 + M[2] * M[2] * b2;
  W[1] = M[3] * M[3] * b0 + M[4] * M[4] * b1 + M[5] * M[5] * b2;
  W[2] = M[6] * M[6] * b0 + M[7] * M[7] * b1 + M[8] * M[8] * b2;
  W[3] = M[3] * M[0] * b0 + M[4] * M[1] * b1 + M[5] * M[2] * b2;
  W[4] = M[6] * M[0] * b0 + M[7] * M[1] * b1 + M[8] * M[2] * b2;
  W[5] = M[3] * M[6] * b0 + M[4] * M[7] * b1 + M[5] * M[8] * b2;
}

template <typename R> __device__ __forceinline__ V3<R> sym_mul(const R W[6], V3<R> a) {
  return V3<R>{W[0] * a.x + W[3] * a.y + W[4] * a.z,
               W[3] * a.x + W[1] * a.y + W[5] * a.z,
               W[4] * a.x + W[5] * a.y + W[2] * a.z};
}

// c + a * b for the contact sweep: one fused multiply-add in FP32; in FP64
// the product and the sum are rounded one by one, as the FP64 oracle does
template <typename R> __device__ __forceinline__ R madd(R a, R b, R c) {
  if constexpr (sizeof(R) == 4) return __builtin_fmaf(a, b, c);
  else return c + a * b;
}

// sym_mul with madd: the same sums in the same order
template <typename R> __device__ __forceinline__ V3<R> sym_madd(const R W[6], V3<R> a) {
  return V3<R>{madd(W[4], a.z, madd(W[3], a.y, W[0] * a.x)),
               madd(W[5], a.z, madd(W[1], a.y, W[3] * a.x)),
               madd(W[2], a.z, madd(W[5], a.y, W[4] * a.x))};
}

// vector3.py:75-113: (t, b, n) with t guessed from the axis of smallest |n_i|
// (the later axis wins ties) and b = unit(n x t), t = b x n.
template <typename R> __device__ __forceinline__ void orthonormal_frame(V3<R> nin, V3<R>& t, V3<R>& b, V3<R>& n) {
  R l = norm(nin);
  n = V3<R>{nin.x / l, nin.y / l, nin.z / l};
  R ax = fabs(n.x), ay = fabs(n.y), az = fabs(n.z);
  V3<R> g = {R(1), R(0), R(0)};
  if (ay <= ax && ay <= az) g = V3<R>{R(0), R(1), R(0)};
  if (az <= ax && az <= ay) g = V3<R>{R(0), R(0), R(1)};
  // the first test (ax smallest) only matters when neither later test fires
  V3<R> bb = cross(n, g);
  R lb = norm(bb);
  b = V3<R>{bb.x / lb, bb.y / lb, bb.z / lb};
  t = cross(b, n);
}

// ---------------------------------------------------------------- SDF grids
template <typename R> struct GridView {
  const R* val;
  const R* cells;   // cell-major copy: cell (i, j, k) holds its 8 corners in the order of load_cell
  int I, J, K;
  R mn[3], mx[3], h[3];
};

// grid3.py:107-123 -- floor((p - min) / h) clipped to [0, dim - 2]
template <typename R> __device__ __forceinline__ void cell_idx(const GridView<R>& g, V3<R> p, int& i, int& j, int& k) {
  R fi = floor((p.x - g.mn[0]) / g.h[0]);
  R fj = floor((p.y - g.mn[1]) / g.h[1]);
  R fk = floor((p.z - g.mn[2]) / g.h[2]);
  // clamp in floating point first so huge values cannot overflow the int cast
  fi = fmin(fmax(fi, R(0)), R(g.I - 2));
  fj = fmin(fmax(fj, R(0)), R(g.J - 2));
  fk = fmin(fmax(fk, R(0)), R(g.K - 2));
  i = (int)fi; j = (int)fj; k = (int)fk;
  if (!(i >= 0)) i = 0;   // NaN input
  if (!(j >= 0)) j = 0;
  if (!(k >= 0)) k = 0;
}

template <typename R> struct Cell { R d000, d001, d010, d011, d100, d101, d110, d111; };

// The 8 corner values of cell (i, j, k), read as two vec4 from the
// cell-major copy of the grid (k_sdf_cells) instead of 8 scattered values:
// (i,j,k), (i+1,j,k), (i,j+1,k), (i+1,j+1,k), then the same at k+1.
template <typename R> __device__ __forceinline__ Cell<R> load_cell(const GridView<R>& g, int i, int j, int k) {
  const V4<R>* p = reinterpret_cast<const V4<R>*>(g.cells) +
                   2 * ((size_t)i + (size_t)(g.I - 1) * ((size_t)j + (size_t)(g.J - 1) * (size_t)k));
  const V4<R> a = p[0], e = p[1];
  Cell<R> c;
  c.d000 = a.x; c.d100 = a.y; c.d010 = a.z; c.d110 = a.w;
  c.d001 = e.x; c.d101 = e.y; c.d011 = e.z; c.d111 = e.w;
  return c;
}

// cell-major copy of one grid (values v, I x J x K nodes, index i + I (j + J k))
template <typename R> __global__ void k_sdf_cells(const R* __restrict__ v, int I, int J, int K, R* __restrict__ out) {
  const long long nc = (long long)(I - 1) * (J - 1) * (K - 1);
  for (long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x; c < nc; c += (long long)gridDim.x * blockDim.x) {
    const int i = (int)(c % (I - 1));
    const long long r = c / (I - 1);
    const int j = (int)(r % (J - 1)), k = (int)(r / (J - 1));
    const long long b = i + (long long)I * (j + (long long)J * k), dj = I, dk = (long long)I * J;
    R* o = out + 8 * c;
    o[0] = v[b]; o[1] = v[b + 1]; o[2] = v[b + dj]; o[3] = v[b + 1 + dj];
    o[4] = v[b + dk]; o[5] = v[b + 1 + dk]; o[6] = v[b + dj + dk]; o[7] = v[b + 1 + dj + dk];
  }
}

// grid3.py:126-177
template <typename R> __device__ __forceinline__ R grid_value(const GridView<R>& g, V3<R> p) {
  int i, j, k;
  cell_idx(g, p, i, j, k);
  Cell<R> c = load_cell(g, i, j, k);
  R s = (p.x - ((R(i) * g.h[0]) + g.mn[0])) / g.h[0];
  R t = (p.y - ((R(j) * g.h[1]) + g.mn[1])) / g.h[1];
  R u = (p.z - ((R(k) * g.h[2]) + g.mn[2])) / g.h[2];
  R x00 = (c.d100 - c.d000) * s + c.d000;
  R x01 = (c.d101 - c.d001) * s + c.d001;
  R x10 = (c.d110 - c.d010) * s + c.d010;
  R x11 = (c.d111 - c.d011) * s + c.d011;
  R y0 = (x10 - x00) * t + x00;
  R y1 = (x11 - x01) * t + x01;
  return (y1 - y0) * u + y0;
}

// grid3.py:180-254 -- local coordinates divided by min_coord (grid3.py:209-211)
template <typename R> __device__ __forceinline__ V3<R> grid_gradient(const GridView<R>& g, V3<R> p) {
  int i, j, k;
  cell_idx(g, p, i, j, k);
  Cell<R> c = load_cell(g, i, j, k);
  R s = (p.x - (R(i) * g.h[0] + g.mn[0])) / g.mn[0];
  R t = (p.y - (R(j) * g.h[1] + g.mn[1])) / g.mn[1];
  R u = (p.z - (R(k) * g.h[2] + g.mn[2])) / g.mn[2];
  R x00 = (c.d100 - c.d000) * s + c.d000;
  R x01 = (c.d101 - c.d001) * s + c.d001;
  R x10 = (c.d110 - c.d010) * s + c.d010;
  R x11 = (c.d111 - c.d011) * s + c.d011;
  R y0 = (x10 - x00) * t + x00;
  R y1 = (x11 - x01) * t + x01;
  R dx00 = c.d100 - c.d000, dx01 = c.d101 - c.d001, dx10 = c.d110 - c.d010, dx11 = c.d111 - c.d011;
  R dy0_ds = (dx10 - dx00) * t + dx00;
  R dy1_ds = (dx11 - dx01) * t + dx01;
  R dy0_dt = x10 - x00;
  R dy1_dt = x11 - x01;
  R dp_ds = (dy1_ds - dy0_ds) * u + dy0_ds;
  R dp_dt = (dy1_dt - dy0_dt) * u + dy0_dt;
  R dp_du = y1 - y0;
  return V3<R>{dp_ds * (R(1) / g.h[0]), dp_dt * (R(1) / g.h[1]), dp_du * (R(1) / g.h[2])};
}

// grid3.py:275-300 (strict comparisons; equality counts as inside)
template <typename R> __device__ __forceinline__ bool grid_inside(const GridView<R>& g, V3<R> p, R boundary) {
  if (p.x > (g.mx[0] - boundary) || p.y > (g.mx[1] - boundary) || p.z > (g.mx[2] - boundary)) return false;
  if (p.x < (g.mn[0] + boundary) || p.y < (g.mn[1] + boundary) || p.z < (g.mn[2] + boundary)) return false;
  return true;
}

// ---------------------------------------------------------------- prox ops
// prox_operators.py:14-34
template <typename R> __device__ __forceinline__ void prox_sphere(R zs, R zt, R zr, R mu, R xn, R& os, R& ot, R& orr) {
  if (xn <= R(0)) { os = ot = orr = R(0); return; }
  R radius = mu * xn;
  R sq = zs * zs + zt * zt + zr * zr;
  if (sq <= radius * radius) { os = zs; ot = zt; orr = zr; return; }
  // FP32: one hardware reciprocal square root (1 ulp) in place of a correctly
  // rounded sqrt and divide; FP64 keeps radius / sqrt(sq) as the reference has it
  R scale;
  if constexpr (sizeof(R) == 4) scale = radius * __builtin_amdgcn_rsqf(sq);
  else scale = radius / sqrt(sq);
  os = zs * scale; ot = zt * scale; orr = zr * scale;
}

// prox_sphere for a lane that holds one of the three values: z projected, sq
// the sum of the three squares (added in prox_sphere's order).  The same
// result; in FP32 by selects (a branch costs a lone wavefront more than the
// arithmetic), in FP64 past a branch, since its square root and division are
// long sequences.
template <typename R> __device__ __forceinline__ R prox_sphere_row(R z, R sq, R mu, R xn) {
  const R radius = mu * xn;
  if constexpr (sizeof(R) == 4) {
    const R f = sq <= radius * radius ? R(1) : radius * __builtin_amdgcn_rsqf(sq);
    const R v = z * f;
    return xn <= R(0) ? R(0) : v;
  } else {
    if (xn <= R(0)) return R(0);
    if (sq <= radius * radius) return z;
    return z * (radius / sqrt(sq));
  }
}

// First term of a velocity-change sum: FP64 starts from 0 as the reference's
// sparse products do (0 + p only differs from p for p = -0); FP32 starts from p.
template <typename R> __device__ __forceinline__ R sum_first(R p) {
  if constexpr (sizeof(R) == 8) return R(0) + p;
  else return p;
}

// proximal_contact/proximal_operators.py:42-139, evaluated in FP64.
struct EllipsoidParams { double tol, expansion; int max_it; };

__device__ __forceinline__ double ell_g(double saa, double sbb, double scc, double sxx, double syy, double szz, double t) {
  return (saa * sxx) / ((saa + t) * (saa + t)) + (sbb * syy) / ((sbb + t) * (sbb + t)) +
         (scc * szz) / ((scc + t) * (scc + t)) - 1.0;
}

// The bisection asks ell_g = n1 / d1 + n2 / d2 + n3 / d3 - 1 two questions only,
// g > 0 and |g| < tol, about 30 times, each with three FP64 divisions in a
// serial chain.  Two shortcuts give the same answers, so the same bits:
//  * ell_side, over the common denominator: both are questions about N - D,
//    with N = n1 d2 d3 + n2 d1 d3 + n3 d1 d2 and D = d1 d2 d3.  Rounding here
//    and in ell_g together stays below 3e-15 (N + D); an answer nearer to its
//    threshold than 1e-14 (N + D), or with a D so small that products
//    underflowed, or one that is not a number, is not `sure`, and the caller
//    then evaluates ell_g;
//  * ell_root: g falls and is convex, so once its root is known the answer at
//    a midpoint away from it is a comparison.
// A lane's bisection took about 9,000 cycles; it is now ~850 before the root,
// ~1,500 for the root and ~90 a level.  27 boxes in FP64, 73 contacts, 50
// sweeps, two solves and two post-stabilisations: 4550 -> 3120 us.
struct EllSide {
  bool pos, near, sure;   // g > 0; |g| < tol
};
__device__ __forceinline__ EllSide ell_side(double n1, double n2, double n3, double d1, double d2, double d3, double tol) {
  const double d23 = d2 * d3;
  const double N = __builtin_fma(n3 * d1, d2, __builtin_fma(n2 * d1, d3, n1 * d23)), D = d1 * d23;
  const double diff = N - D, mag = fabs(diff), tolD = tol * D;
  return EllSide{diff > 0.0, mag < tolD, D > 1e-250 && fmin(mag, fabs(mag - tolD)) > 1e-14 * (N + D)};
}
__device__ __forceinline__ EllSide ell_side_at(double n1, double n2, double n3, double saa, double sbb, double scc,
                                               double sxx, double syy, double szz, double t, double tol) {
  const double a = saa + t, b = sbb + t, c = scc + t;
  EllSide s = ell_side(n1, n2, n3, a * a, b * b, c * c, tol);
  if (!s.sure) {
    const double g = ell_g(saa, sbb, scc, sxx, syy, szz, t);
    s.pos = g > 0.0;
    s.near = fabs(g) < tol;
  }
  return s;
}

// 1 / x to 3e-15 relative: the estimate is good to 2^-24 (largest seen 2^-24.4,
// over 6.7e7 arguments), a Newton step squares that and rounds (2^-48.7)
__device__ __forceinline__ double ell_rcp(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  return __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
}

// Below lo, g > 0 and |g| >= tol; above hi, g <= 0 and |g| >= tol; between
// them (everywhere, if the root was not found) g has to be looked at.
//
// The root by Newton steps on 1 / sqrt(sum) - 1, which is nearly linear in t
// and converges from t = 0 without overshooting, in FP32, and one in FP64.
// With g(r) and the slope m = -g'(r) known, convexity puts the true root
// within 2 |g(r)| / m + rounding of r (g(r) is a sum near 1 of three terms, each
// good to 1e-14).  For t below it g(t) >= m (root - t); for t above it |g| is at
// least what the slope gathers over the first hundredth of (smallest axis
// squared + r), on which it stays above 0.97 m: hi has to lie within that reach.
// (It does not where an axis is thin, g(r) is far above the tolerance and the
// slope is gone before |g| has grown to it.)
struct EllRoot { double lo, hi; };
__device__ __forceinline__ EllRoot ell_root(double n1, double n2, double n3, double saa, double sbb, double scc, double tol) {
  const float f1 = (float)n1, f2 = (float)n2, f3 = (float)n3, e1 = (float)saa, e2 = (float)sbb, e3 = (float)scc;
  float t = 1e-12f;   // (an axis of length zero has no weight, but 0 / 0 at t = 0)
#pragma unroll 1
  for (int i = 0; i < 5; ++i) {
    const float r1 = __builtin_amdgcn_rcpf(e1 + t), r2 = __builtin_amdgcn_rcpf(e2 + t), r3 = __builtin_amdgcn_rcpf(e3 + t);
    const float a1 = f1 * r1 * r1, a2 = f2 * r2 * r2, a3 = f3 * r3 * r3;
    const float S = a1 + a2 + a3, P = a1 * r1 + a2 * r2 + a3 * r3;
    t += S * (__builtin_amdgcn_sqrtf(S) - 1.0f) * __builtin_amdgcn_rcpf(P);
  }
  double r = (double)t, g = 0.0, P = 0.0;
#pragma unroll 1
  for (int i = 0; i < 2; ++i) {
    const double r1 = ell_rcp(saa + r), r2 = ell_rcp(sbb + r), r3 = ell_rcp(scc + r);
    const double a1 = n1 * r1 * r1, a2 = n2 * r2 * r2, a3 = n3 * r3 * r3;
    g = a1 + a2 + a3 - 1.0;
    P = a1 * r1 + a2 * r2 + a3 * r3;
    if (i == 0) r += 0.5 * g * ell_rcp(P);
  }
  const double m = 2.0 * P, eps = fmax(tol, 0.0) + 1e-12;
  const double over = 1.01 * ell_rcp(m) * (2.0 * fabs(g) + 1e-13 + eps / 0.9);
  const double reach = 0.01 * (fmin(saa, fmin(sbb, scc)) + r);
  const bool ok = r > 0.0 && fabs(g) < 1e-8 && 0.9 * m * reach > eps && over > 0.0 && over <= reach && over < 1e300;
  return EllRoot{ok ? r - over : -INFINITY, ok ? r + over : INFINITY};
}

template <typename R>
__device__ __forceinline__ void prox_ellipsoid(R zs_, R zt_, R zr_, R mus_, R mut_, R mur_, R xn_, const EllipsoidParams& ep,
                                               R& os, R& ot, R& orr) {
  double zs = zs_, zt = zt_, zr = zr_, ms = mus_, mt = mut_, mr = mur_, xn = xn_;
  if (xn <= 0.0) { os = ot = orr = R(0); return; }
  if (ms == 0.0 && mt == 0.0 && mr == 0.0) { os = ot = orr = R(0); return; }
  if (ms == mt && ms == mr) { prox_sphere<R>(zs_, zt_, zr_, mus_, xn_, os, ot, orr); return; }
  double a = ms * xn, b = mt * xn, c = mr * xn;
  double m = fmax(fmax(fmax(1.0, a), fmax(b, c)), fmax(fmax(fabs(zs), fabs(zt)), fabs(zr)));
  double scale = 1.0 / m;
  double sa = scale * a, sb = scale * b, sc = scale * c, sx = scale * zs, sy = scale * zt, sz = scale * zr;
  double saa = sa * sa, sbb = sb * sb, scc = sc * sc, sxx = sx * sx, syy = sy * sy, szz = sz * sz;
  // inside the ellipsoid: sxx / saa + syy / sbb + szz / scc - 1 < tol
  const EllSide in = ell_side(sxx, syy, szz, saa, sbb, scc, ep.tol);
  const bool inside = in.sure && ep.tol >= 0.0 ? !in.pos || in.near : (sxx / saa) + (syy / sbb) + (szz / scc) - 1.0 < ep.tol;
  if (inside) { os = zs_; ot = zt_; orr = zr_; return; }
  const double n1 = saa * sxx, n2 = sbb * syy, n3 = scc * szz;
  double t0 = 0.0;
  double t1 = fmax(fmax(sa, sb), sc) * sqrt(sx * sx + sy * sy + sz * sz);
  bool out = ell_side_at(n1, n2, n3, saa, sbb, scc, sxx, syy, szz, t1, ep.tol).pos;
  for (int guard = 0; out && guard < 4096; ++guard) {
    t1 *= ep.expansion;
    out = ell_side_at(n1, n2, n3, saa, sbb, scc, sxx, syy, szz, t1, ep.tol).pos;
  }
  double tk = (t0 + t1) * 0.5;
  const EllRoot root = ell_root(n1, n2, n3, saa, sbb, scc, ep.tol);
  // eight levels at a time without a branch, each lane until its next midpoint
  // is too close to the root or its interval short enough
  int it = 0;
  for (bool go = true; it + 8 <= ep.max_it && __any(go);) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const bool pos = tk < root.lo, neg = tk > root.hi;
      go = go && (pos || neg) && !(fabs(t1 - t0) < ep.tol);
      t0 = go && pos ? tk : t0;
      t1 = go && neg ? tk : t1;
      tk = (t0 + t1) * 0.5;
      it += go ? 1 : 0;
    }
  }
  for (; it < ep.max_it; ++it) {
    if (fabs(t1 - t0) < ep.tol) break;
    const EllSide k = ell_side_at(n1, n2, n3, saa, sbb, scc, sxx, syy, szz, tk, ep.tol);
    if (k.near) break;
    if (k.pos) t0 = tk; else t1 = tk;
    tk = (t0 + t1) * 0.5;
  }
  tk /= scale * scale;
  os = R((a * a * zs) / (a * a + tk));
  ot = R((b * b * zt) / (b * b + tk));
  orr = R((c * c * zr) / (c * c + tk));
}

// out of line: anisotropic friction is the rare case, and inlining its
// bisection into every sweep loop only lengthens the isotropic path's code
template <typename R>
__device__ __attribute__((noinline)) V3<R> prox_ellipsoid_call(R zs, R zt, R zr, R ms, R mt, R mr, R xn, double tol,
                                                              double expansion, int max_it) {
  EllipsoidParams ep{tol, expansion, max_it};
  V3<R> o;
  prox_ellipsoid<R>(zs, zt, zr, ms, mt, mr, xn, ep, o.x, o.y, o.z);
  return o;
}

// ---------------------------------------------------------------- misc
__device__ __forceinline__ uint64_t mix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

__device__ __forceinline__ uint32_t color_draw(uint64_t seed, uint64_t step, uint64_t v, uint64_t rnd, uint32_t n) {
  uint64_t h = mix64(mix64(mix64(mix64(seed) ^ step) ^ v) ^ rnd);
  return (uint32_t)(((h >> 32) * (uint64_t)n) >> 32);
}

// Non-negative doubles order like their bit patterns: max via integer atomics.
__device__ __forceinline__ void atomic_max_nonneg(double* addr, double v) {
  atomicMax(reinterpret_cast<unsigned long long*>(addr), (unsigned long long)__double_as_longlong(v));
}

}  // namespace rbh
