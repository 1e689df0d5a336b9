// Signed-distance grid construction on the GPU (setup time).
//
// The reference builds shape SDFs with libigl's signed_distance
// (rainbow/geometry/grid3.py:320-339, called from api.py:234-241).  Here each
// thread owns one grid node: it computes the exact distance to every triangle
// (closest point by Voronoi-region tests, Ericson, "Real-Time Collision
// Detection" 5.1.5) and the generalized winding number (sum of signed solid
// angles, Van Oosterom & Strackee 1983); the sign is negative where the
// winding number exceeds 1/2.  Arithmetic is FP64 regardless of the step
// precision.  k_sdf does this for every node and triangle; the k_sdf_*
// pipeline below it gives the same values without most of that work.
#pragma once
#include <hip/hip_runtime.h>

namespace rbh {

constexpr int SDF_BLOCK = 256;
constexpr int SDF_TILE = 256;

// squared distance of p to the triangle t, region after region: the form for
// wavefronts of neighbouring nodes, which mostly agree on the region.
__device__ __forceinline__ double tri_sqdist(double px, double py, double pz, const double* t) {
  const double ax = t[0], ay = t[1], az = t[2], bx = t[3], by = t[4], bz = t[5], cx = t[6], cy = t[7], cz = t[8];
  double abx = bx - ax, aby = by - ay, abz = bz - az;
  double acx = cx - ax, acy = cy - ay, acz = cz - az;
  double apx = px - ax, apy = py - ay, apz = pz - az;
  double d1 = abx * apx + aby * apy + abz * apz;
  double d2 = acx * apx + acy * apy + acz * apz;
  double qx, qy, qz;
  if (d1 <= 0.0 && d2 <= 0.0) { qx = ax; qy = ay; qz = az; goto done; }
  {
    double bpx = px - bx, bpy = py - by, bpz = pz - bz;
    double d3 = abx * bpx + aby * bpy + abz * bpz;
    double d4 = acx * bpx + acy * bpy + acz * bpz;
    if (d3 >= 0.0 && d4 <= d3) { qx = bx; qy = by; qz = bz; goto done; }
    double vc = d1 * d4 - d3 * d2;
    if (vc <= 0.0 && d1 >= 0.0 && d3 <= 0.0) {
      double v = d1 / (d1 - d3);
      qx = ax + v * abx; qy = ay + v * aby; qz = az + v * abz; goto done;
    }
    double cpx = px - cx, cpy = py - cy, cpz = pz - cz;
    double d5 = abx * cpx + aby * cpy + abz * cpz;
    double d6 = acx * cpx + acy * cpy + acz * cpz;
    if (d6 >= 0.0 && d5 <= d6) { qx = cx; qy = cy; qz = cz; goto done; }
    double vb = d5 * d2 - d1 * d6;
    if (vb <= 0.0 && d2 >= 0.0 && d6 <= 0.0) {
      double w = d2 / (d2 - d6);
      qx = ax + w * acx; qy = ay + w * acy; qz = az + w * acz; goto done;
    }
    double va = d3 * d6 - d5 * d4;
    if (va <= 0.0 && (d4 - d3) >= 0.0 && (d5 - d6) >= 0.0) {
      double w = (d4 - d3) / ((d4 - d3) + (d5 - d6));
      qx = bx + w * (cx - bx); qy = by + w * (cy - by); qz = bz + w * (cz - bz); goto done;
    }
    double den = 1.0 / (va + vb + vc);
    double v = vb * den, w = vc * den;
    qx = ax + abx * v + acx * w; qy = ay + aby * v + acy * w; qz = az + abz * v + acz * w;
  }
done:
  double dx = px - qx, dy = py - qy, dz = pz - qz;
  return dx * dx + dy * dy + dz * dz;
}

// the same value by selects and one division: the closest point is a + e1 t1 +
// e2 t2 from a corner, an edge (t2 = 0) or the face, chosen in the order of the
// region tests.  For wavefronts whose lanes hold different triangles: a branch
// per region had them run through most of the regions, with a division in four;
// and for lone wavefronts, whose time is that of the chain of instructions.
// The coordinates have to be finite (an edge times zero is zero).
__device__ __forceinline__ double tri_sqdist_select(double px, double py, double pz, const double* t) {
  const double ax = t[0], ay = t[1], az = t[2], bx = t[3], by = t[4], bz = t[5], cx = t[6], cy = t[7], cz = t[8];
  const double abx = bx - ax, aby = by - ay, abz = bz - az;
  const double acx = cx - ax, acy = cy - ay, acz = cz - az;
  const double apx = px - ax, apy = py - ay, apz = pz - az;
  const double bpx = px - bx, bpy = py - by, bpz = pz - bz;
  const double cpx = px - cx, cpy = py - cy, cpz = pz - cz;
  const double d1 = abx * apx + aby * apy + abz * apz, d2 = acx * apx + acy * apy + acz * apz;
  const double d3 = abx * bpx + aby * bpy + abz * bpz, d4 = acx * bpx + acy * bpy + acz * bpz;
  const double d5 = abx * cpx + aby * cpy + abz * cpz, d6 = acx * cpx + acy * cpy + acz * cpz;
  const double vc = d1 * d4 - d3 * d2, vb = d5 * d2 - d1 * d6, va = d3 * d6 - d5 * d4;
  const double e = d4 - d3, f = d5 - d6;
  const bool in_a = d1 <= 0.0 && d2 <= 0.0;
  const bool in_b = !in_a && d3 >= 0.0 && d4 <= d3;
  const bool in_ab = !in_a && !in_b && vc <= 0.0 && d1 >= 0.0 && d3 <= 0.0;
  const bool past = in_a || in_b || in_ab;
  const bool in_c = !past && d6 >= 0.0 && d5 <= d6;
  const bool in_ac = !past && !in_c && vb <= 0.0 && d2 >= 0.0 && d6 <= 0.0;
  const bool in_bc = !past && !in_c && !in_ac && va <= 0.0 && e >= 0.0 && f >= 0.0;
  const bool corner = in_a || in_b || in_c, edge = in_ab || in_ac || in_bc;
  const double num = in_ab ? d1 : in_ac ? d2 : in_bc ? e : 1.0;
  const double den = in_ab ? d1 - d3 : in_ac ? d2 - d6 : in_bc ? e + f : (va + vb + vc);
  const double q = num / den;
  const double t1 = corner ? 0.0 : edge ? q : vb * q, t2 = corner || edge ? 0.0 : vc * q;
  const bool from_b = in_b || in_bc;
  const double ox = in_c ? cx : from_b ? bx : ax, oy = in_c ? cy : from_b ? by : ay, oz = in_c ? cz : from_b ? bz : az;
  const double ex = in_bc ? cx - bx : in_ac ? acx : abx, ey = in_bc ? cy - by : in_ac ? acy : aby,
               ez = in_bc ? cz - bz : in_ac ? acz : abz;
  const double dx = px - (ox + ex * t1 + acx * t2), dy = py - (oy + ey * t1 + acy * t2),
               dz = pz - (oz + ez * t1 + acz * t2);
  return dx * dx + dy * dy + dz * dz;
}

// tan of half the solid angle of triangle t seen from p, as (det, den)
__device__ __forceinline__ void solid_angle_parts(double px, double py, double pz, const double* t, double& det,
                                                  double& den) {
  double ax = t[0] - px, ay = t[1] - py, az = t[2] - pz;
  double bx = t[3] - px, by = t[4] - py, bz = t[5] - pz;
  double cx = t[6] - px, cy = t[7] - py, cz = t[8] - pz;
  double la = sqrt(ax * ax + ay * ay + az * az), lb = sqrt(bx * bx + by * by + bz * bz),
         lc = sqrt(cx * cx + cy * cy + cz * cz);
  det = ax * (by * cz - bz * cy) + ay * (bz * cx - bx * cz) + az * (bx * cy - by * cx);
  den = la * lb * lc + (ax * bx + ay * by + az * bz) * lc + (bx * cx + by * cy + bz * cz) * la +
        (cx * ax + cy * ay + cz * az) * lb;
}

__device__ __forceinline__ double solid_angle(double px, double py, double pz, const double* t) {
  double det, den;
  solid_angle_parts(px, py, pz, t, det, den);
  return 2.0 * atan2(det, den);
}

// The same sum of solid angles without an arctangent per triangle: the
// argument of the product of (den + i det), with the turns past pi counted.
// The half planes are told apart by sign bits, as atan2 does it: a node on a
// triangle has det = -0 and den < 0 there, an angle of -pi and not pi.
// The product is kept near 1 by an approximate reciprocal (its length does
// not matter).  Agrees with the sum of arctangents to rounding.
struct TurnSum {
  double re = 1.0, im = 0.0;
  int turns = 0;
  __device__ __forceinline__ void add(double det, double den) {
    if (det == 0.0 && den == 0.0) return;   // atan2(0, 0): no angle
    const bool up = !signbit(det), was = !signbit(im);
    const double r = re * den - im * det, i = re * det + im * den;
    const bool now = !signbit(i);
    if (up && was && !now) ++turns;
    if (!up && !was && now) --turns;
    const double s = __builtin_amdgcn_rcp(fabs(r) + fabs(i));
    re = r * s;
    im = i * s;
  }
  __device__ __forceinline__ double angle() const { return 2.0 * (atan2(im, re) + 6.28318530717958647692 * turns); }
};

// tri[9 t + 3 k + a] = V[3 T[3 t + k] + a]: the corners of each triangle in
// one record (triangle indices checked on the host)
__global__ void k_sdf_gather(const double* __restrict__ V, const int* __restrict__ T, int nt,
                             double* __restrict__ tri) {
  const long n = 9L * nt;
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    const long t = e / 9;
    const int r = (int)(e - 9 * t);
    tri[e] = V[3L * T[3 * t + r / 3] + r % 3];
  }
}

// tri: 9 doubles per triangle; out[i + I (j + J k)] = signed distance of node (i, j, k).
// SELECT: the closest point by selects.  Up to a wavefront per SIMD (65,536
// nodes) that is 2 to 5 % faster (126 triangles on 12^3 142 us, by branches 150;
// on 38^3 167, 170), beyond it the less work of the branches is (448 on 128^3
// 8.7 ms, by selects 10.1; 500 strewn ones 10.0, 11.0).
constexpr long SDF_SELECT_NODES = 65536;
template <bool SELECT>
__global__ void __launch_bounds__(SDF_BLOCK) k_sdf(const double* __restrict__ tri, int nt, int I, int J, int K,
                                                   double mnx, double mny, double mnz, double hx, double hy, double hz,
                                                   double* __restrict__ out) {
  __shared__ double st[SDF_TILE * 9];
  const long n = (long)I * J * K;
  const long node = (long)blockIdx.x * SDF_BLOCK + threadIdx.x;
  double px = 0, py = 0, pz = 0;
  if (node < n) {
    int i = (int)(node % I);
    int j = (int)((node / I) % J);
    int k = (int)(node / ((long)I * J));
    // grid3.py:88-105: min_coord + spacing * (i, j, k)
    px = mnx + hx * (double)i; py = mny + hy * (double)j; pz = mnz + hz * (double)k;
  }
  double best = INFINITY, wsum = 0.0;
  for (int t0 = 0; t0 < nt; t0 += SDF_TILE) {
    int cnt = min(SDF_TILE, nt - t0);
    for (int e = threadIdx.x; e < cnt * 9; e += SDF_BLOCK) st[e] = tri[(long)t0 * 9 + e];
    __syncthreads();
    if (node < n) {
      for (int e = 0; e < cnt; ++e) {
        const double* t = st + e * 9;
        best = fmin(best, SELECT ? tri_sqdist_select(px, py, pz, t) : tri_sqdist(px, py, pz, t));
        wsum += solid_angle(px, py, pz, t);
      }
    }
    __syncthreads();
  }
  if (node < n) {
    double wn = wsum / (4.0 * 3.14159265358979323846);
    double dist = sqrt(best);
    out[node] = fabs(wn) > 0.5 ? -dist : dist;
  }
}

// ---------------------------------------------------------------- pruned build
// The same values as k_sdf from a fraction of its work (64^3 nodes and 9,680
// triangles: 2.5e9 distances and solid angles, 23.1 ms):
//  * Distance: triangles are sorted into clusters of SDF_CL along a Morton
//    curve; a wavefront owns a small block of nodes and takes the exact
//    distance only to the clusters whose box may hold a nearer triangle, with
//    room for the rounding of those distances (SdfGrid::slack).  The nearest
//    triangle is always among them and its distance is computed by the same
//    expression, so the minimum is the same.
//  * Sign: away from the surface of a closed mesh the winding number is constant.
//    Two neighbouring nodes lie on the same side if either is farther from the
//    surface than from the other, rounding included; nodes are joined so into
//    trees, and the winding number is taken once per tree.  Nodes on the surface itself join
//    no other.  Closed: every edge (vertices welded by position) is used as
//    often in one direction as in the other; for any other (open) mesh every
//    node is a tree of its own.
constexpr int SDF_CL = 32;               // triangles per cluster
constexpr int SDF_CELLS = 4096;          // Morton cells the triangles are sorted by (16 per axis)

// A computed distance, or that of two neighbouring nodes, is good to a few units
// in the last place of the largest coordinate, however small it is itself: near
// the surface of a mesh 10^4 units from the origin, values within 3e-12 of it
// came out otherwise than the plain build's before the slack was given.
constexpr double SDF_SLACK = 256.0 * 2.220446049250313e-16;

struct SdfGrid {
  int I, J, K;
  double mn[3], h[3], mx[3];
  double slack;              // SDF_SLACK of the largest coordinate
  __device__ __forceinline__ double at(int a, int i) const { return mn[a] + h[a] * (double)i; }
};

struct SdfWork {
  const double* V; const int* T; int nv, nt;
  double* tri;               // 9 per triangle, in cluster order
  double* box;               // 6 per cluster: lower, upper corner
  int* cnt;                  // triangles per Morton cell, then the cell's first position (SDF_CELLS + 1)
  int2* pos;                 // per triangle: cell, rank in it
  int* vhash; int vmask;     // welded vertices: table of vertex indices (-1: free)
  int* rep;                  // per vertex: the vertex that stands for its position
  unsigned long long* ekey; int* ebal; int emask;   // edges (lower, upper vertex): uses upwards minus downwards
  int* flags;                // [0] 1: open, [1] roots of a closed mesh
  int* uf;                   // per node: parent
  int* roots;                // nodes without a parent
  signed char* sign;         // per root: 1 inside
  double* out;               // per node: distance, then signed
};

// MurmurHash3's 64-bit finalizer (Austin Appleby, public domain)
__device__ __forceinline__ unsigned sdf_mix(unsigned long long x) {
  x ^= x >> 33; x *= 0xff51afd7ed558ccdull; x ^= x >> 33; x *= 0xc4ceb9fe1a85ec53ull; x ^= x >> 33;
  return (unsigned)x;
}

__global__ void k_sdf_begin(SdfWork w) {
  const int i0 = blockIdx.x * blockDim.x + threadIdx.x, G = gridDim.x * blockDim.x;
  for (int i = i0; i <= SDF_CELLS; i += G) w.cnt[i] = 0;
  for (int i = i0; i <= w.vmask; i += G) w.vhash[i] = -1;
  for (int i = i0; i <= w.emask; i += G) { w.ekey[i] = ~0ull; w.ebal[i] = 0; }
  if (i0 < 2) w.flags[i0] = 0;
}

// rep[v]: the first vertex found at v's position (the table has at least twice
// as many entries as there are vertices)
__global__ void k_sdf_weld(SdfWork w) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= w.nv) return;
  const double x = w.V[3 * v] + 0.0, y = w.V[3 * v + 1] + 0.0, z = w.V[3 * v + 2] + 0.0;   // (-0 as +0)
  unsigned h = sdf_mix((unsigned long long)__double_as_longlong(x) * 3ull +
                       (unsigned long long)__double_as_longlong(y) * 5ull + (unsigned long long)__double_as_longlong(z));
  for (;; ++h) {
    const int o = atomicCAS(&w.vhash[h & (unsigned)w.vmask], -1, v);
    if (o < 0) { w.rep[v] = v; return; }
    if (w.V[3 * o] == x && w.V[3 * o + 1] == y && w.V[3 * o + 2] == z) { w.rep[v] = o; return; }
  }
}

// Morton cell of each triangle's centroid in the grid's box, its rank there;
// its edges
__global__ void k_sdf_tris(SdfWork w, SdfGrid g) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= w.nt) return;
  const int v[3] = {w.T[3 * t], w.T[3 * t + 1], w.T[3 * t + 2]};
  unsigned code = 0;
  for (int a = 0; a < 3; ++a) {
    const double c = (w.V[3 * v[0] + a] + w.V[3 * v[1] + a] + w.V[3 * v[2] + a]) / 3.0;
    const double u = g.mx[a] > g.mn[a] ? (c - g.mn[a]) / (g.mx[a] - g.mn[a]) * 16.0 : 0.0;
    const unsigned q = (unsigned)fmin(15.0, fmax(0.0, u));
    for (int b = 0; b < 4; ++b) code |= ((q >> b) & 1u) << (3 * b + a);
  }
  w.pos[t] = make_int2((int)code, atomicAdd(&w.cnt[code], 1));
  for (int e = 0; e < 3; ++e) {
    const int a = w.rep[v[e]], b = w.rep[v[e == 2 ? 0 : e + 1]];
    if (a == b) continue;
    const unsigned long long key = (unsigned long long)min(a, b) << 32 | (unsigned)max(a, b);
    for (unsigned h = sdf_mix(key);; ++h) {
      const unsigned s = h & (unsigned)w.emask;
      const unsigned long long o = atomicCAS(&w.ekey[s], ~0ull, key);
      if (o == ~0ull || o == key) { atomicAdd(&w.ebal[s], a < b ? 1 : -1); break; }
    }
  }
}

// exclusive prefix sum of the cells' counts, by one workgroup
__global__ void __launch_bounds__(256) k_sdf_cells_scan(SdfWork w) {
  __shared__ int sh[4];
  constexpr int PER = SDF_CELLS / 256;
  int v[PER], sum = 0;
  for (int i = 0; i < PER; ++i) { v[i] = w.cnt[threadIdx.x * PER + i]; sum += v[i]; }
  int tot;
  int acc = block_exclusive_scan(sum, sh, tot);
  for (int i = 0; i < PER; ++i) { w.cnt[threadIdx.x * PER + i] = acc; acc += v[i]; }
}

__global__ void k_sdf_scatter(SdfWork w) {
  const int i0 = blockIdx.x * blockDim.x + threadIdx.x, G = gridDim.x * blockDim.x;
  for (int t = i0; t < w.nt; t += G) {
    const int2 p = w.pos[t];
    double* o = w.tri + 9 * (size_t)(w.cnt[p.x] + p.y);
    for (int e = 0; e < 9; ++e) o[e] = w.V[3 * w.T[3 * t + e / 3] + e % 3];
  }
  for (int i = i0; i <= w.emask; i += G)
    if (w.ebal[i] != 0) w.flags[0] = 1;
}

// cluster boxes, wider by the slack on every side: half a wavefront each
__global__ void __launch_bounds__(256) k_sdf_boxes(SdfWork w, SdfGrid g) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  const double* p = w.tri + 9 * (size_t)min(t, w.nt - 1);   // (a cluster starts inside the list)
  double b[6];
  for (int a = 0; a < 3; ++a) {
    b[a] = fmin(fmin(p[a], p[3 + a]), p[6 + a]);
    b[3 + a] = fmax(fmax(p[a], p[3 + a]), p[6 + a]);
  }
  for (int o = SDF_CL / 2; o > 0; o >>= 1)
    for (int a = 0; a < 3; ++a) {
      b[a] = fmin(b[a], __shfl_xor(b[a], o, 64));
      b[3 + a] = fmax(b[3 + a], __shfl_xor(b[3 + a], o, 64));
    }
  if (t < w.nt && t % SDF_CL == 0)
    for (int a = 0; a < 6; ++a) w.box[6 * (size_t)(t / SDF_CL) + a] = a < 3 ? b[a] - g.slack : b[a] + g.slack;
}

__device__ __forceinline__ double wave_min(double v) {
  for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
  return v;
}

// squared distance of the box [lo, hi] to a cluster's box
__device__ __forceinline__ double sdf_box_gap(const double* lo, const double* hi, const double* box) {
  double s = 0.0;
  for (int a = 0; a < 3; ++a) {
    const double e = fmax(fmax(box[a] - hi[a], lo[a] - box[3 + a]), 0.0);
    s += e * e;
  }
  return s * (1.0 - 1e-9);
}

// Distances of one 2 x 2 x 2 block of nodes per wavefront, 8 lanes to a node
// (each takes every eighth triangle of a cluster; a minimum has no order).
// A first pass over the clusters' first vertices gives an upper bound and the
// cluster to start with; clusters that may hold a nearer triangle for some node
// are then staged in LDS and taken.  Bound by the FP64 distance arithmetic of the triangles left.  (A
// block of 64 nodes, one per lane, left half the device idle on a 32^3 grid
// and kept more clusters per block: 255 us for 448 triangles, now 64; 9,680 of
// a spiky ball on 64^3 2289 us, now 1250.)
constexpr int SDF_SPLIT = 8;
__global__ void __launch_bounds__(256) k_sdf_dist(SdfWork w, SdfGrid g) {
  __shared__ double st[4][SDF_CL * 9];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int bi = (g.I + 1) / 2, bj = (g.J + 1) / 2, bk = (g.K + 1) / 2;
  const long long blk = (long long)blockIdx.x * 4 + wave;
  if (blk >= (long long)bi * bj * bk) return;
  const int i0 = (int)(blk % bi) * 2, j0 = (int)(blk / bi % bj) * 2, k0 = (int)(blk / ((long long)bi * bj)) * 2;
  const int b = lane / SDF_SPLIT, part = lane % SDF_SPLIT;
  const int i = i0 + (b & 1), j = j0 + (b >> 1 & 1), k = k0 + (b >> 2);
  const bool in = i < g.I && j < g.J && k < g.K;
  const double p[3] = {g.at(0, min(i, g.I - 1)), g.at(1, min(j, g.J - 1)), g.at(2, min(k, g.K - 1))};
  const double lo[3] = {g.at(0, i0), g.at(1, j0), g.at(2, k0)};
  const double hi[3] = {g.at(0, min(i0 + 1, g.I - 1)), g.at(1, min(j0 + 1, g.J - 1)), g.at(2, min(k0 + 1, g.K - 1))};
  const int nc = (w.nt + SDF_CL - 1) / SDF_CL;
  double ub = INFINITY;
  int first = 0;
  for (int c = lane; c < nc; c += 64) {
    const double* a = w.tri + 9 * (size_t)c * SDF_CL;
    double u = 0.0;
    for (int x = 0; x < 3; ++x) {
      const double e = fmax(fabs(a[x] - lo[x]), fabs(a[x] - hi[x]));
      u += e * e;
    }
    if (u < ub) { ub = u; first = c; }
  }
  const double least = wave_min(ub);
  first = __shfl(first, __ffsll((unsigned long long)__ballot(ub == least)) - 1, 64);
  ub = least * (1.0 + 1e-9);
  double best = INFINITY;
  auto take = [&](int c) {
    const int n = min(SDF_CL, w.nt - c * SDF_CL);
    const double* src = w.tri + 9 * (size_t)c * SDF_CL;
    for (int e = lane; e < 9 * n; e += 64) st[wave][e] = src[e];
    wave_sync_lds();
    for (int t = part; t < n; t += SDF_SPLIT) best = fmin(best, tri_sqdist_select(p[0], p[1], p[2], st[wave] + 9 * t));
    wave_sync_lds();
    for (int o = 1; o < SDF_SPLIT; o <<= 1) best = fmin(best, __shfl_xor(best, o, 64));
  };
  take(first);
  for (int c0 = 0; c0 < nc; c0 += 64) {
    const int c = c0 + lane;
    const double most = fmin(ub, -wave_min(-best));   // no node's triangle is farther
    unsigned long long m = __ballot(c < nc && c != first && !(sdf_box_gap(lo, hi, w.box + 6 * (size_t)c) > most));
    while (m) {
      const int cc = c0 + __ffsll((long long)m) - 1;
      m &= m - 1;
      if (__ballot(!(sdf_box_gap(p, p, w.box + 6 * (size_t)cc) > best))) take(cc);
    }
  }
  if (in && part == 0) w.out[i + g.I * ((long long)j + (long long)g.J * k)] = sqrt(best);
}

// Each node's parent: of the neighbours on its side (the segment between them
// is shorter than the distance of one of them from the surface, so it does not
// meet the surface) the farthest from the surface, if that is farther than the
// node itself; a tie goes to the lower index.  Parents only climb, so the nodes
// form trees, and a tree lies on one side.  No atomics, and few roots: the local
// maxima of the distance, and the nodes next to or on the surface that no
// neighbour reaches.
__global__ void k_sdf_climb(SdfWork w, SdfGrid g, int n) {
  if (w.flags[0]) return;   // an open mesh
  const int stride[3] = {1, g.I, g.I * g.J}, dim[3] = {g.I, g.J, g.K};
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    const int x[3] = {p % g.I, p / g.I % g.J, p / (g.I * g.J)};
    const double d = w.out[p];
    double top = d;
    int to = p;
    for (int a = 0; a < 3; ++a)
      for (int s = -1; s <= 1; s += 2) {
        if (x[a] + s < 0 || x[a] + s >= dim[a]) continue;
        const int q = p + s * stride[a];
        const double e = w.out[q];
        if (!(fmax(d, e) > g.h[a] * (1.0 + 1e-9) + g.slack)) continue;
        if (e > top || (e == top && q < to)) { top = e; to = q; }
      }
    w.uf[p] = to;
  }
}

// the trees' roots, listed in any order
__global__ void k_sdf_roots(SdfWork w, int n) {
  if (w.flags[0]) return;
  for (int p0 = blockIdx.x * blockDim.x; p0 < n; p0 += gridDim.x * blockDim.x) {
    const int p = p0 + (int)threadIdx.x, lane = (int)(threadIdx.x & 63);
    const bool r = p < n && w.uf[p] == p;
    const unsigned long long m = __ballot(r);
    if (!m) continue;
    int base = 0;
    if (lane == 0) base = atomicAdd(&w.flags[1], __popcll(m));
    base = __shfl(base, 0, 64);
    if (r) w.roots[base + lanes_below(m)] = p;
  }
}

__device__ __forceinline__ void sdf_corners(const SdfWork& w, int t, double* c) {
  for (int e = 0; e < 9; ++e) c[e] = w.V[3 * w.T[3 * t + e / 3] + e % 3];
}

constexpr double SDF_4PI = 4.0 * 3.14159265358979323846;

// sum of the solid angles at p in k_sdf's order, by a wavefront; sh: 64 values
__device__ __forceinline__ double sdf_angles(const SdfWork& w, double px, double py, double pz, double* sh, int lane) {
  double wsum = 0.0;
  for (int t0 = 0; t0 < w.nt; t0 += 64) {
    const int t = t0 + lane, n = min(64, w.nt - t0);
    if (t < w.nt) {
      double c[9];
      sdf_corners(w, t, c);
      sh[lane] = solid_angle(px, py, pz, c);
    }
    wave_sync_lds();
    for (int e = 0; e < n; ++e) wsum += sh[e];
    wave_sync_lds();
  }
  return wsum;
}

// Whether |winding number| > 1/2 at the roots (of an open mesh: at every node),
// from the sum of their solid angles (4 pi wn): a sum in any order decides unless
// it lies near 1/2 (or is not a number); sdf_angles then adds the terms in k_sdf's
// order.  A wavefront per root (a thread each took 0.4 us a triangle in series), or,
// from SDF_MANY roots on, a thread each with the triangles staged in LDS: the threads
// then hide that chain, and a triangle is read once for 256 nodes and not once for
// each (408 triangles with a hole on 51^3 1.03 ms by wavefronts, 1.06 by threads; on
// 58^3 0.96, 0.82; on 128^3 8.3, 6.7; 9,999 on 51^3 7.4, 9.8; on 58^3 10.8, 9.6).
// What is left over the plain build is least for strewn triangles, which cluster
// badly: 500 on 128^3 10.2 ms (plain 10.3).
constexpr int SDF_MANY = 163840;
__global__ void __launch_bounds__(256) k_sdf_sign(SdfWork w, SdfGrid g, int n) {
  __shared__ double st[SDF_TILE * 9];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const bool open = w.flags[0] != 0;
  const int nr = open ? n : w.flags[1];
  auto inside_by = [](double sum) { return fabs(sum / SDF_4PI) > 0.5; };
  auto put = [&](int node, bool inside) {
    if (!open) w.sign[node] = inside ? 1 : 0;
    else if (inside) w.out[node] = -w.out[node];
  };
  auto sure = [](double sum) { return fabs(fabs(sum / SDF_4PI) - 0.5) > 1e-6; };
  if (nr >= SDF_MANY) {
    for (int r0 = blockIdx.x * 256; r0 < nr; r0 += gridDim.x * 256) {
      const int r = r0 + (int)threadIdx.x;
      const bool have = r < nr;
      const int node = have ? (open ? r : w.roots[r]) : 0;
      const double px = g.at(0, node % g.I), py = g.at(1, node / g.I % g.J), pz = g.at(2, node / (g.I * g.J));
      TurnSum ts;
      for (int t0 = 0; t0 < w.nt; t0 += SDF_TILE) {
        const int cnt = min(SDF_TILE, w.nt - t0);
        for (int e = threadIdx.x; e < 9 * cnt; e += 256) st[e] = w.tri[9 * (size_t)t0 + e];
        __syncthreads();
        for (int e = 0; e < cnt; ++e) {
          double det, den;
          solid_angle_parts(px, py, pz, st + 9 * e, det, den);
          ts.add(det, den);
        }
        __syncthreads();
      }
      const double sum = ts.angle();
      bool inside = inside_by(sum);
      for (unsigned long long m = __ballot(have && !sure(sum)); m; m &= m - 1) {
        const int l = __ffsll((long long)m) - 1;
        const bool in = inside_by(sdf_angles(w, __shfl(px, l, 64), __shfl(py, l, 64), __shfl(pz, l, 64), st + 64 * wave, lane));
        if (lane == l) inside = in;
      }
      if (have) put(node, inside);
      __syncthreads();   // st is staged again
    }
    return;
  }
  for (int r = blockIdx.x * 4 + wave; r < nr; r += gridDim.x * 4) {
    const int node = open ? r : w.roots[r];
    const double px = g.at(0, node % g.I), py = g.at(1, node / g.I % g.J), pz = g.at(2, node / (g.I * g.J));
    TurnSum ts;
    for (int t = lane; t < w.nt; t += 64) {
      double c[9], det, den;
      sdf_corners(w, t, c);
      solid_angle_parts(px, py, pz, c, det, den);
      ts.add(det, den);
    }
    double sum = ts.angle();
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    if (!sure(sum)) sum = sdf_angles(w, px, py, pz, st + 64 * wave, lane);   // (uniform over the wavefront)
    if (lane == 0) put(node, inside_by(sum));
  }
}

__global__ void k_sdf_apply(SdfWork w, int n) {
  if (w.flags[0]) return;   // (k_sdf_sign has done it)
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x) {
    int r = p;
    for (int q = w.uf[r]; q != r; q = w.uf[r]) r = q;
    if (w.sign[r]) w.out[p] = -w.out[p];
  }
}

}  // namespace rbh
