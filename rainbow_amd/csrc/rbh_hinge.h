// Hinge joints: the second problem of the prox solve (constraints/hinges.py).
//
// The reference solves the contact problem and the hinge problem in one
// driver loop (gauss_seidel_solver.py:44-94, problems from steppers.py:68-76):
// each sweep updates both, each keeps its own merit, accept/reject and
// r-factors, and the stopping tests use the larger of the two contributions.
// The problems share no unknowns (each sweep recomputes its own w = W J^T x),
// so the hinge problem's sequence of iterates does not depend on the
// contacts.  Here it runs on its own, in two passes of one wavefront per
// scene:
//   pass 0 (before the contact solve, scenes with contacts): max_iter sweeps,
//          recording the hinge contribution of every sweep in h_mer; the
//          contact solve's stopping tests read it;
//   pass 1 (after it): the same sweeps again up to the sweep the joint
//          stopping test ended on -- or, in a scene without contacts, the
//          whole solve with its own stopping tests and residual log -- then
//          W J^T sol per body for the velocity update.
// A hinge sweep is serial over the hinges (Gauss-Seidel); inside one hinge
// the five rows update from the same w (hinges.py:88), one lane per row, and
// the twelve body entries of W J^T delta one lane each.  w, the iterate and
// the accepted solution stay in LDS, and so do the rows of all hinges where
// hinge_launch has them staged; else the rows of the next HINGE_AHEAD hinges are
// loaded from memory while one updates.
// (included inside namespace rbh by rbh_kernels.h)
#pragma once

constexpr int HINGE_BODY_MAX = 1024;   // bodies joined by hinges in one scene (LDS: two V4 each)
constexpr int HINGE_MAX = 1024;        // hinges of one scene (LDS: 5 iterates and 5 accepted values each; FP64 total 144 KB)

// One J row (parent lin, parent ang, child lin, child ang) times body-space
// vectors, term by term in the csr column order of hinges.py:184 (the body of
// lower index first), from zero.
template <typename R>
__device__ __forceinline__ R hinge_rowdot(bool pfirst, const V4<R>* J, V3<R> pl, V3<R> pa, V3<R> cl, V3<R> ca) {
  V4<R> a0 = pfirst ? J[0] : J[2], a1 = pfirst ? J[1] : J[3], a2 = pfirst ? J[2] : J[0], a3 = pfirst ? J[3] : J[1];
  V3<R> b0 = pfirst ? pl : cl, b1 = pfirst ? pa : ca, b2 = pfirst ? cl : pl, b3 = pfirst ? ca : pa;
  R s = R(0);
  s += a0.x * b0.x; s += a0.y * b0.y; s += a0.z * b0.z;
  s += a1.x * b1.x; s += a1.y * b1.y; s += a1.z * b1.z;
  s += a2.x * b2.x; s += a2.y * b2.y; s += a2.z * b2.z;
  s += a3.x * b3.x; s += a3.y * b3.y; s += a3.z * b3.z;
  return s;
}

template <typename R> __device__ __forceinline__ V4<R> v4(V3<R> a) { return V4<R>{a.x, a.y, a.z, R(0)}; }

// Hinges.initialize (hinges.py:28-48): J (:103-185), W J^T, g (:187-218),
// b = J u + J (dt du_ext) + g, diag of J W J^T (0 -> 1), r = 1/diag.
// One workgroup per batch scene, one thread per hinge.
template <typename R> __global__ void __launch_bounds__(64) k_hinge_rows(Dev<R> d) {
  if (aborted(d.err)) return;
  const int slot = d.bs_slot[blockIdx.x];
  const SceneParams& sp = d.sp[slot];
  const R dt = scene_dt(d, slot);
  for (int k = threadIdx.x; k < sp.h_cnt; k += blockDim.x) {
    const int h = sp.h_off + k;
    const int4 id = d.h_ids[h];
    const int P = id.x, C = id.y;
    const Quat<R> qp = quat(d.q[P]), qc = quat(d.q[C]);
    const V3<R> arm_p = qrotate(qp, xyz(d.h_geo[4 * h])), arm_c = qrotate(qc, xyz(d.h_geo[4 * h + 1]));
    V3<R> t, b, n;
    orthonormal_frame(qrotate(qp, xyz(d.h_geo[4 * h + 2])), t, b, n);
    R g[5] = {R(0), R(0), R(0), R(0), R(0)};
    if (sp.use_pre_stab) {
      const V3<R> rp = arm_p + xyz(d.r[P]), rc = arm_c + xyz(d.r[C]);
      const V3<R> u = cross(n, qrotate(qc, xyz(d.h_geo[4 * h + 3])));
      const R rate = R(sp.gap_reduction) / dt;
      g[0] = (rc.x - rp.x) * rate; g[1] = (rc.y - rp.y) * rate; g[2] = (rc.z - rp.z) * rate;
      g[3] = dot(t, u) * rate; g[4] = dot(b, u) * rate;
    }
    R imP, imC, WP[6], WC[6];
    load_W(d, P, imP, WP);
    load_W(d, C, imC, WC);
    const V3<R> z3 = {R(0), R(0), R(0)};
    const V3<R> up_l = xyz(d.v[P]), up_a = xyz(d.w[P]), uc_l = xyz(d.v[C]), uc_a = xyz(d.w[C]);
    const V3<R> dp_l = dt * xyz(d.b_du0[P]), dp_a = dt * xyz(d.b_du1[P]);
    const V3<R> dc_l = dt * xyz(d.b_du0[C]), dc_a = dt * xyz(d.b_du1[C]);
    const bool pfirst = P < C;
    for (int i = 0; i < 5; ++i) {
      V3<R> pl = z3, pa, cl = z3, ca;
      if (i < 3) {
        // rows 0-2: parent [I | -[arm_p]x], child [-I | [arm_c]x]; row i of [a]x
        // is (0, -a.z, a.y), (a.z, 0, -a.x), (-a.y, a.x, 0)
        const V3<R> sp_row = i == 0 ? V3<R>{R(0), -arm_p.z, arm_p.y}
                                    : (i == 1 ? V3<R>{arm_p.z, R(0), -arm_p.x} : V3<R>{-arm_p.y, arm_p.x, R(0)});
        const V3<R> sc_row = i == 0 ? V3<R>{R(0), -arm_c.z, arm_c.y}
                                    : (i == 1 ? V3<R>{arm_c.z, R(0), -arm_c.x} : V3<R>{-arm_c.y, arm_c.x, R(0)});
        pl = V3<R>{R(i == 0), R(i == 1), R(i == 2)};
        cl = -pl;
        pa = -sp_row;
        ca = sc_row;
      } else {
        const V3<R> dir = i == 3 ? t : b;
        pa = dir;
        ca = -dir;
      }
      V4<R> J[4] = {v4(pl), v4(pa), v4(cl), v4(ca)};
      V4<R> WJ[4] = {v4(imP * pl), v4(sym_mul(WP, pa)), v4(imC * cl), v4(sym_mul(WC, ca))};
      const R ju = hinge_rowdot(pfirst, J, up_l, up_a, uc_l, uc_a);
      const R jd = hinge_rowdot(pfirst, J, dp_l, dp_a, dc_l, dc_a);
      const R dg = hinge_rowdot(pfirst, J, xyz(WJ[0]), xyz(WJ[1]), xyz(WJ[2]), xyz(WJ[3]));
      for (int j = 0; j < 4; ++j) {
        d.h_J[20 * h + 4 * i + j] = J[j];
        d.h_WJ[20 * h + 4 * i + j] = WJ[j];
      }
      d.h_b[5 * h + i] = (ju + jd) + g[i];
      d.h_r0[5 * h + i] = R(1) / (dg == R(0) ? R(1) : dg);
    }
  }
}

// w = W J^T x for the scene's hinge bodies (hinges.py:65, :56): one running
// sum per body entry over the body's hinges in hinge order, rows 0..4; x
// holds the scene's rows, row i of hinge h at 5 (h - sp.h_off) + i.
template <typename R>
__device__ __forceinline__ void hinge_body_w(const Dev<R>& d, const SceneParams& sp, const R* x, V4<R>* wl, V4<R>* wa) {
  for (int j = threadIdx.x; j < sp.hb_cnt; j += blockDim.x) {
    const int g = sp.hb_off + j;
    V3<R> sl = {R(0), R(0), R(0)}, sa = {R(0), R(0), R(0)};
    for (int e = d.hb_inc_off[g]; e < d.hb_inc_off[g + 1]; ++e) {
      const int inc = d.hb_inc[e], h = inc >> 1, side = inc & 1;
      for (int i = 0; i < 5; ++i) {
        const R xi = x[5 * (h - sp.h_off) + i];
        const V4<R> l = d.h_WJ[20 * h + 4 * i + 2 * side], a = d.h_WJ[20 * h + 4 * i + 2 * side + 1];
        sl.x += l.x * xi; sl.y += l.y * xi; sl.z += l.z * xi;
        sa.x += a.x * xi; sa.y += a.y * xi; sa.z += a.z * xi;
      }
    }
    wl[j] = v4(sl);
    wa[j] = v4(sa);
  }
}

// Per-hinge constants a lane needs for one Gauss-Seidel update: lanes 0-4
// hold row `lane` (J, b, r0), lanes 0-11 the W J^T entries of body entry
// `lane` for rows 0-4.  Loaded HINGE_AHEAD hinges ahead of their use.
template <typename R> struct HingeRegs {
  int4 id;
  V4<R> J[4];
  R b, r0;
  R wj[5];
};

template <typename R>
__device__ __forceinline__ void hinge_load(const Dev<R>& d, int h, int lane, HingeRegs<R>& g) {
  g.id = d.h_ids[h];
  if (lane < 5) {
    const V4<R>* J = d.h_J + 20 * h + 4 * lane;
    g.J[0] = J[0]; g.J[1] = J[1]; g.J[2] = J[2]; g.J[3] = J[3];
    g.b = d.h_b[5 * h + lane];
    g.r0 = d.h_r0[5 * h + lane];
  }
  if (lane < 12) {
    const int part = lane / 3, c = lane - 3 * part;
    // one element each (a runtime index into a vector register would go through scratch)
    for (int i = 0; i < 5; ++i) g.wj[i] = reinterpret_cast<const R*>(d.h_WJ + 20 * h + 4 * i + part)[c];
  }
}

constexpr int HINGE_AHEAD = 4;   // hinges whose rows are loaded ahead of their update

// One hinge's Gauss-Seidel update on w (LDS) and its iterate x (LDS, rows
// from x0): hinges.py:88 then :101.
template <typename R>
__device__ __forceinline__ void hinge_update(V4<R>* wl, V4<R>* wa, R* x, R* s_delta, int x0, R rs,
                                             const HingeRegs<R>& g, int lane) {
  const int4 id = g.id;
  if (lane < 5) {
    // x_b -= r_b (J w + b)_b with every row of the block from the same w
    const R jw = hinge_rowdot(id.x < id.y, g.J, xyz(wl[id.z]), xyz(wa[id.z]), xyz(wl[id.w]), xyz(wa[id.w]));
    const R xo = x[x0 + lane];
    const R xn = xo - (g.r0 * rs) * (jw + g.b);
    x[x0 + lane] = xn;
    s_delta[lane] = xn - xo;
  }
  // one wavefront: LDS operations stay in issue order, and a fence-free sync
  // keeps the loads of the next hinges in flight (a workgroup barrier would
  // wait for them)
  wave_sync_lds();
  if (lane < 12) {
    // w += W J^T_b delta, one body entry per lane
    const int part = lane / 3, c = lane - 3 * part;
    R t = R(0);
    for (int i = 0; i < 5; ++i) t += g.wj[i] * s_delta[i];
    V4<R>* wv = (part & 1) ? wa : wl;
    R* dst = reinterpret_cast<R*>(wv + (part < 2 ? id.z : id.w)) + c;
    *dst = *dst + t;
  }
  wave_sync_lds();
}

// Bytes of dynamic LDS the hinge solve of a scene needs: w (two V4 per hinge
// body), the iterate x and the accepted solution sol (5 each per hinge).
template <typename R> __host__ __device__ constexpr size_t hinge_lds_bytes(int hb, int nh) {
  return (2 * (size_t)hb * sizeof(V4<R>) + 10 * (size_t)nh * sizeof(R) + 15) & ~(size_t)15;
}

// ---- rows staged in LDS
//
// A sweep is one wavefront's chain of instructions: ~700 cycles an update from
// LDS (12 products summed in order, the five deltas by DPP, 5 more products,
// and reading the next hinge's rows), ~1,000 for w from x, ~1,000 for the merit
// and the decision; from memory every read of a row waited for the cache.
// Chains of 5, 16 and 48 cubes, 100 sweeps, four steps: 1.93, 3.71 and 9.30 ms
// from memory, 1.83, 3.09 and 6.77 staged.
// Up to 64 KB, so that at least two scenes of a batch share a CU: a chain of 83
// hinges in FP32, 42 in FP64 (which of the batches that fit are staged:
// hinge_launch).  The two paths are kernels of their own: in one, the rows in
// registers of one and of the other left the path from memory one wavefront a
// SIMD instead of two (256 links 12.5 ms a step, alone 11.3).
constexpr size_t HINGE_STAGE = 64 * 1024;

template <typename R> struct HingeLds {
  static constexpr int VB = (int)sizeof(V4<R>), SR = (int)sizeof(R);
  int wl, wa, x;             // as in the kernel's layout
  int J, WJ, ids, br, off, inc;   // rows of J (body of lower index first), of W J^T, int4 (parent, child, first, second
                                  // slot), b and r0, the bodies' hinge lists
  // where the rows start: a whole vec4 (an odd number of hinges leaves half of one in FP64)
  __host__ __device__ static constexpr size_t rows_at(int hb, int nh) {
    return (hinge_lds_bytes<R>(hb, nh) + VB - 1) / VB * VB;
  }
  __host__ __device__ static constexpr size_t bytes(int hb, int nh) {
    return rows_at(hb, nh) + (size_t)nh * (40 * VB + 16 + 10 * SR + 8) + 4 * ((size_t)hb + 1);
  }
  __device__ HingeLds(unsigned char* smem, int hb, int nh) {
    wl = lds_addr(smem);
    wa = wl + hb * VB;
    x = wa + hb * VB;
    J = wl + (int)rows_at(hb, nh);
    WJ = J + 20 * nh * VB;
    ids = WJ + 20 * nh * VB;
    br = ids + 16 * nh;
    off = br + 10 * nh * SR;
    inc = off + 4 * (hb + 1);
  }
};

// How a batch's hinge solve is launched: the rows of all its scenes staged, or
// none; the dynamic LDS of a workgroup.
struct HingeLaunch {
  bool staged;
  size_t lds;
};

// n hinged scenes of bodies[i] bodies in hinges[i] hinges on `cus` compute units.
//
// Staged, an update takes 1 / 1.5 of its time from memory as long as a CU has one
// scene; but a scene's workgroup keeps its rows' LDS, so R = LDS / its bytes of
// them share a CU, where up to W = 8 (FP64 4, by their registers) share it from
// memory, at 1.3 + 0.2 w of the staged time for w of them (80 links, 30 sweeps:
// 256 scenes 1.4 ms a step, 512 1.9, 1,024 2.3, 1,280 2.3, 2,048 2.8; staged, with
// R = 2, 1.0, 1.1, 1.9, 2.8 and 3.9).  Either way takes as long as the longest
// scene, or as the CU's scenes R or W at a time; the shorter way is taken.  Short
// scenes stay staged at any number (2,048 of 40 links 1.4 against 1.6, 4,096 of
// 20 1.6 against 2.0, 2,048 of 40 in FP64 2.5 against 3.1).
template <typename R>
HingeLaunch hinge_launch(int cus, int n, const int* bodies, const int* hinges) {
  size_t mem = 16, st = 16;
  double all = 0.0, longest = 0.0;
  for (int i = 0; i < n; ++i) {
    mem = std::max(mem, hinge_lds_bytes<R>(bodies[i], hinges[i]));
    st = std::max(st, HingeLds<R>::bytes(bodies[i], hinges[i]));
    all += hinges[i];
    longest = std::max(longest, (double)hinges[i]);
  }
  if (st > HINGE_STAGE) return HingeLaunch{false, mem};
  const double per_cu = all / cus;                                  // updates a CU has to do
  const double scenes = (double)((n + (long)cus - 1) / cus);        // its scenes
  const double r = std::floor(160.0 * 1024.0 / (double)st), w = std::min(scenes, sizeof(R) == 4 ? 8.0 : 4.0);
  const double t_staged = std::max(longest, std::ceil(scenes / r) * per_cu / scenes);
  const double t_memory = std::max(1.5 * longest, per_cu * (1.3 + 0.2 * w) / w);
  return t_staged <= t_memory ? HingeLaunch{true, st} : HingeLaunch{false, mem};
}

template <typename R> __device__ void hinge_stage(const Dev<R>& d, const SceneParams& sp, const HingeLds<R>& L) {
  constexpr int VB = HingeLds<R>::VB, SR = HingeLds<R>::SR;
  const int lane = threadIdx.x, nh = sp.h_cnt, h0 = sp.h_off;
  for (int i = lane; i < 20 * nh; i += 64) {
    const int h = i / 20, k = i - 20 * h;
    const int4 id = d.h_ids[h0 + h];
    const int to = id.x < id.y ? i : 20 * h + (k ^ 2);   // parent first or child first
    lds_at<V4<R>>(L.J + to * VB) = d.h_J[20 * h0 + i];
    lds_at<V4<R>>(L.WJ + i * VB) = d.h_WJ[20 * h0 + i];
  }
  for (int i = lane; i < 5 * nh; i += 64) {
    lds_at<R>(L.br + i * SR) = d.h_b[5 * h0 + i];
    lds_at<R>(L.br + (5 * nh + i) * SR) = d.h_r0[5 * h0 + i];
  }
  for (int h = lane; h < nh; h += 64) {
    const int4 id = d.h_ids[h0 + h];
    const bool pfirst = id.x < id.y;
    lds_at<int4>(L.ids + 16 * h) = make_int4(id.z, id.w, pfirst ? id.z : id.w, pfirst ? id.w : id.z);
  }
  const int e0 = d.hb_inc_off[sp.hb_off];
  for (int j = lane; j <= sp.hb_cnt; j += 64) lds_at<int>(L.off + 4 * j) = d.hb_inc_off[sp.hb_off + j] - e0;
  for (int e = lane; e < 2 * nh; e += 64) lds_at<int>(L.inc + 4 * e) = d.hb_inc[e0 + e] - 2 * h0;
  for (int i = lane; i < 2 * sp.hb_cnt; i += 64) lds_at<V4<R>>(L.wl + i * VB) = V4<R>{R(0), R(0), R(0), R(0)};
}

// hinge_body_w, one component of a body per lane; x: LDS address of the rows
template <typename R> __device__ __forceinline__ void hinge_body_w_lds(const HingeLds<R>& L, int hb, int x) {
  constexpr int VB = HingeLds<R>::VB, SR = HingeLds<R>::SR;
  for (int t = threadIdx.x; t < 6 * hb; t += 64) {
    const int j = t / 6, k = t - 6 * j, ang = k >= 3, c = ang ? k - 3 : k;
    const int end = lds_at<int>(L.off + 4 * j + 4);
    int e = lds_at<int>(L.off + 4 * j), ahead = lds_at<int>(L.inc + 4 * e);   // (every body has a hinge)
    R s = R(0);
    for (; e < end; ++e) {
      const int inc = ahead, h = inc >> 1, side = inc & 1;
      ahead = lds_at<int>(L.inc + 4 * min(e + 1, end - 1));
      const int w = L.WJ + (20 * h + 2 * side + ang) * VB + c * SR;
#pragma unroll
      for (int i = 0; i < 5; ++i) s += lds_at<R>(w + 4 * i * VB) * lds_at<R>(x + (5 * h + i) * SR);
    }
    lds_at<R>((ang ? L.wa : L.wl) + j * VB + c * SR) = s;
  }
}

// what a lane of the first row needs of a hinge
template <typename R> struct HingeRow {
  V4<R> J[4];
  R b, r0, wj[5];
  int first, second, dst;   // LDS: slots of the bodies in row order, this lane's entry of w
};

template <typename R>
__device__ __forceinline__ void hinge_row(const HingeLds<R>& L, int nh, int h, int lane, HingeRow<R>& g) {
  constexpr int VB = HingeLds<R>::VB, SR = HingeLds<R>::SR;
  const int row = min(lane, 4), part = min(lane / 3, 3), c = lane % 3;
  const int4 id = lds_at<int4>(L.ids + 16 * h);
  for (int k = 0; k < 4; ++k) g.J[k] = lds_at<V4<R>>(L.J + (20 * h + 4 * row + k) * VB);
  g.b = lds_at<R>(L.br + (5 * h + row) * SR);
  g.r0 = lds_at<R>(L.br + (5 * (nh + h) + row) * SR);
  for (int i = 0; i < 5; ++i) g.wj[i] = lds_at<R>(L.WJ + (20 * h + 4 * i + part) * VB + c * SR);
  g.first = id.z * VB;
  g.second = id.w * VB;
  g.dst = ((part & 1) ? L.wa : L.wl) + (part < 2 ? id.x : id.y) * VB + c * SR;
}

// hinge_update from LDS; the five deltas go to the other lanes by DPP.  The
// rows of hinge `next` are read behind this one's w: LDS answers in order, and
// w is what the chain waits for.
template <typename R>
__device__ __forceinline__ void hinge_update_lds(const HingeLds<R>& L, int nh, int h, int next, R rs,
                                                 const HingeRow<R>& g, HingeRow<R>& n, int lane) {
  constexpr int SR = HingeLds<R>::SR;
  const int xa = L.x + (5 * h + min(lane, 4)) * SR;
  const V3<R> b0 = xyz(lds_at<V4<R>>(L.wl + g.first)), b1 = xyz(lds_at<V4<R>>(L.wa + g.first));
  const V3<R> b2 = xyz(lds_at<V4<R>>(L.wl + g.second)), b3 = xyz(lds_at<V4<R>>(L.wa + g.second));
  const R old = lds_at<R>(g.dst), xo = lds_at<R>(xa);
  __builtin_amdgcn_sched_barrier(0);
  hinge_row(L, nh, next, lane, n);
  R s = R(0);
  s += g.J[0].x * b0.x; s += g.J[0].y * b0.y; s += g.J[0].z * b0.z;
  s += g.J[1].x * b1.x; s += g.J[1].y * b1.y; s += g.J[1].z * b1.z;
  s += g.J[2].x * b2.x; s += g.J[2].y * b2.y; s += g.J[2].z * b2.z;
  s += g.J[3].x * b3.x; s += g.J[3].y * b3.y; s += g.J[3].z * b3.z;
  const R xn = xo - (g.r0 * rs) * (s + g.b);
  const R delta = xn - xo;
  R t = R(0);
  t += g.wj[0] * row_bcast<0>(delta);
  t += g.wj[1] * row_bcast<1>(delta);
  t += g.wj[2] * row_bcast<2>(delta);
  t += g.wj[3] * row_bcast<3>(delta);
  t += g.wj[4] * row_bcast<4>(delta);
  if (lane < 5) lds_at<R>(xa) = xn;
  if (lane < 12) lds_at<R>(g.dst) = old + t;
  wave_sync_lds();
}

template <typename R> __device__ __forceinline__ void hinge_sweep_lds(const HingeLds<R>& L, int nh, R rs) {
  const int lane = threadIdx.x;
  HingeRow<R> a, b;
  hinge_row(L, nh, 0, lane, a);
  for (int h = 0; h < nh; h += 2) {
    hinge_update_lds(L, nh, h, min(h + 1, nh - 1), rs, a, b, lane);
    if (h + 1 >= nh) break;
    hinge_update_lds(L, nh, h + 1, min(h + 2, nh - 1), rs, b, a, lane);
  }
}

// One wavefront per batch scene.  pass 0 records the hinge merit
// contributions for the contact solve; pass 1 runs to the joint stop and
// writes hd0/hd1 (see the top of this file).  w, x and the accepted
// solution sol live in LDS, and, STAGED, the rows too.
template <typename R, bool STAGED> __global__ void __launch_bounds__(64) k_hinge_solve(Dev<R> d, int pass) {
  extern __shared__ __align__(32) unsigned char hinge_smem[];
  if (aborted(d.err)) return;
  const int slot = d.bs_slot[blockIdx.x];
  const SceneParams& sp = d.sp[slot];
  SceneState& st = d.ss[slot];
  if (sp.h_cnt == 0) return;
  const bool contacts = st.k_cnt > 0;
  if (pass == 0 && !contacts) return;
  const bool own = pass == 1 && !contacts;   // the hinge problem alone: its own stopping tests and log
  const int n_it = (pass == 1 && contacts) ? (st.exitcode == 0 ? sp.max_iter : st.iterations + 1) : sp.max_iter;
  V4<R>* wl = reinterpret_cast<V4<R>*>(hinge_smem);
  V4<R>* wa = wl + sp.hb_cnt;
  const int lane = threadIdx.x;
  const int h0 = sp.h_off, h1 = sp.h_off + sp.h_cnt, nrow = 5 * sp.h_cnt;
  R* x = reinterpret_cast<R*>(wa + sp.hb_cnt);   // row 5 (h - h0) + i
  R* sol = x + nrow;
  double* res = d.residuals + sp.res_off;
  double* hm = d.h_mer + sp.res_off;
  const HingeLds<R> L(hinge_smem, sp.hb_cnt, sp.h_cnt);   // (STAGED: the launch has room for it)
  if constexpr (STAGED) hinge_stage(d, sp, L);
  for (int i = lane; i < nrow; i += 64) { x[i] = R(0); sol[i] = R(0); }
  if (own)
    for (int i = lane; i < sp.max_iter; i += 64) res[i] = INFINITY;
  __syncthreads();
  const CtlParams cp(sp);
  SolveCtl ctl;
  ctl.iters = sp.max_iter;
  for (int it = 0; it < n_it; ++it) {
    const R rs = R(ctl.rscale);
    if constexpr (STAGED) {
      hinge_body_w_lds(L, sp.hb_cnt, L.x);
      __syncthreads();
      hinge_sweep_lds(L, sp.h_cnt, rs);
      __syncthreads();
    } else {
      __shared__ R s_delta[5];
      hinge_body_w(d, sp, x, wl, wa);
      // rows of the next HINGE_AHEAD hinges in flight while one updates
      HingeRegs<R> ring[HINGE_AHEAD];
#pragma unroll
      for (int k = 0; k < HINGE_AHEAD; ++k)
        if (h0 + k < h1) hinge_load(d, h0 + k, lane, ring[k]);
      __syncthreads();
      for (int hh = h0; hh < h1; hh += HINGE_AHEAD) {
#pragma unroll
        for (int k = 0; k < HINGE_AHEAD; ++k) {
          const int h = hh + k;
          if (h >= h1) break;
          hinge_update(wl, wa, x, s_delta, 5 * (h - h0), rs, ring[k], lane);
          if (h + HINGE_AHEAD < h1) hinge_load(d, h + HINGE_AHEAD, lane, ring[k]);
        }
      }
    }
    double m = 0.0;
    for (int i = lane; i < nrow; i += 64) m = fmax(m, fabs((double)(x[i] - sol[i])));
    m = wave_max(m);
    int dec;
    if (own) {
      dec = ctl.decide(cp, m, lane == 0 ? res : nullptr, it);
    } else {
      dec = ctl.accept_or_reject(cp, m);
      if (pass == 0 && lane == 0) hm[it] = ctl.gm;
    }
    for (int i = lane; i < nrow; i += 64) {
      if (dec & 1) sol[i] = x[i];
      else x[i] = sol[i];
    }
    __syncthreads();
    if (dec & 2) { ctl.iters = it; break; }
  }
  if (pass == 0) return;
  if (own && lane == 0) {
    st.iterations = ctl.iters;
    st.exitcode = ctl.exitcode;
    st.rejects = ctl.rejects;
    st.sweeps = ctl.sweeps;
    st.final_merit = ctl.last_merit;
  }
  // finalize_solution (hinges.py:50-57): W J^T sol per body
  if constexpr (STAGED) hinge_body_w_lds(L, sp.hb_cnt, L.x + nrow * (int)sizeof(R));
  else hinge_body_w(d, sp, sol, wl, wa);
  __syncthreads();
  for (int j = lane; j < sp.hb_cnt; j += 64) {
    const int b = d.hb_body[sp.hb_off + j];
    d.hd0[b] = wl[j];
    d.hd1[b] = wa[j];
  }
}
