// Islands, random colouring, colour order and the proximal Gauss-Seidel /
// Jacobi solve.
//
// Islands: connected components of free bodies linked by contacts (fixed
// bodies have a zero inverse-mass block, so contacts only interact through
// free bodies).  Contacts are regrouped by island ("unit order"); islands are
// packed into colouring units of at most unit_T contacts that never straddle
// a scene.  Each unit is coloured by one workgroup with its state in LDS.
//
// Every body's contacts are solved in the order of their colours (contacts of
// one colour share no free body; serial Gauss-Seidel: of their indices), and the
// iterates depend on nothing else.  All schedules keep that order, so all give
// bitwise the same iterates: dependency levels or colours, one workgroup per
// scene (batched scenes), or lanes spread over many workgroups, whose merits
// meet once per sweep (a single large scene).
#pragma once
// (included inside namespace rbh by rbh_kernels.h)

// ------------------------------------------------------------ islands
__device__ __forceinline__ int uf_find(int* uf, int a) {
  while (true) {
    int p = __atomic_load_n(&uf[a], __ATOMIC_RELAXED);
    if (p == a) return a;
    int gp = __atomic_load_n(&uf[p], __ATOMIC_RELAXED);
    if (gp != p) atomicCAS(&uf[a], p, gp);   // path halving; parents only decrease
    a = p;
  }
}

__device__ __forceinline__ void uf_union(int* uf, int a, int b) {
  while (true) {
    a = uf_find(uf, a);
    b = uf_find(uf, b);
    if (a == b) return;
    if (a > b) { int t = a; a = b; b = t; }
    if (atomicCAS(&uf[b], b, a) == b) return;
  }
}

// reset at the start of the step (k_step_begin): body f's union-find parent
// and contact counters, island label l's counters, unit / sweep lane u
template <typename R> __device__ __forceinline__ void uf_reset(const Dev<R>& d, int f) {
  d.uf[f] = f;
  d.bc_cnt[f] = 0;
  d.bc_fill[f] = 0;
  d.body_claim[f] = -1;
}

template <typename R> __device__ __forceinline__ void isl_reset(const Dev<R>& d, int l) {
  d.isl_cnt[l] = 0;
  d.isl_fill[l] = 0;
}

template <typename R> __global__ void k_uf_union(Dev<R> d) {
  if (aborted(d.err)) return;
  const int nk = *d.n_contacts;
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nk; k += gridDim.x * blockDim.x) {
    int A = d.c_ia[k], B = d.c_ib[k];
    if (!d.b_fixed[A] && !d.b_fixed[B]) uf_union(d.uf, d.b2f[A], d.b2f[B]);
  }
}

// island label: flat root f -> f + bs (scene bs's labels are contiguous);
// contacts without a free body share the extra label bs_foff[bs + 1] + bs
template <typename R> __device__ __forceinline__ int contact_label(const Dev<R>& d, int k) {
  int A = d.c_ia[k], B = d.c_ib[k];
  int f = -1;
  if (!d.b_fixed[A]) f = uf_find(d.uf, d.b2f[A]);
  else if (!d.b_fixed[B]) f = uf_find(d.uf, d.b2f[B]);
  if (f >= 0) return f + d.f_bs[f];
  int bs = d.f_bs[d.b2f[A]];
  return d.bs_foff[bs + 1] + bs;
}

// ctr[key] += 1 for every active lane of the wavefront; returns the lane's
// old value (its slot).  The lanes that share the first active lane's key
// (on a batch scene of one island: the whole wavefront) take one atomic
// together and ranks among themselves; the others add on their own.  An
// island's contacts counted or placed one atomic each serialised in one L2
// channel.  (Slots within one key come in no fixed order; the callers'
// results do not depend on it.)
__device__ __forceinline__ int wave_add_one(int* ctr, int key, bool active) {
  const int lane = (int)(threadIdx.x & 63);
  const unsigned long long act = __ballot(active);
  if (!act) return 0;
  const int first = __ffsll((unsigned long long)act) - 1;
  const int k0 = __shfl(key, first, 64);
  const unsigned long long m = __ballot(active && key == k0);
  int base = 0;
  if (lane == first) base = atomicAdd(&ctr[k0], __popcll(m));
  base = __shfl(base, first, 64);
  if ((m >> lane) & 1ull) return base + __popcll(m & ((1ull << lane) - 1ull));
  return active ? atomicAdd(&ctr[key], 1) : 0;
}

// one contact per lane; the loop runs while any lane of the wavefront has one
template <typename R> __global__ void k_isl_count(Dev<R> d) {
  if (aborted(d.err)) return;
  const int nk = *d.n_contacts;
  const int lane = (int)(threadIdx.x & 63), stride = (int)(gridDim.x * blockDim.x);
  for (int k0 = (int)(blockIdx.x * blockDim.x + (threadIdx.x & ~63u)); k0 < nk; k0 += stride) {
    const int k = k0 + lane;
    const bool act = k < nk;
    int lab = 0;
    if (act) {
      lab = contact_label(d, k);
      d.c_lab[k] = lab;
    }
    (void)wave_add_one(d.isl_cnt, lab, act);
  }
}

template <typename R> __global__ void k_isl_fill(Dev<R> d) {
  if (aborted(d.err)) return;
  const int nk = *d.n_contacts;
  const int lane = (int)(threadIdx.x & 63), stride = (int)(gridDim.x * blockDim.x);
  for (int k0 = (int)(blockIdx.x * blockDim.x + (threadIdx.x & ~63u)); k0 < nk; k0 += stride) {
    const int k = k0 + lane;
    const bool act = k < nk;
    const int lab = act ? d.c_lab[k] : 0;
    const int slot = wave_add_one(d.isl_fill, lab, act);
    if (act) d.uperm[d.isl_off[lab] + slot] = k;
  }
}

// Colouring units of batch scene bs: windows of unit_T contact positions; an
// island joins the window its first position falls in.  Sweep lanes: the
// same with windows of TL_s = unit_T, or, when unit_split > 0, at least
// ceil(K_s / unit_split) positions, so that a scene solved by one workgroup
// has about one lane per wavefront.  Both are unions of whole islands.
template <typename R> __device__ __forceinline__ void scene_pos_range(const Dev<R>& d, int bs, int& p0, int& p1) {
  p0 = d.isl_off[d.bs_foff[bs] + bs];
  p1 = d.isl_off[d.bs_foff[bs + 1] + bs + 1];
}

template <typename R> __global__ void k_unit_count(Dev<R> d) {
  for (int bs = blockIdx.x * blockDim.x + threadIdx.x; bs < d.ns; bs += gridDim.x * blockDim.x) {
    int p0, p1;
    scene_pos_range(d, bs, p0, p1);
    int K = aborted(d.err) ? 0 : p1 - p0;
    int T = d.unit_T, TL = T;
    if (d.unit_split > 0) TL = max(T, (K + d.unit_split - 1) / d.unit_split);
    d.u_cnt[bs] = (K + T - 1) / T;
    d.u_T[bs] = TL;
    d.l_cnt[bs] = (K + TL - 1) / TL;
  }
}

// k_unit_count and the exclusive sums of the scenes' unit and lane counts
// (u_base, l_base with the totals n_units, n_lanes) in one workgroup, one
// launch instead of three, for batches of up to UNIT_SCAN_MAX scenes.
constexpr int UNIT_SCAN_MAX = 8192;

template <typename R> __global__ void __launch_bounds__(SCAN_BLOCK) k_unit_count_scan(Dev<R> d) {
  __shared__ int sh[SCAN_BLOCK / 64];
  const bool ab = aborted(d.err);
  int cu = 0, cl = 0;
  // base <= ns: the tile that holds u_base[ns] and l_base[ns] (the totals) runs
  for (int base = 0; base <= d.ns; base += SCAN_BLOCK) {
    const int bs = base + (int)threadIdx.x;
    int uc = 0, lc = 0;
    if (bs < d.ns) {
      int p0, p1;
      scene_pos_range(d, bs, p0, p1);
      const int K = ab ? 0 : p1 - p0;
      const int T = d.unit_T;
      int TL = T;
      if (d.unit_split > 0) TL = max(T, (K + d.unit_split - 1) / d.unit_split);
      uc = (K + T - 1) / T;
      lc = (K + TL - 1) / TL;
      d.u_cnt[bs] = uc;
      d.u_T[bs] = TL;
      d.l_cnt[bs] = lc;
    }
    int tu, tl;
    const int eu = block_exclusive_scan(uc, sh, tu);
    const int el = block_exclusive_scan(lc, sh, tl);
    if (bs <= d.ns) {
      d.u_base[bs] = cu + eu;
      d.l_base[bs] = cl + el;
    }
    cu += tu;
    cl += tl;
  }
  if (threadIdx.x == 0) {
    *d.n_units = cu;
    *d.n_lanes = cl;
  }
}

template <typename R> __device__ __forceinline__ void unit_reset(const Dev<R>& d, int u) {
  d.u_start[u] = 0x7fffffff;
  d.u_end[u] = 0;
  d.u_ncol[u] = 0;
  d.u_bs[u] = -1;
  d.u_nbody[u] = 0;
  d.l_start[u] = 0x7fffffff;
  d.l_end[u] = 0;
  d.l_bs[u] = -1;
}

template <typename R> __global__ void k_unit_assign(Dev<R> d) {
  if (aborted(d.err)) return;
  const int nu = *d.n_units;
  if (nu > d.cap_units) {
    if (blockIdx.x == 0 && threadIdx.x == 0) { atomicOr(d.err, ERR_CAP_UNITS); atomicMax(d.err + 5, nu); }
    return;
  }
  const int nl = d.nb + d.ns;
  for (int lab = blockIdx.x * blockDim.x + threadIdx.x; lab < nl; lab += gridDim.x * blockDim.x) {
    int cnt = d.isl_cnt[lab];
    if (cnt == 0) continue;
    // batch scene of the label: largest bs with bs_foff[bs] + bs <= lab
    int lo = 0, hi = d.ns - 1;
    while (lo < hi) {
      int mid = (lo + hi + 1) >> 1;
      if (d.bs_foff[mid] + mid <= lab) lo = mid; else hi = mid - 1;
    }
    int bs = lo;
    int p0, p1;
    scene_pos_range(d, bs, p0, p1);
    int start = d.isl_off[lab];
    int j = min(d.u_cnt[bs] - 1, (start - p0) / d.unit_T);
    int u = d.u_base[bs] + j;
    atomicMin(&d.u_start[u], start);
    atomicMax(&d.u_end[u], start + cnt);
    d.u_bs[u] = bs;
    d.isl_unit[lab] = u;
    int jl = min(d.l_cnt[bs] - 1, (start - p0) / d.u_T[bs]);
    int l = d.l_base[bs] + jl;
    atomicMin(&d.l_start[l], start);
    atomicMax(&d.l_end[l], start + cnt);
    d.l_bs[l] = bs;
  }
}

// Free bodies with contacts lie in exactly one island, so in one unit; each
// gets a slot in its unit (where its velocity change lives while the unit is
// solved; the slot order changes no result).
template <typename R> __global__ void k_unit_bodies(Dev<R> d) {
  if (aborted(d.err) || *d.n_units > d.cap_units) return;
  for (int f = blockIdx.x * blockDim.x + threadIdx.x; f < d.nb; f += gridDim.x * blockDim.x) {
    if (d.bc_cnt[f] == 0) { d.f_loc[f] = -1; continue; }
    int root = uf_find(d.uf, f);
    int u = d.isl_unit[root + d.f_bs[root]];
    d.f_unit[f] = u;
    d.f_loc[f] = atomicAdd(&d.u_nbody[u], 1);
  }
}

template <typename R> __global__ void k_unit_blist(Dev<R> d) {
  if (aborted(d.err) || *d.n_units > d.cap_units) return;
  for (int f = blockIdx.x * blockDim.x + threadIdx.x; f < d.nb; f += gridDim.x * blockDim.x) {
    int l = d.f_loc[f];
    if (l >= 0) d.u_blist[d.u_boff[d.f_unit[f]] + l] = d.bb_body[f];
  }
}

// body -> unit-order positions of its contacts (free bodies only)
template <typename R> __global__ void k_csr_count(Dev<R> d) {
  if (aborted(d.err)) return;
  const int nk = *d.n_contacts;
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < nk; p += gridDim.x * blockDim.x) {
    int k = d.uperm[p];
    int A = d.c_ia[k], B = d.c_ib[k];
    if (!d.b_fixed[A]) atomicAdd(&d.bc_cnt[d.b2f[A]], 1);
    if (!d.b_fixed[B]) atomicAdd(&d.bc_cnt[d.b2f[B]], 1);
  }
}

template <typename R> __global__ void k_csr_fill(Dev<R> d) {
  if (aborted(d.err)) return;
  const int nk = *d.n_contacts;
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < nk; p += gridDim.x * blockDim.x) {
    int k = d.uperm[p];
    int A = d.c_ia[k], B = d.c_ib[k];
    if (!d.b_fixed[A]) { int f = d.b2f[A]; d.bc_list[d.bc_off[f] + atomicAdd(&d.bc_fill[f], 1)] = p; }
    if (!d.b_fixed[B]) { int f = d.b2f[B]; d.bc_list[d.bc_off[f] + atomicAdd(&d.bc_fill[f], 1)] = p; }
  }
}

// ------------------------------------------------------------ colouring
// Vivace random colouring per island (proximal_contact/blocking.py:62-111 in
// the deterministic form of oracle/coloring.py).  Node = contact; two
// contacts are adjacent if they share a free body.  Units of up to
// SMALL_UNIT contacts are coloured by one wavefront with the palettes in LDS
// (SMALL_PW words per contact) and, per free body of the unit, bitmaps of the
// colours its contacts drew and won, so that a round costs O(palette words)
// per contact; larger units (and small ones whose palettes or bitmaps would
// not fit) by a workgroup of eight wavefronts, palettes in global memory
// (PALW words per contact; colours of an island stay below twice its size),
// the neighbours found through the bodies' contact lists, the rest of the
// state in LDS up to UNIT_CAP contacts (gfx950: 160 KB of LDS per
// workgroup), in global memory beyond.
constexpr int COLOR_BLOCK = 256;
constexpr int COLOR_UNIT_BLOCK = 512;   // threads colouring one large unit (8 wavefronts)
constexpr int UNIT_CAP = 4096;        // contacts of a large unit staged in LDS
constexpr int LIST_CAP = 8192;        // body-list entries staged in LDS
constexpr int SMALL_UNIT = 256;
constexpr int SMALL_BODY = 32;        // bodies with at most this many contacts are checked entry by entry
constexpr int BODY_BITS = 512;        // words of each per-body colour bitmap array of a small unit
constexpr int SMALL_PW = 4;           // palette words per contact of a small unit (colours below 128)
constexpr int PAIR_HASH = 2 * SMALL_UNIT;   // body-pair table of a small unit's set-up (power of two)
constexpr unsigned short NO_SLOT = 0xffff;

// State of a small unit coloured through per-body colour bitmaps (about 14 KB,
// so that many units share a CU).  Body b of the unit (its slot f_loc) owns
// words [b * bw, (b + 1) * bw) of each bitmap array, bw = palette words in use.
struct BitsColorLds {
  int key[SMALL_UNIT];                // contact index within its scene (draws, ranks)
  int isl[SMALL_UNIT];                // island label
  unsigned short la[SMALL_UNIT], lb[SMALL_UNIT];   // unit slots of the free bodies (NO_SLOT: fixed)
  unsigned short col[SMALL_UNIT], pc[SMALL_UNIT];
  unsigned char done[SMALL_UNIT];     // 0 uncoloured, 1 coloured, 2 won this round
  unsigned pal[SMALL_UNIT * SMALL_PW];
  union {
    struct { unsigned seen[BODY_BITS], dup[BODY_BITS], won[BODY_BITS]; } m;   // rounds
    struct { int cnt[2 * SMALL_UNIT]; unsigned hk[PAIR_HASH]; int hc[PAIR_HASH]; } s;   // set-up
  } u;
  int mx, cmax;
};
static_assert(sizeof(BitsColorLds::u.s) <= sizeof(BitsColorLds::u.m), "set-up tables share the bitmaps' space");

template <int NT, int CAP, int LCAP, int PAL> struct ColorLds {
  // colours a palette can hold (at most PALMAX in either palette layout)
  static constexpr int CC = PALMAX;
  int key[CAP];                       // contact index within its scene (random draws, ranks)
  int fa[CAP], fb[CAP];               // free flat bodies (-1 if fixed)
  unsigned short ao[CAP], ac[CAP], bo[CAP], bcn[CAP];
  unsigned short col[CAP];
  unsigned short pc[CAP];             // palette sizes
  unsigned char done[CAP];            // 0 uncoloured, 1 coloured, 2 won this round
  unsigned short list[LCAP];
  // bodies with more than SMALL_BODY contacts (each holds that many list entries): their lists
  unsigned short bl_off[LCAP / (SMALL_BODY + 1) + 1], bl_cnt[LCAP / (SMALL_BODY + 1) + 1];
  unsigned short ent_off[LCAP], ent_cnt[LCAP]; // per list entry of a smaller body: that body's list (cnt 0: larger body)
  unsigned char lose[CAP];            // drew a colour that another contact of one of its bodies drew
  unsigned seen[NT / 64][CC / 32];    // per wavefront, at the body in hand: colours drawn ...
  unsigned dup[NT / 64][CC / 32];     // ... drawn twice (conflict check), or won (palette removal)
  int nbody;
  unsigned pal[PAL > 0 ? PAL : 1];    // palettes (PAL > 0)
  int nlist, flag, cnt, mx;
  int sh[NT / 64];
};

// colouring state in LDS (unit fits) ...
template <typename S> struct LdsAcc {
  static constexpr bool PER_BODY = true;
  S* s;
  const int* c_lab; const int* uperm; int p0;   // island labels (read only when palettes run empty)
  __device__ int key(int i) const { return s->key[i]; }
  __device__ int isl(int i) const { return c_lab[uperm[p0 + i]]; }
  __device__ int col(int i) const { return s->col[i]; }
  __device__ void set_col(int i, int c) { s->col[i] = (unsigned short)c; }
  __device__ int done(int i) const { return s->done[i]; }
  __device__ void set_done(int i, int v) { s->done[i] = (unsigned char)v; }
  __device__ int pc(int i) const { return s->pc[i]; }
  __device__ void set_pc(int i, int v) { s->pc[i] = (unsigned short)v; }
  __device__ void dec_pc(int i) { atomicSub(reinterpret_cast<unsigned*>(&s->pc[i & ~1]), (i & 1) ? 0x10000u : 1u); }
  // (unrolled so that the list reads of several neighbours are in flight together)
  template <typename F> __device__ void nb(int i, F&& fn) const {
    int fa = s->fa[i];
#pragma unroll 8
    for (int e = s->ao[i], n = s->ao[i] + s->ac[i]; e < n; ++e) { int j = s->list[e]; if (j != i) fn(j); }
#pragma unroll 8
    for (int e = s->bo[i], n = s->bo[i] + s->bcn[i]; e < n; ++e) {
      int j = s->list[e];
      if (j == i) continue;
      if (fa >= 0 && (s->fa[j] == fa || s->fb[j] == fa)) continue;   // met through the first body
      fn(j);
    }
  }
};

// ... or in global memory (unit larger than the LDS capacity)
template <typename R> struct GlbAcc {
  static constexpr bool PER_BODY = false;
  const Dev<R>* d;
  int p0;      // first unit-order position of the unit
  int k_off;   // first contact of the scene
  int* col_arr;
  __device__ int kk(int i) const { return d->uperm[p0 + i]; }
  __device__ int key(int i) const { return kk(i) - k_off; }
  __device__ int isl(int i) const { return d->c_lab[kk(i)]; }
  __device__ int col(int i) const { return col_arr[kk(i)]; }
  __device__ void set_col(int i, int c) { col_arr[kk(i)] = c; }
  __device__ int done(int i) const { return d->g_done[p0 + i]; }
  __device__ void set_done(int i, int v) { d->g_done[p0 + i] = (unsigned char)v; }
  __device__ int pc(int i) const { return d->g_pc[p0 + i]; }
  __device__ void set_pc(int i, int v) { d->g_pc[p0 + i] = v; }
  __device__ void dec_pc(int i) { atomicSub(&d->g_pc[p0 + i], 1); }
  __device__ int free_body(int k, bool second) const {
    int b = second ? d->c_ib[k] : d->c_ia[k];
    return d->b_fixed[b] ? -1 : d->b2f[b];
  }
  template <typename F> __device__ void nb(int i, F&& fn) const {
    int k = kk(i);
    int fa = free_body(k, false), fb = free_body(k, true);
    if (fa >= 0)
      for (int e = d->bc_off[fa], n = e + d->bc_cnt[fa]; e < n; ++e) { int j = d->bc_list[e] - p0; if (j != i) fn(j); }
    if (fb >= 0)
      for (int e = d->bc_off[fb], n = e + d->bc_cnt[fb]; e < n; ++e) {
        int j = d->bc_list[e] - p0;
        if (j == i) continue;
        if (fa >= 0) {
          int kj = d->uperm[p0 + j];
          if (free_body(kj, false) == fa || free_body(kj, true) == fa) continue;
        }
        fn(j);
      }
  }
};

// idx-th set bit of a palette of pw words, or -1
// (palettes of large units live in global memory and are changed by other
// wavefronts' atomics in L2: read them past the vector L1)
__device__ __forceinline__ unsigned pal_word(const unsigned* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ int pal_select(const unsigned* p, int pw, int idx) {
  for (int w = 0; w < pw; ++w) {
    const unsigned pwv = pal_word(p + w);
    int c = __popc(pwv);
    if (idx < c) {
      unsigned m = pwv;
      for (int i = 0; i < idx; ++i) m &= m - 1;   // drop the lowest set bits
      return w * 32 + __ffs(m) - 1;
    }
    idx -= c;
  }
  return -1;
}

// sum over the NT threads of a workgroup (sh: NT / 64 ints)
template <int NT> __device__ __forceinline__ int block_sum(int v, int* sh) {
  v = wave_sum(v);
  if (NT == 64) return v;
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  int tot = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) tot += sh[w];
  __syncthreads();
  return tot;
}

// rounds of blocking.py:78-104 over the K contacts of one unit by NT threads;
// pal: pw words per contact
template <int NT, typename R, typename A>
__device__ void color_rounds(const Dev<R>& d, A& a, int K, unsigned* pal, int pw, unsigned long long seed,
                             unsigned long long stepk, int* sh, int* s_flag, int* s_mx) {
  const int pcap = 32 * pw;
  // words of the palettes that can hold a colour: up to the largest degree,
  // raised when an empty palette grows (kept in *s_mx until the rounds end)
  if (threadIdx.x == 0) *s_mx = 0;
  if constexpr (A::PER_BODY) {
    auto* S = a.s;
    constexpr int CW = sizeof(S->seen[0]) / sizeof(unsigned);
    for (int k = threadIdx.x & 63; k < CW; k += 64) { S->seen[threadIdx.x >> 6][k] = 0; S->dup[threadIdx.x >> 6][k] = 0; }
  }
  __syncthreads();
  // palettes {0, ..., deg-1}
  for (int i = threadIdx.x; i < K; i += NT) {
    int deg = 0;
    a.nb(i, [&](int) { ++deg; });
    if (deg > 0) atomicMax(s_mx, min(deg, pcap));
    if constexpr (A::PER_BODY) a.s->lose[i] = 0;
    unsigned* p = pal + (size_t)i * pw;
    for (int w = 0; w < pw; ++w) {
      int lo = w * 32;
      unsigned m = 0;
      if (deg >= lo + 32) m = 0xffffffffu;
      else if (deg > lo) m = (1u << (deg - lo)) - 1u;
      p[w] = m;
    }
    if (deg > pcap) atomicOr(d.err, ERR_COLORS);
    a.set_pc(i, min(deg, pcap));
    a.set_col(i, 0);
    a.set_done(i, 0);
  }
  __syncthreads();
  int pwe = (*s_mx + 31) / 32;   // palette words in use
  int rnd = 0;
  for (; rnd < MAX_ROUNDS; ++rnd) {
    int left = 0;
    for (int i = threadIdx.x; i < K; i += NT) {
      if (a.done(i)) continue;
      ++left;
      int n = a.pc(i);
      if (n > 0)
        a.set_col(i, pal_select(pal + (size_t)i * pw, pwe,
                                (int)color_draw(seed, stepk, (unsigned long long)a.key(i), (unsigned long long)rnd, (unsigned)n)));
    }
    if (block_sum<NT>(left, sh) == 0) break;
    __syncthreads();
    // keep the draw if no uncoloured neighbour drew the same colour
    if constexpr (A::PER_BODY) {
      // neighbours are the contacts sharing a free body: a draw is lost when
      // another uncoloured contact of one of its bodies drew the same colour.
      // Wavefronts take whole bodies and sweep their contact lists 64 at a time.
      auto* S = a.s;
      const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, pwr = max(pwe, 1);
      unsigned* seen = S->seen[w];
      unsigned* dup = S->dup[w];
      // smaller bodies: every list entry compares its draw with its body's others
      for (int e = threadIdx.x; e < S->nlist; e += NT) {
        const int cnt = S->ent_cnt[e];
        if (!cnt) continue;
        const int j = S->list[e];
        if (a.done(j)) continue;
        const int c = a.col(j), o = S->ent_off[e];
        for (int e2 = o; e2 < o + cnt; ++e2) {
          const int j2 = S->list[e2];
          if (j2 != j && !a.done(j2) && a.col(j2) == c) { S->lose[j] = 1; break; }
        }
      }
      // larger bodies: a wavefront per body
      for (int b = w; b < S->nbody; b += NT / 64) {
        const int off = S->bl_off[b], n = S->bl_cnt[b];
        for (int e = lane; e < n; e += 64) {
          const int j = S->list[off + e];
          if (a.done(j)) continue;
          const int c = a.col(j);
          const unsigned bit = 1u << (c & 31);
          if (atomicOr(&seen[c >> 5], bit) & bit) atomicOr(&dup[c >> 5], bit);
        }
        wave_sync_lds();
        for (int e = lane; e < n; e += 64) {
          const int j = S->list[off + e];
          if (a.done(j)) continue;
          const int c = a.col(j);
          if (dup[c >> 5] & (1u << (c & 31))) S->lose[j] = 1;
        }
        wave_sync_lds();
        for (int k = lane; k < pwr; k += 64) { seen[k] = 0; dup[k] = 0; }
        wave_sync_lds();
      }
      __syncthreads();
      for (int i = threadIdx.x; i < K; i += NT) {
        if (a.done(i)) continue;
        if (!S->lose[i]) a.set_done(i, 2);
        S->lose[i] = 0;
      }
    } else {
      for (int i = threadIdx.x; i < K; i += NT) {
        if (a.done(i)) continue;
        int ci = a.col(i);
        bool ok = true;
        a.nb(i, [&](int j) { if (a.done(j) != 1 && a.col(j) == ci) ok = false; });
        if (ok) a.set_done(i, 2);
      }
    }
    __syncthreads();
    // winners leave their colour out of the palettes of neighbours uncoloured
    // at round start (no-return atomics: nothing waits on them) ...
    if constexpr (A::PER_BODY) {
      // per body: the colours won by its contacts leave the palettes of its
      // uncoloured contacts (a winner's own palette is no longer read)
      auto* S = a.s;
      const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, pwr = max(pwe, 1);
      unsigned* won = S->dup[w];
      // smaller bodies: every uncoloured list entry clears the colours won by its body's others
      for (int e = threadIdx.x; e < S->nlist; e += NT) {
        const int cnt = S->ent_cnt[e];
        if (!cnt) continue;
        const int j = S->list[e];
        if (a.done(j)) continue;
        const int o = S->ent_off[e];
        for (int e2 = o; e2 < o + cnt; ++e2) {
          const int j2 = S->list[e2];
          if (a.done(j2) != 2) continue;
          const int c = a.col(j2);
          (void)__hip_atomic_fetch_and(&pal[(size_t)j * pw + (c >> 5)], ~(1u << (c & 31)), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      // larger bodies: a wavefront per body
      for (int b = w; b < S->nbody; b += NT / 64) {
        const int off = S->bl_off[b], n = S->bl_cnt[b];
        bool any = false;
        for (int e = lane; e < n; e += 64) {
          const int j = S->list[off + e];
          if (a.done(j) != 2) continue;
          const int c = a.col(j);
          atomicOr(&won[c >> 5], 1u << (c & 31));
          any = true;
        }
        if (!__ballot(any)) continue;
        wave_sync_lds();
        for (int e = lane; e < n; e += 64) {
          const int j = S->list[off + e];
          if (a.done(j)) continue;
          for (int k = 0; k < pwr; ++k) {
            const unsigned m = won[k];
            if (m) (void)__hip_atomic_fetch_and(&pal[(size_t)j * pw + k], ~m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        }
        wave_sync_lds();
        for (int k = lane; k < pwr; k += 64) won[k] = 0;
        wave_sync_lds();
      }
    } else {
      for (int i = threadIdx.x; i < K; i += NT) {
        if (a.done(i) != 2) continue;
        int ci = a.col(i);
        unsigned bit = 1u << (ci & 31);
        a.nb(i, [&](int j) {
          if (a.done(j) != 1)
            (void)__hip_atomic_fetch_and(&pal[(size_t)j * pw + (ci >> 5)], ~bit, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
        });
      }
    }
    __syncthreads();
    // ... and the palette sizes of contacts still uncoloured are recounted
    // (a size always equals its palette's popcount)
    for (int i = threadIdx.x; i < K; i += NT) {
      if (a.done(i)) continue;
      const unsigned* p = pal + (size_t)i * pw;
      int n = 0;
      for (int w = 0; w < pwe; ++w) n += __popc(pal_word(p + w));
      a.set_pc(i, n);
    }
    __syncthreads();
    // commit winners
    if (threadIdx.x == 0) *s_flag = 0;
    __syncthreads();
    int moving = 0;   // a winner, or an uncoloured node whose next draw is not forced
    for (int i = threadIdx.x; i < K; i += NT) {
      if (a.done(i) == 2) { a.set_done(i, 1); moving = 1; }
      if (!a.done(i) && a.pc(i) == 0) atomicOr(s_flag, 1);
      if (!a.done(i) && a.pc(i) != 1) moving = 1;
    }
    __syncthreads();
    // No winner and every uncoloured palette a single colour: every later
    // round draws the same colours and keeps none, so the rounds up to
    // MAX_ROUNDS would change nothing; go to the leftovers directly.
    if (block_sum<NT>(moving, sh) == 0) { rnd = MAX_ROUNDS; break; }
    if (*s_flag) {
      // rare: empty palettes get max+1, max+2, ... in increasing contact order
      // per island (max over the island's kept and tentative colours); ranks
      // read only done/pc/isl/key, which stay fixed here
      for (int i = threadIdx.x; i < K; i += NT) d.isl_max[a.isl(i)] = -1;
      __syncthreads();
      for (int i = threadIdx.x; i < K; i += NT) atomicMax(&d.isl_max[a.isl(i)], a.col(i));
      __syncthreads();
      for (int i = threadIdx.x; i < K; i += NT) {
        if (a.done(i) || a.pc(i) != 0) continue;
        int il = a.isl(i), ki = a.key(i), rank = 0;
        for (int j = 0; j < K; ++j)
          if (j != i && !a.done(j) && a.pc(j) == 0 && a.isl(j) == il && a.key(j) < ki) ++rank;
        int c = d.isl_max[il] + 1 + rank;
        if (c >= pcap) { atomicOr(d.err, ERR_COLORS); continue; }
        (void)__hip_atomic_fetch_or(&pal[(size_t)i * pw + (c >> 5)], 1u << (c & 31), __ATOMIC_RELAXED,
                                    __HIP_MEMORY_SCOPE_AGENT);
        atomicMax(s_mx, c + 1);
      }
      __syncthreads();
      pwe = (*s_mx + 31) / 32;
      for (int i = threadIdx.x; i < K; i += NT)
        if (!a.done(i) && a.pc(i) == 0) a.set_pc(i, 1);
      __syncthreads();
    }
  }
  if (rnd >= MAX_ROUNDS) {
    // leftovers get fresh colours max+1, ... in increasing contact order per island
    for (int i = threadIdx.x; i < K; i += NT) d.isl_max[a.isl(i)] = -1;
    __syncthreads();
    for (int i = threadIdx.x; i < K; i += NT) atomicMax(&d.isl_max[a.isl(i)], a.col(i));
    __syncthreads();
    for (int i = threadIdx.x; i < K; i += NT) {
      if (a.done(i)) continue;
      int il = a.isl(i), ki = a.key(i), rank = 0;
      for (int j = 0; j < K; ++j)
        if (j != i && !a.done(j) && a.isl(j) == il && a.key(j) < ki) ++rank;
      int c = d.isl_max[il] + 1 + rank;
      if (c >= pcap) atomicOr(d.err, ERR_COLORS);
      a.set_col(i, min(c, pcap - 1));
    }
    __syncthreads();
  }
  int mx = 0;
  for (int i = threadIdx.x; i < K; i += NT) mx = max(mx, a.col(i) + 1);
  if (threadIdx.x == 0) *s_mx = 0;
  __syncthreads();
  atomicMax(s_mx, mx);
  __syncthreads();
}

// one unit by NT threads with the state S in LDS (global fallback when its
// body lists do not fit)
template <typename R, int NT, int CAP, int LCAP, int PAL>
__device__ void color_unit(const Dev<R>& d, int u, ColorLds<NT, CAP, LCAP, PAL>& s) {
  const int p0 = d.u_start[u], p1 = d.u_end[u];
  const int bs = d.u_bs[u];
  const int slot = d.bs_slot[bs];
  const SceneParams& sp = d.sp[slot];
  const SceneState& st = d.ss[slot];
  const int K = p1 - p0;
  if (sp.scheme == SCHEME_GS) {   // the reference's serial order: contact i is colour i
    for (int i = threadIdx.x; i < K; i += NT) {
      int k = d.uperm[p0 + i];
      d.c_color[k] = k - st.k_off;
    }
    if (threadIdx.x == 0) { d.u_ncol[u] = 0; atomicMax(&d.ss[slot].ncolor, st.k_cnt); }
    return;
  }
  const unsigned long long seed = sp.seed, stepk = (unsigned long long)st.step_index;
  bool fits = K <= min(CAP, d.color_cap);
  if (fits) {
    // stage contacts and the bodies' contact lists (claimed once per body)
    if (threadIdx.x == 0) { s.nlist = 0; s.flag = 0; s.nbody = 0; }
    __syncthreads();
    for (int i = threadIdx.x; i < K; i += NT) {
      int k = d.uperm[p0 + i];
      int A = d.c_ia[k], B = d.c_ib[k];
      int fa = d.b_fixed[A] ? -1 : d.b2f[A];
      int fb = d.b_fixed[B] ? -1 : d.b2f[B];
      s.key[i] = k - st.k_off;
      s.fa[i] = fa;
      s.fb[i] = fb;
      if (fa >= 0) atomicCAS(&d.body_claim[fa], -1, 2 * i);
      if (fb >= 0) atomicCAS(&d.body_claim[fb], -1, 2 * i + 1);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < K; i += NT) {
      for (int side = 0; side < 2; ++side) {
        int f = side ? s.fb[i] : s.fa[i];
        if (f < 0 || d.body_claim[f] != 2 * i + side) continue;
        int n = d.bc_cnt[f];
        int off = atomicAdd(&s.nlist, n);
        if (off + n > LCAP) { atomicOr(&s.flag, 1); continue; }
        for (int e = 0; e < n; ++e) s.list[off + e] = (unsigned short)(d.bc_list[d.bc_off[f] + e] - p0);
        d.body_loc[f] = make_int2(off, n);
        if (n > SMALL_BODY) {
          const int b = atomicAdd(&s.nbody, 1);   // such a body holds more than SMALL_BODY of the <= LCAP entries
          s.bl_off[b] = (unsigned short)off;
          s.bl_cnt[b] = (unsigned short)n;
        }
        for (int e = 0; e < n; ++e) {
          s.ent_off[off + e] = (unsigned short)off;
          s.ent_cnt[off + e] = (unsigned short)(n > SMALL_BODY ? 0 : n);
        }
      }
    }
    __threadfence_block();
    __syncthreads();
    fits = s.flag == 0;
    if (fits) {
      for (int i = threadIdx.x; i < K; i += NT) {
        int2 la = s.fa[i] >= 0 ? d.body_loc[s.fa[i]] : make_int2(0, 0);
        int2 lb = s.fb[i] >= 0 ? d.body_loc[s.fb[i]] : make_int2(0, 0);
        s.ao[i] = (unsigned short)la.x; s.ac[i] = (unsigned short)la.y;
        s.bo[i] = (unsigned short)lb.x; s.bcn[i] = (unsigned short)lb.y;
      }
      __syncthreads();
      LdsAcc<ColorLds<NT, CAP, LCAP, PAL>> a{&s, d.c_lab, d.uperm, p0};
      const int pw = (2 * K + 2 + 31) / 32;
      if (PAL > 0 && K * pw <= PAL)
        color_rounds<NT>(d, a, K, s.pal, pw, seed, stepk, s.sh, &s.flag, &s.mx);
      else
        color_rounds<NT>(d, a, K, d.pal + (size_t)p0 * PALW, PALW, seed, stepk, s.sh, &s.flag, &s.mx);
      for (int i = threadIdx.x; i < K; i += NT) d.c_color[d.uperm[p0 + i]] = s.col[i];
    }
  }
  if (!fits) {
    GlbAcc<R> a{&d, p0, st.k_off, d.c_color};
    color_rounds<NT>(d, a, K, d.pal + (size_t)p0 * PALW, PALW, seed, stepk, s.sh, &s.flag, &s.mx);
  }
  if (threadIdx.x == 0) {
    if (s.mx > 2 * K + 1) atomicOr(d.err, ERR_COLORS);   // beyond the lane's colour offset space
    d.u_ncol[u] = s.mx;
    atomicMax(&d.ss[slot].ncolor, s.mx);
  }
}

static_assert(sizeof(ColorLds<COLOR_UNIT_BLOCK, UNIT_CAP, LIST_CAP, 0>) <= 160 * 1024 - 2048,
              "large-unit colouring state must fit a workgroup's LDS");

// idx-th set bit of an LDS palette of pwe words (the draw's colour), or -1
__device__ __forceinline__ int lds_select(const unsigned* p, int pwe, int idx) {
  for (int w = 0; w < pwe; ++w) {
    unsigned m = p[w];
    const int c = __popc(m);
    if (idx < c) {   // halve the word until the bit is found
      int pos = 0, lo;
      lo = __popc(m & 0xffffu); if (idx >= lo) { idx -= lo; m >>= 16; pos += 16; }
      lo = __popc(m & 0xffu);   if (idx >= lo) { idx -= lo; m >>= 8; pos += 8; }
      lo = __popc(m & 0xfu);    if (idx >= lo) { idx -= lo; m >>= 4; pos += 4; }
      lo = __popc(m & 0x3u);    if (idx >= lo) { idx -= lo; m >>= 2; pos += 2; }
      if (idx >= (int)(m & 1u)) pos += 1;
      return w * 32 + pos;
    }
    idx -= c;
  }
  return -1;
}

__device__ __forceinline__ unsigned pair_hash(unsigned key) { return (key * 2654435761u) >> 23; }   // 9 bits

// The rounds of color_rounds for a unit of up to SMALL_UNIT contacts by one
// wavefront, with a contact's neighbours met through per-body bitmaps instead
// of its bodies' contact lists:
//  * degree = (contacts of body a - 1) + (contacts of body b - 1) - (other
//    contacts between a and b), from per-body counts and a body-pair table;
//  * a draw is lost iff one of its free bodies has the colour in `dup` (drawn
//    by two of its uncoloured contacts in this round);
//  * the colours won on either free body leave the palette of a contact still
//    uncoloured (its palette is read and written by its own lane only).
// The same draws, winners, palettes, fresh colours and leftovers as
// color_rounds, so the same colours.  Palettes hold colours below
// 32 SMALL_PW (leftovers may take larger ones: they need no palette).
// Returns false, having written nothing outside LDS, when the unit is not for
// this path (colouring state forced to global memory) or outgrows it (a
// palette colour of 32 SMALL_PW or more, bitmaps beyond color_bits words);
// color_unit then colours it from the start.
template <typename R>
__device__ bool color_small_bits(const Dev<R>& d, int u, BitsColorLds& s) {
  const int p0 = d.u_start[u], p1 = d.u_end[u], K = p1 - p0;
  const int bs = d.u_bs[u], slot = d.bs_slot[bs];
  const SceneParams& sp = d.sp[slot];
  const SceneState& st = d.ss[slot];
  const int nbu = d.u_nbody[u];
  const int lane = threadIdx.x;
  const int k_off = st.k_off;
  if (sp.scheme == SCHEME_GS) {   // the reference's serial order: contact i is colour i
    for (int i = lane; i < K; i += 64) {
      const int k = d.uperm[p0 + i];
      d.c_color[k] = k - k_off;
    }
    if (lane == 0) { d.u_ncol[u] = 0; atomicMax(&d.ss[slot].ncolor, st.k_cnt); }
    return true;
  }
  if (K > d.color_cap || nbu > 2 * SMALL_UNIT) return false;
  const unsigned long long seed = sp.seed, stepk = (unsigned long long)st.step_index;
  // pcap: the colour space of the unit's lanes (colours of an island stay
  // below twice its size); palettes here hold colours below 32 SMALL_PW
  constexpr int pw = SMALL_PW;
  const int pcap = 32 * ((2 * K + 2 + 31) / 32);
  const int cap = d.color_bits;
  unsigned* const raw = s.u.m.seen;   // the whole union as words
  for (int w = lane; w < 3 * BODY_BITS; w += 64) raw[w] = 0;
  if (lane == 0) { s.mx = 0; s.cmax = 0; }
  __syncthreads();
  // contacts: key, island, body slots; contacts per body and per body pair
  for (int i = lane; i < K; i += 64) {
    const int k = d.uperm[p0 + i];
    const int A = d.c_ia[k], B = d.c_ib[k];
    const int fa = d.b_fixed[A] ? -1 : d.b2f[A], fb = d.b_fixed[B] ? -1 : d.b2f[B];
    const int la = fa >= 0 ? d.f_loc[fa] : NO_SLOT, lb = fb >= 0 ? d.f_loc[fb] : NO_SLOT;
    s.key[i] = k - k_off;
    s.isl[i] = d.c_lab[k];
    s.la[i] = (unsigned short)la;
    s.lb[i] = (unsigned short)lb;
    if (la != NO_SLOT) atomicAdd(&s.u.s.cnt[la], 1);
    if (lb != NO_SLOT) atomicAdd(&s.u.s.cnt[lb], 1);
    if (la != NO_SLOT && lb != NO_SLOT) {
      const unsigned key = (((unsigned)min(la, lb) << 10) | (unsigned)max(la, lb)) + 1u;
      unsigned h = pair_hash(key);
      for (int t = 0; t < PAIR_HASH; ++t, h = (h + 1) & (PAIR_HASH - 1)) {
        const unsigned old = atomicCAS(&s.u.s.hk[h], 0u, key);
        if (old == 0u || old == key) { atomicAdd(&s.u.s.hc[h], 1); break; }
      }
    }
  }
  __syncthreads();
  // palettes {0, ..., deg - 1}
  for (int i = lane; i < K; i += 64) {
    const int la = s.la[i], lb = s.lb[i];
    int deg = 0;
    if (la != NO_SLOT) deg += s.u.s.cnt[la] - 1;
    if (lb != NO_SLOT) deg += s.u.s.cnt[lb] - 1;
    if (la != NO_SLOT && lb != NO_SLOT) {
      const unsigned key = (((unsigned)min(la, lb) << 10) | (unsigned)max(la, lb)) + 1u;
      unsigned h = pair_hash(key);
      for (int t = 0; t < PAIR_HASH; ++t, h = (h + 1) & (PAIR_HASH - 1))
        if (s.u.s.hk[h] == key) { deg -= s.u.s.hc[h] - 1; break; }
    }
    if (deg > 0) atomicMax(&s.mx, deg);
    unsigned* p = s.pal + i * pw;
    for (int w = 0; w < pw; ++w) {
      const int lo = w * 32;
      p[w] = deg >= lo + 32 ? 0xffffffffu : deg > lo ? (1u << (deg - lo)) - 1u : 0u;
    }
    s.pc[i] = (unsigned short)deg;
    s.col[i] = 0;
    s.done[i] = 0;
  }
  __syncthreads();
  for (int w = lane; w < 3 * BODY_BITS; w += 64) raw[w] = 0;
  int pwe = (s.mx + 31) / 32;   // palette words in use
  __syncthreads();
  if (pwe > pw || nbu * max(pwe, 1) > cap) return false;
  unsigned* const seen = s.u.m.seen;
  unsigned* const dup = s.u.m.dup;
  unsigned* const won = s.u.m.won;
  int rnd = 0;
  for (; rnd < MAX_ROUNDS; ++rnd) {
    const int bw = max(pwe, 1);
    // last round's winners are coloured; draws; the colours drawn on each body
    for (int w = lane; w < nbu * bw; w += 64) won[w] = 0;
    int left = 0;
    for (int i = lane; i < K; i += 64) {
      const int dn = s.done[i];
      if (dn == 2) s.done[i] = 1;
      if (dn) continue;
      ++left;
      int c = s.col[i];
      const int n = s.pc[i];
      if (n > 0) {
        c = lds_select(s.pal + i * pw, pwe, (int)color_draw(seed, stepk, (unsigned long long)s.key[i],
                                                             (unsigned long long)rnd, (unsigned)n));
        s.col[i] = (unsigned short)c;
      }
      if (c < 0 || c >= 32 * bw) continue;   // only after a colour-space overflow (ERR_COLORS)
      const unsigned bit = 1u << (c & 31);
      const int la = s.la[i], lb = s.lb[i];
      if (la != NO_SLOT) { const int w = la * bw + (c >> 5); if (atomicOr(&seen[w], bit) & bit) atomicOr(&dup[w], bit); }
      if (lb != NO_SLOT) { const int w = lb * bw + (c >> 5); if (atomicOr(&seen[w], bit) & bit) atomicOr(&dup[w], bit); }
    }
    if (!__any(left)) break;
    __syncthreads();
    // a draw is kept if no other uncoloured contact of either body drew it
    int win = 0;
    for (int i = lane; i < K; i += 64) {
      if (s.done[i]) continue;
      const int c = s.col[i];
      if (c >= 32 * bw) continue;
      const unsigned bit = 1u << (c & 31);
      const int la = s.la[i], lb = s.lb[i];
      const bool lose = (la != NO_SLOT && (dup[la * bw + (c >> 5)] & bit)) ||
                        (lb != NO_SLOT && (dup[lb * bw + (c >> 5)] & bit));
      if (lose) continue;
      s.done[i] = 2;
      win = 1;
      if (la != NO_SLOT) atomicOr(&won[la * bw + (c >> 5)], bit);
      if (lb != NO_SLOT) atomicOr(&won[lb * bw + (c >> 5)], bit);
    }
    __syncthreads();
    // the colours won on its bodies leave the palette of a contact still
    // uncoloured, whose size is recounted
    int moving = win, empty = 0;
    for (int i = lane; i < K; i += 64) {
      if (s.done[i]) continue;
      const int la = s.la[i], lb = s.lb[i];
      unsigned* p = s.pal + i * pw;
      int n = 0;
      for (int w = 0; w < pwe; ++w) {
        unsigned m = 0;
        if (la != NO_SLOT) m |= won[la * bw + w];
        if (lb != NO_SLOT) m |= won[lb * bw + w];
        const unsigned v = p[w] & ~m;
        p[w] = v;
        n += __popc(v);
      }
      s.pc[i] = (unsigned short)n;
      if (n == 0) empty = 1;
      if (n != 1) moving = 1;
    }
    for (int w = lane; w < nbu * bw; w += 64) { seen[w] = 0; dup[w] = 0; }
    // No winner and every uncoloured palette a single colour: every later
    // round draws the same colours and keeps none; go to the leftovers.
    if (!__any(moving)) { rnd = MAX_ROUNDS; break; }
    __syncthreads();
    if (__any(empty)) {
      // empty palettes get max+1, max+2, ... in increasing contact order per
      // island (max over the island's kept and tentative colours)
      for (int i = lane; i < K; i += 64) {
        if (s.done[i] || s.pc[i] != 0) continue;
        const int il = s.isl[i], ki = s.key[i];
        int mx = -1, rank = 0;
        for (int j = 0; j < K; ++j) {
          if (s.isl[j] != il) continue;
          mx = max(mx, (int)s.col[j]);
          if (j != i && !s.done[j] && s.pc[j] == 0 && s.key[j] < ki) ++rank;
        }
        const int c = mx + 1 + rank;
        if (c >= pcap) { atomicOr(d.err, ERR_COLORS); continue; }
        if (c >= 32 * pw) { atomicMax(&s.mx, c + 1); continue; }   // beyond these palettes: start over below
        s.pal[i * pw + (c >> 5)] |= 1u << (c & 31);
        atomicMax(&s.mx, c + 1);
      }
      __syncthreads();
      for (int i = lane; i < K; i += 64)
        if (!s.done[i] && s.pc[i] == 0) s.pc[i] = 1;
      pwe = (s.mx + 31) / 32;
      __syncthreads();
      if (pwe > pw || nbu * max(pwe, 1) > cap) return false;
    }
  }
  if (rnd >= MAX_ROUNDS) {
    // leftovers get fresh colours max+1, ... in increasing contact order per
    // island.  The wavefront walks the (few) leftover contacts together; for
    // each, every lane checks the unit's contacts it holds, and a wavefront max
    // and sum give the island's largest colour (kept or tentative) and the
    // leftover's rank.  (A walk over the whole unit by every leftover's lane
    // made the wavefront run K iterations whenever one contact was left.)
    __syncthreads();
    constexpr int QS = SMALL_UNIT / 64;
    int fresh[QS], il_q[QS], col_q[QS], key_q[QS];
    bool left_q[QS];
#pragma unroll
    for (int q = 0; q < QS; ++q) {
      const int i = lane + 64 * q;
      const bool in = i < K;
      fresh[q] = -1;
      il_q[q] = in ? s.isl[i] : -1;
      col_q[q] = in ? (int)s.col[i] : -1;
      key_q[q] = in ? s.key[i] : 0;
      left_q[q] = in && !s.done[i];
    }
#pragma unroll
    for (int q = 0; q < QS; ++q) {
      unsigned long long m = __ballot(left_q[q]);
      while (m) {                                   // (uniform over the wavefront)
        const int b = __ffsll(m) - 1;
        m &= m - 1;
        const int i = 64 * q + b;
        const int il = s.isl[i], ki = s.key[i];
        int mx = -1, rank = 0;
#pragma unroll
        for (int r = 0; r < QS; ++r) {
          if (il_q[r] != il) continue;              // (-1: no contact)
          mx = max(mx, col_q[r]);
          if (left_q[r] && key_q[r] < ki) ++rank;   // keys are distinct: i itself is not counted
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          mx = max(mx, __shfl_xor(mx, o, 64));
          rank += __shfl_xor(rank, o, 64);
        }
        if (lane == b) fresh[q] = mx + 1 + rank;
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < SMALL_UNIT / 64; ++q) {
      if (fresh[q] < 0) continue;
      if (fresh[q] >= pcap) atomicOr(d.err, ERR_COLORS);
      s.col[lane + 64 * q] = (unsigned short)min(fresh[q], pcap - 1);
    }
    __syncthreads();
  }
  int mx = 0;
  for (int i = lane; i < K; i += 64) {
    mx = max(mx, s.col[i] + 1);
    d.c_color[s.key[i] + k_off] = s.col[i];
  }
  atomicMax(&s.cmax, mx);
  __syncthreads();
  if (lane == 0) {
    if (s.cmax > 2 * K + 1) atomicOr(d.err, ERR_COLORS);   // beyond the lane's colour offset space
    d.u_ncol[u] = s.cmax;
    atomicMax(&d.ss[slot].ncolor, s.cmax);
  }
  return true;
}

// units of up to SMALL_UNIT contacts: one wavefront each, through per-body
// bitmaps; larger units, and those outgrowing the bitmaps, are listed in
// big_list for k_color_units
// (grids of the per-unit and per-lane kernels are capped, and a workgroup
// walks units or lanes in turn: a grid of cap_units workgroups, almost all of
// them without work, costs ~1 ns per workgroup to dispatch)
template <typename R> __global__ void __launch_bounds__(64) k_color_small(Dev<R> d) {
  __shared__ BitsColorLds s;
  if (aborted(d.err)) return;
  const int nu = *d.n_units;
  for (int u = blockIdx.x; u < nu; u += gridDim.x) {
    const int K = d.u_end[u] - d.u_start[u];
    if (K <= 0) continue;
    if ((K > SMALL_UNIT || !color_small_bits<R>(d, u, s)) && threadIdx.x == 0)
      d.big_list[1 + atomicAdd(&d.big_list[0], 1)] = u;
    __syncthreads();   // s is reused by the next unit
  }
}

// the listed units: a workgroup of COLOR_UNIT_BLOCK threads each (a grid of
// at most one workgroup per CU walks the list), neighbours through the
// bodies' contact lists
template <typename R> __global__ void __launch_bounds__(COLOR_UNIT_BLOCK) k_color_units(Dev<R> d) {
  __shared__ ColorLds<COLOR_UNIT_BLOCK, UNIT_CAP, LIST_CAP, 0> s;
  if (aborted(d.err)) return;
  const int n = d.big_list[0];
  for (int i = blockIdx.x; i < n; i += gridDim.x) {
    color_unit<R>(d, d.big_list[1 + i], s);
    __syncthreads();
  }
}

template <typename R> struct ContactRow {
  V3<R> lin[4], angA[4], angB[4];
};

template <typename R>
__device__ __forceinline__ void contact_rows(V4<R> n4, V4<R> rA4, V4<R> rB4, ContactRow<R>& J) {
  V3<R> s, t, n;
  orthonormal_frame(xyz(n4), s, t, n);
  V3<R> rA = xyz(rA4), rB = xyz(rB4);
  J.lin[0] = n; J.lin[1] = s; J.lin[2] = t; J.lin[3] = V3<R>{R(0), R(0), R(0)};
  J.angA[0] = cross(rA, n); J.angA[1] = cross(rA, s); J.angA[2] = cross(rA, t); J.angA[3] = n;
  J.angB[0] = cross(rB, n); J.angB[1] = cross(rB, s); J.angB[2] = cross(rB, t); J.angB[3] = n;
}

// ------------------------------------------------------------ sweep order
// A contact's record in sweep order (s_rec): row r of J at r * ROW as (lin_r,
// b_r | angA_r, r0_r | angB_r, mu_r), both iterates, and the LDS addresses of
// its bodies' records (written by the solve).  mu_1..3 are the friction
// coefficients; under the isotropic projection every row's mu_r is mu_1, the
// only one it reads.  The record after the last contact's stays zero: the null
// contact, which a quad without a contact updates to no effect.
template <typename R> struct Rec {
  static constexpr int ROW = 12 * (int)sizeof(R);
  static constexpr int X0 = 4 * ROW, X1 = X0 + 4 * (int)sizeof(R), LOC = X1 + 4 * (int)sizeof(R);
  static constexpr int BYTES = (LOC + 16 + 4 * (int)sizeof(R) - 1) / (4 * (int)sizeof(R)) * (4 * (int)sizeof(R));
};
static_assert(Rec<float>::BYTES == 240 && Rec<double>::BYTES == 480, "records are whole vec4s");
// 32-bit offsets reach every record of c contacts and the null one
template <typename R> __host__ __device__ constexpr bool rec_addressable(int c) {
  return c < (1 << 24) && ((unsigned long long)c + 1) * Rec<R>::BYTES < (1ull << 32);
}

constexpr int PHASE_Q = 16;      // quads of a wavefront: contacts per phase of a wavefront's sweep
constexpr int PHASE_R = 4;       // rows of 16 lanes of a wavefront: contacts per phase of a narrow lane's sweep
constexpr int LANE_WG = 1, LANE_NARROW = 2, LANE_BITS = 2;   // low bits of l_nph: streamed by the workgroup; narrow if resident
constexpr int PHASE_BITS = 8;    // low bits of an entry of l_phase: contacts of the phase (at most 128); the rest: its first position
// most phases of a lane of K contacts in nc levels: a level of w > 0 contacts
// takes ceil(w / 16) <= 1 + (w - 1) / 16
__device__ __forceinline__ int lane_phases(int K, int nc) { return min(K, nc + K / PHASE_Q); }

__device__ __forceinline__ int wave_inclusive_sum(int v) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(v, o, 64);
    if ((int)(threadIdx.x & 63) >= o) v += y;
  }
  return v;
}

// A free body's slot (index into u_blist); -1 for a fixed one.
template <typename R> __device__ __forceinline__ int body_slot(const Dev<R>& d, int b) {
  if (d.b_fixed[b]) return -1;
  const int f = d.b2f[b];
  return d.u_boff[d.f_unit[f]] + d.f_loc[f];
}

// Gather one contact into the solver arrays at position `pos`; s_loc holds
// the bodies' slots (index into u_blist; -1 for a fixed body).
// ITEMS: also the per-contact items of the global layout
template <typename R> __device__ __forceinline__ void gather_contact(const Dev<R>& d, int pos, int k, bool items, bool iso) {
  const V4<R> mu = d.c_mu[k];
  const V4<R> n = d.c_n[k], rA = d.c_rA[k], rB = d.c_rB[k];
  const int A = d.c_ia[k], B = d.c_ib[k];
  const bool fa = !d.b_fixed[A], fb = !d.b_fixed[B];
  const int sa = body_slot(d, A), sb = body_slot(d, B);
  d.perm[pos] = k;
  d.s_loc[pos] = make_int2(sa, sb);
  if (items) {
    d.s_id[pos] = make_int2(A, B);
    d.s_n[pos] = V4<R>{n.x, n.y, n.z, mu.x};
    d.s_rA[pos] = V4<R>{rA.x, rA.y, rA.z, mu.y};
    d.s_rB[pos] = V4<R>{rB.x, rB.y, rB.z, mu.z};
    d.s_b[pos] = d.c_b[k];
    d.s_r0[pos] = d.c_r0[k];
    const V4<R> z = {R(0), R(0), R(0), R(0)};
    V4<R>* W = d.s_W + 4 * (size_t)pos;
    W[0] = fa ? d.b_W0[A] : z;
    W[1] = fa ? d.b_W1[A] : z;
    W[2] = fb ? d.b_W0[B] : z;
    W[3] = fb ? d.b_W1[B] : z;
    d.x0[pos] = z;
    d.x1[pos] = z;
  }
  // the contact's record, for the quad sweeps
  using X = Rec<R>;
  ContactRow<R> J;
  contact_rows(V4<R>{n.x, n.y, n.z, R(0)}, rA, rB, J);
  const V4<R> bb = d.c_b[k], r0 = d.c_r0[k];
  const R bv[4] = {bb.x, bb.y, bb.z, bb.w}, rv[4] = {r0.x, r0.y, r0.z, r0.w};
  const R mv[4] = {iso ? mu.x : R(0), mu.x, iso ? mu.x : mu.y, iso ? mu.x : mu.z};
  unsigned char* rec = d.s_rec + (size_t)pos * X::BYTES;
  V4<R>* row = reinterpret_cast<V4<R>*>(rec);
  R* x = reinterpret_cast<R*>(rec + X::X0);
  for (int r = 0; r < 4; ++r) {
    row[3 * r] = V4<R>{J.lin[r].x, J.lin[r].y, J.lin[r].z, bv[r]};
    row[3 * r + 1] = V4<R>{J.angA[r].x, J.angA[r].y, J.angA[r].z, rv[r]};
    row[3 * r + 2] = V4<R>{J.angB[r].x, J.angB[r].y, J.angB[r].z, mv[r]};
    x[r] = R(0);
    x[4 + r] = R(0);
  }
}

// steppers.py:15-36 with constraints/post_stabilization.py:21-41, 99-104: the
// post-stabilisation problem keeps the contact problem's rows (J, W J^T and
// r = 1/diag) and sweep order; its right-hand side is the gap of a contact
// deeper than min_gap_value on the normal row and 0 elsewhere, its friction
// rows are projected to zero (mu = 0), and it starts from x = 0.  Rewrites
// the sweep-order arrays of every layout in place (the contact solve is done
// with them) and flags the scenes that have something to correct.
template <typename R> __global__ void k_post_rows(Dev<R> d) {
  if (aborted(d.err)) return;
  const int nk = *d.n_contacts;
  if (nk > d.cap_contacts) return;
  for (int pos = blockIdx.x * blockDim.x + threadIdx.x; pos < nk; pos += gridDim.x * blockDim.x) {
    const int k = d.perm[pos];
    const int slot = d.b_slot[d.c_ia[k]];
    const SceneParams& sp = d.sp[slot];
    if (!sp.use_post_stab) continue;
    const R g = d.c_p[k].w;
    const bool deep = (double)g < -sp.min_gap;
    const R zero = R(0);
    d.s_b[pos] = V4<R>{deep ? g : zero, zero, zero, zero};
    V4<R> n = d.s_n[pos], ra = d.s_rA[pos], rb = d.s_rB[pos];
    n.w = zero; ra.w = zero; rb.w = zero;
    d.s_n[pos] = n; d.s_rA[pos] = ra; d.s_rB[pos] = rb;
    d.x0[pos] = V4<R>{zero, zero, zero, zero};
    d.x1[pos] = V4<R>{zero, zero, zero, zero};
    unsigned char* rec = d.s_rec + (size_t)pos * Rec<R>::BYTES;
    V4<R>* row = reinterpret_cast<V4<R>*>(rec);
    R* x = reinterpret_cast<R*>(rec + Rec<R>::X0);
    for (int r = 0; r < 4; ++r) {
      row[3 * r].w = (r == 0 && deep) ? g : zero;
      row[3 * r + 2].w = zero;
      x[r] = zero;
      x[4 + r] = zero;
    }
    if (deep) d.ss[slot].post_active = 1;
  }
}

// state_storage.py:251-302 with dt = 1 and u = W J^T sol of the
// post-stabilisation problem (steppers.py:33-36): positions only.
template <typename R> __global__ void k_post_integrate(Dev<R> d) {
  const int f = blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= d.nb || aborted(d.err)) return;
  const int b = d.bb_body[f];
  if (d.b_fixed[b]) return;
  const int slot = d.b_slot[b];
  if (!(d.sp[slot].use_post_stab && d.ss[slot].post_active)) return;
  const R one = R(1);
  const V4<R> s0 = d.ws0[b], s1 = d.ws1[b];
  V4<R> r = d.r[b];
  r.x = r.x + s0.x * one; r.y = r.y + s0.y * one; r.z = r.z + s0.z * one;
  Quat<R> q = quat(d.q[b]);
  Quat<R> dq = qprod(Quat<R>{R(0), s1.x, s1.y, s1.z}, q);
  Quat<R> qn = {q.s + dq.s * one * R(0.5), q.x + dq.x * one * R(0.5), q.y + dq.y * one * R(0.5),
                q.z + dq.z * one * R(0.5)};
  qn = qunit(qn);
  d.r[b] = r;
  d.q[b] = V4<R>{qn.s, qn.x, qn.y, qn.z};
}

// level or colour offsets of lane l: 2 K_l + 2 entries (an island's colours stay below
// twice its size, which the colouring checks)
template <typename R> __device__ __forceinline__ const int* lane_coff(const Dev<R>& d, int l) {
  return d.col_off + 2 * ((size_t)d.l_start[l] + l);
}

// State of k_order_lanes (28 KB: five workgroups per CU)
constexpr int ORD_CAP = 2048;      // most contacts of a lane put in dependency levels
constexpr int ORD_BODY = 2046;     // most body slots a lane's contacts may span for it
constexpr unsigned ORD_FIXED = ORD_BODY;   // slot of a fixed body: stays at level 0 (its updates go to the next one)
struct OrderLds {
  int cnt[PALMAX + 1];             // contacts per colour, then the next free position; then the same per level
  unsigned ab[ORD_CAP];            // in colour order: the two bodies' slots (low and high half; ORD_FIXED: fixed)
  unsigned short ord[ORD_CAP];     // in colour order: the contact's unit-order index in the lane
  unsigned short lev[ORD_CAP + 1]; // in colour order: its level
  unsigned short last[ORD_BODY + 2];   // per body slot: level of its last contact so far
  int nc, smin, smax;
};

// exclusive prefix sum of s.cnt[0..n) in place by wavefront 0, copied to coff[0..n] with the total
__device__ __forceinline__ void order_scan(OrderLds& s, int n, int* coff) {
  if (threadIdx.x < 64) {
    int acc = 0;
    for (int c0 = 0; c0 < n; c0 += 64) {
      const int c = c0 + (int)threadIdx.x;
      const int v = c < n ? s.cnt[c] : 0;
      const int x = wave_inclusive_sum(v);
      if (c < n) { coff[c] = acc + x - v; s.cnt[c] = acc + x - v; }
      acc += __shfl(x, 63, 64);
    }
    if (threadIdx.x == 0) coff[n] = acc;
  }
}

// sum over the levels of ceil(width / per), in every lane of the wavefront
__device__ __forceinline__ int count_phases(int nl, const int* coff, int per) {
  const int lane = (int)threadIdx.x & 63;
  int n = 0;
  for (int c = lane; c < nl; c += 64) n += (coff[c + 1] - coff[c] + per - 1) / per;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
  return n;
}

// Whether a resident lane is swept with 16 lanes a contact instead of 4, a
// quarter of the contacts per phase: a row's phase takes about 0.8 of a quad's
// (440 cycles against 550), so it may take up to 5/4 as many.
__device__ __forceinline__ bool narrow_phases(int wide, int narrow) { return 4 * narrow <= 5 * wide; }

// The lane's phases for the streaming sweep, by wavefront 0: at most 16 contacts
// of one level for a wavefront's sweep, a contact per quad of the workgroup for
// the workgroup's.  One wavefront takes about nl / 2 + K / 16 phases, the
// workgroup nl / 2 + K / 64 of about 1.4 times the length (its barrier), but
// only one lane at a time: worth it from levels of 8 contacts on when the group
// has one lane, and 8 times as many as wavefronts it would leave idle.
template <typename R>
__device__ __forceinline__ void order_phases(const Dev<R>& d, int l, int nl, const int* coff) {
  if (threadIdx.x >= 64) return;
  const int p0 = d.l_start[l], K = d.l_end[l] - p0, lane = (int)threadIdx.x;
  const int lanes = d.unit_split > 0 ? min(d.l_cnt[d.l_bs[l]], d.solve_quads / PHASE_Q) : 1;
  const bool wg = K > 8 * lanes * nl;
  const int per = wg ? d.solve_quads : PHASE_Q;
  const bool narrow = narrow_phases(count_phases(nl, coff, PHASE_Q), count_phases(nl, coff, PHASE_R));
  int ph = 0;
  for (int c0 = 0; c0 < nl; c0 += 64) {
    const int c = c0 + lane;
    const int lo = c < nl ? coff[c] : 0, w = c < nl ? coff[c + 1] - lo : 0;
    const int np = (w + per - 1) / per;
    const int inc = wave_inclusive_sum(np);
    unsigned* out = d.l_phase + p0 + ph + inc - np;
    for (int i = 0; i < np; ++i) out[i] = (unsigned)(lo + i * per) << PHASE_BITS | (unsigned)min(per, w - i * per);
    ph += __shfl(inc, 63, 64);
  }
  if (lane == 0)
    d.l_nph[l] = ph << LANE_BITS | (narrow ? LANE_NARROW : 0) | (wg ? LANE_WG : 0);
}

// One workgroup per sweep lane: its positions [l_start, l_end) in sweep order.
//
// The iterates depend only on the order in which each body's contacts are
// solved: by colour, or for the reference's serial Gauss-Seidel by contact
// index.  A lane is therefore swept by dependency level -- a contact's level
// is one more than the highest level of the earlier contacts of its two free
// bodies -- which keeps every body's order (so the iterates are bitwise the
// same) in as few phases as that order allows: the colours of a random
// colouring leave gaps at every body (an island of 677 contacts in a
// 1,500-sphere pile has 114 colours, 93 of them with contacts, and 79 levels;
// one of 1,255 in 48 meshes 345, 306 and 268), and serial Gauss-Seidel has
// one "colour" per contact.  Levels are found by one wavefront walking the
// colours (about 260 cycles each) over LDS tables; a lane too large for them
// keeps its colours.  l_ncol and the colour offsets then count levels.
template <typename R> __device__ __forceinline__ void order_lane(const Dev<R>& d, int l, OrderLds& s) {
  const int p0 = d.l_start[l], p1 = d.l_end[l];
  if (p1 <= p0) return;
  const int K = p1 - p0;
  const bool serial = d.sp[d.bs_slot[d.l_bs[l]]].scheme == SCHEME_GS;
  int* coff = d.col_off + 2 * ((size_t)p0 + l);
  if (threadIdx.x == 0) { s.nc = 0; s.smin = 0x7fffffff; s.smax = -1; }
  __syncthreads();
  int mx = 0, lo = 0x7fffffff, hi = -1;
  for (int i = threadIdx.x; i < K; i += COLOR_BLOCK) {
    const int k = d.uperm[p0 + i];
    if (!serial) mx = max(mx, d.c_color[k] + 1);
    const int a = body_slot(d, d.c_ia[k]), b = body_slot(d, d.c_ib[k]);
    if (a >= 0) { lo = min(lo, a); hi = max(hi, a); }
    if (b >= 0) { lo = min(lo, b); hi = max(hi, b); }
  }
  atomicMax(&s.nc, mx);
  atomicMin(&s.smin, lo);
  atomicMax(&s.smax, hi);
  __syncthreads();
  const int nc = serial ? K : s.nc, s0 = s.smin;
  const bool levels = K <= ORD_CAP && (s.smax < 0 || s.smax - s0 < ORD_BODY);
  // positions by colour: a counting sort (the order inside a colour changes no
  // result), or the contact's rank
  if (!serial) {
    for (int c = threadIdx.x; c <= nc; c += COLOR_BLOCK) s.cnt[c] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < K; i += COLOR_BLOCK) atomicAdd(&s.cnt[d.c_color[d.uperm[p0 + i]]], 1);
    __syncthreads();
    order_scan(s, nc, coff);
    __syncthreads();
  }
  for (int i = threadIdx.x; i < K; i += COLOR_BLOCK) {
    const int k = d.uperm[p0 + i];
    int pos;
    if (serial) {
      pos = 0;
      for (int j = 0; j < K; ++j) pos += d.uperm[p0 + j] < k ? 1 : 0;
      if (!levels) coff[pos] = pos;
    } else {
      pos = atomicAdd(&s.cnt[d.c_color[k]], 1);
    }
    if (levels) {
      const int a = body_slot(d, d.c_ia[k]), b = body_slot(d, d.c_ib[k]);
      s.ab[pos] = (a >= 0 ? (unsigned)(a - s0) : ORD_FIXED) | ((b >= 0 ? (unsigned)(b - s0) : ORD_FIXED) << 16);
      s.ord[pos] = (unsigned short)i;
    } else {
      d.l_pos[p0 + i] = pos;
    }
  }
  if (!levels) {
    if (threadIdx.x == 0) { coff[nc] = K; d.l_ncol[l] = nc; }
    __threadfence_block();
    __syncthreads();
    order_phases(d, l, nc, coff);
    return;
  }
  for (int i = threadIdx.x; i <= (int)ORD_FIXED; i += COLOR_BLOCK) s.last[i] = 0;
  __threadfence_block();
  __syncthreads();
  // levels (from 1), colour after colour; contacts of one colour share no free body
  if (threadIdx.x < 64) {
    const int lane = (int)threadIdx.x;
    int top = 0, q0 = 0, ends = 0;
    unsigned next = s.ab[min(lane, K - 1)];     // the next 64 contacts, read ahead
    for (int c = 0; c < nc; ++c) {
      if (!serial && (c & 63) == 0) ends = s.cnt[min(c + lane, nc - 1)];   // (after the sort: the ends of the colours)
      const int q1 = serial ? c + 1 : __builtin_amdgcn_readlane(ends, c & 63);
      while (q0 < q1) {   // (uniform; no branch on a lane's contact: idle lanes and fixed bodies use spare entries)
        const bool act = q0 + lane < q1;
        const unsigned ab = act ? next : (ORD_FIXED | ORD_FIXED << 16);
        const int a = (int)(ab & 0xffffu), b = (int)(ab >> 16);
        const int v = max(s.last[a], s.last[b]) + 1;
        const int q = act ? q0 + lane : ORD_CAP;
        q0 = min(q0 + 64, q1);
        next = s.ab[min(q0 + lane, K - 1)];
        s.last[a == ORD_FIXED ? ORD_FIXED + 1 : a] = (unsigned short)v;
        s.last[b == ORD_FIXED ? ORD_FIXED + 1 : b] = (unsigned short)v;
        s.lev[q] = (unsigned short)v;
        top = max(top, act ? v : 0);
        wave_sync_lds();
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = max(top, __shfl_xor(top, o, 64));
    if (threadIdx.x == 0) s.nc = top;
  }
  __syncthreads();
  const int nl = s.nc;
  for (int c = threadIdx.x; c <= nl; c += COLOR_BLOCK) s.cnt[c] = 0;
  __syncthreads();
  for (int q = threadIdx.x; q < K; q += COLOR_BLOCK) atomicAdd(&s.cnt[s.lev[q] - 1], 1);
  __syncthreads();
  order_scan(s, nl, coff);
  if (threadIdx.x == 0) d.l_ncol[l] = nl;
  __threadfence_block();
  __syncthreads();
  order_phases(d, l, nl, coff);
  // each contact's position, taken from LDS counters (the order inside a level
  // changes no result)
  for (int q = threadIdx.x; q < K; q += COLOR_BLOCK) d.l_pos[p0 + s.ord[q]] = atomicAdd(&s.cnt[s.lev[q] - 1], 1);
}

template <typename R> __global__ void __launch_bounds__(COLOR_BLOCK) k_order_lanes(Dev<R> d) {
  __shared__ OrderLds s;
  if (aborted(d.err)) return;
  const int nl = *d.n_lanes;
  for (int l = blockIdx.x; l < nl; l += gridDim.x) {
    order_lane(d, l, s);
    __syncthreads();   // s is reused by the next lane
  }
}

// Contacts into sweep order inside their lane, at the positions
// k_order_lanes gave them: GATHER_SPLIT workgroups per lane, each taking every
// GATHER_SPLIT-th run of COLOR_BLOCK positions.  (The positions used to be
// taken here with a global atomic per contact on the lane's per-colour
// counters, which sit in one or two cache lines: the atomics of a lane
// serialised in one L2 channel.)
constexpr int GATHER_SPLIT = 8;
template <typename R> __device__ void gather_lane(const Dev<R>& d, int l) {
  const int p0 = d.l_start[l], p1 = d.l_end[l];
  if (p1 <= p0) return;
  // the items only where the global layout may read them: a group too large
  // for the velocity-only layout, or the post-stabilisation rows
  const int bs = d.l_bs[l];
  const bool iso = d.sp[d.bs_slot[bs]].friction != 1;
  bool items = d.items_nb < 0 || d.sp[d.bs_slot[bs]].use_post_stab;
  if (!items) {
    const int u0 = d.u_base[bs];
    items = d.u_boff[u0 + d.u_cnt[bs]] - d.u_boff[u0] > d.items_nb;
  }
  for (int i = blockIdx.y * COLOR_BLOCK + threadIdx.x; i < p1 - p0; i += GATHER_SPLIT * COLOR_BLOCK) {
    gather_contact(d, p0 + d.l_pos[p0 + i], d.uperm[p0 + i], items, iso);
  }
}

template <typename R> __global__ void __launch_bounds__(COLOR_BLOCK) k_lane_gather(Dev<R> d) {
  if (aborted(d.err)) return;
  const int nl = *d.n_lanes;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < Rec<R>::BYTES / 16)   // the null contact's record
    reinterpret_cast<int4*>(d.s_rec + (size_t)d.cap_contacts * Rec<R>::BYTES)[threadIdx.x] = make_int4(0, 0, 0, 0);
  for (int l = blockIdx.x; l < nl; l += gridDim.x) gather_lane(d, l);
}

// ------------------------------------------------------------ solve
// A workgroup solves a group of sweep lanes: the lanes of one batch scene, or
// a block of the lanes of a single scene spread over a cooperative grid (the
// scene-wide merit then meets in a grid barrier once per sweep).  A group's
// bodies are the slot range [b_lo, b_hi) of u_blist.  Three layouts, chosen
// per group:
//  * resident: everything a sweep touches -- contact records, the lanes'
//    schedules, the bodies' velocity changes and inverse masses -- is staged
//    in LDS once per solve; each wavefront sweeps its own lanes level by level
//    with wavefront-level syncs, and a sweep issues no global memory access;
//  * streaming: the bodies in LDS, contact records read from global memory two
//    phases ahead; a lane with wide levels is swept by the whole workgroup;
//  * global: everything in global memory, lanes swept by the whole workgroup.
// The sweep order inside an island is the same in every layout and schedule,
// so all of them give bitwise the same iterates.
constexpr int SOLVE_BLOCK = 256;
// The scene parameters the friction projection reads, taken into registers
// once per solve: a reference into the scene table would be read again from
// memory after every colour phase's fence.
struct ProxParams {
  double ell_tol, ell_expansion;
  int friction, ell_max_iter;
  __device__ explicit ProxParams(const SceneParams& sp)
      : ell_tol(sp.ell_tol), ell_expansion(sp.ell_expansion), friction(sp.friction), ell_max_iter(sp.ell_max_iter) {}
};

// One row of J w (lin, angA, angB: the row's blocks).  FP64 keeps the
// oracle's sum of four dot products; FP32 sums side A and side B in two
// chains of fused multiply-adds.
template <typename R>
__device__ __forceinline__ R row_jw(V3<R> lin, V3<R> angA, V3<R> angB, V3<R> wlA, V3<R> waA, V3<R> wlB, V3<R> waB) {
  if constexpr (sizeof(R) == 8) {
    return -dot(lin, wlA) - dot(angA, waA) + dot(lin, wlB) + dot(angB, waB);
  } else {
    R a = lin.x * wlA.x;
    a = madd(lin.y, wlA.y, a); a = madd(lin.z, wlA.z, a);
    a = madd(angA.x, waA.x, a); a = madd(angA.y, waA.y, a); a = madd(angA.z, waA.z, a);
    R b = lin.x * wlB.x;
    b = madd(lin.y, wlB.y, b); b = madd(lin.z, wlB.z, b);
    b = madd(angB.x, waB.x, b); b = madd(angB.y, waB.y, b); b = madd(angB.z, waB.z, b);
    return b - a;
  }
}

// z = x - r (J w + b) for one row: xo - r (Jw + b)
template <typename R> __device__ __forceinline__ R row_z(R xo, R r, R jw, R b) { return madd(-r, jw + b, xo); }

// contacts.py:77-95: z = x - r (J w + b); x_n = max(0, z_n); friction prox
template <typename R>
__device__ __forceinline__ V4<R> contact_prox(const ProxParams& pp, const ContactRow<R>& J, V4<R> xo, V4<R> bb,
                                              V4<R> rr, V4<R> mu, V3<R> wlA, V3<R> waA, V3<R> wlB, V3<R> waB,
                                              bool use_old_xn) {
  R Jw[4];
  for (int i = 0; i < 4; ++i) Jw[i] = row_jw(J.lin[i], J.angA[i], J.angB[i], wlA, waA, wlB, waB);
  R z0 = row_z(xo.x, rr.x, Jw[0], bb.x);
  R z1 = row_z(xo.y, rr.y, Jw[1], bb.y);
  R z2 = row_z(xo.z, rr.z, Jw[2], bb.z);
  R z3 = row_z(xo.w, rr.w, Jw[3], bb.w);
  R xn = fmax(R(0), z0);
  R xr = use_old_xn ? xo.x : xn;
  R os, ot, orr;
  if (pp.friction == 1) {
    const V3<R> o = prox_ellipsoid_call<R>(z1, z2, z3, mu.x, mu.y, mu.z, xr, pp.ell_tol, pp.ell_expansion, pp.ell_max_iter);
    os = o.x; ot = o.y; orr = o.z;
  } else {
    prox_sphere<R>(z1, z2, z3, mu.x, xr, os, ot, orr);
  }
  return V4<R>{xn, os, ot, orr};
}

// w += W J^T dx for one body (contacts.py:107); W0 = (I^-1 xx, yy, zz, xy),
// W1 = (I^-1 xz, yz, 1/m, 0); l, g: linear and angular parts of w
template <typename R>
__device__ __forceinline__ void dw_body(V4<R> W0, V4<R> W1, R sign, const ContactRow<R>& J, const V3<R>* ang,
                                        V4<R> dx, V4<R>& l, V4<R>& g) {
  const R im = W1.z;
  const R W[6] = {W0.x, W0.y, W0.z, W0.w, W1.x, W1.y};
  const R dd[4] = {dx.x, dx.y, dx.z, dx.w};
  const R s0 = sign * dd[0];
  R dl[3] = {sum_first(J.lin[0].x * s0), sum_first(J.lin[0].y * s0), sum_first(J.lin[0].z * s0)};
  V3<R> a = {sum_first(s0 * ang[0].x), sum_first(s0 * ang[0].y), sum_first(s0 * ang[0].z)};
  for (int i = 1; i < 4; ++i) {
    const R s = sign * dd[i];
    dl[0] = madd(J.lin[i].x, s, dl[0]); dl[1] = madd(J.lin[i].y, s, dl[1]); dl[2] = madd(J.lin[i].z, s, dl[2]);
    a = V3<R>{madd(s, ang[i].x, a.x), madd(s, ang[i].y, a.y), madd(s, ang[i].z, a.z)};
  }
  const V3<R> da = sym_madd(W, a);
  l = V4<R>{madd(im, dl[0], l.x), madd(im, dl[1], l.y), madd(im, dl[2], l.z), R(0)};
  g = V4<R>{g.x + da.x, g.y + da.y, g.z + da.z, R(0)};
}

__device__ __forceinline__ double absmax4(double a, double b, double c, double e) {
  return fmax(fmax(fabs(a), fabs(b)), fmax(fabs(c), fabs(e)));
}

// one step of a maximum over a wavefront: v against the lane DPP control CTRL names
template <int CTRL, int ROWS = 0xf> __device__ __forceinline__ double dpp_max(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  const int l = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xf, false);
  const int h = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xf, false);
  return fmax(v, __hiloint2double(h, l));
}

// largest v of a wavefront, in every lane.  By DPP: within the rows of 16
// lanes by xor 1, xor 2, half-row and row mirror, then row 0 into 1 and 2
// into 3, then the lower half into the upper (through LDS, as __shfl_xor
// does it, the six steps cost ~900 cycles, three times as much).
__device__ __forceinline__ double wave_max(double v) {
  v = dpp_max<0xb1>(v);          // quad_perm 1, 0, 3, 2
  v = dpp_max<0x4e>(v);          // quad_perm 2, 3, 0, 1
  v = dpp_max<0x141>(v);         // row_half_mirror
  v = dpp_max<0x140>(v);         // row_mirror
  v = dpp_max<0x142, 0xa>(v);    // row_bcast 15 into rows 1 and 3
  v = dpp_max<0x143, 0xc>(v);    // row_bcast 31 into rows 2 and 3
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                          __builtin_amdgcn_readlane(__double2loint(v), 63));
}

__device__ __forceinline__ double block_max(double v, double* sh) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  v = wave_max(v);
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  double m = 0.0;
  for (int i = 0; i < (int)(blockDim.x >> 6); ++i) m = fmax(m, sh[i]);
  __syncthreads();
  return m;
}

// the scene parameters of the accept/reject driver, taken into registers once
// per solve
struct CtlParams {
  double nu_reduce, nu_increase, too_small, abs_tol, rel_tol;
  __device__ explicit CtlParams(const SceneParams& sp)
      : nu_reduce(sp.nu_reduce), nu_increase(sp.nu_increase), too_small(sp.too_small), abs_tol(sp.abs_tol),
        rel_tol(sp.rel_tol) {}
};

// gauss_seidel_solver.py:56-97: accept/reject, r-factor, stopping tests.
struct SolveCtl {
  double last_merit = INFINITY, glast = INFINITY, rscale = 1.0, gm = 0.0;
  int acc = 0, rejects = 0, exitcode = 0, iters = 0, sweeps = 0;
  // accept (bit0) or reject, r-factor update; gm = this problem's contribution
  // to the global merit (its merit, or its last accepted merit on a reject)
  __device__ int accept_or_reject(const CtlParams& sp, double merit) {
    int dec = 0;
    if (merit > last_merit) {
      rscale *= sp.nu_reduce;
      gm = fmax(0.0, last_merit);
      ++rejects;
    } else {
      dec |= 1;
      if (last_merit - merit < sp.too_small) rscale *= sp.nu_increase;
      last_merit = merit;
      gm = fmax(0.0, merit);
    }
    return dec;
  }
  // returns bit0 accept, bit1 stop; `other` is the contribution of the
  // scene's other problem (the hinges) to the global merit of this sweep
  __device__ int decide(const CtlParams& sp, double merit, double* res, int it, double other = 0.0) {
    int dec = accept_or_reject(sp, merit);
    gm = fmax(gm, other);
    if (res) res[it] = gm;
    if (gm < sp.abs_tol) { dec |= 2; exitcode = 1; }
    else if (fabs(gm - glast) < sp.rel_tol * glast) { dec |= 2; exitcode = 2; }
    glast = gm;
    ++sweeps;
    if (dec & 1) acc ^= 1;
    return dec;
  }
};

// the hinge problem's contributions to the sweeps (recorded before the contact
// solve; gauss_seidel_solver.py:47-73 takes the largest over the problems), or
// null
template <typename R> __device__ __forceinline__ const double* hinge_merits(const Dev<R>& d, const SceneParams& sp) {
  return (sp.h_cnt > 0 && !d.post) ? d.h_mer + sp.res_off : nullptr;
}

// the scene's per-sweep merit record: the contact solve's 'residuals', then
// the post-stabilisation solve's 'post_stabilization_residuals'
// (gauss_seidel_solver.py:29-33, 76 with prefix; max_iter entries each)
template <typename R> __device__ __forceinline__ double* residual_record(const Dev<R>& d, const SceneParams& sp) {
  return d.residuals + sp.res_off + (d.post ? max(1, sp.max_iter) : 0);
}

template <typename R> __device__ void write_solve_state(const Dev<R>& d, SceneState& st, const SolveCtl& c) {
  if (d.post) {   // the post-stabilisation solve keeps the contact solve's record
    st.post_iters = c.iters;
    st.post_exit = c.exitcode;
    return;
  }
  st.solved = 1;
  st.iterations = c.iters;
  st.exitcode = c.exitcode;
  st.rejects = c.rejects;
  st.sweeps = c.sweeps;
  st.final_merit = c.last_merit;
}

// The scene-wide merit of sweep `it` in a cooperative launch, which is also
// the sweep's grid barrier.  Workgroup b publishes its merit in slot
// it * G + b: the bits of the non-negative double, or 0 for a merit that is
// not > 0 (a maximum that starts from 0 ignores it).  The slots start as all
// ones, which no published value is.  Wavefront 0 then waits until the
// sweep's G slots are all published and takes their maximum.  Workgroups
// share no other data during the solve, so the slots need no fences.  The
// wait is bounded: it flags ERR_SOLVER and returns false instead of hanging.
// (called by wavefront 0 alone, merit the same in all its lanes)
__device__ __forceinline__ bool grid_merit(unsigned long long* slots, int it, double& merit, int* err) {
  const unsigned G = gridDim.x;
  if (G == 1) return true;
  unsigned long long* row = slots + (size_t)it * G;
  if (threadIdx.x == 0)
    __hip_atomic_store(&row[blockIdx.x], merit > 0.0 ? (unsigned long long)__double_as_longlong(merit) : 0ull,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  double m = 0.0;
  bool ok = true;
  for (unsigned j = threadIdx.x; j < G && ok; j += 64) {
    unsigned long long v = __hip_atomic_load(&row[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (unsigned spins = 0; v == ~0ull;) {
      __builtin_amdgcn_s_sleep(1);
      if (++spins > (1u << 26)) { ok = false; break; }
      v = __hip_atomic_load(&row[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (ok) m = fmax(m, __longlong_as_double((long long)v));
  }
  merit = wave_max(m);
  const bool all_ok = __ballot(!ok) == 0;
  if (threadIdx.x == 0 && !all_ok) atomicOr(err, ERR_SOLVER);
  return all_ok;
}

// The merit of sweep `it` over the workgroup's threads (v each) and, in a
// cooperative launch, over the grid; false if the grid's wait failed.  lone:
// only wavefront 0 swept, so it publishes without waiting for the others.
// The scratch entries alternate between sweeps (sh: 2 x 8 doubles), so one
// barrier per exchange is enough: a workgroup meets another one before an
// entry is written again.
template <typename R, bool COOP>
__device__ __forceinline__ bool sweep_merit(const Dev<R>& d, double v, int it, bool lone, double* sh, int* s_ok,
                                            double& merit) {
  double* s = sh + 8 * (it & 1);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  double m = wave_max(v);
  if (!(COOP && lone)) {
    if (lane == 0) s[wid] = m;
    __syncthreads();
    m = 0.0;
    for (int i = 0; i < (int)(blockDim.x >> 6); ++i) m = fmax(m, s[i]);
  }
  if (COOP) {
    if (!lone) __syncthreads();     // s is read before it is written again
    if (wid == 0) {
      const bool ok = grid_merit(d.merit, it, m, d.err);
      if (lane == 0) { s[0] = m; *s_ok = ok ? 1 : 0; }
    }
    __syncthreads();
    m = s[0];
    merit = m;
    return *s_ok != 0;
  }
  merit = m;
  return true;
}

// Working (wl, wa) and accepted (sl, sa) velocity changes of the bodies (arena arrays).
template <typename R> struct VelStore {
  V4<R>* wl; V4<R>* wa; V4<R>* sl; V4<R>* sa;
};

// the constant rows of one contact and its previous iterate
template <typename R> struct Item {
  int2 loc, id;
  V4<R> n, rA, rB, b, r0, xo, W[4];
};

template <typename R> __device__ __forceinline__ void load_item(const Dev<R>& d, const V4<R>* xa, int kk, Item<R>& it) {
  it.loc = d.s_loc[kk];
  it.id = d.s_id[kk];
  it.n = d.s_n[kk];
  it.rA = d.s_rA[kk];
  it.rB = d.s_rB[kk];
  it.b = d.s_b[kk];
  it.r0 = d.s_r0[kk];
  it.xo = xa[kk];
  const V4<R>* W = d.s_W + 4 * (size_t)kk;
  it.W[0] = W[0]; it.W[1] = W[1]; it.W[2] = W[2]; it.W[3] = W[3];
}

// One contact (contacts.py:77-107).  Gauss-Seidel reads and updates the
// working velocity changes; Jacobi (jacobi_solver.py:6-57) reads the
// accepted ones and adds its change to the working ones.  Returns
// max |x_new - x_old| in FP64.
template <typename R>
__device__ __forceinline__ double update_contact(const ProxParams& pp, const Item<R>& it, VelStore<R>& w,
                                                 V4<R>* xn, int kk, R rs, bool jacobi, bool hybrid) {
  ContactRow<R> J;
  contact_rows(it.n, it.rA, it.rB, J);
  const V4<R> rr = {it.r0.x * rs, it.r0.y * rs, it.r0.z * rs, it.r0.w * rs};
  const V4<R> mu = {it.n.w, it.rA.w, it.rB.w, R(0)};
  const bool fa = it.loc.x >= 0, fb = it.loc.y >= 0;
  const int sa = it.id.x, sb = it.id.y;
  const V4<R> z = {R(0), R(0), R(0), R(0)};
  const V4<R>* rl = jacobi ? w.sl : w.wl;
  const V4<R>* ra = jacobi ? w.sa : w.wa;
  const V4<R> lA = fa ? rl[sa] : z, aA = fa ? ra[sa] : z;
  const V4<R> lB = fb ? rl[sb] : z, aB = fb ? ra[sb] : z;
  const V4<R> x = contact_prox(pp, J, it.xo, it.b, rr, mu, xyz(lA), xyz(aA), xyz(lB), xyz(aB), jacobi && !hybrid);
  xn[kk] = x;
  const V4<R> dx = {x.x - it.xo.x, x.y - it.xo.y, x.z - it.xo.z, x.w - it.xo.w};
  if (fa) {
    V4<R> l = jacobi ? w.wl[sa] : lA, g = jacobi ? w.wa[sa] : aA;
    dw_body(it.W[0], it.W[1], R(-1), J, J.angA, dx, l, g);
    w.wl[sa] = l;
    w.wa[sa] = g;
  }
  if (fb) {
    V4<R> l = jacobi ? w.wl[sb] : lB, g = jacobi ? w.wa[sb] : aB;
    dw_body(it.W[2], it.W[3], R(1), J, J.angB, dx, l, g);
    w.wl[sb] = l;
    w.wa[sb] = g;
  }
  return absmax4((double)x.x - (double)it.xo.x, (double)x.y - (double)it.xo.y, (double)x.z - (double)it.xo.z,
                 (double)x.w - (double)it.xo.w);
}

template <int STRIDE> __device__ __forceinline__ void phase_sync() {
  if (STRIDE == 64) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// One sweep of one lane at positions p0 + [0, K) sorted by colour: STRIDE
// lanes (a wavefront or the workgroup) take the contacts of a colour, in
// passes of STRIDE; colours are separated by a sync.  coff: colour offsets
// Returns this thread's max |dx|.
template <typename R, int STRIDE>
__device__ double sweep_lane(const Dev<R>& d, const ProxParams& pp, VelStore<R>& w, int p0, int nc,
                             const int* coff, bool jacobi, bool hybrid, const V4<R>* xa, V4<R>* xn,
                             R rs, int lane) {
  double m = 0.0;
  if (nc <= 0) return m;
  // pass state: colour c, first position pb of the pass, end hi of colour c, end hn of colour c + 1
  int c = 0;
  int pb = coff[0];
  int hi = coff[1];
  int hn = nc > 1 ? coff[2] : hi;
  // Two item buffers used in turn (no register copies, so the prefetch of
  // one pass stays in flight while the other is computed).
  Item<R> ia, ib;
  bool ha = pb + lane < hi;
  if (ha) load_item(d, xa, p0 + pb + lane, ia);
  auto step = [&](Item<R>& use, bool have, Item<R>& fill, bool& fhave) {
    const bool same = pb + STRIDE < hi;
    int c1, pb1, hi1, hn1;
    if (same) {
      c1 = c; pb1 = pb + STRIDE; hi1 = hi; hn1 = hn;
    } else {
      c1 = c + 1; pb1 = hi; hi1 = hn;
      hn1 = c1 + 1 < nc ? coff[c1 + 2] : hi1;
    }
    fhave = c1 < nc && pb1 + lane < hi1;
    if (fhave) load_item(d, xa, p0 + pb1 + lane, fill);
    if (have) m = fmax(m, update_contact(pp, use, w, xn, p0 + pb + lane, rs, jacobi, hybrid));
    if (!same) phase_sync<STRIDE>();
    c = c1; pb = pb1; hi = hi1; hn = hn1;
  };
  bool hb = false;
  while (true) {
    step(ia, ha, ib, hb);
    if (c >= nc) break;
    step(ib, hb, ia, ha);
    if (c >= nc) break;
  }
  return m;
}

// The lanes and bodies of one solve group.
struct Group {
  int l_lo, l_hi;     // lanes
  int b_lo, b_hi;     // body slots
  bool lead;          // writes the scene's solver state
};

template <typename R, bool COOP, int NT>
__device__ void solve_group(const Dev<R>& d, const int slot, const Group& gr, double* sh_red, int* s_ok) {
  const SceneParams& sp = d.sp[slot];
  SceneState& st = d.ss[slot];
  const int b0 = gr.b_lo, nbody = gr.b_hi - gr.b_lo;
  VelStore<R> w{d.ww0, d.ww1, d.ws0, d.ws1};
  const bool jacobi = sp.scheme == SCHEME_JACOBI || sp.scheme == SCHEME_JACOBI_HYBRID;
  const bool hybrid = sp.scheme == SCHEME_JACOBI_HYBRID;
  const ProxParams pp(sp);
  const CtlParams cp(sp);
  const double* hm = hinge_merits(d, sp);
  double* res = residual_record(d, sp);
  SolveCtl ctl;
  ctl.iters = sp.max_iter;
  for (int it = 0; it < sp.max_iter; ++it) {
    const V4<R>* xa = ctl.acc ? d.x1 : d.x0;
    V4<R>* xn = ctl.acc ? d.x0 : d.x1;
    const R rs = R(ctl.rscale);
    double m = 0.0;
    for (int l = gr.l_lo; l < gr.l_hi; ++l) {
      const int p0 = d.l_start[l], K = d.l_end[l] - p0;
      if (K <= 0) continue;
      m = fmax(m, sweep_lane<R, NT>(d, pp, w, p0, d.l_ncol[l], lane_coff(d, l), jacobi, hybrid, xa, xn, rs,
                                    (int)threadIdx.x));
    }
    double merit;
    if (!sweep_merit<R, COOP>(d, m, it, false, sh_red, s_ok, merit)) return;
    const int dec = ctl.decide(cp, merit, (gr.lead && threadIdx.x == 0) ? res : nullptr, it, hm ? hm[it] : 0.0);
    // accepted sweep: ws <- ww, else ww <- ws
    for (int i = threadIdx.x; i < nbody; i += blockDim.x) {
      const int s = d.u_blist[b0 + i];
      if (dec & 1) { w.sl[s] = w.wl[s]; w.sa[s] = w.wa[s]; }
      else { w.wl[s] = w.sl[s]; w.wa[s] = w.sa[s]; }
    }
    __syncthreads();
    if (dec & 2) { ctl.iters = it; break; }
  }
  // impulses back to contact order; natural-map residual (FP64) with r0
  const V4<R>* xs = ctl.acc ? d.x1 : d.x0;
  double rloc = 0.0, xmax = 0.0;
  const V4<R> z = {R(0), R(0), R(0), R(0)};
  for (int l = gr.l_lo; l < gr.l_hi; ++l) {
    const int p0 = d.l_start[l], K = d.l_end[l] - p0;
    if (K <= 0) continue;
    for (int pos = threadIdx.x; pos < K; pos += blockDim.x) {
      const int kk = p0 + pos;
      Item<R> c;
      load_item(d, xs, kk, c);
      const V4<R> x = c.xo;
      if (!d.post) d.c_imp[d.perm[kk]] = x;
      ContactRow<R> J;
      contact_rows(c.n, c.rA, c.rB, J);
      const V4<R> mu = {c.n.w, c.rA.w, c.rB.w, R(0)};
      const bool fa = c.loc.x >= 0, fb = c.loc.y >= 0;
      const int sa = c.id.x, sb = c.id.y;
      const V4<R> lA = fa ? w.sl[sa] : z, aA = fa ? w.sa[sa] : z;
      const V4<R> lB = fb ? w.sl[sb] : z, aB = fb ? w.sa[sb] : z;
      const V4<R> y = contact_prox(pp, J, x, c.b, c.r0, mu, xyz(lA), xyz(aA), xyz(lB), xyz(aB), false);
      rloc = fmax(rloc, absmax4((double)x.x - (double)y.x, (double)x.y - (double)y.y, (double)x.z - (double)y.z,
                                (double)x.w - (double)y.w));
      xmax = fmax(xmax, absmax4(x.x, x.y, x.z, x.w));
    }
  }
  const double rm = block_max(rloc, sh_red), xm = block_max(xmax, sh_red);
  if (threadIdx.x == 0) {
    if (d.post) {
      // the natural-map residual stays the contact solve's
    } else if (COOP) {
      if (rm > 0.0) atomic_max_nonneg(&st.nat_r, rm);
      if (xm > 0.0) atomic_max_nonneg(&st.nat_x, xm);
    } else {
      st.nat_r = rm;
      st.nat_x = xm;
    }
    if (gr.lead) write_solve_state(d, st, ctl);
  }
}

// value of lane K of each quad (DPP quad_perm(K, K, K, K))
template <int K> __device__ __forceinline__ float quad_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), K * 0x55, 0xf, 0xf, true));
}
template <int K> __device__ __forceinline__ double quad_bcast(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), K * 0x55, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), K * 0x55, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// value of lane K of each row of 16 lanes (DPP row_newbcast)
template <int K> __device__ __forceinline__ float row_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + K, 0xf, 0xf, true));
}
template <int K> __device__ __forceinline__ double row_bcast(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x150 + K, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x150 + K, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
// value of the lane 8 further round its row (DPP row_ror:8)
__device__ __forceinline__ float row_other_half(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, true));
}
__device__ __forceinline__ double row_other_half(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x128, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x128, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// One field of the bodies' LDS records: entry i of a record array with
// BODY_REC vec4s per body.
constexpr int BODY_REC = 6;
enum BodyField { F_WL = 0, F_WA, F_SL, F_SA, F_W0, F_W1 };
template <typename R> struct BodyCol {
  V4<R>* p;
  __device__ __forceinline__ V4<R>& operator[](int i) const { return p[BODY_REC * i]; }
};
// bytes of one body record
template <typename R> __host__ __device__ constexpr int rec_bytes() { return BODY_REC * (int)sizeof(V4<R>); }

// Velocity changes and inverse masses of a group's bodies at the start of its
// LDS, one record each: working (wl, wa) and accepted (sl, sa) velocity
// changes, inverse masses W0 = (I^-1 xx, xy, xz, 1/m), W1 = (I^-1 yy, yz, zz,
// 0) -- so that each row of I^-1 is one value and a pair of neighbours.  A
// contact's loads of one body then share one address.  The
// first record stays zero and stands for every fixed body, the second takes
// the discarded velocity updates of fixed bodies (so no update branches on
// them), the group's bodies follow.
constexpr int BODY_SPARE = 2;
template <typename R> struct BodyLds {
  BodyCol<R> wl, wa, sl, sa, W0, W1;   // (index -2: the zero record)
  __device__ explicit BodyLds(unsigned char* smem) {
    V4<R>* b = reinterpret_cast<V4<R>*>(smem) + BODY_REC * BODY_SPARE;
    wl.p = b; wa.p = b + 1; sl.p = b + 2; sa.p = b + 3; W0.p = b + 4; W1.p = b + 5;
  }
};

// natural-map residual parts of a contact (FP64) from its rows (row r at JL[S r],
// JA[S r], JB[S r]), its final values xs[0..3] and the accepted velocity changes
template <typename R, int S>
__device__ __forceinline__ void quad_finish_contact(const ProxParams& pp, const V4<R>* JL, const V4<R>* JA,
                                                    const V4<R>* JB, const R* xs, const V4<R>& lA, const V4<R>& aA,
                                                    const V4<R>& lB, const V4<R>& aB, V4<R>& x, double& rloc,
                                                    double& xmax) {
  x = V4<R>{xs[0], xs[1], xs[2], xs[3]};
  ContactRow<R> J;
  V4<R> bb, r0;
  R* bp = &bb.x;
  R* rp = &r0.x;
  for (int r = 0; r < 4; ++r) {
    const V4<R> a = JL[S * r], e = JA[S * r], f = JB[S * r];
    J.lin[r] = xyz(a); J.angA[r] = xyz(e); J.angB[r] = xyz(f);
    bp[r] = a.w; rp[r] = e.w;
  }
  const V4<R> mu = {JB[S].w, JB[2 * S].w, JB[3 * S].w, R(0)};
  const V4<R> y = contact_prox(pp, J, x, bb, r0, mu, xyz(lA), xyz(aA), xyz(lB), xyz(aB), false);
  rloc = fmax(rloc, absmax4((double)x.x - (double)y.x, (double)x.y - (double)y.y, (double)x.z - (double)y.z,
                            (double)x.w - (double)y.w));
  xmax = fmax(xmax, absmax4(x.x, x.y, x.z, x.w));
}

// LDS as plain 32-bit addresses: an access costs no address arithmetic beyond
// its own offset
template <typename T> using LdsPtr = __attribute__((address_space(3))) T*;
__device__ __forceinline__ int lds_addr(void* p) { return (int)(unsigned)(size_t)(LdsPtr<unsigned char>)p; }
template <typename T> __device__ __forceinline__ T& lds_at(int addr) { return *(T*)(LdsPtr<T>)(size_t)(unsigned)addr; }

// LDS addresses of a contact's bodies (A and B to read, A and B to write) from
// their slots; body: the address of the group's first record, b0 its first slot
template <typename R> __device__ __forceinline__ int4 contact_bodies(int2 loc, int body, int b0) {
  const int a = body + (loc.x - b0 + BODY_SPARE) * rec_bytes<R>(), b = body + (loc.y - b0 + BODY_SPARE) * rec_bytes<R>();
  const int z = body, t = body + rec_bytes<R>();
  return make_int4(loc.x >= 0 ? a : z, loc.y >= 0 ? b : z, loc.x >= 0 ? a : t, loc.y >= 0 ? b : t);
}

constexpr int RES_LANES = 64;   // lanes of a resident group
constexpr int PHASE_B = 2 * PHASE_Q;   // bytes of one phase of a resident lane's schedule
constexpr int PHASE_PAD = 4;    // phases read past a lane's last one

// LDS of a solve workgroup and the most contacts and bodies a tuning may ask
// for.  H = 1: the half layout, so that two solve workgroups share a CU when a
// batch has more scenes than the device has CUs.
template <typename R, int H = 0> struct ResCap {
  static constexpr int C = (sizeof(R) == 4 ? 384 : 192) >> H;   // contacts: limit of rbh_tuning.resident_contacts
  static constexpr int B = C;                                   // bodies: limit of rbh_tuning.resident_bodies
  static constexpr size_t LDS = (size_t)(H ? 80 : 160) * 1024 - 512;   // dynamic LDS of the launch
  static constexpr size_t BYTES = LDS - 256;                            // of it for the layouts (solve_scratch has the rest)
  // the streaming layout keeps only bodies in the same LDS
  static constexpr int VB = (int)(BYTES / (6 * sizeof(V4<R>))) - BODY_SPARE;
};

// LDS addresses of a resident group of nb bodies, nc contacts, nl lanes: its
// bodies, one record per contact (as in s_rec, the bodies as LDS addresses)
// and the null contact's, the lane table and the lanes' schedules.  A schedule
// lists, phase by phase, the record of each quad's or row's contact (in units
// of 16 bytes; the null contact where it has none).  A phase is at most 16 (4)
// contacts of one level, so a wavefront needs no test of positions against
// level ends, no loop over a wide level, and no branch.  (A narrow lane's
// phases, at most nc + K / 4 of 8 bytes, fit in the nc + K / 16 of 32.)
template <typename R> struct ResLds {
  int body;            // first body record
  int rec, nul;        // first contact record, the null contact's
  int lt, sched;       // lane table (int4: first record, contacts, first phase's place, 2 * phases + 1 if narrow), schedule
  __device__ ResLds(unsigned char* p, int nb, int nc, int nl) {
    body = lds_addr(p);
    rec = body + (nb + BODY_SPARE) * rec_bytes<R>();
    nul = rec + nc * Rec<R>::BYTES;
    lt = nul + Rec<R>::BYTES;
    sched = lt + nl * (int)sizeof(int4);
  }
  static constexpr size_t bytes(int nb, int nc, int nl, int nph) {
    return (size_t)(nb + BODY_SPARE) * rec_bytes<R>() + (size_t)(nc + 1) * Rec<R>::BYTES + (size_t)nl * sizeof(int4) +
           (size_t)(nph + PHASE_PAD) * PHASE_B;
  }
};
static_assert(ResCap<float>::BYTES / 16 < 65536, "a schedule entry addresses LDS in units of 16 bytes");

// sizes of a group's resident data (uniform over the workgroup)
struct GroupSize { int p0, nc, nph, nl; bool wg; };   // wg: a lane is for the whole workgroup (streaming)

template <typename R> __device__ GroupSize group_size(const Dev<R>& d, const Group& gr) {
  GroupSize g{0x7fffffff, 0, 0, 0, false};
  int p1 = 0;
  for (int l = gr.l_lo; l < gr.l_hi; ++l) {
    const int a = d.l_start[l], e = d.l_end[l];
    if (e <= a) continue;
    g.p0 = min(g.p0, a);
    p1 = max(p1, e);
    g.nph += lane_phases(e - a, d.l_ncol[l]);
    g.wg = g.wg || (d.l_nph[l] & LANE_WG);
    ++g.nl;
  }
  g.nc = g.nl ? p1 - g.p0 : 0;
  if (!g.nl) g.p0 = 0;
  return g;
}

template <typename R, int H>
__device__ __forceinline__ bool group_fits(const Dev<R>& d, const Group& gr, const GroupSize& g) {
  const int nb = gr.b_hi - gr.b_lo;
  // (the first bounds keep the sum below from overflowing)
  return g.nc <= min(d.res_cap_c, 4096) && nb <= min(d.res_cap_b, 4096) && g.nl <= RES_LANES &&
         ResLds<R>::bytes(nb, g.nc, g.nl, g.nph) <= ResCap<R, H>::BYTES;
}

// where a contact's record is read from: LDS (resident) or global memory
// (streaming); off: the lane's offset, k: a constant that folds into the load
struct LdsRec {
  int r;
  template <typename T> __device__ __forceinline__ T get(int off, int k = 0) const { return lds_at<T>(r + off + k); }
};
struct GlbRec {
  const unsigned char* base;
  unsigned r;
  template <typename T> __device__ __forceinline__ T get(int off, int k = 0) const {
    return *reinterpret_cast<const T*>(base + (r + (unsigned)off) + k);
  }
};

// A phase of a sweep is one contact by one quad, 16 contacts a wavefront
// (QuadPhase), or one contact by a row of 16 lanes, 4 contacts a wavefront
// (RowPhase); a lane of the problem is swept by one or the other throughout
// (narrow_phases).  Both give the iterates of update_contact bit for bit.
//
// A phase is a serial chain: velocities from LDS, the row products, the
// projection, the velocity update, back to LDS.  With one wavefront per SIMD
// nothing else hides its latency (measured here: 8 cycles per dependent
// vector instruction against 4.5 per independent one, 100 per LDS round trip,
// 33 per saveexec and branch), so:
//  * everything but the velocities is read ahead;
//  * the projection and the choice between the linear and the angular block
//    are selects, not branches;
//  * a row keeps its own projected value: it needs the others' only through
//    the sum of their squares;
//  * the sign of the update (body A minus, body B plus) is applied once, at
//    the end, and a linear update runs through the same multiply-add as an
//    angular one (times 1/m instead of times one).
// A quad's phase is then ~118 instructions and ~570 cycles (0.24 us), bound by
// their issue; with the branches, position tests and a wait for the previous
// phase's writes it took ~1,050.  4,096 spheres, 60 colours, 50 sweeps: solve
// 1613 -> 875 us.
//
// Most levels hold 2 to 4 contacts, so most quads idle, while a lane of a busy
// one computes a whole block.  A row of 16 splits the same sums: a half of J w
// per lane instead of both, one component of a block instead of three, 12
// instead of 17 LDS reads.  A row's phase is ~80 instructions and ~440 cycles,
// now bound by its dependent chain.  4,096 spheres, 59 phases: solve 800 -> 662
// us; 333-sphere Jacobi pile 1761 -> 1672.  (Streamed records stay with quads:
// a row's ten loads cover a quarter of the contacts but cost as much to issue,
// and a shorter phase leaves less time for them; 320 scenes 966 -> 1066 us.)
//
// Interface: LANES per contact; In, what a lane needs of its contact and none
// of which changes during a sweep; Loc, LDS addresses of its bodies; rows,
// loc, bodies and masses fill In; velocities reads what a phase starts from;
// update returns the lane's new iterate and sets nw, its part of the
// velocities after the update, for store.  JAC: Jacobi reads the accepted
// velocity changes (jacobi_solver.py:6-57), Gauss-Seidel the working ones.
template <typename R, bool ISO, bool JAC> struct QuadPhase {
  using X = Rec<R>;
  static constexpr int LANES = 4;
  static constexpr int VB = (int)sizeof(V4<R>), FV = JAC ? F_SL * VB : F_WL * VB;
  using Loc = int4;
  using Out = V4<R>;
  struct In {
    V4<R> jl, ja, jb, W0, W1;   // row q of J, the inverse mass of the block this lane updates
    V3<R> v0, v1, v2, v3;       // rows 0..3 of that block
    R xo;                       // the old iterate
    int oA, oB, own, wr;        // LDS addresses of the bodies read, the one updated, its block's new value
  };
  struct Vel { V4<R> lA, aA, lB, aB, old; };
  int q;
  bool side_b, ang;        // lane 0: linear A, 1: angular A, 2: linear B, 3: angular B
  int row, blk, fo;        // offsets: row q in a record, the block's rows, the block in a body record
  int xro, xwo;            // offsets of the old and the new iterate in a record
  R sgn;
  __device__ QuadPhase(int tid, int acc, int) {
    q = tid & 3;
    side_b = q >= 2;
    ang = q & 1;
    row = q * X::ROW;
    blk = ang ? (side_b ? 2 * VB : VB) : 0;
    fo = ang ? VB : 0;
    xro = (acc ? X::X1 : X::X0) + q * (int)sizeof(R);
    xwo = (acc ? X::X0 : X::X1) + q * (int)sizeof(R);
    sgn = side_b ? R(1) : R(-1);
  }
  template <typename A> __device__ __forceinline__ Loc loc(const A& at) const { return at.template get<int4>(0, X::LOC); }
  __device__ __forceinline__ void bodies(In& n, const Loc& lc) const {
    n.oA = lc.x;
    n.oB = lc.y;
    n.own = side_b ? lc.y : lc.x;
    n.wr = (side_b ? lc.w : lc.z) + fo;
  }
  template <typename A> __device__ __forceinline__ void rows(In& n, const A& at) const {
    n.jl = at.template get<V4<R>>(row);
    n.ja = at.template get<V4<R>>(row, VB);
    n.jb = at.template get<V4<R>>(row, 2 * VB);
    n.xo = at.template get<R>(xro);
    n.v0 = xyz(at.template get<V4<R>>(blk));
    n.v1 = xyz(at.template get<V4<R>>(blk, X::ROW));
    n.v2 = xyz(at.template get<V4<R>>(blk, 2 * X::ROW));
    n.v3 = xyz(at.template get<V4<R>>(blk, 3 * X::ROW));
  }
  __device__ __forceinline__ void masses(In& n) const {
    n.W0 = lds_at<V4<R>>(n.own + F_W0 * VB);
    n.W1 = lds_at<V4<R>>(n.own + F_W1 * VB);
  }
  __device__ __forceinline__ Vel velocities(const In& c) const {
    return Vel{lds_at<V4<R>>(c.oA + FV), lds_at<V4<R>>(c.oA + FV + VB), lds_at<V4<R>>(c.oB + FV),
               lds_at<V4<R>>(c.oB + FV + VB), lds_at<V4<R>>(c.own + fo)};
  }
  __device__ __forceinline__ R update(const ProxParams& pp, const In& c, const Vel& v, R rs, bool hybrid, Out& nw) const {
    // row q of z = x - r (J w + b)  (contacts.py:77-92)
    const R Jw = row_jw(xyz(c.jl), xyz(c.ja), xyz(c.jb), xyz(v.lA), xyz(v.aA), xyz(v.lB), xyz(v.aB));
    const R z = row_z(c.xo, c.ja.w * rs, Jw, c.jl.w);
    // projections (contacts.py:92-95)
    const R z0 = fmax(R(0), z);
    const R xnrm = quad_bcast<0>(z0);
    const R xr = (JAC && !hybrid) ? quad_bcast<0>(c.xo) : xnrm;
    R val;
    if constexpr (ISO) {
      const R zz = z * z;
      const R sq = (quad_bcast<1>(zz) + quad_bcast<2>(zz)) + quad_bcast<3>(zz);
      val = prox_sphere_row<R>(z, sq, c.jb.w, xr);
    } else {
      const R z1 = quad_bcast<1>(z), z2 = quad_bcast<2>(z), z3 = quad_bcast<3>(z);
      const R mu0 = quad_bcast<1>(c.jb.w), mu1 = quad_bcast<2>(c.jb.w), mu2 = quad_bcast<3>(c.jb.w);
      const V3<R> o = prox_ellipsoid_call<R>(z1, z2, z3, mu0, mu1, mu2, xr, pp.ell_tol, pp.ell_expansion, pp.ell_max_iter);
      val = side_b ? (ang ? o.z : o.y) : o.x;
    }
    const R xq = q == 0 ? z0 : val;
    const R dq = xq - c.xo;
    // w += W J^T dx (contacts.py:107), this lane's block
    const R d0 = quad_bcast<0>(dq), d1 = quad_bcast<1>(dq), d2 = quad_bcast<2>(dq), d3 = quad_bcast<3>(dq);
    V3<R> a = {sum_first(d0 * c.v0.x), sum_first(d0 * c.v0.y), sum_first(d0 * c.v0.z)};
    a.x = madd(d1, c.v1.x, a.x); a.y = madd(d1, c.v1.y, a.y); a.z = madd(d1, c.v1.z, a.z);
    a.x = madd(d2, c.v2.x, a.x); a.y = madd(d2, c.v2.y, a.y); a.z = madd(d2, c.v2.z, a.z);
    a.x = madd(d3, c.v3.x, a.x); a.y = madd(d3, c.v3.y, a.y); a.z = madd(d3, c.v3.z, a.z);
    const R W[6] = {c.W0.x, c.W1.x, c.W1.z, c.W0.y, c.W0.z, c.W1.y};   // (xx, yy, zz, xy, xz, yz)
    const V3<R> t = sym_madd(W, a);
    const R s = ang ? sgn : sgn * c.W0.w;
    const V3<R> u = {ang ? t.x : a.x, ang ? t.y : a.y, ang ? t.z : a.z};
    nw = V4<R>{madd(s, u.x, v.old.x), madd(s, u.y, v.old.y), madd(s, u.z, v.old.z), R(0)};
    return xq;
  }
  __device__ __forceinline__ void store(const In& c, const Out& nw) const { lds_at<V4<R>>(c.wr) = nw; }
  // where the lane's new iterate goes in LDS
  __device__ __forceinline__ int x_addr(int r) const { return r + xwo; }
};

// Quad b of a row of 16 lanes updates block b (linear A, angular A, linear B,
// angular B), its lane c component c.  Before that the lanes of the two side-A
// quads sum side A's half of row c's J w, those of the side-B quads side B's,
// which take the others' sums and go on to row c's projection; the side-A
// quads compute along on values that nothing uses, and their iterates and the
// fourth lanes' velocities are stored in the spare body record.
template <typename R, bool ISO, bool JAC> struct RowPhase {
  using X = Rec<R>;
  static constexpr int LANES = 16;
  static constexpr int SR = (int)sizeof(R), VB = (int)sizeof(V4<R>), FV = JAC ? F_SL * VB : F_WL * VB;
  using Loc = int2;        // the lane's side: body to read, body to write
  using Out = R;
  struct In {
    V4<R> jl, js;          // row c of J: linear part and this side's angular one
    R r, xo;               // of row c: r0, the old iterate
    R v0, v1, v2, v3;      // component c of rows 0..3 of the block
    R w0, w1, w2;          // row c of I^-1 (linear blocks: w0 = 1/m)
    int own, wr;           // LDS addresses of the body, of the component's new value
  };
  struct Vel { V4<R> l, a; R old; };
  int c;
  bool ang;
  int row, jso, blk, loc_o, fo, wf, wp;   // offsets
  int xro, xadd;
  unsigned wmul, xmul;     // 1: store, 0: store in the spare record
  int wadd;
  R sgn;
  __device__ RowPhase(int tid, int acc, int body) {
    c = tid & 3;
    const int b = (tid >> 2) & 3;
    const bool side_b = b >= 2;
    ang = b & 1;
    row = c * X::ROW;
    jso = row + (side_b ? 2 * VB : VB);
    blk = (ang ? (side_b ? 2 * VB : VB) : 0) + c * SR;
    loc_o = X::LOC + (side_b ? 4 : 0);
    fo = (ang ? VB : 0) + c * SR;
    wf = F_W0 * VB + (ang ? (c < 3 ? c : 0) : 3) * SR;
    wp = F_W0 * VB + (c == 1 ? 4 : c == 2 ? 5 : 1) * SR;
    const int spare = body + rec_bytes<R>();
    wmul = c < 3 ? 1u : 0u;
    wadd = c < 3 ? fo : spare;
    xro = (acc ? X::X1 : X::X0) + c * SR;
    xmul = b == 2 ? 1u : 0u;
    xadd = b == 2 ? (acc ? X::X0 : X::X1) + c * SR : spare;
    sgn = side_b ? R(1) : R(-1);
    // (factors the compiler does not see through: one multiply-add an address, not a mask, a select and an add)
    asm("" : "+v"(wmul), "+v"(xmul));
  }
  template <typename A> __device__ __forceinline__ Loc loc(const A& at) const {
    return make_int2(at.template get<int>(loc_o), at.template get<int>(loc_o, 8));
  }
  __device__ __forceinline__ void bodies(In& n, const Loc& lc) const {
    n.own = lc.x;
    n.wr = (int)(__umul24((unsigned)lc.y, wmul) + (unsigned)wadd);
  }
  template <typename A> __device__ __forceinline__ void rows(In& n, const A& at) const {
    n.jl = at.template get<V4<R>>(row);
    n.js = at.template get<V4<R>>(jso);
    n.r = at.template get<R>(row, VB + 3 * SR);
    n.xo = at.template get<R>(xro);
    n.v0 = at.template get<R>(blk);
    n.v1 = at.template get<R>(blk, X::ROW);
    n.v2 = at.template get<R>(blk, 2 * X::ROW);
    n.v3 = at.template get<R>(blk, 3 * X::ROW);
  }
  __device__ __forceinline__ void masses(In& n) const {
    n.w0 = lds_at<R>(n.own + wf);
    n.w1 = lds_at<R>(n.own + wp);
    n.w2 = lds_at<R>(n.own + wp + SR);
  }
  __device__ __forceinline__ Vel velocities(const In& k) const {
    return Vel{lds_at<V4<R>>(k.own + FV), lds_at<V4<R>>(k.own + FV + VB), lds_at<R>(k.own + fo)};
  }
  __device__ __forceinline__ R update(const ProxParams& pp, const In& k, const Vel& v, R rs, bool hybrid, Out& nw) const {
    // this side's half of row c of J w, then the row on the side-B quads (row_jw's sums in its order)
    R Jw;
    if constexpr (sizeof(R) == 8) {
      const R lw = dot(xyz(k.jl), xyz(v.l)), aw = dot(xyz(k.js), xyz(v.a));
      Jw = row_other_half(-lw - aw) + lw + aw;
    } else {
      R h = k.jl.x * v.l.x;
      h = madd(k.jl.y, v.l.y, h); h = madd(k.jl.z, v.l.z, h);
      h = madd(k.js.x, v.a.x, h); h = madd(k.js.y, v.a.y, h); h = madd(k.js.z, v.a.z, h);
      Jw = h - row_other_half(h);
    }
    const R z = row_z(k.xo, k.r * rs, Jw, k.jl.w);
    const R z0 = fmax(R(0), z);
    const R xnrm = quad_bcast<0>(z0);
    const R xr = (JAC && !hybrid) ? quad_bcast<0>(k.xo) : xnrm;
    R val;
    if constexpr (ISO) {
      const R zz = z * z;
      const R sq = (quad_bcast<1>(zz) + quad_bcast<2>(zz)) + quad_bcast<3>(zz);
      val = prox_sphere_row<R>(z, sq, k.js.w, xr);
    } else {
      const R z1 = row_bcast<9>(z), z2 = row_bcast<10>(z), z3 = row_bcast<11>(z);
      const R mu0 = row_bcast<9>(k.js.w), mu1 = row_bcast<10>(k.js.w), mu2 = row_bcast<11>(k.js.w);
      const V3<R> o = prox_ellipsoid_call<R>(z1, z2, z3, mu0, mu1, mu2, row_bcast<8>(xr), pp.ell_tol, pp.ell_expansion,
                                             pp.ell_max_iter);
      val = c == 3 ? o.z : c == 2 ? o.y : o.x;
    }
    const R xq = c == 0 ? z0 : val;
    const R dq = xq - k.xo;
    // component c of the block's update
    R a = sum_first(row_bcast<8>(dq) * k.v0);
    a = madd(row_bcast<9>(dq), k.v1, a);
    a = madd(row_bcast<10>(dq), k.v2, a);
    a = madd(row_bcast<11>(dq), k.v3, a);
    const R t = madd(k.w2, quad_bcast<2>(a), madd(k.w1, quad_bcast<1>(a), k.w0 * quad_bcast<0>(a)));
    nw = madd(ang ? sgn : sgn * k.w0, ang ? t : a, v.old);
    return xq;
  }
  __device__ __forceinline__ void store(const In& k, const Out& nw) const { lds_at<R>(k.wr) = nw; }
  __device__ __forceinline__ int x_addr(int r) const { return (int)(__umul24((unsigned)r, xmul) + (unsigned)xadd); }
};

// ---- resident layout: everything a sweep touches in LDS

// One sweep of one resident lane by one wavefront.  Rows, inverse masses and
// iterates are read one phase ahead, the bodies' addresses two ahead and the
// schedule three ahead.
template <typename R, typename P>
__device__ double res_sweep(const ProxParams& pp, const ResLds<R>& L, int4 lt, bool hybrid, int acc, R rs, int lane) {
  using X = Rec<R>;
  constexpr int STEP = 2 * (64 / P::LANES);   // bytes of a phase of the schedule
  struct In : P::In { int xw; };
  const int rec0 = __builtin_amdgcn_readfirstlane(lt.x), K = __builtin_amdgcn_readfirstlane(lt.y);
  const int nph = __builtin_amdgcn_readfirstlane(lt.w) >> 1;
  if (nph <= 0) return 0.0;
  const P ph(lane, acc, L.body);
  int sp = L.sched + __builtin_amdgcn_readfirstlane(lt.z) * PHASE_B + 2 * (lane / P::LANES);
  auto entry = [&](int ahead) { return (int)lds_at<unsigned short>(sp + ahead * STEP) * 16; };
  auto load = [&](int r, const typename P::Loc& lc, In& p) {
    const LdsRec at{r};
    ph.bodies(p, lc);
    ph.rows(p, at);
    ph.masses(p);
    p.xw = ph.x_addr(r);
  };
  int r1 = entry(1), e2 = entry(2);
  In pa, pb;
  typename P::Loc lc1;
  {
    const int r0 = entry(0);
    const typename P::Loc lc0 = ph.loc(LdsRec{r0});
    lc1 = ph.loc(LdsRec{r1});
    load(r0, lc0, pa);
  }
  // the reads above are done when the loop starts: a wait inside it would
  // also wait for the previous phase's writes
  __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
  auto phase = [&](const In& c, In& n) {
    const typename P::Vel v = ph.velocities(c);
    load(r1, lc1, n);
    const int r2 = e2;
    lc1 = ph.loc(LdsRec{r2});
    e2 = entry(3);
    r1 = r2;
    sp += STEP;
    typename P::Out nw;
    const R xq = ph.update(pp, c, v, rs, hybrid, nw);
    ph.store(c, nw);
    lds_at<R>(c.xw) = xq;
    phase_sync<64>();
  };
  for (int p = 0;;) {
    phase(pa, pb);
    if (++p >= nph) break;
    phase(pb, pa);
    if (++p >= nph) break;
  }
  // the merit, max |x_new - x_old| in FP64 (a sweep updates each contact once)
  // 64 contacts per pass, their reads in flight together (past the last
  // contact the last one again)
  const int xr = (acc ? X::X1 : X::X0) + (lane & 3) * (int)sizeof(R), xw = X::X0 + X::X1 + 2 * (lane & 3) * (int)sizeof(R) - xr;
  double m = 0.0;
  for (int i = lane >> 2; i - (lane >> 2) < K; i += 4 * PHASE_Q) {
    R xn[4], xo[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = rec0 + min(i + u * PHASE_Q, K - 1) * X::BYTES;
      xn[u] = lds_at<R>(r + xw);
      xo[u] = lds_at<R>(r + xr);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) m = fmax(m, fabs((double)xn[u] - (double)xo[u]));
  }
  return m;
}

template <typename R, bool ISO, bool JAC>
__device__ __forceinline__ double res_sweep_lane(const ProxParams& pp, const ResLds<R>& L, int4 lt, bool hybrid, int acc,
                                                 R rs, int lane) {
  return lt.w & 1 ? res_sweep<R, RowPhase<R, ISO, JAC>>(pp, L, lt, hybrid, acc, rs, lane)
                  : res_sweep<R, QuadPhase<R, ISO, JAC>>(pp, L, lt, hybrid, acc, rs, lane);
}

// what a group's sweeps are decided with, the same for every sweep
template <typename R> struct Decide {
  CtlParams cp;
  const double* hm;    // the hinges' merits, or null
  double* res;         // the scene's merit record, or null where another thread writes it
  bool lone;           // only wavefront 0 sweeps
  __device__ Decide(const Dev<R>& d, const SceneParams& sp, bool lead, bool lone_)
      : cp(sp), hm(hinge_merits(d, sp)), res(lead && threadIdx.x == 0 ? residual_record(d, sp) : nullptr), lone(lone_) {}
};

// merit meets, accept/reject decided, velocity changes settled (all groups of the scene)
template <typename R, bool COOP>
__device__ __forceinline__ int sweep_decide(const Dev<R>& d, const Decide<R>& by, SolveCtl& ctl, double m, int it,
                                            double* sh_red, int* s_ok, const BodyLds<R>& B, int nb, bool& abort) {
  double merit;
  const double other = by.hm ? by.hm[it] : 0.0;
  if (!sweep_merit<R, COOP>(d, m, it, by.lone, sh_red, s_ok, merit)) { abort = true; return 0; }
  const int dec = ctl.decide(by.cp, merit, by.res, it, other);
  for (int i = threadIdx.x; i < nb; i += blockDim.x) {
    if (dec & 1) { B.sl[i] = B.wl[i]; B.sa[i] = B.wa[i]; }
    else { B.wl[i] = B.sl[i]; B.wa[i] = B.sa[i]; }
  }
  __syncthreads();
  return dec;
}

template <typename R> __device__ void stage_bodies(const Dev<R>& d, const BodyLds<R>& B, int b0, int nb) {
  for (int i = threadIdx.x; i < nb; i += blockDim.x) {
    const int b = d.u_blist[b0 + i];
    B.wl[i] = d.ww0[b]; B.wa[i] = d.ww1[b]; B.sl[i] = d.ws0[b]; B.sa[i] = d.ws1[b];
    const V4<R> w0 = d.b_W0[b], w1 = d.b_W1[b];   // (xx, yy, zz, xy), (xz, yz, 1/m, 0)
    B.W0[i] = V4<R>{w0.x, w0.w, w1.x, w1.z};
    B.W1[i] = V4<R>{w0.y, w1.y, w0.z, R(0)};
  }
  if (threadIdx.x < BODY_SPARE) {
    const V4<R> z = {R(0), R(0), R(0), R(0)};
    const int i = (int)threadIdx.x - BODY_SPARE;
    B.wl[i] = z; B.wa[i] = z; B.sl[i] = z; B.sa[i] = z; B.W0[i] = z; B.W1[i] = z;
  }
}

template <typename R, bool COOP>
__device__ void finish_group(const Dev<R>& d, SceneState& st, const SolveCtl& ctl, bool lead, const BodyLds<R>& B,
                             int b0, int nb, double rloc, double xmax, double* sh_red) {
  for (int i = threadIdx.x; i < nb; i += blockDim.x) {
    const int b = d.u_blist[b0 + i];
    d.ws0[b] = B.sl[i];
    d.ws1[b] = B.sa[i];
  }
  const double rm = block_max(rloc, sh_red), xm = block_max(xmax, sh_red);
  if (threadIdx.x == 0) {
    if (d.post) {
      // the natural-map residual stays the contact solve's
    } else if (COOP) {
      if (rm > 0.0) atomic_max_nonneg(&st.nat_r, rm);
      if (xm > 0.0) atomic_max_nonneg(&st.nat_x, xm);
    } else {
      st.nat_r = rm;
      st.nat_x = xm;
    }
    if (lead) write_solve_state(d, st, ctl);
  }
}

template <typename R, bool COOP, int NT, int H>
__device__ void solve_group_resident(const Dev<R>& d, const int slot, const Group& gr, const GroupSize& gs,
                                     unsigned char* smem, double* sh_red, int* s_ok) {
  using X = Rec<R>;
  constexpr int VB = (int)sizeof(V4<R>);
  const SceneParams& sp = d.sp[slot];
  SceneState& st = d.ss[slot];
  const bool jacobi = sp.scheme == SCHEME_JACOBI || sp.scheme == SCHEME_JACOBI_HYBRID;
  const bool hybrid = sp.scheme == SCHEME_JACOBI_HYBRID;
  const ProxParams pp(sp);
  const bool iso = pp.friction != 1;
  const int b0 = gr.b_lo, nb = gr.b_hi - gr.b_lo;
  const ResLds<R> L(smem, nb, gs.nc, gs.nl);
  const BodyLds<R> B(smem);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nwave = blockDim.x >> 6;
  // stage: lane table (fourth entry: the sweep lane, until its schedule is written), an empty schedule,
  // contact records, bodies
  if (threadIdx.x == 0) {
    int t = 0, o = 0;
    for (int l = gr.l_lo; l < gr.l_hi; ++l) {
      const int a = d.l_start[l], e = d.l_end[l];
      if (e <= a) continue;
      lds_at<int4>(L.lt + 16 * t++) = make_int4(L.rec + (a - gs.p0) * X::BYTES, e - a, o, l);
      o += lane_phases(e - a, d.l_ncol[l]);
    }
  }
  for (int i = threadIdx.x; i < (gs.nph + PHASE_PAD) * PHASE_Q; i += blockDim.x)
    lds_at<unsigned short>(L.sched + 2 * i) = (unsigned short)(L.nul / 16);
  constexpr int WORDS = X::BYTES / 16, LOCW = X::LOC / 16;
  const int4* src = reinterpret_cast<const int4*>(d.s_rec + (size_t)gs.p0 * X::BYTES);
  for (int i = threadIdx.x; i < gs.nc * WORDS; i += blockDim.x)
    if (i % WORDS != LOCW) lds_at<int4>(L.rec + 16 * i) = src[i];
  for (int i = threadIdx.x; i < WORDS; i += blockDim.x)
    if (i != LOCW) lds_at<int4>(L.nul + 16 * i) = make_int4(0, 0, 0, 0);
  for (int i = threadIdx.x; i <= gs.nc; i += blockDim.x)
    lds_at<int4>(L.rec + i * X::BYTES + X::LOC) =
        contact_bodies<R>(i < gs.nc ? d.s_loc[gs.p0 + i] : make_int2(-1, -1), L.body, b0);
  stage_bodies(d, B, b0, nb);
  __syncthreads();
  // schedules: a wavefront per lane, its levels 64 at a time
  for (int t = wave; t < gs.nl; t += nwave) {
    const int4 lt = lds_at<int4>(L.lt + 16 * t);
    const int nc = d.l_ncol[lt.w];
    const int* co = lane_coff(d, lt.w);
    const bool rows16 = d.l_nph[lt.w] & LANE_NARROW;
    const int per = rows16 ? PHASE_R : PHASE_Q;
    int ph = 0;
    for (int c0 = 0; c0 < nc; c0 += 64) {
      const int c = c0 + lane;
      const int lo = c < nc ? co[c] : 0, w = c < nc ? co[c + 1] - lo : 0;
      const int np = (w + per - 1) / per;
      const int inc = wave_inclusive_sum(np);
      const int s0 = L.sched + lt.z * PHASE_B + (ph + inc - np) * 2 * per;
      for (int i = 0; i < w; ++i)   // (slots of one phase are consecutive, and so are its phases)
        lds_at<unsigned short>(s0 + 2 * i) = (unsigned short)((lt.x + (lo + i) * X::BYTES) / 16);
      ph += __shfl(inc, 63, 64);
    }
    if (lane == 0) lds_at<int>(L.lt + 16 * t + 12) = ph << 1 | (rows16 ? 1 : 0);
  }
  __syncthreads();
  const Decide<R> by(d, sp, gr.lead, gs.nl <= 1);
  SolveCtl ctl;
  ctl.iters = sp.max_iter;
  bool abort = false;
  for (int it = 0; it < sp.max_iter; ++it) {
    const R rs = R(ctl.rscale);
    double m = 0.0;
    for (int t = wave; t < gs.nl; t += nwave) {
      const int4 lt = lds_at<int4>(L.lt + 16 * t);
      double ml;
      if (jacobi)
        ml = iso ? res_sweep_lane<R, true, true>(pp, L, lt, hybrid, ctl.acc, rs, lane)
                 : res_sweep_lane<R, false, true>(pp, L, lt, hybrid, ctl.acc, rs, lane);
      else
        ml = iso ? res_sweep_lane<R, true, false>(pp, L, lt, hybrid, ctl.acc, rs, lane)
                 : res_sweep_lane<R, false, false>(pp, L, lt, hybrid, ctl.acc, rs, lane);
      m = fmax(m, ml);
    }
    const int dec = sweep_decide<R, COOP>(d, by, ctl, m, it, sh_red, s_ok, B, nb, abort);
    if (abort) return;
    if (dec & 2) { ctl.iters = it; break; }
  }
  // impulses to contact order; natural-map residual (FP64) with r0; accepted velocity changes out
  double rloc = 0.0, xmax = 0.0;
  for (int i = threadIdx.x; i < gs.nc; i += blockDim.x) {
    const int rec = L.rec + i * X::BYTES;
    const int4 lc = lds_at<int4>(rec + X::LOC);
    const R* xs = &lds_at<R>(rec + (ctl.acc ? X::X1 : X::X0));
    const V4<R>* rows = &lds_at<V4<R>>(rec);
    V4<R> x;
    quad_finish_contact<R, 3>(pp, rows, rows + 1, rows + 2, xs, lds_at<V4<R>>(lc.x + F_SL * VB),
                              lds_at<V4<R>>(lc.x + F_SA * VB), lds_at<V4<R>>(lc.y + F_SL * VB),
                              lds_at<V4<R>>(lc.y + F_SA * VB), x, rloc, xmax);
    if (!d.post) d.c_imp[d.perm[gs.p0 + i]] = x;
  }
  finish_group<R, COOP>(d, st, ctl, gr.lead, B, b0, nb, rloc, xmax, sh_red);
}

// ---- streaming layout: bodies in LDS, contact records in global memory

// One sweep of one lane: its phases from k_order_lanes' list, one contact per
// quad.  WG: by the whole workgroup (up to NT / 4 contacts of a level per
// phase, a workgroup barrier between phases), else by one wavefront.  The
// records of a phase are read from global memory two phases ahead, each lane
// its own row and block, in three register buffers used in turn; a quad
// without a contact reads the null record after the last one.  Bound by the
// phase's chain (QuadPhase::update) as long as the records come from L2.  With rows
// loaded one phase ahead, the block's rows in the phase itself and lanes of
// more than 512 contacts always swept by the workgroup, the solve took: 24
// scenes of ~2,100 contacts 6859 us (now 1406), 320 of ~330 1960 (977),
// 1,500-sphere pile 5278 (2158), 48 meshes 8920 (4300).
template <typename R, bool ISO, bool JAC, bool WG>
__device__ double stream_sweep(const Dev<R>& d, const ProxParams& pp, int l, bool hybrid, int acc, R rs, int tid) {
  using X = Rec<R>;
  using P = QuadPhase<R, ISO, JAC>;
  struct In : P::In { typename P::Loc lc; unsigned off; };
  const int p0 = __builtin_amdgcn_readfirstlane(d.l_start[l]);
  const int nph = __builtin_amdgcn_readfirstlane(d.l_nph[l]) >> LANE_BITS;
  if (nph <= 0) return 0.0;
  const int j = tid / P::LANES, lane = tid & 63;
  const P ph(tid, acc, 0);
  unsigned char* const rec = d.s_rec;
  const unsigned nul = (unsigned)d.cap_contacts * (unsigned)X::BYTES;
  // the list, 64 phases at a time (lane i holds phase i of the run), the next run read ahead
  const unsigned* list = d.l_phase + p0;
  unsigned run = list[min(lane, nph - 1)], ahead = list[min(64 + lane, nph - 1)];
  int base = 0;
  auto fetch = [&](int p, In& n) {
    if (p - base >= 64) { run = ahead; base += 64; ahead = list[min(base + 64 + lane, nph - 1)]; }
    const unsigned e = p < nph ? (unsigned)__builtin_amdgcn_readlane((int)run, p & 63) : 0u;
    const unsigned pos = e >> PHASE_BITS, cnt = e & ((1u << PHASE_BITS) - 1u);
    n.off = (unsigned)j < cnt ? ((unsigned)p0 + pos + (unsigned)j) * (unsigned)X::BYTES : nul;
    const GlbRec at{rec, n.off};
    n.lc = ph.loc(at);
    ph.rows(n, at);
  };
  auto masses = [&](In& n) {
    ph.bodies(n, n.lc);
    ph.masses(n);
  };
  double m = 0.0;
  In a, b, c;
  fetch(0, a);
  fetch(1, b);
  masses(a);
  int p = 0;
  auto phase = [&](In& cur, In& nxt, In& fill) {
    const typename P::Vel v = ph.velocities(cur);
    masses(nxt);
    fetch(p + 2, fill);
    typename P::Out nw;
    const R xq = ph.update(pp, cur, v, rs, hybrid, nw);
    ph.store(cur, nw);
    if (cur.off != nul) *reinterpret_cast<R*>(rec + cur.off + ph.xwo) = xq;
    m = fmax(m, fabs((double)xq - (double)cur.xo));
    if (WG) __syncthreads();
    else phase_sync<64>();
    ++p;
  };
  while (true) {
    phase(a, b, c);
    if (p >= nph) break;
    phase(b, c, a);
    if (p >= nph) break;
    phase(c, a, b);
    if (p >= nph) break;
  }
  return m;
}

template <typename R, bool ISO, bool JAC>
__device__ double stream_lanes(const Dev<R>& d, const ProxParams& pp, const Group& gr, bool hybrid, int acc, R rs) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nwave = blockDim.x >> 6;
  double m = 0.0;
  int t = 0;
  for (int l = gr.l_lo; l < gr.l_hi; ++l) {
    if (d.l_end[l] <= d.l_start[l] || (d.l_nph[l] & LANE_WG)) continue;
    if (t++ % nwave == wave) m = fmax(m, stream_sweep<R, ISO, JAC, false>(d, pp, l, hybrid, acc, rs, lane));
  }
  for (int l = gr.l_lo; l < gr.l_hi; ++l) {   // lanes swept by the workgroup
    if (d.l_end[l] <= d.l_start[l] || !(d.l_nph[l] & LANE_WG)) continue;
    m = fmax(m, stream_sweep<R, ISO, JAC, true>(d, pp, l, hybrid, acc, rs, (int)threadIdx.x));
  }
  return m;
}

template <typename R, bool COOP, int NT, int H>
__device__ void solve_group_stream(const Dev<R>& d, const int slot, const Group& gr, const GroupSize& gs,
                                   unsigned char* smem, double* sh_red, int* s_ok) {
  using X = Rec<R>;
  const SceneParams& sp = d.sp[slot];
  SceneState& st = d.ss[slot];
  const bool jacobi = sp.scheme == SCHEME_JACOBI || sp.scheme == SCHEME_JACOBI_HYBRID;
  const bool hybrid = sp.scheme == SCHEME_JACOBI_HYBRID;
  const ProxParams pp(sp);
  const bool iso = pp.friction != 1;
  const BodyLds<R> B(smem);
  const int body = lds_addr(smem), b0 = gr.b_lo, nb = gr.b_hi - gr.b_lo;
  stage_bodies(d, B, b0, nb);
  // the contacts' bodies as LDS addresses of this group (the null contact's are the same in every group)
  for (int i = threadIdx.x; i < gs.nc; i += blockDim.x)
    *reinterpret_cast<int4*>(d.s_rec + (size_t)(gs.p0 + i) * X::BYTES + X::LOC) =
        contact_bodies<R>(d.s_loc[gs.p0 + i], body, b0);
  if (threadIdx.x == 0)
    *reinterpret_cast<int4*>(d.s_rec + (size_t)d.cap_contacts * X::BYTES + X::LOC) =
        contact_bodies<R>(make_int2(-1, -1), body, b0);
  __syncthreads();
  const Decide<R> by(d, sp, gr.lead, gs.nl <= 1 && !gs.wg);
  SolveCtl ctl;
  ctl.iters = sp.max_iter;
  bool abort = false;
  for (int it = 0; it < sp.max_iter; ++it) {
    const R rs = R(ctl.rscale);
    double m;
    if (jacobi)
      m = iso ? stream_lanes<R, true, true>(d, pp, gr, hybrid, ctl.acc, rs)
              : stream_lanes<R, false, true>(d, pp, gr, hybrid, ctl.acc, rs);
    else
      m = iso ? stream_lanes<R, true, false>(d, pp, gr, hybrid, ctl.acc, rs)
              : stream_lanes<R, false, false>(d, pp, gr, hybrid, ctl.acc, rs);
    const int dec = sweep_decide<R, COOP>(d, by, ctl, m, it, sh_red, s_ok, B, nb, abort);
    if (abort) return;
    if (dec & 2) { ctl.iters = it; break; }
  }
  double rloc = 0.0, xmax = 0.0;
  for (int i = threadIdx.x; i < gs.nc; i += blockDim.x) {
    const unsigned char* rec = d.s_rec + (size_t)(gs.p0 + i) * X::BYTES;
    const int2 lc = d.s_loc[gs.p0 + i];
    const int sa = lc.x >= 0 ? lc.x - b0 : -BODY_SPARE, sb = lc.y >= 0 ? lc.y - b0 : -BODY_SPARE;
    const V4<R>* rows = reinterpret_cast<const V4<R>*>(rec);
    V4<R> x;
    quad_finish_contact<R, 3>(pp, rows, rows + 1, rows + 2, reinterpret_cast<const R*>(rec + (ctl.acc ? X::X1 : X::X0)),
                              B.sl[sa], B.sa[sa], B.sl[sb], B.sa[sb], x, rloc, xmax);
    if (!d.post) d.c_imp[d.perm[gs.p0 + i]] = x;
  }
  finish_group<R, COOP>(d, st, ctl, gr.lead, B, b0, nb, rloc, xmax, sh_red);
}

template <typename R> __device__ __forceinline__ void no_contacts(SceneState& st) {
  st.solved = 0; st.iterations = 0; st.exitcode = 0; st.sweeps = 0; st.rejects = 0; st.final_merit = 0.0;
}

template <typename R, bool COOP, int NT, int H>
__device__ __forceinline__ void solve_dispatch(const Dev<R>& d, int slot, const Group& gr, unsigned char* smem,
                                               double* sh_red, int* s_ok) {
  const GroupSize gs = group_size(d, gr);
  if (group_fits<R, H>(d, gr, gs)) solve_group_resident<R, COOP, NT, H>(d, slot, gr, gs, smem, sh_red, s_ok);
  else if (gr.b_hi - gr.b_lo <= ResCap<R, H>::VB && rec_addressable<R>(d.cap_contacts))
    solve_group_stream<R, COOP, NT, H>(d, slot, gr, gs, smem, sh_red, s_ok);
  else solve_group<R, COOP, NT>(d, slot, gr, sh_red, s_ok);
}

// The solve kernels' reduction scratch (2 x 8 doubles) and flag, at the end
// of the dynamic LDS: with no static LDS the layouts start at LDS address 0,
// so their offsets fold into the LDS instructions.
template <typename R, int H>
__device__ __forceinline__ void solve_scratch(unsigned char* smem, double*& red, int*& ok) {
  red = reinterpret_cast<double*>(smem + ResCap<R, H>::BYTES);
  ok = reinterpret_cast<int*>(red + 16);
}

// One workgroup of NT threads (NT / 64 wavefronts, one per sweep lane) per
// batch scene; H: the LDS layout (0 full, 1 half).
template <typename R, int NT, int H> __global__ void __launch_bounds__(NT) k_solve(Dev<R> d) {
  extern __shared__ __align__(32) unsigned char solve_smem[];
  double* sh_red;
  int* s_ok;
  solve_scratch<R, H>(solve_smem, sh_red, s_ok);
  if (aborted(d.err)) return;
  const int bs = d.bs_order[blockIdx.x];
  const int slot = d.bs_slot[bs];
  const SceneParams& sp = d.sp[slot];
  SceneState& st = d.ss[slot];
  if (d.post && !(sp.use_post_stab && st.post_active)) return;
  double* res = residual_record(d, sp);
  for (int i = threadIdx.x; i < sp.max_iter; i += NT) res[i] = INFINITY;
  if (st.k_cnt == 0) {
    if (threadIdx.x == 0) no_contacts<R>(st);
    return;
  }
  const int u0 = d.u_base[bs], u1 = u0 + d.u_cnt[bs];
  const Group gr{d.l_base[bs], d.l_base[bs] + d.l_cnt[bs], d.u_boff[u0], d.u_boff[u1], true};
  solve_dispatch<R, false, NT, H>(d, slot, gr, solve_smem, sh_red, s_ok);
}

// A single scene (its lanes are its colouring units): the lanes split into
// gridDim.x contiguous blocks, one per workgroup: a cooperative launch if there are several,
// which wait for each other.
template <typename R> __global__ void __launch_bounds__(SOLVE_BLOCK) k_solve_multi(Dev<R> d) {
  extern __shared__ __align__(32) unsigned char solve_smem[];
  double* sh_red;
  int* s_ok;
  solve_scratch<R, 0>(solve_smem, sh_red, s_ok);
  if (aborted(d.err)) return;   // uniform: the flag is set before this launch or not at all
  const int slot = d.bs_slot[0];
  const SceneParams& sp = d.sp[slot];
  SceneState& st = d.ss[slot];
  if (d.post && !(sp.use_post_stab && st.post_active)) return;   // uniform over the grid
  double* res = residual_record(d, sp);
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < sp.max_iter; i += SOLVE_BLOCK) res[i] = INFINITY;
  if (st.k_cnt == 0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) no_contacts<R>(st);
    return;
  }
  const long long nl = *d.n_lanes, G = gridDim.x;
  const int l_lo = (int)(blockIdx.x * nl / G), l_hi = (int)((blockIdx.x + 1) * nl / G);
  const Group gr{l_lo, l_hi, d.u_boff[l_lo], d.u_boff[l_hi], blockIdx.x == 0};
  solve_dispatch<R, true, SOLVE_BLOCK, 0>(d, slot, gr, solve_smem, sh_red, s_ok);
}
