// Edge-collapse (coarsening) pass on the device.
//
//   coarsen_by_size / coarsen_slivers / coarsen / coarsen_verts
//                                    src/Omega_h_coarsen.cpp:29-220
//   check_collapse_class / check_collapse_exposure
//                                    src/Omega_h_check_collapse.cpp:10-117
//   prevent_coarsen_overshoot        src/Omega_h_coarsen_overshoot.cpp:12-49
//   prevent_coarsen_flip             src/Omega_h_coarsen_flip.cpp:14-150,
//                                    src/Omega_h_most_normal.hpp:15-93
//   coarsen_qualities, filter_coarsen_min_qual / _improve
//                                    src/Omega_h_coarsen_qualities.cpp:16-122
//   choose_rails / find_rails        src/Omega_h_collapse_rail.cpp:15-101
//   mark_dead_ents / find_coarsen_domains / coarsen_topology
//                                    src/Omega_h_coarsen_topology.cpp:15-122
//   transfer_coarsen                 src/Omega_h_transfer.cpp:585-619
#include <algorithm>
#include <cstdio>

#include "osh_math.hpp"
#include "osh_passes.hpp"

namespace osh {

namespace {

constexpr I8 kDont = 0;

__device__ __forceinline__ bool collapses(I8 code, int col) { return (code & (1 << col)) != 0; }
__device__ __forceinline__ I8 dont_collapse(I8 code, int col) { return I8(code & ~(1 << col)); }

// the vertices of edges shorter than `shortest`
__global__ void mark_short_edges(LO ne, Real const* lengths, Real shortest, LO const* ev2v,
    I8* vmarks) {
  LO e = thread_index();
  if (e >= ne || !(lengths[e] < shortest)) return;
  vmarks[ev2v[e * 2]] = 1;
  vmarks[ev2v[e * 2 + 1]] = 1;
}

// the collapse directions of each edge: away from its marked ends
// (src/Omega_h_coarsen.cpp:29-47), as far as classification allows
// (check_collapse_class, src/Omega_h_check_collapse.cpp:10-40); `verts` marks
// the vertices that collapse along some edge
__global__ void collapse_codes(LO ne, LO const* ev2v, I8 const* vmarks, I8 const* vdim,
    I8 const* edim, I8* codes, I8* verts) {
  LO e = thread_index();
  if (e >= ne) return;
  LO v[2] = {ev2v[e * 2], ev2v[e * 2 + 1]};
  I8 code = kDont;
  for (int eev = 0; eev < 2; ++eev)
    if (vmarks[v[eev]]) code = I8(code | (1 << eev));
  if (code != kDont) {
    int cds[2] = {vdim[v[0]], vdim[v[1]]};
    int ecd = edim[e];
    if (cds[0] == cds[1]) {
      if (cds[0] != ecd) code = kDont;
    } else {
      for (int col = 0; col < 2; ++col)
        if (cds[col] != ecd) code = dont_collapse(code, col);
    }
  }
  codes[e] = code;
  for (int eev = 0; eev < 2; ++eev)
    if (collapses(code, eev)) verts[v[eev]] = 1;
}

template <int CD>
__device__ __forceinline__ int local_vertex(LO const* cv, LO v) {
  int k = 0;
#pragma unroll
  for (int j = 1; j < CD + 1; ++j)
    if (cv[j] == v) k = j;
  return k;
}

// the cells (faces and tets) of a sweep that looks at each cell's edges and
// sides: job w owns the workgroups [first[w], first[w + 1])
struct CellSweep {
  int n;
  unsigned first[3];
  int dim[2];
  LO ncells[2];
  LO const* c2e[2];
  LO const* cv2v[2];
  LO const* cs2s[2];
  I8* dead_cells[2];
  I8* dead_sides[2];
};

__device__ __forceinline__ int cell_job(CellSweep const& a, LO* c) {
  int w = (a.n > 1 && blockIdx.x >= a.first[1]) ? 1 : 0;
  *c = LO(blockIdx.x - a.first[w]) * kBlock + LO(threadIdx.x);
  return w;
}

constexpr int kLanes = 8;          // threads a key in the product builders below
constexpr int kMaxSideLanes = 32;  // a side's lanes are a 64-bit mask's, shifted into place

// the vertices' metric determinants, which every quality around a vertex
// needs (24 times in a tet mesh)
template <int M>
__global__ void vert_dets(LO nv, Real const* metric, Real* dets) {
  LO v = thread_index();
  if (v >= nv) return;
  constexpr int nc = (M == 2) ? 3 : 6;
  double m[nc];
  for (int k = 0; k < nc; ++k) m[k] = metric[std::size_t(v) * nc + k];
  dets[v] = det<M>(get_symm<M>(m));
}

// coarsen_qualities without its filters: every collapse side's minimum quality
// of the cells that survive, with v_col moved onto v_onto, or -1 for a side
// that is not asked for.  MIXED as in collapse_stars.
struct SideQualities {
  LO const* cands;
  LO const* ev2v;
  LO const* cv2v;
  LO const* v2c_a2ab;
  LO const* v2c_ab2b;
  I8 const* v2c_codes;
  Real const* coords;
  Real const* metric;
  Real const* dets;
  Real qmin;
  I8 const* codes;
  Real* quals;  // by (candidate, direction)
};

// the vertices of a row's cell once its vertex has moved onto v_onto; false if
// it dies
template <int D>
__device__ __forceinline__ bool moved_cell(LO const* cv2v, LO c, int ccv_col, LO v_onto,
    LO (&cv)[D + 1]) {
  bool lives = true;
#pragma unroll
  for (int k = 0; k < D + 1; ++k) {
    cv[k] = cv2v[std::size_t(c) * (D + 1) + k];
    if (k != ccv_col && cv[k] == v_onto) lives = false;
  }
#pragma unroll
  for (int k = 0; k < D + 1; ++k)
    if (k == ccv_col) cv[k] = v_onto;
  return lives;
}

template <int D, int M, bool MIXED>
__global__ void __launch_bounds__(kBlock) coarsen_quality_lanes(LO nt, int lshift,
    SideQualities a) {
  LO t = thread_index();
  if (t >= nt) return;
  LO side = t >> lshift;
  int lanes = 1 << lshift;
  int lane = int(t) & (lanes - 1);
  unsigned long long group = ((1ull << lanes) - 1ull) << (int(threadIdx.x % 64) & ~(lanes - 1));
  LO e = a.cands[side / 2];
  int col = side % 2;
  constexpr int nc = (M == 1) ? 1 : (M == 2 ? 3 : 6);
  bool open = collapses(a.codes[e], col);
  LO v_col = a.ev2v[e * 2 + col];
  LO v_onto = a.ev2v[e * 2 + (1 - col)];
  LO row = open ? a.v2c_a2ab[v_col] : 0;
  LO end = open ? a.v2c_a2ab[v_col + 1] : 0;
  bool rejected = false;
  double const* pp[D + 1];
  double const* ms[D + 1];
  auto points = [&](LO vc, LO (&cv)[D + 1]) {
    if (!moved_cell<D>(a.cv2v, a.v2c_ab2b[vc], code_which_down(a.v2c_codes[vc]), v_onto, cv))
      return false;
    for (int k = 0; k < D + 1; ++k) {
      pp[k] = a.coords + std::size_t(cv[k]) * D;
      ms[k] = a.metric + std::size_t(cv[k]) * nc;
    }
    return true;
  };
  if constexpr (MIXED) {
    float minq = 1.0f;
    bool unclear = false;
    for (LO vc = row + lane; vc < end; vc += lanes) {
      LO cv[D + 1];
      if (!points(vc, cv)) continue;
      float q = f32::element_quality<D, M>(pp, ms, &unclear);
      minq = (q < minq) ? q : minq;
    }
    for (int d = lanes / 2; d > 0; d >>= 1) {
      float o = __shfl_xor(minq, d, 64);
      minq = (o < minq) ? o : minq;
    }
    rejected = open && (__ballot(unclear) & group) == 0ull &&
               double(minq) < a.qmin * (1.0 - double(f32::kScreenBand));
    if (rejected) end = row;
  }
  double minq = 1.0;
  for (LO vc = row + lane; vc < end; vc += lanes) {
    LO cv[D + 1];
    if (!points(vc, cv)) continue;
    double dets[D + 1];
    for (int k = 0; k < D + 1; ++k) dets[k] = a.dets[cv[k]];
    minq = math::min2(minq, element_quality<D, M>(pp, ms, dets));
  }
  for (int d = lanes / 2; d > 0; d >>= 1) minq = math::min2(minq, __shfl_xor(minq, d, 64));
  if (lane == 0) a.quals[side] = (rejected || !open) ? -1.0 : minq;
}

// What a collapsing vertex decides from its star, a wave each:
//  - check_collapse_exposure (src/Omega_h_check_collapse.cpp:64-117): a side is
//    vetoed where a cell around its edge (triangle or tet) has its side opposite
//    the target classified differently from itself;
//  - prevent_coarsen_overshoot: where a new edge would reach max_length;
//  - coarsen_qualities with its filters
//    (src/Omega_h_coarsen_qualities.cpp:16-122): a side is kept when the cells
//    that survive reach qmin and, with `improve`, exceed the old minimum;
//  - choose_rails (src/Omega_h_collapse_rail.cpp:15-60): the shortest edge left,
//    the one of higher quality among equally long ones, the first of those;
//  - the vertex star (verts_across_edges, src/Omega_h_adj.cpp:512-530).
//
// Bound by the issue of vector instructions (all SIMD cycles of a large launch issue
// one, 45 % of them FP64): some 100 operations a new edge, 166 a quality, with
// their correctly rounded divisions.
// A star's vertices are neighbors of all its sides, so they are brought to LDS
// once, and the (target, edge) and (target, cell) pairs of the sides still open
// are dealt out to the lanes together, a few edges or cells of each side at a
// time.  As sweeps of their own with 16 lanes a side, each side gathering the
// star again, exposure, overshoot, qualities and rails took 1.85 ms for 1.9 M
// sides of 275,000 vertices and 165 us for 239,000 sides of which none was
// kept; this takes 1.47 ms and 71 us.
//
// MIXED: FP32 estimates first.  A side is vetoed when an estimated length is
// over max_length by more than the screening band, and measured in FP64 only
// when none is but one lies inside the band; it is rejected when the estimated
// minimum quality is below qmin by more than the band and every cell's
// max-determinant metric was clear, else evaluated in FP64.
struct StarSweep {
  LO nverts;
  LO const* verts;
  LO const* ev2v;
  LO const* e_a2ab;
  LO const* e_ab2b;
  I8 const* e_codes;
  LO const* c_a2ab;
  LO const* c_ab2b;
  I8 const* c_codes;
  LO const* cv2v;
  LO const* c2s;  // the cells' sides
  LO const* f2e;  // 3D: the faces' edges and vertices
  LO const* fv2v;
  I8 const* edim;
  I8 const* sdim;
  I8 const* cdim;
  Real const* coords;
  Real const* metric;
  Real const* lengths;
  Real const* old_quals;  // improve: the elements' qualities (else null)
  Real max_length;
  Real qmin;
  I8 const* codes;
  bool sides_only;  // stop after the overshoot check, with the verdicts in `sides`
  bool checked;     // the codes are those of such a sweep
  I8* large;        // by listed vertex: whether its star does not fit
  unsigned* word;   // receives the tag where one does not (null: not wanted)
  unsigned tag;
  I8* sides;        // by (edge, direction)
  I8* vcand;        // zero on entry
  Real* vqual;
  LO* vrail;
  LO* star;
};

// a wave's star in LDS
template <int D, int M>
struct StarData {
  static constexpr int nc = (M == 1) ? 1 : (M == 2 ? 3 : 6);
  static constexpr int kThreads = 64;
  static constexpr int kEdges = kThreads - 1;  // at most a lane each; kSelf names the last one
  static constexpr int kCells = 128;
  double coords[kThreads * D];
  double metric[kThreads * nc];
  double dets[kThreads];
  double lens[kThreads];
  unsigned long long minq[kThreads];
  LO verts[kThreads];
  unsigned cells[kCells];  // positions of a cell's vertices, a byte each; kSelf: the vertex
  unsigned char list[kThreads];
  I8 edim[kThreads];
  I8 second[kThreads];  // the vertex is its edge's second
  I8 veto[kThreads];
  I8 unsure[kThreads];

  __device__ __forceinline__ static void sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  // lists the sides whose lane says so, in order; how many
  __device__ __forceinline__ int list_sides(bool in, int t) {
    unsigned long long b = __ballot(in);
    sync();
    if (in) list[__popcll(b & ((1ull << t) - 1ull))] = static_cast<unsigned char>(t);
    sync();
    return __popcll(b);
  }
  // op(target, k) for the listed targets and k < n, over the lanes
  template <class Op>
  __device__ __forceinline__ void for_pairs(int nlist, int n, int t, Op const& op) const {
    int at = t / n, k = t % n, step = kThreads / n, rest = kThreads % n;
#pragma unroll 1
    while (at < nlist) {
      op(int(list[at]), k);
      at += step;
      k += rest;
      if (k >= n) {
        k -= n;
        ++at;
      }
    }
  }
  // the same while the sides still stand: few rows of the pairs at a time, the
  // sides vetoed by then left out of the next (a list is some 30 instructions,
  // a quality 500)
  template <class Op>
  __device__ __forceinline__ void for_standing_pairs(int nlist, int n, int t, bool open,
      Op const& op) {
    for (int first = 0; first < n && nlist > 0;) {
      int rows = (nlist > kThreads / 4 ? 2 * kThreads : kThreads) / nlist;
      rows = rows < n - first ? rows : n - first;
#pragma unroll 1
      for (int p = t; p < nlist * rows; p += kThreads) op(int(list[p / rows]), first + p % rows);
      first += rows;
      sync();
      if (first < n) nlist = list_sides(open && !veto[t], t);
    }
  }
  __device__ __forceinline__ static double min_of(double x) {
    for (int d = 32; d > 0; d >>= 1) x = math::min2(x, __shfl_xor(x, d, 64));
    return x;
  }
};
constexpr unsigned kSelf = 0xffu;
constexpr int kLargeStarWord = 2;  // the sets use the words before

// doubles as whole numbers in the same order (atomicMin)
__device__ __forceinline__ unsigned long long ordered(double x) {
  unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(x));
  return (b >> 63) ? ~b : b | (1ull << 63);
}
__device__ __forceinline__ double unordered(unsigned long long b) {
  return __longlong_as_double(
      static_cast<long long>((b >> 63) ? b & ~(1ull << 63) : ~b));
}

// the choice among a vertex's rails so far
struct Rail {
  LO edge = -1;
  double len = 0.0;
  double qual = 0.0;
  __device__ __forceinline__ void visit(LO e, double l, double q) {
    if (edge != -1 && !(l < len || (l == len && q > qual))) return;
    edge = e;
    len = l;
    qual = q;
  }
};

template <int D, int M, bool MIXED>
__device__ __forceinline__ void small_star(StarSweep const& a, LO row, int nedges, LO crow,
    int ncells, int t, StarData<D, M>& s, Rail& rail) {
  using S = StarData<D, M>;
  constexpr int nc = S::nc;
  LO e = -1;
  int eev = 0;
  bool open = false;
  if (t < nedges) {
    e = a.e_ab2b[row + t];
    eev = code_which_down(a.e_codes[row + t]);
    LO u = a.ev2v[e * 2 + 1 - eev];
    open = collapses(a.codes[e], eev);
    if (!a.sides_only) a.star[row + t] = u;
    s.verts[t] = u;
    s.edim[t] = a.edim[e];
    s.second[t] = eev == 1;
    double m[nc];
    for (int k = 0; k < D; ++k) s.coords[t * D + k] = a.coords[std::size_t(u) * D + k];
    for (int k = 0; k < nc; ++k) s.metric[t * nc + k] = m[k] = a.metric[std::size_t(u) * nc + k];
    s.dets[t] = M == 1 ? m[0] : det<M>(get_symm<M>(m));
  }
  s.veto[t] = s.unsure[t] = 0;
  int nopen = s.list_sides(open, t);
  if (!a.checked && nopen) {
    // the ends of the new edge from target w at neighbor u
    auto length_of = [&](auto const& length, int w, int u) {
      int p = s.second[u] ? u : w, q = s.second[u] ? w : u;
      return length(s.coords + p * D, s.coords + q * D, s.metric + p * nc, s.metric + q * nc);
    };
    if constexpr (MIXED) {
      float lmax = float(a.max_length);
      s.for_standing_pairs(nopen, nedges, t, open, [&](int w, int u) {
        if (u == w) return;
        float l = length_of(
            [](auto... x) { return f32::edge_length<D, M>(x...); }, w, u);
        if (l >= lmax * (1.0f + f32::kScreenBand))
          s.veto[w] = 1;
        else if (!(l < lmax * (1.0f - f32::kScreenBand)))
          s.unsure[w] = 1;
      });
      nopen = s.list_sides(open && s.unsure[t] && !s.veto[t], t);
    }
    s.for_standing_pairs(nopen, nedges, t, MIXED ? open && s.unsure[t] : open, [&](int w, int u) {
      if (u == w) return;
      double l = length_of([](auto... x) { return edge_length<D, M>(x...); }, w, u);
      if (l >= a.max_length) s.veto[w] = 1;
    });
    open = open && !s.veto[t];
    nopen = s.list_sides(open, t);
  }
  double vold = 1.79769313486231570815e+308;
  for (int i = t; nopen && i < ncells; i += S::kThreads) {
    LO c = a.c_ab2b[crow + i];
    int at = code_which_down(a.c_codes[crow + i]);
    unsigned pos[D + 1];
    LO cv[D + 1];
#pragma unroll
    for (int k = 0; k < D + 1; ++k) {
      cv[k] = a.cv2v[std::size_t(c) * (D + 1) + k];
      pos[k] = kSelf;
    }
    I8 own = 0, sd[D + 1];
    if (!a.checked) {
      // the side opposite a vertex other than the star's has that one in it
      own = a.cdim[c];
#pragma unroll
      for (int k = 0; k < D + 1; ++k)
        sd[k] = a.sdim[a.c2s[std::size_t(c) * (D + 1) + opposite_template(D, 0, k)]];
    }
    if (a.old_quals && !a.sides_only) vold = math::min2(vold, a.old_quals[c]);
#pragma unroll 2
    for (int j = 0; j < nedges; ++j) {
      LO u = s.verts[j];
#pragma unroll
      for (int k = 0; k < D + 1; ++k)
        if (cv[k] == u) pos[k] = unsigned(j);
    }
    unsigned packed = 0u;
#pragma unroll
    for (int k = 0; k < D + 1; ++k) packed |= pos[k] << (8 * k);
    s.cells[i] = packed;
    if (a.checked) continue;
#pragma unroll
    for (int k = 0; k < D + 1; ++k) {
      if (k == at) continue;
      if (sd[k] != own) s.veto[pos[k] % S::kThreads] = 1;
      if (D == 3) {
        // the triangle's edges from the vertex, each opposite the other's end
        unsigned x = kSelf, y = kSelf;
#pragma unroll
        for (int j = 0; j < D + 1; ++j) {
          if (j == at || j == k) continue;
          y = x;
          x = pos[j];
        }
        x %= S::kThreads;
        y %= S::kThreads;
        if (s.edim[y] != sd[k]) s.veto[x] = 1;
        if (s.edim[x] != sd[k]) s.veto[y] = 1;
      }
    }
  }
  S::sync();
  open = open && !s.veto[t];
  if (a.sides_only) {
    if (t < nedges) a.sides[std::size_t(e) * 2 + eev] = open ? 1 : 0;
    return;
  }
  nopen = s.list_sides(open, t);
  if (nopen == 0) return;
  if (a.old_quals) vold = s.min_of(vold);
  // the positions of cell i's vertices with its vertex moved onto target w;
  // false if it dies
  auto moved = [&](int w, int i, int (&at)[D + 1]) {
    unsigned packed = s.cells[i];
    bool lives = true;
#pragma unroll
    for (int k = 0; k < D + 1; ++k) {
      int j = int((packed >> (8 * k)) & 0xffu);
      lives = lives && j != w;
      at[k] = j == int(kSelf) ? w : j;
    }
    return lives;
  };
  if constexpr (MIXED) {
    // estimated minima, as ordered whole numbers; `unsure`: an unclear metric
    s.unsure[t] = 0;
    s.minq[t] = ordered(1.0);
    S::sync();
    s.for_pairs(nopen, ncells, t, [&](int w, int i) {
      int at[D + 1];
      if (!moved(w, i, at)) return;
      double const* pp[D + 1];
      double const* ms[D + 1];
#pragma unroll
      for (int k = 0; k < D + 1; ++k) {
        pp[k] = s.coords + at[k] * D;
        ms[k] = s.metric + at[k] * nc;
      }
      bool unclear = false;
      float q = f32::element_quality<D, M>(pp, ms, &unclear);
      if (unclear) s.unsure[w] = 1;
      if (q < 1.0f) atomicMin(&s.minq[w], ordered(double(q)));
    });
    S::sync();
    bool rejected =
        !s.unsure[t] && unordered(s.minq[t]) < a.qmin * (1.0 - double(f32::kScreenBand));
    open = open && !rejected;
    nopen = s.list_sides(open, t);
  }
  s.minq[t] = ordered(1.0);
  if (open) s.lens[t] = a.lengths[e];
  s.veto[t] = 0;
  S::sync();
  s.for_standing_pairs(nopen, ncells, t, open, [&](int w, int i) {
    int at[D + 1];
    if (!moved(w, i, at)) return;
    // element_quality, from the positions
    double p[D + 1][D];
    double const* pp[D + 1];
    int best = at[0];
    double maxdet = s.dets[at[0]];
#pragma unroll
    for (int k = 0; k < D + 1; ++k) {
      pp[k] = p[k];
#pragma unroll
      for (int j = 0; j < D; ++j) p[k][j] = s.coords[at[k] * D + j];
      if (s.dets[at[k]] > maxdet) {
        best = at[k];
        maxdet = s.dets[at[k]];
      }
    }
    double q = quality_with<D, M>(pp, get_symm<M>(s.metric + best * nc), maxdet);
    if (q < a.qmin || (a.old_quals && q <= vold))
      s.veto[w] = 1;
    else if (q < 1.0)
      atomicMin(&s.minq[w], ordered(q));
  });
  double minq = unordered(s.minq[t]);
  int nkept = s.list_sides(open && !s.veto[t] && minq >= a.qmin &&
                               (!a.old_quals || minq > vold), t);
  if (t != 0) return;
  for (int i = 0; i < nkept; ++i) {
    int w = s.list[i];
    rail.visit(w, s.lens[w], unordered(s.minq[w]));
  }
  if (nkept) rail.edge = a.e_ab2b[row + rail.edge];
}

// The stars that do not fit a wave's LDS, of any size: their sides (in row order,
// after those of the listed stars before) a wave each, from memory, and then the
// rail of each star from the sides kept.  A few such stars among thousands are
// the usual case, and their sides are all the parallelism there is: a pass over
// a fan of 600 edges takes 0.52 ms in 2D and 0.36 in 3D, 8.5 and 12.8 when one
// wave took a star's sides one after another.  With 129 edges it takes 0.27 and
// 0.29, against 0.38 and 0.48 with a workgroup and its LDS a star; a thousand stars of
// 100 edges are the one case seen where that form was faster (0.70 against 0.86).
struct LargeStars {
  LO nstars;
  LO nsides;
  LO const* stars;    // positions in StarSweep::verts
  LO const* offsets;  // by star: its first side
  I8* kept;           // by side
  Real* quals;        // the minimum quality where kept
};

template <int D, int M, bool MIXED>
__global__ void __launch_bounds__(kBlock) large_star_sides(StarSweep a, LargeStars g) {
  constexpr int nc = StarData<D, M>::nc;
  int lane = int(threadIdx.x) % 64;
  LO step = LO(gridDim.x) * (kBlock / 64);
  for (LO side = LO(blockIdx.x) * (kBlock / 64) + LO(threadIdx.x) / 64; side < g.nsides;
       side += step) {
    LO star = row_of(side, g.nstars, g.offsets);
    LO v = a.verts[g.stars[star]];
    LO row = a.e_a2ab[v], end = a.e_a2ab[v + 1];
    LO crow = a.c_a2ab[v], cend = a.c_a2ab[v + 1];
    LO vw = row + (side - g.offsets[star]);
    LO e = a.e_ab2b[vw];
    int eev = code_which_down(a.e_codes[vw]);
    LO onto = a.ev2v[e * 2 + 1 - eev];
    if (!a.sides_only && lane == 0) {
      a.star[vw] = onto;
      g.kept[side] = 0;
    }
    bool open = collapses(a.codes[e], eev);
    if (open && !a.checked) {
      bool veto = false;
      for (LO vc = crow + lane; vc < cend; vc += 64) {
        LO c = a.c_ab2b[vc];
        int at = code_which_down(a.c_codes[vc]);
        int k_onto = -1;
        for (int k = 0; k < D + 1; ++k)
          if (a.cv2v[std::size_t(c) * (D + 1) + k] == onto) k_onto = k;
        if (k_onto < 0) continue;
        for (int k = 0; k < D + 1; ++k) {
          if (k == at) continue;
          LO f = a.c2s[std::size_t(c) * (D + 1) + opposite_template(D, 0, k)];
          if (k == k_onto) {
            veto = veto || a.sdim[f] != a.cdim[c];
          } else if (D == 3) {
            int j = local_vertex<2>(a.fv2v + std::size_t(f) * 3, onto);
            veto = veto || a.edim[a.f2e[std::size_t(f) * 3 + opposite_template(2, 0, j)]] != a.sdim[f];
          }
        }
      }
      bool unsure = !MIXED;
      bool over = false;
      auto length_of = [&](auto const& length, LO ve) {
        LO e2 = a.e_ab2b[ve];
        int in = code_which_down(a.e_codes[ve]);
        LO out = a.ev2v[e2 * 2 + 1 - in];
        LO p = in == 0 ? onto : out, q = in == 0 ? out : onto;
        return length(a.coords + std::size_t(p) * D, a.coords + std::size_t(q) * D,
            a.metric + std::size_t(p) * nc, a.metric + std::size_t(q) * nc);
      };
      if constexpr (MIXED) {
        float lmax = float(a.max_length);
        for (LO ve = row + lane; ve < end; ve += 64) {
          if (ve == vw) continue;
          float l = length_of([](auto... x) { return f32::edge_length<D, M>(x...); }, ve);
          over = over || l >= lmax * (1.0f + f32::kScreenBand);
          unsure = unsure || !(l < lmax * (1.0f - f32::kScreenBand));
        }
      }
      veto = __any(veto || over);
      if (!veto && __any(unsure)) {
        for (LO ve = row + lane; ve < end && !over; ve += 64)
          if (ve != vw)
            over = length_of([](auto... x) { return edge_length<D, M>(x...); }, ve) >=
                   a.max_length;
        veto = __any(over);
      }
      open = !veto;
    }
    if (a.sides_only) {
      if (lane == 0) a.sides[std::size_t(e) * 2 + eev] = open ? 1 : 0;
      continue;
    }
    if (!open) continue;
    double const* pp[D + 1];
    double const* ms[D + 1];
    auto moved = [&](LO vc) {
      LO cv[D + 1];
      if (!moved_cell<D>(a.cv2v, a.c_ab2b[vc], code_which_down(a.c_codes[vc]), onto, cv))
        return false;
      for (int k = 0; k < D + 1; ++k) {
        pp[k] = a.coords + std::size_t(cv[k]) * D;
        ms[k] = a.metric + std::size_t(cv[k]) * nc;
      }
      return true;
    };
    if constexpr (MIXED) {
      double least = 1.0;
      bool unclear = false;
      for (LO vc = crow + lane; vc < cend; vc += 64)
        if (moved(vc)) least = math::min2(least, f32::element_quality<D, M>(pp, ms, &unclear));
      least = StarData<D, M>::min_of(least);
      if (!__any(unclear) && least < a.qmin * (1.0 - double(f32::kScreenBand))) continue;
    }
    double vold = 1.79769313486231570815e+308;
    double minq = 1.0;
    for (LO vc = crow + lane; vc < cend; vc += 64) {
      if (a.old_quals) vold = math::min2(vold, a.old_quals[a.c_ab2b[vc]]);
      if (!moved(vc)) continue;
      double dets[D + 1];
#pragma unroll
      for (int k = 0; k < D + 1; ++k) dets[k] = M == 1 ? ms[k][0] : det<M>(get_symm<M>(ms[k]));
      minq = math::min2(minq, element_quality<D, M>(pp, ms, dets));
    }
    vold = StarData<D, M>::min_of(vold);
    minq = StarData<D, M>::min_of(minq);
    if (lane == 0 && minq >= a.qmin && (!a.old_quals || minq > vold)) {
      g.kept[side] = 1;
      g.quals[side] = minq;
    }
  }
}

__global__ void large_star_degrees(LO n, LO const* stars, LO const* verts, LO const* a2ab,
    LO* degrees) {
  LO i = thread_index();
  if (i >= n) return;
  LO v = verts[stars[i]];
  degrees[i] = a2ab[v + 1] - a2ab[v];
}

// a wave a star: the kept sides in row order
__global__ void __launch_bounds__(kBlock) large_star_rails(StarSweep a, LargeStars g) {
  LO star = LO(blockIdx.x) * (kBlock / 64) + LO(threadIdx.x) / 64;
  int lane = int(threadIdx.x) % 64;
  if (star >= g.nstars) return;
  LO v = a.verts[g.stars[star]];
  LO row = a.e_a2ab[v], n = a.e_a2ab[v + 1] - row;
  LO first = g.offsets[star];
  Rail rail;
  for (LO base = 0; base < n; base += 64) {
    LO j = base + lane;
    bool kept = j < n && g.kept[first + j];
    LO e = kept ? a.e_ab2b[row + j] : -1;
    double len = kept ? a.lengths[e] : 0.0;
    double q = kept ? g.quals[first + j] : 0.0;
    for (unsigned long long b = __ballot(kept); b; b &= b - 1) {
      int k = __ffsll(static_cast<long long>(b)) - 1;
      rail.visit(__shfl(e, k, 64), __shfl(len, k, 64), __shfl(q, k, 64));
    }
  }
  if (lane != 0 || rail.edge < 0) return;
  a.vcand[v] = 1;
  a.vqual[v] = rail.qual;
  a.vrail[v] = rail.edge;
}

// a wave a star, four stars a workgroup; a star that does not fit is told in
// `large` and by `word`, and left to the sweep above
template <int D, int M, bool MIXED>
__global__ void __launch_bounds__(kBlock, 5) collapse_stars(StarSweep a) {
  constexpr int kStars = kBlock / 64;
  using S = StarData<D, M>;
  __shared__ S data[kStars];
  int star = int(threadIdx.x) / 64, t = int(threadIdx.x) % 64;
  std::int64_t i = std::int64_t(blockIdx.x) * kStars + star;
  if (i >= a.nverts) return;
  LO v = a.verts[i];
  LO row = a.e_a2ab[v], end = a.e_a2ab[v + 1];
  LO crow = a.c_a2ab[v], cend = a.c_a2ab[v + 1];
  bool fits = end - row <= S::kEdges && cend - crow <= S::kCells;
  if (t == 0) a.large[i] = fits ? 0 : 1;
  if (!fits) {
    if (t == 0 && a.word)
      __hip_atomic_store(a.word, a.tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
  Rail rail;
  small_star<D, M, MIXED>(a, row, int(end - row), crow, int(cend - crow), t, data[star], rail);
  if (a.sides_only || t != 0 || rail.edge < 0) return;
  a.vcand[v] = 1;
  a.vqual[v] = rail.qual;
  a.vrail[v] = rail.edge;
}

// drops the candidates' directions that a sweep has vetoed
__global__ void drop_sides(LO n, LO const* cands, I8 const* sides, I8* codes) {
  LO i = thread_index();
  if (i >= n) return;
  LO e = cands[i];
  I8 code = codes[e];
  for (int col = 0; col < 2; ++col)
    if (collapses(code, col) && !sides[std::size_t(e) * 2 + col]) code = dont_collapse(code, col);
  codes[e] = code;
}

__global__ void scatter_codes(LO n, LO const* cands, I8 const* cand_codes, I8* codes) {
  LO i = thread_index();
  if (i < n) codes[cands[i]] = cand_codes[i];
}

// mark_dead_ents (src/Omega_h_coarsen_topology.cpp:15-60): the rails die,
// and so do the cells around a rail and each such cell's side opposite the
// target vertex; rail_col[e] is the collapsing end of rail e (-1 elsewhere),
// onto[v] a key's target vertex
__global__ void mark_rails(LO nv, I8 const* keys, LO const* vrail, LO const* ev2v,
    I8* dead_edges, I8* rail_col, LO* onto) {
  LO v = thread_index();
  if (v >= nv || !keys[v]) return;
  LO e = vrail[v];
  int eev = ev2v[e * 2] == v ? 0 : 1;
  dead_edges[e] = 1;
  rail_col[e] = I8(eev);
  onto[v] = ev2v[e * 2 + 1 - eev];
}

template <int CD>
__device__ __forceinline__ void mark_dead(LO c, CellSweep const& a, int w, LO const* ev2v,
    I8 const* rail_col) {
  if (c >= a.ncells[w]) return;
  constexpr int nepc = (CD == 3) ? 6 : 3;
  for (int j = 0; j < nepc; ++j) {
    LO e = a.c2e[w][std::size_t(c) * nepc + j];
    int col = rail_col[e];
    if (col < 0) continue;
    int ccv_onto =
        local_vertex<CD>(a.cv2v[w] + std::size_t(c) * (CD + 1), ev2v[e * 2 + (1 - col)]);
    a.dead_cells[w][c] = 1;
    a.dead_sides[w][a.cs2s[w][std::size_t(c) * (CD + 1) + opposite_template(CD, 0, ccv_onto)]] =
        1;
  }
}

__global__ void __launch_bounds__(kBlock) mark_dead_cells(CellSweep a, LO const* ev2v,
    I8 const* rail_col) {
  LO c;
  int w = cell_job(a, &c);
  if (a.dim[w] == 3)
    mark_dead<3>(c, a, w, ev2v, rail_col);
  else
    mark_dead<2>(c, a, w, ev2v, rail_col);
}

// a key's products are the live entries of its vertex's row, in row order;
// kLanes threads per vertex count those of every dimension (0 for vertices
// that are no keys)
struct LiveRows {
  int n;
  LO const* a2ab[3];
  LO const* ab2b[3];
  I8 const* dead[3];
  LO* counts[3];
};

__global__ void live_counts(std::int64_t nt, I8 const* keys, LiveRows r) {
  std::int64_t t = thread_index64();
  if (t >= nt) return;
  LO v = LO(t / kLanes);
  int lane = int(t % kLanes);
  bool key = keys[v] != 0;
  for (int d = 0; d < r.n; ++d) {
    LO n = 0;
    if (key) {
      LO end = r.a2ab[d][v + 1];
      for (LO j = r.a2ab[d][v] + lane; j < end; j += kLanes) n += !r.dead[d][r.ab2b[d][j]];
      for (int k = kLanes / 2; k > 0; k >>= 1) n += __shfl_xor(n, k, 64);
    }
    if (lane == 0) r.counts[d][v] = n;
  }
}

// the products of every dimension in one launch: a round of kLanes row entries
// at a time, whose live ones take the next products in row order (a ballot
// gives each its rank; counting the live entries before each one in the row
// cost 28 us a launch on the 64^3 workload)
struct CoarsenRows {
  LO const* a2ab[3];
  LO const* ab2b[3];
  I8 const* codes[3];
  I8 const* dead[3];
  LO const* verts[3];
  LO const* keys2prods[3];
  LO* pv[3];
  LO* psrc[3];
};

__global__ void coarsen_products(std::int64_t nt, LO nkeys, LO const* keys2verts,
    LO const* onto_of, LO const* vert_offsets, CoarsenRows r) {
  std::int64_t t = thread_index64();
  if (t >= nt) return;
  std::int64_t row = t / kLanes;
  int d = int(row / nkeys);
  LO k = LO(row % nkeys);
  int lane = int(t % kLanes);
  int base = int(threadIdx.x % 64) & ~(kLanes - 1);
  int nvd = d + 2;
  LO v = keys2verts[k];
  LO onto = onto_of[v];
  LO e = r.a2ab[d][v + 1];
  LO prod = r.keys2prods[d][k];
  for (LO b = r.a2ab[d][v]; b < e; b += kLanes) {
    LO j = b + lane;
    LO cell = j < e ? r.ab2b[d][j] : 0;
    bool live = j < e && !r.dead[d][cell];
    unsigned mask = unsigned(__ballot(live) >> base) & ((1u << kLanes) - 1u);
    if (live) {
      LO p = prod + __popc(mask & ((1u << lane) - 1u));
      int ccv_col = code_which_down(r.codes[d][j]);
      for (int ccv = 0; ccv < nvd; ++ccv) {
        LO ov = (ccv == ccv_col) ? onto : r.verts[d][std::size_t(cell) * nvd + ccv];
        r.pv[d][std::size_t(p) * nvd + ccv] = vert_offsets[ov];
      }
      r.psrc[d][p] = cell;
    }
    prod += __popc(mask);
  }
}

// ---- prevent_coarsen_flip (src/Omega_h_coarsen_flip.cpp:68-150), taken
// only when AdaptOpts::should_prevent_coarsen_flip is set.  Exposed sides
// (fewer than two elements) around a vertex of a candidate edge "matter", and
// so do their vertices; each such vertex gets a normal, and a collapse
// direction is vetoed when a surviving side that matters around the
// collapsing vertex would turn so that its normal has a dot product below
// 1e-10 with the normal of one of its vertices.

// get_side_vector (src/Omega_h_shape.hpp:276-298): the triangle's
// (b - a) x (c - a) in 3D, -perp(b - a) in 2D
template <int D>
__device__ __forceinline__ void side_vector(double const* const* p, double* out) {
  if (D == 3) {
    double u[3], w[3];
    for (int i = 0; i < 3; ++i) {
      u[i] = p[1][i] - p[0][i];
      w[i] = p[2][i] - p[0][i];
    }
    cross3(u, w, out);
  } else {
    double v0 = p[1][0] - p[0][0], v1 = p[1][1] - p[0][1];
    out[0] = -(-v1);
    out[1] = -v0;
  }
}

template <int D>
__device__ __forceinline__ void normalize_vec(double* v) {
  double l = vnorm<D>(v);
  for (int i = 0; i < D; ++i) v[i] = v[i] / l;
}

__device__ __forceinline__ bool close_rel(double a, double b) {
  double am = math::fabs_(a), bm = math::fabs_(b);
  if (am <= 1e-10 && bm <= 1e-10) return true;
  return math::fabs_(b - a) / math::max2(am, bm) <= 1e-10;
}

// get_most_normal_normal (src/Omega_h_most_normal.hpp:15-93; Aubry and
// Lohner 2008): the centre of the smallest spherical cap holding the n unit
// vectors, from pairs (their normalized bisector) and then from triplets
// (the direction with one dot product with all three, from the inverse of
// the matrix whose rows are the three).  In 2D the normalized sum of the
// first two.  False where the reference's checks fail.
template <int D>
__device__ bool most_normal(int n, double const* N, double* c) {
  if (D == 2) {
    c[0] = N[0] + N[2];
    c[1] = N[1] + N[3];
    normalize_vec<2>(c);
    return true;
  }
  double const tol = 1e-10;
  double scalmin = -1.0;
  c[0] = c[1] = c[2] = 0.0;
  for (int i = 0; i < n; ++i) {
    for (int j = i + 1; j < n; ++j) {
      double b[3];
      for (int k = 0; k < 3; ++k) b[k] = N[i * 3 + k] + N[j * 3 + k];
      normalize_vec<3>(b);
      double scal = dot<3>(b, N + i * 3);
      if (scal < scalmin) continue;
      int l;
      for (l = 0; l < n; ++l)
        if (dot<3>(N + l * 3, b) + tol < scal) break;
      if (l < n) continue;
      for (int k = 0; k < 3; ++k) c[k] = b[k];
      scalmin = scal;
    }
  }
  if (scalmin != -1.0) return true;
  for (int i = 0; i < n; ++i) {
    for (int j = i + 1; j < n; ++j) {
      for (int k = j + 1; k < n; ++k) {
        Mat M;  // columns N_i, N_j, N_k
        for (int r = 0; r < 3; ++r) {
          M.m[0][r] = N[i * 3 + r];
          M.m[1][r] = N[j * 3 + r];
          M.m[2][r] = N[k * 3 + r];
        }
        if (math::fabs_(det<3>(M)) < 1e-6) continue;
        // invert(transpose(M)) * (1, 1, 1) (src/Omega_h_matrix.hpp:89-94,
        // 344-350): rows of the cofactor matrix from the cross products of
        // the transpose's columns, divided by its determinant, summed
        // column by column
        Mat T = transpose<3>(M);
        double bm[3][3];
        for (int a = 0; a < 3; ++a) cross3(T.m[(a + 1) % 3], T.m[(a + 2) % 3], bm[a]);
        double dt = det<3>(T);
        double nc[3];
        for (int r = 0; r < 3; ++r) {
          double s = (bm[r][0] / dt) * 1.0;
          s = s + (bm[r][1] / dt) * 1.0;
          s = s + (bm[r][2] / dt) * 1.0;
          nc[r] = s;
        }
        normalize_vec<3>(nc);
        double scal = dot<3>(nc, N + i * 3);
        if (!close_rel(scal, dot<3>(nc, N + j * 3)) || !close_rel(scal, dot<3>(nc, N + k * 3)))
          return false;
        if (scal < scalmin) continue;
        int l;
        for (l = 0; l < n; ++l)
          if (dot<3>(N + l * 3, nc) + tol < scal) break;
        if (l < n) continue;
        for (int q = 0; q < 3; ++q) c[q] = nc[q];
        scalmin = scal;
      }
    }
  }
  return scalmin > -1.0;
}

__global__ void flip_vert_cands(LO ncands, LO const* cands, LO const* ev2v, I8 const* codes,
    I8* vcand) {
  LO i = thread_index();
  if (i >= ncands) return;
  LO e = cands[i];
  if (codes[e] == kDont) return;
  vcand[ev2v[e * 2]] = 1;
  vcand[ev2v[e * 2 + 1]] = 1;
}

// mark_exposed_sides (src/Omega_h_mark.cpp:12-19) and the sides and
// vertices that matter (src/Omega_h_coarsen_flip.cpp:128-134)
__global__ void flip_sides(LO ns, int nsv, LO const* sv2v, unsigned long long const* side_elems,
    I8 const* vcand, I8* exposed, I8* smatter, I8* vmatter) {
  LO s = thread_index();
  if (s >= ns) return;
  I8 ex = (side_elems[s] >> 32) < 2 ? 1 : 0;
  bool adj = false;
  for (int k = 0; k < nsv; ++k) adj = adj || vcand[sv2v[s * nsv + k]] != 0;
  I8 mt = (adj && ex) ? 1 : 0;
  exposed[s] = ex;
  smatter[s] = mt;
  if (mt)
    for (int k = 0; k < nsv; ++k) vmatter[sv2v[s * nsv + k]] = 1;
}

// compute_flip_normals_dim (src/Omega_h_coarsen_flip.cpp:14-64): zero for
// vertices that do not matter
template <int D>
__global__ void flip_normals(LO nv, LO const* a2ab, LO const* ab2b, LO const* sv2v,
    Real const* coords, I8 const* exposed, I8 const* vmatter, Real* normals, int* error) {
  constexpr int kMaxAdj = (D == 3) ? 24 : 8;
  LO v = thread_index();
  if (v >= nv) return;
  double Nc[D];
  for (int k = 0; k < D; ++k) Nc[k] = 0.0;
  if (vmatter[v]) {
    double N[kMaxAdj * D];
    int n = 0;
    for (LO vs = a2ab[v]; vs < a2ab[v + 1]; ++vs) {
      LO s = ab2b[vs];
      if (!exposed[s]) continue;
      if (n >= kMaxAdj) {
        *error = kFlipNormals;
        return;
      }
      double const* p[D];
      for (int k = 0; k < D; ++k) p[k] = coords + size_t(sv2v[s * D + k]) * D;
      double sv[3];
      side_vector<D>(p, sv);
      for (int k = 0; k < D; ++k) Nc[k] = Nc[k] + sv[k];
      double l = vnorm<D>(sv);
      for (int k = 0; k < D; ++k) N[n * D + k] = sv[k] / l;
      ++n;
    }
    normalize_vec<D>(Nc);
    int i;
    for (i = 0; i < n; ++i)
      if (dot<D>(Nc, N + i * D) < 0.95) break;
    if (i < n && !most_normal<D>(n, N, Nc)) {
      *error = kFlipNormals;
      return;
    }
  }
  for (int k = 0; k < D; ++k) normals[size_t(v) * D + k] = Nc[k];
}

// prevent_coarsen_flip2_dim (src/Omega_h_coarsen_flip.cpp:70-121)
template <int D>
__global__ void flip_veto(LO ncands, LO const* cands, LO const* ev2v, LO const* a2ab,
    LO const* ab2b, I8 const* vs_codes, LO const* sv2v, Real const* coords,
    Real const* normals, I8 const* smatter, I8 const* vmatter, I8* codes) {
  LO i = thread_index();
  if (i >= ncands) return;
  LO e = cands[i];
  I8 code = codes[e];
  if (code == kDont) return;
  for (int col = 0; col < 2; ++col) {
    if (!collapses(code, col)) continue;
    LO v_col = ev2v[e * 2 + col];
    if (!vmatter[v_col]) continue;
    LO v_onto = ev2v[e * 2 + (1 - col)];
    for (LO vs = a2ab[v_col]; vs < a2ab[v_col + 1]; ++vs) {
      LO s = ab2b[vs];
      if (!smatter[s]) continue;
      int ssv_col = vs_codes[vs] >> 3;
      LO sv[D];
      int k;
      for (k = 0; k < D; ++k) sv[k] = sv2v[s * D + k];
      for (k = 0; k < D; ++k)
        if (sv[k] == v_onto) break;
      if (k != D) continue;
      sv[ssv_col] = v_onto;
      double const* p[D];
      for (k = 0; k < D; ++k) p[k] = coords + size_t(sv[k]) * D;
      double sn[3];
      side_vector<D>(p, sn);
      for (k = 0; k < D; ++k)
        if (dot<D>(normals + size_t(sv[k]) * D, sn) < 1e-10) break;
      if (k < D) code = dont_collapse(code, col);
    }
  }
  codes[e] = code;
}

// the whole check on the candidates' codes, in place
void prevent_coarsen_flip(Ctx& c, DMesh& m, LOs const& cands, Bytes& codes) {
  Range range(c, "prevent_coarsen_flip");
  int dim = m.dim;
  int sd = dim - 1;
  LO nv = m.nents[0], ns = m.nents[sd];
  LO ncands = cands.size();
  LO const* ev2v = m.down[1].data();
  LOs const& sv2v = verts_of(c, m, sd);
  Adj const& v2s = ask_up(c, m, 0, sd);
  auto const& se = ask_side_elems(c, m);
  Bytes vcand = fill_i8(c, nv, 0);
  OSH_LAUNCH(flip_vert_cands, ncands, c, cands.data(), ev2v, codes.data(), vcand.data());
  Bytes exposed(c, ns), smatter(c, ns);
  Bytes vmatter = fill_i8(c, nv, 0);
  OSH_LAUNCH(flip_sides, ns, c, sd + 1, sv2v.data(), se.data(), vcand.data(), exposed.data(),
      smatter.data(), vmatter.data());
  Reals normals(c, LO(nv * dim));
  if (dim == 3) {
    OSH_LAUNCH(flip_normals<3>, nv, c, v2s.a2ab.data(), v2s.ab2b.data(), sv2v.data(),
        m.coords.data(), exposed.data(), vmatter.data(), normals.data(), c.error_word());
    OSH_LAUNCH(flip_veto<3>, ncands, c, cands.data(), ev2v, v2s.a2ab.data(), v2s.ab2b.data(),
        v2s.codes.data(), sv2v.data(), m.coords.data(), normals.data(), smatter.data(),
        vmatter.data(), codes.data());
  } else {
    OSH_LAUNCH(flip_normals<2>, nv, c, v2s.a2ab.data(), v2s.ab2b.data(), sv2v.data(),
        m.coords.data(), exposed.data(), vmatter.data(), normals.data(), c.error_word());
    OSH_LAUNCH(flip_veto<2>, ncands, c, cands.data(), ev2v, v2s.a2ab.data(), v2s.ab2b.data(),
        v2s.codes.data(), sv2v.data(), m.coords.data(), normals.data(), smatter.data(),
        vmatter.data(), codes.data());
  }
}

// the determinants of the vertices' metrics (a scalar metric is its own)
Reals metric_dets(Ctx& c, DMesh& m) {
  if (m.metric_ncomps == 1) return m.metric;
  LO nv = m.nents[0];
  Reals d(c, nv);
  if (m.metric_ncomps == 6)
    OSH_LAUNCH(vert_dets<3>, nv, c, m.metric.data(), d.data());
  else
    OSH_LAUNCH(vert_dets<2>, nv, c, m.metric.data(), d.data());
  return d;
}

// a kernel template over dimension, metric dimension and precision
#define OSH_BY_FORM(LAUNCH, dim, md, mixed) \
  do {                                      \
    if (dim == 3 && md == 3 && mixed)       \
      LAUNCH(3, 3, true);                   \
    else if (dim == 3 && md == 3)           \
      LAUNCH(3, 3, false);                  \
    else if (dim == 3 && mixed)             \
      LAUNCH(3, 1, true);                   \
    else if (dim == 3)                      \
      LAUNCH(3, 1, false);                  \
    else if (md == 2 && mixed)              \
      LAUNCH(2, 2, true);                   \
    else if (md == 2)                       \
      LAUNCH(2, 2, false);                  \
    else if (mixed)                         \
      LAUNCH(2, 1, true);                   \
    else                                    \
      LAUNCH(2, 1, false);                  \
  } while (0)

void sweep_stars(Ctx& c, int dim, int md, bool mixed, StarSweep const& a) {
  unsigned blocks = unsigned((std::int64_t(a.nverts) * 64 + kBlock - 1) / kBlock);
#define OSH_STARS(D, M, X) \
  hipLaunchKernelGGL((collapse_stars<D, M, X>), dim3(blocks), dim3(kBlock), 0, c.stream, a)
  OSH_BY_FORM(OSH_STARS, dim, md, mixed);
#undef OSH_STARS
  OSH_HIP(hipGetLastError());
}

// the stars that the sweep has told as large
void sweep_large_stars(Ctx& c, int dim, int md, bool mixed, StarSweep const& a,
    LOs const& stars) {
  LO n = stars.size();
  if (n == 0) return;
  LOs degrees(c, n);
  OSH_LAUNCH(large_star_degrees, n, c, stars.data(), a.verts, a.e_a2ab, degrees.data());
  LargeStars g{};
  LOs offsets = offset_scan(c, degrees, &g.nsides);
  Bytes kept(c, g.nsides);
  Reals quals(c, g.nsides);
  g.nstars = n;
  g.stars = stars.data();
  g.offsets = offsets.data();
  g.kept = kept.data();
  g.quals = quals.data();
  // more waves than the device holds at a time take several sides each
  unsigned blocks = std::min(unsigned((std::int64_t(g.nsides) * 64 + kBlock - 1) / kBlock), 1u << 16);
#define OSH_SIDES(D, M, X) \
  hipLaunchKernelGGL((large_star_sides<D, M, X>), dim3(blocks), dim3(kBlock), 0, c.stream, a, g)
  OSH_BY_FORM(OSH_SIDES, dim, md, mixed);
#undef OSH_SIDES
  OSH_HIP(hipGetLastError());
  if (a.sides_only) return;
  hipLaunchKernelGGL(large_star_rails, dim3(nblocks(n, kBlock / 64)), dim3(kBlock), 0, c.stream, a,
      g);
  OSH_HIP(hipGetLastError());
}

// Up to this many cells the collapsing vertices' rows of all dimensions are
// built at once, in order; beyond, the faces' (and ordered cells') rows are
// built for the chosen keys alone.  The five launches of the second inversion
// take some 25 us; for all candidates it adds about 10 us at 30,000 cells.
constexpr LO kJointCells = 32768;

// the pass's arrays that start out constant, in one launch for the attempt and
// another for the rebuild, or all in the first in small meshes
struct CoarsenArrays {
  bool joint;
  // by vertex
  Bytes wanted;      // collapses of these are tried
  Bytes collapsing;  // those that have a candidate edge
  Bytes cand;        // those that have a rail
  LOs up_zeros, key_up_zeros, side_zeros;
  // by entity
  Bytes dead[4];
  Bytes rail_col;
  KeyedMods km;

  CoarsenArrays(DMesh const& m, Fills& fills, bool with_wanted) {
    joint = m.nents[m.dim] <= kJointCells;
    LO nv = m.nents[0];
    if (with_wanted) wanted = fills.bytes(nv, 0);
    collapsing = fills.bytes(nv, 0);
    cand = fills.bytes(nv, 0);
    up_zeros = fills.ints(nv * (joint ? m.dim : 2), 0);
    if (joint) add_rebuild(m, fills);
  }
  void add_rebuild(DMesh const& m, Fills& fills) {
    for (int d = 1; d <= m.dim; ++d) dead[d] = fills.bytes(m.nents[d], 0);
    rail_col = fills.bytes(m.nents[1], -1);
    prepare_keys(m, 0, 0, m.dim, fills, km);
    if (!joint) key_up_zeros = fills.ints(m.nents[0] * (m.dim - 1), 0);
    side_zeros = fills.ints(m.nents[0] * (m.dim - 1), 0);
  }
};

bool coarsen_verts(Ctx& c, DMesh& m, AdaptOptions const& o, CoarsenArrays& vm,
    bool overshoot_allowed, bool improve, SliverLayers* layers = nullptr) {
  int dim = m.dim;
  LO ne = m.nents[1];
  LO nv = m.nents[0];
  int nc = m.metric_ncomps;
  int md = (nc == 1) ? 1 : dim;
  LO const* ev2v = m.down[1].data();
  Bytes codes(c, ne);
  OSH_LAUNCH(collapse_codes, ne, c, ev2v, vm.wanted.data(), m.class_dim[0].data(),
      m.class_dim[1].data(), codes.data(), vm.collapsing.data());
  LOs verts = collect_marked(c, vm.collapsing);
  if (verts.size() == 0) return false;
  // upward rows only where the candidates look: the collapsing vertices' edges
  // (ordered: the first best rail is kept) and cells (order-free minima)
  Adj v2d[4];
  if (vm.joint) {
    int const highs[3] = {1, 2, 3};
    bool const sorted[3] = {true, true, true};
    marked_ups(c, m, 0, vm.collapsing, dim, highs, sorted, v2d + 1, &vm.up_zeros);
  } else {
    Adj up[2];
    int const highs[2] = {1, dim};
    bool const sorted[2] = {true, false};
    marked_ups(c, m, 0, vm.collapsing, 2, highs, sorted, up, &vm.up_zeros);
    v2d[1] = up[0];
    v2d[dim] = up[1];
  }
  Adj const v2e = v2d[1];
  Adj const v2c = v2d[dim];
  Range quality_range(c, "coarsen_qualities");
  Reals vqual(c, nv);
  LOs vrail(c, nv);
  // the independent set reads the star rows of candidate vertices only
  Adj star;
  star.a2ab = v2e.a2ab;
  star.ab2b = LOs(c, v2e.ab2b.size());
  StarSweep sw{};
  sw.nverts = verts.size();
  sw.verts = verts.data();
  sw.ev2v = ev2v;
  sw.e_a2ab = v2e.a2ab.data();
  sw.e_ab2b = v2e.ab2b.data();
  sw.e_codes = v2e.codes.data();
  sw.c_a2ab = v2c.a2ab.data();
  sw.c_ab2b = v2c.ab2b.data();
  sw.c_codes = v2c.codes.data();
  sw.cv2v = verts_of(c, m, dim).data();
  sw.c2s = m.down[dim].data();
  if (dim == 3) {
    sw.f2e = m.down[2].data();
    sw.fv2v = verts_of(c, m, 2).data();
  }
  sw.edim = m.class_dim[1].data();
  sw.sdim = m.class_dim[dim - 1].data();
  sw.cdim = m.class_dim[dim].data();
  sw.coords = m.coords.data();
  sw.metric = m.metric.data();
  sw.lengths = ask_lengths(c, m).data();
  sw.old_quals = improve ? ask_qualities(c, m).data() : nullptr;
  sw.max_length = overshoot_allowed ? o.max_length_allowed : o.max_length_desired;
  sw.qmin = o.min_quality_allowed;
  sw.codes = codes.data();
  sw.vcand = vm.cand.data();
  sw.vqual = vqual.data();
  sw.vrail = vrail.data();
  sw.star = star.ab2b.data();
  bool mixed = o.precision == 1;
  Bytes large(c, verts.size());
  sw.large = large.data();
  bool any;
  Bytes keys;
  if (o.should_prevent_coarsen_flip) {
    // the flip check looks at the edges that the overshoot check leaves
    LOs cands = collect_marked(c, codes);
    Bytes sides(c, ne * 2);
    sw.sides_only = true;
    sw.sides = sides.data();
    sweep_stars(c, dim, md, mixed, sw);
    LOs stars = collect_marked(c, large);
    sweep_large_stars(c, dim, md, mixed, sw, stars);
    OSH_LAUNCH(drop_sides, cands.size(), c, cands.data(), sides.data(), codes.data());
    prevent_coarsen_flip(c, m, cands, codes);
    sw.sides_only = false;
    sw.checked = true;
    sweep_stars(c, dim, md, mixed, sw);
    sweep_large_stars(c, dim, md, mixed, sw, stars);
    quality_range.end();
    keys = find_indset(c, m, 0, vqual, vm.cand, &any, nullptr, &star);
  } else {
    // few meshes have a large star: the first wait of the independent set brings
    // the word along, and stops it where there is one
    StopWord told{kLargeStarWord, c.wait_tag()};
    sw.word = c.words + told.word;
    sw.tag = told.tag;
    sweep_stars(c, dim, md, mixed, sw);
    quality_range.end();
    keys = find_indset(c, m, 0, vqual, vm.cand, &any, nullptr, &star, &told);
    if (c.word_set(told.word, told.tag)) {
      sweep_large_stars(c, dim, md, mixed, sw, collect_marked(c, large));
      keys = find_indset(c, m, 0, vqual, vm.cand, &any, nullptr, &star);
    }
  }
  if (layers) layers->settle();
  if (!any) return false;
  Range modify_range(c, "modify_ents");
  CellSweep cells{};
  unsigned cell_blocks = 0;
  for (int d = dim; d > 1; --d) {
    int w = cells.n++;
    cells.dim[w] = d;
    cells.ncells[w] = m.nents[d];
    cells.c2e[w] = ask_down(c, m, d, 1, nullptr).data();
    cells.cv2v[w] = verts_of(c, m, d).data();
    cells.cs2s[w] = m.down[d].data();
    cells.first[w] = cell_blocks;
    cell_blocks += nblocks(m.nents[d]);
    cells.first[w + 1] = cell_blocks;
  }
  if (!vm.joint) {
    Fills fills(c);
    vm.add_rebuild(m, fills);
    fills.run();
  }
  Bytes const* dead = vm.dead;
  LOs onto(c, nv);
  OSH_LAUNCH(mark_rails, nv, c, keys.data(), vrail.data(), ev2v, vm.dead[1].data(),
      vm.rail_col.data(), onto.data());
  for (int w = 0; w < cells.n; ++w) {
    cells.dead_cells[w] = vm.dead[cells.dim[w]].data();
    cells.dead_sides[w] = vm.dead[cells.dim[w] - 1].data();
  }
  hipLaunchKernelGGL(mark_dead_cells, dim3(cell_blocks), dim3(kBlock), 0, c.stream, cells, ev2v,
      static_cast<I8 const*>(vm.rail_col.data()));
  OSH_HIP(hipGetLastError());
  // the keys' rows of every dimension, in order: products follow them
  if (!vm.joint) {
    int const hs[2] = {2, 3};
    bool const in_order[2] = {true, true};
    marked_ups(c, m, 0, keys, dim - 1, hs, in_order, v2d + 2, &vm.key_up_zeros);
  }
  KeyedMods& km = vm.km;  // no key vertex has a product vertex
  LiveRows live{};
  live.n = dim;
  for (int d = 1; d <= dim; ++d) {
    km.prod_counts[d] = LOs(c, nv);
    live.a2ab[d - 1] = v2d[d].a2ab.data();
    live.ab2b[d - 1] = v2d[d].ab2b.data();
    live.dead[d - 1] = dead[d].data();
    live.counts[d - 1] = km.prod_counts[d].data();
  }
  OSH_LAUNCH64(live_counts, std::int64_t(nv) * kLanes, c, keys.data(), live);
  plan_keys(c, m, 0, 0, dim, keys, km);
  LO nkeys = km.nkeys;
  LOs const& keys2verts = km.keys2kds;
  ModPlan const* plans = km.plans;
  note_changed_parts(c, m, 0, keys2verts);
  if (o.verbosity >= 2) std::printf("coarsening %d vertices\n", int(nkeys));
  DMesh nw;
  nw.dim = dim;
  nw.metric_ncomps = nc;
  ModOut mo[4];
  rebuild_same(c, m, nw, 0, plans, mo);
  Products prods[4];
  CoarsenRows rows{};
  for (int d = 1; d <= dim; ++d) {
    Products& p = prods[d];
    p.n = km.nprods[d];
    p.keys2prods = km.k2p[d];
    p.verts = LOs(c, p.n * (d + 1));
    p.src = LOs(c, p.n);
    p.src_dim = d;
    rows.a2ab[d - 1] = v2d[d].a2ab.data();
    rows.ab2b[d - 1] = v2d[d].ab2b.data();
    rows.codes[d - 1] = v2d[d].codes.data();
    rows.dead[d - 1] = dead[d].data();
    rows.verts[d - 1] = verts_of(c, m, d).data();
    rows.keys2prods[d - 1] = km.k2p[d].data();
    rows.pv[d - 1] = p.verts.data();
    rows.psrc[d - 1] = p.src.data();
  }
  OSH_LAUNCH64(coarsen_products, std::int64_t(nkeys) * dim * kLanes, c, nkeys, keys2verts.data(), onto.data(),
      plans[0].offsets.data(), rows);
  place_products(c, m, nw, 1, dim, 0, plans, keys2verts, prods, mo);
  match_sides(c, nw, prods, mo, &vm.side_zeros);
  measure_products(c, nw, mo);
  for (auto const& t : m.vtags)
    nw.vtags.push_back(t.with_data(transfer<Real>(c, mo[0], t.ncomps, t.data, nullptr)));
  for (std::size_t t = 0; t < m.itags.size(); ++t)
    nw.itags[t].data[0] =
        transfer<Real>(c, mo[0], m.itags[t].ncomps, m.itags[t].data[0], nullptr);
  transfer_pointwise(c, m, nw, mo[dim], 0, keys2verts, km.k2p[dim], prods[dim].verts);
  conserve_pass(c, m, nw, 1, 0, keys2verts, km.k2p[dim], mo[dim]);
  m = nw;
  return true;
}

}  // namespace

bool coarsen_by_size(Ctx& c, DMesh& m, AdaptOptions const& o) {
  Reals const& lengths = ask_lengths(c, m);
  ask_qualities(c, m);
  Fills fills(c);
  CoarsenArrays vm(m, fills, true);
  fills.run();
  OSH_LAUNCH(mark_short_edges, m.nents[1], c, lengths.data(), o.min_length_desired,
      m.down[1].data(), vm.wanted.data());
  return coarsen_verts(c, m, o, vm, false, false);
}

bool coarsen_slivers(Ctx& c, DMesh& m, AdaptOptions const& o) {
  ask_lengths(c, m);
  Fills fills(c);
  SliverLayers layers(c, m, o.nsliver_layers, fills);
  CoarsenArrays vm(m, fills, false);
  fills.run();
  vm.wanted = mark_down(c, m, m.dim, 0, layers.mark(o.min_quality_desired));
  return coarsen_verts(c, m, o, vm, true, true, &layers);
}

void coarsen_qualities(Ctx& c, DMesh& m, LO ncands, LO const* cands, I8 const* cand_codes,
    Real* out, int precision, Real qmin) {
  if (ncands == 0) return;
  LOs const& cv2v = verts_of(c, m, m.dim);
  Adj const& v2c = ask_up(c, m, 0, m.dim);
  Bytes codes = fill_i8(c, m.nents[1], kDont);
  OSH_LAUNCH(scatter_codes, ncands, c, cands, cand_codes, codes.data());
  Reals dets = metric_dets(c, m);
  SideQualities sq{cands, m.down[1].data(), cv2v.data(), v2c.a2ab.data(), v2c.ab2b.data(),
      v2c.codes.data(), m.coords.data(), m.metric.data(), dets.data(), qmin, codes.data(), out};
  int lanes = c.tuning.coarsen_lanes < kMaxSideLanes ? c.tuning.coarsen_lanes : kMaxSideLanes;
  lanes = fit_lanes(ncands * 2, lanes);
  int lshift = lanes_shift(lanes);
#define OSH_CQ(D, M, X) \
  OSH_LAUNCH((coarsen_quality_lanes<D, M, X>), ncands * 2 * lanes, c, lshift, sq)
  int md = (m.metric_ncomps == 1) ? 1 : m.dim;
  OSH_BY_FORM(OSH_CQ, m.dim, md, precision == 1);
#undef OSH_CQ
}

}  // namespace osh
