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
// (check_collapse_class, src/Omega_h_check_collapse.cpp:10-40)
__global__ void collapse_codes(LO ne, LO const* ev2v, I8 const* vmarks, I8 const* vdim,
    I8 const* edim, I8* codes) {
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
}

// check_collapse_exposure from the cells' side: every cell of dimension CD
// looks at its own edges, and a collapse side whose cell's side opposite the
// target vertex is classified differently from the cell is vetoed (the
// order of the cells does not matter, so no edge -> cell rows are built)
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
  I8 const* cdim[2];
  I8 const* sdim[2];
  I8* dead_cells[2];
  I8* dead_sides[2];
};

template <int CD>
__device__ __forceinline__ void check_exposure(LO c, CellSweep const& a, int w,
    LO const* ev2v, I8 const* codes, I8* veto) {
  if (c >= a.ncells[w]) return;
  constexpr int nepc = (CD == 3) ? 6 : 3;
  // a cell whose sides are all classified like itself vetoes nothing: most
  // cells stop here, before they look at their edges
  I8 own = a.cdim[w][c];
  unsigned differ = 0u;
#pragma unroll
  for (int k = 0; k <= CD; ++k)
    if (a.sdim[w][a.cs2s[w][std::size_t(c) * (CD + 1) + k]] != own) differ |= 1u << k;
  if (differ == 0u) return;
  LO const* cv = a.cv2v[w] + std::size_t(c) * (CD + 1);
  for (int j = 0; j < nepc; ++j) {
    LO e = a.c2e[w][std::size_t(c) * nepc + j];
    I8 code = codes[e];
    if (code == kDont) continue;
    for (int col = 0; col < 2; ++col) {
      if (!collapses(code, col)) continue;
      int ccv_onto = local_vertex<CD>(cv, ev2v[e * 2 + (1 - col)]);
      if ((differ >> opposite_template(CD, 0, ccv_onto)) & 1u) veto[e * 2 + col] = 1;
    }
  }
}

__device__ __forceinline__ int cell_job(CellSweep const& a, LO* c) {
  int w = (a.n > 1 && blockIdx.x >= a.first[1]) ? 1 : 0;
  *c = LO(blockIdx.x - a.first[w]) * kBlock + LO(threadIdx.x);
  return w;
}

__global__ void __launch_bounds__(kBlock) check_exposure_cells(CellSweep a, LO const* ev2v,
    I8 const* codes, I8* veto) {
  LO c;
  int w = cell_job(a, &c);
  if (a.dim[w] == 3)
    check_exposure<3>(c, a, w, ev2v, codes, veto);
  else
    check_exposure<2>(c, a, w, ev2v, codes, veto);
}

// Each collapse side (candidate edge, direction) gets 2^lshift threads
// (Tuning::coarsen_lanes, at most 32 so that an edge's two sides share a
// wave), which split the collapsing vertex's row between them, so that passes
// with few candidates still spread their work over the device.  Minima do not
// depend on how a row is split, so the lane count changes no result.  The two
// sides' verdicts meet through ballots and one lane writes the edge's code.
// The product builders below use kLanes threads per key.
constexpr int kLanes = 8;
constexpr int kMaxSideLanes = 32;

// the lanes of a side and of its edge in the wave
struct SideLanes {
  int lane;
  int base;  // the side's first lane
  unsigned long long side;  // its lanes
  __device__ __forceinline__ SideLanes(LO t, int lshift) {
    int lanes = 1 << lshift;
    lane = int(t) & (lanes - 1);
    base = int(threadIdx.x % 64) & ~(lanes - 1);
    side = ((1ull << lanes) - 1ull) << base;
  }
  __device__ __forceinline__ bool any(bool x) const { return (__ballot(x) & side) != 0ull; }
};

// writes the code of the edge whose sides' verdicts are `keep`
__device__ __forceinline__ void write_code(SideLanes const& s, int lshift, int col, bool keep,
    I8 code, LO e, I8* codes) {
  unsigned long long b = __ballot(keep);
  if (col != 0 || s.lane != 0) return;
  I8 out = code;
  if (!((b >> s.base) & 1ull)) out = dont_collapse(out, 0);
  if (!((b >> (s.base + (1 << lshift))) & 1ull)) out = dont_collapse(out, 1);
  if (out != code) codes[e] = out;
}

// prevent_coarsen_overshoot: a side is vetoed when any new edge would reach
// max_length (the order of the row does not matter); sides vetoed by exposure
// leave their codes here too.  MIXED: FP32 estimates first; a side is vetoed
// when one is over max_length by more than the screening band, and measured
// in FP64 only when none is but one lies inside the band.
template <int D, int M, bool MIXED>
__global__ void overshoot_lanes(LO nt, int lshift, LO const* cands, LO const* ev2v,
    LO const* v2e_a2ab, LO const* v2e_ab2b, I8 const* v2e_codes, Real const* coords,
    Real const* metric, Real max_length, I8 const* exposed, I8* codes) {
  LO t = thread_index();
  if (t >= nt) return;
  LO side = t >> lshift;
  SideLanes s(t, lshift);
  LO e = cands[side / 2];
  int col = side % 2;
  I8 code = codes[e];
  constexpr int nc = (M == 1) ? 1 : (M == 2 ? 3 : 6);
  LO v_col = ev2v[e * 2 + col];
  LO v_onto = ev2v[e * 2 + (1 - col)];
  bool open = collapses(code, col) && !exposed[e * 2 + col];
  LO row = open ? v2e_a2ab[v_col] : 0;
  LO end = open ? v2e_a2ab[v_col + 1] : 0;
  // the ends of the new edge at row entry ve; false for the candidate itself
  auto ends = [&](LO ve, double (&p0)[D], double (&p1)[D], double (&m0)[nc], double (&m1)[nc]) {
    LO e2 = v2e_ab2b[ve];
    if (e2 == e) return false;
    int eev_in = code_which_down(v2e_codes[ve]);
    LO out = ev2v[e2 * 2 + 1 - eev_in];
    LO a = eev_in == 0 ? v_onto : out, b = eev_in == 0 ? out : v_onto;
    for (int k = 0; k < D; ++k) {
      p0[k] = coords[a * D + k];
      p1[k] = coords[b * D + k];
    }
    for (int k = 0; k < nc; ++k) {
      m0[k] = metric[a * nc + k];
      m1[k] = metric[b * nc + k];
    }
    return true;
  };
  double p0[D], p1[D], m0[nc], m1[nc];
  bool veto = false;
  if constexpr (MIXED) {
    bool unsure = false;
    float lmax = float(max_length);
    for (LO ve = row + s.lane; ve < end; ve += (1 << lshift)) {
      if (!ends(ve, p0, p1, m0, m1)) continue;
      float l = f32::edge_length<D, M>(p0, p1, m0, m1);
      veto = veto || l >= lmax * (1.0f + f32::kScreenBand);
      unsure = unsure || !(l < lmax * (1.0f - f32::kScreenBand));
    }
    veto = s.any(veto);
    if (veto || !s.any(unsure)) end = row;
  }
  for (LO ve = row + s.lane; ve < end && !veto; ve += (1 << lshift))
    if (ends(ve, p0, p1, m0, m1)) veto = edge_length<D, M>(p0, p1, m0, m1) >= max_length;
  write_code(s, lshift, col, open && !s.any(veto), code, e, codes);
}

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

// coarsen_qualities with its filters (src/Omega_h_coarsen_qualities.cpp:16-122):
// the minimum quality of the cells that survive a collapse, with v_col moved
// onto v_onto; a side is kept when it reaches qmin and, with `improve`, exceeds
// the old minimum around v_col.  FILTER off: every side's minimum goes to
// quals and nothing is kept or dropped.
//
// Bound by FP64 issue (166 operations a quality and its correctly rounded
// divisions), so work is left out where it decides nothing: the determinants
// come from vert_dets, a lane reads only the metric it uses, and a side stops
// at the first cell below qmin.
//
// MIXED: FP32 estimates first; a side is rejected (quality -1) when their
// minimum is below qmin by more than the band and every element's
// max-determinant metric was clear, else evaluated in FP64.
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
  Real const* old_quals;  // improve: the elements' qualities (else null)
  I8* codes;
  Real* quals;  // by (edge, direction); by (candidate, direction) with FILTER off
};

template <int D, int M, bool MIXED, bool FILTER>
__global__ void __launch_bounds__(kBlock) coarsen_quality_lanes(LO nt, int lshift,
    SideQualities a) {
  LO t = thread_index();
  if (t >= nt) return;
  LO side = t >> lshift;
  SideLanes s(t, lshift);
  int lanes = 1 << lshift;
  LO e = a.cands[side / 2];
  int col = side % 2;
  I8 code = a.codes[e];
  constexpr int nc = (M == 1) ? 1 : (M == 2 ? 3 : 6);
  bool open = collapses(code, col);
  LO v_col = a.ev2v[e * 2 + col];
  LO v_onto = a.ev2v[e * 2 + (1 - col)];
  LO row = open ? a.v2c_a2ab[v_col] : 0;
  LO end = open ? a.v2c_a2ab[v_col + 1] : 0;
  // the vertices of row entry vc's cell after the collapse; false if it dies
  auto moved = [&](LO vc, LO (&cv)[D + 1]) {
    LO c = a.v2c_ab2b[vc];
    int ccv_col = code_which_down(a.v2c_codes[vc]);
    bool lives = true;
#pragma unroll
    for (int k = 0; k < D + 1; ++k) {
      cv[k] = a.cv2v[std::size_t(c) * (D + 1) + k];
      if (k != ccv_col && cv[k] == v_onto) lives = false;
    }
#pragma unroll
    for (int k = 0; k < D + 1; ++k)
      if (k == ccv_col) cv[k] = v_onto;
    return lives;
  };
  bool rejected = false;
  double const* pp[D + 1];
  double const* ms[D + 1];
  if constexpr (MIXED) {
    float minq = 1.0f;
    bool unclear = false;
    for (LO vc = row + s.lane; vc < end; vc += lanes) {
      LO cv[D + 1];
      if (!moved(vc, cv)) continue;
      for (int k = 0; k < D + 1; ++k) {
        pp[k] = a.coords + std::size_t(cv[k]) * D;
        ms[k] = a.metric + std::size_t(cv[k]) * nc;
      }
      float q = f32::element_quality<D, M>(pp, ms, &unclear);
      minq = (q < minq) ? q : minq;
    }
    for (int d = lanes / 2; d > 0; d >>= 1) {
      float o = __shfl_xor(minq, d, 64);
      minq = (o < minq) ? o : minq;
    }
    rejected = open && !s.any(unclear) &&
               double(minq) < a.qmin * (1.0 - double(f32::kScreenBand));
    if (rejected) end = row;
  }
  double minq = 1.0;
  double vold = 1.79769313486231570815e+308;
  for (LO b = row; b < end; b += lanes) {
    LO vc = b + s.lane;
    LO cv[D + 1];
    if (vc < end) {
      if (FILTER && a.old_quals) vold = math::min2(vold, a.old_quals[a.v2c_ab2b[vc]]);
      if (moved(vc, cv)) {
        double dets[D + 1];
        for (int k = 0; k < D + 1; ++k) {
          pp[k] = a.coords + std::size_t(cv[k]) * D;
          ms[k] = a.metric + std::size_t(cv[k]) * nc;
          dets[k] = a.dets[cv[k]];
        }
        minq = math::min2(minq, element_quality<D, M>(pp, ms, dets));
      }
    }
    if (FILTER && s.any(minq < a.qmin)) break;
  }
  for (int d = lanes / 2; d > 0; d >>= 1) {
    minq = math::min2(minq, __shfl_xor(minq, d, 64));
    vold = math::min2(vold, __shfl_xor(vold, d, 64));
  }
  if (rejected || !open) minq = -1.0;
  if constexpr (FILTER) {
    bool keep = open && minq >= a.qmin && (!a.old_quals || minq > vold);
    if (keep && s.lane == 0) a.quals[std::size_t(e) * 2 + col] = minq;
    write_code(s, lshift, col, keep, code, e, a.codes);
  } else {
    if (s.lane == 0) a.quals[side] = minq;
  }
}

__global__ void scatter_codes(LO n, LO const* cands, I8 const* cand_codes, I8* codes) {
  LO i = thread_index();
  if (i < n) codes[cands[i]] = cand_codes[i];
}

// the vertices that would collapse along some candidate edge
__global__ void mark_collapsing_verts(LO ncands, LO const* cands, LO const* ev2v,
    I8 const* codes, I8* vmarks) {
  LO i = thread_index();
  if (i >= ncands) return;
  LO e = cands[i];
  I8 code = codes[e];
  for (int col = 0; col < 2; ++col)
    if (collapses(code, col)) vmarks[ev2v[e * 2 + col]] = 1;
}

// choose_rails (src/Omega_h_collapse_rail.cpp:15-60): each vertex that can
// collapse takes the shortest of its edges that allow it, the one of higher
// quality among equally long ones, the first one of those; and the vertex star
// (verts_across_edges, src/Omega_h_adj.cpp:512-530) of the vertices whose rows
// are built.  kLanes threads per vertex share its row: a chain of some 14
// dependent gathers a vertex otherwise (41 us for the two sweeps on the 64^3
// workload).  A length or quality that is not a number leaves the row to one
// lane, since the choice then depends on the order of the comparisons.
struct Rails {
  LO const* a2ab;
  LO const* ab2b;
  I8 const* v2e_codes;
  I8 const* codes;
  LO const* ev2v;
  Real const* lengths;
  Real const* quals;
};

__device__ __forceinline__ bool better_rail(double len, double q, double best_len,
    double best_q) {
  return len < best_len || (len == best_len && q > best_q);
}

__global__ void choose_rails_kernel(std::int64_t nt, Rails r, I8* vcand, Real* vqual,
    LO* vrail, LO* star) {
  std::int64_t t = thread_index64();
  if (t >= nt) return;
  LO v = LO(t / kLanes);
  int lane = int(t % kLanes);
  LO b = r.a2ab[v], end = r.a2ab[v + 1];
  if (b == end) {
    if (lane == 0) vcand[v] = 0;
    return;
  }
  LO best = -1, at = 0x7fffffff;
  double best_len = 0.0, best_q = 0.0;
  bool nan = false;
  auto visit = [&](LO ve) {
    LO e = r.ab2b[ve];
    int eev = code_which_down(r.v2e_codes[ve]);
    if (!collapses(r.codes[e], eev)) return;
    double len = r.lengths[e];
    double q = r.quals[std::size_t(e) * 2 + eev];
    nan = nan || len != len || q != q;
    if (best == -1 || better_rail(len, q, best_len, best_q)) {
      best = e;
      at = ve;
      best_len = len;
      best_q = q;
    }
  };
  for (LO ve = b + lane; ve < end; ve += kLanes) {
    star[ve] = r.ev2v[r.ab2b[ve] * 2 + (1 - code_which_down(r.v2e_codes[ve]))];
    visit(ve);
  }
  int base = int(threadIdx.x % 64) & ~(kLanes - 1);
  bool any_nan = ((__ballot(nan) >> base) & ((1ull << kLanes) - 1ull)) != 0ull;
  if (any_nan) {
    if (lane != 0) return;
    best = -1;
    for (LO ve = b; ve < end; ++ve) visit(ve);
  } else {
    for (int d = kLanes / 2; d > 0; d >>= 1) {
      LO ob = __shfl_xor(best, d, 64), oa = __shfl_xor(at, d, 64);
      double ol = __shfl_xor(best_len, d, 64), oq = __shfl_xor(best_q, d, 64);
      bool tie = ol == best_len && oq == best_q;
      if (ob >= 0 && (best < 0 || better_rail(ol, oq, best_len, best_q) || (tie && oa < at))) {
        best = ob;
        at = oa;
        best_len = ol;
        best_q = oq;
      }
    }
    if (lane != 0) return;
  }
  vcand[v] = best >= 0 ? 1 : 0;
  vqual[v] = best_q;
  vrail[v] = best;
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

// the lanes of each collapse side
int side_lanes(Ctx& c, LO ncands) {
  int lanes = c.tuning.coarsen_lanes < kMaxSideLanes ? c.tuning.coarsen_lanes : kMaxSideLanes;
  return fit_lanes(ncands * 2, lanes);
}

template <bool FILTER>
void launch_side_qualities(Ctx& c, DMesh& m, LO ncands, int precision, SideQualities const& a) {
  int dim = m.dim;
  int md = (m.metric_ncomps == 1) ? 1 : dim;
  int lanes = side_lanes(c, ncands);
  int lshift = lanes_shift(lanes);
  bool mixed = precision == 1;
#define OSH_CQ(D, M)                                                                       \
  do {                                                                                     \
    if (mixed)                                                                             \
      OSH_LAUNCH((coarsen_quality_lanes<D, M, true, FILTER>), ncands * 2 * lanes, c, lshift, a); \
    else                                                                                   \
      OSH_LAUNCH((coarsen_quality_lanes<D, M, false, FILTER>), ncands * 2 * lanes, c, lshift, a); \
  } while (0)
  if (dim == 3 && md == 3)
    OSH_CQ(3, 3);
  else if (dim == 3)
    OSH_CQ(3, 1);
  else if (md == 2)
    OSH_CQ(2, 2);
  else
    OSH_CQ(2, 1);
#undef OSH_CQ
}

bool coarsen_verts(Ctx& c, DMesh& m, AdaptOptions const& o, Bytes const& vm,
    bool overshoot_allowed, bool improve) {
  int dim = m.dim;
  LO ne = m.nents[1];
  LO nv = m.nents[0];
  int nc = m.metric_ncomps;
  int md = (nc == 1) ? 1 : dim;
  LO const* ev2v = m.down[1].data();
  Bytes codes(c, ne);
  OSH_LAUNCH(collapse_codes, ne, c, ev2v, vm.data(), m.class_dim[0].data(),
      m.class_dim[1].data(), codes.data());
  // the candidate edges: every later sweep runs over this list
  LOs cands = collect_marked(c, codes);
  LO ncands = cands.size();
  if (ncands == 0) return false;
  Fills fills(c);
  Bytes vmarks = fills.bytes(nv, 0);
  Bytes exposed = fills.bytes(2 * ne, 0);
  fills.run();
  OSH_LAUNCH(mark_collapsing_verts, ncands, c, cands.data(), ev2v, codes.data(), vmarks.data());
  CellSweep cells{};
  unsigned cell_blocks = 0;
  for (int d = dim; d > 1; --d) {
    int w = cells.n++;
    cells.dim[w] = d;
    cells.ncells[w] = m.nents[d];
    cells.c2e[w] = ask_down(c, m, d, 1, nullptr).data();
    cells.cv2v[w] = verts_of(c, m, d).data();
    cells.cs2s[w] = m.down[d].data();
    cells.cdim[w] = m.class_dim[d].data();
    cells.sdim[w] = m.class_dim[d - 1].data();
    cells.first[w] = cell_blocks;
    cell_blocks += nblocks(m.nents[d]);
    cells.first[w + 1] = cell_blocks;
  }
  hipLaunchKernelGGL(check_exposure_cells, dim3(cell_blocks), dim3(kBlock), 0, c.stream, cells,
      ev2v, static_cast<I8 const*>(codes.data()), exposed.data());
  OSH_HIP(hipGetLastError());
  // upward rows only where the candidates look: the collapsing vertices' edges
  // (ordered: the first best rail is kept) and cells (order-free minima)
  Adj up[2];
  int const highs[2] = {1, dim};
  bool const sorted[2] = {true, false};
  marked_ups(c, m, 0, vmarks, 2, highs, sorted, up);
  Adj const& v2e = up[0];
  Adj const& v2c = up[1];
  Real max_length = overshoot_allowed ? o.max_length_allowed : o.max_length_desired;
  bool mixed = o.precision == 1;
  int lanes = side_lanes(c, ncands);
  int lshift = lanes_shift(lanes);
  Range overshoot_range(c, "prevent_overshoot");
#define OSH_OV(D, M, X)                                                                    \
  OSH_LAUNCH((overshoot_lanes<D, M, X>), ncands * 2 * lanes, c, lshift, cands.data(), ev2v,  \
      v2e.a2ab.data(), v2e.ab2b.data(), v2e.codes.data(), m.coords.data(), m.metric.data(), \
      max_length, exposed.data(), codes.data())
#define OSH_OV_ALL(X)        \
  if (dim == 3 && md == 3)   \
    OSH_OV(3, 3, X);         \
  else if (dim == 3)         \
    OSH_OV(3, 1, X);         \
  else if (md == 2)          \
    OSH_OV(2, 2, X);         \
  else                       \
    OSH_OV(2, 1, X)
  if (mixed) {
    OSH_OV_ALL(true);
  } else {
    OSH_OV_ALL(false);
  }
#undef OSH_OV_ALL
#undef OSH_OV
  overshoot_range.end();
  if (o.should_prevent_coarsen_flip) prevent_coarsen_flip(c, m, cands, codes);
  // sides without a candidate left are skipped by every sweep below
  Range quality_range(c, "coarsen_qualities");
  Reals quals(c, ne * 2);  // read where a side is kept
  LOs const& cv2v = verts_of(c, m, dim);
  Reals dets = metric_dets(c, m);
  SideQualities sq{cands.data(), ev2v, cv2v.data(), v2c.a2ab.data(), v2c.ab2b.data(),
      v2c.codes.data(), m.coords.data(), m.metric.data(), dets.data(), o.min_quality_allowed,
      improve ? ask_qualities(c, m).data() : (Real const*)nullptr, codes.data(), quals.data()};
  launch_side_qualities<true>(c, m, ncands, o.precision, sq);
  quality_range.end();
  Bytes vcand(c, nv);
  Reals vqual(c, nv);
  LOs vrail(c, nv);
  // the independent set reads the star rows of candidate vertices only
  Adj star;
  star.a2ab = v2e.a2ab;
  star.ab2b = LOs(c, v2e.ab2b.size());
  Rails rails{v2e.a2ab.data(), v2e.ab2b.data(), v2e.codes.data(), codes.data(), ev2v,
      ask_lengths(c, m).data(), quals.data()};
  OSH_LAUNCH64(choose_rails_kernel, std::int64_t(nv) * kLanes, c, rails, vcand.data(), vqual.data(),
      vrail.data(), star.ab2b.data());
  bool any;
  Bytes keys = find_indset(c, m, 0, vqual, vcand, &any, nullptr, &star);
  if (!any) return false;
  Range modify_range(c, "modify_ents");
  Bytes dead[4];
  dead[1] = fills.bytes(ne, 0);
  for (int d = 2; d <= dim; ++d) dead[d] = fills.bytes(m.nents[d], 0);
  Bytes rail_col = fills.bytes(ne, -1);
  fills.run();
  LOs onto(c, nv);
  OSH_LAUNCH(mark_rails, nv, c, keys.data(), vrail.data(), ev2v, dead[1].data(),
      rail_col.data(), onto.data());
  for (int w = 0; w < cells.n; ++w) {
    cells.dead_cells[w] = dead[cells.dim[w]].data();
    cells.dead_sides[w] = dead[cells.dim[w] - 1].data();
  }
  hipLaunchKernelGGL(mark_dead_cells, dim3(cell_blocks), dim3(kBlock), 0, c.stream, cells, ev2v,
      static_cast<I8 const*>(rail_col.data()));
  OSH_HIP(hipGetLastError());
  // the keys' rows of every dimension, in order: products follow them
  Adj v2d[4];
  v2d[1] = v2e;
  {
    int const hs[2] = {2, 3};
    bool const in_order[2] = {true, true};
    marked_ups(c, m, 0, keys, dim - 1, hs, in_order, v2d + 2);
  }
  KeyedMods km;  // no key vertex has a product vertex
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
  match_sides(c, nw, prods, mo);
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
  Bytes vm = fill_i8(c, m.nents[0], 0);
  OSH_LAUNCH(mark_short_edges, m.nents[1], c, lengths.data(), o.min_length_desired,
      m.down[1].data(), vm.data());
  return coarsen_verts(c, m, o, vm, false, false);
}

bool coarsen_slivers(Ctx& c, DMesh& m, AdaptOptions const& o) {
  ask_lengths(c, m);
  Bytes marks = mark_sliver_layers(c, m, o.min_quality_desired, o.nsliver_layers);
  Bytes vm = mark_down(c, m, m.dim, 0, marks);
  return coarsen_verts(c, m, o, vm, true, true);
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
      v2c.codes.data(), m.coords.data(), m.metric.data(), dets.data(), qmin, nullptr,
      codes.data(), out};
  launch_side_qualities<false>(c, m, ncands, precision, sq);
}

}  // namespace osh
