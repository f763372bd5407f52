// Edge-swap pass on the device (3D edge swap over edge loops of up to 7
// tets, 2D edge flip).
//
//   swap_edges / swap_part1 / filter_swap_improve src/Omega_h_swap.cpp:14-55
//   swap3d_ghosted / swap3d_element_based        src/Omega_h_swap3d.cpp:14-84
//   swap3d_qualities                             src/Omega_h_swap3d_qualities.cpp:11-75
//   find_loop                                    src/Omega_h_swap3d_loop.hpp:24-78
//   choose                                       src/Omega_h_swap3d_choice.hpp:16-100
//   swap3d_keys_to_prods / swap3d_topology       src/Omega_h_swap3d_topology.cpp:12-119
//   swap2d_qualities / swap2d_topology           src/Omega_h_swap2d_qualities.cpp:16-72,
//                                                src/Omega_h_swap2d_topology.cpp:11-79
//   transfer_swap / transfer_copy                src/Omega_h_transfer.cpp:631-730
#include <cstdio>

#include "osh_indset.hpp"
#include "osh_math.hpp"
#include "osh_passes.hpp"
#include "osh_swap_tables.hpp"

namespace osh {

namespace {

using swap::Tables;

// The tets around the candidate edges of a swap pass: kRow slots per
// candidate, in the order of the atomics, each the use index tet * 6 +
// local edge.  Only edges with at most swap::kMaxLoop tets can be swapped, so
// a candidate with more just counts them; fixed rows need no scan of counts.
constexpr int kRow = 8;
static_assert(swap::kMaxLoop <= kRow, "a loop fits a row");

struct EdgeRings {
  LO const* cands;     // the candidate edges
  LO const* cand_of;   // candidate index of an edge
  LO const* counts;    // tets around an edge, by edge
  LO const* rows;      // kRow use indices per candidate
  LO const* t2e;       // the elements' edges and their codes
  I8 const* t2e_codes;
};

struct Loop {
  int size;
  LO eev2v[2];
  LO verts[swap::kMaxLoop];
};

// a ring of tets that does not close is a broken mesh: the reference aborts
// (src/Omega_h_swap3d_loop.hpp:71); here the loop is marked broken (size
// -1) and the caller raises kBrokenSwapLoop
__device__ void find_loop(LO edge, LO const* a2ab, LO const* ab2b, I8 const* codes,
    LO const* ev2v, LO const* tv2v, Loop& loop) {
  LO begin = a2ab[edge], end = a2ab[edge + 1];
  loop.size = end - begin;
  if (loop.size > swap::kMaxLoop) return;
  loop.eev2v[0] = ev2v[edge * 2];
  loop.eev2v[1] = ev2v[edge * 2 + 1];
  LO tmp[swap::kMaxLoop][2];
  for (int le = 0; le < loop.size; ++le) {
    LO tet = ab2b[begin + le];
    int rre = code_which_down(codes[begin + le]);
    int rot = code_rotation(codes[begin + le]);
    int rre_opp = opposite_template(3, 1, rre);
    for (int eev = 0; eev < 2; ++eev)
      tmp[le][eev] = tv2v[tet * 4 + down_template(3, 1, rre_opp, rot ^ eev)];
  }
  for (int i = 0; i < loop.size - 1; ++i) {
    int j;
    for (j = i + 1; j < loop.size; ++j)
      if (tmp[j][0] == tmp[i][1]) break;
    if (j >= loop.size) {
      loop.size = -1;
      return;
    }
    LO t0 = tmp[i + 1][0], t1 = tmp[i + 1][1];
    tmp[i + 1][0] = tmp[j][0];
    tmp[i + 1][1] = tmp[j][1];
    tmp[j][0] = t0;
    tmp[j][1] = t1;
  }
  for (int lv = 0; lv < loop.size; ++lv) loop.verts[lv] = tmp[lv][0];
}

template <int M>
__device__ double tet_quality(LO const* v, Real const* coords, Real const* metric) {
  constexpr int nc = (M == 1) ? 1 : 6;
  double p[4][3];
  double m[4][nc];
  double const* pp[4];
  double const* ms[4];
  for (int k = 0; k < 4; ++k) {
    for (int j = 0; j < 3; ++j) p[k][j] = coords[v[k] * 3 + j];
    for (int j = 0; j < nc; ++j) m[k][j] = metric[v[k] * nc + j];
    pp[k] = p[k];
    ms[k] = m[k];
  }
  return element_quality<3, M>(pp, ms);
}

// the FP32 screen of tet_quality (mixed precision); *unsure as in
// f32::element_quality
template <int M>
__device__ float tet_quality32(LO const* v, Real const* coords, Real const* metric,
    bool* unsure) {
  constexpr int nc = (M == 1) ? 1 : 6;
  double p[4][3];
  double m[4][nc];
  double const* pp[4];
  double const* ms[4];
  for (int k = 0; k < 4; ++k) {
    for (int j = 0; j < 3; ++j) p[k][j] = coords[v[k] * 3 + j];
    for (int j = 0; j < nc; ++j) m[k][j] = metric[v[k] * nc + j];
    pp[k] = p[k];
    ms[k] = m[k];
  }
  return f32::element_quality<3, M>(pp, ms, unsure);
}

template <int S, int M>
__device__ float length_between32(LO a, LO b, Real const* coords, Real const* metric) {
  constexpr int nc = (M == 1) ? 1 : (M == 2 ? 3 : 6);
  double p0[S], p1[S], m0[nc], m1[nc];
  for (int k = 0; k < S; ++k) {
    p0[k] = coords[a * S + k];
    p1[k] = coords[b * S + k];
  }
  for (int k = 0; k < nc; ++k) {
    m0[k] = metric[a * nc + k];
    m1[k] = metric[b * nc + k];
  }
  return f32::edge_length<S, M>(p0, p1, m0, m1);
}

template <int S, int M>
__device__ double length_between(LO a, LO b, Real const* coords, Real const* metric) {
  constexpr int nc = (M == 1) ? 1 : (M == 2 ? 3 : 6);
  double p0[S], p1[S], m0[nc], m1[nc];
  for (int k = 0; k < S; ++k) {
    p0[k] = coords[a * S + k];
    p1[k] = coords[b * S + k];
  }
  for (int k = 0; k < nc; ++k) {
    m0[k] = metric[a * nc + k];
    m1[k] = metric[b * nc + k];
  }
  return edge_length<S, M>(p0, p1, m0, m1);
}

__global__ void swap3d_rows(LO nuses, LO const* t2e, I8 const* marks, LO const* cand_of,
    LO* counts, LO* rows) {
  LO i = thread_index();
  if (i >= nuses) return;
  LO e = t2e[i];
  if (!marks[e]) return;
  LO slot = atomicAdd(&counts[e], 1);
  if (slot < kRow) rows[std::size_t(cand_of[e]) * kRow + slot] = i;
}

// The loop of vertices around a candidate edge (find_loop,
// src/Omega_h_swap3d_loop.hpp:24-78) by a group of at least kRow lanes, the
// lanes from `base` on in the wave: lane k < size brings use index `use` and
// returns with the loop's k-th vertex.  The ring starts at the tet with the
// smallest index, and each tet is followed by the one that begins at its last
// vertex.  *ok is false (in every lane) where no such tet is left: the tets
// do not close a ring (the reference aborts,
// src/Omega_h_swap3d_loop.hpp:71).
__device__ __forceinline__ LO ring_vertex(int size, int lane, int base, LO use,
    I8 const* t2e_codes, LO const* tv2v, bool* ok) {
  LO x0 = -1, x1 = -1;
  bool in = lane < size;
  if (in) {
    LO tet = use / 6;
    int rot = code_rotation(t2e_codes[use]);
    int opp = opposite_template(3, 1, int(use % 6));
    x0 = tv2v[tet * 4 + down_template(3, 1, opp, rot)];
    x1 = tv2v[tet * 4 + down_template(3, 1, opp, rot ^ 1)];
  }
  // the lane with the smallest use
  LO least = in ? use : 0x7fffffff;
  for (int d = kRow / 2; d > 0; d >>= 1) {
    LO o = __shfl_xor(least, d, 64);
    least = o < least ? o : least;
  }
  least = __shfl(least, base, 64);  // lanes of the row's first eight hold it
  unsigned long long group = ((1ull << kRow) - 1ull) << base;
  unsigned long long at = __ballot(in && use == least) & group;
  int cur = __ffsll(static_cast<long long>(at)) - 1;
  unsigned long long done = at;
  LO mine = __shfl(x0, cur, 64);
  if (lane != 0) mine = -1;
  *ok = true;
  for (int i = 1; i < size; ++i) {
    LO v = __shfl(x1, cur, 64);
    unsigned long long next = __ballot(in && x0 == v) & group & ~done;
    if (next == 0ull) {
      *ok = false;
      break;
    }
    cur = __ffsll(static_cast<long long>(next)) - 1;
    done |= 1ull << cur;
    if (lane == i) mine = v;
  }
  return mine;
}

// swap3d_qualities (src/Omega_h_swap3d_qualities.cpp:11-75) and choose
// (src/Omega_h_swap3d_choice.hpp:16-100) in one launch: a group of lanes per
// candidate finds the edge's loop, measures each (unique triangle, side) and
// each unique interior edge once, in LDS, values every triangulation and
// takes the best.  A triangulation's value is its minimum triangle quality, or
// -1 when one of its interior edges is longer than max_length; choose() keeps
// the first triangulation whose quality exceeds every earlier kept one
// (starting from 0) and whose edges pass, so it equals the first one attaining
// the largest of these values, when that is positive.
//
// Most candidates of a late pass carry their choice over and return at once,
// so the launch is bound by the latency of one evaluation, not by the FP64
// rate: loops, measures, triangulations and choice in launches of their own,
// with their intermediate arrays, took 32 us where this takes 16 us.
//
// MIXED: an FP32 estimate first.  Its best value, where an interior edge
// counts as too long only when its FP32 length exceeds max_length by more
// than the band, is an upper estimate of the FP64 choice's quality; the
// candidate needs no FP64 when that is below the edge's current minimum
// quality by more than the band, with every element's metric clear and that
// minimum positive.
struct EvalArgs {
  EdgeRings r;
  LO ncands;
  LO const* ev2v;
  LO const* tv2v;
  Real const* coords;
  Real const* metric;
  Real const* elem_quals;
  Real max_length;
  Tables const* tb;
  I8* configs;
  Real* quals;
  I8* keep;
  I8* c_valid;  // null: no cache
  I8* c_cfg;
  I8* c_keep;
  Real* c_q;
  int* error;
};

constexpr int kMinEvalLanes = kRow;

// LDS written by some lanes of a wave and read by others of the same wave
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int M, bool MIXED>
__global__ void __launch_bounds__(kBlock) swap3d_evaluate_kernel(LO nt, int lshift, EvalArgs a) {
  constexpr int kGroups = kBlock / kMinEvalLanes;
  __shared__ double s_tq[kGroups][swap::kMaxUniqueTris];
  __shared__ double s_el[kGroups][swap::kMaxUniqueEdges];
  __shared__ LO s_lv[kGroups][kRow];
  LO t = thread_index();
  if (t >= nt) return;
  int lanes = 1 << lshift;
  LO cand = t >> lshift;
  int lane = int(t) & (lanes - 1);
  int base = int(threadIdx.x % 64) & ~(lanes - 1);
  int g = int(threadIdx.x) >> lshift;
  LO edge = a.r.cands[cand];
  if (a.c_valid && a.c_valid[edge]) {
    if (lane == 0) {
      a.configs[edge] = a.c_cfg[edge];
      if (a.c_keep[edge]) {
        a.keep[edge] = 1;
        a.quals[edge] = a.c_q[edge];
      }
    }
    return;
  }
  int n = a.r.counts[edge];
  Tables const* tb = a.tb;
  // old: the smallest quality around the edge; each lane keeps the first of
  // its triangulations with the largest value above 0
  double old = 1.79769313486231570815e+308;
  int choice = -1;
  double choice_quality = n <= swap::kMaxLoop ? 0.0 : -1.0;
  bool open = n >= 1 && n <= swap::kMaxLoop;
  LO use = 0;
  LO eev[2] = {0, 0};
  if (open) {
    use = lane < n ? a.r.rows[std::size_t(cand) * kRow + lane] : 0;
    bool ok;
    LO v = ring_vertex(n, lane, base, use, a.r.t2e_codes, a.tv2v, &ok);
    if (!ok) {
      if (lane == 0) *a.error = kBrokenSwapLoop;
      open = false;
      choice_quality = -1.0;
    }
    if (lane < kRow) s_lv[g][lane] = v;
    eev[0] = a.ev2v[edge * 2];
    eev[1] = a.ev2v[edge * 2 + 1];
    if (lane < n) old = math::min2(old, a.elem_quals[use / 6]);
    for (int d = kRow / 2; d > 0; d >>= 1) old = math::min2(old, __shfl_xor(old, d, 64));
    old = __shfl(old, base, 64);
    wave_lds_fence();
  }
  bool rejected = false;
  if (open) {
    int ntris = tb->ntris[n], nedges = tb->nuedges[n];
    int nmeshes = tb->mesh_counts[n];
    int mesh_tris = tb->mesh_sizes[n], mesh_edges = tb->nedges[n];
    LO const* lv = s_lv[g];
    double* tq = s_tq[g];
    double* el = s_el[g];
    // the vertices of (triangle i / 2, side i % 2)
    auto tet = [&](int i, LO* tv) {
      int ut = i >> 1;
      bool second = i & 1;
      LO p = lv[tb->tris[n][ut][0]], q = lv[tb->tris[n][ut][1]], r = lv[tb->tris[n][ut][2]];
      tv[0] = p;
      tv[1] = second ? r : q;
      tv[2] = second ? q : r;
      tv[3] = second ? eev[0] : eev[1];
    };
    auto value = [&](int mesh, double lmax) {
      double q = 1.0;
      for (int mt = 0; mt < mesh_tris; ++mt)
        q = math::min2(q, tq[tb->meshes[n][mesh * mesh_tris + mt]]);
      for (int me = 0; me < mesh_edges; ++me)
        if (el[tb->medges[n][mesh * mesh_edges + me]] > lmax) q = -1.0;
      return q;
    };
    if constexpr (MIXED) {
      bool unclear = false;
      for (int i = lane; i < 2 * ntris; i += lanes) {
        LO tv[4];
        tet(i, tv);
        float q = tet_quality32<M>(tv, a.coords, a.metric, &unclear);
        q = q < 1.0f ? q : 1.0f;
        float o = __shfl_xor(q, 1, 64);
        if (!(i & 1)) tq[i >> 1] = double(o < q ? o : q);
      }
      for (int i = lane; i < nedges; i += lanes)
        el[i] = double(length_between32<3, M>(lv[tb->uedges[n][i][0]], lv[tb->uedges[n][i][1]],
            a.coords, a.metric));
      wave_lds_fence();
      double best = -1.0;
      double lmax = a.max_length * (1.0 + double(f32::kScreenBand));
      for (int mesh = lane; mesh < nmeshes; mesh += lanes)
        best = math::max2(best, value(mesh, lmax));
      int unsure = unclear ? 1 : 0;
      for (int d = lanes / 2; d > 0; d >>= 1) {
        best = math::max2(best, __shfl_xor(best, d, 64));
        unsure |= __shfl_xor(unsure, d, 64);
      }
      rejected = ntris != 0 && !unsure && old > 0.0 &&
                 best < old * (1.0 - double(f32::kScreenBand));
      wave_lds_fence();
    }
    if (!rejected) {
      for (int i = lane; i < 2 * ntris; i += lanes) {
        LO tv[4];
        tet(i, tv);
        double q = math::min2(1.0, tet_quality<M>(tv, a.coords, a.metric));
        double o = __shfl_xor(q, 1, 64);
        if (!(i & 1)) tq[i >> 1] = math::min2(q, o);
      }
      for (int i = lane; i < nedges; i += lanes)
        el[i] = length_between<3, M>(lv[tb->uedges[n][i][0]], lv[tb->uedges[n][i][1]], a.coords,
            a.metric);
      wave_lds_fence();
      for (int mesh = lane; mesh < nmeshes; mesh += lanes) {
        double q = value(mesh, a.max_length);
        if (q > choice_quality) {
          choice = mesh;
          choice_quality = q;
        }
      }
      // the largest value, the lowest index on ties
      for (int d = lanes / 2; d > 0; d >>= 1) {
        double oq = __shfl_xor(choice_quality, d, 64);
        int om = __shfl_xor(choice, d, 64);
        if (oq > choice_quality || (oq == choice_quality && om >= 0 &&
                                       (choice < 0 || om < choice))) {
          choice_quality = oq;
          choice = om;
        }
      }
    } else {
      choice_quality = -1.0;
    }
  }
  if (lane != 0) return;
  a.configs[edge] = I8(choice);
  // a key needs a triangulation; with inverted elements the reference can
  // keep an edge without one and then index its tables out of bounds
  bool kept = choice >= 0 && choice_quality > old;
  if (kept) {
    a.keep[edge] = 1;
    a.quals[edge] = choice_quality;
  }
  if (a.c_valid) {
    a.c_cfg[edge] = I8(choice);
    a.c_keep[edge] = I8(kept);
    a.c_q[edge] = choice_quality;
    a.c_valid[edge] = 1;
  }
}

// indset::find over the candidates kept by the choice, through their rows
// (see indset_first_edges and indset_edge for the rounds' rules): a thread or
// a group of lanes per candidate instead of one per edge of the mesh
template <bool FIRST>
__global__ void swap3d_indset(LO nt, int lanes, EdgeRings r, Real const* q, I8 const* old_state,
    I8* new_state, unsigned long long* dom, IndsetWords w) {
  LO t = thread_index();
  if (t >= nt) return;
  LO cand = t / lanes;
  int lane = t % lanes;
  LO v = r.cands[cand];
  I8 s = indset_state<FIRST>(old_state, v);
  I8 res = s;
  if (s == 2) {
    LO const* row = r.rows + std::size_t(cand) * kRow;
    unsigned long long mask = 0;
    int undecided = 0;
    bool out = false;
    if (FIRST) {
      Real qv = q[v];
      int np = r.counts[v] * 6;
      for (int p = lane; p < np; p += lanes) {
        LO u = r.t2e[row[p / 6] / 6 * 6 + p % 6];
        if (u == v || !old_state[u]) continue;
        Real qu = q[u];
        bool beaten = (qu != qv) ? (qu < qv) : (u < v);
        if (beaten) continue;
        undecided = 1;
        mask |= 1ull << p;
      }
      for (int d = lanes / 2; d > 0; d >>= 1) {
        mask |= __shfl_xor(mask, d, 64);
        undecided |= __shfl_xor(undecided, d, 64);
      }
      if (lane == 0) dom[cand] = mask;
    } else {
      mask = dom[cand];
      while (mask && !out) {
        int p = __ffsll(static_cast<long long>(mask)) - 1;
        mask &= mask - 1;
        I8 su = old_state[r.t2e[row[p / 6] / 6 * 6 + p % 6]];
        out = su == 1;
        if (su == 2) undecided = 1;
      }
    }
    res = out ? I8(0) : (undecided ? I8(2) : I8(1));
  }
  if (lane != 0) return;
  new_state[v] = res;
  tell_round(s, res, w);
}

// The rebuild plans of a swap from its keys' rows alone: a key edge and the
// faces and tets around it are no longer the same, the lowest of each stands
// for the key's products, and all else stays (one launch of fills).  Keys share
// no element, so every entity is written for one key only.  Sweeps over every
// edge, face and tet of the mesh (counts, key marks, same entities,
// representatives) took 17 us where this takes 5 us.
struct KeyPlan {
  I8* same[3];    // edges, faces, tets
  LO* counts[3];
  I8* is_key;     // per candidate
  LO* nprods[3];  // per candidate: product edges, faces, tets
  LO* reps[2];    // per candidate: face, tet
  I8* dirty;      // edges whose tets change (null: not wanted)
};

__global__ void swap3d_plan_keys(LO nt, EdgeRings r, I8 const* keys, LO const* t2f,
    Tables const* tb, KeyPlan a) {
  LO t = thread_index();
  if (t >= nt) return;
  LO cand = t / kRow;
  int lane = t % kRow;
  LO e = r.cands[cand];
  if (!keys[e]) {
    if (lane == 0) {
      a.is_key[cand] = 0;
      for (int d = 0; d < 3; ++d) a.nprods[d][cand] = 0;
    }
    return;
  }
  int n = r.counts[e];
  int npt = tb->mesh_sizes[n], npe = tb->nedges[n];
  LO tet = 0x7fffffff, f[2] = {0x7fffffff, 0x7fffffff};
  if (lane < n) {
    LO use = r.rows[std::size_t(cand) * kRow + lane];
    tet = use / 6;
    int opp = opposite_template(3, 1, int(use % 6));
    // the two faces of the tet that hold the edge lie across from the ends of
    // the opposite edge
    for (int k = 0; k < 2; ++k)
      f[k] = t2f[tet * 4 + opposite_template(3, 0, down_template(3, 1, opp, k))];
    if (a.dirty)
      for (int i = 0; i < 6; ++i) a.dirty[r.t2e[tet * 6 + i]] = 1;
  }
  LO trep = tet, frep = f[0] < f[1] ? f[0] : f[1];
  for (int d = kRow / 2; d > 0; d >>= 1) {
    LO o = __shfl_xor(trep, d, 64);
    trep = o < trep ? o : trep;
    o = __shfl_xor(frep, d, 64);
    frep = o < frep ? o : frep;
  }
  LO nf = npt + 2 * npe;
  if (lane < n) {
    a.same[2][tet] = 0;
    a.counts[2][tet] = tet == trep ? 2 * npt : 0;
    for (int k = 0; k < 2; ++k) {
      a.same[1][f[k]] = 0;
      a.counts[1][f[k]] = f[k] == frep ? nf : 0;
    }
  }
  if (lane == 0) {
    a.same[0][e] = 0;
    a.counts[0][e] = npe;
    a.is_key[cand] = 1;
    a.nprods[0][cand] = npe;
    a.nprods[1][cand] = nf;
    a.nprods[2][cand] = 2 * npt;
    a.reps[0][cand] = frep;
    a.reps[1][cand] = trep;
  }
}

// reflect_down for the products of one swap key, searched locally: a side
// of a product (a face of a new tet, an edge of a new face) is a product of
// the same key one dimension down or a surviving side of one of the old tets
// around the key edge, so those are the only candidates (vertices keep their
// numbers in a swap).  `lanes` threads (a power of two up to 64,
// Tuning::side_lanes) share one side's candidates; the one that matches
// writes the side, at the product's new number, and the code match_uses would
// compute.  Faces and tets are one launch: job 0 owns the first workgroups.
struct LocalSides {
  LO nuses;
  LO const* prod_key;
  LO const* k2p_low;
  LO const* pv_high;
  LO const* pv_low;
  LO const* low_prods2new;
  LO const* prods2new;
  LO const* t2low;
  LO const* old_low_verts;
  I8 const* low_same;
  LO const* low_offsets;
  LO* out;
  I8* out_codes;
};

template <int HIGH>
__device__ __forceinline__ void local_side(LO t, int lanes, LO const* keys2edges,
    EdgeRings const& r, LocalSides const& a, int* error) {
  LO u = t / lanes;
  int lane = t % lanes;
  constexpr int LOW = HIGH - 1;
  constexpr int nvh = HIGH + 1;
  constexpr int nvl = LOW + 1;
  constexpr int nlpt = (HIGH == 3) ? 4 : 6;  // faces or edges of an old tet
  bool found = false;
  LO at = 0;
  if (u < a.nuses) {
    LO p = u / nvh;
    int which = u % nvh;
    at = a.prods2new[p] * nvh + which;
    LO key = a.prod_key[p];
    LO av[3];
#pragma unroll
    for (int k = 0; k < nvl; ++k) av[k] = a.pv_high[p * nvh + down_template(HIGH, LOW, which, k)];
    LO q0 = a.k2p_low[key];
    LO nq = a.k2p_low[key + 1] - q0;
    LO e = keys2edges[key];
    LO const* row = r.rows + std::size_t(r.cand_of[e]) * kRow;
    LO ncand = nq + r.counts[e] * nlpt;
    for (LO cnd = lane; cnd < ncand; cnd += lanes) {
      LO id;
      LO bv[3];
      if (cnd < nq) {
        id = a.low_prods2new[q0 + cnd];
#pragma unroll
        for (int k = 0; k < nvl; ++k) bv[k] = a.pv_low[(q0 + cnd) * nvl + k];
      } else {
        LO s = cnd - nq;
        LO o = a.t2low[row[s / nlpt] / 6 * nlpt + s % nlpt];
        if (!a.low_same[o]) continue;
        id = a.low_offsets[o];
#pragma unroll
        for (int k = 0; k < nvl; ++k) bv[k] = a.old_low_verts[o * nvl + k];
      }
      int wd =
          (bv[0] == av[0]) ? 0 : (bv[1] == av[0]) ? 1 : (nvl == 3 && bv[2] == av[0]) ? 2 : -1;
      if (wd < 0) continue;
      I8 code;
      if (nvl == 2) {
        if (av[1] != bv[1 - wd]) continue;
        code = make_code(0, wd, 0);
      } else if (av[1] == bv[(wd + 1) % 3] && av[2] == bv[(wd + 2) % 3]) {
        code = make_code(0, (3 - wd) % 3, 0);
      } else if (av[1] == bv[(wd + 2) % 3] && av[2] == bv[(wd + 1) % 3]) {
        code = make_code(1, (3 - wd) % 3, 0);
      } else {
        continue;
      }
      a.out[at] = id;
      a.out_codes[at] = code;
      found = true;
    }
  }
  // the side's lanes are `lanes` consecutive lanes of one wave
  unsigned long long any = __ballot(found);
  int base = int(threadIdx.x % 64) & ~(lanes - 1);
  unsigned long long group = (lanes >= 64) ? ~0ull : ((1ull << lanes) - 1);
  if (u < a.nuses && lane == 0 && ((any >> base) & group) == 0ull) {
    *error = kReflectDownNoMatch;
    a.out[at] = 0;
    a.out_codes[at] = 0;
  }
}

__global__ void __launch_bounds__(kBlock) swap3d_local_down(int lanes, unsigned face_blocks,
    LO const* keys2edges, EdgeRings r, LocalSides faces, LocalSides tets, int* error) {
  if (blockIdx.x < face_blocks)
    local_side<2>(LO(blockIdx.x) * kBlock + LO(threadIdx.x), lanes, keys2edges, r, faces, error);
  else
    local_side<3>(LO(blockIdx.x - face_blocks) * kBlock + LO(threadIdx.x), lanes, keys2edges, r,
        tets, error);
}

// swap3d_topology (src/Omega_h_swap3d_topology.cpp:12-119): the key list, each
// key's product offsets and representatives from the per-candidate scans, and
// its new edges, faces and tets in template order; kRow threads per candidate
// find a key's loop again and share its products
struct KeyProducts {
  I8 const* is_key;
  LO const* key_off;
  LO const* off[3];   // product offsets by candidate
  LO const* reps[2];  // face and tet representatives by candidate
  LO* keys2edges;
  LO* k2p[3];
  LO* key_reps[3];
  LO* pv[3];
  LO* fkey;
  LO* tkey;
};

__global__ void swap3d_products(LO nt, LO ncands, EdgeRings r, LO const* ev2v, LO const* tv2v,
    I8 const* configs, Tables const* tb, KeyProducts a) {
  LO t = thread_index();
  if (t >= nt) return;
  LO cand = t / kRow;
  int lane = t % kRow;
  if (t == 0)
    for (int d = 0; d < 3; ++d) a.k2p[d][a.key_off[ncands]] = a.off[d][ncands];
  if (!a.is_key[cand]) return;
  LO k = a.key_off[cand];
  LO edge = r.cands[cand];
  int n = r.counts[edge];
  int base = int(threadIdx.x % 64) & ~(kRow - 1);
  LO use = lane < n ? r.rows[std::size_t(cand) * kRow + lane] : 0;
  bool ok;  // the choice has found the same ring
  LO mine = ring_vertex(n, lane, base, use, r.t2e_codes, tv2v, &ok);
  LO lv[kRow];
#pragma unroll
  for (int i = 0; i < kRow; ++i) lv[i] = __shfl(mine, base + i, 64);
  auto vertex = [&](int i) {
    LO v = lv[0];
#pragma unroll
    for (int j = 1; j < kRow; ++j) v = i == j ? lv[j] : v;
    return v;
  };
  LO k2e = a.off[0][cand], k2f = a.off[1][cand], k2t = a.off[2][cand];
  if (lane == 0) {
    a.keys2edges[k] = edge;
    a.k2p[0][k] = k2e;
    a.k2p[1][k] = k2f;
    a.k2p[2][k] = k2t;
    a.key_reps[0][k] = edge;
    a.key_reps[1][k] = a.reps[0][cand];
    a.key_reps[2][k] = a.reps[1][cand];
  }
  int config = configs[edge];
  LO eev2v[2] = {ev2v[edge * 2], ev2v[edge * 2 + 1]};
  int npt = tb->mesh_sizes[n], npe = tb->nedges[n];
  LO* pe = a.pv[0];
  LO* pf = a.pv[1];
  LO* pt = a.pv[2];
  for (int i = lane; i < npe; i += kRow) {
    int ue = tb->medges[n][config * npe + i];
    LO va = vertex(tb->uedges[n][ue][0]);
    LO vb = vertex(tb->uedges[n][ue][1]);
    LO pedge = k2e + i;
    pe[pedge * 2] = va;
    pe[pedge * 2 + 1] = vb;
    for (int eev = 0; eev < 2; ++eev) {
      LO ptri = k2f + 2 * i + eev;
      pf[ptri * 3 + 0] = va;
      pf[ptri * 3 + 1] = vb;
      pf[ptri * 3 + 2] = eev2v[eev];
      a.fkey[ptri] = k;
    }
  }
  for (int i = lane; i < npt; i += kRow) {
    int ut = tb->meshes[n][config * npt + i];
    LO tv[3];
    for (int j = 0; j < 3; ++j) tv[j] = vertex(tb->tris[n][ut][j]);
    LO ptri = k2f + 2 * npe + i;
    for (int j = 0; j < 3; ++j) pf[ptri * 3 + j] = tv[j];
    a.fkey[ptri] = k;
    for (int eev = 0; eev < 2; ++eev) {
      LO ptet = k2t + 2 * i + eev;
      a.tkey[ptet] = k;
      LO nt4[4] = {tv[0], tv[1], tv[2], eev2v[eev]};
      if (eev == 0) {
        LO tmp = nt4[1];
        nt4[1] = nt4[2];
        nt4[2] = tmp;
      }
      for (int j = 0; j < 4; ++j) pt[ptet * 4 + j] = nt4[j];
    }
  }
}

__global__ void loops_kernel(LO n, LO const* edges, LO const* a2ab, LO const* ab2b,
    I8 const* codes, LO const* ev2v, LO const* tv2v, LO* eev2v, LO* verts, LO* sizes,
    int* error) {
  LO i = thread_index();
  if (i >= n) return;
  Loop loop;
  find_loop(edges[i], a2ab, ab2b, codes, ev2v, tv2v, loop);
  if (loop.size < 0) {
    *error = kBrokenSwapLoop;
    sizes[i] = 0;
    return;
  }
  sizes[i] = loop.size;
  if (loop.size > swap::kMaxLoop) return;
  eev2v[i * 2] = loop.eev2v[0];
  eev2v[i * 2 + 1] = loop.eev2v[1];
  for (int k = 0; k < loop.size; ++k) verts[i * swap::kMaxLoop + k] = loop.verts[k];
}

// 2D: the quadrilateral around an interior edge and its flipped diagonal
__device__ void opposite_verts(LO e, LO const* e2t_a2ab, LO const* e2t_ab2b,
    I8 const* e2t_codes, LO const* tv2v, LO* ov) {
  for (int i = 0; i < 2; ++i) {
    LO et = e2t_a2ab[e] + i;
    int tte = code_which_down(e2t_codes[et]);
    int rot = code_rotation(e2t_codes[et]);
    LO t = e2t_ab2b[et];
    ov[rot] = tv2v[t * 3 + opposite_template(2, 1, tte)];
  }
}

template <int M>
__global__ void swap2d_qualities_kernel(LO ncands, LO const* cands, LO const* e2t_a2ab,
    LO const* e2t_ab2b, I8 const* e2t_codes, LO const* ev2v, LO const* tv2v,
    Real const* coords, Real const* metric, Real const* elem_quals, Real max_length,
    I8* keep, Real* quals) {
  LO cand = thread_index();
  if (cand >= ncands) return;
  constexpr int nc = (M == 1) ? 1 : 3;
  LO e = cands[cand];
  LO ov[2];
  opposite_verts(e, e2t_a2ab, e2t_ab2b, e2t_codes, tv2v, ov);
  double q;
  if (length_between<2, M>(ov[0], ov[1], coords, metric) > max_length) {
    q = -1.0;
  } else {
    double minqual = 1.0;
    for (int i = 0; i < 2; ++i) {
      LO ntv[3] = {ev2v[e * 2 + (1 - i)], ov[i], ov[1 - i]};
      double p[3][2];
      double m[3][nc];
      double const* pp[3];
      double const* ms[3];
      for (int k = 0; k < 3; ++k) {
        for (int j = 0; j < 2; ++j) p[k][j] = coords[ntv[k] * 2 + j];
        for (int j = 0; j < nc; ++j) m[k][j] = metric[ntv[k] * nc + j];
        pp[k] = p[k];
        ms[k] = m[k];
      }
      minqual = math::min2(minqual, element_quality<2, M>(pp, ms));
    }
    q = minqual;
  }
  double old = 1.79769313486231570815e+308;
  for (LO j = e2t_a2ab[e]; j < e2t_a2ab[e + 1]; ++j) old = math::min2(old, elem_quals[e2t_ab2b[j]]);
  if (q > old) {
    keep[e] = 1;
    quals[e] = q;
  }
}

__global__ void swap2d_products(LO nkeys, LO const* keys2edges, LO const* e2t_a2ab,
    LO const* e2t_ab2b, I8 const* e2t_codes, LO const* ev2v, LO const* tv2v, LO* pe, LO* pf) {
  LO k = thread_index();
  if (k >= nkeys) return;
  LO e = keys2edges[k];
  LO ov[2];
  opposite_verts(e, e2t_a2ab, e2t_ab2b, e2t_codes, tv2v, ov);
  pe[k * 2] = ov[0];
  pe[k * 2 + 1] = ov[1];
  for (int i = 0; i < 2; ++i) {
    LO* ntv = pf + (k * 2 + i) * 3;
    ntv[0] = ev2v[e * 2 + (1 - i)];
    ntv[1] = ov[i];
    ntv[2] = ov[1 - i];
  }
}

// the context keeps one device copy of the tables
Tables const* device_tables(Ctx& c) {
  if (!c.swap_tables) {
    Tables t = swap::make_tables();
    auto d = std::make_shared<DArray<unsigned char>>(c, LO(sizeof(Tables)));
    upload(c, *d, reinterpret_cast<unsigned char const*>(&t), LO(sizeof(Tables)));
    c.sync();
    c.swap_tables = d;
  }
  return reinterpret_cast<Tables const*>(
      static_cast<DArray<unsigned char>*>(c.swap_tables.get())->data());
}

// `plans` are the rebuild plans of dimensions 1..dim, scanned
void swap_rebuild(Ctx& c, DMesh& m, LOs const& keys2edges, LOs const* k2p, LO const* nprods,
    LOs const* pv, ModPlan const* plans, SwapCache* cache = nullptr,
    Bytes const* dirty = nullptr, EdgeRings const* rings = nullptr,
    LOs const* prod_keys = nullptr, LOs const* side_zeros = nullptr) {
  int dim = m.dim;
  DMesh nw;
  nw.dim = dim;
  nw.linked = m.linked;
  nw.metric_ncomps = m.metric_ncomps;
  nw.nents[0] = m.nents[0];
  nw.coords = m.coords;
  nw.metric = m.metric;
  nw.vtags = m.vtags;
  nw.itags = m.itags;
  nw.class_id[0] = m.class_id[0];
  nw.class_dim[0] = m.class_dim[0];
  ModOut mo[4];
  SwapCache next;
  CacheMove move{cache, &next, dirty};
  rebuild_same(c, m, nw, 1, plans, mo, cache ? &move : nullptr);
  Products prods[4];
  for (int d = 1; d <= dim; ++d) {
    prods[d].n = nprods[d];
    prods[d].keys2prods = k2p[d];
    prods[d].verts = pv[d];
    prods[d].src_dim = 1;  // products come from their key edge
  }
  place_products(c, m, nw, 1, dim, 1, plans, keys2edges, prods, mo, nullptr,
      cache ? next.valid.data() : nullptr);
  if (cache) *cache = next;
  if (rings) {
    // in 3D the products' sides come from a search around each key
    LO most = nprods[2] * 3 > nprods[3] * 4 ? nprods[2] * 3 : nprods[3] * 4;
    int lanes = fit_lanes(most, c.tuning.side_lanes);
    LocalSides s[2];
    unsigned blocks[2];
    for (int d = 2; d <= 3; ++d) {
      LocalSides& a = s[d - 2];
      a.nuses = nprods[d] * (d + 1);
      a.prod_key = prod_keys[d].data();
      a.k2p_low = k2p[d - 1].data();
      a.pv_high = pv[d].data();
      a.pv_low = pv[d - 1].data();
      a.low_prods2new = mo[d - 1].prods2new.data();
      a.prods2new = mo[d].prods2new.data();
      a.t2low = d == 3 ? m.down[3].data() : ask_down(c, m, 3, 1, nullptr).data();
      a.old_low_verts = verts_of(c, m, d - 1).data();
      a.low_same = plans[d - 2].same.data();
      a.low_offsets = plans[d - 2].offsets.data();
      a.out = nw.down[d].data();
      a.out_codes = nw.down_codes[d].data();
      blocks[d - 2] = unsigned((std::int64_t(a.nuses) * lanes + kBlock - 1) / kBlock);
    }
    if (blocks[0] + blocks[1]) {
      hipLaunchKernelGGL(swap3d_local_down, dim3(blocks[0] + blocks[1]), dim3(kBlock), 0,
          c.stream, lanes, blocks[0], keys2edges.data(), *rings, s[0], s[1], c.error_word());
      OSH_HIP(hipGetLastError());
    }
  } else {
    match_sides(c, nw, prods, mo, side_zeros);
  }
  measure_products(c, nw, mo);
  transfer_pointwise(c, m, nw, mo[dim], 1, keys2edges, k2p[dim], pv[dim]);
  conserve_pass(c, m, nw, 2, 1, keys2edges, k2p[dim], mo[dim]);
  m = nw;
}

// what a 3D pass knows about its candidates' rings, with the storage behind it
struct Rings {
  LOs cands, cand_of, rows;
  EdgeRings r{};
};

// the rings of the marked edges; counts: zeros per edge
void build_rings(Ctx& c, DMesh& m, Bytes const& marks, LOs const& counts, Rings& out) {
  out.cands = collect_marked(c, marks, &out.cand_of);
  LO ncands = out.cands.size();
  if (ncands == 0) return;
  Bytes const* codes;
  LOs const& t2e = ask_down(c, m, 3, 1, &codes);
  out.rows = LOs(c, ncands * kRow);
  OSH_LAUNCH(swap3d_rows, m.nents[3] * 6, c, t2e.data(), marks.data(), out.cand_of.data(),
      counts.data(), out.rows.data());
  out.r = EdgeRings{out.cands.data(), out.cand_of.data(), counts.data(), out.rows.data(),
      t2e.data(), codes->data()};
}

// swap3d_qualities (src/Omega_h_swap3d_qualities.cpp:11-75) with the choice
// of each candidate's triangulation (src/Omega_h_swap3d_choice.hpp):
// configs[e] receives the chosen triangulation (-1 for none) and, when it
// improves on the elements around the edge, keep[e] = 1 and quals[e] its
// quality (entries of other edges are left as they are)
void swap3d_evaluate(Ctx& c, DMesh& m, AdaptOptions const& o, Rings const& rings,
    SwapCache* cache, Bytes& configs, Reals& quals, Bytes& keep) {
  Range quality_range(c, "swap3d_qualities");
  LO ncands = rings.cands.size();
  int md = (m.metric_ncomps == 1) ? 1 : 3;
  // one evaluation keeps up to 70 lanes busy (a loop of seven); four lanes
  // to each one that the choice alone is given, 32 by default
  int lanes = 4 * c.tuning.choose_lanes;
  lanes = lanes < kMinEvalLanes ? kMinEvalLanes : (lanes > 64 ? 64 : lanes);
  lanes = fit_lanes(ncands, lanes);
  OSH_CHECK(lanes >= kMinEvalLanes, "swap: too many candidates");
  EvalArgs a{rings.r, ncands, m.down[1].data(), verts_of(c, m, 3).data(), m.coords.data(),
      m.metric.data(), ask_qualities(c, m).data(), o.max_length_allowed, device_tables(c),
      configs.data(), quals.data(), keep.data(), cache ? cache->valid.data() : nullptr,
      cache ? cache->cfg.data() : nullptr, cache ? cache->keep.data() : nullptr,
      cache ? cache->q.data() : nullptr, c.error_word()};
  int lshift = lanes_shift(lanes);
#define OSH_SWE(M, X) OSH_LAUNCH((swap3d_evaluate_kernel<M, X>), ncands * lanes, c, lshift, a)
  bool mixed = o.precision == 1;
  if (md == 3 && mixed)
    OSH_SWE(3, true);
  else if (md == 3)
    OSH_SWE(3, false);
  else if (mixed)
    OSH_SWE(1, true);
  else
    OSH_SWE(1, false);
#undef OSH_SWE
}

bool swap_edges_3d(Ctx& c, DMesh& m, AdaptOptions const& o, SwapCache* cache) {
  ask_lengths(c, m);
  LO ne = m.nents[1], nf = m.nents[2], nt = m.nents[3];
  // every array of the pass that starts out constant, in one launch
  Fills fills(c);
  SliverLayers layers(c, m, o.nsliver_layers, fills);
  Bytes marks = fills.bytes(ne, 0);
  LOs ring_counts = fills.ints(ne, 0);
  Bytes keep = fills.bytes(ne, 0);
  Bytes state[2] = {fills.bytes(ne, 0), fills.bytes(ne, 0)};
  Bytes dirty;
  if (cache) dirty = fills.bytes(ne, 0);
  ModPlan plans[3];
  LO nents[3] = {ne, nf, nt};
  for (int d = 0; d < 3; ++d) {
    plans[d].ent_dim = d + 1;
    plans[d].key_dim = 1;
    plans[d].nold = nents[d];
    plans[d].same = fills.bytes(nents[d], 1);
    plans[d].counts = fills.ints(nents[d], 1);
  }
  if (cache && !cache->valid.exists()) {
    cache->valid = fills.bytes(ne, 0);
    cache->cfg = Bytes(c, ne);
    cache->keep = Bytes(c, ne);
    cache->q = Reals(c, ne);
  }
  fills.run();
  layers.mark_interior_edges(o.min_quality_desired, marks);
  Rings rings;
  build_rings(c, m, marks, ring_counts, rings);
  LO ncands = rings.cands.size();
  if (ncands == 0) return false;
  Bytes configs(c, ne);
  Reals quals(c, ne);
  swap3d_evaluate(c, m, o, rings, cache, configs, quals, keep);
  bool any = false;
  Bytes keys;
  {
    Range indset_range(c, "find_indset");
    DArray<unsigned long long> dom(c, ncands);
    int first_lanes = fit_lanes(ncands, c.tuning.first_lanes);
    keys = indset_rounds(c, ne, keep, state[0], state[1], &any,
        [&](bool first, I8 const* in, I8* out, IndsetWords w) {
          if (first)
            OSH_LAUNCH(swap3d_indset<true>, ncands * first_lanes, c, first_lanes, rings.r,
                quals.data(), in, out, dom.data(), w);
          else
            OSH_LAUNCH(swap3d_indset<false>, ncands, c, 1, rings.r, quals.data(), in, out,
                dom.data(), w);
        });
  }
  layers.settle();
  if (!any) return false;
  Range modify_range(c, "modify_ents");
  // the plans from the keys, then one scan launch and one wait for the keys,
  // their products and the new numbering of edges, faces and tets
  Tables const* tb = device_tables(c);
  Bytes is_key(c, ncands);
  LOs np[3], off[3], reps[2] = {LOs(c, ncands), LOs(c, ncands)};
  LOs key_off(c, ncands + 1);
  ScanJob jobs[kMaxScanJobs];
  jobs[0] = {is_key.data(), kScanNonzero, ncands, key_off.data(), total_slot(c, 0)};
  KeyPlan kp{};
  for (int d = 0; d < 3; ++d) {
    np[d] = LOs(c, ncands);
    off[d] = LOs(c, ncands + 1);
    jobs[d + 1] = {np[d].data(), kScanLO, ncands, off[d].data(), total_slot(c, d + 1)};
    kp.same[d] = plans[d].same.data();
    kp.counts[d] = plans[d].counts.data();
    kp.nprods[d] = np[d].data();
  }
  kp.is_key = is_key.data();
  kp.reps[0] = reps[0].data();
  kp.reps[1] = reps[1].data();
  kp.dirty = cache ? dirty.data() : nullptr;
  OSH_LAUNCH(swap3d_plan_keys, ncands * kRow, c, rings.r, keys.data(), m.down[3].data(), tb, kp);
  int njobs = 4 + modify_scan_jobs(c, plans, 3, jobs + 4, 4);
  offset_scans(c, jobs, njobs);
  c.wait_totals(0x7fu);
  modify_scan_totals(c, plans, 3, 4);
  LO nkeys = read_slot<LO>(c, 0);
  if (o.verbosity >= 2) std::printf("swapping %d 3D edges\n", int(nkeys));
  LOs keys2edges(c, nkeys);
  LOs k2p[4], pv[4];
  LO nprods[4] = {0, 0, 0, 0};
  KeyProducts pr{};
  pr.is_key = is_key.data();
  pr.key_off = key_off.data();
  pr.reps[0] = reps[0].data();
  pr.reps[1] = reps[1].data();
  pr.keys2edges = keys2edges.data();
  for (int d = 1; d <= 3; ++d) {
    nprods[d] = read_slot<LO>(c, d);
    pv[d] = LOs(c, nprods[d] * (d + 1));
    k2p[d] = LOs(c, nkeys + 1);
    plans[d - 1].reps = LOs(c, nkeys);
    pr.off[d - 1] = off[d - 1].data();
    pr.k2p[d - 1] = k2p[d].data();
    pr.key_reps[d - 1] = plans[d - 1].reps.data();
    pr.pv[d - 1] = pv[d].data();
  }
  LOs prod_keys[4];  // the key of each product face and tet
  prod_keys[2] = LOs(c, nprods[2]);
  prod_keys[3] = LOs(c, nprods[3]);
  pr.fkey = prod_keys[2].data();
  pr.tkey = prod_keys[3].data();
  OSH_LAUNCH(swap3d_products, ncands * kRow, c, ncands, rings.r, m.down[1].data(),
      verts_of(c, m, 3).data(), configs.data(), tb, pr);
  note_changed_parts(c, m, 1, keys2edges);
  swap_rebuild(c, m, keys2edges, k2p, nprods, pv, plans, cache, cache ? &dirty : nullptr,
      &rings.r, prod_keys);
  return true;
}

bool swap_edges_2d(Ctx& c, DMesh& m, AdaptOptions const& o) {
  ask_lengths(c, m);
  LO ne = m.nents[1];
  Fills fills(c);
  SliverLayers layers(c, m, o.nsliver_layers, fills);
  Bytes cand = fills.bytes(ne, 0);
  Bytes keep = fills.bytes(ne, 0);
  KeyedMods km;
  km.fixed_prods[1] = 1;
  km.fixed_prods[2] = 2;
  prepare_keys(m, 1, 1, 2, fills, km);
  LOs side_zeros = fills.ints(m.nents[0], 0);
  fills.run();
  layers.mark_interior_edges(o.min_quality_desired, cand);
  Reals quals(c, ne);  // read where an edge is kept
  LOs cands = collect_marked(c, cand);
  if (cands.size() == 0) return false;
  int md = (m.metric_ncomps == 1) ? 1 : 2;
  Adj const& e2t = ask_up(c, m, 1, 2);
  LOs const& tv2v = verts_of(c, m, 2);
  Reals const& eq = ask_qualities(c, m);
  Range quality_range(c, "swap2d_qualities");
  if (md == 2)
    OSH_LAUNCH(swap2d_qualities_kernel<2>, cands.size(), c, cands.data(), e2t.a2ab.data(),
        e2t.ab2b.data(), e2t.codes.data(), m.down[1].data(), tv2v.data(), m.coords.data(),
        m.metric.data(), eq.data(), o.max_length_allowed, keep.data(), quals.data());
  else
    OSH_LAUNCH(swap2d_qualities_kernel<1>, cands.size(), c, cands.data(), e2t.a2ab.data(),
        e2t.ab2b.data(), e2t.codes.data(), m.down[1].data(), tv2v.data(), m.coords.data(),
        m.metric.data(), eq.data(), o.max_length_allowed, keep.data(), quals.data());
  quality_range.end();
  bool any;
  Bytes keys = find_indset(c, m, 1, quals, keep, &any);
  layers.settle();
  if (!any) return false;
  Range modify_range(c, "modify_ents");
  plan_keys(c, m, 1, 1, 2, keys, km);
  note_changed_parts(c, m, 1, km.keys2kds);
  if (o.verbosity >= 2) std::printf("swapping %d 2D edges\n", int(km.nkeys));
  LOs pv[4];
  pv[1] = LOs(c, km.nkeys * 2);
  pv[2] = LOs(c, km.nkeys * 6);
  OSH_LAUNCH(swap2d_products, km.nkeys, c, km.keys2kds.data(), e2t.a2ab.data(),
      e2t.ab2b.data(), e2t.codes.data(), m.down[1].data(), tv2v.data(), pv[1].data(),
      pv[2].data());
  swap_rebuild(c, m, km.keys2kds, km.k2p, km.nprods, pv, km.plans, nullptr, nullptr, nullptr,
      nullptr, &side_zeros);
  return true;
}

}  // namespace

bool swap_edges(Ctx& c, DMesh& m, AdaptOptions const& o, SwapCache* cache) {
  if (m.dim == 3) return swap_edges_3d(c, m, o, cache);
  return swap_edges_2d(c, m, o);
}

namespace {

__global__ void mark_listed(LO n, LO const* list, I8* marks) {
  LO i = thread_index();
  if (i < n) marks[list[i]] = 1;
}

__global__ void gather_choices(LO n, LO const* edges, I8 const* configs, Real const* quals,
    I8 const* keep, LO* out_cfg, Real* out_q) {
  LO i = thread_index();
  if (i >= n) return;
  LO e = edges[i];
  out_cfg[i] = configs[e];
  out_q[i] = keep[e] ? quals[e] : -1.0;
}

}  // namespace

void swap3d_choices(Ctx& c, DMesh& m, AdaptOptions const& o, LOs const& edges,
    LOs& configs_out, Reals& quals_out) {
  OSH_CHECK(m.dim == 3, "swap3d choices need a 3D mesh");
  LO ne = m.nents[1];
  LO n = edges.size();
  Fills fills(c);
  Bytes marks = fills.bytes(ne, 0);
  LOs counts = fills.ints(ne, 0);
  Bytes configs = fills.bytes(ne, -1);
  Bytes keep = fills.bytes(ne, 0);
  fills.run();
  OSH_LAUNCH(mark_listed, n, c, edges.data(), marks.data());
  Rings rings;
  build_rings(c, m, marks, counts, rings);
  Reals quals(c, ne);  // read where an edge is kept
  if (rings.cands.size() > 0)
    swap3d_evaluate(c, m, o, rings, nullptr, configs, quals, keep);
  configs_out = LOs(c, n);
  quals_out = Reals(c, n);
  OSH_LAUNCH(gather_choices, n, c, edges.data(), configs.data(), quals.data(), keep.data(),
      configs_out.data(), quals_out.data());
}

void find_loops(Ctx& c, DMesh& m, LOs const& edges, LOs& eev2v, LOs& loop_verts, LOs& sizes) {
  LO n = edges.size();
  eev2v = fill_lo(c, n * 2, -1);
  loop_verts = fill_lo(c, n * swap::kMaxLoop, -1);
  sizes = LOs(c, n);
  Adj const& e2t = ask_up(c, m, 1, 3);
  LOs const& tv2v = verts_of(c, m, 3);
  OSH_LAUNCH(loops_kernel, n, c, edges.data(), e2t.a2ab.data(), e2t.ab2b.data(),
      e2t.codes.data(), m.down[1].data(), tv2v.data(), eev2v.data(), loop_verts.data(),
      sizes.data(), c.error_word());
}

}  // namespace osh
