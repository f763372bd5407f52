// Topology rebuild, field transfer, independent sets and marking on the
// device.
//
//   modify_ents_adapt / get_mods2reps / get_rep_counts / get_rep2md_order /
//   assign_new_numbering / modify_conn   src/Omega_h_modify.cpp:20-70,141-517
//   (on one rank the global numbers equal the new local numbers, so the
//   modify_globals exchange reduces to the same scan)
//   transfer_common / transfer_inherit_* src/Omega_h_transfer.cpp:149-180
//   indset::find / QualityCompare         src/Omega_h_indset_inline.hpp:12-72,
//                                         src/Omega_h_indset.cpp:5-35
//   mark_down / mark_dual_layers / mark_sliver_layers src/Omega_h_mark.cpp:12-47,190-212
#include "osh_indset.hpp"
#include "osh_math.hpp"
#include "osh_passes.hpp"

namespace osh {

namespace {

// The plans of a pass's dimensions from its keys, given as a mask over the key
// dimension, in one sweep.  A key is no longer the same and counts its
// products; in the dimensions above, an entity is the same when no key is
// among its lower entities, and each key receives the lowest index among the
// entities above it (the first entry of its row of the upward adjacency,
// whose rows are sorted by index), without building that adjacency.  Job w
// owns the workgroups [first[w], first[w + 1]).
struct SameMarks {
  int n;
  unsigned first[5];
  LO nents[4];
  int deg[4];             // lower entities per entity; 0: the key dimension itself
  LO const* lows[4];
  I8* same[4];
  LO* counts[4];
  LO* first_up[4];
  LO const* key_prods;    // products of the key dimension per entity (null: fixed)
  LO fixed_key_prods;
};

__global__ void __launch_bounds__(kBlock) mark_same_kernel(I8 const* keys, SameMarks j) {
  int w = 0;
  while (w + 1 < j.n && blockIdx.x >= j.first[w + 1]) ++w;
  LO h = LO(blockIdx.x - j.first[w]) * kBlock + LO(threadIdx.x);
  if (h >= j.nents[w]) return;
  int deg = j.deg[w];
  if (deg == 0) {
    bool key = keys[h] != 0;
    j.same[w][h] = key ? 0 : 1;
    j.counts[w][h] = key ? (j.key_prods ? j.key_prods[h] : j.fixed_key_prods) : 1;
    return;
  }
  LO const* lows = j.lows[w] + std::size_t(h) * deg;
  I8 r = 1;
  for (int k = 0; k < deg; ++k) {
    LO l = lows[k];
    if (keys[l]) {
      r = 0;
      atomicMin(&j.first_up[w][l], h);
    }
  }
  j.same[w][h] = r;
  j.counts[w][h] = r;
}

// the keys' representatives (get_mods2reps, src/Omega_h_modify.cpp:20-45)
// count their products (get_rep_counts, :47-70): the lowest entity above the
// key, or in the dimension below the key's first lower entity, where the keys
// of one representative are also chained for their order (get_rep2md_order)
struct RepCounts {
  int n;
  LO const* first_up[4];   // dimensions above
  LO const* down[4];       // the dimension below
  int deg[4];
  LO const* prods[4];      // per key-dimension entity (null: fixed)
  LO fixed[4];
  LO* counts[4];
  LO* head;                // per representative below: a key, or -1
  LO* next;                // per key-dimension entity: the chain's next key
};

__global__ void rep_counts_kernel(LO nkd, I8 const* keys, RepCounts j, int* error) {
  LO kd = thread_index();
  if (kd >= nkd || !keys[kd]) return;
  for (int w = 0; w < j.n; ++w) {
    LO r;
    if (j.first_up[w]) {
      r = j.first_up[w][kd];
      if (r == 0x7fffffff) {  // keeps every index in range until the host sees it
        r = 0;
        *error = kKeyWithoutUp;
      }
    } else {
      r = j.down[w][std::size_t(kd) * j.deg[w]];
      j.next[kd] = atomicExch(&j.head[r], kd);
    }
    atomicAdd(&j.counts[w][r], j.prods[w] ? j.prods[w][kd] : j.fixed[w]);
  }
}

// per key (and one past the last): its product offsets and representatives in
// every dimension and, below the key dimension, how many products of earlier
// keys share its representative
struct KeyList {
  int n;
  int kind[4];  // 0: the key dimension, 1: above, -1: below
  LO const* first_up[4];
  LO const* down[4];
  int deg[4];
  LO const* prod_off[4];  // scan of the products per entity (null: fixed)
  LO fixed[4];
  LO* k2p[4];
  LO* reps[4];
  LO nkd;
  LO const* head;
  LO const* next;
  LO* order;  // per key-dimension entity
};

__global__ void list_keys_kernel(LO n, LO nkeys, LO const* keys2kds, KeyList j) {
  LO k = thread_index();
  if (k >= n) return;
  LO kd = k < nkeys ? keys2kds[k] : j.nkd;
  for (int w = 0; w < j.n; ++w) {
    j.k2p[w][k] = j.prod_off[w] ? j.prod_off[w][kd] : k * j.fixed[w];
    if (k == nkeys) continue;
    LO r = kd;
    if (j.kind[w] > 0) {
      r = j.first_up[w][kd];
      r = r == 0x7fffffff ? 0 : r;
    } else if (j.kind[w] < 0) {
      r = j.down[w][std::size_t(kd) * j.deg[w]];
      // one product a key: the order counts the representative's smaller keys
      LO before = 0;
      for (LO o = j.head[r]; o >= 0; o = j.next[o]) before += o < kd;
      j.order[kd] = before * j.fixed[w];
    }
    j.reps[w][k] = r;
  }
}

// a same entity's new number is its offset (assign_new_numbering,
// src/Omega_h_modify.cpp:141-161), whatever its dimension, so one launch moves
// the same entities of every dimension with all they carry: a lower entity's
// or vertex's new number is read from its own dimension's offsets (a same
// entity's lower entities are same entities).  Bound by memory: about 45 bytes
// in and out per edge, 80 per face, 110 per tet; numbering, classification,
// measures and swap choices in launches of their own, through lists of the
// same entities, took 48 us where this takes 16 us (200,000 edges, 338,000
// faces, 167,000 tets).
struct SameDim {
  int dim;
  LO n;
  I8 const* same;  // null: all are
  LO const* offsets;
  LO* old2new;
  LO const* old_down;
  I8 const* old_codes;
  LO const* low_offsets;  // null: lower entities keep their numbers
  LO* down;
  I8* codes;
  LO const* old_verts;
  LO const* vert_offsets;
  LO* verts;
  LO const* old_ids;
  I8 const* old_dims;
  LO* ids;
  I8* dims;
  Real const* old_measure;
  Real* measure;
  // rows of reals (dimension 0: coordinates and metric)
  Real const* old_rows[2];
  Real* rows[2];
  int ncomps[2];
};

struct SameCache {
  I8 const* dirty;
  I8 const* valid;
  I8 const* cfg;
  I8 const* keep;
  Real const* q;
  I8* n_valid;
  I8* n_cfg;
  I8* n_keep;
  Real* n_q;
};

// job w owns the workgroups [first[w], first[w + 1]), so that every branch on
// the dimension is uniform
struct SameJobs {
  int n;
  unsigned first[5];
  SameDim d[4];
  SameCache cache;  // of the edges, when cache.valid
};

__device__ __forceinline__ LO renumber(LO const* offsets, LO l) {
  return offsets ? offsets[l] : l;
}

__global__ void __launch_bounds__(kBlock) rebuild_same_kernel(SameJobs j) {
  int w = 0;
  while (w + 1 < j.n && blockIdx.x >= j.first[w + 1]) ++w;
  SameDim const& a = j.d[w];
  LO o = LO(blockIdx.x - j.first[w]) * kBlock + LO(threadIdx.x);
  if (o >= a.n) return;
  bool keep = !a.same || a.same[o];
  LO x = a.offsets[o];
  if (a.old2new) a.old2new[o] = keep ? x : -1;
  if (!keep) return;
  a.ids[x] = a.old_ids[o];
  a.dims[x] = a.old_dims[o];
  if (a.measure) a.measure[x] = a.old_measure[o];
  if (a.dim == 0) {
    for (int r = 0; r < 2; ++r)
      for (int k = 0; k < a.ncomps[r]; ++k)
        a.rows[r][std::size_t(x) * a.ncomps[r] + k] = a.old_rows[r][std::size_t(o) * a.ncomps[r] + k];
  } else if (a.dim == 1) {
    int2 v = reinterpret_cast<int2 const*>(a.old_down)[o];
    reinterpret_cast<int2*>(a.down)[x] =
        make_int2(renumber(a.low_offsets, v.x), renumber(a.low_offsets, v.y));
    if (j.cache.valid) {
      bool ok = j.cache.valid[o] && !j.cache.dirty[o];
      j.cache.n_valid[x] = I8(ok);
      if (ok) {
        j.cache.n_cfg[x] = j.cache.cfg[o];
        j.cache.n_keep[x] = j.cache.keep[o];
        j.cache.n_q[x] = j.cache.q[o];
      }
    }
  } else if (a.dim == 2) {
    std::size_t so = std::size_t(o) * 3, sx = std::size_t(x) * 3;
    LO l[3], v[3];
    I8 c[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      l[k] = a.old_down[so + k];
      v[k] = a.old_verts[so + k];
      c[k] = a.old_codes[so + k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      a.down[sx + k] = renumber(a.low_offsets, l[k]);
      a.verts[sx + k] = renumber(a.vert_offsets, v[k]);
      a.codes[sx + k] = c[k];
    }
  } else {
    int4 l = reinterpret_cast<int4 const*>(a.old_down)[o];
    int4 v = reinterpret_cast<int4 const*>(a.old_verts)[o];
    reinterpret_cast<int4*>(a.down)[x] =
        make_int4(renumber(a.low_offsets, l.x), renumber(a.low_offsets, l.y),
            renumber(a.low_offsets, l.z), renumber(a.low_offsets, l.w));
    reinterpret_cast<int4*>(a.verts)[x] =
        make_int4(renumber(a.vert_offsets, v.x), renumber(a.vert_offsets, v.y),
            renumber(a.vert_offsets, v.z), renumber(a.vert_offsets, v.w));
    // the four codes are one word
    reinterpret_cast<int*>(a.codes)[x] = reinterpret_cast<int const*>(a.old_codes)[o];
  }
}

// the products' new numbers, following their representative
// (src/Omega_h_modify.cpp:141-161), with their vertex lists and their
// classification, inherited from the entity each came from
// (src/Omega_h_transfer.cpp:20-34,212-267).  A key's products take
// consecutive numbers, so kProdLanes threads per key and dimension share them
// without talking to each other.
constexpr int kProdLanes = 8;

struct PlaceDim {
  LO const* reps;
  LO const* offsets;
  LO const* order;  // products sit after their representative, in this order
  LO const* keys2prods;
  LO* prods2new;
  int nverts;  // 0 for vertices
  LO const* pverts;
  LO* verts;
  LO const* src;  // null: the key
  int src_dim;
  I8 const* src_dims;
  LO const* ids_a;
  I8 const* dims_a;
  LO const* ids_b;
  I8 const* dims_b;
  LO* ids;
  I8* dims;
  LO* src_out;
  I8* zeroed;
};

struct PlaceJobs {
  LO const* keys2kds;
  PlaceDim d[4];
};

__global__ void __launch_bounds__(kBlock) place_products_kernel(std::int64_t nt, LO nkeys,
    PlaceJobs j) {
  std::int64_t t = thread_index64();
  if (t >= nt) return;
  std::int64_t row = t / kProdLanes;
  PlaceDim const& a = j.d[row / nkeys];
  LO k = LO(row % nkeys);
  int lane = int(t % kProdLanes);
  LO first = a.keys2prods[k];
  LO end = a.keys2prods[k + 1];
  LO key = j.keys2kds[k];
  LO base = a.offsets[a.reps[k]];
  if (a.order) base += a.order[key] + 1;
  for (LO p = first + lane; p < end; p += kProdLanes) {
    LO w = base + (p - first);
    a.prods2new[p] = w;
    for (int v = 0; v < a.nverts; ++v)
      a.verts[std::size_t(w) * a.nverts + v] = a.pverts[std::size_t(p) * a.nverts + v];
    LO s = a.src ? a.src[p] : key;
    bool second = a.src_dims && a.src_dims[p] != a.src_dim;
    a.ids[w] = second ? a.ids_b[s] : a.ids_a[s];
    a.dims[w] = second ? a.dims_b[s] : a.dims_a[s];
    if (a.src_out) a.src_out[p] = s;
    if (a.zeroed) a.zeroed[w] = 0;
  }
}

// one launch for a transferred tag: threads [0, nold) copy the old entities
// that survive, the rest place the products' values
// (src/Omega_h_transfer.cpp:631-653)
template <class T>
__global__ void scatter_data(LO n, LO nold, int nc, LO const* old2new, T const* old_data,
    LO const* prods2new, T const* pdata, T* data) {
  LO i = thread_index();
  if (i >= n) return;
  bool prod = i >= nold;
  LO p = i - nold;
  LO w = prod ? prods2new[p] : old2new[i];
  if (w < 0) return;
  T const* from = prod ? pdata + std::size_t(p) * nc : old_data + std::size_t(i) * nc;
  for (int k = 0; k < nc; ++k) data[std::size_t(w) * nc + k] = from[k];
}

// row p of out = row src[p] of in
__global__ void gather_rows(LO n, int nc, LO const* src, Real const* in, Real* out) {
  LO p = thread_index();
  if (p >= n) return;
  for (int k = 0; k < nc; ++k) out[std::size_t(p) * nc + k] = in[std::size_t(src[p]) * nc + k];
}

// transfer_pointwise_tmpl (src/Omega_h_transfer.cpp:515-563): each product
// takes the old element around its key (rows in the order of the upward
// adjacency) in which its centroid has the largest smallest barycentric
// coordinate, the first one on ties (and the first one of all when its
// distance is not a number, which nothing compares below).
//
// kPointLanes threads per product (fewer when they would not fit a launch) share the row and reduce with shuffles: a
// pass has a few thousand products, and one thread per key walked all its
// products' rows one gather after another (292 us a launch on the 14^3 box,
// now under 10 us).
constexpr int kPointLanes = 16;

template <int D>
__global__ void pointwise_kernel(LO nt, int lshift, LO nkeys, LO const* keys2kds, LO const* keys2prods,
    LO const* up_a2ab, LO const* up_ab2b, LO const* old_ev2v, Real const* old_coords,
    LO const* prod_verts, Real const* new_coords, LO* best) {
  LO t = thread_index();
  int lanes = 1 << lshift;
  LO nprods = nt >> lshift;
  LO p = t >> lshift;
  int lane = int(t) & (lanes - 1);
  bool valid = p < nprods;  // groups past the end stay for the shuffles
  LO kd = valid ? keys2kds[row_of(p, nkeys, keys2prods)] : 0;
  LO row = valid ? up_a2ab[kd] : 0;
  LO end = valid ? up_a2ab[kd + 1] : 0;
  double x[3] = {0.0, 0.0, 0.0};
  if (valid) {
    LO v0 = prod_verts[std::size_t(p) * (D + 1)];
    for (int j = 0; j < D; ++j) x[j] = new_coords[std::size_t(v0) * D + j];
    for (int i = 1; i <= D; ++i) {
      LO vi = prod_verts[std::size_t(p) * (D + 1) + i];
      for (int j = 0; j < D; ++j) x[j] = x[j] + new_coords[std::size_t(vi) * D + j];
    }
    for (int j = 0; j < D; ++j) x[j] = x[j] / double(D + 1);
  }
  LO pos = 0x7fffffff;  // the row position of the best element so far
  double bd = __builtin_inf();
  bool first_nan = false;
  for (LO ke = row + lane; ke < end; ke += lanes) {
    LO e = up_ab2b[ke];
    double pp[D + 1][3];
    for (int i = 0; i <= D; ++i) {
      LO v = old_ev2v[std::size_t(e) * (D + 1) + i];
      for (int j = 0; j < D; ++j) pp[i][j] = old_coords[std::size_t(v) * D + j];
    }
    double xi[D + 1];
    barycentric<D>(x, pp, xi);
    double mn = xi[0];
    for (int i = 1; i <= D; ++i) mn = (mn < xi[i]) ? mn : xi[i];
    double dist = -mn;
    if (dist < bd) {
      pos = ke;
      bd = dist;
    }
    if (ke == row && dist != dist) first_nan = true;
  }
  int nan = first_nan ? 1 : 0;
  for (int d = lanes / 2; d > 0; d >>= 1) {
    double od = __shfl_xor(bd, d, 64);
    LO op = __shfl_xor(pos, d, 64);
    nan |= __shfl_xor(nan, d, 64);
    if (od < bd || (od == bd && op < pos)) {
      bd = od;
      pos = op;
    }
  }
  if (valid && lane == 0)
    best[p] = row < end ? up_ab2b[(nan || pos == 0x7fffffff) ? row : pos] : -1;
}

// an inheritance tag of the new entities: survivors keep theirs, products
// inherit as they do their classification
__global__ void inherit_kernel(LO n, LO nold, int nc, LO const* old2new, Real const* old_vals,
    LO const* prods2new, LO const* src, int src_dim, I8 const* src_dims, Real const* vals_a,
    Real const* vals_b, Real* out) {
  LO i = thread_index();
  if (i >= n) return;
  if (i < nold) {
    LO w = old2new[i];
    if (w < 0) return;
    for (int k = 0; k < nc; ++k)
      out[std::size_t(w) * nc + k] = old_vals[std::size_t(i) * nc + k];
    return;
  }
  LO p = i - nold;
  int sd = src_dims ? src_dims[p] : src_dim;
  Real const* from = (sd != src_dim) ? vals_b : vals_a;
  LO s = src[p];
  LO w = prods2new[p];
  for (int k = 0; k < nc; ++k) out[std::size_t(w) * nc + k] = from[std::size_t(s) * nc + k];
}

// an undecided node's next state
template <bool FIRST>
__device__ __forceinline__ I8 indset_node(LO v, LO const* a2ab, LO const* ab2b, Real const* q,
    I8 const* old_state, unsigned long long* dom) {
  LO b = a2ab[v], e = a2ab[v + 1];
  bool undecided = false;
  if (!FIRST && e - b <= kDomBits) {
    unsigned long long mask = dom[v];
    while (mask) {
      int j = __ffsll(static_cast<long long>(mask)) - 1;
      mask &= mask - 1;
      I8 su = old_state[ab2b[b + j]];
      if (su == 1) return 0;
      if (su == 2) undecided = true;
    }
  } else {
    unsigned long long mask = 0;
    Real qv = q[v];
    for (LO j = b; j < e; ++j) {
      LO u = ab2b[j];
      I8 su = indset_state<FIRST>(old_state, u);
      if (su == 0) continue;
      Real qu = q[u];
      bool beaten = (qu != qv) ? (qu < qv) : (u < v);
      if (beaten) continue;
      if (su == 1) return 0;
      undecided = true;
      if (FIRST && j - b < kDomBits) mask |= 1ull << (j - b);
    }
    if (FIRST) dom[v] = mask;
  }
  return undecided ? 2 : 1;
}

template <bool FIRST>
__global__ void indset_iteration(LO n, LO const* a2ab, LO const* ab2b, Real const* q,
    I8 const* old_state, I8* new_state, unsigned long long* dom, IndsetWords w) {
  LO v = thread_index();
  if (v >= n) return;
  I8 s = indset_state<FIRST>(old_state, v);
  I8 r = s == 2 ? indset_node<FIRST>(v, a2ab, ab2b, q, old_state, dom) : s;
  new_state[v] = r;
  tell_round(s, r, w);
}

// the first round for edges with `lanes` threads per edge (a power of two,
// Tuning::first_lanes): each takes every lanes-th row position, and the
// group ORs its findings, so the row's gathers run side by side instead of
// one after another
template <int NEPC>
__global__ void indset_first_edges(LO nt, int lanes, LO const* e2c_a2ab, LO const* e2c_ab2b,
    LO const* c2e, Real const* q, I8 const* cands, I8* new_state, unsigned long long* dom,
    IndsetWords w) {
  LO t = thread_index();
  if (t >= nt) return;
  LO v = t / lanes;
  int lane = t % lanes;
  I8 s = cands[v] ? I8(2) : I8(0);
  unsigned long long mask = 0;
  int undecided = 0;
  if (s == 2) {
    LO b = e2c_a2ab[v], e = e2c_a2ab[v + 1];
    Real qv = q[v];
    LO np = (e - b) * NEPC;
    for (LO p = lane; p < np; p += lanes) {
      LO u = c2e[e2c_ab2b[b + p / NEPC] * NEPC + p % NEPC];
      if (u == v || !cands[u]) continue;
      Real qu = q[u];
      bool beaten = (qu != qv) ? (qu < qv) : (u < v);
      if (beaten) continue;
      undecided = 1;
      if (p < kDomBits) mask |= 1ull << p;
    }
  }
  for (int d = lanes / 2; d > 0; d >>= 1) {
    mask |= __shfl_xor(mask, d, 64);
    undecided |= __shfl_xor(undecided, d, 64);
  }
  if (lane != 0) return;
  I8 r = (s == 2 && !undecided) ? I8(1) : s;
  new_state[v] = r;
  if (s == 2) dom[v] = mask;
  tell_round(s, r, w);
}

// the same round for edges, whose star (edges_across_tris/tets,
// src/Omega_h_adj.cpp:532-589) is the set of other edges of the elements
// around the edge: read through the edge -> element adjacency instead of a
// built star (an edge met twice is checked twice, which changes nothing);
// row position (j, k) is bit j * NEPC + k of `dom`.  Rounds after the first.
template <int NEPC>
__device__ __forceinline__ I8 indset_edge(LO v, LO const* e2c_a2ab, LO const* e2c_ab2b,
    LO const* c2e, Real const* q, I8 const* old_state, unsigned long long const* dom) {
  LO b = e2c_a2ab[v], e = e2c_a2ab[v + 1];
  bool undecided = false;
  if ((e - b) * NEPC <= kDomBits) {
    unsigned long long mask = dom[v];
    while (mask) {
      int p = __ffsll(static_cast<long long>(mask)) - 1;
      mask &= mask - 1;
      I8 su = old_state[c2e[e2c_ab2b[b + p / NEPC] * NEPC + p % NEPC]];
      if (su == 1) return 0;
      if (su == 2) undecided = true;
    }
  } else {
    Real qv = q[v];
    for (LO j = b; j < e; ++j) {
      LO const* ce = c2e + e2c_ab2b[j] * NEPC;
#pragma unroll
      for (int k = 0; k < NEPC; ++k) {
        LO u = ce[k];
        if (u == v) continue;
        I8 su = old_state[u];
        if (su == 0) continue;
        Real qu = q[u];
        bool beaten = (qu != qv) ? (qu < qv) : (u < v);
        if (beaten) continue;
        if (su == 1) return 0;
        undecided = true;
      }
    }
  }
  return undecided ? 2 : 1;
}

template <int NEPC>
__global__ void indset_iteration_edges(LO n, LO const* e2c_a2ab, LO const* e2c_ab2b,
    LO const* c2e, Real const* q, I8 const* old_state, I8* new_state,
    unsigned long long const* dom, IndsetWords w) {
  LO v = thread_index();
  if (v >= n) return;
  I8 s = old_state[v];
  I8 r = s == 2 ? indset_edge<NEPC>(v, e2c_a2ab, e2c_ab2b, c2e, q, old_state, dom) : s;
  new_state[v] = r;
  tell_round(s, r, w);
}

__global__ void mark_down_kernel(LO nl, LO const* a2ab, LO const* ab2b, I8 const* marks, I8* out) {
  LO l = thread_index();
  if (l >= nl) return;
  I8 r = 0;
  for (LO j = a2ab[l]; j < a2ab[l + 1]; ++j)
    if (marks[ab2b[j]]) r = 1;
  out[l] = r;
}

// the same marks by scattering from the marked high entities, for when the
// upward adjacency is not built
__global__ void mark_down_scatter(LO nh, int deg, LO const* hl2l, I8 const* marks, I8* out) {
  LO h = thread_index();
  if (h >= nh || !marks[h]) return;
  for (int j = 0; j < deg; ++j) out[hl2l[h * deg + j]] = 1;
}

__global__ void below_kernel(LO n, Real const* q, Real ceil, I8* out) {
  LO i = thread_index();
  if (i < n) out[i] = q[i] < ceil;
}

// graph_reduce over the dual graph with max (src/Omega_h_graph.cpp:62-80 on
// elements_across_sides, src/Omega_h_adj.cpp:591-657): the max over the
// elements across each side that has two, -128 for an element with none; a
// side with more than two elements (not a manifold mesh) is an error.  The
// first layer: the input is the sliver test q < ceil.
template <int NSPE>
__device__ __forceinline__ I8 dual_max_at(LO e, LO const* es2s,
    unsigned long long const* side_elems, Real const* q, Real ceil, int* error) {
  I8 r = -128;
#pragma unroll
  for (int j = 0; j < NSPE; ++j) {
    unsigned long long w = side_elems[es2s[e * NSPE + j]];
    unsigned count = unsigned(w >> 32);
    if (count == 2) {
      LO o = LO(unsigned(w)) - e;
      I8 x = I8(q[o] < ceil);
      r = (r < x) ? x : r;
    } else if (count > 2) {
      *error = kNonManifoldSide;
    }
  }
  return r;
}

__global__ void dual_max_kernel(LO n, int nspe, LO const* es2s,
    unsigned long long const* side_elems, Real const* q, Real ceil, I8* out, unsigned* word,
    unsigned tag, int* error) {
  LO e = thread_index();
  if (e >= n) return;
  I8 r = nspe == 4 ? dual_max_at<4>(e, es2s, side_elems, q, ceil, error)
                   : dual_max_at<3>(e, es2s, side_elems, q, ceil, error);
  out[e] = r;
  tell(r < 0, word, tag);
}

// The same in a mesh known to be linked (DMesh::linked), without the per-side
// words, whose 660,000 atomics took 18 of a pass's 34 us for four layers at
// 165,000 tets: the few elements of a layer count themselves at their sides,
// and an element is in the next layer when one of its sides has a count that
// is not its own.  A side's counts are two bits a layer of one word.
constexpr int kCountedLayers = 16;
constexpr int kUnlinkedWord = 3;  // the sets and the star sweeps use the others

// the interior edges of an element, marked by the sweep that marks it
struct EdgeMarks {
  LO const* e2e;
  I8 const* edim;
  I8* marks;  // null: not asked for
};

template <int NSPE>
__device__ __forceinline__ void mark_edges(LO e, EdgeMarks const& a) {
  constexpr int nepe = NSPE == 4 ? 6 : 3;
#pragma unroll
  for (int i = 0; i < nepe; ++i) {
    LO ed = a.e2e[std::size_t(e) * nepe + i];
    if (a.edim[ed] == NSPE - 1) a.marks[ed] = 1;
  }
}

template <int NSPE>
__global__ void mark_interior_edges_kernel(LO n, I8 const* elem_marks, EdgeMarks edges) {
  LO e = thread_index();
  if (e < n && elem_marks[e]) mark_edges<NSPE>(e, edges);
}

template <int NSPE>
__global__ void sliver_layer(LO n, int layer, int nlayers, LO const* es2s, Real const* q,
    Real ceil, unsigned* counts, I8* marks, EdgeMarks edges) {
  LO e = thread_index();
  if (e >= n) return;
  LO sides[NSPE];
  bool in = false;
  if (layer == 0) in = q[e] < ceil;
  if (layer != 0 || in) {
#pragma unroll
    for (int j = 0; j < NSPE; ++j) sides[j] = es2s[std::size_t(e) * NSPE + j];
  }
  if (layer != 0) {
    unsigned own = marks[e] != 0;
#pragma unroll
    for (int j = 0; j < NSPE; ++j)
      in = in || ((counts[sides[j]] >> (2 * (layer - 1))) & 3u) > own;
  }
  marks[e] = in;
  if (!in) return;
  if (layer < nlayers) {
#pragma unroll
    for (int j = 0; j < NSPE; ++j) atomicAdd(&counts[sides[j]], 1u << (2 * layer));
  } else if (edges.marks) {
    mark_edges<NSPE>(e, edges);
  }
}

// a later layer, pushed from the marked elements (the first one's output has
// looked at every side): few elements are marked, and the rest read one byte
// instead of four side words (2.5 us against 4.5 us at 167,000 tets).  `out`
// starts at 0; an element without neighbors keeps its -128.
template <int NSPE>
__global__ void push_layer_kernel(LO n, LO const* es2s, unsigned long long const* side_elems,
    I8 const* in, I8* out) {
  LO e = thread_index();
  if (e >= n) return;
  I8 s = in[e];
  if (s == 0) return;
  if (s < 0) {
    out[e] = s;
    return;
  }
#pragma unroll
  for (int j = 0; j < NSPE; ++j) {
    unsigned long long w = side_elems[es2s[std::size_t(e) * NSPE + j]];
    if (unsigned(w >> 32) == 2) out[LO(unsigned(w)) - e] = 1;
  }
}

}  // namespace

void prepare_keys(DMesh const& old, int key_dim, int d0, int d1, Fills& fills, KeyedMods& out) {
  for (int d = d0; d <= d1; ++d) {
    if (d < key_dim) {
      out.plans[d - d0].counts = fills.ints(old.nents[d], 1);
      out.head = fills.ints(old.nents[d], -1);
    } else if (d > key_dim) {
      out.first_up[d] = fills.ints(old.nents[key_dim], 0x7fffffff);
    }
  }
}

void plan_keys(Ctx& c, DMesh& old, int key_dim, int d0, int d1, Bytes const& keys,
    KeyedMods& out) {
  LO nkd = old.nents[key_dim];
  int nd = d1 - d0 + 1;
  OSH_CHECK(nd >= 1 && nd <= 4 && key_dim - d0 <= 1 && key_dim >= d0, "plan_keys: dimensions");
  LOs next;
  SameMarks sm{};
  RepCounts rc{};
  KeyList kl{};
  unsigned blocks = 0;
  for (int d = d0; d <= d1; ++d) {
    ModPlan& plan = out.plans[d - d0];
    plan.ent_dim = d;
    plan.key_dim = key_dim;
    plan.nold = old.nents[d];
    LO const* prods = out.prod_counts[d].exists() ? out.prod_counts[d].data() : nullptr;
    int w = kl.n++;
    kl.kind[w] = d == key_dim ? 0 : (d > key_dim ? 1 : -1);
    kl.fixed[w] = out.fixed_prods[d];
    if (d < key_dim) {
      // every entity stays; without a `same` array all are the same
      OSH_CHECK(!prods, "plan_keys: a fixed count below the keys");
      next = LOs(c, nkd);
      out.order = LOs(c, nkd);
      kl.deg[w] = simplex_degree(key_dim, d);
      kl.down[w] = ask_down(c, old, key_dim, d, nullptr).data();
      kl.head = rc.head = out.head.data();
      rc.next = next.data();
      kl.next = next.data();
      kl.order = out.order.data();
    } else {
      plan.same = Bytes(c, plan.nold);
      plan.counts = LOs(c, plan.nold);
      int v = sm.n;
      sm.first[v] = blocks;
      blocks += nblocks(plan.nold);
      sm.first[v + 1] = blocks;
      sm.nents[v] = plan.nold;
      sm.same[v] = plan.same.data();
      sm.counts[v] = plan.counts.data();
      if (d == key_dim) {
        sm.key_prods = prods;
        sm.fixed_key_prods = out.fixed_prods[d];
      } else {
        sm.deg[v] = simplex_degree(d, key_dim);
        sm.lows[v] = ask_down(c, old, d, key_dim, nullptr).data();
        sm.first_up[v] = out.first_up[d].data();
        kl.first_up[w] = out.first_up[d].data();
      }
      ++sm.n;
    }
    if (d != key_dim) {
      int r = rc.n++;
      rc.first_up[r] = kl.first_up[w];
      rc.down[r] = kl.down[w];
      rc.deg[r] = kl.deg[w];
      rc.prods[r] = prods;
      rc.fixed[r] = kl.fixed[w];
      rc.counts[r] = plan.counts.data();
    }
  }
  hipLaunchKernelGGL(mark_same_kernel, dim3(blocks), dim3(kBlock), 0, c.stream, keys.data(), sm);
  OSH_HIP(hipGetLastError());
  if (rc.n) OSH_LAUNCH(rep_counts_kernel, nkd, c, keys.data(), rc, c.error_word());
  // the keys, their products and every dimension's new numbering by one scan
  // and one wait
  ScanJob jobs[kMaxScanJobs];
  LOs off[4];
  out.keys2kds = LOs(c, nkd);
  int nj = 0;
  jobs[nj++] = {keys.data(), kScanNonzero, nkd, nullptr, total_slot(c, 0),
      out.keys2kds.data()};
  for (int d = d0; d <= d1; ++d) {
    if (!out.prod_counts[d].exists()) continue;
    off[d] = LOs(c, nkd + 1);
    kl.prod_off[d - d0] = off[d].data();
    jobs[nj++] = {out.prod_counts[d].data(), kScanLO, nkd, off[d].data(),
        total_slot(c, 1 + d)};
  }
  nj += modify_scan_jobs(c, out.plans, nd, jobs + nj, 5);
  offset_scans(c, jobs, nj);
  unsigned slots = 1u;
  for (int d = d0; d <= d1; ++d)
    slots |= (out.prod_counts[d].exists() ? 1u << (1 + d) : 0u) | 1u << (5 + d - d0);
  c.wait_totals(slots);
  modify_scan_totals(c, out.plans, nd, 5);
  out.nkeys = read_slot<LO>(c, 0);
  out.keys2kds.shrink(out.nkeys);
  for (int d = d0; d <= d1; ++d) {
    out.nprods[d] = out.prod_counts[d].exists() ? read_slot<LO>(c, 1 + d)
                                                 : out.nkeys * out.fixed_prods[d];
    out.k2p[d] = LOs(c, out.nkeys + 1);
    out.plans[d - d0].reps = LOs(c, out.nkeys);
    kl.k2p[d - d0] = out.k2p[d].data();
    kl.reps[d - d0] = out.plans[d - d0].reps.data();
  }
  kl.nkd = nkd;
  OSH_LAUNCH(list_keys_kernel, out.nkeys + 1, c, out.nkeys, out.keys2kds.data(), kl);
}

int modify_scan_jobs(Ctx& c, ModPlan* plans, int nplans, ScanJob* jobs, int first_slot) {
  for (int i = 0; i < nplans; ++i) {
    ModPlan& p = plans[i];
    p.offsets = LOs(c, p.nold + 1);
    jobs[i] = {p.counts.data(), kScanLO, p.nold, p.offsets.data(),
        total_slot(c, first_slot + i)};
  }
  return nplans;
}

void modify_scan_totals(Ctx& c, ModPlan* plans, int nplans, int first_slot) {
  for (int i = 0; i < nplans; ++i) plans[i].nnew = read_slot<LO>(c, first_slot + i);
}

bool has_tags(DMesh const& m) {
  return !m.vtags.empty() || !m.itags.empty() || !m.etags.empty();
}

void rebuild_same(Ctx& c, DMesh& old, DMesh& nw, int d0, ModPlan const* plans, ModOut* mo,
    CacheMove const* cache) {
  int dim = old.dim;
  bool tags = has_tags(old);
  SameJobs j{};
  unsigned blocks = 0;
  for (int d = d0; d <= dim; ++d) {
    ModPlan const& p = plans[d - d0];
    LO nnew = p.nnew;
    int deg = d + 1;
    mo[d].nold = p.nold;
    mo[d].nnew = nnew;
    nw.nents[d] = nnew;
    SameDim& a = j.d[j.n];
    a.dim = d;
    a.n = p.nold;
    a.same = p.same.exists() ? p.same.data() : nullptr;
    a.offsets = p.offsets.data();
    if (tags) {
      mo[d].old2new = LOs(c, p.nold);
      a.old2new = mo[d].old2new.data();
    }
    nw.class_id[d] = LOs(c, nnew);
    nw.class_dim[d] = Bytes(c, nnew);
    a.old_ids = old.class_id[d].data();
    a.old_dims = old.class_dim[d].data();
    a.ids = nw.class_id[d].data();
    a.dims = nw.class_dim[d].data();
    if (d == 0) {
      nw.coords = Reals(c, nnew * dim);
      nw.metric = Reals(c, nnew * old.metric_ncomps);
      a.old_rows[0] = old.coords.data();
      a.old_rows[1] = old.metric.data();
      a.rows[0] = nw.coords.data();
      a.rows[1] = nw.metric.data();
      a.ncomps[0] = dim;
      a.ncomps[1] = old.metric_ncomps;
    } else {
      nw.down[d] = LOs(c, nnew * deg);
      a.old_down = old.down[d].data();
      a.down = nw.down[d].data();
      a.low_offsets = d > d0 ? plans[d - 1 - d0].offsets.data() : nullptr;
    }
    if (d >= 2) {
      nw.down_codes[d] = Bytes(c, nnew * deg);
      nw.verts[d] = LOs(c, nnew * deg);
      a.old_codes = old.down_codes[d].data();
      a.codes = nw.down_codes[d].data();
      a.old_verts = verts_of(c, old, d).data();
      a.verts = nw.verts[d].data();
      a.vert_offsets = d0 == 0 ? plans[0].offsets.data() : nullptr;
    }
    if (d == 1) {
      nw.length = Reals(c, nnew);
      a.old_measure = ask_lengths(c, old).data();
      a.measure = nw.length.data();
    }
    if (d == dim) {
      nw.quality = Reals(c, nnew);
      a.old_measure = ask_qualities(c, old).data();
      a.measure = nw.quality.data();
    }
    j.first[j.n] = blocks;
    blocks += nblocks(p.nold);
    ++j.n;
    j.first[j.n] = blocks;
  }
  if (cache) {
    LO nnew = nw.nents[1];
    cache->to->valid = Bytes(c, nnew);
    cache->to->cfg = Bytes(c, nnew);
    cache->to->keep = Bytes(c, nnew);
    cache->to->q = Reals(c, nnew);
    j.cache = SameCache{cache->dirty->data(), cache->from->valid.data(),
        cache->from->cfg.data(), cache->from->keep.data(), cache->from->q.data(),
        cache->to->valid.data(), cache->to->cfg.data(), cache->to->keep.data(),
        cache->to->q.data()};
  }
  if (blocks == 0) return;
  hipLaunchKernelGGL(rebuild_same_kernel, dim3(blocks), dim3(kBlock), 0, c.stream, j);
  OSH_HIP(hipGetLastError());
}

void place_products(Ctx& c, DMesh& old, DMesh& nw, int d0, int d1, int plan0,
    ModPlan const* plans, LOs const& keys2kds, Products const* prods, ModOut* mo,
    LOs const* order, I8* new_edges_valid) {
  LO nkeys = keys2kds.size();
  PlaceJobs j{};
  j.keys2kds = keys2kds.data();
  LOs src[4];
  for (int d = d0; d <= d1; ++d) {
    ModPlan const& plan = plans[d - plan0];
    Products const& p = prods[d];
    PlaceDim& a = j.d[d - d0];
    mo[d].nprods = p.n;
    mo[d].prods2new = LOs(c, p.n);
    a.order = plan.key_dim > d ? order->data() : nullptr;
    a.reps = plan.reps.data();
    a.offsets = plan.offsets.data();
    a.keys2prods = p.keys2prods.data();
    a.prods2new = mo[d].prods2new.data();
    if (d >= 1) {
      a.nverts = d + 1;
      a.pverts = p.verts.data();
      a.verts = d == 1 ? nw.down[1].data() : nw.verts[d].data();
    }
    int sd = p.src_dim;
    int other = (p.src_dims.exists() && sd + 1 <= old.dim) ? sd + 1 : sd;
    a.src = p.src.exists() ? p.src.data() : nullptr;
    a.src_dim = sd;
    a.src_dims = p.src_dims.exists() ? p.src_dims.data() : nullptr;
    a.ids_a = old.class_id[sd].data();
    a.dims_a = old.class_dim[sd].data();
    a.ids_b = old.class_id[other].data();
    a.dims_b = old.class_dim[other].data();
    a.ids = nw.class_id[d].data();
    a.dims = nw.class_dim[d].data();
    if (!old.itags.empty()) {
      src[d] = LOs(c, p.n);
      a.src_out = src[d].data();
    }
    if (d == 1) a.zeroed = new_edges_valid;
  }
  int nd = d1 - d0 + 1;
  OSH_LAUNCH64(place_products_kernel, std::int64_t(nkeys) * nd * kProdLanes, c, nkeys, j);
  if (nw.itags.size() != old.itags.size()) nw.itags = old.itags;
  for (int d = d0; d <= d1; ++d) {
    Products const& p = prods[d];
    int sd = p.src_dim;
    int other = (p.src_dims.exists() && sd + 1 <= old.dim) ? sd + 1 : sd;
    for (std::size_t t = 0; t < old.itags.size(); ++t) {
      auto const& a = old.itags[t];
      Reals out(c, mo[d].nnew * a.ncomps);
      OSH_LAUNCH(inherit_kernel, mo[d].nold + p.n, c, mo[d].nold, a.ncomps,
          mo[d].old2new.data(), a.data[d].data(), mo[d].prods2new.data(), src[d].data(), sd,
          p.src_dims.exists() ? p.src_dims.data() : (I8 const*)nullptr, a.data[sd].data(),
          a.data[other].data(), out.data());
      nw.itags[t].data[d] = out;
    }
  }
}

template <class T>
DArray<T> transfer(Ctx& c, ModOut const& mo, int nc, DArray<T> const& old_data,
    DArray<T> const* prod_data) {
  DArray<T> d(c, mo.nnew * nc);
  LO nprods = prod_data ? mo.nprods : 0;
  OSH_LAUNCH(scatter_data<T>, mo.nold + nprods, c, mo.nold, nc, mo.old2new.data(),
      old_data.data(), mo.prods2new.data(), prod_data ? prod_data->data() : (T const*)nullptr,
      d.data());
  return d;
}

template DArray<LO> transfer(Ctx&, ModOut const&, int, DArray<LO> const&, DArray<LO> const*);
template DArray<I8> transfer(Ctx&, ModOut const&, int, DArray<I8> const&, DArray<I8> const*);
template DArray<Real> transfer(Ctx&, ModOut const&, int, DArray<Real> const&, DArray<Real> const*);

void transfer_elem_tags(Ctx& c, DMesh const& old, DMesh& nw, ModOut const& mo,
    LOs const* prod_src) {
  nw.etags.clear();
  LO nprods = mo.nprods;
  for (auto const& t : old.etags) {
    Reals pd;
    if (prod_src) {
      pd = Reals(c, nprods * t.ncomps);
      OSH_LAUNCH(gather_rows, nprods, c, t.ncomps, prod_src->data(), t.data.data(), pd.data());
    }
    nw.etags.push_back(t.with_data(transfer<Real>(c, mo, t.ncomps, t.data,
        prod_src ? &pd : nullptr)));
  }
}

void transfer_pointwise(Ctx& c, DMesh& old, DMesh& nw, ModOut const& mo, int key_dim,
    LOs const& keys2kds, LOs const& keys2prods, LOs const& prod_verts) {
  if (old.etags.empty()) return;
  int dim = old.dim;
  LO nkeys = keys2kds.size();
  Adj const& up = ask_up(c, old, key_dim, dim);
  LOs const& ev2v = verts_of(c, old, dim);
  LO nprods = mo.nprods;
  int lanes = fit_lanes(nprods, kPointLanes);
  int lshift = lanes_shift(lanes);
  LOs best(c, nprods);
  if (dim == 3)
    OSH_LAUNCH(pointwise_kernel<3>, nprods * lanes, c, lshift, nkeys, keys2kds.data(),
        keys2prods.data(),
        up.a2ab.data(), up.ab2b.data(), ev2v.data(), old.coords.data(), prod_verts.data(),
        nw.coords.data(), best.data());
  else
    OSH_LAUNCH(pointwise_kernel<2>, nprods * lanes, c, lshift, nkeys, keys2kds.data(),
        keys2prods.data(),
        up.a2ab.data(), up.ab2b.data(), ev2v.data(), old.coords.data(), prod_verts.data(),
        nw.coords.data(), best.data());
  transfer_elem_tags(c, old, nw, mo, &best);
}

Bytes find_indset(Ctx& c, DMesh& m, int d, Reals const& quality, Bytes const& cands,
    bool* any_cands, Adj const* edge_elems, Adj const* star, StopWord const* stop) {
  Range range(c, "find_indset");
  LO n = m.nents[d];
  if (d == m.dim) {  // src/Omega_h_indset.cpp:29
    if (any_cands) *any_cands = max_i8(c, cands) > 0;
    return cands;
  }
  Adj const* g = nullptr;
  Adj const* e2c = nullptr;
  LO const* c2e = nullptr;
  if (d == 1) {
    e2c = edge_elems ? edge_elems : &ask_up(c, m, 1, m.dim);
    c2e = ask_down(c, m, m.dim, 1, nullptr).data();
  } else {
    g = star ? star : &ask_star(c, m, d);
  }
  Bytes a(c, n), b(c, n);
  DArray<unsigned long long> dom(c, n);
  int first_lanes = fit_lanes(n, c.tuning.first_lanes);
  return indset_rounds(c, n, cands, a, b, any_cands,
      [&](bool first, I8 const* in, I8* out, IndsetWords w) {
        if (g && first)
          OSH_LAUNCH(indset_iteration<true>, n, c, g->a2ab.data(), g->ab2b.data(),
              quality.data(), in, out, dom.data(), w);
        else if (g)
          OSH_LAUNCH(indset_iteration<false>, n, c, g->a2ab.data(), g->ab2b.data(),
              quality.data(), in, out, dom.data(), w);
        else if (first && m.dim == 3)
          OSH_LAUNCH((indset_first_edges<6>), n * first_lanes, c, first_lanes,
              e2c->a2ab.data(), e2c->ab2b.data(), c2e, quality.data(), in, out, dom.data(), w);
        else if (first)
          OSH_LAUNCH((indset_first_edges<3>), n * first_lanes, c, first_lanes,
              e2c->a2ab.data(), e2c->ab2b.data(), c2e, quality.data(), in, out, dom.data(), w);
        else if (m.dim == 3)
          OSH_LAUNCH(indset_iteration_edges<6>, n, c, e2c->a2ab.data(), e2c->ab2b.data(), c2e,
              quality.data(), in, out, dom.data(), w);
        else
          OSH_LAUNCH(indset_iteration_edges<3>, n, c, e2c->a2ab.data(), e2c->ab2b.data(), c2e,
              quality.data(), in, out, dom.data(), w);
      },
      stop);
}

Bytes mark_down(Ctx& c, DMesh& m, int high, int low, Bytes const& marks) {
  if (high == low) return marks;
  if (!m.up[low][high].exists()) {
    Bytes out = fill_i8(c, m.nents[low], 0);
    LOs const& hl2l = ask_down(c, m, high, low, nullptr);
    OSH_LAUNCH(mark_down_scatter, m.nents[high], c, simplex_degree(high, low), hl2l.data(),
        marks.data(), out.data());
    return out;
  }
  Adj const& l2h = ask_up(c, m, low, high);
  Bytes out(c, m.nents[low]);
  OSH_LAUNCH(mark_down_kernel, m.nents[low], c, l2h.a2ab.data(), l2h.ab2b.data(), marks.data(),
      out.data());
  return out;
}

SliverLayers::SliverLayers(Ctx& c, DMesh& m, int nlayers, Fills& fills)
    : c_(c), m_(m), nlayers_(nlayers) {
  if (m.linked && nlayers > 0 && nlayers <= kCountedLayers)
    counts_ = fills.ints(m.nents[m.dim - 1], 0);
}

Bytes SliverLayers::mark(Real qual_ceil) {
  Ctx& c = c_;
  DMesh& m = m_;
  LO ne = m.nents[m.dim];
  Reals const& q = ask_qualities(c, m);
  Bytes marks(c, ne);
  if (nlayers_ == 0) {
    OSH_LAUNCH(below_kernel, ne, c, q.data(), qual_ceil, marks.data());
    return marks;
  }
  LO const* es2s = m.down[m.dim].data();
  EdgeMarks edges{nullptr, m.class_dim[1].data(), edge_marks_};
  if (edge_marks_) edges.e2e = ask_down(c, m, m.dim, 1, nullptr).data();
  if (counts_.exists()) {
    unsigned* counts = reinterpret_cast<unsigned*>(counts_.data());
    for (int k = 0; k <= nlayers_; ++k) {
      if (m.dim == 3)
        OSH_LAUNCH(sliver_layer<4>, ne, c, k, nlayers_, es2s, q.data(), qual_ceil, counts,
            marks.data(), edges);
      else
        OSH_LAUNCH(sliver_layer<3>, ne, c, k, nlayers_, es2s, q.data(), qual_ceil, counts,
            marks.data(), edges);
    }
    return marks;
  }
  auto const& se = ask_side_elems(c, m);
  // the first layer reads the sliver test itself; later ones push, into
  // buffers cleared eight at a time
  tag_ = c.wait_tag();
  OSH_LAUNCH(dual_max_kernel, ne, c, m.dim + 1, es2s, se.data(), q.data(), qual_ceil,
      marks.data(), c.words + kUnlinkedWord, tag_, c.error_word());
  Bytes next[8];
  for (int i = 1; i < nlayers_; ++i) {
    int b = (i - 1) % 8;
    if (b == 0) {
      Fills fills(c);
      for (int k = 0; k < 8 && i + k < nlayers_; ++k) next[k] = fills.bytes(ne, 0);
      fills.run();
    }
    if (m.dim == 3)
      OSH_LAUNCH(push_layer_kernel<4>, ne, c, es2s, se.data(), marks.data(), next[b].data());
    else
      OSH_LAUNCH(push_layer_kernel<3>, ne, c, es2s, se.data(), marks.data(), next[b].data());
    marks = next[b];
  }
  return marks;
}

void SliverLayers::mark_interior_edges(Real qual_ceil, Bytes& edge_marks) {
  Ctx& c = c_;
  DMesh& m = m_;
  edge_marks_ = edge_marks.data();
  Bytes marks = mark(qual_ceil);
  if (counts_.exists()) return;  // the last layer has marked them
  EdgeMarks edges{ask_down(c, m, m.dim, 1, nullptr).data(), m.class_dim[1].data(), edge_marks_};
  if (m.dim == 3)
    OSH_LAUNCH(mark_interior_edges_kernel<4>, m.nents[3], c, marks.data(), edges);
  else
    OSH_LAUNCH(mark_interior_edges_kernel<3>, m.nents[2], c, marks.data(), edges);
}

void SliverLayers::settle() {
  if (tag_) m_.linked = !c_.word_set(kUnlinkedWord, tag_);
}

void default_options(int dim, AdaptOptions& o) {
  o.min_length_desired = 1.0 / __builtin_sqrt(2.0);
  o.max_length_desired = __builtin_sqrt(2.0);
  o.max_length_allowed = o.max_length_desired * 2.0;
  if (dim == 3) {
    o.min_quality_allowed = 0.20;
    o.min_quality_desired = 0.30;
  } else {
    o.min_quality_allowed = 0.30;
    o.min_quality_desired = 0.40;
  }
  o.nsliver_layers = 4;
  o.verbosity = 2;  // EACH_REBUILD
  o.should_refine = 1;
  o.should_coarsen = 1;
  o.should_swap = 1;
  o.should_coarsen_slivers = 1;
  o.length_histogram_min = 0.0;
  o.length_histogram_max = 3.0;
  o.nlength_histogram_bins = 10;
  o.nquality_histogram_bins = 10;
  o.should_prevent_coarsen_flip = 0;
  o.precision = 0;
}

}  // namespace osh
