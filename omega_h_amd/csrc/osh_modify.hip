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
#include "osh_math.hpp"
#include "osh_passes.hpp"

namespace osh {

namespace {

// the same entities of dimension > key dimension: those with no key among
// their lower entities, each counting one new entity; each key also receives
// the lowest index among the entities above it, which is the first entry of
// its row of the upward adjacency (rows are sorted by index), without
// building that adjacency
// the dimensions above the keys in one launch: job w owns the threads
// [start[w], start[w + 1])
struct SameUpJobs {
  LO start[4];
  int deg[3];
  LO const* hl2l[3];
  I8* same[3];
  LO* counts[3];
  LO* first_up[3];
  int n;
};

__global__ void mark_same_up_kernel(LO nt, I8 const* low_marks, SameUpJobs j) {
  LO t = thread_index();
  if (t >= nt) return;
  int w = 0;
  while (w + 1 < j.n && t >= j.start[w + 1]) ++w;
  LO h = t - j.start[w];
  int deg = j.deg[w];
  LO const* hl2l = j.hl2l[w];
  I8 r = 1;
  for (int k = 0; k < deg; ++k) {
    LO l = hl2l[h * deg + k];
    if (low_marks[l]) {
      r = 0;
      atomicMin(&j.first_up[w][l], h);
    }
  }
  j.same[w][h] = r;
  j.counts[w][h] = r;
}

// One sweep over the key-dimension entities starts the plans of every
// dimension of a pass: no key marked, no entity above found yet, and (when
// the key dimension itself is rebuilt) every entity the same, counting one.
struct KeyDimInit {
  I8* key_marks;
  LO* first_up[4];  // per dimension above the keys (null elsewhere)
  I8* same;         // when the key dimension is rebuilt
  LO* counts;
  // with a key mask, the keys are marked in the same sweep: no longer the
  // same, each counting its products
  I8 const* key_mask;
  LO const* key_prod_counts;
};

__global__ void init_key_dim(LO n, KeyDimInit a) {
  LO i = thread_index();
  if (i >= n) return;
  if (a.key_marks) a.key_marks[i] = 0;
  for (int d = 0; d < 4; ++d)
    if (a.first_up[d]) a.first_up[d][i] = 0x7fffffff;
  if (a.same) {
    bool key = a.key_mask && a.key_mask[i];
    a.same[i] = key ? 0 : 1;
    a.counts[i] = key ? a.key_prod_counts[i] : 1;
  }
}

// the keys: marked; when the key dimension is rebuilt, a key is its own
// representative (get_mods2reps, src/Omega_h_modify.cpp:20-45), is no longer
// the same and counts its products (get_rep_counts, :47-70)
__global__ void mark_keys(LO nkeys, LO const* keys2kds, LO const* keys2prods, I8* key_marks,
    I8* same, LO* counts, LO* reps) {
  LO k = thread_index();
  if (k >= nkeys) return;
  LO kd = keys2kds[k];
  if (key_marks) key_marks[kd] = 1;
  if (same) {
    same[kd] = 0;
    counts[kd] = keys2prods[k + 1] - keys2prods[k];
    reps[k] = kd;
  }
}

// representatives of the keys for up to three dimensions in one launch: the
// lowest entity above the key (first_up) or the key's first lower entity
// (down); the representative counts the key's products
struct RepsJob {
  LO const* first_up[3];
  LO const* down[3];
  int deg[3];
  LO const* keys2prods[3];
  LO* reps[3];
  LO* counts[3];
};

__global__ void reps_kernel(LO nt, LO nkeys, LO const* keys2kds, RepsJob j, int* error) {
  LO t = thread_index();
  if (t >= nt) return;
  int w = t / nkeys;
  LO k = t % nkeys;
  LO kd = keys2kds[k];
  LO r;
  if (j.first_up[w]) {
    r = j.first_up[w][kd];
    if (r == 0x7fffffff) {  // keeps every index in range until the host sees it
      r = 0;
      *error = kKeyWithoutUp;
    }
  } else {
    r = j.down[w][kd * j.deg[w]];
  }
  j.reps[w][k] = r;
  atomicAdd(&j.counts[w][r], j.keys2prods[w][k + 1] - j.keys2prods[w][k]);
}

// the same starts with the keys given as a mask over the key dimension and
// their product counts per key-dimension entity: a key of the rebuilt key
// dimension is no longer the same and counts its products; for the
// dimensions above, each key's representative (kept per key-dimension
// entity) counts the key's products
struct MaskedReps {
  LO const* first_up[3];
  LO const* prod_counts[3];
  LO* rep_of[3];
  LO* counts[3];
};

__global__ void reps_masked(LO nt, LO nkd, I8 const* key_mask, MaskedReps j, int* error) {
  LO t = thread_index();
  if (t >= nt) return;
  int w = t / nkd;
  LO kd = t % nkd;
  if (!key_mask[kd]) return;
  LO r = j.first_up[w][kd];
  if (r == 0x7fffffff) {  // keeps every index in range until the host sees it
    r = 0;
    *error = kKeyWithoutUp;
  }
  j.rep_of[w][kd] = r;
  atomicAdd(&j.counts[w][r], j.prod_counts[w][kd]);
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

__global__ void scatter_index(LO n, LO const* a2b, LO* b2a) {
  LO i = thread_index();
  if (i < n) b2a[a2b[i]] = i;
}

__global__ void rep2md_order_kernel(LO nreps, LO const* a2ab, LO const* ab2b, I8 const* codes,
    LO const* md2mod, LO const* keys2prods, LO* order) {
  LO rep = thread_index();
  if (rep >= nreps) return;
  LO offset = 0;
  for (LO j = a2ab[rep]; j < a2ab[rep + 1]; ++j) {
    LO md = ab2b[j];
    LO mod = md2mod[md];
    if (mod >= 0 && code_which_down(codes[j]) == 0) {
      order[md] = offset;
      offset += keys2prods[mod + 1] - keys2prods[mod];
    }
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

__global__ void __launch_bounds__(kBlock) place_products_kernel(LO nt, LO nkeys, PlaceJobs j) {
  LO t = thread_index();
  if (t >= nt) return;
  LO per = nkeys * kProdLanes;
  PlaceDim const& a = j.d[t / per];
  LO k = (t % per) / kProdLanes;
  int lane = t % kProdLanes;
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

// one round of indset::find (src/Omega_h_indset.cpp:5-35).  In the first
// round the states come straight from the candidate marks (2 for a
// candidate, 0 otherwise), so no node is in the set yet.
template <bool FIRST>
__device__ __forceinline__ I8 indset_state(I8 const* old_state, LO x) {
  I8 s = old_state[x];
  return FIRST ? I8(s ? 2 : 0) : s;
}

// A node joins the set once every neighbor that beats it (higher quality,
// or the same quality and a higher index) is out, and leaves once one of
// them is in: a neighbor it beats can be in only after the node is out, so
// this is the round above restated over the beating neighbors alone.  The
// first round records, per candidate, which row positions hold candidates
// that beat it (bits of `dom`); later rounds read the states at those
// positions only, not the qualities.  A row longer than 64 positions is
// read whole every round.
constexpr int kDomBits = 64;

// Each batch of rounds ends with a wait for two words: kUndecidedWord, set by
// the last round's nodes that stay undecided, and kCandWord, set by the first
// round's candidates, so that no reduction over the states is needed.
constexpr int kUndecidedWord = 0;
constexpr int kCandWord = 1;

// one lane a wave stores, and only where the word does not hold the tag yet
__device__ __forceinline__ void tell(bool is, unsigned* word, unsigned tag) {
  unsigned long long b = __ballot(is);
  if (b == 0ull || int(threadIdx.x & 63) != __ffsll(static_cast<long long>(b)) - 1) return;
  if (__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != tag)
    __hip_atomic_store(word, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct IndsetWords {
  unsigned* words;
  unsigned cand_tag;  // 0: not the first round
  unsigned last_tag;  // 0: not the last round of its batch
};

__device__ __forceinline__ void tell_round(I8 before, I8 after, IndsetWords w) {
  if (w.cand_tag) tell(before == 2, w.words + kCandWord, w.cand_tag);
  if (w.last_tag) tell(after == 2, w.words + kUndecidedWord, w.last_tag);
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
// input is `in`, or, when `q` is given, the sliver test q < ceil.
template <int NSPE>
__device__ __forceinline__ I8 dual_max_at(LO e, LO const* es2s,
    unsigned long long const* side_elems, I8 const* in, Real const* q, Real ceil, int* error) {
  I8 r = -128;
#pragma unroll
  for (int j = 0; j < NSPE; ++j) {
    unsigned long long w = side_elems[es2s[e * NSPE + j]];
    unsigned count = unsigned(w >> 32);
    if (count == 2) {
      LO o = LO(unsigned(w)) - e;
      I8 x = q ? I8(q[o] < ceil) : in[o];
      r = (r < x) ? x : r;
    } else if (count > 2) {
      *error = kNonManifoldSide;
    }
  }
  return r;
}

__global__ void dual_max_kernel(LO n, int nspe, LO const* es2s,
    unsigned long long const* side_elems, I8 const* in, Real const* q, Real ceil, I8* out,
    int* error) {
  LO e = thread_index();
  if (e >= n) return;
  out[e] = nspe == 4 ? dual_max_at<4>(e, es2s, side_elems, in, q, ceil, error)
                     : dual_max_at<3>(e, es2s, side_elems, in, q, ceil, error);
}

__global__ void degrees_kernel(LO n, LO const* a2ab, LO const* rows, LO* out) {
  LO i = thread_index();
  if (i >= n) return;
  LO r = rows ? rows[i] : i;
  out[i] = a2ab[r + 1] - a2ab[r];
}

}  // namespace

LOs degrees_of(Ctx& c, LOs const& a2ab, LOs const& rows) {
  LO n = rows.exists() ? rows.size() : a2ab.size() - 1;
  LOs out(c, n);
  OSH_LAUNCH(degrees_kernel, n, c, a2ab.data(), rows.exists() ? rows.data() : (LO const*)nullptr,
      out.data());
  return out;
}

void modify_plans(Ctx& c, DMesh& old, int key_dim, int d0, int d1, LOs const& keys2kds,
    LOs const* keys2prods, ModPlan* plans) {
  LO nkeys = keys2kds.size();
  LO nkd = old.nents[key_dim];
  KeyDimInit init{};
  Bytes key_marks;
  LOs first_up[4];
  bool above = false;
  for (int d = d0; d <= d1; ++d) {
    ModPlan& plan = plans[d - d0];
    plan.ent_dim = d;
    plan.key_dim = key_dim;
    plan.nold = old.nents[d];
    plan.reps = LOs(c, nkeys);
    // same entities: those not adjacent to a key (collect_same); without a
    // `same` array every old entity is the same
    if (d >= key_dim) {
      plan.same = Bytes(c, plan.nold);
      plan.counts = LOs(c, plan.nold);
    }
    if (d > key_dim) {
      first_up[d] = LOs(c, nkd);
      init.first_up[d] = first_up[d].data();
      above = true;
    }
    if (d == key_dim) {
      init.same = plan.same.data();
      init.counts = plan.counts.data();
    }
  }
  if (above) {
    key_marks = Bytes(c, nkd);
    init.key_marks = key_marks.data();
  }
  if (above || init.same) {
    OSH_LAUNCH(init_key_dim, nkd, c, init);
    ModPlan* kp = (key_dim >= d0 && key_dim <= d1) ? &plans[key_dim - d0] : nullptr;
    OSH_LAUNCH(mark_keys, nkeys, c, keys2kds.data(),
        kp ? keys2prods[key_dim].data() : (LO const*)nullptr, init.key_marks,
        kp ? kp->same.data() : (I8*)nullptr, kp ? kp->counts.data() : (LO*)nullptr,
        kp ? kp->reps.data() : (LO*)nullptr);
  }
  RepsJob jobs{};
  int njobs = 0;
  SameUpJobs up{};
  for (int d = d0; d <= d1; ++d) {
    ModPlan& plan = plans[d - d0];
    if (d > key_dim) {
      up.deg[up.n] = simplex_degree(d, key_dim);
      up.hl2l[up.n] = ask_down(c, old, d, key_dim, nullptr).data();
      up.same[up.n] = plan.same.data();
      up.counts[up.n] = plan.counts.data();
      up.first_up[up.n] = first_up[d].data();
      up.start[up.n + 1] = up.start[up.n] + plan.nold;
      ++up.n;
      jobs.first_up[njobs] = first_up[d].data();
    } else if (d < key_dim) {
      plan.counts = fill_lo(c, plan.nold, 1);
      jobs.deg[njobs] = simplex_degree(key_dim, d);
      jobs.down[njobs] = ask_down(c, old, key_dim, d, nullptr).data();
    } else {
      continue;
    }
    jobs.keys2prods[njobs] = keys2prods[d].data();
    jobs.reps[njobs] = plan.reps.data();
    jobs.counts[njobs] = plan.counts.data();
    ++njobs;
  }
  OSH_CHECK(njobs <= 3, "modify_plans: too many dimensions");
  if (up.n) OSH_LAUNCH(mark_same_up_kernel, up.start[up.n], c, key_marks.data(), up);
  if (njobs) OSH_LAUNCH(reps_kernel, njobs * nkeys, c, nkeys, keys2kds.data(), jobs,
      c.error_word());
}

void modify_plans_masked(Ctx& c, DMesh& old, int key_dim, int d1, Bytes const& key_mask,
    LO const* const* prod_counts, ModPlan* plans, LOs* rep_of) {
  LO nkd = old.nents[key_dim];
  KeyDimInit init{};
  LOs first_up[4];
  for (int d = key_dim; d <= d1; ++d) {
    ModPlan& plan = plans[d - key_dim];
    plan.ent_dim = d;
    plan.key_dim = key_dim;
    plan.nold = old.nents[d];
    plan.same = Bytes(c, plan.nold);
    plan.counts = LOs(c, plan.nold);
    if (d > key_dim) {
      first_up[d] = LOs(c, nkd);
      init.first_up[d] = first_up[d].data();
      rep_of[d] = LOs(c, nkd);
    }
  }
  init.same = plans[0].same.data();
  init.counts = plans[0].counts.data();
  init.key_mask = key_mask.data();
  init.key_prod_counts = prod_counts[key_dim];
  OSH_LAUNCH(init_key_dim, nkd, c, init);
  MaskedReps j{};
  int nj = 0;
  SameUpJobs up{};
  for (int d = key_dim + 1; d <= d1; ++d) {
    ModPlan& plan = plans[d - key_dim];
    up.deg[up.n] = simplex_degree(d, key_dim);
    up.hl2l[up.n] = ask_down(c, old, d, key_dim, nullptr).data();
    up.same[up.n] = plan.same.data();
    up.counts[up.n] = plan.counts.data();
    up.first_up[up.n] = first_up[d].data();
    up.start[up.n + 1] = up.start[up.n] + plan.nold;
    ++up.n;
    j.first_up[nj] = first_up[d].data();
    j.prod_counts[nj] = prod_counts[d];
    j.rep_of[nj] = rep_of[d].data();
    j.counts[nj] = plan.counts.data();
    ++nj;
  }
  OSH_CHECK(nj <= 3, "modify_plans_masked: too many dimensions");
  if (up.n) OSH_LAUNCH(mark_same_up_kernel, up.start[up.n], c, key_mask.data(), up);
  if (nj) OSH_LAUNCH(reps_masked, nj * nkd, c, nkd, key_mask.data(), j, c.error_word());
}

int modify_scan_jobs(Ctx& c, ModPlan* plans, int nplans, ScanJob* jobs, int first_slot) {
  for (int i = 0; i < nplans; ++i) {
    ModPlan& p = plans[i];
    p.offsets = LOs(c, p.nold + 1);
    jobs[i] = {p.counts.data(), kScanLO, p.nold, p.offsets.data(),
        slot_ptr<LO>(c, first_slot + i)};
  }
  return nplans;
}

void modify_scan_totals(Ctx& c, ModPlan* plans, int nplans, int first_slot) {
  for (int i = 0; i < nplans; ++i) plans[i].nnew = read_slot<LO>(c, first_slot + i);
}

void modify_scan(Ctx& c, ModPlan* plans, int nplans) {
  OSH_CHECK(nplans >= 1 && nplans <= 4, "modify_scan: too many dimensions");
  ScanJob jobs[kMaxScanJobs];
  int njobs = modify_scan_jobs(c, plans, nplans, jobs, 1);
  offset_scans(c, jobs, njobs);
  c.wait();
  modify_scan_totals(c, plans, nplans, 1);
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
    I8* new_edges_valid) {
  LO nkeys = keys2kds.size();
  PlaceJobs j{};
  j.keys2kds = keys2kds.data();
  LOs src[4];
  LOs order;
  for (int d = d0; d <= d1; ++d) {
    ModPlan const& plan = plans[d - plan0];
    Products const& p = prods[d];
    PlaceDim& a = j.d[d - d0];
    mo[d].nprods = p.n;
    mo[d].prods2new = LOs(c, p.n);
    if (plan.key_dim > d) {
      OSH_CHECK(!order.exists(), "one dimension below the keys");
      LO nkd = old.nents[plan.key_dim];
      order = fill_lo(c, nkd, -1);
      LOs md2mod = fill_lo(c, nkd, -1);
      OSH_LAUNCH(scatter_index, nkeys, c, keys2kds.data(), md2mod.data());
      Adj const& up = ask_up(c, old, d, plan.key_dim);
      OSH_LAUNCH(rep2md_order_kernel, plan.nold, c, up.a2ab.data(), up.ab2b.data(),
          up.codes.data(), md2mod.data(), p.keys2prods.data(), order.data());
      a.order = order.data();
    }
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
  OSH_CHECK(std::int64_t(nkeys) * kProdLanes * nd <= std::int64_t(0x7fffffff),
      "place_products: too many keys");
  OSH_LAUNCH(place_products_kernel, nkeys * kProdLanes * nd, c, nkeys, j);
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
    bool* any_cands, Adj const* edge_elems, Adj const* star) {
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
  // rounds leave decided nodes as they are and take no node from the set, so
  // extra rounds after convergence change nothing: run two rounds before each
  // of the first four checks, then 4, 8 and 16 (long chains of decreasing
  // quality, as on the first coarsening passes of a large smooth mesh, take
  // some 200 rounds and would otherwise spend a wait every two)
  int first_lanes = fit_lanes(n, c.tuning.first_lanes);
  for (LO round = 0;;) {
    OSH_CHECK(round <= n + 1, "independent set does not converge");
    int batch = round < 8 ? 2 : (round < 16 ? 4 : (round < 32 ? 8 : 16));
    unsigned tag = c.wait_tag();
    for (int k = 0; k < batch; ++k, ++round) {
      bool first = round == 0;
      IndsetWords w{c.words, first ? tag : 0u, k == batch - 1 ? tag : 0u};
      I8 const* in = first ? cands.data() : a.data();
      if (g && first)
        OSH_LAUNCH(indset_iteration<true>, n, c, g->a2ab.data(), g->ab2b.data(),
            quality.data(), in, b.data(), dom.data(), w);
      else if (g)
        OSH_LAUNCH(indset_iteration<false>, n, c, g->a2ab.data(), g->ab2b.data(),
            quality.data(), in, b.data(), dom.data(), w);
      else if (first && m.dim == 3)
        OSH_LAUNCH((indset_first_edges<6>), n * first_lanes, c, first_lanes, e2c->a2ab.data(),
            e2c->ab2b.data(), c2e, quality.data(), in, b.data(), dom.data(), w);
      else if (first)
        OSH_LAUNCH((indset_first_edges<3>), n * first_lanes, c, first_lanes, e2c->a2ab.data(),
            e2c->ab2b.data(), c2e, quality.data(), in, b.data(), dom.data(), w);
      else if (m.dim == 3)
        OSH_LAUNCH(indset_iteration_edges<6>, n, c, e2c->a2ab.data(), e2c->ab2b.data(), c2e,
            quality.data(), in, b.data(), dom.data(), w);
      else
        OSH_LAUNCH(indset_iteration_edges<3>, n, c, e2c->a2ab.data(), e2c->ab2b.data(), c2e,
            quality.data(), in, b.data(), dom.data(), w);
      std::swap(a, b);
    }
    c.wait();
    if (any_cands && round == 2) *any_cands = c.word_set(kCandWord, tag);
    if (!c.word_set(kUndecidedWord, tag)) break;
  }
  return a;
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

Bytes mark_sliver_layers(Ctx& c, DMesh& m, Real qual_ceil, int nlayers) {
  LO ne = m.nents[m.dim];
  Reals const& q = ask_qualities(c, m);
  Bytes marks;
  if (nlayers == 0) {
    marks = Bytes(c, ne);
    OSH_LAUNCH(below_kernel, ne, c, q.data(), qual_ceil, marks.data());
    return marks;
  }
  auto const& se = ask_side_elems(c, m);
  // the first layer reads the sliver test itself
  for (int i = 0; i < nlayers; ++i) {
    Bytes next(c, ne);
    OSH_LAUNCH(dual_max_kernel, ne, c, m.dim + 1, m.down[m.dim].data(), se.data(), marks.data(),
        i == 0 ? q.data() : (Real const*)nullptr, qual_ceil, next.data(), c.error_word());
    marks = next;
  }
  return marks;
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
