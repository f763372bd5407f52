// Adjacency derivation on the device.
//
//   transit                 src/Omega_h_adj.cpp:443-510
//   invert_adj              src/Omega_h_adj.cpp:178-263 (count, scan, fill,
//                           then each row ordered by high index so the result
//                           does not depend on atomic order)
//   reflect_down / find_matches src/Omega_h_adj.cpp:297-441
//   verts_across_edges, edges_across_tris/tets, add_edges
//                           src/Omega_h_adj.cpp:512-589, src/Omega_h_graph.cpp:14-40
//   side_elems (the two elements of each side, for elements_across_sides)
//                           src/Omega_h_adj.cpp:591-657
//   find_unique             src/Omega_h_adj.cpp:55-153
#include "osh_mesh.hpp"
#include "osh_passes.hpp"

namespace osh {

int simplex_degree(int from_dim, int to_dim) {
  static int const deg[4][4] = {{1, -1, -1, -1}, {2, 1, -1, -1}, {3, 3, 1, -1}, {4, 6, 4, 1}};
  return deg[from_dim][to_dim];
}

void DMesh::clear_caches() {
  linked = false;
  for (int d = 0; d < 4; ++d) {
    verts[d] = LOs();
    for (int e = 0; e < 4; ++e) up[d][e] = Adj();
  }
  star[0] = star[1] = Adj();
  side_elems = DArray<unsigned long long>();
  dual = Adj();
  size = Reals();
  t2e = LOs();
  t2e_codes = Bytes();
}

namespace {

__device__ __forceinline__ int rotate_index(int n, int index, int rotation) {
  return (index + rotation) % n;
}
__device__ __forceinline__ int invert_rotation(int n, int rotation) {
  return (n - rotation) % n;
}
__device__ __forceinline__ I8 invert_alignment(int n, I8 code) {
  if (code_is_flipped(code)) return code;
  return make_code(0, invert_rotation(n, code_rotation(code)), 0);
}
__device__ __forceinline__ int align_vert_index(int n, int index, I8 code) {
  int r = rotate_index(n, index, code_rotation(code));
  return code_is_flipped(code) ? (r == 0 ? 0 : (1 + ((n - 1) - 1 - (r - 1)))) : r;
}
__device__ __forceinline__ int align_edge_index(int n, int index, I8 code) {
  int r = rotate_index(n, index, code_rotation(code));
  return code_is_flipped(code) ? (n - 1 - r) : r;
}

// first entry of simplex_up_template, src/Omega_h_simplex.hpp:91-229
__device__ __forceinline__ void up_template0(int elem_dim, int bdry_dim, int which,
    int& up, int& which_down, int& flipped) {
  if (elem_dim == 3 && bdry_dim == 0) {
    up = (which == 3) ? 5 : which;
    which_down = (which == 3) ? 1 : 0;
    flipped = 0;
  } else if (elem_dim == 3 && bdry_dim == 1) {
    int const t[6][2] = {{0, 2}, {0, 1}, {0, 0}, {1, 2}, {2, 2}, {3, 2}};
    up = t[which][0];
    which_down = t[which][1];
    flipped = 1;
  } else {
    up = which;
    which_down = 0;
    flipped = 0;
  }
}

// one thread per (high entity, local low entity), so that the gathers of a
// high entity's lows run side by side
template <int HIGH, int LOW>
__global__ void transit_kernel(LO nuses, LO const* hm2m, I8 const* m2hm_codes,
    LO const* ml2l, I8 const* ml_codes, LO* hl2l, I8* codes) {
  LO t = thread_index();
  if (t >= nuses) return;
  constexpr int MID = LOW + 1;
  constexpr int nmph = (HIGH == 3) ? (MID == 2 ? 4 : 6) : 3;
  constexpr int nlpm = MID + 1;
  constexpr int nlph = (HIGH == 3) ? (LOW == 0 ? 4 : 6) : 3;
  LO h = t / nlph;
  int hl = t % nlph;
  {
    int hm, hml, canon_flipped;
    up_template0(HIGH, LOW, hl, hm, hml, canon_flipped);
    LO m = hm2m[h * nmph + hm];
    I8 hm2m_code = invert_alignment(nlpm, m2hm_codes[h * nmph + hm]);
    int ml = (LOW == 0) ? align_vert_index(nlpm, hml, hm2m_code)
                        : align_edge_index(nlpm, hml, hm2m_code);
    hl2l[h * nlph + hl] = ml2l[m * nlpm + ml];
    if (LOW == 1) {
      int region_face_flipped = code_is_flipped(hm2m_code);
      int face_edge_flipped = (code_rotation(ml_codes[m * nlpm + ml]) == 1);
      codes[h * nlph + hl] =
          make_code(0, region_face_flipped ^ face_edge_flipped ^ canon_flipped, 0);
    }
  }
}

// invert_adj in three sweeps over the uses hl = high * deg + which:
//   count_lows: per-low use counts by atomics; each use keeps its slot
//   fill_uses:  ab2hl[a2ab[l] + slot] = hl (slots are in atomic order)
//   rank_uses:  each use counts the uses of its row with a smaller hl and
//               writes itself at that rank, which sorts every row by high
//               index (sort_by_high_index, src/Omega_h_adj.cpp:178-200)
//               and forms the codes of separate_upward_with_codes (:202-217)
// With `marks`, only the rows of marked lows are built (the rest are empty).
// Without `sorted`, rows keep the order of the atomics, for uses that do not
// depend on it (one sweep less).  Several maps are inverted by the same
// launches: job w owns the workgroups [first[w], first[w + 1]).
struct UseJob {
  LO nhl;
  LO const* hl2l;
  I8 const* marks;
  LO* counts;
  LO* slot;
  LO const* a2ab;
  int deg;
  I8 const* down_codes;
  int sorted;
  LO* ab2hl;
  LO* ab2b;
  I8* codes;
};
constexpr int kMaxUseJobs = 3;
struct UseJobs {
  int n;
  unsigned first[kMaxUseJobs + 1];
  UseJob d[kMaxUseJobs];
};

__device__ __forceinline__ int use_job(UseJobs const& j, LO* i) {
  int w = 0;
  while (w + 1 < j.n && blockIdx.x >= j.first[w + 1]) ++w;
  *i = LO(blockIdx.x - j.first[w]) * kBlock + LO(threadIdx.x);
  return w;
}

__device__ __forceinline__ I8 use_code(UseJob const& a, LO hl) {
  int which_down = hl % a.deg;
  return a.down_codes ? make_code(code_is_flipped(a.down_codes[hl]),
                            code_rotation(a.down_codes[hl]), which_down)
                      : make_code(0, 0, which_down);
}

// a workgroup's uses of one low are counted in LDS first, so that the low's
// counter takes one atomic a workgroup: its 64 tets share their vertices several
// times over (18 us a launch on the 64^3 workload against 31 with an atomic a
// use, 5.2 against 7.2 at 10,000 tets).  Slots come in no particular order, which
// the sweeps below do not look at.
__global__ void __launch_bounds__(kBlock) count_lows(UseJobs j) {
  constexpr unsigned kTable = 2 * kBlock;
  constexpr int kTableBits = 9;
  static_assert(kTable == 1u << kTableBits, "a place is the product's high bits");
  __shared__ LO keys[kTable];
  __shared__ LO counts[kTable];
  for (unsigned k = threadIdx.x; k < kTable; k += kBlock) {
    keys[k] = -1;
    counts[k] = 0;
  }
  LO i;
  UseJob const& a = j.d[use_job(j, &i)];
  LO l = i < a.nhl ? a.hl2l[i] : -1;
  if (l >= 0 && a.marks && !a.marks[l]) l = -1;
  __syncthreads();
  unsigned h = 0;
  LO rank = 0;
  if (l >= 0) {
    // the high bits: the low ones give lows a multiple of 512 apart, as on a grid
    // walked across its numbering, the same place (250 us a launch for 2 M
    // triangles of a 512-wide grid, 84 with the high ones)
    h = (unsigned(l) * 2654435761u) >> (32 - kTableBits);
    // at most kBlock lows in twice as many places
    for (;; h = (h + 1) % kTable) {
      LO had = atomicCAS(&keys[h], -1, l);
      if (had == -1 || had == l) break;
    }
    rank = atomicAdd(&counts[h], 1);
  }
  __syncthreads();
  for (unsigned k = threadIdx.x; k < kTable; k += kBlock)
    if (keys[k] >= 0) counts[k] = atomicAdd(&a.counts[keys[k]], counts[k]);
  __syncthreads();
  if (l >= 0) a.slot[i] = counts[h] + rank;
}

__global__ void __launch_bounds__(kBlock) fill_uses(UseJobs j) {
  LO hl;
  UseJob const& a = j.d[use_job(j, &hl)];
  if (hl >= a.nhl) return;
  LO l = a.hl2l[hl];
  if (a.marks && !a.marks[l]) return;
  LO pos = a.a2ab[l] + a.slot[hl];
  if (a.sorted) {
    a.ab2hl[pos] = hl;
  } else {
    a.ab2b[pos] = hl / a.deg;
    a.codes[pos] = use_code(a, hl);
  }
}

__global__ void __launch_bounds__(kBlock) rank_uses(UseJobs j) {
  LO hl;
  UseJob const& a = j.d[use_job(j, &hl)];
  if (hl >= a.nhl) return;
  LO l = a.hl2l[hl];
  if (a.marks && !a.marks[l]) return;
  LO b = a.a2ab[l], e = a.a2ab[l + 1];
  LO rank = 0;
  LO k = b;
  for (; k + 4 <= e; k += 4) {
    LO u[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i] = a.ab2hl[k + i];
#pragma unroll
    for (int i = 0; i < 4; ++i) rank += (u[i] < hl);
  }
  for (; k < e; ++k) rank += (a.ab2hl[k] < hl);
  a.ab2b[b + rank] = hl / a.deg;
  a.codes[b + rank] = use_code(a, hl);
}

struct Invert {
  LO nhigh;
  int deg;
  LO nlow;
  LOs hl2l;
  Bytes const* down_codes;
  Bytes const* marks;
  bool sorted;
};

void invert_adjs(Ctx& c, int n, Invert const* in, Adj* out, LOs const* zeros = nullptr) {
  OSH_CHECK(n >= 1 && n <= kMaxUseJobs, "invert_adjs: too many maps");
  UseJobs j{};
  LOs slot[kMaxUseJobs], ab2hl[kMaxUseJobs];
  ScanJob scans[kMaxUseJobs];
  LOs counts = zeros ? *zeros : LOs();
  if (!zeros) {
    LO total = 0;
    for (int w = 0; w < n; ++w) total += in[w].nlow;
    counts = fill_lo(c, total, 0);
  }
  LO* count = counts.data();
  unsigned blocks = 0;
  for (int w = 0; w < n; ++w) {
    LO nhl = in[w].nhigh * in[w].deg;
    slot[w] = LOs(c, nhl);
    out[w].a2ab = LOs(c, in[w].nlow + 1);
    // with marks the rows hold at most nhl uses; the size stays an upper bound
    out[w].ab2b = LOs(c, nhl);
    out[w].codes = Bytes(c, nhl);
    if (in[w].sorted) ab2hl[w] = LOs(c, nhl);
    j.d[w] = UseJob{nhl, in[w].hl2l.data(), in[w].marks ? in[w].marks->data() : nullptr,
        count, slot[w].data(), out[w].a2ab.data(), in[w].deg,
        in[w].down_codes ? in[w].down_codes->data() : nullptr, in[w].sorted ? 1 : 0,
        in[w].sorted ? ab2hl[w].data() : nullptr, out[w].ab2b.data(), out[w].codes.data()};
    scans[w] = {count, kScanLO, in[w].nlow, out[w].a2ab.data(), nullptr};
    count += in[w].nlow;
    j.first[w] = blocks;
    blocks += nblocks(nhl);
    j.first[w + 1] = blocks;
  }
  j.n = n;
  auto launch = [&](auto kernel, UseJobs const& jobs, unsigned nb) {
    if (nb == 0) return;
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(kBlock), 0, c.stream, jobs);
    OSH_HIP(hipGetLastError());
  };
  launch(count_lows, j, blocks);
  offset_scans(c, scans, n);
  launch(fill_uses, j, blocks);
  UseJobs s{};
  blocks = 0;
  for (int w = 0; w < n; ++w) {
    if (!in[w].sorted) continue;
    s.d[s.n] = j.d[w];
    s.first[s.n++] = blocks;
    blocks += nblocks(j.d[w].nhl);
    s.first[s.n] = blocks;
  }
  launch(rank_uses, s, blocks);
}

Adj invert_adj(Ctx& c, LO nhigh, int deg, LO nlow, LOs const& hl2l, Bytes const* down_codes) {
  Invert in{nhigh, deg, nlow, hl2l, down_codes, nullptr, true};
  Adj out;
  invert_adjs(c, 1, &in, &out);
  return out;
}

// reflect_down: each existing lower entity is listed once, in the row of its
// smallest vertex, and rows are built only for vertices that are the
// smallest vertex of some use.  A use's match has the same vertex set, so it
// sits in the row of the use's smallest vertex; the match is unique, hence it
// is the entity the walk over the full vertex -> lower-entity adjacency finds
// (find_matches, src/Omega_h_adj.cpp:297-422).
template <int NV>
__device__ __forceinline__ LO min_vertex(LO const* v) {
  LO m = v[0];
#pragma unroll
  for (int k = 1; k < NV; ++k) m = (v[k] < m) ? v[k] : m;
  return m;
}

// The four sweeps below take the products of faces and of tets together (a
// job each, owning the workgroups [first[w], first[w + 1])), since neither
// needs the other's result: half the launches, which for the small product
// lists of late passes are the cost.
struct SideDim {
  LO nuses;
  LO const* pverts;
  LO const* prods2new;  // null: products keep their numbers
  LO nl;                // the lower entities and their vertices
  LO const* lv2v;
  LO* counts;
  LO* slot;
  LO const* a2ab;
  int4* rows;
  LO* out;
  I8* codes;
};

struct SideJobs {
  int n;
  int high[2];
  unsigned first[3];
  SideDim d[2];
};

__device__ __forceinline__ int side_job(SideJobs const& j) {
  return (j.n > 1 && blockIdx.x >= j.first[1]) ? 1 : 0;
}
__device__ __forceinline__ LO job_thread(SideJobs const& j, int w) {
  return LO(blockIdx.x - j.first[w]) * kBlock + LO(threadIdx.x);
}

// counts[v] = 1 marks v; a marked row's final slot stays unused
template <int HIGH>
__device__ __forceinline__ void mark_use_min_vert(LO u, SideDim const& a) {
  if (u >= a.nuses) return;
  constexpr int LOW = HIGH - 1;
  LO h = u / (HIGH + 1);
  int which = u % (HIGH + 1);
  LO av[3];
#pragma unroll
  for (int k = 0; k < LOW + 1; ++k)
    av[k] = a.pverts[h * (HIGH + 1) + down_template(HIGH, LOW, which, k)];
  a.counts[min_vertex<LOW + 1>(av)] = 1;
}

__global__ void mark_use_min_verts(SideJobs j) {
  int w = side_job(j);
  if (j.high[w] == 2)
    mark_use_min_vert<2>(job_thread(j, w), j.d[w]);
  else
    mark_use_min_vert<3>(job_thread(j, w), j.d[w]);
}

template <int NVL>
__device__ __forceinline__ void count_min_row(LO l, SideDim const& a) {
  if (l >= a.nl) return;
  LO vm = min_vertex<NVL>(a.lv2v + std::size_t(l) * NVL);
  // unmarked counts stay 0 throughout this kernel, marked ones are >= 1
  a.slot[l] = a.counts[vm] ? atomicAdd(&a.counts[vm], 1) - 1 : -1;
}

__global__ void count_min_rows(SideJobs j) {
  int w = side_job(j);
  if (j.high[w] == 2)
    count_min_row<2>(job_thread(j, w), j.d[w]);
  else
    count_min_row<3>(job_thread(j, w), j.d[w]);
}

// a row entry is {entity, its vertices}, so the match reads no other array
template <int NVL>
__device__ __forceinline__ void fill_min_row(LO l, SideDim const& a) {
  if (l >= a.nl) return;
  LO s = a.slot[l];
  if (s < 0) return;
  LO v[3] = {0, 0, 0};
#pragma unroll
  for (int k = 0; k < NVL; ++k) v[k] = a.lv2v[std::size_t(l) * NVL + k];
  a.rows[a.a2ab[min_vertex<NVL>(v)] + s] = make_int4(l, v[0], v[1], v[2]);
}

__global__ void fill_min_rows(SideJobs j) {
  int w = side_job(j);
  if (j.high[w] == 2)
    fill_min_row<2>(job_thread(j, w), j.d[w]);
  else
    fill_min_row<3>(job_thread(j, w), j.d[w]);
}

// kMatchLanes threads per use share its row; the lane that finds the match
// writes it at the product's new number.  A use without exactly one match
// sets the error word and gets entity 0, which keeps every index in range.
constexpr int kMatchLanes = 4;

template <int HIGH>
__device__ __forceinline__ void match_use(LO t, SideDim const& a, int* error) {
  LO u = t / kMatchLanes;
  int lane = t % kMatchLanes;
  constexpr int LOW = HIGH - 1;
  constexpr int nvh = HIGH + 1;
  constexpr int nvl = LOW + 1;
  int found = 0;
  LO at = 0;
  if (u < a.nuses) {
    LO h = u / (HIGH + 1);
    int which = u % (HIGH + 1);
    at = (a.prods2new ? a.prods2new[h] : h) * nvh + which;
    LO av[3];
#pragma unroll
    for (int k = 0; k < nvl; ++k) av[k] = a.pverts[h * nvh + down_template(HIGH, LOW, which, k)];
    LO vm = min_vertex<nvl>(av);
    LO k0 = a.a2ab[vm], k1 = a.a2ab[vm + 1] - 1;
    for (LO k = k0 + lane; k < k1; k += kMatchLanes) {
      int4 r = a.rows[k];
      LO bv[3] = {r.y, r.z, r.w};
      // wd: the position of the use's first vertex in the candidate
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
      a.out[at] = r.x;
      a.codes[at] = code;
      ++found;
    }
  }
  for (int d = kMatchLanes / 2; d > 0; d >>= 1) found += __shfl_xor(found, d, 64);
  if (u < a.nuses && lane == 0 && found != 1) {
    a.out[at] = 0;
    a.codes[at] = 0;
    *error = kReflectDownNoMatch;
  }
}

__global__ void __launch_bounds__(kBlock) match_uses(SideJobs j, int* error) {
  int w = side_job(j);
  if (j.high[w] == 2)
    match_use<2>(job_thread(j, w), j.d[w], error);
  else
    match_use<3>(job_thread(j, w), j.d[w], error);
}

// per side, the number of elements on it (high 32 bits) and the sum of their
// indices (low 32 bits) by one 64-bit atomic add per element side: with two
// elements, either one finds the other as the sum minus itself
__global__ void side_elems_init(LO ns, unsigned long long* se) {
  LO s = thread_index();
  if (s < ns) se[s] = 0ull;
}

__global__ void side_elems_kernel(LO nuses, int nspe, LO const* es2s, unsigned long long* se) {
  LO i = thread_index();
  if (i >= nuses) return;
  LO e = i / nspe;
  atomicAdd(&se[es2s[i]], (1ull << 32) + static_cast<unsigned long long>(e));
}

// elements_across_sides (src/Omega_h_adj.cpp:591-657) from the per-side
// words: each element lists the other element across each of its sides that
// has two, in side order
__global__ void dual_degrees(LO ne, int nspe, LO const* es2s, unsigned long long const* se,
    LO* deg, int* error) {
  LO e = thread_index();
  if (e >= ne) return;
  LO d = 0;
  for (int j = 0; j < nspe; ++j) {
    unsigned count = unsigned(se[es2s[e * nspe + j]] >> 32);
    if (count == 2) ++d;
    if (count > 2) *error = kNonManifoldSide;
  }
  deg[e] = d;
}

__global__ void dual_fill(LO ne, int nspe, LO const* es2s, unsigned long long const* se,
    LO const* a2ab, LO* ab2b) {
  LO e = thread_index();
  if (e >= ne) return;
  LO k = a2ab[e];
  for (int j = 0; j < nspe; ++j) {
    unsigned long long w = se[es2s[e * nspe + j]];
    if (unsigned(w >> 32) == 2) ab2b[k++] = LO(unsigned(w)) - e;
  }
}

__global__ void verts_across_edges_kernel(LO nve, LO const* ve2e, I8 const* codes,
    LO const* ev2v, LO* vv2v) {
  LO ve = thread_index();
  if (ve >= nve) return;
  LO e = ve2e[ve];
  int eev = code_which_down(codes[ve]);
  vv2v[ve] = ev2v[e * 2 + (1 - eev)];
}

__global__ void edge_star_degrees(LO ne, LO const* e2f_a2ab, LO const* e2t_a2ab, LO* deg) {
  LO e = thread_index();
  if (e >= ne) return;
  LO d = 2 * (e2f_a2ab[e + 1] - e2f_a2ab[e]);
  if (e2t_a2ab) d += e2t_a2ab[e + 1] - e2t_a2ab[e];
  deg[e] = d;
}

__global__ void edge_star_fill(LO ne, LO const* e2f_a2ab, LO const* e2f_ab2b,
    I8 const* e2f_codes, LO const* fe2e, LO const* e2t_a2ab, LO const* e2t_ab2b,
    I8 const* e2t_codes, LO const* te2e, LO const* a2ab, LO* ab2b) {
  LO e = thread_index();
  if (e >= ne) return;
  LO k = a2ab[e];
  for (LO ef = e2f_a2ab[e]; ef < e2f_a2ab[e + 1]; ++ef) {
    LO f = e2f_ab2b[ef];
    int ffe = code_which_down(e2f_codes[ef]);
    ab2b[k++] = fe2e[f * 3 + ((ffe + 1) % 3)];
    ab2b[k++] = fe2e[f * 3 + ((ffe + 2) % 3)];
  }
  if (e2t_a2ab) {
    for (LO er = e2t_a2ab[e]; er < e2t_a2ab[e + 1]; ++er) {
      LO r = e2t_ab2b[er];
      int rre = code_which_down(e2t_codes[er]);
      ab2b[k++] = te2e[r * 6 + opposite_template(3, 1, rre)];
    }
  }
}

}  // namespace

Adj invert_adj_rows(Ctx& c, LO nhigh, int deg, LO nlow, LOs const& hl2l,
    Bytes const* down_codes) {
  return invert_adj(c, nhigh, deg, nlow, hl2l, down_codes);
}

LOs const& verts_of(Ctx& c, DMesh& m, int d) {
  if (d == 1) return m.down[1];
  if (!m.verts[d].exists()) {
    LO n = m.nents[d];
    LOs out(c, n * (d + 1));
    if (d == 2) {
      OSH_LAUNCH((transit_kernel<2, 0>), n * 3, c, m.down[2].data(), m.down_codes[2].data(),
          m.down[1].data(), (I8 const*)nullptr, out.data(), (I8*)nullptr);
    } else {
      Bytes const* codes;
      LOs const& t2e = ask_down(c, m, 3, 1, &codes);
      OSH_LAUNCH((transit_kernel<3, 0>), n * 4, c, t2e.data(), codes->data(), m.down[1].data(),
          (I8 const*)nullptr, out.data(), (I8*)nullptr);
    }
    m.verts[d] = out;
  }
  return m.verts[d];
}

LOs const& ask_down(Ctx& c, DMesh& m, int high, int low, Bytes const** codes) {
  if (low == 0) {
    if (codes) *codes = nullptr;
    return verts_of(c, m, high);
  }
  if (low == high - 1) {
    if (codes) *codes = &m.down_codes[high];
    return m.down[high];
  }
  if (!m.t2e.exists()) {
    LO n = m.nents[3];
    m.t2e = LOs(c, n * 6);
    m.t2e_codes = Bytes(c, n * 6);
    OSH_LAUNCH((transit_kernel<3, 1>), n * 6, c, m.down[3].data(), m.down_codes[3].data(),
        m.down[2].data(), m.down_codes[2].data(), m.t2e.data(), m.t2e_codes.data());
  }
  if (codes) *codes = &m.t2e_codes;
  return m.t2e;
}

void marked_ups(Ctx& c, DMesh& m, int low, Bytes const& marks, int n, int const* highs,
    bool const* sorted, Adj* out, LOs const* zeros) {
  Invert in[kMaxUseJobs];
  OSH_CHECK(n <= kMaxUseJobs, "marked_ups: too many dimensions");
  for (int w = 0; w < n; ++w) {
    Bytes const* codes = nullptr;
    in[w].hl2l = ask_down(c, m, highs[w], low, &codes);
    in[w].down_codes = codes;
    in[w].nhigh = m.nents[highs[w]];
    in[w].deg = simplex_degree(highs[w], low);
    in[w].nlow = m.nents[low];
    in[w].marks = &marks;
    in[w].sorted = sorted[w];
  }
  OSH_CHECK(!zeros || zeros->size() >= n * m.nents[low], "marked_ups: too few zeros");
  invert_adjs(c, n, in, out, zeros);
}

Adj const& ask_up(Ctx& c, DMesh& m, int low, int high) {
  if (!m.up[low][high].exists()) {
    Bytes const* codes = nullptr;
    LOs const& down = ask_down(c, m, high, low, &codes);
    m.up[low][high] = invert_adj(c, m.nents[high], simplex_degree(high, low), m.nents[low],
        down, codes);
  }
  return m.up[low][high];
}

namespace {

// sets the jobs' workgroups for a sweep with n[w] threads in job w; returns
// their number
unsigned side_blocks(SideJobs& j, std::int64_t const* n) {
  unsigned b = 0;
  for (int w = 0; w < j.n; ++w) {
    j.first[w] = b;
    OSH_CHECK(n[w] <= std::int64_t(0x7fffffff), "reflect_down: too many uses");
    b += unsigned((n[w] + kBlock - 1) / kBlock);
    j.first[w + 1] = b;
  }
  return b;
}

void run_sides(Ctx& c, DMesh& m, SideJobs& j, LOs const* zeros = nullptr) {
  LO nv = m.nents[0];
  bool enough = zeros && zeros->size() >= nv * j.n;
  LOs counts = enough ? *zeros : fill_lo(c, nv * j.n, 0);
  LOs slot[2], a2ab[2];
  DArray<int4> rows[2];
  ScanJob scans[2];
  std::int64_t uses[2], lows[2], lanes[2];
  for (int w = 0; w < j.n; ++w) {
    SideDim& a = j.d[w];
    a.counts = counts.data() + std::size_t(w) * nv;
    slot[w] = LOs(c, a.nl);
    a.slot = slot[w].data();
    a2ab[w] = LOs(c, nv + 1);
    a.a2ab = a2ab[w].data();
    // every lower entity in at most one row plus one spare slot per marked row
    rows[w] = DArray<int4>(c, a.nl + nv);
    a.rows = rows[w].data();
    scans[w] = {a.counts, kScanLO, nv, a2ab[w].data(), nullptr};
    uses[w] = a.nuses;
    lows[w] = a.nl;
    lanes[w] = std::int64_t(a.nuses) * kMatchLanes;
  }
  auto launch = [&](auto kernel, std::int64_t const* n, auto... args) {
    unsigned b = side_blocks(j, n);
    if (b == 0) return;
    hipLaunchKernelGGL(kernel, dim3(b), dim3(kBlock), 0, c.stream, j, args...);
    OSH_HIP(hipGetLastError());
  };
  launch(mark_use_min_verts, uses);
  launch(count_min_rows, lows);
  offset_scans(c, scans, j.n);
  launch(fill_min_rows, lows);
  launch(match_uses, lanes, c.error_word());
}

}  // namespace

void reflect_down(Ctx& c, DMesh& m, int high_dim, LO nprods, LOs const& prod_verts,
    LOs& down, Bytes& codes) {
  int low_dim = high_dim - 1;
  LO nuses = nprods * (high_dim + 1);
  down = LOs(c, nuses);
  codes = Bytes(c, nuses);
  if (nuses == 0) return;
  SideJobs j{};
  j.n = 1;
  j.high[0] = high_dim;
  SideDim& a = j.d[0];
  a.nuses = nuses;
  a.pverts = prod_verts.data();
  a.nl = m.nents[low_dim];
  a.lv2v = verts_of(c, m, low_dim).data();
  a.out = down.data();
  a.codes = codes.data();
  run_sides(c, m, j);
}

void match_sides(Ctx& c, DMesh& nw, Products const* prods, ModOut const* mo,
    LOs const* zeros) {
  SideJobs j{};
  for (int d = 2; d <= nw.dim; ++d) {
    if (prods[d].n == 0) continue;
    j.high[j.n] = d;
    SideDim& a = j.d[j.n++];
    a.nuses = prods[d].n * (d + 1);
    a.pverts = prods[d].verts.data();
    a.prods2new = mo[d].prods2new.data();
    a.nl = nw.nents[d - 1];
    a.lv2v = verts_of(c, nw, d - 1).data();
    a.out = nw.down[d].data();
    a.codes = nw.down_codes[d].data();
  }
  if (j.n) run_sides(c, nw, j, zeros);
}

Adj const& ask_star(Ctx& c, DMesh& m, int d) {
  if (!m.star[d].exists()) {
    Adj g;
    if (d == 0) {
      Adj const& v2e = ask_up(c, m, 0, 1);
      g.a2ab = v2e.a2ab;
      g.ab2b = LOs(c, v2e.ab2b.size());
      OSH_LAUNCH(verts_across_edges_kernel, v2e.ab2b.size(), c, v2e.ab2b.data(),
          v2e.codes.data(), m.down[1].data(), g.ab2b.data());
    } else {
      LO ne = m.nents[1];
      Adj const& e2f = ask_up(c, m, 1, 2);
      Adj const* e2t = nullptr;
      LO const* te2e = nullptr;
      if (m.dim == 3) {
        e2t = &ask_up(c, m, 1, 3);
        te2e = ask_down(c, m, 3, 1, nullptr).data();
      }
      LOs deg(c, ne);
      OSH_LAUNCH(edge_star_degrees, ne, c, e2f.a2ab.data(),
          e2t ? e2t->a2ab.data() : (LO const*)nullptr, deg.data());
      LO total;
      g.a2ab = offset_scan(c, deg, &total);
      g.ab2b = LOs(c, total);
      OSH_LAUNCH(edge_star_fill, ne, c, e2f.a2ab.data(), e2f.ab2b.data(), e2f.codes.data(),
          m.down[2].data(), e2t ? e2t->a2ab.data() : (LO const*)nullptr,
          e2t ? e2t->ab2b.data() : (LO const*)nullptr,
          e2t ? e2t->codes.data() : (I8 const*)nullptr, te2e, g.a2ab.data(), g.ab2b.data());
    }
    m.star[d] = g;
  }
  return m.star[d];
}

Adj const& ask_dual(Ctx& c, DMesh& m) {
  if (!m.dual.exists()) {
    int dim = m.dim;
    LO ne = m.nents[dim];
    auto const& se = ask_side_elems(c, m);
    LOs deg(c, ne);
    OSH_LAUNCH(dual_degrees, ne, c, dim + 1, m.down[dim].data(), se.data(), deg.data(),
        c.error_word());
    Adj g;
    LO total;
    g.a2ab = offset_scan(c, deg, &total);
    g.ab2b = LOs(c, total);
    OSH_LAUNCH(dual_fill, ne, c, dim + 1, m.down[dim].data(), se.data(), g.a2ab.data(),
        g.ab2b.data());
    m.dual = g;
  }
  return m.dual;
}

DArray<unsigned long long> const& ask_side_elems(Ctx& c, DMesh& m) {
  if (!m.side_elems.exists()) {
    int dim = m.dim;
    LO ns = m.nents[dim - 1];
    DArray<unsigned long long> se(c, ns);
    OSH_LAUNCH(side_elems_init, ns, c, se.data());
    OSH_LAUNCH(side_elems_kernel, m.nents[dim] * (dim + 1), c, dim + 1, m.down[dim].data(),
        se.data());
    m.side_elems = se;
  }
  return m.side_elems;
}

// ---------------------------------------------------------------- find_unique
namespace {

template <int HIGH, int LOW>
__global__ void form_canonical_uses(LO nuses, LO const* hv2v, LO* uv2v, I64* canon) {
  LO u = thread_index();
  if (u >= nuses) return;
  constexpr int nvh = HIGH + 1;
  constexpr int nlh = (HIGH == 3) ? (LOW == 1 ? 6 : 4) : 3;
  constexpr int deg = LOW + 1;
  LO h = u / nlh;
  int which = u % nlh;
  LO ev[3];
  for (int k = 0; k < deg; ++k) {
    ev[k] = hv2v[h * nvh + down_template(HIGH, LOW, which, k)];
    uv2v[u * deg + k] = ev[k];
  }
  int min_j = 0;
  LO min_v = ev[0];
  for (int j = 1; j < deg; ++j)
    if (ev[j] < min_v) {
      min_j = j;
      min_v = ev[j];
    }
  int rotation = (deg - min_j) % deg;
  LO tmp[3];
  for (int j = 0; j < deg; ++j) tmp[(j + rotation) % deg] = ev[j];
  if (deg == 3 && tmp[2] < tmp[1]) {
    LO t = tmp[1];
    tmp[1] = tmp[2];
    tmp[2] = t;
  }
  for (int j = 0; j < deg; ++j) canon[I64(u) * deg + j] = tmp[j];
}

__global__ void mark_group_ends(LO n, int deg, I64 const* canon, LO const* sorted2u, I8* last) {
  LO s = thread_index();
  if (s >= n) return;
  I8 r = 1;
  if (s < n - 1) {
    LO a = sorted2u[s], b = sorted2u[s + 1];
    r = 0;
    for (int j = 0; j < deg; ++j)
      if (canon[I64(a) * deg + j] != canon[I64(b) * deg + j]) r = 1;
  }
  last[s] = r;
}

__global__ void gather_unique(LO nlow, int deg, LO const* ends, LO const* sorted2u,
    LO const* uv2v, LO* out) {
  LO i = thread_index();
  if (i >= nlow) return;
  LO u = sorted2u[ends[i]];
  for (int j = 0; j < deg; ++j) out[i * deg + j] = uv2v[u * deg + j];
}

}  // namespace

LOs find_unique(Ctx& c, LO nhigh, int high_dim, int low_dim, LOs const& hv2v) {
  int nlh = simplex_degree(high_dim, low_dim);
  int deg = low_dim + 1;
  LO nuses = nhigh * nlh;
  LOs uv2v(c, nuses * deg);
  DArray<I64> canon(c, nuses * deg);
  if (high_dim == 3 && low_dim == 1)
    OSH_LAUNCH((form_canonical_uses<3, 1>), nuses, c, hv2v.data(), uv2v.data(), canon.data());
  else if (high_dim == 3 && low_dim == 2)
    OSH_LAUNCH((form_canonical_uses<3, 2>), nuses, c, hv2v.data(), uv2v.data(), canon.data());
  else
    OSH_LAUNCH((form_canonical_uses<2, 1>), nuses, c, hv2v.data(), uv2v.data(), canon.data());
  LOs sorted2u = sort_by_keys(c, canon, deg);
  Bytes ends(c, nuses);
  OSH_LAUNCH(mark_group_ends, nuses, c, deg, canon.data(), sorted2u.data(), ends.data());
  LOs e2sorted = collect_marked(c, ends);
  LO nlow = e2sorted.size();
  LOs out(c, nlow * deg);
  OSH_LAUNCH(gather_unique, nlow, c, deg, e2sorted.data(), sorted2u.data(), uv2v.data(),
      out.data());
  return out;
}

}  // namespace osh
