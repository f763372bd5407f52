// Internal interfaces shared by the adapt() passes.
#pragma once

#include <functional>

#include "osh_mesh.hpp"

namespace osh {

// mirrors Omega_h::AdaptOpts (src/Omega_h_adapt.hpp:50-77)
struct AdaptOptions {
  Real min_length_desired;
  Real max_length_desired;
  Real max_length_allowed;
  Real min_quality_allowed;
  Real min_quality_desired;
  int nsliver_layers;
  int verbosity;
  int should_refine;
  int should_coarsen;
  int should_swap;
  int should_coarsen_slivers;
  Real length_histogram_min;
  Real length_histogram_max;
  int nlength_histogram_bins;
  int nquality_histogram_bins;
  int should_prevent_coarsen_flip;
  // 0 FP64; 1 mixed: cavity screens in FP32, every cavity the screen does
  // not reject by a margin re-evaluated in FP64 (same mesh, bit for bit)
  int precision;
};

void default_options(int dim, AdaptOptions& o);

// the new numbers of one dimension's entities after modify_ents: old2new
// (-1 for entities that do not survive; built only for meshes that carry
// tags) and, per product, prods2new
struct ModOut {
  LO nold = 0;
  LO nnew = 0;
  LO nprods = 0;
  LOs old2new;
  LOs prods2new;
};

// modify_ents_adapt (src/Omega_h_modify.cpp:468-517) in steps that each cover
// every dimension of a pass in one launch: plan_keys marks the same entities,
// counts the new entities each old one stands for, finds the representatives
// and scans the counts; rebuild_same moves the same entities with all they
// carry; place_products numbers the products; match_sides connects them
struct ModPlan {
  int ent_dim = 0, key_dim = 0;
  LO nold = 0, nnew = 0;
  Bytes same;
  LOs counts, reps, offsets;
};
// what a pass's keys come to.  The caller sets, per rebuilt dimension, the
// products of every key-dimension entity (0 where it is no key), or the fixed
// count of each key.
struct KeyedMods {
  LOs prod_counts[4];
  LO fixed_prods[4] = {0, 0, 0, 0};
  LO nkeys = 0;
  LOs keys2kds;
  LOs k2p[4];
  LO nprods[4] = {0, 0, 0, 0};
  ModPlan plans[4];  // plans[d - d0]
  LOs order;         // of the dimension below the keys, by key-dimension entity
  LOs head;          // by entity of the dimension below the keys
  LOs first_up[4];   // by key-dimension entity
};
// allocates what plan_keys needs to start out constant; `fills` has to run
// before it
void prepare_keys(DMesh const& old, int key_dim, int d0, int d1, Fills& fills, KeyedMods& out);
// the plans of dimensions d0..d1 from the keys, a mask over the key dimension,
// with one wait for everything that depends on the keys
void plan_keys(Ctx& c, DMesh& old, int key_dim, int d0, int d1, Bytes const& keys,
    KeyedMods& out);
// the scans of plans' counts, for a launch of the caller's: the jobs (totals in
// pinned slots first_slot...), then, after the caller's wait, the totals
int modify_scan_jobs(Ctx& c, ModPlan* plans, int nplans, ScanJob* jobs, int first_slot);
void modify_scan_totals(Ctx& c, ModPlan* plans, int nplans, int first_slot);

// the swap choices carried along with the edges (see SwapCache)
struct SwapCache;
struct CacheMove {
  SwapCache const* from;
  SwapCache* to;
  Bytes const* dirty;
};
// the new mesh's arrays of dimensions d0..dim with the same entities in
// place: connectivity, codes and vertex lists renumbered, classification,
// lengths and qualities, and for dimension 0 coordinates and metric, in one
// launch (transfer_common's same part, src/Omega_h_transfer.cpp:149-180, and
// modify_conn, src/Omega_h_modify.cpp:446-466).  plans[d - d0] and mo[d] are
// dimension d's; dimensions below d0 must be set in nw and keep their numbers.
void rebuild_same(Ctx& c, DMesh& old, DMesh& nw, int d0, ModPlan const* plans, ModOut* mo,
    CacheMove const* cache = nullptr);
// the products of one dimension: vertex lists in the new numbering (absent
// for vertices) and the entity each comes from: src[p] of dimension src_dim,
// or src_dims[p]; without src the key itself, of dimension src_dim
struct Products {
  LO n = 0;
  LOs keys2prods;
  LOs verts;
  LOs src;
  int src_dim = 0;
  Bytes src_dims;
};
// numbers the products of dimensions d0..d1 (prods[d], mo[d], plans[d -
// plan0]) and writes their vertex lists and classification, in one launch;
// inheritance tags of those dimensions follow.  order: KeyedMods::order, for
// the dimension below the keys; new_edges_valid, when given, is zeroed at new
// edges.
void place_products(Ctx& c, DMesh& old, DMesh& nw, int d0, int d1, int plan0,
    ModPlan const* plans, LOs const& keys2kds, Products const* prods, ModOut* mo,
    LOs const* order = nullptr, I8* new_edges_valid = nullptr);
// the sides and codes of the placed products of dimensions 2..dim, by their
// vertices among the new mesh's entities (reflect_down); `zeros` (when given
// and long enough): a zero per vertex of the new mesh and such dimension, to be
// used up
void match_sides(Ctx& c, DMesh& nw, Products const* prods, ModOut const* mo,
    LOs const* zeros = nullptr);
// lengths of new edges and qualities of new elements, in one launch
void measure_products(Ctx& c, DMesh& nw, ModOut const* mo);
// every tag of a rebuilt mesh but the vertex tags' and refinement's own
bool has_tags(DMesh const& m);

// new tag data: same entities copy old values, products take prod values
template <class T>
DArray<T> transfer(Ctx& c, ModOut const& mo, int ncomps, DArray<T> const& old_data,
    DArray<T> const* prod_data);
// element tags of the new elements: products take the value of old element
// prod_src[p] (no products when prod_src is null)
void transfer_elem_tags(Ctx& c, DMesh const& old, DMesh& nw, ModOut const& mo,
    LOs const* prod_src);
// transfer_pointwise (src/Omega_h_transfer.cpp:515-583) of the element tags
// for coarsening (key_dim 0) and swap (key_dim 1): prod_verts are the
// products' vertices in the new mesh, whose coordinates are already set
void transfer_pointwise(Ctx& c, DMesh& old, DMesh& nw, ModOut const& mo, int key_dim,
    LOs const& keys2kds, LOs const& keys2prods, LOs const& prod_verts);

// conservative and momentum transfer (osh_conserve.hip): setup_conservation_tags
// (src/Omega_h_conserve.cpp:578-606) zeroes the integral errors at the start
// of adapt(); conserve_pass transfers densities by intersection and the
// errors through one pass (op 0 refine, 1 coarsen, 2 swap; keys of
// dimension key_dim, k2p their element products, after the other element
// transfers of the pass); conserve_correct is correct_integral_errors
// (src/Omega_h_conserve.cpp:799-829) at the end of adapt()
bool conserve_any(DMesh const& m);
void conserve_setup(Ctx& c, DMesh& m);
void conserve_pass(Ctx& c, DMesh& old, DMesh& nw, int op, int key_dim, LOs const& keys2kds,
    LOs const& k2p, ModOut const& mo);
constexpr int kMaxDiffusionSweeps = 100000;
void conserve_correct(Ctx& c, DMesh& m, int max_sweeps);

// *any_cands (when given) tells whether any entity was a candidate; for
// edges, `edge_elems` (when given) is an edge -> element adjacency holding at
// least the rows of the candidate edges; for vertices, `star` (when given) is
// the vertex star holding at least the rows of the candidates.  With `stop`, a
// word (Ctx::words) that earlier kernels may have set to the tag: the rounds end
// at the first wait that brings it, and the set is of no use then
struct StopWord {
  int word;
  unsigned tag;
};
Bytes find_indset(Ctx& c, DMesh& m, int d, Reals const& quality, Bytes const& cands,
    bool* any_cands = nullptr, Adj const* edge_elems = nullptr, Adj const* star = nullptr,
    StopWord const* stop = nullptr);
Bytes mark_down(Ctx& c, DMesh& m, int high, int low, Bytes const& marks);
// mark_sliver_layers: the arrays that start out constant go into `fills`, which
// has to run before mark()
class SliverLayers {
 public:
  SliverLayers(Ctx& c, DMesh& m, int nlayers, Fills& fills);
  Bytes mark(Real qual_ceil);
  // marks (zero so far) of the marked elements' edges of class dimension dim:
  // mark_by_class_dim of their edges
  void mark_interior_edges(Real qual_ceil, Bytes& edge_marks);
  // after a find_indset that follows mark(): records what it has found out
  // about the mesh (DMesh::linked)
  void settle();

 private:
  Ctx& c_;
  DMesh& m_;
  int nlayers_;
  LOs counts_;
  unsigned tag_ = 0;
  I8* edge_marks_ = nullptr;
};

bool refine_by_size(Ctx& c, DMesh& m, AdaptOptions const& o);
bool coarsen_by_size(Ctx& c, DMesh& m, AdaptOptions const& o);
bool coarsen_slivers(Ctx& c, DMesh& m, AdaptOptions const& o);
// The 3D swap choice of each edge (its configuration, whether it improves
// on the edge's elements and the quality it reaches) is a function of the
// tets around the edge, the coordinates and metric of their vertices and
// max_length_allowed only.  Between swap passes of one adapt() nothing else
// moves, so the choices of edges whose tets a pass did not touch carry over
// to the next mesh; `valid` marks them, per edge of the current mesh.
struct SwapCache {
  Bytes valid;
  Bytes cfg;
  Bytes keep;
  Reals q;
  void clear() { *this = SwapCache(); }
};

// with a cache (only for consecutive swap passes of one adapt(), cleared by
// the caller whenever anything else changes the mesh, its metric or the
// options) the 3D pass evaluates only the candidates not carried over
bool swap_edges(Ctx& c, DMesh& m, AdaptOptions const& o, SwapCache* cache = nullptr);
// the swap choices of given interior edges of a 3D mesh (swap3d_qualities
// and the choice of a triangulation): per edge the chosen triangulation (-1
// for none) and the quality of a triangulation that improves on the edge's
// elements (-1 otherwise)
void swap3d_choices(Ctx& c, DMesh& m, AdaptOptions const& o, LOs const& edges,
    LOs& configs_out, Reals& quals_out);

// known-answer hooks used by the tests
Reals refine_qualities(Ctx& c, DMesh& m, LOs const& cands);
// coarsen_qualities (src/Omega_h_coarsen_qualities.cpp:65-88) on device
// arrays, stream-ordered: out[2 i + col] is the quality after collapsing
// candidate i's edge in direction col (-1 where cand_codes[i] does not
// collapse that way).  precision 1 screens in FP32 first: a direction whose
// estimate falls below qmin by more than the band gets -1 instead of its
// FP64 value (the filter that follows rejects it either way).
void coarsen_qualities(Ctx& c, DMesh& m, LO ncands, LO const* cands, I8 const* cand_codes,
    Real* out, int precision, Real qmin);
void find_loops(Ctx& c, DMesh& m, LOs const& edges, LOs& eev2v, LOs& loop_verts, LOs& sizes);

// the batched form (osh_batch.hip): meshes joined into one disjoint mesh
// (part k's entities of every dimension after those of parts < k; the
// vertex tag kPartTag holds each vertex's part), adapted as one, split back
extern char const* const kPartTag;
void join_meshes(Ctx& c, std::vector<DMesh const*> const& parts, DMesh& out);
// first entity and entity count of each part in every dimension; an error
// unless each part is one block and the blocks follow the part order
void part_ranges(Ctx& c, DMesh& m, int nparts, std::vector<LO> first[4],
    std::vector<LO> count[4]);
void split_mesh(Ctx& c, DMesh& m, int nparts, std::vector<DMesh>& out);
// with Ctx::part_changed set, marks the parts of the pass's keys (the part
// of a key's first vertex) as changed; called by every pass with its keys
void note_changed_parts(Ctx& c, DMesh const& m, int key_dim, LOs const& keys2kds);
// the minimum element quality of each part of a joined mesh (a part
// without elements gets +infinity)
std::vector<Real> part_min_quality(Ctx& c, DMesh& m, int nparts);

struct PassRecord {
  int kind;  // 0 refine, 1 coarsen, 2 swap, 3 coarsen slivers
  LO nelems_in;
  LO nelems_out;
  double seconds;
};

// called with the mesh after every pass that changed it (outside the pass's
// timing), for callers that record the mesh pass by pass
using PassHook = std::function<void(DMesh&)>;
bool adapt(Ctx& c, DMesh& m, AdaptOptions const& o, std::vector<PassRecord>* log,
    PassHook const* hook = nullptr);
// adapt() of many meshes at once (the batched form): joined into one
// disjoint mesh whose passes cover every mesh in one launch per kernel, with
// the parts that can no longer change set aside as they appear; each mesh
// ends where adapt() alone leaves it.  Returns adapt()'s result per mesh.
std::vector<int> adapt_batch(Ctx& c, std::vector<DMesh>& meshes, AdaptOptions const& o,
    std::vector<PassRecord>* log);
// approach_metric (src/Omega_h_approach.cpp:83-126): move the metric toward
// the "target_metric" vertex tag; false when there is no target
bool approach_metric(Ctx& c, DMesh& m, AdaptOptions const& o, Real min_step);
// Mesh::set_coords (src/Omega_h_mesh.cpp:365-368): drops the cached lengths,
// qualities and sizes
void set_coords(DMesh& m, Reals const& v);
// warp_to_limit (src/Omega_h_approach.cpp:36-81): move the vertices by the
// "warp" vertex tag as far as quality and lengths allow; false without one
bool warp_to_limit(Ctx& c, DMesh& m, AdaptOptions const& o, bool exit_on_stall, int max_niters);
// get_implied_isos (src/Omega_h_metric.cpp:316-321): nverts values
Reals implied_isos(Ctx& c, DMesh& m);
// compute_ill_metric_dim, fix_for_given_metric, fix, grade_fix_adapt
// (src/Omega_h_fix.cpp:16-176); isotropy 0 anisotropic, 1 iso length,
// 2 iso size; the fix functions return the number of adapt() calls
void ill_metric(Ctx& c, DMesh& m, AdaptOptions const& o, int isotropy);
int fix_for_given_metric(Ctx& c, DMesh& m, AdaptOptions const& o);
int fix(Ctx& c, DMesh& m, AdaptOptions const& o, int isotropy);
int grade_fix_adapt(Ctx& c, DMesh& m, AdaptOptions const& o, int ncomps, Reals const& target);

}  // namespace osh
