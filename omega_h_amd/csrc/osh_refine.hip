// Edge refinement pass on the device.
//
//   refine_by_size / refine_ghosted / refine_element_based src/Omega_h_refine.cpp:17-100
//   refine_qualities (MetricRefineQualities)  src/Omega_h_refine_qualities.cpp:13-86
//   refine_edges_to_pairs / refine_domains_to_pairs / _cuts / combine
//                                             src/Omega_h_refine_topology.cpp:13-203
//   transfer_refine (coords, metric, class, length, quality)
//                                             src/Omega_h_transfer.cpp:182-428
#include <cstdio>

#include "osh_math.hpp"
#include "osh_passes.hpp"

namespace osh {

namespace {

__global__ void gt_kernel(LO n, Real const* a, Real v, I8* out) {
  LO i = thread_index();
  if (i < n) out[i] = a[i] > v;
}

// by edge: whether a candidate's quality reaches qmin, and the quality
struct RefineSeeds {
  Real qmin = 0.0;
  I8* keep = nullptr;
  Real* quals = nullptr;
};

// 2^lshift lanes per candidate edge (consecutive threads of one wave): the
// lanes share the 2 x (elements around the edge) children, each measured
// with the max-determinant metric of its cell-side vertices and the edge
// midpoint, and combine their minima with shuffles.  The minimum does not
// depend on the order (min2 never takes a NaN, and the sign of a zero
// decides nothing downstream: the candidates' qualities are only compared).
template <int D, int M>
__global__ void __launch_bounds__(kBlock) refine_qualities_kernel(LO nt, int lshift,
    LO ncands, LO const* cands, LO const* ev2v, LO const* cv2v, LO const* e2c_a2ab,
    LO const* e2c_ab2b, I8 const* e2c_codes, Real const* coords, Real const* metric,
    Real const* midpt_metrics, Real* out, RefineSeeds seeds) {
  LO t = thread_index();
  int lanes = 1 << lshift;
  LO cand = t >> lshift;
  int lane = t & (lanes - 1);
  // every lane of a group stays for the shuffles; groups past the end (whole
  // groups, as nt is a multiple of the lane count) do no work
  bool valid = t < nt && cand < ncands;
  constexpr int nc = (M == 1) ? 1 : (M == 2 ? 3 : 6);
  double minqual = 1.0;
  LO e = valid ? cands[cand] : 0;
  LO row = valid ? e2c_a2ab[e] : 0;
  LO nchildren = valid ? 2 * (e2c_a2ab[e + 1] - row) : 0;
  double midp[D];
  double mm[nc];
  if (lane < nchildren) {
    for (int j = 0; j < D; ++j)
      midp[j] = (coords[ev2v[e * 2] * D + j] + coords[ev2v[e * 2 + 1] * D + j]) / 2.;
    for (int k = 0; k < nc; ++k) mm[k] = midpt_metrics[cand * nc + k];
  }
  for (LO ch = lane; ch < nchildren; ch += lanes) {
    LO ec = row + ch / 2;
    int eev = ch % 2;
    LO c = e2c_ab2b[ec];
    I8 code = e2c_codes[ec];
    int cce = code_which_down(code);
    int rot = code_rotation(code);
    {
      int cev = eev ^ rot;
      int ccv = down_template(D, 1, cce, cev);
      int ccs = opposite_template(D, 0, ccv);
      double p[D + 1][D];
      double m[D + 1][nc];
      for (int csv = 0; csv < D; ++csv) {
        LO v = cv2v[c * (D + 1) + down_template(D, D - 1, ccs, csv)];
        for (int j = 0; j < D; ++j) p[csv][j] = coords[v * D + j];
        for (int k = 0; k < nc; ++k) m[csv][k] = metric[v * nc + k];
      }
      for (int j = 0; j < D; ++j) p[D][j] = midp[j];
      for (int k = 0; k < nc; ++k) m[D][k] = mm[k];
      double const* pp[D + 1];
      double const* ms[D + 1];
      for (int k = 0; k < D + 1; ++k) {
        pp[k] = p[k];
        ms[k] = m[k];
      }
      if (D == 3) {
        double const* t = pp[1];
        pp[1] = pp[2];
        pp[2] = t;
        t = ms[1];
        ms[1] = ms[2];
        ms[2] = t;
      }
      double q = element_quality<D, M>(pp, ms);
      minqual = math::min2(minqual, q);
    }
  }
  for (int d = lanes / 2; d > 0; d /= 2) minqual = math::min2(minqual, __shfl_xor(minqual, d, 64));
  if (!valid || lane != 0) return;
  if (out) out[cand] = minqual;
  if (seeds.keep) {
    seeds.keep[e] = minqual >= seeds.qmin;
    seeds.quals[e] = minqual;
  }
}

// the rows that refinement products of dimensions 1..3 come from: pairs (the
// entities of the dimension around the key edge, two products each; the edge
// itself in dimension 1) and cuts (the entities one dimension up, one product
// each)
struct RefineRows {
  LO const* pairs_a2ab[3];  // null: none
  LO const* pairs_ab2b[3];
  I8 const* pairs_codes[3];
  LO const* pair_verts[3];
  LO const* cuts_a2ab[3];
  LO const* cuts_ab2b[3];
  I8 const* cuts_codes[3];
  LO const* cut_verts[3];
  LO const* keys2prods[3];
  LO* counts[3];
  LO* pv[3];
  LO* psrc[3];
  I8* psrc_dim[3];
};

// the products of every edge in dimensions 1..n (0 for edges that are no keys)
__global__ void prod_counts(LO nedges, int n, I8 const* keys, RefineRows r) {
  LO e = thread_index();
  if (e >= nedges) return;
  bool key = keys[e] != 0;
  for (int d = 0; d < n; ++d) {
    LO k = 0;
    if (key) {
      k = r.pairs_a2ab[d] ? 2 * (r.pairs_a2ab[d][e + 1] - r.pairs_a2ab[d][e]) : 2;
      if (r.cuts_a2ab[d]) k += r.cuts_a2ab[d][e + 1] - r.cuts_a2ab[d][e];
    }
    r.counts[d][e] = k;
  }
}

// every product's position follows from its row entry, so kRowLanes threads
// per key and dimension share the rows; one thread per key and a launch per
// dimension was a chain of dependent gathers (12 to 24 us a launch)
constexpr int kRowLanes = 8;

template <int ED>
__device__ __forceinline__ void refine_products_of(int lane, LO e, LO mid, LO prod0,
    LO const* ev2v, LO const* vert_offsets, RefineRows const& r) {
  constexpr int nv = ED + 1;
  constexpr int d = ED - 1;
  LO* pv = r.pv[d];
  LO npairs = 1;
  if (ED == 1) {
    if (lane < 2) {
      LO p = prod0 + lane;
      LO end = vert_offsets[ev2v[e * 2 + lane]];
      pv[std::size_t(p) * 2 + lane] = end;
      pv[std::size_t(p) * 2 + 1 - lane] = mid;
      r.psrc[d][p] = e;
      r.psrc_dim[d][p] = 1;
    }
  } else {
    LO row = r.pairs_a2ab[d][e];
    npairs = r.pairs_a2ab[d][e + 1] - row;
    for (LO i = lane; i < 2 * npairs; i += kRowLanes) {
      LO ed = row + i / 2;
      int eev = i % 2;
      LO dom = r.pairs_ab2b[d][ed];
      I8 code = r.pairs_codes[d][ed];
      int dde = code_which_down(code);
      int dev = eev ^ code_rotation(code);
      int ddv = down_template(ED, 1, dde, dev);
      int dds = opposite_template(ED, 0, ddv);
      LO v[nv];
#pragma unroll
      for (int dsv = 0; dsv < ED; ++dsv)
        v[dsv] = vert_offsets[r.pair_verts[d][std::size_t(dom) * nv +
                                              down_template(ED, ED - 1, dds, dsv)]];
      v[ED] = mid;
      if (ED == 3) {
        LO t = v[1];
        v[1] = v[2];
        v[2] = t;
      }
      LO p = prod0 + i;
#pragma unroll
      for (int k = 0; k < nv; ++k) pv[std::size_t(p) * nv + k] = v[k];
      r.psrc[d][p] = dom;
      r.psrc_dim[d][p] = ED;
    }
  }
  if (ED < 3 && r.cuts_a2ab[d]) {
    constexpr int CD = ED < 3 ? ED + 1 : 3;
    LO row = r.cuts_a2ab[d][e], end = r.cuts_a2ab[d][e + 1];
    for (LO ed = row + lane; ed < end; ed += kRowLanes) {
      LO dom = r.cuts_ab2b[d][ed];
      int dde = code_which_down(r.cuts_codes[d][ed]);
      int ddt = opposite_template(CD, 1, dde);
      LO p = prod0 + 2 * npairs + (ed - row);
      for (int dtv = 0; dtv < CD - 1; ++dtv)
        pv[std::size_t(p) * nv + dtv] =
            vert_offsets[r.cut_verts[d][std::size_t(dom) * (CD + 1) +
                                        down_template(CD, CD - 2, ddt, dtv)]];
      pv[std::size_t(p) * nv + CD - 1] = mid;
      r.psrc[d][p] = dom;
      r.psrc_dim[d][p] = CD;
    }
  }
}

__global__ void refine_products(std::int64_t nt, LO nkeys, LO const* keys2edges,
    LO const* keys2mid, LO const* ev2v, LO const* vert_offsets, RefineRows r) {
  std::int64_t t = thread_index64();
  if (t >= nt) return;
  std::int64_t row = t / kRowLanes;
  int d = int(row / nkeys);
  LO k = LO(row % nkeys);
  int lane = int(t % kRowLanes);
  LO e = keys2edges[k];
  LO mid = keys2mid[k];
  LO prod0 = r.keys2prods[d][k];
  if (d == 0)
    refine_products_of<1>(lane, e, mid, prod0, ev2v, vert_offsets, r);
  else if (d == 1)
    refine_products_of<2>(lane, e, mid, prod0, ev2v, vert_offsets, r);
  else
    refine_products_of<3>(lane, e, mid, prod0, ev2v, vert_offsets, r);
}

// the midpoint vertices' coordinates (the mean of the ends) and metrics (the
// ones their candidates' qualities were measured with)
__global__ void place_midpoints(LO nkeys, int dim, int nc, LO const* keys2edges,
    LO const* keys2mid, LO const* ev2v, Real const* old_coords, LO const* cand_of_edge,
    Real const* midpt_metrics, Real* coords, Real* metric) {
  LO k = thread_index();
  if (k >= nkeys) return;
  LO e = keys2edges[k];
  LO w = keys2mid[k];
  LO cand = cand_of_edge[e];
  for (int j = 0; j < dim; ++j) {
    double comp = 0;
    comp += old_coords[ev2v[e * 2] * dim + j];
    comp += old_coords[ev2v[e * 2 + 1] * dim + j];
    comp /= 2;
    coords[w * dim + j] = comp;
  }
  for (int j = 0; j < nc; ++j)
    metric[std::size_t(w) * nc + j] = midpt_metrics[std::size_t(cand) * nc + j];
}

// the mean of a vertex tag over each key edge's ends
__global__ void midpoint_coords(LO nkeys, int dim, LO const* keys2edges, LO const* ev2v,
    Real const* coords, Real* out) {
  LO k = thread_index();
  if (k >= nkeys) return;
  LO e = keys2edges[k];
  for (int j = 0; j < dim; ++j) {
    double comp = 0;
    comp += coords[ev2v[e * 2] * dim + j];
    comp += coords[ev2v[e * 2 + 1] * dim + j];
    comp /= 2;
    out[k * dim + j] = comp;
  }
}

// the qualities of splitting the candidates over an edge -> element adjacency
// with at least their rows: to `out` (when given), and to `seeds` (when set);
// returns the midpoints' metrics
Reals refine_qualities(Ctx& c, DMesh& m, LOs const& cands, Adj const& e2c,
    RefineSeeds const& seeds, Real* out) {
  Range range(c, "refine_qualities");
  LO n = cands.size();
  int dim = m.dim;
  int nc = m.metric_ncomps;
  int md = (nc == 1) ? 1 : dim;
  Reals mm(c, n * nc);
  mident_metrics(c, m, n, cands.data(), mm.data());
  LOs const& cv2v = verts_of(c, m, dim);
  // lanes share a candidate's children
  int lanes = fit_lanes(n, c.tuning.coarsen_lanes);
  int lshift = lanes_shift(lanes);
#define OSH_RQ(D, M)                                                                    \
  OSH_LAUNCH((refine_qualities_kernel<D, M>), n * lanes, c, lshift, n, cands.data(),       \
      m.down[1].data(), cv2v.data(), e2c.a2ab.data(), e2c.ab2b.data(), e2c.codes.data(),    \
      m.coords.data(), m.metric.data(), mm.data(), out, seeds)
  if (dim == 3 && md == 3)
    OSH_RQ(3, 3);
  else if (dim == 3)
    OSH_RQ(3, 1);
  else if (md == 2)
    OSH_RQ(2, 2);
  else
    OSH_RQ(2, 1);
#undef OSH_RQ
  return mm;
}

}  // namespace

Reals refine_qualities(Ctx& c, DMesh& m, LOs const& cands) {
  Reals out(c, cands.size());
  refine_qualities(c, m, cands, ask_up(c, m, 1, m.dim), RefineSeeds{}, out.data());
  return out;
}

bool refine_by_size(Ctx& c, DMesh& m, AdaptOptions const& o) {
  int dim = m.dim;
  LO ne = m.nents[1];
  Reals const& lengths = ask_lengths(c, m);
  ask_qualities(c, m);
  Bytes cand(c, ne);
  OSH_LAUNCH(gt_kernel, ne, c, lengths.data(), o.max_length_desired, cand.data());
  LOs cand_of_edge;
  LOs cands = collect_marked(c, cand, &cand_of_edge);
  if (cands.size() == 0) return false;
  // the candidates' faces and elements; an attempt with a few long edges left
  // (most of the 64^3 workload's) would otherwise invert the whole mesh
  Adj up[2];
  int const highs[2] = {2, 3};
  bool const sorted[2] = {true, true};
  // every array of the pass that starts out constant, in one launch
  Fills fills(c);
  KeyedMods km;
  km.fixed_prods[0] = 1;
  prepare_keys(m, 1, 0, dim, fills, km);
  LOs up_zeros = fills.ints((dim - 1) * ne, 0);
  LOs side_zeros = fills.ints((dim - 1) * (m.nents[0] + cands.size()), 0);
  Bytes initial = fills.bytes(ne, 0);
  fills.run();
  marked_ups(c, m, 1, cand, dim - 1, highs, sorted, up, &up_zeros);
  Adj const& e2c = up[dim - 2];
  Reals edge_quals(c, ne);  // read where an edge is a candidate
  RefineSeeds seeds{o.min_quality_allowed, initial.data(), edge_quals.data()};
  Reals cand_metrics = refine_qualities(c, m, cands, e2c, seeds, nullptr);
  bool any;
  Bytes keys = find_indset(c, m, 1, edge_quals, initial, &any, &e2c);
  if (!any) return false;
  Range modify_range(c, "modify_ents");
  int nc = m.metric_ncomps;
  DMesh nw;
  nw.dim = dim;
  nw.linked = m.linked;
  nw.metric_ncomps = nc;
  RefineRows rows{};
  for (int d = 1; d <= dim; ++d) {
    if (d > 1) {
      Adj const& pr = up[d - 2];
      rows.pairs_a2ab[d - 1] = pr.a2ab.data();
      rows.pairs_ab2b[d - 1] = pr.ab2b.data();
      rows.pairs_codes[d - 1] = pr.codes.data();
      rows.pair_verts[d - 1] = verts_of(c, m, d).data();
    }
    if (d < dim) {
      Adj const& ct = up[d - 1];
      rows.cuts_a2ab[d - 1] = ct.a2ab.data();
      rows.cuts_ab2b[d - 1] = ct.ab2b.data();
      rows.cuts_codes[d - 1] = ct.codes.data();
      rows.cut_verts[d - 1] = verts_of(c, m, d + 1).data();
    }
    km.prod_counts[d] = LOs(c, ne);
    rows.counts[d - 1] = km.prod_counts[d].data();
  }
  OSH_LAUNCH(prod_counts, ne, c, dim, keys.data(), rows);
  plan_keys(c, m, 1, 0, dim, keys, km);
  LO nkeys = km.nkeys;
  LOs const& keys2edges = km.keys2kds;
  LOs const* k2p = km.k2p;
  LO const* nprods = km.nprods;
  ModPlan const* plans = km.plans;
  for (int d = 1; d <= dim; ++d) rows.keys2prods[d - 1] = k2p[d].data();
  note_changed_parts(c, m, 1, keys2edges);
  if (o.verbosity >= 2) std::printf("refining %d edges\n", int(nkeys));
  ModOut mo[4];
  rebuild_same(c, m, nw, 0, plans, mo);
  Products prods[4];
  prods[0].n = nkeys;
  prods[0].keys2prods = k2p[0];
  prods[0].src_dim = 1;
  place_products(c, m, nw, 0, 0, 0, plans, keys2edges, prods, mo, &km.order);
  LO const* keys2mid = mo[0].prods2new.data();
  OSH_LAUNCH(place_midpoints, nkeys, c, dim, nc, keys2edges.data(), keys2mid,
      m.down[1].data(), m.coords.data(), cand_of_edge.data(), cand_metrics.data(),
      nw.coords.data(), nw.metric.data());
  for (int d = 1; d <= dim; ++d) {
    Products& p = prods[d];
    p.n = nprods[d];
    p.keys2prods = k2p[d];
    p.verts = LOs(c, p.n * (d + 1));
    p.src = LOs(c, p.n);
    p.src_dims = Bytes(c, p.n);
    p.src_dim = d;
    rows.pv[d - 1] = p.verts.data();
    rows.psrc[d - 1] = p.src.data();
    rows.psrc_dim[d - 1] = p.src_dims.data();
  }
  OSH_LAUNCH64(refine_products, std::int64_t(nkeys) * dim * kRowLanes, c, nkeys, keys2edges.data(), keys2mid,
      m.down[1].data(), plans[0].offsets.data(), rows);
  place_products(c, m, nw, 1, dim, 0, plans, keys2edges, prods, mo);
  match_sides(c, nw, prods, mo, &side_zeros);
  measure_products(c, nw, mo);
  for (auto const& t : m.vtags) {
    Reals pt(c, nkeys * t.ncomps);
    if (t.kind == 1)
      mident_values(c, m, nkeys, keys2edges.data(), t.data.data(), t.ncomps, pt.data());
    else
      OSH_LAUNCH(midpoint_coords, nkeys, c, t.ncomps, keys2edges.data(), m.down[1].data(),
          t.data.data(), pt.data());
    nw.vtags.push_back(t.with_data(transfer<Real>(c, mo[0], t.ncomps, t.data, &pt)));
  }
  transfer_elem_tags(c, m, nw, mo[dim], &prods[dim].src);
  conserve_pass(c, m, nw, 0, 1, keys2edges, k2p[dim], mo[dim]);
  m = nw;
  return true;
}

}  // namespace osh
