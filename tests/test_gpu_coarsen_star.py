"""Coarsening around vertices with many edges on the GPU against the oracle, bit
for bit: fans whose hub has just as many edges as a wave or a workgroup takes,
one more, and more than both, in 2D (a disk) and 3D (tets around an axis), with
every hub and rim vertex free to collapse by size."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

A = pytest.importorskip("omega_h_amd")


@pytest.fixture(scope="module")
def ctx():
    return A.Context(0)


def fan(dim, n):
    """n triangles around a point, or n tets around an axis, with another ring
    outside, so that the inner rim is interior too"""
    phi = 2 * np.pi * np.arange(n) / n
    ring = np.stack([np.cos(phi), np.sin(phi)], axis=1)
    i = np.arange(n)
    j = (i + 1) % n
    if dim == 2:
        x = np.concatenate([[[0.0, 0.0]], ring, 2 * ring])
        tris = np.concatenate([np.stack([0 * i, 1 + i, 1 + j], axis=1),
                               np.stack([1 + i, 1 + n + i, 1 + n + j], axis=1),
                               np.stack([1 + i, 1 + n + j, 1 + j], axis=1)])
        return tris, x
    x = np.concatenate([[[0, 0, -0.5], [0, 0, 0.5]], np.pad(ring, ((0, 0), (0, 1)))])
    tets = np.stack([0 * i, 0 * i + 1, 2 + i, 2 + j], axis=1)
    p = x[tets]
    vol = np.linalg.det(p[:, 1:] - p[:, :1])
    tets[vol < 0] = tets[vol < 0][:, [1, 0, 2, 3]]
    return tets, x


def classify(m, dim):
    """boundary entities get class dimension dim - 1, the others dim"""
    sides = m.verts(dim - 1).reshape(-1, dim)
    count = np.bincount(m.down(dim)[0], minlength=len(sides))
    on = [np.zeros(m.nents(d), dtype=bool) for d in range(dim + 1)]
    on[dim - 1] = count == 1
    on[0][sides[on[dim - 1]].ravel()] = True
    if dim == 3:
        on[1][m.down(2)[0].reshape(-1, 3)[on[2]].ravel()] = True
    for d in range(dim + 1):
        m.set_class(d, np.zeros(m.nents(d), dtype=np.int32),
                    np.where(on[d], dim - 1, dim).astype(np.int8))


@pytest.mark.parametrize("improve", [False, True])
@pytest.mark.parametrize("dim,n", [(2, 63), (2, 64), (2, 255), (2, 256), (2, 700), (3, 61),
                                   (3, 62), (3, 127), (3, 128), (3, 129), (3, 254), (3, 255),
                                   (3, 600)])
def test_large_stars_match_oracle(ctx, dim, n, improve):
    elems, x = fan(dim, n)
    g = A.Mesh.from_elems(ctx, dim, elems.astype(np.int32).ravel(), len(x))
    g.set_coords(np.ascontiguousarray(x.ravel()))
    g.set_metric(np.full(len(x), 1.0 / 6.0 ** 2), 1)
    classify(g, dim)
    o = O.Mesh.copy_of(g)
    did = []
    for m, opts in ((o, O.default_opts(dim)), (g, ctx.default_opts(dim))):
        opts.verbosity = 0
        opts.min_quality_allowed = 1e-3
        opts.min_quality_desired = 0.9
        did.append(bool(m.coarsen_slivers(opts) if improve else m.coarsen_by_size(opts)))
    assert did[0] and did[1]
    assert [g.nents(d) for d in range(dim + 1)] == [o.nents(d) for d in range(dim + 1)]
    assert g.digests() == o.digests()
