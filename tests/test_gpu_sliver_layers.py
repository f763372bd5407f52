"""adapt() with few and many sliver layers on the GPU against the oracle, bit for
bit: none, the first, the longest that the side counts of a linked mesh hold,
one more, and across the eight buffers of the general form."""
import pytest

import oracle_lib as O
from test_oracle_coarsen_flip import jittered_box

pytestmark = pytest.mark.gpu

A = pytest.importorskip("omega_h_amd")


@pytest.fixture(scope="module")
def ctx():
    return A.Context(0)


@pytest.mark.parametrize("layers", [0, 1, 2, 9, 16, 17])
@pytest.mark.parametrize("dim,n,jitter,h", [(2, 14, 0.45, 0.12), (3, 6, 0.45, 0.3)])
def test_layers_match_oracle(ctx, dim, n, jitter, h, layers):
    meshes = []
    for lib, kw in ((O, {}), (A, {"ctx": ctx})):
        m = jittered_box(lib, dim, n, jitter, h, 3, **kw)
        opts = O.default_opts(dim) if lib is O else ctx.default_opts(dim)
        opts.verbosity = 0
        opts.nsliver_layers = layers
        m.adapt(opts)
        meshes.append(m)
    o, g = meshes
    assert [g.nents(d) for d in range(dim + 1)] == [o.nents(d) for d in range(dim + 1)]
    assert g.digests() == o.digests()
