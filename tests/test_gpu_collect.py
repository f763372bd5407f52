"""collect_marked against numpy on both sides of every line between the forms of
the scan that counts and lists the marks: one tile of 1024, 4096 or 16384 values,
16 tiles whose earlier values each workgroup adds up, two launches, and the
look-back beyond 8192 tiles of 2048."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A = pytest.importorskip("omega_h_amd")


@pytest.fixture(scope="module")
def ctx():
    return A.Context(0)


@pytest.mark.parametrize("share", [0.0, 0.3, 1.0])
@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 4096, 4097, 16384, 16385, 65535, 65536,
                               65537, 8192 * 2048 - 3, 8192 * 2048, 8192 * 2048 + 1, 20_000_001])
def test_marks_of_every_scan_form(ctx, n, share):
    rng = np.random.default_rng(n)
    # any nonzero byte is a mark
    marks = np.where(rng.random(n, dtype=np.float32) < share,
                     rng.choice(np.array([1, -1, 5, -128, 127], dtype=np.int8), size=n), 0)
    print(f"collect n={n} share={share}", flush=True)
    assert np.array_equal(ctx.collect_marked(marks.astype(np.int8)), np.flatnonzero(marks))
