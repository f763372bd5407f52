"""The batched single-pass offset scan (offset_scan, src/Omega_h_int_scan.cpp:10-20)
against numpy's running sums, through the C ABI on device pointers.

Sizes cover empty arrays, one partial tile, the 4096-value tile boundary and
scans of hundreds to thousands of tiles, alone and mixed in one launch, so the
look-back crosses windows of 64 tiles and each job's look-back stays inside
its own tiles.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A = pytest.importorskip("omega_h_amd")


@pytest.fixture(scope="module")
def ctx():
    return A.Context(0)


def run_scans(ctx, arrays):
    from omega_h_amd.hip import DeviceArray
    ins = [DeviceArray(a) for a in arrays]
    outs = [DeviceArray(dtype=np.int32, n=len(a) + 1) for a in arrays]
    ctx.offset_scans([d.ptr for d in ins], [len(a) for a in arrays], [d.ptr for d in outs])
    ctx.synchronize()
    return [o.numpy() for o in outs]


def expected(a):
    return np.concatenate([[0], np.cumsum(a, dtype=np.int64)]).astype(np.int32)


@pytest.mark.parametrize("n", [0, 1, 17, 4095, 4096, 4097, 8192, 100_003, 262_144 + 5,
                               3_000_000, 12_000_000])
def test_single_scan(ctx, n):
    rng = np.random.default_rng(n)
    a = rng.integers(0, 8, size=n, dtype=np.int32)
    (got,) = run_scans(ctx, [a])
    assert np.array_equal(got, expected(a)), n


@pytest.mark.parametrize("n", [1023, 1024, 1025, 16383, 16384, 16385, 20479, 20480, 16 * 4096,
                               16 * 4096 + 1, 8192 * 2048, 8192 * 2048 + 1])
def test_sizes_at_the_edges_of_tiles_and_launch_forms(ctx, n):
    """One tile of 1024, 4096 or 16384 values, the 4096-value tiles of the one-launch form and
    its largest job, and the largest job of the two-launch form."""
    a = np.random.default_rng(n).integers(0, 8, size=n, dtype=np.int32)
    (got,) = run_scans(ctx, [a])
    assert np.array_equal(got, expected(a)), n


@pytest.mark.parametrize("shift", [1, 2, 3])
@pytest.mark.parametrize("n", [5, 16384, 40_001, 300_001])
def test_arrays_at_any_word(ctx, n, shift):
    """Arrays that don't start at a 16-byte boundary."""
    from omega_h_amd.hip import DeviceArray
    a = np.random.default_rng(n).integers(0, 8, size=n + shift, dtype=np.int32)
    d = DeviceArray(a)
    for in_shift, out_shift in ((shift, 0), (0, shift), (shift, shift)):
        o = DeviceArray(np.full(n + 1 + shift, -7, dtype=np.int32))
        ctx.offset_scans([d.ptr + 4 * in_shift], [n], [o.ptr + 4 * out_shift])
        ctx.synchronize()
        got = o.numpy()
        assert np.array_equal(got[out_shift:out_shift + n + 1],
                              expected(a[in_shift:in_shift + n]))
        assert np.all(got[:out_shift] == -7) and np.all(got[out_shift + n + 1:] == -7)


def test_batched_scans_in_one_launch(ctx):
    rng = np.random.default_rng(7)
    for sizes in ([5, 0, 4096, 1], [300_000, 17, 1_000_000, 4097], [2_500_000, 2_500_000],
                  [0, 0, 0], [1000, 5000, 0, 70_000, 4096, 3, 250_000, 9000],
                  [7, 300_000, 0, 4096, 50_000, 1, 200_000, 4097, 12, 100_000, 0, 65_536]):
        arrays = [rng.integers(0, 5, size=n, dtype=np.int32) for n in sizes]
        got = run_scans(ctx, arrays)
        for a, g in zip(arrays, got):
            assert np.array_equal(g, expected(a)), sizes


def test_repeated_scans_keep_the_status_words_apart(ctx):
    # consecutive launches reuse the status words under new epochs
    rng = np.random.default_rng(11)
    for k in range(20):
        a = rng.integers(-3, 4, size=int(rng.integers(1, 600_000)), dtype=np.int32)
        (got,) = run_scans(ctx, [a])
        assert np.array_equal(got, expected(a)), k


def test_bad_scan_arguments_are_refused(ctx):
    from omega_h_amd.hip import DeviceArray
    a = DeviceArray(np.ones(4, np.int32))
    o = DeviceArray(dtype=np.int32, n=5)
    with pytest.raises(A.OshError):
        ctx.offset_scans([a.ptr] * 13, [4] * 13, [o.ptr] * 13)
    with pytest.raises(A.OshError):
        ctx.offset_scans([a.ptr], [-1], [o.ptr])
