"""The searches' quotients by a reciprocal and the re-quantizer's column order
where they can go wrong: values and steps at and past the range that the
reciprocal form admits (both sides of 2^+-60, subnormals, infinities, NaN),
exact ties, every code width, weights and partial codes; equal and NaN column
keys, rows past the LDS and weights and orders that are only 4-byte aligned. All
bit for bit (the quotients are the correctly rounded ones)."""
import numpy as np
import pytest

import sheep_amd as sa
from oracle import bind as ob
from sheep_amd import ingest

pytestmark = pytest.mark.gpu


def _groups(rng, cols):
    """Rows of one kind each: (name, row)."""
    n = rng.standard_normal(cols).astype(np.float32)
    k = rng.integers(0, 16, cols).astype(np.float32)
    out = [("normal", n), ("ties", (k + np.float32(0.5)) * np.float32(0.125)), ("levels", k * np.float32(0.1)),
           ("zero", n * 0), ("const", n * 0 + np.float32(0.3)), ("outlier", np.where(rng.random(cols) < 0.05, n * 1000, n))]
    for e in (-149, -130, -70, -61, -60, -59, -40, 40, 57, 58, 59, 60, 61, 100, 125):
        out.append((f"2^{e}", np.ldexp(n, e).astype(np.float32)))
    return out


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("nbits,rem", [(1, 0), (2, 0), (4, 0), (4, 2), (8, 0), (8, 4), (9, 0), (12, 3), (16, 0)])
def test_grid_search_over_the_range_of_the_quotients(nbits, rem, weighted):
    rng = np.random.default_rng(nbits * 10 + rem)
    cols = 1024
    names, w = zip(*_groups(rng, cols))
    w = np.ascontiguousarray(np.stack(w))
    wt = (rng.random(cols).astype(np.float32) + np.float32(0.1)) if weighted else None
    print(f"grid {nbits} bits rem {rem} weighted {weighted}", flush=True)
    for refit in (0, 1):
        lg, sg = ob.asym_grid(w, 32, nbits, wt, rem=rem, refit=refit, lib=ingest._lib())
        lr, sr = ob.asym_grid(w, 32, nbits, wt, rem=rem, refit=refit)
        for i, name in enumerate(names):
            assert np.array_equal(lg[i], lr[i], equal_nan=True) and np.array_equal(sg[i], sr[i], equal_nan=True), name


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_grid_search_leaves_other_groups_alone(bad):
    # one lane's infinity or NaN sends its wave to the plain division: the
    # other groups' results stay what they are without it
    rng = np.random.default_rng(5)
    w = rng.standard_normal((4, 4096)).astype(np.float32)
    l0, s0 = ob.asym_grid(w, 32, 4, lib=ingest._lib())
    v = w.copy()
    v[1, 70] = bad
    l1, s1 = ob.asym_grid(v, 32, 4, lib=ingest._lib())
    keep = np.ones(l0.shape, bool)
    keep[1, 2] = False
    assert np.array_equal(l0[keep], l1[keep]) and np.array_equal(s0[keep], s1[keep])


@pytest.mark.parametrize("nmax", [3, 15, 255])
def test_field_search_over_the_range_of_the_quotients(nmax):
    rng = np.random.default_rng(nmax)
    cols = 1024
    names, w = zip(*_groups(rng, cols))
    w = np.ascontiguousarray(np.stack(w))
    rows, ng = len(names), cols // 32
    amp = np.abs(w).max(axis=1, keepdims=True)
    dv = np.broadcast_to(np.maximum(amp / np.float32(255 * nmax), np.float32(1e-38)), (rows, ng)).astype(np.float32)
    dm = np.broadcast_to(amp / np.float32(127), (rows, ng)).astype(np.float32)
    q8 = rng.integers(1, 256, (rows, ng)).astype(np.int32)
    mq8 = rng.integers(0, 255, (rows, ng)).astype(np.int32)
    print(f"field nmax {nmax}", flush=True)
    for radius in (0, 2):
        a = ob.field_search(w, dv, dm, q8, mq8, 32, nmax, radius=radius, lib=ingest._lib())
        b = ob.field_search(w, dv, dm, q8, mq8, 32, nmax, radius=radius)
        for i, name in enumerate(names):
            assert np.array_equal(a[0][i], b[0][i]) and np.array_equal(a[1][i], b[1][i]), name


@pytest.mark.parametrize("cols", [256, 768, 4352, 40960, 41216])
def test_column_order(cols):
    # equal maxima (stable order), zero and NaN columns, rows in and past the LDS
    rng = np.random.default_rng(cols)
    w = rng.integers(-6, 7, (3, cols)).astype(np.float32) * np.float32(0.01)
    w[:, cols // 3] = 0.0
    w[1, [5, cols // 2, cols - 1]] = np.nan
    res = ingest.requantize(w, 4)
    want = np.argsort(np.abs(w).max(axis=0), kind="stable")
    assert np.array_equal(res.host()["perm"], want)
    w = np.nan_to_num(w)
    res = ingest.requantize(w, 4, keep_codes=True)
    ref = ob.requant(w, 4)
    h = res.host()
    for k in ("perm", "sd", "sq", "md", "mq", "codes"):
        assert np.array_equal(h[k], ref[k]), k


@pytest.mark.parametrize("given", [False, True])
@pytest.mark.parametrize("cols", [768, 41216])
def test_column_order_of_unaligned_arrays(cols, given):
    # the weights, the order asked for and the order written 4 bytes past a
    # 16-byte boundary: what the aligned call gives, in and past the LDS
    rng = np.random.default_rng(cols)
    rows, nbits = 3, 4
    w = (rng.standard_normal((rows, cols)) * 0.02).astype(np.float32)
    order = rng.permutation(cols).astype(np.int32) if given else None
    got = []
    for off in (0, 4):
        wd = sa.DevBuf(w.nbytes + 16)
        assert sa.lib().sml_hip_h2d(wd.ptr + off, w.ctypes.data, w.nbytes) == 0
        od = None
        if given:
            od = sa.DevBuf(order.nbytes + 16)
            assert sa.lib().sml_hip_h2d(od.ptr + off, order.ctypes.data, order.nbytes) == 0
        r = ingest.Requantized(rows, cols, nbits, True)
        perm = sa.DevBuf(cols * 4 + 16)
        assert ingest._lib().sml_hip_requant(wd.ptr + off, rows, cols, nbits, od.ptr + off if given else None, None, 2,
                                             r._pl(), r.sd.ptr, r.sq.ptr, r.md.ptr, r.mq.ptr, perm.ptr + off,
                                             r.codes.ptr) == 0, sa.lib().sml_hip_last_error()
        h = r.host()
        h["perm"] = perm.read(np.uint8)[off:off + cols * 4].copy().view(np.int32)
        got.append(h)
    if given:
        assert np.array_equal(got[1]["perm"], order)
    for k in ("perm", "sd", "sq", "md", "mq", "codes"):
        assert np.array_equal(got[0][k], got[1][k]), k
    assert all(np.array_equal(a, b) for a, b in zip(got[0]["planes"], got[1]["planes"]))
