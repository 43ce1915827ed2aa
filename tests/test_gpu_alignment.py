"""Buffers at addresses that the copies into LDS do not take: activation codes
and K/V caches off 16-byte boundaries run on the kernels that load them through
registers, and compute what the aligned calls compute to the rounding of the
sums."""
import numpy as np
import pytest

import sheep_amd as sa

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    sa.init(0)


class At:
    """An array on the device `off` bytes past an allocation's start."""

    def __init__(self, arr, off):
        raw = np.zeros(off + arr.nbytes, np.uint8)
        raw[off:] = np.ascontiguousarray(arr).view(np.uint8).reshape(-1)
        self.buf, self.off, self.shape, self.dtype = sa.DevBuf.of(raw), off, arr.shape, arr.dtype
        self.ptr = self.buf.ptr + off

    def read(self):
        return self.buf.read(np.uint8)[self.off:].copy().view(self.dtype).reshape(self.shape)


def matrix(rng, rows, cols, nb):
    planes = [rng.integers(0, 256, rows * cols * b // 8, dtype=np.uint8) for b in ([4] if nb == 4 else [2, 4])]
    sq, mq = (rng.integers(0, 256, (rows, cols // 32)).astype(np.uint8) for _ in range(2))
    sd, md = (rng.uniform(0.5, 2, (rows, cols // 256)).astype(np.float16) for _ in range(2))
    ptrs = (sa.c_void_p * 4)(*([p.ctypes.data for p in planes] + [None] * (4 - len(planes))))
    m = sa.Mat(sa.lib().sml_hip_mat_upload(ptrs, sd.ctypes.data, sq.ctypes.data, md.ctypes.data, mq.ctypes.data,
                                           rows, cols, nb, 0, 0))
    # no weight is larger than its superblock's largest step and min allow
    big = np.repeat(sd.astype(np.float64) * 255 * ((1 << nb) - 1) + md.astype(np.float64) * 128, 256, 1)
    return m, big


@pytest.mark.parametrize("nb", [4, 6])
@pytest.mark.parametrize("off", [4, 8])
@pytest.mark.parametrize("npos", [17, 70])
def test_codes_off_the_copy_alignment(nb, off, npos):
    rng = np.random.default_rng(nb * npos)
    rows, cols = 130, 1536
    (g, big), (u, _) = matrix(rng, rows, cols, nb), matrix(rng, rows, cols, nb)
    q = rng.integers(-127, 128, (npos, cols)).astype(np.int8)
    s = np.repeat(rng.uniform(0.01, 0.02, (npos, cols // 256)).astype(np.float32), 8, 1)
    sums = q.reshape(npos, -1, 32).sum(-1, dtype=np.int32)
    scale, sm = sa.DevBuf.of(s), sa.DevBuf.of(sums)
    got = []
    for o in (0, off):
        qd = At(q, o)
        y, h = sa.DevBuf(npos * rows * 4), sa.DevBuf(npos * rows * 4)
        sa.gemm(g, qd, scale, sm, npos, y, per256=True)
        sa.gemm_swiglu(g, u, qd, scale, sm, npos, h, per256=True)
        got.append([b.read(np.float32).reshape(npos, rows) for b in (y, h)])
    # each side rounds a superblock's two products and sums once, and adds
    # partial sums of up to 8 waves: cols / 256 * 4 + 8 roundings of 2^-24
    mag = (np.abs(q.astype(np.float64)) * np.repeat(s, 32, 1)) @ big.T
    assert np.abs(got[0][0]).max() > 0
    assert np.all(np.abs(got[0][0] - got[1][0]) <= 2 * (cols // 256 * 4 + 8) * 2.0 ** -24 * mag)
    np.testing.assert_allclose(got[1][1], got[0][1], rtol=1e-3, atol=2e-4 * np.abs(got[0][1]).max())


@pytest.mark.parametrize("off", [4, 8])
@pytest.mark.parametrize("heads,kv,n,pos0", [(8, 2, 17, 0), (12, 2, 43, 300)])
def test_caches_off_the_copy_alignment(off, heads, kv, n, pos0):
    rng = np.random.default_rng(n)
    n_ctx = 512
    ang = np.arange(n_ctx)[:, None] * (1e4 ** (-np.arange(64) / 64.0))
    cos, sin = (sa.DevBuf.of(f(ang).astype(np.float32)) for f in (np.cos, np.sin))
    qkv = rng.standard_normal((n, (heads + 2 * kv) * 128)).astype(np.float32)
    kc, vc = (rng.standard_normal((n_ctx, kv * 128)).astype(np.float16) for _ in range(2))
    qd, part = sa.DevBuf.of(qkv), sa.DevBuf(n * heads * 4 * 130 * 4)
    got = []
    for ko, vo in ((0, 0), (off, 0), (0, off)):
        k, v, out = At(kc, ko), At(vc, vo), sa.DevBuf(n * heads * 128 * 4)
        assert sa.lib().sml_hip_attention_prompt(qd.ptr, n, pos0, k.ptr, v.ptr, cos.ptr, sin.ptr, heads, kv, 128, n_ctx,
                                                 part.ptr, out.ptr) == 0, sa.lib().sml_hip_last_error()
        got.append((out.read(np.float32), k.read(), v.read()))
    # scores below 16 here; both forms within (8 + 16) 2^-20 of the largest |V|
    # (the bound of the flash form's own test against float64)
    tol = 2 * 24 * 2.0 ** -20 * np.abs(got[0][2].astype(np.float32)).max()
    for o, k, v in got[1:]:
        assert np.abs(o - got[0][0]).max() <= tol
        np.testing.assert_array_equal(k, got[0][1])
        np.testing.assert_array_equal(v, got[0][2])


@pytest.mark.parametrize("heads,kv,splits", [(3, 1, 3), (5, 5, 3), (7, 1, 4), (1, 1, 1)])
def test_merge_of_odd_splits_into_any_output(monkeypatch, heads, kv, splits):
    # an odd product of heads and splits puts every second row's partials, and
    # the offset the output, on 8- and 4-byte boundaries
    monkeypatch.setenv("SML_PF_NS", str(splits))
    rng = np.random.default_rng(heads)
    n, pos0, n_ctx = 43, 300, 512
    ang = np.arange(n_ctx)[:, None] * (1e4 ** (-np.arange(64) / 64.0))
    cos, sin = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)
    qkv = rng.standard_normal((n, (heads + 2 * kv) * 128)).astype(np.float32)
    kc, vc = (rng.standard_normal((n_ctx, kv * 128)).astype(np.float16) for _ in range(2))
    d = [sa.DevBuf.of(x) for x in (qkv, kc.view(np.uint16), vc.view(np.uint16), cos, sin)]
    got = []
    for off in (0, 4):
        part, out = sa.DevBuf(n * heads * 4 * 130 * 4), At(np.zeros((n, heads, 128), np.float32), off)
        assert sa.lib().sml_hip_attention_prompt(d[0].ptr, n, pos0, d[1].ptr, d[2].ptr, d[3].ptr, d[4].ptr, heads, kv,
                                                 128, n_ctx, part.ptr, out.ptr) == 0, sa.lib().sml_hip_last_error()
        got.append(out.read())
    np.testing.assert_array_equal(got[0], got[1])
    K, V = (d[i].read(np.uint16).view(np.float16).reshape(n_ctx, kv, 128).astype(np.float64) for i in (1, 2))
    p, rep = np.arange(pos0, pos0 + n), heads // kv
    q = qkv[:, :heads * 128].reshape(n, heads, 128).astype(np.float64)
    c, s = cos[p, None].astype(np.float64), sin[p, None].astype(np.float64)
    q = np.concatenate([q[..., :64] * c - q[..., 64:] * s, q[..., :64] * s + q[..., 64:] * c], -1)
    for h in range(heads):
        x = q[:, h] @ K[:pos0 + n, h // rep].T / np.sqrt(128.0)
        big = np.abs(x).max()
        x[np.arange(pos0 + n)[None] > p[:, None]] = -np.inf
        w = np.exp(x - x.max(1, keepdims=True))
        want = (w / w.sum(1, keepdims=True)) @ V[:pos0 + n, h // rep]
        assert np.abs(got[0][:, h] - want).max() <= (8.0 + big) * 2.0 ** -20 * np.abs(V).max(), h
