"""The prompt GEMM's superblock sums (sml_pp_sgemm_*): the whole integer sums on
the matrix cores, at the edges of its tiles and of the integers' range, against
a 64-bit product of the same codes and fields."""
import numpy as np
import pytest

import sheep_amd as sa

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    sa.init(0)


def nibbles(c):
    c = c.reshape(c.shape[0], -1, 4, 32)
    return np.ascontiguousarray(np.stack([c[:, :, 0] | c[:, :, 1] << 4, c[:, :, 2] | c[:, :, 3] << 4], 2))


def matrix(rng, rows, cols, nb, extreme):
    """Codes and fields of a matrix: its handle and its weights in 64 bits."""
    ng, ns, top = cols // 32, cols // 256, (1 << nb) - 1
    codes = np.full((rows, cols), top, np.uint8) if extreme else rng.integers(0, top + 1, (rows, cols)).astype(np.uint8)
    sq = np.full((rows, ng), 255, np.uint8) if extreme else rng.integers(0, 256, (rows, ng)).astype(np.uint8)
    mq = rng.choice([0, 255], (rows, ng)).astype(np.uint8) if extreme else rng.integers(0, 256, (rows, ng)).astype(np.uint8)
    sd, md = (rng.uniform(0.5, 2, (rows, ns)).astype(np.float16) for _ in range(2))
    planes = [nibbles(codes & 15)]
    if nb == 6:
        h = (codes >> 4).reshape(rows, -1, 4, 32)
        planes.insert(0, np.ascontiguousarray(h[:, :, 0] | h[:, :, 1] << 2 | h[:, :, 2] << 4 | h[:, :, 3] << 6))
    ptrs = (sa.c_void_p * 4)(*([p.ctypes.data for p in planes] + [None] * (4 - len(planes))))
    m = sa.Mat(sa.lib().sml_hip_mat_upload(ptrs, sd.ctypes.data, sq.ctypes.data, md.ctypes.data, mq.ctypes.data,
                                           rows, cols, nb, 0, 0))
    sup = np.arange(ng) // 8
    step, low = sd.astype(np.float64)[:, sup] * sq, md.astype(np.float64)[:, sup] * (mq.astype(np.float64) - 127)
    return m, (codes.reshape(rows, ng, 32) * step[:, :, None] + low[:, :, None]).reshape(rows, cols)


def acts(rng, npos, cols, extreme):
    q = (rng.choice([-127, 127], (npos, 1)) * np.ones((1, cols), int) if extreme
         else rng.integers(-127, 128, (npos, cols))).astype(np.int8)
    s = rng.uniform(0.01, 0.02, (npos, cols // 256)).astype(np.float32)
    u = q.reshape(npos, -1, 32).sum(-1, dtype=np.int32)
    dense = q.astype(np.float64) * np.repeat(s, 256, 1)
    bufs = [sa.DevBuf.of(np.ascontiguousarray(x)) for x in (q, np.repeat(s, 8, 1), u)]
    return bufs, dense


@pytest.mark.parametrize("nb", [4, 6])
@pytest.mark.parametrize("rows,cols,npos,extreme", [(1, 256, 17, False), (63, 512, 64, False), (130, 1536, 65, False),
                                                    (257, 768, 129, False), (64, 2048, 200, True)])
def test_sums_at_the_edges(monkeypatch, nb, rows, cols, npos, extreme):
    rng = np.random.default_rng(1000 * nb + rows + npos)
    gate, gw = matrix(rng, rows, cols, nb, extreme)
    up, uw = matrix(rng, rows, cols, nb, extreme)
    (q, s, u), a = acts(rng, npos, cols, extreme)
    got = {}
    for p in ("2", "4", "6", "8"):            # 32 to 128 positions a workgroup
        monkeypatch.setenv("SML_PS_P", p)
        y, h = sa.DevBuf(npos * rows * 4), sa.DevBuf(npos * rows * 4)
        sa.gemm(gate, q, s, u, npos, y, per256=True)
        sa.gemm_swiglu(gate, up, q, s, u, npos, h, per256=True)
        got[p] = [b.read(np.float32).reshape(npos, rows) for b in (y, h)]
    for p in ("2", "6", "8"):
        for x, z in zip(got["4"], got[p]):
            np.testing.assert_array_equal(x, z)
    # each superblock's two products and sums round once: cols / 256 * 4
    # roundings of 2^-24, of terms up to the sum of the magnitudes
    want = a @ gw.T
    mag = np.abs(a) @ np.abs(gw).T
    assert np.all(np.abs(got["4"][0] - want) <= (cols // 256 * 4 + 4) * 2.0 ** -24 * mag)
    g, v = want, a @ uw.T
    hw = g / (1 + np.exp(-np.clip(g, -80, 80))) * v
    np.testing.assert_allclose(got["4"][1], hw, rtol=1e-3, atol=2e-4 * np.abs(hw).max())
