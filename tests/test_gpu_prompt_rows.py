"""Prompt rows: the matrix-core attention (sml_pp_flash, sml_pp_merge) against
float64 at the edges of its 128-row tiles, 64-position blocks and splits, over
scores whose maximum climbs, falls or stays far below zero; and the
row-a-workgroup normalization + quantization (sml_pp_normq, many rows)
against the form that fewer rows take, bit for bit; and the level-1 prompt's
attention (sml_pp_attn, and the decode kernel for few entries) against
decoding, bit for bit."""
import numpy as np
import pytest

import sheep_amd as sa

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    sa.init(0)


def _rotate(x, cos, sin):
    lo, hi = x[..., :64], x[..., 64:]
    return np.concatenate([lo * cos - hi * sin, lo * sin + hi * cos], -1)


@pytest.mark.parametrize("kind", ["flat", "climbing", "falling", "low"])
@pytest.mark.parametrize("heads,kv,n,pos0,n_ctx", [(1, 1, 1, 0, 128), (8, 8, 129, 0, 256), (3, 1, 43, 21, 128),
                                                   (8, 1, 17, 495, 512), (14, 2, 63, 1, 256), (32, 8, 33, 2015, 2048),
                                                   (5, 5, 300, 700, 1024)])
def test_flash_rows_against_float64(heads, kv, n, pos0, n_ctx, kind):
    rng = np.random.default_rng(n * 31 + pos0)
    T, rep = pos0 + n, heads // kv
    ang = np.arange(n_ctx)[:, None] * (1e4 ** (-np.arange(64) / 64.0))
    cos, sin = np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)
    qkv = rng.standard_normal((n, (heads + 2 * kv) * 128)).astype(np.float32)
    kc = rng.standard_normal((n_ctx, kv, 128)).astype(np.float16)
    vc = rng.standard_normal((n_ctx, kv, 128)).astype(np.float16)
    # the keys' weight along the positions, so that a row's running max moves (or not)
    g = {"flat": np.ones(n_ctx), "climbing": np.linspace(0, 6, n_ctx), "falling": np.linspace(6, 0, n_ctx),
         "low": np.full(n_ctx, 4.0)}[kind].astype(np.float32)
    kc = (kc * g[:, None, None]).astype(np.float16)
    if kind == "low":                                     # every score far below zero
        kc[:] = (4.0 * np.sign(rng.standard_normal(128))).astype(np.float16)
        qkv[:, :heads * 128] = 0.0
    d = [sa.DevBuf.of(np.ascontiguousarray(x)) for x in (qkv, kc.view(np.uint16), vc.view(np.uint16), cos, sin)]
    part = sa.DevBuf(n * heads * ((n_ctx + 127) // 128) * 130 * 4)
    out = sa.DevBuf(n * heads * 128 * 4)
    print(f"flash {heads}/{kv} rows {n} at {pos0} {kind}", flush=True)
    assert sa.lib().sml_hip_attention_prompt(d[0].ptr, n, pos0, d[1].ptr, d[2].ptr, d[3].ptr, d[4].ptr, heads, kv, 128,
                                             n_ctx, part.ptr, out.ptr) == 0, sa.lib().sml_hip_last_error()
    got = out.read(np.float32).reshape(n, heads, 128)
    K = d[1].read(np.uint16).view(np.float16).reshape(n_ctx, kv, 128).astype(np.float64)
    V = d[2].read(np.uint16).view(np.float16).reshape(n_ctx, kv, 128).astype(np.float64)
    p = np.arange(pos0, T)
    q = _rotate(qkv[:, :heads * 128].reshape(n, heads, 128).astype(np.float64), cos[p, None].astype(np.float64),
                sin[p, None].astype(np.float64))
    S = 0.0
    for h in range(heads):
        s = q[:, h] @ K[:T, h // rep].T / np.sqrt(128.0)
        s[np.arange(T)[None] > p[:, None]] = -np.inf
        S = max(S, np.abs(s[np.isfinite(s)]).max())
        w = np.exp(s - s.max(1, keepdims=True))
        want = (w / w.sum(1, keepdims=True)) @ V[:T, h // rep]
        # a score is off by the parts of q (2^-22) and 128 float32 sums of
        # random sign (about 2^-21 of its terms); a weight by that and its
        # own two parts (2^-21); both move the output by their share of max |V|
        assert np.abs(got[:, h] - want).max() <= (8.0 + S) * 2.0 ** -20 * np.abs(V[:T]).max(), h


def _read(path, cuts, ids, level, exact, vocab):
    d = sa.Decoder(path, n_ctx=512, exact=exact)
    try:
        d.prompt_mode(level)
        for a, b in zip(cuts, cuts[1:]):
            out = d.prefill(ids[a:b], a, vocab)
        return out, d.step(int(np.argmax(out)), len(ids), vocab)
    finally:
        d.close()


@pytest.mark.parametrize("level,exact", [(1, False), (1, True), (2, False)])
@pytest.mark.parametrize("n_embd,n_head,kv,n_ff", [(384, 3, 1, 1280), (1024, 8, 1, 1152), (2304, 18, 6, 2304)])
@pytest.mark.parametrize("perm,n", [(True, 200), (False, 300)])
def test_many_rows_quantize_as_few(tmp_path, monkeypatch, n_embd, n_head, kv, n_ff, level, exact, perm, n):
    # 192 (permuted) and 256 rows and more in one read against reads of half:
    # the products and the wave-per-position attention do not depend on the cut
    if exact and (n_ff % 256 or n_embd % 256):
        pytest.skip("exact mode batches 256-aligned products")
    monkeypatch.setenv("SML_ATTN_FLASH", "0")
    monkeypatch.setenv("SML_PX_OUT", "0")
    p = tmp_path / "m.ssf"
    sa.synth_model(p, n_layer=2, n_vocab=600, nbits=4, random_perm=perm, seed=n_embd, n_embd=n_embd, n_head=n_head,
                   n_head_kv=kv, n_ff=n_ff)
    ids = np.random.default_rng(n_ff).integers(0, 600, n).astype(np.int32)
    a = _read(p, [0, n], ids, level, exact, 600)
    b = _read(p, [0, n // 2, n], ids, level, exact, 600)
    assert np.abs(a[0]).max() > 0
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("few", ["0", ""])                # a wave per entry; few entries: a workgroup each
@pytest.mark.parametrize("chunk", [128, 64, 32])
@pytest.mark.parametrize("heads,kv,n", [(1, 1, 18), (4, 2, 129), (3, 1, 140), (4, 1, 131), (5, 1, 80), (12, 2, 65),
                                        (7, 1, 64), (8, 1, 150)])
def test_level_1_attention_equals_decoding(tmp_path, monkeypatch, heads, kv, n, chunk, few):
    # every head grouping, splits of each size, entries ending in, at and past
    # a split; two cuts, so that the second reads what the first wrote
    monkeypatch.setenv("SML_ATTN_CHUNK", str(chunk))
    monkeypatch.setenv("SML_ATTN_FEW", few)
    p = tmp_path / "m.ssf"
    sa.synth_model(p, n_layer=2, n_vocab=600, nbits=4, random_perm=True, seed=heads, n_embd=128 * heads, n_head=heads,
                   n_head_kv=kv, n_ff=512)
    ids = np.random.default_rng(n).integers(0, 600, n).astype(np.int32)
    a = _read(p, [0, n], ids, 1, False, 600)
    b = _read(p, [0, n // 3, n], ids, 1, False, 600)
    c = _read(p, [0, n], ids, 0, False, 600)
    assert np.abs(c[0]).max() > 0
    for x, y, z in zip(a, b, c):
        np.testing.assert_array_equal(x, z)
        np.testing.assert_array_equal(y, z)
