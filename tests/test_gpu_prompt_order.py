"""The batched prompt products in a GEMV's float order (sml_pp_gemm_*, sml_pp_xgemm_*):
a prompt read at level 1, or in exact mode, equals reading it a token at a
time bit for bit, whatever the tile edges, code widths and row lengths."""
import numpy as np
import pytest

import sheep_amd as sa

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    sa.init(0)


# rows and columns off the 64-row tiles and 64-position tiles; row lengths of
# 12, 16, 36, 48, 68 and 144 groups: part of the 64-lane tree, a ragged last
# superblock, an odd count of 64-group rounds
SHAPES = {
    "384x1152": dict(n_embd=384, n_head=3, n_head_kv=1, n_ff=1152),
    "512x4608": dict(n_embd=512, n_head=4, n_head_kv=2, n_ff=4608),
    "1536x2176": dict(n_embd=1536, n_head=12, n_head_kv=2, n_ff=2176, qkv_bias=True),
}


def logits(path, ids, level, exact, vocab):
    d = sa.Decoder(path, n_ctx=256, exact=exact)
    try:
        d.prompt_mode(level)
        out = [d.prefill(ids, 0, vocab)]
        out.append(d.step(int(np.argmax(out[0])), len(ids), vocab))      # the cache rows too
        return out
    finally:
        d.close()


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("nb,n,exact", [(4, 17, False), (4, 64, False), (4, 65, False), (4, 150, False),
                                        (2, 70, False), (3, 70, False), (5, 70, False), (6, 70, False),
                                        (7, 70, False), (8, 70, False), (4, 5, True), (4, 65, True), (8, 70, True)])
def test_batched_prompt_equals_stepping(tmp_path, monkeypatch, shape, nb, n, exact):
    if exact and SHAPES[shape]["n_ff"] % 256:
        pytest.skip("exact mode batches 256-aligned products")
    monkeypatch.setenv("SML_PX_OUT", "0")                 # every product of more than 16 rows
    p = tmp_path / "m.ssf"
    sa.synth_model(p, n_layer=2, n_vocab=600, nbits=nb, random_perm=True, seed=7 * nb + n, **SHAPES[shape])
    ids = np.random.default_rng(n).integers(0, 600, n).astype(np.int32)
    for a, b in zip(logits(p, ids, 1, exact, 600), logits(p, ids, 0, exact, 600)):
        assert np.abs(b).max() > 0
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("nb", [4, 8])
@pytest.mark.parametrize("n", [33, 512])
def test_exact_prompt_past_a_workgroup_a_cu(tmp_path, nb, n):
    # 512 positions: 288 and 320 tiles, more than the chip's compute units; 33: a workgroup with an empty quarter
    p = tmp_path / "m.ssf"
    sa.synth_model(p, n_layer=1, n_vocab=600, nbits=nb, random_perm=True, seed=nb, n_embd=2304, n_head=18, n_head_kv=6,
                   n_ff=1280)
    ids = np.random.default_rng(n).integers(0, 600, n).astype(np.int32)
    d = sa.Decoder(p, n_ctx=600, exact=True)
    try:
        out = []
        for level in (1, 0):
            d.prompt_mode(level)
            out.append(d.prefill(ids, 0, 600))
    finally:
        d.close()
    assert np.abs(out[0]).max() > 0
    np.testing.assert_array_equal(out[0], out[1])
