"""Prompts read in several pieces equal reading them a token at a time, bit for
bit: the level-1 attention in slices of rows whose partials fit their buffer
(heads in order, where the slices quantize their outputs, and permuted), and
chunks of 64 positions at level 1 and in exact mode."""
import numpy as np
import pytest

import sheep_amd as sa

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def device():
    sa.init(0)


def read(path, ids, n_ctx, level, exact=False):
    d = sa.Decoder(path, n_ctx=n_ctx, exact=exact)
    try:
        d.prompt_mode(level)
        out = [d.prefill(ids, 0, 600)]
        out.append(d.step(int(np.argmax(out[0])), len(ids), 600))        # the cache rows too
        return out
    finally:
        d.close()


def same(path, n, n_ctx, exact=False):
    ids = np.random.default_rng(n).integers(0, 600, n).astype(np.int32)
    for a, b in zip(read(path, ids, n_ctx, 1, exact), read(path, ids, n_ctx, 0, exact)):
        assert np.abs(b).max() > 0
        np.testing.assert_array_equal(a, b)


# One kv head: splits of 64 positions, while the buffer holds a row's partials at
# splits of 128 for every position of a chunk: slices of 64 + 56, 64 + 1 and
# 256 + 244 rows. In order up to 512 inputs only: stepping such a model sums
# wider gate and up products over 16 lanes a row.
@pytest.mark.parametrize("heads,n_ctx,n,perm", [(4, 128, 120, False), (4, 128, 65, False), (3, 512, 500, False),
                                                (8, 128, 120, True), (3, 512, 500, True)])
@pytest.mark.parametrize("few", ["0", ""])                # a wave per entry; few entries: a workgroup each
def test_level_1_slices_equal_stepping(tmp_path, monkeypatch, heads, n_ctx, n, perm, few):
    monkeypatch.setenv("SML_ATTN_FEW", few)
    p = tmp_path / "m.ssf"
    sa.synth_model(p, n_layer=2, n_vocab=600, nbits=4, random_perm=perm, seed=n, n_embd=128 * heads, n_head=heads,
                   n_head_kv=1, n_ff=512)
    same(p, n, n_ctx)


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("nb,n", [(4, 64), (4, 130), (8, 130)])
def test_chunk_boundaries_equal_stepping(tmp_path, monkeypatch, nb, n, exact):
    monkeypatch.setenv("SML_PB", "64")                    # 130: chunks of 64, 64 and 2
    p = tmp_path / "m.ssf"
    sa.synth_model(p, n_layer=2, n_vocab=600, nbits=nb, random_perm=True, seed=nb, n_embd=512, n_head=4, n_head_kv=2,
                   n_ff=768)
    same(p, n, 256, exact)
