"""A packed chunk's inputs by arrays (BlockManager.chunk_inputs, ops.tile_table) against the lists they are made of."""
import numpy as np
import pytest

from distributed_llm_amd import ops
from distributed_llm_amd.engine import _runtime
from distributed_llm_amd.models.llama import AttnMeta


def test_tokens_positions_slots():
    bm = _runtime.BlockManager(64, 16, False)
    toks = {1: list(range(100, 137)), 2: [7], 3: list(range(16))}
    for k, t in toks.items():
        assert bm.allocate(k, t)[0]
    toks[2].append(9)
    bm.append_token(2, 9)
    spans = [(1, 0, 37), (2, 1, 2), (3, 3, 3), (1, 15, 33)]
    got = bm.chunk_inputs(*(list(v) for v in zip(*spans)))
    want = [sum((toks[k][a:b] for k, a, b in spans), []), sum((list(range(a, b)) for _, a, b in spans), []),
            sum((bm.slots(k, a, b) for k, a, b in spans), [])]
    assert all(g.dtype == np.int32 and g.tolist() == w for g, w in zip(got, want))
    for bad in ((1, 0, 38), (1, -1, 3), (1, 5, 4)):
        with pytest.raises(IndexError):
            bm.chunk_inputs([bad[0]], [bad[1]], [bad[2]])
    with pytest.raises(Exception):
        bm.chunk_inputs([9], [0], [1])


def test_prompts_of_other_lists():
    """What is no list of plain ints goes through the converter, as before."""
    bm = _runtime.BlockManager(8, 16, False)
    assert bm.allocate(1, (1, 2, 3))[0] and bm.allocate(2, [np.int64(4), 5])[0] and bm.allocate(3, [True])[0]
    assert [bm.chunk_inputs([i], [0], [n])[0].tolist() for i, n in ((1, 3), (2, 2), (3, 1))] == [[1, 2, 3], [4, 5], [1]]
    for bad in ([1.5], ["a"], [1 << 31], [None], "ab"):
        with pytest.raises(TypeError):
            bm.allocate(4, bad)
    with pytest.raises(ValueError):
        bm.allocate(4, [])


@pytest.mark.parametrize("lens", [[1], [16, 1, 33], [300, 0, 5], [0], [32] * 7])
@pytest.mark.parametrize("group", [1, 4, 8])
def test_tiles(lens, group):
    for tokens, lists in ((16 // group, ops.build_tiles(lens, group)), (ops.FLASH_ROWS // group, ops.flash_tiles(lens, group))):
        seq, tok0 = ops.tile_table(np.asarray(lens, dtype=np.int64), tokens)
        assert seq.dtype == tok0.dtype == np.int32 and seq.tolist() == lists[0] and tok0.tolist() == lists[1]


def test_latent_tiles():
    meta = AttnMeta(*[None] * 8, host_qlen=[5, 1, 40])
    ts, tt = meta.latent_tiles(4, "cpu", 16)
    assert ts.tolist() == [0, 0, 1] + [2] * 10 and tt.tolist() == [0, 4, 0] + list(range(0, 40, 4))
