"""Blocks that requests open while ``LLMEngine.feed`` gives them single tokens: every one is in the step's block table, whichever way it
gets there."""
import pytest
import torch

from distributed_llm_amd.engine.llm_engine import LLMEngine

DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("device", DEVICES)
def test_single_tokens_across_block_edges(device):
    """Four requests whose blocks fill at different steps, a fifth that arrives and one that ends on the way: the logits of each are those
    of the request by itself (bf16 roundings of another batch's products: 2^-5 of their norm; another position's are as far away as
    they are large)."""
    eng = LLMEngine("tiny-llama-test", device=device, kv_cache_gb=0.1, max_num_seqs=8, max_model_len=256, prefix_cache=False)
    lens, steps = [14, 15, 16, 31, 5], 20
    toks = [[3 + (7 * k + 5 * i) % 200 for i in range(n + steps)] for k, n in enumerate(lens)]

    def alone(k, last):
        out = [eng.feed([(k, toks[k][:lens[k]], [lens[k] - 1])])]
        out += [eng.feed([(k, [toks[k][lens[k] + i]], [0])], end=[k] if i == last - 1 else ()) for i in range(last)]
        return torch.cat(out)

    got = {k: [] for k in range(5)}
    live, fed = [], [0] * 5

    def put(rows, what):
        for k, r in zip(what, rows):
            got[k].append(r)

    for t in range(steps):
        if t == 0:
            live = [0, 1, 2, 3]
            put(eng.feed([(k, toks[k][:lens[k]], [lens[k] - 1]) for k in live]), live)
        if t == 7:      # a step of one prompt; later steps copy the whole table once
            put(eng.feed([(4, toks[4][:lens[4]], [lens[4] - 1])]), [4])
            live.append(4)
        end = [1] if t == 11 else live if t == steps - 1 else []
        put(eng.feed([(k, [toks[k][lens[k] + fed[k]]], [0]) for k in live], end=end), live)
        for k in live:
            fed[k] += 1
        live = [k for k in live if k not in end]
    assert eng.bm.num_free_blocks() == eng.bm.num_blocks and not eng._bt_upd
    for k in range(5):
        want, have = alone(k, fed[k]), torch.stack(got[k])
        assert have.shape == want.shape
        norm = want.norm(dim=-1)
        assert ((have - want).norm(dim=-1) <= 2.0 ** -5 * norm).all()
        assert ((have - want.roll(1, 0)).norm(dim=-1) > 0.25 * norm).all()

