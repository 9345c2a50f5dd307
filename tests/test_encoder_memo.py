"""``MiniLMEncoder.encode`` without a memo: texts that are all new go straight through the forward, every other mix row by row; either way
the rows, the forwards and the counters are those of ``encode_rows``."""
import pytest
import torch

from distributed_llm_amd.models.minilm import MiniLMConfig, MiniLMEncoder

CFG = MiniLMConfig(vocab=2000, hidden=64, layers=1, heads=2, intermediate=128)
FIELDS = ("memo_hits", "memo_misses", "encoded_texts", "batch_hits")


def _encoder(scope=(), memo_size=0):
    enc = MiniLMEncoder(CFG, device="cpu", memo_size=memo_size)
    if scope:
        enc.prefetch(list(scope))
    forward, enc.ran = enc._forward, []
    enc._forward = lambda texts, max_len: enc.ran.append(list(texts)) or forward(texts, max_len)
    return enc


@pytest.mark.parametrize("scope", [(), ("a b", "later")])
@pytest.mark.parametrize("texts", [["a b"], ["a b", "c", "d e f"], ["c", "c"], ["a b", "c", "a b", "c"], ("a b", "c"), ["later", "new"], []])
@pytest.mark.parametrize("memo_size", [0, 8])
def test_as_row_by_row(scope, texts, memo_size):
    a, b = _encoder(scope, memo_size), _encoder(scope, memo_size)
    for _ in range(2):      # (the scope outlives a call)
        got, rows = a.encode(texts), b.encode_rows(texts)
        assert got.shape == (len(texts), CFG.hidden) and got.dtype == torch.float32
        assert all(torch.equal(g, r) for g, r in zip(got, rows))
        assert a.ran == b.ran and [getattr(a, f) for f in FIELDS] == [getattr(b, f) for f in FIELDS]
    got.zero_()             # the caller's own
    assert len(texts) == 0 or float(a.encode(texts).norm(dim=1).min()) > 0.99


def test_duplicates_run_once_and_scope_not_at_all():
    enc = _encoder(("x", "y"))
    enc.encode(["p", "q", "p"])
    assert enc.ran == [["p", "q"]] and (enc.memo_misses, enc.encoded_texts) == (3, 4)
    enc.encode(["x", "r"])
    enc.encode(["y", "x"])
    assert enc.ran[1:] == [["r"]] and enc.batch_hits == 3
    enc.encode(["s", "t"])
    assert enc.ran[2:] == [["s", "t"]] and enc.memo_misses == 6 and enc.memo_hits == 0
