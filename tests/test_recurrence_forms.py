"""Which form of a recurrence a step runs: a long portion is walked in chunks whatever single tokens share its step."""
import types

import torch

from distributed_llm_amd.models.hybrid import HybridModel
from distributed_llm_amd.ops import seqmix


def forms(lens, heads=8):
    T, S, n = sum(lens), len(lens), HybridModel._longest(types.SimpleNamespace(host_qlen=lens))
    return seqmix.scan_in_chunks(T, S, n), seqmix.retention_in_chunks(T, S, heads, n), seqmix.longest_portion(T, S, n) >= seqmix.DELTA_TILE_MIN


def test_mixed_steps():
    assert forms([2000] + [20] * 23) == (True, True, True)
    assert forms([200] + [1] * 31) == (False, True, True)          # a scan of 200 tokens costs less than the others' chunks
    assert forms([200]) == (True, True, True)
    assert forms([20] + [1] * 31, 16) == (False, False, False)
    assert forms([160] * 24) == (True, True, True)


def test_without_the_portions():
    """A caller that does not say: the average.  No sequence, no new token: no chunks."""
    assert seqmix.longest_portion(240, 24, None) == 10 and seqmix.longest_portion(0, 0, None) == 0
    assert not seqmix.scan_in_chunks(2400, 24, None) and seqmix.scan_in_chunks(4800, 24, None)
    assert HybridModel._longest(types.SimpleNamespace(host_qlen=None)) == 1 == HybridModel._longest(types.SimpleNamespace(host_qlen=[1, 0]))


def test_layers_say_their_longest_portion(monkeypatch):
    """Every recurrent mixer hands the step's longest portion to its op."""
    seen = []

    def op(name):
        def f(*a, **k):
            seen.append((name, k["longest"]))
            raise StopIteration
        return f

    for name in ("selective_scan", "retention", "lightning_attention", "delta_rule"):
        monkeypatch.setattr(seqmix, name, op(name))
    for name in ("causal_conv_silu", "conv_state_refill", "paged_gqa_attention", "rope_prep", "attn_prep"):
        monkeypatch.setattr(seqmix, name, lambda *a, **k: torch.zeros(33, 4096))
    monkeypatch.setattr("distributed_llm_amd.models.hybrid._mm", lambda x, w: torch.zeros(33, 4096))
    meta = types.SimpleNamespace(host_qlen=[31, 1, 1], qstart=None, qlen=None, ctx=None, state_rows=None)
    model = HybridModel.__new__(HybridModel)
    model.cfg = types.SimpleNamespace(rms_eps=1e-6)
    model._any_table = lambda: None
    m = types.SimpleNamespace(heads=2, kv_heads=2, dim=4, vdim=4, dt_rank=4, rot=None, inner=4, state=4)

    class Any(dict):
        def __missing__(self, k):
            return torch.zeros(1)

    for run in (lambda: model._mamba(Any(), m, torch.zeros(33, 8), meta, (None, None)),
                lambda: model._retention(Any(), m, torch.zeros(33, 8), None, meta, (None,)),
                lambda: model._delta(Any(), m, torch.zeros(33, 8), meta, (None, None))):
        try:
            run()
        except StopIteration:
            pass
    assert seen == [("selective_scan", 31), ("retention", 31), ("delta_rule", 31)]


def test_chunks_in_order_between():
    """Portions of a few to 64 tokens on few heads: chunks in order, neither token by token nor in parallel."""
    def form(lens, heads, dim, vdim):
        return seqmix.retention_form(sum(lens), len(lens), heads, dim, vdim, max(lens))

    for lens, heads, dim, vdim in (([8], 8, 64, 128), ([16] * 24, 8, 64, 128), ([64], 16, 128, 128), ([8] * 24, 4, 32, 32), ([16] + [1] * 7, 16, 128, 128)):
        assert form(lens, heads, dim, vdim) == (True, True)
    for lens, heads, dim, vdim in (([200], 8, 64, 128), ([96], 16, 128, 128), ([48], 4, 32, 32), ([64] * 24, 16, 128, 128), ([1000] + [1] * 31, 8, 64, 128)):
        assert form(lens, heads, dim, vdim) == (True, False)
    for lens, heads, dim, vdim in (([4], 8, 64, 128), ([1] * 64, 16, 128, 128), ([16] * 24, 16, 128, 128), ([8] * 48, 8, 64, 128), ([], 8, 64, 128)):
        assert not seqmix.retention_form(sum(lens), len(lens), heads, dim, vdim, max(lens, default=None))[0]
    assert form([40], 4, 256, 64) == (True, True)      # widths only the chunks in order take


def test_scan_steps(monkeypatch):
    """A thread takes a channel where no sequence brings more than four tokens, whatever the average."""
    seen = []
    monkeypatch.setattr(seqmix, "_native", lambda x: types.SimpleNamespace(selective_scan=lambda *a: seen.append(a[-2:])))
    for lens in ([1] * 24, [4, 1], [150] + [1] * 63, [16] + [1] * 7, [2000]):
        x, q = torch.zeros(sum(lens), 8), torch.zeros(len(lens), dtype=torch.int32)
        seqmix.selective_scan(x, x, None, None, None, 4, None, None, None, None, q, q, q, q, longest=max(lens))
    assert seen == [(False, True), (False, True), (False, False), (False, False), (True, False)]
