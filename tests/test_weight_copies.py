"""Further copies of a model's weights: when they are laid out, and at whose cost."""
import pytest
import torch

from distributed_llm_amd.models.configs import ModelConfig, filevik_config, sedopel_config
from distributed_llm_amd.models.registry import build_model
from distributed_llm_amd.ops import gemm as G

DENSE = ModelConfig("dense", 256, 2, 4, 2, 64, 512, 512, 10000.0, 1e-5, 512)
SPARSE = ModelConfig("sparse", 256, 2, 4, 2, 64, 512, 512, 10000.0, 1e-5, 512, n_experts=4, experts_per_token=2)

LAYERS = filevik_config({"architecture": "Filevik", "width": 128, "vocab": 512, "norm": {"eps": 1e-6}, "logit_scale": 1.0, "layers": [
    {"type": "latent_attention", "mixer": {"heads": 4, "dim": 32, "rot_dim": 32, "vdim": 32, "kv_rank": 64, "q_rank": 128, "scale": 0.125,
                                           "rot": {"dims": 32, "base": 10000.0}},
     "mlp": {"kind": "moe", "router": {"experts": 4, "top": 2, "scale": 1.0}, "expert": {"ff": 64}, "shared": {"ff": 64}}}] * 2})


def _copies(m):
    return sorted({k for L in m.layers for k in L if k.endswith(("_r", "_p"))}) + (["head"] if m.lm_head_r is not None else [])


def test_a_quarter_of_what_is_free(monkeypatch):
    monkeypatch.delenv("DLLM_REHEARSE_ONE_GPU", raising=False)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d: (4000, 10000))
    assert G.copies_fit(1000, "cuda") and not G.copies_fit(1001, "cuda")
    assert G.copies_fit(500, "cuda", 2000) and not G.copies_fit(501, "cuda", 2000) and not G.copies_fit(1, "cuda", 4000)
    monkeypatch.setenv("DLLM_REHEARSE_ONE_GPU", "1")
    assert not G.copies_fit(1, "cuda")


MODELS = [(DENSE, {"wqkv_f_p", "wqkv_f_r", "wd_r", "head"}), (SPARSE, {"wqkv_f_r", "wo_r", "w13_r", "w2_r", "head"}),
          (LAYERS, {"dqkv_r", "o_r", "experts_r", "head"})]


@pytest.mark.gpu
@pytest.mark.parametrize("cfg,some", MODELS, ids=lambda c: getattr(c, "name", None))
def test_none_where_ranks_share_a_gpu(monkeypatch, cfg, some):
    monkeypatch.delenv("DLLM_REHEARSE_ONE_GPU", raising=False)
    assert some <= set(_copies(build_model(cfg)))
    monkeypatch.setenv("DLLM_REHEARSE_ONE_GPU", "1")
    assert _copies(build_model(cfg)) == []


@pytest.mark.gpu
@pytest.mark.parametrize("cfg,some", MODELS, ids=lambda c: getattr(c, "name", None))
def test_the_pool_comes_first(monkeypatch, cfg, some):
    """Fragment-major copies are laid out behind the paged pool, out of what neither it nor the reserve beside it takes; an engine that has
    no room for them serves without."""
    from distributed_llm_amd.engine import llm_engine as E
    monkeypatch.delenv("DLLM_REHEARSE_ONE_GPU", raising=False)
    seen, alloc, info = [], E.LLMEngine._alloc_kv, torch.cuda.mem_get_info

    def alloc_kv(self, *a):
        seen.append([k for k in _copies(self.model) if not k.endswith("_p")])
        alloc(self, *a)

    monkeypatch.setattr(E.LLMEngine, "_alloc_kv", alloc_kv)
    make = lambda **kw: E.LLMEngine(cfg, device="cuda", max_num_seqs=4, max_model_len=256, prefix_cache=False, **kw)  # noqa: E731
    prompts = [[5, 9, 13], [7] * 20]
    steps = lambda e: [e.feed([(k, p, [len(p) - 1]) for k, p in enumerate(prompts)])] + [  # noqa: E731
        e.feed([(k, [11 + k + i], [0]) for k in range(2)]) for i in range(3)]
    with_copies = make(num_kv_blocks=300)
    assert seen == [[]] and with_copies.num_blocks == 300 and some <= set(_copies(with_copies.model))
    want = torch.cat(steps(with_copies))
    # a device with no more than the reserve free beside the pool that was asked for
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d=None: (int((E.KV_RESERVE_GB + 1) * 2 ** 30), info(d)[1]))
    without = make(kv_cache_gb=8.0)
    assert without.kv_cache_gb == 1.0
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d=None: (int(E.KV_RESERVE_GB * 2 ** 30), info(d)[1]))
    without = make(num_kv_blocks=300)
    assert not [k for k in _copies(without.model) if not k.endswith("_p")]
    got = torch.cat(steps(without))
    # other plans: bf16 roundings of a few layers
    assert float((got - want).norm() / want.norm()) < 2.0 ** -5


LONG = sedopel_config({"architecture": "Sedopel", "width": 128, "vocab": 512, "norm": {"eps": 1e-6}, "layers": [
    {"type": "delta", "mlp": {"kind": "dense", "ff": 4096}, "mixer": {"heads": 2, "kv_heads": 1, "dim": 64, "vdim": 64, "conv": 4}}] * 2})


@pytest.mark.gpu
@pytest.mark.parametrize("cfg,dtype,last", [(LONG, torch.float32, "down_r"), (LAYERS, torch.bfloat16, "uk_r")], ids=["long f32 rows", "uk"])
def test_the_last_copies_cost_no_other_its_place(monkeypatch, cfg, dtype, last):
    """Room for all but the long rows of an f32 model, or all but the key up-projections: only those are missing."""
    asked, room = [], [1 << 40]
    monkeypatch.setattr(G, "copies_fit", lambda extra, device, spare=0: (asked.append(extra), extra <= room[0])[1])
    every = set(_copies(build_model(cfg, dtype=dtype)))
    assert last in every
    mine = sum(asked[:1])      # the projections and the head; what else there is was asked for behind them
    base, asked[:] = set(every) - {last}, []
    room[0] = mine
    monkeypatch.setattr(G, "copies_fit", lambda extra, device, spare=0: (asked.append(extra), len(asked) == 1 and extra <= room[0])[1])
    got = set(_copies(build_model(cfg, dtype=dtype)))
    assert got == base - {"experts_r"} and got
