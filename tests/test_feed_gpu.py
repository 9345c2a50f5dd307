"""Logits of ``LLMEngine.feed`` on their way to the host."""
import pytest
import torch

from distributed_llm_amd.engine.llm_engine import LLMEngine

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    return LLMEngine("tiny-llama-test", device="cuda", kv_cache_gb=0.1, max_num_seqs=8, max_model_len=256, prefix_cache=False)


def test_to_host(eng):
    """Whole, odd and empty numbers of slots, a strided source, and a source rewritten right after."""
    S = eng.READ_SLOT
    for n in (0, 1, S - 1, S, S + 1, 3 * S + 7):
        x = torch.randn(n, 1, device="cuda")
        want = x.clone()
        got = eng._to_host(x)
        x.zero_()
        assert got.shape == (n, 1) and not got.is_cuda and torch.equal(got, want.cpu())
    x = torch.randn(5, 2 * 511, device="cuda")[:, ::2]
    assert torch.equal(eng._to_host(x), x.cpu())


@pytest.mark.parametrize("who", [[0, 1, 2], [1], [2, 0], [1, 1], []])
def test_wanted_rows_of_a_decode_step(eng, who):
    """Any choice of rows, in entry order and repeated, of the same three requests' next step."""
    prompts = [[5, 9, 13], [7] * 20, [3, 4]]
    eng.feed([(k, p, []) for k, p in enumerate(prompts)])
    every = eng.feed([(k, [11 + k], [0]) for k in range(3)], end=range(3))
    eng.feed([(k, p, []) for k, p in enumerate(prompts)])
    got = eng.feed([(k, [11 + k], [0] * who.count(k)) for k in range(3)], end=range(3))
    assert torch.equal(got, every[sorted(who)])


def _filevik(logit_scale):
    from distributed_llm_amd.models.configs import filevik_config
    mlp = {"kind": "moe", "router": {"experts": 4, "top": 2, "scale": 1.0}, "expert": {"ff": 64}, "shared": {"ff": 64}}
    kinds = [{"type": "mamba1", "mixer": {"inner": 128, "state": 16, "dt_rank": 32, "conv": 4}},
             {"type": "latent_attention", "mixer": {"heads": 4, "dim": 32, "rot_dim": 32, "vdim": 32, "kv_rank": 64, "q_rank": 128,
                                                    "scale": 0.125, "rot": {"dims": 32, "base": 10000.0}}}]
    return filevik_config({"architecture": "Filevik", "width": 128, "vocab": 512, "norm": {"eps": 1e-6}, "logit_scale": logit_scale,
                           "layers": [dict(k, mlp=mlp) for k in kinds]})


@pytest.mark.parametrize("what", ["tiny-llama-test", 1.0, 0.5], ids=["llama", "layers", "layers-scaled"])
def test_feed_and_generation_take_turns(what):
    """Given-token steps have graphs of their own beside generation's, over the same buffers and in the same pool: neither changes what the
    other answers, whichever came first, and each step's logits are that step's.  The packed form of the same tokens runs other kernels
    (prompt attention, chunked scans, other products): bf16 roundings of a few layers, 2^-5 of the logits' norm where another position's
    logits are as far away as they are large."""
    from distributed_llm_amd.engine.sampling import SamplingParams
    model = what if isinstance(what, str) else _filevik(what)
    eng = LLMEngine(model, device="cuda", kv_cache_gb=0.1, max_num_seqs=8, max_model_len=256, prefix_cache=False)
    assert eng.use_graphs
    prompts, seqs = ["user: hello", "user: what is a page?", "tell me"], [[5 + 3 * k + i * (7 + k) for i in range(12)] for k in range(3)]
    ask = lambda: [o.token_ids for o in eng.generate(prompts, SamplingParams(max_new_tokens=8, temperature=0.0))]  # noqa: E731

    def steps():
        out = [eng.feed([(k, s[:4], [3]) for k, s in enumerate(seqs)])]
        for i in range(4, 12):
            out.append(eng.feed([(k, [s[i]], [0]) for k, s in enumerate(seqs)], end=range(3) if i == 11 else ()))
        return torch.stack(out, 1)                                     # [request, step, vocab]

    whole = eng.feed([(k, s, list(range(3, 12))) for k, s in enumerate(seqs)], end=range(3)).view(3, 9, -1)
    said = [ask(), ask()]
    fed = [steps()]
    said.append(ask())
    fed.append(steps())
    said += [ask(), ask()]
    fed += [steps(), steps()]
    assert all(a == said[0] for a in said) and all(torch.equal(f, fed[0]) for f in fed)
    got, norm = fed[0], whole.norm(dim=-1)
    assert ((got - whole).norm(dim=-1) <= 2.0 ** -5 * norm).all()
    for other in (whole.roll(1, 1), whole.roll(1, 0)):                 # an earlier step's logits, another request's
        assert ((got - other).norm(dim=-1) > 0.25 * norm).all()
