"""What a launch writes beside its own result: a cleared attention output, the rounded stream widened."""
import pytest
import torch

from distributed_llm_amd.ops import seqmix

pytestmark = pytest.mark.gpu


def _args(T, H, G, d, dv, dtype, cols):
    g = torch.Generator(device="cuda").manual_seed(T + H + d)
    proj = torch.randn(T, cols, device="cuda", generator=g).to(dtype)
    blocks = (T + 15) // 16 + 1
    slots = torch.arange(T, device="cuda", dtype=torch.int32)
    slots[-1] = -1      # a padding row
    pos = torch.arange(T, device="cuda", dtype=torch.int32) % 50
    table = torch.randn(64, d, device="cuda", generator=g)
    return proj, slots, pos, table, blocks


# the last two take the form in 16-byte vectors
@pytest.mark.parametrize("T,H,G,d,dv,dtype", [(1, 2, 1, 8, 3, torch.float32), (5, 3, 3, 10, 6, torch.bfloat16), (16, 8, 2, 64, 64, torch.bfloat16),
                                              (301, 32, 8, 64, 64, torch.bfloat16), (263, 40, 8, 64, 40, torch.bfloat16)])
@pytest.mark.parametrize("odt", [torch.float32, torch.bfloat16])
def test_preps_clear_rows(T, H, G, d, dv, dtype, odt):
    n = H * dv
    if n * odt.itemsize % 4:
        pytest.skip("rows of whole 4-byte words")
    proj, slots, pos, table, blocks = _args(T, H, G, d, dv, dtype, (H + G) * d + G * dv)
    kc, vc = torch.zeros(blocks, G, 16, d, device="cuda", dtype=dtype), torch.zeros(blocks, G, dv, 16, device="cuda", dtype=dtype)
    qs = torch.rand(H, device="cuda") + 0.5
    rot = d // 16 * 16
    z = torch.full((T + 2, n), float("nan"), device="cuda", dtype=odt)
    want = seqmix.attn_prep(proj, H, G, d, dv, table, rot, 1e-6, qs, pos, slots, kc.clone(), vc.clone())
    k2, v2 = kc.clone(), vc.clone()
    got = seqmix.attn_prep(proj, H, G, d, dv, table, rot, 1e-6, qs, pos, slots, k2, v2, z[1:-1])
    assert torch.equal(want, got) and (z[1:-1] == 0).all() and z[0].isnan().all() and z[-1].isnan().all()
    if H % 2 == 0 and G % 2 == 0:      # two maps a head, over the same columns
        w = torch.rand(d, device="cuda")
        vm = torch.zeros(blocks, G // 2, dv, 16, device="cuda", dtype=dtype)
        args = (proj, None, H // 2, G // 2, 2, d, dv, w, w, table, rot, 1e-6, 0.3, pos, slots)
        want = seqmix.qk_norm_prep(*args, kc.clone(), vm.clone())
        z.fill_(float("nan"))
        got = seqmix.qk_norm_prep(*args, kc.clone(), vm.clone(), z[1:-1])
        assert torch.equal(want, got) and (z[1:-1] == 0).all() and z[0].isnan().all() and z[-1].isnan().all()
    with pytest.raises(RuntimeError):
        seqmix.attn_prep(proj, H, G, d, dv, table, rot, 1e-6, qs, pos, slots, k2, v2, z)      # not T rows


# rows in registers (1, 3, 32 entries a thread; parts), rows in two passes
@pytest.mark.parametrize("T,H,groups", [(3, 8, 1), (5, 700, 1), (2, 8192, 1), (2, 8200, 1), (7, 1024, 4), (3, 96, 3), (2, 16640, 4)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_norm_resadd_widens(T, H, groups, dtype):
    g = torch.Generator(device="cuda").manual_seed(H)
    y = torch.randn(T, H, device="cuda", generator=g).to(dtype)
    w, x = torch.rand(H, device="cuda", generator=g), torch.randn(T, H, device="cuda", generator=g)
    want, lp = x.clone(), torch.empty(T, H, device="cuda", dtype=dtype)
    seqmix.norm_resadd(y, w, 1e-6, want, lp, groups)
    got, lp2, wide = x.clone(), torch.empty_like(lp), torch.empty_like(x)
    seqmix.norm_resadd(y, w, 1e-6, got, lp2, groups, x_wide=wide)
    assert torch.equal(want, got) and torch.equal(lp, lp2) and torch.equal(lp.float(), wide)


# less than a wave, more values than a lane keeps, more rotated columns than a wave has lanes; f32 sums of up to 700 squares: some 20
# roundings on the longest way, 2e-5 leaves ten times that
@pytest.mark.parametrize("rank,rot,qn", [(5, 2, 3), (64, 64, 0), (256, 32, 192), (700, 130, 1600)])
@pytest.mark.parametrize("half", [False, True])
def test_latent_write_edges(rank, rot, qn, half):
    from distributed_llm_amd.ops import reference as ref
    T, g = 4, torch.Generator(device="cuda").manual_seed(rank)
    R = lambda *s: torch.randn(*s, device="cuda", generator=g)
    row, w, wq, table = R(T, qn + rank + rot), torch.rand(rank, device="cuda"), torch.rand(max(qn, 1), device="cuda"), R(16, rot)
    slots = torch.tensor([3, -1, 17, 0], device="cuda", dtype=torch.int32)
    pos = torch.tensor([0, 16, 15, 7], device="cuda", dtype=torch.int32)      # the padding token's lies behind the table
    c1, c2 = torch.zeros(2, 16, rank + rot, device="cuda"), torch.zeros(2, 16, rank + rot, device="cuda")
    q = (row[:, :qn], wq) if qn else (None, None)
    a = seqmix.latent_kv_write(row[:, qn:], rank, w, 1e-6, pos, table, slots, c1, half, *q)
    b = ref.latent_kv_write(row[:, qn:], rank, w, 1e-6, pos.clamp(max=15), table, slots, c2, half, *q)
    torch.testing.assert_close(c1, c2, rtol=2e-5, atol=2e-5)
    if qn:
        torch.testing.assert_close(a, b, rtol=2e-5, atol=2e-5)
