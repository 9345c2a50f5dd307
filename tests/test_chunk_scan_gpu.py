"""Chunk-parallel recurrences (csrc/kernels/chunk_scan.hip) against 64-bit recurrences written out here, at the edges
of their chunks (64 tokens), tiles (16, 32, 64, 128 wide) and vectors (4 elements), and beside the token-by-token
kernels.  In 32 bits a result is a sum of at most 64 + d products and one carried state: with roundings of 2^-24 that
act like a random walk the relative error stays below sqrt(64 + 128) 2^-24 times a few (gates, powers), 4e-6."""
import pytest
import torch
import torch.nn.functional as F

from distributed_llm_amd import ops
from distributed_llm_amd.ops import seqmix
from test_seqmix_gpu import batch

pytestmark = pytest.mark.gpu
DEV = "cuda"
EDGES = [([63, 64, 65], [0, 7, 64]), ([1, 0, 200, 16], [3, 2, 0, 0]), ([385], [0])]


@pytest.fixture(autouse=True, scope="module")
def _native():
    assert ops.native_available(), "HIP extension must be built for GPU tests"


def close(got, want, bound):
    assert torch.isfinite(got).all()
    assert float((got.double() - want).norm() / want.norm()) < bound


def recur(q, k, v, dec, state, qlens, starts, rows):
    """S <- dec_t S + k_t v_t^T, y_t = S^T q_t in 64 bits, per sequence; state [slots, H, d, dv] is updated."""
    out, t0 = torch.zeros_like(v), 0
    for s, (n, a) in enumerate(zip(qlens, starts)):
        if n == 0:
            continue
        S = state[rows[s]].clone() if a else torch.zeros_like(state[0])
        for t in range(t0, t0 + n):
            S = dec[t, :, None, None] * S + k[t, :, :, None] * v[t, :, None, :]
            out[t] = (S * q[t, :, :, None]).sum(1)
        state[rows[s]] = S
        t0 += n
    return out


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", EDGES)
@pytest.mark.parametrize("H,d,dv,rot", [(2, 64, 128, 64), (3, 20, 70, 10), (1, 128, 130, 0), (2, 33, 7, 32), (2, 96, 32, 6)])
def test_retention(dt, case, H, d, dv, rot):
    torch.manual_seed(31)
    qlens, starts = case
    T, qstart, qlen, ctx, rows, pos = batch(qlens, starts)
    x = torch.randn(T, 2 * H * d + 2 * H * dv, device=DEV).to(dt)
    table = ops.rope_cos_sin(512, max(rot, 2), 10000.0, DEV)
    dec = torch.tensor([1.0 - 2.0 ** (-2 - 3 * h) for h in range(H)], device=DEV)
    st = torch.randn(len(qlens), H, d, dv, device=DEV)
    s64, s32 = st.double(), st.clone()
    got = seqmix.retention(x, H, d, dv, table, rot, dec, s32, 1e-6, pos, qstart, qlen, ctx, rows, chunked=True)
    y = x.double()
    q, k, v, g = y.split([H * d, H * d, H * dv, H * dv], 1)
    q, k, h2 = q.view(T, H, d).clone(), k.view(T, H, d).clone(), rot // 2
    c, s = (table[pos.long()].double()[:, None, i * h2:(i + 1) * h2] for i in range(2))
    for z in (q, k):
        a, b = z[..., :h2].clone(), z[..., h2:rot].clone()
        z[..., :h2], z[..., h2:rot] = a * c - b * s, b * c + a * s
    o = recur(q, k * d ** -0.5, v.view(T, H, dv), dec.double().expand(T, H), s64, qlens, starts, rows.tolist())
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-6)
    close(got, o.reshape(T, -1) * F.silu(g), 4e-6 if dt == torch.float32 else 4e-3)
    close(s32, s64, 4e-6)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", EDGES)
@pytest.mark.parametrize("H,d,dv", [(3, 128, 128), (2, 40, 48), (1, 5, 6)])
def test_lightning(dt, case, H, d, dv):
    torch.manual_seed(32)
    qlens, starts = case
    T, qstart, qlen, ctx, rows, _ = batch(qlens, starts)
    x = torch.randn(T, 2 * H * d + 2 * H * dv + 4, device=DEV).to(dt)
    dec = torch.tensor([0.5, 0.97, 1.0][:H], device=DEV)
    st, nw = torch.randn(len(qlens), H, d, dv, device=DEV), torch.randn(H * dv, device=DEV)
    s64, s32 = st.double(), st.clone()
    got = seqmix.lightning_attention(x, H, d, dv, dec, s32, 1e-5, nw, qstart, qlen, ctx, rows, chunked=True)
    q, k, v, g, _ = x.double().split([H * d, H * d, H * dv, H * dv, 4], 1)
    o = recur(F.silu(q).view(T, H, d), F.silu(k).view(T, H, d), F.silu(v).view(T, H, dv), dec.double().expand(T, H), s64, qlens, starts,
              rows.tolist()).reshape(T, -1)
    o = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-5) * nw.double() * torch.sigmoid(g)
    close(got, o, 4e-6 if dt == torch.float32 else 4e-3)
    close(s32, s64, 4e-6)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", EDGES)
@pytest.mark.parametrize("H,dv,N,G", [(4, 64, 128, 2), (3, 40, 20, 3), (2, 130, 33, 1), (2, 7, 5, 2)])
def test_ssd(dt, case, H, dv, N, G):
    torch.manual_seed(33)
    qlens, starts = case
    T, qstart, qlen, ctx, rows, _ = batch(qlens, starts)
    xbc = torch.randn(T, H * dv + 2 * G * N, device=DEV).to(dt)
    proj = torch.randn(T, H + 3, device=DEV).to(dt)
    # steep and flat decays: a head that forgets within a few tokens, one that keeps everything
    dt_b, neg_a, D = torch.randn(H, device=DEV), -torch.tensor([8.0, 0.5, 1e-3, 0.05][:H], device=DEV), torch.randn(H, device=DEV)
    st = torch.randn(len(qlens), H, N, dv, device=DEV)
    outs = []
    for chunked in (True, False):
        s64, s32 = st.double(), st.clone()
        got = seqmix.ssd_scan(xbc, proj, 2, H, dv, N, G, dt_b, neg_a, D, s32, qstart, qlen, ctx, rows, chunked=chunked)
        v, B, C = xbc.double().split([H * dv, G * N, G * N], 1)
        B, C = (z.view(T, G, N).repeat_interleave(H // G, 1) for z in (B, C))
        step, v = F.softplus(proj[:, 2:2 + H].double() + dt_b.double(), threshold=40), v.view(T, H, dv)
        o = recur(C, B * step[..., None], v, torch.exp(step * neg_a.double()), s64, qlens, starts, rows.tolist()) + D.double()[:, None] * v
        close(got, o.reshape(T, -1), 4e-6)
        close(s32, s64, 4e-6)
        outs.append(float((got.double() - o.reshape(T, -1)).norm() / o.norm()))
    assert outs[0] < 2 * outs[1] + 1e-7      # as exact as the token-by-token form


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", EDGES + [([31, 32, 33, 2], [1, 0, 32, 0])])
@pytest.mark.parametrize("C,N,R,K", [(256, 16, 8, 4), (70, 5, 3, 2), (300, 32, 0, 1), (8, 17, 4, 4), (264, 33, 2, 3)])
def test_selective_scan(dt, case, C, N, R, K):
    """Chunks of 32 tokens, 8 inputs in flight, 256 channels a workgroup, 8 / 16 / 32 states a thread (33: token by token)."""
    torch.manual_seed(34)
    qlens, starts = case
    T, qstart, qlen, ctx, rows, _ = batch(qlens, starts)
    S = len(qlens)
    xc, dtr = torch.randn(T, C, device=DEV).to(dt), torch.randn(T, C, device=DEV).to(dt)
    dbc, xz = torch.randn(T, R + 2 * N + 1, device=DEV).to(dt), torch.randn(T, 2 * C + 3, device=DEV).to(dt)
    dtb, A, D = torch.randn(C, device=DEV) - 2, -torch.rand(C, N, device=DEV) * 8, torch.randn(C, device=DEV)
    st, cv = torch.randn(S, C, N, device=DEV), torch.randn(S, K - 1, C, device=DEV).to(dt)
    step = F.softplus(dtr.double() + dtb.double(), threshold=40)
    want, s64, t0 = torch.zeros(T, C, dtype=torch.float64, device=DEV), st.double(), 0
    B, Cm = dbc[:, R:R + N].double(), dbc[:, R + N:R + 2 * N].double()
    for s, (n, a) in enumerate(zip(qlens, starts)):
        h = s64[rows[s]].clone() if a else torch.zeros(C, N, dtype=torch.float64, device=DEV)
        for t in range(t0, t0 + n):
            h = torch.exp(step[t, :, None] * A.double()) * h + (step[t] * xc[t].double())[:, None] * B[t]
            want[t] = (h * Cm[t]).sum(1) + D.double() * xc[t].double()
        if n:
            s64[rows[s]] = h
        t0 += n
    want = want * F.silu(xz[:, C:2 * C].double())
    errs, convs = [], []
    for chunked in (True, False):
        s32, c32 = st.clone(), cv.clone()
        got = seqmix.selective_scan(xc, dtr, dtb, A, dbc, R, D, xz, s32, c32, qstart, qlen, ctx, rows, chunked=chunked)
        close(got, want, 4e-6 if dt == torch.float32 else 4e-3)
        close(s32, s64, 4e-6)
        errs.append(float((s32.double() - s64).norm() / s64.norm()))
        convs.append(c32)
    assert torch.equal(*convs) and errs[0] < 2 * errs[1] + 1e-7      # as exact as the token-by-token form


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", EDGES + [([128, 15, 17], [64, 1, 0])])
@pytest.mark.parametrize("H,G,d,dv", [(4, 2, 128, 128), (3, 3, 64, 40), (2, 1, 36, 20), (2, 2, 33, 17), (1, 1, 4, 4), (2, 1, 104, 130)])
@pytest.mark.parametrize("steep", [0.0, 4.0])
def test_delta_rule(dt, case, H, G, d, dv, steep):
    """Tiles of 16 tokens, padded key widths 64 / 128, 16 value columns, rows that are no whole vectors; decays near 1 and
    steep, and keys that repeat, for which the triangular system is furthest from the identity."""
    torch.manual_seed(35)
    qlens, starts = case
    T, qstart, qlen, ctx, rows, _ = batch(qlens, starts)
    S = len(qlens)
    qkv = torch.randn(T, 2 * G * d + H * dv, device=DEV)
    qkv[::3, G * d:2 * G * d] = qkv[:1, G * d:2 * G * d]
    qkv, gba = qkv.to(dt), torch.randn(T, H * dv + 2 * H + 3, device=DEV).to(dt)
    na, dtb, nw = -torch.rand(H, device=DEV) * (0.05 + steep), torch.randn(H, device=DEV), torch.randn(dv, device=DEV)
    st = torch.randn(S, H, dv, d, device=DEV) * 0.5
    q, k, v = qkv.double().split([G * d, G * d, H * dv], 1)
    q, k = (z.view(T, G, d) * torch.rsqrt((z.view(T, G, d) ** 2).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
    q, k = (q * d ** -0.5).repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1)
    v, gate, beta, al = v.view(T, H, dv), *(gba[:, a:b].double() for a, b in ((0, H * dv), (H * dv, H * dv + H), (H * dv + H, H * dv + 2 * H)))
    beta, g = torch.sigmoid(beta), torch.exp(na.double() * F.softplus(al + dtb.double(), threshold=40))
    want, s64, t0 = torch.zeros(T, H, dv, dtype=torch.float64, device=DEV), st.double(), 0
    for s, (n, a) in enumerate(zip(qlens, starts)):
        M = s64[rows[s]].clone() if a else torch.zeros(H, dv, d, dtype=torch.float64, device=DEV)
        for t in range(t0, t0 + n):
            M = g[t, :, None, None] * M
            u = beta[t, :, None] * (v[t] - (M * k[t, :, None]).sum(-1))
            M = M + u[:, :, None] * k[t, :, None]
            want[t] = (M * q[t, :, None]).sum(-1)
        if n:
            s64[rows[s]] = M
        t0 += n
    want = (want * torch.rsqrt((want * want).mean(-1, keepdim=True) + 1e-6) * nw.double()).reshape(T, -1) * F.silu(gate)
    errs = []
    for tiled in (True, False):
        s32 = st.clone()
        got = seqmix.delta_rule(qkv, gba, H, G, d, dv, na, dtb, nw, 1e-6, s32, qstart, qlen, ctx, rows, tiled=tiled)
        close(got, want, 8e-6 if dt == torch.float32 else 4e-3)
        close(s32, s64, 8e-6)
        errs.append((float((s32.double() - s64).norm() / s64.norm()), float((got.double() - want).norm() / want.norm())))
    # as exact as token by token, but for the inverse's own roundings: two of 2^-24 more
    assert errs[0][0] < 1.5 * errs[1][0] + 2.0 ** -23 and errs[0][1] < 1.5 * errs[1][1] + 2.0 ** -23


STEPS = [([1] * 5, [3, 0, 64, 1, 7]), ([1, 0, 3, 2], [0, 5, 9, 0]), ([1], [400])]


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", STEPS)
@pytest.mark.parametrize("H,d,dv,rot", [(2, 64, 128, 64), (16, 128, 128, 0), (3, 20, 36, 10), (1, 256, 64, 32), (2, 5, 4, 0), (2, 64, 256, 6), (2, 33, 7, 32)])
def test_retention_steps(dt, case, H, d, dv, rot):
    """Few new tokens: 4 / 8 / 16 key rows a thread, columns that leave threads idle, widths that are no vectors (the LDS form)."""
    torch.manual_seed(36)
    qlens, starts = case
    T, qstart, qlen, ctx, rows, pos = batch(qlens, starts)
    x = torch.randn(T, 2 * H * d + 2 * H * dv + 3, device=DEV)
    # keys lean on their queries: a first token's output is (q . k) v to unit RMS, whose error is that of q . k over its size, without bound
    # where the two are at right angles
    x[:, H * d:2 * H * d] += x[:, :H * d]
    x = x.to(dt)
    table = ops.rope_cos_sin(512, max(rot, 2), 10000.0, DEV)
    dec = torch.tensor([1.0 - 2.0 ** (-2 - 3 * (h % 4)) for h in range(H)], device=DEV)
    st = torch.randn(len(qlens) + 1, H, d, dv, device=DEV)
    q, k, v, g = x.double()[:, :2 * H * (d + dv)].split([H * d, H * d, H * dv, H * dv], 1)
    q, k, h2 = q.view(T, H, d).clone(), k.view(T, H, d).clone(), rot // 2
    c, s = (table[pos.long()].double()[:, None, i * h2:(i + 1) * h2] for i in range(2))
    for z in (q, k):
        a, b = z[..., :h2].clone(), z[..., h2:rot].clone()
        z[..., :h2], z[..., h2:rot] = a * c - b * s, b * c + a * s
    for form in ("retention", "lightning"):
        s64, s32 = st.double(), st.clone()
        if form == "retention":
            got = seqmix.retention(x, H, d, dv, table, rot, dec, s32, 1e-6, pos, qstart, qlen, ctx, rows, chunked=False)
            o = recur(q, k * d ** -0.5, v.reshape(T, H, dv), dec.double().expand(T, H), s64, qlens, starts, rows.tolist())
            want = (o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-6)).reshape(T, -1) * F.silu(g)
        else:
            nw = torch.randn(H * dv, device=DEV)
            got = seqmix.lightning_attention(x, H, d, dv, dec, s32, 1e-6, nw, qstart, qlen, ctx, rows, chunked=False)
            y = F.silu(x.double()[:, :H * (2 * d + dv)])
            o = recur(*(y[:, i * H * d:i * H * d + H * e].reshape(T, H, e) for i, e in ((0, d), (1, d), (2, dv))), dec.double().expand(T, H), s64,
                      qlens, starts, rows.tolist()).reshape(T, -1)
            want = o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-6) * nw.double() * torch.sigmoid(g)
        close(got, want, 4e-6 if dt == torch.float32 else 4e-3)
        close(s32, s64, 2e-6)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", STEPS)
@pytest.mark.parametrize("C,N,R,K", [(2048, 16, 64, 4), (70, 4, 3, 2), (300, 32, 0, 1), (8, 20, 4, 9), (65, 8, 1, 3), (64, 6, 2, 4)])
def test_scan_steps(dt, case, C, N, R, K):
    """Few new tokens: a thread per channel, 8 / 16 / 32 states in registers, channels that fill no wave, 0 to 8 kept inputs (6 states: the
    form of 16 lanes a channel)."""
    torch.manual_seed(37)
    qlens, starts = case
    T, qstart, qlen, ctx, rows, _ = batch(qlens, starts)
    S = len(qlens)
    xc, dtr = torch.randn(T, C, device=DEV).to(dt), torch.randn(T, C, device=DEV).to(dt)
    dbc, xz = torch.randn(T, R + 2 * N + 1, device=DEV).to(dt), torch.randn(T, 2 * C + 3, device=DEV).to(dt)
    dtb, A, D = torch.randn(C, device=DEV) - 2, -torch.rand(C, N, device=DEV) * 8, torch.randn(C, device=DEV)
    st, cv = torch.randn(S + 1, C, N, device=DEV), torch.randn(S + 1, K - 1, C, device=DEV).to(dt)
    step, want, s64, c2, t0 = F.softplus(dtr.double() + dtb.double(), threshold=40), torch.zeros(T, C, dtype=torch.float64, device=DEV), st.double(), cv.clone(), 0
    for s, (n, a) in enumerate(zip(qlens, starts)):
        h = s64[rows[s]].clone() if a else torch.zeros(C, N, dtype=torch.float64, device=DEV)
        for t in range(t0, t0 + n):
            h = torch.exp(step[t, :, None] * A.double()) * h + (step[t] * xc[t].double())[:, None] * dbc[t, R:R + N].double()
            want[t] = (h * dbc[t, R + N:R + 2 * N].double()).sum(1) + D.double() * xc[t].double()
        if n:
            s64[rows[s]] = h
            old = cv[rows[s]] if a else torch.zeros_like(cv[0])
            c2[rows[s]] = torch.cat([old, xz[t0:t0 + n, :C]])[n:]
        t0 += n
    got = seqmix.selective_scan(xc, dtr, dtb, A, dbc, R, D, xz, st, cv, qstart, qlen, ctx, rows, chunked=False)
    close(got, want * F.silu(xz[:, C:2 * C].double()), 4e-6 if dt == torch.float32 else 4e-3)
    close(st, s64, 4e-6)
    assert torch.equal(cv, c2)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 3, 70])
@pytest.mark.parametrize("S", [0, 3, 130])
def test_rows_of_no_sequence_are_zero(dt, n, S):
    """Padding ahead of, between and behind the sequences, in the forms of a step, of few tokens and of chunks; stale memory under the
    outputs is NaN.  S = 0: every row is padding."""
    torch.manual_seed(38)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    T = S * (n + 1) + 5
    qs, ql = i32([2 + s * (n + 1) for s in range(S)]), i32([n if s % 3 else 0 for s in range(S)])
    cx, rw = ql + 4, i32(list(range(S)))
    live = torch.zeros(T, dtype=torch.bool, device=DEV)
    for a, m in zip(qs.tolist(), ql.tolist()):
        live[a:a + m] = True

    def check(f):
        for w in (T * 70, T * 64, T * 256):          # blocks of these sizes come back from the allocator
            for t in (torch.float32, torch.bfloat16):
                x = torch.full((w,), float("nan"), device=DEV, dtype=t)
                del x
        y = f()
        assert torch.isfinite(y).all() and not y[~live].any()
        if S > 1:
            assert y[live].any()

    H, d, dv, C, N = 2, 16, 32, 64, 16
    x = torch.randn(T, 2 * H * (d + dv), device=DEV).to(dt)
    table, dec = ops.rope_cos_sin(512, 16, 10000.0, DEV), torch.full((H,), 0.9, device=DEV)
    st = torch.randn(max(S, 1), H, d, dv, device=DEV)
    pos = torch.zeros(T, dtype=torch.int32, device=DEV)
    for c in (False, True):
        check(lambda: seqmix.retention(x, H, d, dv, table, 16, dec, st, 1e-6, pos, qs, ql, cx, rw, chunked=c))
    xc, dbc, xz = torch.randn(T, C, device=DEV).to(dt), torch.randn(T, 2 * N, device=DEV).to(dt), torch.randn(T, 2 * C, device=DEV).to(dt)
    A, v, ss = -torch.rand(C, N, device=DEV), torch.zeros(C, device=DEV), torch.zeros(max(S, 1), C, N, device=DEV)
    cv = torch.zeros(max(S, 1), 3, C, device=DEV).to(dt)
    for c in (False, True):
        check(lambda: seqmix.selective_scan(xc, xc, v, A, dbc, 0, v + 1, xz, ss, cv, qs, ql, cx, rw, chunked=c))
        sd, pr = torch.zeros(max(S, 1), H, N, 32, device=DEV), torch.randn(T, H, device=DEV).to(dt)
        check(lambda: seqmix.ssd_scan(torch.cat([xc, dbc], 1), pr, 0, H, 32, N, 1, dec, -dec, dec, sd, qs, ql, cx, rw, chunked=c))
    w = torch.randn(C, 4, device=DEV)
    check(lambda: seqmix.causal_conv_silu(xc, w, v, cv, qs, ql, cx, rw))
    if n == 1:
        check(lambda: seqmix.causal_conv_silu(xc, w, v, cv, qs, ql, cx, rw, refill=True))
