"""Kabanex on the GPU: every kernel of the layer-stack family alone, then the model through the engine
(step graphs, ragged prompt forwards, cache pages and state slots, scheduler), against the plain
float64 implementation of kabanex_oracle.py."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import kabanex_oracle as O
from voice_enabled_browser_automation_amd import ops
from voice_enabled_browser_automation_amd.models.config import KabanexConfig
from voice_enabled_browser_automation_amd.models.kabanex import KabanexModel
from voice_enabled_browser_automation_amd.runtime.engine import LLMEngine
from voice_enabled_browser_automation_amd.runtime.scheduler import TokenScheduler

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"
DTYPES = [torch.float32, torch.bfloat16]
BF16, F32 = torch.bfloat16, torch.float32


def rnd(*shape, seed=0, std=1.0, dtype=F32):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * std).to(dtype)


def rel(got, want):
    return float((got.double().cpu() - want.double()).abs().max() / want.double().abs().max().clamp_min(1e-30))


# ----------------------------------------------------------------------------- rows, norms, projections
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("D,Dp,rows", [(72, 128, 5), (256, 256, 1), (1030, 1152, 33), (4100, 4224, 3), (8192, 8192, 2)])
def test_layernorm_f32(dtype, D, Dp, rows):
    x = rnd(rows, Dp, seed=1, std=3.0) + 20.0    # a mean far from zero: the variance needs the deviations
    w, b = 1 + rnd(D, seed=2, std=0.3), rnd(D, seed=3)
    out = torch.full((rows, Dp), 7.0, dtype=dtype, device=DEV)
    ops.layernorm_f32(x.to(DEV), w.to(DEV), b.to(DEV), eps=1e-3, out=out)
    want = O.layer_norm(x[:, :D].double(), w.double(), b.double(), 1e-3)
    assert rel(out[:, :D], want) < (2e-6 if dtype == F32 else 8e-3)
    assert out[:, D:].abs().sum() == 0


@pytest.mark.parametrize("dtype", DTYPES)
def test_embedding_f32(dtype):
    t = rnd(50, 72, dtype=dtype)
    ids = torch.tensor([3, 49, 0, 3], dtype=torch.int32)
    out = torch.full((4, 128), 7.0, device=DEV)
    ops.embedding_f32(ids.to(DEV), t.to(DEV), out=out)
    assert torch.equal(out[:, :72].cpu(), t[ids.long()].float()) and out[:, 72:].abs().sum() == 0


@pytest.mark.parametrize("M", [1, 3, 16, 17, 40, 64, 130, 300])
@pytest.mark.parametrize("N,K,ns", [(272, 128, 96), (1040, 384, 640), (4096, 1024, 2048)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_linear_split_and_f32_residual(dtype, M, N, K, ns):
    x, w = rnd(M, K, seed=1, dtype=dtype), rnd(N, K, seed=2, std=K ** -0.5, dtype=dtype)
    y = x.double() @ w.double().T
    tol = 3e-6 if dtype == F32 else 8e-3
    wd = ops.TiledWeight(w.to(DEV)) if dtype == BF16 else w.to(DEV)
    out = torch.zeros(M, ns, dtype=dtype, device=DEV)
    wide = torch.zeros(M, N - ns + 64, dtype=dtype, device=DEV)
    ops.linear_split(x.to(DEV), wd, out, wide[:, 32 : 32 + N - ns])
    assert rel(out, y[:, :ns]) < tol
    assert rel(wide[:, 32 : 32 + N - ns], y[:, ns:].clamp_min(0) ** 2) < 2 * tol
    assert wide[:, :32].abs().sum() == 0 and wide[:, 32 + N - ns :].abs().sum() == 0
    # residual stream: small terms onto large rows must not be rounded to 16 bits
    r = rnd(M, N + 16, seed=3, std=300.0)
    rd = r.to(DEV)
    ops.linear(x.to(DEV), wd, out=rd[:, :N], residual=rd[:, :N])
    assert float((rd[:, :N].cpu().double() - r[:, :N].double() - y).abs().max()) < (1e-3 if dtype == F32 else 2e-3)
    assert torch.equal(rd[:, N:].cpu(), r[:, N:])


@pytest.mark.parametrize("N,K", [(1003, 2064), (2048, 6144), (1024, 1024), (3904, 16), (4096, 208), (130, 48), (16416, 80), (2080, 4112)])
def test_gemm_f32_rows_do_not_depend_on_their_company(N, K):
    """A row's results have the same bits alone, in a decoded step and in a prompt, whichever kernel and waves serve it (a
    token's expert does not change with what it is batched with)."""
    gen = torch.Generator(device=DEV).manual_seed(N)
    x, w, r = torch.randn(1100, K, device=DEV, generator=gen), torch.randn(N, K, device=DEV, generator=gen), torch.randn(1100, N, device=DEV, generator=gen)
    E = ops.ext()

    def run(M, epi):
        out, rest = torch.empty(M, {2: N // 2, 6: N // 3}.get(epi, N), device=DEV), torch.empty(M, N - N // 3, device=DEV) if epi == 6 else None
        E.gemm_f32(x[:M], w, out, epi, r[:M] if epi == 1 else None, rest)
        return out if rest is None else torch.cat([out, rest], 1)

    for epi in (0, 1, 6) + ((2,) if N % 32 == 0 else ()):
        want = run(1100, epi)
        for M in (1, 4, 16, 17, 32, 33, 64, 65, 200, 449, 777):
            assert torch.equal(run(M, epi), want[:M]), (epi, M)


@pytest.mark.parametrize("M,N,K", [(1, 1, 16), (16, 1003, 2064), (17, 2080, 48), (32, 16384, 32), (64, 7713, 144),  # rows kernel
                                   (33, 16400, 80), (65, 3904, 16),                # tiles: one / two row blocks, K short of a slice
                                   (200, 4096, 208), (449, 2001, 4112), (641, 3296, 96)])   # 4, 2 and 1 groups of waves
def test_gemm_f32_kernels(M, N, K):
    """Every kernel of the dispatch at remainders of rows, columns and K, all epilogues, X rows apart.  Tolerance: each of K
    additions rounds by 2^-24 of a partial sum, which the sum of |x| |w| bounds, signs at random; an epilogue f(v) turns an error
    d of v into |f'(v)| d and rounds its result a few times."""
    gen = torch.Generator(device=DEV).manual_seed(M * 7 + N)
    randn = lambda *n: torch.randn(*n, device=DEV, generator=gen)  # noqa: E731
    x, w, r = randn(M, K + 12)[:, :K], randn(N, K) * K ** -0.5, randn(M, N)
    y, mag, tol = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T, 2.0 ** -24 * max(4.0, K ** 0.5)
    near = lambda got, want, size: float((got.double() - want).norm()) < tol * float(size.norm()) + 4e-7 * float(want.norm())  # noqa: E731
    E = ops.ext()
    out = torch.full((M, N + 4), 7.0, device=DEV)
    E.gemm_f32(x, w, out[:, :N], 0, None)
    assert near(out[:, :N], y, mag) and bool((out[:, N:] == 7).all())
    E.gemm_f32(x, w, out[:, :N], 1, r)
    assert near(out[:, :N], y + r.double(), mag) and bool((out[:, N:] == 7).all())
    a, b = torch.empty(M, N // 3, device=DEV), torch.empty(M, N - N // 3, device=DEV)
    if N > 2:
        E.gemm_f32(x, w, a, 6, None, b)
        v = y[:, N // 3 :].clamp_min(0)
        assert near(a, y[:, : N // 3], mag[:, : N // 3]) and near(b, v ** 2, 2 * v * mag[:, N // 3 :])
    if N % 32 == 0:
        h = torch.empty(M, N // 2, device=DEV)
        E.gemm_f32(x, w, h, 2, None)
        (g, u), (mg, mu) = (t.view(M, N // 32, 2, 16).unbind(2) for t in (y, mag))
        silu = torch.nn.functional.silu(g)
        assert near(h, (silu * u).reshape(M, N // 2), (1.1 * u.abs() * mg + silu.abs() * mu).reshape(M, N // 2))  # (|silu'| < 1.1)


# ----------------------------------------------------------------------------- cache + rotation
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,dk,dv,rot", [(6, 2, 32, 48, 12), (4, 4, 64, 16, 64), (3, 1, 128, 112, 32)])
def test_qkv_cache_write(dtype, H, G, dk, dv, rot):
    M, bs, nb = 37, 16, 6
    x = rnd(M, H * dk + G * (dk + dv) + 16, seed=1, dtype=dtype)
    pos = torch.arange(M, dtype=torch.int32) + 900
    slots = torch.randperm(nb * bs, generator=torch.Generator().manual_seed(0))[:M]
    slots[5] = -1
    k = torch.zeros(nb, G, bs, dk, dtype=dtype, device=DEV)
    v = torch.zeros(nb, G, dv, bs, dtype=dtype, device=DEV)
    q = torch.zeros(M, H * dk, dtype=dtype, device=DEV)
    rope = ops.rope_table(1000, rot, 250.0, device=DEV)
    ops.qkv_cache_write(x.to(DEV), n_q_heads=H, rot_dims=rot, rope=rope, positions=pos.to(DEV), slots=slots.to(DEV), q_out=q,
                        k_cache=k, v_cache=v)
    xd = x.double()
    wq = O.rotate(xd[:, : H * dk].view(M, H, dk), 250.0, rot, first=900)
    wk = O.rotate(xd[:, H * dk : (H + G) * dk].view(M, G, dk), 250.0, rot, first=900)
    wv = xd[:, (H + G) * dk : (H + G) * dk + G * dv].view(M, G, dv)
    tol = 1e-6 if dtype == F32 else 5e-3
    assert rel(q.view(M, H, dk), wq) < tol
    for m in range(M):
        s = int(slots[m])
        if s >= 0:
            assert rel(k[s // bs, :, s % bs], wk[m]) < 2 * tol and rel(v[s // bs, :, :, s % bs], wv[m]) < 2 * tol
    assert int((k != 0).any(-1).sum()) == G * (M - 1)  # the inert row wrote nothing


# ----------------------------------------------------------------------------- attention
def paged(kn, vn, perm, bs, dtype, extra=3):
    """Natural keys / values [n, G, d] -> caches with the sequence's blocks at perm; other blocks hold rubbish."""
    n, G, dk = kn.shape
    dv = vn.shape[2]
    nb = len(perm) + extra
    k = rnd(nb, G, bs, dk, seed=77, std=30.0, dtype=dtype)
    v = rnd(nb, G, dv, bs, seed=78, std=30.0, dtype=dtype)
    for j in range(n):
        k[perm[j // bs], :, j % bs] = kn[j]
        v[perm[j // bs], :, :, j % bs] = vn[j]
    return k.to(DEV), v.to(DEV)


ATT = [  # H, G, dk, dv, window, keep, bs, n
    (6, 2, 32, 48, 19, 3, 16, 130),
    (4, 4, 64, 16, 64, 0, 16, 200),
    (5, 1, 96, 208, 40, 17, 32, 150),
    (16, 4, 128, 128, 150, 5, 16, 420),
    (8, 8, 64, 80, 16, 16, 16, 90),
    (2, 2, 32, 32, 1000, 4, 16, 100),
    (1, 1, 160, 144, 33, 1, 16, 120),
    (32, 4, 64, 64, 70, 6, 16, 140),
    (20, 1, 32, 32, 30, 2, 16, 90),       # more query heads per kv head than MFMA columns
    (3, 3, 256, 256, 1, 2, 16, 50),       # a window of one
]


def pads(n):
    return 1 << (n - 1).bit_length()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("mixed", [True, False])
@pytest.mark.parametrize("case", ATT, ids=[str(c) for c in ATT])
def test_talk_attention(dtype, mixed, case):
    """Rows form and prefill form over one sequence in scattered blocks.  Some keys stand out (their score
    is far above the others'), at block and tile borders and around the kept ones, so every row just inside
    or just outside of an edge changes visibly if the edge is one off."""
    H, G, dk, dv, window, keep, bs, n = case
    gen = torch.Generator().manual_seed(3)
    u = torch.zeros(dk)
    u[0] = 1.0
    q = rnd(n, H, dk, seed=1, std=0.3) + 2.0 * u
    k = rnd(n, G, dk, seed=2, std=0.3)
    for j in {0, keep - 1, keep, keep + 1, 15, 16, 31, 32, 33, n // 2, n - 20}:
        if 0 <= j < n:
            k[j] += (3.0 + float(torch.rand(1, generator=gen))) * u
    v = rnd(n, G, dv, seed=4)
    q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
    T = (torch.eye(H) + rnd(H, H, seed=5, std=0.4)).to(BF16).float() if mixed else torch.eye(H)
    gate = rnd(n, H + 8, seed=6, dtype=dtype)
    scale = 0.7
    m = O.mask(n, window, keep)
    w = O.talk(O.softmax_weights(q.double(), k.double(), scale, m), T.double())
    want = torch.stack([0.8 * torch.sigmoid(gate[:, h : h + 1].double()) * (w[h] @ v[:, h // (H // G)].double())
                        for h in range(H)], 1).reshape(n, H * dv)
    perm = torch.randperm(-(-n // bs) + 3, generator=gen)[: -(-n // bs)].tolist()
    kc, vc = paged(k, v, perm, bs, dtype)
    table = torch.zeros(4, len(perm) + 2, dtype=torch.int32)
    table[2, : len(perm)] = torch.tensor(perm)
    table, qd = table.to(DEV), q.reshape(n, H * dk).to(DEV)
    max_ctx = len(perm) * bs
    sc = ops.TalkScratch([(H, G, dv, window, keep)], max_ctx, DEV)
    kw = dict(n_q_heads=H, scale=scale, window=window, keep=keep, talk=T.to(DEV) if mixed else None,
              talk_frag=ops.talk_fragment(T, G).to(DEV) if pads(G) * pads(H // G) <= 32 else None, out_scale=0.8, max_ctx=max_ctx, scratch=sc)
    pos = torch.arange(n, dtype=torch.int32, device=DEV)
    sid = torch.full((n,), 2, dtype=torch.int32, device=DEV)
    slots = torch.zeros(n, dtype=torch.int64, device=DEV)
    tol = 5e-6 if dtype == F32 else 1.5e-2

    def run(sel, plan):
        sel = torch.tensor(sel, device=DEV)
        out = torch.full((len(sel), H * dv), float("nan"), dtype=dtype, device=DEV)
        ops.talk_attention(qd[sel], kc, vc, table, pos[sel], sid[sel], slots[sel], gate=gate.to(DEV)[sel], out=out, plan=plan, **kw)
        return out

    assert rel(run(list(range(n)), None), want) < tol
    # whole prompt, odd starts, runs of two, single rows beside runs
    for cuts in ([(0, n)], [(7, 2), (30, n - 35), (3, 1), (n - 1, 1), (16, 17)]):
        sel, runs = [], []
        for a, c in cuts:
            c = min(c, n - a)
            runs.append((len(sel), c))
            sel += list(range(a, a + c))
        got = run(sel, ops.plan_runs(runs, DEV, n - 1))
        assert rel(got, want[sel]) < tol
    # inert rows of a padded step are zero and touch nothing
    slots[5] = -1
    got = run(list(range(12)), None)
    assert got[5].abs().sum() == 0 and rel(got[:5], want[:5]) < tol
    assert sc.counters.abs().sum() == 0


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("case", [(8, 4, 128, 128, 1024, 4, 16, 530),    # one, two and three chunks; groups of 8 rows
                                  (6, 2, 32, 144, 262, 3, 16, 280),      # a window of one chunk and a key; groups of 5, values past 128
                                  (68, 17, 32, 16, 40, 2, 16, 70),       # more heads than lanes; groups of 3 and 2
                                  (132, 12, 32, 16, 100, 2, 16, 150)],   # weights of 256 keys past LDS: 8-tile chunks, no groups
                         ids=str)
def test_talk_attention_chunks_and_groups(dtype, case):
    test_talk_attention(dtype, True, case)


def test_talk_attention_inert_row_in_a_group():
    """A row without a cache slot inside a run is zero; the others are as ever."""
    H, G, dk, dv, n = 4, 2, 32, 16, 21
    q, k, v = (rnd(n, x, d, seed=i, dtype=F32) for i, (x, d) in enumerate(((H, dk), (G, dk), (G, dv))))
    kc, vc = paged(k, v, [0, 1], 16, F32)
    table, pos = torch.tensor([[0, 1]], dtype=torch.int32, device=DEV), torch.arange(n, dtype=torch.int32, device=DEV)
    T = (torch.eye(H) + rnd(H, H, seed=5, std=0.4)).to(DEV)

    def run(slots):
        out = torch.full((n, H * dv), float("nan"), device=DEV)
        ops.talk_attention(q.reshape(n, -1).to(DEV), kc, vc, table, pos, torch.zeros_like(pos), slots, n_q_heads=H, scale=0.3,
                           window=0, keep=0, talk=T, talk_frag=None, gate=None, out_scale=1.0, max_ctx=32,
                           scratch=ops.TalkScratch([(H, G, dv, 0, 0)], 32, DEV), out=out, plan=ops.plan_runs([(0, n)], DEV, n - 1))
        return out

    slots = pos.long()
    want = run(slots.clone())
    slots[6] = -1
    got = run(slots)
    assert got[6].abs().sum() == 0 and torch.equal(got[:6], want[:6]) and torch.equal(got[7:], want[7:])


@pytest.mark.parametrize("n", [21, 400])
def test_inert_row_of_a_group_is_zero_whatever_it_holds(n):
    """A row without a cache slot was never computed: its query may hold anything.  One chunk, and several."""
    H, G, dk, dv = 4, 2, 32, 16
    q, k, v = (rnd(n, x, d, seed=i, dtype=F32) for i, (x, d) in enumerate(((H, dk), (G, dk), (G, dv))))
    blocks = -(-n // 16)
    kc, vc = paged(k, v, list(range(blocks)), 16, F32)
    table, pos = torch.arange(blocks, dtype=torch.int32, device=DEV)[None].contiguous(), torch.arange(n, dtype=torch.int32, device=DEV)
    slots = pos.long()
    inert = [6, n - 2]
    slots[inert] = -1

    def run(q):
        out = torch.full((n, H * dv), float("nan"), device=DEV)
        ops.talk_attention(q.reshape(n, -1).to(DEV), kc, vc, table, pos, torch.zeros_like(pos), slots, n_q_heads=H, scale=0.3,
                           window=0, keep=0, talk=torch.eye(H, device=DEV), talk_frag=None, gate=None, out_scale=1.0, max_ctx=16 * blocks,
                           scratch=ops.TalkScratch([(H, G, dv, 0, 0)], 16 * blocks, DEV), out=out, plan=ops.plan_runs([(0, n)], DEV, n - 1))
        return out

    want = run(q)
    q[inert] = float("nan")
    got = run(q)
    assert got[inert].abs().sum() == 0 and torch.equal(got, want)


def test_prompts_of_rising_length_leave_no_memory_behind():
    """Rows-form prompts of a 32-bit model: what their lengths size goes back with the step, it follows the prompt and not the
    engine's longest context, and two streams have sets of their own."""
    H, G, dk, dv, ctx = 8, 4, 32, 16, 1 << 16
    k, v = (torch.randn(ctx // 16, G, *s, device=DEV) for s in ((16, dk), (dv, 16)))
    table = torch.arange(ctx // 16, dtype=torch.int32, device=DEV)[None].contiguous()
    T = torch.eye(H, device=DEV)
    sc = ops.TalkScratch([(H, G, dv, 0, 0)], ctx, DEV)

    def step(n):
        pos = torch.arange(n, dtype=torch.int32, device=DEV)
        plan = ops.plan_runs([(0, n)], DEV, n - 1)
        q, out = torch.randn(n, H * dk, device=DEV), torch.empty(n, H * dv, device=DEV)
        for _ in range(2):
            ops.talk_attention(q, k, v, table, pos, torch.zeros_like(pos), pos.long(), n_q_heads=H, scale=0.3, window=0, keep=0,
                               talk=T, talk_frag=None, gate=None, out_scale=1.0, max_ctx=ctx, scratch=sc, out=out, plan=plan)
        return plan, out

    step(40)
    torch.cuda.synchronize()
    base, retired = torch.cuda.memory_allocated(), sum(t.numel() for t in ops._SCRATCH_RETIRED)
    for n in (50, 300, 500, 700, 900):
        torch.cuda.reset_peak_memory_stats()
        step(n)
        # scores, statistics and partial sums of n rows in whole groups of 8 and whole chunks of 128 keys, beside the rows' own
        per_row = H * -(-n // 128) * (128 + 4 + dv) * 4
        assert torch.cuda.max_memory_allocated() - base < (n + 8) * per_row + n * (H * (dk + dv) * 4 + 64) + (1 << 20)
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() == base
    assert sum(t.numel() for t in ops._SCRATCH_RETIRED) == retired
    plan, _ = step(60)
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        other = ops.stack.plan_scratch(plan, DEV, 16, 16, 16, 16)
    torch.cuda.synchronize()
    assert len(plan.work) == 2 and all(a.data_ptr() != b.data_ptr() for a, b in zip(other, plan.work[torch.cuda.current_stream().cuda_stream]))


def test_prefill_form_takes_the_usual_sizes():
    part = ops.ext().talk_prefill_part
    for H, G, dk, dv in [(4, 2, 64, 128), (16, 4, 128, 128), (32, 8, 128, 128), (6, 2, 96, 192), (8, 1, 256, 64), (12, 12, 64, 64)]:
        assert part(H, G, dk, dv) > 0
    assert part(40, 1, 64, 64) < 0


def test_attention_with_every_key_visible():
    """window 0: ordinary causal attention."""
    H, G, dk, dv, n = 4, 2, 64, 64, 100
    q, k, v = (rnd(n, x, 64, seed=i, dtype=BF16) for i, x in enumerate((H, G, G)))
    w = O.softmax_weights(q.double(), k.double(), 0.125, torch.ones(n, n).tril().bool())
    want = torch.stack([w[h] @ v[:, h // 2].double() for h in range(H)], 1).reshape(n, -1)
    perm = list(range(7))
    kc, vc = paged(k, v, perm, 16, BF16)
    table = torch.tensor([perm], dtype=torch.int32, device=DEV)
    pos = torch.arange(n, dtype=torch.int32, device=DEV)
    for plan in (None, ops.plan_runs([(0, n)], DEV, n - 1)):
        out = torch.zeros(n, H * dv, dtype=BF16, device=DEV)
        ops.talk_attention(q.reshape(n, -1).to(DEV), kc, vc, table, pos, torch.zeros_like(pos), pos.long(), n_q_heads=H,
                           scale=0.125, window=0, keep=0, talk=None, talk_frag=ops.talk_fragment(torch.eye(H), G).to(DEV), gate=None,
                           out_scale=1.0, max_ctx=112, scratch=ops.TalkScratch([(H, G, dv, 0, 0)], 112, DEV), out=out, plan=plan)
        assert rel(out, want) < 1.5e-2


# ----------------------------------------------------------------------------- recurrence
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("W", [24, 256, 700])
def test_mingru(dtype, W):
    """Rows form and scan form over several runs, continuing and fresh, slow and fast channels."""
    tot, R = 0, []
    for sid, pos0, n in ((2, 0, 1), (0, 5, 33), (3, 0, 64), (1, 100, 2), (4, 1, 95)):
        R.append((sid, pos0, n, tot))
        tot += n
    z, x, g = rnd(tot, W, seed=1, std=2, dtype=dtype), rnd(tot, W, seed=2, dtype=dtype), rnd(tot, W, seed=3, dtype=dtype)
    zb, xb = rnd(W, seed=4, std=3.0), rnd(W, seed=5)
    st0 = rnd(5, W, seed=6, std=5.0)
    want, end = torch.zeros(tot, W, dtype=torch.float64), st0.double().clone()
    for sid, p0, n, r0 in R:
        S = O.min_gru(z[r0 : r0 + n].double() + zb.double(), x[r0 : r0 + n].double() + xb.double(), st0[sid].double() if p0 else None)
        want[r0 : r0 + n], end[sid] = S * O.silu(g[r0 : r0 + n].double()) * 0.7, S[-1]
    y = torch.cat([z, x, g], 1).to(DEV)
    ids = torch.cat([torch.full((n,), s) for s, _, n, _ in R]).int().to(DEV)
    pos = torch.cat([torch.arange(p, p + n) for _, p, n, _ in R]).int().to(DEV)
    for plan in (None, ops.plan_runs([(r0, n) for _, _, n, r0 in R], DEV, 200)):
        st = st0.clone().to(DEV)
        out = torch.zeros(tot, W + 8, dtype=dtype, device=DEV)
        ops.mingru(y[:, :W], y[:, W : 2 * W], y[:, 2 * W :], zb.to(DEV), xb.to(DEV), seq_ids=ids, positions=pos,
                   slots=pos.long(), state=st, out_scale=0.7, out=out[:, :W], plan=plan)
        assert rel(out[:, :W], want) < (1e-5 if dtype == F32 else 8e-3)
        assert rel(st, end) < 1e-5 and out[:, W:].abs().sum() == 0


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [32, 33, 512, 513, 545, 1056, 1300])
def test_mingru_folds_the_chunks_in_front(dtype, n):
    """Runs of one to forty-one chunks, sixteen of which are folded together, behind another run's; slow channels, whose state spans them."""
    W, first = 40, 70
    z, x, g = rnd(first + n, W, seed=1, std=2, dtype=dtype), rnd(first + n, W, seed=2, dtype=dtype), rnd(first + n, W, seed=3, dtype=dtype)
    zb, xb, st0 = rnd(W, seed=4) - 6.0, rnd(W, seed=5), rnd(2, W, seed=6, std=5.0)
    S = O.min_gru(z[first:].double() + zb.double(), x[first:].double() + xb.double(), st0[1].double())
    want = S * O.silu(g[first:].double())
    ids = torch.cat([torch.zeros(first), torch.ones(n)]).int().to(DEV)
    pos = torch.cat([torch.arange(first), torch.arange(9, 9 + n)]).int().to(DEV)
    st, out = st0.clone().to(DEV), torch.zeros(first + n, W, dtype=dtype, device=DEV)
    y = torch.cat([z, x, g], 1).to(DEV)
    ops.mingru(y[:, :W], y[:, W : 2 * W], y[:, 2 * W :], zb.to(DEV), xb.to(DEV), seq_ids=ids, positions=pos, slots=pos.long(), state=st,
               out_scale=1.0, out=out, plan=ops.plan_runs([(0, first), (first, n)], DEV, 2000))
    assert rel(out[first:], want) < (1e-5 if dtype == F32 else 8e-3) and rel(st[1], S[-1]) < 1e-5


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("W,first,pairs", [(256, 0, True), (255, 0, False), (256, 1, False)])
def test_mingru_rounds_one_product(dtype, W, first, pairs):
    """(1 - z) S + z c, bit for bit: of the scan over columns that pair up z c is added unrounded, else and of decoded rows (1 - z) S.
    The gates themselves come from rows that start at c = 1: S = z."""
    n = 20
    y = rnd(n, 3 * W + first, seed=1, dtype=dtype)
    y[:, first + W : first + 2 * W] = y[:, first + W : first + 2 * W].abs()  # (u >= 0: c = u + 1/2)
    one = y.clone()
    one[:, first + W : first + 2 * W] = 0.5
    cols = lambda t: [t.to(DEV)[:, first + i * W : first + (i + 1) * W] for i in range(3)]  # noqa: E731
    none = torch.zeros(W, device=DEV)
    row = torch.arange(n, dtype=torch.int32, device=DEV)
    out = torch.empty(n, W, dtype=dtype, device=DEV)
    z = torch.zeros(n, W, device=DEV)
    ops.mingru(*cols(one), none, none, seq_ids=row, positions=torch.zeros_like(row), slots=row.long(), state=z, out_scale=1.0, out=out)
    z, c, st0 = z.cpu().numpy(), y[:, first + W : first + 2 * W].float().numpy() + np.float32(0.5), rnd(1, W, seed=2)
    for plan in (None, ops.plan_runs([(0, n)], DEV, 100)):
        st = st0.clone().to(DEV)
        ops.mingru(*cols(y), none, none, seq_ids=torch.zeros_like(row), positions=row + 5, slots=row.long(), state=st, out_scale=1.0, out=out, plan=plan)
        S = st0[0].numpy()
        for t in range(n):  # (64 bits of significand hold either sum)
            a, b = (np.float32(1) - z[t], S), (z[t], c[t])
            exact, rounded = (b, a) if plan is not None and pairs else (a, b)
            S = (np.multiply(*exact, dtype=np.longdouble) + (rounded[0] * rounded[1]).astype(np.longdouble)).astype(np.float32)
        assert np.array_equal(st[0].cpu().numpy(), S)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,dk,dv,rot,window,keep,bs", [
    (8, 4, 128, 128, 64, 1024, 4, 16),
    (6, 2, 32, 48, 16, 33, 3, 16),        # half of a fragment step rotates
    (20, 1, 64, 16, 64, 0, 0, 32),        # two column groups; every dimension rotates
    (4, 4, 96, 32, 32, 1, 17, 16),        # a window of one behind kept keys
    (4, 2, 160, 64, 160, 0, 0, 16),       # a head in two pieces, the second in part; pairs across the two
    (8, 2, 256, 32, 64, 48, 2, 16),       # two whole pieces
])
def test_talk_mingru_step(dtype, H, G, dk, dv, rot, window, keep, bs):
    """A decode step's two launches against the ops they stand for, over one set of caches: single rows, runs that start at 0, end
    at, start at and cross tile borders, a run of two chunks of tiles, inert rows between and behind them.  The cache's places of
    the step's own keys and of keys past them hold NaN before the step: the scores may take nothing from there."""
    W, n_seq, per = 40, 7, 24
    runs = [(3, 0, 1), (0, 31, 1), (5, 0, 18), (1, 90, 16), (2, 47, 2), (6, 200, 1), (4, 16, 5)]  # sequence, first position, rows
    ids, pos = [], []
    for s, p0, n in runs:
        ids += [s] * n
        pos += range(p0, p0 + n)
    rows = len(ids) + 2
    live = torch.tensor([True] * 20 + [False] + [True] * (len(ids) - 20) + [False])
    ids, pos = ids[:20] + [5] + ids[20:] + [0], pos[:20] + [0] + pos[20:] + [0]
    table = torch.randperm(n_seq * per, generator=torch.Generator().manual_seed(2)).int().view(n_seq, per)
    posT, idT = torch.tensor(pos), torch.tensor(ids)
    slots = torch.where(live, table[idT, posT // bs].long() * bs + posT % bs, -1)
    kc, vc = rnd(n_seq * per, G, bs, dk, seed=1, dtype=dtype), rnd(n_seq * per, G, dv, bs, seed=2, dtype=dtype)
    for s, p0, n in runs:
        for p in range(p0, min(per * bs, p0 + n + 40)):
            kc[table[s, p // bs], :, p % bs] = float("nan")
    A = H * dk + G * (dk + dv)
    y = rnd(rows, -(-(A + 3 * W + H) // 8) * 8, seed=3, dtype=dtype).to(DEV)
    at = (A, A + W, A + 2 * W)
    T, zb, xb, st = (rnd(*n, seed=i).to(DEV) for i, n in enumerate(((H, H), (W,), (W,), (n_seq, W))))
    rope = ops.rope_table(512, rot, 10000.0, device=DEV)
    sc = ops.TalkScratch([(H, G, dv, window, keep)], per * bs, DEV)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    meta = dict(positions=i32(pos), seq_ids=i32(ids), slots=slots.to(DEV))
    head = dict(n_q_heads=H, rot_dims=rot, rope=rope)
    att = dict(scale=0.4, window=window, keep=keep, talk=T, talk_frag=None, gate=y[:, A + 3 * W : A + 3 * W + H], out_scale=0.8,
               max_ctx=per * bs, scratch=sc)

    def run(fused):
        c = dict(k_cache=kc.clone().to(DEV), v_cache=vc.clone().to(DEV), state=st.clone())
        q, rec = torch.zeros(rows, H * dk, dtype=dtype, device=DEV), torch.zeros(rows, W, dtype=dtype, device=DEV)
        out = torch.full((rows, H * dv), float("nan"), dtype=dtype, device=DEV)
        if fused:
            ops.talk_mingru_step(y, at, zb, xb, table.to(DEV), **head, q_out=q, rec_scale=0.7, rec_out=rec, out=out, **c, **meta, **att)
        else:
            ops.qkv_cache_mingru(y, at, zb, xb, **head, q_out=q, out_scale=0.7, out=rec, **c, **meta)
            ops.talk_attention(q, c["k_cache"], c["v_cache"], table.to(DEV), n_q_heads=H, out=out, **meta, **att)
        torch.cuda.synchronize()
        return out, rec, c["state"], c["k_cache"], c["v_cache"]

    want, got = run(False), run(True)
    for a, b in zip(got[1:], want[1:]):
        assert torch.equal(torch.nan_to_num(a.float(), 1e9), torch.nan_to_num(b.float(), 1e9))
    # (the turned heads may differ by a contraction: the bounds of the attention's own test)
    assert rel(got[0], want[0].cpu()) < (5e-6 if dtype == F32 else 1.5e-2)
    assert got[0][~live].abs().sum() == 0 and sc.counters.abs().sum() == 0


# ----------------------------------------------------------------------------- the model through the engine
CFGS = {
    "odd": O.model_config(72, 101, [
        O.layer_config(6, 2, 20, 24, 12, 19, 3, 40, 56),
        O.layer_config(3, 3, 32, 16, 32, 33, 0, 24, 0, base=5000.0, scale=0.3, ls=1.1, rs=0.4),
        O.layer_config(4, 1, 48, 40, 16, 16, 17, 64, 88)], eps=1e-3),
    "even": O.model_config(384, 512, [
        O.layer_config(8, 4, 64, 64, 32, 48, 4, 256, 512),
        O.layer_config(8, 2, 128, 80, 64, 100, 1, 384, 768, base=1e6)]),
    "one": O.model_config(130, 77, [O.layer_config(1, 1, 32, 16, 2, 5, 1, 1, 33, ls=1.0, rs=1.0)]),
}
LIMIT = {F32: 2e-5, BF16: 3e-2}


def tokens(n, seed, vocab):
    return torch.randint(0, vocab, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


_MODELS = {}


def setup(name, dtype, **kw):
    if (name, dtype) not in _MODELS:
        w = O.random_weights(CFGS[name], 5)
        _MODELS[name, dtype] = (w, KabanexModel(KabanexConfig.from_json(CFGS[name]), weights=w, device=DEV, dtype=dtype))
    w, m = _MODELS[name, dtype]
    return CFGS[name], w, LLMEngine(m, **dict(dict(max_seqs=4, max_model_len=512), **kw))


_WANT = {}


def oracle(name, n, seed):
    key = (name, n, seed)
    if key not in _WANT:
        t = tokens(n, seed, CFGS[name]["vocab"])
        _WANT[key] = (t, O.forward(CFGS[name], O.random_weights(CFGS[name], 5), t))
    return _WANT[key]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(CFGS))
def test_residual_after_every_layer(name, dtype):
    cfg, w, eng = setup(name, dtype)
    t = tokens(50, 9, cfg["vocab"])
    _, res = O.forward(cfg, w, t, layers=True)
    m, seen = eng.model, []
    use_graphs, eng.use_graphs = eng.use_graphs, False
    run = m._layer
    m._layer = lambda li, bufs, M, kv, x, *a: (run(li, bufs, M, kv, x, *a), seen.append(x[:50, : cfg["width"]].clone()))
    try:
        eng.step_batch([(eng.new_sequence([]), t)], [49])
    finally:
        del m._layer
        eng.use_graphs = use_graphs
    assert len(seen) == len(res)
    for g, r in zip(seen, res):
        assert rel(g, r) < (1e-5 if dtype == F32 else 2e-2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", list(CFGS))
@pytest.mark.parametrize("cuts", [[150], [2], [16, 1], [70, 3, 2], [1], [100, 50]], ids=str)
def test_prompts_in_portions(name, dtype, cuts):
    cfg, w, eng = setup(name, dtype)
    t, want = oracle(name, 150, 1)
    seq, out, i, k = eng.new_sequence([]), [], 0, 0
    while i < len(t):
        part = t[i : i + cuts[k % len(cuts)]]
        out.append(eng.step_batch([(seq, part)], range(len(part))).clone())
        i, k = i + len(part), k + 1
    assert O.logit_error(torch.cat(out), want).max() < LIMIT[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", ["odd", "even"])
@pytest.mark.parametrize("big", [False, True])
def test_mixed_batches_with_reused_pages_and_slots(name, dtype, big):
    """Unequal requests in common steps, portions beside single tokens, requests left out of a step, pages
    and slots used again -- against each request alone.  big: steps past the step graphs' rows."""
    lens = (230, 41, 7, 64, 150, 1, 90, 33)
    need = sorted((-(-n // 64) * 4 for n in lens), reverse=True)
    cfg, w, eng = setup(name, dtype, max_seqs=3, kv_blocks=1 + sum(need[:3]))
    reqs = {n: oracle(name, n, 100 + n) for n in lens}
    live, queue, at, got, rng = {}, list(lens), {}, {n: [] for n in lens}, np.random.default_rng(1)
    sids = []
    while queue or live:
        while queue and len(live) < 3:
            n = queue.pop(0)
            live[n], at[n] = eng.new_sequence([]), 0
            sids.append(live[n].sid)
        entries = []
        for n in live:
            if len(live) > 1 and rng.random() < 0.2:
                continue
            k = int(rng.choice([1, 2, 30, 64, 100] if big else [1, 1, 2, 5, 17]))
            entries.append((n, reqs[n][0][at[n] : at[n] + k]))
        if not entries:
            continue
        lg = eng.step_batch([(live[n], p) for n, p in entries], range(sum(len(p) for _, p in entries)))
        i = 0
        for n, p in entries:
            got[n].append(lg[i : i + len(p)].clone())
            i += len(p)
            at[n] += len(p)
        for n in [n for n, _ in entries if at[n] == n]:
            eng.free_sequence(live.pop(n))
    assert len(sids) == len(lens) and len(set(sids)) == 3
    for n in lens:
        assert O.logit_error(torch.cat(got[n]), reqs[n][1]).max() < LIMIT[dtype], n


@pytest.mark.parametrize("dtype", DTYPES)
def test_long_decoding(dtype):
    """Decoding far past every window, through the captured step graph, its first replay included (the
    capture's warm-up forwards must not advance the recurrent state)."""
    t, want = oracle("even", 260, 4)
    cfg, w, eng = setup("even", dtype)
    seq = eng.new_sequence([])
    out = [eng.step_batch([(seq, t[:5])], range(5)).clone()]
    for i in range(5, 260):
        out.append(eng.step_batch([(seq, t[i : i + 1])], [0]).clone())
    assert eng.stats["graph_replays"] >= 250
    assert O.logit_error(torch.cat(out), want).max() < LIMIT[dtype]


@pytest.mark.parametrize("dtype", DTYPES)
def test_graph_replays_match_eager_steps(dtype):
    """Every replay of the step graphs against the same step run eagerly, other work in between."""
    cfg, w, ga = setup("odd", dtype)
    _, _, eb = setup("odd", dtype, use_graphs=False)
    seqs = [(ga.new_sequence([]), eb.new_sequence([])) for _ in range(3)]
    for step in range(12):
        batch = [(p, tokens(1 + (step + i) % 3, 10 * step + i, 101)) for i, p in enumerate(seqs) if (step + i) % 4]
        n = sum(len(t) for _, t in batch)
        a = ga.step_batch([(p[0], t) for p, t in batch], range(n)).clone()
        torch.cuda.synchronize()
        junk = torch.randn(256, 256, device=DEV).sum()  # noqa: F841
        b = eb.step_batch([(p[1], t) for p, t in batch], range(n)).clone()
        assert torch.equal(a, b), step
        for x, y in zip(ga.kv.state, eb.kv.state):
            assert torch.equal(x[:3], y[:3])


def test_far_keys_and_edges_in_decoding():
    """A prompt longer than the window with kept first tokens: decoded logits depend on the first tokens
    and on the last one inside the window, and not on the one just outside (no other layer carries it)."""
    cfg = O.model_config(128, 64, [O.layer_config(4, 2, 32, 32, 16, 40, 3, 16, 64)])
    w = O.random_weights(cfg, 8)
    for k in ("l0.mix.right.o",):
        w[k] = torch.zeros_like(w[k])    # the recurrence reaches past every window: taken out here
    m = KabanexModel(KabanexConfig.from_json(cfg), weights=w, device=DEV, dtype=F32)
    eng = LLMEngine(m, max_seqs=2, max_model_len=256)
    t = tokens(101, 3, 64)

    def last(tt, cut):
        s = eng.new_sequence([])
        if cut:
            eng.step_batch([(s, tt[:cut])])
            for x in tt[cut:-1]:
                eng.step_batch([(s, [x])])
            r = eng.step_batch([(s, tt[-1:])], [0]).clone()
        else:
            r = eng.step_batch([(s, tt)], [len(tt) - 1]).clone()
        eng.free_sequence(s)
        return r

    for cut in (0, 70):
        base = last(t, cut)
        for j, seen in ((0, True), (2, True), (3, False), (100 - 39, True), (100 - 40, False), (50, False)):
            tt = list(t)
            tt[j] = (tt[j] + 1) % 64
            d = float((last(tt, cut) - base).abs().max())
            assert (d > 1e-4) if seen else (d == 0), (cut, j, d)


@pytest.mark.parametrize("dtype", DTYPES)
def test_greedy_generation_through_the_scheduler(dtype):
    cfg, w, eng = setup("even", dtype, max_seqs=2)
    prompts = [tokens(n, 40 + n, 512) for n in (37, 3, 90)]
    outs = TokenScheduler(eng, token_budget=80).generate(prompts, 8)
    for p, o in zip(prompts, outs):
        want = O.forward(cfg, w, p + o)
        for i, tok in enumerate(o):  # (each token is the oracle's choice given the tokens before it, up to near-ties)
            row = want[len(p) - 1 + i]
            assert row.max() - row[tok] < (1e-4 if dtype == F32 else 0.08) * row.std(), (i, tok)


def test_sampling_at_a_temperature_is_reproducible():
    _, _, eng = setup("even", BF16, max_seqs=2)
    p = tokens(20, 1, 512)
    a, b = (TokenScheduler(eng, temperature=1.5, seed=s).generate([p], 12)[0] for s in (3, 3))
    c = TokenScheduler(eng, temperature=1.5, seed=4).generate([p], 12)[0]
    assert a == b and a != c


def test_trace_replay_command(tmp_path):
    cfg = CFGS["odd"]
    w = O.random_weights(cfg, 5)
    O.save_model(str(tmp_path / "m"), cfg, w)
    t, want = oracle("odd", 150, 1)
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": t[:100], "want": [99, 7]}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": t[100:], "want": [49]}, {"id": "b", "tokens": t[:2], "want": [1]}],
              "end": ["a", "b"]}]
    for dtype, lim in (("bfloat16", LIMIT[BF16]), ("float32", LIMIT[F32])):
        r = subprocess.run([os.path.join(ROOT, "bin", "trace_run"), "--model", str(tmp_path / "m"), "--dtype", dtype, "--out",
                            str(tmp_path / dtype), "--max-tokens", "256"], input="".join(json.dumps(s) + "\n" for s in steps),
                           capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stderr[-2000:]
        assert [x for x in r.stdout.split("\n") if x.startswith("done")] == ["done 0", "done 1"]
        got = torch.cat([torch.from_numpy(np.fromfile(tmp_path / dtype / f"{i}.f32", dtype="<f4")).view(-1, 101) for i in (0, 1)])
        assert O.logit_error(got, want[[99, 7, 149, 1]]).max() < lim


def test_intent_engine_serves_a_kabanex_preset():
    from voice_enabled_browser_automation_amd.brain.intent_engine import LLMIntentEngine
    from voice_enabled_browser_automation_amd.contracts import ParseResponse, safe_parse
    from voice_enabled_browser_automation_amd.runtime.weights import load_llm
    from voice_enabled_browser_automation_amd.tokenizer import load_tokenizer

    eng = LLMEngine(load_llm("kabanex-tiny", device=DEV), max_seqs=4, max_model_len=2048)
    brain = LLMIntentEngine(eng, load_tokenizer("llama3"), budget_chars=200, temperature=0.0)
    reqs = [{"text": s, "context": {}} for s in ("scroll down", "search wireless earbuds", "go back")]
    outs = brain.parse_many(reqs)
    assert all(safe_parse(ParseResponse, o).success for o in outs)


def test_native_path_only():
    """Nothing of the model leaves the hand-written kernels (strict native mode would raise)."""
    _, _, eng = setup("even", BF16)
    before = dict(ops.vendor_fallbacks)
    s = eng.new_sequence([])
    eng.step_batch([(s, tokens(150, 2, 512))], [149])
    eng.step_batch([(s, [1])], [0])
    assert ops.vendor_fallbacks == before


@pytest.mark.parametrize("M,N,K,D", [(1, 1024, 6144, 1000), (4, 2048, 2048, 2048), (17, 64, 128, 64), (33, 1024, 6144, 1000), (48, 2032, 2048, 2024), (64, 4096, 512, 4096), (20, 4096, 128, 4090)])
def test_norm_adds_a_projections_slices(M, N, K, D):
    """linear_parts + layernorm_f32(parts): the residual rows and their norm against float64 (one slice and many, a last
    quad that is not whole, padding columns zero)."""
    gen = torch.Generator(device="cuda").manual_seed(M)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    a, w = rnd(M, K).bfloat16(), (rnd(N, K) * K ** -0.5).bfloat16()
    w[D:] = 0
    ld = -(-D // 128) * 128
    x = torch.zeros(M, ld, device="cuda")
    x[:, :D] = rnd(M, D)
    want = x[:, :D].double() + a.double() @ w[:D].double().T
    nw, nb = rnd(D), rnd(D)
    parts = ops.linear_parts(a, ops.TiledWeight(w))
    assert parts.shape[1:] == (M, N) and (parts.shape[0] > 1) == (K > 128)
    out = torch.full((M, ld), 7.0, device="cuda", dtype=torch.bfloat16)
    ops.layernorm_f32(x, nw, nb, eps=1e-5, out=out, parts=parts)
    # (f32 sums of K bf16 products: about sqrt(K) roundings of 2^-24)
    assert rel(x[:, :D], want.cpu()) < 2e-6 and not x[:, D:].any()
    n = torch.nn.functional.layer_norm(want, (D,), nw.double(), nb.double(), 1e-5)
    assert rel(out[:, :D], n.cpu()) < 4e-3 and not out[:, D:].any()
    assert (ops.linear_parts(a[:1], ops.TiledWeight(w)) is None) == (N >= 4096)


@pytest.mark.parametrize("n", [1, 2, 4, 5, 8, 9, 15, 16, 17, 24])
@pytest.mark.parametrize("N,D", [(1024, 1022), (2048, 2048), (4096, 4090)])
def test_norm_adds_any_number_of_slices(n, N, D):
    """Batches of slices (up to 15, 7, 3 in flight by the row's width), each added once and in their order."""
    gen = torch.Generator(device="cuda").manual_seed(n)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen)  # noqa: E731
    x, parts, w = rnd(3, N), rnd(n, 3, N), rnd(D)
    x[:, D:] = 0
    parts[:, :, D:] = 0
    s = parts[0].clone()
    for k in range(1, n):
        s += parts[k]
    want = x + s
    out = torch.empty(3, N, device="cuda")
    ops.layernorm_f32(x, w, None, eps=1e-5, out=out, parts=parts)
    assert torch.equal(x, want)
    # (f32: a mean and a variance of D terms, some sqrt(D) roundings of 2^-24)
    assert rel(out[:, :D], torch.nn.functional.layer_norm(want[:, :D].double(), (D,), w.double(), None, 1e-5).cpu()) < 4e-6


def test_a_projections_slices_are_the_callers():
    """What linear_parts returned stands, whatever is launched before the norm that reads it: another projection's slices, a sum
    of slices, both captured behind it."""
    gen = torch.Generator(device="cuda").manual_seed(5)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=gen).bfloat16()  # noqa: E731
    w, v = ops.TiledWeight(rnd(1024, 4096)), ops.TiledWeight(rnd(1024, 4096))
    a, b = rnd(20, 4096), rnd(20, 4096)
    assert ops.ext().gemm_plan(0, 20, 1024, 4096)[1] > 1
    first = ops.linear_parts(a, w)
    want = first.clone()

    def others():
        return ops.linear_parts(b, v), ops.gemm(b, v, torch.empty(20, 1024, device="cuda", dtype=torch.bfloat16))

    second = others()[0]
    assert torch.equal(first, want) and not torch.equal(second, want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        kept = ops.linear_parts(a, w)
        others()
    for _ in range(3):
        g.replay()
        others()
        assert torch.equal(kept, want)
