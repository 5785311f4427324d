"""GPU: op-level calls that take their parameters with the launch, and penalty histories through
pinned buffers -- issued back to back, with no wait between calls whose parameters differ."""
import numpy as np
import pytest

from momij_amd import synth
from tests.gpu_util import assert_close, dev, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from momij_amd.ops import Context

    c = Context(0)
    yield c
    c.close()


def _trees(rng, M):
    return [list(range(-1, M - 1)), [-1] + [int(rng.integers(0, i)) for i in range(1, M)],
            [-1] + [0] * (M - 1)]


@pytest.mark.parametrize("M,rope,gs", [(1, 64, 64), (9, 128, 128), (64, 32, 64), (17, 0, 64)])
def test_attn_block_back_to_back(ctx, orc, M, rope, gs):
    import torch

    print(f"case: attention calls back to back M={M} rope={rope}", flush=True)
    rng = np.random.default_rng(M)
    H, nQ, nKV, D, win = 2048, 16, 4, 128, 96
    C = win + 64
    cfg = dict(H=H, nQ=nQ, nKV=nKV, D=D, rope_dim=rope, rope_base=1e6, eps=1e-6, window=win, C=C,
               gs=gs)
    aw = synth.attn_weights(rng, H, nQ, nKV, D, gs)
    daw = {k: dev(v) for k, v in aw.items()}
    calls = []
    for L, par in zip((0, 77, 500), _trees(rng, M)):
        h, kc, vc = (synth.normal_f16(rng, s) for s in ((M, H), (nKV, C, D), (nKV, C, D)))
        calls.append((L, par, h, kc, vc, dev(h), dev(kc), dev(vc)))
    torch.cuda.synchronize()
    for L, par, _, _, _, dh, dk, dv in calls:  # the caller's list may go right after the call
        ctx.attn_block(cfg, daw, dh, dk, dv, L, list(par), M)
    ctx.sync()
    for L, par, h, kc, vc, dh, dk, dv in calls:
        ref = orc.attn_block(cfg, aw, h, kc, vc, L, np.asarray(par, np.int32))
        ref = ref[0] if isinstance(ref, tuple) else ref
        assert_close(host(dh), ref, what=f"L={L}")


@pytest.mark.parametrize("n", [1, 2, 33, 64])
def test_accept_greedy_back_to_back(ctx, orc, n):
    import torch

    rng = np.random.default_rng(n)
    runs = []
    for par in _trees(rng, n) * 2:
        tok, am = (rng.integers(0, 3, n).astype(np.int32) for _ in range(2))
        runs.append((par, tok, am, dev(tok), dev(am),
                     torch.full((2 + 2 * n,), -7, dtype=torch.int32, device="cuda")))
    torch.cuda.synchronize()
    for par, _, _, dt, da, out in runs:
        ctx.accept_greedy(dt, par, da, n, out)
    ctx.sync()
    for par, tok, am, _, _, out in runs:
        cur, path, emit = 0, [0], []
        while True:
            kid = next((c for c in range(n) if par[c] == cur and tok[c] == am[cur]), None)
            if kid is None:
                break
            emit.append(int(tok[kid]))
            path.append(kid)
            cur = kid
        o = host(out).tolist()
        assert o[:2] == [len(path) - 1, int(am[cur])]
        assert o[2:2 + len(path)] == path and o[2 + n:2 + n + len(path)] == emit + [int(am[cur])]


def test_histories_back_to_back(ctx, orc):
    """Five calls in flight with histories of growing and shrinking length: each sees its own."""
    import torch

    rng = np.random.default_rng(3)
    V, rows = 5000, 4
    lg = (rng.standard_normal((rows, V)) * 3).astype(np.float32)
    dl = dev(lg)
    opts = dict(top_p=0.8, rep=1.4, pres=0.3, freq=0.2)
    draft = lg.argmax(1)[: rows - 1].astype(np.int32)
    dd = dev(draft)
    runs = []
    for n in (3, 4000, 1, 900, 4999):
        ht = np.sort(rng.choice(V, n, replace=False)).astype(np.int32)
        hc = rng.integers(0, 5, n).astype(np.int32)
        runs.append((ht, hc, torch.empty(2, dtype=torch.int32, device="cuda")))
    torch.cuda.synchronize()
    for i, (ht, hc, out) in enumerate(runs):
        ctx.accept_sampled_ex(dl, rows, V, dd, 1, 9, i, out, 0.9, hist=(ht, hc), **opts)
    ctx.sync()
    for i, (ht, hc, out) in enumerate(runs):
        u = orc.verify_uniforms(9, i, rows)
        ref = orc.accept_sampled_ex(lg, draft, 0.9, 1, u, hist_tok=ht, hist_cnt=hc, **opts)
        assert tuple(int(v) for v in host(out)) == ref, i


def test_history_under_capture_is_refused(ctx):
    """A penalty history is host data of the call: a captured call would replay another's."""
    import torch

    from momij_amd._lib import MomijError

    lg = torch.randn((1, 64), device="cuda")
    d = torch.zeros(1, dtype=torch.int32, device="cuda")
    out = torch.empty(2, dtype=torch.int32, device="cuda")
    hist = (np.arange(4, dtype=np.int32), np.ones(4, np.int32))
    call = dict(rep=1.2, hist=hist)
    ctx.accept_sampled_ex(lg, 1, 64, d, 0, 1, 1, out, 1.0, **call)  # scratch in place
    ctx.sync()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(ctx.stream):
        g.capture_begin(capture_error_mode="thread_local")
        try:
            with pytest.raises(MomijError):
                ctx.accept_sampled_ex(lg, 1, 64, d, 0, 1, 1, out, 1.0, **call)
        finally:
            out.zero_()  # a captured graph of this alone
            g.capture_end()
    torch.cuda.synchronize()
    ctx.accept_sampled_ex(lg, 1, 64, d, 0, 1, 2, out, 1.0, **call)
    ctx.sync()


@pytest.mark.parametrize("op", ["attn_block", "accept_greedy"])
def test_host_trees_under_capture_are_refused(ctx, op):
    """The draft tree (and an attention block's position) is host data of the call too."""
    import torch

    from momij_amd._lib import MomijError

    rng = np.random.default_rng(4)
    H, nQ, nKV, D = 2048, 16, 4, 128
    cfg = dict(H=H, nQ=nQ, nKV=nKV, D=D, rope_dim=64, rope_base=1e6, eps=1e-6, window=96, C=160,
               gs=64)
    aw = {k: dev(v) for k, v in synth.attn_weights(rng, H, nQ, nKV, D, 64).items()}
    h, kc, vc = (dev(synth.normal_f16(rng, s)) for s in ((3, H), (nKV, 160, D), (nKV, 160, D)))
    tok, am = dev(np.array([1, 2, 3], np.int32)), dev(np.array([2, 3, 9], np.int32))
    out = torch.zeros(8, dtype=torch.int32, device="cuda")

    def call():
        if op == "attn_block":
            ctx.attn_block(cfg, aw, h, kc, vc, 10, [-1, 0, 0], 3)
        else:
            ctx.accept_greedy(tok, [-1, 0, 1], am, 3, out)

    torch.cuda.synchronize()
    call()
    ctx.sync()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(ctx.stream):
        g.capture_begin(capture_error_mode="thread_local")
        try:
            with pytest.raises(MomijError):
                call()
        finally:
            out.zero_()  # a captured graph of this alone
            g.capture_end()
    torch.cuda.synchronize()
    call()
    ctx.sync()
    if op == "accept_greedy":
        assert host(out).tolist() == [2, 9, 0, 1, 2, 2, 3, 9]


def test_an_aborted_call_leaves_no_fault(ctx):
    """A wait that ran out its bound (forced by a bound of 0) before a call that reports an abort:
    the call after it reports neither."""
    import torch

    from momij_amd._lib import MomijError

    rng = np.random.default_rng(6)
    mw = {k: (dev(v) if isinstance(v, np.ndarray) else v)
          for k, v in synth.moe_weights(rng, 64, 2048, 1024, 64).items()}
    x = dev(synth.normal_f16(rng, (1, 2048)))
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    faults = 0
    for abort in (False, True, False, True):
        ctx.set_wait_limit(0)
        try:
            # one row: half of the blocks have no up item and check down items' rows at once
            ctx.moe_block(mw, x, y, 1, 3)
        finally:
            ctx.set_wait_limit(1 << 17)
        torch.cuda.synchronize()
        if abort:
            ctx.set_abort(True)
            ctx.set_abort(False)
        try:
            ctx.sync()
        except MomijError as e:
            assert e.status == (5 if abort else 6), e
            faults += not abort
        else:
            assert not abort
        ctx.sync()
    assert faults > 0  # the bound does report
