"""GPU parity of the tile gather's slots, which every block forms from the pairs' expert ids: parts
of an expert with many pairs, pairs without an expert, column blocks with fewer than four (eight)
tiles, and the MoE launch over those slots, against the oracle."""
import numpy as np
import pytest

from momij_amd import synth
from tests.gpu_util import assert_close, dev, host

pytestmark = pytest.mark.gpu

# One fp16 rounding of the result, of either sum: 2 * 2^-11 / sqrt(12) of it on average, a third of
# the bound.
REL = 1e-3


@pytest.fixture(scope="module")
def ctx():
    from momij_amd.ops import Context

    c = Context(0)
    yield c
    c.close()


def _ids(rng, kind, P, E):
    if kind == "one":  # every pair on one expert: more than 64, in parts
        return np.full(P, E - 1, np.int32)
    ids = rng.integers(0, E, P).astype(np.int32)
    if kind == "some":  # pairs that have no expert are left out
        ids[:: 3] = -1
        ids[1:: 7] = 256
    elif kind == "last":  # the last pair alone, after 511 without an expert
        ids[:-1] = -5
    return ids


@pytest.mark.parametrize("M,ktop,E,K,N,gs,kind,add", [
    (64, 8, 256, 512, 64, 64, "any", False),     # 512 pairs over every expert a launch takes
    (64, 8, 3, 1024, 48, 64, "any", False),      # 170 pairs an expert; three tiles of eight
    (64, 8, 2, 2048, 16, 128, "one", False),     # 512 pairs on one expert, one tile
    (64, 1, 1, 2048, 80, 64, "one", True),       # dense rows with residual, five tiles
    (17, 1, 4, 512, 144, 128, "any", True),
    (9, 1, 1, 1024, 2064, 64, "one", True),
    (33, 2, 16, 2048, 208, 64, "some", False),
    (64, 8, 64, 512, 32, 64, "last", False),
    (2, 1, 4, 2048, 5632, 64, "any", False),     # the fewest pairs that take the tile kernel
    (16, 4, 8, 1536, 48, 64, "some", False),     # the general kernel (K = 1536), same table rules
    (5, 8, 256, 4096, 32, 128, "any", False),
])
def test_gather_slots(ctx, orc, M, ktop, E, K, N, gs, kind, add):
    import torch

    print(f"case: slots M={M} ktop={ktop} E={E} K={K} N={N} gs={gs} {kind} add={add}", flush=True)
    rng = np.random.default_rng(M * 1000 + N)
    P = M * ktop
    w, s, b = synth.qweight(rng, (E,), N, K, gs)
    x = synth.normal_f16(rng, (M, K))
    ids = _ids(rng, kind, P, E)
    y0 = synth.normal_f16(rng, (P, N))
    ok = (ids >= 0) & (ids < 256)
    ref = orc.qmm2(x, w, s, b, np.where(ok, ids, 0).astype(np.int32), M, ktop, K, N, gs)
    if add:
        ref = (y0.astype(np.float32) + ref.astype(np.float32)).astype(np.float16)
    ref[~ok] = y0[~ok]
    y, dx, dw, ds, db, di = dev(y0), dev(x), dev(w), dev(s), dev(b), dev(ids)
    torch.cuda.synchronize()
    ctx.gather_qmm2(dx, dw, ds, db, di, y, M, ktop, K, N, gs, epilogue=int(add))
    ctx.sync()
    got = host(y)
    assert (got[~ok] == y0[~ok]).all()
    rel, _ = assert_close(got, ref, what="slots")
    assert rel < REL


def _off(a, by):
    """a on the device, `by` elements past the start of a buffer of its own."""
    import torch

    t = dev(a)
    buf = torch.empty(t.numel() + by, dtype=t.dtype, device="cuda")
    buf[by:].copy_(t.reshape(-1))
    return buf[by:]


@pytest.mark.parametrize("M,ktop,E,K,N,gs,add", [
    (5, 4, 8, 2048, 48, 64, False), (33, 2, 4, 512, 80, 128, False),
    (17, 1, 2, 512, 128, 128, True), (9, 1, 1, 1024, 2048, 64, True),
])
@pytest.mark.parametrize("woff,soff", [(1, 0), (0, 1), (2, 4)])
def test_gather_operands_off_a_line(ctx, orc, M, ktop, E, K, N, gs, add, woff, soff):
    """Codes, scales and biases that start off a 16-byte line (views into a larger buffer)."""
    import torch

    print(f"case: off a line M={M} K={K} N={N} gs={gs} add={add} {woff} {soff}", flush=True)
    rng = np.random.default_rng(M + K + N)
    P = M * ktop
    w, s, b = synth.qweight(rng, (E,), N, K, gs)
    x = synth.normal_f16(rng, (M, K))
    ids = rng.integers(0, E, P).astype(np.int32)
    y0 = synth.normal_f16(rng, (P, N))
    ref = orc.qmm2(x, w, s, b, ids, M, ktop, K, N, gs)
    if add:
        ref = (y0.astype(np.float32) + ref.astype(np.float32)).astype(np.float16)
    y, dx, di = dev(y0), dev(x), dev(ids)
    dw, ds, db = _off(w, woff), _off(s, soff), _off(b, soff)
    torch.cuda.synchronize()
    ctx.gather_qmm2(dx, dw, ds, db, di, y, M, ktop, K, N, gs, epilogue=int(add))
    ctx.sync()
    rel, _ = assert_close(host(y), ref, what="off a line")
    assert rel < REL


@pytest.mark.parametrize("E,I,gs,M,alpha", [
    (64, 512, 64, 1, False), (64, 512, 64, 16, True), (64, 512, 128, 32, False),  # ranked, I 512
    (64, 1024, 64, 33, False), (64, 512, 64, 64, True),  # the first rows past the ranked forms
    (72, 1024, 64, 1, False), (256, 512, 64, 5, True), (256, 1024, 128, 64, False),
    (8, 1024, 64, 64, False),  # every row on every expert: 64 pairs of each
    # five pairs an expert and just fewer: 16-wave blocks, and two of eight
    (40, 512, 128, 25, True), (40, 1024, 128, 25, False), (40, 512, 64, 24, False),
])
def test_moe_slots(ctx, orc, E, I, gs, M, alpha):
    import torch

    print(f"case: moe slots E={E} I={I} gs={gs} M={M} alpha={alpha}", flush=True)
    rng = np.random.default_rng(E + I + M)
    H = 2048
    mw = synth.moe_weights(rng, E, H, I, gs)
    if alpha:
        for k, n in (("up_gate", 2 * I), ("down", H)):
            a = rng.uniform(0.005, 0.02, (E, n)).astype(np.float16)
            mw[k + "_s"] = np.repeat(a[..., None], mw[k + "_s"].shape[-1], -1)
            mw[k + "_b"] = -mw[k + "_s"]
            mw[k + "_alpha"] = a
    x = synth.normal_f16(rng, (M, H))
    ref, ri, rs = orc.moe_block(mw, x, prenorm=True, residual=True)
    dmw = {k: (dev(v) if isinstance(v, np.ndarray) else v) for k, v in mw.items()}
    dx, y = dev(x), torch.empty((M, H), dtype=torch.float16, device="cuda")
    inds = torch.empty((M, 8), dtype=torch.int32, device="cuda")
    sc = torch.empty((M, 8), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    for _ in range(2):  # the second call finds the first one's scratch
        ctx.moe_block(dmw, dx, y, M, 3, inds, sc)
    ctx.sync()
    assert (host(inds) == ri).all()
    assert_close(host(y), ref, what="moe")
    # a row's result does not depend on the rows that share its pass: the one-row call, bit for bit
    y1 = torch.empty((1, H), dtype=torch.float16, device="cuda")
    for r in {0, M // 2, M - 1}:
        xr = dx[r:r + 1].contiguous()
        torch.cuda.synchronize()
        ctx.moe_block(dmw, xr, y1, 1, 3)
        ctx.sync()
        assert torch.equal(y1[0], y[r])


@pytest.mark.parametrize("H,E,I,gs,k,M", [
    (2048, 12, 1024, 64, 4, 2), (2048, 60, 512, 128, 8, 33), (2048, 4, 2048, 64, 2, 64),  # both
    (4096, 16, 1024, 64, 4, 9), (4096, 64, 512, 128, 8, 64), (4096, 12, 2048, 64, 3, 17),  # down
    (2048, 16, 1536, 64, 4, 5), (2048, 10, 1536, 128, 4, 40),  # up
    (4096, 12, 1536, 64, 8, 17), (4096, 16, 4096, 128, 2, 3),  # neither
])
def test_moe_shapes_without_the_routed_launch(ctx, orc, H, E, I, gs, k, M):
    """Shapes the fused router does not take (experts not a multiple of 8, H 4096) or that lack a
    tile kernel for one product: either product on the tile kernel, the other on the general one,
    both, or neither."""
    import torch

    print(f"case: moe shape H={H} E={E} I={I} gs={gs} k={k} M={M}", flush=True)
    rng = np.random.default_rng(H + E + I + M)
    mw = synth.moe_weights(rng, E, H, I, gs, top_k=k)
    x = synth.normal_f16(rng, (M, H))
    ref, ri, _ = orc.moe_block(mw, x, prenorm=True, residual=True)
    dmw = {n: (dev(v) if isinstance(v, np.ndarray) else v) for n, v in mw.items()}
    dx, y = dev(x), torch.empty((M, H), dtype=torch.float16, device="cuda")
    inds = torch.empty((M, k), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    for _ in range(2):  # the second call finds the first one's scratch
        ctx.moe_block(dmw, dx, y, M, 3, inds)
    ctx.sync()
    assert (host(inds) == ri).all()
    rel, _ = assert_close(host(y), ref, what="moe")
    assert rel < 5e-3  # fp16 between the stages, as the block's other shapes


@pytest.mark.parametrize("E,I,gs,M", [
    (16, 512, 64, 40), (40, 1024, 64, 64), (256, 512, 128, 17), (12, 1024, 64, 20),  # from ids
    (64, 1024, 64, 9), (64, 1024, 64, 24), (64, 512, 64, 12),  # ranked in the product's launch
])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_a_row_that_overflowed_keeps_to_itself(ctx, E, I, gs, M, bad):
    """A row whose router logits are NaN still picks experts that exist (and, by the fused router,
    distinct ones), and the rows that share its pass come out as without it, bit for bit."""
    import torch

    print(f"case: overflowed row E={E} I={I} gs={gs} M={M} {bad}", flush=True)
    rng = np.random.default_rng(E + I + M)
    H, k = 2048, 8
    mw = synth.moe_weights(rng, E, H, I, gs, top_k=k)
    dmw = {n: (dev(v) if isinstance(v, np.ndarray) else v) for n, v in mw.items()}
    x = synth.normal_f16(rng, (M, H))
    r = M // 2
    outs = []
    for v in (None, bad):
        xv = x.copy()
        if v is not None:
            xv[r, 5] = v
        dx, y = dev(xv), torch.empty((M, H), dtype=torch.float16, device="cuda")
        inds = torch.full((M, k), -1, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        ctx.moe_block(dmw, dx, y, M, 3, inds)
        ctx.sync()
        outs.append((host(y).view(np.uint16), host(inds)))
    (y0, i0), (y1, i1) = outs
    rest = np.arange(M) != r
    assert (y0[rest] == y1[rest]).all() and (i0[rest] == i1[rest]).all()
    assert i1[r].min() >= 0 and i1[r].max() < E
    assert E % 8 or len(set(i1[r].tolist())) == k
