"""GPU: attention over chunks, over groups of chunks a block, and with a pass's query tiles over
several blocks: the split of the work changes no bit of a row."""
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


# keys around a group's edge (256) and the line past which groups are taken (40 chunks); rows
# around a tile (4 rows), two tiles (a block's) and the widest pass
@pytest.mark.parametrize("M,L,window,rope", [
    (9, 2431, 0, 0), (13, 2560, 0, 64), (64, 2600, 0, 128), (33, 4095, 2600, 64),
    (17, 1023, 1024, 32), (64, 250, 0, 64), (5, 3, 0, 64)])
def test_rows_equal_one_row_passes(ctx, orc, M, L, window, rope):
    import torch

    print(f"case: attention split M={M} L={L} window={window} rope={rope}", flush=True)
    rng = np.random.default_rng(M * L)
    H, nQ, nKV, D, gs = 2048, 16, 4, 128, 64
    C = window + 64 if window else (L + M + 63) // 64 * 64
    cfg = dict(H=H, nQ=nQ, nKV=nKV, D=D, rope_dim=rope, rope_base=1e6, eps=1e-6, window=window,
               C=C, gs=gs)
    aw = synth.attn_weights(rng, H, nQ, nKV, D, gs)
    daw = {k: dev(v) for k, v in aw.items()}
    h, kc, vc = (synth.normal_f16(rng, s) for s in ((M, H), (nKV, C, D), (nKV, C, D)))
    dh, dk, dv = dev(h), dev(kc), dev(vc)
    one, k1, v1 = dev(h), dev(kc), dev(vc)
    torch.cuda.synchronize()
    ctx.attn_block(cfg, daw, dh, dk, dv, L, None, M)
    for r in range(M):
        ctx.attn_block(cfg, daw, one[r:r + 1], k1, v1, L + r, None, 1)
    ctx.sync()
    for got, ref in ((dh, one), (dk, k1), (dv, v1)):
        assert (host(got).view(np.uint16) == host(ref).view(np.uint16)).all()
    tree = [-1] + [int(rng.integers(max(0, i - 6), i)) for i in range(1, M)]
    for parents in (list(range(-1, M - 1)), tree):
        ref = orc.attn_block(cfg, aw, h, kc, vc, L, np.asarray(parents, np.int32))
        dh, dk, dv = dev(h), dev(kc), dev(vc)
        torch.cuda.synchronize()
        ctx.attn_block(cfg, daw, dh, dk, dv, L, parents, M)
        ctx.sync()
        assert_close(host(dh), ref[0], what=f"M={M} L={L}")


# query heads a KV head of 1, 2, 3, 4, 8 and 16; the o-projection's widths of the tile kernel (512,
# 1024, 2048) and of the general one; rows around its 16-row groups
@pytest.mark.parametrize("nQ,nKV,gs,M,L,window", [
    (4, 4, 64, 17, 300, 0), (4, 1, 128, 1, 70, 96), (8, 4, 128, 5, 0, 0), (8, 1, 64, 64, 2600, 0),
    (8, 8, 64, 33, 100, 96), (12, 4, 128, 16, 500, 96), (16, 1, 64, 40, 65, 0),
    (32, 4, 128, 13, 2500, 0), (32, 2, 64, 64, 129, 96)])
def test_head_shapes(ctx, orc, nQ, nKV, gs, M, L, window):
    import torch

    print(f"case: attention heads {nQ}/{nKV} gs={gs} M={M} L={L} window={window}", flush=True)
    rng = np.random.default_rng(nQ * M + L)
    H, D = 2048, 128
    C = window + 64 if window else (L + M + 63) // 64 * 64
    cfg = dict(H=H, nQ=nQ, nKV=nKV, D=D, rope_dim=64, rope_base=1e6, eps=1e-6, window=window, C=C,
               gs=gs)
    aw = synth.attn_weights(rng, H, nQ, nKV, D, gs)
    daw = {k: dev(v) for k, v in aw.items()}
    h, kc, vc = (synth.normal_f16(rng, s) for s in ((M, H), (nKV, C, D), (nKV, C, D)))
    tree = [-1] + [int(rng.integers(max(0, i - 6), i)) for i in range(1, M)]
    for parents in (list(range(-1, M - 1)), tree):
        ref = orc.attn_block(cfg, aw, h, kc, vc, L, np.asarray(parents, np.int32))
        dh, dk, dv = dev(h), dev(kc), dev(vc)
        torch.cuda.synchronize()
        ctx.attn_block(cfg, daw, dh, dk, dv, L, parents, M)
        ctx.sync()
        rel, _ = assert_close(host(dh), ref[0], what=f"{nQ}/{nKV} M={M}")
        assert rel < 5e-3  # fp16 between the block's stages
        slots = [(L + r) % C for r in range(M)]
        assert_close(host(dk)[:, slots], ref[1][:, slots], what="new K")
        assert_close(host(dv)[:, slots], ref[2][:, slots], what="new V")
