"""GPU: a prompt's 64-row chunks sharing a wide pass give the same bits as passes of their own."""
import numpy as np
import pytest

from momij_amd import _lib
from momij_amd._lib import MomijError

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from momij_amd.ops import Context

    c = Context(0)
    yield c
    c.close()


def _engine(ctx, E, I, gs, alpha, top_k, capacity, n_layers=2, full=True, heads=(16, 4)):
    import torch

    from momij_amd.engine import MapleLikeConfig, VerifyEngine, random_model

    kinds = ["sliding_attention", "full" if full else "sliding_attention"] * n_layers
    wins, ropes = MapleLikeConfig.maple_layer_mix(n_layers, 96, 64, kinds)
    cfg = MapleLikeConfig(n_layers=n_layers, E=E, I=I, gs=gs, top_k=top_k, vocab=2048, window=96,
                          kv_capacity=capacity, layer_window=wins, layer_rope_dim=ropes,
                          n_heads=heads[0], n_kv_heads=heads[1])
    layers, *rest = random_model(cfg, seed=E + I)
    if alpha:  # scale alpha, bias -alpha in every group of a row
        for lw in layers:
            for nm in ("up_gate", "down"):
                m = lw["moe"]
                al = m[nm + "_s"][..., 0].contiguous()
                m[nm + "_s"] = al[..., None].expand_as(m[nm + "_s"]).contiguous()
                m[nm + "_b"] = -m[nm + "_s"]
                m[nm + "_alpha"] = al
    torch.cuda.synchronize()
    return VerifyEngine(ctx, cfg, layers, *rest), cfg


def _cache(eng, cfg):
    import torch

    class View:
        def __init__(self, p):
            self.__cuda_array_interface__ = dict(
                data=(p, False), shape=(cfg.n_kv_heads, cfg.kv_capacity, cfg.head_dim),
                typestr="<f2", version=2)

    return [torch.as_tensor(View(p), device="cuda").cpu().numpy().view(np.uint16)
            for l in range(cfg.n_layers) for p in eng.kv(l)]


# experts with one slot and with many (8 experts, all routed by every row), each group size, rows
# with and without one alpha, both down widths
@pytest.mark.parametrize("E,I,gs,alpha,top_k", [
    (64, 1024, 64, False, 8), (256, 512, 128, True, 8), (8, 1024, 128, False, 8),
    (40, 512, 64, True, 3), (16, 1024, 64, True, 4), (24, 512, 128, False, 1)])
def test_wide_equals_chunk_passes(ctx, E, I, gs, alpha, top_k):
    import torch

    print(f"case: wide prefill E={E} I={I} gs={gs} alpha={alpha} top_k={top_k}", flush=True)
    eng, cfg = _engine(ctx, E, I, gs, alpha, top_k, 640)
    rng = np.random.default_rng(E)
    logits = torch.zeros((_lib.MJ_MAX_ROWS, cfg.vocab), device="cuda")
    for n in (65, 200, 256, 257, 500):
        prompt = rng.integers(0, cfg.vocab, n).tolist()
        eng.rewind(0)
        for i in range(0, n, 64):  # passes of their own
            last = eng.step_chain_feeds(prompt[i:i + 64])
        ref = _cache(eng, cfg)
        eng.set_capture(logits=logits)
        eng.rewind(n - len(last))
        eng.step_chain_feeds(prompt[n - len(last):])
        ref_logits = logits[:len(last)].clone()
        for capture in (True, False):
            eng.set_capture(logits=logits if capture else None)
            eng.rewind(0)
            logits.zero_()
            torch.cuda.synchronize()
            assert eng.prefill(prompt) == last[-1] and eng.offset == n
            for a, b in zip(_cache(eng, cfg), ref):
                assert (a == b).all(), n
            if capture:
                assert torch.equal(logits[:len(last)], ref_logits), n
    eng.close()


@pytest.mark.parametrize("heads", [(4, 4), (8, 1), (8, 4), (16, 16), (4, 2)])
def test_wide_head_shapes(ctx, heads):
    eng, cfg = _engine(ctx, 16, 512, 128, False, 4, 320, heads=heads)
    rng = np.random.default_rng(sum(heads))
    for n in (65, 250, 300):
        prompt = rng.integers(0, cfg.vocab, n).tolist()
        eng.rewind(0)
        for i in range(0, n, 64):
            last = eng.step_chain_feeds(prompt[i:i + 64])
        ref = _cache(eng, cfg)
        eng.rewind(0)
        assert eng.prefill(prompt) == last[-1]
        for a, b in zip(_cache(eng, cfg), ref):
            assert (a == b).all(), n
    eng.close()


def test_wide_refusals(ctx):
    """A bad token, or a prompt past the capacity, is refused at its chunk, the chunks before it
    committed."""
    eng, cfg = _engine(ctx, 16, 512, 64, False, 4, 320)
    prompt = [int(t) for t in np.random.default_rng(1).integers(0, cfg.vocab, 400)]
    for bad, at, status in ((prompt[:150] + [cfg.vocab] + prompt[150:200], 128, 4),
                            ([-1] + prompt[:100], 0, 4), (prompt, 320, 7)):
        eng.rewind(0)
        with pytest.raises(MomijError) as e:
            eng.prefill(bad)
        assert e.value.status == status and eng.offset == at, (e.value, eng.offset)
    eng.close()


def test_wide_in_a_wrapped_ring(ctx):
    """Passes of more rows than the ring has slots past the window, from offsets all around it."""
    eng, cfg = _engine(ctx, 16, 512, 64, False, 4, 160, full=False)
    rng = np.random.default_rng(5)
    prompt = rng.integers(0, cfg.vocab, 700).tolist()
    for i in range(0, 700, 50):
        last = eng.step_chain_feeds(prompt[i:i + 50])
    ref = _cache(eng, cfg)
    for at in (0, 64, 150, 299, 444):
        eng.rewind(0)
        for i in range(0, at, 64):
            eng.step_chain_feeds(prompt[i:min(i + 64, at)])
        assert eng.prefill(prompt[at:]) == last[-1]
        for a, b in zip(_cache(eng, cfg), ref):
            assert (a == b).all(), at
    eng.close()


def test_wide_past_the_deep_line(ctx):
    """Full attention from passes whose parts attend together to passes whose keys are too many."""
    eng, cfg = _engine(ctx, 16, 512, 64, False, 4, 2944)
    prompt = np.random.default_rng(8).integers(0, cfg.vocab, 2900).tolist()
    for i in range(0, 2900, 64):
        last = eng.step_chain_feeds(prompt[i:i + 64])
    ref = _cache(eng, cfg)
    for at in (0, 2200):
        eng.rewind(0)
        for i in range(0, at, 64):
            eng.step_chain_feeds(prompt[i:min(i + 64, at)])
        assert eng.prefill(prompt[at:]) == last[-1]
        for a, b in zip(_cache(eng, cfg), ref):
            assert (a == b).all(), at
    eng.close()


def test_wide_abort_leaves_its_start_valid(ctx):
    """A prefill cut off in a wide pass goes on from the model's offset to the uninterrupted state:
    what the pass had overwritten of the window before it is back.  Compared 100 rows further on,
    with every one of them still in the cache: the first of them read the keys that went back."""
    import threading
    import time

    eng, cfg = _engine(ctx, 64, 1024, 64, False, 8, 160, n_layers=6, full=False)
    prompt = np.random.default_rng(6).integers(0, cfg.vocab, 3000).tolist()
    eng.prefill(prompt)
    eng.rewind(0)
    t0 = time.perf_counter()
    eng.prefill(prompt)
    t_full = time.perf_counter() - t0
    cut = 0
    for k in range(8):
        eng.rewind(0)
        timer = threading.Timer(t_full * (0.15 + 0.08 * k), lambda: ctx.set_abort(True))
        timer.start()
        try:
            eng.prefill(prompt)
        except MomijError as e:
            assert e.status == 5
            cut += 1
        timer.join()
        ctx.set_abort(False)
        print(f"cut at offset {eng.offset}", flush=True)
        to = eng.offset + 100
        if to <= len(prompt):
            got = eng.prefill(prompt[to - 100:to])
            kv = _cache(eng, cfg)
            eng.rewind(0)
            assert eng.prefill(prompt[:to]) == got
            for a, b in zip(_cache(eng, cfg), kv):
                assert (a == b).all()
    assert cut > 0
    eng.close()


def test_wide_failure_leaves_its_start_valid(ctx):
    """The same where the pass ends with an error: a wait that ran out its bound in an earlier call
    (forced by a bound of 0) is reported by the prefill that follows it."""
    import torch

    from momij_amd import synth

    eng, cfg = _engine(ctx, 16, 512, 64, False, 4, 160, full=False)
    rng = np.random.default_rng(9)
    # 100 rows from 150: the last 36 take the slots of keys that the first ones need, and every row
    # is still in the cache at the end
    prompt = rng.integers(0, cfg.vocab, 250).tolist()
    want = eng.prefill(prompt)
    ref = _cache(eng, cfg)
    mw = synth.moe_weights(rng, 64, 2048, 1024, 64)
    dmw = {n: (torch.from_numpy(v.view(np.int32) if v.dtype == np.uint32 else v).cuda()
               if isinstance(v, np.ndarray) else v) for n, v in mw.items()}
    x = torch.from_numpy(synth.normal_f16(rng, (1, 2048))).cuda()
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    reported = 0
    for _ in range(4):
        eng.rewind(0)
        eng.prefill(prompt[:150])
        ctx.set_wait_limit(0)
        try:
            # one row: half of the blocks have no up item and check down items' rows at once
            ctx.moe_block(dmw, x, y, 1, 3)
        finally:
            ctx.set_wait_limit(1 << 17)
        try:
            got = eng.prefill(prompt[150:])
        except MomijError as e:
            assert e.status == 6 and eng.offset == 150, e
            reported += 1
            got = eng.prefill(prompt[150:])
        assert got == want
        for a, b in zip(_cache(eng, cfg), ref):
            assert (a == b).all()
    assert reported > 0
    eng.close()
