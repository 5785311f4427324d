"""GPU: the first call after the context's scratch has grown gives what the next one gives.

The scratch is cleared when it is allocated.  The clear must be through before the call's own
kernels write there, whatever else the device is doing: here the default stream, which the library's
streams do not wait for, is busy for a few to some hundred microseconds when the call is made."""
import pytest

pytestmark = pytest.mark.gpu


def _calls():
    """name: call(ctx, busy) -> out tensors, of the op-level entries, at shapes whose scratch is
    large: the clear then takes longer than the first kernels."""
    import torch

    from momij_amd import synth

    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    n = lambda *s: torch.randn(s, generator=gen, device="cuda").half()
    H, nQ, nKV, D, gs, M, L = 2048, 16, 4, 128, 64, 64, 6000
    q = lambda lead, N, K: synth.torch_qweight(gen, lead, N, K, gs)
    qw, qs, qb = q((), (nQ + 2 * nKV) * D, H)
    ow, os_, ob = q((), H, nQ * D)
    aw = dict(norm_w=n(H), qkv_w=qw, qkv_s=qs, qkv_b=qb, q_norm_w=n(D), k_norm_w=n(D), o_w=ow,
              o_s=os_, o_b=ob)
    cfg = dict(H=H, nQ=nQ, nKV=nKV, D=D, rope_dim=64, rope_base=1e6, eps=1e-6, window=0, C=L + M,
               gs=gs)
    h, kc, vc = n(M, H), n(nKV, L + M, D), n(nKV, L + M, D)

    def attn(ctx, busy):
        out = h.clone(), kc.clone(), vc.clone()
        torch.cuda.synchronize()
        torch.cuda._sleep(busy)
        ctx.attn_block(cfg, aw, *out, L, None, M)
        return out

    E, I = 16, 1024
    mw = dict(norm_w=n(H), router_w=(0.02 * n(E, H)), E=E, top_k=8, H=H, I=I, gs=gs, eps=1e-6)
    for name, N, K in (("up_gate", 2 * I, H), ("down", H, I)):
        mw[name + "_w"], mw[name + "_s"], mw[name + "_b"] = q((E,), N, K)

    def moe(ctx, busy):
        out = torch.empty_like(h)
        torch.cuda.synchronize()
        torch.cuda._sleep(busy)
        ctx.moe_block(mw, h, out, M, 3)
        return (out,)

    V, rows = 151936, 64
    logits = torch.randn((rows, V), generator=gen, device="cuda")
    draft = logits.argmax(1)[: rows - 1].to(torch.int32).contiguous()
    logits[torch.arange(rows - 1), draft.long()] += 14.0

    def accept(ctx, busy):
        out = torch.empty(2, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        torch.cuda._sleep(busy)
        ctx.accept_sampled_ex(logits, rows, V, draft, 1, 3, 9, out, 0.9, top_p=0.9, pres=0.01)
        return (out,)

    x, ids = n(512, H), torch.zeros(512, dtype=torch.int32, device="cuda")

    def gather(ctx, busy):
        out = torch.empty((512, qw.shape[0]), dtype=torch.float16, device="cuda")
        torch.cuda.synchronize()
        torch.cuda._sleep(busy)
        ctx.gather_qmm2(x, qw, qs, qb, ids, out, 512, 1, H, qw.shape[0], gs)
        return (out,)

    return dict(attn=attn, moe=moe, accept=accept, gather=gather)


def test_first_call_after_growth():
    import torch

    from momij_amd.ops import Context

    wrong = []
    for name, call in _calls().items():
        for busy in (1, 4000, 16000, 32000, 64000, 96000, 128000, 192000, 256000, 512000):  # clocks
            ctx = Context(0)
            first = call(ctx, busy)
            ctx.sync()
            torch.cuda.synchronize()
            again = call(ctx, 1)
            ctx.sync()
            if not all(torch.equal(a, b) for a, b in zip(first, again)):
                wrong.append((name, busy))
            ctx.close()
    assert not wrong, wrong
