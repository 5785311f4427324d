"""GPU parity of the penalties at the edges of a row's slices and of the history's search: every
token bit for bit the oracle's, the caller's logits untouched."""
import numpy as np
import pytest

from tests.gpu_util import dev, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from momij_amd.ops import Context

    c = Context(0)
    yield c
    c.close()


# fewer ids than slices, rows whose length is no multiple of 4, the widest row; histories of one
# id, of one round of requests, one more, and of a search
@pytest.mark.parametrize("V", [20, 33, 4096, 40001, 196608])
@pytest.mark.parametrize("n_hist", [0, 1, 2048, 2049, 30000])
def test_penalties(ctx, orc, V, n_hist):
    import torch

    print(f"case: penalties V={V} n_hist={n_hist}", flush=True)
    rng = np.random.default_rng(V + n_hist)
    rows = 9
    lg = (rng.standard_normal((rows, V)) * 2).astype(np.float32)
    tok = np.sort(rng.choice(V, min(n_hist, V), replace=False)).astype(np.int32)
    if n_hist:  # the ends of slices among the history
        span = (V // 4 + 31) // 32 * 4 if V % 4 == 0 else (V + 31) // 32
        tok[0], tok[-1] = min(0, tok[0]), V - 1
        if len(tok) > 4 and V > 4 * span:
            tok = np.unique(np.concatenate([tok, [span - 1, span, 2 * span]])).astype(np.int32)
    cnt = rng.integers(0, 4, len(tok)).astype(np.int32)
    # drafts the rows favour: repeated, in the history and not
    draft = rng.integers(0, V, rows - 1).astype(np.int32)
    draft[3] = draft[1]
    if len(tok):
        draft[2], draft[6] = tok[0], tok[-1]
    for r in range(rows - 1):
        lg[r, draft[r]] += 12.0
    dl, dd = dev(lg), dev(draft)
    for trial, (rep, pres, freq, top_p) in enumerate([(1.3, 0.0, 0.0, 1.0), (1.0, 0.4, 0.7, 0.9),
                                                      (0.8, -0.2, 0.1, 1.0)]):
        out = torch.empty(2, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        kw = dict(top_p=top_p, rep=rep, pres=pres, freq=freq)
        ctx.accept_sampled_ex(dl, rows, V, dd, 1, 11, trial, out, 0.9,
                              hist=(tok, cnt) if len(tok) else None, **kw)
        ctx.sync()
        u = orc.verify_uniforms(11, trial, rows)
        ref = orc.accept_sampled_ex(lg, draft, 0.9, 1, u, hist_tok=tok, hist_cnt=cnt, **kw)
        assert tuple(int(v) for v in host(out)) == ref, (trial, V, n_hist)
    assert (host(dl).view(np.uint32) == lg.view(np.uint32)).all()


@pytest.mark.parametrize("V", [1, 31, 33, 4096, 40001, 196608])
@pytest.mark.parametrize("rows", [1, 9, 64])
def test_without_penalties(ctx, orc, V, rows):
    """The row maxima alone: fewer ids than slices, rows of no multiple of 4 and rows that start
    off a 16-byte line, the maximum in the first and the last id."""
    import torch

    print(f"case: no penalties V={V} rows={rows}", flush=True)
    rng = np.random.default_rng(V + rows)
    lg = (rng.standard_normal((rows, V)) * 2).astype(np.float32)
    draft = rng.integers(0, V, rows - 1).astype(np.int32)
    for r in range(rows - 1):
        lg[r, draft[r]] += 12.0
    lg[0, 0] = 30.0
    lg[-1, V - 1] = 40.0
    buf = torch.zeros(rows * V + 4, dtype=torch.float32, device="cuda")
    dd = dev(draft) if rows > 1 else torch.zeros(1, dtype=torch.int32, device="cuda")
    for off, top_p in ((0, 1.0), (0, 0.8), (1, 1.0)):
        dl = buf[off:off + rows * V]
        dl.copy_(dev(lg).reshape(-1))
        out = torch.empty(2, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        ctx.accept_sampled_ex(dl, rows, V, dd, 1, 5, off, out, 0.9, top_p=top_p)
        ctx.sync()
        u = orc.verify_uniforms(5, off, rows)
        ref = orc.accept_sampled_ex(lg, draft, 0.9, 1, u, top_p=top_p)
        assert tuple(int(v) for v in host(out)) == ref, (off, top_p)
