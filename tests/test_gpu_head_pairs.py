"""GPU parity of the fp16 head past 32 rows, both groups of rows in one launch: vocabularies of one
strip, of fewer strips than blocks and of a ragged last one, both piece lengths."""
import numpy as np
import pytest

from tests.gpu_util import assert_close, dev, host

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from momij_amd.ops import Context

    c = Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("M,K,V", [(33, 2048, 16), (33, 256, 4111), (48, 2048, 4111),
                                   (64, 256, 30001), (64, 2048, 9000)])
def test_lm_head_two_groups(ctx, orc, M, K, V):
    import torch

    print(f"case: head of two row groups M={M} K={K} V={V}", flush=True)
    rng = np.random.default_rng(M + K + V)
    w = (rng.standard_normal((V, K)) * 0.02).astype(np.float16)
    x = rng.standard_normal((M, K)).astype(np.float16)
    dw, dx = dev(w), dev(x)
    am, one = (torch.full((M,), -1, dtype=torch.int32, device="cuda") for _ in range(2))
    lg, lg1 = (torch.zeros((M, V), dtype=torch.float32, device="cuda") for _ in range(2))
    lse = torch.zeros(M, dtype=torch.float32, device="cuda")
    ban = dev(np.array([0, V - 1], np.int32))
    torch.cuda.synchronize()
    ctx.lm_head_verify(dx, dw, M, K, V, am, None, lg, banned=ban, n_banned=2, temperature=0.9,
                       out_lse=lse)
    for r in range(M):  # the one-row calls, bit for bit
        ctx.lm_head_verify(dx[r:r + 1], dw, 1, K, V, one[r:r + 1], None, lg1[r:r + 1], banned=ban,
                           n_banned=2)
    ctx.sync()
    assert torch.equal(lg, lg1) and torch.equal(am, one)
    ref = orc.lm_head_logits(x, w)
    assert_close(host(lg), ref, rel_tol=1e-5, abs_tol=1e-4, what="logits")
    keep = np.ones(V, bool)
    keep[[0, V - 1]] = False
    z = ref[:, keep].astype(np.float64) / 0.9
    want = np.log(np.exp(z - z.max(1, keepdims=True)).sum(1)) + z.max(1)
    assert np.abs(host(lse) - want).max() < 3e-5  # the head's log-sum-exp bar
