"""GPU parity of the nucleus selection at its edges: widths about its blocks of 2048 ids and 1024-id
sums, targets of nothing and of almost everything, rows whose kept mass is one id or a tie group
cut at its last id.  Every token bit for bit the oracle's."""
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


@pytest.mark.parametrize("V", [16, 17, 1023, 1025, 2047, 2048, 2049, 40001, 196608])
@pytest.mark.parametrize("shape", ["flat", "peaked", "ties", "wide"])
def test_nucleus_edges(ctx, orc, V, shape):
    import torch

    print(f"case: nucleus V={V} {shape}", flush=True)
    rng = np.random.default_rng(V)
    lg = rng.standard_normal((1, V)).astype(np.float32)
    if shape == "peaked":
        lg[0, V - 1] = 60.0  # one id holds the whole mass
    elif shape == "ties":
        lg = np.round(lg)  # few values: the cut falls in a tie group, or at one's end
    elif shape == "wide":
        lg *= 40.0  # most e underflow to zero; masses below 2^-40 truncate
    out = torch.empty(2, dtype=torch.int32, device="cuda")
    dl, dd = dev(lg), dev(np.zeros(1, np.int32))
    for trial, top_p in enumerate([0.0, 1e-6, 0.25, 0.5, 0.9, 0.99999]):
        torch.cuda.synchronize()
        ctx.accept_sampled_ex(dl, 1, V, dd, 0, 5, trial, out, 0.8, top_p=top_p)
        ctx.sync()
        u = orc.verify_uniforms(5, trial, 1)
        ref = orc.accept_sampled_ex(lg, np.zeros(0, np.int32), 0.8, 0, u, top_p=top_p)
        assert tuple(int(v) for v in host(out)) == ref, (V, shape, top_p)
