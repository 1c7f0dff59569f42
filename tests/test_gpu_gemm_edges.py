"""The expected side's GEMMs at the edges of their tiles and depth parts, against the oracle's scores (the serving
tests' tolerance)."""
import numpy as np
import pytest
import torch

from oracle import serve_check
from tests.test_gpu_serve import run_gpu
from tests.test_oracle_golden import gemm_slack, z_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("m", [1, 32, 33, 64, 65, 129, 260])
@pytest.mark.parametrize("k,n", [(64, 128), (128, 200), (448, 1000), (704, 4224), (2112, 8200)])
def test_serving_rows_and_depths(m, k, n, dt):
    """Row tiles of 32, 64 and 128 with their remainders; depths of one segment (fewer than the waves), of uneven
    shares, and of several parts; outputs of one column tile, a narrower last block, and several tiles."""
    g = torch.Generator().manual_seed(m * 7 + k + n)
    t = torch.bfloat16 if dt == "bf16" else torch.float16
    x = torch.randn(m, k, generator=g).to(t)
    W = (torch.randn(n, k, generator=g) * 0.05).to(t)
    y = (x.float() @ W.float().t()).to(t)
    xf, Wf, yf = (v.float().numpy() for v in (x, W, y))
    zs, st, _ = run_gpu(xf, Wf, None, yf, dt)
    o = serve_check.check_static(xf, yf, serve_check.layer_constants(Wf, None, 128, dt, seed=1), dtype=dt, seed=1)
    ok = z_close(zs.reshape(-1), o.z.reshape(-1), gemm_slack(o.csb, o.den).reshape(-1))
    assert ok.all(), (np.nonzero(~ok)[0][:5], zs.reshape(-1)[~ok][:5], o.z.reshape(-1)[~ok][:5])
    assert st[0, 2] == 1 and st[0, 3] == 0
