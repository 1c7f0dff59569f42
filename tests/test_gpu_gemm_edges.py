"""The expected side's GEMMs at the edges of their tiles and depth parts, against the oracle's scores (the serving
tests' tolerance)."""
import numpy as np
import pytest
import torch

from oracle import abft, serve_check
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


def _operand(rows, cols, layout, g, t, std):
    """(rows, cols) of dtype t in a layout: row- or column-contiguous, at an odd offset of odd-strided storage, or with
    neither stride one."""
    if layout == "rows":
        return (torch.randn(rows, cols, generator=g) * std).to(t).cuda()
    if layout == "cols":
        return (torch.randn(cols, rows, generator=g) * std).to(t).cuda().t()
    if layout == "odd":
        return (torch.randn(rows, cols + 5, generator=g) * std).to(t).cuda()[:, 3:3 + cols]
    if layout == "cols_odd":
        return (torch.randn(cols, rows + 5, generator=g) * std).to(t).cuda()[:, 3:3 + rows].t()
    if layout == "expanded":
        return (torch.randn(1, cols, generator=g) * std).to(t).cuda().expand(rows, cols)
    return (torch.randn(rows, 2 * cols, generator=g) * std).to(t).cuda()[:, ::2]


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("la", ["rows", "cols", "odd", "cols_odd", "expanded", "strided"])
@pytest.mark.parametrize("m,k,n,lb", [(1, 1, 1, "rows"), (3, 64, 130, "cols"), (37, 63, 128, "rows"),
                                      (128, 128, 256, "cols"), (131, 65, 300, "odd"), (257, 1030, 513, "cols_odd"),
                                      (514, 320, 4300, "rows")])
def test_training_operand_layouts(m, k, n, lb, la, dt):
    """Every layout of A through the GEMM its strides and depth pick, every checksum's score against the oracle's."""
    from sdcguard_amd import matmul_zscores
    g = torch.Generator().manual_seed(m + k + n)
    t = torch.bfloat16 if dt == "bf16" else torch.float16
    A, B = _operand(m, k, la, g, t, 1.0), _operand(k, n, lb, g, t, 0.1)
    C = (A.float().cpu() @ B.float().cpu()).to(t)
    scores = torch.full((1, m, -(-n // 128), 2), -7.0, device="cuda")
    row = matmul_zscores(A, B, C.cuda(), scores_out=scores).result.tolist()
    o = abft.zscores(A.float().cpu().numpy(), B.float().cpu().numpy(), C.float().numpy(), dtype=dt, seed=1)
    z = scores.cpu().numpy().reshape(-1)
    ok = z_close(z, o.z.reshape(-1), gemm_slack(o.csb, o.den).reshape(-1))
    assert ok.all(), (np.nonzero(~ok)[0][:5], z[~ok][:5], o.z.reshape(-1)[~ok][:5])
    assert row[2] == 0


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("n,block", [(5, 128), (9, 8), (130, 7), (300, 100), (257, 127), (1000, 128)])
@pytest.mark.parametrize("batch", [0, 3])
def test_narrow_blocks(n, block, batch, dt):
    """Blocks narrower than 128, rows at any 2-byte address, fewer columns than one 16-byte load."""
    from sdcguard_amd import matmul_zscores
    m, k = 67, 40
    g = torch.Generator().manual_seed(n + block)
    t = torch.bfloat16 if dt == "bf16" else torch.float16
    lead = (batch,) if batch else ()
    A, B = torch.randn(*lead, m, k, generator=g).to(t), (torch.randn(*lead, k, n, generator=g) * 0.1).to(t)
    C = (A.float() @ B.float()).to(t)
    scores = torch.full((max(1, batch), m, -(-n // min(block, n)), 2), -7.0, device="cuda")
    matmul_zscores(A.cuda(), B.cuda(), C.cuda(), block=block, scores_out=scores)
    o = abft.zscores(A.float().numpy(), B.float().numpy(), C.float().numpy(), block=block, dtype=dt, seed=1)
    z = scores.cpu().numpy().reshape(-1)
    ok = z_close(z, o.z.reshape(-1), gemm_slack(o.csb, o.den).reshape(-1))
    assert ok.all(), (np.nonzero(~ok)[0][:5], z[~ok][:5], o.z.reshape(-1)[~ok][:5])


def _scores_match(A, B, C, dt, **kw):
    """Every score and the count of unjudged ones against the oracle's."""
    from sdcguard_amd import matmul_zscores
    m, n = C.shape
    scores = torch.full((1, m, -(-n // 128), 2), -7.0, device="cuda")
    row = matmul_zscores(A, B, C, scores_out=scores, **kw).result.tolist()
    o = abft.zscores(*(t.float().cpu().numpy() for t in (A, B, C)), dtype=dt, seed=1, **kw)
    z = scores.cpu().numpy().reshape(-1)
    ok = z_close(z, o.z.reshape(-1), gemm_slack(o.csb, o.den).reshape(-1))
    assert ok.all(), (np.nonzero(~ok)[0][:5], z[~ok][:5], o.z.reshape(-1)[~ok][:5])
    assert row[2] == int((o.z < 0).sum())
    return z.reshape(m, -1), o


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("m,k,n,la,lc", [(131, 65, 300, "odd", "rows"), (130, 64, 257, "rows", "odd"),
                                         (257, 130, 513, "cols_odd", "cols"), (67, 5, 9, "rows", "rows"),
                                         (37, 63, 130, "strided", "strided")])
def test_nonfinite_at_the_edges(m, k, n, la, lc, bad, dt):
    """NaN and infinities at the ends of rows, columns, narrow blocks and depth, in each operand: the pairs that hold
    them get the oracle's verdict, and rows and blocks beside them are judged as without them."""
    g = torch.Generator().manual_seed(m + k)
    t = torch.bfloat16 if dt == "bf16" else torch.float16
    A, B, C = _operand(m, k, la, g, t, 1.0), _operand(k, n, "rows", g, t, 0.1), _operand(m, n, lc, g, t, 1.0)
    C.copy_((A.float() @ B.float()).to(t))
    clean, _ = _scores_match(A, B, C, dt)
    last = n - 1
    for T, i, j in ((C, m - 1, last), (C, 0, 0), (C, m // 2, last - last % 128 - 1 if n > 128 else 0), (C, 3, last - last % 128),
                    (A, m - 1, k - 1), (A, 0, k - 1), (A, m - 2, 0)):
        kept = T[i, j].clone()
        T[i, j] = bad
        z, _ = _scores_match(A, B, C, dt)
        others = torch.arange(m).numpy() != i
        assert np.array_equal(z[others], clean[others])
        T[i, j] = kept
    for i, j in ((k - 1, last), (0, 0)):
        kept = B[i, j].clone()
        B[i, j] = bad
        z, o = _scores_match(A, B, C, dt)
        blocks = np.arange(z.shape[1]) // 2 != j // 128
        assert np.array_equal(z[:, blocks], clean[:, blocks])
        B[i, j] = kept


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("la", ["rows", "odd", "cols", "strided"])
@pytest.mark.parametrize("lc", ["rows", "cols"])
def test_many_planes(la, lc, dt):
    """A deep product of few rows and columns: more depth parts than a scoring pass loads at once, for both ways of reading C."""
    from sdcguard_amd import _lib
    m, k, n = 300, 8256, 260
    g = torch.Generator().manual_seed(9)
    t = torch.bfloat16 if dt == "bf16" else torch.float16
    A, B, C = _operand(m, k, la, g, t, 1.0), _operand(k, n, "rows", g, t, 0.02), _operand(m, n, lc, g, t, 1.0)
    C.copy_((A.float() @ B.float()).to(t))
    C[m - 1, n - 1] += 8.0
    z, o = _scores_match(A, B, C, dt)
    assert (z > 6).any()


@pytest.mark.parametrize("dt,scale", [("fp16", 1e-4), ("fp16", 4e-4), ("bf16", 3e-10)])
@pytest.mark.parametrize("n,lc", [(256, "rows"), (300, "rows"), (300, "odd"), (9, "rows"), (300, "cols"), (300, "strided")])
def test_subnormal_outputs(n, lc, dt, scale):
    """fp16 outputs below the normal range, and bf16 ones whose squares are below fp32's, keep their sums and norms."""
    m, k = 70, 64
    g = torch.Generator().manual_seed(n)
    t = torch.bfloat16 if dt == "bf16" else torch.float16
    A, B, C = _operand(m, k, "rows", g, t, scale), _operand(k, n, "rows", g, t, scale), _operand(m, n, lc, g, t, 1.0)
    C.copy_((A.float() @ B.float()).to(t))
    _scores_match(A, B, C, dt, abs_floor=1e-30)
