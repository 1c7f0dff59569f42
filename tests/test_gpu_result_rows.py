"""Result rows of passes with many workgroups: the row holds the worst score of all, whether it starts at zero (every
workgroup may raise it) or already holds another call's worst."""
import struct

import pytest
import torch

pytestmark = pytest.mark.gpu


def _z(key: int) -> float:
    return struct.unpack("<f", struct.pack("<I", (int(key) >> 32) & 0xFFFFFFFF))[0]


def _holds_worst(row, scores):
    """row[0]: the largest score and a place that has it; row[1]: the same score with its noise."""
    flat = scores.reshape(-1)
    key = int(row[0])
    assert _z(key) == float(flat.max()) == _z(int(row[1]))
    assert float(flat[key & 0xFFFFFFFF]) == _z(key)


@pytest.mark.parametrize("m,k,n", [(1, 256, 128), (129, 256, 136), (1152, 128, 896), (1024, 128, 1024), (2048, 512, 6144)])
def test_linear_rows(m, k, n):
    from sdcguard_amd import LayerChecksums
    from sdcguard_amd.linear import check_linear_both
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    w = (torch.randn(n, k, device="cuda", generator=g) * 0.05).bfloat16()
    y = torch.nn.functional.linear(x, w)
    cs = LayerChecksums(w, None, 128)
    nb, mb = -(-n // 128), -(-m // 128)
    cols, rows = torch.empty(m, nb, 2, device="cuda"), torch.empty(n, mb, 2, device="cuda")
    for _ in range(3):
        state, row = check_linear_both(x, w, None, y, cs, col_scores=cols, row_scores=rows)
        _holds_worst(state.tolist(), cols)
        _holds_worst(row.tolist(), rows)
    kept = state.clone(), row.clone()
    check_linear_both(x, w, None, y, cs, state=state, row_result=row)
    assert torch.equal(state[:2], kept[0][:2]) and torch.equal(row, kept[1])
    y[m // 2, n // 2] += 64.0                                # a worse call into the same rows
    check_linear_both(x, w, None, y, cs, state=state, row_result=row, col_scores=cols, row_scores=rows)
    _holds_worst(state.tolist(), cols)
    _holds_worst(row.tolist(), rows)
    assert _z(state[0]) > _z(kept[0][0]) and _z(row[0]) > _z(kept[1][0])


@pytest.mark.parametrize("mode,m,k,n", [("fp8", 1, 64, 8), ("fp8", 130, 96, 200), ("fp8", 4032, 64, 128),
                                        ("fp8", 4096, 64, 128), ("fp8", 2048, 1024, 6144),
                                        ("fp8", 2048, 96, 6143), ("int8", 2048, 128, 6144)])
def test_quant_rows(mode, m, k, n):
    from sdcguard_amd import modes
    g = torch.Generator(device="cuda").manual_seed(m + k)
    if mode == "int8":
        a = torch.randint(-127, 128, (m, k), device="cuda", generator=g, dtype=torch.int32).to(torch.int8)
        b = torch.randint(-127, 128, (k, n), device="cuda", generator=g, dtype=torch.int32).to(torch.int8)
        c = (a.double() @ b.double()).to(torch.int32)
        c[5, 7] += 1
        c[m - 1, n - 1] -= 1
        sa = sb = None
    else:
        a = torch.randn(m, k, device="cuda", generator=g).to(torch.float8_e4m3fn)
        b = torch.randn(k, n, device="cuda", generator=g).to(torch.float8_e4m3fn)
        sa, sb = (torch.rand(s, device="cuda", generator=g) + 0.5 for s in (m, n))
        c = ((a.float() @ b.float()) * sa[:, None] * sb).bfloat16()
    consts = modes.QuantChecksums.make(b, sb)
    z = torch.empty(m, -(-n // 128), device="cuda")
    for _ in range(3):
        row = modes.quant_zscores(a, consts, c, sa=sa, scores_out=z).result.tolist()
        _holds_worst(row, z)
        assert row[2:] == [int((z > 6).sum()), 0]
    if mode == "int8":                                       # the last wrong block's place
        assert row[0] & 0xFFFFFFFF == m * z.shape[1] - 1 and row[2] == 2


def _product(m, k, n, la, lc, batch, dt, g):
    """A, B and C = A @ B (fp32), A and C in a layout: rows or columns contiguous, or rows at odd addresses."""
    lead = (batch,) if batch else ()
    a, b = (torch.randn(*lead, *s, device="cuda", generator=g).to(dt) for s in ((m, k), (k, n)))
    c = a.float() @ b.float()

    def lay(t, how):
        if how == "cols":
            return t.transpose(-1, -2).contiguous().transpose(-1, -2)
        if how == "odd":
            return torch.cat([t[..., :3], t, t[..., :2]], -1)[..., 3:3 + t.shape[-1]]
        return t
    return lay(a, la), b, lambda d: lay(c.to(d), lc)


# (each path of the expected side's GEMM before the scores: whole lines, 32- and 64-row tiles, unaligned rows, contiguous
# columns, neither, batches; below and past 64 scoring workgroups; C by rows, at odd addresses and by columns)
@pytest.mark.parametrize("m,k,n,la,lc,batch", [
    (1, 64, 128, "rows", "rows", 0), (32, 64, 64500, "rows", "rows", 0), (60, 128, 35000, "rows", "rows", 0),
    (2016, 64, 1024, "rows", "rows", 0), (2048, 64, 1024, "rows", "rows", 0), (8192, 64, 1024, "rows", "odd", 0),
    (2048, 65, 1030, "odd", "rows", 0), (5000, 90, 700, "cols", "rows", 0), (1500, 64, 3000, "rows", "cols", 0),
    (20000, 100, 300, "cols", "cols", 0), (300, 64, 500, "rows", "rows", 24), (2048, 1000, 1024, "odd", "cols", 0)])
def test_training_rows(m, k, n, la, lc, batch):
    from sdcguard_amd import matmul_zscores
    g = torch.Generator(device="cuda").manual_seed(m + n)
    a, b, c = _product(m, k, n, la, lc, batch, torch.bfloat16, g)
    c = c(torch.bfloat16)
    nb = -(-n // 128)
    z = torch.empty(max(1, batch), m, nb, 2, device="cuda")
    bad = torch.cat([c[..., :3], c], -1)[..., 3:] if lc == "odd" else c.clone(memory_format=torch.preserve_format)
    bad[..., m // 2, n // 2] += 1e4
    for out in (bad, c, bad, c):                             # (a worst call before each clean one: stale slots would hide it)
        row = matmul_zscores(a, b, out, scores_out=z).result.tolist()
        _holds_worst(row, z)
        assert row[2] == 0 and (_z(row[0]) > 6.0) == (out is bad)


@pytest.mark.parametrize("m,k,n,lc,batch", [(1, 64, 128, "rows", 0), (1008, 64, 1024, "rows", 0), (1024, 64, 1024, "rows", 0),
                                            (3000, 65, 1030, "odd", 0), (300, 40, 500, "rows", 24)])
def test_precise_rows(m, k, n, lc, batch):
    from sdcguard_amd.checksum import matmul_zscores_acc
    g = torch.Generator(device="cuda").manual_seed(m + n)
    a, b, c = _product(m, k, n, "rows", lc, batch, torch.bfloat16, g)
    c = c(torch.float32)
    z = torch.empty(max(1, batch), m, -(-n // 128), 2, device="cuda")
    bad = c.clone()
    bad[..., m // 2, n // 2] += 1e4
    for out in (bad, c, bad, c):
        row = matmul_zscores_acc(a, b, out, scores_out=z).result.tolist()
        _holds_worst(row, z)
        assert row[2] == 0 and (_z(row[0]) > 6.0) == (out is bad)
