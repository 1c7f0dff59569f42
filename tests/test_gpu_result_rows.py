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


@pytest.mark.parametrize("m,k,n", [(1, 256, 128), (129, 256, 136), (2048, 512, 6144)])
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


@pytest.mark.parametrize("mode,m,k,n", [("fp8", 1, 64, 8), ("fp8", 130, 96, 200), ("fp8", 2048, 1024, 6144),
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
