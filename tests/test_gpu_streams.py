"""Tensors kept on a layer's constants (its parts in other orders, its packed table), used from several streams, inside a
captured graph and in inference mode.  Constants made elsewhere come without them: the first check makes them."""
import pytest
import torch

pytestmark = pytest.mark.gpu

M, K, N = 16, 1024, 384


def _elsewhere(t):
    """The same constants as another program would hand them over: nothing kept on them."""
    return t.as_strided(t.shape, t.stride()).clone(memory_format=torch.preserve_format)


def _serving(dt, by_row):
    from sdcguard_amd import LayerChecksums
    from sdcguard_amd.serve import check_static_impl
    g = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn(M, K, device="cuda", generator=g).to(dt)
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.05).to(dt)
    y = torch.nn.functional.linear(x, w)
    parts, *rest = LayerChecksums(w, None, 128).tensors(False)
    parts = parts.contiguous() if by_row else _elsewhere(parts)
    rest[7] = _elsewhere(rest[7])

    def check(state, scores):
        check_static_impl(x, y, parts, *rest, state, 0, 6.0, 1e-30, scores_out=scores)
    return check, (M, N // 128, 2), (parts, rest[7])


def _quant(kind):
    from sdcguard_amd import modes
    g = torch.Generator(device="cuda").manual_seed(K + 1)
    if kind == "int8":
        a, b = (torch.randint(-127, 128, s, device="cuda", generator=g, dtype=torch.int32).to(torch.int8)
                for s in ((M, K), (K, N)))
        c = (a.double() @ b.double()).to(torch.int32)
        c[3, 200] += 1
    else:
        a, b = (torch.randn(*s, device="cuda", generator=g).to(torch.float8_e4m3fn) for s in ((M, K), (K, N)))
        c = a.float() @ b.float()
    own = modes.QuantChecksums.make(b)
    consts = modes.QuantChecksums(own.kind, K, N, own.block, _elsewhere(own.parts), own.bfrob, own.bcol)

    def check(state, scores):
        modes.quant_zscores(a, consts, c, scores_out=scores, out=state)
    return check, (M, N // 128), (consts.parts,)


CASES = {"bf16": lambda: _serving(torch.bfloat16, False), "fp16": lambda: _serving(torch.float16, False),
         "by_row": lambda: _serving(torch.bfloat16, True), "int8": lambda: _quant("int8"), "fp8": lambda: _quant("fp8")}


def _buffers(shape):
    return torch.zeros(4, dtype=torch.int64, device="cuda").view(1, 4) if len(shape) == 3 else \
        torch.zeros(4, dtype=torch.int64, device="cuda"), torch.full(shape, -7.0, device="cuda")


def _forget(owners):
    for o in owners:
        for name in list(vars(o)):
            delattr(o, name)


@pytest.mark.parametrize("case", sorted(CASES))
def test_first_check_on_one_stream_next_on_another(case):
    """The second stream's check waits for what the first one's check is still to make."""
    check, shape, owners = CASES[case]()
    state, want = _buffers(shape)
    check(state, want)
    want = want.clone()
    assert (want != -7.0).all()
    one, two = torch.cuda.Stream(), torch.cuda.Stream()
    big = torch.randn(4096, 4096, device="cuda")
    bufs = [_buffers(shape) for _ in range(3)]
    for s, b in zip((one, two), bufs):                       # (both streams' workspaces are there)
        with torch.cuda.stream(s):
            check(*b)
    torch.cuda.synchronize()
    _forget(owners)
    with torch.cuda.stream(one):
        for _ in range(20):
            big = big @ big * 1e-3                           # some milliseconds
        check(*bufs[0])
    with torch.cuda.stream(two):
        bufs[1][1].fill_(-7.0)
        check(*bufs[1])
        check(*bufs[1])
    two.synchronize()
    assert torch.equal(bufs[1][1], want)
    one.synchronize()
    assert torch.equal(bufs[0][1], want)
    check(*bufs[2])
    assert torch.equal(bufs[2][1], want)


@pytest.mark.parametrize("case", sorted(CASES))
def test_first_check_inside_a_graph(case):
    """What a capture made is not taken by later calls, and each replay makes its own."""
    check, shape, owners = CASES[case]()
    state, want = _buffers(shape)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        check(state, want)
    torch.cuda.synchronize()
    want = want.clone()
    _forget(owners)
    gstate, got = _buffers(shape)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        check(gstate, got)
    state, eager = _buffers(shape)
    check(state, eager)                                      # before any replay
    assert torch.equal(eager, want)
    for _ in range(3):
        got.fill_(-7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        check(state, eager)
        assert torch.equal(eager, want)


@pytest.mark.parametrize("k", [64, 128, 200, 512])
def test_constants_of_inference_mode(k):
    """Tensors of inference mode have no version counter."""
    from sdcguard_amd import LayerChecksums
    from sdcguard_amd.serve import check_static_impl
    with torch.inference_mode():
        x, w = torch.randn(M, k, device="cuda").bfloat16(), torch.randn(N, k, device="cuda").bfloat16()
        y = torch.nn.functional.linear(x, w)
        cs = LayerChecksums(w, None, 128)
        state, z = torch.zeros(1, 4, dtype=torch.int64, device="cuda"), torch.full((M, 3, 2), -7.0, device="cuda")
        check_static_impl(x, y, *cs.tensors(False), state, 0, 6.0, 1e-30, scores_out=z)
        again = torch.full_like(z, -7.0)
        check_static_impl(x, y, _elsewhere(cs.parts), *cs.tensors(False)[1:], state, 0, 6.0, 1e-30, scores_out=again)
    assert (z >= 0).all() and float(z.max()) < 6.0 and float((z - again).abs().max()) < 1e-2
    assert int(state[0, 2]) == 2


@pytest.mark.parametrize("query", ["raw", "stream"])
def test_current_stream_handle(query, monkeypatch):
    """The handle of torch's raw query, and of the stream object where a torch has no such query."""
    from sdcguard_amd import _lib
    if query == "stream":
        monkeypatch.setattr(_lib, "_current_raw_stream", None)
    t, side = torch.zeros(1, device="cuda"), torch.cuda.Stream()
    assert _lib.stream_of(t) == torch.cuda.current_stream().cuda_stream == torch.cuda.default_stream().cuda_stream
    with torch.cuda.stream(side):
        assert _lib.stream_of(t) == side.cuda_stream
        assert _lib._raw_stream(torch.device("cuda")) == side.cuda_stream
