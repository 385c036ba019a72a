"""GPU parity of the fp32 attention forward where its 32-key blocks share out
unevenly over the waves and workgroups of a query block, against float64.

Bound per element: scores are float32 sums of D products, so |ds| <= (D + 4)
2^-24 scale sum |q k|; a weight's relative error is 2 |ds| plus the exponentials'
2^-22, one more 2^-22 for each of the N / 32 rescales; O sums N products. With w
the weights, |error| <= (2 (2 max |ds| + (N / 32 + 2) 2^-22) + (N + 8) 2^-24)
sum w |v|."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

U = 2.0 ** -24


def _cuda():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def _inputs(heads, N, D, dev, seed=41):
    g = torch.Generator("cpu").manual_seed(seed)
    # keys that grow along the sequence: the running maximum moves block by block
    ramp = torch.linspace(0.2, 2.0, N).view(1, 1, N, 1)
    q, k, v = (torch.randn((1, heads, N, D), generator=g) for _ in range(3))
    return q.to(dev), (k * ramp).to(dev), v.to(dev)


def _check(got, q, k, v, what):
    N, D = q.shape[2:]
    scale = D ** -0.5
    q64, k64, v64 = (t.double() for t in (q, k, v))
    w = torch.softmax(scale * (q64 @ k64.transpose(2, 3).contiguous()), -1)
    ds = (D + 4) * U * scale * (q64.abs() @ k64.abs().transpose(2, 3).contiguous()).amax(-1, keepdim=True)
    bound = (2 * (2 * ds + (N // 32 + 2) * 2.0 ** -22) + (N + 8) * U) * (w @ v64.abs())
    err = (got.double() - w @ v64).abs()
    print(f"[parity] fp32 blocks {what}: max {float(err.max()):.2e}", flush=True)
    assert bool((err <= bound).all())


CASES = [
    # heads, N: 32-key blocks per wave
    (1, 32),       # one wave, one block
    (2, 64),       # two waves
    (3, 96),       # three of four waves have one
    (1, 128),      # one each
    (2, 160),      # two and one; from here on split over workgroups
    (1, 512),      # one each in four parts
    (4, 320),
    (1, 1056),     # 33 blocks over 32 waves
    (3, 1184),     # two parts, four and five
    (40, 224),     # more workgroups than compute units
]


@pytest.mark.parametrize("kt", [False, True], ids=["natural", "kt"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("heads,N", CASES)
def test_fp32_blocks_parity(heads, N, D, kt):
    dev = _cuda()
    from grammar.attention import flash_attention_fwd
    print(f"[case] fp32 blocks heads={heads} N={N} D={D} kt={kt}", flush=True)
    q, k, v = _inputs(heads, N, D, dev)
    out = torch.full((1, heads, N + 1, D + 8), float("nan"), device=dev)
    kk = k.transpose(2, 3).contiguous() if kt else k
    flash_attention_fwd(q, kk, v, k_transposed=kt, out=out[:, :, :N, :D])
    again = flash_attention_fwd(q, kk, v, k_transposed=kt)
    torch.cuda.synchronize()
    assert torch.equal(out[:, :, :N, :D], again)
    assert torch.isnan(out[:, :, N:]).all() and torch.isnan(out[..., D:]).all()
    _check(again, q, k, v, (heads, N, D, kt))


@pytest.mark.parametrize("kt", [False, True], ids=["natural", "kt"])
def test_fp32_blocks_wide_row_strides(kt):
    """Rows of V and K^T 2^27 elements apart: past the 32-bit lane offsets."""
    dev = _cuda()
    from grammar.attention import flash_attention_fwd
    N = D = 64
    row = 1 << 27
    need = (63 * row + 2 * D) * 4
    if torch.cuda.mem_get_info(dev)[0] < need + (4 << 30):
        pytest.skip("needs 34 GB of device memory")
    print(f"[case] fp32 wide row strides kt={kt}", flush=True)
    q, k, v = _inputs(1, N, D, dev)
    buf = torch.empty(need // 4, device=dev)
    vw = buf.as_strided((1, 1, N, D), (row, row, row, 1))
    vw.copy_(v)
    kk = k
    if kt:
        kk = buf.as_strided((1, 1, D, N), (row, row, row, 1), D)
        kk.copy_(k.transpose(2, 3))
    got = flash_attention_fwd(q, kk, vw, k_transposed=kt)
    torch.cuda.synchronize()
    _check(got, q, k, v, ("wide", kt))
    del buf, vw, kk
    torch.cuda.empty_cache()


@pytest.mark.parametrize("heads,N,D", [(1, 512, 64), (4, 320, 64), (3, 1184, 128)])
def test_fp32_split_without_memory_for_its_workspace(heads, N, D):
    """A key split whose workspace cannot be allocated runs unsplit and reports
    success, and the failed allocation is not found by a later call."""
    dev = _cuda()
    from grammar import runtime as rt
    from grammar.attention import flash_attention_fwd
    print(f"[case] fp32 without a workspace heads={heads} N={N} D={D}", flush=True)
    q, k, v = _inputs(heads, N, D, dev)
    split = flash_attention_fwd(q, k, v)
    rt.check(rt.lib().gr_selftest_f32_no_workspace(1))
    try:
        whole = flash_attention_fwd(q, k, v)
        assert "workspace" in rt.last_error()            # the hook was reached
    finally:
        rt.check(rt.lib().gr_selftest_f32_no_workspace(0))
    again = flash_attention_fwd(q, k, v)
    torch.cuda.synchronize()
    _check(whole, q, k, v, ("no workspace", heads, N, D))
    assert torch.equal(split, again)


def test_fp32_graph_replay_beside_eager_splits():
    """A captured split's partials are not those of eager calls that split in
    other shapes on the capturing stream: replayed on another stream beside them,
    both keep their results."""
    dev = _cuda()
    from grammar.attention import bind_flash_attention
    graph_in, eager_in = _inputs(1, 512, 64, dev), _inputs(4, 320, 64, dev, seed=42)
    s, t = torch.cuda.Stream(), torch.cuda.Stream()
    print("[case] fp32 graph replay beside eager splits", flush=True)
    with torch.cuda.stream(s):
        s.wait_stream(torch.cuda.default_stream())
        run, out = bind_flash_attention(*graph_in, stream=s)
        eager, eout = bind_flash_attention(*eager_in, stream=s)
        run()
        eager()
        s.synchronize()
        want, ewant = out.clone(), eout.clone()
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            run()
    for _ in range(20):
        out.zero_()
        eout.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(t):
            for _ in range(8):
                graph.replay()
        for _ in range(8):
            eager()
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(eout, ewant)
