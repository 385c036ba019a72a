"""Device memory that a call allocates for itself belongs to the stream it
launches on: dropped, it goes back to that stream and to no other."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _cuda():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.device("cuda:0")


def _free_bytes(handle):
    """Bytes the caching allocator holds free for the stream `handle`."""
    return sum(b["size"] for seg in torch.cuda.memory_snapshot() if seg["stream"] == handle
               for b in seg["blocks"] if b["state"] == "inactive")


def test_the_null_streams_handle_is_the_default_stream():
    dev = _cuda()
    from grammar import runtime as rt
    from grammar.gemm import gemm
    assert torch.cuda.default_stream(dev).cuda_stream == 0
    assert rt.torch_stream(0, dev).cuda_stream == 0
    size = 40 << 20
    ws = rt.workspace(size, dev, 0)
    ptr = ws.data_ptr()
    del ws
    assert torch.empty(size, dtype=torch.uint8, device=dev).data_ptr() == ptr
    a, b = torch.randn(24, 4096, device=dev).half(), torch.randn(4096, 1376, device=dev).half()
    assert rt.lib().gr_gemm_workspace(rt.GR_F16, 1, 24, 1376, 4096) > 0
    assert torch.equal(gemm(a, b, stream=0), gemm(a, b))


def _decode(stream):
    from grammar.attention import flash_attention_decode
    q, kv = torch.randn(4, 8, 32, 128, device="cuda").half(), torch.randn(4, 8, 2048, 128, device="cuda").half()
    return 8 * 4 * 8 * 32 * 130 * 4, lambda: flash_attention_decode(q, kv, kv, splits=8, stream=stream)


def _decode_default_splits(stream):
    from grammar.attention import decode_splits, flash_attention_decode
    q, kv = torch.randn(1, 64, 4, 128, device="cuda").half(), torch.randn(1, 64, 4096, 128, device="cuda").half()
    s = decode_splits(1, 64, 4, 4096)
    assert s > 1
    return s * 64 * 4 * 130 * 4, lambda: flash_attention_decode(q, kv, kv, stream=stream)


def _bwd(stream):
    from grammar import runtime as rt
    from grammar.attention import flash_attention_bwd, flash_attention_fwd_train
    q = torch.randn(2, 1024, 64, 64, device="cuda").half().transpose(1, 2)      # copies of 16 MiB are made
    o, lse = flash_attention_fwd_train(q, q, q)
    o = o.transpose(1, 2).contiguous().transpose(1, 2)
    return int(rt.lib().gr_attn_bwd_workspace(2, 64, 1024, 64)) + 5 * q.numel() * 2, \
        lambda: flash_attention_bwd(q, q, q, o, o, lse, stream=stream)


def _mlp(stream):
    from grammar import runtime as rt
    from grammar.gemm import mlp_fwd
    x, w1, w2 = (torch.randn(*s, device="cuda").half() / 16 for s in ((24, 2048), (2048, 32768), (32768, 2048)))
    split = int(rt.lib().gr_mlp_fwd_workspace(rt.GR_F16, 24, 2048, 32768))
    return 24 * 32768 * 2 + split, lambda: mlp_fwd(x, w1, w2, stream=stream)


@pytest.mark.parametrize("raw", [False, True], ids=["stream", "handle"])
@pytest.mark.parametrize("call", [_decode, _decode_default_splits, _bwd, _mlp], ids=lambda f: f.__name__[1:])
def test_scratch_goes_back_to_the_launch_stream(call, raw):
    dev = _cuda()
    side = torch.cuda.Stream()
    print(f"[case] scratch of {call.__name__} raw={raw}", flush=True)
    torch.manual_seed(3)
    size, run = call(side.cuda_stream if raw else side)
    torch.manual_seed(3)
    want = call(None)[1]()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = _free_bytes(0), _free_bytes(side.cuda_stream)
    got = run()
    torch.cuda.synchronize()
    assert _free_bytes(side.cuda_stream) - before[1] >= size
    for g, w in zip(got if isinstance(got, tuple) else (got,), want if isinstance(want, tuple) else (want,)):
        assert torch.equal(g, w)


def test_per_thread_streams_do_not_share_memory():
    """hipStreamPerThread is one handle for another stream in every host
    thread: what one thread drops with work in flight, no other thread gets."""
    dev = _cuda()
    import threading
    from grammar import runtime as rt
    from grammar.gemm import gemm
    size, handle = 48 << 20, 2
    a, b = torch.randn(24, 4096, device=dev).half(), torch.randn(4096, 1376, device=dev).half()
    want = gemm(a, b)
    torch.cuda.synchronize()
    got, dropped, checked = {}, threading.Event(), threading.Event()

    def first():
        ws = rt.workspace(size, dev, handle)
        with torch.cuda.stream(rt.torch_stream(handle, dev)):
            torch.cuda._sleep(50_000_000)
        got["first"] = ws.data_ptr()
        del ws
        got["busy"] = not rt.torch_stream(handle, dev).query()
        dropped.set()
        checked.wait(30)
        got["c"] = gemm(a, b, stream=handle)
        rt.torch_stream(handle, dev).synchronize()

    def second():
        dropped.wait(30)
        got["second"] = rt.workspace(size, dev, handle).data_ptr()
        checked.set()

    threads = [threading.Thread(target=f) for f in (first, second)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert got["busy"] and got["second"] != got["first"]
    assert torch.equal(got["c"], want)
