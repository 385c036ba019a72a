"""Device memory that a call allocates for itself belongs to the stream it
launches on: dropped, it goes back to that stream and to no other."""
import threading

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
