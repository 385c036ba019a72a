"""GPU parity of the GEMM launches that gr_gemm picks by shape (no tile named):
32- and 64-row tiles, and K split over workgroups with a merge launch, against
float64 products of the same rounded inputs.

Bound per element: the result is a float32 sum of K exact products rounded once
to the storage type, so |error| <= |c| u + K 2^-24 sum |a b| with u = 2^-11
(fp16) or 2^-8 (bf16); relu and silu have slopes of at most 1.1, and silu adds a
few float32 roundings of its own (covered by 2^-20 |c|)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _cuda():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


CASES = [
    # batch, M, N, K, dtype, epilogue, b_kmajor, split expected
    (1, 1, 8, 64, "fp16", "none", False, False),          # 32-row tile: one k tile, the narrowest C
    (1, 32, 136, 96, "bf16", "silu", False, False),       # a half k tile at the end, ragged columns
    (2, 7, 264, 160, "fp16", "relu", True, False),
    (1, 24, 1376, 1056, "bf16", "silu", False, True),     # parts of whole and half k tiles
    (1, 31, 520, 4096, "fp16", "none", True, True),
    (3, 17, 264, 1024, "fp16", "relu", False, True),      # a batch with a split
    (1, 33, 136, 64, "fp16", "none", True, False),        # 64-row tile
    (1, 65, 264, 96, "bf16", "relu", False, False),
    (1, 100, 264, 2080, "fp16", "silu", False, True),
    (2, 64, 136, 2080, "bf16", "none", True, True),
    (1, 129, 1032, 1056, "fp16", "none", False, True),
    (1, 65, 8200, 4096, "bf16", "none", False, True),     # 128 x 128 split
    (1, 200, 8200, 8192, "fp16", "silu", False, True),    # 256 x 256 split
    (1, 200, 4104, 8224, "bf16", "none", True, True),     # and on 32-deep k tiles
    (1, 1000, 520, 64, "fp16", "relu", False, False),     # 256 x 128
    (1, 520, 3000, 96, "bf16", "none", False, False),     # 128 x 128, 32-deep k tiles
    (1, 700, 11000, 64, "bf16", "silu", False, False),    # bound by the store of C: 256 x 256
    (2, 1000, 8200, 224, "fp16", "none", True, False),    # 32-deep k tiles
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_picked_plan_parity(case):
    dev = _cuda()
    from grammar import runtime as rt
    from grammar.gemm import gemm
    z, M, N, K, dt, epi, km, split = case
    print(f"[case] picked gemm {case}", flush=True)
    tdt = {"fp16": torch.float16, "bf16": torch.bfloat16}[dt]
    assert (rt.lib().gr_gemm_workspace(rt.dtype_code(tdt), z, M, N, K) > 0) == split
    g = torch.Generator("cpu").manual_seed(17)
    a = torch.randn((z, M, K), generator=g).to(tdt).to(dev)
    b = (torch.randn((z, N, K) if km else (z, K, N), generator=g) / np.sqrt(K)).to(tdt).to(dev)
    out = torch.full((z, M + 1, N + 8), float("nan"), dtype=tdt, device=dev)    # a margin that must stay as it is
    gemm(a, b, epilogue=epi, alpha=0.5, b_kmajor=km, out=out[:, :M, :N])
    again = gemm(a, b, epilogue=epi, alpha=0.5, b_kmajor=km)
    torch.cuda.synchronize()
    assert torch.equal(out[:, :M, :N], again)
    assert torch.isnan(out[:, M:].float()).all() and torch.isnan(out[:, :, N:].float()).all()
    a64, b64 = a.double(), (b.transpose(1, 2).contiguous() if km else b).double()
    ref = 0.5 * (a64 @ b64)
    mag = 0.5 * (a64.abs() @ b64.abs())
    ref = ref.clamp(min=0) if epi == "relu" else ref * torch.sigmoid(ref) if epi == "silu" else ref
    u = 2.0 ** -11 if dt == "fp16" else 2.0 ** -8
    tiny = 2.0 ** -24                                       # fp16 subnormals
    bound = ref.abs() * (u + 2.0 ** -20) + 1.1 * K * 2.0 ** -24 * mag + tiny
    err = (again.double() - ref).abs()
    print(f"[parity] picked gemm {case}: max-abs {float(err.max()):.2e}", flush=True)
    assert bool((err <= bound).all())


def test_split_on_a_side_stream_and_through_the_c_abi_without_workspace():
    """The split's workspace belongs to the launch's stream; gr_gemm (no
    workspace) runs the same call whole-K, and a workspace too small for the
    split is not written."""
    dev = _cuda()
    import ctypes
    from grammar import runtime as rt
    from grammar.gemm import gemm
    g = torch.Generator("cpu").manual_seed(18)
    M, N, K = 24, 1376, 4096
    a = torch.randn((M, K), generator=g).half().to(dev)
    b = (torch.randn((K, N), generator=g) / 64).half().to(dev)
    ref = (a.double() @ b.double())
    L = rt.lib()
    need = L.gr_gemm_workspace(rt.GR_F16, 1, M, N, K)
    assert need > 0
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    outs = [gemm(a, b, stream=side) for _ in range(3)]
    outs.append(gemm(a, b, stream=side.cuda_stream))
    ws = torch.zeros(need - 16, dtype=torch.uint8, device=dev)
    st = [rt._ll2(0, K), rt._ll2(0, N), rt._ll2(0, N)]
    c = torch.empty((M, N), dtype=torch.float16, device=dev)
    p = [ctypes.c_void_p(t.data_ptr()) for t in (a, b, c)]
    rt.check(L.gr_gemm_ws(*p, rt.GR_F16, 1, M, N, K, *st, 0, 0, 1.0, ctypes.c_void_p(ws.data_ptr()), ws.numel(),
                          rt._stream_ptr(None)))
    d = torch.empty_like(c)
    p[2] = ctypes.c_void_p(d.data_ptr())
    rt.check(L.gr_gemm(*p, rt.GR_F16, 1, M, N, K, *st, 0, 0, 1.0, 0, 0, rt._stream_ptr(None)))
    torch.cuda.synchronize()
    for o in (*outs, c, d):
        assert float((o.double() - ref).norm() / ref.norm()) <= 4e-4      # fp16 rounding: 2^-11 / sqrt(3)
    for o in outs[1:]:
        assert torch.equal(o, outs[0])
    assert rt.lib().gr_gemm_workspace(rt.GR_F32, 1, M, N, K) == 0
