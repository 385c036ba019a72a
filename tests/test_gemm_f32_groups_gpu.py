"""GPU parity of the fp32 GEMM's k-group body (32 x 32 blocks, K over the four
waves of a workgroup): gr_gemm calls that name no tile and leave CUs idle, and
rendered stages, against float64.

Bound per element: float32 products summed in eight chains that are then
added, so |error| <= (K / 8 + 16) 2^-24 sum |a b| before the epilogue; relu and
silu have slopes of at most 1.1, silu's own float32 steps 2^-20 |c|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _cuda():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


CASES = [
    # batch, M, N, K, epilogue, b_kmajor
    (1, 64, 64, 32, "none", False),       # two k tiles: two of four waves have work
    (1, 64, 64, 64, "none", False),       # one tile per wave, no turn of the ring
    (1, 128, 128, 208, "relu", True),     # 13 tiles: one wave takes four, the others three
    (2, 64, 128, 80, "none", False),
    (1, 128, 64, 40, "silu", True),       # 8-deep k tiles
    (3, 128, 64, 288, "silu", False),
    (1, 256, 512, 1024, "none", True),
    (1, 1056, 96, 2048, "relu", False),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_f32_groups_parity(case):
    dev = _cuda()
    from grammar.gemm import gemm
    z, M, N, K, epi, km = case
    print(f"[case] fp32 groups {case}", flush=True)
    g = torch.Generator("cpu").manual_seed(31)
    a = torch.randn((z, M, K), generator=g).to(dev)
    b = (torch.randn((z, N, K) if km else (z, K, N), generator=g) / np.sqrt(K)).to(dev)
    out = torch.full((z, M + 1, N + 4), float("nan"), device=dev)
    c = gemm(a, b, epilogue=epi, alpha=0.5, b_kmajor=km, out=out[:, :M, :N])
    again = gemm(a, b, epilogue=epi, alpha=0.5, b_kmajor=km)
    torch.cuda.synchronize()
    assert torch.equal(c, again)
    assert torch.isnan(out[:, M:]).all() and torch.isnan(out[:, :, N:]).all()
    a64, b64 = a.double(), (b.transpose(1, 2).contiguous() if km else b).double()
    ref = 0.5 * (a64 @ b64)
    mag = 0.5 * (a64.abs() @ b64.abs())
    ref = ref.clamp(min=0) if epi == "relu" else ref * torch.sigmoid(ref) if epi == "silu" else ref
    err = (again.double() - ref).abs()
    bound = 1.1 * (K / 8 + 16) * 2.0 ** -24 * mag + 2.0 ** -20 * ref.abs()
    print(f"[parity] fp32 groups {case}: max {float(err.max()):.2e}", flush=True)
    assert bool((err <= bound).all())


@pytest.mark.parametrize("tile,dims", [(64, (256, 512, 1024)), (32, (64, 96, 160)), (128, (128, 256, 384))])
def test_rendered_stages_on_k_groups(tile, dims):
    """The fp32 MLP + LayerNorm program with its residual merged into the second
    GEMM: every GEMM stage runs on k groups and matches float64."""
    dev = _cuda()
    import run_mlp_search as RM
    from grammar import rewrites as R
    from grammar.hip_module import load_module
    from grammar.kernel_ast import emit_module
    M, D, F = dims
    print(f"[case] rendered k groups tile {tile} {dims}", flush=True)
    p = RM.build_mlp_ln(M, D, F, tile=tile)
    p = R.merge(p, p.body[2], p.body[3])
    p = R.merge(p, p.body[0], p.body[1])
    mod = load_module(emit_module(p))
    gemms = [s for s in mod.plan["steps"] if s["lowering"] == "gemm"]
    assert len(gemms) == 2 and all(s["tiles"]["k_groups"] == 4 and s["block"] == [256, 1, 1] for s in gemms)
    ins = RM.mlp_inputs(M, D, F, "fp32", seed=6, device=dev)
    t = mod.run_with([ins[n] for n in mod.inputs])
    torch.cuda.synchronize()
    x, w1, w2 = (ins[n].double() for n in ("X", "W1", "W2"))
    h = torch.relu(x @ w1)
    r = h @ w2 + x
    ref = (r - r.mean(1, keepdim=True)) / torch.sqrt(r.var(1, unbiased=False, keepdim=True) + 1e-5)
    for name, want in (("a", h), ("r", r), ("out", ref)):
        err = float((t[name].double() - want).norm() / want.norm())
        print(f"[parity] rendered k groups {name}: rel {err:.2e}", flush=True)
        assert err <= 2e-6
