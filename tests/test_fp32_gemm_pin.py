"""The knob kgroups pins an fp32 GEMM stage to its program's tile (1) or to 32 x
32 blocks with K over four waves (4); without it the shape decides."""
import pytest

from grammar.hip_backend import parse_plan
from grammar.kernel_ast import emit_module, program_from_key, structural_key


def _stage(p, out):
    src = emit_module(p)
    step = [s for s in parse_plan(src)["steps"] if s["kernel"] == f"t_{out}_kernel"][0]
    return src, src.split(f"void t_{out}_kernel(")[1].split("\n}\n")[0], step


def test_pinned_tile_and_pinned_groups():
    import run_mlp_search as RM
    p = RM.build_mlp_ln(256, 512, 1024, tile=64)
    loop = p.body[0]
    free, body, step = _stage(p, loop.out)
    assert "a.kgroups = 4;" in body and step["tiles"]["k_groups"] == 4 and step["grid"] == [8 * 32, 1, 1]
    key = structural_key(p)
    loop.knobs["kgroups"] = 1                    # the named 64 x 64 tile
    src, body, step = _stage(p, loop.out)
    assert "kgroups" not in body and "gr_gemm_f32_body<64, 64, 32, 2, 2" in body
    assert step["tiles"] == {"block_m": 64, "block_n": 64, "block_k": 32}
    assert step["grid"] == [4 * 16, 1, 1] and step["block"] == [256, 1, 1]
    assert structural_key(p) != key and structural_key(program_from_key(structural_key(p))) == structural_key(p)
    assert emit_module(program_from_key(structural_key(p))).count("a.kgroups = 4;") == src.count("a.kgroups = 4;")
    loop.knobs["kgroups"] = 4                    # what the shape decides here
    assert _stage(p, loop.out)[1:] == _stage(RM.build_mlp_ln(256, 512, 1024, tile=64), loop.out)[1:]
    del loop.knobs["kgroups"]
    assert emit_module(p) == free and structural_key(p) == key
    q = RM.build_mlp_ln(2048, 2048, 2048, tile=128)      # full grids keep their tile unless pinned
    assert "kgroups" not in _stage(q, q.body[0].out)[1]
    q.body[0].knobs["kgroups"] = 4
    assert _stage(q, q.body[0].out)[2]["grid"] == [64 * 64, 1, 1]


def test_pin_and_split_k():
    """A K split over workgroups runs the program's tile, pinned or not."""
    import run_mlp_search as RM
    for pin in (None, 1, 4):
        p = RM.build_mlp_ln(256, 512, 1024, tile=64)
        p.body[0].knobs["ksplit"] = 2
        if pin:
            p.body[0].knobs["kgroups"] = pin
        body, step = _stage(p, p.body[0].out)[1:]
        assert "kgroups" not in body and step["grid"][2] == 2 and step["tiles"]["ksplit"] == 2


@pytest.mark.gpu
@pytest.mark.parametrize("pin", [1, 4])
def test_pinned_stages_parity(pin):
    """Both lowerings of one program against float64 (float32 sums: 2e-6)."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import run_mlp_search as RM
    from grammar.hip_module import load_module
    print(f"[case] fp32 GEMM stages pinned to kgroups={pin}", flush=True)
    p = RM.build_mlp_ln(128, 192, 320, tile=64)
    for loop in p.body:
        loop.knobs["kgroups"] = pin
    mod = load_module(emit_module(p))
    gemms = [s for s in mod.plan["steps"] if s["lowering"] == "gemm"]
    assert len(gemms) == 2 and all((s["tiles"].get("k_groups", 1) == 4) == (pin == 4) for s in gemms)
    ins = RM.mlp_inputs(128, 192, 320, "fp32", seed=8, device=torch.device("cuda:0"))
    out = mod.fn(*[ins[n] for n in mod.inputs])
    torch.cuda.synchronize()
    x, w1, w2 = (ins[n].double() for n in ("X", "W1", "W2"))
    r = torch.relu(x @ w1) @ w2 + x
    ref = (r - r.mean(1, keepdim=True)) / torch.sqrt(r.var(1, unbiased=False, keepdim=True) + 1e-5)
    assert float((out.double() - ref).norm() / ref.norm()) <= 2e-6
