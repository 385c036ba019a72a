"""A module call whose stage takes more arguments than a few."""
import pytest

from grammar.hip_backend import parse_plan
from grammar.kernel_ast import Compute, Load, ParallelLoop, Program, Store, emit_module

torch = pytest.importorskip("torch")


def _sum_program(n):
    loads = [Load(f"i{j:03d}", ["n", "m"]) for j in range(n)]
    body, s = list(loads), loads[0]
    for ld in loads[1:]:
        s = Compute("add", [s, ld])
        body.append(s)
    shapes = {f"i{j:03d}": (64, 64) for j in range(n)}
    return Program({**shapes, "o": (64, 64)}, [ParallelLoop("o", (32, 32), ("n", "m"), body + [Store("o", s, ["n", "m"])])])


@pytest.mark.gpu
@pytest.mark.parametrize("inputs", [63, 64, 100])      # with the output 64, 65 and 101 arguments
def test_a_stage_of_many_arguments(inputs):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from grammar.hip_module import load_module
    print(f"[case] a stage of {inputs} inputs", flush=True)
    src = emit_module(_sum_program(inputs))
    assert [len(s["args"]) for s in parse_plan(src)["steps"]] == [inputs + 1]
    mod = load_module(src)
    g = torch.Generator("cpu").manual_seed(53)
    ins = [torch.randint(-8, 8, (64, 64), generator=g).float().cuda() for _ in range(inputs)]
    out = mod.fn(*ins)
    torch.cuda.synchronize()
    assert torch.equal(out, torch.stack(ins).sum(0))        # whole numbers: exact
