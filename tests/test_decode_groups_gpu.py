"""GPU parity of the decode launches' key groups (5 to 64 queries) and of the
merge of their parts, against attention in float64 on the GPU.

Bound: relative 2-norm at most the storage type's unit roundoff (2^-11 fp16,
2^-8 bf16), as for the attention forward."""
import math

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CASES = [
    # B, H, Nq, N, D, dtype, splits
    (1, 2, 5, 32, 64, "fp16", 1),         # one key tile: three of four groups idle
    (1, 2, 32, 96, 128, "bf16", 1),
    (2, 3, 33, 224, 64, "bf16", 1),       # two waves, 31 queries past the end
    (1, 3, 64, 1056, 128, "fp16", 4),     # four parts: lane groups merge a row each
    (1, 5, 40, 1056, 64, "fp16", 5),      # five: a wave per row
    (2, 1, 17, 3104, 128, "bf16", 16),
    (1, 1, 9, 2144, 64, "bf16", 67),      # more parts than lanes in the merge
    (1, 1, 3, 2144, 128, "fp16", 67),     # streaming kernel, the same merge
    (1, 7, 1, 1024, 64, "bf16", 3),
    (1, 2, 100, 544, 64, "fp16", 2),      # four waves, 32-key tiles, no groups
    (1, 300, 33, 256, 128, "bf16", 1),    # more heads than compute units, D 128, few keys: one group of 64-key tiles
    (3, 100, 5, 480, 128, "fp16", 1),     # of 32-key tiles
    (1, 300, 9, 512, 128, "fp16", 1),     # groups again
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_decode_groups_parity(case):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from grammar.attention import flash_attention_decode
    B, H, Nq, N, D, dt, splits = case
    print(f"[case] decode groups {case}", flush=True)
    tdt = {"fp16": torch.float16, "bf16": torch.bfloat16}[dt]
    g = torch.Generator("cpu").manual_seed(37)
    q = torch.randn((B, H, Nq, D), generator=g)
    # keys climb from part to part, so the parts and groups end with different bases
    k = torch.randn((B, H, N + 64, D), generator=g) + (torch.arange(N + 64).float() * 2 / N).view(1, 1, -1, 1)
    v = torch.randn((B, H, N + 64, D), generator=g)
    q, k, v = (t.to(tdt).cuda() for t in (q, k, v))
    k, v = k[:, :, :N], v[:, :, :N]                       # a cache with room for more
    store = torch.full((B, H, Nq + 1, D), float("nan"), dtype=tdt, device="cuda")
    o = flash_attention_decode(q, k, v, splits=splits, out=store[:, :, :Nq])
    torch.cuda.synchronize()
    assert torch.isnan(store[:, :, Nq].float()).all()
    ref = torch.empty((B, H, Nq, D), dtype=torch.float64, device="cuda")
    for b in range(B):
        for h in range(H):
            s = q[b, h].double() @ k[b, h].double().t().contiguous() / math.sqrt(D)
            ref[b, h] = torch.softmax(s, dim=1) @ v[b, h].double()
    err = float((o.double() - ref).norm() / ref.norm())
    print(f"[parity] decode groups {case}: rel {err:.2e}", flush=True)
    assert err <= (2.0 ** -11 if dt == "fp16" else 2.0 ** -8)


@pytest.mark.parametrize("Nq,N,D,splits", [(40, 2144, 64, 0), (9, 1024, 128, 0), (64, 544, 64, 3)])
def test_decode_unscaled_queries_in_parts(Nq, N, D, splits):
    """fp16 with scale 1.0: Q as given, one wave per 32 queries, no key groups."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from grammar.attention import decode_splits, flash_attention_decode
    assert splits or decode_splits(1, 2, Nq, N, groups=False) > 1
    print(f"[case] decode unscaled Nq={Nq} N={N} D={D} splits={splits}", flush=True)
    g = torch.Generator("cpu").manual_seed(43)
    # scores of unit variance, climbing by 2 over the keys
    q = torch.randn((1, 2, Nq, D), generator=g)
    k = (torch.randn((1, 2, N, D), generator=g) + (torch.arange(N).float() * 2 / N).view(1, 1, -1, 1)) / D ** 0.5
    v = torch.randn((1, 2, N, D), generator=g)
    q, k, v = (t.half().cuda() for t in (q, k, v))
    o = flash_attention_decode(q, k, v, scale=1.0, splits=splits)
    torch.cuda.synchronize()
    ref = torch.softmax(q.double() @ k.double().transpose(2, 3).contiguous(), dim=-1) @ v.double()
    err = float((o.double() - ref).norm() / ref.norm())
    print(f"[parity] decode unscaled: rel {err:.2e}", flush=True)
    assert err <= 2.0 ** -11


@pytest.mark.parametrize("Nq", [1, 3, 40])
def test_decode_default_parts_fit_a_given_workspace(Nq):
    """splits = 0 with a workspace of fewer parts than the default takes those;
    one that does not hold two is refused."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from grammar import runtime as rt
    from grammar.attention import decode_splits, flash_attention_decode
    print(f"[case] decode given workspace Nq={Nq}", flush=True)
    H, N, D = 4, 8192, 64
    g = torch.Generator("cpu").manual_seed(59)
    q, kv = (torch.randn((1, H, n, D), generator=g).bfloat16().cuda() for n in (Nq, N))
    assert decode_splits(1, H, Nq, N) > 4
    need = int(rt.lib().gr_attn_decode_workspace(1, H, Nq, D, 4))
    ws = torch.empty(need + 16, dtype=torch.uint8, device="cuda")
    assert torch.equal(flash_attention_decode(q, kv, kv, workspace=ws), flash_attention_decode(q, kv, kv, splits=4))
    big = torch.empty(64 * need, dtype=torch.uint8, device="cuda")
    assert torch.equal(flash_attention_decode(q, kv, kv, workspace=big), flash_attention_decode(q, kv, kv))
    with pytest.raises(ValueError):
        flash_attention_decode(q, kv, kv, workspace=ws[:need // 4 + 16])
