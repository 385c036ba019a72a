"""GPU parity of the attention forward's picked workgroup shapes (no tile named):
key groups inside a workgroup and part-filled last query tiles, against
attention computed in float64 on the GPU from the same rounded inputs.

Bound: relative 2-norm at most the storage type's unit roundoff (2^-11 fp16,
2^-8 bf16). O's own rounding gives u / sqrt(3) of it, the rounding of P (one of
2^-11 / 2^-8 per probability, averaged over the keys) less; row log-sum-exps
are float32 sums of those rounded P: 2e-3 absolute, as the training tests."""
import math

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DT = {"fp16": torch.float16, "bf16": torch.bfloat16}
U = {"fp16": 2.0 ** -11, "bf16": 2.0 ** -8}


def _cuda():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def _reference(q, k, v, causal):
    """(O, row log-sum-exp) in float64; k as [B, H, N, D]."""
    q, k, v = q.double(), k.double(), v.double()
    s = torch.stack([torch.stack([qh @ kh.t().contiguous() for qh, kh in zip(qb, kb)]) for qb, kb in zip(q, k)])
    s = s / math.sqrt(q.shape[-1])
    if causal:
        n = s.shape[-1]
        s = s.masked_fill(torch.ones(n, n, dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    return torch.matmul(torch.softmax(s, dim=-1), v.contiguous()), torch.logsumexp(s, dim=-1)


CASES = [
    # B, H, N, D, dtype, causal, k_transposed, the picked (queries, key groups, keys per tile)
    (1, 1, 64, 64, "fp16", False, False, (128, 1, 64)),  # one query tile of 4 waves, half of them past the end
    (1, 1, 192, 64, "bf16", True, False, (32, 4, 32)),  # 1 wave x 4 groups
    (1, 3, 320, 64, "fp16", True, True, (32, 4, 32)),  # 10 key tiles: groups of unequal count
    (2, 2, 512, 64, "bf16", False, True, (32, 4, 32)),
    (1, 1, 2048, 64, "fp16", True, False, (32, 8, 32)),  # 1 wave x 8 groups
    (1, 2, 1344, 64, "bf16", False, False, (32, 4, 32)),
    (1, 15, 2432, 64, "bf16", False, False, (128, 1, 128)),
    (1, 86, 640, 64, "bf16", False, False, (128, 1, 128)),  # 128-query tiles of 128 keys
    (1, 86, 640, 64, "fp16", False, True, (128, 1, 128)),
    (1, 16, 1024, 64, "fp16", False, False, (64, 2, 64)),  # 2 waves x 2 groups
    (1, 32, 320, 64, "bf16", True, True, (64, 2, 64)),
    (1, 12, 1408, 64, "bf16", False, False, (128, 2, 64)),  # 4 waves x 2 groups
    (2, 32, 448, 64, "fp16", True, True, (128, 2, 64)),  # the last tile half-filled
    (1, 48, 704, 64, "bf16", False, True, (256, 1, 64)),  # 256-query tiles, ragged
    (2, 32, 1344, 64, "fp16", False, False, (128, 1, 64)),  # 128-query tiles, one group, ragged
    (3, 16, 1344, 64, "fp16", False, True, (64, 1, 64)),  # 64-query tiles, one group
    (1, 1, 64, 128, "bf16", True, False, (128, 1, 64)),
    (1, 2, 320, 128, "fp16", True, True, (64, 4, 32)),  # 2 waves x 4 groups
    (1, 12, 1344, 128, "bf16", False, True, (64, 4, 32)),
    (1, 3, 1984, 128, "fp16", False, False, (64, 4, 32)),
    (2, 32, 384, 128, "bf16", True, False, (128, 2, 64)),  # 4 waves x 2 groups
    (1, 12, 1408, 128, "fp16", False, True, (128, 2, 64)),
    (2, 12, 1344, 128, "bf16", False, False, (64, 1, 64)),  # 64-query tiles, one group
    (2, 32, 1344, 128, "fp16", True, True, (128, 1, 64)),
    (1, 85, 960, 128, "fp16", True, True, (256, 1, 64)),  # 256-query causal tiles, ragged
    (1, 85, 960, 128, "bf16", True, False, (256, 1, 64)),
    (1, 32, 1344, 128, "fp16", False, False, (256, 1, 64)),  # 256-query tiles, ragged
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_picked_shape_parity(case):
    dev = _cuda()
    from grammar.attention import flash_attention_fwd, flash_attention_fwd_train, picked_shape
    B, H, N, D, dt, causal, kt, shape = case
    assert picked_shape(B, H, N, D, dt, causal=causal, k_transposed=kt) == shape
    if not kt:
        assert picked_shape(B, H, N, D, dt, causal=causal, train=True) == shape
    print(f"[case] picked attention {case}", flush=True)
    g = torch.Generator("cpu").manual_seed(19)
    q, k, v = (torch.randn((B, N, H, D), generator=g).to(DT[dt]).to(dev).transpose(1, 2) for _ in range(3))
    kk = k.transpose(2, 3).contiguous() if kt else k
    store = torch.full((B, N + 1, H, D), float("nan"), dtype=DT[dt], device=dev)       # row N stays as it is
    o = flash_attention_fwd(q, kk, v, causal=causal, k_transposed=kt, out=store[:, :N].transpose(1, 2))
    again = flash_attention_fwd(q.contiguous(), kk, v.contiguous(), causal=causal, k_transposed=kt)
    torch.cuda.synchronize()
    assert torch.isnan(store[:, N].float()).all()
    assert torch.equal(o, again)
    ref, lse_ref = _reference(q, k, v, causal)
    err = float((o.double() - ref).norm() / ref.norm())
    print(f"[parity] picked attention {case}: rel {err:.2e}", flush=True)
    assert err <= U[dt]
    if not kt:
        o2, lse = flash_attention_fwd_train(q, k, v, causal=causal)
        torch.cuda.synchronize()
        assert float((o2.double() - ref).norm() / ref.norm()) <= U[dt]
        assert float((lse.double() - lse_ref).abs().max()) <= 2e-3


def test_part_filled_256_query_causal_tiles_at_head_dim_64():
    dev = _cuda()
    from grammar.attention import flash_attention_fwd_train, picked_shape
    H, N, D = 122, 4032, 64
    assert picked_shape(1, H, N, D, "bf16", causal=True, train=True) == (256, 1, 64)
    print(f"[case] picked attention {H} heads N {N} D {D} causal", flush=True)
    g = torch.Generator("cuda").manual_seed(29)
    q, k, v = (torch.randn((1, H, N, D), generator=g, device=dev).bfloat16() for _ in range(3))
    o, lse = flash_attention_fwd_train(q, k, v, causal=True)
    for h in (0, 61, H - 1):
        ref, lse_ref = _reference(q[:, h:h + 1], k[:, h:h + 1], v[:, h:h + 1], True)
        assert float((o[:, h:h + 1].double() - ref).norm() / ref.norm()) <= U["bf16"]
        assert float((lse[:, h:h + 1].double() - lse_ref).abs().max()) <= 2e-3


@pytest.mark.parametrize("D,N,causal,dt", [(64, 448, False, "fp16"), (64, 2048, True, "fp16"), (128, 832, False, "bf16"),
                                           (128, 1024, True, "fp16")])
def test_groups_merge_bases_far_apart(D, N, causal, dt):
    """Keys that climb along the queries' common direction: the groups end with
    different exponent bases, and within a group the base moves."""
    dev = _cuda()
    from grammar.attention import flash_attention_fwd
    print(f"[case] groups far apart D={D} N={N} causal={causal} {dt}", flush=True)
    g = torch.Generator("cpu").manual_seed(23)
    q = torch.randn((1, 2, N, D), generator=g) + 1.0
    climb = 3.0 * (torch.arange(N).float() / N) + 2.0 * (torch.arange(N) // 32 % 4).float()
    k = torch.randn((1, 2, N, D), generator=g) + climb.view(1, 1, N, 1)
    v = torch.randn((1, 2, N, D), generator=g)
    q, k, v = (t.to(DT[dt]).to(dev) for t in (q, k, v))
    o = flash_attention_fwd(q, k, v, causal=causal)
    torch.cuda.synchronize()
    ref, _ = _reference(q, k, v, causal)
    # scores reach about 60: the fp16 path's pre-scaled Q rounds them by up to
    # 60 log2(e) 2^-11 = 0.04 in the exponent, 3 % of a probability at worst
    err = float((o.double() - ref).norm() / ref.norm())
    print(f"[parity] groups far apart: rel {err:.2e}", flush=True)
    assert torch.isfinite(o.float()).all() and err <= (1e-2 if dt == "fp16" else 2.0 ** -8)
