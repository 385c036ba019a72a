"""GPU attention where the exponent bases of a row's key tiles, key groups and
key parts lie 120 to 140 powers of two apart, against float64.

Every query row selects one pattern of scores, in powers of two: one 32-key
block low (at -x), a key near the row's maximum in a later block, all other
keys at -200. The kernels take a row's base from its first tile (of a group or
a part), so the late key's probability may stand far above that base, and the
base may have to be brought to another one's by a factor near the smallest
float32.

Bound per element: a probability is rounded once to the storage type (unit
roundoff u: 2^-9 bf16, 2^-11 fp16) in the numerator and in the row sum, and the
result once, so |error| <= (3 u + 2^-14) sum w |v|, with 2^-14 for fp16's
subnormal probabilities (N 2^-25) and the float32 exponents (200 * 2^-23)."""
import math

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DT = {"fp16": torch.float16, "bf16": torch.bfloat16}
U = {"fp16": 2.0 ** -11, "bf16": 2.0 ** -9}
SCALE = math.log(2.0) / 2          # with queries of 2: scores are keys' entries in powers of two


def _cuda():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def _patterns(N):
    """[patterns, N] scores: the low block, the distance to the late key's block
    and how low, so that some pattern meets any group's or part's first tile."""
    out = []
    for x in (120, 127, 128, 140):
        for low, step in ((0, 1), (0, 4), (1, 1), (1, 4), (1, 8), (2, 2), (2, 4), (3, 4), (4, 1), (4, 2), (4, 8), (6, 4),
                          (8, 2), (8, 8)):
            late, last = 32 * (low + step) + 5, 32 * (low + 2 * step) + 9
            if last >= N:
                continue
            e = torch.full((N,), -200.0)
            e[0] = 0.0
            e[32 * low:32 * low + 32] = -float(x)
            e[late] = -0.5
            if low == 0:
                e[last] = 1.0          # the base moves once more, past the late key
            out.append(e)
    return torch.stack(out)


def _inputs(B, H, Nq, N, D, dt, dev):
    pat = _patterns(N)
    assert len(pat) <= D
    g = torch.Generator("cpu").manual_seed(47)
    q = torch.zeros((B, H, Nq, D))
    q.scatter_(3, torch.randint(0, len(pat), (B, H, Nq, 1), generator=g), 2.0)
    k = torch.zeros((B, H, N, D))
    k[..., :len(pat)] = pat.t()
    v = 3.0 * torch.randn((B, H, N, D), generator=g)
    return tuple(t.to(DT[dt]).to(dev) for t in (q, k, v))


def _check(o, q, k, v, dt, causal, what, lse=None):
    s = SCALE * (q.double() @ k.double().transpose(2, 3).contiguous())
    if causal:
        s = s.masked_fill(torch.ones(s.shape[2:], dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    w = torch.softmax(s, dim=-1)
    err = (o.double() - w @ v.double()).abs()
    bound = (3 * U[dt] + 2.0 ** -14) * (w @ v.double().abs())
    bad = ~(err <= bound)
    print(f"[parity] bases {what}: {int(bad.any(-1).sum())} rows of {bad[..., 0].numel()} outside", flush=True)
    assert not bool(bad.any())
    if lse is not None:                  # the sum's relative error, as an absolute one of its logarithm
        assert bool(((lse.double() - torch.logsumexp(s, dim=-1)).abs() <= U[dt] + 2.0 ** -14).all())


CASES = [
    # H, N, D, causal, k_transposed, block_m, block_n (0, 0: the picked shape)
    (4, 512, 64, False, False, 0, 0),      # 1 wave x 4 key groups of 32 keys
    (1, 2048, 64, True, False, 0, 0),      # 1 x 8
    (16, 1024, 64, False, True, 0, 0),     # 2 x 2 of 64 keys
    (2, 832, 128, False, False, 0, 0),     # 2 x 4 of 32 keys
    (64, 384, 128, True, True, 0, 0),      # 4 x 2 of 64 keys
    (2, 1024, 64, False, False, 256, 128),
    (2, 1024, 64, True, True, 64, 32),
    (2, 1024, 64, False, False, 129, 64),  # the pipelined schedule
    (2, 1024, 64, False, True, 256, 64),   # fp16: two waves per SIMD
    (2, 1024, 128, False, True, 256, 64),  # two waves per SIMD
    (2, 1024, 128, True, True, 256, 64),
    (2, 1024, 128, False, False, 128, 64),
]


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_forward_bases_far_apart(case, dt):
    dev = _cuda()
    from grammar.attention import flash_attention_fwd, flash_attention_fwd_train
    H, N, D, causal, kt, bm, bn = case
    print(f"[case] bases {case} {dt}", flush=True)
    q, k, v = _inputs(1, H, N, N, D, dt, dev)
    kk = k.transpose(2, 3).contiguous() if kt else k
    o = flash_attention_fwd(q, kk, v, causal=causal, k_transposed=kt, scale=SCALE, block_m=bm, block_n=bn)
    torch.cuda.synchronize()
    _check(o, q, k, v, dt, causal, (case, dt))
    if not kt:
        o, lse = flash_attention_fwd_train(q, k, v, causal=causal, scale=SCALE, block_m=bm, block_n=bn)
        torch.cuda.synchronize()
        _check(o, q, k, v, dt, causal, (case, dt, "train"), lse)


@pytest.mark.parametrize("dt", ["bf16", "fp16"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Nq,splits", [(1, 4), (3, 1), (40, 1), (17, 4), (64, 8), (100, 1), (100, 4)])
def test_decode_bases_far_apart(Nq, splits, D, dt):
    dev = _cuda()
    from grammar.attention import flash_attention_decode
    N = 1024
    print(f"[case] decode bases Nq={Nq} splits={splits} D={D} {dt}", flush=True)
    q, k, v = _inputs(1, 64 if Nq < 5 else 2, Nq, N, D, dt, dev)
    o = flash_attention_decode(q, k, v, scale=SCALE, splits=splits)
    torch.cuda.synchronize()
    _check(o, q, k, v, dt, False, (Nq, splits, D, dt))
