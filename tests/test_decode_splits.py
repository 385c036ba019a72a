"""The key parts that decode calls take by default (host-side rule)."""
import pytest

torch = pytest.importorskip("torch")


def test_parts_without_key_groups():
    """fp16 with scale log2(e) > 1 runs one wave per query tile and part: its
    parts fill two workgroups per compute unit."""
    from grammar.attention import _key_groups, decode_splits, decode_splits_noalloc
    assert [decode_splits(1, h, 40, n, groups=False) for h, n in
            ((1, 16384), (1, 512), (8, 8192), (64, 8192), (129, 8192), (200, 8192), (512, 8192))] == \
        [64, 2, 32, 8, 4, 3, 1]
    assert decode_splits_noalloc(1, 1, 40, 16384, 64, groups=False) == 64
    assert not _key_groups(torch.float16, 1.0) and not _key_groups(torch.float16, 0.7)
    assert _key_groups(torch.float16, 0.125) and _key_groups(torch.bfloat16, 1.0)


# B * H, queries, N, D -> parts
LINES = [
    (1, 1, 512, 64, 1), (1, 1, 544, 64, 2), (8, 1, 8192, 128, 32), (16, 1, 4128, 128, 16), (85, 1, 768, 64, 3),
    (86, 1, 992, 64, 1), (86, 1, 1024, 64, 2), (128, 1, 4128, 128, 2), (129, 1, 4096, 128, 1), (512, 1, 16384, 128, 1),
    (8, 2, 512, 64, 1), (8, 2, 544, 64, 2), (8, 2, 288, 128, 2), (8, 4, 256, 64, 1), (8, 4, 288, 64, 2),
    (8, 3, 3104, 64, 24), (8, 4, 8192, 64, 32), (64, 2, 4096, 64, 6), (64, 3, 4096, 64, 8), (129, 4, 992, 64, 1),
    (129, 4, 1024, 64, 3), (129, 2, 992, 128, 1), (129, 2, 1024, 128, 3), (255, 4, 512, 64, 1), (255, 2, 1024, 128, 2),
    (300, 3, 8192, 64, 1),
    (8, 40, 512, 64, 1), (8, 40, 3104, 64, 12), (16, 64, 8192, 64, 16), (128, 5, 4096, 64, 2), (129, 5, 4096, 64, 1),
    (129, 5, 8192, 64, 2), (150, 64, 8192, 128, 3), (256, 5, 4096, 128, 1), (300, 5, 8192, 128, 2), (512, 5, 16384, 64, 1),
    (64, 128, 4096, 128, 8),
]


@pytest.mark.parametrize("heads,Nq,N,D,parts", LINES)
def test_lines_of_the_default_parts(heads, Nq, N, D, parts):
    from grammar.attention import decode_splits
    assert decode_splits(1, heads, Nq, N, D=D) == parts
