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
