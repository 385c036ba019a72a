"""Lines of the shape picks at 256 compute units (host arithmetic)."""
import pytest

pytest.importorskip("torch")


@pytest.mark.parametrize("H,N,D,causal,shape", [
    (200, 320, 64, False, (64, 1, 64)),      # many short workgroups: 64 x 64 before a part-empty 128 x 64
    (300, 192, 64, True, (64, 1, 64)),
    (200, 448, 64, True, (64, 1, 64)),
    (200, 576, 64, False, (128, 1, 64)),     # nine key tiles: the larger tile
    (128, 320, 64, False, (256, 1, 64)),     # three workgroups per CU at most
    (12, 4096, 64, False, (256, 1, 64)),     # not 64 queries x 2 groups in three rounds
    (16, 1024, 64, False, (64, 2, 64)),      # one workgroup per CU
])
def test_attention_64_query_tiles(H, N, D, causal, shape):
    from grammar.attention import picked_shape
    assert picked_shape(1, H, N, D, "bf16", causal=causal) == shape
