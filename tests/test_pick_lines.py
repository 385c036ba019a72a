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


def test_rendered_fp32_stages_follow_the_library_rule():
    """The rule for 32 x 32 blocks with K over four waves is written in the
    library and in the renderer."""
    import itertools
    from grammar import runtime as rt
    from grammar.hip_backend import _gemm_f32_groups
    L = rt.lib()
    picked = 0
    for M, N, nk, batch, km, bm, bn, cus in itertools.product((32, 128, 256, 768, 4096), (64, 512, 800, 4096), (1, 4, 5, 32, 256),
                                                              (1, 3), (0, 1), (32, 64, 128), (32, 64, 128), (256, 64)):
        if M % bm == 0 and N % bn == 0:
            want = bool(L.gr_gemm_f32_groups(batch, M, N, nk, km, bm, bn, cus))
            assert _gemm_f32_groups(M, N, nk, batch, bool(km), bm, bn, cus) == want, (M, N, nk, batch, km, bm, bn, cus)
            picked += want
    assert picked > 100


@pytest.mark.parametrize("M,N,nk,kmajor,bm,bn,groups", [
    (256, 512, 64, False, 64, 64, True), (512, 1024, 64, True, 64, 64, True), (1024, 1024, 64, False, 64, 64, False),
    (640, 1152, 32, False, 64, 64, True),          # three rounds of blocks: 46.4 us the whole program, 47.3 on the tile
    (640, 1152, 32, True, 64, 64, False),          # K-major
    (960, 1152, 44, False, 32, 32, True), (960, 1152, 44, True, 64, 64, True),    # five rounds against two part-filled ones
    (960, 1152, 16, False, 64, 64, False), (1024, 1024, 44, False, 32, 32, False), (1024, 1536, 44, False, 64, 64, False),
    (1024, 512, 4, True, 32, 32, True), (1024, 2048, 4, True, 32, 32, False),     # 8 rounds: 11.6 us, 7.1 on the tile
    (768, 4096, 64, False, 128, 128, False),       # 12 rounds: 98 us, 79 on the tile
    (2048, 1024, 16, False, 128, 128, True), (1536, 1408, 12, True, 128, 128, False),
    (2048, 800, 64, True, 128, 32, True),          # 7 rounds against two-wave tiles: 102 us, 143 on the tile
    (4096, 512, 12, True, 64, 32, False), (2048, 512, 12, True, 64, 32, True),
])
def test_fp32_groups_lines(M, N, nk, kmajor, bm, bn, groups):
    from grammar import runtime as rt
    assert bool(rt.lib().gr_gemm_f32_groups(1, M, N, nk, kmajor, bm, bn, 256)) == groups
