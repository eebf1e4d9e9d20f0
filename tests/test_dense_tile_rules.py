"""The host's rules for dense tiled products, asked of the built library: which of them multiply K's runs in workgroups of their own, and
which hand their strips to XCDs in runs; and which tiled products, dense or routed, send float32 results past the caches."""

import pytest


@pytest.mark.parametrize("M,N,K,apart", [
    # up to 64 rows: wherever there are fewer strips than CUs, the other kernel of so few rows being slower
    (17, 2048, 2048, True), (48, 16384, 2048, True), (48, 20480, 2048, True), (64, 24576, 4096, True), (17, 28672, 6144, True), (64, 32640, 2048, True),
    (64, 32768, 2048, False), (17, 32768, 8192, False),
    # up to 192 rows of long K likewise
    (192, 8192, 4096, True), (192, 8192, 6144, True), (65, 12288, 4096, True), (65, 8192, 2048, True), (128, 8192, 2048, True),
    # many rows and enough tiles: the form that walks all of K
    (192, 8192, 2048, False), (128, 12288, 2048, False), (512, 2048, 2048, False), (512, 3072, 2048, False), (384, 4096, 3072, False), (512, 3072, 6144, False),
    (512, 3072, 8192, True), (512, 2048, 3072, True),
    # as many tiles as CUs: none, however long K is
    (256, 8192, 16384, False), (512, 4096, 28672, False), (2048, 1024, 16384, False)])
def test_runs_apart(M, N, K, apart):
    from llmx_amd import ops
    ks = ops._split_k(-(-N // 16), K)
    floats = ops.lib().llmx_gemm_tile_runs_scratch(M, N, K, ops.EPI_STORE, ks, 0)
    assert (floats > 0) == apart
    assert floats % (M * N) == 0 and floats // (M * N) in ((2, 3, 4, 5, 6, 7, 8) if apart else (0,))


@pytest.mark.parametrize("strips,row_tiles,wide,runs", [
    (12, 16, True, False), (20, 16, True, False), (28, 32, True, False), (30, 16, True, False), (42, 16, True, False), (52, 16, True, False), (68, 32, True, False),
    (20, 16, False, False), (28, 16, False, False), (42, 8, False, False), (84, 8, False, False), (100, 4, False, False), (130, 2, False, False),
    (21, 16, True, True), (43, 8, True, True), (85, 16, False, True), (21, 2, False, True),
    (50, 16, True, True), (54, 4, True, True), (84, 16, True, True), (594, 2, True, True), (114, 4, False, True),
    (21, 1, False, False), (514, 1, False, False), (1187, 1, False, True), (1562, 1, False, True), (594, 1, True, True), (125, 1, True, False),
    (16, 16, True, False), (1024, 1, False, False), (800, 4, True, False)])
def test_strips_handed_to_xcds_in_runs(strips, row_tiles, wide, runs):
    from llmx_amd import ops
    assert ops.lib().llmx_gemm_tile_strip_runs(strips, row_tiles, int(wide)) == int(runs)


# both sides of every line: bytes of the results (8 MB routed, 48 MB dense, 10 MB beside weights of 512 MB), rows of whole lines
@pytest.mark.parametrize("at,M,N,K,ldc,groups,streams", [
    (0, 683, 3072, 1536, 3072, 256, True), (0, 682, 3072, 1536, 3072, 256, False), (0, 4096, 512, 128, 512, 24, True), (0, 4095, 512, 128, 512, 24, False),
    (0, 8192, 3076, 1536, 3076, 256, False), (0, 8192, 3076, 1536, 3104, 256, True), (0, 8192, 3074, 1536, 3104, 256, False), (64, 8192, 3072, 1536, 3072, 256, False),
    (128, 8192, 3072, 1536, 3072, 256, True), (16, 64, 200064, 3072, 200064, 0, False),
    (0, 14, 200064, 3072, 200064, 0, True), (0, 13, 200064, 3072, 200064, 0, False), (0, 20, 131072, 2048, 131072, 0, True), (0, 90, 131040, 2048, 131040, 0, False),
    (0, 1536, 8192, 3072, 8192, 0, True), (0, 1535, 8192, 3072, 8192, 0, False), (0, 96, 131072, 64, 131072, 0, True), (0, 768, 2048, 2048, 2048, 0, False),
    (0, 400, 8192, 32768, 8192, 0, True), (0, 64, 200068, 3072, 200068, 0, False), (0, 2048, 9220, 2048, 9220, 0, False)])
def test_results_past_the_caches(at, M, N, K, ldc, groups, streams):
    from llmx_amd import ops
    assert ops.lib().llmx_gemm_tile_streams_out(4096 + at, M, N, K, ldc, groups) == int(streams)
