"""The GEMM planner (gemm_plan) on the host: which kernel, tile height and K split a batch gets. The GPU tests of the
kernels take their sizes from plans that are asserted here or there, so that they run what they name."""
from gemm_plan import QKV, REF_ROWS, RESID, RSNAKE, SNAKE, STORE, STORE_KS, STORE_OTHER, STORE_ROWS, SWIGLU


def test_input_projection_fits_one_round(plan):
    """A short K (3 taps of 64 channels, six hi|lo K tiles) with a workspace: the one-round kernel without a split.
    The reference graph's input projection of two 8 s samples."""
    p = plan(STORE, [(344, 1024, 2 * 64 * 3, 3)], pair=1)
    assert p.kernel == "gemm_hl2_kernel<0>" and p.splits == 1 and p.tiles > 64


def test_one_step_fits_one_round(plan):
    """The shortest K there is (one 64-channel step), with and without a workspace, paired and f32 rows."""
    for ws in (0, 1 << 20):
        for pair in (0, 1):
            p = plan(STORE, [(33, 128, 128, 1)], ws=ws, pair=pair)
            assert p.kernel == "gemm_hl2_kernel<0>" and p.splits == 1, (ws, pair, p)


def test_stream_k_kernels(plan):
    """Stream-K: plain batches run the kernel with the plain K loop alone, a batch with one half-width-W problem
    the one with both; the snake convs never stream."""
    for epi in (QKV, SWIGLU):   # 297 tiles: a second round of 41
        p = plan(epi, [(384, 99 * 128, 4096, 1)], half=0)
        assert p.sk == 1 and p.kernel == "gemm_sk_kernel<%d>" % epi, p
    mixed = [(344, 5632, 2048 * 3, 3, 1, 1), (308, 5632, 1024, 1, 0, 0)]
    p = plan(SWIGLU, mixed)
    assert p.sk == 1 and p.kernel == "gemm_sk_hl_kernel<3>", p
    for epi in (SNAKE, RSNAKE):
        p = plan(epi, [(200, 1024, 8192, 1)], half=0)
        assert p.sk == 0 and p.kernel == "gemm_pipe_kernel<%d>" % epi, p


def test_sizes_of_the_one_round_gpu_tests(plan):
    """Every tile height of the one-round hi|lo kernel is run by the GPU tests in all four epilogues, at edges of the
    tiles, with one K step, odd numbers of steps and K splits."""
    for M, height in STORE_ROWS:
        for K in STORE_KS:
            p = plan(STORE, [(M, 4096, 2 * K, 1)], split_waves=1)
            assert p.kernel == "gemm_hl2_kernel<0>" and p.height == height, (M, K, p)
    for M, N, K, height, splits in STORE_OTHER:
        p = plan(STORE, [(M, N, 2 * K, 1)], split_waves=1)
        assert p.kernel == "gemm_hl2_kernel<0>" and (p.height, p.splits) == (height, splits), (M, N, K, p)
    H, F = 1024, 2816
    for M, want in REF_ROWS.items():
        got = (plan(QKV, [(M, 3 * H, 2 * H, 1)]).height, plan(SWIGLU, [(M, 2 * F, 2 * H * 3, 3)], pair=1).height,
               plan(RESID, [(M, H, 2 * H, 1)], split_waves=1).height,
               plan(RESID, [(M, H, 2 * F * 3, 3)], split_waves=1).height)
        assert got == want, (M, got)
    for epi in range(3):
        assert {32, 64, 96, 128} <= {h for hs in REF_ROWS.values() for h in (hs[epi:epi + 1] if epi < 2 else hs[2:])}
