"""The GEMM planner (gemm_plan) on the host: which kernel, tile height and K split a batch gets. The GPU tests of the
kernels take their sizes from plans that are asserted here or there, so that they run what they name."""
from gemm_plan import QKV, RESID, STORE, SWIGLU


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
