"""The search windows a plan accepts against the LDS of the kernel that evaluates them."""
import ctypes as C

import pytest

WIDEST = {16: 32, 32: 64, 48: 96, 64: 128, 96: 79, 128: 45}  # points per axis


@pytest.mark.gpu
@pytest.mark.parametrize("N", sorted(WIDEST))
def test_widest_window_fits_its_kernel(torch_gpu, ctx, N):
    """The need is the launched kernel's own: two tables of E x (N/2 + 1) complex values per launch, and at least the
    exchange of a round of pencils and the twiddles beside them."""
    from ettk_amd import lib

    need = getattr(lib.load(), "_ZN4ettk19fft3_ccc_window_ldsEii")
    need.argtypes, need.restype = [C.c_int, C.c_int], C.c_size_t
    E, H = WIDEST[N], N // 2 + 1
    pencils = (H + 1) // 2 if N == 128 else H
    assert need(N, E) <= 160 * 1024
    assert need(N, E) - need(N, 0) == 16 * E * H
    assert need(N, 0) >= 8 * N * pencils + 16 * N


@pytest.mark.gpu
@pytest.mark.parametrize("N,widest", [(96, 19.5), (128, 11.0)])
def test_wider_windows_are_refused(torch_gpu, ctx, N, widest):
    from ettk_amd.abi import default_params
    from ettk_amd.lib import EttkError, Plan

    plan = Plan(ctx, default_params(N, 8, trans_restrict=8.0))
    try:
        plan.set_restrictions(180.0, widest)
        for window in (widest + 0.5, -1.0):
            with pytest.raises(EttkError, match="search window too large for this box size"):
                plan.set_restrictions(180.0, window)
        plan.set_restrictions(180.0, 8.0)
    finally:
        plan.close()
