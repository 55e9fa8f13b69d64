"""Large results on their way to host memory (download_staged, so3.hip): the routes by destination, and what is left where
something the fast route needs cannot be had.  The function is called by its C++ name in the built library, with a ring
made of zero bytes (its default state), so that the route can be read from the ring."""
import ctypes as C

import numpy as np
import pytest

SYMBOL = "_ZN4ettk15download_stagedERNS_12DownloadRingEPvPKvmP12ihipStream_t"
PIECE = 2 << 20


class Ring:
    def __init__(self):
        self.mem = (C.c_uint64 * 64)()  # pinned pointer, its bytes, four events

    @property
    def bytes(self):
        return self.mem[1]


def download(ring, dst, src):
    from ettk_amd import lib

    fn = getattr(lib.load(), SYMBOL)
    fn.argtypes, fn.restype = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_size_t, C.c_void_p], None
    fn(C.addressof(ring.mem), dst.ctypes.data, src.data_ptr(), dst.nbytes, None)


def source(torch, n):
    t = torch.arange(n, dtype=torch.int64, device="cuda") * 0x9E3779B9
    torch.cuda.synchronize()
    return t, t.cpu().numpy()


@pytest.mark.gpu
def test_pinned_destination_is_one_transfer(torch_gpu, ctx):
    """A destination that the card writes by itself takes no detour through the slots; ordinary memory does."""
    src, want = source(torch_gpu, 5 * PIECE // 8 + 3)
    pinned = torch_gpu.zeros(want.size, dtype=torch_gpu.int64, pin_memory=True).numpy()
    ring = Ring()
    download(ring, pinned, src)
    assert np.array_equal(pinned, want)
    assert ring.bytes == 0
    pageable = np.zeros_like(want)
    download(ring, pageable, src)
    assert np.array_equal(pageable, want)
    assert ring.bytes == 4 * PIECE


@pytest.mark.gpu
@pytest.mark.parametrize("extra", [-1, 0, 1, PIECE // 8])
def test_slots_are_emptied_by_the_caller_where_no_thread_starts(torch_gpu, ctx, extra):
    """With the process at its limit of threads the calling thread empties all four slots, over 9 pieces and a remainder."""
    import resource

    src, want = source(torch_gpu, 9 * PIECE // 8 + extra)
    ring, got = Ring(), np.zeros_like(want)
    download(ring, got, src)  # allocates the slots
    assert np.array_equal(got, want)
    got[:] = 0
    soft, hard = resource.getrlimit(resource.RLIMIT_NPROC)
    resource.setrlimit(resource.RLIMIT_NPROC, (1, hard))
    try:
        download(ring, got, src)
    finally:
        resource.setrlimit(resource.RLIMIT_NPROC, (soft, hard))
    assert np.array_equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("pairs", [3, 20])
def test_correlations_into_pinned_memory(torch_gpu, ctx, pairs):
    """The public call with its result in pinned memory, below and above one piece, against pageable memory."""
    from ettk_amd.abi import default_params
    from ettk_amd.lib import Plan, check

    B = 16
    g = np.random.default_rng(pairs)
    sig, pat = g.standard_normal((2, pairs, 2 * B, 2 * B))
    plan = Plan(ctx, default_params(32, B))
    try:
        want = plan.so3_correlate(sig, pat)
        got = torch_gpu.zeros(want.size, dtype=torch_gpu.float64, pin_memory=True).numpy().reshape(want.shape)
        dp = C.POINTER(C.c_double)
        check(plan.lib.ettk_so3_correlate_batch(plan.h, pairs, sig.ctypes.data_as(dp), pat.ctypes.data_as(dp),
                                                got.ctypes.data_as(dp)))
        assert np.array_equal(got, want)
    finally:
        plan.close()
