"""ettk_profile_query finds what ran: the names its documentation gives, and the form a strided pass took."""
import re
from pathlib import Path

import numpy as np
import pytest

from conftest import to_dev

HEADER = Path(__file__).resolve().parents[1] / "include" / "ettk_align.h"


@pytest.mark.gpu
def test_documented_names_are_recorded(torch_gpu, ctx):
    from ettk_amd.abi import Particle, default_params
    from ettk_amd.lib import Plan
    from ettk_amd.synth import blob_reference

    text = HEADER.read_text()
    names = re.findall(r'"(k_\w+(?:<\d+>)?)"', text[text.index("Measurement hooks"):])
    assert len(names) >= 3
    N = 64
    ref = to_dev(torch_gpu, blob_reference(N, seed=3))
    plan = Plan(ctx, default_params(N, 8))
    half = torch_gpu.empty((1, N, N, N // 2 + 1), dtype=torch_gpu.complex64, device="cuda")
    try:
        plan.set_reference(ref)
        ctx.profile(True)
        plan.ccc(ref[None], [Particle()], [0], np.eye(4)[None])
        ctx.fft3(ctx.FFT_R2C, N, 1, ref, half)
        got = {n: ctx.profile_query(n)[1] for n in names}
    finally:
        ctx.profile(False)
        plan.close()
    assert all(got.values()), got


@pytest.mark.gpu
@pytest.mark.parametrize("n,ran,other", [(64, "k_fft_strided", "k_fft_col"), (96, "k_fft_col", "k_fft_strided"),
                                         (256, "k_fft_col", "k_fft_strided")])
def test_strided_pass_is_recorded_as_what_ran(torch_gpu, ctx, n, ran, other):
    x = torch_gpu.zeros((1, n, n, n), dtype=torch_gpu.float32, device="cuda")
    half = torch_gpu.empty((1, n, n, n // 2 + 1), dtype=torch_gpu.complex64, device="cuda")
    torch_gpu.cuda.synchronize()
    try:
        ctx.profile(True)
        ctx.fft3(ctx.FFT_R2C, n, 1, x, half)
        assert ctx.profile_query(f"{ran}<{n}>")[1] == (2 if n > 128 else 1)
        assert ctx.profile_query(f"{other}<{n}>")[1] == 0
    finally:
        ctx.profile(False)
