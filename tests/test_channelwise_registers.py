"""Generated channel-wise units as the compiler reports them: a channel count that leaves lanes without a channel must not cost registers."""

import re
import subprocess

import pytest

from cuequivariance_amd import cue, jit
from cuequivariance_amd.tables import U1dTables


@pytest.mark.parametrize("channels,degrees,code", [(24, 2, 1), (40, 2, 1), (24, 3, 0)])  # code: float32, float64
def test_backward_of_masked_channels_does_not_spill(jit_on, monkeypatch, channels, degrees, code):
    """One SIMD holds two wavefronts of the backward for whole groups of lanes (32 channels, l <= 2 float64, l <= 3 float32); with branches around the
    stores of lanes that have a channel the same kernels spilled 70 to 750 registers."""
    run, seen = subprocess.run, {}

    def recording(cmd, **kw):
        r = run([*cmd, "-Rpass-analysis=kernel-resource-usage"], **kw)
        seen["report"] = r.stderr
        return r

    monkeypatch.setattr(jit.subprocess, "run", recording)
    irreps = lambda mul: cue.Irreps("O3", "+".join(f"{mul}x{k}{'eo'[k % 2]}" for k in range(degrees + 1)))
    e = cue.descriptors.channelwise_tensor_product(irreps(channels), irreps(1), "+".join(f"{k}{'eo'[k % 2]}" for k in range(degrees + 1)))
    assert jit.ensure_specialised(U1dTables.from_polynomial(e.polynomial.flatten_coefficient_modes().squeeze_modes()), code)
    scratch, kernel = {}, None
    for line in seen["report"].splitlines():
        if (m := re.search(r"Function Name: (\S+)", line)) is not None:
            kernel = m.group(1)
        elif (m := re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line)) is not None:
            scratch[kernel] = int(m.group(1))
    backward = {k: v for k, v in scratch.items() if "bwd_kernel" in k}
    assert len(backward) >= 4 and not any(backward.values()), backward
