"""Units of the general generator (``codegen/general.py``) as the compiler reports them: that some launches share the list of an output
row among wavefronts must not cost any kernel registers that it has with one wavefront (most outputs are never shared, and a kernel's
bound holds in all its launches)."""

import re
import subprocess

import pytest

from cuequivariance_amd import cue, jit
from cuequivariance_amd.tables import U1dTables

REPORT = "-Rpass-analysis=kernel-resource-usage"


def _scratch(report: str) -> dict:
    """{kernel: bytes of scratch memory per lane} of a compiler report."""
    out, kernel = {}, None
    for line in report.splitlines():
        if (m := re.search(r"Function Name: \S*(out\d+)_kernel", line)) is not None:
            kernel = m.group(1)
        elif (m := re.search(r"ScratchSize \[bytes/lane\]: (\d+)", line)) is not None:
            out[kernel] = int(m.group(1))
    return out


@pytest.mark.parametrize("code", [0, 1])  # float32, float64
@pytest.mark.parametrize("lout", [0, 1])
def test_no_kernel_spills_more_than_with_one_wavefront(jit_on, tmp_path, monkeypatch, lout, code):
    """All gradients of the gradients of a product basis (force training): 64 channels, degrees up to 2 into 0 or up to 1."""
    run, seen = subprocess.run, {}

    def recording(cmd, **kw):
        r = run([*cmd, REPORT] if REPORT not in cmd else cmd, **kw)
        source, = (c for c in cmd if c.endswith(".hip"))
        seen.update(source=open(source).read(), scratch=_scratch(r.stderr), cmd=cmd)
        return r

    monkeypatch.setattr(jit.subprocess, "run", recording)
    irreps = lambda l: cue.Irreps("O3", "+".join(f"64x{k}{'eo'[k % 2]}" for k in range(l + 1)))
    e, _ = cue.mace.symmetric_contraction(irreps(2), irreps(lout), range(1, 4))
    t = U1dTables.from_polynomial(e.polynomial.flatten_coefficient_modes().squeeze_modes())
    second = t.backward((True, True)).backward((True, True, True))
    assert jit.ensure_specialised(second, code, general=True)
    built = seen["scratch"]
    assert len(built) == 3

    # the same kernels when no launch may have more than one wavefront a block
    source = tmp_path / "one.hip"
    source.write_text(re.sub(r"__launch_bounds__\(\d+\)", "__launch_bounds__(64)", seen["source"]))
    cmd = [c for c in seen["cmd"] if not c.endswith((".hip", ".so")) and c not in ("-shared", "-o") and not c.startswith(("-L", "-l:", "-Wl"))]
    r = run([*cmd, *([] if REPORT in cmd else [REPORT]), "--cuda-device-only", "-c", str(source), "-o", str(tmp_path / "one.o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    one = _scratch(r.stderr)
    assert one.keys() == built.keys()
    assert all(built[k] <= one[k] for k in one), (built, one)
