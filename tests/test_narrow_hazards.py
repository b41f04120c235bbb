"""The SwiGLU, int8 and many-wave forms of the skinny GEMM tie their MFMA
accumulators by inline asm as the plain ones do: the same scan of the
gfx950 assembly (see test_pinned_hazards.py) over narrow_dma_kernel and
narrow_lds_kernel."""
import re
import subprocess

import pytest

from test_pinned_hazards import (HIPCC, PKG, REPO, _acc_regs, _operands, _touches,
                                 _unsettled_acc_read, _unsettled_acc_write, _valu_hazards)


@pytest.fixture(scope="module")
def bodies():
    import pathlib
    if not pathlib.Path(HIPCC).exists():
        pytest.skip("hipcc not available")
    out = subprocess.run(
        [HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17",
         "-Wno-unused-command-line-argument",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         f"-I{REPO / 'include'}", f"-I{PKG / 'csrc'}", "--cuda-device-only", "-S",
         str(PKG / "csrc" / "u15h_kernels.hip"), "-o", "-"],
        capture_output=True, text=True, timeout=600, check=True).stdout
    found, name = {}, None
    for raw in out.splitlines():
        if re.match(r"^_Z\S*narrow_(?:dma|lds|pack)_kernel\S*:", raw):
            name = raw.split(":")[0]
            found[name] = []
        elif name is not None:
            s = raw.strip()
            if s.startswith(".amdhsa_kernel") or raw.startswith(".Lfunc_end"):
                name = None
            elif s and not s.startswith((";", ".")) and not s.endswith(":"):
                found[name].append(s)
    assert found
    return found


def test_tied_accumulators_and_wait_states(bodies):
    for name, body in bodies.items():
        mfma = [s for s in body if s.startswith("v_mfma")]
        assert mfma, name
        assert not _valu_hazards(body), (name, _valu_hazards(body)[:3])
        assert _unsettled_acc_read(body) is None, (name, _unsettled_acc_read(body))
        assert _unsettled_acc_write(body) is None, (name, _unsettled_acc_write(body))
        acc = _acc_regs(body)
        idx = [i for i, s in enumerate(body) if s.startswith("v_mfma")]
        assert not any(_touches(s, acc) for s in body[idx[0]:idx[-1]]
                       if not s.startswith("v_mfma")), name
        for s in mfma:
            assert _operands(s)[0] == _operands(s)[3], s
