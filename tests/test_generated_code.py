"""Waits in the gfx950 code of the kernels whose LDS DMAs are inline assembly.

The compiler counts no DMA that it did not issue itself, so where a kernel
relies on one, or must not drain one, shows only in the assembly that hipcc
makes of the sources (compiled here; no GPU needed)."""
import os
import re
import subprocess

import pytest

from flaggems_vllm import _native


@pytest.fixture(scope="module")
def mla_asm(tmp_path_factory):
    """{kernel name: its instructions and labels} of sparse_mla_decode.hip."""
    out = str(tmp_path_factory.mktemp("asm") / "mla.s")
    flags = [f for f in _native.HIPCC_FLAGS if f not in ("-fPIC", "-shared")]
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), *flags, "-S", "--cuda-device-only",
                    f"-I{_native._INCLUDE}", f"-I{_native._CSRC}",
                    os.path.join(_native._CSRC, "sparse_mla_decode.hip"), "-o", out], check=True, capture_output=True)
    text, kernels = open(out).read(), {}
    for m in re.finditer(r"^_ZN\w*?\d+(sparse_mla_\w+?_kernel)\w*:[^\n]*\n(.*?)^\.Lfunc_end", text, re.S | re.M):
        lines = (line.split(";")[0].strip() for line in m.group(2).split("\n"))
        kernels.setdefault(m.group(1), [line for line in lines if line and not line.startswith((".p2align", ".loc"))])
    return kernels


def test_pair_kernel_waits_for_its_length_dmas(mla_asm):
    """The barrier that hands the top-k lengths over (the first past the chunk
    loops) waits for every DMA of the wave, also where a half has had no
    chunk to wait for."""
    code = mla_asm["sparse_mla_decode_pair_kernel"]
    last = max(i for i, line in enumerate(code) if line.startswith("v_mfma"))
    at = next(i for i in range(last, len(code)) if code[i].startswith("s_barrier"))
    before = code[at - 4:at]
    assert any(re.match(r"s_waitcnt\b.*vmcnt\(0\)", line) for line in before), before
