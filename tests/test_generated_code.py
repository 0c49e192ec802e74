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


@pytest.mark.parametrize("kernel", ["decode", "decode_pieces", "decode_split", "decode_pair"])
def test_no_wait_drains_a_gather(mla_asm, kernel):
    """Behind a raw gather (its scale words go last), no wait for vector
    memory before q's loads go out (the first gather), nor before the current
    chunk's scores, 32 MFMAs, are made (the chunk loops'): either would also
    wait for the gather, which is meant to land under them.  The gather under
    the first chunk is left out where that chunk has code of its own (its
    scores wait for q), and so is the paired kernel's first (its q addresses
    are reloaded registers)."""
    code, seen = mla_asm[f"sparse_mla_{kernel}_kernel"], []
    for i, line in enumerate(code):
        if not line.startswith("global_load_lds_dword "):
            continue
        at = next((j for j in range(i, len(code)) if code[j].startswith(("v_mfma", "global_load_dwordx4"))), None)
        if at is None:
            continue
        first = code[at].startswith("global_load_dwordx4")
        end = at if first else [j for j in range(at, len(code)) if code[j].startswith("v_mfma")][31]
        seen.append((first, [x for x in code[i:end] if re.match(r"s_waitcnt\b.*vmcnt", x)]))
    if kernel == "decode_pair":
        seen = [s for s in seen if not s[0]]
        assert len(seen) == 1
    else:
        assert [s[0] for s in seen] == [True, False, False]
        del seen[1]
    assert not any(waits for _, waits in seen), seen
