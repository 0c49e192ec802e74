"""What shows only in the gfx950 assembly that hipcc makes of the sources
(compiled here; no GPU needed): the waits of the kernels whose LDS DMAs are
inline assembly, which the compiler does not count, and the registers that set
how many waves a SIMD holds."""
import os
import re
import subprocess

import pytest

from flaggems_vllm import _native


def _assembly(source, out):
    flags = [f for f in _native.HIPCC_FLAGS if f not in ("-fPIC", "-shared")]
    subprocess.run([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), *flags, "-S", "--cuda-device-only",
                    f"-I{_native._INCLUDE}", f"-I{_native._CSRC}", os.path.join(_native._CSRC, source), "-o", str(out)],
                   check=True, capture_output=True)
    return open(out).read()


@pytest.fixture(scope="module")
def mla_asm(tmp_path_factory):
    """{kernel name: its instructions and labels} of sparse_mla_decode.hip."""
    text, kernels = _assembly("sparse_mla_decode.hip", tmp_path_factory.mktemp("asm") / "mla.s"), {}
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


def test_paged_logits_registers(tmp_path):
    """Vector registers of the paged indexer logits, which loads each key tile's
    successor into the same registers: four waves per SIMD up to 64 heads (128
    registers), three at 128 heads with MXFP4 queries (168), and no spills."""
    text = _assembly("mqa_logits.hip", tmp_path / "mqa.s")
    seen = {}
    for m in re.finditer(r"\.name:\s+\S*paged_mqa_logits_kernelILb(\d)ELi(\d)E\S*\n(.*?)\.wavefront_size", text, re.S):
        count, spills = (int(re.search(rf"\.vgpr_{k}:\s+(\d+)", m.group(3)).group(1)) for k in ("count", "spill_count"))
        assert spills == 0
        key = (m.group(1) == "1", 16 * int(m.group(2)))
        seen[key] = max(count, seen.get(key, 0))
    assert set(seen) == {(fp4, heads) for fp4 in (False, True) for heads in (16, 32, 64, 128)}
    for (fp4, heads), count in seen.items():
        assert count <= (128 if heads <= 64 else 168 if fp4 else 256), (fp4, heads, count)
