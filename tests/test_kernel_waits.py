"""LDS-direct loads and the barriers that publish them, in the built code.

``s_barrier`` does not wait for a wave's outstanding LDS-direct loads, and the
compiler adds a wait only ahead of that wave's own LDS reads: a wave without any
must wait by itself. A run on the GPU shows a missing wait only when a load
happens to be late, so the instructions are read instead: the attention kernels
are compiled to assembly and every path from such a load to the next barrier has
to pass ``s_waitcnt vmcnt(0)``.
"""

import os
import re
import shutil
import subprocess

import pytest

import build_hip

HIPCC = shutil.which(build_hip.HIPCC)
DMA_FORMS = (
    [(d, "ROWS_DMA", c, w, 1) for d in (64, 128) for c in (0, 1) for w in (0, 1)]
    + [(128, "PAGES_DMA", 1, w, 1) for w in (0, 1)]
    + [(d, "PAGES_DMA", 1, w, 3) for d in (64, 128) for w in (0, 1)]
)


def unwaited_barriers(lines):
    """Barriers (line numbers) that an LDS-direct load can reach in flight."""
    label = {}
    for i, line in enumerate(lines):
        m = re.match(r"(\.L\w+):", line)
        if m:
            label[m.group(1)] = i
    seen = set()
    found = set()
    work = [(0, False)]
    while work:
        i, flying = work.pop()
        while i < len(lines) and (i, flying) not in seen:
            seen.add((i, flying))
            op, _, args = lines[i].strip().partition(" ")
            args = args.split(";")[0]
            if op.startswith("global_load_lds") or (
                op.startswith("buffer_load") and re.search(r"\blds\b", args)
            ):
                flying = True
            elif op == "s_waitcnt" and "vmcnt(0)" in args:
                flying = False
            elif op == "s_barrier" and flying:
                found.add(i)
            elif op.startswith("s_cbranch") or op == "s_branch":
                work.append((label[args.strip()], flying))
                if op == "s_branch":
                    break
            elif op == "s_endpgm":
                break
            i += 1
    return sorted(found)


def kernels(asm: str):
    """(name, instruction lines) of each function in an assembly listing."""
    asm = asm.replace("\t", " ")
    for m in re.finditer(r"^(_Z\w+):.*?^\.Lfunc_end\d+:", asm, re.M | re.S):
        yield m.group(1), m.group(0).splitlines()[1:]


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc")
@pytest.mark.parametrize("fast_math", [False, True])
def test_prefill_attention_waits_for_lds_loads(tmp_path, fast_math):
    src = tmp_path / "forms.hip"
    src.write_text(
        '#include "mfma_attention.h"\nnamespace {\n'
        + "".join(
            "template __global__ void mfma_attn::prefill_attention_kernel"
            f"<{d}, mfma_attn::{s}, {bool(c):d}, {bool(w):d}, {p}>"
            "(const mfma_attn::PrefillArgs);\n"
            for d, s, c, w, p in DMA_FORMS
        )
        + "}\n"
    )
    out = tmp_path / "forms.s"
    subprocess.run(
        [HIPCC, "-S", "--cuda-device-only", str(src), "-o", str(out),
         f"--offload-arch={build_hip.ARCH}", "-O3", "-std=c++17",
         f"-I{build_hip.CSRC}", *build_hip.DEVICE_FLAGS,
         *(["-ffast-math"] if fast_math else [])],
        check=True, capture_output=True, env={**os.environ, "TMPDIR": str(tmp_path)},
    )
    listed = list(kernels(out.read_text()))
    assert len(listed) == len(DMA_FORMS)
    for name, lines in listed:
        text = "\n".join(lines)
        assert "global_load_lds" in text and "s_barrier" in text, name
        assert not unwaited_barriers(lines), name


def test_skipped_wait_is_seen():
    body = """
 global_load_lds_dwordx4 v[2:3], off
 s_cbranch_vccz .LBB0_2
 s_waitcnt vmcnt(0)
.LBB0_2:
 s_barrier
 s_endpgm""".splitlines()
    assert unwaited_barriers(body) == [5]
    assert not unwaited_barriers(body[:1] + body[1:2] + body[3:])
