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


def compiled(src, tmp_path, fast_math):
    """{name: instruction lines} of a source's kernels."""
    out = tmp_path / "kernels.s"
    subprocess.run(
        [HIPCC, "-S", "--cuda-device-only", str(src), "-o", str(out),
         f"--offload-arch={build_hip.ARCH}", "-O3", "-std=c++17",
         f"-I{build_hip.CSRC}", *build_hip.DEVICE_FLAGS,
         *(["-ffast-math"] if fast_math else [])],
        check=True, capture_output=True, env={**os.environ, "TMPDIR": str(tmp_path)},
    )
    return dict(kernels(out.read_text()))


def in_flight(lines):
    """(most LDS-direct loads in flight at each barrier, by line, over all paths;
    lines with other vector accesses before the last barrier: they would be counted
    too)"""
    label = {m.group(1): i for i, x in enumerate(lines) if (m := re.match(r"(\.L\w+):", x))}
    most, others, seen = {}, set(), set()
    work = [(0, 0)]
    while work:
        i, n = work.pop()
        while i < len(lines) and (i, n) not in seen:
            seen.add((i, n))
            op, _, args = lines[i].strip().partition(" ")
            args = args.split(";")[0]
            if re.match(r"(buffer|global|flat|scratch)_", op):
                if re.search(r"\blds\b", args):
                    n = min(n + 1, 64)
                else:
                    others.add(i)
            elif op == "s_waitcnt" and (m := re.search(r"vmcnt\((\d+)\)", args)):
                n = min(n, int(m.group(1)))
            elif op == "s_barrier":
                most[i] = max(n, most.get(i, 0))
            elif op.startswith("s_cbranch") or op == "s_branch":
                work.append((label[args.strip()], n))
                if op == "s_branch":
                    break
            elif op == "s_endpgm":
                break
            i += 1
    return most, {i for i in others if i < max(most)}


def ring_faults(lines, loads: int, slots: int):
    """What is wrong with the counted waits of a ring of ``slots`` steps, ``loads``
    LDS-direct loads each (a wave's). At a barrier the step that follows has landed,
    the loads of the ``slots`` - 2 after it may be in flight. Ahead of the first one,
    which short products reach by another branch, the wait is looked for by its
    count: those and the loads of the last step that go out early."""
    most, others = in_flight(lines)
    rest = sorted(most)[1:]
    early = loads if slots == 2 else (loads + 1) // 2
    waits = {int(x) for line in lines[: max(most)] for x in re.findall(r"vmcnt\((\d+)\)", line)}
    faults = [f"another access, line {i}" for i in sorted(others)]
    faults += [
        f"{most[i]} loads in flight at line {i}" for i in rest if most[i] > loads * (slots - 2)
    ]
    if waits != {0, loads * (slots - 2), loads * (slots - 2) + early}:
        faults.append(f"waits for {waits}")
    return faults


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc")
def test_product_rings_count_their_loads(tmp_path):
    listed = compiled(os.path.join(build_hip.CSRC, "dense_gemm.hip"), tmp_path, True)
    assert len(listed) == 18  # the encoder's tiles with either epilogue, those of many rows
    for name, lines in listed.items():
        tn, tm, wn, wm, slots, _ = map(int, re.findall(r"Li(\d+)E", name))
        loads = (tn + tm) // 8 // (wn * wm)
        assert sum(bool(re.search(r"\blds\b", x)) for x in lines) >= 2 * loads, name
        assert not ring_faults(lines, loads, slots), name
        # mistakes in the listing are seen: a count too high, an access more
        waits = [i for i, x in enumerate(lines) if re.search(rf"vmcnt\({loads * (slots - 2)}\)", x)]
        late = list(lines)
        for i in waits:
            late[i] = f" s_waitcnt vmcnt({loads * (slots - 2) + 1})"
        assert ring_faults(late, loads, slots), name
        assert ring_faults([" global_load_dword v0, v[0:1], off"] + lines, loads, slots), name


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc")
def test_few_row_rings_count_their_loads(tmp_path):
    listed = compiled(os.path.join(build_hip.CSRC, "skinny_gemm.hip"), tmp_path, True)
    listed = {n: x for n, x in listed.items() if "dense_gemm_kernel" in n}
    # 12 tiles and 2 for long rows with four epilogues, but those of dense_gemm.hip
    assert len(listed) == 54
    for name, lines in listed.items():
        tn, tm, wn, wm, slots, _ = map(int, re.findall(r"Li(\d+)E", name))
        loads = (tn + tm) // 8 // (wn * wm)
        lines = [re.sub(r"global_load_lds_dwordx4 (.*)", r"global_load_dwordx4 \1 lds", x)
                 for x in lines]
        assert sum(bool(re.search(r"\blds\b", x)) for x in lines) >= 2 * loads, name
        assert not ring_faults(lines, loads, slots), name


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
    listed = compiled(src, tmp_path, fast_math)
    assert len(listed) == len(DMA_FORMS)
    for name, lines in listed.items():
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


def unpublished_reads(lines):
    """Reads of an LDS word at a fixed address (their lines, by address) that a path
    from a write of it reaches without a barrier between: other waves may not see the
    value. An address is the last constant moved to its register above."""
    label, const, access = {}, {}, {}
    for i, line in enumerate(lines):
        if m := re.match(r"(\.L\w+):", line):
            label[m.group(1)] = i
            continue
        op, _, args = line.strip().partition(" ")
        args = args.split(";")[0]
        if m := re.match(r"ds_(read|write)_b(32|64|128)$", op):
            regs = re.findall(r"v\[?(\d+)", args)
            at = const.get(int(regs[1 if m.group(1) == "read" else 0]))
            if at is not None:
                off = re.search(r"offset:(\d+)", args)
                at += int(off.group(1)) if off else 0
                words = range(at, at + int(m.group(2)) // 8, 4)
                access[i] = (m.group(1), set(words))
        if not re.match(r"(ds_write|global_store|buffer_store|s_|v_cmp)", op):
            if m := re.match(r"v(\d+)\b|v\[(\d+):(\d+)\]", args):
                lo, hi = (m.group(1),) * 2 if m.group(1) else m.group(2, 3)
                for r in range(int(lo), int(hi) + 1):
                    const.pop(r, None)
        if m := re.match(r"v_mov_b32(?:_e32)? v(\d+), (0x[0-9a-f]+|\d+)$",
                         line.strip().split(";")[0].strip()):
            const[int(m.group(1))] = int(m.group(2), 0)
    found = {}
    for start, (kind, words) in access.items():
        if kind != "write":
            continue
        seen, work = set(), [start + 1]
        while work:
            i = work.pop()
            while i < len(lines) and i not in seen:
                seen.add(i)
                op, _, args = lines[i].strip().partition(" ")
                if op in ("s_barrier", "s_endpgm"):
                    break
                if access.get(i, ("",))[0] == "read" and words & access[i][1]:
                    found.setdefault(min(words), set()).add(i)
                if op.startswith("s_cbranch") or op == "s_branch":
                    work.append(label[args.split(";")[0].strip()])
                    if op == "s_branch":
                        break
                i += 1
    return found


@pytest.mark.skipif(HIPCC is None, reason="needs hipcc")
@pytest.mark.parametrize("fast_math", [False, True])
def test_sampler_publishes_what_it_shares(tmp_path, fast_math):
    """What one thread of the sampler with limits leaves in LDS for the block: a run
    shows a missing barrier only when a wave happens to be ahead."""
    listed = compiled(os.path.join(build_hip.CSRC, "sampling.hip"), tmp_path, fast_math)
    (lines,) = [x for n, x in listed.items() if "topk_topp_sample" in n]
    assert not unpublished_reads(lines)
    # taken from the listing, each of the first pass's last barriers is missed
    barriers = [i for i, x in enumerate(lines) if x.strip().startswith("s_barrier")]
    assert any(
        unpublished_reads(lines[:i] + [""] + lines[i + 1 :]) for i in barriers
    )


def test_unpublished_read_is_seen():
    body = """
 v_mov_b32_e32 v1, 0x40
 s_cbranch_execz .LBB0_2
 ds_write_b32 v1, v2 offset:4
.LBB0_2:
 v_mov_b32_e32 v3, 0x44
 ds_read_b32 v4, v3
 s_endpgm""".splitlines()
    assert unpublished_reads(body) == {0x44: {6}}
    assert not unpublished_reads(body[:5] + [" s_barrier"] + body[5:])
    assert not unpublished_reads(body[:5] + [" v_mov_b32_e32 v3, 0x48"] + body[6:])
