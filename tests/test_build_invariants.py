"""Properties of the generated code that the sources rely on but cannot state themselves,
checked on the compiler's assembly listing (no GPU needed)."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "ellm_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fno-strict-aliasing", "-Xclang", "-target-feature",
         "-Xclang", "-packed-fp32-ops", "-Wno-int-to-pointer-cast", "--cuda-device-only", "-S"]


_listings = {}


def _listing(name, tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    if name not in _listings:
        out = tmp_path / (name + ".s")
        subprocess.run([HIPCC, *FLAGS, "-o", str(out), os.path.join(CSRC, name)], check=True,
                       capture_output=True, timeout=600)
        _listings[name] = out.read_text()
    return _listings[name]


def test_one_head_tile_kernels_leave_m0_to_the_inline_asm(tmp_path):
    """project_mid.hip sets M0 (the LDS address of a direct-to-LDS load) inside inline asm that
    cannot declare the write; that is sound only while the compiler keeps nothing of its own in
    M0, i.e. never indexes registers through it in these kernels."""
    text = _listing("project_mid.hip", tmp_path)
    code = [l.split(";")[0] for l in text.splitlines()]
    uses = [l for l in code if re.search(r"\bm0\b", l)]
    assert uses and all(re.fullmatch(r"\s*s_mov_b32 m0, s\d+\s*", l) for l in uses), \
        [l for l in uses if not re.fullmatch(r"\s*s_mov_b32 m0, s\d+\s*", l)][:5]
    assert not any("movrel" in l or "s_set_gpr_idx" in l for l in code)


def test_tile_kernel_leaves_m0_to_the_inline_asm(tmp_path):
    """The same for project.hip: every tile of it, the 256 x 256 ones and the one-head ones of the last round, is loaded
    that way."""
    text = _listing("project.hip", tmp_path)
    code = [l.split(";")[0] for l in text.splitlines()]
    uses = [l for l in code if re.search(r"\bm0\b", l)]
    assert uses and all(re.fullmatch(r"\s*s_mov_b32 m0, s\d+\s*", l) for l in uses)
    assert not any("movrel" in l or "s_set_gpr_idx" in l for l in code)


def test_chunk_kernels_leave_m0_to_the_inline_asm(tmp_path):
    """The same for prefill.hip, whose tile kernel fetches the tiles of long walks straight into LDS."""
    text = _listing("prefill.hip", tmp_path)
    code = [l.split(";")[0] for l in text.splitlines()]
    uses = [l for l in code if re.search(r"\bm0\b", l)]
    assert uses and all(re.fullmatch(r"\s*s_mov_b32 m0, s\d+\s*", l) for l in uses)
    assert not any("movrel" in l or "s_set_gpr_idx" in l for l in code)


def _ahead(lines, jumps, at, left):
    """Lines of the instructions within `left` wait states ahead of line `at`, along every path that leads there."""
    found, seen, work = set(), set(), [(at - 1, left, False)]
    while work:
        n, left, jumped = work.pop()
        while n >= 0 and left > 0 and (n, left) not in seen:
            seen.add((n, left))
            text = lines[n].strip()
            if (label := re.match(r"(\.LBB\d+_\d+):", text)):
                work += [(j, left, True) for j in jumps.get(label.group(1), [])]
            elif text and not text.startswith(".") and not text.endswith(":"):
                if not jumped and re.match(r"s_(branch|endpgm|setpc)", text):
                    break                                # nothing falls through from there
                found.add(n)
                nop = re.match(r"s_nop\s+(\d+)", text)
                left -= int(nop.group(1)) + 1 if nop else 1
            n, jumped = n - 1, False
    return found


def _scalars(text):
    out = set()
    for m in re.finditer(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", text):
        out |= set(range(int(m.group(1)), int(m.group(2)) + 1)) if m.group(1) else {int(m.group(3))}
    return out


@pytest.mark.parametrize("name", ["project.hip", "project_mid.hip", "prefill.hip"])
def test_descriptors_of_loads_in_inline_asm_are_not_fresh_from_the_vector_unit(name, tmp_path):
    """A scalar register written by a vector instruction (v_readfirstlane, v_readlane of a spilled one, v_cmp) may be
    read by a memory instruction five wait states later.  The compiler keeps that distance for its own loads, not for
    those in inline asm: their descriptor and offset registers must not have been written within it."""
    text = _listing(name, tmp_path)
    assert set(re.findall(r"\.sgpr_spill_count:\s*(\d+)", text)) == {"0"}
    lines = [re.split(r";|//", l)[0].rstrip() for l in text.splitlines()]
    jumps = {}
    for n, l in enumerate(lines):
        if (m := re.match(r"\s+s_c?branch\w*\s+(\.LBB\d+_\d+)", l)):
            jumps.setdefault(m.group(1), []).append(n)
    loads = [n for n, l in enumerate(lines) if re.search(r"buffer_load_dwordx4 .* lds$", l)]
    assert loads
    for at in loads:
        reads = _scalars(lines[at])
        for n in _ahead(lines, jumps, at, 5):
            if lines[n].strip().startswith("v_"):
                m = re.match(r"\s*(v_\w+)\s+([^,]+)(?:,\s*([^,]+))?", lines[n])
                written = _scalars(m.group(2)) | (_scalars(m.group(3) or "") if "_co_" in m.group(1) else set())
                assert not written & reads, (lines[n], lines[at])


@pytest.mark.parametrize("name", ["project.hip", "project_mid.hip", "project_small.hip", "prefill.hip", "decode.hip",
                                  "decode_balanced.hip", "kv_cache.hip", "attn_general.hip", "attn_general_chunk.hip",
                                  "attn_general_step.hip"])
def test_hot_kernels_do_not_spill(name, tmp_path):
    text = _listing(name, tmp_path)
    sizes = [int(x) for x in re.findall(r"\.private_segment_fixed_size:\s*(\d+)", text)]
    assert sizes and all(v == 0 for v in sizes), sizes


def _loops(lines):
    """(first, last) line ranges of backward branches: label ... s_cbranch to that label."""
    labels = {}
    for n, l in enumerate(lines):
        m = re.match(r"^(\.LBB\d+_\d+):", l)
        if m:
            labels[m.group(1)] = n
    out = []
    for n, l in enumerate(lines):
        m = re.match(r"\s+s_cbranch_\w+\s+(\.LBB\d+_\d+)", l)
        if m and m.group(1) in labels and labels[m.group(1)] < n:
            out.append((labels[m.group(1)], n))
    return out


@pytest.mark.parametrize("name,in_loop", [("project.hip", 0)])
def test_projection_kernels_keep_scratch_out_of_their_matrix_loops(name, in_loop, tmp_path):
    """The 256 x 256 tile kernel runs eight waves, two a SIMD, at up to 256 registers a lane: whatever the register
    allocator does with the epilogue's values, the K loop never touches scratch (the kernel has none
    today: test_hot_kernels_do_not_spill)."""
    text = _listing(name, tmp_path)
    lines = [l.split(";")[0] for l in text.splitlines()]
    for first, last in _loops(lines):
        body = lines[first:last + 1]
        if any("v_mfma" in l for l in body):
            assert sum("scratch_" in l for l in body) <= in_loop, (name, first, last)
