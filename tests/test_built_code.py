"""Properties of the kernels that no run shows reliably, looked for in the built library's own instructions."""
import glob
import itertools
import os
import re
import shutil
import subprocess

import pytest

from tiny_llm_amd.kernels import library

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{name: instructions} of every kernel of the library."""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    tmp = tmp_path_factory.mktemp("listing")
    lib = shutil.copy(library.find_or_build(verbose=False), tmp / "kernels.so")
    subprocess.run([OBJDUMP, "--offloading", str(lib)], cwd=tmp, check=True, stdout=subprocess.DEVNULL)
    found, name = {}, None
    for part in sorted(glob.glob(str(tmp / f"*{library.ARCH}*"))):
        text = subprocess.run([OBJDUMP, "-d", part], check=True, capture_output=True, text=True).stdout
        for line in text.splitlines():
            if m := re.match(r"[0-9a-f]+ <(\S+)>:", line):
                name = m[1]
                found[name] = []
            elif name and line.startswith("\t"):
                found[name].append(line.split("//")[0].strip())
    assert found
    return found


def exchanges(lines, count):
    """Whether a listing passes blocks of `count` vectors through LDS in order: writes of a block and reads of a block in turn,
    all writes of it before the first read and all reads before the next write."""
    ops = [line.split()[0] for line in lines]
    ops = [o[3:7] for o in ops if o in ("ds_write_b128", "ds_read_b128")]
    runs = [(o, len(list(g))) for o, g in itertools.groupby(ops)]
    return bool(runs) and all(n % count == 0 for _, n in runs)


def main_loop(lines):
    """A kernel's instructions up to the barrier behind its main loop."""
    return lines[:next(i for i, line in enumerate(lines) if line.startswith("s_barrier"))]


def test_the_check_of_exchanges_finds_what_it_is_for():
    write, read = ["ds_write_b128 v1, v[2:5]"], ["ds_read_b128 v[2:5], v1"]
    assert exchanges(write * 4 + read * 4 + write * 4 + read * 4, 4)
    assert not exchanges(write * 3 + read + write + read * 3, 4)
    assert not exchanges(write * 4 + read * 3 + write * 4 + read, 4)
    assert not exchanges([], 4)


def test_a_wave_reads_a_block_once_it_is_written_whole(kernels):
    """The products of 6 to 64 rows turn whole lines into operands through LDS of a wave's own, without a barrier: the order of
    its instructions is all that keeps a block whole."""
    seen = 0
    for name, lines in kernels.items():
        m = re.search(r"gemm_stripe_(bf16_kernelILi(\d+)E|set_kernelI)Li(\d+)ELi(\d+)E", name)
        if not m:
            continue
        mt, ct, tk = int(m[2] or 1), int(m[3]), int(m[4])
        assert exchanges(main_loop(lines), (mt + ct) * tk // 32), name
        seen += 1
    assert seen


def scalar_offsets(lines):
    """The scalar offsets of a listing's buffer loads."""
    return [re.split(r",\s*(?![^\[]*\])", line)[3].split()[0] for line in lines if line.startswith("buffer_load_")]


def test_rows_beyond_a_matrix_are_beyond_a_lane_s_own_offset(kernels):
    """The kernels that fetch whole lines ask for rows beyond the matrices and for blocks beyond the inner size, and rely on the
    buffers' ends: of an offset only a lane's own part is sure to be compared with them."""
    assert scalar_offsets(["buffer_load_dwordx4 v[8:11], v94, s[4:7], s14 offen", "buffer_load_dword v8, v94, s[4:7], 0 offen"]) == ["s14", "0"]
    seen = 0
    for name, lines in kernels.items():
        if "gemm_stripe_" in name or "gemm_f32_lines_" in name:
            offsets = scalar_offsets(lines)
            seen += len(offsets)
            assert set(offsets) <= {"0"}, name
    assert seen
