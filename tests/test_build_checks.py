"""CPU tests of the build-time assembly check for inline-asm loads
(vllm-exact_amd/check_async_loads.py): it must reject a destination register touched before
the covering wait (straight line, through a branch, around a loop), a path that ends
uncovered, and compiler-generated M0 use, and accept the same code once a wait covers it; and of
the registers of the built kernels."""
import re
import struct
import subprocess
import sys
from pathlib import Path

import msgpack

ROOT = Path(__file__).resolve().parents[1]
CHECK = ROOT / "vllm-exact_amd" / "check_async_loads.py"


def run(tmp_path, body):
    asm = tmp_path / "k.s"
    asm.write_text("_Zkernel:\n" + body + "\n.Lfunc_end0:\n")
    return subprocess.run([sys.executable, str(CHECK), str(asm), "_Zkernel"], capture_output=True, text=True)


LOAD = ";;#ASMSTART\nglobal_load_dwordx4 v[4:7], v[0:1], off\n;;#ASMEND\n"


def test_accepts_covered_load(tmp_path):
    r = run(tmp_path, LOAD + "global_load_dwordx4 v[8:11], v[2:3], off\ns_waitcnt vmcnt(1)\nv_mov_b32 v5, 0\ns_endpgm")
    assert r.returncode == 0, r.stdout


def test_rejects_touch_before_wait(tmp_path):
    r = run(tmp_path, LOAD + "v_mov_b32 v5, 0\ns_waitcnt vmcnt(0)\ns_endpgm")
    assert r.returncode == 1 and "v_mov_b32 v5" in r.stdout


def test_rejects_wait_that_does_not_cover(tmp_path):
    # vmcnt(1) with no younger memory operation leaves this load possibly in flight
    r = run(tmp_path, LOAD + "s_waitcnt vmcnt(1)\nv_add_u32_e32 v1, v6, v1\ns_waitcnt vmcnt(0)\ns_endpgm")
    assert r.returncode == 1


def test_rejects_touch_on_branch_path(tmp_path):
    body = (LOAD + "s_cbranch_scc1 .LBB0_2\ns_waitcnt vmcnt(0)\ns_branch .LBB0_3\n.LBB0_2:\nv_mov_b32 v7, 1\n"
            ".LBB0_3:\ns_waitcnt vmcnt(0)\ns_endpgm")
    r = run(tmp_path, body)
    assert r.returncode == 1 and "v_mov_b32 v7" in r.stdout


def test_rejects_uncovered_end_and_loop_reuse(tmp_path):
    assert run(tmp_path, LOAD + "s_endpgm").returncode == 1
    body = (".LBB0_1:\n" + LOAD + "v_mfma_i32_16x16x64_i8 a[0:3], v[4:7], v[4:7], a[0:3]\n"
            "s_cbranch_scc1 .LBB0_1\ns_waitcnt vmcnt(0)\ns_endpgm")
    assert run(tmp_path, body).returncode == 1


def test_rejects_compiler_m0_use(tmp_path):
    r = run(tmp_path, "s_mov_b32 m0, s2\n" + LOAD + "s_waitcnt vmcnt(0)\ns_endpgm")
    assert r.returncode == 1 and "m0" in r.stdout


def kernel_metadata(lib):
    """The kernels' metadata (AMDGPU notes, msgpack) of every gfx950 code object in the library."""
    data, pos = lib.read_bytes(), 0
    while (pos := data.find(b"\x7fELF", pos)) >= 0:
        if struct.unpack_from("<H", data, pos + 18)[0] == 224:  # e_machine: EM_AMDGPU
            shoff, = struct.unpack_from("<Q", data, pos + 40)
            shentsize, shnum = struct.unpack_from("<HH", data, pos + 58)
            for i in range(shnum):
                _, kind, _, _, offset = struct.unpack_from("<IIQQQ", data, pos + shoff + i * shentsize)
                if kind == 7:  # SHT_NOTE: sizes of the name and of the contents, type, name padded to 4
                    name, size, _ = struct.unpack_from("<III", data, pos + offset)
                    at = pos + offset + 12 + (name + 3) // 4 * 4
                    yield from msgpack.unpackb(data[at:at + size]).get("amdhsa.kernels", [])
        pos += 4


def test_kernels_use_no_scratch():
    """No kernel spills, but paged decode away from the default constants (16 keys a step, 4 waves):
    its steps of 64 keys or 8 waves of many heads have more accumulators than registers."""
    kernels = list(kernel_metadata(ROOT / "vllm-exact_amd" / "vllm_exact" / "libvllm_exact_amd.so"))
    assert len(kernels) > 100
    for k in kernels:
        paged = re.search(r"paged_partial_kernelILi\d+ELi\d+ELi(\d+)ELi(\d+)E", k[".name"])
        if not paged or paged.groups() == ("1", "4"):
            assert k[".private_segment_fixed_size"] == 0, k[".name"]
