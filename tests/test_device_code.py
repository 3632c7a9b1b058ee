"""Properties of the built device code that running it cannot show (no GPU needed).

Global->LDS loads (global_load_lds_dword) write LDS when their data arrives and
count in vmcnt; LDS reads count in lgkmcnt, and nothing orders the two. A wave
that stages rows over a tile it has just read therefore has to wait for its reads
first (lgkmcnt), else a load that returns early replaces values still to be
read. The wait is missing or there in the instructions, so the test reads those:
no path through any kernel may reach a global->LDS load with an LDS read of the
wave outstanding.

The loads are inline assembly, whose registers the compiler has to accept: staging
code compiles without a warning, and the build stops at one.
"""
import glob
import os
import re
import shutil
import subprocess

import pytest

from tridsolver_amd import _lib
from tridsolver_amd import build as B

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
INSTR = re.compile(r"^\t(\S+)(.*?)// 0*([0-9A-F]+):(?: [0-9A-F]{8})+(?: <(.*)\+0x([0-9a-f]+)>)?")
HEAD = re.compile(r"^0*([0-9a-f]+) <(.*)>:")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> [(address, mnemonic, operands, branch target or None)] of every
    kernel that has a global->LDS load."""
    if not os.path.exists(_lib.LIBPATH):
        pytest.fail("libtridhip.so is not built (python -m tridsolver_amd.build)")
    tmp = tmp_path_factory.mktemp("device_code")
    lib = shutil.copy(_lib.LIBPATH, tmp)
    subprocess.run([OBJDUMP, "--offloading", os.path.basename(lib)], cwd=tmp, check=True,
                   capture_output=True)
    found = {}
    for obj in sorted(glob.glob(str(tmp / "*gfx950"))):
        text = subprocess.run([OBJDUMP, "-d", obj], check=True, capture_output=True,
                              text=True).stdout
        if "global_load_lds" not in text:
            continue
        name, start, code = None, {}, {}
        for line in text.splitlines():
            m = HEAD.match(line)
            if m:
                name = m.group(2)
                start[name], code[name] = int(m.group(1), 16), []
                continue
            m = INSTR.match(line)
            if m and name:
                target = None
                if m.group(5):
                    target = start[m.group(4)] + int(m.group(5), 16)
                elif "branch" in m.group(1):  # a branch to the kernel's first instruction
                    target = start[name]
                code[name].append((int(m.group(3), 16), m.group(1), m.group(2), target))
        found.update({k: v for k, v in code.items()
                      if any(op.startswith("global_load_lds") for _, op, _, _ in v)})
    assert found, "no kernel with a global->LDS load in the library"
    return found


def unordered_stages(code):
    """Addresses of global->LDS loads that some path reaches with an LDS read
    outstanding. LDS operations complete in order, so a read with k of them behind
    it is done after a wait for lgkmcnt <= k; the state is the smallest such k on
    any path, None with no read outstanding."""
    at = {a: i for i, (a, _, _, _) in enumerate(code)}
    none = 1 << 30
    state, bad, work = {0: none}, set(), [0]
    while work:
        i = work.pop()
        k = state[i]
        while True:
            addr, op, args, target = code[i]
            if op.startswith("ds_read"):
                k = 0
            elif op.startswith("ds_"):
                k += k < none
            elif op == "s_waitcnt":
                m = re.search(r"lgkmcnt\((\d+)\)", args)
                if m and int(m.group(1)) <= k:
                    k = none
            elif op.startswith("global_load_lds") and k < none:
                bad.add(addr)
            if target is not None:
                j = at[target]
                if k < state.get(j, none + 1):
                    state[j] = k
                    work.append(j)
            if op in ("s_branch", "s_endpgm") or i + 1 == len(code):
                break
            i += 1
            if i in state or target is not None:  # a block's first instruction
                if k >= state.get(i, none + 1):
                    break
                state[i] = k
    return sorted(bad)


def test_the_scan_finds_a_missing_wait():
    """The scan on hand-written sequences: a read right before the load, one behind a
    wait that does not reach it, one on a loop's back edge, and the sound forms."""
    def scan(*ops):
        ops = [o if isinstance(o, tuple) else (o,) for o in ops]
        return unordered_stages([(i, *o, *("", None)[len(o) - 1:]) for i, o in enumerate(ops)])
    lds, end = "global_load_lds_dword", "s_endpgm"
    assert scan("ds_read2_b64", lds, end) == [1]
    assert scan("ds_read_b64", ("s_waitcnt", " lgkmcnt(0)"), lds, end) == []
    assert scan("ds_read_b64", ("s_waitcnt", " vmcnt(0)"), lds, end) == [2]
    assert scan("ds_read_b64", "ds_write_b64", ("s_waitcnt", " lgkmcnt(1)"), lds, end) == []
    assert scan("ds_write_b64", "ds_read_b64", ("s_waitcnt", " lgkmcnt(1)"), lds, end) == [3]
    assert scan(lds, "ds_read_b64", ("s_cbranch_scc1", "", 0), end) == [0]
    assert scan(("s_cbranch_scc1", "", 2), "ds_read_b64", lds, end) == [2]


def test_no_stage_over_lds_reads_in_flight(kernels):
    bad = {name: ["%x" % a for a in found[:4]] for name, code in kernels.items()
           for found in [unordered_stages(code)] if found}
    assert not bad, "global->LDS loads behind unfinished LDS reads: %s" % bad


def test_staging_compiles_without_warnings(tmp_path):
    src = tmp_path / "stage.hip"
    src.write_text('#include "wide_core.hpp"\n'
                   '__global__ void k(const double *a, double *o, int N, int64_t nsys) {\n'
                   '  extern __shared__ double t[];\n'
                   '  trid::wide::wide_stage<double, 16, 256, 2, false>(\n'
                   '      a, trid::hyb::lds_address(t), 0, threadIdx.x, 4096u, N, nsys);\n'
                   '  trid::hyb::stage_wait_all();\n'
                   '  o[threadIdx.x] = t[threadIdx.x];\n'
                   '}\n')
    r = subprocess.run([B.HIPCC] + [f for f in B.CFLAGS if f != "-Werror"] +
                       ["-I" + B.CSRC, "-c", str(src), "-o", str(tmp_path / "stage.o")],
                       capture_output=True, text=True)
    assert r.returncode == 0 and "warning:" not in r.stderr, r.stderr[:2000]
    assert "-Werror" in B.CFLAGS


def test_registers_of_the_largest_fp32_workgroups(tmp_path):
    """The strided FP32 kernel at 16 rows of 128 bytes runs up to 1024 threads; two such
    workgroups share a CU only at 64 VGPRs or fewer."""
    lib = shutil.copy(_lib.LIBPATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", os.path.basename(lib)], cwd=tmp_path, check=True,
                   capture_output=True)
    found = {}
    for obj in glob.glob(str(tmp_path / "*gfx950")):
        notes = subprocess.run([os.path.join(os.path.dirname(OBJDUMP), "llvm-readelf"), "--notes",
                                obj], check=True, capture_output=True, text=True).stdout
        for name, vgprs in re.findall(r"\.symbol: +(\S+)\.kd.*?\.vgpr_count: +(\d+)", notes, re.S):
            if "hybrid_wide_kernelIfLi16ELi128E" in name:
                found[name] = int(vgprs)
    assert len(found) == 4 and max(found.values()) <= 64, found
