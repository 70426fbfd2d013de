"""Build rules the GPU found the hard way, checked on the CPU by cross-compiling every kernel source to gfx950 assembly.

Rule 1: no packed fp32 operation (v_pk_fma_f32 / v_pk_mul_f32 / v_pk_add_f32) in any kernel.  hipcc -O3 forms them by itself from ordinary
float code, and the forms that read the high dword of a VGPR src1 pair in the low lane return wrong results while another wave of the same
SIMD issues MFMAs (profiles/r04_pkfma_probe.txt) -- parity-green and bit-stable alone, wrong beside a neighbour.  The libraries are built
with the feature off (build.FLAGS); this test compiles with the same flags and looks at what came out.

Rule 2: no scratch memory in the kernels of the language models' library and in the talker's persistent launches.  A tile kernel whose epilogue outgrew the
compiler's unrolling kept its accumulators there -- right results, 25 us more per launch.  The all-pass launch that ends in the step's tail is the one
exception: its two calls that are not inlined have a stack, once a launch."""
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from ht_vllm_omni_amd import build as B

CSRC = B.CSRC
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
PACKED = re.compile(r"^\s*(v_pk_(?:fma|mul|add)_f32)\b")


def _asm(name, tmp_path, defines=()):
    out = os.path.join(tmp_path, name + ".s")
    subprocess.run([HIPCC, *B.FLAGS, *B.EXTRA.get(name, []), *defines, "-S", "--cuda-device-only", os.path.join(CSRC, name), "-o", out],
                   check=True, capture_output=True, timeout=900)
    return open(out).read().split("\n")


def packed_fp32(lines):
    return [l.strip() for l in lines if PACKED.match(l)]


def scratch_bytes(lines):
    return [int(m.group(1)) for m in (re.match(r"^; ScratchSize: (\d+)", l) for l in lines) if m]


def kernel_scratch(lines):
    """{kernel: scratch bytes a lane}: the first size behind each kernel's label"""
    out, name = {}, None
    for l in lines:
        m = re.match(r"^(_Z\w+):", l)
        name = m.group(1) if m else name
        m = re.match(r"^; ScratchSize: (\d+)", l)
        if m and "_kernel" in name:
            out.setdefault(name, int(m.group(1)))
    return out


def test_the_scanner_sees_the_form():
    got = packed_fp32(["_Zk:", "\tv_pk_fma_f32 v[0:1], v[2:3], v[4:5], v[0:1] op_sel:[0,1,0]", "\tv_pk_mul_f32 v[0:1], v[2:3], v[4:5]",
                       "\tv_pk_add_f32 v[0:1], v[2:3], s[4:5]", "\tv_pk_fma_f16 v0, v1, v2, v3", "\tv_fma_f32 v0, v1, v2, v3"])
    assert len(got) == 3


def test_the_feature_is_off_in_the_flags():
    f = B.FLAGS
    i = f.index("-packed-fp32-ops")
    assert f[i - 3:i] == ["-Xclang", "-target-feature", "-Xclang"]


# both builds: the product, and the diagnostics build (-DOMNI_DEBUG_HOOKS turns the policy knobs into run-time variables: other code)
@pytest.mark.parametrize("defines", [(), ("-DOMNI_DEBUG_HOOKS",)], ids=["product", "debug-hooks"])
@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_no_kernel_holds_a_packed_fp32_op(tmp_path, defines):
    names = sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))
    with ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as pool:
        asms = list(pool.map(lambda n: _asm(n, str(tmp_path), defines), names))
    bad = [(n, x) for n, lines in zip(names, asms) for x in packed_fp32(lines)]
    assert sum(len(a) for a in asms) > 10000
    assert not bad, f"{len(bad)} packed fp32 ops, e.g. {bad[:4]}"
    if not defines:
        chains = {}
        for n in ("cp_chain.hip", "bb_chain.hip"):
            chains |= kernel_scratch(asms[names.index(n)])
        tail = {k for k in chains if "cp_chain_kernelILi64ELi" in k and "ELi0E" not in k}
        assert len(chains) > 20 and len(tail) == 2
        assert all(chains[k] <= 352 for k in tail) and not any(v for k, v in chains.items() if k not in tail), {k: v for k, v in chains.items() if v}
        scratch = {n: scratch_bytes(lines) for n, lines in zip(names, asms) if n in B.DECODER_SOURCES}
        assert sum(map(len, scratch.values())) > 50
        assert not any(map(any, scratch.values())), {n: v for n, v in scratch.items() if any(v)}


@pytest.mark.skipif(not os.path.exists(B.LIB_DECODER), reason="libomni_decoder.so is not built")
def test_no_kernel_of_runs_that_nothing_reaches():
    """32 row groups of 16 rows are all 512 rows of S that omni_decay_rec takes: no form by 32 columns holds 32 rows a thread.  16 groups need it."""
    code = open(B.LIB_DECODER, "rb").read()
    assert b"rec_run_kernelILi8ELi16E" in code and b"rec_run_kernelILi16ELi32E" in code
    assert b"rec_run_kernelILi8ELi32E" not in code


# (kernel, rows, tiles of a workgroup in o_proj, gate_up and the last stage, a workgroup may run gate_up without down_proj)
LAYER_LAUNCHES = [("wide", 16, 1, 3, 1, True), ("wide", 32, 1, 6, 2, False), ("wide", 64, 2, 12, 4, False), ("small", 16, 1, 2, 1, True),
                  ("small", 32, 1, 6, 2, True), ("small", 48, 1, 6, 4, False), ("small", 64, 1, 6, 4, False)]


@pytest.mark.parametrize("kernel,rows,o,gu,last,alone", LAYER_LAUNCHES)
def test_a_layer_launch_combines_over_nothing_that_is_still_read(tmp_path, kernel, rows, o, gu, last, alone):
    """LDS of the backbone's layer launches: the three areas of o_proj, gate_up and down_proj do not meet; the last stage's never meets down_proj's, and
    where a workgroup runs gate_up and no down_proj -- no barrier between -- it does not meet gate_up's."""
    src = tmp_path / "areas.cpp"
    src.write_text(f"""
#include "bb_areas.h"
constexpr BbAreas a = bb_areas_{kernel}({rows});
constexpr bool apart(int x, int nx, int y, int ny) {{ return x + bb_area(nx) <= y || y + bb_area(ny) <= x; }}
static_assert(apart(a.o, {o}, a.gate_up, {gu}) && apart(a.o, {o}, a.down, {o}) && apart(a.gate_up, {gu}, a.down, {o}), "three areas");
static_assert(apart(a.last, {last}, a.down, {o}), "the last stage over down_proj's");
static_assert({str(not alone).lower()} || apart(a.last, {last}, a.gate_up, {gu}), "the last stage over gate_up's");
static_assert(a.down + bb_area({o}) <= a.total && a.last + bb_area({last}) <= a.total && a.total * 4 <= 160 * 1024, "total");
""")
    subprocess.run(["g++", "-std=c++17", "-fsyntax-only", "-I", CSRC, str(src)], check=True, timeout=60)
