"""Register budget of the sweep kernels, read from the compiler's resource
report (hipcc -Rpass-analysis=kernel-resource-usage, device code only).

The sweeps are bound by VALU issue and latency; two allocation accidents cost
a third or more of a kernel's speed without changing a single result: a
private array the compiler cannot keep in registers (ScratchSize > 0, e.g. a
selection between two structs made through a pointer), and a body one
register over the 256 that two waves per SIMD allow (one wave per SIMD).
This pins both for the throughput kernels: no scratch anywhere, and at least
two waves per SIMD for the gamma = 5/3 Sod sweeps of both precisions and for
the batch kernels of the gamma = 5/3 and mixed forms.  Runs on the CPU
(cross-compilation only)."""
import os
import re
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

from hydropad_amd import build

FIELDS = {"VGPRs": "vgpr", "AGPRs": "agpr", "ScratchSize [bytes/lane]": "scratch", "Occupancy [waves/SIMD]": "waves"}


def resources(src):
    cmd = [build.hipcc()] + build.flags("fast") + ["-Rpass-analysis=kernel-resource-usage", "--cuda-device-only",
                                                  "-c", os.path.join(build.CSRC, src), "-o", os.devnull]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    out, cur = {}, None
    for line in r.stderr.splitlines():
        m = re.search(r"remark: Function Name: (\S+)", line)
        if m:
            cur = out.setdefault(m.group(1), {})
            continue
        m = re.search(r"remark:\s+([A-Za-z/\[\] ]+): (\d+)", line)
        if cur is not None and m and m.group(1).strip() in FIELDS:
            cur[FIELDS[m.group(1).strip()]] = int(m.group(2))
    return out


@pytest.fixture(scope="module")
def report():
    with ThreadPoolExecutor(2) as ex:
        fast, batch = ex.map(resources, ["hp_kernels_fast.hip", "hp_batch_kernels.hip"])
    return fast, batch


def test_no_kernel_uses_scratch(report):
    for rep in report:
        assert rep, "no resource remarks parsed"
        for name, r in rep.items():
            assert r.get("scratch", 0) == 0, (name, r)


def test_throughput_sweeps_keep_two_waves(report):
    fast, batch = report
    # FastMath53 sweeps without gravity, expansion terms or fused expansion
    sod = [n for n in fast if "FastMath53" in n and re.search(r"E[df](Li[23]E)?Lb0ELb0ELb0E", n)]
    assert len(sod) == 6, sod
    held = [n for n in batch if "batch_" in n and ("FastMath53" in n or re.search(r"FastMathEf", n))]
    assert len(held) == 18, held
    for n in sod + held:
        assert batch.get(n, fast.get(n))["waves"] >= 2, (n, batch.get(n, fast.get(n)))


FIELDS["LDS Size [bytes/block]"] = "lds"
LDS_PER_CU = 160 << 10


def test_stream_window_is_sized_by_the_block(report):
    """The y/z sweeps' LDS window is asked for at launch, for the threads a
    block has (hp_set_tiling's block): reserved for 256 threads whatever the
    block, a 64-thread block's single wave held 53 KB and a CU three of them."""
    sweeps = {n: r for n, r in report[0].items() if "sweep_stream" in n}
    assert len(sweeps) == 48
    for name, r in sweeps.items():
        assert r["lds"] < 1024, (name, r)


CLAIMS = """
#include <cstdio>
#include "hp_tiling.h"
int main()
{
    for (int g53 = 0; g53 < 2; ++g53)
        for (int x = 0; x < 2; ++x)
            std::printf("%d %d %d %d\\n", g53, x, hp::stream_waves(g53, x), hp::batch_x_waves(g53, x));
}
"""


def test_kernels_hold_the_waves_their_launches_fill(report, tmp_path):
    """The segment length of a y/z sweep and the batch's grids are sized to the
    waves per SIMD that hp_tiling.h states: each kernel holds exactly those, by
    its registers and, for the y/z sweeps, by the LDS of its window (26
    doubles a thread, 30 with gravity, in blocks of 256)."""
    (tmp_path / "claims.cpp").write_text(CLAIMS)
    exe = str(tmp_path / "claims")
    subprocess.run(["g++", "-std=c++17", "-I", build.CSRC, str(tmp_path / "claims.cpp"), "-o", exe], check=True)
    stream, batch_x = {}, {}
    for line in subprocess.run([exe], capture_output=True, text=True, check=True).stdout.split("\n")[:-1]:
        g53, x, s, b = map(int, line.split())
        stream[g53, x], batch_x[g53, x] = s, b
    checked = 0
    for rep in report:
        for name, r in rep.items():
            g53 = "FastMath53" in name
            form = re.search(r"FastMath(?:53)?E([df])(?:Li[23]E)?Lb([01])E", name)
            if "stream" in name:
                grav = "sweep_stream" in name and form.group(2) == "1"
                lds = max(r["lds"], (30 if grav else 26) * 8 * 256 + (r["lds"] if "sweep_stream" in name else 0))
                assert min(r["waves"], LDS_PER_CU // lds) == stream[g53, grav], (name, r)
            elif "batch_x" in name:
                assert r["waves"] == batch_x[g53, form.group(1) == "f"], (name, r)
            else:
                continue
            checked += 1
    assert checked == 48 + 16 + 8
