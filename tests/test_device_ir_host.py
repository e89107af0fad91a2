"""What the device code tells the compiler, read from the LLVM IR that hipcc
makes of it before any optimisation (about a second a file, no GPU)."""
import os
import re
import subprocess

import pytest

from vissatsatellitestereo_amd import build


@pytest.fixture(scope="module")
def pm_ir(tmp_path_factory):
    """Functions of vsm_pm.hip as {mangled name: [lines, the head first]}."""
    try:
        cc = build.hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    out = tmp_path_factory.mktemp("ir") / "pm.ll"
    cmd = [cc] + build.flags("gfx950") + ["--offload-device-only", "-S", "-emit-llvm", "-fno-discard-value-names",
                                          "-Xclang", "-disable-llvm-passes",
                                          os.path.join(build.CSRC, "vsm_pm.hip"), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True, text=True)
    funcs, cur = {}, None
    for line in out.read_text().splitlines():
        m = re.match(r"define .*@([\w.$]+)\(", line)
        if m:
            cur = funcs.setdefault(m.group(1), [])
        if cur is not None:
            cur.append(line)
        if line == "}":
            cur = None
    return funcs


def _find(lines, pattern):
    return [i for i, line in enumerate(lines) if re.search(pattern, line)]


def test_lanes_exchange_units_in_order(pm_ir):
    """A lane reads the unit that another lane of its wave wrote into the LDS
    row its own draw count was read from: the writes and the reads are ordered
    for the compiler (release, wave barrier, acquire), and so are the reads of
    the counts and the weights' writes before them."""
    order = [f for f in pm_ir if "wave_lds_order" in f]
    assert len(order) == 1
    body = pm_ir[order[0]]
    steps = [_find(body, p) for p in (r'fence syncscope\("wavefront"\) release', r"@llvm\.amdgcn\.wave\.barrier",
                                      r'fence syncscope\("wavefront"\) acquire')]
    assert all(len(s) == 1 for s in steps) and steps[0] < steps[1] < steps[2]
    tiles = [f for f in pm_ir if "13halfstep_tile" in f]
    assert len(tiles) >= 8
    for f in tiles:
        lines = pm_ir[f]
        (made,) = _find(lines, r"store ptr .*, ptr %slot\.ascast")
        (got,) = _find(lines, r"store i32 .*, ptr %got\.ascast")
        uses = [i for i in _find(lines, r"load ptr, ptr %slot\.ascast") if i < got]
        writes, read = uses[:-1], uses[-1]
        assert writes and read < got
        calls = _find(lines, rf"call .*@{order[0]}\(")
        assert any(made < i < writes[0] for i in calls), f
        assert any(writes[-1] < i < read for i in calls), f


def test_half_step_writes_no_descriptor(pm_ir):
    """k_halfstep promises that nothing writes the view descriptors while it
    runs (noalias, read only), so no pointer through which it could write one
    is among its arguments: the half-step counters are an array of ints."""
    kernels = [f for f in pm_ir if "10k_halfstep" in f]
    assert len(kernels) >= 8
    for f in kernels:
        head = pm_ir[f][0]
        assert re.search(r"noalias \S* ?%views", head), head
        args = subprocess.run(["c++filt", f], check=True, capture_output=True, text=True).stdout.strip()
        args = args[args.index("(") + 1:].split(", ")
        assert "vsm::ViewDesc const*" in args and "vsm::ViewDesc*" not in args, args
