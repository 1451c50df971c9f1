"""Register and private-memory budgets of the hot kernels (compiler remarks
of the gfx950 build; no GPU).  A kernel whose arguments or registers fall back
to private memory runs several times slower, so the budgets are checked here."""
import re
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def resource_usage(tmp_path):
    sys.path.insert(0, str(ROOT / "trixilw.jl_amd"))
    import build

    out = tmp_path / "probe.so"
    cmd = [build.hipcc(), *build.HIPCC_FLAGS, "-Rpass-analysis=kernel-resource-usage", "-o", str(out),
           str(build.CSRC / "tlw_capi.hip")]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    usage, cur = {}, None
    for ln in r.stderr.splitlines():
        m = re.search(r"remark:\s+(Function Name|ScratchSize \[bytes/lane\]|Occupancy \[waves/SIMD\]): (\S+)", ln)
        if not m:
            continue
        if m.group(1) == "Function Name":
            cur = m.group(2)
            usage[cur] = {}
        else:
            usage[cur][m.group(1).split()[0]] = int(m.group(2))
    return usage


@pytest.fixture(scope="module")
def usage(tmp_path_factory):
    return resource_usage(tmp_path_factory.mktemp("res"))


def test_hot_kernels_stay_out_of_private_memory(usage):
    vol = {k: v for k, v in usage.items() if "k_volume" in k}
    surf = {k: v for k, v in usage.items() if "k_surface" in k}
    assert vol and surf
    for name, u in surf.items():
        assert u["ScratchSize"] == 0, (name, u)
    for name, u in vol.items():
        # a few spilled registers at most: the curvilinear N=4 kernels without shock capturing
        # spill 12 to 24 B, the 15-element N=4 kernel 12 B, the others nothing
        spills = re.match(r"_ZN3tlw8k_volumeILi4ELi\d+ELi\dELb0ELb[01]ELb1E", name) or "ILi4ELi15ELi0ELb0ELb0ELb0E" in name
        assert u["ScratchSize"] <= (24 if spills else 0), (name, u)
        # the Navier-Stokes LW, MDRK stage-2 and adaptive wall kernels (KIND 4, 9 and 10)
        # run at one wave per SIMD by design, their wall terms in accumulation
        # registers: no private memory at all
        wall = re.match(r"_ZN3tlw8k_volumeILi\dELi\d+ELi(4|9|10)E", name) is not None
        if wall:
            assert u["ScratchSize"] == 0 and u["Occupancy"] >= 1, (name, u)
        else:
            assert u["Occupancy"] >= 2, (name, u)


def test_adjoint_kernels_stay_out_of_private_memory(usage):
    adj = {k: v for k, v in usage.items() if re.match(r"_ZN3tlw\d+k_adj", k)}
    # LW, MDRK and shock-capturing steps, each with its face records, at both degrees
    assert len(adj) == 2 * (2 + 4 + 2), sorted(adj)
    for name, u in adj.items():
        # the N=4 LW kernel holds the derivatives of four Taylor levels and spills 84 B
        lw4 = re.match(r"_ZN3tlw9k_adjointILi4E", name) is not None
        assert u["ScratchSize"] <= (84 if lw4 else 0), (name, u)
