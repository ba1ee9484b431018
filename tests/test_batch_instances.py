"""The kernel instance that runs a group of the batched solve (no GPU needed):
a group of few k must not reserve the LDS of waves it does not launch, nor run
the instance whose register budget spills."""
import os
import re
import subprocess

import pytest

from test_device_code import LLVM, _code_objects

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SIMT = os.path.join(ROOT, "tests", "simt")
CU_LDS = 160 * 1024
CU_SIMDS = 4


@pytest.fixture(scope="module")
def rule():
    """{(slots, batch): (waves launched, waves of the instance, its LDS bytes)}"""
    r = subprocess.run(["make", "-C", SIMT, "simt_batch"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-3000:] + r.stderr[-3000:]
    out = subprocess.run([os.path.join(SIMT, "simt_batch"), "rule"], check=True, capture_output=True, text=True).stdout
    rows = [tuple(map(int, ln.split())) for ln in out.splitlines()]
    return {row[:2]: row[2:] for row in rows}


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{(slots, waves): (LDS bytes, scratch bytes per lane)} of the built batched kernels"""
    got = {}
    for co in _code_objects(tmp_path_factory.mktemp("co")):
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", str(co)], check=True,
                               capture_output=True, text=True).stdout
        for k in re.split(r"\n  - \.a", notes)[1:]:
            m = re.search(r"\.name:\s+\S*deb_forward_batched_kernelILi(\d+)ELi(\d+)E", k)
            if m:
                size = [int(re.search(rf"\.{f}_segment_fixed_size:\s+(\d+)", k).group(1)) for f in ("group", "private")]
                got[int(m.group(1)), int(m.group(2))] = tuple(size)
    assert got, "no batched kernel in the library"
    return got


@pytest.mark.parametrize("slots", range(1, 7))
def test_small_groups_share_a_cu(rule, slots):
    """Groups of up to four waves: the LDS of a CU holds as many as its SIMDs take at one wave each, and from two
    slots on they run an instance with the registers of one wave per SIMD."""
    for batch in range(1, 65):
        waves, inst, lds = rule[slots, batch]
        assert 1 <= waves <= min(batch, inst)
        if waves <= CU_SIMDS:
            assert (CU_SIMDS // waves) * lds <= CU_LDS, (batch, waves, inst, lds)
            assert inst <= CU_SIMDS or slots == 1, (batch, waves, inst)
        assert lds <= CU_LDS


@pytest.mark.parametrize("slots", range(1, 7))
def test_instances_are_built_as_the_rule_counts(rule, kernels, slots):
    """Every instance that the rule picks is in the library with the LDS it counts, and up to two slots those of at
    most four waves keep their state out of scratch memory."""
    for batch in range(1, 65):
        waves, inst, lds = rule[slots, batch]
        assert kernels[slots, inst][0] == lds, (batch, inst)
        if slots <= 2 and inst <= CU_SIMDS:
            assert kernels[slots, inst][1] == 0, (batch, inst)
