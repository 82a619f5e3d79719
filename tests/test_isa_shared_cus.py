"""What a default launch of each persistent kernel takes of a compute unit.

A persistent launch waits for all of its workgroups, so two of them on one GPU both
end only if every workgroup of both finds room.  Launches that ran beside each other,
or beside the default serving loop (one workgroup per CU), keep doing so: a default
launch takes at most what that loop leaves of a CU's registers, which is also no more
than half of them, and at most half of its LDS."""
import os
import re

import pytest

from test_isa_barrier_loops import _HAVE_HIPCC, _compile, kernel_registers

CSRC = os.path.join("csrc")
VGPRS, LDS = 512, 160 * 1024  # per SIMD and lane, per CU

# kernel (a pattern of its symbol) -> file, threads of a workgroup, workgroups per CU
DEFAULT = {
    r"5k_bfsI": ("graph", 512, 1),
    r"6k_ssspI": ("graph", 512, 1),
    r"10k_pagerankILi\dELi3E": ("graph", 256, 3),
    r"10k_pagerankILi\dELi1E": ("graph", 256, 4),
    r"10k_scan_u32I": ("scan", 512, 1),
    # no workgroup of these waits for one that has not started: one has to find room
    r"12k_scan_batchI": ("batch", 512, 1),
    r"14k_reduce_batch": ("batch", 256, 1),
}

# the 64-source SSSP by kind: workgroups per CU, and the registers that these launches
# leave to others (what 4 workgroups of 113 and of 104 registers left)
MSSP = {r"6k_msspILi2E": (6, 480), r"6k_msspILi[013-7]E": (5, 416)}


def _granule(v):
    return -(-v // 8) * 8


def kernel_lds(asm):
    """Map kernel symbol -> LDS bytes."""
    out, fn = {}, None
    for line in asm.splitlines():
        m = re.match(r"^\s*\.amdhsa_kernel (\S+)", line)
        if m:
            fn = m.group(1)
        m = re.match(r"^\s*\.amdhsa_group_segment_fixed_size (\d+)", line)
        if m and fn:
            out[fn] = int(m.group(1))
    return out


@pytest.fixture(scope="module")
def asm():
    from concurrent.futures import ThreadPoolExecutor
    names = sorted({"serve"} | {f for f, _, _ in DEFAULT.values()} | {"mssp"})
    with ThreadPoolExecutor(max_workers=4) as ex:
        return dict(zip(names, ex.map(lambda n: _compile(os.path.join(CSRC, n + ".hip")), names)))


@pytest.mark.skipif(not _HAVE_HIPCC, reason="hipcc absent")
def test_default_launches_leave_room_for_another(asm):
    loop = [v for k, v in kernel_registers(asm["serve"]).items() if "k_serve" in k]
    assert len(loop) == 1
    left = VGPRS - _granule(loop[0][1])
    assert left >= VGPRS // 2
    for pattern, (name, threads, per_cu) in DEFAULT.items():
        regs, lds = kernel_registers(asm[name]), kernel_lds(asm[name])
        hits = [k for k in regs if re.search(pattern, k)]
        assert hits, pattern
        for k in hits:
            took = per_cu * threads // 256 * _granule(regs[k][1])
            assert took <= VGPRS // 2, (k, took)
            assert per_cu * lds[k] <= LDS // 2, (k, lds[k])


@pytest.mark.skipif(not _HAVE_HIPCC, reason="hipcc absent")
def test_mssp_leaves_what_it_left(asm):
    regs, lds = kernel_registers(asm["mssp"]), kernel_lds(asm["mssp"])
    for pattern, (per_cu, most) in MSSP.items():
        hits = [k for k in regs if re.search(pattern, k)]
        assert hits, pattern
        for k in hits:
            assert per_cu * _granule(regs[k][1]) <= most, (k, regs[k])
            assert per_cu * lds[k] <= LDS
