"""The geometry search of the persistent recurrences (haste_hip_plan_tiles), swept on the host
over hidden sizes, batch sizes and device shapes: whatever it finds must be a geometry the
kernels can run."""
import ctypes

import pytest

from haste_amd import lib as hlib

DEVICES = [(256, 8), (256, 0), (128, 4), (304, 8), (64, 1)]
BATCHES = [1, 3, 4, 8, 9, 16, 31, 32, 64, 100, 128, 200, 256, 512]


def _plan(lib, cus, xcds, gates, N, H):
    out = (ctypes.c_int * 16)()
    rc = lib.haste_hip_plan_tiles(cus, xcds, gates, N, H, out)
    assert rc == 0
    return list(out[:8]), list(out[8:])


@pytest.mark.parametrize("cus,xcds", DEVICES)
@pytest.mark.parametrize("gates", [3, 4])
def test_every_geometry_found_is_one_the_kernels_can_run(cus, xcds, gates):
    lib = hlib.load()
    lib.haste_hip_plan_tiles.restype = ctypes.c_int
    sizes = list(range(16, 4097, 16)) + [1, 5, 37, 100, 300, 500, 1001, 1300, 2049]
    resident = 0
    for H in sizes:
        for N in BATCHES:
            for which, plan in zip(("forward", "backward"), _plan(lib, cus, xcds, gates, N, H)):
                found, nb, hs, ct, gx, gy, reg, groups = plan
                where = (which, cus, xcds, gates, N, H, plan)
                if not found:
                    assert plan == [0] * 8, where
                    continue
                assert nb in (4, 8, 16, 32, 64), where
                if which == "forward":  # the gate columns of the workgroup's units fit its slice
                    assert hs in (4, 8, 16) and gates * hs <= 16 * ct, where
                assert gx == -(-H // hs) and gy == -(-N // nb), where
                # one workgroup per CU, all on the chip at once
                assert gx * gy <= cus, where
                # part of the slice in registers: tall tiles only, whole batches of 8 groups, and
                # some of the slice stays in LDS
                if reg:
                    resident += 1
                    assert nb >= 16 and reg % 8 == 0 and 0 < reg < groups, where
    if cus >= 256:
        assert resident > 0  # the sweep reaches the register-resident range


def test_plan_tiles_refuses_bad_arguments():
    lib = hlib.load()
    lib.haste_hip_plan_tiles.restype = ctypes.c_int
    out = (ctypes.c_int * 16)()
    assert lib.haste_hip_plan_tiles(256, 8, 5, 4, 64, out) != 0
    assert lib.haste_hip_plan_tiles(256, 8, 4, 0, 64, out) != 0
    assert lib.haste_hip_plan_tiles(256, 8, 4, 4, 64, None) != 0
    assert lib.haste_hip_plan_tiles(0, 8, 4, 4, 64, out) != 0


def test_plan_recurrence_refuses_bad_arguments():
    lib = hlib.load()
    good = (256, 8, 4, 4, 0, 30, 64, 512, 512)
    assert _plan_pass(lib, *good)[0] == 0
    for at, value in [(0, -1), (0, 0), (2, 5), (2, 2), (3, 2), (5, 0), (6, 0), (7, 0), (8, -3)]:
        bad = list(good)
        bad[at] = value
        assert _plan_pass(lib, *bad)[0] != 0, bad
    assert _plan_pass(lib, *good, workspace=64)[0] != 0
    assert lib.haste_hip_plan_recurrence(*good, ctypes.c_size_t(0), None) != 0


PASSES = [(gates, size, backward) for gates in (3, 4) for size in (4, 8) for backward in (0, 1)]


def _plan_pass(lib, cus, xcds, gates, size, backward, T, N, C, H, workspace=0):
    out = (ctypes.c_int * 8)()
    rc = lib.haste_hip_plan_recurrence(cus, xcds, gates, size, backward, T, N, C, H, ctypes.c_size_t(workspace), out)
    return rc, list(out)


@pytest.mark.parametrize("cus,xcds", DEVICES + [(128, 0), (64, 2), (32, 1)])
@pytest.mark.parametrize("gates,size,backward", PASSES)
def test_every_pass_has_a_kernel(cus, xcds, gates, size, backward):
    """Whatever is chosen for a pass can be launched, on every device shape: with XCDs, without (the placement could not
    be looked at, was switched off or turned out wrong) and with fewer of them."""
    lib = hlib.load()
    sizes = sorted(set(list(range(16, 1025, 16)) + [1, 5, 37, 100, 129, 257, 300, 321, 385, 500, 511, 770, 777, 800, 816, 1100, 2048, 4096]))
    batches = sorted(set(BATCHES + list(range(1, 130, 4)) + [33, 40, 65, 72, 80]))
    kernels = set()
    for H in sizes:
        for N in batches:
            for T in (2, 30):
                rc, plan = _plan_pass(lib, cus, xcds, gates, size, backward, T, N, 18, H)
                assert rc == 0, (cus, xcds, gates, size, backward, T, N, H, rc)
                kernels.add(plan[0])
                if plan[0] > 1:
                    assert plan[3] * plan[4] <= cus and plan[1] * plan[2] * plan[4] >= N
    every = {0, 4} if size == 8 else {0, 2, 3}
    assert kernels == every if (cus, xcds) == (256, 8) else kernels <= every if xcds else kernels <= every - {3}


@pytest.mark.parametrize("gates", [3, 4])
def test_single_steps(gates):
    """One kernel for a step of up to 8 rows of any size, and of more rows up to a size that depends on what else there
    is; a workspace too small for its sums leaves larger batches what they ran on before."""
    lib = hlib.load()
    for N, C, H, single in [(1, 512, 512, 1), (8, 64, 4096, 1), (9, 512, 512, 1), (128, 512, 512, 1), (64, 64, 2048, 1),
                            (16, 512, 4096, 0), (128, 64, 3000, 0), (1024, 512, 512, 0),
                            # beyond what stays on chip: as long as there is no more than a tile per CU, and few blocks
                            (16, 64, 2560, 0), (96, 64, 1280, 1), (112, 64, 1152, 0), (80, 64, 1536, 0),
                            (160, 512, 1024, 1)]:
        rc, plan = _plan_pass(lib, 256, 8, gates, 4, 0, 1, N, C, H)
        assert rc == 0 and (plan[0] == 1) == bool(single), (N, C, H, rc, plan)
    # the sums of a step of 64 rows take 2 MiB; its all-steps kernel asks for less
    rc, plan = _plan_pass(lib, 256, 8, gates, 4, 0, 1, 64, 16, 512, workspace=(2 << 20) - 4096)
    assert rc == 0 and plan[0] > 1, (rc, plan)
    rc, plan = _plan_pass(lib, 256, 8, gates, 4, 0, 1, 8, 512, 512, workspace=100 << 10)
    assert rc == 0 and plan[0] == 1, (rc, plan)


def test_double_groups_of_8_rows_have_an_xcd_each():
    """Groups of 8 rows rather than 16 pay where a group's workgroups share an XCD: with XCDs, as far as there are, and not
    without."""
    lib = hlib.load()
    for gates in (3, 4):
        for N, H in [(64, 512), (40, 256), (8, 64)]:
            for backward in (0, 1):
                rows = {}
                for cus, xcds in [(256, 8), (256, 0), (128, 4), (256, 16)]:
                    rc, plan = _plan_pass(lib, cus, xcds, gates, 8, backward, 30, N, 18, H)
                    assert rc == 0
                    rows[cus, xcds] = (plan[1], plan[5])
                assert rows[256, 8] == (8, 1), (gates, N, H, backward)
                assert rows[256, 0] == (16, 0), (gates, N, H, backward)
                # four XCDs of 32 CUs: four groups
                assert rows[128, 4] == ((8, 1) if N <= 32 else (16, 1 if N <= 64 and H <= 512 else 0)), (gates, N, H, backward)
                # sixteen XCDs of 16 CUs: 256 units
                assert (rows[256, 16][0] == 8) == (H <= 256), (gates, N, H, backward)


@pytest.mark.parametrize("gates,size,backward", PASSES)
def test_a_workspace_of_the_stated_size_decides_nothing(gates, size, backward):
    """A pass that was lent haste_hip_workspace_bytes(), or what a rehearsal asked for, runs what it runs with a workspace
    that grows; one with less than it needs is refused or runs what needs less."""
    lib = hlib.load()
    lib.haste_hip_workspace_bytes.restype = ctypes.c_size_t
    fewer = 0
    for T in (1, 2, 30, 300):
        for N in BATCHES + [20, 48, 96]:
            for C, H in [(1, 1), (64, 128), (18, 257), (512, 300), (512, 512), (75, 512), (33, 800), (512, 1024), (2048, 1536)]:
                where = (gates, size, backward, T, N, C, H)
                own = _plan_pass(lib, 256, 8, gates, size, backward, T, N, C, H)
                assert own[0] == 0, where
                stated = lib.haste_hip_workspace_bytes(T, N, C, H)
                assert own[1][6] * 1024 <= stated + 1024, where
                for lent in (stated, own[1][6] * 1024):
                    rc, plan = _plan_pass(lib, 256, 8, gates, size, backward, T, N, C, H, lent)
                    assert rc == 0 and plan[:6] == own[1][:6], (where, lent)
                rc, plan = _plan_pass(lib, 256, 8, gates, size, backward, T, N, C, H, own[1][6] * 512)
                fewer += rc != 0 or plan[:6] != own[1][:6]
    assert fewer > 0


def test_the_tests_of_the_split_recurrences_reach_them():
    """The shapes that tests/test_gpu_split_recurrence.py means to run on the bf16 matrix cores do, on eight XCDs of 32 CUs."""
    import test_gpu_split_recurrence as t
    lib = hlib.load()

    def kernel(gates, backward, T, N, H, C):
        rc, plan = _plan_pass(lib, 256, 8, gates, 4, backward, T, N, C, H)
        assert rc == 0
        return plan[0], plan[1]
    heights = set()
    for gates in (3, 4):
        for backward, shapes, C in ((0, t.FORWARD, 18), (0, t.EXTREME_FORWARD, 13), (1, t.BACKWARD, 12), (1, t.EXTREME_BACKWARD, 8),
                                    (0, [(100, N, 512) for _, N in t.FP32_ERRORS], 512),
                                    (1, [(100, N, 512) for _, N in t.FP32_ERRORS], 512)):
            for T, N, H in shapes:
                which, rows = kernel(gates, backward, T, N, H, C)
                assert which == 3, (gates, backward, T, N, H)
                heights.add((gates, backward, shapes is t.EXTREME_FORWARD or shapes is t.EXTREME_BACKWARD, rows))
        for T, N, H in t.BESIDE_BACKWARD + t.EXTREME_BESIDE_BACKWARD:
            assert kernel(gates, 1, T, N, H, 12)[0] == 2, (gates, T, N, H)
    # every tile height, ordinary values and extreme ones
    assert heights == {(gates, backward, extreme, rows) for gates in (3, 4) for extreme in (False, True)
                       for backward, rows in ((0, 4), (0, 8), (0, 16), (1, 8), (1, 16))}


def test_the_tests_of_the_cut_recurrences_reach_them():
    """The shapes that tests/test_gpu_cut_recurrence.py means to run on groups of several XCDs do, on eight XCDs of 32 CUs, where a
    pass has enough steps; every number of XCDs per group and of batch tiles is among them."""
    import test_gpu_cut_recurrence as t
    lib = hlib.load()
    seen = set()
    for gates in (3, 4):
        for backward in (0, 1):
            for T, N, H in t.SHAPES + t.EXTREME + [t.MANY_NANS, (5, 50, 700), (5, 20, 1300), (4, 40, 1300)]:
                rc, plan = _plan_pass(lib, 256, 8, gates, 4, backward, T, N, 12, H)
                assert rc == 0 and plan[0] == 3 and plan[3] > 32, (gates, backward, T, N, H, plan)
                seen.add((backward, plan[3] // 32, min(plan[2], 3)))
                rc, few = _plan_pass(lib, 256, 8, gates, 4, backward, 3, N, 12, H)
                assert rc == 0 and few[0] != 3, (gates, backward, N, H)
    assert {(b, xcds) for b, xcds, _ in seen} == {(b, xcds) for b in (0, 1) for xcds in (2, 4, 8)}
    assert {(b, tiles) for b, _, tiles in seen} == {(b, tiles) for b in (0, 1) for tiles in (1, 2, 3)}


@pytest.mark.parametrize("gates,backward,N,H,cut", [
    (4, 0, 128, 544, 1), (4, 0, 64, 544, 0), (4, 0, 40, 672, 1), (4, 0, 28, 1024, 0), (4, 0, 160, 2048, 1),
    (3, 0, 28, 800, 1), (3, 0, 72, 736, 0), (3, 0, 144, 800, 0), (3, 0, 40, 1056, 0), (3, 0, 52, 1056, 1), (3, 0, 160, 1536, 1),
    (4, 1, 96, 544, 0), (4, 1, 72, 640, 0), (4, 1, 72, 624, 1), (4, 1, 160, 848, 1), (4, 1, 160, 2048, 1),
    (3, 1, 144, 528, 0), (3, 1, 80, 672, 0), (3, 1, 48, 1056, 0), (3, 1, 40, 1312, 1)])
def test_where_the_cut_recurrences_are_taken(gates, backward, N, H, cut):
    """Where the batch tiles of the other kernels have many rows for every batch tile a group goes through, as measured."""
    rc, plan = _plan_pass(hlib.load(), 256, 8, gates, 4, backward, 60, N, 64, H)
    assert rc == 0 and (plan[0] == 3 and plan[3] > 32) == bool(cut), plan


def test_workspace_bytes_of_the_cut_recurrences():
    """Nothing else is in use beside them, and calls of more rows never take them: they do not add to the bound, and a buffer
    of its size is enough for them."""
    lib = hlib.load()
    lib.haste_hip_workspace_bytes.restype = ctypes.c_size_t
    assert lib.haste_hip_workspace_bytes(50, 64, 512, 2048) < 380 << 20
    assert lib.haste_hip_workspace_bytes(4, 200, 64, 2048) < 440 << 20
    for gates in (3, 4):
        for backward in (0, 1):
            for N, H in [(1, 1024), (64, 2048), (160, 1408), (160, 2048), (20, 736)]:
                rc, plan = _plan_pass(lib, 256, 8, gates, 4, backward, 60, N, 64, H)
                lent = lib.haste_hip_workspace_bytes(60, N, 64, H)
                assert rc == 0 and _plan_pass(lib, 256, 8, gates, 4, backward, 60, N, 64, H, lent)[1][:6] == plan[:6]
