"""The bookkeeping of the matrix-core prefill launches without a GPU: ``research_amd/csrc/prefill_plan.h`` (the
header the host entry points and the kernels share) compiled with g++ into ``tests/host/prefill_plan_replay.cpp``.
The pieces a workgroup's tiles are cut into cover the tiles once; the groups that the workgroups of one (sequence,
kv head) run in turn cover the groups once and stay within what the launch was sized for; the split rule picks the
cheapest admissible split of its own cost model; the workspace size is the layout the kernels index."""

import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "host", "prefill_plan_replay.cpp")


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("pfplan") / "libprefill_plan_replay.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-o", lib, SRC], check=True)
    dll = ctypes.CDLL(lib)
    dll.pa_plan_pieces.argtypes = [ctypes.c_int] * 3 + [ctypes.c_char_p, ctypes.c_int]
    dll.pa_plan_groups.argtypes = [ctypes.c_int] * 3 + [ctypes.POINTER(ctypes.c_int), ctypes.c_char_p, ctypes.c_int]
    dll.pa_plan_splits.argtypes = [ctypes.c_longlong, ctypes.c_int, ctypes.c_longlong, ctypes.c_int, ctypes.c_longlong]
    dll.pa_plan_ragged_groups.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_int, ctypes.c_int] + [ctypes.c_longlong] * 4 + [ctypes.c_int] * 2
    dll.pa_plan_units.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_int, ctypes.c_longlong] + [ctypes.c_int] * 3
    dll.pa_plan_units.restype = ctypes.c_longlong
    dll.pa_plan_dense.argtypes = [ctypes.c_longlong, ctypes.c_longlong, ctypes.c_int]
    dll.pa_plan_cost.argtypes = [ctypes.c_longlong, ctypes.c_int, ctypes.c_longlong, ctypes.c_int]
    dll.pa_plan_cost.restype = ctypes.c_longlong
    dll.pa_plan_ws_bytes.argtypes = [ctypes.c_longlong, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    dll.pa_plan_ws_bytes.restype = ctypes.c_ulonglong
    dll.pa_plan_groups_per_workgroup.argtypes = [ctypes.c_int, ctypes.c_longlong, ctypes.c_int, ctypes.c_int]
    return dll


def _ok(rc, err):
    assert rc == 0, err.value.decode()


def test_pieces_cover_the_tiles_once(plan):
    err = ctypes.create_string_buffer(256)
    rng = np.random.default_rng(0)
    for n_all in list(range(0, 40)) + rng.integers(40, 6000, 200).tolist():
        for n_splits in range(1, 9):
            _ok(plan.pa_plan_pieces(int(rng.integers(0, 3000)), int(n_all), n_splits, err, 256), err)


def test_groups_of_a_sequence_are_each_run_once(plan):
    """As the host sizes the launch: gpw groups per workgroup, ceil(groups / gpw) workgroups along y."""
    err = ctypes.create_string_buffer(256)
    most = ctypes.c_int(0)
    for groups in range(1, 130):
        for gpw in range(1, 9):
            n_chunks = -(-groups // gpw)
            # a shorter sequence of the same launch has fewer groups than the launch was sized for
            for group_end in {groups, max(1, groups // 2), max(1, groups - 1), 1}:
                _ok(plan.pa_plan_groups(group_end, n_chunks, gpw, ctypes.byref(most), err, 256), err)
            _ok(plan.pa_plan_groups(groups, n_chunks, gpw, ctypes.byref(most), err, 256), err)
            assert most.value == -(-groups // n_chunks)


def test_zigzag_order_balances_causal_work(plan):
    """Group g of a dense causal prompt runs g + 1 tiles: with the groups dealt from the front in even rounds and
    from the back in odd ones the workgroups' tile counts differ by less than one round's spread."""
    groups, gpw = 64, 8
    n_chunks = groups // gpw
    totals = []
    for chunk in range(n_chunks):
        mine = [i * n_chunks + (n_chunks - 1 - chunk if i & 1 else chunk) for i in range(gpw)]
        totals.append(sum(g + 1 for g in mine))
    assert max(totals) - min(totals) == 0
    straight = [sum(i * n_chunks + chunk + 1 for i in range(gpw)) for chunk in range(n_chunks)]
    assert max(straight) - min(straight) == gpw * (n_chunks - 1)


class Launch:
    """What a launch of the kernels with the assembly loop is planned as on 256 compute units (``prefill_launch`` of ``prefill.hip``).
    ``rows``: of q, all prompts' (0: not known); ``keys``: that the block tables can describe."""

    def __init__(self, plan, hq, hkv, d, batch, most, rows, keys):
        self.plan, self.hkv, self.batch, self.rows, self.keys, self.n_rep = plan, hkv, batch, rows, keys, hq // hkv
        self.tasks, self.tile = (4, 32) if d > 128 else (8, 64)
        self.groups = -(-(-(-most // 32) * self.n_rep) // self.tasks)
        self.part_bytes = rows * hq * ((256 if d > 128 else 128 if d > 64 else 64 if d > 32 else 32) + 2) * 4
        self.gpw = 1
        if d <= 128:
            equal = plan.pa_plan_groups_per_workgroup(hkv, self.groups, batch, 256)
            self.gpw = plan.pa_plan_ragged_groups(equal, self.groups, hkv, batch, rows, most, 256 // self.n_rep, keys, 64, 256)

    def units(self, gpw=1):
        return self.plan.pa_plan_units(self.hkv, -(-self.groups // gpw), self.batch, self.rows, self.n_rep, 32, self.tasks * gpw)

    def splits(self):
        return self.plan.pa_plan_splits(self.units(), 256, self.keys, self.tile, self.part_bytes)

    def dense(self):
        return self.rows > 0 and bool(self.plan.pa_plan_dense(self.units(self.gpw), self.hkv * -(-self.groups // self.gpw) * self.batch, 256))


def unequal_prompts(n, most):
    """Rows of ``n`` prompts and the tokens before them: two have ``most`` rows, one has none, the others up to half as many."""
    rng = np.random.default_rng(n)
    chunk = rng.integers(0, most // 2 + 1, size=n)
    chunk[[1, n // 2, n - 1]] = most, 0, most
    return [int(x) for x in chunk], [int(x) for x in rng.integers(most, 2 * most, size=n)]


# (head size, query heads, kv heads, prompts, the longest's rows, groups of a workgroup): launches whose workgroups are numbered by the chunks that have
# rows (test_gpu_prefill_split.py runs them): more than 64 sequences, and workgroups of one group and of two
NUMBERED = [(128, 8, 2, 110, 130, 2), (64, 8, 2, 66, 260, 1), (256, 6, 3, 70, 80, 1), (128, 8, 2, 12, 1200, 1), (128, 12, 2, 110, 80, 2), (32, 8, 4, 40, 260, 2)]


@pytest.mark.parametrize("d,hq,hkv,n,most,gpw", NUMBERED)
def test_which_unequal_prompts_are_numbered_by_rows(plan, d, hq, hkv, n, most, gpw):
    chunk, prefix = unequal_prompts(n, most)
    keys = -(-max(c + p for c, p in zip(chunk, prefix)) // 16) * 16
    at = Launch(plan, hq, hkv, d, n, most, sum(chunk), keys)
    assert at.dense() and at.gpw == gpw
    assert not Launch(plan, hq, hkv, d, n, most, 0, keys).dense()  # (a call that does not know how many rows)


@pytest.mark.parametrize("cus", [256, 304, 64])
def test_split_rule_is_the_cheapest_admissible_split(plan, cus):
    rng = np.random.default_rng(cus)
    for i in range(800):
        workgroups = int(rng.integers(1, 4 * cus))
        max_keys = int(rng.integers(64, 400000 if i % 2 else 12800))
        part = int(rng.integers(0, 1 << 25))
        s = plan.pa_plan_splits(workgroups, cus, max_keys, 64, part)
        tiles = max_keys // 64
        assert 1 <= s <= 8
        if s > 1:
            assert tiles // s >= 8  # a piece keeps enough tiles to pay for its set-up
        cost = lambda k: plan.pa_plan_cost(workgroups, cus, tiles, k) + (9 + 2 * k * part // 4500000 if k > 1 else 0)  # (and the merge)
        admissible = [k for k in range(1, 9) if k == 1 or tiles // k >= 8]
        # (the rule stops at the first split that is too fine, so the admissible ones are 1 .. some k)
        assert admissible == list(range(1, len(admissible) + 1))
        assert cost(s) == min(cost(k) for k in admissible)
        assert all(cost(k) > cost(s) for k in admissible if k < s)  # the smaller on ties
    # launches that fill the device several times over stay whole
    assert plan.pa_plan_splits(64 * cus, cus, 1 << 20, 64, 64 * cus * 133120) == 1


def test_launches_and_their_pieces(plan):
    splits = lambda *a: Launch(plan, *a).splits()
    # the long-context shapes of bench.py, whose 64 and 128 workgroups leave compute units idle, and its batch of 32, which does not
    assert splits(8, 2, 128, 1, 2048, 2048, 202048) == 4
    assert splits(8, 2, 256, 1, 2048, 2048, 202048) == 2
    assert splits(32, 8, 128, 32, 256, 32 * 256, 2304) == 1 and splits(32, 8, 256, 32, 256, 32 * 256, 2304) == 1
    assert splits(8, 2, 128, 1, 150, 150, 1024) == 1       # 16 tiles: the merge costs what half of them do
    assert splits(8, 2, 128, 7, 248, 7 * 248, 4184) == 4   # few rows behind a long prefix: 56 workgroups
    assert splits(32, 8, 128, 64, 256, 64 * 256, 16384) == 1


@pytest.mark.parametrize("tasks", [8, 4])
def test_units_are_about_the_groups_with_rows(plan, tasks):
    """Between a group for every sequence and what the longest prompt's length would give all, and no further
    from the groups there are than the last task and group of each sequence, and the reserve of one in sixteen, can make it."""
    rng = np.random.default_rng(tasks)
    count = lambda n, n_rep: -(-(-(-n // 32) * n_rep) // tasks)
    for _ in range(400):
        n_rep, batch, most, hkv = int(rng.integers(1, 20)), int(rng.integers(1, 300)), int(rng.integers(1, 1500)), int(rng.integers(1, 9))
        lens = rng.integers(1, most + 1, size=batch)
        lens[0] = most
        upper, real = count(most, n_rep) * batch, sum(count(int(n), n_rep) for n in lens)
        got = plan.pa_plan_units(hkv, count(most, n_rep), batch, int(lens.sum()), n_rep, 32, tasks)
        assert got % hkv == 0 and hkv * batch <= got <= hkv * upper
        # (what a sequence's last task and last group lack lies between nothing and twice what is counted for them; floors and ceilings: 2)
        step = next(x for x in (8, 4, 2, 1) if x <= tasks and n_rep % x == 0)
        assert abs(got // hkv - real) <= batch * (n_rep + tasks - step) / (2 * tasks) + batch / 16 + 2


def test_workgroups_are_numbered_by_rows_where_that_is_a_round_less(plan):
    assert all(not plan.pa_plan_dense(u, u, 256) for u in (1, 160, 255, 256, 257, 512, 700))           # equal prompts: nothing to gain
    assert [plan.pa_plan_dense(u, 300, 256) for u in (159, 160, 256, 257)] == [0, 1, 1, 0]             # a round instead of two, well filled
    assert [plan.pa_plan_dense(u, 1152, 256) for u in (800, 927, 928, 1024, 1025)] == [0, 0, 1, 1, 0]  # 4 instead of 5
    assert [plan.pa_plan_dense(u, 1152, 256) for u in (256 + 159, 256 + 160)] == [0, 1]                # 2 instead of 5


def test_workspace_size_is_the_layout_the_kernels_index(plan):
    # part_o float[row][head][piece][D] + part_ml float[row][head][piece][2]
    for total_q, hq, d, s in [(2048, 8, 128, 4), (150, 8, 256, 2), (7, 3, 32, 8)]:
        assert plan.pa_plan_ws_bytes(total_q, hq, d, s) == total_q * hq * s * (d + 2) * 4
    assert plan.pa_plan_ws_bytes(2048, 8, 128, 1) == 0 and plan.pa_plan_ws_bytes(2048, 8, 128, 0) == 0


def test_groups_per_workgroup_leaves_a_workgroup_per_compute_unit(plan):
    rng = np.random.default_rng(3)
    for _ in range(500):
        hkv, groups, batch, cus = int(rng.integers(1, 17)), int(rng.integers(1, 200)), int(rng.integers(1, 300)), 256
        g = plan.pa_plan_groups_per_workgroup(hkv, groups, batch, cus)
        assert 1 <= g <= min(8, groups)
        fills = lambda k: hkv * -(-groups // k) * batch >= cus
        assert g == 1 or fills(g)
        assert all(not fills(k) for k in range(g + 1, min(8, groups) + 1))
    assert plan.pa_plan_groups_per_workgroup(8, 8, 64, 256) == 8    # dense 64 x 512
    assert plan.pa_plan_groups_per_workgroup(8, 4, 32, 256) == 4    # c3: all 4 groups of a (sequence, kv head)
    assert plan.pa_plan_groups_per_workgroup(2, 8, 1, 256) == 1     # one long chunk: nothing to spare
