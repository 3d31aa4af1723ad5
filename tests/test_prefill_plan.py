"""How prefill launches are cut (csrc/prefill_plan.h, no device code), by itself on the CPU, against the recorded times of
both forms and all numbers of parts."""
import math
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("plan") / "prefill_plan")
    subprocess.check_call(["g++", "-std=c++17", "-O2", "-Wall", "-Wextra", "-o", exe, os.path.join(HERE, "prefill_plan.cpp")])

    def run(sizes):
        """[(shape, rows, keys before, window)] -> ["<pairs>x<parts>"]"""
        lines = "".join("%d %d %d %s\n" % (before, rows, window, shape.replace("/", " ")) for shape, rows, before, window in sizes)
        out = subprocess.run([exe], input=lines, capture_output=True, text=True, timeout=60, check=True).stdout.splitlines()
        assert len(out) == len(sizes) and all(o.endswith(" 0") for o in out)
        return ["x".join(o.split()[:2]) for o in out]
    return run


def recorded():
    for line in open(os.path.join(HERE, "..", "profiles", "prefill_parts.txt")):
        if line.count("|") == 4 and line[0].isdigit():
            size, before, now, _, times = line.split("|")
            shape, *rest = size.split()
            yield (shape, *map(int, rest)), before.strip(), now.strip(), {k: float(v) for k, v in (t.split(":") for t in times.split())}


def test_what_is_picked_is_near_the_best_and_not_slower_than_before(plan):
    rows = list(recorded())
    assert len(rows) == 1199
    picks = plan([r[0] for r in rows])
    off, worse = {"64": [], "128": [], "256": []}, []
    for (size, before, now, us), pick in zip(rows, picks):
        assert pick == now, (size, pick, now)
        if pick in us:                                       # (numbers of parts between the recorded ones)
            off[size[0].split("/")[2]].append(us[pick] / min(us.values()))
            if us[pick] > 1.025 * us[before]:
                worse.append(size)
    for hd, ratios in off.items():
        assert len(ratios) >= 300 and sum(map(math.log, ratios)) / len(ratios) < 0.01 and max(ratios) < 1.25, hd
    # the two sizes that the rule's comment names
    assert worse == [("8/4/256", 33, 16000, 0), ("8/2/256", 2048, 100, 128)]


# blocks of unequal length in one to two rounds of workgroups, and two workgroups to a compute unit at head dim 64
@pytest.mark.parametrize("shape,rows,before,window", [("16/8/256", 1501, 0, 0), ("16/8/256", 1501, 200, 0), ("8/8/128", 3000, 0, 0), ("16/8/128", 1501, 0, 0),
                                                      ("16/16/64", 1501, 0, 0), ("16/16/64", 3000, 0, 0), ("32/8/64", 3000, 0, 512)])
def test_two_pairs_where_workgroups_are_more_than_units(plan, shape, rows, before, window):
    assert plan([(shape, rows, before, window)]) == ["2x1"]


# blocks of equal length: whole rounds
@pytest.mark.parametrize("shape,rows,before,window", [("16/8/256", 1501, 0, 512), ("16/8/128", 1501, 4000, 512), ("16/8/128", 3000, 0, 0), ("32/8/128", 2048, 0, 0)])
def test_four_pairs_where_a_second_round_would_be_whole(plan, shape, rows, before, window):
    assert plan([(shape, rows, before, window)]) == ["4x1"]


def test_any_sizes_are_cut(plan):
    # smallest and largest, windows longer than what there is, every group of heads
    plan([(shape, rows, before, window) for shape in ("1/1/64", "2/1/128", "4/1/256", "8/1/64", "64/64/128", "64/8/256")
          for rows in (1, 31, 32, 33, 4096, 131072) for before in (0, 1, 126975) if rows + before <= 131072
          for window in (0, 1, 31, 4096, 131072)])
