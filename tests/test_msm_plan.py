"""The MSM sizing arithmetic the device buffers are allocated from
(nkr-zkp_amd/csrc/msm_plan.h), compiled for the CPU: window choice, the lane
rule, the bounds of a batch's partial sums and folds against the numbering the
planning kernel uses, and the schedules' buffers; schedules with zero entries
included, and a zero divisor must raise an error instead of ending the process
(SIGFPE)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def plan_bin(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("needs g++")
    out = str(tmp_path_factory.mktemp("plan") / "msm_plan_check")
    subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", "-Werror", "-I" + os.path.join(ROOT, "nkr-zkp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "msm_plan_check.cpp"), "-o", out], check=True)
    return out


def ask(binary, lines):
    res = subprocess.run([binary], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True)
    return res.stdout.strip().splitlines()


def test_window_choice_covers_the_scalar(plan_bin):
    ns = sorted({1, 2, 3, 5, 7, 100, 1000, 4097} | {1 << k for k in range(0, 25)} | {(1 << k) + 1 for k in range(1, 24)})
    out = ask(plan_bin, [f"plan {n} 0" for n in ns])
    for n, line in zip(ns, out):
        c, W, B = map(int, line.split())
        assert 4 <= c <= 16 and B == 1 << (c - 1)
        assert c * W >= 255 and c * (W - 1) < 255          # W signed digits cover 255 bits, none wasted
        assert 254 - c * (W - 1) >= 4 or c in (4, 16)        # the top window keeps at least 4 bits
        if n >= 1 << 20:
            assert c == 16


def test_default_target_is_the_groups_own_rule(plan_bin):
    """The lane setting's default, 19, gives each group its measured rule, so
    that setting it back restores the default; any other value is 2^value
    lanes whatever the number of entries."""
    own = [line.split() for line in ask(plan_bin, ["lanes 0 19", "lanes 1 19"])]
    assert own == ["65536 131072 262144 393216 4194304 16777216 33554432".split(),
                   "65536 65536 131072 262144 524288 2097152 8388608".split()]
    for target in (10, 12, 18, 20, 22, 24):
        for line in ask(plan_bin, [f"lanes 0 {target}", f"lanes 1 {target}"]):
            assert line.split()[:4] == [str(1 << target)] * 4


def test_a_minimum_binds_its_own_job_only(plan_bin):
    """Entries per lane of a launch, and of a job with a minimum (the witness
    MSMs may have one, H, in the same launch, has none); never 0."""
    rng = np.random.default_rng(3)
    entries = [0, 1, 65535, 65536, 65537, (1 << 22) - 1, 1 << 22, 1 << 24, (1 << 25) - 1, 1 << 25, 1 << 34]
    entries += [int(e) for e in 2 ** rng.uniform(0, 33, 20)]
    lanes = {0: [(1 << 22, 1), (1 << 24, 2), (1 << 25, 4), (1 << 60, 6)],
             1: [(1 << 21, 1), (1 << 23, 2), (1 << 60, 4)]}
    for g2 in (0, 1):
        for minimum in (1, 64):
            got = list(map(int, ask(plan_bin, [f"piece {g2} 19 {minimum} " + " ".join(map(str, entries))])[0].split()))
            for e, launch, job in zip(entries, got[::2], got[1::2]):
                n = 65536 * next(k for below, k in lanes[g2] if e < below)
                assert launch == max(1, -(-e // n)) and job == max(launch, minimum), (g2, minimum, e)


def test_b_query_plan(plan_bin):
    """bs1 and bs2 use the witness's plan while more than three quarters of the
    columns are finite, else their own width for what is left, whatever width
    the witness was given."""
    n = 1 << 17
    out = ask(plan_bin, [f"bplan {n} {c} {f}" for c in (0, 13) for f in (n, n - n // 4 + 1, n - n // 4, 1300, 1, 0)]
              + [f"plan {k} 0" for k in (n, n - n // 4, 1300, 1)])
    own = [int(line.split()[0]) for line in out[12:]]
    for c, got in ((own[0], out[:6]), (13, out[6:12])):
        assert [tuple(map(int, g.split())) for g in got] == \
            [(n, c), (n, c), (n - n // 4, own[1]), (1300, own[2]), (1, own[3]), (1, own[3])]
    assert own[2] <= 10
    # a plan of its own always has fewer terms
    for cols in (1, 2, 3, 4, 5):
        for f in range(cols + 1):
            got, plan = ask(plan_bin, [f"bplan {cols} 9 {f}", f"plan {max(1, f)} 0"])
            same = max(1, f) == cols or f > cols - cols // 4
            assert got.split() == ([str(cols), "9"] if same else [str(max(1, f)), plan.split()[0]]), (cols, f)
    # the witness itself stays at 15 bits
    assert ask(plan_bin, [f"bplan {1 << 21} 0 {1 << 21}", f"bplan {1 << 22} 0 {1 << 21}"]) == \
        [f"{1 << 21} 15", f"{1 << 21} 15"]


def test_fold_launches_are_what_the_plan_uses(plan_bin):
    """The launches issued are those the planning kernel's own fold loop (64:1
    while a bucket has more than 128 partial sums) can fill, for the largest
    bucket each lane count allows: two for the default lanes, never an empty
    third."""
    def loop(m):
        n = 0
        while m > 128:
            m, n = -(-m // 64), n + 1
        return n
    ms = [0, 1, 128, 129, 8192, 8193, (1 << 19), (1 << 19) + 1, (1 << 24) + 1] + \
        [lanes + 1 for lanes in (65536, 131072, 262144, 393216)]
    got = list(map(int, ask(plan_bin, [f"launches {m}" for m in ms])))
    assert got == [loop(m) for m in ms]
    assert got == [0, 0, 0, 1, 1, 2, 2, 3, 3, 2, 2, 2, 2]


def spread(rng, shape, entries, B):
    """Entries per bucket."""
    if shape == "one":
        counts = np.zeros(B, dtype=np.int64)
        counts[rng.integers(B)] = entries
    elif shape == "uniform":
        counts = np.full(B, entries // B, dtype=np.int64)
        counts[: entries % B] += 1
    elif shape == "singles":
        counts = np.zeros(B, dtype=np.int64)
        counts[rng.permutation(B)[: min(B, entries)]] = 1
    else:
        counts = rng.multinomial(entries, rng.dirichlet(np.full(B, 0.02)))
    return counts


@pytest.mark.parametrize("g2,target", [(0, 19), (1, 19), (0, 10), (1, 12), (0, 22), (1, 24)])
def test_buffer_bounds_cover_every_plan(plan_bin, g2, target):
    """What the layout allocates (msm_sizes, from the most entries its jobs can
    have) against the plan of a launch: every lane takes an equal run of its
    job's entries, the partial of lane l and bucket k goes to slot l + k of the
    job, and buckets of more than 128 partials are folded 64:1 launch by launch.
    Distributions from one bucket to all, batches of one to five jobs, full and
    nearly empty ones, at and around the lane rule's limits."""
    rng = np.random.default_rng(100 * target + g2)
    batches = [[(1, 8)], [(60000, 256)], [(1 << 21, 4096), (1 << 21, 4096), (9, 16), ((1 << 22) + 7, 1 << 15)],
               [(1 << 19, 64)] * 5, [((1 << 25) + 1, 1 << 15), (3, 4)], [(5000, 2)] * 3]
    for jobs in batches:
        entries, buckets = sum(e for e, _ in jobs), sum(B for _, B in jobs)
        for shape in ("one", "uniform", "singles", "skewed"):
            for fill in (1.0, 0.37, 1e-4, 0.0):
                counts = [spread(rng, shape, int(e * fill), B) for e, B in jobs]
                E = sum(int(c.sum()) for c in counts)
                sizes, piece = ask(plan_bin, [f"sizes {g2} {target} {len(jobs)} {entries} {buckets}",
                                              f"piece {g2} {target} 1 {E}"])
                lanes_cap, pool, rec_cap, complete, launches, *folds = map(int, sizes.split())
                p = int(piece.split()[0])
                base, cap = folds[::2], folds[1::2]
                lanes_before = b_off = 0
                ms = []
                for c in counts:
                    end = np.cumsum(c)
                    beg, k = end - c, np.arange(c.size)
                    first, last = beg // p, np.where(c > 0, (end - 1) // p, -1)
                    used = c > 0
                    # slots of one job: a bucket's come after the ones before it
                    lo, hi = (first + k)[used], (last + k)[used]
                    assert (lo[1:] > hi[:-1]).all()
                    lanes = -(-int(end[-1]) // p)
                    assert hi.size == 0 or hi[-1] < lanes + c.size
                    assert (hi + lanes_before + b_off < lanes_cap + buckets).all()
                    lanes_before, b_off = lanes_before + lanes, b_off + c.size
                    ms.append(np.where(used, last - first + 1, 0))
                assert lanes_before <= lanes_cap
                m, issued = np.concatenate(ms), 0
                while (m > 128).any():
                    assert issued < launches <= 4
                    folded = -(-m[m > 128] // 64)
                    assert folded.size <= rec_cap and folded.sum() <= cap[issued]
                    assert base[issued] >= lanes_cap + buckets and base[issued] + cap[issued] <= pool
                    assert issued == 0 or base[issued] >= base[issued - 1] + cap[issued - 1]
                    m = np.where(m > 128, -(-m // 64), m)
                    issued += 1
                assert buckets * 64 + 5 * 64 * len(jobs) == complete


def test_schedule_bytes_count_every_buffer(plan_bin):
    """The sorted list (whole blocks of four), the bucket starts and the two
    levels of their prefix, and the sort workgroups' counts."""
    for n, c in ((1, 4), (5, 7), (255, 0), (257, 8), (65537, 0), (1 << 20, 16)):
        C, W, B = map(int, ask(plan_bin, [f"plan {n} {c}"])[0].split())
        blocks = max(1, min(256, -(-n // 256)))
        words = [-(-n * W // 4) * 4, B + 1, B, -(-B // 64), blocks * B]
        assert list(map(int, ask(plan_bin, [f"schedule {n} {c}"])[0].split())) == words + [4 * sum(words)]


def test_bad_sizes_raise_instead_of_crashing(plan_bin):
    out = ask(plan_bin, ["divup 10 0", "divup 10 3", "plan 0 0", "plan 1024 17", f"plan {1 << 28} 15"])
    assert out[0].startswith("error internal sizing error")
    assert out[1] == "4"
    assert out[2].startswith("error MSM needs at least one term")
    assert out[3].startswith("error MSM window")
    assert out[4].startswith("error MSM too large")
