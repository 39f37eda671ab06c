"""The prefill launch plan (prefill_plan.h) on the host: when latent attention takes 128 rows per workgroup instead of 64, and
when the tokens of a row block are split."""
import ctypes
import heapq
import random
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def build_probe(directory):
    """Compiles tests/prefill_plan_probe.cc with the host compiler; returns groups(num_seqs, tokens, ...) -> 1 or 2."""
    out = directory / "libprefillplanprobe.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{ROOT / 'include'}",
                    f"-I{ROOT / 'infinicore_amd' / 'csrc'}", str(ROOT / "tests" / "prefill_plan_probe.cc"), "-o", str(out)],
                   check=True, capture_output=True, text=True)
    lib = ctypes.CDLL(str(out))
    lib.latentPrefillProbe.argtypes = [ctypes.POINTER(ctypes.c_longlong), ctypes.c_float]

    lib.splitPrefillProbe.argtypes = [ctypes.POINTER(ctypes.c_longlong)] * 2
    lib.splitPrefillProbe.restype = ctypes.c_float

    def split(num_seqs, tokens, table_tokens, heads=32, kv_heads=8, head_size=128, value_size=None, units=256):
        args = (ctypes.c_longlong * 10)(num_seqs, tokens, heads, kv_heads, value_size or head_size, 16, -(-table_tokens // 16),
                                        units, False, head_size)
        out = (ctypes.c_longlong * 8)()
        cost = lib.splitPrefillProbe(args, out)
        return dict(zip(("tiled", "parts", "merge", "from", "bytes", "acc", "ml", "flags"), out), cost=cost)

    def groups(num_seqs, tokens, table_tokens, heads=16, kv_heads=1, value_size=512, alibi=False, scale=0.04, units=256):
        args = (ctypes.c_longlong * 9)(num_seqs, tokens, heads, kv_heads, value_size, 16, -(-table_tokens // 16), units, alibi)
        return lib.latentPrefillProbe(args, scale)

    groups.split = split
    return groups


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    return build_probe(tmp_path_factory.mktemp("plan"))


@pytest.fixture(autouse=True)
def no_knobs(monkeypatch):
    for k in ("INFINIOP_AMD_PREFILL_GROUPS", "INFINIOP_AMD_PREFILL_KERNEL", "INFINIOP_AMD_PREFILL_PARTS", "INFINIOP_AMD_PREFILL_MERGE_POLLS"):
        monkeypatch.delenv(k, raising=False)


def makespan(new, hist, group, block_rows, units=256):
    """Time of the batch in tokens of a 64-row block: workgroups start in grid order, each on the compute unit that is free
    first. The grid has the longest blocks first where it is one to six rounds of workgroups, else the last sequence first and
    within it the blocks that see most. A block of 128 rows takes 1.4 x as long as one of 64 over the same tokens; the start
    of a block is worth some 40 tokens."""
    blocks = []
    for n, h in reversed(list(zip(new, hist))):
        rows = n * group
        blocks += [h + (min((b + 1) * block_rows, rows) - 1) // group + 1 for b in reversed(range(-(-rows // block_rows)))]
    grid = sum(new) * group // block_rows + len(new)
    if units < grid <= 6 * units:
        blocks.sort(reverse=True)
    free = [0.0] * units
    end = 0.0
    for sees in blocks:
        t = heapq.heappop(free) + (40 + sees) * (1.4 if block_rows == 128 else 1.0)
        end = max(end, t)
        heapq.heappush(free, t)
    return end


def test_128_rows_are_taken_only_where_they_are_not_slower(probe):
    """Batches of equal and of ragged lengths, with and without history, on tables as wide as the longest sequence."""
    rng = random.Random(3)
    taken = 0
    for _ in range(250):
        seqs = int(2 ** rng.uniform(0, 6))
        top = max(1, int(rng.uniform(900, 5000) / seqs))
        low = top if rng.random() < 0.5 else max(1, int(top * rng.uniform(0.125, 1)))
        longest = 0 if rng.random() < 0.4 else int(16 * 2 ** rng.uniform(0, 9))
        shortest = longest if rng.random() < 0.5 else int(longest * rng.uniform(0.125, 1))
        new = [rng.randint(low, top) for _ in range(seqs)]
        hist = [rng.randint(shortest, longest) for _ in range(seqs)]
        if probe(seqs, sum(new), max(n + h for n, h in zip(new, hist))) == 2:
            taken += 1
            t64, t128 = makespan(new, hist, 16, 64), makespan(new, hist, 16, 128)
            # 1.05: rows of the batch are counted from the average length, and the history of one sequence in whole pages
            assert t128 <= 1.05 * t64, (new, hist, t64, t128)
    assert taken > 50


@pytest.mark.parametrize("seqs,new,history,want", [
    (1, 1024, 8192, 1),   # one round of either
    (1, 1100, 0, 1), (1, 2000, 0, 1), (2, 900, 0, 1), (4, 300, 0, 1),  # a second round of short blocks
    (1, 2000, 1000, 1), (1, 2000, 4000, 2),                             # one sequence: by its history
    (2, 900, 2000, 1),                                                  # several: their lengths are not known
    (4, 640, 2000, 1),                                                  # three rounds against two
    (1, 3200, 0, 2), (4, 1000, 2000, 2), (400, 8, 0, 2), (16, 320, 4000, 2),
])
def test_rounds(probe, seqs, new, history, want):
    assert probe(seqs, seqs * new, new + history) == want


def test_only_the_shape_that_has_the_kernel_takes_128_rows(probe):
    assert probe(16, 16 * 320, 4000) == 2
    assert probe(16, 16 * 320, 4000, value_size=576) == 1
    assert probe(16, 16 * 320, 4000, alibi=True) == 1
    assert probe(16, 16 * 320, 4000, scale=-1.0) == 1
    assert probe(16, 16 * 320, 4000, scale=0.0) == 1
    assert probe(2, 2 * 320, 4000, heads=128) == 2  # 40 960 rows per sequence
    assert probe(16, 16 * 320, 4000, units=1024) == 1


# ---- splitting -------------------------------------------------------------------------------------------------

def parts_of(plan, tokens, step):
    """splitSteps of prefill_split.h: the parts that a row block seeing `tokens` gets, and the steps of each."""
    steps = -(-tokens // step)
    parts = 1
    if tokens >= plan["from"]:
        each = max(int((tokens * plan["cost"]) ** 0.5), 128)
        parts = min(plan["parts"], steps, -(-tokens // each))
    per = -(-steps // parts)
    return -(-steps // per), per


def row_blocks(new, group):
    return sum(-(-n * group // 64) for n in new)


def test_splits_fit_their_workspace_and_the_device(probe, monkeypatch):
    """Over shapes, lengths and forced numbers of parts: the row blocks that a batch can have fit the grid, every row of every
    part its region, and what a block is cut into covers its steps."""
    rng = random.Random(7)
    split_plans = 0
    for _ in range(3000):
        heads, kv_heads = rng.choice([(32, 8), (16, 16), (28, 4), (8, 1), (64, 8), (40, 8), (5, 1)])
        head = rng.choice([64, 128, 192, 256, 576])
        value = 512 if head == 576 and rng.random() < 0.8 else head
        seqs = int(2 ** rng.uniform(0, 7))
        new = [rng.choice([0, 1, rng.randint(1, 30), rng.randint(1, 600)]) for _ in range(seqs)]
        if sum(new) == 0:
            continue
        total = sum(new) if rng.random() < 0.9 else max(1, sum(new) - 3)  # (cum_seq_lens_q may say more than q holds)
        table = int(16 * 2 ** rng.uniform(0, 11))
        if rng.random() < 0.3:
            monkeypatch.setenv("INFINIOP_AMD_PREFILL_PARTS", str(rng.choice([1, 2, 7, 64])))
        else:
            monkeypatch.delenv("INFINIOP_AMD_PREFILL_PARTS", raising=False)
        plan = probe.split(seqs, total, table, heads, kv_heads, head, value)
        if plan["parts"] <= 1:
            assert plan["bytes"] == 0
            continue
        split_plans += 1
        group = heads // kv_heads
        grid = (total * group // 64 + seqs) * kv_heads
        if total == sum(new):
            assert row_blocks(new, group) * kv_heads <= grid
        rows = grid * plan["parts"] * 64
        assert plan["acc"] >= rows * value * 4 and plan["ml"] >= rows * 8 and plan["flags"] >= (rows + grid * 32) * 8
        assert all(plan[k] % 256 == 0 for k in ("acc", "ml", "flags"))
        assert plan["bytes"] == plan["acc"] + plan["ml"] + plan["flags"] + 256
        assert plan["parts"] <= 64 and plan["merge"] in (1, 2, 4, 8)
        step = 32 if head in (192, 576) else 64
        for tokens in (1, 127, 128, 129, 255, 257, table // 2 + 1, table):
            used, per = parts_of(plan, tokens, step)
            steps = -(-tokens // step)
            assert 1 <= used <= plan["parts"] and (used - 1) * per < steps <= used * per
            assert used <= -(-tokens // 128)  # a part per 128 tokens at most
    assert split_plans > 500


@pytest.mark.parametrize("seqs,new,table,head,heads,kv_heads,parts", [
    (1, 3, 5800, 128, 32, 8, 2), (1, 128, 8000, 128, 32, 8, 2), (4, 64, 4000, 128, 32, 8, 2), (16, 5, 2000, 128, 32, 8, 2),
    (1, 3, 5800, 576, 16, 1, 2), (1, 128, 8000, 256, 28, 4, 2), (4, 3, 32768, 64, 16, 16, 2),
    (1, 3, 250, 128, 32, 8, 1), (4, 64, 500, 128, 32, 8, 1), (16, 512, 4000, 128, 32, 8, 1), (4, 3000, 3000, 128, 32, 8, 1)])
def test_who_is_split(probe, seqs, new, table, head, heads, kv_heads, parts):
    plan = probe.split(seqs, seqs * new, table, heads, kv_heads, head, 512 if head == 576 else head)
    assert (plan["parts"] >= 2) == (parts == 2)


@pytest.mark.parametrize("head,heads,kv_heads,whole,cut", [(64, 16, 16, 300, 900), (128, 32, 8, 250, 700), (192, 32, 8, 150, 500),
                                                         (256, 28, 4, 150, 500), (576, 16, 1, 127, 350)])
def test_short_blocks_stay_whole_on_wide_tables(probe, head, heads, kv_heads, whole, cut):
    step = 32 if head in (192, 576) else 64
    for table in (4096, 32768):
        plan = probe.split(1, 3, table, heads, kv_heads, head, 512 if head == 576 else head)
        assert plan["parts"] > 1
        assert parts_of(plan, whole, step)[0] == 1 and parts_of(plan, cut, step)[0] > 1
