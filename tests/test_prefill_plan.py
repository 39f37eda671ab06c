"""The prefill launch plan (prefill_plan.h) on the host: when latent attention takes 128 rows per workgroup instead of 64."""
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

    def groups(num_seqs, tokens, table_tokens, heads=16, kv_heads=1, value_size=512, alibi=False, scale=0.04, units=256):
        args = (ctypes.c_longlong * 9)(num_seqs, tokens, heads, kv_heads, value_size, 16, -(-table_tokens // 16), units, alibi)
        return lib.latentPrefillProbe(args, scale)

    return groups


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    return build_probe(tmp_path_factory.mktemp("plan"))


@pytest.fixture(autouse=True)
def no_knobs(monkeypatch):
    for k in ("INFINIOP_AMD_PREFILL_GROUPS", "INFINIOP_AMD_PREFILL_KERNEL"):
        monkeypatch.delenv(k, raising=False)


def makespan(new, hist, group, block_rows, units=256):
    """Time of the batch in tokens of a 64-row block: workgroups start in grid order (last sequence first, within it the
    blocks that see most first), each on the compute unit that is free first. A block of 128 rows takes 1.4 x as long as
    one of 64 over the same tokens; the start of a block is worth some 40 tokens."""
    free = [0.0] * units
    end = 0.0
    for n, h in reversed(list(zip(new, hist))):
        rows = n * group
        for b in reversed(range(-(-rows // block_rows))):
            sees = h + (min((b + 1) * block_rows, rows) - 1) // group + 1
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
