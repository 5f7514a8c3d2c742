"""The kernel core built for the host (same window decomposition, runs,
deferral and Pass-1 code as the gfx950 kernels) against the oracle."""
import numpy as np
import pytest

from pilon_amd.abi import default_config
from tests import corehost as CH
from tests import kat_cases as K
from tests.helpers import assert_same_region, assert_same_stats


def oracle():
    from oracle import oracle as O
    return O


@pytest.mark.parametrize("make", K.ALL, ids=[f.__name__ for f in K.ALL])
@pytest.mark.parametrize("W", [64, 1024])
def test_kat_core_host(make, W):
    case = make()
    b = K.batch_of(case)
    cfg = default_config(**case.get("cfg", {}))
    ref = oracle().run_region(cfg, case["ref"], case["start"], case["stop"], [b], name="ctg")
    got = CH.run(cfg, case["ref"].encode(), b, [(case["start"], case["stop"])], W=W, name="ctg")[0]
    assert got["status"] == 0
    assert_same_region(got["pile"], got["calls"], ref, make.__name__)
    assert_same_stats(got["stats"], ref["stats"])
    assert got["changes"] == ref["changes"] and got["bases"] == ref["bases"]


@pytest.mark.parametrize("make", K.LONG, ids=[f.__name__ for f in K.LONG])
def test_kat_long_read_core_host(make):
    """The long-read cases: the reads walked with their longReadType, and
    excludeMotifs on the change list."""
    from pilon_amd.abi import BAM_TYPES
    case = make()
    cfg = default_config(**case.get("cfg", {}))
    sets = K.sets_of(case)
    ref = oracle().run_region(cfg, case["ref"], case["start"], case["stop"], [b for b, _ in sets], name="ctg",
                              set_types=[BAM_TYPES[t] for _, t in sets])
    b, lrt, kinds = K.merged_of(case)
    got = CH.run(cfg, case["ref"].encode(), b, [(case["start"], case["stop"])], W=64, name="ctg", lrt=lrt,
                 set_kinds=kinds)[0]
    assert got["status"] == 0
    assert_same_region(got["pile"], got["calls"], ref, make.__name__)
    assert_same_stats(got["stats"], ref["stats"])
    assert got["changes"] == ref["changes"] and got["bases"] == ref["bases"]


@pytest.mark.parametrize("lr", ["nanopore", "pacbio"])
def test_synthetic_long_read_core_host(lr):
    """A c2-shaped contig (error indels, N runs) piled as one long-read BAM:
    every homopolymer and CC_GG motif of the random draft meets the reads'
    indels and bases."""
    from pilon_amd.abi import BAM_TYPES
    from pilon_amd.synth import SynthData, preset
    p = preset("c2", scale=0.04)
    p.update({"n_rate": 0.001, "err_indel_rate": 0.004})
    d = SynthData(p)
    cfg = default_config(longread=1)
    draft, b = d.draft(0), d.batch(0)
    L = len(draft)
    regions = [(1, L // 2), (L // 2 + 1, L), (7, L - 5)]
    lrt = np.full(b.n, K.LR_TYPE[lr], np.uint8)
    got = CH.run(cfg, draft, b, regions, W=512, name=d.names[0], lrt=lrt, set_kinds=2 if lr == "nanopore" else 0)
    for (s, e), g in zip(regions, got):
        ref = oracle().run_region(cfg, draft, s, e, [b], name=d.names[0], set_types=[BAM_TYPES[lr]])
        assert g["status"] == ref["status"] == 0
        assert_same_region(g["pile"], g["calls"], ref, f"{lr} {s}-{e}")
        assert_same_stats(g["stats"], ref["stats"])
        assert g["changes"] == ref["changes"] and g["bases"] == ref["bases"]
    # the long-read rules changed the pileup: indel quality sums differ from a frags run
    plain = oracle().run_region(cfg, draft, 1, L // 2, [b], name=d.names[0])
    assert not np.array_equal(plain["pile"], got[0]["pile"])


@pytest.mark.parametrize("name,scale,extra", [
    ("c1", 1.0, {}),
    ("c2", 0.04, {"n_rate": 0.001, "err_indel_rate": 0.002}),
    ("c5", 0.004, {}),
])
def test_synthetic_core_host(name, scale, extra):
    p = __import__("pilon_amd.synth", fromlist=["preset"]).preset(name, scale=scale)
    p.update(extra)
    from pilon_amd.synth import SynthData
    d = SynthData(p)
    cfg = default_config()
    draft, b = d.draft(0), d.batch(0)
    L = len(draft)
    regions = [(1, L // 3), (L // 3 + 1, 2 * L // 3), (2 * L // 3 + 1, L), (1, L)]
    for W in (256, 2048):
        got = CH.run(cfg, draft, b, regions, W=W, name=d.names[0])
        for (s, e), g in zip(regions, got):
            ref = oracle().run_region(cfg, draft, s, e, [b], name=d.names[0])
            assert g["status"] == ref["status"] == 0
            assert_same_region(g["pile"], g["calls"], ref, f"{name} {s}-{e} W={W}")
            assert_same_stats(g["stats"], ref["stats"])
            assert g["changes"] == ref["changes"] and g["bases"] == ref["bases"]


def test_edge_detected_by_core_host():
    case = K.case_insertion_rotation(start=14)
    got = CH.run(default_config(), case["ref"].encode(), K.batch_of(case), [(14, 40)], W=64)[0]
    assert got["status"] == 4


@pytest.mark.parametrize("read_len", [700, 9500])
@pytest.mark.parametrize("lr,W", [("nanopore", 64), ("pacbio", 512)])
def test_long_reads_by_segments_core_host(read_len, lr, W):
    """Reads of many windows piled by the segments each window can touch."""
    from pilon_amd.abi import BAM_TYPES
    from tests.test_gpu_longread import long_data
    name, draft, b = long_data(read_len, 7 + read_len)
    cfg = default_config(longread=1, min_qual=3)
    lrt = np.full(b.n, K.LR_TYPE[lr], np.uint8)
    regions = [(1, len(draft)), (1001, 9000)]
    got = CH.run(cfg, draft, b, regions, W=W, name=name, lrt=lrt, set_kinds=2 if lr == "nanopore" else 0)
    assert any(g["status"] == 0 for g in got)
    for (s, e), g in zip(regions, got):
        ref = oracle().run_region(cfg, draft, s, e, [b], name=name, set_types=[BAM_TYPES[lr]])
        assert g["status"] == ref["status"]
        if g["status"] == 0:
            assert_same_region(g["pile"], g["calls"], ref, f"{lr} {s}-{e}")
            assert_same_stats(g["stats"], ref["stats"])
            assert g["changes"] == ref["changes"] and g["bases"] == ref["bases"]


@pytest.mark.parametrize("n_recs,rec_cap,spill_cap,whole", [
    ([0, 128, 129, 5], 1000, 1, True), ([300, 300, 2], 1000, 344, True),       # the list just holds the spilled ones
    ([300, 300, 2], 1000, 343, False), ([128, 400, 10, 200], 4000, 16, False),  # ... and does not
    ([300, 300, 2], 500, 344, False), ([300, 300, 2], 500, 10, False),          # an overfull record buffer
])
def test_no_unwritten_record_is_read(n_recs, rec_cap, spill_cap, whole):
    """A column's scan of its window's records meets every one of them, or,
    where they did not all find room, none that the batch did not write."""
    bad, seen = CH.evidence(n_recs, 128, rec_cap, spill_cap)
    assert bad == 0
    assert (list(seen) == n_recs) == whole


def test_kept_scratch_makes_no_call_fail():
    """A lane's scratch stays for its next call, up to a bound, and goes back
    when any allocation finds no memory, unless a call is using it."""
    assert CH.lib().ch_scratch() == 0


def test_cost_bins_order_every_window():
    """Any cost falls in a bin of the table, more work never in a later one,
    and windows placed by their bins fill the queue's slots once each."""
    bin_of = CH.lib().ch_cost_bin
    costs = [0, 1, 15, 16, 17, 31, 32, 255, 256, 4095, 4096, 65_534, 65_535, 65_536, 2 ** 19 - 1, 2 ** 19, 557_056,
             2 ** 20, 2 ** 24 - 1, 2 ** 31 - 1, 2 ** 31, 2 ** 40]
    bins = [bin_of(c) for c in costs]
    assert all(0 <= b < 256 for b in bins) and bins == sorted(bins, reverse=True)
    assert all(bin_of(c) >= bin_of(c + 1) for c in range(70_000))
    rng = np.random.default_rng(3)
    cost = np.concatenate([np.full(2000, 300), rng.integers(0, 2 ** 24, 500), [6, 6, 6, 2 ** 20, 2 ** 31]])
    b = np.array([bin_of(int(c)) for c in cost])
    start = np.concatenate([[0], np.cumsum(np.bincount(b, minlength=256))[:-1]])
    taken = np.zeros(256, int)
    slot = []
    for x in b:                                    # k_plan's counts, k_heads' slots
        slot.append(start[x] + taken[x])
        taken[x] += 1
    assert sorted(slot) == list(range(len(cost)))
    c = np.minimum(cost, 65_535)[np.argsort(slot)]
    assert np.all(c[1:] <= 1.0625 * c[:-1] + 1)
