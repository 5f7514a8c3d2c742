"""Windows at the edges of the 32-bit counters against the oracle: as many
reads at one column as a counter holds and one more (slid bases and indels
count too), records and walked reads that just fit their buffers, reads of
many clips, and every MAPQ and quality that a counter can meet."""
import numpy as np
import pytest

from pilon_amd.abi import default_config
from pilon_amd.reads import pack_reads
from tests.helpers import assert_same_region, assert_same_stats

pytestmark = pytest.mark.gpu


def reads_of(case, n, ref, rng):
    def read(a, cigar="60M", seq=None, lo=0, hi=42, mapq=60):
        seq = seq if seq is not None else ref[a:a + 60]
        return dict(pos=a + 1, cigar=cigar, seq=seq, qual=[int(x) for x in rng.integers(lo, hi, len(seq))], mapq=mapq)
    # (a window of the column's reads and no others: 4095 is the last narrow one)
    out = [] if case == "reads" else [read(int(a), mapq=int(rng.integers(0, 61))) for a in rng.integers(0, len(ref) - 60, 300)]
    if case == "reads":          # every base at the largest quality and MAPQ
        out += [read(700, lo=126, hi=128, mapq=254 if k % 3 else 60) for k in range(n)]
    elif case == "events":       # slid deletions (an A after the run of Ts) and insertions
        out += [read(700, mapq=40) for _ in range(n - 60)]
        for k in range(60):
            if k % 2:
                out.append(read(700, "30M1D30M", ref[700:730] + ref[731:761]))
            else:
                out.append(read(700, "30M2I30M", ref[700:730] + "GA" + ref[730:760]))
    elif case == "walked":       # reads with an N
        out += [read(700, seq=ref[700:730] + "N" + ref[731:760]) for _ in range(n)]
    elif case == "clips":
        out += [read(700 + k % 9, "5S2S48M3S2S", ref[700:760]) for k in range(n)]
    return out


@pytest.mark.parametrize("case,n", [("reads", 3700), ("reads", 4095), ("reads", 4096), ("events", 3900), ("events", 4200),
                                    ("walked", 256), ("walked", 257), ("clips", 1), ("clips", 200)])
@pytest.mark.parametrize("min_qual,block", [(0, 256), (30, 512), (-1, 256)])
def test_narrow_counter_edges(case, n, min_qual, block):
    from oracle import oracle as O
    from pilon_amd.engine import Context
    print(f"case: {case} {n}, min_qual {min_qual}, block {block}", flush=True)
    rng = np.random.default_rng(n)
    s = [("ACGT"[x]) for x in rng.integers(0, 4, 1600)]
    s[726:740] = "TTTTTTTTTTTTTA"
    ref = "".join(s)
    b = pack_reads(reads_of(case, n, ref, rng))
    cfg = default_config(min_qual=min_qual)
    ctx = Context(cfg, device=0)
    try:
        ctx.ref_upload(0, "ctg", ref)
        rid = ctx.readset_upload(0, b)
        pile, calls, stats = ctx.batch_run([(0, 1, 1600, rid)], window=512, block=block, persistent=1)
        changes, _ = ctx.batch_fix()
    finally:
        ctx.close()
    want = O.run_region(cfg, ref.encode(), 1, 1600, [b], name="ctg")
    assert want["status"] == 0
    assert_same_region(pile, calls, want, f"{case} {n}")
    assert_same_stats(stats[0], want["stats"], f"{case} {n}")
    assert changes == want["changes"]
