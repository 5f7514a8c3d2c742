"""Indel evidence and candidate order of a batch against the oracle: windows
whose records just fit their LDS buffer (128) and spill beyond it, at one
column and over many, with the windows taken in their own order and, when
more than the launch holds at once, in cost order; more spilled records than
their list holds at first, on a context that held another set's records; a
window of more reads than the cost order tells apart among them."""
import numpy as np
import pytest

from pilon_amd.abi import default_config
from pilon_amd.reads import pack_reads
from tests.helpers import assert_same_region, assert_same_stats

pytestmark = pytest.mark.gpu


def indel_reads(ref, sites, seed):
    """60-base reads, `n` per (locus, op, length) site carrying the indel 30
    bases in (two insertion strings, so that majorities differ)."""
    rng = np.random.default_rng(seed)
    out = []
    for locus, op, ln, n in sites:
        a = locus - 31
        for k in range(n):
            q = [int(x) for x in rng.integers(20, 41, 60 + (ln if op == "I" else 0))]
            if op == "I":
                ins = ("GATC" if k % 4 else "GTTC")[:ln]
                out.append(dict(pos=a + 1, cigar=f"30M{ln}I30M", seq=ref[a:a + 30] + ins + ref[a + 30:a + 60], qual=q))
            else:
                out.append(dict(pos=a + 1, cigar=f"30M{ln}D30M", seq=ref[a:a + 30] + ref[a + 30 + ln:a + 60 + ln],
                                qual=q[:60]))
    return out


@pytest.mark.parametrize("n", [127, 128, 129, 700])
@pytest.mark.parametrize("window,persistent", [(64, 1), (512, 0)])
def test_window_record_buffer(n, window, persistent):
    from oracle import oracle as O
    from pilon_amd.engine import Context
    print(f"case: {n} records in one column, window {window}", flush=True)
    rng = np.random.default_rng(n)
    ref = "".join("ACGT"[x] for x in rng.integers(0, 4, 4000))
    sites = [(1100, "I", 4, n), (1900, "D", 3, n // 2), (1920, "I", 2, n - n // 2)]
    sites += [(2600 + 9 * k, "I" if k % 2 else "D", 1 + k % 4, 1 + k % 9) for k in range(60)]
    b = pack_reads(indel_reads(ref, sites, n))
    cfg = default_config()
    ctx = Context(cfg, device=0)
    try:
        ctx.ref_upload(0, "ctg", ref)
        rid = ctx.readset_upload(0, b)
        pile, calls, stats = ctx.batch_run([(0, 1, 4000, rid)], window=window, block=256, persistent=persistent)
        changes, _ = ctx.batch_fix()
        text, _ = ctx.batch_vcf()
    finally:
        ctx.close()
    want = O.run_region(cfg, ref.encode(), 1, 4000, [b], name="ctg", vcf=O.VCF_ON)
    assert want["status"] == 0
    assert_same_region(pile, calls, want, f"{n} records")
    assert_same_stats(stats[0], want["stats"], f"{n} records")
    assert changes == want["changes"]
    assert text == want["vcf"]


def test_more_spilled_than_the_list_holds():
    """16,720 spilled records (the list starts at 16,384) at the columns where
    an earlier batch of another read set left its own, then that set again."""
    from oracle import oracle as O
    from pilon_amd.engine import Context
    print("case: spill list overflow over an earlier batch's records", flush=True)
    rng = np.random.default_rng(5)
    ref = "".join("ACGT"[x] for x in rng.integers(0, 4, 20_000))
    few = pack_reads(indel_reads(ref, [(64 * w + 41, "I", 4, 110) for w in range(1, 300)], 1))
    out = indel_reads(ref, [(64 * w + 41, "I", 3, 1800) for w in range(150, 160)], 2)
    for r in out:                                  # an N: walked, so the read set's segments do not tell
        r["seq"] = r["seq"][:3] + "N" + r["seq"][4:]
    many = pack_reads(out)
    cfg = default_config()
    want = [O.run_region(cfg, ref.encode(), 1, len(ref), [b], name="ctg") for b in (few, many)]
    ctx = Context(cfg, device=0)
    try:
        ctx.ref_upload(0, "ctg", ref)
        ids = [ctx.readset_upload(0, b) for b in (few, many)]
        for k in (0, 1, 0):
            pile, calls, stats = ctx.batch_run([(0, 1, len(ref), ids[k])], window=64, block=256, persistent=1)
            changes, _ = ctx.batch_fix()
            assert_same_region(pile, calls, want[k], f"set {k}")
            assert_same_stats(stats[0], want[k]["stats"], f"set {k}")
            assert changes == want[k]["changes"]
    finally:
        ctx.close()


def test_candidates_over_many_blocks():
    """Contigs whose candidate masks fill several list blocks, more windows
    than the launch holds at once (cost order), regions of a single locus
    among them: every region's changes in order."""
    import ctypes as C
    from oracle import oracle as O
    from pilon_amd.engine import Context, lib
    from pilon_amd.synth import SynthData, preset
    p = preset("c3", scale=0.01)
    p.update(coverage=25, snv_rate=0.01, indel_rate=0.002, lens=p["lens"] + [300_001])
    print("case: candidates over many blocks", flush=True)
    d = SynthData(p)
    cfg = default_config()
    ctx = Context(cfg, device=0)
    try:
        ids = []
        for i in range(d.n):
            ctx.ref_upload(i, d.names[i], d.draft(i))
            ids.append(ctx.readset_upload(i, d.batch(i)))
        regions = [(i, 1, len(d.draft(i)), ids[i]) for i in range(d.n)] + [(0, 500, 500, ids[0])]
        _, _, stats = ctx.batch_run(regions, window=64, block=256, persistent=1, copy_out=False)
        changes, fasta = ctx.batch_fix(element=list(range(len(regions))))
        el = np.arange(len(regions), dtype=np.int32)
        ptr, clen, flen = C.c_void_p(), C.c_int64(), C.c_int64()
        assert lib().pl_batch_fix(ctx.h, el.ctypes.data, len(el), C.byref(ptr), C.byref(clen), None, C.byref(flen)) == 0
        assert C.string_at(ptr, clen.value).decode() == changes and flen.value == len(fasta)
        lib().pl_free(ptr)
    finally:
        ctx.close()
    want_c = ""
    for (i, s, e, _), st in zip(regions, stats):
        w = O.run_region(cfg, d.draft(i), s, e, [d.batch(i)], name=d.names[i])
        assert w["status"] == 0
        assert_same_stats(st, w["stats"], f"{i}:{s}-{e}")
        want_c += w["changes"]
    assert changes == want_c
    assert changes.count("\n") > 2000


def test_very_deep_window_in_cost_order():
    """A window of 70,000 reads (costs are told apart up to 65,535), one of
    66,000 and a contig's last, of a position, among more windows than the
    launch holds at once: every window is piled."""
    from oracle import oracle as O
    from pilon_amd.engine import Context
    print("case: very deep windows in cost order", flush=True)
    rng = np.random.default_rng(11)
    n = 64 * 2600 + 1
    ref = "".join("ACGT"[x] for x in rng.integers(0, 4, n))
    starts = np.concatenate([np.full(70_000, 64 * 900 + 20), np.full(66_000, 64 * 2100 + 20),
                             rng.integers(0, n - 30, 20_000)])
    b = pack_reads([dict(pos=int(a) + 1, cigar="30M", seq=ref[a:a + 30], qual=[30] * 30, mapq=40 + int(a) % 3)
                    for a in np.sort(starts)])
    cfg = default_config()
    want = O.run_region(cfg, ref.encode(), 1, n, [b], name="ctg")
    assert want["status"] == 0
    ctx = Context(cfg, device=0)
    try:
        ctx.ref_upload(0, "ctg", ref)
        rid = ctx.readset_upload(0, b)
        for window in (64, 512):
            pile, calls, stats = ctx.batch_run([(0, 1, n, rid)], window=window, block=256, persistent=1)
            assert_same_region(pile, calls, want, f"window {window}")
            assert_same_stats(stats[0], want["stats"], f"window {window}")
    finally:
        ctx.close()
