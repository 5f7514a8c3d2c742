"""Long-read BAMs (--nanopore, --pacbio) on the GPU against the oracle:
resident long-read sets through the batched form (pileup, calls, stats,
.changes and FASTA with excludeMotifs), and a region that mixes a frags BAM
with a nanopore BAM through the plain form (reads of both kinds merged,
each piled by its own BAM's rules)."""
import numpy as np
import pytest

from pilon_amd.abi import BAM_TYPES, default_config
from tests.helpers import assert_same_region, assert_same_stats

pytestmark = pytest.mark.gpu


def data():
    from pilon_amd.synth import SynthData, preset
    p = preset("c2", scale=0.04)
    p.update({"n_rate": 0.001, "err_indel_rate": 0.004, "n_indel": 40})
    return SynthData(p)


@pytest.mark.parametrize("lr", ["nanopore", "pacbio"])
def test_long_read_set_batched(lr):
    from oracle import oracle as O
    from pilon_amd.engine import Context, contig_regions
    print(f"case: resident {lr} set, batched", flush=True)
    d = data()
    cfg = default_config(longread=1)
    draft, b = d.draft(0), d.batch(0)
    L = len(draft)
    ctx = Context(cfg, device=0)
    try:
        ctx.ref_upload(0, d.names[0], draft)
        rid = ctx.readset_upload(0, b, bam_type=lr)
        regions = contig_regions(L, 60_000)
        pile, calls, stats = ctx.batch_run([(0, s, e, rid) for s, e in regions], persistent=1)
        changes, fasta = ctx.batch_fix()
    finally:
        ctx.close()
    want_c, want_f = O.process_regions_output(cfg, [(d.names[0], draft)], [(0, s, e) for s, e in regions],
                                              lambda k: [b], set_types=[BAM_TYPES[lr]])
    off = 0
    for k, (s, e) in enumerate(regions):
        ref = O.run_region(cfg, draft, s, e, [b], name=d.names[0], set_types=[BAM_TYPES[lr]])
        assert ref["status"] == 0
        n = e - s + 1
        assert_same_region(pile[:, off:off + n], calls[off:off + n], ref, f"{lr} {s}-{e}")
        assert_same_stats(stats[k], ref["stats"], f"{lr} {s}-{e}")
        off += n
    assert changes == want_c
    assert fasta == want_f
    # the long-read rules matter here: the frags reading of the same reads differs
    plain = O.run_region(cfg, draft, 1, regions[0][1], [b], name=d.names[0])
    assert not np.array_equal(plain["pile"], pile[:, :regions[0][1]])


def test_frags_and_nanopore_region():
    from oracle import oracle as O
    from pilon_amd.engine import Context, PileUpRegion
    print("case: region with a frags and a nanopore BAM", flush=True)
    d = data()
    cfg = default_config(longread=1)
    draft, b = d.draft(0), d.batch(0)
    L = len(draft)
    idx = np.arange(b.n)
    Fs, Ns = b.take(idx[idx % 3 != 0]), b.take(idx[idx % 3 == 0])
    ctx = Context(cfg, device=0)
    try:
        ctx.ref_upload(1, d.names[0], draft)
        for s, e in ((1, L), (1001, L - 999)):
            pr = PileUpRegion(ctx, 1, s, e)
            pr.addReads(Fs)
            pr.addReads(Ns, bam_type="nanopore")
            pr.postProcess()
            changes, bases = pr.fix()
            pr.close()
            ref = O.run_region(cfg, draft, s, e, [Fs, Ns], name=d.names[0], set_types=[0, 3])
            assert ref["status"] == 0
            assert_same_region(pr.pile, pr.calls, ref, f"mixed {s}-{e}")
            assert_same_stats(pr.stats, ref["stats"], f"mixed {s}-{e}")
            assert changes == ref["changes"] and bases == ref["bases"]
    finally:
        ctx.close()


def long_data(read_len, seed):
    """A contig with homopolymer and tandem runs (indels slide far) under
    unpaired reads of read_len, an indel every 30 bases, some clipped, some
    with N (walked)."""
    from pilon_amd.reads import ReadBatch
    from pilon_amd.synth import SynthData, preset
    p = preset("c1", scale=0.4, seed=seed)
    p.update(read_len=read_len, insert_mean=read_len, insert_sd=0, coverage=15, err_indel_rate=0.03, err_indel_max=3,
             sub_rate=0.02, clip_frac=0.3, clip_min=5, clip_max=400, n_rate=2e-5, qual_lo=0, qual_hi=25, repeat_copies=3,
             repeat_len=2000)
    d = SynthData(p)
    b = d.batch(0)
    b = ReadBatch(b.pos, np.zeros_like(b.tlen), b.flag & 0xA010, b.mapq, b.cigar_off, b.cigar, b.seq_off, b.bases2,
                  b.quals, b.exo_read, b.exo_off, b.nib)
    draft = bytearray(d.draft(0))
    for k in range(40):                       # runs the reads' indels are normalised along
        a = 500 + 900 * k
        draft[a:a + 70] = (b"A" * 70 if k % 3 == 0 else b"CAG" * 23 + b"C" if k % 3 == 1 else b"CCAGG" * 14)
    return d.names[0], bytes(draft), b


@pytest.mark.parametrize("read_len", [700, 3001, 9500])
@pytest.mark.parametrize("lr,window,block", [("nanopore", 512, 256), ("pacbio", 64, 512), ("nanopore", 1024, 1024)])
def test_long_reads_by_segments(read_len, lr, window, block):
    """Reads of many windows, whose segments each window takes its own part
    of: read lengths below and above the short sets' scan margin, windows of
    one and several chunks of reads."""
    from oracle import oracle as O
    from pilon_amd.engine import Context, contig_regions
    print(f"case: {lr} reads of {read_len}, window {window}", flush=True)
    name, draft, b = long_data(read_len, 7 + read_len)
    cfg = default_config(longread=1, min_qual=3)
    ctx = Context(cfg, device=0)
    try:
        ctx.ref_upload(0, name, draft)
        rid = ctx.readset_upload(0, b, bam_type=lr)
        rid2 = ctx.readset_upload_many([(0, b, lr)])[0]
        regions = [(1, len(draft)), (1001, 9000)]
        want = [O.run_region(cfg, draft, s, e, [b], name=name, set_types=[BAM_TYPES[lr]]) for s, e in regions]
        regions = [x for x, w in zip(regions, want) if w["status"] == 0]
        want = [w for w in want if w["status"] == 0]
        assert want
        for ids in (rid, rid2):
            pile, calls, stats = ctx.batch_run([(0, s, e, ids) for s, e in regions], window=window, block=block,
                                               persistent=1)
            off = 0
            for (s, e), st, w in zip(regions, stats, want):
                n = e - s + 1
                assert_same_region(pile[:, off:off + n], calls[off:off + n], w, f"{lr} {s}-{e}")
                assert_same_stats(st, w["stats"], f"{lr} {s}-{e}")
                off += n
    finally:
        ctx.close()


def read_of_ops(ref, pos, ops, rng):
    """A read at 0-based pos with these (op, length) pairs: the reference's
    bases where it matches, random ones where it inserts or is clipped."""
    seq, at = "", pos
    for op, n in ops:
        if op in "IS":
            seq += "".join("ACGT"[x] for x in rng.integers(0, 4, n))
        else:
            seq += ref[at:at + n] if op == "M" else ""
            at += n
    return dict(pos=pos + 1, cigar="".join(f"{n}{op}" for op, n in ops), seq=seq, mapq=int(rng.integers(5, 61)),
                qual=[int(x) for x in rng.integers(3, 41, len(seq))])


@pytest.mark.parametrize("n_ops", [1, 2, 63, 64, 65, 127, 128, 129, 300])
@pytest.mark.parametrize("ends", ["plain", "clipped", "inner_clip", "lead_del", "lead_ins"])
def test_long_reads_of_any_op_count(n_ops, ends):
    """Reads whose ops just fill the rounds of 64 a wave takes of them, with
    clips at their ends (or, walked, between ops) and indels first."""
    from oracle import oracle as O
    from pilon_amd.engine import Context
    from pilon_amd.reads import pack_reads
    print(f"case: long reads of {n_ops} ops, {ends}", flush=True)
    rng = np.random.default_rng(n_ops)
    ref = "".join("ACGT"[x] for x in rng.integers(0, 4, 6000))
    ref = ref[:900] + "A" * 40 + "CAG" * 30 + ref[1030:2000] + "CCAGG" * 30 + ref[2150:]
    reads = []
    for k in range(24):
        ops = [("M", int(rng.integers(3, 14))) if i % 2 == 0 else ("ID"[int(rng.integers(0, 2))], int(rng.integers(1, 4)))
               for i in range(n_ops)]
        if ends == "clipped":
            ops = [("S", 7)] + ops + [("S", 9)]
        elif ends == "inner_clip" and k % 2:
            ops.insert(len(ops) // 2, ("S", 5))
        elif ends == "lead_del":
            ops = [("D", 2)] + ops
        elif ends == "lead_ins":
            ops = [("I", 3)] + ops
        reads.append(read_of_ops(ref, int(rng.integers(600, 1400)), ops, rng))
    b = pack_reads(reads)
    cfg = default_config(longread=1, flank=0)
    want = O.run_region(cfg, ref.encode(), 1, len(ref), [b], name="ctg", set_types=[BAM_TYPES["nanopore"]])
    assert want["status"] == 0
    ctx = Context(cfg, device=0)
    try:
        ctx.ref_upload(0, "ctg", ref)
        for rid in (ctx.readset_upload(0, b, bam_type="nanopore"), ctx.readset_upload_many([(0, b, "nanopore")])[0]):
            pile, calls, stats = ctx.batch_run([(0, 1, len(ref), rid)], window=256, block=256, persistent=1)
            assert_same_region(pile, calls, want, f"{n_ops} ops, {ends}")
            assert_same_stats(stats[0], want["stats"], f"{n_ops} ops, {ends}")
    finally:
        ctx.close()
