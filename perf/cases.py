"""The work a user of this library has it do, as cases to measure.

A case names a form of the library (a region polished on its own, a batch of
whole contigs, a request stream, the VCF, tracks or K-mer graph passes) and
the size and kind of its data: contig lengths, depth, read length, how the
reads differ from the draft.  Everything goes through include/pilon_hip.h, by
pilon_amd.engine's classes or, where a host program takes the library's
arrays as they are (batch statistics, K-mers), by its ctypes binding; reads
come from the package's seeded generator.  Every result is a whole number or
a byte, so outputs compare exactly.  Texts come back in arrays of a size that
depends on the case alone, zero past their end.
"""
import ctypes as C
import math

import numpy as np

from pilon_amd import engine
from pilon_amd.abi import PlBatchOpts, PlRegionStats, default_config
from pilon_amd.engine import Context, PileUpRegion, Server
from pilon_amd.reads import ReadBatch
from pilon_amd.synth import SynthData, lognormal_lengths, serve_requests

# How reads differ from the draft, after the benchmark's configurations: a
# clean small genome; a GC-rich one with MAPQ-0 repeats; a many-contig
# assembly; a diploid with 250-base reads, deep hotspots and clipped
# breakpoints; long reads with frequent indels.
PROFILES = {
    "clean": dict(gc=0.5, read_len=150, insert_mean=400, insert_sd=40, sub_rate=0.003, snv_rate=0.002,
                  indel_rate=0.0002, indel_max=10),
    "repeats": dict(gc=0.65, read_len=150, insert_mean=400, insert_sd=40, sub_rate=0.005, err_indel_rate=0.0002,
                    err_indel_max=3, clip_frac=1 / 200, clip_min=10, clip_max=60, improper_frac=0.01,
                    snv_rate=0.0001, indel_rate=0.00002, indel_max=10, repeat_copies=10, repeat_len=2000),
    "contigs": dict(gc=0.5, read_len=150, insert_mean=350, insert_sd=35, sub_rate=0.005, err_indel_rate=0.0002,
                    err_indel_max=3, clip_frac=1 / 200, clip_min=10, clip_max=60, improper_frac=0.01,
                    snv_rate=0.0001, indel_rate=0.00002, indel_max=10),
    "diploid": dict(gc=0.5, read_len=250, insert_mean=500, insert_sd=50, sub_rate=0.005, err_indel_rate=0.0002,
                    err_indel_max=3, improper_frac=0.01, snv_rate=0.0001, indel_rate=0.00002, indel_max=10,
                    het_rate=0.001, n_hotspots=1, hotspot_len=2000, hotspot_cov=2000, n_breakpoints=50,
                    bp_clip_frac=1.0, bp_clip_min=30, bp_clip_max=200),
    "nanopore": dict(gc=0.5, sub_rate=0.02, err_indel_rate=0.03, err_indel_max=3, snv_rate=0.001,
                     indel_rate=0.0002, indel_max=10, qual_lo=5, qual_hi=25),
}


def listed():
    return [
        # One short region of a resident contig: the latency of a single call.
        {"name": "region-2kb", "kind": "region", "profile": "clean", "genome": 100_000, "contigs": 1, "depth": 40,
         "size": 2_000},
        # One BAM region as Pilon's own loop has it: reads handed over from
        # the host, piled, fixed.
        {"name": "host-region-100kb", "kind": "host_region", "profile": "clean", "genome": 100_000, "contigs": 1,
         "depth": 40},
        # Contigs polished in one call whose pileup the caller reads back.
        {"name": "batch-copy-200kb", "kind": "batch", "profile": "contigs", "genome": 200_000, "contigs": 11,
         "depth": 60, "copy": True, "graph": False, "tuned": False},
        # The benchmark's form: a many-contig assembly resident on the
        # device, repeated through a captured graph at the tuned shape.
        {"name": "batch-24mb", "kind": "batch", "profile": "contigs", "genome": 24_000_000, "contigs": 1_201,
         "depth": 60, "copy": False, "graph": True, "tuned": True},
        # A bacterial chromosome's worth at high depth, with repeats.
        {"name": "batch-deep-2mb", "kind": "batch", "profile": "repeats", "genome": 2_000_003, "contigs": 1,
         "depth": 100, "copy": False, "graph": False, "tuned": False},
        # A diploid draft, 250-base reads, a 2,000x hotspot.
        {"name": "batch-diploid-2mb", "kind": "batch", "profile": "diploid", "genome": 2_000_000, "contigs": 2,
         "depth": 80, "copy": False, "graph": False, "tuned": False},
        # A long-read BAM (--nanopore).
        {"name": "nanopore-400kb", "kind": "nanopore", "profile": "nanopore", "genome": 400_000, "contigs": 2,
         "depth": 40, "read_len": 6_001},
        # A request stream over resident contigs, changes and fixed bases
        # fetched for each request.
        {"name": "serve-96", "kind": "serve", "profile": "contigs", "genome": 2_000_000, "contigs": 4, "depth": 50,
         "requests": 96, "lanes": 4},
        # The whole-genome VCF of a finished batch, streamed to the caller.
        {"name": "vcf-400kb", "kind": "vcf", "profile": "contigs", "genome": 400_000, "contigs": 21, "depth": 60},
        # The 13 tracks and Pilon.bed of a finished batch.
        {"name": "tracks-500kb", "kind": "tracks", "profile": "contigs", "genome": 500_000, "contigs": 25,
         "depth": 60},
        # The assembler's K-mer graph of one break's recruited reads ...
        {"name": "kmer-1500", "kind": "kmer", "profile": "contigs", "genome": 3_751, "contigs": 1, "depth": 60,
         "k": 47},
        # ... and of a large recruitment.
        {"name": "kmer-60000", "kind": "kmer", "profile": "contigs", "genome": 150_000, "contigs": 1, "depth": 60,
         "k": 47},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["region", "host_region", "batch", "batch", "batch", "nanopore", "serve", "vcf", "tracks", "kmer"])
    depth = rng.randint(20, 100)
    c = {"kind": kind, "contigs": 1, "depth": depth}
    if kind == "region":
        c.update(profile="clean", genome=_log_int(rng, 60_000, 400_000), size=_log_int(rng, 500, 50_000))
    elif kind == "host_region":
        c.update(profile="clean", genome=_log_int(rng, 5_000, 150_000), depth=rng.randint(20, 60))
    elif kind == "batch":
        p = rng.choice(["contigs", "contigs", "repeats", "diploid"])
        copy = rng.random() < 0.2
        n = _log_int(rng, 50_000, 400_000) if copy else _log_int(rng, 100_000, 24_000_000 if p == "contigs" else 2_000_000)
        graph = not copy and rng.random() < 0.4
        c.update(profile=p, genome=n, contigs=max(1, n // 20_000 + rng.randint(-2, 2)) if p == "contigs" else rng.randint(1, 3),
                 copy=copy, graph=graph, tuned=graph)
        if p == "contigs":
            c["depth"] = rng.randint(30, 60)
    elif kind == "nanopore":
        c.update(profile="nanopore", genome=_log_int(rng, 60_000, 400_000), contigs=rng.randint(1, 3),
                 depth=rng.randint(15, 50), read_len=_log_int(rng, 1_500, 12_000))
    elif kind == "serve":
        c.update(profile="contigs", genome=_log_int(rng, 400_000, 2_000_000), contigs=rng.randint(1, 5),
                 depth=rng.randint(30, 60), requests=_log_int(rng, 8, 96), lanes=rng.choice([1, 2, 4]))
    elif kind == "vcf":
        c.update(profile="contigs", genome=_log_int(rng, 30_000, 400_000), contigs=rng.randint(1, 20))
    elif kind == "tracks":
        c.update(profile="contigs", genome=_log_int(rng, 30_000, 500_000), contigs=rng.randint(1, 20))
    else:
        c.update(profile="contigs", genome=_log_int(rng, 2_001, 150_000), depth=rng.randint(20, 60),
                 k=rng.choice([31, 47]))
    return c


def _lengths(case):
    n, g = case["contigs"], case["genome"]
    if n >= 10:      # a draft assembly's contigs: log-normal, a few large
        return [int(x) for x in lognormal_lengths(n, 8000, 1.35, 1000, 2_000_000, g, 1003)]
    return [g // n + (1 if i < g % n else 0) for i in range(n)]


def _serve_most(case):
    """The longest request: at most 200 kb, and a contig."""
    return min(200_000, case["genome"] // case["contigs"])


def _data(case, seed):
    p = dict(PROFILES[case["profile"]], seed=seed + 1, lens=_lengths(case), coverage=case["depth"])
    if "read_len" in case:
        p.update(read_len=case["read_len"], insert_mean=case["read_len"], insert_sd=0)
    return SynthData(p)


def _unpaired(b):
    """The batch's reads as a long-read BAM has them: no mates."""
    return ReadBatch(b.pos, np.zeros_like(b.tlen), b.flag & 0xA010, b.mapq, b.cigar_off, b.cigar, b.seq_off, b.bases2,
                     b.quals, b.exo_read, b.exo_off, b.nib)


def _resident(case, data, cfg, bam_type="frags"):
    """A context holding the data's contigs and reads, and their whole-contig regions."""
    ctx = Context(cfg, device=0)
    lens = []
    for i in range(data.n):
        d = data.draft(i)
        lens.append(len(d))
        ctx.ref_upload(i, data.names[i], d)
    reads = [_unpaired(data.batch(i)) if bam_type == "nanopore" else data.soa(i) for i in range(data.n)]
    ids = ctx.readset_upload_many([(i, reads[i], bam_type) for i in range(data.n)])
    return ctx, ids, [(i, 1, lens[i], ids[i]) for i in range(data.n)]


def prepare(case, seed):
    data = _data(case, seed)
    kind = case["kind"]
    cfg = default_config(longread=1) if kind == "nanopore" else default_config()
    if kind == "host_region":
        ctx = Context(cfg, device=0)
        draft = data.draft(0)
        ctx.ref_upload(0, data.names[0], draft)
        return {"case": case, "ctx": ctx, "reads": data.batch(0), "size": len(draft)}
    if kind == "kmer":
        return {"case": case, "ctx": Context(cfg, device=0), "reads": data.batch(0)}
    ctx, ids, regions = _resident(case, data, cfg, "nanopore" if kind == "nanopore" else "frags")
    s = {"case": case, "ctx": ctx, "regions": regions}
    if kind == "region":
        # a start clear of the planted indels: Pilon throws where one is
        # normalised to before its region
        pos, op, _ = data.variants(0)
        start = 1_000 + seed % (case["genome"] - case["size"] - 5_000)
        while np.any((op != 0) & (np.abs(pos - start) < 60)):
            start += 61
        s.update(start=start, stop=start + case["size"] - 1, set=ids[0])
    elif kind == "serve":
        s["requests"] = [(c, a, b, ids[c])
                         for c, a, b in serve_requests(data, case["requests"], 2_000, _serve_most(case), seed=seed)]
        s["server"] = Server(ctx, lanes=case["lanes"], max_batch=64, mem_budget=2 << 30, keep_fix=True)
    elif kind in ("vcf", "tracks"):
        ctx.batch_run(regions, window=512, block=256, persistent=1, copy_out=False, want_stats=False)
    if kind in ("batch", "nanopore"):
        s["descs"] = ctx.batch_descs(regions)
    return s


def _text(b, cap):
    """The bytes b at the front of cap bytes."""
    b = b.encode() if isinstance(b, str) else b
    if len(b) > cap:
        raise ValueError("%d bytes of output, room for %d" % (len(b), cap))
    out = np.zeros(cap, np.uint8)
    out[:len(b)] = np.frombuffer(b, np.uint8)
    return out


def _changes_cap(loci):
    """Room for the .changes lines of this many loci: one line of up to about
    60 bytes per planted or miscalled variant, at most one in 100 loci."""
    return 65_536 + loci


def _region(reg):
    reg.postProcess()
    changes, bases = reg.fix()
    out = {"pile": reg.pile, "calls": reg.calls.view(np.int64), "stats": np.array(list(reg.stats.values()), np.int64),
           "changes": _text(changes, _changes_cap(reg.size)), "bases": _text(bases, reg.size + 10_000)}
    reg.close()
    return out


STATS = np.dtype([(f, np.int64 if t is C.c_int64 else np.int32) for f, t in PlRegionStats._fields_], align=True)


def _batch(s, graph=False, tuned=False, copy=False):
    ctx, descs, n = s["ctx"], s["descs"], len(s["regions"])
    G = sum(e - b + 1 for _, b, e, _ in s["regions"])
    opts = PlBatchOpts(window=0 if tuned else 512, block=0 if tuned else 256, persistent=1, use_graph=int(graph),
                       copy_out=int(copy))
    stats = np.zeros(n, STATS)
    pile = np.zeros((engine.NFIELDS, G), np.int32) if copy else None
    calls = np.zeros(G, np.int64) if copy else None
    status = engine.lib().pl_batch_run(ctx.h, descs, n, C.byref(opts), pile.ctypes.data if copy else None,
                                       calls.ctypes.data if copy else None, stats.ctypes.data)
    if status:
        raise RuntimeError(engine.lib().pl_last_error().decode())
    changes, _ = ctx.batch_fix(want_fasta=False)
    out = {"changes": _text(changes, _changes_cap(G)), **{f: stats[f] for f in STATS.names}}
    if copy:
        out.update(pile=pile, calls=calls)
    return out


def _serve(s):
    srv, case = s["server"], s["case"]
    order = {srv.submit(*r): k for k, r in enumerate(s["requests"])}
    srv.drain()
    res = sorted(srv.poll(max_n=4096), key=lambda r: order[r["ticket"]])
    changes, bases = [], []
    for r in res:
        if r["status"] == 0:
            c, b = srv.fetch_fix(r["ticket"])
            changes.append(c)
            bases.append(b)
    loci = case["requests"] * _serve_most(case)
    return {"status": np.array([r["status"] for r in res], np.int32),
            "stats": np.array([list(r["stats"].values()) for r in res], np.int64),
            "changes": _text("".join(changes), _changes_cap(loci)), "bases": _text(b"".join(bases), loci + 65_536)}


def _kmer(s):
    L, soa = engine.lib(), s["reads"].soa()
    ks, nx, al = C.c_void_p(), C.c_void_p(), C.c_void_p()
    n, ms = C.c_int64(), C.c_double()
    K = s["case"]["k"]
    status = L.pl_kmer_graph(s["ctx"].h, C.byref(soa), K, 5, C.byref(ks), C.byref(nx), C.byref(al), C.byref(n),
                             C.byref(ms))
    if status:
        raise RuntimeError(L.pl_last_error().decode())
    cap = 4 * s["case"]["genome"] + 4096
    out = {"n": n.value, "kmers": _text(C.string_at(ks, K * n.value), K * cap),
           "next": _text(C.string_at(nx, n.value), cap), "alt": _text(C.string_at(al, n.value), cap)}
    for p in (ks, nx, al):
        L.pl_free(p)
    return out


def _vcf(s):
    text = np.zeros(200 * s["case"]["genome"] + 65_536, np.uint8)
    at = 0

    def write(data, n):
        nonlocal at
        C.memmove(text.ctypes.data + at, data, n)
        at += n

    n, _ = s["ctx"].batch_vcf_stream(write, raw=True)
    return {"n": n, "vcf": text}


def _tracks(s):
    values, _ = s["ctx"].batch_tracks()
    bed, _ = s["ctx"].batch_bed()
    return {"values": values, "bed": _text(bed, 65_536 + s["case"]["genome"])}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "region":
        reg = PileUpRegion(state["ctx"], 0, state["start"], state["stop"])
        reg.useReadSet(state["set"])
        return _region(reg)
    if kind == "host_region":
        reg = PileUpRegion(state["ctx"], 0, 1, state["size"])
        reg.addReads(state["reads"])
        return _region(reg)
    if kind == "batch":
        return _batch(state, case["graph"], case["tuned"], case["copy"])
    if kind == "nanopore":
        return _batch(state)
    return {"serve": _serve, "vcf": _vcf, "tracks": _tracks, "kmer": _kmer}[kind](state)


def work(case):
    """Bytes one pass cannot do without: per read its 16-byte header, a CIGAR
    word (one per indel too for long reads), 2-bit bases and qualities; per
    position 18 counters, the call and the reference; per formatted locus its
    text."""
    kind, g = case["kind"], case["genome"]
    L = case.get("read_len") or PROFILES[case["profile"]]["read_len"]
    ops = 1 + 2 * L * PROFILES[case["profile"]].get("err_indel_rate", 0)
    per_base = (16 + 4 * ops) / L + 1.25

    def pile(n):
        return n * (80.25 + case["depth"] * per_base)

    if kind == "region":
        n = pile(case["size"])
    elif kind == "serve":
        hi = _serve_most(case)
        n = pile(case["requests"] * (hi - 2_000) / math.log(hi / 2_000))
    elif kind == "vcf":          # 14 counters and the call in, about 125 bytes of text out
        n = g * (64 + 125)
    elif kind == "tracks":       # 14 counters, the call and a GC value in, 13 values and an issue byte out
        n = g * (65 + 53)
    elif kind == "kmer":         # reads in, K-mers with their two edges out (about twice the genome's loci)
        n = g * case["depth"] * 1.25 + 2 * g * (case["k"] + 2)
    else:
        n = pile(g)
        if case["profile"] == "diploid":
            n += case["contigs"] * 4_000_000 * per_base
    return {"bytes": float(n), "flops": 0.0}


def tolerance(case):
    return "exact"
