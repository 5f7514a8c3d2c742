"""The K-mer graph's byte order and grouping on the device against the
oracle's: counts of kept K-mers about the limit of the counted order (8,192)
and above it, K-mers that agree in their first 16 bases (a handful, and more
than one thread orders), codes other than A, C, G, T among them; K-mers whose
hashes agree in their low bits, in batches of few occurrences."""
import numpy as np
import pytest

from pilon_amd.abi import default_config
from pilon_amd.reads import pack_reads

pytestmark = pytest.mark.gpu


def reads_of(kind, n, K, rng):
    """Reads of K + 1 bases, each K-mer in `depth` of them."""
    out = []
    for i in range(n):
        seq = "".join(rng.choice(list("ACGT"), K + 1))
        if kind == "prefix":                     # 8 to a 16-base prefix
            seq = "".join("ACGT"[(i // 8 >> (2 * b)) & 3] for b in range(16)) + seq[16:]
        elif kind == "one_prefix":
            seq = "ACGTTGCATTGACCAG" + seq[16:]
        elif kind == "codes" and i % 3 == 0:
            seq = seq[:K // 2] + "RYMN"[i % 4] + seq[K // 2 + 1:]
        out.append(seq)
    return out


@pytest.mark.parametrize("kind,n,K", [("plain", 4095, 47), ("plain", 4097, 47), ("plain", 9000, 16), ("plain", 300, 7),
                                      ("prefix", 6000, 47), ("one_prefix", 200, 47), ("one_prefix", 5000, 33),
                                      ("codes", 3000, 48), ("codes", 5000, 31)])
def test_kmer_byte_order(kind, n, K):
    from oracle import oracle as O
    from pilon_amd.engine import Context
    print(f"case: kmer order {kind} n={n} K={K}", flush=True)
    rng = np.random.default_rng(n + K)
    depth = 3
    reads = []
    for seq in reads_of(kind, n, K, rng):
        for _ in range(depth):
            reads.append(dict(pos=1, cigar=f"{K + 1}M", seq=seq, qual=[int(x) for x in rng.integers(2, 41, K + 1)],
                              mapq=int(rng.integers(0, 61))))
    b = pack_reads(reads, sort=False)
    cfg = default_config()
    ctx = Context(cfg, device=0)
    try:
        for min_depth in (depth, 1):
            got, _ = ctx.kmer_graph(b, K=K, min_depth=min_depth)
            st, ref = O.kmer_graph(cfg, b, K=K, min_depth=min_depth)
            assert st == 0 and len(ref) >= min(n, 200)
            assert got == ref
    finally:
        ctx.close()


@pytest.mark.parametrize("occ", [1, 1024, 1025, 131_072, 131_073, 524_288, 524_289])
def test_kmer_sort_sizes(occ):
    """Occurrences, all of different K-mers, that just fill the tiles of each
    form of the radix sort, and one more."""
    from oracle import oracle as O
    from pilon_amd.engine import Context
    print(f"case: kmer sort of {occ} occurrences", flush=True)
    K, per = 24, 256
    rng = np.random.default_rng(occ)
    lens = [per] * (occ // per) + ([occ % per] if occ % per else [])
    b = pack_reads([dict(pos=1, cigar=f"{n + K}M", seq="".join(np.array(list("ACGT"))[rng.integers(0, 4, n + K)]),
                         qual=[30] * (n + K), mapq=40) for n in lens], sort=False)
    cfg = default_config()
    ctx = Context(cfg, device=0)
    try:
        got, _ = ctx.kmer_graph(b, K=K, min_depth=1)
    finally:
        ctx.close()
    st, ref = O.kmer_graph(cfg, b, K=K, min_depth=1)
    assert st == 0 and len(ref) > occ // 2
    assert got == ref


def words_hash(codes):
    """kmer_hash of K-mers given as [n, K] base indices: the 64-bit key the
    occurrences are grouped by."""
    n, K = codes.shape
    words = (K + 7) // 8
    nib = np.zeros((n, 8 * words), np.uint64)
    nib[:, :K] = 1 << codes.astype(np.uint64)
    h = np.full(n, np.uint64((0x9e3779b97f4a7c15 * (words + 1)) & (2 ** 64 - 1)))
    with np.errstate(over="ignore"):
        for w in range(words):
            x = np.zeros(n, np.uint64)
            for j in range(8):
                x = (x << np.uint64(4)) | nib[:, 8 * w + j]
            h = (h ^ x) * np.uint64(0xff51afd7ed558ccd)
            h ^= h >> np.uint64(33)
        h *= np.uint64(0xc4ceb9fe1a85ec53)
        return h ^ (h >> np.uint64(29))


def sharing_pair(bits, K, rng):
    """Two K-mers whose hashes agree in their low `bits` bits and differ above."""
    seen = {}
    while True:
        codes = rng.integers(0, 4, (4096, K))
        for c, h in zip(codes, words_hash(codes)):
            low = int(h) & ((1 << bits) - 1)
            if low in seen and seen[low][1] != int(h):
                return seen[low][0], c
            seen[low] = (c, int(h))


@pytest.mark.parametrize("bits,depth,fill", [(8, 3, 0), (16, 5, 0), (16, 5, 100), (24, 5, 200), (24, 9, 2000), (32, 5, 1000)])
def test_kmer_shared_hash_bits(bits, depth, fill):
    """Two K-mers that share the low bits of their hashes, in alternate reads
    of a batch of 12 to 4,018 occurrences: each is found with all of its
    occurrences."""
    from oracle import oracle as O
    from pilon_amd.engine import Context
    print(f"case: K-mers sharing {bits} hash bits, {2 * (2 * depth + fill)} occurrences", flush=True)
    K = 23
    rng = np.random.default_rng(bits + fill)
    pair = sharing_pair(bits, K, rng)
    seqs = []
    for _ in range(depth):
        for c in pair:
            seqs.append("".join("ACGT"[x] for x in c) + "ACGT"[int(rng.integers(0, 4))])
    seqs += ["".join("ACGT"[x] for x in rng.integers(0, 4, K + 1)) for _ in range(fill)]
    b = pack_reads([dict(pos=1, cigar=f"{K + 1}M", seq=s, qual=[30] * (K + 1)) for s in seqs], sort=False)
    cfg = default_config()
    ctx = Context(cfg, device=0)
    try:
        for min_depth in (depth, 2):
            got, _ = ctx.kmer_graph(b, K=K, min_depth=min_depth)
            st, ref = O.kmer_graph(cfg, b, K=K, min_depth=min_depth)
            assert st == 0
            assert {"".join("ACGT"[x] for x in c) for c in pair} <= {k[0] for k in ref}
            assert got == ref
    finally:
        ctx.close()
