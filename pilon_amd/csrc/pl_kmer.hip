// pl_kmer.hip — the host side of the assembler's K-mer graph (included at
// the end of pl_engine.hip): the reads go to the device, the occurrences
// are emitted and grouped by K-mer (an LSD radix sort by some bits of a
// 64-bit hash of the K-mer; should two distinct K-mers share them, stable
// sorts by the K-mer's own words, last word first), summed and called per
// K-mer, and the kept K-mers put in byte order and written as text, by the
// k_kmer_* kernels.

namespace {

// bits of x's binary form
int bits_of(int64_t x) {
  int b = 0;
  for (; x; x >>= 1) b++;
  return b;
}

pl_status kmer_graph(pl_ctx* c, const pl_read_soa* R, int32_t K, int32_t min_depth, char** kmers, uint8_t** next,
                     uint8_t** alt, int64_t* n_out, double* device_ms) {
  *kmers = nullptr; *next = nullptr; *alt = nullptr; *n_out = 0;
  if (K < 1 || K > 8 * PL_KMER_WORDS) return fail(PL_E_INVAL, "K = %d outside [1, %d]", K, 8 * PL_KMER_WORDS);
  const int64_t n = R->n_reads;
  if (n < 0 || (n > 0 && (!R->seq_off || !R->bases2 || !R->quals || !R->flag || !R->mapq)))
    return fail(PL_E_INVAL, "incomplete read batch");
  // occurrences per read (both strands of every offset 0 .. L-K-1), the
  // nibble offset of each non-ACGT read, and the stream sizes
  std::vector<int64_t> occ((size_t)n + 1, 0), exo((size_t)n, -1);
  int64_t nreads = 0, nib_bytes = 1, longest = 0;
  for (int64_t i = 0; i < n; i++) {
    const int64_t L = R->seq_off[i + 1] - R->seq_off[i];
    occ[(size_t)i + 1] = occ[(size_t)i] + (L > K ? 2 * (L - K) : 0);
    if (L > K) nreads++;
    longest = std::max(longest, L);
  }
  for (int64_t k = 0; k < R->n_exotic; k++) {
    const int64_t r = R->exo_read[k];
    if (r < 0 || r >= n) return fail(PL_E_INVAL, "exotic read index %lld outside the batch", (long long)r);
    exo[(size_t)r] = R->exo_off[k];
    const int64_t L = R->seq_off[r + 1] - R->seq_off[r];
    nib_bytes = std::max<int64_t>(nib_bytes, (R->exo_off[k] + L + 1) / 2);
  }
  if (nreads >= 100000)
    return fail(PL_E_INVAL, "%lld reads longer than K: Assembler.addRead would prune its map at 100,000",
                (long long)nreads);
  const int64_t N = occ[(size_t)n];
  if (N >= ((int64_t)1 << 31)) return fail(PL_E_INVAL, "too many K-mer occurrences (%lld)", (long long)N);
  if (N == 0) return PL_OK;
  const int64_t S = R->seq_off[n];
  HIPCHK(hipSetDevice(c->device));
  Lane* L = &c->main;
  hipStream_t st = L->stream;
  ScratchBufs B(L);
  KmerArgs A;
  std::memset(&A, 0, sizeof A);
  A.n_reads = n;
  A.n_occ = (uint32_t)N;
  A.K = K;
  A.words = (K + 7) / 8;
  A.default_qual = c->pc.default_qual;
  A.min_qual = c->pc.min_qual;
  A.min_depth = min_depth;
  int64_t *dso, *dexo, *docc;
  uint8_t *db2, *dmq, *dnib;
  int8_t* dq;
  uint16_t* dfl;
  pl_status s;
  if ((s = B.get(&dso, 8 * ((size_t)n + 1))) || (s = B.get(&db2, (size_t)(S + 3) / 4 + 8)) ||
      (s = B.get(&dq, (size_t)S + 8)) || (s = B.get(&dfl, 2 * (size_t)n)) || (s = B.get(&dmq, (size_t)n)) ||
      (s = B.get(&dexo, 8 * (size_t)n)) || (s = B.get(&dnib, (size_t)nib_bytes)) || (s = B.get(&docc, 8 * ((size_t)n + 1))))
    return s;
  HIPCHK(hipMemcpyAsync(dso, R->seq_off, 8 * ((size_t)n + 1), hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(db2, R->bases2, (size_t)(S + 3) / 4, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(dq, R->quals, (size_t)S, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(dfl, R->flag, 2 * (size_t)n, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(dmq, R->mapq, (size_t)n, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(dexo, exo.data(), 8 * (size_t)n, hipMemcpyHostToDevice, st));
  if (R->n_exotic) HIPCHK(hipMemcpyAsync(dnib, R->nib, (size_t)nib_bytes, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(docc, occ.data(), 8 * ((size_t)n + 1), hipMemcpyHostToDevice, st));
  A.seq_off = dso; A.bases2 = db2; A.quals = dq; A.flag = dfl; A.mapq = dmq; A.exo_of = dexo; A.nib = dnib;
  A.occ_off = docc;
  const uint32_t nocc = (uint32_t)N;
  // Hash bits the order is by: twice those of N, so that of N distinct
  // K-mers two share them in about half the calls at worst and, of the third
  // or less that are distinct in reads with errors, in a few of a hundred.
  // At least 32: the low word is compared whole, so a shorter order would cut
  // the run of a K-mer wherever another shares its bits.
  const int bits = std::min(64, std::max(32, (2 * bits_of(N) + 7) / 8 * 8));
  A.hmask = bits >= 64 ? ~0u : (1u << (bits - 32)) - 1u;
  A.cap = (uint32_t)(N / std::max(min_depth, 1)) + 1;
  SortRecs a, b;
  uint32_t* counts;                                          // list_n, out_n, flags[2]
  if ((s = B.get(&A.kw, 4 * (size_t)PL_KMER_STRIDE * (size_t)N)) || (s = B.get(&a.lo, 4 * (size_t)N)) || (s = B.get(&a.hi, 4 * (size_t)N)) || (s = B.get(&a.v, 4 * (size_t)N)) ||
      (s = B.get(&b.lo, 4 * (size_t)N)) || (s = B.get(&b.hi, 4 * (size_t)N)) || (s = B.get(&b.v, 4 * (size_t)N)) ||
      (s = B.get(&A.list, 4 * (size_t)A.cap)) || (s = B.get(&counts, 16)) ||
      (s = B.get(&A.out_kw, 4 * (size_t)A.words * (size_t)A.cap)) || (s = B.get(&A.out_next, (size_t)A.cap)) ||
      (s = B.get(&A.out_alt, (size_t)A.cap)))
    return s;
  A.list_n = counts;
  A.out_n = counts + 1;
  A.flags = counts + 2;
  EventPair ev;
  HIPCHK(ev.create());
  HIPCHK(hipEventRecord(ev.e0, st));
  const unsigned gb = (unsigned)((N + 255) / 256);
  A.hlo = a.lo; A.hhi = a.hi; A.perm = a.v;
  if (longest <= PL_KMER_WAVE_BASES) k_kmer_emit<true><<<dim3((unsigned)((n + 3) / 4)), dim3(256), 0, st>>>(A);
  else k_kmer_emit<false><<<dim3((unsigned)n), dim3(256), 0, st>>>(A);
  HIPCHK(hipGetLastError());
  if ((s = radix_sort(L, a, b, nocc, bits))) return s;
  // m records in word order (src[w] + record * stride: word w), last word first
  auto sort_by_words = [&](uint32_t* const* src, uint32_t stride, uint32_t m) -> pl_status {
    const unsigned g = (m + 255) / 256;
    k_iota<<<dim3(std::min<unsigned>(g, 4096)), dim3(256), 0, st>>>(a.v, (int32_t)m, counts);
    for (int w = A.words - 1; w >= 0; w--) {
      k_kmer_gather<<<dim3(g), dim3(256), 0, st>>>(src[w], stride, a.v, m, a.lo);
      if (pl_status e = radix_sort(L, a, b, m, 32)) return e;
    }
    return PL_OK;
  };
  uint32_t hc[4] = {0, 0, 0, 0};
  auto counted = [&]() -> pl_status {
    HIPCHK(hipMemcpyAsync(hc, counts, 16, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    return PL_OK;
  };
  // PILON_HIP_KMER_WORD_SORT in the environment takes the word order without
  // a collision (tests compare it with the hash order's graph)
  bool by_words = std::getenv("PILON_HIP_KMER_WORD_SORT") != nullptr;
  for (;; by_words = true) {
    if (by_words) {
      uint32_t* src[PL_KMER_WORDS];
      uint32_t *head, *seg;
      for (int w = 0; w < A.words; w++) src[w] = A.kw + w;
      if ((s = B.get(&head, 4 * (size_t)N)) || (s = B.get(&seg, 4 * ((size_t)N + 1)))) return s;
      if ((s = sort_by_words(src, PL_KMER_STRIDE, nocc))) return s;
      A.hlo = a.lo; A.hhi = a.hi; A.perm = a.v;
      k_kmer_heads<<<dim3(gb), dim3(256), 0, st>>>(A, head);
      if ((s = scan_u32(L, head, seg, N))) return s;
      k_kmer_number<<<dim3(gb), dim3(256), 0, st>>>(A, head, seg);
    }
    A.hlo = a.lo; A.hhi = a.hi; A.perm = a.v;
    HIPCHK(hipMemsetAsync(counts, 0, 16, st));
    k_kmer_list<<<dim3((unsigned)((N + 256 * PL_KMER_LIST_PER - 1) / (256 * PL_KMER_LIST_PER))), dim3(256), 0, st>>>(A);
    HIPCHK(hipGetLastError());
    if ((s = counted())) return s;
    if (hc[0]) k_kmer_call<<<dim3((unsigned)(((int64_t)hc[0] * 16 + 255) / 256)), dim3(256), 0, st>>>(A);
    HIPCHK(hipGetLastError());
    if ((s = counted())) return s;
    if (!hc[2] || by_words) break;                            // else two K-mers share the hash bits
  }
  const uint32_t nk = hc[1];
  uint8_t* dtext = nullptr;
  const size_t tb = ((size_t)K * nk + 255) & ~(size_t)255, nb = ((size_t)nk + 255) & ~(size_t)255;
  if (nk) {
    const unsigned gk = (nk + 255) / 256;
    if (nk <= PL_KMER_RANK_MAX) {
      HIPCHK(hipMemsetAsync(a.lo, 0, 4 * (size_t)nk, st));
      k_kmer_rank<<<dim3(gk, (nk + PL_KMER_RANK_TILE - 1) / PL_KMER_RANK_TILE), dim3(256), 0, st>>>(A, nk, a.lo);
      k_kmer_place<<<dim3(gk), dim3(256), 0, st>>>(a.lo, nk, a.v);
    } else {
      k_kmer_keys<<<dim3(gk), dim3(256), 0, st>>>(A, nk, a.lo, a.hi, a.v);
      if ((s = radix_sort(L, a, b, nk, 64))) return s;
      if (A.words > 2) {
        k_kmer_ties<<<dim3(gk), dim3(256), 0, st>>>(A, nk, a.lo, a.hi, a.v);
        HIPCHK(hipGetLastError());
        if ((s = counted())) return s;
        if (hc[3]) {
          uint32_t* src[PL_KMER_WORDS];
          for (int w = 0; w < A.words; w++) src[w] = A.out_kw + (size_t)w * A.cap;
          if ((s = sort_by_words(src, 1, nk))) return s;
        }
      }
    }
    HIPCHK(hipGetLastError());
    if ((s = B.get(&dtext, tb + 2 * nb))) return s;
    const size_t threads = std::max<size_t>(((size_t)K * nk + 3) / 4, nk);
    k_kmer_text<<<dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st>>>(A, nk, a.v, dtext, dtext + tb,
                                                                              dtext + tb + nb);
    HIPCHK(hipGetLastError());
  }
  HIPCHK(hipEventRecord(ev.e1, st));
  char* ko = (char*)malloc((size_t)K * nk + 1);
  uint8_t* no = (uint8_t*)malloc((size_t)nk + 1);
  uint8_t* ao = (uint8_t*)malloc((size_t)nk + 1);
  s = ko && no && ao ? PL_OK : fail(PL_E_OOM, "host allocation failed");
  if (!s && nk && !(s = copy_to_host(L, ko, dtext, (size_t)K * nk)) && !(s = copy_to_host(L, no, dtext + tb, nk)))
    s = copy_to_host(L, ao, dtext + tb + nb, nk);
  float t = 0.f;
  if (!s && (hipEventSynchronize(ev.e1) != hipSuccess || hipEventElapsedTime(&t, ev.e0, ev.e1) != hipSuccess))
    s = fail(PL_E_DEVICE, "K-mer graph events");
  if (s) { free(ko); free(no); free(ao); return s; }
  *kmers = ko; *next = no; *alt = ao; *n_out = nk;
  if (device_ms) *device_ms = t;
  return PL_OK;
}

}  // namespace

extern "C" {

pl_status pl_kmer_graph(pl_ctx* c, const pl_read_soa* reads, int32_t K, int32_t min_depth, char** kmers,
                        uint8_t** next, uint8_t** alt, int64_t* n, double* device_ms) {
  if (!c || !reads || !kmers || !next || !alt || !n) return fail(PL_E_INVAL, "null argument");
  return kmer_graph(c, reads, K, min_depth, kmers, next, alt, n, device_ms);
}

}  // extern "C"
