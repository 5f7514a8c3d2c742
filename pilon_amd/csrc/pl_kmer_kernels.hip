// pl_kmer_kernels.hip — the K-mer pileups of Pilon's local assembler
// (Assembler.addReads / addToPileups / buildGraph, Assembler.scala:46-85,
// 131-153) on the device.  Included at the end of pl_kernels.hip.
//
//   k_kmer_emit   one workgroup per read, one thread per K-mer occurrence
//                 (strand, offset): the K-mer as 4-bit BAM codes packed in
//                 six 32-bit words (first base most significant), their
//                 hash, and the base after it with its quality and the
//                 read's MAPQ;
//   (an LSD radix sort of the occurrences by the low bits of a 64-bit hash
//   of the six words; by the six words themselves only if two distinct
//   K-mers share those bits)
//   k_kmer_list   the K-mers with at least minDepth occurrences;
//   k_kmer_call   16 lanes per listed K-mer: PileUp.add of its occurrences
//                 (each one's words checked against the first's) and, at
//                 depth >= minDepth, BaseCall: kGraph's base and, when not
//                 homozygous, altGraph's;
//   k_kmer_rank, k_kmer_place, or a radix sort and k_kmer_ties: the kept K-mers in byte
//                 order; k_kmer_text writes them.

#define PL_KMER_WORDS 6          // K <= 48: eight 4-bit codes per word
#define PL_KMER_STRIDE 8         // words per occurrence in kw: one 32-byte record (unused words zero)
#define PL_KMER_VAL 6            // ... whose word 6 is code | qual << 8 | mapq << 16 of the base after it

struct KmerArgs {
  int64_t n_reads;
  const int64_t* seq_off;        // [n_reads + 1]
  const uint8_t* bases2;
  const int8_t* quals;
  const uint16_t* flag;
  const uint8_t* mapq;
  const int64_t* exo_of;         // [n_reads] first nibble of a non-ACGT read, -1 otherwise
  const uint8_t* nib;
  const int64_t* occ_off;        // [n_reads + 1] first occurrence of each read
  uint32_t n_occ;
  int32_t K, words;
  int32_t default_qual, min_qual, min_depth;
  uint32_t* kw;                  // [n_occ][PL_KMER_STRIDE] each occurrence's words and value together
  uint32_t *hlo, *hhi, *perm;    // [n_occ] the K-mer's hash and the occurrence, then in K-mer order
  uint32_t hmask;                // bits of hhi the order is by
  uint32_t* list;                // first sorted occurrence of each listed K-mer
  uint32_t* list_n;
  uint32_t* flags;               // [0]: a K-mer's occurrences differ in their words; [1]: a long run of equal keys
  // the kept K-mers: their words with each code replaced by its rank in byte order
  uint32_t cap;                  // room for them (the listed ones)
  uint32_t* out_n;
  uint32_t* out_kw;              // [PL_KMER_WORDS][cap]
  uint8_t* out_next;
  uint8_t* out_alt;
};

namespace {

// 4-bit BAM code of base j of read r (getReadString)
__device__ __forceinline__ uint32_t kmer_code(const KmerArgs& A, int64_t r, int64_t j) {
  const int64_t x = A.exo_of[r];
  if (x >= 0) {
    const int64_t k = x + j;
    return (A.nib[k >> 1] >> ((k & 1) ? 0 : 4)) & 15u;
  }
  const int64_t k = A.seq_off[r] + j;
  return 1u << ((A.bases2[k >> 2] >> (2 * (k & 3))) & 3u);
}

// a 64-bit mix of the K-mer's words (a grouping key: equal words give
// equal hashes; k_kmer_call checks that equal hashes hold equal words)
__device__ __forceinline__ uint64_t kmer_hash(const uint32_t* w, int words) {
  uint64_t h = 0x9e3779b97f4a7c15ull * (uint64_t)(words + 1);
  for (int k = 0; k < words; k++) {
    h = (h ^ w[k]) * 0xff51afd7ed558ccdull;
    h ^= h >> 33;
  }
  h *= 0xc4ceb9fe1a85ec53ull;
  return h ^ (h >> 29);
}

// Bases.complement (Bases.scala:47-53): A<->T, C<->G, any other code kept
__device__ __forceinline__ uint32_t kmer_comp(uint32_t c) {
  return c == 1u ? 8u : c == 8u ? 1u : c == 2u ? 4u : c == 4u ? 2u : c;
}

__device__ __forceinline__ int32_t kmer_qual(const KmerArgs& A, int64_t r, int64_t j) {
  return (A.flag[r] & PL_RF_NO_QUAL) ? A.default_qual : (int32_t)A.quals[A.seq_off[r] + j];
}

}  // namespace

// the occurrence's outputs: its K-mer words, their hash, the next base
__device__ __forceinline__ void kmer_store(const KmerArgs& A, int64_t t, const uint32_t* w, uint32_t next,
                                           int32_t qual, uint32_t mapq) {
  uint4* rec = (uint4*)(A.kw + (int64_t)t * PL_KMER_STRIDE);
  static_assert(PL_KMER_WORDS <= PL_KMER_VAL && PL_KMER_STRIDE == 8, "two 16-byte halves per occurrence");
  uint32_t v[PL_KMER_STRIDE];
#pragma unroll
  for (int k = 0; k < PL_KMER_STRIDE; k++) v[k] = (k < PL_KMER_WORDS && k < A.words) ? w[k] : 0u;
  v[PL_KMER_VAL] = next | ((uint32_t)(uint8_t)(int8_t)qual << 8) | (mapq << 16);
  rec[0] = make_uint4(v[0], v[1], v[2], v[3]);
  rec[1] = make_uint4(v[4], v[5], v[6], v[7]);
  const uint64_t h = kmer_hash(w, A.words);
  A.hlo[t] = (uint32_t)h;
  A.hhi[t] = (uint32_t)(h >> 32) & A.hmask;
  A.perm[t] = (uint32_t)t;
}

#define PL_KMER_LDS_BASES 8192   // reads up to this long are staged in LDS
#define PL_KMER_WAVE_BASES (PL_KMER_LDS_BASES / 4)   // ... by a wave each, when all are up to this long

// One read per workgroup, or per wave (WAVE: no read of the batch is longer
// than PL_KMER_WAVE_BASES; a 150-base read is three rounds of a wave, and a
// workgroup each for 60,000 of them spent its time starting): the read's
// codes, forward and reverse-complemented, packed eight to a 32-bit word
// (first code most significant) in LDS; each occurrence's K-mer is then six
// funnel shifts of that stream.  Occurrence 2*o + rc of the read is the
// K-mer at offset o of the forward (rc = 0) or reverse-complement (rc = 1)
// sequence (Assembler.addRead, Assembler.scala:65-85).
template <bool WAVE>
__global__ void __launch_bounds__(256) k_kmer_emit(KmerArgs A) {
  constexpr int PER = WAVE ? 4 : 1, BD = 256 / PER, SPAN = PL_KMER_LDS_BASES / 8 / PER + 8;
  __shared__ uint32_t sfw[PER][SPAN], srw[PER][SPAN];
  const int sub = WAVE ? threadIdx.x >> 6 : 0, tid = WAVE ? threadIdx.x & 63 : threadIdx.x;
  uint32_t *fw = sfw[sub], *rw = srw[sub];
  const int64_t r = (int64_t)blockIdx.x * PER + sub;
  if (r >= A.n_reads) return;
  const int64_t t0 = A.occ_off[r], t1 = A.occ_off[r + 1];
  if (t1 <= t0) return;
  const int64_t L = A.seq_off[r + 1] - A.seq_off[r];
  const uint32_t mapq = A.mapq[r];
  if (!WAVE && L > PL_KMER_LDS_BASES) {
    // a long read: each occurrence reads its K + 1 codes itself
    for (int64_t t = t0 + tid; t < t1; t += BD) {
      const int64_t local = t - t0;
      const bool rc = local & 1;
      const int64_t o = local >> 1;
      uint32_t w[PL_KMER_WORDS] = {0, 0, 0, 0, 0, 0};
      for (int j = 0; j < A.K; j++) {
        const int64_t p = o + j;
        const uint32_t c = rc ? kmer_comp(kmer_code(A, r, L - 1 - p)) : kmer_code(A, r, p);
        w[j >> 3] |= c << (28 - 4 * (j & 7));
      }
      const int64_t pn = o + A.K;
      const uint32_t next = rc ? kmer_comp(kmer_code(A, r, L - 1 - pn)) : kmer_code(A, r, pn);
      const int32_t qual = rc ? kmer_qual(A, r, L - 1 - pn) : kmer_qual(A, r, pn);
      kmer_store(A, t, w, next, qual, mapq);
    }
    return;
  }
  const int nw = (int)((L + 7) / 8);
  for (int k = tid; k < nw + 8; k += BD) {
    uint32_t f = 0, b = 0;
    for (int j = 0; j < 8; j++) {
      const int64_t p = 8 * (int64_t)k + j;
      if (p < L) {
        f |= kmer_code(A, r, p) << (28 - 4 * j);
        b |= kmer_comp(kmer_code(A, r, L - 1 - p)) << (28 - 4 * j);
      }
    }
    fw[k] = f;
    rw[k] = b;
  }
  // (a wave's LDS operations complete in order)
  if constexpr (WAVE) __builtin_amdgcn_wave_barrier();
  else __syncthreads();
  const int K = A.K;
  for (int64_t t = t0 + tid; t < t1; t += BD) {
    const int64_t local = t - t0;
    const bool rc = local & 1;
    const int o = (int)(local >> 1);
    const uint32_t* sw = rc ? rw : fw;
    const int a = o >> 3, sh = 4 * (o & 7);
    uint32_t w[PL_KMER_WORDS];
#pragma unroll
    for (int k = 0; k < PL_KMER_WORDS; k++) {
      const uint32_t hi = sw[a + k], lo = sw[a + k + 1];
      w[k] = sh ? (hi << sh) | (lo >> (32 - sh)) : hi;
    }
    // codes past the K-th are zero
#pragma unroll
    for (int k = 0; k < PL_KMER_WORDS; k++) {
      const int keep = K - 8 * k;
      w[k] = keep >= 8 ? w[k] : keep <= 0 ? 0u : (w[k] & ~(0xffffffffu >> (4 * keep)));
    }
    const int pn = o + K;
    const uint32_t next = (sw[pn >> 3] >> (28 - 4 * (pn & 7))) & 15u;
    const int32_t qual = rc ? kmer_qual(A, r, L - 1 - pn) : kmer_qual(A, r, pn);
    kmer_store(A, t, w, next, qual, mapq);
  }
}

// keys[i] = word w of the i-th K-mer or occurrence in the current order
// (record r's word at src[r * stride])
__global__ void __launch_bounds__(256) k_kmer_gather(const uint32_t* src, uint32_t stride, const uint32_t* perm,
                                                     uint32_t n, uint32_t* keys) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) keys[i] = src[(int64_t)perm[i] * stride];
}

// occurrences in word order: 1 where a K-mer begins
__global__ void __launch_bounds__(256) k_kmer_heads(KmerArgs A, uint32_t* head) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= A.n_occ) return;
  const uint32_t* x = A.kw + (int64_t)A.perm[i] * PL_KMER_STRIDE;
  const uint32_t* y = A.kw + (int64_t)A.perm[i ? i - 1 : 0] * PL_KMER_STRIDE;
  uint32_t h = i == 0;
  for (int k = 0; k < A.words; k++) h |= x[k] != y[k];
  head[i] = h;
}
// ... and each K-mer's number in place of its hash
__global__ void __launch_bounds__(256) k_kmer_number(KmerArgs A, const uint32_t* head, const uint32_t* seg) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < A.n_occ) { A.hlo[i] = seg[i] + head[i]; A.hhi[i] = 0; }
}

// The K-mers with min_depth occurrences or more: only they can reach that
// depth, and in reads with errors most K-mers occur once.
#define PL_KMER_LIST_PER 8       // occurrences a thread: one atomic on the list per 2,048
__global__ void __launch_bounds__(256) k_kmer_list(KmerArgs A) {
  __shared__ uint32_t s_n, s_base;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  const uint32_t more = A.min_depth > 1 ? (uint32_t)A.min_depth - 1u : 0u;
  const uint32_t b0 = blockIdx.x * (256u * PL_KMER_LIST_PER) + threadIdx.x;
  uint32_t take = 0, at[PL_KMER_LIST_PER];
#pragma unroll
  for (int k = 0; k < PL_KMER_LIST_PER; k++) {
    const uint32_t i = b0 + 256u * k;
    bool t = false;
    if (i < A.n_occ) {
      const uint32_t lo = A.hlo[i], hi = A.hhi[i];
      const bool head = i == 0 || A.hlo[i - 1] != lo || A.hhi[i - 1] != hi;
      t = head && more < A.n_occ - i && A.hlo[i + more] == lo && A.hhi[i + more] == hi;
    }
    at[k] = wave_append(&s_n, t);
    if (t) take |= 1u << k;
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_n) s_base = atomicAdd(A.list_n, s_n);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PL_KMER_LIST_PER; k++)
    if (take >> k & 1u) A.list[s_base + at[k]] = b0 + 256u * k;
}

// a code's rank among the codes in the byte order of their letters, nibble-wise
__device__ __forceinline__ uint32_t kmer_ranks(uint32_t w) {
  // rank of code c in nibble c: = A C M G R S V T W Y H K D B N
  const uint64_t R = 0x92476fecdba58310ull;
  uint32_t r = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) r |= (uint32_t)((R >> (4 * ((w >> (4 * k)) & 15u))) & 15u) << (4 * k);
  return r;
}

// PileUp.add (PileUp.scala:75-84) of a listed K-mer's occurrences, contiguous
// after the sort, then buildGraph's call (Assembler.scala:131-150), 16 lanes
// a K-mer: the occurrences' values and words come through the permutation,
// so what counts is how many of these loads are in flight (a lane per K-mer,
// eight at a time, took 590 us for 12.4 M occurrences, all K-mers included).
__global__ void __launch_bounds__(256) k_kmer_call(KmerArgs A) {
  const uint32_t g = (blockIdx.x * blockDim.x + threadIdx.x) >> 4;
  const int lane = threadIdx.x & 63, gl = lane & 15;
  const uint32_t n = *A.list_n;
  const bool in = g < n;
  Col c;
  for (int b = 0; b < 4; b++) { c.bc[b] = 0; c.qs[b] = 0; }
  c.mqSum = c.qSum = c.deletions = c.insertions = c.insQual = c.delQual = 0;
  const uint32_t i0 = in ? A.list[g] : 0u;
  const uint32_t lo = A.hlo[i0], hi = A.hhi[i0];
  const uint4* first = (const uint4*)(A.kw + (int64_t)A.perm[i0] * PL_KMER_STRIDE);
  const uint4 f0 = first[0], f1 = first[1];
  bool more = in;
  for (uint32_t i = i0 + gl; __ballot(more); i += 16) {
    const bool same = more && i < A.n_occ && A.hlo[i] == lo && A.hhi[i] == hi;
    if (same) {
      const uint32_t p = A.perm[i];
      const uint4* r = (const uint4*)(A.kw + (int64_t)p * PL_KMER_STRIDE);
      const uint4 r0 = r[0], r1 = r[1];
      const uint32_t v = r1.z;
      if (((r0.x ^ f0.x) | (r0.y ^ f0.y) | (r0.z ^ f0.z) | (r0.w ^ f0.w) | (r1.x ^ f1.x) | (r1.y ^ f1.y)) != 0)
        A.flags[0] = 1;
      const uint32_t code = v & 15u;
      const int bi = code == 1u ? 0 : code == 2u ? 1 : code == 4u ? 2 : code == 8u ? 3 : -1;
      const int32_t qual = (int32_t)(int8_t)(uint8_t)(v >> 8);
      const int32_t mq1 = (int32_t)(v >> 16) + 1;
      if (bi >= 0 && qual >= A.min_qual) {
        // each sum by a constant index, so the column stays in registers
        const int64_t qm = (int64_t)j_mul(qual, mq1);
#pragma unroll
        for (int b = 0; b < 4; b++) {
          c.bc[b] += bi == b ? 1 : 0;
          c.qs[b] += bi == b ? qm : 0;
        }
        c.mqSum = j_add(c.mqSum, mq1);
        c.qSum = j_add(c.qSum, qual);
      }
    }
    more = ((__ballot(same) >> (lane & 48)) & 0xffffull) == 0xffffull;   // the K-mer may go on
  }
#pragma unroll
  for (int d = 1; d < 16; d <<= 1) {
#pragma unroll
    for (int b = 0; b < 4; b++) {
      c.bc[b] += __shfl_xor((int)c.bc[b], d, 64);
      c.qs[b] += __shfl_xor((long long)c.qs[b], d, 64);
    }
    c.mqSum = j_add(c.mqSum, __shfl_xor(c.mqSum, d, 64));
    c.qSum = j_add(c.qSum, __shfl_xor(c.qSum, d, 64));
  }
  const bool keep = in && gl == 0 && c.depth() >= A.min_depth;
  __shared__ uint32_t s_n, s_base;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  const uint32_t slot = wave_append(&s_n, keep);
  __syncthreads();
  if (threadIdx.x == 0 && s_n) s_base = atomicAdd(A.out_n, s_n);
  __syncthreads();
  if (!keep) return;
  const uint32_t k = s_base + slot;
  const BaseFacts f = base_facts(c);
  const uint32_t w[PL_KMER_WORDS] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y};
#pragma unroll
  for (int x = 0; x < PL_KMER_WORDS; x++)
    if (x < A.words) A.out_kw[(int64_t)x * A.cap + k] = kmer_ranks(w[x]);
  A.out_next[k] = (uint8_t)"ACGTN"[f.base];
  A.out_alt[k] = f.homo ? (uint8_t)0 : (uint8_t)"ACGT"[f.alt];
}

// ------------------------------------------------------------- byte order
// A kept K-mer's words are ranks of letters, so their order is the letters'.
__device__ __forceinline__ bool kmer_before(const KmerArgs& A, uint32_t a, uint32_t b, int w0) {
  for (int w = w0; w < A.words; w++) {
    const uint32_t x = A.out_kw[(int64_t)w * A.cap + a], y = A.out_kw[(int64_t)w * A.cap + b];
    if (x != y) return x < y;
  }
  return false;
}

// Few K-mers (PL_KMER_RANK_MAX): each one's place is the number of K-mers
// before it, a thread counting them in PL_KMER_RANK_TILE keys staged in LDS
// and adding to rank (zero at first).  Two launches where the radix sort
// takes 16 to 40: graphs of 2,000 / 8,000 / 16,000 / 48,000 kept K-mers 166 /
// 175 / 191 / 538 us by counting, 230 / 235 / 249 / 340 by sorting (even at
// 24,000).
#define PL_KMER_RANK_MAX 8192
#define PL_KMER_RANK_TILE 512
__global__ void __launch_bounds__(256) k_kmer_rank(KmerArgs A, uint32_t n, uint32_t* rank) {
  __shared__ uint64_t keys[PL_KMER_RANK_TILE];
  const uint32_t* k1 = A.out_kw + (A.words > 1 ? A.cap : 0);
  const uint32_t j0 = blockIdx.y * PL_KMER_RANK_TILE;
  for (uint32_t k = threadIdx.x; k < PL_KMER_RANK_TILE; k += 256)
    keys[k] = j0 + k < n ? ((uint64_t)A.out_kw[j0 + k] << 32) | k1[j0 + k] : ~0ull;   // (none is all ones)
  __syncthreads();
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint64_t key = ((uint64_t)A.out_kw[i] << 32) | k1[i];
  uint32_t r = 0;
#pragma unroll 8
  for (uint32_t k = 0; k < PL_KMER_RANK_TILE; k++) {
    const uint64_t o = keys[k];
    r += o < key ? 1u : 0u;
    if (o == key && j0 + k < n && j0 + k != i && kmer_before(A, j0 + k, i, 2)) r++;
  }
  if (r) atomicAdd(&rank[i], r);
}
__global__ void __launch_bounds__(256) k_kmer_place(const uint32_t* rank, uint32_t n, uint32_t* order) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) order[rank[i]] = i;
}

// sort records of the kept K-mers by their first two words
__global__ void __launch_bounds__(256) k_kmer_keys(KmerArgs A, uint32_t n, uint32_t* lo, uint32_t* hi, uint32_t* v) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  hi[i] = A.out_kw[i];
  lo[i] = A.words > 1 ? A.out_kw[A.cap + i] : 0u;
  v[i] = i;
}

// K-mers that agree in their first two words (16 bases) into order, each run
// of them by the thread at its head; a run too long for that sets flags[1]
// (the host then sorts by all the words).
#define PL_KMER_RUN 32
__global__ void __launch_bounds__(256) k_kmer_ties(KmerArgs A, uint32_t n, const uint32_t* lo, const uint32_t* hi,
                                                   uint32_t* order) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i + 1 >= n) return;
  const uint32_t a = lo[i], b = hi[i];
  if (lo[i + 1] != a || hi[i + 1] != b) return;
  if (i > 0 && lo[i - 1] == a && hi[i - 1] == b) return;
  uint32_t e = i + 2;
  while (e < n && lo[e] == a && hi[e] == b && e - i <= PL_KMER_RUN) e++;
  if (e - i > PL_KMER_RUN) { A.flags[1] = 1; return; }
  for (uint32_t j = i + 1; j < e; j++) {
    const uint32_t x = order[j];
    uint32_t k = j;
    for (; k > i && kmer_before(A, x, order[k - 1], 2); k--) order[k] = order[k - 1];
    order[k] = x;
  }
}

// The K-mers' letters in order (four a thread), then their two edges.
__global__ void __launch_bounds__(256) k_kmer_text(KmerArgs A, uint32_t n, const uint32_t* order, uint8_t* text,
                                                   uint8_t* next, uint8_t* alt) {
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t total = (uint64_t)n * (uint32_t)A.K;
  if (4 * t < total) {
    uint32_t i = (uint32_t)((4 * t) / (uint32_t)A.K), j = (uint32_t)(4 * t - (uint64_t)i * (uint32_t)A.K), out = 0;
    uint32_t k = order[i];
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const uint32_t r = (A.out_kw[(int64_t)(j >> 3) * A.cap + k] >> (28 - 4 * (j & 7u))) & 15u;
      out |= (uint32_t)(uint8_t)"=ABCDGHKMNRSTVWY"[r] << (8 * b);
      if (++j == (uint32_t)A.K) { j = 0; i++; k = order[i < n ? i : n - 1]; }
    }
    *(uint32_t*)(text + 4 * t) = out;                          // (text has room for whole words)
  }
  if (t < n) { next[t] = A.out_next[order[t]]; alt[t] = A.out_alt[order[t]]; }
}
