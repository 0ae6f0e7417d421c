// The block search: exact scoring of large batches from a doc-block-major copy of
// a float index.  Included by gs_search.hip inside its namespace.
//
// Documents are cut into blocks of 64.  Of each block the copy holds
//  * the head rows: the weights of the index's 128 longest lists as int8 levels,
//    [64][128], the A operand of int8 matrix products, and
//  * the tail words: its postings of all other terms, one 32-bit word each (tail
//    rank, doc in the block, 10-bit weight level), ordered by list length, so that
//    a wave's 64 words meet neighbouring table entries.
// A workgroup owns a block and up to 512 queries.  It adds the tail postings of
// the block into an LDS tile of 16-bit sums [query][doc] -- each posting finds the
// queries holding its term in a table of the batch -- and then runs the heavy
// terms' products with those sums as the C operand, so that the scores come out in
// registers, where they are compared with the queries' thresholds.  Nothing of
// size [queries x docs] goes through HBM.
//
// Exactness.  Per query the sums are integers in units of 1 / C score:
//  * heavy term h: a_h lv, lv = rint(w L / W_h) with W_h = max |w| of the list, L =
//    255 levels (127 when the index holds negative weights), a_h = rint(q_h C W_h /
//    L), |a_h| <= 16383, q_h = the query's summed weight of h.  Its error is at
//    most |q_h| C W_h / (2 L) + L / 2.
//  * a tail occurrence: v 2^r, v = floor(qi lv / 2^10 + 1/2), lv = rint(w 511 /
//    W_t), qi = rint(q Ct 2^10 W_t / 511), Ct = C / 2^r.  Its error is at most
//    3/4 2^r + |q| C W_t / (2 * 511).  Ct keeps every sum of v within 16 bits.
// With 255 levels the head rows hold lv - 128, which lowers a doc's sum by 128 sum
// a_h, a constant of the query (kq).  a_h = 128 ah + al is taken as two int8
// limbs: sum a_h lv = sum al lv + 2^7 sum ah lv, each an exact int32 sum.  The
// error bounds give the selection margin as in k_query_prep, so every doc that can
// reach the top k is rescored in fp64 and the answers are the fp64 scatter-add's.

typedef int32_t gs_v16i __attribute__((ext_vector_type(16)));

constexpr int kBlkDocs = GS_BLOCK_DOCS;
constexpr int kBlkHeavy = GS_BLOCK_HEAVY;
constexpr int kBlkMaxQ = 512;      // queries of one workgroup
constexpr int kBlkThreads = 512;   // 8 waves, two workgroups per CU
constexpr int kBlkMinCand = 128;   // emitted scores a workgroup collects in LDS, at least
constexpr size_t kBlkLds = 80 * 1024 - 64;  // LDS of one of two workgroups on a CU, less the static part
constexpr int kBlkGroups = 5;      // 64-word groups of a wave whose lookups are in flight together
constexpr int kBlkClosed = 0x7FFFFFFF;  // threshold of a query that emits nothing: above every score
constexpr uint32_t kBlkPast = 0xFFFFFFFFu;  // candidate count of a query that is given up: past any slots
constexpr float kBlkTiny = 1e-30f; // lists with a smaller max |w| are scored as zeros
static_assert(kBlkDocs == 64 && kBlkHeavy % 64 == 0 && kBlkHeavy <= 256, "the kernels' tiles");

// Byte of row i (a doc of a block, or a query of a 16-query column), heavy term h
// in an operand of v_mfma_i32_16x16x64_i8 as a wave loads it, 16 bytes per lane: lane
// = row % 16 + 16 (h % 64 / 16), the 1 KiB of (row / 16, h / 64) contiguous.
__host__ __device__ constexpr int blk_at(int i, int h) {
    return (((i >> 4) * (kBlkHeavy / 64) + (h >> 6)) * 64 + ((h & 63) >> 4) * 16 + (i & 15)) * 16 + (h & 15);
}

// ---------------------------------------------------------------------- the copy

// Tail ranks in 256 buckets, 16 per octave of the rank: close enough to sorted for
// neighbouring words to share table lines, at one counting pass.
__device__ __forceinline__ int blk_bucket(int x) {
    return min((int)(__float_as_uint((float)(x + 1)) >> 19) - (127 << 4), 255);
}

// What the fill needs of a term, in one 8-byte look-up per posting: its rank and
// the levels per unit of weight (0 for a list of tiny weights).
__global__ void k_blk_terms(const int32_t *__restrict__ rank, const float *__restrict__ max_abs, int32_t V,
                            int32_t levels, uint2 *__restrict__ info) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= V) return;
    const int rk = rank[t];
    const float W = max_abs[t];
    const float per = W > kBlkTiny ? (rk < kBlkHeavy ? (float)levels : 511.0f) / W : 0.0f;
    info[t] = make_uint2((uint32_t)rk, __float_as_uint(per));
}

// One workgroup per block of 64 docs, from the doc-major copy.  The tail words of
// a block start at its first posting's index (row_ptr[64 b]); count[b] of them.  The
// postings are read once: head levels and bucket counts, the tail words kept in LDS
// (a block with more than kBlkStage postings reads them again), then put into their
// buckets.  The look-ups bound it, about one line per clock of each CU's vector cache:
// 1.06e9 postings 5.2 ms, 10.6 with two look-ups per posting in two sweeps.
constexpr int kBlkStage = 9216;
template <int WT>
__global__ void __launch_bounds__(512)
    k_blk_fill(const int64_t *__restrict__ row_ptr, const int32_t *__restrict__ fterm, const void *__restrict__ fw,
               int64_t n_docs, const uint2 *__restrict__ info, int32_t levels, int8_t *__restrict__ head,
               uint32_t *__restrict__ tail, int32_t *__restrict__ count, int32_t *__restrict__ negative) {
    using store_t = typename gs_weight<WT>::store_t;
    constexpr int UN = 8, NT = 512;
    __shared__ __align__(16) int8_t s_head[kBlkDocs * kBlkHeavy];
    __shared__ uint32_t s_word[kBlkStage];
    __shared__ int32_t s_row[kBlkDocs + 1];
    __shared__ uint32_t s_cnt[256], s_wave[4];
    const int tid = threadIdx.x;
    const int64_t doc0 = (int64_t)blockIdx.x * kBlkDocs;
    const int64_t base = row_ptr[doc0];
    const store_t *wall = reinterpret_cast<const store_t *>(fw);
    const uint32_t absent = levels == 255 ? 0x80808080u : 0u;
    for (int i = tid; i < kBlkDocs * kBlkHeavy / 4; i += NT) reinterpret_cast<uint32_t *>(s_head)[i] = absent;
    if (tid < 256) s_cnt[tid] = 0;
    if (tid <= kBlkDocs) s_row[tid] = (int32_t)(row_ptr[min(doc0 + tid, n_docs)] - base);
    __syncthreads();
    const int n = s_row[kBlkDocs];
    const bool staged = n <= kBlkStage;
    constexpr uint32_t kNone = 0xFFFFFFFFu;  // no tail word: tail ranks are below 65535
    bool neg = false;
    // f(i, tail word or kNone) for every posting i; heavy levels are stored when `first`
    auto sweep = [&](bool first, auto &&f) {
        for (int i0 = tid; i0 < n; i0 += NT * UN) {
            int32_t t[UN];
            float w[UN];
            uint2 in[UN];
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int i = min(i0 + u * NT, n - 1);
                t[u] = fterm[base + i];
                w[u] = (float)gs_weight<WT>::decode(wall[base + i]);
            }
#pragma unroll
            for (int u = 0; u < UN; ++u) in[u] = info[t[u]];
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const int i = i0 + u * NT;
                if (i >= n) continue;
                const int rk = (int)in[u].x;
                uint32_t word = kNone;
                if (rk >= 0) {
                    int d = 0;  // the row holding posting i: s_row[d] <= i < s_row[d + 1]
#pragma unroll
                    for (int b = kBlkDocs / 2; b >= 1; b >>= 1)
                        if (s_row[d + b] <= i) d += b;
                    const int lv = (int)rintf(w[u] * __uint_as_float(in[u].y));
                    if (rk >= kBlkHeavy) {
                        word = ((uint32_t)min(max(lv, -511), 511) << 22) | ((uint32_t)d << 16) |
                               (uint32_t)(rk - kBlkHeavy);
                    } else if (first) {
                        s_head[blk_at(d, rk)] =
                            (int8_t)(levels == 255 ? min(max(lv, 0), 255) - 128 : min(max(lv, -127), 127));
                    }
                    neg = neg || w[u] < 0.0f;
                }
                f(i, word);
            }
        }
    };
    sweep(true, [&](int i, uint32_t word) {
        if (staged) s_word[i] = word;
        if (word != kNone) atomicAdd(&s_cnt[blk_bucket((int)(word & 0xFFFFu))], 1u);
    });
    __syncthreads();
    uint32_t c = 0, inc = 0;
    if (tid < 256) {
        c = s_cnt[tid];
        inc = gs_wave_incl_scan(c);
        if (gs_lane() == 63) s_wave[tid >> 6] = inc;
    }
    __syncthreads();
    if (tid < 256) {
        uint32_t at = inc - c;
        for (int w = 0; w < (tid >> 6); ++w) at += s_wave[w];
        s_cnt[tid] = at;
        if (tid == 255) count[blockIdx.x] = (int32_t)(at + c);
    }
    __syncthreads();
    uint32_t *out = tail + base;
    auto place = [&](int, uint32_t word) {
        if (word != kNone) out[atomicAdd(&s_cnt[blk_bucket((int)(word & 0xFFFFu))], 1u)] = word;
    };
    if (staged)
        for (int i = tid; i < n; i += NT) place(i, s_word[i]);
    else
        sweep(false, place);
    uint4 *oh = reinterpret_cast<uint4 *>(head + (int64_t)blockIdx.x * (kBlkDocs * kBlkHeavy));
    for (int i = tid; i < kBlkDocs * kBlkHeavy / 16; i += NT) oh[i] = reinterpret_cast<const uint4 *>(s_head)[i];
    if (levels == 255 && __ballot(neg) && gs_lane() == 0) atomicOr(negative, 1);
}

// ---------------------------------------------------------------------- the batch

// Stride of the order in which the `all` blocks of a collection are taken: coprime to
// it and about its golden section, so that the blocks of any run of places lie evenly
// over the whole collection.  Thresholds are fixed while a launch runs, each launch
// takes as many docs as all before it, and their candidates number about k a launch
// only if the docs so far are a fair sample of the rest.  In id order they are not
// where docs lie in topical, date or length order (8.8M docs sorted by the weight of
// their mid-frequency terms, 512 queries, k = 1000: 11.9 ms in id order, rows past
// their candidate slots among them, 5.4 in this one; sorted by length 8.4 and 5.4; in
// no order 4.99 and 5.01).
inline int32_t blk_stride(int32_t all) {
    int64_t x = std::max<int64_t>(1, (int64_t)(0.6180339887498949 * all));
    while (std::gcd(x, (int64_t)all) != 1) ++x;
    return (int32_t)(x % all);
}

struct BlkQueries {
    const int32_t *qt;
    const float *qw;
    int32_t B, T, V, Q, slots, n_tail;
    const int32_t *rank, *heavy, *dup;
    const float *max_abs;
    int32_t levels;
    int8_t *alimb;   // [slots / 16][2 limbs][16 x 128] of the heavy terms' integer query weights (blk_at)
    int32_t *shift;  // [slots] r
    int32_t *kq;     // [slots] 128 sum a_h (255 levels)
    double *ct;      // [slots] Ct; 0: no entries (padding, or a row for the dense path)
    uint2 *tab;      // [chunks][n_tail] entries of each tail term: [x, y)
    uint32_t *ent;   // [chunks][ent_ld] qi << 12 | 8 times the query's place in the chunk
    int64_t ent_ld;
    uint32_t *total;  // [chunks] entries handed out
    uint32_t *mfix, *tau, *cnt;
    const int64_t *row_ptr;  // of the blocks, in the order they are taken in (blk_stride):
    const int32_t *count;
    int32_t all, stride;
    uint4 *place;  // [all] first word (x, y), number of words and block of each place
};

// One wave per query slot: C, r and Ct (top of the file), the heavy limbs, the
// margin, the counts of the tail terms' entries.  Slots past B get zero limbs, and
// so do queries without a feasible C: non-finite weights and no term, whose margin
// 2^31 - 1 and lack of candidates send their row to the dense path, and too many
// terms or too wide a margin, whose row is flagged as past its candidate slots.
__global__ void __launch_bounds__(256) k_blk_prep(const BlkQueries a) {
    __shared__ double s_q[4][kBlkHeavy];
    const int wv = threadIdx.x >> 6;
    const int q = (int)((blockIdx.x * (int64_t)blockDim.x + threadIdx.x) >> 6);
    const int lane = gs_lane();
    if (q >= a.slots) return;
    int8_t *lim = a.alimb + (int64_t)(q >> 4) * (2 * 16 * kBlkHeavy);
    constexpr int kLimb = 16 * kBlkHeavy;  // bytes from a column's low limbs to its high ones
    if (q >= a.B) {
        for (int h = lane; h < kBlkHeavy; h += 64) lim[blk_at(q & 15, h)] = lim[kLimb + blk_at(q & 15, h)] = 0;
        if (lane == 0) {
            a.shift[q] = 0;
            a.kq[q] = 0;
            a.ct[q] = 0.0;
        }
        return;
    }
    for (int h = lane; h < kBlkHeavy; h += 64) s_q[wv][h] = 0.0;
    gs_wave_sync();
    const int32_t *qrow = a.qt + (int64_t)q * a.T;
    const float *wrow = a.qw + (int64_t)q * a.T;
    double M = 0.0, n = 0.0, TQ = 0.0, nT = 0.0, Z = 0.0;
    for (int j = lane; j < a.T; j += 64) {
        const int32_t t = qrow[j];
        if ((uint32_t)t >= (uint32_t)a.V) continue;
        const int rk = a.rank[t];
        if (rk < 0) continue;  // an empty list
        const double m = 1.0 + (double)a.dup[t];
        const double x = (double)wrow[j];
        const float W = a.max_abs[t];
        const double p = fabs(x) * (double)W * m;
        M += p;
        n += m;
        if (!(W > kBlkTiny)) Z += p;
        if (rk < kBlkHeavy) {
            __hip_atomic_fetch_add(&s_q[wv][rk], x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        } else {
            TQ += p;
            nT += m;
        }
    }
    gs_wave_sync();
    double hmax = 0.0, hsum = 0.0, hn = 0.0;  // max and sum of |q_h| W_h, heavy terms held
    double hq[kBlkHeavy / 64];
    float hW[kBlkHeavy / 64];
#pragma unroll
    for (int u = 0; u < kBlkHeavy / 64; ++u) {
        const int h = u * 64 + lane;
        const int32_t t = a.heavy[h];
        hq[u] = s_q[wv][h];
        hW[u] = t >= 0 ? a.max_abs[t] : 0.0f;
        const double p = fabs(hq[u]) * (double)hW[u];
        hmax = fmax(hmax, p);
        hsum += p;
        hn += hq[u] != 0.0;
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        M += __shfl_xor(M, d, 64);
        n += __shfl_xor(n, d, 64);
        TQ += __shfl_xor(TQ, d, 64);
        nT += __shfl_xor(nT, d, 64);
        Z += __shfl_xor(Z, d, 64);
        hmax = fmax(hmax, __shfl_xor(hmax, d, 64));
        hsum += __shfl_xor(hsum, d, 64);
        hn += __shfl_xor(hn, d, 64);
    }
    M *= 1.0 + 1e-12;  // fp64 rounding of the sums themselves
    TQ *= 1.0 + 1e-12;
    hsum *= 1.0 + 1e-12;
    const double L = (double)a.levels;
    // C W_h |q_h| / L + 1/2 <= 16383;  sum |v| <= Ct TQ + 3/2 nT <= 32766
    const double room = 32766.0 - 1.5 * nT;
    double C = hmax > 0.0 ? 16382.0 * L / hmax : INFINITY;
    int r = 0;
    double Ct;
    if (TQ > 0.0) {
        const double most = room / TQ;
        const double ratio = C / most;
        while (r < 14 && ldexp(1.0, r + 1) <= ratio) ++r;
        C = fmin(C, ldexp(most, r));
        Ct = ldexp(C, -r);
    } else {
        Ct = C;
    }
    const double inf = INFINITY;
    bool ok = M > 0.0 && M < inf && room > 0.0 && C > 0.0 && C < 1e30 && Ct > 0.0;
    // errors in units of 1 / C (rintf of an fp32 quotient: 0.5002 of a level)
    const double E = 0.5002 / L * hsum * C + 0.5 * L * hn + nT * ldexp(0.75, r) + 0.5002 / 511.0 * TQ * C + Z * C;
    const double g64 = (2.0 * n + 2.0) * 0x1p-53 / (1.0 - (2.0 * n + 2.0) * 0x1p-53);
    double mf = ceil(2.0 * (E * (1.0 + 1e-9) + g64 * M * C)) + 2.0;
    ok = ok && mf < 2147483647.0;
    // the limbs
    int sum = 0;
    bool fits = true;
#pragma unroll
    for (int u = 0; u < kBlkHeavy / 64; ++u) {
        const double x = ok ? rint(hq[u] * C * (double)hW[u] / L) : 0.0;
        fits = fits && fabs(x) <= 16383.0;
        const int av = fits ? (int)x : 0;
        sum += av;
        lim[blk_at(q & 15, u * 64 + lane)] = (int8_t)(av & 127);
        lim[kLimb + blk_at(q & 15, u * 64 + lane)] = (int8_t)(av >> 7);
    }
    if (__ballot(!fits)) {
        ok = false;
#pragma unroll
        for (int u = 0; u < kBlkHeavy / 64; ++u)
            lim[blk_at(q & 15, u * 64 + lane)] = lim[kLimb + blk_at(q & 15, u * 64 + lane)] = 0;
    }
    sum = (int)gs_wave_sum((uint32_t)sum);
    if (lane == 0) {
        a.shift[q] = ok ? r : 0;
        a.kq[q] = ok && a.levels == 255 ? 128 * sum : 0;
        a.ct[q] = ok ? Ct : 0.0;
        a.mfix[q] = ok ? (uint32_t)mf : 0x7FFFFFFFu;
        a.tau[q] = 0;
        a.cnt[q] = !ok && M > 0.0 && M < inf ? kBlkPast : 0;
    }
    if (!ok) return;
    uint2 *tab = a.tab + (int64_t)(q / a.Q) * a.n_tail;
    for (int j = lane; j < a.T; j += 64) {
        const int32_t t = qrow[j];
        if ((uint32_t)t >= (uint32_t)a.V) continue;
        const int rk = a.rank[t];
        if (rk >= kBlkHeavy) atomicAdd(&tab[rk - kBlkHeavy].y, 1u);
    }
}

// Words of the bitmap of the tail terms with entries.
__host__ __device__ constexpr int blk_live_words(int n_tail) { return (n_tail + 63) / 64; }

// Entry ranges from the counts: 1024 terms per workgroup take consecutive ranges,
// the workgroups' runs in any order.  (x, y) <- (begin, begin): k_blk_entries
// advances y to the range's end.
__global__ void __launch_bounds__(1024) k_blk_ranges(uint2 *__restrict__ tab, int32_t n_tail,
                                                     uint32_t *__restrict__ total, uint64_t *__restrict__ live) {
    __shared__ uint32_t s_wave[16], s_base;
    const int x = blockIdx.x * 1024 + threadIdx.x;
    uint2 *t = tab + (int64_t)blockIdx.y * n_tail;
    const int wave = threadIdx.x >> 6;
    const uint32_t c = x < n_tail ? t[x].y : 0u;
    const uint32_t inc = gs_wave_incl_scan(c);
    if (gs_lane() == 63) s_wave[wave] = inc;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t tot = 0;
        for (int w = 0; w < 16; ++w) tot += s_wave[w];
        s_base = tot ? atomicAdd(total + blockIdx.y, tot) : 0u;
    }
    __syncthreads();
    uint32_t at = s_base + inc - c;
    for (int w = 0; w < wave; ++w) at += s_wave[w];
    if (x < n_tail) t[x] = make_uint2(at, at);
    const uint64_t has = __ballot(c != 0);
    if (gs_lane() == 0 && x < n_tail) live[(int64_t)blockIdx.y * blk_live_words(n_tail) + (x >> 6)] = has;
}

__global__ void __launch_bounds__(256) k_blk_entries(const BlkQueries a) {
    const int64_t n = (int64_t)a.B * a.T;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int q = (int)(i / a.T);
        const int32_t t = a.qt[i];
        if ((uint32_t)t >= (uint32_t)a.V) continue;
        const int rk = a.rank[t];
        const double ct = a.ct[q];
        if (rk < kBlkHeavy || !(ct > 0.0)) continue;
        const int c = q / a.Q;
        const int qi = (int)rint((double)a.qw[i] * ct * 1024.0 * (double)a.max_abs[t] / 511.0);  // |qi| < 2^17
        const uint32_t at = atomicAdd(&a.tab[(int64_t)c * a.n_tail + rk - kBlkHeavy].y, 1u);
        a.ent[(int64_t)c * a.ent_ld + at] = ((uint32_t)qi << 12) | (uint32_t)(q - c * a.Q) * 8u;
    }
    // where the places' words lie, in their order: neighbouring workgroups of k_blk_score
    // read neighbouring entries (from the arrays by block each block waited for two
    // misses of L2, 45 of 5000 us at 8.8M docs, 512 queries)
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < a.all; p += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t b = (uint32_t)((uint64_t)(p * a.stride) % (uint32_t)a.all);
        const uint64_t s = (uint64_t)a.row_ptr[(int64_t)b * kBlkDocs];
        a.place[p] = make_uint4((uint32_t)s, (uint32_t)(s >> 32), (uint32_t)a.count[b], b);
    }
}

// ---------------------------------------------------------------------- scoring

struct BlkArgs {
    const int8_t *head;
    const uint32_t *tail;
    const uint4 *place;        // BlkQueries::place
    int32_t place0, n_places;  // places of this launch
    int32_t Q, B, chunks, n_tail;
    int32_t sets;  // workgroups per chunk, each taking every sets-th place
    const int8_t *alimb;
    const int32_t *shift, *kq;
    const uint2 *tab;
    const uint32_t *ent;
    const uint64_t *live;
    int64_t ent_ld;
    const uint32_t *tau, *mfix;
    uint32_t *cnt, *cand_doc, *cand_key;
    int32_t cap;
    // emitted scores, one list per workgroup (k_blk_deal hands them to the queries)
    uint32_t *out_q, *out_doc, *out_key, *out_n;
    int32_t out_cap;
    int32_t collect;  // scores a workgroup collects in LDS
    uint32_t *seed;  // SEED: [slots][seed_ld] scores (0 for non-positive ones), by place
    int64_t seed_ld;
};

// Workgroup barrier that orders LDS accesses only: loads from global memory stay in
// flight across it (__syncthreads waits for them).
__device__ __forceinline__ void blk_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// LDS of a scoring workgroup for Q queries: the tile, the live tail terms, thresholds,
// kq and 2^r; and the scores it collects in the rest of half a CU's.
constexpr size_t blk_lds_fixed(int Q, int n_tail) {
    return (size_t)Q * (kBlkDocs * 2 + 4 + 4 + 4) + (size_t)blk_live_words(n_tail) * 8;
}
constexpr int blk_collect(int Q, int n_tail) {
    const size_t fixed = blk_lds_fixed(Q, n_tail);
    const size_t n = fixed < kBlkLds ? (kBlkLds - fixed) / 12 : 0;
    return n < kBlkMinCand ? kBlkMinCand : n > 2048 ? 2048 : (int)n;
}
static_assert(blk_lds_fixed(kBlkMaxQ, 65535) + kBlkMinCand * 12 <= kBlkLds,
              "two scoring workgroups must fit a CU's LDS at the most tail terms");

// One workgroup takes blocks of 64 docs in turn, all Q queries of its chunk at once
// (k_blk_prep ...; the scheme is at the top of the file).  Per block:
//  1. tail: wave w takes word groups w, w + 8, ...; lane: one posting.  A posting of
//     a term the batch holds (a bitmap in LDS) looks its entries up and reads up to
//     four per 16-byte load, one ds_add_u32 each into the tile, whose words hold two
//     docs: a negative sum borrows from the upper one, which the decoding undoes (both
//     sums fit 16 bits).  The look-ups of the other postings' lanes point past their
//     buffers and go nowhere: the vector cache takes about one line per clock.
//  2. products: wave w takes 16-query columns w, w + 8, ...: its C operands are the
//     tile's sums (cleared as they are read), A the block's head rows (held in
//     registers, loaded under the tail), B the queries' limbs, loaded a column ahead.
//  3. scores at or above their query's threshold are collected in LDS and go to the
//     workgroup's own list between blocks.  (With a slot, a histogram count and a bin
//     maximum per candidate as device atomics, those took 1.1 of 3.0 ms at 2.2M docs,
//     512 queries: thresholds are raised between launches instead, k_blk_tau.  Stored
//     to the list at once, each store held the next column's limbs up, since loads and
//     stores share a counter: 1.2 of 3.8 ms at 4.4M docs.)
// The tile's 8-byte pieces (4 docs of a query) are XOR-swizzled by the query, so
// that a wave's C reads (16 queries x 4 pieces) spread over the banks.
// SEED: the scores themselves go to `seed`, for the first threshold.
// What bounds it: by the counters no unit alone.  8.8M docs, 512 queries, k = 1000:
// 4.4 ms for all launches, where the hybrid search's products and scorer took 1.7 +
// 5.4, with the vector ALU issuing 58% of the time, the vector cache at 0.50 lines per
// clock and CU, LDS 18%, MFMA 11%, HBM at a tenth; 14.5 of 16 waves per CU are there,
// and wait half of their time for a block's chain of loads (words, look-ups, entries,
// head rows) and its barriers.  Emission is about 12% (k = 10: 0.6 ms less).  (256
// heavy terms: 64 more registers of head rows, so half the waves, 3.8 ms at 4.4M docs
// against 2.6.  At 128 they cost 204 tail adds per doc instead of 91, and win.)
template <bool SEED>
__global__ void __launch_bounds__(kBlkThreads, 4) k_blk_score(const BlkArgs a) {
    constexpr int NW = kBlkThreads / 64;
    constexpr int KB = kBlkHeavy / 64;
    constexpr int RT = kBlkDocs / 16;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    __shared__ uint32_t s_nc, s_listed, s_open;  // scores collected, and in the workgroup's list; queries that emit
    unsigned char *tile = lds_raw;
    uint32_t *s_live = reinterpret_cast<uint32_t *>(lds_raw + (size_t)a.Q * (kBlkDocs * 2));
    int32_t *s_thr = reinterpret_cast<int32_t *>(s_live + 2 * blk_live_words(a.n_tail));
    int32_t *s_kq = s_thr + a.Q, *s_mul = s_kq + a.Q;  // s_mul: 2^r
    uint32_t *s_cq = reinterpret_cast<uint32_t *>(s_mul + a.Q), *s_cd = s_cq + a.collect, *s_ck = s_cd + a.collect;

    const int tid = threadIdx.x, lane = gs_lane();
    const int wave = gs_uniform(tid >> 6);
    // workgroup i runs on XCD i % 8: the chunks of a set of blocks share an XCD
    const int per_xcd = (a.sets * a.chunks + 7) / 8;
    const int lin = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (lin >= a.sets * a.chunks) return;
    const int chunk = lin % a.chunks;
    const int q0 = chunk * a.Q;  // first slot of the chunk
    const uint2 *tab = a.tab + (int64_t)chunk * a.n_tail;
    const uint32_t *ent = a.ent + (int64_t)chunk * a.ent_ld;
    const int nct = a.Q >> 4;
    const int last = a.place0 + a.n_places;

    for (int i = tid; i < a.Q * (kBlkDocs * 2 / 16); i += kBlkThreads)
        reinterpret_cast<uint4 *>(tile)[i] = make_uint4(0, 0, 0, 0);
    if (tid == 0) s_nc = s_listed = s_open = 0;
    __syncthreads();
    for (int i = tid; i < a.Q; i += kBlkThreads) {
        const int kq = a.kq[q0 + i];
        s_kq[i] = kq;
        s_mul[i] = 1 << a.shift[q0 + i];
        // the threshold on the products' own scale (kq below the score); slots past B never
        // emit, nor do queries past their candidate slots, whose rows are done elsewhere
        int64_t th = kBlkClosed;
        if (!SEED && q0 + i < a.B && a.cnt[q0 + i] <= (uint32_t)a.cap)
            th = (int64_t)emit_threshold(a.tau[q0 + i], a.mfix[q0 + i]) - kq;
        s_thr[i] = (int)(th > kBlkClosed ? kBlkClosed : th);
        if (s_thr[i] != kBlkClosed) s_open = 1;
    }
    const int n_live = 2 * blk_live_words(a.n_tail);
    const uint32_t *live = reinterpret_cast<const uint32_t *>(a.live) + (int64_t)chunk * n_live;
    for (int i = tid; i < n_live; i += kBlkThreads) s_live[i] = live[i];
    __syncthreads();
    if (!SEED && !s_open) {
        if (tid == 0) a.out_n[lin] = 0;
        return;
    }
    const auto r_tab = gs_rsrc(tab, (uint32_t)a.n_tail * 8u);
    const auto r_ent = gs_rsrc(ent, (uint32_t)(a.ent_ld * 4));

    // score i of the workgroup's list; one past its end goes straight to its query's candidates
    auto to_list = [&](uint32_t i, uint32_t q, uint32_t doc, uint32_t key) {
        if (i < (uint32_t)a.out_cap) {
            const int64_t o = (int64_t)lin * a.out_cap + i;
            a.out_q[o] = q;
            a.out_doc[o] = doc;
            a.out_key[o] = key;
            return;
        }
        const uint32_t slot = atomicAdd(a.cnt + q, 1u);
        if (slot < (uint32_t)a.cap) {
            a.cand_doc[(int64_t)q * a.cap + slot] = doc;
            a.cand_key[(int64_t)q * a.cap + slot] = key;
        } else {  // the query is past its slots: no more of it from this workgroup
            __hip_atomic_store(s_thr + (q - q0), kBlkClosed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    };
    // the collected scores to the list; the whole workgroup, after a barrier
    auto flush = [&]() {
        const uint32_t nc = min(s_nc, (uint32_t)a.collect), at = s_listed;
        for (uint32_t i = tid; i < nc; i += kBlkThreads) to_list(at + i, s_cq[i], s_cd[i], s_ck[i]);
        blk_barrier();
        if (tid == 0) {
            s_nc = 0;
            s_listed = at + nc;
        }
        blk_barrier();
    };
    // the first words of a block are loaded before the previous block's products
    auto load_words = [&](const uint32_t *words, int n, int g0, uint32_t (&wd)[kBlkGroups]) {
#pragma unroll
        for (int u = 0; u < kBlkGroups; ++u) wd[u] = words[max(min(g0 + u * NW * 64 + lane, n - 1), 0)];
    };
    auto load_limbs = [&](int ct, gs_v4i (&l)[KB], gs_v4i (&h)[KB]) {
        const int8_t *ap = a.alimb + (int64_t)((q0 >> 4) + ct) * (2 * 16 * kBlkHeavy) + lane * 16;
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            l[kb] = *reinterpret_cast<const gs_v4i *>(ap + kb * 1024);
            h[kb] = *reinterpret_cast<const gs_v4i *>(ap + 16 * kBlkHeavy + kb * 1024);
        }
    };
    int place = a.place0 + lin / a.chunks;
    auto first_word = [&](const uint4 &p) { return a.tail + (int64_t)((uint64_t)p.y << 32 | p.x); };
    uint4 here = a.place[place];
    const uint32_t *words = first_word(here);
    int n = (int)here.z;
    uint32_t wd[kBlkGroups];
    if (n > 0) load_words(words, n, wave * 64, wd);

    for (; place < last; place += a.sets) {
        const int64_t doc0 = (int64_t)here.w * kBlkDocs;
        gs_v4i av[RT][KB];
        auto load_head = [&]() {
            const int8_t *hp = a.head + doc0 * kBlkHeavy + lane * 16;
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int kb = 0; kb < KB; ++kb)
                    av[rt][kb] = *reinterpret_cast<const gs_v4i *>(hp + (rt * KB + kb) * 1024);
        };
        if (wave * 64 >= n) load_head();
        for (int g0 = wave * 64; g0 < n; g0 += NW * 64 * kBlkGroups) {
            // (every load below is issued, whatever its lanes need: a load under a branch
            // would be waited for there, and they would not be in flight together)
            uint2 be[kBlkGroups];
#pragma unroll
            for (int u = 0; u < kBlkGroups; ++u) {
                const uint32_t x = wd[u] & 0xFFFFu;
                const uint32_t use = (s_live[x >> 5] >> (x & 31u)) & (uint32_t)(g0 + u * NW * 64 + lane < n);
                be[u] = gs_bload64(r_tab, use & 1u ? (int)(x * 8u) : -8);  // past the table: an empty range
            }
            if (g0 == wave * 64) load_head();  // behind the first look-ups, which wait for less
            uint32_t ahead[kBlkGroups];
            load_words(words, n, g0 + NW * 64 * kBlkGroups, ahead);
            // the first four entries of every posting at once: most terms have no more
            gs_u32x4 en[kBlkGroups];
#pragma unroll
            for (int u = 0; u < kBlkGroups; ++u)
                en[u] = __builtin_amdgcn_raw_buffer_load_b128(r_ent, be[u].x < be[u].y ? (int)(be[u].x * 4u) : -16, 0, 0);
#pragma unroll
            for (int u = 0; u < kBlkGroups; ++u) {
                const uint32_t w = wd[u];
                const int lv = (int)w >> 22;
                const uint32_t dpart = ((w >> 15) & 0x78u) | ((w >> 15) & 4u);
                const int sh = (int)((w >> 16) & 1u) << 4;
                const uint32_t end = be[u].y;
                auto add4 = [&](const gs_u32x4 &x, uint32_t e) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        if (e + i < end) {
                            const int v = (__mul24((int)x[i] >> 12, lv) + 512) >> 10;
                            const uint32_t t = x[i] & 0xFF8u;  // query * 8
                            const uint32_t at = (t << 4) + (dpart ^ (t & 0x78u));
                            lds_add<uint32_t>(reinterpret_cast<uint32_t *>(tile + at), (uint32_t)v << sh);
                        }
                    }
                };
                add4(en[u], be[u].x);
                // further entries, eight at a time (the array is padded to whole loads)
                for (uint32_t e = be[u].x + 4; e < end; e += 8) {
                    const gs_u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(r_ent, (int)(e * 4u), 0, 0);
                    const gs_u32x4 y = __builtin_amdgcn_raw_buffer_load_b128(r_ent, (int)(e * 4u), 16, 0);
                    add4(x, e);
                    add4(y, e + 4);
                }
            }
#pragma unroll
            for (int u = 0; u < kBlkGroups; ++u) wd[u] = ahead[u];
        }
        gs_v4i bl[KB], bh[KB];
        load_limbs(min(wave, nct - 1), bl, bh);
        if (place + a.sets < last) {
            here = a.place[place + a.sets];
            words = first_word(here);
            n = (int)here.z;
            if (n > 0) load_words(words, n, wave * 64, wd);
        }
        blk_barrier();

        for (int ct = wave; ct < nct; ct += NW) {
            gs_v4i nl[KB], nh[KB];
            load_limbs(min(ct + NW, nct - 1), nl, nh);  // the next column's
            const int ql = ct * 16 + (lane & 15);  // query of the chunk
            const int mul = s_mul[ql];
            const int thr = s_thr[ql];
            const int kq = s_kq[ql];
            uint2 *tq = reinterpret_cast<uint2 *>(tile + ql * (kBlkDocs * 2));
            gs_v16i s;  // lane: docs 16 rt + 4 (lane / 16) + i of query ql at 4 rt + i
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                uint2 *pc = tq + ((rt * 4 + (lane >> 4)) ^ (lane & 15));
                const uint2 tv = *pc;
                *pc = make_uint2(0, 0);
                gs_v4i c0 = {__mul24((int)(int16_t)tv.x, mul), __mul24((int)(tv.x + 0x8000u) >> 16, mul),
                             __mul24((int)(int16_t)tv.y, mul), __mul24((int)(tv.y + 0x8000u) >> 16, mul)};
                gs_v4i c1 = {0, 0, 0, 0};
#pragma unroll
                for (int kb = 0; kb < KB; ++kb) {
                    c0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[rt][kb], bl[kb], c0, 0, 0, 0);
                    c1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(av[rt][kb], bh[kb], c1, 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) s[4 * rt + i] = c0[i] + (c1[i] << 7);
            }
            const int d = 4 * (lane >> 4);
            if constexpr (SEED) {
#pragma unroll
                for (int rt = 0; rt < RT; ++rt)
                    *reinterpret_cast<uint4 *>(a.seed + (int64_t)(q0 + ql) * a.seed_ld + (int64_t)place * kBlkDocs +
                                               rt * 16 + d) =
                        make_uint4((uint32_t)max(s[4 * rt] + kq, 0), (uint32_t)max(s[4 * rt + 1] + kq, 0),
                                   (uint32_t)max(s[4 * rt + 2] + kq, 0), (uint32_t)max(s[4 * rt + 3] + kq, 0));
            } else {
                int top = s[0];
#pragma unroll
                for (int j = 1; j < 16; ++j) top = max(top, s[j]);
                if (__ballot(top >= thr)) {
                    const uint32_t q = (uint32_t)(q0 + ql);
                    uint32_t over = 0;  // docs that found the collection full: bit j
#pragma unroll
                    for (int j = 0; j < 16; ++j) {
                        if (s[j] >= thr) {
                            const uint32_t at = atomicAdd(&s_nc, 1u);
                            if (at < (uint32_t)a.collect) {
                                s_cq[at] = q;
                                s_cd[at] = (uint32_t)(doc0 + (j >> 2) * 16 + d + (j & 3));
                                s_ck[at] = (uint32_t)(s[j] + kq);
                            } else {
                                over |= 1u << j;
                            }
                        }
                    }
                    // the first launches, whose thresholds are low (j is uniform: s[j] is an
                    // indexed register)
                    if (__ballot(over != 0)) {
#pragma unroll 1
                        for (int j = 0; j < 16; ++j) {
                            const int v = s[j];
                            if (over >> j & 1u)
                                to_list(atomicAdd(&s_listed, 1u), q, (uint32_t)(doc0 + (j >> 2) * 16 + d + (j & 3)),
                                        (uint32_t)(v + kq));
                        }
                    }
                }
            }
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                bl[kb] = nl[kb];
                bh[kb] = nh[kb];
            }
        }
        blk_barrier();
        if (!SEED && s_nc > (uint32_t)a.collect / 4) flush();
    }
    if (!SEED) {
        flush();
        if (tid == 0) a.out_n[lin] = min(s_listed, (uint32_t)a.out_cap);
    }
}

// Hands a scoring launch's lists to the queries: one workgroup per list counts its
// queries in LDS, reserves each query's slots with one atomic and writes them.
__global__ void __launch_bounds__(512)
    k_blk_deal(const uint32_t *__restrict__ out_q, const uint32_t *__restrict__ out_doc,
               const uint32_t *__restrict__ out_key, const uint32_t *__restrict__ out_n, int32_t out_cap, int32_t chunks,
               int32_t Q, int32_t cap, uint32_t *__restrict__ cnt, uint32_t *__restrict__ cand_doc,
               uint32_t *__restrict__ cand_key) {
    __shared__ uint32_t s_n[kBlkMaxQ], s_at[kBlkMaxQ];
    const int tid = threadIdx.x;
    const uint32_t q0 = (uint32_t)((int)(blockIdx.x % chunks) * Q);
    const int64_t o = (int64_t)blockIdx.x * out_cap;
    const uint32_t n = out_n[blockIdx.x];
    if (n == 0) return;
    s_n[tid] = 0;
    __syncthreads();
    for (uint32_t i = tid; i < n; i += 512) {
        atomicAdd(&s_n[out_q[o + i] - q0], 1u);
    }
    __syncthreads();
    s_at[tid] = s_n[tid] ? atomicAdd(cnt + q0 + tid, s_n[tid]) : 0u;
    __syncthreads();
    for (uint32_t i = tid; i < n; i += 512) {
        const uint32_t q = out_q[o + i];
        const uint32_t slot = atomicAdd(&s_at[q - q0], 1u);
        if (slot < (uint32_t)cap) {
            cand_doc[(int64_t)q * cap + slot] = out_doc[o + i];
            cand_key[(int64_t)q * cap + slot] = out_key[o + i];
        }
    }
}

// Threshold of each query: the lower edge of the highest bin with at least k
// scores at or above it, of the seed docs' scores (cnt null: n of them) or of the
// candidates so far (at most n).  One workgroup per query.
__global__ void __launch_bounds__(256)
    k_blk_tau(const uint32_t *__restrict__ score, int64_t ld, int32_t n, const uint32_t *__restrict__ cnt, int32_t k,
              uint32_t *__restrict__ tau) {
    __shared__ uint32_t s_hist[GS_HIST_BINS], s_wave[4];
    const int q = blockIdx.x, tid = threadIdx.x;
    for (int i = tid; i < GS_HIST_BINS; i += 256) s_hist[i] = 0;
    __syncthreads();
    const uint32_t *row = score + (int64_t)q * ld;
    if (cnt && cnt[q] > (uint32_t)n) return;  // past its slots: k_blk_score emits nothing of it
    const int m = cnt ? (int)cnt[q] : n;
    for (int i0 = tid; i0 < m; i0 += 256 * 8) {
        uint32_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = i0 + u * 256 < m ? row[i0 + u * 256] : 0u;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (v[u]) atomicAdd(&s_hist[gs_bin_of((float)v[u])], 1u);
    }
    __syncthreads();
    uint32_t c[8], sum = 0;  // bins 2047 - 8 tid - j
#pragma unroll
    for (int j = 0; j < 8; ++j) sum += (c[j] = s_hist[GS_HIST_BINS - 1 - 8 * tid - j]);
    const uint32_t inc = gs_wave_incl_scan(sum);
    if (gs_lane() == 63) s_wave[tid >> 6] = inc;
    __syncthreads();
    uint32_t before = inc - sum;
    for (int w = 0; w < (tid >> 6); ++w) before += s_wave[w];
    if (before < (uint32_t)k && before + sum >= (uint32_t)k) {
        int j = 0;
        while (before + c[j] < (uint32_t)k) before += c[j++];
        const uint32_t t = int_threshold_of_bin((uint32_t)(GS_HIST_BINS - 1 - 8 * tid - j));
        if (t > tau[q]) tau[q] = t;
    }
}
