// Exact top-k selection of one row per workgroup (1024 threads), shared by the
// search pipeline and the dense-row entry points.
//
// Entries expose a monotone unsigned key (larger score -> larger key) and a
// unique doc id; the order is key descending, doc ascending.  A radix select
// finds a cut on the key (and, where keys tie at the k-th, on the doc id); the
// entries past the cut are collected into LDS and sorted with Batcher's bitonic
// network.  What bounds such a selection is the chain of passes and barriers of
// its one workgroup, not bytes, so
//  * a list that fits the threads' registers or LDS is read once (SelKeys,
//    SelKeysLds), a longer one eight entries per thread at a time;
//  * the digits start at the highest bit in which the keys differ (the first
//    digit of keys sharing their top bits would send every LDS add to one bin);
//  * the select stops as soon as what lies at or above the current digit fits
//    the sort buffer, which holds twice k;
//  * the sort takes up to three strides per pass over LDS, eight entries per
//    thread in registers: 22 passes and barriers instead of 55 for 1024 entries.
// Final sort of ~1065 rescored entries to 1000: 42 -> 33 us at 512 rows, 82 -> 62
// at 1024; the k-th of the candidates (9 K of 512 rows, 38 K of 16): 66 -> 23 and
// 74 -> 28 us against digits from the top bit, re-read lists and one stride per
// barrier.  (48 keys per thread in registers instead of LDS spilled: 57 us.)
#pragma once

#include "gs_common.h"

namespace gs {

constexpr int kSelThreads = 1024;
constexpr int kMaxK = 8192;  // LDS sort capacity


// Entry i of the sort buffer lies at sel_pos(i): one entry of padding after every
// eight, so that threads sorting eight consecutive entries each start in
// different LDS banks.
__host__ __device__ constexpr int sel_pos(int i) { return i + (i >> 3); }

// LDS of one selection: the radix state (static) ...
struct SelStatic {
    uint32_t hist[256];
    unsigned long long kmin, kmax;  // of the eligible keys
    uint64_t prefix;
    uint32_t kr;         // entries still to take at the current prefix
    uint32_t above;      // entries above the current prefix
    uint32_t tie_total;  // entries at the current prefix
    uint32_t doc_prefix;
    uint32_t n_sel;
};
// ... and each thread's view of it plus the dynamic sort buffer (key, doc).
struct SelShared {
    SelStatic &s;
    uint64_t *key;
    uint32_t *doc;
    int cap;
    __device__ uint64_t key_at(int i) const { return key[sel_pos(i)]; }
    __device__ uint32_t doc_at(int i) const { return doc[sel_pos(i)]; }
};

// Sort-buffer entries for a selection of k: a power of two (bitonic sort), at
// least 2 k where that fits, so that the radix select can stop early.
__host__ __device__ constexpr int sel_cap(int k) {
    int c = 512;
    while (c < 2 * k && c < kMaxK) c <<= 1;
    return c;
}
inline size_t sel_lds_bytes(int k) { return (size_t)sel_pos(sel_cap(k)) * (sizeof(uint64_t) + sizeof(uint32_t)); }
// Raises a selection kernel's dynamic LDS limit when sel_lds_bytes(k) exceeds
// the 64 KiB default.
inline hipError_t sel_attr(const void *fn, size_t lds) {
    return lds > 65536 ? hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) : hipSuccess;
}

extern __shared__ __align__(16) unsigned char gs_sel_lds[];

// The view of a selection kernel launched with sel_lds_bytes(k) of dynamic LDS.
__device__ __forceinline__ SelShared sel_view(SelStatic &st, int k) {
    const int cap = sel_cap(k);
    uint64_t *key = reinterpret_cast<uint64_t *>(gs_sel_lds);
    return SelShared{st, key, reinterpret_cast<uint32_t *>(key + sel_pos(cap)), cap};
}

// Wave-wide search of a 256-bin histogram: the digit at which the running count
// (from digit 255 down when `desc`, from 0 up otherwise) reaches kr, and the
// count of the bins before it.  Lane l holds four consecutive bins; a wave scan
// of their sums finds the lane, which walks its four.  All lanes return both.
__device__ __forceinline__ void sel_find_digit(const uint32_t *hist, uint32_t kr, bool desc, int &digit,
                                               uint32_t &before) {
    const int lane = gs_lane();
    uint32_t h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) h[i] = hist[desc ? 255 - (4 * lane + i) : 4 * lane + i];
    const uint32_t tot = h[0] + h[1] + h[2] + h[3];
    const uint32_t incl = gs_wave_incl_scan(tot);
    const uint32_t excl = incl - tot;
    const uint64_t bal = __ballot(excl < kr && kr <= incl);
    if (!bal) {  // kr beyond the total (not reached by a consistent histogram): last digit
        digit = desc ? 0 : 255;
        before = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63) - hist[digit];
        return;
    }
    const int L = __ffsll((unsigned long long)bal) - 1;
    int dg = 0;
    uint32_t cum = excl;
    if (lane == L) {
        int i = 0;
        for (; i < 3; ++i) {
            if (cum + h[i] >= kr) break;
            cum += h[i];
        }
        dg = desc ? 255 - (4 * lane + i) : 4 * lane + i;
    }
    digit = __builtin_amdgcn_readlane(dg, L);
    before = (uint32_t)__builtin_amdgcn_readlane((int)cum, L);
}

// Entries of a selection source expose a monotone key and a unique doc id.
struct SrcCand32 {  // candidate list with 32-bit keys
    const uint32_t *key;
    const uint32_t *doc;
    int64_t n;
    __device__ uint64_t k(int64_t i) const { return key[i]; }
    __device__ uint32_t d(int64_t i) const { return doc[i]; }
};
struct SrcCand64 {  // rescored list with 64-bit keys
    const uint64_t *key;
    const uint32_t *doc;
    int64_t n;
    __device__ uint64_t k(int64_t i) const { return key[i]; }
    __device__ uint32_t d(int64_t i) const { return doc[i]; }
};
struct SrcRowF64 {  // dense fp64 row, doc = column
    const double *v;
    int64_t n;
    __device__ uint64_t k(int64_t i) const { return gs_key_f64(v[i]); }
    __device__ uint32_t d(int64_t i) const { return (uint32_t)i; }
};
struct SrcRowU32 {
    const uint32_t *v;
    int64_t n;
    __device__ uint64_t k(int64_t i) const { return v[i]; }
    __device__ uint32_t d(int64_t i) const { return (uint32_t)i; }
};
struct SrcCandF32 {  // compacted (column, fp32 value) candidates
    const float *val;
    const int32_t *idx;
    int64_t n;
    __device__ uint64_t k(int64_t i) const { return gs_key_f32(val[i]); }
    __device__ uint32_t d(int64_t i) const { return (uint32_t)idx[i]; }
};
struct SrcRowF32 {  // dense fp32 row, optionally only entries >= tau
    const float *v;
    int64_t n;
    uint32_t min_key;
    __device__ uint64_t k(int64_t i) const {
        const uint32_t kk = gs_key_f32(v[i]);
        return kk >= min_key ? (uint64_t)kk + 1 : 0;  // 0 = filtered out
    }
    __device__ uint32_t d(int64_t i) const { return (uint32_t)i; }
};

// Dense row (fp64 or uint32 values, doc = column) past a cutoff: only the
// entries after (ck, cd) in (key desc, doc asc) order take part, as key + 1 (a
// finite score's key is below 2^64 - 1); the others read 0, filtered out.  With
// `cut` false every entry takes part.  Successive selections of up to kMaxK
// entries, each after the previous one's last entry, give a top-k of any k.
template <bool F64>
struct SrcRowAfter {
    const void *v;
    int64_t n;
    uint64_t ck;
    uint32_t cd;
    bool cut;
    __device__ uint64_t k(int64_t i) const {
        const uint64_t kk = F64 ? gs_key_f64(reinterpret_cast<const double *>(v)[i])
                                : (uint64_t)reinterpret_cast<const uint32_t *>(v)[i];
        const bool after = !cut || kk < ck || (kk == ck && (uint32_t)i > cd);
        return after ? kk + 1 : 0;
    }
    __device__ uint32_t d(int64_t i) const { return (uint32_t)i; }
};

__device__ __forceinline__ bool sel_before(uint64_t ka, uint32_t da, uint64_t kb, uint32_t db) {
    return ka > kb || (ka == kb && da < db);
}

// LV strides (s << (LV - 1), ..., s) of the bitonic merge of runs of `size`: each
// thread holds 2^LV entries s apart.
template <int LV>
__device__ void sort_strides(SelShared &sh, int np, int size, int s_log2) {
    constexpr int M = 1 << LV;
    for (int g = threadIdx.x; g < np >> LV; g += blockDim.x) {
        const int base = ((g >> s_log2) << (s_log2 + LV)) | (g & ((1 << s_log2) - 1));
        const bool up = (base & size) == 0;
        uint64_t k[M];
        uint32_t d[M];
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const int at = sel_pos(base + (j << s_log2));
            k[j] = sh.key[at];
            d[j] = sh.doc[at];
        }
#pragma unroll
        for (int h = M / 2; h >= 1; h >>= 1) {
#pragma unroll
            for (int j = 0; j < M; ++j) {
                if (j & h) continue;
                const bool swap = up == sel_before(k[j | h], d[j | h], k[j], d[j]);
                const uint64_t ka = swap ? k[j | h] : k[j], kb = swap ? k[j] : k[j | h];
                const uint32_t da = swap ? d[j | h] : d[j], db = swap ? d[j] : d[j | h];
                k[j] = ka;
                k[j | h] = kb;
                d[j] = da;
                d[j | h] = db;
            }
        }
#pragma unroll
        for (int j = 0; j < M; ++j) {
            const int at = sel_pos(base + (j << s_log2));
            sh.key[at] = k[j];
            sh.doc[at] = d[j];
        }
    }
    __syncthreads();
}

// Bitonic sort of entries [0, n) of the sort buffer into (key desc, doc asc).
__device__ void block_sort(SelShared &sh, int n) {
    int np = 1;
    while (np < n) np <<= 1;
    for (int i = n + threadIdx.x; i < np; i += blockDim.x) {
        sh.key[sel_pos(i)] = 0;
        sh.doc[sel_pos(i)] = 0xFFFFFFFFu;
    }
    __syncthreads();
    for (int m = 1; (1 << m) <= np; ++m) {
        for (int rem = m; rem > 0;) {
            const int lv = rem % 3 ? rem % 3 : 3;
            rem -= lv;
            if (lv == 3) sort_strides<3>(sh, np, 1 << m, rem);
            else if (lv == 2) sort_strides<2>(sh, np, 1 << m, rem);
            else sort_strides<1>(sh, np, 1 << m, rem);
        }
    }
}

// The keys of a source as a selection's passes read them: R entries per thread in
// registers when the source has at most R * kSelThreads, else eight loads per
// thread in flight on every pass.
template <int R, class K, class Src>
struct SelKeys {
    const Src &src;
    K kk[R];
    __device__ explicit SelKeys(const Src &s) : src(s) {
        if (cached())
#pragma unroll
            for (int u = 0; u < R; ++u) {
                const int64_t i = (int64_t)u * kSelThreads + threadIdx.x;
                kk[u] = i < src.n ? (K)src.k(i) : K(0);
            }
    }
    __device__ bool cached() const { return src.n <= (int64_t)R * kSelThreads; }
    template <class F>
    __device__ void each(F &&f) const {
        if (cached()) {
#pragma unroll
            for (int u = 0; u < R; ++u) {
                const int64_t i = (int64_t)u * kSelThreads + threadIdx.x;
                if (i < src.n) f(i, (uint64_t)kk[u]);
            }
            return;
        }
        for (int64_t i0 = threadIdx.x; i0 < src.n; i0 += 8 * kSelThreads) {
            K b[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t i = i0 + u * kSelThreads;
                b[u] = i < src.n ? (K)src.k(i) : K(0);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int64_t i = i0 + u * kSelThreads;
                if (i < src.n) f(i, (uint64_t)b[u]);
            }
        }
    }
};

// The same with the first `held` keys in LDS (32-bit keys): tens of thousands of
// them, in loops short enough for the instruction cache.
template <class Src>
struct SelKeysLds {
    const Src &src;
    uint32_t *lds;
    int held;
    __device__ SelKeysLds(const Src &s, uint32_t *buf, int cap) : src(s), lds(buf), held(s.n < cap ? (int)s.n : cap) {
        for (int i0 = threadIdx.x; i0 < held; i0 += 8 * kSelThreads) {
            uint32_t b[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) b[u] = i0 + u * kSelThreads < held ? (uint32_t)src.k(i0 + u * kSelThreads) : 0u;
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (i0 + u * kSelThreads < held) lds[i0 + u * kSelThreads] = b[u];
        }
        __syncthreads();
    }
    template <class F>
    __device__ void each(F &&f) const {
#pragma unroll 4
        for (int i = threadIdx.x; i < held; i += kSelThreads) f((int64_t)i, (uint64_t)lds[i]);
        for (int64_t i = held + threadIdx.x; i < src.n; i += kSelThreads) f(i, src.k(i));
    }
};

// Radix select of the k-th largest key (k <= the eligible entries; keys of 0 are
// ignored when `skip_zero`).  With stop > 0 it ends as soon as the entries at or
// above the current digit number at most `stop`.  Returns the cut: every entry
// above it and sh.s.kr of the sh.s.tie_total entries at it (low bits cleared by
// an early stop, which sets kr = tie_total) are the selection.  Whole workgroup.
template <class Keys>
__device__ uint64_t sel_cut(const Keys &keys, int k, uint32_t stop, SelShared &sh, bool skip_zero) {
    if (threadIdx.x == 0) {
        sh.s.kmin = ~0ull;
        sh.s.kmax = 0;
    }
    __syncthreads();
    uint64_t lo = ~0ull, hi = 0;
    keys.each([&](int64_t, uint64_t kk) {
        if (skip_zero && kk == 0) return;
        lo = kk < lo ? kk : lo;
        hi = kk > hi ? kk : hi;
    });
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        const uint64_t ol = __shfl_xor((unsigned long long)lo, d, 64), oh = __shfl_xor((unsigned long long)hi, d, 64);
        lo = ol < lo ? ol : lo;
        hi = oh > hi ? oh : hi;
    }
    if (gs_lane() == 0) {
        atomicMin(&sh.s.kmin, (unsigned long long)lo);
        atomicMax(&sh.s.kmax, (unsigned long long)hi);
    }
    __syncthreads();
    const uint64_t kmin = sh.s.kmin, kmax = sh.s.kmax;
    int left = kmin < kmax ? 64 - __clzll((long long)(kmin ^ kmax)) : 0;  // key bits still open
    uint64_t pre = left >= 64 ? 0 : (kmax >> left) << left;
    if (threadIdx.x == 0) {
        sh.s.kr = (uint32_t)k;
        sh.s.above = 0;
        sh.s.tie_total = 0xFFFFFFFFu;  // no bit open: the tie count is taken by the caller's doc pass
    }
    __syncthreads();
    while (left > 0) {
        const int bits = left < 8 ? left : 8, shift = left - bits;
        const uint64_t hmask = left >= 64 ? 0ull : ~0ull << left;
        if (threadIdx.x < 256) sh.s.hist[threadIdx.x] = 0;
        __syncthreads();
        keys.each([&](int64_t, uint64_t kk) {
            if (skip_zero && kk == 0) return;
            if ((kk & hmask) == pre) atomicAdd(&sh.s.hist[(kk >> shift) & ((1u << bits) - 1u)], 1u);
        });
        __syncthreads();
        if (threadIdx.x < 64) {
            int dg;
            uint32_t cum;
            sel_find_digit(sh.s.hist, sh.s.kr, true, dg, cum);
            if (threadIdx.x == 0) {
                sh.s.kr -= cum;
                sh.s.above += cum;
                sh.s.prefix = pre | ((uint64_t)dg << shift);
                sh.s.tie_total = sh.s.hist[dg];
            }
        }
        __syncthreads();
        pre = sh.s.prefix;
        left = shift;
        if (stop && sh.s.above + sh.s.tie_total <= stop) {
            __syncthreads();
            if (threadIdx.x == 0) sh.s.kr = sh.s.tie_total;
            break;
        }
    }
    __syncthreads();
    return pre;
}

// Exact top-k of a source by (key desc, doc asc).  Keys equal to 0 are ignored
// when `skip_zero` (used by filtered sources).  Returns the number selected
// (min(k, #entries)), sorted in sh.key/sh.doc.  K: the keys' type (32 or 64 bits).
template <class K, class Src>
__device__ int block_topk(const Src &src, int k, SelShared &sh, bool skip_zero) {
    const SelKeys<sizeof(K) == 8 ? 4 : 8, K, Src> keys(src);
    if (threadIdx.x == 0) sh.s.n_sel = 0;
    __syncthreads();
    uint32_t n_elig = src.n > 0xFFFFFFFFll ? 0xFFFFFFFFu : (uint32_t)src.n;
    if (skip_zero) {
        uint32_t local = 0;
        keys.each([&](int64_t, uint64_t kk) { local += kk != 0; });
        local = gs_wave_sum(local);
        if (gs_lane() == 0) atomicAdd(&sh.s.n_sel, local);
        __syncthreads();
        n_elig = sh.s.n_sel;
        __syncthreads();
        if (threadIdx.x == 0) sh.s.n_sel = 0;
    }
    uint64_t kstar = 0;
    uint32_t dstar = 0xFFFFFFFFu;
    if (n_elig > (uint32_t)sh.cap) {
        kstar = sel_cut(keys, k, (uint32_t)sh.cap, sh, skip_zero);
        const uint32_t need = sh.s.kr;  // ties at kstar to take, by smallest doc
        if (sh.s.tie_total > need) {
            if (threadIdx.x == 0) sh.s.doc_prefix = 0;
            __syncthreads();
            for (int shift = 24; shift >= 0; shift -= 8) {
                for (int b = threadIdx.x; b < 256; b += blockDim.x) sh.s.hist[b] = 0;
                __syncthreads();
                const uint32_t pre = sh.s.doc_prefix;
                const uint32_t hmask = shift + 8 >= 32 ? 0u : (~0u << (shift + 8));
                keys.each([&](int64_t i, uint64_t kk) {
                    if (kk != kstar) return;
                    const uint32_t dd = src.d(i);
                    if ((dd & hmask) == pre) atomicAdd(&sh.s.hist[(dd >> shift) & 255u], 1u);
                });
                __syncthreads();
                if (threadIdx.x < 64) {
                    int dg;
                    uint32_t cum;
                    sel_find_digit(sh.s.hist, sh.s.kr, false, dg, cum);
                    if (threadIdx.x == 0) {
                        sh.s.kr -= cum;
                        sh.s.doc_prefix = pre | ((uint32_t)dg << shift);
                    }
                }
                __syncthreads();
            }
            dstar = sh.s.doc_prefix;
        }
    }
    __syncthreads();
    keys.each([&](int64_t i, uint64_t kk) {
        if ((skip_zero && kk == 0) || kk < kstar) return;
        const uint32_t dd = src.d(i);
        // an early stop leaves kstar's low bits clear and takes everything at or above it
        if (kk == kstar && dd > dstar) return;
        const uint32_t s = atomicAdd(&sh.s.n_sel, 1u);
        if (s < (uint32_t)sh.cap) {
            sh.key[sel_pos((int)s)] = kk;
            sh.doc[sel_pos((int)s)] = dd;
        }
    });
    __syncthreads();
    int c = (int)sh.s.n_sel;
    if (c > sh.cap) c = sh.cap;
    __syncthreads();
    block_sort(sh, c);
    return c < k ? c : k;
}


}  // namespace gs
