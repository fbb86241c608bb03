// hk_sort.hip -- order a raw line list by centre on the device.
//
// The reference sorts each chunk of lines by nu with thrust::sort_by_key and
// then gathers every field through the permutation (Sort_kernel /
// Copy_kernel, heliosk.cu:1147-1171, voigt.h:843-866).  Here lines are ordered by
// (nu, line index), so lines with equal centres keep their input order (a
// stable sort by nu): through buckets that fit in LDS where the list's length
// allows it (further down), else by merging (nu, index) pairs:
//   * pair_block_sort_kernel: runs of 8192 pairs sorted by one workgroup in
//     LDS -- 8 pairs per thread sorted in registers by a bitonic network,
//     then merge rounds in LDS, each thread placing its 8 outputs after a
//     merge-path search;
//   * pair_merge_kernel: runs of w pairs merged into runs of 2w; each
//     workgroup emits 2048 outputs of one merged pair after one merge-path
//     split, with both input slices staged in LDS;
//   * the last pass writes the sorted centres into the output list and the
//     permutation, and gather_kernel moves the other seven fields.
#include <climits>

#include <algorithm>

#include "hk_internal.h"

namespace {

constexpr int kNT = 1024;                 // threads of the block sort
constexpr int kIPT = 8;                   // pairs per thread
constexpr int kRun = kNT * kIPT;          // pairs per LDS-sorted run (8192)
constexpr int kMergeE = 8;                // outputs per thread in a merge pass
constexpr int kMB = 256 * kMergeE;        // outputs per merge workgroup (2048)
constexpr int64_t kMaxSortLines = 0x7fffffff;
constexpr int64_t kWideSplitLines = (int64_t)1 << 20;

// (key, index) order: by key, then by index.
__device__ __forceinline__ bool pless(double ka, int32_t ia, double kb, int32_t ib) {
    return ka < kb || (ka == kb && ia < ib);
}

// LDS slot of pair i where one thread owns IPT pairs: their starts are an odd
// number of slots apart, with a spare slot after every IPT pairs if IPT is even.
template <int IPT>
__device__ __forceinline__ int slot(int i) { return IPT % 2 ? i : i + i / IPT; }
constexpr int kSlots = kRun + kRun / kIPT;

// Sorts the len pairs (sk, si)[slot(i)] of LDS, by the threads of a workgroup
// of at least len / IPT: IPT pairs per thread sorted in registers (bitonic
// network, or odd-even transposition where IPT is no power of two), then merge
// rounds, each thread placing its IPT outputs after a merge-path search.
// less(ka, ia, kb, ib) is a strict order in which a pair of index LAST comes
// behind all others.  Returns after a barrier.
template <int IPT, class Idx, class Less>
__device__ __forceinline__ void lds_sort_pairs(double *sk, Idx *si, int len, int last, Less less) {
    const int t = threadIdx.x;
    const int np = (len + IPT - 1) / IPT * IPT;
    const int d0 = t * IPT;
    const bool act = d0 < np;
    double vk[IPT];
    int vi[IPT];
    auto order = [&](int i, int l, bool up) {
        const bool sw = up == less(vk[l], vi[l], vk[i], vi[i]);
        if (sw) {
            const double tk = vk[i]; vk[i] = vk[l]; vk[l] = tk;
            const int ti = vi[i]; vi[i] = vi[l]; vi[l] = ti;
        }
    };
    if (act) {
#pragma unroll
        for (int q = 0; q < IPT; ++q) {
            const bool in = d0 + q < len;
            vk[q] = in ? sk[slot<IPT>(d0 + q)] : INFINITY;
            vi[q] = in ? (int)si[slot<IPT>(d0 + q)] : last;
        }
        if constexpr ((IPT & (IPT - 1)) == 0) {
#pragma unroll
            for (int k = 2; k <= IPT; k <<= 1) {
#pragma unroll
                for (int j = k >> 1; j > 0; j >>= 1) {
#pragma unroll
                    for (int i = 0; i < IPT; ++i)
                        if ((i ^ j) > i) order(i, i ^ j, (i & k) == 0);
                }
            }
        } else {
#pragma unroll
            for (int k = 0; k < IPT; ++k) {
#pragma unroll
                for (int i = k & 1; i + 1 < IPT; i += 2) order(i, i + 1, true);
            }
        }
    }
    __syncthreads();
    if (act) {
#pragma unroll
        for (int q = 0; q < IPT; ++q) {
            sk[slot<IPT>(d0 + q)] = vk[q];
            si[slot<IPT>(d0 + q)] = (Idx)vi[q];
        }
    }
    for (int L = IPT; L < np; L <<= 1) {
        __syncthreads();
        if (act) {
            const int ps = d0 / (2 * L) * (2 * L);
            const int na = min(L, np - ps), nb = min(L, np - ps - na);
            const int diag = d0 - ps, a0 = ps, b0 = ps + na;
            int lo = max(0, diag - nb), hi = min(diag, na);
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                const int am = slot<IPT>(a0 + mid), bm = slot<IPT>(b0 + diag - mid - 1);
                if (!less(sk[bm], (int)si[bm], sk[am], (int)si[am]))
                    lo = mid + 1;
                else
                    hi = mid;
            }
            int a = lo, b = diag - lo;
            double ka = a < na ? sk[slot<IPT>(a0 + a)] : INFINITY;
            double kb = b < nb ? sk[slot<IPT>(b0 + b)] : INFINITY;
            int ia = a < na ? (int)si[slot<IPT>(a0 + a)] : last;
            int ib = b < nb ? (int)si[slot<IPT>(b0 + b)] : last;
#pragma unroll
            for (int q = 0; q < IPT; ++q) {
                const bool ta = b >= nb || (a < na && !less(kb, ib, ka, ia));
                vk[q] = ta ? ka : kb;
                vi[q] = ta ? ia : ib;
                if (ta) {
                    ++a;
                    ka = a < na ? sk[slot<IPT>(a0 + a)] : INFINITY;
                    ia = a < na ? (int)si[slot<IPT>(a0 + a)] : last;
                } else {
                    ++b;
                    kb = b < nb ? sk[slot<IPT>(b0 + b)] : INFINITY;
                    ib = b < nb ? (int)si[slot<IPT>(b0 + b)] : last;
                }
            }
        }
        __syncthreads();
        if (act) {
#pragma unroll
            for (int q = 0; q < IPT; ++q) {
                sk[slot<IPT>(d0 + q)] = vk[q];
                si[slot<IPT>(d0 + q)] = (Idx)vi[q];
            }
        }
    }
    __syncthreads();
}

__global__ __launch_bounds__(kNT) void pair_block_sort_kernel(const double *__restrict__ key,
                                                              int64_t n,
                                                              double *__restrict__ okey,
                                                              int32_t *__restrict__ oidx) {
    __shared__ double sk[kSlots];
    __shared__ int32_t si[kSlots];
    const int t = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * kRun;
    const int len = (int)std::min<int64_t>(kRun, n - base);
    for (int i = t; i < len; i += kNT) {
        sk[slot<kIPT>(i)] = key[base + i];
        si[slot<kIPT>(i)] = (int32_t)(base + i);
    }
    __syncthreads();
    lds_sort_pairs<kIPT>(sk, si, len, INT_MAX, pless);
    for (int i = t; i < len; i += kNT) {
        okey[base + i] = sk[slot<kIPT>(i)];
        oidx[base + i] = si[slot<kIPT>(i)];
    }
}

// First a in [max(0, diag-nb), min(diag, na)] with A[a] after B[diag-a-1], by
// a wave (WIDE: 64 probes a round, so a range of 2.5e5 takes three rounds of
// loads; halving it 18, a merge pass over it 17 us against 13) or by one lane:
// long lists are bound by memory, and 64 probes a round move as much as the merge
// itself (2.2e7 lines: 354 us a pass, halving 338).
template <bool WIDE>
__device__ __forceinline__ int64_t pair_split(const double *Ak, const int32_t *Ai, int64_t na,
                                              const double *Bk, const int32_t *Bi, int64_t nb,
                                              int64_t diag) {
    int64_t lo = std::max<int64_t>(0, diag - nb), hi = std::min<int64_t>(diag, na);
    if (!WIDE) {
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1, bm = diag - mid - 1;
            if (!pless(Bk[bm], Bi[bm], Ak[mid], Ai[mid])) lo = mid + 1; else hi = mid;
        }
        return lo;
    }
    while (lo < hi) {
        const int64_t step = (hi - lo + 63) >> 6;
        const int64_t mid = lo + (threadIdx.x & 63) * step;
        const int64_t bm = diag - mid - 1;
        const bool before = mid < hi && !pless(Bk[bm], Bi[bm], Ak[mid], Ai[mid]);
        const int c = __popcll(__ballot(before));
        if (c == 0) break;
        hi = std::min(hi, lo + c * step);
        lo += (c - 1) * step + 1;
    }
    return lo;
}

template <bool WIDE>
__global__ __launch_bounds__(256) void pair_merge_kernel(const double *__restrict__ ik,
                                                         const int32_t *__restrict__ ii,
                                                         double *__restrict__ ok,
                                                         int32_t *__restrict__ oi, int64_t n,
                                                         int64_t w) {
    __shared__ double sAk[kMB], sBk[kMB];
    __shared__ int32_t sAi[kMB], sBi[kMB];
    __shared__ int64_t sp[2];
    const int t = threadIdx.x;
    const int64_t o0 = (int64_t)blockIdx.x * kMB;
    if (o0 >= n) return;
    const int64_t ps = o0 / (2 * w) * (2 * w);
    const int64_t na = std::min(w, n - ps), nb = std::min(w, n - ps - na);
    const double *Ak = ik + ps, *Bk = Ak + na;
    const int32_t *Ai = ii + ps, *Bi = Ai + na;
    const int64_t d0 = o0 - ps, d1 = std::min(d0 + kMB, na + nb);
    if (WIDE) {
        if (t < 128) {
            const int64_t a = pair_split<WIDE>(Ak, Ai, na, Bk, Bi, nb, t < 64 ? d0 : d1);
            if ((t & 63) == 0) sp[t >> 6] = a;
        }
    } else {                                    // (scalar loads: the diagonals are uniform)
        if (t == 0) sp[0] = pair_split<WIDE>(Ak, Ai, na, Bk, Bi, nb, d0);
        if (t == 64) sp[1] = pair_split<WIDE>(Ak, Ai, na, Bk, Bi, nb, d1);
    }
    __syncthreads();
    const int64_t a0 = sp[0], a1 = sp[1], b0 = d0 - a0, b1 = d1 - a1;
    const int la = (int)(a1 - a0), lb = (int)(b1 - b0), tot = (int)(d1 - d0);
    for (int i = t; i < la; i += 256) { sAk[i] = Ak[a0 + i]; sAi[i] = Ai[a0 + i]; }
    for (int i = t; i < lb; i += 256) { sBk[i] = Bk[b0 + i]; sBi[i] = Bi[b0 + i]; }
    __syncthreads();
    const int d = t * kMergeE;
    double vk[kMergeE];
    int32_t vi[kMergeE];
    int cnt = 0;
    if (d < tot) {
        int lo = max(0, d - lb), hi = min(d, la);
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            const int bm = d - mid - 1;
            if (!pless(sBk[bm], sBi[bm], sAk[mid], sAi[mid])) lo = mid + 1; else hi = mid;
        }
        int a = lo, b = d - lo;
        cnt = min(kMergeE, tot - d);
        for (int q = 0; q < cnt; ++q) {
            const bool ta = b >= lb || (a < la && !pless(sBk[b], sBi[b], sAk[a], sAi[a]));
            vk[q] = ta ? sAk[a] : sBk[b];
            vi[q] = ta ? sAi[a] : sBi[b];
            if (ta) ++a; else ++b;
        }
    }
    // outputs are written from registers: the slices in LDS are not reused
    for (int q = 0; q < cnt; ++q) {
        ok[o0 + d + q] = vk[q];
        oi[o0 + d + q] = vi[q];
    }
}

struct Fields {
    const double *src[6];
    double *dst[6];
    const int32_t *iso_src;
    int32_t *iso_dst;
};

// out_f[i] = in_f[perm[i]] for S, EL, A, delta, vy, n and iso.
__global__ __launch_bounds__(256) void gather_kernel(const int32_t *__restrict__ perm, int64_t n,
                                                     Fields f) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * 256) {
        const int64_t j = perm[i];
#pragma unroll
        for (int k = 0; k < 6; ++k) f.dst[k][i] = f.src[k][j];
        if (f.iso_src) f.iso_dst[i] = f.iso_src[j];
    }
}

// ---------------------------------------------------------------------------
// Lists of kBucketMinLines to kBucketMaxLines: a sample sort that moves each
// line's 60 bytes twice instead of its (centre, index) pair through every merge
// pass and then six fields and iso through a random gather.
//   * kOver samples per bucket (one from each of nb kOver equal strips of the
//     list, at a hashed place) are sorted by (centre, index); every kOver-th is
//     a splitter.  Splitters compare centre and index, so equal centres spread
//     over buckets as others do;
//   * bucket_count_kernel finds each line's bucket by binary search in LDS and
//     counts; bucket_scan_kernel turns the counts into bucket starts;
//   * bucket_scatter_kernel writes the lines as 64-byte records into their
//     buckets, in no particular order, a quad of lanes per record (a lane
//     writing its own record in four pieces: 443 us at 1e7 lines, this 397);
//   * bucket_sort_kernel sorts a bucket's (centre, index) in LDS -- which makes
//     the result independent of that order -- and writes the fields.
// A bucket is half full on average; with 32 samples each, about one in 3e5
// is too long and is ranked by counting instead.
// Bound by memory: 4 x 60 bytes a line, half of it in scattered 64-byte pieces.
// Whole sort, merge passes and gather against this: 65536 lines 197 and 195 us,
// 1e6 437 and 288, 1e7 3200 and 1120, 2e7 7530 and 2020; at 20000 lines 156
// and 169, so shorter lists keep the merge passes, as do longer ones than
// kMaxBuckets buckets in LDS can hold.
// ---------------------------------------------------------------------------
constexpr int kBIPT = 5;                        // pairs per thread of a bucket sort
constexpr int kMaxBuckets = 8192;
// Threads of a bucket sort, the lines it can hold and the mean it is given:
// 512 (2560, 1280) while kMaxBuckets such buckets hold the list, else 1024.
constexpr int bucket_threads(int64_t n) { return n <= (int64_t)kMaxBuckets * 1280 ? 512 : 1024; }
constexpr int bucket_mean(int nt) { return nt * kBIPT / 2; }
constexpr int kOver = 32;
constexpr int64_t kBucketMaxLines = (int64_t)kMaxBuckets * bucket_mean(1024);
constexpr int64_t kBucketMinLines = 65536;
constexpr int kScatNT = 1024, kScatE = 16;      // lines per scatter workgroup: 16384

// A line as 64 bytes: nu, S, EL, A, delta, vy, n, (iso, place in the input).
struct alignas(64) LineRec {
    int4 q[4];
};

// 4 x 4 transpose of 16-byte pieces over a quad of lanes: piece p of lane r
// and piece r of lane p change places, so that the quad reads and writes
// each of its four records as one 64-byte access.
template <int CTRL>
__device__ __forceinline__ int4 quad_move(const int4 &v) {
    return make_int4(__builtin_amdgcn_mov_dpp(v.x, CTRL, 0xf, 0xf, true),
                     __builtin_amdgcn_mov_dpp(v.y, CTRL, 0xf, 0xf, true),
                     __builtin_amdgcn_mov_dpp(v.z, CTRL, 0xf, 0xf, true),
                     __builtin_amdgcn_mov_dpp(v.w, CTRL, 0xf, 0xf, true));
}

__device__ __forceinline__ int4 pick(bool c, const int4 &a, const int4 &b) {
    return make_int4(c ? a.x : b.x, c ? a.y : b.y, c ? a.z : b.z, c ? a.w : b.w);
}

template <int CTRL>
__device__ __forceinline__ void quad_swap(bool odd, int4 &a, int4 &b) {
    const int4 r = quad_move<CTRL>(pick(odd, a, b));
    a = pick(odd, r, a);
    b = pick(odd, b, r);
}

__device__ __forceinline__ void quad_transpose(int4 (&v)[4]) {
    const int l = threadIdx.x & 3;
    quad_swap<0xB1>(l & 1, v[0], v[1]);         // lanes 1 0 3 2
    quad_swap<0xB1>(l & 1, v[2], v[3]);
    quad_swap<0x4E>(l & 2, v[0], v[2]);         // lanes 2 3 0 1
    quad_swap<0x4E>(l & 2, v[1], v[3]);
}

__device__ __forceinline__ void quad_lanes(int x, int (&o)[4]) {
    o[0] = __builtin_amdgcn_mov_dpp(x, 0x00, 0xf, 0xf, true);
    o[1] = __builtin_amdgcn_mov_dpp(x, 0x55, 0xf, 0xf, true);
    o[2] = __builtin_amdgcn_mov_dpp(x, 0xAA, 0xf, 0xf, true);
    o[3] = __builtin_amdgcn_mov_dpp(x, 0xFF, 0xf, 0xf, true);
}

__device__ __forceinline__ double as_double(int lo, int hi) { return __hiloint2double(hi, lo); }

struct Columns {
    const double *src[7];
    double *dst[7];
    const int32_t *iso_src;
    int32_t *iso_dst;
};

// Place of sample i of ns in a list of n: one per strip, increasing with i.
__device__ __forceinline__ int64_t sample_pos(int64_t i, int64_t ns, int64_t n) {
    const int64_t a = i * n / ns, b = (i + 1) * n / ns;
    uint32_t h = (uint32_t)i * 2654435761u;
    h ^= h >> 16;
    h *= 2246822519u;
    h ^= h >> 13;
    return a + (int64_t)(h % (uint32_t)max((int64_t)1, b - a));
}

__global__ __launch_bounds__(256) void sample_kernel(const double *__restrict__ nu, int64_t n,
                                                     int64_t ns, double *__restrict__ sample,
                                                     uint32_t *__restrict__ total, int nb) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < ns) sample[i] = nu[sample_pos(i, ns, n)];
    if (i < nb) total[i] = 0u;
}

// Splitters (centre, index) from the sorted samples.
__global__ __launch_bounds__(256) void splitter_kernel(const double *__restrict__ k,
                                                       const int32_t *__restrict__ id, int64_t ns,
                                                       int64_t n, int nb,
                                                       double *__restrict__ sk,
                                                       int32_t *__restrict__ si) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= nb - 1) return;
    const int64_t q = (int64_t)(b + 1) * kOver;
    const int64_t s = min(max((int64_t)id[q], (int64_t)0), ns - 1);
    sk[b] = k[q];
    si[b] = (int32_t)sample_pos(s, ns, n);
}

__global__ __launch_bounds__(1024) void bucket_count_kernel(const double *__restrict__ nu,
                                                            int64_t n, int nb,
                                                            const double *__restrict__ spk,
                                                            const int32_t *__restrict__ spi,
                                                            uint16_t *__restrict__ bucket,
                                                            uint32_t *__restrict__ total) {
    __shared__ double sk[kMaxBuckets];
    __shared__ int32_t si[kMaxBuckets];
    __shared__ uint32_t hist[kMaxBuckets];
    const int t = threadIdx.x;
    for (int b = t; b < nb; b += 1024) {
        if (b < nb - 1) { sk[b] = spk[b]; si[b] = spi[b]; }
        hist[b] = 0u;
    }
    __syncthreads();
    for (int64_t i = (int64_t)blockIdx.x * 1024 + t; i < n; i += (int64_t)gridDim.x * 1024) {
        const double k = nu[i];
        int lo = 0, hi = nb - 1;                // splitters before (k, i)
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            const double s = sk[mid];
            if (s < k || (s == k && si[mid] <= (int32_t)i)) lo = mid + 1; else hi = mid;
        }
        bucket[i] = (uint16_t)lo;
        atomicAdd(&hist[lo], 1u);
    }
    __syncthreads();
    for (int b = t; b < nb; b += 1024)
        if (hist[b]) atomicAdd(&total[b], hist[b]);
}

// start[b] = lines in the buckets before b (b = 0..nb); cursor = a copy.
__global__ __launch_bounds__(1024) void bucket_scan_kernel(const uint32_t *__restrict__ total,
                                                           int nb, uint32_t *__restrict__ start,
                                                           uint32_t *__restrict__ cursor) {
    __shared__ uint32_t s[1024];
    const int t = threadIdx.x;
    constexpr int E = kMaxBuckets / 1024;
    uint32_t v[E], sum = 0;
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int b = t * E + q;
        v[q] = sum;
        sum += b < nb ? total[b] : 0u;
    }
    s[t] = sum;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const uint32_t x = t >= off ? s[t - off] : 0u;
        __syncthreads();
        s[t] += x;
        __syncthreads();
    }
    const uint32_t base = s[t] - sum;
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int b = t * E + q;
        if (b < nb) { start[b] = base + v[q]; cursor[b] = base + v[q]; }
    }
    if (t == 1023) start[nb] = s[1023];
}

__global__ __launch_bounds__(kScatNT) void bucket_scatter_kernel(Columns f, int64_t n, int nb,
                                                                 const uint16_t *__restrict__ bucket,
                                                                 uint32_t *__restrict__ cursor,
                                                                 LineRec *__restrict__ rec) {
    __shared__ uint32_t hist[kMaxBuckets];
    const int t = threadIdx.x;
    const int64_t base = (int64_t)blockIdx.x * (kScatNT * kScatE);
    for (int b = t; b < nb; b += kScatNT) hist[b] = 0u;
    __syncthreads();
    int at[kScatE];                             // bucket, then place; -1 past the end
    uint32_t rk[kScatE];
#pragma unroll
    for (int q = 0; q < kScatE; ++q) {
        const int64_t i = base + q * kScatNT + t;
        at[q] = i < n ? (int)bucket[i] : -1;
        rk[q] = at[q] >= 0 ? atomicAdd(&hist[at[q]], 1u) : 0u;
    }
    __syncthreads();
    for (int b = t; b < nb; b += kScatNT) {
        const uint32_t c = hist[b];
        if (c) hist[b] = atomicAdd(&cursor[b], c);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kScatE; ++q)
        if (at[q] >= 0) at[q] = (int)(hist[at[q]] + rk[q]);
#pragma unroll 2
    for (int q = 0; q < kScatE; ++q) {
        const int64_t i = base + q * kScatNT + t;
        const int64_t j = min(i, n - 1);
        int4 v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const double a = f.src[2 * k][j];
            v[k].x = __double2loint(a);
            v[k].y = __double2hiint(a);
            if (k < 3) {
                const double b = f.src[2 * k + 1][j];
                v[k].z = __double2loint(b);
                v[k].w = __double2hiint(b);
            }
        }
        v[3].z = f.iso_src ? f.iso_src[j] : 0;
        v[3].w = (int)j;
        quad_transpose(v);
        int o[4];
        quad_lanes(at[q], o);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (o[r] >= 0) rec[o[r]].q[t & 3] = v[r];
    }
}

__device__ __forceinline__ void put_record(const Columns &f, int64_t o, const int4 (&v)[4]) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        f.dst[2 * k][o] = as_double(v[k].x, v[k].y);
        if (k < 3) f.dst[2 * k + 1][o] = as_double(v[k].z, v[k].w);
    }
    if (f.iso_dst) f.iso_dst[o] = v[3].z;
}

__device__ __forceinline__ double rec_key(const LineRec &r) { return as_double(r.q[0].x, r.q[0].y); }

template <int NT>
__global__ __launch_bounds__(NT, 8) void bucket_sort_kernel(const LineRec *__restrict__ rec,
                                                            const uint32_t *__restrict__ start,
                                                            Columns f) {
    constexpr int kCap = NT * kBIPT;
    __shared__ double sk[kCap];
    __shared__ uint16_t si[kCap];
    __shared__ int32_t id[kCap];
    constexpr int kLast = 0xffff;
    const int t = threadIdx.x;
    const uint32_t s0 = start[blockIdx.x];
    const int cnt = (int)(start[blockIdx.x + 1] - s0);
    const LineRec *r = rec + s0;
    if (cnt <= kCap) {
        for (int i = t; i < cnt; i += NT) {
            sk[i] = rec_key(r[i]);
            id[i] = r[i].q[3].w;
            si[i] = (uint16_t)i;
        }
        __syncthreads();
        // by centre, then by the line's place in the input
        lds_sort_pairs<kBIPT>(sk, si, cnt, kLast, [&](double ka, int ia, double kb, int ib) {
            if (ka != kb) return ka < kb;
            if (ia == kLast || ib == kLast) return ia < ib;
            return id[ia] < id[ib];
        });
        for (int i0 = 0; i0 < cnt; i0 += NT) {
            const int i = i0 + t;
            int o[4];
            quad_lanes(min((int)si[min(i, cnt - 1)], cnt - 1), o);
            int4 v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = r[o[k]].q[t & 3];
            quad_transpose(v);
            if (i < cnt) put_record(f, (int64_t)s0 + i, v);
        }
        return;
    }
    // a bucket beyond the cap: each line's rank by counting
    for (int i0 = 0; i0 < cnt; i0 += NT) {
        const int i = i0 + t;
        const LineRec a = r[min(i, cnt - 1)];
        const double ka = rec_key(a);
        int rank = 0;
        for (int j0 = 0; j0 < cnt; j0 += kCap) {
            const int m = min(kCap, cnt - j0);
            __syncthreads();
            for (int j = t; j < m; j += NT) { sk[j] = rec_key(r[j0 + j]); id[j] = r[j0 + j].q[3].w; }
            __syncthreads();
            for (int j = 0; j < m; ++j) rank += pless(sk[j], id[j], ka, a.q[3].w) ? 1 : 0;
        }
        if (i < cnt) put_record(f, (int64_t)s0 + rank, a.q);
    }
}

int grid_for(int64_t n) {
    int64_t b = (n + 255) / 256;
    return (int)(b < 65536 ? (b > 0 ? b : 1) : 65536);
}

int merge_passes(int64_t n) {
    int p = 0;
    for (int64_t w = kRun; w < n; w *= 2) ++p;
    return p;
}

// The pairs (key[i], i), sorted: into (k0, i0) or (k1, i1); returns which.
int sort_pairs(const double *key, int64_t n, double *k0, int32_t *i0, double *k1, int32_t *i1,
               hipStream_t s, int &which) {
    const unsigned nrun = (unsigned)((n + kRun - 1) / kRun);
    hipLaunchKernelGGL(pair_block_sort_kernel, dim3(nrun), dim3(kNT), 0, s, key, n, k0, i0);
    HK_LAUNCH_CHECK();
    double *ck = k0, *nk = k1;
    int32_t *ci = i0, *ni = i1;
    which = 0;
    const unsigned nblk = (unsigned)((n + kMB - 1) / kMB);
    for (int64_t wl = kRun; wl < n; wl *= 2) {
        if (n <= kWideSplitLines)
            hipLaunchKernelGGL(pair_merge_kernel<true>, dim3(nblk), dim3(256), 0, s, ck, ci, nk, ni, n,
                               wl);
        else
            hipLaunchKernelGGL(pair_merge_kernel<false>, dim3(nblk), dim3(256), 0, s, ck, ci, nk, ni,
                               n, wl);
        HK_LAUNCH_CHECK();
        std::swap(ck, nk);
        std::swap(ci, ni);
        which ^= 1;
    }
    return HK_OK;
}

// Workspace of the merge passes: two ping-pong pairs of (key, index) arrays.
size_t pair_bytes(int64_t n) {
    const size_t kb = hk::align_up((size_t)n * sizeof(double), 256);
    const size_t ib = hk::align_up((size_t)n * sizeof(int32_t), 256);
    return 2 * (kb + ib) + 256;
}

struct BucketLayout {
    int nb;
    int64_t ns;
    size_t rec, k0, i0, k1, i1, spk, spi, bucket, total, start, cursor, bytes;
};

bool use_buckets(int64_t n) { return n >= kBucketMinLines && n <= kBucketMaxLines; }

BucketLayout bucket_layout(int64_t n) {
    BucketLayout L;
    const int mean = bucket_mean(bucket_threads(n));
    L.nb = (int)((n + mean - 1) / mean);
    L.ns = (int64_t)L.nb * kOver;
    size_t o = 0;
    auto take = [&](size_t b) { const size_t at = o; o = hk::align_up(o + b, 256); return at; };
    L.rec = take((size_t)n * sizeof(LineRec));
    L.k0 = take((size_t)L.ns * sizeof(double));
    L.i0 = take((size_t)L.ns * sizeof(int32_t));
    L.k1 = take((size_t)L.ns * sizeof(double));
    L.i1 = take((size_t)L.ns * sizeof(int32_t));
    L.spk = take((size_t)L.nb * sizeof(double));
    L.spi = take((size_t)L.nb * sizeof(int32_t));
    L.bucket = take((size_t)n * sizeof(uint16_t));
    L.total = take((size_t)L.nb * sizeof(uint32_t));
    L.start = take((size_t)(L.nb + 1) * sizeof(uint32_t));
    L.cursor = take((size_t)L.nb * sizeof(uint32_t));
    L.bytes = o + 256;
    return L;
}

int bucket_sort(const Columns &f, int64_t n, char *w, hipStream_t s) {
    const BucketLayout L = bucket_layout(n);
    double *k[2] = {(double *)(w + L.k0), (double *)(w + L.k1)};
    int32_t *id[2] = {(int32_t *)(w + L.i0), (int32_t *)(w + L.i1)};
    uint32_t *total = (uint32_t *)(w + L.total), *start = (uint32_t *)(w + L.start);
    uint32_t *cursor = (uint32_t *)(w + L.cursor);
    uint16_t *bucket = (uint16_t *)(w + L.bucket);
    double *spk = (double *)(w + L.spk);
    int32_t *spi = (int32_t *)(w + L.spi);
    LineRec *rec = (LineRec *)(w + L.rec);
    // the samples go through the record area: it is free until the scatter
    double *sample = (double *)rec;
    hipLaunchKernelGGL(sample_kernel, dim3((unsigned)((L.ns + 255) / 256)), dim3(256), 0, s,
                       f.src[0], n, L.ns, sample, total, L.nb);
    HK_LAUNCH_CHECK();
    int which = 0;
    if (int e = sort_pairs(sample, L.ns, k[0], id[0], k[1], id[1], s, which)) return e;
    hipLaunchKernelGGL(splitter_kernel, dim3((unsigned)((L.nb + 255) / 256)), dim3(256), 0, s,
                       k[which], id[which], L.ns, n, L.nb, spk, spi);
    HK_LAUNCH_CHECK();
    const unsigned gc = (unsigned)std::min<int64_t>((n + 8191) / 8192, 256);
    hipLaunchKernelGGL(bucket_count_kernel, dim3(gc), dim3(1024), 0, s, f.src[0], n, L.nb, spk, spi,
                       bucket, total);
    HK_LAUNCH_CHECK();
    hipLaunchKernelGGL(bucket_scan_kernel, dim3(1), dim3(1024), 0, s, total, L.nb, start, cursor);
    HK_LAUNCH_CHECK();
    const unsigned gs = (unsigned)((n + kScatNT * kScatE - 1) / (kScatNT * kScatE));
    hipLaunchKernelGGL(bucket_scatter_kernel, dim3(gs), dim3(kScatNT), 0, s, f, n, L.nb, bucket,
                       cursor, rec);
    HK_LAUNCH_CHECK();
    if (bucket_threads(n) == 512)
        hipLaunchKernelGGL(bucket_sort_kernel<512>, dim3((unsigned)L.nb), dim3(512), 0, s, rec, start,
                           f);
    else
        hipLaunchKernelGGL(bucket_sort_kernel<1024>, dim3((unsigned)L.nb), dim3(1024), 0, s, rec,
                           start, f);
    HK_LAUNCH_CHECK();
    return HK_OK;
}

}  // namespace

extern "C" size_t hk_lines_sort_workspace_bytes(int64_t nlines) {
    if (nlines < 0 || nlines > kMaxSortLines) return 0;
    return use_buckets(nlines) ? std::max(pair_bytes(nlines), bucket_layout(nlines).bytes + 256)
                               : pair_bytes(nlines);
}

extern "C" int hk_lines_sort(const hk_lines *in, hk_lines *out, void *workspace, size_t bytes,
                             hk_stream_t stream) {
    HK_CHECK_ARG(in && out, "hk_lines_sort: null argument");
    const int64_t n = in->nlines;
    HK_CHECK_ARG(n >= 0 && n <= kMaxSortLines, "hk_lines_sort: %lld lines (at most %lld per call)",
                 (long long)n, (long long)kMaxSortLines);
    HK_CHECK_ARG(in->form >= HK_FORM_HITRAN && in->form <= HK_FORM_SUPERLINE,
                 "hk_lines_sort: unknown line form %d", in->form);
    const double *src[7] = {in->nu, in->S, in->EL, in->A, in->delta, in->vy, in->n};
    const double *dst[7] = {out->nu, out->S, out->EL, out->A, out->delta, out->vy, out->n};
    if (n > 0) {
        for (int k = 0; k < 7; ++k) {
            HK_CHECK_ARG(src[k] && dst[k], "hk_lines_sort: field %d is NULL", k);
            HK_CHECK_ARG(src[k] != dst[k], "hk_lines_sort: field %d sorted in place", k);
        }
        HK_CHECK_ARG(!in->iso || (out->iso && out->iso != in->iso),
                     "hk_lines_sort: iso needs a distinct output array");
    }
    const size_t need = pair_bytes(n);
    if (bytes < need) {
        hk::set_error("hk_lines_sort: workspace of %zu bytes, %zu needed", bytes, need);
        return HK_ERR_WORKSPACE;
    }
    HK_CHECK_ARG(workspace, "hk_lines_sort: null workspace");
    // scalar fields travel with the lines
    const int niso = in->niso, form = in->form;
    double mass[HK_MAX_ISO], ab[HK_MAX_ISO], ss[HK_MAX_ISO];
    for (int k = 0; k < HK_MAX_ISO; ++k) {
        mass[k] = in->iso_mass[k]; ab[k] = in->iso_ab[k]; ss[k] = in->iso_sscale[k];
    }
    const double mad = in->max_abs_delta;
    const int32_t *iso_src = in->iso;
    out->nlines = n;
    out->niso = niso;
    out->form = form;
    for (int k = 0; k < HK_MAX_ISO; ++k) {
        out->iso_mass[k] = mass[k]; out->iso_ab[k] = ab[k]; out->iso_sscale[k] = ss[k];
    }
    out->max_abs_delta = mad;
    if (n == 0) return HK_OK;

    hipStream_t s = (hipStream_t)stream;
    char *w = (char *)hk::align_up((size_t)workspace, 256);
    // a workspace without room for the records still takes the merge passes
    if (use_buckets(n) && bytes >= bucket_layout(n).bytes + 256) {
        Columns c;
        for (int k = 0; k < 7; ++k) { c.src[k] = src[k]; c.dst[k] = (double *)dst[k]; }
        c.iso_src = iso_src;
        c.iso_dst = iso_src ? (int32_t *)out->iso : nullptr;
        return bucket_sort(c, n, w, s);
    }
    const size_t kb = hk::align_up((size_t)n * sizeof(double), 256);
    const size_t ib = hk::align_up((size_t)n * sizeof(int32_t), 256);
    double *k0 = (double *)w;
    int32_t *i0 = (int32_t *)(w + kb);
    double *k1 = (double *)(w + kb + ib);
    int32_t *i1 = (int32_t *)(w + 2 * kb + ib);
    // the last pass writes the sorted centres into out->nu
    const bool odd = merge_passes(n) % 2 != 0;
    int which = 0;
    if (int e = sort_pairs(src[0], n, odd ? k0 : (double *)dst[0], i0, odd ? (double *)dst[0] : k1,
                           i1, s, which))
        return e;
    const int32_t *ci = which ? i1 : i0;
    Fields f;
    for (int k = 0; k < 6; ++k) {
        f.src[k] = src[k + 1];
        f.dst[k] = (double *)dst[k + 1];
    }
    f.iso_src = iso_src;
    f.iso_dst = iso_src ? (int32_t *)out->iso : nullptr;
    hipLaunchKernelGGL(gather_kernel, dim3(grid_for(n)), dim3(256), 0, s, ci, n, f);
    HK_LAUNCH_CHECK();
    return HK_OK;
}
