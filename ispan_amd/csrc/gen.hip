// Device-side producers of the iSpan CSR layout: seeded synthetic edge
// lists (R-MAT, lattice) and an edge-list -> CSR-pair builder (sort, drop
// self-loops, deduplicate, offsets, transpose).  This is
// the format producer of graph_converter/txt_to_bin_{fw,bw}_int.cpp
// (:31-217), which does not deduplicate; here both directions are built in
// one pass over sorted (src,dst) keys.
//
// Randomness is a counter hash of (seed, draw index), so the edge multiset
// depends on nothing but the parameters.
#include <string.h>

#include <cstring>
#include <hip/hip_runtime.h>
#include <rocprim/rocprim.hpp>

#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <string>
#include <type_traits>

#include "common.h"

namespace ispan {

namespace {

// SplitMix64 finaliser (Steele, Lea, Flood 2014) as a stateless mixer.
__host__ __device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

uint64_t stream_base(uint64_t seed, uint64_t tag) {
    return mix64(seed * 0x632BE59BD9B4E019ull + tag * 0xD1B54A32D192ED03ull + 1ull);
}

// A directed edge as one sort key: src above the low `bits` bits, dst in
// them, bits = id_bits(V).  An absent edge is any self-loop, (0, 0) where
// there is nothing to keep: self-loops are dropped after the sort, so absent
// edges need no value outside the 2 * bits bits that are sorted.
int id_bits(int64_t V) {
    int b = 1;
    while (b < 31 && ((int64_t)1 << b) < V) ++b;
    return b;
}

template <class K>
__device__ __forceinline__ K edge_key(uint32_t s, uint32_t d, int bits) {
    return (K)(((K)s << bits) | (K)d);
}

// R-MAT draw e: at each of `scale` bit levels (most significant first) a
// 32-bit draw picks the quadrant: r < t1 (0,0), r < t2 (0,1), r < t3 (1,0),
// else (1,1).  Two levels share one 64-bit hash.
template <class K>
__global__ void k_rmat(int32_t V, int scale, int64_t m, uint32_t t1, uint32_t t2, uint32_t t3, uint64_t base, int bits,
                       K* keys) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < m; e += (int64_t)gridDim.x * blockDim.x) {
        uint32_t s = 0, d = 0;
        uint64_t h = 0;
        for (int k = 0; k < scale; ++k) {
            if ((k & 1) == 0) h = mix64(base ^ (((uint64_t)e << 5) | (uint64_t)(k >> 1)));
            const uint32_t r = (k & 1) ? (uint32_t)(h >> 32) : (uint32_t)h;
            const uint32_t sb = r >= t2;
            const uint32_t db = (r >= t1 && r < t2) || r >= t3;
            s |= sb << (scale - 1 - k);
            d |= db << (scale - 1 - k);
        }
        keys[e] = (s < (uint32_t)V && d < (uint32_t)V) ? edge_key<K>(s, d, bits) : (K)0;
    }
}

// n x n lattice: draw i < L covers lattice edge i (horizontal edges first,
// row-major), slots 2i and 2i+1; then L/100 uniform random directed edges.
template <class K>
__global__ void k_grid(int32_t n, uint32_t tb, uint64_t b1, uint64_t b2, int bits, K* keys) {
    const int64_t H = (int64_t)n * (n - 1), L = 2 * H, R = L / 100;
    const uint64_t V = (uint64_t)n * (uint64_t)n;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < L + R;
         i += (int64_t)gridDim.x * blockDim.x) {
        if (i < L) {
            int64_t u, v;
            if (i < H) {
                const int64_t r = i / (n - 1), c = i % (n - 1);
                u = r * n + c;
                v = u + 1;
            } else {
                const int64_t j = i - H;
                const int64_t r = j / n, c = j % n;
                u = r * n + c;
                v = u + n;
            }
            const uint64_t h = mix64(b1 ^ (uint64_t)i);
            const K uv = edge_key<K>((uint32_t)u, (uint32_t)v, bits), vu = edge_key<K>((uint32_t)v, (uint32_t)u, bits);
            if ((uint32_t)h < tb) {
                keys[2 * i] = uv;
                keys[2 * i + 1] = vu;
            } else {
                keys[2 * i] = (h >> 63) == 0 ? uv : vu;
                keys[2 * i + 1] = 0;
            }
        } else {
            const int64_t k = i - L;
            const uint64_t h = mix64(b2 ^ (uint64_t)k);
            const uint64_t s = ((h & 0xffffffffull) * V) >> 32, d = ((h >> 32) * V) >> 32;
            keys[2 * L + k] = edge_key<K>((uint32_t)s, (uint32_t)d, bits);
        }
    }
}

template <class K>
__global__ void k_pack(const int32_t* __restrict__ src, const int32_t* __restrict__ dst, int64_t m, int32_t V,
                       int bits, K* __restrict__ keys, int32_t* bad) {
    int wrong = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t s = src[i], d = dst[i];
        const bool ok = s >= 0 && s < V && d >= 0 && d < V;
        wrong |= !ok;
        keys[i] = ok ? edge_key<K>((uint32_t)s, (uint32_t)d, bits) : (K)0;
    }
    if (wrong) atomicOr(bad, 1);
}

// Row offsets come with a pass over the keys in row order: where a key's row
// is larger than the one before it, the rows in between and its own begin at
// its position.  (A binary search per row, bounded per 256 or 1024 rows, was
// bound by its scattered probes: 60 us for 2^20 rows over 16 M keys, twice a
// build.)  A lane writes up to kLaneRows rows itself, the wave the rest of a
// gap, and a gap of more than kGapRows rows is cut into pieces that k_gaps
// fills, one block each, so that a hole in the ids does not hold up one wave:
// of kGapRows rows, or in a large gap of so many that there are kGapPieces.
// (2 x 10^9 rows, one key: 36.0 ms of kernels with one lane listing 490,000
// pieces, 3.3 now; a search per row took 3.2.  Of 1,000 keys: 33.8, 5.1, 17.9.)
constexpr int kLaneRows = 4;
constexpr int kGapRows = 4096;
constexpr int kGapPieces = 8192;
constexpr int kGapBlocks = 2048;
struct Gap {
    int32_t lo, n, pos;
};
struct Rows {
    int32_t* beg;
    Gap* gaps;        // gap_capacity(V) entries
    int32_t* n_gaps;  // zero before the pass
};
// Pieces are full but for one per gap, and a gap has more than kGapRows rows.
int64_t gap_capacity(int64_t V) { return 2 * (V / kGapRows) + 2; }

// beg[r0 + 1 .. r1] = pos, for every lane's own r0, r1, pos (r1 <= r0: none).
// All 64 lanes call it.
__device__ __forceinline__ void begin_rows(const Rows& R, int32_t r0, int32_t r1, int32_t pos) {
    const int lane = threadIdx.x & 63;
    const int32_t n = r1 - r0;
#pragma unroll
    for (int k = 0; k < kLaneRows; ++k)
        if (k < n) R.beg[r0 + 1 + k] = pos;
    uint64_t more = __ballot(n > kLaneRows);
    while (more) {
        const int l = __ffsll((unsigned long long)more) - 1;
        more &= more - 1;
        const int32_t lo = __builtin_amdgcn_readlane(r0, l) + 1 + kLaneRows, hi = __builtin_amdgcn_readlane(r1, l);
        const int32_t p = __builtin_amdgcn_readlane(pos, l);
        if (hi - lo < kGapRows) {
            for (int32_t k = lane; k <= hi - lo; k += 64) R.beg[lo + k] = p;  // hi + 64 may be past int32
        } else {
            const int32_t rows = hi - lo + 1;
            const int32_t size = max(kGapRows, (rows / kGapPieces | 63) + 1);
            const int32_t pieces = (int32_t)(((int64_t)rows + size - 1) / size);
            int32_t at = 0;
            if (lane == 0) at = atomicAdd(R.n_gaps, pieces);
            at = __builtin_amdgcn_readfirstlane(at);
            for (int32_t k = lane; k < pieces; k += 64)
                R.gaps[at + k] = Gap{lo + k * size, min(size, rows - k * size), p};
        }
    }
}

__global__ void k_gaps(Rows R) {
    const int32_t n = *R.n_gaps;
    for (int32_t g = blockIdx.x; g < n; g += gridDim.x) {
        const Gap x = R.gaps[g];
        const int32_t head = min(x.n, (4 - (x.lo & 3)) & 3), quads = (x.n - head) / 4, tail = head + quads * 4;
        int32_t* beg = R.beg + x.lo;
        int4* wide = reinterpret_cast<int4*>(beg + head);  // the array starts aligned
        const int t = threadIdx.x;
        if (t < head) beg[t] = x.pos;
        if (t < x.n - tail) beg[tail + t] = x.pos;
        for (int32_t k = t; k < quads; k += blockDim.x) wide[k] = int4{x.pos, x.pos, x.pos, x.pos};
    }
}

// Sorted keys -> kept keys (the first of equal ones, no self-loops).  A wave
// owns a chunk of consecutive keys; k_keep_count counts what each keeps, and
// after a prefix sum over the chunks k_keep writes them in order, with their
// low halves as the adjacency, and the row offsets.  Bound by memory: two
// reads of the keys and one write.
//
// A chunk has kKeepChunk keys, or fewer (in whole steps of 64) where that would
// be less than kKeepFull chunks: with few keys over many rows the waves are
// needed for the rows (2^24 rows, 70,000 keys: 777 us of kernels with 1024
// keys a wave, 201 with 64, 463 with a search per row).
constexpr int kKeepChunk = 1024;
constexpr int kKeepFull = 2048;
constexpr int kKeepWaves = 4;
int keep_chunk(int64_t m) {
    return (int)std::max<int64_t>(64, std::min<int64_t>(kKeepChunk, (m / kKeepFull + 63) & ~(int64_t)63));
}

// f(valid, key, keep, previous key) for the 64 keys of every step.
template <class K, class F>
__device__ __forceinline__ void each_key(const K* __restrict__ keys, int64_t m, int bits, int per, int64_t chunk,
                                         F&& f) {
    const int lane = threadIdx.x & 63;
    const K low = ((K)1 << bits) - 1;
    const int64_t i0 = chunk * per, i1 = min(i0 + per, m);
    for (int64_t ib = i0; ib < i1; ib += 64) {
        const int64_t i = ib + lane;
        const bool valid = i < i1;
        const K k = valid ? keys[i] : 0, before = valid && i > 0 ? keys[i - 1] : 0;
        f(i, valid, k, valid && (K)(k >> bits) != (k & low) && (i == 0 || before != k), before);
    }
}

template <class K>
__global__ __launch_bounds__(64 * kKeepWaves) void k_keep_count(const K* __restrict__ keys, int64_t m, int bits, int per,
                                                                int64_t chunks, int32_t* __restrict__ counts) {
    for (int64_t c = (int64_t)blockIdx.x * kKeepWaves + threadIdx.x / 64; c < chunks; c += (int64_t)gridDim.x * kKeepWaves) {
        int n = 0;
        each_key<K>(keys, m, bits, per, c, [&](int64_t, bool, K, bool keep, K) { n += __popcll(__ballot(keep)); });
        if ((threadIdx.x & 63) == 0) counts[c] = n;
    }
}

template <class K>
__global__ __launch_bounds__(64 * kKeepWaves) void k_keep(const K* __restrict__ keys, int64_t m, int bits, int per,
                                                          int64_t chunks, const int64_t* __restrict__ start,
                                                          K* __restrict__ kept, int32_t* __restrict__ adj, Rows R,
                                                          int32_t V) {
    const int lane = threadIdx.x & 63;
    const K low = ((K)1 << bits) - 1;
    for (int64_t c = (int64_t)blockIdx.x * kKeepWaves + threadIdx.x / 64; c < chunks; c += (int64_t)gridDim.x * kKeepWaves) {
        int64_t p = start[c];
        each_key<K>(keys, m, bits, per, c, [&](int64_t i, bool valid, K k, bool keep, K before) {
            const uint64_t mask = __ballot(keep);
            const int64_t q = p + __popcll(mask & ((1ull << lane) - 1));
            if (keep) {
                kept[q] = k;
                adj[q] = (int32_t)(k & low);
            }
            const int32_t row = (int32_t)(k >> bits);
            begin_rows(R, i == 0 ? -1 : (int32_t)(before >> bits), valid ? row : -1, (int32_t)q);
            p += __popcll(mask);
            const bool last = i == m - 1;  // the rows after the last key's
            if (__ballot(last)) begin_rows(R, row, last ? V : -1, (int32_t)p);
        });
    }
}

// Kept keys in (dst, src) order -> the transposed rows.
template <class K>
__global__ __launch_bounds__(64 * kKeepWaves) void k_transposed(const K* __restrict__ keys, int64_t E, int bits, int per,
                                                                int64_t chunks, int32_t* __restrict__ adj, Rows R,
                                                                int32_t V) {
    const K low = ((K)1 << bits) - 1;
    for (int64_t c = (int64_t)blockIdx.x * kKeepWaves + threadIdx.x / 64; c < chunks; c += (int64_t)gridDim.x * kKeepWaves)
        each_key<K>(keys, E, bits, per, c, [&](int64_t i, bool valid, K k, bool, K before) {
            if (valid) adj[i] = (int32_t)(k >> bits);
            const int32_t row = (int32_t)(k & low);
            begin_rows(R, i == 0 ? -1 : (int32_t)(before & low), valid ? row : -1, (int32_t)i);
            const bool last = i == E - 1;
            if (__ballot(last)) begin_rows(R, row, last ? V : -1, (int32_t)E);
        });
}

__global__ void k_widen_keys(const uint32_t* __restrict__ k, int64_t m, uint64_t* out) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = (uint64_t)k[i] << 32;
}

// beg[v] = first i with keys[i] >= v<<32 over sorted keys.
__global__ void k_beg_from_keys(const uint64_t* __restrict__ keys, int64_t m, int32_t V, int32_t* beg) {
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v <= V; v += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t key = (uint64_t)v << 32;
        int64_t lo = 0, hi = m;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (keys[mid] < key) lo = mid + 1;
            else hi = mid;
        }
        beg[v] = (int32_t)lo;
    }
}

#define GK(call)                                                             \
    do {                                                                     \
        hipError_t e_ = (call);                                              \
        if (e_ != hipSuccess) {                                              \
            (void)hipGetLastError(); /* or the next launch reports it */     \
            err = std::string(#call) + ": " + hipGetErrorString(e_);         \
            rc = e_ == hipErrorOutOfMemory ? -3 : -4;                        \
            goto done;                                                       \
        }                                                                    \
    } while (0)

constexpr int kGrid = 4096;

}  // namespace

// A builder's scratch: the keys twice, the counts and starts of their chunks,
// the gaps of one direction, and three counters (gaps of each direction, bad
// endpoints).
template <class K>
struct BuildMem {
    K *keys, *alt;
    int32_t* counts;
    int64_t* start;  // first kept position of every chunk, then their total
    Gap* gaps;
    int32_t* n;
    int per;  // keys a chunk
    int64_t chunks;

    BuildMem(void* base, int32_t V, int64_t m, size_t* bytes = nullptr) {
        per = keep_chunk(m);
        chunks = (m + per - 1) / per;
        size_t off = 0;
        auto take = [&](size_t size) {
            char* p = static_cast<char*>(base) + off;
            off += (size + 255) & ~(size_t)255;
            return static_cast<void*>(p);
        };
        keys = static_cast<K*>(take((size_t)std::max<int64_t>(m, 1) * sizeof(K)));
        alt = static_cast<K*>(take((size_t)std::max<int64_t>(m, 1) * sizeof(K)));
        counts = static_cast<int32_t*>(take((size_t)(chunks + 1) * 4));
        start = static_cast<int64_t*>(take((size_t)(chunks + 1) * 8));
        gaps = static_cast<Gap*>(take((size_t)gap_capacity(V) * sizeof(Gap)));
        n = static_cast<int32_t*>(take(12));
        if (bytes) *bytes = off;
    }
};

// How keys are sorted.  By radix passes from 2^18 keys on: the library's own
// line, 2^20, has merges up to there, whose time steps up with the size (64-bit
// keys, 40 / 17 bits: 200,000 keys 67 / 63 us merged, 99 / 63 by passes; 400,000
// keys 123 / 118 and 106 / 68; a million 177 / 170 and 123 / 80).  And 1024
// threads of 8 keys a block, which for 64-bit keys is faster than its choice
// from 2.5 M keys on (16 M keys of 40 bits 547 -> 510 us) and otherwise equal.
using KeySort = rocprim::radix_sort_config<
    rocprim::default_config, rocprim::default_config,
    rocprim::radix_sort_onesweep_config<rocprim::kernel_config<1024, 8>, rocprim::kernel_config<1024, 8>, 8,
                                        rocprim::block_radix_rank_algorithm::match>,
    1 << 18>;

// M.keys[0, m) (edge_key form) -> CSR pair; M.n is zero.  Only the 2 * bits
// bits of a key are sorted, in 32-bit keys when they fit (V <= 65536); the
// kept keys, then in (src, dst) order, are sorted by dst alone for the
// transposed rows: the sort is stable, so each row stays in src order.  At
// 2^20 vertices that is 5 + 3 radix passes instead of the 8 + 8 of full 64-bit
// keys.
template <class K>
int csr_from_keys(hipStream_t s, Workspace& sort, const BuildMem<K>& M, int32_t V, int64_t m, int32_t** fwb,
                  int32_t** fwa, int32_t** bwb, int32_t** bwa, int64_t* E_out, std::string& err) {
    int rc = 0;
    const int bits = id_bits(V);
    const int per = M.per;
    const int64_t chunks = M.chunks;
    const int keep_grid = (int)std::max<int64_t>(1, std::min<int64_t>(kGrid, (chunks + kKeepWaves - 1) / kKeepWaves));
    size_t b1 = 0, b2 = 0;
    int64_t E = 0;
    rocprim::double_buffer<K> buf(M.keys, M.alt);
    if (m > 0) {
        GK(rocprim::radix_sort_keys<KeySort>(nullptr, b1, buf, (size_t)m, 0, 2 * bits, s));
        GK(rocprim::exclusive_scan(nullptr, b2, M.counts, M.start, (int64_t)0, (size_t)chunks + 1,
                                   rocprim::plus<int64_t>(), s));
        GK(sort.ensure(std::max(b1, b2) + 256));
        b1 = b2 = sort.cap;
        GK(rocprim::radix_sort_keys<KeySort>(sort.p, b1, buf, (size_t)m, 0, 2 * bits, s));
        hipLaunchKernelGGL(k_keep_count<K>, dim3(keep_grid), dim3(64 * kKeepWaves), 0, s, buf.current(), m, bits,
                           per, chunks, M.counts);
        GK(hipGetLastError());
        // one entry more than chunks: the last start is the total (the last
        // count is not read into it)
        GK(rocprim::exclusive_scan(sort.p, b2, M.counts, M.start, (int64_t)0, (size_t)chunks + 1,
                                   rocprim::plus<int64_t>(), s));
        GK(hipMemcpyAsync(&E, M.start + chunks, 8, hipMemcpyDeviceToHost, s));
        GK(hipStreamSynchronize(s));
    }
    if (E > INT32_MAX) {
        err = "edge count exceeds int32";
        rc = -1;
        goto done;
    }
    GK(hipMalloc(fwb, ((size_t)V + 1) * 4));
    GK(hipMalloc(bwb, ((size_t)V + 1) * 4));
    GK(hipMalloc(fwa, (size_t)std::max<int64_t>(E, 1) * 4));
    GK(hipMalloc(bwa, (size_t)std::max<int64_t>(E, 1) * 4));
    if (E > 0) {
        K* kept = buf.alternate();
        Rows R{*fwb, M.gaps, M.n};
        hipLaunchKernelGGL(k_keep<K>, dim3(keep_grid), dim3(64 * kKeepWaves), 0, s, buf.current(), m, bits, per, chunks,
                           M.start, kept, *fwa, R, V);
        GK(hipGetLastError());
        hipLaunchKernelGGL(k_gaps, dim3(kGapBlocks), dim3(256), 0, s, R);
        GK(hipGetLastError());
        buf = rocprim::double_buffer<K>(kept, buf.current());
        // fewer keys can take another of the sort's methods, with more scratch
        GK(rocprim::radix_sort_keys<KeySort>(nullptr, b1, buf, (size_t)E, 0, bits, s));
        GK(sort.ensure(b1));
        b1 = sort.cap;
        GK(rocprim::radix_sort_keys<KeySort>(sort.p, b1, buf, (size_t)E, 0, bits, s));
        R.beg = *bwb;
        R.n_gaps = M.n + 1;
        hipLaunchKernelGGL(k_transposed<K>, dim3(keep_grid), dim3(64 * kKeepWaves), 0, s, buf.current(), E, bits, per,
                           (E + per - 1) / per, *bwa, R, V);
        GK(hipGetLastError());
        hipLaunchKernelGGL(k_gaps, dim3(kGapBlocks), dim3(256), 0, s, R);
        GK(hipGetLastError());
    } else {
        GK(launch_fill_i32(*fwb, 0, (int64_t)V + 1, kGrid, s));
        GK(launch_fill_i32(*bwb, 0, (int64_t)V + 1, kGrid, s));
    }
    GK(hipStreamSynchronize(s));
    *E_out = E;
done:
    return rc;
}

// Stable CSR of one direction: rows in input order, duplicates and
// self-loops kept (the byte layout of graph_converter/txt_to_bin_fw_int.cpp
// :146-181).  key[i] = row of edge i, val[i] = its other endpoint.
int csr_stable_one(hipStream_t s, int32_t V, int64_t m, const int32_t* key, const int32_t* val, int32_t** beg,
                   int32_t** adj, std::string& err) {
    int rc = 0;
    uint32_t *k2 = nullptr, *kin = nullptr;
    int32_t* v2 = nullptr;
    void* tmp = nullptr;
    size_t bytes = 0;
    uint64_t* keys64 = nullptr;
    *beg = *adj = nullptr;
    unsigned end_bit = 1;
    while (end_bit < 32 && ((int64_t)1 << end_bit) < (int64_t)V) ++end_bit;
    GK(hipMalloc(&kin, (size_t)std::max<int64_t>(m, 1) * 4));
    GK(hipMalloc(&k2, (size_t)std::max<int64_t>(m, 1) * 4));
    GK(hipMalloc(&v2, (size_t)std::max<int64_t>(m, 1) * 4));
    GK(hipMalloc(adj, (size_t)std::max<int64_t>(m, 1) * 4));
    GK(hipMalloc(beg, ((size_t)V + 1) * 4));
    GK(hipMalloc(&keys64, (size_t)std::max<int64_t>(m, 1) * 8));
    if (m > 0) {
        GK(hipMemcpyAsync(kin, key, (size_t)m * 4, hipMemcpyDeviceToDevice, s));
        GK(rocprim::radix_sort_pairs(nullptr, bytes, kin, k2, val, v2, (size_t)m, 0, end_bit, s));
        GK(hipMalloc(&tmp, bytes + 256));
        bytes += 256;
        GK(rocprim::radix_sort_pairs(tmp, bytes, kin, k2, val, v2, (size_t)m, 0, end_bit, s));
        GK(hipMemcpyAsync(*adj, v2, (size_t)m * 4, hipMemcpyDeviceToDevice, s));
        hipLaunchKernelGGL(k_widen_keys, dim3(kGrid), dim3(256), 0, s, k2, (int64_t)m, keys64);
        GK(hipGetLastError());
    }
    hipLaunchKernelGGL(k_beg_from_keys, dim3(kGrid), dim3(256), 0, s, keys64, (int64_t)m, V, *beg);
    GK(hipGetLastError());
    GK(hipStreamSynchronize(s));
done:
    for (void* p : {(void*)kin, (void*)k2, (void*)v2, tmp, (void*)keys64})
        if (p) (void)hipFree(p);
    if (rc) {
        if (*beg) (void)hipFree(*beg);
        if (*adj) (void)hipFree(*adj);
        *beg = *adj = nullptr;
    }
    return rc;
}

int launched(std::string& err) {
    const hipError_t e = hipGetLastError();
    if (e == hipSuccess) return 0;
    err = std::string("kernel launch: ") + hipGetErrorString(e);
    return e == hipErrorOutOfMemory ? -3 : -4;
}

// Scratch for m edges over V vertices and, on it, fill(memory) (which writes
// the keys) and csr_from_keys.
template <class K, class Fill>
int csr_from_filled(hipStream_t s, GenScratch& w, int32_t V, int64_t m, Fill&& fill, int32_t** fwb, int32_t** fwa,
                    int32_t** bwb, int32_t** bwa, int64_t* E, std::string& err) {
    int rc = 0;
    size_t bytes = 0;
    BuildMem<K> size(nullptr, V, m, &bytes);
    *fwb = *fwa = *bwb = *bwa = nullptr;
    GK(w.m.ensure(bytes));
    {
        const BuildMem<K> M(w.m.p, V, m);
        GK(launch_fill_i32(M.n, 0, 3, 1, s));
        rc = fill(M);
        if (!rc) rc = csr_from_keys<K>(s, w.sort, M, V, m, fwb, fwa, bwb, bwa, E, err);
    }
done:
    if (rc) {
        (void)hipStreamSynchronize(s);  // nothing queued may outlive what is freed
        for (int32_t** p : {fwb, fwa, bwb, bwa}) {
            if (*p) (void)hipFree(*p);
            *p = nullptr;
        }
    }
    if (w.m.cap + w.sort.cap > kKeepScratch) {
        w.m.release();
        w.sort.release();
    }
    return rc;
}

template <class Fill>
int csr_from(hipStream_t s, GenScratch& w, int32_t V, int64_t m, Fill&& fill, int32_t** fwb, int32_t** fwa,
             int32_t** bwb, int32_t** bwa, int64_t* E, std::string& err) {
    if (2 * id_bits(V) <= 32) return csr_from_filled<uint32_t>(s, w, V, m, fill, fwb, fwa, bwb, bwa, E, err);
    return csr_from_filled<uint64_t>(s, w, V, m, fill, fwb, fwa, bwb, bwa, E, err);
}

int gen_rmat_device(hipStream_t s, GenScratch& w, int32_t V, double ef, double a, double b, double c, uint64_t seed,
                    int32_t** fwb, int32_t** fwa, int32_t** bwb, int32_t** bwa, int64_t* E, std::string& err) {
    if (V <= 0 || ef < 0 || a < 0 || b < 0 || c < 0 || a + b + c > 1.0) return -1;
    int scale = 0;
    while (((int64_t)1 << scale) < (int64_t)V) ++scale;
    const int64_t m = llround(ef * (double)V);
    const double S = 4294967296.0;
    const uint32_t t1 = (uint32_t)(a * S), t2 = (uint32_t)((a + b) * S), t3 = (uint32_t)((a + b + c) * S);
    auto fill = [&](const auto& M) {
        using K = std::remove_pointer_t<decltype(M.keys)>;
        hipLaunchKernelGGL(k_rmat<K>, dim3(kGrid), dim3(256), 0, s, V, scale, m, t1, t2, t3, stream_base(seed, 1),
                           id_bits(V), M.keys);
        return launched(err);
    };
    return csr_from(s, w, V, m, fill, fwb, fwa, bwb, bwa, E, err);
}

int gen_grid_device(hipStream_t s, GenScratch& w, int32_t n, double p_bidir, uint64_t seed, int32_t** fwb,
                    int32_t** fwa, int32_t** bwb, int32_t** bwa, int64_t* E, std::string& err) {
    if (n < 2 || (int64_t)n * n > INT32_MAX || p_bidir < 0 || p_bidir > 1) return -1;
    const int64_t L = 2 * (int64_t)n * (n - 1), R = L / 100, m = 2 * L + R;
    const uint32_t tb = (uint32_t)(p_bidir * 4294967296.0);
    auto fill = [&](const auto& M) {
        using K = std::remove_pointer_t<decltype(M.keys)>;
        hipLaunchKernelGGL(k_grid<K>, dim3(kGrid), dim3(256), 0, s, n, tb, stream_base(seed, 2), stream_base(seed, 3),
                           id_bits((int64_t)n * n), M.keys);
        return launched(err);
    };
    return csr_from(s, w, n * n, m, fill, fwb, fwa, bwb, bwa, E, err);
}

int build_csr_device(hipStream_t s, GenScratch& w, int32_t V, int64_t m, const int32_t* src, const int32_t* dst,
                     int32_t** fwb, int32_t** fwa, int32_t** bwb, int32_t** bwa, int64_t* E, std::string& err) {
    if (V < 0 || m < 0) return -1;
    auto fill = [&](const auto& M) {
        using K = std::remove_pointer_t<decltype(M.keys)>;
        if (m == 0) return 0;
        int32_t bad = 0;
        hipLaunchKernelGGL(k_pack<K>, dim3(kGrid), dim3(256), 0, s, src, dst, m, V, id_bits(V), M.keys, M.n + 2);
        if (int e = launched(err)) return e;
        if (hipMemcpyAsync(&bad, M.n + 2, 4, hipMemcpyDeviceToHost, s) != hipSuccess ||
            hipStreamSynchronize(s) != hipSuccess) {
            err = "reading the edge check failed";
            return -4;
        }
        if (bad) {
            err = "edge endpoint outside [0, V)";
            return -2;
        }
        return 0;
    };
    return csr_from(s, w, V, m, fill, fwb, fwa, bwb, bwa, E, err);
}

}  // namespace ispan
