// The giant-SCC phase as one cooperative, persistent kernel: trim-1-first and
// the pivot (src/trim_1_gfq.h:9-33, src/scc_common.h:92-150), the forward
// and backward direction-optimising traversals (src/fw_bw.h:396-698,
// 944-1248) and the relabelling of what they found, with grid-wide barriers
// between levels instead of host round trips.
//
// Every block runs the same control flow: each barrier gives all blocks the
// same totals, they take the same top-down/bottom-up decision, so every block
// passes the same barriers.  Data written by other
// blocks before a barrier is read with plain loads after a barrier that
// invalidates the caches, and with device-coherent loads after one that does
// not; device-coherent loads are also kept for what other blocks change
// during the same phase.
#include "common.h"
#include "device_util.h"

namespace ispan {
using namespace dev;

namespace {

// Polls that a barrier waits at most, each a round trip past the L2 and a short
// sleep (10 s and more in all); beyond them the kernel aborts.
constexpr int kSpinCap = 1 << 24;
constexpr int kBarWords = 8;       // payload words a barrier can carry per block
static_assert(kBarWords * 2 * 8 == kBarBytesPerBlock, "two record buffers of 8-byte words");
// One 1024-thread block per CU: every block invalidates its caches after a
// barrier, so fewer, larger blocks make the barrier cheaper.
constexpr int kGBlock = 1024;
constexpr int kW = kGBlock / kWave;

// Per-direction state of the joint traversal (the same in every block).
struct Dir {
    int32_t mode;     // 0 top-down, 1 bottom-up, 2 top-down to exhaustion
    int32_t L;        // levels done
    int32_t visited;  // vertices claimed, the roots excluded
    int32_t nq, nh;   // next level's queue entries and hub work items (nq: the finds to gather, before a gathering level)
};
// What the traversal goes on with (Smem::flow): which directions are still
// traversing; which had a bottom-up level last and have a top-down one next,
// which starts from the bitmaps instead of a queue.
constexpr int kLive = 1, kGather = 4, kFailed = 16;  // of direction d: kLive << d, kGather << d

struct Smem {
    Dir dir[2];
    int flow;
    int32_t off[kGBlock];    // top-down tile: exclusive degree prefix, first edge
    int32_t start[kGBlock];
    int tmp[kW];
    int64_t red[kW];
    int64_t red2[kW];
    int32_t bi[kW];
    alignas(16) uint32_t bv[kBarWords][kW];  // a barrier's payload per wave
    int64_t tot[2][kBarWords];               // its totals over the grid, per reading wave
    int ok[2];
    int steps;  // levels a narrow frontier may still take in its block
    int32_t narrow[2][kW];  // the same: every wave's staged entries, and their edges
    int32_t wcnt[2][kW];    // block flushes: per-wave counts and bases of up to two counters
    int32_t wbase[2][kW];
    int32_t hv[kW][kWave];  // per-wave staged hub vertices: id, first edge, degree
    int32_t hs[kW][kWave];
    int32_t hd[kW][kWave];
};

// Per-wave staging, kPairCap 8-byte entries a wave: top-down queue entries,
// or kWaveBuf vertex ids in the phases that queue ids.  It is dynamic LDS,
// placed after Smem, so that Smem's arrays stay within the 64 KB an LDS
// instruction's immediate offset reaches.
constexpr int kPairCap = 512;
static_assert(kWaveBuf * 4 <= kPairCap * 8, "the id view fits the staging");
static_assert((kPairCap & (kPairCap - 1)) == 0, "the in-place ring indexes with a mask");
extern __shared__ uint64_t stage_lds[];

// The launch's arguments, read from the kernel argument segment.  args()
// hides where the address comes from, so that what a phase reads of them is
// loaded in that phase: read once at the start they take more scalar
// registers than there are, and every use of a spilled one is a move from a
// vector register's lane.
typedef const GiantArgs __attribute__((address_space(4))) KernelArgs;
__device__ __forceinline__ KernelArgs& kernel_args() {
    KernelArgs* p = (KernelArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *p;
}

struct Ctx {
    __device__ KernelArgs& args() const { return kernel_args(); }
    int G, b, tid, lane, wave;
    Smem& sm;
    uint32_t nbar;  // barriers this launch has passed (the same in every block)
    int64_t edges_td, edges_bu, found_td, found_bu;  // work counters of this wave (wave-uniform)
    // this wave's staging, as 8-byte entries or as ids
    __device__ uint64_t* stage() const { return stage_lds + wave * kPairCap; }
    __device__ int32_t* stage32() const { return reinterpret_cast<int32_t*>(stage()); }
};

// Waits until every vector-memory access this wave has issued (loads,
// stores, atomics) has completed: s_waitcnt vmcnt(0), with no cache
// maintenance.  An sc1 store or a device atomic has completed once it is
// visible at device scope, so after this wait the wave's device-coherent
// writes are visible to every other XCD.  (A release fence does not give
// this: at workgroup scope it emits no wait at all, since the block's waves
// share one L1; at agent scope it also writes back the whole L2.)
__device__ __forceinline__ void wait_vm() { __builtin_amdgcn_s_waitcnt(0x0F70); }  // vmcnt(0), others unchanged

// Grid barrier that carries a payload.  Every block publishes one record, NW
// (4 or 8) 8-byte words of {tag, 32-bit value}, and wave 0 of every block
// reads every block's record until all of them bear this barrier's tag: one
// store and one read across the chip, with nothing passed on in between.
// What the blocks contribute comes with the arrival itself, so a reduction
// costs no further round trip.  A counter tree (32 group counters, a top
// counter, a generation word) needs three dependent atomics, and carried
// sums add an exchange and an add at each of its levels; same box, 256 blocks
// of 1024 threads, back to back: 4.2 us with 2 sums and 5.3 us with 4, against
// 2.1 us with 4 words and 2.8 us with 8 here.
//
// Lane l of the reading wave takes word l % NW of record l / NW, then the
// same of the next 64 / NW records, so a load instruction covers 512
// consecutive bytes; one record a lane takes 3.1 and 4.4 us instead.  A lane
// has 16 loads in flight (more spill), so with 8 words the records of 256
// blocks take two waves, or two rounds of one wave where the barrier also
// acquires: only one wave may do that (four at once: 8.9 us a barrier).
//
// Tags: each barrier's is one more than the last, counted on over the
// launches on one state (GiantArgs::bar_base), so no record left from before
// bears it, and the records need no clearing.  Consecutive barriers use the
// two record buffers in turn: a block writes a buffer again only after a
// barrier that every block reached after reading it.
//
// Memory protocol: everything a block writes for other blocks is written
// device-coherently (atomics or st_agent), so arriving needs no L2
// writeback.  It does need every one of those writes to have completed
// before the record is written, and they are issued by all 16 waves while
// only wave 0 writes the record: so every wave waits for its own accesses
// (wait_vm) before the block barrier.  A block that reads a record of this
// tag therefore sees every write its block made before the barrier, once it
// invalidates its L1 and its XCC's L2 (device-scope acquire) or reads the
// data with device-coherent loads.
//
// ACQ: after the wait, invalidate this CU's L1 and this XCC's L2 (agent
// acquire), so that plain loads see what other blocks wrote before the
// barrier.  Without it only coherent loads and atomics may read such data
// (and loads that tolerate stale values).
//
// src() gives lane w < NW of wave 0 the block's word w, after the block
// barrier; fold.take(record, value) is called in the reading waves for every
// word of every record (lanes as above), then fold.finish() once per wave.
//
// Returns false (and flags an error) if the wait exceeds kSpinCap.
template <int NW, bool ACQ, class Src, class Fold>
__device__ __forceinline__ bool gsync_with(Ctx& c, Src src, Fold& fold) {
    static_assert(NW == 4 || NW == 8, "record size");
    constexpr int kReaders = ACQ ? 1 : NW / 4;  // reading waves
    Smem& sm = c.sm;
    const uint32_t nb = ++c.nbar;
    wait_vm();  // this wave's writes for other blocks have completed
    __syncthreads();
    if (c.wave < kReaders) {
        KernelArgs& a = c.args();
        const uint32_t tag = a.bar_base + nb;
        uint64_t* rec = a.bar + (int64_t)(tag & 1) * c.G * kBarWords;
        if (c.wave == 0) {
            const uint32_t mine = src();  // by every lane
            if (c.lane < NW) st_agent(&rec[c.b * NW + c.lane], ((uint64_t)tag << 32) | mine);
        }
        if (c.tid == 0) {  // diagnostics: barriers arrived at, and passed
            a.dbg[c.b] = (int32_t)nb;
            a.dbg[c.G + c.b] = (int32_t)nb - 1;
        }
        constexpr int K = 16;  // loads a lane has in flight
        const int words = c.G * NW;
        int ok = 1;
        for (int base = c.wave * K * kWave; base < words && ok; base += kReaders * K * kWave) {
            uint64_t x[K];
            uint32_t todo = 0;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                x[k] = 0;
                todo |= base + k * kWave + c.lane < words ? 1u << k : 0u;
            }
            int spins = 0;
            while (true) {
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if ((todo >> k) & 1u) x[k] = load_agent(&rec[base + k * kWave + c.lane]);
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if ((uint32_t)(x[k] >> 32) == tag) todo &= ~(1u << k);
                if (!__ballot(todo != 0)) break;
                __builtin_amdgcn_s_sleep(1);
                if (++spins > kSpinCap) {
                    if (c.lane == 0) atomicOr(&a.gs->err.v, 1);
                    ok = 0;
                    break;
                }
            }
#pragma unroll
            for (int k = 0; k < K; ++k) fold.take((base + k * kWave + c.lane) / NW, (uint32_t)x[k]);
        }
        fold.finish(sm, c.wave);
        if (ACQ) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // this CU's L1 and this XCC's L2
        else __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        if (c.lane == 0) sm.ok[c.wave] = ok;
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(kReaders == 1 ? sm.ok[0] : (sm.ok[0] & sm.ok[1]));
}

// The payload as each wave stages it: word w's value of this wave, the same
// in every lane.
template <int NW>
__device__ __forceinline__ void stage_words(Ctx& c, const uint32_t (&v)[NW]) {
    uint32_t x = v[0];
#pragma unroll
    for (int w = 1; w < NW; ++w) x = c.lane == w ? v[w] : x;
    if (c.lane < NW) c.sm.bv[c.lane][c.wave] = x;
}

// Sum of word lane % kBarWords over the waves.
__device__ __forceinline__ uint32_t staged_sum(const Smem& sm, int lane) {
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < kW; ++i) s += sm.bv[lane & (kBarWords - 1)][i];
    return s;
}

// Folds the lanes that hold the same word (lane % NW), op over them; every
// lane gets its word's result.
template <int NW, class T, class Op>
__device__ __forceinline__ T fold_lanes(T s, Op op) {
#pragma unroll
    for (int d = NW; d < kWave; d <<= 1) s = op(s, (T)__shfl_xor(s, d, kWave));
    return s;
}

// Totals of every word into sm.tot.
template <int NW>
struct SumFold {
    uint64_t s = 0;
    __device__ void take(int, uint32_t x) { s += x; }
    __device__ void finish(Smem& sm, int wave) {
        s = fold_lanes<NW>(s, [](uint64_t p, uint64_t q) { return p + q; });
        if (lane_id() < NW) sm.tot[wave][lane_id()] = (int64_t)s;
    }
};

// Barrier whose payload is summed: v holds each wave's values (the same in
// every lane); out receives the totals.
template <int NW, bool ACQ>
__device__ __forceinline__ bool gsync_sum(Ctx& c, const uint32_t (&v)[NW], int64_t (&out)[NW]) {
    stage_words<NW>(c, v);
    SumFold<NW> f;
    if (!gsync_with<NW, ACQ>(c, [&c]() { return staged_sum(c.sm, c.lane); }, f)) return false;
#pragma unroll
    for (int w = 0; w < NW; ++w)
        out[w] = lane_get((NW == 8 && !ACQ) ? c.sm.tot[0][w] + c.sm.tot[1][w] : c.sm.tot[0][w], 0);
    return true;
}

struct NoFold {
    __device__ void take(int, uint32_t) {}
    __device__ void finish(Smem&, int) {}
};

// Barrier without a payload.
template <bool ACQ = true>
__device__ __forceinline__ bool gsync(Ctx& c) {
    NoFold f;
    return gsync_with<4, ACQ>(c, []() { return 0u; }, f);
}

// The largest (product, -id) over the records of {product high, product low,
// id, survivors}, and the survivors' sum, into sm.tot[0][0..2].
struct PivotFold {
    int64_t bestp = 0;
    int32_t besti = INT32_MAX;
    uint64_t surv = 0;
    __device__ void take(int, uint32_t x) {
        // the four words of a record lie in the four lanes of a quad
        const int32_t y = (int32_t)x;
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, y, 0x00, 0xF, 0xF, false);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, y, 0x55, 0xF, 0xF, false);
        const int32_t id = __builtin_amdgcn_update_dpp(0, y, 0xAA, 0xF, 0xF, false);
        const int64_t p = (int64_t)(((uint64_t)hi << 32) | lo);
        if (pivot_better(p, id, bestp, besti)) {
            bestp = p;
            besti = id;
        }
        surv += x;  // of lanes 3, 7, ..: the others' sums are not used
    }
    __device__ void finish(Smem& sm, int) {
#pragma unroll
        for (int d = 4; d < kWave; d <<= 1) {
            const int64_t op = __shfl_xor(bestp, d, kWave);
            const int32_t oi = __shfl_xor(besti, d, kWave);
            if (pivot_better(op, oi, bestp, besti)) {
                bestp = op;
                besti = oi;
            }
        }
        surv = fold_lanes<4>(surv, [](uint64_t p, uint64_t q) { return p + q; });
        if (lane_id() == 3) {
            sm.tot[0][0] = bestp;
            sm.tot[0][1] = besti;
            sm.tot[0][2] = (int64_t)surv;
        }
    }
};

// Totals of every word but word 2, whose largest value is taken, into
// sm.tot[0], and into sm.tot[1][0] the sum of word 0 over the blocks before
// this one.
struct PostFold {
    int b;
    uint64_t s = 0, pre = 0;
    __device__ void take(int rec, uint32_t x) {
        s = (lane_id() & 7) == 2 ? max(s, (uint64_t)x) : s + x;
        pre += rec < b ? x : 0u;
    }
    __device__ void finish(Smem& sm, int) {
        const bool mx = (lane_id() & 7) == 2;
        s = fold_lanes<8>(s, [mx](uint64_t p, uint64_t q) { return mx ? max(p, q) : p + q; });
        pre = fold_lanes<8>(pre, [](uint64_t p, uint64_t q) { return p + q; });
        if (lane_id() < 8) sm.tot[0][lane_id()] = (int64_t)s;
        if (lane_id() == 0) sm.tot[1][0] = (int64_t)pre;
    }
};

// Sum of a per-thread value over the block (every thread gets it).
__device__ __forceinline__ int64_t block_sum(int64_t x, Smem& sm) {
    static_assert(kW == 16, "one DPP row holds the wave totals");
    x = wave_sum(x);
    if (lane_id() == 0) sm.red[wave_id()] = x;
    __syncthreads();
    x = row_incl(sm.red[lane_id() & 15], (int64_t)0, [](int64_t a, int64_t b) { return a + b; });
    x = lane_get(x, 15);
    __syncthreads();
    return x;
}

// Per-wave staging of hub vertices in LDS; a flush turns them into
// kGiantChunk-edge work items with one atomic for the whole batch.
struct HubStage {
    int32_t* v;
    int32_t* s;
    int32_t* d;
    int n;              // wave-uniform fill
    uint32_t sent = 0;  // work items written so far (wave-uniform)
    int chunk = kGiantChunk;  // edges per work item
};

__device__ __forceinline__ void hub_flush(HubStage& hs, HubItem* hout, int32_t* hn_out) {
    if (hs.n == 0) return;
    wave_sync();
    const int lane = lane_id();
    int32_t v = 0, s0 = 0, nch = 0;
    if (lane < hs.n) {
        v = hs.v[lane];
        s0 = hs.s[lane];
        nch = (hs.d[lane] + hs.chunk - 1) / hs.chunk;
    }
    const int incl = wave_incl_scan(nch);
    int base = 0;
    if (lane == kWave - 1) base = atomicAdd(hn_out, incl);
    base = lane_get(base, kWave - 1) + incl - nch;
    hs.sent += (uint32_t)lane_get(incl, kWave - 1);
    for (int k = 0; k < nch; ++k) {
        st_agent(&hout[base + k].v, v);
        st_agent(&hout[base + k].start, s0 + k * hs.chunk);
    }
    hs.n = 0;
    wave_sync();
}

__device__ __forceinline__ void hub_push(HubStage& hs, bool pred, int32_t v, int32_t s0, int32_t d, HubItem* hout,
                                         int32_t* hn_out) {
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    const int c = __popcll(m);
    if (hs.n + c > kWave) hub_flush(hs, hout, hn_out);
    if (pred) {
        const int i = hs.n + __popcll(m & lanemask_lt());
        hs.v[i] = v;
        hs.s[i] = s0;
        hs.d[i] = d;
    }
    hs.n += c;
}

// End-of-phase flushes of every wave's staged entries with one allocation
// per block: each wave's count goes through LDS, thread 0 reserves the
// block's total.  (One allocation per wave would put up to 4096 atomics on
// one counter at the end of every level.)  All threads call them.
// Room for every wave's entries in up to two global counters: lane 0 of
// each wave posts its counts, lanes 0-15 of wave 0 (one DPP row) scan them,
// one lane takes both counters' atomics back to back, and every wave reads
// its bases.  Two block barriers.  sm.wbase is rewritten only after the next
// call's first barrier, which every wave reaches after reading its bases.
__device__ __forceinline__ void block_reserve2(Ctx& c, int n0, int32_t* count0, int n1, int32_t* count1, int& base0,
                                               int& base1) {
    static_assert(kW == 16, "the wave counts fill one DPP row");
    Smem& sm = c.sm;
    if (c.lane == 0) {
        sm.wcnt[0][c.wave] = n0;
        sm.wcnt[1][c.wave] = n1;
    }
    __syncthreads();
    if (c.wave == 0) {
        const int x = c.lane < kW ? sm.wcnt[0][c.lane] : 0, y = c.lane < kW ? sm.wcnt[1][c.lane] : 0;
        const int xi = row_incl(x, 0, [](int p, int q) { return p + q; });
        const int yi = row_incl(y, 0, [](int p, int q) { return p + q; });
        const int xt = lane_get(xi, kW - 1), yt = lane_get(yi, kW - 1);
        int xb = 0, yb = 0;
        if (c.lane == 0) {
            if (xt) xb = atomicAdd(count0, xt);
            if (yt) yb = atomicAdd(count1, yt);
        }
        xb = lane_get(xb, 0);
        yb = lane_get(yb, 0);
        if (c.lane < kW) {
            sm.wbase[0][c.lane] = xb + xi - x;
            sm.wbase[1][c.lane] = yb + yi - y;
        }
    }
    __syncthreads();
    base0 = sm.wbase[0][c.wave];
    base1 = sm.wbase[1][c.wave];
}

__device__ __forceinline__ int block_reserve(Ctx& c, int wave_count, int32_t* gcount) {
    int base, unused;
    block_reserve2(c, wave_count, gcount, 0, gcount, base, unused);
    return base;
}

__device__ __forceinline__ void block_flush(Ctx& c, WaveQueue& wq, int32_t* gq, int32_t* gcount) {
    const int base = block_reserve(c, wq.n, gcount);
    for (int i = c.lane; i < wq.n; i += kWave) st_agent(&gq[base + i], wq.buf[i]);
    wq.n = 0;
    wave_sync();
}

// A top-down queue entry: a vertex's first edge (high half) and degree (low
// half), which is all a top-down level needs to walk the vertex's list, so
// it loads no offsets; the claim that queues a vertex has just loaded them.
__device__ __forceinline__ uint64_t qentry(int32_t s0, int32_t d) {
    return ((uint64_t)(uint32_t)s0 << 32) | (uint32_t)d;
}
__device__ __forceinline__ int32_t qentry_start(uint64_t e) { return (int32_t)(uint32_t)(e >> 32); }
__device__ __forceinline__ int32_t qentry_degree(uint64_t e) { return (int32_t)(uint32_t)e; }

// A wave's staged top-down queue entries (in LDS) and its fill.
struct PairQueue {
    uint64_t* buf;
    int n;              // wave-uniform
    uint32_t sent = 0;  // entries written to the next level's queue so far (wave-uniform)
};

__device__ __forceinline__ void pq_flush(PairQueue& pq, uint64_t* gq, int32_t* gcount) {
    if (pq.n == 0) return;
    wave_sync();
    int base = 0;
    if (lane_id() == 0) base = atomicAdd(gcount, pq.n);
    base = lane_get(base, 0);
    for (int i = lane_id(); i < pq.n; i += kWave) st_agent(&gq[base + i], pq.buf[i]);
    pq.sent += (uint32_t)pq.n;
    pq.n = 0;
    wave_sync();
}

__device__ __forceinline__ void pq_push(PairQueue& pq, bool pred, uint64_t e, uint64_t* gq, int32_t* gcount) {
    const uint64_t m = __ballot(pred);
    if (m == 0) return;
    const int c = __popcll(m);
    if (pq.n + c > kPairCap) pq_flush(pq, gq, gcount);
    if (pred) pq.buf[pq.n + __popcll(m & lanemask_lt())] = e;
    pq.n += c;
}

// The end-of-level flush of the queue and of the staged hub vertices (as work
// items), with one reservation round.
__device__ __forceinline__ void block_flush_both(Ctx& c, PairQueue& pq, uint64_t* gq, int32_t* gcount, HubStage& hs,
                                                 HubItem* hout, int32_t* hn_out) {
    int32_t v = 0, s0 = 0, nch = 0;
    if (c.lane < hs.n) {
        v = hs.v[c.lane];
        s0 = hs.s[c.lane];
        nch = (hs.d[c.lane] + hs.chunk - 1) / hs.chunk;
    }
    const int incl = wave_incl_scan(nch);
    int qb, hb;
    block_reserve2(c, pq.n, gcount, lane_get(incl, kWave - 1), hn_out, qb, hb);
    for (int i = c.lane; i < pq.n; i += kWave) st_agent(&gq[qb + i], pq.buf[i]);
    hb += incl - nch;
    for (int k = 0; k < nch; ++k) {
        st_agent(&hout[hb + k].v, v);
        st_agent(&hout[hb + k].start, s0 + k * hs.chunk);
    }
    pq.sent += (uint32_t)pq.n;
    hs.sent += (uint32_t)lane_get(incl, kWave - 1);
    pq.n = 0;
    hs.n = 0;
    wave_sync();
}

// Pushes a newly claimed vertex for expansion at the next level: vertices of
// degree >= kGiantHubDeg become kGiantChunk-edge work items, others go to
// the queue (degree-0 vertices have nothing to expand).  All lanes call it.
__device__ __forceinline__ void push_next(bool claim, int32_t w, const int32_t* __restrict__ beg, PairQueue& pq,
                                          uint64_t* qout, int32_t* qn_out, HubStage& hs, HubItem* hout,
                                          int32_t* hn_out, int64_t& pushed_edges,
                                          int32_t hub_deg = kGiantHubDeg) {
    int32_t d = 0, s0 = 0;
    if (claim) {
        s0 = beg[w];
        d = beg[w + 1] - s0;
        pushed_edges += d;
    }
    hub_push(hs, claim && d >= hub_deg, w, s0, d, hout, hn_out);
    pq_push(pq, claim && d > 0 && d < hub_deg, qentry(s0, d), qout, qn_out);
}

// Claims K targets per lane, each as wave_try_claim does, and loads the
// offsets of every candidate while the claim atomics are in flight: a
// claimed vertex's degree costs no round trip of its own.  All lanes call it.
//
// kAskListed: without the allowed bits.  What a traversal reaches over an edge
// is allowed exactly if its own list in that direction is not empty (the edge
// is in its other list, and only vertices with both are active), so the
// offsets say it too, read before the claim and only for targets not yet
// visited.  That is one more round trip and a third fewer requests: for a chip
// full of waves that expand in place, which random requests bound (this card:
// 27 G/s atomics, 65 G/s loads past the L2), 4096^2 grid 3.72 -> 3.62 ms.
// kAskFresh: the same, and `allow` holds vertices that are not to be claimed.
enum { kAskAllowed, kAskListed, kAskFresh };
template <int K, int ASK = kAskAllowed>
__device__ __forceinline__ void claim_with_degree(const bool (&want)[K], const int32_t (&w)[K],
                                                  const uint64_t* __restrict__ allow, uint64_t* vis,
                                                  const int32_t* __restrict__ beg, bool (&claim)[K],
                                                  int32_t (&s0)[K], int32_t (&d)[K]) {
    const int lane = lane_id();
    uint64_t al[K], vi[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        al[k] = 0;
        vi[k] = 0;
        if (want[k]) {
            al[k] = ASK == kAskListed ? ~0ull : allow[w[k] >> 6];
            if (ASK == kAskFresh) al[k] = ~al[k];
            vi[k] = vis[w[k] >> 6];
        }
    }
    bool cand[K];
#pragma unroll
    for (int k = 0; k < K; ++k) cand[k] = want[k] && ((al[k] & ~vi[k]) >> (w[k] & 63)) & 1ull;
    int32_t e1[K];
    auto load_offsets = [&]() {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            s0[k] = 0;
            e1[k] = 0;
            if (cand[k]) {
                s0[k] = beg[w[k]];
                e1[k] = beg[w[k] + 1];
            }
        }
    };
    if (ASK != kAskAllowed) {
        load_offsets();
#pragma unroll
        for (int k = 0; k < K; ++k) cand[k] = cand[k] && e1[k] > s0[k];
    }
    uint64_t incl[K], excl[K];
    int end[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int32_t key = cand[k] ? (w[k] >> 6) : -1 - lane;  // lanes without a candidate: runs of their own
        // key of lane - 1: DPP within rows, the three row starts by readlane
        int32_t pkey = row_shr<1>(key, key);
        {
            const int32_t k15 = lane_get(key, 15), k31 = lane_get(key, 31), k47 = lane_get(key, 47);
            pkey = lane == 16 ? k15 : lane == 32 ? k31 : lane == 48 ? k47 : pkey;
        }
        const uint64_t heads = __ballot(lane == 0 || pkey != key);
        const uint64_t le = lane == kWave - 1 ? ~0ull : ((2ull << lane) - 1);
        const int start = 63 - __clzll(heads & le);
        const uint64_t after = heads & ~le;
        end[k] = after ? __ffsll((unsigned long long)after) - 2 : kWave - 1;
        // OR over lanes start..lane: scans within rows, then the carries of
        // runs that cross a row boundary, row by row
        uint64_t in = cand[k] ? 1ull << (w[k] & 63) : 0ull;
        uint64_t y = row_shr<1>(in, 0ull);
        if (lane - 1 >= start) in |= y;
        y = row_shr<2>(in, 0ull);
        if (lane - 2 >= start) in |= y;
        y = row_shr<4>(in, 0ull);
        if (lane - 4 >= start) in |= y;
        y = row_shr<8>(in, 0ull);
        if (lane - 8 >= start) in |= y;
        const uint64_t c15 = lane_get(in, 15);
        if (lane >= 16 && lane < 32 && start <= 15) in |= c15;
        const uint64_t c31 = lane_get(in, 31);
        if (lane >= 32 && lane < 48 && start <= 31) in |= c31;
        const uint64_t c47 = lane_get(in, 47);
        if (lane >= 48 && start <= 47) in |= c47;
        // the run's OR before this lane
        uint64_t ex = row_shr<1>(in, 0ull);
        ex = lane == 16 ? c15 : lane == 32 ? c31 : lane == 48 ? c47 : ex;
        if (lane == start) ex = 0;
        incl[k] = in;
        excl[k] = ex;
    }
    unsigned long long old[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        old[k] = 0;
        if (lane == end[k] && incl[k])
            old[k] = atomicOr(reinterpret_cast<unsigned long long*>(vis + (w[k] >> 6)), (unsigned long long)incl[k]);
    }
    if (ASK == kAskAllowed) load_offsets();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint64_t o = __shfl(old[k], end[k], kWave);
        claim[k] = cand[k] && !((o | excl[k]) & (1ull << (w[k] & 63)));
        d[k] = claim[k] ? e1[k] - s0[k] : 0;
    }
}

// push_next for K claimed targets whose offsets are known.
template <int K>
__device__ __forceinline__ void push_found_n(const bool (&claim)[K], const int32_t (&w)[K], const int32_t (&s0)[K],
                                             const int32_t (&d)[K], PairQueue& wq, uint64_t* qout, int32_t* qn_out,
                                             HubStage& hs, HubItem* hout, int32_t* hn_out, int64_t& pushed_edges) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
        pushed_edges += d[k];
        hub_push(hs, claim[k] && d[k] >= kGiantHubDeg, w[k], s0[k], d[k], hout, hn_out);
        pq_push(wq, claim[k] && d[k] > 0 && d[k] < kGiantHubDeg, qentry(s0[k], d[k]), qout, qn_out);
    }
}

// A frontier that is all in one tile, so in one block, goes on there without
// grid barriers: the block takes what it claimed as its next tile while that
// has at most kNarrowBlock edges, and its first wave alone, with no block
// barriers either, while it has at most kNarrowWave.  A level of a few edges
// costs 11 us across the grid, nearly all of it barrier and round trips that
// do no work, and about 4 us in a block and under 1 us in a wave.  More edges than
// a couple of steps of one block go back to the grid, which also bounds how
// long one block expands a growing region alone.
constexpr int kNarrowWave = 256;
constexpr int kNarrowBlock = 2048;
// Such levels in a row, while the other direction waits at the barrier and
// when it has finished: counted as levels of a wave, one of a block as the
// kNarrowCost wave levels whose time it takes.  128, 64 and 16 with every
// level counted as one gave lattices of 60^2 192, 281 and 358 us and of 2000^2
// 1.46, 1.45 and 1.68 ms; 256 and 512 gave what 128 gives.
constexpr int kNarrowShort = 128, kNarrowLong = 16384, kNarrowCost = 4;

// The adj index of this lane's edge, less the edge's number eb + lane, for
// edges eb to eb + kWave - 1 of up to kWave entries, one a lane, that begin at
// edge `off` (ascending) and at adj index `st`; a lane past the last edge gets
// some value.  The source of edge e is the last entry j with off_j <= e.
// Every entry has an edge, so that is the number of entries that begin at or
// before e, less one: those before the chunk, and those whose bit is set up to
// e's in the chunk's word of beginnings (an OR over the wave by DPP).  A
// binary search of the offsets in LDS is six dependent reads.
__device__ __forceinline__ int32_t edge_entry(bool valid, int off, int32_t st, int eb) {
    const int rel = off - eb;
    const int before = __popcll(__ballot(valid && rel < 0));
    uint64_t begins = row_incl((uint64_t)(valid && rel >= 0 && rel < kWave ? 1ull << rel : 0ull), (uint64_t)0,
                               [](uint64_t x, uint64_t y) { return x | y; });
    begins = lane_get(begins, 15) | lane_get(begins, 31) | lane_get(begins, 47) | lane_get(begins, 63);
    const int pos = before + __popcll(begins & (lanemask_lt() | (1ull << lane_id()))) - 1;
    return __shfl(st - off, pos, kWave);
}

// Top-down to exhaustion (mode 2) without level barriers in the thin parts:
// a wave expands the vertices it claimed itself, in the same level, instead
// of publishing them for the next level -- the reference's asynchronous
// top-down (src/fw_bw.h:506-544, 1068-1106), where each thread keeps
// expanding its own circular queue.  The wave's LDS staging buffer is that
// queue: up to kWave pending entries per step are flattened (wave-level
// degree scan) and walked one edge per lane; new claims of degree below
// kGiantHubDeg go back into the queue, hubs become next-level work items,
// and when the queue is full -- or after max_steps steps, so that a region
// one wave holds is shared again -- entries go to the next level's queue.
// Claims stay exact (the same wave-combined atomics), so the reach set and
// the found counts are those of a level-synchronous traversal; only the
// level at which a vertex is expanded changes.  With FRESH, what is in `before`
// is not claimed, besides what is in vis.  All lanes call it.
template <bool FRESH>
__device__ __forceinline__ void expand_local(Ctx& c, PairQueue& wq, int32_t root, const int32_t* __restrict__ beg,
                                             const int32_t* __restrict__ adj, const uint64_t* __restrict__ before,
                                             uint64_t* vis, uint64_t* qout, int32_t* qn_out, HubStage& hs,
                                             HubItem* hout, int32_t* hn_out, int64_t& my_found, int max_steps) {
    uint64_t* buf = wq.buf;
    constexpr int mask = kPairCap - 1;
    int head = 0, n = wq.n;  // pending: buf[head .. n) modulo kPairCap
    wave_sync();
    for (; n > head && max_steps > 0; --max_steps) {
        const int k = min(kWave, n - head);
        int32_t st = 0, dg = 0;
        if (c.lane < k) {
            const uint64_t q = buf[(head + c.lane) & mask];
            st = qentry_start(q);
            dg = qentry_degree(q);
        }
        const int incl = wave_incl_scan(dg);
        const int total = lane_get(incl, kWave - 1);
        head += k;
        c.edges_td += total;
        const int off = incl - dg;  // this entry's first edge of the step
        wave_sync();  // the queue entries are read: their places may be written
        for (int eb = 0; eb < total; eb += kWave) {
            const int e = eb + c.lane;
            const int32_t src = edge_entry(c.lane < k, off, st, eb);
            bool want[1];
            int32_t w[1];
            w[0] = e < total ? adj[src + e] : 0;
            want[0] = e < total && w[0] != root;
            bool claim[1];
            int32_t s0[1], d[1];
            claim_with_degree<1, FRESH ? kAskFresh : kAskListed>(want, w, before, vis, beg, claim, s0, d);
            my_found += claim[0];
            hub_push(hs, claim[0] && d[0] >= kGiantHubDeg, w[0], s0[0], d[0], hout, hn_out);
            const bool keep = claim[0] && d[0] > 0 && d[0] < kGiantHubDeg;
            const uint64_t m = __ballot(keep);
            const int cnt = __popcll(m);
            if (cnt && n - head + cnt <= kPairCap) {
                if (keep) buf[(n + __popcll(m & lanemask_lt())) & mask] = qentry(s0[0], d[0]);
                n += cnt;
            } else if (cnt) {  // the queue is full: these go to the next level
                int base = 0;
                if (c.lane == 0) base = atomicAdd(qn_out, cnt);
                base = lane_get(base, 0);
                wq.sent += (uint32_t)cnt;
                if (keep) st_agent(&qout[base + __popcll(m & lanemask_lt())], qentry(s0[0], d[0]));
            }
        }
        wave_sync();  // the entries pushed are read next step
    }
    const int left = n - head;  // the step budget ran out: the next level takes them
    if (left > 0) {
        int base = 0;
        if (c.lane == 0) base = atomicAdd(qn_out, left);
        base = lane_get(base, 0);
        for (int i = c.lane; i < left; i += kWave) st_agent(&qout[base + i], buf[(head + i) & mask]);
        wq.sent += (uint32_t)left;
    }
    wq.n = 0;
    wave_sync();
}

// The frontier of a narrow region in one wave: expand_local for at most kWave
// entries of at most kNarrowWave edges together at a time, and only while
// that is everything that is pending and no hub turned up; what is left then
// stays staged in wq, for the block to go on with.  Returns the steps that
// are left of max_steps.
//
// Such a step is one serial chain of round trips and dependent instructions,
// so it is cut to what a step cannot do without.  Nobody else claims in this
// direction meanwhile (the frontier is all in this wave, the other blocks
// wait at the grid's barrier), so the claims are made in LDS, on copies of the
// visited words: kSets of them, by word number modulo kSets, each beside what
// it was in memory, which gets the new bits when another word takes the place
// and at the end.  That leaves two round trips a step, the list and the
// offsets of what it names, mostly cache hits, where there are four with the
// visited bits read and then claimed in memory.  While a step's edges fit the
// wave, the entries stay in the registers of the lanes that claimed them, and
// no lane branches except where a word is missing or a hub turns up.  A
// chain of 10^4 levels of about two vertices: 1.6 us a level in expand_local,
// 0.94 with the copies, 0.71 with both.  The copies lie in the other waves'
// staging, which is empty while they wait at the block's barrier.
__device__ __forceinline__ int expand_wave(Ctx& c, PairQueue& wq, int32_t root, const int32_t* __restrict__ beg,
                                           const int32_t* __restrict__ adj, const uint64_t* __restrict__ allow,
                                           uint64_t* vis, HubStage& hs, HubItem* hout, int32_t* hn_out,
                                           int32_t nwords, int64_t& my_found, int max_steps) {
    constexpr int kSets = 256, kStep = kWave - 1;
    static_assert(2 * kSets <= kPairCap && kSets % kWave == 0 && kW >= 3, "the copies fit two waves' staging");
    static_assert(kNarrowWave <= kPairCap, "a step's claims fit the staging");
    uint64_t* buf = wq.buf;
    unsigned long long* seen = reinterpret_cast<unsigned long long*>(buf + kPairCap);  // visited, or not to be visited
    unsigned long long* had = seen + kSets;                                            // the same as it is in memory
    int32_t* word = reinterpret_cast<int32_t*>(buf + 2 * kPairCap);                    // the word's number
    unsigned long long* mem = reinterpret_cast<unsigned long long*>(vis);
    if (wq.n > kWave || hs.n > 0) return max_steps;
    for (int i = c.lane; i < kSets; i += kWave) {
        word[i] = -1;
        seen[i] = 0;
        had[i] = 0;
    }
    int32_t st = 0, dg = 0;  // an entry a lane, in any lane; dg = 0 is none
    if (c.lane < wq.n) {
        const uint64_t q = buf[c.lane];
        st = qentry_start(q);
        dg = qentry_degree(q);
    }
    wave_sync();
    int staged = 0;  // entries in buf, when they are too many for the lanes
    for (; max_steps > 0; --max_steps) {
        const int incl = wave_incl_scan(dg);
        const int total = lane_get(incl, kWave - 1);
        if (total == 0 || total > kNarrowWave) break;
        c.edges_td += total;
        const int off = incl - dg;
        int n = 0;
        for (int eb = 0; eb < total; eb += kStep) {
            // Edges eb to eb + kStep - 1, one a lane.  An entry sends where
            // its list lies, less its offset, to the lane of its first edge;
            // an edge's entry is then at the last such lane up to its own,
            // or began before the chunk.  (The last lane has no edge: what is
            // not to be sent goes there.  kBias keeps a sent value from 0.)
            constexpr int kBias = kNarrowWave + 1;
            const int rel = off - eb;
            const bool starts = dg > 0 && rel >= 0 && rel < kStep;
            const int got = __builtin_amdgcn_ds_permute((starts ? rel : kStep) * 4, st - off + kBias);
            const uint64_t heads = __ballot(got != 0 && c.lane < kStep) & ((2ull << c.lane) - 1);
            int32_t src = __shfl(got, 63 - __clzll((long long)(heads | 1)), kWave) - kBias;
            if (eb) {
                const uint64_t before = __ballot(dg > 0 && rel < 0);
                const int32_t cur = lane_get(st - off, 63 - __clzll((long long)before));
                src = heads ? src : cur;
            }
            const int e = eb + c.lane;
            const bool edge = c.lane < kStep && e < total;
            const int32_t w = adj[edge ? src + e : lane_get(src, 0) + eb];
            const int32_t s0 = beg[w], d = beg[w + 1] - s0;
            const bool cand = edge && w != root;
            const int32_t wd = w >> 6;
            const int set = wd & (kSets - 1);
            const unsigned long long bit = 1ull << (w & 63);
            bool here = word[set] == wd;
            unsigned long long old = ~0ull;
            if (__ballot(cand && !here)) {
                wait_vm();  // what earlier words left is in memory
                // the missing words, and in the other lanes the words around
                // the first of them: vertices that follow each other along a
                // path mostly have ids close together
                const uint64_t missing = __ballot(cand && !here);
                const int32_t near = lane_get(wd, __ffsll((unsigned long long)missing) - 1) + c.lane - kWave / 2;
                const bool miss = cand && !here;
                const int32_t take = miss ? wd : near;
                const int at = take & (kSets - 1);
                const bool fill = miss || (near >= 0 && near < nwords && word[at] != near);
                unsigned long long now = 0, left = 0;
                int32_t from = 0;
                if (fill) {
                    now = load_agent(&vis[take]) | ~allow[take];
                    from = word[at];
                    left = seen[at] & ~had[at];
                }
                wave_sync();
                if (fill) word[at] = take;
                wave_sync();
                if (fill && word[at] == take) {  // of several words for one place, one has it
                    if (left) atomicOr(mem + from, left);
                    seen[at] = now;
                    had[at] = now;
                }
                wave_sync();
                here = word[set] == wd;
                if (__ballot(cand && !here)) {  // the others, and a word that was here until now, in memory
                    wait_vm();
                    if (cand && !here && (allow[wd] & bit)) old = atomicOr(mem + wd, bit);
                    wait_vm();
                }
            }
            const unsigned long long was = atomicOr(&seen[set], cand && here ? bit : 0ull);
            old = here ? was : old;
            const bool claim = cand && !(old & bit);
            my_found += claim;
            hub_push(hs, claim && d >= kGiantHubDeg, w, s0, d, hout, hn_out);
            const bool keep = claim && d > 0 && d < kGiantHubDeg;
            if (total <= kStep) {
                st = s0;
                dg = keep ? d : 0;
            } else {
                const uint64_t m = __ballot(keep);
                if (keep) buf[n + __popcll(m & lanemask_lt())] = qentry(s0, d);
                n += __popcll(m);
            }
        }
        if (total > kStep) {
            wave_sync();
            uint64_t q = 0;
            if (n > kWave)
                staged = n;
            else if (c.lane < n)
                q = buf[c.lane];
            st = qentry_start(q);
            dg = qentry_degree(q);
            wave_sync();
        }
        if (staged || hs.n > 0) {
            --max_steps;
            break;
        }
    }
    if (staged == 0) {
        const uint64_t m = __ballot(dg > 0);
        if (dg > 0) buf[__popcll(m & lanemask_lt())] = qentry(st, dg);
        staged = __popcll(m);
    }
    wave_sync();
    for (int i = c.lane; i < kSets; i += kWave) {
        const unsigned long long left = seen[i] & ~had[i];
        if (left) atomicOr(mem + word[i], left);
    }
    wait_vm();  // the other waves claim from memory
    wq.n = staged;
    return max_steps;
}

// Level-synchronous top-down levels are expanded in place (as in mode 2)
// once their input gives every wave at least this many vertices.  Five
// 4096^2 lattices: 3.65 ms on average with 12, 3.70 with 11, 3.72 with 10 and
// 3.69 with 14 (8 and 16: three of them, 3.88 and 3.89), smaller ones alike;
// R-MAT flat.
constexpr int kLocalPerWave = 12;

// The first top-down level after bottom-up ones goes on from the finds in place
// while there are at most this many for each wave, and else queues them for the
// next level: a wave's words have what they have, and where the finds are many
// some waves have most of their edges (R-MAT's degrees follow the id bits).
// With the defaults few are left.  Always in place, and by this rule: beta = 1 on
// 3 M vertices at edge factor 3 2.38 / 0.50 ms, on R-MAT of 700 K and 8 M vertices
// 0.63 / 0.31 and 2.9 / 1.38; with 8, 32 or 64 the same.  Never in place: by the
// defaults 700 K vertices 151 us against 137, a lattice of 500^2 623 against 577.
constexpr int kGatherLocal = 16;

// A batch's roots, the vertices of most edges of its graphs, are the whole
// level 0: their lists are cut into items of a block's step, from kSeedHubDeg
// edges on where the items' room allows.  With kGiantChunk edges an item and
// up to 64 lists of less than kGiantHubDeg in a tile a few blocks had most of
// the level (400 graphs, 660 K edges a direction: the level 97 -> 64 us).
constexpr int kSeedChunk = kGBlock;
constexpr int kSeedHubDeg = kWave;
static_assert(kSeedChunk >= 2 * kGiantHubDeg, "giant_hub_capacity holds such items");

// What a wave's part of a level came to: per-thread counts and wave-uniform
// queue totals.
struct Level {
    int found;          // vertices this thread claimed
    int edges;          // out-degree sum of what it pushed (top-down), entries it scanned (bottom-up)
    uint32_t nq, nh;    // queue entries and work items this wave wrote for the next level
};

// One level of one direction: top-down over the level's queue and hub items
// (then, where it applies, in place), or bottom-up over the candidate
// bitmap.  Forward: from the pivot along
// out-edges, claiming active vertices into fvis.  Backward: along in-edges,
// claiming active vertices into bvis, not only those of the forward set: the
// giant SCC is fvis & bvis either way (a path from v to the pivot lies in
// the forward set when v does), and the two directions then need not wait
// for each other.
__device__ __forceinline__ void level_work(Ctx& c, int mode, int32_t L, int32_t nq, int32_t nh_in, int dir, int32_t root,
                                           int narrow_steps, bool half, bool gather, Level& lv) {
    KernelArgs& a = c.args();
    Smem& sm = c.sm;
    const bool bw = dir != 0;
    const int32_t* beg = bw ? a.bwb : a.fwb;  // expansion (top-down) direction
    const int32_t* adj = bw ? a.bwa : a.fwa;
    const int32_t* rbeg = bw ? a.fwb : a.bwb;  // bottom-up scans the reverse direction
    const int32_t* radj = bw ? a.fwa : a.bwa;
    const int32_t* rfirst = bw ? a.fw_first : a.bw_first;
    const uint64_t* allow = a.act;
    uint64_t* snap = bw ? a.snapb : a.snap;
    // what is visited: from the gathering level on, the bitmap that the
    // bottom-up levels left in snap
    uint64_t* vis = mode == 2 ? snap : bw ? a.bvis : a.fvis;
    uint64_t* q0 = bw ? a.qb0 : a.q0;
    uint64_t* q1 = bw ? a.qb1 : a.q1;
    HubItem* h0 = bw ? a.hb0 : a.h0;
    HubItem* h1 = bw ? a.hb1 : a.h1;
    GiantState* gs = a.gs;
    PairQueue pq{c.stage(), 0};    // top-down: staged next-level entries
    WaveQueue wq{c.stage32(), 0};  // bottom-up: the same LDS, parked misses (ids)
    HubStage hs{sm.hv[c.wave], sm.hs[c.wave], sm.hd[c.wave], 0};
    // half: this direction has half of every block's waves (bottom-up only)
    const int wpb = half ? kW / 2 : kW;
    const int64_t total_waves = (int64_t)c.G * wpb;
    const int64_t gwave = (int64_t)c.b * wpb + (half ? c.wave % (kW / 2) : c.wave);
    auto is_vis = [vis](int32_t u, int32_t) { return bit_of(vis, u); };
    const bool multi = a.n_roots > 0;
    int64_t my_found = 0, fedges = 0;
    const uint64_t* qin = (L & 1) ? q1 : q0;
    uint64_t* qout = (L & 1) ? q0 : q1;
    const HubItem* hin = (L & 1) ? h1 : h0;
    HubItem* hout = (L & 1) ? h0 : h1;
    int32_t* qn_out = &gs->qn[dir][(L + 1) % 3].v;
    int32_t* hn_out = &gs->hn[dir][(L + 1) % 3].v;
    const bool topdown = mode != 1;
    // the level trace is kept by one thread of the block: of its part that has
    // this direction, where each direction has half of the waves
    const bool tr = a.trace && L < kLevelTrace && c.tid % (wpb * kWave) == 0;
    const int64_t tl0 = tr ? (int64_t)wall_clock64() : 0;
    if (topdown && gather) {
        // ---- the first top-down level after bottom-up ones: each wave takes
        // the last level's finds of its words, an even share of up to 64 at a
        // time, and goes on from them in place (64 whatever the size left a
        // lattice of 500^2 to 61 waves, 0.56 ms a direction).  No queue and no
        // barrier lie between the finds and their expansion (a gather pass
        // that queued them for a level of their own: 29 us for both at R-MAT
        // s24).
        // Some waves expand while others still gather, so the claims must not
        // show among the finds: a vertex queued by both would be one entry
        // more than the queues and hub lists have room for.  The bitmap that
        // the finds were made in (`found`) therefore stays as it is, and
        // claims, of vertices outside it, go into snap (what was visited
        // before the last level), to which each wave adds the finds it takes.
        // After the level snap holds all that is visited, and the later levels
        // and the phases after them go by it.
        const uint64_t* found = bw ? a.bvis : a.fvis;
        const int64_t share = min((a.nwords + total_waves - 1) / total_waves, (int64_t)kWave);
        for (int64_t wb = gwave * share; wb < a.nwords; wb += total_waves * share) {
            const int64_t w = wb + c.lane;
            uint64_t nw = 0;
            if (c.lane < share && w < a.nwords) nw = found[w] & ~vis[w];
            if (nw) atomicOr(reinterpret_cast<unsigned long long*>(vis + w), (unsigned long long)nw);
            uint64_t busy = __ballot(nw != 0);
            while (busy) {
                const int l = __ffsll((unsigned long long)busy) - 1;
                busy &= busy - 1;
                const uint64_t m = lane_get(nw, l);
                const int32_t v = (int32_t)((wb + l) * 64 + c.lane);
                push_next((m >> c.lane) & 1ull, v, beg, pq, qout, qn_out, hs, hout, hn_out, fedges);
            }
        }
        if (a.td_local > 0 && nq <= kGatherLocal * total_waves)
            expand_local<true>(c, pq, root, beg, adj, found, vis, qout, qn_out, hs, hout, hn_out, my_found,
                               a.td_local);
        block_flush_both(c, pq, qout, qn_out, hs, hout, hn_out);
        lv = Level{(int)my_found, (int)fedges, pq.sent, hs.sent};
    } else if (topdown) {
        // ---- top-down: tiles of the queue, then hub work items; level 0
        // expands the root's list in kGiantChunk-edge pieces.
        int64_t n = 0, nh = 0;
        int32_t rchunk = kGiantChunk;  // level 0: edges per piece of the root's list
        if (L == 0 && !multi) {
            if (c.b == 0 && c.tid == 0)
                atomicOr(reinterpret_cast<unsigned long long*>(vis + (root >> 6)), 1ull << (root & 63));
            // the root's list in about one piece per block
            const int32_t rdeg = beg[root + 1] - beg[root];
            rchunk = max(256, ((rdeg + c.G - 1) / c.G + 63) & ~63);
            rchunk = min(rchunk, kGiantChunk);
            nh = (rdeg + rchunk - 1) / rchunk;
        } else {
            n = nq;
            nh = nh_in;
            if (L == 0) rchunk = kSeedChunk;
            if (n < 0 || n > a.V || nh < 0 || nh > a.hub_cap) {  // cannot happen with exact claims
                if (c.tid == 0) atomicOr(&gs->err.v, 4);
                n = 0;
                nh = 0;
            }
        }
        if (n == 0 && nh == 0) return;
        static_assert((kGBlock & (kGBlock - 1)) == 0, "tile size");
        // entries per tile: a power of two from 64 to kGBlock, the
        // smallest that needs no more tiles than blocks, so a small
        // frontier is spread over many blocks
        int tile = kGBlock;
        while (tile > kWave && (int64_t)(tile / 2) * c.G >= n) tile /= 2;
        const int64_t ntiles = (n + tile - 1) / tile;
        // the backward direction's tiles start half the grid away, so that
        // when both directions' levels are small (fewer tiles than blocks)
        // they run on different blocks at the same time
        const int64_t b0 = bw ? ((int64_t)c.b + c.G / 2) % c.G : c.b;
        const bool narrow = a.td_local > 0 && mode == 0 && ntiles + nh == 1;  // mode 2 goes on in place below
        for (int64_t u = b0; u < ntiles + nh; u += c.G) {
            // a tile: queue entries on threads 0..tile-1; a hub item is a
            // tile of one entry on thread 0
            bool hub = u >= ntiles;
            int32_t st = 0, dg = 0;
            if (!hub) {
                const int64_t i = u * tile + c.tid;
                if (c.tid < tile && i < n) {
                    const uint64_t q = load_agent(&qin[i]);
                    st = qentry_start(q);
                    dg = qentry_degree(q);
                }
            } else if (c.tid == 0) {
                int32_t v = root;
                if (L == 0 && !multi) {
                    st = beg[root] + (int32_t)(u - ntiles) * rchunk;
                } else {
                    v = load_agent(&hin[u - ntiles].v);
                    st = load_agent(&hin[u - ntiles].start);
                }
                dg = min(rchunk, beg[v + 1] - st);
            }
            while (true) {
                int excl, total;
                block_excl_scan<kW>(dg, excl, total, sm.tmp);
                sm.off[c.tid] = excl;
                sm.start[c.tid] = st;
                if (c.wave == 0) c.edges_td += total;
                __syncthreads();
                for (int eb = 0; eb < total; eb += kGBlock) {
                    // the source of edge e is the last j with off[j] <= e
                    // (off[0] = 0, non-decreasing), found by a fixed-depth
                    // search; a hub item's is its one entry
                    const int e = eb + c.tid;
                    int pos = 0;
                    if (!hub) {
#pragma unroll
                        for (int sp = kGBlock / 2; sp > 0; sp >>= 1)
                            if (sm.off[pos + sp] <= e) pos += sp;
                    }
                    int32_t w[1] = {0};
                    if (e < total) w[0] = adj[sm.start[pos] + (e - sm.off[pos])];
                    const bool want[1] = {e < total && w[0] != root};
                    bool claim[1];
                    int32_t s0[1], dw[1];
                    claim_with_degree<1>(want, w, allow, vis, beg, claim, s0, dw);
                    my_found += claim[0];
                    push_found_n<1>(claim, w, s0, dw, pq, qout, qn_out, hs, hout, hn_out, fedges);
                }
                __syncthreads();
                if (!narrow) break;
                // the only tile: take what it claimed as the next one
                if (total <= kWave) {  // only the first wave had edges
                    if (c.wave == 0) {
                        narrow_steps = expand_wave(c, pq, root, beg, adj, allow, vis, hs, hout, hn_out, (int32_t)a.nwords,
                                                   my_found, narrow_steps);
                        fedges = c.lane < hs.n ? hs.d[c.lane] : 0;
                        for (int i = c.lane; i < pq.n; i += kWave) fedges += qentry_degree(pq.buf[i]);
                    }
                }
                // Every wave decides by itself from all waves' counts.  They have
                // arrays of their own: a wave that leaves writes its flush
                // counts (wcnt) with no barrier in between, while others may
                // still be reading these.  They are written again only after
                // the barriers of another round, or after the grid's.
                const int work = wave_sum((int)fedges);
                if (c.tid == 0) sm.steps = narrow_steps;
                if (c.lane == 0) {
                    sm.narrow[0][c.wave] = pq.n;
                    sm.narrow[1][c.wave] = (hs.n > 0 || pq.sent > 0 || hs.sent > 0) ? kNarrowBlock + 1 : min(work, kNarrowBlock + 1);
                }
                __syncthreads();
                const int cnt = sm.narrow[0][c.lane & 15];
                const int ci = row_incl(cnt, 0, [](int x, int y) { return x + y; });
                const int wi = row_incl(sm.narrow[1][c.lane & 15], 0, [](int x, int y) { return x + y; });
                const int entries = lane_get(ci, kW - 1), edges = lane_get(wi, kW - 1);
                const int base = lane_get(ci - cnt, c.wave);
                narrow_steps = __builtin_amdgcn_readfirstlane(sm.steps) - kNarrowCost;
                if (entries == 0 || entries > kGBlock || edges > kNarrowBlock || narrow_steps <= 0) break;
                wave_sync();
                for (int i = c.lane; i < pq.n; i += kWave) {
                    const uint64_t q = pq.buf[i];
                    sm.off[base + i] = qentry_degree(q);
                    sm.start[base + i] = qentry_start(q);
                }
                pq.n = 0;
                fedges = 0;
                __syncthreads();
                st = c.tid < entries ? sm.start[c.tid] : 0;
                dg = c.tid < entries ? sm.off[c.tid] : 0;
                hub = false;
                __syncthreads();
            }
        }
        // in place: in top-down to exhaustion, and in any later top-down
        // level whose input gives every wave at least kLocalPerWave
        // vertices.  Where the frontier is small (the start of a
        // traversal on a high-diameter graph) a few waves would expand a
        // growing region alone: levels of up to 256-65536 entries
        // expanded so took the 4096^2 grid from 5.09 to 5.8-6.5 ms.
        if (a.td_local > 0 && (mode == 2 || (L > 0 && nh == 0 && n >= kLocalPerWave * total_waves)))
            expand_local<false>(c, pq, root, beg, adj, nullptr, vis, qout, qn_out, hs, hout, hn_out, my_found,
                                a.td_local);
        block_flush_both(c, pq, qout, qn_out, hs, hout, hn_out);
        lv = Level{(int)my_found, (int)fedges, pq.sent, hs.sent};
    } else {
        // ---- bottom-up over the candidate bitmap, one wave per group of
        // kU consecutive 64-vertex words; only that wave writes those
        // words in this level.  Each stage issues its kU loads (first
        // in-neighbours, their visited bits) before any result is used.
        // Nothing is queued: each word's visited bits before the level go
        // to `snap`, and a switch back to top-down takes vis & ~snap.
        constexpr int kU = 8;       // dense words per group
        constexpr int kSparse = 8;  // at most this many candidates: a lane's own work
        constexpr int kS = 4;       // sparse candidates per lane per step
        int scanned = 0;
        // candidates whose first probe misses are parked in the wave's LDS
        // buffer and scanned 64 at a time, one per lane, so their load
        // chains overlap instead of idling the other 63 lanes
        int nmiss = 0;  // wave-uniform
        auto scan_misses = [&]() {
            wave_sync();
            int32_t pv = -1;  // found in the previous batch: set behind this batch's loads
            for (int i0 = 0; i0 < nmiss; i0 += kWave) {
                const int i = i0 + c.lane;
                int32_t v = 0, p = 0, e = 0;
                if (i < nmiss) {
                    v = wq.buf[i];
                    p = rbeg[v] + 1;
                    e = rbeg[v + 1];
                }
                if (pv >= 0) atomicOr(reinterpret_cast<unsigned long long*>(vis + (pv >> 6)), 1ull << (pv & 63));
                pv = -1;
                const bool found = wave_any_edge(i < nmiss && p < e, p, e, v, radj, is_vis, scanned);
                if (found) {
                    pv = v;
                    my_found += 1;
                }
            }
            if (pv >= 0) atomicOr(reinterpret_cast<unsigned long long*>(vis + (pv >> 6)), 1ull << (pv & 63));
            nmiss = 0;
            wave_sync();
        };
        // misses with more list to scan go to the wave's buffer (all lanes call)
        auto park_misses = [&](bool miss, int32_t v) {
            const uint64_t mm = __ballot(miss);
            if (!mm) return;
            if (nmiss + __popcll(mm) > kWaveBuf) scan_misses();
            if (miss) wq.buf[nmiss + __popcll(mm & lanemask_lt())] = v;
            nmiss += __popcll(mm);
        };
        // A wave step covers kWave / kBUrun runs of kBUrun consecutive words
        // spread over the whole id range (run r of the step is run
        // cb + r * total_waves + gwave), so that the id ranges where the
        // work concentrates are shared by all blocks.
        constexpr int kBUrun = 8;
        const int64_t nruns = (a.nwords + kBUrun - 1) / kBUrun;
        // All waves sweep the id range in the same order (band by band:
        // vertices found early help later probes of the level hit), and
        // within a band wave g takes run (g * bu_mult) mod total_waves, a
        // permutation: with plain indices a block's runs would share
        // fixed bits of their vertex ids, and in graphs whose degrees
        // follow id bits (R-MAT) the blocks' work would differ severalfold.
        // (gwave and bu_mult are less than all waves of the grid, at most
        // 65536, also where a direction has half of them: the product fits
        // 32 bits, and bu_mult, coprime to all of them, is so to the half)
        const int64_t pg = (int64_t)(((uint32_t)gwave * (uint32_t)a.bu_mult) % (uint32_t)total_waves);
        for (int64_t cb = 0; cb < nruns; cb += total_waves * (kWave / kBUrun)) {
            // lane j loads one word; then only words with candidates are
            // worked on, kU of them at a time
            const int64_t run = cb + (int64_t)(c.lane / kBUrun) * total_waves + pg;
            const int64_t wl = run * kBUrun + (c.lane % kBUrun);
            uint64_t lvw = 0, lcand = 0;
            if (wl < a.nwords) {
                lvw = vis[wl];
                lcand = allow[wl] & ~lvw;
            }
            // words with more than kSparse candidates: the wave works on
            // kU of them at a time, one lane per vertex
            const bool dense = __popcll(lcand) > kSparse;
            uint64_t busy = __ballot(dense);
            // Found bits of group member u wait in lane u and go out as
            // one atomic instruction behind the next group's loads: a
            // load's wait also waits for the atomics issued before it.
            int64_t pw = 0;
            uint64_t pm = 0;
            while (busy) {
                uint64_t group = 0;  // the kU words worked on, as lanes of wl / lcand
                int32_t f[kU];
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    f[u] = -1;
                    if (busy) {
                        const int l = __ffsll((unsigned long long)busy) - 1;
                        busy &= busy - 1;
                        group |= 1ull << l;
                        if ((lane_get(lcand, l) >> c.lane) & 1ull) f[u] = rfirst[lane_get(wl, l) * 64 + c.lane];
                    }
                }
                if (pm) atomicOr(reinterpret_cast<unsigned long long*>(vis + pw), (unsigned long long)pm);
                pm = 0;
                uint32_t hits = 0, listed = 0;  // bit u: first neighbour visited / list not empty
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    listed |= f[u] >= 0 ? 1u << u : 0u;
                    hits |= (f[u] >= 0 && bit_of(vis, f[u])) ? 1u << u : 0u;
                }
                // rolled, so that the miss scan is in the code once
#pragma unroll 1
                for (int u = 0; group; ++u, group &= group - 1) {
                    const int l = __ffsll((unsigned long long)group) - 1;
                    const uint64_t cm = lane_get(lcand, l);
                    const int64_t w = lane_get(wl, l);
                    const bool is_c = (cm >> c.lane) & 1ull;
                    const bool hit = (hits >> u) & 1u;  // f is -1 unless a candidate
                    scanned += is_c;
                    park_misses(!hit && ((listed >> u) & 1u), (int32_t)(w * 64 + c.lane));
                    // found bits are set within the level: later probes
                    // already see them
                    const uint64_t fm = __ballot(hit);
                    if (c.lane == u) {
                        pw = w;
                        pm = fm;
                    }
                    my_found += hit;
                }
            }
            if (tr && cb == 0)
                atomicMax(reinterpret_cast<unsigned long long*>(&gs->lv_cp[dir][L][3]),
                          (unsigned long long)((int64_t)wall_clock64() - tl0));
            // sparse words: each lane works through its own word's
            // candidates, kS at a time, and sets its found bits at once
            uint64_t mine = dense ? 0ull : lcand, fm_lane = 0;
            while (__ballot(mine != 0)) {
                uint64_t group = mine;  // its lowest kS bits are this step's candidates
                int32_t f[kS];
#pragma unroll
                for (int k = 0; k < kS; ++k) {
                    f[k] = -1;
                    if (mine) {
                        f[k] = rfirst[wl * 64 + __ffsll((unsigned long long)mine) - 1];
                        mine &= mine - 1;
                    }
                }
                uint32_t hits = 0, listed = 0;
#pragma unroll
                for (int k = 0; k < kS; ++k) {
                    listed |= f[k] >= 0 ? 1u << k : 0u;
                    hits |= (f[k] >= 0 && bit_of(vis, f[k])) ? 1u << k : 0u;
                }
#pragma unroll 1
                for (int k = 0; k < kS; ++k) {
                    const int bit = __ffsll((unsigned long long)group) - 1;  // -1: none left
                    group &= group ? group - 1 : 0;
                    const bool hit = (hits >> k) & 1u;
                    scanned += bit >= 0;
                    park_misses(!hit && ((listed >> k) & 1u), (int32_t)(wl * 64 + bit));
                    if (hit) {
                        fm_lane |= 1ull << bit;
                        my_found += 1;
                    }
                }
            }
            if (pm) atomicOr(reinterpret_cast<unsigned long long*>(vis + pw), (unsigned long long)pm);
            if (fm_lane) atomicOr(reinterpret_cast<unsigned long long*>(vis + wl), (unsigned long long)fm_lane);
            if (wl < a.nwords) st_agent(&snap[wl], lvw);  // the gather's "visited before this level"
        }
        if (tr)
            atomicMax(reinterpret_cast<unsigned long long*>(&gs->lv_cp[dir][L][1]),
                      (unsigned long long)((int64_t)wall_clock64() - tl0));
        scan_misses();
        if (tr)
            atomicMax(reinterpret_cast<unsigned long long*>(&gs->lv_cp[dir][L][2]),
                      (unsigned long long)((int64_t)wall_clock64() - tl0));
        lv = Level{(int)my_found, scanned, 0, 0};  // bottom-up pushes nothing
    }
}

// The giant's traversals: forward and backward in the same levels, one grid
// barrier per level for both (fw_bfs_fq_queue, src/fw_bw.h:396-698, and
// bw_bfs_fq_queue, :944-1248, which the reference runs one after the
// other).  Each direction switches top-down / bottom-up / top-down to
// exhaustion on its own, by the reference's rules on alpha, beta and gamma
// (src/fw_bw.h:576-624) with set_size the active count for both; a
// direction that has finished idles while the other goes on.  Returns false
// after a failed barrier.  With a.n_roots > 0 every listed root seeds both
// directions (*seeded_out of them).  The directions' state is in sm.dir.
//
// Wave 0 alone takes the decisions after a barrier and leaves them in LDS: the
// block's 16 waves share four SIMDs, so a few hundred instructions that all of
// them execute take four times as long (2.8 us a level against 1.0).
__device__ __forceinline__ bool traverse_joint(Ctx& c, int32_t root, int64_t set_size, int64_t* seeded_out) {
    KernelArgs& a = c.args();
    Smem& sm = c.sm;
    GiantState* gs = a.gs;
    if (c.tid == 0) {
        sm.dir[0] = sm.dir[1] = Dir{0, 0, 0, 0, 0};
        sm.flow = kLive | kLive << 1;
    }
    *seeded_out = 1;
    if (a.n_roots > 0) {
        // level-0 input of both directions: every graph's root, marked
        // visited, queued or split into hub items like any claimed vertex
        int seeded = 0;
        uint32_t cnt[4];
        for (int dir = 0; dir < 2; ++dir) {
            PairQueue wq{c.stage(), 0};
            HubStage hs{sm.hv[c.wave], sm.hs[c.wave], sm.hd[c.wave], 0, 0, kSeedChunk};
            const int32_t* beg = dir ? a.bwb : a.fwb;
            uint64_t* vis = dir ? a.bvis : a.fvis;
            uint64_t* q0 = dir ? a.qb0 : a.q0;
            HubItem* h0 = dir ? a.hb0 : a.h0;
            int64_t unused = 0;
            const bool fits = a.n_roots + beg[a.V] / kSeedChunk <= a.hub_cap;
            for (int64_t ib = (int64_t)c.b * kGBlock + c.wave * kWave; ib < a.n_roots; ib += (int64_t)c.G * kGBlock) {
                const int64_t i = ib + c.lane;
                const int32_t r = i < a.n_roots ? a.roots[i] : -1;
                const bool ok = r >= 0 && r < a.V;
                if (ok) atomicOr(reinterpret_cast<unsigned long long*>(vis + (r >> 6)), 1ull << (r & 63));
                if (dir == 0) seeded += ok;
                push_next(ok, r, beg, wq, q0, &gs->qn[dir][0].v, hs, h0, &gs->hn[dir][0].v, unused,
                          fits ? kSeedHubDeg : kGiantHubDeg);
            }
            block_flush_both(c, wq, q0, &gs->qn[dir][0].v, hs, h0, &gs->hn[dir][0].v);
            cnt[2 * dir] = wq.sent;
            cnt[2 * dir + 1] = hs.sent;
        }
        int64_t r[8];
        if (!gsync_sum<8, true>(c, {(uint32_t)wave_sum(seeded), 0, cnt[0], cnt[1], 0, 0, cnt[2], cnt[3]}, r))
            return false;
        *seeded_out = r[0];
        if (c.tid == 0) {
            sm.dir[0].nq = (int32_t)r[2];
            sm.dir[0].nh = (int32_t)r[3];
            sm.dir[1].nq = (int32_t)r[6];
            sm.dir[1].nh = (int32_t)r[7];
        }
    }
    __syncthreads();
    while (true) {
        const int flow = lane_get(sm.flow, 0);
        if (!(flow & (kLive | kLive << 1))) break;
        const bool tr = a.trace != 0;
        const int64_t tl0 = tr ? (int64_t)wall_clock64() : 0;
        // One copy of the level's code serves both directions: the
        // instruction cache (64 KB for two CUs) does not hold two.
        // Two bottom-up levels, which have no block barriers inside, run side
        // by side on half of every block's waves each: a small one is a chain
        // of round trips, and the two chains then overlap (same box: 700 K
        // vertices 183 -> 174 us, 3 M at edge factor 3 271 -> 250 us, R-MAT s24
        // 383 -> 364 us).
        const bool both = (flow & (kLive | kLive << 1)) == (kLive | kLive << 1);
        const bool half = both && lane_get(sm.dir[0].mode, 0) == 1 && lane_get(sm.dir[1].mode, 0) == 1;
        uint32_t pay[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 1
        for (int it = 0; it < (half ? 1 : 2); ++it) {
            const int dir = half ? __builtin_amdgcn_readfirstlane(c.wave / (kW / 2)) : it;
            if (!(flow & (kLive << dir))) continue;
            const int mode = lane_get(sm.dir[dir].mode, 0);
            const int32_t L = lane_get(sm.dir[dir].L, 0);
            const int64_t edges0 = c.edges_td;
            Level lv{0, 0, 0, 0};
            level_work(c, mode, L, lane_get(sm.dir[dir].nq, 0), lane_get(sm.dir[dir].nh, 0), dir, root,
                       both ? kNarrowShort : kNarrowLong, half, (flow & (kGather << dir)) != 0, lv);
            lv.found = wave_sum(lv.found);
            lv.edges = wave_sum(lv.edges);
            // this wave's part of the work counters
            const bool td = mode != 1;
            if (td) {
                c.found_td += (uint32_t)lv.found;
            } else {
                c.found_bu += (uint32_t)lv.found;
                c.edges_bu += (uint32_t)lv.edges;
            }
            if (tr && L < kLevelTrace && c.lane == 0) {
                using ull = unsigned long long;
                if (c.edges_td > edges0)
                    atomicAdd(reinterpret_cast<ull*>(&gs->lv_edges[dir][L]), (ull)(c.edges_td - edges0));
                if (c.wave % (half ? kW / 2 : kW) == 0) {  // the direction's first wave of each block
                    const ull wt = (ull)((int64_t)wall_clock64() - tl0);
                    if (!td) atomicMax(reinterpret_cast<ull*>(&gs->lv_cp[dir][L][0]), (ull)(uint32_t)lv.edges);
                    atomicMax(reinterpret_cast<ull*>(&gs->lv_wmax[dir][L]), wt);
                    atomicMax(reinterpret_cast<ull*>(&gs->lv_wmin[dir][L]), ~wt);
                    if (!td && dir == 0 && c.b < 1024 && gs->bu1_scan[c.b] == 0) {
                        gs->bu1_scan[c.b] = (uint32_t)lv.edges + 1;
                        gs->bu1_work[c.b] = (int64_t)wt;
                    }
                }
            }
            if (dir) {
                pay[4] = (uint32_t)lv.found;
                pay[5] = (uint32_t)lv.edges;
                pay[6] = lv.nq;
                pay[7] = lv.nh;
            } else {
                pay[0] = (uint32_t)lv.found;
                pay[1] = (uint32_t)lv.edges;
                pay[2] = lv.nq;
                pay[3] = lv.nh;
            }
        }
        // counters of level L+2: last used in level L-1, first written in level
        // L+1 (reset here, before the barrier)
        if (c.b == 0 && c.tid < 2) {
            const int32_t L = sm.dir[c.tid].L;
            st_agent(&gs->qn[c.tid][(L + 2) % 3].v, 0);
            st_agent(&gs->hn[c.tid][(L + 2) % 3].v, 0);
        }
        // Top-down levels read what other blocks wrote in the level before
        // through coherent loads (queue entries, hub items, counts), a
        // candidate bitmap that is fixed during the traversal, and visited
        // bits only as a hint for the claim atomics: their barriers skip the
        // L2 invalidation (the acquire below catches up where needed).
        stage_words<8>(c, pay);
        SumFold<8> fold;
        if (!gsync_with<8, false>(c, [&c]() { return staged_sum(c.sm, c.lane); }, fold)) return false;
        if (c.wave == 0) {
            // per direction: the level's totals, the end test and the switches
            bool acquire = false;
            int next = 0;
#pragma unroll 1
            for (int dir = 0; dir < 2; ++dir) {
                if (!(flow & (kLive << dir))) continue;
                auto total = [&](int w) {
                    return lane_get(sm.tot[0][4 * dir + w], 0) + lane_get(sm.tot[1][4 * dir + w], 0);
                };
                const int64_t found = total(0);
                const int64_t next_edges = total(1);  // top-down levels: exact work of the next level
                const int32_t nq = (int32_t)total(2), nh = (int32_t)total(3);
                int mode = lane_get(sm.dir[dir].mode, 0);
                const int32_t L = lane_get(sm.dir[dir].L, 0) + 1;  // levels done now
                const int64_t visited = lane_get(sm.dir[dir].visited, 0) + found;
                const bool td = mode != 1;
                if (c.b == 0 && c.lane == 0 && L <= kLevelTrace) {
                    gs->lv_ts[dir][L - 1] = wall_clock64();
                    gs->lv_found[dir][L - 1] = found;
                    gs->lv_mode[dir][L - 1] = td ? 0 : 1;
                    if (!td) gs->lv_edges[dir][L - 1] = next_edges;
                }
                int bits = 0;
                // a top-down level ends the traversal when it hands nothing on
                // (it may have found something and expanded it in place, or
                // only handed on what it gathered)
                if (td ? nq == 0 && nh == 0 && (found == 0 || a.td_local > 0) : found == 0) {
                    acquire = true;  // what follows reads the visited bits exactly
                    if (dir == 0 && c.b == 0 && c.lane == 0) gs->ts[2] = wall_clock64();  // the forward one's end
                } else if ((int64_t)L > (int64_t)a.V + 2) {
                    if (c.lane == 0) atomicOr(&gs->err.v, 2);
                    bits = kFailed;
                } else {
                    bits = kLive << dir;
                    if (mode == 0) {
                        const double ef = a.switch_rule ? (double)next_edges : (double)found * a.avg_degree;
                        const double er = (double)(set_size - visited) * a.avg_degree;
                        if (er / a.alpha < ef) mode = 1;
                    }
                    // bottom-up levels and the gather read visited bits exactly
                    if (!td || mode == 1) acquire = true;
                    if (!td && ((set_size * 1.0 / a.beta) > found || L - 1 > a.gamma)) {  // this level was bottom-up
                        mode = 2;
                        bits |= kGather << dir;
                    }
                }
                next |= bits;
                const int32_t finds = (int32_t)found;
                if (c.lane == 0)
                    sm.dir[dir] = Dir{mode, L, (int32_t)visited, (bits & (kGather << dir)) ? finds : nq, nh};
            }
            if (acquire) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // as a barrier with ACQ does
            if (c.lane == 0) sm.flow = next;
        }
        __syncthreads();
        if (lane_get(sm.flow, 0) & kFailed) return false;
    }
    return true;
}

// ---- phases after the giant (run when GiantArgs::rest != 0) --------------

// One trim-1 sweep (trim_1_from_fq_gfq, src/trim_1_gfq.h:365-458) over
// fin[0, n): act is updated in place, survivors are pushed to fout.
// trimmed and kept: this wave's counts (the same in every lane).
// With lo >= 0 the block sweeps only fin[lo, lo + n), entries it wrote
// itself, so no barrier has to make other blocks' entries visible first.
__device__ __forceinline__ void trim_sweep(Ctx& c, const int32_t* fin, int64_t n, int32_t* fout, int32_t* fcount,
                                           int64_t lo, int& trimmed, int& kept) {
    KernelArgs& a = c.args();
    WaveQueue wq{c.stage32(), 0};
    const uint64_t* act = a.act;
    auto live = [act](int32_t w, int32_t self) { return w != self && bit_of(act, w); };
    int scanned = 0;
    trimmed = kept = 0;
    const bool local = lo >= 0;
    const int64_t first = local ? c.wave * kWave : (int64_t)c.b * kGBlock + c.wave * kWave;
    const int64_t step = local ? kGBlock : (int64_t)c.G * kGBlock;
    if (local) fin += lo;
    for (int64_t ib = first; ib < n; ib += step) {
        const int64_t i = ib + c.lane;
        int32_t v = 0;
        bool alive = false;
        if (i < n) {
            v = local ? load_agent(&fin[i]) : fin[i];
            alive = bit_of(a.act, v);
        }
        const bool out = wave_any_edge(alive, alive ? a.fwb[v] : 0, alive ? a.fwb[v + 1] : 0, v, a.fwa, live, scanned);
        const bool in =
            wave_any_edge(alive && out, alive ? a.bwb[v] : 0, alive ? a.bwb[v + 1] : 0, v, a.bwa, live, scanned);
        const bool trim = alive && !(out && in);
        if (trim) {
            st_agent(&a.lab[v], v);
            atomicAnd(reinterpret_cast<unsigned long long*>(a.act + (v >> 6)), ~(1ull << (v & 63)));
        }
        trimmed += __popcll(__ballot(trim));
        kept += __popcll(__ballot(alive && !trim));
        wq_push<true>(wq, alive && !trim, v, fout, fcount);
    }
    block_flush(c, wq, fout, fcount);
}

// ---- small-SCC strategies after the trims (wcc_mode 1 and 2), run by
// k_tail: a second cooperative launch on the same stream, made only when the
// giant phase leaves active vertices.  A kernel of their own keeps k_giant's
// code (and its register allocation) as it is.
// col[v] = smallest id of v's WCC in the active subgraph, by label
// propagation over in- and out-edges with jumps along the colour chain, to a
// fixed point (coloring_wcc, src/color_propagation.h:468-593, which keeps
// the largest id).  The count of changed vertices rides on the barrier, so
// every block leaves after the same sweep.
__device__ __forceinline__ bool lp_wcc(Ctx& c, const int32_t* q, int64_t n, int64_t& rounds) {
    KernelArgs& a = c.args();
    const int64_t nthreads = (int64_t)c.G * kGBlock;
    const int64_t gt = (int64_t)c.b * kGBlock + c.tid;
    int32_t* col = a.parent;
    for (int64_t i = gt; i < n; i += nthreads) st_agent(&col[q[i]], q[i]);
    if (!gsync(c)) return false;
    for (rounds = 1;; ++rounds) {
        int changed = 0;
        for (int64_t i = gt; i < n; i += nthreads) {
            const int32_t v = q[i];
            const int32_t c0 = load_agent(&col[v]);
            int32_t m = c0;
            for (int dir = 0; dir < 2; ++dir) {
                const int32_t* beg = dir ? a.bwb : a.fwb;
                const int32_t* adj = dir ? a.bwa : a.fwa;
                const int32_t e = beg[v + 1];
                for (int32_t k = beg[v]; k < e; ++k) {
                    const int32_t w = adj[k];
                    if (w != v && bit_of(a.act, w)) m = min(m, load_agent(&col[w]));
                }
            }
            // colours are ids of active members: follow the chain (at most
            // 100 hops, as the reference's path compression)
            for (int hop = 0; hop < 100; ++hop) {
                const int32_t nx = load_agent(&col[m]);
                if (nx >= m) break;
                m = nx;
            }
            if (m < c0) {
                atomicMin(&col[v], m);
                ++changed;
            }
        }
        int64_t r[4];
        if (!gsync_sum<4, true>(c, {(uint32_t)wave_sum(changed), 0, 0, 0}, r)) return false;
        if (r[0] == 0) return true;
        if (rounds > (int64_t)a.V + 2) {
            if (c.tid == 0) atomicOr(&a.gs->err.v, 2);
            return false;
        }
    }
}

__device__ __forceinline__ int32_t key_colour(uint64_t k) { return (int32_t)(uint32_t)k; }

// Sweeps of a fixed-point iteration by one block over its own vertices, until
// one of them changes nothing there or `most` are done: between two
// grid barriers, so what came from other blocks goes as far as it can.  A
// block's vertices are neighbours in the queue, which is ascending, so most
// edges of a graph with local ids stay inside it.  sweep() returns what this
// thread changed; the sum over the sweeps comes back.
constexpr int kBlockSweeps = 16;
// With more vertices than this for each thread of the grid, a block sweeps
// once: its sweep takes longer than the grid barrier it saves, and with many
// vertices most edges lead out of the block's slices.  Up to 16 times against
// once: random DAGs of 4-cycles, 3 M vertices 67 / 46 ms, 1 M with 6 edges each
// 55 / 46, 200,000 with 20 edges 96 / 96; edges to the next 12 ids, 4 M vertices
// 1.81 / 1.15 s, 1 M 0.27 / 0.18, 300,000 34.9 / 46.2 ms, 20,000 with 2 edges
// 1.95 / 2.11.  The rule is the same for all blocks on purpose: where some
// sweep once and some 16 times (by their own lists, or by a time limit), the
// former wait for the latter, 20,000 vertices with 20 edges each 86 for 46 ms.
constexpr int kBlockSweepsPer = 2;
template <class Sweep>
__device__ __forceinline__ int block_sweeps(Ctx& c, bool one, int most, Sweep sweep) {
    int all = 0;
    for (int k = 0; k < most; ++k) {
        const int changed = sweep();
        all += changed;
        wait_vm();  // the other waves' next sweep reads it
        if (!__syncthreads_or(changed)) return one ? 0 : all;  // alone: that was the fixed point
    }
    return all;
}

// colour_scc's barrier, with the sum of x over the threads: of the grid, or
// of one block while the others have left.
template <bool ACQ>
__device__ __forceinline__ bool colour_sync(Ctx& c, bool one, int x, int64_t& sum) {
    if (!one) {
        int64_t r[4];
        if (!gsync_sum<4, ACQ>(c, {(uint32_t)wave_sum(x), 0, 0, 0}, r)) return false;
        sum = r[0];
        return true;
    }
    wait_vm();
    sum = block_sum(x, c.sm);
    if (ACQ) {
        if (c.wave == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        __syncthreads();
    }
    return true;
}

// The colouring SCC method (graph_color, src/color_propagation.h:9-467).  A
// vertex's priority is (active out-degree + 5) x active in-degree
// (degree_rank, :9-58; clipped to 31 bits here, which can only change ties:
// the priority chooses the work, never the labels).  Each round every active
// vertex takes the largest (priority, id) key among the vertices that reach
// it: propagation over in-edges with jumps along the colour chain
// (color_propagation, :64-200), to a fixed point.  A vertex whose key is its
// own is a root, and the vertices of its colour that reach it are its SCC
// (color_identify, :203-260; here a fixed point of backward sweeps for all
// roots at once instead of one search per root).  Those SCCs are labelled
// with their smallest id and leave the active set; the rest start the next
// round with their own keys again (color_init, :262-290).  Each round labels
// at least the SCC of the largest key of every weakly connected piece.
//
// Nearly all of it is barriers and round trips: about 25 sweeps a round over
// a chain of 20,000 SCCs.  So blocks sweep on their own between barriers,
// barriers within a round skip the acquire (keys, stamps and minima are read
// coherently), entries are read four at a time, and a rest of at most a block's
// threads is left to one block: k_tail 924 -> 590 us there, 300 SCCs
// 400 -> 283.
__device__ __forceinline__ bool colour_scc(Ctx& c, int& cur, int64_t n, int s, int64_t& rounds, int64_t& sccs) {
    KernelArgs& a = c.args();
    GiantState* gs = a.gs;
    const int64_t nthreads = (int64_t)c.G * kGBlock;
    const int64_t gt = (int64_t)c.b * kGBlock + c.tid;
    auto buf = [&a](int k) { return k ? a.fq : a.fq_alt; };
    using ull = unsigned long long;
    // List entries whose keys or stamps are read together.  They come from past
    // the L2, the active bits mostly from it, and after the first rounds most
    // entries are active no more: only those that are get read.  (All of them
    // at once, which saves the bits' round trip: random DAGs of 20,000 and 1 M
    // vertices with 20 and 6 edges each 46 and 73 ms, 39 and 47 this way.)
    constexpr int kAhead = 4;
    {  // degree rank, once, into parent
        const int32_t* q = buf(cur);
        for (int64_t i = gt; i < n; i += nthreads) {
            const int32_t v = q[i];
            int64_t od = 0, id = 0;
            for (int32_t k = a.fwb[v]; k < a.fwb[v + 1]; ++k) od += bit_of(a.act, a.fwa[k]);
            for (int32_t k = a.bwb[v]; k < a.bwb[v + 1]; ++k) id += bit_of(a.act, a.bwa[k]);
            st_agent(&a.parent[v], (int32_t)min<int64_t>((od + 5) * id, INT32_MAX));
        }
    }
    sccs = 0;
    for (rounds = 1;; ++rounds) {
        const bool one = n <= kGBlock;
        if (one && c.b != 0) return true;
        const int most = n > kBlockSweepsPer * nthreads ? 1 : kBlockSweeps;
        const int32_t* q = buf(cur);
        int32_t* qn = buf(cur ^ 1);
        int32_t* cnt = &gs->fqn[s % 3].v;  // last read three rounds (or sweeps) ago
        if (c.b == 0 && c.tid == 0) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int64_t i = gt; i < n; i += nthreads) {
            const int32_t v = q[i];
            st_agent(&a.ckey[v], ((uint64_t)(uint32_t)load_agent(&a.parent[v]) << 32) | (uint32_t)v);
            st_agent(&a.stamp[v], -1);
        }
        int64_t got;
        if (!colour_sync<false>(c, one, 0, got)) return false;
        for (int64_t it = 0;; ++it) {  // largest key among the vertices that reach v
            const int changed = block_sweeps(c, one, most, [&]() {
                int ch = 0;
                for (int64_t i = gt; i < n; i += nthreads) {
                    const int32_t v = q[i];
                    const uint64_t k0 = load_agent(&a.ckey[v]);
                    uint64_t k = k0;
                    const int32_t end = a.bwb[v + 1];
                    for (int32_t e = a.bwb[v]; e < end; e += kAhead) {
                        int32_t w[kAhead];
                        bool on[kAhead];
                        uint64_t kw[kAhead];
#pragma unroll
                        for (int j = 0; j < kAhead; ++j) w[j] = a.bwa[min(e + j, end - 1)];
#pragma unroll
                        for (int j = 0; j < kAhead; ++j) on[j] = e + j < end && w[j] != v && bit_of(a.act, w[j]);
#pragma unroll
                        for (int j = 0; j < kAhead; ++j) kw[j] = on[j] ? load_agent(&a.ckey[w[j]]) : 0;
#pragma unroll
                        for (int j = 0; j < kAhead; ++j) k = max(k, kw[j]);
                    }
                    for (int hop = 0; hop < 100; ++hop) {  // the colour's own key, and so on
                        const uint64_t kc = load_agent(&a.ckey[key_colour(k)]);
                        if (kc <= k) break;
                        k = kc;
                    }
                    if (k > k0) {
                        atomicMax(reinterpret_cast<ull*>(&a.ckey[v]), (ull)k);
                        ++ch;
                    }
                }
                return ch;
            });
            if (!colour_sync<false>(c, one, changed, got)) return false;
            if (got == 0) break;
            if (it > (int64_t)a.V + 2) {
                if (c.tid == 0) atomicOr(&gs->err.v, 2);
                return false;
            }
        }
        for (int64_t i = gt; i < n; i += nthreads) {  // roots
            const int32_t v = q[i];
            if (key_colour(load_agent(&a.ckey[v])) == v) {
                st_agent(&a.stamp[v], v);
                st_agent(&a.aux[v], v);
            }
        }
        if (!colour_sync<false>(c, one, 0, got)) return false;
        for (int64_t it = 0;; ++it) {  // v joins its colour's SCC through an out-neighbour in it
            const int changed = block_sweeps(c, one, most, [&]() {
                int ch = 0;
                for (int64_t i = gt; i < n; i += nthreads) {
                    const int32_t v = q[i];
                    if (load_agent(&a.stamp[v]) >= 0) continue;
                    const int32_t r = key_colour(load_agent(&a.ckey[v]));
                    const int32_t end = a.fwb[v + 1];
                    for (int32_t e = a.fwb[v]; e < end; e += kAhead) {
                        int32_t u[kAhead], su[kAhead];
                        bool on[kAhead];
#pragma unroll
                        for (int j = 0; j < kAhead; ++j) u[j] = a.fwa[min(e + j, end - 1)];
#pragma unroll
                        for (int j = 0; j < kAhead; ++j) on[j] = e + j < end && u[j] != v && bit_of(a.act, u[j]);
#pragma unroll
                        for (int j = 0; j < kAhead; ++j) su[j] = on[j] ? load_agent(&a.stamp[u[j]]) : -1;
                        bool join = false;
#pragma unroll
                        for (int j = 0; j < kAhead; ++j) join = join || su[j] == r;
                        if (join) {
                            st_agent(&a.stamp[v], r);
                            ++ch;
                            break;
                        }
                    }
                }
                return ch;
            });
            if (!colour_sync<false>(c, one, changed, got)) return false;
            if (got == 0) break;
            if (it > (int64_t)a.V + 2) {
                if (c.tid == 0) atomicOr(&gs->err.v, 2);
                return false;
            }
        }
        for (int64_t i = gt; i < n; i += nthreads) {  // smallest member per SCC
            const int32_t v = q[i];
            const int32_t r = load_agent(&a.stamp[v]);
            if (r >= 0 && r != v) atomicMin(&a.aux[r], v);
        }
        if (!colour_sync<false>(c, one, 0, got)) return false;
        // label the SCCs found, take them out of the active set, queue the rest
        WaveQueue wq{c.stage32(), 0};
        int found = 0;
        for (int64_t ib = (int64_t)c.b * kGBlock + c.wave * kWave; ib < n; ib += nthreads) {
            const int64_t i = ib + c.lane;
            int32_t v = 0, r = -1;
            if (i < n) {
                v = q[i];
                r = load_agent(&a.stamp[v]);
                if (r >= 0) {
                    st_agent(&a.lab[v], load_agent(&a.aux[r]));
                    atomicAnd(reinterpret_cast<ull*>(a.act + (v >> 6)), ~(1ull << (v & 63)));
                    found += r == v;
                }
            }
            wq_push<true>(wq, i < n && r < 0, v, qn, cnt);
        }
        block_flush(c, wq, qn, cnt);
        if (!colour_sync<true>(c, one, found, got)) return false;  // the active set and the queue are read plainly
        sccs += got;
        n = load_agent(cnt);
        cur ^= 1;
        ++s;
        if (n == 0) return true;
        if (rounds > (int64_t)a.V + 2) {
            if (c.tid == 0) atomicOr(&gs->err.v, 2);
            return false;
        }
    }
}

// Trims and WCC after the giant.  Returns false after a failed barrier.
// Pattern checks: a vertex with more entries than this in either list is
// checked by a whole wave instead of one lane.
constexpr int kPatternLong = 32;

// own_lo / own_n: the slice of the active queue this block wrote; the first
// trim sweep takes only it, so the queue needs no barrier before it (one is
// taken when no sweep comes first).
__device__ __forceinline__ bool rest_phase(Ctx& c, int64_t fq0, int64_t n, int64_t own_lo, int64_t own_n,
                                           int64_t& n_left) {
    KernelArgs& a = c.args();
    GiantState* gs = a.gs;
    int cur = 1, s = 0;
    auto buf = [&a](int k) { return k ? a.fq : a.fq_alt; };
    int64_t prev = fq0, trim1 = 0, p2 = 0, p3 = 0;
    int it = 0;
    const int64_t nthreads = (int64_t)c.G * kGBlock;
    const int64_t gt = (int64_t)c.b * kGBlock + c.tid;
    // Sweep s pushes at fqn[s % 3]; what it kept is summed by its barrier.
    // It clears fqn[(s + 1) % 3] for the next sweep: that counter was last
    // used in sweep s - 2, before the barrier that ended it.
    auto sweep = [&]() -> bool {
        if (c.b == 0 && c.tid == 0)
            __hip_atomic_store(&gs->fqn[(s + 1) % 3].v, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int t, kept;
        trim_sweep(c, buf(cur), s == 0 ? own_n : n, buf(cur ^ 1), &gs->fqn[s % 3].v, s == 0 ? own_lo : -1, t, kept);
        int64_t r[4];
        if (!gsync_sum<4, true>(c, {(uint32_t)t, (uint32_t)kept, 0, 0}, r)) return false;
        trim1 += r[0];
        n = r[1];
        cur ^= 1;
        ++s;
        return true;
    };
    // P7: up to trim_times sweeps with the theta stop rule (src/scc_core.cpp:562-602);
    // the first comparison is against the pre-giant queue, as there.
    while (prev > 0 && it < a.trim_times && n > 0) {
        if (!sweep()) return false;
        if (prev - n < prev * a.theta) break;
        prev = n;
        ++it;
    }
    bool wcc = false;
    if (n > 0 && s == 0 && !gsync(c)) return false;  // no sweep: the queue's barrier
    if (n > 0) {
        // P8-P10: pattern detection against the current act, then commit.
        // Over the active queue (trim_*_from_fq, src/trim_2_3.h:146-283,
        // 482-677, 881-1080) or, with trim_scope 1, over every active vertex
        // of the graph (trim_*_from_graph, src/trim_2_3.h:9-144, 287-480,
        // 682-879): the same detections, a different walk.
        const int32_t* f = buf(cur);
        auto each_active = [&](auto&& fn) {
            if (a.trim_scope) {
                for (int64_t w = gt; w < a.nwords; w += nthreads) {
                    uint64_t m = a.act[w];
                    while (m) {
                        fn((int32_t)(w * 64 + __ffsll((unsigned long long)m) - 1));
                        m &= m - 1;
                    }
                }
            } else {
                for (int64_t i = gt; i < n; i += nthreads) {
                    const int32_t v = f[i];
                    if (bit_of(a.act, v)) fn(v);
                }
            }
        };
        // A lane checks its own vertex, except one with a long list (a lane
        // would walk it entry by entry): those are queued in the wave's LDS
        // buffer and checked afterwards by the whole wave, 64 entries a step.
        {
            int32_t* lq = c.stage32();
            int32_t& nlq = c.sm.wcnt[0][c.wave];
            if (c.lane == 0) nlq = 0;
            wave_sync();
            each_active([&](int32_t v) {
                const int32_t dv = max(a.fwb[v + 1] - a.fwb[v], a.bwb[v + 1] - a.bwb[v]);
                if (dv > kPatternLong) {
                    const int slot = atomicAdd(&nlq, 1);
                    if (slot < kWaveBuf) {
                        lq[slot] = v;
                        return;
                    }
                }
                pattern_check(a.fwb, a.fwa, a.bwb, a.bwa, a.lab, a.stamp, a.act, v);
            });
            wave_sync();
            const int nl = min(nlq, kWaveBuf);
            for (int j = 0; j < nl; ++j)
                pattern_check<true>(a.fwb, a.fwa, a.bwb, a.bwa, a.lab, a.stamp, a.act, lq[j]);
        }
        if (!gsync(c)) return false;
        int c2 = 0, c3 = 0;
        each_active([&](int32_t v) {
            if (a.lab[v] >= 0) {
                atomicAnd(reinterpret_cast<unsigned long long*>(a.act + (v >> 6)), ~(1ull << (v & 63)));
                if (a.stamp[v] == 2) ++c2;
                else ++c3;
            }
        });
        int64_t r[4];
        if (!gsync_sum<4, true>(c, {(uint32_t)wave_sum(c2), (uint32_t)wave_sum(c3), 0, 0}, r)) return false;
        p2 = r[0];
        p3 = r[1];
        // P11: one more trim-1 sweep
        if (!sweep()) return false;
        // (wcc_mode 1 and 2 run in k_tail, launched when something is left)
        if (n > 0 && a.wcc_mode == 0) {
            // P12: WCC by union-find; parent = smallest id of the WCC.  A
            // vertex starts under the smallest active neighbour among the
            // first entries of its lists, if that is smaller, then under its
            // root by that: no atomics, and most edges then find both ends
            // under one root in two loads (12,500 WCCs of 28 vertices: 102 ->
            // 26 us with the passes and barriers before the hooks, which take
            // 55 us without the second pass).
            constexpr int32_t kFirstEntries = 4;
            const int32_t* g = buf(cur);
            for (int64_t i = gt; i < n; i += nthreads) {
                const int32_t v = g[i];
                int32_t m = v;
                for (int dir = 0; dir < 2; ++dir) {
                    const int32_t* adj = dir ? a.bwa : a.fwa;
                    const int32_t p = (dir ? a.bwb : a.fwb)[v], e = min((dir ? a.bwb : a.fwb)[v + 1], p + kFirstEntries);
                    for (int32_t k = p; k < e; ++k) {
                        const int32_t w = adj[k];
                        if (w < m && bit_of(a.act, w)) m = w;
                    }
                }
                st_agent(&a.parent[v], m);
            }
            if (!gsync<false>(c)) return false;
            // every vertex under its root so far: the hooks' walks are short
            for (int64_t i = gt; i < n; i += nthreads) {
                const int32_t v = g[i];
                st_agent(&a.parent[v], uf_find(a.parent, v));
            }
            if (!gsync<false>(c)) return false;
            for (int64_t i = gt; i < n; i += nthreads) {
                const int32_t v = g[i];
                const int32_t e = a.fwb[v + 1];
                int32_t x = v;
                for (int32_t k = a.fwb[v]; k < e; ++k) {
                    const int32_t w = a.fwa[k];
                    if (w == v || !bit_of(a.act, w)) continue;
                    int32_t y = w;
                    while (true) {
                        x = uf_root(a.parent, x);
                        y = uf_root(a.parent, y);
                        if (x == y) break;
                        if (x < y) {
                            const int32_t t = x;
                            x = y;
                            y = t;
                        }
                        if (atomicCAS(&a.parent[x], x, y) == x) {
                            x = y;
                            break;
                        }
                    }
                }
            }
            if (!gsync(c)) return false;
            for (int64_t i = gt; i < n; i += nthreads) {
                const int32_t v = g[i];
                st_agent(&a.parent[v], uf_find(a.parent, v));
            }
            wcc = true;
        }
    }
    if (c.b == 0 && c.tid == 0) {
        gs->n_final = n;
        gs->final_sel = cur;
        gs->trim1 = trim1;
        gs->pat2 = p2;
        gs->pat3 = p3;
        gs->sweeps = s;
        gs->wcc_done = wcc;
        a.fq_n_ctl[cur] = (int32_t)n;
    }
    n_left = n;
    return true;
}

// Labels of words [wb, we), the block's own: the giant's from its bitmap, the
// vertices' own ids elsewhere, and for the vertices the giant phase left (a.act
// then, a.snap later) -1 into the context's array, or, FINAL, what the
// context's array says by then into the caller's.  One word per lane: a wave
// loads its share of the words, up to 64 at once, then writes them four words
// at a time, four consecutive labels a lane (coalesced 1 KB stores, no loads in
// the loop but for the vertices left).  (64 whatever there are left the 43
// words a block of 700 K vertices to one wave: 162 us a solve against 154.)
//
// The caller's array is written at the very end, when no barrier is left that
// could fail and nobody reads the graph any more: it stays as it was if the
// solve fails, and may lie over the graph's arrays.  (A copy after the launch
// instead reads and writes the labels once more and costs another host wait:
// R-MAT s24 403 -> 387 us, 700 K vertices 203 -> 190 us.)
template <bool FINAL>
__device__ __forceinline__ void write_labels(Ctx& c, int64_t wb, int64_t we, bool traversed, int32_t gmin) {
    KernelArgs& a = c.args();
    const bool multi = a.n_roots > 0;
    int32_t* lab = FINAL ? a.lab2 : a.lab;
    const uint64_t* left = FINAL ? a.snap : a.act;
    const bool wide = (reinterpret_cast<uintptr_t>(lab) & 15) == 0;
    const int share = (int)min(((we - wb + kW - 1) / kW + 3) & ~(int64_t)3, (int64_t)kWave);
    for (int64_t base = wb + (int64_t)c.wave * share; base < we; base += (int64_t)kW * share) {
        const int64_t w = base + c.lane;
        uint64_t ac = 0, g = 0, sw = 0;
        if (w < we) {
            ac = left[w];
            g = traversed ? a.bvis[w] : 0ull;
            sw = a.sel ? a.sel[w] : ~0ull;  // unselected vertices keep whatever label they had
        }
        const int nw = (int)min<int64_t>(share, we - base);
        const int q = (c.lane & 15) * 4;  // this lane's first bit in its word
        for (int j = 0; j < nw; j += 4) {
            const int src = j + (c.lane >> 4);  // this lane's word in the group of four
            const uint64_t aj = lane_from(ac, src), gj = lane_from(g, src), sj = lane_from(sw, src);
            if (src >= nw) continue;
            const int64_t v0 = (base + src) * 64 + q;
            int32_t l[4];
            bool all = v0 + 3 < a.V;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int64_t v = v0 + k;
                const bool gi = (gj >> (q + k)) & 1ull, rest = (aj >> (q + k)) & 1ull;
                l[k] = gi ? (multi ? (int32_t)v : gmin) : (rest ? -1 : (int32_t)v);
                if (FINAL && !gi && rest) l[k] = a.lab[v];
                all = all && ((sj >> (q + k)) & 1ull);
            }
            if (all && wide) {
                st_agent4(&lab[v0], l[0], l[1], l[2], l[3]);
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (v0 + k < a.V && ((sj >> (q + k)) & 1ull)) st_agent(&lab[v0 + k], l[k]);
            }
        }
    }
}

}  // namespace

__global__ __launch_bounds__(kGBlock) void k_giant(const GiantArgs) {
    KernelArgs& a = kernel_args();
    __shared__ Smem sm;
    Ctx c{(int)gridDim.x, (int)blockIdx.x, (int)threadIdx.x, lane_id(), wave_id(), sm, 0, 0, 0, 0, 0};
    GiantState* gs = a.gs;
    // Block 0 clears the state and the control block.  No other block writes
    // either before the first barrier (whose records are not part of them),
    // so none has to wait for it, and the barrier waits for the stores.
    if (c.b == 0) {
        int64_t* p = reinterpret_cast<int64_t*>(gs);
        for (int i = c.tid; i < a.state_words; i += kGBlock) st_agent(&p[i], (int64_t)0);
        int64_t* q = reinterpret_cast<int64_t*>(a.ctl);
        for (int i = c.tid; i < a.ctl_words; i += kGBlock) st_agent(&q[i], (int64_t)0);
    }
    const int64_t total_waves = (int64_t)c.G * kW;
    const int64_t gwave = (int64_t)c.b * kW + c.wave;
    const bool stamp = c.b == 0 && c.tid == 0;  // phase timestamps (constant-rate clock)
    const unsigned long long t_begin = wall_clock64();  // launch ramp: when each block started

    // ---- phase A: trim-1-first (raw degree 0 either way), act bitmap,
    // cleared traversal bitmaps, pivot = largest out*in (lowest id on ties).
    int64_t bestp = 0, surv = 0;
    int32_t besti = INT32_MAX;
    // a wave takes kUA consecutive words at a time and issues all their offset
    // loads before it uses any of them; lane i loads beg[v] once and takes
    // beg[v + 1] from lane i + 1 (lane 63 from the next word's lane 0)
    constexpr int kUA = 16;
    // lane u < kUA holds the previous step's word w0 + u until the next
    // step's loads are out: a load's wait also waits for earlier stores
    int64_t pword = -1;
    uint64_t pmine = 0;
    for (int64_t w0 = gwave * kUA; w0 < a.nwords; w0 += total_waves * kUA) {
        int32_t fo[kUA], bo[kUA];
#pragma unroll
        for (int u = 0; u < kUA; ++u) {
            const int64_t v = (w0 + u) * 64 + c.lane;
            fo[u] = v <= a.V ? a.fwb[v] : 0;
            bo[u] = v <= a.V ? a.bwb[v] : 0;
        }
        int32_t fl = 0, bl = 0;  // offsets of the vertex after the last word
        const int64_t vl = (w0 + kUA) * 64;
        if (c.lane == kWave - 1 && vl <= a.V) {
            fl = a.fwb[vl];
            bl = a.bwb[vl];
        }
        // vertices outside the selection never become active: lane u < kUA
        // loads word w0 + u's selection
        const uint64_t lsel = (c.lane < kUA && w0 + c.lane < a.nwords) ? (a.sel ? a.sel[w0 + c.lane] : ~0ull) : 0ull;
        if (pword >= 0) {
            st_agent(&a.act[pword], pmine);
            st_agent(&a.fvis[pword], (uint64_t)0);
            st_agent(&a.bvis[pword], (uint64_t)0);
            pword = -1;
        }
        uint64_t mine = 0;  // lane u < kUA keeps word w0 + u's survivors
#pragma unroll
        for (int u = 0; u < kUA; ++u) {
            const int64_t w = w0 + u, v = w * 64 + c.lane;
            const int32_t f0 = u + 1 < kUA ? lane_get(fo[u + 1 < kUA ? u + 1 : u], 0) : fl;
            const int32_t b0 = u + 1 < kUA ? lane_get(bo[u + 1 < kUA ? u + 1 : u], 0) : bl;
            int32_t fn = __shfl_down(fo[u], 1, kWave), bn = __shfl_down(bo[u], 1, kWave);
            if (c.lane == kWave - 1) {
                fn = f0;
                bn = b0;
            }
            const uint64_t sw = lane_get(lsel, u);
            const bool on = v < a.V && ((sw >> c.lane) & 1ull);
            const int32_t od = fn - fo[u], id = bn - bo[u];
            const bool s = on && od > 0 && id > 0;
            if (s) {
                const int64_t p = a.wrap32 ? (int64_t)(int32_t)((uint32_t)od * (uint32_t)id) : (int64_t)od * id;
                if (p > 0 && pivot_better(p, (int32_t)v, bestp, besti)) {
                    bestp = p;
                    besti = (int32_t)v;
                }
            }
            const uint64_t m = __ballot(s);
            if (c.lane == u) mine = m;
        }
        if (c.lane < kUA && w0 + c.lane < a.nwords) {
            pword = w0 + c.lane;
            pmine = mine;
            surv += __popcll(mine);
        }
    }
    if (pword >= 0) {
        st_agent(&a.act[pword], pmine);
        st_agent(&a.fvis[pword], (uint64_t)0);
        st_agent(&a.bvis[pword], (uint64_t)0);
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
        const int64_t op = __shfl_xor(bestp, d, kWave);
        const int32_t oi = __shfl_xor(besti, d, kWave);
        if (pivot_better(op, oi, bestp, besti)) {
            bestp = op;
            besti = oi;
        }
    }
    surv = wave_sum(surv);
    if (c.lane == 0) {
        sm.red2[c.wave] = bestp;
        sm.bi[c.wave] = besti;
        sm.red[c.wave] = surv;
    }
    const unsigned long long t_arrive = a.trace ? wall_clock64() : 0;
    // the barrier carries each block's candidate and survivor count
    PivotFold pf;
    const bool go = gsync_with<4, true>(
        c,
        [&]() {
            int64_t p = sm.red2[c.lane & 15];
            int32_t id = sm.bi[c.lane & 15];
            const int64_t n = row_incl(sm.red[c.lane & 15], (int64_t)0, [](int64_t x, int64_t y) { return x + y; });
#pragma unroll
            for (int d = kW / 2; d > 0; d >>= 1) {
                const int64_t op = __shfl_xor(p, d, kWave);
                const int32_t oi = __shfl_xor(id, d, kWave);
                if (pivot_better(op, oi, p, id)) {
                    p = op;
                    id = oi;
                }
            }
            const uint32_t nn = (uint32_t)lane_get(n, kW - 1);
            return c.lane == 0 ? (uint32_t)((uint64_t)p >> 32) : c.lane == 1 ? (uint32_t)p : c.lane == 2 ? (uint32_t)id : nn;
        },
        pf);
    if (!go) return;
    bestp = lane_get(sm.tot[0][0], 0);
    besti = (int32_t)lane_get(sm.tot[0][1], 0);
    const int64_t fq0 = lane_get(sm.tot[0][2], 0);
    if (a.trace && c.tid == 0) {  // min as max of ~t (the state starts at 0)
        using ull = unsigned long long;
        atomicMax(reinterpret_cast<ull*>(&gs->t_start[0]), ~t_begin);
        atomicMax(reinterpret_cast<ull*>(&gs->t_start[1]), t_begin);
        atomicMax(reinterpret_cast<ull*>(&gs->t_arrive[0]), ~t_arrive);
        atomicMax(reinterpret_cast<ull*>(&gs->t_arrive[1]), t_arrive);
    }
    const int32_t root = (a.n_roots == 0 && bestp > 0 && besti < a.V) ? besti : -1;
    if (stamp) {
        gs->ts[0] = (int64_t)t_begin;
        gs->ts[1] = wall_clock64();
    }

    int64_t fw_count = 0, bw_reach = 0, fw_levels = 0, bw_levels = 0;
    int32_t gmin = root;
    const bool multi = a.n_roots > 0;
    const bool traversed = multi || root >= 0;
    if (traversed) {
        int64_t seeded = 0;
        if (!traverse_joint(c, root, fq0, &seeded)) return;
        fw_count = sm.dir[0].visited + seeded;
        bw_reach = sm.dir[1].visited + seeded;
        fw_levels = sm.dir[0].L;
        bw_levels = sm.dir[1].L;
    }
    if (stamp) {
        if (!traversed) gs->ts[2] = wall_clock64();
        gs->ts[3] = wall_clock64();  // both directions done
    }

    // ---- post: giant labels, act minus giant, every label written once;
    // each block owns a contiguous word range so the rebuilt active queue
    // comes out ascending without atomics.  First the block's words are
    // narrowed and counted, and the giant's smallest id (its label: no larger
    // than the pivot, which the giant contains) is found among words up to
    // the pivot's; the barrier after the counts reduces it as its key.
    const int64_t per = (a.nwords + c.G - 1) / c.G;
    const int64_t wb = min((int64_t)c.b * per, a.nwords), we = min(wb + per, a.nwords);
    const bool want_min = traversed && !multi;
    // a direction that ended top-down after bottom-up levels has its visited
    // bits in its snapshot
    const bool fsnap = traversed && sm.dir[0].mode == 2, bsnap = traversed && sm.dir[1].mode == 2;
    int64_t cnt = 0, gcnt = 0;
    int32_t mn = INT32_MAX;
    for (int64_t w = wb + c.tid; w < we; w += kGBlock) {
        const uint64_t a0 = a.act[w];
        uint64_t g = 0;
        if (traversed) {  // the giant: reached both ways; bvis keeps only it
            const uint64_t fw = fsnap ? a.snap[w] : a.fvis[w], bw = bsnap ? a.snapb[w] : a.bvis[w];
            g = fw & bw;
            if (fsnap) st_agent(&a.fvis[w], fw);
            if (bsnap || g != bw) st_agent(&a.bvis[w], g);
        }
        if (g) st_agent(&a.act[w], a0 & ~g);
        // the vertices left at -1 below: only they can still be unlabelled at
        // the end (the traversal no longer reads this bitmap)
        st_agent(&a.snap[w], a0 & ~g);
        cnt += __popcll(a0 & ~g);
        gcnt += __popcll(g);
        if (want_min && g && w <= (root >> 6)) mn = min(mn, (int32_t)(w * 64 + __ffsll((unsigned long long)g) - 1));
    }
    const int wmn = wave_min(mn);
    const uint32_t key = wmn < INT32_MAX ? (uint32_t)(INT32_MAX - wmn) : 0u;
    if (a.trace && c.tid == 0) atomicMax((unsigned long long*)&gs->post_cp[0], (unsigned long long)wall_clock64());
    // (vertices, and entries read top-down, once each: a block's fit 32 bits;
    // bottom-up levels read lists again and again, so that count goes in two)
    constexpr int kLowBits = 20;
    stage_words<8>(c, {(uint32_t)wave_sum((int)cnt), (uint32_t)wave_sum((int)gcnt), key, (uint32_t)c.edges_td,
                       (uint32_t)c.edges_bu & ((1u << kLowBits) - 1), (uint32_t)c.found_td, (uint32_t)c.found_bu,
                       (uint32_t)(c.edges_bu >> kLowBits)});
    {
        PostFold f{c.b};
        auto src = [&]() {
            if (c.lane != 2) return staged_sum(sm, c.lane);
            uint32_t k = 0;
            for (int i = 0; i < kW; ++i) k = max(k, sm.bv[2][i]);
            return k;
        };
        if (!gsync_with<8, true>(c, src, f)) return;
    }
    if (want_min) gmin = (int32_t)((int64_t)INT32_MAX - lane_get(sm.tot[0][2], 0));
    int64_t off = lane_get(sm.tot[1][0], 0);  // active vertices of the blocks before this one
    const int64_t tot = lane_get(sm.tot[0][0], 0);
    const int64_t giant = lane_get(sm.tot[0][1], 0);
    if (a.trace && c.tid == 0) atomicMax((unsigned long long*)&gs->post_cp[1], (unsigned long long)wall_clock64());
    // the labels; the vertices left get theirs later
    write_labels<false>(c, wb, we, traversed, gmin);
    // this block's slice of the queue, the active vertices of its own words.
    // The first trim sweep takes it alone (no barrier before it): a sweep
    // clears act bits only of the vertices it sweeps, so no block's sweep
    // touches the words another block is still listing.
    const int64_t own_lo = off;
    for (int64_t base = wb; base < we; base += kGBlock) {
        const int64_t w = base + c.tid;
        const uint64_t m = w < we ? a.act[w] : 0ull;
        int excl, total;
        block_excl_scan<kW>(__popcll(m), excl, total, sm.tmp);
        uint64_t mm = m;
        int64_t o = off + excl;
        while (mm) {
            const int bit = __ffsll((unsigned long long)mm) - 1;
            st_agent(&a.fq[o++], (int32_t)(w * 64 + bit));
            mm &= mm - 1;
        }
        off += total;
    }
    if (a.trace && c.tid == 0) atomicMax((unsigned long long*)&gs->post_cp[2], (unsigned long long)wall_clock64());
    if (c.b == 0) {
        if (c.tid == 0) {
            gs->root = root;
            gs->fq0 = fq0;
            gs->fw_count = fw_count;
            gs->giant = giant;
            gs->bw_reach = bw_reach;
            gs->gmin = gmin;
            gs->fq_n = tot;
            gs->fw_levels = fw_levels;
            gs->bw_levels = bw_levels;
            gs->work[0] = sm.tot[0][3];
            gs->work[1] = sm.tot[0][4] + (sm.tot[0][7] << kLowBits);
            gs->work[2] = sm.tot[0][5];
            gs->work[3] = sm.tot[0][6];
            *a.fq_n_out = (int32_t)tot;
            gs->ts[4] = wall_clock64();
        }
    }
    if (a.rest) {
        __syncthreads();  // the block's queue slice is written
        int64_t n_left = 0;
        if (!rest_phase(c, fq0, tot, own_lo, off - own_lo, n_left)) return;
        if (n_left == 0) {
            // Every label is final (the rest phase's last barrier acquired
            // them).  The post phase gave every selected vertex outside the
            // post-time active set (`snap`) a label >= 0, so only that set
            // is checked for -1, each block over its own word range.
            int64_t left = 0;
            for (int64_t w = wb + c.tid; w < we; w += kGBlock) {
                uint64_t m = a.snap[w];
                while (m) {
                    const int64_t v = w * 64 + __ffsll((unsigned long long)m) - 1;
                    left += a.lab[v] < 0;
                    m &= m - 1;
                }
            }
            left = block_sum(left, sm);
            if (c.tid == 0) {
                if (left) atomicAdd(reinterpret_cast<unsigned long long*>(&gs->unlabelled), (unsigned long long)left);
                if (c.b == 0) gs->unl_checked = 1;
            }
            if (a.lab2) write_labels<true>(c, wb, we, traversed, gmin);
        }
        if (stamp) gs->ts[5] = wall_clock64();
    }
    if (stamp) gs->bar_next = a.bar_base + c.nbar;
}

__global__ __launch_bounds__(kGBlock) void k_tail(const GiantArgs) {
    KernelArgs& a = kernel_args();
    __shared__ Smem sm;
    GiantState* gs = a.gs;
    if (gs->err.v != 0) return;  // k_giant failed; the host reports its error
    const int64_t n = gs->n_final;
    int cur = (int)gs->final_sel;
    if (n == 0) return;
    Ctx c{(int)gridDim.x, (int)blockIdx.x, (int)threadIdx.x, lane_id(), wave_id(), sm, 0, 0, 0, 0, 0};
    const bool lead = c.b == 0 && c.tid == 0;
    int64_t rounds = 0, sccs = 0;
    if (a.wcc_mode == 1) {  // P12 by label propagation: parent = smallest id of the WCC
        if (!lp_wcc(c, cur ? a.fq : a.fq_alt, n, rounds)) return;
        if (lead) {
            gs->wcc_done = 1;
            gs->tail_rounds = rounds;
        }
    } else if (a.wcc_mode == 2) {  // P12-P14 replaced: nothing is left for the mice phase
        if (!colour_scc(c, cur, n, (int)gs->sweeps, rounds, sccs)) return;
        if (lead) {
            gs->n_final = 0;
            gs->final_sel = cur;
            gs->tail_rounds = rounds;
            gs->tail_sccs = sccs;
            a.fq_n_ctl[cur] = 0;
        }
    }
    if (lead) {
        gs->bar_next = a.bar_base + c.nbar;
        gs->ts[5] = wall_clock64();
    }
}

// first[v] = the first entry of v's list (-1 if empty): the bottom-up sweep's
// first probe reads 4 dense bytes instead of a cache line of the list.
__global__ void k_first(const int32_t* __restrict__ beg, const int32_t* __restrict__ adj, int32_t V, int32_t* first) {
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += (int64_t)gridDim.x * blockDim.x)
        first[v] = beg[v + 1] > beg[v] ? adj[beg[v]] : -1;
}

constexpr size_t kStageBytes = (size_t)kW * kPairCap * 8;  // dynamic LDS of k_giant and k_tail

int giant_max_blocks_per_cu() {
    for (const void* k : {reinterpret_cast<const void*>(k_giant), reinterpret_cast<const void*>(k_tail)})
        if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kStageBytes) != hipSuccess)
            return 0;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_giant, kGBlock, kStageBytes) != hipSuccess) return 0;
    return nb;
}

int64_t giant_bu_mult(int grid) {
    const int64_t t = (int64_t)grid * kW;
    int64_t m = 2654435761ll % t;  // Knuth's multiplicative hash constant, then the next value coprime to t
    for (;; ++m) {
        int64_t x = m, y = t;
        while (y) {
            const int64_t r = x % y;
            x = y;
            y = r;
        }
        if (x == 1) return m;
    }
}

hipError_t launch_giant(const GiantArgs& a, Ctl* ctl, int grid, hipStream_t s, hipEvent_t before) {
    static_assert(kGiantStateHead % 8 == 0 && sizeof(Ctl) % 8 == 0 && sizeof(GiantState) % 8 == 0, "state sizes");
    hipError_t e;
    if (before && (e = hipEventRecord(before, s)) != hipSuccess) return e;
    GiantArgs copy = a;
    copy.ctl = ctl;
    copy.state_words = (int32_t)((a.trace ? sizeof(GiantState) : kGiantStateHead) / 8);
    copy.ctl_words = (int32_t)(sizeof(Ctl) / 8);
    void* args[] = {&copy};
    return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_giant), dim3(grid), dim3(kGBlock), args,
                                      kStageBytes, s);
}

hipError_t launch_tail(const GiantArgs& a, int grid, hipStream_t s) {
    GiantArgs copy = a;
    void* args[] = {&copy};
    return hipLaunchCooperativeKernel(reinterpret_cast<const void*>(k_tail), dim3(grid), dim3(kGBlock), args,
                                      kStageBytes, s);
}

hipError_t launch_first(const int32_t* beg, const int32_t* adj, int32_t V, int32_t* first, int grid, hipStream_t s) {
    hipLaunchKernelGGL(k_first, dim3(grid), dim3(256), 0, s, beg, adj, V, first);
    return hipGetLastError();
}

}  // namespace ispan
