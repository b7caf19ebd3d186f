// gfx950 kernels of the iSpan SCC pipeline.
//
// Per-vertex state in HBM:
//   lab[V]   int32   -1 while unassigned, else the canonical SCC label
//   act[W]   uint64  bit v: v is still unassigned (W = ceil(V/64))
//   fvis[W]  uint64  bit v: reached by the forward traversal from the pivot
//   bvis[W]  uint64  bit v: reached by the backward traversal inside fvis
// The bitmaps are 2 MB each at V = 2^24, so the random probes of the
// traversals stay in L2/MALL while adjacency is streamed from HBM.
#include <algorithm>

#include "common.h"
#include "device_util.h"

namespace ispan {

using namespace dev;


// ------------------------------------------------------------------ reset

__global__ void k_reset_ctl(Ctl* ctl) {
    int32_t* p = reinterpret_cast<int32_t*>(ctl);
    for (int i = threadIdx.x; i < (int)(sizeof(Ctl) / 4); i += blockDim.x) p[i] = 0;
}

__global__ void k_fill_i32(int32_t* p, int32_t v, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// ---------------------------------------- P1-P3: trim-1-first, queue, pivot
// trim_1_first (src/trim_1_gfq.h:9-33) + generate_frontier_queue
// (src/trim_1_gfq.h:486-529) + pivot_selection_from_fq (src/scc_common.h:
// 92-150) in one sweep over the two offset arrays.  Each 4096-vertex tile
// compacts its survivors in ascending order with one global atomic; the
// pivot is the largest out*in, lowest id on ties, reduced by the last block.
__global__ __launch_bounds__(kBlock) void k_trim1_first(const int32_t* __restrict__ fwb, const int32_t* __restrict__ bwb,
                                                        int32_t V, int32_t* __restrict__ lab, uint64_t* act,
                                                        uint64_t* fvis, uint64_t* bvis, int32_t* __restrict__ fq,
                                                        int32_t* q0, Ctl* ctl, PivotPart* part, int wrap32) {
    constexpr int J = kTrimTile / kBlock;
    __shared__ int s_off[J * (kBlock / kWave)];
    __shared__ int64_t s_bp[kBlock / kWave];
    __shared__ int32_t s_bi[kBlock / kWave];
    __shared__ int s_last;
    const int tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    int64_t bestp = 0;
    int32_t besti = INT32_MAX;
    const int64_t ntiles = ((int64_t)V + kTrimTile - 1) / kTrimTile;
    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int64_t base = tile * kTrimTile;
        uint64_t masks[J];
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int64_t v = base + j * kBlock + tid;
            bool surv = false;
            if (v < V) {
                const int32_t od = fwb[v + 1] - fwb[v];
                const int32_t id = bwb[v + 1] - bwb[v];
                surv = od > 0 && id > 0;
                lab[v] = surv ? -1 : (int32_t)v;
                if (surv) {
                    int64_t p = wrap32 ? (int64_t)(int32_t)((uint32_t)od * (uint32_t)id) : (int64_t)od * id;
                    if (p > 0 && pivot_better(p, (int32_t)v, bestp, besti)) {
                        bestp = p;
                        besti = (int32_t)v;
                    }
                }
            }
            const uint64_t m = __ballot(surv);
            masks[j] = m;
            const int64_t first = base + j * kBlock + wave * kWave;
            if (lane == 0) {
                if (first < V) {
                    act[first >> 6] = m;
                    fvis[first >> 6] = 0;
                    bvis[first >> 6] = 0;
                }
                s_off[j * (kBlock / kWave) + wave] = __popcll(m);
            }
        }
        __syncthreads();
        if (wave == 0) {
            const int c = s_off[lane];
            const int incl = wave_incl_scan(c);
            const int total = lane_get(incl, kWave - 1);
            int b = 0;
            if (lane == 0 && total) b = atomicAdd(&ctl->fq_n[0], total);
            b = lane_get(b, 0);
            s_off[lane] = b + incl - c;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < J; ++j) {
            if ((masks[j] >> lane) & 1ull)
                fq[s_off[j * (kBlock / kWave) + wave] + __popcll(masks[j] & lanemask_lt())] =
                    (int32_t)(base + j * kBlock + tid);
        }
        __syncthreads();
    }
    // block reduction of the pivot candidate
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
        int64_t op = __shfl_xor(bestp, d, kWave);
        int32_t oi = __shfl_xor(besti, d, kWave);
        if (pivot_better(op, oi, bestp, besti)) {
            bestp = op;
            besti = oi;
        }
    }
    if (lane == 0) {
        s_bp[wave] = bestp;
        s_bi[wave] = besti;
    }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < kBlock / kWave; ++w)
            if (pivot_better(s_bp[w], s_bi[w], bestp, besti)) {
                bestp = s_bp[w];
                besti = s_bi[w];
            }
        part[blockIdx.x].prod = bestp;
        part[blockIdx.x].id = besti;
        __threadfence();
        const unsigned prev = atomicAdd(&ctl->done_blocks, 1u);
        s_last = prev == gridDim.x - 1;
    }
    __syncthreads();
    if (!s_last) return;
    // last block: global pivot and traversal start state
    __threadfence();
    bestp = 0;
    besti = INT32_MAX;
    for (int b = tid; b < (int)gridDim.x; b += kBlock) {
        const int64_t p = load_agent(&part[b].prod);
        const int32_t i = load_agent(&part[b].id);
        if (pivot_better(p, i, bestp, besti)) {
            bestp = p;
            besti = i;
        }
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
        int64_t op = __shfl_xor(bestp, d, kWave);
        int32_t oi = __shfl_xor(besti, d, kWave);
        if (pivot_better(op, oi, bestp, besti)) {
            bestp = op;
            besti = oi;
        }
    }
    if (lane == 0) {
        s_bp[wave] = bestp;
        s_bi[wave] = besti;
    }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < kBlock / kWave; ++w)
            if (pivot_better(s_bp[w], s_bi[w], bestp, besti)) {
                bestp = s_bp[w];
                besti = s_bi[w];
            }
        const int32_t root = (bestp > 0 && besti < V) ? besti : -1;
        ctl->root = root;
        ctl->done_blocks = 0;
        ctl->giant_min = root;
        ctl->q_n[0] = root >= 0 ? 1 : 0;
        ctl->q_n[1] = 0;
        ctl->hub_n[0] = ctl->hub_n[1] = 0;
        ctl->levels = 0;
        if (root >= 0) {
            atomicOr(reinterpret_cast<unsigned long long*>(fvis + (root >> 6)), 1ull << (root & 63));
            q0[0] = root;
        }
    }
}

// ------------------------------------------------------- traversal levels
// Top-down level (fw_bfs_fq_queue / bw_bfs_fq_queue sync and async top-down
// branches, src/fw_bw.h:453-478,506-544 and :992-1026,1066-1108).  A block
// stages 256 frontier vertices, scans their degrees in LDS and walks the
// block's combined edge range with all 256 threads (coalesced adjacency
// reads).  Vertices of degree >= kHubDeg are split into kHubChunk-edge work
// items for k_td_hub, which every level runs last.
template <bool BW>
__global__ __launch_bounds__(kBlock) void k_td(const int32_t* __restrict__ beg, const int32_t* __restrict__ adj,
                                               const uint64_t* __restrict__ allow, uint64_t* vis,
                                               const int32_t* __restrict__ qin, int32_t* qout, HubItem* hub_out,
                                               Ctl* ctl, int par) {
    __shared__ int32_t s_off[kBlock];
    __shared__ int32_t s_start[kBlock];
    __shared__ int s_tmp[kBlock / kWave];
    __shared__ int32_t s_wbuf[kBlock / kWave][kWaveBuf];
    const int tid = threadIdx.x;
    const int n = ctl->q_n[par];
    int32_t* qn_out = &ctl->q_n[par ^ 1];
    int32_t* hub_n = &ctl->hub_n[par];
    WaveQueue wq{s_wbuf[wave_id()], 0};
    int gmin = INT32_MAX;
    int64_t edges = 0, found = 0;
    for (int64_t tb = (int64_t)blockIdx.x * kBlock; tb < n; tb += (int64_t)gridDim.x * kBlock) {
        const int64_t i = tb + tid;
        int32_t start = 0, deg = 0;
        if (i < n) {
            const int32_t v = qin[i];
            start = beg[v];
            deg = beg[v + 1] - start;
            if (deg >= kHubDeg) {
                const int nch = (deg + kHubChunk - 1) / kHubChunk;
                const int h = atomicAdd(hub_n, nch);
                for (int c = 0; c < nch; ++c) hub_out[h + c] = HubItem{v, start + c * kHubChunk};
                deg = 0;
            }
        }
        int excl, total;
        block_excl_scan(deg, excl, total, s_tmp);
        s_off[tid] = excl;
        s_start[tid] = start;
        if (tid == 0) edges += total;
        __syncthreads();
        for (int eb = 0; eb < total; eb += kBlock) {
            const int e = eb + tid;
            bool claim = false;
            int32_t w = 0;
            if (e < total) {
                int lo = 0, hi = kBlock - 1;  // last j with s_off[j] <= e
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (s_off[mid] <= e) lo = mid;
                    else hi = mid - 1;
                }
                w = adj[s_start[lo] + (e - s_off[lo])];
                claim = try_claim(w, allow, vis);
            }
            wq_push(wq, claim, w, qout, qn_out);
            found += claim;
            if (BW && claim) gmin = min(gmin, w);
        }
        __syncthreads();
    }
    wq_flush(wq, qout, qn_out);
    wave_add64(&ctl->work_edges[0], edges);
    wave_add64(&ctl->work_found[0], found);
    if (BW) {
        gmin = wave_min(gmin);
        if (lane_id() == 0 && gmin != INT32_MAX) atomicMin(&ctl->giant_min, gmin);
    }
}

// Hub work items of this level; also the level's bookkeeping: the input
// count q_n[par] is consumed (k_td has completed) and reset, and the next
// level's hub counter is cleared.
template <bool BW>
__global__ __launch_bounds__(kBlock) void k_td_hub(const int32_t* __restrict__ beg, const int32_t* __restrict__ adj,
                                                   const uint64_t* __restrict__ allow, uint64_t* vis,
                                                   const HubItem* __restrict__ hub_in, int32_t* qout, Ctl* ctl,
                                                   int par) {
    __shared__ int32_t s_wbuf[kBlock / kWave][kWaveBuf];
    const int tid = threadIdx.x;
    if (blockIdx.x == 0 && tid == 0) {
        if (ctl->q_n[par] > 0) ctl->levels += 1;
        ctl->q_n[par] = 0;
        ctl->hub_n[par ^ 1] = 0;
    }
    const int nh = ctl->hub_n[par];
    int32_t* qn_out = &ctl->q_n[par ^ 1];
    WaveQueue wq{s_wbuf[wave_id()], 0};
    int gmin = INT32_MAX;
    int64_t edges = 0, found = 0;
    for (int h = blockIdx.x; h < nh; h += gridDim.x) {
        const HubItem it = hub_in[h];
        const int32_t end = min(it.start + kHubChunk, beg[it.v + 1]);
        if (tid == 0) edges += end - it.start;
        for (int32_t eb = it.start; eb < end; eb += kBlock) {
            const int32_t e = eb + tid;
            bool claim = false;
            int32_t w = 0;
            if (e < end) {
                w = adj[e];
                claim = try_claim(w, allow, vis);
            }
            wq_push(wq, claim, w, qout, qn_out);
            found += claim;
            if (BW && claim) gmin = min(gmin, w);
        }
    }
    wq_flush(wq, qout, qn_out);
    wave_add64(&ctl->work_edges[1], edges);
    wave_add64(&ctl->work_found[1], found);
    if (BW) {
        gmin = wave_min(gmin);
        if (lane_id() == 0 && gmin != INT32_MAX) atomicMin(&ctl->giant_min, gmin);
    }
}

// Bottom-up sweep (the Rsync branches, src/fw_bw.h:480-505 and :1040-1064).
// Candidates come from the bitmaps (allow & ~vis), 2048 vertices per tile
// compacted into LDS; each candidate scans its reverse-direction edges and
// stops at the first visited neighbour.  Bits set during the sweep are seen
// by later checks (asynchronous, as in the reference).  Every vertex found
// is also pushed, so a switch to top-down needs no gather pass.
template <bool BW>
__global__ __launch_bounds__(kBlock) void k_bu(const int32_t* __restrict__ beg, const int32_t* __restrict__ adj,
                                               const uint64_t* __restrict__ allow, uint64_t* vis, int32_t* qout,
                                               Ctl* ctl, int par, int64_t nwords) {
    __shared__ int32_t s_list[kBuTileWords * 64];
    __shared__ int s_n;
    __shared__ int32_t s_wbuf[kBlock / kWave][kWaveBuf];
    const int tid = threadIdx.x, lane = lane_id();
    if (blockIdx.x == 0 && tid == 0) {
        ctl->levels += 1;
        ctl->q_n[par] = 0;
        ctl->hub_n[par ^ 1] = 0;
    }
    int32_t* qn_out = &ctl->q_n[par ^ 1];
    WaveQueue wq{s_wbuf[wave_id()], 0};
    int gmin = INT32_MAX;
    int scanned = 0, nfound = 0;
    auto visited = [vis](int32_t u, int32_t) { return bit_of(vis, u); };
    for (int64_t t = blockIdx.x; t * kBuTileWords < nwords; t += gridDim.x) {
        if (wave_id() == 0) {
            const int64_t wi = t * kBuTileWords + lane;
            uint64_t m = 0;
            if (lane < kBuTileWords && wi < nwords) m = allow[wi] & ~vis[wi];
            const int c = __popcll(m);
            const int incl = wave_incl_scan(c);
            int o = incl - c;
            while (m) {
                const int b = __ffsll((unsigned long long)m) - 1;
                s_list[o++] = (int32_t)((wi << 6) + b);
                m &= m - 1;
            }
            if (lane == kWave - 1) s_n = incl;
        }
        __syncthreads();
        const int n = s_n;
        for (int kb = 0; kb < n; kb += kBlock) {
            const int k = kb + tid;
            const bool have = k < n;
            const int32_t v = have ? s_list[k] : 0;
            const int32_t p = have ? beg[v] : 0;
            const int32_t end = have ? beg[v + 1] : 0;
            const bool found = wave_any_edge(have, p, end, v, adj, visited, scanned);
            if (found)
                atomicOr(reinterpret_cast<unsigned long long*>(vis + (v >> 6)), 1ull << (v & 63));
            wq_push(wq, found, v, qout, qn_out);
            nfound += found;
            if (BW && found) gmin = min(gmin, v);
        }
        __syncthreads();
    }
    wq_flush(wq, qout, qn_out);
    wave_add64(&ctl->work_edges[2], scanned);
    wave_add64(&ctl->work_found[2], nfound);
    if (BW) {
        gmin = wave_min(gmin);
        if (lane_id() == 0 && gmin != INT32_MAX) atomicMin(&ctl->giant_min, gmin);
    }
}

// Backward traversal start: the pivot (src/fw_bw.h:972-976).
__global__ void k_bw_init(uint64_t* bvis, int32_t* q0, Ctl* ctl) {
    const int32_t root = ctl->root;
    ctl->q_n[0] = root >= 0 ? 1 : 0;
    ctl->q_n[1] = 0;
    ctl->hub_n[0] = ctl->hub_n[1] = 0;
    ctl->levels = 0;
    if (root >= 0) {
        bvis[root >> 6] |= 1ull << (root & 63);
        q0[0] = root;
        ctl->giant_min = root;
    }
}

__global__ __launch_bounds__(kBlock) void k_popcount(const uint64_t* __restrict__ bm, int64_t nwords, int64_t* out) {
    int c = 0;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < nwords; i += (int64_t)gridDim.x * kBlock)
        c += __popcll(bm[i]);
    c = wave_sum(c);
    if (lane_id() == 0 && c) atomicAdd(reinterpret_cast<unsigned long long*>(out), (unsigned long long)c);
}

// ------------------------------------------------------------ after giant
// Giant members get the giant's smallest id; act loses them; the active
// queue fq is rebuilt from the bitmap (ascending within each wave).
__global__ __launch_bounds__(kBlock) void k_post_giant(int32_t V, int32_t* __restrict__ lab, uint64_t* act,
                                                       const uint64_t* __restrict__ bvis, int32_t* fq, Ctl* ctl) {
    __shared__ int32_t s_wbuf[kBlock / kWave][kWaveBuf];
    const int32_t gmin = ctl->giant_min;
    WaveQueue wq{s_wbuf[wave_id()], 0};
    int32_t* cnt = &ctl->fq_n[1];
    for (int64_t tb = (int64_t)blockIdx.x * kBlock; tb < V; tb += (int64_t)gridDim.x * kBlock) {
        const int64_t v = tb + threadIdx.x;
        const bool in = v < V;
        uint64_t g = 0, a = 0;
        if (in) {
            g = bvis[v >> 6];
            a = act[v >> 6];
        }
        const bool giant = in && ((g >> (v & 63)) & 1ull);
        const bool keep = in && ((a >> (v & 63)) & 1ull) && !giant;
        if (giant) lab[v] = gmin;
        const uint64_t mk = __ballot(keep);
        if (lane_id() == 0 && in && g) act[v >> 6] = mk;
        wq_push(wq, keep, (int32_t)v, fq, cnt);
    }
    wq_flush(wq, fq, cnt);
}

// ---------------------------------------------------------------- trim-1
// trim_1_from_fq_gfq (src/trim_1_gfq.h:365-458): an active vertex with no
// active non-self out-neighbour or no active non-self in-neighbour is a
// singleton SCC.  act is updated in place, so later checks in the same sweep
// see it; survivors are compacted into fq[sel^1].
__global__ void k_prep_sweep(Ctl* ctl, int sel) {
    ctl->fq_n[sel ^ 1] = 0;
    ctl->trimmed = 0;
}

__global__ __launch_bounds__(kBlock) void k_trim1(const int32_t* __restrict__ fwb, const int32_t* __restrict__ fwa,
                                                  const int32_t* __restrict__ bwb, const int32_t* __restrict__ bwa,
                                                  int32_t* __restrict__ lab, uint64_t* act,
                                                  const int32_t* __restrict__ fq_in, int32_t* fq_out, Ctl* ctl,
                                                  int sel) {
    __shared__ int32_t s_wbuf[kBlock / kWave][kWaveBuf];
    const int n = ctl->fq_n[sel];
    int32_t* cnt = &ctl->fq_n[sel ^ 1];
    WaveQueue wq{s_wbuf[wave_id()], 0};
    int trimmed = 0, scanned = 0;
    auto live = [act](int32_t w, int32_t self) { return w != self && bit_of(act, w); };
    for (int64_t tb = (int64_t)blockIdx.x * kBlock; tb < n; tb += (int64_t)gridDim.x * kBlock) {
        const int64_t i = tb + threadIdx.x;
        int32_t v = 0;
        bool alive = false;
        if (i < n) {
            v = fq_in[i];
            alive = bit_of(act, v);
        }
        const bool out = wave_any_edge(alive, alive ? fwb[v] : 0, alive ? fwb[v + 1] : 0, v, fwa, live, scanned);
        const bool in =
            wave_any_edge(alive && out, alive ? bwb[v] : 0, alive ? bwb[v + 1] : 0, v, bwa, live, scanned);
        const bool trim = alive && !(out && in);
        if (trim) {
            lab[v] = v;
            atomicAnd(reinterpret_cast<unsigned long long*>(act + (v >> 6)), ~(1ull << (v & 63)));
            ++trimmed;
        }
        wq_push(wq, alive && !trim, v, fq_out, cnt);
    }
    wq_flush(wq, fq_out, cnt);
    trimmed = wave_sum(trimmed);
    if (lane_id() == 0 && trimmed) atomicAdd(&ctl->trimmed, trimmed);
}

// ---------------------------------------------------------- size-2/3 trims
// trim_2_from_fq (src/trim_2_3.h:146-283), trim_3_1_from_fq (:482-677) and
// trim_3_2_from_fq (:881-1080), checked against act as it stands when the
// kernel starts: detections only write lab (and the pattern size into
// stamp); act is cleared afterwards by k_pattern_commit.  With a fixed
// active set every detected group is an SCC of the active subgraph, so two
// detections of one vertex always agree on its label.

__global__ __launch_bounds__(kBlock) void k_pattern(const int32_t* __restrict__ fwb, const int32_t* __restrict__ fwa,
                                                    const int32_t* __restrict__ bwb, const int32_t* __restrict__ bwa,
                                                    int32_t* lab, int32_t* stamp, const uint64_t* __restrict__ act,
                                                    const int32_t* __restrict__ fq, const Ctl* ctl, int sel) {
    const int n = ctl->fq_n[sel];
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t a = fq[i];
        if (bit_of(act, a)) pattern_check(fwb, fwa, bwb, bwa, lab, stamp, act, a);
    }
}

__global__ __launch_bounds__(kBlock) void k_pattern_commit(const int32_t* __restrict__ lab, uint64_t* act,
                                                           const int32_t* __restrict__ stamp,
                                                           const int32_t* __restrict__ fq, Ctl* ctl, int sel) {
    const int n = ctl->fq_n[sel];
    int c2 = 0, c3 = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t v = fq[i];
        if (lab[v] >= 0 && bit_of(act, v)) {
            atomicAnd(reinterpret_cast<unsigned long long*>(act + (v >> 6)), ~(1ull << (v & 63)));
            if (stamp[v] == 2) ++c2;
            else ++c3;
        }
    }
    c2 = wave_sum(c2);
    c3 = wave_sum(c3);
    if (lane_id() == 0) {
        if (c2) atomicAdd(&ctl->pattern2, c2);
        if (c3) atomicAdd(&ctl->pattern3, c3);
    }
}

// ------------------------------------------------------------------- WCC
// Weakly connected components of the active subgraph (the role of
// coloring_wcc, src/color_propagation.h:468-593, and openmp_wcc's CAS union,
// src/openmp_wcc.hpp:86-114).  Union-find: each active edge links the larger
// root under the smaller one with a CAS, then every vertex jumps to its
// root, so parent[v] = smallest id of v's WCC.  Out-edges of active vertices
// cover every active edge once.
__global__ __launch_bounds__(kBlock) void k_uf_init(const int32_t* __restrict__ fq, int32_t* parent, const Ctl* ctl,
                                                    int sel) {
    const int n = ctl->fq_n[sel];
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        parent[fq[i]] = fq[i];
}

__global__ __launch_bounds__(kBlock) void k_uf_hook(const int32_t* __restrict__ fwb, const int32_t* __restrict__ fwa,
                                                    const uint64_t* __restrict__ act, const int32_t* __restrict__ fq,
                                                    int32_t* parent, const Ctl* ctl, int sel) {
    const int n = ctl->fq_n[sel];
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t v = fq[i];
        for (int32_t k = fwb[v]; k < fwb[v + 1]; ++k) {
            const int32_t w = fwa[k];
            if (w == v || !bit_of(act, w)) continue;
            int32_t a = v, b = w;
            while (true) {
                a = uf_root(parent, a);
                b = uf_root(parent, b);
                if (a == b) break;
                if (a < b) {
                    const int32_t t = a;
                    a = b;
                    b = t;
                }
                if (atomicCAS(&parent[a], a, b) == a) break;
            }
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_uf_compress(const int32_t* __restrict__ fq, int32_t* parent,
                                                        const Ctl* ctl, int sel) {
    const int n = ctl->fq_n[sel];
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t v = fq[i];
        parent[v] = uf_find(parent, v);
    }
}

// Label propagation variant (coloring_wcc's scheme with the smallest id):
// color[v] = min over active in/out neighbours, then pointer jumping, until
// a sweep changes nothing.
__global__ __launch_bounds__(kBlock) void k_lp_sweep(const int32_t* __restrict__ fwb, const int32_t* __restrict__ fwa,
                                                     const int32_t* __restrict__ bwb, const int32_t* __restrict__ bwa,
                                                     const uint64_t* __restrict__ act, const int32_t* __restrict__ fq,
                                                     int32_t* color, Ctl* ctl, int sel) {
    const int n = ctl->fq_n[sel];
    int changed = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t v = fq[i];
        int32_t c = load_agent(&color[v]);
        const int32_t c0 = c;
        for (int dir = 0; dir < 2; ++dir) {
            const int32_t* beg = dir == 0 ? bwb : fwb;
            const int32_t* adj = dir == 0 ? bwa : fwa;
            for (int32_t k = beg[v]; k < beg[v + 1]; ++k) {
                const int32_t w = adj[k];
                if (w == v || !bit_of(act, w)) continue;
                c = min(c, load_agent(&color[w]));
            }
        }
        if (c < c0) {
            atomicMin(&color[v], c);
            changed = 1;
        }
    }
    if (__ballot(changed) && lane_id() == 0) atomicOr(&ctl->changed, 1);
}

__global__ __launch_bounds__(kBlock) void k_lp_jump(const int32_t* __restrict__ fq, int32_t* color, const Ctl* ctl,
                                                    int sel) {
    const int n = ctl->fq_n[sel];
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t v = fq[i];
        int32_t r = load_agent(&color[v]);
        for (int hop = 0; hop < 100; ++hop) {
            const int32_t nr = load_agent(&color[r]);
            if (nr == r) break;
            r = nr;
        }
        atomicMin(&color[v], r);
    }
}

__global__ void k_clear_changed(Ctl* ctl) { ctl->changed = 0; }

// ------------------------------------------------------------------ mice
// init_fw_sa + mice_fw_bw (src/fw_bw.h:1548-1691) regrouped: the members of
// each WCC are brought together (k_wcc_*), and one wave owns a WCC.  Grouping
// is a counting sort by WCC root: a member's place in its WCC is its count on
// the root's counter, in no particular order.

// The roots' counters cleared.
__global__ __launch_bounds__(kBlock) void k_wcc_reset(const int32_t* __restrict__ fq, int32_t n,
                                                      const int32_t* __restrict__ wcc, int32_t* cnt, Ctl* ctl) {
    if (blockIdx.x == 0 && threadIdx.x == 0) ctl->unlabelled = 0;  // counted again after the mice
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t v = fq[i];
        if (wcc[v] == v) cnt[v] = 0;
    }
}

// slot[v] = v's place in its WCC; cnt[root] = the WCC's size.  The queue is in
// ascending id order for the most part, so lanes of a wave often share a
// root: up to kSlotRounds roots are counted once per wave.
constexpr int kSlotRounds = 4;
__global__ __launch_bounds__(kBlock) void k_wcc_slots(const int32_t* __restrict__ fq, int32_t n,
                                                      const int32_t* __restrict__ wcc, int32_t* cnt, int32_t* slot,
                                                      int32_t* stamp) {
    const int lane = lane_id();
    const int64_t waves = (int64_t)gridDim.x * (kBlock / kWave);
    for (int64_t base = ((int64_t)blockIdx.x * (kBlock / kWave) + wave_id()) * kWave; base < n; base += waves * kWave) {
        const int64_t i = base + lane;
        const int32_t v = i < n ? fq[i] : 0;
        const int32_t r = i < n ? wcc[v] : -1;
        bool todo = i < n;
        int32_t at = 0;
        for (int k = 0; k < kSlotRounds; ++k) {
            const uint64_t m = __ballot(todo);
            if (!m) break;
            const int lead = __ffsll((unsigned long long)m) - 1;
            const int32_t L = lane_get(r, lead);
            const uint64_t same = __ballot(todo && r == L);
            int32_t b = 0;
            if (lane == lead) b = atomicAdd(&cnt[L], __popcll(same));
            b = lane_get(b, lead);
            if (todo && r == L) {
                at = b + __popcll(same & lanemask_lt());
                todo = false;
            }
        }
        if (todo) at = atomicAdd(&cnt[r], 1);
        if (i < n) {
            slot[v] = at;
            stamp[v] = -1;
        }
    }
}

// Every WCC's range of the member array and its entry in the list of WCCs; the
// number of WCCs and the largest.  A block takes one piece of the queue, adds
// up its WCCs first and reserves for all of them with one atomic per counter
// (one per 256 vertices took 58 us for 318,000: 11 ns each on one address).
constexpr int kRangeBlocks = 256;
__global__ __launch_bounds__(kBlock) void k_wcc_ranges(const int32_t* __restrict__ fq, int32_t n,
                                                       const int32_t* __restrict__ wcc, const int32_t* __restrict__ cnt,
                                                       int32_t* first, int32_t* roots, Ctl* ctl) {
    constexpr int NW = kBlock / kWave;
    __shared__ int s_tmp[NW];
    __shared__ int s_part[3][NW];
    __shared__ int s_at[2];
    const int64_t per = (((int64_t)n + gridDim.x - 1) / gridDim.x + kBlock - 1) / kBlock * kBlock;
    const int64_t lo = min((int64_t)blockIdx.x * per, (int64_t)n), hi = min(lo + per, (int64_t)n);
    int members = 0, found = 0, largest = 0;
    for (int64_t i = lo + threadIdx.x; i < hi; i += kBlock) {
        const int32_t v = fq[i];
        if (wcc[v] != v) continue;
        members += cnt[v];
        largest = max(largest, cnt[v]);
        ++found;
    }
    members = wave_sum(members);
    found = wave_sum(found);
    largest = -wave_min(-largest);
    if (lane_id() == 0) {
        s_part[0][wave_id()] = members;
        s_part[1][wave_id()] = found;
        s_part[2][wave_id()] = largest;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int m = 0, f = 0, l = 0;
        for (int w = 0; w < NW; ++w) {
            m += s_part[0][w];
            f += s_part[1][w];
            l = max(l, s_part[2][w]);
        }
        if (f) {
            s_at[0] = atomicAdd(&ctl->wcc_members, m);
            s_at[1] = atomicAdd(&ctl->n_wcc, f);
            atomicMax(&ctl->max_wcc, l);
        }
    }
    __syncthreads();
    int at_m = s_at[0], at_f = s_at[1];  // read only where the block found a WCC
    for (int64_t base = lo; base < hi; base += kBlock) {
        const int64_t i = base + threadIdx.x;
        const int32_t v = i < hi ? fq[i] : 0;
        const bool root = i < hi && wcc[v] == v;
        int m, f, all_m, all_f;
        block_excl_scan(root ? cnt[v] : 0, m, all_m, s_tmp);
        block_excl_scan(root ? 1 : 0, f, all_f, s_tmp);
        if (root) {
            first[v] = at_m + m;
            roots[at_f + f] = v;
        }
        at_m += all_m;
        at_f += all_f;
    }
}

__global__ __launch_bounds__(kBlock) void k_wcc_members(const int32_t* __restrict__ fq, int32_t n,
                                                        const int32_t* __restrict__ wcc,
                                                        const int32_t* __restrict__ first,
                                                        const int32_t* __restrict__ slot, int32_t* member) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t v = fq[i];
        member[first[wcc[v]] + slot[v]] = v;
    }
}

// SCCs of a WCC of n <= 64 * W vertices by one wave, from the transitive
// closure of its out-edges: lane l holds the rows of vertices l, l + 64, ..,
// W words each, in registers.  Active neighbours of a member are members
// (an edge joins their WCCs), and members are unlabelled until the end here,
// so an unlabelled neighbour's slot is its column.  Warshall's step k ORs row
// k into the rows that have bit k: n steps of a few instructions, however long
// the paths are, where a search per SCC costs a round trip per level (WCCs of
// 28 vertices in 8 groups: 526 -> 25 us for 12,500 of them).
constexpr int kLongList = 64;  // a longer list is scanned by the whole wave
template <int W>
__device__ __forceinline__ void closure_sccs(const int32_t* __restrict__ fwb, const int32_t* __restrict__ fwa,
                                             int32_t* lab, const int32_t* __restrict__ slot,
                                             const int32_t* __restrict__ member, int32_t n, uint64_t* s_row) {
    const int lane = lane_id();
    int32_t id[W];
    uint64_t R[W][W];
#pragma unroll
    for (int a = 0; a < W; ++a) {
        const int32_t i = a * kWave + lane;
        id[a] = i < n ? member[i] : -1;
#pragma unroll
        for (int b = 0; b < W; ++b) R[a][b] = 0;
        const int32_t p = i < n ? fwb[id[a]] : 0, e = i < n ? fwb[id[a] + 1] : 0;
        if (e - p <= kLongList) {
            for (int32_t k = p; k < e; ++k) {
                const int32_t w = fwa[k];
                if (load_agent(&lab[w]) != -1) continue;
                const int32_t j = slot[w];
#pragma unroll
                for (int b = 0; b < W; ++b)
                    if (W == 1 || (j >> 6) == b) R[a][b] |= 1ull << (j & 63);
            }
        }
        uint64_t pend = __ballot(e - p > kLongList);
        while (pend) {
            const int l = __ffsll((unsigned long long)pend) - 1;
            pend &= pend - 1;
            const int32_t p0 = lane_get(p, l), e0 = lane_get(e, l);
            if (lane < W) s_row[lane] = 0;
            wave_sync();
            for (int32_t k = p0 + lane; k < e0; k += kWave) {
                const int32_t w = fwa[k];
                if (load_agent(&lab[w]) != -1) continue;
                const int32_t j = slot[w];
                atomicOr(reinterpret_cast<unsigned long long*>(&s_row[j >> 6]), 1ull << (j & 63));
            }
            wave_sync();
            if (lane == l) {
#pragma unroll
                for (int b = 0; b < W; ++b) R[a][b] = s_row[b];
            }
            wave_sync();
        }
    }
#pragma unroll
    for (int c = 0; c < W; ++c) {
        const int m = min(kWave, n - c * kWave);
        for (int k = 0; k < m; ++k) {
            uint64_t row[W];
#pragma unroll
            for (int b = 0; b < W; ++b) row[b] = lane_get(R[c][b], k);
#pragma unroll
            for (int a = 0; a < W; ++a) {
                const uint64_t take = 0 - ((R[a][c] >> k) & 1ull);
#pragma unroll
                for (int b = 0; b < W; ++b) R[a][b] |= row[b] & take;
            }
        }
    }
    // a vertex's SCC: itself and the members it reaches and that reach it;
    // the label is the smallest id of them
    int32_t mn[W];
#pragma unroll
    for (int a = 0; a < W; ++a) mn[a] = id[a];
#pragma unroll
    for (int c = 0; c < W; ++c) {
        const int m = min(kWave, n - c * kWave);
        for (int k = 0; k < m; ++k) {
            const int32_t idk = lane_get(id[c], k);
            uint64_t row[W];  // whom k reaches
#pragma unroll
            for (int b = 0; b < W; ++b) row[b] = lane_get(R[c][b], k);
#pragma unroll
            for (int a = 0; a < W; ++a)
                if (((R[a][c] >> k) & (row[a] >> lane)) & 1ull) mn[a] = min(mn[a], idk);
        }
    }
    // every lane has read the labels it needed: the closure used them all
#pragma unroll
    for (int a = 0; a < W; ++a)
        if (a * kWave + lane < n) st_agent(&lab[id[a]], mn[a]);
}

// Larger WCCs: the wave repeatedly takes an unlabelled member as pivot, runs a
// FW search (visit stamp = pivot) and a BW search inside the WCC, whose queue
// then holds the pivot's SCC, and labels that with its smallest id.
constexpr int kClosureMax = 256;  // largest WCC taken by its closure (4 words a row)
__global__ __launch_bounds__(kBlock) void k_mice(const int32_t* __restrict__ fwb, const int32_t* __restrict__ fwa,
                                                 const int32_t* __restrict__ bwb, const int32_t* __restrict__ bwa,
                                                 int32_t* lab, int32_t* stamp, const int32_t* __restrict__ roots,
                                                 const int32_t* __restrict__ cnt, const int32_t* __restrict__ first,
                                                 const int32_t* __restrict__ slot, const int32_t* __restrict__ member,
                                                 const Ctl* ctl, int32_t* qbuf, int32_t max_wcc) {
    __shared__ int s_tail[kBlock / kWave];
    __shared__ uint64_t s_rows[kBlock / kWave][kClosureMax / kWave];
    if (max_wcc > 0 && ctl->max_wcc > max_wcc) return;  // left to the caller's other method
    const int lane = lane_id(), wave = wave_id();
    const int nw = ctl->n_wcc;
    const int waves = gridDim.x * (kBlock / kWave);
    for (int idx = blockIdx.x * (kBlock / kWave) + wave; idx < nw; idx += waves) {
        const int32_t root = lane_get(roots[idx], 0);
        const int32_t s = lane_get(first[root], 0), n = lane_get(cnt[root], 0);
        if (n <= kClosureMax) {
            if (n <= kWave) closure_sccs<1>(fwb, fwa, lab, slot, member + s, n, s_rows[wave]);
            else if (n <= 2 * kWave) closure_sccs<2>(fwb, fwa, lab, slot, member + s, n, s_rows[wave]);
            else closure_sccs<4>(fwb, fwa, lab, slot, member + s, n, s_rows[wave]);
            continue;
        }
        const int32_t e = s + n;
        int32_t* q = qbuf + s;
        int32_t cursor = s;
        while (true) {
            // next pivot: the next member still unlabelled
            int32_t pj = -1;
            for (int32_t b = cursor; b < e; b += kWave) {
                const int32_t j = b + lane;
                const bool fr = j < e && load_agent(&lab[member[j]]) == -1;
                const uint64_t m = __ballot(fr);
                if (m) {
                    pj = b + __ffsll((unsigned long long)m) - 1;
                    break;
                }
            }
            if (pj < 0) break;
            cursor = pj + 1;
            const int32_t pv = member[pj];
            int32_t found = 0;
            for (int phase = 0; phase < 2; ++phase) {
                const int32_t* beg = phase == 0 ? fwb : bwb;
                const int32_t* adj = phase == 0 ? fwa : bwa;
                if (lane == 0) {
                    if (phase == 0) stamp[pv] = pv;
                    else lab[pv] = pv;
                    q[0] = pv;
                    s_tail[wave] = 1;
                }
                wave_sync();
                int32_t head = 0, tail = 1;
                while (head < tail) {
                    const int32_t lo = head, hi = tail;
                    head = hi;
                    for (int32_t b = lo; b < hi; b += kWave) {
                        const int32_t i = b + lane;
                        if (i < hi) {
                            const int32_t x = load_agent(&q[i]);
                            for (int32_t k = beg[x]; k < beg[x + 1]; ++k) {
                                const int32_t w = adj[k];
                                if (load_agent(&lab[w]) != -1) continue;
                                bool claim;
                                if (phase == 0)
                                    claim = load_agent(&stamp[w]) != pv && atomicExch(&stamp[w], pv) != pv;
                                else
                                    claim = load_agent(&stamp[w]) == pv && atomicCAS(&lab[w], -1, pv) == -1;
                                if (claim) q[atomicAdd(&s_tail[wave], 1)] = w;
                            }
                        }
                    }
                    wave_sync();
                    tail = s_tail[wave];
                    wave_sync();
                }
                found = tail;
            }
            int32_t mn = INT32_MAX;
            for (int32_t i = lane; i < found; i += kWave) mn = min(mn, load_agent(&q[i]));
            mn = wave_min(mn);
            if (mn != pv)
                for (int32_t i = lane; i < found; i += kWave) st_agent(&lab[load_agent(&q[i])], mn);
            wave_sync();
        }
    }
}

// ---------------------------------------------------------------- checks
// sel (optional): only the selected vertices count.
__global__ __launch_bounds__(kBlock) void k_count_unlabelled(const int32_t* __restrict__ lab, int32_t V,
                                                             const uint64_t* __restrict__ sel, Ctl* ctl) {
    int c = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < V; i += (int64_t)gridDim.x * blockDim.x)
        c += (!sel || ((sel[i >> 6] >> (i & 63)) & 1ull)) && lab[i] < 0;
    c = wave_sum(c);
    if (lane_id() == 0 && c) atomicAdd(&ctl->unlabelled, c);
}

// Work statistics of the last solve: edges incident to the FW set (out) and
// to the giant (in), and the SCC count.
__global__ __launch_bounds__(kBlock) void k_stats(const int32_t* __restrict__ fwb, const int32_t* __restrict__ bwb,
                                                  const int32_t* __restrict__ lab, const uint64_t* __restrict__ fvis,
                                                  const uint64_t* __restrict__ bvis, int32_t V, Ctl* ctl) {
    int64_t fe = 0, be = 0;
    int ns = 0;
    for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < V; v += (int64_t)gridDim.x * blockDim.x) {
        if (bit_of(fvis, (int32_t)v)) fe += fwb[v + 1] - fwb[v];
        if (bit_of(bvis, (int32_t)v)) be += bwb[v + 1] - bwb[v];
        ns += lab[v] == v;
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
        fe += __shfl_xor(fe, d, kWave);
        be += __shfl_xor(be, d, kWave);
    }
    ns = wave_sum(ns);
    if (lane_id() == 0) {
        if (fe) atomicAdd(reinterpret_cast<unsigned long long*>(&ctl->fw_edges), (unsigned long long)fe);
        if (be) atomicAdd(reinterpret_cast<unsigned long long*>(&ctl->bw_edges), (unsigned long long)be);
        if (ns) atomicAdd(reinterpret_cast<unsigned long long*>(&ctl->n_scc), (unsigned long long)ns);
    }
}

// Structural check of a CSR pair: beg[0] == 0, beg non-decreasing, beg[V] == E,
// every adjacency id in [0, V); and, where the caller has room for it, every
// list's first entry (-1 if empty), which the bottom-up sweep probes first.
// Half of the blocks take each direction.  Bound by the one read of the lists;
// a thread has kAhead loads in flight.  V 2 M, E 32 M: 62 us (272 MB, and the
// lines of the first entries again), where a pass a direction and two for the
// first entries took 99.
__global__ __launch_bounds__(kBlock) void k_check_csr(CsrPair P, int32_t V, int64_t E, Ctl* ctl) {
    constexpr int kAhead = 8;
    const int dir = blockIdx.x & 1;
    const int32_t* __restrict__ beg = P.beg[dir];
    const int32_t* __restrict__ adj = P.adj[dir];
    int32_t* first = P.first[dir];
    int bad = 0;
    const int64_t stride = (int64_t)(gridDim.x / 2) * kBlock;
    const int64_t t = (int64_t)(blockIdx.x / 2) * kBlock + threadIdx.x;
    if (t == 0) bad += beg[0] != 0 || (int64_t)beg[V] != E;
    for (int64_t kb = t; kb < E; kb += kAhead * stride) {
        int32_t x[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) x[u] = kb + u * stride < E ? adj[kb + u * stride] : 0;
#pragma unroll
        for (int u = 0; u < kAhead; ++u) bad += x[u] < 0 || x[u] >= V;
    }
    for (int64_t vb = t; vb < V; vb += kAhead * stride) {
        int32_t b[kAhead], e[kAhead], f[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int64_t v = min(vb + u * stride, (int64_t)V - 1);
            b[u] = beg[v];
            e[u] = beg[v + 1];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            bad += vb + u * stride < V && b[u] > e[u];
            // offsets are not known to be right yet: none is followed out of the lists
            const bool some = first && e[u] > b[u] && b[u] >= 0 && b[u] < E;
            f[u] = some ? adj[b[u]] : -1;
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (first && vb + u * stride < V) first[vb + u * stride] = f[u];
    }
    bad = wave_sum(bad);
    if (lane_id() == 0 && bad) atomicAdd(&ctl->bad_csr, bad);
}

// ---------------------------------------------------- SCC size histogram
// Extends get_scc_result (src/load_print.cpp:24-60), which tallies SCC
// sizes in a std::map but prints only count classes.
//
// Canonical labels: the vertex whose label is its own id is its SCC's
// smallest, so every size starts at 1 with a plain store there, and only the
// other vertices of an SCC are counted by atomics.
constexpr int kHistGrid = 512;  // blocks: each ends with one atomic per common address

// Four consecutive labels from v (16-byte load; entries past V are -1).
__device__ __forceinline__ int4 load4(const int32_t* __restrict__ p, int64_t v, int32_t V) {
    if (v + 3 < V) return *reinterpret_cast<const int4*>(p + v);
    return int4{v < V ? p[v] : -1, v + 1 < V ? p[v + 1] : -1, v + 2 < V ? p[v + 2] : -1, -1};
}

__global__ __launch_bounds__(kBlock) void k_size_roots(const int32_t* __restrict__ lab, int32_t V, int32_t* size,
                                                       int64_t* out) {
    if (blockIdx.x == 0 && threadIdx.x < kHistSlots) out[threadIdx.x] = 0;
    for (int64_t v = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * 4; v < V; v += (int64_t)gridDim.x * kBlock * 4) {
        const int4 l = load4(lab, v, V);
        const int4 r{l.x == v, l.y == v + 1, l.z == v + 2, l.w == v + 3};
        if (v + 3 < V) {
            *reinterpret_cast<int4*>(size + v) = r;
        } else {
            size[v] = r.x;
            if (v + 1 < V) size[v + 1] = r.y;
            if (v + 2 < V) size[v + 2] = r.z;
        }
    }
}

// size[lab[v]] += 1 for every vertex that is not its SCC's smallest.  Atomics
// on one address run one after the other over the whole chip (11 ns each), so
// the label of a large SCC must not cost one per wave step: each thread counts
// on while the label stays the same, and then adds to the block's table in
// LDS, which takes the first kSizeSlots labels or so that the block meets (the
// large ones are met early) and goes out at the end, one atomic an entry.
// The whole histogram call, 2 M vertices in one SCC, and in two, four, ten and
// a hundred with ids at random: 41, 47, 58, 64 and 96 us (a combined atomic
// per wave step: 389, 743, 1451, 6245 and 1833; without the table, only the
// block's most frequent label added up: 39, 7387, 8012, 6116 and 1675).
constexpr int kSizeSlots = 512;
constexpr int kSizeProbes = 4;
__global__ __launch_bounds__(kBlock) void k_scc_sizes(const int32_t* __restrict__ lab, int32_t V, int32_t* size) {
    __shared__ int32_t s_lab[kSizeSlots];
    __shared__ int s_cnt[kSizeSlots];
    for (int i = threadIdx.x; i < kSizeSlots; i += kBlock) {
        s_lab[i] = -1;
        s_cnt[i] = 0;
    }
    __syncthreads();
    auto add = [&](int32_t l, int n) {
        uint32_t at = (uint32_t)l * 2654435761u >> 23;  // Knuth's multiplicative hash: 9 bits
        for (int k = 0; k < kSizeProbes; ++k, at = (at + 1) & (kSizeSlots - 1)) {
            int32_t have = s_lab[at];
            if (have == -1) {
                have = atomicCAS(&s_lab[at], -1, l);
                if (have == -1) have = l;
            }
            if (have == l) {
                atomicAdd(&s_cnt[at], n);
                return;
            }
        }
        atomicAdd(&size[l], n);
    };
    int32_t cur = -1;  // this thread's current label and how often it met it
    int cnt = 0;
    auto meet = [&](int32_t l, int64_t v) {
        if (l < 0 || l == v) return;
        if (l != cur) {
            if (cnt) add(cur, cnt);
            cur = l;
            cnt = 0;
        }
        ++cnt;
    };
    for (int64_t v = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * 4; v < V; v += (int64_t)gridDim.x * kBlock * 4) {
        const int4 l = load4(lab, v, V);
        meet(l.x, v);
        meet(l.y, v + 1);
        meet(l.z, v + 2);
        meet(l.w, v + 3);
    }
    if (cnt) add(cur, cnt);
    __syncthreads();
    for (int i = threadIdx.x; i < kSizeSlots; i += kBlock)
        if (s_cnt[i]) atomicAdd(&size[s_lab[i]], s_cnt[i]);
}

// Log2 bins of the SCC sizes (bin k: sizes in [2^k, 2^(k+1))), per block in
// LDS, plus the largest size, the counts of sizes 1, 2, 3 and the SCC
// count: out[0..63] bins, out[64] largest, out[65..67] sizes 1-3, out[68]
// total.  Sizes up to 3, nearly all of them, are counted in registers (one
// LDS bin for all of a wave's lanes took 292 us at 2 M vertices).
__global__ __launch_bounds__(kBlock) void k_scc_hist(const int32_t* __restrict__ size, int32_t V, int64_t* out) {
    constexpr int NW = kBlock / kWave;
    __shared__ int s_bin[64];
    __shared__ int s_part[5][NW];
    if (threadIdx.x < 64) s_bin[threadIdx.x] = 0;
    __syncthreads();
    int largest = 0, c1 = 0, c2 = 0, c3 = 0, tot = 0;
    auto meet = [&](int c) {
        if (c <= 0) return;
        c1 += c == 1;
        c2 += c == 2;
        c3 += c == 3;
        ++tot;
        if (c > 3) atomicAdd(&s_bin[31 - __clz(c)], 1);
        largest = max(largest, c);
    };
    for (int64_t v = ((int64_t)blockIdx.x * kBlock + threadIdx.x) * 4; v < V; v += (int64_t)gridDim.x * kBlock * 4) {
        const int4 c = load4(size, v, V);
        meet(c.x);
        meet(c.y);
        meet(c.z);
        meet(c.w);
    }
    c1 = wave_sum(c1);
    c2 = wave_sum(c2);
    c3 = wave_sum(c3);
    tot = wave_sum(tot);
    largest = -wave_min(-largest);
    if (lane_id() == 0) {
        const int w = wave_id();
        s_part[0][w] = c1;
        s_part[1][w] = c2;
        s_part[2][w] = c3;
        s_part[3][w] = tot;
        s_part[4][w] = largest;
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        int x[5] = {0, 0, 0, 0, 0};
        for (int w = 0; w < NW; ++w) {
            for (int k = 0; k < 4; ++k) x[k] += s_part[k][w];
            x[4] = max(x[4], s_part[4][w]);
        }
        const int t = threadIdx.x;
        const int bin = s_bin[t] + (t == 0 ? x[0] : t == 1 ? x[1] + x[2] : 0);
        if (bin) atomicAdd(reinterpret_cast<unsigned long long*>(&out[t]), (unsigned long long)bin);
        const int y = t == 0 ? x[4] : t < 4 ? x[t - 1] : t == 4 ? x[3] : 0;  // out[64..68]
        if (t == 0 && y) atomicMax(reinterpret_cast<unsigned long long*>(&out[64]), (unsigned long long)y);
        else if (t > 0 && t < 5 && y) atomicAdd(reinterpret_cast<unsigned long long*>(&out[64 + t]), (unsigned long long)y);
    }
}

// ------------------------------------------------------------- launchers

#define LAUNCH(kern, grid, ...)                                  \
    do {                                                         \
        hipLaunchKernelGGL(kern, dim3(grid), dim3(kBlock), 0, s, __VA_ARGS__); \
        return hipGetLastError();                                \
    } while (0)

hipError_t launch_reset_ctl(Ctl* ctl, hipStream_t s) { LAUNCH(k_reset_ctl, 1, ctl); }

hipError_t launch_fill_i32(int32_t* p, int32_t v, int64_t n, int grid, hipStream_t s) {
    LAUNCH(k_fill_i32, grid, p, v, n);
}

hipError_t launch_trim1_first(const int32_t* fwb, const int32_t* bwb, int32_t V, int32_t* lab, uint64_t* act,
                              uint64_t* fvis, uint64_t* bvis, int32_t* fq, int32_t* q0, Ctl* ctl, PivotPart* part,
                              int pivot_wrap32, int grid, hipStream_t s) {
    LAUNCH(k_trim1_first, grid, fwb, bwb, V, lab, act, fvis, bvis, fq, q0, ctl, part, pivot_wrap32);
}

hipError_t launch_td_level(bool bw, const int32_t* beg, const int32_t* adj, const uint64_t* allow, uint64_t* vis,
                           int32_t* const q[2], HubItem* const hub[2], Ctl* ctl, int par, int grid, hipStream_t s,
                           hipEvent_t ev_mid) {
    if (bw)
        hipLaunchKernelGGL(k_td<true>, dim3(grid), dim3(kBlock), 0, s, beg, adj, allow, vis, q[par], q[par ^ 1],
                           hub[par], ctl, par);
    else
        hipLaunchKernelGGL(k_td<false>, dim3(grid), dim3(kBlock), 0, s, beg, adj, allow, vis, q[par], q[par ^ 1],
                           hub[par], ctl, par);
    if (ev_mid) (void)hipEventRecord(ev_mid, s);
    if (bw)
        hipLaunchKernelGGL(k_td_hub<true>, dim3(grid), dim3(kBlock), 0, s, beg, adj, allow, vis, hub[par],
                           q[par ^ 1], ctl, par);
    else
        hipLaunchKernelGGL(k_td_hub<false>, dim3(grid), dim3(kBlock), 0, s, beg, adj, allow, vis, hub[par],
                           q[par ^ 1], ctl, par);
    return hipGetLastError();
}

hipError_t launch_bu_level(bool bw, const int32_t* beg, const int32_t* adj, const uint64_t* allow, uint64_t* vis,
                           int32_t* const q[2], HubItem* const hub[2], Ctl* ctl, int par, int64_t nwords, int grid,
                           hipStream_t s) {
    (void)hub;
    if (bw) {
        LAUNCH(k_bu<true>, grid, beg, adj, allow, vis, q[par ^ 1], ctl, par, nwords);
    } else {
        LAUNCH(k_bu<false>, grid, beg, adj, allow, vis, q[par ^ 1], ctl, par, nwords);
    }
}

hipError_t launch_bw_init(uint64_t* bvis, int32_t* q0, Ctl* ctl, hipStream_t s) {
    hipLaunchKernelGGL(k_bw_init, dim3(1), dim3(1), 0, s, bvis, q0, ctl);
    return hipGetLastError();
}

hipError_t launch_popcount(const uint64_t* bm, int64_t nwords, int64_t* out, int grid, hipStream_t s) {
    LAUNCH(k_popcount, grid, bm, nwords, out);
}

hipError_t launch_post_giant(int32_t V, int32_t* lab, uint64_t* act, const uint64_t* bvis, int32_t* fq, Ctl* ctl,
                             int grid, hipStream_t s) {
    LAUNCH(k_post_giant, grid, V, lab, act, bvis, fq, ctl);
}

hipError_t launch_trim1_sweep(const int32_t* fwb, const int32_t* fwa, const int32_t* bwb, const int32_t* bwa,
                              int32_t* lab, uint64_t* act, int32_t* const fq[2], Ctl* ctl, int sel, int grid,
                              hipStream_t s) {
    hipLaunchKernelGGL(k_prep_sweep, dim3(1), dim3(1), 0, s, ctl, sel);
    LAUNCH(k_trim1, grid, fwb, fwa, bwb, bwa, lab, act, fq[sel], fq[sel ^ 1], ctl, sel);
}

hipError_t launch_pattern_trim(const int32_t* fwb, const int32_t* fwa, const int32_t* bwb, const int32_t* bwa,
                               int32_t* lab, int32_t* stamp, const uint64_t* act, const int32_t* fq, Ctl* ctl,
                               int sel, int grid, hipStream_t s) {
    LAUNCH(k_pattern, grid, fwb, fwa, bwb, bwa, lab, stamp, act, fq, ctl, sel);
}

hipError_t launch_pattern_commit(int32_t* lab, uint64_t* act, const int32_t* stamp, const int32_t* fq, Ctl* ctl,
                                 int sel, int grid, hipStream_t s) {
    LAUNCH(k_pattern_commit, grid, lab, act, stamp, fq, ctl, sel);
}

hipError_t launch_wcc_uf(const int32_t* fwb, const int32_t* fwa, const uint64_t* act, const int32_t* fq,
                         int32_t* parent, Ctl* ctl, int sel, int grid, hipStream_t s) {
    hipLaunchKernelGGL(k_uf_init, dim3(grid), dim3(kBlock), 0, s, fq, parent, ctl, sel);
    hipLaunchKernelGGL(k_uf_hook, dim3(grid), dim3(kBlock), 0, s, fwb, fwa, act, fq, parent, ctl, sel);
    LAUNCH(k_uf_compress, grid, fq, parent, ctl, sel);
}

hipError_t launch_lp_round(const int32_t* fwb, const int32_t* fwa, const int32_t* bwb, const int32_t* bwa,
                           const uint64_t* act, const int32_t* fq, int32_t* color, Ctl* ctl, int sel, int grid,
                           hipStream_t s) {
    hipLaunchKernelGGL(k_clear_changed, dim3(1), dim3(1), 0, s, ctl);
    hipLaunchKernelGGL(k_lp_sweep, dim3(grid), dim3(kBlock), 0, s, fwb, fwa, bwb, bwa, act, fq, color, ctl, sel);
    LAUNCH(k_lp_jump, grid, fq, color, ctl, sel);
}

hipError_t launch_uf_init(const int32_t* fq, int32_t* parent, Ctl* ctl, int sel, int grid, hipStream_t s) {
    LAUNCH(k_uf_init, grid, fq, parent, ctl, sel);
}

hipError_t launch_mice(const int32_t* fwb, const int32_t* fwa, const int32_t* bwb, const int32_t* bwa, int32_t* lab,
                       int32_t* stamp, const int32_t* fq, int32_t n, const int32_t* wcc, const MiceBuf& m, Ctl* ctl,
                       int32_t max_wcc, int grid, hipStream_t s) {
    const int g = (int)std::max<int64_t>(1, std::min<int64_t>(grid, ((int64_t)n + kBlock - 1) / kBlock));
    hipLaunchKernelGGL(k_wcc_reset, dim3(g), dim3(kBlock), 0, s, fq, n, wcc, m.cnt, ctl);
    hipLaunchKernelGGL(k_wcc_slots, dim3(g), dim3(kBlock), 0, s, fq, n, wcc, m.cnt, m.slot, stamp);
    hipLaunchKernelGGL(k_wcc_ranges, dim3(std::min(g, kRangeBlocks)), dim3(kBlock), 0, s, fq, n, wcc, m.cnt, m.first, m.roots, ctl);
    hipLaunchKernelGGL(k_wcc_members, dim3(g), dim3(kBlock), 0, s, fq, n, wcc, m.first, m.slot, m.member);
    // a wave per WCC, of which there are at most n
    const int gm = (int)std::max<int64_t>(1, std::min<int64_t>(grid, ((int64_t)n + kBlock / kWave - 1) / (kBlock / kWave)));
    LAUNCH(k_mice, gm, fwb, fwa, bwb, bwa, lab, stamp, m.roots, m.cnt, m.first, m.slot, m.member, ctl, m.queue,
           max_wcc);
}

hipError_t launch_count_unlabelled(const int32_t* lab, int32_t V, const uint64_t* sel, Ctl* ctl, int grid,
                                   hipStream_t s) {
    LAUNCH(k_count_unlabelled, grid, lab, V, sel, ctl);
}

hipError_t launch_check_csr(const CsrPair& pair, int32_t V, int64_t E, Ctl* ctl, int grid, hipStream_t s) {
    LAUNCH(k_check_csr, std::max(grid & ~1, 2), pair, V, E, ctl);
}

hipError_t launch_stats(const int32_t* fwb, const int32_t* bwb, const int32_t* lab, const uint64_t* fvis,
                        const uint64_t* bvis, int32_t V, Ctl* ctl, int grid, hipStream_t s) {
    LAUNCH(k_stats, grid, fwb, bwb, lab, fvis, bvis, V, ctl);
}

hipError_t launch_scc_histogram(const int32_t* lab, int32_t V, int32_t* size, int64_t* out, hipStream_t s) {
    static_assert(kHistSlots <= kBlock, "one thread clears one slot");
    const int grid = (int)std::max<int64_t>(1, std::min<int64_t>(kHistGrid, ((int64_t)V + 4 * kBlock - 1) / (4 * kBlock)));
    hipLaunchKernelGGL(k_size_roots, dim3(grid), dim3(kBlock), 0, s, lab, V, size, out);
    hipLaunchKernelGGL(k_scc_sizes, dim3(grid), dim3(kBlock), 0, s, lab, V, size);
    LAUNCH(k_scc_hist, grid, size, V, out);
}

}  // namespace ispan
