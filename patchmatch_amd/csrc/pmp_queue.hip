// pmp_queue.hip -- the work-queue kernels and the batched form.
//
// Every stage is one launch of a persistent kernel whose blocks walk a list
// of work items over all slots of a descriptor set:
//   k_init_q       random init + initial score; items (slot, 64x4 tile), the
//                  tile's reference taps staged in LDS
//   k_score_q      score of the working planes; items (slot, 64x4 tile)
//   k_propagate_q  one or several red-black passes; items (slot, tile of 64 R
//                  same-colour pixels), split into 8 contiguous bands, one per
//                  XCD, each taken through atomic heads (take_tile)
//   k_copyback_q, k_median_q (x2), k_postfilter_q   finalize; items (slot, row)
// Descriptors (SlotDesc) and work lists live in device memory and are read
// with scalar loads (constant address space); launches carry only pointers,
// so a captured hipGraph of a whole densification replays for any slots with
// the same iteration count.  The view count is a run-time value (views in
// groups of at most 4, per-view scores parked in LDS): one kernel serves
// keyframes of every size and view count in the same launch.
#include <math.h>
#include <string.h>

#include <algorithm>

#include "pmp_trace.h"
#include "pmp_internal.h"
#include "pmp_math.h"
#include "pmp_queue.h"
#include "pmp_score.h"
#include "pmp_tile.h"

#define PMP_CONST __attribute__((address_space(4)))

namespace pmp {

// Slot holding `item` (uniform binary search) and the item's index in it.
__device__ __forceinline__ int list_find(const WorkList PMP_CONST* L, int item, int& local) {
    int lo = 0, hi = L->n - 1;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (item < L->end[mid]) hi = mid;
        else lo = mid + 1;
    }
    local = item - (lo ? L->end[lo - 1] : 0);
    return L->slot[lo];
}

__device__ __forceinline__ const SlotDesc& slot_ref(const SlotDesc PMP_CONST* slots, int s) {
    return *(const SlotDesc*)(slots + s);
}

__global__ void k_fill_u32(unsigned int* __restrict__ p, int n, unsigned int v) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) p[k] = v;
}

// An init tile is 4 rows x 64 columns, one row per wave.  Its reference
// patch and bearing-table entries (the tile plus a halo of half each side,
// coordinates clamped: only interior pixels, whose taps lie inside the image,
// read them) are staged in LDS, as for a propagation tile, so that the tap
// reads never wait behind the neighbour gathers issued before them.  The planes
// are random, so each pixel's patches lie elsewhere and the gathers' cache
// lines bound the kernel; by quads of lanes (score_wave) a 1920x960 keyframe
// with 6 views takes 1.05 ms, with a plane per lane 1.25.  With one view only
// a quarter of a quad's lanes have one to accumulate, and a plane per lane is
// the faster form (queue_run).
constexpr int kInitRows = 4;
constexpr int kInitStageRows = kInitRows + 2 * kMaxHalf;
// A wave owns kOwn pixels of the tile: 64, or 32 or 16 where the launch would
// leave the chip idle (queue_run), which takes fewer rounds of score_wave.
// kOwn 0: 64 pixels, a plane per lane.
template <int kOwn>
struct InitShared {
    static constexpr bool kLanes = kOwn == 0;
    static constexpr int kPix = kLanes ? 64 : kOwn;     // a wave's pixels
    static constexpr int kWaves = 64 * kInitRows / kPix;
    QuadTap walk[kLanes ? 1 : kQuadTaps];
    std::conditional_t<kLanes, LaneShared, QuadShared> eval[kWaves];
    float4 rs[64 * kInitRows];
    float4 plane[64 * kInitRows];
    float score[64 * kInitRows];
    float2 row[kInitStageRows];
    float2 col[kTileCols];
    float sWc[256];
    float ic[64 * kInitRows];
    uint8_t ref[kInitStageRows * kTileCols];
};
static_assert(64 + 2 * kMaxHalf <= kTileCols, "init tile columns");

// Waits for the previous tile's readers first.
template <int kOwn>
__device__ __forceinline__ LdsTaps stage_init_tile(const KfArgs& a, InitShared<kOwn>& st, int tx, int ty) {
    constexpr int NT = 64 * InitShared<kOwn>::kWaves;
    const int r0 = ty * kInitRows - a.half, c0 = 64 * tx - a.half;
    const int nr = kInitRows + 2 * a.half, nc = 64 + 2 * a.half;
    __syncthreads();
    for (int e = threadIdx.x; e < nc; e += NT) st.col[e] = a.coltab[min(max(c0 + e, 0), a.W - 1)];
    for (int e = threadIdx.x; e < nr; e += NT) st.row[e] = a.rowtab[min(max(r0 + e, 0), a.H - 1)];
    for (int e = threadIdx.x; e < nr * nc; e += NT) {
        const int r = e / nc, c = e - r * nc;
        const int y = min(max(r0 + r, 0), a.H - 1), x = min(max(c0 + c, 0), a.W - 1);
        st.ref[r * kTileCols + c] = a.ref[(size_t)y * a.W + x];
    }
    __syncthreads();
    return LdsTaps{st.row, st.col, st.ref, r0, c0};
}

// kScore: only score the working planes (pmp_score_plane_depth); otherwise
// random initialisation + score + snapshot (RandomInitialization,
// PatchMatchCuda.cu:210-270, depthmap.cc:656-663).
template <bool kZero, bool kScore, int kOwn>
__global__ __launch_bounds__(64 * InitShared<kOwn>::kWaves) void k_init_q(const SlotDesc PMP_CONST* slots,
                                                                        const BatchHdr PMP_CONST* hdr) {
    __shared__ InitShared<kOwn> st;
    const WorkList PMP_CONST* L = &hdr->init;
    const int total = L->total;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    constexpr int PW = InitShared<kOwn>::kPix;
    const bool owner = PW == 64 || lane < PW;   // lanes beyond own no pixel but take part in the evaluations
    const int t = PW * wave + (owner ? lane : 0);
    int cur = -1;
    for (int item = blockIdx.x; item < total; item += gridDim.x) {
        int local;
        const int s = list_find(L, item, local);
        const SlotDesc& d = slot_ref(slots, s);
        const KfArgs& a = d.a;
        if (s != cur) {
            __syncthreads();
            load_wc(a.Wc, st.sWc);
            if constexpr (kOwn != 0) load_walk(a, st.walk);
            cur = s;
        }
        const int tx = local % d.nbx_init, ty = local / d.nbx_init;
        const LdsTaps tp = stage_init_tile(a, st, tx, ty);
        const int j = tx * 64 + (t & 63);
        const int i = ty * kInitRows + (t >> 6);
        const bool in = owner && i < a.H && j < a.W;
        const bool scored = in && in_score_grid(a, i, j);
        const size_t k = in ? (size_t)i * a.W + j : 0;
        float p0 = 0.0f, p1 = 0.0f, p2 = 0.0f, dep = 0.0f;
        if constexpr (kScore) {
            if (scored) {
                const float4 p = d.plane[k];
                p0 = p.x; p1 = p.y; p2 = p.z;
            }
        } else {
            if (in && in_init_grid(a, i, j)) random_plane(a, i, j, p0, p1, p2, dep);
        }
        RefStat rs = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        if (scored) rs = ref_stats(a, tp, st.sWc, i, j);
        if (owner) {
            st.rs[t] = make_float4(rs.mx, rs.inv, rs.mxc, rs.vx);
            st.ic[t] = rs.Ic;
            st.plane[t] = make_float4(p0, p1, p2, 0.0f);
        }
        wave_exchange();   // a wave reads its own pixels' entries
        auto at = [&](int p, int& row, int& col) {
            row = (p >> 6) + a.half;
            col = (p & 63) + a.half;
        };
        auto job = [&](int l, int& jt, float& px, float& py, float& pz) {
            jt = PW * wave + l;
            const float4 p = st.plane[jt];
            px = p.x; py = p.y; pz = p.z;
        };
        auto put = [&](int l, float v) { st.score[PW * wave + l] = v; };
        if constexpr (kOwn == 0)
            score_lanes<kZero>(a, tp, st.sWc, st.rs, st.ic, at, job, put, __ballot(scored), &st.eval[wave].sv[0][0]);
        else
            score_wave<kZero>(a, tp, st.walk, st.sWc, st.rs, st.ic, at, job, put, __ballot(scored), st.eval[wave]);
        const float sc = scored ? st.score[t] : __uint_as_float(0xFFFFFFFFu);   // cudaMemset(score, 0xFF) (depthmap.cc:657)
        if constexpr (kScore) {
            if (scored) d.score[k] = sc;
        } else if (in) {
            const float4 pl = make_float4(p0, p1, p2, 0.0f);
            d.plane[k] = pl; d.depth[k] = dep; d.score[k] = sc;
            d.iplane[k] = pl; d.idepth[k] = dep; d.iscore[k] = sc;
        }
    }
}

// Debug pass epochs (SlotDesc::epochs).  A tile about to run red-black pass
// pp must have completed pp passes, and each of the 8 tiles around it (whose
// maps its candidates and the other colour's pixels come from, 3 pixels at
// most across a tile edge) pp or pp + 1: the previous pass wrote them and this
// one writes only the colour that pass pp does not read.  Anything else (a
// tile skipped, run twice, or run before the pass before it finished) adds to
// the violation count.  Tiles of one launch may see each other's stores or not;
// both values are allowed.
__device__ __forceinline__ void epoch_enter(const SlotDesc& d, int tx, int ty, int pp) {
    if (threadIdx.x != 0) return;
    unsigned int* e = d.epochs;
    const int nbx = d.nbx_prop, nby = d.nby_prop;
    unsigned int bad = 0;
    for (int dy = -1; dy <= 1; ++dy)
        for (int dx = -1; dx <= 1; ++dx) {
            const int x = tx + dx, y = ty + dy;
            if (x < 0 || y < 0 || x >= nbx || y >= nby) continue;
            const unsigned int v = __hip_atomic_load(&e[y * nbx + x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const bool ok = (dx == 0 && dy == 0) ? v == (unsigned int)pp : (v == (unsigned int)pp || v == (unsigned int)pp + 1u);
            bad += ok ? 0u : 1u;
        }
    if (bad) atomicAdd(&e[nbx * nby], bad);
}

// After every lane's map writes of the tile: its epoch becomes pp + 1.
__device__ __forceinline__ void epoch_leave(const SlotDesc& d, int tx, int ty, int pp) {
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        __hip_atomic_store(&d.epochs[ty * d.nbx_prop + tx], (unsigned int)pp + 1u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---- all red-black passes of a call in one launch
// A tile may run pass p + 1 as soon as it and the 8 tiles around it have
// completed pass p: they wrote what it reads, and, since they in turn wait for
// this tile, none of them is ahead by more than one pass, which writes only
// the colour that this one does not read.  So the tail of a pass, when its
// last tiles leave compute units idle, overlaps the next pass.
//
// Every block takes tiles of its own XCD's band (home) and of bands that are
// behind it.  Pass-0 tiles are handed out in list order through a ticket per
// band.  A tile that completes pass p counts itself in at the 9 tiles it may
// release (arrivals, one count per pass parity: a neighbour cannot complete
// pass p + 2 before this tile has completed p + 1, so the counts of one parity
// never mix two passes); the last of a tile's arrivals puts (tile, p + 1) into
// its band's ring, from which blocks take tiles in that order.
//
// No block waits while it holds a tile, and none takes a ring entry that has
// not been announced, so some block progresses whatever part of the grid is
// resident: a tile that is ready lies in a ring, and any running block that
// has no work looks through all rings.  The two waits for another block's
// store (a ring slot announced but not written yet, one taken but not read
// yet) are for blocks that are past every other wait.
//
// The hand-over is ordered by fences: a completed tile's maps are released
// before its arrivals, the last arrival acquires the others' and releases all
// before the ring entry, and the wave that takes the entry acquires them for its
// block.
//
// heads: four words per band, each in a cache line of its own.  A block takes an
// entry by a permit (ready, counted down) and then a ticket (ring): where most
// blocks want the same band, each does two additions, while a compare-and-swap
// of the ring's head let one of them through per 2.7 us (eight 960x480
// keyframes, one view, in a single band: 157 ms, 15.4 now; 640x320, 2 views,
// from a warped result: 2.89, 2.53 now).
__device__ __forceinline__ unsigned int* head_of(unsigned int* heads, int kind, int band) {
    return heads + (kind * 8 + band) * kHeadStride;
}
// A block without work looks again after 64 x 64 cycles, then after up to
// kMaxNaps times that: the looks share a few cache lines with the others' atomics.
constexpr int kNap = 64, kMaxNaps = 4;
enum { kHeadFirst = 0, kHeadRing = 1, kHeadTail = 2, kHeadReady = 3 };   // pass-0 tickets; ring entries taken, announced, ready

__device__ __forceinline__ int load_agent(const unsigned int* p) {
    return (int)__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int band_lo(int total, int band, int nb) { return (int)(((long long)total * band) / nb); }

// Takes the block's next (tile, pass) into sh.item (-1: nothing is left to
// take) and sh.pass: from the band that is furthest behind among those with a
// tile to take, its own on a tie.  (Own band first whatever its pass let a
// keyframe's cheap bands run ahead of its dear ones, whose last passes then ran
// on few tiles: a 1920x960 keyframe whose bottom eighth starts from random
// planes and the rest from a warped result took 17.3 ms for 4 passes.)  Called
// by the block's first wave; lane b < 8 looks at band home + b.
template <int R, int F>
__device__ __forceinline__ void take_tile(const BatchHdr PMP_CONST* hdr, int passes, unsigned int* heads, int bands,
                                          PropShared<R, F>& sh) {
    const int total = hdr->prop.total;
    unsigned int* ring = hdr->sync + 2 * (size_t)total;
    const int nb = bands ? 8 : 1;
    const int home = bands ? (int)(blockIdx.x & 7) : 0;
    const int lane = threadIdx.x;
    const int band = (home + lane) & (nb - 1);
    const int lo = band_lo(total, band, nb), n = band_lo(total, band + 1, nb) - lo;
    unsigned int* h0 = head_of(heads, kHeadFirst, band);
    unsigned int* hr = head_of(heads, kHeadRing, band);
    unsigned int* ready = head_of(heads, kHeadReady, band);
    int item = -1, pass = 0, naps = 1;
    for (;;) {
        int level = 0x7FFFFFFF;          // the pass (about, in the ring) of the band's next tile
        bool left = false;
        if (lane < nb && n > 0) {
            if (load_agent(h0) < n) {
                level = 0;
            } else if (passes > 1) {
                const int q = load_agent(hr);
                left = q < n * (passes - 1);
                if (load_agent(ready) > 0) level = 1 + q / n;
            }
        }
        int best = level;
#pragma unroll
        for (int k = 1; k < 8; k <<= 1) best = min(best, __shfl_xor(best, k, 64));
        const unsigned long long at = __ballot(lane < nb && level == best && level != 0x7FFFFFFF);
        if (at == 0ull) {
            if (__ballot(left) == 0ull) break;
            for (int k = 0; k < naps; ++k) __builtin_amdgcn_s_sleep(kNap);
            naps = min(2 * naps, kMaxNaps);
            continue;
        }
        bool got = false;
        if (lane == __ffsll((long long)at) - 1) {
            if (level == 0) {
                const int h = (int)atomicAdd(h0, 1u);
                got = h < n;
                item = lo + h;
                pass = 0;
            } else if ((int)atomicSub(ready, 1u) > 0) {
                const unsigned int q = atomicAdd(hr, 1u);
                unsigned int v;
                while ((v = atomicExch(&ring[lo + q % (unsigned int)n], 0u)) == 0u) __builtin_amdgcn_s_sleep(1);
                got = true;
                item = (int)(v & 0xFFFFFFu);
                pass = (int)(v >> 24);
            } else {
                atomicAdd(ready, 1u);   // the last one went to another block
            }
            if (got) {
                sh.item = item;
                sh.pass = pass;
            }
        }
        if (__any(got)) return;
    }
    if (lane == 0) sh.item = -1;
}

constexpr int kVmcnt0 = 0x0F70;   // s_waitcnt vmcnt(0), no other counter

// The block's tile (list index item, at (tx, ty) of slot d) has completed
// pass `pass` of the launch, which is not the last: counts it in at the tiles
// around it and announces those that are now ready.  Called by every thread.
__device__ __forceinline__ void release_tiles(const BatchHdr PMP_CONST* hdr, const SlotDesc& d, unsigned int* heads,
                                              int bands, int item, int tx, int ty, int pass) {
    // every wave's stores have left its compute unit before the barrier
    // (vmcnt(0)), and one wave releases them all: a fence by every wave, each
    // writing back and invalidating caches, cost 4-12 % of a densification with
    // one or two views (1920x960, 1 view, 25 taps, 3 iterations: 5.35 ms, 4.80
    // now)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(kVmcnt0);
    __syncthreads();
    if (threadIdx.x >= 9) return;
    // the wait for the write-back, which the compiler leaves out where it sees
    // no store of the wave's own in flight
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    __builtin_amdgcn_s_waitcnt(kVmcnt0);
    const int total = hdr->prop.total;
    const int nb = bands ? 8 : 1;
    const int nbx = d.nbx_prop, nby = d.nby_prop;
    const int x = tx + (int)threadIdx.x % 3 - 1, y = ty + (int)threadIdx.x / 3 - 1;
    if (x < 0 || y < 0 || x >= nbx || y >= nby) return;
    const int t = item - (ty * nbx + tx) + y * nbx + x;
    const int around = (min(x + 1, nbx - 1) - max(x - 1, 0) + 1) * (min(y + 1, nby - 1) - max(y - 1, 0) + 1);
    const int arrived = (int)atomicAdd(&hdr->sync[(size_t)(pass & 1) * total + t], 1u) + 1;
    if (arrived != around * (pass / 2 + 1)) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "agent");   // the other arrivals' maps, with the ring entry
    int band = (int)(((long long)t * nb) / total);
    while (t >= band_lo(total, band + 1, nb)) ++band;
    const int lo = band_lo(total, band, nb), n = band_lo(total, band + 1, nb) - lo;
    const int q = (int)atomicAdd(head_of(heads, kHeadTail, band), 1u);
    unsigned int* slot = hdr->sync + 2 * (size_t)total + lo + q % n;
    while (atomicCAS(slot, 0u, ((unsigned int)(pass + 1) << 24) | (unsigned int)t) != 0u) __builtin_amdgcn_s_sleep(1);
    atomicAdd(head_of(heads, kHeadReady, band), 1u);
}

// One launch over `passes` red-black passes of every slot, the first being
// pass `first` of the call.
//
// A block has 64 threads to each wave of its form (prop_shape).
template <int R, int F>
constexpr int kPropThreads = 64 * PropShared<R, F>::kWaves;
template <bool kZero, int R, int F>
__global__ __launch_bounds__((kPropThreads<R, F>))
    __attribute__((amdgpu_waves_per_eu(F != kLane || kZero ? 4 : 1))) void k_propagate_q(
    const SlotDesc PMP_CONST* slots, const BatchHdr PMP_CONST* hdr, int first, int passes,
    unsigned int* __restrict__ heads, unsigned long long* __restrict__ counters, int bands) {
    __shared__ PropShared<R, F> sh;
    const WorkList PMP_CONST* L = &hdr->prop;
    unsigned int n_eval = 0, n_cand = 0;   // of the wave
    int cur = -1;
    for (;;) {
        if (threadIdx.x < 64) {
            take_tile(hdr, passes, heads, bands, sh);
            // the maps that the ring entry hands over (release_tiles), before the block reads any
            if (passes > 1) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        __syncthreads();
        const int item = sh.item, pass = sh.pass;
        __syncthreads();
        if (item < 0) break;
        int local;
        const int s = list_find(L, item, local);
        const SlotDesc& d = slot_ref(slots, s);
        if (s != cur) {
            load_wc(d.a.Wc, sh.sWc);
            if constexpr (F != kLane) load_walk(d.a, sh.walk);
            cur = s;
        }
        const int pp = d.pass0 + first + pass;
        const int tx = local % d.nbx_prop, ty = local / d.nbx_prop;
        if (d.epochs) epoch_enter(d, tx, ty, pp);
        propagate_tile<kZero, R, F>(d.a, sh, d.plane, d.depth, d.score, pp >> 1, pp & 1, tx, ty,
                                     item & (PropShared<R, F>::kWaves - 1), n_eval, n_cand);
        if (d.epochs) epoch_leave(d, tx, ty, pp);
        if (pass + 1 < passes) release_tiles(hdr, d, heads, bands, item, tx, ty, pass);
    }
    count_add_wave(&counters[0], n_eval);
    count_add_wave(&counters[1], n_cand);
}

__global__ __launch_bounds__(256) void k_copyback_q(const SlotDesc PMP_CONST* slots, const BatchHdr PMP_CONST* hdr) {
    const WorkList PMP_CONST* L = &hdr->rows;
    for (int item = blockIdx.x; item < L->total; item += gridDim.x) {
        int i;
        const SlotDesc& d = slot_ref(slots, list_find(L, item, i));
        for (int j = threadIdx.x; j < d.a.W; j += blockDim.x)
            copyback_pixel(d.a, d.mask, d.iplane, d.idepth, d.iscore, d.plane, d.depth, d.score, d.oplane, d.odepth,
                           d.oscore, d.onghbr, d.min_var, d.inv_T, i, j);
    }
}

__global__ __launch_bounds__(256) void k_median_q(const SlotDesc PMP_CONST* slots, const BatchHdr PMP_CONST* hdr,
                                                  int second) {
    const WorkList PMP_CONST* L = &hdr->rows;
    for (int item = blockIdx.x; item < L->total; item += gridDim.x) {
        int i;
        const SlotDesc& d = slot_ref(slots, list_find(L, item, i));
        if (!d.postprocess) continue;
        const float* src = second ? d.tmp0 : d.odepth;
        float* dst = second ? d.tmp1 : d.tmp0;
        for (int j = threadIdx.x; j < d.a.W; j += blockDim.x) median3_pixel(src, dst, d.a.W, d.a.H, i, j);
    }
}

__global__ __launch_bounds__(256) void k_postfilter_q(const SlotDesc PMP_CONST* slots,
                                                      const BatchHdr PMP_CONST* hdr) {
    const WorkList PMP_CONST* L = &hdr->rows;
    for (int item = blockIdx.x; item < L->total; item += gridDim.x) {
        int i;
        const SlotDesc& d = slot_ref(slots, list_find(L, item, i));
        if (!d.postprocess) continue;
        for (int j = threadIdx.x; j < d.a.W; j += blockDim.x)
            postfilter_pixel(d.tmp1, d.odepth, d.oscore, (size_t)i * d.a.W + j, d.rel_thr, d.a.min_depth,
                             d.a.max_depth, d.min_score);
    }
}

// ---------------------------------------------------------------- host side

int desc_alloc(pmp_ctx* ctx, DescSet& d, int cap) {
    d.cap = cap;
    PMP_HIP(ctx, hipHostMalloc((void**)&d.h_slots, cap * sizeof(SlotDesc), hipHostMallocDefault));
    PMP_HIP(ctx, hipHostMalloc((void**)&d.h_hdr, sizeof(BatchHdr), hipHostMallocDefault));
    PMP_HIP(ctx, hipMalloc(&d.d_slots, cap * sizeof(SlotDesc)));
    PMP_HIP(ctx, hipMalloc(&d.d_hdr, sizeof(BatchHdr)));
    PMP_HIP(ctx, hipMalloc(&d.d_heads, std::max(kMaxPasses * kFirstWords, kHeadWords) * sizeof(unsigned int)));
    PMP_HIP(ctx, hipEventCreateWithFlags(&d.uploaded, hipEventDisableTiming));
    return PMP_OK;
}

void desc_free(DescSet& d) {
    for (auto& kv : d.graphs) {
        (void)hipGraphExecDestroy(kv.second.second);
        (void)hipGraphDestroy(kv.second.first);
    }
    if (d.h_slots) (void)hipHostFree(d.h_slots);
    if (d.h_hdr) (void)hipHostFree(d.h_hdr);
    if (d.d_slots) (void)hipFree(d.d_slots);
    if (d.d_hdr) (void)hipFree(d.d_hdr);
    if (d.d_heads) (void)hipFree(d.d_heads);
    if (d.d_sync) (void)hipFree(d.d_sync);
    if (d.uploaded) (void)hipEventDestroy(d.uploaded);
    d = DescSet();
}

int desc_begin(pmp_ctx* ctx, DescSet& d) {
    if (d.pending) {
        PMP_HIP(ctx, hipEventSynchronize(d.uploaded));
        d.pending = false;
    }
    return PMP_OK;
}

int desc_upload(pmp_ctx* ctx, DescSet& d, int n, hipStream_t stream) {
    PMP_HIP(ctx, hipMemcpyAsync(d.d_slots, d.h_slots, n * sizeof(SlotDesc), hipMemcpyHostToDevice, stream));
    PMP_HIP(ctx, hipMemcpyAsync(d.d_hdr, d.h_hdr, sizeof(BatchHdr), hipMemcpyHostToDevice, stream));
    PMP_HIP(ctx, hipEventRecord(d.uploaded, stream));
    d.pending = true;
    return PMP_OK;
}

void queue_free(pmp_ctx* ctx) {
    QueueState* q = ctx->queue;
    if (!q) return;
    desc_free(q->plain);
    desc_free(q->batch);
    for (auto& b : q->bufs) free_slot(b);
    delete q;
    ctx->queue = nullptr;
}

int queue_state(pmp_ctx* ctx, QueueState*& out) {
    if (!ctx->queue) {
        QueueState* q = new (std::nothrow) QueueState();
        if (!q) return set_error(ctx, PMP_ENOMEM, "queue state");
        ctx->queue = q;
        int rc = desc_alloc(ctx, q->plain, 1);
        if (!rc) rc = desc_alloc(ctx, q->batch, kMaxSlots);
        if (rc) {
            queue_free(ctx);
            return rc;
        }
        PMP_HIP(ctx, hipDeviceGetAttribute(&q->cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
        q->bufs.resize(kMaxSlots);
    }
    out = ctx->queue;
    return PMP_OK;
}

void fill_list(WorkList& L, int n, const int* items) {
    L.n = 0;
    L.total = 0;
    for (int s = 0; s < n; ++s) {
        if (items[s] <= 0) continue;
        L.total += items[s];
        L.slot[L.n] = s;
        L.end[L.n] = L.total;
        L.n++;
    }
}

int slot_fill(pmp_ctx* ctx, const pmp_params* params, const pmp_keyframe& kf, const SlotBuf& b, const uint8_t* dmask,
              int pass0, hipStream_t stream, SlotDesc& d, int items[2]) {
    pmp_params pk = *params;
    if (kf.min_depth > 0.0f) pk.min_depth = kf.min_depth;
    if (kf.max_depth > 0.0f) pk.max_depth = kf.max_depth;
    memset(&d, 0, sizeof(d));
    int rc = build_args(ctx, &pk, kf.ref_id, kf.n_views, kf.view_ids, (const double*)&kf.ref_pose,
                        (const double*)kf.view_poses, stream, d.a);
    if (rc) return rc;
    const int W = d.a.W, H = d.a.H;
    if ((size_t)W * H > b.cap) return set_error(ctx, PMP_ESTATE, "keyframe maps are smaller than the keyframe");
    d.plane = b.plane; d.depth = b.depth; d.score = b.score;
    d.iplane = b.iplane; d.idepth = b.idepth; d.iscore = b.iscore;
    d.oplane = b.oplane; d.odepth = b.odepth; d.oscore = b.oscore; d.onghbr = b.onghbr;
    d.tmp0 = b.tmp0; d.tmp1 = b.tmp1;
    d.mask = dmask;
    if (!dmask && kf.mask_id >= 0) {
        auto im = ctx->images.find((uint64_t)kf.mask_id);
        if (im == ctx->images.end()) return set_error(ctx, PMP_ENOTFOUND, "unknown mask image id");
        if (im->second.W != W || im->second.H != H)
            return set_error(ctx, PMP_EINVAL, "mask image size differs from the reference");
        d.mask = im->second.gray;
    }
    d.min_var = pk.min_patch_sd * pk.min_patch_sd;
    d.inv_T = (float)(1.0 / (double)d.a.T);
    d.rel_thr = pk.median_rel_thr;
    d.min_score = pk.min_score;
    d.postprocess = pk.postprocess;
    d.pass0 = pass0;
    d.nbx_init = (W + 63) / 64;
    d.nbx_prop = ((W + 1) / 2 + kTileSame - 1) / kTileSame;
    items[0] = d.nbx_init * ((H + 3) / 4);
    items[1] = H;
    return PMP_OK;
}

int slot_tiles(SlotDesc& d, int rows) {
    const int trows = 64 * rows / kTileSame;   // rows of a propagation tile
    d.nby_prop = (d.a.H + trows - 1) / trows;
    return d.nbx_prop * d.nby_prop;
}

// The kernel of a form and tile size, and its block size.  Tiles of 8 rows
// have no kWide kernel: one block of it would be 2048 threads.
struct PropKernel {
    const void* fn;
    int threads;
};
template <bool kZero, int R, int F>
static PropKernel prop_kernel_of() { return {(const void*)k_propagate_q<kZero, R, F>, kPropThreads<R, F>}; }
template <bool kZero, int F>
static PropKernel prop_kernel_f(int rows) {
    if (rows == 2) return prop_kernel_of<kZero, 2, F>();
    if (rows == 4) return prop_kernel_of<kZero, 4, F>();
    return prop_kernel_of<kZero, 8, F == kWide ? kQuad : F>();
}
template <bool kZero>
static PropKernel prop_kernel_z(int form, int rows) {
    if (form == kLane) return prop_kernel_f<kZero, kLane>(rows);
    if (form == kWide) return prop_kernel_f<kZero, kWide>(rows);
    return prop_kernel_f<kZero, kQuad>(rows);
}
static PropKernel prop_kernel(bool zero, int form, int rows) {
    return zero ? prop_kernel_z<true>(form, rows) : prop_kernel_z<false>(form, rows);
}

static bool is_default(const pmp_batch_config& c) {
    return c.tile_rows == kDefaultConfig.tile_rows && c.blocks_per_cu == kDefaultConfig.blocks_per_cu;
}

void prop_shape(const QueueState& q, const pmp_batch_config& c, int n, const int* slot, const SlotDesc* slots,
                bool single, QueueRun& r) {
    // work: the pixels of one colour in units of 64; chip: waves at four to a
    // SIMD; gain: what kLane wins over kQuad, per unit of work about 2 with one
    // view, 1 with two, 0 with three and -3 with more
    double work = 0.0, gain = 0.0;
    int views = 0;
    for (int k = 0; k < n; ++k) {
        const KfArgs& a = slots[slot ? slot[k] : k].a;
        const double w = (double)a.W * a.H / 128.0;
        work += w;
        gain += w * (a.N >= 4 ? -3.0 : 3.0 - a.N);
        views = std::max(views, (int)a.N);
    }
    const double chip = 16.0 * q.cus;
    // Measured on densifications of 4 iterations, ms as kLane / kQuad / kWide,
    // each with the tile rows below:
    // - Below one and three quarters of the chip kWide: its tiles take four
    //   times the waves that the other forms have for the same pixels, which
    //   leave the chip idle there (480x240, 2 views: 2.2 / 2.9 / 1.7; 960x480,
    //   8 views: 13.9 / 13.7 / 11.2; 1280x640, 8 views: 20.7 / 21.3 / 20.1;
    //   1440x720, 4 views: 13.5 / 12.8 / 14.3).
    // - Above, kQuad: a quad's gathers fall into one patch (1920x960: 4 views
    //   23.5 / 21.6 / 25.9, 6 views 34.9 / 33.6 / 37.1; 2880x1440, 10 views: 152
    //   / 131 / 135).
    // - With one to three views some lanes of a quad have no view to
    //   accumulate, so kLane, where it fills the chip well enough: one view
    //   from 640x320 (1.73 / 2.26 / 1.74), two from 960x480 (3.79 / 4.23 / 4.32;
    //   800x400: 3.19 / 4.11 / 3.10), three from there up to 1680x840 (960x480:
    //   5.2 / 5.6 / 5.3; 1280x640: 7.8 / 8.5 / 9.2; 1680x840: 13.3 / 13.2 /
    //   16.2).
    const double lane_from = views == 1 ? 0.375 : 0.75, lane_to = views == 3 ? 2.5 : 1e30;
    if (views <= 3 && work > lane_from * chip && work < lane_to * chip)
        r.form = kLane;
    else if (work < 1.75 * chip)
        r.form = kWide;
    else
        // - A launch over keyframes of several view counts takes what most of its
        //   work is better with (eight of 960x480: seven with 1 view and one with
        //   4 18.7 / 20.0, seven with 2 and one with 10 33.9 / 34.7, four with 2
        //   and four with 4 33.5 / 32.2).
        r.form = gain > 0.0 ? kLane : kQuad;
    // kQuad, 1440x720, 4 views: 13.0 ms with 8 rows, 14.4 with 4, 12.9 with 2
    // (1920x960, 6 views: 33.1, 33.4, 35.0); with a launch per pass, whose last
    // tiles leave compute units idle, 15.5 with 8, 14.0 with 4, 14.3 with 2.  kWide, 640x320, 4 views: 3.4 with 2,
    // 3.5 with 4.  kLane: pmp_queue.h
    r.rows = !is_default(c) ? c.tile_rows : r.form == kLane ? 4 : r.form == kWide ? 2 : single ? 4 : 8;
    if (r.form == kWide && r.rows == 8) r.form = kQuad;
}

static int check_config(pmp_ctx* ctx, const pmp_batch_config& c) {
    if (c.tile_rows != 2 && c.tile_rows != 4 && c.tile_rows != 8)
        return set_error(ctx, PMP_EINVAL, "tile_rows must be 2, 4 or 8");
    if (c.blocks_per_cu < 0 || c.blocks_per_cu > 32) return set_error(ctx, PMP_EINVAL, "blocks_per_cu must be in [0, 32]");
    return PMP_OK;
}

// Persistent grid: the configured blocks per CU, capped by (and defaulting
// to) what fits on a CU at once; a multiple of 8 with per-XCD bands.
int queue_run(pmp_ctx* ctx, const QueueState& q, const pmp_batch_config& c, bool zero, bool post, const BatchHdr& h,
              const SlotDesc* slots, QueueRun& r) {
    const int tiles = h.prop.total;
    int occ = 0;
    const PropKernel kern = prop_kernel(zero, r.form, r.rows);
    PMP_HIP(ctx, hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern.fn, kern.threads, 0));
    if (occ < 1) occ = 1;
    int bpc = (c.blocks_per_cu <= 0 || c.blocks_per_cu > occ) ? occ : c.blocks_per_cu;
    // one plane per lane: with 12 waves' gathers a CU's L1 is full (16 waves: 2-4 % slower)
    if (c.blocks_per_cu <= 0 && r.form == kLane) bpc = std::min(bpc, std::max(1, 12 / r.rows));
    // blocks beyond one per tile would only look for work
    if (tiles > 0) bpc = std::min(bpc, (tiles + q.cus - 1) / q.cus);
    // One launch over all passes pays where the blocks in flight hold less
    // than two thirds of the tiles (1920x960, 4 views, 4 iterations: 21.5
    // against 24.6 ms; 640x320, 4 views: 3.4 against 4.2 ms).  Otherwise most
    // tiles are in flight at once and wait for each other tile by tile, while
    // the launches' own barrier leaves the last ones whole compute units
    // (480x240, 4 views, 4 iterations: 3.3 against 2.3 ms).
    // However many tiles there are to a block, the one launch is no slower (kLane,
    // 4 iterations: eight of 960x480, 1 view 14.7 / 15.1, 4600x2300 43.1 / 42.9,
    // eight of 2880x1440, 2 views 217.6 / 215.6; kQuad, 3 iterations: 5760x2880, 4
    // views 192 / 195, eight of 2880x1440 329 / 331).
    r.fused = 2 * tiles >= 3 * q.cus * bpc;
    // a block of 16 waves fits on a CU once, of 8 twice: while every tile has
    // one, its planes are scored in one or two rounds instead of four (init of
    // 320x160, 8 views: 72 us, 108 with four; of 480x240: 114 and 123); beyond,
    // the small blocks fill the chip better (640x320, 2 views: 82 us, 107 with
    // 16 waves).
    // There, a plane per lane with one view (us against quads: 640x320 58 / 66,
    // 1920x960 271 / 285, 3840x1920 1069 / 1061), with two or three up to six
    // tiles to a CU (800x400: 95 / 98 and 110 / 112; 960x480: 124 / 127 and 152
    // / 144), and with any but four up to four (640x320: 5 views 127 / 136, 4
    // views 117 / 115, 10 views 229 / 231; 720x360: 10 views 287 / 276).
    int views = 0;
    for (int k = 0; k < h.init.n; ++k) views = std::max(views, (int)slots[h.init.slot[k]].a.N);
    r.init_own = h.init.total <= q.cus       ? 16
                 : h.init.total <= 2 * q.cus ? 32
                 : views == 1 || (views <= 3 && h.init.total <= 6 * q.cus) ||
                         (views != 4 && h.init.total <= 4 * q.cus)
                     ? 0
                     : 64;
    r.zero = zero;
    r.post = post;
    r.bands = c.xcd_bands ? 1 : 0;
    r.blocks = q.cus * bpc;
    if (r.bands) r.blocks = (r.blocks + 7) / 8 * 8;
    return PMP_OK;
}

#define PMP_QPTRS                                                             \
    const SlotDesc PMP_CONST* sl = (const SlotDesc PMP_CONST*)d.d_slots;     \
    const BatchHdr PMP_CONST* hd = (const BatchHdr PMP_CONST*)d.d_hdr;

static int grid_blocks(pmp_ctx* ctx) {
    QueueState* q = ctx->queue;
    return (q && q->cus > 0 ? q->cus : 256) * 8;
}

// Before the launches of the propagation kernel: their band heads, the
// evaluation counters and, for one launch over several passes, the tiles'
// arrivals and the rings.
__global__ void k_clear(const BatchHdr PMP_CONST* hdr, unsigned int* __restrict__ heads, int head_words,
                        unsigned int* __restrict__ counters, int sync) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x, step = gridDim.x * blockDim.x;
    for (int t = k; t < head_words; t += step) heads[t] = 0u;
    if (k < 4) counters[k] = 0u;
    if (sync)
        for (int t = k; t < 3 * hdr->prop.total; t += step) hdr->sync[t] = 0u;
}

int q_clear(pmp_ctx* ctx, hipStream_t s, DescSet& d, const QueueRun& r, int passes) {
    PMP_QPTRS
    (void)sl;
    // a fill kernel, not memset nodes: the sequence may be captured
    const bool one = r.fused && passes > 1;
    const int words = one ? kHeadWords : kFirstWords * std::max(passes, 1);
    hipLaunchKernelGGL(k_clear, dim3(one ? 64 : (words + 255) / 256), dim3(256), 0, s, hd, d.d_heads, words,
                       (unsigned int*)ctx->counters, one ? 1 : 0);
    PMP_HIP(ctx, hipGetLastError());
    return PMP_OK;
}

int ensure_sync(pmp_ctx* ctx, DescSet& d, size_t tiles) {
    if (tiles > kMaxTiles) return set_error(ctx, PMP_EINVAL, "too many propagation tiles in one call");
    if (tiles > d.sync_cap) {
        PMP_HIP(ctx, hipStreamSynchronize(ctx->stream));
        if (d.d_sync) (void)hipFree(d.d_sync);
        d.d_sync = nullptr;
        d.sync_cap = 0;
        PMP_HIP(ctx, hipMalloc(&d.d_sync, 3 * tiles * sizeof(unsigned int)));
        d.sync_cap = tiles;
    }
    d.h_hdr->sync = d.d_sync;
    return PMP_OK;
}

template <bool kScore, int kOwn>
static void launch_init_own(hipStream_t s, dim3 grd, const SlotDesc PMP_CONST* sl, const BatchHdr PMP_CONST* hd,
                            bool zero) {
    const dim3 blk(64 * InitShared<kOwn>::kWaves);
    if (zero) hipLaunchKernelGGL((k_init_q<true, kScore, kOwn>), grd, blk, 0, s, sl, hd);
    else hipLaunchKernelGGL((k_init_q<false, kScore, kOwn>), grd, blk, 0, s, sl, hd);
}
template <bool kScore>
static int launch_init(pmp_ctx* ctx, hipStream_t s, const SlotDesc PMP_CONST* sl, const BatchHdr PMP_CONST* hd,
                       const QueueRun& r) {
    const unsigned n = (unsigned)grid_blocks(ctx);
    if (r.init_own == 16) launch_init_own<kScore, 16>(s, dim3(n / 8), sl, hd, r.zero);
    else if (r.init_own == 32) launch_init_own<kScore, 32>(s, dim3(n / 4), sl, hd, r.zero);
    else if (r.init_own == 0) launch_init_own<kScore, 0>(s, dim3(n), sl, hd, r.zero);
    else launch_init_own<kScore, 64>(s, dim3(n), sl, hd, r.zero);
    PMP_HIP(ctx, hipGetLastError());
    return PMP_OK;
}

int q_init(pmp_ctx* ctx, hipStream_t s, DescSet& d, const QueueRun& r) {
    PMP_QPTRS
    return launch_init<false>(ctx, s, sl, hd, r);
}

int q_score(pmp_ctx* ctx, hipStream_t s, DescSet& d, const QueueRun& r) {
    PMP_QPTRS
    return launch_init<true>(ctx, s, sl, hd, r);
}

// One launch over passes [first, first + passes), with the heads of launch `launch`.
static int launch_prop(pmp_ctx* ctx, hipStream_t s, DescSet& d, const QueueRun& r, int launch, int first, int passes) {
    PMP_QPTRS
    unsigned int* heads = d.d_heads + (size_t)launch * kFirstWords;
    unsigned long long* counters = ctx->counters;
    int bands = r.bands;
    void* args[] = {(void*)&sl, (void*)&hd, &first, &passes, &heads, &counters, &bands};
    const PropKernel kern = prop_kernel(r.zero, r.form, r.rows);
    PMP_HIP(ctx, hipLaunchKernel(kern.fn, dim3((unsigned)r.blocks), dim3((unsigned)kern.threads), args, 0, s));
    return PMP_OK;
}

int q_prop(pmp_ctx* ctx, hipStream_t s, DescSet& d, const QueueRun& r, int passes) {
    if (r.fused) return passes > 0 ? launch_prop(ctx, s, d, r, 0, 0, passes) : PMP_OK;
    int rc = PMP_OK;
    for (int p = 0; p < passes && !rc; ++p) rc = launch_prop(ctx, s, d, r, p, p, 1);
    return rc;
}

int q_finalize(pmp_ctx* ctx, hipStream_t s, DescSet& d, const QueueRun& r) {
    PMP_QPTRS
    const dim3 grd((unsigned)grid_blocks(ctx)), blk(256);
    hipLaunchKernelGGL(k_copyback_q, grd, blk, 0, s, sl, hd);
    if (r.post) {
        hipLaunchKernelGGL(k_median_q, grd, blk, 0, s, sl, hd, 0);
        hipLaunchKernelGGL(k_median_q, grd, blk, 0, s, sl, hd, 1);
        hipLaunchKernelGGL(k_postfilter_q, grd, blk, 0, s, sl, hd);
    }
    PMP_HIP(ctx, hipGetLastError());
    return PMP_OK;
}

int q_fill_u32(pmp_ctx* ctx, hipStream_t s, unsigned int* p, size_t n, unsigned int v) {
    for (size_t off = 0; off < n; off += (size_t)1 << 30) {
        const size_t m = (n - off) < ((size_t)1 << 30) ? (n - off) : ((size_t)1 << 30);
        hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, p + off, (int)m, v);
    }
    PMP_HIP(ctx, hipGetLastError());
    return PMP_OK;
}

int epochs_arm(pmp_ctx* ctx, hipStream_t s, int n, SlotDesc* slots, const int* tiles, int pass0) {
    if (!ctx->epoch_mode) return PMP_OK;
    size_t need = 0;
    for (int k = 0; k < n; ++k) need += (size_t)tiles[k] + 1;
    if (need > ctx->epochs_cap) {
        if (ctx->epochs) (void)hipFree(ctx->epochs);
        ctx->epochs = nullptr;
        ctx->epochs_cap = 0;
        PMP_HIP(ctx, hipMalloc(&ctx->epochs, need * sizeof(unsigned int)));
        ctx->epochs_cap = need;
    }
    // fill kernels on the stream, ahead of the (possibly graph-replayed) passes
    size_t off = 0;
    int rc;
    for (int k = 0; k < n; ++k) {
        unsigned int* seg = ctx->epochs + off;
        if ((rc = q_fill_u32(ctx, s, seg, (size_t)tiles[k], (unsigned int)pass0))) return rc;
        if ((rc = q_fill_u32(ctx, s, seg + tiles[k], 1, 0u))) return rc;
        if (k == 0 && ctx->epoch_mode == 2 && (rc = q_fill_u32(ctx, s, seg, 1, (unsigned int)pass0 + 1u))) return rc;
        slots[k].epochs = seg;
        off += (size_t)tiles[k] + 1;
    }
    ctx->epoch_tiles.assign(tiles, tiles + n);
    ctx->epoch_words = need;
    return PMP_OK;
}

static int q_sequence(pmp_ctx* ctx, hipStream_t s, DescSet& d, const QueueRun& r, int passes) {
    int rc;
    if ((rc = q_clear(ctx, s, d, r, passes))) return rc;
    int tp = timing_begin(ctx, kStageInit);
    if ((rc = q_init(ctx, s, d, r))) return rc;
    timing_end(ctx, tp);
    if (passes > 0) {
        tp = timing_begin(ctx, kStagePropagate, passes);
        if ((rc = q_prop(ctx, s, d, r, passes))) return rc;
        timing_end(ctx, tp);
    }
    tp = timing_begin(ctx, kStageFinalize);
    rc = q_finalize(ctx, s, d, r);
    timing_end(ctx, tp);
    return rc;
}

int q_densify(pmp_ctx* ctx, hipStream_t s, DescSet& d, const QueueRun& r, int passes, bool use_graph) {
    // per-stage timing needs events between the launches: no graph then
    if (!use_graph || ctx->timing) return q_sequence(ctx, s, d, r, passes);
    const GraphKey key{passes, (r.zero ? 1 : 0) + 2 * r.form, r.rows, r.blocks, r.bands, (r.post ? 1 : 0) + (r.fused ? 2 : 0) + 4 * r.init_own};
    auto it = d.graphs.find(key);
    if (it == d.graphs.end()) {
        hipGraph_t g = nullptr;
        hipGraphExec_t ge = nullptr;
        PMP_HIP(ctx, hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        int rc = q_sequence(ctx, s, d, r, passes);
        hipError_t e = hipStreamEndCapture(s, &g);
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (e != hipSuccess) return check_hip(ctx, e, "hipStreamEndCapture");
        e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
        if (e != hipSuccess) {
            (void)hipGraphDestroy(g);
            return check_hip(ctx, e, "hipGraphInstantiate");
        }
        it = d.graphs.emplace(key, std::make_pair(g, ge)).first;
    }
    PMP_HIP(ctx, hipGraphLaunch(it->second.second, s));
    return PMP_OK;
}

// ---------------------------------------------------------------- batched form

// Descriptors, propagation shape (r) and work lists for n keyframes (all from
// pass 0), uploaded to the batch set.
// arm: pass epochs for this batch (pmp_batch_densify; the autotuner reruns
// passes from the same maps and does not arm them)
static int batch_prepare(pmp_ctx* ctx, QueueState* q, const pmp_params* params, int n, const pmp_keyframe* kfs,
                         const pmp_batch_config& c, QueueRun& r, bool arm) {
    int rc = check_params(ctx, params);
    if (rc) return rc;
    if (params->iterations > kMaxPasses / 2) return set_error(ctx, PMP_EINVAL, "iterations must be <= 64");
    // the slots' maps may be reallocated and the staging copy rewritten
    PMP_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if ((rc = desc_begin(ctx, q->batch))) return rc;
    if (!ctx->counters) {
        PMP_HIP(ctx, hipMalloc(&ctx->counters, 4 * sizeof(unsigned long long)));
        PMP_HIP(ctx, hipMemsetAsync(ctx->counters, 0, 4 * sizeof(unsigned long long), ctx->stream));
    }
    int it_init[kMaxSlots], it_prop[kMaxSlots], it_rows[kMaxSlots];
    for (int k = 0; k < n; ++k) {
        auto ir = ctx->images.find(kfs[k].ref_id);
        if (ir == ctx->images.end()) return set_error(ctx, PMP_ENOTFOUND, "unknown reference image id");
        if ((rc = ensure_slot(ctx, q->bufs[k], ir->second.W, ir->second.H))) return rc;
        int items[2];
        rc = slot_fill(ctx, params, kfs[k], q->bufs[k], nullptr, 0, ctx->stream, q->batch.h_slots[k], items);
        if (rc) return rc;
        it_init[k] = items[0];
        it_rows[k] = items[1];
    }
    prop_shape(*q, c, n, nullptr, q->batch.h_slots, false, r);
    for (int k = 0; k < n; ++k) it_prop[k] = slot_tiles(q->batch.h_slots[k], r.rows);
    fill_list(q->batch.h_hdr->init, n, it_init);
    fill_list(q->batch.h_hdr->prop, n, it_prop);
    fill_list(q->batch.h_hdr->rows, n, it_rows);
    if ((rc = ensure_sync(ctx, q->batch, (size_t)q->batch.h_hdr->prop.total))) return rc;
    if (arm && (rc = epochs_arm(ctx, ctx->stream, n, q->batch.h_slots, it_prop, 0))) return rc;
    return desc_upload(ctx, q->batch, n, ctx->stream);
}

}  // namespace pmp

using namespace pmp;

extern "C" {

int pmp_batch_densify(pmp_ctx* ctx, const pmp_params* params, int32_t n, const pmp_keyframe* kfs) {
    TraceRange trace_range("pmp_batch_densify");
    if (!ctx || !params || !kfs) return PMP_EINVAL;
    if (n < 1 || n > kMaxSlots) return set_error(ctx, PMP_EINVAL, "batch size must be in [1, PMP_MAX_BATCH]");
    PMP_ON_DEVICE(ctx);
    QueueState* q = nullptr;
    int rc = queue_state(ctx, q);
    if (rc) return rc;
    q->n_last = 0;
    QueueRun r;
    if ((rc = batch_prepare(ctx, q, params, n, kfs, q->cfg, r, true))) return rc;
    if ((rc = queue_run(ctx, *q, q->cfg, params->edge_mode == PMP_EDGE_ZERO, params->postprocess != 0,
                        *q->batch.h_hdr, q->batch.h_slots, r)))
        return rc;
    q->last = r;
    if ((rc = q_densify(ctx, ctx->stream, q->batch, r, 2 * params->iterations, q->cfg.use_graph != 0))) return rc;
    q->n_last = n;
    ctx->densify_calls += n;
    return PMP_OK;
}

int pmp_batch_get_maps(pmp_ctx* ctx, int32_t k, float* plane4, float* depth, float* score, int32_t* nghbr) {
    if (!ctx) return PMP_EINVAL;
    PMP_ON_DEVICE(ctx);
    QueueState* q = ctx->queue;
    if (!q || k < 0 || k >= q->n_last) return set_error(ctx, PMP_EINVAL, "no such keyframe in the last batch");
    const SlotBuf& b = q->bufs[k];
    const size_t P = (size_t)b.W * b.H;
    HostCopy c[4];
    int n = 0;
    if (plane4) c[n++] = flat_copy(plane4, b.oplane, P * 16);
    if (depth) c[n++] = flat_copy(depth, b.odepth, P * 4);
    if (score) c[n++] = flat_copy(score, b.oscore, P * 4);
    if (nghbr) c[n++] = flat_copy(nghbr, b.onghbr, P * 4);
    return copy_to_host(ctx, c, n);
}

int pmp_batch_set_config(pmp_ctx* ctx, const pmp_batch_config* cfg) {
    if (!ctx || !cfg) return PMP_EINVAL;
    PMP_ON_DEVICE(ctx);
    int rc = check_config(ctx, *cfg);
    if (rc) return rc;
    QueueState* q = nullptr;
    if ((rc = queue_state(ctx, q))) return rc;
    q->cfg = *cfg;
    return PMP_OK;
}

int pmp_batch_get_config(pmp_ctx* ctx, pmp_batch_config* cfg) {
    if (!ctx || !cfg) return PMP_EINVAL;
    PMP_ON_DEVICE(ctx);
    QueueState* q = nullptr;
    int rc = queue_state(ctx, q);
    if (rc) return rc;
    *cfg = q->cfg;
    return PMP_OK;
}

int pmp_batch_autotune(pmp_ctx* ctx, const pmp_params* params, int32_t n, const pmp_keyframe* kfs,
                       pmp_batch_config* best) {
    TraceRange trace_range("pmp_batch_autotune");
    if (!ctx || !params || !kfs) return PMP_EINVAL;
    if (n < 1 || n > kMaxSlots) return set_error(ctx, PMP_EINVAL, "batch size must be in [1, PMP_MAX_BATCH]");
    PMP_ON_DEVICE(ctx);
    QueueState* q = nullptr;
    int rc = queue_state(ctx, q);
    if (rc) return rc;
    q->n_last = 0;
    hipEvent_t e0, e1;
    PMP_HIP(ctx, hipEventCreate(&e0));
    PMP_HIP(ctx, hipEventCreate(&e1));
    pmp_batch_config found = q->cfg;
    float best_ms = 3.0e38f;
    const int rows_set[3] = {2, 4, 8};
    const bool zero = params->edge_mode == PMP_EDGE_ZERO;
    for (int ri = 0; ri < 3 && rc == 0; ++ri) {
        pmp_batch_config c = q->cfg;
        c.tile_rows = rows_set[ri];
        c.blocks_per_cu = 32;
        QueueRun r;
        if ((rc = batch_prepare(ctx, q, params, n, kfs, c, r, false))) break;
        if ((rc = queue_run(ctx, *q, c, zero, false, *q->batch.h_hdr, q->batch.h_slots, r))) break;
        const int occ = r.blocks / (q->cus > 0 ? q->cus : 1);   // blocks per CU that fit (rounding aside)
        // at least 8 waves per CU: fewer leave SIMDs idle and measured 1.3-4x
        // slower, and their trials are the longest
        const int waves = prop_kernel(zero, r.form, r.rows).threads / 64;   // of a block
        const int bpc_min = std::min(occ, (8 + waves - 1) / waves);
        for (int bpc = bpc_min; bpc <= occ && rc == 0; ++bpc) {
            for (int bands = 0; bands <= 1 && rc == 0; ++bands) {
                c.blocks_per_cu = bpc;
                c.xcd_bands = bands;
                if ((rc = queue_run(ctx, *q, c, zero, false, *q->batch.h_hdr, q->batch.h_slots, r))) break;
                // same starting maps for every candidate: init, then time every
                // pass.  The first passes score random planes (most candidates
                // survive pre-rejection, the gathers scatter); the converged
                // ones pre-reject most candidates and are instruction-bound.
                // The shapes rank differently on the two kinds, so a prefix of
                // passes misranks them.
                const int timed = 2 * params->iterations;
                if ((rc = q_clear(ctx, ctx->stream, q->batch, r, timed))) break;
                if ((rc = q_init(ctx, ctx->stream, q->batch, r))) break;
                hipError_t e = hipEventRecord(e0, ctx->stream);
                if (e == hipSuccess) rc = q_prop(ctx, ctx->stream, q->batch, r, timed);
                if (e == hipSuccess && rc == 0) e = hipEventRecord(e1, ctx->stream);
                if (e == hipSuccess && rc == 0) e = hipEventSynchronize(e1);
                float ms = 0.0f;
                if (e == hipSuccess && rc == 0) e = hipEventElapsedTime(&ms, e0, e1);
                if (e != hipSuccess) rc = check_hip(ctx, e, "autotune timing");
                if (rc) break;
                if (ms < best_ms) {
                    best_ms = ms;
                    found = c;
                }
            }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    q->cfg = found;
    if (best) *best = found;
    return PMP_OK;
}

}  // extern "C"
