// pmp_tile.h -- per-tile and per-pixel device code shared by the one-keyframe
// kernels (pmp_estimator.hip) and the work-queue kernels over many keyframes
// (pmp_batch.hip).
#pragma once
#include <type_traits>

#include "pmp_internal.h"
#include "pmp_math.h"
#include "pmp_score.h"

namespace pmp {

// Colour-weight table into LDS; every thread of the (1-D) block takes part.
__device__ __forceinline__ void load_wc(const float* wc, float* sWc) {
    for (int k = threadIdx.x; k < 256; k += blockDim.x) sWc[k] = wc[k];
    __syncthreads();
}

__device__ __forceinline__ void count_add(unsigned long long* ctr, unsigned int v) {
    // one atomic per wave (all 64 lanes active; per-lane counts are < 2^16)
    unsigned int s = v;
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if ((threadIdx.x & 63) == 0 && s) atomicAdd(ctr, (unsigned long long)s);
}

// The same for a count that is the wave's, not the lane's.
__device__ __forceinline__ void count_add_wave(unsigned long long* ctr, unsigned int v) {
    if ((threadIdx.x & 63) == 0 && v) atomicAdd(ctr, (unsigned long long)v);
}

// A keyframe's tap walk (quad_tap) into LDS; every thread of the block takes part.
__device__ __forceinline__ void load_walk(const KfArgs& a, QuadTap* tab) {
    const int n = (a.T + 3) / 4 * 4;
    for (int k = threadIdx.x; k < n; k += blockDim.x) tab[k] = quad_tap(a, k);
    __syncthreads();
}

// ---- red-black pass
// A tile is 2R rows x 32 same-colour pixels (64 columns); its pixel t < 64R is
// at row i = 2R by + t / 32, column j = 2 (32 bx + t % 32) + ((i + colour) & 1),
// i.e. every pixel of colour (i+j)&1 == colour once.  A thread owns one pixel
// (kWide: a quarter of a wave's threads do) and decides for it.  Candidates are at odd
// distance (1 or 3), so they have the other colour and are not written by
// this pass.
//
// Propagation candidates are scored by whichever waves of the block are
// free, in packed sweeps, and their raw scores handed back to the owning
// threads, which apply the penalty and the acceptance test in candidate order:
//   1. every pixel tests its 8 candidates against its state at entry (the
//      exact pre-rejection below); the (candidate, pixel) pairs that pass are
//      listed candidate-major and scored in one sweep over the block's waves;
//   2. each pixel then walks its candidates in order against its running state
//      (the test is repeated: an acceptance changes the plane and the score it
//      is tested against).  A candidate that passes there but did not pass at
//      entry has no score yet: the pixel stops and lists every later candidate
//      that can still pass at all (1 - f_d above its current score: the plane
//      factor is at most 1 and the score only grows), and a second sweep scores
//      those of all such pixels before the walks go on.  After it no walk
//      stops again, so a tile takes at most two sweeps.
// A candidate's raw score depends only on its plane and the pixel, so where
// and when it is computed does not matter: each pixel's sequence of decisions
// is that of a loop over its own candidates, and the results are identical.
// Scores computed for candidates that an acceptance makes unnecessary are
// spent work (counted as evaluations).
// srow/scol/sref: the tile's rows and columns of the bearing tables and of
// the reference image, with the patch halo (LdsTaps).
// pl: the other colour's planes of the tile and 3 pixels around it, where its
// candidates are (cand_plane).
// walk: the keyframe's tap walk; eval: each wave's exchange area; rs, ic: the
// pixels' reference moments.
// res[c * 64R + t]: raw score of candidate c of pixel t; job: the sweep's
// (candidate << 9 | pixel) list.
constexpr int kPlaneCols = kTileSame + 3;   // one colour's pixels in a row of the tile and 3 columns each side
// How a propagation block evaluates planes: kLane one per lane, 64 to a wave;
// kQuad one per four lanes; kWide as kQuad with four times the waves to a tile
// (chosen by prop_shape).
enum PropForm { kLane = 0, kQuad = 1, kWide = 2 };
struct LaneShared {
    float sv[kMaxViews][64];
};
template <int R, int F>
struct PropShared {
    static constexpr int kPix = 64 * R;              // pixels of a tile
    static constexpr int kOwn = F == kWide ? 16 : 64;   // of them, a wave's own
    static constexpr int kWaves = kPix / kOwn;
    static constexpr int kRows = kPix / kTileSame;   // tile rows
    QuadTap walk[F == kLane ? 1 : kQuadTaps];
    std::conditional_t<F == kLane, LaneShared, QuadShared> eval[kWaves];
    float4 rs[kPix];
    union {
        float4 pl[(kRows + 6) * kPlaneCols];
        struct {                      // a refinement trial: its planes and their scores
            float4 trial[kPix];
            float trial_score[kPix];
        };
    };
    float2 srow[kRows + 2 * kMaxHalf];
    float2 scol[kTileCols];
    float sWc[256];
    union {
        struct {
            float res[8 * kPix];
            uint16_t job[8 * kPix];
        };
        float z[12 * kPix];           // normals of four refinement trials per pixel
    };
    float ic[kPix];
    int cnt[8 * kWaves];
    int item, pass;
    uint8_t sref[(kRows + 2 * kMaxHalf) * kTileCols];
};

// The maps that tiles of one launch hand each other (pass fusion: a tile of
// pass p + 1 runs beside tiles of pass p) go through agent-scope accesses:
// the XCDs' L2 caches are not coherent with each other for plain ones within
// a launch.  The taking of a tile orders them (take_tile, release_tiles).
__device__ __forceinline__ float load_map(const float* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_map(float* p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float4 load_map4(const float4* p) {
    const unsigned long long* q = (const unsigned long long*)p;
    const unsigned long long a = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long b = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return make_float4(u2f((uint32_t)a), u2f((uint32_t)(a >> 32)), u2f((uint32_t)b), u2f((uint32_t)(b >> 32)));
}
__device__ __forceinline__ void store_map4(float4* p, float4 v) {
    unsigned long long* q = (unsigned long long*)p;
    __hip_atomic_store(q, (unsigned long long)f2u(v.x) | ((unsigned long long)f2u(v.y) << 32), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(q + 1, (unsigned long long)f2u(v.z) | ((unsigned long long)f2u(v.w) << 32), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// Offset (di, dj) of propagation candidate c: (0,+1) (+1,0) (0,-1) (-1,0)
// (0,+3) (+3,0) (0,-3) (-3,0) (PatchMatchCuda.cu:305)
__device__ __forceinline__ void cand_offset(int c, int& di, int& dj) {
    const int dist = (c < 4) ? 1 : 3, dir = c & 3;
    di = (dir == 1) ? dist : (dir == 3) ? -dist : 0;
    dj = (dir == 0) ? dist : (dir == 2) ? -dist : 0;
}

// 1 - f_d of candidate plane pn: the largest penalty factor it can have for a
// pixel with bearing b and entry depth d0 (PatchMatchCuda.cu:323-326), whatever
// the running plane.
__device__ __forceinline__ float cand_bound(const KfArgs& a, float4 pn, float bx, float by, float bz, float d0,
                                           float inv_d0) {
    const float s = fma_(pn.z, bz, fma_(pn.y, by, pn.x * bx));
    const float dn = rcp_pos(clampf(abs_(s), 1e-6f, 1e30f));
    const float rel = (d0 - dn) * inv_d0;
    const float fd = exp_((rel * rel) * -a.depth_penalty);
    return 1.0f - fd;
}

// Penalty and acceptance precondition of candidate plane pn for a pixel with
// bearing b, entry depth d0 and running plane h and score sc
// (PatchMatchCuda.cu:323-332).  acosf(prod/norm) is NaN, i.e. the candidate
// is rejected, unless |prod| <= norm; |score| <= 1, so the penalised score
// cannot exceed f, and f <= sc rejects it before it is scored.
__device__ __forceinline__ bool cand_test(const KfArgs& a, float4 pn, float bx, float by, float bz, float d0,
                                          float inv_d0, float h0, float h1, float h2, float sc, float& f) {
    const float gd = cand_bound(a, pn, bx, by, bz, d0, inv_d0);
    const float prod = fma_(h2, pn.z, fma_(h1, pn.y, h0 * pn.x));
    const float ex = h0 - pn.x, ey = h1 - pn.y, ez = h2 - pn.z;
    const float nrm = sqrt_(fma_(ez, ez, fma_(ey, ey, ex * ex)));
    f = 0.0f;
    if (nrm > 0.0f && abs_(prod) <= nrm) {
        const float ratio = clampf(prod * rcp_pos(clampf(nrm, 1e-30f, 1e30f)), -1.0f, 1.0f);
        const float ac = acos_(ratio);
        const float fp = exp_((ac * ac) * -a.plane_penalty);
        f = gd * (1.0f - fp);
        return f > sc;
    }
    return false;
}

// A propagation tile is TR = 64 R / kTileSame rows by 2 kTileSame columns
// (kTileSame same-colour pixels per row; each wave covers 64 / kTileSame
// rows).  Taller, narrower tiles than one row per wave shrink the views' cache
// footprint of a tile's patches.  stage_tile copies the rows
// [tby TR - half, tby TR + TR + half) and columns [2 kTileSame tbx - half,
// 2 kTileSame (tbx + 1) + half) of the reference image and of the bearing
// tables into sh (coordinates outside the image are clamped; only interior
// pixels, whose taps lie inside the image, read them), and the other colour's
// planes of the tile and 3 pixels around it (0 outside the image, where no
// interior pixel's candidate lies).  Waits for the previous tile's readers
// first.
template <int R, int F>
__device__ __forceinline__ LdsTaps stage_tile(const KfArgs& a, PropShared<R, F>& sh, const float4* plane, int colour,
                                              int tbx, int tby) {
    constexpr int NT = 64 * PropShared<R, F>::kWaves;
    constexpr int TR = PropShared<R, F>::kRows;
    const int r0 = tby * TR - a.half, c0 = 2 * kTileSame * tbx - a.half;
    const int nr = TR + 2 * a.half, nc = 2 * kTileSame + 2 * a.half;
    __syncthreads();
    const int pr0 = tby * TR - 3, pc0 = 2 * kTileSame * tbx - 3;
    for (int e = threadIdx.x; e < (TR + 6) * kPlaneCols; e += NT) {
        const int r = e / kPlaneCols, q = e - r * kPlaneCols;
        const int y = pr0 + r, x = pc0 + 2 * q + ((y + pc0 + colour + 1) & 1);
        const bool in = y >= 0 && y < a.H && x >= 0 && x < a.W;
        sh.pl[e] = in ? load_map4(&plane[(size_t)y * a.W + x]) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    for (int e = threadIdx.x; e < nc; e += NT) {
        const int x = min(max(c0 + e, 0), a.W - 1);
        sh.scol[e] = a.coltab[x];
    }
    for (int e = threadIdx.x; e < nr; e += NT) {
        const int y = min(max(r0 + e, 0), a.H - 1);
        sh.srow[e] = a.rowtab[y];
    }
    for (int e = threadIdx.x; e < nr * nc; e += NT) {
        const int r = e / nc, c = e - r * nc;
        const int y = min(max(r0 + r, 0), a.H - 1), x = min(max(c0 + c, 0), a.W - 1);
        sh.sref[r * kTileCols + c] = a.ref[(size_t)y * a.W + x];
    }
    __syncthreads();
    return LdsTaps{sh.srow, sh.scol, sh.sref, r0, c0};
}

// The staged plane of candidate c of the tile's pixel t.
template <int R, int F>
__device__ __forceinline__ float4 cand_plane(const PropShared<R, F>& sh, int t, int colour, int tby, int c) {
    int di, dj;
    cand_offset(c, di, dj);
    const int row = t / kTileSame;
    const int col = 2 * (t % kTileSame) + ((tby * PropShared<R, F>::kRows + row + colour) & 1);
    return sh.pl[(row + di + 3) * kPlaneCols + ((col + dj + 3) >> 1)];
}

// One tile of one red-black pass by a block whose waves own PW pixels each
// (pixel t = PW wave + lane, lanes beyond PW own none but take part in the
// evaluations).  sh.sWc and sh.walk hold the keyframe's tables; rot is the wave
// that takes the first packed jobs.
template <bool kZero, int R, int F>
__device__ __forceinline__ void propagate_tile(const KfArgs& a, PropShared<R, F>& sh, float4* __restrict__ plane,
                                               float* __restrict__ depth, float* __restrict__ score, int it,
                                               int colour, int tbx, int tby, int rot, unsigned int& n_eval,
                                               unsigned int& n_cand) {
    using Sh = PropShared<R, F>;
    constexpr int NP = Sh::kPix, NW = Sh::kWaves, TR = Sh::kRows, PW = Sh::kOwn;
    constexpr int NJ = F == kLane ? 64 : 16;   // planes a wave scores at a time
    const float* sWc = sh.sWc;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const bool owner = PW == 64 || lane < PW;
    const int t = PW * wave + (owner ? lane : 0);
    const int i = tby * TR + t / kTileSame;
    const int j = 2 * (tbx * kTileSame + t % kTileSame) + ((i + colour) & 1);
    const bool active = owner && i < a.H && j < a.W && in_prop_grid(a, i, j);
    const size_t k = active ? (size_t)i * a.W + j : 0;
    // row and column of pixel p in the tile copies
    auto at = [&](int p, int& row, int& col) {
        const int y = p / kTileSame;
        row = y + a.half;
        col = 2 * (p % kTileSame) + ((tby * TR + y + colour) & 1) + a.half;
    };

    const LdsTaps tp = stage_tile(a, sh, plane, colour, tbx, tby);
    auto evaluate = [&](const auto& job, const auto& put, unsigned long long live) {
        if constexpr (F == kLane)
            score_lanes<kZero>(a, tp, sWc, sh.rs, sh.ic, at, job, put, live, &sh.eval[wave].sv[0][0]);
        else
            score_wave<kZero>(a, tp, sh.walk, sWc, sh.rs, sh.ic, at, job, put, live, sh.eval[wave]);
    };
    float sc = 0.0f, h0 = 0.0f, h1 = 0.0f, h2 = 0.0f, bx = 0.0f, by = 0.0f, bz = 0.0f, d0 = 1.0f, inv_d0 = 1.0f;
    {
        RefStat rs = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        if (active) {
            sc = load_map(&score[k]);
            const float4 pk = load_map4(&plane[k]);
            d0 = load_map(&depth[k]);
            rs = ref_stats(a, tp, sWc, i, j);
            h0 = pk.x; h1 = pk.y; h2 = pk.z;
            tap_bearing(tp, i, j, bx, by, bz);
            inv_d0 = rcp(d0);
        }
        if (owner) {
            sh.rs[t] = make_float4(rs.mx, rs.inv, rs.mxc, rs.vx);
            sh.ic[t] = rs.Ic;
        }
    }

    // 1. propagation (PatchMatchCuda.cu:311-338), in the order of cand_offset
    unsigned int want = 0;     // bit c: candidate c is to be scored in the next sweep
    const unsigned long long alive = __ballot(active);
    n_cand += (unsigned int)__popcll(alive) * (8u + (unsigned int)a.n_refine);
    if (active) {
#pragma unroll 1
        for (int c = 0; c < 8; ++c) {
            const float4 pn = cand_plane(sh, t, colour, tby, c);
            float f;
            if (cand_test(a, pn, bx, by, bz, d0, inv_d0, h0, h1, h2, sc, f)) want |= 1u << c;
        }
    }
    unsigned int listed = want;   // bit c: candidate c has a score (or will after the sweep)
    int cpos = 0;                 // the next candidate of this pixel's walk
#pragma unroll 1
    for (;;) {
        // the sweep's list, candidate-major: per (candidate, wave) counts, then offsets
#pragma unroll 1
        for (int c = 0; c < 8; ++c) {
            const unsigned long long bal = __ballot((want >> c) & 1u);
            if (lane == 0) sh.cnt[c * NW + wave] = __popcll(bal);
        }
        __syncthreads();
        int J = 0;
#pragma unroll 1
        for (int c = 0; c < 8; ++c) {
            int woff = 0, tot = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const int cw = sh.cnt[c * NW + w];
                woff += (w < wave) ? cw : 0;
                tot += cw;
            }
            const bool on = (want >> c) & 1u;
            const unsigned long long bal = __ballot(on);
            if (on) sh.job[J + woff + __popcll(bal & ((1ull << lane) - 1ull))] = (uint16_t)((c << 9) | t);
            J += tot;
        }
        J = __builtin_amdgcn_readfirstlane(J);
        if (J == 0) break;   // the same in every thread
        __syncthreads();
        // score the list: NJ jobs per wave and turn, from wave rot on
#pragma unroll 1
        for (int g0 = NJ * ((wave - rot) & (NW - 1)); g0 < J; g0 += NJ * NW) {
            const int n = min(J - g0, NJ);
            auto job = [&](int l, int& jt, float& px, float& py, float& pz) {
                const unsigned int e = sh.job[g0 + (l < n ? l : 0)];
                jt = (int)(e & 511u);
                const float4 pn = cand_plane(sh, jt, colour, tby, (int)(e >> 9));
                px = pn.x; py = pn.y; pz = pn.z;
            };
            auto put = [&](int l, float s) {
                const unsigned int e = sh.job[g0 + l];
                sh.res[(e >> 9) * NP + (e & 511u)] = s;
            };
            evaluate(job, put, ~0ull >> (64 - n));
            n_eval += n;
        }
        __syncthreads();
        // walk the candidates in order against the running state, up to the
        // first one that passes but has no score
        want = 0;
        if (active) {
            while (cpos < 8) {
                const float4 pn = cand_plane(sh, t, colour, tby, cpos);
                float f;
                if (cand_test(a, pn, bx, by, bz, d0, inv_d0, h0, h1, h2, sc, f)) {
                    if (!((listed >> cpos) & 1u)) break;
                    const float sh_ = sh.res[cpos * NP + t] * f;
                    if (sh_ > sc) { h0 = pn.x; h1 = pn.y; h2 = pn.z; sc = sh_; }
                }
                ++cpos;
            }
            if (cpos < 8) {
                // stopped: list this and every later unscored candidate that can still pass
#pragma unroll 1
                for (int c = cpos; c < 8; ++c) {
                    if ((listed >> c) & 1u) continue;
                    const float4 pn = cand_plane(sh, t, colour, tby, c);
                    if (c == cpos || cand_bound(a, pn, bx, by, bz, d0, inv_d0) > sc) want |= 1u << c;
                }
                listed |= want;
            }
        }
    }
    // 2. refinement (PatchMatchCuda.cu:340-395); its normals and planes lie where
    // the sweeps' scores, lists and planes were, which the other waves may
    // still read
    __syncthreads();
    float dcur = 1.0f, c0 = 0.0f, c1 = 0.0f, c2 = 0.0f;
    if (active) {
        dcur = depth_of_plane(bx, by, bz, h0, h1, h2);
        c0 = h0; c1 = h1; c2 = h2;
    }
#pragma unroll 1
    for (int n = 0; n < a.n_refine; ++n) {
        // the normals of four trials at a time, in the pixel's own LDS column
        if ((n & 3) == 0 && owner) {
#pragma unroll 1
            for (int b = 0; b < 3; ++b) {
                float z0, z1, z2, z3;
                refine_block(a, (uint32_t)(i * a.W + j), it, 3 * (n >> 2) + b, z0, z1, z2, z3);
                float* zt = &sh.z[4 * b * NP + t];
                zt[0] = z0; zt[NP] = z1; zt[2 * NP] = z2; zt[3 * NP] = z3;
            }
        }
        const float* zt = &sh.z[3 * (n & 3) * NP + t];
        const float ra = zt[0], rb = zt[NP], rc = zt[2 * NP];
        const float dh = dcur * exp_(a.dr[n] * ra);
        const float nx = fma_(a.nr[n], ra, c0);
        const float ny = fma_(a.nr[n], rb, c1);
        const float nz = fma_(a.nr[n], rc, c2);
        float q0, q1, q2;
        tap_bearing(tp, i, j, bx, by, bz);
        plane_from_depth_normal(bx, by, bz, dh, nx, ny, nz, q0, q1, q2);
        if (owner) sh.trial[t] = make_float4(q0, q1, q2, dh);
        wave_exchange();
        auto job = [&](int l, int& jt, float& px, float& py, float& pz) {
            jt = PW * wave + l;
            const float4 pn = sh.trial[jt];
            px = pn.x; py = pn.y; pz = pn.z;
        };
        auto put = [&](int l, float s) { sh.trial_score[PW * wave + l] = s; };
        evaluate(job, put, alive);
        n_eval += (unsigned int)__popcll(alive);
        if (active && sh.trial_score[t] > sc) {
            const float4 pn = sh.trial[t];
            c0 = pn.x; c1 = pn.y; c2 = pn.z; dcur = pn.w;
            sc = sh.trial_score[t];
        }
        wave_exchange();
    }
    tap_bearing(tp, i, j, bx, by, bz);
    if (active) {
        store_map(&score[k], sc);
        store_map4(&plane[k], make_float4(c0, c1, c2, 0.0f));
        store_map(&depth[k], depth_of_plane(bx, by, bz, c0, c1, c2));
    }
}

// ---- finalize
// Copy-back of ComputePatchMatch: masked pixels keep the AssignMatrices values
// (depth 0, plane 0, score -1, nghbr 0); unmasked pixels take the maps after
// RandomInitialization (depthmap.cc:673-687) unless they are inside the window
// [ps-2, dim-ps-2) (depthmap.cc:731-732), where they take the final maps, or
// 0 when the patch variance is below min_patch_sd^2 (depthmap.cc:739-743).
__device__ __forceinline__ void copyback_pixel(const KfArgs& a, const uint8_t* __restrict__ mask,
                                               const float4* __restrict__ ip, const float* __restrict__ id,
                                               const float* __restrict__ is, const float4* __restrict__ fp,
                                               const float* __restrict__ fd, const float* __restrict__ fs,
                                               float4* __restrict__ op, float* __restrict__ od,
                                               float* __restrict__ os, int32_t* __restrict__ on, float min_var,
                                               float inv_T, int i, int j) {
    const int W = a.W, H = a.H;
    const size_t k = (size_t)i * W + j;
    const int ps = a.half + 2;
    const int lo = ps - 2, hi_r = H - ps - 2, hi_c = W - ps - 2;
    float4 pl = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float dep = 0.0f, sc = -1.0f;
    int ng = 0;
    if (mask == nullptr || mask[k]) {
        if (i >= lo && i < hi_r && j >= lo && j < hi_c) {
            bool low = false;
            if (min_var > 0.0f) {
                float sum = 0.0f;
                for (int k1 = -a.half; k1 <= a.half; k1 += a.stride)
                    for (int k2 = -a.half; k2 <= a.half; k2 += a.stride)
                        sum = sum + (float)a.ref[(size_t)(i + k1) * W + (j + k2)];
                const float mean = sum * inv_T;
                float s2 = 0.0f;
                for (int k1 = -a.half; k1 <= a.half; k1 += a.stride)
                    for (int k2 = -a.half; k2 <= a.half; k2 += a.stride) {
                        float e = (float)a.ref[(size_t)(i + k1) * W + (j + k2)] - mean;
                        s2 = fma_(e, e, s2);
                    }
                low = (s2 * inv_T) < min_var;
            }
            if (!low) {
                dep = fd[k]; sc = fs[k];
                const float4 f = fp[k];
                pl = make_float4(f.x, f.y, f.z, 0.0f);
            } else {
                sc = 0.0f;
            }
            ng = 1;
        } else {
            dep = id[k]; sc = is[k];
            const float4 f = ip[k];
            pl = make_float4(f.x, f.y, f.z, 0.0f);
        }
    }
    op[k] = pl; od[k] = dep; os[k] = sc; on[k] = ng;
}

// 3x3 median with replicated border (cv::medianBlur, ksize 3, CV_32F)
__device__ __forceinline__ void median3_pixel(const float* __restrict__ src, float* __restrict__ dst, int W, int H,
                                              int i, int j) {
    float v[9];
    int n = 0;
#pragma unroll
    for (int a = -1; a <= 1; ++a) {
        const int ii = min(max(i + a, 0), H - 1);
#pragma unroll
        for (int b = -1; b <= 1; ++b) {
            const int jj = min(max(j + b, 0), W - 1);
            v[n++] = src[(size_t)ii * W + jj];
        }
    }
    // median of 9 by a fixed exchange network (the value equals any sort's v[4])
#pragma unroll
    for (int p = 0; p <= 4; ++p)
#pragma unroll
        for (int b = p + 1; b < 9; ++b) {
            const float lo = fminf(v[p], v[b]);
            const float hi = fmaxf(v[p], v[b]);
            v[p] = lo;
            v[b] = hi;
        }
    dst[(size_t)i * W + j] = v[4];
}

// PostProcess test (depthmap.cc:1189-1196): the float ratio |d - m| / d against
// the double threshold (fabs of a float is float there, 0.05 a double literal)
__device__ __forceinline__ void postfilter_pixel(const float* __restrict__ med, float* __restrict__ depth,
                                                 float* __restrict__ score, size_t k, double rel_thr,
                                                 float min_depth, float max_depth, float min_score) {
    const float d = depth[k], m = med[k], sc = score[k];
    if (d == 0.0f || (double)(__builtin_fabsf(d - m) / d) > rel_thr || d < min_depth || d > max_depth ||
        sc <= min_score) {
        depth[k] = 0.0f;
        score[k] = -1.0f;
    } else {
        depth[k] = m;
    }
}

}  // namespace pmp
