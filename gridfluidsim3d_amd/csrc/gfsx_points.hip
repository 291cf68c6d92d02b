// gfsx_points.hip -- MAC samples and Runge-Kutta steps of point arrays (the
// ParticleAdvector calls, particleadvector.cpp:209-455) over grid bricks
// staged in LDS, on gfx950.
//
// The points are AoS triples in any order; FluidSimulation shuffles its
// particles every step (fluidsimulation.cpp:3211-3223), so neighbouring
// points rarely share a cell and sampling the grid straight from memory is
// bound by scattered L2 reads (tricubic: 192 taps a sample).  Here the points
// are first gathered by bricks of 8^3 cells, in no particular order inside a
// brick: every output depends on its own point only, so the results are the
// same bits whatever the order (and the same as the direct kernels give).
//
//   1. k_pt_count: per work-group, a histogram of its points' bricks in LDS
//      (one word per brick), added to the global counts with one atomic per
//      brick the work-group met.
//   2. k_pt_scan: brick starts, and the work list: bricks cut into chunks of
//      at most CHUNK points.  Bricks of fewer than SPARSE points are in no
//      chunk; their points lie together behind all others.
//   3. k_pt_place: the histogram again, each point's rank in it kept, one
//      atomic per brick met reserving the work-group's range; the points are
//      written there with their index (16 bytes each).
//   4. k_pt_brick: one work-group per chunk stages the u, v, w boxes and
//      samples them.  A stage that leaves the boxes is sampled from global
//      memory (trilinear), or its point goes to a list (tricubic: 192 loads
//      in the kernel's loop would take its registers).
//   5. k_pt_slow: the listed points and the sparse bricks', sampled from
//      global memory.
//
// Bound: the tricubic brick kernel by LDS reads and VALU (64 taps and 84 FMAs
// a component), the passes around it by memory (12 B read twice, 16 B written
// and read twice, 12 B written per point, scattered where the input is).
// 2.65M shuffled points on 128x97x112, RK4: 4.78 ms (direct) -> 0.34 ms, of
// which the brick kernel 0.26 (0.46 before its points were ordered by cell);
// one sample 1.05 -> 0.16 ms, 84 us of it the brick kernel.

#include "gfsx_internal.h"
#include "gfsx_sample.h"
#include "gfsx_device.h"

#include <algorithm>

namespace gfsx {

namespace {

constexpr int PNT = 1024;            // threads of the count and place kernels
constexpr int PITEMS = 16;           // most points per thread there
constexpr uint32_t CHUNK = 2048;     // most points of one brick work-group
constexpr uint32_t SPARSE = 32;      // bricks below this size are not staged
constexpr int SLOW_BLOCKS = 1024;
constexpr uint32_t kMaxBins = 40000; // histogram words that fit a CU's 160 KB of LDS

// The brick frame of a grid: bricks of 8^3 cells, i fastest, then one bin
// for the points outside the grid (their samples are 0).
struct PointGrid {
    int gbx, gby, gbz;
    uint32_t nbin;       // gbx*gby*gbz + 1
    float inv;           // 1/dx
    float limf[3];
};

// A point's brick.  FP32: a point within rounding of a cell face may be
// given the neighbouring brick, whose boxes hold its stencil too.
__device__ __forceinline__ uint32_t point_bin(const PointGrid &g, float x, float y, float z) {
    if (!(x >= 0.0f && y >= 0.0f && z >= 0.0f && x < g.limf[0] && y < g.limf[1] && z < g.limf[2]))
        return g.nbin - 1u;
    const int bx = min((int)(x * g.inv) >> 3, g.gbx - 1);
    const int by = min((int)(y * g.inv) >> 3, g.gby - 1);
    const int bz = min((int)(z * g.inv) >> 3, g.gbz - 1);
    return (uint32_t)bx + (uint32_t)g.gbx * ((uint32_t)by + (uint32_t)g.gby * (uint32_t)bz);
}

__device__ __forceinline__ uint32_t load_bin(const PointGrid &g, const float *__restrict__ pos,
                                             int64_t p) {
    return point_bin(g, gld(pos, 3 * p), gld(pos, 3 * p + 1), gld(pos, 3 * p + 2));
}

// items points per thread (at most PITEMS): the work-group's points are
// [blockIdx * items * PNT, ...), item m the m-th run of PNT of them.
__global__ __launch_bounds__(PNT) void k_pt_count(PointGrid g, const float *__restrict__ pos,
                                                  int64_t n, int items,
                                                  uint32_t *__restrict__ count) {
    extern __shared__ uint32_t s_hist[];
    for (uint32_t b = threadIdx.x; b < g.nbin; b += PNT) s_hist[b] = 0u;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * items * PNT + threadIdx.x;
    for (int m = 0; m < items; m++) {
        const int64_t p = base + (int64_t)m * PNT;
        if (p < n) atomicAdd(&s_hist[load_bin(g, pos, p)], 1u);
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < g.nbin; b += PNT) {
        const uint32_t c = s_hist[b];
        if (c) atomicAdd(&count[b], c);
    }
}

// One work-group: cursor[b] = first slot of bin b, the sparse ones' from the
// end of the n points down, and the chunk list (bin, first slot, points);
// meta[0] = chunks, meta[1] (the slow list's count) = 0, meta[2] = points of
// the sparse bins.
__global__ __launch_bounds__(PNT) void k_pt_scan(uint32_t nbin, uint32_t n,
                                                 const uint32_t *__restrict__ count,
                                                 uint32_t *__restrict__ cursor,
                                                 uint4 *__restrict__ chunks,
                                                 uint32_t *__restrict__ meta) {
    __shared__ uint32_t s_p[PNT / 64], s_c[PNT / 64], s_s[PNT / 64];
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    uint32_t p0 = 0, c0 = 0, s0 = 0;
    for (uint32_t b0 = 0; b0 < nbin; b0 += PNT) {
        const uint32_t b = b0 + (uint32_t)t;
        const uint32_t all = b < nbin ? count[b] : 0u;
        const bool sparse = all < SPARSE && b != nbin - 1u;
        const uint32_t np = sparse ? 0u : all, ns = sparse ? all : 0u;
        const uint32_t nc = (np + CHUNK - 1u) / CHUNK;
        const uint32_t ip = wave_inclusive_sum(np), ic = wave_inclusive_sum(nc),
                       is = wave_inclusive_sum(ns);
        if (lane == 63) {
            s_p[wid] = ip;
            s_c[wid] = ic;
            s_s[wid] = is;
        }
        __syncthreads();
        uint32_t ps = p0 + ip - np, cs = c0 + ic - nc, ss = s0 + is, pt = 0, ct = 0, st = 0;
        for (int w = 0; w < PNT / 64; w++) {
            const uint32_t a = s_p[w], c = s_c[w], d = s_s[w];
            if (w < wid) {
                ps += a;
                cs += c;
                ss += d;
            }
            pt += a;
            ct += c;
            st += d;
        }
        if (b < nbin) cursor[b] = sparse ? n - ss : ps;
        // equal shares of the bin's points
        for (uint32_t k = 0; k < nc; k++) {
            const uint32_t f = (uint32_t)((uint64_t)np * k / nc), e = (uint32_t)((uint64_t)np * (k + 1) / nc);
            chunks[cs + k] = make_uint4(b, ps + f, e - f, 0u);
        }
        p0 += pt;
        c0 += ct;
        s0 += st;
        __syncthreads();
    }
    if (t == 0) {
        meta[0] = c0;
        meta[1] = 0u;
        meta[2] = s0;
    }
}

__global__ __launch_bounds__(PNT) void k_pt_place(PointGrid g, const float *__restrict__ pos,
                                                  int64_t n, int items,
                                                  uint32_t *__restrict__ cursor,
                                                  float4 *__restrict__ rec) {
    extern __shared__ uint32_t s_hist[];
    for (uint32_t b = threadIdx.x; b < g.nbin; b += PNT) s_hist[b] = 0u;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * items * PNT + threadIdx.x;
    uint32_t bin[PITEMS], rank[PITEMS];
#pragma unroll
    for (int m = 0; m < PITEMS; m++) {
        const int64_t p = base + (int64_t)m * PNT;
        if (m < items && p < n) {
            bin[m] = load_bin(g, pos, p);
            rank[m] = atomicAdd(&s_hist[bin[m]], 1u);
        }
    }
    __syncthreads();
    // each bin's count becomes the first slot of this work-group's range
    for (uint32_t b = threadIdx.x; b < g.nbin; b += PNT) {
        const uint32_t c = s_hist[b];
        if (c) s_hist[b] = atomicAdd(&cursor[b], c);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < PITEMS; m++) {
        const int64_t p = base + (int64_t)m * PNT;
        if (m < items && p < n) {
            const float x = gld(pos, 3 * p), y = gld(pos, 3 * p + 1), z = gld(pos, 3 * p + 2);
            rec[s_hist[bin[m]] + rank[m]] = make_float4(x, y, z, __uint_as_float((uint32_t)p));
        }
    }
}

// What one call computes per point.
struct PointJob {
    MacGrid g;
    RkConsts c;
    int order;          // 0: the sample; 1..4: a Runge-Kutta step
    float *out;         // AoS, by point index
};

// A sample from the staged boxes (edge E, origin (lx,ly,lz)); false, with
// out untouched, when a stencil leaves them.
template <int ST, int E, bool P2>
__device__ __forceinline__ bool box_sample(const MacGrid &g, const float *b0, const float *b1,
                                           const float *b2, int lx, int ly, int lz, const float q[3],
                                           float out[3]) {
    if (!(q[0] >= 0.0f && q[1] >= 0.0f && q[2] >= 0.0f && q[0] < g.limf[0] && q[1] < g.limf[1] &&
          q[2] < g.limf[2])) {
        out[0] = out[1] = out[2] = 0.0f;
        return true;
    }
    const AxisCoords cx = axis_coords_t<P2>(q[0], g.inv_dx);
    const AxisCoords cy = axis_coords_t<P2>(q[1], g.inv_dx);
    const AxisCoords cz = axis_coords_t<P2>(q[2], g.inv_dx);
    if (!in_box<ST, E>(cx, cy, cz, lx, ly, lz)) return false;
    const int b = (cx.ib - lx) + E * ((cy.ib - ly) + E * (cz.ib - lz));
    out[0] = box_comp_at<ST, E>(b0 + b + (cx.ia - cx.ib), cx.ta, cy.tb, cz.tb);
    out[1] = box_comp_at<ST, E>(b1 + b + E * (cy.ia - cy.ib), cx.tb, cy.ta, cz.tb);
    out[2] = box_comp_at<ST, E>(b2 + b + E * E * (cz.ia - cz.ib), cx.tb, cy.tb, cz.ta);
    return true;
}

// One Runge-Kutta step (rk_step's arithmetic) with samples by smp(q, out),
// which returns false where it cannot sample; then so does this.
template <class Smp>
__device__ __forceinline__ bool rk_with(int order, const RkConsts &c, const float x0[3],
                                        const float k1[3], float x1[3], Smp &&smp) {
    float q[3], k2[3], k3[3], k4[3];
    if (order == 1) {
#pragma unroll
        for (int a = 0; a < 3; a++) x1[a] = x0[a] + c.full * k1[a];
        return true;
    }
#pragma unroll
    for (int a = 0; a < 3; a++) q[a] = x0[a] + c.half * k1[a];
    if (!smp(q, k2)) return false;
    if (order == 2) {
#pragma unroll
        for (int a = 0; a < 3; a++) x1[a] = x0[a] + c.full * k2[a];
        return true;
    }
    const float h3 = order == 3 ? c.three_q : c.half;
#pragma unroll
    for (int a = 0; a < 3; a++) q[a] = x0[a] + h3 * k2[a];
    if (!smp(q, k3)) return false;
    if (order == 3) {
#pragma unroll
        for (int a = 0; a < 3; a++)
            x1[a] = x0[a] + c.ninth * ((2.0f * k1[a] + 3.0f * k2[a]) + 4.0f * k3[a]);
        return true;
    }
#pragma unroll
    for (int a = 0; a < 3; a++) q[a] = x0[a] + c.full * k3[a];
    if (!smp(q, k4)) return false;
#pragma unroll
    for (int a = 0; a < 3; a++)
        x1[a] = x0[a] + c.sixth * (((k1[a] + 2.0f * k2[a]) + 2.0f * k3[a]) + k4[a]);
    return true;
}

__device__ __forceinline__ void store_point(const PointJob &j, const float4 &r, const float o[3]) {
    const size_t p = 3 * (size_t)__float_as_uint(r.w);
    gst(j.out, p, o[0]);
    gst(j.out, p + 1, o[1]);
    gst(j.out, p + 2, o[2]);
}

// A Runge-Kutta step stages one cell more around the brick than a sample.
template <int ST, bool RK> struct PointBox {
    static constexpr int E = RK ? gbrick::Box<ST>::E : gbrick::Box<ST>::EO;
    static constexpr int LO = RK ? gbrick::Box<ST>::LO : gbrick::Box<ST>::LOO;
};

template <int ST, bool RK, bool P2>
__device__ __forceinline__ void point_brick(const PointGrid &pg, const PointJob &j,
                                            const float4 *__restrict__ rec,
                                            const uint4 *__restrict__ chunks,
                                            uint32_t *__restrict__ slow, uint32_t *meta) {
    using B = PointBox<ST, RK>;
    constexpr int CELLS = gbrick::GB * gbrick::GB * gbrick::GB;
    constexpr int PER = (int)CHUNK / gbrick::NT;
    __shared__ float s_box[3][B::E * B::E * B::E];
    __shared__ uint32_t s_cell[CELLS];       // points per cell, then their first place
    __shared__ uint16_t s_ord[CHUNK];        // the chunk's points in cell order
    __shared__ uint32_t s_wsum[gbrick::NT / 64];
    // the points to list, a bit each: a wave's 64 points of a pass share a word
    constexpr int WORDS = (int)CHUNK / 64;
    __shared__ uint64_t s_slow[ST == 0 ? 1 : WORDS];
    __shared__ uint32_t s_slow_at[ST == 0 ? 1 : WORDS];
    const uint32_t nchunk = gld(meta, 0);
    const uint32_t per = (nchunk + 7u) / 8u;
    // consecutive bricks share box halos: keep them on one XCD
    const uint32_t c = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || c >= nchunk) return;
    const uint4 ch = chunks[c];
    const int t = threadIdx.x, lane = t & 63;
    const bool outside = ch.x == pg.nbin - 1u;
    const int gx = (int)(ch.x % (uint32_t)pg.gbx), gy = (int)(ch.x / (uint32_t)pg.gbx % (uint32_t)pg.gby),
              gz = (int)(ch.x / ((uint32_t)pg.gbx * (uint32_t)pg.gby));
    const int lx = 8 * gx - B::LO, ly = 8 * gy - B::LO, lz = 8 * gz - B::LO;
    if (!outside) {
        float *const bx[3] = {s_box[0], s_box[1], s_box[2]};
        float m[3];
        stage_mac_boxes<B::E>(bx, j.g.f, j.g.ni, j.g.nj, j.g.nk, lx, ly, lz, m);
    }
    // the chunk's points in the order of their cells: lanes of one cell then
    // read the same LDS words and neighbouring cells' lanes different banks
    // (in any order inside a cell)
    static_assert(CELLS == 2 * gbrick::NT, "two cells per thread in the scan");
    s_cell[t] = 0u;
    s_cell[t + gbrick::NT] = 0u;
    if (ST != 0 && t < WORDS) s_slow[t] = 0ull;
    __syncthreads();
    uint32_t cr[PER];   // cell << 16 | rank in it
#pragma unroll
    for (int m = 0; m < PER; m++) {
        const uint32_t e = (uint32_t)(t + m * gbrick::NT);
        if (e < ch.z) {
            const float4 r = rec[ch.y + e];
            const int ci = min(max((int)(r.x * pg.inv) - 8 * gx, 0), 7);
            const int cj = min(max((int)(r.y * pg.inv) - 8 * gy, 0), 7);
            const int ck = min(max((int)(r.z * pg.inv) - 8 * gz, 0), 7);
            const uint32_t cell = (uint32_t)(ci + 8 * (cj + 8 * ck));
            cr[m] = (cell << 16) | atomicAdd(&s_cell[cell], 1u);
        }
    }
    __syncthreads();
    {
        const uint32_t a = s_cell[2 * t], b = s_cell[2 * t + 1];
        uint32_t tot;
        const uint32_t at = block_exclusive_sum(a + b, s_wsum, tot);
        s_cell[2 * t] = at;
        s_cell[2 * t + 1] = at + a;
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < PER; m++) {
        const uint32_t e = (uint32_t)(t + m * gbrick::NT);
        if (e < ch.z) s_ord[s_cell[cr[m] >> 16] + (cr[m] & 0xFFFFu)] = (uint16_t)e;
    }
    __syncthreads();
    auto smp = [&](const float q[3], float out[3]) {
        const bool in = box_sample<ST, B::E, P2>(j.g, s_box[0], s_box[1], s_box[2], lx, ly, lz, q, out);
        if (ST != 0 || in) return in;
        float unused[3];
        sample_mac<0, false>(j.g, nullptr, nullptr, nullptr, q[0], q[1], q[2], out, unused);
        return true;
    };
    for (uint32_t e = (uint32_t)t; e < ch.z; e += gbrick::NT) {
        const uint32_t q = ch.y + s_ord[e];
        const float4 r = rec[q];
        const float x0[3] = {r.x, r.y, r.z};
        float k1[3], o[3];
        bool done = smp(x0, k1);
        if (RK) {
            if (done) done = rk_with(j.order, j.c, x0, k1, o, smp);
        } else if (done) {
            validate3(k1);
#pragma unroll
            for (int a = 0; a < 3; a++) o[a] = k1[a];
        }
        if (done) store_point(j, r, o);
        if (ST != 0) {
            const uint64_t mk = __ballot(!done);
            if (mk && lane == 0) s_slow[e >> 6] = mk;
        }
    }
    if (ST == 0) return;
    // the chunk's listed points: one atomic for all of them
    __syncthreads();
    if (t < 64) {
        const uint32_t n = t < WORDS ? (uint32_t)__popcll(s_slow[t]) : 0u;
        const uint32_t inc = wave_inclusive_sum(n), tot = __shfl(inc, 63, 64);
        uint32_t at = 0;
        if (tot && t == 0) at = atomicAdd(&meta[1], tot);
        at = __shfl(at, 0, 64);
        if (t < WORDS) s_slow_at[t] = at + inc - n;
    }
    __syncthreads();
    for (int w = t >> 6; w < WORDS; w += gbrick::NT / 64) {
        const uint64_t mk = s_slow[w];
        if ((mk >> lane) & 1ull)
            slow[s_slow_at[w] + (uint32_t)__popcll(mk & ((1ull << lane) - 1ull))] =
                ch.y + s_ord[64 * w + lane];
    }
}

template <int ST, bool RK, bool P2>
__global__ __launch_bounds__(gbrick::NT, ST == 0 ? 6 : 4) void k_pt_brick(
    PointGrid pg, PointJob j, const float4 *__restrict__ rec, const uint4 *__restrict__ chunks,
    uint32_t *__restrict__ slow, uint32_t *meta) {
    point_brick<ST, RK, P2>(pg, j, rec, chunks, slow, meta);
}

template <int ST>
__global__ __launch_bounds__(kBlock) void k_pt_slow(PointJob j, uint32_t n,
                                                   const float4 *__restrict__ rec,
                                                   const uint32_t *__restrict__ slow,
                                                   const uint32_t *__restrict__ meta) {
    const uint32_t ns = meta[1], all = ns + meta[2];
    for (uint32_t e = blockIdx.x * kBlock + threadIdx.x; e < all; e += gridDim.x * kBlock) {
        const float4 r = rec[e < ns ? slow[e] : n - (all - e)];
        const float x0[3] = {r.x, r.y, r.z};
        float k1[3], o[3], unused[3];
        sample_mac<ST, false>(j.g, nullptr, nullptr, nullptr, x0[0], x0[1], x0[2], k1, unused);
        if (ST == 0 || j.order > 0) {
            rk_step<ST>(j.g, j.order, j.c, x0, k1, o);
            store_point(j, r, o);
        } else {
            validate3(k1);
            store_point(j, r, k1);
        }
    }
}

}  // namespace

int64_t points_bins(int ni, int nj, int nk) {
    return (int64_t)((ni + 7) / 8) * ((nj + 7) / 8) * ((nk + 7) / 8) + 1;
}

bool points_by_brick(int64_t n, int ni, int nj, int nk, int order, int stencil) {
    const int64_t bins = points_bins(ni, nj, nk);
    if (bins > (int64_t)kMaxBins || n >= ((int64_t)1 << 31) || n < kPointsPerBrick * (bins - 1))
        return false;
    if (stencil == 0)
        return order >= 3 && n >= (order == 3 ? 2 : 1) * kPointsMinLinear &&
               n >= kPointsPerBrickLinear * (bins - 1);
    return n >= (order >= 2 ? kPointsMinCubicRk : kPointsMinCubic);
}

size_t points_workspace(int64_t n, int ni, int nj, int nk) {
    const int64_t nb = points_bins(ni, nj, nk);
    // records, slow list, counts, cursors, meta, chunk list
    return 16 * (size_t)n + 4 * (size_t)n + 8 * (size_t)nb + 64 +
           16 * (size_t)(nb + n / CHUNK + 1) + 5 * 256;
}

void points_run(void *work, const float *pos, int64_t n, const MacGrid &g, int order, double dt,
                int stencil, float *out, hipStream_t s) {
    PointGrid pg;
    pg.gbx = (g.ni + 7) / 8;
    pg.gby = (g.nj + 7) / 8;
    pg.gbz = (g.nk + 7) / 8;
    pg.nbin = (uint32_t)points_bins(g.ni, g.nj, g.nk);
    pg.inv = (float)g.inv_dx;
    for (int a = 0; a < 3; a++) pg.limf[a] = g.limf[a];
    char *at = static_cast<char *>(work);
    auto take = [&](size_t bytes) {
        char *p = at;
        at += (bytes + 255) & ~(size_t)255;
        return p;
    };
    const size_t nchunk = (size_t)(pg.nbin + n / CHUNK + 1);
    float4 *rec = (float4 *)take(16 * (size_t)n);
    uint4 *chunks = (uint4 *)take(16 * nchunk);
    uint32_t *slow = (uint32_t *)take(4 * (size_t)n);
    uint32_t *count = (uint32_t *)take(4 * (size_t)pg.nbin);
    uint32_t *cursor = (uint32_t *)take(4 * (size_t)pg.nbin);
    uint32_t *meta = (uint32_t *)take(12);
    PointJob j;
    j.g = g;
    j.c = rk_consts(dt);
    j.order = order;
    j.out = out;
    fill_u32(count, 0u, (int64_t)pg.nbin, s);
    // about 512 work-groups, each of 1 to PITEMS points per thread, and of
    // half as many points as histogram words (which each clears and reads)
    const int items = (int)std::min<int64_t>(
        std::max<int64_t>({n / ((int64_t)512 * PNT), (int64_t)pg.nbin / (2 * PNT), 1}), PITEMS);
    const unsigned nblk = grid_for(n, (int64_t)items * PNT);
    const size_t lds = 4 * (size_t)pg.nbin;
    hipLaunchKernelGGL(k_pt_count, dim3(nblk), dim3(PNT), lds, s, pg, pos, n, items, count);
    GFSX_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_pt_scan, dim3(1), dim3(PNT), 0, s, pg.nbin, (uint32_t)n,
                       (const uint32_t *)count, cursor, chunks, meta);
    GFSX_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_pt_place, dim3(nblk), dim3(PNT), lds, s, pg, pos, n, items, cursor, rec);
    GFSX_LAUNCH_CHECK();
    int e = 0;
    const bool p2 = std::frexp(g.inv_dx, &e) == 0.5 && e > -100 && e < 100;
    // (a trilinear sample is not taken here: points_by_brick)
    if (stencil == 0 && order == 0) throw Error("points_run: no trilinear sample by bricks");
    auto *kern = stencil == 0 ? (p2 ? k_pt_brick<0, true, true> : k_pt_brick<0, true, false>)
               : order > 0    ? (p2 ? k_pt_brick<1, true, true> : k_pt_brick<1, true, false>)
                              : (p2 ? k_pt_brick<1, false, true> : k_pt_brick<1, false, false>);
    hipLaunchKernelGGL(kern, dim3((unsigned)(8 * ((nchunk + 7) / 8))), dim3(gbrick::NT), 0, s, pg, j,
                       (const float4 *)rec, (const uint4 *)chunks, slow, meta);
    GFSX_LAUNCH_CHECK();
    auto *slowk = stencil == 0 ? k_pt_slow<0> : k_pt_slow<1>;
    hipLaunchKernelGGL(slowk, dim3(SLOW_BLOCKS), dim3(kBlock), 0, s, j, (uint32_t)n,
                       (const float4 *)rec, (const uint32_t *)slow, (const uint32_t *)meta);
    GFSX_LAUNCH_CHECK();
}

}  // namespace gfsx
