// gfsx_remove.hip -- particle removal after the step, on gfx950:
// FluidSimulation::_removeMarkerParticlesInSolidCells and
// _removeMarkerParticles (fluidsimulation.cpp:1985-1988, 3213-3243).
//
// Particles in solid cells are dropped; a cell keeps at most max_per_cell
// particles.  The reference keeps the first ones of a rand() shuffle of the
// whole array; here a cell keeps the max_per_cell particles with the
// smallest SplitMix64 key of (seed, input index), a seeded order that is the
// same on every run and every machine.  The particles are grouped by cell
// (in any order inside one: the keys decide); k_remove_cells lists the solid
// and the over-full cells; k_remove_wave takes one listed cell of up to
// WAVE_MAX particles per wave, counts the smaller keys of each of its keys and
// drops the particles past the cap; k_remove_select does the same for larger
// cells, one work-group each, by a radix select over the cell's keys (eight
// byte passes, each a 256-bucket histogram in LDS: linear in the cell's
// count).  k_remove_count and a scan give each block of particles its first
// output index and k_remove_compact copies the kept particles in input order.
//
// Bound: the copy, by memory (56 bytes per particle with labels).  5.65M
// particles on 128x113x128, some 7 thousand over-full cells of 101..160: 0.94
// ms with one work-group and eight radix passes per over-full cell (0.50 ms of
// it; now 26 us), every particle's cell looked up again (0.09) and the cells
// ordered inside (0.06); now 0.30 ms, 66 us of it the copy (4.8 TB/s).

#include "gfsx_internal.h"

#include <algorithm>

namespace gfsx {

namespace {

inline unsigned blocks_for(int64_t n) {
    return (unsigned)std::max<int64_t>((n + kBlock - 1) / kBlock, 1);
}

// SplitMix64 (Steele, Lea, Flood 2014; constants of Vigna's splitmix64.c):
// a bijection of i for a fixed seed, so keys never tie
__device__ __forceinline__ uint64_t removal_key(uint64_t seed, uint64_t i) {
    uint64_t z = seed + (i + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

constexpr uint32_t WAVE_MAX = 256;   // particles of a cell that one wave decides

// The cells some of whose particles go, one thread per cell: solid cells
// with particles and over-full cells of up to WAVE_MAX particles from the
// front of the list (nfull[0]), larger ones from its back (nfull[1]).
__global__ __launch_bounds__(kBlock) void k_remove_cells(RemoveArgs r) {
    const uint32_t b = blockIdx.x * kBlock + threadIdx.x;
    const int lane = threadIdx.x & 63;
    bool wave = false, group = false;
    if (b < r.bg.nbin) {
        const uint32_t len = r.start[b + 1] - r.start[b];
        const bool solid = r.solid && len > 0 && r.solid[b];
        if (solid || len > (uint32_t)r.max_per_cell) {
            group = !solid && len > WAVE_MAX;
            wave = !group;
        }
    }
    const uint64_t mw = __ballot(wave), mg = __ballot(group);
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t w0 = 0, g0 = 0;
    if (lane == 0) {
        if (mw) w0 = atomicAdd(&r.nfull[0], (uint32_t)__popcll(mw));
        if (mg) g0 = atomicAdd(&r.nfull[1], (uint32_t)__popcll(mg));
    }
    w0 = __shfl(w0, 0, 64);
    g0 = __shfl(g0, 0, 64);
    if (wave) r.full[w0 + (uint32_t)__popcll(mw & below)] = b;
    if (group) r.full[r.full_cap - 1u - (g0 + (uint32_t)__popcll(mg & below))] = b;
}

// One wave per listed cell (grid-stride).  A solid cell loses every
// particle; an over-full one those with max_per_cell or more smaller keys
// (keys are distinct).  The keys pass through LDS in the wave's own part.
__global__ __launch_bounds__(kBlock) void k_remove_wave(RemoveArgs r) {
    __shared__ uint64_t s_key[kBlock / 64][WAVE_MAX];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint32_t nlist = r.nfull[0], stride = gridDim.x * (kBlock / 64);
    for (uint32_t c = blockIdx.x * (kBlock / 64) + (uint32_t)wid; c < nlist; c += stride) {
        const uint32_t b = r.full[c];
        const uint32_t q0 = r.start[b], len = r.start[b + 1] - q0;
        if (r.solid && r.solid[b]) {
            for (uint32_t e = (uint32_t)lane; e < len; e += 64u) r.keep[r.perm[q0 + e]] = 0;
            continue;
        }
        constexpr int PER = (int)WAVE_MAX / 64;
        uint32_t p[PER], rank[PER];
        uint64_t key[PER];
#pragma unroll
        for (int m = 0; m < PER; m++) {
            const uint32_t e = (uint32_t)(lane + 64 * m);
            p[m] = e < len ? r.perm[q0 + e] : 0u;
            key[m] = removal_key(r.seed, (uint64_t)p[m]);
            rank[m] = 0;
            if (e < len) s_key[wid][e] = key[m];
        }
        // (a wave's LDS accesses are in order; keep the compiler's too)
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
        for (uint32_t e = 0; e < len; e++) {
            const uint64_t k = s_key[wid][e];
#pragma unroll
            for (int m = 0; m < PER; m++) rank[m] += k < key[m];
        }
#pragma unroll
        for (int m = 0; m < PER; m++)
            if ((uint32_t)(lane + 64 * m) < len && rank[m] >= (uint32_t)r.max_per_cell) r.keep[p[m]] = 0;
        __builtin_amdgcn_wave_barrier();
        __threadfence_block();
    }
}

// One work-group per larger over-full cell (grid-stride over the list's
// back): the max_per_cell-th smallest key of the cell, byte by byte from the
// top, then keep[p] = 0 for the particles whose key is above it.  Keys are
// distinct (a bijection of the index), so exactly max_per_cell are kept.
static_assert(kBlock == 256, "one histogram bucket per thread");

__global__ __launch_bounds__(kBlock) void k_remove_select(RemoveArgs r) {
    __shared__ uint32_t hist[256];
    __shared__ uint64_t s_prefix;
    __shared__ uint32_t s_rank;
    const uint32_t nfull = r.nfull[1];
    const int t = threadIdx.x;
    for (uint32_t c = blockIdx.x; c < nfull; c += gridDim.x) {
        const uint32_t b = r.full[r.full_cap - 1u - c];
        const uint32_t q0 = r.start[b], q1 = r.start[b + 1];
        if (t == 0) {
            s_prefix = 0ull;
            s_rank = (uint32_t)r.max_per_cell;   // 1-based rank still to find
        }
        for (int pass = 7; pass >= 0; pass--) {
            const int sh = 8 * pass;
            hist[t] = 0u;   // kBlock == 256 buckets
            __syncthreads();
            const uint64_t prefix = s_prefix;
            for (uint32_t q = q0 + t; q < q1; q += kBlock) {
                const uint64_t key = removal_key(r.seed, (uint64_t)r.perm[q]);
                // the bytes above this pass match the prefix found so far
                const bool match = pass == 7 || (key >> (sh + 8)) == (prefix >> (sh + 8));
                if (match) atomicAdd(&hist[(key >> sh) & 255u], 1u);
            }
            __syncthreads();
            if (t == 0) {
                uint32_t rank = s_rank, d = 0;
                while (hist[d] < rank) {
                    rank -= hist[d];
                    d++;
                }
                s_rank = rank;
                s_prefix = prefix | ((uint64_t)d << sh);
            }
            __syncthreads();
        }
        const uint64_t kth = s_prefix;
        for (uint32_t q = q0 + t; q < q1; q += kBlock) {
            const uint32_t p = r.perm[q];
            if (removal_key(r.seed, (uint64_t)p) > kth) r.keep[p] = 0;
        }
        __syncthreads();
    }
}

// Particles per work-group of the count and the compaction: item m of a
// block is its m-th run of kBlock particles.
constexpr int ITEMS = 4;
constexpr int64_t TILE = (int64_t)ITEMS * kBlock;

// Kept particles of every block of TILE.
__global__ __launch_bounds__(kBlock) void k_remove_count(RemoveArgs r) {
    __shared__ uint32_t s_n[kBlock / 64];
    const int64_t base = (int64_t)blockIdx.x * TILE + threadIdx.x;
    uint32_t n = 0;
#pragma unroll
    for (int m = 0; m < ITEMS; m++) {
        const int64_t p = base + (int64_t)m * kBlock;
        n += (uint32_t)__popcll(__ballot(p < r.n && r.keep[p]));
    }
    if ((threadIdx.x & 63) == 0) s_n[threadIdx.x >> 6] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t tot = 0;
        for (int w = 0; w < kBlock / 64; w++) tot += s_n[w];
        r.count[blockIdx.x] = tot;
    }
}

__global__ __launch_bounds__(kBlock) void k_remove_compact(RemoveArgs r) {
    __shared__ uint32_t s_n[ITEMS][kBlock / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int64_t base = (int64_t)blockIdx.x * TILE + threadIdx.x;
    bool keep[ITEMS];
    uint32_t o[ITEMS];
#pragma unroll
    for (int m = 0; m < ITEMS; m++) {
        const int64_t p = base + (int64_t)m * kBlock;
        keep[m] = p < r.n && r.keep[p];
        const uint64_t mk = __ballot(keep[m]);
        o[m] = (uint32_t)__popcll(mk & ((1ull << lane) - 1ull));
        if (lane == 0) s_n[m][wid] = (uint32_t)__popcll(mk);
    }
    __syncthreads();
    uint32_t at = r.dst[blockIdx.x];
#pragma unroll
    for (int m = 0; m < ITEMS; m++)
#pragma unroll
        for (int w = 0; w < kBlock / 64; w++) {
            if (w == wid) o[m] += at;
            at += s_n[m][w];
        }
    for (int c = 0; c < 3; c++) {
        float x[ITEMS], v[ITEMS];
#pragma unroll
        for (int m = 0; m < ITEMS; m++) {
            const int64_t p = base + (int64_t)m * kBlock;
            x[m] = keep[m] ? gld(r.x[c], p) : 0.0f;
            v[m] = keep[m] ? gld(r.v[c], p) : 0.0f;
        }
#pragma unroll
        for (int m = 0; m < ITEMS; m++)
            if (keep[m]) {
                gst(r.xo[c], o[m], x[m]);
                gst(r.vo[c], o[m], v[m]);
            }
    }
    if (r.id_out) {
#pragma unroll
        for (int m = 0; m < ITEMS; m++) {
            const int64_t p = base + (int64_t)m * kBlock;
            if (keep[m]) r.id_out[o[m]] = r.id_in ? r.id_in[p] : (uint32_t)p;
        }
    }
}

}  // namespace

int64_t remove_blocks(int64_t n) { return std::max<int64_t>((n + TILE - 1) / TILE, 1); }

void remove_mark(const RemoveArgs &r, hipStream_t s) {
    fill_u8(r.keep, 1, r.n, s);
    fill_u32(r.nfull, 0u, 2, s);
    if (r.n > 0) {
        hipLaunchKernelGGL(k_remove_cells, dim3(blocks_for(r.bg.nbin)), dim3(kBlock), 0, s, r);
        GFSX_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_remove_wave, dim3(2048), dim3(kBlock), 0, s, r);
        GFSX_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_remove_select, dim3(1024), dim3(kBlock), 0, s, r);
        GFSX_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_remove_count, dim3((unsigned)remove_blocks(r.n)), dim3(kBlock), 0, s, r);
    GFSX_LAUNCH_CHECK();
}

void remove_compact(const RemoveArgs &r, hipStream_t s) {
    if (r.n <= 0) return;
    hipLaunchKernelGGL(k_remove_compact, dim3((unsigned)remove_blocks(r.n)), dim3(kBlock), 0, s, r);
    GFSX_LAUNCH_CHECK();
}

}  // namespace gfsx
