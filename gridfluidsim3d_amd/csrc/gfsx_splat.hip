// gfsx_splat.hip -- P2G of point arrays onto a node grid for any radius
// (CLScalarField::addPointValues / addPoints, clscalarfield.cpp:68-301) on
// gfx950: a stable sort of the points by cell whose records the gather reads
// in sequence.
//
// The bin cells (gfsx_internal.h, BinGrid) are grouped in bricks of 8^3; the
// sort places brick after brick, cell after cell inside a brick (i fastest)
// and point index order inside a cell:
//
//   1. k_sp_count / k_sp_starts / k_sp_place: every point's record (x, y, z,
//      value; 16 bytes) and index into its brick's range, by histograms of
//      the bricks in LDS (the order inside a brick is not fixed yet).
//   2. k_sp_cells: one work-group per brick counts its cells in LDS, and
//      writes each record to its cell at the rank of its index there; the
//      512 cell starts go to a table (brick * 512 + cell, so a cell's end is
//      the next entry).  A brick of more than CAP points is only grouped by
//      cell there; k_sp_rank gives its records their places, RANK_TILE of
//      them per work-group.
//   3. k_sp_gather: every node sums the records of its candidate cells, rows
//      in (k, j) order, then cell order, then index order: a fixed order, so
//      results are bit-identical run to run.  k_sp_gather_sparse does the
//      same where no brick holds more than two points per cell on average.
//
// Bound: the gather by L2 reads (a lane's records are 16 bytes apart, a
// wave's spread over a cache line per cell), the passes before it by
// scattered memory.  The gather through a permutation of unsorted AoS points
// read 16 bytes from a random place per candidate (64-odd per node at 8
// points per cell).  3.85M shuffled points with values on 131x97x113, R = dx,
// with weights, per component: 1.44 -> 0.33 ms (gather 1.14 -> 0.10, sort
// 0.30 -> 0.20); 0.73M points on 160x121x144, R = 2.5 dx: 0.94 -> 0.32 ms.

#include "gfsx_internal.h"
#include "gfsx_device.h"

#include <algorithm>

namespace gfsx {

namespace {

constexpr int SNT = 1024;             // threads of the count and place kernels
constexpr int SITEMS = 16;            // most points per thread there
constexpr uint32_t kMaxBricks = 40000;   // histogram words that fit a CU's 160 KB of LDS
constexpr uint32_t CAP = 6144;        // points of a brick ordered in LDS
constexpr int CELLS = 512;            // cells of a brick
constexpr uint32_t RANK_TILE = 256;   // points of a crowded brick that a work-group ranks
constexpr size_t RANK_BLOCKS = 2048;  // its work-groups
constexpr uint32_t kSparse = 2 * CELLS;   // most points of a brick for k_sp_gather_sparse

struct SplatGrid {
    BinGrid bg;
    int gb[3];          // bricks per axis
    uint32_t nbrick;    // their number; also the bin of the points outside the bins
};

// A point's brick and its cell there; bin_of's arithmetic.
__device__ __forceinline__ uint32_t brick_of(const SplatGrid &g, float x, float y, float z,
                                             uint32_t &cell) {
    const float px = x - g.bg.off[0], py = y - g.bg.off[1], pz = z - g.bg.off[2];
    const double fi = floor((double)px * g.bg.inv_dx) + g.bg.pad[0];
    const double fj = floor((double)py * g.bg.inv_dx) + g.bg.pad[1];
    const double fk = floor((double)pz * g.bg.inv_dx) + g.bg.pad[2];
    cell = 0;
    if (!(fi >= 0.0 && fj >= 0.0 && fk >= 0.0 && fi < (double)g.bg.b[0] &&
          fj < (double)g.bg.b[1] && fk < (double)g.bg.b[2]))
        return g.nbrick;
    const uint32_t i = (uint32_t)fi, j = (uint32_t)fj, k = (uint32_t)fk;
    cell = (i & 7u) | ((j & 7u) << 3) | ((k & 7u) << 6);
    return (i >> 3) + (uint32_t)g.gb[0] * ((j >> 3) + (uint32_t)g.gb[1] * (k >> 3));
}

__global__ __launch_bounds__(SNT) void k_sp_count(SplatGrid g, const float *__restrict__ pos,
                                                  int64_t n, int items,
                                                  uint32_t *__restrict__ count) {
    extern __shared__ uint32_t s_hist[];
    for (uint32_t b = threadIdx.x; b <= g.nbrick; b += SNT) s_hist[b] = 0u;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * items * SNT + threadIdx.x;
    for (int m = 0; m < items; m++) {
        const int64_t p = base + (int64_t)m * SNT;
        uint32_t cell;
        if (p < n)
            atomicAdd(&s_hist[brick_of(g, gld(pos, 3 * p), gld(pos, 3 * p + 1), gld(pos, 3 * p + 2),
                                       cell)], 1u);
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b <= g.nbrick; b += SNT) {
        const uint32_t c = s_hist[b];
        if (c) atomicAdd(&count[b], c);
    }
}

// One work-group: first[b] (b = 0..nbrick+1), the placing cursors, in
// first[nbrick+2] the points of the fullest brick, and in first[nbrick+3] the
// count of k_sp_rank's tiles, cleared.
__global__ __launch_bounds__(SNT) void k_sp_starts(uint32_t nbrick, const uint32_t *__restrict__ count,
                                                   uint32_t *__restrict__ first,
                                                   uint32_t *__restrict__ cursor) {
    __shared__ uint32_t s_w[SNT / 64];
    __shared__ uint32_t s_most;
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    uint32_t at = 0, most = 0;
    if (t == 0) s_most = 0u;
    for (uint32_t b0 = 0; b0 <= nbrick; b0 += SNT) {
        const uint32_t b = b0 + (uint32_t)t;
        const uint32_t c = b <= nbrick ? count[b] : 0u;
        const uint32_t inc = wave_inclusive_sum(c);
        if (b < nbrick) most = max(most, c);
        if (lane == 63) s_w[wid] = inc;
        __syncthreads();
        uint32_t s = at + inc - c;
        for (int w = 0; w < SNT / 64; w++) {
            const uint32_t v = s_w[w];
            if (w < wid) s += v;
            at += v;
        }
        if (b <= nbrick) {
            first[b] = s;
            cursor[b] = s;
        }
        __syncthreads();
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, d, 64));
    if (lane == 0) atomicMax(&s_most, most);
    __syncthreads();
    if (t == 0) {
        first[nbrick + 1] = at;
        first[nbrick + 2] = s_most;
        first[nbrick + 3] = 0u;
    }
}

__global__ __launch_bounds__(SNT) void k_sp_place(SplatGrid g, const float *__restrict__ pos,
                                                  const float *__restrict__ val, int64_t n,
                                                  int items, uint32_t *__restrict__ cursor,
                                                  float4 *__restrict__ rec,
                                                  uint32_t *__restrict__ idx) {
    extern __shared__ uint32_t s_hist[];
    for (uint32_t b = threadIdx.x; b <= g.nbrick; b += SNT) s_hist[b] = 0u;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * items * SNT + threadIdx.x;
    uint32_t bin[SITEMS], rank[SITEMS];
#pragma unroll
    for (int m = 0; m < SITEMS; m++) {
        const int64_t p = base + (int64_t)m * SNT;
        if (m < items && p < n) {
            uint32_t cell;
            bin[m] = brick_of(g, gld(pos, 3 * p), gld(pos, 3 * p + 1), gld(pos, 3 * p + 2), cell);
            rank[m] = atomicAdd(&s_hist[bin[m]], 1u);
        }
    }
    __syncthreads();
    // each brick's count becomes the first slot of this work-group's range
    for (uint32_t b = threadIdx.x; b <= g.nbrick; b += SNT) {
        const uint32_t c = s_hist[b];
        if (c) s_hist[b] = atomicAdd(&cursor[b], c);
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < SITEMS; m++) {
        const int64_t p = base + (int64_t)m * SNT;
        if (m < items && p < n) {
            const uint32_t q = s_hist[bin[m]] + rank[m];
            rec[q] = make_float4(gld(pos, 3 * p), gld(pos, 3 * p + 1), gld(pos, 3 * p + 2),
                                 val ? gld(val, p) : 1.0f);
            idx[q] = (uint32_t)p;
        }
    }
}

// One work-group per brick: its records from rec (any order) to out (by
// cell, then point index), and its cells' starts.  Ranks inside a cell come
// from counting the cell's smaller indices, 8 at 8 points per cell.  A brick
// of more than CAP points leaves that count, which grows as the square, to
// k_sp_rank: its points grouped by cell (index and place in rec) in spill, and
// their tiles appended to tiles (brick, tile), *ntile of them.
__global__ __launch_bounds__(CELLS) void k_sp_cells(SplatGrid g, const uint32_t *__restrict__ first,
                                                     const float4 *__restrict__ rec,
                                                     const uint32_t *__restrict__ idx,
                                                     uint2 *__restrict__ spill,
                                                     uint2 *__restrict__ tiles,
                                                     uint32_t *__restrict__ ntile,
                                                     float4 *__restrict__ out,
                                                     uint32_t *__restrict__ start) {
    __shared__ uint32_t s_cell[CELLS + 1];    // points per cell, then the cell's first place
    __shared__ uint32_t s_cur[CELLS];
    __shared__ uint32_t s_idx[CAP];           // point indices, grouped by cell
    __shared__ uint32_t s_src[CAP];           // cell << 16 | place in rec
    __shared__ uint32_t s_wsum[CELLS / 64];
    const int t = threadIdx.x;
    const uint32_t b = blockIdx.x;
    const uint32_t q0 = first[b], N = first[b + 1] - q0;
    uint32_t *st = start + (size_t)b * CELLS;
    if (b == g.nbrick - 1 && t == 0) start[(size_t)g.nbrick * CELLS] = q0 + N;
    if (N == 0) {
        st[t] = q0;
        return;
    }
    s_cell[t] = 0u;
    __syncthreads();
    for (uint32_t e = t; e < N; e += CELLS) {
        const float4 r = rec[q0 + e];
        uint32_t cell;
        brick_of(g, r.x, r.y, r.z, cell);
        atomicAdd(&s_cell[cell], 1u);
    }
    __syncthreads();
    {
        // one cell per thread
        const int lane = t & 63, wid = t >> 6;
        const uint32_t n = s_cell[t], inc = wave_inclusive_sum(n);
        if (lane == 63) s_wsum[wid] = inc;
        __syncthreads();
        uint32_t at = inc - n;
        for (int w = 0; w < wid; w++) at += s_wsum[w];
        s_cell[t] = s_cur[t] = at;
        st[t] = q0 + at;
        if (t == 0) s_cell[CELLS] = N;
    }
    __syncthreads();
    if (N <= CAP) {
        for (uint32_t e = t; e < N; e += CELLS) {
            const float4 r = rec[q0 + e];
            uint32_t cell;
            brick_of(g, r.x, r.y, r.z, cell);
            const uint32_t at = atomicAdd(&s_cur[cell], 1u);
            s_idx[at] = idx[q0 + e];
            s_src[at] = (cell << 16) | e;
        }
        __syncthreads();
        for (uint32_t e = t; e < N; e += CELLS) {
            const uint32_t sc = s_src[e], mine = s_idx[e];
            const uint32_t c0 = s_cell[sc >> 16], c1 = s_cell[(sc >> 16) + 1];
            uint32_t rank = 0;
            for (uint32_t k = c0; k < c1; k++) rank += s_idx[k] < mine;
            out[q0 + c0 + rank] = rec[q0 + (sc & 0xFFFFu)];
        }
        return;
    }
    for (uint32_t e = t; e < N; e += CELLS) {
        const float4 r = rec[q0 + e];
        uint32_t cell;
        brick_of(g, r.x, r.y, r.z, cell);
        spill[q0 + atomicAdd(&s_cur[cell], 1u)] = make_uint2(idx[q0 + e], e);
    }
    const uint32_t nt = (N + RANK_TILE - 1u) / RANK_TILE;
    if (t == 0) s_wsum[0] = atomicAdd(ntile, nt);
    __syncthreads();
    for (uint32_t k = t; k < nt; k += CELLS) tiles[s_wsum[0] + k] = make_uint2(b, k);
}

// The records of the crowded bricks to their places, a tile of RANK_TILE
// grouped points at a time (grid-stride over the tiles): as in k_sp_cells, a
// point's rank is the number of smaller indices in its cell.  A cell's points
// lie together, so a wave reads the same few words; a cell's tiles are spread
// over the chip.  Whole calls on a 48^3 grid, R = dx, as measured with the
// brick's one work-group ranking them / now: 1M points in one brick 329 / 8.2
// ms (5 of it the gather of the crowded nodes, 0.3 this kernel), 0.2M 16.6 /
// 1.6, 16 points in every cell 251 / 196 us, 32 573 / 371; 20 thousand points
// in one cell 5.5 ms.
__global__ __launch_bounds__(RANK_TILE) void k_sp_rank(SplatGrid g, const uint32_t *__restrict__ first,
                                                       const uint32_t *__restrict__ start,
                                                       const float4 *__restrict__ rec,
                                                       const uint2 *__restrict__ spill,
                                                       const uint2 *__restrict__ tiles,
                                                       const uint32_t *__restrict__ ntile,
                                                       float4 *__restrict__ out) {
    const uint32_t nt = *ntile;
    for (uint32_t n = blockIdx.x; n < nt; n += gridDim.x) {
        const uint2 tile = tiles[n];
        const uint32_t q0 = first[tile.x], q1 = first[tile.x + 1u];
        const uint32_t p = q0 + tile.y * RANK_TILE + threadIdx.x;
        if (p >= q1) continue;
        const uint2 me = spill[p];
        const float4 r = rec[q0 + me.y];
        uint32_t cell;
        const uint32_t id = brick_of(g, r.x, r.y, r.z, cell) * (uint32_t)CELLS + cell;
        const uint32_t c0 = start[id], c1 = start[id + 1u];
        uint32_t rank = 0;
#pragma unroll 8
        for (uint32_t k = c0; k < c1; k++) rank += spill[k].x < me.x;
        out[c0 + rank] = r;
    }
}

// A record's terms of one node: K (and K val) at squared distance dxy + vz^2,
// dxy = vx^2 + vy^2.  The roundings are written out, so that a node's sums do
// not depend on which gather takes it; they are those of the cell sort's
// gather.  in false: the record adds nothing.
__device__ __forceinline__ float square_xy(float vx, float vy) { return fmaf(vx, vx, vy * vy); }

template <bool HAS_VAL>
__device__ __forceinline__ void add_record(float dxy, float vz, float inv_r2, float val, bool in,
                                           float &s, float &w) {
    const float d2 = fmaf(vz, vz, dxy);
    const float b = fmaxf(fmaf(-d2, inv_r2, 1.0f), 0.0f);
    const float a = in ? b : 0.0f, a2 = a * a;
    const float q = fmaf(4.0f / 9.0f, a, 5.0f / 9.0f);
    // only inside the radius (scalarfield.cpp:191-196): a value that is not
    // finite must not reach the nodes beyond it
    if (HAS_VAL) s = fmaf(a2 * q, in && d2 * inv_r2 < 1.0f ? val : 0.0f, s);
    else s = fmaf(a2, q, s);
    w = fmaf(a2, q, w);
}

// One thread per column of kseg nodes along z.  A node's candidate cells
// along an axis are D consecutive ones (dhi - dlo + 1), so the cells of one
// plane reach D nodes of the column: the thread walks the planes upwards,
// reads each candidate record once for all of them (its x and y distances
// are shared) and keeps their sums in registers, slot m for node
// plane - dhi + m.  A node's own terms still come plane by plane, row by row
// and in cell order.  A row's cells are one range per brick they lie in; two
// records are loaded ahead of the sums, and one past the range adds K = 0.
// COLUMN false: kseg is 1, one slot.
template <bool HAS_VAL, int D, bool COLUMN>
__global__ __launch_bounds__(kBlock) void k_sp_gather(SplatGrid g, NodeGrid ng, double dx,
                                                      float inv_r2, int kseg,
                                                      const uint32_t *__restrict__ most,
                                                      const uint32_t *__restrict__ start,
                                                      const float4 *__restrict__ rec,
                                                      float *__restrict__ S, float *__restrict__ W) {
    constexpr int AHEAD = 2;
    if (most && *most <= kSparse) return;   // k_sp_gather_sparse does it
    const int64_t col = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    const int64_t ncol = (int64_t)ng.n[0] * ng.n[1];
    if (col >= ncol) return;
    const int i = (int)(col % ng.n[0]), j = (int)(col / ng.n[0]);
    const int k0 = (int)blockIdx.y * kseg, k1 = min(k0 + kseg, ng.n[2]);
    // node position in the shifted frame, rounded as
    // Grid3d::GridIndexToPosition does (grid3d.h:79-81)
    const float gx = (float)((float)i * dx);
    const float gy = (float)((float)j * dx);
    const int ilo = max(i + ng.dlo[0], 0), ihi = min(i + ng.dhi[0], g.bg.b[0] - 1);
    const int jlo = max(j + ng.dlo[1], 0), jhi = min(j + ng.dhi[1], g.bg.b[1] - 1);
    const size_t stride = (size_t)ng.n[0] * ng.n[1];
    constexpr int M = COLUMN ? D : 1;
    float s[M], w[M], gz[M];
#pragma unroll
    for (int m = 0; m < M; m++) s[m] = w[m] = 0.0f;
    for (int bk = k0 + ng.dlo[2]; bk <= k1 - 1 + ng.dhi[2]; bk++) {
        const int kk = COLUMN ? bk - ng.dhi[2] : k0;   // the node of slot 0
        if (bk >= 0 && bk < g.bg.b[2]) {
#pragma unroll
            for (int m = 0; m < M; m++) gz[m] = (float)((float)(kk + m) * dx);
            for (int bj = jlo; bj <= jhi; bj++) {
                const uint32_t row = (uint32_t)g.gb[0] *
                                     ((uint32_t)(bj >> 3) + (uint32_t)g.gb[1] * (uint32_t)(bk >> 3));
                const uint32_t cjk = (uint32_t)((bj & 7) << 3) | (uint32_t)((bk & 7) << 6);
                for (int a = ilo; a <= ihi;) {
                    const int e = min(ihi, a | 7);
                    const uint32_t id = ((row + (uint32_t)(a >> 3)) << 9) | cjk | (uint32_t)(a & 7);
                    const uint32_t q0 = start[id], q1 = start[id + (uint32_t)(e - a) + 1u];
                    for (uint32_t q = q0; q < q1; q += AHEAD) {
                        float4 r[AHEAD];
#pragma unroll
                        for (int u = 0; u < AHEAD; u++) r[u] = rec[min(q + (uint32_t)u, q1 - 1u)];
#pragma unroll
                        for (int u = 0; u < AHEAD; u++) {
                            // p -= offset, then v = gpos - p (scalarfield.cpp:168,186-188)
                            const float vx = gx - (r[u].x - ng.off[0]);
                            const float vy = gy - (r[u].y - ng.off[1]);
                            const float pz = r[u].z - ng.off[2];
                            const float dxy = square_xy(vx, vy);
                            const bool in = q + (uint32_t)u < q1;
#pragma unroll
                            for (int m = 0; m < M; m++) {
                                // (the same for all lanes)
                                if (COLUMN && (kk + m < k0 || kk + m >= k1)) continue;
                                add_record<HAS_VAL>(dxy, gz[m] - pz, inv_r2, r[u].w, in, s[m], w[m]);
                            }
                        }
                    }
                    a = e + 1;
                }
            }
        }
        // the node of slot 0 has all its planes: accumulate into the caller's
        // arrays (clscalarfield.cpp:1448-1449)
        if (COLUMN ? kk >= k0 : bk == k0 + ng.dhi[2]) {
            const size_t f = (size_t)col + stride * (size_t)kk;
            S[f] += s[0];
            if (W) W[f] += w[0];
        }
#pragma unroll
        for (int m = 0; m + 1 < M; m++) {
            s[m] = s[m + 1];
            w[m] = w[m + 1];
        }
        if (COLUMN) s[M - 1] = w[M - 1] = 0.0f;
    }
}

// The same sums in the same order where cells hold few points.  A row is then
// mostly a wait for its two starts and for the wave's longest lane (0.26 points
// per cell: 1.6 records in a row of 6 cells, 5 to 6 in the longest of 64 lanes):
// all of a plane's starts are loaded together, its ranges that are not empty
// kept in LDS, and a thread goes through them as one sequence, so a wave waits
// for its longest lane once a plane.  A row's cells (at most 8) lie in at most
// two bricks.  0.73M points on 160x121x144, R = 2.5 dx: the call 410 -> 317 us.
// Where cells are full, lanes on different rows no longer share cache
// lines: splats of evenly spread points by rows / as one sequence at 1, 2, 4
// and 8 points per cell, R = dx: 189/177, 282/277, 266/284, 670/888 us; R = 2.5
// dx: 750/524, 1189/1005, 1611/2129, 3981/8717 us.  Hence kSparse, two points
// per cell in the fullest brick.
template <bool HAS_VAL, int D, bool COLUMN>
__global__ __launch_bounds__(kBlock) void k_sp_gather_sparse(SplatGrid g, NodeGrid ng, double dx,
                                                      float inv_r2, int kseg,
                                                      const uint32_t *__restrict__ most,
                                                      const uint32_t *__restrict__ start,
                                                      const float4 *__restrict__ rec,
                                                      float *__restrict__ S, float *__restrict__ W) {
    // the calling thread's own column only: no barrier
    __shared__ uint2 s_range[2 * D][kBlock];
    if (*most > kSparse) return;   // k_sp_gather does it
    const int64_t col = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    const int64_t ncol = (int64_t)ng.n[0] * ng.n[1];
    if (col >= ncol) return;
    const int i = (int)(col % ng.n[0]), j = (int)(col / ng.n[0]);
    const int k0 = (int)blockIdx.y * kseg, k1 = min(k0 + kseg, ng.n[2]);
    // node position in the shifted frame, rounded as
    // Grid3d::GridIndexToPosition does (grid3d.h:79-81)
    const float gx = (float)((float)i * dx);
    const float gy = (float)((float)j * dx);
    const int ilo = max(i + ng.dlo[0], 0), ihi = min(i + ng.dhi[0], g.bg.b[0] - 1);
    const int jlo = max(j + ng.dlo[1], 0), jhi = min(j + ng.dhi[1], g.bg.b[1] - 1);
    const size_t stride = (size_t)ng.n[0] * ng.n[1];
    constexpr int M = COLUMN ? D : 1;
    float s[M], w[M], gz[M];
#pragma unroll
    for (int m = 0; m < M; m++) s[m] = w[m] = 0.0f;
    for (int bk = k0 + ng.dlo[2]; bk <= k1 - 1 + ng.dhi[2]; bk++) {
        const int kk = COLUMN ? bk - ng.dhi[2] : k0;   // the node of slot 0
        if (bk >= 0 && bk < g.bg.b[2]) {
#pragma unroll
            for (int m = 0; m < M; m++) gz[m] = (float)((float)(kk + m) * dx);
            // the plane's ranges of records, every start loaded before any is used
            uint32_t q0[2 * D], q1[2 * D];
#pragma unroll
            for (int y = 0; y < D; y++) {
                const int bj = jlo + y;
                const uint32_t row = (uint32_t)g.gb[0] *
                                     ((uint32_t)(bj >> 3) + (uint32_t)g.gb[1] * (uint32_t)(bk >> 3));
                const uint32_t cjk = (uint32_t)((bj & 7) << 3) | (uint32_t)((bk & 7) << 6);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int a = h ? (ilo | 7) + 1 : ilo, e = h ? ihi : min(ihi, ilo | 7);
                    const bool some = bj <= jhi && a <= e;
                    const uint32_t id = ((row + (uint32_t)(a >> 3)) << 9) | cjk | (uint32_t)(a & 7);
                    q0[2 * y + h] = start[some ? id : 0u];
                    q1[2 * y + h] = start[some ? id + (uint32_t)(e - a) + 1u : 0u];
                }
            }
            int nr = 0;
#pragma unroll
            for (int c = 0; c < 2 * D; c++) {
                if (q0[c] < q1[c]) s_range[nr++][threadIdx.x] = make_uint2(q0[c], q1[c]);
            }
            bool live = nr > 0;
            uint2 at = make_uint2(0u, 0u);
            if (live) at = s_range[0][threadIdx.x];
            float4 r = rec[at.x];
            for (int c = 0; live;) {
                // the next record, loaded ahead of this one's sums
                bool more = true;
                if (++at.x >= at.y) {
                    more = ++c < nr;
                    if (more) at = s_range[c][threadIdx.x];
                }
                const float4 rn = rec[more ? at.x : 0u];
                const float vx = gx - (r.x - ng.off[0]);
                const float vy = gy - (r.y - ng.off[1]);
                const float pz = r.z - ng.off[2];
                const float dxy = square_xy(vx, vy);
#pragma unroll
                for (int m = 0; m < M; m++) {
                    if (COLUMN && (kk + m < k0 || kk + m >= k1)) continue;
                    add_record<HAS_VAL>(dxy, gz[m] - pz, inv_r2, r.w, true, s[m], w[m]);
                }
                r = rn;
                live = more;
            }
        }
        // the node of slot 0 has all its planes: accumulate into the caller's
        // arrays (clscalarfield.cpp:1448-1449)
        if (COLUMN ? kk >= k0 : bk == k0 + ng.dhi[2]) {
            const size_t f = (size_t)col + stride * (size_t)kk;
            S[f] += s[0];
            if (W) W[f] += w[0];
        }
#pragma unroll
        for (int m = 0; m + 1 < M; m++) {
            s[m] = s[m + 1];
            w[m] = w[m + 1];
        }
        if (COLUMN) s[M - 1] = w[M - 1] = 0.0f;
    }
}

using Gather = void (*)(SplatGrid, NodeGrid, double, float, int, const uint32_t *, const uint32_t *,
                        const float4 *, float *, float *);

template <int D>
Gather gather_kernel(bool val, bool column, bool sparse) {
    if (sparse)
        return column ? (val ? k_sp_gather_sparse<true, D, true> : k_sp_gather_sparse<false, D, true>)
                      : (val ? k_sp_gather_sparse<true, D, false> : k_sp_gather_sparse<false, D, false>);
    return column ? (val ? k_sp_gather<true, D, true> : k_sp_gather<false, D, true>)
                  : (val ? k_sp_gather<true, D, false> : k_sp_gather<false, D, false>);
}

int64_t bricks(const BinGrid &bg) {
    int64_t b = 1;
    for (int a = 0; a < 3; a++) b *= (bg.b[a] + 7) / 8;
    return b;
}

}  // namespace

// The gather of few points with a radius of one cell on a large grid is short,
// and the bricks' passes before it take longer than the cell sort's.  Cell sort /
// bricks, us per call, R = dx: 128^3 nodes, 3 thousand points 73 / 59, 100
// thousand 93 / 77; 160^3 89 / 90, 117 / 120; 200^3 122 / 124, 160 / 191, 250
// thousand 192 / 190; R = 1.7 dx: 200^3 191 / 172 and 300 / 238.
bool splat_by_brick(int64_t n, const BinGrid &bg, double reach, int64_t nnode) {
    const int64_t few = reach <= 1.0 && nnode > ((int64_t)3 << 20) ? nnode / 32 : 0;
    return reach <= 4.0 && n >= few && n < ((int64_t)1 << 31) && bricks(bg) < (int64_t)kMaxBricks;
}

// Most tiles of crowded bricks: a brick's last one may hold a single point,
// but a crowded brick holds more than CAP.
static size_t rank_tiles(int64_t n) {
    return (size_t)n / RANK_TILE + (size_t)n / CAP + 1;
}

size_t splat_workspace(int64_t n, const BinGrid &bg) {
    const size_t nb = (size_t)bricks(bg);
    // records twice, indices, crowded bricks' groups and tiles; counts, starts, cursors, cell starts
    return (16 + 16 + 8 + 4) * (size_t)n + 8 * rank_tiles(n) + 3 * 4 * (nb + 4) +
           4 * (nb * CELLS + 1) + 9 * 256;
}

void splat_run(void *work, const float *pos, const float *val, int64_t n, const BinGrid &bins,
               const NodeGrid &nodes, double radius, double dx, float *S, float *W, hipStream_t st) {
    const int64_t nnode = (int64_t)nodes.n[0] * nodes.n[1] * nodes.n[2];
    if (nnode <= 0) return;
    SplatGrid g;
    g.bg = bins;
    for (int a = 0; a < 3; a++) g.gb[a] = (bins.b[a] + 7) / 8;
    g.nbrick = (uint32_t)bricks(bins);
    char *at = static_cast<char *>(work);
    auto take = [&](size_t bytes) {
        char *p = at;
        at += (bytes + 255) & ~(size_t)255;
        return p;
    };
    const size_t nn = (size_t)n;
    float4 *rec = (float4 *)take(16 * nn), *out = (float4 *)take(16 * nn);
    uint2 *spill = (uint2 *)take(8 * nn);
    uint2 *tiles = (uint2 *)take(8 * rank_tiles(n));
    uint32_t *idx = (uint32_t *)take(4 * nn);
    uint32_t *count = (uint32_t *)take(4 * (size_t)(g.nbrick + 1));
    uint32_t *first = (uint32_t *)take(4 * (size_t)(g.nbrick + 4));
    uint32_t *cursor = (uint32_t *)take(4 * (size_t)(g.nbrick + 1));
    uint32_t *start = (uint32_t *)take(4 * ((size_t)g.nbrick * CELLS + 1));
    fill_u32(count, 0u, (int64_t)g.nbrick + 1, st);
    // about 512 work-groups, each of 1 to SITEMS points per thread, and of
    // half as many points as histogram words (which each clears and reads)
    const int items = (int)std::min<int64_t>(
        std::max<int64_t>({n / ((int64_t)512 * SNT), (int64_t)g.nbrick / (2 * SNT), 1}), SITEMS);
    const unsigned nblk = grid_for(n, (int64_t)items * SNT);
    const size_t lds = 4 * ((size_t)g.nbrick + 1);
    hipLaunchKernelGGL(k_sp_count, dim3(nblk), dim3(SNT), lds, st, g, pos, n, items, count);
    GFSX_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_sp_starts, dim3(1), dim3(SNT), 0, st, g.nbrick, (const uint32_t *)count,
                       first, cursor);
    GFSX_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_sp_place, dim3(nblk), dim3(SNT), lds, st, g, pos, val, n, items, cursor,
                       rec, idx);
    GFSX_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_sp_cells, dim3(g.nbrick), dim3(CELLS), 0, st, g, (const uint32_t *)first,
                       (const float4 *)rec, (const uint32_t *)idx, spill, tiles,
                       first + g.nbrick + 3, out, start);
    GFSX_LAUNCH_CHECK();
    if (n > (int64_t)CAP) {
        hipLaunchKernelGGL(k_sp_rank, dim3((unsigned)std::min<size_t>(rank_tiles(n), RANK_BLOCKS)),
                           dim3(RANK_TILE), 0, st, g, (const uint32_t *)first,
                           (const uint32_t *)start, (const float4 *)rec, (const uint2 *)spill,
                           (const uint2 *)tiles, (const uint32_t *)(first + g.nbrick + 3), out);
        GFSX_LAUNCH_CHECK();
    }
    const float inv_r2 = (float)(1.0 / (radius * radius));
    // Columns of 1 to 16 nodes, about 8192 waves of them (and no more
    // segments than a grid's y extent holds): longer columns read less,
    // shorter ones fill the chip.  0.27M nodes, columns of 1 / 4: 22 / 52 us
    // of gather; 2.8M nodes at R = 2.5 dx, the whole call with columns of
    // 1 / 3 / 5 / 8: 644 / 442 / 410 / 427 us by rows.
    const int kseg = (int)std::max<int64_t>(
        std::min<int64_t>(std::max<int64_t>(nnode / (64 * 8192), 1), 16), nodes.n[2] / 65535 + 1);
    const dim3 grid(grid_for((int64_t)nodes.n[0] * nodes.n[1], kBlock), grid_for(nodes.n[2], kseg));
    const int D = nodes.dhi[2] - nodes.dlo[2] + 1;
    const Gather kern = D == 2   ? gather_kernel<2>(val, kseg > 1, false)
                        : D == 4 ? gather_kernel<4>(val, kseg > 1, false)
                        : D == 6 ? gather_kernel<6>(val, kseg > 1, false)
                                 : gather_kernel<8>(val, kseg > 1, false);
    // The sparse gather's starts cost it more than its sums: past a radius of
    // one cell, columns of up to 3 nodes where the above gives fewer, and with
    // few points for the nodes 2048 waves of them.  100^3 nodes, columns of 1 / 3
    // / 7, us per call: R = 4 dx, 100 points 188 / 110 / 91, 62 thousand evenly
    // spread 243 / 151 / 128, in a ball 321 / 288 / 373; R = 1.7 dx 89 / 73 / 76
    // and 89 / 88 / 115; R = dx (128^3, columns of 4 / 8, 30 thousand) 75 / 87.
    const bool few = 32 * n < nnode;
    const int ksp = D == 2 ? kseg : (int)std::max<int64_t>(
        kseg, std::min<int64_t>(nnode / (64 * (few ? 2048 : 4096)), few ? 16 : 3));
    const Gather sparse = D == 2   ? gather_kernel<2>(val, ksp > 1, true)
                          : D == 4 ? gather_kernel<4>(val, ksp > 1, true)
                          : D == 6 ? gather_kernel<6>(val, ksp > 1, true)
                                   : gather_kernel<8>(val, ksp > 1, true);
    // the fullest brick, known on the device, decides which of the two works;
    // where the points' mean exceeds the line the rows do it anyway (3.85M
    // points in 3315 bricks: an empty launch saved)
    const uint32_t *most = n <= (int64_t)kSparse * g.nbrick ? first + g.nbrick + 2 : nullptr;
    if (most) {
        hipLaunchKernelGGL(sparse, dim3(grid.x, grid_for(nodes.n[2], ksp)), dim3(kBlock), 0, st, g,
                           nodes, dx, inv_r2, ksp, most,
                           (const uint32_t *)start, (const float4 *)out, S, W);
        GFSX_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(kern, grid, dim3(kBlock), 0, st, g, nodes, dx, inv_r2, kseg, most,
                       (const uint32_t *)start, (const float4 *)out, S, W);
    GFSX_LAUNCH_CHECK();
}

}  // namespace gfsx
