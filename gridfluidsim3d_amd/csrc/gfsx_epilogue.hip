// gfsx_epilogue.hip -- FluidSimulation's stages around the transfer: the
// face fill after P2G and the velocity extrapolation, on gfx950.
//
// After the P2G gather has written the normalised values n and the weights
// W of every face (no body force yet):
//
//   1. k_fs_layers: the cell layer grid of
//      MACVelocityField::extrapolateVelocityField (macvelocityfield.cpp:
//      577-664): fluid cells (a particle, not solid; fluidsimulation.cpp:
//      1990-2017) 0, then one 6-neighbour dilation per layer through
//      non-solid cells, up to seven layers per launch on bit rows in LDS;
//      solid cells are marked -2 so that no test matches them.
//   2. k_fs_faces, the fill: FluidSimulation::_advectVelocityFieldU/V/W
//      (fluidsimulation.cpp:2597-2730): faces bordering fluid keep n where
//      W > 1e-9 (isValueSet, :2575-2585), else the FP64 average of their 26
//      neighbours (|n| > 0 for U, :2630; isValueSet for V, W, :2675,2720);
//      other faces 0.  The snapshot takes that field; the field gets the
//      body force on faces bordering fluid (:2766-2805, 3306).  And the
//      classification: each face's extrapolation layer (at most one) and its
//      neighbours bordering the layer before, listed by layer per segment of
//      SEG faces.
//   3. k_fs_extrapolate, one launch per layer L that changes the listed faces
//      of layer L only: on both the snapshot and
//      the field (:3307, 3334), faces that border layer L, not layer L-1 and
//      no solid cell take the FP64 average of their 6 same-component
//      neighbours that border layer L-1, or 0 when that sum is 0
//      (macvelocityfield.cpp:616-760).  Within one layer the faces written
//      never border layer L-1 and the faces read always do, so the launch
//      reads only values of earlier layers, as the reference's in-place loop
//      does.
//
// Bound: latency and the passes over all faces, of which one is left (the
// fill reads two floats and writes two per face).  157x93x121, 5.3M faces,
// seven layers: 280 us with a launch over all cells per dilation (77), a fill
// (30), a classification (36) and a launch over all faces per layer (130); now
// 147: cell words 9, layers 16, faces 62, extrapolation 7 x 8.6.
//
// Everything here is integer work or a fixed-order FP64 sum per face:
// results are bit-identical to the sequential restatement.

#include "gfsx_internal.h"

#include <algorithm>

namespace gfsx {

namespace {

constexpr int8_t kSolid = -2;

inline unsigned blocks_for(int64_t n) {
    return (unsigned)std::max<int64_t>((n + kBlock - 1) / kBlock, 1);
}

__device__ __forceinline__ int8_t layer_at(const FsEpilogue &e, int i, int j, int k) {
    return e.layer[(uint32_t)i + (uint32_t)e.ni * ((uint32_t)j + (uint32_t)e.nj * (uint32_t)k)];
}

// the face of component c at (i,j,k) borders a cell whose layer is v
// (FluidMaterialGrid::isFaceBorderingMaterialU/V/W, fluidmaterialgrid.cpp:119-143)
__device__ __forceinline__ bool face_borders(const FsEpilogue &e, int c, int i, int j, int k,
                                             int v) {
    const int a = c == 0 ? i : (c == 1 ? j : k);
    const int na = c == 0 ? e.ni : (c == 1 ? e.nj : e.nk);
    const int li = i - (c == 0), lj = j - (c == 1), lk = k - (c == 2);
    if (a == na) return layer_at(e, li, lj, lk) == v;
    if (a > 0) return layer_at(e, i, j, k) == v || layer_at(e, li, lj, lk) == v;
    return layer_at(e, i, j, k) == v;
}

// ---- the cell layers

namespace lay {
constexpr int H = 7;                       // layers per launch: the halo of a tile
constexpr int TX = 64 - 2 * H, TY = 8, TZ = 8;   // cells of a tile: rows of 64 bits with the halo
constexpr int RY = TY + 2 * H, RZ = TZ + 2 * H, ROWS = RY * RZ;
constexpr int NT = 512;
constexpr int AHEAD = 8;                   // rows a wave loads at a time
}  // namespace lay

// The state of cell (i,j,k) before any dilation: -3 outside the grid, kSolid,
// 0 fluid, -1 neither.
__device__ __forceinline__ int cell_state(const FsEpilogue &e, int i, int j, int k) {
    if ((unsigned)i >= (unsigned)e.ni || (unsigned)j >= (unsigned)e.nj || (unsigned)k >= (unsigned)e.nk)
        return -3;
    const uint32_t t = (uint32_t)i + (uint32_t)e.ni * ((uint32_t)j + (uint32_t)e.nj * (uint32_t)k);
    bool fluid;
    if (e.fluid) {
        // the cell's bit in its P2G brick's mask (brick bins: the 8 P2G
        // bricks of each G2P brick consecutive)
        const int bx = i >> 2, by = j >> 2, bz = k >> 2;
        const uint32_t g = (uint32_t)(bx >> 1) +
                           (uint32_t)e.gbx * ((uint32_t)(by >> 1) + (uint32_t)e.gby * (uint32_t)(bz >> 1));
        const uint32_t bin = e.kb0 + ((g << 3) | (uint32_t)((bx & 1) | ((by & 1) << 1) | ((bz & 1) << 2)));
        const int bit = (i & 3) + 4 * (j & 3) + 16 * (k & 3);
        fluid = (e.fluid[bin] >> bit) & 1ull;
    } else {
        // the cell's bin in the sort's padded bin grid
        const uint32_t b = (uint32_t)(i + 1) + (uint32_t)e.b[0] *
                           ((uint32_t)(j + 1) + (uint32_t)e.b[1] * (uint32_t)(k + 1));
        fluid = e.start[b + 1] > e.start[b];
    }
    if (e.solid && e.solid[t]) return kSolid;
    return fluid ? 0 : -1;
}

// The cells as bits, 64 along x to a word (nw words a row): fluid, or open
// (neither fluid nor solid); one wave per word, four words in flight.
__global__ __launch_bounds__(kBlock) void k_fs_pack(FsEpilogue e, uint32_t nw, uint32_t words) {
    constexpr int PER = 4;
    const int lane = threadIdx.x & 63;
    const uint32_t w0 = (blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)) * PER;
    int v[PER];
#pragma unroll
    for (int m = 0; m < PER; m++) {
        const uint32_t w = w0 + (uint32_t)m, row = w / nw;
        v[m] = w < words ? cell_state(e, (int)(w % nw) * 64 + lane, (int)(row % (uint32_t)e.nj),
                                      (int)(row / (uint32_t)e.nj))
                         : -3;
    }
#pragma unroll
    for (int m = 0; m < PER; m++) {
        const uint64_t fluid = __ballot(v[m] == 0), open = __ballot(v[m] == -1);
        if (lane == 0 && w0 + (uint32_t)m < words) e.bits[w0 + (uint32_t)m] = make_ulonglong2(fluid, open);
    }
}

// Layers l0 + 1 .. l0 + n (n <= H) of a tile of TX x TY x TZ cells.  A row of
// the tile with its halo is a 64-bit word along x, so a dilation is a few word
// operations per row; the halo is as deep as the dilations, so what is wrong
// at its rim never reaches the tile.  FIRST (l0 = 0): the cells' states come
// from k_fs_pack's words, and every cell is written; later launches
// start from the layers up to l0 (another tile may already have written
// deeper ones: such a cell counts as unreached here, as it is) and write the
// cells they reach.
template <bool FIRST>
__global__ __launch_bounds__(lay::NT) void k_fs_layers(FsEpilogue e, int l0, int n) {
    using namespace lay;
    __shared__ uint64_t s_open[ROWS];        // neither solid nor reached before
    __shared__ uint64_t s_r[H + 1][ROWS];    // reached after each dilation
    const int t = threadIdx.x, lane = t & 63, wid = t >> 6;
    const uint32_t tx = (uint32_t)(e.ni + TX - 1) / TX, ty = (uint32_t)(e.nj + TY - 1) / TY;
    const int x0 = (int)(blockIdx.x % tx) * TX, y0 = (int)(blockIdx.x / tx % ty) * TY,
              z0 = (int)(blockIdx.x / (tx * ty)) * TZ;
    if (FIRST) {
        if (t < ROWS) {
            // the row's 64 cells from x0 - H, out of two words
            const int j = y0 - H + t % RY, k = z0 - H + t / RY, x = x0 - H;
            const int nw = (e.ni + 63) / 64, w = x >> 6, sh = x & 63;
            const bool in = (unsigned)j < (unsigned)e.nj && (unsigned)k < (unsigned)e.nk;
            const size_t row = in ? (size_t)nw * ((size_t)j + (size_t)e.nj * (size_t)k) : 0;
            ulonglong2 lo = make_ulonglong2(0ull, 0ull), hi = lo;
            if (in && w >= 0) lo = e.bits[row + (size_t)w];
            if (in && w + 1 < nw && sh) hi = e.bits[row + (size_t)(w + 1)];
            s_r[0][t] = sh ? (lo.x >> sh) | (hi.x << (64 - sh)) : lo.x;
            s_open[t] = sh ? (lo.y >> sh) | (hi.y << (64 - sh)) : lo.y;
        }
    } else {
        for (int r0 = wid; r0 < ROWS; r0 += AHEAD * (NT / 64)) {
            int v[AHEAD];
#pragma unroll
            for (int m = 0; m < AHEAD; m++) {
                const int r = r0 + m * (NT / 64);
                const int i = x0 - H + lane, j = y0 - H + r % RY, k = z0 - H + r / RY;
                const bool in = r < ROWS && (unsigned)i < (unsigned)e.ni &&
                                (unsigned)j < (unsigned)e.nj && (unsigned)k < (unsigned)e.nk;
                v[m] = in ? (int)layer_at(e, i, j, k) : -3;
                if (v[m] > l0) v[m] = -1;
            }
#pragma unroll
            for (int m = 0; m < AHEAD; m++) {
                const int r = r0 + m * (NT / 64);
                const uint64_t in = __ballot(v[m] >= 0), open = __ballot(v[m] == -1);
                if (lane == 0 && r < ROWS) {
                    s_r[0][r] = in;
                    s_open[r] = open;
                }
            }
        }
    }
    __syncthreads();
    for (int s = 1; s <= n; s++) {
        if (t < ROWS) {
            const uint64_t *p = s_r[s - 1];
            const int y = t % RY, z = t / RY;
            const uint64_t w = p[t];
            uint64_t near = (w << 1) | (w >> 1);
            if (y > 0) near |= p[t - 1];
            if (y < RY - 1) near |= p[t + 1];
            if (z > 0) near |= p[t - RY];
            if (z < RZ - 1) near |= p[t + RY];
            s_r[s][t] = w | (near & s_open[t]);
        }
        __syncthreads();
    }
    for (int c = t; c < TX * TY * TZ; c += NT) {
        const int x = c % TX, y = (c / TX) % TY, z = c / (TX * TY);
        const int i = x0 + x, j = y0 + y, k = z0 + z;
        if (i >= e.ni || j >= e.nj || k >= e.nk) continue;
        const int r = (y + H) + RY * (z + H), b = x + H;
        int v = -1;
        if ((s_open[r] >> b) & 1ull) {
            // the dilation that reached the cell
            for (int s = n; s >= 1 && ((s_r[s][r] >> b) & 1ull); s--) v = l0 + s;
            if (!FIRST && v < 0) continue;
        } else {
            if (!FIRST) continue;
            v = ((s_r[0][r] >> b) & 1ull) ? 0 : kSolid;
        }
        e.layer[(uint32_t)i + (uint32_t)e.ni * ((uint32_t)j + (uint32_t)e.nj * (uint32_t)k)] = (int8_t)v;
    }
}

static_assert(lay::ROWS <= lay::NT, "a thread per row");

// ---- the faces

constexpr int SEG = 1024;   // faces of a segment: 10 bits of an entry, 6 of its neighbours

// The segment sg: its component, its first face and how many it has.
__device__ __forceinline__ int segment(const FsEpilogue &e, uint32_t sg, uint32_t &f0, uint32_t &nf) {
    const int c = sg < e.nseg[0] ? 0 : (sg < e.nseg[0] + e.nseg[1] ? 1 : 2);
    f0 = (sg - (c > 0 ? e.nseg[0] : 0u) - (c > 1 ? e.nseg[1] : 0u)) * (uint32_t)SEG;
    const uint32_t tot = (uint32_t)(e.ni + (c == 0)) * (uint32_t)(e.nj + (c == 1)) * (uint32_t)(e.nk + (c == 2));
    nf = min(tot - f0, (uint32_t)SEG);
    return c;
}

// The value before the forces of a face bordering fluid that W did not set:
// the mean of its set neighbours.
__device__ float mean_of_set(const FsEpilogue &e, int c, int i, int j, int k, const int d[3]) {
    const float *n = c == 0 ? e.n[0] : (c == 1 ? e.n[1] : e.n[2]);
    const float *w = c == 0 ? e.w[0] : (c == 1 ? e.w[1] : e.w[2]);
    double avg = 0.0, weight = 0.0;
    for (int nk = k - 1; nk <= k + 1; nk++)
        for (int nj = j - 1; nj <= j + 1; nj++)
            for (int ni = i - 1; ni <= i + 1; ni++) {
                if (ni == i && nj == j && nk == k) continue;
                if ((unsigned)ni >= (unsigned)d[0] || (unsigned)nj >= (unsigned)d[1] ||
                    (unsigned)nk >= (unsigned)d[2])
                    continue;
                const uint32_t g = (uint32_t)ni + (uint32_t)d[0] * ((uint32_t)nj + (uint32_t)d[1] * (uint32_t)nk);
                const float nv = n[g];
                const bool use = c == 0 ? fabsf(nv) > 0.0f : (double)w[g] > 1e-9;
                if (use) {
                    avg += (double)nv;
                    weight += 1.0;
                }
            }
    return weight > 0.0 ? (float)(avg / weight) : 0.0f;
}

// One work-group per segment: the fill of its faces, and the list of those
// with an extrapolation layer, grouped by layer (in any order inside one):
// entry = place in the segment | mask of the neighbours that border the layer
// before << 10; off[L - 1] .. off[L] the entries of layer L.
//
// The layer L at which a face is extrapolated: L borders it, L-1 does not, no
// solid does, 1 <= L <= layers (macvelocityfield.cpp:694-706).  A face borders
// at most two cells, so at most one L fits.
__global__ __launch_bounds__(kBlock) void k_fs_faces(FsEpilogue e) {
    constexpr int ITEMS = SEG / kBlock;
    constexpr int MAXL = 100;   // layers at most
    __shared__ uint32_t s_cnt[MAXL + 1];
    __shared__ uint32_t s_off[MAXL + 2];
    const int t = threadIdx.x;
    if (t <= MAXL) s_cnt[t] = 0u;
    uint32_t f0, nf;
    const int c = segment(e, blockIdx.x, f0, nf);
    const int d[3] = {e.ni + (c == 0), e.nj + (c == 1), e.nk + (c == 2)};
    const int na = c == 0 ? e.ni : (c == 1 ? e.nj : e.nk);
    float *grid = c == 0 ? e.grid[0] : (c == 1 ? e.grid[1] : e.grid[2]);
    float *old = c == 0 ? e.old[0] : (c == 1 ? e.old[1] : e.old[2]);
    const bool on = c == 0 ? e.grav_on[0] : (c == 1 ? e.grav_on[1] : e.grav_on[2]);
    const float gd = c == 0 ? e.grav_delta[0] : (c == 1 ? e.grav_delta[1] : e.grav_delta[2]);
    __syncthreads();
    const float *fn = c == 0 ? e.n[0] : (c == 1 ? e.n[1] : e.n[2]);
    const float *fw = c == 0 ? e.w[0] : (c == 1 ? e.w[1] : e.w[2]);
    // every item's cell layers, then values, are loaded before any is used
    int L[ITEMS], fi[ITEMS], fj[ITEMS], fk[ITEMS], lo[ITEMS], hi[ITEMS];
    uint32_t ent[ITEMS], rank[ITEMS];
    float val[ITEMS], wgt[ITEMS];
#pragma unroll
    for (int m = 0; m < ITEMS; m++) {
        const uint32_t l = (uint32_t)(t + m * kBlock);
        const uint32_t o = f0 + min(l, nf - 1u);
        const uint32_t row = o / (uint32_t)d[0];
        const int i = fi[m] = (int)(o - row * (uint32_t)d[0]);
        const int j = fj[m] = (int)(row % (uint32_t)d[1]), k = fk[m] = (int)(row / (uint32_t)d[1]);
        // the layers of the cells on either side (-3: no cell)
        const int a = c == 0 ? i : (c == 1 ? j : k);
        hi[m] = a < na ? layer_at(e, i, j, k) : -3;
        lo[m] = a > 0 ? layer_at(e, i - (c == 0), j - (c == 1), k - (c == 2)) : -3;
    }
#pragma unroll
    for (int m = 0; m < ITEMS; m++) {
        const uint32_t o = f0 + min((uint32_t)(t + m * kBlock), nf - 1u);
        const bool set = hi[m] == 0 || lo[m] == 0;
        val[m] = set ? gld(fn, o) : 0.0f;
        wgt[m] = set ? gld(fw, o) : 0.0f;
    }
#pragma unroll
    for (int m = 0; m < ITEMS; m++) {
        const uint32_t l = (uint32_t)(t + m * kBlock), o = f0 + l;
        L[m] = 0;
        if (l >= nf) continue;
        const bool set = hi[m] == 0 || lo[m] == 0;
        if (set && !((double)wgt[m] > 1e-9)) val[m] = mean_of_set(e, c, fi[m], fj[m], fk[m], d);
        gst(old, (size_t)o, val[m]);
        gst(grid, (size_t)o, set && on ? val[m] + gd : val[m]);
        if (hi[m] == kSolid || lo[m] == kSolid) continue;
        int f = 0;
        if (hi[m] >= 1 && lo[m] != hi[m] - 1) f = hi[m];
        if (lo[m] >= 1 && hi[m] != lo[m] - 1 && (f == 0 || lo[m] < f)) f = lo[m];
        if (f == 0 || f > e.layers) continue;
        uint32_t mask = 0;
        const int i = fi[m], j = fj[m], k = fk[m];
        const int nb[6][3] = {{i - 1, j, k}, {i + 1, j, k}, {i, j - 1, k},
                              {i, j + 1, k}, {i, j, k - 1}, {i, j, k + 1}};
#pragma unroll
        for (int q = 0; q < 6; q++) {
            const int x = nb[q][0], y = nb[q][1], z = nb[q][2];
            if ((unsigned)x >= (unsigned)d[0] || (unsigned)y >= (unsigned)d[1] ||
                (unsigned)z >= (unsigned)d[2])
                continue;
            if (face_borders(e, c, x, y, z, f - 1)) mask |= 1u << q;
        }
        L[m] = f;
        ent[m] = l | (mask << 10);
        rank[m] = atomicAdd(&s_cnt[f], 1u);
    }
    __syncthreads();
    if (t == 0) {
        uint32_t at = 0;
        for (int f = 1; f <= e.layers; f++) {
            s_off[f] = at;
            at += s_cnt[f];
        }
        s_off[e.layers + 1] = at;
    }
    __syncthreads();
    if (t <= e.layers) e.foff[(size_t)blockIdx.x * (size_t)(e.layers + 1) + t] = (uint16_t)s_off[t + 1];
#pragma unroll
    for (int m = 0; m < ITEMS; m++)
        if (L[m] > 0) e.fent[(size_t)blockIdx.x * SEG + s_off[L[m]] + rank[m]] = (uint16_t)ent[m];
}

// one layer: every face of layer L takes the FP64 average of its masked
// neighbours (in the order -x, +x, -y, +y, -z, +z), 0 when that sum is 0,
// on both grids; one work-group per segment (a segment along the fluid's
// surface can lie in one layer whole)
__global__ __launch_bounds__(kBlock) void k_fs_extrapolate(FsEpilogue e, int L) {
    const uint32_t sg = blockIdx.x;
    const uint16_t *off = e.foff + (size_t)sg * (size_t)(e.layers + 1);
    const uint32_t e0 = off[L - 1], e1 = off[L];
    if (e0 == e1) return;
    uint32_t f0, nf;
    const int c = segment(e, sg, f0, nf);
    const uint32_t d0 = (uint32_t)(e.ni + (c == 0)), d1 = (uint32_t)(e.nj + (c == 1));
    const uint32_t step[3] = {1u, d0, d0 * d1};
    float *grid = c == 0 ? e.grid[0] : (c == 1 ? e.grid[1] : e.grid[2]);
    float *old = c == 0 ? e.old[0] : (c == 1 ? e.old[1] : e.old[2]);
    for (uint32_t n = e0 + threadIdx.x; n < e1; n += kBlock) {
        const uint32_t cl = e.fent[(size_t)sg * SEG + n];
        const uint32_t o = f0 + (cl & (uint32_t)(SEG - 1)), mask = cl >> 10;
        double sg_ = 0.0, so = 0.0, cnt = 0.0;
#pragma unroll
        for (int q = 0; q < 6; q++) {
            if (!(mask & (1u << q))) continue;
            const uint32_t g = (q & 1) ? o + step[q >> 1] : o - step[q >> 1];
            sg_ += (double)grid[g];
            so += (double)old[g];
            cnt += 1.0;
        }
        grid[o] = sg_ == 0.0 ? 0.0f : (float)(sg_ / cnt);
        old[o] = so == 0.0 ? 0.0f : (float)(so / cnt);
    }
}

// ---- collision fix (fluidsimulation.cpp:3145-3207, collision.cpp:303-449)
// FP32 vec3 and FP64 scalar maths as the reference evaluates them; products
// and sums are rounded one by one (no fused multiply-add), as on the CPU.

__device__ __forceinline__ bool solid_at(const FsEpilogue &e, int i, int j, int k) {
    return (unsigned)i < (unsigned)e.ni && (unsigned)j < (unsigned)e.nj &&
           (unsigned)k < (unsigned)e.nk &&
           e.solid[(uint32_t)i + (uint32_t)e.ni * ((uint32_t)j + (uint32_t)e.nj * (uint32_t)k)] != 0;
}

// Grid3d::positionToGridIndex then the solid test; out of the grid is not solid
__device__ __forceinline__ bool point_in_solid(const FsEpilogue &e, float x, float y, float z) {
    const double inv = 1.0 / e.dx;
    const double fi = floor(__dmul_rn((double)x, inv));
    const double fj = floor(__dmul_rn((double)y, inv));
    const double fk = floor(__dmul_rn((double)z, inv));
    if (!(fi >= 0.0 && fj >= 0.0 && fk >= 0.0 && fi < e.ni && fj < e.nj && fk < e.nk)) return false;
    return solid_at(e, (int)fi, (int)fj, (int)fk);
}

// Collision::getLineSegmentVoxelIntersection: the first solid voxel on p0 -> p1
__device__ bool segment_voxel(const FsEpilogue &e, const float a[3], const float b[3], int vox[3]) {
    const float invdx = (float)(1.0 / e.dx);
    float p0[3], p1[3];
    for (int c = 0; c < 3; c++) {
        p0[c] = __fmul_rn(a[c], invdx);
        p1[c] = __fmul_rn(b[c], invdx);
    }
    int g0[3], g1[3], sgn[3];
    for (int c = 0; c < 3; c++) {
        g0[c] = (int)floor((double)p0[c]);
        g1[c] = (int)floor((double)p1[c]);
        sgn[c] = g1[c] > g0[c] ? 1 : g1[c] < g0[c] ? -1 : 0;
    }
    double v[3];
    for (int c = 0; c < 3; c++)
        v[c] = p1[c] == p0[c] ? 1.0 : (double)__fsub_rn(p1[c], p0[c]);
    const double vxvy = __dmul_rn(v[0], v[1]), vxvz = __dmul_rn(v[0], v[2]);
    const double vyvz = __dmul_rn(v[1], v[2]);
    const double gp0 = g0[0] + (g1[0] > g0[0] ? 1 : 0);
    const double gp1 = g0[1] + (g1[1] > g0[1] ? 1 : 0);
    const double gp2 = g0[2] + (g1[2] > g0[2] ? 1 : 0);
    double errx = __dmul_rn(__dsub_rn(gp0, (double)p0[0]), vyvz);
    double erry = __dmul_rn(__dsub_rn(gp1, (double)p0[1]), vxvz);
    double errz = __dmul_rn(__dsub_rn(gp2, (double)p0[2]), vxvy);
    const double derrx = __dmul_rn((double)sgn[0], vyvz);
    const double derry = __dmul_rn((double)sgn[1], vxvz);
    const double derrz = __dmul_rn((double)sgn[2], vxvy);
    int gx = g0[0], gy = g0[1], gz = g0[2];
    // the walk reaches the end voxel in |dgx| + |dgy| + |dgz| steps
    const long long steps = llabs((long long)g1[0] - g0[0]) + llabs((long long)g1[1] - g0[1]) +
                            llabs((long long)g1[2] - g0[2]) + 1;
    for (long long it = 0; it <= steps; it++) {
        if (solid_at(e, gx, gy, gz)) {
            vox[0] = gx;
            vox[1] = gy;
            vox[2] = gz;
            return true;
        }
        if (gx == g1[0] && gy == g1[1] && gz == g1[2]) break;
        const double xr = fabs(errx), yr = fabs(erry), zr = fabs(errz);
        if (sgn[0] != 0 && (sgn[1] == 0 || xr < yr) && (sgn[2] == 0 || xr < zr)) {
            gx += sgn[0];
            errx = __dadd_rn(errx, derrx);
        } else if (sgn[1] != 0 && (sgn[2] == 0 || yr < zr)) {
            gy += sgn[1];
            erry = __dadd_rn(erry, derry);
        } else if (sgn[2] != 0) {
            gz += sgn[2];
            errz = __dadd_rn(errz, derrz);
        }
    }
    return false;
}

// Collision::rayIntersectsAABB, with the reference's test of dir.x where
// dir.z is clamped
__device__ bool ray_aabb(const float p0[3], const float d[3], const float bmin[3],
                         const float bmax[3], float hit[3]) {
    const double eps = 1e-10;
    float dir[3] = {d[0], d[1], d[2]};
    if (fabs((double)dir[0]) < eps) dir[0] = dir[0] < 0 ? (float)-eps : (float)eps;
    if (fabs((double)dir[1]) < eps) dir[1] = dir[1] < 0 ? (float)-eps : (float)eps;
    if (fabs((double)dir[0]) < eps) dir[2] = dir[2] < 0 ? (float)-eps : (float)eps;
    float inv[3];
    for (int c = 0; c < 3; c++) inv[c] = (float)(1.0 / (double)dir[c]);
    double tmin = 0.0, tmax = 0.0;
    for (int c = 0; c < 3; c++) {
        const double t1 = (double)__fmul_rn(__fsub_rn(bmin[c], p0[c]), inv[c]);
        const double t2 = (double)__fmul_rn(__fsub_rn(bmax[c], p0[c]), inv[c]);
        if (c == 0) {
            tmin = fmin(t1, t2);
            tmax = fmax(t1, t2);
        } else {
            tmin = fmax(tmin, fmin(t1, t2));
            tmax = fmin(tmax, fmax(t1, t2));
        }
    }
    if (tmax > fmax(tmin, 0.0)) {
        const float tf = (float)tmin;
        for (int c = 0; c < 3; c++) hit[c] = __fadd_rn(p0[c], __fmul_rn(dir[c], tf));
        return true;
    }
    return false;
}

__global__ __launch_bounds__(kBlock) void k_fs_collide(FsEpilogue e) {
    const int64_t p = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    if (p >= e.np) return;
    float b[3] = {e.x1[0][p], e.x1[1][p], e.x1[2][p]};
    if (!point_in_solid(e, b[0], b[1], b[2])) return;
    const int64_t p0 = e.x0_perm ? (int64_t)e.x0_perm[p] : p;
    const float a[3] = {e.x0[0][p0], e.x0[1][p0], e.x0[2][p0]};
    float r[3] = {a[0], a[1], a[2]};
    int vox[3];
    if (segment_voxel(e, a, b, vox)) {
        float d[3];
        for (int c = 0; c < 3; c++) d[c] = __fsub_rn(b[c], a[c]);
        const float lsq = __fadd_rn(__fadd_rn(__fmul_rn(d[0], d[0]), __fmul_rn(d[1], d[1])),
                                    __fmul_rn(d[2], d[2]));
        const float len = (float)sqrt((double)lsq);
        const float inv = (float)(1.0 / (double)len);
        float rn[3], bmin[3], bmax[3], hit[3];
        for (int c = 0; c < 3; c++) {
            rn[c] = __fmul_rn(d[c], inv);
            bmin[c] = (float)__dmul_rn((double)(float)vox[c], e.dx);
            bmax[c] = __fadd_rn(bmin[c], (float)e.dx);
        }
        if (ray_aabb(a, rn, bmin, bmax, hit)) {
            const float back = (float)(0.05 * e.dx);
            float q[3];
            for (int c = 0; c < 3; c++) q[c] = __fsub_rn(hit[c], __fmul_rn(rn[c], back));
            if (!point_in_solid(e, q[0], q[1], q[2]))
                for (int c = 0; c < 3; c++) r[c] = q[c];
        }
    }
    for (int c = 0; c < 3; c++) e.x1[c][p] = r[c];
}

}  // namespace

void fs_collide(const FsEpilogue &e, hipStream_t s) {
    if (e.np <= 0 || !e.solid) return;
    hipLaunchKernelGGL(k_fs_collide, dim3(blocks_for(e.np)), dim3(kBlock), 0, s, e);
    GFSX_LAUNCH_CHECK();
}

uint32_t fs_segments(FsEpilogue &e) {
    uint32_t all = 0;
    for (int c = 0; c < 3; c++) {
        const int64_t nf = (int64_t)(e.ni + (c == 0)) * (e.nj + (c == 1)) * (e.nk + (c == 2));
        e.nseg[c] = (uint32_t)((nf + SEG - 1) / SEG);
        all += e.nseg[c];
    }
    return all;
}

size_t fs_words(const FsEpilogue &e) { return (size_t)((e.ni + 63) / 64) * (size_t)e.nj * (size_t)e.nk; }

size_t fs_entries(const FsEpilogue &e) {
    return (size_t)(e.nseg[0] + e.nseg[1] + e.nseg[2]) * SEG;
}

void fs_epilogue(const FsEpilogue &e, hipStream_t s) {
    auto tiles = [](int n, int t) { return (unsigned)((n + t - 1) / t); };
    const dim3 grid(tiles(e.ni, lay::TX) * tiles(e.nj, lay::TY) * tiles(e.nk, lay::TZ));
    const uint32_t nw = tiles(e.ni, 64), words = (uint32_t)fs_words(e);
    hipLaunchKernelGGL(k_fs_pack, dim3(blocks_for((int64_t)words * 16)), dim3(kBlock), 0, s, e, nw, words);
    GFSX_LAUNCH_CHECK();
    for (int l0 = 0; l0 < e.layers; l0 += lay::H) {
        hipLaunchKernelGGL(l0 == 0 ? k_fs_layers<true> : k_fs_layers<false>, grid, dim3(lay::NT), 0, s,
                           e, l0, std::min(e.layers - l0, lay::H));
        GFSX_LAUNCH_CHECK();
    }
    const uint32_t nseg = e.nseg[0] + e.nseg[1] + e.nseg[2];
    hipLaunchKernelGGL(k_fs_faces, dim3(nseg), dim3(kBlock), 0, s, e);
    GFSX_LAUNCH_CHECK();
    // a layer's launch changes only faces of that layer and reads only faces
    // bordering the layer before
    for (int L = 1; L <= e.layers; L++) {
        hipLaunchKernelGGL(k_fs_extrapolate, dim3(nseg), dim3(kBlock), 0, s, e, L);
        GFSX_LAUNCH_CHECK();
    }
}

}  // namespace gfsx
