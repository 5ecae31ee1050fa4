// region.hip -- the stages around the bilateral filter in
// okano_3_0/SimpleRegionDetect.cu:287-312: LocalCluster before it and
// ConnectRegion after it, for gfx950.
//
// LocalCluster (okano_3_0/LocalCluster.cu:45-153): the reference spreads a
// pixel's eight directional walks over eight threads and a shared array.  Here
// one lane per pixel makes the walks' first step, which settles most pixels,
// and eight lanes run the walks of each other one; the averages are formed and
// summed with the same FP32 operations in the same order (-ffp-contract=off,
// IEEE division), so the u8 result is the reference's.
// The reference addresses every read as data + y * pitch + x from the ROI
// origin and its walks reach 2 (pntRange - 1) pixels from the centre while
// the guard band is pntRange + 2 wide; reads here use the same linear
// address, clamped into the allocation the caller declares.  A workgroup
// stages its tile of 64 columns and 16, 32 or 64 rows plus the walks' reach in
// LDS by that rule; for reaches too large for LDS one lane walks all eight
// directions of a pixel in global memory.
//
// ConnectRegion (okano_3_0/ConnectRegion.cu:789-1043): 8-connected
// components of pixels whose gray values lie in [minGray, maxGray], each
// labelled by its minimum raster index.  The reference gets there with
// shared-memory labelling per block and rounds of border merging; here the
// runs of each 64 x 64 tile are labelled in LDS, which leaves a handful of
// tile-local roots, then the runs that touch across tile edges join those by a
// lock-free union-find pass in global memory (atomicMin on roots, parents
// always smaller than children, so every loop ends), then each tile-local root
// is pointed at its global root and its area added there -- the result does
// not depend on the order the unions run in.  No pass keeps a label per pixel.
// The area filter, the raster-order
// renumbering and the u8 output follow the reference, including its area
// launch covering only rows below 256 * ceil(floor((H + 4) / 32) / 8)
// (ConnectRegion.cu:45, :957-967) and never dropping a root whose counted
// area is 0.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>

#include "bf_internal.h"

namespace bfimpl {
namespace region {

// ------------------------------------------------------------ LocalCluster

struct LcArgs {
    const uint8_t *in;        // ROI origin
    int64_t pitch;
    int64_t lo, hi;           // readable byte offsets from `in`: [lo, hi)
    uint8_t *out;
    int64_t out_pitch;
    int W, H;
    int pnt_range, pnt_count;
    float gap, diffe;
    int pro_black, pro_white;
};

__device__ __forceinline__ uint32_t lc_read(const LcArgs &a, int y, int x)
{
    int64_t off = (int64_t)y * a.pitch + x;
    off = off < a.lo ? a.lo : (off >= a.hi ? a.hi - 1 : off);
    return a.in[off];
}

__device__ __forceinline__ uint8_t lc_sat_u8(float q)
{
    if (!(q > 0.0f)) return 0;
    if (q >= 255.0f) return 255;
    return (uint8_t)(int)q;
}

// The filter of one pixel (x, y) whose value is cv; rd(dx, dy) returns the
// byte at (x + dx, y + dy) by the linear-address rule of lc_read.
template <typename Read>
__device__ __forceinline__ uint8_t lc_pixel(const LcArgs &a, int x, int y, uint32_t cv, Read rd)
{
    const int sx = a.pnt_range + 2, ex = a.W - a.pnt_range - 2;
    const int sy = a.pnt_range + 2, ey = a.H - a.pnt_range - 2;
    if (x < sx || x > ex || y < sy || y > ey || (int)cv <= a.pro_black || (int)cv >= a.pro_white)
        return (uint8_t)cv;
    // directions {dx, dy} of LocalCluster.cu:14-19
    const int ddx_t[8] = { 1, 1, 0, -1, -1, -1, 0, 1 };
    const int ddy_t[8] = { 0, -1, -1, -1, 0, 1, 1, 1 };
    const float fcv = (float)cv;
    float temp[8];
#pragma unroll
    for (int z = 0; z < 8; z++) {
        const int ddx = ddx_t[z], ddy = ddy_t[z];
        uint32_t cuv = rd(ddx, ddy);
        uint32_t pre1 = rd(-ddx, -ddy);
        uint32_t pre2 = cv;
        uint32_t latt1 = rd(2 * ddx, 2 * ddy);
        float sum = fcv;
        int i, k = 0;
        for (i = 1; i < a.pnt_range; i++) {
            if (fabsf(fcv - (float)cuv) > a.gap) break;
            k += 2;
            const uint32_t latt2 = rd(k * ddx, k * ddy);
            const float side1 = (float)(pre1 + pre2);
            const float side2 = (float)(latt1 + latt2);
            if (fabsf(side1 - side2) > a.diffe) break;
            pre1 = pre2;
            pre2 = cuv;
            cuv = latt1;
            latt1 = latt2;
            sum += (float)cuv;
        }
        temp[z] = sum / (float)i;
    }
    int mark = 0;
    for (int j = 8 - a.pnt_count; j > 0; j--) {
#pragma unroll
        for (int i = 0; i < 8; i++)
            if (fabsf(temp[i] - fcv) >= fabsf(temp[mark] - fcv)) mark = i;
#pragma unroll
        for (int i = 0; i < 8; i++) temp[i] = i == mark ? fcv : temp[i];
    }
    float sumag = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; j++) sumag += temp[j];
    sumag -= (float)((8 - a.pnt_count) * (int)cv);
    const float q = sumag / (float)a.pnt_count;
    return q > 255.0f ? 255 : lc_sat_u8(q);
}

// Every read straight from global memory (any pntRange).
__global__ void __launch_bounds__(256) local_cluster_kernel(LcArgs a)
{
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= a.W || y >= a.H) return;
    a.out[(int64_t)y * a.out_pitch + x] =
        lc_pixel(a, x, y, lc_read(a, y, x),
                 [&](int dx, int dy) { return lc_read(a, y + dy, x + dx); });
}

// A 64 x th tile with a halo of `halo` = 2 (pntRange - 1) pixels (the walks'
// reach) staged in LDS by lc_read's address rule, so every read sees the
// byte the global-read kernel would.
//
// The eight walks of a pixel end on their first step far more often than
// not (noise sigma 10 against gap and diffe 10: four of five), and a walk
// that ends there leaves the average at the centre's value.  With 1 <=
// pntCount <= 8 the 8 - pntCount averages furthest from the centre are
// replaced by it, so a pixel with no more surviving walks than that is
// (8 cv - (8 - n) cv) / n = cv, exactly.  Phase 1 therefore only makes the
// first step's two tests (integers: every operand is a sum of bytes, so the
// comparisons are the floating ones), one pixel per lane, writes those
// pixels and queues the others in LDS.  Phase 2 runs the queued pixels with
// eight lanes each, one per direction, so that the walks of a pixel and of
// its neighbours in the queue proceed together; the lanes' averages are
// ranked and summed across the eight lanes with DPP moves.
// Bound by VALU issue: one lane walking the eight directions of a pixel in
// turn paid every direction's longest walk among 64 pixels and nine
// divisions (about 1,290 issue slots per 64 pixels; 198 here, VALU 72% busy).
// 2048 x 1536, pntRange 8, noise 10: 114 -> 26 us a call.  Eight waves per
// workgroup measured 26.4 us, four 27.2, sixteen 35.3.
constexpr int kLcTw = 64, kLcThMax = 64, kLcWaves = 8;
constexpr int64_t kLcMaxLds = 48 * 1024;   // larger halos read global memory

// value of lane (lane ^ X) within each group of eight lanes, X = 1..7
template <int X>
__device__ __forceinline__ int lc_xor8(int v)
{
    if constexpr (X >= 4) v = __builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, true);   // lane ^ 7
    constexpr int Q = X >= 4 ? (X ^ 7) : X;                                           // quad part
    if constexpr (Q == 1) v = __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);
    if constexpr (Q == 2) v = __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);
    if constexpr (Q == 3) v = __builtin_amdgcn_mov_dpp(v, 0x1B, 0xF, 0xF, true);
    return v;
}

// value of lane K of each quad
template <int K>
__device__ __forceinline__ float lc_quad_bcast(float v)
{
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), K * 0x55, 0xF, 0xF, true));
}

// 1 when lane ^ X is replaced before this lane: further from the centre
// (distances as the bits of non-negative floats), or as far and later in
// direction order (later = 1 when direction z ^ X comes after z).
template <int X>
__device__ __forceinline__ int lc_before(int dev, int later)
{
    return lc_xor8<X>(dev) + later > dev ? 1 : 0;
}

// SP: staged bytes per row (64 columns and both halos).
template <int SP>
__global__ void __launch_bounds__(64 * kLcWaves) local_cluster_lds_kernel(LcArgs a, int halo, int th)
{
    extern __shared__ __align__(16) uint8_t s_img[];
    const int sh = th + 2 * halo;
    uint16_t *queue = reinterpret_cast<uint16_t *>(s_img + SP * sh);
    int *qcount = reinterpret_cast<int *>(queue + kLcTw * th);
    const int x0 = blockIdx.x * kLcTw, y0 = blockIdx.y * th;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (threadIdx.x == 0) *qcount = 0;
    // Row r of the tile is the linear range from (y0 - halo + r, x0 - halo).
    // A row inside the allocation is read as aligned dwords (the second of a
    // pair only where the row is misaligned: it then holds a wanted byte);
    // any other is clamped byte by byte as in lc_read.
    const int need = kLcTw + 2 * halo;                // bytes of a row that can be read
    for (int r = wave; r < sh; r += kLcWaves) {
        const int64_t row = (int64_t)(y0 - halo + r) * a.pitch + (x0 - halo);
        if (row >= a.lo && row + SP <= a.hi) {
            const uintptr_t p = reinterpret_cast<uintptr_t>(a.in + row);
            const uint32_t mis = (uint32_t)(p & 3);
            const uint32_t *src = reinterpret_cast<const uint32_t *>(p - mis);
#pragma unroll
            for (int c = lane; c < SP / 4; c += 64) {
                const uint32_t lo = src[c], hi = src[c + (mis ? 1 : 0)];
                *reinterpret_cast<uint32_t *>(s_img + r * SP + 4 * c) =
                    __builtin_amdgcn_alignbyte(hi, lo, mis);
            }
        } else {
            for (int c = lane; c < need; c += 64) {
                int64_t off = row + c;
                off = off < a.lo ? a.lo : (off >= a.hi ? a.hi - 1 : off);
                s_img[r * SP + c] = a.in[off];
            }
        }
    }
    __syncthreads();
    const uint32_t gap = (uint32_t)a.gap, diffe = (uint32_t)a.diffe;
    // surviving walks a pixel may have and still be its own value
    const int spare = a.pnt_count >= 1 && a.pnt_count <= 8 ? 8 - a.pnt_count : -1;
    const int x = x0 + lane;
    const bool xin = x >= a.pnt_range + 2 && x <= a.W - a.pnt_range - 2 && x < a.W;
    const uint32_t gap_bias = 0x7FFFFFFFu - gap, diffe_bias = 0x7FFFFFFFu - diffe;
    uint8_t *orow = a.out + (int64_t)(y0 + wave) * a.out_pitch + x;
    for (int ly = wave; ly < th; ly += kLcWaves, orow += kLcWaves * a.out_pitch) {
        const int y = y0 + ly;
        if (y >= a.H) break;                          // whole waves
        // the 5 x 5 window from its top-left corner
        const uint8_t *w = s_img + (ly + halo - 2) * SP + lane + halo - 2;
        const uint32_t cv = w[2 * SP + 2];
        constexpr int dxs[8] = { 1, 1, 0, -1, -1, -1, 0, 1 }, dys[8] = { 0, -1, -1, -1, 0, 1, 1, 1 };
        uint32_t n1[8], n2[8], ended = 0;
#pragma unroll
        for (int z = 0; z < 8; z++) {
            n1[z] = w[(2 + dys[z]) * SP + 2 + dxs[z]];
            n2[z] = w[(2 + 2 * dys[z]) * SP + 2 + 2 * dxs[z]];
        }
        // a test that fails carries its sum past 2^31: the larger sum's top
        // bit says whether the walk ended
#pragma unroll
        for (int z = 0; z < 8; z++) {
            const uint32_t g = __builtin_amdgcn_sad_u16(cv, n1[z], gap_bias);
            const uint32_t d = __builtin_amdgcn_sad_u16(cv + n1[(z + 4) & 7], 2 * n2[z], diffe_bias);
            ended = __builtin_amdgcn_alignbit(ended, g > d ? g : d, 31);
        }
        const int alive = a.pnt_range <= 1 ? 0 : 8 - __popc(ended);   // no steps: every average is cv
        const bool more = xin && y >= a.pnt_range + 2 && y <= a.H - a.pnt_range - 2 &&
                          (int)cv > a.pro_black && (int)cv < a.pro_white && alive > spare;
        const uint64_t m = __ballot(more);
        if (m) {
            int at = 0;
            if (lane == 0) at = atomicAdd(qcount, __popcll(m));
            at = __builtin_amdgcn_readfirstlane(at);
            const int before = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
            if (more) queue[at + before] = (uint16_t)(ly * kLcTw + lane);
        }
        if (!more && x < a.W) *orow = (uint8_t)cv;
    }
    __syncthreads();
    const int nq = __builtin_amdgcn_readfirstlane(*qcount);
    const int z = lane & 7;                           // this lane's direction
    const int zy = z == 0 || z == 4 ? 0 : (z < 4 ? -1 : 1);
    const int zx = z == 2 || z == 6 ? 0 : (z < 2 || z == 7 ? 1 : -1);
    const int dir = zy * SP + zx;
    const int l1 = z & 1 ? 0 : 1, l2 = z & 2 ? 0 : 1, l4 = z & 4 ? 0 : 1;
    for (int q0 = wave * 8; q0 < nq; q0 += 8 * kLcWaves) {      // whole waves
        const int q = q0 + (lane >> 3);
        const int e = queue[q < nq ? q : nq - 1];
        int pos = (e / kLcTw + halo) * SP + (e & (kLcTw - 1)) + halo;
        const uint32_t cv = s_img[pos];
        const float fcv = (float)cv;
        uint32_t cuv = s_img[pos + dir], pre1 = s_img[pos - dir], pre2 = cv;
        uint32_t latt1 = s_img[pos + 2 * dir], sum = cv;
        int i;
        for (i = 1; i < a.pnt_range; i++) {
            if (__builtin_amdgcn_sad_u16(cv, cuv, 0) > gap) break;
            pos += 2 * dir;
            const uint32_t latt2 = s_img[pos];
            if (__builtin_amdgcn_sad_u16(pre1 + pre2, latt1 + latt2, 0) > diffe) break;
            pre1 = pre2;
            pre2 = cuv;
            cuv = latt1;
            latt1 = latt2;
            sum += cuv;
        }
        float temp = (float)sum / (float)i;
        const int dev = __float_as_int(fabsf(temp - fcv));
        // Rounds that each replace the last of the furthest averages take
        // them in (distance, direction) order: this lane's place in it.
        const int rank = lc_before<1>(dev, l1) + lc_before<2>(dev, l2) + lc_before<3>(dev, l2) +
                         lc_before<4>(dev, l4) + lc_before<5>(dev, l4) + lc_before<6>(dev, l4) +
                         lc_before<7>(dev, l4);
        if (rank < 8 - a.pnt_count) temp = fcv;
        // the eight averages in direction order, from 0 (valid in lanes 0..3
        // of each group)
        const float rev = __int_as_float(lc_xor8<7>(__float_as_int(temp)));
        float sumag = 0.0f;
        sumag += lc_quad_bcast<0>(temp);
        sumag += lc_quad_bcast<1>(temp);
        sumag += lc_quad_bcast<2>(temp);
        sumag += lc_quad_bcast<3>(temp);
        sumag += lc_quad_bcast<3>(rev);
        sumag += lc_quad_bcast<2>(rev);
        sumag += lc_quad_bcast<1>(rev);
        sumag += lc_quad_bcast<0>(rev);
        sumag -= (float)((8 - a.pnt_count) * (int)cv);
        const float v = sumag / (float)a.pnt_count;
        if (z == 0 && q < nq)
            a.out[(int64_t)(y0 + e / kLcTw) * a.out_pitch + x0 + (e & (kLcTw - 1))] =
                v > 255.0f ? 255 : lc_sat_u8(v);
    }
}

// ----------------------------------------------------------- ConnectRegion

__device__ __forceinline__ int cr_load(const int *L, int i)
{
    return __hip_atomic_load(L + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Root of x, pointing x further up at every step of the walk: a region
// that spans many tiles starts as long chains of their roots, and as every
// union re-points the node it starts from, the walks double their stride as
// they go (path halving, which re-points each visited node once, took 26.3
// us for the border pass of a 4096 x 4096 image, this 24.6).  Parents are never larger than their children, so the walk ends,
// and a node is only ever pointed at an ancestor it keeps (trees only ever
// merge).  A hook another lane makes meanwhile on x could be overwritten,
// but x was no longer a root, so that lane's union loop does not stop there
// and merges the trees through x's former parent.
__device__ __forceinline__ int cr_find_pull(int *L, int x)
{
    int p = cr_load(L, x);
    if (p == x) return x;
    while (true) {
        const int gp = cr_load(L, p);
        if (gp == p) return p;
        __hip_atomic_store(L + x, gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        p = gp;
    }
}

// Lock-free union (the larger root is hooked under the smaller one with
// atomicMin; a failed hook means that root was hooked meanwhile, and the
// loop continues from its new parent, a strictly smaller index).
__device__ void cr_unite(int *L, int a, int b)
{
    while (true) {
        a = cr_find_pull(L, a);
        b = cr_find_pull(L, b);
        if (a == b) return;
        if (a < b) {
            const int old = atomicMin(L + b, a);
            if (old == b) return;
            b = old;
        } else {
            const int old = atomicMin(L + a, b);
            if (old == a) return;
            a = old;
        }
    }
}

struct CrArgs {
    const uint8_t *in;
    int64_t pitch;
    uint8_t *out;
    int64_t out_pitch;
    int W, H;
    int tiles_x;
    int runs;                 // run entries of a tile row (most it can hold)
    int min_gray, max_gray;
    int min_area, max_area;
    int covered;              // rows the area count covers
    uint64_t *fg;             // per row and tile: foreground pixels
    uint64_t *root;           // likewise: tile-local roots
    uint64_t *kept;           // likewise: global roots the area filter keeps
    uint16_t *run_root;       // per row, tile and run: its root's index in the tile
    int *parent;              // per pixel, set at tile-local roots only
    int *area;                // likewise: the area, later the u8 number
    int *rowcount;            // kept roots of a row
};

__device__ __forceinline__ bool cr_fg(const CrArgs &a, uint32_t v)
{
    return (int)v >= a.min_gray && (int)v <= a.max_gray;
}

__device__ __forceinline__ bool cr_kept_area(const CrArgs &a, int ar)
{
    return !(ar != 0 && (ar < a.min_area || ar > a.max_area));
}

// Labels work on 64 x 64 tiles and, inside them, on runs: a tile row is a
// 64-bit foreground mask and a 16-bit root for each of its runs (at most
// 32).  A tile of 4,096 pixels has a handful of roots, so the passes after
// the tile pass (unions across tile edges, areas, numbers) touch a few
// thousand words; no pass reads or writes a label per pixel, and the output
// pass finds a pixel's run by counting run starts in its row's mask.  A
// pixel outside the gray range is a region of its own: it takes part (as a
// root without runs) only where its area, 1, or 0 in the rows the reference
// does not count, is kept.
constexpr int kCrT = 64;
constexpr int kCrRuns = kCrT / 2;
constexpr int kCrMaxRows = 1 << 26;     // rows are refused from here on (64 threads a row: 2^32)
constexpr int kCrRow = kCrRuns + 1;      // run entries of a row in LDS (odd: rows fall in different banks)

__device__ __forceinline__ int lds_load(const int *L, int i)
{
    return __hip_atomic_load(L + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Lock-free union of the trees that a and b lie in: both walks take a step
// at a time together, and end as soon as they meet (cr_unite's rule on LDS).
__device__ void l_unite(int *L, int a, int b)
{
    while (a != b) {
        const int pa = lds_load(L, a), pb = lds_load(L, b);
        if (pa != a || pb != b) {
            a = pa;
            b = pb;
        } else if (a < b) {
            const int old = atomicMin(L + b, a);
            if (old == b) return;
            b = old;
        } else {
            const int old = atomicMin(L + a, b);
            if (old == a) return;
            a = old;
        }
    }
}

__device__ __forceinline__ uint64_t cr_starts(uint64_t m) { return m & ~(m << 1); }

// Columns (as bits) of row u that touch the run of row m starting at bit
// `s` (a single set bit), diagonals included.
__device__ __forceinline__ uint64_t cr_touched(uint64_t m, uint64_t u, uint64_t s)
{
    const uint64_t run = m & ~(m + s) & ~(s - 1);   // the carry clears the run that starts at s
    return u & (run | (run << 1) | (run >> 1));
}

// Index of the run of row m that holds the lowest bit of t (t within m).
__device__ __forceinline__ int cr_run_of(uint64_t m, uint64_t t)
{
    return __popcll(cr_starts(m) & (t ^ (t - 1))) - 1;
}

// Tile pass.  Rows become masks (16 pixels a thread), and four threads a row
// walk its runs.  Every run hooks onto the first run above that it touches,
// with a plain store, and pointer jumping points each run at its tree's
// root; what is left are the runs that touch a second run above, whose
// unions find both roots at once.  Runs are numbered in raster order, so a
// root is the component's first run.  A tile whose rows hold at most one run
// each (most tiles of an image are inside one region) needs none of that: a
// row's component starts at the last row above it that touches nothing,
// which a ballot over the rows tells.
// (Bound by LDS latency.  4096 x 4096 with quiet noise, a band of it around
// the gray limit: 28 us, 17 us where nothing is noise; uniting all rows at
// once through chains of up to 64 links took 82 us, a lane per pixel with
// these hooks 80 us, and a lane per row 78 us.)
__global__ void __launch_bounds__(256) cr_local_kernel(CrArgs a)
{
    __shared__ int loc[kCrT * kCrRow];             // parent run of a run
    __shared__ uint32_t cnt[kCrT * kCrRow / 2];    // areas, two 16-bit sums per word
    __shared__ uint8_t col[kCrT * kCrRow];         // a run's first column
    __shared__ uint64_t mask[kCrT];                // foreground of a row, written in 16-bit parts
    typedef uint16_t __attribute__((may_alias)) mask_part_t;
    const int ty = (int)blockIdx.x / a.tiles_x, tx = (int)blockIdx.x - ty * a.tiles_x;
    const int x0 = tx * kCrT, y0 = ty * kCrT;
    const int lane = (int)threadIdx.x & 63;
    const int row = (int)threadIdx.x >> 2, part = (int)threadIdx.x & 3, gy = y0 + row;
    {
        // sixteen pixels of row `row`: four dwords, read at their alignment
        // where the tile's row is whole, else byte by byte
        uint32_t w[4] = {};
        const int gx = x0 + 16 * part, left = a.W - gx;
        uint32_t in = left >= 16 ? 0xFFFFu : (left > 0 ? (1u << left) - 1u : 0u);
        if (gy >= a.H) in = 0;
        if (in == 0xFFFFu) {
            const uintptr_t p = reinterpret_cast<uintptr_t>(a.in + (int64_t)gy * a.pitch + gx);
            const uint32_t mis = (uint32_t)(p & 3);
            const uint32_t *src = reinterpret_cast<const uint32_t *>(p - mis);
            uint32_t d[5];
#pragma unroll
            for (int j = 0; j < 4; j++) d[j] = src[j];
            d[4] = src[mis ? 4 : 3];
#pragma unroll
            for (int j = 0; j < 4; j++) w[j] = __builtin_amdgcn_alignbyte(d[j + 1], d[j], mis);
        } else {
            for (int b = 0; b < 16; b++)
                if ((in >> b) & 1) w[b >> 2] |= (uint32_t)a.in[(int64_t)gy * a.pitch + gx + b] << (8 * (b & 3));
        }
        uint32_t bits = 0;
#pragma unroll
        for (int b = 0; b < 16; b++) bits |= cr_fg(a, (w[b >> 2] >> (8 * (b & 3))) & 0xFFu) ? 1u << b : 0u;
        reinterpret_cast<mask_part_t *>(mask)[threadIdx.x] = (mask_part_t)(bits & in);
    }
    for (int k = (int)threadIdx.x; k < kCrT * kCrRow / 2; k += 256) cnt[k] = 0;
    __syncthreads();
    const uint64_t m = mask[row], st = cr_starts(m);
    const int n = __popcll(st), li = row * kCrRow, lu = li - kCrRow;
    // this thread's runs are part, part + 4, ... (at most eight): where each
    // points, in the end its root
    const int mine = n > part ? (n - part + 3) / 4 : 0;
    int p[8];
    const uint64_t mr = mask[lane], ur = lane > 0 ? mask[lane - 1] : 0;
    if (__all((cr_starts(mr) & (cr_starts(mr) - 1)) == 0)) {
        // every wave sees the same rows
        const uint64_t breaks = __ballot((ur & (mr | (mr << 1) | (mr >> 1))) == 0);
        p[0] = (63 - __clzll((long long)(breaks & ((2ull << row) - 1ull)))) * kCrRow;
        if (mine) {
            col[li] = (uint8_t)(__ffsll((unsigned long long)m) - 1);
            if (gy < a.covered) atomicAdd(cnt + (p[0] >> 1), (uint32_t)__popcll(m) << (16 * (p[0] & 1)));
        }
    } else {
        const uint64_t u = row > 0 ? mask[row - 1] : 0;
        uint64_t own = st;
        for (int j = 0; j < part; j++) own &= own - 1;
        auto next4 = [](uint64_t v) {
#pragma unroll
            for (int j = 0; j < 4; j++) v &= v - 1;
            return v;
        };
        uint32_t extra = 0;                         // those that touch a second run above
        uint64_t r = own;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (!__any(j < mine)) break;
            if (j < mine) {
                const int k = part + 4 * j;
                const uint64_t t = cr_touched(m, u, r & (~r + 1));
                p[j] = li + k;
                if (t) {
                    p[j] = lu + cr_run_of(u, t);
                    if (cr_starts(u) & t & (t - 1)) extra |= 1u << j;
                }
                loc[li + k] = p[j];
                col[li + k] = (uint8_t)(__ffsll((unsigned long long)r) - 1);
                r = next4(r);
            }
        }
        // Whatever a wave reads of another's entries is an ancestor, so the
        // rounds need no barrier between them (what they leave is walked).
        // Entries are read four at a time.
        auto step = [&](int h, bool store) {
            int q[4];
            bool moved = false;
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (h + j < mine) q[j] = lds_load(loc, p[h + j]);
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (h + j < mine) {
                    moved = moved || q[j] != p[h + j];
                    if (store)
                        __hip_atomic_store(loc + li + part + 4 * (h + j), q[j], __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
                    p[h + j] = q[j];
                }
            return moved;
        };
        auto jump = [&](int rounds) {
            __syncthreads();
            for (int round = 0; round < rounds; round++) {
                step(0, true);
                if (__any(mine > 4)) step(4, true);
            }
        };
        jump(4);
        jump(3);
        __syncthreads();
        r = own;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if (!__any((extra >> j) != 0)) break;
            if ((extra >> j) & 1) {
                const uint64_t t = cr_touched(m, u, r & (~r + 1));
                uint64_t more = cr_starts(u) & t & (t - 1);   // starts past the first touched column
                while (more) {
                    l_unite(loc, p[j], lu + cr_run_of(u, more));
                    more &= more - 1;
                }
            }
            r = next4(r);
        }
        __syncthreads();
        while (__any(step(0, false))) {}
        if (__any(mine > 4))
            while (__any(step(4, false))) {}
        if (gy < a.covered) {
            r = own;
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (j < mine) {
                    const uint64_t s = r & (~r + 1);
                    atomicAdd(cnt + (p[j] >> 1), (uint32_t)__popcll(m & ~(m + s) & ~(s - 1)) << (16 * (p[j] & 1)));
                    r = next4(r);
                }
        }
    }
    __syncthreads();
    // the runs' roots as tile indexes; each root's parent (itself) and area
    uint64_t roots = 0;
    if (gy < a.H) {
        const int64_t at = (int64_t)gy * a.tiles_x + tx;
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (j < mine) {
                const int k = part + 4 * j, c = col[p[j]];
                a.run_root[at * a.runs + k] = (uint16_t)(p[j] / kCrRow * kCrT + c);
                if (p[j] == li + k) {
                    roots |= 1ull << c;
                    const int g = gy * a.W + x0 + c;
                    a.parent[g] = g;
                    a.area[g] = (int)((cnt[p[j] >> 1] >> (16 * (p[j] & 1))) & 0xFFFFu);
                }
            }
        // single pixels outside the gray range that the area filter keeps
        const int one = gy < a.covered ? 1 : 0;
        if (cr_kept_area(a, one)) {
            for (int c = 16 * part; c < 16 * part + 16 && x0 + c < a.W; c++)
                if (!((m >> c) & 1)) {
                    roots |= 1ull << c;
                    const int g = gy * a.W + x0 + c;
                    a.parent[g] = g;
                    a.area[g] = one;
                }
        }
    }
    // the row's four threads hold parts of its root mask
    uint32_t lo = (uint32_t)roots, hi = (uint32_t)(roots >> 32);
    lo |= (uint32_t)__builtin_amdgcn_mov_dpp((int)lo, 0xB1, 0xF, 0xF, true);
    hi |= (uint32_t)__builtin_amdgcn_mov_dpp((int)hi, 0xB1, 0xF, 0xF, true);
    lo |= (uint32_t)__builtin_amdgcn_mov_dpp((int)lo, 0x4E, 0xF, 0xF, true);
    hi |= (uint32_t)__builtin_amdgcn_mov_dpp((int)hi, 0x4E, 0xF, 0xF, true);
    if (gy < a.H && part == 0) {
        const int64_t at = (int64_t)gy * a.tiles_x + tx;
        a.fg[at] = m;
        a.root[at] = ((uint64_t)hi << 32) | lo;
    }
}

// Global index of the tile-local root of the pixel in row y, column c of
// tile column tx, whose row's mask there is m; -1 outside the gray range.
__device__ __forceinline__ int cr_local_root(const CrArgs &a, int y, int tx, uint64_t m, int c)
{
    if (!((m >> c) & 1)) return -1;
    const int l = a.run_root[((int64_t)y * a.tiles_x + tx) * a.runs + cr_run_of(m, 1ull << c)];
    return ((y & ~(kCrT - 1)) + (l >> 6)) * a.W + tx * kCrT + (l & (kCrT - 1));
}

// The same for the pixel at (x, y), which may lie outside the image.
__device__ __forceinline__ int cr_local_root_at(const CrArgs &a, int x, int y)
{
    if (x < 0 || x >= a.W || y < 0 || y >= a.H) return -1;
    const int tx = x / kCrT;
    return cr_local_root(a, y, tx, a.fg[(int64_t)y * a.tiles_x + tx], x & (kCrT - 1));
}

// Unites the pairs (ri, ro) of the lanes that have one, each different pair
// once (the runs of one region that noise has cut meet across an edge many
// times, with the same two roots).
__device__ __forceinline__ void cr_unite_pairs(int *parent, bool has, int ri, int ro, int lane)
{
    uint64_t todo = __ballot(has), chosen = 0;
    while (todo) {
        const int l0 = __ffsll((unsigned long long)todo) - 1;
        const int a0 = __builtin_amdgcn_readlane(ri, l0), b0 = __builtin_amdgcn_readlane(ro, l0);
        todo &= ~__ballot(ri == a0 && ro == b0);
        chosen |= 1ull << l0;
    }
    if ((chosen >> lane) & 1) cr_unite(parent, ri, ro);
}

// Border pass: the pairs of 8-neighbours in different tiles.  One wave per
// tile edge: the top edge (64 pixels of the tile's first row) against the
// row above, the left edge (64 pixels of its first column) against the
// column to the left, each line extended by one pixel past both ends (the
// corner diagonals).  Pixels along an edge are joined where they touch
// inside their own tile, so the run rule of the tile pass applies with the
// edge as the line: one union per pair of touching runs.  A right edge is
// the next tile's left edge (its NE pairs are that edge's SW pairs).
__global__ void __launch_bounds__(256) cr_union_kernel(CrArgs a, int ntiles)
{
    const int lane = (int)threadIdx.x & 63;
    const int64_t e = (int64_t)blockIdx.x * 4 + ((int)threadIdx.x >> 6);   // 2 * tile + (0 top, 1 left)
    if (e >= 2 * (int64_t)ntiles) return;                        // whole waves
    const int tile = (int)(e >> 1), ty = tile / a.tiles_x;
    const int x0 = (tile - ty * a.tiles_x) * kCrT, y0 = ty * kCrT;
    const bool top = (e & 1) == 0;
    if (top ? y0 == 0 : x0 == 0) return;
    // this pixel (x, y) and its neighbour across the edge (xo, yo); the
    // line's step from one lane to the next is (dx, dy)
    const int x = top ? x0 + lane : x0, y = top ? y0 : y0 + lane;
    const int dx = top ? 1 : 0, dy = top ? 0 : 1;
    const int xo = top ? x : x - 1, yo = top ? y - 1 : y;
    const int ri = cr_local_root_at(a, x, y), ro = cr_local_root_at(a, xo, yo);
    // the other line's pixels before and after this one (past the ends: read)
    int rb = __shfl_up(ro, 1), ra = __shfl_down(ro, 1);
    if (lane == 0) rb = cr_local_root_at(a, xo - dx, yo - dy);
    if (lane == 63) ra = cr_local_root_at(a, xo + dx, yo + dy);
    const uint64_t fm = __ballot(ri >= 0);
    const bool f = ri >= 0, o = ro >= 0;
    const bool start = lane == 0 || !((fm >> (lane - 1)) & 1);
    const bool end = lane == 63 || !((fm >> (lane + 1)) & 1);
    const bool first = f && (o ? (start || rb < 0) : (start && rb >= 0));
    cr_unite_pairs(a.parent, first, ri, o ? ro : rb, lane);
    cr_unite_pairs(a.parent, f && !o && end && ra >= 0, ri, ra, lane);
}

// Path compression and areas: a workgroup takes 4 * `per` tiles, four at a
// time with four threads per tile row, which walk the row's local roots,
// point each at its global root and add its area there.  One region can hold
// a root in every tile, and atomics on one counter serialise (about 12 ns
// each), so equal roots are added up first in the wave, then over the
// workgroup in a small LDS table (a root whose slot is taken adds directly).
constexpr int kCrSlots = 64;

__global__ void __launch_bounds__(1024) cr_area_kernel(CrArgs a, int ntiles, int per)
{
    __shared__ int key[kCrSlots], sum_of[kCrSlots];
    const int lane = (int)threadIdx.x & 63;
    if (threadIdx.x < kCrSlots) {
        key[threadIdx.x] = -1;
        sum_of[threadIdx.x] = 0;
    }
    __syncthreads();
    for (int b = 0; b < per; b++) {
        const int tile = ((int)blockIdx.x * per + b) * 4 + ((int)threadIdx.x >> 8);
        const int ty = tile / a.tiles_x, tx = tile - ty * a.tiles_x;
        const int y = ty * kCrT + (((int)threadIdx.x & 255) >> 2), c0 = ((int)threadIdx.x & 3) * 16;
        uint32_t bits = 0;
        if (tile < ntiles && y < a.H) bits = (uint32_t)(a.root[(int64_t)y * a.tiles_x + tx] >> c0) & 0xFFFFu;
        while (__any(bits != 0)) {
            int g = -1, ar = 0;
            if (bits) {
                const int r = y * a.W + tx * kCrT + c0 + __ffs(bits) - 1;
                bits &= bits - 1;
                // Other workgroups store to these entries meanwhile: whatever
                // a read finds of that is an ancestor, so it need not see
                // their stores (reads and stores at device scope cost the
                // call 0.8 us on 1021 x 767), but each has to be one access.
                auto entry = [&](int i) {
                    return __hip_atomic_load(a.parent + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                };
                int up = entry(r);
                do {
                    g = up;
                    up = entry(g);
                } while (up != g);
                if (g != r) {
                    __hip_atomic_store(a.parent + r, g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                    ar = a.area[r];
                } else {
                    g = -1;
                }
            }
            uint64_t rem = __ballot(ar > 0);
            while (rem) {
                const int l0 = __ffsll((unsigned long long)rem) - 1;
                const int g0 = __builtin_amdgcn_readlane(g, l0);
                int sum = g == g0 ? ar : 0;
                const uint64_t eq = __ballot(g == g0);
                if (eq & (eq - 1)) {
#pragma unroll
                    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
                }
                if (lane == l0) {
                    const int slot = (int)(((uint32_t)g0 * 0x9E3779B1u) >> 26);
                    const int old = atomicCAS(key + slot, -1, g0);
                    if (old == -1 || old == g0)
                        atomicAdd(sum_of + slot, sum);
                    else
                        atomicAdd(a.area + g0, sum);
                }
                rem &= ~eq;
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < kCrSlots && key[threadIdx.x] >= 0) atomicAdd(a.area + key[threadIdx.x], sum_of[threadIdx.x]);
}

// One wave per row (of every 4 * gridDim.x): which roots are kept, and how
// many.  The areas are read here for the last time; from here on a.area holds
// the u8 numbers, 0 until cr_number_kernel sets those of the first 256 kept
// roots.
__global__ void __launch_bounds__(256) cr_kept_kernel(CrArgs a)
{
    const int lane = (int)threadIdx.x & 63;
    for (int y = (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6); y < a.H; y += (int)gridDim.x * 4) {   // whole waves
        int count = 0;
        for (int tx = lane; tx < a.tiles_x; tx += 64) {
            uint64_t bits = a.root[(int64_t)y * a.tiles_x + tx], kept = 0;
            while (bits) {
                const uint64_t bit = bits & (~bits + 1);
                const int r = y * a.W + tx * kCrT + __ffsll((unsigned long long)bits) - 1;
                bits ^= bit;
                if (a.parent[r] == r) {
                    if (cr_kept_area(a, a.area[r])) kept |= bit;
                    a.area[r] = 0;
                }
            }
            a.kept[(int64_t)y * a.tiles_x + tx] = kept;
            count += __popcll(kept);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) count += __shfl_xor(count, off);
        if (lane == 0) a.rowcount[y] = count;
    }
}

// Raster-order numbers (one workgroup): kept roots before each row by a scan
// of the row counts, then the rows that hold one of the first 256 (at most
// 256 rows) number theirs.  Number s is the output byte s + 1; the others
// (and 255, whose byte wraps) keep 0.
__global__ void __launch_bounds__(1024) cr_number_kernel(CrArgs a)
{
    __shared__ int part[16], row_of[256], off_of[256], nrows;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = (a.H + 1023) / 1024;
    const int64_t first = (int64_t)tid * per;
    const int y0 = (int)(first < a.H ? first : a.H), y1 = (int)(first + per < a.H ? first + per : a.H);
    int sum = 0;
    for (int y = y0; y < y1; y++) sum += a.rowcount[y];
    int scan = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int t = __shfl_up(scan, off);
        if (lane >= off) scan += t;
    }
    if (lane == 63) part[wave] = scan;
    if (tid == 0) nrows = 0;
    __syncthreads();
    int next = scan - sum;
    for (int w = 0; w < wave; w++) next += part[w];
    for (int y = y0; y < y1 && next < 256; y++) {
        const int c = a.rowcount[y];
        if (c > 0) {
            const int k = atomicAdd(&nrows, 1);
            row_of[k] = y;
            off_of[k] = next;
        }
        next += c;
    }
    __syncthreads();
    const int n = nrows;
    for (int k = wave; k < n; k += 16) {
        const int y = row_of[k];
        int base = off_of[k];
        for (int tx0 = 0; tx0 < a.tiles_x && base < 256; tx0 += 64) {
            const int tx = tx0 + lane;
            uint64_t bits = tx < a.tiles_x ? a.kept[(int64_t)y * a.tiles_x + tx] : 0;
            const int c = __popcll(bits);
            int incl = c;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int t = __shfl_up(incl, off);
                if (lane >= off) incl += t;
            }
            int s = base + incl - c;
            while (bits && s < 256) {
                a.area[y * a.W + tx * kCrT + __ffsll((unsigned long long)bits) - 1] = (s + 1) & 255;
                bits &= bits - 1;
                s++;
            }
            base += __builtin_amdgcn_readlane(incl, 63);
        }
    }
}

// Output: the number of each of a tile's runs is looked up once into an LDS
// table; a thread then writes four adjacent pixels, each the number of the
// run its row's mask puts it in.
__global__ void __launch_bounds__(256) cr_output_kernel(CrArgs a)
{
    __shared__ uint8_t number[kCrT * kCrRuns];
    const int ty = (int)blockIdx.x / a.tiles_x, tx = (int)blockIdx.x - ty * a.tiles_x;
    const int x0 = tx * kCrT, y0 = ty * kCrT;
    // this thread's rows of the second part: 16 threads a row, 4 rows
    const int q = (int)threadIdx.x & 15;
    uint64_t m[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int y = y0 + 16 * j + ((int)threadIdx.x >> 4);
        m[j] = y < a.H ? a.fg[(int64_t)y * a.tiles_x + tx] : 0;
    }
    {
        const int row = (int)threadIdx.x >> 2, part = (int)threadIdx.x & 3, y = y0 + row;
        if (y < a.H) {
            const int64_t at = (int64_t)y * a.tiles_x + tx;
            const int n = __popcll(cr_starts(a.fg[at]));
            for (int k = part; k < n; k += 4) {
                const int l = a.run_root[at * a.runs + k];
                number[row * kCrRuns + k] =
                    (uint8_t)a.area[a.parent[(y0 + (l >> 6)) * a.W + x0 + (l & (kCrT - 1))]];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int row = 16 * j + ((int)threadIdx.x >> 4), y = y0 + row, x = x0 + 4 * q;
        if (y >= a.H || x >= a.W) continue;
        const uint64_t st = cr_starts(m[j]);
        const uint32_t mine = (uint32_t)(m[j] >> (4 * q)) & 15u, starts = (uint32_t)(st >> (4 * q)) & 15u;
        int k = __popcll(st & ((1ull << (4 * q)) - 1ull)) - 1;
        uint32_t v = 0;
        if (mine == 15u && !(starts & 14u)) {       // one run, starting here or before
            v = number[row * kCrRuns + k + (int)(starts & 1u)] * 0x01010101u;
        } else {
            const bool singles = cr_kept_area(a, y < a.covered ? 1 : 0);
#pragma unroll
            for (int b = 0; b < 4; b++) {
                k += (int)((starts >> b) & 1u);
                uint32_t s = 0;
                if ((mine >> b) & 1u)
                    s = number[row * kCrRuns + k];
                else if (singles && x + b < a.W)
                    s = (uint32_t)a.area[y * a.W + x + b] & 0xFFu;
                v |= s << (8 * b);
            }
        }
        uint8_t *o = a.out + (int64_t)y * a.out_pitch + x;
        if (x + 4 <= a.W) {
            __builtin_memcpy(o, &v, 4);
        } else {
            for (int b = 0; x + b < a.W; b++) o[b] = (uint8_t)(v >> (8 * b));
        }
    }
}

}  // namespace region
}  // namespace bfimpl

using namespace bfimpl;
using namespace bfimpl::region;

namespace {

bool view_ok(const bf_image_view *v)
{
    return v && v->data && v->width > 0 && v->height > 0 && v->pitch >= v->width;
}

}  // namespace

extern "C" {

int bf_local_cluster(const bf_image_view *in, int64_t alloc_lo, int64_t alloc_hi,
                     const bf_image_view *out, const bf_local_cluster_params *p, void *stream)
{
    if (!in || !out || !p || !in->data || !out->data) {
        set_error("null argument");
        return kNullPointer;
    }
    if (!view_ok(in) || !view_ok(out)) {
        set_error("empty or malformed view");
        return kInvalidData;
    }
    if (alloc_lo == 0 && alloc_hi == 0) {          // the ROI itself
        alloc_hi = (int64_t)(in->height - 1) * in->pitch + in->width;
    }
    if (alloc_lo > 0 || alloc_hi < (int64_t)(in->height - 1) * in->pitch + in->width) {
        set_error("declared allocation does not contain the ROI");
        return kInvalidData;
    }
    LcArgs a{};
    a.in = in->data;
    a.pitch = in->pitch;
    a.lo = alloc_lo;
    a.hi = alloc_hi;
    a.out = out->data;
    a.out_pitch = out->pitch;
    a.W = std::min(in->width, out->width);
    a.H = std::min(in->height, out->height);
    a.pnt_range = p->pnt_range;
    a.pnt_count = p->pnt_count;
    a.gap = (float)p->gap_thred;
    a.diffe = (float)p->diffe_thred;
    a.pro_black = p->pro_black;
    a.pro_white = p->pro_white;
    // The walks reach 2 (pntRange - 1) pixels from the centre, and 2 at least.
    // A halo whose 16-row tile exceeds the LDS bound reads global memory;
    // the others take the tallest tile (fewer halo rows per pixel) that
    // still gives every CU several workgroups.
    const int64_t halo = std::max<int64_t>(2, 2 * ((int64_t)a.pnt_range - 1));
    if ((kLcTw + 2 * halo) * (16 + 2 * halo) > kLcMaxLds) {
        hipLaunchKernelGGL(local_cluster_kernel, dim3((a.W + 63) / 64, (a.H + 3) / 4), dim3(256), 0,
                           (hipStream_t)stream, a);
    } else {
        // staged row: 64 columns and two halos, as one of three compiled
        // pitches (halo <= 16, 32 and 96 pixels)
        const int sp = halo <= 16 ? 96 : (halo <= 32 ? 128 : 256);
        int cus = 0;
        BF_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, current_device()));
        const int64_t tx = (a.W + kLcTw - 1) / kLcTw;
        auto lds_of = [&](int rows) {
            return (size_t)sp * (rows + 2 * halo) + sizeof(uint16_t) * kLcTw * rows + sizeof(int);
        };
        int th = kLcThMax;
        while (th > 16 && (tx * ((a.H + th - 1) / th) < 4 * (int64_t)cus || lds_of(th) > 64 * 1024)) th /= 2;
        const dim3 grid((unsigned)tx, (a.H + th - 1) / th);
        const auto kern = sp == 96 ? local_cluster_lds_kernel<96>
                                   : (sp == 128 ? local_cluster_lds_kernel<128> : local_cluster_lds_kernel<256>);
        hipLaunchKernelGGL(kern, grid, dim3(64 * kLcWaves), lds_of(th), (hipStream_t)stream, a, (int)halo, th);
    }
    BF_HIP(hipGetLastError());
    return kOk;
}

int bf_connect_region(const bf_image_view *in, const bf_image_view *out, int32_t min_area,
                      int32_t max_area, int32_t min_gray, int32_t max_gray, void *stream)
{
    if (!in || !out || !in->data || !out->data) {
        set_error("null argument");
        return kNullPointer;
    }
    if (!view_ok(in) || !view_ok(out)) {
        set_error("empty or malformed view");
        return kInvalidData;
    }
    const int W = std::min(in->width, out->width), H = std::min(in->height, out->height);
    if ((int64_t)W * H > 0x7FFFFFFF) {
        set_error("image too large for 32-bit labels");
        return kInvalidData;
    }
    // A launch holds fewer than 2^32 threads in a dimension; the passes that
    // follow a refused one would work on scratch it has not set.
    if (H >= kCrMaxRows) {
        set_error("image taller than 2^26 - 1 rows");
        return kInvalidData;
    }
    hipStream_t s = (hipStream_t)stream;
    int cus = 0;
    BF_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, current_device()));
    const size_t n = (size_t)W * H;
    const int tiles_x = (W + kCrT - 1) / kCrT, tiles_y = (H + kCrT - 1) / kCrT;
    const int ntiles = tiles_x * tiles_y;
    const int runs = (std::min(W, kCrT) + 1) / 2;
    // foreground, root and kept masks; parents and numbers; row counts; run roots
    const size_t masks = (size_t)H * tiles_x;
    const size_t bytes = 3 * masks * sizeof(uint64_t) + (2 * n + H) * sizeof(int) +
                         masks * runs * sizeof(uint16_t);
    void *work = nullptr;
    BF_HIP(hipMallocAsync(&work, bytes, s));
    CrArgs a{};
    a.in = in->data;
    a.pitch = in->pitch;
    a.out = out->data;
    a.out_pitch = out->pitch;
    a.W = W;
    a.H = H;
    a.tiles_x = tiles_x;
    a.runs = runs;
    a.min_gray = min_gray;
    a.max_gray = max_gray;
    a.min_area = min_area;
    a.max_area = max_area;
    a.covered = std::min(H, 256 * ((((H + 4) / 32) + 7) / 8));
    a.fg = static_cast<uint64_t *>(work);
    a.root = a.fg + masks;
    a.kept = a.root + masks;
    a.parent = reinterpret_cast<int *>(a.kept + masks);
    a.area = a.parent + n;
    a.rowcount = a.area + n;
    a.run_root = reinterpret_cast<uint16_t *>(a.rowcount + H);
    hipLaunchKernelGGL(cr_local_kernel, dim3(ntiles), dim3(256), 0, s, a);
    hipLaunchKernelGGL(cr_union_kernel, dim3((unsigned)((2 * (int64_t)ntiles + 3) / 4)), dim3(256), 0, s, a, ntiles);
    // Eight tiles a workgroup where that still gives every CU two, four below.
    // Fewer workgroups add fewer sums to a region that spans the image; the
    // whole call on square images, noise 2, four / eight tiles, in us: 65.6 /
    // 70.1 at 2048, 92.5 / 92.4 at 3000, 122.0 / 121.6 at 3600, 122.5 / 119.2
    // at 4096, 217 / 204 at 6000, 300 / 276 at 8192 (sixteen: 280).
    const int per = ntiles >= 2 * 8 * cus ? 2 : 1;
    hipLaunchKernelGGL(cr_area_kernel, dim3((ntiles + 4 * per - 1) / (4 * per)), dim3(1024), 0, s, a, ntiles, per);
    hipLaunchKernelGGL(cr_kept_kernel, dim3((unsigned)std::min((H + 3) / 4, 1 << 22)), dim3(256), 0, s, a);
    hipLaunchKernelGGL(cr_number_kernel, dim3(1), dim3(1024), 0, s, a);
    hipLaunchKernelGGL(cr_output_kernel, dim3(ntiles), dim3(256), 0, s, a);
    hipError_t e = hipGetLastError();
    hipError_t f = hipFreeAsync(work, s);
    if (e != hipSuccess) return hip_fail(e, "bf_connect_region");
    if (f != hipSuccess) return hip_fail(f, "bf_connect_region");
    return kOk;
}

}  // extern "C"
