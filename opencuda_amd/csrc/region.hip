// region.hip -- the stages around the bilateral filter in
// okano_3_0/SimpleRegionDetect.cu:287-312: LocalCluster before it and
// ConnectRegion after it, for gfx950.
//
// LocalCluster (okano_3_0/LocalCluster.cu:45-153): one lane per pixel runs
// the eight directional walks the reference spreads over eight threads and
// a shared array, with the same FP32 operations in the same order
// (-ffp-contract=off, IEEE division), so the u8 result is the reference's.
// The reference addresses every read as data + y * pitch + x from the ROI
// origin and its walks reach 2 (pntRange - 1) pixels from the centre while
// the guard band is pntRange + 2 wide; reads here use the same linear
// address, clamped into the allocation the caller declares.  A workgroup
// stages its 64 x 16 tile plus the walks' reach in LDS by that rule.
//
// ConnectRegion (okano_3_0/ConnectRegion.cu:789-1043): 8-connected
// components of pixels whose gray values lie in [minGray, maxGray], each
// labelled by its minimum raster index.  The reference gets there with
// shared-memory labelling per block and rounds of border merging; here each
// 64 x 64 tile is labelled in LDS, then the runs that touch across tile
// edges are joined by a lock-free union-find pass in global memory
// (atomicMin on roots, parents always smaller than children, so every loop
// ends), then path compression -- the result does not depend on the order
// the unions run in.  Areas, the area filter, the raster-order
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

// Root of x: parents are never larger than their children, so the walk ends.
__device__ __forceinline__ int cr_find(const int *L, int x)
{
    int p = cr_load(L, x);
    while (p != x) {
        x = p;
        p = cr_load(L, x);
    }
    return x;
}

// Root of x with path halving: each visited node is re-pointed to its
// grandparent, an ancestor it keeps (trees only ever merge), so parents stay
// smaller than children.  A hook another lane makes meanwhile on a node
// this walk re-points could be overwritten, but such a node was no longer a
// root, so that lane's union loop does not stop there and merges the trees
// through the node's former parent.
__device__ __forceinline__ int cr_find_halving(int *L, int x)
{
    while (true) {
        const int p = cr_load(L, x);
        if (p == x) return x;
        const int gp = cr_load(L, p);
        if (gp == p) return p;
        __hip_atomic_store(L + x, gp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        x = gp;
    }
}

// Lock-free union (the larger root is hooked under the smaller one with
// atomicMin; a failed hook means that root was hooked meanwhile, and the
// loop continues from its new parent, a strictly smaller index).
__device__ void cr_unite(int *L, int a, int b)
{
    while (true) {
        a = cr_find_halving(L, a);
        b = cr_find_halving(L, b);
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
    int min_gray, max_gray;
    int min_area, max_area;
    int covered;              // rows the area count covers
    int *label, *area, *seq, *rowcount, *rowoff;
};

__device__ __forceinline__ bool cr_fg(const CrArgs &a, uint32_t v)
{
    return (int)v >= a.min_gray && (int)v <= a.max_gray;
}

// Areas start at zero (every label is written by the tile pass).
__global__ void cr_init_kernel(CrArgs a)
{
    const int64_t n = (int64_t)a.W * a.H;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        a.area[i] = 0;
}

// Tile pass: each 64 x 64 tile labels its own pixels in LDS with the same
// lock-free union (LDS atomics), then writes every pixel's label as the
// global index of its tile-local root.  Row-major order inside a tile is
// the global order restricted to it, so a local root is the component's
// smallest global index within the tile, never larger than its children.
// (64 x 64 measured fastest on MI355X, 4096^2 chain image: 64 x 16 2.88 ms,
// 64 x 32 2.69, 64 x 64 2.48, 64 x 128 2.98, 128 x 64 3.47 -- taller tiles
// halve the border unions and the depth of the global trees, while wider
// ones lengthen the LDS union chains.)
constexpr int kCrTw = 64, kCrTh = 64;

__device__ __forceinline__ int lds_load(const int *L, int i)
{
    return __hip_atomic_load(L + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ int l_find(const int *L, int x)
{
    int p = lds_load(L, x);
    while (p != x) {
        x = p;
        p = lds_load(L, x);
    }
    return x;
}

__device__ void l_unite(int *L, int a, int b)
{
    while (true) {
        a = l_find(L, a);
        b = l_find(L, b);
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

constexpr int kCrLocalThreads = 256;    // 512 and 1024 measured no faster

// A tile row is one wave (kCrTw = 64): its foreground runs are linked to
// their first pixel with a ballot (no atomics), and a run is united with
// the row above once per run it touches there: through N at the first of
// its pixels under each above segment, through NW / NE at its ends when N
// is background there (a diagonal neighbour next to a foreground N pixel is
// in that pixel's run already).
static_assert(kCrTw == 64, "one wave per tile row");

__global__ void __launch_bounds__(kCrLocalThreads) cr_local_kernel(CrArgs a)
{
    constexpr int kWaves = kCrLocalThreads / 64;
    __shared__ int loc[kCrTw * kCrTh];
    __shared__ uint64_t fgrow[kCrTh];            // foreground bits of each tile row
    const int x0 = blockIdx.x * kCrTw, y0 = blockIdx.y * kCrTh;
    const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    const int gx = x0 + lane;
    const uint64_t upto = lane == 63 ? ~0ull : (2ull << lane) - 1ull;   // lanes 0..lane
    for (int ly = wave; ly < kCrTh; ly += kWaves) {
        const int gy = y0 + ly;
        const bool f = gx < a.W && gy < a.H && cr_fg(a, a.in[(int64_t)gy * a.pitch + gx]);
        const uint64_t m = __ballot(f);
        const uint64_t starts = m & ~(m << 1);   // foreground with background on the left
        const int s = f ? 63 - __clzll((long long)(starts & upto)) : lane;
        loc[ly * kCrTw + lane] = ly * kCrTw + s;
        if (lane == 0) fgrow[ly] = m;
    }
    __syncthreads();
    for (int ly = 1 + wave; ly < kCrTh; ly += kWaves) {
        const uint64_t m = fgrow[ly], u = fgrow[ly - 1];
        if (!((m >> lane) & 1)) continue;
        const int i = ly * kCrTw + lane;
        const bool start = lane == 0 || !((m >> (lane - 1)) & 1);
        const bool end = lane == 63 || !((m >> (lane + 1)) & 1);
        const bool n = (u >> lane) & 1;
        const bool nw = lane > 0 && ((u >> (lane - 1)) & 1);
        const bool ne = lane < 63 && ((u >> (lane + 1)) & 1);
        if (n && (start || !nw)) l_unite(loc, i, i - kCrTw);
        if (!n && start && nw) l_unite(loc, i, i - kCrTw - 1);
        if (!n && end && ne) l_unite(loc, i, i - kCrTw + 1);
    }
    __syncthreads();
    for (int ly = wave; ly < kCrTh; ly += kWaves) {
        const int gy = y0 + ly;
        if (gx >= a.W || gy >= a.H) continue;
        const int root = l_find(loc, ly * kCrTw + lane);
        a.label[gy * a.W + gx] = (y0 + root / kCrTw) * a.W + x0 + (root & (kCrTw - 1));
    }
}

// Border pass: the pairs of 8-neighbours in different tiles.  One wave per
// tile edge: the top edge (64 pixels of the tile's first row) against the
// row above, the left edge (64 pixels of its first column) against the
// column to the left, each line extended by one pixel past both ends (the
// corner diagonals).  Pixels along an edge are joined where they touch
// inside their own tile, so the run rule of the tile pass applies with the
// edge as the line: one union per pair of touching runs.  A right edge is
// the next tile's left edge (its NE pairs are that edge's SW pairs).
__global__ void __launch_bounds__(256) cr_union_kernel(CrArgs a, int tiles_x, int ntiles)
{
    const int lane = (int)threadIdx.x & 63;
    const int e = (int)blockIdx.x * 4 + ((int)threadIdx.x >> 6);   // 2 * tile + (0 top, 1 left)
    const int tile = e >> 1;
    if (tile >= ntiles) return;                                  // whole waves
    const int x0 = tile % tiles_x * kCrTw, y0 = tile / tiles_x * kCrTh;
    const bool top = (e & 1) == 0;
    if (top ? y0 == 0 : x0 == 0) return;
    // this pixel (x, y) and its neighbour across the edge (xo, yo); the
    // line's step from one lane to the next is (dx, dy)
    const int x = top ? x0 + lane : x0, y = top ? y0 : y0 + lane;
    const int dx = top ? 1 : 0, dy = top ? 0 : 1;
    const int xo = top ? x : x - 1, yo = top ? y - 1 : y;
    auto fg_at = [&](int px, int py) {
        return px >= 0 && px < a.W && py >= 0 && py < a.H &&
               cr_fg(a, a.in[(int64_t)py * a.pitch + px]);
    };
    const bool f = fg_at(x, y), o = fg_at(xo, yo);
    const uint64_t fm = __ballot(f), om = __ballot(o);
    // the other line's pixels before and after this one (past the ends: read)
    const bool ob = lane > 0 ? ((om >> (lane - 1)) & 1) : fg_at(xo - dx, yo - dy);
    const bool oa = lane < 63 ? ((om >> (lane + 1)) & 1) : fg_at(xo + dx, yo + dy);
    if (!f) return;
    const bool start = lane == 0 || !((fm >> (lane - 1)) & 1);
    const bool end = lane == 63 || !((fm >> (lane + 1)) & 1);
    const int idx = y * a.W + x, io = yo * a.W + xo, step = dy * a.W + dx;
    if (o && (start || !ob)) cr_unite(a.label, idx, io);
    if (!o && start && ob) cr_unite(a.label, idx, io - step);
    if (!o && end && oa) cr_unite(a.label, idx, io + step);
}

// Path compression and areas in one pass: one wave per row walks it in
// 64-pixel chunks, replaces every label by its root (the unions are all
// done, so a root is the same whichever lane finds it; a walk through a
// label another wave has already replaced reaches the same root), and for
// the rows below a.covered adds the areas per root.  Inside a chunk the
// lane that starts a run of equal roots adds the run; the run that reaches
// the chunk's end is carried, with a wave-uniform label and count, into the
// next chunk.  A row's first
// long run (>= 32 pixels) names its "hot" label, whose later runs are
// summed in the wave and added once at the row's end: in a large region
// broken by many small ones (here 1.26M runs on a 4096^2 image, half of them
// one region's) every run would otherwise be an atomic on the same
// counter, and those serialise.
__global__ void __launch_bounds__(256) cr_area_kernel(CrArgs a)
{
    const int lane = threadIdx.x & 63;
    const int y = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (y >= a.H) return;                           // whole waves
    int *row = a.label + (int64_t)y * a.W;
    const bool counted = y < a.covered;             // wave-uniform
    int cur = -1, cnt = 0;                          // carried run
    int hot = -1, hot_cnt = 0;                      // the row's hot label and its sum
    // a finished run of `lab` (wave-uniform): to the hot sum or one atomic
    auto flush = [&](int lab, int c) {
        if (lab < 0 || c <= 0) return;
        if (lab == hot) {
            hot_cnt += c;
        } else if (hot < 0 && c >= 32) {
            hot = lab;
            hot_cnt = c;
        } else if (lane == 0) {
            atomicAdd(a.area + lab, c);
        }
    };
    for (int x0 = 0; x0 < a.W; x0 += 64) {
        const int n = min(64, a.W - x0);            // pixels in this chunk
        // path compression: the root, written back for the later passes
        const int l = lane < n ? cr_find(a.label, y * a.W + x0 + lane) : -1;
        if (lane < n)
            __hip_atomic_store(row + x0 + lane, l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!counted) continue;
        int prev = __shfl_up(l, 1);
        if (lane == 0) prev = cur;
        const bool start = lane < n && l != prev;
        const uint64_t starts = __ballot(start);
        // runs that start and end inside the chunk: the hot label's are
        // summed across the wave, the others added by their start lane
        int len = 0;
        if (start) {
            const uint64_t later = lane == 63 ? 0ull : (starts >> (lane + 1)) << (lane + 1);
            if (later) len = __ffsll((unsigned long long)later) - 1 - lane;
        }
        const bool to_hot = len > 0 && l == hot;
        if (len > 0 && !to_hot) atomicAdd(a.area + l, len);
        if (__ballot(to_hot)) {
            int sum = to_hot ? len : 0;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
            hot_cnt += sum;
        }
        const int first = starts ? __ffsll((unsigned long long)starts) - 1 : n;
        cnt += first;                               // the carried run goes on to `first`
        if (starts) {
            flush(cur, cnt);
            const int last = 63 - __clzll((long long)starts);
            cur = __shfl(l, last);
            cnt = n - last;
        }
    }
    if (!counted) return;
    flush(cur, cnt);
    if (lane == 0 && hot >= 0) atomicAdd(a.area + hot, hot_cnt);
}

__device__ __forceinline__ bool cr_kept_root(const CrArgs &a, int i)
{
    if (a.label[i] != i) return false;
    const int ar = a.area[i];
    return !(ar != 0 && (ar < a.min_area || ar > a.max_area));
}

// One wave per row: kept roots in the row.
__global__ void __launch_bounds__(64) cr_rowcount_kernel(CrArgs a)
{
    const int y = blockIdx.x;
    int count = 0;
    for (int x0 = 0; x0 < a.W; x0 += 64) {
        const int x = x0 + (int)threadIdx.x;
        const bool k = x < a.W && cr_kept_root(a, y * a.W + x);
        count += __popcll(__ballot(k));
    }
    if (threadIdx.x == 0) a.rowcount[y] = count;
}

// Exclusive scan of the row counts (one workgroup).
__global__ void __launch_bounds__(1024) cr_scan_kernel(CrArgs a)
{
    __shared__ int part[1024];
    __shared__ int carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (int base = 0; base < a.H; base += 1024) {
        const int i = base + (int)threadIdx.x;
        const int v = i < a.H ? a.rowcount[i] : 0;
        part[threadIdx.x] = v;
        __syncthreads();
        for (int off = 1; off < 1024; off <<= 1) {
            const int t = threadIdx.x >= (unsigned)off ? part[threadIdx.x - off] : 0;
            __syncthreads();
            part[threadIdx.x] += t;
            __syncthreads();
        }
        if (i < a.H) a.rowoff[i] = carry + part[threadIdx.x] - v;
        __syncthreads();
        if (threadIdx.x == 1023) carry += part[1023];
        __syncthreads();
    }
}

// One wave per row: raster-order numbers of the kept roots (-1 for the
// other roots and for numbers >= 256).
__global__ void __launch_bounds__(64) cr_number_kernel(CrArgs a)
{
    const int y = blockIdx.x;
    const uint64_t below = (1ull << threadIdx.x) - 1ull;
    int next = a.rowoff[y];
    for (int x0 = 0; x0 < a.W; x0 += 64) {
        const int x = x0 + (int)threadIdx.x;
        const int i = y * a.W + x;
        const bool in = x < a.W;
        const bool root = in && a.label[i] == i;
        const bool k = in && cr_kept_root(a, i);
        const uint64_t m = __ballot(k);
        if (root) {
            const int s = next + __popcll(m & below);
            a.seq[i] = (k && s < 256) ? s : -1;
        }
        next += __popcll(m);
    }
}

__global__ void __launch_bounds__(256) cr_output_kernel(CrArgs a)
{
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= a.W || y >= a.H) return;
    const int s = a.seq[a.label[y * a.W + x]];
    a.out[(int64_t)y * a.out_pitch + x] = (uint8_t)(s + 1);
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
    hipStream_t s = (hipStream_t)stream;
    const size_t n = (size_t)W * H;
    const size_t bytes = (3 * n + 2 * (size_t)H) * sizeof(int);
    int *work = nullptr;
    BF_HIP(hipMallocAsync(reinterpret_cast<void **>(&work), bytes, s));
    CrArgs a{};
    a.in = in->data;
    a.pitch = in->pitch;
    a.out = out->data;
    a.out_pitch = out->pitch;
    a.W = W;
    a.H = H;
    a.min_gray = min_gray;
    a.max_gray = max_gray;
    a.min_area = min_area;
    a.max_area = max_area;
    a.covered = std::min(H, 256 * ((((H + 4) / 32) + 7) / 8));
    a.label = work;
    a.area = work + n;
    a.seq = work + 2 * n;
    a.rowcount = work + 3 * n;
    a.rowoff = work + 3 * n + H;
    const int flat = (int)std::min<size_t>((n + 255) / 256, 65536);
    const dim3 g2((W + 63) / 64, (H + 3) / 4);
    hipLaunchKernelGGL(cr_init_kernel, dim3(flat), dim3(256), 0, s, a);
    hipLaunchKernelGGL(cr_local_kernel, dim3((W + kCrTw - 1) / kCrTw, (H + kCrTh - 1) / kCrTh),
                       dim3(kCrLocalThreads), 0, s, a);
    {
        const int tiles_x = (W + kCrTw - 1) / kCrTw, tiles_y = (H + kCrTh - 1) / kCrTh;
        const int edges = 2 * tiles_x * tiles_y;
        hipLaunchKernelGGL(cr_union_kernel, dim3((edges + 3) / 4), dim3(256), 0, s, a, tiles_x,
                           tiles_x * tiles_y);
    }
    hipLaunchKernelGGL(cr_area_kernel, dim3((H + 3) / 4), dim3(256), 0, s, a);
    hipLaunchKernelGGL(cr_rowcount_kernel, dim3(H), dim3(64), 0, s, a);
    hipLaunchKernelGGL(cr_scan_kernel, dim3(1), dim3(1024), 0, s, a);
    hipLaunchKernelGGL(cr_number_kernel, dim3(H), dim3(64), 0, s, a);
    hipLaunchKernelGGL(cr_output_kernel, g2, dim3(256), 0, s, a);
    hipError_t e = hipGetLastError();
    hipError_t f = hipFreeAsync(work, s);
    if (e != hipSuccess) return hip_fail(e, "bf_connect_region");
    if (f != hipSuccess) return hip_fail(f, "bf_connect_region");
    return kOk;
}

}  // extern "C"
