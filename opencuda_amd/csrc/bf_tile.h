// bf_tile.h -- device building blocks shared by the exact-filter kernels
// (bf_exact.hip: single image, tile lists, sample check; bf_ring_batch.hip:
// batches of canonical-template jobs).  Not a public header.
//
// LDS is addressed by byte offset through address-space-3 pointers.  The
// kernels that use these helpers declare no static LDS, so the dynamic
// allocation starts at LDS address 0 and a v_sad_u8 result is usable as a
// ds_read address unchanged.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>

#include "bf_internal.h"

namespace bfimpl {

constexpr int kModeRef = BF_MODE_REF;

struct KArgs {
    DevJob job0;                 // used when njobs == 1
    const DevJob *jobs;          // device job table (njobs > 1)
    int32_t njobs;
    int32_t ntiles;              // static tile count (no tile_list)
    const int32_t *tile_list;    // optional: global tile ids to run
    const int32_t *tile_count;   // device count of tile_list entries
    int32_t *counter;            // optional work-queue counter
    int32_t pad;
};

// Dynamic LDS layout (no static __shared__ objects, so it starts at LDS
// address 0 and every gather address is a plain byte offset):
//   [0, 16)                  work-queue slot
//   [16, 16 + TILE_BYTES)    staged input tile (byte-replicated u32)
//   [16 + TILE_BYTES, ...)   fused weight table, (nrows + 1) x 256 floats
constexpr uint32_t kTileOff = 16;

// LDS is addressed by byte offset through address-space-3 pointers.  The
// kernel declares no static LDS, so the dynamic allocation starts at LDS
// address 0 (checked by the .group_segment_fixed_size of 0 in the code
// object) and a v_sad_u8 result is usable as a ds_read address unchanged.
typedef __attribute__((address_space(3))) uint32_t lds_word;
typedef __attribute__((address_space(3))) float lds_float;

__device__ __forceinline__ uint32_t lds_u32(uint32_t byte_addr)
{
    return *(const lds_word *)(size_t)byte_addr;
}

__device__ __forceinline__ float lds_f32(uint32_t byte_addr)
{
    return *(const lds_float *)(size_t)byte_addr;
}

__device__ __forceinline__ void lds_store_u32(uint32_t byte_addr, uint32_t v)
{
    *(lds_word *)(size_t)byte_addr = v;
}

// Read-only tables (jobs, taps) are read through the constant address
// space: they never change during a launch, and this lets the compiler use
// scalar loads for the wave-uniform tap stream.
#define BF_CONST __attribute__((address_space(4)))
template <class T>
__device__ __forceinline__ const BF_CONST T *as_const(const T *p)
{
    return (const BF_CONST T *)(p);
}

// Images and tables are in global memory.  Pointers that a kernel reads from
// a job table are generic ones to the compiler; through them it would use
// flat accesses, which count as LDS accesses too, and with one of those in
// flight every wait for an LDS read has to wait for all of them.
#define BF_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ BF_GLOBAL T *as_global(T *p)
{
    return (BF_GLOBAL T *)(p);
}

__device__ __forceinline__ uint8_t to_u8(float q)
{
    if (!(q > 0.0f)) return 0;          // NaN (0/0) and non-positive
    if (q >= 255.0f) return 255;
    return (uint8_t)(int)q;             // truncation toward zero
}

__device__ __forceinline__ int clampi(int v, int lo, int hi)
{
    return v < lo ? lo : (v > hi ? hi : v);
}

// Find the job owning global tile `tile` (jobs sorted by tile_begin).
__device__ __forceinline__ int find_job(const BF_CONST DevJob *jobs, int njobs, int tile)
{
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].tile_begin <= tile) lo = mid; else hi = mid - 1;
    }
    return lo;
}

template <int TW, int TGY, int HALO>
struct Geo {
    static constexpr int TH = 4 * TGY;
    static constexpr int TCOLS = TW + 2 * HALO;
    static constexpr int TROWS = TH + 2 * HALO;
    static constexpr int TILE_BYTES = TCOLS * TROWS * 4;
    static constexpr int NT = TW * TGY;
};

typedef __attribute__((address_space(3))) uint8_t lds_byte;

__device__ __forceinline__ uint32_t lds_u8(uint32_t byte_addr)
{
    return *(const lds_byte *)(size_t)byte_addr;
}

// Stage the clamped input rectangle (rows ys .. ys+ROWS-1, columns xs ..
// xs+COLS-1, clamped to the input view) into LDS at `base`, row-major with
// COLS elements per row: byte-replicated u32 elements (the exact kernels'
// v_sad_u8 form) or, with BYTES, plain bytes.  NT threads (ids 0..NT-1)
// share the work.
template <int COLS, int ROWS, int NT, bool BYTES>
__device__ __forceinline__ void stage_rect(const DevJob &job, int xs, int ys, uint32_t base,
                                           int tid)
{
    constexpr uint32_t ESZ = BYTES ? 1u : 4u;
    const int wmax = job.in_w - 1, hmax = job.in_h - 1;
    auto put = [&](int e, uint32_t byte) {
        if (BYTES)
            *(lds_byte *)(size_t)(base + (uint32_t)e) = (uint8_t)byte;
        else
            lds_store_u32(base + (uint32_t)e * ESZ, byte * 0x01010101u);
    };
    if (xs >= 0 && xs + COLS <= job.in_w) {
        // Interior columns: aligned 16-byte loads covering [xs, xs+COLS).
        // Bytes outside that span are dropped; they lie in the same aligned
        // 16-byte block as a byte of the row, hence in mapped memory.
        constexpr int NCH = (COLS + 15) / 16 + 1;  // chunks per row
        for (int e = tid; e < ROWS * NCH; e += NT) {
            const int r = e / NCH, ch = e - r * NCH;
            const int gy = clampi(ys + r, 0, hmax);
            const uint8_t *row = job.in + (int64_t)gy * job.in_pitch;
            const uintptr_t a0 = reinterpret_cast<uintptr_t>(row + xs) & ~(uintptr_t)15;
            const uintptr_t ca = a0 + 16 * (uintptr_t)ch;
            const intptr_t first = (intptr_t)ca - (intptr_t)reinterpret_cast<uintptr_t>(row + xs);
            if (first >= COLS) continue;
            typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
            const u32x4_t w = *as_global(reinterpret_cast<const u32x4_t *>(ca));
#pragma unroll
            for (int b = 0; b < 16; b++) {
                const int c = (int)first + b;
                if (c >= 0 && c < COLS) put(r * COLS + c, (w[b >> 2] >> (8 * (b & 3))) & 0xFFu);
            }
        }
    } else {
        for (int e = tid; e < ROWS * COLS; e += NT) {
            const int r = e / COLS, c = e - r * COLS;
            const int gy = clampi(ys + r, 0, hmax);
            const int gx = clampi(xs + c, 0, wmax);
            put(e, as_global(job.in)[(int64_t)gy * job.in_pitch + gx]);
        }
    }
}

// Stage the clamped input tile (rows Y0-HALO .., cols X0-HALO ..) into LDS
// as byte-replicated u32.
template <int TW, int TGY, int HALO>
__device__ __forceinline__ void load_tile(const DevJob &job, int X0, int Y0, int tid)
{
    using G = Geo<TW, TGY, HALO>;
    stage_rect<G::TCOLS, G::TROWS, G::NT, false>(job, X0 - HALO, Y0 - HALO, kTileOff, tid);
}

// Fused weight table: W[row][d] = rowg[row] * range[d]; row `nrows` = 0, or
// range[d] itself where the job's further rows are not fused (erow).
// Separate-table mode: just E[d].
template <int NT>
__device__ __forceinline__ void build_lut(const DevJob &job, uint32_t lut_base, int tid)
{
    if (job.sep) {
        for (int d = tid; d < 256; d += NT)
            lds_store_u32(lut_base + (uint32_t)d * 4, __float_as_uint(as_global(job.range)[d]));
        return;
    }
    if constexpr (NT % 256 == 0) {
        // Each thread keeps one column d (its range value loaded once); the
        // row a wave writes is the same for all its lanes, so its spatial
        // weight is a scalar load.  (A loop over flat indices waited for
        // two vector loads per entry, ~30 round trips before the first
        // tile of a launch or of a job with other tables.)
        const int d = tid & 255;
        const float rd = as_global(job.range)[d];
        const int r0 = __builtin_amdgcn_readfirstlane(tid >> 8);
        for (int row = r0; row <= job.nrows; row += NT / 256) {
            const float w = row < job.nrows ? as_const(job.rowg)[row] * rd : (job.erow ? rd : 0.0f);
            lds_store_u32(lut_base + (uint32_t)(row * 256 + d) * 4, __float_as_uint(w));
        }
    } else {
        const int n = (job.nrows + 1) * 256;
        for (int e = tid; e < n; e += NT) {
            const int row = e >> 8, d = e & 255;
            float w = job.erow ? as_global(job.range)[d] : 0.0f;
            if (row < job.nrows) w = as_global(job.rowg)[row] * as_global(job.range)[d];
            lds_store_u32(lut_base + (uint32_t)e * 4, __float_as_uint(w));
        }
    }
}

// ------------------------------------------------------------------------
// Unrolled variant for the canonical ring template (the one the GAUSS
// factory emits, TemplateFactory.cu:1092-1168).  Its taps come ring by ring,
// so the taps of a radius are a prefix of those of every larger one, and so
// are the rows of the fused table (one per distinct q = dy^2 + dx^2, in order
// of first appearance).  One kernel per staged halo therefore holds the tap
// list of its largest radius, with every tap's tile offset and table row
// compiled in (ds_read immediates; the compiler schedules across taps
// freely), and leaves it at the ring of the job's radius.  The host checks
// that the template really is the canonical one (same offsets, one weight per
// q) before choosing these kernels.

struct RingTap {
    int dy, dx, row;
    int side;      // 0: the ring's top/bottom rows; 1: right column; 2: left column
    bool first;    // first tap of its side column in this ring (j = -i + 1)
};

// The taps of rings 0 .. N.
template <int N>
struct RingTaps {
    static constexpr int T = (2 * N + 1) * (2 * N + 1);
    RingTap t[T];
    int rows[N + 1];       // table rows used by rings 0 .. i
    int xrow[N + 1];       // row of the first tap of ring i + 1 (REF's extra tap at radius i)
    constexpr RingTaps() : t{}, rows{}, xrow{}
    {
        int row_of[2 * (N + 1) * (N + 1) + 1] = {};   // row + 1 of q, 0 = not seen
        int n = 0, nrows = 0;
        for (int i = 0; i <= N; i++) {
            for (int j = (i == 0 ? 0 : -i + 1); j <= i; j++) {
                const int pts[4][2] = { { i, j }, { -i, j }, { j, i }, { j, -i } };
                for (int k = 0; k < (i == 0 ? 1 : 4); k++) {
                    const int dy = pts[k][0], dx = pts[k][1], q = dy * dy + dx * dx;
                    if (row_of[q] == 0) row_of[q] = ++nrows;
                    const int side = k < 2 ? 0 : k - 1;
                    t[n++] = RingTap{ dy, dx, row_of[q] - 1, side, side != 0 && j == -i + 1 };
                }
            }
            rows[i] = nrows;
            const int q = (i + 1) * (i + 1) + i * i;
            xrow[i] = row_of[q] ? row_of[q] - 1 : nrows;
        }
    }
};

template <int N>
inline constexpr RingTaps<N> kRing{};

constexpr int ring_first(int i) { return i == 0 ? 0 : (2 * i - 1) * (2 * i - 1); }   // first tap of ring i

// Smallest tap offset (in tile elements) of rings 0 .. N: the unrolled
// kernels address every fetch from one base placed there, so all ds_read
// offsets are non-negative immediates and no per-tap base register is needed.
template <int N, int TCOLS>
constexpr int ring_min_offset()
{
    int m = 0;
    for (int c = 0; c < RingTaps<N>::T; c++) {
        const int o = kRing<N>.t[c].dy * TCOLS + kRing<N>.t[c].dx;
        m = o < m ? o : m;
    }
    return m;
}

// Rows of the fused table a workgroup's LDS holds beside its tile and one
// more row.  Radii with more rows (16 and up: 135 or 136 rows at r = 16 against
// 122 beside 64 x 64 tiles and 134 beside 64 x 32 ones) keep the first ones
// fused; a tap of any other row reads E[d] from that last row
// and forms the factor g * E[d] itself, the product the fused rows hold,
// with the same single rounding.
template <int TW, int TGY, int HALO>
constexpr int ring_fused_rows()
{
    return (160 * 1024 - (int)kTileOff - Geo<TW, TGY, HALO>::TILE_BYTES) / 1024 - 1;
}

// Taps scheduled together between fences in the unrolled kernels: a fence
// after every ring_group() taps of the whole list (windows that start anew at
// each ring measured 3% slower).  us on 2048 x 2048, noise 10, one image:
//   REF flat from 4 to 16 taps, slower at 2 (506 at r = 15);
//   STD r = 3: 29.6 at 28 taps, 30.5 at 36 and more, 30.8 at 20;
//   STD r = 5, 7, 9, 11: 69.8, 125.6, 202, 311 at 60; 73.1, 129.6, 209, 321
//     at 20; 94, 155, 255, 316 at 64 (the registers then cost a workgroup);
//   STD r = 13, 15: 447, 579 at 20; 444, 581 at 40; 447, 592 at 48;
//   STD r = 18: 838 at 36, 841 at 30, 868 at 28, 855 at 52.
// The batch kernel holds both modes and keeps to windows whose registers
// leave two workgroups a CU (BATCH), six waves a SIMD to r = 8: STD r = 5, 7
// on 64 x 32 tiles of 4096 x 2048: 161.0, 269.2 at 24 taps, 158.7, 267.2 at 28,
// 156.5, 265.9 at 32 (r = 6 and 4 then slower), 161.0, 285.9 at 36.
template <int MODE, int HALO, bool BATCH>
constexpr int ring_group()
{
    if (MODE == kModeRef) return 4;
    if (BATCH) return HALO <= 8 ? 28 : (HALO <= 12 ? 24 : 40);
    return HALO <= 4 ? 28 : (HALO <= 12 ? 60 : (HALO <= 16 ? 20 : 36));
}

template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}

template <int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Smallest radius of a halo class (halo_class in bf_exact.hip: multiples of 4).
constexpr int halo_min_radius(int halo) { return halo - 3; }

// MINR: the smallest radius the kernel is used for.  Its rings are straight
// code; a branch before each of them measured 1% (REF) to 4% (STD) slower.
template <int MODE, int TW, int TGY, int HALO, int MINR, int GROUP>
__device__ __forceinline__ void tile_ring(const DevJob &job, int X0, int Y0, int lx, int gy)
{
    using G = Geo<TW, TGY, HALO>;
    constexpr uint32_t LUT_BASE = kTileOff + G::TILE_BYTES;
    constexpr int ROWB = G::TCOLS * 4;
    constexpr int FUSED = ring_fused_rows<TW, TGY, HALO>();
    const uint32_t lane = kTileOff + (uint32_t)(((4 * gy + HALO) * G::TCOLS + lx + HALO) * 4);
    const uint32_t c0 = lds_u32(lane), c1 = lds_u32(lane + ROWB);
    const uint32_t c2 = lds_u32(lane + 2 * ROWB), c3 = lds_u32(lane + 3 * ROWB);
    float t0 = 0.0f, t1 = 0.0f, t2 = 0.0f, t3 = 0.0f;
    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
    constexpr int MINB = ring_min_offset<HALO, G::TCOLS>() * 4;
    uint32_t tbase = lane + (uint32_t)MINB;         // >= 0: the halo covers every tap
    // Kept opaque: folded into `lane`, the taps above and left of the pixel
    // would need negative offsets, which ds_read's unsigned offset field
    // cannot hold (each such fetch then costs a v_add_u32).
    asm volatile("" : "+v"(tbase));
    uint32_t wp[2][4] = {};                         // STD: side-column windows (right, left)
    float wf[2][4] = {};
    // Gathers address W[row][d] as (4d + LUT_BASE) + row*1024; every 64 rows
    // have a base of their own, so that the offset fits the 16-bit field.
    // gs: the spatial weights of the ring's rows past FUSED, by min(|dy|, |dx|)
    auto tap = [&](auto ci, const float *gs) __attribute__((always_inline)) {
        constexpr RingTap tp = kRing<HALO>.t[decltype(ci)::value];
        constexpr int TAPB = (tp.dy * G::TCOLS + tp.dx) * 4 - MINB;   // >= 0
        constexpr bool SEP = tp.row >= FUSED;
        constexpr int LROW = SEP ? FUSED : tp.row;
        constexpr uint32_t WB = LUT_BASE + (uint32_t)(LROW / 64) * 65536u;
        constexpr uint32_t WOFF = (uint32_t)(LROW & 63) * 1024u;
        constexpr int AY = tp.dy < 0 ? -tp.dy : tp.dy, AX = tp.dx < 0 ? -tp.dx : tp.dx;
        auto weight = [&](uint32_t p, uint32_t c) __attribute__((always_inline)) {
            const float f = lds_f32(__builtin_amdgcn_sad_u8(p, c, WB) + WOFF);
            if constexpr (SEP)
                return gs[AY < AX ? AY : AX] * f;
            else
                return f;
        };
        if constexpr (MODE == kModeRef) {
            const uint32_t p = lds_u32(tbase + TAPB);
            const float pf = (float)(p & 0xFFu);
            const float f0 = weight(p, c0), f1 = weight(p, c1), f2 = weight(p, c2), f3 = weight(p, c3);
            t0 = t0 + f0 * pf; s0 = s0 + f0;
            t1 = t1 + f1 * pf; s1 = s1 + f1;
            t2 = t2 + f2 * pf; s2 = s2 + f2;
            t3 = t3 + f3 * pf; s3 = s3 + f3;
        } else {
            // Own window per row: row k reads tile row k + dy.  Along a side
            // column of a ring (dx = +-i, dy = j = -i+1 .. i, taps four apart
            // in ring order) row k at dy = j reads the pixel row k+1 read at
            // dy = j - 1: a window of the four pixels rows j .. j+3 of that
            // column (bytes and their float values) slides down one row per
            // tap, so such a tap fetches and converts one pixel, not four.
            uint32_t p0, p1, p2, p3;
            float q0, q1, q2, q3;
            if constexpr (tp.side != 0) {
                constexpr int sd = tp.side - 1;
                if constexpr (tp.first) {
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        wp[sd][m] = lds_u32(tbase + TAPB + m * ROWB);
                        wf[sd][m] = (float)(wp[sd][m] & 0xFFu);
                    }
                } else {
#pragma unroll
                    for (int m = 0; m < 3; m++) {
                        wp[sd][m] = wp[sd][m + 1];
                        wf[sd][m] = wf[sd][m + 1];
                    }
                    wp[sd][3] = lds_u32(tbase + TAPB + 3 * ROWB);
                    wf[sd][3] = (float)(wp[sd][3] & 0xFFu);
                }
                p0 = wp[sd][0]; p1 = wp[sd][1]; p2 = wp[sd][2]; p3 = wp[sd][3];
                q0 = wf[sd][0]; q1 = wf[sd][1]; q2 = wf[sd][2]; q3 = wf[sd][3];
            } else {
                p0 = lds_u32(tbase + TAPB); p1 = lds_u32(tbase + TAPB + ROWB);
                p2 = lds_u32(tbase + TAPB + 2 * ROWB); p3 = lds_u32(tbase + TAPB + 3 * ROWB);
                q0 = (float)(p0 & 0xFFu); q1 = (float)(p1 & 0xFFu);
                q2 = (float)(p2 & 0xFFu); q3 = (float)(p3 & 0xFFu);
            }
            const float f0 = weight(p0, c0), f1 = weight(p1, c1), f2 = weight(p2, c2), f3 = weight(p3, c3);
            t0 = t0 + f0 * q0; s0 = s0 + f0;
            t1 = t1 + f1 * q1; s1 = s1 + f1;
            t2 = t2 + f2 * q2; s2 = s2 + f2;
            t3 = t3 + f3 * q3; s3 = s3 + f3;
        }
    };
    // Keep the schedule local (a group of taps in flight), as the loop
    // version does: without a fence the compiler issues every gather of
    // the window first and spills them.  The empty asm reads and writes
    // the accumulators and clobbers memory, so neither the adds nor the
    // LDS reads move across it; it emits no instruction.
    auto fence = [&]() __attribute__((always_inline)) {
        asm volatile("" : "+v"(t0), "+v"(t1), "+v"(t2), "+v"(t3), "+v"(s0), "+v"(s1),
                     "+v"(s2), "+v"(s3)::"memory");
    };
    const int radius = __builtin_amdgcn_readfirstlane(job.radius);
    tap(std::integral_constant<int, 0>{}, nullptr);
    static_for<HALO>([&](auto ri) {
        constexpr int I = decltype(ri)::value + 1, C0 = ring_first(I), N = 8 * I;
        if constexpr (I > MINR)
            if (radius < I) return;
        // Weights of the ring's rows past the fused ones (q = I^2 + j^2),
        // loaded into scalar registers before the first tap: a scalar load
        // beside the taps would make each wait for every LDS read in flight.
        float gs[I + 1] = {};
        static_for<I + 1>([&](auto ji) {
            constexpr int J = decltype(ji)::value;
            // the ring's first tap with that q: (I, J), or (I, -J) where J = I
            constexpr int row = kRing<HALO>.t[C0 + 4 * (J + I - 1)].row;
            if constexpr (row >= FUSED) {
                gs[J] = as_const(job.rowg)[row];
                asm volatile("" : "+s"(gs[J]));
            }
        });
        static_for<N>([&](auto ci) {
            constexpr int C = C0 + decltype(ci)::value;
            tap(std::integral_constant<int, C>{}, gs);
            if constexpr (C % GROUP == GROUP - 1) fence();
        });
    });
    if constexpr (MODE == kModeRef) {
        // the extra tap (r + 1, -r): the one tap whose place the kernel reads
        const uint32_t p = lds_u32(lane + (uint32_t)(((radius + 1) * G::TCOLS - radius) * 4));
        const float pf = (float)(p & 0xFFu);
        const int xrow = __builtin_amdgcn_readfirstlane(job.xrow);
        const bool sep = xrow >= FUSED;
        const uint32_t wb = LUT_BASE + (uint32_t)(sep ? FUSED : xrow) * 1024u;
        float f0 = lds_f32(__builtin_amdgcn_sad_u8(p, c0, wb)), f1 = lds_f32(__builtin_amdgcn_sad_u8(p, c1, wb));
        float f2 = lds_f32(__builtin_amdgcn_sad_u8(p, c2, wb)), f3 = lds_f32(__builtin_amdgcn_sad_u8(p, c3, wb));
        if (sep) {
            const float g = as_const(job.rowg)[xrow];
            f0 = g * f0; f1 = g * f1; f2 = g * f2; f3 = g * f3;
        }
        t0 = t0 + f0 * pf; s0 = s0 + f0;
        t1 = t1 + f1 * pf; s1 = s1 + f1;
        t2 = t2 + f2 * pf; s2 = s2 + f2;
        t3 = t3 + f3 * pf; s3 = s3 + f3;
    }
    const int x = X0 + lx, y0 = Y0 + 4 * gy;
    if (x < job.W) {
        BF_GLOBAL uint8_t *o = as_global(job.out) + (int64_t)y0 * job.out_pitch + x;
        if (y0 < job.H) o[0] = to_u8(t0 / s0);
        if (y0 + 1 < job.H) o[job.out_pitch] = to_u8(t1 / s1);
        if (y0 + 2 < job.H) o[2 * job.out_pitch] = to_u8(t2 / s2);
        if (y0 + 3 < job.H) o[3 * job.out_pitch] = to_u8(t3 / s3);
    }
}

// hipFuncSetAttribute once per kernel (thread-safe static initialisation):
// allow the dynamic LDS of a kernel to reach the CU's 160 KB.
template <auto K>
hipError_t allow_full_lds()
{
    static const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(K),
                                                    hipFuncAttributeMaxDynamicSharedMemorySize,
                                                    160 * 1024);
    return e;
}

// Workgroups of `kern` (NT threads, lds bytes) that run at once on the
// device; 0 when one does not fit.  The answer depends on nothing else, so a
// thread keeps its last few (the queries are most of a small launch's host
// time).
inline int resident_groups(const void *kern, int nt, size_t lds)
{
    struct Entry {
        const void *kern;
        size_t lds;
        int nt, dev, groups;
    };
    constexpr int kEntries = 8;
    thread_local Entry last[kEntries] = {};
    thread_local int next = 0;
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess) return -1;
    for (const Entry &e : last)
        if (e.kern == kern && e.lds == lds && e.nt == nt && e.dev == dev) return e.groups;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, nt, lds) != hipSuccess)
        return -1;
    last[next] = Entry{ kern, lds, nt, dev, cus * per_cu };
    next = (next + 1) % kEntries;
    return cus * per_cu;
}

}  // namespace bfimpl
