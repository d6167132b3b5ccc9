/* HIP kernels for the SES mesh path on CDNA4 (gfx950, wave64).
 *
 * Floating-point expressions that decide labels, cube indices or vertex positions are written
 * in the evaluation order of the reference kernel they follow and the library is compiled with
 * -ffp-contract=off, so each operation rounds once (IEEE single precision, correctly rounded
 * division and sqrt).  Integer outputs (cell ids, atom order, labels, cube indices, vertex and
 * triangle ids) are therefore bit-identical to a host evaluation of the same formulas.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qs_common.h"
#include "qs_kernels.h"
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "qs_mc_table.h"

/* field-pass-2 tiles: x, y, z extents (P2R_TX in x for the fixed-radius kernel, whose halo costs
   (16 + 2R) / 16 in x) */
#define P2_TX 8
#define P2_TY 8
#define P2_TZ 32
#define P2R_TX 16 /* x extent of the fixed-radius kernel's tiles (halo cost (16 + 2R) / 16 in x) */

__constant__ uint64_t c_tri[256] = QS_TRI_PACKED_DATA;

/* cube corners and edges (see qs_mc_table.h): edge e runs from corner offset kEdgeLow[e] along
   axis kEdgeAxis[e]; packed into bit masks so that per-lane lookups are shifts, not loads */
constexpr int8_t kEdgeLow[12][3] = {{0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 0}, {0, 0, 1}, {1, 0, 1},
                                    {0, 1, 1}, {0, 0, 1}, {0, 0, 0}, {1, 0, 0}, {1, 1, 0}, {0, 1, 0}};
constexpr int8_t kEdgeAxis[12] = {0, 1, 0, 1, 0, 1, 0, 1, 2, 2, 2, 2};
constexpr uint32_t edge_low_bits(int c)
{
    uint32_t m = 0;
    for (int e = 0; e < 12; e++) m |= (uint32_t)(kEdgeLow[e][c] != 0) << e;
    return m;
}
constexpr uint32_t edge_axis_bits()
{
    uint32_t m = 0;
    for (int e = 0; e < 12; e++) m |= (uint32_t)kEdgeAxis[e] << (2 * e);
    return m;
}
constexpr uint32_t kEdgeLX = edge_low_bits(0), kEdgeLY = edge_low_bits(1), kEdgeLZ = edge_low_bits(2);
constexpr uint32_t kEdgeAX = edge_axis_bits();
static_assert(kEdgeLX == 0x622u && kEdgeLY == 0xC44u && kEdgeLZ == 0xF0u && kEdgeAX == 0xAA4444u, "edge tables");
/* the same, five bits per edge: low corner's z offset, x offset, y offset, axis (two bits) */
constexpr uint64_t edge_packed()
{
    uint64_t m = 0;
    for (int e = 0; e < 12; e++)
        m |= (uint64_t)(kEdgeLow[e][2] | kEdgeLow[e][0] << 1 | kEdgeLow[e][1] << 2 | kEdgeAxis[e] << 3) << (5 * e);
    return m;
}
constexpr uint64_t kEdgePacked = edge_packed();

/* ------------------------------------------------------------------------------------------ */
/* small helpers                                                                                */

__device__ __forceinline__ int iclamp(int f, int a, int b) { return max(a, min(f, b)); }

/* gridToSpace Kernels.cu:124-127: origin + (float)i * dx, two roundings */
__device__ __forceinline__ float grid_pos(float o, int i, float dx)
{
    float t = (float)i * dx;
    return o + t;
}

/* spaceToGrid Kernels.cu:119-123: truncation of (p - o) / dx */
__device__ __forceinline__ int cell_of(float p, float o, float dx) { return (int)((p - o) / dx); }

/* one axis' term of dist3_sq */
__device__ __forceinline__ float sq_dist(float a, float b)
{
    const float e = a - b;
    return e * e;
}

/* fast_distance Kernels.cu:149-155, left to right, IEEE sqrt */
/* the squared sum under dist3's root, with dist3's roundings */
__device__ __forceinline__ float dist3_sq(float ax, float ay, float az, float bx, float by, float bz)
{
    float ex = ax - bx, ey = ay - by, ez = az - bz;
    float x = ex * ex;
    float y = ey * ey;
    float z = ez * ez;
    float s = x + y;
    return s + z;
}

/* sqrtf, correctly rounded.  For a normal x or +inf the hardware root is within one ulp of the
   correctly rounded one, and Tuckerman's rounding test on the residuals of its two neighbours
   (exact FMAs) selects it; zero, denormal and NaN inputs take the general routine. */
__device__ __forceinline__ float sqrt_rn(float x)
{
    if (!(x >= 1.17549435e-38f)) return sqrtf(x);
    const float s = __builtin_amdgcn_sqrtf(x);
    const float sm = __uint_as_float(__float_as_uint(s) - 1u), sp = __uint_as_float(__float_as_uint(s) + 1u);
    float r = s;
    if (__builtin_fmaf(-sm, s, x) <= 0.0f) r = sm;
    if (__builtin_fmaf(-sp, s, x) > 0.0f) r = sp;
    return r;
}

__device__ __forceinline__ float dist3(float ax, float ay, float az, float bx, float by, float bz)
{
    float ex = ax - bx, ey = ay - by, ez = az - bz;
    float x = ex * ex;
    float y = ey * ey;
    float z = ez * ez;
    float s = x + y;
    s = s + z;
    return sqrtf(s);
}

__device__ __forceinline__ int tri_entry(uint64_t packed, int k) { return (int)((packed >> (4 * k)) & 0xF); }

/* number of triangles of a packed case: nibble k is 0xF exactly for k >= 3 * ntri (k < 16) */
__device__ __forceinline__ int tri_count_packed(uint64_t p)
{
    const uint64_t f = p & (p >> 1) & (p >> 2) & (p >> 3) & 0x1111111111111111ull; /* bit 4k: nibble k is 0xF */
    return (int)(__builtin_ctzll(f | (1ull << 63)) >> 2) / 3;
}

__device__ __forceinline__ int tri_count(int ci) { return tri_count_packed(c_tri[ci]); }

/* Segment lookups.  A prefix array pre (n + 1 non-decreasing entries, pre[n] = total) comes with
   a coarse index: coarse[k] = the segment holding item k << shift.  Segment of item v: start at
   coarse[v >> shift] and step forward past the segments that end at or before v (segments are
   long next to 2^shift items, so this is usually no step at all). */
template <int SHIFT, typename T>
__device__ __forceinline__ int seg_coarse(const T *__restrict__ pre, const uint32_t *__restrict__ coarse, T v)
{
    int j = (int)coarse[v >> SHIFT];
    while (pre[j + 1] <= v) j++;
    return j;
}

/* Workgroups are dealt to the eight XCDs round-robin (block b runs on XCD b % 8), and each XCD
   has its own L2.  This renumbers the blocks of an nb-block launch in groups of 8*C: inside a group
   each XCD runs C consecutive logical blocks, so neighbouring tiles share an L2 (their halo reads
   hit there and their partial output lines merge there before going to HBM), while the groups
   still spread every region of the grid over all eight XCDs.  A bijection on [0, nb): the last,
   incomplete group keeps its order.  Grid tiles use C = 8; per-vertex gathers, whose neighbours
   lie about one grid plane (a few thousand vertices) away, use C = 64. */
template <uint32_t C>
__device__ __forceinline__ uint32_t xcd_group(uint32_t b, uint32_t nb)
{
    constexpr uint32_t G = 8 * C;
    if (b >= nb / G * G) return b;
    const uint32_t w = b % G;
    return b - w + (w & 7u) * C + (w >> 3);
}
constexpr uint32_t XCD_CHUNK = 8;
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nb) { return xcd_group<XCD_CHUNK>(b, nb); }
/* the same renumbering with a group size chosen at launch (c >= 1) */
__device__ __forceinline__ uint32_t xcd_group_rt(uint32_t b, uint32_t nb, uint32_t c)
{
    const uint32_t G = 8 * c;
    if (b >= nb / G * G) return b;
    const uint32_t w = b % G;
    return b - w + (w & 7u) * c + (w >> 3);
}

/* molecule of block b of a batched launch, and the block's index inside the molecule */
__device__ __forceinline__ int batch_mol(const QsBatch &B, uint32_t b, uint32_t &local)
{
    if (!B.coarse) { /* one molecule: mols[0] */
        local = b;
        return 0;
    }
    const int j = seg_coarse<QS_COARSE_BLOCKS>(B.bpre, B.coarse, b);
    local = b - B.bpre[j];
    return B.mid ? B.mid[j] : j;
}

/* index of the segment of a sorted prefix array (n + 1 entries) that holds item v */
__device__ __forceinline__ int seg_of(const uint32_t *__restrict__ pre, int n, uint32_t v)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (pre[mid] <= v) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

/* segment of v for a wavefront whose items usually share one: the first active lane's segment
   is found with scalar loads, the others fall back to their own lookup (coarse == nullptr: one
   segment) */
__device__ __forceinline__ int seg_of_wave(const uint32_t *__restrict__ pre, const uint32_t *__restrict__ coarse, uint32_t v)
{
    if (!coarse) return 0;
    const uint32_t v0 = __builtin_amdgcn_readfirstlane(v);
    const int m0 = __builtin_amdgcn_readfirstlane(seg_coarse<QS_COARSE_ITEMS>(pre, coarse, v0));
    if (v >= pre[m0] && v < pre[m0 + 1]) return m0;
    return seg_coarse<QS_COARSE_ITEMS>(pre, coarse, v);
}

/* inclusive scan over the wave's lanes (all active): six data-parallel-primitive adds, where a
   shuffle through LDS per step made the scans bound by its latency */
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x)
{
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false); /* lane - 1, - 2, - 4, - 8 of the row of 16 */
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false);
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false); /* last lane of the row below, to rows 1 and 3 */
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false); /* lane 31, to rows 2 and 3 */
    return x;
}
/* the next (previous) lane's v; lane 63 (0) gets edge */
__device__ __forceinline__ uint64_t lane_above(uint64_t v, uint64_t edge)
{
    const int lo = __builtin_amdgcn_update_dpp((int)(uint32_t)edge, (int)(uint32_t)v, 0x130, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(uint32_t)(edge >> 32), (int)(uint32_t)(v >> 32), 0x130, 0xf, 0xf, false);
    return (uint64_t)(uint32_t)hi << 32 | (uint32_t)lo;
}
__device__ __forceinline__ uint64_t lane_below(uint64_t v, uint64_t edge)
{
    const int lo = __builtin_amdgcn_update_dpp((int)(uint32_t)edge, (int)(uint32_t)v, 0x138, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(uint32_t)(edge >> 32), (int)(uint32_t)(v >> 32), 0x138, 0xf, 0xf, false);
    return (uint64_t)(uint32_t)hi << 32 | (uint32_t)lo;
}
/* the largest of the wave's values */
__device__ __forceinline__ uint32_t wave_max(uint32_t x)
{
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false));
    x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false));
    return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}
/* lane 63's value */
__device__ __forceinline__ uint32_t wave_last(uint32_t x) { return (uint32_t)__builtin_amdgcn_readlane((int)x, 63); }

/* exclusive scan over the block; returns this thread's prefix, *total the block sum */
template <int NT>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t *total, uint32_t *lds)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint32_t x = wave_incl_scan(v);
    if (lane == 63) lds[wid] = x;
    __syncthreads();
    uint32_t below = 0, all = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; w++) {
        const uint32_t t = lds[w];
        below += (w < wid) ? t : 0u;
        all += t;
    }
    *total = all;
    __syncthreads();
    return x - v + below;
}

template <int NT>
__device__ __forceinline__ uint32_t block_sum(uint32_t v, uint32_t *lds)
{
    uint32_t t;
    block_excl_scan<NT>(v, &t, lds);
    return t;
}

/* sum of sums[0 .. b) for b <= 64, in every lane of the wave (a scan whose tile count is small
   takes its tiles' offsets this way instead of from a launch that scans the tile sums) */
template <int STRIDE = 1>
__device__ __forceinline__ uint32_t wave_sum_below(const uint32_t *__restrict__ sums, uint32_t b)
{
    const uint32_t lane = threadIdx.x & 63;
    return wave_last(wave_incl_scan((lane < b) ? sums[STRIDE * lane] : 0u));
}

/* bit position of the r-th set bit (from 0) of m, which has more than r */
__device__ __forceinline__ int nth_bit32(uint32_t m, uint32_t r)
{
    int b = 0;
#pragma unroll
    for (int h = 16; h >= 1; h >>= 1) {
        const uint32_t c = (uint32_t)__popc(m & ((1u << h) - 1u));
        const bool up = r >= c;
        r -= up ? c : 0u;
        m >>= up ? h : 0;
        b += up ? h : 0;
    }
    return b;
}

__device__ __forceinline__ int nth_bit(uint64_t w, uint32_t r)
{
    const uint32_t low = (uint32_t)__popc((uint32_t)w);
    const bool up = r >= low;
    return (up ? 32 : 0) + nth_bit32((uint32_t)(up ? w >> 32 : w), up ? r - low : r);
}

/* ------------------------------------------------------------------------------------------ */
/* device-wide exclusive scan of uint32 (reduce tiles, scan tile sums, scan tiles)              */

#define SCAN_NT 256
#define SCAN_IPT 8
#define SCAN_TILE (SCAN_NT * SCAN_IPT)

__global__ void __launch_bounds__(SCAN_NT) k_tile_reduce(const uint32_t *__restrict__ in, uint64_t n,
                                                         uint32_t *__restrict__ sums)
{
    __shared__ uint32_t lds[SCAN_NT / 64 + 1];
    uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE;
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        uint64_t i = base + (uint64_t)k * SCAN_NT + threadIdx.x;
        if (i < n) s += in[i];
    }
    uint32_t t = block_sum<SCAN_NT>(s, lds);
    if (threadIdx.x == 0) sums[blockIdx.x] = t;
}

/* out[i] = offsets[tile] + exclusive prefix inside the tile; in may alias out.  With self_sums
   (at most QS_SCAN_SELF_TILES tiles) the tile's offset is the sum of the tile sums before it. */
__global__ void __launch_bounds__(SCAN_NT) k_tile_scan(const uint32_t *in, uint32_t *out, uint64_t n,
                                                       const uint32_t *__restrict__ offsets,
                                                       uint32_t *__restrict__ total, const uint32_t *__restrict__ self_sums)
{
    __shared__ uint32_t lds[SCAN_NT / 64 + 1];
    uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_IPT;
    uint32_t v[SCAN_IPT];
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        uint64_t i = base + k;
        v[k] = (i < n) ? in[i] : 0u;
        s += v[k];
    }
    uint32_t tot;
    uint32_t pre = block_excl_scan<SCAN_NT>(s, &tot, lds);
    uint32_t off = offsets ? offsets[blockIdx.x] : (self_sums ? wave_sum_below(self_sums, blockIdx.x) : 0u);
    uint32_t run = off + pre;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        uint64_t i = base + k;
        if (i < n) out[i] = run;
        run += v[k];
    }
    if (total && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *total = off + tot;
}

/* a row word's counts, packed by k_mc_count: vertices (at most 4 x 64), triangles (at most 5 x 64)
   and polygonised cubes (at most 64) */
__device__ __forceinline__ uint32_t word_counts(uint32_t nv, uint32_t nt, uint32_t nc) { return nv | nt << 9 | nc << 18; }
__device__ __forceinline__ uint32_t word_verts(uint32_t c) { return c & 511u; }
__device__ __forceinline__ uint32_t word_tris(uint32_t c) { return (c >> 9) & 511u; }
__device__ __forceinline__ uint32_t word_cubes(uint32_t c) { return c >> 18; }

/* Marching-cubes word scans in one pass: per row word its vertex, triangle and cube counts and
   "active" flag (any nonzero) are scanned together.  Plane 0 = triangles, 1 = vertices, 2 = active
   words, 3 = cubes; the count kernel adds up each tile's four sums, which lie together. */
/* block p: exclusive scan of plane p of the tile sums in place, total to totals[p], plane 3's to
   totals[4]: totals[3] (the degenerate-triangle count, accumulated later) starts at zero */
__global__ void __launch_bounds__(SCAN_NT) k_scan_planes(uint32_t *__restrict__ sums, uint64_t ntiles,
                                                         uint32_t *__restrict__ totals)
{
    __shared__ uint32_t lds[SCAN_NT / 64 + 1];
    uint32_t *plane = sums + blockIdx.x; /* every fourth entry */
    uint32_t carry = 0;
    for (uint64_t b0 = 0; b0 < ntiles; b0 += SCAN_TILE) {
        const uint64_t base = b0 + (uint64_t)threadIdx.x * SCAN_IPT;
        uint32_t v[SCAN_IPT], s = 0;
#pragma unroll
        for (int k = 0; k < SCAN_IPT; k++) {
            v[k] = (base + k < ntiles) ? plane[4 * (base + k)] : 0u;
            s += v[k];
        }
        uint32_t tot;
        uint32_t run = carry + block_excl_scan<SCAN_NT>(s, &tot, lds);
#pragma unroll
        for (int k = 0; k < SCAN_IPT; k++) {
            if (base + k < ntiles) plane[4 * (base + k)] = run;
            run += v[k];
        }
        carry += tot;
    }
    if (threadIdx.x == 0) totals[blockIdx.x + (blockIdx.x >= 3u ? 1u : 0u)] = carry;
    if (blockIdx.x == 0 && threadIdx.x == 0) totals[3] = 0u;
}

/* An active word with items [first, first + count) is where every 256-item block whose first
   item lies in that range starts: it writes those blocks' start (its index in the active list),
   below the start array's capacity cap. */
__device__ __forceinline__ void mark_block_starts(uint32_t *__restrict__ start, uint32_t cap, uint32_t first, uint32_t count,
                                                  uint32_t r)
{
    for (uint32_t b = (first + 255u) >> 8; b < cap && (b << 8) < first + count; b++) start[b] = r;
}

/* per word: first vertex (vbw) and first triangle (tbw); active words listed in order; with
   bs.vstart, the first active word of every 256-vertex and 256-cube block, and the triangle
   blocks' counters cleared */
__global__ void __launch_bounds__(SCAN_NT) k_mc_scan4(const uint32_t *__restrict__ cnt, uint64_t n, const uint32_t *__restrict__ sums,
                                                      uint32_t *__restrict__ vbw, uint32_t *__restrict__ tbw,
                                                      uint32_t *__restrict__ list, uint32_t *__restrict__ avb,
                                                      uint32_t *__restrict__ acb, uint32_t list_base, int self,
                                                      uint32_t *__restrict__ totals, QsBlockStarts bs)
{
    if (bs.zero)
        for (uint32_t i = blockIdx.x * SCAN_NT + threadIdx.x; i < bs.nzero; i += gridDim.x * SCAN_NT) bs.zero[i] = 0u;
    /* (self: sums holds the raw tile sums of at most QS_SCAN_SELF_TILES tiles, each tile adds up
       the ones before it, and the last tile writes totals = {triangles, vertices, active, 0, cubes}) */
    /* wave w of the block takes words [w * 512, (w + 1) * 512) of the tile, 64 consecutive words
       per load; the scans run per group of 64 in order, carried across groups, and each group's active words are listed in order by ballot */
    __shared__ uint32_t wsum[4][SCAN_NT / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)wid * (64 * SCAN_IPT) + lane;
    const uint64_t below = (1ull << lane) - 1ull;
    uint32_t cw[SCAN_IPT], pv[SCAN_IPT], pt[SCAN_IPT], pc[SCAN_IPT], pa[SCAN_IPT];
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const uint64_t i = base + 64 * k;
        cw[k] = (i < n) ? cnt[i] : 0u;
    }
    uint32_t rv = 0, rt = 0, rc = 0, ra = 0; /* the wave's earlier groups */
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        /* triangles and cubes of a group of 64 words are scanned in one register (at most 64 x 320
           and 64 x 64) */
        const uint32_t own = word_tris(cw[k]) | word_cubes(cw[k]) << 16;
        const uint32_t xv = wave_incl_scan(word_verts(cw[k])), xt = wave_incl_scan(own);
        const uint64_t am = __ballot(cw[k] != 0u);
        pv[k] = rv + xv - word_verts(cw[k]);
        pt[k] = rt + ((xt - own) & 0xFFFFu);
        pc[k] = rc + ((xt - own) >> 16);
        pa[k] = ra + (uint32_t)__popcll(am & below);
        rv += wave_last(xv);
        const uint32_t last = wave_last(xt);
        rt += last & 0xFFFFu;
        rc += last >> 16;
        ra += (uint32_t)__popcll(am);
    }
    if (lane == 0) {
        wsum[0][wid] = rv;
        wsum[1][wid] = rt;
        wsum[2][wid] = ra;
        wsum[3][wid] = rc;
    }
    __syncthreads();
    uint32_t ov, ot, oa, oc;
    if (self) {
        ot = wave_sum_below<4>(sums, blockIdx.x);
        ov = wave_sum_below<4>(sums + 1, blockIdx.x);
        oa = wave_sum_below<4>(sums + 2, blockIdx.x);
        oc = wave_sum_below<4>(sums + 3, blockIdx.x);
        if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
            uint32_t tv = ov, tt = ot, ta = oa, tc = oc;
            for (int w = 0; w < SCAN_NT / 64; w++) {
                tv += wsum[0][w];
                tt += wsum[1][w];
                ta += wsum[2][w];
                tc += wsum[3][w];
            }
            totals[0] = tt;
            totals[1] = tv;
            totals[2] = ta;
            totals[3] = 0u;
            totals[4] = tc;
        }
    } else {
        ot = sums[4 * (size_t)blockIdx.x];
        ov = sums[4 * (size_t)blockIdx.x + 1];
        oa = sums[4 * (size_t)blockIdx.x + 2];
        oc = sums[4 * (size_t)blockIdx.x + 3];
    }
    for (int w = 0; w < wid; w++) {
        ov += wsum[0][w];
        ot += wsum[1][w];
        oa += wsum[2][w];
        oc += wsum[3][w];
    }
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const uint64_t i = base + 64 * k;
        if (i < n) {
            vbw[i] = ov + pv[k];
            tbw[i] = ot + pt[k];
            if (cw[k]) {
                const uint32_t r = oa + pa[k];
                avb[r] = ov + pv[k];
                acb[r] = oc + pc[k];
                list[r] = list_base + (uint32_t)i;
                if (bs.vstart) {
                    mark_block_starts(bs.vstart, bs.nv, ov + pv[k], word_verts(cw[k]), r);
                    mark_block_starts(bs.tstart, bs.nt, oc + pc[k], word_cubes(cw[k]), r);
                }
            }
        }
    }
}

/* The generic scan in one block of SCAN1_NT threads for at most QS_SCAN1_MAX entries: one launch
   instead of three.  The block runs over chunks of SCAN1_NT * SCAN_IPT entries in
   order, each wave 64 consecutive entries per load as above, carrying the running totals. */
#define SCAN1_NT 1024
#define SCAN1_W (SCAN1_NT / 64)

/* this wave's offset (waves below it) and the chunk total, from the per-wave sums */
__device__ __forceinline__ void scan1_offsets(const uint32_t *wsum, int wid, uint32_t &below, uint32_t &all)
{
    below = 0u;
    all = 0u;
#pragma unroll
    for (int w = 0; w < SCAN1_W; w++) {
        const uint32_t s = wsum[w];
        below += (w < wid) ? s : 0u;
        all += s;
    }
}

/* exclusive prefix of the wave's SCAN_IPT groups of 64 in place; returns the wave's total */
__device__ __forceinline__ uint32_t wave_groups_scan(uint32_t (&v)[SCAN_IPT])
{
    uint32_t run = 0;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const uint32_t x = wave_incl_scan(v[k]);
        v[k] = run + x - v[k];
        run += wave_last(x);
    }
    return run;
}

/* generic exclusive scan (in may equal out); total to *total if given */
__global__ void __launch_bounds__(SCAN1_NT) k_scan1(const uint32_t *in, uint32_t *out, uint64_t n, uint32_t *__restrict__ total)
{
    __shared__ uint32_t wsum[SCAN1_W];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t carry = 0;
    for (uint64_t c0 = 0; c0 < n; c0 += SCAN1_NT * SCAN_IPT) {
        const uint64_t base = c0 + (uint64_t)wid * (64 * SCAN_IPT) + lane;
        uint32_t v[SCAN_IPT];
#pragma unroll
        for (int k = 0; k < SCAN_IPT; k++) v[k] = (base + 64 * k < n) ? in[base + 64 * k] : 0u;
        const uint32_t run = wave_groups_scan(v);
        if (lane == 0) wsum[wid] = run;
        __syncthreads();
        uint32_t below, all;
        scan1_offsets(wsum, wid, below, all);
#pragma unroll
        for (int k = 0; k < SCAN_IPT; k++)
            if (base + 64 * k < n) out[base + 64 * k] = carry + below + v[k];
        carry += all;
        __syncthreads(); /* wsum is written again for the next chunk */
    }
    if (total && threadIdx.x == 0) *total = carry;
}

/* ------------------------------------------------------------------------------------------ */
/* bounding box (getMinMax CudaSurf.cu:149-174): partial boxes per molecule, then one wave    */

#define BB_NT 256
#define BB_NV 8 /* min x,y,z, max x,y,z, max radius, count of non-finite inputs */
#define BB_PMAX 256 /* partial boxes per molecule at most */

__device__ __forceinline__ void bb_combine(float *v, const float *w)
{
    for (int c = 0; c < 3; c++) v[c] = fminf(v[c], w[c]);
    for (int c = 3; c < 7; c++) v[c] = fmaxf(v[c], w[c]);
    v[7] += w[7];
}

/* the wave's lanes combined (minima, maxima and a sum of small integer counts: the same box in any
   order) */
__device__ __forceinline__ void bb_wave(float *v)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        float w[BB_NV];
#pragma unroll
        for (int c = 0; c < BB_NV; c++) w[c] = __shfl_xor(v[c], d, 64);
        bb_combine(v, w);
    }
}

/* block (p, m) of P partial boxes per molecule: atoms off[m] + p*NT + k*P*NT + t of molecule m ->
   part[m][p] (off == nullptr: one molecule, atoms [o0, o1)).  Bound by the latency of its loads:
   four atoms per thread are in flight. */
template <int NT>
__global__ void __launch_bounds__(NT) k_bbox_part(const float *__restrict__ pos, const float *__restrict__ rad,
                                                  const uint32_t *__restrict__ off, uint32_t o0, uint32_t o1,
                                                  float *__restrict__ part)
{
    const uint32_t P = gridDim.x;
    __shared__ float s[NT / 64][BB_NV];
    const int m = blockIdx.y, p = blockIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    float v[BB_NV] = {100000.0f, 100000.0f, 100000.0f, -100000.0f, -100000.0f, -100000.0f, 0.0f, 0.0f};
    const uint32_t beg = off ? off[m] : o0, end = off ? off[m + 1] : o1;
    for (uint32_t i0 = beg + p * NT + threadIdx.x; i0 < end; i0 += 4 * P * NT) {
        float q[4][4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            /* (past the end the thread's first atom again; 32-bit wrap-around included) */
            const uint32_t j = i0 + k * P * NT, i = (j < end && j >= i0) ? j : i0;
#pragma unroll
            for (int c = 0; c < 3; c++) q[k][c] = pos[3 * (size_t)i + c];
            q[k][3] = rad[i];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                v[c] = fminf(v[c], q[k][c]);
                v[3 + c] = fmaxf(v[3 + c], q[k][c]);
                if (!isfinite(q[k][c])) v[7] += 1.0f;
            }
            v[6] = fmaxf(v[6], q[k][3]);
            if (!isfinite(q[k][3])) v[7] += 1.0f;
        }
        if (i0 + 4 * P * NT < i0) break; /* (the index would wrap around) */
    }
    bb_wave(v);
    if (lane == 0)
        for (int c = 0; c < BB_NV; c++) s[wid][c] = v[c];
    __syncthreads();
    if (threadIdx.x < BB_NV) {
        const int c = threadIdx.x;
        float r = s[0][c];
        for (int w = 1; w < NT / 64; w++) r = c < 3 ? fminf(r, s[w][c]) : (c < 7 ? fmaxf(r, s[w][c]) : r + s[w][c]);
        part[((size_t)m * P + p) * BB_NV + c] = r;
    }
}

/* one wavefront per molecule: combine its P partial boxes, lane k taking partials k, k + 64, ... */
__global__ void __launch_bounds__(64) k_bbox_final(const float *__restrict__ part, int P, float *__restrict__ out)
{
    const int m = blockIdx.x, lane = threadIdx.x;
    float v[BB_NV] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY, -INFINITY, 0.0f};
    for (int p = lane; p < P; p += 64) {
        float w[BB_NV];
#pragma unroll
        for (int c = 0; c < BB_NV; c++) w[c] = part[((size_t)m * P + p) * BB_NV + c];
        bb_combine(v, w);
    }
    bb_wave(v);
    if (lane < BB_NV) {
        float r = v[0];
#pragma unroll
        for (int c = 1; c < BB_NV; c++) r = (lane == c) ? v[c] : r;
        out[BB_NV * m + lane] = r;
    }
}

/* ------------------------------------------------------------------------------------------ */
/* atom hashing and cell ordering                                                              */

/* hashAtoms Kernels.cu:185-216: cell id x-major (global over the batch); count atoms per cell.
   key[atom] = (cell, the atom's rank among its cell's atoms in the order the counts were taken):
   the scatter gives it a place in its cell with that rank, and k_place orders the cell's atoms. */
__global__ void __launch_bounds__(256) k_hash_count(QsBatch B, const float *__restrict__ pos, int2 *__restrict__ key,
                                                    uint32_t *__restrict__ count)
{
    uint32_t lb;
    const QsMol &M = B.mols[batch_mol(B, blockIdx.x, lb)];
    const uint32_t i = lb * 256 + threadIdx.x;
    if (i >= M.n_atoms) return;
    const QsGrid G = M.G;
    const size_t ga = (size_t)M.atom_off + i;
    /* in range for every atom by construction of the grid; clamped only as a memory guard */
    int cx = iclamp(cell_of(pos[3 * ga + 0], G.ox, G.dxn), 0, G.gn - 1);
    int cy = iclamp(cell_of(pos[3 * ga + 1], G.oy, G.dxn), 0, G.gn - 1);
    int cz = iclamp(cell_of(pos[3 * ga + 2], G.oz, G.dxn), 0, G.gn - 1);
    int h = (int)M.cell_off + ((G.gn * G.gn * cx) + (G.gn * cy) + cz);
    key[ga] = make_int2(h, (int)atomicAdd(&count[h], 1u));
}

__global__ void __launch_bounds__(256) k_scatter(const int2 *__restrict__ key, int n, const uint32_t *__restrict__ start,
                                                 int *__restrict__ slot)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int2 hr = key[i];
    slot[start[hr.x] + (uint32_t)hr.y] = i;
}

/* ------------------------------------------------------------------------------------------ */
/* field pass 1: probeIntersection + computeInOrOut Kernels.cu:344-475                         */
/*
 * Labels are kept as two bit masks per 64-voxel z-word of every (x, y) row: "outside" (no
 * admissible atom within r + probe) and "shell" (within r + probe of one, within r - dx of none);
 * a voxel in neither is inside.  Bits for z >= g are 0; the last layer of each axis is outside
 * (never written by the reference, CudaSurf.cu:664).
 *
 * k_pass1_rows: one wavefront per row word of up to four adjacent rows.  The lanes take the
 * candidate atoms of the rows (the atoms of the neighbour cells any of their voxels would visit),
 * and each lane computes, for its atom and each row, the z-interval of voxels it reaches.  Along a row the single-precision distance
 * sqrt((x^2 + y^2) + z^2) is non-increasing then non-decreasing in z (every rounding is
 * monotone), so {z : d(z) < T} is an interval; it is located from the closed-form estimate and
 * then pinned by evaluating the reference's float predicate at its ends.  A voxel counts an atom
 * only if the atom's cell is one of the 27 (clamped) cells it would visit, as in the reference.
 * The wave ORs the lanes' interval masks.  Cost per row word: a few hundred instructions,
 * instead of ~44 candidate atoms per voxel.
 */

/* OR of v over the 64 lanes (all active), returned wave-uniform: row shifts inside each 16-lane
   row, then row broadcasts, leave the total in lane 63 */
__device__ __forceinline__ uint32_t wave_or_u32(uint32_t v)
{
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true); /* row_shr:1 */
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true); /* row_shr:2 */
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true); /* row_shr:4 */
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true); /* row_shr:8 */
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false); /* row_bcast:15 */
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false); /* row_bcast:31 */
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ uint64_t wave_or_u64(uint64_t v)
{
    return ((uint64_t)wave_or_u32((uint32_t)(v >> 32)) << 32) | wave_or_u32((uint32_t)v);
}

/* bits [a, b] (inclusive, 0 <= a, b <= 63) */
__device__ __forceinline__ uint64_t bit_range(int a, int b)
{
    if (a > b) return 0ull;
    uint64_t hi = (b >= 63) ? ~0ull : ((2ull << b) - 1ull);
    uint64_t lo = (1ull << a) - 1ull;
    return hi & ~lo;
}

/* bits of the word starting at z0 for z < L */
__device__ __forceinline__ uint64_t bits_below(int L, int z0)
{
    int n = L - z0;
    return n <= 0 ? 0ull : (n >= 64 ? ~0ull : ((1ull << n) - 1ull));
}

/* smallest float s with sqrtf(s) >= T (T > 0), so that for v >= 0: sqrtf(v) < T <=> v < s.
   Every step uses the correctly rounded sqrtf, so the comparison is the reference's. */
__device__ __forceinline__ float sqrt_threshold(float T)
{
    if (!(T > 0.0f)) return -1.0f;
    float s = T * T;
    for (int i = 0; i < 8 && sqrt_rn(s) < T; i++) s = __uint_as_float(__float_as_uint(s) + 1u);
    for (int i = 0; i < 8 && s > 0.0f; i++) {
        float q = __uint_as_float(__float_as_uint(s) - 1u);
        if (sqrt_rn(q) >= T) s = q;
        else break;
    }
    return s;
}

/* one atom seen from one row: fl(S + fl(e(z)^2)) with S = fl(x^2 + y^2), e(z) = az - pz(z) */
struct RowAtom {
    float az, S, dx, oz;
    __device__ __forceinline__ float Zf(int z) const
    {
        float pz = grid_pos(oz, z, dx);
        float e = az - pz;
        return e * e;
    }
    __device__ __forceinline__ bool pred(int z, float ss) const
    {
        float v = S + Zf(z);
        return v < ss;
    }
};

/* exact [L, R] within [zlo, zhi] where the predicate holds; zb = its argmin in [zlo, zhi];
   L > R if none.  zc is the atom's z in voxel units; zc -+ h only start the exact walks, so the
   hardware root (within an ulp) serves for h. */
__device__ __forceinline__ void row_interval(const RowAtom &A, float ss, int zlo, int zhi, int zb, float zc, float inv_dx,
                                             int &L, int &R)
{
    L = 1;
    R = 0;
    if (zlo > zhi || !A.pred(zb, ss)) return;
    float h2 = ss - A.S;
    float h = (h2 > 0.0f) ? __builtin_amdgcn_sqrtf(h2) * inv_dx : 0.0f;
    int l = iclamp((int)ceilf(zc - h), zlo, zb);
    if (A.pred(l, ss)) {
        while (l > zlo && A.pred(l - 1, ss)) l--;
    } else {
        while (l < zb && !A.pred(l, ss)) l++;
    }
    int r = iclamp((int)floorf(zc + h), zb, zhi);
    if (A.pred(r, ss)) {
        while (r < zhi && A.pred(r + 1, ss)) r++;
    } else {
        while (r > zb && !A.pred(r, ss)) r--;
    }
    L = l;
    R = r;
}

/* the interval of row_interval from its closed form (qs_closed_interval), or false */
__device__ __forceinline__ bool fast_interval(float h2, float zc, float inv_dx, float eps, int zlo, int zhi, int &L, int &R)
{
    return qs_closed_interval(__builtin_amdgcn_sqrtf(h2), h2, zc, inv_dx, eps, zlo, zhi, L, R);
}

/* an atom's float thresholds of its near (r + probe) and inside (r - dx) tests, and its
   neighbour-cell y and z (packed) */
__device__ __forceinline__ float4 atom_aux(const float4 &a, const QsGrid &G, int acy, int acz)
{
    return make_float4(sqrt_threshold(QS_PROBE + a.w), sqrt_threshold(a.w - G.dx), __int_as_float((acy << 16) | acz), 0.0f);
}

/* per atom in cell order, once: the atom (perm gives its input index) as float4 x, y, z, r, the
   exact float thresholds of its near (r + probe) and inside (r - dx) tests, and its neighbour-cell
   y and z (packed) */
__global__ void __launch_bounds__(256) k_gather_aux(QsBatch B, const int *__restrict__ perm, const float *__restrict__ pos,
                                                    const float *__restrict__ rad, float4 *__restrict__ sx,
                                                    float4 *__restrict__ aux)
{
    uint32_t lb;
    const QsMol &M = B.mols[batch_mol(B, blockIdx.x, lb)];
    const uint32_t i = lb * 256 + threadIdx.x;
    if (i >= M.n_atoms) return;
    const QsGrid G = M.G;
    const size_t k = (size_t)M.atom_off + i;
    const int id = perm[k];
    const float4 a = make_float4(pos[3 * (size_t)id], pos[3 * (size_t)id + 1], pos[3 * (size_t)id + 2], rad[id]);
    sx[k] = a;
    aux[k] = atom_aux(a, G, iclamp(cell_of(a.y, G.oy, G.dxn), 0, G.gn - 1), iclamp(cell_of(a.z, G.oz, G.dxn), 0, G.gn - 1));
}

/* Every atom to its place in the order (cell, index), the order a stable sort by cell id gives
   (thrust::sort CudaSurf.cu:610-612): its cell's first place plus the number of the cell's atoms (in
   slot, in any order) of lower index; with the gathered atom as k_gather_aux writes it, and every cell's
   range (sortCell Kernels.cu:306-341).  Bound by the gathers of the atoms.  With a thread per cell that
   sorted its atoms in place, a gather after it and a clear before, all steps of the cells of 50,000
   atoms took 33 us instead of 27, of 200,000 49 instead of 40, of a million 136 instead of 128 (and
   159 with a thread per atom in input order, whose writes are then scattered). */
__global__ void __launch_bounds__(256) k_place(QsBatch B, const uint32_t *__restrict__ start,
                                               const int *__restrict__ slot, uint32_t ncell, const float *__restrict__ pos,
                                               const float *__restrict__ rad, int *__restrict__ perm, int2 *__restrict__ cse,
                                               float4 *__restrict__ sx, float4 *__restrict__ aux)
{
    for (uint32_t c = blockIdx.x * 256u + threadIdx.x; c < ncell; c += gridDim.x * 256u) {
        const uint32_t b = start[c], e = start[c + 1];
        cse[c] = b == e ? make_int2(QS_EMPTY, QS_EMPTY) : make_int2((int)b, (int)e);
    }
    uint32_t lb;
    const QsMol &M = B.mols[batch_mol(B, blockIdx.x, lb)];
    const uint32_t i = lb * 256 + threadIdx.x;
    if (i >= M.n_atoms) return;
    const QsGrid G = M.G;
    /* (threads go by place, not by atom: gathers of atoms, but writes next to each other) */
    const uint32_t id = (uint32_t)slot[M.atom_off + i];
    const float4 a = make_float4(pos[3 * (size_t)id], pos[3 * (size_t)id + 1], pos[3 * (size_t)id + 2], rad[id]);
    const int cx = iclamp(cell_of(a.x, G.ox, G.dxn), 0, G.gn - 1), cy = iclamp(cell_of(a.y, G.oy, G.dxn), 0, G.gn - 1),
              cz = iclamp(cell_of(a.z, G.oz, G.dxn), 0, G.gn - 1);
    const uint32_t h = M.cell_off + (uint32_t)((G.gn * G.gn * cx) + (G.gn * cy) + cz), b = start[h], e = start[h + 1];
    uint32_t at = b;
    for (uint32_t q = b; q < e; q++) at += slot[q] < (int)id ? 1u : 0u;
    perm[at] = (int)id;
    sx[at] = a;
    aux[at] = atom_aux(a, G, cy, cz);
}

/* Cells of a molecule of at most PER * 1,024 atoms and CELLS_MAX cells in one block: hashing, counts,
   their scan and the order (cell, index) in LDS, and with GATHER the gathered atoms, with the results
   of k_hash_count, the scan, k_scatter and k_place.  Bound by the latency of its
   few dependent steps, where those launches (and a clear) each had that of a launch; an atom's place
   within its cell is the number of the cell's atoms of lower index, so nothing is sorted.  The cells
   of 300 atoms took 24 us and take 9, of 2,000 atoms 26 and 14.
   With put, the run's one molecule comes in the arguments and goes to *put for the later launches. */
constexpr uint32_t CELLS_NT = 1024;
template <int PER, bool GATHER>
__global__ void __launch_bounds__(CELLS_NT) k_cells(const QsMol *__restrict__ mols, QsMol one, QsMol *__restrict__ put,
                                                    const float *__restrict__ pos, const float *__restrict__ rad,
                                                    uint32_t *__restrict__ start, int *__restrict__ perm, int2 *__restrict__ cse,
                                                    float4 *__restrict__ sx, float4 *__restrict__ aux)
{
    static_assert(PER % 4 == 0 && PER * CELLS_NT < 65536, "atoms four at a time, 16-bit places");
    extern __shared__ uint32_t cells_lds[];
    __shared__ uint32_t wsum[CELLS_NT / 64];
    if (put && threadIdx.x == 0) *put = one;
    const QsMol &M = put ? one : mols[blockIdx.x];
    const QsGrid G = M.G;
    const int gn = G.gn;
    const uint32_t n = M.n_atoms, a0 = M.atom_off, ncell = (uint32_t)(gn * gn * gn), c0 = M.cell_off;
    uint16_t *const cnt = (uint16_t *)cells_lds; /* atoms per cell, then the cells' first places */
    uint16_t *const slot = (uint16_t *)(cells_lds + ncell / 2 + 1); /* atoms by cell, in the order they were counted */
    for (uint32_t c = threadIdx.x; c <= ncell / 2; c += CELLS_NT) cells_lds[c] = 0u;
    __syncthreads();
    uint32_t hr[PER]; /* cell << 16 | rank in the cell */
#pragma unroll
    for (uint32_t k0 = 0; k0 < PER; k0 += 4) {
        if (k0 * CELLS_NT >= n) break;
        float p[4][3];
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
            const float *__restrict__ q = pos + 3 * (size_t)(a0 + min((k0 + k) * CELLS_NT + threadIdx.x, n - 1u));
            p[k][0] = q[0];
            p[k][1] = q[1];
            p[k][2] = q[2];
        }
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
            const int cx = iclamp(cell_of(p[k][0], G.ox, G.dxn), 0, gn - 1), cy = iclamp(cell_of(p[k][1], G.oy, G.dxn), 0, gn - 1),
                      cz = iclamp(cell_of(p[k][2], G.oz, G.dxn), 0, gn - 1);
            const uint32_t h = (uint32_t)((gn * gn * cx) + (gn * cy) + cz);
            const uint32_t half = 16u * (h & 1u); /* (counts of two cells in a word) */
            uint32_t r = 0;
            if ((k0 + k) * CELLS_NT + threadIdx.x < n) r = (atomicAdd(&cells_lds[h >> 1], 1u << half) >> half) & 0xFFFFu;
            hr[k0 + k] = h << 16 | r;
        }
    }
    __syncthreads();
    /* exclusive scan of the counts: a wave takes consecutive groups of 64 */
    const uint32_t lane = threadIdx.x & 63, wid = threadIdx.x >> 6, ng = (ncell + CELLS_NT - 1) / CELLS_NT;
    uint32_t run = 0;
    for (uint32_t k = 0; k < ng; k++) {
        const uint32_t c = (wid * ng + k) * 64u + lane;
        const uint32_t v = c < ncell ? cnt[c] : 0u, x = wave_incl_scan(v);
        if (c < ncell) cnt[c] = (uint16_t)(run + x - v);
        run += wave_last(x);
    }
    if (lane == 0) wsum[wid] = run;
    if (threadIdx.x == 0) cnt[ncell] = (uint16_t)n;
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < wid; w++) before += wsum[w];
    for (uint32_t k = 0; k < ng; k++) {
        const uint32_t c = (wid * ng + k) * 64u + lane;
        if (c < ncell) {
            const uint32_t v = cnt[c] + before;
            cnt[c] = (uint16_t)v;
            start[c0 + c] = a0 + v;
        }
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) start[c0 + ncell] = a0 + n;
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < PER; k++) {
        const uint32_t i = k * CELLS_NT + threadIdx.x;
        if (i < n) slot[cnt[hr[k] >> 16] + (hr[k] & 0xFFFFu)] = (uint16_t)i;
    }
    for (uint32_t c = threadIdx.x; c < ncell; c += CELLS_NT) {
        const uint32_t b = cnt[c], e = cnt[c + 1];
        cse[c0 + c] = b == e ? make_int2(QS_EMPTY, QS_EMPTY) : make_int2((int)(a0 + b), (int)(a0 + e));
    }
    __syncthreads();
    const float inv_gn = 1.0f / (float)gn;
#pragma unroll
    for (uint32_t k = 0; k < PER; k++) {
        const uint32_t i = k * CELLS_NT + threadIdx.x;
        if (i < n) {
            const uint32_t h = hr[k] >> 16, b = cnt[h], e = cnt[h + 1];
            uint32_t at = a0 + b;
            for (uint32_t q = b; q < e; q++) at += slot[q] < i ? 1u : 0u;
            perm[at] = (int)(a0 + i);
            if constexpr (GATHER) {
                const float *__restrict__ p = pos + 3 * (size_t)(a0 + i);
                const float4 a = make_float4(p[0], p[1], p[2], rad[a0 + i]);
                /* the cell's z and y: h < 2^16, so the quotients are exact */
                const int xy = (int)(((float)h + 0.5f) * inv_gn), cz = (int)h - gn * xy;
                const int cy = xy - gn * (int)(((float)xy + 0.5f) * inv_gn);
                sx[at] = a;
                aux[at] = atom_aux(a, G, cy, cz);
            }
        }
    }
}

/* rows per wavefront: R consecutive y rows (R * dx <= neighbour-cell size, so they span at most
   two neighbour cells in y and the candidate set is at most 3 x 4 cell columns) */
#define P1_RMAX 4
#define P1_QCAP 128

__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__global__ void __launch_bounds__(256) k_pass1_rows(QsBatch B, const uint32_t *__restrict__ cstart_all,
                                                    const float4 *__restrict__ sx, const float4 *__restrict__ aux,
                                                    uint64_t *__restrict__ outm_all, uint64_t *__restrict__ shellm_all)
{
    __shared__ int queue_all[4][P1_QCAP];
    /* wave-uniform values go through readfirstlane so that they live in scalar registers */
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int *queue = queue_all[wid];
    uint32_t lb;
    const QsMol &M = B.mols[batch_mol(B, blockIdx.x, lb)];
    const QsGrid G = M.G;
    const int g = G.g, gn = G.gn, W = (int)M.W, R = M.rows_per_wave;
    const uint32_t *__restrict__ cstart = cstart_all + M.cell_off;
    uint64_t *__restrict__ outm = outm_all + M.word_off;
    uint64_t *__restrict__ shellm = shellm_all + M.word_off;
    /* one wavefront per group of R rows, looping over the rows' W words: the group's setup
       (molecule, rows, x and y cells) is paid once */
    const int nby = (g + 4 * R - 1) / (4 * R);
    const int by = (int)(lb % (uint32_t)nby);
    const int x = M.p1_lo + (int)(lb / (uint32_t)nby);
    const int x1 = M.p1_hi;
    const int y0 = (by * 4 + wid) * R;
    if (y0 >= g || x >= x1) return; /* whole wavefront */
    const int ny = min(R, g - y0);
    if (x >= g - 1) {
        for (int w = 0; w < W; w++) {
            const int nvalid = min(64, g - w * 64);
            const uint64_t valid = (nvalid >= 64) ? ~0ull : ((1ull << nvalid) - 1ull);
            if (lane < ny) {
                size_t widx = ((size_t)x * g + y0 + lane) * W + w;
                outm[widx] = valid;
                shellm[widx] = 0ull;
            }
        }
        return;
    }
    const float dx = G.dx, inv_dx = 1.0f / G.dx;
    const float px = grid_pos(G.ox, x, dx);
    const int cx = cell_of(px, G.ox, G.dxn);
    float py[P1_RMAX];
    int cyl[P1_RMAX], cyh[P1_RMAX];
#pragma unroll
    for (int k = 0; k < P1_RMAX; k++) {
        int yk = min(y0 + min(k, ny - 1), g - 1);
        py[k] = grid_pos(G.oy, yk, dx);
        int cy = cell_of(py[k], G.oy, G.dxn);
        cyl[k] = iclamp(cy - 1, 0, gn - 1);
        cyh[k] = iclamp(cy + 1, 0, gn - 1);
    }
    for (int w = 0; w < W; w++) {
        const int z0 = w * 64;
        const int nvalid = min(64, g - z0);
        const uint64_t valid = (nvalid >= 64) ? ~0ull : ((1ull << nvalid) - 1ull);
        wave_lds_sync(); /* the previous word's queue reads are done */
        /* this lane's voxel z cell; the wave's cells are monotone in the lane */
        const int zl = min(z0 + lane, g - 1);
        const int cz = cell_of(grid_pos(G.oz, zl, dx), G.oz, G.dxn);
        const int czmin = __builtin_amdgcn_readfirstlane(cz), czmax = __builtin_amdgcn_readlane(cz, 63);
        const int D = czmax - czmin + 1; /* distinct z cells + 1 */
        const int zc0 = iclamp(czmin - 1, 0, gn - 1), zc1 = iclamp(czmax + 1, 0, gn - 1);
        const int xa = iclamp(cx - 1, 0, gn - 1), xb = iclamp(cx + 1, 0, gn - 1);
        const int ya = cyl[0], yb = cyh[P1_RMAX - 1];
        /* candidate atoms: up to 3 x 4 contiguous ranges of the cell-ordered array */
        int rs[12], pre[13];
        pre[0] = 0;
    #pragma unroll
        for (int i = 0; i < 3; i++) {
    #pragma unroll
            for (int j = 0; j < 4; j++) {
                int k = 4 * i + j;
                int xc = xa + i, yc = ya + j;
                int len = 0, st = 0;
                if (xc <= xb && yc <= yb) {
                    int h0 = (xc * gn + yc) * gn + zc0;
                    st = (int)cstart[h0];
                    len = (int)cstart[h0 + (zc1 - zc0) + 1] - st;
                }
                rs[k] = st;
                pre[k + 1] = pre[k] + len;
            }
        }
        const int total = pre[12];
        const int zmax = min(z0 + 63, g - 2); /* labelled voxels: z <= g-2 (z = g-1 is outside) */
        if (total == 0) {
            /* no atom can reach these rows: every voxel is outside */
            if (lane < ny) {
                const size_t widx = ((size_t)x * g + y0 + lane) * W + w;
                outm[widx] = valid;
                shellm[widx] = 0ull;
            }
            continue;
        }
        /* tab (lane j) = number of lanes whose z cell is < czmin + j, j = 0..D */
        int tab = (lane >= D) ? 64 : 0;
        if (D < 64) {
            for (int d = 1; d < D; d++) {
                uint64_t m = __ballot(cz < czmin + d);
                if (lane == d) tab = __popcll(m);
            }
        }
        uint64_t m_in[P1_RMAX], m_near[P1_RMAX];
    #pragma unroll
        for (int k = 0; k < P1_RMAX; k++) m_in[k] = m_near[k] = 0ull;

        /* interval work for up to 64 queued atoms, one per lane */
        auto process = [&](int count) {
            const int id = (lane < count) ? queue[lane] : -1;
            float4 a = make_float4(0.f, 0.f, 0.f, 0.f), ax = make_float4(0.f, 0.f, 0.f, 0.f);
            int acz = czmin, acy = 0;
            if (id >= 0) {
                a = sx[id];
                ax = aux[id];
                const int packed = __float_as_int(ax.z);
                acy = packed >> 16;
                acz = packed & 0xFFFF;
            }
            /* voxels whose z cell admits the atom's z cell: lanes [La, Ra] */
            int La, Ra;
            if (D < 64) {
                int j1 = acz - 1 - czmin, j2 = acz + 2 - czmin;
                int t1 = __shfl(tab, iclamp(j1, 0, 63), 64);
                int t2 = __shfl(tab, iclamp(j2, 0, 63), 64);
                La = (j1 <= 0) ? 0 : (j1 >= D ? 64 : t1);
                Ra = ((j2 >= D) || (acz == gn - 1)) ? 63 : ((j2 <= 0) ? -1 : t2 - 1);
            } else {
                const int alo = iclamp(cz - 1, 0, gn - 1), ahi = iclamp(cz + 1, 0, gn - 1);
                int lo_i = 0, hi_i = 64;
                for (int it = 0; it < 7; it++) {
                    int mid = (lo_i + hi_i) >> 1;
                    int v = __shfl(ahi, min(mid, 63), 64);
                    if (lo_i < hi_i) {
                        if (v >= acz) hi_i = mid;
                        else lo_i = mid + 1;
                    }
                }
                La = lo_i;
                lo_i = 0;
                hi_i = 64;
                for (int it = 0; it < 7; it++) {
                    int mid = (lo_i + hi_i) >> 1;
                    int v = __shfl(alo, min(mid, 63), 64);
                    if (lo_i < hi_i) {
                        if (v > acz) hi_i = mid;
                        else lo_i = mid + 1;
                    }
                }
                Ra = lo_i - 1;
            }
            if (id < 0) return;
            const int zlo = z0 + La, zhi = min(z0 + Ra, zmax);
            if (zlo > zhi) return;
            const float sN = ax.x, sD = ax.y;
            const float ex = a.x - px;
            const float X = ex * ex;
            const float zc = (a.z - G.oz) * inv_dx;
            RowAtom A;
            A.az = a.z;
            A.dx = dx;
            A.oz = G.oz;
            const int zb0 = iclamp((int)floorf(zc), zlo, zhi);
    #pragma unroll
            for (int k = 0; k < P1_RMAX; k++) {
                if (k >= ny) break;
                if (acy < cyl[k] || acy > cyh[k]) continue; /* row's y cell does not admit the atom */
                float ey = a.y - py[k];
                float Y = ey * ey;
                A.S = X + Y;
                if (!(A.S < sN)) continue;
                int zb = zb0;
                if (zb + 1 <= zhi && A.Zf(zb + 1) < A.Zf(zb)) zb = zb + 1;
                int L, Rr;
                row_interval(A, sN, zlo, zhi, zb, zc, inv_dx, L, Rr);
                if (L > Rr) continue;
                m_near[k] |= bit_range(L - z0, Rr - z0);
                if (!(A.S < sD)) continue;
                row_interval(A, sD, L, Rr, zb, zc, inv_dx, L, Rr);
                if (L <= Rr) m_in[k] |= bit_range(L - z0, Rr - z0);
            }
        };

        /* candidates that can reach one of the rows (xy distance below r + probe) are queued */
        int qn = 0;
        const float pymin = py[0], pymax = py[ny - 1];
        for (int base = 0; base < total; base += 64) {
            const int kk = base + lane;
            int id = -1;
    #pragma unroll
            for (int q = 0; q < 12; q++)
                if (kk >= pre[q] && kk < pre[q + 1]) id = rs[q] + (kk - pre[q]);
            bool keep = false;
            if (id >= 0) {
                const float4 a = sx[id];
                const float sN = aux[id].x;
                const float ex = a.x - px;
                const float X = ex * ex;
                const float yy = fminf(fmaxf(a.y, pymin), pymax); /* nearest row y */
                const float ey = a.y - yy;
                const float Y = ey * ey;
                keep = (X + Y) < sN * 1.0001f + 1e-6f; /* conservative: exact tests follow */
            }
            const uint64_t km = __ballot(keep);
            if (keep) queue[qn + __popcll(km & ((1ull << lane) - 1ull))] = id;
            qn += __popcll(km);
            wave_lds_sync();
            if (qn >= 64) {
                process(64);
                wave_lds_sync();
                const int rest = qn - 64;
                int moved = (lane < rest) ? queue[64 + lane] : 0;
                wave_lds_sync();
                if (lane < rest) queue[lane] = moved;
                wave_lds_sync();
                qn = rest;
            }
        }
        if (qn > 0) process(qn);

    #pragma unroll
        for (int k = 0; k < P1_RMAX; k++) {
            m_in[k] = wave_or_u64(m_in[k]);
            m_near[k] = wave_or_u64(m_near[k]);
        }
        if (lane < ny) {
            uint64_t mi = 0ull, mn = 0ull;
    #pragma unroll
            for (int k = 0; k < P1_RMAX; k++)
                if (lane == k) {
                    mi = m_in[k];
                    mn = m_near[k];
                }
            const int y = y0 + lane;
            uint64_t lab = (zmax >= z0 && y < g - 1) ? bit_range(0, zmax - z0) : 0ull;
            mi &= lab;
            mn &= lab;
            size_t widx = ((size_t)x * g + y) * W + w;
            outm[widx] = valid & ~(mi | mn);
            shellm[widx] = mn & ~mi;
        }
    }
}

/* OR bits [L, R] (absolute z) into a row's words in LDS (32-bit halves of the row words).  An
   interval of at most 32 voxels takes one or two of them, from one 64-bit shift. */
__device__ __forceinline__ void lds_or_range(uint32_t *row, int L, int R)
{
    const int n = R - L;
    uint32_t *w = row + (L >> 5);
    if (n < 32) {
        const uint64_t m = (uint64_t)(~0u >> (31 - n)) << (L & 31);
        atomicOr(w, (uint32_t)m);
        if (m >> 32) atomicOr(w + 1, (uint32_t)(m >> 32));
        return;
    }
    atomicOr(w, ~0u << (L & 31));
    for (w++; w < row + (R >> 5); w++) atomicOr(w, ~0u);
    atomicOr(w, ~0u >> (31 - (R & 31)));
}

/* Field pass 1 by scatter into LDS: one block per slab of up to P1S_MAXROWS consecutive y rows of
   one x plane, all z.  Each candidate atom (x cells cx-1..cx+1 times the slab's y cells, every z
   cell) takes the rows whose y cell admits it and, lane by lane, ORs its exact near and inside
   z-intervals (the ones of k_pass1_rows) into the slab's two masks.  The z-intervals are clipped
   to the voxels whose z cell admits the atom, so each voxel sees exactly the atoms of its 27
   neighbour cells, as in probeIntersection (Kernels.cu:394-475); inside wins over near, which
   makes the result independent of the order of the ORs.
   Bound by VALU issue over the (atom, row) pairs, 730 an atom at 0.2 A.  Three things keep a pair
   short: its interval comes from the closed form (fast_interval), not from walking the predicate;
   the inside intervals, which one pair in seven has at 0.5 A, are taken apart from the near ones,
   so that the lanes without one do not wait; and an interval of 32 voxels is ORed with one 64-bit
   shift.  50,000 atoms at 0.2 A 0.313 -> 0.185 ms, 256 molecules at 0.5 A 1.05 -> 0.60 ms, a million
   atoms at 0.5 A 0.87 -> 0.49 ms; with the row prefixes by data-parallel primitives instead of
   shuffles through LDS 0.170, 0.56 and 0.45. */
#define P1S_MAXROWS 256   /* rows per slab block at most (row indexes in the queue are 8-bit) */
#define P1S_DEFROWS 64    /* rows per slab block when no tuned count is set */
#define P1S_MAXCOL 256
/* a wave takes its queued atoms as (atom, row) items when twice the item rounds of 64 are fewer than
   the largest row count of one atom, i.e. when walking atoms would leave most lanes idle (an item
   costs the shuffles of its atom's values).  Pass 1 on the 50,000-atom 0.2 A mesh and on 256
   molecules at 0.5 A: ratio 1 0.208 and 0.775 ms, 3/2 0.191 and 0.612, 2 0.185 and 0.600, 3 0.186
   and 0.622. */
#define P1_FLAT 2
__global__ void __launch_bounds__(256) k_pass1_slab(QsBatch B, const uint32_t *__restrict__ cstart_all,
                                                    const float4 *__restrict__ sx, const float4 *__restrict__ aux,
                                                    uint64_t *__restrict__ outm_all, uint64_t *__restrict__ shellm_all,
                                                    uint64_t *__restrict__ negm_all, uint64_t *__restrict__ zerom_all,
                                                    uint8_t *__restrict__ tflag, uint8_t tmark,
                                                    uint32_t *__restrict__ clear, uint32_t nclear)
{
    /* counters that a later launch adds to */
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < nclear; i += gridDim.x * 256u) clear[i] = 0u;
    extern __shared__ __align__(16) uint64_t p1s_dyn[];
    __shared__ uint32_t colpre[P1S_MAXCOL + 1], colst[P1S_MAXCOL];
    __shared__ int q_id[4][P1_QCAP], q_rows[4][P1_QCAP], q_z[4][P1_QCAP];
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t lb;
    const QsMol &M = B.mols[batch_mol(B, blockIdx.x, lb)];
    const QsGrid G = M.G;
    const int g = G.g, gn = G.gn, W = (int)M.W, YB = M.slab_rows;
    const uint32_t *__restrict__ cstart = cstart_all + M.cell_off;
    uint64_t *__restrict__ outm = outm_all + M.word_off;
    uint64_t *__restrict__ shellm = shellm_all + M.word_off;
    const int nyb = (g + YB - 1) / YB;
    const int x = M.p1_lo + (int)(lb / (uint32_t)nyb);
    const int y0 = (int)(lb % (uint32_t)nyb) * YB;
    if (x >= M.p1_hi) return; /* whole block */
    const int ny = min(YB, g - y0);
    const size_t wbase = ((size_t)x * g + y0) * W;
    uint64_t *__restrict__ negm = negm_all ? negm_all + M.word_off : nullptr;
    uint64_t *__restrict__ zerom = zerom_all ? zerom_all + M.word_off : nullptr;
    if (x >= g - 1) {
        /* the last plane is not labelled: outside */
        for (int t = threadIdx.x; t < ny * W; t += 256) {
            const int w = t % W;
            outm[wbase + t] = bits_below(g, w * 64);
            shellm[wbase + t] = 0ull;
            if (negm) {
                negm[wbase + t] = 0ull;
                zerom[wbase + t] = 0ull;
            }
        }
        return;
    }
    uint64_t *nearw = p1s_dyn, *insw = p1s_dyn + (size_t)YB * W;
    /* yfirst[c] (zfirst[c]) = first y (z) whose neighbour cell is >= c, g if none; c = 0..gn+1 */
    int *yfirst = (int *)(p1s_dyn + 2 * (size_t)YB * W), *zfirst = yfirst + (gn + 2);
    for (int t = threadIdx.x; t < ny * W; t += 256) nearw[t] = insw[t] = 0ull;
    for (int t = threadIdx.x; t < gn + 2; t += 256) yfirst[t] = zfirst[t] = g;
    __syncthreads();
    const float dx = G.dx, inv_dx = 1.0f / G.dx;
    const float eps0 = qs_interval_eps0(G.oz, g, dx, inv_dx), eps1 = qs_interval_eps1(inv_dx);
    const float ymargin = qs_row_margin(G.oy, g, dx, inv_dx), ymargin_r = qs_row_margin_r(inv_dx);
    for (int i = threadIdx.x; i < g; i += 256) {
        const int cy = min(cell_of(grid_pos(G.oy, i, dx), G.oy, G.dxn), gn + 1);
        const int cyp = i ? min(cell_of(grid_pos(G.oy, i - 1, dx), G.oy, G.dxn), gn + 1) : -1;
        for (int c = cyp + 1; c <= cy; c++) yfirst[c] = i;
        const int cz = min(cell_of(grid_pos(G.oz, i, dx), G.oz, G.dxn), gn + 1);
        const int czp = i ? min(cell_of(grid_pos(G.oz, i - 1, dx), G.oz, G.dxn), gn + 1) : -1;
        for (int c = czp + 1; c <= cz; c++) zfirst[c] = i;
    }
    /* labelled rows of the slab: y <= g - 2 */
    const int ylast = min(y0 + ny - 1, g - 2);
    const float px = grid_pos(G.ox, x, dx);
    const int cx = cell_of(px, G.ox, G.dxn);
    const int xa = iclamp(cx - 1, 0, gn - 1), xb = iclamp(cx + 1, 0, gn - 1);
    const int ya = iclamp(cell_of(grid_pos(G.oy, y0, dx), G.oy, G.dxn) - 1, 0, gn - 1);
    const int yb = iclamp(cell_of(grid_pos(G.oy, max(ylast, y0), dx), G.oy, G.dxn) + 1, 0, gn - 1);
    const int nyc = yb - ya + 1, ncol = (xb - xa + 1) * nyc;
    /* candidate columns: every z cell of (xc, yc), contiguous in the cell-ordered atoms */
    uint32_t len = 0;
    if ((int)threadIdx.x < ncol) {
        const int xc = xa + (int)threadIdx.x / nyc, yc = ya + (int)threadIdx.x % nyc;
        const size_t h0 = ((size_t)xc * gn + yc) * gn;
        colst[threadIdx.x] = cstart[h0];
        len = cstart[h0 + gn] - cstart[h0];
    }
    /* exclusive prefix of the column lengths (ncol <= 256) */
    {
        const uint32_t v = wave_incl_scan(len);
        __shared__ uint32_t wsum[4];
        if (lane == 63) wsum[wid] = v;
        __syncthreads();
        uint32_t add = 0;
        for (int k = 0; k < wid; k++) add += wsum[k];
        colpre[threadIdx.x + 1] = add + v;
        if (threadIdx.x == 0) colpre[0] = 0;
    }
    __syncthreads();
    const int total = (int)colpre[ncol];
    const int rows_hi = ylast - y0; /* rows 0..rows_hi of the slab are labelled */
    int *qid = q_id[wid], *qrows = q_rows[wid], *qz = q_z[wid];

    /* The wave's queued atoms, lane k < count holding atom k: first their near intervals, then
       their inside ones.  Each lane walks its own atom's rows, unless the row counts are so uneven
       that most lanes would idle: the atoms' rows are then items pre_k .. pre_k + rows - 1 that the
       lanes take 64 at a time, each with its atom's values from the lane that holds it.  An (atom,
       row) pair gives the atom's exact z-interval in the row, ORed into the slab's mask (the ORs are
       order-independent).  One loop body serves both ways and both masks: four copies of it took
       32 KB of code.  Called by the whole wave. */
    auto process = [&](int count) {
        int rr = 0, zr = 0, nr[2] = {0, 0}, r0[2] = {0, 0};
        float X = 0.0f, sN = 0.0f, sD = 0.0f, zc = 0.0f, az = 0.0f, ay = 0.0f;
        if (lane < count) {
            const int id = qid[lane];
            rr = qrows[lane];
            zr = qz[lane];
            r0[0] = rr & 0xFF;
            nr[0] = (rr >> 8) - r0[0] + 1;
            const float4 a = sx[id], ax = aux[id];
            sN = ax.x;
            sD = ax.y;
            const float ex = a.x - px;
            X = ex * ex;
            zc = (a.z - G.oz) * inv_dx;
            az = a.z;
            ay = a.y;
            if (X < sD) {
                const float h = __builtin_amdgcn_sqrtf(sD - X) * inv_dx, yc = (ay - G.oy) * inv_dx - (float)y0;
                const float ym = ymargin + ymargin_r * (a.w + QS_PROBE);
                r0[1] = max(qs_row_lo(yc, h, ym), r0[0]);
                nr[1] = max(min(qs_row_hi(yc, h, ym), rr >> 8) - r0[1] + 1, 0);
            }
        }
#pragma unroll 1
        for (int p = 0; p < 2; p++) {
            const int n = p ? nr[1] : nr[0], first = p ? r0[1] : r0[0];
            const float thr = p ? sD : sN;
            uint32_t *const mask = (uint32_t *)(p ? insw : nearw);
            int pre = (int)wave_incl_scan((uint32_t)n);
            const int nitems = (int)wave_last((uint32_t)pre), most = (int)wave_max((uint32_t)n);
            pre -= n; /* exclusive */
            const bool walk = P1_FLAT * ((nitems + 63) >> 6) >= most;
            const int rounds = walk ? most : (nitems + 63) >> 6;
#pragma unroll 1
            for (int it = 0; it < rounds; it++) {
                bool on = it < n;
                int yr = first + it, iz = zr;
                float iX = X, ithr = thr, izc = zc, iaz = az, iay = ay;
                if (!walk) {
                    const int j = it * 64 + lane;
                    /* the item's atom: the last lane whose first item is at or below j */
                    int o = 0;
#pragma unroll
                    for (int step = 32; step >= 1; step >>= 1)
                        if (__shfl(pre, o + step, 64) <= j) o += step;
                    iX = __shfl(X, o, 64);
                    ithr = __shfl(thr, o, 64);
                    izc = __shfl(zc, o, 64);
                    iaz = __shfl(az, o, 64);
                    iay = __shfl(ay, o, 64);
                    iz = __shfl(zr, o, 64);
                    yr = __shfl(first, o, 64) + j - __shfl(pre, o, 64);
                    on = j < nitems;
                }
                if (!on) continue;
                const float ey = iay - grid_pos(G.oy, y0 + yr, dx);
                const float Y = ey * ey;
                const float S = iX + Y;
                if (!(S < ithr)) continue;
                const int zlo = iz & 0xFFFF, zhi = iz >> 16;
                int L, Rr;
                if (!fast_interval(ithr - S, izc, inv_dx, eps0 + eps1 * ithr, zlo, zhi, L, Rr)) {
                    RowAtom A;
                    A.az = iaz;
                    A.S = S;
                    A.dx = dx;
                    A.oz = G.oz;
                    int zb = iclamp((int)floorf(izc), zlo, zhi);
                    if (zb + 1 <= zhi && A.Zf(zb + 1) < A.Zf(zb)) zb = zb + 1;
                    row_interval(A, ithr, zlo, zhi, zb, izc, inv_dx, L, Rr);
                }
                if (L <= Rr) lds_or_range(mask + (size_t)yr * (2 * W), L, Rr);
            }
        }
    };

    int qn = 0;
    if (rows_hi >= 0) {
        /* (one place calls process: its code is inlined once) */
        bool more = true;
        for (int base = wid * 64; more; base += 256) {
            more = base < total;
            const int k = base + lane;
            bool keep = false;
            int id = 0, rows = 0, zr = 0;
            if (k < total) {
                int lo = 0, hi = ncol - 1;
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if ((int)colpre[mid] <= k) lo = mid;
                    else hi = mid - 1;
                }
                id = (int)colst[lo] + (k - (int)colpre[lo]);
                const float4 a = sx[id], ax = aux[id];
                const float ex = a.x - px;
                const float X = ex * ex;
                if (X < ax.x) {
                    const int packed = __float_as_int(ax.z);
                    const int acy = packed >> 16, acz = packed & 0xFFFF;
                    /* rows whose y cell admits the atom: cy >= acy - 1, and cy <= acy + 1 unless acy is the last cell */
                    int ylo = yfirst[max(acy - 1, 0)];
                    int yhi = (acy == gn - 1) ? g - 1 : yfirst[acy + 2] - 1;
                    /* rows the atom can reach in y (a superset: the exact test is per row) */
                    const float h = __builtin_amdgcn_sqrtf(ax.x - X) * inv_dx, yc = (a.y - G.oy) * inv_dx;
                    const float ym = ymargin + ymargin_r * (a.w + QS_PROBE);
                    ylo = max(ylo, qs_row_lo(yc, h, ym));
                    yhi = min(yhi, qs_row_hi(yc, h, ym));
                    const int r0 = max(ylo - y0, 0), r1 = min(yhi - y0, rows_hi);
                    /* voxels whose z cell admits the atom, labelled ones only (z <= g - 2) */
                    const int zlo = zfirst[max(acz - 1, 0)];
                    const int zhi = min((acz == gn - 1) ? g - 1 : zfirst[acz + 2] - 1, g - 2);
                    keep = r0 <= r1 && zlo <= zhi;
                    rows = r0 | (r1 << 8);
                    zr = zlo | (zhi << 16);
                }
            }
            const uint64_t km = __ballot(keep);
            if (keep) {
                const int slot = qn + __popcll(km & ((1ull << lane) - 1ull));
                qid[slot] = id;
                qrows[slot] = rows;
                qz[slot] = zr;
            }
            qn += __popcll(km);
            wave_lds_sync();
            if (qn >= 64 || (!more && qn > 0)) {
                process(min(qn, 64));
                wave_lds_sync();
                if (qn <= 64) {
                    qn = 0;
                    continue;
                }
                const int rest = qn - 64;
                int m0 = 0, m1 = 0, m2 = 0;
                if (lane < rest) {
                    m0 = qid[64 + lane];
                    m1 = qrows[64 + lane];
                    m2 = qz[64 + lane];
                }
                wave_lds_sync();
                if (lane < rest) {
                    qid[lane] = m0;
                    qrows[lane] = m1;
                    qz[lane] = m2;
                }
                wave_lds_sync();
                qn = rest;
            }
        }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < ny * W; t += 256) {
        const int yr = t / W, w = t - yr * W;
        const uint64_t valid = bits_below(g, w * 64);
        uint64_t mi = 0ull, mn = 0ull;
        if (yr <= rows_hi) {
            mi = insw[t];
            mn = nearw[t];
        }
        outm[wbase + t] = valid & ~(mi | mn);
        const uint64_t sh = mn & ~mi;
        shellm[wbase + t] = sh;
        if (negm) {
            /* the sign words of a voxel without a shell voxel in its pass-2 tile: inside (-dx)
               is negative, outside (the probe radius) is not, no field value is zero; field
               pass 2 rewrites the tiles that hold a shell voxel, which it finds marked here */
            negm[wbase + t] = valid & (mi | mn);
            zerom[wbase + t] = 0ull;
            if (sh && tflag && M.tile_off != ~0u && x >= M.p2_lo && x < M.p2_hi) {
                const uint32_t nbz = (uint32_t)(g + P2_TZ - 1) / P2_TZ, nby = (uint32_t)(g + P2_TY - 1) / P2_TY;
                const uint32_t tyx = ((uint32_t)(x - M.p2_lo) / P2R_TX) * nby + (uint32_t)(y0 + yr) / P2_TY;
                if ((uint32_t)sh) tflag[M.tile_off + tyx * nbz + 2 * w] = tmark;
                if (sh >> 32) tflag[M.tile_off + tyx * nbz + 2 * w + 1] = tmark;
            }
        }
    }
}

/* per-voxel form (27 cells per voxel, as the reference); cross-check of k_pass1_rows */
__global__ void __launch_bounds__(256) k_pass1_direct(QsBatch B, const int2 *__restrict__ cse_all,
                                                      const float4 *__restrict__ sx, uint64_t *__restrict__ outm_all,
                                                      uint64_t *__restrict__ shellm_all)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    uint32_t lb;
    const QsMol &M = B.mols[batch_mol(B, blockIdx.x, lb)];
    const QsGrid G = M.G;
    const int g = G.g, W = (int)M.W;
    const int2 *__restrict__ cse = cse_all + M.cell_off;
    uint64_t *__restrict__ outm = outm_all + M.word_off;
    uint64_t *__restrict__ shellm = shellm_all + M.word_off;
    const int nby = (g + 3) / 4;
    const int w = (int)(lb % (uint32_t)W);
    const int y = (int)((lb / (uint32_t)W) % (uint32_t)nby) * 4 + wid;
    const int x = M.p1_lo + (int)(lb / ((uint32_t)W * nby));
    if (y >= g || x >= M.p1_hi) return;
    const int z = w * 64 + lane;
    uint8_t res = QS_OUT;
    if (x < g - 1 && y < g - 1 && z < g - 1) {
        const float dx = G.dx;
        float px = grid_pos(G.ox, x, dx), py = grid_pos(G.oy, y, dx), pz = grid_pos(G.oz, z, dx);
        int cx = cell_of(px, G.ox, G.dxn), cy = cell_of(py, G.oy, G.dxn), cz = cell_of(pz, G.oz, G.dxn);
        const int gn = G.gn;
        bool near = false, inside = false;
        for (int a = -1; a <= 1 && !inside; a++) {
            int ix = iclamp(cx + a, 0, gn - 1);
            for (int b = -1; b <= 1 && !inside; b++) {
                int iy = iclamp(cy + b, 0, gn - 1);
                for (int c = -1; c <= 1 && !inside; c++) {
                    int iz = iclamp(cz + c, 0, gn - 1);
                    int2 se = cse[(gn * gn * ix) + (gn * iy) + iz];
                    if (se.x >= QS_EMPTY) continue;
                    for (int id = se.x; id < se.y; id++) {
                        float4 at = sx[id];
                        float d = dist3(at.x, at.y, at.z, px, py, pz);
                        if (d < at.w - dx) {
                            inside = true;
                            break;
                        }
                        if (d < (QS_PROBE + at.w)) near = true;
                    }
                }
            }
        }
        res = inside ? QS_IN : (near ? QS_SHELL : QS_OUT);
    }
    uint64_t mo = __ballot(z < g && res == QS_OUT);
    uint64_t ms = __ballot(z < g && res == QS_SHELL);
    if (lane == 0) {
        size_t widx = ((size_t)x * g + y) * W + w;
        outm[widx] = mo;
        shellm[widx] = ms;
    }
}

/* ------------------------------------------------------------------------------------------ */
/* field pass 2 (distanceFieldRefine Kernels.cu:478-545)                                        */
/*
 * For a shell voxel v the reference takes the minimum, over "outside" voxels q of the (2r+1)^3
 * window clamped to the grid, of the single-precision distance between their world positions.
 * Every such float distance lies within delta of dx*sqrt(n) for the integer n = |q - v|^2, and
 * norms that differ give distances further apart than 2*delta, so the minimum is attained among
 * the outside voxels whose norm lies within [nmin, nmax(nmin)], nmin being the exact smallest
 * norm.  The tile kernel finds nmin with three separable integer passes in LDS (z by bit scan
 * of the outside mask, then y, then x) and evaluates the reference's float distance only for
 * those candidates.  The result is the reference's value bit for bit.
 */


/* bits [s, s + len) of a row of W mask words (bit i <-> z = s + i), zero outside [0, 64 W) */
__device__ __forceinline__ uint64_t row_bits(const uint64_t *__restrict__ rp, int W, int s, int len)
{
    int w0 = s >> 6; /* floor */
    int sh = s & 63;
    uint64_t a = (w0 >= 0 && w0 < W) ? rp[w0] : 0ull;
    uint64_t v = a >> sh;
    if (sh) {
        uint64_t b = (w0 + 1 >= 0 && w0 + 1 < W) ? rp[w0 + 1] : 0ull;
        v |= b << (64 - sh);
    }
    if (len < 64) v &= (1ull << len) - 1ull;
    return v;
}

size_t qs_pass2_lds_bytes(int r)
{
    size_t LX = P2_TX + 2 * r, LY = P2_TY + 2 * r;
    size_t dt = (3 * r * r < 255) ? 1 : 2;
    return LX * LY * 8 + P2_TX * P2_TY * 4 + LX * LY * P2_TZ * dt + LX * P2_TY * P2_TZ * dt;
}

/* sign (field < 0) and zero (field == 0) bits of the field, one ballot per wave-half: lanes 0-31
   are the 32 voxels (gx, gy, tz0..tz0+31), lanes 32-63 the same z range of row gy + 1 */
__device__ __forceinline__ void emit_sign_bits(uint32_t *__restrict__ negm, uint32_t *__restrict__ zerom, int W, int g,
                                               int gx, int gy, int tz0, bool valid, float res)
{
    const int lane = threadIdx.x & 63;
    uint64_t n = __ballot(valid && res < 0.0f);
    uint64_t zr = __ballot(valid && res == 0.0f);
    if ((lane & 31) == 0 && valid) {
        size_t w32 = ((size_t)gx * g + gy) * (2 * (size_t)W) + (tz0 >> 5);
        negm[w32] = (uint32_t)(lane ? (n >> 32) : n);
        zerom[w32] = (uint32_t)(lane ? (zr >> 32) : zr);
    }
}

template <typename DT>
__global__ void __launch_bounds__(256) k_pass2_tile(QsBatch B, const uint64_t *__restrict__ outm_all,
                                                    const uint64_t *__restrict__ shellm_all,
                                                    float *__restrict__ field_all,
                                                    uint32_t *__restrict__ negm_all, uint32_t *__restrict__ zerom_all,
                                                    const int *__restrict__ offs, const int *__restrict__ norm_start,
                                                    const int *__restrict__ enum_end)
{
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int s_flags;
    constexpr int INF = (sizeof(DT) == 1) ? 0xFF : 0xFFFF;
    uint32_t lb;
    const QsMol &M = B.mols[batch_mol(B, blockIdx.x, lb)];
    const QsGrid G = M.G;
    const int r = G.r, g = G.g, W = (int)M.W;
    const uint64_t *__restrict__ outm = outm_all + M.word_off;
    const uint64_t *__restrict__ shellm = shellm_all + M.word_off;
    float *__restrict__ field = field_all + M.vox_off;
    uint32_t *__restrict__ negm = negm_all + 2 * M.word_off;
    uint32_t *__restrict__ zerom = zerom_all + 2 * M.word_off;
    const int x0 = M.p2_lo, x1 = M.p2_hi;
    const uint32_t nbx = (g + P2_TZ - 1) / P2_TZ, nby = (g + P2_TY - 1) / P2_TY;
    const int bidx = (int)(lb % nbx), bidy = (int)((lb / nbx) % nby), bidz = (int)(lb / (nbx * nby));
    const int LX = P2_TX + 2 * r, LY = P2_TY + 2 * r, LZ = P2_TZ + 2 * r;
    uint64_t *rows = (uint64_t *)smem;
    uint32_t *own = (uint32_t *)(smem + (size_t)LX * LY * 8);
    DT *DZ = (DT *)(smem + (size_t)LX * LY * 8 + P2_TX * P2_TY * 4);
    DT *DY = DZ + (size_t)LX * LY * P2_TZ;
    const int tz0 = bidx * P2_TZ, ty0 = bidy * P2_TY, tx0 = x0 + bidz * P2_TX;
    if (threadIdx.x == 0) s_flags = 0;
    __syncthreads();

    /* 1. outside bits of the haloed tile; shell bits of the tile */
    int fl = 0;
    for (int row = threadIdx.x; row < LX * LY; row += 256) {
        int lx = row / LY, ly = row - lx * LY;
        int gx = tx0 - r + lx, gy = ty0 - r + ly;
        uint64_t m = 0ull;
        /* planes outside [p1_lo, p1_hi) are not stored (and are read by no output voxel) */
        if (gx >= M.p1_lo && gx < M.p1_hi && gy >= 0 && gy < g)
            m = row_bits(outm + ((size_t)gx * g + gy) * W, W, tz0 - r, LZ);
        rows[row] = m;
        if (m) fl |= 2;
    }
    for (int t = threadIdx.x; t < P2_TX * P2_TY; t += 256) {
        int tx = t / P2_TY, ty = t - tx * P2_TY;
        int gx = tx0 + tx, gy = ty0 + ty;
        uint32_t m = 0u;
        if (gx < x1 && gx < g && gy < g) m = (uint32_t)row_bits(shellm + ((size_t)gx * g + gy) * W, W, tz0, P2_TZ);
        own[t] = m;
        if (m) fl |= 1;
    }
    if (fl) atomicOr(&s_flags, fl);
    __syncthreads();
    const int flags = s_flags;

    const int ty = threadIdx.x / P2_TZ, tz = threadIdx.x - ty * P2_TZ;
    const int gy = ty0 + ty, gz = tz0 + tz;
    const bool vyz = gy < g && gz < g;
    const float dx = G.dx;
    if (flags != 3) {
        /* no shell voxel, or no outside voxel within reach: outside -> probe, else -dx */
        for (int tx = 0; tx < P2_TX; tx++) {
            int gx = tx0 + tx;
            if (gx >= x1 || gx >= g) break;
            bool out = (rows[(size_t)(tx + r) * LY + (ty + r)] >> (tz + r)) & 1ull;
            float res = out ? QS_PROBE : -dx;
            const uint32_t om = own[tx * P2_TY + ty];
            if (vyz && ((om >> tz) & 1u)) field[((size_t)gx * g + gy) * g + gz] = res;
            emit_sign_bits(negm, zerom, W, g, gx, gy, tz0, vyz, res);
        }
        return;
    }

    /* 2. z: squared distance to the nearest outside voxel within |c| <= r along each row */
    for (int w = threadIdx.x; w < LX * LY * P2_TZ; w += 256) {
        int row = w / P2_TZ, z = w - row * P2_TZ;
        uint64_t m = rows[row];
        int best = INF;
        if (m) {
            int c = z + r;
            uint64_t up = m >> c;
            if (up) {
                int d = __builtin_ctzll(up);
                if (d <= r) best = d * d;
            }
            uint64_t dn = m & ((2ull << c) - 1ull);
            if (dn) {
                int d = c - (63 - __builtin_clzll(dn));
                if (d <= r) best = min(best, d * d);
            }
        }
        DZ[w] = (DT)best;
    }
    __syncthreads();

    /* 3. y */
    for (int w = threadIdx.x; w < LX * P2_TY * P2_TZ; w += 256) {
        int lx = w / (P2_TY * P2_TZ);
        int rem = w - lx * (P2_TY * P2_TZ);
        int yy = rem / P2_TZ, z = rem - yy * P2_TZ;
        int best = INF;
        for (int b = -r; b <= r; b++) {
            int v = DZ[((size_t)lx * LY + (yy + r + b)) * P2_TZ + z];
            if (v != INF) best = min(best, v + b * b);
        }
        DY[w] = (DT)best;
    }
    __syncthreads();

    /* 4. x, then the field value of each output voxel */
    const float vy = grid_pos(G.oy, gy, dx), vz = grid_pos(G.oz, gz, dx);
    for (int tx = 0; tx < P2_TX; tx++) {
        int gx = tx0 + tx;
        if (gx >= x1 || gx >= g) break;
        bool out = (rows[(size_t)(tx + r) * LY + (ty + r)] >> (tz + r)) & 1ull;
        bool shell = (own[tx * P2_TY + ty] >> tz) & 1u;
        float res;
        if (!vyz || out) {
            res = QS_PROBE;
        } else if (!shell) {
            res = -dx;
        } else {
            int nmin = INF;
            for (int a = -r; a <= r; a++) {
                int v = DY[((size_t)(tx + r + a) * P2_TY + ty) * P2_TZ + tz];
                if (v != INF) nmin = min(nmin, v + a * a);
            }
            if (nmin == INF) {
                res = -dx;
            } else {
                const float vx = grid_pos(G.ox, gx, dx);
                float min_dist = 100000.0f;
                if (enum_end[nmin] == norm_start[nmin + 1]) {
                    /* only norm nmin can attain the minimum: trace the minimisers back through the
                       separable passes (a with a^2 + DY = nmin, then b with b^2 + DZ = DY, then
                       c = +-sqrt(DZ) where the voxel is outside) */
                    for (int a = -r; a <= r; a++) {
                        int dy = DY[((size_t)(tx + r + a) * P2_TY + ty) * P2_TZ + tz];
                        if (dy == INF || dy + a * a != nmin) continue;
                        for (int b = -r; b <= r; b++) {
                            int dz = DZ[((size_t)(tx + r + a) * LY + (ty + r + b)) * P2_TZ + tz];
                            if (dz == INF || dz + b * b != dy) continue;
                            int c = (int)sqrtf((float)dz);
                            uint64_t m = rows[(size_t)(tx + r + a) * LY + (ty + r + b)];
                            const float qx = grid_pos(G.ox, gx + a, dx), qy = grid_pos(G.oy, gy + b, dx);
                            if ((m >> (tz + r + c)) & 1ull)
                                min_dist = fminf(dist3(qx, qy, grid_pos(G.oz, gz + c, dx), vx, vy, vz), min_dist);
                            if (c && ((m >> (tz + r - c)) & 1ull))
                                min_dist = fminf(dist3(qx, qy, grid_pos(G.oz, gz - c, dx), vx, vy, vz), min_dist);
                        }
                    }
                } else {
                    for (int k = norm_start[nmin]; k < enum_end[nmin]; k++) {
                        int o = offs[k];
                        int a = (int)(int8_t)(o & 0xFF), b = (int)(int8_t)((o >> 8) & 0xFF), c = (int)(int8_t)((o >> 16) & 0xFF);
                        uint64_t m = rows[(size_t)(tx + r + a) * LY + (ty + r + b)];
                        if (!((m >> (tz + r + c)) & 1ull)) continue;
                        float d = dist3(grid_pos(G.ox, gx + a, dx), grid_pos(G.oy, gy + b, dx), grid_pos(G.oz, gz + c, dx),
                                        vx, vy, vz);
                        min_dist = fminf(d, min_dist);
                    }
                }
                res = (min_dist < 999.0f) ? (QS_PROBE - min_dist) : -dx;
            }
        }
        if (vyz && shell)
            field[((size_t)gx * g + gy) * g + gz] = res;
        emit_sign_bits(negm, zerom, W, g, gx, gy, tz0, vyz, res);
    }
}

/* squared distance from bit z + R of row m to its nearest set bit within R; z < 32 and 2R < 32,
   so bits z .. z + 2R are the low bits of one 32-bit funnel shift.  Branch free: bits above the
   window are cleared and a sentinel stands at bit 31, so a row with no set bit within R gives a
   distance of at least 31 - R and a square of at least (31 - R)^2 >= 484, above INF = 255 (every
   in-window norm is at most 3R^2 <= 243 for R <= 9); callers clamp it to INF. */
template <int R>
__device__ __forceinline__ uint32_t zdist2(uint64_t m, int z)
{
    static_assert(2 * R < 31 && (31 - R) * (31 - R) > 255, "window wider than a funnel shift");
    const uint32_t w = __builtin_amdgcn_alignbit((uint32_t)(m >> 32), (uint32_t)m, (uint32_t)z); /* bit k = m bit z + k */
    const uint32_t ws = (w & ((1u << (2 * R + 1)) - 1u)) | 0x80000000u;
    const uint32_t up = (uint32_t)__builtin_ctz(ws >> R);               /* nearest set bit at or above the centre */
    const uint32_t dn = (uint32_t)__builtin_clz((ws << (31 - R)) | 1u); /* at or below it (31: none) */
    const uint32_t d = min(up, dn);
    return d * d;
}

/* Field pass 2 for a fixed window half-width R (probeIntersection's second pass,
   Kernels.cu:478-545), one 16 x 8 x 32 tile per block:
   - the tile's own shell and outside bits; a tile without a shell voxel writes its sign words only;
   - the outside rows of the tile and its R halo in LDS;
   - the voxels whose value the mesh can read (QsBand) and the signs of the others, by dilating the
     outside bits 32 voxels at a time; a tile with none of them is done;
   - for those, the exact minimal squared norm n_min by separable minima: z distances from the row
     bits, y minima (with the masks of the attaining y offsets) for the columns they read, x minima;
   - the exact float distance of the minimisers, traced back through the masks (or enumerated
     from a norm-sorted table where another norm could tie), rooted once;
   - the field of those voxels at their grid places, and every voxel's sign bits.
   Bound by VALU issue and, at R = 7, by LDS reads of the dilated rows.  Evaluating every shell
   voxel with an outside voxel in reach (28 to 38 % of the shell; 8 to 15 % are read) by x minima and
   trace took 0.592 ms on the 50,000-atom 0.2 A mesh (R 7), 0.610 on 200,000 atoms at 0.3 A (R 5) and
   0.923 on 100 frames of 10,000 atoms at 0.5 A (R 3); this takes 0.425, 0.382 and 0.555. */

/* entry it of a per-plane bit list: the plane lx with cpre[lx] <= it < cpre[lx + 1] (binary
   search) and the z of the (it - cpre[lx])-th set bit of cmask[lx] */
template <int LX>
__device__ __forceinline__ void list_column(const uint32_t *cpre, const uint32_t *cmask, uint32_t it, int &lx, int &z)
{
    int lo = 0;
#pragma unroll
    for (int step = 32; step >= 1; step >>= 1)
        if (lo + step < LX && cpre[lo + step] <= it) lo += step;
    lx = lo;
    uint32_t w = cmask[lo], k = it - cpre[lo];
    int zz = 0;
#pragma unroll
    for (int h = 16; h >= 1; h >>= 1) {
        const uint32_t c = (uint32_t)__builtin_popcount(w & ((1u << h) - 1u));
        if (k >= c) {
            k -= c;
            w >>= h;
            zz += h;
        }
    }
    z = zz;
}

template <int R>
__global__ void __launch_bounds__(256) k_pass2_r(QsBatch B, const uint64_t *__restrict__ outm_all,
                                                 const uint64_t *__restrict__ shellm_all, float *__restrict__ field_all, uint32_t *__restrict__ negm_all,
                                                 uint32_t *__restrict__ zerom_all, const int *__restrict__ offs,
                                                 const int *__restrict__ norm_start, const int *__restrict__ enum_end,
                                                 QsNormFlags nf, QsBand band, const uint8_t *__restrict__ tflag, uint8_t tmark,
                                                 uint32_t xchunk)
{
    constexpr int LX = P2R_TX + 2 * R, LY = P2_TY + 2 * R, LZ = P2_TZ + 2 * R;
    constexpr int INF = 255;
    static_assert(LZ <= 64 && 3 * R * R < INF, "window too wide for this kernel");
    constexpr int NR = LX * LY;
    __shared__ uint64_t rows[NR];
    /* ownout: the own rows' outside bits, read only by a tile without a shell voxel */
    __shared__ uint32_t own[P2R_TX * P2_TY], ownout[P2R_TX * P2_TY];
    /* y offsets (bit b + R) attaining each DY value */
    using BMask = typename std::conditional<(2 * R + 1 <= 8), uint8_t,
                                            typename std::conditional<(2 * R + 1 <= 16), uint16_t, uint32_t>::type>::type;
    /* first the rows' own 32 voxels dilated by 0 .. R along z (dil[c * NR + row]), then the y minima
       (DY) and their masks (BM) */
    constexpr int NDY = LX * P2_TY * P2_TZ;
    __shared__ uint32_t pool[(R + 1) * NR * 4 > NDY * (1 + (int)sizeof(BMask)) ? (R + 1) * NR : NDY * (1 + (int)sizeof(BMask)) / 4];
    uint32_t *const dil = pool;
    uint8_t *const DY = (uint8_t *)pool;
    BMask *const BM = (BMask *)(pool + NDY / 4);
    /* y-pass work list: per halo x plane lx, the z columns (bit z) that need y minima, and the
       exclusive prefix of their counts (cpre[LX] = total) */
    __shared__ uint32_t shx[P2R_TX], cmask[LX], cpre[LX + 1];
    /* norms whose minimisers are traced back (bit n), from nf */
    __shared__ uint32_t nfw[8];
    /* half-lengths along z of the balls of norms below band.hi (0) and up to band.lo (1) at x and y
       offsets |a|, |b| (255: none) */
    __shared__ uint8_t zlen[2][R + 1][R + 1];
    /* per own (x, y) row of the tile: the voxels whose minimisers are to be traced back, its sign
       words and its zero words */
    __shared__ uint32_t strace[P2R_TX * P2_TY], sneg[P2R_TX * P2_TY], szero[P2R_TX * P2_TY];
    uint32_t lb;
    /* each XCD takes xchunk consecutive tiles at a time (whole rows of z tiles: the y and z halos
       of a tile are then mostly read by tiles of the same XCD, from its L2) */
    const uint32_t bt = xcd_group_rt(blockIdx.x, gridDim.x, xchunk);
    /* a tile without a shell voxel keeps the sign words field pass 1 wrote for it (the launch's
       tile marks are in its block order: an unmarked tile leaves after one load) */
    if (tflag && tflag[bt] != tmark) return;
    const QsMol &M = B.mols[batch_mol(B, bt, lb)];
    const QsGrid G = M.G;
    const int g = G.g, W = (int)M.W;
    const uint64_t *__restrict__ outm = outm_all + M.word_off;
    const uint64_t *__restrict__ shellm = shellm_all + M.word_off;
    float *__restrict__ field = field_all + M.vox_off;
    uint32_t *__restrict__ negm = negm_all + 2 * M.word_off;
    uint32_t *__restrict__ zerom = zerom_all + 2 * M.word_off;
    const int x1 = M.p2_hi;
    const uint32_t nbx = (g + P2_TZ - 1) / P2_TZ, nby = (g + P2_TY - 1) / P2_TY;
    const int tz0 = (int)(lb % nbx) * P2_TZ, ty0 = (int)((lb / nbx) % nby) * P2_TY;
    const int tx0 = M.p2_lo + (int)(lb / (nbx * nby)) * P2R_TX;
    const int ty = threadIdx.x >> 5, tz = threadIdx.x & 31;
    const int gy = ty0 + ty, gz = tz0 + tz;
    const bool vyz = gy < g && gz < g;
    const float dx = G.dx;

    /* the outside rows of the tile and its R halo into LDS; fl: some row has an outside voxel.  A row's
       R + 32 + R bits lie in the 32-bit words before, at and after the tile's, which are one load; a
       row outside the planes [p1_lo, p1_hi), which are all that is stored, reads another one and is
       cleared (no output voxel reads it).  All loads are in flight before the first is used.  (Two
       64-bit words under branches, one row after the other, took 0.440 instead of 0.425 ms on the
       50,000-atom 0.2 A mesh and 0.393 instead of 0.382 on 200,000 atoms at 0.3 A.) */
    int fl = 0;
    auto load_rows = [&]() {
        struct __attribute__((packed, aligned(4))) U3 {
            uint32_t x, y, z;
        };
        constexpr int NL = (LX * LY + 255) / 256;
        const int zw = tz0 >> 5;
        const bool first = zw == 0;
        const uint32_t kc = zw + 1 < 2 * W ? ~0u : 0u;
        const uint32_t *__restrict__ o32 = (const uint32_t *)outm + (first ? 0 : zw - 1);
        U3 w[NL];
        bool ok[NL];
#pragma unroll
        for (int k = 0; k < NL; k++) {
            const int row = min((int)threadIdx.x + 256 * k, LX * LY - 1);
            const int lx = row / LY, ly = row - lx * LY;
            const int gx = tx0 - R + lx, gy_ = ty0 - R + ly;
            ok[k] = gx >= M.p1_lo && gx < M.p1_hi && gy_ >= 0 && gy_ < g;
            w[k] = *(const U3 *)(o32 + (size_t)(ok[k] ? gx * g + gy_ : M.p1_lo * g) * (2 * (size_t)W));
        }
#pragma unroll
        for (int k = 0; k < NL; k++) {
            const int row = (int)threadIdx.x + 256 * k;
            if (row >= LX * LY) break;
            const uint32_t wa = first ? 0u : w[k].x, wb = first ? w[k].x : w[k].y, wc = (first ? w[k].y : w[k].z) & kc;
            const uint32_t kk = ok[k] ? ~0u : 0u;
            const uint32_t lo = __builtin_amdgcn_alignbit(wb, wa, 32 - R) & kk;
            const uint32_t hi = __builtin_amdgcn_alignbit(wc, wb, 32 - R) & kk & ((1u << (LZ - 32)) - 1u);
            rows[row] = (uint64_t)hi << 32 | lo;
            fl |= (lo | hi) != 0u;
            /* bit z of d: an outside voxel within c of z (bit z + R of the row is z) */
            uint32_t d = __builtin_amdgcn_alignbit(hi, lo, R);
            dil[row] = d;
#pragma unroll
            for (int c = 1; c <= R; c++) {
                d |= __builtin_amdgcn_alignbit(hi, lo, R - c) | __builtin_amdgcn_alignbit(hi, lo, R + c);
                dil[c * NR + row] = d;
            }
        }
    };
    /* a tile marked by field pass 1 has a shell voxel: its halo rows are loaded together with its
       own rows, and the first barrier reduces fl */
    const bool marked = tflag != nullptr;

    /* the tile's own shell bits (threads 0-127) and outside bits (threads 128-255) first: an
       unmarked tile without a shell voxel (outside the molecule or deep inside it) is finished
       from them alone, without its halo */
    static_assert(P2R_TX * P2_TY == 128, "one thread per own row of each mask");
    static_assert(P2_TZ == 32, "a tile's z range is one half of a row word");
    if (threadIdx.x < 8) {
        const int t = threadIdx.x;
        const uint64_t w = t < 2 ? nf.w[0] : (t < 4 ? nf.w[1] : (t < 6 ? nf.w[2] : nf.w[3]));
        nfw[t] = (uint32_t)(w >> (32 * (t & 1)));
    }
    if (threadIdx.x < 2 * (R + 1) * (R + 1)) {
        const int set = threadIdx.x / ((R + 1) * (R + 1)), ab = threadIdx.x - set * (R + 1) * (R + 1);
        const int a = ab / (R + 1), b = ab - a * (R + 1);
        const int rem = (set ? band.lo : band.hi - 1) - a * a - b * b; /* c^2 <= rem */
        int c = rem < 0 ? 255 : min((int)__builtin_amdgcn_sqrtf((float)rem + 0.5f), R);
        if (band.all && !set) c = R; /* the whole window */
        zlen[set][a][b] = (uint8_t)c;
    }
    int has_shell;
    {
        const int t = threadIdx.x & 127, tx = t / P2_TY, ty_ = t - tx * P2_TY;
        const int gx = tx0 + tx, gy_ = ty0 + ty_;
        const uint64_t *__restrict__ src = threadIdx.x < 128 ? shellm : outm;
        uint32_t m = 0u;
        if (gx < x1 && gx < g && gy_ < g) {
            /* the tile's 32 z of the row are one half of a row word (tz0 is a multiple of 32) */
            m = (uint32_t)(src[((size_t)gx * g + gy_) * W + (tz0 >> 6)] >> (tz0 & 63));
        }
        /* with band.edge: the row's outside words R + 1 steps away along x and y, and the ones next
           to its own along z (a place outside the grid reads the row's own word and is masked), in
           flight with the halo rows */
        uint32_t ew[7] = {0u, 0u, 0u, 0u, 0u, 0u, 0u}, ek[7] = {0u, 0u, 0u, 0u, 0u, 0u, 0u};
        if (band.edge && threadIdx.x < 128 && gx < x1 && gx < g && gy_ < g) {
            const uint32_t *__restrict__ o32 = (const uint32_t *)outm + ((size_t)gx * g + gy_) * (2 * (size_t)W) + (tz0 >> 5);
            const ptrdiff_t wy = 2 * (ptrdiff_t)W, wx = g * wy;
            const bool k[7] = {true, tz0 > 0, (tz0 >> 5) + 1 < 2 * W, gx - (R + 1) >= M.p1_lo, gx + (R + 1) < M.p1_hi,
                               gy_ - (R + 1) >= 0, gy_ + (R + 1) < g};
            const ptrdiff_t at[7] = {0, -1, 1, -(R + 1) * wx, (R + 1) * wx, -(R + 1) * wy, (R + 1) * wy};
#pragma unroll
            for (int i = 0; i < 7; i++) {
                ew[i] = o32[k[i] ? at[i] : 0];
                ek[i] = k[i] ? ~0u : 0u;
            }
        }
        if (marked) load_rows();
#pragma unroll
        for (int i = 0; i < 7; i++) ew[i] &= ek[i];
        /* the row's voxels with an outside voxel R + 1 steps away along an axis */
        const uint32_t far = (ew[0] << (R + 1) | ew[1] >> (31 - R)) | (ew[0] >> (R + 1) | ew[2] << (31 - R)) | ew[3] | ew[4] | ew[5] | ew[6];
        if (threadIdx.x < 128) {
            strace[t] = szero[t] = 0u;
            sneg[t] = far;
            own[t] = m;
        } else {
            ownout[t] = m;
        }
        /* marked: the tile has a shell voxel, and the barrier tells whether an outside voxel is
           within reach instead */
        has_shell = __syncthreads_or(marked ? fl : (threadIdx.x < 128 && m != 0u));
    }
    if (!marked && !has_shell) {
        /* no field values to store (only shell voxels hold one; the others are the probe radius
           outside and -dx inside): the sign words are the complemented outside bits */
        const uint32_t zvalid = (tz0 + P2_TZ <= g) ? ~0u : ((1u << (g - tz0)) - 1u);
        if (threadIdx.x < P2R_TX * P2_TY) {
            const int tx = threadIdx.x / P2_TY, ty_ = threadIdx.x - tx * P2_TY;
            const int gx = tx0 + tx, gy_ = ty0 + ty_;
            if (gx < x1 && gx < g && gy_ < g) {
                const size_t w32 = ((size_t)gx * g + gy_) * (2 * (size_t)W) + (tz0 >> 5);
                negm[w32] = ~ownout[threadIdx.x] & zvalid;
                zerom[w32] = 0u;
            }
        }
        return;
    }
    /* index of own voxel (tx, ty, tz) in the field */
    auto fidx = [&](int tx, int ty_, int tz_) { return ((size_t)(tx0 + tx) * g + (ty0 + ty_)) * g + (tz0 + tz_); };

    if (!marked) load_rows();
    if (!(marked ? has_shell : __syncthreads_or(fl))) {
        /* no outside voxel within reach: every voxel of the tile is -dx */
        for (int tx = 0; tx < P2R_TX; tx++) {
            int gx = tx0 + tx;
            if (gx >= x1 || gx >= g) break;
            if ((band.all || band.edge) && vyz && ((own[tx * P2_TY + ty] >> tz) & 1u)) field[fidx(tx, ty, tz)] = -dx;
            emit_sign_bits(negm, zerom, W, g, gx, gy, tz0, vyz, -dx);
        }
        return;
    }

    /* Which voxels are near enough to the surface to be read (QsBand), and the signs of the others,
       for 32 voxels of a row at a time: the outside bits dilated by the ball of norms below band.hi
       (strace) and by the one up to band.lo (szero), each clipped to the window.  A ball is a disc of
       (x, y) offsets with a z length each, so a row is the OR of the rows at those offsets, dilated
       along z (dil).  A lane takes two rows, each wave some of the x offsets; offsets x = -a and a
       have the same lengths, which the lanes hold per y offset.  (From the x minima of every shell voxel
       instead, with the y minima of every column a shell voxel reads, this took more than half of
       the kernel at 0.5 A.) */
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    {
        const int r0 = ((lane >> 2) + R) * LY + 2 * (lane & 3); /* + (y offset + R), + x offset * LY */
#pragma unroll 1
        for (int set = 0; set < 2; set++) {
            uint32_t acc0 = 0u, acc1 = 0u;
            /* wave w takes the x offsets w, 7 - w and 8 + w (discs of about the same total width) */
#pragma unroll 1
            for (int i = 0; i < 3; i++) {
                const int a = i == 0 ? wid : (i == 1 ? 7 - wid : 8 + wid);
                if (a > R) continue;
                const int c = lane <= 2 * R ? (int)zlen[set][a][lane < R ? R - lane : lane - R] : 255;
                const int at = c * NR + lane; /* per y offset + R = lane */
                const uint64_t some = __ballot(c != 255); /* y offsets -nb .. nb, or none */
                const int nb = (int)__popcll(some) >> 1;
                if (!some) continue;
                const uint32_t *const pu = dil + r0 + a * LY, *const pv = dil + r0 - a * LY;
#pragma unroll 4
                for (int b = R - nb; b <= R + nb; b++) {
                    const int o = __builtin_amdgcn_readlane(at, b);
                    acc0 |= pu[o] | pv[o];
                    acc1 |= pu[o + 1] | pv[o + 1];
                }
            }
            uint32_t *const acc = set ? szero : strace;
            const int t = (lane >> 2) * P2_TY + 2 * (lane & 3);
            if (acc0) atomicOr(&acc[t], acc0);
            if (acc1) atomicOr(&acc[t + 1], acc1);
        }
    }
    __syncthreads();
    bool any = false;
    if (threadIdx.x < 128) {
        const int t = threadIdx.x, tx = t / P2_TY, ty_ = t - tx * P2_TY;
        const bool in = tx0 + tx < x1 && tx0 + tx < g && ty0 + ty_ < g;
        const uint32_t valid = !in ? 0u : (tz0 + P2_TZ <= g ? ~0u : (1u << (g - tz0)) - 1u);
        const uint32_t hi = strace[t], lo = szero[t], far = sneg[t], sh = own[t] & valid, o = dil[(tx + R) * LY + ty_ + R];
        const uint32_t tr = sh & ((hi & ~lo) | (far & ~hi));
        /* negative: inside, and shell beyond the band (a traced voxel's bits follow from its value) */
        strace[t] = tr;
        sneg[t] = valid & ~o & ~(sh & lo) & ~tr;
        szero[t] = 0u;
        any = tr != 0u;
        if (band.all) /* shell voxels without an outside voxel in the window: -dx */
            for (uint32_t w = sh & ~hi; w; w &= w - 1u) field[fidx(tx, ty_, __builtin_ctz(w))] = -dx;
        /* the traced voxels of each own x plane, over its P2_TY rows (consecutive lanes) */
        uint32_t sx = tr;
#pragma unroll
        for (int k = 1; k < P2_TY; k *= 2) sx |= (uint32_t)__shfl_xor((int)sx, k);
        if (ty_ == 0) shx[tx] = sx;
    }
    if (__syncthreads_or(any)) {
    /* every y minimum starts unreachable; only listed columns are computed */
    for (int i = threadIdx.x; i < NDY / 4; i += 256) pool[i] = 0x01010101u * INF;
    /* the work list: columns needed by a traced voxel with an outside voxel within R of their z
       in some row (else every minimum is INF, as filled) */
    static_assert(LX <= 64, "one lane per halo x plane");
    if (threadIdx.x < 64) {
        const int lx = threadIdx.x;
        uint32_t c = 0;
        if (lx < LX) {
            /* a column (lx, z) is read by the x taps of traced voxels of own planes lx - 2R .. lx */
            uint32_t need = 0;
#pragma unroll
            for (int tx = 0; tx < P2R_TX; tx++)
                if (tx >= lx - 2 * R && tx <= lx) need |= shx[tx];
            uint64_t o = 0;
#pragma unroll
            for (int ly = 0; ly < LY; ly++) o |= rows[lx * LY + ly];
            /* bit z: any of bits z .. z + 2R (bit k of a row is z = k - R) */
            uint64_t near = 0;
#pragma unroll
            for (int k = 0; k <= 2 * R; k++) near |= o >> k;
            c = (uint32_t)near & need;
            cmask[lx] = c;
        }
        const uint32_t cnt = (uint32_t)__builtin_popcount(c);
        const uint32_t inc = wave_incl_scan(cnt);
        if (lx < LX) cpre[lx] = inc - cnt;
        if (lx == LX - 1) cpre[LX] = inc;
    }
    __syncthreads();
    const uint32_t ntodo = cpre[LX];

    /* z then y, one listed (lx, z) column per thread: the squared z distance of each row to its
       nearest outside voxel within R, straight from the row bits, then the y minima over 2R+1 rows */
    if constexpr (2 * R + 1 <= 16) {
        /* two y outputs per 32-bit register (16-bit halves): the tap sums, minima and equality
           masks in packed 16-bit integer arithmetic */
        typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
        /* 2^1, 2^2, 2^4, 2^8 per lane, opaque so that the mask bits stay packed multiply-adds */
        u16x2 pw[4] = {{2, 2}, {4, 4}, {16, 16}, {256, 256}};
#pragma unroll
        for (int i = 0; i < 4; i++) asm volatile("" : "+v"(pw[i]));
        for (uint32_t it = threadIdx.x; it < ntodo; it += 256) {
            int lx, z;
            list_column<LX>(cpre, cmask, it, lx, z);
            uint32_t v[LY];
#pragma unroll
            for (int ly = 0; ly < LY; ly++) v[ly] = zdist2<R>(rows[lx * LY + ly], z);
            u16x2 P[LY - 1];
#pragma unroll
            for (int k = 0; k < LY - 1; k++) P[k] = __builtin_bit_cast(u16x2, v[k] | (v[k + 1] << 16));
#pragma unroll
            for (int yy = 0; yy < P2_TY; yy += 2) {
                /* taps below 2^11 (z squares below 1024 plus 49): no 16-bit lane overflows */
                constexpr int NT = 2 * R + 1;
                u16x2 sb[NT], t[NT];
#pragma unroll
                for (int b = 0; b < NT; b++) {
                    const uint16_t c = (uint16_t)((b - R) * (b - R));
                    sb[b] = P[yy + b] + (u16x2){c, c};
                    t[b] = sb[b];
                }
                /* minimum as a tree (no chain of dependent packed operations) */
#pragma unroll
                for (int s = 1; s < NT; s *= 2)
#pragma unroll
                    for (int b = 0; b + s < NT; b += 2 * s) t[b] = __builtin_elementwise_min(t[b], t[b + s]);
                const u16x2 best = t[0];
                /* tie mask: best + 1 - tap saturates to 1 at a minimum and to 0 elsewhere; the
                   bits are combined as a tree as well, pairs of taps first */
                const u16x2 best1 = best + (u16x2){1, 1};
#pragma unroll
                for (int b = 0; b < NT; b++) t[b] = __builtin_elementwise_sub_sat(best1, sb[b]);
#pragma unroll
                for (int s = 1, l = 0; s < NT; s *= 2, l++)
#pragma unroll
                    for (int b = 0; b + s < NT; b += 2 * s) t[b] = t[b + s] * pw[l] + t[b];
                const u16x2 mm = t[0];
                const uint32_t bb = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(best, (u16x2){(uint16_t)INF, (uint16_t)INF}));
                const uint32_t mw = __builtin_bit_cast(uint32_t, mm);
                DY[(lx * P2_TY + yy) * P2_TZ + z] = (uint8_t)bb;
                DY[(lx * P2_TY + yy + 1) * P2_TZ + z] = (uint8_t)(bb >> 16);
                BM[(lx * P2_TY + yy) * P2_TZ + z] = (BMask)(mw & 0xFFFFu);
                BM[(lx * P2_TY + yy + 1) * P2_TZ + z] = (BMask)(mw >> 16);
            }
        }
    } else
    for (uint32_t it = threadIdx.x; it < ntodo; it += 256) {
        int lx, z;
        list_column<LX>(cpre, cmask, it, lx, z);
        int v[LY];
#pragma unroll
        for (int ly = 0; ly < LY; ly++) v[ly] = (int)zdist2<R>(rows[lx * LY + ly], z);
#pragma unroll
        for (int yy = 0; yy < P2_TY; yy++) {
            int best = INF;
#pragma unroll
            for (int b = 0; b <= 2 * R; b++) best = min(best, v[yy + b] + (b - R) * (b - R));
            uint32_t bm = 0;
#pragma unroll
            for (int b = 0; b <= 2 * R; b++) bm |= (uint32_t)(v[yy + b] + (b - R) * (b - R) == best) << b;
            DY[(lx * P2_TY + yy) * P2_TZ + z] = (uint8_t)best;
            BM[(lx * P2_TY + yy) * P2_TZ + z] = (BMask)bm;
        }
    }
    __syncthreads();

    /* the block's marked voxels, 64 at a time per wave in row order: the x minimum and the offsets
       attaining it, the minimisers traced back through the y masks, and their exact float distance.
       (Traced as soon as a wave had queued 64, from inside an unrolled loop over the x minima, the
       kernel had 16 copies of the trace, 60 KB of code.) */
    auto trace_voxel = [&](int tx, int ty_, int tz_) {
        const int gx = tx0 + tx, gy_ = ty0 + ty_, gz_ = tz0 + tz_;
        /* the x offsets (bit a + R) attaining the minimal norm */
        int nmin = INF;
        uint32_t amask = 0;
        if constexpr (2 * R + 1 <= 16) {
            /* taps a = 2k, 2k + 1 in the 16-bit halves of t[k] (an odd last tap is padded with the
               largest value, which neither lowers the minimum nor equals it); the tie bits are
               taken as in the y pass, then combined by packed multiply-adds: the low halves end up
               holding the even taps' bits at their places, the high halves the odd ones' one place
               lower */
            typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
            constexpr int NT = 2 * R + 1, NP = (NT + 1) / 2;
            u16x2 t[NP];
#pragma unroll
            for (int k = 0; k < NP; k++) {
                const int a0 = 2 * k, a1 = 2 * k + 1;
                const uint32_t lo = DY[((tx + a0) * P2_TY + ty_) * P2_TZ + tz_];
                const uint32_t hi = (a1 < NT) ? (uint32_t)DY[((tx + a1) * P2_TY + ty_) * P2_TZ + tz_] : 0xFFFFu;
                const uint16_t c0 = (uint16_t)((a0 - R) * (a0 - R)), c1 = (a1 < NT) ? (uint16_t)((a1 - R) * (a1 - R)) : (uint16_t)0;
                t[k] = __builtin_bit_cast(u16x2, lo | (hi << 16)) + (u16x2){c0, c1};
            }
            u16x2 m = t[0];
#pragma unroll
            for (int k = 1; k < NP; k++) m = __builtin_elementwise_min(m, t[k]);
            nmin = (int)min(m.x, m.y);
            const u16x2 n1 = (u16x2){(uint16_t)(nmin + 1), (uint16_t)(nmin + 1)};
#pragma unroll
            for (int k = 0; k < NP; k++) t[k] = __builtin_elementwise_sub_sat(n1, t[k]);
            /* 4, 16, 256 per lane, opaque so that the combination stays packed multiply-adds */
            u16x2 pw[3] = {{4, 4}, {16, 16}, {256, 256}};
#pragma unroll
            for (int i = 0; i < 3; i++) asm volatile("" : "+v"(pw[i]));
#pragma unroll
            for (int st = 1, l = 0; st < NP; st *= 2, l++)
#pragma unroll
                for (int k = 0; k + st < NP; k += 2 * st) t[k] = t[k + st] * pw[l] + t[k];
            amask = (uint32_t)t[0].x | ((uint32_t)t[0].y << 1);
        } else {
#pragma unroll
            for (int a = 0; a <= 2 * R; a++) nmin = min(nmin, (int)DY[((tx + a) * P2_TY + ty_) * P2_TZ + tz_] + (a - R) * (a - R));
#pragma unroll
            for (int a = 0; a <= 2 * R; a++)
                amask |= (uint32_t)((int)DY[((tx + a) * P2_TY + ty_) * P2_TZ + tz_] + (a - R) * (a - R) == nmin) << a;
        }
        const float vx = grid_pos(G.ox, gx, dx), vy = grid_pos(G.oy, gy_, dx), vz = grid_pos(G.oz, gz_, dx);
        /* the smallest squared distance, rooted once at the end: sqrtf rounds correctly and is
           monotone, so the root of the minimum is the minimum of the roots */
        float min_sq = __builtin_inff();
        if (nmin >= INF) {
            /* no outside voxel in the window: -dx */
        } else if ((nfw[nmin >> 5] >> (nmin & 31)) & 1u) {
            /* trace the minimisers back through the separable passes: the x offsets, their y offsets
               from the recorded masks, and the nearest outside voxels of those rows along z (one
               loop over the (x, y) offsets, as the lanes' numbers of x and of y offsets differ: an
               outer and an inner one, with a root for the z offset and 64-bit shifts of the row for
               its two ends, took 0.611 instead of 0.581 ms on 100 frames of 10,000 atoms at 0.5 A
               and 0.869 instead of 0.825 on 256 molecules) */
            int at = 0;             /* own voxel (tx + R + a, ty_) as the row of DY and BM */
            uint32_t bmask = 0;
            float ex2 = 0.0f;
            while (amask | bmask) {
                if (!bmask) {
                    const int a = __builtin_ctz(amask);
                    amask &= amask - 1u;
                    at = tx + a;
                    bmask = BM[(at * P2_TY + ty_) * P2_TZ + tz_];
                    ex2 = sq_dist(grid_pos(G.ox, gx + a - R, dx), vx);
                }
                const int b = __builtin_ctz(bmask);
                bmask &= bmask - 1u;
                const uint64_t m = rows[at * LY + ty_ + b];
                const uint32_t w = __builtin_amdgcn_alignbit((uint32_t)(m >> 32), (uint32_t)m, (uint32_t)tz_);
                const int up = __builtin_ctz((w >> R) | 0x80000000u), dn = __builtin_clz((w << (31 - R)) | 1u);
                const int c = min(up, dn);
                const float exy = ex2 + sq_dist(grid_pos(G.oy, gy_ + b - R, dx), vy);
                const float su = exy + sq_dist(grid_pos(G.oz, gz_ + c, dx), vz);
                const float sd = exy + sq_dist(grid_pos(G.oz, gz_ - c, dx), vz);
                min_sq = fminf(min_sq, up <= dn ? su : sd);
                min_sq = fminf(min_sq, dn <= up ? sd : su);
            }
        } else {
#pragma unroll 1
            for (int k = norm_start[nmin]; k < enum_end[nmin]; k++) {
                int o = offs[k];
                int a = (int)(int8_t)(o & 0xFF), b = (int)(int8_t)((o >> 8) & 0xFF), c = (int)(int8_t)((o >> 16) & 0xFF);
                uint64_t m = rows[(tx + R + a) * LY + (ty_ + R + b)];
                if (!((m >> (tz_ + R + c)) & 1ull)) continue;
                float d = dist3_sq(grid_pos(G.ox, gx + a, dx), grid_pos(G.oy, gy_ + b, dx), grid_pos(G.oz, gz_ + c, dx), vx, vy,
                                   vz);
                min_sq = fminf(d, min_sq);
            }
        }
        const float min_dist = sqrt_rn(min_sq);
        const float res = (min_dist < 999.0f) ? (QS_PROBE - min_dist) : -dx;
        field[fidx(tx, ty_, tz_)] = res;
        if (res < 0.0f) atomicOr(&sneg[tx * P2_TY + ty_], 1u << tz_);
        if (res == 0.0f) atomicOr(&szero[tx * P2_TY + ty_], 1u << tz_);
    };
    {
        /* lane l's rows are 2 l and 2 l + 1 */
        const uint32_t m0 = strace[2 * lane], m1 = strace[2 * lane + 1];
        const uint32_t n0 = (uint32_t)__popc(m0), nn = n0 + (uint32_t)__popc(m1);
        uint32_t pre = wave_incl_scan(nn);
        const uint32_t total = wave_last(pre);
        pre -= nn; /* exclusive */
#pragma unroll 1
        for (uint32_t base = 64u * (uint32_t)wid; base < total; base += 256u) {
            const uint32_t j = base + (uint32_t)lane;
            /* the item's pair of rows: the last lane whose first item is at or below j */
            int o = 0;
#pragma unroll
            for (int step = 32; step >= 1; step >>= 1)
                if ((uint32_t)__shfl((int)pre, o + step, 64) <= j) o += step;
            uint32_t r = j - (uint32_t)__shfl((int)pre, o, 64);
            const uint32_t on0 = (uint32_t)__shfl((int)n0, o, 64);
            const uint32_t om0 = (uint32_t)__shfl((int)m0, o, 64), om1 = (uint32_t)__shfl((int)m1, o, 64);
            const bool second = r >= on0;
            r -= second ? on0 : 0u;
            const int row = 2 * o + (second ? 1 : 0);
            if (j < total) trace_voxel(row / P2_TY, row % P2_TY, nth_bit32(second ? om1 : om0, r));
        }
    }
    __syncthreads();
    }
    /* the wave's sign and zero words: lane = x (0-15) | row bit << 4 | zero word << 5 */
    {
        const int tx = lane & 15, ty_ = 2 * wid + ((lane >> 4) & 1);
        const int gx = tx0 + tx, gy_ = ty0 + ty_;
        if (gx < x1 && gx < g && gy_ < g) {
            const size_t w32 = ((size_t)gx * g + gy_) * (2 * (size_t)W) + (tz0 >> 5);
            if (lane < 32) negm[w32] = sneg[tx * P2_TY + ty_];
            else zerom[w32] = szero[tx * P2_TY + ty_];
        }
    }
}

__device__ __forceinline__ bool mask_bit(const uint64_t *__restrict__ m, int g, int W, int x, int y, int z)
{
    return (m[((size_t)x * g + y) * W + (z >> 6)] >> (z & 63)) & 1ull;
}

/* direct (2r+1)^3 window, one thread per voxel: any r; also a cross-check of the tile kernel */
__global__ void __launch_bounds__(256) k_pass2_direct(QsBatch B, const uint64_t *__restrict__ outm_all,
                                                      const uint64_t *__restrict__ shellm_all,
                                                      float *__restrict__ field_all,
                                                      uint32_t *__restrict__ negm_all, uint32_t *__restrict__ zerom_all)
{
    uint32_t lb;
    const QsMol &M = B.mols[batch_mol(B, blockIdx.x, lb)];
    const QsGrid G = M.G;
    const int g = G.g, r = G.r, W = (int)M.W;
    const uint64_t *__restrict__ outm = outm_all + M.word_off;
    const uint64_t *__restrict__ shellm = shellm_all + M.word_off;
    float *__restrict__ field = field_all + M.vox_off;
    uint32_t *__restrict__ negm = negm_all + 2 * M.word_off;
    uint32_t *__restrict__ zerom = zerom_all + 2 * M.word_off;
    const uint32_t nbx = (g + 63) / 64, nby = (g + 3) / 4;
    const int bidx = (int)(lb % nbx);
    int z = bidx * 64 + (threadIdx.x & 63);
    int y = (int)((lb / nbx) % nby) * 4 + (threadIdx.x >> 6);
    int x = M.p2_lo + (int)(lb / (nbx * nby));
    const int x1 = M.p2_hi;
    if (x >= x1 || y >= g) return;
    const bool valid = z < g;
    const float dx = G.dx;
    float res;
    bool shell = false;
    if (!valid || mask_bit(outm, g, W, x, y, z)) {
        res = QS_PROBE;
    } else if (!(shell = mask_bit(shellm, g, W, x, y, z))) {
        res = -dx;
    } else {
        float vx = grid_pos(G.ox, x, dx), vy = grid_pos(G.oy, y, dx), vz = grid_pos(G.oz, z, dx);
        float min_dist = 100000.0f;
        for (int a = -r; a <= r; a++) {
            int qx = iclamp(x + a, 0, g - 1);
            for (int b = -r; b <= r; b++) {
                int qy = iclamp(y + b, 0, g - 1);
                for (int c = -r; c <= r; c++) {
                    int qz = iclamp(z + c, 0, g - 1);
                    if (!mask_bit(outm, g, W, qx, qy, qz)) continue;
                    float d = dist3(grid_pos(G.ox, qx, dx), grid_pos(G.oy, qy, dx), grid_pos(G.oz, qz, dx), vx, vy, vz);
                    min_dist = fminf(d, min_dist);
                }
            }
        }
        res = (min_dist < 999.0f) ? (QS_PROBE - min_dist) : -dx;
    }
    if (shell) field[((size_t)x * g + y) * g + z] = res;
    uint64_t n = __ballot(valid && res < 0.0f), zr = __ballot(valid && res == 0.0f);
    if ((threadIdx.x & 63) == 0) {
        size_t w32 = ((size_t)x * g + y) * (2 * (size_t)W) + 2 * (size_t)bidx;
        negm[w32] = (uint32_t)n;
        negm[w32 + 1] = (uint32_t)(n >> 32);
        zerom[w32] = (uint32_t)zr;
        zerom[w32 + 1] = (uint32_t)(zr >> 32);
    }
}

/* sign and zero bits of a caller-given field (stage-wise entry point) */
__global__ void __launch_bounds__(256) k_field_signs(const float *__restrict__ F, int g, int W, uint32_t *__restrict__ negm,
                                                     uint32_t *__restrict__ zerom)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int w = blockIdx.x, y = blockIdx.y * 4 + wid, x = blockIdx.z;
    if (y >= g) return;
    const int z = w * 64 + lane;
    const float f = (z < g) ? F[((size_t)x * g + y) * g + z] : 1.0f;
    uint64_t n = __ballot(f < 0.0f), zr = __ballot(f == 0.0f);
    if (lane == 0) {
        size_t w32 = ((size_t)x * g + y) * (2 * (size_t)W) + 2 * (size_t)w;
        negm[w32] = (uint32_t)n;
        negm[w32 + 1] = (uint32_t)(n >> 32);
        zerom[w32] = (uint32_t)zr;
        zerom[w32 + 1] = (uint32_t)(zr >> 32);
    }
}

void qs_launch_field_signs(const float *F, int g, int W, uint32_t *negm, uint32_t *zerom, hipStream_t s)
{
    dim3 grid((unsigned)W, (unsigned)((g + 3) / 4), (unsigned)g);
    hipLaunchKernelGGL(k_field_signs, grid, dim3(256), 0, s, F, g, W, negm, zerom);
}

/* labels (u8, 0 outside 1 shell 2 inside) -> masks, for stage-wise entry points */
__global__ void __launch_bounds__(256) k_labels_to_masks(const uint8_t *__restrict__ labels, int g, int W,
                                                         uint64_t *__restrict__ outm, uint64_t *__restrict__ shellm)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int w = blockIdx.x, y = blockIdx.y * 4 + wid, x = blockIdx.z;
    if (y >= g) return;
    int z = w * 64 + lane;
    uint8_t l = (z < g) ? labels[((size_t)x * g + y) * g + z] : 0xFF;
    uint64_t mo = __ballot(l == QS_OUT), ms = __ballot(l == QS_SHELL);
    if (lane == 0) {
        outm[((size_t)x * g + y) * W + w] = mo;
        shellm[((size_t)x * g + y) * W + w] = ms;
    }
}

/* ------------------------------------------------------------------------------------------ */
/* marching cubes with edge-id welding                                                         */
/*
 * Every grid point p owns four vertex slots: the edges from p along +x, +y, +z (slots 0..2) and
 * p itself (slot 3).  An edge carries a vertex when its end points differ in sign (field < 0)
 * and it lies on a polygonised cube; when the non-negative end is exactly zero the vertex is
 * that grid point instead (all such edges then share one vertex).  Vertex ids are the ranks of
 * the occupied slots in (point, slot) order, so they come from one prefix sum and welding is
 * exact.  Triangles follow cube order and the case table's order.
 */

/*
 * Marching cubes on the sign bits of the field.  Field pass 2 writes, per 64-voxel row word,
 * N (field < 0) and Z (field == 0).  For every row word k_mc_count forms with 64-bit logic
 *   the four vertex-slot masks of its points (edge +x, +y, +z with a sign change inside the
 *   emission window and a non-zero non-negative end; the point itself when it is zero and an
 *   incident in-window edge ends negative), and
 *   the mask of polygonised cubes (cube origin in [0, lim)^3, corners not all of one sign),
 * and counts vertices and triangles.  An exclusive scan over row words in linear (x, y, w) order
 * gives each word's first vertex and triangle id; inside a word, a point's vertices come after
 * those of the points below it (popcounts of the slot masks), in slot order x, y, z, point --
 * the (point, slot) order.  Emission and smoothing run only on words that own something.
 */

struct MCView {
    const uint64_t *__restrict__ N;
    const uint64_t *__restrict__ Zm;
    const uint64_t *__restrict__ S4; /* 4 slot masks per row word */
    const uint32_t *__restrict__ vbw; /* first vertex id per row word */
    int g, W, lim;

    __device__ __forceinline__ size_t widx(int x, int y, int z) const { return ((size_t)x * g + y) * W + (z >> 6); }
    __device__ __forceinline__ bool nbit(int x, int y, int z) const { return (N[widx(x, y, z)] >> (z & 63)) & 1ull; }
    __device__ __forceinline__ int cube_index(int x, int y, int z) const
    {
        int ci = (int)nbit(x, y, z);
        ci |= (int)nbit(x + 1, y, z) << 1;
        ci |= (int)nbit(x + 1, y + 1, z) << 2;
        ci |= (int)nbit(x, y + 1, z) << 3;
        ci |= (int)nbit(x, y, z + 1) << 4;
        ci |= (int)nbit(x + 1, y, z + 1) << 5;
        ci |= (int)nbit(x + 1, y + 1, z + 1) << 6;
        ci |= (int)nbit(x, y + 1, z + 1) << 7;
        return ci;
    }
};

/* countVertexPerCell MarchingCubes.cu:571-658 in word form: slot masks and per-word counts */
__global__ void __launch_bounds__(256) k_mc_count(QsBatch B, const uint64_t *__restrict__ N_all,
                                                  const uint64_t *__restrict__ Zm_all, uint64_t *__restrict__ S4_all,
                                                  uint32_t *__restrict__ cnt_all, uint64_t *__restrict__ NT_all,
                                                  uint32_t *__restrict__ sums, uint64_t scan_w0)
{
    uint32_t lb;
    const QsMol &M = B.mols[batch_mol(B, xcd_block(blockIdx.x, gridDim.x), lb)];
    const QsGrid G = M.G;
    const int g = G.g, lim = G.lim, W = (int)M.W;
    const uint64_t *__restrict__ N = N_all + M.word_off;
    const uint64_t *__restrict__ Zm = Zm_all + M.word_off;
    uint64_t *__restrict__ S4 = S4_all + 4 * M.word_off;
    uint32_t *__restrict__ cnt = cnt_all + M.word_off;
    const uint32_t nbx = ((uint32_t)g * W + 255) / 256;
    const int idx = (int)(lb % nbx) * 256 + threadIdx.x;
    const int x = M.mc_lo + (int)(lb / nbx);
    if (x >= M.mc_hi) return; /* whole block */
    uint32_t counts = 0;
    if (idx < g * W) {
    const int y = idx / W, w = idx - y * W;
    const int z0 = w * 64;
    const size_t wi = ((size_t)x * g + y) * W + w;
    const uint64_t valid = bits_below(g, z0);
    const uint64_t wlt = bits_below(lim, z0) & valid;     /* z < lim */
    const uint64_t wle = bits_below(lim + 1, z0) & valid; /* z <= lim */
    const uint64_t zm1 = (w == 0) ? ~1ull : ~0ull;         /* z >= 1 */

    /* the word and its neighbours one step along x, y and w, loaded together without branches: a
       neighbour outside the grid reads the word itself and is masked to zero (the point itself
       is inside the grid).  Bound by the address unit, which takes 16 cycles for a wave's load: the
       neighbours along w come from the neighbour lanes (count and scans of 1M atoms at 0.5 A 144 us
       with thirteen loads, 139 with seven; of 100 frames of 10,000 atoms 176 and 169) */
    const size_t sx = (size_t)g * W;
    const uint64_t *__restrict__ np = N + wi;
    const uint64_t *__restrict__ zp = Zm + wi;
    const bool hx = x + 1 < g, hy = y + 1 < g, hw = w + 1 < W;
    const size_t ox = hx ? sx : 0, oy = hy ? (size_t)W : 0, ow = hw ? 1 : 0;
    const uint64_t mx = hx ? ~0ull : 0ull, my = hy ? ~0ull : 0ull, mw = hw ? ~0ull : 0ull;
    const uint64_t n00 = np[0], z00 = zp[0];
    const uint64_t n10 = np[ox] & mx, z10 = zp[ox] & mx;
    const uint64_t n01 = np[oy] & my, z01 = zp[oy] & my;
    /* the cube's far x, y corner, and the next words of its top corners: the next lane's words, but
       for lane 63 */
    const uint64_t n11 = np[ox + oy] & mx & my;
    uint64_t e00 = 0, ez00 = 0, e10 = 0, e01 = 0, e11 = 0, d00 = 0;
    if ((threadIdx.x & 63) == 63) {
        e00 = np[ow];
        ez00 = zp[ow];
        e10 = np[ox + ow] & mx;
        e01 = np[oy + ow] & my;
        e11 = np[ox + oy + ow] & mx & my;
    }
    if ((threadIdx.x & 63) == 0) d00 = np[w > 0 ? -1 : 0];
    const uint64_t n00p = lane_above(n00, e00) & mw, z00p = lane_above(z00, ez00) & mw, n10p = lane_above(n10, e10) & mw;
    const uint64_t n01p = lane_above(n01, e01) & mw, n11p = lane_above(n11, e11) & mw;
    const uint64_t n00m = lane_below(n00, d00) & (w > 0 ? ~0ull : 0ull);
    const uint64_t n00_up = (n00 >> 1) | (n00p << 63); /* bit z = N[z+1] */
    const uint64_t n00_dn = (n00 << 1) | (n00m >> 63); /* bit z = N[z-1] */
    const uint64_t z00_up = (z00 >> 1) | (z00p << 63);

    /* edge masks under condition masks rather than branches (a branch would take its word's
       load with it and wait on it alone) */
    const uint64_t kx = (x + 1 < g && x < lim && y <= lim) ? ~0ull : 0ull;
    const uint64_t ky = (y + 1 < g && x <= lim && y < lim) ? ~0ull : 0ull;
    const uint64_t kz = (x <= lim && y <= lim) ? ~0ull : 0ull;
    const uint64_t ex = (n00 ^ n10) & ~((n00 & z10) | (~n00 & z00)) & wle & kx;
    const uint64_t ey = (n00 ^ n01) & ~((n00 & z01) | (~n00 & z00)) & wle & ky;
    const uint64_t ez = (n00 ^ n00_up) & ~((n00 & z00_up) | (~n00 & z00)) & wlt & kz;
    uint64_t pt = 0;
    if (z00) {
        uint64_t nb = 0;
        if (x + 1 < g && x < lim && y <= lim) nb |= n10 & wle;
        if (x >= 1 && x - 1 < lim && y <= lim) nb |= *(np - sx) & wle;
        if (y + 1 < g && x <= lim && y < lim) nb |= n01 & wle;
        if (y >= 1 && x <= lim && y - 1 < lim) nb |= *(np - W) & wle;
        if (x <= lim && y <= lim) nb |= (n00_up & wlt) | (n00_dn & zm1 & wle);
        pt = z00 & nb;
    }
    uint32_t nv = (uint32_t)(__popcll(ex) + __popcll(ey) + __popcll(ez) + __popcll(pt));
    /* slot masks are read only for the words that hold vertices */
    if (nv) {
        S4[4 * wi + 0] = ex;
        S4[4 * wi + 1] = ey;
        S4[4 * wi + 2] = ez;
        S4[4 * wi + 3] = pt;
    }
    uint32_t nt = 0, nc = 0;
    if (x < lim && x < M.cube_hi && y < lim) {
        const uint64_t c0 = n00, c1 = n10, c2 = n11, c3 = n01;
        const uint64_t c4 = n00_up;
        const uint64_t c5 = (n10 >> 1) | (n10p << 63);
        const uint64_t c6 = (n11 >> 1) | (n11p << 63);
        const uint64_t c7 = (n01 >> 1) | (n01p << 63);
        const uint64_t all = c0 & c1 & c2 & c3 & c4 & c5 & c6 & c7;
        const uint64_t any = c0 | c1 | c2 | c3 | c4 | c5 | c6 | c7;
        const uint64_t act = any & ~all & wlt;
        /* triangles per cube as three bit planes (counts < 8), for the word's 64 cubes at once.
           For a cube with negative corners S (neither none nor all), the table's count is
           |S| - 2 f - 4 h: f is the number of faces whose four corners are in S, and h marks the
           cases whose two corners outside S are opposite ends of a body diagonal.  (The table
           gives k - 2 triangles per component of S with k cut edges; the cut edges number
           3 |S| - 2 e(S) for e(S) edges inside S, and the components |S| - e(S) + f, except for
           the ring of six corners around a body diagonal: one component, which the table
           triangulates as two, one triangle at each corner outside S.)  Checked against every
           case of the table. */
        const auto fadd = [](uint64_t a, uint64_t b, uint64_t c, uint64_t &carry) {
            const uint64_t ab = a ^ b;
            carry = (a & b) | (c & ab);
            return ab ^ c;
        };
        uint64_t a1, b1, e1, t1;
        const uint64_t a0 = fadd(c0, c1, c2, a1), b0 = fadd(c3, c4, c5, b1);
        const uint64_t d0 = c6 ^ c7, d1 = c6 & c7;
        const uint64_t s0 = fadd(a0, b0, d0, e1);    /* |S| bit 0 */
        const uint64_t t0 = fadd(a1, b1, d1, t1);    /* weight-2 sum of the carries */
        const uint64_t s1 = t0 ^ e1, s2 = t1 ^ (t0 & e1); /* |S| bits 1 and 2 (bit 3: all set) */
        const uint64_t fz0 = c0 & c1 & c2 & c3, fz1 = c4 & c5 & c6 & c7, fy0 = c0 & c1 & c4 & c5;
        const uint64_t fy1 = c2 & c3 & c6 & c7, fx0 = c0 & c3 & c4 & c7, fx1 = c1 & c2 & c5 & c6;
        uint64_t x1, y1;
        const uint64_t x0 = fadd(fz0, fz1, fy0, x1), y0 = fadd(fy1, fx0, fx1, y1);
        const uint64_t f0 = x0 ^ y0, f1 = x1 ^ y1 ^ (x0 & y0); /* f mod 4 (f <= 3 unless all set) */
        /* |S| = 6 with no full face: the two corners outside S are a body diagonal */
        const uint64_t h = ~s0 & s1 & s2 & ~(fz0 | fz1 | fy0 | fy1 | fx0 | fx1);
        /* k = |S| - 2 f - 4 h mod 8, bit by bit */
        const uint64_t p0 = s0 & act, p1 = (s1 ^ f0) & act, p2 = (s2 ^ f1 ^ (~s1 & f0) ^ h) & act;
        nt = (uint32_t)(__popcll(p0) + 2 * __popcll(p1) + 4 * __popcll(p2));
        nc = (uint32_t)__popcll(p0 | p1 | p2);
        if (nt) {
            uint64_t *__restrict__ NT = NT_all + 3 * (M.word_off + wi);
            NT[0] = p0;
            NT[1] = p1;
            NT[2] = p2;
        }
    }
    counts = word_counts(nv, nt, nc);
    cnt[wi] = counts;
    }
    /* The block's counts go to the sums of their scan tiles: one tile, or two where the block crosses a
       boundary (then wave by wave).  A launch that reads all counts again for that took 21 us on the
       50,000-atom 0.2 A mesh and 30 on 256 molecules at 0.5 A; four adds per wave took 10 and 27 more
       than it. */
    __shared__ unsigned long long part[4][2];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint64_t s0 = M.word_off + (uint64_t)x * g * W - scan_w0;
    const uint32_t b0 = (lb % nbx) * 256u, tile = (uint32_t)((s0 + (uint32_t)idx) / SCAN_TILE);
    const uint32_t t0 = (uint32_t)((s0 + b0) / SCAN_TILE), t1 = (uint32_t)((s0 + min(b0 + 255u, (uint32_t)(g * W) - 1u)) / SCAN_TILE);
    for (uint32_t t = t0; t <= t1; t++) {
        const uint32_t c = tile == t ? counts : 0u;
        const uint32_t na = (uint32_t)__popcll(__ballot(c != 0u));
        unsigned long long p0 = 0ull, p1 = 0ull;
        if (na) {
            /* (at most 64 x 256 vertices, 64 x 320 triangles, 64 x 64 cubes) */
            const uint32_t vt = wave_last(wave_incl_scan(word_verts(c) | word_tris(c) << 16));
            p0 = (unsigned long long)(vt >> 16) | (unsigned long long)(vt & 0xFFFFu) << 32;
            p1 = (unsigned long long)na | (unsigned long long)wave_last(wave_incl_scan(word_cubes(c))) << 32;
        }
        if (lane < 2) part[wid][lane] = lane ? p1 : p0;
        __syncthreads();
        if (threadIdx.x < 2) {
            const unsigned long long p = part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
            if (p) atomicAdd((unsigned long long *)sums + 2 * (size_t)t + lane, p);
        }
        __syncthreads(); /* part is written again for the next tile */
    }
}

/* row word wi of a grid -> (x, y, word) */
__device__ __forceinline__ void decode_word(uint32_t wi, int g, int W, int &x, int &y, int &w)
{
    const int row = (int)(wi / (uint32_t)W);
    w = (int)(wi - (uint32_t)row * W);
    x = row / g;
    y = row - x * g;
}

/* last index k in [lo, hi] with a[k] <= v, given a[lo] <= v; a non-decreasing */
__device__ __forceinline__ uint32_t last_le(const uint32_t *__restrict__ a, uint32_t lo, uint32_t hi, uint32_t v)
{
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (a[mid] <= v) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

/* first active word of every 256-item block of a launch over items [0, n): active word k holds
   items [base[k], base[k + 1]) (the last one up to n), so block b starts in the word whose range
   holds item 256 b.  Words may hold items beyond n (a slab's scan counts the vertices of the next
   slab's first plane, which that slab emits): blocks stop at n.  One launch serves the vertex
   launch (blockIdx.y 0) and the triangle launch (1), whose items are cubes. */
struct QsStarts {
    const uint32_t *base; /* first item of each active word */
    uint32_t n;           /* items the launch covers */
    const uint32_t *d_n;  /* the item count on the device (within n), or null */
    uint32_t *start;      /* first active word of each 256-item block */
    uint32_t *zero;       /* nzero counters the item kernel adds to, cleared here */
    uint32_t nzero;
};

__global__ void __launch_bounds__(256) k_block_starts(QsStarts sv, QsStarts st, uint32_t nact,
                                                      const uint32_t *__restrict__ d_nact)
{
    const QsStarts A = blockIdx.y ? st : sv;
    /* counts on the device (when given) within the launch's bounds nact, n */
    if (d_nact) nact = min(*d_nact, nact);
    uint32_t n = A.n;
    if (A.d_n) n = min(*A.d_n, n);
    const uint32_t k0 = blockIdx.x * 256u + threadIdx.x;
    for (uint32_t i = k0; i < A.nzero; i += gridDim.x * 256u) A.zero[i] = 0u;
    for (uint32_t k = k0; k < nact; k += gridDim.x * 256u) {
        const uint32_t b0 = (A.base[k] + 255u) >> 8;
        const uint32_t e = (k + 1 < nact) ? min(A.base[k + 1], n) : n;
        for (uint32_t b = b0; (b << 8) < e; b++) A.start[b] = k;
    }
}

/* The active words that hold a block's items, staged in LDS: their first items and word
   indices, and the block's molecule when one molecule holds them all (else -1). */
struct ItemWords {
    uint32_t k0, nk;
    int mol;
    uint32_t base[257], word[257];
};

__device__ __forceinline__ void stage_item_words(ItemWords &S, const uint32_t *__restrict__ base,
                                                 const uint32_t *__restrict__ list, const uint32_t *__restrict__ start,
                                                 uint32_t nact, uint32_t nblocks, uint32_t blk, const uint64_t *__restrict__ wpre,
                                                 const uint32_t *__restrict__ wcoarse)
{
    const uint32_t k0 = start[blk];
    const uint32_t k1 = (blk + 1 < nblocks) ? start[blk + 1] : nact - 1u;
    const uint32_t nk = k1 - k0 + 1u;
    if (threadIdx.x == 0) {
        S.k0 = k0;
        S.nk = nk;
        S.mol = 0;
        if (wcoarse) { /* (nullptr: one molecule) */
            const int m0 = seg_coarse<QS_COARSE_ITEMS>(wpre, wcoarse, (uint64_t)list[k0]);
            const int m1 = seg_coarse<QS_COARSE_ITEMS>(wpre, wcoarse, (uint64_t)list[k1]);
            S.mol = (m0 == m1) ? m0 : -1;
        }
    }
    if (nk <= 257u)
        for (uint32_t t = threadIdx.x; t < nk; t += 256) {
            S.base[t] = base[k0 + t];
            S.word[t] = list[k0 + t];
        }
    __syncthreads();
}

/* active word (index into the active list, and its row word) of item i of the block */
__device__ __forceinline__ void item_word(const ItemWords &S, const uint32_t *__restrict__ base,
                                          const uint32_t *__restrict__ list, uint32_t i, uint32_t &k, uint32_t &wi,
                                          uint32_t &first)
{
    uint32_t lo = 0, hi = min(S.nk, 257u) - 1u;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (S.base[mid] <= i) lo = mid;
        else hi = mid - 1;
    }
    k = S.k0 + lo;
    wi = S.word[lo];
    first = S.base[lo];
    /* (opaque, so that these stay LDS reads: merged with the loads below they become flat loads) */
    asm volatile("" : "+v"(wi), "+v"(first));
    if (S.nk > 257u) { /* not staged */
        k = last_le(base, S.k0, S.k0 + S.nk - 1u, i);
        wi = list[k];
        first = base[k];
    }
}

/* Field value of voxel z of grid row `row` (= x * g + y).  Field pass 2 stores shell voxels only (of
   them those that its QsBand keeps: callers read no others), at their grid places; every other voxel is the probe radius outside and -dx inside, read from the
   outside and shell masks (W words per row), which are loaded together with the place.  shellm ==
   nullptr: F holds every voxel. */
__device__ __forceinline__ float field_at(const float *__restrict__ F, const uint64_t *__restrict__ outm,
                                          const uint64_t *__restrict__ shellm, size_t row, int g, int W, int z, float dx)
{
    const float f = F[row * g + z];
    if (!shellm) return f;
    const size_t wi = row * W + (z >> 6);
    const uint64_t sh = shellm[wi], ou = outm[wi];
    const int b = z & 63;
    return ((sh >> b) & 1ull) ? f : (((ou >> b) & 1ull) ? QS_PROBE : -dx);
}

/* every voxel of one molecule's field in grid order (out) from the stored shell values (F) and the
   masks: a wave per mask word, a lane per voxel */
__global__ void __launch_bounds__(256) k_field_expand(const float *__restrict__ F, const uint64_t *__restrict__ outm,
                                                      const uint64_t *__restrict__ shellm, float *__restrict__ out, int g, int W,
                                                      float dx)
{
    const size_t wi = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wi >= (size_t)g * g * W) return;
    const size_t row = wi / W;
    const int b = threadIdx.x & 63, z = (int)(wi - row * W) * 64 + b;
    if (z >= g) return;
    const bool sh = (shellm[wi] >> b) & 1ull, o = (outm[wi] >> b) & 1ull;
    out[row * g + z] = sh ? F[row * g + z] : (o ? QS_PROBE : -dx);
}

void qs_launch_field_expand(const float *F, const uint64_t *outm, const uint64_t *shellm, float *out, int g, int W, float dx,
                            hipStream_t s)
{
    const size_t n = (size_t)g * g * W;
    if (!n) return;
    k_field_expand<<<(unsigned)((n + 3) / 4), 256, 0, s>>>(F, outm, shellm, out, g, W, dx);
}

/* ------------------------------------------------------------------------------------------ */
/* closest atom per vertex (computeClosestAtom Kernels.cu:547-604)                              */
/* The reference visits the 27 clamped cells x-major, z fastest, and keeps the first atom whose
   rounded distance is strictly below the best so far.  The three z cells of an (x, y) column are
   consecutive cells, so their atoms are one contiguous range in that same order; a cell the clamp
   visits twice cannot improve on its first visit. */

/* The walk as the reference's, with a root for every atom whose squared sum is below the best
   one's (sqrtf is monotone: no other can win): for the vertices closest_one cannot decide. */
__device__ __noinline__ int closest_walk(const float4 *__restrict__ sx, const uint32_t *__restrict__ cstart, int gn, int cx, int cy,
                                         int cz, float px, float py, float pz)
{
    const int z0 = iclamp(cz - 1, 0, gn - 1), z1 = iclamp(cz + 1, 0, gn - 1);
    int best = -1;
    float min_d = 999999.0f, min_s = INFINITY;
    for (int k = 0; k < 9; k++) {
        const int ix = iclamp(cx + k / 3 - 1, 0, gn - 1), iy = iclamp(cy + k % 3 - 1, 0, gn - 1);
        const int h = (gn * gn * ix) + (gn * iy);
        const int hi = (int)cstart[h + z1 + 1];
        for (int id = (int)cstart[h + z0]; id < hi; id++) {
            const float4 at = sx[id];
            const float sq = dist3_sq(at.x, at.y, at.z, px, py, pz);
            if (sq < min_s) {
                const float d = sqrt_rn(sq);
                if (d < min_d) {
                    min_d = d;
                    min_s = sq;
                    best = id;
                }
            }
        }
    }
    return best;
}

/* One axis of a vertex's 3 x 3 x 3 cells: its own cell o, and the squared distance that an atom of
   the cell below (o - 1) or above (o + 1) is away at least (infinite where the clamp leaves none).
   A cell's atoms lie beyond its boundary up to the rounding of cell_of, which margin covers. */
struct AxisCells {
    int o;
    float dn2, up2;
    __device__ __forceinline__ bool near_dn() const { return dn2 < up2; }
    __device__ __forceinline__ int nr() const { return near_dn() ? o - 1 : o + 1; }
    __device__ __forceinline__ int fr() const { return near_dn() ? o + 1 : o - 1; }
    __device__ __forceinline__ float nr2() const { return fminf(dn2, up2); }
    __device__ __forceinline__ float fr2() const { return fmaxf(dn2, up2); }
};
__device__ __forceinline__ AxisCells axis_cells(float p, float org, float dxn, int gn, float margin)
{
    AxisCells A;
    /* (clamped to one cell off the grid, where the reference's three clamped cells are the same as
       further off: the neighbours' indexes hold for any p) */
    const int c = iclamp(cell_of(p, org, dxn), -1, gn);
    const float f = p - org;
    A.o = iclamp(c, 0, gn - 1);
    const float dn = fmaxf(f - (float)A.o * dxn - margin, 0.0f), up = fmaxf((float)(A.o + 1) * dxn - f - margin, 0.0f);
    A.dn2 = iclamp(c - 1, 0, gn - 1) == A.o ? INFINITY : dn * dn;
    A.up2 = iclamp(c + 1, 0, gn - 1) == A.o ? INFINITY : up * up;
    return A;
}

/* A column's three z cells around z cell o as places in the cell-sorted atoms: below [a, b), own
   [b, c), above [c, d), read in one load (past the column's ends they hold its neighbours' places,
   past the last cell the padding of the array: callers use those of cells that exist only) */
struct ColumnStarts {
    int a, b, c, d;
};
__device__ __forceinline__ ColumnStarts column_starts(const uint32_t *__restrict__ cstart, int h, int o)
{
    struct __attribute__((packed, aligned(4))) U4 {
        int x, y, z, w;
    };
    const U4 e = *(const U4 *)(cstart + (h + max(o - 1, 0)));
    ColumnStarts C;
    C.a = e.x;
    C.b = o ? e.y : e.x;
    C.c = o ? e.z : e.y;
    C.d = o ? e.w : e.z;
    return C;
}

/* closest atom of vertex v (position p) of molecule M, relative to its first atom (-1: none).
   Bound by the L1's lookups: a lane's gather of an atom or of a column's places takes one each,
   nearly independent of its width.  So the eight cells of the vertex's octant (its own and the nearer
   neighbour on each axis) come first, and of the other 19 only those are visited whose boundary is
   not further than the best atom so far: 9 atoms per vertex instead of 24, 33 iterations per wave
   instead of 47 (most vertices need none of the 19, as the closest atom is about 1.9 A away and the
   far cells at least 1.6); and a column's places are one load.  All 27 cells, two loads per column,
   took 0.185 ms on the 50,000-atom 0.2 A mesh and 0.907 ms on 256 molecules at 0.5 A; this takes
   0.126 and 0.716 (0.134 and 0.756 with two loads per column; the far columns walked from a mask of
   those to visit, their places loaded when it is their turn, 0.143 and 0.777).
   A loop that roots every improving candidate pays for the root on almost every iteration, so the
   loop keeps the smallest squared sum, its atom and the second smallest sum, with no branch.
   Rounded roots of two sums can only be equal when the sums agree to 2^-22, so unless the two
   smallest agree to 1e-6 the atom of the smallest one is the reference's, whatever the order of the
   visit (a cell is left out only if its atoms' sums are 1e-4 above); else the vertex is walked
   again in the reference's order with the roots. */
__device__ __forceinline__ int closest_one(const QsMol &M, float px, float py, float pz, const uint32_t *__restrict__ cstart_all,
                                           const float4 *__restrict__ sx, const int *__restrict__ perm, int sorted_ids)
{
    const QsGrid G = M.G;
    const uint32_t *__restrict__ cstart = cstart_all + M.cell_off;
    const int gn = G.gn;
    const float margin = (float)(gn + 1) * G.dxn * 1e-6f; /* 8 roundings at the grid's extent */
    const AxisCells X = axis_cells(px, G.ox, G.dxn, gn, margin), Y = axis_cells(py, G.oy, G.dxn, gn, margin),
                    Z = axis_cells(pz, G.oz, G.dxn, gn, margin);
    int best = -1;
    float min_s = INFINITY, next_s = INFINITY;
    const auto walk = [&](int lo, int hi) {
        for (int id = lo; id < hi; id++) {
            const float4 at = sx[id];
            const float sq = dist3_sq(at.x, at.y, at.z, px, py, pz);
            next_s = __builtin_amdgcn_fmed3f(sq, min_s, next_s); /* second smallest: min_s <= next_s */
            best = (sq < min_s) ? id : best;
            min_s = (sq < min_s) ? sq : min_s;
        }
    };
    const auto column = [&](int ix, int iy) { return (gn * gn * ix) + (gn * iy); };
    const bool zdn = Z.near_dn();
    const float xn2 = X.nr2(), xf2 = X.fr2(), yn2 = Y.nr2(), yf2 = Y.fr2(), zf2 = Z.fr2();
    const bool xn = xn2 < INFINITY, yn = yn2 < INFINITY, zn = Z.nr2() < INFINITY;
    const int xnr = xn ? X.nr() : X.o, ynr = yn ? Y.nr() : Y.o;
    /* the octant's four columns: own and near z cell; the far z cell's range is kept for later */
    int flo[4], fhi[4];
    {
        int lo[4], hi[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const ColumnStarts C = column_starts(cstart, column(k & 1 ? xnr : X.o, k & 2 ? ynr : Y.o), Z.o);
            const bool is = (!(k & 1) || xn) && (!(k & 2) || yn);
            lo[k] = zn && zdn ? C.a : C.b;
            hi[k] = is ? (zn && !zdn ? C.d : C.c) : 0;
            flo[k] = zdn ? C.c : C.a;
            fhi[k] = zdn ? C.d : C.b;
        }
#pragma unroll
        for (int k = 0; k < 4; k++) walk(lo[k], hi[k]);
    }
    {
        /* the far cells in reach */
        const float lim = fminf(min_s * 1.0001f, 3.0e38f);
        const float near2[4] = {0.0f, xn2, yn2, xn2 + yn2};
        const float far2[5] = {xf2, xf2 + yn2, yf2, xn2 + yf2, xf2 + yf2};
        const int ix[5] = {X.fr(), X.fr(), X.o, xnr, X.fr()}, iy[5] = {Y.o, ynr, Y.fr(), Y.fr(), Y.fr()};
        int lo[5], hi[5];
#pragma unroll
        for (int k = 0; k < 5; k++) {
            lo[k] = hi[k] = 0;
            if (far2[k] <= lim) {
                const ColumnStarts C = column_starts(cstart, column(ix[k], iy[k]), Z.o);
                lo[k] = far2[k] + Z.dn2 <= lim ? C.a : C.b;
                hi[k] = far2[k] + Z.up2 <= lim ? C.d : C.c;
            }
        }
#pragma unroll
        for (int k = 0; k < 4; k++) walk(flo[k], near2[k] + zf2 <= lim ? fhi[k] : 0);
#pragma unroll
        for (int k = 0; k < 5; k++) walk(lo[k], hi[k]);
    }
    if (!(next_s > min_s * 1.000001f) && best >= 0)
        best = closest_walk(sx, cstart, gn, cell_of(px, G.ox, G.dxn), cell_of(py, G.oy, G.dxn), cell_of(pz, G.oz, G.dxn), px, py, pz);
    /* atom indices are returned relative to the molecule's first atom */
    return (best < 0) ? -1 : ((sorted_ids ? best : perm[best]) - (int)M.atom_off);
}

__global__ void __launch_bounds__(256) k_closest_atom(const QsMol *__restrict__ mols, const uint32_t *__restrict__ vpre,
                                                      const uint32_t *__restrict__ vcoarse, const float *__restrict__ vert,
                                                      uint32_t nv, const uint32_t *__restrict__ d_nv, QsClosest A)
{
    if (d_nv) nv = min(*d_nv, nv); /* the device count within the launch's pool */
    const uint32_t nb = (nv + 255u) >> 8;
    /* persistent blocks over the 256-vertex blocks (on XCDs as in k_mc_emit) */
    for (uint32_t vb = blockIdx.x; vb < nb; vb += gridDim.x) {
        const uint32_t v = xcd_group<64>(vb, nb) * 256u + threadIdx.x;
        if (v >= nv) continue;
        const QsMol &M = mols[seg_of_wave(vpre, vcoarse, v)];
        A.atom[v] = closest_one(M, vert[3 * (size_t)v], vert[3 * (size_t)v + 1], vert[3 * (size_t)v + 2], A.cstart, A.sx, A.perm,
                                A.sorted_ids);
    }
}

/* ------------------------------------------------------------------------------------------ */
/* vertices (vertexInterp/lerp MarchingCubes.cu:715-734, edge oriented low->high), one thread per
   vertex: its word from the active words' first vertex ids, its point and slot from the word's
   four slot masks (vertex ids run over the word's points in z order, slots x, y, z, point).
   ATOMS: the vertex's closest atom in the same pass (A). */
/* triangles (generateTriangleVerticesSMEM MarchingCubes.cu:736-851 order), one thread per
   polygonised cube (two triangles on average): its word from the active words' first cubes, its
   place from the word's triangle-count planes.  Bound by the dependent memory trips of a block
   (block start, word list, planes, corner masks) and by VALU issue, so both are paid once per cube:
   the thread loads the sign words, slot masks and vertex counts of the cube's four (x, y) columns
   together, and every corner's vertex id comes from them.  One thread per triangle, three corners'
   masks each, took 0.20 ms on the 50,000-atom 0.2 A mesh and 0.92 ms on 256 molecules at 0.5 A
   (47 M triangles); this takes 0.14 and 0.56 ms.  (64 registers for eight waves per SIMD, with
   spills, were slower than 66 with seven: emission 1.11 against 1.06 ms.) */
/* The two are launches of their own (VERT or TRI) or, for a small mesh, whose time is that of the
   launches in turn, one launch whose first nbv blocks are the vertices': 7 us of 25 less on 2,000
   atoms at 0.5 A. */
template <bool VERT, bool TRI, bool ATOMS>
__global__ void __launch_bounds__(256) k_mc_emit(const QsMol *__restrict__ mols, const uint64_t *__restrict__ wpre,
                                                 const uint32_t *__restrict__ wcoarse, const uint32_t *__restrict__ list,
                                                 const uint32_t *__restrict__ avb, const uint32_t *__restrict__ vstart,
                                                 uint32_t nact, uint32_t nv, const uint64_t *__restrict__ S4_all,
                                                 const float *__restrict__ F_all, const uint64_t *__restrict__ outm_all,
                                                 const uint64_t *__restrict__ shellm_all, float *__restrict__ vert,
                                                 uint64_t *__restrict__ vkey, const uint32_t *__restrict__ d_counts,
                                                 const uint32_t *__restrict__ acb, const uint32_t *__restrict__ tstart,
                                                 uint32_t ncube, uint32_t ntri, const uint64_t *__restrict__ N,
                                                 const uint32_t *__restrict__ cnt, const uint32_t *__restrict__ vbw,
                                                 const uint32_t *__restrict__ tbw, const uint64_t *__restrict__ NT,
                                                 int *__restrict__ tri, uint32_t vbase, uint32_t *__restrict__ deg_blk,
                                                 uint32_t *__restrict__ deg_total, QsClosest A, uint32_t nbv)
{
    __shared__ ItemWords S;
    if constexpr (VERT) {
    if (!TRI || blockIdx.x < nbv) {
    /* with d_counts (triangles, vertices, active words) the counts come from the device, the
       launch covering the pool of nv vertices: blocks past the count leave at once */
    if (d_counts) {
        nact = d_counts[2];
        nv = min(d_counts[1], nv);
    }
    const uint32_t nb = (nv + 255u) >> 8;
    /* persistent blocks over the 256-vertex blocks: block vb runs on XCD vb % 8 and the renumbering keeps
       neighbouring rows' words on one L2, but not in a block's later turns, whose XCD is the grid's
       remainder by 8 away (nor the cubes' blocks behind nbv of vertices).  Grids rounded to a multiple of 8
       took the same time: 2 M separate spheres' vertices at 1.0 A, in 8 turns, 322 and 325 us in all. */
    for (uint32_t vb = blockIdx.x; vb < nb; vb += VERT && TRI ? nbv : gridDim.x) {
    const uint32_t blk = xcd_group<64>(vb, nb);
    stage_item_words(S, avb, list, vstart, nact, nb, blk, wpre, wcoarse);
    const uint32_t v = blk * 256u + threadIdx.x;
    if (v < nv) {
    uint32_t k, wi, first;
    item_word(S, avb, list, v, k, wi, first);
    const uint32_t local = v - first;
    const QsMol &M = mols[S.mol >= 0 ? S.mol : seg_coarse<QS_COARSE_ITEMS>(wpre, wcoarse, (uint64_t)wi)];
    const QsGrid G = M.G;
    const int g = G.g;
    int x, y, w;
    decode_word((uint32_t)(wi - M.word_off), g, (int)M.W, x, y, w);
    const uint64_t *__restrict__ m = S4_all + 4 * (size_t)wi;
    const uint64_t m0 = m[0], m1 = m[1], m2 = m[2], m3 = m[3];
    /* the point: smallest b whose slots below b + 1 exceed local */
    int lo = 0, hi = 63;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        const uint64_t below = (2ull << mid) - 1ull;
        const uint32_t c = (uint32_t)(__popcll(m0 & below) + __popcll(m1 & below) + __popcll(m2 & below) + __popcll(m3 & below));
        if (c > local) hi = mid;
        else lo = mid + 1;
    }
    const int b = lo;
    const uint64_t below = (1ull << b) - 1ull;
    uint32_t r = local - (uint32_t)(__popcll(m0 & below) + __popcll(m1 & below) + __popcll(m2 & below) + __popcll(m3 & below));
    const uint32_t bits = (uint32_t)((m0 >> b) & 1ull) | (uint32_t)((m1 >> b) & 1ull) << 1 |
                          (uint32_t)((m2 >> b) & 1ull) << 2 | (uint32_t)((m3 >> b) & 1ull) << 3;
    uint32_t bb = bits;
    while (r) {
        bb &= bb - 1u;
        r--;
    }
    const int sl = bb ? __builtin_ctz(bb) : 3;
    const int z = w * 64 + b;
    const float dx = G.dx;
    const size_t pidx = ((size_t)x * g + y) * g + z;
    const float C[3] = {grid_pos(G.ox, x, dx), grid_pos(G.oy, y, dx), grid_pos(G.oz, z, dx)};
    float P[3] = {C[0], C[1], C[2]};
    if (sl < 3) {
        const float *__restrict__ F = F_all + M.vox_off;
        const uint64_t *__restrict__ om = outm_all + M.word_off;
        const uint64_t *__restrict__ sm = shellm_all ? shellm_all + M.word_off : nullptr;
        const size_t row = (size_t)x * g + y;
        const int W = (int)M.W;
        const float f0 = field_at(F, om, sm, row, g, W, z, dx);
        const float f1 = field_at(F, om, sm, row + (sl == 0 ? (size_t)g : (sl == 1 ? 1 : 0)), g, W, z + (sl == 2), dx);
        float B[3] = {C[0], C[1], C[2]};
        B[sl] = C[sl] + dx;
        const float t = (0.0f - f0) / (f1 - f0);
#pragma unroll
        for (int c3 = 0; c3 < 3; c3++) {
            float dd = B[c3] - C[c3];
            float s = t * dd;
            P[c3] = C[c3] + s;
        }
    }
    vert[3 * (size_t)v + 0] = P[0];
    vert[3 * (size_t)v + 1] = P[1];
    vert[3 * (size_t)v + 2] = P[2];
    vkey[v] = ((uint64_t)pidx << 2) | (uint64_t)sl;
    if constexpr (ATOMS) A.atom[v] = closest_one(M, P[0], P[1], P[2], A.cstart, A.sx, A.perm, A.sorted_ids);
    }
    __syncthreads(); /* S is staged again for the next block */
    }
    return;
    }
    }
    if constexpr (TRI) {
    __shared__ uint32_t S_before[4][256]; /* per cube: vertices before its four columns' lower points */
    /* counts from the device as for the vertices; triangles past the pool are not written */
    if (d_counts) {
        nact = d_counts[2];
        ncube = min(d_counts[4], ncube);
    }
    const uint32_t nb = (ncube + 255u) >> 8;
    /* persistent blocks over the 256-cube blocks, as for the vertices */
    for (uint32_t vb = blockIdx.x - (VERT ? nbv : 0u); vb < nb; vb += gridDim.x - (VERT ? nbv : 0u)) {
    const uint32_t blk = xcd_group<64>(vb, nb);
    stage_item_words(S, acb, list, tstart, nact, nb, blk, wpre, wcoarse);
    const uint32_t cube = blk * 256u + threadIdx.x;
    /* sl: the vertex slots of the eight corners, byte q = x | y << 1 for the column, bit
       2 slot + z in it; has: the columns whose words own vertices (the masks of others are not
       written, and only an edge that ends in a zero point asks for them) */
    uint32_t first_tri = 0, nt = 0, sl = 0, has = 0, cs = 0;
    uint64_t table = 0;
    if (cube < ncube) {
        uint32_t k, wi, first;
        item_word(S, acb, list, cube, k, wi, first);
        const QsMol &M = mols[S.mol >= 0 ? S.mol : seg_coarse<QS_COARSE_ITEMS>(wpre, wcoarse, (uint64_t)wi)];
        const size_t W = M.W, gW = (size_t)M.G.g * W;
        const uint64_t p0 = NT[3 * (size_t)wi], p1 = NT[3 * (size_t)wi + 1], p2 = NT[3 * (size_t)wi + 2];
        const int b = nth_bit(p0 | p1 | p2, cube - first);
        const uint64_t below = (1ull << b) - 1ull;
        first_tri = tbw[wi] + (uint32_t)(__popcll(p0 & below) + 2 * __popcll(p1 & below) + 4 * __popcll(p2 & below));
        nt = (uint32_t)((p0 >> b) & 1ull) + 2u * (uint32_t)((p1 >> b) & 1ull) + 4u * (uint32_t)((p2 >> b) & 1ull);
        uint64_t s[4][4], nw[4];
        uint32_t vb4[4], nv4[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const size_t cw = wi + (q & 1 ? gW : 0) + (q & 2 ? W : 0);
            nw[q] = N[cw];
            nv4[q] = word_verts(cnt[cw]);
            vb4[q] = vbw[cw];
#pragma unroll
            for (int a = 0; a < 4; a++) s[q][a] = S4_all[4 * cw + a];
        }
        uint32_t sg = 0; /* sign bits, bit 2 q + z */
#pragma unroll
        for (int q = 0; q < 4; q++) {
            uint32_t m = 0, before = vb4[q];
#pragma unroll
            for (int a = 0; a < 4; a++) {
                before += (uint32_t)__popcll(s[q][a] & below);
                m |= ((uint32_t)(s[q][a] >> b) & 3u) << (2 * a);
            }
            S_before[q][threadIdx.x] = before;
            sl |= m << (8 * q);
            has |= (nv4[q] ? 1u : 0u) << q;
            sg |= ((uint32_t)(nw[q] >> b) & 3u) << (2 * q);
        }
        if (b == 63) { /* the cube's top corners are in the next words */
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const size_t cw = wi + (q & 1 ? gW : 0) + (q & 2 ? W : 0) + 1;
                sg |= (uint32_t)(N[cw] & 1ull) << (2 * q + 1);
                uint32_t m = 0;
#pragma unroll
                for (int a = 0; a < 4; a++) m |= (uint32_t)(S4_all[4 * cw + a] & 1ull) << (2 * a + 1);
                if (word_verts(cnt[cw])) {
                    /* (a word without vertices below has none of its own slots set) */
                    sl = (has >> q) & 1u ? sl : sl & ~(255u << (8 * q));
                    if (!((has >> q) & 1u)) S_before[q][threadIdx.x] = vbw[cw];
                    has |= 1u << q;
                    sl |= m << (8 * q);
                }
            }
        }
        /* the table's corner order goes round the (x, y) columns 00, 10, 11, 01 */
        const uint32_t lo4 = (sg & 1u) | (sg >> 1 & 2u) | (sg >> 4 & 4u) | (sg >> 1 & 8u);
        const uint32_t hi4 = (sg >> 1 & 1u) | (sg >> 2 & 2u) | (sg >> 5 & 4u) | (sg >> 2 & 8u);
        cs = lo4 | hi4 << 4;
        table = c_tri[cs];
    }
#pragma unroll 1
    for (uint32_t j = 0; j < 5u; j++) {
        const bool on = j < nt && first_tri + j < ntri;
        if (!__ballot(on)) break;
        uint32_t c[3] = {0u, 1u, 2u};
        const uint32_t t = first_tri + j;
        if (on) {
            const uint32_t corners = (uint32_t)(table >> (12u * j));
#pragma unroll
            for (int i = 0; i < 3; i++) {
                const uint32_t e = (corners >> (4 * i)) & 15u;
                const uint32_t d = (uint32_t)(kEdgePacked >> (5u * e));
                uint32_t z = d & 1u, q = (d >> 1) & 3u, a2 = (d >> 2) & 6u; /* a2 = 2 axis */
                uint32_t at = 8u * q + z;                                    /* the corner's slot 0 */
                if (!((sl >> (at + a2)) & (has >> q) & 1u)) {
                    /* the edge has no vertex of its own: its non-negative end is exactly zero and
                       is the vertex (the point slot, after the point's edges) */
                    if ((cs >> (4 * z + (q ^ (q >> 1)))) & 1u) {
                        q |= (a2 == 0 ? 1u : 0u) | (a2 == 2 ? 2u : 0u);
                        z |= a2 == 4 ? 1u : 0u;
                        at = 8u * q + z;
                    }
                    a2 = 6u;
                }
                /* the corner's slots below this one, and all slots of the corner below it */
                const uint32_t lower = __builtin_amdgcn_ubfe(sl, at, a2) & 0x55u;
                const uint32_t under = __builtin_amdgcn_ubfe(sl, 8u * q, 8u * z) & 0x55u;
                c[i] = vbase + S_before[q][threadIdx.x] + (uint32_t)(__popc(lower) + __popc(under));
            }
            tri[3 * (size_t)t + 0] = (int)c[0];
            tri[3 * (size_t)t + 1] = (int)c[1];
            tri[3 * (size_t)t + 2] = (int)c[2];
        }
        /* triangles with a repeated corner (zero grid points) are dropped from the output
           (CudaSurf.cu:820-829): counted here per 256-triangle block and in total */
        uint64_t dm = __ballot(c[0] == c[1] || c[1] == c[2] || c[0] == c[2]);
        if (dm) {
            if ((threadIdx.x & 63) == (uint32_t)__builtin_ctzll(dm)) atomicAdd(deg_total, (uint32_t)__popcll(dm));
            while (dm) {
                const uint32_t lead = (uint32_t)__builtin_ctzll(dm);
                const uint32_t tb = (uint32_t)__shfl((int)(t >> 8), (int)lead, 64);
                const uint64_t same = __ballot((t >> 8) == tb) & dm;
                if ((threadIdx.x & 63) == lead) atomicAdd(&deg_blk[tb], (uint32_t)__popcll(same));
                dm &= ~same;
            }
        }
    }
    __syncthreads(); /* S is staged again for the next block */
    }
    }
}

/* ------------------------------------------------------------------------------------------ */
/* Laplacian smoothing (SmoothMesh.cpp:45-63, 96-124) in Jacobi form on the GPU                 */
/*
 * A vertex's neighbour list is, triangle by triangle in triangle order, the two other corners
 * in the order the reference pushes them (corner 0: 1,2; corner 1: 0,2; corner 2: 0,1).  Every
 * triangle that uses an edge vertex lies in one of the 4 cubes around that edge, every triangle
 * that uses a point vertex in one of the 8 cubes around that point, and triangle order is cube
 * order then case-table order.  So the list is walked from the case table, cube by cube in
 * order, without being stored; the sums run in that order, reading the previous pass.
 */
__device__ __forceinline__ void push_pair(const float *__restrict__ src, uint32_t a, uint32_t b, float &sx, float &sy,
                                          float &sz)
{
    const float *q0 = src + 3 * (size_t)a;
    sx = sx + q0[0];
    sy = sy + q0[1];
    sz = sz + q0[2];
    const float *q1 = src + 3 * (size_t)b;
    sx = sx + q1[0];
    sy = sy + q1[1];
    sz = sz + q1[2];
}

/* first triangle id of polygonised cube (x, y, z) (bit b of word wi): the word's first triangle
   tbw[wi] plus the triangles of the word's cubes below b, from its triangle-count bit planes */
__device__ __forceinline__ uint32_t cube_first_tri(const uint64_t *__restrict__ NT, const uint32_t *__restrict__ tbw, size_t wi,
                                                   int b)
{
    const uint64_t *np = NT + 3 * wi;
    const uint64_t below = (1ull << b) - 1ull;
    return tbw[wi] + (uint32_t)(__popcll(np[0] & below) + 2 * __popcll(np[1] & below) + 4 * __popcll(np[2] & below));
}

/* The grid records the smoothing walk reads (one molecule's view of the batch arrays) */
struct SmoothView {
    MCView V;
    const uint64_t *__restrict__ NT;
    const uint32_t *__restrict__ tbw;
};

__device__ __forceinline__ SmoothView smooth_view(const QsMol &M, const uint64_t *__restrict__ N_all,
                                                  const uint64_t *__restrict__ Zm_all, const uint64_t *__restrict__ S4_all,
                                                  const uint32_t *__restrict__ vbw_all, const uint64_t *__restrict__ NT_all,
                                                  const uint32_t *__restrict__ tbw_all)
{
    SmoothView S;
    S.V.N = N_all + M.word_off;
    S.V.Zm = Zm_all + M.word_off;
    S.V.S4 = S4_all + 4 * M.word_off;
    S.V.vbw = vbw_all + M.word_off;
    S.V.g = M.G.g;
    S.V.W = (int)M.W;
    S.V.lim = M.G.lim;
    S.NT = NT_all + 3 * M.word_off;
    S.tbw = tbw_all + M.word_off;
    return S;
}

/* The incident cubes of an edge vertex: the 4 cubes around the edge in cube order (offsets -1 / 0
   of the two other axes, major first); every one inside the grid contains the sign change, so it
   is polygonised and its word's triangle records exist.  Their first triangles and counts (0 for
   a cube outside the grid, and for a point slot) are loaded here, all four before any is used. */
__device__ __forceinline__ void smooth_edge_cubes(const uint64_t *__restrict__ NT, const uint32_t *__restrict__ tbw, int g, int W,
                                                  int lim, int x, int y, int z, int sl, int (&nt4)[4], uint32_t (&tb4)[4])
{
    /* the cube at the point, and the one below it, lie in the grid on each axis */
    const bool xo = x < lim, yo = y < lim, zo = z < lim;
    const bool xl = x > 0 && x <= lim, yl = y > 0 && y <= lim, zl = z > 0 && z <= lim;
    const uint32_t row = (uint32_t)x * (uint32_t)g + (uint32_t)y;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        /* below the point on which axes (bit 1 of k: not on the first of the two others, bit 0: not
           on the second) */
        const bool hi = k >> 1, lo = k & 1;
        const bool dx = sl != 0 && !hi, dy = sl == 0 ? !hi : (sl == 2 && !lo), dz = sl != 2 && !lo;
        const bool ok = sl < 3 && (dx ? xl : xo) && (dy ? yl : yo) && (dz ? zl : zo);
        const int cz = z - (dz ? 1 : 0);
        const uint32_t wi = ok ? (row - (dx ? (uint32_t)g : 0u) - (dy ? 1u : 0u)) * (uint32_t)W + (uint32_t)(cz >> 6) : 0u;
        const uint64_t *__restrict__ np = NT + 3 * (size_t)wi;
        const uint64_t p0 = np[0], p1 = np[1], p2 = np[2];
        const uint32_t b = (uint32_t)cz & 63u, h = b & 31u, bit = 1u << h, below = bit - 1u;
        const bool top = b >= 32u;
        const uint32_t ml = top ? ~0u : below, mh = top ? below : 0u;
        tb4[k] = tbw[wi] + (uint32_t)(__popc((uint32_t)p0 & ml) + __popc((uint32_t)(p0 >> 32) & mh)) +
                 2u * (uint32_t)(__popc((uint32_t)p1 & ml) + __popc((uint32_t)(p1 >> 32) & mh)) +
                 4u * (uint32_t)(__popc((uint32_t)p2 & ml) + __popc((uint32_t)(p2 >> 32) & mh));
        const uint32_t q0 = top ? (uint32_t)(p0 >> 32) : (uint32_t)p0, q1 = top ? (uint32_t)(p1 >> 32) : (uint32_t)p1,
                       q2 = top ? (uint32_t)(p2 >> 32) : (uint32_t)p2;
        nt4[k] = ok ? (int)(((q0 >> h) & 1u) | ((q1 >> h) & 1u) << 1 | ((q2 >> h) & 1u) << 2) : 0;
    }
}

/* Triangles a smoothing thread takes per round.  Bound by the memory round trips of the gathers:
   one triangle at a time is two dependent trips each (its corners, then the positions), about 18
   triangles for the longest lane of a wave.  Four at a time measured 0.228 -> 0.185 ms on the
   50,000-atom 0.2 A mesh, 1.02 -> 0.80 ms on 256 molecules at 0.5 A (23.8 M vertices); two
   0.195 and 0.854, three 0.191 and 0.815, six 0.196 and 0.845 (registers). */
constexpr int SM_U = 4;

/* vertex v's Jacobi sum over the neighbour list walked from its cubes, written to dst: an edge
   vertex's, from the cubes of smooth_edge_cubes, U triangles per round */
template <int U>
__device__ __forceinline__ void smooth_edge(uint32_t v, const int (&nt4)[4], const uint32_t (&tb4)[4], const int *__restrict__ tri,
                                            const float *__restrict__ src, float *__restrict__ dst)
{
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
    uint32_t cnt = 0;
    /* the four cubes' triangles as one sequence, U at a time: their corners are loaded
       together, then the other corners' positions together, then added in order */
    const int s1 = nt4[0], s2 = s1 + nt4[1], s3 = s2 + nt4[2], total = s3 + nt4[3];
    const uint32_t d0 = tb4[0], d1 = tb4[1] - (uint32_t)s1, d2 = tb4[2] - (uint32_t)s2, d3 = tb4[3] - (uint32_t)s3;
    for (int j = 0; j < total; j += U) {
        uint32_t a[U], b[U], c[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = min(j + u, total - 1);
            const uint32_t t = (uint32_t)i + (i < s1 ? d0 : (i < s2 ? d1 : (i < s3 ? d2 : d3)));
            const int *tt = tri + 3 * (size_t)t;
            a[u] = (uint32_t)tt[0];
            b[u] = (uint32_t)tt[1];
            c[u] = (uint32_t)tt[2];
        }
        bool hit[U];
        float q[U][6];
#pragma unroll
        for (int u = 0; u < U; u++) {
            hit[u] = j + u < total && (a[u] == v || b[u] == v || c[u] == v);
            const float *q0 = src + 3 * (size_t)(hit[u] ? (a[u] == v ? b[u] : a[u]) : v);
            const float *q1 = src + 3 * (size_t)(hit[u] ? (c[u] == v ? b[u] : c[u]) : v);
#pragma unroll
            for (int e = 0; e < 3; e++) {
                q[u][e] = q0[e];
                q[u][3 + e] = q1[e];
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (!hit[u]) continue;
            sx = sx + q[u][0];
            sy = sy + q[u][1];
            sz = sz + q[u][2];
            sx = sx + q[u][3];
            sy = sy + q[u][4];
            sz = sz + q[u][5];
            cnt += 2;
        }
    }
    const float fc = (float)cnt;
    dst[3 * (size_t)v + 0] = sx / fc;
    dst[3 * (size_t)v + 1] = sy / fc;
    dst[3 * (size_t)v + 2] = sz / fc;
}

/* a point vertex's, from the 8 cubes around it */
__device__ __forceinline__ void smooth_point(const SmoothView &S, uint32_t v, int x, int y, int z, const int *__restrict__ tri,
                                             const float *__restrict__ src, float *__restrict__ dst)
{
    const int g = S.V.g, W = S.V.W, lim = S.V.lim;
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
    uint32_t cnt = 0;
    /* a zero grid point: the 8 cubes around it, every corner that is this vertex */
    for (int k = 0; k < 8; k++) {
        const int cx = x - 1 + (k >> 2), cy = y - 1 + ((k >> 1) & 1), cz = z - 1 + (k & 1);
        if (cx < 0 || cy < 0 || cz < 0 || cx >= lim || cy >= lim || cz >= lim) continue;
        const int ci = S.V.cube_index(cx, cy, cz);
        const int nt = tri_count(ci);
        if (!nt) continue;
        const uint32_t tb = cube_first_tri(S.NT, S.tbw, ((size_t)cx * g + cy) * W + (cz >> 6), cz & 63);
        for (int t = 0; t < nt; t++) {
            const int *tt = tri + 3 * (size_t)(tb + t);
            const uint32_t a = (uint32_t)tt[0], b = (uint32_t)tt[1], c = (uint32_t)tt[2];
            if (a == v) { push_pair(src, b, c, sx, sy, sz); cnt += 2; }
            if (b == v) { push_pair(src, a, c, sx, sy, sz); cnt += 2; }
            if (c == v) { push_pair(src, a, b, sx, sy, sz); cnt += 2; }
        }
    }
    const float fc = (float)cnt;
    dst[3 * (size_t)v + 0] = sx / fc;
    dst[3 * (size_t)v + 1] = sy / fc;
    dst[3 * (size_t)v + 2] = sz / fc;
}

/* grid point (x, y, z) and slot of a vertex key (grid point index << 2 | slot; a molecule's grid
   has fewer than 2^32 points) */
__device__ __forceinline__ void vertex_point(uint64_t key, int g, int &x, int &y, int &z, int &sl)
{
    sl = (int)(key & 3ull);
    const uint32_t p = (uint32_t)(key >> 2), ug = (uint32_t)g;
    const uint32_t xy = p / ug;
    z = (int)(p - xy * ug);
    x = (int)(xy / ug);
    y = (int)(xy - (uint32_t)x * ug);
}

/* ------------------------------------------------------------------------------------------ */
/* degenerate-triangle filter (CudaSurf.cu:820-829), order preserving: block b of 256 triangles
   writes its kept ones from position 256 b - dpre[b] on, dpre being the exclusive prefix of the
   per-block degenerate counts */
__device__ __forceinline__ bool tri_degenerate(const int *__restrict__ tri, uint32_t t)
{
    const int x = tri[3 * (size_t)t], y = tri[3 * (size_t)t + 1], z = tri[3 * (size_t)t + 2];
    return !(x != y && y != z && x != z);
}

/* ONE: one molecule.  Its read-back {totals[0..3], first vertices (0, nv), kept triangles before its
   first and last (0, nt - *ndeg)} and the last two pairs (vpre, kept) are written here too.
   self: dpre holds the per-block counts themselves (at most TRI_SELF_BLOCKS of them) and each block
   adds up those before it, which only happens when there is something to drop. */
template <bool ONE>
__device__ __forceinline__ void tri_compact(const int *__restrict__ tri, uint32_t nt, const uint32_t *__restrict__ dpre,
                                            const uint32_t *__restrict__ totals, int *__restrict__ out,
                                            const uint32_t *__restrict__ d_nt, int self, uint32_t nv, uint32_t *__restrict__ vpre,
                                            uint32_t *__restrict__ kept, uint32_t *__restrict__ rb, uint32_t bid, uint32_t nblocks)
{
    __shared__ uint32_t wkeep[4], lds[256 / 64 + 1];
    const uint32_t ndeg = totals[3];
    if (ONE && bid == 0 && threadIdx.x < 8) {
        const uint32_t t = threadIdx.x, all_t = d_nt ? *d_nt : nt, all_v = d_nt ? totals[1] : nv;
        const uint32_t end = t == 5 ? all_v : (t == 7 ? all_t - ndeg : 0u);
        rb[t] = t < 4 ? totals[t] : end;
        if (t >= 6) kept[t - 6] = end;
        else if (t >= 4) vpre[t - 4] = end;
    }
    if (ndeg == 0) return; /* nothing to drop: the caller keeps the input array */
    if (d_nt) nt = min(*d_nt, nt); /* the device count within the launch's pool */
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    /* persistent blocks over the 256-triangle blocks */
    for (uint32_t b = bid; b * 256u < nt; b += nblocks) {
        const uint32_t t = b * 256u + threadIdx.x;
        const bool keep = t < nt && !tri_degenerate(tri, t);
        const uint64_t km = __ballot(keep);
        if (lane == 0) wkeep[wid] = (uint32_t)__popcll(km);
        __syncthreads();
        uint32_t before;
        if (ONE && self) {
            uint32_t x = 0;
            for (uint32_t k = threadIdx.x; k < b; k += 256u) x += dpre[k];
            before = block_sum<256>(x, lds);
        } else {
            before = dpre[b];
        }
        uint32_t o = b * 256u - before + (uint32_t)__popcll(km & ((1ull << lane) - 1ull));
        for (int k = 0; k < wid; k++) o += wkeep[k];
        if (keep) {
            out[3 * (size_t)o] = tri[3 * (size_t)t];
            out[3 * (size_t)o + 1] = tri[3 * (size_t)t + 1];
            out[3 * (size_t)o + 2] = tri[3 * (size_t)t + 2];
        }
        __syncthreads(); /* wkeep is written again for the next block */
    }
}

template <bool ONE>
__global__ void __launch_bounds__(256) k_tri_compact(const int *__restrict__ tri, uint32_t nt,
                                                     const uint32_t *__restrict__ dpre, const uint32_t *__restrict__ totals,
                                                     int *__restrict__ out, const uint32_t *__restrict__ d_nt, int self, uint32_t nv,
                                                     uint32_t *__restrict__ vpre, uint32_t *__restrict__ kept,
                                                     uint32_t *__restrict__ rb)
{
    tri_compact<ONE>(tri, nt, dpre, totals, out, d_nt, self, nv, vpre, kept, rb, blockIdx.x, gridDim.x);
}

/* ------------------------------------------------------------------------------------------ */
/* triangles and vertices that a smoothing block stages in LDS at most (10 bits per corner) */
constexpr uint32_t SM_TRI = 1408, SM_VERT = 1024;
/* expected vertices above which blocks stage: a smaller mesh is bound by a block's chain of loads, which
   staging makes longer (2,000 atoms at 0.5 A: 9 us without, 12 with) */
constexpr uint32_t SM_STAGED_MIN = 1u << 19;

/* one Jacobi pass, one thread per vertex.  A polygonised cube's triangles are consecutive from
   its first triangle id (its word's triangle base plus the triangle-count planes below it), and
   its count is its bit of those planes, so each incident triangle's other corners are read from
   the triangle array.  An edge vertex is a corner of exactly the triangles whose case-table entry
   is its cube edge (no other edge of the cube shares its id), so it finds them by id.
   Bound by the address unit when every vertex gathers them from memory: eight triangles and the
   other corners' positions are about 50 gathers, though neighbouring vertices share them.  With
   STAGED a block loads them once, in order, into LDS: its 256 vertices lie in consecutive grid rows
   [ra, rb] (row = x g + y), so their triangles lie in two ranges of the triangle array, the rows
   [ra - 1, rb] of their own plane and of the plane below, and those triangles' corners in three
   ranges of the vertices, the rows [ra - 1, rb + 1] of the planes below, own and above: about 1,150
   triangles and 900 vertices.  A triangle is kept as its corners' places among the staged vertices.
   A block whose ranges are larger (1 to 3 % of them) or whose vertices belong to two molecules
   gathers from memory.  Then bound by VALU issue, and by waves in flight: 64 registers, so the
   triangles' loads end before the positions' begin.  On 256 molecules at 0.5 A gathers took 0.793 ms
   and this takes 0.566, on the 50,000-atom 0.2 A mesh 0.188 and 0.156, on 1M atoms at 0.5 A (two passes)
   0.660 and 0.537.
   COMPACT: blocks from nbs on filter the triangles, which the pass only reads too (one molecule, the
   work of k_tri_compact<true>): on a small mesh, a chain of short launches, one launch less (2,000
   atoms at 0.5 A: 129 -> 118 us in all). */
template <bool STAGED, bool COMPACT>
__global__ void __launch_bounds__(256, STAGED ? 8 : 1) k_smooth(const QsMol *__restrict__ mols, const uint32_t *__restrict__ vpre,
                                                   const uint32_t *__restrict__ vcoarse, const uint64_t *__restrict__ wpre,
                                                   const uint32_t *__restrict__ wcoarse, const uint32_t *__restrict__ list,
                                                   const uint32_t *__restrict__ vstart, const uint64_t *__restrict__ N_all,
                                                   const uint64_t *__restrict__ Zm_all, const uint64_t *__restrict__ S4_all,
                                                   const uint32_t *__restrict__ vbw_all, const uint64_t *__restrict__ vkey,
                                                   uint32_t nv, uint32_t ntri, const uint64_t *__restrict__ NT_all,
                                                   const uint32_t *__restrict__ tbw_all, const int *__restrict__ tri,
                                                   const float *__restrict__ src, float *__restrict__ dst,
                                                   const uint32_t *__restrict__ d_counts, QsCompact K, uint32_t nbs)
{
    const uint32_t nblocks = COMPACT ? nbs : gridDim.x;
    if constexpr (COMPACT) {
        if (blockIdx.x >= nbs) {
            tri_compact<true>(tri, ntri, K.deg_blk, d_counts, K.out, d_counts, 1, 0u, K.vpre, K.kept, K.rb, blockIdx.x - nbs,
                              gridDim.x - nbs);
            return;
        }
    }
    __shared__ uint32_t s_tri[STAGED ? SM_TRI : 1];           /* corners' places, in bits 2, 12 and 22 on */
    __shared__ float s_pos[3][STAGED ? SM_VERT : 1];
    /* a mesh larger than the pools (the run is repeated with larger ones) has ids past them: nothing
       to smooth then */
    if (d_counts[1] > nv || d_counts[0] > ntri) return;
    nv = d_counts[1];
    const uint32_t nact = d_counts[2];
    const uint32_t nb = (nv + 255u) >> 8;
    /* persistent blocks over the 256-vertex blocks (on XCDs as in k_mc_emit) */
    for (uint32_t vb = blockIdx.x; vb < nb; vb += nblocks) {
        const uint32_t blk = xcd_group<64>(vb, nb), v = blk * 256u + threadIdx.x;
        bool staged = false;
        if constexpr (STAGED) {
            const uint32_t w0 = list[vstart[blk]], w1 = list[blk + 1 < nb ? vstart[blk + 1] : nact - 1u];
            const int m0 = wcoarse ? __builtin_amdgcn_readfirstlane(seg_coarse<QS_COARSE_ITEMS>(wpre, wcoarse, (uint64_t)w0)) : 0;
            const int m1 = wcoarse ? __builtin_amdgcn_readfirstlane(seg_coarse<QS_COARSE_ITEMS>(wpre, wcoarse, (uint64_t)w1)) : 0;
            if (m0 == m1) {
                const QsMol &M = mols[m0];
                const int g = M.G.g, W = (int)M.W, last = g * g - 1; /* (the last row holds nothing) */
                const int ra = (int)((w0 - (uint32_t)M.word_off) / (uint32_t)W), rb = (int)((w1 - (uint32_t)M.word_off) / (uint32_t)W);
                const uint32_t *__restrict__ vbw = vbw_all + M.word_off, *__restrict__ tbw = tbw_all + M.word_off;
                /* the ranges of triangles (t, own plane and below) and vertices (u, own, below,
                   above), and how many entries come before each in LDS */
                const auto at = [&](int r) { return (size_t)iclamp(r, 0, last) * W; };
                const uint32_t t0 = tbw[at(ra - 1)], t1 = tbw[at(ra - g - 1)];
                const uint32_t na = tbw[at(rb + 1)] - t0, nt = na + tbw[at(rb - g + 1)] - t1;
                const uint32_t u0 = vbw[at(ra - 1)], u1 = vbw[at(ra - g - 1)], u2 = vbw[at(ra + g - 1)];
                const uint32_t nu0 = vbw[at(rb + 2)] - u0, nu1 = nu0 + vbw[at(rb - g + 2)] - u1, nu = nu1 + vbw[at(rb + g + 2)] - u2;
                /* (and the rows' points, as offsets from the block's first, are exact in float) */
                staged = nt - 1u < SM_TRI && nu - 1u < SM_VERT && (uint64_t)(rb - ra + 1) * (uint32_t)g < (1u << 20);
                if (staged) {
                    /* all of a thread's triangles, then all of its positions, are loaded before any is
                       used (past the end the last one again) */
                    constexpr uint32_t KT = (SM_TRI + 255u) / 256u, KV = SM_VERT / 256u;
                    int tt[KT][3];
#pragma unroll
                    for (uint32_t k = 0; k < KT; k++) {
                        const uint32_t i = min(k * 256u + threadIdx.x, nt - 1u);
                        const int *__restrict__ q = tri + 3 * (size_t)(i + (i < na ? t0 : t1 - na));
#pragma unroll
                        for (int c = 0; c < 3; c++) tt[k][c] = q[c];
                    }
                    const uint64_t key = vkey[min(v, nv - 1u)];
                    /* (the ranges' ids ascend from the plane below to the one above; where the rows are so
                       empty that two ranges overlap, the later one's place is every use's) */
                    const auto place = [&](int id) { return (uint32_t)id - ((uint32_t)id >= u2 ? u2 - nu1 : ((uint32_t)id >= u0 ? u0 : u1 - nu0)); };
#pragma unroll
                    for (uint32_t k = 0; k < KT; k++)
                        if (k * 256u + threadIdx.x < nt)
                            s_tri[k * 256u + threadIdx.x] = place(tt[k][0]) << 2 | place(tt[k][1]) << 12 | place(tt[k][2]) << 22;
                    float pp[KV][3];
#pragma unroll
                    for (uint32_t k = 0; k < KV; k++) {
                        const uint32_t i = min(k * 256u + threadIdx.x, nu - 1u);
                        const float *__restrict__ q = src + 3 * (size_t)(i + (i < nu0 ? u0 : (i < nu1 ? u1 - nu0 : u2 - nu1)));
#pragma unroll
                        for (int c = 0; c < 3; c++) pp[k][c] = q[c];
                    }
                    /* the vertex's point: key >> 2 = row g + z */
                    const float inv_g = 1.0f / (float)g;
                    const int xa = ra / g, o = (int)((uint32_t)(key >> 2) - (uint32_t)ra * (uint32_t)g);
                    const int dr = (int)(((float)o + 0.5f) * inv_g), z = o - dr * g, r = ra + dr - xa * g;
                    const int dx_ = (int)(((float)r + 0.5f) * inv_g), x = xa + dx_, y = r - dx_ * g, sl = (int)(key & 3ull);
                    /* its four cubes' first triangles (as places in LDS) and counts */
                    int nt4[4];
                    uint32_t tb4[4];
                    smooth_edge_cubes(NT_all + 3 * M.word_off, tbw, g, W, M.G.lim, x, y, z, sl, nt4, tb4);
#pragma unroll
                    for (uint32_t k = 0; k < KV; k++)
                        if (k * 256u + threadIdx.x < nu)
#pragma unroll
                            for (int c = 0; c < 3; c++) s_pos[c][k * 256u + threadIdx.x] = pp[k][c];
                    __syncthreads();
                    if (v < nv) {
                        if (sl < 3) {
                            /* cubes 2 and 3, and all of an x edge's, lie in the own plane */
                            const uint32_t lo = sl == 0 ? 0u - t0 : na - t1;
                            const int s1 = nt4[0], s2 = s1 + nt4[1], s3 = s2 + nt4[2], total = s3 + nt4[3];
                            const uint32_t d0 = tb4[0] + lo, d1 = tb4[1] + lo - (uint32_t)s1, d2 = tb4[2] - t0 - (uint32_t)s2,
                                           d3 = tb4[3] - t0 - (uint32_t)s3, me = place((int)v) << 2;
                            const auto pos = [&](int c, uint32_t b) { return *(const float *)((const char *)s_pos[c] + b); };
                            float sx = 0.0f, sy = 0.0f, sz = 0.0f;
                            uint32_t cnt = 0;
#pragma unroll 2
                            for (int i = 0; i < total; i++) {
                                const uint32_t p = s_tri[(uint32_t)i + (i < s1 ? d0 : (i < s2 ? d1 : (i < s3 ? d2 : d3)))];
                                const uint32_t a = p & 0xFFCu, b = (p >> 10) & 0xFFCu, c = (p >> 20) & 0xFFCu;
                                if (a == me || b == me || c == me) {
                                    const uint32_t q0 = a == me ? b : a, q1 = c == me ? b : c;
                                    sx = sx + pos(0, q0);
                                    sy = sy + pos(1, q0);
                                    sz = sz + pos(2, q0);
                                    sx = sx + pos(0, q1);
                                    sy = sy + pos(1, q1);
                                    sz = sz + pos(2, q1);
                                    cnt += 2;
                                }
                            }
                            const float fc = (float)cnt;
                            dst[3 * (size_t)v + 0] = sx / fc;
                            dst[3 * (size_t)v + 1] = sy / fc;
                            dst[3 * (size_t)v + 2] = sz / fc;
                        } else {
                            const SmoothView S = smooth_view(M, N_all, Zm_all, S4_all, vbw_all, NT_all, tbw_all);
                            smooth_point(S, v, x, y, z, tri, src, dst);
                        }
                    }
                    __syncthreads(); /* the next block is staged */
                }
            }
        }
        if (!staged && v < nv) {
            const QsMol &M = mols[seg_of_wave(vpre, vcoarse, v)];
            const SmoothView S = smooth_view(M, N_all, Zm_all, S4_all, vbw_all, NT_all, tbw_all);
            int x, y, z, sl;
            vertex_point(vkey[v], S.V.g, x, y, z, sl);
            if (sl < 3) {
                int nt4[4];
                uint32_t tb4[4];
                smooth_edge_cubes(S.NT, S.tbw, S.V.g, S.V.W, S.V.lim, x, y, z, sl, nt4, tb4);
                smooth_edge<STAGED ? 1 : SM_U>(v, nt4, tb4, tri, src, dst);
            } else {
                smooth_point(S, v, x, y, z, tri, src, dst);
            }
        }
    }
}

/* ------------------------------------------------------------------------------------------ */
/* Laplacian smoothing over a triangle array (SmoothMesh.cpp:45-63, 96-124), for meshes built in
 * x-slabs, whose grid records do not outlive their slab.  Each vertex's incidences (corner index
 * 3 t + j of triangle t) are listed per vertex and sorted, so the Jacobi sums run over the
 * reference's neighbour list in its push order -- triangle by triangle, corner 0: 1,2; corner 1:
 * 0,2; corner 2: 0,1 -- as k_smooth walks it from the grid records: the results are the same bits. */
/* (corner ids outside [0, nv) are skipped: they cannot occur, and a mistake shows as a mesh
   difference rather than a stray write) */
__global__ void __launch_bounds__(256) k_incid_count(const int *__restrict__ tri, uint64_t ncorner, uint32_t nv,
                                                     uint32_t *__restrict__ cnt)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= ncorner) return;
    const uint32_t v = (uint32_t)tri[i];
    if (v < nv) atomicAdd(&cnt[v], 1u);
}

__global__ void __launch_bounds__(256) k_incid_fill(const int *__restrict__ tri, uint64_t ncorner, uint32_t nv,
                                                    const uint32_t *__restrict__ start, uint32_t *__restrict__ cursor,
                                                    uint32_t *__restrict__ ent)
{
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= ncorner) return;
    const uint32_t v = (uint32_t)tri[i];
    if (v < nv) ent[start[v] + atomicAdd(&cursor[v], 1u)] = (uint32_t)i;
}

/* each vertex's incidences in increasing corner index (insertion sort; a few per vertex) */
__global__ void __launch_bounds__(256) k_incid_sort(const uint32_t *__restrict__ start, uint32_t nv, uint32_t *__restrict__ ent)
{
    const uint32_t v = blockIdx.x * 256 + threadIdx.x;
    if (v >= nv) return;
    const uint32_t a = start[v], b = start[v + 1];
    for (uint32_t i = a + 1; i < b; i++) {
        const uint32_t x = ent[i];
        uint32_t j = i;
        while (j > a && ent[j - 1] > x) {
            ent[j] = ent[j - 1];
            j--;
        }
        ent[j] = x;
    }
}

/* one Jacobi pass over the listed incidences */
__global__ void __launch_bounds__(256) k_smooth_incid(const uint32_t *__restrict__ start, const uint32_t *__restrict__ ent,
                                                      const int *__restrict__ tri, uint32_t nv, const float *__restrict__ src,
                                                      float *__restrict__ dst)
{
    const uint32_t v = xcd_group<64>(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    if (v >= nv) return;
    float sx = 0.0f, sy = 0.0f, sz = 0.0f;
    uint32_t cnt = 0;
    for (uint32_t k = start[v], e = start[v + 1]; k < e; k++) {
        const uint32_t c = ent[k];
        const uint32_t t = c / 3u, j = c - 3u * t;
        const int *tt = tri + 3 * (size_t)t;
        const uint32_t a = min((uint32_t)tt[j == 0 ? 1 : 0], nv - 1u), b = min((uint32_t)tt[j == 2 ? 1 : 2], nv - 1u);
        push_pair(src, a, b, sx, sy, sz);
        cnt += 2;
    }
    const float fc = (float)cnt;
    dst[3 * (size_t)v + 0] = sx / fc;
    dst[3 * (size_t)v + 1] = sy / fc;
    dst[3 * (size_t)v + 2] = sz / fc;
}

/* ------------------------------------------------------------------------------------------ */
/* Per-vertex normals (the normals field that MeshData leaves commented out, SmoothMesh.h:34):
 * the unit field gradient at the vertex's marching-cubes position.  The gradient at a grid point
 * is the central difference (one-sided at the grid faces) of the field; an edge vertex blends
 * its two end points' gradients with the vertex's edge parameter t, a zero-point vertex takes
 * its point's.  The field grows outwards (negative inside), so the normals point outwards. */
/* one molecule's field, addressed by grid row (x * g + y) and z */
struct FieldView {
    const float *F;
    const uint64_t *outm, *shellm;
    int g, W;
    float dx;
    __device__ __forceinline__ float at(size_t row, int z) const { return field_at(F, outm, shellm, row, g, W, z, dx); }
};

/* derivative along axis a (0 x, 1 y, 2 z) at grid point (row, z), whose coordinate on that axis is i */
__device__ __forceinline__ float grad_axis(const FieldView &F, size_t row, int z, int a, int i, int g, float dx)
{
    const size_t dr = a == 0 ? (size_t)g : (a == 1 ? 1 : 0);
    const int dz = a == 2;
    if (i > 0 && i < g - 1) return (F.at(row + dr, z + dz) - F.at(row - dr, z - dz)) / (2.0f * dx);
    if (i == 0) return (F.at(row + dr, z + dz) - F.at(row, z)) / dx;
    return (F.at(row, z) - F.at(row - dr, z - dz)) / dx;
}

__global__ void __launch_bounds__(256) k_vertex_normals(const QsMol *__restrict__ mols, const uint32_t *__restrict__ vpre,
                                                        const uint32_t *__restrict__ vcoarse, const uint64_t *__restrict__ vkey,
                                                        uint32_t nv, const float *__restrict__ F_all,
                                                        const uint64_t *__restrict__ outm_all,
                                                        const uint64_t *__restrict__ shellm_all, float *__restrict__ out)
{
    const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    const QsMol &M = mols[seg_of_wave(vpre, vcoarse, v)];
    const int g = M.G.g;
    const float dx = M.G.dx;
    const FieldView F{F_all + M.vox_off, outm_all + M.word_off,
                      shellm_all ? shellm_all + M.word_off : nullptr, g, (int)M.W, dx};
    const uint64_t key = vkey[v];
    const int sl = (int)(key & 3ull);
    const uint32_t p = (uint32_t)(key >> 2), ug = (uint32_t)g;
    const uint32_t xy = p / ug;
    int c[3];
    c[2] = (int)(p - xy * ug);
    c[0] = (int)(xy / ug);
    c[1] = (int)(xy - (uint32_t)c[0] * ug);
    const size_t row = (size_t)c[0] * g + c[1];
    const int z = c[2];
    float n[3];
#pragma unroll
    for (int a = 0; a < 3; a++) n[a] = grad_axis(F, row, z, a, c[a], g, dx);
    if (sl < 3) {
        const size_t rq = row + (sl == 0 ? (size_t)g : (sl == 1 ? 1 : 0));
        const int zq = z + (sl == 2);
        const float f0 = F.at(row, z), f1 = F.at(rq, zq);
        const float t = (0.0f - f0) / (f1 - f0);
        const float s = 1.0f - t;
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const float g1 = grad_axis(F, rq, zq, a, c[a] + (a == sl), g, dx);
            n[a] = s * n[a] + t * g1;
        }
    }
    const float len = sqrtf(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
    const float inv = len > 0.0f ? 1.0f / len : 0.0f;
    out[3 * (size_t)v + 0] = n[0] * inv;
    out[3 * (size_t)v + 1] = n[1] * inv;
    out[3 * (size_t)v + 2] = n[2] * inv;
}

/* Per-vertex colours (the colors field that MeshData leaves commented out, SmoothMesh.h:35): the
   colour of the vertex's closest atom, from a per-atom RGBA table laid out like the atom input
   (a batch's molecules concatenated); a vertex without a closest atom gets (0, 0, 0, 0).  When the
   ids are in the reference's cell-sorted convention (perm != nullptr), the id is mapped back to
   the input order through perm (sorted position -> input index, batch-global) first. */
__global__ void __launch_bounds__(256) k_vertex_colors(const QsMol *__restrict__ mols, const uint32_t *__restrict__ vpre,
                                                       const uint32_t *__restrict__ vcoarse, const int *__restrict__ atom,
                                                       const int *__restrict__ perm, uint32_t nv,
                                                       const float4 *__restrict__ table, float4 *__restrict__ out)
{
    const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    const QsMol &M = mols[seg_of_wave(vpre, vcoarse, v)];
    const int a = atom[v];
    if (a < 0) {
        out[v] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const uint32_t in = perm ? (uint32_t)perm[M.atom_off + (uint32_t)a] : M.atom_off + (uint32_t)a;
    out[v] = table[in];
}

/* ------------------------------------------------------------------------------------------ */
/* Per-molecule first vertex and first triangle of a batch, from the word scans: molecule m's are
   the exclusive scans at its first row word (wpre[m]; at or past the scanned words nw for a
   molecule without words, whose mesh is empty and starts at the totals).  vpre / tpre get nmol + 1 entries, the last one the
   totals (counts[1] vertices, counts[0] triangles).  In the same launch, the coarse index of the
   vertex prefix: entry k (of ncoarse, enough for a pool of vertices) = the last molecule whose
   first vertex is at or before vertex k << QS_COARSE_ITEMS, searched over the same first
   vertices read from the word scan. */
__device__ __forceinline__ uint32_t mol_first_vertex(const uint32_t *__restrict__ vbw, const uint64_t *__restrict__ wpre,
                                                     uint64_t nw, int nmol, const uint32_t *__restrict__ counts, int m)
{
    const uint64_t w = (m < nmol) ? wpre[m] : nw;
    return (w < nw) ? vbw[w] : counts[1];
}

__global__ void __launch_bounds__(256) k_mesh_bases(const uint32_t *__restrict__ vbw, const uint32_t *__restrict__ tbw,
                                                    const uint64_t *__restrict__ wpre, uint64_t nw, int nmol,
                                                    const uint32_t *__restrict__ counts, uint32_t *__restrict__ vpre,
                                                    uint64_t *__restrict__ tpre, uint32_t *__restrict__ coarse,
                                                    uint32_t ncoarse)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i <= (uint32_t)nmol) {
        const int m = (int)i;
        const uint64_t w = (m < nmol) ? wpre[m] : nw;
        vpre[m] = (w < nw) ? vbw[w] : counts[1];
        tpre[m] = (w < nw) ? tbw[w] : counts[0];
    }
    if (i < ncoarse) {
        const uint64_t t = (uint64_t)i << QS_COARSE_ITEMS;
        int lo = 0, hi = nmol - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if ((uint64_t)mol_first_vertex(vbw, wpre, nw, nmol, counts, mid) <= t) lo = mid;
            else hi = mid - 1;
        }
        coarse[i] = (uint32_t)lo;
    }
}

/* degenerate triangles per 256-triangle block (and their total, added to *deg_total), as the
   triangle kernel counts them: for triangle arrays assembled from several launches */
__global__ void __launch_bounds__(256) k_deg_count(const int *__restrict__ tri, uint32_t nt, uint32_t *__restrict__ deg_blk,
                                                   uint32_t *__restrict__ deg_total)
{
    __shared__ uint32_t lds[256 / 64 + 1];
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    const uint32_t d = (t < nt && tri_degenerate(tri, t)) ? 1u : 0u;
    const uint32_t sum = block_sum<256>(d, lds);
    if (threadIdx.x == 0) {
        deg_blk[blockIdx.x] = sum;
        if (sum) atomicAdd(deg_total, sum);
    }
}

/* kept triangles before each of n boundaries idx[i] (molecule starts and the end) */
__global__ void __launch_bounds__(256) k_tri_kept_before(const int *__restrict__ tri, const uint32_t *__restrict__ dpre,
                                                         const uint64_t *__restrict__ idx, int n, uint32_t tcap,
                                                         uint32_t *__restrict__ out, const uint32_t *__restrict__ totals,
                                                         const uint32_t *__restrict__ vpre, uint32_t *__restrict__ rb)
{
    /* with rb: the run's read-back in one array, {totals[0..3], vpre[0..n), out[0..n)} */
    if (rb && blockIdx.x == 0)
        for (int j = (int)threadIdx.x; j < 4 + n; j += 256) rb[j] = (j < 4) ? totals[j] : vpre[j - 4];
    /* one wave per boundary: the degenerate triangles of the boundary's 256-triangle block below
       it, four per lane, counted by ballot */
    const int i = blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n) return;
    /* (boundaries past the triangle pool occur only when the mesh overflowed it) */
    const uint32_t t = (uint32_t)min(idx[i], (uint64_t)tcap);
    const uint32_t b = t >> 8;
    uint32_t d = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t u = (b << 8) + (uint32_t)(64 * k + lane);
        d += (uint32_t)__popcll(__ballot(u < t && tri_degenerate(tri, u)));
    }
    if (lane == 0) {
        out[i] = t - dpre[b] - d;
        if (rb) rb[4 + n + i] = t - dpre[b] - d;
    }
}

/* one molecule's record, from the launch's arguments, and a clear of n counters */
__global__ void __launch_bounds__(256) k_put_mol(QsMol m, QsMol *__restrict__ dst, uint32_t *__restrict__ clear, uint32_t n)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) *dst = m;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) clear[i] = 0u;
}

/* plain device copy (16-byte vectors, grid-stride): the reference point for traffic counters */
__global__ void __launch_bounds__(256) k_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst, uint64_t n16)
{
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += (uint64_t)gridDim.x * 256) dst[i] = src[i];
}

/* a mesh's three arrays (4-byte items) to the caller's, in one launch, its corner ids less v0: small
   ones are bound by the start of each copy, not by its bytes */
__device__ __forceinline__ void copy_items(const uint32_t *__restrict__ src, uint32_t *__restrict__ dst, size_t n, uint32_t v0)
{
    const size_t i0 = (size_t)blockIdx.x * 256 + threadIdx.x, step = (size_t)gridDim.x * 256;
    const size_t n4 = (((uintptr_t)src | (uintptr_t)dst) & 15u) ? 0 : n / 4;
    for (size_t i = i0; i < n4; i += step) {
        const uint4 q = ((const uint4 *)src)[i];
        ((uint4 *)dst)[i] = make_uint4(q.x - v0, q.y - v0, q.z - v0, q.w - v0);
    }
    for (size_t i = 4 * n4 + i0; i < n; i += step) dst[i] = src[i] - v0;
}
__global__ void __launch_bounds__(256) k_copy_mesh(const uint32_t *__restrict__ v, const uint32_t *__restrict__ a,
                                                   const uint32_t *__restrict__ t, uint32_t nv, uint32_t nt, uint32_t v0,
                                                   uint32_t *__restrict__ dv, uint32_t *__restrict__ da,
                                                   uint32_t *__restrict__ dt)
{
    copy_items(v, dv, 3 * (size_t)nv, 0u);
    copy_items(a, da, nv, 0u);
    copy_items(t, dt, 3 * (size_t)nt, v0);
}

/* triangles of a batch with vertex indices local to their molecule */
__global__ void __launch_bounds__(256) k_tri_localize(const int *__restrict__ tri, uint32_t nt, const uint32_t *__restrict__ tpre,
                                                      const uint32_t *__restrict__ vpre, int nmol, int *__restrict__ out)
{
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nt) return;
    const int v0 = (int)vpre[seg_of(tpre, nmol, t)];
    for (int c = 0; c < 3; c++) out[3 * (size_t)t + c] = tri[3 * (size_t)t + c] - v0;
}

/* ------------------------------------------------------------------------------------------ */
/* launchers                                                                                    */

static inline unsigned nblk(uint64_t n, unsigned b) { return (unsigned)((n + b - 1) / b); }

/* Launches over a pool of items whose count lives on the device have blocks that loop over 256-item
   blocks up to the count (blocks past it leave at once), at most g_persist_blocks, by default without
   limit.  With one block per item block of the mesh these gather-bound kernels were faster than with
   fewer, longer-lived blocks (smoothing +15 % and closest atom +11 % with 2048 blocks, +19 % and +50 %
   with 1024, on the 50,000-atom 0.2 A mesh). */
static uint32_t g_persist_blocks = 1u << 30;

void qs_set_persistent_blocks(uint32_t n) { g_persist_blocks = std::max<uint32_t>(8u, n & ~7u); }
uint32_t qs_persistent_blocks(void) { return g_persist_blocks; }

static inline unsigned pgrid(uint64_t nb)
{
    return nb <= g_persist_blocks ? (unsigned)std::max<uint64_t>(nb, 1) : g_persist_blocks;
}

/* blocks of the triangle compaction at most: it streams, or leaves at once where nothing is dropped,
   which 335,000 blocks over the pool of 256 molecules at 0.5 A took 70 us for */
constexpr unsigned COMPACT_BLOCKS = 4096;

/* partial boxes per molecule: about 8 atoms per thread of the largest molecule, 1 to BB_PMAX */
/* (a single molecule of up to 8,192 atoms is one block of 1,024 threads and one launch) */
int qs_bbox_parts(uint32_t max_atoms, int nmol)
{
    if (nmol == 1 && max_atoms <= 8192u) return 1;
    const uint32_t p = (max_atoms + 8 * BB_NT - 1) / (8 * BB_NT);
    return (int)std::min<uint32_t>(std::max<uint32_t>(p, 1u), BB_PMAX);
}

size_t qs_bbox_part_floats(int nmol, int parts) { return (size_t)nmol * parts * BB_NV; }

void qs_launch_bbox(const float *pos, const float *rad, const uint32_t *off, uint32_t o0, uint32_t o1, int nmol, int parts,
                    float *part, float *out, hipStream_t s)
{
    /* one partial box per molecule is its box (part[m][0] and out[m] are at the same offset) */
    if (parts == 1 && nmol == 1) {
        hipLaunchKernelGGL(k_bbox_part<1024>, dim3(1, 1), dim3(1024), 0, s, pos, rad, off, o0, o1, out);
        return;
    }
    hipLaunchKernelGGL(k_bbox_part<BB_NT>, dim3(parts, nmol), dim3(BB_NT), 0, s, pos, rad, off, o0, o1, parts == 1 ? out : part);
    if (parts == 1) return;
    hipLaunchKernelGGL(k_bbox_final, dim3(nmol), dim3(64), 0, s, part, parts, out);
}

void qs_launch_hash_count(QsBatch B, uint32_t nblocks, const float *pos, int2 *key, uint32_t *count, hipStream_t s)
{
    hipLaunchKernelGGL(k_hash_count, dim3(nblocks), dim3(256), 0, s, B, pos, key, count);
}

void qs_launch_scatter(const int2 *key, int n, const uint32_t *start, int *slot, hipStream_t s)
{
    hipLaunchKernelGGL(k_scatter, dim3(nblk(n, 256)), dim3(256), 0, s, key, n, start, slot);
}

void qs_launch_place(QsBatch B, uint32_t nblocks, const uint32_t *start, const int *slot, uint32_t ncell, const float *pos,
                     const float *rad, int *perm, int2 *cse, float4 *sx, float4 *aux, hipStream_t s)
{
    hipLaunchKernelGGL(k_place, dim3(nblocks), dim3(256), 0, s, B, start, slot, ncell, pos, rad, perm, cse, sx, aux);
}

void qs_launch_gather_aux(QsBatch B, uint32_t nblocks, const int *perm, const float *pos, const float *rad, float4 *sx,
                          float4 *aux, hipStream_t s)
{
    hipLaunchKernelGGL(k_gather_aux, dim3(nblocks), dim3(256), 0, s, B, perm, pos, rad, sx, aux);
}

int qs_pass1_rows_per_wave(QsGrid G)
{
    /* R rows per wavefront with R * dx <= neighbour-cell size */
    int R = (int)(G.dxn / G.dx);
    return R < 1 ? 1 : (R > P1_RMAX ? P1_RMAX : R);
}

/* tuned rows per pass-1 block by voxel size (qs_set_tuned_rows): a short list, looked up by the
   nearest voxel size within 1 % */
static float g_rows_dx[16];
static int g_rows_v[16];
static int g_rows_n = 0;

int qs_set_tuned_rows(float dx, int rows)
{
    if (!(dx > 0.0f)) {
        g_rows_n = 0; /* dx <= 0 clears the table */
        return 0;
    }
    for (int i = 0; i < g_rows_n; i++)
        if (std::fabs(g_rows_dx[i] - dx) <= 0.01f * dx) {
            g_rows_v[i] = rows;
            return 0;
        }
    if (g_rows_n == 16) return -1;
    g_rows_dx[g_rows_n] = dx;
    g_rows_v[g_rows_n++] = rows;
    return 0;
}

int qs_pass1_slab_rows(QsGrid G, int W)
{
    /* 64 rows (or the tuned count for this voxel size, up to 256); both masks in at most 12 KB of LDS
       (a tuned count from a workload of small grids would otherwise give a large grid slabs that
       are too tall: pass 1 of the million-atom shell at 0.5 A, 12 words per row, took 1.22 ms with
       256-row slabs and 0.86 ms with the 64 rows of this cap (0.81 ms with 85), of a 200,000-atom
       molecule at 0.3 A, 11 words per row, 0.64 ms with 93 rows and 0.48 ms with 69, at 0.5 A, 7
       words per row, about 0.30 ms with 146 rows and 0.25 ms with 109); at most 80 neighbour
       cells of y per slab, so the candidate columns (3 x cells times the y cells + 2) stay
       within 256 */
    int yb = P1S_DEFROWS;
    for (int i = 0; i < g_rows_n; i++)
        if (std::fabs(g_rows_dx[i] - G.dx) <= 0.01f * G.dx && g_rows_v[i] >= 1) yb = std::min(P1S_MAXROWS, g_rows_v[i]);
    yb = std::min(yb, std::max(1, 768 / std::max(W, 1)));
    yb = std::min(yb, std::max(1, (int)(80.0f * G.dxn / G.dx)));
    return yb;
}

int qs_pass1_mode(bool direct, bool rows) { return direct ? 2 : (rows ? 1 : 0); }

uint32_t qs_pass1_blocks(const QsMol &M, int mode)
{
    const QsGrid &G = M.G;
    const uint32_t nx = (uint32_t)std::max(M.p1_hi - M.p1_lo, 0);
    if (mode == 2) return M.W * nblk(G.g, 4) * nx;
    if (mode == 1) return nblk(G.g, 4 * M.rows_per_wave) * nx;
    return nblk(G.g, M.slab_rows) * nx;
}

size_t qs_pass1_lds_bytes(const QsMol &M, int mode)
{
    if (mode != 0) return 0;
    return (size_t)16 * M.slab_rows * M.W + (size_t)8 * (M.G.gn + 2);
}

void qs_launch_pass1(QsBatch B, uint32_t nblocks, int mode, size_t lds_bytes, const uint32_t *cstart, const float4 *sx,
                     const float4 *aux, uint64_t *outm, uint64_t *shellm, uint64_t *negm, uint64_t *zerom, uint8_t *tflag,
                     uint8_t tmark, uint32_t *clear, uint32_t nclear, hipStream_t s)
{
    if (mode == 1)
        hipLaunchKernelGGL(k_pass1_rows, dim3(nblocks), dim3(256), 0, s, B, cstart, sx, aux, outm, shellm);
    else
        hipLaunchKernelGGL(k_pass1_slab, dim3(nblocks), dim3(256), lds_bytes, s, B, cstart, sx, aux, outm, shellm, negm, zerom,
                           tflag, tmark, clear, nclear);
}

void qs_launch_pass1_direct(QsBatch B, uint32_t nblocks, const int2 *cse, const float4 *sx, uint64_t *outm, uint64_t *shellm,
                            hipStream_t s)
{
    hipLaunchKernelGGL(k_pass1_direct, dim3(nblocks), dim3(256), 0, s, B, cse, sx, outm, shellm);
}

/* field pass 2 kernel choice for half-window r: 0 fixed-R kernel (r <= 9), 1 runtime-r tile
   kernel, 2 direct window */
int qs_pass2_path(int r, bool direct)
{
    if (direct) return 2;
    if (r >= 1 && r <= 9) return 0;
    if (qs_pass2_lds_bytes(r) <= 65536 && 2 * r + P2_TZ <= 64) return 1;
    return 2;
}

uint32_t qs_pass2_blocks(const QsMol &M, int path)
{
    const QsGrid &G = M.G;
    const uint32_t nx = (uint32_t)std::max(M.p2_hi - M.p2_lo, 0);
    if (path == 2) return nblk(G.g, 64) * nblk(G.g, 4) * nx;
    return nblk(G.g, P2_TZ) * nblk(G.g, P2_TY) * nblk(nx, path == 0 ? P2R_TX : P2_TX);
}

/* one launch for a group of molecules sharing r (and so the path) */
void qs_launch_pass2(QsBatch B, uint32_t nblocks, int r, int path, const uint64_t *outm, const uint64_t *shellm,
                     float *field, uint32_t *negm, uint32_t *zerom, const int *offs, const int *norm_start, const int *enum_end,
                     QsNormFlags nf, QsBand band, const uint8_t *tflag, uint8_t tmark, uint32_t xchunk, hipStream_t s)
{
    if (path == 0) {
        xchunk = std::max(xchunk, 1u);
#define QS_P2R(RR)                                                                                                    \
    case RR:                                                                                                          \
        hipLaunchKernelGGL(k_pass2_r<RR>, dim3(nblocks), dim3(256), 0, s, B, outm, shellm, field, negm, zerom, \
                           offs, norm_start, enum_end, nf, band, tflag, tmark, xchunk);                                            \
        return;
        switch (r) {
            QS_P2R(1)
            QS_P2R(2)
            QS_P2R(3)
            QS_P2R(4)
            QS_P2R(5)
            QS_P2R(6)
            QS_P2R(7)
            QS_P2R(8)
            QS_P2R(9)
        default:
            break;
        }
#undef QS_P2R
    }
    if (path <= 1) {
        hipLaunchKernelGGL(k_pass2_tile<uint16_t>, dim3(nblocks), dim3(256), qs_pass2_lds_bytes(r), s, B, outm, shellm,
                           field, negm, zerom, offs, norm_start, enum_end);
        return;
    }
    hipLaunchKernelGGL(k_pass2_direct, dim3(nblocks), dim3(256), 0, s, B, outm, shellm, field, negm, zerom);
}

void qs_launch_labels_to_masks(const uint8_t *labels, int g, int W, uint64_t *outm, uint64_t *shellm, hipStream_t s)
{
    dim3 grid((unsigned)W, nblk(g, 4), (unsigned)g);
    hipLaunchKernelGGL(k_labels_to_masks, grid, dim3(256), 0, s, labels, g, W, outm, shellm);
}

uint32_t qs_mc_count_blocks(const QsMol &M)
{
    return nblk((uint64_t)M.G.g * M.W, 256) * (uint32_t)std::max(M.mc_hi - M.mc_lo, 0);
}

void qs_launch_mc_count(QsBatch B, uint32_t nblocks, const uint64_t *N, const uint64_t *Zm, uint64_t *S4, uint32_t *cnt,
                        uint64_t *NT, uint32_t *sums, uint64_t scan_w0, hipStream_t s)
{
    hipLaunchKernelGGL(k_mc_count, dim3(nblocks), dim3(256), 0, s, B, N, Zm, S4, cnt, NT, sums, scan_w0);
}

void qs_launch_mc_emit(const QsMol *mols, const uint64_t *wpre, const uint32_t *wcoarse, const uint32_t *list, uint32_t nact,
                       const uint32_t *avb, uint32_t *vstart, uint32_t nv, const uint64_t *S4, const float *F,
                       const uint64_t *outm, const uint64_t *shellm, float *vert, uint64_t *vkey,
                       const uint32_t *acb, uint32_t *tstart, uint32_t ncube, uint32_t ntri, const uint64_t *N, const uint32_t *cnt,
                       const uint32_t *vbw, const uint32_t *tbw, const uint64_t *NT, int *tri, uint32_t vbase, uint32_t *deg_blk,
                       uint32_t *deg_total, const uint32_t *d_counts, hipStream_t s, const QsClosest *atoms, bool starts_ready,
                       uint32_t block_items)
{
    if (!nact || (!nv && !ntri)) return;
    /* the per-block degenerate counts start at zero (the triangle kernel adds to them), over the
       whole pool of ntri triangles */
    const uint32_t nzero = ntri ? ntri / 256 + 1 : 0u;
    const QsStarts sv = {avb, nv, d_counts ? d_counts + 1 : nullptr, vstart, nullptr, 0u};
    const QsStarts st = {acb, ncube, d_counts ? d_counts + 4 : nullptr, tstart, deg_blk, nzero};
    if (!starts_ready)
        hipLaunchKernelGGL(k_block_starts, dim3(pgrid(nblk(std::max<uint32_t>(nact, nzero), 256)), 2), dim3(256), 0, s, sv, st,
                           nact, d_counts ? d_counts + 2 : nullptr);
    const unsigned gv = nv ? pgrid(nblk(std::min(nv, block_items), 256)) : 0u,
                   gt = ntri ? pgrid(nblk(std::min(ncube, block_items), 256)) : 0u;
    if (atoms && gv && gt) {
        hipLaunchKernelGGL((k_mc_emit<true, true, true>), dim3(gv + gt), dim3(256), 0, s, mols, wpre, wcoarse, list, avb,
                                                                                          vstart, nact, nv, S4, F, outm, shellm,
                                                                                          vert, vkey, d_counts, acb, tstart,
                                                                                          ncube, ntri, N, cnt, vbw, tbw, NT,
                                                                                          tri, vbase, deg_blk, deg_total,
                                                                                          *atoms, gv);
        return;
    }
    if (gv && atoms)
        hipLaunchKernelGGL((k_mc_emit<true, false, true>), dim3(gv), dim3(256), 0, s, mols, wpre, wcoarse, list, avb, vstart,
                                                                                      nact, nv, S4, F, outm, shellm, vert, vkey,
                                                                                      d_counts, acb, tstart, ncube, ntri, N,
                                                                                      cnt, vbw, tbw, NT, tri, vbase, deg_blk,
                                                                                      deg_total, *atoms, 0u);
    else if (gv)
        hipLaunchKernelGGL((k_mc_emit<true, false, false>), dim3(gv), dim3(256), 0, s, mols, wpre, wcoarse, list, avb, vstart,
                                                                                       nact, nv, S4, F, outm, shellm, vert,
                                                                                       vkey, d_counts, acb, tstart, ncube, ntri,
                                                                                       N, cnt, vbw, tbw, NT, tri, vbase,
                                                                                       deg_blk, deg_total, QsClosest{}, 0u);
    if (gt)
        hipLaunchKernelGGL((k_mc_emit<false, true, false>), dim3(gt), dim3(256), 0, s, mols, wpre, wcoarse, list, avb, vstart,
                                                                                       nact, nv, S4, F, outm, shellm, vert,
                                                                                       vkey, d_counts, acb, tstart, ncube, ntri,
                                                                                       N, cnt, vbw, tbw, NT, tri, vbase,
                                                                                       deg_blk, deg_total, QsClosest{}, 0u);
}

void qs_launch_smooth(const QsMol *mols, const uint32_t *vpre, const uint32_t *vcoarse, const uint64_t *wpre, const uint32_t *wcoarse,
                      const uint32_t *list, const uint32_t *vstart, const uint64_t *N, const uint64_t *Zm, const uint64_t *S4,
                      const uint32_t *vbw, const uint64_t *vkey, uint32_t nv, uint32_t ntri, const uint64_t *NT,
                      const uint32_t *tbw, const int *tri, const float *src, float *dst, const uint32_t *d_counts, uint32_t expect,
                      uint32_t block_items, const QsCompact *compact, hipStream_t s)
{
    if (!nv) return;
    const dim3 grid(pgrid(nblk(std::min(nv, block_items), 256)));
    if (compact) {
        const unsigned nbs = grid.x, nbc = std::max(1u, std::min(nblk(ntri, 256), COMPACT_BLOCKS));
        hipLaunchKernelGGL((k_smooth<false, true>), dim3(nbs + nbc), dim3(256), 0, s, mols, vpre, vcoarse, wpre, wcoarse, list, vstart,
                           N, Zm, S4, vbw, vkey, nv, ntri, NT, tbw, tri, src, dst, d_counts, *compact, nbs);
    } else if (std::min(nv, expect) > SM_STAGED_MIN) {
        hipLaunchKernelGGL((k_smooth<true, false>), grid, dim3(256), 0, s, mols, vpre, vcoarse, wpre, wcoarse, list, vstart, N, Zm, S4,
                           vbw, vkey, nv, ntri, NT, tbw, tri, src, dst, d_counts, QsCompact{}, 0u);
    } else {
        hipLaunchKernelGGL((k_smooth<false, false>), grid, dim3(256), 0, s, mols, vpre, vcoarse, wpre, wcoarse, list, vstart, N, Zm,
                           S4, vbw, vkey, nv, ntri, NT, tbw, tri, src, dst, d_counts, QsCompact{}, 0u);
    }
}

void qs_launch_vertex_normals(const QsMol *mols, const uint32_t *vpre, const uint32_t *vcoarse, const uint64_t *vkey, uint32_t nv,
                              const float *F, const uint64_t *outm, const uint64_t *shellm, float *out,
                              hipStream_t s)
{
    if (!nv) return;
    hipLaunchKernelGGL(k_vertex_normals, dim3(nblk(nv, 256)), dim3(256), 0, s, mols, vpre, vcoarse, vkey, nv, F, outm, shellm,
                       out);
}

void qs_launch_vertex_colors(const QsMol *mols, const uint32_t *vpre, const uint32_t *vcoarse, const int *atom,
                             const int *perm, uint32_t nv, const float4 *table, float4 *out, hipStream_t s)
{
    if (!nv) return;
    hipLaunchKernelGGL(k_vertex_colors, dim3(nblk(nv, 256)), dim3(256), 0, s, mols, vpre, vcoarse, atom, perm, nv, table,
                       out);
}

void qs_launch_closest_atom(const QsMol *mols, const uint32_t *vpre, const uint32_t *vcoarse, const QsClosest &A,
                            const float *vert, uint32_t nv, const uint32_t *d_nv, uint32_t block_items, hipStream_t s)
{
    if (!nv) return;
    hipLaunchKernelGGL(k_closest_atom, dim3(pgrid(nblk(std::min(nv, block_items), 256))), dim3(256), 0, s, mols, vpre, vcoarse, vert, nv,
                       d_nv, A);
}

size_t qs_cells_lds_bytes(const QsMol &m)
{
    const uint64_t ncell = (uint64_t)m.G.gn * m.G.gn * m.G.gn;
    if (m.n_atoms > CELLS_ATOMS || ncell > CELLS_MAX) return 0;
    return ((size_t)ncell / 2 + 1) * 4 + ((size_t)m.n_atoms * 2 + 3) / 4 * 4;
}

void qs_launch_cells(const QsMol *mols, int nmol, const QsMol *one, size_t lds, bool gather, const float *pos, const float *rad, uint32_t *start,
                     int *perm, int2 *cse, float4 *sx, float4 *aux, hipStream_t s)
{
    QsMol *const put = one ? (QsMol *)mols : nullptr;
    const QsMol m = one ? *one : QsMol{};
    if (gather)
        hipLaunchKernelGGL((k_cells<CELLS_GATHER / CELLS_NT, true>), dim3(nmol), dim3(CELLS_NT), lds, s, mols, m, put, pos, rad,
                           start, perm, cse, sx, aux);
    else
        hipLaunchKernelGGL((k_cells<CELLS_ATOMS / CELLS_NT, false>), dim3(nmol), dim3(CELLS_NT), lds, s, mols, m, put, pos, rad,
                           start, perm, cse, sx, aux);
}

void qs_launch_put_mol(const QsMol &m, QsMol *dst, uint32_t *clear, uint32_t n, hipStream_t s)
{
    hipLaunchKernelGGL(k_put_mol, dim3(std::min(std::max(nblk(n, 1024), 1u), 512u)), dim3(256), 0, s, m, dst, clear, n);
}

void qs_launch_copy(const void *src, void *dst, uint64_t bytes, hipStream_t s)
{
    const uint64_t n16 = bytes / 16;
    if (!n16) return;
    const uint64_t blocks = std::min<uint64_t>((n16 + 255) / 256, 8192);
    hipLaunchKernelGGL(k_copy, dim3((unsigned)blocks), dim3(256), 0, s, (const uint4 *)src, (uint4 *)dst, n16);
}

void qs_launch_copy_mesh(const float *v, const int *a, const int *t, uint32_t nv, uint32_t nt, uint32_t v0, float *dv, int *da,
                         int *dt, hipStream_t s)
{
    const size_t items = 4 * (size_t)nv + 3 * (size_t)nt;
    if (!items) return;
    hipLaunchKernelGGL(k_copy_mesh, dim3((unsigned)std::min<size_t>((items / 4 + 255) / 256 + 1, 2048)), dim3(256), 0, s,
                       (const uint32_t *)v, (const uint32_t *)a, (const uint32_t *)t, nv, nt, v0, (uint32_t *)dv, (uint32_t *)da,
                       (uint32_t *)dt);
}

void qs_launch_tri_localize(const int *tri, uint32_t nt, const uint32_t *tpre, const uint32_t *vpre, int nmol, int *out,
                            hipStream_t s)
{
    if (nt == 0) return;
    hipLaunchKernelGGL(k_tri_localize, dim3(nblk(nt, 256)), dim3(256), 0, s, tri, nt, tpre, vpre, nmol, out);
}

void qs_launch_tri_compact(const int *tri, uint32_t nt, const uint32_t *dpre, const uint32_t *totals, int *out,
                           const uint32_t *d_nt, hipStream_t s)
{
    if (!nt) return;
    hipLaunchKernelGGL(k_tri_compact<false>, dim3(std::min(nblk(nt, 256), COMPACT_BLOCKS)), dim3(256), 0, s, tri, nt, dpre, totals,
                       out, d_nt, 0, 0u, (uint32_t *)nullptr, (uint32_t *)nullptr, (uint32_t *)nullptr);
}

void qs_launch_tri_compact_one(const int *tri, uint32_t nt, const uint32_t *dpre, bool self, const uint32_t *totals, int *out,
                               const uint32_t *d_nt, uint32_t nv, uint32_t *vpre, uint32_t *kept, uint32_t *rb, hipStream_t s)
{
    hipLaunchKernelGGL(k_tri_compact<true>, dim3(std::max(1u, std::min(nblk(nt, 256), COMPACT_BLOCKS))), dim3(256), 0, s, tri, nt,
                       dpre, totals, out, d_nt, self ? 1 : 0, nv, vpre, kept, rb);
}

void qs_launch_tri_kept_before(const int *tri, const uint32_t *dpre, const uint64_t *idx, int n, uint32_t tcap, uint32_t *out,
                               const uint32_t *totals, const uint32_t *vpre, uint32_t *rb, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_tri_kept_before, dim3(nblk(n, 4)), dim3(256), 0, s, tri, dpre, idx, n, tcap, out, totals, vpre, rb);
}

/* scan helpers */
void qs_launch_mc_scans(const uint32_t *cnt, uint64_t nw, uint32_t *sums, uint32_t *vbw,
                        uint32_t *tbw, uint32_t *list, uint32_t *avb, uint32_t *acb, uint32_t *totals, uint32_t list_base,
                        hipStream_t s, QsBlockStarts bs)
{
    if (!nw) return;
    const uint64_t ntiles = qs_scan_tiles(nw);
    const int self = ntiles <= QS_SCAN_SELF_TILES;
    if (!self) hipLaunchKernelGGL(k_scan_planes, dim3(4), dim3(SCAN_NT), 0, s, sums, ntiles, totals);
    hipLaunchKernelGGL(k_mc_scan4, dim3((unsigned)ntiles), dim3(SCAN_NT), 0, s, cnt, nw, sums, vbw, tbw, list,
                       avb, acb, list_base, self, totals, bs);
}

uint64_t qs_scan_tiles(uint64_t n) { return (n + SCAN_TILE - 1) / SCAN_TILE; }

void qs_launch_tile_reduce(const uint32_t *in, uint64_t n, uint32_t *sums, hipStream_t s)
{
    hipLaunchKernelGGL(k_tile_reduce, dim3((unsigned)qs_scan_tiles(n)), dim3(SCAN_NT), 0, s, in, n, sums);
}

void qs_launch_scan1(const uint32_t *in, uint32_t *out, uint64_t n, uint32_t *total, hipStream_t s)
{
    hipLaunchKernelGGL(k_scan1, dim3(1), dim3(SCAN1_NT), 0, s, in, out, n, total);
}

void qs_launch_tile_scan(const uint32_t *in, uint32_t *out, uint64_t n, const uint32_t *offsets, uint32_t *total,
                         hipStream_t s, const uint32_t *self_sums)
{
    hipLaunchKernelGGL(k_tile_scan, dim3((unsigned)qs_scan_tiles(n)), dim3(SCAN_NT), 0, s, in, out, n, offsets, total,
                       self_sums);
}

void qs_launch_smooth_incid_build(const int *tri, uint32_t nt, uint32_t nv, uint32_t *cnt, uint32_t *start, uint32_t *ent,
                                  hipStream_t s)
{
    const uint64_t nc = 3 * (uint64_t)nt;
    if (!nc || !nv) return;
    /* start[] (nv + 1 entries) holds the exclusive prefix of cnt[]; cnt[] is reused as the fill
       cursors, so the caller clears it between the scan and this fill */
    hipLaunchKernelGGL(k_incid_fill, dim3(nblk(nc, 256)), dim3(256), 0, s, tri, nc, nv, start, cnt, ent);
    hipLaunchKernelGGL(k_incid_sort, dim3(nblk(nv, 256)), dim3(256), 0, s, start, nv, ent);
}

void qs_launch_incid_count(const int *tri, uint32_t nt, uint32_t nv, uint32_t *cnt, hipStream_t s)
{
    const uint64_t nc = 3 * (uint64_t)nt;
    if (!nc || !nv) return;
    hipLaunchKernelGGL(k_incid_count, dim3(nblk(nc, 256)), dim3(256), 0, s, tri, nc, nv, cnt);
}

void qs_launch_smooth_incid(const uint32_t *start, const uint32_t *ent, const int *tri, uint32_t nv, const float *src,
                            float *dst, hipStream_t s)
{
    if (!nv) return;
    hipLaunchKernelGGL(k_smooth_incid, dim3(nblk(nv, 256)), dim3(256), 0, s, start, ent, tri, nv, src, dst);
}

void qs_launch_deg_count(const int *tri, uint32_t nt, uint32_t *deg_blk, uint32_t *deg_total, hipStream_t s)
{
    if (!nt) return;
    hipLaunchKernelGGL(k_deg_count, dim3(nblk(nt, 256)), dim3(256), 0, s, tri, nt, deg_blk, deg_total);
}

void qs_launch_mesh_bases(const uint32_t *vbw, const uint32_t *tbw, const uint64_t *wpre, uint64_t nw, int nmol,
                          const uint32_t *counts, uint32_t *vpre, uint64_t *tpre, uint32_t *vcoarse, uint32_t ncoarse, hipStream_t s)
{
    hipLaunchKernelGGL(k_mesh_bases, dim3(nblk(std::max<uint64_t>((uint64_t)nmol + 1, ncoarse), 256)), dim3(256), 0, s, vbw, tbw,
                       wpre, nw, nmol, counts, vpre, tpre, vcoarse, ncoarse);
}

uint32_t qs_pass2_tiles(const QsMol &M) { return qs_pass2_blocks(M, 0); }
uint32_t qs_pass2_ztiles(const QsMol &M) { return (uint32_t)((M.G.g + P2_TZ - 1) / P2_TZ); }
