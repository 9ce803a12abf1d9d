// Point cloud -> voxels with up to max_points points each, replacing the sequential CPU loop of
// points_to_voxel_3d (include/point2voxel.h:412-512, called from sphconv/utils/voxelize.py:126-214)
// and the coordinate transforms of sphconv/utils/coord_transform.py:8-118.
//
// The reference walks the points in order: a point outside the grid is skipped; a point in a
// new cell opens the next voxel, unless max_voxels are open already -- then the whole loop
// stops; a voxel keeps its first max_points points.  The same result without the sequential
// loop:
//   1. vox_clear_kernel    zeroes the outputs and resets the workspace (one launch)
//   2. vox_insert_kernel   system coordinates (float32, operation by operation as numpy does it) and
//                          the cell of every point; the cells of a workgroup's points meet in a table in LDS, and each
//                          of them enters a hash table (open addressing, at most half full), with the number of its
//                          points and the smallest of their indices (atomic sum and minimum)
//   3. one scan            over the points: those that open a cell count as one voxel and as their cell's number of
//                          points, so the sums in front of one are its voxel number and the start of its cell's segment
//                          of the point list; they go to the cell's record.  The point that would open voxel number
//                          max_voxels is where the reference's loop stops: every later point is dropped
//   4. vox_scatter_kernel  writes every point into its cell's segment (in any order)
//   5. vox_write_kernel    a point's place in its voxel = the number of smaller point indices in its
//                          segment (counted until max_points are found: such a point is dropped);
//                          segments of more than 256 points are walked by the whole wave, 64 entries at a time
// Which slot a cell gets, and the order inside a segment, depend on the order the atomics land in;
// no output does.  Nothing is allocated; table, segments and the scan's state live in the caller's workspace.
#include "common.h"

#include <cstring>

#include "scan.h"

namespace {

enum { SYS_SPHERICAL = 0, SYS_LSPHERICAL, SYS_CYLINDER, SYS_LCYLINDER, SYS_HYBRID, SYS_LHYBRID, SYS_COUNT };

struct VoxParams {
    int system, nfeat, append_mode, max_points, max_voxels;
    float lo[3], vs[3];   // lower bound and voxel size per system coordinate
    int grid[3];
    unsigned long long cells;
};

// (c0, c1, c2) of a point in the chosen system; every operation rounded to float32 on its own
__device__ __forceinline__ void system_coords(const float *p, int system, float (&c)[3])
{
    const float x = p[0], y = p[1], z = p[2];
    const float x2y2 = __fadd_rn(__fmul_rn(x, x), __fmul_rn(y, y));
    const float d = __fsqrt_rn(x2y2);
    const float phi = asinf(__fdiv_rn(y, d));
    c[1] = phi;
    if (system == SYS_CYLINDER || system == SYS_LCYLINDER) {
        c[0] = system == SYS_CYLINDER ? d : logf(d);
        c[2] = z;
        return;
    }
    const float r = __fsqrt_rn(__fadd_rn(x2y2, __fmul_rn(z, z)));
    c[2] = acosf(__fdiv_rn(z, r));
    switch (system) {
    case SYS_SPHERICAL: c[0] = r; break;
    case SYS_LSPHERICAL: c[0] = logf(r); break;
    case SYS_HYBRID: c[0] = d; break;
    default: c[0] = logf(d); break;
    }
}

// bins (idx of c0, c1, c2) or false if the point is outside the grid (point2voxel.h:447-457)
__device__ __forceinline__ bool cell_of(const float (&c)[3], const VoxParams &q, int (&bin)[3])
{
    bool ok = true;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const float f = floorf(__fdiv_rn(__fsub_rn(c[i], q.lo[i]), q.vs[i]));
        ok = ok && f >= 0.f && f < (float)q.grid[i]; // false for NaN
        bin[i] = ok ? (int)f : 0;
    }
    return ok;
}

// cell of point i as the table's key, or `cells` for a point that is skipped
__device__ __forceinline__ uint64_t point_cell(const float *points, int i, const VoxParams &q, const long long *cell_in)
{
    if (cell_in) {
        const long long c = cell_in[i];
        return c >= 0 && (unsigned long long)c < q.cells ? (uint64_t)c : (uint64_t)q.cells;
    }
    float c[3];
    int bin[3];
    system_coords(points + (long)i * q.nfeat, q.system, c);
    // the reference indexes its map [c2 bin][c1 bin][c0 bin]
    if (cell_of(c, q, bin)) return ((uint64_t)bin[2] * q.grid[1] + bin[1]) * q.grid[0] + bin[0];
    return q.cells;
}

constexpr uint64_t kEmptyKey = ~0ull;
constexpr int kFills = 10;
constexpr int kFillBlocks = 128;  // workgroups per range
constexpr int kLongSegment = 256; // longer segments are walked by the wave together

// up to kFills ranges of 32-bit words, each set to its value (or to two values in turn: an even number of words, aligned
// to 16 bytes): blockIdx.y = range
struct VoxFills {
    int32_t *p[kFills];
    long words[kFills];
    int32_t value[kFills], odd_value[kFills];
};

__global__ __launch_bounds__(256) void vox_clear_kernel(VoxFills f)
{
    int32_t *p = f.p[blockIdx.y];
    const long n = f.words[blockIdx.y];
    const int32_t v = f.value[blockIdx.y], w = f.odd_value[blockIdx.y];
    const long t = (long)blockIdx.x * 256 + threadIdx.x, step = (long)gridDim.x * 256;
    if (((uintptr_t)p & 15) == 0) {
        const int4 v4 = make_int4(v, w, v, w);
        for (long i = t; i < n / 4; i += step) ((int4 *)p)[i] = v4;
        if (t < (n & 3)) p[(n & ~3L) + t] = (t & 1) ? w : v;
    } else {
        for (long i = t; i < n; i += step) p[i] = v;
    }
}

// tbits = log2 of the table's slots.  slot_place[i]: the point's slot (-1: outside the grid) and its place in the slot's
// segment, the places given in the order of arrival: from the front (>= 0) to the points of the workgroup that brought the
// cell, from the back (-1, -2, ...) to all others.
// Device-wide atomics bound it (about 24 per ns over the chip), so there are few: what a workgroup's points have in common
// is settled in LDS, and the workgroup that brings a cell needs one, the compare-and-swap, and stores its points' number
// and smallest index where nobody else does (`brought`); the others add to `later` (smallest index, number).  123 k points
// in 24 k cells: 17.4 us with three atomics per point, 13.6 us this way.
constexpr int kInsertThreads = 512, kInsertSlots = 1024; // (at most half full too)
__global__ __launch_bounds__(kInsertThreads) void vox_insert_kernel(const float *points, int n, VoxParams q, const long long *cell_in,
                                                                    int tbits, unsigned long long *keys, int2 *brought,
                                                                    int2 *later, int2 *slot_place, long long *cell_out)
{
    __shared__ unsigned long long s_key[kInsertSlots];
    __shared__ int s_first[kInsertSlots], s_count[kInsertSlots], s_slot[kInsertSlots], s_base[kInsertSlots];
    const int i = blockIdx.x * kInsertThreads + threadIdx.x;
    for (int e = threadIdx.x; e < kInsertSlots; e += kInsertThreads) {
        s_key[e] = kEmptyKey;
        s_first[e] = INT_MAX;
        s_count[e] = 0;
    }
    __syncthreads();
    const uint64_t key = i < n ? point_cell(points, i, q, cell_in) : (uint64_t)q.cells;
    if (cell_out && i < n) cell_out[i] = key == q.cells ? -1 : (long long)key;
    const bool inside = key != q.cells;
    const uint64_t hash = key * 0x9E3779B97F4A7C15ull;
    int e = 0, place = 0;
    bool opens = false; // the first of the workgroup's points to bring this cell
    if (inside) {
        e = (int)(hash >> (64 - 10));
        for (;;) {
            const unsigned long long seen = atomicCAS(&s_key[e], (unsigned long long)kEmptyKey, (unsigned long long)key);
            opens = seen == kEmptyKey;
            if (opens || seen == key) break;
            e = (e + 1) & (kInsertSlots - 1);
        }
        place = atomicAdd(&s_count[e], 1);
        atomicMin(&s_first[e], i);
    }
    __syncthreads();
    if (opens) {
        const unsigned mask = (1u << tbits) - 1u;
        unsigned slot = (unsigned)(hash >> (64 - tbits));
        unsigned long long seen;
        // the table has at least twice as many slots as there are points: a free one is always met
        for (;;) {
            seen = atomicCAS(&keys[slot], (unsigned long long)kEmptyKey, (unsigned long long)key);
            if (seen == kEmptyKey || seen == key) break;
            slot = (slot + 1) & mask;
        }
        if (seen == kEmptyKey) {
            brought[slot] = make_int2(s_first[e], s_count[e]);
            s_base[e] = -1;
        } else {
            atomicMin(&later[slot].x, s_first[e]);
            s_base[e] = atomicAdd(&later[slot].y, s_count[e]);
        }
        s_slot[e] = (int)slot;
    }
    __syncthreads();
    if (i < n) slot_place[i] = inside ? make_int2(s_slot[e], s_base[e] < 0 ? place : ~(s_base[e] + place)) : make_int2(-1, 0);
}

// What the scan reads: per point that opens a cell one voxel (upper half) and the cell's points (lower 30 bits).
constexpr int kPairShift = 30;
constexpr int kPointItems = 4; // points per thread of the scan
struct OpenedCells {
    const int2 *brought, *later, *slot_place;
    __device__ __forceinline__ unsigned long long operator()(long i) const
    {
        const int s = slot_place[i].x;
        if (s < 0) return 0ull;
        const int2 b = brought[s], l = later[s];
        return min(b.x, l.x) == (int)i ? (1ull << kPairShift) + (unsigned)(b.y + l.y) : 0ull;
    }
};
// ... and where the sums go: rec[slot] = (first and last + 1 of its segment, its voxel number, the point that opened it)
struct CellRecords {
    const int2 *slot_place;
    int4 *rec;
    int32_t *stop, *voxel_num;
    int max_voxels;
    template <int ITEMS>
    __device__ __forceinline__ void tile(long base, long, unsigned long long before, const unsigned long long (&incl)[ITEMS]) const
    {
        constexpr unsigned long long kLow = (1ull << kPairShift) - 1;
#pragma unroll
        for (int j = 0; j < ITEMS; j++) {
            const unsigned long long excl = j ? incl[j - 1] : before;
            if (incl[j] == excl) continue;
            const int i = (int)(base + j), vid = (int)(excl >> kPairShift);
            rec[slot_place[i].x] = make_int4((int)(excl & kLow), (int)(incl[j] & kLow), vid, i);
            if (vid == max_voxels) *stop = i; // exactly one such point, if any
        }
    }
    __device__ __forceinline__ void all(unsigned long long sum) const { *voxel_num = min((int)(sum >> kPairShift), max_voxels); }
};

__global__ __launch_bounds__(256) void vox_scatter_kernel(const int2 *slot_place, const int4 *rec, int n, int32_t *seg)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int2 sp = slot_place[i];
    if (sp.x < 0) return;
    const int4 r = rec[sp.x];
    seg[(sp.y >= 0 ? r.x : r.y) + sp.y] = i;
}

__global__ __launch_bounds__(256) void vox_write_kernel(const float *points, int n, VoxParams q, const unsigned long long *keys,
                                                        const int2 *slot_place, const int4 *rec, const int32_t *seg,
                                                        const int32_t *stop, float *voxels, float *mask, int32_t *coors,
                                                        int32_t *num_points)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const int s = i < n ? slot_place[i].x : -1;
    int vid = 0, h = 0, s0 = 0, s1 = 0;
    bool live = s >= 0;
    if (live) {
        const int4 r = rec[s];
        s0 = r.x; s1 = r.y; vid = r.z; h = r.w;
        live = vid < q.max_voxels && i < *stop;
    }
    // place among the cell's points = smaller indices in the segment
    int rank = 0;
    const bool wide = live && s1 - s0 > kLongSegment;
    if (live && !wide)
        for (int p = s0; p < s1 && rank < q.max_points; p++) rank += seg[p] < i;
    for (unsigned long long todo = __ballot(wide); todo; todo &= todo - 1) {
        const int l = __ffsll((long long)todo) - 1;
        const int ti = __shfl(i, l, 64), t1 = __shfl(s1, l, 64);
        int r = 0;
        for (int p = __shfl(s0, l, 64); p < t1 && r < q.max_points; p += 64)
            r += __popcll(__ballot(p + lane < t1 && seg[p + lane] < ti));
        if (lane == l) rank = r;
    }
    if (!live || rank >= q.max_points) return;
    if (i == h) {
        const uint64_t key = keys[s];
        const uint64_t t = key / q.grid[0];
        coors[3 * (long)vid] = (int)(t / q.grid[1]);       // c2 bin
        coors[3 * (long)vid + 1] = (int)(t % q.grid[1]);   // c1 bin
        coors[3 * (long)vid + 2] = (int)(key % q.grid[0]); // c0 bin
    }
    const int width = q.append_mode == 1 ? q.nfeat + 3 : q.nfeat;
    float *dst = voxels + ((long)vid * q.max_points + rank) * width;
    const float *p = points + (long)i * q.nfeat;
    if (q.append_mode == 2) {
        float c[3];
        system_coords(p, q.system, c);
        dst[0] = c[0]; dst[1] = c[1]; dst[2] = c[2]; dst[3] = p[3];
    } else {
        for (int f = 0; f < q.nfeat; f++) dst[f] = p[f];
        if (q.append_mode == 1) {
            float c[3];
            system_coords(p, q.system, c);
            dst[q.nfeat] = c[0]; dst[q.nfeat + 1] = c[1]; dst[q.nfeat + 2] = c[2];
        }
    }
    mask[(long)vid * q.max_points + rank] = 1.f;
    atomicMax(&num_points[vid], rank + 1);
}

struct VoxLayout {
    int tbits;
    long T; // slots of the table: a power of two, at least twice the points
    size_t keys, later, brought, rec, slot_place, seg, stop, state, state_words, total;
};

inline size_t al256(size_t x) { return (x + 255) & ~(size_t)255; }

inline VoxLayout vox_layout(int n)
{
    VoxLayout l;
    const size_t nn = (size_t)(n > 0 ? n : 1);
    l.tbits = 10;
    while ((1ull << l.tbits) < 2 * nn) l.tbits++;
    l.T = 1L << l.tbits;
    size_t o = 0;
    l.keys = o; o += al256((size_t)l.T * 8);
    l.later = o; o += al256((size_t)l.T * 8);
    l.brought = o; o += al256((size_t)l.T * 8);
    l.rec = o; o += al256((size_t)l.T * 16);
    l.slot_place = o; o += al256(nn * 8);
    l.seg = o; o += al256(nn * 4);
    l.stop = o; o += 256;
    l.state = o;
    l.state_words = (size_t)sph_scan::state_ints((long)nn, kPointItems);
    o += al256(sph_scan::state_bytes((long)nn, kPointItems));
    l.total = o;
    return l;
}

inline unsigned blocks(long n) { return (unsigned)((n + 255) / 256); }

} // namespace

SPH_EXPORT size_t sph_points_to_voxel_workspace(int n, int g0, int g1, int g2)
{
    if (n < 0 || n > (1 << 29) || g0 <= 0 || g1 <= 0 || g2 <= 0) return 0;
    return vox_layout(n).total;
}

SPH_EXPORT int sph_points_to_voxel(const float *points, int n, int nfeat, int system, float lo0, float lo1, float lo2,
                                   float vs0, float vs1, float vs2, int g0, int g1, int g2, int max_points,
                                   int max_voxels, int append_mode, float *voxels, float *mask, int32_t *coors,
                                   int32_t *num_points, int32_t *voxel_num, const long long *cell_in,
                                   long long *cell_out, void *workspace, size_t workspace_bytes, void *stream)
{
    SPH_REQUIRE(n >= 0 && n <= (1 << 29) && nfeat >= 4 && max_points > 0 && max_voxels > 0 && g0 > 0 && g1 > 0 && g2 > 0,
                SPH_ERR_ARG, "sph_points_to_voxel: bad sizes (points need x, y, z, intensity; at most 2^29 points)");
    SPH_REQUIRE(system >= 0 && system < SYS_COUNT && append_mode >= 0 && append_mode <= 2, SPH_ERR_ARG,
                "sph_points_to_voxel: unknown coordinate system %d or append mode %d", system, append_mode);
    SPH_REQUIRE(vs0 != 0.f && vs1 != 0.f && vs2 != 0.f, SPH_ERR_ARG, "sph_points_to_voxel: empty range");
    SPH_REQUIRE(voxels && mask && coors && num_points && voxel_num && workspace && (n == 0 || points), SPH_ERR_ARG,
                "sph_points_to_voxel: null pointer");
    SPH_REQUIRE((uintptr_t)workspace % 256 == 0, SPH_ERR_ARG, "sph_points_to_voxel: workspace must be 256-byte aligned");
    VoxParams q;
    q.system = system; q.nfeat = nfeat; q.append_mode = append_mode; q.max_points = max_points; q.max_voxels = max_voxels;
    q.lo[0] = lo0; q.lo[1] = lo1; q.lo[2] = lo2; q.vs[0] = vs0; q.vs[1] = vs1; q.vs[2] = vs2;
    q.grid[0] = g0; q.grid[1] = g1; q.grid[2] = g2;
    q.cells = (unsigned long long)g0 * g1 * g2;
    SPH_REQUIRE(q.cells / g0 / g1 == (unsigned long long)g2 && q.cells < (1ull << 63), SPH_ERR_ARG,
                "sph_points_to_voxel: grid %d x %d x %d has too many cells", g0, g1, g2);
    const VoxLayout l = vox_layout(n);
    SPH_REQUIRE(workspace_bytes >= l.total, SPH_ERR_ARG, "sph_points_to_voxel: workspace of %zu bytes, %zu needed",
                workspace_bytes, l.total);
    hipStream_t st = (hipStream_t)stream;
    char *ws = (char *)workspace;
    unsigned long long *keys = (unsigned long long *)(ws + l.keys);
    int2 *later = (int2 *)(ws + l.later), *brought = (int2 *)(ws + l.brought);
    int32_t *seg = (int32_t *)(ws + l.seg), *stop = (int32_t *)(ws + l.stop);
    int2 *slot_place = (int2 *)(ws + l.slot_place);
    int4 *rec = (int4 *)(ws + l.rec);

    const int width = append_mode == 1 ? nfeat + 3 : nfeat;
    const long nv = (long)max_voxels * max_points;
    VoxFills f;
    int nf = 0;
    auto fill_pairs = [&](void *p, long pairs, int32_t v, int32_t w) {
        f.p[nf] = (int32_t *)p; f.words[nf] = 2 * pairs; f.value[nf] = v; f.odd_value[nf] = w;
        nf++;
    };
    auto fill = [&](void *p, long words, int32_t v) {
        f.p[nf] = (int32_t *)p; f.words[nf] = words; f.value[nf] = f.odd_value[nf] = v;
        nf++;
    };
    fill(voxels, nv * width, 0);
    fill(mask, nv, 0);
    fill(coors, 3L * max_voxels, 0);
    fill(num_points, (long)max_voxels, 0);
    if (n == 0) fill(voxel_num, 1L, 0); // else it is written once, by the scan: the host may be watching it
    if (n > 0) {
        fill(keys, 2 * l.T, -1);
        fill_pairs(later, l.T, INT_MAX, 0);
        fill(stop, 1L, n);
        fill(ws + l.state, (long)l.state_words, 0);
    }
    hipLaunchKernelGGL(vox_clear_kernel, dim3(kFillBlocks, nf), dim3(256), 0, st, f);
    int rc = sph_check_launch("sph_points_to_voxel(clear)");
    if (rc || n == 0) return rc;
    hipLaunchKernelGGL(vox_insert_kernel, dim3(sph_div_up(n, kInsertThreads)), dim3(kInsertThreads), 0, st, points, n, q, cell_in,
                       l.tbits, keys, brought, later, slot_place, cell_out);
    rc = sph_check_launch("sph_points_to_voxel(cells)");
    if (rc) return rc;
    const hipError_t e = sph_scan::launch_from<sph_scan::PlusPair, kPointItems>(
        sph_scan::FromFunction<OpenedCells>{OpenedCells{brought, later, slot_place}}, CellRecords{slot_place, rec, stop, voxel_num, max_voxels},
        (long)n, ws + l.state, st, /*clear_state=*/false);
    if (e != hipSuccess) {
        sph_set_error("sph_points_to_voxel: scan: %s", hipGetErrorString(e));
        return SPH_ERR_LAUNCH;
    }
    hipLaunchKernelGGL(vox_scatter_kernel, dim3(blocks(n)), dim3(256), 0, st, (const int2 *)slot_place, (const int4 *)rec, n, seg);
    hipLaunchKernelGGL(vox_write_kernel, dim3(blocks(n)), dim3(256), 0, st, points, n, q, (const unsigned long long *)keys,
                       (const int2 *)slot_place, (const int4 *)rec, (const int32_t *)seg, (const int32_t *)stop, voxels, mask, coors,
                       num_points);
    return sph_check_launch("sph_points_to_voxel");
}

// ---------------------------------------------------------------------------
// What follows the voxeliser on the way to a sparse tensor: the mean of a voxel's points (SimpleVoxel,
// sphconv/vfe.py:210-228) and the batch's coordinates (merge_batch_torch, sphconv/datagen.py:53-74).  As tensor
// operations these are three and two or more launches of a few microseconds each for 24 000 voxels.
// ---------------------------------------------------------------------------
static __global__ __launch_bounds__(256) void voxel_mean_kernel(const float *voxels, const int32_t *num, int nv, int max_points,
                                                                int width, int nf, float *out)
{
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    const long v = t / nf;
    const int f = (int)(t - v * nf);
    if (v >= nv) return;
    const float *p = voxels + v * max_points * width + f;
    float s = 0.f;
    for (int j = 0; j < max_points; j++) s += p[(long)j * width];
    out[t] = __fdiv_rn(s, (float)num[v]);
}

SPH_EXPORT int sph_voxel_mean(const float *voxels, const int32_t *num_points, int nv, int max_points, int width, int nf,
                              float *out, void *stream)
{
    SPH_REQUIRE(nv >= 0 && max_points > 0 && nf > 0 && width >= nf, SPH_ERR_ARG, "sph_voxel_mean: bad sizes");
    if (nv == 0) return SPH_OK;
    SPH_REQUIRE(voxels && num_points && out, SPH_ERR_ARG, "sph_voxel_mean: null pointer");
    hipLaunchKernelGGL(voxel_mean_kernel, dim3(blocks((long)nv * nf)), dim3(256), 0, (hipStream_t)stream, voxels, num_points, nv,
                       max_points, width, nf, out);
    return sph_check_launch("sph_voxel_mean");
}

namespace {
struct CoordParts {
    const int32_t *p[SPH_MAX_BATCH_PARTS]; // [rows, 3] each
    int first[SPH_MAX_BATCH_PARTS + 1];    // first output row of every part
    int n;
};
} // namespace

static __global__ __launch_bounds__(256) void batch_coordinates_kernel(CoordParts c, int4 *out)
{
    const int r = blockIdx.x * 256 + threadIdx.x;
    if (r >= c.first[c.n]) return;
    int b = 0;
    while (r >= c.first[b + 1]) b++;
    const int32_t *p = c.p[b] + 3L * (r - c.first[b]);
    out[r] = make_int4(b, p[0], p[1], p[2]);
}

SPH_EXPORT int sph_batch_coordinates(const int32_t *const *parts, const int32_t *rows, int nparts, int32_t *out, void *stream)
{
    SPH_REQUIRE(parts && rows && nparts > 0 && nparts <= SPH_MAX_BATCH_PARTS && (uintptr_t)out % 16 == 0, SPH_ERR_ARG,
                "sph_batch_coordinates: 1 to %d parts and a 16-byte aligned output", SPH_MAX_BATCH_PARTS);
    CoordParts c;
    c.n = nparts;
    c.first[0] = 0;
    for (int b = 0; b < nparts; b++) {
        SPH_REQUIRE(rows[b] >= 0 && (rows[b] == 0 || parts[b]), SPH_ERR_ARG, "sph_batch_coordinates: null part");
        c.p[b] = parts[b];
        c.first[b + 1] = c.first[b] + rows[b];
    }
    const int total = c.first[nparts];
    if (total == 0) return SPH_OK;
    SPH_REQUIRE(out, SPH_ERR_ARG, "sph_batch_coordinates: null output");
    hipLaunchKernelGGL(batch_coordinates_kernel, dim3(blocks(total)), dim3(256), 0, (hipStream_t)stream, c, (int4 *)out);
    return sph_check_launch("sph_batch_coordinates");
}
