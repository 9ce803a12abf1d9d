// COO -> per-column compressed layout (sph_init_tensor), replacing the dense
// occupancy grid + per-fiber atomics of init_tensor (src/sphconv/tensor.cu:78-127,
// fillGridKernel 21-36, reorderFeatureKernel 39-76): rows are sorted by their linear
// cell index (b, s0, s1, s2), which orders fibers by column and, inside a fiber, by
// ascending S2 -- one legal, deterministic serialisation of the reference's output
// (its order inside a fiber is the order in which atomics happen to land).
//
// No sort: a row's place is the start of its column plus its rank inside the column, and one bit per cell says both:
//   1. coo_clear_kernel  zeroes the bitmap, the scan's state and the status words (one launch)
//   2. coo_mark_kernel   every row sets its cell's bit in its column's bitmap (one 64-bit atomic without a result:
//                        nothing waits for it)
//   3. sum-scan (scan.h) of the columns' bit counts, made from the bitmap as they are read -> z_ptr
//   4. coo_place_kernel  rank = set bits of the column below s2 (popcounts of up to S2/64 words); writes the
//                        permutation, moves the feature row and reports the status; z_idx and
//                        the rows' columns come from the row or from the bitmap.  Rows that
//                        share a cell set one bit between them: their number is what the bits are short of the rows.
// (the reference keeps four bytes per cell for the same purpose, tensor.cu:21-36.)
// What bounds it: the random accesses, one atomic and one feature row per input row.  623 k rows in random order on a
// 4x64x2048x64 grid, 16 fp16 channels: 118 us in eight launches with per-column counters, slots, a scatter into segments
// and a walk of each row's segment; 66 us in four launches now.
// A bitmap of more than 1 GiB (8.6e9 cells) falls back to that walk, which needs memory by rows only:
//   coo_count_kernel    slot = atomicAdd(count[column]) per row (arrival order, only used to park the row inside its
//                       column's segment); sum-scan -> z_ptr
//   coo_scatter_kernel  (s2, row) -> segment position start + slot
//   coo_rank_kernel     every row counts the entries of its column with a smaller s2: that rank is its final
//                       position, whatever the arrival order was
// No memory is allocated: bitmap or segments and the scan's state live in the caller's workspace.
#include "common.h"

#include <cstring>

#include "scan.h"

namespace {

inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

inline size_t sum_scan_bytes(int ncol) { return sph_scan::state_bytes(ncol); }

struct RankLayout {
    size_t slot, seg_z, seg_row, temp, temp_bytes, total;
};

inline RankLayout rank_layout(int n, int ncol)
{
    RankLayout l;
    const size_t nn = (size_t)(n > 0 ? n : 1);
    size_t o = 0;
    l.slot = o; o += align256(nn * 4);
    l.seg_z = o; o += align256(nn * 4);
    l.seg_row = o; o += align256(nn * 4);
    l.temp = o;
    l.temp_bytes = sum_scan_bytes(ncol);
    l.total = l.temp_bytes ? o + align256(l.temp_bytes) : 0;
    return l;
}

constexpr size_t kBitmapMaxBytes = (size_t)1 << 30; // grids whose bitmap would be larger are ranked by the walk

// Columns per thread of the scan of the columns' bit counts.  With eight, 32 768 columns of eight words are sixteen
// workgroups that fetch 128 KB each: 12.8 us.  So the columns of deep grids go one to a thread as long as the workgroups
// stay few (they take a number each, one after the other, at 20 ns).
constexpr int kWideScanCols = 65536;
inline int scan_items(int ncol, int words) { return words > 1 && ncol <= kWideScanCols ? 1 : sph_scan::kItems; }

struct BitLayout {
    size_t bits, bits_bytes, temp, temp_bytes, total;
    int words; // 64-bit words per column
};

inline BitLayout bit_layout(int ncol, int S2)
{
    BitLayout l;
    l.words = (S2 + 63) / 64;
    l.bits = 0;
    l.bits_bytes = (size_t)ncol * l.words * sizeof(unsigned long long);
    l.temp = align256(l.bits_bytes);
    l.temp_bytes = sph_scan::state_bytes(ncol, scan_items(ncol, l.words));
    l.total = l.temp_bytes ? l.temp + align256(l.temp_bytes) : 0;
    return l;
}

inline bool by_bitmap(int ncol, int S2)
{
    return (double)ncol * ((S2 + 63) / 64) * 8.0 <= (double)kBitmapMaxBytes;
}

__global__ void fill_zero_kernel(int32_t *p, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// bitmap and scan state, which follow each other in the workspace (n16 16-byte words), and the status words
__global__ __launch_bounds__(256) void coo_clear_kernel(uint4 *p, long n16, int32_t *status)
{
    const long step = (long)gridDim.x * 256;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n16; i += step) p[i] = make_uint4(0, 0, 0, 0);
    if (blockIdx.x == 0 && threadIdx.x < 2) status[threadIdx.x] = 0;
}

__global__ void copy_status_kernel(const int32_t *status, int32_t *host_status)
{
    if (threadIdx.x == 0) *(unsigned long long *)host_status = *(const unsigned long long *)status;
}

struct CooGrid {
    int B, S0, S1, S2, words; // words: 64-bit words of a column's bitmap
};
__device__ __forceinline__ bool coo_inside(const int4 &c, const CooGrid &g)
{
    return (unsigned)c.x < (unsigned)g.B && (unsigned)c.y < (unsigned)g.S0 && (unsigned)c.z < (unsigned)g.S1 &&
           (unsigned)c.w < (unsigned)g.S2;
}

// Whether a wave's rows lie strewn over the grid: more than a quarter of them are not among the next columns of the row before.
__device__ __forceinline__ bool coo_strewn(const int4 &c, const CooGrid &g)
{
    const unsigned col = ((unsigned)c.x * g.S0 + (unsigned)c.y) * g.S1 + (unsigned)c.z;
    const unsigned before = (unsigned)__shfl_up((int)col, 1, 64);
    return __popcll(__ballot((threadIdx.x & 63) != 0 && col - before > 32u)) > 16;
}

// *strewn (zero before, may be null): set where one of the sampled waves finds its rows so
__global__ __launch_bounds__(256) void coo_mark_kernel(const int32_t *idx, int n, CooGrid g, unsigned long long *bits, int32_t *status,
                                                       int32_t *strewn)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int4 c = ((const int4 *)idx)[i]; // (b, s0, s1, s2)
    if (strewn && blockIdx.x % 8 == 0 && coo_strewn(c, g) && threadIdx.x % 64 == 0) *strewn = 1;
    if (!coo_inside(c, g)) {
        atomicAdd(&status[0], 1);
        return;
    }
    const int col = (c.x * g.S0 + c.y) * g.S1 + c.z;
    atomicOr(&bits[(size_t)col * g.words + (c.w >> 6)], 1ull << (c.w & 63));
}

// rows of a column, from its bitmap (what the scan reads)
template <int WORDS> // words per column where that is known to the compiler: their loads are then in flight together; 0: any
struct ColumnRows {
    const unsigned long long *bits;
    int words;
    __device__ __forceinline__ int operator()(long col) const
    {
        int n = 0;
        if constexpr (WORDS > 0) {
            const unsigned long long *p = bits + (size_t)col * WORDS;
#pragma unroll
            for (int w = 0; w < WORDS; w++) n += __popcll(p[w]);
        } else {
            for (int w = 0; w < words; w++) n += __popcll(bits[(size_t)col * words + w]);
        }
        return n;
    }
};

template <int WORDS>
inline hipError_t scan_columns(const unsigned long long *bits, int words, int32_t *z_ptr, int ncol, void *state, hipStream_t st)
{
    const sph_scan::FromFunction<ColumnRows<WORDS>> rows{ColumnRows<WORDS>{bits, words}};
    const sph_scan::ToArray out{z_ptr, nullptr};
    if (scan_items(ncol, words) == 1) return sph_scan::launch_from<sph_scan::Plus, 1>(rows, out, ncol, state, st, /*clear_state=*/false);
    return sph_scan::launch_from<sph_scan::Plus, sph_scan::kItems>(rows, out, ncol, state, st, /*clear_state=*/false);
}

struct CooRows {
    const int32_t *z_ptr;
    const unsigned long long *bits;
    int32_t *z_idx, *permutation, *row_cols; // row_cols may be null
    const char *feature;                     // null: no rows to move
    char *out;
    int32_t *status, *host_status;           // host_status (may be null): the same two words where the host reads them
    const int32_t *strewn;                   // null: the rows write z_idx and row_cols; else the columns do where *strewn is not 0
};

// Whether the columns may write what their bits say of their rows, a thread each: where the bitmap has few words more than there are
// rows, and the columns are neither deep nor full (a thread goes through its words and rows one by one).  us of the call, 32-byte
// features, by rows : by columns, rows in random order:
//   623 k rows, 524 k columns of 64 bins 78.5 : 65.8      140 k, 524 k columns 31.2 : 30.1    94 k, 131 k columns 19.2 : 18.3
//   35 k, 131 k columns 14.4 : 14.9     4000, 4096 columns 10.9 : 11.2   (what the mark kernel found is read in front of all else)
//   20 k, 1024 columns 12.3 : 15.7      200 k, 4096 columns of 128 bins 24.9 : 34.4     200 k, 1024 columns of 4096 bins 55.7 : 120
// Rows that come in the columns' order write next to one another, and the columns would cost more than they save (623 k rows 38.3 :
// 40.8): the mark kernel looks at the order of an eighth of the rows, and the place kernel goes by what it found (39.2).
inline bool coo_by_columns(int n, int ncol, int words)
{
    return n >= 65536 && words <= 4 && 4 * (double)n >= (double)ncol * words && n <= 8 * (double)ncol;
}

// What a column's bits say of its rows, a thread per column: their S2 coordinates and their column.
__device__ __forceinline__ void coo_columns(int col, int n, const CooGrid &g, const CooRows &r)
{
    if (col >= g.B * g.S0 * g.S1) return;
    int pos = col ? r.z_ptr[col - 1] : 0;
    for (int w = 0; w < g.words; w++)
        for (unsigned long long m = r.bits[(size_t)col * g.words + w]; m && pos < n; m &= m - 1, pos++) {
            r.z_idx[pos] = w * 64 + __ffsll((long long)m) - 1;
            if (r.row_cols) r.row_cols[pos] = col;
        }
}

// gpr threads per row, one 16-byte (G) granule of its features each; gpr = 1 without features.  z_idx and row_cols are written by
// rows, two 4-byte writes to lines of their own for each where the rows come in no order, or there (coo_by_columns) by
// workgroups of the columns behind those of the rows (row_blocks).
template <typename G>
__global__ __launch_bounds__(256) void coo_place_kernel(const int32_t *idx, int n, CooGrid g, CooRows r, int gpr, int row_blocks)
{
    const bool by_columns = r.strewn && *r.strewn != 0;
    if ((int)blockIdx.x >= row_blocks) {
        if (by_columns) coo_columns((blockIdx.x - row_blocks) * 256 + threadIdx.x, n, g, r);
        return;
    }
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t == 0) {
        const int outside = r.status[0], ncol = g.B * g.S0 * g.S1;
        const int dup = n - outside - r.z_ptr[ncol - 1];
        r.status[1] = dup;
        if (r.host_status) {
            // one 8-byte store: the host may be watching the pair
            *(unsigned long long *)r.host_status = ((unsigned long long)(unsigned)dup << 32) | (unsigned)outside;
        }
    }
    const int i = gpr == 1 ? (int)t : (int)(t / gpr);
    const int q = gpr == 1 ? 0 : (int)(t - (long)i * gpr);
    if (i >= n) return;
    const int4 c = ((const int4 *)idx)[i];
    if (!coo_inside(c, g)) return;
    const int col = (c.x * g.S0 + c.y) * g.S1 + c.z;
    const unsigned long long *cb = r.bits + (size_t)col * g.words;
    const int wz = c.w >> 6;
    int rank = __popcll(cb[wz] & ((1ull << (c.w & 63)) - 1ull));
    for (int w = 0; w < wz; w++) rank += __popcll(cb[w]);
    const int pos = (col ? r.z_ptr[col - 1] : 0) + rank;
    if ((unsigned)pos >= (unsigned)n) return;
    if (q == 0) {
        r.permutation[i] = pos;
        if (!by_columns) {
            r.z_idx[pos] = c.w;
            if (r.row_cols) r.row_cols[pos] = col;
        }
    }
    if (r.feature) ((G *)r.out)[(long)pos * gpr + q] = ((const G *)r.feature)[(long)i * gpr + q];
}

__global__ void coo_count_kernel(const int32_t *idx, int n, int B, int S0, int S1, int S2, int32_t *counts, int32_t *slot,
                                 int32_t *status)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int4 c = ((const int4 *)idx)[i]; // (b, s0, s1, s2)
    const bool ok = (unsigned)c.x < (unsigned)B && (unsigned)c.y < (unsigned)S0 && (unsigned)c.z < (unsigned)S1 &&
                    (unsigned)c.w < (unsigned)S2;
    int sl = -1;
    if (ok) sl = atomicAdd(&counts[(c.x * S0 + c.y) * S1 + c.z], 1);
    else atomicAdd(&status[0], 1);
    slot[i] = sl;
}

__global__ void coo_scatter_kernel(const int32_t *idx, int n, int S0, int S1, const int32_t *z_ptr, const int32_t *slot,
                                   int32_t *seg_z, int32_t *seg_row)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int sl = slot[i];
    if (sl < 0) return;
    const int4 c = ((const int4 *)idx)[i];
    const int col = (c.x * S0 + c.y) * S1 + c.z;
    const int pos = (col ? z_ptr[col - 1] : 0) + sl;
    if ((unsigned)pos >= (unsigned)n) return;
    seg_z[pos] = c.w;
    seg_row[pos] = i;
}

__global__ void coo_rank_kernel(const int32_t *idx, int n, int S0, int S1, int S2, const int32_t *z_ptr, const int32_t *slot,
                                const int32_t *seg_z, const int32_t *seg_row, int32_t *z_idx, int32_t *permutation,
                                int32_t *status)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (slot[i] < 0) return;
    const int4 c = ((const int4 *)idx)[i];
    const int col = (c.x * S0 + c.y) * S1 + c.z;
    const int start = col ? z_ptr[col - 1] : 0;
    int end = min(z_ptr[col], n);
    int rank = 0, dup = 0;
    if (end - start > S2) { // more rows than bins: duplicates for sure; keep the walk bounded
        dup = 1;
        end = start + S2;
    }
    for (int j = start; j < end; j++) {
        const int z = seg_z[j];
        rank += z < c.w;
        dup += (z == c.w && seg_row[j] < i);
    }
    if (dup) atomicAdd(&status[1], dup);
    const int pos = start + rank;
    if ((unsigned)pos < (unsigned)n) {
        z_idx[pos] = c.w;
        permutation[i] = pos;
    }
}

} // namespace

SPH_EXPORT size_t sph_init_tensor_workspace(int n, int B, int S0, int S1, int S2)
{
    if (n < 0 || B <= 0 || S0 <= 0 || S1 <= 0 || S2 <= 0) return 0;
    if ((double)B * S0 * S1 >= 2147483648.0) return 0;
    if (by_bitmap(B * S0 * S1, S2)) return bit_layout(B * S0 * S1, S2).total;
    return rank_layout(n, B * S0 * S1).total;
}

// count, scan, scatter, rank by a walk of the column's segment (grids whose bitmap would not fit)
static int init_tensor_by_rank(const int32_t *indices, int n, int B, int S0, int S1, int S2, int32_t *z_idx, int32_t *z_ptr,
                               int32_t *permutation, int32_t *status, void *workspace, size_t workspace_bytes,
                               hipStream_t st)
{
    const int ncol = B * S0 * S1;
    const RankLayout l = rank_layout(n, ncol);
    SPH_REQUIRE(l.total != 0, SPH_ERR_LAUNCH, "sph_init_tensor: temporary storage query failed");
    SPH_REQUIRE(workspace_bytes >= l.total, SPH_ERR_ARG, "sph_init_tensor: workspace of %zu bytes, %zu needed",
                workspace_bytes, l.total);
    char *ws = (char *)workspace;
    int32_t *slot = (int32_t *)(ws + l.slot), *seg_z = (int32_t *)(ws + l.seg_z), *seg_row = (int32_t *)(ws + l.seg_row);
    hipLaunchKernelGGL(fill_zero_kernel, dim3((ncol + 255) / 256), dim3(256), 0, st, z_ptr, ncol);
    hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(64), 0, st, status, 2);
    int rc = sph_check_launch("sph_init_tensor(fill)");
    if (rc || n == 0) return rc;
    const dim3 grid((n + 255) / 256), block(256);
    hipLaunchKernelGGL(coo_count_kernel, grid, block, 0, st, indices, n, B, S0, S1, S2, z_ptr, slot, status);
    rc = sph_check_launch("sph_init_tensor(count)");
    if (rc) return rc;
    hipError_t e = sph_scan::launch(z_ptr, z_ptr, ncol, ws + l.temp, st);
    if (e != hipSuccess) {
        sph_set_error("sph_init_tensor: scan: %s", hipGetErrorString(e));
        return SPH_ERR_LAUNCH;
    }
    hipLaunchKernelGGL(coo_scatter_kernel, grid, block, 0, st, indices, n, S0, S1, (const int32_t *)z_ptr,
                       (const int32_t *)slot, seg_z, seg_row);
    hipLaunchKernelGGL(coo_rank_kernel, grid, block, 0, st, indices, n, S0, S1, S2, (const int32_t *)z_ptr, (const int32_t *)slot,
                       (const int32_t *)seg_z, (const int32_t *)seg_row, z_idx, permutation, status);
    return sph_check_launch("sph_init_tensor(rank)");
}

// Granules of a row up to which the place kernel moves the features itself (each granule's thread finds the row's
// place again, from cached words); longer rows are moved by sph_permute_rows.
constexpr int kPlaceGranules = 16;

SPH_EXPORT int sph_init_tensor_rows(const int32_t *indices, int n, int B, int S0, int S1, int S2, const void *feature,
                                    int row_bytes, int32_t *z_idx, int32_t *z_ptr, int32_t *permutation, int32_t *row_cols,
                                    void *out_feature, int32_t *status, int32_t *host_status, void *workspace,
                                    size_t workspace_bytes, void *stream)
{
    const char *who = "sph_init_tensor";
    SPH_REQUIRE(n >= 0 && B > 0 && S0 > 0 && S1 > 0 && S2 > 0, SPH_ERR_ARG, "%s: bad sizes", who);
    SPH_REQUIRE((double)B * S0 * S1 < 2147483648.0, SPH_ERR_UNSUPPORTED, "%s: more than 2^31 columns", who);
    SPH_REQUIRE(z_ptr && status && workspace && (n == 0 || (indices && z_idx && permutation)), SPH_ERR_ARG, "%s: null pointer", who);
    SPH_REQUIRE((uintptr_t)indices % 16 == 0 && (uintptr_t)workspace % 256 == 0 && (uintptr_t)host_status % 8 == 0, SPH_ERR_ARG,
                "%s: indices must be 16-byte aligned, the workspace 256-byte aligned, the host's status words 8-byte aligned", who);
    SPH_REQUIRE(!feature || (out_feature && row_bytes > 0), SPH_ERR_ARG, "%s: feature rows without a place to go", who);
    const int ncol = B * S0 * S1;
    hipStream_t st = (hipStream_t)stream;
    const bool move = feature && n > 0;
    int rc;
    if (!by_bitmap(ncol, S2)) {
        rc = init_tensor_by_rank(indices, n, B, S0, S1, S2, z_idx, z_ptr, permutation, status, workspace, workspace_bytes, st);
        if (rc) return rc;
        if (row_cols && n > 0 && (rc = sph_row_columns(z_ptr, ncol, n, row_cols, stream))) return rc;
        if (move && (rc = sph_permute_rows(feature, permutation, n, row_bytes, 0, out_feature, stream))) return rc;
        if (host_status) hipLaunchKernelGGL(copy_status_kernel, dim3(1), dim3(64), 0, st, (const int32_t *)status, host_status);
        return sph_check_launch(who);
    }
    const BitLayout l = bit_layout(ncol, S2);
    SPH_REQUIRE(l.total != 0, SPH_ERR_LAUNCH, "%s: temporary storage query failed", who);
    SPH_REQUIRE(workspace_bytes >= l.total, SPH_ERR_ARG, "%s: workspace of %zu bytes, %zu needed", who, workspace_bytes, l.total);
    char *ws = (char *)workspace;
    CooGrid g{B, S0, S1, S2, l.words};
    CooRows r{z_ptr, (const unsigned long long *)(ws + l.bits), z_idx, permutation, row_cols, nullptr, nullptr, status, host_status, nullptr};
    // (the second word of the scan's state is nobody's, and cleared with it)
    int32_t *strewn = coo_by_columns(n, ncol, l.words) ? (int32_t *)(ws + l.temp) + 1 : nullptr;
    r.strewn = strewn;
    const long n16 = (long)(l.total / 16);
    hipLaunchKernelGGL(coo_clear_kernel, dim3((unsigned)(n16 < 256L * 2048 ? (n16 + 255) / 256 : 2048)), dim3(256), 0, st,
                       (uint4 *)workspace, n16, status);
    const dim3 block(256);
    if (n > 0)
        hipLaunchKernelGGL(coo_mark_kernel, dim3(sph_div_up(n, 256)), block, 0, st, indices, n, g, (unsigned long long *)(ws + l.bits), status,
                           strewn);
    hipError_t e;
    switch (l.words) {
    case 1: e = scan_columns<1>(r.bits, 1, z_ptr, ncol, ws + l.temp, st); break;
    case 2: e = scan_columns<2>(r.bits, 2, z_ptr, ncol, ws + l.temp, st); break;
    case 4: e = scan_columns<4>(r.bits, 4, z_ptr, ncol, ws + l.temp, st); break;
    case 8: e = scan_columns<8>(r.bits, 8, z_ptr, ncol, ws + l.temp, st); break;
    default: e = scan_columns<0>(r.bits, l.words, z_ptr, ncol, ws + l.temp, st); break;
    }
    if (e != hipSuccess) {
        sph_set_error("%s: scan: %s", who, hipGetErrorString(e));
        return SPH_ERR_LAUNCH;
    }
    const uintptr_t al = (uintptr_t)feature | (uintptr_t)out_feature | (uintptr_t)row_bytes;
    const int gran = al % 16 == 0 ? 16 : (al % 4 == 0 ? 4 : (al % 2 == 0 ? 2 : 1));
    const bool here = move && row_bytes / gran <= kPlaceGranules;
    int gpr = 1;
    if (here) {
        r.feature = (const char *)feature;
        r.out = (char *)out_feature;
        gpr = row_bytes / gran;
    }
    const int row_blocks = (int)(((long)n * gpr + 255) / 256 + (n == 0));
    const dim3 grid((unsigned)row_blocks + (unsigned)(strewn ? sph_div_up(ncol, 256) : 0));
    switch (here ? gran : 16) {
    case 16: hipLaunchKernelGGL(coo_place_kernel<uint4>, grid, block, 0, st, indices, n, g, r, gpr, row_blocks); break;
    case 4: hipLaunchKernelGGL(coo_place_kernel<uint32_t>, grid, block, 0, st, indices, n, g, r, gpr, row_blocks); break;
    case 2: hipLaunchKernelGGL(coo_place_kernel<uint16_t>, grid, block, 0, st, indices, n, g, r, gpr, row_blocks); break;
    default: hipLaunchKernelGGL(coo_place_kernel<uint8_t>, grid, block, 0, st, indices, n, g, r, gpr, row_blocks); break;
    }
    rc = sph_check_launch(who);
    if (rc) return rc;
    if (move && !here) return sph_permute_rows(feature, permutation, n, row_bytes, 0, out_feature, stream);
    return SPH_OK;
}

SPH_EXPORT int sph_init_tensor(const int32_t *indices, int n, int B, int S0, int S1, int S2, int32_t *z_idx,
                               int32_t *z_ptr, int32_t *permutation, int32_t *status, void *workspace,
                               size_t workspace_bytes, void *stream)
{
    return sph_init_tensor_rows(indices, n, B, S0, S1, S2, nullptr, 0, z_idx, z_ptr, permutation, nullptr, nullptr, status,
                                nullptr, workspace, workspace_bytes, stream);
}
