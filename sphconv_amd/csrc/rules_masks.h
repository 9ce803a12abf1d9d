// Rule generation by occupancy masks for books kept by stationary row only (included by rules.hip).
#pragma once
#include "rules_tile.h"

namespace {

// The mask join of rules_tile.h with a thread per stationary row and its results stored as they are made: a book without groups
// needs no table in LDS, so none is cleared, filled and read back, and what LDS holds (8 KB) lets sixteen workgroups share a
// compute unit.  A fiber is read sixteen entries at a time; a row's place among its entries is a population count, and the three
// offsets of a fiber share it.
// What bounds it: the table's bytes (13.8 KB a tile, written at 4.0 TB/s with 12 744 tiles), on small grids four dependent
// loads.  us, the mask join with the table in LDS -> now: 12 744 tiles 78.0 -> 44.1, 4056 tiles 30.3 -> 17.9, 1248 tiles 16.1 ->
// 11.6, 512 tiles 10.5 -> 7.8, 64 tiles 9.6 -> 8.5.
// That is for columns alike.  Where sparse columns lie beside full ones, a tile of more than 64 columns walks: one entry at a
// time that took up to twice the mask join's time (5.9 entries a column on average, 865 tiles 14.8 : 26.0), the first two of nine fibers
// and then eight of three at once 16.1 (307 tiles 10.9 : 13.3, 2588 tiles 27.1 : 20.6).  Two passes of masks over such a
// tile were slower (22.1), and so was a walk from 32 columns on, for columns of four entries (1003 tiles 7.3 : 6.3 -> 7.8).
// Left to it: transposed books, books with groups, kernels of more than 32 offsets (their masks outgrow the LDS), short grids with
// few rows to a column (masks_build_ok).
constexpr int kNbrThreads = R;
constexpr int kNbrCols = 64; // distinct columns of a tile that masks are made for

// On short grids the tile's chain counts, and with few rows to a column a tile has many columns, their fibers more than a thread each:
// stride 2 on a full grid of four bins, two rows to a column, 125 tiles 7.5 : 8.6 us, 375 tiles 9.0 : 9.5, 750 tiles 11.6 : 10.3;
// with three 75 tiles 7.2 : 8.1, with nearly four 63 tiles 9.1 : 7.3.
inline bool masks_build_ok(const BuildArgs &a, bool transposed, int KV, int ntiles)
{
    return !transposed && a.long_fibers && KV <= 32 && a.book.tile_nbr && !a.book.grp_gather && a.cv.p2 <= 64 - a.P.n2 &&
           (double)a.Q.n2 * a.cv.s2 < (1 << 22) && a.p_rows < (1 << 28) && (ntiles > 512 || a.q_rows >= 3.5 * a.B * a.Q.n0 * a.Q.n1);
}

inline size_t masks_lds(int K01) { return (size_t)kNbrCols * K01 * (sizeof(unsigned long long) + sizeof(int)) + kNbrCols * sizeof(int4); }

// K01T, K2T: the kernel's number of (k0, k1) and of k2, or 0 for those of the call.  HINT: the rows' columns are given.
template <bool HINT, int K01T, int K2T>
__global__ __launch_bounds__(kNbrThreads) void build_nbr_kernel(BuildArgs a)
{
    extern __shared__ __attribute__((aligned(16))) unsigned long long s_mask[]; // [K01][ncols], bit v + p2: an entry with S2 coordinate v
    __shared__ int s_col[R], s_first[2 * (kNbrThreads / kWave)], s_flag[2];
    __shared__ unsigned long long s_heads[R / kWave];
    __shared__ int s_last, s_bad[2], s_general;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    if ((int)blockIdx.x >= a.tile_blocks) {
        sph_pack_fragments(a.pack, (int)(blockIdx.x - a.tile_blocks) * kNbrThreads + tid);
        return;
    }
    const int tile = sph_xcd_tile(blockIdx.x, (a.q_rows + R - 1) / R);
    const int r0 = tile * R;
    if (r0 >= a.q_rows) return; // grid is padded to a multiple of the XCD count
    const int nrows = min(R, a.q_rows - r0);
    const int K01 = K01T ? K01T : a.cv.K0 * a.cv.K1, K2 = K2T ? K2T : a.cv.K2, KV = K01 * K2;
    int4 *s_cols = (int4 *)(s_mask + kNbrCols * K01);  // of a distinct column: its place on the gathered grid
    int *s_start = (int *)(s_cols + kNbrCols);         // [K01][ncols] first entry of the fiber
    int32_t *dst = a.book.tile_nbr + (long)tile * KV * R + tid;

    bool live = tid < nrows;
    const int r = r0 + min(tid, nrows - 1);
    const int zz = a.q_idx[r];
    const int q_ncol = a.B * a.Q.n0 * a.Q.n1;
    int c, hint_e = 0, hint_s = 0;
    bool inside = true;
    if constexpr (HINT) {
        const int hint = a.q_rowcol[r];
        inside = (unsigned)hint < (unsigned)q_ncol;
        c = inside ? hint : 0;
        hint_e = a.q_ptr[c];
        hint_s = a.q_ptr[max(c - 1, 0)];
    } else {
        search_columns<kNbrThreads>(a.q_ptr, q_ncol, a.q_rows, r0, r0 + nrows, s_col, s_first, s_flag, []() {});
        c = s_col[tid];
        live = live && c >= 0;
        c = max(c, 0);
    }
    const __amdgpu_buffer_rsrc_t r_idx = __builtin_amdgcn_make_buffer_rsrc((void *)a.p_idx, 0, a.p_rows * 4, 0x00020000);
    const unsigned inv_k1 = (65536u + a.cv.K1 - 1) / a.cv.K1;
    int cj, ncols, y0b, y1b, colb;
    for (bool first = true;; first = false) { // once, or twice where a column is wrong
    const bool first_col = c == 0;
    const int b = (int)div_by((uint32_t)c, a.by_q01);
    const int rem = c - b * (a.Q.n0 * a.Q.n1);
    const int c0 = (int)div_by((uint32_t)rem, a.by_q1), c1 = rem - c0 * a.Q.n1;
    y0b = c0 * a.cv.s0 - a.cv.p0;
    y1b = c1 * a.cv.s1 - a.cv.p1;
    colb = b * a.P.n0;
    // the tile's distinct columns, numbered in the rows' order (a column met again behind another one gets a second number)
    int before = __shfl_up(c, 1, kWave);
    if (tid == kWave - 1) s_last = c;
    if (tid == 0) s_general = 0;
    if (wave == 0) {
        const unsigned long long heads = __ballot(tid == 0 || c != before);
        if (lane == 0) s_heads[0] = heads;
    }
    lds_barrier();
    if (wave != 0) {
        if (lane == 0) before = s_last;
        const unsigned long long heads = __ballot(c != before);
        if (lane == 0) s_heads[1] = heads;
    }
    const unsigned long long h0 = s_heads[0];
    const unsigned long long mine = wave ? __ballot(c != before) : h0;
    cj = __popcll(mine & ((2ull << lane) - 1)) - 1 + (wave ? __popcll(h0) : 0);
    if (((mine >> lane) & 1) && cj < kNbrCols) s_cols[cj] = make_int4(y0b, y1b, colb, 0);
    lds_barrier();
    ncols = __popcll(h0) + __popcll(s_heads[1]);

    // every (column, k0, k1) fiber once into a mask of 64 bins
    if (ncols <= kNbrCols) {
        const float inv = __builtin_amdgcn_rcpf((float)ncols);
        for (int it = tid; it < ncols * K01; it += kNbrThreads) {
            const int k01 = (int)(((float)it + 0.5f) * inv), j = it - k01 * ncols;
            const int k0 = (int)(((unsigned)k01 * inv_k1) >> 16), k1 = k01 - k0 * a.cv.K1;
            const int4 at = s_cols[j];
            const int y0 = at.x + k0, y1 = at.y + k1;
            const bool ok = (unsigned)y0 < (unsigned)a.P.n0 && (unsigned)y1 < (unsigned)a.P.n1;
            int st, e;
            fiber_range(a.p_ptr, ok ? (at.z + y0) * a.P.n1 + y1 : 0, a.p_rows, st, e);
            const int n = ok ? e - st : 0;
            unsigned lo = 0, hi = 0;
            int prev = -1;
            bool bad = false;
            for (int t = 0; t < n; t += 16) {
                typedef int int4v __attribute__((ext_vector_type(4)));
                int4v v[4];
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = __builtin_amdgcn_raw_buffer_load_b128(r_idx, (st + t) * 4 + 16 * q, 0, 0);
#pragma unroll
                for (int q = 0; q < 16; q++) {
                    const int z = v[q / 4][q % 4];
                    if (t + q < n) {
                        bad |= (z <= prev) | (z >= a.P.n2);
                        prev = z;
                        const unsigned bit = 1u << ((z + a.cv.p2) & 31);
                        const bool high = ((z + a.cv.p2) & 32) != 0;
                        lo |= high ? 0u : bit;
                        hi |= high ? bit : 0u;
                    }
                }
            }
            if (bad) s_general = 1;
            s_mask[it] = (unsigned long long)hi << 32 | lo;
            s_start[it] = st;
        }
    }
    if (!HINT || !first) {
        lds_barrier();
        break;
    }
    const unsigned long long wrong = __ballot(live & !(inside & ((first_col ? 0 : hint_s) <= r) & (r < hint_e)));
    if (lane == 0) s_bad[wave] = wrong != 0;
    lds_barrier();
    if (!__builtin_amdgcn_readfirstlane(s_bad[0] | s_bad[1])) break;
    int above = q_ncol; // the first column whose rows end behind r
    for (c = 0; c < above;) {
        const int mid = (c + above) / 2;
        if (a.q_ptr[mid] > r) above = mid;
        else c = mid + 1;
    }
    live = live && c < q_ncol;
    c = min(c, q_ncol - 1);
    }

    if (ncols <= kNbrCols && !__builtin_amdgcn_readfirstlane(s_general)) {
        const int sh = zz * a.cv.s2; // the offset k2's bin is sh + k2
        const bool reach = live && (unsigned)sh < 64u;
        const unsigned long long below = (1ull << (sh & 63)) - 1;
        auto line = [&](int k01) {
            const unsigned long long m = reach ? s_mask[k01 * ncols + cj] : 0ull;
            int at = s_start[k01 * ncols + cj] + __popcll(m & below);
            const unsigned w = (unsigned)(m >> (sh & 63));
            for (int k2 = 0; k2 < K2; k2++) {
                const int has = (w >> k2) & 1;
                dst[(k01 * K2 + k2) * R] = has ? at : -1;
                at += has;
            }
        };
        if constexpr (K01T > 0) {
#pragma unroll
            for (int k01 = 0; k01 < K01T; k01++) line(k01);
        } else {
            for (int k01 = 0; k01 < K01; k01++) line(k01);
        }
        return;
    }
    // Fibers that do not ascend or leave the bins, or a tile of many short ones: every row walks its own, several at a time.
    for (int k = 0; k < KV; k++) dst[k * R] = -1;
    constexpr int kWalk = 9; // fibers at a time
    for (int base = 0; base < K01; base += kWalk) {
        int st[kWalk], n[kWalk];
#pragma unroll
        for (int i = 0; i < kWalk; i++) {
            st[i] = n[i] = 0;
            const int k01 = base + i;
            if (k01 >= K01) continue;
            const int k0 = (int)(((unsigned)k01 * inv_k1) >> 16), k1 = k01 - k0 * a.cv.K1;
            const int y0 = y0b + k0, y1 = y1b + k1;
            const bool ok = live && (unsigned)y0 < (unsigned)a.P.n0 && (unsigned)y1 < (unsigned)a.P.n1;
            const int pc = ok ? (colb + y0) * a.P.n1 + y1 : 0;
            const int from = a.p_ptr[max(pc - 1, 0)], to = a.p_ptr[pc];
            st[i] = pc > 0 ? from : 0;
            n[i] = ok ? to : 0;
        }
#pragma unroll
        for (int i = 0; i < kWalk; i++) {
            st[i] = clampi(st[i], 0, a.p_rows);
            n[i] = clampi(n[i], 0, a.p_rows) - st[i];
        }
        auto pair = [&](int i, int t, int z) {
            const int k2 = z - (zz * a.cv.s2 - a.cv.p2);
            if (t < n[i] && (unsigned)k2 < (unsigned)K2) dst[((base + i) * K2 + k2) * R] = st[i] + t;
        };
        int v[kWalk][2]; // the first two entries of every fiber, then eight at a time of three fibers (a line of the grid, mostly)
#pragma unroll
        for (int i = 0; i < kWalk; i++)
#pragma unroll
            for (int q = 0; q < 2; q++) v[i][q] = __builtin_amdgcn_raw_buffer_load_b32(r_idx, (st[i] + q) * 4, 0, 0);
#pragma unroll
        for (int i = 0; i < kWalk; i++)
#pragma unroll
            for (int q = 0; q < 2; q++) pair(i, q, v[i][q]);
#pragma unroll
        for (int i0 = 0; i0 < kWalk; i0 += 3) {
            const int most = max(n[i0], max(n[i0 + 1], n[i0 + 2]));
            for (int t = 2; __any(most > t); t += 8) {
                int u[3][8];
#pragma unroll
                for (int i = 0; i < 3; i++)
#pragma unroll
                    for (int q = 0; q < 8; q++) u[i][q] = __builtin_amdgcn_raw_buffer_load_b32(r_idx, (st[i0 + i] + t + q) * 4, 0, 0);
#pragma unroll
                for (int i = 0; i < 3; i++)
#pragma unroll
                    for (int q = 0; q < 8; q++) pair(i0 + i, t + q, u[i][q]);
            }
        }
    }
}

} // namespace
