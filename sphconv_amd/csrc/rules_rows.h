// Rule generation with a thread per stationary row, for long grids (included by rules.hip).
#pragma once
#include <climits>
#include <type_traits>

#include "rules_tile.h"

namespace {

// The kernel of rules_tile.h is made for the length of one tile's chain: 256 threads, two or more items of work each, and on
// large grids a vector ALU that is 90 % busy with 2460 instructions a tile.  This one is made for few of them (1310): a thread
// has one row and takes the entries of its NL x C columns column by column, keeps the offsets it found a pair at as bits
// of one register, and writes only the pairs it found (the table needs no clearing and is read where a bit is set).  A wave
// takes its own 64 rows through all offsets: a ballot per offset, counts in the lanes of one register, one exchange of counts
// between the tile's two waves.  The pairs go to their slots tagged with their owner's row, and out sixteen bytes at a time.
// Books with up to 32 offsets and rows below 2^24.  The rows' columns come from the caller's table or from a search by the
// workgroup (in a tile with a table entry that turns out wrong every thread searches for its row's own).
// What bounds it: the vector ALU, 72 % busy over the kernel (5890 tiles), between the ends of nine workgroups' rounds.
// us, the kernel of rules_tile.h -> this one, with the rows' columns (without), columns of one to three entries as a scan has
// them: submanifold 3x3x3 530 tiles 7.8 -> 6.9 (8.7 -> 8.0), 930 tiles 8.6 -> 7.2 (9.5 -> 8.4), 2400 tiles 15.9 -> 12.8 (18.4 ->
// 15.2), 5890 tiles 31.8 -> 21.5 (37.8 -> 26.9); 3x3x1 530 tiles 6.5 -> 6.1 (7.5 -> 7.1), 1x3x3 6.0 -> 5.1 (7.0 -> 5.9); stride 2
// transposed 1100 tiles 19.0 -> 12.9, 2400 tiles 32.1 -> 21.3.  A call among others gains more: three scans of 926 tiles in
// flight 21.7 -> 19.5 us a scan.
// Asking for as many lines and columns as the call has, instead of three by three, is what keeps small kernels
// here: 1x3x3 as three lines 530 tiles 6.7, 4800 tiles 16.8, as one 5.1 and 10.9; 3x1x1 with stride 2 transposed 1100 tiles 9.0, now 6.1.
// On the way: with the checks of the rows' columns before the pointers are asked for, entries past a column's second one by one,
// the table read an offset at a time, and masks kept from the counting for the placing (54 scalar registers, spilled), no faster
// than the general kernel (32 and 72 us); a test of every column before its third entry 10 % slower.
constexpr int kRowThreads = R;
constexpr int kRowTag = 24; // a pair in the slot array: gathered row, and the owner's row in the tile from this bit on

// Lines of the gathered grid a row can pair with.
inline int rows_lines(const BuildArgs &a, bool transposed) { return transposed ? (a.cv.K0 + a.cv.s0 - 1) / a.cv.s0 : a.cv.K0; }

inline bool rows_build_ok(const BuildArgs &a, bool transposed, int KV, int ntiles)
{
    const int nlines = rows_lines(a, transposed);
    // Entries a column of the gathered side holds on average.  A round takes as long as the wave's longest column needs, so what
    // has many or uneven ones stays with the kernels of rules_tile.h until there are tiles enough.  us, theirs : this one's,
    // submanifold 3x3x3:
    //   1 to 3 entries in 60 % of the columns   530 tiles  7.8 :  6.9   930 tiles  8.6 :  7.2   2400 tiles 15.9 : 12.8
    //   Poisson, 1.2 a column                   530 tiles  7.7 :  8.0   930 tiles  8.6 :  8.7   2400 tiles 15.9 : 14.5
    //   Poisson, 3.9 a column                   600 tiles  9.8 : 10.5  1300 tiles 13.0 : 12.6   3000 tiles 22.9 : 20.7
    //   3.9, in a third of the columns          600 tiles 12.2 : 15.5  1300 tiles 16.4 : 17.5   3000 tiles 28.8 : 28.7
    //   512 bins, 8.0 in a third                600 tiles 15.7 : 21.2  1300 tiles 18.9 : 22.9   3000 tiles 32.5 : 39.5
    // A row of a transposed book meets at most two columns of three on each line; what it replaces there is, up to 64 bins and
    // from four entries on, the join by masks.  Stride 2 transposed:
    //   64 bins, 12.5 entries a column   1100 tiles 19.0 : 12.9   2400 tiles 32.1 : 21.3  (32 entries 4101 tiles 34.0 : 36.9)
    //   256 bins, 13                     1100 tiles 14.2 : 15.0   1700 tiles 19.5 : 16.9   3000 tiles 27.7 : 26.1
    //   256 bins, 25                     1100 tiles 17.5 : 18.4   1700 tiles 24.3 : 21.6   3000 tiles 34.9 : 32.6
    //   256 bins, 48                     1100 tiles 22.9 : 24.6   3000 tiles, in a fifth of the columns 61.0 : 63.5
    // (at 914 tiles 10.9 : 11.4).
    const double each = a.p_rows / ((double)a.B * a.P.n0 * a.P.n1);
    int line;
    if (transposed) line = each < 4.0 || (a.long_fibers && each <= 16.0) ? 1024 : (!a.long_fibers && each <= 32.0 ? 1536 : INT_MAX);
    else line = a.long_fibers || each > 4.0 ? INT_MAX : (each <= 1.5 ? 512 : 2048);
    // the coordinates' products are signed 24-bit ones: an axis, stride or padding of up to 2^22 (a coordinate and a padding
    // add up) keeps every factor below 2^23; columns are divided by unsigned ones
    const int most = 1 << 22;
    const bool small = a.Q.n0 <= most && a.Q.n1 <= most && a.Q.n2 <= most && (double)a.B * a.P.n0 <= most && a.P.n1 <= most &&
                       a.cv.s0 <= most && a.cv.s1 <= most && a.cv.s2 <= most && a.cv.p0 <= most && a.cv.p1 <= most;
    // groups are stored sixteen bytes at a time; the caller's arrays need not be aligned to that
    const bool aligned = (((uintptr_t)a.book.grp_gather | (uintptr_t)a.book.grp_owner) & 15) == 0;
    return small && aligned && ntiles > line && a.lines >= 1 && nlines <= 3 && KV <= 32 && a.book.grp_gather && !a.book.tile_nbr &&
           a.p_rows < (1 << kRowTag) && (double)a.B * a.Q.n0 * a.Q.n1 < (1 << 24) && (double)a.B * a.P.n0 * a.P.n1 < (1 << 24);
}

// Groups whose slots are in LDS at a time (a tile has 33 to 36 at the densities of a scan): with the table 16.7 KB at 27
// offsets, nine workgroups on a compute unit.
constexpr int kRowGroups = 40;
// LDS behind the table [R][KV]: the slots, the counts of both waves, a flag of each.
constexpr size_t kRowScratch = (size_t)kRowGroups * SPH_GROUP * 4 + 2 * 32 * 4 + 2 * 4;

// KVT: the kernel volume, or 32 for any up to that.  HINT: the rows' columns are given (and checked), else searched for.
// LATER: entries a column's later rounds take at most (4, or 2 where registers count: rows_kernel).
template <bool TRANSPOSED, int C, int NL, int KVT, bool HINT, int LATER = 4>
__global__ __launch_bounds__(kRowThreads) void build_rows_kernel(BuildArgs a)
{
    extern __shared__ __attribute__((aligned(16))) int32_t s_nbr[];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    if ((int)blockIdx.x >= a.tile_blocks) {
        sph_pack_fragments(a.pack, (int)(blockIdx.x - a.tile_blocks) * kRowThreads + tid);
        return;
    }
    const int tile = sph_xcd_tile(blockIdx.x, (a.q_rows + R - 1) / R);
    const int K12 = a.cv.K1 * a.cv.K2, KV = KVT < 32 ? KVT : a.cv.K0 * K12, K2 = a.cv.K2;
    const int r0 = tile * R;
    if (r0 >= a.q_rows) return; // grid is padded to a multiple of the XCD count
    const int nrows = min(R, a.q_rows - r0);
    int *s_slot = s_nbr + R * KV;                              // [kRowGroups * SPH_GROUP] pairs, tagged, or -1
    int *s_cnt = s_slot + kRowGroups * SPH_GROUP;          // [2][32] pairs of an offset in a wave's rows
    int *s_bad = s_cnt + 2 * 32;                               // [2] the wave met a wrong column

    // the row and its column, which is believed before it is checked: the first pointers are on their way by then
    bool live = tid < nrows;
    const int r = r0 + min(tid, nrows - 1);
    const int zz = a.q_idx[r];
    const int q_ncol = a.B * a.Q.n0 * a.Q.n1, p_ncol = a.B * a.P.n0 * a.P.n1;
    int c, hint_e = 0, hint_s = 0;
    bool inside = true, first_col = false;
    if constexpr (HINT) {
        const int hint = a.q_rowcol[r];
        inside = (unsigned)hint < (unsigned)q_ncol;
        c = inside ? hint : 0;
        first_col = c == 0;
        hint_e = a.q_ptr[c];
        hint_s = a.q_ptr[max(c - 1, 0)];
    } else {
        __shared__ int s_col[R], s_first[2 * (kRowThreads / kWave)], s_flag[2];
        search_columns<kRowThreads>(a.q_ptr, q_ncol, a.q_rows, r0, r0 + nrows, s_col, s_first, s_flag, []() {});
        c = s_col[tid];
        live = live && c >= 0;
        c = max(c, 0);
    }

    const __amdgpu_buffer_rsrc_t r_ptr = __builtin_amdgcn_make_buffer_rsrc((void *)a.p_ptr, 0, p_ncol * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t r_idx = __builtin_amdgcn_make_buffer_rsrc((void *)a.p_idx, 0, a.p_rows * 4, 0x00020000);
    const int dy = TRANSPOSED ? -1 : 1, dline = TRANSPOSED ? a.cv.s0 * K12 : K12, dcol = TRANSPOSED ? -a.cv.s1 * K2 : K2;
    const int nlines = TRANSPOSED ? (a.cv.K0 + a.cv.s0 - 1) / a.cv.s0 : a.cv.K0;
    const int off_z = TRANSPOSED ? zz + a.cv.p2 : a.cv.p2 - __mul24(zz, a.cv.s2); // k2 = off_z +- v
    int p[NL][C + 1], slot;
    bool line_ok[NL], col_ok[C];
    for (bool first = true;; first = false) { // once, or twice where a column is wrong
    const int b = (int)div_by((uint32_t)c, a.by_q01);
    const int rem = c - (int)__umul24((unsigned)b, (unsigned)(a.Q.n0 * a.Q.n1));
    const int c0 = (int)div_by((uint32_t)rem, a.by_q1), c1 = rem - (int)__umul24((unsigned)c0, (unsigned)a.Q.n1);
    // Line j of the gathered grid: coordinate y0 + j * dy on the first axis; its columns ya, ya + 1, .. of which [lo, hi) are
    // in the grid and within the kernel; offset of (line j, column ya + i): slot + j * dline + i * dcol + k2.
    int y0, ya, rem0 = 0, lo;
    slot = 0;
    if (!TRANSPOSED) {
        y0 = __mul24(c0, a.cv.s0) - a.cv.p0;
        ya = __mul24(c1, a.cv.s1) - a.cv.p1;
        lo = max(0, -ya);
    } else { // k_d = x_d + p_d - y_d * s_d: the highest column and the first line have the smallest offsets
        const int t0 = c0 + a.cv.p0, t1 = c1 + a.cv.p1;
        int yb;
        if (((a.cv.s0 & (a.cv.s0 - 1)) | (a.cv.s1 & (a.cv.s1 - 1))) == 0) {
            y0 = t0 >> (__ffs(a.cv.s0) - 1);
            yb = t1 >> (__ffs(a.cv.s1) - 1);
        } else {
            y0 = t0 / a.cv.s0;
            yb = t1 / a.cv.s1;
        }
        rem0 = t0 - __mul24(y0, a.cv.s0);
        ya = yb - (a.lines - 1);
        const int k1a = t1 - __mul24(ya, a.cv.s1); // offset of column ya: the only one that can be too large
        slot = __mul24(rem0, K12) + __mul24(k1a, K2);
        lo = max(k1a >= a.cv.K1 ? 1 : 0, -ya);
    }
    const int hi = min(a.lines, a.P.n1 - ya); // (a.lines is at most C)
#pragma unroll
    for (int i = 0; i < C; i++) col_ok[i] = live && i >= lo && i < hi;
    const int pc0 = __mul24(__mul24(b, a.P.n0) + y0, a.P.n1) + ya;

    // the pointers that bound a line's columns
#pragma unroll
    for (int j = 0; j < NL; j++) {
        line_ok[j] = j < nlines && (unsigned)(y0 + j * dy) < (unsigned)a.P.n0 && (!TRANSPOSED || rem0 + j * a.cv.s0 < a.cv.K0);
        const int at = (pc0 + j * dy * a.P.n1 - 1) * 4;
#pragma unroll
        for (int q = 0; q <= C; q++) p[j][q] = __builtin_amdgcn_raw_buffer_load_b32(r_ptr, max(at, 0) + 4 * q, 0, 0);
        if (__any(at < 0)) { // in front of the array's first element are zeros, where the grid's first column begins
#pragma unroll
            for (int q = 0; q <= C; q++) {
                const int x = __builtin_amdgcn_raw_buffer_load_b32(r_ptr, max(at + 4 * q, 0), 0, 0);
                p[j][q] = at + 4 * q < 0 ? 0 : x;
            }
        }
    }
    if (first)
        for (int i = tid; i < kRowGroups * SPH_GROUP / 4; i += kRowThreads) ((int4 *)s_slot)[i] = make_int4(-1, -1, -1, -1);
    if (!HINT || !first) break;
    __builtin_amdgcn_sched_barrier(0); // (nothing above waits for the pointers of the row's own column)
    const int own_s = first_col ? 0 : hint_s;
    const unsigned long long bad = __ballot(live & !(inside & (own_s <= r) & (r < hint_e)));
    if (lane == 0) s_bad[wave] = bad != 0;
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

    // entries t = 0 and 1 of every column, all on their way together, then 2 and 3 (or to 5) where a lane has them, then four at a
    // time of the columns that have any left for one of the wave's rows
    int at[NL][C], n[NL][C]; // at: byte offset of the column's first entry
#pragma unroll
    for (int j = 0; j < NL; j++) {
#pragma unroll
        for (int q = 0; q <= C; q++) p[j][q] = (int)min((unsigned)p[j][q], (unsigned)a.p_rows);
#pragma unroll
        for (int i = 0; i < C; i++) {
            at[j][i] = p[j][i] * 4;
            n[j][i] = col_ok[i] && line_ok[j] ? p[j][i + 1] - p[j][i] : 0;
        }
    }
    unsigned found = 0; // bit k: a pair at offset k
    const int tag = tid << kRowTag;
    int32_t *mine = s_nbr + __mul24(tid, KV);
    auto entries = [&](int t, auto number, auto uneven) { // entries t, t + 1, .. of all columns, or (uneven) of those that have one
        constexpr int N = decltype(number)::value;
        int v[NL][C][N];
        bool go[NL][C];
#pragma unroll
        for (int j = 0; j < NL; j++)
#pragma unroll
            for (int i = 0; i < C; i++) {
                go[j][i] = !decltype(uneven)::value || __any(n[j][i] > t);
                if (go[j][i]) {
#pragma unroll
                    for (int q = 0; q < N; q++) v[j][i][q] = __builtin_amdgcn_raw_buffer_load_b32(r_idx, at[j][i] + 4 * t + 4 * q, 0, 0);
                }
            }
#pragma unroll
        for (int j = 0; j < NL; j++)
#pragma unroll
            for (int i = 0; i < C; i++) {
                if (!go[j][i]) continue;
#pragma unroll
                for (int q = 0; q < N; q++) {
                    int z = v[j][i][q];
                    asm volatile("" : "+v"(z)); // (the load stays where it was asked for, and does not move behind the condition)
                    const int k2 = TRANSPOSED ? off_z - __mul24(z, a.cv.s2) : off_z + z;
                    if ((n[j][i] > t + q) & ((unsigned)k2 < (unsigned)K2)) {
                        const int k = k2 + slot + j * dline + i * dcol;
                        found |= 1u << k;
                        mine[k] = p[j][i] + (tag + t + q);
                    }
                }
            }
    };
    int most = 0;
#pragma unroll
    for (int j = 0; j < NL; j++)
#pragma unroll
        for (int i = 0; i < C; i++) most = max(most, n[j][i]);
    const std::integral_constant<int, 2> two;
    const std::integral_constant<int, 4> four;
    entries(0, two, std::false_type());
    if constexpr (LATER == 2) {
        for (int t = 2; __any(most > t); t += 2) entries(t, two, std::false_type());
    } else if (__any(most > 4)) {
        entries(2, four, std::false_type());
        for (int t = 6; __any(most > t); t += 4) entries(t, four, std::true_type());
    } else if (__any(most > 2)) {
        entries(2, two, std::false_type());
    }

    constexpr int kBatch = 9; // offsets taken together: table entries read at once, and tests against the number of offsets
    // pairs of every offset in the wave's rows: lane k of `count`
    int count = 0;
#pragma unroll
    for (int kb = 0; kb < KVT; kb += kBatch)
        if (KVT < 32 || kb < KV) {
#pragma unroll
            for (int k = kb; k < kb + kBatch && k < KVT; k++)
                if (KVT < 32 || k < KV) {
                    const int pop = __popcll(__builtin_amdgcn_ballot_w64((found & (1u << k)) != 0));
                    asm("v_writelane_b32 %0, %1, %2" : "+v"(count) : "s"(pop), "n"(k));
                }
        }
    if (lane < 32) s_cnt[wave * 32 + lane] = count;
    lds_barrier();
    const int cnt0 = lane < 32 ? s_cnt[lane] : 0, total = cnt0 + (lane < 32 ? s_cnt[32 + lane] : 0);
    const int groups = (total + SPH_GROUP - 1) / SPH_GROUP;
    const int incl = wave_inclusive_sum(groups), first = incl - groups; // first group of offset `lane`
    const int ngrp = __builtin_amdgcn_readlane(incl, kWave - 1);
    const long gbase = (long)tile * a.cap;
    if (wave == 0) {
        if (lane <= KV) a.book.tile_koff[(long)tile * (KV + 1) + lane] = (uint16_t)first;
        if (lane == 0) a.book.tile_ngrp[tile] = ngrp;
    } else {
        for (int g = 0; __any(g < groups); g++)
            if (g < groups) a.book.grp_k[gbase + first + g] = lane;
    }
    const int begin = first * SPH_GROUP + (wave ? cnt0 : 0); // slot of the wave's first pair of offset `lane`
    // the pairs of groups w0 .. w0 + kRowGroups - 1 to their slots
    auto to_slots = [&](int w0, bool all) {
#pragma unroll
        for (int kb = 0; kb < KVT; kb += kBatch) {
            if (KVT == 32 && kb >= KV) continue;
            int e[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; i++) e[i] = mine[min(kb + i, KV - 1)];
            asm volatile("" : "+v"(found)); // (masks of all offsets made beforehand would not fit the scalar registers)
#pragma unroll
            for (int i = 0; i < kBatch; i++) {
                const int k = kb + i;
                if (k < KVT && (KVT < 32 || k < KV)) {
                    const unsigned long long m = __builtin_amdgcn_ballot_w64((found & (1u << k)) != 0);
                    const bool here = __builtin_amdgcn_inverse_ballot_w64(m);
                    const int s = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0)) +
                                  (__builtin_amdgcn_readlane(begin, k) - w0 * SPH_GROUP);
                    if (here & (all | ((unsigned)s < (unsigned)(kRowGroups * SPH_GROUP)))) s_slot[s] = e[i];
                }
            }
        }
    };
    auto store = [&](int w0, int n) {
        const int quads = n * (SPH_GROUP / 4);
        int4 *gat = (int4 *)(a.book.grp_gather + (gbase + w0) * SPH_GROUP), *own = (int4 *)(a.book.grp_owner + (gbase + w0) * SPH_GROUP);
        for (int i = tid; i < quads; i += kRowThreads) {
            const int4 x = ((const int4 *)s_slot)[i];
            const int v4[4] = {x.x, x.y, x.z, x.w};
            int gv[4], ov[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                gv[q] = v4[q] < 0 ? -1 : v4[q] & ((1 << kRowTag) - 1);
                ov[q] = v4[q] < 0 ? -1 : r0 + (int)((unsigned)v4[q] >> kRowTag);
            }
            gat[i] = make_int4(gv[0], gv[1], gv[2], gv[3]);
            own[i] = make_int4(ov[0], ov[1], ov[2], ov[3]);
        }
    };
    if (ngrp <= kRowGroups) {
        to_slots(0, true);
        lds_barrier();
        store(0, ngrp);
        return;
    }
    for (int w0 = 0; w0 < ngrp; w0 += kRowGroups) { // dense neighbourhoods
        if (w0) {
            lds_barrier();
            for (int i = tid; i < kRowGroups * SPH_GROUP / 4; i += kRowThreads) ((int4 *)s_slot)[i] = make_int4(-1, -1, -1, -1);
            lds_barrier();
        }
        to_slots(w0, false);
        lds_barrier();
        store(w0, min(ngrp - w0, kRowGroups));
    }
}

// The kernel for the call's number of lines and of columns on a line (one to three each); with the loops' lengths fixed for 27
// offsets of stride 1, of stride 2 transposed, and of two columns by three lines.
// The rounds of four entries take 84 registers there where rounds of two take 56, and leave less room for the convolution of the
// scan before.  Up to the line where the relay has the compute units to itself, rounds of two are the better ones for scans in flight:
// us a scan, 64 -> 64 fp16 on three streams, four : two, 1 to 3 entries in 60 % of the columns 930 tiles 17.5 : 17.2, 1100 tiles
// 20.7 : 20.4, 1900 tiles 31.0 : 31.1, 4000 tiles 58.5 : 58.7 (Poisson columns 18.0 : 18.1, 21.0 : 21.2, 32.4 : 33.0, 60.9 : 62.3);
// a call on its own 1300 tiles 8.4 : 8.7, 5890 tiles 22.5 : 23.4.
constexpr int kRowFlightTiles = 1280;
template <bool TRANSPOSED, bool HINT>
inline void (*rows_kernel(const BuildArgs &a, int KV, int ntiles))(BuildArgs)
{
    constexpr int cube = TRANSPOSED ? 2 : 3;
    const int nl = rows_lines(a, TRANSPOSED), c = a.lines;
    if (KV == 27 && c == cube && nl == cube) {
        if (!TRANSPOSED && book_says(&a.book) == SPH_RUN_IN_FLIGHT && ntiles <= kRowFlightTiles)
            return build_rows_kernel<false, 3, 3, 27, HINT, 2>;
        return build_rows_kernel<TRANSPOSED, cube, cube, 27, HINT>;
    }
    if (KV == 27 && c == 2 && nl == 3) return build_rows_kernel<TRANSPOSED, 2, 3, 27, HINT>;
#define SPH_ROWS(C, NL) if (c == C && nl == NL) return build_rows_kernel<TRANSPOSED, C, NL, 32, HINT>;
    SPH_ROWS(1, 1) SPH_ROWS(1, 2) SPH_ROWS(1, 3) SPH_ROWS(2, 1) SPH_ROWS(2, 2) SPH_ROWS(2, 3) SPH_ROWS(3, 1) SPH_ROWS(3, 2)
#undef SPH_ROWS
    return build_rows_kernel<TRANSPOSED, 3, 3, 32, HINT>;
}

} // namespace
