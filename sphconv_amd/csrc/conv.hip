// Gather-GEMM-scatter convolution for gfx950 (wave64, MFMA 16x16 tiles).
//
// Forward / dgrad (sph_conv_apply): the tile's pairs arrive as groups of 16 (one
// kernel offset per group).  Fast kernel (conv_wave_kernel): one wave owns a
// 128-row tile (x 64 output columns), gathers each group's 16 feature rows straight
// into MFMA operand registers (16 B per lane), multiplies by the pre-packed weight
// fragments of that offset and adds the result into its private LDS accumulator
// tile; the tile is written to HBM once, with the epilogue fused.  No barriers, no
// atomics, summation order fixed by the book.  Long grids go to relay.hip, which keeps the
// weight in registers.  conv_apply_kernel is the general
// fallback for unaligned or very long rows.  When the book also keeps its pairs by
// stationary row (dense neighbourhoods), conv_rows_kernel_* walks (offset, block of 16
// rows) steps with the accumulators in registers instead; with rows of up to 64 bytes and
// up to 64 output columns conv_rows_win_kernel does so from a copy of the gathered rows
// in LDS.  Before these, rows_hold.hip takes long grids of up to 32 columns, whose weight it
// keeps in LDS, and rows_split.hip grids that do not fill the chip with a wave per tile and
// rows that its larger windows hold.
#include "common.h"
#include "pack.h"
#include "conv_wave.h"
#include "relay.h"
#include "rows_split.h"
#include "rows_hold.h"

#include <cstdlib>

namespace {

// ---------------------------------------------------------------------------
// Weight packing (layout and element copy: pack.h)
// ---------------------------------------------------------------------------
__global__ void pack_weight_kernel(SphPackJobs p)
{
    sph_pack_fragments(p, (int)(blockIdx.x * blockDim.x + threadIdx.x));
}

constexpr int kMetaGroups = 32; // groups whose indices are staged in LDS at a time

// General kernel (any row length and alignment; used when the rows are not a
// multiple of 16 bytes or longer than 256 bytes): NW waves per tile, wave w owns
// columns [16w, 16w+16), one group at a time, every wave gathers for itself.
// The MFMA is issued transposed: D^T[16 owner columns, 16 pairs] = W^T x A^T, so
// lane l ends up with columns 4*(l/16)..+3 of pair l%16.  NSTEP is always 0 (row
// length taken from the arguments).
template <sph_dtype DT, int NW, int NSTEP>
__global__ __launch_bounds__(NW * kWave) void conv_apply_kernel(ConvArgs a)
{
    typedef typename Traits<DT>::elem elem;
    typedef typename Traits<DT>::acc4 acc4;
    constexpr int LDW = NW * 16 + 4; // accumulator row stride in 32-bit words (16-byte multiple)
    extern __shared__ __attribute__((aligned(16))) uint32_t s_acc[]; // [R][LDW]
    __shared__ int s_k[kMetaGroups];
    __shared__ int2 s_meta[kMetaGroups * SPH_GROUP]; // (gathered row, owner row - r0)

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;
    const int tile = sph_xcd_tile(blockIdx.x, (a.book.rows + R - 1) / R);
    const int r0 = tile * R;
    if (r0 >= a.book.rows) return; // grid is padded to a multiple of the XCD count
    const int nrows = min(R, a.book.rows - r0);

    // each wave clears and later updates only its own 16 columns
    for (int i = lane; i < R * 4; i += kWave)
        *(int4v *)&s_acc[(i >> 2) * LDW + wave * 16 + (i & 3) * 4] = int4v{0, 0, 0, 0};

    const int ngrp = a.book.tile_ngrp[tile];
    const long gb0 = (long)tile * a.cap;
    const int acc_col = wave * 16 + (lane >> 4) * 4;
    const char *wlane = a.wp + (long)wave * (kWave * 16) + lane * 16;
    const long wstep = (long)NW * (kWave * 16);           // bytes between steps of one offset
    const int nsteps = NSTEP > 0 ? NSTEP : a.nsteps;

    for (int c0 = 0; c0 < ngrp; c0 += kMetaGroups) {
        const int nc = min(kMetaGroups, ngrp - c0);
        if (c0) __syncthreads(); // every wave is done with the previous chunk's indices
        for (int i = tid; i < nc * SPH_GROUP; i += NW * kWave) {
            int gi = a.book.grp_gather[(gb0 + c0) * SPH_GROUP + i];
            int rl = a.book.grp_owner[(gb0 + c0) * SPH_GROUP + i] - r0;
            if ((unsigned)rl >= (unsigned)nrows || (unsigned)gi >= (unsigned)a.feat_rows) gi = rl = -1;
            s_meta[i] = make_int2(gi, rl);
        }
        for (int i = tid; i < nc; i += NW * kWave) s_k[i] = a.book.grp_k[gb0 + c0 + i];
        __syncthreads();

        {
            for (int g = 0; g < nc; g++) {
                const int2 m = s_meta[g * SPH_GROUP + (lane & 15)];
                const char *wk = wlane + (long)s_k[g] * nsteps * wstep;
                acc4 d = {0, 0, 0, 0};
                for (int st = 0; st < nsteps; st++) {
                    int4v fa = load_a_frag<DT>(a, m.x, st, lane);
                    int4v fb = *(const int4v *)(wk + st * wstep);
                    d = mfma_step<DT>(fb, fa, d);
                }
                if (m.y >= 0) acc_add4<DT>(&s_acc[m.y * LDW + acc_col], d);
            }
        }
    }
    __syncthreads();

    // epilogue: LDS tile -> out rows [r0, r0+nrows), all ndim columns
    elem *out = (elem *)a.out + (long)r0 * a.ndim;
    constexpr int VE = 16 / (int)sizeof(elem);
    if (a.aligned_out) {
        const int cpr = a.ndim / VE; // 16-byte chunks per row
        for (int i = tid; i < nrows * cpr; i += NW * kWave) {
            int row = i / cpr, ch = i - row * cpr;
            union { int4v v; elem e[VE]; } u;
#pragma unroll
            for (int j = 0; j < VE; j++)
                u.e[j] = to_elem<DT>(epilogue_value<DT>(a, s_acc[row * LDW + ch * VE + j], ch * VE + j));
            *(int4v *)(out + (long)row * a.ndim + ch * VE) = u.v;
        }
    } else {
        for (int i = tid; i < nrows * a.ndim; i += NW * kWave) {
            int row = i / a.ndim, c = i - row * a.ndim;
            out[i] = to_elem<DT>(epilogue_value<DT>(a, s_acc[row * LDW + c], c));
        }
    }
}

// ---------------------------------------------------------------------------

template <sph_dtype DT, int NS, int CT, bool MASKED>
__global__ __launch_bounds__(128) void conv_wave_kernel(ConvArgs a, int nwtot)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t s_acc[]; // [R + 1][LDW]
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;              // block of CT*16 columns
    const int tile = sph_xcd_tile(blockIdx.x, (a.book.rows + R - 1) / R);
    const int r0 = tile * R;
    if (r0 >= a.book.rows) return;
    const int nrows = min(R, a.book.rows - r0);
    const int col0 = wave * CT * 16;           // first column of this wave
    const int ngrp = min(max(a.book.tile_ngrp[tile], 0), a.cap);
    const BookMeta meta(a.book, a.cap, tile, ngrp, r0, nrows, a.feat_rows);
    conv_wave_groups<DT, NS, CT, MASKED>(a, nwtot, meta, ngrp, s_acc, col0, lane, true);
    conv_wave_store<DT, CT>(a, nwtot, s_acc, col0, r0, nrows, lane, kWave);
}

// Two tiles at a time, for fp32 rows of 196 to 256 bytes into 33 to 64 columns, where a group of 16 pairs takes 64 matrix instructions of
// 32 cycles, empty slots or not.  At LiDAR sparsity a tile has about one group at an offset and five pairs in it: the last groups
// of two neighbouring tiles at an offset are merged where their pairs fit one.  Two waves take 32 columns each of 256
// accumulator rows, as much LDS for a wave as one that takes 64 columns of one tile.  A row's sum is in conv_wave_kernel's order.
// Where merging would save less than a quarter of the groups, or the list has no room, each wave takes one tile as conv_wave_kernel does.
// What bounds it: in conv_wave_kernel the matrix cores, 69 % of the time with two slots of three empty; here the rows and fragments,
// 12 KB for a group and wave (a quarter more than half of what one wave with all columns loads), and two round trips more to make the list.
// us, 64 -> 64: strided layer of eight 64x512x512 scans, 2848 tiles, 117.7 -> 96.4.  Rows and fragments requested as far ahead as conv_wave_groups does, two groups of 1024 cycles:
// no gain (124); five 104 to 112, six 102 to 108 (behind 62 loads a wave cannot have more counted).
constexpr int kPairRoom = 104;   // merged groups that fit the LDS beside the accumulators of two workgroups per compute unit
constexpr int kPairRows = 2 * R;
constexpr int kPairLists = kPairRoom * (SPH_GROUP * 5 + 4 + 4 + 1); // gat, desc, count of the first, own, gk
// The merged groups into 32 columns of the two tiles' rows.  A group is 32 matrix instructions here, half as long as in conv_wave_groups, so rows
// and fragments are requested kPairAhead groups ahead (a wave has its SIMD to itself: 512 registers).
constexpr int kPairAhead = 6;
template <int NS, bool MASKED>
__device__ __forceinline__ void pair_groups(const ConvArgs &a, int nwtot, const int32_t *gat, const unsigned char *own, const unsigned char *gk,
                                            int total, uint32_t *s_acc, int col0, int lane)
{
    constexpr int CT = 2, D = kPairAhead;
    const int LDW = nwtot * 16 + 4, wstep = nwtot * (kWave * 16);
    const __amdgpu_buffer_rsrc_t r_feat = __builtin_amdgcn_make_buffer_rsrc((void *)a.feat, 0, a.feat_rows * a.row_bytes, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_w = __builtin_amdgcn_make_buffer_rsrc((void *)a.wp, 0, a.book.KV * NS * wstep, kRsrcFlags);
    const int w_lane = (col0 / 16) * (kWave * 16) + lane * 16, chunk = (lane >> 4) * 16, acc_lane = (col0 + (lane >> 4) * 4) * 4;
    if (total == 0) { // tiles without a pair (rows no output reaches): there is no last group to ask for in a group's place
        conv_wave_clear<CT, kPairRows>(s_acc, LDW, col0, lane);
        return;
    }
    int4v x[D][NS], w[D][NS][CT];
    struct Entry { int gi, k; };
    auto entry = [&](int j) -> Entry { // (behind the last group: that one again)
        const int g = min(j, total - 1);
        return Entry{gat[g * SPH_GROUP + (lane & 15)], gk[g]};
    };
    auto acc_row = [&](int j) -> uint32_t * {
        const int g = min(j, total - 1), at = g * SPH_GROUP + (lane & 15);
        const int row = j < total && gat[at] >= 0 ? own[at] : kPairRows;
        return (uint32_t *)((char *)s_acc + (int)__umul24(row, LDW * 4) + acc_lane);
    };
    auto load = [&](const Entry &e, int4v (&xs)[NS], int4v (&ws)[NS][CT], int st) {
        const int off = (int)__umul24((unsigned)max(e.gi, 0), (unsigned)a.row_bytes) + chunk, k = __builtin_amdgcn_readfirstlane(e.k);
        xs[st] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(r_feat, off + st * 64, 0, 0));
#pragma unroll
        for (int c = 0; c < CT; c++)
            ws[st][c] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(r_w, w_lane + st * wstep + c * (kWave * 16), k * (NS * wstep), 0));
    };
#pragma unroll
    for (int d = 0; d < D; d++) {
        const Entry e = entry(d);
#pragma unroll
        for (int st = 0; st < NS; st++) load(e, x[d], w[d], st);
        __builtin_amdgcn_sched_barrier(0);
    }
    conv_wave_clear<CT, kPairRows>(s_acc, LDW, col0, lane);
    Entry next = entry(D);
    uint32_t *p = acc_row(0);
    for (int j0 = 0; j0 < total; j0 += D) {
#pragma unroll
        for (int d = 0; d < D; d++) {
            const int j = j0 + d;
            float4v acc[CT];
#pragma unroll
            for (int c = 0; c < CT; c++) acc[c] = *(const float4v *)(p + c * 16);
            const Entry e = next;
            next = entry(j + D + 1);
            uint32_t *p_next = acc_row(j + 1);
#pragma unroll
            for (int st = 0; st < NS; st++) {
                int4v v = x[d][st];
                if constexpr (MASKED) {
                    const bool live = st * 64 + chunk < a.row_bytes;
                    v = live ? v : int4v{0, 0, 0, 0};
                }
#pragma unroll
                for (int c = 0; c < CT; c++) acc[c] = mfma_step<SPH_F32>(w[d][st][c], v, acc[c]);
                load(e, x[d], w[d], st);
            }
#pragma unroll
            for (int c = 0; c < CT; c++) *(float4v *)(p + c * 16) = acc[c];
            p = p_next;
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

template <int NS, bool MASKED>
__global__ __launch_bounds__(2 * kWave) __attribute__((amdgpu_waves_per_eu(1))) void conv_wave_pair_kernel(ConvArgs a, int nwtot)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t s_acc[]; // [kPairRows + 1][LDW], then the merged groups
    const int LDW = nwtot * 16 + 4;
    int32_t *s_gat = (int32_t *)(s_acc + (kPairRows + 1) * LDW), *s_desc = s_gat + kPairRoom * SPH_GROUP, *s_first = s_desc + kPairRoom;
    unsigned char *s_own = (unsigned char *)(s_first + kPairRoom), *s_gk = s_own + kPairRoom * SPH_GROUP;
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int ntiles = (a.book.rows + R - 1) / R, npairs = (ntiles + 1) / 2;
    const int pair = sph_xcd_tile(blockIdx.x, npairs);
    if (pair >= npairs) return; // whole workgroups leave
    const int r0 = pair * kPairRows, nrows = min(kPairRows, a.book.rows - r0), KV = a.book.KV;
    const int col0 = wave * 32;
    const int tile[2] = {2 * pair, min(2 * pair + 1, ntiles - 1)};
    const bool two = 2 * pair + 1 < ntiles;

    // (each offset can save one group, so with more than four of them to an offset merging is out of the question)
    int ng[2];
#pragma unroll
    for (int t = 0; t < 2; t++) ng[t] = t == 0 || two ? min(max(a.book.tile_ngrp[tile[t]], 0), a.cap) : 0;
    const bool few = ng[0] + ng[1] <= 4 * KV;
    // lane k: the tiles' groups at offset k, and how many slots of the last ones are taken (both waves find the same)
    int g0[2] = {}, n[2] = {}, taken[2] = {};
    if (few) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const unsigned short *ko = a.book.tile_koff + (long)tile[t] * (KV + 1) + min(lane, KV - 1);
            g0[t] = min((int)ko[0], a.cap);
            n[t] = lane < KV && (t == 0 || two) ? min(max((int)ko[1] - g0[t], 0), a.cap - g0[t]) : 0;
        }
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int g = min(g0[t] + max(n[t] - 1, 0), a.cap - 1);
            const int4v *e = (const int4v *)(a.book.grp_gather + ((long)tile[t] * a.cap + g) * SPH_GROUP);
            int last = 0;
#pragma unroll
            for (int i = 0; i < SPH_GROUP / 4; i++) {
                const int4v v = e[i];
#pragma unroll
                for (int j = 0; j < 4; j++) last = v[j] >= 0 ? i * 4 + j + 1 : last;
            }
            taken[t] = last;
        }
    }
    const bool merge = n[0] > 0 && n[1] > 0 && taken[0] + taken[1] <= SPH_GROUP;
    const int mine = n[0] + n[1] - (merge ? 1 : 0);
    const int incl = wave_inclusive_sum(mine);
    const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
    const int apart = __builtin_amdgcn_readlane(wave_inclusive_sum(n[0] + n[1]), kWave - 1);
    if (few && total <= kPairRoom && total * 4 <= apart * 3) {
        // where group j of the list comes from: the group of the first tile in the low half, of the second in the high one (0xffff: none)
        if (wave == 0)
            for (int i = 0, j = incl - mine; i < mine; i++, j++) {
                const bool both = merge && i == n[0] - 1;
                const bool first = i < n[0];
                const int ib = merge ? i - n[0] + 1 : i - n[0]; // the second tile's: its last one first, where it is merged
                const int gb = merge ? (ib == 0 ? n[1] - 1 : ib - 1) : ib;
                s_desc[j] = (first ? g0[0] + i : 0xffff) | (!first || both ? g0[1] + gb : 0xffff) << 16;
                s_first[j] = first ? (both ? taken[0] : SPH_GROUP) : 0;
                s_gk[j] = (unsigned char)lane;
            }
        lds_barrier();
        for (int i = tid; i < total * SPH_GROUP; i += 2 * kWave) {
            const int j = i / SPH_GROUP, s = i % SPH_GROUP, d = s_desc[j], nf = s_first[j];
            const bool first = s < nf;
            const unsigned g = first ? d & 0xffff : (unsigned)d >> 16;
            const long slot = ((long)(first ? tile[0] : tile[1]) * a.cap + min(g, (unsigned)a.cap - 1)) * SPH_GROUP + (first ? s : s - nf);
            const int gi = a.book.grp_gather[slot], ow = a.book.grp_owner[slot] - r0;
            const bool ok = g != 0xffff && (unsigned)gi < (unsigned)a.feat_rows && (unsigned)ow < (unsigned)nrows;
            s_gat[i] = ok ? gi : -1;
            s_own[i] = (unsigned char)ow;
        }
        lds_barrier();
        pair_groups<NS, MASKED>(a, nwtot, s_gat, s_own, s_gk, total, s_acc, col0, lane);
        conv_wave_store<SPH_F32, 2>(a, nwtot, s_acc, col0, r0, nrows, lane, kWave);
    } else {
        // too full for the list, or for merging to pay: a wave takes all columns of one tile
        const int first = wave * R;
        if (first < nrows) {
            const int mine = wave ? ng[1] : ng[0];
            const BookMeta meta(a.book, a.cap, 2 * pair + wave, mine, r0, nrows, a.feat_rows);
            conv_wave_clear<4, R - 1>(s_acc + first * LDW, LDW, 0, lane); // (the row for slots without a pair is both waves', and nobody's result)
            conv_wave_groups<SPH_F32, NS, 4, MASKED, kPairRows>(a, nwtot, meta, mine, s_acc, 0, lane, false);
            conv_wave_store<SPH_F32, 4>(a, nwtot, s_acc + first * LDW, 0, r0 + first, min(R, nrows - first), lane, kWave);
        }
    }
}
inline size_t pair_lds(int nwtot) { return (size_t)(kPairRows + 1) * (nwtot * 16 + 4) * 4 + kPairLists; }

// The same with two helper waves per tile (up to 64 output columns, rows of up to 128 bytes).  A submanifold book
// has a run of up to eight full groups at the middle offset (every row's pair with itself), which all use one set
// of weight fragments: the helper waves load those fragments once, take the run's groups between them, multiply
// from zero and store the products to the owners' accumulator rows behind wave 0's clear and before its first
// sum, while wave 0's first rows and fragments are on their way.  Wave 0's chain is then the tile's other groups
// only (26 instead of 34 at LiDAR sparsity), and the run costs 8 fragment loads instead of 64.  A tile whose middle
// offset holds fewer than two groups (strided books) is wave 0's alone, and the helper waves leave at once.
constexpr int kRunHelpers = 2;
template <sph_dtype DT, int NS, int CT, bool MASKED>
__global__ __launch_bounds__(kWave * (1 + kRunHelpers)) __attribute__((amdgpu_waves_per_eu(3))) void conv_wave_run_kernel(ConvArgs a, int nwtot)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t s_acc[]; // [R + 1][LDW]
    constexpr int kRun = (R / SPH_GROUP + kRunHelpers - 1) / kRunHelpers;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;
    const int tile = sph_xcd_tile(blockIdx.x, (a.book.rows + R - 1) / R);
    const int r0 = tile * R;
    if (r0 >= a.book.rows) return;
    const int nrows = min(R, a.book.rows - r0);
    const int KV = a.book.KV, kc = KV / 2;
    const int ngrp = min(max(a.book.tile_ngrp[tile], 0), a.cap);
    const unsigned short *ko = a.book.tile_koff + (long)tile * (KV + 1) + kc;
    const int run_lo = min((int)ko[0], ngrp);
    const int run_n = min(max((int)ko[1] - run_lo, 0), min(ngrp - run_lo, R / SPH_GROUP));
    const bool shared = run_n >= 2; // workgroup-uniform
    if (wave == 0) {
        const BookMeta meta(a.book, a.cap, tile, shared ? ngrp - run_n : ngrp, r0, nrows, a.feat_rows, run_lo, shared ? run_n : 0);
        conv_wave_groups<DT, NS, CT, MASKED>(a, nwtot, meta, meta.ngrp, s_acc, 0, lane, true, shared ? 2 : 0);
    } else {
        if (!shared) return;
        const BookMeta meta(a.book, a.cap, tile, ngrp, r0, nrows, a.feat_rows);
        conv_run_store<DT, NS, CT, MASKED, kRun>(a, nwtot, meta, kc, run_lo + wave - 1, kRunHelpers, run_lo + run_n, lane, s_acc,
                                                 nullptr, -1, 0, true);
        lds_barrier();
    }
    if (shared) { // the helper waves have waited for the tile: all three write it out
        lds_barrier();
        conv_wave_store<DT, CT>(a, nwtot, s_acc, 0, r0, nrows, tid, kWave * (1 + kRunHelpers));
    } else {
        conv_wave_store<DT, CT>(a, nwtot, s_acc, 0, r0, nrows, lane, kWave);
    }
}

// A grid that the chip holds at once lasts as long as one tile's chain of groups, so the S waves of a workgroup share the
// tile's groups: each adds its share into accumulators of its own (up to 64 output columns), and the copies are summed as
// the tile is written, in the waves' order.  S is the most that still lets every tile be resident (LDS); see
// split_waves().  A tile whose groups are few is all set-up and store; one of a denser stage (70 to 100 groups) is where
// this counts.
template <sph_dtype DT, int NS, int CT, bool MASKED, int S>
__global__ __launch_bounds__(kWave * S) __attribute__((amdgpu_waves_per_eu(1))) void conv_wave_split_kernel(ConvArgs a, int nwtot)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t s_acc[]; // [S][R + 1][LDW]
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;
    const int tile = sph_xcd_tile(blockIdx.x, (a.book.rows + R - 1) / R);
    const int r0 = tile * R;
    if (r0 >= a.book.rows) return;
    const int nrows = min(R, a.book.rows - r0);
    const int ngrp = min(max(a.book.tile_ngrp[tile], 0), a.cap);
    int base, n;
    group_share(ngrp, S, wave, base, n);
    BookMeta meta(a.book, a.cap, tile, n, r0, nrows, a.feat_rows);
    meta.base = base;
    conv_wave_groups<DT, NS, CT, MASKED>(a, nwtot, meta, n, s_acc + wave * (R + 1) * (nwtot * 16 + 4), 0, lane, true);
    lds_barrier();
    conv_wave_store<DT, CT, S>(a, nwtot, s_acc, 0, r0, nrows, tid, kWave * S);
}

// ---------------------------------------------------------------------------
// Walk by stationary row (book.tile_nbr): for dense neighbourhoods.
//
// The grouped kernel above pays per group of 16 pairs (weight fragments through the L1,
// an LDS read-modify-write of the owners' accumulators), which is the right price when a
// row has two or three pairs.  From about ten pairs per row upwards it is cheaper to take
// every (offset, block of 16 consecutive rows) in turn, whatever it holds: the 16 gathered
// rows (zeros where a row has no pair at this offset) times the offset's weight, added to
// accumulators that never leave the registers (8 blocks x 64 columns = 128 per lane).
// 27 weight loads per tile instead of one per group, no accumulators in LDS, no owner
// indirection; the price is one MFMA step per (offset, block) even when it is nearly empty.
// One wave per tile and 64 output columns.  The tile's table is staged in LDS; gathers are
// requested two to four stages (of 4 sixteen-byte chunks per lane) ahead of their use.
// Measured at 64->64 fp16 on a full grid: 164 us against 387 us by groups; without any
// load the same instruction stream takes 91 us, twice what its MFMAs alone need (independent
// 16x16x32 MFMAs issue every 16 cycles): a stage's selects, LDS exchange and waits are in
// series with its MFMAs, and two waves per SIMD do not cover them.
// ---------------------------------------------------------------------------
// (Short grids, and long ones of 128-byte rows whose rows lie close together, share a row's offsets between waves: rows_split.hip; long
// grids into 17 to 32 columns keep the weight in LDS: rows_hold.hip.)
template <sph_dtype DT, int NS, int CT, bool MASKED>
__device__ __forceinline__ void conv_rows_body(const ConvArgs &a, int nwtot)
{
    typedef typename Traits<DT>::elem elem;
    typedef typename Traits<DT>::acc4 acc4;
    constexpr int NB = R / SPH_GROUP;      // blocks of 16 rows
    constexpr int BPS = 4 / NS;            // blocks per stage: a stage gathers up to 4 sixteen-byte chunks per lane
    constexpr int SPK = NB / BPS;         // stages per offset
    // measured: 128-byte rows want four stages of gathers in flight and one set of weight registers; 64-byte
    // rows (few MFMAs per stage) two stages and the next offset's weights requested an offset ahead
    constexpr int D = NS >= 2 ? 4 : 2;     // stages in flight
    constexpr int KW = NS >= 2 ? 1 : 2;    // sets of weight fragment registers
    constexpr int U = (D > SPK * KW) ? D : SPK * KW; // stages per unrolled round (all powers of two)
    extern __shared__ __attribute__((aligned(16))) int32_t s_nb[]; // [KV][R] gathered row or -1

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;          // block of CT*16 columns
    const int tile = sph_xcd_tile(blockIdx.x, (a.book.rows + R - 1) / R);
    const int r0 = tile * R;
    if (r0 >= a.book.rows) return; // whole workgroups leave: no barrier is missed
    const int nrows = min(R, a.book.rows - r0);
    const int col0 = wave * CT * 16;
    const int KV = a.book.KV;
    const int S = KV * SPK;
    const char *wlane = a.wp + ((long)(wave * CT)) * (kWave * 16) + lane * 16;
    const long wstep = (long)nwtot * (kWave * 16);

    // the tile's table goes to LDS once (validated on the way): every stage then finds its rows
    // with one LDS read per block instead of a dependent global load
    {
        const int4v *src = (const int4v *)(a.book.tile_nbr + (long)tile * KV * R);
        for (int i = tid; i < KV * R / 4; i += blockDim.x) {
            int4v v = src[i];
            v.x = (unsigned)v.x < (unsigned)a.feat_rows ? v.x : -1;
            v.y = (unsigned)v.y < (unsigned)a.feat_rows ? v.y : -1;
            v.z = (unsigned)v.z < (unsigned)a.feat_rows ? v.z : -1;
            v.w = (unsigned)v.w < (unsigned)a.feat_rows ? v.w : -1;
            ((int4v *)s_nb)[i] = v;
        }
    }
    __syncthreads();

    // Gathers are requested with the four lanes of a quad on the four 16-byte chunks of ONE row's 64-byte
    // step (one tag look-up per quad; with a lane per row of the MFMA layout every quad would touch four
    // rows).  They reach the MFMA layout (lane = pair + 16 * chunk) through a wave-private LDS buffer:
    // [chunk set][16 rows][80 bytes] (the 16-byte pad makes both the write and the read conflict-free).
    // With 64-byte rows (one step) the exchange costs more than the look-ups it saves: there a lane loads
    // its MFMA operand directly.
    constexpr bool QUAD = NS >= 2;
    constexpr int kTrRow = 80, kTrSet = SPH_GROUP * kTrRow;
    char *tr = (char *)(s_nb + KV * R) + (tid / kWave) * (BPS * NS * kTrSet);
    int4v fa[D][BPS][NS], fw[KW][NS][CT];
    int rq[D][BPS];
    acc4 acc[NB][CT];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int c = 0; c < CT; c++) acc[j][c] = acc4{0, 0, 0, 0};

    // stage s = (k, q): offset k = s / SPK, blocks q*BPS .. q*BPS+BPS-1 of the tile, every 64-byte step of
    // their rows; stages past the end re-read the last offset
    auto issue = [&](int s, int q, int4v (&f)[BPS][NS], int (&rows)[BPS]) {
        const int k = min(s / SPK, KV - 1);
#pragma unroll
        for (int j = 0; j < BPS; j++) {
            rows[j] = s_nb[k * R + (q * BPS + j) * SPH_GROUP + (QUAD ? lane >> 2 : lane & 15)];
            const char *row = a.feat + (long)max(rows[j], 0) * a.row_bytes;
#pragma unroll
            for (int st = 0; st < NS; st++) {
                const int off = st * 64 + (QUAD ? lane & 3 : lane >> 4) * 16;
                f[j][st] = *(const int4v *)(row + (off < a.row_bytes ? off : 0));
            }
        }
    };
    auto load_w = [&](int k, int4v (&w)[NS][CT]) {
        const char *wk = wlane + (long)min(k, KV - 1) * NS * wstep;
#pragma unroll
        for (int st = 0; st < NS; st++)
#pragma unroll
            for (int c = 0; c < CT; c++) w[st][c] = *(const int4v *)(wk + st * wstep + (long)c * (kWave * 16));
    };

#pragma unroll
    for (int p = 0; p < KW; p++) load_w(p, fw[p]);
#pragma unroll
    for (int u = 0; u < D; u++) issue(u, u % SPK, fa[u], rq[u]);
    for (int s0 = 0; s0 < S; s0 += U) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int s = s0 + u;
            const int d = u % D, q = u % SPK, p = (u / SPK) % KW; // compile-time after unrolling
            __builtin_amdgcn_sched_barrier(0);
            if (s < S) {
                // zeros for rows without a pair and beyond the row's end; quad layout -> LDS -> MFMA layout
                int4v x[BPS][NS];
#pragma unroll
                for (int j = 0; j < BPS; j++)
#pragma unroll
                    for (int st = 0; st < NS; st++) {
                        bool live = rq[d][j] >= 0;
                        if constexpr (MASKED) live = live && (st * 64 + (QUAD ? lane & 3 : lane >> 4) * 16 < a.row_bytes);
                        x[j][st] = live ? fa[d][j][st] : int4v{0, 0, 0, 0};
                        if constexpr (QUAD)
                            *(int4v *)(tr + (j * NS + st) * kTrSet + (lane >> 2) * kTrRow + (lane & 3) * 16) = x[j][st];
                    }
                if constexpr (QUAD) {
                    asm volatile("" ::: "memory"); // other lanes' chunks: keep the reads behind the writes
#pragma unroll
                    for (int j = 0; j < BPS; j++)
#pragma unroll
                        for (int st = 0; st < NS; st++)
                            x[j][st] = *(const int4v *)(tr + (j * NS + st) * kTrSet + (lane & 15) * kTrRow + (lane >> 4) * 16);
                }
                asm volatile("" ::: "memory");
#pragma unroll
                for (int j = 0; j < BPS; j++)
#pragma unroll
                    for (int st = 0; st < NS; st++)
#pragma unroll
                        for (int c = 0; c < CT; c++)
                            acc[q * BPS + j][c] = mfma_step<DT>(fw[p][st][c], x[j][st], acc[q * BPS + j][c]);
            }
            __builtin_amdgcn_sched_barrier(0);
            // the offset is done: its weight registers take the fragments of offset k + KW; the row buffers
            // just consumed take stage s + D
            if (q == SPK - 1) load_w(s / SPK + KW, fw[p]);
            issue(s + D, (u + D) % SPK, fa[d], rq[d]);
        }
    }

    // epilogue: a lane holds four consecutive columns of one row per block and column tile
    const bool plain = DT != SPH_I8 && !a.scale && !a.shift && !a.relu;
    const bool relu = DT != SPH_I8 && a.relu;
    float sc[CT][4], sh[CT][4];
#pragma unroll
    for (int c = 0; c < CT; c++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int col = min(col0 + c * 16 + (lane >> 4) * 4 + j, a.ndim - 1);
            sc[c][j] = a.scale ? a.scale[col] : 1.f;
            sh[c][j] = (DT != SPH_I8 && a.shift) ? a.shift[col] : 0.f;
        }
    elem *out = (elem *)a.out + (long)r0 * a.ndim;
    auto store_block = [&](int b, const acc4 (&ac)[CT]) {
        const int row = b * SPH_GROUP + (lane & 15);
        if (row >= nrows) return;
#pragma unroll
        for (int c = 0; c < CT; c++) {
            const int col = col0 + c * 16 + (lane >> 4) * 4;
            if (col >= a.ndim) continue;
            union { elem e[4]; uint32_t w[sizeof(elem)]; } u;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float v = DT == SPH_I8 ? (float)(int)ac[c][j] : (float)ac[c][j];
                if (!plain) {
                    v = v * sc[c][j] + sh[c][j];
                    if (relu) v = v > 0.f ? v : 0.f;
                }
                u.e[j] = to_elem<DT>(v);
            }
            uint32_t *dst = (uint32_t *)(out + (long)row * a.ndim + col);
#pragma unroll
            for (int q = 0; q < (int)sizeof(elem); q++) dst[q] = u.w[q];
        }
    };
#pragma unroll
    for (int j = 0; j < NB; j++) store_block(j, acc[j]);
}

// The accumulators of a wave are CT*32 registers; the wrappers tell the compiler how many waves per
// SIMD to leave room for (4 column tiles: 2, 2 tiles: 3, 1 tile: 4), i.e. how many registers the
// gathers in flight may take.
template <sph_dtype DT, int NS, int CT, bool MASKED>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2))) void conv_rows_kernel_w2(ConvArgs a, int nwtot)
{
    conv_rows_body<DT, NS, CT, MASKED>(a, nwtot);
}
template <sph_dtype DT, int NS, int CT, bool MASKED>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(3))) void conv_rows_kernel_w3(ConvArgs a, int nwtot)
{
    conv_rows_body<DT, NS, CT, MASKED>(a, nwtot);
}
template <sph_dtype DT, int NS, int CT, bool MASKED>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(4))) void conv_rows_kernel_w4(ConvArgs a, int nwtot)
{
    conv_rows_body<DT, NS, CT, MASKED>(a, nwtot);
}

// ---------------------------------------------------------------------------
// By stationary row, gathered rows staged in LDS: rows of up to 64 bytes (one MFMA K step), up to 64
// output columns, one or two waves per tile.
//
// With one K step a (offset, block) step is one or two MFMAs behind a gather of 16 rows; the plain by-row
// kernel then waits for its gathers (every one a miss of the vector L1: a tile's 27 offsets ask for each
// neighbouring row about ten times, with the other waves' traffic in between).  The rows a tile's offsets
// gather lie close together in the feature array: for 9 consecutive offsets (one value of k0 in a 3x3x3
// kernel) they are the tile's own range of rows of one line of the grid, a column more on either side.
// So the offsets are taken in phases of 9: the tile's waves, with 128 or 64 rows each, find the range [lo, hi]
// of rows the phase gathers, bring it to LDS as it lies (direct global -> LDS loads, all in flight at once),
// rewrite the phase's table as one byte per (offset, row) (place in the window; slots without a pair point at
// a row of zeros behind it), and every step's gather is then one 16-byte LDS read per lane, with nothing to
// select afterwards.  A phase whose rows do not fit the window (a tile that straddles two lines of the grid,
// strided layers with wide footprints) gathers from the feature array instead.  The order of summation
// per row is the plain kernel's (offsets ascending), so results are bit-identical.
// What bounds it: the round trips of the windows.  On 12 744 tiles, 32 -> 32, waves wait for memory 58 % of their
// time, the vector memory path is 64 % busy (two fifths of it weight fragments), the LDS 37 %, the matrix cores 27 %.
// With one wave per tile (256 registers: two waves per SIMD) there was less to fill the waits with; two halve a
// wave's accumulators and table, so three waves share a SIMD, with one window for two of them, at the price of
// twice the weight loads.  us, one wave a tile -> two, fp16: 32 -> 32 on 12 744 tiles (10.9 pairs a row)
// 154.6 -> 146.7, 16 -> 32 149.0 -> 140.1; on 4056 tiles (24.8 pairs) 74.3 -> 61.2; on 1248 tiles 23.3 -> 18.2 (where one
// wave is the better one: win_one_wave).  With the registers of one wave there was no room for 64 columns either; with two it
// depends (win_ok).  Held to four waves per SIMD (128 registers) it spills and takes 245 us.
// ---------------------------------------------------------------------------
constexpr int kWinPhase = 9;           // offsets per window
constexpr int kWinBytes = 16 * 1024;   // bytes of feature rows a window holds (up to 255 rows)
constexpr int kWinTab = kWinPhase * R; // one byte per (offset, row)
constexpr int kWinMaxRows = 255;       // most rows of a window: a byte names any of them or the row of zeros

// W: waves of a tile, R / W rows each, with one window.
template <sph_dtype DT, int CT, bool MASKED, int W>
__global__ __launch_bounds__(W * kWave) __attribute__((amdgpu_waves_per_eu(CT == 4 || W == 1 ? 2 : 3))) void conv_rows_win_kernel(ConvArgs a, int nwtot)
{
    typedef typename Traits<DT>::elem elem;
    typedef typename Traits<DT>::acc4 acc4;
    constexpr int RW = R / W;                // rows of a wave
    constexpr int RL = RW / kWave;           // of which a lane brings the table's entries
    constexpr int NB = RW / SPH_GROUP;       // blocks of 16 rows
    constexpr int HB = CT == 4 ? 2 : 4;      // blocks per stage
    constexpr int SPO = NB / HB;             // stages per offset
    constexpr int WR = 3;                    // sets of weight fragments: requested three offsets ahead
    static_assert(kWinPhase % WR == 0, "the ring must divide a phase");
    extern __shared__ __attribute__((aligned(16))) char s_mem[];
    __shared__ int2 s_range[2][W];   // rows a wave's part of the phase gathers, by the phase's parity
    const int lane = threadIdx.x & (kWave - 1);
    const int part = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    uint8_t *s_tab = (uint8_t *)s_mem + part * (kWinPhase * RW); // [kWinPhase][SPO][16 rows][HB blocks], a wave's own
    char *s_win = s_mem + kWinTab;           // the window's rows, as they lie in the feature array
    int32_t *s_tab32 = (int32_t *)s_win + part * (kWinPhase * RW); // a phase without a window: [kWinPhase][RW] rows of the feature array

    const int tile = sph_xcd_tile(blockIdx.x, (a.book.rows + R - 1) / R);
    const int r0 = tile * R;
    if (r0 >= a.book.rows) return;
    const int nrows = min(R, a.book.rows - r0);
    const int KV = a.book.KV;
    const int rb = a.row_bytes;
    const int nph = (KV + kWinPhase - 1) / kWinPhase;
    const char *wlane = a.wp + lane * 16;
    const long wstep = (long)nwtot * (kWave * 16);
    const int chunk = lane >> 4;
    const bool live_chunk = chunk * 16 < rb;
    const int choff = live_chunk ? chunk * 16 : 0;

    acc4 acc[NB][CT];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int c = 0; c < CT; c++) acc[j][c] = acc4{0, 0, 0, 0};

    int tn[kWinPhase][RL]; // the next phase's table, on its way while this phase is worked through
    auto load_tab = [&](int ph) {
        const int k0 = min(ph, nph - 1) * kWinPhase;
        const int32_t *src = a.book.tile_nbr + ((long)tile * KV + k0) * R + part * RW + lane;
#pragma unroll
        for (int i = 0; i < kWinPhase; i++)
#pragma unroll
            for (int r = 0; r < RL; r++) tn[i][r] = src[min(i, KV - 1 - k0) * R + r * kWave];
    };
    auto load_w = [&](int k, int4v (&w)[CT]) {
        const char *wk = wlane + (long)min(k, KV - 1) * wstep;
#pragma unroll
        for (int c = 0; c < CT; c++) w[c] = *(const int4v *)(wk + (long)c * (kWave * 16));
    };

    int4v wr[WR][CT];
    load_tab(0);
#pragma unroll
    for (int i = 0; i < WR; i++) load_w(i, wr[i]);
    for (int ph = 0; ph < nph; ph++) {
        const int k0 = ph * kWinPhase;
        const int nk = min(kWinPhase, KV - k0);
        // this phase's table: validate, find the range of rows it gathers
        int t[kWinPhase][RL], lo = 0x7fffffff, hi = -1;
#pragma unroll
        for (int i = 0; i < kWinPhase; i++)
#pragma unroll
            for (int r = 0; r < RL; r++) {
                t[i][r] = (i < nk && (unsigned)tn[i][r] < (unsigned)a.feat_rows) ? tn[i][r] : -1;
                lo = (int)min((unsigned)lo, (unsigned)t[i][r]); // (-1 is the largest unsigned number)
                hi = max(hi, t[i][r]);
            }
        lo = ~wave_max_last(~lo); // lowest: 0x7fffffff, a lane without a pair, is the least of the complements
        hi = wave_max_last(hi);
        // direct loads write LDS behind the back of the LDS unit's own queue: the last phase's reads must
        // have returned before the window is overwritten
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (lane == kWave - 1) s_range[ph & 1][part] = make_int2(lo, hi);
        lds_barrier();
        lo = min(s_range[ph & 1][0].x, s_range[ph & 1][W - 1].x);
        hi = max(s_range[ph & 1][0].y, s_range[ph & 1][W - 1].y);
        lo = __builtin_amdgcn_readfirstlane(lo);
        hi = __builtin_amdgcn_readfirstlane(hi);
        if (hi < 0) { // no pair at these offsets
            load_tab(ph + 1);
#pragma unroll
            for (int i = 0; i < WR; i++) load_w(k0 + kWinPhase + i, wr[i]);
            continue;
        }
        // a window holds rows lo..hi and, behind them, one row of zeros that slots without a pair read
        const int nrow = hi - lo + 1;
        const bool win = nrow <= kWinMaxRows && nrow * rb <= kWinBytes;
        if (win) {
#pragma unroll
            for (int i = 0; i < kWinPhase; i++)
#pragma unroll
                for (int r = 0; r < RL; r++) {
                    const int blk = r * (kWave / SPH_GROUP) + (lane >> 4);
                    s_tab[i * RW + blk / HB * (SPH_GROUP * HB) + (lane & 15) * HB + blk % HB] =
                        (uint8_t)(t[i][r] >= 0 ? t[i][r] - lo : nrow);
                }
            // lane l of load i fills the 16 bytes at i * 1024 + l * 16 of the window
            const int nbytes = nrow * rb;
            const int nld = (nbytes + kWave * 16 - 1) / (kWave * 16);
            const char *src = a.feat + (long)lo * rb;
            for (int i = part; i < nld; i += W) {
                const char *g = src + min((i * kWave + lane) * 16, nbytes - 16);
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)g,
                                                 (__attribute__((address_space(3))) void *)(s_win + i * (kWave * 16)), 16, 0, 0);
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            lds_barrier();
            load_tab(ph + 1);
            if (lane * 16 < rb) *(int4v *)(s_win + nbytes + lane * 16) = int4v{0, 0, 0, 0}; // behind the loads: their last kilobyte may reach here
            // stages (offset, HB blocks): table entries two stages ahead, rows one stage ahead
            constexpr int ns = kWinPhase * SPO;
            auto tab = [&](int st, int (&id)[HB]) {
                const int sc = min(st, ns - 1);
                const uint8_t *p = s_tab + (sc / SPO) * RW + (sc % SPO) * (SPH_GROUP * HB) + (lane & 15) * HB;
                const uint32_t pk = HB == 4 ? *(const uint32_t *)p : *(const uint16_t *)p;
#pragma unroll
                for (int j = 0; j < HB; j++) id[j] = (pk >> (8 * j)) & 255;
            };
            auto rows = [&](const int (&id)[HB], int4v (&x)[HB]) {
#pragma unroll
                for (int j = 0; j < HB; j++) {
                    // lanes on 16-byte chunks behind the row's end read zeros too
                    const int r = (MASKED && !live_chunk) ? nrow : id[j];
                    x[j] = *(const int4v *)(s_win + (__umul24(r, rb) + choff));
                }
            };
            int id1[HB], id2[HB];
            int4v x1[HB];
            tab(0, id1);
            tab(1, id2);
            rows(id1, x1);
            auto round = [&](int k9) {
#pragma unroll
                for (int i = 0; i < WR; i++) {
#pragma unroll
                    for (int h = 0; h < SPO; h++) {
                        const int st = (k9 + i) * SPO + h;
                        int4v xc[HB];
#pragma unroll
                        for (int j = 0; j < HB; j++) { xc[j] = x1[j]; id1[j] = id2[j]; }
                        rows(id1, x1);
                        tab(st + 2, id2);
#pragma unroll
                        for (int j = 0; j < HB; j++)
#pragma unroll
                            for (int c = 0; c < CT; c++) acc[h * HB + j][c] = mfma_step<DT>(wr[i][c], xc[j], acc[h * HB + j][c]);
                    }
                    load_w(k0 + k9 + i + WR, wr[i]);
                }
            };
            // a whole phase as straight-line code (the compiler then counts the weight loads in flight exactly);
            // offsets past the kernel's last find a table of empty slots
#pragma unroll
            for (int k9 = 0; k9 < kWinPhase; k9 += WR) round(k9);
        } else {
            // the rows lie too far apart: gathers from the feature array, one offset at a time
#pragma unroll
            for (int i = 0; i < kWinPhase; i++)
#pragma unroll
                for (int r = 0; r < RL; r++) s_tab32[i * RW + r * kWave + lane] = t[i][r];
            load_tab(ph + 1);
#pragma unroll 1
            for (int k9 = 0; k9 < nk; k9++) {
                int4v w[CT];
                load_w(k0 + k9, w);
#pragma unroll
                for (int h = 0; h < SPO; h++) {
                    int id[HB];
                    int4v x[HB];
#pragma unroll
                    for (int j = 0; j < HB; j++) {
                        id[j] = s_tab32[k9 * RW + (h * HB + j) * SPH_GROUP + (lane & 15)];
                        x[j] = *(const int4v *)(a.feat + (long)max(id[j], 0) * rb + choff);
                    }
#pragma unroll
                    for (int j = 0; j < HB; j++) {
                        bool live = id[j] >= 0;
                        if constexpr (MASKED) live = live && live_chunk;
                        const int4v y = live ? x[j] : int4v{0, 0, 0, 0};
#pragma unroll
                        for (int c = 0; c < CT; c++) acc[h * HB + j][c] = mfma_step<DT>(w[c], y, acc[h * HB + j][c]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int i = 0; i < WR; i++) load_w(k0 + kWinPhase + i, wr[i]);
        }
    }

    // epilogue: a lane holds four consecutive columns of one row per block and column tile
    const bool plain = DT != SPH_I8 && !a.scale && !a.shift && !a.relu;
    const bool relu = DT != SPH_I8 && a.relu;
    float sc[CT][4], sh[CT][4];
#pragma unroll
    for (int c = 0; c < CT; c++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int col = min(c * 16 + (lane >> 4) * 4 + j, a.ndim - 1);
            sc[c][j] = a.scale ? a.scale[col] : 1.f;
            sh[c][j] = (DT != SPH_I8 && a.shift) ? a.shift[col] : 0.f;
        }
    elem *out = (elem *)a.out + (long)r0 * a.ndim;
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int row = part * RW + b * SPH_GROUP + (lane & 15);
        if (row >= nrows) continue;
#pragma unroll
        for (int c = 0; c < CT; c++) {
            const int col = c * 16 + (lane >> 4) * 4;
            if (col >= a.ndim) continue;
            union { elem e[4]; uint32_t w[sizeof(elem)]; } u;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float v = DT == SPH_I8 ? (float)(int)acc[b][c][j] : (float)acc[b][c][j];
                if (!plain) {
                    v = v * sc[c][j] + sh[c][j];
                    if (relu) v = v > 0.f ? v : 0.f;
                }
                u.e[j] = to_elem<DT>(v);
            }
            uint32_t *dst = (uint32_t *)(out + (long)row * a.ndim + col);
#pragma unroll
            for (int q = 0; q < (int)sizeof(elem); q++) dst[q] = u.w[q];
        }
    }
}

inline int elem_size(sph_dtype dt) { return sph_elem_size(dt); }
inline int frag_elems(sph_dtype dt) { return sph_frag_elems(dt); }
inline int pad_waves(int ndim) { return sph_pad_waves(ndim); }
inline int num_steps(sph_dtype dt, int kdim) { return sph_num_steps(dt, kdim); }

template <sph_dtype DT, int NW, int NSTEP>
int launch_conv_ns(const ConvArgs &a, int ntiles, hipStream_t st)
{
    size_t lds = (size_t)R * (NW * 16 + 4) * sizeof(uint32_t);
    int rc = set_lds(conv_apply_kernel<DT, NW, NSTEP>, lds);
    if (rc) return rc;
    hipLaunchKernelGGL((conv_apply_kernel<DT, NW, NSTEP>), dim3(sph_xcd_grid(ntiles)), dim3(NW * kWave), lds, st, a);
    return sph_check_launch("sph_conv_apply");
}

template <sph_dtype DT, int NS, int CT, bool MASKED, int S>
int launch_conv_split(const ConvArgs &a, int nwtot, int ntiles, size_t lds, hipStream_t st)
{
    int rc = set_lds(conv_wave_split_kernel<DT, NS, CT, MASKED, S>, lds);
    if (rc) return rc;
    hipLaunchKernelGGL((conv_wave_split_kernel<DT, NS, CT, MASKED, S>), dim3(sph_xcd_grid(ntiles)), dim3(kWave * S), lds, st, a, nwtot);
    return sph_check_launch("sph_conv_apply");
}

// Only for books that are said to be thin.  The list costs a pair of tiles its two round trips whether it then pays or not, and a workgroup of two
// tiles is 5 % slower than two of one where it does not.  By pairs to a row, two tiles : one, 64 -> 64, 1100 to 4000 tiles: strided layers 1.0 to 1.25
// pairs 0.78 to 0.92 of the time, 1.45 0.87 to 0.97, 1.6 0.92 to 1.04, 2 and more 1.04 to 1.13.  Submanifold layers, whose middle offset is full,
// gain only from 1.35 to 2 pairs (0.86 to 0.98) and lose up to 0.3 below and 0.1 above; how many theirs are is not known before they are
// counted on the GPU (the share of the grid's cells that is taken says 1.1 for 1.1 pairs where voxels lie anywhere, and for 1.6 where they
// lie along surfaces).
// Not below 641 tiles, where conv_wave_split_kernel shares a tile's groups between waves or the chip is not filled (64 -> 64, two tiles : those,
// 304 tiles 31.2 : 30.2, 475 tiles 69 : 42; 606 tiles of stride 2x1x1 38.6 : 36.3, of stride 2x2x2 0.90), and not for smaller kernels, whose
// offsets have more pairs each (18 offsets 1.03 to 1.10).
inline bool pair_ok(const ConvArgs &a, int nwtot, int ntiles)
{
    return nwtot == 4 && book_says(&a.book) == SPH_THIN && a.book.KV >= 27 && a.book.KV <= kWave && a.book.tile_koff &&
           (uintptr_t)a.book.grp_gather % 16 == 0 && ntiles > 640;
}

template <sph_dtype DT, int NS, int CT, bool MASKED>
int launch_conv_wave(const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
    size_t lds = (size_t)(R + 1) * (nwtot * 16 + 4) * sizeof(uint32_t); // + scratch row
    const int waves = (nwtot + CT - 1) / CT;
    // one wave's worth of columns, rows of up to 128 bytes: helper waves for the middle offset's run (fp32 rows
    // of 128 bytes into 64 columns do not fit the registers three waves per SIMD leave)
    // (narrow layers on large grids keep the one-wave kernel: a group is one fragment load and one MFMA there,
    // and the helper waves' barriers cost a full chip more than the run saves: 16 -> 16 on 4912 tiles 22.6 / 25.8 us)
    constexpr bool kRunKernel = NS <= 2 && !(DT == SPH_F32 && NS == 2 && CT == 4);
    const bool helpers = kRunKernel && waves == 1 && a.book.tile_koff && book_has_run(&a.book) && (NS * CT >= 4 || ntiles <= 1024);
    if constexpr (DT == SPH_F32 && NS == 4 && CT == 4) {
        if (pair_ok(a, nwtot, ntiles)) {
            const size_t lds2 = pair_lds(nwtot);
            int rc = set_lds(conv_wave_pair_kernel<NS, MASKED>, lds2);
            if (rc) return rc;
            hipLaunchKernelGGL((conv_wave_pair_kernel<NS, MASKED>), dim3(sph_xcd_grid((ntiles + 1) / 2)), dim3(2 * kWave), lds2, st, a, nwtot);
            return sph_check_launch("sph_conv_apply");
        }
    }
    if (waves == 1) {
        const int s = split_waves(DT, a.row_bytes, nwtot, helpers, ntiles, lds, 0);
        if (s == 4) return launch_conv_split<DT, NS, CT, MASKED, 4>(a, nwtot, ntiles, 4 * lds, st);
        if (s == 2) return launch_conv_split<DT, NS, CT, MASKED, 2>(a, nwtot, ntiles, 2 * lds, st);
    }
    if constexpr (kRunKernel) {
        if (helpers) {
            int rc = set_lds(conv_wave_run_kernel<DT, NS, CT, MASKED>, lds);
            if (rc) return rc;
            hipLaunchKernelGGL((conv_wave_run_kernel<DT, NS, CT, MASKED>), dim3(sph_xcd_grid(ntiles)), dim3(kWave * (1 + kRunHelpers)),
                               lds, st, a, nwtot);
            return sph_check_launch("sph_conv_apply");
        }
    }
    int rc = set_lds(conv_wave_kernel<DT, NS, CT, MASKED>, lds);
    if (rc) return rc;
    hipLaunchKernelGGL((conv_wave_kernel<DT, NS, CT, MASKED>), dim3(sph_xcd_grid(ntiles)), dim3(waves * kWave), lds, st, a, nwtot);
    return sph_check_launch("sph_conv_apply");
}

template <sph_dtype DT, int NS, int CT>
int launch_conv_wave_m(const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
    // rows that end inside the last 64-byte step need its tail masked
    if (a.row_bytes < NS * 64) return launch_conv_wave<DT, NS, CT, true>(a, nwtot, ntiles, st);
    return launch_conv_wave<DT, NS, CT, false>(a, nwtot, ntiles, st);
}

template <sph_dtype DT, int NS>
int launch_conv_wave_ct(const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
    switch (nwtot) { // at most two waves per workgroup (launch bound of the kernel)
    case 1: return launch_conv_wave_m<DT, NS, 1>(a, nwtot, ntiles, st);
    case 2: return launch_conv_wave_m<DT, NS, 2>(a, nwtot, ntiles, st);
    default:
        // int8 rows are 64 bytes: on a full chip two waves per tile (32 columns each, the rows gathered twice)
        // are faster than one (2464 tiles, 27 offsets: 50.5 -> 45.5 us; what relay.hip does not take comes here: up to 9
        // offsets, unaligned output); with 128-byte fp16 rows they are slower (123 -> 151 us)
        // (up to 64 output columns only: more would be four waves, beyond the kernel's launch bound).  A book with a
        // run at its middle offset takes one wave of 64 columns and two helper waves instead (36.7 -> 35.1 us).
        if constexpr (DT == SPH_I8)
            if (ntiles > 1024 && nwtot <= 4 && !book_has_run(&a.book)) return launch_conv_wave_m<DT, NS, 2>(a, nwtot, ntiles, st);
        return launch_conv_wave_m<DT, NS, 4>(a, nwtot, ntiles, st);
    }
}

// Whether a layer of one K step that rows_hold.hip and rows_split.hip leave goes through the window.  With up to 32 columns on grids of
// more than 1024 tiles; into 64 columns what arrives is 27 offsets in 16 bits and int8 on 961 to 1024 tiles and beyond 1900, and other kernels from 641
// or 769 tiles on (win_first).  Two waves of a tile have only two waves of a SIMD beside them then, and it depends.  Times with the
// window over times without, 3x3x3 but where said, 0.4 of the bins:
//   tiles             800  1000  1100  1250  1500  1800  2000  3000  4000
//   fp16 32 -> 64                                              0.80  0.84
//   int8 64 -> 64                                              0.72  0.82
//   fp32, 5x3x3                        0.90  0.93                    0.88
//   fp16, 3x3x1      0.78  0.81  1.43  1.43  1.42  1.24  1.35  1.26  1.35   (one phase: nothing overlaps its window)
//   fp16, 2x2x2      0.92  0.93  1.49  1.52  1.56  1.40  1.43  1.37  1.54   (a phase costs nine offsets; 3x2x2 alike)
//   fp16, stride 2         0.95        1.33        1.11  1.22  0.99  1.02   (3.2 gathered rows to a row: windows too small)
template <sph_dtype DT, int CT>
bool win_ok(const ConvArgs &a, int ntiles)
{
    if (CT < 4) return ntiles > 1024;
    if (a.book.KV % kWinPhase != 0 || a.feat_rows > 2.0 * a.book.rows) return false;
    if (a.book.KV == kWinPhase) return ntiles > 768 && ntiles <= 1024;
    if (DT == SPH_F32) return ntiles > 768 && (ntiles <= 1280 || a.book.KV > 4 * kWinPhase);
    // (without it 2048 tiles are on the chip at once: 2037 tiles, 6.9 pairs a row, fp16 32 -> 64 1.09, 16 -> 64 1.16; int8 1.04)
    if (DT != SPH_I8 && ntiles > 1920 && ntiles <= 2048) return false;
    return true;
}

// One wave per tile instead of two (32 columns): with two 1536 tiles are on the chip at once, with one 2048.  us, one : two:
// fp16 32 -> 32 1500 tiles 23.9 : 19.7, 1800 tiles 24.9 : 27.7, 2300 tiles 39.5 : 31.3, 4000 tiles 52.0 : 51.1; fp32 16 -> 32 1250
// tiles 66.2 : 52.6, 2000 tiles 71.4 : 86.5, 3300 tiles 135.2 : 130.5, 4000 tiles 138.8 : 146.0 (its matrix cores leave fewer waits to fill).
template <sph_dtype DT>
bool win_one_wave(int ntiles) { return (ntiles > 1536 && ntiles <= 2048) || (DT == SPH_F32 && ntiles > 3584); }

// Before the kernels of rows_split.hip: kernels of other than 27 offsets into 64 columns, from 769 tiles on (45 offsets 32 -> 64 1001 tiles 33 : 42
// us, 512 tiles 27 : 22.5; 1x3x3 1001 tiles 14 : 19).
template <sph_dtype DT>
bool win_first(const ConvArgs &a, int nwtot, int ntiles)
{
    return a.nsteps == 1 && nwtot == 4 && a.book.KV != 27 && ntiles > 768 && win_ok<DT, 4>(a, ntiles);
}

template <sph_dtype DT, int NS, int CT, bool MASKED>
int launch_conv_rows_m(const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
    const int waves = (nwtot + CT - 1) / CT;
    // the table, and for 128-byte rows a wave's exchange buffer (up to 4 chunk sets of 16 rows x 80 bytes)
    const size_t lds = (size_t)a.book.KV * R * sizeof(int32_t) + (NS >= 2 ? (size_t)waves * 4 * SPH_GROUP * 80 : 0);
    const dim3 grid(sph_xcd_grid(ntiles)), block(waves * kWave);
    if constexpr (NS == 1) {
        // one K step, up to 64 columns: the gathered rows go through an LDS window
        if (waves == 1 && win_ok<DT, CT>(a, ntiles)) {
            const size_t lds_win = kWinTab + kWinBytes + 64;
            if constexpr (CT == 2) {
                if (win_one_wave<DT>(ntiles)) {
                    hipLaunchKernelGGL((conv_rows_win_kernel<DT, CT, MASKED, 1>), grid, dim3(kWave), lds_win, st, a, nwtot);
                    return sph_check_launch("sph_conv_apply");
                }
            }
            hipLaunchKernelGGL((conv_rows_win_kernel<DT, CT, MASKED, 2>), grid, dim3(2 * kWave), lds_win, st, a, nwtot);
            return sph_check_launch("sph_conv_apply");
        }
    }
    if constexpr (CT >= 4) hipLaunchKernelGGL((conv_rows_kernel_w2<DT, NS, CT, MASKED>), grid, block, lds, st, a, nwtot);
    else if constexpr (CT == 2) hipLaunchKernelGGL((conv_rows_kernel_w3<DT, NS, CT, MASKED>), grid, block, lds, st, a, nwtot);
    else hipLaunchKernelGGL((conv_rows_kernel_w4<DT, NS, CT, MASKED>), grid, block, lds, st, a, nwtot);
    return sph_check_launch("sph_conv_apply");
}

template <sph_dtype DT, int NS, int CT>
int launch_conv_rows(const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
    if (a.row_bytes < NS * 64) return launch_conv_rows_m<DT, NS, CT, true>(a, nwtot, ntiles, st);
    return launch_conv_rows_m<DT, NS, CT, false>(a, nwtot, ntiles, st);
}

template <sph_dtype DT, int NS>
int launch_conv_rows_ct(const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
    switch (nwtot) {
    case 1: return launch_conv_rows<DT, NS, 1>(a, nwtot, ntiles, st);
    case 2: return launch_conv_rows<DT, NS, 2>(a, nwtot, ntiles, st);
    default: return launch_conv_rows<DT, NS, 4>(a, nwtot, ntiles, st);
    }
}

template <sph_dtype DT, int NW>
int launch_conv(const ConvArgs &a, int ntiles, hipStream_t st)
{
    // by stationary row, when the book keeps that form (rows of up to 128 bytes; its table must fit LDS)
    if (rows_path_ok(a)) {
        if (sph_rows_hold_ok(DT, a, NW, ntiles)) return sph_rows_hold_launch(DT, a, st);
        if (!win_first<DT>(a, NW, ntiles) && sph_rows_split_ok(DT, a, NW, ntiles)) return sph_rows_split_launch(DT, a, NW, ntiles, st);
        if (a.nsteps == 1) return launch_conv_rows_ct<DT, 1>(a, NW, ntiles, st);
        return launch_conv_rows_ct<DT, 2>(a, NW, ntiles, st);
    }
    // the one-wave-per-tile kernel addresses the feature array through a buffer descriptor with 31-bit offsets
    // made by a 24-bit multiply
    const bool small = (double)a.feat_rows * a.row_bytes < 2147483648.0 && a.feat_rows < (1 << 24);
    if (a.aligned_in && a.feat_rows > 0 && small) {
        if (sph_relay_ok(DT, a, NW, ntiles)) return sph_relay_launch(DT, a, NW, ntiles, st);
        switch (a.nsteps) {
        case 1: return launch_conv_wave_ct<DT, 1>(a, NW, ntiles, st);
        case 2: return launch_conv_wave_ct<DT, 2>(a, NW, ntiles, st);
        case 4: return launch_conv_wave_ct<DT, 4>(a, NW, ntiles, st);
        default: break;
        }
    }
    return launch_conv_ns<DT, NW, 0>(a, ntiles, st); // rows not a multiple of 16 bytes, or more than 256 bytes, or 2 GiB of them
}

template <sph_dtype DT>
int launch_conv_nw(const ConvArgs &a, int nw, int ntiles, hipStream_t st)
{
    switch (nw) {
    case 1: return launch_conv<DT, 1>(a, ntiles, st);
    case 2: return launch_conv<DT, 2>(a, ntiles, st);
    case 4: return launch_conv<DT, 4>(a, ntiles, st);
    default: return launch_conv<DT, 8>(a, ntiles, st);
    }
}

} // namespace

SPH_EXPORT size_t sph_weight_packed_bytes(sph_dtype dt, int KV, int kdim, int ndim)
{
    if (KV <= 0 || kdim <= 0 || ndim <= 0 || (int)dt < 0 || (int)dt > 3) return 0;
    return (size_t)KV * num_steps(dt, kdim) * pad_waves(ndim) * kWave * 16;
}

SPH_EXPORT int sph_weight_pack(sph_dtype dt, const void *w, int KV, int kdim, int ndim, long stride_k,
                               long stride_kk, long stride_n, void *packed, void *stream)
{
    int rc = sph_pack_args_ok("sph_weight_pack", dt, w, packed, KV, kdim, ndim);
    if (rc) return rc;
    SPH_REQUIRE((uintptr_t)packed % 16 == 0, SPH_ERR_ARG, "sph_weight_pack: packed weight must be 16-byte aligned");
    SphPackJobs p;
    p.job[0] = sph_pack_job(dt, w, KV, kdim, ndim, stride_k, stride_kk, stride_n, packed);
    p.job[1].total = 0;
    hipLaunchKernelGGL(pack_weight_kernel, dim3(sph_div_up(p.job[0].total, 64)), dim3(64), 0, (hipStream_t)stream, p);
    return sph_check_launch("sph_weight_pack");
}

SPH_EXPORT int sph_weight_packs(const sph_pack_desc *packs, int npacks, void *stream)
{
    SphPackJobs p;
    int rc = sph_pack_jobs("sph_weight_packs", packs, npacks, &p);
    if (rc) return rc;
    const int total = sph_pack_total(p.job);
    if (total == 0) return SPH_OK;
    hipLaunchKernelGGL(pack_weight_kernel, dim3(sph_div_up(total, 64)), dim3(64), 0, (hipStream_t)stream, p);
    return sph_check_launch("sph_weight_packs");
}

SPH_EXPORT int sph_conv_apply(sph_dtype dt, const void *feature, int feature_rows, int kdim,
                              const void *packed_w, int ndim, const sph_book *book,
                              const sph_epilogue *epi, void *out, void *stream)
{
    SPH_REQUIRE(book_ok(book), SPH_ERR_ARG, "sph_conv_apply: bad book");
    SPH_REQUIRE(packed_w && feature_rows >= 0 && (feature_rows == 0 || feature), SPH_ERR_ARG, "sph_conv_apply: null pointer");
    SPH_REQUIRE((int)dt >= 0 && (int)dt <= 3, SPH_ERR_ARG, "sph_conv_apply: unknown dtype %d", (int)dt);
    SPH_REQUIRE(kdim > 0 && kdim <= SPH_MAX_CHANNELS, SPH_ERR_UNSUPPORTED,
                "sph_conv_apply: %d input channels not in 1..%d", kdim, SPH_MAX_CHANNELS);
    SPH_REQUIRE(ndim > 0 && ndim <= 128, SPH_ERR_UNSUPPORTED, "sph_conv_apply: %d output channels not in 1..128", ndim);
    SPH_REQUIRE(dt != SPH_I8 || (epi && epi->scale), SPH_ERR_ARG, "sph_conv_apply: int8 needs per-channel scales");
    if (book->rows == 0) return SPH_OK;
    SPH_REQUIRE(out, SPH_ERR_ARG, "sph_conv_apply: null output");
    const int es = elem_size(dt);
    ConvArgs a;
    a.feat = (const char *)feature;
    a.feat_rows = feature_rows;
    a.kdim = kdim;
    a.row_bytes = kdim * es;
    a.wp = (const char *)packed_w;
    a.nsteps = num_steps(dt, kdim);
    a.ndim = ndim;
    a.book = *book;
    a.cap = sph_book_cap(book->KV);
    a.scale = epi ? epi->scale : nullptr;
    a.shift = epi ? epi->shift : nullptr;
    a.relu = epi ? epi->relu : 0;
    a.out = (char *)out;
    a.aligned_in = (a.row_bytes % 16 == 0) && ((uintptr_t)feature % 16 == 0);
    a.aligned_out = ((ndim * es) % 16 == 0) && ((uintptr_t)out % 16 == 0);
    SPH_REQUIRE((uintptr_t)packed_w % 16 == 0, SPH_ERR_ARG, "sph_conv_apply: packed weight must be 16-byte aligned");
    SPH_REQUIRE(book_has_groups(book) || rows_path_ok(a), SPH_ERR_ARG,
                "sph_conv_apply: the book holds no groups and this call cannot go by rows (rows of 16-byte multiples up to "
                "128 bytes, 16-byte aligned arrays)");
    const int nw = pad_waves(ndim), nt = sph_book_tiles(book->rows);
    hipStream_t st = (hipStream_t)stream;
    switch (dt) {
    case SPH_F32: return launch_conv_nw<SPH_F32>(a, nw, nt, st);
    case SPH_F16: return launch_conv_nw<SPH_F16>(a, nw, nt, st);
    case SPH_BF16: return launch_conv_nw<SPH_BF16>(a, nw, nt, st);
    default: return launch_conv_nw<SPH_I8>(a, nw, nt, st);
    }
}
