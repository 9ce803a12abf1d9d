// By-row convolution (gfx950) with a row's offsets shared by the waves of a workgroup: short grids, where one wave's walk over
// all offsets is what the kernel lasts, and longer ones of 128-byte rows, whose gathers are the bound of the kernels of conv.hip.
// A row's sum is four or eight waves' sums (offsets w, w + 4, ... or w + 8, ...), added in a fixed order.
#include "rows_split.h"
#include <type_traits>

namespace {

constexpr unsigned kNoRow = 0x80000000u; // a byte offset beyond every feature array (below 2 GiB): such a load returns zeros
constexpr int kPhase = 9, kPhases = 3;   // offsets that share a window, windows of a tile
constexpr int kSplitKV = kPhase * kPhases;

template <typename T> __device__ __forceinline__ T pick_of(bool second, T x, T y) { return second ? y : x; }

// four columns of a row
template <sph_dtype DT, typename F>
__device__ __forceinline__ void store_four(const ConvArgs &a, typename Traits<DT>::elem *out, typename Traits<DT>::acc4 v, const F &sc, const F &sh)
{
    typedef typename Traits<DT>::elem elem;
    const bool relu = DT != SPH_I8 && a.relu;
    union { elem e[4]; uint32_t w[sizeof(elem)]; } u;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float x = DT == SPH_I8 ? (float)(int)v[j] : (float)v[j];
        x = x * sc[j] + sh[j]; // (1 and 0 where the call has none: the sum itself)
        if (relu) x = x > 0.f ? x : 0.f;
        u.e[j] = to_elem<DT>(x);
    }
#pragma unroll
    for (int q = 0; q < (int)sizeof(elem); q++) ((uint32_t *)out)[q] = u.w[q];
}

// A workgroup takes NB blocks of 16 rows and up to 64 columns; wave w takes offsets w, w + W, ..., KC of them in flight: the
// table's entries, then the gathered rows and the weight fragments, all requested at once and counted exactly.  Slots
// without a pair read zeros from out of the array's range.  The waves' sums meet in LDS.
// What bounds it: three memory round trips and the sums' exchange (64 tiles, 64 -> 64: 6.8 us, 2.3 of them a launch that
// does nothing), where a wave that walked all 27 offsets for two blocks lasted 16.7 on a quarter of the compute units; on
// grids that fill the chip the gathers, 27 rows for every row.
template <sph_dtype DT, int NS, int CT, bool MASKED, int NB, int W, int KC>
__global__ __launch_bounds__(W * kWave) __attribute__((amdgpu_waves_per_eu(W / 4)))
void conv_rows_short_kernel(ConvArgs a, int nwtot)
{
    typedef typename Traits<DT>::elem elem;
    typedef typename Traits<DT>::acc4 acc4;
    constexpr int RB = NB * SPH_GROUP; // rows of a workgroup
    constexpr int NF = NB * CT;        // accumulators of a wave
    static_assert(W % CT == 0, "the fragments a wave writes lie in one column tile");
    // Rows of 128 bytes are asked for with the four lanes of a quad on a row's 64 bytes (one look-up in the nearest cache for
    // four) and brought to the operands' order, lane = row + 16 * chunk, through a wave's own part of LDS.
    constexpr bool QUAD = NS == 2;
    constexpr int kTrRow = 80, kTrSet = SPH_GROUP * kTrRow; // (padded rows: writes and reads without conflicts)
    constexpr int kWaveLds = NF * kWave * 16 > (QUAD ? NB * NS * kTrSet : 0) ? NF * kWave * 16 : NB * NS * kTrSet;
    __shared__ __attribute__((aligned(16))) char s_mem[W * kWaveLds];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int unit = sph_xcd_tile(blockIdx.x, (a.book.rows + RB - 1) / RB);
    const int r0 = unit * RB;
    if (r0 >= a.book.rows) return;
    const int KV = a.book.KV;
    const int col0 = blockIdx.y * (CT * 16);
    const int tile = r0 / R;
    const int32_t *tab = a.book.tile_nbr + (long)tile * KV * R + (r0 - tile * R) + (QUAD ? lane >> 2 : lane & 15);
    char *tr = s_mem + wave * kWaveLds;
    const int wstep = nwtot * (kWave * 16);
    const __amdgpu_buffer_rsrc_t r_feat = __builtin_amdgcn_make_buffer_rsrc((void *)a.feat, 0, a.feat_rows * a.row_bytes, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_w = __builtin_amdgcn_make_buffer_rsrc((void *)a.wp, 0, KV * NS * wstep, kRsrcFlags);
    const int wlane = (col0 / 16) * (kWave * 16) + lane * 16;
    const int chunk = (QUAD ? lane & 3 : lane >> 4) * 16;

    acc4 acc[NB][CT];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int c = 0; c < CT; c++) acc[j][c] = acc4{0, 0, 0, 0};

    int id[KC][NB];
    auto load_tab = [&](int k0) {
#pragma unroll
        for (int i = 0; i < KC; i++)
#pragma unroll
            for (int j = 0; j < NB; j++) id[i][j] = tab[min(k0 + i * W, KV - 1) * R + j * SPH_GROUP];
    };
    load_tab(wave);
    for (int k0 = wave; k0 < KV; k0 += KC * W) {
        int4v fw[KC][NS][CT], fa[KC][NB][NS];
#pragma unroll
        for (int i = 0; i < KC; i++) {
            const int wk = min(k0 + i * W, KV - 1) * (NS * wstep);
#pragma unroll
            for (int st = 0; st < NS; st++)
#pragma unroll
                for (int c = 0; c < CT; c++)
                    fw[i][st][c] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(r_w, wlane + st * wstep + c * (kWave * 16), wk, 0));
        }
#pragma unroll
        for (int i = 0; i < KC; i++) {
            const unsigned lim = k0 + i * W < KV ? a.feat_rows : 0; // an offset behind the last has no pairs
#pragma unroll
            for (int j = 0; j < NB; j++) {
                const unsigned off = (unsigned)id[i][j] < lim ? (unsigned)(id[i][j] * a.row_bytes + chunk) : kNoRow;
#pragma unroll
                for (int st = 0; st < NS; st++) {
                    const unsigned o = MASKED && st * 64 + chunk >= a.row_bytes ? kNoRow : off + st * 64;
                    fa[i][j][st] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(r_feat, o, 0, 0));
                }
            }
        }
        if (k0 + KC * W < KV) load_tab(k0 + KC * W);
#pragma unroll
        for (int i = 0; i < KC; i++) {
            if constexpr (QUAD) { // (a wave's accesses of LDS keep their order)
#pragma unroll
                for (int j = 0; j < NB; j++)
#pragma unroll
                    for (int st = 0; st < NS; st++) *(int4v *)(tr + (j * NS + st) * kTrSet + (lane >> 2) * kTrRow + (lane & 3) * 16) = fa[i][j][st];
                asm volatile("" ::: "memory");
#pragma unroll
                for (int j = 0; j < NB; j++)
#pragma unroll
                    for (int st = 0; st < NS; st++) fa[i][j][st] = *(const int4v *)(tr + (j * NS + st) * kTrSet + (lane & 15) * kTrRow + (lane >> 4) * 16);
                asm volatile("" ::: "memory");
            }
#pragma unroll
            for (int st = 0; st < NS; st++)
#pragma unroll
                for (int j = 0; j < NB; j++)
#pragma unroll
                    for (int c = 0; c < CT; c++) acc[j][c] = mfma_step<DT>(fw[i][st][c], fa[i][j][st], acc[j][c]);
        }
    }

    // the waves' sums meet in LDS (the exchange above is over: a wave's part of both is its own), wave by wave; a wave writes fragments wave, wave + W, ...
    const int col = col0 + (wave % CT) * 16 + (lane >> 4) * 4;
    float sc[4], sh[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int cj = min(col + j, a.ndim - 1);
        sc[j] = a.scale ? a.scale[cj] : 1.f;
        sh[j] = (DT != SPH_I8 && a.shift) ? a.shift[cj] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int c = 0; c < CT; c++) *(acc4 *)(tr + ((j * CT + c) * kWave + lane) * 16) = acc[j][c];
    lds_barrier();
#pragma unroll
    for (int f0 = 0; f0 < NF; f0 += W) {
        const int f = f0 + wave;
        if (f >= NF) break;
        acc4 v = *(const acc4 *)(s_mem + (f * kWave + lane) * 16);
#pragma unroll
        for (int w = 1; w < W; w++) v += *(const acc4 *)(s_mem + w * kWaveLds + (f * kWave + lane) * 16);
        const int row = r0 + (f / CT) * SPH_GROUP + (lane & 15);
        if (row < a.book.rows && col < a.ndim) store_four<DT>(a, (elem *)a.out + (long)row * a.ndim + col, v, sc, sh);
    }
}

// 27 offsets, the rows that a workgroup gathers in LDS: a workgroup takes NB blocks of 16 rows and up to 64 columns, its four
// waves every fourth offset of all rows.  The rows that nine consecutive offsets gather (one k0 of a 3x3x3 kernel) are one
// stretch of the feature array (two where the rows straddle lines of the grid): three windows, brought by direct loads that are
// all in flight at once, at multiples of a load's rows; the table is rewritten to places in LDS.  A row's 16-byte chunks lie
// exchanged by its place (chunk ^ place), so that 16 rows' chunks, which the operands take together, lie in different banks; the
// table holds places with that folded in, and an address is an exclusive or.  Empty slots point at a row of zeros.  The offsets of a window
// that finds no room are left out, and follow from the feature array.  The waves' sums meet in LDS, halves of the blocks
// first, then quarters.
// Every offset's weight passes the compute unit's vector memory path once for NB * 16 rows (216 KiB at 64 -> 64), the rows
// three times at most, where gathers bring each row 27 times: 290 KiB for 128 rows against 660.
// What bounds it, 64 -> 64 fp16 on 3996 tiles (129 us, plain kernel 167; the matrix cores need 55 at the 2.0 GHz it runs at): two workgroups
// are on a compute unit (LDS 79 KiB, 242 registers), each 28 k cycles: table 4.7 k, windows 2.5 k, places 1.9 k, products 11.8 k (7.2 k alone
// on its SIMD), exchange 3.9 k, store 2.4 k; the one's products run beside the other's rest.  Blocks of 64 rows take the
// weights twice: 165.
template <sph_dtype DT, int NS, int CT, bool MASKED, int NB>
__global__ __launch_bounds__(4 * kWave) __attribute__((amdgpu_waves_per_eu(2)))
void conv_rows_split_kernel(ConvArgs a, int nwtot, int cap_rows)
{
    typedef typename Traits<DT>::elem elem;
    typedef typename Traits<DT>::acc4 acc4;
    constexpr int W = 4;
    constexpr int DX = NB >= 8 ? 2 : 1; // blocks that rows are read ahead of their products
    constexpr int RB = NB * SPH_GROUP; // rows of a workgroup
    constexpr int CH = NS * 4;         // 16-byte chunks of a row in LDS
    constexpr int RPL = kWave / CH;    // rows one wave-wide load brings
    constexpr int TPR = 4 * kWave / RB;     // waves that share a row's entries while the table is read
    constexpr int TE = (kPhase + TPR - 1) / TPR; // entries of a thread and phase
    static_assert(RB >= kWave, "a wave reads whole offsets");
    static_assert(W == 4 && kSplitKV <= 32, "every fourth bit of a word");
    extern __shared__ __attribute__((aligned(16))) char s_mem[];
    uint16_t *s_tab = (uint16_t *)s_mem;                       // [kSplitKV][16 rows][NB]
    char *s_win = s_mem + kSplitKV * RB * 2;                         // rows, chunks swizzled
    __shared__ int2 s_range[kPhases][W];
    __shared__ int2 s_range2[kPhases][W];
    __shared__ __attribute__((aligned(16))) float s_sc[2][CT * 16]; // the columns' scale and shift
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int unit = sph_xcd_tile(blockIdx.x, (a.book.rows + RB - 1) / RB);
    const int r0 = unit * RB;
    if (r0 >= a.book.rows) return;
    const int col0 = blockIdx.y * (CT * 16);
    const int tile = r0 / R;
    const int32_t *tab = a.book.tile_nbr + (long)tile * kSplitKV * R + (r0 - tile * R);
    const int wstep = nwtot * (kWave * 16);
    const int rb = a.row_bytes;
    const __amdgpu_buffer_rsrc_t r_feat = __builtin_amdgcn_make_buffer_rsrc((void *)a.feat, 0, a.feat_rows * rb, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_w = __builtin_amdgcn_make_buffer_rsrc((void *)a.wp, 0, kSplitKV * NS * wstep, kRsrcFlags);
    const int wlane = (col0 / 16) * (kWave * 16) + lane * 16;

    // the thread's part of the table: row trow, offsets tpart, tpart + TPR, ... of every phase
    int t[kPhases][TE];
    const int trow = lane + wave % (RB / kWave) * kWave, tpart = wave / (RB / kWave);
#pragma unroll
    for (int p = 0; p < kPhases; p++)
#pragma unroll
        for (int i = 0; i < TE; i++) t[p][i] = tab[(p * kPhase + min(tpart + i * TPR, kPhase - 1)) * R + trow];
    auto load_w = [&](int k, int4v (&w)[NS][CT]) {
        const int wk = min(k, kSplitKV - 1) * (NS * wstep);
#pragma unroll
        for (int st = 0; st < NS; st++)
#pragma unroll
            for (int c = 0; c < CT; c++)
                w[st][c] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(r_w, wlane + st * wstep + c * (kWave * 16), wk, 0));
    };
    int4v fw[2][NS][CT];
    load_w(wave, fw[0]);
    load_w(wave + W, fw[1]);

    if (tid < CT * 16) {
        const int c = min(col0 + tid, a.ndim - 1);
        s_sc[0][tid] = a.scale ? a.scale[c] : 1.f;
        s_sc[1][tid] = DT != SPH_I8 && a.shift ? a.shift[c] : 0.f;
    }
    int lo[kPhases], hi[kPhases];
#pragma unroll
    for (int p = 0; p < kPhases; p++) {
        lo[p] = 0x7fffffff;
        hi[p] = -1;
#pragma unroll
        for (int i = 0; i < TE; i++) {
            t[p][i] = (unsigned)t[p][i] < (unsigned)a.feat_rows ? t[p][i] : -1; // (a wave's last offset may be there twice)
            lo[p] = (int)min((unsigned)lo[p], (unsigned)t[p][i]);
            hi[p] = max(hi[p], t[p][i]);
        }
    }
#pragma unroll
    for (int p = 0; p < kPhases; p++) {
        lo[p] = ~wave_max_last(~lo[p]);
        hi[p] = wave_max_last(hi[p]);
        if (lane == kWave - 1) s_range[p][wave] = make_int2(lo[p], hi[p]);
    }
    if (tid < CH) *(int4v *)(s_win + tid * 16) = int4v{0, 0, 0, 0}; // row 0
    lds_barrier();
    int n1[kPhases], lo2[kPhases], n2[kPhases], base[kPhases], base2[kPhases], need = 0;
#pragma unroll
    for (int p = 0; p < kPhases; p++) {
        int l = 0x7fffffff, h = -1;
#pragma unroll
        for (int w = 0; w < W; w++) { const int2 v = s_range[p][w]; l = min(l, v.x); h = max(h, v.y); }
        lo[p] = __builtin_amdgcn_readfirstlane(l);
        hi[p] = __builtin_amdgcn_readfirstlane(h);
        n1[p] = hi[p] < 0 ? 0 : hi[p] - lo[p] + 1;
        lo2[p] = 0x7fffffff; n2[p] = 0; base2[p] = 0;
        need += min(n1[p], 1 << 24);
    }
    if (need > cap_rows - RPL * (kPhases + 1)) {
        // the rows of a tile that straddles two lines of the grid lie in two places
        const int seg = cap_rows / (2 * kPhases);
#pragma unroll
        for (int p = 0; p < kPhases; p++) {
            int h1 = -1, l2 = 0x7fffffff;
            const int cut = lo[p] + seg;
#pragma unroll
            for (int i = 0; i < TE; i++) {
                h1 = max(h1, t[p][i] < cut ? t[p][i] : -1);
                l2 = (int)min((unsigned)l2, (unsigned)(t[p][i] < cut ? -1 : t[p][i]));
            }
            h1 = wave_max_last(h1);
            l2 = ~wave_max_last(~l2);
            if (lane == kWave - 1) s_range2[p][wave] = make_int2(l2, h1);
        }
        lds_barrier();
#pragma unroll
        for (int p = 0; p < kPhases; p++) {
            int l2 = 0x7fffffff, h1 = -1;
#pragma unroll
            for (int w = 0; w < W; w++) { const int2 v = s_range2[p][w]; l2 = min(l2, v.x); h1 = max(h1, v.y); }
            l2 = __builtin_amdgcn_readfirstlane(l2);
            h1 = __builtin_amdgcn_readfirstlane(h1);
            if (n1[p] > seg && l2 != 0x7fffffff && l2 > h1 + 1) { n1[p] = h1 - lo[p] + 1; lo2[p] = l2; n2[p] = hi[p] - l2 + 1; }
        }
    }
    // Windows begin at multiples of a load's rows (row 0 holds zeros), so that a lane's place in the swizzle does not depend on
    // the load: a load of RPL rows is a scalar step on from the last.  Rows behind a window's last are the array's next rows
    // (or its last row again) in places nothing points to.
    int used = RPL;
    bool fits[kPhases];
    const int lrow = lane / CH, f_lane = NS == 2 ? (lrow & 7) : ((lrow >> 1) & 3);
    const int c_lane = ((lane & (CH - 1)) ^ f_lane) * 16;
    const int src_lane = lrow * rb + ((!MASKED || c_lane < rb) ? c_lane : 0);
    const int last = (a.feat_rows - 1) * rb + rb - 16;
#pragma unroll
    for (int p = 0; p < kPhases; p++) {
        base[p] = used;
        const int r1 = (n1[p] + RPL - 1) & -RPL, r2 = (n2[p] + RPL - 1) & -RPL;
        fits[p] = n1[p] <= cap_rows && n2[p] <= cap_rows && used + r1 + r2 <= cap_rows;
        if (!fits[p]) continue;
        base2[p] = used + r1;
        used += r1 + r2;
        const int first = src_lane + (int)((unsigned)lo[p] * rb), first2 = src_lane + (int)((unsigned)lo2[p] * rb);
        for (int i = wave * RPL; i < n1[p]; i += W * RPL)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r_feat, (__attribute__((address_space(3))) void *)(s_win + (base[p] + i) * (CH * 16)), 16,
                                                     min(first + i * rb, last), 0, 0, 0);
        for (int i = wave * RPL; i < n2[p]; i += W * RPL)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r_feat, (__attribute__((address_space(3))) void *)(s_win + (base2[p] + i) * (CH * 16)), 16,
                                                     min(first2 + i * rb, last), 0, 0, 0);
    }
    // the table: place of the row in LDS, its swizzle folded in
#pragma unroll
    for (int p = 0; p < kPhases; p++) {
        if (!fits[p])
#pragma unroll
            for (int i = 0; i < TE; i++) t[p][i] = -1;
        const int d1 = base[p] - lo[p], d2 = base2[p] - lo2[p];
#pragma unroll
        for (int i = 0; i < TE; i++) {
            const int k9 = min(tpart + i * TPR, kPhase - 1);
            int at = t[p][i] + (n2[p] > 0 && t[p][i] >= lo2[p] ? d2 : d1);
            at = t[p][i] >= 0 ? at : 0;
            const int f = NS == 2 ? (at & 7) : ((at >> 1) & 3);
            s_tab[((p * kPhase + k9) * SPH_GROUP + (trow & 15)) * NB + trow / SPH_GROUP] = (uint16_t)(at * CH | f);
        }
    }
    acc4 acc[NB][CT];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int c = 0; c < CT; c++) acc[j][c] = acc4{0, 0, 0, 0};
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();

    const int chunk = lane >> 4;
    const bool live0 = !MASKED || chunk * 16 < rb, live1 = !MASKED || NS == 1 || 64 + chunk * 16 < rb;
    const int ok_mask = (fits[0] ? 1 : 0) | (fits[1] ? 2 : 0) | (fits[2] ? 4 : 0);
    // rows one block ahead of their products, the table one offset ahead
    auto load_ix = [&](int k, uint32_t (&ix)[NB / 2]) {
        const uint32_t *p = (const uint32_t *)(s_tab + (min(k, kSplitKV - 1) * SPH_GROUP + (lane & 15)) * NB);
#pragma unroll
        for (int q = 0; q < NB / 2; q++) ix[q] = p[q];
    };
    auto load_x = [&](const uint32_t (&ix)[NB / 2], int j, int4v (&x)[NS]) {
        const int e = (j & 1) ? (ix[j / 2] >> 16) : (ix[j / 2] & 0xffff);
        const int at = (e ^ chunk) << 4;
        x[0] = *(const int4v *)(s_win + (live0 ? at : 0));
        if constexpr (NS == 2) x[1] = *(const int4v *)(s_win + (live1 ? at ^ 64 : 0));
    };
    uint32_t ix0[NB / 2], ix1[NB / 2];
    int4v x[2 * DX][NS];
    auto step = [&](int knext, const uint32_t (&ix)[NB / 2], uint32_t (&ixn)[NB / 2], int4v (&w)[NS][CT]) {
#pragma unroll
        for (int j = 0; j < NB; j++) {
            if (j == 0) load_ix(knext, ixn);
            if (j < NB - DX) load_x(ix, j + DX, x[(j + DX) % (2 * DX)]);
            else load_x(ixn, j + DX - NB, x[(j + DX) % (2 * DX)]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int st = 0; st < NS; st++)
#pragma unroll
                for (int c = 0; c < CT; c++) acc[j][c] = mfma_step<DT>(w[st][c], x[j % (2 * DX)][st], acc[j][c]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // The first run of phases whose windows have room; the others follow (a list of the offsets of any such phases made this loop 1 to 4 %
    // slower where all have room).
    const int fit0 = __builtin_ctz(ok_mask | 1 << kPhases), fit1 = fit0 + __builtin_ctz(~(ok_mask >> fit0));
    auto from = [&](int p) { return p * kPhase + ((wave - p * kPhase) & (W - 1)); }; // the wave's first offset of a phase
    const int kend = min(fit1, kPhases) * kPhase;
    int k = from(fit0);
    if (fit0) {
        load_w(k, fw[0]);
        __builtin_amdgcn_sched_barrier(0); // (in the loop's order: what it then waits for is counted)
        load_w(k + W, fw[1]);
        __builtin_amdgcn_sched_barrier(0);
    }
    load_ix(k, ix0);
#pragma unroll
    for (int j = 0; j < DX; j++) load_x(ix0, j, x[j]);
    for (; k + W < kend; k += 2 * W) {
        step(k + W, ix0, ix1, fw[0]);
        load_w(k + 2 * W, fw[0]);
        __builtin_amdgcn_sched_barrier(0);
        step(k + 2 * W, ix1, ix0, fw[1]);
        load_w(k + 3 * W, fw[1]);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (k < kend) step(k, ix0, ix1, fw[0]);
    if (ok_mask != 7) {
        // Windows that found no room: their rows from the feature array, G blocks at a time and the next ones on their way, also into
        // the next offset, whose part of the table is there an offset ahead.  Columns of 150 rows (two windows of three have no room),
        // 5210 tiles, 64 -> 64 fp16: 1.05 of the time of conv_rows_kernel_w2, 32 -> 64 fp32 0.99.  With these offsets among the products
        // above as well (rows of zeros) and an offset's loads waited for here before the next one's were asked for 1.31 and 1.39.
        constexpr bool QUAD = NS == 2;     // as in conv_rows_short_kernel
        constexpr int G = 2, U = NB / G, kTrRow = 80, kTrSet = SPH_GROUP * kTrRow;
        static_assert(U % 2 == 0, "two units in flight, and an offset begins with the first");
        if (QUAD) lds_barrier(); // the waves are through with the windows: each turns its rows in a part of them
        char *tr = s_win + wave * (G * NS * kTrSet);
        const int qrow = QUAD ? lane >> 2 : lane & 15, qchunk = (QUAD ? lane & 3 : lane >> 4) * 16;
        unsigned qadd[NS]; // (a chunk beyond the row's end: out of range with any row added, which is below 2^31)
#pragma unroll
        for (int st = 0; st < NS; st++) qadd[st] = !MASKED || st * 64 + qchunk < rb ? st * 64 + qchunk : kNoRow;
        auto load_id = [&](int k, int (&id)[NB]) {
#pragma unroll
            for (int j = 0; j < NB; j++) id[j] = tab[min(k, kSplitKV - 1) * R + j * SPH_GROUP + qrow];
        };
        auto gather = [&](int k, const int (&id)[NB], int u, int4v (&v)[G][NS]) {
            const unsigned lim = k < kSplitKV ? a.feat_rows : 0;
#pragma unroll
            for (int g = 0; g < G; g++) {
#pragma unroll
                for (int st = 0; st < NS; st++) {
                    const unsigned off = (unsigned)id[u * G + g] < lim ? (unsigned)(id[u * G + g] * rb) + qadd[st] : kNoRow;
                    v[g][st] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(r_feat, off, 0, 0));
                }
            }
        };
        unsigned rest = 0; // the wave's offsets there, one bit each
#pragma unroll
        for (int p = 0; p < kPhases; p++) rest |= p < fit0 || p >= fit1 ? ((1u << kPhase) - 1) << (p * kPhase) : 0;
        rest &= 0x11111111u << wave;
        auto next_of = [&](unsigned &left) {
            const int k = left ? __builtin_ctz(left) : kSplitKV;
            left &= left - 1;
            return k;
        };
        int k0 = next_of(rest), k1 = next_of(rest);
        int id0[NB], id1[NB];
        int4v v[2][G][NS];
        if (k0 < kSplitKV) {
            load_w(k0, fw[0]);
            load_id(k0, id0);
            load_id(k1, id1);
#pragma unroll
            for (int u = 0; u < 2; u++) gather(k0, id0, u, v[u]);
        }
        while (k0 < kSplitKV) {
            const int k2 = next_of(rest);
            int id2[NB];
            if constexpr (NB < 8) load_id(k2, id2);
#pragma unroll
            for (int u = 0; u < U; u++) {
                int4v y[G][NS];
                if constexpr (QUAD) { // (a wave's accesses of LDS keep their order)
#pragma unroll
                    for (int g = 0; g < G; g++)
#pragma unroll
                        for (int st = 0; st < NS; st++) *(int4v *)(tr + (g * NS + st) * kTrSet + (lane >> 2) * kTrRow + (lane & 3) * 16) = v[u & 1][g][st];
                    asm volatile("" ::: "memory");
                } else {
#pragma unroll
                    for (int g = 0; g < G; g++) y[g][0] = v[u & 1][g][0];
                }
                __builtin_amdgcn_sched_barrier(0);
                if (u + 2 < U) gather(k0, id0, u + 2, v[u & 1]);
                else gather(k1, id1, u + 2 - U, v[u & 1]);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (QUAD) {
#pragma unroll
                    for (int g = 0; g < G; g++)
#pragma unroll
                        for (int st = 0; st < NS; st++) y[g][st] = *(const int4v *)(tr + (g * NS + st) * kTrSet + (lane & 15) * kTrRow + (lane >> 4) * 16);
                    asm volatile("" ::: "memory");
                }
#pragma unroll
                for (int st = 0; st < NS; st++)
#pragma unroll
                    for (int g = 0; g < G; g++)
#pragma unroll
                        for (int c = 0; c < CT; c++) acc[u * G + g][c] = mfma_step<DT>(fw[0][st][c], y[g][st], acc[u * G + g][c]);
                __builtin_amdgcn_sched_barrier(0);
            }
            load_w(k1, fw[0]);
#pragma unroll
            for (int j = 0; j < NB; j++) id0[j] = id1[j];
            if constexpr (NB < 8) {
#pragma unroll
                for (int j = 0; j < NB; j++) id1[j] = id2[j];
            } else load_id(k2, id1);
            k0 = k1;
            k1 = k2;
        }
    }

    // the waves' sums meet in LDS: halves of the blocks first, then quarters
    lds_barrier();
    acc4 *s_x = (acc4 *)s_win;
    constexpr int H = NB / 2, Q = NB / 4;
    acc4 half[H][CT], quart[Q][CT];
    const bool up = wave & 2, odd = wave & 1;
#pragma unroll
    for (int j = 0; j < H; j++)
#pragma unroll
        for (int c = 0; c < CT; c++) s_x[((wave ^ 2) * H * CT + j * CT + c) * kWave + lane] = pick_of(up, acc[H + j][c], acc[j][c]);
    lds_barrier();
#pragma unroll
    for (int j = 0; j < H; j++)
#pragma unroll
        for (int c = 0; c < CT; c++) half[j][c] = pick_of(up, acc[j][c], acc[H + j][c]) + s_x[(wave * H * CT + j * CT + c) * kWave + lane];
    lds_barrier();
#pragma unroll
    for (int j = 0; j < Q; j++)
#pragma unroll
        for (int c = 0; c < CT; c++) s_x[((wave ^ 1) * Q * CT + j * CT + c) * kWave + lane] = pick_of(odd, half[Q + j][c], half[j][c]);
    lds_barrier();
#pragma unroll
    for (int j = 0; j < Q; j++)
#pragma unroll
        for (int c = 0; c < CT; c++) quart[j][c] = pick_of(odd, half[j][c], half[Q + j][c]) + s_x[(wave * Q * CT + j * CT + c) * kWave + lane];

    const int row0 = r0 + ((up ? H : 0) + (odd ? Q : 0)) * SPH_GROUP + (lane & 15);
    elem *out = (elem *)a.out + (long)row0 * a.ndim + col0 + chunk * 4;
#pragma unroll
    for (int c = 0; c < CT; c++) {
        const float4v sc = *(const float4v *)&s_sc[0][c * 16 + chunk * 4], sh = *(const float4v *)&s_sc[1][c * 16 + chunk * 4];
        const bool in = col0 + c * 16 + chunk * 4 < a.ndim;
#pragma unroll
        for (int b = 0; b < Q; b++)
            if (in && row0 + b * SPH_GROUP < a.book.rows) store_four<DT>(a, out + (long)b * SPH_GROUP * a.ndim + c * 16, quart[b][c], sc, sh);
    }
}


template <sph_dtype DT, int NS, int CT, bool MASKED, int NB, int W, int KC>
int launch_short(const ConvArgs &a, int nwtot, hipStream_t st)
{
    const int units = sph_div_up(a.book.rows, NB * SPH_GROUP);
    hipLaunchKernelGGL((conv_rows_short_kernel<DT, NS, CT, MASKED, NB, W, KC>), dim3(sph_xcd_grid(units), sph_div_up(nwtot, CT)),
                       dim3(W * kWave), 0, st, a, nwtot);
    return sph_check_launch("sph_conv_apply");
}

template <sph_dtype DT, int NS, int CT, bool MASKED, int NB>
int launch_split(const ConvArgs &a, int nwtot, hipStream_t st, int lds)
{
    constexpr int tab = kSplitKV * NB * SPH_GROUP * 2;
    constexpr int least = tab + 4 * (NB / 2) * CT * 1024; // the exchange of the waves' sums
    lds = lds < least ? least : lds;
    const int cap_rows = (lds - tab) / (NS * 64);
    if (int rc = set_lds(conv_rows_split_kernel<DT, NS, CT, MASKED, NB>, lds)) return rc;
    const int units = sph_div_up(a.book.rows, NB * SPH_GROUP);
    hipLaunchKernelGGL((conv_rows_split_kernel<DT, NS, CT, MASKED, NB>), dim3(sph_xcd_grid(units), sph_div_up(nwtot, CT)),
                       dim3(4 * kWave), lds, st, a, nwtot, cap_rows);
    return sph_check_launch("sph_conv_apply");
}

// Which kernel takes a call.  T: tiles times blocks of 64 columns.
enum Way { kNone, kShort1, kShort2, kByOffset, kSplit4, kSplit8 };

// us at 3x3x3, 0.4 of the bins of a grid of depth 32 ("to a row": stride 2, gathered rows to a row), the way that is taken against its
// neighbours; plain: conv_rows_kernel_* of conv.hip (with four waves a tile up to 1024 tiles, as it was), win: conv_rows_win_kernel.
//   16 / 32 rows a workgroup up to 32 / 64 tiles (one for every compute unit): 64 -> 64 fp16 26 tiles 5.5 : 6.6 : plain 16.7, 51 tiles
//     6.8 : 9.6, 66 tiles 10.3 : split 8.6; one K step and up to 32 columns, 91 tiles 5.1 : split 5.8, 131 tiles 6.7 : 6.4
//   64 rows, an offset at a time (kByOffset) where no window helps: 5x3x3 64 -> 64 512 tiles 42 : plain 53, 3x3x1 16 : 20 (1001 tiles
//     28 : 33, 2000 tiles 57 : 38); 7.2 to a row 260 tiles 24 : 33, 511 tiles 35 : 40, 999 tiles 69 : 80; 3.6 to a row 511 tiles 28 : split
//     32 : 35, 999 tiles 60 : 57 : 71; fp32 32 -> 32 3.6 to a row 999 tiles 72 : split 89 : 93, 4000 tiles 271 : 304 : 348 (before its rows
//     were asked for by quads, which took 64 -> 64 511 tiles of 7.2 to a row from 40 to 35)
//   64 rows with windows (kSplit4) up to 256 tiles, 128 rows (kSplit8) beyond, 64 -> 64 fp16: 201 tiles 12.2 : 13.1 : plain 18.7; 400 tiles
//     21.1 : 18.9 : 31; 1001 tiles 41.8 : 34.8 : 59.5; 3996 tiles 165 : 129 : 167.  fp32, whose matrix cores are the bound, up to 32 columns
//     always (32 -> 32 3996 tiles 252 : 254 : 344), 64 up to 512 (700 tiles 97 : 94).  3.6 to a row 1399 tiles 71 : 79
//   one K step: 32 -> 64 1401 tiles 33 : win 39, 2000 tiles 48 : 55, 2997 tiles 70 : 68; fp32 16 -> 64 3996 tiles 250 : 265; 32 -> 32 1001
//     tiles 16 : plain 27, 1401 tiles 22 : win 19 (fp32 16 -> 32 51 : 54, 2000 tiles 72 : 69); 32 -> 64 3.6 to a row 4000 tiles 106 : 117;
//     32 -> 32 3.6 to a row 511 tiles kByOffset 12 : split 15, 4000 tiles split 74 : win 88, 2.8 to a row 4000 tiles 64.5 : 64.9
// Which windows find room decides between kSplit4, kSplit8 and the kernels without them (kByOffset; plain or win from 1025 tiles on).  A window holds a
// plane's rows, which lie between its first and last column (sph_book.middle_run says how many), and the workgroup's own stretch of a line.
// Times over those of the kernels before the windows came, 17 680 calls (500 to 9000 tiles, 0.3 to 0.8 of the bins, columns of 5 to 170 rows,
// strides 1x1x1, 1x2x2, 2x2x2 and 2x1x1), by three, two, one of three with room: 64 -> 64 fp16 kSplit8 0.71 to 0.80, 0.83 to 0.97, 0.98 to 1.07; where
// more than 1.9 are gathered to a row kSplit4's three 0.92, its two 1.10 to 1.18; 64 -> 128 the same, two 1.04 to 1.16.  One K step into 64
// columns, more than 2 to a row: kSplit4 0.81 to 0.92, 0.87 to 1.03, 0.98 to 1.12, more than 5 to a row 0.9, 1.11, 1.22.  The lines by T beside that:
//   fp32 two K steps into 32: an offset at a time 0.64 to 0.84 beyond 1152 tiles, windows 0.66 to 1.0 (into 16, up to 2048 tiles, 0.8 of the former);
//     into 64: an offset at a time 0.78 to 0.95, windows 0.75 to 1.05 (three with room, 1300 to 5500 tiles, 0.76 to 0.90; 330 tiles 0.63, an offset at a time 0.78), beyond 6000 tiles 1.03, 0.96 to 1.11
//   rows shorter than 64 bytes into 64 columns, 16 bits and int8, up to 2 to a row: kSplit4 0.55 to 0.95 (three with room, where conv_rows_win_kernel
//     has room as well, 7000 tiles 0.99, 0.90 to 1.14; two, 1900 tiles and more 0.95 to 1.13); 2 to 5 to a row: three 0.65 to 0.97, two or one 0.73 to 0.98 up to
//     1100 tiles, 1.0 to 1.19 beyond but for 2200 (0.86 to 0.92: a round of plain is 2048); more: an offset at a time 0.72 to 0.84 up to 800 tiles
//   rows of 64 bytes into 64 columns, up to 2 to a row: 961 to 1024 tiles of submanifold books are one round of conv_rows_win_kernel (995 tiles 1.05, int8 1.07 to 1.10
//     of it; strided 1000 tiles 0.70 to 0.80);
//     1700 tiles 0.74 of it, 2000 0.8 to 0.97, 16 bits with fewer than three with room 1.07 to 1.18
//   one K step into 16 and 32 columns: fp32 into 16, fewer than three with room, 700 and 1000 tiles: an offset at a time 1.03 to 1.05, windows to 1.15 (four waves of
//     one tile were faster there); 16 bits into 32, up to 1024 tiles, three with room 0.64 (16 -> 32 0.75), an offset at a time 0.71, two or one with
//     room 0.8 to 1.0; 16 -> 32 fp16, more than 2.4 to a row, 1700 tiles: 0.76, windows 1.00
//   two blocks of columns: up to 1152 tiles of rows windows in any case (1040 tiles 0.75, neither 1.0), one K step beyond only where three have room to spare (1.0
//     per row, columns of 60 and 70 rows 1.07 to 1.20)
// Over 37 076 other calls (130 to 5500 tiles, 0.25 to 0.75 of the bins, 24 widths and types): 0.81 of the time before the windows, 234 calls more than 6 % and
// 71 more than 10 % slower (1.31 at most); by T and the rows to a row alone 0.885, 6029, 4981 and 2.16.
//   8 offsets, 45 offsets, 16 bits, one K step into 64 columns: 645 tiles 1.04 to 1.09, 990 tiles 1.10 of plain or the window kernel
//   65 to 128 columns of other than 27 offsets: 512 tiles (9 offsets 64 -> 128 f16 520 tiles 0.93, 650 1.07, 1000 1.38 of plain)

// LDS of a workgroup of 64 rows: what four, three or two of them on a compute unit leave each (where their registers let as many be
// there: up to 128 of a lane four, 168 three), by the rows its windows should hold (about half
// of the gathered rows to a row lie on a window's line, and a column or two more on either side)
template <int NS>
int split4_lds(const ConvArgs &a)
{
    const double to_a_row = (double)a.feat_rows / a.book.rows;
    const double rows = kPhases * (64 * (to_a_row > 2 ? to_a_row / 2 : 1.0) + 32);
    const double need = (rows * NS * 64 + kSplitKV * 64 * 2) / 1024;
    return (NS == 2 && to_a_row > 1.5 ? 79 : need <= 39 ? 39 : need <= 52 ? 52 : 79) * 1024;
}
constexpr int kSplit8Lds = 79 * 1024;

// Of the three windows of `rows` rows, on average, those that find room in so much LDS.
template <int NS>
int windows_with_room(const ConvArgs &a, int rows, int lds)
{
    const int cap_rows = (lds - kSplitKV * rows * 2) / (NS * 64);
    const double window = plane_window(a, rows);
    return kPhases * window <= cap_rows ? kPhases : 2 * window <= cap_rows ? 2 : 1;
}

template <sph_dtype DT, int NS, int CT>
Way pick_way(const ConvArgs &a, int nwtot, int ntiles)
{
    const double to_a_row = (double)a.feat_rows / a.book.rows;
    const long T = (long)ntiles * sph_div_up(nwtot, CT);
    const int KV = a.book.KV;
    const bool f32 = DT == SPH_F32, half = DT == SPH_F16 || DT == SPH_BF16;
    if (T <= 32) return kShort1;
    if (KV != kSplitKV) {
        if (T <= 64 && KV >= 16) return kShort2;
        return T <= (half && NS == 1 && nwtot == 4 && (KV <= 8 || KV > kSplitKV) ? 640 : 1024) ? kByOffset : kNone;
    }
    if (T <= (NS == 1 && CT <= 2 ? 128 : 64)) return kShort2;
    const int room4 = windows_with_room<NS>(a, 64, split4_lds<NS>(a)), room8 = NS == 2 ? windows_with_room<NS>(a, 128, kSplit8Lds) : 0;
    const bool two_blocks = nwtot > 4, many = T > (two_blocks ? 2304 : 1024);
    if (NS == 2 && f32) {
        if (CT < 4) return to_a_row <= 2.4 && room4 == 3 && T <= (CT == 1 ? 2048 : 1152) ? kSplit4 : kByOffset;
        if (to_a_row <= (T <= 384 ? 2.4 : 1.3) && room4 == 3 && (T <= 512 || T > 1024)) return T <= 512 ? kSplit4 : kSplit8;
        return T <= 6000 ? kByOffset : kNone;
    }
    if (NS == 2) {
        if (to_a_row > (CT == 4 ? 2.5 : 2.4)) {
            if (T <= 1024) return kByOffset;
            return to_a_row > 5 || T > 1400 ? kNone : room4 == 3 ? kSplit4 : kByOffset;
        }
        if (CT < 4 || !many) return T <= 256 ? kSplit4 : kSplit8;
        if (room8 == 3) return kSplit8;
        if (two_blocks) return kNone;
        return to_a_row >= 1.9 && room4 == 3 ? kSplit4 : room8 == 2 ? kSplit8 : kNone;
    }
    if (CT == 4 && f32) {
        if (T <= 1900 || (to_a_row <= 2 && (T <= 6000 || room4 == 3))) return kSplit4;
        return T <= 6000 && (room4 == 3 || (room4 == 2 && to_a_row <= 5)) ? kSplit4 : kNone;
    }
    if (CT == 4) {
        if (!two_blocks && a.row_bytes < 64) {
            const bool win = plane_window(a, R) <= 255; // conv_rows_win_kernel's has room for a tile
            if (to_a_row > 5) return T <= 768 ? kByOffset : kNone;
            if (to_a_row > 2) return room4 == 3 || T <= 1152 || (T > 2048 && T <= 2304) ? kSplit4 : kNone;
            return !win || T <= (room4 == 3 ? 6000 : 1700) ? kSplit4 : kNone;
        }
        const bool win_round = T > 960 && T <= 1024 && to_a_row <= 1.3 && book_plane_stride(&a.book) == 1;
        if (!two_blocks && to_a_row <= 2) return !win_round && T <= (room4 == 3 || !half ? 2048 : 1900) ? kSplit4 : kNone;
        if (!many) return kSplit4;
        if (two_blocks) return to_a_row <= 4.5 && windows_with_room<NS>(a, 64, split4_lds<NS>(a) * 9 / 10) == 3 ? kSplit4 : kNone;
        if (room4 == 3) return kSplit4;
        return to_a_row <= 5 && (room4 == 2 || (T <= 2700 && book_plane_stride(&a.book) == 1)) ? kSplit4 : kNone;
    }
    if (to_a_row <= 2.4) {
        if (T > (f32 ? 1536 : 1024)) return kNone;
        return room4 == 3 || (f32 && CT == 2) || many ? kSplit4 : kByOffset;
    }
    if (CT == 1) return T <= (f32 ? 1024 : 640) ? kByOffset : T <= 1024 ? kSplit4 : kNone;
    if (f32) return T <= 640 ? kByOffset : kSplit4;
    return T <= 2048 ? kByOffset : to_a_row > 3.3 ? kSplit4 : kNone;
}

template <sph_dtype DT, int NS, int CT, bool MASKED>
int launch_m(const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
    switch (pick_way<DT, NS, CT>(a, nwtot, ntiles)) {
    case kShort1: return launch_short<DT, NS, CT, MASKED, 1, 8, 4>(a, nwtot, st);
    case kShort2: return launch_short<DT, NS, CT, MASKED, 2, 8, 4>(a, nwtot, st);
    case kSplit4: return launch_split<DT, NS, CT, MASKED, 4>(a, nwtot, st, split4_lds<NS>(a));
    case kSplit8:
        if constexpr (NS == 2) return launch_split<DT, NS, CT, MASKED, 8>(a, nwtot, st, kSplit8Lds);
    default: return launch_short<DT, NS, CT, MASKED, 4, 4, 1>(a, nwtot, st);
    }
}

template <sph_dtype DT, int NS, int CT>
int launch_ct(const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
    if (a.row_bytes < NS * 64) return launch_m<DT, NS, CT, true>(a, nwtot, ntiles, st);
    return launch_m<DT, NS, CT, false>(a, nwtot, ntiles, st);
}

template <sph_dtype DT, int NS>
int launch_ns(const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
    switch (nwtot) {
    case 1: return launch_ct<DT, NS, 1>(a, nwtot, ntiles, st);
    case 2: return launch_ct<DT, NS, 2>(a, nwtot, ntiles, st);
    default: return launch_ct<DT, NS, 4>(a, nwtot, ntiles, st);
    }
}

template <sph_dtype DT>
int launch_dt(const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
    return a.nsteps == 1 ? launch_ns<DT, 1>(a, nwtot, ntiles, st) : launch_ns<DT, 2>(a, nwtot, ntiles, st);
}

} // namespace

bool sph_rows_split_ok(sph_dtype dt, const ConvArgs &a, int nwtot, int ntiles)
{
    if ((double)a.feat_rows * a.row_bytes >= 2147483648.0) return false; // lane offsets are 31-bit
    const int ct = nwtot < 4 ? nwtot : 4;
    auto way = [&](auto type) {
        constexpr sph_dtype DT = decltype(type)::value;
        if (a.nsteps == 1) return ct == 1 ? pick_way<DT, 1, 1>(a, nwtot, ntiles) : ct == 2 ? pick_way<DT, 1, 2>(a, nwtot, ntiles) : pick_way<DT, 1, 4>(a, nwtot, ntiles);
        return ct == 1 ? pick_way<DT, 2, 1>(a, nwtot, ntiles) : ct == 2 ? pick_way<DT, 2, 2>(a, nwtot, ntiles) : pick_way<DT, 2, 4>(a, nwtot, ntiles);
    };
    if (dt == SPH_F32) return way(std::integral_constant<sph_dtype, SPH_F32>()) != kNone;
    if (dt == SPH_I8) return way(std::integral_constant<sph_dtype, SPH_I8>()) != kNone;
    return way(std::integral_constant<sph_dtype, SPH_F16>()) != kNone;
}

int sph_rows_split_launch(sph_dtype dt, const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
    switch (dt) {
    case SPH_F32: return launch_dt<SPH_F32>(a, nwtot, ntiles, st);
    case SPH_F16: return launch_dt<SPH_F16>(a, nwtot, ntiles, st);
    case SPH_BF16: return launch_dt<SPH_BF16>(a, nwtot, ntiles, st);
    default: return launch_dt<SPH_I8>(a, nwtot, ntiles, st);
    }
}
