// By-row convolution (gfx950) on long grids, rows of up to 64 bytes (one MFMA K step) into 17 to 32 columns: the weight of all
// offsets stays in a compute unit's LDS while its waves walk through the grid.
//
// One workgroup of twelve waves per compute unit; a wave takes units of 64 rows, one after the other, and shares nothing but the
// weight with the others.  As in conv_rows_win_kernel of conv.hip the offsets go in phases of nine: the rows a phase gathers lie close
// together and come to LDS as they lie, the phase's table is rewritten as one byte per (offset, row), and every gather is an LDS
// read.  A wave works one phase ahead: while it multiplies, the next phase's window is on its way to registers and the
// table of the one after that behind it, also from one unit to the next.  The sums are in the order of conv_rows_win_kernel.
// What bounds it: a wave's own chain (LDS reads, products, and between phases the table: 44 % of its time it waits, 23 % for
// its turn) with three waves on a SIMD; the LDS is 43 % busy, the vector memory path 41, the vector units 35, the matrix cores 29.
// There the weight, 2 KB for every offset and 64 rows, was two fifths of the vector memory path's work (64 % busy) and stood behind
// the windows in its queue.  us, 3x3x3, 12 744 tiles of 10.9 pairs a row, f16: 16 -> 32 140 -> 119, 32 -> 32 147 -> 132.
// Measured and not kept: the window a phase ahead with the weight still from memory 167 (waves wait for weights behind windows);
// one wave for 128 rows 217; eleven waves with windows of 132 rows 127 and 135; rows of 64 bytes as they lie instead of in planes
// 15 of 35 million LDS cycles are bank conflicts.
#include "rows_hold.h"

namespace {

constexpr int kPhase = 9;            // offsets per window
constexpr int kRows = 64;            // rows of a unit, which a wave takes
constexpr int kWinRows64 = 116;      // rows of 64 bytes that a wave's window holds, the row of zeros among them
constexpr int kWin = kWinRows64 * 64; // its bytes
constexpr int kTab = kPhase * kRows; // bytes of a phase's table
constexpr int kMaxRows = 255;        // most rows of a window: a byte names any of them or the row of zeros
constexpr int kWaves = 12;           // three on a SIMD
constexpr int CT = 2;                // tiles of 16 columns
constexpr int kAffine = 2 * 64 * 4;  // bytes of scale and shift
constexpr int kPerWave = kWin + 2 * kTab;
constexpr int kCUs = 256;

template <sph_dtype DT, bool MASKED>
__global__ __launch_bounds__(kWaves * kWave) __attribute__((amdgpu_waves_per_eu(3))) void conv_rows_hold_kernel(ConvArgs a)
{
    typedef typename Traits<DT>::elem elem;
    typedef typename Traits<DT>::acc4 acc4;
    typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
    constexpr int NB = kRows / SPH_GROUP;              // blocks of 16 rows
    constexpr int NP = (kWin + kWave * 16 - 1) / (kWave * 16);  // loads of a window
    constexpr int OPL = kWave * 4 / kRows;             // offsets per load of the table
    constexpr int NT = (kPhase + OPL - 1) / OPL;       // loads of a phase's table
    static_assert(NP <= kPhase, "a phase has room for the next one's loads");
    extern __shared__ __attribute__((aligned(16))) char s_mem[];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int KV = a.book.KV, rb = a.row_bytes;
    const int nph = (KV + kPhase - 1) / kPhase;
    const bool plain = DT != SPH_I8 && !a.scale && !a.shift && !a.relu;
    const bool relu = DT != SPH_I8 && a.relu;

    // shared: scale and shift, the weight's fragments as they lie; a wave's own: the window, and two phases' tables
    // ([kPhase][16 rows][NB blocks] bytes)
    float *s_scale = (float *)s_mem, *s_shift = s_scale + 64;
    char *s_w = s_mem + kAffine, *s_win = s_w + KV * CT * (kWave * 16) + wave * kPerWave, *s_tabs = s_win + kWin;
    for (int i = threadIdx.x; i < KV * CT * kWave; i += kWaves * kWave) ((int4v *)s_w)[i] = ((const int4v *)a.wp)[i];
    if (threadIdx.x < 64) {
        const int col = min((int)threadIdx.x, a.ndim - 1);
        s_scale[threadIdx.x] = a.scale ? a.scale[col] : 1.f;
        s_shift[threadIdx.x] = DT != SPH_I8 && a.shift ? a.shift[col] : 0.f;
    }
    __syncthreads(); // the only one: from here on every wave goes its own way

    // An XCD's workgroups walk through a contiguous run of units side by side: their windows come from its L2.
    const int ntiles = (a.book.rows + R - 1) / R, units = ntiles * (R / kRows);
    const int xcd = blockIdx.x % SPH_NUM_XCD, wgs = gridDim.x / SPH_NUM_XCD;
    const int u_end = (int)((long)units * (xcd + 1) / SPH_NUM_XCD), u_step = wgs * kWaves;
    int u = (int)((long)units * xcd / SPH_NUM_XCD) + (int)(blockIdx.x / SPH_NUM_XCD) * kWaves + wave;
    if (u >= u_end) return;

    const int chunk = lane >> 4;
    const bool live_chunk = chunk * 16 < rb;
    const int choff = live_chunk ? chunk * 16 : 0;
    const int t_off = lane / (kRows / 4), t_row = lane % (kRows / 4) * 4; // a lane's offset in a load of the table, and its first of four rows
    const int t_dst = t_off * kRows + t_row % SPH_GROUP * NB + t_row / SPH_GROUP;
    // Rows of 64 bytes lie as four planes of 16-byte chunks: the sixteen lanes that read the same chunk of neighbouring rows find
    // them side by side (row by row they lie in a quarter of the banks), and so do those that write four rows.
    constexpr int kPlane = kWinRows64 * 16;
    static_assert(kPlane % 256 == 64, "four planes, four quarters of the banks");
    const int w_dst = MASKED ? lane * 16 : (lane & 3) * kPlane + (lane >> 2) * 16;
    int4v tn[NT]; // the table of the phase after the next, on its way
    auto table = [&](int unit) {
        return __builtin_amdgcn_make_buffer_rsrc((void *)(a.book.tile_nbr + (long)(unit / (R / kRows)) * KV * R + unit % (R / kRows) * kRows), 0,
                                                 KV * R * 4 - unit % (R / kRows) * kRows * 4, kRsrcFlags);
    };
    auto load_tab = [&](int unit, int ph) { // (behind a phase's last offset: that one's entries again, which change nothing)
        const __amdgpu_buffer_rsrc_t r = table(unit);
        const int nk = min(kPhase, KV - ph * kPhase);
#pragma unroll
        for (int i = 0; i < NT; i++)
            tn[i] = (int4v)__builtin_amdgcn_raw_buffer_load_b128(r, (min(i * OPL + t_off, nk - 1) * R + t_row) * 4, ph * kPhase * (R * 4), 0);
    };
    // A phase's table, which has arrived, to LDS.  lo: the lowest row the phase gathers; nrow: how many
    // from there to the highest; bytes: of its window, 0 where it has none.
    struct Phase { int lo, nrow, bytes; };
    auto prepare = [&](int ph, int parity) -> Phase {
        char *tab = s_tabs + parity * kTab + t_dst;
        const int nk = min(kPhase, KV - ph * kPhase);
        unsigned lo = ~0u; // (-1, no pair, is the largest unsigned number)
        int hi = -1;
#pragma unroll
        for (int i = 0; i < NT; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                lo = min(lo, (unsigned)tn[i][e]);
                hi = max(hi, tn[i][e]);
            }
        lo = min(lo, 0x7fffffffu);
        const int low = __builtin_amdgcn_readlane(~wave_max_last(~(int)lo), kWave - 1); // the least of the complements is the largest
        hi = __builtin_amdgcn_readlane(wave_max_last(hi), kWave - 1);
        Phase p = {low, hi < 0 ? 0 : hi - low + 1, 0};
        // (a row behind the array's end, which no table of the library's own names: the walk without a window looks at every entry)
        if (p.nrow <= kMaxRows && (p.nrow + 1) * rb <= kWin && hi < a.feat_rows) {
            p.bytes = p.nrow * rb;
#pragma unroll
            for (int i = 0; i < NT; i++)
                if ((i + 1) * OPL <= kPhase || i * OPL + t_off < kPhase) {
#pragma unroll
                    for (int e = 0; e < 4; e++) { // (-1 - low is a large unsigned number)
                        const unsigned v = min((unsigned)(tn[i][e] - low), (unsigned)p.nrow);
                        tab[i * OPL * kRows + e * NB] = (char)v;
                    }
                }
            if (nk < kPhase) { // empty slots behind the kernel's last offset
#pragma unroll
                for (int i = 0; i < NT; i++)
                    if (i * OPL + t_off >= nk && i * OPL + t_off < kPhase) {
#pragma unroll
                        for (int e = 0; e < 4; e++) tab[i * OPL * kRows + e * NB] = (char)p.nrow;
                    }
            }
        }
        return p;
    };
    // Loads of a phase's window: bytes as they lie in the feature array, zeros behind them.
    uint4v piece[NP];
    auto load_piece = [&](const __amdgpu_buffer_rsrc_t &r, int i) { piece[i] = __builtin_amdgcn_raw_buffer_load_b128(r, lane * 16, i * (kWave * 16), 0); };
    auto window = [&](const Phase &p) { return __builtin_amdgcn_make_buffer_rsrc((void *)(a.feat + (long)p.lo * rb), 0, p.bytes, kRsrcFlags); };

    load_tab(u, 0);
    Phase next = prepare(0, 0);
    {
        const __amdgpu_buffer_rsrc_t r = window(next);
#pragma unroll
        for (int i = 0; i < NP; i++) load_piece(r, i);
    }
    if (nph > 1) load_tab(u, 1);
    else if (u + u_step < u_end) load_tab(u + u_step, 0);
    int parity = 0;
    for (; u < u_end; u += u_step) {
        acc4 acc[NB][CT];
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int c = 0; c < CT; c++) acc[j][c] = acc4{0, 0, 0, 0};
        for (int ph = 0; ph < nph; ph++, parity ^= 1) {
            const Phase cur = next;
            const char *tab = s_tabs + parity * kTab, *w = s_w + ph * kPhase * CT * (kWave * 16) + lane * 16;
            const int nk = min(kPhase, KV - ph * kPhase);
#pragma unroll
            for (int i = 0; i < NP; i++)
                if ((i + 1) * kWave * 16 <= kWin || (i * kWave + lane) * 16 < kWin) *(uint4v *)(s_win + w_dst + i * (MASKED ? kWave * 16 : kWave * 4)) = piece[i];
            // the phase after this one, and the table of the one after that
            const bool last = ph == nph - 1;
            const int u1 = last ? u + u_step : u, p1 = last ? 0 : ph + 1;
            next = Phase{0, 0, 0};
            if (u1 < u_end) {
                next = prepare(p1, parity ^ 1);
                const int u2 = p1 == nph - 1 ? u1 + u_step : u1, p2 = p1 == nph - 1 ? 0 : p1 + 1;
                if (u2 < u_end) load_tab(u2, p2);
            }
            const __amdgpu_buffer_rsrc_t r = window(next);
            if (cur.bytes > 0) {
                // table entries two offsets ahead, rows and weights one
                auto entries = [&](int o) { return *(const uint32_t *)(tab + min(o, kPhase - 1) * kRows + (lane & 15) * NB); };
                auto rows = [&](uint32_t pk, int4v (&x)[NB]) {
#pragma unroll
                    for (int j = 0; j < NB; j++) {
                        // lanes on 16-byte chunks behind the row's end read zeros too
                        const int row = (MASKED && !live_chunk) ? cur.nrow : (pk >> (8 * j)) & 255;
                        x[j] = *(const int4v *)(s_win + (MASKED ? (int)__umul24(row, rb) + choff : row * 16 + chunk * kPlane));
                    }
                };
                auto weights = [&](int o, int4v (&f)[CT]) {
#pragma unroll
                    for (int c = 0; c < CT; c++) f[c] = *(const int4v *)(w + (min(o, nk - 1) * CT + c) * (kWave * 16));
                };
                uint32_t e1 = entries(0), e2 = entries(1);
                int4v x[2][NB], f[2][CT];
                rows(e1, x[0]);
                weights(0, f[0]);
                // offsets past the kernel's last find a table of empty slots
#pragma unroll
                for (int o = 0; o < kPhase; o++) {
                    if (o + 1 < kPhase) {
                        rows(e2, x[(o + 1) & 1]);
                        weights(o + 1, f[(o + 1) & 1]);
                        e2 = entries(o + 2);
                    }
                    if (o < NP) load_piece(r, o);
#pragma unroll
                    for (int j = 0; j < NB; j++)
#pragma unroll
                        for (int c = 0; c < CT; c++) acc[j][c] = mfma_step<DT>(f[o & 1][c], x[o & 1][j], acc[j][c]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                // the rows lie too far apart: gathers from the feature array, three offsets at a time (zeros from behind its end for
                // slots without a pair and for lanes on chunks behind the row's end)
                const __amdgpu_buffer_rsrc_t rt = table(u), rf = __builtin_amdgcn_make_buffer_rsrc((void *)a.feat, 0, a.feat_rows * rb, kRsrcFlags);
                const int n = cur.nrow > 0 ? nk : 0;
#pragma unroll 1
                for (int o = 0; o < n; o += 3) {
                    int id[3][NB];
                    uint4v x[3][NB];
#pragma unroll
                    for (int k = 0; k < 3; k++)
#pragma unroll
                        for (int j = 0; j < NB; j++)
                            id[k][j] = __builtin_amdgcn_raw_buffer_load_b32(rt, (j * SPH_GROUP + (lane & 15)) * 4, (ph * kPhase + min(o + k, n - 1)) * (R * 4), 0);
#pragma unroll
                    for (int k = 0; k < 3; k++)
#pragma unroll
                        for (int j = 0; j < NB; j++) {
                            const unsigned row = o + k < n ? min((unsigned)id[k][j], (unsigned)a.feat_rows) : a.feat_rows;
                            x[k][j] = __builtin_amdgcn_raw_buffer_load_b128(rf, row * rb + (live_chunk ? choff : a.feat_rows * rb), 0, 0);
                        }
#pragma unroll
                    for (int k = 0; k < 3; k++) {
                        int4v f[CT];
#pragma unroll
                        for (int c = 0; c < CT; c++) f[c] = *(const int4v *)(w + (min(o + k, n - 1) * CT + c) * (kWave * 16));
#pragma unroll
                        for (int j = 0; j < NB; j++)
#pragma unroll
                            for (int c = 0; c < CT; c++) acc[j][c] = mfma_step<DT>(f[c], (int4v)x[k][j], acc[j][c]);
                    }
                }
#pragma unroll
                for (int i = 0; i < NP; i++) load_piece(r, i);
            }
        }

        // a lane holds four consecutive columns of one row per block and column tile
        const int nrows = a.book.rows - u * kRows;
        elem *out = (elem *)a.out + (long)u * kRows * a.ndim;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int row = b * SPH_GROUP + (lane & 15);
            if (row >= nrows) continue;
#pragma unroll
            for (int c = 0; c < CT; c++) {
                const int col = c * 16 + (lane >> 4) * 4;
                if (col >= a.ndim) continue;
                union { elem e[4]; uint32_t w[sizeof(elem)]; } v;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    float y = DT == SPH_I8 ? (float)(int)acc[b][c][j] : (float)acc[b][c][j];
                    if (!plain) {
                        y = y * s_scale[col + j] + s_shift[col + j];
                        if (relu) y = y > 0.f ? y : 0.f;
                    }
                    v.e[j] = to_elem<DT>(y);
                }
                uint32_t *dst = (uint32_t *)(out + (long)row * a.ndim + col);
#pragma unroll
                for (int q = 0; q < (int)sizeof(elem); q++) dst[q] = v.w[q];
            }
        }
    }
}

inline size_t hold_lds(int KV) { return (size_t)kAffine + (size_t)KV * CT * (kWave * 16) + (size_t)kWaves * kPerWave; }

template <sph_dtype DT>
int launch(const ConvArgs &a, hipStream_t st)
{
    const size_t lds = hold_lds(a.book.KV);
    auto go = [&](auto kernel) -> int {
        if (int rc = set_lds(kernel, lds)) return rc;
        hipLaunchKernelGGL(kernel, dim3(kCUs), dim3(kWaves * kWave), lds, st, a);
        return sph_check_launch("sph_conv_apply");
    };
    return a.row_bytes < 64 ? go(conv_rows_hold_kernel<DT, true>) : go(conv_rows_hold_kernel<DT, false>);
}

} // namespace

// The weight and twelve waves' windows have to fit the LDS (up to 29 offsets).  Times of this kernel over those of conv.hip, 3x3x3:
//   tiles                       1100  1300  1540  1800  2040  2500  3100  4000  6000  9000 12700
//   f16 32 -> 32, 0.4 of bins   1.15  1.16  1.03  1.28  1.24  1.01  0.94  0.97  0.90  0.87  0.88
//   f16 16 -> 32                1.06  1.05  1.03  1.27  1.28  1.02  0.99  0.98  0.88  0.86  0.90
//   fp32 16 -> 32               1.00  0.97  0.97  1.38  1.37  0.98  1.02  1.05  0.95  0.96  0.99   (3x3x1: 0.81 0.78 0.85 at the end)
//   int8 64 -> 32               1.09  1.08  0.95  1.26  1.21  0.99  0.89  0.95  0.84  0.80  0.83
//   stride 2, f16 16 -> 32      0.86  0.73  0.89  0.77  0.83  0.78  0.73  0.60  0.60  0.55  0.58   (its window of 64 rows' gathers fits, that of
//   stride 2, bf16 24 -> 24     0.90  0.89  0.91  0.91  0.93  0.84  0.89  0.79  0.75  0.71  0.73    128 rows' does not)
//   stride 2, f16 32 -> 32      1.12  1.08  1.08  1.30  1.24  1.12  1.17  1.06  0.99  1.00  1.06   (neither fits)
//   stride 1,2,2, f16 32 -> 32  1.43  1.35  1.16  1.53  1.52  1.44  1.44  1.39  1.35  1.37  1.48   (that of 128 rows fits)
//   stride 1,2,2, f16 16 -> 32  1.00  0.95  0.85  1.03  1.01  0.95  0.95  0.91  0.84  0.84  0.87
// 16 columns gain nothing (f16 16 -> 16 1.07 to 1.11 on the longest grids), 45 offsets leave room for eight waves (1.08).
// Rows of 64 bytes in 16 bits and int8 only where the caller says how far apart a plane's rows lie: those of 64 rows have to find room among 116
// (7500 tiles, 97 rows 0.76 to 0.87, 103 rows 0.86 to 0.90, 114 rows 1.06 to 1.17, 138 rows 1.34 to 1.64, 184 rows 1.16 to 1.42), as a phase without a
// window is three round trips of gathers for every three offsets; or those of 128 rows find none in the other kernel's window either (248 rows 1.16
// to 1.41, 298 and more 0.81 to 0.91).  fp32, which waits for its matrix cores, gains in any case (0.75 to 0.96).  A window for every three offsets of a phase
// without one takes registers that the usual one then misses: 29 rows a column 1.18 to 1.44, but 13 rows 1.08 to 1.13 where it was 0.88 to 0.93.
// A round of the chip's 3072 waves (1536 tiles) that is mostly empty counts on short grids: strided layers on 1537 to 2303 tiles, and on 3073 to 3455, are
// not taken in fp32 (4 -> 32 1.08 to 1.23), and from 1537 to 2047 not in 16 bits where columns are deep (29 rows 1.17 to 1.32; 8 and 13 rows 0.56
// to 0.8; of stride 2 with two gathered rows to a row, 25 to 50 rows, 0.71 to 0.82).  Kernels of nine offsets or fewer are one phase, with nothing to work ahead of (8 offsets 1.06 to 1.28).
bool sph_rows_hold_ok(sph_dtype dt, const ConvArgs &a, int nwtot, int ntiles)
{
    if (a.nsteps != 1 || nwtot != CT || hold_lds(a.book.KV) > 160 * 1024 || (double)a.feat_rows * a.row_bytes >= 1073741824.0) return false;
    const double gathered = a.feat_rows / (double)a.book.rows; // to a row
    const bool said = book_plane_rows(&a.book) > 0;
    const double window = plane_window(a, kRows);
    if (a.row_bytes > 48) {
        if (gathered > 1.25) return false;
        if (dt != SPH_F32 && !(said && (window <= 104 || plane_window(a, R) > 280))) return false;
    }
    if (ntiles > 5000) return true;
    if (gathered <= 2 || ntiles <= 1024 || a.book.KV <= kPhase) return false;
    if (dt == SPH_F32) return ntiles <= 1536 || (ntiles >= 2304 && (ntiles <= 3072 || ntiles >= 3456));
    return ntiles <= 1536 || ntiles >= 2048 || (said && (window <= 170 || book_plane_rows(&a.book) <= 32));
}

int sph_rows_hold_launch(sph_dtype dt, const ConvArgs &a, hipStream_t st)
{
    switch (dt) {
    case SPH_F32: return launch<SPH_F32>(a, st);
    case SPH_F16: return launch<SPH_F16>(a, st);
    case SPH_BF16: return launch<SPH_BF16>(a, st);
    default: return launch<SPH_I8>(a, st);
    }
}
