// Gather-GEMM-scatter convolution by groups with the weight stationary in registers (gfx950), for long grids.
//
// The kernels of conv.hip give a tile of 128 rows to a workgroup, which loads the weight fragments of a group with the
// group: 8 of the 10 KiB that a group of 16 pairs takes through the compute unit's vector memory path at 64 -> 64 in 16 bit.
// All 27 offsets' fragments are 216 KiB, which no LDS holds but a compute unit's registers do (512 KiB).  So here a workgroup is
// as large as a compute unit and stays for many tiles; three stages of waves keep the fragments of a third of the offsets each,
// and the tiles pass from stage to stage, one barrier a tile, with their accumulators in LDS (four tiles in flight):
//   stage 3 gives a tile its first sums (the middle offset's run, or zeros),
//   stages 0, 1, 2 add their offsets' groups, one stage at a time, so that no two waves add to a row at once,
//   stage 3 writes the tile out with the epilogue and begins the next one in its place.
// With 64 output columns two waves share a stage, 32 columns each (the fragments of nine offsets for 64 columns of 128-byte rows
// are 288 registers, and one wave a SIMD waits for its own chain: 81 us against 78 where 126 was the start); with fewer columns a
// compute unit holds two or three workgroups.  A row's sum begins with its middle pair and goes on with the offsets ascending.
//
// What bounds it: not one unit.  8 scans of 64 -> 64 bf16, 5890 tiles, inputs from memory: 126 us before, 78 now; a tile's step
// is 5700 cycles of the two SIMDs with two gathering waves, the LDS busy 44 % of it, the texture addresser 60 %, the matrix
// cores 16 %, a wave's wait for LDS and rows the rest; without row loads 71.  An accumulator row costs the LDS most at its write
// (measured alone: 246 bytes a clock read, 77 written, 51 written where rows are strewn).  Strided 32 -> 64 fp16, 12 744 tiles,
// 165 -> 109 us (LDS 59 %); int8 64 -> 64, 2376 tiles, 39 -> 31; 64 -> 64 fp16, 2376 tiles, 56 -> 37; 32 -> 64 fp32 96 -> 65.
// Without an effect: the next group's sums read early or late, accumulator rows without bank conflicts among neighbours, indices
// requested two passes ahead, wave priorities.
#include "relay.h"

namespace {

constexpr int kRelayStages = 4;  // tiles in flight = accumulator tiles in LDS
constexpr int kRelayPart = 9;    // offsets a gathering wave keeps the fragments of
constexpr int kOut = (int)0x80000000u; // lane offset beyond every array the kernel reads (all are below 2 GiB): the load returns zeros

// A workgroup has NH waves per stage, each with CW column tiles of sixteen of the NH * CW.
template <int CT> struct RelayShape {
    static constexpr int NH = CT == 4 ? 2 : 1, CW = CT / NH;
    static constexpr int kThreads = kRelayStages * NH * kWave;
    static constexpr int LDW = CT * 16 + 4;
    static constexpr int kTileBytes = (R + 1) * LDW * 4;
};

// Fragments of offset k for the CW column tiles of block `half`.  Row m of tile c is column CW * 4 * (m / 4) + 4 * c + m % 4 of
// the block, so that a lane, which holds four rows of each tile's product, holds CW * 4 CONSECUTIVE columns.
template <int NS, int CT, int CW>
__device__ __forceinline__ void relay_weight(__amdgpu_buffer_rsrc_t r_w, int k, int half, int lane, int4v (&fw)[NS][CW])
{
#pragma unroll
    for (int c = 0; c < CW; c++) {
        const int m = lane & 15, col = half * CW * 16 + CW * 4 * (m >> 2) + 4 * c + (m & 3);
        const int off = (col >> 4) * (kWave * 16) + ((lane & 48) | (col & 15)) * 16;
#pragma unroll
        for (int st = 0; st < NS; st++)
            fw[st][c] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(r_w, off + (k * NS + st) * CT * (kWave * 16), 0, 0));
    }
}

// v holds four values per lane of sixteen, one for each quarter of the wave: out[u] = quarter u's, in all quarters.
__device__ __forceinline__ void quarters(int v, int (&out)[4])
{
    const auto a = __builtin_amdgcn_permlane16_swap((unsigned)v, (unsigned)v, false, false);       // quarters 0 0 2 2 and 1 1 3 3
    const auto b = __builtin_amdgcn_permlane32_swap(a[0], a[0], false, false);
    const auto c = __builtin_amdgcn_permlane32_swap(a[1], a[1], false, false);
    out[0] = (int)b[0];
    out[2] = (int)b[1];
    out[1] = (int)c[0];
    out[3] = (int)c[1];
}

// A gathering wave: offsets k0 .. k0 + 8 of every tile, columns of block `half`.  It goes over a tile in passes: pass p takes
// group p of each of its up to nine offsets (one pass on most scenes; 1.4 at 3.3 pairs per row).  Slot j of a pass is offset k0 + j; the rows of slot j
// are in register set j % 5 and are requested when slot j - 5 or j + 4 is done, their indices a pass before that.
template <sph_dtype DT, int NS, int CT, bool MASKED, bool RUN>
__device__ __forceinline__ void relay_gather(const ConvArgs &a, char *s_acc, int stage, int half, int lane, int first, int step, int n)
{
    typedef typename Traits<DT>::acc4 acc4;
    typedef RelayShape<CT> S;
    constexpr int CW = S::CW;
    constexpr int NJ = kRelayPart, NF = 5;
    static_assert(NJ == 9, "the order of the requests is written for nine offsets");
    const int KV = a.book.KV, kc = KV / 2;
    const int part = (KV + kRelayStages - 2) / (kRelayStages - 1), k0 = stage * part; // offsets of a wave (at most NJ), and the first
    const int ntiles = (a.book.rows + R - 1) / R;
    const __amdgpu_buffer_rsrc_t r_feat = __builtin_amdgcn_make_buffer_rsrc((void *)a.feat, 0, a.feat_rows * a.row_bytes, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_w = __builtin_amdgcn_make_buffer_rsrc((void *)a.wp, 0, KV * NS * CT * kWave * 16, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_gat = __builtin_amdgcn_make_buffer_rsrc((void *)a.book.grp_gather, 0, ntiles * a.cap * SPH_GROUP * 4, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_own = __builtin_amdgcn_make_buffer_rsrc((void *)a.book.grp_owner, 0, ntiles * a.cap * SPH_GROUP * 4, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_ko = __builtin_amdgcn_make_buffer_rsrc((void *)a.book.tile_koff, 0, ntiles * (KV + 1) * 2, kRsrcFlags);
    const int slot_lane = (lane & 15) * 4;
    const int chunk = (lane >> 4) * 16;
    const unsigned bit = 1u << (lane >> 4);
    const int acc_lane = half * (CW * 64) + (lane >> 4) * (CW * 16); // byte offset of the lane's CW * 4 columns inside an accumulator row
    // lane j < part follows offset k0 + j
    const int k_lane = min(k0 + min(lane, part), KV);
    const int k_next = (lane < part && !(RUN && k_lane == kc)) ? min(k_lane + 1, KV) : k_lane;

    int4v fw[NJ][NS][CW];
#pragma unroll
    for (int j = 0; j < NJ; j++) relay_weight<NS, CT, CW>(r_w, k0 + j, half, lane, fw[j]);

    // the workgroup's tiles are first, first + step, ...: n of them
    const int tile_end = first + n * step, tile_last = tile_end - step;
    auto load_ko = [&](int t, int &lo, int &hi) {
        const int at = min(t, tile_last) * (KV + 1);
        lo = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r_ko, k_lane * 2, at * 2, 0);
        hi = (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r_ko, k_next * 2, at * 2, 0);
    };
    // the pass whose indices are requested next: group f_p of every offset of tile f_tile
    int f_tile = first, f_p = 0, f_lo, f_hi, x_lo, x_hi;
    load_ko(f_tile, f_lo, f_hi);
    load_ko(f_tile + step, x_lo, x_hi);

    int4v fa[NF][NS];   // gathered rows
    int own[NJ];        // LDS addresses of their owners' accumulators
    int gi[3], ow[3];   // indices of slots 0..3 (a quarter of the wave each), 4 (all quarters alike) and 5..8
    unsigned mask0, mask1;
    bool last0, last1;
    int tile0, tile1, buf0, buf1;

    // where group f_p of each offset begins (byte offset), which offsets have one, whether none has another
    auto pass_groups = [&](unsigned &mask, bool &last) -> int {
        const int g = f_lo + f_p;
        const bool valid = g < f_hi && f_tile < tile_end;
        last = __builtin_amdgcn_ballot_w64(g + 1 < f_hi) == 0;
        mask = (unsigned)__builtin_amdgcn_ballot_w64(valid);
        return valid ? (f_tile * a.cap + g) * (SPH_GROUP * 4) : kOut;
    };
    auto advance = [&](bool last) {
        f_tile = last ? f_tile + step : f_tile;
        f_p = last ? 0 : f_p + 1;
        f_lo = last ? x_lo : f_lo;
        f_hi = last ? x_hi : f_hi;
        load_ko(f_tile + step, x_lo, x_hi);
    };
    auto load_idx = [&](int i, int at) {
        gi[i] = __builtin_amdgcn_raw_buffer_load_b32(r_gat, at, 0, 0);
        ow[i] = __builtin_amdgcn_raw_buffer_load_b32(r_own, at, 0, 0);
    };
    auto place = [&](int at, int i) { // the lane's index entry: slots i, i + 1, ... for the quarters of the wave
        return __shfl(at, i + (lane >> 4), kWave) + slot_lane;
    };
    // byte offset of the row to gather and accumulator address of a pair; a slot without a pair gathers zeros and adds them
    // to the scratch row
    auto finish = [&](int i, bool live, int tile, int buf, int &off, int &acc) {
        const int r0 = tile * R, nrows = min(R, a.book.rows - r0), rl = ow[i] - r0;
        const bool ok = live && (unsigned)rl < (unsigned)nrows && (unsigned)gi[i] < (unsigned)a.feat_rows;
        off = ok ? (int)__umul24((unsigned)gi[i], (unsigned)a.row_bytes) : kOut;
        acc = (int)__umul24((unsigned)(ok ? rl : R), (unsigned)(S::LDW * 4)) + buf;
    };
    auto finish4 = [&](int i, int j, unsigned mask, int tile, int buf, int (&off)[4]) {
        int o, c, ac[4];
        finish(i, ((mask >> j) & bit) != 0, tile, buf, o, c);
        quarters(o, off);
        quarters(c, ac);
#pragma unroll
        for (int u = 0; u < 4; u++) own[j + u] = ac[u] + acc_lane;
    };
    auto finish1 = [&](int j, unsigned mask, int tile, int buf, int &off) {
        int c;
        finish(1, ((mask >> j) & 1) != 0, tile, buf, off, c);
        own[j] = c + acc_lane;
    };
    auto gather = [&](int j, int off) {
#pragma unroll
        for (int st = 0; st < NS; st++)
            fa[j % NF][st] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(r_feat, off + chunk + st * 64, 0, 0));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto tail = [&](int4v x, int st) { // rows shorter than the steps: zeros behind their end
        if constexpr (MASKED) x = st * 64 + chunk < a.row_bytes ? x : int4v{0, 0, 0, 0};
        return x;
    };
    // the indices of the pass after the next: slots 0..4 at once, where those of slots 5..8 are to `at5`
    int at5;
    auto look_ahead = [&](unsigned &mask, bool &last) {
        const int at = pass_groups(mask, last);
        load_idx(0, place(at, 0));
        load_idx(1, __builtin_amdgcn_readlane(at, 4) + slot_lane);
        at5 = place(at, 5);
    };
    auto next_buf = [&](int buf) { return buf == (kRelayStages - 1) * S::kTileBytes ? 0 : buf + S::kTileBytes; };
    {
        look_ahead(mask0, last0);
        load_idx(2, at5);
        tile0 = first;
        buf0 = 0;
        __builtin_amdgcn_sched_barrier(0);
        int off[4], off4;
        finish4(0, 0, mask0, tile0, buf0, off);
        finish1(4, mask0, tile0, buf0, off4);
        advance(last0);
        look_ahead(mask1, last1);
        tile1 = f_tile;
        buf1 = last0 ? next_buf(buf0) : buf0;
        __builtin_amdgcn_sched_barrier(0);
        gather(4, off4);
#pragma unroll
        for (int u = 0; u < 4; u++) gather(u, off[u]);
    }
    int done = 0; // tiles finished
    for (int i = 0; i <= stage; i++) lds_barrier(); // the first tile is there
    for (;;) {
        acc4 d[2][CW]; // sums of the even and the odd slots' groups
#pragma unroll
        for (int c = 0; c < CW; c++) d[0][c] = *(const acc4 *)(s_acc + own[0] + c * 16);
        int off[4], off4, tile2;
        unsigned mask2;
        bool last2;
        finish4(2, 5, mask0, tile0, buf0, off);
        load_idx(2, at5);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            acc4 (&dj)[CW] = d[j & 1];
            if ((mask0 >> j) & 1) {
#pragma unroll
                for (int c = 0; c < CW; c++)
#pragma unroll
                    for (int st = 0; st < NS; st++) dj[c] = mfma_step<DT>(fw[j][st][c], tail(fa[j % NF][st], st), dj[c]);
#pragma unroll
                for (int c = 0; c < CW; c++) *(acc4 *)(s_acc + own[j] + c * 16) = dj[c];
            }
            __builtin_amdgcn_sched_barrier(0);
            // the next group's sums, read behind the write of this one's, which the LDS keeps in order (into registers of their
            // own: after a skipped group the compiler would wait for the reads that are still on their way into these)
            if (j + 1 < NJ) {
#pragma unroll
                for (int c = 0; c < CW; c++) d[(j + 1) & 1][c] = *(const acc4 *)(s_acc + own[j + 1] + c * 16);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (j < 4) {
                gather(j + 5, off[j]);
            } else if (j == 4) {
                finish4(0, 0, mask1, tile1, buf1, off);
                finish1(4, mask1, tile1, buf1, off4);
                advance(last1);
                look_ahead(mask2, last2);
                tile2 = f_tile;
                __builtin_amdgcn_sched_barrier(0);
                gather(4, off4);
            } else {
                gather(j - 5, off[j - 5]);
            }
        }
        if (last0) {
            lds_barrier();
            if (++done == n) break;
        }
        buf0 = buf1;
        if (last1) buf1 = next_buf(buf1);
        mask0 = mask1, last0 = last1, tile0 = tile1;
        mask1 = mask2, last1 = last2, tile1 = tile2;
    }
}

// The wave at both ends of a tile's way.  It gives a tile its first sums: the products of the middle offset's run (RUN: every
// row with itself, its weight fragments stay in registers) or zeros; and when the tile has passed the gathering waves it
// writes it out with the epilogue.  EPI: 0 = the sums as they are, 1 = scale and shift, 2 = and ReLU.
template <sph_dtype DT, int NS, int CT, bool MASKED, bool RUN, int EPI>
__device__ __forceinline__ void relay_ends(const ConvArgs &a, char *s_acc, int half, int lane, int first, int step, int n)
{
    typedef typename Traits<DT>::acc4 acc4;
    typedef typename Traits<DT>::elem elem;
    typedef RelayShape<CT> S;
    constexpr int RH = R / S::NH;                          // rows of a tile that this wave takes: from `half` * RH
    constexpr int NB = RH / SPH_GROUP;
    constexpr int VE = 16 / (int)sizeof(elem);             // columns of a 16-byte store
    constexpr int kRowChunks = CT * 16 / VE;               // stores of a row
    constexpr int kChunks = RH * kRowChunks / kWave;       // a lane's stores of a tile
    constexpr int kBatch = kChunks < 4 ? kChunks : 4;      // in work at a time
    const int KV = a.book.KV, kc = KV / 2;
    const int ntiles = (a.book.rows + R - 1) / R;
    const __amdgpu_buffer_rsrc_t r_feat = __builtin_amdgcn_make_buffer_rsrc((void *)a.feat, 0, a.feat_rows * a.row_bytes, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_w = __builtin_amdgcn_make_buffer_rsrc((void *)a.wp, 0, KV * NS * CT * kWave * 16, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_gat = __builtin_amdgcn_make_buffer_rsrc((void *)a.book.grp_gather, 0, ntiles * a.cap * SPH_GROUP * 4, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_own = __builtin_amdgcn_make_buffer_rsrc((void *)a.book.grp_owner, 0, ntiles * a.cap * SPH_GROUP * 4, kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_ko = __builtin_amdgcn_make_buffer_rsrc((void *)a.book.tile_koff, 0, ntiles * (KV + 1) * 2, kRsrcFlags);
    const int chunk = (lane >> 4) * 16;
    const int tile_last = first + (n - 1) * step;

    int4v fw[NS][CT];
    if constexpr (RUN) relay_weight<NS, CT, CT>(r_w, kc, 0, lane, fw);

    // a lane's columns are the same in all its stores
    const int ch = lane % kRowChunks;
    float sc[VE], sh[VE];
#pragma unroll
    for (int j = 0; j < VE; j++) {
        const int col = min(ch * VE + j, a.ndim - 1);
        sc[j] = a.scale ? a.scale[col] : 1.f;
        sh[j] = (DT != SPH_I8 && a.shift) ? a.shift[col] : 0.f;
    }

    int4v fa[NB][NS];              // rows of the run, in their rows' places, of the tile that begins next
    int gi[RH / kWave], ow[RH / kWave]; // indices of the tile after it,
    bool in_run[RH / kWave];            // and whether the run is that long (what is read behind its end are zeros, not "no row")
    unsigned short x_lo, x_hi;     // groups of the run, the tile after that
    unsigned long long stray[RH / kWave] = {}; // its rows that the run has no pair for in their places, a bit for each
    auto load_ko = [&](int t) {
        const int at = min(t, tile_last) * (KV + 1);
        x_lo = __builtin_amdgcn_raw_buffer_load_b16(r_ko, kc * 2, at * 2, 0);
        x_hi = __builtin_amdgcn_raw_buffer_load_b16(r_ko, kc * 2 + 2, at * 2, 0);
    };
    auto load_idx = [&](int t) { // entry r of the run is row r's, if every row has its pair
#pragma unroll
        for (int h = 0; h < RH / kWave; h++) {
            const int at = x_lo * SPH_GROUP + half * RH + h * kWave + lane;
            in_run[h] = at < x_hi * SPH_GROUP;
            const int off = in_run[h] ? (min(t, tile_last) * a.cap * SPH_GROUP + at) * 4 : kOut;
            gi[h] = __builtin_amdgcn_raw_buffer_load_b32(r_gat, off, 0, 0);
            ow[h] = __builtin_amdgcn_raw_buffer_load_b32(r_own, off, 0, 0);
        }
    };
    // the rows of tile t, and the indices of the two tiles behind it
    auto gather = [&](int t) {
        const int r0 = min(t, tile_last) * R, nrows = min(R, a.book.rows - r0);
        int off[RH / kWave][4];
#pragma unroll
        for (int h = 0; h < RH / kWave; h++) {
            const int row = half * RH + h * kWave + lane;
            const bool here = row < nrows && in_run[h] && ow[h] == r0 + row && (unsigned)gi[h] < (unsigned)a.feat_rows;
            stray[h] = __builtin_amdgcn_ballot_w64(row < nrows && !here);
            quarters(here ? (int)__umul24((unsigned)gi[h], (unsigned)a.row_bytes) : kOut, off[h]);
        }
        load_idx(t + step);
        load_ko(t + 2 * step);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int h = 0; h < RH / kWave; h++)
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int st = 0; st < NS; st++)
                    fa[h * 4 + u][st] = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(r_feat, off[h][u] + chunk + st * 64, 0, 0));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto tail = [&](int4v x, int st) {
        if constexpr (MASKED) x = st * 64 + chunk < a.row_bytes ? x : int4v{0, 0, 0, 0};
        return x;
    };
    auto begin = [&](int t, char *tile) {
        char *p = tile + (half * RH + (lane & 15)) * (S::LDW * 4) + (lane >> 4) * (CT * 16);
        acc4 d[NB][CT];
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int c = 0; c < CT; c++) d[b][c] = acc4{0, 0, 0, 0};
        if constexpr (RUN) {
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int st = 0; st < NS; st++)
#pragma unroll
                    for (int c = 0; c < CT; c++) d[b][c] = mfma_step<DT>(fw[st][c], tail(fa[b][st], st), d[b][c]);
        }
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int c = 0; c < CT; c++) *(acc4 *)(p + b * SPH_GROUP * S::LDW * 4 + c * 16) = d[b][c];
        if constexpr (RUN) {
            unsigned long long any = 0;
#pragma unroll
            for (int h = 0; h < RH / kWave; h++) any |= stray[h];
            if (any) {
                // Rows without their pair start from zero (their products are those of a row of zeros, which is not the same where
                // the weight is not finite), and pairs that are not in their rows' places are added group by group.
#pragma unroll
                for (int h = 0; h < RH / kWave; h++)
                    if ((stray[h] >> lane) & 1)
                        for (int c = 0; c < CT * 4; c++)
                            *(acc4 *)(tile + (half * RH + h * kWave + lane) * (S::LDW * 4) + c * 16) = acc4{0, 0, 0, 0};
                const int r0 = t * R, nrows = min(R, a.book.rows - r0);
                const unsigned short *ko = a.book.tile_koff + (long)t * (KV + 1) + kc;
                const int lo = ko[0], hi = min((int)ko[1], a.cap);
                for (int g = lo; g < hi; g++) {
                    const long slot = ((long)t * a.cap + g) * SPH_GROUP + (lane & 15);
                    const int in = a.book.grp_gather[slot], rl = a.book.grp_owner[slot] - r0;
                    const bool ok = (unsigned)rl < (unsigned)nrows && (unsigned)in < (unsigned)a.feat_rows && rl != (g - lo) * SPH_GROUP + (lane & 15) &&
                                    rl / RH == half;
                    const int off = ok ? (int)__umul24((unsigned)in, (unsigned)a.row_bytes) : kOut;
                    char *q = tile + (ok ? rl : R) * (S::LDW * 4) + (lane >> 4) * (CT * 16);
                    acc4 e[CT];
#pragma unroll
                    for (int c = 0; c < CT; c++) e[c] = *(const acc4 *)(q + c * 16);
#pragma unroll
                    for (int st = 0; st < NS; st++) {
                        const int4v x = __builtin_bit_cast(int4v, __builtin_amdgcn_raw_buffer_load_b128(r_feat, off + chunk + st * 64, 0, 0));
#pragma unroll
                        for (int c = 0; c < CT; c++) e[c] = mfma_step<DT>(fw[st][c], tail(x, st), e[c]);
                    }
#pragma unroll
                    for (int c = 0; c < CT; c++) *(acc4 *)(q + c * 16) = e[c];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            gather(t + step);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // (stores through a descriptor that ends with the tile's last row: none of them is behind a branch, so the compiler
    // knows how many are in flight and the rows of the run do not wait for them)
    const int row_bytes = a.ndim * (int)sizeof(elem);
    const int out_lane = ch * VE < a.ndim ? (half * RH + lane / kRowChunks) * row_bytes + ch * 16 : kOut;
    auto end = [&](int t, const char *tile) {
        const int r0 = t * R, nrows = min(R, a.book.rows - r0);
        const __amdgpu_buffer_rsrc_t r_out = __builtin_amdgcn_make_buffer_rsrc(a.out + (long)r0 * row_bytes, 0, nrows * row_bytes, kRsrcFlags);
        const char *from = tile + (half * RH + lane / kRowChunks) * (S::LDW * 4) + ch * (VE * 4);
#pragma unroll
        for (int i0 = 0; i0 < kChunks; i0 += kBatch) {
            acc4 f[kBatch][VE / 4];
#pragma unroll
            for (int i = 0; i < kBatch; i++)
#pragma unroll
                for (int j = 0; j < VE / 4; j++) f[i][j] = *(const acc4 *)(from + (i0 + i) * (kWave / kRowChunks) * (S::LDW * 4) + j * 16);
#pragma unroll
            for (int i = 0; i < kBatch; i++) {
                union { elem e[VE]; int4v v; } u;
#pragma unroll
                for (int j = 0; j < VE; j++) {
                    float v = (float)f[i][j / 4][j % 4];
                    if constexpr (EPI > 0) v = v * sc[j] + sh[j];
                    if constexpr (EPI > 1) v = v > 0.f ? v : 0.f;
                    u.e[j] = to_elem<DT>(v);
                }
                __builtin_amdgcn_raw_buffer_store_b128(u.v, r_out, out_lane + (i0 + i) * (kWave / kRowChunks) * row_bytes, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (RUN) {
        load_ko(first);
        load_idx(first);
        load_ko(first + step);
        gather(first);
    }
    // n + kRelayStages barriers: the first kRelayStages tiles begin, then one ends and the next takes its place.  (Loops of their
    // own: the compiler counts the loads and stores in flight for every path into a loop.)
    char *tile = s_acc;
    auto next = [&]() {
        tile = tile == s_acc + (kRelayStages - 1) * S::kTileBytes ? s_acc : tile + S::kTileBytes;
        lds_barrier();
    };
    int s = 0;
    for (; s < min(n, kRelayStages); s++) {
        begin(first + s * step, tile);
        next();
    }
    for (; s < kRelayStages; s++) next();
    for (; s < n; s++) {
        end(first + (s - kRelayStages) * step, tile);
        begin(first + s * step, tile);
        next();
    }
    for (; s < n + kRelayStages; s++) {
        end(first + (s - kRelayStages) * step, tile);
        next();
    }
}

// GPC: workgroups a CU holds.
template <sph_dtype DT, int NS, int CT, bool MASKED, bool RUN, int GPC>
__global__ __launch_bounds__(RelayShape<CT>::kThreads) __attribute__((amdgpu_waves_per_eu(GPC * RelayShape<CT>::NH, GPC * RelayShape<CT>::NH)))
void conv_relay_kernel(ConvArgs a, int slots)
{
    extern __shared__ __attribute__((aligned(16))) char s_relay[]; // [kRelayStages][R + 1][LDW] accumulators
    constexpr int NH = RelayShape<CT>::NH;
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int stage = wave / NH, half = wave % NH;
    const int ntiles = (a.book.rows + R - 1) / R;
    const int per_xcd = (ntiles + SPH_NUM_XCD - 1) / SPH_NUM_XCD;
    const int xcd = blockIdx.x % SPH_NUM_XCD, slot = blockIdx.x / SPH_NUM_XCD;
    const int first = xcd * per_xcd + slot, end = min((xcd + 1) * per_xcd, ntiles);
    if (first >= end) return; // the whole workgroup
    const int n = (end - first + slots - 1) / slots;
    // Every wave meets n + kRelayStages barriers: a tile's first sums are there behind the first, stage w takes it behind
    // w more, and behind kRelayStages it is written out.
    if (stage == kRelayStages - 1) {
        if (DT != SPH_I8 && !a.scale && !a.shift && !a.relu) relay_ends<DT, NS, CT, MASKED, RUN, 0>(a, s_relay, half, lane, first, slots, n);
        else if (DT == SPH_I8 || !a.relu) relay_ends<DT, NS, CT, MASKED, RUN, 1>(a, s_relay, half, lane, first, slots, n);
        else relay_ends<DT, NS, CT, MASKED, RUN, 2>(a, s_relay, half, lane, first, slots, n);
    } else {
        relay_gather<DT, NS, CT, MASKED, RUN>(a, s_relay, stage, half, lane, first, slots, n);
        for (int i = stage + 1; i < kRelayStages; i++) lds_barrier();
    }
}

template <sph_dtype DT, int NS, int CT, bool MASKED, bool RUN, int GPC>
int relay_launch(const ConvArgs &a, int ntiles, hipStream_t st)
{
    const size_t lds = kRelayStages * RelayShape<CT>::kTileBytes;
    auto kernel = conv_relay_kernel<DT, NS, CT, MASKED, RUN, GPC>;
    hipError_t e = hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) {
        sph_set_error("hipFuncSetAttribute(%zu bytes of LDS): %s", lds, hipGetErrorString(e));
        return SPH_ERR_LAUNCH;
    }
    const int per_xcd = sph_div_up(ntiles, SPH_NUM_XCD), room = 32 * GPC;
    const int slots = per_xcd < room ? per_xcd : room;
    hipLaunchKernelGGL(kernel, dim3(slots * SPH_NUM_XCD), dim3(RelayShape<CT>::kThreads), lds, st, a, slots);
    return sph_check_launch("sph_conv_apply");
}

template <sph_dtype DT, int NS, int CT, int GPC>
int relay_launch_m(const ConvArgs &a, int ntiles, hipStream_t st)
{
    const bool masked = a.row_bytes < NS * 64;
    if (book_has_run(&a.book))
        return masked ? relay_launch<DT, NS, CT, true, true, GPC>(a, ntiles, st) : relay_launch<DT, NS, CT, false, true, GPC>(a, ntiles, st);
    return masked ? relay_launch<DT, NS, CT, true, false, GPC>(a, ntiles, st) : relay_launch<DT, NS, CT, false, false, GPC>(a, ntiles, st);
}

} // namespace

// Tiles above which the relay is the faster one (a tile takes five steps, so a short grid is all start and end), in a call on its
// own and with three scans in flight, where the kernels of conv.hip fill one another's ends and the relay, which takes whole
// compute units, keeps the others out.  us of rules + convolution, conv.hip : relay, alone and in flight, scans of 1.5 to 2 pairs a row:
//   64 -> 64 fp16   1065 tiles 38.1 : 33.1, 23.1 : 24.0   1207 tiles 42.0 : 33.8, 26.7 : 26.4   2003 tiles 57.2 : 45.0, 47.5 : 38.3
//   32 -> 64 fp16   1065 tiles 29.4 : 27.1, 14.7 : 17.9   1804 tiles 37.2 : 36.1, 28.5 : 27.9   2205 tiles 44.8 : 40.5, 34.4 : 32.8
//   64 -> 64 int8   1065 tiles 30.7 : 28.9, 16.1 : 19.1   1804 tiles 39.0 : 36.3, 28.0 : 28.7   2205 tiles 47.1 : 40.9, 35.2 : 33.6
//   32 -> 32 fp32   1207 tiles 37.8 : 41.1, 27.0 : 31.8   1355 tiles 50.7 : 44.7, 29.6 : 34.3   2205 tiles 64.0 : 54.8, 47.7 : 47.2
//   32 -> 64 fp32   1065 tiles 63.8 : 51.8, 39.4 : 39.4   1207 tiles 76.2 : 52.7, 44.0 : 42.5   2205 tiles 106  : 76.9, 80.0 : 67.4
//   32 -> 32 fp16   2205 tiles 35.1 : 29.8, 25.7 : 24.0
//   16 -> 32 fp32   2205 tiles 44.4 : 39.9, 31.8 : 33.3   2609 tiles 50.0 : 45.5, 37.5 : 37.9   3212 tiles 59.8 : 51.9, 47.3 : 45.1
//   16 -> 16 fp16   2205 tiles 23.6 : 24.9, 15.1 : 16.4   3212 tiles 32.8 : 32.2, 25.3 : 24.2   4215 tiles 42.7 : 38.5, 33.9 : 30.5
//    4 -> 16 fp32   3212 tiles 36.4 : 39.3, 27.2 : 29.8   4215 tiles 47.0 : 46.5, 36.5 : 37.1   6013 tiles 64.8 : 60.8, 54.6 : 50.5
// Kernels of up to nine offsets stay with conv.hip: their weight is a third and a tile's groups meet three stages unevenly (3x3x1 64 -> 64 of
// stride 2 on 5029 tiles 62.4 : 51.4, submanifold on 4871 tiles 49.5 : 58.3).
static int relay_line(sph_dtype dt, int nsteps, int nwtot, bool in_flight)
{
    const int fragments = nsteps * nwtot; // of one offset: what the relay keeps in registers and the others load with every group
    if (fragments == 1) return 3584;
    if (fragments == 2) return in_flight ? 2560 : 2048;
    if (!in_flight) return dt == SPH_F32 && nwtot == 2 ? 1280 : 1024;
    if (dt == SPH_F32 && nwtot == 4) return 1152;
    return fragments == 8 ? 1280 : 1920;
}

bool sph_relay_ok(sph_dtype dt, const ConvArgs &a, int nwtot, int ntiles)
{
    const int KV = a.book.KV;
    if (!a.aligned_in || !a.aligned_out || a.nsteps > 2 || nwtot > 4) return false;
    if (KV <= kRelayPart || KV > (kRelayStages - 1) * kRelayPart) return false;
    if ((double)ntiles * a.cap * SPH_GROUP * 4 >= 2147483648.0) return false; // 32-bit offsets into the book
    return ntiles > relay_line(dt, a.nsteps, nwtot, book_says(&a.book) == SPH_RUN_IN_FLIGHT);
}

int sph_relay_launch(sph_dtype dt, const ConvArgs &a, int nwtot, int ntiles, hipStream_t st)
{
#define SPH_RELAY(DT, NS, CT, OCC) if (dt == DT && a.nsteps == NS && nwtot == CT) return relay_launch_m<DT, NS, CT, OCC>(a, ntiles, st);
#define SPH_RELAY_TYPE(DT) \
    SPH_RELAY(DT, 2, 4, 1) SPH_RELAY(DT, 1, 4, 1) SPH_RELAY(DT, 2, 2, 2) SPH_RELAY(DT, 1, 2, 2) SPH_RELAY(DT, 2, 1, 3) SPH_RELAY(DT, 1, 1, 3)
    SPH_RELAY_TYPE(SPH_F32) SPH_RELAY_TYPE(SPH_F16) SPH_RELAY_TYPE(SPH_BF16) SPH_RELAY_TYPE(SPH_I8)
    sph_set_error("sph_conv_apply: no such form");
    return SPH_ERR_UNSUPPORTED;
}
