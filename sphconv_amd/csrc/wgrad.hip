// Weight gradient for gfx950 (sph_conv_wgrad): sums of outer products over a rule book's pairs.
#include "common.h"
#include "pack.h"
#include "conv_wave.h"

#include <utility>

namespace {

struct WgradArgs {
    const char *feat;
    int in_rows, iC;
    const char *dout;
    int out_rows, oC;
    sph_book book;
    const int32_t *list_in, *list_out; // the book's two lists: input rows and output rows of the groups
    int cap, ntiles, nchunk;
    float *partial;
    int *flags;      // wave kernel: one per partial slot, 1 = the slot was written
    int nslice;      // stage kernel: workgroups per chunk at the centre offset (slices h, h + nslice, ... each)
    int all_slices;  // stage kernel: every offset has its later slices' workgroups (small grids), not only the centre
    int chunk_tiles; // wave kernel: tiles of a chunk
    int nparts;      // wave kernel: workgroups that share a chunk's groups at the centre offset
};

constexpr int kWgThreads = 256;
constexpr int kWgWaves = kWgThreads / kWave;
constexpr int kMaxTilesPerWave = 16; // (128/16)^2 / 4 waves

template <sph_dtype DT>
__global__ __launch_bounds__(kWgThreads) void wgrad_kernel(WgradArgs a)
{
    typedef typename Traits<DT>::elem elem;
    constexpr int KW = Traits<DT>::KW;
    constexpr int PB = 4 * KW;            // pairs per batch = K of one super step
    constexpr int LDP = PB + 16 / (int)sizeof(elem); // padded pair stride, keeps 16-byte alignment
    extern __shared__ char s_raw[];
    const int iCp = (a.iC + 15) & ~15, oCp = (a.oC + 15) & ~15;
    elem *At = (elem *)s_raw;               // [iCp][LDP]
    elem *Gt = At + (long)iCp * LDP;        // [oCp][LDP]
    __shared__ int s_in[PB], s_out[PB];

    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int KV = a.book.KV;
    const int k = blockIdx.x / a.nchunk, chunk = blockIdx.x - k * a.nchunk;
    const int tpc = (a.ntiles + a.nchunk - 1) / a.nchunk;
    const int t0 = chunk * tpc, t1 = min(t0 + tpc, a.ntiles);
    const int MI = iCp / 16, NI = oCp / 16, MT = MI * NI;

    float4v acc[kMaxTilesPerWave];
#pragma unroll
    for (int j = 0; j < kMaxTilesPerWave; j++) acc[j] = float4v{0, 0, 0, 0};

    for (int t = t0; t < t1; t++) {
        const int g0 = a.book.tile_koff[(long)t * (KV + 1) + k];
        const int g1 = a.book.tile_koff[(long)t * (KV + 1) + k + 1];
        for (int gb = g0; gb < g1; gb += PB / SPH_GROUP) {
            __syncthreads(); // previous batch fully consumed
            if (tid < PB) {
                int g = gb + tid / SPH_GROUP;
                int vi = -1, vo = -1;
                if (g < g1) {
                    long slot = ((long)t * a.cap + g) * SPH_GROUP + (tid & (SPH_GROUP - 1));
                    vi = a.list_in[slot];
                    vo = a.list_out[slot];
                }
                if ((unsigned)vi >= (unsigned)a.in_rows || (unsigned)vo >= (unsigned)a.out_rows) vi = vo = -1;
                s_in[tid] = vi;
                s_out[tid] = vo;
            }
            __syncthreads();
            for (int e = tid; e < PB * iCp; e += kWgThreads) {
                int p = e / iCp, c = e - p * iCp;
                int row = s_in[p];
                elem v = (elem)0;
                if (row >= 0 && c < a.iC) v = ((const elem *)a.feat)[(long)row * a.iC + c];
                At[c * LDP + p] = v;
            }
            for (int e = tid; e < PB * oCp; e += kWgThreads) {
                int p = e / oCp, c = e - p * oCp;
                int row = s_out[p];
                elem v = (elem)0;
                if (row >= 0 && c < a.oC) v = ((const elem *)a.dout)[(long)row * a.oC + c];
                Gt[c * LDP + p] = v;
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < kMaxTilesPerWave; j++) {
                int ti = wave + j * kWgWaves;
                if (ti < MT) {
                    int mi = ti / NI, ni = ti - mi * NI;
                    int4v fa = *(const int4v *)(At + (mi * 16 + (lane & 15)) * LDP + (lane >> 4) * KW);
                    int4v fb = *(const int4v *)(Gt + (ni * 16 + (lane & 15)) * LDP + (lane >> 4) * KW);
                    acc[j] = mfma_step<DT>(fa, fb, acc[j]);
                }
            }
        }
    }
    float *part = a.partial + ((long)k * a.nchunk + chunk) * a.iC * a.oC;
#pragma unroll
    for (int j = 0; j < kMaxTilesPerWave; j++) {
        int ti = wave + j * kWgWaves;
        if (ti < MT) {
            int mi = ti / NI, ni = ti - mi * NI;
            int co = ni * 16 + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                int ci = mi * 16 + (lane >> 4) * 4 + r;
                if (ci < a.iC && co < a.oC) part[(long)ci * a.oC + co] = acc[j][r];
            }
        }
    }
}

template <typename OUT>
__global__ void wgrad_reduce_kernel(const float *partial, int KV, int nchunk, int per_k, OUT *dw)
{
    long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (long)KV * per_k) return;
    int k = (int)(i / per_k), e = (int)(i - (long)k * per_k);
    const float *p = partial + (long)k * nchunk * per_k + e;
    float s = 0.f;
    for (int c = 0; c < nchunk; c++) s += p[(long)c * per_k];
    dw[i] = (OUT)s;
}

// ---------------------------------------------------------------------------
constexpr int kWsBlock = 64;   // channels per block side

// Narrow layers of 16 bits (blocks of up to four tiles; of eight on books of up to four tiles of rows): through LDS.  A row is two to four lanes' loads of 16 bytes here; turning it
// in registers, as wgrad_wave_kernel does, takes pieces of 4 or 8 bytes, as many loads as a row of 64 channels (16->16 on 14 599
// tiles 66 us here, 116 there; 32->32 118 : 130; 64->16 on 2 437 tiles 32 : 34; 24->40 the other way round, 173 : 137).
// Work item = (offset k, chunk of 64 tiles, slice of 64 groups of that chunk's groups at
// k, 64x64 block of [iC,oC]).  A chunk holds at most 64*8 groups per offset.  Slicing by groups,
// not tiles, is what balances the grid: a submanifold book has 8 groups per tile at the centre
// offset and about one elsewhere.  nslice workgroups (8 or 4) share the centre offset, workgroup h
// takes slices h, h + nslice, ..., and one takes the whole of every other offset; on small grids
// (all_slices) every offset has nslice.  A workgroup whose first slice lies beyond the chunk's real
// group count exits at once.
// The four waves of the workgroup take the slice's batches (32 pairs) round
// robin and never synchronise until the end: a wave gathers the batch's feature rows and
// d_out rows with 16-byte loads into its own LDS area in natural [pair][channel] order,
// and reads MFMA operands with the pair index as the K dimension through transposing
// LDS reads.  The block lives in registers;
// the workgroup's four blocks are summed through LDS into one fp32 partial, and
// wgrad_slot_reduce_kernel adds the written slots in a fixed order.
// ---------------------------------------------------------------------------
constexpr int kWsTiles = 64;   // tiles per chunk (one lane each)
constexpr int kWsSlice = 64;   // groups per slice
constexpr int kWsSlices = 8;   // most workgroups per chunk at the centre offset (workgroup h takes slices h, h + nslice, ...);
                               // WgradArgs::nslice = 8 on books of up to 16 chunks, 4 on larger ones

typedef short short4v __attribute__((ext_vector_type(4)));

// MFMA operand of 16 channels x one batch of pairs from a staging area laid out
// [pair][channel], row stride rs bytes: lane (m = lane%16, q = lane/16)
// receives pairs 8q..8q+7 of channel m through two transposing reads (element j of lane
// 4a+b = the b-th element at the address given by lane a+4j of the same 16 lanes).
__device__ __forceinline__ int wgrad_frag_offset(int rs, int lane)
{
    const int s = lane & 15, q = lane >> 4;
    return (8 * q + (s >> 2)) * rs + 4 * (s & 3) * 2;
}
__device__ __forceinline__ int4v wgrad_frag(const char *p, int rs)
{
    typedef __attribute__((address_space(3))) short4v lds_s4;
    short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)p);
    short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)(p + 4 * rs));
    union { struct { short4v l, h; } s; int4v v; } u;
    u.s.l = lo; u.s.h = hi;
    return u.v;
}

template <sph_dtype DT, int MI, int NI>
__global__ __launch_bounds__(256, 2) void wgrad_stage_kernel(WgradArgs a)
{
    typedef typename Traits<DT>::elem elem;
    constexpr int E = (int)sizeof(elem);
    static_assert(E == 2, "16-bit types");
    constexpr int GPB = 2;                             // groups per batch: one MFMA super step of 32 pairs
    constexpr int PB = GPB * SPH_GROUP;                // pairs per batch
    // MI, NI: 16-channel tiles of the block's two sides (1, 2 or 4, up to 8 together; narrower blocks are zero padded).
    // A batch of rows of MI tiles is MI 16-byte loads per lane.
    extern __shared__ __attribute__((aligned(16))) char s_raw[];

    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int KV = a.book.KV;
    // Work items u = chunk*KV + k are dealt to the XCDs in contiguous runs (workgroups go to
    // the XCDs round robin): the offsets of one chunk gather the same ~2 MiB of rows, which
    // then stay in that XCD's L2.  The slice index is slowest, so that the first slices --
    // often the only ones with work -- spread over all XCDs and start first.
    const int items = KV * a.nchunk, items_grid = (items + SPH_NUM_XCD - 1) / SPH_NUM_XCD * SPH_NUM_XCD;
    int h, chunk, k;
    if ((int)blockIdx.x < items_grid) {
        h = 0;
        const int u = sph_xcd_tile(blockIdx.x, items);
        if (u >= items) return;
        chunk = u / KV;
        k = u - chunk * KV;
    } else {
        // Later slices: a submanifold book has 8 groups per tile at the centre offset and about one elsewhere, and
        // a workgroup without work still costs its dispatch (three quarters of the grid found none when every offset
        // had four).  So only the centre offset has them, numbered first, and at the other offsets the first
        // workgroup takes every slice -- unless the grid is small (all_slices): then a dense book's offsets need
        // their four workgroups each to fill the chip, and they follow the centre's.
        const int kc = KV / 2, v = (int)blockIdx.x - items_grid, nc = (a.nslice - 1) * a.nchunk;
        if (v < nc) {
            h = 1 + v / a.nchunk;
            chunk = v % a.nchunk;
            k = kc;
        } else {
            const int r = v - nc, per = a.nchunk * (KV - 1);
            if (!a.all_slices || KV == 1 || r >= (a.nslice - 1) * per) return;
            h = 1 + r / per;
            const int q = r % per, kk = q % (KV - 1);
            chunk = q / (KV - 1);
            k = kk + (kk >= kc ? 1 : 0);
        }
    }
    const int slice_step = (a.all_slices || k == KV / 2) ? a.nslice : 1;
    const int sbn = (a.oC + kWsBlock - 1) / kWsBlock;
    const int ci0 = (blockIdx.y / sbn) * kWsBlock, co0 = (blockIdx.y % sbn) * kWsBlock;
    const int cA = min(kWsBlock, a.iC - ci0), cG = min(kWsBlock, a.oC - co0);
    const int slot = (k * a.nchunk + chunk) * a.nslice + h;

    // groups of this offset in the chunk's tiles: lane = tile, prefix sums over the wave
    const int t0 = chunk * kWsTiles;
    int g0 = 0, n = 0;
    if (t0 + lane < a.ntiles) {
        const unsigned short *ko = a.book.tile_koff + (long)(t0 + lane) * (KV + 1) + k;
        g0 = min((int)ko[0], a.cap);
        n = min(max((int)ko[1] - g0, 0), min(a.cap - g0, R / SPH_GROUP));
    }
    const int incl = wave_inclusive_sum(n); // lane shifts of the vector ALU, no LDS round trip per step
    const int total = __builtin_amdgcn_readlane(incl, kWave - 1);
    if (slice_step == 1 && tid < a.nslice - 1 && blockIdx.y == 0) a.flags[slot + 1 + tid] = 0; // slots nobody fills
    if (h * kWsSlice >= total) {
        if (tid == 0 && blockIdx.y == 0) a.flags[slot] = 0;
        return;
    }

    // wave-private staging: feature rows then d_out rows, [pair][channels + 16 bytes]
    constexpr int rsA = MI * 16 * E + 16, rsG = NI * 16 * E + 16;
    const int cprA = cA * E / 16, cprG = cG * E / 16;      // real 16-byte chunks per row
    char *xa = s_raw + (size_t)wave * PB * (rsA + rsG);
    char *xg = xa + PB * rsA;
    for (int i = lane; i < PB * (rsA + rsG) / 16; i += kWave) ((int4v *)xa)[i] = int4v{0, 0, 0, 0};

    float4v acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++) acc[i][j] = float4v{0, 0, 0, 0};

    // Per-lane constants of the row copies: which pair and 16-byte chunk each of the lane's
    // loads moves, its offset in the source row and in the staging area (-1: none).
    int pairA[MI], srcA[MI], dstA[MI], pairG[NI], srcG[NI], dstG[NI];
    // (rows of 32, 64 or 128 bytes are 2, 4 or 8 chunks: a shift instead of the forty instructions of a division)
    const bool p2A = (cprA & (cprA - 1)) == 0, p2G = (cprG & (cprG - 1)) == 0;
    const int shA = __ffs(cprA) - 1, shG = __ffs(cprG) - 1;
#pragma unroll
    for (int it = 0; it < MI; it++) {
        const int i = it * kWave + lane;
        const int pa = p2A ? i >> shA : i / cprA, ca = i - pa * cprA;
        pairA[it] = min(pa, PB - 1); srcA[it] = ci0 * E + ca * 16; dstA[it] = pa < PB ? pa * rsA + ca * 16 : -1;
    }
#pragma unroll
    for (int it = 0; it < NI; it++) {
        const int i = it * kWave + lane;
        const int pg = p2G ? i >> shG : i / cprG, cg = i - pg * cprG;
        pairG[it] = min(pg, PB - 1); srcG[it] = co0 * E + cg * 16; dstG[it] = pg < PB ? pg * rsG + cg * 16 : -1;
    }
    const unsigned strideA = a.iC * E, strideG = a.oC * E;   // arrays are below 4 GiB (checked by the launcher)

    // Book slot of every group of a slice: lane l looks up flattened group s0+l (the tile
    // whose prefix range holds it, by binary search over the tile lanes) once per slice.
    const long slot_max = (long)a.ntiles * a.cap * SPH_GROUP - 1;
    auto slot_bases = [&](int s0) -> int {
        const int f = s0 + lane;
        int lo = 0;
#pragma unroll
        for (int step = kWave / 2; step >= 1; step >>= 1) {
            const int v = __shfl(incl, lo + step - 1, kWave);
            if (v <= f) lo += step;
        }
        lo = min(lo, kWave - 1);
        const int g = __shfl(g0, lo, kWave) + f - (__shfl(incl, lo, kWave) - __shfl(n, lo, kWave));
        const long sl = ((long)(t0 + lo) * a.cap + g) * SPH_GROUP;
        return (int)min(max(sl, 0L), slot_max - (SPH_GROUP - 1));   // ntiles*cap*16 fits 31 bits (checked by the launcher)
    };
    // Book entries of batch b of the slice: lane l < 32 loads the gathered (input) row of pair
    // l%PB, lane 32+l its owner (output) row.  The load is unconditional; the value is only
    // looked at once all of the wave's index loads are on their way.
    auto load_idx = [&](int bases, int s0, int s1, int b, bool &valid) -> int {
        const int pr = lane & (PB - 1);
        const int fl = GPB * b + (pr >> 4);                 // group within the slice
        valid = s0 + fl < s1;
        const int base = __shfl(bases, fl & (kWave - 1), kWave);
        return (lane < 32 ? a.list_in : a.list_out)[base + (pr & 15)];
    };
    // Row loads are unconditional (clamped to row 0; in_rows and out_rows are positive here)
    // so that several batches stay in flight; slots without a pair are zeroed when the rows
    // are staged.  Returns the mask of pairs that exist.
    auto gather = [&](int idx, int4v (&ra)[MI], int4v (&rg)[NI]) -> unsigned {
        // all lane exchanges first, then all loads: one wait on the LDS queue instead of one per row
        const int other = __shfl_xor(idx, 32, kWave);
        int rowA[MI], rowG[NI];
#pragma unroll
        for (int it = 0; it < MI; it++) rowA[it] = __shfl(idx, pairA[it], kWave);
#pragma unroll
        for (int it = 0; it < NI; it++) rowG[it] = __shfl(idx, 32 + pairG[it], kWave);
        __builtin_amdgcn_sched_barrier(0);
        const unsigned ok = (unsigned)__ballot(idx >= 0 && other >= 0);
#pragma unroll
        for (int it = 0; it < MI; it++)
            ra[it] = *(const int4v *)(a.feat + ((unsigned)max(rowA[it], 0) * strideA + (unsigned)srcA[it]));
#pragma unroll
        for (int it = 0; it < NI; it++)
            rg[it] = *(const int4v *)(a.dout + ((unsigned)max(rowG[it], 0) * strideG + (unsigned)srcG[it]));
        return ok;
    };
    auto stage = [&](unsigned ok, const int4v (&ra)[MI], const int4v (&rg)[NI]) {
#pragma unroll
        for (int it = 0; it < MI; it++)
            if (dstA[it] >= 0) *(int4v *)(xa + dstA[it]) = ((ok >> pairA[it]) & 1) ? ra[it] : int4v{0, 0, 0, 0};
#pragma unroll
        for (int it = 0; it < NI; it++)
            if (dstG[it] >= 0) *(int4v *)(xg + dstG[it]) = ((ok >> pairG[it]) & 1) ? rg[it] : int4v{0, 0, 0, 0};
    };
    const char *fragA = xa + wgrad_frag_offset(rsA, lane), *fragG = xg + wgrad_frag_offset(rsG, lane);
    auto multiply = [&]() {
        int4v fa[MI], fb[NI];
#pragma unroll
        for (int i = 0; i < MI; i++) fa[i] = wgrad_frag(fragA + i * 16 * E, rsA);
#pragma unroll
        for (int i = 0; i < NI; i++) fb[i] = wgrad_frag(fragG + i * 16 * E, rsG);
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++) acc[i][j] = mfma_step<DT>(fa[i], fb[j], acc[i][j]);
    };

    // Per slice, this wave owns batches wave, wave+4, ... (at most NB).  All their index
    // entries are requested at once; then the rows run DEPTH-1 batches ahead of their
    // staging through DEPTH register sets, and staging runs one batch ahead of the MFMAs.
    // The single staging area is safe because LDS operations of a wave execute in order.
    constexpr int NB = kWsSlice / GPB / 4;
    constexpr int DEPTH = 3;
    for (int s0 = h * kWsSlice; s0 < total; s0 += slice_step * kWsSlice) {
        const int s1 = min(total, s0 + kWsSlice);
        const int nbatch = (s1 - s0 + GPB - 1) / GPB;
        const int bases = slot_bases(s0);
        int idx[NB];
        bool valid[NB];
#pragma unroll
        for (int j = 0; j < NB; j++) idx[j] = load_idx(bases, s0, s1, wave + 4 * j, valid[j]);
#pragma unroll
        for (int j = 0; j < NB; j++)
            idx[j] = (valid[j] && (unsigned)idx[j] < (unsigned)(lane < 32 ? a.in_rows : a.out_rows)) ? idx[j] : -1;
        int4v ra[DEPTH][MI], rg[DEPTH][NI];
        unsigned ok[DEPTH];
#pragma unroll
        for (int j = 0; j < DEPTH - 1; j++)
            if (j < NB) ok[j] = gather(idx[j], ra[j], rg[j]);
#pragma unroll
        for (int j = 0; j < NB; j++) {
            if (wave + 4 * j < nbatch) {     // wave-uniform
                if (j + DEPTH - 1 < NB)
                    ok[(j + DEPTH - 1) % DEPTH] = gather(idx[j + DEPTH - 1], ra[(j + DEPTH - 1) % DEPTH], rg[(j + DEPTH - 1) % DEPTH]);
                if (j > 0) multiply();      // batch j-1, from LDS
                asm volatile("" ::: "memory");    // keep the staging writes behind the transposing reads
                stage(ok[j % DEPTH], ra[j % DEPTH], rg[j % DEPTH]);
                asm volatile("" ::: "memory");
            }
        }
        if (wave < nbatch) multiply();      // the last staged batch
    }

    // Sum the four waves' blocks through LDS (over the staging areas), pairwise: (0+2, 1+3),
    // then (0+1).  The partial is stored in accumulator order -- tile (i,j), lane, 4 values:
    // element [16i + 4(lane/16) + r][16j + lane%16] -- as 16-byte stores; the reduction kernel
    // puts it back in [iC,oC] order.
    float4v *red = (float4v *)s_raw;
    constexpr int BLK = MI * NI * kWave;   // float4 per block
    __syncthreads();
    if (wave >= 2) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++) red[(wave - 2) * BLK + (i * NI + j) * kWave + lane] = acc[i][j];
    }
    __syncthreads();
    if (wave < 2) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++) acc[i][j] += red[wave * BLK + (i * NI + j) * kWave + lane];
    }
    __syncthreads();
    if (wave == 1) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++) red[(i * NI + j) * kWave + lane] = acc[i][j];
    }
    __syncthreads();
    if (wave == 0) {
        float4v *part = (float4v *)(a.partial + ((long)slot * gridDim.y + blockIdx.y) * (kWsBlock * kWsBlock));
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++) part[(i * NI + j) * kWave + lane] = acc[i][j] + red[(i * NI + j) * kWave + lane];
        if (lane == 0 && blockIdx.y == 0) a.flags[slot] = 1;
    }
}

// ---------------------------------------------------------------------------
// wgrad, fast path (rows are whole 16-byte chunks).
//
// Work item = (offset k, chunk of up to 192 tiles, part of that chunk's groups at k, 64x64 block of [iC,oC]).  A submanifold
// book has eight groups a tile at the centre offset and about one at the others, so eight workgroups share the centre's; where no offset
// stands out each has one.  The grid is one round of workgroups of about the same number of groups (on long books whole rounds), and
// each ends with one partial block.
// The workgroup's four waves take its batches (64 pairs; 16 for fp32) round robin and never synchronise until the end.
// The contraction runs over pairs and memory has channels side by side, so both operands have to be turned; a wave does that
// in its registers.  fp32: lane (m = lane % 16, q = lane / 16) loads channels MI m .. MI m + MI - 1 of pair 4 s + q for the
// s-th MFMA, and the loaded words are the operands as they are: row m of tile i is channel MI m + i.  16 bits: lane
// (c = lane % 8, half, q) loads channels 2 MI c .. of eight pairs, 16 bytes at 64 channels; lanes eight apart exchange halves
// (one DPP move a word) and a byte permutation per two pairs then makes a tile's operand.
// Slots without a pair read zeros from out of the array's range.  The block lives in registers;
// the workgroup's four blocks are summed through LDS into one fp32 partial, and
// wgrad_slot_reduce_kernel adds the written slots in a fixed order.
//
// What bounds it: a 16-bit batch costs a compute unit 16 loads' addresses (16 cycles each), 32 matrix instructions of 16 cycles on
// one of four SIMDs, and some 150 vector instructions for the exchange and the addresses; the rows come from L2 (2.3 times
// each at fourteen pairs to a row).  Through LDS, as wgrad_stage_kernel below 64 channels, a row was written, read back and waited for
// on top: 64x64 f16 on eight 64x512x32 scans (2 412 tiles) 42 -> 29 us and the sum of the partials 7.7 -> 6.0, fewer of them; 64x64 fp32
// on the strided layer of eight 64x512x512 scans 61 -> 40; 24->40 bf16 on eight ragged grids 38 -> 27 (45 and 31 with
// workgroups kept for a centre that these books have not).
// Loads stand between the matrix instructions: in one burst all waves of the chip ask at the same time and then all wait
// (43 : 33 us).  A wave that has no batch left leaves the unrolled pipeline instead of skipping its stages: behind a skipped
// load the compiler cannot tell how many are on their way and waits for all of them.
//
// The book is the layer's forward one or its transposed one (list_in, list_out): a strided layer on scattered voxels has
// its pairs in 3.1 times fewer tiles stationary on the input rows, with groups more than twice as full (64->64 fp32 on
// eight 64x512x512 scans, stride 2, with the kernel through LDS: 117 us from the forward book, 59 us from the transposed one with the
// empty fours left out; 24->40 bf16: 52 -> 38 us).
//
// Where the kernel through LDS was the faster one still: long books of nearly full grids with 32 channels on a side in 16 bits, whose offsets
// all have seven groups a tile and whose centre's workgroups have an eighth of the others' work (9002 tiles of 24 pairs a row, 32->64 f16
// 403 : 476 us; of 11 pairs a row 242 : 253, of 3.7 128 : 104).  A book does not say how full its grid is before its groups are counted on the GPU.
// ---------------------------------------------------------------------------
constexpr int kWsMost = 192, kWsMostLight = 128; // most tiles of a chunk, and where a compute unit holds more than two workgroups
constexpr int kWsPer = 4;      // most of a lane (even)
constexpr int kWsParts = 8;    // most workgroups that share a chunk's groups at the centre offset
static_assert(kWsMost <= kWsPer * kWave, "a chunk's tiles fit the lanes");
constexpr int kWsLeast = 24;   // groups of a centre offset's share: six for every wave

// f(0), f(1), ... until one says no
template <class F, int... J> __device__ __forceinline__ void each_while(F &&f, std::integer_sequence<int, J...>)
{
    (void)(f(std::integral_constant<int, J>()) && ...);
}

// a lane's channels of one pair, in 32-bit words
template <int WORDS> struct WgRow {
    uint32_t w[WORDS];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, unsigned off)
    {
        if constexpr (WORDS == 1) w[0] = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
        else if constexpr (WORDS == 2) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
            w[0] = v[0]; w[1] = v[1];
        } else {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
            w[0] = v[0]; w[1] = v[1]; w[2] = v[2]; w[3] = v[3];
        }
    }
};

// x = [x0 | x1], y = [y0 | y1], the halves of every sixteen lanes -> x = [x0 | y0], y = [x1 | y1]
__device__ __forceinline__ void swap_eights(uint32_t &x, uint32_t &y)
{
    const int u = __builtin_amdgcn_update_dpp((int)x, (int)y, 0x128, 0xf, 0xc, false); // row_ror:8 into lanes 8 to 15
    const int v = __builtin_amdgcn_update_dpp((int)y, (int)x, 0x128, 0xf, 0x3, false); // and into lanes 0 to 7
    x = (uint32_t)u;
    y = (uint32_t)v;
}

// BIG: arrays of 2^24 rows or more (a row's offset is then a 32-bit product, which takes four times a 24-bit one's time).
template <sph_dtype DT, int MI, int NI, bool BIG>
__global__ __launch_bounds__(256, 2) void wgrad_wave_kernel(WgradArgs a)
{
    typedef typename Traits<DT>::elem elem;
    constexpr int E = (int)sizeof(elem);
    constexpr bool HALF = E == 2;
    constexpr int GPB = HALF ? 4 : 1;                  // groups per batch: two MFMA steps of 32 pairs, or four of 4
    constexpr int SLICE = HALF ? 64 : 48;              // groups whose entries are asked for together
    constexpr int NB = SLICE / GPB / 4, DEPTH = HALF ? 2 : 3;
    static_assert(NB % DEPTH == 0, "the ring must divide a slice");
    constexpr int PL = HALF ? 8 : 4;                   // loads of a lane for a batch's rows of one side
    // MI, NI: 16-channel tiles of the block's two sides (1, 2 or 4, 16 bits 2 or 4; narrower blocks are padded).
    extern __shared__ __attribute__((aligned(16))) char s_raw[];

    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int KV = a.book.KV;
    // Work items u = chunk * (KV - 1 + nparts) + (offset, or a further part of the centre's) are dealt to the XCDs in contiguous
    // runs (workgroups go to the XCDs round robin): the offsets of a chunk walk through the same rows at about the same pace, which
    // then come from that XCD's L2.
    const int per_chunk = KV - 1 + a.nparts, items = per_chunk * a.nchunk;
    const int u = sph_xcd_tile(blockIdx.x, items);
    if (u >= items) return;
    const int chunk = u / per_chunk, idx_in = u - chunk * per_chunk;
    const int k = idx_in < KV ? idx_in : KV / 2, h = idx_in < KV ? 0 : idx_in - KV + 1;
    const int sbn = (a.oC + kWsBlock - 1) / kWsBlock;
    const int ci0 = (blockIdx.y / sbn) * kWsBlock, co0 = (blockIdx.y % sbn) * kWsBlock;
    const int cA = min(kWsBlock, a.iC - ci0), cG = min(kWsBlock, a.oC - co0);
    const int slot = (k * a.nchunk + chunk) * a.nparts + h;

    // groups of this offset in the chunk's tiles: a lane has `per` neighbouring tiles, prefix sums over the wave
    const int t0 = chunk * a.chunk_tiles, t1 = min(t0 + a.chunk_tiles, a.ntiles), per = (a.chunk_tiles + kWave - 1) / kWave;
    // (kept in the wave's own part of LDS: a tile's first group at this offset, and how many, 0 to 8, from bit 16 on)
    unsigned *s_tile = (unsigned *)(s_raw + 2 * MI * NI * kWave * 16) + wave * (kWsPer * kWave);
    int n_lane = 0;
    unsigned short ko[kWsPer][2] = {};
#pragma unroll
    for (int i = 0; i < kWsPer; i += 2)
        if (i < per) { // wave-uniform; all that are asked for are on their way together
#pragma unroll
            for (int u = i; u < i + 2; u++) {
                const unsigned short *p = a.book.tile_koff + (long)min(t0 + lane * per + min(u, per - 1), a.ntiles - 1) * (KV + 1) + k;
                ko[u][0] = p[0];
                ko[u][1] = p[1];
            }
        }
#pragma unroll
    for (int i = 0; i < kWsPer; i++) {
        if (i >= per) break; // wave-uniform
        const int g0 = min((int)ko[i][0], a.cap);
        const int n = t0 + lane * per + i < t1 ? min(max((int)ko[i][1] - g0, 0), min(a.cap - g0, R / SPH_GROUP)) : 0;
        s_tile[lane * per + i] = (unsigned)g0 | (unsigned)n << 16;
        n_lane += n;
    }
    const int incl = wave_inclusive_sum(n_lane);
    const int all = __builtin_amdgcn_readlane(incl, kWave - 1);
    // This workgroup's share of them: every parts-th batch, so that the workgroups of a chunk walk through its rows together
    // (group i of the share is group (i / GPB * parts + h) * GPB + i % GPB of the chunk).
    const int parts = k == KV / 2 ? max(min(a.nparts, all / kWsLeast), 1) : 1;
    const int round = GPB * parts, total = h < parts ? all / round * GPB + min(max(all % round - h * GPB, 0), GPB) : 0;
    if (k != KV / 2 && tid < a.nparts - 1 && blockIdx.y == 0) a.flags[slot + 1 + tid] = 0; // slots nobody fills
    if (total == 0) {
        if (tid == 0 && blockIdx.y == 0) a.flags[slot] = 0;
        return;
    }

    const unsigned strideA = a.iC * E, strideG = a.oC * E;
    const __amdgpu_buffer_rsrc_t r_a = __builtin_amdgcn_make_buffer_rsrc((void *)a.feat, 0, (int)((unsigned)a.in_rows * strideA), kRsrcFlags);
    const __amdgpu_buffer_rsrc_t r_g = __builtin_amdgcn_make_buffer_rsrc((void *)a.dout, 0, (int)((unsigned)a.out_rows * strideG), kRsrcFlags);
    // fp32: lane (m, q) loads channels MI m .. of pair 4 i + q.  16 bits: lane (c, half, q) = (lane % 8, lane / 8 % 2, lane / 16)
    // loads channels 2 MI c .. of pair 32 half + 8 q + i.
    const int q = lane >> 4, piece = HALF ? lane & 7 : lane & 15;
    constexpr int PA = HALF ? 2 * MI : MI, PG = HALF ? 2 * NI : NI; // channels of a piece
    // (what lanes behind the block's last channel read ends in rows and columns of the block that nobody looks at)
    const unsigned chanA = (ci0 + (piece * PA < cA ? piece * PA : 0)) * E, chanG = (co0 + (piece * PG < cG ? piece * PG : 0)) * E;

    float4v acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NI; j++) acc[i][j] = float4v{0, 0, 0, 0};

    // Book slot of every group of a slice: lane l looks up flattened group s0 + l, once per slice: the lane whose prefix range
    // holds it by binary search, the tile among that lane's by counting down.
    const long slot_max = (long)a.ntiles * a.cap * SPH_GROUP - 1;
    auto slot_bases = [&](int s0) -> int {
        const int f = ((s0 + lane) / GPB * parts + h) * GPB + (s0 + lane) % GPB;
        int lo = 0;
#pragma unroll
        for (int step = kWave / 2; step >= 1; step >>= 1) {
            const int v = __shfl(incl, lo + step - 1, kWave);
            if (v <= f) lo += step;
        }
        lo = min(lo, kWave - 1);
        const int before = __shfl(incl, max(lo - 1, 0), kWave);
        int left = f - (lo ? before : 0), t = lo * per, g = 0;
        bool done = false;
#pragma unroll
        for (int i = 0; i < kWsPer; i++) {
            if (i >= per) break; // wave-uniform
            const unsigned x = s_tile[lo * per + i];
            const int n = x >> 16;
            const bool here = !done && left < n;
            g = here ? (int)(x & 0xffff) + left : g;
            done |= here;
            t += done ? 0 : 1;
            left -= n;
        }
        t += t0;
        const long sl = ((long)t * a.cap + g) * SPH_GROUP;
        return (int)min(max(sl, 0L), slot_max - (SPH_GROUP - 1));   // ntiles*cap*16 fits 31 bits (checked by the launcher)
    };
    // Book entries of batch b of the slice's ng groups.  16 bits: a lane has one pair's gathered (input) row and owner (output)
    // row.  fp32: lane l < 32 the gathered row of pair l % 16, lane 32 + l its owner row.
    struct Entry { int x, y; };
    auto load_idx = [&](int bases, int ng, int b) -> Entry {
        const int pr = lane & (HALF ? kWave - 1 : SPH_GROUP - 1), fl = GPB * b + (pr >> 4);
        const int at = __shfl(bases, fl, kWave) + (pr & 15); // (a slice has no more groups than a wave lanes)
        Entry e;
        if constexpr (HALF) { e.x = a.list_in[at]; e.y = a.list_out[at]; }
        else { e.x = (lane < 32 ? a.list_in : a.list_out)[at]; e.y = 0; }
        if (fl >= ng) e.x = e.y = -1;
        return e;
    };
    // A batch's rows.  An entry that names no row counts as the row behind the last, whose bytes read as zeros.
    struct Rows { WgRow<PA * E / 4> a[PL]; WgRow<PG * E / 4> g[PL]; unsigned long long some; };
    auto offset = [&](int entry, unsigned rows, unsigned stride) -> int {
        const unsigned row = min((unsigned)entry, rows);
        return (int)(BIG ? row * stride : __umul24(row, stride));
    };
    struct Offsets { int a, g; unsigned la, lg; }; // a lane's pair's, and those of the lane's next load
    auto offsets = [&](const Entry &e, Rows &r) -> Offsets {
        Offsets o;
        if constexpr (HALF) {
            o.a = offset(e.x, a.in_rows, strideA);
            o.g = offset(e.y, a.out_rows, strideG);
        } else {
            o.a = o.g = offset(e.x, lane < 32 ? a.in_rows : a.out_rows, lane < 32 ? strideA : strideG);
            r.some = __ballot(e.x >= 0);
        }
        return o;
    };
    auto aim = [&](Offsets &o, int i) {
        const int pr = HALF ? (lane >> 3 & 1) * 32 + 8 * q + i : 4 * i + q;
        o.la = (unsigned)__builtin_amdgcn_ds_bpermute(pr * 4, o.a) + chanA;
        o.lg = (unsigned)__builtin_amdgcn_ds_bpermute((HALF ? pr : 32 + pr) * 4, o.g) + chanG;
    };
    auto load_row = [&](const Offsets &o, Rows &r, int i) {
        r.a[i].load(r_a, o.la);
        r.g[i].load(r_g, o.lg);
    };
    auto load_rows = [&](const Entry &e, Rows &r) {
        Offsets o = offsets(e, r);
#pragma unroll
        for (int i = 0; i < PL; i++) {
            aim(o, i);
            load_row(o, r, i);
        }
    };
    // fp32 takes the pairs four at a time and leaves out fours without one (a group's pairs come first, its padding
    // behind): at 32 cycles an MFMA the padding was most of what the kernel did on a strided layer's books, whose groups hold
    // five pairs of sixteen.
    // `then`: what to ask for meanwhile.  Its loads go out between the products: asked for in one go they hold the wave up until the
    // compute unit's address path has taken them, all waves of a compute unit end up doing so at the same time, and loads and
    // products take turns instead of running beside one another.
    auto multiply = [&](Rows &r, const Entry &then, Rows &to) {
        Offsets o = offsets(then, to);
        if constexpr (!HALF) {
#pragma unroll
            for (int s = 0; s < 4; s++) {
                aim(o, s);
                load_row(o, to, s);
                if (!(r.some >> (4 * s) & 15)) continue; // wave-uniform
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int j = 0; j < NI; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, r.a[s].w[i]),
                                                                         __builtin_bit_cast(float, r.g[s].w[j]), acc[i][j], 0, 0, 0);
            }
        } else {
            // both halves of sixteen lanes come to have the same pairs, half the channels of a piece each: words 0 .. MI/2-1 of the
            // first 32 pairs, MI/2 .. of the others
            aim(o, 0);
#pragma unroll
            for (int d = 0; d < NI / 2; d++)
#pragma unroll
                for (int p = 0; p < PL; p++) swap_eights(r.g[p].w[d], r.g[p].w[d + NI / 2]);
            __builtin_amdgcn_sched_barrier(0);
            auto turn = [&](const auto (&rows)[PL], int word, int odd) -> int4v { // a channel of the lane's eight pairs
                int4v f;
#pragma unroll
                for (int d = 0; d < 4; d++) // low halves or high halves of the two pairs' words
                    f[d] = (int)__builtin_amdgcn_perm(rows[2 * d + 1].w[word], rows[2 * d].w[word], odd ? 0x07060302u : 0x05040100u);
                return f;
            };
            constexpr int LOADS = PL / (2 * MI); // rows asked for behind each of the 2 MI groups of products
#pragma unroll
            for (int s = 0; s < 2; s++) {
                int4v fb[NI];
#pragma unroll
                for (int j = 0; j < NI; j++) fb[j] = turn(r.g, s * (NI / 2) + j / 2, j & 1);
#pragma unroll
                for (int i = 0; i < MI; i++) {
                    if (s == 0 && i % 2 == 0) {
#pragma unroll
                        for (int p = 0; p < PL; p++) swap_eights(r.a[p].w[i / 2], r.a[p].w[i / 2 + MI / 2]);
                    }
                    const int4v fa = turn(r.a, s * (MI / 2) + i / 2, i & 1);
#pragma unroll
                    for (int l = 0; l < LOADS; l++) {
                        const int at = (s * MI + i) * LOADS + l;
                        load_row(o, to, at);
                        if (at + 1 < PL) aim(o, at + 1);
                    }
#pragma unroll
                    for (int j = 0; j < NI; j++) acc[i][j] = mfma_step<DT>(fa, fb[j], acc[i][j]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };

    // This wave: batches wave, wave + 4, ... of every slice, NB of them.  A batch's entries are asked for two batches ahead of its
    // rows, its rows (DEPTH - 1) ahead of its products, also into the next slice.
    int bases = slot_bases(0);
    Entry e0 = load_idx(bases, total, wave), e1, e2;
    Rows r[DEPTH];
#pragma unroll
    for (int j = 0; j < DEPTH - 1; j++) {
        if (j) e0 = load_idx(bases, total, wave + 4 * j);
        load_rows(e0, r[j]);
    }
    e1 = load_idx(bases, total, wave + 4 * (DEPTH - 1));
    for (int s0 = 0;; s0 += SLICE) {
        const int ng = total - s0; // groups from here on; the last slice's batches end before NB
        const int mine = ((ng + GPB - 1) / GPB - wave + 3) / 4;
        const int later = slot_bases(s0 + SLICE);
        // (leaving, not skipping: with a way round a batch the compiler, which counts the loads in flight on every way to an
        // instruction, waits for all of them in every batch)
        auto batch = [&](auto number) -> bool {
            constexpr int j = decltype(number)::value;
            if (j >= mine) return false; // wave-uniform
            constexpr int at = j + DEPTH; // the batch behind the one whose rows are asked for now
            e2 = at < NB ? load_idx(bases, ng, wave + 4 * at) : load_idx(later, ng - SLICE, wave + 4 * (at - NB));
            __builtin_amdgcn_sched_barrier(0);
            multiply(r[j % DEPTH], e1, r[(j + DEPTH - 1) % DEPTH]);
            e1 = e2;
            return true;
        };
        each_while(batch, std::make_integer_sequence<int, NB>());
        if (ng <= SLICE) break;
        bases = later;
    }

    // Sum the four waves' blocks through LDS, pairwise: (0+2, 1+3),
    // then (0+1).  The partial is stored in accumulator order -- tile (i,j), lane, 4 values:
    // element [MI (4(lane/16) + r) + i][NI (lane%16) + j] -- as 16-byte stores; the reduction kernel
    // puts it back in [iC,oC] order.
    float4v *red = (float4v *)s_raw;
    constexpr int BLK = MI * NI * kWave;   // float4 per block
    if (wave >= 2) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++) red[(wave - 2) * BLK + (i * NI + j) * kWave + lane] = acc[i][j];
    }
    __syncthreads();
    if (wave < 2) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++) acc[i][j] += red[wave * BLK + (i * NI + j) * kWave + lane];
    }
    __syncthreads();
    if (wave == 1) {
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++) red[(i * NI + j) * kWave + lane] = acc[i][j];
    }
    __syncthreads();
    if (wave == 0) {
        float4v *part = (float4v *)(a.partial + ((long)slot * gridDim.y + blockIdx.y) * (kWsBlock * kWsBlock));
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NI; j++) part[(i * NI + j) * kWave + lane] = acc[i][j] + red[(i * NI + j) * kWave + lane];
        if (lane == 0 && blockIdx.y == 0) a.flags[slot] = 1;
    }
}

// Which channel of a block's side row (or column) m of tile i is, tiles of them.
enum { kWsRows, kWsWords, kWsHalves };
__device__ __forceinline__ int wgrad_channel(int m, int i, int tiles, int layout)
{
    if (layout == kWsRows) return 16 * i + m;                  // staged rows, channel by channel
    if (layout == kWsWords) return tiles * m + i;              // lane m has a piece of `tiles` channels
    return tiles * (2 * (m & 7) + (m >> 3)) + i;               // and, behind the exchange, half m / 8 of piece m % 8
}

// dw[k][ci][co] = sum of the written slots of offset k, in slot order.  A slot holds one
// 64x64 block per (iC,oC) block pair, each in accumulator order of MI x NI tiles (see
// wgrad_wave_kernel).  A thread owns one 16-byte item of a block (four ci of one co), so the
// slots are read as they were written; a workgroup covers 32 consecutive items, its 8 groups of
// 32 threads each add every 8th slot (up to sixteen loads in flight), and the 8 sub-sums are added in a
// fixed order.
template <typename OUT>
__global__ __launch_bounds__(256) void wgrad_slot_reduce_kernel(const float *partial, const int *flags, int slots_per_k,
                                                                int iC, int oC, int mi_tiles, int ni_tiles, int layout, OUT *dw)
{
    __shared__ float4v s_sum[8][32];
    __shared__ unsigned long long s_flags[16];
    const int k = blockIdx.z, b = blockIdx.y, t = threadIdx.x & 31, j = threadIdx.x >> 5;
    const int q = blockIdx.x * 32 + t;       // 16-byte item of the block, in accumulator order
    const int sbn = (oC + kWsBlock - 1) / kWsBlock, nblk = ((iC + kWsBlock - 1) / kWsBlock) * sbn;
    const int tile = q >> 6, lane = q & 63;
    const bool live = tile < mi_tiles * ni_tiles;
    const long blk = (long)kWsBlock * kWsBlock, step = (long)nblk * blk;
    const float *p = partial + ((long)k * slots_per_k * nblk + b) * blk + q * 4;
    const int *f = flags + (long)k * slots_per_k;
    float4v s = {0.f, 0.f, 0.f, 0.f};
    // The flags of 1024 slots at a time become 16 ballot words in LDS, so that a thread's data loads do not
    // wait for flag loads: per round a thread takes its 16 candidates of two words (slots j, j+8, ... of each),
    // the loads of the written ones in flight together, and adds them in slot order.
    for (int base = 0; base < slots_per_k; base += 1024) {
        __syncthreads();
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const int c = base + w * 256 + (int)threadIdx.x;
            const unsigned long long m = __ballot(c < slots_per_k && f[c] != 0);
            if ((threadIdx.x & (kWave - 1)) == 0) s_flags[w * 4 + (threadIdx.x >> 6)] = m;
        }
        __syncthreads();
        if (!live) continue;
        const int nwords = min(16, (slots_per_k - base + 63) >> 6);
        for (int w0 = 0; w0 < nwords; w0 += 2) {
            const unsigned long long m0 = s_flags[w0] >> j, m1 = w0 + 1 < nwords ? s_flags[w0 + 1] >> j : 0ull;
            float4v v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) {
                const unsigned long long m = u < 8 ? m0 : m1;
                const int cc = base + (w0 + (u >> 3)) * 64 + j + 8 * (u & 7);
                v[u] = float4v{0.f, 0.f, 0.f, 0.f};
                if ((m >> (8 * (u & 7))) & 1ull) v[u] = *(const float4v *)(p + cc * step);
            }
#pragma unroll
            for (int u = 0; u < 16; u++) s += v[u];
        }
    }
    s_sum[j][t] = s;
    __syncthreads();
    if (j == 0 && live) {
        float4v r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int g = 0; g < 8; g++) r += s_sum[g][t];
        // accumulator order inside the block: tile (i, j), lane, value v are row 4 (lane / 16) + v and column lane % 16
        const int co = (b % sbn) * kWsBlock + wgrad_channel(lane & 15, tile % ni_tiles, ni_tiles, layout);
        if (co < oC) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int ci = (b / sbn) * kWsBlock + wgrad_channel((lane >> 4) * 4 + v, tile / ni_tiles, mi_tiles, layout);
                if (ci < iC) dw[((long)k * iC + ci) * oC + co] = (OUT)r[v];
            }
        }
    }
}

inline int wgrad_chunks(int ntiles) { return ntiles < 32 ? (ntiles < 1 ? 1 : ntiles) : 32; }

// 16-channel tiles of one side of the widest block: 1, 2 or 4
inline int wgrad_tiles(int channels)
{
    const int t = sph_div_up(channels < kWsBlock ? channels : kWsBlock, 16);
    return t <= 1 ? 1 : (t <= 2 ? 2 : 4);
}
inline int wgrad_blocks(int iC, int oC) { return sph_div_up(iC, kWsBlock) * sph_div_up(oC, kWsBlock); }
inline size_t wgrad_stage_lds(int mi, int ni)
{
    const size_t stage = (size_t)4 * 2 * SPH_GROUP * ((mi * 32 + 16) + (ni * 32 + 16));
    const size_t red = (size_t)2 * mi * ni * kWave * 4 * sizeof(float); // two waves' blocks at once
    return stage > red ? stage : red;
}
inline int wgrad_stage_chunks(int ntiles) { return ntiles < 1 ? 1 : sph_div_up(ntiles, kWsTiles); }
// two waves' blocks at once, and behind them every wave's tiles
inline size_t wgrad_wave_lds(int mi, int ni) { return (size_t)2 * mi * ni * kWave * 4 * sizeof(float) + 4 * kWsPer * kWave * sizeof(unsigned); }
// Workgroups of wgrad_wave_kernel on a compute unit, by its registers (197 to 256, 141 to 194 for a side of 64 channels, 113 at most).
inline int wgrad_wave_occupancy(bool f32, int mi, int ni) { return mi * ni >= 16 || !f32 ? 2 : (mi * ni >= 8 ? 3 : 4); }
// Does the middle offset hold far more pairs than the others?  The caller says so; a layer with as many rows out as in is taken for one too.
inline bool wgrad_run(const WgradArgs &a) { return book_has_run(&a.book) || a.in_rows == a.out_rows; }
struct WavePlan { int nchunk, nparts; };
// Chunks of a book's tiles, and workgroups that share a chunk's groups at the centre offset: one round of workgroups of about the same number of
// groups each.  A submanifold book has eight groups a tile at the centre and about one at the others, so eight share the centre's; of small
// kernels (most of their offsets' pairs are there) four.  Where no offset stands out one: with eight the others' workgroups were four
// times as long as the centre's and half the chip idle (2x2x2 stride 2, 64->64 f16, 998 tiles 20.3 us through LDS, 23.9 with eight, 18.4 with
// one; fp32, transposed book of 16 611 tiles 259, 511, 187).
// A round: with whole chunks to an XCD (sixteen of them, six workgroups at the centre) 3 % fewer lines come from memory, and the centre's
// workgroups last a third longer than the others: 32.9 : 29.0 us.
// An offset has at most 256 partial blocks in a round: few workgroups add up those of a small kernel (1x1x1, 2005 tiles, 32->64 f16: 504 blocks
// 19.8 us, 252 17.3).
// A small book's chunks are eight, or of 48 tiles for 27 offsets (fp32: 16) if that is more, and in 16 bits of no fewer than eight tiles: each more
// writes a block for every offset and one for each of the centre's workgroups, and the sum of them then lasts longer than
// the chunks' loads are shorter (608 tiles, 64->64 f16: 19 chunks 23 us, 13 20.5; nine offsets: 8 chunks 21, 38 18; a full grid of 16 tiles,
// 27 offsets: 2 chunks 16.2, 1 chunk 20.0).  In fp32 a chunk's chain of products is longer (a full grid of 462 tiles, 64->64: 15 chunks
// 125 us, 10 181; of 16 tiles: 8 chunks 16.3, 2 28.5).
// A long book's chunks hold 192 tiles at most, 128 where a compute unit has three workgroups or four: the offsets of a longer chunk fall so far
// behind each other that their rows are no longer in the XCD's L2 (64->64 f16, a full grid of 9002 tiles: chunks of 300 tiles 574 us, through LDS 537;
// 32->32 fp32, stride 2, transposed book of 7057 tiles: chunks of 236 tiles 170, 96 tiles 143, through LDS 131).
inline WavePlan wgrad_wave_plan(int ntiles, int KV, int blocks, int occupancy, bool f32, bool run)
{
    const int nparts = !run ? 1 : (KV >= 16 ? kWsParts : kWsParts / 2);
    const int slots = 256 / nparts, all = 256 * occupancy / ((KV - 1 + nparts) * blocks), fit = all < slots ? all : slots, round = fit < 1 ? 1 : fit;
    const int of27 = (f32 ? 16 : 48) * KV / 27, least = run ? (f32 ? 8 : 16) : 4, tiles = of27 > least ? of27 : least;
    if (ntiles < tiles * round) {
        const int most = f32 ? ntiles : sph_div_up(ntiles, 8);
        const int n = sph_div_up(ntiles, tiles) < 8 ? 8 : sph_div_up(ntiles, tiles);
        const int r = n < round ? n : round, m = r < most ? r : most;
        return WavePlan{m < 1 ? 1 : m, nparts};
    }
    int n = round;
    while (sph_div_up(ntiles, n) > (occupancy > 2 ? kWsMostLight : kWsMost)) n += round;
    return WavePlan{n, nparts};
}
inline bool wgrad_wave_ok(sph_dtype dt, int iC, int oC)
{
    const int e = sph_elem_size(dt);
    return (iC * e) % 16 == 0 && (oC * e) % 16 == 0;
}

template <sph_dtype DT>
int launch_wgrad(const WgradArgs &a0, void *dw, bool f32_out, hipStream_t st)
{
    typedef typename Traits<DT>::elem elem;
    const int KV = a0.book.KV;
    const int per_k = a0.iC * a0.oC;
    const long total = (long)KV * per_k;
    const bool aligned = ((uintptr_t)a0.feat % 16 == 0) && ((uintptr_t)a0.dout % 16 == 0);
    const bool small = (double)a0.in_rows * a0.iC * sizeof(elem) < 4294966784.0 &&
                       (double)a0.out_rows * a0.oC * sizeof(elem) < 4294966784.0 &&
                       (double)a0.ntiles * a0.cap * SPH_GROUP < 2147483648.0;
    if (wgrad_wave_ok(DT, a0.iC, a0.oC) && aligned && small && a0.in_rows > 0 && a0.out_rows > 0) {
        WgradArgs a = a0;
        constexpr bool F32 = sizeof(elem) == 4;
        const int sb = wgrad_blocks(a.iC, a.oC);
        int mi = wgrad_tiles(a.iC), ni = wgrad_tiles(a.oC), slots, layout;
        // (books of four tiles or less: with 32 channels on one side this kernel's shorter way to its first product is 0.6 us of 9)
        if (!F32 && (mi * ni <= 4 || (mi * ni == 8 && a.ntiles <= 4))) {
            a.nchunk = wgrad_stage_chunks(a.ntiles);
            // the centre offset's chain is what a small book's kernel lasts: eight workgroups share it there; on large
            // books four, which halves the partial blocks to write and add
            a.nslice = a.nchunk <= 16 ? kWsSlices : kWsSlices / 2;
            slots = a.nchunk * a.nslice;
            layout = kWsRows;
            a.flags = (int *)(a.partial + (size_t)KV * slots * sb * kWsBlock * kWsBlock);
            // later slices for every offset only where the whole grid stays small (measured: a full 4x4x128x4 grid, one
            // chunk, 15 us with them and 33 us without; 8 chunks 32 against 35 us; from 12 chunks on the shorter grid wins)
            a.all_slices = KV * a.nchunk * 4 <= 1024;
            const dim3 grid(sph_xcd_grid(KV * a.nchunk) + (a.nslice - 1) * a.nchunk * (a.all_slices ? KV : 1), sb), block(256);
            if constexpr (!F32) {
#define SPH_WGRAD_CASE(M, N) \
    if (mi == M && ni == N) hipLaunchKernelGGL((wgrad_stage_kernel<DT, M, N>), grid, block, wgrad_stage_lds(M, N), st, a);
                SPH_WGRAD_CASE(1, 1) SPH_WGRAD_CASE(1, 2) SPH_WGRAD_CASE(1, 4) SPH_WGRAD_CASE(2, 1) SPH_WGRAD_CASE(2, 2) SPH_WGRAD_CASE(4, 1)
                SPH_WGRAD_CASE(2, 4) SPH_WGRAD_CASE(4, 2)
#undef SPH_WGRAD_CASE
            }
        } else {
            const WavePlan plan = wgrad_wave_plan(a.ntiles, KV, sb, wgrad_wave_occupancy(F32, mi, ni), F32, wgrad_run(a));
            a.nchunk = plan.nchunk;
            a.nparts = plan.nparts;
            a.chunk_tiles = sph_div_up(a.ntiles, a.nchunk);
            slots = a.nchunk * a.nparts;
            layout = F32 ? kWsWords : kWsHalves;
            a.flags = (int *)(a.partial + (size_t)KV * slots * sb * kWsBlock * kWsBlock);
            const dim3 grid(sph_xcd_grid((KV - 1 + a.nparts) * a.nchunk), sb), block(256);
            const bool big = a.in_rows >= (1 << 24) || a.out_rows >= (1 << 24);
#define SPH_WGRAD_CASE(M, N)                                                                                       \
    if (mi == M && ni == N) {                                                                                      \
        if (big) hipLaunchKernelGGL((wgrad_wave_kernel<DT, M, N, true>), grid, block, wgrad_wave_lds(M, N), st, a); \
        else hipLaunchKernelGGL((wgrad_wave_kernel<DT, M, N, false>), grid, block, wgrad_wave_lds(M, N), st, a);    \
    }
            if constexpr (F32) {
                SPH_WGRAD_CASE(1, 1) SPH_WGRAD_CASE(1, 2) SPH_WGRAD_CASE(1, 4) SPH_WGRAD_CASE(2, 1) SPH_WGRAD_CASE(2, 2) SPH_WGRAD_CASE(4, 1)
            }
            SPH_WGRAD_CASE(2, 4) SPH_WGRAD_CASE(4, 2) SPH_WGRAD_CASE(4, 4)
#undef SPH_WGRAD_CASE
        }
        int rc = sph_check_launch("sph_conv_wgrad");
        if (rc) return rc;
        const dim3 grid((unsigned)(mi * ni * 2), sb, KV);
        if (f32_out)
            hipLaunchKernelGGL(wgrad_slot_reduce_kernel<float>, grid, dim3(256), 0, st, a.partial, a.flags, slots, a.iC, a.oC, mi, ni, layout, (float *)dw);
        else
            hipLaunchKernelGGL(wgrad_slot_reduce_kernel<elem>, grid, dim3(256), 0, st, a.partial, a.flags, slots, a.iC, a.oC, mi, ni, layout, (elem *)dw);
        return sph_check_launch("sph_conv_wgrad(reduce)");
    }
    const WgradArgs &a = a0;
    constexpr int LDP = 4 * Traits<DT>::KW + 16 / (int)sizeof(elem);
    const int iCp = (a.iC + 15) & ~15, oCp = (a.oC + 15) & ~15;
    size_t lds = (size_t)(iCp + oCp) * LDP * sizeof(elem);
    hipLaunchKernelGGL(wgrad_kernel<DT>, dim3(KV * a.nchunk), dim3(kWgThreads), lds, st, a);
    int rc = sph_check_launch("sph_conv_wgrad");
    if (rc) return rc;
    if (f32_out)
        hipLaunchKernelGGL(wgrad_reduce_kernel<float>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                           a.partial, KV, a.nchunk, per_k, (float *)dw);
    else
        hipLaunchKernelGGL(wgrad_reduce_kernel<elem>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                           a.partial, KV, a.nchunk, per_k, (elem *)dw);
    return sph_check_launch("sph_conv_wgrad(reduce)");
}

} // namespace

SPH_EXPORT size_t sph_wgrad_partial_elems(int KV, int iC, int oC, int out_rows)
{
    if (KV <= 0 || iC <= 0 || oC <= 0) return 0;
    const int ntiles = sph_book_tiles(out_rows);
    const size_t general = (size_t)KV * wgrad_chunks(ntiles) * iC * oC;
    // whichever kernel and type takes it
    size_t slots = (size_t)KV * wgrad_stage_chunks(ntiles) * kWsSlices;
    for (int i = 0; i < 4; i++)
        for (int occupancy = 2; occupancy <= 4; occupancy++) {
            const WavePlan p = wgrad_wave_plan(ntiles, KV, wgrad_blocks(iC, oC), occupancy, i & 1, i & 2);
            const size_t wave = (size_t)KV * p.nchunk * p.nparts;
            slots = wave > slots ? wave : slots;
        }
    const size_t blocks = (size_t)sph_div_up(iC, kWsBlock) * sph_div_up(oC, kWsBlock);
    const size_t fast = slots * blocks * kWsBlock * kWsBlock + slots; // 64x64 blocks + one flag word per slot
    return general > fast ? general : fast;
}

// `book`: stationary on the output rows, or on the input rows (`transposed`); other_rows: the rows its groups gather
static int conv_wgrad(sph_dtype dt, const void *feature, int iC, const void *d_out, int oC, const sph_book *book, int other_rows,
                      bool transposed, float *partial, void *d_weight, int d_weight_f32, void *stream)
{
    SPH_REQUIRE(book_ok(book) && book_has_groups(book), SPH_ERR_ARG, "sph_conv_wgrad: bad book (it must hold its groups)");
    SPH_REQUIRE(partial && d_weight, SPH_ERR_ARG, "sph_conv_wgrad: null pointer");
    SPH_REQUIRE(dt == SPH_F32 || dt == SPH_F16 || dt == SPH_BF16, SPH_ERR_UNSUPPORTED,
                "sph_conv_wgrad: dtype %d has no weight gradient", (int)dt);
    SPH_REQUIRE(iC > 0 && iC <= 128 && oC > 0 && oC <= 128, SPH_ERR_UNSUPPORTED,
                "sph_conv_wgrad: channels %d->%d not in 1..128", iC, oC);
    const int in_rows = transposed ? book->rows : other_rows, out_rows = transposed ? other_rows : book->rows;
    SPH_REQUIRE((in_rows == 0 || feature) && (out_rows == 0 || d_out), SPH_ERR_ARG, "sph_conv_wgrad: null pointer");
    WgradArgs a;
    a.feat = (const char *)feature;
    a.in_rows = in_rows;
    a.iC = iC;
    a.dout = (const char *)d_out;
    a.out_rows = out_rows;
    a.oC = oC;
    a.book = *book;
    a.list_in = transposed ? book->grp_owner : book->grp_gather;
    a.list_out = transposed ? book->grp_gather : book->grp_owner;
    a.cap = sph_book_cap(book->KV);
    a.ntiles = sph_book_tiles(book->rows);
    a.nchunk = wgrad_chunks(a.ntiles);
    a.partial = partial;
    a.flags = nullptr;
    a.nslice = a.all_slices = a.chunk_tiles = a.nparts = 0;
    hipStream_t st = (hipStream_t)stream;
    switch (dt) {
    case SPH_F32: return launch_wgrad<SPH_F32>(a, d_weight, true, st);
    case SPH_F16: return launch_wgrad<SPH_F16>(a, d_weight, d_weight_f32 != 0, st);
    default: return launch_wgrad<SPH_BF16>(a, d_weight, d_weight_f32 != 0, st);
    }
}

SPH_EXPORT int sph_conv_wgrad(sph_dtype dt, const void *feature, int in_rows, int iC, const void *d_out,
                              int oC, const sph_book *fwd_book, float *partial, void *d_weight, int d_weight_f32,
                              void *stream)
{
    return conv_wgrad(dt, feature, iC, d_out, oC, fwd_book, in_rows, false, partial, d_weight, d_weight_f32, stream);
}

SPH_EXPORT int sph_conv_wgrad_transposed(sph_dtype dt, const void *feature, int iC, const void *d_out, int out_rows, int oC,
                                         const sph_book *t_book, float *partial, void *d_weight, int d_weight_f32, void *stream)
{
    return conv_wgrad(dt, feature, iC, d_out, oC, t_book, out_rows, true, partial, d_weight, d_weight_f32, stream);
}
