// Weight packing shared by the stand-alone kernel (sph_weight_pack) and by the rule kernel
// launch that carries it as extra workgroups (sph_rules_build_pack).
//
// packed[k][step][ntile][lane][KW] holds weight element (k, kk, n) with
//   kk = step*4*KW + KW*(lane/16) + j,  n = ntile*16 + lane%16,  KW = 16 / element size,
// zero padded: the order in which an MFMA lane reads its 16-byte operand fragment.
// The copy is a permutation of elements, so it only depends on the element size.
#pragma once
#include "common.h"

struct SphPackJob {
    const void *w;
    void *packed;
    int elem_size;          // 1, 2 or 4 bytes of an element of the packed copy
    int narrow;             // 0: w holds elements of that size; 1 / 2: w is fp32, rounded to fp16 / bf16 on the way
    int KV, kdim, ndim, nsteps, ntn;
    long sk, skk, sn;       // element strides of w over (k, kk, n)
    int total;              // 16-byte fragments of the packed copy
};

static inline int sph_elem_size(sph_dtype dt) { return dt == SPH_F32 ? 4 : (dt == SPH_I8 ? 1 : 2); }
static inline int sph_frag_elems(sph_dtype dt) { return 16 / sph_elem_size(dt); }
// output-column tiles of 16, padded to 1, 2, 4 or 8
static inline int sph_pad_waves(int ndim)
{
    int nt = sph_div_up(ndim, 16);
    return nt <= 1 ? 1 : (nt <= 2 ? 2 : (nt <= 4 ? 4 : 8));
}
// MFMA super steps (64 bytes of every row each) of a contraction over kdim elements
static inline int sph_num_steps(sph_dtype dt, int kdim) { return sph_div_up(kdim, 4 * sph_frag_elems(dt)); }
static inline SphPackJob sph_pack_job(sph_dtype dt, const void *w, int KV, int kdim, int ndim, long sk, long skk,
                                      long sn, void *packed, int w_f32 = 0)
{
    SphPackJob p;
    p.w = w; p.packed = packed; p.elem_size = sph_elem_size(dt);
    p.narrow = !w_f32 || dt == SPH_F32 ? 0 : (dt == SPH_F16 ? 1 : 2);
    p.KV = KV; p.kdim = kdim; p.ndim = ndim;
    p.nsteps = sph_num_steps(dt, kdim); p.ntn = sph_pad_waves(ndim);
    p.sk = sk; p.skk = skk; p.sn = sn;
    p.total = KV * p.nsteps * p.ntn * 64;
    return p;
}
// argument checks shared by the entry points that pack; returns 0 or an error code (message set)
static inline int sph_pack_args_ok(const char *who, sph_dtype dt, const void *w, void *packed, int KV, int kdim, int ndim)
{
    if (!w || !packed) { sph_set_error("%s: null pointer", who); return SPH_ERR_ARG; }
    if ((int)dt < 0 || (int)dt > 3) { sph_set_error("%s: unknown dtype %d", who, (int)dt); return SPH_ERR_ARG; }
    if (KV <= 0 || KV > SPH_MAX_KV) { sph_set_error("%s: kernel volume %d not in 1..%d", who, KV, SPH_MAX_KV); return SPH_ERR_UNSUPPORTED; }
    if (kdim <= 0 || kdim > SPH_MAX_CHANNELS) { sph_set_error("%s: %d input channels not in 1..%d", who, kdim, SPH_MAX_CHANNELS); return SPH_ERR_UNSUPPORTED; }
    if (ndim <= 0 || ndim > 128) { sph_set_error("%s: %d output channels not in 1..128", who, ndim); return SPH_ERR_UNSUPPORTED; }
    return SPH_OK;
}

// Up to two jobs share a launch: a training step wants the weight for its forward pass and, transposed, for dgrad.
struct SphPackJobs {
    SphPackJob job[2]; // total == 0: no job
};
static inline int sph_pack_total(const SphPackJob *jobs) { return jobs[0].total + jobs[1].total; }
static inline int sph_pack_jobs(const char *who, const sph_pack_desc *d, int n, SphPackJobs *out)
{
    out->job[0].total = out->job[1].total = 0;
    if (n < 0 || n > 2 || (n > 0 && !d)) { sph_set_error("%s: 0 to 2 weights can be packed, not %d", who, n); return SPH_ERR_ARG; }
    for (int i = 0; i < n; i++) {
        int rc = sph_pack_args_ok(who, d[i].dt, d[i].w, d[i].packed, d[i].KV, d[i].kdim, d[i].ndim);
        if (rc) return rc;
        if (d[i].w_f32 && d[i].dt == SPH_I8) { sph_set_error("%s: an fp32 weight has no int8 copy", who); return SPH_ERR_ARG; }
        if ((uintptr_t)d[i].packed % 16) { sph_set_error("%s: packed weight must be 16-byte aligned", who); return SPH_ERR_ARG; }
        out->job[i] = sph_pack_job(d[i].dt, d[i].w, d[i].KV, d[i].kdim, d[i].ndim, d[i].stride_k, d[i].stride_kk,
                                   d[i].stride_n, d[i].packed, d[i].w_f32);
    }
    return SPH_OK;
}

#ifdef __HIPCC__
// Fragment i of the job.  T: element of the packed copy, S: element of w.  A lane's 16 bytes are put together in
// registers and stored at once (one division chain per 16 bytes instead of one per element); the 16 lanes of a column
// tile read neighbouring columns (forward weights) or 16 bytes of one column each (transposed ones).
template <typename T, typename S>
__device__ __forceinline__ void sph_pack_fragment_as(const SphPackJob &p, int i)
{
    constexpr int KW = 16 / (int)sizeof(T);
    const int lane = i & 63;
    int t = i >> 6;
    const int nt = t % p.ntn;
    t /= p.ntn;
    const int st = t % p.nsteps, k = t / p.nsteps;
    const int kk0 = st * 4 * KW + KW * (lane >> 4), n = nt * 16 + (lane & 15);
    const S *src = (const S *)p.w + k * p.sk + kk0 * p.skk + n * p.sn;
    union { T e[KW]; uint4 v; } u;
#pragma unroll
    for (int j = 0; j < KW; j++) u.e[j] = (kk0 + j < p.kdim && n < p.ndim) ? (T)src[j * p.skk] : (T)0;
    ((uint4 *)p.packed)[i] = u.v;
}

// fragment i of the job, whatever its types (a permutation of elements, so equal types go by their size)
__device__ __forceinline__ void sph_pack_fragment(const SphPackJob &p, int i)
{
    if (i >= p.total) return;
    if (p.narrow == 1) sph_pack_fragment_as<_Float16, float>(p, i);
    else if (p.narrow == 2) sph_pack_fragment_as<__bf16, float>(p, i);
    else if (p.elem_size == 2) sph_pack_fragment_as<uint16_t, uint16_t>(p, i);
    else if (p.elem_size == 4) sph_pack_fragment_as<uint32_t, uint32_t>(p, i);
    else sph_pack_fragment_as<uint8_t, uint8_t>(p, i);
}

__device__ __forceinline__ void sph_pack_fragments(const SphPackJobs &p, int i)
{
    if (i < p.job[0].total) sph_pack_fragment(p.job[0], i);
    else sph_pack_fragment(p.job[1], i - p.job[0].total);
}
#endif
