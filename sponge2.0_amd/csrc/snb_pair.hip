// snb_pair.hip -- LJ + erfc-screened Coulomb over the half neighbor list, and
// the PME exclusion correction.
//
// Pair kernel (stands in for Lennard_Jones_And_Direct_Coulomb_Device,
// Lennard_Jones_force.cpp:43-136): one wavefront per row i of the reference
// layout half list; 64 lanes stride the row (coalesced 256-byte reads of the
// padded int table), gather j's packed {x, y, z, q} record and LJ type, and
// evaluate the pair in float with the library's own exp/erfc/rsqrt.  Every
// per-pair term is rounded to int64 fixed point before it is added, so the
// i-sums (wave reduction) and the j-scatter (64-bit integer atomics) give the
// same bits in any order.  Energies and virials of a pair go to row atom i,
// as in the reference; they are written once per row with plain stores.
#include "snb_internal.h"

__device__ __forceinline__ void pbc_disp(float& dx, float& dy, float& dz, const SnbBox& box)
{
    float sx = (dx * box.rc[0] + dy * box.rc[1]) + dz * box.rc[3];
    float sy = dy * box.rc[2] + dz * box.rc[4];
    float sz = dz * box.rc[5];
    float kx = floorf(sx + 0.5f), ky = floorf(sy + 0.5f), kz = floorf(sz + 0.5f);
    dx = dx - ((kx * box.c[0] + ky * box.c[1]) + kz * box.c[3]);
    dy = dy - (ky * box.c[2] + kz * box.c[4]);
    dz = dz - kz * box.c[5];
}

// Element i of an array addressed with a 32-bit byte offset: the load can use
// the scalar-base + unsigned vector-offset form (the offset is computed in 32
// bits, which holds for every array of this library).
template <class T>
__device__ __forceinline__ T ld32(const T* __restrict__ base, unsigned i)
{
    return *(const T*)((const char*)base + i * (unsigned)sizeof(T));
}

__device__ __forceinline__ int64_t wave_sum(int64_t v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// a value that is the same in the whole wavefront, in a scalar register
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float unif(float v) { return __int_as_float(uni(__float_as_int(v))); }

// x + (x of the lane CTRL selects), lanes permuted by DPP within rows of 16
template <int CTRL>
__device__ __forceinline__ int64_t add_dpp(int64_t x)
{
    const int lo = (int)x, hi = (int)(x >> 32);
    const unsigned l2 = (unsigned)__builtin_amdgcn_mov_dpp(lo, CTRL, 0xf, 0xf, true);
    const int h2 = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xf, 0xf, true);
    return x + (int64_t)(((uint64_t)(unsigned)h2 << 32) | l2);
}

// minimum over the wavefront, in every lane (a NaN counts as no value)
__device__ __forceinline__ float wave_min(float v)
{
    auto step = [&](int w) { v = fminf(v, __int_as_float(w)); };
    step(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x128, 0xf, 0xf, true));
    step(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x124, 0xf, 0xf, true));
    step(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x122, 0xf, 0xf, true));
    step(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x121, 0xf, 0xf, true));
    const int i = __float_as_int(v);
    return fminf(fminf(__int_as_float(__builtin_amdgcn_readlane(i, 0)),
                       __int_as_float(__builtin_amdgcn_readlane(i, 16))),
                 fminf(__int_as_float(__builtin_amdgcn_readlane(i, 32)),
                       __int_as_float(__builtin_amdgcn_readlane(i, 48))));
}

// Sums of three values over the wavefront: lanes 0..15 return the sum of x,
// lanes 16..31 and 48..63 that of z, lanes 32..47 that of y.  The halves and
// then the rows of 16 lanes are folded onto each other with two values in
// flight (permlane swaps), the rows by rotations: 21 vector instructions and
// no LDS, where a butterfly of each value takes 36 LDS permutes and their waits.
__device__ __forceinline__ int64_t wave_sum3(int64_t x, int64_t y, int64_t z)
{
    auto swap32 = [](int64_t a, int64_t b) -> int64_t {
        const auto l = __builtin_amdgcn_permlane32_swap((int)a, (int)b, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap((int)(a >> 32), (int)(b >> 32), false,
                                                        false);
        return (int64_t)(((uint64_t)h[0] << 32) | l[0]) + (int64_t)(((uint64_t)h[1] << 32) | l[1]);
    };
    auto swap16 = [](int64_t a, int64_t b) -> int64_t {
        const auto l = __builtin_amdgcn_permlane16_swap((int)a, (int)b, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap((int)(a >> 32), (int)(b >> 32), false,
                                                        false);
        return (int64_t)(((uint64_t)h[0] << 32) | l[0]) + (int64_t)(((uint64_t)h[1] << 32) | l[1]);
    };
    const int64_t xy = swap32(x, y);  // lanes 0..31: x, 32..63: y
    const int64_t zz = swap32(z, z);  // both halves: z
    int64_t v = swap16(xy, zz);       // rows: x, z, y, z
    v = add_dpp<0x128>(v);            // row_ror:8
    v = add_dpp<0x124>(v);
    v = add_dpp<0x122>(v);
    return add_dpp<0x121>(v);
}

__device__ __forceinline__ void atomic_add_i64(int64_t* p, int64_t v)
{
    atomicAdd((unsigned long long*)p, (unsigned long long)v);
}

// Force factor of one pair (Lennard_Jones_force.cpp:73-97): LJ plus the
// erfc-screened Coulomb term, float arithmetic of the library's own math,
// the Coulomb shape from the Hermite table (ctab, SNB_COUL_N float4 pieces).
// A, B and qq may carry a common power-of-two scale; the result then carries
// it exactly (every operation is a product or difference of scaled terms).
__device__ __forceinline__ float pair_force_factor(float r2, float A, float B, float qq,
                                                   float beta, float cscale,
                                                   const float4* ctab)
{
    float rinv = snb_rsqrtf(r2);
    float r = r2 * rinv;
    float rinv2 = rinv * rinv;
    float rinv6 = (rinv2 * rinv2) * rinv2;
    float flj = ((B - A * rinv6) * rinv6) * rinv2;
    float t;
    int k = snb_coul_piece(beta * r, cscale, &t);
    float4 c = ctab[k];
    float fc = (qq * (rinv2 * rinv)) * snb_coul_eval(t, c.x, c.y, c.z, c.w);
    return flj - fc;
}

// The Coulomb part alone: pair_force_factor with A = B = 0 returns 0 - this.
__device__ __forceinline__ float pair_coulomb_factor(float r2, float qq, float beta, float cscale,
                                                     const float4* ctab)
{
    const float rinv = snb_rsqrtf(r2);
    const float r = r2 * rinv;
    const float rinv2 = rinv * rinv;
    float t;
    const int k = snb_coul_piece(beta * r, cscale, &t);
    const float4 c = ctab[k];
    return (qq * (rinv2 * rinv)) * snb_coul_eval(t, c.x, c.y, c.z, c.w);
}

template <bool NEED_ENERGY, bool NEED_VIRIAL>
__device__ __forceinline__ void k_lj_direct_body(
    int n, const snb_atom_group* __restrict__ nl, const float4* __restrict__ atoms,
    const int* __restrict__ type, const float* __restrict__ lj_a,
    const float* __restrict__ lj_b, const float4* __restrict__ coul_tab, float cscale,
    SnbBox box, float rc2, float beta,
    int64_t* __restrict__ fx, int64_t* __restrict__ e_atom, int64_t* __restrict__ vir,
    unsigned bid, unsigned nbid)
{
    const int lane = threadIdx.x & 63;
    const int waves = nbid * 4;
    for (int i = bid * 4 + (threadIdx.x >> 6); i < n; i += waves)
    {
        const snb_atom_group g = nl[i];
        const float4 ai = atoms[i];
        const int ti = type[i];
        int64_t sx = 0, sy = 0, sz = 0, elj = 0, ec = 0;
        int64_t v0 = 0, v1 = 0, v2 = 0, v3 = 0, v4 = 0, v5 = 0;
        for (int k = lane; k < g.atom_numbers; k += 64)
        {
            const int j = g.atom_serial[k];
            const float4 aj = atoms[j];
            // Get_Periodic_Displacement(r_j, r_i) (Lennard_Jones_force.cpp:72)
            float dx = aj.x - ai.x, dy = aj.y - ai.y, dz = aj.z - ai.z;
            pbc_disp(dx, dy, dz, box);
            float r2 = (dx * dx + dy * dy) + dz * dz;
            if (!(r2 < rc2)) continue;
            const int p = snb_lj_pair_index(ti, type[j]);
            const float A = lj_a[p], B = lj_b[p];
            const float fa = pair_force_factor(r2, A, B, ai.w * aj.w, beta, cscale, coul_tab);
            float fxv = fa * dx, fyv = fa * dy, fzv = fa * dz;
            int64_t ix = snb_to_fixed(fxv), iy = snb_to_fixed(fyv), iz = snb_to_fixed(fzv);
            sx += ix;
            sy += iy;
            sz += iz;
            atomic_add_i64(fx + j, -ix);
            atomic_add_i64(fx + n + j, -iy);
            atomic_add_i64(fx + 2 * n + j, -iz);
            if (NEED_ENERGY)
            {
                // energies in FP64 from the (exact) float displacement
                double ddx = dx, ddy = dy, ddz = dz;
                double r2d = (ddx * ddx + ddy * ddy) + ddz * ddz;
                double rd = __builtin_sqrt(r2d);
                double rid = 1.0 / rd;
                double ri2 = rid * rid;
                double ri6 = (ri2 * ri2) * ri2;
                elj += snb_to_fixed_d((((double)A * (1.0 / 12.0)) * ri6 - (double)B * (1.0 / 6.0)) *
                                      ri6);
                double gd;
                const double erfcd = snb_erfc_parts_d((double)beta * rd, &gd);
                ec += snb_to_fixed_d((((double)ai.w * (double)aj.w) * erfcd) * rid);
            }
            if (NEED_VIRIAL)
            {
                v0 += snb_to_fixed(-(fxv * dx));
                v1 += snb_to_fixed(-(fxv * dy + fyv * dx));
                v2 += snb_to_fixed(-(fyv * dy));
                v3 += snb_to_fixed(-(fxv * dz + fzv * dx));
                v4 += snb_to_fixed(-(fyv * dz + fzv * dy));
                v5 += snb_to_fixed(-(fzv * dz));
            }
        }
        sx = wave_sum(sx);
        sy = wave_sum(sy);
        sz = wave_sum(sz);
        if (NEED_ENERGY)
        {
            elj = wave_sum(elj);
            ec = wave_sum(ec);
        }
        if (NEED_VIRIAL)
        {
            v0 = wave_sum(v0); v1 = wave_sum(v1); v2 = wave_sum(v2);
            v3 = wave_sum(v3); v4 = wave_sum(v4); v5 = wave_sum(v5);
        }
        if (lane == 0)
        {
            atomic_add_i64(fx + i, sx);
            atomic_add_i64(fx + n + i, sy);
            atomic_add_i64(fx + 2 * n + i, sz);
            if (NEED_ENERGY)
            {
                e_atom[i] += elj;
                e_atom[(size_t)n + i] += ec;
            }
            if (NEED_VIRIAL)
            {
                vir[i] += v0;
                vir[(size_t)n + i] += v1;
                vir[(size_t)2 * n + i] += v2;
                vir[(size_t)3 * n + i] += v3;
                vir[(size_t)4 * n + i] += v4;
                vir[(size_t)5 * n + i] += v5;
            }
        }
    }
}

template <bool NEED_ENERGY, bool NEED_VIRIAL>
__global__ void __launch_bounds__(256) k_lj_direct(
    int n, const snb_atom_group* __restrict__ nl, const float4* __restrict__ atoms,
    const int* __restrict__ type, const float* __restrict__ lj_a,
    const float* __restrict__ lj_b, const float4* __restrict__ coul_tab, float cscale,
    SnbBox box, float rc2, float beta,
    int64_t* __restrict__ fx, int64_t* __restrict__ e_atom, int64_t* __restrict__ vir)
{
    k_lj_direct_body<NEED_ENERGY, NEED_VIRIAL>(
        n, nl, atoms, type, lj_a, lj_b, coul_tab, cscale, box, rc2, beta, fx, e_atom, vir,
        blockIdx.x, gridDim.x);
}

struct LjDirectArgs
{
    int n;
    const snb_atom_group* nl;
    const float4* atoms;
    const int* type;
    const float* lj_a;
    const float* lj_b;
    const float4* coul_tab;
    float cscale;
    SnbBox box;
    float rc2;
    float beta;
    int64_t* fx;
    int64_t* e_atom;
    int64_t* vir;
};

template <bool NEED_ENERGY, bool NEED_VIRIAL>
__global__ void __launch_bounds__(256) k_lj_direct_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const LjDirectArgs& a = snb_seg<LjDirectArgs>(t, bid, nbid);
    k_lj_direct_body<NEED_ENERGY, NEED_VIRIAL>(
        a.n, a.nl, a.atoms, a.type, a.lj_a, a.lj_b, a.coul_tab, a.cscale, a.box, a.rc2, a.beta,
        a.fx, a.e_atom, a.vir, bid, nbid);
}

// Force-only steps of the row kernel for small systems, on request: every
// atom's force accumulators in LDS (3 x n int64, n <= SNB_LJ_LDS_MAX), each workgroup a
// run of SNB_LJ_LDS_ROWS consecutive rows, and one global add per nonzero
// sum at the end.  The same integer sums as the global atomics of
// k_lj_direct, with about a quarter of the global atomics: where several
// small systems share the device (a step batch), the atomics' throughput,
// not their latency, bounds the row kernel.
#define SNB_LJ_LDS_MAX 2560
#define SNB_LJ_LDS_ROWS 64
__device__ __forceinline__ void k_lj_lds_body(
    int n, const snb_atom_group* __restrict__ nl, const float4* __restrict__ atoms,
    const int* __restrict__ type, const float* __restrict__ lj_a,
    const float* __restrict__ lj_b, const float4* __restrict__ coul_tab, float cscale,
    SnbBox box, float rc2, float beta, int64_t* __restrict__ fx, unsigned bid, unsigned nbid)
{
    extern __shared__ long long acc[];  // [3][n]
    for (int t = threadIdx.x; t < 3 * n; t += blockDim.x) acc[t] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
    const int r0 = (int)bid * SNB_LJ_LDS_ROWS;
    const int r1 = r0 + SNB_LJ_LDS_ROWS < n ? r0 + SNB_LJ_LDS_ROWS : n;
    for (int i = r0 + wave; i < r1; i += nwave)
    {
        const snb_atom_group g = nl[i];
        const float4 ai = atoms[i];
        const int ti = type[i];
        int64_t sx = 0, sy = 0, sz = 0;
        for (int k = lane; k < g.atom_numbers; k += 64)
        {
            const int j = g.atom_serial[k];
            const float4 aj = atoms[j];
            float dx = aj.x - ai.x, dy = aj.y - ai.y, dz = aj.z - ai.z;
            pbc_disp(dx, dy, dz, box);
            float r2 = (dx * dx + dy * dy) + dz * dz;
            if (!(r2 < rc2)) continue;
            const int p = snb_lj_pair_index(ti, type[j]);
            const float fa =
                pair_force_factor(r2, lj_a[p], lj_b[p], ai.w * aj.w, beta, cscale, coul_tab);
            const int64_t ix = snb_to_fixed(fa * dx), iy = snb_to_fixed(fa * dy),
                          iz = snb_to_fixed(fa * dz);
            sx += ix;
            sy += iy;
            sz += iz;
            atomicAdd((unsigned long long*)&acc[j], (unsigned long long)(-ix));
            atomicAdd((unsigned long long*)&acc[n + j], (unsigned long long)(-iy));
            atomicAdd((unsigned long long*)&acc[2 * n + j], (unsigned long long)(-iz));
        }
        sx = wave_sum(sx);
        sy = wave_sum(sy);
        sz = wave_sum(sz);
        if (lane == 0)
        {
            atomicAdd((unsigned long long*)&acc[i], (unsigned long long)sx);
            atomicAdd((unsigned long long*)&acc[n + i], (unsigned long long)sy);
            atomicAdd((unsigned long long*)&acc[2 * n + i], (unsigned long long)sz);
        }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < n; t += blockDim.x)
    {
        const long long vx = acc[t], vy = acc[n + t], vz = acc[2 * n + t];
        if (vx) atomic_add_i64(fx + t, vx);
        if (vy) atomic_add_i64(fx + n + t, vy);
        if (vz) atomic_add_i64(fx + 2 * n + t, vz);
    }
}

__global__ void __launch_bounds__(1024) k_lj_lds(
    int n, const snb_atom_group* __restrict__ nl, const float4* __restrict__ atoms,
    const int* __restrict__ type, const float* __restrict__ lj_a,
    const float* __restrict__ lj_b, const float4* __restrict__ coul_tab, float cscale,
    SnbBox box, float rc2, float beta, int64_t* __restrict__ fx)
{
    k_lj_lds_body(n, nl, atoms, type, lj_a, lj_b, coul_tab, cscale, box, rc2, beta, fx,
                  blockIdx.x, gridDim.x);
}

struct LjLdsArgs
{
    int n;
    const snb_atom_group* nl;
    const float4* atoms;
    const int* type;
    const float* lj_a;
    const float* lj_b;
    const float4* coul_tab;
    float cscale;
    SnbBox box;
    float rc2;
    float beta;
    int64_t* fx;
};

__global__ void __launch_bounds__(1024) k_lj_lds_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const LjLdsArgs& a = snb_seg<LjLdsArgs>(t, bid, nbid);
    k_lj_lds_body(a.n, a.nl, a.atoms, a.type, a.lj_a, a.lj_b, a.coul_tab, a.cscale, a.box,
                  a.rc2, a.beta, a.fx, bid, nbid);
}

// Force-only steps of the row kernel for small systems over the list in both
// directions: a workgroup per atom i sums the pairs of all its neighbours, those
// of lower ids with the displacement and sign of their own row's entry, so the
// terms are the ones that k_lj_direct rounds and scatters, each evaluated on
// both sides.  Twice the pair math (230 k pairs at 1,500 atoms: under 1 us of
// the device) for none of its three 64-bit global atomics per pair, whose
// throughput (about 31 per ns) is what bounds k_lj_direct.  Reads the caller's coordinates and
// charges and the square parameter table: no packing kernel precedes it.  At
// 1,500 atoms 25.4 us and 2 for packing -> 5.3 us, in a triclinic cell of 7,200
// 60 with packing -> 16.
// A list with rows cut at max_nb (*cut) is taken in one direction with the
// atomics, as k_lj_direct takes it.
__device__ __forceinline__ void k_lj_full_body(
    int n, const snb_atom_group* __restrict__ nl, const uint16_t* __restrict__ lo_rows,
    const int* __restrict__ lo_count, const snb_vector* __restrict__ crd,
    const float* __restrict__ charge, const int* __restrict__ type,
    const float2* __restrict__ ab2, int ntypes, const float4* __restrict__ coul_tab, float cscale,
    const SnbBox& box, float rc2, float beta, int64_t* __restrict__ fx,
    const int* __restrict__ cut, int* __restrict__ status, unsigned bid)
{
    __shared__ float4 ctab[SNB_COUL_N];
    __shared__ unsigned long long sum[3];
    const int i = uni(bid), tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
    const snb_atom_group g = nl[i];
    const int lo_n = lo_count[i];
    const bool both = *cut == 0;
    const snb_vector ri = crd[i];
    const float qi2 = charge[i] * 4294967296.0f;  // 2^32 fixed-point scale
    const float2* abrow = ab2 + (size_t)type[i] * ntypes;
    const uint16_t* lo_row = lo_rows + (size_t)i * n;
    ctab[tid] = coul_tab[tid];
    if (tid < 3) sum[tid] = 0;
    if (tid == 0 &&
        !(__builtin_isfinite(ri.x) && __builtin_isfinite(ri.y) && __builtin_isfinite(ri.z)))
        atomicOr(status, SNB_FLAG_NONFINITE_CRD);
    __syncthreads();
    const int hi_n = g.atom_numbers, cnt = hi_n + (both ? lo_n : 0);
    int64_t sx = 0, sy = 0, sz = 0;
    for (int k0 = wave * 128; k0 < cnt; k0 += 512)
    {
        int jj[2];
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            const int k = k0 + 64 * h + lane;
            jj[h] = k < hi_n ? g.atom_serial[k] : (k < cnt ? (int)lo_row[k - hi_n] : i);
        }
        snb_vector rj[2];
        float qj[2];
        int tj[2];
        float2 AB[2];
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            rj[h] = crd[jj[h]];
            qj[h] = charge[jj[h]];
            tj[h] = type[jj[h]];
        }
#pragma unroll
        for (int h = 0; h < 2; h++) AB[h] = abrow[tj[h]];
#pragma unroll
        for (int h = 0; h < 2; h++)
        {
            const int j = jj[h];
            float dx = rj[h].x - ri.x, dy = rj[h].y - ri.y, dz = rj[h].z - ri.z;
            // the row of the lower id takes the displacement from it to the other
            const bool lo = j < i;
            if (lo)
            {
                dx = -dx;
                dy = -dy;
                dz = -dz;
            }
            pbc_disp(dx, dy, dz, box);
            const float r2 = (dx * dx + dy * dy) + dz * dz;
            if (j == i || !(r2 < rc2)) continue;
            const float fa2 =
                pair_force_factor(r2, AB[h].x, AB[h].y, qi2 * qj[h], beta, cscale, ctab);
            const int64_t ix = snb_fixed_from_scaled(fa2 * dx),
                          iy = snb_fixed_from_scaled(fa2 * dy),
                          iz = snb_fixed_from_scaled(fa2 * dz);
            const int64_t m = lo ? -1 : 0;  // the higher id's force: the negated integers
            sx += (ix ^ m) - m;
            sy += (iy ^ m) - m;
            sz += (iz ^ m) - m;
            if (!both)
            {
                atomic_add_i64(fx + j, -ix);
                atomic_add_i64(fx + n + j, -iy);
                atomic_add_i64(fx + 2 * n + j, -iz);
            }
        }
    }
    if (wave * 128 < cnt)
    {
        const int64_t v = wave_sum3(sx, sy, sz);
        if ((lane & 15) == 0 && lane < 48)
            atomicAdd(&sum[lane == 0 ? 0 : (lane == 32 ? 1 : 2)], (unsigned long long)v);
    }
    __syncthreads();
    if (tid < 3) atomic_add_i64(fx + (size_t)tid * n + i, (int64_t)sum[tid]);
}

__global__ void __launch_bounds__(256) k_lj_full(
    int n, const snb_atom_group* __restrict__ nl, const uint16_t* __restrict__ lo_rows,
    const int* __restrict__ lo_count, const snb_vector* __restrict__ crd,
    const float* __restrict__ charge, const int* __restrict__ type,
    const float2* __restrict__ ab2, int ntypes, const float4* __restrict__ coul_tab, float cscale,
    SnbBox box, float rc2, float beta, int64_t* __restrict__ fx, const int* __restrict__ cut,
    int* __restrict__ status)
{
    k_lj_full_body(n, nl, lo_rows, lo_count, crd, charge, type, ab2, ntypes, coul_tab, cscale, box,
                   rc2, beta, fx, cut, status, blockIdx.x);
}

struct LjFullArgs
{
    int n;
    const snb_atom_group* nl;
    const uint16_t* lo_rows;
    const int* lo_count;
    const snb_vector* crd;
    const float* charge;
    const int* type;
    const float2* ab2;
    int ntypes;
    const float4* coul_tab;
    float cscale;
    SnbBox box;
    float rc2;
    float beta;
    int64_t* fx;
    const int* cut;
    int* status;
};

__global__ void __launch_bounds__(256) k_lj_full_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const LjFullArgs& a = snb_seg<LjFullArgs>(t, bid, nbid);
    k_lj_full_body(a.n, a.nl, a.lo_rows, a.lo_count, a.crd, a.charge, a.type, a.ab2, a.ntypes,
                   a.coul_tab, a.cscale, a.box, a.rc2, a.beta, a.fx, a.cut, a.status, bid);
}

int snb_launch_lj_direct(snb_context* ctx, const snb_atom_group* nl, const snb_vector* crd,
                         const float* charge, const SnbBox& box, float beta, int need_energy,
                         int need_virial)
{
    int n = ctx->n;
    if (n <= 0) return SNB_OK;
    float rc2 = ctx->lj.cutoff * ctx->lj.cutoff;
    const int row_mode = ctx->lj.row_lds;
    const bool force_only = !need_energy && !need_virial;
    // both directions: the library's own list, kept that way by its rebuild
    const SnbNl& L = ctx->nl;
    if (force_only && row_mode < 0 && L.init && L.built && !L.windowed && L.lo_rows && nl == L.dnl)
    {
        snb_prof_begin(ctx, SNB_PROF_PAIR);
        if (snb_rec) snb_rec->weight_next = (double)n;
        SNB_LAUNCH_B(k_lj_full, k_lj_full_batch, LjFullArgs, dim3(n), dim3(256), 0, ctx->stream, n,
                     nl, L.lo_rows, L.lo_count, crd, charge, ctx->type, ctx->lj.ab2,
                     ctx->lj.ntypes, ctx->lj.coul, ctx->lj.coul_scale, box, rc2, beta, ctx->fx,
                     L.cell_count + L.ncell, ctx->status);
        snb_prof_end(ctx, SNB_PROF_PAIR);
        SNB_CHECK(hipGetLastError());
        return SNB_OK;
    }
    int rc = snb_launch_pack_atoms(ctx, crd, charge);
    if (rc) return rc;
    // LDS accumulators: on request, or for another list in a recorded step batch
    if (force_only && n <= SNB_LJ_LDS_MAX && (row_mode > 0 || (row_mode < 0 && snb_rec)))
    {
        snb_prof_begin(ctx, SNB_PROF_PAIR);
        SNB_LAUNCH_B(k_lj_lds, k_lj_lds_batch, LjLdsArgs,
                     dim3((n + SNB_LJ_LDS_ROWS - 1) / SNB_LJ_LDS_ROWS), dim3(1024),
                     sizeof(long long) * 3 * (size_t)n, ctx->stream, n, nl, ctx->atom4,
                     ctx->type, ctx->lj.a, ctx->lj.b, ctx->lj.coul, ctx->lj.coul_scale, box, rc2,
                     beta, ctx->fx);
        snb_prof_end(ctx, SNB_PROF_PAIR);
        SNB_CHECK(hipGetLastError());
        return SNB_OK;
    }
    int blocks = (n + 3) / 4;
    if (blocks > 65535 * 4) blocks = 65535 * 4;
    snb_prof_begin(ctx, SNB_PROF_PAIR);
#define SNB_LJ_LAUNCH(E, V)                                                                   \
    SNB_LAUNCH_B((k_lj_direct<E, V>), (k_lj_direct_batch<E, V>), LjDirectArgs, dim3(blocks),   \
                 dim3(256), 0, ctx->stream, n, nl, ctx->atom4, ctx->type, ctx->lj.a, ctx->lj.b, \
                 ctx->lj.coul, ctx->lj.coul_scale, box, rc2, beta, ctx->fx, ctx->e_atom,        \
                 ctx->vir_atom)
    if (need_energy && need_virial)
        SNB_LJ_LAUNCH(true, true);
    else if (need_energy)
        SNB_LJ_LAUNCH(true, false);
    else if (need_virial)
        SNB_LJ_LAUNCH(false, true);
    else
        SNB_LJ_LAUNCH(false, false);
#undef SNB_LJ_LAUNCH
    snb_prof_end(ctx, SNB_PROF_PAIR);
    SNB_CHECK(hipGetLastError());
    return SNB_OK;
}

// MPI_PME_Excluded_Force_With_Atom_Energy_Correction (PM_force.cpp:1743-1814)
// with exclude_factor 1: for j in excl(i), f = qq (erf(x) - 2x/sqrt(pi)
// e^{-x^2}) r^-3 dr on i and -f on j, energy -qq erf(x)/r and virial to i,
// evaluated in FP64.  One thread per atom i; i-sums in registers, j-terms by
// integer atomics (a few per atom).
template <bool NEED_ENERGY, bool NEED_VIRIAL>
__device__ __forceinline__ void k_excl_body(int n, const snb_vector* __restrict__ crd,
                                              const float* __restrict__ charge,
                                              SnbBox box, float beta,
                                              const int* __restrict__ ex_start,
                                              const int* __restrict__ ex_list,
                                              const int* __restrict__ ex_num,
                                              int64_t* __restrict__ fx,
                                              int64_t* __restrict__ e_atom,
                                              int64_t* __restrict__ vir,
    unsigned bid, unsigned nbid)
{
    int i = bid * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int cnt = ex_num[i];
    if (cnt <= 0) return;
    int s0 = ex_start[i];
    const snb_vector ri = crd[i];
    const float4 ai = make_float4(ri.x, ri.y, ri.z, charge[i]);
    int64_t sx = 0, sy = 0, sz = 0, e = 0;
    int64_t v0 = 0, v1 = 0, v2 = 0, v3 = 0, v4 = 0, v5 = 0;
    for (int k = s0; k < s0 + cnt; k++)
    {
        int j = ex_list[k];
        const snb_vector rj = crd[j];
        const float4 aj = make_float4(rj.x, rj.y, rj.z, charge[j]);
        float dx = aj.x - ai.x, dy = aj.y - ai.y, dz = aj.z - ai.z;
        pbc_disp(dx, dy, dz, box);
        // FP64 from the float displacement: the erf part of an excluded pair is
        // a small difference of large terms in float arithmetic
        double ddx = dx, ddy = dy, ddz = dz;
        double r2d = (ddx * ddx + ddy * ddy) + ddz * ddz;
        double rd = __builtin_sqrt(r2d);
        double rid = 1.0 / rd;
        double gd;
        const double erfd = 1.0 - snb_erfc_parts_d((double)beta * rd, &gd);
        const double hd = erfd - gd;
        double qq = (double)ai.w * (double)aj.w;
        double fa = (qq * hd) * ((rid * rid) * rid);
        double fxv = fa * ddx, fyv = fa * ddy, fzv = fa * ddz;
        int64_t ix = snb_to_fixed_d(fxv), iy = snb_to_fixed_d(fyv), iz = snb_to_fixed_d(fzv);
        sx += ix;
        sy += iy;
        sz += iz;
        atomic_add_i64(fx + j, -ix);
        atomic_add_i64(fx + n + j, -iy);
        atomic_add_i64(fx + 2 * n + j, -iz);
        if (NEED_ENERGY) e += snb_to_fixed_d(-((qq * erfd) * rid));
        if (NEED_VIRIAL)
        {
            v0 += snb_to_fixed_d(-(fxv * ddx));
            v1 += snb_to_fixed_d(-(fxv * ddy + fyv * ddx));
            v2 += snb_to_fixed_d(-(fyv * ddy));
            v3 += snb_to_fixed_d(-(fxv * ddz + fzv * ddx));
            v4 += snb_to_fixed_d(-(fyv * ddz + fzv * ddy));
            v5 += snb_to_fixed_d(-(fzv * ddz));
        }
    }
    atomic_add_i64(fx + i, sx);
    atomic_add_i64(fx + n + i, sy);
    atomic_add_i64(fx + 2 * n + i, sz);
    if (NEED_ENERGY) e_atom[(size_t)2 * n + i] += e;
    if (NEED_VIRIAL)
    {
        vir[i] += v0;
        vir[(size_t)n + i] += v1;
        vir[(size_t)2 * n + i] += v2;
        vir[(size_t)3 * n + i] += v3;
        vir[(size_t)4 * n + i] += v4;
        vir[(size_t)5 * n + i] += v5;
    }
}

template <bool NEED_ENERGY, bool NEED_VIRIAL>
__global__ void __launch_bounds__(256) k_excl(int n, const snb_vector* __restrict__ crd,
                                              const float* __restrict__ charge,
                                              SnbBox box, float beta,
                                              const int* __restrict__ ex_start,
                                              const int* __restrict__ ex_list,
                                              const int* __restrict__ ex_num,
                                              int64_t* __restrict__ fx,
                                              int64_t* __restrict__ e_atom,
                                              int64_t* __restrict__ vir)
{
    k_excl_body<NEED_ENERGY, NEED_VIRIAL>(
        n, crd, charge, box, beta, ex_start, ex_list, ex_num, fx, e_atom, vir, blockIdx.x,
        gridDim.x);
}

struct ExclArgs
{
    int n;
    const snb_vector* crd;
    const float* charge;
    SnbBox box;
    float beta;
    const int* ex_start;
    const int* ex_list;
    const int* ex_num;
    int64_t* fx;
    int64_t* e_atom;
    int64_t* vir;
};

template <bool NEED_ENERGY, bool NEED_VIRIAL>
__global__ void __launch_bounds__(256) k_excl_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const ExclArgs& a = snb_seg<ExclArgs>(t, bid, nbid);
    k_excl_body<NEED_ENERGY, NEED_VIRIAL>(
        a.n, a.crd, a.charge, a.box, a.beta, a.ex_start, a.ex_list, a.ex_num, a.fx, a.e_atom, a.vir,
        bid, nbid);
}

int snb_launch_excl_to(hipStream_t s, int n, const snb_vector* crd, const float* charge,
                       const SnbBox& box, float beta, const int* ex_start, const int* ex_list,
                       const int* ex_num, int need_energy, int need_virial, int64_t* fx,
                       int64_t* e_atom, int64_t* vir)
{
    if (n <= 0) return SNB_OK;
    dim3 g((n + 255) / 256);
#define SNB_EX_LAUNCH(E, V)                                                                  \
    SNB_LAUNCH_B((k_excl<E, V>), (k_excl_batch<E, V>), ExclArgs, g, dim3(256), 0, s, n, crd, \
                 charge, box, beta, ex_start, ex_list, ex_num, fx, e_atom, vir)
    if (need_energy && need_virial)
        SNB_EX_LAUNCH(true, true);
    else if (need_energy)
        SNB_EX_LAUNCH(true, false);
    else if (need_virial)
        SNB_EX_LAUNCH(false, true);
    else
        SNB_EX_LAUNCH(false, false);
#undef SNB_EX_LAUNCH
    SNB_CHECK(hipGetLastError());
    return SNB_OK;
}

int snb_launch_excl(snb_context* ctx, const snb_vector* crd, const float* charge,
                    const SnbBox& box, float beta,
                    const int* ex_start, const int* ex_list, const int* ex_num,
                    int need_energy, int need_virial, int64_t* fx)
{
    if (ctx->n <= 0) return SNB_OK;
    snb_prof_begin(ctx, SNB_PROF_EXCL);
    int rc = snb_launch_excl_to(ctx->stream, ctx->n, crd, charge, box, beta, ex_start, ex_list,
                                ex_num, need_energy, need_virial, fx, ctx->e_atom,
                                ctx->vir_atom);
    snb_prof_end(ctx, SNB_PROF_EXCL);
    return rc;
}

// Scaled 1-4 LJ and plain Coulomb of the 1-4 pairs (stands in for
// Dihedral_14_LJ_CF_Force_With_Atom_Energy_And_Virial_Device, nb14.cpp:7-100).
// One thread per pair.  The force is float, in the reference's operation
// order: dr = pbc(r_b - r_a), 1/r^2 and 1/r as a double quotient rounded to
// float, charges below 1e-10 in magnitude raised to 1e-10, f = -A r^-14 +
// B r^-8 - cf qa qb r^-3; +f dr on a and -f dr on b, rounded to fixed point.
// Energies in FP64 from the float displacement with the reference's
// constants (cf qa qb / r and 0.08333333 A r^-12 - 0.1666666 B r^-6), kept
// per pair and added to atom a; the virial -f dr (x) dr goes to atom a.
// 1/r uses sqrtf (correctly rounded) where the reference takes norm3df.
template <bool NEED_ENERGY, bool NEED_VIRIAL>
__global__ void __launch_bounds__(256) k_nb14(int m, int n, const int* __restrict__ a14,
                                              const int* __restrict__ b14,
                                              const float* __restrict__ A14,
                                              const float* __restrict__ B14,
                                              const float* __restrict__ cf14,
                                              const snb_vector* __restrict__ crd,
                                              const float* __restrict__ charge, SnbBox box,
                                              int64_t* __restrict__ fx,
                                              int64_t* __restrict__ e_nb14,
                                              int64_t* __restrict__ pair_e,
                                              int64_t* __restrict__ vir)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m) return;
    const int i = a14[k], j = b14[k];
    const snb_vector ri = crd[i], rj = crd[j];
    float dx = rj.x - ri.x, dy = rj.y - ri.y, dz = rj.z - ri.z;
    pbc_disp(dx, dy, dz, box);
    const float dr2 = (dx * dx + dy * dy) + dz * dz;
    const float dr_2 = (float)(1.0 / (double)dr2);
    const float dr_4 = dr_2 * dr_2;
    const float dr_8 = dr_4 * dr_4;
    const float dr_14 = (dr_8 * dr_4) * dr_2;
    const float dr_1 = (float)(1.0 / (double)sqrtf(dr2));
    float qi = charge[i], qj = charge[j];
    if ((double)fabsf(qi) < 1e-10) qi = (float)1e-10;
    if ((double)fabsf(qj) < 1e-10) qj = (float)1e-10;
    const float A = A14[k], B = B14[k], cf = cf14[k];
    const float fcf = ((-((cf * dr_2) * dr_1)) * qi) * qj;
    const float flj = (-A) * dr_14 + B * dr_8;
    const float f = flj + fcf;
    const float fxv = f * dx, fyv = f * dy, fzv = f * dz;
    const int64_t ix = snb_to_fixed(fxv), iy = snb_to_fixed(fyv), iz = snb_to_fixed(fzv);
    atomic_add_i64(fx + i, ix);
    atomic_add_i64(fx + n + i, iy);
    atomic_add_i64(fx + 2 * n + i, iz);
    atomic_add_i64(fx + j, -ix);
    atomic_add_i64(fx + n + j, -iy);
    atomic_add_i64(fx + 2 * n + j, -iz);
    if (NEED_ENERGY)
    {
        const double ddx = dx, ddy = dy, ddz = dz;
        const double r2d = (ddx * ddx + ddy * ddy) + ddz * ddz;
        const double d1 = 1.0 / __builtin_sqrt(r2d);
        const double d2 = 1.0 / r2d;
        const double d4 = d2 * d2, d8 = d4 * d4;
        const int64_t pc = snb_to_fixed_d((((double)cf * d1) * (double)qi) * (double)qj);
        const int64_t pl = snb_to_fixed_d(((0.08333333 * (double)A) * d4) * d8 -
                                          ((0.1666666 * (double)B) * d4) * d2);
        pair_e[k] = pl;
        pair_e[m + k] = pc;
        atomic_add_i64(e_nb14 + i, pl + pc);
    }
    if (NEED_VIRIAL)
    {
        atomic_add_i64(vir + i, snb_to_fixed(-(fxv * dx)));
        atomic_add_i64(vir + (size_t)n + i, snb_to_fixed(-(fxv * dy + fyv * dx)));
        atomic_add_i64(vir + (size_t)2 * n + i, snb_to_fixed(-(fyv * dy)));
        atomic_add_i64(vir + (size_t)3 * n + i, snb_to_fixed(-(fxv * dz + fzv * dx)));
        atomic_add_i64(vir + (size_t)4 * n + i, snb_to_fixed(-(fyv * dz + fzv * dy)));
        atomic_add_i64(vir + (size_t)5 * n + i, snb_to_fixed(-(fzv * dz)));
    }
}

int snb_launch_nb14(snb_context* ctx, const snb_vector* crd, const float* charge,
                    const SnbBox& box, int need_energy, int need_virial, int64_t* fx)
{
    const SnbNb14& M = ctx->nb14;
    const int m = M.count, n = ctx->n;
    if (m <= 0) return SNB_OK;
    dim3 g((m + 255) / 256);
#define SNB_NB14_LAUNCH(E, V)                                                                \
    SNB_LAUNCH((k_nb14<E, V>), g, dim3(256), 0, ctx->stream, m, n, M.a, M.b, M.A, M.B, \
                       M.cf, crd, charge, box, fx, ctx->e_atom + 3 * (size_t)n, M.pair_e,      \
                       ctx->vir_atom)
    if (need_energy && need_virial)
        SNB_NB14_LAUNCH(true, true);
    else if (need_energy)
        SNB_NB14_LAUNCH(true, false);
    else if (need_virial)
        SNB_NB14_LAUNCH(false, true);
    else
        SNB_NB14_LAUNCH(false, false);
#undef SNB_NB14_LAUNCH
    SNB_CHECK(hipGetLastError());
    return SNB_OK;
}

// Harmonic bonds (stands in for Bond_Force_With_Atom_Energy_And_Virial_Device,
// bond/bond.cpp:15-64): dr = pbc(r_a - r_b), r = |dr| (sqrtf, where the
// reference calls norm3df), f = -(2 k (r - r0)) / r * dr on a and -f on b in
// the reference's float order, fixed point; the energy k (r - r0)^2 in FP64
// from the float displacement, kept per bond and added to atom a; the virial
// f (x) dr to atom a.
template <bool NEED_ENERGY, bool NEED_VIRIAL>
__global__ void __launch_bounds__(256) k_bond(int m, int n, const int* __restrict__ ba,
                                              const int* __restrict__ bb,
                                              const float* __restrict__ bk,
                                              const float* __restrict__ br0,
                                              const snb_vector* __restrict__ crd, SnbBox box,
                                              int64_t* __restrict__ fx,
                                              int64_t* __restrict__ e_bond,
                                              int64_t* __restrict__ pair_e,
                                              int64_t* __restrict__ vir)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= m) return;
    const int i = ba[k], j = bb[k];
    const snb_vector ri = crd[i], rj = crd[j];
    float dx = ri.x - rj.x, dy = ri.y - rj.y, dz = ri.z - rj.z;
    pbc_disp(dx, dy, dz, box);
    const float r = sqrtf((dx * dx + dy * dy) + dz * dz);
    const float kk = bk[k], r0 = br0[k];
    const float d = r - r0;
    const float g = (2.0f * d) * kk;
    const float s = (-g) / r;
    const float fxv = s * dx, fyv = s * dy, fzv = s * dz;
    const int64_t ix = snb_to_fixed(fxv), iy = snb_to_fixed(fyv), iz = snb_to_fixed(fzv);
    atomic_add_i64(fx + i, ix);
    atomic_add_i64(fx + n + i, iy);
    atomic_add_i64(fx + 2 * n + i, iz);
    atomic_add_i64(fx + j, -ix);
    atomic_add_i64(fx + n + j, -iy);
    atomic_add_i64(fx + 2 * n + j, -iz);
    if (NEED_ENERGY)
    {
        const double ddx = dx, ddy = dy, ddz = dz;
        const double dd = __builtin_sqrt((ddx * ddx + ddy * ddy) + ddz * ddz) - (double)r0;
        const int64_t pe = snb_to_fixed_d(((double)kk * dd) * dd);
        pair_e[k] = pe;
        atomic_add_i64(e_bond + i, pe);
    }
    if (NEED_VIRIAL)
    {
        atomic_add_i64(vir + i, snb_to_fixed(fxv * dx));
        atomic_add_i64(vir + (size_t)n + i, snb_to_fixed(fxv * dy + fyv * dx));
        atomic_add_i64(vir + (size_t)2 * n + i, snb_to_fixed(fyv * dy));
        atomic_add_i64(vir + (size_t)3 * n + i, snb_to_fixed(fxv * dz + fzv * dx));
        atomic_add_i64(vir + (size_t)4 * n + i, snb_to_fixed(fyv * dz + fzv * dy));
        atomic_add_i64(vir + (size_t)5 * n + i, snb_to_fixed(fzv * dz));
    }
}

int snb_launch_bond(snb_context* ctx, const snb_vector* crd, const SnbBox& box, int need_energy,
                    int need_virial, int64_t* fx)
{
    const SnbBond& M = ctx->bond;
    const int m = M.count, n = ctx->n;
    if (m <= 0) return SNB_OK;
    dim3 g((m + 255) / 256);
#define SNB_BOND_LAUNCH(E, V)                                                               \
    SNB_LAUNCH((k_bond<E, V>), g, dim3(256), 0, ctx->stream, m, n, M.a, M.b, M.k,    \
                       M.r0, crd, box, fx, ctx->e_atom + 4 * (size_t)n, M.pair_e,            \
                       ctx->vir_atom)
    if (need_energy && need_virial)
        SNB_BOND_LAUNCH(true, true);
    else if (need_energy)
        SNB_BOND_LAUNCH(true, false);
    else if (need_virial)
        SNB_BOND_LAUNCH(false, true);
    else
        SNB_BOND_LAUNCH(false, false);
#undef SNB_BOND_LAUNCH
    SNB_CHECK(hipGetLastError());
    return SNB_OK;
}

// ---------------------------------------------------------------------------
// windowed path
// ---------------------------------------------------------------------------
// Packs coordinates and charges in sorted (cell) order: satom[s] = (crd, q) of
// atom order[s]; raises the non-finite flag.
__device__ __forceinline__ void k_pack_sorted_body(int n, const int* __restrict__ order,
                              const snb_vector* __restrict__ crd, const float* __restrict__ charge,
                              float4* __restrict__ satom, int* __restrict__ status,
    unsigned bid, unsigned nbid)
{
    int s = bid * blockDim.x + threadIdx.x;
    if (s >= n) return;
    int id = order[s];
    snb_vector r = crd[id];
    satom[s] = make_float4(r.x, r.y, r.z, charge[id]);
    if (!(__builtin_isfinite(r.x) && __builtin_isfinite(r.y) && __builtin_isfinite(r.z)))
        atomicOr(status, SNB_FLAG_NONFINITE_CRD);
}

__global__ void k_pack_sorted(int n, const int* __restrict__ order,
                              const snb_vector* __restrict__ crd, const float* __restrict__ charge,
                              float4* __restrict__ satom, int* __restrict__ status)
{
    k_pack_sorted_body(n, order, crd, charge, satom, status, blockIdx.x, gridDim.x);
}

struct PackSortedArgs
{
    int n;
    const int* order;
    const snb_vector* crd;
    const float* charge;
    float4* satom;
    int* status;
};

__global__ void k_pack_sorted_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const PackSortedArgs& a = snb_seg<PackSortedArgs>(t, bid, nbid);
    k_pack_sorted_body(a.n, a.order, a.crd, a.charge, a.satom, a.status, bid, nbid);
}

// One workgroup per block of a x b columns x S z-cells (snb_window.h).  The
// workgroup keeps int64 force accumulators for every atom of its window in
// LDS; a wavefront evaluates one row at a time (64 lanes over its entries,
// two entries per lane in flight so the gathers of one overlap the other),
// adds -f to the j slot (ds_add_u64) and, after a wave reduction, +sum f to
// the row's own slot.  At the end the accumulators go to the stage buffer;
// k_stage_gather sums each atom's stage entries.  Windows larger than the LDS
// capacity fall back to integer atomics on the global accumulators.
// Per-atom energies and virials go, as in the reference, to the lower atom id
// of the pair: row-owner sums when the owner is the lower id, otherwise
// integer atomics on the j atom's entry of the sorted-order arrays (the j
// atoms of one row lie in a few neighbouring cells, so a wavefront's adds
// fall on few cache lines); k_stage_gather moves the sorted-order sums to the
// id-ordered arrays.  With ref_attr == 0 every pair's terms stay with the row
// owner.

// Periodic displacement.  ORTHO (diagonal cell) drops the off-diagonal terms
// and takes k = rint(s) for floor(s + 0.5).  For every pair that can reach
// the cutoff this is the reference's arithmetic bit for bit: s lies within
// rc / L < 1/2 of an integer there, so both give the same k.  The two differ
// only for s within an ulp of a half-integer, i.e. for pairs half a box
// length apart, which are beyond the cutoff either way.
template <bool ORTHO>
__device__ __forceinline__ void win_disp(float& dx, float& dy, float& dz, const SnbBox& box)
{
    if (ORTHO)
    {
        const float kx = rintf(dx * box.rc[0]);
        const float ky = rintf(dy * box.rc[2]);
        const float kz = rintf(dz * box.rc[5]);
        dx = dx - kx * box.c[0];
        dy = dy - ky * box.c[2];
        dz = dz - kz * box.c[5];
    }
    else
        pbc_disp(dx, dy, dz, box);
}

// adds to the accumulators of a window slot (x, y, z side by side: one address
// and two offsets)
__device__ __forceinline__ void lds_add3(long long* acc, int slot, int64_t x, int64_t y, int64_t z)
{
    unsigned long long* a =
        (unsigned long long*)((char*)acc + __umul24((unsigned)slot, 24u));
    atomicAdd(a, (unsigned long long)x);
    atomicAdd(a + 1, (unsigned long long)y);
    atomicAdd(a + 2, (unsigned long long)z);
}

struct WinRowSums
{
    int64_t sx, sy, sz, elj, ec, v0, v1, v2, v3, v4, v5;
};

// Everything one in-cutoff pair contributes: f (force on the row atom i) to
// the register sums, the j share to the j accumulator, the row owner's share
// of energy/virial to the register sums.  A2, B2 and qi2 carry the 2^32
// fixed-point scale (exact power-of-two scaling), so f comes out scaled and
// its conversion is one double add.  The LDS accumulators hold the negated
// force (j receives +f, the row atom -sum f at the row's end), which saves
// the 64-bit negation per pair; the global arrays of the overflow mode hold
// the force itself.
template <bool NEED_ENERGY, bool NEED_VIRIAL>
__device__ __forceinline__ void win_pair(WinRowSums& S, float dx, float dy, float dz, float r2,
                                         float A2, float B2, float qi2, float qj, float beta,
                                         float cscale, const float4* ctab,
                                         int slot, int sj, bool ov, long long* acc,
                                         int n, const int* __restrict__ order,
                                         int64_t* __restrict__ fx, int ref_attr, int id_i,
                                         int64_t* __restrict__ e_sorted,
                                         int64_t* __restrict__ v_sorted)
{
    const float fa2 = pair_force_factor(r2, A2, B2, qi2 * qj, beta, cscale, ctab);
    const float fx2 = fa2 * dx, fy2 = fa2 * dy, fz2 = fa2 * dz;
    int64_t ix = snb_fixed_from_scaled(fx2), iy = snb_fixed_from_scaled(fy2),
            iz = snb_fixed_from_scaled(fz2);
    S.sx += ix;
    S.sy += iy;
    S.sz += iz;
    if (!ov)
    {
        lds_add3(acc, slot, ix, iy, iz);
    }
    else
    {
        int idj = order[sj];
        atomic_add_i64(fx + idj, -ix);
        atomic_add_i64(fx + n + idj, -iy);
        atomic_add_i64(fx + 2 * n + idj, -iz);
    }
    if (NEED_ENERGY || NEED_VIRIAL)
    {
        // the lower id takes the pair's terms
        const bool to_j = ref_attr && order[sj] < id_i;
        if (NEED_ENERGY)
        {
            // unscaled parameters (2^-32 scaling is exact)
            const float A = A2 * 2.3283064365386963e-10f, B = B2 * 2.3283064365386963e-10f;
            const float qi = qi2 * 2.3283064365386963e-10f;
            double ddx = dx, ddy = dy, ddz = dz;
            double r2d = (ddx * ddx + ddy * ddy) + ddz * ddz;
            double rd = __builtin_sqrt(r2d);
            double rid = 1.0 / rd;
            double ri2 = rid * rid;
            double ri6 = (ri2 * ri2) * ri2;
            int64_t pl = snb_to_fixed_d((((double)A * (1.0 / 12.0)) * ri6 -
                                         (double)B * (1.0 / 6.0)) * ri6);
            double gd;
            const double erfcd = snb_erfc_parts_d((double)beta * rd, &gd);
            int64_t pc = snb_to_fixed_d((((double)qi * (double)qj) * erfcd) * rid);
            if (to_j)
            {
                atomic_add_i64(e_sorted + sj, pl);
                atomic_add_i64(e_sorted + n + sj, pc);
            }
            else
            {
                S.elj += pl;
                S.ec += pc;
            }
        }
        if (NEED_VIRIAL)
        {
            const float fxv = fx2 * 2.3283064365386963e-10f, fyv = fy2 * 2.3283064365386963e-10f,
                        fzv = fz2 * 2.3283064365386963e-10f;
            int64_t p0 = snb_to_fixed(-(fxv * dx));
            int64_t p1 = snb_to_fixed(-(fxv * dy + fyv * dx));
            int64_t p2 = snb_to_fixed(-(fyv * dy));
            int64_t p3 = snb_to_fixed(-(fxv * dz + fzv * dx));
            int64_t p4 = snb_to_fixed(-(fyv * dz + fzv * dy));
            int64_t p5 = snb_to_fixed(-(fzv * dz));
            if (to_j)
            {
                atomic_add_i64(v_sorted + sj, p0);
                atomic_add_i64(v_sorted + (size_t)n + sj, p1);
                atomic_add_i64(v_sorted + (size_t)2 * n + sj, p2);
                atomic_add_i64(v_sorted + (size_t)3 * n + sj, p3);
                atomic_add_i64(v_sorted + (size_t)4 * n + sj, p4);
                atomic_add_i64(v_sorted + (size_t)5 * n + sj, p5);
            }
            else
            {
                S.v0 += p0; S.v1 += p1; S.v2 += p2; S.v3 += p3; S.v4 += p4; S.v5 += p5;
            }
        }
    }
}

// window slot -> sorted index: the LDS map, or a search of the range table
// when the window did not fit
__device__ __forceinline__ int win_slot_sorted(int slot, bool ov, const int* slot_s,
                                               const int* rfirst, const int* rpref, int nrange)
{
    if (!ov) return slot_s[slot];
    int lo = 0, hi = nrange - 1;
    while (lo < hi)
    {
        int mid = (lo + hi + 1) >> 1;
        if (rpref[mid] <= slot)
            lo = mid;
        else
            hi = mid - 1;
    }
    return rfirst[lo] + (slot - rpref[lo]);
}

// Force-only steps: one workgroup per block, whose window map (slot -> sorted
// index) and list units come ready-made from the rebuild (k_stage_inverse).  A unit is up to 128 entries of one row's near or far part;
// the units are dealt to the 16 wavefronts in contiguous runs of equal cost
// (a row may be shared by two), so that all of them finish together, and lane
// l of a wavefront holds what its unit l needs (64 units at a time).  A unit's
// values go to scalar registers as it comes up.  Per iteration of the software
// pipeline: the window slots of unit t + 1 (its list entries arrived during
// unit t - 1), the LJ parameters of unit t (its types arrived during unit
// t - 1), types and positions of unit t + 1, list entries of unit t + 2, then
// the pairs of unit t, two entries per lane.  The two register sets alternate
// (the loop body is written out twice), so no value is copied while its load
// is in flight.
//   - Far units hold pairs beyond rc + skin/4 at the rebuild: distances only;
//     a pair that has come into range loads its type and parameters then.
//   - A row whose type has no LJ with any type (nolj: the hydrogens of a
//     TIP3P water) skips the type and parameter gathers and the LJ terms,
//     which would be exact zeros.
//   - Where the window's atoms spread over less than half the box along an
//     axis, every minimum-image count of the block is zero there and
//     d - 0 * L = d, so those instructions are skipped.
// A window beyond the LDS capacity (OV) adds to the global accumulators
// instead and looks slots up in the global map.
//
// Bound by vector issue (IEEE-only math in a fixed order, about 62
// instructions per pair, 50 per unit and entry pair around them) at 16
// wavefronts a CU, which the window's LDS allows.  Against a loop of whole
// rows dealt round robin, with row metadata in vector registers and wave sums
// through LDS: 93,000 atoms (34.6M entries) 148 -> 119 us and 65.8M -> 50.3M
// vector instructions, 1,000,002 atoms 1583 -> 1337 us, 9,000 atoms 68 -> 54,
// 24,999 atoms 57 -> 48 (kernel alone).  Rows dealt round robin left the
// first wavefront of a block waiting 18 of 52 us for the last one.
struct WinUnits
{
    int at, desc, type, slot, si;  // desc: u_kind, u_last, u_rem below
    float4 a;
};

// lane's unit first + lane of those before `end`
__device__ __forceinline__ WinUnits win_load_units(const int4* __restrict__ units, int first,
                                                   int end, const float4* __restrict__ satom,
                                                   const int* __restrict__ stype,
                                                   const int* __restrict__ nolj)
{
    WinUnits m = {SNB_NL16_PAD, 3 << 6, 0, 0, 0, {0, 0, 0, 0}};
    const int t = first + (int)(threadIdx.x & 63);
    if (t < end)
    {
        const int4 u = units[t];
        m.si = u.x;
        m.at = u.y;
        m.slot = u.z;
        m.type = stype[u.x];
        m.a = satom[u.x];
        const int kind = (u.w & SNB_UNIT_FAR) ? 2 : (nolj[m.type] ? 1 : 0);
        m.desc = kind << 6 | ((u.w & SNB_UNIT_LAST) ? 256 : 0) | (u.w & 255) << 9;
    }
    return m;
}

template <bool ORTHO, bool OV>
__device__ __forceinline__ void win_force_units(
    int n, WinUnits m, const int4* __restrict__ units, int u_first, int u_end,
    const uint16_t* __restrict__ nl16, const float4* __restrict__ satom,
    const int* __restrict__ stype, const int* __restrict__ order,
    const float2* __restrict__ ab2, const int* __restrict__ nolj, int ntypes, float cscale,
    const SnbBox& box, float rc2, float beta, int64_t* __restrict__ fx, const float4* ctab,
    long long* acc, const int* slot_s, const int* __restrict__ wslots, int wrap_x, int wrap_y,
    int wrap_z)
{
    const int lane = threadIdx.x & 63;
    auto lane_of = [](int v, int l) { return __builtin_amdgcn_readlane(v, l); };
    auto lane_off = [](float v, int l) -> float {
        return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
    };
    // a unit in one word: kind (0 near, LJ; 1 near, no LJ; 2 far; 3 none),
    // whether it is the row's last, entries (at most 128)
    auto u_kind = [](int u) { return (u >> 6) & 3; };
    auto u_far = [](int u) { return (u & 128) != 0; };
    auto u_last = [](int u) { return (u & 256) != 0; };
    auto u_rem = [](int u) { return u >> 9; };
    struct Rec
    {
        int sla, slb, tja, tjb;
        unsigned sja, sjb;
        float4 aja, ajb;
    };
    // list entries lane and lane + 64 of a unit, unchecked beyond its end
    // (the list has SNB_NL16_PAD spare entries on either side)
    auto entries = [&](int u, int at, int& ea, int& eb) {
        const unsigned o = (unsigned)at + (u_far(u) ? 127u - (unsigned)lane : (unsigned)lane);
        ea = (int)ld32(nl16 - SNB_NL16_PAD, o);
        eb = (int)ld32(nl16 - SNB_NL16_PAD + (u_far(u) ? -64 : 64), o);
    };
    auto slots = [&](Rec& q, int u, int ea, int eb) {
        const int rem = u_rem(u);
        q.sla = lane < rem ? ea : 0;
        q.slb = lane + 64 < rem ? eb : 0;
        q.sja = (unsigned)(OV ? wslots[q.sla] : slot_s[q.sla]);
        q.sjb = (unsigned)(OV ? wslots[q.slb] : slot_s[q.slb]);
    };
    auto records = [&](Rec& q, int u) {
        if (u_kind(u) == 0)
        {
            q.tja = ld32(stype, q.sja);
            q.tjb = ld32(stype, q.sjb);
        }
        q.aja = ld32(satom, q.sja);
        q.ajb = ld32(satom, q.sjb);
    };
    int64_t sx = 0, sy = 0, sz = 0;
    // fa2 * d on row atom i, the opposite on j (A2, B2 and qq carry 2^32)
    auto give = [&](float fa2, float dx, float dy, float dz, int slot, unsigned sj) {
        const int64_t ix = snb_fixed_from_scaled(fa2 * dx), iy = snb_fixed_from_scaled(fa2 * dy),
                      iz = snb_fixed_from_scaled(fa2 * dz);
        sx += ix;
        sy += iy;
        sz += iz;
        if (!OV)
            lds_add3(acc, slot, ix, iy, iz);
        else
        {
            const int idj = order[sj];
            atomic_add_i64(fx + idj, -ix);
            atomic_add_i64(fx + n + idj, -iy);
            atomic_add_i64(fx + 2 * n + idj, -iz);
        }
    };
    int C = 0, N = 0, E = 0, e_at = 0, c = 0;  // the units of the three stages, C's lane
    auto step = [&](Rec& cur, Rec& nxt, int ea, int eb, int& fa, int& fb) {
        // the wrap flags are tested as integers (an empty statement:
        // otherwise their booleans are kept in lanes)
        int wx = uni(wrap_x), wy = uni(wrap_y), wz = uni(wrap_z);
        asm volatile("" : "+s"(wx), "+s"(wy), "+s"(wz));
        const int kind = u_kind(C), rem = u_rem(C);
        const float2* abrow = ab2 + lane_of(m.type, c) * ntypes;
        float2 ABa = {0, 0}, ABb = {0, 0};
        // the entries first: they are the last loads of the iteration
        // before, and waiting for them behind the parameter gathers would
        // wait for those too
        slots(nxt, N, ea, eb);
        asm volatile("" : "+v"(nxt.sla), "+v"(nxt.slb));
        if (kind == 0)
        {
            ABa = ld32(abrow, (unsigned)cur.tja);
            ABb = ld32(abrow, (unsigned)cur.tjb);
        }
        records(nxt, N);
        entries(E, e_at, fa, fb);
        const float xi = lane_off(m.a.x, c), yi = lane_off(m.a.y, c), zi = lane_off(m.a.z, c);
        const float qi2 = lane_off(m.a.w, c) * 4294967296.0f;  // 2^32
        float dxa = cur.aja.x - xi, dya = cur.aja.y - yi, dza = cur.aja.z - zi;
        float dxb = cur.ajb.x - xi, dyb = cur.ajb.y - yi, dzb = cur.ajb.z - zi;
        if (ORTHO)
        {
            if (wx)
            {
                dxa = dxa - rintf(dxa * box.rc[0]) * box.c[0];
                dxb = dxb - rintf(dxb * box.rc[0]) * box.c[0];
            }
            if (wy)
            {
                dya = dya - rintf(dya * box.rc[2]) * box.c[2];
                dyb = dyb - rintf(dyb * box.rc[2]) * box.c[2];
            }
            if (wz)
            {
                dza = dza - rintf(dza * box.rc[5]) * box.c[5];
                dzb = dzb - rintf(dzb * box.rc[5]) * box.c[5];
            }
        }
        else
        {
            pbc_disp(dxa, dya, dza, box);
            pbc_disp(dxb, dyb, dzb, box);
        }
        const float r2a = (dxa * dxa + dya * dya) + dza * dza;
        const float r2b = (dxb * dxb + dyb * dyb) + dzb * dzb;
        const bool ina = lane < rem && r2a < rc2, inb = lane + 64 < rem && r2b < rc2;
        if (kind == 0)
        {
            if (ina)
                give(pair_force_factor(r2a, ABa.x, ABa.y, qi2 * cur.aja.w, beta, cscale, ctab),
                     dxa, dya, dza, cur.sla, cur.sja);
            if (inb)
                give(pair_force_factor(r2b, ABb.x, ABb.y, qi2 * cur.ajb.w, beta, cscale, ctab),
                     dxb, dyb, dzb, cur.slb, cur.sjb);
        }
        else if (kind == 1)
        {
            if (ina)
                give(-pair_coulomb_factor(r2a, qi2 * cur.aja.w, beta, cscale, ctab), dxa, dya,
                     dza, cur.sla, cur.sja);
            if (inb)
                give(-pair_coulomb_factor(r2b, qi2 * cur.ajb.w, beta, cscale, ctab), dxb, dyb,
                     dzb, cur.slb, cur.sjb);
        }
        else if (__any(ina || inb))
        {
            // rare: pairs that came into range since the rebuild
            for (int h = 0; h < 2; h++)
                if (h ? inb : ina)
                {
                    const unsigned sj = h ? cur.sjb : cur.sja;
                    const float2 AB = ld32(abrow, (unsigned)ld32(stype, sj));
                    give(pair_force_factor(h ? r2b : r2a, AB.x, AB.y,
                                           qi2 * (h ? cur.ajb.w : cur.aja.w), beta, cscale, ctab),
                         h ? dxb : dxa, h ? dyb : dya, h ? dzb : dza, h ? cur.slb : cur.sla, sj);
                }
        }
        if (u_last(C) || c == 63)
        {
            // the end of the row (or of this wavefront's part of it): its own force
            const int64_t v = wave_sum3(sx, sy, sz);
            sx = sy = sz = 0;
            const int slot_i = lane_of(m.slot, c), si = lane_of(m.si, c);
            if ((lane & 15) == 0 && lane < 48)
            {
                const int d = lane == 0 ? 0 : (lane == 32 ? 1 : 2);
                if (!OV)  // the LDS accumulators hold the negated force
                    atomicAdd((unsigned long long*)&acc[3 * slot_i + d], (unsigned long long)(-v));
                else
                    atomic_add_i64(fx + (size_t)d * n + order[si], v);
            }
        }
    };
    for (int t0 = u_first; t0 < u_end; t0 += 64)
    {
        if (t0 > u_first) m = win_load_units(units, t0, u_end, satom, stype, nolj);
        const int T = u_end - t0 < 64 ? u_end - t0 : 64;
        // this wavefront's part of its last row ends with its last unit
        int desc = m.desc;
        if (lane == T - 1) desc |= 256;
        Rec r0 = {}, r1 = {};
        int e0a, e0b, e1a, e1b, e2a = 0, e2b = 0;
        C = lane_of(desc, 0);
        N = lane_of(desc, 1);
        E = lane_of(desc, 2);
        e_at = lane_of(m.at, 2);
        c = 0;
        entries(C, lane_of(m.at, 0), e0a, e0b);
        entries(N, lane_of(m.at, 1), e1a, e1b);
        slots(r0, C, e0a, e0b);
        records(r0, C);
        // lanes from T on describe no unit; beyond lane 63 the value of lane
        // 63 stands in (its entries are loaded and not used)
        auto shift = [&]() {
            const int l = c + 3 < 63 ? c + 3 : 63;
            c = c + 1;
            C = N;
            N = E;
            E = lane_of(desc, l);
            e_at = lane_of(m.at, l);
        };
        while (true)
        {
            step(r0, r1, e1a, e1b, e2a, e2b);
            if (c + 1 >= T) break;
            shift();
            step(r1, r0, e2a, e2b, e1a, e1b);
            if (c + 1 >= T) break;
            shift();
        }
    }
}

template <bool ORTHO>
__device__ __forceinline__ void k_pair_win_body(
    int n, int wcap, const uint16_t* __restrict__ nl16, const float4* __restrict__ satom,
    const int* __restrict__ stype, const int* __restrict__ order,
    const float2* __restrict__ ab2, const int* __restrict__ nolj, int ntypes,
    const float4* __restrict__ coul_tab, float cscale, SnbBox box, float rc2, float beta,
    const int* __restrict__ stage_base, const int* __restrict__ wslots,
    const int4* __restrict__ units, const int* __restrict__ unit_run,
    long long* __restrict__ stage, size_t stage_cap, int64_t* __restrict__ fx,
    const int* __restrict__ perm, int jdirect, unsigned bid, unsigned nbid)
{
    extern __shared__ long long smem[];
    float4* ctab = (float4*)smem;                  // [SNB_COUL_N]
    long long* acc = smem + 2 * SNB_COUL_N;        // [wcap][3]
    int* slot_s = (int*)(acc + 3 * (size_t)wcap);  // [wcap]
    float* range = (float*)(slot_s + wcap);        // [16][6]: min, max of x, y, z per wavefront
    const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
    const int w = uni(perm[bid]);  // heaviest blocks first
    const int base = uni(stage_base[w]), total = uni(stage_base[w + 1]) - base;
    const int* run = unit_run + w * SNB_UNIT_RUNS + wave;
    const int u_first = uni(run[0]), u_end = uni(run[1]);
    WinUnits m = win_load_units(units, u_first, u_end, satom, stype, nolj);
    if (tid < SNB_COUL_N) ctab[tid] = coul_tab[tid];
    const bool ov = total > wcap;
    const int* slot_map = wslots + base;
    if (!ov)
    {
        const float inf = __builtin_inff();
        float lo[3] = {inf, inf, inf}, hi[3] = {-inf, -inf, -inf};
        for (int t = tid; t < total; t += blockDim.x)
        {
            const int sj = slot_map[t];
            slot_s[t] = sj;
            if (ORTHO)
            {
                const float4 a = satom[sj];
                lo[0] = fminf(lo[0], a.x);
                lo[1] = fminf(lo[1], a.y);
                lo[2] = fminf(lo[2], a.z);
                hi[0] = fmaxf(hi[0], a.x);
                hi[1] = fmaxf(hi[1], a.y);
                hi[2] = fmaxf(hi[2], a.z);
            }
        }
        for (int t = tid; t < 3 * total; t += blockDim.x) acc[t] = 0;
        if (ORTHO)
            for (int d = 0; d < 3; d++)
            {
                const float a = wave_min(lo[d]), b = -wave_min(-hi[d]);
                if (lane == 0)
                {
                    range[6 * wave + d] = a;
                    range[6 * wave + 3 + d] = b;
                }
            }
    }
    __syncthreads();
    if (!ov)
    {
        // |d| <= spread for every pair of the block, so that 0.49 leaves
        // rint(d / L) = 0 with room for the rounding of the quotient (an
        // infinite coordinate makes the spread infinite, and a NaN one fails
        // the distance test with or without the image)
        int wrap[3] = {1, 1, 1};
        if (ORTHO)
            for (int d = 0; d < 3; d++)
            {
                const int q = 6 * (lane & 15) + d;
                const float spread = -wave_min(-range[q + 3]) - wave_min(range[q]);
                wrap[d] = uni(spread * box.rc[d == 0 ? 0 : (d == 1 ? 2 : 5)] < 0.49f ? 0 : 1);
            }
        win_force_units<ORTHO, false>(n, m, units, u_first, u_end, nl16, satom, stype, order, ab2,
                                      nolj, ntypes, cscale, box, rc2, beta, fx, ctab, acc, slot_s,
                                      slot_map, wrap[0], wrap[1], wrap[2]);
    }
    else
        win_force_units<ORTHO, true>(n, m, units, u_first, u_end, nl16, satom, stype, order, ab2,
                                     nolj, ntypes, cscale, box, rc2, beta, fx, ctab, acc, slot_s,
                                     slot_map, 1, 1, 1);
    __syncthreads();
    if (jdirect)
    {
        // the window's sums go straight to the id-ordered accumulators
        // (integer sums, so the order of the adds does not matter); slots
        // that received nothing are skipped
        if (!ov)
            for (int t = tid; t < total; t += blockDim.x)
            {
                const long long vx = acc[3 * t], vy = acc[3 * t + 1], vz = acc[3 * t + 2];
                if ((vx | vy | vz) == 0) continue;
                const int id = order[slot_s[t]];
                if (vx) atomic_add_i64(fx + id, -vx);
                if (vy) atomic_add_i64(fx + n + id, -vy);
                if (vz) atomic_add_i64(fx + 2 * n + id, -vz);
            }
        return;
    }
    for (int t = tid; t < 3 * total; t += blockDim.x)
    {
        const size_t d = 3 * (size_t)base + t;
        if (d >= 3 * stage_cap) break;  // cannot happen: stage holds n x invmax
        stage[d] = ov ? 0 : -acc[t];
    }
}

template <bool ORTHO>
__global__ void __launch_bounds__(1024) k_pair_win(
    int n, int wcap, const uint16_t* __restrict__ nl16, const float4* __restrict__ satom,
    const int* __restrict__ stype, const int* __restrict__ order,
    const float2* __restrict__ ab2, const int* __restrict__ nolj, int ntypes,
    const float4* __restrict__ coul_tab, float cscale, SnbBox box, float rc2, float beta,
    const int* __restrict__ stage_base, const int* __restrict__ wslots,
    const int4* __restrict__ units, const int* __restrict__ unit_run,
    long long* __restrict__ stage, size_t stage_cap, int64_t* __restrict__ fx,
    const int* __restrict__ perm, int jdirect)
{
    k_pair_win_body<ORTHO>(n, wcap, nl16, satom, stype, order, ab2, nolj, ntypes, coul_tab, cscale,
                           box, rc2, beta, stage_base, wslots, units, unit_run, stage, stage_cap,
                           fx, perm, jdirect, blockIdx.x, gridDim.x);
}

struct PairWinArgs
{
    int n;
    int wcap;
    const uint16_t* nl16;
    const float4* satom;
    const int* stype;
    const int* order;
    const float2* ab2;
    const int* nolj;
    int ntypes;
    const float4* coul_tab;
    float cscale;
    SnbBox box;
    float rc2;
    float beta;
    const int* stage_base;
    const int* wslots;
    const int4* units;
    const int* unit_run;
    long long* stage;
    size_t stage_cap;
    int64_t* fx;
    const int* perm;
    int jdirect;
};

template <bool ORTHO>
__global__ void __launch_bounds__(1024) k_pair_win_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const PairWinArgs& a = snb_seg<PairWinArgs>(t, bid, nbid);
    k_pair_win_body<ORTHO>(a.n, a.wcap, a.nl16, a.satom, a.stype, a.order, a.ab2, a.nolj, a.ntypes,
                           a.coul_tab, a.cscale, a.box, a.rc2, a.beta, a.stage_base, a.wslots,
                           a.units, a.unit_run, a.stage, a.stage_cap, a.fx, a.perm, a.jdirect, bid,
                           nbid);
}

// Energy and virial steps: the same block and window, rows instead of units.
template <bool NEED_ENERGY, bool NEED_VIRIAL, bool ORTHO>
__device__ __forceinline__ void k_pair_ev_body(
    int n, SnbWin W, const int* __restrict__ start, const int* __restrict__ sorted_cell,
    const int* __restrict__ row_count, const int* __restrict__ row_split,
    const uint16_t* __restrict__ nl16, int max_nb,
    const float4* __restrict__ satom, const int* __restrict__ stype,
    const int* __restrict__ order, const float2* __restrict__ ab2, int ntypes,
    const float4* __restrict__ coul_tab, float cscale, SnbBox box, float rc2, float beta,
    const int* __restrict__ stage_base, long long* __restrict__ stage, size_t stage_cap,
    int64_t* __restrict__ fx, int64_t* __restrict__ e_sorted, int64_t* __restrict__ v_sorted,
    int ref_attr, const int* __restrict__ perm, unsigned bid, unsigned nbid)
{
    extern __shared__ long long smem[];
    float4* ctab = (float4*)smem;                   // [SNB_COUL_N]
    long long* acc = smem + 2 * SNB_COUL_N;         // [wcap][3]
    int* slot_s = (int*)(acc + 3 * (size_t)W.wcap);  // [wcap]
    int* rfirst = slot_s + W.wcap;                  // [128]
    int* rpref = rfirst + SNB_WIN_MAX_RANGES;       // [129]
    const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
    const int nwave = blockDim.x >> 6;
    const int w = uni(perm[bid]);  // heaviest blocks first
    if (tid < SNB_COUL_N) ctab[tid] = coul_tab[tid];
    int x0, y0, z0;
    snb_win_block(W, w, x0, y0, z0);
    x0 = uni(x0);
    y0 = uni(y0);
    z0 = uni(z0);
    // range table: sizes, then a wave-0 scan
    int rsz = 0;
    if (tid < SNB_WIN_MAX_RANGES)
    {
        int f = 0;
        if (tid < W.nrange)
        {
            int fc, nc;
            snb_win_range_cells(W, x0, y0, z0, tid, fc, nc);
            f = start[fc];
            rsz = nc > 0 ? start[fc + nc] - f : 0;
        }
        rfirst[tid] = f;
        rpref[tid + 1] = rsz;
    }
    __syncthreads();
    if (wave == 0)
    {
        int a0 = rpref[lane + 1], a1 = rpref[lane + 65];
        int i0 = a0, i1 = a1;
        for (int off = 1; off < 64; off <<= 1)
        {
            int u0 = __shfl_up(i0, off), u1 = __shfl_up(i1, off);
            if (lane >= off)
            {
                i0 += u0;
                i1 += u1;
            }
        }
        int t0 = __shfl(i0, 63);
        rpref[lane + 1] = i0;
        rpref[lane + 65] = t0 + i1;
        if (lane == 0) rpref[0] = 0;
    }
    __syncthreads();
    const int total = uni(rpref[SNB_WIN_MAX_RANGES]);
    const bool ov = total > W.wcap;
    if (!ov)
    {
        for (int k = wave; k < W.nrange; k += nwave)
        {
            const int b0 = uni(rpref[k]), cnt = uni(rpref[k + 1]) - b0, f = uni(rfirst[k]);
            for (int t = lane; t < cnt; t += 64) slot_s[b0 + t] = f + t;
        }
        for (int t = tid; t < 3 * total; t += blockDim.x) acc[t] = 0;
    }
    __syncthreads();
    for (int col = 0; col < W.a * W.b; col++)
    {
        int ua = col / W.b, vb = col - ua * W.b;
        if (x0 + ua >= W.nx || y0 + vb >= W.ny) continue;
        int colbase = ((x0 + ua) * W.ny + (y0 + vb)) * W.nz;
        int z1 = z0 + W.s < W.nz ? z0 + W.s : W.nz;
        int r0 = start[colbase + z0], r1 = start[colbase + z1];
        for (int si = r0 + wave; si < r1; si += nwave)
        {
            const int cnt = row_count[si], split = row_split[si];
            const unsigned row0 = (unsigned)si * (unsigned)max_nb;  // n * max_nb < 2^31
            const float4 ai = satom[si];
            const float qi2 = ai.w * 4294967296.0f;  // 2^32 fixed-point scale
            const unsigned trow = (unsigned)(stype[si] * ntypes);
            const int id_i = (NEED_ENERGY || NEED_VIRIAL) && ref_attr ? order[si] : 0;
            WinRowSums S = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
            // two entries per lane at a time; each step fetches its records
            // when it starts: the FP64 energies and row sums leave no
            // registers for a second set of records
            auto entry = [&](int k) -> int {
                return k < cnt ? (int)ld32(nl16, row0 + (unsigned)snb_row_entry(k, split, max_nb))
                               : -1;
            };
            auto sorted_of = [&](int sl) -> unsigned {
                return sl >= 0 ? (unsigned)win_slot_sorted(sl, ov, slot_s, rfirst, rpref, W.nrange)
                               : (unsigned)si;
            };
            int sla = 0, slb = 0, tja = 0, tjb = 0;
            unsigned sja = 0, sjb = 0;
            float4 aja = {0, 0, 0, 0}, ajb = {0, 0, 0, 0};
            auto records = [&](int k) {
                sla = entry(k + lane);
                slb = entry(k + 64 + lane);
                sja = sorted_of(sla);
                sjb = sorted_of(slb);
                aja = ld32(satom, sja);
                ajb = ld32(satom, sjb);
                tja = ld32(stype, sja);
                tjb = ld32(stype, sjb);
            };
            for (int k0 = 0; k0 < cnt; k0 += 128)
            {
                records(k0);
                const float2 ABa = ld32(ab2, trow + (unsigned)tja);
                const float2 ABb = ld32(ab2, trow + (unsigned)tjb);
                float dxa = aja.x - ai.x, dya = aja.y - ai.y, dza = aja.z - ai.z;
                float dxb = ajb.x - ai.x, dyb = ajb.y - ai.y, dzb = ajb.z - ai.z;
                win_disp<ORTHO>(dxa, dya, dza, box);
                win_disp<ORTHO>(dxb, dyb, dzb, box);
                const float r2a = (dxa * dxa + dya * dya) + dza * dza;
                const float r2b = (dxb * dxb + dyb * dyb) + dzb * dzb;
                // keep the parameter gathers ahead of the branches (the
                // compiler would otherwise sink them into the branches, where
                // their latency is not hidden behind the distance test); an
                // empty statement that reads the registers, nothing is emitted
                asm volatile("" ::"v"(ABa.x), "v"(ABa.y), "v"(ABb.x), "v"(ABb.y));
                if (sla >= 0 && r2a < rc2)
                    win_pair<NEED_ENERGY, NEED_VIRIAL>(S, dxa, dya, dza, r2a, ABa.x, ABa.y, qi2,
                                                       aja.w, beta, cscale, ctab, sla, sja, ov,
                                                       acc, n, order, fx, ref_attr, id_i,
                                                       e_sorted, v_sorted);
                if (slb >= 0 && r2b < rc2)
                    win_pair<NEED_ENERGY, NEED_VIRIAL>(S, dxb, dyb, dzb, r2b, ABb.x, ABb.y, qi2,
                                                       ajb.w, beta, cscale, ctab, slb, sjb, ov,
                                                       acc, n, order, fx, ref_attr, id_i,
                                                       e_sorted, v_sorted);
            }
            int64_t sx = wave_sum(S.sx), sy = wave_sum(S.sy), sz = wave_sum(S.sz);
            int64_t elj = 0, ec = 0, v0 = 0, v1 = 0, v2 = 0, v3 = 0, v4 = 0, v5 = 0;
            if (NEED_ENERGY)
            {
                elj = wave_sum(S.elj);
                ec = wave_sum(S.ec);
            }
            if (NEED_VIRIAL)
            {
                v0 = wave_sum(S.v0); v1 = wave_sum(S.v1); v2 = wave_sum(S.v2);
                v3 = wave_sum(S.v3); v4 = wave_sum(S.v4); v5 = wave_sum(S.v5);
            }
            if (lane == 0)
            {
                if (!ov)
                {
                    int cz = sorted_cell[si] % W.nz;
                    int k = snb_win_range_of(W, z0, ua, vb + 2, cz - z0 + 2);
                    int slot_i = rpref[k] + (si - rfirst[k]);
                    // negated-force convention of the LDS accumulators
                    lds_add3(acc, slot_i, -sx, -sy, -sz);
                }
                else
                {
                    int idi = order[si];
                    atomic_add_i64(fx + idi, sx);
                    atomic_add_i64(fx + n + idi, sy);
                    atomic_add_i64(fx + 2 * n + idi, sz);
                }
                // other rows' lower-id terms may land on si as well
                // (ref_attr: the arrays were cleared before the launch)
                if (NEED_ENERGY)
                {
                    if (ref_attr)
                    {
                        atomic_add_i64(e_sorted + si, elj);
                        atomic_add_i64(e_sorted + (size_t)n + si, ec);
                    }
                    else
                    {
                        e_sorted[si] = elj;
                        e_sorted[(size_t)n + si] = ec;
                    }
                }
                if (NEED_VIRIAL)
                {
                    const int64_t vv[6] = {v0, v1, v2, v3, v4, v5};
                    for (int c = 0; c < 6; c++)
                    {
                        if (ref_attr)
                            atomic_add_i64(v_sorted + (size_t)c * n + si, vv[c]);
                        else
                            v_sorted[(size_t)c * n + si] = vv[c];
                    }
                }
            }
        }
    }
    __syncthreads();
    // stage_base + total stays within the stage: it holds n x invmax slots
    const size_t base = 3 * (size_t)stage_base[w];
    for (int t = tid; t < 3 * total; t += blockDim.x)
    {
        if (base + t >= 3 * stage_cap) break;
        stage[base + t] = ov ? 0 : -acc[t];
    }
}

template <bool NEED_ENERGY, bool NEED_VIRIAL, bool ORTHO>
__global__ void __launch_bounds__(1024) k_pair_ev(
    int n, SnbWin W, const int* __restrict__ start, const int* __restrict__ sorted_cell,
    const int* __restrict__ row_count, const int* __restrict__ row_split,
    const uint16_t* __restrict__ nl16, int max_nb,
    const float4* __restrict__ satom, const int* __restrict__ stype,
    const int* __restrict__ order, const float2* __restrict__ ab2, int ntypes,
    const float4* __restrict__ coul_tab, float cscale, SnbBox box, float rc2, float beta,
    const int* __restrict__ stage_base, long long* __restrict__ stage, size_t stage_cap,
    int64_t* __restrict__ fx, int64_t* __restrict__ e_sorted, int64_t* __restrict__ v_sorted,
    int ref_attr, const int* __restrict__ perm)
{
    k_pair_ev_body<NEED_ENERGY, NEED_VIRIAL, ORTHO>(
        n, W, start, sorted_cell, row_count, row_split, nl16, max_nb, satom, stype, order, ab2,
        ntypes, coul_tab, cscale, box, rc2, beta, stage_base, stage, stage_cap, fx, e_sorted,
        v_sorted, ref_attr, perm, blockIdx.x, gridDim.x);
}

struct PairEvArgs
{
    int n;
    SnbWin W;
    const int* start;
    const int* sorted_cell;
    const int* row_count;
    const int* row_split;
    const uint16_t* nl16;
    int max_nb;
    const float4* satom;
    const int* stype;
    const int* order;
    const float2* ab2;
    int ntypes;
    const float4* coul_tab;
    float cscale;
    SnbBox box;
    float rc2;
    float beta;
    const int* stage_base;
    long long* stage;
    size_t stage_cap;
    int64_t* fx;
    int64_t* e_sorted;
    int64_t* v_sorted;
    int ref_attr;
    const int* perm;
};

template <bool NEED_ENERGY, bool NEED_VIRIAL, bool ORTHO>
__global__ void __launch_bounds__(1024) k_pair_ev_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const PairEvArgs& a = snb_seg<PairEvArgs>(t, bid, nbid);
    k_pair_ev_body<NEED_ENERGY, NEED_VIRIAL, ORTHO>(
        a.n, a.W, a.start, a.sorted_cell, a.row_count, a.row_split, a.nl16, a.max_nb, a.satom,
        a.stype, a.order, a.ab2, a.ntypes, a.coul_tab, a.cscale, a.box, a.rc2, a.beta, a.stage_base,
        a.stage, a.stage_cap, a.fx, a.e_sorted, a.v_sorted, a.ref_attr, a.perm, bid, nbid);
}

// Per sorted atom: sum of its stage entries into the id-ordered accumulators
// (plus the row-owner energies / virials on those steps).
__device__ __forceinline__ void k_stage_gather_body(int n, const int* __restrict__ inv_count,
                               const int* __restrict__ inv_list, int invmax,
                               const long long* __restrict__ stage, size_t stage_cap,
                               const int* __restrict__ order,
                               int64_t* __restrict__ fx, int need_energy, int need_virial,
                               const int64_t* __restrict__ e_sorted,
                               const int64_t* __restrict__ v_sorted, int64_t* __restrict__ e_atom,
                               int64_t* __restrict__ vir,
    unsigned bid, unsigned nbid)
{
    int s = bid * blockDim.x + threadIdx.x;
    if (s >= n) return;
    int id = order[s];
    int m = inv_count[s];
    if (m > invmax) m = invmax;
    int64_t sx = 0, sy = 0, sz = 0;
    const int* lst = inv_list + (size_t)s * invmax;
    for (int k = 0; k < m; k++)
    {
        if ((size_t)lst[k] >= stage_cap) continue;
        const long long* p = stage + 3 * (size_t)lst[k];
        sx += p[0];
        sy += p[1];
        sz += p[2];
    }
    fx[id] += sx;
    fx[n + id] += sy;
    fx[2 * n + id] += sz;
    if (need_energy)
    {
        e_atom[id] += e_sorted[s];
        e_atom[(size_t)n + id] += e_sorted[(size_t)n + s];
    }
    if (need_virial)
        for (int c = 0; c < 6; c++) vir[(size_t)c * n + id] += v_sorted[(size_t)c * n + s];
}

__global__ void k_stage_gather(int n, const int* __restrict__ inv_count,
                               const int* __restrict__ inv_list, int invmax,
                               const long long* __restrict__ stage, size_t stage_cap,
                               const int* __restrict__ order,
                               int64_t* __restrict__ fx, int need_energy, int need_virial,
                               const int64_t* __restrict__ e_sorted,
                               const int64_t* __restrict__ v_sorted, int64_t* __restrict__ e_atom,
                               int64_t* __restrict__ vir)
{
    k_stage_gather_body(
        n, inv_count, inv_list, invmax, stage, stage_cap, order, fx, need_energy, need_virial,
        e_sorted, v_sorted, e_atom, vir, blockIdx.x, gridDim.x);
}

struct StageGatherArgs
{
    int n;
    const int* inv_count;
    const int* inv_list;
    int invmax;
    const long long* stage;
    size_t stage_cap;
    const int* order;
    int64_t* fx;
    int need_energy;
    int need_virial;
    const int64_t* e_sorted;
    const int64_t* v_sorted;
    int64_t* e_atom;
    int64_t* vir;
};

__global__ void k_stage_gather_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const StageGatherArgs& a = snb_seg<StageGatherArgs>(t, bid, nbid);
    k_stage_gather_body(
        a.n, a.inv_count, a.inv_list, a.invmax, a.stage, a.stage_cap, a.order, a.fx, a.need_energy,
        a.need_virial, a.e_sorted, a.v_sorted, a.e_atom, a.vir, bid, nbid);
}

int snb_launch_lj_window(snb_context* ctx, const snb_vector* crd, const float* charge,
                         const SnbBox& box, float beta, int need_energy, int need_virial)
{
    int n = ctx->n;
    if (n <= 0) return SNB_OK;
    SnbNl& L = ctx->nl;
    const SnbWin& W = L.win;
    hipStream_t s = ctx->stream;
    SNB_LAUNCH_B(k_pack_sorted, k_pack_sorted_batch, PackSortedArgs, dim3((n + 255) / 256),
                 dim3(256), 0, s, n, L.order, crd, charge, ctx->satom, ctx->status);
    float rc2 = ctx->lj.cutoff * ctx->lj.cutoff;
    size_t lds = 28 * (size_t)W.wcap + SNB_WIN_FIXED_LDS;
    if (L.win_lds_set != lds)
    {
        // dynamic LDS above 64 KiB is granted per kernel
        const void* fns[8] = {
            (const void*)k_pair_win<true>, (const void*)k_pair_win<false>,
            (const void*)k_pair_ev<true, true, true>, (const void*)k_pair_ev<true, false, true>,
            (const void*)k_pair_ev<false, true, true>, (const void*)k_pair_ev<true, true, false>,
            (const void*)k_pair_ev<true, false, false>, (const void*)k_pair_ev<false, true, false>};
        for (const void* f : fns)
            SNB_CHECK(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        L.win_lds_set = lds;
    }
    // diagonal cell and rcell: the displacement skips the zero terms
    const bool ortho = box.c[1] == 0.0f && box.c[3] == 0.0f && box.c[4] == 0.0f &&
                       box.rc[1] == 0.0f && box.rc[3] == 0.0f && box.rc[4] == 0.0f;
    // Force-only steps: the blocks add their window forces to the accumulators
    // by atomics, or write them to the stage (one slot per window atom) which
    // k_stage_gather sums.  What decides are the rounds of blocks over the
    // compute units, one block on each at a time: in two rounds or less they
    // all end together, and no block's arithmetic runs beside their adds; in
    // more rounds it does, and the gather comes on top of the pair kernel.  Ten
    // whole steps, stage / atomics in us, on 256 compute units:
    //   490 to 512 blocks: 66,000 atoms 1729 / 1767, 81,000 1705 / 1758,
    //     93,000 (8 A) 1924 / 1973, (10 A) 2237 / 2309, 108,000 2057 / 2136,
    //     150,000 2656 / 2651;
    //   612 and more: 87,000 (612) 1969 / 1825, (960) 2293 / 2062, 126,000
    //     (700) 2510 / 2318, 150,000 (1000) 3527 / 3141, 1,000,000 22340 / 19412.
    // The stage is kept to the sizes where two rounds are worth most of 2 to 4%
    // of the step: a pair call by itself, with no other stream beside it, pays 4
    // to 24% for the gather at any size (66,000 107 / 93 us, 93,000 123 / 117,
    // at 8 A 105 / 84, 108,000 122 / 117); below, 24,000 to 61,500 atoms are within 3% either
    // way, and from 135,000 on the step gains nothing any more.
    int jdirect = ctx->lj.j_direct;
    if (jdirect < 0)
    {
        const bool two_rounds = W.nblock <= 2 * ctx->num_cu;
        jdirect = (two_rounds && n >= 65536 && n <= 98304) ? 0 : 1;
    }
    if (need_energy || need_virial) jdirect = 0;
    const int ref_attr = ctx->lj.owner_attribution ? 0 : 1;
    int rc;
    if (ref_attr && need_energy && (rc = snb_launch_fill_i64(s, ctx->e_sorted, 2 * (size_t)n)))
        return rc;
    if (ref_attr && need_virial && (rc = snb_launch_fill_i64(s, ctx->v_sorted, 6 * (size_t)n)))
        return rc;
    snb_prof_begin(ctx, SNB_PROF_PAIR);
    // recorded step batches: the work of a workgroup is its rows
    if (snb_rec) snb_rec->weight_next = (double)n / W.nblock;
#define SNB_EV_LAUNCH(E, V, O)                                                                   \
    SNB_LAUNCH_B((k_pair_ev<E, V, O>), (k_pair_ev_batch<E, V, O>), PairEvArgs, dim3(W.nblock),   \
                 dim3(1024), lds, s, n, W, L.cell_start, L.sorted_cell, L.row_count,             \
                 L.row_split, L.nl16, L.max_nb, ctx->satom, ctx->stype, L.order, ctx->lj.ab2,    \
                 ctx->lj.ntypes, ctx->lj.coul, ctx->lj.coul_scale, box, rc2, beta, L.stage_base, \
                 L.stage, (size_t)n * L.invmax, ctx->fx, ctx->e_sorted, ctx->v_sorted, ref_attr, \
                 L.block_perm)
#define SNB_WIN_LAUNCH(O)                                                                       \
    if (need_energy && need_virial)                                                             \
        SNB_EV_LAUNCH(true, true, O);                                                           \
    else if (need_energy)                                                                       \
        SNB_EV_LAUNCH(true, false, O);                                                          \
    else if (need_virial)                                                                       \
        SNB_EV_LAUNCH(false, true, O);                                                          \
    else                                                                                        \
        SNB_LAUNCH_B(k_pair_win<O>, k_pair_win_batch<O>, PairWinArgs, dim3(W.nblock), dim3(1024), \
                     lds, s, n, W.wcap, L.nl16, ctx->satom, ctx->stype, L.order, ctx->lj.ab2,    \
                     ctx->lj.nolj, ctx->lj.ntypes, ctx->lj.coul, ctx->lj.coul_scale, box, rc2,   \
                     beta, L.stage_base, L.wslots, L.units, L.unit_run, L.stage,                 \
                     (size_t)n * L.invmax, ctx->fx, L.block_perm, jdirect);
    if (ortho)
    {
        SNB_WIN_LAUNCH(true)
    }
    else
    {
        SNB_WIN_LAUNCH(false)
    }
#undef SNB_WIN_LAUNCH
#undef SNB_EV_LAUNCH
    snb_prof_end(ctx, SNB_PROF_PAIR);
    SNB_CHECK(hipGetLastError());
    if (jdirect) return SNB_OK;
    SNB_LAUNCH_B(k_stage_gather, k_stage_gather_batch, StageGatherArgs, dim3((n + 255) / 256),
                 dim3(256), 0, s, n, L.inv_count, L.inv_list, L.invmax, L.stage,
                 (size_t)n * L.invmax, L.order, ctx->fx, need_energy, need_virial, ctx->e_sorted,
                 ctx->v_sorted, ctx->e_atom, ctx->vir_atom);
    SNB_CHECK(hipGetLastError());
    return SNB_OK;
}
