// snb_nlwin.hip -- neighbor-list build for the windowed pair path.
//
// After the cell sort (snb_nl.hip), one workgroup per cell builds the rows of
// its atoms: the candidates of the forward half-stencil (13 columns, runs of
// up to five z-cells, see snb_window.h) are staged in LDS, tested 64 at a time
// and the survivors are stored as 16-bit slots of the owning block's window.  The same pair set
// as the reference's half list results -- every unordered pair within
// rc + skin once, minus exclusions decided on the lower atom id as the
// reference does (neighbor_list.cpp:594-665) -- only the row that holds a
// pair differs.  When the reference-layout list is wanted (the public d_nl),
// it is derived from these rows (export) and each row sorted.
#include "snb_internal.h"

// Range table of the window of block (x0, y0, z0) into LDS: first sorted index
// and exclusive slot prefix of each range; one wavefront, two ranges per lane.
// Caller synchronises before reading.
__device__ void win_table_wave(const SnbWin& W, const int* __restrict__ start, int x0, int y0,
                               int z0, int lane, int* first, int* pref)
{
    int sz[2], fs[2];
    for (int h = 0; h < 2; h++)
    {
        int k = lane + 64 * h;
        sz[h] = 0;
        fs[h] = 0;
        if (k < W.nrange)
        {
            int fc, nc;
            snb_win_range_cells(W, x0, y0, z0, k, fc, nc);
            fs[h] = start[fc];
            sz[h] = nc > 0 ? start[fc + nc] - fs[h] : 0;
        }
    }
    // exclusive prefix over k = lane, then k = lane + 64
    int tot0 = sz[0], inc0 = sz[0], inc1 = sz[1];
    for (int off = 1; off < 64; off <<= 1)
    {
        int a = __shfl_up(inc0, off);
        int b = __shfl_up(inc1, off);
        if (lane >= off)
        {
            inc0 += a;
            inc1 += b;
        }
    }
    tot0 = __shfl(inc0, 63);
    first[lane] = fs[0];
    first[lane + 64] = fs[1];
    pref[lane] = inc0 - sz[0];
    pref[lane + 64] = tot0 + inc1 - sz[1];
    if (lane == 63) pref[SNB_WIN_MAX_RANGES] = tot0 + inc1;
}

__device__ __forceinline__ bool excluded_pair(int id_a, int id_b, const int* __restrict__ ex_start,
                                              const int* __restrict__ ex_list,
                                              const int* __restrict__ ex_num)
{
    // the reference deletes hi from row lo when hi is in lo's list, testing
    // membership only between the list's first and last entries
    if (!ex_num) return false;
    int lo = id_a < id_b ? id_a : id_b, hi = id_a < id_b ? id_b : id_a;
    int en = ex_num[lo];
    if (en <= 0) return false;
    int es = ex_start[lo];
    if (hi < ex_list[es] || hi > ex_list[es + en - 1]) return false;
    for (int t = es; t < es + en; t++)
        if (ex_list[t] == hi) return true;
    return false;
}

__device__ __forceinline__ void win_block_of_cell(const SnbWin& W, int c, int& cx, int& cy,
                                                  int& cz, int& x0, int& y0, int& z0)
{
    cz = c % W.nz;
    cy = (c / W.nz) % W.ny;
    cx = c / (W.nz * W.ny);
    x0 = (cx / W.a) * W.a;
    y0 = (cy / W.b) * W.b;
    z0 = (cz / W.s) * W.s;
}

// Candidate capacity of one LDS chunk.  1408 candidates (22 groups, 32 KB of
// LDS) hold a mean stencil of ~1,360 atoms at 6 A cells; four workgroups then
// fit a CU beside the reciprocal pipeline's.
#define SNB_NLC_CAP 1408
#define SNB_NLC_MAXRUN 63
#define SNB_NLC_WAVES 8

// One 512-thread workgroup per cell.  The candidates are the cell's forward
// stencil: 13 columns of up to 5 cells, one run per cell, at most 63 runs, in
// chunks of SNB_NLC_CAP.  Candidate order is column, z (unwrapped), sorted
// index, so a row lists its entries in that order; the first run is the cell
// itself, where only larger sorted indices count.  For a diagonal box each
// atom first marks the stencil cells whose box lies within the list radius
// of its (wrapped) position, with a margin over float rounding; groups of 64
// candidates that lie in unmarked cells only are skipped for that atom.
//
// What bounds this kernel is the number of instructions per pair of (atom,
// group).  A wavefront keeps a group of candidates in its lanes and goes over
// the cell's atoms, whose positions are scalars; the two distance comparisons
// are the ballots of the row's near and far entries, which lane a keeps for
// atom a.  The minimum image is one shift per candidate wherever every atom of
// the cell has the same one (rounding is monotone, so the extremes of the
// cell's positions decide); where they differ the pair is folded by itself.
// Row positions come from prefix sums of the ballots' counts over the groups,
// then the wavefront writes its groups' entries.  About 45 instructions per
// (atom, group), half of them scalar, where a wavefront per row took 85: 292 us
// -> 262 at 45,000 atoms and 10 A while the widest cell set the time, 134 over
// cells of equal width.
//
// The distance is taken as q_i - q_j for the row atom i.  The reference takes
// it from the higher id to the lower; the two agree bit for bit (negation is
// exact) except where floorf(s + 0.5) rounds differently at |s| = k + 1/2,
// i.e. where the minimum image is half a box away in that dimension.  With
// >= 5 cells of >= (rc + skin)/2 per axis that is >= 1.25 (rc + skin), so
// such a pair fails the test either way.
#define SNB_NLC_GROUPS (SNB_NLC_CAP / 64)
typedef float SnbF4 __attribute__((ext_vector_type(4)));
typedef const SnbF4 __attribute__((address_space(4)))* SnbConstF4;

__device__ __forceinline__ float readlane_f(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// v of the lane that DPP control C names, the lane's own where that has none
template <int C>
__device__ __forceinline__ float dpp_f(float v)
{
    const int x = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(x, x, C, 0xf, 0xf, false));
}

// smallest and largest of the wavefront's values (NaN left out)
__device__ __forceinline__ float wave_fmin(float v)
{
    v = fminf(v, dpp_f<0x111>(v));  // row_shr 1, 2, 4, 8: rows of 16
    v = fminf(v, dpp_f<0x112>(v));
    v = fminf(v, dpp_f<0x114>(v));
    v = fminf(v, dpp_f<0x118>(v));
    v = fminf(v, dpp_f<0x142>(v));  // lane 15 of a row to the next row, then lane 31
    v = fminf(v, dpp_f<0x143>(v));
    return readlane_f(v, 63);
}

__device__ __forceinline__ float wave_fmax(float v) { return -wave_fmin(-v); }

__device__ __forceinline__ int mbcnt(uint64_t mask)
{
    return (int)__builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                          __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

// v with lane l's value replaced by the scalar x (no clang builtin names it)
extern "C" __device__ unsigned snb_writelane(unsigned x, unsigned l, unsigned v) __asm(
    "llvm.amdgcn.writelane.i32");

__device__ __forceinline__ uint64_t lane_value(uint2 v, int l)
{
    return (uint64_t)(unsigned)__builtin_amdgcn_readlane((int)v.x, l) |
           ((uint64_t)(unsigned)__builtin_amdgcn_readlane((int)v.y, l) << 32);
}

template <bool ORTHO>
__device__ __forceinline__ void k_nl_build_cell_body(
    const int* __restrict__ need, SnbWin W, const int* __restrict__ start,
    const float4* __restrict__ sorted_crd, SnbBox box, float cs2,
    const int* __restrict__ ex_start, const int* __restrict__ ex_list,
    const int* __restrict__ ex_num, const int2* __restrict__ ex_rng, int max_nb, float near2,
    uint16_t* __restrict__ nl16, int* __restrict__ row_count, int* __restrict__ row_split,
    int* __restrict__ status, float wx, float wy, float wz,
    unsigned bid, unsigned nbid)
{
    if (need[0] == 0) return;
    __shared__ int first[SNB_WIN_MAX_RANGES];
    __shared__ int pref[SNB_WIN_MAX_RANGES + 1];
    __shared__ uint4 masks[SNB_NLC_GROUPS][64];    // near and far ballots of (group, atom)
    __shared__ uint16_t cnts[SNB_NLC_GROUPS][64];  // their counts: near | far << 8
    __shared__ uint16_t cslot[SNB_NLC_CAP];
    __shared__ uint64_t reach_s[64];
    __shared__ int run_off[SNB_NLC_MAXRUN + 1];
    __shared__ int run_p0[SNB_NLC_MAXRUN];
    __shared__ int run_slot0[SNB_NLC_MAXRUN];
    const int c = bid;
    const int cb = start[c], m = start[c + 1] - cb;
    if (m == 0) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cz = c % W.nz, cy = (c / W.nz) % W.ny, cx = c / (W.nz * W.ny);
    const int x0 = (cx / W.a) * W.a, y0 = (cy / W.b) * W.b, z0 = (cz / W.s) * W.s;
    if (wave == 0) win_table_wave(W, start, x0, y0, z0, lane, first, pref);
    __syncthreads();
    if (pref[SNB_WIN_MAX_RANGES] > 65535)
    {
        // the window does not fit 16-bit slots: no rows, flagged
        for (int a = tid; a < m; a += blockDim.x)
        {
            row_count[cb + a] = 0;
            row_split[cb + a] = 0;
        }
        if (tid == 0) atomicOr(status, SNB_FLAG_NL_OVERFLOW);
        return;
    }
    if (wave == 0)
    {
        // lane r builds run r: the own column holds 3 cells (cz .. cz + 2),
        // the 12 others 5 (cz - 2 .. cz + 2); sizes are then scanned
        int size = 0;
        if (lane < SNB_NLC_MAXRUN)
        {
            int col, zu;
            if (lane < 3)
            {
                col = 0;
                zu = cz + lane;
            }
            else
            {
                col = 1 + (lane - 3) / 5;
                zu = cz - 2 + (lane - 3) % 5;
            }
            int dx, dy;
            if (col < 3)
            {
                dx = 0;
                dy = col;
            }
            else
            {
                dx = 1 + (col - 3) / 5;
                dy = (col - 3) % 5 - 2;
            }
            const int u = (cx - x0) + dx, v = (cy - y0) + dy + 2;
            const int base = (snb_wrap(cx + dx, W.nx) * W.ny + snb_wrap(cy + dy, W.ny)) * W.nz;
            // zu unwrapped: the window range and the order of the cells
            const int zw = snb_wrap(zu, W.nz);
            const int k = snb_win_range_of(W, z0, u, v, zu - z0 + 2);
            const int p0 = start[base + zw], p1 = start[base + zw + 1];
            run_p0[lane] = p0;
            run_slot0[lane] = pref[k] + (p0 - first[k]);
            size = p1 - p0;
        }
        int incl = size;
        for (int off = 1; off < 64; off <<= 1)
        {
            const int up = __shfl_up(incl, off);
            if (lane >= off) incl += up;
        }
        if (lane < SNB_NLC_MAXRUN) run_off[lane] = incl - size;
        if (lane == SNB_NLC_MAXRUN - 1) run_off[SNB_NLC_MAXRUN] = incl;
    }
    __syncthreads();
    const int total = __builtin_amdgcn_readfirstlane(run_off[SNB_NLC_MAXRUN]);
    const SnbConstF4 cell_crd = (SnbConstF4)(sorted_crd + cb);
    // lane r: where run r lies in the stencil
    const int rcol = lane < 3 ? 0 : 1 + (lane - 3) / 5;
    const int rdx = rcol < 3 ? 0 : 1 + (rcol - 3) / 5;
    const int rdy = rcol < 3 ? rcol : (rcol - 3) % 5 - 2;
    const int rdz = lane < 3 ? lane : (lane - 3) % 5 - 2;
    for (int a0 = 0; a0 < m; a0 += 64)
    {
        const int ma = m - a0 < 64 ? m - a0 : 64;
        // lane a: atom a0 + a of the cell
        float4 qa = make_float4(__builtin_nanf(""), 0.0f, 0.0f, 0.0f);
        qa.y = qa.z = qa.x;
        int ilo = 0, iwid = 0;  // the id window of its exclusions
        if (lane < ma)
        {
            qa = sorted_crd[cb + a0 + lane];
            if (ex_num)
            {
                const int2 r = ex_rng[__float_as_int(qa.w)];
                ilo = r.x >= 0 ? r.x : ~r.x;
                iwid = r.y - ilo + 1;
            }
        }
        // stencil cells within reach of atom a: per axis the gap from its
        // wrapped position (the binning's arithmetic) to the cell, a lower
        // bound of the minimum-image distance
        for (int a = wave; a < ma; a += SNB_NLC_WAVES)
        {
            uint64_t reach = ~0ull;
            if (ORTHO)
            {
                const float qx = readlane_f(qa.x, a), qy = readlane_f(qa.y, a),
                            qz = readlane_f(qa.z, a);
                const float xw = qx - floorf(qx / box.c[0]) * box.c[0];
                const float yw = qy - floorf(qy / box.c[2]) * box.c[2];
                const float zw = qz - floorf(qz / box.c[5]) * box.c[5];
                auto gap = [](int d, int c, float x, float w) -> float {
                    float g = d > 0 ? (float)(c + d) * w - x
                                    : (d < 0 ? x - (float)(c + d + 1) * w : 0.0f);
                    return g > 0.0f ? g : 0.0f;
                };
                const float gx = gap(rdx, cx, xw, wx), gy = gap(rdy, cy, yw, wy),
                            gz = gap(rdz, cz, zw, wz);
                reach = __ballot(lane < SNB_NLC_MAXRUN &&
                                 (gx * gx + gy * gy) + gz * gz < cs2 + 0.05f);
            }
            if (lane == 0) reach_s[a] = reach;
        }
        const float lo3[3] = {wave_fmin(qa.x), wave_fmin(qa.y), wave_fmin(qa.z)};
        const float hi3[3] = {wave_fmax(qa.x), wave_fmax(qa.y), wave_fmax(qa.z)};
        __syncthreads();
        const uint64_t reach_a = lane < ma ? reach_s[lane] : 0ull;
        int near0 = 0, far0 = 0;  // the entries of row a so far
        for (int chunk0 = 0; chunk0 < total; chunk0 += SNB_NLC_CAP)
        {
            const int clen = total - chunk0 < SNB_NLC_CAP ? total - chunk0 : SNB_NLC_CAP;
            const int ngroup = (clen + 63) >> 6;
            for (int k = wave; k < ngroup; k += SNB_NLC_WAVES)
            {
                const int t = k * 64 + lane, g0 = chunk0 + k * 64;
                const bool valid = t < clen;
                // the last run starting at or before the candidate (empty runs
                // share offsets)
                const int g = valid ? g0 + lane : chunk0 + clen - 1;
                int lo = 0, hi = SNB_NLC_MAXRUN - 1;
                while (lo < hi)
                {
                    const int mid = (lo + hi + 1) >> 1;
                    if (run_off[mid] <= g)
                        lo = mid;
                    else
                        hi = mid - 1;
                }
                const int off = g - run_off[lo];
                const float4 qj = sorted_crd[run_p0[lo] + off];
                const int id_j = __float_as_int(qj.w);
                cslot[t] = (uint16_t)(run_slot0[lo] + off);
                int jlo = 0, jwid = 0;
                if (ex_num)
                {
                    const int2 r = ex_rng[id_j];
                    jlo = r.x >= 0 ? r.x : ~r.x;
                    jwid = r.y - jlo + 1;
                }
                // the image shifts, where they are the same for the whole cell
                const float qj3[3] = {qj.x, qj.y, qj.z};
                float sh[3] = {0.0f, 0.0f, 0.0f};
                bool same = ORTHO;
                if (ORTHO)
                {
                    const float rc3[3] = {box.rc[0], box.rc[2], box.rc[5]};
                    const float c3[3] = {box.c[0], box.c[2], box.c[5]};
#pragma unroll
                    for (int d = 0; d < 3; d++)
                    {
                        // rint(s) == floorf(s + 0.5) for every pair within
                        // rc + skin (s lies within (rc + skin)/L < 1/2 of an
                        // integer); they differ only half a box away
                        const float k0 = rintf((lo3[d] - qj3[d]) * rc3[d]);
                        const float k1 = rintf((hi3[d] - qj3[d]) * rc3[d]);
                        same = same && k0 == k1;
                        sh[d] = k0 * c3[d];
                        asm volatile("" : "+v"(sh[d]));  // here, not once per atom
                    }
                }
                const bool fold = __ballot(!same) != 0;
                const int r0 = __builtin_amdgcn_readlane(lo, 0);
                const int r1 = __builtin_amdgcn_readlane(lo, 63);
                const uint64_t live = __ballot(valid);
                const bool own = g0 < m;
                uint64_t todo = __ballot((reach_a & (((2ull << (r1 - r0)) - 1ull) << r0)) != 0);
                uint2 mnear = make_uint2(0u, 0u), mfar = make_uint2(0u, 0u);
                while (todo)
                {
                    const int a = __builtin_ctzll(todo);
                    todo &= todo - 1;
                    const SnbF4 qi = cell_crd[a0 + a];
                    const int id_i = __float_as_int(qi.w);
                    float ddx = qi.x - qj.x, ddy = qi.y - qj.y, ddz = qi.z - qj.z;
                    if (!fold)
                    {
                        ddx = ddx - sh[0];
                        ddy = ddy - sh[1];
                        ddz = ddz - sh[2];
                    }
                    else if (ORTHO)
                    {
                        const float kx = rintf(ddx * box.rc[0]);
                        const float ky = rintf(ddy * box.rc[2]);
                        const float kz = rintf(ddz * box.rc[5]);
                        ddx = ddx - kx * box.c[0];
                        ddy = ddy - ky * box.c[2];
                        ddz = ddz - kz * box.c[5];
                    }
                    else
                    {
                        float sx = (ddx * box.rc[0] + ddy * box.rc[1]) + ddz * box.rc[3];
                        float sy = ddy * box.rc[2] + ddz * box.rc[4];
                        float sz = ddz * box.rc[5];
                        float kx = floorf(sx + 0.5f), ky = floorf(sy + 0.5f),
                              kz = floorf(sz + 0.5f);
                        ddx = ddx - ((kx * box.c[0] + ky * box.c[1]) + kz * box.c[3]);
                        ddy = ddy - (ky * box.c[2] + kz * box.c[4]);
                        ddz = ddz - kz * box.c[5];
                    }
                    const float d2 = (ddx * ddx + ddy * ddy) + ddz * ddz;
                    uint64_t ok = __ballot(d2 < cs2) & live;
                    const uint64_t nearp = __ballot(d2 < near2);
                    // the cell's own atoms come first: larger sorted index only
                    if (own && g0 <= a0 + a)
                    {
                        const int skip = a0 + a - g0 + 1;
                        ok = skip < 64 ? ok & (~0ull << skip) : 0ull;
                    }
                    // the lower id's list decides; its id window rules out
                    // most pairs without touching the list, and decides alone
                    // for a list of consecutive ids (first stored >= 0)
                    const int wlo = __builtin_amdgcn_readlane(ilo, a);
                    const int wwid = __builtin_amdgcn_readlane(iwid, a);
                    const uint64_t maybe =
                        (__ballot((unsigned)(id_j - wlo) < (unsigned)wwid) |
                         __ballot((unsigned)(id_i - jlo) < (unsigned)jwid)) & ok;
                    if (maybe)
                    {
                        bool ex = false;
                        if ((maybe >> lane) & 1)
                        {
                            const int lo_id = id_i < id_j ? id_i : id_j;
                            const int hi_id = id_i < id_j ? id_j : id_i;
                            const int2 rl = ex_rng[lo_id];
                            if (hi_id >= (rl.x >= 0 ? rl.x : ~rl.x) && hi_id <= rl.y)
                                ex = rl.x >= 0 ||
                                     excluded_pair(id_i, id_j, ex_start, ex_list, ex_num);
                        }
                        ok &= ~__ballot(ex);
                    }
                    const uint64_t mn = ok & nearp, mf = ok & ~nearp;
                    mnear.x = snb_writelane((unsigned)mn, a, mnear.x);
                    mnear.y = snb_writelane((unsigned)(mn >> 32), a, mnear.y);
                    mfar.x = snb_writelane((unsigned)mf, a, mfar.x);
                    mfar.y = snb_writelane((unsigned)(mf >> 32), a, mfar.y);
                }
                masks[k][lane] = make_uint4(mnear.x, mnear.y, mfar.x, mfar.y);
                cnts[k][lane] = (uint16_t)((__popc(mnear.x) + __popc(mnear.y)) |
                                           ((__popc(mfar.x) + __popc(mfar.y)) << 8));
            }
            __syncthreads();
            // Near pairs (within rc + skin/4, the ones that can come into
            // range before the next rebuild) from the front, the rest from
            // the back: the pair kernel meets them in that order and whole
            // wavefronts of far pairs skip the force evaluation.
            for (int k = 0; k < ngroup; k++)
            {
                if (k % SNB_NLC_WAVES == wave)
                {
                    const uint4 mk = masks[k][lane];
                    const int slot = cslot[k * 64 + lane];
                    uint64_t todo = __ballot((mk.x | mk.y | mk.z | mk.w) != 0);
                    while (todo)
                    {
                        const int a = __builtin_ctzll(todo);
                        todo &= todo - 1;
                        const uint64_t mn = lane_value(make_uint2(mk.x, mk.y), a);
                        const uint64_t mf = lane_value(make_uint2(mk.z, mk.w), a);
                        const int pn = __builtin_amdgcn_readlane(near0, a) + mbcnt(mn);
                        const int pf = max_nb - 1 - __builtin_amdgcn_readlane(far0, a) - mbcnt(mf);
                        const int pos = __builtin_amdgcn_inverse_ballot_w64(mn) ? pn : pf;
                        if (__builtin_amdgcn_inverse_ballot_w64(mn | mf) &&
                            (unsigned)pos < (unsigned)max_nb)
                            nl16[(size_t)(cb + a0 + a) * max_nb + pos] = (uint16_t)slot;
                    }
                }
                const int v = cnts[k][lane];
                near0 += v & 255;
                far0 += v >> 8;
            }
            __syncthreads();
        }
        if (wave == 0 && lane < ma)
        {
            // an overflowing row (flagged) keeps max_nb valid slots
            row_count[cb + a0 + lane] = near0 + far0 < max_nb ? near0 + far0 : max_nb;
            row_split[cb + a0 + lane] = near0 < max_nb ? near0 : max_nb;
            if (near0 + far0 > max_nb) atomicOr(status, SNB_FLAG_NL_OVERFLOW);
        }
    }
}

template <bool ORTHO>
__global__ void __launch_bounds__(64 * SNB_NLC_WAVES, 8) k_nl_build_cell(
    const int* __restrict__ need, SnbWin W, const int* __restrict__ start,
    const float4* __restrict__ sorted_crd, SnbBox box, float cs2,
    const int* __restrict__ ex_start, const int* __restrict__ ex_list,
    const int* __restrict__ ex_num, const int2* __restrict__ ex_rng, int max_nb, float near2,
    uint16_t* __restrict__ nl16, int* __restrict__ row_count, int* __restrict__ row_split,
    int* __restrict__ status, float wx, float wy, float wz)
{
    k_nl_build_cell_body<ORTHO>(
        need, W, start, sorted_crd, box, cs2, ex_start, ex_list, ex_num, ex_rng, max_nb, near2,
        nl16, row_count, row_split, status, wx, wy, wz, blockIdx.x, gridDim.x);
}

struct NlBuildCellArgs
{
    const int* need;
    SnbWin W;
    const int* start;
    const float4* sorted_crd;
    SnbBox box;
    float cs2;
    const int* ex_start;
    const int* ex_list;
    const int* ex_num;
    const int2* ex_rng;
    int max_nb;
    float near2;
    uint16_t* nl16;
    int* row_count;
    int* row_split;
    int* status;
    float wx;
    float wy;
    float wz;
};

template <bool ORTHO>
__global__ void __launch_bounds__(64 * SNB_NLC_WAVES, 8) k_nl_build_cell_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const NlBuildCellArgs& a = snb_seg<NlBuildCellArgs>(t, bid, nbid);
    k_nl_build_cell_body<ORTHO>(
        a.need, a.W, a.start, a.sorted_crd, a.box, a.cs2, a.ex_start, a.ex_list, a.ex_num, a.ex_rng,
        a.max_nb, a.near2, a.nl16, a.row_count, a.row_split, a.status, a.wx, a.wy, a.wz, bid, nbid);
}

// The rows of the block at (x0, y0, z0), 64 at a time, column by column:
// visit(row or beyond the column's end, column, near entries, far entries).
template <class V>
__device__ __forceinline__ void each_block_rows(const SnbWin& W, int x0, int y0, int z0, int lane,
                                                const int* __restrict__ start,
                                                const int* __restrict__ row_count,
                                                const int* __restrict__ row_split, V&& visit)
{
    const int z1 = z0 + W.s < W.nz ? z0 + W.s : W.nz;
    for (int ua = 0; ua < W.a; ua++)
        for (int vb = 0; vb < W.b; vb++)
        {
            if (x0 + ua >= W.nx || y0 + vb >= W.ny) continue;
            const int colbase = ((x0 + ua) * W.ny + (y0 + vb)) * W.nz;
            const int e = start[colbase + z1];
            for (int s0 = start[colbase + z0]; s0 < e; s0 += 64)
            {
                const int si = s0 + lane;
                int near = 0, far = 0;
                if (si < e)
                {
                    near = row_split[si];
                    far = row_count[si] - near;
                }
                visit(si, ua * W.wv + vb + 2, near, far);
            }
        }
}

// Units of one row (snb_window.h) and their cost in the pair kernel's
// instructions: about 50 for any unit, 60 more per 64 near entries.
__device__ __forceinline__ int units_of(int near, int far)
{
    return ((near + 127) >> 7) + ((far + 127) >> 7);
}
__device__ __forceinline__ int unit_cost(bool far, int entries)
{
    return far ? 50 : (entries > 64 ? 170 : 110);
}
__device__ __forceinline__ int row_cost(int near, int far)
{
    const int rest = near & 127;
    return (near >> 7) * unit_cost(false, 128) + (rest ? unit_cost(false, rest) : 0) +
           ((far + 127) >> 7) * unit_cost(true, 0);
}

// Window atoms, units and cost of every block (one wavefront per block).
__device__ __forceinline__ void k_win_sizes_body(const int* __restrict__ need, SnbWin W,
                                                  const int* __restrict__ start,
                                                  const int* __restrict__ row_count,
                                                  const int* __restrict__ row_split,
                                                  int* __restrict__ win_size,
                                                  int* __restrict__ unit_count,
                                                  int* __restrict__ work,
    unsigned bid, unsigned nbid)
{
    if (need[0] == 0) return;
    const int w = bid, lane = threadIdx.x;
    int x0, y0, z0;
    snb_win_block(W, w, x0, y0, z0);
    int size = 0;
    for (int k = lane; k < W.nrange; k += 64)
    {
        int fc, nc;
        snb_win_range_cells(W, x0, y0, z0, k, fc, nc);
        size += nc > 0 ? start[fc + nc] - start[fc] : 0;
    }
    int cost = 0, count = 0;
    each_block_rows(W, x0, y0, z0, lane, start, row_count, row_split,
                    [&](int, int, int near, int far) {
                        cost += row_cost(near, far);
                        count += units_of(near, far);
                    });
    for (int off = 32; off > 0; off >>= 1)
    {
        size += __shfl_xor(size, off);
        cost += __shfl_xor(cost, off);
        count += __shfl_xor(count, off);
    }
    if (lane == 0)
    {
        win_size[w] = size;
        unit_count[w] = count;
        work[w] = cost;
    }
}

__global__ void __launch_bounds__(64) k_win_sizes(const int* __restrict__ need, SnbWin W,
                                                  const int* __restrict__ start,
                                                  const int* __restrict__ row_count,
                                                  const int* __restrict__ row_split,
                                                  int* __restrict__ win_size,
                                                  int* __restrict__ unit_count,
                                                  int* __restrict__ work)
{
    k_win_sizes_body(need, W, start, row_count, row_split, win_size, unit_count, work, blockIdx.x,
                     gridDim.x);
}

struct WinSizesArgs
{
    const int* need;
    SnbWin W;
    const int* start;
    const int* row_count;
    const int* row_split;
    int* win_size;
    int* unit_count;
    int* work;
};

__global__ void __launch_bounds__(64) k_win_sizes_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const WinSizesArgs& a = snb_seg<WinSizesArgs>(t, bid, nbid);
    k_win_sizes_body(a.need, a.W, a.start, a.row_count, a.row_split, a.win_size, a.unit_count,
                     a.work, bid, nbid);
}

// The units of the block whose window table is (first, pref), by one
// wavefront: units[base ..), and the first unit of each of the 16 wavefronts
// of the pair kernel's workgroup, which take contiguous runs of equal cost.
__device__ void write_units(const SnbWin& W, int w, int x0, int y0, int z0, int lane,
                            const int* __restrict__ start, const int* __restrict__ row_count,
                            const int* __restrict__ row_split, int max_nb, const int* first,
                            const int* pref, int cost, int base, int end,
                            int4* __restrict__ units, int* __restrict__ unit_run)
{
    int* run = unit_run + w * SNB_UNIT_RUNS;
    if (lane < SNB_UNIT_RUNS) run[lane] = lane == 0 ? base : end;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    int c0 = 0, t0 = base;  // cost and units before this batch of rows
    const float per_cost = (float)(SNB_UNIT_RUNS - 1) / (float)(cost > 0 ? cost : 1);
    each_block_rows(W, x0, y0, z0, lane, start, row_count, row_split, [&](int si, int col, int near,
                                                                         int far) {
        // the column's own z-cells do not wrap: part 1 of its run when the
        // run starts below z = 0, else part 0
        const int k = 2 * col + (z0 < 2 ? 1 : 0);
        const int slot_d = pref[k] - first[k];
        const int rc = row_cost(near, far), rn = units_of(near, far);
        int ce = rc, te = rn;
        for (int off = 1; off < 64; off <<= 1)
        {
            const int a = __shfl_up(ce, off), b = __shfl_up(te, off);
            if (lane >= off)
            {
                ce += a;
                te += b;
            }
        }
        int c = c0 + ce - rc, t = t0 + te - rn;
        const int near_u = (near + 127) >> 7;
        for (int j = 0; j < rn; j++)
        {
            const bool is_far = j >= near_u;
            const int k0 = (is_far ? j - near_u : j) << 7;
            const int left = (is_far ? far : near) - k0, entries = left < 128 ? left : 128;
            const int at = si * max_nb + (is_far ? max_nb - 128 - k0 : k0) + SNB_NL16_PAD;
            units[t] = make_int4(si, at, si + slot_d,
                                 entries | (is_far ? SNB_UNIT_FAR : 0) |
                                     (j + 1 == rn ? SNB_UNIT_LAST : 0));
            // wavefront v starts at the unit that holds its share's first
            // cost, or after it when that lies in the unit's second half
            const int uc = unit_cost(is_far, entries);
            int v = (int)((float)c * per_cost) - 1;  // at or below the first share >= c
            for (v = v < 1 ? 1 : v; v < SNB_UNIT_RUNS - 1; v++)
            {
                const int share = (int)((long long)cost * v / (SNB_UNIT_RUNS - 1));
                if (share >= c + uc) break;
                if (share >= c) run[v] = 2 * (share - c) < uc ? t : t + 1;
            }
            c += uc;
            t++;
        }
        c0 += __shfl(ce, 63);
        t0 += __shfl(te, 63);
    });
}

// Per block: the atom of every window slot (wslots, at the slot's stage
// position) and that position in the atom's list (the per-step gather sums
// these); one of the four wavefronts writes the block's units instead.
__device__ __forceinline__ void k_stage_inverse_body(
    const int* __restrict__ need, SnbWin W, const int* __restrict__ start,
    const int* __restrict__ stage_base, int* __restrict__ inv_count, int* __restrict__ inv_list,
    int invmax, int* __restrict__ wslots, int wslots_cap, int* __restrict__ status,
    const int* __restrict__ row_count, const int* __restrict__ row_split, int max_nb,
    const int* __restrict__ work, const int* __restrict__ unit_base, int4* __restrict__ units,
    int* __restrict__ unit_run, unsigned bid, unsigned nbid)
{
    if (need[0] == 0) return;
    __shared__ int first[SNB_WIN_MAX_RANGES];
    __shared__ int pref[SNB_WIN_MAX_RANGES + 1];
    int w = bid, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nwave = blockDim.x >> 6;
    int x0, y0, z0;
    snb_win_block(W, w, x0, y0, z0);
    if (wave == 0) win_table_wave(W, start, x0, y0, z0, lane, first, pref);
    __syncthreads();
    if (wave == nwave - 1)
    {
        write_units(W, w, x0, y0, z0, lane, start, row_count, row_split, max_nb, first, pref,
                    work[w], unit_base[w], unit_base[w + 1], units, unit_run);
        return;
    }
    int base = stage_base[w];
    for (int k = wave; k < W.nrange; k += nwave - 1)
    {
        // ranges beyond nrange are empty, so pref[k + 1] is defined for k < nrange <= 128
        int cnt = pref[k + 1] - pref[k];
        for (int t = lane; t < cnt; t += 64)
        {
            int s = first[k] + t;
            const int at = base + pref[k] + t;
            if (at < wslots_cap) wslots[at] = s;
            int idx = atomicAdd(&inv_count[s], 1);
            if (idx < invmax)
                inv_list[(size_t)s * invmax + idx] = at;
            else
                atomicOr(status, SNB_FLAG_NL_OVERFLOW);
        }
    }
}

__global__ void __launch_bounds__(256) k_stage_inverse(
    const int* __restrict__ need, SnbWin W, const int* __restrict__ start,
    const int* __restrict__ stage_base, int* __restrict__ inv_count, int* __restrict__ inv_list,
    int invmax, int* __restrict__ wslots, int wslots_cap, int* __restrict__ status,
    const int* __restrict__ row_count, const int* __restrict__ row_split, int max_nb,
    const int* __restrict__ work, const int* __restrict__ unit_base, int4* __restrict__ units,
    int* __restrict__ unit_run)
{
    k_stage_inverse_body(need, W, start, stage_base, inv_count, inv_list, invmax, wslots,
                         wslots_cap, status, row_count, row_split, max_nb, work, unit_base, units,
                         unit_run, blockIdx.x, gridDim.x);
}

struct StageInverseArgs
{
    const int* need;
    SnbWin W;
    const int* start;
    const int* stage_base;
    int* inv_count;
    int* inv_list;
    int invmax;
    int* wslots;
    int wslots_cap;
    int* status;
    const int* row_count;
    const int* row_split;
    int max_nb;
    const int* work;
    const int* unit_base;
    int4* units;
    int* unit_run;
};

__global__ void __launch_bounds__(256) k_stage_inverse_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const StageInverseArgs& a = snb_seg<StageInverseArgs>(t, bid, nbid);
    k_stage_inverse_body(a.need, a.W, a.start, a.stage_base, a.inv_count, a.inv_list, a.invmax,
                         a.wslots, a.wslots_cap, a.status, a.row_count, a.row_split, a.max_nb,
                         a.work, a.unit_base, a.units, a.unit_run, bid, nbid);
}

// slot -> sorted index through the LDS range table (binary search)
__device__ __forceinline__ int win_slot_to_sorted(const SnbWin& W, const int* first,
                                                  const int* pref, int slot)
{
    int lo = 0, hi = W.nrange - 1;
    while (lo < hi)
    {
        int mid = (lo + hi + 1) >> 1;
        if (pref[mid] <= slot)
            lo = mid;
        else
            hi = mid - 1;
    }
    // skip empty ranges that share the prefix
    return first[lo] + (slot - pref[lo]);
}

// Reference-layout rows, one workgroup per window block: the block's window
// table and, when the window fits, the atom id of every window slot are built
// once in LDS; then every internal row of the block's cells sends each pair
// to row min(id) as max(id).  Pairs whose lower id is the row's own atom are
// appended by the wavefront with one counter add per 64 entries.  The others
// go to rows of other window atoms: a first pass counts them per window slot
// in LDS, each slot reserves one range of its row with a single counter add,
// and a second pass places the entries in that range with LDS counters.  A
// window beyond the map takes one counter add per such entry instead.  The
// order within a row follows the appends (rows are sorted afterwards when
// asked for).
#define SNB_EXPORT_MAP_CAP 8192
__global__ void __launch_bounds__(1024) k_nl_export_block(
    const int* __restrict__ need, SnbWin W, const int* __restrict__ start,
    const int* __restrict__ order, const int* __restrict__ row_count,
    const int* __restrict__ row_split, const uint16_t* __restrict__ nl16, int max_nb,
    int* __restrict__ pub_count, int* __restrict__ serial)
{
    if (need[0] == 0) return;
    __shared__ int first[SNB_WIN_MAX_RANGES];
    __shared__ int pref[SNB_WIN_MAX_RANGES + 1];
    __shared__ int wid[SNB_EXPORT_MAP_CAP];  // atom id of each window slot
    __shared__ int fwd[SNB_EXPORT_MAP_CAP];  // appends to each slot's row, then its next position
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nwave = (int)(blockDim.x >> 6);
    int x0, y0, z0;
    snb_win_block(W, blockIdx.x, x0, y0, z0);
    if (wave == 0) win_table_wave(W, start, x0, y0, z0, lane, first, pref);
    __syncthreads();
    const int total = pref[SNB_WIN_MAX_RANGES];
    const bool use_map = total <= SNB_EXPORT_MAP_CAP;
    if (use_map)
        for (int slot = tid; slot < total; slot += blockDim.x)
        {
            wid[slot] = order[win_slot_to_sorted(W, first, pref, slot)];
            fwd[slot] = 0;
        }
    __syncthreads();
    // the block's own cells (the last block of an axis may be partial); the
    // cells (x0 + u, y0 + v, z0 .. z0 + zs - 1) are consecutive
    const int xa = W.nx - x0 < W.a ? W.nx - x0 : W.a;
    const int yb = W.ny - y0 < W.b ? W.ny - y0 : W.b;
    const int zs = W.nz - z0 < W.s ? W.nz - z0 : W.s;
    auto each_row = [&](auto&& visit) {
        for (int u = 0; u < xa; u++)
            for (int v = 0; v < yb; v++)
            {
                const int c0 = ((x0 + u) * W.ny + (y0 + v)) * W.nz + z0;
                const int sb = start[c0], se = start[c0 + zs];
                for (int srow = sb + wave; srow < se; srow += nwave) visit(srow);
            }
    };
    const uint64_t lower = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    if (use_map)
    {
        each_row([&](int srow) {
            const int id_i = order[srow];
            const int cnt = row_count[srow], split = row_split[srow];
            const uint16_t* row = nl16 + (size_t)srow * max_nb;
            for (int k = lane; k < cnt; k += 64)
            {
                const int slot = row[snb_row_entry(k, split, max_nb)];
                if (wid[slot] < id_i) atomicAdd(&fwd[slot], 1);
            }
        });
        __syncthreads();
        for (int slot = tid; slot < total; slot += blockDim.x)
        {
            const int c = fwd[slot];
            if (c > 0) fwd[slot] = atomicAdd(&pub_count[wid[slot]], c);
        }
        __syncthreads();
        each_row([&](int srow) {
            const int id_i = order[srow];
            const int cnt = row_count[srow], split = row_split[srow];
            const uint16_t* row = nl16 + (size_t)srow * max_nb;
            int* own_row = serial + (size_t)id_i * max_nb;
            for (int k0 = 0; k0 < cnt; k0 += 64)
            {
                const int k = k0 + lane;
                int slot = 0, id_j = -1;
                if (k < cnt)
                {
                    slot = row[snb_row_entry(k, split, max_nb)];
                    id_j = wid[slot];
                }
                const bool own = id_j > id_i;
                const uint64_t m = __ballot(own);
                int base = 0;
                if (lane == 0 && m) base = atomicAdd(&pub_count[id_i], (int)__popcll(m));
                base = __shfl(base, 0);
                if (own)
                {
                    const int pos = base + (int)__popcll(m & lower);
                    if (pos < max_nb) own_row[pos] = id_j;
                }
                else if (id_j >= 0)
                {
                    const int pos = atomicAdd(&fwd[slot], 1);
                    if (pos < max_nb) serial[(size_t)id_j * max_nb + pos] = id_i;
                }
            }
        });
        return;
    }
    each_row([&](int srow) {
        const int id_i = order[srow];
        const int cnt = row_count[srow], split = row_split[srow];
        const uint16_t* row = nl16 + (size_t)srow * max_nb;
        int* own_row = serial + (size_t)id_i * max_nb;
        for (int k0 = 0; k0 < cnt; k0 += 64)
        {
            const int k = k0 + lane;
            int id_j = -1;
            if (k < cnt)
                id_j = order[win_slot_to_sorted(W, first, pref,
                                                row[snb_row_entry(k, split, max_nb)])];
            const bool own = id_j > id_i;
            const uint64_t m = __ballot(own);
            int base = 0;
            if (lane == 0 && m) base = atomicAdd(&pub_count[id_i], (int)__popcll(m));
            base = __shfl(base, 0);
            if (own)
            {
                const int pos = base + (int)__popcll(m & lower);
                if (pos < max_nb) own_row[pos] = id_j;
            }
            else if (id_j >= 0)
            {
                const int pos = atomicAdd(&pub_count[id_j], 1);
                if (pos < max_nb) serial[(size_t)id_j * max_nb + pos] = id_i;
            }
        }
    });
}

// ATOM_GROUP::atom_numbers of every public row (rows in append order).
__global__ void k_nl_pub_counts(const int* __restrict__ need, int n,
                                const int* __restrict__ pub_count, int max_nb,
                                snb_atom_group* __restrict__ nl, int* __restrict__ status)
{
    if (need[0] == 0) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int c = pub_count[i];
    if (c > max_nb)
    {
        atomicOr(status, SNB_FLAG_NL_OVERFLOW);
        c = max_nb;
    }
    nl[i].atom_numbers = c;
    nl[i].ghost_numbers = 0;
}

// Sorts each public row ascending (bitonic, one wavefront per row) and sets
// ATOM_GROUP::atom_numbers.
#define SNB_SORT_CAP 4096
__global__ void __launch_bounds__(64) k_nl_pub_finish(const int* __restrict__ need, int n,
                                                      const int* __restrict__ pub_count,
                                                      int max_nb, int* __restrict__ serial,
                                                      snb_atom_group* __restrict__ nl,
                                                      int* __restrict__ status)
{
    if (need[0] == 0) return;
    __shared__ int v[SNB_SORT_CAP];
    int i = blockIdx.x, lane = threadIdx.x;
    int c = pub_count[i];
    if (c > max_nb)
    {
        if (lane == 0) atomicOr(status, SNB_FLAG_NL_OVERFLOW);
        c = max_nb;
    }
    if (lane == 0)
    {
        nl[i].atom_numbers = c;
        nl[i].ghost_numbers = 0;
    }
    if (c <= 1 || c > SNB_SORT_CAP) return;
    int P = 1;
    while (P < c) P <<= 1;
    int* row = serial + (size_t)i * max_nb;
    for (int t = lane; t < P; t += 64) v[t] = t < c ? row[t] : 0x7fffffff;
    __syncthreads();
    for (int k = 2; k <= P; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1)
        {
            for (int t = lane; t < P; t += 64)
            {
                int p = t ^ j;
                if (p > t)
                {
                    int a = v[t], b = v[p];
                    bool up = (t & k) == 0;
                    if ((a > b) == up)
                    {
                        v[t] = b;
                        v[p] = a;
                    }
                }
            }
            __syncthreads();
        }
    for (int t = lane; t < c; t += 64) row[t] = v[t];
}

// The same sort with one wavefront per row and four rows per workgroup, each
// wavefront in its own LDS slab (rows up to SNB_SORT_WAVE_CAP entries); the
// compare-exchange stages need no workgroup barrier because a wavefront
// executes its LDS operations in order.
#define SNB_SORT_WAVE_CAP 2048
__global__ void __launch_bounds__(256) k_nl_pub_finish_wave(const int* __restrict__ need, int n,
                                                           const int* __restrict__ pub_count,
                                                           int max_nb, int* __restrict__ serial,
                                                           snb_atom_group* __restrict__ nl,
                                                           int* __restrict__ status)
{
    if (need[0] == 0) return;
    __shared__ int slab[4][SNB_SORT_WAVE_CAP];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = blockIdx.x * 4 + wave;
    if (i >= n) return;
    int c = pub_count[i];
    if (c > max_nb)
    {
        if (lane == 0) atomicOr(status, SNB_FLAG_NL_OVERFLOW);
        c = max_nb;
    }
    if (lane == 0)
    {
        nl[i].atom_numbers = c;
        nl[i].ghost_numbers = 0;
    }
    if (c <= 1) return;
    int* v = slab[wave];
    int P = 1;
    while (P < c) P <<= 1;
    int* row = serial + (size_t)i * max_nb;
    for (int t = lane; t < P; t += 64) v[t] = t < c ? row[t] : 0x7fffffff;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int k = 2; k <= P; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1)
        {
            for (int t = lane; t < P; t += 64)
            {
                const int p = t ^ j;
                if (p > t)
                {
                    const int a = v[t], b = v[p];
                    const bool up = (t & k) == 0;
                    if ((a > b) == up)
                    {
                        v[t] = b;
                        v[p] = a;
                    }
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    for (int t = lane; t < c; t += 64) row[t] = v[t];
}

// Test hook: the internal rows with atom ids, indexed by the owner's id.
__global__ void __launch_bounds__(64) k_nl_copy_internal(int n, SnbWin W,
                                                         const int* __restrict__ start,
                                                         const int* __restrict__ sorted_cell,
                                                         const int* __restrict__ order,
                                                         const int* __restrict__ row_count,
                                                         const int* __restrict__ row_split,
                                                         const uint16_t* __restrict__ nl16,
                                                         int max_nb, int* __restrict__ counts,
                                                         int* __restrict__ rows)
{
    __shared__ int first[SNB_WIN_MAX_RANGES];
    __shared__ int pref[SNB_WIN_MAX_RANGES + 1];
    int s = blockIdx.x, lane = threadIdx.x;
    int cx, cy, cz, x0, y0, z0;
    win_block_of_cell(W, sorted_cell[s], cx, cy, cz, x0, y0, z0);
    win_table_wave(W, start, x0, y0, z0, lane, first, pref);
    __syncthreads();
    int id_i = order[s];
    int cnt = row_count[s], split = row_split[s];
    if (lane == 0) counts[id_i] = cnt;
    for (int k = lane; k < cnt; k += 64)
        rows[(size_t)id_i * max_nb + k] = order[win_slot_to_sorted(
            W, first, pref, nl16[(size_t)s * max_nb + snb_row_entry(k, split, max_nb)])];
}

// Per sorted position: its LJ type, no stage entries yet.  Per atom id (with
// exclusions): first and last entry of its exclusion list (an empty window
// (1, 0) when it has none), the window the reference tests before searching
// the list (neighbor_list.cpp:594-665).
__device__ __forceinline__ void k_win_atoms_body(const int* __restrict__ need, int n,
                                                 const int* __restrict__ order,
                                                 const int* __restrict__ type,
                                                 int* __restrict__ stype,
                                                 int* __restrict__ inv_count,
                                                 const int* __restrict__ ex_start,
                                                 const int* __restrict__ ex_list,
                                                 const int* __restrict__ ex_num,
                                                 int2* __restrict__ ex_rng,
    unsigned bid, unsigned nbid)
{
    if (need[0] == 0) return;
    int i = bid * blockDim.x + threadIdx.x;
    if (i >= n) return;
    stype[i] = type[order[i]];
    inv_count[i] = 0;
    if (!ex_num) return;
    int en = ex_num[i];
    int2 r = make_int2(1, 0);
    if (en > 0)
    {
        int es = ex_start[i];
        r = make_int2(ex_list[es], ex_list[es + en - 1]);
        // a list that is exactly first, first + 1, ..., last holds every id of
        // its window, so the window test alone decides; other lists are
        // marked (first stored as ~first) and searched
        bool run = r.y - r.x == en - 1;
        for (int t = 1; run && t < en; t++) run = ex_list[es + t] == r.x + t;
        if (!run) r.x = ~r.x;
    }
    ex_rng[i] = r;
}

__global__ void k_win_atoms(const int* __restrict__ need, int n, const int* __restrict__ order,
                            const int* __restrict__ type, int* __restrict__ stype,
                            int* __restrict__ inv_count, const int* __restrict__ ex_start,
                            const int* __restrict__ ex_list, const int* __restrict__ ex_num,
                            int2* __restrict__ ex_rng)
{
    k_win_atoms_body(need, n, order, type, stype, inv_count, ex_start, ex_list, ex_num, ex_rng,
                     blockIdx.x, gridDim.x);
}

struct WinAtomsArgs
{
    const int* need;
    int n;
    const int* order;
    const int* type;
    int* stype;
    int* inv_count;
    const int* ex_start;
    const int* ex_list;
    const int* ex_num;
    int2* ex_rng;
};

__global__ void k_win_atoms_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const WinAtomsArgs& a = snb_seg<WinAtomsArgs>(t, bid, nbid);
    k_win_atoms_body(a.need, a.n, a.order, a.type, a.stype, a.inv_count, a.ex_start, a.ex_list,
                     a.ex_num, a.ex_rng, bid, nbid);
}

// Launch order of the pair kernel's blocks: descending work (ties by block
// index), one workgroup bitonic sort; identity when there are more blocks
// than SNB_ORDER_CAP.
#define SNB_ORDER_CAP 4096
__device__ __forceinline__ void block_order(int nblock, const int* __restrict__ work,
                                            int* __restrict__ perm)
{
    __shared__ long long key[SNB_ORDER_CAP];
    if (nblock > SNB_ORDER_CAP)
    {
        for (int t = threadIdx.x; t < nblock; t += blockDim.x) perm[t] = t;
        return;
    }
    int P = 1;
    while (P < nblock) P <<= 1;
    // key: -work in the high word, index in the low word; padding sorts last
    for (int t = threadIdx.x; t < P; t += blockDim.x)
        key[t] = t < nblock ? (-(long long)work[t]) * 4294967296ll + (long long)t
                            : 0x7fffffffffffffffll;
    __syncthreads();
    for (int k = 2; k <= P; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1)
        {
            for (int t = threadIdx.x; t < P; t += blockDim.x)
            {
                int q = t ^ j;
                if (q > t)
                {
                    long long a = key[t], b = key[q];
                    bool up = (t & k) == 0;
                    if ((a > b) == up)
                    {
                        key[t] = b;
                        key[q] = a;
                    }
                }
            }
            __syncthreads();
        }
    for (int t = threadIdx.x; t < nblock; t += blockDim.x)
        perm[t] = (int)(key[t] & 0xffffffffll);  // low word: the block index (>= 0)
}

// out[k] = in[0] + .. + in[k - 1] for k = 0 .. n, by one workgroup of 1024
__device__ __forceinline__ void block_scan(const int* __restrict__ in, int* __restrict__ out, int n)
{
    __shared__ int part[1024];
    const int t = threadIdx.x, chunk = (n + 1023) / 1024;
    const int b = min(t * chunk, n), e = min(b + chunk, n);
    int s = 0;
    for (int i = b; i < e; i++) s += in[i];
    part[t] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1)
    {
        const int v = t >= off ? part[t - off] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int run = t > 0 ? part[t - 1] : 0;
    for (int i = b; i < e; i++)
    {
        const int v = in[i];
        out[i] = run;
        run += v;
    }
    if (t == 1023) out[n] = part[1023];
}

// Three workgroups: first stage slot of every block, first unit of every
// block, the launch order.
__device__ __forceinline__ void k_block_tables_body(const int* __restrict__ need, int nblock,
                                                    const int* __restrict__ win_size,
                                                    int* __restrict__ stage_base,
                                                    const int* __restrict__ unit_count,
                                                    int* __restrict__ unit_base,
                                                    const int* __restrict__ work,
                                                    int* __restrict__ perm,
    unsigned bid, unsigned nbid)
{
    if (need[0] == 0) return;
    if (bid == 2)
        block_order(nblock, work, perm);
    else
        block_scan(bid == 0 ? win_size : unit_count, bid == 0 ? stage_base : unit_base, nblock);
}

__global__ void __launch_bounds__(1024) k_block_tables(const int* __restrict__ need, int nblock,
                                                       const int* __restrict__ win_size,
                                                       int* __restrict__ stage_base,
                                                       const int* __restrict__ unit_count,
                                                       int* __restrict__ unit_base,
                                                       const int* __restrict__ work,
                                                       int* __restrict__ perm)
{
    k_block_tables_body(need, nblock, win_size, stage_base, unit_count, unit_base, work, perm,
                        blockIdx.x, gridDim.x);
}

struct BlockTablesArgs
{
    const int* need;
    int nblock;
    const int* win_size;
    int* stage_base;
    const int* unit_count;
    int* unit_base;
    const int* work;
    int* perm;
};

__global__ void __launch_bounds__(1024) k_block_tables_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const BlockTablesArgs& a = snb_seg<BlockTablesArgs>(t, bid, nbid);
    k_block_tables_body(a.need, a.nblock, a.win_size, a.stage_base, a.unit_count, a.unit_base,
                        a.work, a.perm, bid, nbid);
}

// Clears p[0 .. n) on rebuild steps only.
__device__ __forceinline__ void k_fill_need_body(const int* __restrict__ need, int* __restrict__ p, int n,
    unsigned bid, unsigned nbid)
{
    if (need[0] == 0) return;
    int i = bid * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void k_fill_need(const int* __restrict__ need, int* __restrict__ p, int n)
{
    k_fill_need_body(need, p, n, blockIdx.x, gridDim.x);
}

struct FillNeedArgs
{
    const int* need;
    int* p;
    int n;
};

__global__ void k_fill_need_batch(SnbSegTab t)
{
    unsigned bid, nbid;
    const FillNeedArgs& a = snb_seg<FillNeedArgs>(t, bid, nbid);
    k_fill_need_body(a.need, a.p, a.n, bid, nbid);
}

// Called after the cell sort of a rebuild (same device flag).
int snb_launch_nl_window(snb_context* ctx, const SnbBox& box, const int* ex_start,
                         const int* ex_list, const int* ex_num)
{
    SnbNl& L = ctx->nl;
    hipStream_t s = ctx->stream;
    int n = ctx->n;
    const SnbWin& W = L.win;
    SNB_LAUNCH_B(k_win_atoms, k_win_atoms_batch, WinAtomsArgs, dim3((n + 255) / 256), dim3(256), 0,
                 s, L.need, n, L.order, ctx->type, ctx->stype, L.inv_count, ex_start, ex_list,
                 ex_num, L.ex_rng);
    float w[3];
    snb_cell_widths(L, box, w);
    const bool ortho = box.c[1] == 0.0f && box.c[3] == 0.0f && box.c[4] == 0.0f &&
                       box.rc[1] == 0.0f && box.rc[3] == 0.0f && box.rc[4] == 0.0f;
    if (ortho)
        SNB_LAUNCH_B(k_nl_build_cell<true>, k_nl_build_cell_batch<true>, NlBuildCellArgs,
                     dim3(L.ncell), dim3(64 * SNB_NLC_WAVES), 0, s, L.need, W, L.cell_start, L.sorted_crd, box,
                     L.cs2, ex_start, ex_list, ex_num, L.ex_rng, L.max_nb, L.near2, L.nl16,
                     L.row_count, L.row_split, ctx->status, w[0], w[1], w[2]);
    else
        SNB_LAUNCH_B(k_nl_build_cell<false>, k_nl_build_cell_batch<false>, NlBuildCellArgs,
                     dim3(L.ncell), dim3(64 * SNB_NLC_WAVES), 0, s, L.need, W, L.cell_start, L.sorted_crd, box,
                     L.cs2, ex_start, ex_list, ex_num, L.ex_rng, L.max_nb, L.near2, L.nl16,
                     L.row_count, L.row_split, ctx->status, w[0], w[1], w[2]);
    SNB_LAUNCH_B(k_win_sizes, k_win_sizes_batch, WinSizesArgs, dim3(W.nblock), dim3(64), 0, s,
                 L.need, W, L.cell_start, L.row_count, L.row_split, L.win_size, L.unit_count,
                 L.block_work);
    SNB_LAUNCH_B(k_block_tables, k_block_tables_batch, BlockTablesArgs, dim3(3), dim3(1024), 0, s,
                 L.need, W.nblock, L.win_size, L.stage_base, L.unit_count, L.unit_base,
                 L.block_work, L.block_perm);
    SNB_LAUNCH_B(k_stage_inverse, k_stage_inverse_batch, StageInverseArgs, dim3(W.nblock),
                 dim3(256), 0, s, L.need, W, L.cell_start, L.stage_base, L.inv_count, L.inv_list,
                 L.invmax, L.wslots, n * L.invmax, ctx->status, L.row_count, L.row_split, L.max_nb,
                 L.block_work, L.unit_base, L.units, L.unit_run);
    SNB_CHECK(hipGetLastError());
    if (L.export_mode)
    {
        SNB_LAUNCH_B(k_fill_need, k_fill_need_batch, FillNeedArgs, dim3((n + 255) / 256), dim3(256),
                     0, s, L.need, L.pub_count, n);
        SNB_LAUNCH(k_nl_export_block, dim3(W.nblock), dim3(1024), 0, s, L.need, W, L.cell_start,
                   L.order, L.row_count, L.row_split, L.nl16, L.max_nb, L.pub_count, L.serial);
        if (L.export_mode == 1)
            SNB_LAUNCH(k_nl_pub_counts, dim3((n + 255) / 256), dim3(256), 0, s, L.need, n,
                       L.pub_count, L.max_nb, L.dnl, ctx->status);
        else if (L.max_nb <= SNB_SORT_WAVE_CAP)
            SNB_LAUNCH(k_nl_pub_finish_wave, dim3((n + 3) / 4), dim3(256), 0, s, L.need, n,
                       L.pub_count, L.max_nb, L.serial, L.dnl, ctx->status);
        else
            SNB_LAUNCH(k_nl_pub_finish, dim3(n), dim3(64), 0, s, L.need, n, L.pub_count, L.max_nb,
                       L.serial, L.dnl, ctx->status);
        SNB_CHECK(hipGetLastError());
    }
    return SNB_OK;
}

int snb_launch_nl_copy_internal(snb_context* ctx, int* counts, int* rows)
{
    SnbNl& L = ctx->nl;
    if (ctx->n <= 0) return SNB_OK;
    SNB_LAUNCH(k_nl_copy_internal,
               dim3(ctx->n), dim3(64), 0, ctx->stream, ctx->n, L.win, L.cell_start, L.sorted_cell, L.order, L.row_count, L.row_split, L.nl16, L.max_nb, counts, rows);
    SNB_CHECK(hipGetLastError());
    return SNB_OK;
}
