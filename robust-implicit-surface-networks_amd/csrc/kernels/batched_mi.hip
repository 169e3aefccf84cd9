// Batched form of the material-interface path (src/material_interface.cpp:53-447).
//
// The plain form's stages (highest material, filter, CSR, cut lists, the
// per-tet cut by table or lane group, boundary-face pairing, extraction,
// dedup, coordinates, faces) with every size kept on
// the device: buffers are allocated to capacities, launches are sized by the
// capacities and read the live counts from device memory (clamped, and
// skipped once a count overflowed).  So the path after the first kernel is one
// captured graph per workspace, replayed on every run and for any values: the
// first kernel, launched with the values, leaves their address for it.  An
// overflow grows the workspace and captures again.  The closing kernel
// publishes the counters into pinned host memory and clears them, so a replay
// needs no copies.  A complex beyond the lane-group cut's capacity sends the
// run to the plain form.
#include <algorithm>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>

#include "kernels_ia.h"
#include "kernels_mi.h"
#include "pipeline.h"
#include "scan_sort.h"

namespace rin {

namespace {

// device counters of one run
enum MICtr : uint32_t {
    M_DEGEN = 0,   // vertices with tied maxima
    M_ACTIVE,      // active tets
    M_LIST,        // cut list sizes [4], histogram [3], 3..4 / 5..8 counts, largest count (k_bucket_scan)
    M_WORDS = M_LIST + 10,  // record words
    M_VO, M_FO, M_FV,  // vertex occurrences, faces, face corners
    M_NV,          // vertices after dedup
    M_FIT,         // active (tet, material) entries: the CSR's total
    M_EMIT,        // tet-boundary faces among the faces (MIEmits)
    M_ABORT,       // a count exceeded its capacity: later stages process nothing
    M_N
};
// kMiHuge: a tet has more than 8 materials (the wide cut takes it)
constexpr uint32_t kMiOverflow = 1u << 8, kMiPlain = 1u << 9, kMiHuge = 1u << 10;
constexpr int kMiPub = 32;
static_assert(M_N <= kMiPub, "published counters");

struct MICaps {
    uint32_t active = 0, fit = 0, words = 0, vo = 0, fo = 0, fv = 0;
    uint32_t huge = 0;  // the captured path holds the wide cut
};

__global__ void k_mi_zero(uint32_t* ctr, uint32_t* errs) {
    if (threadIdx.x < M_N) ctr[threadIdx.x] = 0;
    if (threadIdx.x < 64) errs[threadIdx.x] = 0;
}

// Filter, CSR, active list, cut lists and record slots by tiles of 1280 tets
// (a workgroup of 256 lanes, five consecutive tets a lane: a cube of a regular
// grid): a count pass leaves each tet's material mask and each tile's sums,
// one workgroup turns the sums into prefixes and totals and checks the
// capacities, a fill pass places the tile's tets.  Three launches for what
// took thirteen (a scan of three fields over every tet, the lists' count,
// scan and fill, the slots' bounds and scan, checks and copies): 41 us at 65^3
// vertices and 8 materials, from 100.
constexpr uint32_t kMiLanes = 256, kMiTile = 5 * kMiLanes;
enum MITileField {
    MT_FIT = 0, MT_ACTIVE, MT_LIST, MT_WORDS = MT_LIST + 4,  // prefixes: the CSR, active tets, four lists, slot words
    MT_HIST,                     // totals: two, three and more materials
    MT_N34 = MT_HIST + 3, MT_N58, MT_KMAX, MT_N = 16
};
constexpr int kMiPrefixes = MT_WORDS + 1;
struct MITile {
    uint32_t v[MT_N];
};

// The highest materials at a tet's corners are active; so is every material
// above the lowest of those at two corners or more
// (src/material_interface.cpp:94-152).  Few tets have two materials among
// their corners' highest, so each lane finds its own tets' and the workgroup
// then takes those together, a lane a corner, the loads of eight materials in
// flight (a lane a tet left one lane in twenty busy through 4 F dependent
// loads: 102 us at 100^3 vertices and 18 materials against 65).
__global__ void __launch_bounds__(kMiLanes) k_mi_count_tiles(GridView g, const double* const* vref, uint32_t F,
                                                             const uint64_t* __restrict__ hm, int tables,
                                                             uint64_t* __restrict__ amask,
                                                             MITile* __restrict__ tiles) {
    const double* __restrict__ vals = *vref;
    __shared__ uint64_t s_mask[kMiTile];
    __shared__ uint16_t s_list[kMiTile];
    __shared__ uint32_t s_n;
    const uint64_t V = g.V;
    const uint32_t t0 = blockIdx.x * kMiTile, tid = threadIdx.x;
    if (tid == 0) s_n = 0;
    __syncthreads();
    auto put = [&](uint32_t local, uint64_t u) {
        s_mask[local] = u;
        if (__popcll(u) >= 2) s_list[atomicAdd(&s_n, 1u)] = (uint16_t)local;
    };
    if (g.regular) {
        const uint32_t cube = blockIdx.x * kMiLanes + tid;
        if ((uint64_t)cube * 5 < g.T) {
            const uint32_t R = (uint32_t)g.res, N = R + 1;
            const uint32_t i = cube / (R * R), rem = cube - i * (R * R), j = rem / R, k = rem - j * R;
            const uint32_t b = i * N * N + j * N + k;
            const uint32_t c[8] = {b, b + N * N, b + N * N + N, b + N, b + 1, b + N * N + 1, b + N * N + N + 1, b + N + 1};
            uint64_t h[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) h[q] = hm[c[q]];
            const bool even = ((i + j + k) & 1u) == 0;
            // both parities' tets with indices known here, then one select
#pragma unroll
            for (int q = 0; q < 5; ++q) {
                constexpr auto& E = dev::kCubeTetEven;
                constexpr auto& O = dev::kCubeTetOdd;
                const uint64_t e = h[E[q][0]] | h[E[q][1]] | h[E[q][2]] | h[E[q][3]];
                const uint64_t o = h[O[q][0]] | h[O[q][1]] | h[O[q][2]] | h[O[q][3]];
                put(5 * tid + q, even ? e : o);
            }
        }
    } else {
        for (uint32_t q = tid; q < kMiTile; q += kMiLanes) {
            const uint64_t t = (uint64_t)t0 + q;
            if (t >= g.T) continue;
            uint32_t v[4];
            dev::tet_corners(g, t, v);
            put(q, hm[v[0]] | hm[v[1]] | hm[v[2]] | hm[v[3]]);
        }
    }
    __syncthreads();
    const uint32_t n = s_n;
    for (uint32_t x = tid >> 2; x < n; x += kMiLanes / 4) {
        const uint32_t local = s_list[x], c = tid & 3;
        uint32_t v[4];
        dev::tet_corners(g, (uint64_t)t0 + local, v);
        const double* at = vals + (c == 0 ? v[0] : (c == 1 ? v[1] : (c == 2 ? v[2] : v[3])));
        const uint64_t u = s_mask[local];
        double mn = 1.79769313486231570815e308;
        for (uint64_t m = u; m; m &= m - 1) {
            const double y = at[(uint64_t)(__ffsll((unsigned long long)m) - 1) * V];
            if (y < mn) mn = y;
        }
        uint64_t above = 0;
        for (uint32_t j0 = 0; j0 < F; j0 += 8) {
            double y[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) y[q] = at[(uint64_t)(j0 + q < F ? j0 + q : 0) * V];
#pragma unroll
            for (int q = 0; q < 8; ++q) above |= (uint64_t)(j0 + q < F && y[q] > mn) << (j0 + q);
        }
        // materials above at two corners or more, over the tet's four lanes
        const uint64_t p = __shfl_xor(above, 1, 64), both = above & p, any = above | p;
        const uint64_t both2 = __shfl_xor(both, 2, 64), any2 = __shfl_xor(any, 2, 64);
        if (c == 0) s_mask[local] = u | both | both2 | (any & any2);
    }
    __syncthreads();
    uint32_t s[MT_N];
#pragma unroll
    for (int f = 0; f < MT_N; ++f) s[f] = 0;
    for (uint32_t q = 0; q < 5; ++q) {
        const uint32_t local = 5 * tid + q;
        const uint64_t t = (uint64_t)t0 + local;
        if (t >= g.T) continue;
        const uint64_t m = s_mask[local];
        const int k = __popcll(m);
        if (k < 2) continue;
        s[MT_FIT] += (uint32_t)k;
        s[MT_ACTIVE] += 1;
        const int b = bucket_of_k(k, tables);
#pragma unroll
        for (int z = 0; z < 4; ++z) s[MT_LIST + z] += b == z;
        s[MT_WORDS] += rec_bound(1, k);
        s[MT_HIST] += k == 2;
        s[MT_HIST + 1] += k == 3;
        s[MT_HIST + 2] += k > 3;
        s[MT_N34] += k == 3 || k == 4;
        s[MT_N58] += k >= 5 && k <= 8;
        s[MT_KMAX] = max(s[MT_KMAX], (uint32_t)k);
    }
    for (uint32_t q = tid; q < kMiTile; q += kMiLanes) {
        const uint64_t t = (uint64_t)t0 + q;
        if (t < g.T) amask[t] = s_mask[q];
    }
    __shared__ uint32_t red[kMiLanes / 64][MT_N];
#pragma unroll
    for (int f = 0; f < MT_N; ++f) {
        uint32_t x = s[f];
        for (int d = 32; d > 0; d >>= 1) {
            const uint32_t y = __shfl_xor(x, d, 64);
            x = f == MT_KMAX ? max(x, y) : x + y;
        }
        if ((tid & 63) == 0) red[tid >> 6][f] = x;
    }
    __syncthreads();
    if (tid < MT_N) {
        uint32_t x = red[0][tid];
        for (uint32_t w = 1; w < kMiLanes / 64; ++w) x = tid == MT_KMAX ? max(x, red[w][tid]) : x + red[w][tid];
        tiles[blockIdx.x].v[tid] = x;
    }
}

// a count beyond its capacity stops the later stages (and asks the host to
// grow the workspace); the cut lists' sizes are zeroed then, so the cut
// kernels read nothing out of range
__device__ inline void mi_check(uint32_t* ctr, const MICaps& c, uint32_t* errs) {
    bool over = ctr[M_ACTIVE] > c.active || ctr[M_FIT] > c.fit || ctr[M_WORDS] > c.words || ctr[M_VO] > c.vo ||
                ctr[M_FO] > c.fo || ctr[M_FV] > c.fv;
    if (over) {
        ctr[M_ABORT] = 1;
        errs[0] |= kMiOverflow;
    }
    // tets beyond 8 materials take the wide cut (a path captured without it
    // stops here and is captured again with it); beyond its capacity the
    // plain form reports them
    if (ctr[M_LIST + 9] > 8) {
        errs[0] |= kMiHuge;
        if (!c.huge) ctr[M_ABORT] = 1;
    }
    if (ctr[M_LIST + 9] > (uint32_t)kMaxHuge) errs[0] |= kMiPlain;
    if (ctr[M_ABORT])
        for (int q = 0; q < 4; ++q) ctr[M_LIST + q] = 0;
}
__global__ void k_mi_check(uint32_t* ctr, MICaps c, uint32_t* errs) {
    if (threadIdx.x == 0) mi_check(ctr, c, errs);
}

// The tile sums into exclusive prefixes (the first kMiPrefixes fields), the
// totals into the counters, and the capacity check; one workgroup, a wavefront
// a field, 16 consecutive tiles a lane.
__global__ void __launch_bounds__(1024) k_mi_tile_scan(MITile* __restrict__ ts, uint32_t n, uint64_t T, uint32_t* ctr,
                                                       MICaps c, uint32_t* errs, uint32_t* __restrict__ csr_off,
                                                       uint32_t* __restrict__ rec_off) {
    constexpr int P = 1024 + 1024 / 16;  // a pad word every 16 against bank conflicts
    __shared__ uint32_t sm[MT_N][P];
    __shared__ uint32_t tot[MT_N];
    __shared__ uint32_t wrapped;  // tot[MT_WORDS] has passed 2^32
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    static_assert(MT_N == 16, "a wavefront a field");
    if (threadIdx.x < MT_N) tot[threadIdx.x] = 0;
    if (threadIdx.x == 0) wrapped = 0;
    for (uint32_t base = 0; base < n; base += 1024) {
        const uint32_t i = base + threadIdx.x;
        const int pi = threadIdx.x + threadIdx.x / 16;
        MITile x = {};
        if (i < n) x = ts[i];
        for (int f = 0; f < MT_N; ++f) sm[f][pi] = x.v[f];
        __syncthreads();
        {
            const int f = wave, e0 = 16 * lane, p0 = e0 + e0 / 16;
            uint32_t sum = 0;
            for (int e = 0; e < 16; ++e) sum = f == MT_KMAX ? max(sum, sm[f][p0 + e]) : sum + sm[f][p0 + e];
            if (f < kMiPrefixes) {
                uint32_t inc = sum;
                bool wrap = false;
                for (int d = 1; d < 64; d <<= 1) {
                    const uint32_t o = __shfl_up(inc, d, 64);
                    if (lane >= d) {
                        inc += o;
                        wrap |= inc < o;
                    }
                }
                wrap |= tot[f] + inc < inc;
                if (f == MT_WORDS && wrap) wrapped = 1;
                uint32_t run = tot[f] + inc - sum;
                for (int e = 0; e < 16; ++e) {
                    const uint32_t v = sm[f][p0 + e];
                    sm[f][p0 + e] = run;
                    run += v;
                }
                sum = __shfl(inc, 63, 64);
            } else {
                for (int d = 32; d > 0; d >>= 1) {
                    const uint32_t y = __shfl_xor(sum, d, 64);
                    sum = f == MT_KMAX ? max(sum, y) : sum + y;
                }
            }
            if (lane == 0) tot[f] = f == MT_KMAX ? max(tot[f], sum) : tot[f] + sum;
        }
        __syncthreads();
        if (i < n)
            for (int f = 0; f < kMiPrefixes; ++f) ts[i].v[f] = sm[f][pi];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        ctr[M_FIT] = tot[MT_FIT];
        ctr[M_ACTIVE] = tot[MT_ACTIVE];
        for (int q = 0; q < 4; ++q) ctr[M_LIST + q] = tot[MT_LIST + q];
        for (int q = 0; q < 3; ++q) ctr[M_LIST + 4 + q] = tot[MT_HIST + q];
        ctr[M_LIST + 7] = tot[MT_N34];
        ctr[M_LIST + 8] = tot[MT_N58];
        ctr[M_LIST + 9] = tot[MT_KMAX];
        ctr[M_WORDS] = wrapped ? 0xFFFFFFFFu : tot[MT_WORDS];  // (past any capacity)
        csr_off[T] = tot[MT_FIT];
        mi_check(ctr, c, errs);
        if (!ctr[M_ABORT]) rec_off[tot[MT_ACTIVE]] = tot[MT_WORDS];
    }
}

__global__ void __launch_bounds__(kMiLanes) k_mi_fill_tiles(uint64_t T, const uint64_t* __restrict__ amask,
                                                            const MITile* __restrict__ tiles,
                                                            const uint32_t* __restrict__ abort, int tables,
                                                            uint32_t* __restrict__ csr_off, uint32_t* __restrict__ rank,
                                                            uint8_t* __restrict__ fit, uint32_t* __restrict__ act,
                                                            uint8_t* __restrict__ act_k, uint32_t* __restrict__ rec_off,
                                                            uint32_t* __restrict__ rec_loc, uint32_t* __restrict__ l0,
                                                            uint32_t* __restrict__ l1, uint32_t* __restrict__ l2,
                                                            uint32_t* __restrict__ l3) {
    if (*abort) return;
    __shared__ uint64_t s_mask[kMiTile];
    __shared__ uint32_t s_off[kMiTile], s_rank[kMiTile];
    __shared__ uint64_t w0[kMiLanes / 64], w1[kMiLanes / 64];
    __shared__ uint32_t w2[kMiLanes / 64];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint64_t t0 = (uint64_t)blockIdx.x * kMiTile;
    const MITile pre = tiles[blockIdx.x];
    for (uint32_t q = tid; q < kMiTile; q += kMiLanes) s_mask[q] = t0 + q < T ? amask[t0 + q] : 0;
    __syncthreads();
    // per lane: active materials and tets (20 bits each is enough: a tile
    // holds 1280 tets of at most 64), the four lists' tets, the slot words
    uint64_t a = 0, b = 0;
    uint32_t w = 0;
    for (uint32_t q = 0; q < 5; ++q) {
        const int k = __popcll(s_mask[5 * tid + q]);
        if (k < 2) continue;
        a += (uint64_t)k | 1ull << 32;
        b += 1ull << (16 * bucket_of_k(k, tables));
        w += rec_bound(1, k);
    }
    uint64_t ia = a, ib = b;
    uint32_t iw = w;
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t oa = __shfl_up(ia, d, 64), ob = __shfl_up(ib, d, 64);
        const uint32_t ow = __shfl_up(iw, d, 64);
        if ((int)lane >= d) {
            ia += oa;
            ib += ob;
            iw += ow;
        }
    }
    if (lane == 63) {
        w0[wave] = ia;
        w1[wave] = ib;
        w2[wave] = iw;
    }
    __syncthreads();
    ia -= a;
    ib -= b;
    iw -= w;
    for (uint32_t x = 0; x < wave; ++x) {
        ia += w0[x];
        ib += w1[x];
        iw += w2[x];
    }
    uint32_t o = pre.v[MT_FIT] + (uint32_t)ia, r = pre.v[MT_ACTIVE] + (uint32_t)(ia >> 32), at = pre.v[MT_WORDS] + iw;
    uint32_t p[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) p[q] = pre.v[MT_LIST + q] + ((uint32_t)(ib >> (16 * q)) & 0xffffu);
    for (uint32_t q = 0; q < 5; ++q) {
        const uint32_t local = 5 * tid + q;
        uint64_t m = s_mask[local];
        const int k = __popcll(m);
        s_off[local] = o;
        s_rank[local] = r;
        if (k < 2) continue;
        act[r] = (uint32_t)(t0 + local);
        act_k[r] = (uint8_t)k;
        rec_off[r] = at;
        rec_loc[r] = at;
        const int z = bucket_of_k(k, tables);
        if (z == 0) l0[p[0]++] = r;
        if (z == 1) l1[p[1]++] = r;
        if (z == 2) l2[p[2]++] = r;
        if (z == 3) l3[p[3]++] = r;
        for (uint32_t x = o; m; m &= m - 1) fit[x++] = (uint8_t)(__ffsll((unsigned long long)m) - 1);
        o += (uint32_t)k;
        ++r;
        at += rec_bound(1, k);
    }
    __syncthreads();
    for (uint32_t q = tid; q < kMiTile; q += kMiLanes)
        if (t0 + q < T) {
            csr_off[t0 + q] = s_off[q];
            rank[t0 + q] = s_rank[q];
        }
}

// The tables and the lane-group cuts of four and of five to eight materials
// in one launch of wavefronts, the longest first: the lists share no output,
// and each cut's time is the latency of its longest tet (59 + 65 us one after
// the other at 65^3 vertices and 8 materials, and 34 us of tables; together
// 66 us).  One launch rather than graph branches: kernels with this much
// private memory stay on one queue.
struct MICutArgs {
    GridView g;
    ValsRef vals;
    const uint32_t* act;
    const uint8_t* act_k;
    const uint32_t* csr_off;
    const uint8_t* fit;
    const uint32_t* list[3];
    Count n[3];
    const uint32_t* rec_off;
    uint32_t* rec_loc;
    uint16_t* rec;
    uint32_t *cnt, *errs, *labels;
    MITablesDev tables;
    uint32_t base2, base3;
    MI3Snap snap;
};
__global__ void __launch_bounds__(64) k_mi_cuts(MICutArgs A, uint32_t nb5, uint32_t nb4, uint32_t nbt) {
    __shared__ union U {
        dev::WaveMI<CBig> big;
        dev::WaveMI<CMed> med;
        MI3Pat pats[81];
        __device__ U() {}
    } u;
    const uint32_t b = blockIdx.x;
    if (b < nb5)
        cut_group_role<CBig, 64, true>(&u.big, b, nb5, A.g, A.vals, A.act, A.act_k, A.csr_off, A.fit, A.list[2], A.n[2],
                                       A.rec_off, A.rec, A.cnt, A.errs, 0, 0u, A.labels, A.snap);
    else if (b < nb5 + nb4)
        cut_group_role<CMed, 64, true>(&u.med, b - nb5, nb4, A.g, A.vals, A.act, A.act_k, A.csr_off, A.fit, A.list[1],
                                       A.n[1], A.rec_off, A.rec, A.cnt, A.errs, 0, 0u, A.labels, A.snap);
    else
        mi_table_role(u.pats, b - nb5 - nb4, nbt, A.g, A.vals, A.act, A.csr_off, A.fit, A.list[0], count_of(A.n[0]),
                      nullptr, 0u, A.rec_off, A.rec, A.cnt, A.errs, A.tables, A.labels, A.rec_loc, A.base2, A.base3);
}

// closes the face arrays, publishes the counters and the union of the error
// flags into pinned host memory, and clears both for the next run
__global__ void k_mi_close(uint32_t* ctr, uint32_t* errs, uint32_t cap_fo, uint32_t* f_vstart, uint32_t* f_tfstart,
                           uint32_t* pub) {
    const uint32_t nf = ctr[M_FO] < cap_fo ? ctr[M_FO] : cap_fo;
    if (threadIdx.x == 0 && !ctr[M_ABORT]) {
        f_vstart[nf] = ctr[M_FV];
        f_tfstart[nf] = nf;
    }
    if (threadIdx.x < M_N) pub[threadIdx.x] = ctr[threadIdx.x];
    uint32_t e = errs[threadIdx.x];
    for (int d = 32; d > 0; d >>= 1) e |= __shfl_xor(e, d, 64);
    if (threadIdx.x == 0) pub[kMiPub] = e;
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x < M_N) ctr[threadIdx.x] = 0;
    errs[threadIdx.x] = 0;
}

unsigned blocks_for(uint64_t n) { return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>((n + 255) / 256, 65535)); }

int bits_of(uint64_t x) {
    int b = 0;
    while (b < 64 && (x >> b)) ++b;
    return b;
}

}  // namespace

struct MIWorkspace {
    DevMem mem;
    MICaps cap;
    bool in_use = false;
    // per vertex / tet (fixed by the grid)
    DBuf<const double*> vals_at;  // the run's values, left by its first kernel for the captured ones
    DBuf<uint64_t> hm, amask;
    DBuf<MITile> tiles;
    DBuf<uint32_t> csr_off, rank;
    // per active tet
    DBuf<uint8_t> fit, act_k;
    DBuf<uint32_t> act, blists, rec_off, cnt, labels;
    // each active tet's record location: its slot (rec_off), or for a table
    // tet the table's record, whose words follow the slots in rec (at
    // tab_base2 and tab_base3)
    DBuf<uint32_t> rec_loc;
    uint32_t tab_base2 = 0, tab_base3 = 0;
    DBuf<uint16_t> rec;
    DBuf<uint2> emit_at;      // MIEmits
    DBuf<uint32_t> emit_list;
    unsigned cut_blocks[2] = {0, 0};
    bool wide = false;  // the path holds the cut of more than 8 materials, once a run needs it
    // per occurrence, face
    DBuf<uint16_t> oj, fq_l;
    DBuf<uint64_t> okey;
    DBuf<uint32_t> cv, cf, cfv, oa, fq_a, fq_vs, fve;
    DBuf<uint8_t> fq_m;
    // dedup
    DBuf<uint32_t> first, mo, hslot, vrank, vid, first_occ, tile_first, star_head;
    DBuf<uint8_t> star_ent;
    // explicit meshes: first-occurrence hash table (key + 1, ~smallest occurrence), zero
    // between runs: the assign pass clears the slots a run used
    DBuf<unsigned long long> hkey;
    DBuf<uint32_t> hmx;
    int hbits = 0;
    bool hash_dirty = false;  // a run stopped with entries left: clear before the next
    // outputs
    DBuf<uint32_t> v_tet, v_sv, f_vstart, f_verts, f_tfstart, f_tf_tet;
    DBuf<uint16_t> v_j, f_tf_local;
    DBuf<uint8_t> v_ss, v_fn, f_func;
    DBuf<double> xyz;
    DBuf<uint32_t> ctr, errs;
    uint32_t* pub_h = nullptr;
    uint32_t* pub_d = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hipEvent_t ev[2] = {nullptr, nullptr};
    bool ctr_clear = false;  // counters and error flags are zero (left so by the last run)
    void drop_graph() {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
    }
    ~MIWorkspace() {
        drop_graph();
        for (auto e : ev)
            if (e) (void)hipEventDestroy(e);
        if (pub_h) (void)hipHostFree(pub_h);
    }
};

struct MIPlan {
    std::mutex mu;
    std::vector<std::shared_ptr<MIWorkspace>> ws;
};

struct MIPlanCache {
    std::mutex mu;
    std::map<uint32_t, std::shared_ptr<MIPlan>> plans;  // by material count
    std::shared_ptr<MIPlan> get(uint32_t F) {
        std::lock_guard<std::mutex> l(mu);
        auto& p = plans[F];
        if (!p) p = std::make_shared<MIPlan>();
        return p;
    }
};

std::shared_ptr<void> make_mi_plan_cache() { return std::make_shared<MIPlanCache>(); }

namespace {

// W.cap says what the buffers hold: it is empty from the first change to them
// until the last has its size, so a growth that fails midway (no memory) leaves
// a workspace that the next run allocates anew
void alloc_mi(MIWorkspace& W, const Grid& g, const MICaps& c, hipStream_t s) {
    DevMem& m = W.mem;
    W.drop_graph();
    const uint64_t V = g.view.V, T = g.view.T;
    const MITablesRaw TR = mi_tables_device(s);
    if ((uint64_t)c.words + 1 + TR.n_w2 + TR.n_w3 >= record_limit(1ull << 32))
        throw NeedsPlainForm("the record slots exceed 2^32 words");
    W.cap = MICaps{};
    if (!W.errs.p) {
        W.hm.alloc(m, V);
        W.amask.alloc(m, T);
        W.vals_at.alloc(m, 1);
        W.tiles.alloc(m, T / kMiTile + 1);
        W.csr_off.alloc(m, T + 1);
        W.rank.alloc(m, T + 1);
        W.ctr.alloc(m, 64);
        W.errs.alloc(m, 64);
    }
    const uint64_t A = c.active;
    W.fit.alloc(m, c.fit + 1);
    W.act_k.alloc(m, A + 1);
    W.act.alloc(m, A + 1);
    W.blists.alloc(m, 4 * (A + 1));
    W.rec_off.alloc(m, A + 2);
    W.rec_loc.alloc(m, A + 2);
    {
        // the slots, then the two tables' record words (copied once per allocation)
        W.tab_base2 = (uint32_t)c.words + 1;
        W.tab_base3 = W.tab_base2 + (uint32_t)TR.n_w2;
        W.rec.alloc(m, (uint64_t)W.tab_base3 + TR.n_w3 + 1);
        RIN_HIP(hipMemcpyAsync(W.rec.p + W.tab_base2, TR.w2, 2 * TR.n_w2, hipMemcpyDeviceToDevice, s));
        RIN_HIP(hipMemcpyAsync(W.rec.p + W.tab_base3, TR.w3, 2 * TR.n_w3, hipMemcpyDeviceToDevice, s));
    }
    W.cnt.alloc(m, 3 * A + 3);
    W.labels.alloc(m, A + 1);
    W.emit_at.alloc(m, A + 1);
    W.emit_list.alloc(m, c.fo + 1);
    W.cv.alloc(m, A + 2);
    W.cf.alloc(m, A + 2);
    W.cfv.alloc(m, A + 2);
    // thread cuts (four and five to eight materials): a lane per tet with
    // its complex in LDS, two lanes (one for the larger complexes) a
    // wavefront, grids striding over their lists
    W.cut_blocks[0] = (unsigned)std::min<uint64_t>((A + 1) / 2 + 1, 4096);
    W.cut_blocks[1] = (unsigned)std::min<uint64_t>(A + 1, 2048);
    W.okey.alloc(m, c.vo + 1);
    W.oa.alloc(m, c.vo + 1);
    W.oj.alloc(m, c.vo + 1);
    W.fq_a.alloc(m, c.fo + 1);
    W.fq_l.alloc(m, c.fo + 1);
    W.fq_m.alloc(m, 2 * (uint64_t)c.fo + 2);
    W.fq_vs.alloc(m, c.fo + 1);
    W.fve.alloc(m, c.fv + 1);
    for (auto* b : {&W.first, &W.mo, &W.vrank, &W.first_occ}) b->alloc(m, c.vo + 1);
    if (g.view.regular) {
        W.tile_first.alloc(m, (c.vo + kDedupTile - 1) / kDedupTile + 1);
        upload_star_tables(m, W.star_head, W.star_ent, s);
    } else {
        // a table of at least twice the occurrence capacity, cleared once here
        W.vid.alloc(m, c.vo + 1);
        W.hslot.alloc(m, c.vo + 1);
        W.hbits = 10;
        while ((1ull << W.hbits) < 2ull * (c.vo + 1)) ++W.hbits;
        W.hkey.alloc(m, 1ull << W.hbits);
        W.hmx.alloc(m, 1ull << W.hbits);
        RIN_HIP(hipMemsetAsync(W.hkey.p, 0, 8ull << W.hbits, s));
        RIN_HIP(hipMemsetAsync(W.hmx.p, 0, 4ull << W.hbits, s));
        W.hash_dirty = false;
    }
    W.v_tet.alloc(m, c.vo + 1);
    W.v_j.alloc(m, c.vo + 1);
    W.v_ss.alloc(m, c.vo + 1);
    W.v_sv.alloc(m, 4 * (uint64_t)c.vo + 4);
    W.v_fn.alloc(m, 4 * (uint64_t)c.vo + 4);
    W.xyz.alloc(m, 3 * (uint64_t)c.vo + 3);
    W.f_vstart.alloc(m, c.fo + 1);
    W.f_tfstart.alloc(m, c.fo + 1);
    W.f_verts.alloc(m, c.fv + 1);
    W.f_tf_tet.alloc(m, c.fo + 1);
    W.f_tf_local.alloc(m, c.fo + 1);
    W.f_func.alloc(m, 2 * (uint64_t)c.fo + 2);
    if (!W.pub_h) {
        RIN_HIP(hipHostMalloc((void**)&W.pub_h, (kMiPub + 1) * sizeof(uint32_t),
                              hipHostMallocMapped | hipHostMallocCoherent));
        RIN_HIP(hipHostGetDevicePointer((void**)&W.pub_d, W.pub_h, 0));
    }
    W.cap = c;
}

// the whole path on stream s; every launch is sized by capacities and reads
// the live counts from the workspace
void mi_path(MIWorkspace& W, const Grid& g, uint32_t F, const MITablesDev& TT, hipStream_t s) {
    const GridView& G = g.view;
    const uint64_t T = G.T;
    MICaps c = W.cap;
    c.huge = W.wide ? 1u : 0u;
    uint32_t* ctr = W.ctr.p;
    const uint32_t* abort = ctr + M_ABORT;
    const ValsRef vals{nullptr, W.vals_at.p};
    // cut lists: the tables take two and three materials, lane groups four
    // to eight.  RIN_CUT_FORM=wave or thread turns the tables off and cuts
    // every tet up to eight materials by lane groups or by a lane each.
    const char* form = std::getenv("RIN_CUT_FORM");
    const bool all_thread = form && !std::strcmp(form, "thread");
    const bool all_wave = form && !std::strcmp(form, "wave");
    const int tables = (all_thread || all_wave) ? 0 : 1;
    uint32_t* bl[4];
    for (int q = 0; q < 4; ++q) bl[q] = W.blists.p + (uint64_t)q * (c.active + 1);
    // filter, CSR, lists and slots (src/material_interface.cpp:94-152)
    const uint32_t ntiles = (uint32_t)((T + kMiTile - 1) / kMiTile);
    hipLaunchKernelGGL(k_mi_count_tiles, dim3(ntiles), dim3(kMiLanes), 0, s, G, W.vals_at.p, F,
                       (const uint64_t*)W.hm.p, tables, W.amask.p, W.tiles.p);
    hipLaunchKernelGGL(k_mi_tile_scan, dim3(1), dim3(1024), 0, s, W.tiles.p, ntiles, T, ctr, c, W.errs.p, W.csr_off.p,
                       W.rec_off.p);
    hipLaunchKernelGGL(k_mi_fill_tiles, dim3(ntiles), dim3(kMiLanes), 0, s, T, (const uint64_t*)W.amask.p,
                       (const MITile*)W.tiles.p, abort, tables, W.csr_off.p, W.rank.p, W.fit.p, W.act.p, W.act_k.p,
                       W.rec_off.p, W.rec_loc.p, bl[0], bl[1], bl[2], bl[3]);
    const Count NA(ctr + M_ACTIVE, c.active, abort);
    const Count n1(ctr + M_LIST + 1, c.active, abort), n2(ctr + M_LIST + 2, c.active, abort);
    // the cuts start from the 3-material table's complex after three
    // materials (RIN_MI3_START=0: from the tet)
    const char* ms = std::getenv("RIN_MI3_START");
    MICutArgs U;
    U.g = G;
    U.vals = vals;
    U.act = W.act.p;
    U.act_k = W.act_k.p;
    U.csr_off = W.csr_off.p;
    U.fit = W.fit.p;
    for (int q = 0; q < 3; ++q) U.list[q] = bl[q];
    U.n[0] = Count(ctr + M_LIST, c.active, abort);
    U.n[1] = n1;
    U.n[2] = n2;
    U.rec_off = W.rec_off.p;
    U.rec_loc = W.rec_loc.p;
    U.rec = W.rec.p;
    U.cnt = W.cnt.p;
    U.errs = W.errs.p;
    U.labels = W.labels.p;
    U.tables = TT;
    U.base2 = W.tab_base2;
    U.base3 = W.tab_base3;
    U.snap = (ms && !std::strcmp(ms, "0")) ? MI3Snap{nullptr, nullptr, nullptr}
                                           : MI3Snap{TT.pat3, TT.snap_off3, TT.snap3};
    if (all_thread) {
        hipLaunchKernelGGL((k_cut_lds<CMed, true, 2>), dim3(W.cut_blocks[0]), dim3(2), 0, s, G, vals,
                           (const uint32_t*)W.act.p, (const uint8_t*)W.act_k.p, (const uint32_t*)W.csr_off.p,
                           (const uint8_t*)W.fit.p, n1, 1, 4, (uint32_t)0, (const uint32_t*)W.rec_off.p, W.rec.p,
                           W.cnt.p, W.errs.p, (const uint32_t*)bl[1], W.labels.p);
        hipLaunchKernelGGL((k_cut_lds<CBig, true, 1>), dim3(W.cut_blocks[1]), dim3(1), 0, s, G, vals,
                           (const uint32_t*)W.act.p, (const uint8_t*)W.act_k.p, (const uint32_t*)W.csr_off.p,
                           (const uint8_t*)W.fit.p, n2, 5, 8, (uint32_t)0, (const uint32_t*)W.rec_off.p, W.rec.p,
                           W.cnt.p, W.errs.p, (const uint32_t*)bl[2], W.labels.p);
    } else {
        const unsigned nb5 = (unsigned)std::min<uint64_t>(c.active + 1, 1024);
        const unsigned nb4 = (unsigned)std::min<uint64_t>(c.active + 1, 2048);
        const unsigned nbt = (unsigned)std::min<uint64_t>((c.active + 63) / 64 + 1, 16384);
        hipLaunchKernelGGL(k_mi_cuts, dim3(nb5 + nb4 + nbt), dim3(64), 0, s, U, nb5, nb4, nbt);
    }
    if (W.wide) {
        const MI3Snap none{nullptr, nullptr, nullptr};
        hipLaunchKernelGGL((k_cut_group<CWideMI, 64, true>), dim3((unsigned)std::min<uint64_t>(c.active + 1, 512)),
                           dim3(64), 0, s, G, vals, (const uint32_t*)W.act.p, (const uint8_t*)W.act_k.p,
                           (const uint32_t*)W.csr_off.p, (const uint8_t*)W.fit.p, (const uint32_t*)bl[3],
                           Count(ctr + M_LIST + 3, c.active, abort), (const uint32_t*)W.rec_off.p, W.rec.p, W.cnt.p,
                           W.errs.p, 0, (uint32_t)0, W.labels.p, none);
    }
    // extraction (src/extract_mesh.cpp:569-986): boundary-face pairing, then
    // occurrences in the reference's creation order
    MIArgs A;
    A.g = G;
    A.act = W.act.p;
    A.csr_off = W.csr_off.p;
    A.rank = W.rank.p;
    A.rec_loc = W.rec_loc.p;
    A.nbr = g.nbr.p;
    A.fit = W.fit.p;
    A.rec = W.rec.p;
    A.n_active = NA;
    const MIEmits E{W.emit_at.p, W.emit_list.p, c.fo, ctr + M_EMIT};
    hipLaunchKernelGGL(k_mi_pair, dim3(blocks_for(c.active)), dim3(256), 0, s, A, (const uint32_t*)W.labels.p, E,
                       W.cnt.p);
    {
        const uint32_t* in[3] = {W.cnt.p, W.cnt.p + 1, W.cnt.p + 2};
        uint32_t* out[3] = {W.cv.p, W.cf.p, W.cfv.p};
        uint32_t* tot[3] = {ctr + M_VO, ctr + M_FO, ctr + M_FV};
        scan3_u32(W.mem, in, 3, out, NA, tot, s);
    }
    hipLaunchKernelGGL(k_mi_check, dim3(1), dim3(64), 0, s, ctr, c, W.errs.p);
    hipLaunchKernelGGL(k_mi_extract, dim3(blocks_for(c.active)), dim3(256), 0, s, A, E,
                       (const uint32_t*)W.cv.p, (const uint32_t*)W.cf.p, (const uint32_t*)W.cfv.p, W.okey.p, W.oa.p,
                       W.oj.p, W.fq_a.p, W.fq_l.p, W.fq_m.p, W.fq_vs.p, W.fve.p);
    // vertex dedup: on regular grids each key's first occurrence by its
    // simplex's star, on explicit meshes by an atomic hash table (left empty);
    // ids in the order of the first occurrences
    const Count NVO(ctr + M_VO, c.vo, abort);
    const uint32_t *vid = W.vid.p, *mo = nullptr;
    if (G.regular) {
        const unsigned tgrid = (unsigned)((c.vo + kDedupTile - 1) / kDedupTile);
        StarArgs S;
        S.res = G.res;
        S.edge_shift = 14;
        S.face_shift = 20;
        S.own = 1;
        S.okey = W.okey.p;
        S.oa = W.oa.p;
        S.act = W.act.p;
        S.rank = RankOf{W.rank.p, W.act.p, nullptr};
        S.voff = W.cv.p;
        S.star_head = W.star_head.p;
        S.star_ent = W.star_ent.p;
        S.first = W.first.p;
        S.mo = W.mo.p;
        S.n_active = ctr + M_ACTIVE;
        S.tile_first = W.tile_first.p;
        hipLaunchKernelGGL(k_dedup_star, dim3(tgrid), dim3(256), 0, s, NVO, S);
        hipLaunchKernelGGL(k_dedup_tile_scan, dim3(1), dim3(1024), 0, s, NVO, W.tile_first.p, ctr + M_NV);
        hipLaunchKernelGGL(k_dedup_rank, dim3(tgrid), dim3(256), 0, s, NVO, (const uint32_t*)W.first.p,
                           (const uint32_t*)W.tile_first.p, W.vrank.p, W.first_occ.p);
        vid = W.vrank.p;
        mo = W.mo.p;
    } else {
        hipLaunchKernelGGL(k_hash_insert, dim3(blocks_for(c.vo)), dim3(256), 0, s, NVO, (const uint64_t*)W.okey.p,
                           W.hkey.p, W.hmx.p, W.hbits, W.hslot.p, W.errs.p);
        hipLaunchKernelGGL(k_hash_first, dim3(blocks_for(c.vo)), dim3(256), 0, s, NVO, (const uint32_t*)W.hslot.p,
                           (const uint32_t*)W.hmx.p, W.first.p, W.mo.p);
        scan_u32(W.mem, W.first.p, W.vrank.p, NVO, ctr + M_NV, s);
        hipLaunchKernelGGL(k_dedup_assign, dim3(blocks_for(c.vo)), dim3(256), 0, s, NVO, (const uint32_t*)W.mo.p,
                           (const uint32_t*)W.first.p, (const uint32_t*)W.vrank.p, W.vid.p, W.first_occ.p,
                           (const uint32_t*)W.hslot.p, W.hkey.p, W.hmx.p);
    }
    // coordinates and faces
    const Count NV(ctr + M_NV, c.vo, abort), NF(ctr + M_FO, c.fo, abort), NFV(ctr + M_FV, c.fv, abort);
    hipLaunchKernelGGL(k_vert_fields_mi, dim3(blocks_for(c.vo)), dim3(256), 0, s, G, vals, (const uint32_t*)W.act.p,
                       (const uint32_t*)W.csr_off.p, (const uint8_t*)W.fit.p, (const uint32_t*)W.rec_loc.p,
                       (const uint16_t*)W.rec.p, (const uint32_t*)W.first_occ.p, (const uint32_t*)W.oa.p,
                       (const uint16_t*)W.oj.p, NV, W.v_tet.p, W.v_j.p, W.v_ss.p, W.v_sv.p, W.v_fn.p, W.xyz.p);
    hipLaunchKernelGGL(k_mi_face_out, dim3(blocks_for(c.fo)), dim3(256), 0, s, NF, (const uint32_t*)W.act.p,
                       (const uint32_t*)W.fq_a.p, (const uint16_t*)W.fq_l.p, (const uint8_t*)W.fq_m.p,
                       (const uint32_t*)W.fq_vs.p, (const uint32_t*)W.fve.p, vid, mo, NFV,
                       W.f_vstart.p, W.f_verts.p, W.f_tfstart.p, W.f_tf_tet.p, W.f_tf_local.p, W.f_func.p);
    hipLaunchKernelGGL(k_mi_close, dim3(1), dim3(64), 0, s, ctr, W.errs.p, c.fo, W.f_vstart.p, W.f_tfstart.p,
                       W.pub_d);
    RIN_HIP(hipGetLastError());
}

MICaps grow_caps(const MICaps& have, const uint32_t* pub, uint64_t T) {
    // a count past its capacity grows that capacity by a quarter over the
    // count; a stage that never ran (an earlier overflow) doubles its capacity
    auto g = [](uint32_t have_c, uint32_t seen) -> uint32_t {
        const uint64_t want = seen > have_c ? (uint64_t)seen + seen / 4 + 64 : (uint64_t)have_c;
        return (uint32_t)std::min<uint64_t>(want, 0xFFFFFFF0u);
    };
    MICaps c;
    const bool ran = !pub[M_ABORT];
    c.active = g(have.active, pub[M_ACTIVE]);
    c.fit = g(have.fit, pub[M_FIT]);
    c.words = g(have.words, pub[M_WORDS]);
    c.vo = g(have.vo, pub[M_VO]);
    c.fo = g(have.fo, pub[M_FO]);
    c.fv = g(have.fv, pub[M_FV]);
    if (!ran) {
        // later stages did not count: make room in proportion to the tets
        c.fit = std::max<uint32_t>(c.fit, 3 * c.active);
        c.words = std::max<uint32_t>(c.words, 160 * c.active);
        c.vo = std::max<uint32_t>(c.vo, 8 * c.active);
        c.fo = std::max<uint32_t>(c.fo, 4 * c.active);
        c.fv = std::max<uint32_t>(c.fv, 16 * c.active);
    }
    (void)T;
    return c;
}

}  // namespace

void run_batched_mi(DevMem& ctx_mem, const Grid& g, const Values& val, uint32_t flags, RunOut& out, hipStream_t s) {
    (void)ctx_mem;
    if (flags & (RUN_CUT_ONLY | RUN_REVERSE | RUN_NO_LOOKUP))
        throw NeedsPlainForm("the -R check and lookups off run the plain form");
    if (val.grid_id != g.id) throw std::invalid_argument("values were made on another grid");
    ensure_nbr(ctx_mem, g, s);
    auto* cache = static_cast<MIPlanCache*>(g.mi_plans.get());
    std::shared_ptr<MIPlan> planp = cache->get(val.F);
    MIPlan& P = *planp;
    std::lock_guard<std::mutex> lock(P.mu);
    std::shared_ptr<MIWorkspace> W;
    for (auto& w : P.ws)
        if (!w->in_use) {
            W = w;
            break;
        }
    if (!W) {
        W = std::make_shared<MIWorkspace>();
        P.ws.push_back(W);
    }
    MIWorkspace& w = *W;
    const MITablesDev TT = mi_tables_view(mi_tables_device(s));
    const uint64_t T = g.view.T;
    uint32_t pub[kMiPub + 1];
    bool ok = false;
    for (int attempt = 0; attempt < 8 && !ok; ++attempt) {
        if (!w.cap.active) {
            MICaps c0;
            c0.active = (uint32_t)std::min<uint64_t>(T, 1024 + T / 16);
            c0.fit = 3 * c0.active;
            c0.words = 160 * c0.active;
            c0.vo = 8 * c0.active;
            c0.fo = 4 * c0.active;
            c0.fv = 16 * c0.active;
            alloc_mi(w, g, c0, s);
        }
        if (!w.exec) {
            // recorded once per workspace capacity: the graph holds no pointer
            // to the values, which the first kernel of a run leaves for it
            const int kbits = 2 + std::max({bits_of(g.view.V), bits_of(g.view.n_edge_ids) + 12,
                                            bits_of(g.view.n_face_ids) + 18, bits_of(w.cap.active) + 10});
            if (kbits > 63) throw NeedsPlainForm("simplex keys exceed 63 bits for this mesh");
            for (auto& e : w.ev)
                if (!e) RIN_HIP(hipEventCreate(&e));
            hipGraph_t gr = nullptr;
            RIN_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed));
            try {
                mi_path(w, g, val.F, TT, s);
            } catch (...) {
                (void)hipStreamEndCapture(s, &gr);
                if (gr) (void)hipGraphDestroy(gr);
                throw;
            }
            RIN_HIP(hipStreamEndCapture(s, &gr));
            w.graph = gr;
            RIN_HIP(hipGraphInstantiate(&w.exec, gr, nullptr, nullptr, 0));
        }
        if (w.hash_dirty) {
            RIN_HIP(hipMemsetAsync(w.hkey.p, 0, 8ull << w.hbits, s));
            RIN_HIP(hipMemsetAsync(w.hmx.p, 0, 4ull << w.hbits, s));
            w.hash_dirty = false;
        }
        if (!w.ctr_clear) hipLaunchKernelGGL(k_mi_zero, dim3(1), dim3(64), 0, s, w.ctr.p, w.errs.p);
        w.ctr_clear = false;
        RIN_HIP(hipEventRecord(w.ev[0], s));
        // highest materials (src/material_interface.cpp:53-92), with the values
        hipLaunchKernelGGL(k_highest_mi, dim3(blocks_for(g.view.V)), dim3(256), 0, s, (const double*)val.vals.p,
                           g.view.V, val.F, w.hm.p, (uint32_t*)nullptr, w.ctr.p + M_DEGEN, w.vals_at.p);
        RIN_HIP(hipGraphLaunch(w.exec, s));
        RIN_HIP(hipEventRecord(w.ev[1], s));
        RIN_HIP(hipStreamSynchronize(s));
        w.ctr_clear = true;  // the run's closing kernel cleared them
        float ms = 0;
        RIN_HIP(hipEventElapsedTime(&ms, w.ev[0], w.ev[1]));
        std::memcpy(pub, w.pub_h, sizeof(pub));
        uint32_t e = pub[kMiPub];
        // a stopped or failed run may leave table entries
        if (w.hkey.p && ((e & ~kMiHuge) || ((e & kMiHuge) && !w.wide))) w.hash_dirty = true;
        if (e & kMiPlain) throw NeedsPlainForm("a tet has more materials than the device cut holds");
        if ((e & kMiHuge) && !w.wide) {
            // first run with such tets: the path captured again with the wide cut
            w.wide = true;
            w.drop_graph();
            continue;
        }
        e &= ~kMiHuge;
        if (e & kMiOverflow) {
            alloc_mi(w, g, grow_caps(w.cap, pub, T), s);
            continue;
        }
        if (e) {
            out.err = e;
            throw NeedsPlainForm("a complex exceeds the batched cut's capacities or the predicate range");
        }
        out.times.ms.push_back({"batched path (one graph)", ms});
        ok = true;
    }
    if (!ok) throw std::runtime_error("batched material-interface workspace did not converge");
    w.in_use = true;
    out.mi = true;
    out.flags = flags;
    out.T = T;
    out.F = val.F;
    out.num_degenerate = pub[M_DEGEN];
    out.n_active = out.num_intersecting = pub[M_ACTIVE];
    out.n_fit = pub[M_FIT];
    for (int q = 0; q < 3; ++q) out.nb[q] = pub[M_LIST + 4 + q];
    out.n_cut34 = pub[M_LIST + 7];
    out.n_cut58 = pub[M_LIST + 8];
    out.n_verts = pub[M_NV];
    out.n_faces = pub[M_FO];
    out.n_face_verts = pub[M_FV];
    out.n_tet_faces = pub[M_FO];
    out.n_vert_occ = pub[M_VO];
    out.n_face_occ = pub[M_FO];
    out.n_face_occ_verts = pub[M_FV];
    auto& vw = out.view;
    vw.fit = w.fit.p;
    vw.csr_off = w.csr_off.p;
    vw.act = w.act.p;
    vw.rank_of_tet = w.rank.p;
    vw.rec_off = w.rec_off.p;
    vw.rec = w.rec.p;
    vw.rec_loc = w.rec_loc.p;
    vw.v_tet = w.v_tet.p;
    vw.v_j = w.v_j.p;
    vw.v_ss = w.v_ss.p;
    vw.v_sv = w.v_sv.p;
    vw.v_fn = w.v_fn.p;
    vw.xyz = w.xyz.p;
    vw.f_vstart = w.f_vstart.p;
    vw.f_verts = w.f_verts.p;
    vw.f_tfstart = w.f_tfstart.p;
    vw.f_tf_tet = w.f_tf_tet.p;
    vw.f_tf_local = w.f_tf_local.p;
    vw.f_func = w.f_func.p;
    std::weak_ptr<MIPlan> wp = planp;
    MIWorkspace* raw = W.get();
    out.hold = std::shared_ptr<void>(nullptr, [W, wp, raw](void*) {
        if (auto p = wp.lock()) {
            std::lock_guard<std::mutex> l(p->mu);
            raw->in_use = false;
        }
    });
}

}  // namespace rin
