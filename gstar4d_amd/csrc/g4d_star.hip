// gStar4D for MI355X — 4D stars on the lifted points and parallel star splaying.
//
// Reference behaviour restated (GD/ = GDelaunay/):
//   initial cones            GD/GDelaunay/GDelPredKernels.cu:45-231
//   beneath marking          GD/GDelaunay/GDelPredKernels.cu:233-420
//   hole stitching           GD/GDelaunay/GDelKernels.cu:518-783
//   drowned insertions       GD/GDelaunay/GDelKernels.cu:1459-1527, GD/GDelaunay/GDelHost.cu:817-875
//   containment proofs       GD/GDelaunay/GDelPredKernels.cu:427-626
//   triangle insertions      GD/GDelaunay/GDelKernels.cu:818-939
//   history                  GD/GDelaunay/GDelKernels.cu:984-1068,1625-1677
//   tetra output             GD/GDelaunay/GDelKernels.cu:1097-1191, GD/GDelaunay/GDelPredKernels.cu:628-692
//
// MI355X design.  A pass's plan lists its stars by size.  A group of 16 lanes builds a star of up to 32
// link vertices (four stars a wave), a wave one of up to 256, a work-group larger ones.  The star's
// link (a triangulated 2-sphere) lives in LDS, beyond 1,024 vertices in HBM: local vertex table with
// coordinates relative to the star point, triangles with local vertices and adjacency.  Each lane owns
// triangle slots (lane, lane + lanes, ...) and keeps for each the four cofactors of the lifted 4x4
// determinant, in registers (in LDS in the exact kernels, in HBM in the global-memory one), so the
// beneath test of a new vertex v against triangle (a,b,c) is one 4-term dot product:
//     orient4(a,b,c,s,v) = v'x*Mx - v'y*My + v'z*Mz - v'l*Ml      (primes: relative to s)
// with a forward-error bound from the cofactor permanents.  A star with an uncertain sign goes, untouched,
// to a kernel that has the exact predicate with SoS.  The hole boundary after freeing beneath
// triangles is found in parallel (edges of freed triangles whose neighbour survives), slots are
// assigned with a prefix sum over a free-slot stack, and the fan's adjacency is closed through two
// per-vertex maps (boundary edge starting / ending at each vertex).  The whole insertion list of a star
// runs inside one kernel, so there is no host loop per insertion index.
#include "g4d_predicates.h"
#include <algorithm>
#include <climits>
#include <cstdlib>
#include <type_traits>

#include "g4d_star.h"

namespace g4d {

static constexpr uint32_t TF_ALIVE = 1u << 27;
static constexpr uint32_t TF_CHECKED = 1u << 28;
static constexpr uint32_t TF_VIS = 1u << 29;
static constexpr uint32_t TF_FRESH = 1u << 30;
static constexpr uint32_t TF_UNSURE = 1u << 26; // global-memory kernel only (its flags word holds no vertices)

__device__ __forceinline__ int tvert(uint32_t t, int i) { return (int)((t >> (9 * i)) & 511u); }
__device__ __forceinline__ uint32_t tpack(int a, int b, int c, uint32_t fl)
{
    return (uint32_t)a | ((uint32_t)b << 9) | ((uint32_t)c << 18) | fl;
}

// HBM triangle: bits 0..26 vertices, 27..56 adjacency (10 bits each), 57 checked.
__device__ __forceinline__ uint64_t hpack(int a, int b, int c, int o0, int o1, int o2, bool checked)
{
    return (uint64_t)a | ((uint64_t)b << 9) | ((uint64_t)c << 18) | ((uint64_t)o0 << 27) | ((uint64_t)o1 << 37) |
           ((uint64_t)o2 << 47) | ((uint64_t)(checked ? 1 : 0) << 57);
}
__device__ __forceinline__ int hvert(uint64_t t, int i) { return (int)((t >> (9 * i)) & 511u); }
__device__ __forceinline__ int hopp(uint64_t t, int i) { return (int)((t >> (27 + 10 * i)) & 1023u); }
__device__ __forceinline__ bool hchecked(uint64_t t) { return (t >> 57) & 1u; }

// Wide format (stars with >= STAR_WIDE_MIN link vertices): two words per triangle.
static constexpr uint64_t W21 = (1ull << 21) - 1;
__device__ __forceinline__ uint64_t wpack3(int a, int b, int c)
{
    return (uint64_t)a | ((uint64_t)b << 21) | ((uint64_t)c << 42);
}
__device__ __forceinline__ int wfield(uint64_t w, int i) { return (int)((w >> (21 * i)) & W21); }

// Local vertex indices of triangle t of a star stored at tpool + to.
__device__ __forceinline__ void star_tri_verts(const uint64_t *tpool, int64_t to, int t, bool wide, int *v)
{
    if (wide) {
        const uint64_t w = tpool[to + 2 * (int64_t)t];
        v[0] = wfield(w, 0);
        v[1] = wfield(w, 1);
        v[2] = wfield(w, 2);
    } else {
        const uint64_t h = tpool[to + t];
        v[0] = hvert(h, 0);
        v[1] = hvert(h, 1);
        v[2] = hvert(h, 2);
    }
}

// Per triangle slot: cofactors C[0..3] and permanents P[0..3], stored component-major so that the
// lanes of a wave, each reading its own slot, touch consecutive 8-byte words.
template <int TMAX, bool CACHED>
struct StarCof {
    double cof[8][TMAX];
};
template <int TMAX>
struct StarCof<TMAX, false> {
};

template <int VMAX, bool CACHED>
struct StarLds : StarCof<2 * VMAX, CACHED> {
    static constexpr int TMAX = 2 * VMAX;
    int vid[VMAX];
    double vc[VMAX][4];
    uint32_t tv[TMAX];
    union {
        uint16_t to[TMAX][4]; // neighbours across the edges opposite vertices 0-2 (fourth unused)
        uint64_t to64[TMAX];  // the same rows read as one word each
    };
    int16_t vstart[VMAX];
    int16_t vend[VMAX];
    uint16_t freel[TMAX];
    uint16_t be_a[TMAX], be_b[TMAX], be_u[TMAX], be_slot[TMAX];
    uint8_t be_j[TMAX];
    int ins[VMAX];
    int16_t ins_local[VMAX];
    uint8_t present[VMAX];
    uint16_t remap[TMAX];
    uint16_t vremap[VMAX];
    int sc[4];
};

// Cofactors and permanents of the triangle (r0, r1, r2) into the component-major slot table.
template <int TMAX>
__device__ __forceinline__ void lds_cofactors(const double *r0, const double *r1, const double *r2,
                                              double (*cof)[TMAX], int slot)
{
    double C[4], P[4];
    tri_cofactors(r0, r1, r2, C, P);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        cof[j][slot] = C[j];
        cof[4 + j][slot] = P[j];
    }
}

// Exclusive scan across the wave of per-lane counts below 2^BITS; returns the prefix, the total
// in *tot.  One ballot and a lane-masked bit count per bit: no cross-lane data movement.
template <int BITS>
__device__ __forceinline__ int wave_excl(int v, int *tot)
{
    int pre = 0, all = 0;
#pragma unroll
    for (int b = 0; b < BITS; b++) {
        const uint64_t m = __ballot((v >> b) & 1);
        pre += (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u)) << b;
        all += __popcll(m) << b;
    }
    *tot = all;
    return pre;
}

// Bits needed for counts up to x.
__host__ __device__ constexpr int count_bits(int x) { return x < 2 ? 1 : 1 + count_bits(x >> 1); }

// Insertion pairs of a link triangle with global vertices (a, b, c) (GD/GDelaunay/GDelKernels.cu:
// 818-939): when it is unchecked, each cyclic edge (u, w) with u < w gives (u<<32 | w); there
// are one or two such edges, the unused entry is STAR_PAIR_NONE.
struct TriPairs {
    uint64_t x, y;
};
__device__ __forceinline__ TriPairs star_tri_pairs(int a, int b, int c, bool unchecked)
{
    uint64_t e0 = STAR_PAIR_NONE, e1 = STAR_PAIR_NONE;
    if (unchecked) {
        const int u[3] = {a, b, c};
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const int x = u[i], y = u[(i + 1) % 3];
            if (x < y) {
                const uint64_t k = ((uint64_t)(uint32_t)x << 32) | (uint32_t)y;
                if (e0 == STAR_PAIR_NONE) e0 = k;
                else e1 = k;
            }
        }
    }
    return TriPairs{e0, e1};
}

// The LDS star kernels run one wave per work-group.  A wave's LDS operations complete in
// order, so ordering its LDS traffic needs only a compiler-level barrier at wavefront scope;
// unlike __syncthreads() this does not wait for the wave's outstanding global stores.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Appends star s to a list (lane 0), flagging a buffer error when the list is full.
__device__ __forceinline__ void star_list_push(int *list, int64_t cap, unsigned long long *counter, int s,
                                               unsigned long long *cnt)
{
    if (__lane_id() == 0) {
        const unsigned long long k = atomicAdd(counter, 1ull);
        if ((int64_t)k < cap) list[k] = s;
        else atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_BUFFER);
    }
}

// New history of star s: its old history (mode 1) merged with this pass's insertions ins[0, m)
// (sorted, disjoint from the old list) into the star's new region.  Returns the old length.
__device__ __forceinline__ int star_history_merge(const StarParams &p, int s, const int *ins, int m, int tid, int nt)
{
    const int64_t ho = p.nhoff[s];
    if (p.mode == 0) {
        for (int i = tid; i < m; i += nt) p.hpool[ho + i] = ins[i];
        return 0;
    }
    const int64_t hb = p.hoff[s];
    const int hn = p.hnum[s];
    const int *old = p.hpool + hb;
    for (int i = tid; i < hn; i += nt) {
        const int x = old[i];
        int lo = 0, hi = m;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (ins[mid] < x) lo = mid + 1;
            else hi = mid;
        }
        p.hpool[ho + i + lo] = x;
    }
    for (int i = tid; i < m; i += nt) {
        const int x = ins[i];
        int lo = 0, hi = hn;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (old[mid] < x) lo = mid + 1;
            else hi = mid;
        }
        p.hpool[ho + i + lo] = x;
    }
    return hn;
}

// Points star s's record at its rebuilt regions (one thread, after every read of the old
// record and regions).
__device__ __forceinline__ void star_commit(const StarParams &p, int s, int vcount, int64_t vo, int tcount, int64_t to,
                                            int hcount)
{
    p.vnum[s] = vcount;
    p.voff[s] = vo;
    p.tnum[s] = tcount;
    p.toff[s] = to;
    p.hnum[s] = hcount;
    p.hoff[s] = p.nhoff[s];
}

// EXACT = false: filters only.  A star with an inconclusive orientation is handed to
// p.exact_list untouched (its output is written only at the end), so the kernel carries no
// multiprecision code.  Its registers then have room for the cofactors of the lane's own slots, with
// two permanents each (the largest of the three coordinates', and the lift's), which only that lane
// reads: without them in LDS a 256-vertex star takes 25 KB instead of 57 and six waves share a CU
// instead of two.  At the occupancies below 50 to 150 bytes a lane of other values spill.
template <int VMAX, bool EXACT>
__device__ __forceinline__ void star_body(const StarParams &p, int nitems, int bid, int nblk)
{
    constexpr bool REGC = !EXACT;
    constexpr bool COUNT = !EXACT && VMAX == STAR_VMAX_T0; // the statistics are the 32-vertex kernel's
    using Lds = StarLds<VMAX, !REGC>;
    constexpr int TMAX = Lds::TMAX;
    constexpr int KPL = TMAX / 64, UNROLL = REGC ? KPL : 1;
    __shared__ Lds L;
    double rc[REGC ? KPL : 1][4], rp[REGC ? KPL : 1][2];
    const int lane = threadIdx.x;
    unsigned long long *cnt = p.cnt;

    if (EXACT && p.nlist_dev) {
        const unsigned long long c = *p.nlist_dev;
        nitems = c < (unsigned long long)nitems ? (int)c : nitems;
    }
    // A list no longer than the grid is spread one star per work-group, without the queue;
    // work-groups beyond its length leave at once (thousands of idle work-groups contending for
    // the queue counter cost ~0.3 ms).  Longer lists go through the work queue in chunks: one
    // atomic per STAR_CHUNK stars for the filter-only kernels (many small stars), per star for
    // the exact ones (uneven cost).
    constexpr int CHUNK = EXACT ? 1 : STAR_CHUNK;
    const bool one_each = nitems <= nblk;
    if (bid >= nitems) return;
    bool first = true;
    int nfilt = 0, ncof = 0; // this lane's cofactor-filter evaluations and cofactor computations
    unsigned long long npairs = 0, ndrown = 0; // the wave's
    for (;;) {
        int base = 0;
        if (one_each) {
            base = first ? bid : nitems;
            first = false;
        } else {
            if (lane == 0) base = (int)atomicAdd(&cnt[p.work_counter], (unsigned long long)CHUNK);
            base = __shfl(base, 0, 64);
        }
        if (base >= nitems) break;
        const int bend = one_each ? base + 1 : (base + CHUNK < nitems ? base + CHUNK : nitems);
#pragma unroll 1
        for (int item = base; item < bend; item++) {
            const int s = p.star_list[item];
            if (s < 0) continue; // on another tier's list
            const int64_t ib = p.ins_off[s];
            const int m = (int)(p.ins_off[s + 1] - ib);
            const int vn = p.mode ? p.vnum[s] : 0;
            const int need = vn + m;
            const int lim = VMAX < p.lds_limit ? VMAX : p.lds_limit;
            if (need > lim) {
                if (EXACT) star_list_push(p.defer_list, p.defer_cap, &cnt[p.defer_counter], s, cnt);
                else if (lane == 0) // not the list of this tier
                    atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_BUFFER);
                continue;
            }
            if (p.mode == 0 && m < 4) {
                if (lane == 0) {
                    atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_CONE);
                    p.vnum[s] = 0;
                    p.tnum[s] = 0;
                }
                continue;
            }
            if (p.mode == 1 && m == 0) continue; // untouched star: stays where it is
            const double sx = p.pts[3 * (int64_t)s], sy = p.pts[3 * (int64_t)s + 1], sz = p.pts[3 * (int64_t)s + 2];
            // Insertion q takes link-vertex slot vn + q; every insertion's coordinates are fetched
            // here at once instead of one dependent load per insertion step.  (In mode 0 the
            // first four form the initial simplex, set up below.)
            const int q0 = p.mode ? 0 : 4;
            for (int q = lane; q < m; q += 64) {
                const int g = (int)(uint32_t)p.ins_keys[ib + q];
                L.ins[q] = g;
                L.ins_local[q] = -1;
                if (q >= q0) {
                    L.vid[vn + q] = g;
                    rel_coords(p.pts, g, sx, sy, sz, L.vc[vn + q]);
                }
            }
            int T, nfree = 0;
            if (p.mode == 1) {
                const int tn = p.tnum[s];
                const int64_t vi = p.voff[s], ti = p.toff[s];
                for (int v = lane; v < vn; v += 64) {
                    const int g = p.vpool[vi + v];
                    L.vid[v] = g;
                    rel_coords(p.pts, g, sx, sy, sz, L.vc[v]);
                }
                for (int t = lane; t < tn; t += 64) {
                    const uint64_t h = p.tpool[ti + t];
                    L.tv[t] = tpack(hvert(h, 0), hvert(h, 1), hvert(h, 2), TF_ALIVE | (hchecked(h) ? TF_CHECKED : 0u));
                    L.to[t][0] = (uint16_t)hopp(h, 0);
                    L.to[t][1] = (uint16_t)hopp(h, 1);
                    L.to[t][2] = (uint16_t)hopp(h, 2);
                }
                T = tn;
            } else {
                // initial 4-simplex (GD/GDelaunay/GDelPredKernels.cu:45-158)
                int l[4];
                for (int i = 0; i < 4; i++) l[i] = (int)(uint32_t)p.ins_keys[ib + i];
                const double *pp[5] = {p.pts + 3 * (int64_t)l[0], p.pts + 3 * (int64_t)l[1], p.pts + 3 * (int64_t)l[2],
                                       p.pts + 3 * (int64_t)l[3], p.pts + 3 * (int64_t)s};
                const int idx[5] = {l[0], l[1], l[2], l[3], s};
                const int o = EXACT ? orient4_full(pp, idx, cnt) : filter_insphere(pp);
                if (!EXACT && o == 0) {
                    star_list_push(p.exact_list, p.exact_cap, &cnt[p.exact_counter], s, cnt);
                    continue;
                }
                const bool sw = o < 0;
                if (sw) {
                    const int t = l[0];
                    l[0] = l[1];
                    l[1] = t;
                }
                if (lane < 4) {
                    L.vid[lane] = l[lane];
                    rel_coords(p.pts, l[lane], sx, sy, sz, L.vc[lane]);
                    // cone triangles (link triangles seen from the star point) and adjacency
                    const int lt[4][3] = {{1, 2, 3}, {0, 3, 2}, {0, 1, 3}, {0, 2, 1}};
                    L.tv[lane] = tpack(lt[lane][0], lt[lane][1], lt[lane][2], TF_ALIVE);
                    L.to[lane][0] = (uint16_t)lt[lane][0];
                    L.to[lane][1] = (uint16_t)lt[lane][1];
                    L.to[lane][2] = (uint16_t)lt[lane][2];
                    const int local = (lane < 2 && sw) ? 1 - lane : lane;
                    L.ins_local[lane] = (int16_t)local;
                }
                T = 4;
            }
            wave_sync();
            // The cofactors of this lane's slots k of the mask: registers are filled by rounds, a slot
            // of each lane per round, so that a few new triangles spread over the lanes cost a
            // round or two and not one for every k that some lane needs.
            auto cofactors = [&](unsigned km) {
                if constexpr (REGC) {
                    while (__ballot(km != 0)) {
                        const int k = km ? __builtin_ctz(km) : KPL;
                        double C[4], P[4];
                        if (km) {
                            const uint32_t t = L.tv[lane + 64 * k];
                            tri_cofactors(L.vc[tvert(t, 0)], L.vc[tvert(t, 1)], L.vc[tvert(t, 2)], C, P);
                            L.tv[lane + 64 * k] = t & ~TF_FRESH;
                            if (COUNT) ncof++;
                        }
#pragma unroll
                        for (int i = 0; i < KPL; i++)
                            if (i == k) {
#pragma unroll
                                for (int j = 0; j < 4; j++) rc[i][j] = C[j];
                                rp[i][0] = fmax(P[0], fmax(P[1], P[2]));
                                rp[i][1] = P[3];
                            }
                        km &= km - 1;
                    }
                } else {
#pragma unroll 1
                    for (int k = 0; k < KPL; k++)
                        if ((km >> k) & 1) {
                            const int slot = lane + 64 * k;
                            const uint32_t t = L.tv[slot];
                            lds_cofactors<TMAX>(L.vc[tvert(t, 0)], L.vc[tvert(t, 1)], L.vc[tvert(t, 2)], L.cof, slot);
                            L.tv[slot] = t & ~TF_FRESH;
                            if (COUNT) ncof++;
                        }
                }
            };
            cofactors(T > lane ? (unsigned)((1ull << ((T - lane + 63) / 64)) - 1ull) : 0u);
            bool failed = false, unsure = false;
            for (int q = q0; q < m; q++) {
                const int gv = L.ins[q];
                const int Vn = vn + q;
                const double r[4] = {L.vc[Vn][0], L.vc[Vn][1], L.vc[Vn][2], L.vc[Vn][3]};
                int nv = 0;
                unsigned vm = 0; // bit k: slot lane + 64 k sees the vertex
                unsigned um = 0; // bit k: its filter is inconclusive
                const double rsum = fabs(r[0]) + fabs(r[1]) + fabs(r[2]);
#pragma unroll UNROLL
                for (int k = 0; k < KPL; k++) {
                    const int slot = lane + 64 * k;
                    if (REGC && 64 * k >= T) break; // wave-uniform: a small star in a large tier
                    if (slot < T) {
                        const uint32_t t = L.tv[slot];
                        if ((t & (TF_ALIVE | TF_VIS)) == TF_ALIVE) {
                            if (COUNT) nfilt++;
                            int sg;
                            if constexpr (REGC) {
                                sg = cofactor_filter_sign2(r, rsum, rc[k], rp[k][0], rp[k][1]);
                            } else {
                                double c[8];
#pragma unroll
                                for (int j = 0; j < 8; j++) c[j] = L.cof[j][slot];
                                sg = cofactor_filter_sign(r, c, c + 4);
                            }
                            if (sg == 0) um |= 1u << k;
                            if (sg < 0) {
                                L.tv[slot] = t | TF_VIS;
                                vm |= 1u << k;
                                nv++;
                            }
                        }
                    }
                }
                if (__ballot(um != 0)) {
                    if (!EXACT) {
                        unsure = true;
                        break;
                    }
                    // The inconclusive slots of the whole wave in one list (be_slot is free until the
                    // new triangles), decided 64 at a time: slot by slot in their owners' lanes a
                    // 256-vertex star paid up to eight exact evaluations per insertion, each with
                    // a few lanes active.
                    const int nu = __popc(um);
                    const int uinc = g4d_wave_incl_sum(nu), nutot = __builtin_amdgcn_readlane(uinc, 63);
                    int upos = uinc - nu;
#pragma unroll 1
                    for (int k = 0; k < KPL; k++)
                        if ((um >> k) & 1) L.be_slot[upos++] = (uint16_t)(lane + 64 * k);
                    wave_sync();
                    for (int x = lane; x < nutot; x += 64) {
                        const int slot = L.be_slot[x];
                        const uint32_t t = L.tv[slot];
                        const int a = L.vid[tvert(t, 0)], b = L.vid[tvert(t, 1)], c = L.vid[tvert(t, 2)];
                        const double *pp[5] = {p.pts + 3 * (int64_t)a, p.pts + 3 * (int64_t)b, p.pts + 3 * (int64_t)c,
                                               p.pts + 3 * (int64_t)s, p.pts + 3 * (int64_t)gv};
                        const int idx[5] = {a, b, c, s, gv};
                        if (orient4_full(pp, idx, cnt) < 0) L.tv[slot] = t | TF_VIS;
                    }
                    wave_sync();
#pragma unroll 1
                    for (int k = 0; k < KPL; k++)
                        if (((um >> k) & 1) && (L.tv[lane + 64 * k] & TF_VIS)) {
                            vm |= 1u << k;
                            nv++;
                        }
                }
                const int vinc = g4d_wave_incl_sum(nv);
                const int vbase = vinc - nv, nvis = __builtin_amdgcn_readlane(vinc, 63);
                if (nvis == 0) continue; // drowned at insertion
                if (lane == 0) L.ins_local[q] = (int16_t)Vn;
                // the visible slots join the free list (positions nfree .. nfree + nvis - 1)
                {
                    int fpos = nfree + vbase;
#pragma unroll 1
                    for (int k = 0; k < KPL; k++)
                        if ((vm >> k) & 1) L.freel[fpos++] = (uint16_t)(lane + 64 * k);
                }
                wave_sync();
                // Hole boundary: the edges of visible triangles whose neighbour is not visible, in
                // the order of the visible list; entry x is taken by lane x mod 64.  The edge's
                // position in the neighbour u is that of u's vertex off the edge.
                int nbtot = 0;
                for (int x0 = 0; x0 < nvis; x0 += 64) {
                    const int x = x0 + lane;
                    const bool own = x < nvis;
                    uint32_t t = 0u;
                    uint64_t o = 0ull;
                    if (own) {
                        const int slot = L.freel[nfree + x];
                        t = L.tv[slot];
                        o = L.to64[slot];
                    }
                    uint32_t tu[3] = {TF_VIS, TF_VIS, TF_VIS};
                    if (own)
#pragma unroll
                        for (int i = 0; i < 3; i++) tu[i] = L.tv[(int)(o >> (16 * i)) & (TMAX - 1)];
                    int nb = 0;
#pragma unroll
                    for (int i = 0; i < 3; i++) nb += (tu[i] & TF_VIS) ? 0 : 1;
                    const int binc = g4d_wave_incl_sum(nb);
                    int e = nbtot + binc - nb;
#pragma unroll
                    for (int i = 0; i < 3; i++) {
                        if (tu[i] & TF_VIS) continue;
                        const int a = tvert(t, (i + 1) % 3), b = tvert(t, (i + 2) % 3);
                        const int u0 = tvert(tu[i], 0), u1 = tvert(tu[i], 1);
                        if (e < TMAX) {
                            L.be_a[e] = (uint16_t)a;
                            L.be_b[e] = (uint16_t)b;
                            L.be_u[e] = (uint16_t)(o >> (16 * i));
                            L.be_j[e] = (uint8_t)((u0 != a && u0 != b) ? 0 : ((u1 != a && u1 != b) ? 1 : 2));
                        }
                        e++;
                    }
                    nbtot += __builtin_amdgcn_readlane(binc, 63);
                }
                // The visible triangles keep their words, TF_VIS marking them dead, until a new
                // triangle takes the slot: boundary edge k takes free slot nfree_tot - 1 - k (the
                // visible ones first) or, past the free list, slot T + k - nfree_tot.
                const int nfree_tot = nfree + nvis;
                const int newT = T + (nbtot > nfree_tot ? nbtot - nfree_tot : 0);
                if (nbtot > TMAX || nbtot < 3 || newT > TMAX || Vn + 1 > VMAX) {
                    failed = true;
                    break;
                }
                wave_sync();
                for (int k = lane; k < nbtot; k += 64) {
                    const int slot = k < nfree_tot ? L.freel[nfree_tot - 1 - k] : T + (k - nfree_tot);
                    const int a = L.be_a[k], b = L.be_b[k], u = L.be_u[k];
                    L.be_slot[k] = (uint16_t)slot;
                    L.tv[slot] = tpack(a, b, Vn, TF_ALIVE | TF_FRESH);
                    L.to[slot][2] = (uint16_t)u;
                    L.to[u][L.be_j[k]] = (uint16_t)slot;
                    L.vstart[a] = (int16_t)slot;
                    L.vend[b] = (int16_t)slot;
                }
                wave_sync();
                for (int k = lane; k < nbtot; k += 64) {
                    const int slot = L.be_slot[k];
                    L.to[slot][0] = (uint16_t)L.vstart[L.be_b[k]];
                    L.to[slot][1] = (uint16_t)L.vend[L.be_a[k]];
                }
                nfree = nfree_tot - (nbtot < nfree_tot ? nbtot : nfree_tot);
                T = newT;
                // the link writes above touch only the new slots' neighbour rows: the cofactor
                // pass below (triangle words, coordinates, this lane's cofactor columns) needs no
                // barrier after them
                unsigned fm = 0;
#pragma unroll UNROLL
                for (int k = 0; k < KPL; k++) {
                    if (REGC && 64 * k >= T) break;
                    if (lane + 64 * k < T && (L.tv[lane + 64 * k] & TF_FRESH)) fm |= 1u << k;
                }
                cofactors(fm);
                // No barrier before the next step: its filter reads and writes only this lane's
                // own slots and cofactor columns and the listed coordinates, and its first barrier
                // precedes any read of another lane's words.
            }
            wave_sync();
            if (unsure) {
                star_list_push(p.exact_list, p.exact_cap, &cnt[p.exact_counter], s, cnt);
                wave_sync();
                continue;
            }
            if (failed) {
                if (lane == 0) {
                    atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_HOLE);
                    p.vnum[s] = 0;
                    p.tnum[s] = 0;
                }
                wave_sync();
                continue;
            }
            // ---- finalize: link set, drowned insertions, compaction, pairs, history ----
            const int V = need; // drowned insertions' slots are never referenced and drop out
            for (int v = lane; v < V; v += 64) L.present[v] = 0;
            wave_sync();
#pragma unroll 1
            for (int k = 0; k < KPL; k++) {
                const int slot = lane + 64 * k;
                if (slot < T) {
                    const uint32_t t = L.tv[slot];
                    if ((t & (TF_ALIVE | TF_VIS)) == TF_ALIVE) {
                        L.present[tvert(t, 0)] = 1;
                        L.present[tvert(t, 1)] = 1;
                        L.present[tvert(t, 2)] = 1;
                    }
                }
            }
            wave_sync();
            int drowned = 0;
            for (int b0 = 0; b0 < m; b0 += 64) {
                const int q = b0 + lane, lv = q < m ? L.ins_local[q] : 0;
                const bool dr = q < m && (lv < 0 || !L.present[lv]);
                if (q < m) p.dflag[ib + q] = dr ? 1 : 0;
                drowned += __popcll(__ballot(dr));
            }
            // vertex compaction
            const int64_t vo = p.nvoff[s], to = p.ntoff[s];
            int vcount = 0;
            for (int base = 0; base < V; base += 64) {
                const int v = base + lane;
                const bool pr = v < V && L.present[v];
                int tot;
                const int rk = g4d_wave_excl_count(pr, &tot);
                if (pr) {
                    L.vremap[v] = (uint16_t)(vcount + rk);
                    p.vpool[vo + vcount + rk] = L.vid[v];
                }
                vcount += tot;
            }
            int tcount = 0;
            for (int base = 0; base < T; base += 64) {
                const int t = base + lane;
                const bool al = t < T && (L.tv[t] & (TF_ALIVE | TF_VIS)) == TF_ALIVE;
                int tot;
                const int rk = g4d_wave_excl_count(al, &tot);
                if (al) L.remap[t] = (uint16_t)(tcount + rk);
                tcount += tot;
            }
            if (tcount > 2 * need - 4 || tcount != 2 * vcount - 4) {
                // not a triangulated 2-sphere: report instead of writing past the star's region
                if (lane == 0) {
                    atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_HOLE);
                    p.vnum[s] = 0;
                    p.tnum[s] = 0;
                }
                wave_sync();
                continue;
            }
            wave_sync();
            const int64_t pb = 2 * (to - p.tbase);
            int npair = 0;
            for (int base = 0; base < T; base += 64) {
                const int t = base + lane;
                uint32_t tt = 0;
                if (t < T) tt = L.tv[t];
                TriPairs pr{STAR_PAIR_NONE, STAR_PAIR_NONE};
                if (t < T && (tt & (TF_ALIVE | TF_VIS)) == TF_ALIVE) {
                    const int a = tvert(tt, 0), b = tvert(tt, 1), c = tvert(tt, 2);
                    const int d = L.remap[t];
                    p.tpool[to + d] = hpack(L.vremap[a], L.vremap[b], L.vremap[c], L.remap[L.to[t][0]],
                                            L.remap[L.to[t][1]], L.remap[L.to[t][2]], true);
                    pr = star_tri_pairs(L.vid[a], L.vid[b], L.vid[c], !(tt & TF_CHECKED));
                }
                // the star's pairs, dense, in triangle order
                const int np = (pr.x != STAR_PAIR_NONE ? 1 : 0) + (pr.y != STAR_PAIR_NONE ? 1 : 0);
                int tot;
                const int at = npair + wave_excl<2>(np, &tot);
                if (np > 0) p.pairbuf[pb + at] = pr.x;
                if (np > 1) p.pairbuf[pb + at + 1] = pr.y;
                npair += tot;
            }
            if (lane == 0) p.pcount[s] = npair;
            npairs += npair;
            ndrown += drowned;
            const int hn = star_history_merge(p, s, L.ins, m, lane, 64);
            wave_sync();
            if (lane == 0) star_commit(p, s, vcount, vo, tcount, to, hn + m);
            wave_sync();
        }
    }
    if (COUNT) {
        const int wf = g4d_wave_sum(nfilt), wc = g4d_wave_sum(ncof);
        if (lane == 0) {
            atomicAdd(&cnt[G4D_CNT_ORIENT4], (unsigned long long)wf);
            atomicAdd(&cnt[G4D_CNT_COFACTOR], (unsigned long long)wc);
        }
    }
    if (lane == 0) {
        if (npairs) atomicAdd(&cnt[G4D_CNT_PAIRS], npairs);
        if (ndrown) atomicAdd(&cnt[G4D_CNT_DROWNED], ndrown);
    }
}

// The 32-vertex tier with one star a wave, selectable: 3.2 KB of LDS, five waves per SIMD (96 VGPRs, 148
// bytes spilled).  At 4,194,304 uniform points 46.8 ms where the grouped kernel below takes 15.3.
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(5, 8))) k_star32(StarParams p, int nitems)
{
    star_body<STAR_VMAX_T0, false>(p, nitems, blockIdx.x, gridDim.x);
}

// The exact predicates' callee takes 256 VGPRs, 34 to 43 AGPRs and 2,368 bytes of scratch a lane (the
// integer forms for wide coordinates): one wave per SIMD.  Bound by that callee's latency in the few
// lanes whose signs are open.
template <int VMAX>
__global__ void __launch_bounds__(64) k_star_exact(StarParams p, int nitems)
{
    star_body<VMAX, true>(p, nitems, blockIdx.x, gridDim.x);
}

// The filter-only tiers above 32: the registers that each occupancy leaves, measured on 1,000,000
// clustered points (12 passes): 64 vertices at 3, 4, 5 waves per SIMD 11.0, 9.9, 10.5 ms; 128 at
// 2, 3 waves 9.5, 8.3 ms; 256 at 2 waves 8.5 ms.  With cofactors in LDS and no 128-vertex tier
// the 64-vertex stars took 11.7 ms and all larger ones 38.8.
template <int VMAX, int WPE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE, 8))) k_star(StarParams p, int nitems)
{
    star_body<VMAX, false>(p, nitems, blockIdx.x, gridDim.x);
}

// ------------------------------------------------------------------------------------
// Grouped 32-vertex star kernel: one star per group of GL lanes, 64 / GL stars per wave.
//
// The one-star-per-wave kernel leaves most lanes idle on a star of this tier (at most 60
// triangle slots, about 27 live) and pays its chain of ballots and wave-level barriers per
// insertion of one star; here the chain is shared by 64 / GL stars.  Each lane owns KPL =
// 64 / GL triangle slots (gl, gl + GL, ...) and keeps their cofactors and permanents in
// registers (only the owning lane ever reads or writes them), so a star's LDS holds only its
// link vertices, triangles and hole-boundary lists (2 KB).  Every barrier and ballot is
// reached by the whole wave in uniform control flow: the insertion loop runs to the largest
// insertion count of the wave's stars, and a group with nothing to do in a step has its work
// masked off.  Filters only (no multiprecision code): a star with an inconclusive orientation
// goes to p.exact_list untouched; a star beyond the tier is left to the plan's lists.
//
// Bound by vector instructions (two thirds of the issue slots at three waves per SIMD, of them a
// fifth FP64), with the LDS pipe half busy.  At 4,194,304 uniform points (G = 512) its passes took
// 22.3 ms with 16-bit indices and the permanents of every triangle; 2 KB a star, which lets four waves
// share a SIMD, one word per boundary edge, the cheap bound in place of the permanents (70 instructions
// a triangle slot before, 43 now) and packed scans: 15.3 ms.
// ------------------------------------------------------------------------------------

static constexpr uint32_t GF_ALIVE = 1u << 31; // a triangle of the star as it stands (the sign of the word)

struct StarGrpLds {
    static constexpr int VMAX = STAR_VMAX_T0;
    static constexpr int TMAX = 2 * VMAX;
    double vc[VMAX][4];
    int vid[VMAX];
    uint32_t tv[TMAX];
    uint32_t to[TMAX]; // neighbours across the edges opposite vertices 0-2, a byte each
    union {
        uint32_t be[TMAX]; // hole boundary: a, b, u | j << 6, then the edge's slot, a byte each
        struct {           // finalisation
            uint8_t present[VMAX], vremap[VMAX], remap[TMAX];
        };
    };
    uint8_t freel[TMAX];
    uint8_t vstart[VMAX], vend[VMAX];
    uint8_t ord[VMAX]; // insertion order: list indices by distance to the star point
    // 2,112 bytes: bytes for indices (all below 64), so that four waves fit each SIMD; at 64 mod 256
    // the groups' blocks start 16 banks apart (mod 64), and accesses of the groups at the same
    // offsets meet in no bank.
    uint8_t pad[32];
};
static_assert(sizeof(StarGrpLds) % 256 == 64, "group blocks start 16 banks apart");
static_assert(StarGrpLds::TMAX <= 64, "indices fit their bytes, slots the boundary word's six bits");

// Ballot of this lane's group of GL lanes, shifted down to bit 0.
template <int GL>
__device__ __forceinline__ uint64_t grp_ballot(bool pred, int g)
{
    const uint64_t m = __ballot(pred);
    return GL == 64 ? m : (m >> (g * GL)) & ((1ull << GL) - 1ull);
}

// Inclusive prefix sums over each DPP row of 16 lanes (row_shr 1, 2, 4, 8) and every lane's row
// total (row_ror 8, 4, 2, 1); lanes whose shifted source lies outside the row add 0.  Every lane
// of the wave must be active.
__device__ __forceinline__ int row16_scan(int v, int *tot)
{
    int x = v, a = v;
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
    a += __builtin_amdgcn_update_dpp(0, a, 0x128, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
    a += __builtin_amdgcn_update_dpp(0, a, 0x124, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
    a += __builtin_amdgcn_update_dpp(0, a, 0x122, 0xf, 0xf, false);
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
    a += __builtin_amdgcn_update_dpp(0, a, 0x121, 0xf, 0xf, false);
    *tot = a;
    return x;
}

// Exclusive scan of per-lane counts below 2^BITS within the group; total in *tot.  Groups of 16
// lanes are DPP rows and scan any counts whose group sum stays below 2^31.
template <int GL, int BITS>
__device__ __forceinline__ int grp_excl(int v, int g, int gl, int *tot)
{
    if constexpr (GL == 16) return row16_scan(v, tot) - v;
    const uint64_t below = gl == 0 ? 0ull : (~0ull >> (64 - gl));
    int pre = 0, all = 0;
#pragma unroll
    for (int b = 0; b < BITS; b++) {
        const uint64_t m = grp_ballot<GL>((v >> b) & 1, g);
        pre += __popcll(m & below) << b;
        all += __popcll(m) << b;
    }
    *tot = all;
    return pre;
}

// Exclusive scans within the group, and totals, of NF flags (BITS = 1) or counts below 2^BITS each: in
// groups of 16 lanes the fields travel packed through one scan.
template <int GL, int BITS, int NF>
__device__ __forceinline__ void grp_excl_n(const int (&v)[NF], int g, int gl, int (&pre)[NF], int (&tot)[NF])
{
    if constexpr (GL == 16) {
        constexpr int W = 4 + BITS; // sums up to 16 (2^BITS - 1)
        static_assert(NF * W <= 32, "packed sums fit a word");
        uint32_t pk = 0u;
#pragma unroll
        for (int k = 0; k < NF; k++) pk |= (uint32_t)v[k] << (W * k);
        int t;
        const uint32_t x = (uint32_t)row16_scan((int)pk, &t) - pk;
#pragma unroll
        for (int k = 0; k < NF; k++) {
            pre[k] = (int)((x >> (W * k)) & ((1u << W) - 1u));
            tot[k] = (int)(((uint32_t)t >> (W * k)) & ((1u << W) - 1u));
        }
    } else {
#pragma unroll
        for (int k = 0; k < NF; k++) pre[k] = grp_excl<GL, BITS>(v[k], g, gl, &tot[k]);
    }
}

// A triangle slot's cofactors with the four permanents in FP64, or (PF) with tri_cofactors_m's bound on
// them in FP32; rs2 = |x| + |y| + |z| + l of r2.
template <bool PF> struct GrpBound {
    double p[4];
};
template <> struct GrpBound<true> {
    float m;
};
__device__ __forceinline__ void grp_cofactors(const double *r0, const double *r1, const double *r2, double, double,
                                              double *C, GrpBound<false> &P)
{
    tri_cofactors(r0, r1, r2, C, P.p);
}
__device__ __forceinline__ void grp_cofactors(const double *r0, const double *r1, const double *r2, double a2, double rs2,
                                              double *C, GrpBound<true> &P)
{
    P.m = (float)tri_cofactors_m(r0, r1, r2, a2, rs2, C);
}
// The vertex being inserted: its row's sums, and for PF the factors of the bound.  What decides whether a
// star goes to the exact kernel (whose triangles come in another order) is 32 u rs max_j P_j with the
// largest permanent rounded up to FP32; the bound m is no smaller than that, its roundings (2^-24 in FP32,
// a dozen in FP64) within the 2^-20 and what the denormals lose within tiny.  A sign that it leaves open is
// decided by the permanents themselves (grp_filter_tail).
struct GrpRow {
    double a, rs, as, tiny;
};
__device__ __forceinline__ GrpRow grp_row(const double *r)
{
    GrpRow w;
    w.a = fabs(r[0]) + fabs(r[1]) + fabs(r[2]);
    w.rs = w.a + r[3];
    w.as = 32.0 * 1.1102230246251565e-16 * (1.0 + 0x1p-20) * w.rs;
    w.tiny = fma(w.as, 3e-45, 1e-249);
    return w;
}
__device__ __forceinline__ int grp_filter_sign(const double *r, const GrpRow &, const double *C, const GrpBound<false> &P)
{
    return cofactor_filter_sign(r, C, P.p);
}
__device__ __forceinline__ int grp_filter_sign(const double *r, const GrpRow &w, const double *C, const GrpBound<true> &P)
{
    const double val = fma(r[3], C[3], fma(r[2], C[2], fma(r[1], C[1], r[0] * C[0])));
    const double bnd = fma(w.as, (double)P.m, w.tiny);
    return val > bnd ? 1 : (-val > bnd ? -1 : 0);
}
__device__ __forceinline__ int grp_filter_tail(const double *r0, const double *r1, const double *r2,
                                                         const double *r)
{
    double C[4], P[4];
    tri_cofactors(r0, r1, r2, C, P);
    const float p = __double2float_ru(fmax(fmax(P[0], P[1]), fmax(P[2], P[3])));
    const double val = fma(r[3], C[3], fma(r[2], C[2], fma(r[1], C[1], r[0] * C[0])));
    const double per = (fabs(r[0]) + fabs(r[1]) + fabs(r[2]) + r[3]) * (double)p;
    const double bnd = 32.0 * 1.1102230246251565e-16 * per;
    if (!(per > 1e-250)) return 0;
    return val > bnd ? 1 : (-val > bnd ? -1 : 0);
}

// Largest value over the wave for non-negative v: maxima within each 16-lane row by DPP row
// rotations (8, 4, 2, 1), then the four rows' maxima read into scalars.  Every lane must be
// active.
__device__ __forceinline__ int wave_max_i(int v)
{
    int x = v;
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x124, 0xf, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x122, 0xf, 0xf, false));
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x121, 0xf, 0xf, false));
    const int r0 = __builtin_amdgcn_readlane(x, 0), r1 = __builtin_amdgcn_readlane(x, 16);
    const int r2 = __builtin_amdgcn_readlane(x, 32), r3 = __builtin_amdgcn_readlane(x, 48);
    return max(max(r0, r1), max(r2, r3));
}

template <int GL, bool PF, bool COUNT = true>
__device__ __forceinline__ void star_body_grp(const StarParams &p, int nitems, int bid, int nblk)
{
    constexpr int NG = 64 / GL;
    constexpr int VMAX = StarGrpLds::VMAX, TMAX = StarGrpLds::TMAX;
    constexpr int KPL = TMAX / GL;
    __shared__ StarGrpLds Ls[NG];
    __shared__ int order[NG * STAR_CHUNK]; // the chunk's items by insertion count
    const int lane = threadIdx.x, g = lane / GL;
    int gl = lane % GL;
    StarGrpLds &L = Ls[g];
    unsigned long long *cnt = p.cnt;

    // Work unit: a batch of NG consecutive list entries, one per group.  As many batches as
    // work-groups or fewer: one batch each, no queue; otherwise STAR_CHUNK batches per atomic.
    const int nbatch = (nitems + NG - 1) / NG;
    const bool one_each = nbatch <= nblk;
    if (bid >= nbatch) return;
    bool first = true;
    int nfilt = 0, ncof = 0;
    unsigned long long npairs = 0, ndrown = 0; // the wave's
    for (;;) {
        int base = 0;
        if (one_each) {
            base = first ? bid : nbatch;
            first = false;
        } else {
            if (lane == 0) base = (int)atomicAdd(&cnt[p.work_counter], (unsigned long long)STAR_CHUNK);
            base = __shfl(base, 0, 64);
        }
        if (base >= nbatch) break;
        const int bend = one_each ? base + 1 : (base + STAR_CHUNK < nbatch ? base + STAR_CHUNK : nbatch);
        // The chunk's stars are dealt to batches in order of their insertion counts, so that the
        // four stars of a batch (which step through their insertions in lock-step) need about as
        // many steps each; within a chunk of 32 consecutive stars the order keeps their locality.
        {
            const int nit = (bend - base) * NG;
            const int my = base * NG + lane;
            int key = INT_MAX;
            if (lane < nit && my < nitems) {
                const int s = p.star_list[my];
                key = s < 0 ? 0 : (int)(p.ins_off[s + 1] - p.ins_off[s]);
            }
            int rank = 0;
#pragma unroll
            for (int j = 0; j < NG * STAR_CHUNK; j++) {
                const int kj = __shfl(key, j, 64);
                rank += (kj < key || (kj == key && j < lane)) ? 1 : 0;
            }
            if (lane < nit) order[rank] = my;
            wave_sync();
        }
#pragma unroll 1
        for (int batch = base; batch < bend; batch++) {
            // addresses made from gl are made again for each batch: kept across it they would cost
            // more registers than four waves per SIMD leave
            asm volatile("" : "+v"(gl));
            const int item = order[(batch - base) * NG + g];
            // ---- this group's star: checks, then its link and insertions into LDS ----
            const int entry = item < nitems ? p.star_list[item] : -1;
            bool act = entry >= 0; // below: on another tier's list
            const int s = act ? entry : 0;
            const int64_t ib = act ? p.ins_off[s] : 0;
            const int m = act ? (int)(p.ins_off[s + 1] - ib) : 0;
            const int vn = act && p.mode ? p.vnum[s] : 0;
            const int need = vn + m;
            const int lim = VMAX < p.lds_limit ? VMAX : p.lds_limit;
            if (act && need > lim) { // not the list of this tier
                if (gl == 0) atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_BUFFER);
                act = false;
            }
            if (act && p.mode == 0 && m < 4) {
                if (gl == 0) {
                    atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_CONE);
                    p.vnum[s] = 0;
                    p.tnum[s] = 0;
                }
                act = false;
            }
            if (act && p.mode == 1 && m == 0) act = false;
            double sx = 0.0, sy = 0.0, sz = 0.0;
            if (act) {
                sx = p.pts[3 * (int64_t)s];
                sy = p.pts[3 * (int64_t)s + 1];
                sz = p.pts[3 * (int64_t)s + 2];
            }
            const int q0 = p.mode ? 0 : 4;
            // Every listed vertex q takes link-vertex slot vn + q (the cone's four included).
            if (act) {
                for (int q = gl; q < m; q += GL) {
                    const int gv = (int)(uint32_t)p.ins_keys[ib + q];
                    L.vid[vn + q] = gv;
                    rel_coords(p.pts, gv, sx, sy, sz, L.vc[vn + q]);
                }
            }
#pragma unroll
            for (int k = 0; k < KPL; k++) L.tv[gl + GL * k] = 0u;
            wave_sync();
            // Insertion order: nearest to the star point first (ties by list index).  The star
            // that results does not depend on the order (the link is the unique convex hull of
            // the lifted points as seen from the star point, the drowned flags mark listed
            // vertices absent from it, the pairs come from its unchecked triangles), but near
            // vertices are almost all in it: inserted first, they leave the far ones to be
            // rejected by the filter alone, and fewer triangles are made and undone.
            if (act)
                for (int q = gl; q < m; q += GL) {
                    const double dq = L.vc[vn + q][3];
                    int rank = 0;
                    for (int k0 = 0; k0 < m; k0 += 4) { // four reads in flight (indices kept below m)
                        double dk[4];
#pragma unroll
                        for (int i = 0; i < 4; i++) dk[i] = L.vc[vn + (k0 + i < m ? k0 + i : m - 1)][3];
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const int k = k0 + i;
                            rank += (k < m && (dk[i] < dq || (dk[i] == dq && k < q))) ? 1 : 0;
                        }
                    }
                    L.ord[rank] = (uint8_t)q;
                }
            wave_sync();
            int T = 0, nfree = 0;
            bool unsure = false, failed = false;
            if (act && p.mode == 1) {
                const int tn = p.tnum[s];
                const int64_t vi = p.voff[s], ti = p.toff[s];
                for (int v = gl; v < vn; v += GL) {
                    const int gv = p.vpool[vi + v];
                    L.vid[v] = gv;
                    rel_coords(p.pts, gv, sx, sy, sz, L.vc[v]);
                }
                for (int t = gl; t < tn; t += GL) {
                    const uint64_t h = p.tpool[ti + t];
                    L.tv[t] = tpack(hvert(h, 0), hvert(h, 1), hvert(h, 2), GF_ALIVE | (hchecked(h) ? TF_CHECKED : 0u));
                    L.to[t] = (uint32_t)hopp(h, 0) | ((uint32_t)hopp(h, 1) << 8) | ((uint32_t)hopp(h, 2) << 16);
                }
                T = tn;
            } else if (act) {
                // initial 4-simplex (GD/GDelaunay/GDelPredKernels.cu:45-158) on the first four
                // vertices of the insertion order; slot c[i] holds cone vertex i
                int c[4];
                for (int i = 0; i < 4; i++) c[i] = L.ord[i];
                // the cone's coordinates relative to the star point, as listed in LDS (vn = 0)
                const double *pr[4] = {L.vc[c[0]], L.vc[c[1]], L.vc[c[2]], L.vc[c[3]]};
                const int o = filter_insphere_rel(pr);
                if (o == 0) {
                    unsure = true; // pushed to the exact list below, untouched
                } else {
                    if (o < 0) {
                        const int t = c[0];
                        c[0] = c[1];
                        c[1] = t;
                    }
                    if (gl < 4) {
                        const int lt[4][3] = {{1, 2, 3}, {0, 3, 2}, {0, 1, 3}, {0, 2, 1}};
                        L.tv[gl] = tpack(c[lt[gl][0]], c[lt[gl][1]], c[lt[gl][2]], GF_ALIVE);
                        L.to[gl] = (uint32_t)(lt[gl][0] | (lt[gl][1] << 8) | (lt[gl][2] << 16));
                    }
                    T = 4;
                }
            }
            wave_sync();
            bool live = act && !unsure; // the group is building its star
            // declared here, not before the loop over batches: their registers are free outside the insertions
            double C[KPL][4];
            GrpBound<PF> P[KPL];
#pragma unroll
            for (int k = 0; k < KPL; k++) {
                const int slot = gl + GL * k;
                if (live && slot < T) {
                    const uint32_t t = L.tv[slot];
                    const double *r2 = L.vc[tvert(t, 2)];
                    const double a2 = fabs(r2[0]) + fabs(r2[1]) + fabs(r2[2]);
                    grp_cofactors(L.vc[tvert(t, 0)], L.vc[tvert(t, 1)], r2, a2, a2 + r2[3], C[k], P[k]);
                    if (COUNT) ncof++;
                }
            }
            // ---- insertions: every group steps through its list in lock-step ----
            const int qend = wave_max_i(live ? m : 0);
            int jnext = L.ord[q0 < m ? q0 : 0];
            for (int q = q0; q < qend; q++) {
                bool step = live && q < m;
                const int j = step ? jnext : 0; // the list index inserted in this step
                jnext = L.ord[q + 1 < m ? q + 1 : 0]; // the next step's, read a step ahead
                const int Vn = vn + j;
                // this lane's triangle words, read together (every slot index is below TMAX)
                uint32_t tk[KPL];
#pragma unroll
                for (int k = 0; k < KPL; k++) tk[k] = L.tv[gl + GL * k];
                double r[4] = {0.0, 0.0, 0.0, 0.0};
                if (step) {
                    r[0] = L.vc[Vn][0];
                    r[1] = L.vc[Vn][1];
                    r[2] = L.vc[Vn][2];
                    r[3] = L.vc[Vn][3];
                }
                const GrpRow w = grp_row(r);
                int nv = 0;
                unsigned vm = 0; // bit k: slot gl + GL k sees the vertex
                unsigned um = 0; // bit k: the sign is open
                bool unc = false;
#pragma unroll
                for (int k = 0; k < KPL; k++) {
                    if (step && (int)tk[k] < 0) {
                        if (COUNT) nfilt++;
                        const int sg = grp_filter_sign(r, w, C[k], P[k]);
                        if (sg == 0) um |= 1u << k;
                        if (sg < 0) {
                            L.tv[gl + GL * k] = tk[k] & ~GF_ALIVE;
                            vm |= 1u << k;
                            nv++;
                        }
                    }
                }
                if constexpr (!PF) unc = um != 0;
                else if (__builtin_expect(__ballot(um != 0) != 0ull, 0)) {
                    for (; um; um &= um - 1) {
                        const int k = __builtin_ctz(um), slot = gl + GL * k;
                        const uint32_t t = L.tv[slot];
                        const int sg = grp_filter_tail(L.vc[tvert(t, 0)], L.vc[tvert(t, 1)], L.vc[tvert(t, 2)], L.vc[Vn]);
                        if (sg == 0) unc = true;
                        if (sg < 0) {
                            L.tv[slot] = t & ~GF_ALIVE;
                            vm |= 1u << k;
                            nv++;
                        }
                    }
                }
                // every group drowned its vertex at once, or idles: nothing changes in this step
                if (__ballot(step && (nv > 0 || unc)) == 0ull) continue;
                int nvis, vbase;
                bool gunc;
                if constexpr (GL == 16) {
                    // one row scan of two counts: visible triangles (bits 0-7, at most TMAX) and
                    // inconclusive lanes (bits 8-12)
                    static_assert(TMAX < 256, "packed counts fit their fields");
                    const int pk = nv | (unc ? 1 << 8 : 0);
                    int tot;
                    vbase = (row16_scan(pk, &tot) - pk) & 255;
                    nvis = tot & 255;
                    gunc = (tot >> 8) != 0;
                } else {
                    gunc = grp_ballot<GL>(unc, g) != 0ull;
                    vbase = grp_excl<GL, count_bits(KPL)>(nv, g, gl, &nvis);
                }
                if (gunc) {
                    unsure = true;
                    live = false;
                    step = false;
                }
                if (nvis == 0) step = false; // drowned at insertion
                // the visible slots join the free list (positions nfree .. nfree + nvis - 1)
                if (step) {
                    int fpos = nfree + vbase;
#pragma unroll
                    for (int k = 0; k < KPL; k++)
                        if ((vm >> k) & 1) L.freel[fpos++] = (uint8_t)(gl + GL * k);
                }
                wave_sync();
                // Hole boundary: the edges of visible triangles whose neighbour is not visible, in
                // the order of the visible list; its entry x is taken by lane x mod GL.  The edge's
                // position in the neighbour u is that of u's vertex off the edge (all triangles turn
                // the same way round: the edge runs the other way in u).
                int nbtot = 0;
                for (int x0 = 0; __ballot(step && x0 < nvis) != 0ull; x0 += GL) {
                    const int x = x0 + gl;
                    const bool own = step && x < nvis;
                    uint32_t t = 0u, o = 0u;
                    if (own) {
                        const int slot = L.freel[nfree + x];
                        t = L.tv[slot];
                        o = L.to[slot];
                    }
                    uint32_t tu[3] = {0u, 0u, 0u};
                    if (own)
#pragma unroll
                        for (int i = 0; i < 3; i++) tu[i] = L.tv[(o >> (8 * i)) & (TMAX - 1)];
                    int nb = 0;
#pragma unroll
                    for (int i = 0; i < 3; i++) nb += (int)(tu[i] >> 31);
                    int tot;
                    int e = nbtot + grp_excl<GL, 2>(nb, g, gl, &tot);
#pragma unroll
                    for (int i = 0; i < 3; i++) {
                        if ((int)tu[i] >= 0) continue;
                        const int a = tvert(t, (i + 1) % 3), b = tvert(t, (i + 2) % 3);
                        // u has the edge as b, a
                        const int j = tvert(tu[i], 0) == b ? 2 : (tvert(tu[i], 1) == b ? 0 : 1);
                        if (e < TMAX)
                            L.be[e] = (uint32_t)(a | (b << 8) | (j << 22)) | (((o >> (8 * i)) & (TMAX - 1)) << 16);
                        e++;
                    }
                    nbtot += tot;
                }
                // The visible triangles keep their words, no longer alive, until a new triangle takes
                // the slot: boundary edge k takes free slot nfree_tot - 1 - k (the visible ones first)
                // or, past the free list, slot T + k - nfree_tot.
                const int nfree_tot = nfree + nvis;
                const int newT = T + (nbtot > nfree_tot ? nbtot - nfree_tot : 0);
                if (step && (nbtot > TMAX || nbtot < 3 || newT > TMAX || Vn + 1 > VMAX)) {
                    failed = true;
                    live = false;
                    step = false;
                }
                wave_sync();
                if (step)
                    for (int k = gl; k < nbtot; k += GL) {
                        const int slot = k < nfree_tot ? L.freel[nfree_tot - 1 - k] : T + (k - nfree_tot);
                        const uint32_t e = L.be[k];
                        const int a = (int)(e & 255u), b = (int)((e >> 8) & 255u), u = (int)((e >> 16) & 63u),
                                  j = (int)((e >> 22) & 3u);
                        L.be[k] = (e & 0x3fffffu) | ((uint32_t)slot << 24);
                        L.tv[slot] = tpack(a, b, Vn, GF_ALIVE);
                        reinterpret_cast<uint8_t *>(&L.to[u])[j] = (uint8_t)slot;
                        L.vstart[a] = (uint8_t)slot;
                        L.vend[b] = (uint8_t)slot;
                    }
                wave_sync();
                if (step) {
                    for (int k = gl; k < nbtot; k += GL) {
                        const uint32_t e = L.be[k];
                        L.to[e >> 24] = (uint32_t)L.vstart[(e >> 8) & 255u] | ((uint32_t)L.vend[e & 255u] << 8) |
                                        (e & 0x3f0000u);
                    }
                    nfree = nfree_tot - (nbtot < nfree_tot ? nbtot : nfree_tot);
                    T = newT;
                }
                // the link writes above touch only the new slots' neighbour rows: the cofactor
                // pass below (triangle words and coordinates) needs no barrier after them.  The new
                // triangles are those alive whose third vertex, here this lane's own r, is Vn.
#pragma unroll
                for (int k = 0; k < KPL; k++) tk[k] = L.tv[gl + GL * k];
                const uint32_t fresh = step ? (uint32_t)Vn | (GF_ALIVE >> 18) : ~0u;
#pragma unroll
                for (int k = 0; k < KPL; k++) {
                    const uint32_t t = tk[k];
                    if ((t >> 18) == fresh) {
                        grp_cofactors(L.vc[tvert(t, 0)], L.vc[tvert(t, 1)], r, w.a, w.rs, C[k], P[k]);
                        if (COUNT) ncof++;
                    }
                }
                // No barrier before the next step: its filter reads and writes only this lane's
                // own slots and the listed coordinates, and its first barrier precedes any read
                // of another lane's words.
            }
            wave_sync();
            // ---- outcome per group ----
            if (act && unsure && gl == 0) {
                const unsigned long long k = atomicAdd(&cnt[p.exact_counter], 1ull);
                if ((int64_t)k < p.exact_cap) p.exact_list[k] = s;
                else atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_BUFFER);
            }
            if (act && failed && gl == 0) {
                atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_HOLE);
                p.vnum[s] = 0;
                p.tnum[s] = 0;
            }
            bool fin = act && !unsure && !failed;
            // ---- finalize: link set, drowned insertions, compaction, pairs, history ----
            const int V = need; // drowned insertions' slots are never referenced and drop out
            if (fin)
                for (int v = gl; v < V; v += GL) L.present[v] = 0;
            // this lane's live triangle words (0 for dead and unused slots), read together
            uint32_t tf[KPL];
#pragma unroll
            for (int k = 0; k < KPL; k++) {
                const uint32_t t = L.tv[gl + GL * k];
                tf[k] = fin && (int)t < 0 ? t : 0u;
            }
            wave_sync();
#pragma unroll
            for (int k = 0; k < KPL; k++)
                if (tf[k]) {
                    L.present[tvert(tf[k], 0)] = 1;
                    L.present[tvert(tf[k], 1)] = 1;
                    L.present[tvert(tf[k], 2)] = 1;
                }
            wave_sync();
#pragma unroll
            for (int b0 = 0; b0 < VMAX; b0 += GL) {
                const int q = b0 + gl;
                bool dr = false;
                if (fin && q < m) {
                    dr = !L.present[vn + q]; // a vertex that never entered is in no triangle
                    p.dflag[ib + q] = dr ? 1 : 0;
                }
                ndrown += __popcll(__ballot(dr));
            }
            const int64_t vo = fin ? p.nvoff[s] : 0, to = fin ? p.ntoff[s] : 0;
            // ranks of the link's vertices and of the live triangles, scanned together
            constexpr int VPL = VMAX / GL;
            int fl[VPL + KPL], rk[VPL + KPL], ct[VPL + KPL];
#pragma unroll
            for (int i = 0; i < VPL; i++) fl[i] = fin && gl + GL * i < V && L.present[gl + GL * i] ? 1 : 0;
#pragma unroll
            for (int k = 0; k < KPL; k++) fl[VPL + k] = tf[k] ? 1 : 0;
            grp_excl_n<GL, 1, VPL + KPL>(fl, g, gl, rk, ct);
            int vcount = 0, tcount = 0;
#pragma unroll
            for (int i = 0; i < VPL; i++) {
                const int v = gl + GL * i;
                if (fl[i]) {
                    L.vremap[v] = (uint8_t)(vcount + rk[i]);
                    p.vpool[vo + vcount + rk[i]] = L.vid[v];
                }
                vcount += ct[i];
            }
#pragma unroll
            for (int k = 0; k < KPL; k++) {
                rk[VPL + k] += tcount;
                if (tf[k]) L.remap[gl + GL * k] = (uint8_t)rk[VPL + k];
                tcount += ct[VPL + k];
            }
            if (fin && (tcount > 2 * need - 4 || tcount != 2 * vcount - 4)) {
                // not a triangulated 2-sphere: report instead of writing past the star's region
                if (gl == 0) {
                    atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_HOLE);
                    p.vnum[s] = 0;
                    p.tnum[s] = 0;
                }
                fin = false;
            }
            wave_sync();
            const int64_t pb = 2 * (to - p.tbase);
            // every slot's output word and pairs first (their reads overlap), then the pair scans
            TriPairs prk[KPL];
#pragma unroll
            for (int k = 0; k < KPL; k++) {
                const int t = gl + GL * k;
                const uint32_t tt = fin ? tf[k] : 0u;
                prk[k] = TriPairs{STAR_PAIR_NONE, STAR_PAIR_NONE};
                if (tt) {
                    const int a = tvert(tt, 0), b = tvert(tt, 1), c = tvert(tt, 2);
                    const uint32_t o = L.to[t];
                    p.tpool[to + rk[VPL + k]] = hpack(L.vremap[a], L.vremap[b], L.vremap[c], L.remap[o & 255u],
                                                      L.remap[(o >> 8) & 255u], L.remap[(o >> 16) & 255u], true);
                    prk[k] = star_tri_pairs(L.vid[a], L.vid[b], L.vid[c], !(tt & TF_CHECKED));
                }
            }
            // the star's pairs, dense, in triangle order
            int np[KPL], pat[KPL], ptot[KPL], npair = 0;
#pragma unroll
            for (int k = 0; k < KPL; k++)
                np[k] = (prk[k].x != STAR_PAIR_NONE ? 1 : 0) + (prk[k].y != STAR_PAIR_NONE ? 1 : 0);
            grp_excl_n<GL, 2, KPL>(np, g, gl, pat, ptot);
#pragma unroll
            for (int k = 0; k < KPL; k++) {
                const int64_t at = pb + npair + pat[k];
                if (np[k] > 0) p.pairbuf[at] = prk[k].x;
                if (np[k] > 1) p.pairbuf[at + 1] = prk[k].y;
                npair += ptot[k];
            }
            // groups not finalised count none
#pragma unroll
            for (int j = 0; j < NG; j++) npairs += __builtin_amdgcn_readlane(npair, j * GL);
            int hn = 0;
            if (fin) {
                if (gl == 0) p.pcount[s] = npair;
                hn = star_history_merge(p, s, L.vid + vn, m, gl, GL);
            }
            wave_sync();
            if (fin && gl == 0) star_commit(p, s, vcount, vo, tcount, to, hn + m);
            wave_sync();
        }
    }
    if (COUNT) {
        const int wf = g4d_wave_sum(nfilt), wc = g4d_wave_sum(ncof);
        if (lane == 0) {
            atomicAdd(&cnt[G4D_CNT_ORIENT4], (unsigned long long)wf);
            atomicAdd(&cnt[G4D_CNT_COFACTOR], (unsigned long long)wc);
        }
    }
    if (lane == 0) {
        if (npairs) atomicAdd(&cnt[G4D_CNT_PAIRS], npairs);
        if (ndrown) atomicAdd(&cnt[G4D_CNT_DROWNED], ndrown);
    }
}

__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3, 8))) k_star32g16(StarParams p, int nitems)
{
    star_body_grp<16, false>(p, nitems, blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3, 8))) k_star32g16f(StarParams p, int nitems)
{
    star_body_grp<16, true>(p, nitems, blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) k_star32g16f4(StarParams p, int nitems)
{
    star_body_grp<16, true>(p, nitems, blockIdx.x, gridDim.x);
}

__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) k_star32g32f(StarParams p, int nitems)
{
    star_body_grp<32, true>(p, nitems, blockIdx.x, gridDim.x);
}

// A late pass's two tiers (32 and, merged, 64 to 256 vertices) in one launch: work-groups below nb take
// batches of p's list, the others stars of q's.  Both finish when their longest star does (some
// 35 us each), which this pays once.  The larger tier's 256 registers and both LDS blocks (33.9 KB)
// leave one wave per SIMD, 1,024 work-groups on the chip; such a pass has some four keys a star, so
// 6,144 keys come to some 1,300 stars, 330 batches beside a few hundred larger stars.  One launch
// against two: 1,000 uniform points (five late passes) 1.20 and 1.34 ms a call, 7,000 1.77 and 1.81,
// 100,000 4.72 and 4.89, 300,000 6.36 and 6.54.
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2, 8))) k_star_late(StarParams p, int nb,
                                                                                            StarParams q)
{
    if ((int)blockIdx.x < nb) star_body_grp<16, true, false>(p, p.nlist, blockIdx.x, nb);
    else star_body<STAR_VMAX_T2, false>(q, q.nlist, blockIdx.x - nb, gridDim.x - nb);
}

// The 32-vertex filter-only kernel variant of a launch: the caller's choice, else the
// G4D_STAR_T0 environment variable (measurement), else the measured best: four stars per wave with
// the FP32 bound at four waves per SIMD, 15.3 ms of star kernel at 4,194,304 uniform points (G = 512)
// against 18.1 at three (18.4 with the FP64 permanents), 22.6 for two stars per wave and 46.8 for one.
static int star_t0_variant(int requested)
{
    if (requested >= 0 && requested < STAR_T0_NUM) return requested;
    static int env = -2;
    if (env == -2) {
        const char *e = getenv("G4D_STAR_T0");
        env = e ? atoi(e) : -1;
        if (env < 0 || env >= STAR_T0_NUM) env = -1;
    }
    return env >= 0 ? env : STAR_T0_G16F4;
}

static_assert(G4D_CNT_QUEUE0 + 7 <= G4D_CNT_PAIRS, "seven queue heads must fit the counter block");
static_assert(G4D_CNT_NUM < 64, "counter masks are 64 bits wide");

__global__ void k_zero_counters(unsigned long long *cnt, uint64_t mask)
{
    const int i = threadIdx.x;
    if (i < G4D_CNT_NUM && ((mask >> i) & 1u)) cnt[i] = 0ull;
}

hipError_t launch_zero_counters(unsigned long long *cnt, uint64_t mask, hipStream_t s)
{
    if ((mask >> G4D_CNT_NUM) != 0u) return hipErrorInvalidValue; // beyond the block
    hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, s, cnt, mask);
    return hipGetLastError();
}

hipError_t launch_star_late(const StarParams &p, const StarParams &q, hipStream_t s)
{
    if (!p.star_list || p.nlist <= 0 || !q.star_list || q.nlist <= 0 || p.nlist_dev || q.nlist_dev ||
        p.lds_limit > STAR_LDS_LIMIT)
        return hipErrorInvalidValue;
    const int nb = std::min(4096, (p.nlist + 3) / 4);
    hipLaunchKernelGGL(k_star_late, dim3(nb + std::min(1536, q.nlist)), dim3(64), 0, s, p, nb, q);
    return hipGetLastError();
}

bool star_late_variant(int requested) { return star_t0_variant(requested) == STAR_T0_G16F4; }

hipError_t launch_star_kernel(const StarParams &p, int vmax, bool exact, int nblocks, hipStream_t s)
{
    const int nitems = p.nlist;
    if (nitems <= 0) return hipSuccess;
    if (!p.star_list || (exact ? !p.defer_list : p.nlist_dev != nullptr)) return hipErrorInvalidValue;
    if (p.lds_limit > STAR_LDS_LIMIT) return hipErrorInvalidValue; // local ids must fit 9 bits
    if (nblocks > nitems) nblocks = nitems;
    if (exact) {
        if (vmax == STAR_VMAX_T0)
            hipLaunchKernelGGL(HIP_KERNEL_NAME(k_star_exact<STAR_VMAX_T0>), dim3(nblocks), dim3(64), 0, s, p, nitems);
        else if (vmax == STAR_VMAX_T1)
            hipLaunchKernelGGL(HIP_KERNEL_NAME(k_star_exact<STAR_VMAX_T1>), dim3(nblocks), dim3(64), 0, s, p, nitems);
        else if (vmax == STAR_VMAX_T2)
            hipLaunchKernelGGL(HIP_KERNEL_NAME(k_star_exact<STAR_VMAX_T2>), dim3(nblocks), dim3(64), 0, s, p, nitems);
        else
            return hipErrorInvalidValue;
    } else if (vmax == STAR_VMAX_T0) {
        const int v = star_t0_variant(p.t0_variant);
        if (v == STAR_T0_WAVE) {
            hipLaunchKernelGGL(k_star32, dim3(nblocks), dim3(64), 0, s, p, nitems);
        } else {
            // one work-group per resident wave (256 CUs x 4 SIMDs x the variant's occupancy), or
            // one per batch of stars when the list is shorter
            const int per_simd = v <= STAR_T0_G16F ? 3 : 4;
            const int ng = v == STAR_T0_G32F ? 2 : 4;
            const int nb = std::max(1, std::min(1024 * per_simd, (nitems + ng - 1) / ng));
            if (v == STAR_T0_G16) hipLaunchKernelGGL(k_star32g16, dim3(nb), dim3(64), 0, s, p, nitems);
            else if (v == STAR_T0_G16F) hipLaunchKernelGGL(k_star32g16f, dim3(nb), dim3(64), 0, s, p, nitems);
            else if (v == STAR_T0_G16F4) hipLaunchKernelGGL(k_star32g16f4, dim3(nb), dim3(64), 0, s, p, nitems);
            else hipLaunchKernelGGL(k_star32g32f, dim3(nb), dim3(64), 0, s, p, nitems);
        }
    } else if (vmax == STAR_VMAX_T1) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_star<STAR_VMAX_T1, 4>), dim3(nblocks), dim3(64), 0, s, p, nitems);
    } else if (vmax == STAR_VMAX_TM) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_star<STAR_VMAX_TM, 3>), dim3(nblocks), dim3(64), 0, s, p, nitems);
    } else if (vmax == STAR_VMAX_T2) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_star<STAR_VMAX_T2, 2>), dim3(nblocks), dim3(64), 0, s, p, nitems);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------
// Wide star kernel: stars of up to VMAX link vertices plus insertions in LDS, one work-group of NT
// threads per star, filters only.  A thread owns the slots tid, tid + NT, ... and keeps their
// cofactors in registers as the one-wave kernels do; the step is theirs too, with work-group
// barriers (five a step, one per scan and one before each pass that reads what others wrote).
// Slots are counted in the order of the global-memory kernel below, as if 512 threads owned them, so
// a star leaves either kernel with the same triangles in the same order.
//
// That kernel keeps these arrays in HBM, 64 bytes of cofactors a slot among them, and reads them
// through L2 once per insertion; it now takes the stars beyond 1,024 and those whose filters are
// inconclusive.  On 1,000,000 clustered points (11,766 stars of 257-2,283 over six passes) it took
// 35.4 ms; 512 vertices take 4.7 ms here, 1,024 6.8 ms, and the few larger ones 6.9 ms there, each a
// chain of its insertions.  (512 vertices with 256 threads at 2 waves per SIMD 5.6 ms, with 512
// threads 5.8 ms.)
// ------------------------------------------------------------------------------------

static constexpr int STAR_ORDER = 512; // threads whose slot order both kernels follow

template <int VMAX, int NT>
struct StarWideLds {
    static constexpr int TMAX = 2 * VMAX;
    double vc[VMAX][4];
    union {
        uint16_t tv[TMAX][4]; // local vertices 0-2, flags (TW_*)
        uint64_t tv64[TMAX];
    };
    union {
        uint16_t to[TMAX][4]; // neighbours across the edges opposite vertices 0-2 (fourth unused)
        uint64_t to64[TMAX];
    };
    int vid[VMAX], ins[VMAX];
    uint16_t vstart[VMAX], vend[VMAX], freel[TMAX];
    union {
        struct {
            uint16_t a[TMAX], b[TMAX], u[TMAX], slot[TMAX];
            uint8_t j[TMAX];
        } be; // hole boundary
        struct {
            uint16_t remap[TMAX], vremap[VMAX];
            uint8_t present[VMAX];
        } fin; // finalisation
    };
    int16_t ins_local[VMAX];
    int red[4][NT / 64]; // rows 0 and 1: the filters' counts by turns; 2 and 3: the other scans
    int item;
};

static constexpr uint32_t TW_ALIVE = 1u, TW_CHECKED = 2u, TW_VIS = 4u, TW_FRESH = 8u;

__device__ __forceinline__ uint64_t wtri(int a, int b, int c, uint32_t fl)
{
    return (uint64_t)(uint32_t)a | ((uint64_t)(uint32_t)b << 16) | ((uint64_t)(uint32_t)c << 32) | ((uint64_t)fl << 48);
}
__device__ __forceinline__ int wtv(uint64_t t, int i) { return (int)((t >> (16 * i)) & 0xffffu); }
__device__ __forceinline__ uint32_t wfl(uint64_t t) { return (uint32_t)(t >> 48); }

// Exclusive prefix over the work-group of packed counts and their total; `add` joins the wave's
// total (wave-uniform).  One barrier, so no row of red may serve two calls without a barrier between
// the first call's reads and the second's write: consecutive calls use different rows.
template <int NT>
__device__ __forceinline__ int wide_excl(int v, int add, int *red, int *tot)
{
    const int lane = __lane_id(), w = threadIdx.x >> 6;
    const int inc = g4d_wave_incl_sum(v);
    if (lane == 63) red[w] = inc + add;
    __syncthreads();
    int base = 0, all = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; i++) {
        const int x = red[i];
        if (i < w) base += x;
        all += x;
    }
    *tot = all;
    return base + inc - v;
}

template <int VMAX, int NT, int WPE>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(WPE, 8))) k_star_wide(StarParams p, int nitems)
{
    using Lds = StarWideLds<VMAX, NT>;
    constexpr int TMAX = Lds::TMAX, KPL = TMAX / NT, H = STAR_ORDER / NT;
    static_assert(H * NT == STAR_ORDER && TMAX < 4096, "packed counts of 12 bits");
    __shared__ Lds L;
    const int tid = threadIdx.x;
    unsigned long long *cnt = p.cnt;
    double rc[KPL][4], rp[KPL][2];
    unsigned long long npairs = 0, ndrown = 0; // of the work-group, and of the wave
    for (;;) {
        __syncthreads(); // the previous star is done with L
        if (tid == 0) L.item = (int)atomicAdd(&cnt[p.work_counter], 1ull);
        __syncthreads();
        if (L.item >= nitems) break;
        const int s = p.star_list[L.item];
        const int64_t ib = p.ins_off[s];
        const int m = (int)(p.ins_off[s + 1] - ib);
        const int vn = p.mode ? p.vnum[s] : 0;
        const int need = vn + m;
        if (need > VMAX || (p.mode == 0 && m < 4)) {
            if (tid == 0) {
                atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)(need > VMAX ? G4D_DEV_ERR_BUFFER : G4D_DEV_ERR_CONE));
                p.vnum[s] = 0;
                p.tnum[s] = 0;
            }
            continue;
        }
        if (p.mode == 1 && m == 0) continue; // untouched star: stays where it is
        const bool in_wide = vn >= STAR_WIDE_MIN;
        const double sx = p.pts[3 * (int64_t)s], sy = p.pts[3 * (int64_t)s + 1], sz = p.pts[3 * (int64_t)s + 2];
        const int q0 = p.mode ? 0 : 4;
        for (int q = tid; q < m; q += NT) {
            const int g = (int)(uint32_t)p.ins_keys[ib + q];
            L.ins[q] = g;
            L.ins_local[q] = -1;
            if (q >= q0) {
                L.vid[vn + q] = g;
                rel_coords(p.pts, g, sx, sy, sz, L.vc[vn + q]);
            }
        }
        int T, nfree = 0;
        bool unsure = false, failed = false;
        if (p.mode == 1) {
            const int tn = p.tnum[s];
            const int64_t vi = p.voff[s], ti = p.toff[s];
            for (int v = tid; v < vn; v += NT) {
                const int g = p.vpool[vi + v];
                L.vid[v] = g;
                rel_coords(p.pts, g, sx, sy, sz, L.vc[v]);
            }
            for (int t = tid; t < tn; t += NT) {
                if (in_wide) {
                    const uint64_t w0 = p.tpool[ti + 2 * (int64_t)t], w1 = p.tpool[ti + 2 * (int64_t)t + 1];
                    L.tv64[t] = wtri(wfield(w0, 0), wfield(w0, 1), wfield(w0, 2), TW_ALIVE | ((w0 >> 63) ? TW_CHECKED : 0u));
                    L.to64[t] = wtri(wfield(w1, 0), wfield(w1, 1), wfield(w1, 2), 0u);
                } else {
                    const uint64_t h = p.tpool[ti + t];
                    L.tv64[t] = wtri(hvert(h, 0), hvert(h, 1), hvert(h, 2), TW_ALIVE | (hchecked(h) ? TW_CHECKED : 0u));
                    L.to64[t] = wtri(hopp(h, 0), hopp(h, 1), hopp(h, 2), 0u);
                }
            }
            T = tn;
        } else {
            // initial 4-simplex (GD/GDelaunay/GDelPredKernels.cu:45-158)
            int l[4];
            for (int i = 0; i < 4; i++) l[i] = (int)(uint32_t)p.ins_keys[ib + i];
            const double *pp[5] = {p.pts + 3 * (int64_t)l[0], p.pts + 3 * (int64_t)l[1], p.pts + 3 * (int64_t)l[2],
                                   p.pts + 3 * (int64_t)l[3], p.pts + 3 * (int64_t)s};
            const int o = filter_insphere(pp);
            unsure = o == 0;
            const bool sw = o < 0;
            if (tid < 4) {
                const int from = (tid < 2 && sw) ? 1 - tid : tid;
                L.vid[tid] = l[from];
                rel_coords(p.pts, l[from], sx, sy, sz, L.vc[tid]);
                const int lt[4][3] = {{1, 2, 3}, {0, 3, 2}, {0, 1, 3}, {0, 2, 1}};
                L.tv64[tid] = wtri(lt[tid][0], lt[tid][1], lt[tid][2], TW_ALIVE);
                L.to64[tid] = wtri(lt[tid][0], lt[tid][1], lt[tid][2], 0u);
                L.ins_local[tid] = (int16_t)from;
            }
            T = 4;
        }
        __syncthreads();
        // the cofactors of this thread's slots k of the mask, by rounds (as in star_body)
        auto cofactors = [&](unsigned km) {
            while (__ballot(km != 0)) {
                const int k = km ? __builtin_ctz(km) : KPL;
                double C[4], P[4];
                if (km) {
                    const uint64_t t = L.tv64[tid + NT * k];
                    tri_cofactors(L.vc[wtv(t, 0)], L.vc[wtv(t, 1)], L.vc[wtv(t, 2)], C, P);
                    L.tv[tid + NT * k][3] = (uint16_t)(wfl(t) & ~TW_FRESH);
                }
#pragma unroll
                for (int i = 0; i < KPL; i++)
                    if (i == k) {
#pragma unroll
                        for (int j = 0; j < 4; j++) rc[i][j] = C[j];
                        rp[i][0] = fmax(P[0], fmax(P[1], P[2]));
                        rp[i][1] = P[3];
                    }
                km &= km - 1;
            }
        };
        cofactors(T > tid ? (1u << ((T - tid + NT - 1) / NT)) - 1u : 0u);
        for (int q = q0; q < m && !unsure; q++) {
            const int Vn = vn + q;
            const double r[4] = {L.vc[Vn][0], L.vc[Vn][1], L.vc[Vn][2], L.vc[Vn][3]};
            const double rsum = fabs(r[0]) + fabs(r[1]) + fabs(r[2]);
            unsigned vm = 0;
            bool unc = false;
            int nv = 0; // per half of the slot order, 12 bits each
#pragma unroll
            for (int k = 0; k < KPL; k++) {
                const int slot = tid + NT * k;
                if (slot < T) {
                    const uint32_t f = L.tv[slot][3];
                    if ((f & (TW_ALIVE | TW_VIS)) == TW_ALIVE) {
                        const int sg = cofactor_filter_sign2(r, rsum, rc[k], rp[k][0], rp[k][1]);
                        unc = unc || sg == 0;
                        if (sg < 0) {
                            L.tv[slot][3] = (uint16_t)(f | TW_VIS);
                            vm |= 1u << k;
                            nv += (k % H) ? 1 << 12 : 1;
                        }
                    }
                }
            }
            int all;
            const int pre = wide_excl<NT>(nv, __ballot(unc) ? 1 << 24 : 0, L.red[q & 1], &all);
            if (all >> 24) {
                unsure = true;
                break;
            }
            const int nvis = (all & 0xfff) + ((all >> 12) & 0xfff);
            if (nvis == 0) continue; // drowned at insertion
            if (tid == 0) L.ins_local[q] = (int16_t)Vn;
            {
                // only the part of `pre` below bit 24 counts; the flag bits of earlier waves are zero here
                int f0 = nfree + (pre & 0xfff), f1 = nfree + (all & 0xfff) + ((pre >> 12) & 0xfff);
#pragma unroll
                for (int k = 0; k < KPL; k++)
                    if ((vm >> k) & 1) L.freel[(k % H) ? f1++ : f0++] = (uint16_t)(tid + NT * k);
            }
            __syncthreads();
            // hole boundary in the order of the visible list (see star_body)
            int nbtot = 0;
            for (int x0 = 0, row = 2; x0 < nvis; x0 += NT, row ^= 1) {
                const int x = x0 + tid;
                uint64_t t = 0ull, o = 0ull, tu[3];
                bool edge[3] = {false, false, false};
                if (x < nvis) {
                    const int slot = L.freel[nfree + x];
                    t = L.tv64[slot];
                    o = L.to64[slot];
#pragma unroll
                    for (int i = 0; i < 3; i++) {
                        tu[i] = L.tv64[wtv(o, i)];
                        edge[i] = !(wfl(tu[i]) & TW_VIS);
                    }
                }
                int tot;
                int e = nbtot + wide_excl<NT>((int)edge[0] + (int)edge[1] + (int)edge[2], 0, L.red[row], &tot);
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    if (!edge[i]) continue;
                    const int a = wtv(t, (i + 1) % 3), b = wtv(t, (i + 2) % 3);
                    const int u0 = wtv(tu[i], 0), u1 = wtv(tu[i], 1);
                    if (e < TMAX) {
                        L.be.a[e] = (uint16_t)a;
                        L.be.b[e] = (uint16_t)b;
                        L.be.u[e] = (uint16_t)wtv(o, i);
                        L.be.j[e] = (uint8_t)((u0 != a && u0 != b) ? 0 : ((u1 != a && u1 != b) ? 1 : 2));
                    }
                    e++;
                }
                nbtot += tot;
            }
            const int nfree_tot = nfree + nvis;
            const int newT = T + (nbtot > nfree_tot ? nbtot - nfree_tot : 0);
            if (nbtot > TMAX || nbtot < 3 || newT > TMAX || Vn + 1 > VMAX) {
                failed = true;
                break;
            }
            __syncthreads();
            for (int k = tid; k < nbtot; k += NT) {
                const int slot = k < nfree_tot ? L.freel[nfree_tot - 1 - k] : T + (k - nfree_tot);
                const int a = L.be.a[k], b = L.be.b[k], u = L.be.u[k];
                L.be.slot[k] = (uint16_t)slot;
                L.tv64[slot] = wtri(a, b, Vn, TW_ALIVE | TW_FRESH);
                L.to[slot][2] = (uint16_t)u;
                L.to[u][L.be.j[k]] = (uint16_t)slot;
                L.vstart[a] = (uint16_t)slot;
                L.vend[b] = (uint16_t)slot;
            }
            __syncthreads();
            for (int k = tid; k < nbtot; k += NT) {
                const int slot = L.be.slot[k];
                L.to[slot][0] = L.vstart[L.be.b[k]];
                L.to[slot][1] = L.vend[L.be.a[k]];
            }
            nfree = nfree_tot - (nbtot < nfree_tot ? nbtot : nfree_tot);
            T = newT;
            unsigned fm = 0;
#pragma unroll
            for (int k = 0; k < KPL; k++)
                if (tid + NT * k < T && (L.tv[tid + NT * k][3] & TW_FRESH)) fm |= 1u << k;
            cofactors(fm);
            // No barrier before the next step, as in star_body: its filter touches this thread's own
            // slots and the listed coordinates, and its scan's barrier comes before the rest.
        }
        __syncthreads();
        if (unsure) {
            if (tid < 64) star_list_push(p.exact_list, p.exact_cap, &cnt[p.exact_counter], s, cnt);
            continue;
        }
        // ---- finalize: link set, drowned insertions, compaction, pairs, history ----
        for (int v = tid; v < need; v += NT) L.fin.present[v] = 0;
        __syncthreads();
        if (!failed)
            for (int t = tid; t < T; t += NT) {
                const uint64_t w = L.tv64[t];
                if ((wfl(w) & (TW_ALIVE | TW_VIS)) == TW_ALIVE)
                    for (int i = 0; i < 3; i++) L.fin.present[wtv(w, i)] = 1;
            }
        __syncthreads();
        const int64_t vo = p.nvoff[s], to = p.ntoff[s];
        int vcount = 0, tcount = 0, row = 2;
        if (!failed) {
            for (int b0 = 0; b0 < m; b0 += NT) {
                const int q = b0 + tid, lv = q < m ? L.ins_local[q] : 0;
                const bool dr = q < m && (lv < 0 || !L.fin.present[lv]);
                if (q < m) p.dflag[ib + q] = dr ? 1 : 0;
                ndrown += __popcll(__ballot(dr));
            }
            for (int base = 0; base < need; base += NT, row ^= 1) {
                const int v = base + tid;
                const bool pr = v < need && L.fin.present[v];
                int tot;
                const int at = vcount + wide_excl<NT>(pr ? 1 : 0, 0, L.red[row], &tot);
                if (pr) {
                    L.fin.vremap[v] = (uint16_t)at;
                    p.vpool[vo + at] = L.vid[v];
                }
                vcount += tot;
            }
            for (int base = 0; base < T; base += NT, row ^= 1) {
                const int t = base + tid;
                const bool al = t < T && (L.tv[t][3] & (TW_ALIVE | TW_VIS)) == TW_ALIVE;
                int tot;
                const int at = tcount + wide_excl<NT>(al ? 1 : 0, 0, L.red[row], &tot);
                if (al) L.fin.remap[t] = (uint16_t)at;
                tcount += tot;
            }
        }
        const bool wide = vcount >= STAR_WIDE_MIN;
        const int64_t words = wide ? 2 * (int64_t)tcount : tcount;
        if (failed || words > star_tcap_words(need) || tcount != 2 * vcount - 4) {
            // not a triangulated 2-sphere: report instead of writing past the star's region
            if (tid == 0) {
                atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_HOLE);
                p.vnum[s] = 0;
                p.tnum[s] = 0;
            }
            continue;
        }
        __syncthreads();
        const int64_t pb = 2 * (to - p.tbase);
        int npair = 0;
        for (int base = 0; base < T; base += NT, row ^= 1) {
            const int t = base + tid;
            const uint64_t w = t < T ? L.tv64[t] : 0ull;
            TriPairs pr{STAR_PAIR_NONE, STAR_PAIR_NONE};
            if ((wfl(w) & (TW_ALIVE | TW_VIS)) == TW_ALIVE) {
                const int a = wtv(w, 0), b = wtv(w, 1), cc = wtv(w, 2);
                const int ra = L.fin.vremap[a], rb = L.fin.vremap[b], rcc = L.fin.vremap[cc];
                const int o0 = L.fin.remap[L.to[t][0]], o1 = L.fin.remap[L.to[t][1]], o2 = L.fin.remap[L.to[t][2]];
                const int64_t d = L.fin.remap[t];
                if (wide) {
                    p.tpool[to + 2 * d] = wpack3(ra, rb, rcc) | (1ull << 63);
                    p.tpool[to + 2 * d + 1] = wpack3(o0, o1, o2);
                } else {
                    p.tpool[to + d] = hpack(ra, rb, rcc, o0, o1, o2, true);
                }
                pr = star_tri_pairs(L.vid[a], L.vid[b], L.vid[cc], !(wfl(w) & TW_CHECKED));
            }
            // the star's pairs, dense, in triangle order
            const int np = (pr.x != STAR_PAIR_NONE ? 1 : 0) + (pr.y != STAR_PAIR_NONE ? 1 : 0);
            int tot;
            const int64_t at = npair + wide_excl<NT>(np, 0, L.red[row], &tot);
            if (np > 0) p.pairbuf[pb + at] = pr.x;
            if (np > 1) p.pairbuf[pb + at + 1] = pr.y;
            npair += tot;
        }
        if (tid == 0) p.pcount[s] = npair;
        npairs += npair;
        const int hn = star_history_merge(p, s, L.ins, m, tid, NT);
        __syncthreads(); // every read of the old record and regions before the switch
        if (tid == 0) star_commit(p, s, vcount, vo, tcount, to, hn + m);
    }
    if ((tid & 63) == 0) {
        if (tid == 0 && npairs) atomicAdd(&cnt[G4D_CNT_PAIRS], npairs);
        if (ndrown) atomicAdd(&cnt[G4D_CNT_DROWNED], ndrown);
    }
}

hipError_t launch_star_wide(const StarParams &p, int vmax, hipStream_t s)
{
    if (p.nlist <= 0) return hipSuccess;
    if (!p.star_list) return hipErrorInvalidValue;
    // at most one work-group per resident one: LDS takes 50 KB at 512 vertices, 100 KB at 1,024
    if (vmax == STAR_VMAX_W1)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_star_wide<STAR_VMAX_W1, 256, 3>), dim3(std::min(p.nlist, 768)), dim3(256), 0, s,
                           p, p.nlist);
    else if (vmax == STAR_VMAX_W2)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_star_wide<STAR_VMAX_W2, 512, 2>), dim3(std::min(p.nlist, 256)), dim3(512), 0, s,
                           p, p.nlist);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------
// Global-memory star kernel: the same insertion / finalisation as k_star for stars whose link exceeds
// the LDS kernels' capacity, and with exact predicates for the wide ones' inconclusive stars.  A
// work-group of 512 threads per star; the star's working arrays (32-bit local indices, cached
// cofactors per triangle slot) live in a per-block HBM workspace sized for the largest such star of
// the pass.
// ------------------------------------------------------------------------------------

static constexpr int GSTAR_NT = STAR_ORDER; // threads per star in the global-memory kernel

// Exclusive prefix sum of v over the work-group's threads in thread order; total in *tot.
// red: GSTAR_NT / 64 ints of LDS.  Every thread of the work-group must call it.
__device__ __forceinline__ int block_excl(int v, int *tot, int *red)
{
    const int lane = __lane_id(), w = threadIdx.x >> 6;
    const int inc = g4d_wave_incl_sum(v);
    if (lane == 63) red[w] = inc;
    __syncthreads();
    int base = 0, all = 0;
    for (int i = 0; i < GSTAR_NT / 64; i++) {
        const int x = red[i];
        if (i < w) base += x;
        all += x;
    }
    __syncthreads();
    *tot = all;
    return base + inc - v;
}

struct GWork {
    int *vid, *vstart, *vend, *ins, *ins_local, *vremap;
    double *vc;   // 4 per vertex
    int *tva;     // 3 local vertices per triangle slot
    uint32_t *tfl;
    int *to;      // 3 adjacency slots per triangle slot
    double *cof;  // 8 per triangle slot: cofactors, permanents
    int *freel, *be_a, *be_b, *be_u, *be_slot, *be_j, *remap;
    uint8_t *present;
};

__host__ __device__ inline int64_t gwork_layout(char *base, int vcap, GWork *w)
{
    const int64_t V = vcap, T = 2 * (int64_t)vcap;
    int64_t off = 0;
    auto take = [&](int64_t bytes) -> char * {
        char *r = base ? base + off : nullptr;
        off += (bytes + 255) & ~(int64_t)255;
        return r;
    };
    GWork t;
    t.vc = (double *)take(32 * V);
    t.cof = (double *)take(64 * T);
    t.vid = (int *)take(4 * V);
    t.vstart = (int *)take(4 * V);
    t.vend = (int *)take(4 * V);
    t.ins = (int *)take(4 * V);
    t.ins_local = (int *)take(4 * V);
    t.vremap = (int *)take(4 * V);
    t.tva = (int *)take(12 * T);
    t.tfl = (uint32_t *)take(4 * T);
    t.to = (int *)take(12 * T);
    t.freel = (int *)take(4 * T);
    t.be_a = (int *)take(4 * T);
    t.be_b = (int *)take(4 * T);
    t.be_u = (int *)take(4 * T);
    t.be_slot = (int *)take(4 * T);
    t.be_j = (int *)take(4 * T);
    t.remap = (int *)take(4 * T);
    t.present = (uint8_t *)take(V);
    if (w) *w = t;
    return off;
}

int64_t star_global_bytes(int vcap) { return gwork_layout(nullptr, vcap, nullptr); }

__global__ void __launch_bounds__(GSTAR_NT) k_star_global(StarParams p, const int *list, int nitems, char *ws,
                                                          int64_t ws_stride, int vcap)
{
    __shared__ int red[GSTAR_NT / 64];
    const int tid = threadIdx.x;
    unsigned long long *cnt = p.cnt;
    GWork L;
    gwork_layout(ws + (int64_t)blockIdx.x * ws_stride, vcap, &L);
    const int TMAX = 2 * vcap;

    for (int item = blockIdx.x; item < nitems; item += gridDim.x) {
        const int s = list[item];
        const int64_t ib = p.ins_off[s];
        const int m = (int)(p.ins_off[s + 1] - ib);
        const int vn = p.mode ? p.vnum[s] : 0;
        const bool in_wide = vn >= STAR_WIDE_MIN;
        if (vn + m > vcap || (p.mode == 0 && m < 4)) {
            if (tid == 0) {
                atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)(vn + m > vcap ? G4D_DEV_ERR_STAR_CAPACITY
                                                                                  : G4D_DEV_ERR_CONE));
                p.vnum[s] = 0;
                p.tnum[s] = 0;
            }
            continue;
        }
        if (p.mode == 1 && m == 0) continue; // untouched star: stays where it is
        const double sx = p.pts[3 * (int64_t)s], sy = p.pts[3 * (int64_t)s + 1], sz = p.pts[3 * (int64_t)s + 2];
        // insertion q takes link-vertex slot vn + q (mode 0: the first four form the simplex)
        const int q0 = p.mode ? 0 : 4;
        for (int q = tid; q < m; q += GSTAR_NT) {
            const int g = (int)(uint32_t)p.ins_keys[ib + q];
            L.ins[q] = g;
            L.ins_local[q] = -1;
            if (q >= q0) {
                L.vid[vn + q] = g;
                rel_coords(p.pts, g, sx, sy, sz, L.vc + 4 * (vn + q));
            }
        }
        int T, nfree = 0;
        if (p.mode == 1) {
            const int tn = p.tnum[s];
            const int64_t vi = p.voff[s], ti = p.toff[s];
            for (int v = tid; v < vn; v += GSTAR_NT) {
                const int g = p.vpool[vi + v];
                L.vid[v] = g;
                rel_coords(p.pts, g, sx, sy, sz, L.vc + 4 * v);
            }
            for (int t = tid; t < tn; t += GSTAR_NT) {
                int a[3], o[3];
                bool chk;
                if (in_wide) {
                    const uint64_t w0 = p.tpool[ti + 2 * (int64_t)t], w1 = p.tpool[ti + 2 * (int64_t)t + 1];
                    for (int i = 0; i < 3; i++) {
                        a[i] = wfield(w0, i);
                        o[i] = wfield(w1, i);
                    }
                    chk = (w0 >> 63) & 1u;
                } else {
                    const uint64_t h = p.tpool[ti + t];
                    for (int i = 0; i < 3; i++) {
                        a[i] = hvert(h, i);
                        o[i] = hopp(h, i);
                    }
                    chk = hchecked(h);
                }
                for (int i = 0; i < 3; i++) {
                    L.tva[3 * t + i] = a[i];
                    L.to[3 * t + i] = o[i];
                }
                L.tfl[t] = TF_ALIVE | (chk ? TF_CHECKED : 0u);
            }
            T = tn;
        } else {
            // initial 4-simplex (GD/GDelaunay/GDelPredKernels.cu:45-158)
            int l[4];
            for (int i = 0; i < 4; i++) l[i] = (int)(uint32_t)p.ins_keys[ib + i];
            const double *pp[5] = {p.pts + 3 * (int64_t)l[0], p.pts + 3 * (int64_t)l[1], p.pts + 3 * (int64_t)l[2],
                                   p.pts + 3 * (int64_t)l[3], p.pts + 3 * (int64_t)s};
            const int idx[5] = {l[0], l[1], l[2], l[3], s};
            const bool sw = orient4_full(pp, idx, cnt) < 0;
            if (sw) {
                const int t = l[0];
                l[0] = l[1];
                l[1] = t;
            }
            if (tid < 4) {
                L.vid[tid] = l[tid];
                rel_coords(p.pts, l[tid], sx, sy, sz, L.vc + 4 * tid);
                const int lt[4][3] = {{1, 2, 3}, {0, 3, 2}, {0, 1, 3}, {0, 2, 1}};
                for (int i = 0; i < 3; i++) {
                    L.tva[3 * tid + i] = lt[tid][i];
                    L.to[3 * tid + i] = lt[tid][i];
                }
                L.tfl[tid] = TF_ALIVE;
                L.ins_local[tid] = (tid < 2 && sw) ? 1 - tid : tid;
            }
            T = 4;
        }
        __syncthreads();
        for (int slot = tid; slot < T; slot += GSTAR_NT)
            tri_cofactors(L.vc + 4 * L.tva[3 * slot], L.vc + 4 * L.tva[3 * slot + 1], L.vc + 4 * L.tva[3 * slot + 2],
                          L.cof + 8 * slot, L.cof + 8 * slot + 4);
        bool failed = false;
        for (int q = q0; q < m; q++) {
            const int gv = L.ins[q];
            const int Vn = vn + q;
            const double r[4] = {L.vc[4 * Vn], L.vc[4 * Vn + 1], L.vc[4 * Vn + 2], L.vc[4 * Vn + 3]};
            int nv = 0, nunc = 0;
            for (int slot = tid; slot < T; slot += GSTAR_NT) {
                const uint32_t f = L.tfl[slot];
                if (!(f & TF_ALIVE)) continue;
                const int sg = cofactor_filter_sign(r, L.cof + 8 * slot, L.cof + 8 * slot + 4);
                if (sg == 0) {
                    L.tfl[slot] = f | TF_UNSURE;
                    nunc++;
                } else if (sg < 0) {
                    L.tfl[slot] = f | TF_VIS;
                    nv++;
                }
            }
            // Triangles the filter cannot decide are gathered into one list (be_slot is free until
            // the hole boundary) and decided exactly one per thread, so that the block's threads
            // share the exact work instead of each wave stalling on its own few slots.  Below 2^15
            // slots one scan serves both counts (each total is at most T), packed in 16-bit halves.
            int vbase, nvis, nunc_tot, ub;
            if (T < 32768) {
                int both;
                const int pre = block_excl(nv | (nunc << 16), &both, red);
                vbase = pre & 0xffff;
                nvis = both & 0xffff;
                ub = pre >> 16;
                nunc_tot = both >> 16;
            } else {
                ub = block_excl(nunc, &nunc_tot, red);
                vbase = block_excl(nv, &nvis, red);
            }
            // rare: the registers that the call takes are saved here and not around the loop
            if (__builtin_expect(nunc_tot > 0, 0)) {
                for (int slot = tid; slot < T && nunc > 0; slot += GSTAR_NT)
                    if (L.tfl[slot] & TF_UNSURE) {
                        L.be_slot[ub++] = slot;
                        nunc--;
                    }
                __syncthreads();
                for (int k = tid; k < nunc_tot; k += GSTAR_NT) {
                    const int slot = L.be_slot[k];
                    const int a = L.vid[L.tva[3 * slot]], b = L.vid[L.tva[3 * slot + 1]], c = L.vid[L.tva[3 * slot + 2]];
                    const double *pp[5] = {p.pts + 3 * (int64_t)a, p.pts + 3 * (int64_t)b, p.pts + 3 * (int64_t)c,
                                           p.pts + 3 * (int64_t)s, p.pts + 3 * (int64_t)gv};
                    const int idx[5] = {a, b, c, s, gv};
                    const int sg = orient4_full(pp, idx, cnt);
                    const uint32_t f = L.tfl[slot] & ~TF_UNSURE;
                    L.tfl[slot] = sg < 0 ? (f | TF_VIS) : f;
                }
                __syncthreads();
                // each thread counts the beneath triangles among its own slots again
                nv = 0;
                for (int slot = tid; slot < T; slot += GSTAR_NT) nv += (L.tfl[slot] & TF_VIS) ? 1 : 0;
                vbase = block_excl(nv, &nvis, red);
            }
            if (nvis == 0) continue; // drowned at insertion
            if (tid == 0) L.ins_local[q] = Vn;
            __syncthreads();
            // hole boundary: edges of freed triangles whose neighbour survives
            int nb = 0;
            for (int slot = tid; slot < T; slot += GSTAR_NT)
                if (L.tfl[slot] & TF_VIS)
                    for (int i = 0; i < 3; i++) nb += (L.tfl[L.to[3 * slot + i]] & TF_VIS) ? 0 : 1;
            int nbtot;
            int e = block_excl(nb, &nbtot, red);
            if (nbtot > TMAX || nbtot < 3) {
                failed = true;
                break;
            }
            int fpos = nfree + vbase;
            for (int slot = tid; slot < T; slot += GSTAR_NT) {
                if (!(L.tfl[slot] & TF_VIS)) continue;
                for (int i = 0; i < 3; i++) {
                    const int u = L.to[3 * slot + i];
                    if (L.tfl[u] & TF_VIS) continue;
                    int j = 0;
                    while (j < 2 && L.to[3 * u + j] != slot) j++;
                    L.be_a[e] = L.tva[3 * slot + (i + 1) % 3];
                    L.be_b[e] = L.tva[3 * slot + (i + 2) % 3];
                    L.be_u[e] = u;
                    L.be_j[e] = j;
                    e++;
                }
                L.freel[fpos++] = slot;
            }
            __syncthreads();
            const int nfree_tot = nfree + nvis;
            for (int slot = tid; slot < T; slot += GSTAR_NT)
                if (L.tfl[slot] & TF_VIS) L.tfl[slot] = 0u;
            for (int k = tid; k < nbtot; k += GSTAR_NT)
                L.be_slot[k] = k < nfree_tot ? L.freel[nfree_tot - 1 - k] : T + (k - nfree_tot);
            const int newT = T + (nbtot > nfree_tot ? nbtot - nfree_tot : 0);
            if (newT > TMAX || Vn + 1 > vcap) {
                failed = true;
                break;
            }
            __syncthreads();
            for (int k = tid; k < nbtot; k += GSTAR_NT) {
                const int slot = L.be_slot[k], a = L.be_a[k], b = L.be_b[k], u = L.be_u[k];
                L.tva[3 * slot] = a;
                L.tva[3 * slot + 1] = b;
                L.tva[3 * slot + 2] = Vn;
                L.tfl[slot] = TF_ALIVE | TF_FRESH;
                L.to[3 * slot + 2] = u;
                L.to[3 * u + L.be_j[k]] = slot;
                L.vstart[a] = slot;
                L.vend[b] = slot;
            }
            __syncthreads();
            for (int k = tid; k < nbtot; k += GSTAR_NT) {
                const int slot = L.be_slot[k];
                L.to[3 * slot] = L.vstart[L.be_b[k]];
                L.to[3 * slot + 1] = L.vend[L.be_a[k]];
            }
            nfree = nfree_tot - (nbtot < nfree_tot ? nbtot : nfree_tot);
            T = newT;
            __syncthreads();
            for (int slot = tid; slot < T; slot += GSTAR_NT) {
                const uint32_t f = L.tfl[slot];
                if (f & TF_FRESH) {
                    tri_cofactors(L.vc + 4 * L.tva[3 * slot], L.vc + 4 * L.tva[3 * slot + 1],
                                  L.vc + 4 * L.tva[3 * slot + 2], L.cof + 8 * slot, L.cof + 8 * slot + 4);
                    L.tfl[slot] = f & ~TF_FRESH;
                }
            }
            __syncthreads();
        }
        if (failed) {
            if (tid == 0) {
                atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_HOLE);
                p.vnum[s] = 0;
                p.tnum[s] = 0;
            }
            __syncthreads();
            continue;
        }
        // ---- finalize: link set, drowned insertions, compaction, pairs, history ----
        const int V = vn + m; // drowned insertions' slots are never referenced and drop out
        for (int v = tid; v < V; v += GSTAR_NT) L.present[v] = 0;
        __syncthreads();
        for (int slot = tid; slot < T; slot += GSTAR_NT)
            if (L.tfl[slot] & TF_ALIVE)
                for (int i = 0; i < 3; i++) L.present[L.tva[3 * slot + i]] = 1;
        __syncthreads();
        int ndrown = 0; // the wave's
        for (int b0 = 0; b0 < m; b0 += GSTAR_NT) {
            const int q = b0 + tid, lv = q < m ? L.ins_local[q] : 0;
            const bool dr = q < m && (lv < 0 || !L.present[lv]);
            if (q < m) p.dflag[ib + q] = dr ? 1 : 0;
            ndrown += __popcll(__ballot(dr));
        }
        if ((tid & 63) == 0 && ndrown) atomicAdd(&cnt[G4D_CNT_DROWNED], (unsigned long long)ndrown);
        const int64_t vo = p.nvoff[s], to = p.ntoff[s];
        int vcount = 0;
        for (int base = 0; base < V; base += GSTAR_NT) {
            const int v = base + tid;
            const bool pr = v < V && L.present[v];
            int tot;
            const int rk = block_excl(pr ? 1 : 0, &tot, red);
            if (pr) {
                L.vremap[v] = vcount + rk;
                p.vpool[vo + vcount + rk] = L.vid[v];
            }
            vcount += tot;
        }
        int tcount = 0;
        for (int base = 0; base < T; base += GSTAR_NT) {
            const int t = base + tid;
            const bool al = t < T && (L.tfl[t] & TF_ALIVE);
            int tot;
            const int rk = block_excl(al ? 1 : 0, &tot, red);
            if (al) L.remap[t] = tcount + rk;
            tcount += tot;
        }
        const bool wide = vcount >= STAR_WIDE_MIN;
        const int64_t words = wide ? 2 * (int64_t)tcount : tcount;
        if (words > star_tcap_words(vn + m) || tcount != 2 * vcount - 4) {
            if (tid == 0) {
                atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_HOLE);
                p.vnum[s] = 0;
                p.tnum[s] = 0;
            }
            __syncthreads();
            continue;
        }
        __syncthreads();
        const int64_t pb = 2 * (to - p.tbase);
        int64_t npair = 0;
        for (int base = 0; base < T; base += GSTAR_NT) {
            const int t = base + tid;
            const uint32_t f = t < T ? L.tfl[t] : 0u;
            TriPairs pr{STAR_PAIR_NONE, STAR_PAIR_NONE};
            if (f & TF_ALIVE) {
                const int a = L.tva[3 * t], b = L.tva[3 * t + 1], c = L.tva[3 * t + 2];
                const int ra = L.vremap[a], rb = L.vremap[b], rc = L.vremap[c];
                const int o0 = L.remap[L.to[3 * t]], o1 = L.remap[L.to[3 * t + 1]], o2 = L.remap[L.to[3 * t + 2]];
                const int64_t d = L.remap[t];
                if (wide) {
                    p.tpool[to + 2 * d] = wpack3(ra, rb, rc) | (1ull << 63);
                    p.tpool[to + 2 * d + 1] = wpack3(o0, o1, o2);
                } else {
                    p.tpool[to + d] = hpack(ra, rb, rc, o0, o1, o2, true);
                }
                pr = star_tri_pairs(L.vid[a], L.vid[b], L.vid[c], !(f & TF_CHECKED));
            }
            // the star's pairs, dense, in triangle order
            const int np = (pr.x != STAR_PAIR_NONE ? 1 : 0) + (pr.y != STAR_PAIR_NONE ? 1 : 0);
            int tot;
            const int64_t at = npair + block_excl(np, &tot, red);
            if (np > 0) p.pairbuf[pb + at] = pr.x;
            if (np > 1) p.pairbuf[pb + at + 1] = pr.y;
            npair += tot;
        }
        if (tid == 0) {
            p.pcount[s] = (int)npair;
            atomicAdd(&cnt[G4D_CNT_PAIRS], (unsigned long long)npair);
        }
        const int hn = star_history_merge(p, s, L.ins, m, tid, GSTAR_NT);
        __syncthreads();
        if (tid == 0) star_commit(p, s, vcount, vo, tcount, to, hn + m);
        __syncthreads();
    }
}

hipError_t launch_star_global(const StarParams &p, const int *list, int nitems, char *ws, int64_t ws_stride, int vcap,
                              int nblocks, hipStream_t s)
{
    if (nitems <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_star_global, dim3(nblocks), dim3(GSTAR_NT), 0, s, p, list, nitems, ws, ws_stride, vcap);
    return hipGetLastError();
}

__global__ void k_need_max(StarParams p, const int *list, int nitems, unsigned long long *out)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nitems; i += gridDim.x * blockDim.x) {
        const int s = list[i];
        const int64_t need = (p.ins_off[s + 1] - p.ins_off[s]) + (p.mode ? p.vnum[s] : 0);
        atomicMax(out, (unsigned long long)need);
    }
}

hipError_t launch_need_max(const StarParams &p, const int *list, int nitems, unsigned long long *out, hipStream_t s)
{
    if (nitems <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_need_max, dim3(g4d_blocks(nitems, 256, 1024)), dim3(256), 0, s, p, list, nitems, out);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------
// Containment proofs for drowned insertions (GD/GDelaunay/GDelPredKernels.cu:427-520).
// exVert is the lowest link vertex; the proof triangle is the unique live triangle
// without exVert whose three edges give one orient4(s, v, exVert, edge) sign.
// ------------------------------------------------------------------------------------

// EXACT = false: filters only, over all tasks; a task with an inconclusive orientation goes to
// p.xlist.  EXACT = true: the tasks listed in p.xlist, with exact predicates and SoS.
// Minimum over the GL lanes of a group (GL a power of two dividing 64).
template <int GL>
__device__ __forceinline__ int grp_min(int v)
{
    // minima within each 16-lane DPP row (rotations 8, 4, 2, 1); a whole-wave group then reads
    // the four rows' minima into scalars.  Every lane of the group must be active.
    static_assert(GL == 16 || GL == 64, "groups are DPP rows or the whole wave");
    int x = v;
    x = min(x, __builtin_amdgcn_update_dpp(x, x, 0x128, 0xf, 0xf, false));
    x = min(x, __builtin_amdgcn_update_dpp(x, x, 0x124, 0xf, 0xf, false));
    x = min(x, __builtin_amdgcn_update_dpp(x, x, 0x122, 0xf, 0xf, false));
    x = min(x, __builtin_amdgcn_update_dpp(x, x, 0x121, 0xf, 0xf, false));
    if constexpr (GL == 64)
        x = min(min(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
                min(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
    return x;
}

// One task per group of GL lanes: the filter pass takes 16 lanes per task (four tasks per
// wave; a star has about 27 link triangles, so a whole wave per task left most lanes idle),
// the exact pass a whole wave.  The lanes of a group stay together: every loop that ends in a
// group reduction has a trip count uniform over the group.
template <bool EXACT, int GL>
__global__ void __launch_bounds__(64) k_proofs(ProofParams p)
{
    constexpr int NG = 64 / GL;
    const int lane = threadIdx.x, g = lane / GL, gl = lane % GL;
    // the counts come from the device, so that no host round trip precedes either launch
    const int64_t nc = (int64_t)p.cnt[EXACT ? G4D_CNT_APPEND5 : G4D_CNT_TASKS];
    const int64_t nt = min(nc, EXACT ? p.xcap : p.ntasks);
    for (int64_t it = (int64_t)blockIdx.x * NG + g; it < nt; it += (int64_t)gridDim.x * NG) {
        const int64_t task = EXACT ? p.xlist[it] : it;
        const uint64_t tk = p.tasks[task];
        const int s = (int)(tk >> 32), v = (int)(uint32_t)tk;
        const int vn = p.vnum[s], tn = p.tnum[s];
        const bool wide = vn >= STAR_WIDE_MIN;
        const int64_t vo = p.voff[s], to = p.toff[s];
        int mn = 0x7fffffff;
        for (int i = gl; i < vn; i += GL) mn = min(mn, p.vpool[vo + i]);
        const int ex = grp_min<GL>(mn);
        int k0 = 0x7fffffff, k1 = 0x7fffffff, k2 = 0x7fffffff;
        bool unc = false;
        for (int t = gl; t < tn; t += GL) {
            int lv[3];
            star_tri_verts(p.tpool, to, t, wide, lv);
            const int a = p.vpool[vo + lv[0]], b = p.vpool[vo + lv[1]], c = p.vpool[vo + lv[2]];
            if (a == ex || b == ex || c == ex) continue;
            const int tri[3] = {a, b, c};
            int o[3];
            bool ok = true;
            for (int i = 0; i < 3 && ok; i++) {
                const int pv = tri[i], tv2 = tri[(i + 1) % 3];
                const double *pp[5] = {p.pts + 3 * (int64_t)s, p.pts + 3 * (int64_t)v, p.pts + 3 * (int64_t)ex,
                                       p.pts + 3 * (int64_t)pv, p.pts + 3 * (int64_t)tv2};
                if (EXACT) {
                    const int idx[5] = {s, v, ex, pv, tv2};
                    o[i] = orient4_full(pp, idx, p.cnt);
                } else {
                    o[i] = filter_insphere(pp);
                    if (o[i] == 0) {
                        unc = true;
                        ok = false;
                    }
                }
                if (i > 0 && o[i] != o[0]) ok = false;
            }
            if (!ok) continue;
            int x0 = a, x1 = b, x2 = c, tmp;
            if (x0 > x1) { tmp = x0; x0 = x1; x1 = tmp; }
            if (x1 > x2) { tmp = x1; x1 = x2; x2 = tmp; }
            if (x0 > x1) { tmp = x0; x0 = x1; x1 = tmp; }
            if (x0 < k0 || (x0 == k0 && (x1 < k1 || (x1 == k1 && x2 < k2)))) {
                k0 = x0;
                k1 = x1;
                k2 = x2;
            }
        }
        // the group's verdict: any inconclusive filter sends the task to the exact pass
        if (!EXACT && grp_min<GL>(unc ? 0 : 1) == 0) {
            if (gl == 0) {
                const unsigned long long k = atomicAdd(&p.cnt[G4D_CNT_APPEND5], 1ull);
                if ((int64_t)k < p.xcap) p.xlist[k] = task;
                else atomicOr(&p.cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_BUFFER);
            }
            continue;
        }
        const int b0 = grp_min<GL>(k0);
        const int b1 = grp_min<GL>(k0 == b0 ? k1 : 0x7fffffff);
        const int b2 = grp_min<GL>((k0 == b0 && k1 == b1) ? k2 : 0x7fffffff);
        if (gl == 0) {
            uint64_t *o = p.out + 4 * task;
            if (b0 == 0x7fffffff) {
                atomicOr(&p.cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_PROOF);
                o[0] = o[1] = o[2] = o[3] = ~0ull;
            } else {
                const int xs[4] = {ex, b0, b1, b2};
                for (int j = 0; j < 4; j++) {
                    const int a = v < xs[j] ? v : xs[j], b = v < xs[j] ? xs[j] : v;
                    o[j] = ((uint64_t)(uint32_t)a << 32) | (uint32_t)b;
                }
            }
        }
    }
}

hipError_t launch_proofs(const ProofParams &p, bool exact, hipStream_t s)
{
    const int64_t nt = exact ? p.xcap : p.ntasks;
    if (nt <= 0) return hipSuccess;
    if (exact) {
        const int nb = (int)(nt < 1024 ? nt : 1024);
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_proofs<true, 64>), dim3(nb), dim3(64), 0, s, p);
    } else {
        const int64_t nw = (nt + 3) / 4; // four tasks per wave
        const int nb = (int)(nw < 65536 ? nw : 65536);
        hipLaunchKernelGGL(HIP_KERNEL_NAME(k_proofs<false, 16>), dim3(nb), dim3(64), 0, s, p);
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------
// Drowned pairs, mutual removal (GD/GDelaunay/GDelHost.cu:832-875), history filter,
// reciprocation, capacities
// ------------------------------------------------------------------------------------

// Exclusive prefix of v over the work-group's threads (NT of them) and the total; red holds NT / 64 values
// and is free again when every thread has passed the next barrier.  T is int, or int64_t where a tile's
// sum can pass 2^31: 4,096 stars of 131,074 vertices (a set of two skew lines, some 135,000 points) take
// 2^31 triangle words.
template <int NT, typename T>
__device__ __forceinline__ T list_excl(T v, T *red, T *tot)
{
    T inc;
    if constexpr (sizeof(T) == 8) inc = g4d_wave_incl_sum64(v);
    else inc = g4d_wave_incl_sum(v);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 63) red[w] = inc;
    __syncthreads();
    T base = 0, all = 0;
#pragma unroll
    for (int i = 0; i < NT / 64; i++) {
        const T x = red[i];
        if (i < w) base += x;
        all += x;
    }
    *tot = all;
    return base + inc - v;
}
static constexpr int LA_THREADS = 256;

// Whether a pass has stars left for the exact or the global-memory kernel, which the host launches when
// it sees their counts: its lists are not complete yet.
__device__ __forceinline__ bool pass_open(const unsigned long long *cnt)
{
    return cnt[G4D_CNT_APPEND4] != 0 || cnt[G4D_CNT_XL] != 0;
}

// Key of drowned insertion k = star << 32 | vertex: the pair in order, then who inserted whom.
__device__ __forceinline__ uint64_t drown_key(uint64_t k)
{
    const uint32_t st = (uint32_t)(k >> 32), v = (uint32_t)k;
    const uint32_t mn = st < v ? st : v, mx = st < v ? v : st;
    return ((uint64_t)mn << 33) | ((uint64_t)mx << 1) | (uint64_t)(st == mn ? 0 : 1);
}

// Proof task of the sorted drowned key k between its neighbours (all ones at the ends), or
// STAR_PAIR_NONE when the drowning is mutual.
__device__ __forceinline__ uint64_t drown_task(uint64_t k, uint64_t prev, uint64_t next)
{
    const uint64_t pair = k >> 1;
    if ((prev >> 1) == pair || (next >> 1) == pair) return STAR_PAIR_NONE;
    const uint32_t mn = (uint32_t)(k >> 33), mx = (uint32_t)(pair & 0xffffffffu);
    return (k & 1) ? (((uint64_t)mx << 32) | mn) : (((uint64_t)mn << 32) | mx);
}

// Sorts n keys in LDS (n a power of two, at least 128) with NT threads.  A step's pairs are at most 64
// apart within the 128 keys of a wave's 64 pairs, so the work-group meets only around the wider
// steps (6 of 55 for 1,024 keys, 15 of 78 for 4,096).
template <int NT>
__device__ __forceinline__ void lds_bitonic(uint64_t *a, int n)
{
    for (int k = 2; k <= n; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int x = threadIdx.x; x < n / 2; x += NT) {
                const int i = ((x & ~(j - 1)) << 1) | (x & (j - 1)), l = i | j;
                const uint64_t u = a[i], w = a[l];
                if ((u > w) == ((i & k) == 0)) {
                    a[i] = w;
                    a[l] = u;
                }
            }
            if (j > 64 || (j == 1 && k > 64)) __syncthreads();
            else wave_sync();
        }
    __syncthreads();
}

// A tile of 16 flags a thread; HBM bound (one byte an insertion, 16 more for a drowned one).
__global__ void __launch_bounds__(LA_THREADS) k_drown_keys(const uint64_t *ins_keys, const uint8_t *dflag, int64_t m,
                                                           uint64_t *keys, unsigned long long *cnt)
{
    __shared__ int red[LA_THREADS / 64];
    __shared__ unsigned long long base;
    const int64_t i0 = ((int64_t)blockIdx.x * LA_THREADS + threadIdx.x) * 16;
    uint32_t bits = 0;
    if (i0 < m) {
        const uint4 f = *reinterpret_cast<const uint4 *>(dflag + i0);
        const uint32_t w[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
        for (int j = 0; j < 16; j++) bits |= ((w[j >> 2] >> (8 * (j & 3))) & 1u) << j;
        if (m - i0 < 16) bits &= (1u << (m - i0)) - 1u;
    }
    int tot;
    const int at = list_excl<LA_THREADS, int>(__popc(bits), red, &tot);
    if (threadIdx.x == 0 && tot) base = atomicAdd(&cnt[G4D_CNT_DROWN_KEYS], (unsigned long long)tot);
    __syncthreads();
    uint64_t *out = keys + base + at;
    for (; bits; bits &= bits - 1) *out++ = drown_key(ins_keys[i0 + __builtin_ctz(bits)]);
}

hipError_t launch_drown_keys(const uint64_t *ins_keys, const uint8_t *dflag, int64_t m, uint64_t *keys,
                             unsigned long long *cnt, hipStream_t s)
{
    if (m <= 0) return hipSuccess;
    const int64_t nb = (m + 16 * LA_THREADS - 1) / (16 * LA_THREADS);
    if (nb > INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_drown_keys, dim3((unsigned)nb), dim3(LA_THREADS), 0, s, ins_keys, dflag, m, keys, cnt);
    return hipGetLastError();
}

static constexpr int NM_ITEMS = 8;
__global__ void __launch_bounds__(LA_THREADS) k_nonmutual(const uint64_t *keys, int64_t m, uint64_t *tasks,
                                                          unsigned long long *cnt)
{
    __shared__ int red[LA_THREADS / 64];
    __shared__ unsigned long long base;
    const int64_t b0 = (int64_t)blockIdx.x * (LA_THREADS * NM_ITEMS) + threadIdx.x;
    uint64_t task[NM_ITEMS];
    int c = 0;
#pragma unroll
    for (int j = 0; j < NM_ITEMS; j++) {
        const int64_t i = b0 + j * LA_THREADS;
        task[j] = STAR_PAIR_NONE;
        if (i >= m) continue;
        task[j] = drown_task(keys[i], i > 0 ? keys[i - 1] : ~0ull, i + 1 < m ? keys[i + 1] : ~0ull);
        c += task[j] != STAR_PAIR_NONE ? 1 : 0;
    }
    int tot;
    int at = list_excl<LA_THREADS>(c, red, &tot);
    if (threadIdx.x == 0 && tot) base = atomicAdd(&cnt[G4D_CNT_TASKS], (unsigned long long)tot);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NM_ITEMS; j++)
        if (task[j] != STAR_PAIR_NONE) tasks[base + at++] = task[j];
}

hipError_t launch_nonmutual(const uint64_t *keys, int64_t m, uint64_t *tasks, unsigned long long *cnt, hipStream_t s)
{
    if (m <= 0) return hipSuccess;
    const int64_t nb = (m + LA_THREADS * NM_ITEMS - 1) / (LA_THREADS * NM_ITEMS);
    if (nb > INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_nonmutual, dim3((unsigned)nb), dim3(LA_THREADS), 0, s, keys, m, tasks, cnt);
    return hipGetLastError();
}

// The drowned insertions of a late round, at most DROWN_SMALL of them, to proof tasks in one launch:
// the keys collected in LDS, a bitonic sort, and the tasks of the ones that are not mutual, in the
// place of three launches and the gaps between them.  Bound by latency: 13-17 us for up to a thousand
// drowned, 24 us for 1,700 of 4,600 insertions, as long as the three kernels alone took; 39 us for lists
// that the sort pads to 4,096.
__global__ void __launch_bounds__(1024) k_drown_small(const uint64_t *ins_keys, const uint8_t *dflag, int m, int nd,
                                                      uint64_t *tasks, unsigned long long *cnt)
{
    __shared__ uint64_t a[DROWN_SMALL];
    __shared__ int have, ntask;
    const int tid = threadIdx.x, lane = __lane_id();
    if (nd < 0) { // launched ahead of the host's look at the pass
        if (pass_open(cnt)) return;
        nd = (int)min(cnt[G4D_CNT_DROWNED], (unsigned long long)DROWN_SMALL);
        if (nd == 0) return;
    }
    int n = 128;
    while (n < nd) n <<= 1;
    for (int i = tid; i < n; i += 1024) a[i] = ~0ull;
    if (tid == 0) have = ntask = 0;
    __syncthreads();
    // four flags a thread: their keys' reads are the chain here
    for (int i0 = tid * 4; i0 < m; i0 += 1024 * 4) {
        const uint32_t f = *reinterpret_cast<const uint32_t *>(dflag + i0);
        uint64_t k[4];
        bool d[4];
        int c = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            d[j] = i0 + j < m && ((f >> (8 * j)) & 1u);
            k[j] = d[j] ? ins_keys[i0 + j] : 0ull;
            c += d[j] ? 1 : 0;
        }
        int at = c ? atomicAdd(&have, c) : 0;
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (d[j]) {
                if (at < DROWN_SMALL) a[at] = drown_key(k[j]);
                at++;
            }
    }
    __syncthreads();
    lds_bitonic<1024>(a, n);
    const int c = min(have, DROWN_SMALL);
    for (int i0 = 0; i0 < c; i0 += 1024) {
        const int i = i0 + tid;
        uint64_t task = STAR_PAIR_NONE;
        if (i < c) task = drown_task(a[i], i > 0 ? a[i - 1] : ~0ull, i + 1 < c ? a[i + 1] : ~0ull);
        const uint64_t mk = __ballot(task != STAR_PAIR_NONE);
        int at = 0;
        if (lane == 0 && mk) at = atomicAdd(&ntask, __popcll(mk));
        at = __builtin_amdgcn_readfirstlane(at) + __popcll(mk & ((1ull << lane) - 1ull));
        if (task != STAR_PAIR_NONE) tasks[at] = task;
    }
    __syncthreads();
    if (tid == 0) cnt[G4D_CNT_TASKS] = (unsigned long long)ntask;
}

hipError_t launch_drown_small(const uint64_t *ins_keys, const uint8_t *dflag, int64_t m, int64_t nd, uint64_t *tasks,
                              unsigned long long *cnt, hipStream_t s)
{
    if (nd == 0 || m <= 0) return hipSuccess;
    if (nd > DROWN_SMALL || m > (nd < 0 ? DROWN_SMALL : DROWN_SMALL_INS)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_drown_small, dim3(1), dim3(1024), 0, s, ins_keys, dflag, (int)m, (int)nd, tasks, cnt);
    return hipGetLastError();
}

// One pass from the stars' pair regions and the proofs' pairs to the appended keys.  An edge is in the
// links of some five stars, which lie near each other in the list: a wave walks rows of consecutive
// stars (16 lanes a star), drops the pairs that its work-group has lately seen, and queues the others,
// so that the histories' binary searches (some six dependent reads each) run in full waves, two a lane.
// What is new is staged and leaves with one atomic: all of them meet at one counter, and with a
// stage of 160 instead of 672 the first pass below took 4.4 ms.  Bound by the searches' latency and
// divergent lines.  4,194,304 uniform points, 12 rounds: 2.5 ms, of which the first pass 1.5; a search per
// pair where it is read, with nothing dropped or queued, 3.75 and 2.1.
static constexpr int NP_LANE = 2, NP_DRAIN = 64 * NP_LANE, NP_QUEUE = NP_DRAIN + 64, NP_STAGE = 672, NP_WIDE = 128,
                     NP_SEEN = 1024, NP_ROW = 1024;

__global__ void __launch_bounds__(LA_THREADS) k_new_pairs(NewPairs p)
{
    constexpr int W = LA_THREADS / 64, G = LA_THREADS / 16;
    __shared__ uint64_t queue_[W][NP_QUEUE], stage_[W][NP_STAGE], seen[NP_SEEN];
    __shared__ int nwide;
    __shared__ uint16_t wide[NP_ROW];
    const int tid = threadIdx.x, sub = tid & 15, lane = tid & 63, wv = tid >> 6;
    uint64_t *queue = queue_[wv], *stage = stage_[wv];
    int nq = 0, ns = 0; // this wave's
    if (p.ahead && pass_open(p.cnt)) return;
    for (int i = tid; i < NP_SEEN; i += LA_THREADS) seen[i] = STAR_PAIR_NONE;
    if (tid == 0) nwide = 0;
    __syncthreads();
    // All of these are called by whole waves.
    auto add = [&](int n) {
        unsigned long long base = 0;
        if (lane == 0) base = atomicAdd(&p.cnt[G4D_CNT_NEW_PAIRS], (unsigned long long)n);
        return __shfl(base, 0, 64);
    };
    auto flush = [&](int n, unsigned long long base) {
        wave_sync();
        for (int i = lane; i < n; i += 64) {
            const uint64_t k = stage[i];
            reinterpret_cast<ulonglong2 *>(p.keys)[base + i] = make_ulonglong2(k, (k << 32) | (k >> 32));
        }
        wave_sync();
        ns = 0;
    };
    // The last n <= NP_DRAIN pairs of the queue: new when b is not in a's history.
    auto drain = [&](int n) {
        wave_sync();
        uint64_t k[NP_LANE];
        int64_t h[NP_LANE];
        int lo[NP_LANE], hi[NP_LANE];
        nq -= n;
#pragma unroll
        for (int j = 0; j < NP_LANE; j++) {
            const int i = j * 64 + lane;
            k[j] = i < n ? queue[nq + i] : STAR_PAIR_NONE;
        }
#pragma unroll
        for (int j = 0; j < NP_LANE; j++) {
            const bool v = k[j] != STAR_PAIR_NONE;
            const uint32_t a = v ? (uint32_t)(k[j] >> 32) : 0u;
            h[j] = p.hoff[a];
            hi[j] = v ? p.hnum[a] : 0;
            lo[j] = 0;
        }
        for (;;) {
            bool more = false;
#pragma unroll
            for (int j = 0; j < NP_LANE; j++) more = more || lo[j] < hi[j];
            if (!__ballot(more)) break;
            int mid[NP_LANE];
            uint32_t x[NP_LANE];
#pragma unroll
            for (int j = 0; j < NP_LANE; j++) {
                mid[j] = (lo[j] + hi[j]) >> 1;
                // a search that is over reads the pool's first word, so that all reads leave together
                x[j] = (uint32_t)p.hpool[lo[j] < hi[j] ? h[j] + mid[j] : 0];
            }
#pragma unroll
            for (int j = 0; j < NP_LANE; j++) {
                const bool in = lo[j] < hi[j], less = x[j] < (uint32_t)k[j], same = x[j] == (uint32_t)k[j];
                if (in && less) lo[j] = mid[j] + 1;
                if (in && !less) hi[j] = mid[j];
                if (in && same) k[j] = STAR_PAIR_NONE, hi[j] = lo[j]; // found: not new
            }
        }
        wave_sync();
#pragma unroll
        for (int j = 0; j < NP_LANE; j++) {
            const bool f = k[j] != STAR_PAIR_NONE;
            const uint64_t mk = __ballot(f);
            if (f) stage[ns + __popcll(mk & ((1ull << lane) - 1ull))] = k[j];
            ns += __popcll(mk);
        }
        if (ns > NP_STAGE - NP_DRAIN) flush(ns, add(ns));
    };
    auto put = [&](bool have, uint64_t k) {
        const uint32_t a = (uint32_t)(k >> 32), b = (uint32_t)k;
        bool f = have && a < b;
        if (f) {
            // an entry is read and written whole (64-bit LDS accesses); one that another pair takes
            // only means another look
            uint64_t *e = &seen[(a * 0x9e3779b1u ^ b * 0x85ebca6bu) >> (32 - __builtin_ctz(NP_SEEN))];
            f = __hip_atomic_load(e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != k;
            if (f) __hip_atomic_store(e, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        const uint64_t mk = __ballot(f);
        if (f) queue[nq + __popcll(mk & ((1ull << lane) - 1ull))] = k;
        nq += __popcll(mk);
        if (nq >= NP_DRAIN) drain(NP_DRAIN);
    };
    const int row = max(G, min(NP_ROW, (p.nitems / (int)gridDim.x + G - 1) / G * G));
    for (int64_t r0 = (int64_t)blockIdx.x * row; r0 < p.nitems; r0 += (int64_t)gridDim.x * row) {
        // 16 stars of the row a step, four of them this wave's
        const int nrow = (int)min((int64_t)row, p.nitems - r0);
        // the reads of a step (list entry, then count and region, then the first pairs) are made one, two
        // and three steps ahead: each waits for the one before
        auto star = [&](int64_t i) { // ~s: on a tier's list
            const int s = p.list[i];
            return s < 0 ? ~s : s;
        };
        auto entry = [&](int i) { return i < nrow ? star(r0 + i) : -1; };
        struct Region {
            int c;
            int64_t off;
        };
        auto region = [&](int s) { return s >= 0 ? Region{p.pcount[s], p.ntoff[s]} : Region{0, p.tbase}; };
        auto pair = [&](const Region &g, int k) { return k < g.c ? p.pairbuf[2 * (g.off - p.tbase) + k] : 0ull; };
        const int i1 = 4 * wv + (lane >> 4);
        Region g0 = region(entry(i1)), g1 = region(entry(i1 + G));
        int s2 = entry(i1 + 2 * G);
        uint64_t pr0 = pair(g0, sub);
        for (int i0 = 4 * wv; i0 < nrow; i0 += G) {
            const int i = i0 + (lane >> 4);
            const int s3 = entry(i + 3 * G);
            const Region g2 = region(s2);
            const uint64_t pr1 = pair(g1, sub);
            int c = g0.c;
            if (c > NP_WIDE) {
                if (sub == 0) wide[atomicAdd(&nwide, 1)] = (uint16_t)i;
                c = 0;
            }
            const int cmax = g4d_wave_max(c);
            uint64_t pr = pr0;
            for (int k0 = 0; k0 < cmax; k0 += 16) {
                const int k = k0 + sub;
                const uint64_t next = pair(g0, k + 16); // read ahead of this one's searches
                put(k < c, pr);
                pr = next;
            }
            g0 = g1;
            g1 = g2;
            s2 = s3;
            pr0 = pr1;
        }
        __syncthreads();
        // stars with many pairs: all waves together
        const int nw = nwide;
        __syncthreads();
        if (nw == 0) continue;
        if (tid == 0) nwide = 0;
        for (int w = 0; w < nw; w++) {
            const int s = star(r0 + wide[w]), c = p.pcount[s];
            const uint64_t *src = p.pairbuf + 2 * (p.ntoff[s] - p.tbase);
            for (int k0 = 64 * wv; k0 < c; k0 += LA_THREADS) put(k0 + lane < c, k0 + lane < c ? src[k0 + lane] : 0ull);
        }
        __syncthreads(); // wide[] and nwide are free again
    }
    const int64_t np = 4 * min((int64_t)p.cnt[G4D_CNT_TASKS], p.ntasks);
    for (int64_t k0 = ((int64_t)blockIdx.x * W + wv) * 64; k0 < np; k0 += (int64_t)gridDim.x * LA_THREADS)
        put(k0 + lane < np, k0 + lane < np ? p.proofs[k0 + lane] : 0ull);
    while (nq > 0) drain(min(nq, NP_DRAIN));
    // what the waves have left, with one atomic
    __shared__ int left[W];
    __shared__ unsigned long long rest;
    if (lane == 0) left[wv] = ns;
    __syncthreads();
    int before = 0, all = 0;
    for (int w = 0; w < W; w++) {
        if (w < wv) before += left[w];
        all += left[w];
    }
    if (tid == 0) rest = all ? atomicAdd(&p.cnt[G4D_CNT_NEW_PAIRS], (unsigned long long)all) : 0ull;
    __syncthreads();
    flush(ns, rest + before);
}

hipError_t launch_new_pairs(const NewPairs &p, hipStream_t s)
{
    const int64_t work = std::max<int64_t>(16 * (int64_t)p.nitems, 4 * p.ntasks);
    if (work <= 0) return hipSuccess;
    if (!p.list && p.nitems > 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_new_pairs, dim3(g4d_blocks(work, LA_THREADS, 2048)), dim3(LA_THREADS), 0, s, p);
    return hipGetLastError();
}

// Region sizes of star s with m insertions.
__device__ __forceinline__ void plan_sizes(const PassPlan &p, int s, int m, int *v, int64_t *t, int *h)
{
    *v = p.vnum[s] + m;
    *t = star_tcap_words(*v);
    *h = p.hnum[s] + m;
}

// A star on a tier's list is marked on the pass's list (~s): the 32-vertex kernel must not look at its
// record, which the other tier's kernel may have rebuilt already, to see that it is not its own.
__device__ __forceinline__ void plan_star(const PassPlan &p, int s, int64_t first, int m, unsigned long long item,
                                          int64_t v, int64_t t, int64_t h, bool tiered)
{
    p.ins_off[s] = first;
    p.ins_off[s + 1] = first + m; // the following star's first, when that has insertions too
    p.list[item] = tiered ? ~s : s;
    p.nvoff[s] = v;
    p.ntoff[s] = t;
    p.nhoff[s] = h;
    p.pcount[s] = 0;
}

// Tier of a star above 32, -1 for one that the 32-vertex kernel takes.  A pass of few keys sends all of
// tiers 64 to 256 to the 256-vertex kernel: its resident waves hold them all, the tiers number a star's
// slots alike, and the stars' chains of insertions run side by side and not launch after launch
// (100,000 uniform points, six late passes: 1.15 -> 0.30 ms; up to some 1,500 stars, four keys each).
static constexpr int TIER_MERGE_KEYS = 6144;
__device__ __forceinline__ int star_tier(int need, int lim, bool merge)
{
    if (need <= min(STAR_VMAX_T0, lim)) return -1;
    if (need <= min(STAR_VMAX_T2, lim)) return merge || need > STAR_VMAX_TM ? 2 : (need > STAR_VMAX_T1 ? 1 : 0);
    if (lim < STAR_LDS_LIMIT) return 5; // a lowered limit sends every larger star to the global-memory kernel
    return need <= STAR_VMAX_W1 ? 3 : (need <= STAR_VMAX_W2 ? 4 : 5);
}
__device__ __forceinline__ void tier_put(const PassPlan &p, int tier, int k, int s)
{
    p.tier[tier >> 1][(tier & 1) ? p.n - 1 - k : k] = s;
}

// A tile of keys is read once, in order, into LDS (a thread that reads its own eight in a row loads
// every line eight times); the keys that start a star's run are listed, and a thread plans a few
// stars in a row.  Only the tile's last run has its end searched for, by doubling steps.  The tile's
// stars take list entries and regions with one atomic per counter, in key order within the tile.
// Bound by those atomics' one cache line and the stars' scattered records: star creation
// at 4,194,304 uniform points 0.23 ms (0.42 with tiles of 2,048 keys).
static constexpr int PP_ITEMS = 16, PP_TILE = LA_THREADS * PP_ITEMS;
__global__ void __launch_bounds__(LA_THREADS) k_pass_plan(PassPlan p, const uint64_t *keys, int64_t m, const int64_t *dev_m)
{
    __shared__ uint32_t sid[PP_TILE];
    __shared__ uint16_t first[PP_TILE + 1];
    __shared__ int runs_[LA_THREADS / 64];
    __shared__ int64_t red[3][LA_THREADS / 64];
    __shared__ unsigned long long base[4];
    __shared__ int last_len, tn[STAR_TIERS + 2]; // per tier, above 64, largest beyond the tiers
    if (dev_m) m = min(m, *dev_m);
    const int64_t t0 = (int64_t)blockIdx.x * PP_TILE;
    if (t0 >= m) return;
    const int nt = (int)min((int64_t)PP_TILE, m - t0), tid = threadIdx.x;
    const bool merge = m <= TIER_MERGE_KEYS;
    if (tid < STAR_TIERS + 2) tn[tid] = 0;
    {
        uint64_t k[PP_ITEMS];
#pragma unroll
        for (int j = 0; j < PP_ITEMS; j++) k[j] = keys[t0 + min(j * LA_THREADS + tid, nt - 1)];
#pragma unroll
        for (int j = 0; j < PP_ITEMS; j++) sid[j * LA_THREADS + tid] = (uint32_t)(k[j] >> 32);
    }
    const uint32_t before = tid == 0 && t0 > 0 ? (uint32_t)(keys[t0 - 1] >> 32) : 0u;
    __syncthreads();
    // starts of runs: a wave takes 64 keys in a row at a time
    const int lane = tid & 63, wv = tid >> 6;
    constexpr int PER = PP_TILE / (LA_THREADS / 64); // keys of a wave
    uint64_t fl[PER / 64];
    int mine = 0;
#pragma unroll
    for (int j = 0; j < PER / 64; j++) {
        const int i = wv * PER + j * 64 + lane;
        const bool f = i < nt && (i > 0 ? sid[i - 1] != sid[i] : t0 == 0 || before != sid[0]);
        fl[j] = __ballot(f);
        mine += __popcll(fl[j]);
    }
    if (lane == 0) runs_[wv] = mine;
    __syncthreads();
    int at = 0, runs = 0;
    for (int w = 0; w < LA_THREADS / 64; w++) {
        if (w < wv) at += runs_[w];
        runs += runs_[w];
    }
#pragma unroll
    for (int j = 0; j < PER / 64; j++) {
        if ((fl[j] >> lane) & 1) first[at + __popcll(fl[j] & ((1ull << lane) - 1))] = (uint16_t)(wv * PER + j * 64 + lane);
        at += __popcll(fl[j]);
    }
    __syncthreads();
    if (runs == 0) return; // all of one run from an earlier tile
    if (tid == 0) {
        const uint32_t s = sid[nt - 1];
        int64_t lo = t0 + nt - 1, step = 1; // keys[lo] is s
        while (lo + step < m && (uint32_t)(keys[lo + step] >> 32) == s) {
            lo += step;
            step *= 2;
        }
        int64_t hi = min(lo + step, m);
        while (lo + 1 < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if ((uint32_t)(keys[mid] >> 32) == s) lo = mid;
            else hi = mid;
        }
        last_len = (int)(lo + 1 - t0 - first[runs - 1]);
    }
    __syncthreads();
    const int R = (runs + LA_THREADS - 1) / LA_THREADS, r0 = min(tid * R, runs), r1 = min(r0 + R, runs);
    int64_t v = 0, t = 0, h = 0;
    for (int r = r0; r < r1; r++) {
        int dv, dh;
        int64_t dt;
        plan_sizes(p, (int)sid[first[r]], r + 1 < runs ? first[r + 1] - first[r] : last_len, &dv, &dt, &dh);
        v += dv;
        t += dt;
        h += dh;
        const int tier = star_tier(dv, p.lds_limit, merge);
        if (tier >= 0) {
            atomicAdd(&tn[tier], 1);
            if (dv > min(STAR_VMAX_T1, p.lds_limit)) atomicAdd(&tn[STAR_TIERS], 1);
            if (tier == STAR_TIERS - 1) atomicMax(&tn[STAR_TIERS + 1], dv);
        }
    }
    int64_t tv, tt, th;
    const int64_t ev = list_excl<LA_THREADS>(v, red[0], &tv), et = list_excl<LA_THREADS>(t, red[1], &tt),
                  eh = list_excl<LA_THREADS>(h, red[2], &th);
    if (tid < 4) {
        const int64_t add[4] = {runs, tv, tt, th};
        const int c[4] = {G4D_CNT_ACTIVE, G4D_CNT_NEED_V, G4D_CNT_NEED_T, G4D_CNT_NEED_H};
        base[tid] = atomicAdd(&p.cnt[c[tid]], (unsigned long long)add[tid]);
    } else if (tid >= 64 && tid < 64 + STAR_TIERS + 2) {
        const int i = tid - 64, c = tn[i];
        if (c && i < STAR_TIERS) tn[i] = (int)atomicAdd(&p.cnt[G4D_CNT_TIER0 + i], (unsigned long long)c); // now a cursor
        else if (c && i == STAR_TIERS) atomicAdd(&p.cnt[G4D_CNT_OVER64], (unsigned long long)c);
        else if (c) atomicMax(&p.cnt[G4D_CNT_NEED_MAX], (unsigned long long)c);
    }
    __syncthreads();
    int64_t vo = p.base[0] + (int64_t)base[1] + ev, to = p.base[1] + (int64_t)base[2] + et,
            ho = p.base[2] + (int64_t)base[3] + eh;
    for (int r = r0; r < r1; r++) {
        const int s = (int)sid[first[r]], len = r + 1 < runs ? first[r + 1] - first[r] : last_len;
        int dv, dh;
        int64_t dt;
        plan_sizes(p, s, len, &dv, &dt, &dh);
        const int tier = star_tier(dv, p.lds_limit, merge);
        plan_star(p, s, t0 + first[r], len, base[0] + r, vo, to, ho, tier >= 0);
        if (tier >= 0) tier_put(p, tier, atomicAdd(&tn[tier], 1), s);
        vo += dv;
        to += dt;
        ho += dh;
    }
}

hipError_t launch_pass_plan(const PassPlan &p, const uint64_t *keys, int64_t m, const int64_t *dev_m, hipStream_t s)
{
    const int64_t nb = (m + PP_TILE - 1) / PP_TILE;
    if (nb <= 0) return hipSuccess;
    if (nb > INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_pass_plan, dim3((unsigned)nb), dim3(LA_THREADS), 0, s, p, keys, m, dev_m);
    return hipGetLastError();
}

// Late rounds insert a few thousand keys or fewer, and every one of the sort, unique, compaction and
// scan launches they took cost 3-10 us with a host round trip between some: 20 launches and four
// round trips.  One work-group does all of it in LDS: a bitonic sort (78 steps for 4,096
// keys), repeats removed, runs listed, region sizes scanned; bound by its barriers and LDS latency: 11 us
// for lists that the sort pads to 512 keys, 18 for 1,024, 40 to 44 for 4,096.
// With the appended lists before it a call on 1,000 points makes 178 launches instead of 331 (2.40 ->
// 1.70 ms), on 100,000 330 instead of 656 (7.1 -> 6.25 ms).
static constexpr int SR_THREADS = 1024;

__global__ void __launch_bounds__(SR_THREADS) k_small_round(PassPlan p, uint64_t *keys)
{
    __shared__ uint64_t a[STAR_ROUND_SMALL], b[STAR_ROUND_SMALL];
    __shared__ int first[STAR_ROUND_SMALL + 1];
    __shared__ int red[2][SR_THREADS / 64];
    __shared__ int64_t sum[3][SR_THREADS / 64];
    __shared__ int tn[STAR_TIERS + 2];
    const int tid = threadIdx.x;
    const unsigned long long np = p.cnt[G4D_CNT_NEW_PAIRS];
    if (np == 0 || np > STAR_ROUND_SMALL / 2) return;
    const int m = 2 * (int)np;
    int n = 128;
    while (n < m) n <<= 1;
    for (int i = tid; i < n; i += SR_THREADS) a[i] = i < m ? keys[i] : ~0ull;
    __syncthreads();
    lds_bitonic<SR_THREADS>(a, n);
    // repeats out, in order
    int cnt = 0;
    for (int i0 = 0, r = 0; i0 < m; i0 += SR_THREADS, r ^= 1) {
        const int i = i0 + tid;
        const bool f = i < m && (i == 0 || a[i] != a[i - 1]);
        int tot;
        const int at = cnt + list_excl<SR_THREADS>(f ? 1 : 0, red[r], &tot);
        if (f) {
            b[at] = a[i];
            keys[at] = a[i];
        }
        cnt += tot;
    }
    __syncthreads();
    // runs of one star
    int runs = 0;
    for (int i0 = 0, r = 0; i0 < cnt; i0 += SR_THREADS, r ^= 1) {
        const int i = i0 + tid;
        const bool f = i < cnt && (i == 0 || (b[i] >> 32) != (b[i - 1] >> 32));
        int tot;
        const int at = runs + list_excl<SR_THREADS>(f ? 1 : 0, red[r], &tot);
        if (f) first[at] = i;
        runs += tot;
    }
    if (tid == 0) first[runs] = cnt;
    __syncthreads();
    int64_t vo = p.base[0], to = p.base[1], ho = p.base[2];
    if (tid < STAR_TIERS + 2) tn[tid] = 0;
    __syncthreads();
    for (int r0 = 0; r0 < runs; r0 += SR_THREADS) {
        const int r = r0 + tid;
        int s = 0, len = 0, dv = 0, dh = 0;
        int64_t dt = 0;
        if (r < runs) {
            s = (int)(uint32_t)(b[first[r]] >> 32);
            len = first[r + 1] - first[r];
            plan_sizes(p, s, len, &dv, &dt, &dh);
        }
        int64_t tv, tt, th;
        const int64_t ev = list_excl<SR_THREADS, int64_t>(dv, sum[0], &tv), et = list_excl<SR_THREADS>(dt, sum[1], &tt),
                      eh = list_excl<SR_THREADS, int64_t>(dh, sum[2], &th);
        if (r < runs) {
            const int tier = star_tier(dv, p.lds_limit, true); // at most STAR_ROUND_SMALL keys
            plan_star(p, s, first[r], len, r, vo + ev, to + et, ho + eh, tier >= 0);
            if (tier >= 0) {
                tier_put(p, tier, atomicAdd(&tn[tier], 1), s);
                if (dv > min(STAR_VMAX_T1, p.lds_limit)) atomicAdd(&tn[STAR_TIERS], 1);
                if (tier == STAR_TIERS - 1) atomicMax(&tn[STAR_TIERS + 1], dv);
            }
        }
        vo += tv;
        to += tt;
        ho += th;
        __syncthreads();
    }
    if (tid == 0) {
        p.cnt[G4D_CNT_INS] = cnt;
        p.cnt[G4D_CNT_ACTIVE] = runs;
        p.cnt[G4D_CNT_NEED_V] = vo - p.base[0];
        p.cnt[G4D_CNT_NEED_T] = to - p.base[1];
        p.cnt[G4D_CNT_NEED_H] = ho - p.base[2];
    }
    static_assert(G4D_CNT_OVER64 == G4D_CNT_TIER0 + STAR_TIERS && G4D_CNT_NEED_MAX == G4D_CNT_OVER64 + 1 &&
                      STAR_ROUND_SMALL <= TIER_MERGE_KEYS,
                  "one row of counters; small rounds merge the tiers");
    if (tid < STAR_TIERS + 2) p.cnt[G4D_CNT_TIER0 + tid] = (unsigned long long)tn[tid];
}

hipError_t launch_small_round(const PassPlan &p, uint64_t *keys, hipStream_t s)
{
    hipLaunchKernelGGL(k_small_round, dim3(1), dim3(SR_THREADS), 0, s, p, keys);
    return hipGetLastError();
}

__global__ void k_reciprocate(uint64_t *keys, int64_t m)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t k = keys[i];
        keys[m + i] = (k << 32) | (k >> 32);
    }
}

hipError_t launch_reciprocate(uint64_t *keys, int64_t m, hipStream_t s)
{
    if (m <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_reciprocate, dim3(g4d_blocks(m, 256, 65536)), dim3(256), 0, s, keys, m);
    return hipGetLastError();
}

__global__ void k_live_sizes(int n, const int *vnum, const int *tnum, const int *hnum, int64_t *vsz, int64_t *tsz,
                             int64_t *hsz)
{
    for (int s = blockIdx.x * blockDim.x + threadIdx.x; s < n; s += gridDim.x * blockDim.x) {
        const int v = vnum[s];
        vsz[s] = v;
        tsz[s] = v >= STAR_WIDE_MIN ? 2 * (int64_t)tnum[s] : tnum[s];
        hsz[s] = hnum[s];
    }
}

hipError_t launch_live_sizes(int n, const int *vnum, const int *tnum, const int *hnum, int64_t *vsz, int64_t *tsz,
                             int64_t *hsz, hipStream_t s)
{
    hipLaunchKernelGGL(k_live_sizes, dim3(g4d_blocks(n, 256, 65536)), dim3(256), 0, s, n, vnum, tnum, hnum, vsz, tsz,
                       hsz);
    return hipGetLastError();
}

// 16 lanes a star, whose regions hold some 16 to 30 elements; stars of more than 16 rounds are copied by
// their whole wave afterwards.  Bound by the records' scattered reads and the copies; a wave per star
// left most lanes idle: 4,000,000 stars of 1.5 GB 2.06 ms, this 1.08.
__global__ void __launch_bounds__(256) k_repack(int n, const int *vnum, const int64_t *voff, const int *tnum,
                                                const int64_t *toff, const int *hnum, const int64_t *hoff,
                                                const int *vpool, const uint64_t *tpool, const int *hpool,
                                                const int64_t *vdst, const int64_t *tdst, const int64_t *hdst,
                                                int *vpool2, uint64_t *tpool2, int *hpool2)
{
    const int lane = threadIdx.x & 63, sub = lane & 15;
    const int64_t w0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6, nw = ((int64_t)gridDim.x * blockDim.x) >> 6;
    auto copy = [&](int s, int at, int step, bool big) {
        const int v = vnum[s], h = hnum[s];
        const int64_t tw = v >= STAR_WIDE_MIN ? 2 * (int64_t)tnum[s] : tnum[s];
        if (!big && max((int64_t)max(v, h), tw) > 256) return true;
        const int64_t vi = voff[s], ti = toff[s], hi = hoff[s], vo = vdst[s], to = tdst[s], ho = hdst[s];
        for (int i = at; i < v; i += step) vpool2[vo + i] = vpool[vi + i];
        for (int64_t i = at; i < tw; i += step) tpool2[to + i] = tpool[ti + i];
        for (int i = at; i < h; i += step) hpool2[ho + i] = hpool[hi + i];
        return false;
    };
    for (int64_t s0 = 4 * w0; s0 < n; s0 += 4 * nw) {
        const int64_t s = s0 + (lane >> 4);
        const bool big = s < n && copy((int)s, sub, 16, false);
        const uint64_t mk = __ballot(big);
        for (int g = 0; g < 4; g++)
            if ((mk >> (16 * g)) & 1) copy((int)(s0 + g), lane, 64, true);
    }
}

hipError_t launch_repack(int n, const int *vnum, const int64_t *voff, const int *tnum, const int64_t *toff,
                         const int *hnum, const int64_t *hoff, const int *vpool, const uint64_t *tpool,
                         const int *hpool, const int64_t *vdst, const int64_t *tdst, const int64_t *hdst, int *vpool2,
                         uint64_t *tpool2, int *hpool2, hipStream_t s)
{
    hipLaunchKernelGGL(k_repack, dim3(g4d_blocks(n, 16, 65536)), dim3(256), 0, s, n, vnum, voff, tnum, toff, hnum, hoff,
                       vpool, tpool, hpool, vdst, tdst, hdst, vpool2, tpool2, hpool2);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------
// Output tetrahedra: owner triangles (star id below its three link vertices) whose exact
// orient3d(v0, v1, v2, star) is negative; upper-hull and flat ones are dropped.
// ------------------------------------------------------------------------------------

// Keep flag of an owner triangle decided by the exact orient3d (bit 58 of a packed word, bit
// 63 of the second word of a wide one); clear as written by the star kernels.
__device__ __forceinline__ uint64_t *out_keep_word(const OutParams &p, int64_t to, int t, bool wide)
{
    return p.tpool + to + (wide ? 2 * (int64_t)t + 1 : (int64_t)t);
}
__device__ __forceinline__ uint64_t out_keep_bit(bool wide) { return wide ? (1ull << 63) : (1ull << 58); }

// The output passes give each star a group of OUT_GL lanes, one lane per link triangle in turn
// (a star has ~27 link triangles): four stars per wave step, so that each wave keeps four
// stars' chains of dependent reads (star record, triangle words, link ids, points) in flight
// instead of two.
static constexpr int OUT_GL = 16;
static constexpr int OUT_NG = 64 / OUT_GL;

// A wave takes up to 16 stars at a time: their records are read together, lane per star, and handed to
// the groups; a group's link ids wait in two registers a lane, read beside the triangle words.
struct OutStar {
    int tn, vn;
    int64_t vo, to;
};
__device__ __forceinline__ OutStar out_star_read(const OutParams &p, int s0)
{
    const int s = s0 + (int)(threadIdx.x & 15);
    if (s >= p.n) return OutStar{0, 0, 0, 0};
    return OutStar{p.tnum[s], p.vnum[s], p.voff[s], p.toff[s]};
}
__device__ __forceinline__ OutStar out_star_of(const OutStar &r, int i)
{
    return OutStar{__shfl(r.tn, i, 64), __shfl(r.vn, i, 64), (int64_t)__shfl((long long)r.vo, i, 64),
                   (int64_t)__shfl((long long)r.to, i, 64)};
}
struct OutLink {
    int v[2];
    bool regs; // no star of the wave's four has more than 32 link vertices
};
__device__ __forceinline__ OutLink out_link_read(const OutParams &p, const OutStar &r, int gl)
{
    OutLink l;
    l.regs = __ballot(r.vn > 32) == 0ull;
    l.v[0] = l.regs && gl < r.vn ? p.vpool[r.vo + gl] : 0;
    l.v[1] = l.regs && gl + 16 < r.vn ? p.vpool[r.vo + 16 + gl] : 0;
    return l;
}
// Link vertex lv of this lane's star (every lane of the wave calls it).
__device__ __forceinline__ int out_link(const OutParams &p, const OutStar &r, const OutLink &l, int lv, bool have)
{
    if (!l.regs) return have ? p.vpool[r.vo + lv] : 0;
    const int src = (int)(threadIdx.x & 48) | (lv & 15);
    const int a = __shfl(l.v[0], src, 64), b = __shfl(l.v[1], src, 64);
    return lv < 16 ? a : b;
}

// Decision pass: every owner triangle whose orient3d filter says "lower hull" gets its keep bit and is
// counted for its star; inconclusive ones go to the list for the exact pass.  One triangle in four is
// its star's, so the wave queues them and gathers the points and decides for 64 at a time.  Bound by
// those gathers and the triangle words: 4,194,304 uniform points 0.87 ms, 1.46 with a gather and a
// decision for the owners of each 64 triangles where they stood.  Below OF_WIDE_N stars a wave takes
// four, one after another being as long as the pass then (1,000 points: 12.6 us with 16).
static constexpr int OF_QUEUE = 128, OF_WIDE_N = 1 << 17;
__global__ void __launch_bounds__(256) k_out_flag(OutParams p, uint64_t *list, int64_t cap, int ng)
{
    __shared__ int4 tri_[4][OF_QUEUE]; // a, b, c, t
    __shared__ uint8_t own_[4][OF_QUEUE]; // which of the 16 stars
    __shared__ int kept_[4][16];
    const int lane = threadIdx.x & 63, grp = lane / OUT_GL, gl = lane % OUT_GL, wv = threadIdx.x >> 6;
    int4 *tri = tri_[wv];
    uint8_t *own = own_[wv];
    int *kept = kept_[wv];
    const int w0 = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6), nw = (int)((gridDim.x * blockDim.x) >> 6);
    const int64_t step = 4 * (int64_t)ng * nw;
    OutStar next = out_star_read(p, (int)min(4 * (int64_t)ng * w0, (int64_t)p.n));
    for (int64_t s0 = 4 * (int64_t)ng * w0; s0 < p.n; s0 += step) {
        const OutStar rec = next;
        next = out_star_read(p, (int)min(s0 + step, (int64_t)p.n));
        if (lane < 16) kept[lane] = 0;
        int nq = 0;
        // decides the last n <= 64 of the queue
        auto drain = [&](int n) {
            wave_sync();
            nq -= n;
            int o = 1, st = 0;
            int4 q = make_int4(0, 0, 0, 0);
            if (lane < n) {
                q = tri[nq + lane];
                st = own[nq + lane];
                const double *pp[4] = {p.pts + 3 * (int64_t)q.x, p.pts + 3 * (int64_t)q.y, p.pts + 3 * (int64_t)q.z,
                                       p.pts + 3 * (s0 + st)};
                o = filter_orient3d(pp);
            }
            const int64_t to = (int64_t)__shfl((long long)rec.to, st, 64);
            const bool wide = __shfl(rec.vn, st, 64) >= STAR_WIDE_MIN;
            if (o < 0) {
                *out_keep_word(p, to, q.w, wide) |= out_keep_bit(wide);
                atomicAdd(&kept[st], 1);
            }
            if (__ballot(o == 0)) {
                const long long k = g4d_wave_append(o == 0, &p.cnt[G4D_CNT_OUT_EXACT]);
                if (o == 0 && k < cap) list[k] = ((uint64_t)(uint32_t)(s0 + st) << 32) | (uint32_t)q.w;
            }
            wave_sync();
        };
#pragma unroll 1
        for (int g = 0; g < ng; g++) {
            const int i = 4 * g + grp, s = (int)s0 + i;
            const OutStar r = out_star_of(rec, i);
            const OutLink l = out_link_read(p, r, gl);
            const bool wide = r.vn >= STAR_WIDE_MIN;
            const int tmax = wave_max_i(r.tn);
            for (int t0 = 0; t0 < tmax; t0 += OUT_GL) {
                const int t = t0 + gl;
                int lv[3] = {0, 0, 0};
                if (t < r.tn) star_tri_verts(p.tpool, r.to, t, wide, lv);
                int a[3];
#pragma unroll
                for (int j = 0; j < 3; j++) a[j] = out_link(p, r, l, lv[j], t < r.tn);
                const bool f = t < r.tn && s < a[0] && s < a[1] && s < a[2];
                const uint64_t m = __ballot(f);
                if (f) {
                    const int at = nq + __popcll(m & ((1ull << lane) - 1ull));
                    tri[at] = make_int4(a[0], a[1], a[2], t);
                    own[at] = (uint8_t)i;
                }
                nq += __popcll(m);
                if (nq >= 64) drain(64);
            }
        }
        if (nq > 0) drain(nq);
        if (lane < 4 * ng && s0 + lane < p.n) p.star_tet_count[s0 + lane] = kept[lane];
        wave_sync();
    }
}

// Exact pass over the inconclusive owner triangles: keep (and count) those with orient3d < 0.
__global__ void k_out_exact(OutParams p, const uint64_t *list, int64_t m)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x) {
        const int s = (int)(list[i] >> 32), t = (int)(uint32_t)list[i];
        const bool wide = p.vnum[s] >= STAR_WIDE_MIN;
        const int64_t vo = p.voff[s], to = p.toff[s];
        int lv[3];
        star_tri_verts(p.tpool, to, t, wide, lv);
        const int a = p.vpool[vo + lv[0]], b = p.vpool[vo + lv[1]], cc = p.vpool[vo + lv[2]];
        const double *pp[4] = {p.pts + 3 * (int64_t)a, p.pts + 3 * (int64_t)b, p.pts + 3 * (int64_t)cc,
                               p.pts + 3 * (int64_t)s};
        if (exact_orient3d(pp, p.cnt) < 0) {
            *out_keep_word(p, to, t, wide) |= out_keep_bit(wide);
            atomicAdd(reinterpret_cast<unsigned long long *>(&p.star_tet_count[s]), 1ull);
        }
    }
}

// Write pass, a group of OUT_GL lanes per star: the kept triangles of each star at its scanned offset,
// in triangle order.
__global__ void __launch_bounds__(256) k_out_write(OutParams p)
{
    const int lane = threadIdx.x & 63, grp = lane / OUT_GL, gl = lane % OUT_GL;
    const uint64_t gmask = ((OUT_GL == 64 ? 0ull : (1ull << OUT_GL)) - 1ull) << (grp * OUT_GL);
    const int w0 = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6), nw = (int)((gridDim.x * blockDim.x) >> 6);
    const uint64_t below = ((1ull << lane) - 1ull) & gmask;
    for (int s0 = OUT_NG * w0; s0 < p.n; s0 += OUT_NG * nw) {
        const int s = s0 + grp;
        const bool has = s < p.n;
        const int tn = has ? p.tnum[s] : 0;
        const bool wide = has && p.vnum[s] >= STAR_WIDE_MIN;
        const int64_t vo = has ? p.voff[s] : 0, to = has ? p.toff[s] : 0;
        int64_t k = has ? p.star_tet_off[s] : 0;
        const int tmax = wave_max_i(tn);
        for (int t0 = 0; t0 < tmax; t0 += OUT_GL) {
            const int t = t0 + gl;
            const bool keep = t < tn && (*out_keep_word(p, to, t, wide) & out_keep_bit(wide));
            const uint64_t m = __ballot(keep);
            if (keep) {
                int lv[3];
                star_tri_verts(p.tpool, to, t, wide, lv);
                int4 q;
                q.x = p.vpool[vo + lv[0]];
                q.y = p.vpool[vo + lv[1]];
                q.z = p.vpool[vo + lv[2]];
                q.w = s;
                if (p.perm) q = make_int4(p.perm[q.x], p.perm[q.y], p.perm[q.z], p.perm[q.w]);
                reinterpret_cast<int4 *>(p.tets)[k + __popcll(m & below)] = q;
            }
            k += __popcll(m & gmask);
        }
    }
}

hipError_t launch_out_flag(const OutParams &p, uint64_t *list, int64_t cap, hipStream_t s)
{
    // 16 stars a wave, four where that would leave the chip short of waves
    const int ng = p.n >= OF_WIDE_N ? 4 : 1;
    hipLaunchKernelGGL(k_out_flag, dim3(g4d_blocks(p.n, 16 * ng, 16384)), dim3(256), 0, s, p, list, cap, ng);
    return hipGetLastError();
}

hipError_t launch_out_exact(const OutParams &p, const uint64_t *list, int64_t m, hipStream_t s)
{
    if (m <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_out_exact, dim3(g4d_blocks(m, 64, 1024)), dim3(64), 0, s, p, list, m);
    return hipGetLastError();
}

hipError_t launch_out_write(const OutParams &p, hipStream_t s)
{
    hipLaunchKernelGGL(k_out_write, dim3(g4d_blocks((int64_t)p.n * 64, 256, 16384)), dim3(256), 0, s, p);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------
// Star consistency (kerCheckStarConsistency / checkIfStarHasTriangle, GD/GDelaunay/
// GDelKernels.cu:1193-1271): link triangle (a, b, c) of star s stands for tetrahedron
// {s, a, b, c}, so star a must hold a link triangle with the vertex set {s, b, c}, and likewise
// stars b and c.  Vertex sets are compared without orientation, as the reference does.
// ------------------------------------------------------------------------------------

// Does star u hold a link triangle with vertex set {x, y, z} (global ids)?
__device__ bool star_has_triangle(const OutParams &p, int u, int x, int y, int z)
{
    if (u < 0 || u >= p.n) return false;
    const int vn = p.vnum[u], tn = p.tnum[u];
    const int64_t vo = p.voff[u], to = p.toff[u];
    int lx = -1, ly = -1, lz = -1;
    for (int v = 0; v < vn; v++) {
        const int g = p.vpool[vo + v];
        lx = g == x ? v : lx;
        ly = g == y ? v : ly;
        lz = g == z ? v : lz;
    }
    if (lx < 0 || ly < 0 || lz < 0) return false;
    const bool wide = vn >= STAR_WIDE_MIN;
    for (int t = 0; t < tn; t++) {
        int lv[3];
        star_tri_verts(p.tpool, to, t, wide, lv);
        const bool hx = lv[0] == lx || lv[1] == lx || lv[2] == lx;
        const bool hy = lv[0] == ly || lv[1] == ly || lv[2] == ly;
        const bool hz = lv[0] == lz || lv[1] == lz || lv[2] == lz;
        if (hx && hy && hz) return true;
    }
    return false;
}

// One half-wave per star, one lane per link triangle; cnt[G4D_CNT_APPEND5] counts the link
// triangles that fail, cnt[G4D_CNT_APPEND4] those checked.
__global__ void __launch_bounds__(256) k_star_consistency(OutParams p)
{
    const int lane = threadIdx.x & 63, half = lane >> 5, hl = lane & 31;
    const int w0 = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6), nw = (int)((gridDim.x * blockDim.x) >> 6);
    int bad = 0, seen = 0;
    for (int s0 = 2 * w0; s0 < p.n; s0 += 2 * nw) {
        const int s = s0 + half;
        const bool has = s < p.n;
        const int tn = has ? p.tnum[s] : 0;
        const bool wide = has && p.vnum[s] >= STAR_WIDE_MIN;
        const int64_t vo = has ? p.voff[s] : 0, to = has ? p.toff[s] : 0;
        const int tmax = max(tn, __shfl_xor(tn, 32, 64));
        for (int t0 = 0; t0 < tmax; t0 += 32) {
            const int t = t0 + hl;
            if (t >= tn) continue;
            int lv[3];
            star_tri_verts(p.tpool, to, t, wide, lv);
            const int g[3] = {p.vpool[vo + lv[0]], p.vpool[vo + lv[1]], p.vpool[vo + lv[2]]};
            bool ok = true;
            for (int i = 0; i < 3 && ok; i++) ok = star_has_triangle(p, g[i], s, g[(i + 1) % 3], g[(i + 2) % 3]);
            seen++;
            bad += ok ? 0 : 1;
        }
    }
    const int wb = g4d_wave_sum(bad), ws = g4d_wave_sum(seen);
    if (lane == 0) {
        if (wb) atomicAdd(&p.cnt[G4D_CNT_APPEND5], (unsigned long long)wb);
        atomicAdd(&p.cnt[G4D_CNT_APPEND4], (unsigned long long)ws);
    }
}

hipError_t launch_star_consistency(const OutParams &p, hipStream_t s)
{
    if (p.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_star_consistency, dim3(g4d_blocks((int64_t)p.n * 32, 256, 16384)), dim3(256), 0, s, p);
    return hipGetLastError();
}

__device__ __forceinline__ void face_of(const int *tt, int i, int *f)
{
    int q = 0;
#pragma unroll
    for (int j = 0; j < 4; j++)
        if (j != i) f[q++] = tt[j];
    int tmp;
    if (f[0] > f[1]) { tmp = f[0]; f[0] = f[1]; f[1] = tmp; }
    if (f[1] > f[2]) { tmp = f[1]; f[1] = f[2]; f[2] = tmp; }
    if (f[0] > f[1]) { tmp = f[0]; f[0] = f[1]; f[1] = tmp; }
}

__global__ void k_adjacency(const int *tets, int64_t nt, int *opp, uint32_t *table, uint64_t mask,
                            unsigned long long *cnt)
{
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < nt; t += (int64_t)gridDim.x * blockDim.x) {
        const int *tt = tets + 4 * t;
        for (int i = 0; i < 4; i++) {
            int f[3];
            face_of(tt, i, f);
            uint64_t h = (uint64_t)(uint32_t)f[0] * 0x9E3779B97F4A7C15ull ^ (uint64_t)(uint32_t)f[1] * 0xC2B2AE3D27D4EB4Full ^
                         (uint64_t)(uint32_t)f[2] * 0x165667B19E3779F9ull;
            h ^= h >> 29;
            h *= 0xBF58476D1CE4E5B9ull;
            h ^= h >> 32;
            uint64_t slot = h & mask;
            const uint32_t mine = (uint32_t)((t << 2) | i) + 1u;
            for (uint64_t probe = 0; probe <= mask; probe++) {
                uint32_t cur = atomicCAS(&table[slot], 0u, mine);
                if (cur == 0u) break; // first occurrence stored
                const int64_t t2 = (int64_t)((cur - 1u) >> 2);
                const int i2 = (int)((cur - 1u) & 3u);
                int g[3];
                face_of(tets + 4 * t2, i2, g);
                if (g[0] == f[0] && g[1] == f[1] && g[2] == f[2]) {
                    if (atomicCAS(&opp[4 * t2 + i2], -1, (int)t) != -1)
                        atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_FACE);
                    opp[4 * t + i] = (int)t2;
                    break;
                }
                slot = (slot + 1) & mask;
            }
        }
    }
}

__device__ __forceinline__ uint64_t face_hash(const int *f)
{
    uint64_t h = (uint64_t)(uint32_t)f[0] * 0x9E3779B97F4A7C15ull ^ (uint64_t)(uint32_t)f[1] * 0xC2B2AE3D27D4EB4Full ^
                 (uint64_t)(uint32_t)f[2] * 0x165667B19E3779F9ull;
    h ^= h >> 29;
    h *= 0xBF58476D1CE4E5B9ull;
    h ^= h >> 32;
    return h;
}

// Tiled variant for the pipeline's output, whose tetrahedra come grouped by owner star in
// Morton order: a work-group first pairs the faces of its ADJ_TETS consecutive tetrahedra in an
// LDS hash table (most interior faces have both tetrahedra in the same tile), and only the
// faces left unpaired go through the global table as in k_adjacency.  512-tetrahedron tiles
// (24.6 KB of LDS) measured faster than 1,024 and 2,048 at 4M points: residency wins over the
// extra global inserts of the smaller tiles.
static constexpr int ADJ_TETS = 512;
static constexpr int ADJ_HASH = 4096;

__global__ void __launch_bounds__(256) k_adjacency_tiled(const int *tets, int64_t nt, int *opp, uint32_t *table,
                                                         uint64_t mask, unsigned long long *cnt)
{
    __shared__ int4 lt[ADJ_TETS];
    __shared__ uint32_t tab[ADJ_HASH];
    __shared__ uint32_t done[ADJ_TETS * 4 / 32];
    for (int64_t tile = blockIdx.x; tile * ADJ_TETS < nt; tile += gridDim.x) {
        const int64_t t0 = tile * ADJ_TETS;
        const int nloc = (int)(nt - t0 < ADJ_TETS ? nt - t0 : ADJ_TETS);
        for (int k = threadIdx.x; k < nloc; k += blockDim.x) lt[k] = reinterpret_cast<const int4 *>(tets)[t0 + k];
        for (int k = threadIdx.x; k < ADJ_HASH; k += blockDim.x) tab[k] = 0u;
        for (int k = threadIdx.x; k < ADJ_TETS * 4 / 32; k += blockDim.x) done[k] = 0u;
        __syncthreads();
        for (int lf = threadIdx.x; lf < 4 * nloc; lf += blockDim.x) {
            const int k = lf >> 2, i = lf & 3;
            int f[3];
            face_of(reinterpret_cast<const int *>(&lt[k]), i, f);
            uint32_t h = (uint32_t)face_hash(f) & (ADJ_HASH - 1);
            for (int probe = 0; probe < ADJ_HASH; probe++) { // fewer faces than slots: ends
                const uint32_t cur = atomicCAS(&tab[h], 0u, (uint32_t)lf + 1u);
                if (cur == 0u) break;
                const int other = (int)cur - 1;
                int g[3];
                face_of(reinterpret_cast<const int *>(&lt[other >> 2]), other & 3, g);
                if (g[0] == f[0] && g[1] == f[1] && g[2] == f[2]) {
                    const uint32_t was = atomicOr(&done[other >> 5], 1u << (other & 31));
                    if (was & (1u << (other & 31))) atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_FACE);
                    atomicOr(&done[lf >> 5], 1u << (lf & 31));
                    opp[4 * (t0 + (other >> 2)) + (other & 3)] = (int)(t0 + k);
                    opp[4 * (t0 + k) + i] = (int)(t0 + (other >> 2));
                    break;
                }
                h = (h + 1) & (ADJ_HASH - 1);
            }
        }
        __syncthreads();
        for (int lf = threadIdx.x; lf < 4 * nloc; lf += blockDim.x) {
            if (done[lf >> 5] & (1u << (lf & 31))) continue;
            const int k = lf >> 2, i = lf & 3;
            const int64_t t = t0 + k;
            int f[3];
            face_of(reinterpret_cast<const int *>(&lt[k]), i, f);
            uint64_t slot = face_hash(f) & mask;
            const uint32_t mine = (uint32_t)((t << 2) | i) + 1u;
            for (uint64_t probe = 0; probe <= mask; probe++) {
                const uint32_t cur = atomicCAS(&table[slot], 0u, mine);
                if (cur == 0u) break;
                const int64_t t2 = (int64_t)((cur - 1u) >> 2);
                const int i2 = (int)((cur - 1u) & 3u);
                int g[3];
                face_of(tets + 4 * t2, i2, g);
                if (g[0] == f[0] && g[1] == f[1] && g[2] == f[2]) {
                    if (atomicCAS(&opp[4 * t2 + i2], -1, (int)t) != -1)
                        atomicOr(&cnt[G4D_CNT_ERROR], (unsigned long long)G4D_DEV_ERR_FACE);
                    opp[4 * t + i] = (int)t2;
                    break;
                }
                slot = (slot + 1) & mask;
            }
        }
        __syncthreads();
    }
}

hipError_t launch_adjacency_tiled(const int *tets, int64_t nt, int *opp, uint32_t *table, int64_t table_size,
                                  unsigned long long *cnt, hipStream_t s)
{
    if (nt <= 0) return hipSuccess;
    HIP_CHECK_RET(hipMemsetAsync(table, 0, sizeof(uint32_t) * (size_t)table_size, s));
    HIP_CHECK_RET(hipMemsetAsync(opp, 0xff, sizeof(int) * 4 * (size_t)nt, s));
    const int64_t tiles = (nt + ADJ_TETS - 1) / ADJ_TETS;
    hipLaunchKernelGGL(k_adjacency_tiled, dim3((unsigned)(tiles < 65536 ? tiles : 65536)), dim3(256), 0, s, tets, nt,
                       opp, table, (uint64_t)(table_size - 1), cnt);
    return hipGetLastError();
}

hipError_t launch_adjacency(const int *tets, int64_t nt, int *opp, uint32_t *table, int64_t table_size,
                            unsigned long long *cnt, hipStream_t s)
{
    if (nt <= 0) return hipSuccess;
    HIP_CHECK_RET(hipMemsetAsync(table, 0, sizeof(uint32_t) * (size_t)table_size, s));
    HIP_CHECK_RET(hipMemsetAsync(opp, 0xff, sizeof(int) * 4 * (size_t)nt, s));
    hipLaunchKernelGGL(k_adjacency, dim3(g4d_blocks(nt, 256, 65536)), dim3(256), 0, s, tets, nt, opp, table,
                       (uint64_t)(table_size - 1), cnt);
    return hipGetLastError();
}

__global__ void k_gather_i64(const int64_t *a, const int64_t *idx, int64_t m, int64_t *out)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x)
        out[i] = a[idx[i]];
}

hipError_t launch_gather_i64(const int64_t *a, const int64_t *idx, int64_t m, int64_t *out, hipStream_t s)
{
    if (m <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather_i64, dim3(g4d_blocks(m, 256, 65536)), dim3(256), 0, s, a, idx, m, out);
    return hipGetLastError();
}

__global__ void k_batch_localize(int *tets, int *opp, int64_t nt, const int *pt_set, const int64_t *pt_off,
                                 const int64_t *tet_off, const int *perm)
{
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < nt; t += (int64_t)gridDim.x * blockDim.x) {
        const int st = pt_set[tets[4 * t]];
        const int base = (int)pt_off[st];
        for (int i = 0; i < 4; i++) tets[4 * t + i] = perm[tets[4 * t + i]] - base;
        if (opp)
            for (int i = 0; i < 4; i++) {
                const int o = opp[4 * t + i];
                opp[4 * t + i] = o < 0 ? -1 : (int)(o - tet_off[st]);
            }
    }
}

hipError_t launch_batch_localize(int *tets, int *opp, int64_t nt, const int *pt_set, const int64_t *pt_off,
                                 const int64_t *tet_off, const int *perm, hipStream_t s)
{
    if (nt <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_batch_localize, dim3(g4d_blocks(nt, 256, 65536)), dim3(256), 0, s, tets, opp, nt, pt_set,
                       pt_off, tet_off, perm);
    return hipGetLastError();
}

} // namespace g4d
