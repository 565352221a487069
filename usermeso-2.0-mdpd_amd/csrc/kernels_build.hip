// Neighbor-rebuild phase of the mdpd355 engine: periodic wrap, cell keys,
// counting sort by cell + per-particle rank of the sub-bin key inside its
// cell, gather into the other buffer, per-particle neighbor-row build, commit.
//
// Replaces, for one or many periodic boxes at once:
//   MesoAtom::sort_local            src/USER-MESO/atom_meso.cu:271-387
//   MesoNeighbor::binning_meso      src/USER-MESO/neighbor_meso.cu:390-683
//   MesoNeighbor::full_bin_meso     src/USER-MESO/neigh_build_meso.cu:17-127,286-449
//   Domain::pbc + MesoComm::borders (on-device periodic images instead of ghosts)
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace mdpd {

#pragma clang fp contract(off)

// The neighbor-row build of a pool walks a worklist of the cells to list
// (k_scan_apply appends them); one system (the plain path) keeps one wave
// per cell slot: its slots are few and the list would only add its own cost.
__host__ __device__ inline bool nlist_listed(const PoolDev &P) { return !P.one; }

// particle at p with packed image flags img wrapped into the box (Domain::pbc
// in FP32)
__device__ inline void wrap_particle(const SysDev *d, float4 &p, int &img)
{
    float c[3] = {p.x, p.y, p.z};
    int im[3] = {(img & 1023) - 512, ((img >> 10) & 1023) - 512, ((img >> 20) & 1023) - 512};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float flo = d->lo[a], fhi = d->hi[a], prd = d->L[a];
        float v = c[a];
        if (v < flo) { v = v + prd; im[a] -= 1; }
        if (v >= fhi) { v = v - prd; v = fmaxf(v, flo); im[a] += 1; }
        c[a] = v;
    }
    p.x = c[0]; p.y = c[1]; p.z = c[2];
    img = ((im[0] + 512) & 1023) | (((im[1] + 512) & 1023) << 10) | (((im[2] + 512) & 1023) << 20);
}

// bin coordinates b of a wrapped position and its 12-bit sub-bin Morton code
__device__ inline uint32_t particle_bins(const SysDev *d, const float4 &p, int b[3])
{
    const float c[3] = {p.x, p.y, p.z};
    uint32_t sub[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        // bin: (int)((x - lo) * bininv + 1.0), FP64, clamped to the interior
        const double t = ((double)c[a] - d->lo_d[a]) * d->bininv_d[a];
        const double u = t + 1.0;
        int bb = (int)u;
        bb = bb > d->mbin[a] - 2 ? d->mbin[a] - 2 : bb;
        bb = bb < 1 ? 1 : bb;
        b[a] = bb;
        // sub-bin: (x - (bin-1) * binsize) * 16 * bininv (atom_meso.cu:298-300)
        const double off = (double)(uint32_t)(bb - 1) * d->binsize_d[a];
        const double rel = (double)c[a] - off;
        const double sc = rel * (16.0 * d->bininv_d[a]);
        int ss = (int)sc;
        ss = ss > 15 ? 15 : ss;
        ss = ss < 0 ? 0 : ss;
        sub[a] = (uint32_t)ss;
    }
    // four bits per axis, bit i to bit 3 i (+ axis)
    uint32_t z = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
        z |= ((sub[a] & 1) | (sub[a] & 2) << 2 | (sub[a] & 4) << 4 | (sub[a] & 8) << 6) << a;
    return z;
}

// --------------------------------------------------------------------------
// K1: wrap into the box (Domain::pbc in FP32), reference sort key, sub-cell
// slot (cell slot * SUBCELLS + top bits of the sub-bin key), arrival rank
// inside the sub-cell.  `commit`: the commit of the pass before is still to
// come (the scan makes it, when nobody here reads its fields any more), so
// the decision it is going to make and the buffer it makes current are worked
// out here, and the decision goes to d->due for the scan's workgroups.
// --------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_keys(PoolDev P, int commit)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) {
        P.work_count[0] = 0;                              // this rebuild's worklist starts empty
        // one system: the row build's waves read this word, not the flag that
        // their commit clears
        if (P.one) P.work_count[1] = due_after(P.sys, commit) ? 1 : 0;
    }
    if (i >= P.nact) return;
    const int s = P.one ? 0 : P.wave_sys[i >> 6];
    if (s < 0) return;
    SysDev *d = P.sys + s;
    const bool due = due_after(d, commit);
    if (i == d->part_base) d->due = due ? 1 : 0;
    if (!due) return;
    // the wave stays whole (the slot's run below is found across lanes);
    // lanes past the system's last particle only take part in that
    const bool valid = i < d->part_base + d->n;
    int gc = -1;
    if (valid) {
    const int cur = d->sel ^ (commit && !d->overflow ? 1 : 0), cura = d->sela;
    float4 p = P.pos[cur][i];
    int img = P.image[cura][i];
    wrap_particle(d, p, img);
    P.pos[cur][i] = p;
    P.image[cura][i] = img;
    int b[3];
    const uint32_t z2 = particle_bins(d, p, b);
    const int lin = (b[0] - 1) + d->nb[0] * ((b[1] - 1) + d->nb[1] * (b[2] - 1));
    gc = (d->cell_base + P.cell_rank[d->cell_base + lin]) * SUBCELLS + (int)(z2 >> SUBCELL_SHIFT);
    P.pcell[i] = gc;
    P.psub[i] = (int)z2;
    }
    // arrival slots: the particles are still nearly in the last build's
    // order, so neighboring lanes mostly share a sub-cell; each run of equal
    // sub-cells takes its slots with one atomic (the order of arrival inside
    // a sub-cell does not matter: the rank in k_sortgather decides)
    const int lane = threadIdx.x & 63;
    const int prev = __shfl_up(gc, 1, 64);
    const bool head = valid && (lane == 0 || prev != gc);
    const uint64_t heads = __builtin_amdgcn_ballot_w64(head);
    const uint64_t below = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);    // lanes 0..lane
    const uint64_t hb = heads & below;
    const int h = hb ? 63 - __clzll(hb) : 0;                                // this lane's run head
    const uint64_t later = heads & ~below;
    const int nvalid = __popcll(__builtin_amdgcn_ballot_w64(valid));
    const int next = later ? min(__ffsll((long long)later) - 1, nvalid) : nvalid;
    int base = 0;
    if (head) base = atomicAdd(P.cell_count + gc, next - lane);
    base = __shfl(base, h, 64);
    if (valid) P.pslot[i] = base + (lane - h);
}

// --------------------------------------------------------------------------
// K2: exclusive scan of sub-cell counts in (cell Morton rank, sub-cell)
// order, per system, from its first particle slot; clears the counts for the
// next rebuild.  Chunks of SCAN_CH counts, two launches without waits:
//   k_scan_sums   per chunk: its total, to chunk_sum[first cell slot + chunk]
//   k_scan_apply  per chunk: exclusive scan of its counts from the sum of the
//                 totals before it (each workgroup adds them up itself: one
//                 load per thread up to a million sub-cells, where a launch
//                 between the two cost a pass 3 us and more); in a pool also
//                 each cell's particle range by linear cell id and the
//                 worklist of occupied cells for the row build
// Grid (G, nsys): workgroup g of a system takes chunks g, g + G, ...
// --------------------------------------------------------------------------
constexpr int SCAN_BLK = 256, SCAN_PER = 16, SCAN_CH = SCAN_BLK * SCAN_PER;

// exclusive scan of one value per thread over the workgroup; returns the
// workgroup total through *total
__device__ inline int block_excl_scan(int x, int *wsum, int *total)
{
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int incl = wave_incl_scan(x);
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    int before = 0, all = 0;
    for (int k = 0; k < SCAN_BLK / 64; ++k) {
        const int y = wsum[k];
        before += k < w ? y : 0;
        all += y;
    }
    __syncthreads();
    *total = all;
    return before + incl - x;
}

__global__ void __launch_bounds__(SCAN_BLK) k_scan_sums(PoolDev P, int commit, int split, int seeded)
{
    const SysDev *d = P.sys + blockIdx.y;
    // a finished system is not due; the commit ends no system that is
    const bool due = d->active && d->due;
    if (commit && blockIdx.x == 0 && threadIdx.x == 0) commit_system(P, blockIdx.y, commit, split, seeded);
    if (!due) return;
    __shared__ int wsum[SCAN_BLK / 64];
    const int nc = d->ncell * SUBCELLS, base = d->cell_base * SUBCELLS;
    for (int c0 = blockIdx.x * SCAN_CH; c0 < nc; c0 += gridDim.x * SCAN_CH) {
        // clamped loads, all in flight; entries past the end count 0
        int sum = 0;
#pragma unroll
        for (int u = 0; u < SCAN_PER; ++u) {
            const int c = c0 + u * SCAN_BLK + (int)threadIdx.x;
            const int v = P.cell_count[base + min(c, nc - 1)];
            sum += c < nc ? v : 0;
        }
        int total;
        block_excl_scan(sum, wsum, &total);
        if (threadIdx.x == 0) P.chunk_sum[d->cell_base + c0 / SCAN_CH] = total;
    }
}

__global__ void __launch_bounds__(SCAN_BLK) k_scan_apply(PoolDev P)
{
    const SysDev *d = P.sys + blockIdx.y;
    if (!d->active || !d->stale) return;
    __shared__ int buf[SCAN_CH];
    __shared__ int wsum[SCAN_BLK / 64];
    __shared__ int s_wl[SCAN_BLK / 64 + 1];                // worklist: wave counts, the chunk's base
    const int nc = d->ncell * SUBCELLS, base = d->cell_base * SUBCELLS;
    const int t = threadIdx.x;
    for (int c0 = blockIdx.x * SCAN_CH; c0 < nc; c0 += gridDim.x * SCAN_CH) {
        int before = 0;
        for (int k = t; k < c0 / SCAN_CH; k += SCAN_BLK) before += P.chunk_sum[d->cell_base + k];
        // coalesced load into LDS (counts cleared), SCAN_PER consecutive
        // counts per thread, workgroup scan, coalesced store
#pragma unroll
        for (int u = 0; u < SCAN_PER; ++u) {
            const int c = c0 + u * SCAN_BLK + t;
            const int v = P.cell_count[base + min(c, nc - 1)];
            buf[u * SCAN_BLK + t] = c < nc ? v : 0;
        }
#pragma unroll
        for (int u = 0; u < SCAN_PER; ++u) {
            const int c = c0 + u * SCAN_BLK + t;
            if (c < nc) P.cell_count[base + c] = 0;
        }
        __syncthreads();
        int v[SCAN_PER], sum = 0;
        for (int k = 0; k < SCAN_PER; ++k) { v[k] = buf[t * SCAN_PER + k]; sum += v[k]; }
        static_assert(SCAN_PER % SUBCELLS == 0 && SCAN_CH % SUBCELLS == 0, "whole cells per thread");
        constexpr int CPT = SCAN_PER / SUBCELLS;                 // cells per thread
        int cst[CPT];                                            // first particle of each
        int total;
        int run = d->part_base + block_excl_scan(sum, wsum, &total);
        block_excl_scan(before, wsum, &total);
        run += total;
        if (t == 0 && c0 + SCAN_CH >= nc) P.cell_start[base + nc] = d->part_base + d->n;
#pragma unroll
        for (int k = 0; k < SCAN_PER; ++k) {
            if (k % SUBCELLS == 0) cst[k / SUBCELLS] = run;
            buf[t * SCAN_PER + k] = run;
            run += v[k];
        }
        // pools: every cell's particle range by linear cell id, and the cells
        // holding particles appended to the neighbor-row worklist with their
        // system, coordinates and range, in cell-slot order within the chunk
        // (one atomic per workgroup and chunk: same-address atomics
        // serialize); counts past the system's end are zero and not listed
        if (nlist_listed(P)) {
            const int cell0 = d->cell_base + (c0 + t * SCAN_PER) / SUBCELLS;
            int xyz[CPT], full = 0;
#pragma unroll
            for (int q = 0; q < CPT; ++q) {
                const bool in = c0 + t * SCAN_PER + q * SUBCELLS < nc;
                int m = 0;
#pragma unroll
                for (int u = 0; u < SUBCELLS; ++u) m += v[q * SUBCELLS + u];
                xyz[q] = in ? P.cell_xyz[cell0 + q] : 0;
                if (in) {
                    const int lin = (xyz[q] & 1023) + d->nb[0] * (((xyz[q] >> 10) & 1023) + d->nb[1] * ((xyz[q] >> 20) & 1023));
                    P.cell_lse[d->cell_base + lin] = make_int2(cst[q], cst[q] + m);
                }
                full |= (m > 0 ? 1 : 0) << q;
            }
            const int cnt = __popc(full);
            const int lane = t & 63, wv = t >> 6;
            const int incl = wave_incl_scan(cnt);
            if (lane == 63) s_wl[wv] = incl;
            __syncthreads();
            if (t == 0) {
                int tot = 0;
                for (int k = 0; k < SCAN_BLK / 64; ++k) tot += s_wl[k];
                s_wl[SCAN_BLK / 64] = tot > 0 ? atomicAdd(P.work_count, tot) : 0;
            }
            __syncthreads();
            int o = s_wl[SCAN_BLK / 64] + incl - cnt;
            for (int k = 0; k < wv; ++k) o += s_wl[k];
#pragma unroll
            for (int q = 0; q < CPT; ++q) {
                if (full >> q & 1) {
                    int m = 0;
#pragma unroll
                    for (int u = 0; u < SUBCELLS; ++u) m += v[q * SUBCELLS + u];
                    P.cell_work[o++] = make_int4((int)blockIdx.y, xyz[q], cst[q], cst[q] + m);
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < SCAN_PER; ++u) {
            const int k = u * SCAN_BLK + t;
            if (c0 + k < nc) P.cell_start[base + c0 + k] = buf[k];
        }
        __syncthreads();
    }
}

// --------------------------------------------------------------------------
// The same scan for one system in one launch: workgroup g adds up all the
// counts before its chunk itself, which costs it reads (four chunks a round:
// the last of the 14 workgroups for the 54,000 sub-cells of a 97,000-particle
// slab makes four rounds) where k_scan_sums costs a launch, 1.6 us idle and 4.7
// us working.  Other workgroups may still read a chunk's counts, so k_scatter
// clears them.
// --------------------------------------------------------------------------
constexpr int SCAN1_BLK = 1024, SCAN1_CH = SCAN1_BLK * 4;
constexpr int SCAN1_MAX = 40;          // chunks: past that the last workgroup's reads (10 rounds) cost the launches saved

__global__ void __launch_bounds__(SCAN1_BLK) k_scan_one(PoolDev P, int commit, int split, int seeded)
{
    const SysDev *d = P.sys;
    const bool due = P.work_count[1] != 0;
    if (commit && blockIdx.x == 0 && threadIdx.x == 0) commit_system(P, 0, commit, split, seeded);
    if (!due) return;
    __shared__ int s_before[SCAN1_BLK / WAVE], s_own[SCAN1_BLK / WAVE];
    const int nc = d->ncell * SUBCELLS;                    // a multiple of four
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int c0 = blockIdx.x * SCAN1_CH, c = c0 + 4 * t;
    const int4 *cnt4 = (const int4 *)P.cell_count;
    int before = 0;
    for (int k = 0; k < c0; k += 4 * SCAN1_CH) {
        int4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            v[u] = k + u * SCAN1_CH < c0 ? cnt4[(k + u * SCAN1_CH) / 4 + t] : make_int4(0, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 4; ++u) before += v[u].x + v[u].y + v[u].z + v[u].w;
    }
    const int4 own = c < nc ? cnt4[c / 4] : make_int4(0, 0, 0, 0);
    const int sum = own.x + own.y + own.z + own.w;
    const int incl = wave_incl_scan(sum);
    before = wave_sum(before);
    if (lane == 63) {
        s_own[wv] = incl;
        s_before[wv] = before;
    }
    __syncthreads();
    int run = d->part_base + incl - sum;
    for (int k = 0; k < SCAN1_BLK / WAVE; ++k) run += s_before[k] + (k < wv ? s_own[k] : 0);
    if (c < nc) {
        const int4 st = make_int4(run, run + own.x, run + own.x + own.y, run + own.x + own.y + own.z);
        ((int4 *)P.cell_start)[c / 4] = st;
        if (c + 4 == nc) P.cell_start[nc] = d->part_base + d->n;
    }
}

// --------------------------------------------------------------------------
// K3: scatter particle indices into their sub-cell segments (arrival order),
// the sub-bin key beside each (in cl, for the ranks of k_sortgather); with
// `clear` the sub-cell counts of the one system are cleared here.
// --------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_scatter(PoolDev P, int clear)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.nact) return;
    const int s = P.one ? 0 : P.wave_sys[i >> 6];
    if (s < 0) return;
    SysDev *d = P.sys + s;
    if (!d->active || !d->stale) return;
    if (clear)
        for (int c = i; c < d->ncell * SUBCELLS; c += P.nact) P.cell_count[c] = 0;
    if (i >= d->part_base + d->n) return;
    const int f = P.cell_start[P.pcell[i]] + P.pslot[i];
    P.tmp[f] = i;
    P.cl[f] = P.psub[i];
}

// --------------------------------------------------------------------------
// K4: one thread per particle, by its previous slot i: its rank in its
// sub-cell by (sub-bin key, previous index) -- with the sub-cells in key
// order this is the stable sort of the 2-level Morton key -- gives its sorted
// slot; every per-particle array moves there in the other buffer (loads in
// the previous order, issued while the rank is found; stores scattered).
// --------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_sortgather(PoolDev P)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.nact) return;
    const int s = P.one ? 0 : P.wave_sys[i >> 6];
    if (s < 0) return;
    const SysDev *d = P.sys + s;
    if (!d->active || !d->stale) return;
    if (i >= d->part_base + d->n) return;
    const int cell = P.pcell[i];
    const int key = P.psub[i];
    const int cur = d->sel, cura = d->sela;
    const float4 p = P.pos[cur][i];
    float4 v = P.vel[cur][i];
    const int tg = P.tag[cura][i];
    const int mk = P.mask[cura][i], og = P.origin[cura][i], im = P.image[cura][i];
    const float ph = P.phi[cura][i];
    const int start = P.cell_start[cell], end = P.cell_start[cell + 1];
    // four members' keys in flight per round trip (loads clamped to the
    // segment, members past its end not counted)
    int rank = 0;
    for (int g0 = start; g0 < end; g0 += 4) {
        int kg[4], jg[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int g = min(g0 + u, end - 1);
            kg[u] = P.cl[g];
            jg[u] = P.tmp[g];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            rank += g0 + u < end && ((kg[u] < key) || (kg[u] == key && jg[u] < i));
    }
    const int dst = start + rank;
    if (d->phase == PH_FRESH) {
        // a newly loaded system: signatures of its first force pass
        const uint32_t sg = d->style == STYLE_MDPD ? sig_mdpd(tg, d->seed_cur)
                                                   : sig_dpd(tg, d->seed_cur, v.x, v.y, v.z);
        v.w = __uint_as_float(sg);
    }
    P.pos[cur ^ 1][dst] = p;
    P.vel[cur ^ 1][dst] = v;
    P.xhold[dst] = p;
    P.tag[cura ^ 1][dst] = tg;
    P.mask[cura ^ 1][dst] = mk;
    P.origin[cura ^ 1][dst] = og;
    P.image[cura ^ 1][dst] = im;
    P.phi[cura ^ 1][dst] = ph;
}

// --------------------------------------------------------------------------
// K1 to K4 for one small system in one launch: a workgroup holds the sub-cell
// counts and the sort keys in LDS, each thread up to SORT1_PER particles.  A
// step without a re-sort saves the idle time of three launches, a step with
// one pays ~340 instructions per particle on one CU (sort_one_limit weighs the
// two).  `commit`: the previous step's
// commit (COMMIT_DECIDE) is made here first, one launch of 2.7 us less.
// --------------------------------------------------------------------------
constexpr int SORT1_BLK = 1024, SORT1_PER = 10, SORT1_N = SORT1_BLK * SORT1_PER, SORT1_SUB = 16384;

template <int PER>
__global__ void __launch_bounds__(SORT1_BLK) k_sort_one(PoolDev P, int commit, int seeded)
{
    __shared__ __align__(16) int s_cnt[SORT1_SUB + 4];     // counts, then first slots
    __shared__ uint32_t s_key[SORT1_N];                    // sub-bin key << 14 | previous index, by sub-cell
    __shared__ int s_wave[SORT1_BLK / WAVE], s_now[3];      // stale, sel, sela after the commit
    SysDev *d = P.sys;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    if (t == 0) {
        if (commit) commit_system(P, 0, commit, 0, seeded);
        s_now[0] = d->active && d->stale;
        s_now[1] = d->sel;
        s_now[2] = d->sela;
    }
    __syncthreads();
    const int stale = s_now[0], cur = s_now[1], cura = s_now[2];
    if (t == 0) P.work_count[1] = stale;                   // the row build's flag
    if (!stale) return;
    const int n = d->n, nsub = d->ncell * SUBCELLS;        // part_base and cell_base are 0
    for (int c = 4 * t; c < nsub; c += 4 * SORT1_BLK) *(int4 *)(s_cnt + c) = make_int4(0, 0, 0, 0);
    __syncthreads();
    uint32_t pk[PER];                                      // sub-cell << 12 | sub-bin key
    int slot[PER];                                         // arrival rank in the sub-cell
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int i = k * SORT1_BLK + t;
        if (k * SORT1_BLK >= n) break;
        if (i < n) {
            float4 p = P.pos[cur][i];
            int img = P.image[cura][i], b[3];
            wrap_particle(d, p, img);
            const uint32_t z2 = particle_bins(d, p, b);
            const int lin = (b[0] - 1) + d->nb[0] * ((b[1] - 1) + d->nb[1] * (b[2] - 1));
            const int gc = P.cell_rank[lin] * SUBCELLS + (int)(z2 >> SUBCELL_SHIFT);
            pk[k] = (uint32_t)gc << 12 | z2;
            slot[k] = atomicAdd(s_cnt + gc, 1);
        }
    }
    __syncthreads();
    // exclusive scan, sixteen counts per thread
    int4 v[4];
    int sum = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int c = 16 * t + 4 * u;
        v[u] = c < nsub ? *(const int4 *)(s_cnt + c) : make_int4(0, 0, 0, 0);
        sum += v[u].x + v[u].y + v[u].z + v[u].w;
    }
    const int incl = wave_incl_scan(sum);
    if (lane == 63) s_wave[wv] = incl;
    __syncthreads();
    int run = incl - sum;
    for (int k = 0; k < wv; ++k) run += s_wave[k];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int c = 16 * t + 4 * u;
        const int4 st = make_int4(run, run + v[u].x, run + v[u].x + v[u].y, run + v[u].x + v[u].y + v[u].z);
        run = st.w + v[u].w;
        if (c < nsub) {
            *(int4 *)(s_cnt + c) = st;
            ((int4 *)P.cell_start)[c / 4] = st;
        }
    }
    if (t == 0) s_cnt[nsub] = P.cell_start[nsub] = n;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int i = k * SORT1_BLK + t;
        if (k * SORT1_BLK >= n) break;
        if (i < n) s_key[s_cnt[pk[k] >> 12] + slot[k]] = (pk[k] & 4095u) << 14 | (uint32_t)i;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int i = k * SORT1_BLK + t;
        if (k * SORT1_BLK >= n) break;
        if (i < n) {
            float4 p = P.pos[cur][i];
            const float4 vel = P.vel[cur][i];
            int img = P.image[cura][i];
            const int tg = P.tag[cura][i], mk = P.mask[cura][i], og = P.origin[cura][i];
            const float ph = P.phi[cura][i];
            wrap_particle(d, p, img);
            const int gc = (int)(pk[k] >> 12);
            const uint32_t key = (pk[k] & 4095u) << 14 | (uint32_t)i;
            const int lo = s_cnt[gc], hi = s_cnt[gc + 1];
            int dst = lo;
            for (int g = lo; g < hi; ++g) dst += s_key[g] < key;
            P.pos[cur ^ 1][dst] = p;
            P.vel[cur ^ 1][dst] = vel;
            P.xhold[dst] = p;
            P.tag[cura ^ 1][dst] = tg;
            P.mask[cura ^ 1][dst] = mk;
            P.origin[cura ^ 1][dst] = og;
            P.image[cura ^ 1][dst] = img;
            P.phi[cura ^ 1][dst] = ph;
        }
    }
}

// --------------------------------------------------------------------------
// K5: neighbor rows, one wave per cell.  A centre's row lists every
// (j, image) of the 27 stencil cells of its cell -- stencil cell k has offset
// (k%3-1, k/3%3-1, k/9-1), periodic images shift by +-L -- in stencil order,
// then j ascending, with (float) r^2 <= (float)(rc+skin)^2, itself excluded.
// r^2 = fma(dz, dz, fma(dy, dy, dx dx)): the reference's
// `dx * dx + dy * dy + dz * dz` (neigh_build_meso.cu:86-93) as its -O3 build
// (nvcc, floating-point contraction on by default) evaluates it.  The set is
// the reference's (neigh_build_meso.cu:58-118).
//
// All centres of a cell share the stencil, so the wave walks the stencil's
// candidates 64 at a time, one per lane (coalesced loads, image shift applied
// once), NL_ITER iterations held in registers, and tests them against one
// centre after another (the centre's position is uniform).  The lanes that
// pass append in lane order (ballot + mbcnt) to an LDS copy of the centre's
// row, which keeps the row order; the copy is stored to the chunked row
// layout once per centre and batch.  The workgroup is one wave.
// Rows are built from the positions of the last build (xhold), which the
// cells were sorted by: right after the re-sort they equal the sorted
// positions; with relist (the row width grew) every sorted system gets back
// exactly the rows of its last build, whatever steps it has taken since, so
// the rebuild trigger (displacement from xhold) keeps its guarantee.
// relist selects the systems not flagged stale, otherwise the stale ones.
//
// A pool's rebuild walks the worklist k_scan_apply made: the cells holding
// particles of the systems re-sorted this pass, each with its system,
// coordinates and particle range; a listed cell reads its 27 neighbor ranges
// from the linear range table.  A pool's cell slots are
// mostly empty (a droplet fills a quarter of its box) or belong to systems
// not re-sorted, and dispatching one workgroup per cell slot costs ~0.2 ns
// each whether it works or exits (136 us per pass for 650,000 slots), so a
// grid of at most NL_GRID waves takes the list instead, XCD x the x-th eighth
// of it in strides, so that cells next to each other in Morton order share
// that XCD's L2 (batched droplets: rebuild phase 0.379 -> 0.278 ms per pass).
// A relist covers every cell slot, one wave per slot.
// --------------------------------------------------------------------------
constexpr int NL_ITER = 7;             // candidate tiles per batch: 448 candidates (a cell's stencil averages ~370)
constexpr int NL_WAVES = 8;            // waves per SIMD of the worklist walk (61 VGPRs; measured
                                       // faster than seven)
// its waves: one per NL_PART particle slots, about what the cells of a liquid
// hold (waves without a cell cost their dispatch, 14 us for 65,536, 3.8 us for
// the 13,000 of 24 droplets, 8 and 32 slots measured the same within 1%;
// fewer waves than cells balance uneven cells worse), at most NL_GRID
// (measured against 7,168 and 16,384 at 256 droplets)
constexpr int NL_PART = 16, NL_GRID = 65536;

typedef float float3v __attribute__((ext_vector_type(3)));

// LISTED: e = (system, packed coordinates, first particle, end) of a listed
// cell, whose neighbor cells' ranges come from the linear table; otherwise
// e.x = a cell slot, looked up through its system and the Morton rank table
template <bool LISTED>
__device__ __attribute__((always_inline)) void nlist_cell(const PoolDev &P, int4 e, int relist, int part, int parts,
                                                          int *s_row)
{
    int s, xyz, c0, c1, cs = e.x;
    if (LISTED) {
        s = e.x; xyz = e.y; c0 = e.z; c1 = e.w;
    } else {
        s = P.one ? 0 : P.cell_sys[cs];
        if (s < 0) return;
    }
    SysDev *d = P.sys + s;
    const int cb = d->cell_base;
    if (!LISTED) {
        if (relist && (!d->active || d->stale != 0)) return;       // a relist: the systems not flagged stale
        if (cs < cb || cs >= cb + d->ncell) return;       // the end slot holds no cell
        c0 = P.cell_start[cs * SUBCELLS];
        c1 = P.cell_start[(cs + 1) * SUBCELLS];
        if (c0 >= c1) return;
    }
    const int lane = threadIdx.x;
    const float4 *pos = P.xhold;
    // stencil table: lane k < 27 holds cell k's first particle, its length and
    // image code
    int kst = 0, klen = 0;
    uint32_t kcode = IMG_ZERO;
    if (lane < 27) {
        if (!LISTED) xyz = P.cell_xyz[cs];
        const int cx = xyz & 1023, cy = (xyz >> 10) & 1023, cz = (xyz >> 20) & 1023;
        const int nb0 = d->nb[0], nb1 = d->nb[1], nb2 = d->nb[2];
        int nx = cx + lane % 3 - 1, ny = cy + lane / 3 % 3 - 1, nz = cz + lane / 9 - 1;
        int sx = 0, sy = 0, sz = 0;
        if (nx < 0) { nx += nb0; sx = -1; } else if (nx >= nb0) { nx -= nb0; sx = 1; }
        if (ny < 0) { ny += nb1; sy = -1; } else if (ny >= nb1) { ny -= nb1; sy = 1; }
        if (nz < 0) { nz += nb2; sz = -1; } else if (nz >= nb2) { nz -= nb2; sz = 1; }
        const int lin = nx + nb0 * (ny + nb1 * nz);
        if (LISTED) {
            const int2 r = P.cell_lse[cb + lin];
            kst = r.x;
            klen = r.y - r.x;
        } else {
            const int rank = P.cell_rank[cb + lin];
            kst = P.cell_start[(cb + rank) * SUBCELLS];
            klen = P.cell_start[(cb + rank + 1) * SUBCELLS] - kst;
        }
        kcode = (uint32_t)((sx + 1) + 3 * (sy + 1) + 9 * (sz + 1));
    }
    const int kend = wave_incl_scan(klen);
    const int kpre = kend - klen;                           // candidates before cell k
    const int ntot = __builtin_amdgcn_readlane(kend, 26);
    const float rc2 = d->rc2_list;
    const float Lx = d->L[0], Ly = d->L[1], Lz = d->L[2];
    const int maxnbr = P.maxnbr;
    // a cell away from the box's edges has no shifted candidate
    const bool images = __builtin_amdgcn_ballot_w64(lane < 27 && kcode != (uint32_t)IMG_ZERO) != 0;
    for (int cg = c0; cg < c1; cg += WAVE) {
        const int ng = min(WAVE, c1 - cg);
        int cntv = 0;                                       // lane l: row length of centre cg + l
        const float4 pg = pos[min(cg + lane, c1 - 1)];      // lane l: position of centre cg + l
        for (int tb = 0; tb < ntot; tb += NL_ITER * WAVE) {
            // candidates tb + 64 m + lane.  A candidate's stencil cell is the
            // last one that starts at or before it: the cells leave their
            // number where they start, a running maximum spreads it, and all
            // the positions load together (a search per candidate, six
            // shuffles in a row, made each tile wait for its load before the
            // next one's search; with the entries stored below without a
            // branch on where the centre is: 480,000 particles 91 -> 86 us a
            // step, 256 droplets 119 -> 112, 32,000 15.4 -> 14.4).
            float3v q[NL_ITER];
            int qe[NL_ITER];
            const int nm = min(NL_ITER, (ntot - tb + WAVE - 1) / WAVE);
#pragma unroll
            for (int m = 0; m < NL_ITER; ++m) s_row[m * WAVE + lane] = 0;
            __syncthreads();
            if (klen > 0 && (unsigned)(kpre - tb) < NL_ITER * WAVE) s_row[kpre - tb] = lane;
            __syncthreads();
            const uint64_t begun = __builtin_amdgcn_ballot_w64(klen > 0 && kpre <= tb);
            int carry = begun ? 63 - __clzll(begun) : 0;
#pragma unroll
            for (int m = 0; m < NL_ITER; ++m) qe[m] = s_row[m * WAVE + lane];
            __syncthreads();
#pragma unroll
            for (int m = 0; m < NL_ITER; ++m) {
                const int k = max(wave_scan(qe[m], [](int x, int y) { return max(x, y); }), carry);
                carry = __builtin_amdgcn_readlane(k, 63);
                const int t = tb + m * WAVE + lane;
                // every shuffle with the whole wave active (a lane reads a
                // source lane's register only while that lane is active)
                const int j0 = __shfl(kst - kpre, k);
                uint32_t code = IMG_ZERO;
                if (images) code = (uint32_t)__shfl((int)kcode, k);
                qe[m] = (int)((uint32_t)(t < ntot ? j0 + t : c0) | (code << IMG_SHIFT));
            }
#pragma unroll
            for (int m = 0; m < NL_ITER; ++m) q[m] = *(const float3v *)(pos + ((uint32_t)qe[m] & IDX_MASK));
#pragma unroll
            for (int m = 0; m < NL_ITER; ++m) {
                if (tb + m * WAVE + lane >= ntot) q[m].x = __builtin_inff();     // no candidate
                if (images) {
                    int sx, sy, sz;
                    image_decode((uint32_t)qe[m] >> IMG_SHIFT, sx, sy, sz);
                    q[m].x += (float)sx * Lx;
                    q[m].y += (float)sy * Ly;
                    q[m].z += (float)sz * Lz;
                }
            }
            for (int c = cg + part; c < cg + ng; c += parts) {
                const int cl = c - cg;
                const float pcx = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pg.x), cl));
                const float pcy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pg.y), cl));
                const float pcz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pg.z), cl));
                const int q0 = __builtin_amdgcn_readlane(cntv, cl);     // row length before this batch
                int n = 0;                                  // hits of this batch, staged in LDS
#pragma unroll
                for (int m = 0; m < NL_ITER; ++m) {
                    if (m >= nm) break;
                    const float dx = pcx - q[m].x, dy = pcy - q[m].y, dz = pcz - q[m].z;
                    const float r2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                    const uint64_t mask = __builtin_amdgcn_ballot_w64(r2 <= rc2);
                    if (mask) {
                        if (__builtin_amdgcn_inverse_ballot_w64(mask))
                            s_row[n + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u))] = qe[m];
                        n += __popcll(mask);
                    }
                }
                // this batch's entries of centre c: rows [q0, ...) in the
                // chunked layout, entries past the row width dropped (the
                // count marks the overflow).  The centre itself is among the
                // hits once in its whole row (stencil cell 13, the only one
                // with a zero image shift, distance 0): that entry is left
                // out and the entries after it move up by one.
                __syncthreads();
                const int selfe = (int)((uint32_t)c | (IMG_ZERO << IMG_SHIFT));
                int *row = P.nlist + nbr_at(c, 0, maxnbr);
                int shift = 0;
                for (int k0 = 0; k0 < n; k0 += WAVE) {
                    const int k = k0 + lane, v = s_row[k];                                  // n <= NL_ITER * WAVE
                    const uint64_t in = __builtin_amdgcn_ballot_w64(k < n);
                    const uint64_t sb = __builtin_amdgcn_ballot_w64(v == selfe) & in;       // the lane holding the centre
                    const uint64_t after = sb ? ~(sb | (sb - 1)) : 0;                       // and those past it
                    const uint32_t q = (uint32_t)(q0 + k - shift - (__builtin_amdgcn_inverse_ballot_w64(after) ? 1 : 0));
                    if (__builtin_amdgcn_inverse_ballot_w64(in & ~sb) && q < (uint32_t)maxnbr)
                        row[(q & ~(uint32_t)(NBR_CHUNK - 1)) * WAVE + (q & (uint32_t)(NBR_CHUNK - 1))] = v;
                    if (sb) shift = 1;
                }
                __syncthreads();
                if (lane == cl) cntv = q0 + n - shift;
            }
        }
        const bool mine = lane < ng && (parts == 1 || lane % parts == part);
        if (mine) P.ncount[cg + lane] = cntv;
        if (__ballot(mine && cntv > maxnbr) && lane == 0) atomicOr(&d->overflow, 1);
    }
}

// Commit after a rebuild: the sorted data in the other buffers becomes current.
__device__ inline void commit_rebuild_sys(const PoolDev &P, int s)
{
    SysDev *d = P.sys + s;
    if (!d->active || !d->stale) return;
    d->sel ^= 1;
    d->sela ^= 1;
    d->stale = 0;
    d->ago = 0;
    d->builds += 1;
}

// one wave per cell slot (a relist, or one system): eight waves per SIMD
// (seven candidate tiles in registers, no spills), measured faster than seven
__global__ void __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(8, 8))) k_nlist(PoolDev P, int relist, int ncells, int lparts, int nseed)
{
    __shared__ int s_row[NL_ITER * WAVE];                   // one centre's entries of one batch
    const int nu = ncells << lparts;                        // 2^lparts waves share a cell's centres
    const int b = (int)blockIdx.x - nseed;
    if (b < 0) { next_seeds(P, blockIdx.x); return; }
    if (!relist) {
        // the one system, when k_keys found it stale; its rebuild is committed
        // here: the row build reads only its geometry and the flag word
        if (P.work_count[1] == 0) return;
        if (b == 0 && threadIdx.x == 0) commit_rebuild_sys(P, 0);
    }
    const int u = xcd_logical(b, nu), cs = u >> lparts;     // cell slot (Morton rank order)
    if (cs < ncells)
        nlist_cell<false>(P, make_int4(cs, 0, 0, 0), relist, u & ((1 << lparts) - 1), 1 << lparts, s_row);
}

// the worklist walk; it also commits the rebuild of every re-sorted system
// (the row build reads only their geometry, and the next kernel sees the
// flipped buffers), which saves a launch per pass
__global__ void __launch_bounds__(WAVE) __attribute__((amdgpu_waves_per_eu(NL_WAVES, NL_WAVES))) k_nlist_listed(PoolDev P)
{
    __shared__ int s_row[NL_ITER * WAVE];
    for (int s = blockIdx.x * WAVE + threadIdx.x; s < P.nsys; s += gridDim.x * WAVE) commit_rebuild_sys(P, s);
    // gridDim.x is a multiple of NXCD; workgroup b runs on XCD b % NXCD
    const int n = *P.work_count;
    const int x = blockIdx.x % NXCD, per = gridDim.x / NXCD;
    const int hi = (int)((long long)n * (x + 1) / NXCD);
    for (int w = (int)((long long)n * x / NXCD) + blockIdx.x / NXCD; w < hi; w += per)
        nlist_cell<true>(P, P.cell_work[w], 0, 0, 1, s_row);
}

// overflow flags of the sorted systems cleared before their rows are rebuilt
// in place (k_nlist sets them again if the rows are still too narrow)
__global__ void k_clear_overflow(PoolDev P)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= P.nsys) return;
    SysDev *d = P.sys + s;
    if (d->active && !d->stale) d->overflow = 0;
}

// --------------------------------------------------------------------------
// The reference's 2-level Morton keys of one system's particles at the last
// build, in sorted order (parity hook; the sort itself orders sub-cells).
// --------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_sort_keys(PoolDev P, unsigned long long *out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const SysDev *d = P.sys;
    if (i >= d->n) return;
    int b[3];
    const uint32_t z2 = particle_bins(d, P.xhold[i], b);
    out[i] = (morton3((uint32_t)b[0], (uint32_t)b[1], (uint32_t)b[2]) << d->l1_shift) | z2;
}

// --------------------------------------------------------------------------
// Signatures of the current step (setup only; in the step loop the fused
// force epilogue writes them for the following step).
// --------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_signatures(PoolDev P)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= P.nact) return;
    const int s = P.wave_sys[i >> 6];
    if (s < 0) return;
    SysDev *d = P.sys + s;
    if (!d->active || i >= d->part_base + d->n) return;
    const uint32_t st = premix<64>(d->seed, (uint32_t)d->step);
    float4 v = P.vel[d->sel][i];
    const int tag = P.tag[d->sela][i];
    const uint32_t sg = d->style == STYLE_MDPD ? sig_mdpd(tag, st) : sig_dpd(tag, st, v.x, v.y, v.z);
    v.w = __uint_as_float(sg);
    P.vel[d->sel][i] = v;
}

// ----------------------------------------------------------------------------
// host launchers
// ----------------------------------------------------------------------------
static inline int nblk(int n, int b) { return (n + b - 1) / b; }
// One system of few cells: four waves share a cell's centres, each listing the
// stencil for itself (1,000 particles: 21 -> 13 us; every cell of a larger
// system has its wave at once anyway, and the launch grows by 0.2 ns a wave).
constexpr int NL_FEW = 2560, NL_LPARTS = 2;

static void launch_nlist(const PoolDev &P, int relist, bool seeds, hipStream_t st)
{
    if (P.ncact <= 0) return;
    if (relist || !nlist_listed(P)) {
        const int lparts = P.one && P.ncact <= NL_FEW ? NL_LPARTS : 0;
        hipLaunchKernelGGL(k_nlist, dim3(xcd_grid(P.ncact << lparts) + (seeds ? seed_grid(P) : 0)), dim3(WAVE), 0, st, P,
                           relist, P.ncact, lparts, seeds ? seed_grid(P) : 0);
    } else
        hipLaunchKernelGGL(k_nlist_listed, dim3(std::min(NL_GRID, xcd_grid(std::min(P.ncact, P.nact / NL_PART)))), dim3(WAVE), 0, st, P);
}

// A step with the one-launch sort against the four launches, us (DPD fluid of
// density 3; mDPD droplets within 2 us of it), by the steps between re-sorts:
//   particles   1             2             3             4             none due
//   1,000       25.2 / 31.5   21.0 / 26.7   19.4 / 24.8   18.8 / 24.0   16.7 / 21.3
//   3,500       33.0 / 32.8   25.1 / 27.5   22.2 / 25.4   20.9 / 24.5   17.0 / 21.7
//   5,000       38.4 / 33.4   28.0 / 27.8   24.3 / 25.7   22.6 / 24.8   17.3 / 21.8
//   7,000       44.6 / 34.7   31.3 / 28.6   26.7 / 26.4   24.4 / 25.3   17.7 / 22.2
//   9,000       50.6 / 35.6   34.4 / 29.2   28.9 / 26.9   26.1 / 25.8   18.0 / 22.5
// One launch gains 4.5 us on a step without a re-sort and loses ~2.7 ns per
// particle past 3,300 on a step with one: even at 3,300 + 1,650 (period - 1).
int sort_one_limit(int period)
{
    return (int)std::min<long long>(SORT1_N, 3300 + 1650 * ((long long)std::max(period, 1) - 1));
}

hipError_t launch_rebuild(const PoolDev &P, int split, int commit, hipStream_t st)
{
    if (P.nact == 0) return hipSuccess;
    if (commit != COMMIT_FINAL && commit != COMMIT_PHASED && commit != COMMIT_DECIDE) return hipErrorInvalidValue;
    const bool fseed = first_seeds(split, P.nact / WAVE);
    const int seeded = P.one || fseed ? 1 : 0;
    if (P.one && P.nact <= std::min(P.sort1, SORT1_N) && (P.ncellslots - 1) * SUBCELLS <= SORT1_SUB) {
        if (P.nact <= SORT1_BLK)
            hipLaunchKernelGGL((k_sort_one<1>), dim3(1), dim3(SORT1_BLK), 0, st, P, commit, seeded);
        else
            hipLaunchKernelGGL((k_sort_one<SORT1_PER>), dim3(1), dim3(SORT1_BLK), 0, st, P, commit, seeded);
        launch_nlist(P, 0, !fseed, st);
        return hipGetLastError();
    }
    const dim3 g(nblk(P.nact, 256)), b(256);
    hipLaunchKernelGGL(k_keys, g, b, 0, st, P, commit);
    const long long nsub = P.maxsub > 0 ? (long long)P.maxsub : (long long)P.ncellslots * SUBCELLS;
    const bool scan_one = P.one && nblk((int)nsub, SCAN1_CH) <= SCAN1_MAX;
    if (scan_one) {
        hipLaunchKernelGGL(k_scan_one, dim3(nblk((int)nsub, SCAN1_CH)), dim3(SCAN1_BLK), 0, st, P, commit, split, seeded);
    } else {
        // workgroups per system for the chunked scan: as many as the largest
        // system has chunks, up to 64 (smaller systems' extra workgroups exit)
        const int nch = (int)((nsub + SCAN_CH - 1) / SCAN_CH);
        const int gs = std::max(1, std::min(64, nch));
        hipLaunchKernelGGL(k_scan_sums, dim3(gs, P.nsys), dim3(SCAN_BLK), 0, st, P, commit, split, seeded);
        hipLaunchKernelGGL(k_scan_apply, dim3(gs, P.nsys), dim3(SCAN_BLK), 0, st, P);
    }
    hipLaunchKernelGGL(k_scatter, g, b, 0, st, P, scan_one ? 1 : 0);
    hipLaunchKernelGGL(k_sortgather, g, b, 0, st, P);
    launch_nlist(P, 0, P.one && !fseed, st);
    return hipGetLastError();
}

hipError_t launch_nlist_only(const PoolDev &P, hipStream_t st)
{
    if (P.nact == 0) return hipSuccess;
    launch_nlist(P, 0, false, st);
    return hipGetLastError();
}

hipError_t launch_relist(const PoolDev &P, hipStream_t st)
{
    if (P.nact == 0) return hipSuccess;
    hipLaunchKernelGGL(k_clear_overflow, dim3(nblk(P.nsys, 64)), dim3(64), 0, st, P);
    launch_nlist(P, 1, false, st);
    return hipGetLastError();
}

hipError_t launch_sort_keys(const PoolDev &P, unsigned long long *out, hipStream_t st)
{
    if (!P.one || !out) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_sort_keys, dim3(nblk(P.nact, 256)), dim3(256), 0, st, P, out);
    return hipGetLastError();
}

hipError_t launch_signatures(const PoolDev &P, hipStream_t st)
{
    hipLaunchKernelGGL(k_signatures, dim3(nblk(P.nact, 256)), dim3(256), 0, st, P);
    return hipGetLastError();
}

}  // namespace mdpd
