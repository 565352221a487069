// Per-step passes of the mdpd355 engine: local density, initial half-kick,
// and the pair-force pass with velocity-Verlet fused into its epilogue.
//
// Replaces, per step (ModifiedVerlet::run, src/USER-MESO/mvv_meso.cu:321-564):
//   FixArbitraryBoundaryRho::pre_force / gpu_compute_rho   fix_aboundary_rho_meso.cu:119-212
//   MesoPairMDPD::compute / gpu_mdpd                        pair_mdpd_meso.cu:93-293
//   MesoPairDPD::compute / gpu_dpd                          pair_dpd_meso.cu:91-266
//   FixNVEMeso::initial_integrate / final_integrate         fix_nve_meso.cu:63-199
//   MesoFixAddForce::post_force                             fix_addforce_meso.cu:72-108
//   dp2sp_merged signatures                                 atom_vec_mdpd_atomic_meso.cu:140-206
//
// Each step the first pass (density for mDPD, a filter pass for DPD) walks the
// full neighbor rows (cutoff + skin) and writes, per particle, the compact row
// of entries inside the pair cutoff; the force pass then walks only those.
// Compact rows are staged per lane in LDS and stored as whole coalesced rows.
//
// Launch shape: the first and force passes run one workgroup per 64-particle
// tile with SPLIT waves sharing the tile's rows, or, up to WIDE_TILES tiles,
// with eight to twelve that keep those waves' sums; systems are padded to 256
// slots; workgroup ids are remapped so each of the 8 XCDs sweeps one
// contiguous particle range.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>

namespace mdpd {

constexpr int BLK = 256;

// A wave that holds a particle past skin/2 says so in its system's flag: a
// plain store, the same from every wave (same-address device-scope atomics
// serialize across the XCDs and cost ~50 ns each), and none on most steps.
__device__ inline void flag_moved(SysDev *d, bool moved)
{
    if (__builtin_amdgcn_ballot_w64(moved) != 0 && (threadIdx.x & 63) == 0) d->moved = 1;
}

// a - (b + s L) with a single rounding.  Adding s L to the neighbor's
// coordinate first rounds at the magnitude of L (half an ulp of L: 4.8e-7 at
// L = 8), an error in r that the density weight (r_d - r)^2 amplifies for a
// neighbor near r_d.  Here the difference a - b and its exact rounding error
// (Knuth's TwoSum) come first; a - b lies within r_c + skin of s L, so for
// L >= 2 (r_c + skin) subtracting s L is exact (Sterbenz) and the error term
// is added back last, giving the correctly rounded displacement.  With s = 0
// the result equals a - b bit for bit.
__device__ inline float image_diff(float a, float b, float sl)
{
    const float d = a - b;
    const float bv = d - a;
    const float e = (a - (d - bv)) + (-b - bv);
    return (d - sl) + e;
}

// displacement r_i - (r_j + s L) of a neighbor entry with image code `code`
__device__ inline void pair_delta(const float4 &pi, const float4 &q, uint32_t code, const SysDev *d, float &dx,
                                  float &dy, float &dz)
{
    if (code == IMG_ZERO) {
        dx = pi.x - q.x; dy = pi.y - q.y; dz = pi.z - q.z;
    } else {
        int sx, sy, sz;
        image_decode(code, sx, sy, sz);
        dx = image_diff(pi.x, q.x, (float)sx * d->L[0]);
        dy = image_diff(pi.y, q.y, (float)sy * d->L[1]);
        dz = image_diff(pi.z, q.z, (float)sz * d->L[2]);
    }
}

// r^2 with the fusion spelled out, so the first pass's compaction test and
// the force pass's cutoff test see the same bits
__device__ inline float dist2(float dx, float dy, float dz) { return fmaf(dz, dz, fmaf(dy, dy, dx * dx)); }

__device__ inline float pair_rsq(const float4 &pi, const float4 &q, uint32_t code, const SysDev *d)
{
    float dx, dy, dz;
    pair_delta(pi, q, code, d, dx, dy, dz);
    return dist2(dx, dy, dz);
}

// --------------------------------------------------------------------------
// first pass: density rho_i = m_i * sum_j w(r_ij) over 1e-20 <= r^2 < rd^2
// (no self term; fix_aboundary_rho_meso.cu:131-164), and the compact rows of
// entries with r^2 < rc^2 for the force pass.  WITH_RHO = false is the DPD
// filter pass (no density).
//
// One workgroup per 64-particle tile; wave w of SPLIT walks the chunks of
// row entries 8k..8k+7 with k = w mod SPLIT and writes its compact entries
// to compact rows t * SPLIT + w, so the force pass can give the same rows to
// the same wave.
// Partial densities are summed in LDS in wave order (deterministic).
// --------------------------------------------------------------------------
// the density weight of a neighbor at r = sqrt(rsq) < h, (h - r)^2 or Lucy's
// (h + 3 r) (h - r)^3, as the two factors of the fused multiply-add that adds
// it to a sum (both passes below round alike); rsq < 0: zero
__device__ inline float2 weight_factors(float h, float rsq, bool lucy)
{
    const float r = __builtin_amdgcn_sqrtf(rsq);
    const float hm = h - r;
    const float g = lucy ? fmaf(r, 3.f, h) * hm * hm : hm;
    return rsq < 0.f ? make_float2(0.f, 0.f) : make_float2(hm, g);
}

// system of a tile; one system (the plain path) holds them all
__device__ inline int tile_system(const PoolDev &P, int tile) { return P.one ? 0 : P.wave_sys[tile]; }

// density of particle i from its weight sum, and the record the force pass of
// a one-type system gathers (position and density in one 16-byte load)
template <bool WITH_RHO>
__device__ inline void finish_density(const PoolDev &P, const SysDev *d, int i, const float4 &pi, float sum)
{
    if (WITH_RHO) {
        const int mk = P.mask[d->sela][i];
        const int ti = __float_as_int(pi.w);
        const float r = (mk & d->rho_bit) ? P.mass[d->mass_base + ti] * d->rho_factor * sum : 0.f;
        P.rho[i] = r;
        P.pr[i] = make_float4(pi.x, pi.y, pi.z, r);
    } else if (d->style == STYLE_MDPD) {
        // mDPD without the density fix: zero density (P.rho keeps its zeros)
        P.pr[i] = make_float4(pi.x, pi.y, pi.z, 0.f);
    }
}

template <bool WITH_RHO, int SPLIT>
__global__ void __launch_bounds__(WAVE * SPLIT) k_first(PoolDev P, int ntiles, int nseed)
{
    constexpr int STAGE = 32 / SPLIT;   // LDS-staged compact entries per lane (measured best)
    __shared__ int s_c[SPLIT][STAGE * WAVE];
    __shared__ float s_sum[SPLIT][WAVE];
    const int b = (int)blockIdx.x - (SPLIT == 1 ? nseed : 0);
    if (SPLIT == 1 && b < 0) { next_seeds(P, blockIdx.x); return; }
    const int tile = xcd_logical(b, ntiles);
    if (tile >= ntiles) return;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i = tile * WAVE + lane;
    const int s = tile_system(P, tile);
    if (s < 0) return;
    const SysDev *d = P.sys + s;
    if (!d->active || d->overflow) return;    // an overflowed system waits for wider rows
    const bool valid = i < d->part_base + d->n;
    const float4 *pos = P.pos[d->sel];
    const int maxnbr = P.maxnbr;
    const size_t tbase = (size_t)tile * maxnbr * WAVE + lane;
    const int *row = P.nlist + nbr_at(i, 0, maxnbr);
    int *crow = P.clist + tbase;
    int cnt = 0;
    float4 pi = make_float4(0.f, 0.f, 0.f, 0.f);
    if (valid) {
        pi = pos[i];
        cnt = min(P.ncount[i], maxnbr);
    }
    const float h = d->rd, h2 = h * h;
    const float rc2 = d->rc2_max;
    const bool lucy = d->lucy;
    float sum = 0.f;
    int nc = 0;
    // ROOM: the staging area is known to hold this entry (no spill check)
    auto visit = [&](uint32_t e, const float4 &q, auto room) {
        const float rsq = pair_rsq(pi, q, e >> IMG_SHIFT, d);
        if (WITH_RHO && rsq < h2 && rsq >= 1e-20f) {
            const float2 f = weight_factors(h, rsq, lucy);
            sum = fmaf(f.x, f.y, sum);
        }
        if (rsq < rc2 && rsq >= 1e-20f) {
            if constexpr (decltype(room)::value) {
                s_c[w][nc * WAVE + lane] = (int)e;
            } else {
                if (nc < STAGE) s_c[w][nc * WAVE + lane] = (int)e;
                else crow[(size_t)(nc * SPLIT + w) * WAVE] = (int)e;
            }
            ++nc;
        }
    };
    // a chunk of eight entries (two 16-byte loads) and their eight position
    // gathers in flight per lane, the next chunk's entries loading meanwhile;
    // wave w takes chunks w, w + SPLIT, ... and visits them in row order.
    // With one wave per tile (SPLIT 1) the LDS staging, not registers, limits
    // occupancy, so a wave takes U = 2 chunks per iteration: sixteen gathers
    // in flight, the next two chunks' entries loading meanwhile.
    constexpr int U = SPLIT == 1 ? 2 : 1;
    const int nch = (cnt + NBR_CHUNK - 1) / NBR_CHUNK;
    const int4 *row4 = (const int4 *)row;
    int4 ea[U], eb[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        ea[u] = make_int4(0, 0, 0, 0);
        eb[u] = ea[u];
        const int cu = w + u * SPLIT;
        if (cu < nch) {
            ea[u] = row4[(size_t)cu * (NBR_CHUNK * WAVE / 4)];
            eb[u] = row4[(size_t)cu * (NBR_CHUNK * WAVE / 4) + 1];
        }
    }
    for (int c = w; c < nch; c += SPLIT * U) {
        uint32_t e[U * NBR_CHUNK];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            e[u * NBR_CHUNK + 0] = (uint32_t)ea[u].x; e[u * NBR_CHUNK + 1] = (uint32_t)ea[u].y;
            e[u * NBR_CHUNK + 2] = (uint32_t)ea[u].z; e[u * NBR_CHUNK + 3] = (uint32_t)ea[u].w;
            e[u * NBR_CHUNK + 4] = (uint32_t)eb[u].x; e[u * NBR_CHUNK + 5] = (uint32_t)eb[u].y;
            e[u * NBR_CHUNK + 6] = (uint32_t)eb[u].z; e[u * NBR_CHUNK + 7] = (uint32_t)eb[u].w;
            const int cn = c + (U + u) * SPLIT;
            if (cn < nch) {
                ea[u] = row4[(size_t)cn * (NBR_CHUNK * WAVE / 4)];
                eb[u] = row4[(size_t)cn * (NBR_CHUNK * WAVE / 4) + 1];
            }
        }
        float4 q[U * NBR_CHUNK];
        if constexpr (SPLIT == 1) {
            // past the row's end a lane takes itself (r = 0, skipped), so only
            // the room in the staging area is left to check, by iteration
            // (256 droplets 214 -> 210 us; with two or four waves per tile it
            // costs registers: 480,000 particles 80 -> 86)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int left = cnt - (c + u) * NBR_CHUNK;
                if (__builtin_amdgcn_ballot_w64(left < NBR_CHUNK) != 0)
#pragma unroll
                    for (int k = 0; k < NBR_CHUNK; ++k)
                        if (k >= left) e[u * NBR_CHUNK + k] = (uint32_t)i | ((uint32_t)IMG_ZERO << IMG_SHIFT);
            }
#pragma unroll
            for (int k = 0; k < U * NBR_CHUNK; ++k) q[k] = pos[e[k] & IDX_MASK];
            if (__builtin_amdgcn_ballot_w64(nc + U * NBR_CHUNK > STAGE) == 0) {
#pragma unroll
                for (int k = 0; k < U * NBR_CHUNK; ++k) visit(e[k], q[k], std::true_type{});
            } else {
#pragma unroll
                for (int k = 0; k < U * NBR_CHUNK; ++k) visit(e[k], q[k], std::false_type{});
            }
        } else {
            // when every active lane's row covers all of this iteration's
            // entries and its staging area has room for all of them, the
            // per-entry row-end and staging checks are skipped (same result)
            const bool full = (c + (U - 1) * SPLIT + 1) * NBR_CHUNK <= cnt && nc + U * NBR_CHUNK <= STAGE;
            if (__builtin_amdgcn_ballot_w64(!full) == 0) {
#pragma unroll
                for (int k = 0; k < U * NBR_CHUNK; ++k) q[k] = pos[e[k] & IDX_MASK];
#pragma unroll
                for (int k = 0; k < U * NBR_CHUNK; ++k) visit(e[k], q[k], std::true_type{});
            } else {
#pragma unroll
                for (int k = 0; k < U * NBR_CHUNK; ++k) {
                    const int p = (c + (k / NBR_CHUNK) * SPLIT) * NBR_CHUNK + k % NBR_CHUNK;
                    q[k] = pos[(p < cnt ? e[k] : (uint32_t)i) & IDX_MASK];
                }
#pragma unroll
                for (int k = 0; k < U * NBR_CHUNK; ++k) {
                    const int p = (c + (k / NBR_CHUNK) * SPLIT) * NBR_CHUNK + k % NBR_CHUNK;
                    if (p < cnt) visit(e[k], q[k], std::false_type{});
                }
            }
        }
    }
    // coalesced store of the staged rows
    const int ncmax = wave_max(min(nc, STAGE));
    for (int t = 0; t < ncmax; ++t)
        if (t < nc) crow[(size_t)(t * SPLIT + w) * WAVE] = s_c[w][t * WAVE + lane];
    P.ccount[ccount_at(tile, w, lane)] = nc;
    if (WITH_RHO) {
        s_sum[w][lane] = sum;
        __syncthreads();
        if (w == 0)
            for (int k = 1; k < SPLIT; ++k) sum += s_sum[k][lane];
    }
    if (w == 0 && valid) finish_density<WITH_RHO>(P, d, i, pi, sum);
}

// --------------------------------------------------------------------------
// The first pass with one wave per row chunk of a tile (split 2 and 4): lane
// l of wave k holds chunk k of particle l, its eight gathers in flight at
// once.  Each wave leaves its in-cutoff counts and its weight factors in LDS,
// places its compact entries after those of the sub-row's earlier chunks, and
// wave w adds up sub-row w's weights in row order.  Rounds of FS_WAVES chunks.
// --------------------------------------------------------------------------
template <int SPLIT>
constexpr int FS_WAVES = SPLIT == 2 ? 10 : 12;

template <bool WITH_RHO, int SPLIT>
__global__ void __launch_bounds__(WAVE * FS_WAVES<SPLIT>) k_first_wide(PoolDev P, int ntiles, int nseed)
{
    constexpr int NW = FS_WAVES<SPLIT>;
    static_assert(NW % SPLIT == 0, "a wave keeps its sub-row from round to round");
    __shared__ float2 s_w[WITH_RHO ? NW * NBR_CHUNK : 1][WAVE];    // weight factors of each entry
    __shared__ int s_n[NW][WAVE];                                  // in-cutoff entries of each chunk
    __shared__ float s_sum[SPLIT][WAVE];
    const int b = (int)blockIdx.x - nseed;
    if (b < 0) { next_seeds(P, blockIdx.x); return; }
    const int tile = xcd_logical(b, ntiles);
    if (tile >= ntiles) return;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int i = tile * WAVE + lane;
    const int s = tile_system(P, tile);
    if (s < 0) return;
    const SysDev *d = P.sys + s;
    if (!d->active || d->overflow) return;    // an overflowed system waits for wider rows
    const bool valid = i < d->part_base + d->n;
    const float4 *pos = P.pos[d->sel];
    const int maxnbr = P.maxnbr;
    int *crow = P.clist + (size_t)tile * maxnbr * WAVE + lane;
    float4 pi = make_float4(0.f, 0.f, 0.f, 0.f);
    int cnt = 0;
    if (valid) {
        pi = pos[i];
        cnt = min(P.ncount[i], maxnbr);
    }
    const float h = d->rd, h2 = h * h;
    const float rc2 = d->rc2_max;
    const bool lucy = d->lucy;
    const int4 *row4 = (const int4 *)(P.nlist + nbr_at(i, 0, maxnbr));
    float sum = 0.f;
    int base = 0;                             // compact entries of this wave's sub-row in earlier rounds
    for (int c0 = 0;; c0 += NW) {
        const int c = c0 + wv, left = cnt - c * NBR_CHUNK;      // this chunk's entries, if fewer than eight
        uint32_t e[NBR_CHUNK];
        int flags = 0;
        if (left > 0) {
            const int4 ea = row4[(size_t)c * (NBR_CHUNK * WAVE / 4)], eb = row4[(size_t)c * (NBR_CHUNK * WAVE / 4) + 1];
            e[0] = (uint32_t)ea.x; e[1] = (uint32_t)ea.y; e[2] = (uint32_t)ea.z; e[3] = (uint32_t)ea.w;
            e[4] = (uint32_t)eb.x; e[5] = (uint32_t)eb.y; e[6] = (uint32_t)eb.z; e[7] = (uint32_t)eb.w;
            float4 q[NBR_CHUNK];
#pragma unroll
            for (int k = 0; k < NBR_CHUNK; ++k) q[k] = pos[(k < left ? e[k] : (uint32_t)i) & IDX_MASK];
#pragma unroll
            for (int k = 0; k < NBR_CHUNK; ++k) {
                const float rsq = pair_rsq(pi, q[k], k < left ? e[k] >> IMG_SHIFT : IMG_ZERO, d);
                const bool in = k < left && rsq >= 1e-20f;
                if (WITH_RHO) s_w[wv * NBR_CHUNK + k][lane] = weight_factors(h, in && rsq < h2 ? rsq : -1.f, lucy);
                flags |= (in && rsq < rc2 ? 1 : 0) << k;
            }
        }
        s_n[wv][lane] = __popc((unsigned)flags);
        __syncthreads();
        int at = base;                        // compact entries of the sub-row before this chunk
#pragma unroll
        for (int k = 0; k < NW / SPLIT; ++k) {
            const int x = s_n[k * SPLIT + wv % SPLIT][lane];
            at += k * SPLIT + wv % SPLIT < wv ? x : 0;
            base += x;
        }
        int r = at * SPLIT + wv % SPLIT;
#pragma unroll
        for (int k = 0; k < NBR_CHUNK; ++k)
            if (flags >> k & 1) {
                crow[(size_t)r * WAVE] = (int)e[k];
                r += SPLIT;
            }
        if (WITH_RHO && wv < SPLIT) {
            for (int k = wv; k < NW; k += SPLIT) {
                const int m = cnt - (c0 + k) * NBR_CHUNK;
                if (m > 0)
#pragma unroll
                    for (int x = 0; x < NBR_CHUNK; ++x) {
                        const float2 f = s_w[k * NBR_CHUNK + x][lane];
                        sum = fmaf(f.x, f.y, sum);
                    }
            }
        }
        if (__builtin_amdgcn_ballot_w64(cnt > (c0 + NW) * NBR_CHUNK) == 0) break;
        __syncthreads();                      // the next round reuses the slots
    }
    if (wv < SPLIT) {
        P.ccount[ccount_at(tile, wv, lane)] = base;
        s_sum[wv][lane] = sum;
    }
    __syncthreads();
    if (wv == 0 && valid) {
        float tot = s_sum[0][lane];
#pragma unroll
        for (int k = 1; k < SPLIT; ++k) tot += s_sum[k][lane];
        finish_density<WITH_RHO>(P, d, i, pi, tot);
    }
}

// --------------------------------------------------------------------------
// initial half-kick + drift from the stored force (first step of a run)
// --------------------------------------------------------------------------
__device__ inline uint32_t next_signature(const SysDev *d, int tag, float vx, float vy, float vz)
{
    return d->style == STYLE_MDPD ? sig_mdpd(tag, d->seed_next) : sig_dpd(tag, d->seed_next, vx, vy, vz);
}

__global__ void __launch_bounds__(BLK) k_initial(PoolDev P, int nlogical)
{
    const int lb = xcd_logical(blockIdx.x, nlogical);
    if (lb >= nlogical) return;
    const int i = lb * BLK + threadIdx.x;
    const int s = P.wave_sys[(lb * BLK) >> 6];
    if (s < 0) return;
    SysDev *d = P.sys + s;
    if (!d->active) return;
    int moved = 0;
    if (i < d->part_base + d->n) {
        const int cur = d->sel;
        float4 p = P.pos[cur][i];
        float4 v = P.vel[cur][i];
        const float4 f = P.frc[i];
        const int mk = P.mask[d->sela][i];
        if (mk & d->nve_bit) {
            const float dtfm = d->dtf * P.minv[d->mass_base + __float_as_int(p.w)];
            v.x += dtfm * f.x; v.y += dtfm * f.y; v.z += dtfm * f.z;
            p.x += d->dt * v.x; p.y += d->dt * v.y; p.z += d->dt * v.z;
        }
        v.w = __uint_as_float(next_signature(d, P.tag[d->sela][i], v.x, v.y, v.z));
        P.pos[cur ^ 1][i] = p;
        P.vel[cur ^ 1][i] = v;
        const float4 h = P.xhold[i];
        const float ex = p.x - h.x, ey = p.y - h.y, ez = p.z - h.z;
        moved = ex * ex + ey * ey + ez * ez > d->trig2;
    }
    if (!d->fix_arb) flag_moved(d, moved);          // else k_aboundary does, from the final positions
}

// --------------------------------------------------------------------------
// pair force (+ fused velocity-Verlet) over the compact rows.  One workgroup
// per 64-particle tile; wave w of SPLIT takes compact rows t * SPLIT + w (the
// ones the first pass wrote for it); partial sums meet in LDS and wave 0 adds
// them in wave order, then runs the integration epilogue.
// --------------------------------------------------------------------------
struct PairC {
    float rc, rc2, rcinv, rd, rdinv, a, b, gamma, sigma, expw;
};

__device__ inline PairC load_coef(const float *tab, int idx)
{
    const float *c = tab + idx * NCOEF;
    PairC q;
    q.rc = c[C_RC]; q.rc2 = c[C_RC2]; q.rcinv = c[C_RCINV]; q.rd = c[C_RD]; q.rdinv = c[C_RDINV];
    q.a = c[C_A]; q.b = c[C_B]; q.gamma = c[C_GAMMA]; q.sigma = c[C_SIGMA]; q.expw = c[C_EXPW];
    return q;
}

template <bool EV>
struct Acc {
    static constexpr int N = EV ? 10 : 3;
    float v[N];
    __device__ Acc() { for (int k = 0; k < N; ++k) v[k] = 0.f; }
};

// One pair: displacement, F / r and (EV) its energy.
// TEST = false: the entry is known to pass the cutoff test (a one-type
// system's compact row holds exactly the entries with
// 1e-20 <= r^2 < rc^2, r^2 computed from the same positions by dist2, and
// the system's largest cutoff is its only one).
// yx: dx.dv starts from the y product, as it does for the odd last entry of
// the rows (or row parts) that the loops below walk in pairs; its rounding is
// part of a trajectory, which grows any difference, so every kernel keeps it.
// Energy: en * eg, added with one rounding (eg = 1: en, which has had its own).
// DPD of one type keeps the factors apart so that every kernel rounds alike.
struct PairF {
    float dx, dy, dz, fpair, en, eg;
};

// styles whose energy is kept as two factors
constexpr bool en_factors(int style) { return style == STYLE_DPD; }

template <int STYLE, bool EV, bool TEST = true>
__device__ inline PairF pair_eval(const float4 &pi, const float4 &vi, float rho_i, const float4 &q, const float4 &vj,
                                  float rho_j, uint32_t code, const PairC &c, float dtis, const SysDev *d, bool yx)
{
    PairF o;
    float dx, dy, dz;
    pair_delta(pi, q, code, d, dx, dy, dz);
    const float rsq = dist2(dx, dy, dz);
    const bool in = !TEST || (rsq < c.rc2 && rsq >= 1e-20f);
    const float rinv = __builtin_amdgcn_rsqf(rsq);
    const float r = rsq * rinv;
    const float dvx = vi.x - vj.x, dvy = vi.y - vj.y, dvz = vi.z - vj.z;
    const float dot = fmaf(dz, dvz, yx ? fmaf(dx, dvx, dy * dvy) : fmaf(dy, dvy, dx * dvx));
    const float wc = 1.f - r * c.rcinv;
    const float xi = pair_gaussian(__float_as_uint(vi.w), __float_as_uint(vj.w));
    // sigma / sqrt(dt): uniform for a one-type system away from walls
    const float sdt = c.sigma * dtis;
    float fpair, en = 0.f, eg = 1.f;
    if (STYLE == STYLE_MDPD) {
        // pair_mdpd_meso.cu:156-191: F = [A wc + B (rho_i + rho_j) wr
        //   - gamma wc^2 (dx.dv)/r + sigma wc xi / sqrt(dt)] / r, evaluated as
        // [wc (A + sigma' xi - gamma wc (dx.dv)/r) + B (rho_i + rho_j) wr] / r
        const float wcr = fmaxf(1.f - r * c.rdinv, 0.f);
        const float rr = rho_i + rho_j;
        float t = fmaf(sdt, xi, c.a);
        t = fmaf(-(c.gamma * wc * rinv), dot, t);
        fpair = fmaf(c.b * rr, wcr, t * wc) * rinv;
        if (EV) en = 0.5f * c.a * c.rc * wc * wc + 0.5f * c.b * c.rd * rr * wcr * wcr;
    } else {
        // pair_dpd_meso.cu:145-175: F = [a0 wc - gamma wr^2 (dx.dv)/r
        //   + sigma wr xi / sqrt(dt)] / r, evaluated as
        // [a0 wc + wr (sigma' xi - gamma wr (dx.dv)/r)] / r
        const float wr = c.expw == 1.f ? wc : powf(wc, c.expw);
        const float t = fmaf(-(c.gamma * wr * rinv), dot, sdt * xi);
        fpair = fmaf(c.a, wc, wr * t) * rinv;
        if (EV) {
            en = 0.5f * c.a * c.rc * wc;
            if (TEST) en = en * wc;
            else eg = wc;
        }
    }
    o.dx = dx; o.dy = dy; o.dz = dz;
    o.fpair = in ? fpair : 0.f;
    o.en = in ? en : 0.f;
    o.eg = eg;
    return o;
}

// a += the pair's terms.  The fused multiply-adds are spelled out: the two
// force kernels below sum the same pairs in the same order and must agree
// bit for bit.
template <bool EV>
__device__ inline void pair_add(Acc<EV> &a, const PairF &o)
{
    a.v[0] = fmaf(o.dx, o.fpair, a.v[0]);
    a.v[1] = fmaf(o.dy, o.fpair, a.v[1]);
    a.v[2] = fmaf(o.dz, o.fpair, a.v[2]);
    if (EV) {
        a.v[3] = fmaf(o.en, o.eg, a.v[3]);
        a.v[4] = fmaf(o.dx * o.dx, o.fpair, a.v[4]);
        a.v[5] = fmaf(o.dy * o.dy, o.fpair, a.v[5]);
        a.v[6] = fmaf(o.dz * o.dz, o.fpair, a.v[6]);
        a.v[7] = fmaf(o.dx * o.dy, o.fpair, a.v[7]);
        a.v[8] = fmaf(o.dx * o.dz, o.fpair, a.v[8]);
        a.v[9] = fmaf(o.dy * o.dz, o.fpair, a.v[9]);
    }
}

template <int STYLE, bool EV, bool TEST = true>
__device__ inline void pair_term(Acc<EV> &a, const float4 &pi, const float4 &vi, float rho_i, const float4 &q,
                                 const float4 &vj, float rho_j, uint32_t code, const PairC &c, float dtis,
                                 const SysDev *d, bool yx)
{
    pair_add<EV>(a, pair_eval<STYLE, EV, TEST>(pi, vi, rho_i, q, vj, rho_j, code, c, dtis, d, yx));
}

// Force of particle i known: its outputs (EV) and, in a stepping mode, the
// half-kicks, drift, next signature (SIG: already known, it reads no
// velocity) and displacement test.  Returns whether it moved past skin / 2.
template <int MODE, bool EV, bool STEP, bool SIG>
__device__ inline int finish_particle(const PoolDev &P, SysDev *d, int i, int cur, const float4 &pi, const float4 &vi,
                                      int ti, int mk, const Acc<EV> &a, uint32_t sig)
{
    float fx = a.v[0], fy = a.v[1], fz = a.v[2];
    if (mk & d->add_bit) { fx += d->add[0]; fy += d->add[1]; fz += d->add[2]; }
    if (EV) {
        P.frc[i] = make_float4(fx, fy, fz, 0.5f * a.v[3]);
        const size_t cap = (size_t)P.cap;
        P.vir[i] = 0.5f * a.v[4]; P.vir[cap + i] = 0.5f * a.v[5]; P.vir[2 * cap + i] = 0.5f * a.v[6];
        P.vir[3 * cap + i] = 0.5f * a.v[7]; P.vir[4 * cap + i] = 0.5f * a.v[8]; P.vir[5 * cap + i] = 0.5f * a.v[9];
    }
    if (STEP) {
        // which half-kicks this pass applies: the pooled engine decides per
        // system, the plain engine per launch
        const int ph = MODE == MODE_PHASED ? d->phase : (MODE == MODE_FINAL ? (int)PH_LAST : (int)PH_RUN);
        float vx = vi.x, vy = vi.y, vz = vi.z;
        float4 pn = pi;
        if ((mk & d->nve_bit) && ph != PH_FRESH) {
            const float dtfm = d->dtf * P.minv[d->mass_base + ti];
            vx += dtfm * fx; vy += dtfm * fy; vz += dtfm * fz;             // final_integrate
        }
        if (ph == PH_LAST) {
            P.pos[cur ^ 1][i] = pi;
            P.vel[cur ^ 1][i] = make_float4(vx, vy, vz, vi.w);
            P.vend[i] = make_float4(vx, vy, vz, 0.f);
            if (MODE == MODE_PHASED) P.frc[i] = make_float4(fx, fy, fz, 0.f);
        } else {
            if (MODE == MODE_FUSED_OUT) P.vend[i] = make_float4(vx, vy, vz, 0.f);
            if (mk & d->nve_bit) {
                const float dtfm = d->dtf * P.minv[d->mass_base + ti];
                vx += dtfm * fx; vy += dtfm * fy; vz += dtfm * fz;         // next initial_integrate
                pn.x += d->dt * vx; pn.y += d->dt * vy; pn.z += d->dt * vz;
            }
            const uint32_t sg = SIG ? sig : next_signature(d, P.tag[d->sela][i], vx, vy, vz);
            P.pos[cur ^ 1][i] = pn;
            P.vel[cur ^ 1][i] = make_float4(vx, vy, vz, __uint_as_float(sg));
            const float4 h = P.xhold[i];
            const float ex = pn.x - h.x, ey = pn.y - h.y, ez = pn.z - h.z;
            return fmaf(ez, ez, fmaf(ex, ex, ey * ey)) > d->trig2;
        }
    }
    return 0;
}

template <int STYLE, int MODE, bool UNI, int SPLIT>
__global__ void __launch_bounds__(WAVE * SPLIT)
    __attribute__((amdgpu_waves_per_eu(SPLIT > 1 && (MODE == MODE_FUSED || MODE == MODE_PHASED) ? 6 : 1))) k_force(PoolDev P, int tile0, int ntiles)
{
    // HARVEST re-evaluates the last pass of a finished pooled system from the
    // state that pass read, which its commit left in the other buffer; it
    // adds energy and virial and changes no state
    constexpr bool EV = MODE != MODE_FUSED && MODE != MODE_PHASED;
    constexpr bool STEP = MODE != MODE_SETUP && MODE != MODE_HARVEST;
    constexpr int NA = Acc<EV>::N;
    __shared__ float s_acc[SPLIT > 1 ? SPLIT - 1 : 1][NA][WAVE];
    // lane-balanced pair loop (see below): one wave per tile, one type
    constexpr bool BAL = SPLIT == 1 && UNI;
    constexpr int TAIL_CAP = BAL ? 192 : 1;
    __shared__ float4 s_pi[BAL ? WAVE : 1], s_vi[BAL ? WAVE : 1];
    __shared__ float s_ri[BAL ? WAVE : 1];
    __shared__ float s_tail[TAIL_CAP * NA];
    __shared__ int s_own[TAIL_CAP];
    // the same between a wave's sub-rows (two or four waves per tile)
    constexpr int NB = SPLIT > 1 ? SPLIT : 1, NL = SPLIT > 1 ? WAVE : 1;
    __shared__ float4 s_bp[NB][NL], s_bv[NB][NL], s_bt[NB][NL];
    __shared__ float s_br[NB][NL], s_bphi[NB][NL], s_be[EV ? NB : 1][EV ? NL : 1];
    constexpr bool EG = EV && en_factors(STYLE);
    __shared__ float s_bg[EG ? NB : 1][EG ? NL : 1];
    __shared__ int s_who[NB][NL];
    const int lt = xcd_logical(blockIdx.x, ntiles);
    if (lt >= ntiles) return;
    const int tile = tile0 + lt;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i = tile * WAVE + lane;
    const int s = tile_system(P, tile);
    if (s < 0) return;
    SysDev *d = P.sys + s;
    if (!d->active && MODE != MODE_HARVEST) return;
    if (UNI != (d->ntypes == 1)) return;     // host launches the matching variant
    // a system waiting for wider neighbor rows is skipped by the stepping
    // passes (no state change until the host has regrown the rows), and a
    // pool may mix styles: each launch takes the systems of its style
    if (STEP && d->overflow) return;
    if ((MODE == MODE_PHASED || MODE == MODE_HARVEST) && d->style != STYLE) return;
    // a finished system, at the split of its last pass
    if (MODE == MODE_HARVEST && (d->phase != PH_DONE || d->split_last != SPLIT)) return;
    const bool valid = i < d->part_base + d->n;
    const int cur = MODE == MODE_HARVEST ? d->sel ^ 1 : d->sel;
    const float4 *pos = P.pos[cur];
    const float4 *vel = P.vel[cur];
    const int *maskv = P.mask[d->sela];
    float4 pi = make_float4(0.f, 0.f, 0.f, 0.f), vi = pi;
    float rho_i = 0.f, phi_i = 0.f;
    int ti = 0, cnt = 0, mk = 0;
    if (valid) {
        pi = pos[i];
        vi = vel[i];
        ti = __float_as_int(pi.w);
        mk = maskv[i];
        if (STYLE == STYLE_MDPD) rho_i = P.rho[i];
        cnt = P.ccount[ccount_at(tile, w, lane)];
    }
    // arbitrary boundary: a mobile particle scales gamma / sigma of its pairs
    // with wall particles by its wall fraction (pair_mdpd_meso.cu:169-185)
    const bool arb_i = STYLE == STYLE_MDPD && d->pair_arb && (mk & d->pair_mobile_bit);
    if (arb_i) phi_i = P.phi[d->sela][i];
    const int wall_bit = d->pair_wall_bit;
    auto wall_scale_of = [&](PairC &c, uint32_t j, bool arb, float phi) {
        if (arb && (maskv[j] & wall_bit)) {
            const float ratio = wall_ratio(phi, c.rc);
            c.gamma *= ratio;
            c.sigma *= __builtin_amdgcn_sqrtf(ratio);
        }
    };
    auto wall_scale = [&](PairC &c, uint32_t j) { wall_scale_of(c, j, arb_i, phi_i); };
    const float dtis = d->dtinvsqrt;
    const float *coef = P.coef + d->coef_base;
    const int nt = d->ntypes;
    PairC cu;
    if (UNI) cu = load_coef(coef, 0);
    const int maxnbr = P.maxnbr;
    const int *crow = P.clist + (size_t)tile * maxnbr * WAVE + lane;
    Acc<EV> a;
    // pairs [t, end) of this lane's compact row, four gathers in flight (one
    // type) or two
    // neighbor j's position (q.w: its type bits, used by several types) and
    // density; one type of mDPD takes both from the first pass's x, y, z,
    // rho record with one 16-byte load
    auto nbr = [&](uint32_t j, float4 &q, float &rj) {
        if (UNI && STYLE == STYLE_MDPD) {
            q = P.pr[j];
            rj = q.w;
        } else {
            q = pos[j];
            rj = STYLE == STYLE_MDPD ? P.rho[j] : 0.f;
        }
    };
    auto walk = [&](int t, int end) {
        if (UNI) {
            for (; t + 4 <= end; t += 4) {
                uint32_t e[4], j[4];
                float4 q[4], vv[4];
                float rj[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    e[u] = (uint32_t)crow[(size_t)((t + u) * SPLIT + w) * WAVE];
                    j[u] = e[u] & IDX_MASK;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    nbr(j[u], q[u], rj[u]);
                    vv[u] = vel[j[u]];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    PairC c = cu;
                    wall_scale(c, j[u]);
                    pair_term<STYLE, EV, !UNI>(a, pi, vi, rho_i, q[u], vv[u], rj[u], e[u] >> IMG_SHIFT, c, dtis, d,
                                               false);
                }
            }
        }
        for (; t + 2 <= end; t += 2) {
            const uint32_t e0 = (uint32_t)crow[(size_t)(t * SPLIT + w) * WAVE];
            const uint32_t e1 = (uint32_t)crow[(size_t)((t + 1) * SPLIT + w) * WAVE];
            const uint32_t j0 = e0 & IDX_MASK, j1 = e1 & IDX_MASK;
            float4 q0, q1;
            float r0, r1;
            nbr(j0, q0, r0);
            nbr(j1, q1, r1);
            const float4 w0 = vel[j0], w1 = vel[j1];
            PairC c0 = UNI ? cu : load_coef(coef, ti * nt + __float_as_int(q0.w));
            PairC c1 = UNI ? cu : load_coef(coef, ti * nt + __float_as_int(q1.w));
            wall_scale(c0, j0);
            wall_scale(c1, j1);
            pair_term<STYLE, EV, !UNI>(a, pi, vi, rho_i, q0, w0, r0, e0 >> IMG_SHIFT, c0, dtis, d, false);
            pair_term<STYLE, EV, !UNI>(a, pi, vi, rho_i, q1, w1, r1, e1 >> IMG_SHIFT, c1, dtis, d, false);
        }
        if (t < end) {
            const uint32_t e0 = (uint32_t)crow[(size_t)(t * SPLIT + w) * WAVE];
            const uint32_t j0 = e0 & IDX_MASK;
            float4 q0;
            float r0;
            nbr(j0, q0, r0);
            PairC c0 = UNI ? cu : load_coef(coef, ti * nt + __float_as_int(q0.w));
            wall_scale(c0, j0);
            pair_term<STYLE, EV, !UNI>(a, pi, vi, rho_i, q0, vel[j0], r0, e0 >> IMG_SHIFT, c0, dtis, d, true);
        }
    };
    // Lane balance (one wave per tile, one type, no wall scaling): a wave
    // runs as long as its longest row, ~1.5x its mean row.  The first M
    // entries of every row (M: the mean row, raised until the rest fits
    // TAIL_CAP) are walked by their own lane; the entries past M, the tails,
    // laid out one after another in particle order, are dealt to all 64
    // lanes.  A tail pair's terms go to the LDS slot of its position, and
    // each particle adds its slots, in row order, after its own M entries.
    bool balanced = false;
    if constexpr (BAL) balanced = !(STYLE == STYLE_MDPD && d->pair_arb);
    if (balanced) {
        const int tot = wave_sum(cnt);
        int M = tot >> 6;
        int tail = wave_sum(max(cnt - M, 0));
        for (int it = 0; tail > TAIL_CAP && it < 4; ++it) {
            M += (tail - TAIL_CAP + WAVE - 1) / WAVE;
            tail = wave_sum(max(cnt - M, 0));
        }
        if (tail > TAIL_CAP) {          // rows too uneven: the longest row sets M
            M = wave_max(cnt);
            tail = 0;
        }
        walk(0, min(cnt, M));
        if (tail > 0) {
            const int sur = max(cnt - M, 0);
            const int first = wave_incl_scan(sur) - sur;     // this particle's first tail slot
            s_pi[lane] = pi;
            s_vi[lane] = vi;
            s_ri[lane] = rho_i;
            for (int f0 = 0; f0 < TAIL_CAP; f0 += WAVE) s_own[f0 + lane] = 0;
            __syncthreads();
            if (sur > 0) s_own[first] = lane;
            __syncthreads();
            const int *ctile = P.clist + (size_t)tile * maxnbr * WAVE;
            int carry = 0;
            for (int f0 = 0; f0 < tail; f0 += WAVE) {
                const int f = f0 + lane;
                // owner: the last particle whose tail starts at or before f,
                // spread from where the tails start (a search of six
                // shuffles per round takes four registers more)
                const int p = max(wave_scan(s_own[f], [](int x, int y) { return max(x, y); }), carry);
                carry = __builtin_amdgcn_readlane(p, 63);
                const int t = M + f - __shfl(first, p);
                const bool act = f < tail;
                // a lane past the last tail evaluates its own particle with
                // itself (r = 0: terms not finite) and stores nothing
                const uint32_t e = act ? (uint32_t)ctile[(size_t)t * WAVE + p]
                                       : ((uint32_t)i | ((uint32_t)IMG_ZERO << IMG_SHIFT));
                const uint32_t j = e & IDX_MASK;
                float4 q;
                float rj;
                nbr(j, q, rj);
                Acc<EV> b;
                pair_term<STYLE, EV, !UNI>(b, s_pi[p], s_vi[p], s_ri[p], q, vel[j], rj, e >> IMG_SHIFT, cu, dtis, d,
                                           true);
                if (act)
                    for (int k = 0; k < NA; ++k) s_tail[k * TAIL_CAP + f] = b.v[k];
            }
            __syncthreads();
            for (int f = first; f < first + sur; ++f)
                for (int k = 0; k < NA; ++k) a.v[k] += s_tail[k * TAIL_CAP + f];
        }
    } else if constexpr (SPLIT > 1) {
        // Two or four waves per tile: a wave's sub-rows are shorter and vary
        // more.  The first M entries (the mean, raised until at most one wave
        // of entries is left) are walked by their own lane, the rest dealt one
        // to a lane; their terms come back through LDS and are added in row
        // order with the same fused multiply-adds, so the sums are those of a
        // plain walk.  Instead of loops over fours, twos and ones down to the
        // longest row: 480,000 particles 126 -> 119 us, 122,000 (several
        // types, walls) 35 -> 32, 97,000 25 -> 23, 40,000 15.2 -> 14.9.
        // Reading a row past its end (to M, within the tile's rows: an even
        // number of them to each wave) needs no branch per entry.
        constexpr int B = UNI ? 4 : 2;      // pairs in flight
        int M = (wave_sum(cnt) + WAVE * 2 - 1) / (WAVE * 2) * 2;
        int tail = wave_sum(max(cnt - M, 0));
        while (tail > WAVE) {
            M += ((tail - 1) / WAVE + 1) / 2 * 2;
            tail = wave_sum(max(cnt - M, 0));
        }
        const uint32_t self = (uint32_t)i | ((uint32_t)IMG_ZERO << IMG_SHIFT);     // r = 0: not added
        for (int t = 0; t < M; t += B) {
            if (__builtin_amdgcn_ballot_w64(t < cnt) == 0) break;
            uint32_t e[B];
            float4 q[B], vv[B];
            float rj[B];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                if (t + u >= M) break;
                e[u] = (uint32_t)crow[(size_t)((t + u) * SPLIT + w) * WAVE];
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                if (t + u >= M) break;
                e[u] = t + u < cnt ? e[u] : self;
                nbr(e[u] & IDX_MASK, q[u], rj[u]);
                vv[u] = vel[e[u] & IDX_MASK];
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                if (t + u >= M) break;
                PairC c = UNI ? cu : load_coef(coef, ti * nt + (t + u < cnt ? __float_as_int(q[u].w) : 0));
                wall_scale(c, e[u] & IDX_MASK);
                const PairF o = pair_eval<STYLE, EV, !UNI>(pi, vi, rho_i, q[u], vv[u], rj[u], e[u] >> IMG_SHIFT, c,
                                                           dtis, d, u % 2 == 0 && t + u == cnt - 1);
                if (t + u < cnt) pair_add<EV>(a, o);
            }
        }
        if (tail > 0) {
            const int sur = max(cnt - M, 0);
            const int first = wave_incl_scan(sur) - sur;     // this particle's first tail entry
            s_bp[w][lane] = pi;
            s_bv[w][lane] = vi;
            s_br[w][lane] = rho_i;
            // wall_ratio takes no fraction past 1/2: 1 stands for a particle
            // whose pairs are not scaled (a bit of s_who for it takes a
            // register more, 65, and a wave per SIMD from several types: split
            // 4, 122,400 particles 31.7 -> 33.1 us)
            s_bphi[w][lane] = arb_i ? fminf(phi_i, 0.5f) : 1.f;
            // entry k of the tail: its particle, its row position, odd last entry
            for (int k = 0; k < sur; ++k)
                s_who[w][first + k] = lane | (M + k) << 6 | ((cnt & 1) && M + k == cnt - 1 ? 1 << 30 : 0);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const bool act = lane < tail;
            const int who = act ? s_who[w][lane] : lane, p = who & 63, t = who >> 6 & 0xFFFFFF;
            uint32_t e = self;
            if (act) e = (uint32_t)(crow - lane)[(size_t)(t * SPLIT + w) * WAVE + p];
            const uint32_t j = e & IDX_MASK;
            float4 q;
            float rj;
            nbr(j, q, rj);
            const float4 vj = vel[j], pp = s_bp[w][p];
            const float ph = s_bphi[w][p];
            PairC c = UNI ? cu : load_coef(coef, __float_as_int(pp.w) * nt + (act ? __float_as_int(q.w) : 0));
            wall_scale_of(c, j, ph <= 0.5f, ph);
            const PairF o = pair_eval<STYLE, EV, !UNI>(pp, s_bv[w][p], s_br[w][p], q, vj, rj, e >> IMG_SHIFT, c, dtis, d,
                                                       who >> 30 & 1);
            s_bt[w][lane] = make_float4(o.dx, o.dy, o.dz, o.fpair);
            if (EV) s_be[w][lane] = o.en;
            if (EG) s_bg[w][lane] = o.eg;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            for (int f = first; f < first + sur; ++f) {
                const float4 x = s_bt[w][f];
                pair_add<EV>(a, PairF{x.x, x.y, x.z, x.w, EV ? s_be[w][f] : 0.f, EG ? s_bg[w][f] : 1.f});
            }
        }
    } else {
        walk(0, cnt);
    }
    if (SPLIT > 1) {
        if (w > 0)
            for (int k = 0; k < NA; ++k) s_acc[w - 1][k][lane] = a.v[k];
        __syncthreads();
        if (w == 0)
            for (int q = 0; q < SPLIT - 1; ++q)
                for (int k = 0; k < NA; ++k) a.v[k] += s_acc[q][k][lane];
    }
    if (w > 0) return;
    int moved = 0;
    if (valid) moved = finish_particle<MODE, EV, STEP, false>(P, d, i, cur, pi, vi, ti, mk, a, 0u);
    if ((MODE == MODE_FUSED || MODE == MODE_FUSED_OUT || MODE == MODE_PHASED) && !d->fix_arb) flag_moved(d, moved);
}

// --------------------------------------------------------------------------
// The same pass with FW_WAVES waves sharing a tile's compact rows (split 2
// and 4): lane l of wave k evaluates particle l's pairs of rows k,
// k + FW_WAVES, ... (row t * SPLIT + w holds entry t of sub-row w), FW_ROWS
// of them with their gathers in flight at once, and leaves each pair's terms
// in LDS; then a wave per sub-row and force component adds them in row order,
// and the sub-rows' sums are added in order, so a particle's sum is that of a
// loop over its row.  One more wave computes the mDPD signatures of the next
// step meanwhile (they read only the tags).
// --------------------------------------------------------------------------
constexpr int FW_WAVES = 8, FW_ROWS = 5;

template <int STYLE, int MODE, bool UNI, int SPLIT>
__global__ void __launch_bounds__(WAVE * (FW_WAVES + 1)) k_force_wide(PoolDev P, int tile0, int ntiles)
{
    constexpr bool EV = MODE != MODE_FUSED && MODE != MODE_PHASED;
    constexpr bool STEP = MODE != MODE_SETUP && MODE != MODE_HARVEST;
    constexpr int NA = Acc<EV>::N;
    constexpr int R = FW_WAVES * FW_ROWS;              // rows per round
    constexpr int NU = EV ? SPLIT : 3 * SPLIT;         // sums: sub-row x component (EV: all components)
    constexpr int UPW = (NU + FW_WAVES - 1) / FW_WAVES;
    static_assert(FW_WAVES % SPLIT == 0, "a wave's rows belong to one sub-row");
    __shared__ float s_d[3][R][WAVE], s_f[R][WAVE];    // dx, dy, dz and F / r of each pair
    constexpr bool EG = EV && en_factors(STYLE);
    __shared__ float s_en[EV ? R : 1][WAVE], s_eg[EG ? R : 1][WAVE];
    __shared__ float s_acc[SPLIT][NA][WAVE];
    __shared__ uint32_t s_sig[WAVE];
    const int lt = xcd_logical(blockIdx.x, ntiles);
    if (lt >= ntiles) return;
    const int tile = tile0 + lt;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int i = tile * WAVE + lane;
    const int s = tile_system(P, tile);
    if (s < 0) return;
    SysDev *d = P.sys + s;
    if (!d->active && MODE != MODE_HARVEST) return;
    if (UNI != (d->ntypes == 1)) return;     // host launches the matching variant
    if (STEP && d->overflow) return;
    if ((MODE == MODE_PHASED || MODE == MODE_HARVEST) && d->style != STYLE) return;
    if (MODE == MODE_HARVEST && (d->phase != PH_DONE || d->split_last != SPLIT)) return;
    const bool valid = i < d->part_base + d->n;
    const int cur = MODE == MODE_HARVEST ? d->sel ^ 1 : d->sel;
    const float4 *pos = P.pos[cur];
    const float4 *vel = P.vel[cur];
    const int *maskv = P.mask[d->sela];
    int n[SPLIT];
#pragma unroll
    for (int w = 0; w < SPLIT; ++w) n[w] = valid ? P.ccount[ccount_at(tile, w, lane)] : 0;
    float4 pi = make_float4(0.f, 0.f, 0.f, 0.f), vi = pi;
    float rho_i = 0.f, phi_i = 0.f;
    int mk = 0;
    if (valid) {
        pi = pos[i];
        vi = vel[i];
        mk = maskv[i];
        if (STYLE == STYLE_MDPD) rho_i = P.rho[i];
    }
    if (wv == FW_WAVES && STEP && STYLE == STYLE_MDPD)
        s_sig[lane] = valid ? sig_mdpd(P.tag[d->sela][i], d->seed_next) : 0u;
    // a mobile particle's wall fraction scales its pairs with wall particles
    // (pair_mdpd_meso.cu:169-185)
    const bool arb_i = STYLE == STYLE_MDPD && d->pair_arb && (mk & d->pair_mobile_bit);
    if (arb_i) phi_i = P.phi[d->sela][i];
    const int ti = __float_as_int(pi.w);
    const float dtis = d->dtinvsqrt;
    const float *coef = P.coef + d->coef_base;
    const int nt = d->ntypes, wall_bit = d->pair_wall_bit;
    PairC cu;
    if (UNI) cu = load_coef(coef, 0);
    const int maxnbr = P.maxnbr;
    const int *crow = P.clist + (size_t)tile * maxnbr * WAVE + lane;
    int nmax = n[0], nw = n[0];
#pragma unroll
    for (int w = 1; w < SPLIT; ++w) {
        nmax = max(nmax, n[w]);
        nw = wv % SPLIT == w ? n[w] : nw;
    }
    Acc<EV> a;                                // EV: all components of one sub-row
    float sum[UPW];
#pragma unroll
    for (int k = 0; k < UPW; ++k) sum[k] = 0.f;
    for (int r0 = 0;; r0 += R) {
        if (wv < FW_WAVES) {
            uint32_t e[FW_ROWS];
            float4 q[FW_ROWS], vv[FW_ROWS];
            float rj[FW_ROWS];
#pragma unroll
            for (int u = 0; u < FW_ROWS; ++u) {
                const int r = r0 + u * FW_WAVES + wv;
                // a lane without this row takes itself (stored nowhere)
                e[u] = (uint32_t)i | ((uint32_t)IMG_ZERO << IMG_SHIFT);
                if (r / SPLIT < nw) e[u] = (uint32_t)crow[(size_t)r * WAVE];
            }
#pragma unroll
            for (int u = 0; u < FW_ROWS; ++u) {
                const uint32_t j = e[u] & IDX_MASK;
                if (UNI && STYLE == STYLE_MDPD) {
                    q[u] = P.pr[j];
                    rj[u] = q[u].w;
                } else {
                    q[u] = pos[j];
                    rj[u] = STYLE == STYLE_MDPD ? P.rho[j] : 0.f;
                }
                vv[u] = vel[j];
            }
#pragma unroll
            for (int u = 0; u < FW_ROWS; ++u) {
                const int r = r0 + u * FW_WAVES + wv;
                const bool on = r / SPLIT < nw;
                if (__builtin_amdgcn_ballot_w64(on) == 0) break;
                PairC c;
                if (UNI) c = cu;
                else c = load_coef(coef, ti * nt + (on ? __float_as_int(q[u].w) : 0));
                if (arb_i && (maskv[e[u] & IDX_MASK] & wall_bit)) {
                    const float ratio = wall_ratio(phi_i, c.rc);
                    c.gamma *= ratio;
                    c.sigma *= __builtin_amdgcn_sqrtf(ratio);
                }
                const PairF o = pair_eval<STYLE, EV, !UNI>(pi, vi, rho_i, q[u], vv[u], rj[u], e[u] >> IMG_SHIFT, c,
                                                           dtis, d, (nw & 1) && r / SPLIT == nw - 1);
                const int k = u * FW_WAVES + wv;
                s_d[0][k][lane] = o.dx;
                s_d[1][k][lane] = o.dy;
                s_d[2][k][lane] = o.dz;
                s_f[k][lane] = o.fpair;
                if (EV) s_en[k][lane] = o.en;
                if (EG) s_eg[k][lane] = o.eg;
            }
        }
        __syncthreads();
        if (EV) {
            if (wv < SPLIT)
                for (int k = wv; k < R && (r0 + k) / SPLIT < nw; k += SPLIT) {
                    PairF o;
                    o.dx = s_d[0][k][lane]; o.dy = s_d[1][k][lane]; o.dz = s_d[2][k][lane];
                    o.fpair = s_f[k][lane]; o.en = s_en[k][lane];
                    o.eg = EG ? s_eg[k][lane] : 1.f;
                    pair_add<EV>(a, o);
                }
        } else if (wv < FW_WAVES) {
#pragma unroll
            for (int y = 0; y < UPW; ++y) {
                // component comp of sub-row wv % SPLIT
                const int comp = (y * FW_WAVES + wv) / SPLIT;
                if (comp < 3)
                    for (int k0 = wv % SPLIT; k0 < R; k0 += 4 * SPLIT) {
                        if (__builtin_amdgcn_ballot_w64((r0 + k0) / SPLIT < nw) == 0) break;
                        float x[4], f[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const int k = min(k0 + u * SPLIT, R - 1);
                            x[u] = s_d[comp][k][lane];
                            f[u] = s_f[k][lane];
                        }
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const int k = k0 + u * SPLIT;
                            sum[y] = k < R && (r0 + k) / SPLIT < nw ? fmaf(x[u], f[u], sum[y]) : sum[y];
                        }
                    }
            }
        }
        if (__builtin_amdgcn_ballot_w64(nmax * SPLIT > r0 + R) == 0) break;
        __syncthreads();                      // the next round reuses the slots
    }
    if (EV) {
        if (wv < SPLIT)
            for (int k = 0; k < NA; ++k) s_acc[wv][k][lane] = a.v[k];
    } else if (wv < FW_WAVES) {
#pragma unroll
        for (int y = 0; y < UPW; ++y)
            if ((y * FW_WAVES + wv) / SPLIT < 3) s_acc[wv % SPLIT][(y * FW_WAVES + wv) / SPLIT][lane] = sum[y];
    }
    __syncthreads();
    if (wv > 0) return;
    for (int k = 0; k < NA; ++k) {
        a.v[k] = s_acc[0][k][lane];
#pragma unroll
        for (int w = 1; w < SPLIT; ++w) a.v[k] += s_acc[w][k][lane];
    }
    int moved = 0;
    if (valid)
        moved = finish_particle<MODE, EV, STEP, STYLE == STYLE_MDPD>(P, d, i, cur, pi, vi, ti, mk, a, s_sig[lane]);
    if ((MODE == MODE_FUSED || MODE == MODE_FUSED_OUT || MODE == MODE_PHASED) && !d->fix_arb) flag_moved(d, moved);
}

// --------------------------------------------------------------------------
// Wall branch of aboundary/rho/meso after the initial integrate
// (FixArbitraryBoundaryRho::post_integrate / gpu_aboundary,
// fix_aboundary_rho_meso.cu:220-317): wall fraction phi_i and wall normal of
// each mobile particle from the wall particles within cut_phi (every entry of
// its neighbor row, positions after the drift), bounce-back when
// phi_i > phi_c (v <- -v + 2 max(0, v.n) n, x <- x - v dtf/m + dt v_new),
// then the system's displacement flag from the final positions.  Works on the
// buffer the pass just wrote (sel ^ 1, before the step commit); one wave per
// 64-particle tile.  `pooled`: apply only to systems whose pass integrated.
// --------------------------------------------------------------------------
__global__ void __launch_bounds__(WAVE) k_aboundary(PoolDev P, int ntiles, int pooled)
{
    const int tile = xcd_logical(blockIdx.x, ntiles);
    if (tile >= ntiles) return;
    const int s = P.wave_sys[tile];
    if (s < 0) return;
    const SysDev *d = P.sys + s;
    if (!d->active || !d->fix_arb || d->overflow) return;
    if (pooled && d->phase == PH_LAST) return;
    const int lane = threadIdx.x;
    const int i = tile * WAVE + lane;
    const bool valid = i < d->part_base + d->n;
    const int sa = d->sela;
    float4 *pos = P.pos[d->sel ^ 1];
    float4 *vel = P.vel[d->sel ^ 1];
    const int *mask = P.mask[sa];
    int moved = 0;
    if (valid) {
        float4 p = pos[i];
        // the rows do not change between builds: the first wall pass after a
        // build records which of them hold a wall particle, and the later
        // passes skip the others (no wall neighbor: phi stays 0, no bounce)
        const bool fresh = d->ago == 0;
        if ((mask[i] & d->fix_mobile_bit) && (fresh || P.wall_near[i])) {
            const int maxnbr = P.maxnbr;
            const int cnt = min(P.ncount[i], maxnbr);
            int near = 0;
            const int4 *row4 = (const int4 *)(P.nlist + nbr_at(i, 0, maxnbr));
            const float c = d->cut_phi, c2 = c * c;
            const int wbit = d->fix_wall_bit;
            float phi = 0.f, nx = 0.f, ny = 0.f, nz = 0.f;
            // the row in chunks of eight entries, the next chunk's masks and
            // positions and the entries of the one after it loading meanwhile
            // (two waves per SIMD: nothing else hides the chain of entry,
            // mask, position; 122,000 particles 25 -> 18 us); terms added in
            // row order
            const int nch = (cnt + NBR_CHUNK - 1) / NBR_CHUNK;
            int4 ea = make_int4(0, 0, 0, 0), eb = ea;
            auto entries = [&](int ch) {
                if (ch < nch) {
                    ea = row4[(size_t)ch * (NBR_CHUNK * WAVE / 4)];
                    eb = row4[(size_t)ch * (NBR_CHUNK * WAVE / 4) + 1];
                }
            };
            uint32_t e[NBR_CHUNK];
            int m[NBR_CHUNK];
            float4 q[NBR_CHUNK];
            // past the row's end a lane takes itself, which is not a wall
            auto gather = [&](int ch, uint32_t *eo, int *mo, float4 *qo) {
                const uint32_t en[NBR_CHUNK] = {(uint32_t)ea.x, (uint32_t)ea.y, (uint32_t)ea.z, (uint32_t)ea.w,
                                                (uint32_t)eb.x, (uint32_t)eb.y, (uint32_t)eb.z, (uint32_t)eb.w};
#pragma unroll
                for (int k = 0; k < NBR_CHUNK; ++k) {
                    const bool in = ch * NBR_CHUNK + k < cnt;
                    eo[k] = in ? en[k] : (uint32_t)i;
                    mo[k] = mask[eo[k] & IDX_MASK];
                    qo[k] = pos[eo[k] & IDX_MASK];
                    if (!in) mo[k] = 0;
                }
            };
            entries(0);
            gather(0, e, m, q);
            entries(1);
            for (int ch = 0; ch < nch; ++ch) {
                uint32_t e1[NBR_CHUNK];
                int m1[NBR_CHUNK];
                float4 q1[NBR_CHUNK];
                gather(ch + 1, e1, m1, q1);
                entries(ch + 2);
#pragma unroll
                for (int k = 0; k < NBR_CHUNK; ++k) {
                    if (!(m[k] & wbit)) continue;
                    near = 1;
                    float dx, dy, dz;
                    pair_delta(p, q[k], e[k] >> IMG_SHIFT, d, dx, dy, dz);
                    const float rsq = dx * dx + dy * dy + dz * dz;
                    if (!(rsq < c2)) continue;
                    const float rinv = __builtin_amdgcn_rsqf(rsq);
                    const float r = fmaxf(rsq * rinv, 1e-10f);
                    const float dd = c - r;
                    phi += (c + 3.f * r) * dd * dd * dd * d->phi_factor;
                    const float g = r * dd * dd * d->dw_factor * rinv;
                    nx -= g * dx; ny -= g * dy; nz -= g * dz;
                }
#pragma unroll
                for (int k = 0; k < NBR_CHUNK; ++k) {
                    e[k] = e1[k];
                    m[k] = m1[k];
                    q[k] = q1[k];
                }
            }
            if (fresh) P.wall_near[i] = near;
            P.phi[sa][i] = phi;
            if (phi > d->phi_c) {
                const float inv = __builtin_amdgcn_rsqf(nx * nx + ny * ny + nz * nz);
                nx *= inv; ny *= inv; nz *= inv;
                float4 v = vel[i];
                const float dtfm = d->dtf * P.minv[d->mass_base + __float_as_int(p.w)];
                const float ox = p.x - v.x * dtfm, oy = p.y - v.y * dtfm, oz = p.z - v.z * dtfm;
                const float tmp = fmaxf(0.f, v.x * nx + v.y * ny + v.z * nz);
                v.x = -v.x + 2.f * tmp * nx;
                v.y = -v.y + 2.f * tmp * ny;
                v.z = -v.z + 2.f * tmp * nz;
                p.x = ox + d->dt * v.x;
                p.y = oy + d->dt * v.y;
                p.z = oz + d->dt * v.z;
                if (d->style == STYLE_DPD)      // the DPD signature reads v
                    v.w = __uint_as_float(sig_dpd(P.tag[sa][i], d->seed_next, v.x, v.y, v.z));
                pos[i] = p;
                vel[i] = v;
            }
        }
        const float4 h = P.xhold[i];
        const float ex = p.x - h.x, ey = p.y - h.y, ez = p.z - h.z;
        moved = ex * ex + ey * ey + ez * ez > d->trig2;
    }
    flag_moved(P.sys + s, moved);
}

// --------------------------------------------------------------------------
// Step commit, one thread per system, after a pass that wrote the other
// buffer: FINAL (end-of-run half-kick) only flips the buffer; DECIDE (plain
// engine) and PHASED (pooled engine) also advance the step and the seed and
// make the reneighbor decision of Neighbor::decide (src/neighbor.cpp:
// 1216-1290) on the device: after `ago` steps since the last build, rebuild
// when ago >= delay, ago % every == 0 and (no check, or a particle moved more
// than skin/2 since the last build); PHASED also follows each system's
// lifecycle.  A system whose rows overflowed was skipped by the pass and is
// not advanced.  Between the steps of one graph the next rebuild phase makes
// the commit instead (launch_rebuild): a launch of one workgroup costs every
// step 2 to 3 us whatever it does (97,000 particles: a step 94 -> 91.4 us,
// 40,000 particles 59.4 -> 57.7).
// --------------------------------------------------------------------------
__global__ void __launch_bounds__(WAVE) k_commit_step(PoolDev P, int kind, int split, int seeded)
{
    const int s = blockIdx.x * WAVE + threadIdx.x;
    if (s < P.nsys) commit_system(P, s, kind, split, seeded);
}

// --------------------------------------------------------------------------
// Admission: one launch unpacks the input blocks of up to ADMIT_LIST submitted
// systems (blockIdx.y: one of the list), read in place from the pinned host
// memory they were packed in, and derives the rest (creation indices, owners
// of tiles and cell slots, cleared counts).  A launch per system reads 350 KB
// of a droplet in 16 us, latency for the most part; sixteen together take 123
// us, 46 GB/s (256 droplets: 4.1 -> 2.0 ms).
// --------------------------------------------------------------------------
constexpr int ADMIT_LIST = 16;
struct AdmitList {
    AdmitItem item[ADMIT_LIST];
};

__global__ void __launch_bounds__(256) k_admit(PoolDev P, AdmitList list)
{
    const AdmitItem &a = list.item[blockIdx.y];
    const InLayout &in = a.in;
    const char *src = a.block;
    const int s = a.slot, pb = a.part_base, cb = a.cell_base;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0) {
        const SysDev *d = (const SysDev *)(src + in.sys);
        const int *w = (const int *)d;
        int *o = (int *)(P.sys + s);
        for (int q = threadIdx.x; q < (int)(sizeof(SysDev) / 4); q += blockDim.x) o[q] = w[q];
        const float *cf = (const float *)(src + in.coef), *ms = (const float *)(src + in.mass);
        const int c0 = s * MAXTYPES * MAXTYPES * NCOEF, m0 = s * MAXTYPES;
        for (int q = threadIdx.x; q < in.ncoef; q += blockDim.x) P.coef[c0 + q] = cf[q];
        for (int q = threadIdx.x; q < in.nt; q += blockDim.x) {
            P.mass[m0 + q] = ms[q];
            P.minv[m0 + q] = ms[in.nt + q];
        }
    }
    if (k < in.nc1) {
        P.cell_rank[cb + k] = ((const int *)(src + in.rank))[k];
        P.cell_xyz[cb + k] = ((const int *)(src + in.xyz))[k];
        P.cell_sys[cb + k] = s;
        for (int q = 0; q < SUBCELLS; ++q) P.cell_count[(cb + k) * SUBCELLS + q] = 0;
    }
    if (k < in.npad / WAVE) P.wave_sys[pb / WAVE + k] = s;
    if (k >= in.npad) return;
    const int i = pb + k;
    const bool live = k < in.n;                            // padding slots are inert
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f), v = x;
    if (live) {
        x = ((const float4 *)(src + in.pos))[k];
        const float *u = (const float *)(src + in.vel) + 3 * (size_t)k;
        v = make_float4(u[0], u[1], u[2], 0.f);
    }
    P.pos[0][i] = x;
    P.vel[0][i] = v;
    P.tag[0][i] = live ? ((const int *)(src + in.tag))[k] : 0;
    P.mask[0][i] = live ? ((const int *)(src + in.mask))[k] : 0;
    P.origin[0][i] = live ? k : -1;
    P.image[0][i] = live ? ((const int *)(src + in.image))[k] : 512 | (512 << 10) | (512 << 20);
    P.phi[0][i] = live && in.has_phi ? ((const float *)(src + in.phi))[k] : 0.f;
}

// --------------------------------------------------------------------------
// Finished pooled systems (blockIdx.y: one of the list): current state, last
// force evaluation and descriptor packed into one block in the system's own
// neighbor-row range, which no pass reads once it has stopped (x, v, f | tag,
// mask, image | rho, virial | SysDev, each array npad long, in creation
// order), so the host copies one range.  Runs after the HARVEST force pass,
// which reads the other buffer.  The system's tiles and cell slots are
// unmapped here (no kernel after it finds the system through them); the host
// frees the ranges once the copy has landed.  A creation index outside the
// system would leave a slot of the block unwritten: it is reported in `bad`.
// --------------------------------------------------------------------------
constexpr int HARVEST_LIST = 64;
struct HarvestList {
    int slot[HARVEST_LIST];
};

__global__ void __launch_bounds__(256) k_harvest(PoolDev P, HarvestList list, int *bad)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const SysDev *d = P.sys + list.slot[blockIdx.y];
    const int pb = d->part_base, npad = d->npad;
    char *dst = (char *)(P.nlist + (size_t)pb * P.maxnbr);
    if (blockIdx.x == 0) {
        const int *src = (const int *)d;
        int *o = (int *)(dst + (size_t)npad * HARVEST_SLOT_BYTES);
        for (int w = threadIdx.x; w < (int)(sizeof(SysDev) / 4); w += blockDim.x) o[w] = src[w];
    }
    for (int c = k, nc = d->ncell + 1; c < nc; c += gridDim.x * blockDim.x) P.cell_sys[d->cell_base + c] = -1;
    if (k < npad / WAVE) P.wave_sys[pb / WAVE + k] = -1;
    if (k >= d->n) return;
    const int i = pb + k, cur = d->sel, cura = d->sela;
    const int c = P.origin[cura][i];                          // creation index
    if (c < 0 || c >= d->n) {
        bad[list.slot[blockIdx.y]] = 1;
        return;
    }
    const size_t n = npad;
    float4 *o4 = (float4 *)dst;
    o4[c] = P.pos[cur][i];
    o4[n + c] = P.vel[cur][i];
    o4[2 * n + c] = P.frc[i];
    int *oi = (int *)(o4 + 3 * n);
    oi[c] = P.tag[cura][i];
    oi[n + c] = P.mask[cura][i];
    oi[2 * n + c] = P.image[cura][i];
    float *of = (float *)(oi + 3 * n);
    of[c] = P.rho[i];
#pragma unroll
    for (int m = 0; m < 6; ++m) of[(m + 1) * n + c] = P.vir[(size_t)m * P.cap + i];
}

// --------------------------------------------------------------------------
// One system's per-atom quantity in creation order (the host copies one block
// and only widens it).
// --------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_gather(PoolDev P, int field, int *out, int *bad)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const SysDev *d = P.sys;
    if (i >= d->n) return;
    const int sel = d->sel, sela = d->sela;
    const int c = P.origin[sela][i];
    if (c < 0 || c >= d->n) {
        *bad = 1;
        return;
    }
    float *of = (float *)out;
    auto put3 = [&](const float4 &q) { of[3 * c] = q.x; of[3 * c + 1] = q.y; of[3 * c + 2] = q.z; };
    switch (field) {
    case G_X: put3(P.pos[sel][i]); break;
    case G_V: put3(P.vel[sel][i]); break;
    case G_F: put3(P.frc[i]); break;
    case G_EPAIR: of[c] = P.frc[i].w; break;
    case G_RHO: of[c] = P.rho[i]; break;
    case G_PHI: of[c] = P.phi[sela][i]; break;
    case G_VIRIAL:
        for (int m = 0; m < 6; ++m) of[6 * c + m] = P.vir[(size_t)m * P.cap + i];
        break;
    case G_TAG: out[c] = P.tag[sela][i]; break;
    case G_TYPE: out[c] = __float_as_int(P.pos[sel][i].w) + 1; break;
    case G_MASK: out[c] = P.mask[sela][i]; break;
    case G_IMAGE: {
        const int im = P.image[sela][i];
        out[3 * c] = (im & 1023) - 512;
        out[3 * c + 1] = ((im >> 10) & 1023) - 512;
        out[3 * c + 2] = ((im >> 20) & 1023) - 512;
        break;
    }
    }
}

// --------------------------------------------------------------------------
// stateless helpers (parity tests)
// --------------------------------------------------------------------------
__global__ void k_pair_gaussian(const uint32_t *a, const uint32_t *b, float *out, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = pair_gaussian(a[i], b[i]);
}

__global__ void k_premix(const uint32_t *a, const uint32_t *b, uint32_t *out, int n, int rounds)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t v0 = a[i], v1 = b[i];
    tea_rounds(v0, v1, rounds);
    out[i] = v0 ^ v1;
}

// ----------------------------------------------------------------------------
// launchers
// ----------------------------------------------------------------------------
// Tiles up to which a split of 2 or 4 takes the wide kernels: two of their
// workgroups per CU, all of them resident at once.  A short launch is one
// tile's chain of loads and of ~6.5 cycles per dependent instruction, which
// the wide kernels cut (16 tiles: first pass 10.9 -> 6.8 us, force pass 12.5
// -> 7.3 us; 500 tiles of the DPD fluid: step 1.04x faster); past that their
// tiles queue and the two-wave kernels' occupancy wins (626 tiles: 13.4 and
// 15.3 us against 13.2 and 16.3; 1,513 tiles: step 0.89x).
constexpr int WIDE_TILES = 512;

bool first_seeds(int split, int nt) { return split == 1 || nt <= WIDE_TILES; }

template <bool WITH_RHO>
static hipError_t launch_first_t(const PoolDev &P, int split, int nt, hipStream_t st)
{
    const int ns = first_seeds(split, nt) ? seed_grid(P) : 0;       // seed workgroups, then the tiles
    const dim3 g(ns + xcd_grid(nt));
    const bool wide = nt <= WIDE_TILES;
    if (split == 1)
        hipLaunchKernelGGL((k_first<WITH_RHO, 1>), g, dim3(WAVE), 0, st, P, nt, ns);
    else if (split == 2 && wide)
        hipLaunchKernelGGL((k_first_wide<WITH_RHO, 2>), g, dim3(WAVE * FS_WAVES<2>), 0, st, P, nt, ns);
    else if (split == 2)
        hipLaunchKernelGGL((k_first<WITH_RHO, 2>), g, dim3(WAVE * 2), 0, st, P, nt, ns);
    else if (split == 4 && wide)
        hipLaunchKernelGGL((k_first_wide<WITH_RHO, 4>), g, dim3(WAVE * FS_WAVES<4>), 0, st, P, nt, ns);
    else if (split == 4)
        hipLaunchKernelGGL((k_first<WITH_RHO, 4>), g, dim3(WAVE * 4), 0, st, P, nt, ns);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_first(const PoolDev &P, bool with_rho, int split, hipStream_t st)
{
    const int nt = P.nact / WAVE;
    if (nt == 0) return hipSuccess;
    if (P.maxnbr % NBR_ALIGN) return hipErrorInvalidValue;   // a split wave's compact rows must fit
    return with_rho ? launch_first_t<true>(P, split, nt, st) : launch_first_t<false>(P, split, nt, st);
}

hipError_t launch_commit_step(const PoolDev &P, int kind, int split, bool after_pass, hipStream_t st)
{
    if (P.nsys == 0) return hipSuccess;
    const int seeded = after_pass && (P.one || first_seeds(split, P.nact / WAVE)) ? 1 : 0;
    hipLaunchKernelGGL(k_commit_step, dim3((P.nsys + WAVE - 1) / WAVE), dim3(WAVE), 0, st, P, kind, split, seeded);
    return hipGetLastError();
}

hipError_t launch_aboundary(const PoolDev &P, int pooled, hipStream_t st)
{
    const int nt = P.nact / WAVE;
    if (nt == 0) return hipSuccess;
    hipLaunchKernelGGL(k_aboundary, dim3(xcd_grid(nt)), dim3(WAVE), 0, st, P, nt, pooled);
    return hipGetLastError();
}

hipError_t launch_admit(const PoolDev &P, const AdmitItem *items, int count, hipStream_t st)
{
    static_assert(sizeof(PoolDev) + sizeof(AdmitList) <= 4096, "kernel arguments");
    for (int q0 = 0; q0 < count; q0 += ADMIT_LIST) {
        const int m = count - q0 < ADMIT_LIST ? count - q0 : ADMIT_LIST;
        AdmitList list;
        int threads = 0;
        for (int q = 0; q < ADMIT_LIST; ++q) {
            const AdmitItem &a = items[q0 + (q < m ? q : 0)];
            const InLayout &in = a.in;
            if (!a.block || a.slot < 0 || a.part_base < 0 || a.part_base % 256 || in.npad % 256 || in.n > in.npad ||
                a.part_base + in.npad > P.cap || a.cell_base < 0 || a.cell_base + in.nc1 > P.ncellslots ||
                in.ncoef > MAXTYPES * MAXTYPES * NCOEF || in.nt > MAXTYPES)
                return hipErrorInvalidValue;
            list.item[q] = a;
            threads = std::max(threads, std::max(in.npad, in.nc1));
        }
        hipLaunchKernelGGL(k_admit, dim3((threads + 255) / 256, m), dim3(256), 0, st, P, list);
    }
    return hipGetLastError();
}

hipError_t launch_harvest(const PoolDev &P, const int *slots, int count, int npad_max, int *bad, hipStream_t st)
{
    // the packed block fits the rows: maxnbr entries per slot, at least NBR_ALIGN
    static_assert(sizeof(SysDev) <= 256 * (4 * NBR_ALIGN - HARVEST_SLOT_BYTES), "harvest block fits the rows");
    if (P.maxnbr < NBR_ALIGN || npad_max <= 0 || npad_max > P.cap || !bad) return hipErrorInvalidValue;
    for (int q0 = 0; q0 < count; q0 += HARVEST_LIST) {
        HarvestList list{};
        const int m = count - q0 < HARVEST_LIST ? count - q0 : HARVEST_LIST;
        for (int q = 0; q < m; ++q) {
            list.slot[q] = slots[q0 + q];
            if (list.slot[q] < 0 || list.slot[q] >= P.nsys) return hipErrorInvalidValue;
        }
        hipLaunchKernelGGL(k_harvest, dim3((npad_max + 255) / 256, m), dim3(256), 0, st, P, list, bad);
    }
    return hipGetLastError();
}

hipError_t launch_gather(const PoolDev &P, int field, int *out, int *bad, hipStream_t st)
{
    if (!P.one || field < G_X || field > G_IMAGE || !out || !bad) return hipErrorInvalidValue;
    if (P.nact == 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather, dim3((P.nact + 255) / 256), dim3(256), 0, st, P, field, out, bad);
    return hipGetLastError();
}

hipError_t launch_initial(const PoolDev &P, hipStream_t st)
{
    const int nl = P.nact / BLK;
    if (nl == 0) return hipSuccess;
    hipLaunchKernelGGL(k_initial, dim3(xcd_grid(nl)), dim3(BLK), 0, st, P, nl);
    return hipGetLastError();
}

template <int STYLE, int MODE, bool UNI>
static hipError_t launch_force_t(const PoolDev &P, int split, int t0, int nt, hipStream_t st)
{
    const dim3 g(xcd_grid(nt)), bw(WAVE * (FW_WAVES + 1));
    const bool wide = nt <= WIDE_TILES;
    if (split == 1)
        hipLaunchKernelGGL((k_force<STYLE, MODE, UNI, 1>), g, dim3(WAVE), 0, st, P, t0, nt);
    else if (split == 2 && wide)
        hipLaunchKernelGGL((k_force_wide<STYLE, MODE, UNI, 2>), g, bw, 0, st, P, t0, nt);
    else if (split == 2)
        hipLaunchKernelGGL((k_force<STYLE, MODE, UNI, 2>), g, dim3(WAVE * 2), 0, st, P, t0, nt);
    else if (split == 4 && wide)
        hipLaunchKernelGGL((k_force_wide<STYLE, MODE, UNI, 4>), g, bw, 0, st, P, t0, nt);
    else if (split == 4)
        hipLaunchKernelGGL((k_force<STYLE, MODE, UNI, 4>), g, dim3(WAVE * 4), 0, st, P, t0, nt);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

template <int STYLE, int MODE>
static hipError_t launch_force_s(const PoolDev &P, bool uni, int split, int t0, int nt, hipStream_t st)
{
    return uni ? launch_force_t<STYLE, MODE, true>(P, split, t0, nt, st)
               : launch_force_t<STYLE, MODE, false>(P, split, t0, nt, st);
}

hipError_t launch_force(const PoolDev &P, int style, int mode, bool uni, int split, hipStream_t st)
{
    return launch_force_range(P, style, mode, uni, split, 0, P.nact / WAVE, st);
}

hipError_t launch_force_range(const PoolDev &P, int style, int mode, bool uni, int split, int t0, int nt,
                              hipStream_t st)
{
    if (nt <= 0) return hipSuccess;
    if (t0 < 0 || t0 + nt > P.cap / WAVE) return hipErrorInvalidValue;
#define MDPD_FORCE_CASE(S, M) \
    if (style == S && mode == M) return launch_force_s<S, M>(P, uni, split, t0, nt, st);
    MDPD_FORCE_CASE(STYLE_MDPD, MODE_SETUP)
    MDPD_FORCE_CASE(STYLE_MDPD, MODE_FUSED)
    MDPD_FORCE_CASE(STYLE_MDPD, MODE_FUSED_OUT)
    MDPD_FORCE_CASE(STYLE_MDPD, MODE_FINAL)
    MDPD_FORCE_CASE(STYLE_MDPD, MODE_PHASED)
    MDPD_FORCE_CASE(STYLE_MDPD, MODE_HARVEST)
    MDPD_FORCE_CASE(STYLE_DPD, MODE_SETUP)
    MDPD_FORCE_CASE(STYLE_DPD, MODE_FUSED)
    MDPD_FORCE_CASE(STYLE_DPD, MODE_FUSED_OUT)
    MDPD_FORCE_CASE(STYLE_DPD, MODE_FINAL)
    MDPD_FORCE_CASE(STYLE_DPD, MODE_PHASED)
    MDPD_FORCE_CASE(STYLE_DPD, MODE_HARVEST)
#undef MDPD_FORCE_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_pair_gaussian(const uint32_t *a, const uint32_t *b, float *out, int n, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_pair_gaussian, dim3((n + 255) / 256), dim3(256), 0, st, a, b, out, n);
    return hipGetLastError();
}

hipError_t launch_premix(const uint32_t *a, const uint32_t *b, uint32_t *out, int n, int rounds, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_premix, dim3((n + 255) / 256), dim3(256), 0, st, a, b, out, n, rounds);
    return hipGetLastError();
}

}  // namespace mdpd
