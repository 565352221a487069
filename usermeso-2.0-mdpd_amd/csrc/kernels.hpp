// Host-side launchers for the mdpd355 kernels.
#pragma once

#include "common.hpp"

namespace mdpd {

enum ForceMode : int {
    MODE_SETUP = 0,      // forces (+energy/virial) of the current state, no state change
    MODE_FUSED = 1,      // force, final half-kick, next initial half-kick + drift
    MODE_FUSED_OUT = 2,  // MODE_FUSED and also write f, e, virial, end-of-step v
    MODE_FINAL = 3,      // force and final half-kick only (end of a run)
    MODE_PHASED = 4,     // pooled engine: each system follows its own SysPhase
    MODE_HARVEST = 5,    // pooled engine, finished system: f, e, virial of its last pass
};

// rebuild phase: wrap, keys, sort, gather, neighbor rows, commit (stale systems only)
// split: of the pass that follows; commit: the commit that the pass before,
// at the same split, has left to this phase (its CommitKind after_pass), or 0
hipError_t launch_rebuild(const PoolDev &P, int split, int commit, hipStream_t st);
// particle slots up to which one system that re-sorts every `period` steps is
// better off with the one-launch sort
int sort_one_limit(int period);
hipError_t launch_nlist_only(const PoolDev &P, hipStream_t st);
// neighbor rows of every sorted active system rebuilt in place (row width grew)
hipError_t launch_relist(const PoolDev &P, hipStream_t st);
hipError_t launch_signatures(const PoolDev &P, hipStream_t st);
// one system: its sort keys at the last build, in sorted order
hipError_t launch_sort_keys(const PoolDev &P, unsigned long long *out, hipStream_t st);

// per step
// first pass of a step: density (mDPD with the density fix) and compact rows
hipError_t launch_first(const PoolDev &P, bool with_rho, int split, hipStream_t st);
hipError_t launch_initial(const PoolDev &P, hipStream_t st);
// after launch_initial or a force pass
// kind: CommitKind; split = waves per tile of the pass; after_pass: a rebuild
// phase and a first pass of that split have run since the last commit
hipError_t launch_commit_step(const PoolDev &P, int kind, int split, bool after_pass, hipStream_t st);
// whether a first pass of this split over nt tiles computes the seeds the
// step's commit moves on to; otherwise, for one system, the row build does
bool first_seeds(int split, int nt);
hipError_t launch_force(const PoolDev &P, int style, int mode, bool uni, int split, hipStream_t st);
// the same over the 64-particle tiles [tile0, tile0 + ntiles) only
hipError_t launch_force_range(const PoolDev &P, int style, int mode, bool uni, int split, int tile0, int ntiles,
                              hipStream_t st);
// wall branch of aboundary/rho/meso (wall fraction, bounce-back, displacement
// flags) on the buffer a pass just wrote; pooled: only systems that integrated
hipError_t launch_aboundary(const PoolDev &P, int pooled, hipStream_t st);
// pooled engine: a submitted system's input block (InLayout, readable from the
// device) unpacked into slots [part_base, + npad) and cell slots [cell_base,
// + nc1) of buffer 0, descriptor slot s
struct InLayout {
    size_t pos, vel, tag, mask, image, phi, rank, xyz, coef, mass, sys, bytes;
    int n, npad, nc1, ncoef, nt, has_phi;
    InLayout() = default;
    InLayout(int n_, int npad_, int nc1_, int ncoef_, int nt_, bool phi_)
        : n(n_), npad(npad_), nc1(nc1_), ncoef(ncoef_), nt(nt_), has_phi(phi_ ? 1 : 0)
    {
        size_t at = 0;
        auto take = [&](size_t b) { const size_t o = at; at += (b + 15) / 16 * 16; return o; };
        pos = take(sizeof(float4) * n);
        vel = take(sizeof(float) * 3 * n);
        tag = take(sizeof(int) * n);
        mask = take(sizeof(int) * n);
        image = take(sizeof(int) * n);
        phi = take(has_phi ? sizeof(float) * n : 0);
        rank = take(sizeof(int) * nc1);
        xyz = take(sizeof(int) * nc1);
        coef = take(sizeof(float) * ncoef);
        mass = take(sizeof(float) * 2 * nt);            // m, 1 / m
        sys = take(sizeof(SysDev));
        bytes = at;
    }
};
// a submitted system on its way in: block (InLayout, readable from the
// device), descriptor slot, first particle and cell slot
struct AdmitItem {
    InLayout in;
    const char *block;
    int slot, part_base, cell_base;
};
hipError_t launch_admit(const PoolDev &P, const AdmitItem *items, int count, hipStream_t st);

// pooled engine, finished systems in descriptor slots[0 .. count): each one's
// results in creation order, packed at the start of its own neighbor-row range
// (harvest_dst), harvest_bytes(npad) bytes:
//   float4 x[npad] | float4 v[npad] | float4 f[npad] (w: pair energy) |
//   int tag[npad], mask[npad], image[npad] | float rho[npad] |
//   float virial[6][npad] | SysDev
constexpr size_t HARVEST_SLOT_BYTES = 3 * 16 + 3 * 4 + 4 + 6 * 4;
inline size_t harvest_bytes(size_t npad) { return npad * HARVEST_SLOT_BYTES + sizeof(SysDev); }
inline size_t harvest_dst(const PoolDev &P, int part_base) { return (size_t)part_base * P.maxnbr; }
// bad: a word per descriptor slot, writable from the device; set to 1 when a
// particle of that system has no valid creation index (its results are not whole)
hipError_t launch_harvest(const PoolDev &P, const int *slots, int count, int npad_max, int *bad, hipStream_t st);

// one system: a per-atom quantity in creation order, gather_words(field) 4-byte
// words per particle (floats, or ints from G_TAG on; image unpacked, type 1-based)
enum GatherField : int { G_X = 0, G_V, G_F, G_EPAIR, G_RHO, G_PHI, G_VIRIAL, G_TAG, G_TYPE, G_MASK, G_IMAGE };
constexpr int gather_words(int field)
{
    return field == G_X || field == G_V || field == G_F || field == G_IMAGE ? 3 : field == G_VIRIAL ? 6 : 1;
}
// bad: one word, as for launch_harvest
hipError_t launch_gather(const PoolDev &P, int field, int *out, int *bad, hipStream_t st);

// observables (accumulate into device histograms of nbin + 1 slots, slot nbin
// counting the samples; a system whose rows overflowed is not sampled)
hipError_t launch_rdf(const PoolDev &P, unsigned *hist, int nbin, float rc, int gi, int gj, hipStream_t st);
hipError_t launch_profile(const PoolDev &P, unsigned *count, int nbin, int axis, int g, hipStream_t st);
// rdf/fast/meso and density/meso of every pooled system that has them and
// samples this pass
hipError_t launch_obs_pool(const PoolDev &P, hipStream_t st);

// stateless helpers for parity tests
hipError_t launch_pair_gaussian(const uint32_t *a, const uint32_t *b, float *out, int n, hipStream_t st);
hipError_t launch_premix(const uint32_t *a, const uint32_t *b, uint32_t *out, int n, int rounds, hipStream_t st);

}  // namespace mdpd
