// hm_types.hpp -- layouts shared by the host engine and the gfx950 kernels.
//
// Device memory layout of one bunch (all FP64 unless noted):
//   z[n], dE[n]                 particle state, SoA (data_structures.jl:26-29)
//   hist[2][nbins] (uint32)     line-density counts; turn t fills half t&1 while
//                               the bin phase clears the other half
//   P[nbins]                    wake potential at the bin centres (previous turn)
//   P2[nbins][2]                the same as neighbour pairs, one 16-byte gather per particle
//   lam[nbins]                  delta(c_i, 0.15) line-density kernel (wakefield.jl:219-221)
//   What[nJ][F]   (complex)     FFT of the wake blocks, fixed for one evolve call
//   X[nA][F]      (complex)     FFT of the packed line-density blocks of a turn
//   Y[nA][F]      (complex)     their products with the wake spectra, summed
//                               per output block (before its inverse FFT)
//   part[ntiles][16][4]         per-wave sums of each tile (sum z, sum z^2,
//                               sum dE'-dE_init, particles not binned)
//   ipart[ntiles][16]           per-wave sums of each tile of the interpolated
//                               potential (E0 update)
//   moments[ntiles][4]          per-tile sums of z, z^2, dE, dE^2 (initial / final spreads)
//   red[nred][4]                slice sums of the per-bunch reductions, and cnt
//                               (uint32), the slices of the running reduction
//                               counted in so far (zero between reductions)
//   sc                          TurnScalars of the current turn
//   out[8]                      sigma_E0, sigma_z0, sigma_E, sigma_z, E0, ...
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hm_rules.hpp"

namespace hm {

constexpr double kTwoPi = 6.283185307179586;   // Julia's 2π as Float64
constexpr double kPi = 3.141592653589793;
constexpr double kSpeedLight = 299792458.0;    // src/constants.jl:5

enum BunchFlags : uint32_t {
    F_WAKE = 1u,       // use_wakefield
    F_ETA = 2u,        // update_eta
    F_E0 = 4u,         // update_E0
    F_SR = 8u,         // SR_damping
    F_QE = 16u,        // use_excitation
    F_INJ = 32u,       // injected normals instead of Philox
    F_CHARGE = 64u,    // fixed wake current (charge extension / stage entry)
    F_GHIST = 128u,    // the histogram is not whole in LDS: hwin of its bins are, or none
    F_LAG = 256u,      // wake table by lag behind the source: bin k feels bins k+j (causal)
    F_CIC = 512u,      // the pass deposits the interpolation weights of the new z (cic)
    F_CACHED = 1024u,  // z and dE of a windowed histogram's bunch go through the caches
};

// Cloud-in-cell deposit (F_CIC).  The E0 update needs sum_i interp(P_t, z_i)
// over the post-drift z of turn t, with P_t known only after the histogram of
// those z.  The interpolation is linear in P: with (k_i, w_i) the cell and
// weight of z_i, the sum is sum_k (N_k - S_k) P_t[k] + S_k P_t[k+1], where
// N_k counts the particles of cell k and S_k adds their weights.  The pass
// adds W_i = round(w_i 2^51): integer sums, so they do not depend on the order
// of the additions, and 2^-52 of a weight is as fine as the weight's own FP64
// rounding.  In LDS a cell is a pair of 64-bit counters: N_k (from bit
// kCicCountBit) with the sum of W >> 32, and the sum of W's low words, so a
// particle costs two atomics at one address; the count's field bounds a run
// to kCicRunPairs pairs between two flushes.  In global memory: hi[nbins],
// lo[nbins] (64-bit; the flush carries lo's high word into hi, so lo stays
// exact in a double), then n[nbins + 1] (32-bit; n[nbins] counts NaN
// positions).
constexpr double kCicScale = 2251799813685248.0;   // 2^51
constexpr int kCicCountBit = 42;
constexpr int64_t kCicRunPairs = (int64_t)1 << 20;

// the all-physics-on configuration the turn pass is specialised for, and the
// flags that select the pass's code path
constexpr uint32_t kStdFlags = F_WAKE | F_ETA | F_E0 | F_SR | F_QE;
constexpr uint32_t kPhysMask = F_WAKE | F_ETA | F_E0 | F_SR | F_QE | F_INJ;

// Slots of the count of a turn's particles that are not binned: one 64-byte
// line each, so that the pass's workgroups (one addition per run at most) do
// not queue at one address.
constexpr int kUnbSlots = 64;

// Scalars of one turn of one bunch (evolution.jl:300-304 plus the pending
// state of the fused pass).  Written by k_init / k_finalize, read by the
// per-particle kernels.
struct TurnScalars {
    double E0, gamma0, beta0, eta0, rf;
    double inv_rf;     // 1/rf (the phase-to-z conversion, utils.jl:476)
    double denom;      // (beta0*beta0)*E0, drift denominator (evolution.jl:338)
    double kcoef;      // (2 pi h)/denom: the phase coefficient is eta * kcoef
    double coeff_c;    // constant-eta phase coefficient (evolution.jl:157)
    double damp;       // 1 - dU/dE (synchrotron_radiation.jl:44-45)
    double exc;        // sqrt(1-(1-dU/dE)^2) * sigma_E0 (quantum_excitation.jl:58-59)
    double m_prev;     // mean energy change still to subtract (evolution.jl:429-434)
    double sigma_z, current, n_h;   // bin phase of this turn (wake bunches)
    double sum_dE;     // sum over the bunch of dE'-dE_init of this turn (evolution.jl:419-429)
    int32_t pending_kick;   // 1: the previous turn's wake kick is still to be applied
    int32_t pending_m;      // 1: m_prev still to be subtracted
    int32_t drift_skip;     // apply_phase_advance! skip condition of this turn
    int32_t drift_skipped_count;
    int64_t turn;           // turns completed in this call
    int32_t centre_bin;     // interpolation cell of this turn's centroid: the LDS windows
                            // of P are placed around it (placement changes no result)
    int32_t pad_;
};

struct BunchDev {
    double *z, *dE;
    int64_t n, npairs;
    int64_t pairs_per_tile;
    int32_t tile_begin, ntiles;
    uint32_t flags;
    int32_t nbins;
    // physics constants of the call
    double mass, inv_mass, voltage, alpha_c, phis, sin_phis, radius, freq_rf, two_pi_h;
    double sigma_E0;   // initial energy spread (drives QE and the wake current)
    double pf;         // particle factor of evolution.jl:377-383 (depends on n only)
    double charge;     // fixed current when F_CHARGE
    double E0_init;
    uint64_t seed;
    int64_t turn_offset;
    const double *normals;   // device, [turns][n] when F_INJ
    // histogram / interpolation grids (evolution.jl:270-274, wakefield.jl:38-42)
    double e_first, e_last, inv_step;
    double c_first, c_last, inv_s;
    double u_last;        // (c_last - c_first) * inv_s: the interpolation coordinate of the last centre
    uint32_t *hist;       // [2][hist_half]: half (turn & 1) is this turn's, bin b at spread32
    double *P;
    double *P2;           // interleaved pairs (P[k], P[k+1]), k < nbins (P[nbins] := 0)
    const double *lam;
    const double *What;   // interleaved complex [nJ][F][2]
    const double *tw;     // interleaved complex [F/2][2], exp(-2 pi i k / F)
    double *X;            // interleaved complex [nA][F][2]: FFT(g_a + i g_{a-1}) (nJ > 1)
    double *Y;            // interleaved complex [nA][F][2]: sum_j X_{o-j} FFT(W_j), or null
    int32_t B, F, logF, nA, nJ;
    int32_t win;          // entries of P the pass stages in LDS (0: all gathers global)
    int32_t iwin;         // entries of P the interpolation sums stage in LDS
    double *part, *ipart, *moments, *out;
    double *red;          // [nred][4]
    uint32_t *cnt;
    int32_t nred;
    int32_t hwin;         // F_GHIST: bins counted in LDS (even; 0: all in global memory)
    int32_t nslabs;       // F_GHIST with hwin: the bunch's runs, one slab of counts each
    uint32_t *slabs;      // [nslabs][hwin / 2], two 16-bit counts per word
    int32_t cic_off;      // F_CIC: byte offset of the pass's LDS deposit
    int32_t cic_tiles;    // F_CIC: tiles of a run between two flushes of the deposit
    TurnScalars *sc;
    double *mon;          // device [n_turns][4] turn monitor or null
    int32_t spread;            // where counter i of hist and cic lies: spread32, spread64
    unsigned long long *cic;   // F_CIC: this turn's deposit (cic_* below; zero between turns)
    uint32_t *unb;             // [2][kUnbSlots][16]: this turn's particles not binned, behind hist;
                               // null where no k_reduce_fwd reads them
};

// The counters that every workgroup of the pass adds to (histogram, deposit)
// use the first 128 of every 256 bytes where spreads_counters says so
// (BunchDev::spread is ~31, else 0).
__host__ __device__ inline int spread32(int spread, int i) { return i + (i & spread); }
__host__ __device__ inline int spread64(int spread, int i) { return i + (i & (spread >> 1)); }
// 32-bit words of one half of a histogram, 64-bit words of a deposit's hi or lo
__host__ __device__ inline int hist_half(int nbins) { return (nbins + 31) / 32 * 64; }
__host__ __device__ inline int cic_half(int nbins) { return (nbins + 15) / 16 * 32; }
// the deposit: hi, lo (64-bit), then n (32-bit) and the count of NaN positions
__host__ __device__ inline size_t cic_words(int nbins) {
    return 2 * (size_t)cic_half(nbins) + (size_t)hist_half(nbins) / 2 + 1;
}

// A run of a workgroup: `count` consecutive entries, from `begin`, of a tile
// order, all of one bunch; its slab of the bunch's windowed histogram.
struct RunDev {
    int32_t bunch, begin, count, slab;
};

// LDS of a turn-pass workgroup for one bunch: its histogram (nbins counts, with
// F_GHIST hwin 16-bit ones), then a window of `win` entries of the previous turn's
// potential, P[lo .. lo+win), for the wake-kick gathers, then with F_CIC the
// deposit's counters at cic_off.
__host__ __device__ inline int pass_hist_bytes(const BunchDev &B) {
    if (!(B.flags & F_WAKE)) return 0;
    return (((B.flags & F_GHIST) ? B.hwin * 2 : B.nbins * 4) + 15) & ~15;
}

__host__ __device__ inline int cic_bytes(int nbins) { return 16 * nbins; }
__host__ __device__ inline int pass_cic_bytes(const BunchDev &B) {
    return (B.flags & F_CIC) ? cic_bytes(B.nbins) : 0;
}
// the pass's dynamic LDS for one bunch
__host__ __device__ inline int pass_lds_bytes(const BunchDev &B) {
    return (B.flags & F_CIC) ? B.cic_off + pass_cic_bytes(B) : pass_hist_bytes(B) + 8 * B.win;
}

// first entry of a window of w entries of P centred on `centre`; even, so that
// the window is read by 16-byte loads
__host__ __device__ inline int window_lo(int centre, int w, int nbins) {
    const int lo = centre - w / 2;
    return (lo < 0 ? 0 : (lo > nbins - w ? nbins - w : lo)) & ~1;
}

}  // namespace hm
