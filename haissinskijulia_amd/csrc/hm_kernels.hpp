// hm_kernels.hpp -- launch wrappers of the gfx950 kernels (hm_kernels.hip).
// Every wrapper checks nothing itself: the engine validates shapes and
// buffer sizes before it calls one.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hm_types.hpp"

namespace hm {

constexpr int kPassThreads = 1024;     // turn-pass / moments / interp-sum block
constexpr int kConvThreads = 256;      // convolution block
constexpr int kConvMaxThreads = 1024;  // and the largest, for long transforms
constexpr int kConvInvThreads = 1024;  // phase-B convolution block (spectral sums in flight)
constexpr int kFinalThreads = 256;     // per-bunch set-up and moment blocks
// Per-bunch reductions of the per-wave tile sums: each workgroup sums one
// slice of kRedEntries entries (kRedPer per thread); the last slice of a bunch
// to finish adds the slice sums in order.
constexpr int kRedThreads = 256;
constexpr int kRedPer = 4;
constexpr int kRedEntries = kRedThreads * kRedPer;
constexpr int kInterpThreads = 1024;   // LDS-staged interpolation sums
// partial sums per tile are kept per wave of the 1024-thread pass and
// interpolation-sum workgroups: part[ntiles][kTileWaves][4], ipart[ntiles][kTileWaves]
constexpr int kTileWaves = 16;
static_assert(kPassThreads == 64 * kTileWaves && kInterpThreads == 64 * kTileWaves,
              "per-wave tile sums assume 1024-thread workgroups");
// slices of the reductions of a bunch with ntiles tiles
inline int red_slices(int ntiles) {
    const int e = (ntiles > 0 ? ntiles : 1) * kTileWaves;
    return (e + kRedEntries - 1) / kRedEntries;
}
constexpr int kMaxFFT = 8192;          // largest LDS FFT (128 KiB of complex FP64)
constexpr int kAutoFFTBlock = 1024;    // default convolution block (F = 2048)

// CONV_SPEC + CONV_OUT replace CONV_INV where the spectra of a frequency
// chunk fit the LDS (conv_spec_fits)
enum ConvKind { CONV_FUSED = 0, CONV_FWD = 1, CONV_INV = 2, CONV_SPEC = 3, CONV_OUT = 4 };
constexpr int kConvKinds = 5;
// Frequencies per CONV_SPEC workgroup, 1 to 16 (F and the result are powers of
// two, so the chunks tile F): one (frequency, output block) pair per thread of
// 256 threads, of up to 1024 where 256 workgroups remain -- two frequencies are
// a quarter of a cache line (131072 bins, 128 blocks: 13.8 -> 10.6 us by eight).
__host__ __device__ inline int spec_chunk(int nA, int F) {
    int c = 16;
    while (c > 1 && (c > F || c * nA > kConvMaxThreads || (c * nA > kConvThreads && F / c < 256)))
        c >>= 1;
    return c;
}
inline size_t conv_spec_lds(int nA, int nJ, int F) {
    return (size_t)(nA + nJ) * (size_t)spec_chunk(nA, F) * 16;
}
inline bool conv_spec_fits(int nA, int nJ, int F, int lds_max) {
    return conv_spec_lds(nA, nJ, F) + 1024 <= (size_t)lds_max;
}

// zero `bytes` (a multiple of 4) at p by a kernel (no memset node: callers may
// capture the stream)
hipError_t launch_zero(void *p, size_t bytes, hipStream_t s);
// Up to kCopyList copies of 4-byte words between pinned host and device memory
// by one kernel, which reads and writes the host's memory itself; a piece
// without a source is cleared.  A copy call or a launch each took about 4 us of
// the host and 2 to 3 of the stream, a pageable copy 15 to 25: a call of 4000
// particles and 10 turns took 476 us with them, 370 so.
constexpr int kCopyList = 32;
struct CopyList {
    struct {
        void *dst;
        const void *src;
        uint32_t words;
    } e[kCopyList];
};
hipError_t launch_copies(const CopyList &l, int n, hipStream_t s);

// allow the dynamic-LDS kernels the device's LDS per block (best effort)
hipError_t configure_kernels(int max_dynamic_lds);

// per-tile sums of z, z^2, dE, dE^2; mode 1 first applies the pending wake
// kick and re-centre (the epilogue of the last turn)
hipError_t launch_moments(const BunchDev *bds, const int32_t *tile_bunch, int ntiles, int mode,
                          int grid, int lds_entries, hipStream_t s);
// per-bunch spreads from the tile sums; mode 0 -> out[0..1], mode 1 -> out[2..8]
hipError_t launch_moments_final(const BunchDev *bds, const int32_t *bunch_list, int nb, int mode,
                                hipStream_t s);
hipError_t launch_init(const BunchDev *bds, const int32_t *bunch_list, int nb, hipStream_t s);
// `grid` workgroups over the tile order, workgroup g taking the runs
// [rr[g], rr[g+1]); lds_bytes = the largest per-bunch histogram + potential
// window; std_only: every bunch has (flags & kPhysMask) == kStdFlags, two bins
// or more and (F_GHIST) hwin > 0; unb: some bunch's particles not binned are
// counted (BunchDev::unb); keep_z: z stays in the caches (Batch::keep_z_)
hipError_t launch_turn_pass(const BunchDev *bds, const int32_t *order, const RunDev *runs,
                            const int32_t *rr, int grid, int slices, size_t lds, int std_only,
                            int unb, bool keep_z, hipStream_t s);
// `turns` turns of bunches without a wake and without the E0 update: items
// cover the listed bunches' pairs
constexpr int kFreeThreads = 256;
hipError_t launch_free_turns(const BunchDev *bds, const RunDev *items, int nitems,
                             const int32_t *bunch_list, int nlist, int turns, hipStream_t s);
// items are (bunch, block) pairs, for CONV_SPEC (bunch, frequency chunk)
// pairs; Fmax is the largest FFT length among them, for CONV_SPEC the largest
// conv_spec_lds of their bunches in bytes
hipError_t launch_conv(int kind, const BunchDev *bds, const int32_t *items, int nitems, int Fmax,
                       hipStream_t s, int threads = kConvThreads);
// interpolation sums of the wake + update_E0 bunches: `grid` workgroups over
// their tile order (runs as for the pass); lds_bytes = 8 x the largest iwin;
// deep: one workgroup per CU, eight streaming loads in flight per thread
hipError_t launch_interp_sum(const BunchDev *bds, const int32_t *order, const RunDev *runs,
                             const int32_t *rr, int grid, size_t lds_bytes, bool deep,
                             bool keep_z, hipStream_t s);
// the slabs of the windowed histograms added up: items are (bunch, group of 512
// bins of its window) pairs
hipError_t launch_hist_slabs(const BunchDev *bds, const int32_t *items, int nitems, hipStream_t s);
// per-bunch reduction of the pass's tile sums into the turn scalars (sum of
// dE'-dE_init; sigma_z, current, binned count, centroid cell of a wake bunch),
// and of the interpolation sums into the E0 update.  items holds nitems
// (bunch, slice) pairs, red_slices(ntiles) slices per bunch.
// launch_reduce_fwd: the pass's sums, and phase A of the convolutions of the
// nitems (bunch, block) items
hipError_t launch_reduce_fwd(const BunchDev *bds, const int32_t *red, int nred, const int32_t *items,
                             int nitems, int Fmax, hipStream_t s);
hipError_t launch_finalize(const BunchDev *bds, const int32_t *items, int nitems, hipStream_t s);
// the same bits with one 1024-thread workgroup per listed bunch and no
// cross-workgroup count; lds: 8 bytes per bin of the largest grid with a deposit
hipError_t launch_finalize_whole(const BunchDev *bds, const int32_t *bunch_list, int nb, size_t lds,
                                 hipStream_t s);
// The whole bin phase (the reduction, the convolution and the finalize) of
// each listed bunch in one 1024-thread workgroup: the same bits as the
// launches of those phases.  For bunches of at most kBinWholeMaxTiles tiles
// without interpolation sums; lds = the largest bin_whole_layout(...).bytes
// among them.
constexpr int kBinWholeMaxTiles = 256;
// LDS of k_bin_whole for one bunch (byte offsets, 16-aligned): the
// convolution's X[nA][F] (and for nJ > 1 FFT(W)[nJ][F] and Y[nA][F]), then
// for a wake bunch this turn's counts[nb], the line-density kernel[nb], the
// potential[nb] and the FFT twiddles[F/2], then for a deposit bunch its
// hi/lo[2 nb] and n[nb + 1].
struct BinWholeLayout {
    size_t hist, lam, pot, tw, cic, bytes;
};
__host__ __device__ inline size_t align16(size_t b) { return (b + 15) & ~(size_t)15; }
__host__ __device__ inline BinWholeLayout bin_whole_layout(int nb, int nA, int nJ, int F,
                                                           bool cic) {
    BinWholeLayout L;
    const size_t conv = nb > 0 ? (size_t)(nJ <= 1 ? nA : 2 * nA + nJ) * (size_t)F * 16 : 0;
    L.hist = conv;
    L.lam = L.hist + align16((size_t)nb * 4);
    L.pot = L.lam + align16((size_t)nb * 8);
    L.tw = L.pot + align16((size_t)nb * 8);   // double2: every region starts 16-aligned
    L.cic = L.tw + (nb > 0 ? (size_t)(F / 2) * 16 : 0);
    L.bytes = L.cic + (cic ? align16((size_t)nb * 16 + ((size_t)nb + 1) * 4) : 0);
    return L;
}
hipError_t launch_bin_whole(const BunchDev *bds, const int32_t *bunch_list, int nb, size_t lds,
                            hipStream_t s);
// The same for the bunches that fit k_bin_64's arrangement: blocks of 64 bins
// (what the tuned table gives 256 to 1024 bins), at most 16 of them, a wake of
// more than one block (one block has nothing to sum), at most four reduction
// slices, and the whole potential in the pass's window `win` (k_bin_64 leaves
// the neighbour-pair table out).  Same bits; in a turn 9.4 us against 17.7 us
// at 1024 bins, 7.7 against 12.7 us at 512.  Its LDS fits in
// bin_whole_layout(...).bytes.
inline bool fits_bin_64(bool wake, int nbins, int win, int nA, int nJ, int F, int nred) {
    return wake && F == 128 && nbins >= 2 && nA <= 16 && nJ > 1 && nJ <= 16 && nred <= 4 && win >= nbins;
}
hipError_t launch_bin_64(const BunchDev *bds, const int32_t *bunch_list, int nb, size_t lds,
                         hipStream_t s);
// Broadband resonators of a lag-indexed wake table, (R_s [Ohm], f_r [Hz], Q)
// each, passed by value.
constexpr int kMaxResonators = 8;
struct ResonatorSet {
    int32_t n;
    double Rs[kMaxResonators], fr[kMaxResonators], Q[kMaxResonators];
};
// W[j] = sum of the resonators' wakes at s = j * step, j < nb
hipError_t launch_resonator_table(double *W, int nb, double step, const ResonatorSet &rs,
                                  hipStream_t s);
// the reference's W(c) and delta kernel of the bin centres (either may be NULL;
// nb < 2^28, 1e-200 < zw <= 1e300)
hipError_t launch_reference_tables(double *W, double *lam, int nb, double zw, double wf, double ws,
                                   double inv_ctau, double s_inv, double ef, hipStream_t s);
// FFT of the wake blocks: What[j] = FFT_F(W[jB .. jB+B) zero-padded)
hipError_t launch_fft_wake(const BunchDev *bd_dev, const double *W, int nJ, int F,
                           hipStream_t s);

// stage kernels (unit parity entry points)
hipError_t launch_stage_rf(double V, double sphis, double rf, double phis, const double *z,
                           double *dE, int64_t n, hipStream_t s);
hipError_t launch_stage_qe(double exc, const double *r, double *dE, int64_t n, hipStream_t s);
hipError_t launch_stage_sr(double damp, double *dE, int64_t n, hipStream_t s);
hipError_t launch_stage_drift(int update_eta, const TurnScalars *sc_dev, double mass,
                              double alpha_c, double phis, double *z, const double *dE, int64_t n,
                              hipStream_t s);
hipError_t launch_stage_hist(const double *z, int64_t n, double e_first, double e_last,
                             double inv_step, int nb, uint32_t *hist, int use_lds, hipStream_t s);
hipError_t launch_stage_interp_kick(const double *z, double *dE, int64_t n, const double *P,
                                    double c0, double c1, double inv, int nb, hipStream_t s);
hipError_t launch_stage_normals(uint64_t seed, int64_t turn, int64_t i0, int64_t n, double *out,
                                hipStream_t s);
hipError_t launch_generate(uint64_t seed, double mu_z, double sz, double mu_E, double sE,
                           double *z, double *dE, int64_t n, hipStream_t s);
hipError_t launch_turn_scalars(const BunchDev *bd_dev, double E0, TurnScalars *out,
                               hipStream_t s);
// two-pass statistics of device arrays z, dE (n >= 2): stats[0..4] = (mean z,
// mean dE, std z, std dE, cor(z, dE)); part holds 3 * kStatBlocks doubles
constexpr int kStatBlocks = 1024;
hipError_t launch_pair_stats(const double *z, const double *dE, int64_t n, double *stats,
                             double *part, hipStream_t s);
// generate_particles for n >= 2 (sample-covariance MvNormal): writes z, dE,
// work[0..2] = Cholesky factor (l11, l21, l22) and the pair statistics of
// the bunch at work[4..8]; work holds kGenWorkDoubles doubles
constexpr int kGenWorkDoubles = 12 + 3 * kStatBlocks;
hipError_t launch_generate_particles(uint64_t seed, double mu_z, double mu_E, double sz, double sE,
                                     double *z, double *dE, int64_t n, double *work,
                                     hipStream_t s);
// device-to-device copy of n doubles (n even) by a plain grid-stride kernel
hipError_t launch_stream_copy(const double *src, double *dst, int64_t n, int blocks, hipStream_t s);

}  // namespace hm
