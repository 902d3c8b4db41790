// hm_kernels.hip -- gfx950 kernels of the longitudinal turn loop.
//
// One turn of the reference (src/evolution.jl:295-456) is, per bunch:
//   k_turn_pass   one coalesced read and write of (z, dE) per particle:
//                 the previous turn's wake kick and E0 re-centre, then RF kick
//                 (rf_kick.jl:84-87), quantum excitation (quantum_excitation.jl
//                 :58-71), SR damping (synchrotron_radiation.jl:44-56) and the
//                 drift (evolution.jl:330-347); it bins the new z into an
//                 LDS-privatised histogram (utils.jl:351-401) and writes
//                 deterministic per-wave partial sums of each tile.
//   k_reduce_fwd  one workgroup per slice of 1024 of those sums; the last
//                 slice of a bunch to finish adds the slice sums in order:
//                 sigma_z, the wake current (evolution.jl:373-386), the
//                 binned count and the sum of the energy changes; beside
//                 them the line density's blocks transformed.
//   k_conv_*      the rest of the line-density convolution with the wake
//                 (wakefield.jl:186-319) by blocked LDS FFTs.
//   k_interp_sum  (update_E0 with the wake) sum of the interpolated potential
//                 over the post-drift z, which the E0 update of
//                 evolution.jl:404-435 needs before the next turn.
//   k_finalize    E0 update and the scalars of the next turn.
//
// All floating-point work is FP64.  Multiplies and adds of the per-particle path
// are never contracted (-ffp-contract=off); fused ones are written out in the
// elementary functions (hm_math.hpp, bm_radius) and in steps that are exact or
// round once by them (the uniforms, the deposit's weights, the bin centres).
// Divides by per-turn constants are multiplies by their reciprocals.  Sums are
// reduced in a fixed order, so a run is bitwise reproducible.
#include <hip/hip_runtime.h>
#include <math.h>

#include "hm_kernels.hpp"

// a*b + k with the polynomial constant k in scalar registers.  Written as
// plain fma, the compiler keeps the ~30 constants of the pass in vector
// registers and copies one into the accumulator before every v_fmac; this
// form needs no copy and leaves the vector registers to the particles.
__device__ __forceinline__ double fma_sk(double a, double b, double k) {
    double d;
    asm("v_fma_f64 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(b), "s"(k));
    return d;
}
#define HM_QUAL __device__ __forceinline__
#define HM_FMAK(a, b, k) ::fma_sk(a, b, k)
#include "hm_math.hpp"

namespace hm {

struct DevOps {
    static __device__ __forceinline__ double rcp(double a) { return __builtin_amdgcn_rcp(a); }
    static __device__ __forceinline__ double frexp_mant(double u) {
        return __builtin_amdgcn_frexp_mant(u);
    }
    static __device__ __forceinline__ int frexp_exp(double u) { return __builtin_amdgcn_frexp_exp(u); }
};

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------

__host__ __device__ inline double jl_max(double a, double b) {
    // Julia's max for floats: NaN wins
    if (a != a) return a;
    if (b != b) return b;
    return (b > a) ? b : a;
}

// compute_global_std from reduced sums (utils.jl:589-605)
__device__ inline double gstd_from_sums(double s, double s2, double nd) {
    const int64_t n = (int64_t)nd;
    if (n <= 1) return 0.0;
    const double mean = s / (double)n;
    const double var = (s2 / (double)n) - (mean * mean);
    return sqrt(jl_max(0.0, var * (double)n / (double)(n - 1)));
}

// Scalars of a turn from the current E0 (evolution.jl:300-304,157;
// synchrotron_radiation.jl:44-45; quantum_excitation.jl:58-59).
__device__ inline void turn_scalars(const BunchDev &B, double E0, TurnScalars &s) {
    s.E0 = E0;
    s.gamma0 = E0 / B.mass;
    const double ig2 = 1.0 / (s.gamma0 * s.gamma0);
    s.beta0 = sqrt(jl_max(0.0, 1.0 - ig2));
    s.eta0 = B.alpha_c - ig2;
    s.rf = (s.beta0 <= 0.0) ? INFINITY : (B.freq_rf * kTwoPi) / (s.beta0 * kSpeedLight);
    s.inv_rf = 1.0 / s.rf;
    s.denom = (s.beta0 * s.beta0) * E0;
    s.kcoef = B.two_pi_h / s.denom;
    s.coeff_c = (B.two_pi_h * s.eta0) / s.denom;
    const double x = E0 / 1e9;
    const double d = ((4.0 * 8.85e-5) * ((x * x) * x)) / B.radius;
    s.damp = 1.0 - d;
    const double om = 1.0 - d;
    s.exc = sqrt(1.0 - (om * om)) * B.sigma_E0;
    s.drift_skip = (!(B.flags & F_ETA)) && (s.beta0 <= 0.0 || E0 == 0.0 || s.rf == 0.0);
}

// sin for the RF kick; arguments far from the bucket (|x| >= 2^19) go to the
// device library, out of line so the common path keeps its registers
__device__ __noinline__ double sin_far(double x) { return sin(x); }

__device__ __forceinline__ double dsin(double x) {
    if (__builtin_expect(!(__builtin_fabs(x) < fm::kReduceMax), 0)) return sin_far(x);
    return fm::sin_reduced(x);
}

// Physics flags of a pass: FX != 0 fixes them at compile time (the common
// all-on configuration), FX == 0 reads them from the bunch.
template <uint32_t FX>
struct Flags {
    uint32_t rt;
    __device__ __forceinline__ bool has(uint32_t f) const {
        return FX ? ((FX & f) != 0) : ((rt & f) != 0);
    }
};

// Philox4x32-10 (Salmon et al., SC'11); the 32x32 -> 64 products give the
// high and low words in one multiply.  Forced inline: with constant or
// wave-uniform counter words the first rounds' products are scalar or leave
// the loop.
__device__ __forceinline__ void philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                              uint32_t k0, uint32_t k1, uint32_t x[4]) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
        const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
        // three-input xor in one instruction (truth table 0x96 = a ^ b ^ c)
        const uint32_t n0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c1, k0, 0x96);
        const uint32_t n2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c3, k1, 0x96);
        c1 = (uint32_t)p1;
        c3 = (uint32_t)p0;
        c0 = n0;
        c2 = n2;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
        // the round keys are uniform: recomputed per round by scalar adds
        // rather than twenty of them held (and spilled) across the pass
        asm volatile("" : "+s"(k0), "+s"(k1));
    }
    x[0] = c0; x[1] = c1; x[2] = c2; x[3] = c3;
}

// sqrt(x) for the Box-Muller radius, 0 <= x <= 74 (u1 >= 2^-53): one
// Goldschmidt step from the hardware reciprocal-square-root estimate and one
// Newton correction, within an ulp of the rounded root.  x = 0 (u1 = 1) gives
// 2^-500 instead of 0.
__device__ __forceinline__ double bm_radius(double x) {
    x = __builtin_fmax(x, 0x1p-1000);
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = __builtin_fma(-h, g, 0.5);
    g = __builtin_fma(g, r, g);
    h = __builtin_fma(h, r, h);
    const double d = __builtin_fma(-g, g, x);
    return __builtin_fma(d, h, g);
}

// Box-Muller (1958) on one Philox block: u1 in (0,1], u2 in [0,1), 53 bits each
__device__ __forceinline__ void box_muller(const uint32_t x[4], double &n0, double &n1) {
    // (a 2^26 + b + 1) 2^-53 and (a 2^26 + b) 2^-53, every step exact
    const double u1 = __builtin_fma((double)(x[0] >> 5), 0x1p-27,
                                    __builtin_fma((double)(x[1] >> 6), 0x1p-53, 0x1p-53));
    const double u2 = __builtin_fma((double)(x[2] >> 5), 0x1p-27, (double)(x[3] >> 6) * 0x1p-53);
    const double r = bm_radius(-2.0 * fm::log_pos<DevOps>(u1));
    double s, c;
    fm::sincos_reduced(kTwoPi * u2, s, c);
    n0 = r * c;
    n1 = r * s;
}

// QE normals of particle pair p < 2^32 at absolute turn t (a bunch has fewer
// than 2^31 pairs): the counter's second word is the constant 0, which makes
// one product of the second round uniform too
__device__ __forceinline__ void qe_pair_normals32(uint64_t seed, uint32_t p, uint32_t t, double &n0,
                                                  double &n1) {
    uint32_t x[4];
    philox4x32_10(p, 0u, t, 0u, (uint32_t)seed, (uint32_t)(seed >> 32), x);
    box_muller(x, n0, n1);
}

// QE normals of particle pair p at absolute turn t
__device__ __forceinline__ void qe_pair_normals(uint64_t seed, uint64_t p, uint32_t t, double &n0,
                                                double &n1) {
    uint32_t x[4];
    philox4x32_10((uint32_t)p, (uint32_t)(p >> 32), t, 0u, (uint32_t)seed, (uint32_t)(seed >> 32), x);
    box_muller(x, n0, n1);
}

// zero_alloc_interpolation! index and weight (wakefield.jl:38-42,64-78) for
// nb >= 2.  interp_index clamps z to [c0, c1] by one v_max_f64 and one
// v_min_f64, which map a NaN z to c0; the reference's clamp keeps the NaN, its
// weight u - floor(u) is NaN and so is the interpolated value (cell 0 for the
// index, as the clamp of a converted NaN gives), which interp_index selects
// back.
//
// interp_index_pass, the turn pass's form, clamps the coordinate
// u = (z - c0) * inv to [0, u1], u1 = (c1 - c0) * inv, instead of z to
// [c0, c1]: the same u for every z that is not NaN, since rounding is
// monotonic (z > c1 gives u >= u1, z < c0 gives u <= 0, and the clamped
// z = c0 gives +0).  u is an arithmetic result, so the clamp needs no
// canonicalising of z and the ends, and it is never NaN (max with 0 drops a
// NaN): a NaN z lands on cell 0 with weight 0, and k = min(int(floor(u)),
// nb - 2) lies in [0, nb - 2] without a NaN select or a lower bound.  In the
// turn pass a NaN-z particle's dE turns NaN through the RF term of the same
// pass whatever its kick, so no result depends on that weight (the
// cloud-in-cell deposit counts a NaN z apart).
__device__ __forceinline__ void interp_index_pass(double z, double c0, double u1, double inv,
                                                  int nb, int &k, double &w) {
    const double v = __builtin_fmax((z - c0) * inv, 0.0);
    double u;   // fmin without a canonicalised copy of u1 (v is an arithmetic result, u1 finite)
    asm("v_min_f64 %0, %1, %2" : "=v"(u) : "v"(v), "s"(u1));
    k = min((int)u, nb - 2);           // truncation: u >= 0
    w = __builtin_amdgcn_fract(u);     // u - floor(u), exact
}
__device__ __forceinline__ void interp_index(double z, double c0, double c1, double inv, int nb,
                                             int &k, double &w) {
    const double cl = __builtin_fmin(__builtin_fmax(z, c0), c1);
    const double u = (cl - c0) * inv;
    const double fu = floor(u);
    const int kk = (fu == fu) ? (int)fu : 0;
    k = min(max(kk, 0), nb - 2);
    w = (z == z) ? u - fu : z;
}

// the interpolated value (wakefield.jl:94-102)
__device__ __forceinline__ double interp_pot(const double *__restrict__ P, double z, double c0,
                                             double c1, double inv, int nb) {
    if (nb <= 1) return nb == 1 ? P[0] : 0.0;
    int k;
    double w;
    interp_index(z, c0, c1, inv, nb, k, w);
    return P[k] * (1.0 - w) + P[k + 1] * w;
}

// the slots of `turn`'s count of particles that are not binned
__device__ __forceinline__ uint32_t *unb_of(const BunchDev &B, int64_t turn) {
    return B.unb + (int)(turn & 1) * (kUnbSlots * 16);
}
// `turn`'s half of the two-turn histogram buffer
__device__ __forceinline__ uint32_t *hist_of(const BunchDev &B, int64_t turn) {
    return B.hist + (int)(turn & 1) * hist_half(B.nbins);
}

// histogram bin of calculate_local_histogram! (utils.jl:387-397); -1 = not counted
// (z >= e0 makes z - e0, u and b non-negative: only z = e1 needs the clamp)
__device__ __forceinline__ int hist_bin(double z, double e0, double e1, double inv, int nb) {
    if (!((z >= e0) & (z <= e1))) return -1;
    const double u = (z - e0) * inv;
    const int b = (int)floor(u);
    return min(b, nb - 1);
}

// One DPP lane move of a double (two 32-bit moves with the same control);
// lanes whose row is not in ROWS receive 0.0.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xF, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// v[lane ^ OFF] + v[lane] for OFF = 32, 16, 8, 4, 2, 1 by lane swaps and DPP
// moves: the same sum as with __shfl_xor (an addition's operands commute)
// without its trip through LDS, whose latency is most of a butterfly's.
template <int OFF>
__device__ __forceinline__ double add_xor(double v) {
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
    if constexpr (OFF == 32) {
        const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        return __longlong_as_double(((long long)h[0] << 32) | l[0]) +
               __longlong_as_double(((long long)h[1] << 32) | l[1]);
    } else if constexpr (OFF == 16) {
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        return __longlong_as_double(((long long)h[0] << 32) | l[0]) +
               __longlong_as_double(((long long)h[1] << 32) | l[1]);
    } else if constexpr (OFF == 8) {
        return v + dpp_move<0x128, 0xF>(v);                       // row_ror:8
    } else if constexpr (OFF == 4) {
        return v + dpp_move<0x1B, 0xF>(dpp_move<0x141, 0xF>(v));  // half-row mirror, quad mirror
    } else if constexpr (OFF == 2) {
        return v + dpp_move<0x4E, 0xF>(v);                        // quad_perm [2,3,0,1]
    } else {
        return v + dpp_move<0xB1, 0xF>(v);                        // quad_perm [1,0,3,2]
    }
}
// the butterfly sum over the wave, offsets 32 down to 1; every lane gets it
__device__ __forceinline__ double butterfly(double v) {
    v = add_xor<32>(v);
    v = add_xor<16>(v);
    v = add_xor<8>(v);
    v = add_xor<4>(v);
    v = add_xor<2>(v);
    return add_xor<1>(v);
}

// Deterministic block sum of NV values: wave butterflies, then the waves in
// order.  The result is valid in thread 0.  s_red holds NV * 16 doubles.
template <int NV>
__device__ inline void block_sum(double (&v)[NV], double *s_red, int nw = (int)(blockDim.x >> 6)) {
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = butterfly(v[k]);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) s_red[k * 16 + wave] = v[k];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            double s = 0.0;
            for (int w = 0; w < nw; ++w) s += s_red[k * 16 + w];
            v[k] = s;
        }
    }
}

// Butterfly sum of NV values over one wave; every lane gets the result.
template <int NV>
__device__ __forceinline__ void wave_sum(double (&v)[NV]) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off, 64);
    }
}

// Sum of NV values over one wave in lane 63, by DPP lane moves (no LDS):
// within each row of 16 lanes by quad permutes (lane ^ 1, lane ^ 2), the
// half-row and the row mirror, which leave the row's sum in all of its lanes
// (each step adds two equal partial sums, in either order the same bits);
// then rows 1 and 3 add rows 0 and 2 (row_bcast:15) and row 3 adds row 1
// (row_bcast:31): lane 63 holds (R3 + R2) + (R1 + R0).  A fixed order.
template <int NV>
__device__ __forceinline__ void wave_total(double (&v)[NV]) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        double x = v[k];
        x = x + dpp_move<0xB1, 0xF>(x);    // quad_perm [1,0,3,2]
        x = x + dpp_move<0x4E, 0xF>(x);    // quad_perm [2,3,0,1]
        x = x + dpp_move<0x141, 0xF>(x);   // row_half_mirror
        x = x + dpp_move<0x140, 0xF>(x);   // row_mirror
        x = x + dpp_move<0x142, 0xA>(x);   // row_bcast:15 into rows 1, 3
        x = x + dpp_move<0x143, 0x8>(x);   // row_bcast:31 into row 3
        v[k] = x;
    }
}

// The wave totals of four values, in a fixed order, the total of v[q] in the
// lanes with (lane & 3) == q (lane 60 + q among them).  The quantities are
// transposed across lanes while they are summed: lanes l and l^1 exchange two
// values each and keep the sums of the other two, lanes l and l^2 one, so
// after two steps every lane holds one quantity summed over its quad; four
// more steps (row rotations by 4 and 8, then the rows by lane xor 16 and 32)
// sum it over the wave.  A third of the instructions of four wave_total<1>.
__device__ __forceinline__ double wave_total4(const double (&v)[4]) {
    const int l = (int)threadIdx.x & 63;
    const bool odd = (l & 1) != 0, hi = (l & 2) != 0;
    // quad_perm [1,0,3,2]: quantities 0, 2 (even lanes) or 1, 3 (odd lanes)
    const double ka = (odd ? v[1] : v[0]) + dpp_move<0xB1, 0xF>(odd ? v[0] : v[1]);
    const double kb = (odd ? v[3] : v[2]) + dpp_move<0xB1, 0xF>(odd ? v[2] : v[3]);
    double k = hi ? kb : ka;
    const double s = hi ? ka : kb;
    k = k + dpp_move<0x4E, 0xF>(s);      // quad_perm [2,3,0,1]: quantity l & 3
    k = k + dpp_move<0x124, 0xF>(k);     // row_ror:4
    k = k + dpp_move<0x128, 0xF>(k);     // row_ror:8
    k = k + __shfl_xor(k, 16, 64);
    k = k + __shfl_xor(k, 32, 64);
    return k;
}

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ int bitrev(int m, int logF) {
    return (int)(__brev((unsigned)m) >> (32 - logF));
}

__device__ __forceinline__ double2 cadd(double2 a, double2 b) {
    return make_double2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ double2 csub(double2 a, double2 b) {
    return make_double2(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ double2 conj2(double2 a) { return make_double2(a.x, -a.y); }

// In-place radix-2 decimation-in-time FFT of X[F] in LDS, bit-reversed input,
// natural-order output, twiddles tw[k] = exp(-2 pi i k / F).  Stage s pairs
// X[i] and X[i + 2^s] (i with bit s clear, k = i mod 2^s) with twiddle
// tw[k << (logF-1-s)].  The stages run in pairs (s, s+1) as radix-2^2
// butterflies: each thread takes the four points base + {0,1,2,3}*2^s
// through both stages in registers, the same additions and products as the
// two radix-2 stages (the same bits) with half the barriers and LDS round
// trips; an odd stage count starts with one radix-2 stage.  nblk blocks of F
// points, X + b*F, are transformed side by side.
__device__ void fft_dit_forward(double2 *X, int F, int logF, const double2 *__restrict__ tw,
                                int nblk = 1) {
    int s = 0;
    if (logF & 1) {   // stage 0 alone: pairs (2b, 2b+1), twiddle tw[0]
        __syncthreads();
        for (int b = threadIdx.x; b < nblk * (F >> 1); b += blockDim.x) {
            const double2 a = X[2 * b];
            const double2 t = cmul(X[2 * b + 1], tw[0]);
            X[2 * b] = cadd(a, t);
            X[2 * b + 1] = csub(a, t);
        }
        s = 1;
    }
    for (; s + 1 < logF; s += 2) {
        const int h = 1 << s, tsh = logF - 1 - s;
        __syncthreads();
        for (int u = threadIdx.x; u < nblk * (F >> 2); u += blockDim.x) {
            const int q = u & ((F >> 2) - 1);
            const int k = q & (h - 1);
            const int i0 = ((u >> (logF - 2)) << logF) + (((q >> s) << (s + 2)) | k);
            const double2 w1 = tw[k << tsh];              // stage s, both pairs
            const double2 wa = tw[k << (tsh - 1)];        // stage s+1, pair (0, 2)
            const double2 wb = tw[(k + h) << (tsh - 1)];  // stage s+1, pair (1, 3)
            const double2 x0 = X[i0], x1 = X[i0 + h], x2 = X[i0 + 2 * h], x3 = X[i0 + 3 * h];
            double2 t = cmul(x1, w1);
            const double2 a0 = cadd(x0, t), a1 = csub(x0, t);
            t = cmul(x3, w1);
            const double2 a2 = cadd(x2, t), a3 = csub(x2, t);
            t = cmul(a2, wa);
            X[i0] = cadd(a0, t);
            X[i0 + 2 * h] = csub(a0, t);
            t = cmul(a3, wb);
            X[i0 + h] = cadd(a1, t);
            X[i0 + 3 * h] = csub(a1, t);
        }
    }
    __syncthreads();
}

// Unnormalised inverse FFT (decimation in frequency, conjugate twiddles):
// natural-order input, output y[m] at X[bitrev(m)].  Stage s (from logF-1
// down to 0) takes a = X[i], c = X[i + 2^s] to a + c and (a - c) conj(w),
// w = tw[k << (logF-1-s)]; stages run in pairs (s, s-1) as radix-2^2
// butterflies on base + {0, 2^(s-1), 2^s, 2^s + 2^(s-1)}, with the same
// operations as the radix-2 stages, and an odd stage count ends with stage 0
// alone.  nblk blocks side by side, as in fft_dit_forward.
__device__ void fft_dif_inverse(double2 *X, int F, int logF, const double2 *__restrict__ tw,
                                int nblk = 1) {
    int s = logF - 1;
    for (; s >= 1; s -= 2) {
        const int h = 1 << s, h2 = h >> 1, tsh = logF - 1 - s;
        __syncthreads();
        for (int u = threadIdx.x; u < nblk * (F >> 2); u += blockDim.x) {
            const int q = u & ((F >> 2) - 1);
            const int k = q & (h2 - 1);
            const int i0 = ((u >> (logF - 2)) << logF) + (((q >> (s - 1)) << (s + 1)) | k);
            const double2 wa = conj2(tw[k << tsh]);          // stage s, pair (0, 2)
            const double2 wb = conj2(tw[(k + h2) << tsh]);   // stage s, pair (1, 3)
            const double2 wc = conj2(tw[k << (tsh + 1)]);    // stage s-1, both pairs
            const double2 x0 = X[i0], x1 = X[i0 + h2], x2 = X[i0 + h], x3 = X[i0 + h + h2];
            const double2 a0 = cadd(x0, x2), a2 = cmul(csub(x0, x2), wa);
            const double2 a1 = cadd(x1, x3), a3 = cmul(csub(x1, x3), wb);
            X[i0] = cadd(a0, a1);
            X[i0 + h2] = cmul(csub(a0, a1), wc);
            X[i0 + h] = cadd(a2, a3);
            X[i0 + h + h2] = cmul(csub(a2, a3), wc);
        }
    }
    if (s == 0) {   // stage 0 alone: pairs (2b, 2b+1), twiddle conj(tw[0])
        __syncthreads();
        const double2 w = conj2(tw[0]);
        for (int b = threadIdx.x; b < nblk * (F >> 1); b += blockDim.x) {
            const double2 a = X[2 * b], c = X[2 * b + 1];
            X[2 * b] = cadd(a, c);
            X[2 * b + 1] = cmul(csub(a, c), w);
        }
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// per-particle turn (fused)
// ---------------------------------------------------------------------------

struct PassCtx {
    double rf, inv_rf, phis, sin_phis, voltage, exc, damp, inv_mass, gamma0, alpha_c, kcoef,
        coeff_c, m_prev;
    int pending_kick, pending_m, drift_skip;
    uint32_t flags;
    const double *P;
    double c0, c1, u1, inv_s, e0, e1, inv_step;
    int nb;
};

__device__ inline void load_ctx(const BunchDev &B, PassCtx &c) {
    const TurnScalars &s = *B.sc;
    c.rf = s.rf;
    c.inv_rf = s.inv_rf;
    c.phis = B.phis;
    c.sin_phis = B.sin_phis;
    c.voltage = B.voltage;
    c.exc = s.exc;
    c.damp = s.damp;
    c.inv_mass = B.inv_mass;
    c.gamma0 = s.gamma0;
    c.alpha_c = B.alpha_c;
    c.kcoef = s.kcoef;
    c.coeff_c = s.coeff_c;
    // 0 when no re-centre is pending: subtracting it then changes nothing
    // (x - 0 = x for every x, -0 and NaN included)
    c.m_prev = s.pending_m ? s.m_prev : 0.0;
    c.pending_kick = s.pending_kick;
    c.pending_m = s.pending_m;
    c.drift_skip = s.drift_skip;
    c.flags = B.flags;
    c.P = B.P;
    c.c0 = B.c_first;
    c.c1 = B.c_last;
    c.u1 = B.u_last;
    c.inv_s = B.inv_s;
    c.e0 = B.e_first;
    c.e1 = B.e_last;
    c.inv_step = B.inv_step;
    c.nb = B.nbins;
}

// The previous turn's wake kick (wakefield.jl:342-344) and E0 re-centre
// (evolution.jl:434), applied at the start of this pass.
__device__ __forceinline__ double apply_pending(const PassCtx &c, double z, double e) {
    if (c.pending_kick) e = e - interp_pot(c.P, z, c.c0, c.c1, c.inv_s, c.nb);
    if (c.pending_m) e = e - c.m_prev;
    return e;
}

// phase advance (evolution.jl:331-344 with update_eta, :159-165 without)
template <uint32_t FX>
__device__ __forceinline__ double drift(const PassCtx &c, Flags<FX> fl, double z, double e) {
    if (fl.has(F_ETA)) {
        const double gp = c.gamma0 + e * c.inv_mass;
        // 1/gp^2 ~ 3e-8 enters eta ~ 1e-3 as a correction: one Newton step
        const double eta = c.alpha_c - fm::rcp1<DevOps>(gp * gp);
        const double coeff = eta * c.kcoef;
        double phi = -((z * c.rf) - c.phis);
        phi = phi + coeff * e;
        return ((-phi) + c.phis) * c.inv_rf;
    } else if (!c.drift_skip) {
        double phi = -((z * c.rf) - c.phis);
        phi = phi + c.coeff_c * e;
        return ((-phi) + c.phis) * c.inv_rf;
    }
    return z;
}

// The RF kick's energy change of a particle at z (rf_kick.jl:85-86); it
// does not depend on the particle's energy.
__device__ __forceinline__ double rf_term(const PassCtx &c, double z) {
    const double phi0 = ((-z) * c.rf) + c.phis;                    // rf_kick.jl:85
    return c.voltage * (dsin(phi0) - c.sin_phis);                  // rf_kick.jl:86
}

// RF (its term precomputed by rf_term), QE, SR and drift of one particle;
// returns dE' - dE_init via de_turn.
template <uint32_t FX>
__device__ __forceinline__ void advance_rest(const PassCtx &c, Flags<FX> fl, double &z, double &e,
                                             double rf, double r, double &de_turn) {
    const double e_init = e;
    e = e + rf;                                                    // rf_kick.jl:86
    if (fl.has(F_QE)) e = e + c.exc * r;                           // quantum_excitation.jl:70
    if (fl.has(F_SR)) e = e * c.damp;                              // synchrotron_radiation.jl:55
    z = drift(c, fl, z, e);
    de_turn = e - e_init;
}

// RF, QE, SR and drift of one particle; returns dE' - dE_init via de_turn.
template <uint32_t FX>
__device__ __forceinline__ void advance(const PassCtx &c, Flags<FX> fl, double &z, double &e,
                                        double r, double &de_turn) {
    advance_rest(c, fl, z, e, rf_term(c, z), r, de_turn);
}

// Explicit address spaces.  Pointers read from a BunchDev are generic to the
// compiler, and a choice between LDS and global memory merges into one
// generic access: both become flat instructions, which wait on the LDS and
// the vector-memory counters together.  The pass therefore names global
// memory (address space 1) and reaches its LDS through the kernel's own
// dynamic-LDS symbol.
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) double g_f64;
typedef __attribute__((address_space(1))) f64x2 g_f64x2;
typedef __attribute__((address_space(1))) uint32_t g_u32;
typedef __attribute__((address_space(1))) uint8_t g_u8;
typedef __attribute__((address_space(1))) unsigned long long g_u64;

// a deposit's counts n, and behind them the count of NaN positions
__device__ __forceinline__ g_u32 *cic_n(const BunchDev &B) {
    return (g_u32 *)(B.cic + 2 * cic_half(B.nbins));
}

__device__ __forceinline__ double2 ld2(const g_f64x2 *a) {
    const f64x2 v = *a;
    return make_double2(v.x, v.y);
}
__device__ __forceinline__ void st2(g_f64x2 *a, double x, double y) {
    f64x2 v;
    v.x = x;
    v.y = y;
    *a = v;
}
// streaming (nontemporal) 16-byte load: for arrays far larger than the caches
__device__ __forceinline__ double2 ldnt(const g_f64x2 *a) {
    const f64x2 v = __builtin_nontemporal_load(a);
    return make_double2(v.x, v.y);
}
// one or the other
template <bool NT>
__device__ __forceinline__ double2 ldp(const g_f64x2 *a) {
    return NT ? ldnt(a) : ld2(a);
}
// streaming (nontemporal) 16-byte store
__device__ __forceinline__ void stnt(g_f64x2 *a, double x, double y) {
    f64x2 v;
    v.x = x;
    v.y = y;
    __builtin_nontemporal_store(v, a);
}
template <bool NT>
__device__ __forceinline__ void stp(g_f64x2 *a, double x, double y) {
    if (NT) stnt(a, x, y);
    else st2(a, x, y);
}
// P[k]*(1-w) + P[k+1]*w from the neighbour-pair table entry (P[k], P[k+1])
__device__ __forceinline__ double gather_interp(const g_f64x2 *q, double w) {
    const f64x2 v = *q;
    return v.x * (1.0 - w) + v.y * w;
}

// whether the bunch's particles are read and written through the caches
__device__ __forceinline__ bool cached(const BunchDev &B) { return (B.flags & F_CACHED) != 0; }

__device__ __forceinline__ uint8_t *pass_lds() {
    extern __shared__ __align__(16) uint8_t s_lds[];
    return s_lds;
}

// the workgroup's count of particles that are not binned
__device__ __forceinline__ uint32_t &pass_unbinned() {
    __shared__ uint32_t s_unb;
    return s_unb;
}

// the next unit of the workgroup's run, and the single particle of an odd
// bunch: z, its energy change, and 1 if it is not binned
__device__ __forceinline__ int &pass_next() {
    __shared__ int s_next;
    return s_next;
}
__device__ __forceinline__ double (&pass_odd())[3] {
    __shared__ double s_odd[3];
    return s_odd;
}

// Copies the w entries from P to LDS, both 16-byte aligned, by 16-byte loads,
// kStageLoads in flight per thread (eight spend registers and gain nothing).  In
// 8-byte loads a window of 97 KB took 3 us of a pass and 128 KB 3 us of an
// interpolation sum: a turn of 1e6 particles and 16384 bins 62 -> 57 us with
// this and clear_lds.
constexpr int kStageLoads = 4;
__device__ __forceinline__ void stage_window(double *s, const double *P, int w) {
    const g_u8 *p = (const g_u8 *)P;
    uint8_t *d = reinterpret_cast<uint8_t *>(s);
    const unsigned end = (unsigned)(w >> 1) * 16u, step = blockDim.x * 16u;
    unsigned t = threadIdx.x * 16u;
    asm volatile("" : "+v"(t));   // not hoisted out of a loop over runs: it has no registers to spare
    for (unsigned b = 0; b < end; b += kStageLoads * step) {
        f64x2 x[kStageLoads];
#pragma unroll
        for (int u = 0; u < kStageLoads; ++u)
            if (b + u * step < end) x[u] = *(const g_f64x2 *)(p + min(b + u * step + t, end - 16u));
#pragma unroll
        for (int u = 0; u < kStageLoads; ++u)
            if (b + u * step + t < end) *reinterpret_cast<f64x2 *>(d + b + u * step + t) = x[u];
    }
    if ((w & 1) && t == 0) s[w - 1] = P[w - 1];
}
// Clears `bytes` (a multiple of 16) of LDS.
__device__ __forceinline__ void clear_lds(uint8_t *s, int bytes) {
    unsigned t = threadIdx.x;
    asm volatile("" : "+v"(t));   // as in stage_window
    uint4 *s4 = reinterpret_cast<uint4 *>(s);
    for (unsigned b = t; b < (unsigned)bytes / 16; b += blockDim.x) s4[b] = make_uint4(0u, 0u, 0u, 0u);
}

// HM: the histogram is in LDS, straight in global memory, or its window from bin
// hlo in 16-bit LDS counts and the rest in global memory.  v[3] counts
// the particles that are not binned (a branch most waves skip), n_bad (CIC
// only) the NaN positions among them, one atomic each.
enum HistMode { kHistGlobal = 0, kHistLds = 1, kHistWindow = 2 };
template <int HM, bool CIC>
__device__ __forceinline__ void bin_and_sum(const PassCtx &c, g_u32 *ghist, int spread, int hlo,
                                            int hwin, g_u32 *n_bad, double z, double (&v)[4]) {
    v[0] += z;
    v[1] += z * z;
    // hist_bin with its range test as the branch: in range, u = (z - e0) * inv
    // is >= 0, and its conversion to int (truncation) is floor(u)
    if ((z >= c.e0) & (z <= c.e1)) {
        const int b = min((int)((z - c.e0) * c.inv_step), c.nb - 1);
        const unsigned w = (unsigned)(b - hlo);
        if (HM == kHistLds)
            atomicAdd(reinterpret_cast<uint32_t *>(pass_lds()) + b, 1u);
        else if (HM == kHistWindow && w < (unsigned)hwin)
            atomicAdd(reinterpret_cast<uint32_t *>(pass_lds()) + (w >> 1), 1u << (16 * (w & 1)));
        else
            __hip_atomic_fetch_add(ghist + spread32(spread, b), 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    } else {
        v[3] += 1.0;
        if (CIC && z != z)
            __hip_atomic_fetch_add(n_bad, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// The cloud-in-cell deposit of one post-drift z (F_CIC) into the LDS counters
// at byte offset cb: the cell and weight the next pass's kick takes for it
// (interp_index_pass).  round(w 2^51) is the low 52 bits of the double
// 2^52 + w 2^51, formed by one fused multiply-add (one rounding; w in [0, 1),
// so the sum stays below 2^53).  A NaN z lands in cell 0; bin_and_sum counts
// it, which makes the sum NaN.
__device__ __forceinline__ void cic_deposit(const PassCtx &c, int cb, double z) {
    int k;
    double w;
    interp_index_pass(z, c.c0, c.u1, c.inv_s, c.nb, k, w);
    unsigned long long *cell = reinterpret_cast<unsigned long long *>(pass_lds() + cb) + 2 * k;
    const unsigned long long y = (unsigned long long)__double_as_longlong(
        __builtin_fma(w, kCicScale, 2.0 * kCicScale));
    atomicAdd(cell, (1ull << kCicCountBit) | ((unsigned)(y >> 32) & 0xfffffu));   // W >> 32 <= 2^19
    atomicAdd(cell + 1, y & 0xffffffffull);
}

// A value that every lane holds, as a scalar: the turn scalars are read through
// a pointer that the kernel also writes near, so the compiler keeps them in
// vector registers and takes the branches on them lane by lane.
__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// The fused pass over a run of tiles.  FX = kStdFlags is the common configuration
// with the flags folded at compile time; FX = 0 handles any other.  Both
// evaluate the same expressions, so a bunch gets the same bits from either.
// HM: where the histogram is (bin_and_sum), in LDS at offset 0; the window of P
// follows at byte hb.
//
// One call covers the run's tiles run[0..cnt) of bunch B (indices into the
// tile table, in ascending order but not necessarily adjacent: a bunch shared
// by several workgroups has its tiles dealt to them in turn).  Tiles are whole
// multiples of the block size, so thread t's pairs in tile lt are
// lt*ppt + t + k*kPassThreads in ascending k, exactly as for a tile taken
// alone; the 64 consecutive t of a tile are a unit, with sums of its own.  The
// waves take the run's units one by one from a counter in LDS, the next one
// while they work on the last: with every wave bound to the same 64 threads of
// each tile, the older waves of a SIMD ran ahead, and the last of the younger
// ones ran alone (1e7 particles: a pass of 69.7 -> 68.3 us; 28 bunches: 165.7 ->
// 159.4; 24 served jobs: 30.2 -> 29.2).  The loop over a unit is uniform: one chunk of
// kPassThreads pairs per step, its addresses a scalar base plus the lane's
// offset, the next chunk (the next unit's first at a unit's end) prefetched;
// only the last chunk of a bunch may be shorter, and its lanes past the end
// re-read its last pair and skip the rest.  A unit's sums are written at its end.
// The pass is bound by vector instructions below about 1e8 particles: with
// per-thread 64-bit positions and bounds the same loop spent 16 of them per
// pair on addresses, and 130 per tile on spilled scalars (a turn of a scan of 28
// bunches, most tiles of one to four pairs per thread: 240 -> 213 us; 24 served
// jobs 33.0 -> 30.3 ms; 1e7 particles 124 -> 121 us a turn).
// KM, how the kick reads P: kFullWindow (the LDS window holds the whole table:
// no global gathers), kGatherFirst or kPrefetchFirst (a partial window, the
// particles outside it gather from global memory; see the loop body).
// CIC: the bunch's post-drift z are also deposited (cic_deposit) into the LDS
// counters at byte cb.
// NTZ, NTE: z, dE are streamed past the caches, which are left to the bin
// phase's tables.
// With FX = kStdFlags the kick is applied from the first turn on: P is zero
// before it, and subtracting 0 changes nothing.
enum KickMode { kFullWindow = 0, kGatherFirst = 1, kPrefetchFirst = 2 };
template <uint32_t FX, int HM, int KM, bool CIC, bool NTZ, bool NTE = true>
__device__ __forceinline__ void turn_pass_run(const BunchDev &B, const int32_t *__restrict__ run,
                                              int cnt, unsigned t0, int hb, int cb, int unb) {
    PassCtx c;
    load_ctx(B, c);
    const Flags<FX> fl{c.flags};
    const bool wake = fl.has(F_WAKE);
    const TurnScalars &sc = *B.sc;
    const int64_t n = B.n;
    // pair indices are unsigned 32-bit: a bunch has at most 2^31 pairs
    const unsigned ppt = (unsigned)B.pairs_per_tile;
    const unsigned full = (unsigned)(n >> 1);       // pairs with two particles
    const int tb = B.tile_begin;
    const uint32_t tabs = (uint32_t)uni((int)(uint32_t)(B.turn_offset + sc.turn));
    const bool inj = fl.has(F_INJ);
    const bool qe = fl.has(F_QE);
    const g_f64 *nrm = inj ? (const g_f64 *)(B.normals + sc.turn * n) : nullptr;
    const uint64_t seed = B.seed;
    const bool kick = FX ? true : uni(c.pending_kick) != 0;
    const bool kick2 = kick && (FX ? true : c.nb >= 2);
    const bool rec = uni(c.pending_m) != 0;
    const int wlo = KM == kFullWindow ? 0 : uni(window_lo(sc.centre_bin, B.win, c.nb));
    const unsigned wpairs = (unsigned)max(B.win - 1, 0);   // pair starts inside the window
    const double *sP = reinterpret_cast<const double *>(pass_lds() + hb);
    const g_f64x2 *P2 = (const g_f64x2 *)B.P2;
    g_f64 *zp = (g_f64 *)B.z;
    g_f64 *ep = (g_f64 *)B.dE;
    g_u32 *ghist = (g_u32 *)hist_of(B, sc.turn);
    const int spread = HM == kHistLds ? 0 : B.spread, hwin = B.hwin;
    const int hlo = HM == kHistWindow ? uni(window_lo(sc.centre_bin, hwin, c.nb)) : 0;
    g_u32 *n_bad = CIC ? cic_n(B) + hist_half(c.nb) : nullptr;
    const int lane = (int)threadIdx.x & 63;
    const int lw = 31 - __builtin_clz(blockDim.x >> 6);   // log2 of the waves
    const int units = cnt << lw;
    constexpr unsigned step = kPassThreads;

    // pair `base` + (byte offset / 16) of the z or dE array
    auto at = [](g_f64 *a, unsigned base, unsigned off) -> g_f64x2 * {
        return (g_f64x2 *)((g_u8 *)a + (int64_t)base * 16 + off);
    };
    // a unit's partial sums: no workgroup barrier per tile, so a wave never
    // waits for the others of its workgroup between tiles
    auto flush = [&](const double (&v)[4], int lt, int slot) {
        const double tot = wave_total4(v);
        g_f64 *o = (g_f64 *)B.part + 4 * ((int64_t)lt * kTileWaves + slot);
        if (lane >= 60) o[lane - 60] = tot;
        if (unb && lane == 63 && tot != 0.0) atomicAdd(&pass_unbinned(), (uint32_t)tot);
    };
    // The single particle of an odd bunch sits in the bunch's last tile, the
    // last of this run if the run has it, and belongs to that tile's first
    // thread, whose unit adds it last.  Its turn is out of the loop over the
    // units, so that it does not add to the loop's register pressure.
    const int lt_last = run[cnt - 1] - tb;
    const bool odd = (n & 1) && t0 == 0 && (int64_t)full >= (int64_t)lt_last * ppt &&
                     (int64_t)full < min((int64_t)(lt_last + 1) * ppt, B.npairs);
    if (odd) {
        if (threadIdx.x == 0) {
            const int64_t i = n - 1;
            double z0 = zp[i], e0 = ep[i], r0 = 0.0, r1 = 0.0;
            if (qe) {
                if (inj) r0 = nrm[i];
                else qe_pair_normals32(seed, full, tabs, r0, r1);
            }
            e0 = apply_pending(c, z0, e0);
            double d0, v[4] = {0.0, 0.0, 0.0, 0.0};
            advance(c, fl, z0, e0, r0, d0);
            if (wake) bin_and_sum<HM, CIC>(c, ghist, spread, hlo, hwin, n_bad, z0, v);
            if (CIC) cic_deposit(c, cb, z0);
            zp[i] = z0;
            ep[i] = e0;
            pass_odd()[0] = z0;
            pass_odd()[1] = d0;
            pass_odd()[2] = v[3];
        }
        __syncthreads();
    }
    double v[4];   // sum z, sum z^2, sum (dE'-dE_init), not binned
    // a chunk's byte offset for a thread; lanes past the end take its last pair
    auto offset = [&](unsigned tid, unsigned lim) -> unsigned { return min(tid, lim - 1) * 16u; };
    // unit u: its tile, and its lanes' threads of the tile
    auto tile_of = [&](int u) { return run[u >> lw] - tb; };
    auto tid_of = [&](int u) { return t0 + (unsigned)((u & ((1 << lw) - 1)) << 6) + (unsigned)lane; };
    double2 zn = make_double2(0.0, 0.0), en = make_double2(0.0, 0.0);
    int u = uni((int)(threadIdx.x >> 6));
    int lt = tile_of(u);
    unsigned tid = tid_of(u);
    {
        const unsigned b0 = (unsigned)lt * ppt, lim = min(full - b0, step);   // b0 <= full
        if (lim > 0) {
            const unsigned off = offset(tid, lim);
            zn = ldp<NTZ>(at(zp, b0, off));
            en = ldp<NTE>(at(ep, b0, off));
        }
    }
    // the first chunk completes here (s_waitcnt vmcnt(0)), so that in the loop
    // the pair in hand is never taken for an outstanding load and the waits
    // there count only the loads issued in the loop
    __builtin_amdgcn_s_waitcnt(0x0F70);
    while (u < units) {
        const unsigned p0 = (unsigned)lt * ppt;
        const unsigned p1 = min(p0 + ppt, full);
        int un = units;   // the next unit; a single tile has one for each wave
        if (cnt > 1) {
            if (lane == 0) un = atomicAdd(&pass_next(), 1);
            un = uni(un);
        }
        const int ltn = un < units ? tile_of(un) : lt;
        const unsigned tidn = un < units ? tid_of(un) : tid;
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = 0.0;
        for (unsigned base = p0; base < p1; base += step) {
            const double2 zz = zn, ee = en;
            const unsigned lim = min(p1 - base, step);
            // The previous turn's potential at (P[k], P[k+1]): read from the LDS
            // window (clamped index, always valid), replaced by one 16-byte
            // global gather for the particles outside a partial window.  With
            // gather_first the gathers are issued before the next pair's
            // prefetch and consumed after the RF and QE terms, whose
            // arithmetic covers their latency.  Otherwise the prefetch goes
            // first.  The order of the loads changes no result.
            constexpr bool gather = KM != kFullWindow;
            constexpr bool gather_first = KM == kGatherFirst;
            // the next chunk (the next unit's first at a unit's end); past the
            // end of the run, or where that tile has no pair of two particles,
            // the tile's first chunk or this one is read again and not used,
            // so the load is unconditional and zn, en need no copy of their
            // old value
            auto prefetch = [&]() {
                const bool more = base + step < p1;
                unsigned bn = more ? base + step : (unsigned)ltn * ppt;
                if (bn >= full) bn = base;
                const unsigned off = offset(more ? tid : tidn, min(full - bn, step));
                zn = ldp<NTZ>(at(zp, bn, off));
                en = ldp<NTE>(at(ep, bn, off));
            };
            if (!gather_first) prefetch();
            // set and read only when kick2 (no per-pair clearing)
            double w0, w1;
            double2 q0, q1;
            if (kick2) {
                int k0, k1;
                interp_index_pass(zz.x, c.c0, c.u1, c.inv_s, c.nb, k0, w0);
                interp_index_pass(zz.y, c.c0, c.u1, c.inv_s, c.nb, k1, w1);
                if (!gather) {
                    q0 = make_double2(sP[k0], sP[k0 + 1]);
                    q1 = make_double2(sP[k1], sP[k1 + 1]);
                } else {
                    const unsigned j0 = (unsigned)(k0 - wlo), j1 = (unsigned)(k1 - wlo);
                    // any window of the all-flags pass (its histogram's share of
                    // the LDS leaves at least two entries) has wpairs >= 1
                    if (FX != 0 || wpairs) {
                        const unsigned i0 = min(j0, wpairs - 1), i1 = min(j1, wpairs - 1);
                        q0 = make_double2(sP[i0], sP[i0 + 1]);
                        q1 = make_double2(sP[i1], sP[i1 + 1]);
                    }
                    if (j0 >= wpairs) q0 = ld2(P2 + k0);
                    if (j1 >= wpairs) q1 = ld2(P2 + k1);
                }
            }
            if (gather_first) prefetch();
            double rf0 = 0.0, rf1 = 0.0;
            if (gather_first) {
                rf0 = rf_term(c, zz.x);
                rf1 = rf_term(c, zz.y);
            }
            double r0 = 0.0, r1 = 0.0;
            if (qe) {
                if (inj) {   // turn rows of an odd bunch are only 8-byte aligned
                    const int64_t p = (int64_t)base + min(tid, lim - 1);
                    r0 = nrm[2 * p];
                    r1 = nrm[2 * p + 1];
                } else {
                    qe_pair_normals32(seed, base + tid, tabs, r0, r1);
                }
            }
            double z0 = zz.x, z1 = zz.y, e0 = ee.x, e1 = ee.y;
            if (kick) {
                if (kick2) {
                    e0 = e0 - (q0.x * (1.0 - w0) + q0.y * w0);
                    e1 = e1 - (q1.x * (1.0 - w1) + q1.y * w1);
                } else {
                    const double pc = ((const g_f64 *)c.P)[0];
                    e0 = e0 - pc;
                    e1 = e1 - pc;
                }
            }
            // with update_E0 every turn but the first has a re-centre pending,
            // and m_prev is 0 when none is: the all-flags pass subtracts it
            // without a select
            if (fl.has(F_E0) || rec) {
                e0 = e0 - c.m_prev;
                e1 = e1 - c.m_prev;
            }
            double d0, d1;
            if (gather_first) {
                advance_rest(c, fl, z0, e0, rf0, r0, d0);
                advance_rest(c, fl, z1, e1, rf1, r1, d1);
            } else {
                advance(c, fl, z0, e0, r0, d0);
                advance(c, fl, z1, e1, r1, d1);
            }
            // The prefetched pair is complete before this pair's stores are
            // issued: a wait for a load behind a store would wait for the store.
            __builtin_amdgcn_s_waitcnt(0x0F70);
            if (tid < lim) {
                if (wake) {
                    bin_and_sum<HM, CIC>(c, ghist, spread, hlo, hwin, n_bad, z0, v);
                    bin_and_sum<HM, CIC>(c, ghist, spread, hlo, hwin, n_bad, z1, v);
                }
                if (CIC) {
                    cic_deposit(c, cb, z0);
                    cic_deposit(c, cb, z1);
                }
                v[2] += d0;
                v[2] += d1;
                stp<NTZ>(at(zp, base, tid * 16u), z0, z1);
                stp<NTE>(at(ep, base, tid * 16u), e0, e1);
            }
        }
        if (odd && lt == lt_last && tid == (unsigned)lane && lane == 0) {   // the unit of slot 0
            v[0] += pass_odd()[0];
            v[1] += pass_odd()[0] * pass_odd()[0];
            v[3] += pass_odd()[2];
            v[2] += pass_odd()[1];
        }
        if (!wake) { v[0] = 0.0; v[1] = 0.0; }
        flush(v, lt, uni((int)(tid >> 6)));
        u = un;
        lt = ltn;
        tid = tidn;
    }
}

// Adds the LDS histogram of bunch B, and the count of particles not binned, into
// this turn's global counts; a windowed one goes to the run's slab as it is.
__device__ inline void flush_hist(const BunchDev &B, int slab, int unb) {
    if (!(B.flags & F_WAKE)) return;
    __syncthreads();
    if (unb && threadIdx.x == 0) {
        const uint32_t u = pass_unbinned();
        if (u && B.unb)
            __hip_atomic_fetch_add((g_u32 *)unb_of(B, B.sc->turn) + 16 * (blockIdx.x % kUnbSlots), u,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!pass_hist_bytes(B)) return;
    int t = (int)threadIdx.x;
    asm volatile("" : "+v"(t));   // as in stage_window
    const uint32_t *s_hist = reinterpret_cast<const uint32_t *>(pass_lds());
    if (B.flags & F_GHIST) {
        const int words = B.hwin / 2;
        g_u32 *o = (g_u32 *)B.slabs + (int64_t)slab * words;
        for (int w = t; w < words; w += blockDim.x) o[w] = s_hist[w];
        return;
    }
    g_u32 *g = (g_u32 *)hist_of(B, B.sc->turn);
    const int sp = B.spread;
    for (int b = t; b < B.nbins; b += blockDim.x) {
        const uint32_t h = s_hist[b];
        if (h)
            __hip_atomic_fetch_add(g + spread32(sp, b), h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (B.flags & F_CIC) {   // and the deposit into this turn's counters
        const int nb = B.nbins;
        const ulonglong2 *sC = reinterpret_cast<const ulonglong2 *>(pass_lds() + B.cic_off);
        g_u64 *gH = (g_u64 *)B.cic, *gL = gH + cic_half(nb);
        g_u32 *gN = cic_n(B);
        for (int b = t; b < nb; b += blockDim.x) {
            const ulonglong2 c = sC[b];
            if (!c.x) continue;
            __hip_atomic_fetch_add(gN + spread32(sp, b), (uint32_t)(c.x >> kCicCountBit), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_add(gH + spread64(sp, b), (c.x & ((1ull << kCicCountBit) - 1)) + (c.y >> 32),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_add(gL + spread64(sp, b), c.y & 0xffffffffull, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// Clears the LDS histogram of bunch B and loads its potential window (zero
// before the first turn's bin phase; the all-flags pass reads it from the start).
template <uint32_t FX>
__device__ inline void stage_bunch(const BunchDev &B, int unb) {
    __syncthreads();   // the previous bunch's LDS is no longer read
    if (threadIdx.x == 0) {
        if (unb) pass_unbinned() = 0u;
        pass_next() = (int)(blockDim.x >> 6);   // each wave starts with the unit of its number
    }
    const int hb = pass_hist_bytes(B);
    clear_lds(pass_lds(), hb);
    if (B.flags & F_CIC) clear_lds(pass_lds() + B.cic_off, cic_bytes(B.nbins));
    const TurnScalars &sc = *B.sc;
    if ((FX || sc.pending_kick) && B.win > 0)
        stage_window(reinterpret_cast<double *>(pass_lds() + hb),
                     B.P + window_lo(sc.centre_bin, B.win, B.nbins), B.win);
    __syncthreads();
}

// Whether the all-flags pass prefetches before its gathers although its window is
// partial (the same bits): the loop waits for both together, and where most
// particles gather, the prefetch, which has the longer way, is better issued
// first.  A window of less than a seventh of the table, from 31657 bins on.  Pass
// of 8e7, 1e8 and 2e8 particles, gathers first and prefetch first, us:
//   24576 bins    564, 563      655, 661     1314, 1325
//   30000         602, 603      692, 700     1335, 1323
//   32000         646, 620      717, 693     1396, 1374
//   34560         750, 710      798, 774     1545, 1527
//   36000         784, 768      835, 825     1646, 1625
//   40700         948, 907     1003, 962     1978, 1882
// and of 1e7 particles, 34560 bins: 93, 92.
__device__ __forceinline__ bool small_window(const BunchDev &B) { return 7 * B.win < B.nbins; }

// The fused pass over a tile order.  Each workgroup takes its runs
// (runs[rr[g]..rr[g+1]): consecutive entries of the pass's tile order of one
// bunch, with about the same number of pairs as every other workgroup's, one
// workgroup per CU), and for each stages the bunch's LDS, streams the run and
// flushes the histogram.  The per-tile sums depend on the tile and the block
// size only, not on which workgroup takes the tile.  The runs are found on the
// host: found in the kernel, from the tile table, they cost two dependent
// scalar loads per tile before the first byte was streamed.  Launched with half
// the threads, two consecutive workgroups share a range, each with the tiles'
// lower or upper eight waves and LDS tables of its own.
template <uint32_t FX, bool NTZ>
__device__ __forceinline__ void turn_pass_blocks(const BunchDev *__restrict__ bds,
                                                 const int32_t *__restrict__ order,
                                                 const RunDev *__restrict__ runs,
                                                 const int32_t *__restrict__ rr, int unb) {
    const unsigned slices = kPassThreads / blockDim.x;
    const unsigned g = blockIdx.x / slices, slice = blockIdx.x % slices;
    const unsigned t0 = slice * blockDim.x;
    const int r1 = rr[g + 1];
    for (int r = rr[g]; r < r1; ++r) {
        const RunDev rd = runs[r];
        const BunchDev &B = bds[rd.bunch];
        stage_bunch<FX>(B, unb);
        const int hb = pass_hist_bytes(B);
        const int32_t *run = order + rd.begin;
        const int cnt = rd.count;
        // a partial window of P: gather first in the pass with compile-time
        // flags (only it has the registers), prefetch first in the generic one
        constexpr int kPartial = FX != 0 ? kGatherFirst : kPrefetchFirst;
        const bool full = B.win >= B.nbins;
        const int cb = B.cic_off;
        if (B.flags & F_CIC) {   // the deposit comes with the whole table
            turn_pass_run<FX, kHistLds, kFullWindow, true, NTZ>(B, run, cnt, t0, hb, cb, unb);
        } else if (!(B.flags & F_GHIST)) {   // a bunch without a wake among them
            if (full)
                turn_pass_run<FX, kHistLds, kFullWindow, false, NTZ>(B, run, cnt, t0, hb, cb, unb);
            else if (FX != 0 && small_window(B))
                turn_pass_run<FX, kHistLds, kPrefetchFirst, false, NTZ>(B, run, cnt, t0, hb, cb, unb);
            else
                turn_pass_run<FX, kHistLds, kPartial, false, NTZ>(B, run, cnt, t0, hb, cb, unb);
        } else if (FX != 0 || B.hwin > 0) {
            if (cached(B))
                turn_pass_run<FX, kHistWindow, kPartial, false, false, false>(B, run, cnt, t0, hb, cb, unb);
            else
                turn_pass_run<FX, kHistWindow, kPartial, false, NTZ>(B, run, cnt, t0, hb, cb, unb);
        } else {
            turn_pass_run<FX, kHistGlobal, kPrefetchFirst, false, NTZ>(B, run, cnt, t0, hb, cb, unb);
        }
        flush_hist(B, rd.slab + (int)slice, unb);
    }
}

template <bool NTZ>
__global__ __launch_bounds__(kPassThreads) void k_turn_pass(const BunchDev *__restrict__ bds,
                                                            const int32_t *__restrict__ order,
                                                            const RunDev *__restrict__ runs,
                                                            const int32_t *__restrict__ rr, int unb) {
    turn_pass_blocks<0, NTZ>(bds, order, runs, rr, unb);
}

// the same for tables whose bunches all have exactly kStdFlags, two bins or more
// and some of their histogram in LDS
template <bool NTZ>
__global__ __launch_bounds__(kPassThreads) void k_turn_pass_std(const BunchDev *__restrict__ bds,
                                                                const int32_t *__restrict__ order,
                                                                const RunDev *__restrict__ runs,
                                                                const int32_t *__restrict__ rr, int unb) {
    turn_pass_blocks<kStdFlags, NTZ>(bds, order, runs, rr, unb);
}

// ---------------------------------------------------------------------------
// turns without a wake and without the E0 update
// ---------------------------------------------------------------------------

// `turns` turns of bunches whose turns need nothing of the other particles (no
// wake, no E0 update: the turn scalars stay as they are): a thread carries its
// pair through all of them in registers, by the pass's own expressions, so the
// bits are those of one pass per turn.  Bound by vector instructions (about
// 270 per pair and turn) instead of 64 bytes of memory per pair and turn and
// two launches: 3e6 particles x 200 turns 6.6 ms by passes, 2.2 ms so.
// 256-thread workgroups of one item (consecutive pairs of one bunch) each:
// with nothing shared between waves they fill the SIMDs evenly.
__global__ __launch_bounds__(kFreeThreads) void k_free_turns(const BunchDev *__restrict__ bds,
                                                             const RunDev *__restrict__ items,
                                                             int turns) {
    const RunDev it = items[blockIdx.x];
    const BunchDev &B = bds[it.bunch];
    PassCtx c;
    load_ctx(B, c);
    c.drift_skip = uni(c.drift_skip);
    const Flags<0> fl{B.flags};
    const bool inj = fl.has(F_INJ), qe = fl.has(F_QE);
    const int64_t n = B.n, turn = B.sc->turn;
    const uint32_t t0 = (uint32_t)uni((int)(uint32_t)(B.turn_offset + turn));
    const unsigned end = (unsigned)it.begin + (unsigned)it.count;
    const unsigned full = (unsigned)(n >> 1);   // pairs with two particles
    g_f64 *zp = (g_f64 *)B.z;
    g_f64 *ep = (g_f64 *)B.dE;
    double2 zn = make_double2(0.0, 0.0), en = make_double2(0.0, 0.0);
    // pair q of the item, where it has two particles
    auto prefetch = [&](unsigned q) {
        if (q >= min(end, full)) return;
        zn = ldnt((const g_f64x2 *)zp + q);
        en = ldnt((const g_f64x2 *)ep + q);
    };
    prefetch((unsigned)it.begin + threadIdx.x);
    for (unsigned p = (unsigned)it.begin + threadIdx.x; p < end; p += kFreeThreads) {
        const int64_t i = 2 * (int64_t)p;
        const bool two = p < full;   // else the single particle of an odd bunch
        double z0 = zn.x, z1 = zn.y, e0 = en.x, e1 = en.y;
        if (!two) {
            z0 = zp[i];
            e0 = ep[i];
            z1 = e1 = 0.0;
        }
        prefetch(p + kFreeThreads);   // on its way during this pair's turns
        for (int t = 0; t < turns; ++t) {
            double r0 = 0.0, r1 = 0.0, d;
            if (qe) {
                if (inj) {
                    const g_f64 *nrm = (const g_f64 *)(B.normals + (turn + t) * n) + i;
                    r0 = nrm[0];
                    if (two) r1 = nrm[1];
                } else {
                    qe_pair_normals32(B.seed, p, t0 + (uint32_t)t, r0, r1);
                }
            }
            advance(c, fl, z0, e0, r0, d);
            advance(c, fl, z1, e1, r1, d);
        }
        if (two) {
            stnt((g_f64x2 *)(zp + i), z0, z1);
            stnt((g_f64x2 *)(ep + i), e0, e1);
        } else {
            zp[i] = z0;
            ep[i] = e0;
        }
    }
}

// after k_free_turns: finish_on's bookkeeping of `turns` such turns, one
// workgroup per listed bunch
__global__ __launch_bounds__(kFreeThreads) void k_free_finish(const BunchDev *__restrict__ bds,
                                                              const int32_t *__restrict__ list,
                                                              int turns) {
    const BunchDev &B = bds[list[blockIdx.x]];
    TurnScalars &s = *B.sc;
    const int64_t turn = s.turn;
    if (B.mon)
        for (int t = threadIdx.x; t < turns; t += kFreeThreads) B.mon[4 * (turn + t) + 2] = s.E0;
    __syncthreads();   // every thread has read the turn
    if (threadIdx.x == 0) {
        if (s.drift_skip) s.drift_skipped_count += turns;
        s.turn = turn + turns;
    }
}

// ---------------------------------------------------------------------------
// bin phase: sigma_z, current, line density, blocked FFT convolution
// ---------------------------------------------------------------------------
//
// P_k = I * sum_{j<=k} W_j g_{k-j},  g_i = lam_i * (cnt_i / n_h).
// With block size B and F = 2B, output block o is
//   Re(IFFT(Y_o))[0,B) + Im(IFFT(Y_o))[B,2B),
//   Y_o = sum_j X_{o-j} FFT(W_j),   X_a = FFT(g_a + i g_{a-1}),
// since each block product g_a * W_j is real, has length 2B-1 <= F (no
// wrap), and lands on output blocks a+j (first half) and a+j+1 (second half).

// One slice of a per-bunch reduction: the sum of entries [r*kRedEntries,
// (r+1)*kRedEntries) of a per-wave partial array of n entries, NV doubles
// each (NV = 1 or 4).  Thread t adds entries r*kRedEntries + t + k*kRedThreads
// in ascending k (all loads in flight at once), then block_sum adds the
// threads in its fixed order: the slice sum depends on n and r only.  Valid
// in thread 0.
template <int NV>
__device__ inline void slice_sum(const double *a, int n, int r, double (&v)[NV], double *s_red) {
    const int e0 = r * kRedEntries + (int)threadIdx.x;
    double x[kRedPer][NV];
#pragma unroll
    for (int k = 0; k < kRedPer; ++k) {
        const int e = e0 + k * kRedThreads;
        if constexpr (NV == 4) {
            double2 lo = make_double2(0.0, 0.0), hi = make_double2(0.0, 0.0);
            if (e < n) {
                const g_f64x2 *q = (const g_f64x2 *)a + 2 * (int64_t)e;
                lo = ld2(q);
                hi = ld2(q + 1);
            }
            x[k][0] = lo.x;
            x[k][1] = lo.y;
            x[k][2] = hi.x;
            x[k][3] = hi.y;
        } else {
            x[k][0] = e < n ? ((const g_f64 *)a)[e] : 0.0;
        }
    }
#pragma unroll
    for (int k = 0; k < kRedPer; ++k)
#pragma unroll
        for (int j = 0; j < NV; ++j) v[j] += x[k][j];
    block_sum<NV>(v, s_red, kRedThreads / 64);
}

// Counts slice r of bunch B in, its NV sums (thread 0's v) first stored at
// red[r].  Returns true in every thread of the workgroup that counts the
// bunch's last slice in; there thread 0 receives in t the sums of all slices,
// added in slice order, and the count is reset for the next reduction.  The
// count's read-modify-write is acquire-release at device scope, so the last
// slice sees every slice's stores whichever XCD wrote them; its threads read
// the slice sums side by side (one round trip), thread 0 adds them.
template <int NV>
__device__ inline bool slices_done(const BunchDev &B, int r, const double (&v)[NV],
                                   double (&t)[NV]) {
    __shared__ int s_last;
    __shared__ double s_slice[kRedThreads][NV];
    if (B.nred == 1) {   // one slice: nothing to count or to exchange
#pragma unroll
        for (int j = 0; j < NV; ++j) t[j] = v[j];
        return true;
    }
    g_f64 *red = (g_f64 *)B.red;
    g_u32 *cnt = (g_u32 *)B.cnt;
    if (threadIdx.x == 0) {
#pragma unroll
        for (int j = 0; j < NV; ++j)
            __hip_atomic_store(red + 4 * r + j, v[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const uint32_t before =
            __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        s_last = before + 1 == (uint32_t)B.nred;
    }
    __syncthreads();
    if (!s_last) return false;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
    for (int j = 0; j < NV; ++j) t[j] = 0.0;
    for (int q0 = 0; q0 < B.nred; q0 += kRedThreads) {
        const int q = q0 + (int)threadIdx.x;
        if (q < B.nred) {
            double x[NV];
#pragma unroll
            for (int j = 0; j < NV; ++j)
                x[j] = __hip_atomic_load(red + 4 * q + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int j = 0; j < NV; ++j) s_slice[threadIdx.x][j] = x[j];
        }
        __syncthreads();
        if (threadIdx.x == 0)
            for (int k = 0; k < kRedThreads && q0 + k < B.nred; ++k)
#pragma unroll
                for (int j = 0; j < NV; ++j) t[j] += s_slice[k][j];
        __syncthreads();
    }
    if (threadIdx.x == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// The turn scalars from the reduced pass sums t = {sum z, sum z^2,
// sum (dE'-dE_init), particles not binned}.
// bin_scalars_on updates the turn scalars sc in place (the bin phase in one
// workgroup keeps them in registers).
__device__ inline void bin_scalars_on(const BunchDev &B, const double (&t)[4], TurnScalars &sc) {
    sc.sum_dE = t[2];
    if (!(B.flags & F_WAKE)) return;
    const double sz = gstd_from_sums(t[0], t[1], (double)B.n);
    const double mz = t[0] / (double)B.n;
    sc.sigma_z = sz;
    sc.current = (B.flags & F_CHARGE)
                     ? B.charge
                     : (((B.pf / sc.E0) / (kTwoPi * B.radius)) * sz) /
                           (sc.eta0 * (B.sigma_E0 * B.sigma_E0));
    sc.n_h = (double)B.n - t[3];
    const double kc = floor((mz - B.c_first) * B.inv_s);
    const double top = (double)(B.nbins - 1);
    sc.centre_bin = (kc == kc) ? (int)(kc < 0.0 ? 0.0 : (kc > top ? top : kc)) : 0;
    if (B.mon) {   // turn monitor: centroid and sigma_z after the drift, binned count
        double *m = B.mon + 4 * sc.turn;
        m[0] = mz;
        m[1] = sz;
        m[3] = sc.n_h;
    }
}

__device__ inline void bin_scalars(const BunchDev &B, const double (&t)[4]) {
    bin_scalars_on(B, t, *B.sc);
}

// The sums t over the nred slices of the pass's per-wave sums by one 1024-thread
// workgroup (k_bin_whole), with the arithmetic of slice_sum (256 threads) and
// slices_done: the workgroup's four groups of four waves take four slices at a
// time, each group exactly as a 256-thread slice workgroup, and thread 0 adds
// the slice sums in slice order.  Same bits as the sliced form, without its count
// across workgroups.
__device__ inline void whole_sum(const BunchDev &B, double (&t)[4]) {
    constexpr int NV = 4;
    __shared__ double s_red[4][NV * 16];
    __shared__ double s_slice[4][NV];
    const int n = B.ntiles * kTileWaves, nred = B.nred;
    const int g = (int)threadIdx.x >> 8, tl = (int)threadIdx.x & 255;
    const int lane = tl & 63, wave = tl >> 6;
#pragma unroll
    for (int j = 0; j < NV; ++j) t[j] = 0.0;
    for (int r0 = 0; r0 < nred; r0 += 4) {
        const int r = r0 + g;
        double v[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j) v[j] = 0.0;
        if (r < nred) {   // slice_sum's loads and order, thread tl of slice r
            const int e0 = r * kRedEntries + tl;
            double x[kRedPer][NV];
#pragma unroll
            for (int k = 0; k < kRedPer; ++k) {
                const int e = e0 + k * kRedThreads;
                double2 lo = make_double2(0.0, 0.0), hi = make_double2(0.0, 0.0);
                if (e < n) {
                    const g_f64x2 *q = (const g_f64x2 *)B.part + 2 * (int64_t)e;
                    lo = ld2(q);
                    hi = ld2(q + 1);
                }
                x[k][0] = lo.x;
                x[k][1] = lo.y;
                x[k][2] = hi.x;
                x[k][3] = hi.y;
            }
#pragma unroll
            for (int k = 0; k < kRedPer; ++k)
#pragma unroll
                for (int j = 0; j < NV; ++j) v[j] += x[k][j];
        }
        // block_sum's order within the group: wave butterflies, then its four waves
#pragma unroll
        for (int j = 0; j < NV; ++j) v[j] = butterfly(v[j]);
        if (lane == 0)
#pragma unroll
            for (int j = 0; j < NV; ++j) s_red[g][j * 16 + wave] = v[j];
        __syncthreads();
        if (tl == 0)
#pragma unroll
            for (int j = 0; j < NV; ++j) {
                double x = 0.0;
                for (int w = 0; w < 4; ++w) x += s_red[g][j * 16 + w];
                s_slice[g][j] = x;
            }
        __syncthreads();
        if (threadIdx.x == 0)   // slices_done: one slice as it is, else from zero in order
            for (int q = 0; q < 4 && r0 + q < nred; ++q)
#pragma unroll
                for (int j = 0; j < NV; ++j) t[j] = nred == 1 ? s_slice[q][j] : t[j] + s_slice[q][j];
        __syncthreads();
    }
}

// The counts of the LDS windows, slab by slab, added to this turn's histogram:
// a workgroup takes 256 words (512 bins) of one bunch's window, each of its
// four groups of waves a quarter of the slabs with 16 loads in flight.  Before
// k_reduce_fwd, which moves the centroid that places the window.  Bound by the
// 25 MB of 256 slabs: 8 us with its launch, where flushing 49152 bins of every
// workgroup by atomics would take about 28 (14 us per 6.3e6 of them).
__global__ __launch_bounds__(1024) void k_hist_slabs(const BunchDev *__restrict__ bds,
                                                     const int32_t *__restrict__ items) {
    __shared__ uint32_t s_part[4][512];
    const BunchDev &B = bds[items[2 * blockIdx.x]];
    const int words = B.hwin / 2, col = (int)threadIdx.x & 255, grp = (int)threadIdx.x >> 8;
    const int w = items[2 * blockIdx.x + 1] * 256 + col;
    const g_u32 *slab = (const g_u32 *)B.slabs + min(w, words - 1);
    const int n = B.nslabs, q = (n + 3) / 4, s1 = min(n, (grp + 1) * q);
    uint32_t lo = 0, hi = 0;
    for (int s = grp * q; s < s1; s += 16) {
        uint32_t x[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) x[u] = s + u < s1 ? slab[(int64_t)(s + u) * words] : 0u;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            lo += x[u] & 0xffffu;
            hi += x[u] >> 16;
        }
    }
    s_part[grp][2 * col] = lo;
    s_part[grp][2 * col + 1] = hi;
    __syncthreads();
    const int b = (int)threadIdx.x;   // 512 bins on the first 512 threads
    const int i = items[2 * blockIdx.x + 1] * 512 + b;
    if (b < 512 && i < B.hwin) {
        const TurnScalars &sc = *B.sc;
        uint32_t *h = hist_of(B, sc.turn) +
                      spread32(B.spread, window_lo(sc.centre_bin, B.hwin, B.nbins) + i);
        *h += s_part[0][b] + s_part[1][b] + s_part[2][b] + s_part[3][b];
    }
}

// Once per turn and bunch, after the pass: the pass's per-wave sums reduced
// into the turn scalars.  sum (dE'-dE_init) for the E0 update; for a wake
// bunch sigma_z (evolution.jl:357), the wake current (evolution.jl:373-386),
// the binned count, and the interpolation cell of the centroid (where the LDS
// windows of P are placed; the placement changes no result); the turn
// monitor's centroid, sigma_z and binned count.  One workgroup per slice.
__device__ __forceinline__ void bin_reduce(const BunchDev &B, int r) {
    __shared__ double s_red[4 * 16];
    if (!(B.flags & (F_WAKE | F_E0))) return;
    double v[4] = {0.0, 0.0, 0.0, 0.0};   // sum z, sum z^2, sum (dE'-dE_init), not binned
    slice_sum<4>(B.part, B.ntiles * kTileWaves, r, v, s_red);
    double t[4];
    if (!slices_done<4>(B, r, v, t) || threadIdx.x != 0) return;
    bin_scalars(B, t);
}

// g_i = lam_i * (cnt_i / n_h) (wakefield.jl:210,238).  A wake table by lag
// (F_LAG) is convolved causally, P_k = I sum_j W_j g_{k+j}: the index
// convolution of the reversed density, written back reversed (store_block).
__device__ __forceinline__ double line_density(const BunchDev &B, const uint32_t *h, int i,
                                               double inv_nh) {
    if (B.flags & F_LAG) i = B.nbins - 1 - i;
    return B.lam[i] * ((double)h[spread32(B.spread, i)] * inv_nh);
}

// sX <- bit-reversed g_a + i g_{a-1}, zero-padded to F
__device__ inline void load_packed(double2 *sX, const BunchDev &B, int a, double inv_nh) {
    const int nb = B.nbins, Bk = B.B, F = B.F, logF = B.logF;
    const uint32_t *h = hist_of(B, B.sc->turn);
    for (int m = threadIdx.x; m < F; m += blockDim.x) {
        double re = 0.0, im = 0.0;
        if (m < Bk) {
            const int i = a * Bk + m;
            if (i < nb) re = line_density(B, h, i, inv_nh);
            if (a >= 1) im = line_density(B, h, i - Bk, inv_nh);
        }
        sX[bitrev(m, logF)] = make_double2(re, im);
    }
}

// clears bins [aB, aB+B) of the histogram half the next turn fills (nothing
// reads it during this turn)
__device__ inline void clear_next_hist(const BunchDev &B, int a) {
    const int nb = B.nbins, Bk = B.B;
    uint32_t *h = hist_of(B, B.sc->turn + 1);
    for (int m = threadIdx.x; m < Bk; m += blockDim.x)
        if (a * Bk + m < nb) h[spread32(B.spread, a * Bk + m)] = 0u;
}

// writes P[i] and its two places in the neighbour-pair table,
// P2[i].x = P[i] and P2[i-1].y = P[i] (P2[nb-1].y stays 0)
__device__ __forceinline__ void put_potential(const BunchDev &B, int i, double v) {
    B.P[i] = v;
    if (B.P2) {
        B.P2[2 * i] = v;
        if (i >= 1) B.P2[2 * i - 1] = v;
    }
}

// P block o from the unnormalised inverse FFT in LDS
__device__ inline void store_block(const BunchDev &B, const double2 *sX, int o, double cur) {
    const int nb = B.nbins, Bk = B.B, logF = B.logF;
    const double scale = cur / (double)B.F;
    for (int m = threadIdx.x; m < Bk; m += blockDim.x) {
        const int i = o * Bk + m;
        if (i >= nb) continue;
        const double2 y0 = sX[bitrev(m, logF)];
        const double2 y1 = sX[bitrev(m + Bk, logF)];
        put_potential(B, (B.flags & F_LAG) ? nb - 1 - i : i, (y0.x + y1.y) * scale);
    }
}

__device__ inline void zero_block(const BunchDev &B, int o) {
    const int nb = B.nbins, Bk = B.B;
    for (int m = threadIdx.x; m < Bk; m += blockDim.x) {
        const int i = o * Bk + m;
        if (i < nb) put_potential(B, (B.flags & F_LAG) ? nb - 1 - i : i, 0.0);
    }
}

// one workgroup per output block, wake support within one block (nJ <= 1)
__global__ __launch_bounds__(kConvThreads) void k_conv_fused(const BunchDev *__restrict__ bds,
                                                             const int32_t *__restrict__ items) {
    extern __shared__ double2 sX[];
    const BunchDev &B = bds[items[2 * blockIdx.x]];
    const int o = items[2 * blockIdx.x + 1];
    const double nh = B.sc->n_h, cur = B.sc->current;
    clear_next_hist(B, o);
    if (nh == 0.0 || B.nJ == 0) {   // wakefield.jl:305-311
        zero_block(B, o);
        return;
    }
    const double2 *tw = reinterpret_cast<const double2 *>(B.tw);
    const double2 *What = reinterpret_cast<const double2 *>(B.What);
    load_packed(sX, B, o, 1.0 / nh);
    fft_dit_forward(sX, B.F, B.logF, tw);
    for (int k = threadIdx.x; k < B.F; k += blockDim.x) sX[k] = cmul(sX[k], What[k]);
    fft_dif_inverse(sX, B.F, B.logF, tw);
    store_block(B, sX, o, cur);
}

// phase A of the blocked convolution: X_a = FFT(g_a + i g_{a-1})
__device__ __forceinline__ void conv_fwd(const BunchDev &B, int a, double nh) {
    extern __shared__ double2 sX[];
    clear_next_hist(B, a);
    if (nh == 0.0) return;
    load_packed(sX, B, a, 1.0 / nh);
    fft_dit_forward(sX, B.F, B.logF, reinterpret_cast<const double2 *>(B.tw));
    double2 *X = reinterpret_cast<double2 *>(B.X) + (int64_t)a * B.F;
    for (int k = threadIdx.x; k < B.F; k += blockDim.x) X[k] = sX[k];
}

__global__ __launch_bounds__(kConvThreads) void k_conv_fwd(const BunchDev *__restrict__ bds,
                                                           const int32_t *__restrict__ items) {
    const BunchDev &B = bds[items[2 * blockIdx.x]];
    conv_fwd(B, items[2 * blockIdx.x + 1], B.sc->n_h);
}

// The reductions of the pass's sums (the first nred workgroups, bin_reduce) and
// phase A of the convolutions in one launch.  Phase A needs of the reductions
// only the binned count, which it takes from the pass's counts of particles
// not binned (the same whole number).  In launches of their own the two took
// 5 to 7 us each, one after the other: 1e6 particles, 16384 bins: 56.5 -> 52.4 us a
// turn; 1e7, 8192 bins: 120 -> 117; 28 bunches of 4096 bins, which had one
// workgroup per bunch for the reductions: 212 -> 210.
__global__ __launch_bounds__(kConvMaxThreads) void k_reduce_fwd(const BunchDev *__restrict__ bds,
                                                             const int32_t *__restrict__ red, int nred,
                                                             const int32_t *__restrict__ items) {
    if ((int)blockIdx.x < nred) {
        if ((int)threadIdx.x >= kRedThreads) return;   // whole waves, before any barrier
        bin_reduce(bds[red[2 * blockIdx.x]], red[2 * blockIdx.x + 1]);
        return;
    }
    const int32_t *it = items + 2 * ((int)blockIdx.x - nred);
    const BunchDev &B = bds[it[0]];
    const int64_t turn = B.sc->turn;
    const int lane = (int)threadIdx.x & 63;
    int c = (int)((g_u32 *)unb_of(B, turn))[16 * lane];   // every wave: kUnbSlots lanes
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if (it[1] == 0 && (int)threadIdx.x < kUnbSlots) ((g_u32 *)unb_of(B, turn + 1))[16 * lane] = 0u;
    conv_fwd(B, it[1], (double)(B.n - (int64_t)(uint32_t)c));
}

// phase B1: Y_o[k] = sum_{j <= min(o, nJ-1)} X_{o-j}[k] FFT(W_j)[k] for every
// output block o, one chunk of spec_chunk(nA, F) frequencies of one bunch per
// workgroup.  The chunk's columns of X and of the wake spectra are staged in
// LDS once (every X_a and W_j is read from memory once per turn, instead of
// once per output block as in k_conv_inv); a thread takes one (frequency,
// output block) pair.  The products are added in ascending j from zero, as in
// k_conv_inv, so Y_o and the potential are the same bits on either path.
__global__ __launch_bounds__(kConvMaxThreads) void k_conv_spec(const BunchDev *__restrict__ bds,
                                                            const int32_t *__restrict__ items) {
    extern __shared__ double2 sS[];
    const BunchDev &B = bds[items[2 * blockIdx.x]];
    const int c = items[2 * blockIdx.x + 1];
    if (B.sc->n_h == 0.0) return;   // k_conv_out writes a zero potential
    const int F = B.F, nA = B.nA, nJ = B.nJ;
    const int kc = spec_chunk(nA, F), k0 = c * kc;
    double2 *sXc = sS;               // [nA][kc]
    double2 *sWc = sS + nA * kc;     // [nJ][kc]
    const double2 *X = reinterpret_cast<const double2 *>(B.X);
    const double2 *What = reinterpret_cast<const double2 *>(B.What);
    for (int i = threadIdx.x; i < nA * kc; i += blockDim.x) {
        const int a = i / kc, kk = i - a * kc;
        sXc[i] = X[(int64_t)a * F + k0 + kk];
    }
    for (int i = threadIdx.x; i < nJ * kc; i += blockDim.x) {
        const int j = i / kc, kk = i - j * kc;
        sWc[i] = What[(int64_t)j * F + k0 + kk];
    }
    __syncthreads();
    double2 *Y = reinterpret_cast<double2 *>(B.Y);
    for (int i = threadIdx.x; i < nA * kc; i += blockDim.x) {
        const int o = i / kc, kk = i - o * kc;
        double2 acc = make_double2(0.0, 0.0);
        const int jmax = min(o, nJ - 1);
#pragma unroll 4
        for (int j = 0; j <= jmax; ++j) {
            const double2 t = cmul(sXc[(o - j) * kc + kk], sWc[j * kc + kk]);
            acc = make_double2(acc.x + t.x, acc.y + t.y);
        }
        Y[(int64_t)o * F + k0 + kk] = acc;
    }
}

// phase B2: inverse FFT of Y_o, P block o
__global__ __launch_bounds__(kConvMaxThreads) void k_conv_out(const BunchDev *__restrict__ bds,
                                                           const int32_t *__restrict__ items) {
    extern __shared__ double2 sX[];
    const BunchDev &B = bds[items[2 * blockIdx.x]];
    const int o = items[2 * blockIdx.x + 1];
    const double nh = B.sc->n_h, cur = B.sc->current;
    if (nh == 0.0) {
        zero_block(B, o);
        return;
    }
    const int F = B.F;
    const double2 *Y = reinterpret_cast<const double2 *>(B.Y) + (int64_t)o * F;
    for (int k = threadIdx.x; k < F; k += blockDim.x) sX[k] = Y[k];
    fft_dif_inverse(sX, F, B.logF, reinterpret_cast<const double2 *>(B.tw));
    store_block(B, sX, o, cur);
}

// phase B (where the spectra of a chunk exceed the LDS): Y_o = sum_j
// X_{o-j} FFT(W_j), inverse FFT, P block o.  The products are summed in j
// order; four j at a time have their loads in flight.
__global__ __launch_bounds__(kConvInvThreads) void k_conv_inv(const BunchDev *__restrict__ bds,
                                                              const int32_t *__restrict__ items) {
    extern __shared__ double2 sX[];
    const BunchDev &B = bds[items[2 * blockIdx.x]];
    const int o = items[2 * blockIdx.x + 1];
    const double nh = B.sc->n_h, cur = B.sc->current;
    if (nh == 0.0) {
        zero_block(B, o);
        return;
    }
    const int F = B.F;
    const int jmax = min(o, B.nJ - 1);
    const double2 *X = reinterpret_cast<const double2 *>(B.X);
    const double2 *What = reinterpret_cast<const double2 *>(B.What);
    for (int k = threadIdx.x; k < F; k += blockDim.x) {
        double2 acc = make_double2(0.0, 0.0);
        int j = 0;
        for (; j + 4 <= jmax + 1; j += 4) {
            double2 xa[4], wa[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                xa[u] = X[(int64_t)(o - j - u) * F + k];
                wa[u] = What[(int64_t)(j + u) * F + k];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const double2 t = cmul(xa[u], wa[u]);
                acc = make_double2(acc.x + t.x, acc.y + t.y);
            }
        }
        for (; j <= jmax; ++j) {
            const double2 t = cmul(X[(int64_t)(o - j) * F + k], What[(int64_t)j * F + k]);
            acc = make_double2(acc.x + t.x, acc.y + t.y);
        }
        sX[k] = acc;
    }
    fft_dif_inverse(sX, F, B.logF, reinterpret_cast<const double2 *>(B.tw));
    store_block(B, sX, o, cur);
}

// Broadband resonator wake [V/C] at distance s >= 0 behind the source
// (Chao, Physics of Collective Beam Instabilities, eq. 2.84):
// W(s) = 2 a Rs e^{-a s/c} [cos(wb s/c) - (a/wb) sin(wb s/c)], a = w_r/(2Q),
// wb = sqrt(w_r^2 - a^2); W(0) = a Rs, half the jump.  Overdamped (Q < 1/2)
// and critical forms by cosh/sinh and the limit.
__device__ inline double resonator_wake(double s, double Rs, double fr, double Q) {
    const double wr = kTwoPi * fr;
    const double a = wr / (2.0 * Q);
    if (s < 0.0) return 0.0;
    if (s == 0.0) return a * Rs;
    const double tau = s / kSpeedLight;
    const double env = 2.0 * a * Rs * exp(-a * tau);
    const double d = wr * wr - a * a;
    if (d > 0.0) {
        const double wb = sqrt(d);
        return env * (cos(wb * tau) - (a / wb) * sin(wb * tau));
    } else if (d < 0.0) {
        const double wb = sqrt(-d);
        return env * (cosh(wb * tau) - (a / wb) * sinh(wb * tau));
    }
    return env * (1.0 - a * tau);
}

// the resonators' wake table by lag (set-up of an evolve call)
__global__ void k_resonator_table(double *__restrict__ W, int nb, double step, ResonatorSet rs) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nb) return;
    const double s = (double)j * step;
    double w = 0.0;
    for (int r = 0; r < rs.n; ++r) w += resonator_wake(s, rs.Rs[r], rs.fr[r], rs.Q[r]);
    W[j] = w;
}

// The reference's tables of the bin centres (set-up of an evolve call): its
// wake W(c) (wakefield.jl:115-118) and the delta kernel (utils.jl:58-66), each
// where asked for (ef = 0: the constant s_inv).  The centre is the correctly rounded zw num / nb: with
// zw num = p + e and the quotient q of p, the remainder p + e - q nb is exact
// (both parts are multiples of q's last place, less than nb of them), and
// q plus the remainder's quotient rounds once: that quotient's own rounding is
// 2^-53 of it, while its distance from a half of the last place is zero or at
// least 1 / (4 nb).  Needs nb < 2^28 and no under- or overflow in p and e.
// On the host, by 128-bit integers and libm, the two tables of 131072 bins took
// 3.8 of the 14.5 ms of a call of 50 turns of 1e7 particles (0.5 of 6.7 ms with
// 16384 bins, 100 turns of 1e6 particles).
__global__ void k_reference_tables(double *__restrict__ W, double *__restrict__ lam, int nb,
                                   double zw, double wf, double ws, double inv_ctau, double s_inv,
                                   double ef) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nb) return;
    const double num = (double)(2 * i + 1 - nb), den = (double)nb;
    const double p = zw * num, e = __builtin_fma(zw, num, -p);
    const double q = p / den;
    const double c = q + (__builtin_fma(-q, den, p) + e) / den;
    if (W) W[i] = c > 0.0 ? 0.0 : (wf * exp(c * inv_ctau)) * cos(ws * c);
    if (lam) lam[i] = ef == 0.0 ? s_inv : s_inv * exp((c * c) * ef);
}

// FFT of one wake block per workgroup (set-up of an evolve call)
__global__ __launch_bounds__(kConvThreads) void k_fft_wake(const BunchDev *__restrict__ bd,
                                                           const double *__restrict__ W) {
    extern __shared__ double2 sX[];
    const BunchDev &B = *bd;
    const int j = blockIdx.x, Bk = B.B, F = B.F, logF = B.logF, nb = B.nbins;
    for (int m = threadIdx.x; m < F; m += blockDim.x) {
        const int i = j * Bk + m;
        const double w = (m < Bk && i < nb) ? W[i] : 0.0;
        sX[bitrev(m, logF)] = make_double2(w, 0.0);
    }
    fft_dit_forward(sX, F, logF, reinterpret_cast<const double2 *>(B.tw));
    double2 *out = reinterpret_cast<double2 *>(const_cast<double *>(B.What)) + (int64_t)j * F;
    for (int k = threadIdx.x; k < F; k += blockDim.x) out[k] = sX[k];
}

// ---------------------------------------------------------------------------
// E0 update support, moments, init, finalize
// ---------------------------------------------------------------------------

// interp_sum_run for tiles of at least G pairs per thread (G = 4 or 8): per
// tile, groups of G pairs per thread.  The sums over a run of tiles [lt0, lt1) of bunch
// B of the interpolated potential at the post-drift z, one sum per tile and
// wave.  The run first stages B.iwin entries of P around the
// centroid in LDS (the whole table unless it exceeds the LDS); particles
// outside the window read the pair table P2.  Each thread takes its pairs
// of a tile in groups of G, in ascending order, with the next group's
// streaming loads (the next tile's first group at a tile's end) issued before
// this group's sums; the group loop has the same trip count in every lane.
// A tile's sums therefore depend on the tile and the block size only (not on G).
template <int G, bool FULLW, bool NT>
__device__ __forceinline__ void interp_sum_run_tiles(const BunchDev &B, const int32_t *__restrict__ run,
                                                     int nrun) {
    extern __shared__ __align__(16) double sP[];
    const int nb = B.nbins;
    const double *__restrict__ P = B.P;
    const int w = B.iwin;
    const int wlo = window_lo(B.sc->centre_bin, w, nb);
    const unsigned wpairs = (unsigned)(w - 1);
    __syncthreads();   // the previous run's window is no longer read
    stage_window(sP, P + wlo, w);
    __syncthreads();
    const int64_t n = B.n, ppt = B.pairs_per_tile, full = n >> 1;
    const int64_t bs = kInterpThreads;
    const int K = (int)(ppt / bs);   // pairs of each thread in a full tile
    const double c0 = B.c_first, c1 = B.c_last, inv = B.inv_s;
    const g_f64 *zp = (const g_f64 *)B.z;
    const g_f64x2 *P2 = (const g_f64x2 *)B.P2;
    const g_f64x2 *zpair = (const g_f64x2 *)zp;
    const int tid = (int)threadIdx.x, ibs = (int)bs;
    // pair offsets within a tile are 32-bit; tile bases are uniform
    // The ring's loads are issued unconditionally (a lane without a next pair
    // reads pair 0 and ignores it), so that every wait for a slot is the same
    // count of younger loads.  Needs a two-particle pair: full >= 1.
    const bool ring = nb >= 2 && full >= 1;
    // the j-th tile of the run, and its two-particle pairs
    auto tile_of = [&](int j) { return run[j] - B.tile_begin; };
    auto lim_of = [&](int lt) {
        const int64_t p0 = (int64_t)lt * ppt;
        return (int)(min(min(p0 + ppt, B.npairs), full) - p0);
    };
    double2 zn[G];
    if (ring) {
        const int lt = tile_of(0), lim0 = lim_of(lt);
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int r = tid + u * ibs;
            zn[u] = ldp<NT>((u < K && r < lim0) ? zpair + (int64_t)lt * ppt + r : zpair);
        }
    }
    for (int j = 0; j < nrun; ++j) {
        const int lt = tile_of(j);
        const int64_t p0 = (int64_t)lt * ppt;
        const int lim = lim_of(lt);   // two-particle pairs of this tile
        double v[1] = {0.0};
        if (ring) {
            for (int k = 0; k < K; k += G) {
                // the next group: the rest of this tile, else the next tile's first
                const g_f64x2 *nbase = zpair + p0;
                int nr = 0, nlim = 0, nk = 0;
                if (k + G < K) {
                    nr = tid + (k + G) * ibs;
                    nlim = lim;
                    nk = K - (k + G);
                } else if (j + 1 < nrun) {
                    const int ltn = tile_of(j + 1);
                    nbase = zpair + (int64_t)ltn * ppt;
                    nr = tid;
                    nlim = lim_of(ltn);
                    nk = K;
                }
                // a ring of G slots: slot u's next load is issued as soon as
                // its current pair is taken
#pragma unroll
                for (int u = 0; u < G; ++u) {
                    const double2 zz = zn[u];
                    const int r = nr + u * ibs;
                    zn[u] = ldp<NT>((u < nk && r < nlim) ? nbase + r : zpair);
                    if (k + u >= K || tid + (k + u) * ibs >= lim) continue;
                    int k0, k1;
                    double w0, w1;
                    interp_index(zz.x, c0, c1, inv, nb, k0, w0);
                    interp_index(zz.y, c0, c1, inv, nb, k1, w1);
                    const unsigned j0 = (unsigned)(k0 - wlo), j1 = (unsigned)(k1 - wlo);
                    const unsigned i0 = min(j0, wpairs - 1), i1 = min(j1, wpairs - 1);
                    double t0 = sP[i0] * (1.0 - w0) + sP[i0 + 1] * w0;
                    double t1 = sP[i1] * (1.0 - w1) + sP[i1 + 1] * w1;
                    // outside the window: the pair table, with the wait in the branch
                    if (!FULLW && j0 >= wpairs) t0 = gather_interp(P2 + k0, w0);
                    if (!FULLW && j1 >= wpairs) t1 = gather_interp(P2 + k1, w1);
                    v[0] += t0;
                    v[0] += t1;
                }
            }
        } else if (nb < 2) {
            for (int64_t p = p0 + threadIdx.x; p < p0 + lim; p += bs) v[0] += P[0] + P[0];
        }
        if ((n & 1) && threadIdx.x == 0 && full >= p0 && full < min(p0 + ppt, B.npairs))
            v[0] += interp_pot(P, zp[n - 1], c0, c1, inv, nb);
        wave_sum<1>(v);   // (the DPP reduction slows this loop's streaming)
        if ((threadIdx.x & 63) == 0) B.ipart[(int64_t)lt * kTileWaves + (threadIdx.x >> 6)] = v[0];
    }
}

// interp_sum_run for tiles of one to three pairs per thread.  The sums over a
// run of tiles [lt0, lt1) of bunch B of the interpolated potential at the
// post-drift z (the E0 update of a wake bunch), one sum per tile and wave.
// The run first stages B.iwin entries of P around the
// centroid in LDS (the whole table unless it exceeds the LDS); particles
// outside the window read the pair table P2.  Each thread takes its pairs of
// the run in order -- pair j in tile lt0 + j/K at offset threadIdx.x +
// (j%K)*blockDim.x, K pairs per thread and tile -- through a ring of four
// streaming loads in flight, so a tile of one pair per thread costs no
// pipeline start.  A tile's sum is written when its last pair is added; it
// depends on the tile and the block size only.
template <bool FULLW, bool NT>
__device__ __forceinline__ void interp_sum_run_flat(const BunchDev &B, const int32_t *__restrict__ run,
                                                    int nrun) {
    extern __shared__ __align__(16) double sP[];
    const int nb = B.nbins;
    const double *__restrict__ P = B.P;
    const int w = B.iwin;
    const int wlo = window_lo(B.sc->centre_bin, w, nb);
    const unsigned wpairs = (unsigned)(w - 1);
    __syncthreads();   // the previous run's window is no longer read
    stage_window(sP, P + wlo, w);
    __syncthreads();
    const int64_t n = B.n, ppt = B.pairs_per_tile, full = n >> 1;
    const int tid = (int)threadIdx.x, ibs = kInterpThreads;
    const int K = (int)(ppt / ibs);   // pairs of each thread in a full tile
    const double c0 = B.c_first, c1 = B.c_last, inv = B.inv_s;
    const g_f64 *zp = (const g_f64 *)B.z;
    const g_f64x2 *P2 = (const g_f64x2 *)B.P2;
    const g_f64x2 *zpair = (const g_f64x2 *)zp;
    // two-particle pairs of tile lt (32-bit offsets within a tile)
    auto lim_of = [&](int lt) {
        const int64_t p0 = (int64_t)lt * ppt;
        return (int)(min(min(p0 + ppt, B.npairs), full) - p0);
    };
    // tile lt is complete: the single particle of an odd bunch (thread 0, the
    // bunch's last tile), then the per-wave sums
    auto flush = [&](double &v, int lt) {
        const int64_t p0 = (int64_t)lt * ppt;
        if ((n & 1) && threadIdx.x == 0 && full >= p0 && full < min(p0 + ppt, B.npairs))
            v += interp_pot(P, zp[n - 1], c0, c1, inv, nb);
        double s1[1] = {v};
        wave_total<1>(s1);
        if ((threadIdx.x & 63) == 63) B.ipart[(int64_t)lt * kTileWaves + (threadIdx.x >> 6)] = s1[0];
        v = 0.0;
    };
    auto tile_of = [&](int j) { return run[j] - B.tile_begin; };
    if (nb < 2 || full < 1) {   // a one-bin table, or no two-particle pair
        for (int j = 0; j < nrun; ++j) {
            const int lt = tile_of(j);
            double v = 0.0;
            const int lim = lim_of(lt);
            if (nb < 2)
                for (int r = tid; r < lim; r += ibs) v += P[0] + P[0];
            flush(v, lt);
        }
        return;
    }
    // The ring's loads are issued unconditionally (a lane without a next pair
    // reads pair 0 and ignores it), so that every wait for a slot is the same
    // count of younger loads.  The load and compute cursors are uniform.
    int lj = 0, lk = 0;   // the load cursor: entry lj of the run, pair lk of the thread
    auto load_next = [&]() -> double2 {
        const int r = tid + lk * ibs;
        const int llt = lj < nrun ? tile_of(lj) : 0;
        const bool ok = lj < nrun && r < lim_of(llt);
        const double2 x = ldp<NT>(ok ? zpair + (int64_t)llt * ppt + r : zpair);
        if (++lk == K) {
            lk = 0;
            ++lj;
        }
        return x;
    };
    double2 zn[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) zn[u] = load_next();
    const int J = nrun * K;
    int cj = 0, clt = tile_of(0), ck = 0, clim = lim_of(clt);
    double v = 0.0;
    for (int j = 0; j < J; j += 4) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (j + u >= J) break;
            const double2 zz = zn[u];
            zn[u] = load_next();
            if (tid + ck * ibs < clim) {
                int k0, k1;
                double w0, w1;
                interp_index(zz.x, c0, c1, inv, nb, k0, w0);
                interp_index(zz.y, c0, c1, inv, nb, k1, w1);
                const unsigned j0 = (unsigned)(k0 - wlo), j1 = (unsigned)(k1 - wlo);
                const unsigned i0 = min(j0, wpairs - 1), i1 = min(j1, wpairs - 1);
                double t0 = sP[i0] * (1.0 - w0) + sP[i0 + 1] * w0;
                double t1 = sP[i1] * (1.0 - w1) + sP[i1 + 1] * w1;
                // outside the window: the pair table, with the wait in the branch
                if (!FULLW && j0 >= wpairs) t0 = gather_interp(P2 + k0, w0);
                if (!FULLW && j1 >= wpairs) t1 = gather_interp(P2 + k1, w1);
                v += t0;
                v += t1;
            }
            if (++ck == K) {   // the last pair of tile clt
                flush(v, clt);
                ck = 0;
                if (++cj < nrun) {
                    clt = tile_of(cj);
                    clim = lim_of(clt);
                }
            }
        }
    }
}

// Both forms add each thread's pairs of a tile in ascending order and reduce
// them per wave in a fixed order (the large-tile form by a butterfly through
// LDS permutes, the small-tile form by DPP moves).  Which form a bunch takes
// depends on its size alone.  The per-tile groups cost less bookkeeping for
// large tiles, the run-wide ring no pipeline start per tile for small ones.
// FULLW: the window holds the whole table (no gathers), so the compiler's
// waits for the ring's slots count only the ring's own loads.
template <int G, bool FULLW, bool NT>
__device__ __forceinline__ void interp_sum_run_w(const BunchDev &B, const int32_t *run, int nrun) {
    if (G > 4 && B.pairs_per_tile >= G * (int64_t)kInterpThreads)
        interp_sum_run_tiles<G, FULLW, NT>(B, run, nrun);
    else if (B.pairs_per_tile >= 4 * (int64_t)kInterpThreads)
        interp_sum_run_tiles<4, FULLW, NT>(B, run, nrun);
    else
        interp_sum_run_flat<FULLW, NT>(B, run, nrun);
}

template <int G, bool NTZ>
__device__ __forceinline__ void interp_sum_run(const BunchDev &B, const int32_t *run, int nrun) {
    if (B.iwin >= B.nbins)
        interp_sum_run_w<G, true, NTZ>(B, run, nrun);
    else if (!cached(B))
        interp_sum_run_w<G, false, NTZ>(B, run, nrun);
    else
        interp_sum_run_w<G, false, false>(B, run, nrun);
}

// The interpolation sums of the wake + update_E0 bunches over a tile table:
// each workgroup walks its runs of the sums' tile order (a bunch shared by
// several workgroups has its tiles dealt to them in turn, as in the pass).
template <int G, bool NTZ>
__device__ __forceinline__ void interp_sum_blocks(const BunchDev *__restrict__ bds,
                                                  const int32_t *__restrict__ order,
                                                  const RunDev *__restrict__ runs,
                                                  const int32_t *__restrict__ rr) {
    const int r1 = rr[blockIdx.x + 1];
    for (int r = rr[blockIdx.x]; r < r1; ++r) {
        const RunDev rd = runs[r];
        const BunchDev &B = bds[rd.bunch];
        if ((B.flags & F_WAKE) && (B.flags & F_E0) && !(B.flags & F_CIC))
            interp_sum_run<G, NTZ>(B, order + rd.begin, rd.count);
    }
}

// At most 64 VGPRs, so that two workgroups fit a CU when both windows fit its
// LDS; rings of four loads.
template <bool NTZ>
__global__ __launch_bounds__(kInterpThreads) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_interp_sum(
    const BunchDev *__restrict__ bds, const int32_t *__restrict__ order,
    const RunDev *__restrict__ runs, const int32_t *__restrict__ rr) {
    interp_sum_blocks<4, NTZ>(bds, order, runs, rr);
}

// One workgroup per CU (a window of P larger than half the LDS): the
// registers of four waves per SIMD allow rings of eight loads.
template <bool NTZ>
__global__ __launch_bounds__(kInterpThreads) void k_interp_sum_deep(
    const BunchDev *__restrict__ bds, const int32_t *__restrict__ order,
    const RunDev *__restrict__ runs, const int32_t *__restrict__ rr) {
    interp_sum_blocks<8, NTZ>(bds, order, runs, rr);
}

// Per-tile sums of z, z^2, dE, dE^2 (the initial and final spreads,
// evolution.jl:245-253,461-467); mode 1 first applies the last turn's pending
// wake kick and re-centre (the epilogue) and writes dE back.  The tile is read
// in the turn pass's layout, 16-byte (z, z) and (dE, dE) pairs, thread t taking
// pairs lt*ppt + t + k*1024, two pairs' loads in flight; the single particle
// of an odd bunch goes to thread 0 of the bunch's last tile.  LP: the kick
// reads P from the LDS copy sP (the whole table) instead of global memory.
template <bool LP>
__device__ inline void moments_tile(const BunchDev &B, int lt, int mode, const double *sP,
                                    double *s_red) {
    const int64_t ppt = B.pairs_per_tile;
    const int64_t p0 = (int64_t)lt * ppt;
    const int64_t p1 = min(p0 + ppt, B.npairs);
    const int64_t full = B.n >> 1;                  // pairs with two particles
    const int64_t pf = min(p1, full);
    PassCtx c;
    if (mode == 1) load_ctx(B, c);
    const bool kick = (mode == 1) && c.pending_kick;
    const bool rec = (mode == 1) && c.pending_m;
    g_f64 *zp = (g_f64 *)B.z;
    g_f64 *ep = (g_f64 *)B.dE;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    auto one = [&](double z, double e) -> double {
        if (kick)                                                           // wakefield.jl:342-344
            e = e - (LP ? interp_pot(sP, z, c.c0, c.c1, c.inv_s, c.nb)
                        : interp_pot(c.P, z, c.c0, c.c1, c.inv_s, c.nb));
        if (rec) e = e - c.m_prev;                                          // evolution.jl:434
        v[0] += z;
        v[1] += z * z;
        v[2] += e;
        v[3] += e * e;
        return e;
    };
    constexpr int64_t kStep = kPassThreads;
    for (int64_t p = p0 + threadIdx.x; p < pf; p += 2 * kStep) {
        const int64_t q = p + kStep;
        const bool two = q < pf;
        const double2 za = ldnt((const g_f64x2 *)(zp + 2 * p));
        const double2 ea = ldnt((const g_f64x2 *)(ep + 2 * p));
        double2 zb = make_double2(0.0, 0.0), eb = make_double2(0.0, 0.0);
        if (two) {
            zb = ldnt((const g_f64x2 *)(zp + 2 * q));
            eb = ldnt((const g_f64x2 *)(ep + 2 * q));
        }
        const double a0 = one(za.x, ea.x), a1 = one(za.y, ea.y);
        if (kick || rec) stnt((g_f64x2 *)(ep + 2 * p), a0, a1);
        if (two) {
            const double b0 = one(zb.x, eb.x), b1 = one(zb.y, eb.y);
            if (kick || rec) stnt((g_f64x2 *)(ep + 2 * q), b0, b1);
        }
    }
    if ((B.n & 1) && full >= p0 && full < p1 && threadIdx.x == 0) {
        const int64_t i = B.n - 1;
        const double e = one(zp[i], ep[i]);
        if (kick || rec) ep[i] = e;
    }
    block_sum<4>(v, s_red);
    if (threadIdx.x == 0) {
        double *o = B.moments + 4 * (int64_t)lt;
        o[0] = v[0]; o[1] = v[1]; o[2] = v[2]; o[3] = v[3];
    }
}

// The tiles of a table, tile = blockIdx.x + k*gridDim.x.  With dynamic LDS
// (lds_entries > 0: the epilogue), a workgroup copies a bunch's potential
// into its LDS once for its tiles of that bunch when the bunch has a kick
// pending and its table fits; the per-tile arithmetic is the same either way.
__global__ __launch_bounds__(kPassThreads) void k_moments(const BunchDev *__restrict__ bds,
                                                          const int32_t *__restrict__ tile_bunch,
                                                          int ntiles, int mode, int lds_entries) {
    __shared__ double s_red[4 * 16];
    extern __shared__ __align__(16) double s_pot[];
    int staged = -1;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        __syncthreads();   // s_red and s_pot of the previous tile are no longer read
        const int bi = tile_bunch[tile];
        const BunchDev &B = bds[bi];
        const int lt = tile - B.tile_begin;
        const bool lp = mode == 1 && B.sc->pending_kick && B.nbins >= 2 &&
                        B.nbins <= lds_entries;
        if (lp && staged != bi) {
            for (int k = threadIdx.x; k < B.nbins; k += blockDim.x) s_pot[k] = B.P[k];
            staged = bi;
            __syncthreads();
        }
        if (lp)
            moments_tile<true>(B, lt, mode, s_pot, s_red);
        else
            moments_tile<false>(B, lt, mode, nullptr, s_red);
    }
}

__global__ __launch_bounds__(kFinalThreads) void k_moments_final(const BunchDev *__restrict__ bds,
                                                                 const int32_t *__restrict__ list,
                                                                 int mode) {
    __shared__ double s_red[4 * 16];
    const BunchDev &B = bds[list[blockIdx.x]];
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int t = threadIdx.x; t < B.ntiles; t += blockDim.x) {
        v[0] += B.moments[4 * t];
        v[1] += B.moments[4 * t + 1];
        v[2] += B.moments[4 * t + 2];
        v[3] += B.moments[4 * t + 3];
    }
    block_sum<4>(v, s_red);
    if (threadIdx.x == 0) {
        const double sE = gstd_from_sums(v[2], v[3], (double)B.n);
        const double sz = gstd_from_sums(v[0], v[1], (double)B.n);
        if (mode == 0) {
            B.out[0] = sE;
            B.out[1] = sz;
        } else {
            const TurnScalars &s = *B.sc;
            B.out[2] = sE;
            B.out[3] = sz;
            B.out[4] = s.E0;
            B.out[5] = (double)s.drift_skipped_count;
            B.out[6] = (double)s.turn;
            B.out[7] = (B.n > 0) ? v[0] / (double)B.n : 0.0;   // centroid z
            B.out[8] = (B.n > 0) ? v[2] / (double)B.n : 0.0;   // centroid dE
        }
    }
}

__global__ __launch_bounds__(kFinalThreads) void k_init(const BunchDev *__restrict__ bds,
                                                        const int32_t *__restrict__ list) {
    const BunchDev &B = bds[list[blockIdx.x]];
    if (threadIdx.x == 0) {
        TurnScalars s = {};
        turn_scalars(B, B.E0_init, s);
        s.m_prev = 0.0;
        s.pending_kick = 0;
        s.pending_m = 0;
        s.drift_skipped_count = 0;
        s.turn = 0;
        s.centre_bin = B.nbins / 2;   // the windows start at the middle of the grid
        *B.sc = s;
    }
}

// The E0 update (evolution.jl:419-429) from this turn's sums (psum: the sum of
// the interpolated potential over the bunch), and the scalars of the next turn.
// finish_on updates the turn scalars s in place.
__device__ inline void finish_on(const BunchDev &B, double psum, TurnScalars &s) {
    const uint32_t fl = B.flags;
    double E0 = s.E0;
    if (s.drift_skip) s.drift_skipped_count += 1;
    if (fl & F_E0) {                                  // evolution.jl:419-429
        const double mean = (s.sum_dE - psum) / (double)B.n;
        E0 = E0 + mean;
        s.m_prev = mean;
        s.pending_m = 1;
    } else {
        s.pending_m = 0;
    }
    s.pending_kick = (fl & F_WAKE) ? 1 : 0;
    if (B.mon) B.mon[4 * s.turn + 2] = E0;   // turn monitor: E0 after the turn
    s.turn += 1;
    turn_scalars(B, E0, s);
}

__device__ inline void finish_turn(const BunchDev &B, double psum) {
    TurnScalars s = *B.sc;
    finish_on(B, psum, s);
    *B.sc = s;
}

// The sum over the bunch of the interpolated potential from the cloud-in-cell
// deposit (F_CIC): sum_k (N_k - S_k) P[k] + S_k P[k+1] with
// S_k = (hi_k 2^32 + lo_k) / 2^51, over the cells with particles (a cell
// without particles adds nothing, even where P is not finite); NaN when some
// particle's weight was not finite (as its interpolated value is).  Threads
// [0, kRedThreads) take cells k = t + kRedThreads*j in ascending j and clear
// them for the next turn; the waves' sums are added in wave order.  Valid in
// thread 0; every thread of the workgroup calls it, and the sliced and the
// whole-bunch finalize get the same bits from it.
__device__ inline double cic_psum(const BunchDev &B, double *s_red) {
    const int nb = B.nbins;
    const int sp = B.spread;
    g_u64 *H = (g_u64 *)B.cic, *Lo = H + cic_half(nb);
    g_u32 *N = cic_n(B);
    const g_f64 *P = (const g_f64 *)B.P;
    if ((int)threadIdx.x < kRedThreads) {
        // U cells per thread at a time, every load of the group issued before
        // its arithmetic (the loads of empty cells read zeros and are not used)
        constexpr int U = 8;
        double v = 0.0;
        for (int k0 = (int)threadIdx.x; k0 < nb - 1; k0 += U * kRedThreads) {
            uint32_t cnt[U];
            unsigned long long hi[U], lo[U];
            double p0[U], p1[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = k0 + u * kRedThreads;
                const bool in = k < nb - 1;
                cnt[u] = in ? N[spread32(sp, k)] : 0u;
                hi[u] = in ? H[spread64(sp, k)] : 0ull;
                lo[u] = in ? Lo[spread64(sp, k)] : 0ull;
                p0[u] = in ? P[k] : 0.0;
                p1[u] = in ? P[k + 1] : 0.0;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (cnt[u]) {
                    const double sk = ((double)hi[u] * 0x1p32 + (double)lo[u]) * (1.0 / kCicScale);
                    v += ((double)cnt[u] - sk) * p0[u] + sk * p1[u];
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = k0 + u * kRedThreads;
                if (cnt[u]) {
                    N[spread32(sp, k)] = 0u;
                    H[spread64(sp, k)] = 0ull;
                    Lo[spread64(sp, k)] = 0ull;
                }
            }
        }
        v = butterfly(v);
        if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
    }
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0) {
        for (int w = 0; w < kRedThreads / 64; ++w) t += s_red[w];
        const uint32_t bad = N[hist_half(nb)];
        N[hist_half(nb)] = 0u;
        if (bad) t = __builtin_nan("");
    }
    return t;
}

// finish_turn after the sum of the interpolation sums, one workgroup per slice
// (a cloud-in-cell bunch: its deposit's sum in slice 0, zero in the others)
__global__ __launch_bounds__(kRedThreads) void k_finalize(const BunchDev *__restrict__ bds,
                                                          const int32_t *__restrict__ items) {
    __shared__ double s_red[16];
    const BunchDev &B = bds[items[2 * blockIdx.x]];
    const int r = items[2 * blockIdx.x + 1];
    const uint32_t fl = B.flags;
    double v[1] = {0.0};   // sum of the interpolated P (the sum of dE'-dE_init is in sc)
    if ((fl & F_E0) && (fl & F_WAKE)) {
        if (!(fl & F_CIC))
            slice_sum<1>(B.ipart, B.ntiles * kTileWaves, r, v, s_red);
        else if (r == 0)
            v[0] = cic_psum(B, s_red);
    }
    double t[1];
    if (!slices_done<1>(B, r, v, t) || threadIdx.x != 0) return;
    finish_turn(B, t[0]);
}

// cic_psum by a 1024-thread workgroup: four times the threads load the cells and
// form their terms, which go through LDS (sT[nb]) to the 256 threads that add
// them as cic_psum does (an empty cell's term is 0, which changes no sum): the
// same bits.  28 bunches of 4096 bins: 13.2 us by 256 threads, 6.5 us so.
__device__ inline double cic_psum_whole(const BunchDev &B, double *sT, double *s_red) {
    const int nb = B.nbins, sp = B.spread, t = (int)threadIdx.x;
    g_u64 *H = (g_u64 *)B.cic, *Lo = H + cic_half(nb);
    g_u32 *N = cic_n(B);
    const g_f64 *P = (const g_f64 *)B.P;
    constexpr int U = 4;
    for (int k0 = t; k0 < nb - 1; k0 += U * 1024) {
        uint32_t cnt[U];
        unsigned long long hi[U], lo[U];
        double p0[U], p1[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 1024;
            const bool in = k < nb - 1;
            cnt[u] = in ? N[spread32(sp, k)] : 0u;
            hi[u] = in ? H[spread64(sp, k)] : 0ull;
            lo[u] = in ? Lo[spread64(sp, k)] : 0ull;
            p0[u] = in ? P[k] : 0.0;
            p1[u] = in ? P[k + 1] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * 1024;
            double term = 0.0;
            if (cnt[u]) {
                const double sk = ((double)hi[u] * 0x1p32 + (double)lo[u]) * (1.0 / kCicScale);
                term = ((double)cnt[u] - sk) * p0[u] + sk * p1[u];
                N[spread32(sp, k)] = 0u;
                H[spread64(sp, k)] = 0ull;
                Lo[spread64(sp, k)] = 0ull;
            }
            if (k < nb - 1) sT[k] = term;
        }
    }
    uint32_t bad = 0;
    if (t == 0) bad = N[hist_half(nb)];
    __syncthreads();
    if (t < kRedThreads) {
        double v = 0.0;
        for (int k = t; k < nb - 1; k += kRedThreads) v += sT[k];
        v = butterfly(v);
        if ((t & 63) == 0) s_red[t >> 6] = v;
    }
    __syncthreads();
    double r = 0.0;
    if (t == 0) {
        for (int w = 0; w < kRedThreads / 64; ++w) r += s_red[w];
        N[hist_half(nb)] = 0u;
        if (bad) r = __builtin_nan("");
    }
    return r;
}

// k_finalize with one 1024-thread workgroup per bunch: the slices' sums of
// slice_sum sixteen at a time, four per group of four waves with all their
// loads in flight, added in slice order as slices_done adds them; a
// cloud-in-cell bunch's sum as slices_done adds slice 0's and the zeros.  The
// same bits without the count across workgroups and its exchange through
// memory (two slices: 6.3 us by two workgroups, 4.5 us so; sixteen slices, one
// CU's reading of 128 KB, gain nothing).
__global__ __launch_bounds__(1024) void k_finalize_whole(const BunchDev *__restrict__ bds,
                                                         const int32_t *__restrict__ list) {
    extern __shared__ __align__(16) double sT[];
    __shared__ double s_red[16][4];
    const BunchDev &B = bds[list[blockIdx.x]];
    const uint32_t fl = B.flags;
    const int t = (int)threadIdx.x, g = t >> 8, tl = t & 255, nred = B.nred;
    TurnScalars sc;
    if (t == 0) sc = *B.sc;
    double psum = 0.0;
    if ((fl & F_E0) && (fl & F_WAKE)) {
        if (fl & F_CIC) {
            const double d = cic_psum_whole(B, sT, s_red[0]);
            psum = nred == 1 ? d : 0.0 + d;
        } else {
            const g_f64 *a = (const g_f64 *)B.ipart;
            const int n = B.ntiles * kTileWaves;
            for (int r0 = 0; r0 < nred; r0 += 16) {
                double x[4][kRedPer];
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int k = 0; k < kRedPer; ++k) {
                        const int e = (r0 + 4 * q + g) * kRedEntries + tl + k * kRedThreads;
                        x[q][k] = e < n ? a[e] : 0.0;
                    }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    double v = 0.0;
#pragma unroll
                    for (int k = 0; k < kRedPer; ++k) v += x[q][k];
                    v = butterfly(v);
                    if ((tl & 63) == 0) s_red[4 * q + g][tl >> 6] = v;
                }
                __syncthreads();
                if (t < 64) {
                    double v = 0.0;
                    for (int w = 0; w < 4; ++w) v += s_red[t & 15][w];
                    for (int q = 0; q < 16 && r0 + q < nred; ++q) {
                        const double w = __shfl(v, q, 64);
                        psum = nred == 1 ? w : psum + w;
                    }
                }
                __syncthreads();
            }
        }
    }
    if (t == 0) {
        finish_on(B, psum, sc);
        *B.sc = sc;
    }
}

// cic_psum over the deposit and the potential staged in LDS (sN[nb+1],
// sH[2 nb], sP[nb]): the same cells per thread in the same order, the same
// expressions, so the same bits; the global counters are cleared as there.
__device__ inline double cic_psum_lds(const BunchDev &B, const uint32_t *sN,
                                      const unsigned long long *sH, const double *sP,
                                      double *s_red) {
    const int nb = B.nbins;
    const int sp = B.spread;
    g_u64 *H = (g_u64 *)B.cic, *Lo = H + cic_half(nb);
    g_u32 *N = cic_n(B);
    if ((int)threadIdx.x < kRedThreads) {
        double v = 0.0;
        for (int k = (int)threadIdx.x; k < nb - 1; k += kRedThreads) {
            const uint32_t cnt = sN[k];
            if (cnt) {
                const double sk = ((double)sH[k] * 0x1p32 + (double)sH[nb + k]) * (1.0 / kCicScale);
                v += ((double)cnt - sk) * sP[k] + sk * sP[k + 1];
                N[spread32(sp, k)] = 0u;
                H[spread64(sp, k)] = 0ull;
                Lo[spread64(sp, k)] = 0ull;
            }
        }
        v = butterfly(v);
        if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
    }
    __syncthreads();
    double t = 0.0;
    if (threadIdx.x == 0) {
        for (int w = 0; w < kRedThreads / 64; ++w) t += s_red[w];
        const uint32_t bad = sN[nb];
        N[hist_half(nb)] = 0u;
        if (bad) t = __builtin_nan("");
    }
    return t;
}

// The bin phase of a small bunch in one 1024-thread workgroup, in place of
// k_reduce_fwd, the convolution kernels and k_finalize.  Everything it reads
// is staged first, side by side (the turn scalars in thread 0's registers,
// this turn's counts, the line-density kernel, the wake spectra, the FFT
// twiddles, the deposit), so the phase waits on memory about twice instead
// of once per step.  Then: the pass sums reduced as whole_sum does (the sliced form's
// bits) into the turn scalars; the line density of every block packed and
// transformed side by side (nA blocks of F points); the spectral sums Y_o =
// sum_j X_{o-j} FFT(W_j) added in ascending j from zero, as k_conv_inv adds
// them, one (block, frequency) pair per thread; the inverse transforms side
// by side; P and P2 (and P in LDS); the E0 update from the deposit as
// k_finalize_whole.  Every value is the same expression of the same operands
// as on the launch-per-phase path, so the bunch gets the same bits either
// way.  LDS layout: bin_whole_layout.
__device__ inline void bin_phase_whole(const BunchDev &B) {
    extern __shared__ __align__(16) uint8_t s_bw[];
    __shared__ double s_nh, s_cur, s_red[16];
    const uint32_t fl = B.flags;
    const bool wake = (fl & F_WAKE) != 0;
    const bool cic = wake && (fl & F_E0) && (fl & F_CIC);
    const int nb = B.nbins, nA = B.nA, F = B.F, logF = B.logF, Bk = B.B, nJ = B.nJ;
    BinWholeLayout L = bin_whole_layout(wake ? nb : 0, nA, nJ, F, cic);
    double2 *sX = reinterpret_cast<double2 *>(s_bw);
    double2 *sW = sX + nA * F, *sY = sW + nJ * F;
    uint32_t *sHist = reinterpret_cast<uint32_t *>(s_bw + L.hist);
    double *sLam = reinterpret_cast<double *>(s_bw + L.lam);
    double *sP = reinterpret_cast<double *>(s_bw + L.pot);
    double2 *sTw = reinterpret_cast<double2 *>(s_bw + L.tw);
    unsigned long long *sH = reinterpret_cast<unsigned long long *>(s_bw + L.cic);
    uint32_t *sN = reinterpret_cast<uint32_t *>(sH + 2 * nb);
    const int sp = B.spread;
    TurnScalars sc;
    if (threadIdx.x == 0) sc = *B.sc;
    const int64_t turn = B.sc->turn;
    if (wake) {
        const uint32_t *h = hist_of(B, turn);
        for (int i = threadIdx.x; i < nb; i += blockDim.x) {
            sHist[i] = h[spread32(sp, i)];
            sLam[i] = B.lam[i];
        }
        if (nJ > 1) {
            const double2 *What = reinterpret_cast<const double2 *>(B.What);
            for (int u = threadIdx.x; u < nJ * F; u += blockDim.x) sW[u] = What[u];
        }
        const double2 *twg = reinterpret_cast<const double2 *>(B.tw);
        for (int u = threadIdx.x; u < F / 2; u += blockDim.x) sTw[u] = twg[u];
        if (cic) {
            const g_u64 *C = (const g_u64 *)B.cic;
            const g_u32 *N = cic_n(B);
            for (int i = threadIdx.x; i < nb; i += blockDim.x) {
                sH[i] = C[spread64(sp, i)];
                sH[nb + i] = C[cic_half(nb) + spread64(sp, i)];
                sN[i] = N[spread32(sp, i)];
            }
            if (threadIdx.x == 0) sN[nb] = N[hist_half(nb)];
        }
    }
    if (fl & (F_WAKE | F_E0)) {
        double t[4];
        whole_sum(B, t);   // its barriers also publish the staged LDS
        if (threadIdx.x == 0) {
            bin_scalars_on(B, t, sc);
            s_nh = sc.n_h;
            s_cur = sc.current;
        }
    }
    __syncthreads();
    if (wake) {
        const double nh = s_nh, cur = s_cur;
        const double2 *tw = sTw;   // the twiddles from LDS: no global load per FFT stage
        uint32_t *hn = hist_of(B, turn + 1);   // the next turn's half, cleared
        for (int i = threadIdx.x; i < nb; i += blockDim.x) hn[spread32(sp, i)] = 0u;
        if (nh == 0.0 || nJ == 0) {   // wakefield.jl:305-311
            for (int i = threadIdx.x; i < nb; i += blockDim.x) {
                put_potential(B, i, 0.0);
                sP[i] = 0.0;
            }
        } else {
            const double inv_nh = 1.0 / nh;
            auto dens = [&](int i) {   // line_density from the staged counts
                if (fl & F_LAG) i = nb - 1 - i;
                return sLam[i] * ((double)sHist[i] * inv_nh);
            };
            for (int u = threadIdx.x; u < nA * F; u += blockDim.x) {   // load_packed, every block
                const int a = u >> logF, m = u & (F - 1);
                double re = 0.0, im = 0.0;
                if (m < Bk) {
                    const int i = a * Bk + m;
                    if (i < nb) re = dens(i);
                    if (a >= 1) im = dens(i - Bk);
                }
                sX[a * F + bitrev(m, logF)] = make_double2(re, im);
            }
            fft_dit_forward(sX, F, logF, tw, nA);
            double2 *sR = sX;   // the spectra to invert
            if (nJ <= 1) {      // k_conv_fused's product
                const double2 *What = reinterpret_cast<const double2 *>(B.What);
                for (int u = threadIdx.x; u < nA * F; u += blockDim.x)
                    sX[u] = cmul(sX[u], What[u & (F - 1)]);
            } else {
                for (int u = threadIdx.x; u < nA * F; u += blockDim.x) {
                    const int o = u >> logF, k = u & (F - 1);
                    const int jmax = min(o, nJ - 1);
                    double2 acc = make_double2(0.0, 0.0);
                    for (int j = 0; j <= jmax; ++j) {
                        const double2 t = cmul(sX[(o - j) * F + k], sW[j * F + k]);
                        acc = make_double2(acc.x + t.x, acc.y + t.y);
                    }
                    sY[u] = acc;
                }
                sR = sY;
            }
            fft_dif_inverse(sR, F, logF, tw, nA);
            const double scale = cur / (double)F;
            for (int u = threadIdx.x; u < nA * Bk; u += blockDim.x) {   // store_block, every block
                const int o = u / Bk, m = u - o * Bk;
                const int i = o * Bk + m;
                if (i >= nb) continue;
                const double2 y0 = sR[o * F + bitrev(m, logF)];
                const double2 y1 = sR[o * F + bitrev(m + Bk, logF)];
                const int k = (fl & F_LAG) ? nb - 1 - i : i;
                const double v = (y0.x + y1.y) * scale;
                put_potential(B, k, v);
                sP[k] = v;
            }
        }
    }
    __syncthreads();   // P in LDS before the deposit's sum reads it
    double t = 0.0;
    if (cic) {
        const double d = cic_psum_lds(B, sN, sH, sP, s_red);
        t = B.nred == 1 ? d : 0.0 + d;
    }
    if (threadIdx.x == 0) {
        finish_on(B, t, sc);
        *B.sc = sc;
    }
}

// LDS ordering within one wave: its LDS operations execute in order, so only
// the compiler has to keep them so.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A workgroup barrier for data exchanged through LDS alone: __syncthreads also
// waits for the wave's outstanding global loads and stores.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The radix-2^2 butterflies of fft_dit_forward and fft_dif_inverse on four
// points in registers.
__device__ __forceinline__ void dit_pair(double2 (&x)[4], double2 w1, double2 wa, double2 wb) {
    double2 t = cmul(x[1], w1);
    const double2 a0 = cadd(x[0], t), a1 = csub(x[0], t);
    t = cmul(x[3], w1);
    const double2 a2 = cadd(x[2], t), a3 = csub(x[2], t);
    t = cmul(a2, wa);
    x[0] = cadd(a0, t);
    x[2] = csub(a0, t);
    t = cmul(a3, wb);
    x[1] = cadd(a1, t);
    x[3] = csub(a1, t);
}
// x holds points 0, h2, h, h + h2 of the inverse butterfly
__device__ __forceinline__ void dif_pair(double2 (&x)[4], double2 wa, double2 wb, double2 wc) {
    const double2 a0 = cadd(x[0], x[2]), a2 = cmul(csub(x[0], x[2]), wa);
    const double2 a1 = cadd(x[1], x[3]), a3 = cmul(csub(x[1], x[3]), wb);
    x[0] = cadd(a0, a1);
    x[1] = cmul(csub(a0, a1), wc);
    x[2] = cadd(a2, a3);
    x[3] = cmul(csub(a2, a3), wc);
}
__device__ __forceinline__ double2 dpp_swap1(double2 v) {   // the neighbouring lane's (lane ^ 1)
    return make_double2(dpp_move<0xB1, 0xF>(v.x), dpp_move<0xB1, 0xF>(v.y));
}

// k_bin_whole for the grids whose blocks are 64 bins (fits_bin_64: F = 128, at
// most 16 blocks, more than one wake block): the same products, sums and
// twiddles in the same order, so the same bits, arranged for latency.
// - A block's 32 butterflies stay in one half-wave from the packing to the last
//   stage, four points and all nine twiddles of a thread in registers: the
//   stages exchange through LDS without workgroup barriers, and the first
//   (its other inputs are the zero padding) and the last (half of its outputs
//   are needed, each from a neighbouring lane) cost no LDS pass.
// - The spectral sums take two consecutive output blocks per thread, so a wake
//   and a line-density value are read once per two products; every SIMD's
//   waves have the same number of products.
// - The phase's barriers order LDS only, so a load is waited for where its
//   value is used and not at the next barrier.
// - The binned count comes from the counts themselves, so the transforms do
//   not wait for the pass sums, which the waves that have no butterflies
//   reduce meanwhile; one of their lanes (kScalarThread) does the scalars.
// It is bound by LDS bandwidth: 264 KB for the forward transforms and 320 KB for
// the spectral sums of 1024 bins, at 128 B a cycle.  Measured in a turn: 1024
// bins 17.7 us (k_bin_whole) -> 9.4 us, 512 bins 12.7 -> 7.7 us.
constexpr int kScalarThread = 512;
// A point's place in its block in LDS: the stages' strides (2, 8 and 32 points of
// 16 bytes) and the contiguous reads then spread over all banks.
__device__ __forceinline__ int swz64(int e) { return e ^ ((e >> 3) & 7) ^ ((e >> 2) & 8); }
__global__ __launch_bounds__(1024) void k_bin_64(const BunchDev *__restrict__ bds,
                                                 const int32_t *__restrict__ list) {
    const BunchDev &B = bds[list[blockIdx.x]];
    extern __shared__ __align__(16) uint8_t s_bw[];
    __shared__ double s_sum[4][4 * 16], s_cur, s_red[16];
    __shared__ uint32_t s_cnt[16];
    __shared__ double2 s_tw[126];   // w1, wa, wb of stages (1,2): 2 each, (3,4): 8 each, (5,6): 32 each
    constexpr int F = 128, Bk = 64, logF = 7;
    const uint32_t fl = B.flags;
    const int nb = B.nbins, nA = B.nA, nJ = B.nJ, nred = B.nred;
    const bool cic = (fl & F_E0) && (fl & F_CIC);
    double2 *sX = reinterpret_cast<double2 *>(s_bw);
    double2 *sW = sX + nA * F, *sY = sW + nJ * F;
    double *sG = reinterpret_cast<double *>(sY + nA * F);   // the line density, nA * 64
    double *sP = sG + nA * Bk;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int sp = B.spread;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The first loads, all in flight together: the twiddles for LDS, s_tw[tid] =
    // w1, wa or wb (c = 0, 1, 2) of stage pair r at butterfly index k, by waves 0
    // and 1; the turn; both halves' counts (this turn's is known a load later).
    // Without branches: the compiler waited for all of them before the first
    // one's, and loaded the twiddles after (1024 bins: 9.6 -> 9.4 us).
    double2 twv = make_double2(0.0, 0.0);
    if (wave < 2) {
        const int r = (tid >= 6) + (tid >= 30), q = tid - 6 * r - 18 * (r >> 1);
        const int k = q & ((2 << (2 * r)) - 1), c = q >> (2 * r + 1), m = max(c - 1, 0);
        twv = ld2((const g_f64x2 *)B.tw + min((k + (m << (2 * r + 1))) << (5 - 2 * r - min(c, 1)), 63));
    }
    const int64_t turn = *(const __attribute__((address_space(1))) int64_t *)&B.sc->turn;
    const g_u32 *hist = (const g_u32 *)B.hist;
    const int bin = min(tid, nb - 1);
    const uint32_t h0 = hist[spread32(sp, bin)], h1 = hist[hist_half(nb) + spread32(sp, bin)];
    const double lam = ((const g_f64 *)B.lam)[bin];
    if (tid < 126) s_tw[tid] = twv;
    const uint32_t hc = tid < nb ? ((turn & 1) ? h1 : h0) : 0u;
    {
        uint32_t c = hc;
        c += __builtin_amdgcn_update_dpp(0, c, 0xB1, 0xF, 0xF, false);
        c += __builtin_amdgcn_update_dpp(0, c, 0x4E, 0xF, 0xF, false);
        c += __builtin_amdgcn_update_dpp(0, c, 0x141, 0xF, 0xF, false);
        c += __builtin_amdgcn_update_dpp(0, c, 0x140, 0xF, 0xF, false);
        c += __builtin_amdgcn_update_dpp(0, c, 0x142, 0xA, 0xF, false);
        c += __builtin_amdgcn_update_dpp(0, c, 0x143, 0x8, 0xF, false);
        if (lane == 63) s_cnt[wave] = c;   // row sums, then the rows into lane 63
    }
    lds_barrier();
    uint32_t total = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) total += s_cnt[w];
    const double nh = (double)total;
    if (tid < nb) ((g_u32 *)hist_of(B, turn + 1))[spread32(sp, tid)] = 0u;   // the next turn's half
    const double inv_nh = 1.0 / nh;
    if (tid < nA * Bk)   // line_density, in the convolution's order
        sG[(fl & F_LAG) && tid < nb ? nb - 1 - tid : tid] = tid < nb ? lam * ((double)hc * inv_nh) : 0.0;
    lds_barrier();
    // The other loads, by the waves without butterflies and while those run:
    // waves 8-15 the wake spectra and the pass sums, waves 12-15 this turn's
    // deposit as well.  (Issued before the density was packed, they held up
    // its barrier: a CU takes about 16 cycles for each 16-byte-per-lane load.)
    const int q = tid & 31, blk = tid >> 5;   // this thread's butterfly and its block
    const bool fft = wave < 8 && blk < nA;
    double2 R[12];   // waves 8-15: the pass sums' loads, then the spectra's; waves 0-7: the
                     // twiddles, 3 r + {0, 1, 2} = w1, wa, wb of stages 2r+1, 2r+2
    uint32_t cnt[4] = {0u, 0u, 0u, 0u};
    unsigned long long hi[4] = {0ull, 0ull, 0ull, 0ull}, lo[4] = {0ull, 0ull, 0ull, 0ull};
    uint32_t bad = 0;
    g_u64 *H = (g_u64 *)B.cic, *Lo = H + cic_half(nb);
    g_u32 *N = cic_n(B);
    const int ct = tid - 768;   // cic_psum's thread
    const int npart = B.ntiles * kTileWaves, tl = tid & 255;
    // group g of the pass sums (whole_sum's slices): waves 8-11 the even ones, 12-15 the odd ones
    auto load_part = [&](int g) {
#pragma unroll
        for (int k = 0; k < kRedPer; ++k) {
            const int e = g * kRedEntries + tl + k * kRedThreads;
            double2 a = make_double2(0.0, 0.0), b = make_double2(0.0, 0.0);
            if (e < npart) {
                const g_f64x2 *p = (const g_f64x2 *)B.part + 2 * (int64_t)e;
                a = ld2(p);
                b = ld2(p + 1);
            }
            R[2 * k] = a;
            R[2 * k + 1] = b;
        }
    };
    const int g0 = wave >= 12 ? 1 : 0;
    const int nW = nJ * F;
    if (wave >= 8) {
        const g_f64x2 *Wg = (const g_f64x2 *)B.What;
#pragma unroll
        for (int u = 0; u < 4; ++u) R[8 + u] = ld2(Wg + min(tid - 512 + 512 * u, nW - 1));
        if (g0 < nred) load_part(g0);
        if (cic && wave >= 12) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = ct + u * kRedThreads;
                if (k < nb - 1) {
                    cnt[u] = N[spread32(sp, k)];
                    hi[u] = H[spread64(sp, k)];
                    lo[u] = Lo[spread64(sp, k)];
                }
            }
        }
    }
    if (wave >= 8) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (tid - 512 + 512 * u < nW) sW[tid - 512 + 512 * u] = R[8 + u];
        // the pass sums' slices, block_sum's order within the group
        for (int g = g0; g < nred; g += 2) {
            if (g > 1) load_part(g);
            double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < kRedPer; ++k) {
                v[0] += R[2 * k].x;
                v[1] += R[2 * k].y;
                v[2] += R[2 * k + 1].x;
                v[3] += R[2 * k + 1].y;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[j] = butterfly(v[j]);
                if (lane == 0) s_sum[g][j * 16 + (tl >> 6)] = v[j];
            }
        }
    }
    const bool conv = nh != 0.0;   // else the potential is zero (wakefield.jl:305-311)
    if (fft) {
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const int hh = 2 << (2 * r), k = q & (hh - 1), t0 = r == 0 ? 0 : (r == 1 ? 6 : 30);
#pragma unroll
            for (int c = 0; c < 3; ++c) R[3 * r + c] = s_tw[t0 + c * hh + k];
        }
    }
    // the thread's places in its block at the stage pairs' strides
    const int e1 = ((q >> 1) << 3) | (q & 1), e3 = ((q >> 3) << 5) | (q & 7);
    if (conv && fft) {
        // stages 1 and 2 on packed points 8 (q >> 1) + (q & 1) + {0, 2, 4, 6},
        // which stage 0 leaves equal in pairs: input bitrev(8 (q >> 1) + 2 j)
        double2 y[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = blk * Bk + bitrev(8 * (q >> 1) + 2 * j, logF);
            y[j] = make_double2(sG[i], blk >= 1 ? sG[i - Bk] : 0.0);
        }
        dit_pair(y, R[0], R[1], R[2]);
        double2 *X = sX + blk * F;
#pragma unroll
        for (int j = 0; j < 4; ++j) X[swz64(e1 + 2 * j)] = y[j];
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = X[swz64(e3 + 8 * j)];
        dit_pair(y, R[3], R[4], R[5]);
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; ++j) X[swz64(e3 + 8 * j)] = y[j];
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = X[swz64(q + 32 * j)];
        dit_pair(y, R[6], R[7], R[8]);
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; ++j) X[swz64(q + 32 * j)] = y[j];
    }
    lds_barrier();
    if (conv) {
        // output blocks o0 = 2 og and o0 + 1 at frequency k.  og by wave pair, so
        // that every SIMD's four waves (w, w + 4, ...) have 68 products
        constexpr unsigned kGroups = 0x31462057u;   // 7, 5, 0, 2, 6, 4, 1, 3
        const int o0 = 2 * (int)((kGroups >> (4 * (wave >> 1))) & 7u);
        const int k = (wave & 1) * 64 + lane, kx = swz64(k);
        if (o0 < nA) {
            double2 a0 = make_double2(0.0, 0.0), a1 = a0;
            double2 x0 = sX[o0 * F + kx], x1 = o0 + 1 < nA ? sX[(o0 + 1) * F + kx] : a0;
            double2 w = sW[k];
            // step j: X_{o0-j}, X_{o0+1-j} times FFT(W_j); the next step's two
            // values are read before this step's products
            const int jm = min(o0, nJ - 1);
            for (int j = 0; j <= jm; ++j) {
                const double2 wn = sW[min(j + 1, nJ - 1) * F + k];
                const double2 xn = sX[max(o0 - j - 1, 0) * F + kx];
                a0 = cadd(a0, cmul(x0, w));
                a1 = cadd(a1, cmul(x1, w));
                x1 = x0;
                x0 = xn;
                w = wn;
            }
            if (jm + 1 < nJ) a1 = cadd(a1, cmul(x1, w));   // j = o0 + 1: block o0 + 1 alone
            sY[o0 * F + kx] = a0;
            if (o0 + 1 < nA) sY[(o0 + 1) * F + kx] = a1;
        }
    }
    lds_barrier();
    TurnScalars sc;
    if (tid == kScalarThread) {   // whole_sum's and slices_done's order
        sc = *B.sc;
        if (cic) bad = N[hist_half(nb)];
        double t[4] = {0.0, 0.0, 0.0, 0.0};
        for (int r = 0; r < nred; ++r)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                double s = 0.0;
                for (int w = 0; w < 4; ++w) s += s_sum[r][j * 16 + w];
                t[j] = nred == 1 ? s : t[j] + s;
            }
        bin_scalars_on(B, t, sc);
        s_cur = sc.current;
    }
    g_f64 *P = (g_f64 *)B.P;
    double2 y[4];
    if (conv && fft) {
        double2 *Y = sY + blk * F;
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = Y[swz64(q + 32 * j)];
        dif_pair(y, conj2(R[7]), conj2(R[8]), conj2(R[6]));
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; ++j) Y[swz64(q + 32 * j)] = y[j];
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = Y[swz64(e3 + 8 * j)];
        dif_pair(y, conj2(R[4]), conj2(R[5]), conj2(R[3]));
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; ++j) Y[swz64(e3 + 8 * j)] = y[j];
        wave_lds_fence();
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = Y[swz64(e1 + 2 * j)];
        dif_pair(y, conj2(R[1]), conj2(R[2]), conj2(R[0]));
    }
    lds_barrier();   // the current (kScalarThread)
    if (conv && fft) {
        // stage 0 on points 8 (q >> 1) + 2 j (this lane or its neighbour, even q)
        // and the one after it (odd q): output m = bitrev(8 (q >> 1) + 2 j) is
        // Re of their sum plus Im of their difference times tw[0]; even lanes
        // take j = 0, 1, odd lanes j = 2, 3
        const bool odd = q & 1;
        const double2 s0 = dpp_swap1(odd ? y[0] : y[2]), s1 = dpp_swap1(odd ? y[1] : y[3]);
        const double2 w0 = conj2(ld2((const g_f64x2 *)B.tw));
        const double scale = s_cur / (double)F;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const double2 s = u ? s1 : s0;
            const double2 a = odd ? s : y[u], c = odd ? y[2 + u] : s;
            const int i = blk * Bk + bitrev(8 * (q >> 1) + 2 * (u + (odd ? 2 : 0)), logF);
            const double2 d = csub(a, c);
            const double p = (cadd(a, c).x + (d.x * w0.y + d.y * w0.x)) * scale;
            if (i < nb) {
                const int k = (fl & F_LAG) ? nb - 1 - i : i;
                P[k] = p;
                sP[k] = p;
            }
        }
    } else if (!conv && tid < nb) {
        P[tid] = 0.0;
        sP[tid] = 0.0;
    }
    lds_barrier();
    double t = 0.0;
    if (cic) {   // cic_psum's cells per thread and order
        if (wave >= 12) {
            double a = 0.0;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = ct + u * kRedThreads;
                if (cnt[u]) {
                    const double sk = ((double)hi[u] * 0x1p32 + (double)lo[u]) * (1.0 / kCicScale);
                    a += ((double)cnt[u] - sk) * sP[k] + sk * sP[k + 1];
                    N[spread32(sp, k)] = 0u;
                    H[spread64(sp, k)] = 0ull;
                    Lo[spread64(sp, k)] = 0ull;
                }
            }
            a = butterfly(a);
            if (lane == 0) s_red[wave - 12] = a;
        }
        lds_barrier();
        if (tid == kScalarThread) {
            for (int w = 0; w < kRedThreads / 64; ++w) t += s_red[w];
            if (bad) {
                N[hist_half(nb)] = 0u;
                t = __builtin_nan("");
            }
            if (nred != 1) t = 0.0 + t;
        }
    }
    if (tid == kScalarThread) {
        finish_on(B, t, sc);
        *B.sc = sc;
    }
}

__global__ __launch_bounds__(1024) void k_bin_whole(const BunchDev *__restrict__ bds,
                                                    const int32_t *__restrict__ list) {
    bin_phase_whole(bds[list[blockIdx.x]]);
}

__global__ void k_turn_scalars(const BunchDev *__restrict__ bd, double E0, TurnScalars *out) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        TurnScalars s = {};
        turn_scalars(*bd, E0, s);
        *out = s;
    }
}

// ---------------------------------------------------------------------------
// stage kernels (unit parity); the same device functions as the fused pass
// ---------------------------------------------------------------------------

__global__ void k_stage_rf(double V, double sphis, double rf, double phis,
                           const double *__restrict__ z, double *__restrict__ dE, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const double phi = ((-z[i]) * rf) + phis;
        dE[i] = dE[i] + V * (dsin(phi) - sphis);
    }
}

__global__ void k_stage_qe(double exc, const double *__restrict__ r, double *__restrict__ dE,
                           int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dE[i] = dE[i] + exc * r[i];
}

__global__ void k_stage_sr(double damp, double *__restrict__ dE, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dE[i] = dE[i] * damp;
}

__global__ void k_stage_drift(int update_eta, const TurnScalars *__restrict__ scp, double mass,
                              double alpha_c, double phis, double *__restrict__ z,
                              const double *__restrict__ dE, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const TurnScalars &s = *scp;
    PassCtx c = {};
    c.rf = s.rf;
    c.inv_rf = s.inv_rf;
    c.phis = phis;
    c.inv_mass = 1.0 / mass;
    c.gamma0 = s.gamma0;
    c.alpha_c = alpha_c;
    c.kcoef = s.kcoef;
    c.coeff_c = s.coeff_c;
    c.drift_skip = s.drift_skip;
    c.flags = update_eta ? F_ETA : 0u;
    z[i] = drift(c, Flags<0>{c.flags}, z[i], dE[i]);
}

__global__ __launch_bounds__(kPassThreads) void k_stage_hist(const double *__restrict__ z,
                                                             int64_t n, double e0, double e1,
                                                             double inv, int nb,
                                                             uint32_t *__restrict__ ghist,
                                                             int use_lds) {
    extern __shared__ uint32_t s_hist[];
    uint32_t *h = use_lds ? s_hist : ghist;
    if (use_lds) {
        for (int b = threadIdx.x; b < nb; b += blockDim.x) s_hist[b] = 0u;
        __syncthreads();
    }
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int b = hist_bin(z[i], e0, e1, inv, nb);
        if (b >= 0) atomicAdd(&h[b], 1u);
    }
    if (use_lds) {
        __syncthreads();
        for (int b = threadIdx.x; b < nb; b += blockDim.x)
            if (s_hist[b]) atomicAdd(&ghist[b], s_hist[b]);
    }
}

__global__ void k_stage_interp_kick(const double *__restrict__ z, double *__restrict__ dE,
                                    int64_t n, const double *__restrict__ P, double c0, double c1,
                                    double inv, int nb) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dE[i] -= interp_pot(P, z[i], c0, c1, inv, nb);
}

__global__ void k_stage_normals(uint64_t seed, int64_t turn, int64_t i0, int64_t n,
                                double *__restrict__ out) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int64_t i = i0 + k;
    double a, b;
    qe_pair_normals(seed, (uint64_t)i >> 1, (uint32_t)turn, a, b);
    out[k] = (i & 1) ? b : a;
}

__global__ void k_generate(uint64_t seed, double mu_z, double sz, double mu_E, double sE,
                           double *__restrict__ z, double *__restrict__ dE, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t x[4];
    philox4x32_10((uint32_t)i, (uint32_t)((uint64_t)i >> 32), 0u, 1u, (uint32_t)seed,
                  (uint32_t)(seed >> 32), x);
    double a, b;
    box_muller(x, a, b);
    z[i] = mu_z + sz * a;
    dE[i] = mu_E + sE * b;
}

// generate_particles (evolution.jl:42-133) for n >= 2, step 1: one workgroup
// forms the sample covariance of m = min(n, 10000) independent samples
// (stream 2, regenerated from their counters for the second pass): mean-
// centred sums with m-1 normalisation (:75-82), variances floored at 1e-18,
// the diagonal lifted when the smallest eigenvalue is below 1e-12 (:89-94),
// then the lower Cholesky factor of the MvNormal (:97-101) -> L[0..2].
__device__ __forceinline__ void gen_sample(uint64_t seed, int64_t j, uint32_t stream, double &a,
                                           double &b) {
    uint32_t x[4];
    philox4x32_10((uint32_t)j, (uint32_t)((uint64_t)j >> 32), 0u, stream, (uint32_t)seed,
                  (uint32_t)(seed >> 32), x);
    box_muller(x, a, b);
}

__global__ __launch_bounds__(1024) void k_gen_cov(uint64_t seed, double mu_z, double mu_E,
                                                  double sz, double sE, int64_t m,
                                                  double *__restrict__ L) {
    __shared__ double s_red[3 * 16];
    __shared__ double s_mean[2];
    double v[3] = {0.0, 0.0, 0.0};
    for (int64_t j = threadIdx.x; j < m; j += blockDim.x) {
        double a, b;
        gen_sample(seed, j, 2u, a, b);
        v[0] += mu_z + sz * a;
        v[1] += mu_E + sE * b;
    }
    double w[2] = {v[0], v[1]};
    block_sum<2>(w, s_red);
    if (threadIdx.x == 0) {
        s_mean[0] = w[0] / (double)m;
        s_mean[1] = w[1] / (double)m;
    }
    __syncthreads();
    const double mz = s_mean[0], me = s_mean[1];
    v[0] = v[1] = v[2] = 0.0;
    for (int64_t j = threadIdx.x; j < m; j += blockDim.x) {
        double a, b;
        gen_sample(seed, j, 2u, a, b);
        const double dz = (mu_z + sz * a) - mz, de = (mu_E + sE * b) - me;
        v[0] += dz * dz;
        v[1] += de * de;
        v[2] += dz * de;
    }
    block_sum<3>(v, s_red);
    if (threadIdx.x == 0) {
        const double md = (double)(m - 1);
        double a = v[0] / md, c = v[1] / md;
        const double b = v[2] / md;
        a = a < 1e-18 ? 1e-18 : a;
        c = c < 1e-18 ? 1e-18 : c;
        // smallest eigenvalue as det / largest: no cancellation when a << c
        const double h = (a - c) * 0.5;
        const double lmax = (a + c) * 0.5 + sqrt(h * h + b * b);
        const double lmin = (a * c - b * b) / lmax;
        if (lmin < 1e-12) {
            const double lift = 1e-12 - lmin;
            a += lift;
            c += lift;
        }
        const double l11 = sqrt(a);
        const double l21 = b / l11;
        L[0] = l11;
        L[1] = l21;
        L[2] = sqrt(c - l21 * l21);
    }
}

// step 2: particle i = mu + L xi, xi the stream-1 normals of particle i
__global__ void k_gen_mvn(uint64_t seed, double mu_z, double mu_E, const double *__restrict__ L,
                          double *__restrict__ z, double *__restrict__ dE, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double l11 = L[0], l21 = L[1], l22 = L[2];
    double x1, x2;
    gen_sample(seed, i, 1u, x1, x2);
    z[i] = mu_z + l11 * x1;
    dE[i] = mu_E + (l21 * x1 + l22 * x2);
}

// Two-pass statistics of (z, dE): means, compute_std (utils.jl:531-544) and
// Statistics.cor (the emittance figure of merit, figures_of_merit.jl:36-47).
// Block b sums [b*chunk, (b+1)*chunk); mode 0 sums the values, mode 1 the
// squared deviations and the cross product about stats[0..1].
__global__ __launch_bounds__(1024) void k_pair_sums(int mode, const double *__restrict__ z,
                                                    const double *__restrict__ dE, int64_t n,
                                                    int64_t chunk, const double *__restrict__ stats,
                                                    double *__restrict__ part) {
    __shared__ double s_red[3 * 16];
    const int64_t i0 = (int64_t)blockIdx.x * chunk;
    const int64_t i1 = min(n, i0 + chunk);
    double v[3] = {0.0, 0.0, 0.0};
    const double cz = mode ? stats[0] : 0.0, ce = mode ? stats[1] : 0.0;
    for (int64_t i = i0 + threadIdx.x; i < i1; i += blockDim.x) {
        if (mode) {
            const double a = z[i] - cz, b = dE[i] - ce;
            v[0] += a * a;
            v[1] += b * b;
            v[2] += a * b;
        } else {
            v[0] += z[i];
            v[1] += dE[i];
        }
    }
    block_sum<3>(v, s_red);
    if (threadIdx.x == 0) {
        part[3 * blockIdx.x] = v[0];
        part[3 * blockIdx.x + 1] = v[1];
        part[3 * blockIdx.x + 2] = v[2];
    }
}

// mode 0: stats[0..1] = means; mode 1: stats[2..3] = sample standard
// deviations of z and dE, stats[4] = their correlation
__global__ __launch_bounds__(256) void k_pair_sums_final(int mode, const double *__restrict__ part,
                                                         int nblocks, int64_t n,
                                                         double *__restrict__ stats) {
    __shared__ double s_red[3 * 16];
    double v[3] = {0.0, 0.0, 0.0};
    for (int b = threadIdx.x; b < nblocks; b += blockDim.x) {
        v[0] += part[3 * b];
        v[1] += part[3 * b + 1];
        v[2] += part[3 * b + 2];
    }
    block_sum<3>(v, s_red);
    if (threadIdx.x == 0) {
        if (mode == 0) {
            stats[0] = v[0] / (double)n;
            stats[1] = v[1] / (double)n;
        } else {
            const double vz = v[0] / (double)(n - 1), ve = v[1] / (double)(n - 1);
            stats[2] = sqrt(jl_max(0.0, vz));   // compute_std: sqrt(max(0, variance))
            stats[3] = sqrt(jl_max(0.0, ve));
            double r = v[2] / sqrt(v[0] * v[1]);   // Statistics.cor, clamped to [-1, 1]
            stats[4] = (r != r) ? r : (r > 1.0 ? 1.0 : (r < -1.0 ? -1.0 : r));
        }
    }
}

// Plain device copy (16 B per lane per step, streaming loads and stores,
// 64 workgroups of 1024 per CU): the HBM ceiling of a kernel that reads and
// writes each byte once, and the calibration of the HBM byte counters.
// grid-stride copy with four 16-byte loads of each thread in flight before
// its stores (the fastest form of a sweep over grid, block size and loads in
// flight on MI355X)
__global__ __launch_bounds__(1024) void k_stream_copy(const f64x2 *__restrict__ src,
                                                      f64x2 *__restrict__ dst, int64_t n2) {
    const int64_t st = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n2; i += 4 * st) {
        f64x2 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + u * st < n2) v[u] = __builtin_nontemporal_load(src + i + u * st);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + u * st < n2) __builtin_nontemporal_store(v[u], dst + i + u * st);
    }
}

// ---------------------------------------------------------------------------
// launch wrappers
// ---------------------------------------------------------------------------

static inline unsigned blocks_for(int64_t n, int t) { return (unsigned)((n + t - 1) / t); }

hipError_t configure_kernels(int lds) {
    const void *fns[] = {(const void *)k_turn_pass<true>, (const void *)k_turn_pass<false>,
                         (const void *)k_turn_pass_std<true>, (const void *)k_turn_pass_std<false>,
                         (const void *)k_conv_fused,
                         (const void *)k_conv_fwd, (const void *)k_reduce_fwd,
                         (const void *)k_conv_inv,
                         (const void *)k_conv_spec, (const void *)k_conv_out,
                         (const void *)k_fft_wake, (const void *)k_stage_hist,
                         (const void *)k_interp_sum<true>, (const void *)k_interp_sum<false>,
                         (const void *)k_interp_sum_deep<true>, (const void *)k_interp_sum_deep<false>,
                         (const void *)k_bin_whole, (const void *)k_bin_64};
    hipError_t last = hipSuccess;
    for (const void *f : fns) {
        hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) last = e;
    }
    return last;
}

hipError_t launch_stream_copy(const double *src, double *dst, int64_t n, int blocks, hipStream_t s) {
    if (n <= 1) return hipSuccess;
    hipLaunchKernelGGL(k_stream_copy, dim3((unsigned)blocks), dim3(1024), 0, s,
                       reinterpret_cast<const f64x2 *>(src), reinterpret_cast<f64x2 *>(dst), n / 2);
    return hipGetLastError();
}

hipError_t launch_moments(const BunchDev *bds, const int32_t *tb, int ntiles, int mode,
                          int grid, int lds_entries, hipStream_t s) {
    if (ntiles <= 0) return hipSuccess;
    grid = grid > 0 ? min(grid, ntiles) : ntiles;
    hipLaunchKernelGGL(k_moments, dim3(grid), dim3(kPassThreads), (size_t)lds_entries * 8, s, bds,
                       tb, ntiles, mode, lds_entries);
    return hipGetLastError();
}

hipError_t launch_moments_final(const BunchDev *bds, const int32_t *list, int nb, int mode,
                                hipStream_t s) {
    if (nb <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_moments_final, dim3(nb), dim3(kFinalThreads), 0, s, bds, list, mode);
    return hipGetLastError();
}

hipError_t launch_init(const BunchDev *bds, const int32_t *list, int nb, hipStream_t s) {
    if (nb <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_init, dim3(nb), dim3(kFinalThreads), 0, s, bds, list);
    return hipGetLastError();
}

hipError_t launch_turn_pass(const BunchDev *bds, const int32_t *order, const RunDev *runs,
                            const int32_t *rr, int grid, int slices, size_t lds, int std_only,
                            int unb, bool keep_z, hipStream_t s) {
    if (grid <= 0) return hipSuccess;
    const dim3 blocks((unsigned)(grid * slices)), threads((unsigned)(kPassThreads / slices));
    auto *k = std_only ? (keep_z ? k_turn_pass_std<false> : k_turn_pass_std<true>)
                       : (keep_z ? k_turn_pass<false> : k_turn_pass<true>);
    hipLaunchKernelGGL(k, blocks, threads, lds, s, bds, order, runs, rr, unb);
    return hipGetLastError();
}

hipError_t launch_free_turns(const BunchDev *bds, const RunDev *items, int nitems,
                             const int32_t *list, int nlist, int turns, hipStream_t s) {
    if (nitems <= 0 || turns <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_free_turns, dim3((unsigned)nitems), dim3(kFreeThreads), 0, s, bds, items,
                       turns);
    hipLaunchKernelGGL(k_free_finish, dim3((unsigned)nlist), dim3(kFreeThreads), 0, s, bds, list,
                       turns);
    return hipGetLastError();
}

// A butterfly per thread and stage of the longest transform (2048 points, 131072
// bins: k_reduce_fwd 13.1 -> 11.3 us, k_conv_out 11.2 -> 9.6 by 1024 threads)
static unsigned fft_threads(int Fmax) {
    return (unsigned)std::min(std::max(Fmax / 2, kConvThreads), kConvMaxThreads);
}

hipError_t launch_conv(int kind, const BunchDev *bds, const int32_t *items, int nitems, int Fmax,
                       hipStream_t s, int threads) {
    if (nitems <= 0) return hipSuccess;
    const size_t lds = (size_t)Fmax * 16;
    if (kind == CONV_FUSED)
        hipLaunchKernelGGL(k_conv_fused, dim3(nitems), dim3(kConvThreads), lds, s, bds, items);
    else if (kind == CONV_FWD)
        hipLaunchKernelGGL(k_conv_fwd, dim3(nitems), dim3(kConvThreads), lds, s, bds, items);
    else if (kind == CONV_INV)
        hipLaunchKernelGGL(k_conv_inv, dim3(nitems), dim3(kConvInvThreads), lds, s, bds, items);
    else if (kind == CONV_SPEC)
        hipLaunchKernelGGL(k_conv_spec, dim3(nitems), dim3((unsigned)threads), (size_t)Fmax, s, bds,
                           items);
    else
        hipLaunchKernelGGL(k_conv_out, dim3(nitems), dim3(fft_threads(Fmax)), lds, s, bds, items);
    return hipGetLastError();
}

hipError_t launch_interp_sum(const BunchDev *bds, const int32_t *order, const RunDev *runs,
                             const int32_t *rr, int grid, size_t lds_bytes, bool deep,
                             bool keep_z, hipStream_t s) {
    if (grid <= 0) return hipSuccess;
    auto *k = deep ? (keep_z ? k_interp_sum_deep<false> : k_interp_sum_deep<true>)
                   : (keep_z ? k_interp_sum<false> : k_interp_sum<true>);
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(kInterpThreads), lds_bytes, s, bds, order, runs,
                       rr);
    return hipGetLastError();
}

hipError_t launch_finalize(const BunchDev *bds, const int32_t *items, int nitems, hipStream_t s) {
    if (nitems <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_finalize, dim3(nitems), dim3(kRedThreads), 0, s, bds, items);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void k_copies(CopyList l) {
    const uint32_t n = l.e[blockIdx.x].words, st = gridDim.y * 256u;
    g_u32 *d = (g_u32 *)l.e[blockIdx.x].dst;
    const g_u32 *s = (const g_u32 *)l.e[blockIdx.x].src;
    if (!l.e[blockIdx.x].src) {
        for (uint32_t i = blockIdx.y * 256u + threadIdx.x; i < n; i += st) d[i] = 0u;
        return;
    }
    for (uint32_t i = blockIdx.y * 256u + threadIdx.x; i < n; i += 4 * st) {
        uint32_t x[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) x[u] = s[min(i + u * st, n - 1)];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
            if (i + u * st < n) d[i + u * st] = x[u];
    }
}

hipError_t launch_copies(const CopyList &l, int n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    uint32_t words = 0;
    for (int k = 0; k < n; ++k) words = std::max(words, l.e[k].words);
    const uint32_t gy = std::min<uint32_t>(64, (words + 1023) / 1024);
    hipLaunchKernelGGL(k_copies, dim3((unsigned)n, std::max<uint32_t>(gy, 1)), dim3(256), 0, s, l);
    return hipGetLastError();
}

hipError_t launch_hist_slabs(const BunchDev *bds, const int32_t *items, int nitems, hipStream_t s) {
    if (nitems <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_hist_slabs, dim3(nitems), dim3(1024), 0, s, bds, items);
    return hipGetLastError();
}

hipError_t launch_reduce_fwd(const BunchDev *bds, const int32_t *red, int nred, const int32_t *items,
                             int nitems, int Fmax, hipStream_t s) {
    if (nred + nitems <= 0) return hipSuccess;
    static_assert(kRedThreads <= kConvThreads, "one launch for both");
    hipLaunchKernelGGL(k_reduce_fwd, dim3(nred + nitems), dim3(nitems > 0 ? fft_threads(Fmax) : kRedThreads),
                       nitems > 0 ? (size_t)Fmax * 16 : 0, s, bds, red, nred, items);
    return hipGetLastError();
}

hipError_t launch_bin_whole(const BunchDev *bds, const int32_t *list, int nb, size_t lds,
                            hipStream_t s) {
    if (nb <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_bin_whole, dim3(nb), dim3(1024), lds, s, bds, list);
    return hipGetLastError();
}

hipError_t launch_bin_64(const BunchDev *bds, const int32_t *list, int nb, size_t lds,
                         hipStream_t s) {
    if (nb <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_bin_64, dim3(nb), dim3(1024), lds, s, bds, list);
    return hipGetLastError();
}

hipError_t launch_finalize_whole(const BunchDev *bds, const int32_t *list, int nb, size_t lds,
                                 hipStream_t s) {
    if (nb <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_finalize_whole, dim3(nb), dim3(1024), lds, s, bds, list);
    return hipGetLastError();
}

__global__ void k_zero(uint32_t *__restrict__ p, int64_t words) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0u;
}

hipError_t launch_zero(void *p, size_t bytes, hipStream_t s) {
    const int64_t words = (int64_t)(bytes / 4);
    if (words <= 0) return hipSuccess;
    const int64_t b = (words + 255) / 256;
    hipLaunchKernelGGL(k_zero, dim3((unsigned)(b < 1024 ? b : 1024)), dim3(256), 0, s,
                       static_cast<uint32_t *>(p), words);
    return hipGetLastError();
}

hipError_t launch_resonator_table(double *W, int nb, double step, const ResonatorSet &rs,
                                  hipStream_t s) {
    hipLaunchKernelGGL(k_resonator_table, dim3(blocks_for(nb, 256)), dim3(256), 0, s, W, nb, step,
                       rs);
    return hipGetLastError();
}

hipError_t launch_reference_tables(double *W, double *lam, int nb, double zw, double wf, double ws,
                                   double inv_ctau, double s_inv, double ef, hipStream_t s) {
    if (nb <= 0 || (!W && !lam)) return hipSuccess;
    hipLaunchKernelGGL(k_reference_tables, dim3(blocks_for(nb, 256)), dim3(256), 0, s, W, lam, nb, zw,
                       wf, ws, inv_ctau, s_inv, ef);
    return hipGetLastError();
}

hipError_t launch_fft_wake(const BunchDev *bd, const double *W, int nJ, int F, hipStream_t s) {
    if (nJ <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fft_wake, dim3(nJ), dim3(kConvThreads), (size_t)F * 16, s, bd, W);
    return hipGetLastError();
}

hipError_t launch_stage_rf(double V, double sphis, double rf, double phis, const double *z,
                           double *dE, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stage_rf, dim3(blocks_for(n, 256)), dim3(256), 0, s, V, sphis, rf, phis,
                       z, dE, n);
    return hipGetLastError();
}

hipError_t launch_stage_qe(double exc, const double *r, double *dE, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stage_qe, dim3(blocks_for(n, 256)), dim3(256), 0, s, exc, r, dE, n);
    return hipGetLastError();
}

hipError_t launch_stage_sr(double damp, double *dE, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stage_sr, dim3(blocks_for(n, 256)), dim3(256), 0, s, damp, dE, n);
    return hipGetLastError();
}

hipError_t launch_stage_drift(int update_eta, const TurnScalars *sc, double mass, double alpha_c,
                              double phis, double *z, const double *dE, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stage_drift, dim3(blocks_for(n, 256)), dim3(256), 0, s, update_eta, sc,
                       mass, alpha_c, phis, z, dE, n);
    return hipGetLastError();
}

hipError_t launch_stage_hist(const double *z, int64_t n, double e0, double e1, double inv, int nb,
                             uint32_t *hist, int use_lds, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    int64_t blocks = blocks_for(n, kPassThreads);
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(k_stage_hist, dim3((unsigned)blocks), dim3(kPassThreads),
                       use_lds ? (size_t)nb * 4 : 0, s, z, n, e0, e1, inv, nb, hist, use_lds);
    return hipGetLastError();
}

hipError_t launch_stage_interp_kick(const double *z, double *dE, int64_t n, const double *P,
                                    double c0, double c1, double inv, int nb, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stage_interp_kick, dim3(blocks_for(n, 256)), dim3(256), 0, s, z, dE, n,
                       P, c0, c1, inv, nb);
    return hipGetLastError();
}

hipError_t launch_stage_normals(uint64_t seed, int64_t turn, int64_t i0, int64_t n, double *out,
                                hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stage_normals, dim3(blocks_for(n, 256)), dim3(256), 0, s, seed, turn, i0,
                       n, out);
    return hipGetLastError();
}

hipError_t launch_generate(uint64_t seed, double mu_z, double sz, double mu_E, double sE,
                           double *z, double *dE, int64_t n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_generate, dim3(blocks_for(n, 256)), dim3(256), 0, s, seed, mu_z, sz, mu_E,
                       sE, z, dE, n);
    return hipGetLastError();
}

hipError_t launch_generate_particles(uint64_t seed, double mu_z, double mu_E, double sz, double sE,
                                     double *z, double *dE, int64_t n, double *work,
                                     hipStream_t s) {
    if (n < 2) return hipSuccess;
    double *L = work;
    hipLaunchKernelGGL(k_gen_cov, dim3(1), dim3(1024), 0, s, seed, mu_z, mu_E, sz, sE,
                       n < 10000 ? n : (int64_t)10000, L);
    hipLaunchKernelGGL(k_gen_mvn, dim3(blocks_for(n, 256)), dim3(256), 0, s, seed, mu_z, mu_E,
                       (const double *)L, z, dE, n);
    return launch_pair_stats(z, dE, n, work + 4, work + 12, s);
}

hipError_t launch_pair_stats(const double *z, const double *dE, int64_t n, double *stats,
                             double *part, hipStream_t s) {
    if (n < 2) return hipSuccess;
    const int64_t nbl = (n + 1023) / 1024;
    const int nb = (int)(nbl < kStatBlocks ? nbl : kStatBlocks);
    const int64_t chunk = (n + nb - 1) / nb;
    for (int mode = 0; mode < 2; ++mode) {
        hipLaunchKernelGGL(k_pair_sums, dim3(nb), dim3(1024), 0, s, mode, z, dE, n, chunk,
                           (const double *)stats, part);
        hipLaunchKernelGGL(k_pair_sums_final, dim3(1), dim3(256), 0, s, mode, (const double *)part,
                           nb, n, stats);
    }
    return hipGetLastError();
}

hipError_t launch_turn_scalars(const BunchDev *bd, double E0, TurnScalars *out, hipStream_t s) {
    hipLaunchKernelGGL(k_turn_scalars, dim3(1), dim3(64), 0, s, bd, E0, out);
    return hipGetLastError();
}

}  // namespace hm
