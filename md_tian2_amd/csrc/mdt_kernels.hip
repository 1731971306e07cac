// mdt_kernels.hip -- CDNA4 (gfx950) kernels for batched EMT forces and the
// md_tian2 propagators.
//
// k_replica: calc_force, one workgroup per replica (trajectory t, bead b).
//   phase 0: stage the replica in LDS;
//   phase 1: the rows of neighbours, (index | periodic-image code << 11), kept from
//            an earlier launch or built by a minimum-image scan of all atoms;
//   phase 2 (pass A): every unordered pair once, by its owner atom:
//            sigma_k += csig(tk,tn) f_sigma_tn(r) and sigma_n += csig(tn,tk)
//            f_sigma_tk(r); then per atom s, dens, E_coh + vref and
//            G_a = dE/dsigma_a;
//   phase 3 (pass B): the pair's dE/dr (density part through G of both
//            atoms, pair-potential part directly) gives +F on the owner and
//            -F on the partner (Newton's third law); then set_acceleration.
//   Every sum is one of integers, or of FP64 multiples of a grid: results are
//   bitwise reproducible whatever order the lanes' atomics land in.
// k_traj_classical (one-bead batches) and k_prop / k_com_ring (the others):
//   propagate_2 of the previous step, propagate_1, COM removal and (P > 1)
//   the ring-polymer free step (src/md_algo.f90:37-106, src/rpmd.f90:309-452).
#include <hip/hip_runtime.h>

#include "mdt_device.h"
#include "mdt_math.h"
#include "mdt_philox.h"

#define MDT_NBR_IDX_BITS 11
#define MDT_NBR_IDX_MASK 0x7FF

namespace {

// Tables every lane indexes by atom type: kept in LDS (divergent indices).
struct LdsTypes {
    double bs0[MDT_MAXT], kdb[MDT_MAXT], betaeta2[MDT_MAXT];
    double e0[MDT_MAXT], lambda[MDT_MAXT], v0[MDT_MAXT], kappa[MDT_MAXT], n0[MDT_MAXT];
    double densc[MDT_MAXT];
    double etaT[MDT_MAXT], kdbT[MDT_MAXT];  // -eta2, -kdb in mdt_exp_t's unit
    double csig[MDT_MAXT * MDT_MAXT], etad[MDT_MAXT * MDT_MAXT], wv[MDT_MAXT * MDT_MAXT];
    double exptab[MDT_EXP_TAB_N];
    int owner[MDT_MAXT], pair_on[MDT_MAXT * MDT_MAXT];
    // FP32 copies for the single-precision pair terms; *_l2 carry a factor
    // log2(e) so that exp(-a x) = 2^(-a_l2 x)
    float f_eta2l2[MDT_MAXT], f_kdbl2[MDT_MAXT], f_kdb[MDT_MAXT];
    float f_csig[MDT_MAXT * MDT_MAXT], f_etad[MDT_MAXT * MDT_MAXT], f_wv[MDT_MAXT * MDT_MAXT];
};
struct LdsTables : LdsTypes {
    double eta2[MDT_MAXT];
    double csig48[MDT_MAXT * MDT_MAXT];  // csig * 2^48: partner sigma terms in fixed-point units
    double shift[27 * 3];  // cartesian lattice translation of each image code
    int algo[MDT_MAXT], is_proj[MDT_MAXT];
};

#define MDT_LOG2E 1.4426950408889634

struct CellRegs {
    double h[9], ih[9];
};

__device__ __forceinline__ void load_cell(const BatchView &bv, int t, CellRegs &c) {
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        c.h[k] = bv.cell[9 * t + k];
        c.ih[k] = bv.icell[9 * t + k];
    }
}

template <int TPA>
__device__ __forceinline__ double group_sum(double v) {
#pragma unroll
    for (int o = 1; o < TPA; o <<= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Langevin coefficients, src/md_algo.f90:165-198 (langevin_1) and :253-285
struct LanCoef {
    double c0, c1, c2, sr, sv, crv;
};

__device__ __forceinline__ LanCoef lan_coef(double fric, double dt, double temp, bool exact) {
#pragma clang fp contract(off)
    LanCoef L;
    const double xidt = fric * dt;
    const double xidt2 = xidt * xidt;
    const double ixidt = dt / xidt;
    if (exact) {
        L.c0 = exp(-xidt);
        L.c1 = (1 - L.c0) * ixidt;
        L.c2 = (1 - L.c1 / dt) * ixidt;
        L.sr = ixidt * sqrt(temp * (2 * xidt - 3 + 4 * L.c0 - L.c0 * L.c0));
        L.sv = sqrt(temp * (1 - L.c0 * L.c0));
        const double om = 1 - L.c0;
        L.crv = ixidt * temp * (om * om) / (L.sr * L.sv);
    } else {
        L.c0 = 1 - xidt + 0.5 * xidt2;
        L.c1 = (1 - 0.5 * xidt + 2 * MDT_TWELFTH * xidt2) * dt;
        L.c2 = (0.5 - 2 * MDT_TWELFTH * xidt + 0.5 * MDT_TWELFTH * xidt2) * dt;
        L.sr = dt * sqrt(temp * (8 * MDT_TWELFTH * xidt - 0.5 * xidt2));
        L.sv = sqrt(2 * temp * xidt * (1 - xidt));
        L.crv = 0.5 * sqrt(3.0) * (1 - 0.125 * xidt);
    }
    return L;
}

// the branch test of md_algo.f90:176 for one bead (1e-2 is a default-real literal)
__device__ __forceinline__ bool lan_big(double fric, double dt) { return fric * dt > (double)1e-2f; }

// ldfa, src/md_algo.f90:506-570: friction [1/fs] from the EMT density
__device__ __forceinline__ double ldfa(double dens, double mass, int *bad) {
#pragma clang fp contract(off)
    const double convert = 1.00794 * MDT_AMU2MASS;
    const double lo = (double)(-1e-12f), hi = (double)0.36f;
    double fric;
    if (lo <= dens && dens <= hi) {
        const double c[12] = {0.0802484, -1.12851, 9.28508, 2.10064, -843.419, 8.85354e3,
                              -4.89023e4, 1.6741e5, -3.67098e5, 5.03476e5, -3.9426e5, 1.34763e5};
        fric = 0.0;
        double temp = dens;
#pragma unroll
        for (int j = 0; j < 12; ++j) {
            fric = fric + c[j] * temp;
            temp = temp * dens;
        }
    } else if (dens > hi) {
        fric = 0.001 * (4.7131 - exp(-4.41305 * dens));
    } else {
        *bad = 1;
        fric = 0.0;
    }
    return fric * convert / MDT_HBAR / mass;
}

__device__ void load_types(LdsTypes &T, const EmtConst *__restrict__ ec, int lane, int nthr) {
    for (int k = lane; k < MDT_MAXT; k += nthr) {
        T.bs0[k] = ec->betas0[k];
        T.kdb[k] = ec->kappadbeta[k];
        T.betaeta2[k] = ec->betaeta2[k];
        T.e0[k] = ec->e0[k];
        T.lambda[k] = ec->lambda[k];
        T.v0[k] = ec->v0[k];
        T.kappa[k] = ec->kappa[k];
        T.n0[k] = ec->n0[k];
        T.densc[k] = ec->densc[k];
        T.etaT[k] = -ec->eta2[k] * MDT_EXP_K;
        T.kdbT[k] = -ec->kappadbeta[k] * MDT_EXP_K;
        T.owner[k] = ec->owner[k];
        T.f_eta2l2[k] = (float)(ec->eta2[k] * MDT_LOG2E);
        T.f_kdbl2[k] = (float)(ec->kappadbeta[k] * MDT_LOG2E);
        T.f_kdb[k] = (float)ec->kappadbeta[k];
    }
    for (int k = lane; k < MDT_MAXT * MDT_MAXT; k += nthr) {
        T.csig[k] = ec->csig[k];
        T.etad[k] = ec->etad[k];
        T.wv[k] = ec->wv[k];
        T.pair_on[k] = ec->pair_on[k];
        T.f_csig[k] = (float)ec->csig[k];
        T.f_etad[k] = (float)ec->etad[k];
        T.f_wv[k] = (float)ec->wv[k];
    }
}

__device__ void load_exptab(LdsTypes &T, int lane, int nthr) {
    const double et[MDT_EXP_TAB_N] = MDT_EXP_TAB_INIT;
    for (int k = lane; k < MDT_EXP_TAB_N; k += nthr) T.exptab[k] = et[k];
}

__device__ void load_tables(LdsTables &T, const EmtConst *__restrict__ ec, const PropConst *__restrict__ pc,
                            const CellRegs &cell, int lane, int nthr) {
    load_types(T, ec, lane, nthr);
    for (int k = lane; k < MDT_MAXT; k += nthr) {
        T.eta2[k] = ec->eta2[k];
        T.algo[k] = pc->algo[k];
        T.is_proj[k] = pc->is_proj[k];
    }
    for (int k = lane; k < MDT_MAXT * MDT_MAXT; k += nthr) T.csig48[k] = ec->csig[k] * 281474976710656.0;  // exact (power of two)
    for (int c = lane; c < 27; c += nthr) {
        const double m0 = (double)(c % 3 - 1), m1 = (double)((c / 3) % 3 - 1), m2 = (double)(c / 9 - 1);
        T.shift[3 * c + 0] = cell.h[0] * m0 + cell.h[3] * m1 + cell.h[6] * m2;
        T.shift[3 * c + 1] = cell.h[1] * m0 + cell.h[4] * m1 + cell.h[7] * m2;
        T.shift[3 * c + 2] = cell.h[2] * m0 + cell.h[5] * m1 + cell.h[8] * m2;
    }
    load_exptab(T, lane, nthr);
}

}  // namespace

// Fixed-point scales of the LDS accumulators that receive pair
// contributions from other lanes: integer addition is associative, so the
// totals do not depend on the order in which lanes add them.
#define MDT_W48 281474976710656.0            // 2^48
#define MDT_IW48 (1.0 / 281474976710656.0)
#define MDT_F_SCALE 4398046511104.0          // 2^42: force up to 2.1e6 eV/A, step 2.3e-13
#define MDT_F_ISCALE (1.0 / 4398046511104.0)

// Round-to-nearest-even of y to int64, returned with the rounded value as a
// double in *r.  For |y| < 2^51 adding 1.5 * 2^52 leaves rint(y) in the low
// mantissa bits (the sum lies in [2^52, 2^53), where the spacing is 1 and the
// default rounding is to nearest even), so the integer is the difference of
// two bit patterns: three instructions instead of the f64 -> i64 expansion.
// fix_round_small requires |y| < 2^51; its callers vote across the wave and
// take rint, the conversion and the overflow test (the callers' 9e18 bound)
// only when some lane's |y| is larger, so the common case issues neither.
#define MDT_RND_MAGIC 6755399441055744.0  // 1.5 * 2^52
__device__ __forceinline__ long long fix_round_small(double y, double *r) {
    const double t = y + MDT_RND_MAGIC;
    *r = t - MDT_RND_MAGIC;
    return __double_as_longlong(t) - __double_as_longlong(MDT_RND_MAGIC);
}

// sigma contributions span ~1e3 (close contact) down to ~1e-35 (pairs at the
// cut-off) and an isolated atom's sigma sits near the reference's 1e-30
// clamp, where G = dE/dsigma ~ 1/sigma: a sum with relative precision at
// any magnitude is needed.  Three int64 words at 2^-48, 2^-96 and 2^-144
// hold each contribution exactly down to 4.5e-44 (each conversion step is an
// exact power-of-two scaling and an exact subtraction of the rounded part).
__device__ __forceinline__ void sig_add_scaled(unsigned long long *hi, unsigned long long *mid,
                                               unsigned long long *lo, double y, int *bad) {
    // y: the contribution times 2^48 (callers fold the power of two into a
    // constant, an exact scaling).  The overflow test sits in the slow path
    // of the wave-uniform vote.
    double h, m, l;
    long long ih;
    if (__all(fabs(y) < 2251799813685248.0)) {  // 2^51
        ih = fix_round_small(y, &h);
    } else {
        if (!(fabs(y) < 9.0e18)) {
            *bad |= MDT_ST_FIXED_OVERFLOW;
            return;
        }
        h = rint(y);
        ih = (long long)h;
    }
    const double y1 = (y - h) * MDT_W48;  // |y1| <= 2^47
    const long long im = fix_round_small(y1, &m);
    const long long il = fix_round_small((y1 - m) * MDT_W48, &l);  // |.| <= 2^47
    atomicAdd(hi, (unsigned long long)ih);
    if (im != 0) atomicAdd(mid, (unsigned long long)im);
    if (il != 0) atomicAdd(lo, (unsigned long long)il);
}

__device__ __forceinline__ double sig_value(unsigned long long hi, unsigned long long mid, unsigned long long lo) {
    return (((double)(long long)lo * MDT_IW48 + (double)(long long)mid) * MDT_IW48 + (double)(long long)hi) *
           MDT_IW48;
}

// y: the contribution in fixed-point units (times the accumulator's scale)
__device__ __forceinline__ void fx_add_scaled(unsigned long long *acc, double y, int *bad) {
    double r;
    if (__all(fabs(y) < 2251799813685248.0)) {  // 2^51, wave-uniform branch
        atomicAdd(acc, (unsigned long long)fix_round_small(y, &r));
    } else if (fabs(y) < 9.0e18) {
        atomicAdd(acc, (unsigned long long)(long long)rint(y));
    } else {
        *bad |= MDT_ST_FIXED_OVERFLOW;
    }
}
__device__ __forceinline__ void fx_add(unsigned long long *acc, double x, double scale, int *bad) {
    fx_add_scaled(acc, x * scale, bad);
}

// s, embedded density, E_coh + vref and G = dE/dsigma of an atom of type tk
// with total sigma (src/pes_emt_mod.f90:793-869 and :871-972)
__device__ __forceinline__ void emt_atom(const LdsTypes &T, int tk, double sig, double *Gk, double *Ek, double *dn) {
    const double clamp30 = (double)1e-30f;  // pes_emt_mod.f90:793-794
    const double sc = sig > clamp30 ? sig : clamp30;
    const double sl = sc > MDT_TOLERANCE ? sc : MDT_TOLERANCE;
    const double sv = -log(sl * MDT_TWELFTH) / T.betaeta2[tk];
    *dn = T.n0[tk] * exp(T.densc[tk] * sv);
    const double el = exp(-T.lambda[tk] * sv);
    const double ek = exp(-T.kappa[tk] * sv);
    *Ek = T.e0[tk] * ((1 + T.lambda[tk] * sv) * el - 1) + 6 * T.v0[tk] * ek;
    const double D = T.e0[tk] * T.lambda[tk] * T.lambda[tk] * (sv * el) + 6 * T.v0[tk] * T.kappa[tk] * ek;
    *Gk = -D / (T.betaeta2[tk] * sc);
}

// Image along one axis of a pair whose folded fractional difference x lies
// within 1e-4 of +-1/2 -- in a cell of even width, atoms of perfect lattice
// layers sit exactly half a cell apart.  The reference's minimum image
// (src/universe_mod.f90:411-428) rounds s = isimbox (r_j - r_i) of the
// unfolded positions half away from zero (anint), so the tie goes to the
// image that expression, evaluated in its order without fused
// multiply-adds, picks; returns m with x - m equal to its reduced
// coordinate (s - anint(s) is odd in r_j - r_i, so the pair's order does
// not matter).  (ia, ib, ic) = isimbox(axis, 1..3); ra, rb the x, y, z of
// the two atoms.
__device__ __forceinline__ double tie_dot(double ia, double ib, double ic, double d0, double d1, double d2) {
#pragma clang fp contract(off)
    return ia * d0 + ib * d1 + ic * d2;
}
__device__ __forceinline__ double tie_image(double ia, double ib, double ic, double ra0, double ra1, double ra2, double rb0,
                                         double rb1, double rb2, double x) {
#pragma clang fp contract(off)
    const double s = tie_dot(ia, ib, ic, ra0 - rb0, ra1 - rb1, ra2 - rb2);
    return rint(x - (s - round(s)));
}

// One atom of a replica in LDS: position, G = dE/dsigma~ (pass B) and the first
// accumulator word.  40 bytes, so that random atoms spread over all banks (32
// would put every x on an eighth of them).
struct PairRec {
    double x, y, z, g;
    unsigned long long w;
};

// Sums that do not depend on the order of their terms.  A term v is rounded to a
// multiple of a power of two, the grid: t = v + C with C = 1.5 * 2^52 grids
// leaves v / grid in t's mantissa, so t's bits less C's are the integer that a
// 64-bit LDS atomic adds (C's low word is 0: one subtraction), and t - C is the
// rounded term, whose sums in registers are exact in FP64 (multiples of the grid
// below 2^53 of them).  Results are bitwise reproducible whatever order the
// atomics land in, however a row of neighbours is cut into lanes and whichever
// of its two atoms owns a pair.  (FP64 LDS atomics would save the subtraction, but
// on random addresses they take 21 cycles a wavefront, 64-bit integer ones 11.)
//   sigma: 2^-42 (|v| < 512) and 2^-88 for the rest;
//   forces: 2^-43 eV/A (|v| < 256 eV/A).  The words hold up to 1.05e6 eV/A, 700 times
//   the largest pair force of the shipped parameter sets; 2^-42 would hold twice as
//   much and double the error of a run's state (4096 x 145 atoms, 200 steps, against
//   64 bits: 2.8e-13 with 2^-43, 5.5e-13 with 2^-42).
// Larger terms are converted by rint and added by themselves; those beyond 2^63
// grids, and NaN, are flagged (MDT_ST_FIXED_OVERFLOW) and left out.
// A lane sums the terms of its piece of a row, whose order is the list's, as rounded
// FP64 terms: exact while the lane's sum stays below 2^53 grids, 1024 eV/A or
// sigma 2048; beyond that it is rounded, the same in every run but not however the
// row is cut.  Atoms whose partners come in no fixed order (flat lists) sum integers.
// Energies are summed in registers: 2^-33 eV (sums below 1e6 eV) and 2^-70 for
// the rest.
#define MDT_SIG_C1 1536.0                         // 1.5 * 2^(52 - 42)
#define MDT_SIG_C2 2.1827872842550278e-11         // 1.5 * 2^(52 - 88)
#define MDT_SIG_FAST 511.0
#define MDT_FRC_C 768.0                           // 1.5 * 2^(52 - 43)
#define MDT_FRC_FAST 255.0
#define MDT_EPR_C1 786432.0                       // 1.5 * 2^(52 - 33)
#define MDT_EPR_C2 5.7220458984375e-06            // 1.5 * 2^(52 - 70)
#define MDT_P42 4398046511104.0
#define MDT_P43 8796093022208.0
#define MDT_P46 70368744177664.0

// Below this sigma~ (of the near pairs) the words' absolute step shows in a
// relative sense, and the atom's force scales with sigma~ itself down to the
// reference's 1e-30 clamp: its sigma~ is summed again over all partners as plain
// FP64 terms, in an order that depends on the atoms alone.
#define MDT_SIG_VTINY 2.3283064365386963e-10  // 2^-32

#define MDT_ANY_IMAGE 31   // image code of a kept pair that may round either way
#define MDT_FLAT_CAP 128   // listed near partners of one such atom (with more it tests every atom in both passes)

// the integer of t = v + C (C's low word is 0)
__device__ __forceinline__ unsigned long long grid_int(double t, double C) {
    union {
        double d;
        struct {
            uint32_t lo, hi;
        } w;
        unsigned long long u;
    } a, c;
    a.d = t;
    c.d = C;
    a.w.hi -= c.w.hi;
    return a.u;
}
// v as an integer of grids (scale: grids per unit) and rounded, any size
__device__ __forceinline__ unsigned long long grid_any(double v, double scale, double *r, int *bad) {
    double y = rint(v * scale);
    if (!(fabs(y) < 9.0e18)) {
        *bad |= MDT_ST_FIXED_OVERFLOW;
        y = 0.0;
    }
    *r = y / scale;
    return (unsigned long long)(long long)y;
}
// the two words of a sigma term below MDT_SIG_FAST; *h, *l: the rounded parts
__device__ __forceinline__ void sig_words(double v, unsigned long long *u1, unsigned long long *u2, double *h, double *l) {
    const double t = v + MDT_SIG_C1;
    *u1 = grid_int(t, MDT_SIG_C1);
    *h = t - MDT_SIG_C1;
    const double t2 = (v - *h) + MDT_SIG_C2;
    *u2 = grid_int(t2, MDT_SIG_C2);
    *l = t2 - MDT_SIG_C2;
}
// a sigma term from MDT_SIG_FAST on: its first word (step 2e-13) is enough;
// adds it to *p and returns it rounded
__device__ double sig_large(unsigned long long *p, double v, int *bad) {
    double h;
    const unsigned long long u = grid_any(v, MDT_P42, &h, bad);
    atomicAdd(p, u);
    return h;
}
__device__ __forceinline__ double sig_sum(unsigned long long w1, unsigned long long w2) {
    return (double)(long long)w1 * (1.0 / MDT_P42) + (double)(long long)w2 * (1.0 / (MDT_P42 * MDT_P46));
}
__device__ __forceinline__ double frc_sum(unsigned long long w) { return (double)(long long)w * (1.0 / MDT_P43); }
// LDS += a sum of rounded terms (a multiple of the grid, C as in grid_int)
__device__ __forceinline__ void add_sum(unsigned long long *p, double v, double C, double scale, int *bad) {
    unsigned long long u;
    double r;
    if (__builtin_expect(fabs(v) < C * (1.0 / 3.0), 1))  // 2^51 grids
        u = grid_int(v + C, C);
    else
        u = grid_any(v, scale, &r, bad);
    atomicAdd(p, u);
}

// Minimum image of the pair (k, n) of a replica staged in LDS (positions p,
// fractional components in [-0.2, 1.2)): d = p_k - p_n - shift[code] (4 doubles a code), code
// the rounding m of the fractional difference (in {-1, 0, 1}^3, the list
// scan's image code).  The rounding is decided in FP32 from ihf (H^-1, 9
// floats, column major; error ~1e-7 against the 1e-4 tie window); a component
// within 1e-4 of +-1/2 takes the reference's image from the FP64 H^-1 ihg and
// the unfolded positions -- xr (SoA, N per component) in global memory, or, xr NULL,
// the staged ones: no atom was folded -- as tie_image does.  Returns |d|^2.
__device__ __forceinline__ double pair_image(const float *ihf, const double *ihg, const double *shift, const PairRec &pk,
                                             const PairRec &pn, const double *xr, int N, int k, int n, double d[3],
                                             int *codep) {
    const double cx = pk.x - pn.x, cy = pk.y - pn.y, cz = pk.z - pn.z;
    const float ex = (float)cx, ey = (float)cy, ez = (float)cz;
    const float f0 = ihf[0] * ex + ihf[3] * ey + ihf[6] * ez;
    const float f1 = ihf[1] * ex + ihf[4] * ey + ihf[7] * ez;
    const float f2 = ihf[2] * ex + ihf[5] * ey + ihf[8] * ez;
    float m0 = rintf(f0), m1 = rintf(f1), m2 = rintf(f2);
    const bool t0 = fabsf(f0 - m0) > 0.4999f, t1 = fabsf(f1 - m1) > 0.4999f, t2 = fabsf(f2 - m2) > 0.4999f;
    if (t0 | t1 | t2) {  // rare: the exact fractional difference and the reference's tie rule
        if (xr) {
            const double a0 = xr[k], a1 = xr[N + k], a2 = xr[2 * N + k];
            const double b0 = xr[n], b1 = xr[N + n], b2 = xr[2 * N + n];
            if (t0) m0 = (float)tie_image(ihg[0], ihg[3], ihg[6], a0, a1, a2, b0, b1, b2, ihg[0] * cx + ihg[3] * cy + ihg[6] * cz);
            if (t1) m1 = (float)tie_image(ihg[1], ihg[4], ihg[7], a0, a1, a2, b0, b1, b2, ihg[1] * cx + ihg[4] * cy + ihg[7] * cz);
            if (t2) m2 = (float)tie_image(ihg[2], ihg[5], ihg[8], a0, a1, a2, b0, b1, b2, ihg[2] * cx + ihg[5] * cy + ihg[8] * cz);
        } else {  // tie_image's x is its s
            if (t0) m0 = (float)round(tie_dot(ihg[0], ihg[3], ihg[6], cx, cy, cz));
            if (t1) m1 = (float)round(tie_dot(ihg[1], ihg[4], ihg[7], cx, cy, cz));
            if (t2) m2 = (float)round(tie_dot(ihg[2], ihg[5], ihg[8], cx, cy, cz));
        }
    }
    const int code = ((int)m0 + 1) + 3 * ((int)m1 + 1) + 9 * ((int)m2 + 1);
    d[0] = cx - shift[4 * code];
    d[1] = cy - shift[4 * code + 1];
    d[2] = cz - shift[4 * code + 2];
    *codep = code;
    return fma(d[2], d[2], fma(d[1], d[1], d[0] * d[0]));
}

// Hides v's derivation from the optimiser (an empty asm with a register
// operand; no instruction is emitted): in a loop that usually runs once,
// addresses derived from v are then formed per iteration instead of being
// strength-reduced into one induction register per array.
__device__ __forceinline__ void opaque(int &v) { asm volatile("" : "+v"(v)); }

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// LDS += the wavefront's integers (p the same in every lane: left to itself the
// compiler adds such lanes up one by one)
__device__ __forceinline__ void add_uniform(unsigned long long *p, unsigned long long v) {
    if (__ballot(v != 0) == 0) return;  // the wavefront has none
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(p, v);
}

// a b rounded, whatever it is added to: a pair's distance and terms have the same
// bits in rows, flat lists and direct sums
template <class F>
__device__ __forceinline__ F mul_rn(F a, F b) {
#pragma clang fp contract(off)
    return a * b;
}

// Pair ownership: each unordered pair is evaluated once, by its owner; the
// owner alternates with index parity, which gives every atom about half of
// its neighbours.
__device__ __forceinline__ bool owns(int k, int n) { return (k < n) != (((k + n) & 1) != 0); }

// calc_force for one replica per workgroup.
//
// What bounds it: with enough replicas the issue of vector instructions (about 60 %
// of the cycles; about 165 a pair and lane in both passes together) beside the LDS (51 %:
// positions, exponential table, atomics), with few of them the latency of its
// phases.  H/Au 6x6x4, 4096 replicas of 3 k near pairs: 166 us a step with the
// propagator, 263 before rows were sorted pieces; H/Pt 8x8x6, 2048 replicas: 281 us
// a launch (mean, builds included), 494 before.
//  * Rows.  The owned half lists hold the near pairs (r <= rnear) of the
//    atoms of one EMT type, the majority (bv.bulk); their constants are
//    uniform, so a pair needs no type.  A row is cut into equal pieces, one a
//    lane, sorted by length, so that a wavefront's lanes end together; the
//    pieces' sums meet in the order-free words.  The entries lie in HBM in the
//    order the wavefronts read them, two a word, one word a lane and iteration
//    (coalesced, and no LDS: a replica of 145 atoms takes 14 KB of it instead of 33).
//  * Flat lists.  The few atoms of the other EMT type (at most
//    MDT_FLAT_MAX: the projectile) get the list of their near partners at
//    every launch, by a minimum-image test of every atom, one partner per lane
//    in the passes.  They are the fast atoms, so the rows are kept while the
//    slower ones move.  Universes with more of them (MIXED) hold every pair in
//    rows and look the types up.
//  * Kept rows.  They serve until an atom that is in them has moved half the
//    skin.  Positions stay unfolded (fractional components in [-0.2, 1.2);
//    others are folded by the fold of the build), so an entry's image code stays
//    what it was at the build: a launch only reads them.
//  * Rows for one launch (lists not kept, or fresh positions at every call).  Few
//    workgroups read them in LDS as scanned, tpa lanes per atom, with every type in
//    them (MIXED): no cut, no sort, and no flat lists, whose three phases of
//    their own cost 3 k cycles each to a workgroup that waits for latency
//    (100 replicas of 37 atoms, 150 steps: 3.45 ms, 3.68 with kept rows).  Many
//    workgroups cut them as ever: rows in LDS would leave 3 of 5 workgroups a CU
//    (4096 replicas of 145 atoms: 0.41 ms a call, 0.36 cut).
//  * The scan tests two candidates of an atom at a time and looks for images that
//    round either way only along axes where such a pair can be near (new
//    positions of 4096 x 145 atoms: 0.39 -> 0.36 ms a call).
//  * A pair's terms have the same bits in rows of one type, rows of all types, flat
//    lists and direct sums: products that an addition could fuse are written
//    out (mul_rn, fma).
//  * The pair terms of two entries are evaluated without a branch between them, so
//    that one's chain of dependent instructions fills the other's gaps.
// PREC (arithmetic of the pair terms):
//   0: FP64 throughout;
//   1: the cut-off function, the sigma and pair-potential exponentials and
//      their products in FP32;
//   2: only the cut-off exponential exp(acut (r - rcut)) and theta in FP32,
//      the sigma and pair-potential exponentials in FP64 (for metals whose
//      embedding stiffness makes FP32 sigma / V terms miss 1e-6 eV/atom and
//      1e-5 eV/A, e.g. Pt with V0 = 21.7 eV).
// In every mode the geometry (differences, r, the exponent arguments
// r - rcut and r - beta s0, which carry factors up to acut ~ 26/A), the
// per-atom embedding terms, G and every accumulation stay FP64.
// JUDGE: FP64 EMT forces of the selected replicas compared with
// bv.judge_f (the network's judge); nothing else is written.
// MAXB: the largest workgroup of the instantiation, 512, or 1024 for size
// classes of more than 512 atoms x threads per atom, whose few replicas
// would otherwise leave each CU two waves per SIMD.
template <bool MIXED, int PREC, bool JUDGE, int MAXB>
__global__ void __launch_bounds__(MAXB, 4)
    k_replica(const EmtConst *__restrict__ ecg, BatchView bv, int add_fin) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ LdsTypes T;
    __shared__ double s_sh[27 * 4];  // lattice translations of the image codes, 32 bytes each
    __shared__ double s_cell[18];    // H, H^-1
    __shared__ float s_ihf[9];       // H^-1 in FP32
    __shared__ double s_ep[2];       // energy words: pair energies - 2 (atoms' energies)
    __shared__ int s_flat[MDT_FLAT_MAX], s_fcnt[MDT_FLAT_MAX];
    __shared__ uint16_t s_flist[MIXED ? 1 : MDT_FLAT_MAX * MDT_FLAT_CAP];
    __shared__ int s_np[64], s_hist[64];  // pieces at each length limit, of each length
    __shared__ int s_cb[64];              // stream offset of each chunk of 64 pieces
    __shared__ int s_nflat, s_R, s_slow, s_anyfold, s_folded;
    const int rep = bv.rep_list ? bv.rep_list[blockIdx.x] : bv.rep0 + (int)blockIdx.x;
    if (bv.only && !bv.only[rep]) return;                          // whole block: uniform
    if (bv.skip && bv.skip[rep]) return;                           // whole block: uniform
    if (JUDGE && (rep % bv.judge_mod) != bv.judge_phase) return;   // whole block: uniform
    const int t = bv.rep_traj[rep];
    if (bv.done && bv.done[t]) return;  // frozen trajectory (whole block: uniform)
    const int b = bv.rep_bead[rep];
    const int N = bv.traj_N[t];
    const int cap = bv.nbcap < N - 1 ? bv.nbcap : (N > 1 ? N - 1 : 1);  // entries per row
    const int capg = (bv.nbcap + 7) & ~7;                               // stride of the rows in HBM
    const long long soff = bv.traj_soff[t];
    const long long roff = soff + (long long)b * 3 * N;  // x block of this replica
    const long long doff = soff / 3 + (long long)b * N;   // dens / fixed block
    const long long aoff = bv.traj_aoff[t];
    const double *xr = bv.x + roff;
    const int nthr = blockDim.x;
    const int lane = threadIdx.x, wl = lane & 63, wave = lane >> 6, nwaves = nthr >> 6;
    const int bulk = bv.bulk;
    load_types(T, ecg, lane, nthr);
    load_exptab(T, lane, nthr);
    if (lane < 18) s_cell[lane] = lane < 9 ? bv.cell[9 * t + lane] : bv.icell[9 * t + lane - 9];
    if (lane < 27) {
        const double m0 = (double)(lane % 3 - 1), m1 = (double)((lane / 3) % 3 - 1), m2 = (double)(lane / 9 - 1);
        const double *h = bv.cell + 9 * t;
#pragma unroll
        for (int q = 0; q < 3; ++q) s_sh[4 * lane + q] = h[q] * m0 + h[q + 3] * m1 + h[q + 6] * m2;
    }
    const double *s_h = s_cell, *s_ih = s_cell + 9;

    // LDS: words W2, W3 | records | typ | tiny.  sigma takes two words (record
    // and W2), forces all three.  W2 and W3 hold the scan's FP32 coordinates.
    unsigned long long *w2 = (unsigned long long *)smem_raw, *w3 = w2 + N;
    PairRec *rec = (PairRec *)(w3 + N);
    uint8_t *typ = (uint8_t *)(rec + N);
    uint8_t *tiny = typ + N;
    // HBM, per block slot: the stream of pieces, the piece table (atom | length
    // << 11), the chunks' offsets in the stream; rows as scanned (those of batches
    // too small to fill the GPU in LDS: mdt_replica_lists)
    uint32_t *stream = bv.rl_lists + (long long)blockIdx.x * bv.rl_stride;
    uint32_t *rows = stream + bv.rl_rows, *chunk = stream + bv.rl_chunk;
    // (never one pointer to either: that makes every access a flat one)
    const bool lds_scan = bv.rl_scan < 0;
    uint16_t *lrow = (uint16_t *)(smem_raw + ((58 * N + 7) & ~7)), *grow = (uint16_t *)(stream + bv.rl_scan);
    int bad_local = 0;

    // Verlet skin: the rows of this block slot are built with rnear + skin and
    // kept while no atom in them moved more than skin / 2 since.  A pair's
    // rounded image is then the build's, unless a fractional component of
    // the difference lay within skin / width of +-1/2 at the build: such a pair is
    // listed if any image it can round to lies within rnear + skin, with
    // the code MDT_ANY_IMAGE, and takes its image at every launch from the
    // current positions.  (The pairs beyond rnear never come from a row.)
    const double skin = bv.rl_skin, rnear = ecg->rnear, cutr = ecg->cutr;
    int2 *valid = bv.rl_valid ? bv.rl_valid + blockIdx.x : nullptr;
    // x: 0, or 1 | fold << 1 | slow << 2 | row pieces << 3; y: the EMT constants' generation
    const int kept = valid && valid->y == ecg->gen ? valid->x : 0;
    bool keep = valid != nullptr;
    if (keep && !kept) {
        const double *ih = bv.icell + 9 * t;
        const double b0 = sqrt(ih[0] * ih[0] + ih[3] * ih[3] + ih[6] * ih[6]) * skin;
        const double b1 = sqrt(ih[1] * ih[1] + ih[4] * ih[4] + ih[7] * ih[7]) * skin;
        const double b2 = sqrt(ih[2] * ih[2] + ih[5] * ih[5] + ih[8] * ih[8]) * skin;
        keep = b0 < 0.05 && b1 < 0.05 && b2 < 0.05;
    }
    double *ref = keep ? bv.rl_ref + (long long)blockIdx.x * 3 * bv.rl_ns : nullptr;

    // ---- phase 0: stage ----
    if (lane < 9) s_ihf[lane] = (float)bv.icell[9 * t + lane];
    if (lane < 64) {
        s_np[lane] = s_hist[lane] = 0;
        s_cb[lane] = kept && lane < ((kept >> 3) + 63) / 64 ? chunk[lane] : 0;
    }
    if (lane == 0) {
        s_nflat = 0;
        s_anyfold = s_folded = 0;
        s_slow = kept >> 2 & 1;
        s_R = kept >> 3;
        s_ep[0] = s_ep[1] = 0.0;
    }
    // loads that the passes and the output wait for otherwise: the lane's first
    // piece, its atom's mass and fixed bits
    uint32_t info0 = 0, word0 = 0;
    int off0 = 0;
    if (kept && lane < kept >> 3) {
        info0 = rows[lane];
        off0 = chunk[wave];
    }
    double mass0 = 1.0;
    int fixed0 = 0;
    if (!JUDGE && lane < N) {
        mass0 = bv.mass[aoff + lane];
        fixed0 = bv.fixed[doff + lane];
    }
    __syncthreads();  // s_nflat
    // An atom whose fractional position leaves [-0.2, 1.2) is folded into the
    // cell; an atom in kept rows as at their build (there, for a fold of zero,
    // nothing is looked at: kept & 2 tells whether any was not).
    auto fold = [&](double &x, double &y, double &z, double rx, double ry, double rz, float4 *f) {
        const double f0 = s_ih[0] * rx + s_ih[3] * ry + s_ih[6] * rz;
        const double f1 = s_ih[1] * rx + s_ih[4] * ry + s_ih[7] * rz;
        const double f2 = s_ih[2] * rx + s_ih[5] * ry + s_ih[8] * rz;
        const double g0 = (f0 >= -0.2 && f0 < 1.2) ? 0.0 : floor(f0);
        const double g1 = (f1 >= -0.2 && f1 < 1.2) ? 0.0 : floor(f1);
        const double g2 = (f2 >= -0.2 && f2 < 1.2) ? 0.0 : floor(f2);
        if (f) *f = make_float4((float)(f0 - g0), (float)(f1 - g1), (float)(f2 - g2), 0.f);
        if (g0 == 0.0 && g1 == 0.0 && g2 == 0.0) return false;
        s_folded = 1;  // benign race: every writer stores 1
        x -= s_h[0] * g0 + s_h[3] * g1 + s_h[6] * g2;
        y -= s_h[1] * g0 + s_h[4] * g1 + s_h[7] * g2;
        z -= s_h[2] * g0 + s_h[5] * g1 + s_h[8] * g2;
        return true;
    };
    // staged for a scan: folded position, fractional one and type
    float4 *f4 = (float4 *)w2;
    auto stage = [&](int i, int ty, double x, double y, double z) {
        if (keep) {
            ref[i] = x;
            ref[bv.rl_ns + i] = y;
            ref[2 * bv.rl_ns + i] = z;
        }
        float4 f;
        if (fold(x, y, z, x, y, z, &f) && (MIXED || ty == bulk)) s_anyfold = 1;  // benign race: every writer stores 1
        f.w = __int_as_float(ty);
        rec[i].x = x;
        rec[i].y = y;
        rec[i].z = z;
        f4[i] = f;
    };
    int moved = 0;
    for (int i = lane; i < N; i += nthr) {
        const int ty = bv.type[aoff + i];
        typ[i] = (uint8_t)ty;
        double x = xr[i], y = xr[N + i], z = xr[2 * N + i];
        const bool rowed = MIXED || ty == bulk;
        if (!rowed && T.owner[ty]) {
            const int q = atomicAdd(&s_nflat, 1);  // the order is free
            if (q < MDT_FLAT_MAX) {
                s_flat[q] = i;
                s_fcnt[q] = 0;
            }
        }
        rec[i].g = 0.0;
        if (!kept) {
            stage(i, ty, x, y, z);
            continue;
        }
        if (rowed) {
            const double rx = ref[i], ry = ref[bv.rl_ns + i], rz = ref[2 * bv.rl_ns + i];
            const double d0 = x - rx, d1 = y - ry, d2 = z - rz;
            if (!(d0 * d0 + d1 * d1 + d2 * d2 <= 0.25 * skin * skin)) moved = 1;
            if (kept & 2) fold(x, y, z, rx, ry, rz, nullptr);
        } else {
            fold(x, y, z, x, y, z, nullptr);
        }
        rec[i].x = x;
        rec[i].y = y;
        rec[i].z = z;
        rec[i].w = w2[i] = w3[i] = 0;
    }
    if (kept && lane < kept >> 3) word0 = stream[off0 + wl];
    const bool reuse = !__syncthreads_or(moved) && kept;
    const unsigned long long below = (wl == 0) ? 0ull : ((~0ull) >> (64 - wl));

    // ---- phase 1: rows ----
    // few workgroups and rows for this launch only: they are read where the scan
    // put them, in LDS, tpa lanes per row (cutting and sorting them costs 6 us)
    // (launches that want this hold all types in their rows: the row loop of one type has no test for it)
    const bool direct = MIXED && !keep && lds_scan;
    const int sh = bv.tpa_shift;
    if (!reuse) {
        if (kept) {  // the rows are stale
            if (lane == 0) s_slow = 0;
            for (int i = lane; i < N; i += nthr) stage(i, typ[i], xr[i], xr[N + i], xr[2 * N + i]);
            __syncthreads();
        }
        const double *xt = s_folded ? xr : nullptr;  // the unfolded positions are the staged ones
        // The scan only decides membership: FP32 fractional differences, r^2
        // from the cell metric H^T H with the bound widened by 1e-4; the
        // passes test r <= rnear in FP64.  A fractional difference within
        // 1e-4 of +-1/2 takes its image from the reference's expression (in rows
        // that are kept: MDT_ANY_IMAGE).
        // tpa lanes per atom; only the owned candidates are visited, in
        // increasing index: below k those of the other parity (a = (k + 1) / 2
        // of them), above k those of the same parity.
        // row lengths go to the record's word
        float g00, g11, g22, g01, g02, g12;  // H^T H, cell vectors = columns of H
        {
            const double *h = s_h;
            g00 = (float)(h[0] * h[0] + h[1] * h[1] + h[2] * h[2]);
            g11 = (float)(h[3] * h[3] + h[4] * h[4] + h[5] * h[5]);
            g22 = (float)(h[6] * h[6] + h[7] * h[7] + h[8] * h[8]);
            g01 = (float)(2 * (h[0] * h[3] + h[1] * h[4] + h[2] * h[5]));
            g02 = (float)(2 * (h[0] * h[6] + h[1] * h[7] + h[2] * h[8]));
            g12 = (float)(2 * (h[3] * h[6] + h[4] * h[7] + h[5] * h[8]));
        }
        const double rn = keep ? rnear + skin : rnear;
        // components beyond these can round either way (2: none can, the cell is so wide
        // along the axis that such a pair is beyond rn in any image)
        auto margin = [&](int a) {
            const float *ih = s_ihf + a;
            const float inv = sqrtf(ih[0] * ih[0] + ih[3] * ih[3] + ih[6] * ih[6]);  // 1 / width
            const float mg = 0.4999f - (keep ? (float)skin * inv : 0.f);
            return mg > 1.001f * (float)rn * inv ? 2.f : mg;
        };
        const float mg0 = margin(0), mg1 = margin(1), mg2 = margin(2);
        // (of the pairs of types; one lane each)
        const int nt = ecg->ntypes;
        const bool all_on = MIXED ? __all(wl >= nt * nt || T.pair_on[wl / nt * MDT_MAXT + wl % nt])
                                  : T.pair_on[bulk * MDT_MAXT + bulk] != 0;
        const float cut2f = (float)(rn * rn * (1.0 + 1e-4));
        const int tpa = 1 << sh, apb = nthr >> sh;
        const unsigned long long gmask = ((1ull << tpa) - 1ull) << ((wl >> sh) << sh);
        const int mmax = N / 2 + 1;
        const int sub = lane & (tpa - 1);
        for (int k0 = 0; k0 < N; k0 += apb) {
            const int k = k0 + (lane >> sh);
            const int tk = k < N ? typ[k] : 0;
            const bool act = k < N && (MIXED || (tk == bulk && all_on));
            const float4 pk = act ? f4[k] : make_float4(0.f, 0.f, 0.f, 0.f);
            const int a_lo = (k + 1) >> 1;
            int c = 0;
            // candidate n of this lane's atom: listed (and the entry's code)?
            auto test = [&](int n, const float4 &pn, bool ok, int &code) {
                const int tn = __float_as_int(pn.w);
                ok = ok && (MIXED ? (all_on || T.pair_on[tk * MDT_MAXT + tn]) : tn == bulk);
                const float e0 = pk.x - pn.x, e1 = pk.y - pn.y, e2 = pk.z - pn.z;
                float m0f = rintf(e0), m1f = rintf(e1), m2f = rintf(e2);
                float d0 = e0 - m0f, d1 = e1 - m1f, d2 = e2 - m2f;
                const bool t0 = fabsf(d0) > mg0, t1 = fabsf(d1) > mg1, t2 = fabsf(d2) > mg2;
                const bool tie = ok && (t0 | t1 | t2);
                if (tie && !keep) {
                    const PairRec ck = rec[k], cn = rec[n];
                    const double cx = ck.x - cn.x, cy = ck.y - cn.y, cz = ck.z - cn.z;
                    const double *ih = s_ih;
                    if (xt) {
                        const double a0 = xt[k], a1 = xt[N + k], a2 = xt[2 * N + k];
                        const double b0 = xt[n], b1 = xt[N + n], b2 = xt[2 * N + n];
                        if (t0) m0f = (float)tie_image(ih[0], ih[3], ih[6], a0, a1, a2, b0, b1, b2, ih[0] * cx + ih[3] * cy + ih[6] * cz);
                        if (t1) m1f = (float)tie_image(ih[1], ih[4], ih[7], a0, a1, a2, b0, b1, b2, ih[1] * cx + ih[4] * cy + ih[7] * cz);
                        if (t2) m2f = (float)tie_image(ih[2], ih[5], ih[8], a0, a1, a2, b0, b1, b2, ih[2] * cx + ih[5] * cy + ih[8] * cz);
                    } else {
                        if (t0) m0f = (float)round(tie_dot(ih[0], ih[3], ih[6], cx, cy, cz));
                        if (t1) m1f = (float)round(tie_dot(ih[1], ih[4], ih[7], cx, cy, cz));
                        if (t2) m2f = (float)round(tie_dot(ih[2], ih[5], ih[8], cx, cy, cz));
                    }
                    d0 = e0 - m0f;
                    d1 = e1 - m1f;
                    d2 = e2 - m2f;
                }
                auto metric = [&](float d0, float d1, float d2) {
                    return d0 * (g00 * d0 + g01 * d1 + g02 * d2) + d1 * (g11 * d1 + g12 * d2) + g22 * d2 * d2;
                };
                float r2 = metric(d0, d1, d2);
                code = (int)(m0f + 3.f * m1f + (9.f * m2f + 13.f));
                if (tie && keep) {
                    code = MDT_ANY_IMAGE;
                    for (int q = 1; q < 8; ++q)
                        r2 = fminf(r2, metric(d0 - (t0 && (q & 1) ? copysignf(1.f, d0) : 0.f),
                                              d1 - (t1 && (q & 2) ? copysignf(1.f, d1) : 0.f),
                                              d2 - (t2 && (q & 4) ? copysignf(1.f, d2) : 0.f)));
                }
                return ok && r2 <= cut2f;
            };
            auto put = [&](int n, bool in, int code, int pos) {
                if (in) {
                    const uint16_t ent = (uint16_t)(n | (code << MDT_NBR_IDX_BITS));
                    const uint32_t at = (uint32_t)(k * capg + pos);
                    if (pos >= cap) {
                        bad_local |= MDT_ST_NBR_OVERFLOW;
                    } else {
                        if (lds_scan)
                            lrow[at] = ent;
                        else
                            grow[at] = ent;
                        if (code == MDT_ANY_IMAGE) s_slow = 1;  // benign race: every writer stores 1
                    }
                }
            };
            // two candidates at a time, so that one's reads and chain fill the other's gaps
            const int below_k = (k + 1) & 1, above_k = k + 2 - 2 * a_lo;
            auto scan = [&](auto one) {
                for (int m0 = sub; m0 - sub < mmax; m0 += 2 * tpa) {
                    const int m1 = m0 + tpa;
                    const int na = 2 * m0 + (m0 < a_lo ? below_k : above_k), nb = 2 * m1 + (m1 < a_lo ? below_k : above_k);
                    const float4 pa = f4[na < N ? na : N - 1], pb = f4[nb < N ? nb : N - 1];
                    int codea, codeb;
                    const bool ina = test(na, pa, act && na < N, codea), inb = test(nb, pb, act && nb < N, codeb);
                    one(na, ina, codea);
                    one(nb, inb, codeb);
                }
            };
            if (sh == 0)
                scan([&](int n, bool in, int code) {
                    put(n, in, code, c);
                    c += in ? 1 : 0;
                });
            else  // the atom's lanes in order
                scan([&](int n, bool in, int code) {
                    const unsigned long long m = __ballot(in) & gmask;
                    put(n, in, code, c + __popcll(m & below));
                    c += __popcll(m);
                });
            c = c < cap ? c : cap;
            if (direct) {
                const uint32_t info = k < N ? (uint32_t)(k | ((c - sub + tpa - 1) >> sh) << MDT_NBR_IDX_BITS) : 0u;
                if (k < N) rows[(k << sh) + sub] = info;
                if (k0 == 0) info0 = info;
            } else if (k < N && sub == 0) {
                rec[k].w = c;
            }
        }
        __syncthreads();
        if (direct) {
            if (lane == 0) s_R = N << sh;
        } else {
        // Row table: rows in equal pieces of at most L, the shortest L that gives
        // at most `lim` pieces -- one per lane, or two where that leaves less
        // than a quarter of the lanes to split with --, in order of length, so that
        // a wavefront's lanes have the same (145 atoms on 192 lanes: 57 wavefront
        // iterations for 49 full ones' worth of pairs, 72 unsorted).
        {
            const int magic = 65536 / (wl + 2) + 1;  // x / (wl + 2) for x < 256
            int np = 0;
            for (int k = wave; k < N; k += nwaves) {
                const int c = (int)rec[k].w;
                np += c > 190 ? 0x10000 : ((c + wl + 1) * magic) >> 16;
            }
            atomicAdd(&s_np[wl], np);
        }
        __syncthreads();
        // (few workgroups: the last wavefront is left to the flat lists)
        const int lim0 = (N + nthr / 4 + nthr - 1) / nthr * nthr - (lds_scan && nwaves > 3 ? 64 : 0);
        const int lim = lim0 < N + nthr ? lim0 : N + nthr;
        const unsigned long long fit = __ballot(s_np[wl] <= lim);
        const int L = fit ? __builtin_ctzll(fit) + 2 : 4096;  // none fits: one piece per row
        // pieces of atom k: m of length l + 1 after ns - m of length l
        auto cut = [&](int k, int &ns, int &l, int &m) {
            const int c = (int)rec[k].w;
            ns = (c + L - 1) / L;
            l = ns ? c / ns : 0;
            m = c - l * ns;
        };
        for (int k = lane; k < N; k += nthr) {
            int ns, l, m;
            cut(k, ns, l, m);
            if (m) atomicAdd(&s_hist[l + 1 < 63 ? l + 1 : 63], m);
            if (ns > m) atomicAdd(&s_hist[l < 63 ? l : 63], ns - m);
        }
        __syncthreads();
        int off = s_hist[wl];  // pieces of this length or longer
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_down(off, o, 64);
            if (wl + o < 64) off += y;
        }
        if (lane == 0) s_R = off;
        const int np = s_hist[wl];
        off -= np;
        __syncthreads();
        if (wave == 0) {
            s_hist[wl] = off;
            // chunks that start among the pieces of this length: their stream words
            const int len = wl < 63 ? wl : fit ? L : cap;
            for (int c = (off + 63) >> 6; 64 * c < off + np; ++c) s_cb[c] = 64 * ((len + 1) >> 1);
        }
        __syncthreads();
        if (wave == 0) {  // offsets
            int v = s_cb[wl];
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(v, o, 64);
                if (wl >= o) v += y;
            }
            s_cb[wl] = v - s_cb[wl];
        }
        __syncthreads();
        // tpa lanes per atom again, a piece each: the table and, two entries a
        // word, a word per lane and row of the chunk, the stream
        for (int k0 = 0; k0 < N; k0 += apb) {
            const int k = k0 + (lane >> sh);
            if (k >= N) continue;
            int ns, l, m;
            cut(k, ns, l, m);
            for (int j = sub; j < ns; j += tpa) {
                const int len = l + (j >= ns - m ? 1 : 0);
                const int st = j * l + (j > ns - m ? j - (ns - m) : 0);
                const int p = atomicAdd(&s_hist[len < 63 ? len : 63], 1);  // the order is free
                rows[p] = (uint32_t)(k | len << MDT_NBR_IDX_BITS);
                const int src = k * capg + st;
                uint32_t *dst = stream + s_cb[p >> 6] + (p & 63);
                for (int e = 0; e < len; e += 2) {
                    const int e1 = e + 1 < len ? e + 1 : e;
                    dst[32 * e] = lds_scan ? lrow[src + e] | (uint32_t)lrow[src + e1] << 16
                                           : grow[src + e] | (uint32_t)grow[src + e1] << 16;
                }
            }
        }
        }
        __syncthreads();
        for (int i = lane; i < N; i += nthr) rec[i].w = w2[i] = w3[i] = 0;
        if (keep) {
            if (lane < (s_R + 63) / 64) chunk[lane] = s_cb[lane];
            if (lane == 0)  // read by the next launch
                *valid = make_int2(1 | (s_anyfold ? 2 : 0) | (s_slow ? 4 : 0) | s_R << 3, ecg->gen);
        }
    }
    const double *xt = s_folded ? xr : nullptr;
    // ---- flat lists: the near partners of the atoms outside the majority type ----
    // (two of those atoms with each other: listed at the lower index)
    auto flat_pair = [&](int h, int n, double d[3], double &r2, int &code) {
        if (n == h || !T.pair_on[typ[h] * MDT_MAXT + typ[n]] || (typ[n] != bulk && n < h)) return false;
        r2 = pair_image(s_ihf, bv.icell + 9 * t, s_sh, rec[h], rec[n], xt, N, h, n, d, &code);
        // (r2 = 0 is near; an atom without a position has no partners, as in the scan)
        return r2 == r2 && !(mul_rn(r2, mdt_rsqrt(r2)) > rnear);
    };
    const int nflat = MIXED ? 0 : (s_nflat < MDT_FLAT_MAX ? s_nflat : MDT_FLAT_MAX);
    for (int f = 0; f < nflat; ++f) {
        for (int n0 = 0; n0 < N; n0 += nthr) {
            double d[3], r2;
            int code = 0;
            const bool in = n0 + lane < N && flat_pair(s_flat[f], n0 + lane, d, r2, code);
            const unsigned long long m = __ballot(in);
            int base = 0;
            if (wl == 0 && m) base = atomicAdd(&s_fcnt[f], __popcll(m));  // the order is free
            base = __builtin_amdgcn_readfirstlane(base);
            const int pos = base + __popcll(m & below);
            if (in && pos < MDT_FLAT_CAP)
                s_flist[f * MDT_FLAT_CAP + pos] = (uint16_t)((n0 + lane) | (code << MDT_NBR_IDX_BITS));
        }
    }
    __syncthreads();
    const int R = s_R;
    const bool slow = s_slow != 0;  // entries without a fixed image
    if (!reuse && !direct && lane < R) {
        info0 = rows[lane];
        word0 = stream[s_cb[wave] + wl];
    }

    // ---- pair terms ----
    const double acut = ecg->acut, rcut = ecg->rcut;
    const float acutf = (float)acut, acutl2f = (float)(acut * MDT_LOG2E);
    // exp(acut (r - rcut)) in FP32; the bound (beyond the cut-off) keeps terms that
    // are multiplied by 0 finite
    auto cut_exp = [&](double r) { return mdt_exp2f(fminf(acutl2f * (float)(r - rcut), 100.0f)); };
    // theta and, for its derivative, rt1 = acut e1 theta
    auto theta = [&](double r, double *rt1) {
        if constexpr (PREC == 0) {
            const double e1 = mdt_exp_ab(r - rcut, acut * MDT_EXP_K, T.exptab);
            const double th = mdt_rcp(1 + e1);
            *rt1 = acut * e1 * th;
            return th;
        } else {
            const float e1 = cut_exp(r);
            const float th = mdt_rcpf(1.0f + e1);
            *rt1 = (double)(acutf * e1 * th);
            return (double)th;
        }
    };
    // sigma terms of the pair of types (tk, tn) at r: on k and on n
    auto sigma_terms = [&](int tk, int tn, double r, double &own, double &other) {
        if constexpr (PREC == 1) {
            const float e1 = cut_exp(r);
            const float th = mdt_rcpf(1.0f + e1);
            const float fsn = th * mdt_exp2f(-T.f_eta2l2[tn] * (float)(r - T.bs0[tn]));
            const float fsk = (tn == tk) ? fsn : th * mdt_exp2f(-T.f_eta2l2[tk] * (float)(r - T.bs0[tk]));
            own = (double)(T.f_csig[tk * MDT_MAXT + tn] * fsn);
            other = (double)(T.f_csig[tn * MDT_MAXT + tk] * fsk);
        } else {
            double rt1;
            const double th = theta(r, &rt1);
            const double fsn = th * mdt_exp_ab(T.etaT[tn], r - T.bs0[tn], T.exptab);
            const double fsk = (tn == tk) ? fsn : th * mdt_exp_ab(T.etaT[tk], r - T.bs0[tk], T.exptab);
            own = mul_rn(T.csig[tk * MDT_MAXT + tn], fsn);
            other = mul_rn(T.csig[tn * MDT_MAXT + tk], fsk);
        }
    };
    // dE/dr of the pair: density part through G of both atoms, pair (V) part
    // directly; and the pair energy
    auto force_terms = [&](int tk, int tn, double r, double Gk, double Gn, double &c, double &ep) {
        if (tn < tk) {  // one order of the sums, whichever of the two asks
            const int u = tk;
            tk = tn;
            tn = u;
            const double g = Gk;
            Gk = Gn;
            Gn = g;
        }
        const int kn = tk * MDT_MAXT + tn, nk = tn * MDT_MAXT + tk;
        if constexpr (PREC == 1) {
            const float e1 = cut_exp(r);
            const float th = mdt_rcpf(1.0f + e1);
            const float ae = acutf * e1;  // theta' / theta = ae th
            const float drn = (float)(r - T.bs0[tn]);
            const float fsn = th * mdt_exp2f(-T.f_eta2l2[tn] * drn);
            const float fvn = th * mdt_exp2f(-T.f_kdbl2[tn] * drn);
            if (tn == tk) {  // one element: one set of pair constants (kn == nk)
                const float fv = T.f_wv[kn] * fvn;
                c = fma((double)(T.f_csig[kn] * (fmaf(ae, th, T.f_etad[kn]) * fsn)), Gk + Gn, (double)(fmaf(ae, th, T.f_kdb[tn]) * fv));
                ep = (double)(2.0f * fv);
                return;
            }
            const float drk = (float)(r - T.bs0[tk]);
            const float fsk = th * mdt_exp2f(-T.f_eta2l2[tk] * drk);
            const float fvk = th * mdt_exp2f(-T.f_kdbl2[tk] * drk);
            const float ta = T.f_csig[kn] * (fmaf(ae, th, T.f_etad[kn]) * fsn);
            const float tb = T.f_csig[nk] * (fmaf(ae, th, T.f_etad[nk]) * fsk);
            const float tv = 0.5f * fmaf(T.f_wv[kn], fmaf(ae, th, T.f_kdb[tn]) * fvn, T.f_wv[nk] * (fmaf(ae, th, T.f_kdb[tk]) * fvk));
            c = fma(Gk, (double)ta, fma(Gn, (double)tb, (double)tv));
            ep = (double)fmaf(T.f_wv[kn], fvn, T.f_wv[nk] * fvk);
        } else {
            double rt1;
            const double th = theta(r, &rt1);
            const double drn = r - T.bs0[tn];
            const double fsn = th * mdt_exp_ab(T.etaT[tn], drn, T.exptab);
            const double fvn = th * mdt_exp_ab(T.kdbT[tn], drn, T.exptab);
            if (tn == tk) {
                const double fv = T.wv[kn] * fvn;
                c = fma(T.csig[kn] * ((T.etad[kn] + rt1) * fsn), Gk + Gn, (T.kdb[tn] + rt1) * fv);
                ep = 2.0 * fv;
            } else {
                const double drk = r - T.bs0[tk];
                const double fsk = th * mdt_exp_ab(T.etaT[tk], drk, T.exptab);
                const double fvk = th * mdt_exp_ab(T.kdbT[tk], drk, T.exptab);
                const double vn = T.wv[kn] * fvn, vk = T.wv[nk] * fvk;
                const double v = fma(T.kdb[tn] + rt1, vn, (T.kdb[tk] + rt1) * vk);
                c = fma(Gk * T.csig[kn], (T.etad[kn] + rt1) * fsn,
                        fma(Gn * T.csig[nk], (T.etad[nk] + rt1) * fsk, 0.5 * v));
                ep = vn + vk;
            }
        }
    };
    // a listed pair (entry q) of the atom at (xk, yk, zk): its vector; returns r^2
    auto listed = [&](unsigned q, double xk, double yk, double zk, const PairRec &pn, double &dx, double &dy, double &dz) {
        const double *sft = s_sh + 4 * (q >> MDT_NBR_IDX_BITS);
        dx = (xk - pn.x) - sft[0];
        dy = (yk - pn.y) - sft[1];
        dz = (zk - pn.z) - sft[2];
        return fma(dz, dz, fma(dy, dy, dx * dx));
    };
    // a pair's force crs d, added to n; its rounded components, as integers in u
    auto add_force = [&](int n, double crs, const double *d, double g[3], unsigned long long u[3]) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const double tq = fma(crs, d[q], MDT_FRC_C);
            u[q] = grid_int(tq, MDT_FRC_C);
            g[q] = tq - MDT_FRC_C;
        }
        atomicAdd(&rec[n].w, u[0]);
        atomicAdd(&w2[n], u[1]);
        atomicAdd(&w3[n], u[2]);
    };
    // a term of either pass from the fast limit on (rare): added by itself, to n and to k
    auto add_large = [&](int k, int n, double crs, const double *d) {
#pragma unroll 1
        for (int q = 0; q < 3; ++q) {
            double g;
            const unsigned long long u = grid_any(crs * d[q], MDT_P43, &g, &bad_local);
            unsigned long long *w = q == 0 ? &rec[n].w : (q == 1 ? w2 : w3) + n;
            atomicAdd(w, u);
            w = q == 0 ? &rec[k].w : (q == 1 ? w2 : w3) + k;
            atomicAdd(w, 0ull - u);
        }
    };
    // a row's pair (one type, its constants uniform): the sigma term of either atom, the force terms
    const int ub = MIXED ? 0 : bulk, ubb = ub * MDT_MAXT + ub;
    const double u_bs0 = ecg->betas0[ub], u_etaT = -ecg->eta2[ub] * MDT_EXP_K, u_kdbT = -ecg->kappadbeta[ub] * MDT_EXP_K;
    const double u_csig = ecg->csig[ubb], u_etad = ecg->etad[ubb], u_wv = ecg->wv[ubb], u_kdb = ecg->kappadbeta[ub];
    const float uf_eta = -(float)(ecg->eta2[ub] * MDT_LOG2E), uf_kdbl2 = -(float)(ecg->kappadbeta[ub] * MDT_LOG2E);
    const float uf_csig = (float)u_csig, uf_etad = (float)u_etad, uf_wv = (float)u_wv, uf_kdb = (float)u_kdb;
    auto bulk_sigma = [&](double r) {
        if constexpr (PREC == 1) {
            const float th = mdt_rcpf(1.0f + cut_exp(r));
            return (double)(uf_csig * (th * mdt_exp2f(uf_eta * (float)(r - u_bs0))));
        } else {
            double rt1;
            return mul_rn(u_csig, theta(r, &rt1) * mdt_exp_ab(u_etaT, r - u_bs0, T.exptab));
        }
    };
    auto bulk_force = [&](double r, double G2, double &c, double &ep) {  // G2: G of both atoms
        if constexpr (PREC == 1) {
            const float e1 = cut_exp(r);
            const float th = mdt_rcpf(1.0f + e1);
            const float ae = acutf * e1;  // theta' / theta = ae th
            const float dr = (float)(r - u_bs0);
            const float fs = th * mdt_exp2f(uf_eta * dr), fv = uf_wv * (th * mdt_exp2f(uf_kdbl2 * dr));
            c = fma((double)(uf_csig * (fmaf(ae, th, uf_etad) * fs)), G2, (double)(fmaf(ae, th, uf_kdb) * fv));
            ep = (double)(2.0f * fv);
        } else {
            double rt1;
            const double th = theta(r, &rt1);
            const double dr = r - u_bs0;
            const double fs = th * mdt_exp_ab(u_etaT, dr, T.exptab);
            const double fv = u_wv * (th * mdt_exp_ab(u_kdbT, dr, T.exptab));
            c = fma(u_csig * ((u_etad + rt1) * fs), G2, (u_kdb + rt1) * fv);
            ep = 2.0 * fv;
        }
    };
    // the lane's piece of round rb / nthr: the wavefront with the longest pieces of
    // one round has the shortest of the next
    auto piece_of = [&](int rb) {
        return rb + wl + ((rb / nthr & 1) ? nthr - 64 - 64 * wave : 64 * wave);
    };
    // The pairs of the lane's piece, atom k at (x, y, z): eval(n, G, r2, in) gives a
    // pair's terms (in false: none), add(n, terms, d) adds them; a lane's terms of a
    // `size` from lim on go to large(n, terms, d), which clears them.  Two entries at
    // a time without a branch between them.
    auto each_entry = [&](int r0, int k, int len, double x, double y, double z, double lim, auto eval, auto add,
                          auto large) {
        const uint32_t *src = stream + (direct ? 0 : s_cb[r0 >> 6]) + (r0 & 63);
        const uint16_t *row = lrow + k * capg + (r0 & ((1 << sh) - 1));  // direct
        const int last = 32 * (len - 1 & ~1);  // of the piece's words
        // entries e and e + 1 (the last one twice in an odd piece)
        auto word = [&](int e) {
            if (!direct) return src[32 * e < last ? 32 * e : last];
            const int e0 = e < len ? e : len - 1, e1 = e + 1 < len ? e + 1 : len - 1;
            return (uint32_t)row[e0 << sh] | (uint32_t)row[e1 << sh] << 16;
        };
        if (len == 0) return;  // a lane without an entry of its row (direct)
        uint32_t cur = !direct && r0 == lane ? word0 : word(0);
        double d[3], g[3];
        if (!slow) {
            for (int e = 0; e < len; e += 2) {
                const uint32_t q = cur;
                cur = word(e + 2);
                const PairRec a0 = rec[q & MDT_NBR_IDX_MASK], a1 = rec[q >> 16 & MDT_NBR_IDX_MASK];
                const double r0 = listed(q & 0xFFFF, x, y, z, a0, d[0], d[1], d[2]);
                const double r1 = listed(q >> 16, x, y, z, a1, g[0], g[1], g[2]);
                const int n0 = q & MDT_NBR_IDX_MASK, n1 = q >> 16 & MDT_NBR_IDX_MASK;
                auto t0 = eval(n0, a0.g, r0, true), t1 = eval(n1, a1.g, r1, e + 1 < len);
                if (__builtin_expect(!(fmax(t0.size, t1.size) < lim) || t0.size + t1.size != t0.size + t1.size, 0)) {
                    if (!(t0.size < lim)) large(n0, t0, d);
                    if (!(t1.size < lim)) large(n1, t1, g);
                }
                add(n0, t0, d);
                add(n1, t1, g);
            }
        } else {
            for (int e = 0; e < len; ++e) {
                const unsigned q = e & 1 ? cur >> 16 : cur & 0xFFFF;
                if (e & 1) cur = word(e + 1);
                const int n = q & MDT_NBR_IDX_MASK;
                const PairRec pn = rec[n];
                double r2;
                int code;
                if (q >> MDT_NBR_IDX_BITS == MDT_ANY_IMAGE) {
                    r2 = pair_image(s_ihf, bv.icell + 9 * t, s_sh, rec[k], pn, xt, N, k, n, d, &code);
                    // in a skewed cell its image may be anywhere; the terms of a pair
                    // beyond rnear count 0 times and stay finite up to 2 rnear
                    r2 = r2 > 4.0 * rnear * rnear ? 4.0 * rnear * rnear : r2;
                } else {
                    r2 = listed(q, x, y, z, pn, d[0], d[1], d[2]);
                }
                auto tm = eval(n, pn.g, r2, true);
                if (!(tm.size < lim)) large(n, tm, d);
                add(n, tm, d);
            }
        }
    };
    // f(n, d, r2) for the near partners of flat atom number q, one per lane from the
    // last wavefront on, which has the shortest pieces, or none
    auto each_flat = [&](int q, auto f) {
        const int h = s_flat[q], c = s_fcnt[q];
        const PairRec ph = rec[h];
        for (int e = lane + 64 < nthr ? lane + 64 : lane + 64 - nthr; e < (c <= MDT_FLAT_CAP ? c : N); e += nthr) {
            double d[3], r2;
            int n = e, code;
            if (c <= MDT_FLAT_CAP) {
                const unsigned ent = s_flist[q * MDT_FLAT_CAP + e];
                n = ent & MDT_NBR_IDX_MASK;
                r2 = listed(ent, ph.x, ph.y, ph.z, rec[n], d[0], d[1], d[2]);
            } else if (!flat_pair(h, n, d, r2, code)) {
                continue;
            }
            f(n, d, r2);
        }
    };

    // ---- phase 2: pass A, sigma ----
    for (int rb = 0; rb < R; rb += nthr) {
        const int r0 = piece_of(rb);
        if (r0 >= R) continue;
        const uint32_t info = rb == 0 ? info0 : rows[r0];
        const int k = info & MDT_NBR_IDX_MASK, len = info >> MDT_NBR_IDX_BITS;
        const double xk = rec[k].x, yk = rec[k].y, zk = rec[k].z;
        const int tk = MIXED ? typ[k] : 0;
        double s1 = 0.0, s2 = 0.0;
        struct Sig {
            double size, own, other;
        };
        each_entry(
            r0, k, len, xk, yk, zk, MDT_SIG_FAST,
            [&](int n, double, double r2, bool in) {
                const double r = mul_rn(r2, mdt_rsqrt(r2));
                Sig v;
                if constexpr (MIXED)
                    sigma_terms(tk, typ[n], r, v.own, v.other);
                else
                    v.own = v.other = bulk_sigma(r);
                const double on = in && !(r > rnear) ? 1.0 : 0.0;  // r > rnear: in the skin; a factor, not a branch
                v.own *= on;
                v.other *= on;
                v.size = MIXED ? fmax(v.own, v.other) : v.own;
                return v;
            },
            [&](int n, const Sig &v, const double *) {
                double h, l;
                unsigned long long u1, u2;
                sig_words(v.own, &u1, &u2, &h, &l);
                s1 += h;
                s2 += l;
                if constexpr (MIXED) sig_words(v.other, &u1, &u2, &h, &l);
                atomicAdd(&rec[n].w, u1);
                atomicAdd(&w2[n], u2);
            },
            [&](int n, Sig &v, const double *) {
                sig_large(&rec[k].w, v.own, &bad_local);
                sig_large(&rec[n].w, v.other, &bad_local);
                v.own = v.other = 0.0;
            });
        add_sum(&rec[k].w, s1, MDT_SIG_C1, MDT_P42, &bad_local);
        add_sum(&w2[k], s2, MDT_SIG_C2, MDT_P42 * MDT_P46, &bad_local);
    }
    for (int q = 0; q < nflat; ++q) {
        const int h = s_flat[q];
        unsigned long long s1 = 0, s2 = 0;
        each_flat(q, [&](int n, const double *d, double r2) {
            double own, other, hi, lo;
            unsigned long long u1, u2;
            sigma_terms(typ[h], typ[n], mul_rn(r2, mdt_rsqrt(r2)), own, other);
            if (!(own < MDT_SIG_FAST && other < MDT_SIG_FAST)) {
                sig_large(&rec[h].w, own, &bad_local);
                sig_large(&rec[n].w, other, &bad_local);
                return;
            }
            sig_words(own, &u1, &u2, &hi, &lo);
            s1 += u1;
            s2 += u2;
            sig_words(other, &u1, &u2, &hi, &lo);
            atomicAdd(&rec[n].w, u1);
            atomicAdd(&w2[n], u2);
        });
        add_uniform(&rec[h].w, s1);
        add_uniform(&w2[h], s2);
    }
    __syncthreads();

    // ---- tiny atoms: sigma~ of the near pairs below MDT_SIG_TINY; their
    // pairs beyond rnear from a minimum-image test of all atoms, a wavefront
    // per atom (lanes over partners: an order of the atoms' own).  A tiny
    // atom's share is summed by its own scan (below MDT_SIG_VTINY over the near
    // pairs too, in place of its words), the other atoms' through their words.
    int any = 0;
    for (int k = lane; k < N; k += nthr) {
        uint8_t ty = 0;
        if (T.owner[typ[k]]) {
            const double s = sig_sum(rec[k].w, w2[k]);
            ty = s < MDT_SIG_TINY ? (s < MDT_SIG_VTINY ? 2 : 1) : 0;
        }
        tiny[k] = ty;
        any |= ty;
    }
    const bool anytiny = __syncthreads_or(any);
    // the partners n of tiny atom k: within the cut-off, and beyond rnear unless `near`
    auto partner = [&](int k, int n, bool near, double d[3], double &r, double &ri) {
        if (n == k || !T.pair_on[typ[k] * MDT_MAXT + typ[n]]) return false;
        int code;
        const double r2 = pair_image(s_ihf, bv.icell + 9 * t, s_sh, rec[k], rec[n], xt, N, k, n, d, &code);
        ri = mdt_rsqrt(r2);
        r = mul_rn(r2, ri);
        return (near || r > rnear) && r <= cutr;
    };
    // calls f(k) for every tiny atom, each on one wavefront
    auto each_tiny = [&](auto f) {
        int at = 0;
        for (int t0 = 0; t0 < N; t0 += 64) {
            unsigned long long tm = __ballot(t0 + wl < N && tiny[t0 + wl] != 0);
            for (; tm; tm &= tm - 1, ++at)
                if (at % nwaves == wave) f(t0 + __builtin_ctzll(tm));
        }
    };
    if (anytiny) {
        each_tiny([&](int k) {
            const int tk = typ[k];
            const bool near = tiny[k] == 2;
            double sig = 0.0;
            for (int n0 = wl; n0 < N; n0 += 64) {
                int n = n0;
                opaque(n);
                double d[3], r, ri;
                if (!partner(k, n, near, d, r, ri)) continue;
                double own, other, hi, lo;
                unsigned long long u1, u2;
                sigma_terms(tk, typ[n], r, own, other);
                sig += own;
                if (r > rnear && !tiny[n]) {
                    sig_words(other, &u1, &u2, &hi, &lo);  // beyond rnear: far below MDT_SIG_FAST
                    atomicAdd(&rec[n].w, u1);
                    atomicAdd(&w2[n], u2);
                }
            }
            sig = wave_sum(sig);
            if (wl == 0) w3[k] = __double_as_longlong(sig);
        });
        __syncthreads();
    }

    // ---- per atom: s, dens, E_coh + vref, G = dE/dsigma ----
    double ep1 = 0.0, ep2 = 0.0;
    auto add_energy = [&](double ep) {
        const double h = (ep + MDT_EPR_C1) - MDT_EPR_C1;
        ep1 += h;
        ep2 += ((ep - h) + MDT_EPR_C2) - MDT_EPR_C2;
    };
    for (int k = lane; k < N; k += nthr) {
        const int tk = typ[k];
        double Gk = 0.0, Ek = 0.0;
        if (T.owner[tk]) {
            double dn;
            const double sig = (tiny[k] == 2 ? 0.0 : sig_sum(rec[k].w, w2[k])) + __longlong_as_double(w3[k]);
            emt_atom(T, tk, sig, &Gk, &Ek, &dn);
            if (!JUDGE) bv.dens[doff + k] = dn;  // raw EMT density (pes_emt_mod.f90:855,861)
        }
        rec[k].g = Gk;
        add_energy(-2.0 * Ek);
        rec[k].w = w2[k] = w3[k] = 0;  // force words from here on
    }
    __syncthreads();

    // ---- phase 3: pass B, pair forces and pair energies ----
    // each pair's dE/dr gives +F on the owner and -F on the partner
    // (Newton's third law)
    for (int rb = 0; rb < R; rb += nthr) {
        const int r0 = piece_of(rb);
        if (r0 >= R) continue;
        const uint32_t info = rb == 0 ? info0 : rows[r0];
        const int k = info & MDT_NBR_IDX_MASK, len = info >> MDT_NBR_IDX_BITS;
        const double xk = rec[k].x, yk = rec[k].y, zk = rec[k].z, Gk = rec[k].g;
        const int tk = MIXED ? typ[k] : 0;
        double fx = 0.0, fy = 0.0, fz = 0.0;
        struct Frc {
            double size, crs, ep;
        };
        each_entry(
            r0, k, len, xk, yk, zk, MDT_FRC_FAST,
            [&](int n, double Gn, double r2, bool in) {
                const double ri = mdt_rsqrt(r2);
                const double r = mul_rn(r2, ri);
                double c;
                Frc v;
                if constexpr (MIXED)
                    force_terms(tk, typ[n], r, Gk, Gn, c, v.ep);
                else
                    bulk_force(r, Gk + Gn, c, v.ep);
                const double on = in && !(r > rnear) ? 1.0 : 0.0;
                c *= on;
                v.ep *= on;
                v.size = fabs(c);
                v.crs = c * ri;
                return v;
            },
            [&](int n, const Frc &v, const double *d) {
                double g[3];
                unsigned long long u[3];
                add_energy(v.ep);
                add_force(n, v.crs, d, g, u);
                fx -= g[0];
                fy -= g[1];
                fz -= g[2];
            },
            [&](int n, Frc &v, const double *d) {
                add_large(k, n, v.crs, d);
                v.crs = 0.0;
            });
        add_sum(&rec[k].w, fx, MDT_FRC_C, MDT_P43, &bad_local);
        add_sum(&w2[k], fy, MDT_FRC_C, MDT_P43, &bad_local);
        add_sum(&w3[k], fz, MDT_FRC_C, MDT_P43, &bad_local);
    }
    // the pair (k, n) of an atom k that a wavefront's lanes share: -F on k in fk
    auto pair_forces = [&](int k, int n, const double *d, double r, double ri, unsigned long long fk[3]) {
        double c, ep, g[3];
        unsigned long long u[3];
        force_terms(typ[k], typ[n], r, rec[k].g, rec[n].g, c, ep);
        add_energy(ep);
        if (!(fabs(c) < MDT_FRC_FAST)) {
            add_large(k, n, c * ri, d);
            return;
        }
        add_force(n, c * ri, d, g, u);
#pragma unroll
        for (int q = 0; q < 3; ++q) fk[q] -= u[q];
    };
    for (int q = 0; q < nflat; ++q) {
        const int h = s_flat[q];
        unsigned long long fk[3] = {0, 0, 0};
        each_flat(q, [&](int n, const double *d, double r2) {
            const double ri = mdt_rsqrt(r2);
            pair_forces(h, n, d, mul_rn(r2, ri), ri, fk);
        });
        add_uniform(&rec[h].w, fk[0]);
        add_uniform(&w2[h], fk[1]);
        add_uniform(&w3[h], fk[2]);
    }
    // the pairs beyond rnear of the tiny atoms, a pair of two by its owner
    if (anytiny)
        each_tiny([&](int k) {
            unsigned long long fk[3] = {0, 0, 0};
            for (int n0 = wl; n0 < N; n0 += 64) {
                int n = n0;
                opaque(n);
                double d[3], r, ri;
                if ((tiny[n] && !owns(k, n)) || !partner(k, n, false, d, r, ri)) continue;
                pair_forces(k, n, d, r, ri, fk);
            }
            add_uniform(&rec[k].w, fk[0]);
            add_uniform(&w2[k], fk[1]);
            add_uniform(&w3[k], fk[2]);
        });
    ep1 = wave_sum(ep1);
    ep2 = wave_sum(ep2);
    if (wl == 0) {
        unsafeAtomicAdd(&s_ep[0], ep1);
        unsafeAtomicAdd(&s_ep[1], ep2);
    }
    __syncthreads();
    // ---- judge mode: compare with the given forces, write nothing else ----
    if constexpr (JUDGE) {
        double sq = 0.0, mx = 0.0;
        for (int k = lane; k < N; k += nthr) {
            const int tk = typ[k];
            for (int cc = 0; cc < 3; ++cc) {
                const double F = T.owner[tk] ? frc_sum(cc == 0 ? rec[k].w : cc == 1 ? w2[k] : w3[k]) : 0.0;
                const double d = F - bv.judge_f[roff + (long long)cc * N + k];
                sq += d * d;
                mx = fabs(d) > mx ? fabs(d) : mx;
            }
        }
        // fixed-order block reduction through jr[] (wave partials, then wave 0)
        for (int o = 32; o > 0; o >>= 1) {
            sq += __shfl_xor(sq, o, 64);
            const double m2 = __shfl_xor(mx, o, 64);
            mx = m2 > mx ? m2 : mx;
        }
        __shared__ double jr[32];
        if (wl == 0) {
            jr[2 * wave] = sq;
            jr[2 * wave + 1] = mx;
        }
        __syncthreads();
        if (lane == 0) {
            double s2 = 0.0, m2 = 0.0;
            for (int w = 0; w < nwaves; ++w) {
                s2 += jr[2 * w];
                m2 = jr[2 * w + 1] > m2 ? jr[2 * w + 1] : m2;
            }
            bv.judge_acc[3 * rep] += s2;
            bv.judge_acc[3 * rep + 1] += 3.0 * N;
            bv.judge_acc[3 * rep + 2] = m2 > bv.judge_acc[3 * rep + 2] ? m2 : bv.judge_acc[3 * rep + 2];
        }
        if (bad_local) atomicOr(&bv.status[t], bad_local);
        return;
    }

    // ---- phase 4: set_acceleration (force.f90:89-98), outputs ----
    for (int k = lane; k < N; k += nthr) {
        double F[3] = {frc_sum(rec[k].w), frc_sum(w2[k]), frc_sum(w3[k])};
        if (!T.owner[typ[k]]) F[0] = F[1] = F[2] = 0.0;
        if (add_fin) {
            F[0] += bv.f[roff + k];
            F[1] += bv.f[roff + N + k];
            F[2] += bv.f[roff + 2 * N + k];
        }
        const int fb = k == lane ? fixed0 : bv.fixed[doff + k];
        const double mass = k == lane ? mass0 : bv.mass[aoff + k];
        bv.f[roff + k] = F[0];
        bv.f[roff + N + k] = F[1];
        bv.f[roff + 2 * N + k] = F[2];
        bv.a[roff + k] = (fb & 1) ? 0.0 : F[0] / mass;
        bv.a[roff + N + k] = (fb & 2) ? 0.0 : F[1] / mass;
        bv.a[roff + 2 * N + k] = (fb & 4) ? 0.0 : F[2] / mass;
    }
    if (lane == 0) bv.epot[bv.traj_eoff[t] + b] = -0.5 * (s_ep[0] + s_ep[1]);
    if (bad_local) atomicOr(&bv.status[t], bad_local);
}

// ---------------------------------------------------------------------------
// collect_trajectory_characteristics after propagate_2 of step step_prev
// (src/trajectory_info.f90:47-263) for trajectory t: centroids, the
// projectile (atom 0) against every other atom (min image).  Reads x, v and
// f of the projectile and x of every atom from global memory (written
// before the caller's barrier); every lane of the block calls it.  Returns
// (block-uniform) whether the trajectory left the box and is frozen from
// this step.
__device__ bool traj_observe(const PropConst &pc, const int *s_proj, const BatchView &bv, int t, int N, int P,
                             long long soff, long long aoff, int lane, int nthr, uint32_t step_prev,
                             double *s_rmin, int *s_done) {
#pragma clang fp contract(off)
#define OX(c, b, i) (soff + ((long long)(b) * 3 + (c)) * N + (i))
        // centroids, the projectile (atom 0) against every other atom (min image)
        double cx = 0.0, cy = 0.0, cz = 0.0, vz = 0.0;
        int fnz = 0, above = 1, below = 1;
        for (int b = 0; b < P; ++b) {
            cx += bv.x[OX(0, b, 0)];
            cy += bv.x[OX(1, b, 0)];
            cz += bv.x[OX(2, b, 0)];
            vz += bv.v[OX(2, b, 0)];
            if (bv.f[OX(0, b, 0)] != 0.0 || bv.f[OX(1, b, 0)] != 0.0 || bv.f[OX(2, b, 0)] != 0.0) fnz = 1;
            if (!(bv.x[OX(2, b, 0)] > bv.obs_ul)) above = 0;
            if (!(bv.x[OX(2, b, 0)] < bv.obs_ll)) below = 0;
        }
        cx /= P;
        cy /= P;
        cz /= P;
        vz /= P;
        double h[9], ih[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            h[k] = bv.cell[9 * t + k];
            ih[k] = bv.icell[9 * t + k];
        }
        double rmin = 1.0e300;
        for (int i = 1 + lane; i < N; i += nthr) {
            const int ty = bv.type[aoff + i];
        const int pb = (pc.mixed && !s_proj[ty]) ? 1 : P;
            double ax = 0.0, ay = 0.0, az = 0.0;
            for (int b = 0; b < pb; ++b) {
                ax += bv.x[OX(0, b, i)];
                ay += bv.x[OX(1, b, i)];
                az += bv.x[OX(2, b, i)];
            }
            const double d0 = cx - ax / pb, d1 = cy - ay / pb, d2 = cz - az / pb;
            double s0 = ih[0] * d0 + ih[3] * d1 + ih[6] * d2;
            double s1 = ih[1] * d0 + ih[4] * d1 + ih[7] * d2;
            double s2 = ih[2] * d0 + ih[5] * d1 + ih[8] * d2;
            s0 -= round(s0);
            s1 -= round(s1);
            s2 -= round(s2);
            const double e0 = h[0] * s0 + h[3] * s1 + h[6] * s2;
            const double e1 = h[1] * s0 + h[4] * s1 + h[7] * s2;
            const double e2 = h[2] * s0 + h[5] * s1 + h[8] * s2;
            const double r = sqrt(e0 * e0 + e1 * e1 + e2 * e2);
            rmin = r < rmin ? r : rmin;
        }
        for (int o = 32; o > 0; o >>= 1) {
            const double y = __shfl_xor(rmin, o, 64);
            rmin = y < rmin ? y : rmin;
        }
        if ((lane & 63) == 0) s_rmin[lane >> 6] = rmin;
        __syncthreads();
        if (lane == 0) {
            for (int w = 1; w < (nthr + 63) / 64; ++w) rmin = s_rmin[w] < rmin ? s_rmin[w] : rmin;
            TrajObs &o = bv.obs[t];
            const int istep = (int)(step_prev - bv.obs_step0);
            if (rmin < o.cl_appr) {
                o.cl_appr = rmin;
                o.cl_appr_step = istep;
            }
            o.cl_last = rmin;
            o.last_step = istep;
            o.adsorbed_prev = o.adsorbed;
            if (!o.adsorbed && rmin < bv.ads_start) o.adsorbed = 1;
            if (o.adsorbed && rmin > bv.ads_end) o.adsorbed = 0;
            if (cz < o.r_min[2]) {
                o.r_min[0] = cx;
                o.r_min[1] = cy;
                o.r_min[2] = cz;
            }
            if (fnz) o.t_int += pc.dt;
            const int down = vz < 0.0;
            if (down != o.moving_down) {
                ++o.turning_points;
                o.moving_down = down;
            }
            *s_done = bv.obs_exit && (above || below);
            if (*s_done) {
                o.exit_step = istep;
                bv.done[t] = 1;
            }
        }
        __syncthreads();
    return *s_done != 0;
#undef OX
}

// The propagator updates shared by k_prop and k_traj_classical, in the
// reference's operation order with FMA contraction off (the pragma's flag
// stays on the instructions after inlining): both kernels then give
// bitwise the same states, whatever code surrounds the updates.
// langevin_2 (md_algo.f90:253-285) and langevin_1 (:165-198):
__device__ __forceinline__ double lan_w(const LanCoef &L) {
#pragma clang fp contract(off)
    return L.sv * sqrt(1 - L.crv * L.crv);
}
__device__ __forceinline__ double lan_v2(const LanCoef &L, double w, double v, double a, double eta) {
#pragma clang fp contract(off)
    return v + L.c2 * a + w * eta;
}
__device__ __forceinline__ double lan_x1(const LanCoef &L, double dt, double r, double v, double a, double eta) {
#pragma clang fp contract(off)
    return r + L.c1 * v + L.c2 * dt * a + L.sr * eta;
}
__device__ __forceinline__ double lan_v1(const LanCoef &L, double v, double a, double eta) {
#pragma clang fp contract(off)
    return L.c0 * v + (L.c1 - L.c2) * a + L.sv * L.crv * eta;
}
// velocity Verlet half step and drift (md_algo.f90:108-131, 226-245)
__device__ __forceinline__ double verlet_v(double v, double dt, double a) {
#pragma clang fp contract(off)
    return v + 0.5 * dt * a;
}
__device__ __forceinline__ double verlet_x(double x, double dt, double vn) {
#pragma clang fp contract(off)
    return x + dt * vn;
}

// ---------------------------------------------------------------------------
// The propagators of batches with ring polymers, PILE or Andersen atoms or
// one-bead slabs of more than 256 atoms.  One lane per atom-bead; a
// workgroup holds every bead of a run of atoms (PropChunk, at most 256
// atom-beads), so that all couplings but one -- the branch test of
// langevin_1 over an atom's beads, the spring forces, the normal-mode
// transforms -- stay inside it, and a trajectory spreads over as many
// workgroups as it has work for.  The one coupling across atoms,
// remove_com_velocity, takes the chunks' partial sums to a second launch.
//
// flags bit0: propagate_2, bit1: propagate_1, bit2: ring-polymer step (atoms
// with one bead only get f = 0 from it, as calc_force zeroes f), bit3: the COM
// velocity is removed after propagate_1 (k_com_ring follows, which also
// takes the transforms of the ring-polymer step, since those read the
// corrected velocities).
// step_base (graph replays): when non-null, *step_base is added to both step
// numbers, which are then offsets within the captured chunk.
// Mixed bead mode (pc.mixed): atoms of non-projectile types are classical --
// one bead, kept in bead 0 (the other bead slots are not read): their
// Langevin / Andersen temperature is kB T / m, PILE acts on their single
// mode, positions advance in propagate_1 and the ring-polymer step skips
// them; in the COM sum a classical atom counts as P identical beads.
//
// Memory bound: about 200 B per atom-bead and launch.  64 trajectories of
// H/Pt 8x8x6 with 32 beads (788k atom-beads, 3136 chunks) take 46 us in
// k_prop and 33 us in k_com_ring, against 511 us with one workgroup of 256
// lanes per trajectory (64 of 256 CUs, x and v through global memory between
// the phases); 192 uneven H/Au trajectories 38 against 401 us; 384 mixed
// trajectories of H/Pt 6x6x4 14 + 10 against 41 us.
// ---------------------------------------------------------------------------

// The chunk of this workgroup.  Workgroups go round the 8 XCDs in launch
// order, so consecutive chunks -- which share cache lines, their rows of
// [bead][component][atom] being short -- are given to one XCD.
__device__ __forceinline__ int chunk_of_block(int nchunk) {
    const int per = (nchunk + 7) >> 3;
    return ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
}

// C (P x P, column-major cjk(j,k)) to LDS in columns of P + 1 entries: the
// forward transform reads down a column per lane, and columns P apart would
// share their banks.  Every lane calls it; the caller synchronises.
__device__ __forceinline__ void load_cjk(double *C, const double *cjk, int P, int lane, int nthr) {
    for (int k = lane; k < P * P; k += nthr) C[(k / P) * (P + 1) + k % P] = cjk[k];
}

// The exact free step of one atom's ring polymer (do_ring_polymer_step,
// rpmd.f90:309-452) on x, v of the lane's atom-bead: forward transform and
// harmonic rotation of mode k = the lane's bead, then back.  s_x, s_v:
// 3 x 256 LDS words each, holding the chunk's x and v ([component][slot],
// slot = bead na + atom of the chunk); on: the lane's atom takes part.
// Every lane of the block calls it; x and v of fixed components stay.
__device__ __forceinline__ void ring_transform(double (*s_x)[256], double (*s_v)[256], const double *C, bool on, int a,
                                               int k, int na, int P, double mass, double temp_k, double dt, uint8_t fb,
                                               double x[3], double v[3]) {
    const int lane = threadIdx.x;
    const int ld = P + 1;
    double p[3] = {0.0, 0.0, 0.0}, q[3] = {0.0, 0.0, 0.0};
    if (on) {
        for (int j = 0; j < P; ++j) {
            const double cj = C[j + ld * k];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                p[c] = p[c] + (mass * s_v[c][j * na + a]) * cj;
                q[c] = q[c] + s_x[c][j * na + a] * cj;
            }
        }
        const double betaN = 1.0 / (MDT_KB * temp_k * P);
        const double twown = 2.0 / betaN / MDT_HBAR;
        double p1 = 1.0, p2 = 0.0, p3 = dt / mass, p4 = 1.0;
        const int fk = (k <= P / 2) ? k : P - k;  // mirrored modes share a frequency
        if (fk > 0) {
            const double wk = twown * sin(fk * (MDT_PI / P));
            const double wt = wk * dt, wm = wk * mass;
            const double cw = cos(wt), sw = sin(wt);
            p1 = cw;
            p2 = -wm * sw;
            p3 = sw / wm;
            p4 = cw;
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double pn = p[c] * p1 + q[c] * p2;
            q[c] = p[c] * p3 + q[c] * p4;
            p[c] = pn;
        }
    }
    __syncthreads();
    if (on)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            s_v[c][lane] = p[c];
            s_x[c][lane] = q[c];
        }
    __syncthreads();
    if (on) {
        double rr[3] = {0.0, 0.0, 0.0}, vv[3] = {0.0, 0.0, 0.0};
        for (int j = 0; j < P; ++j) {
            const double cj = C[k + ld * j];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                rr[c] = rr[c] + s_x[c][j * na + a] * cj;
                vv[c] = vv[c] + s_v[c][j * na + a] * cj / mass;
            }
        }
#pragma unroll
        for (int c = 0; c < 3; ++c)
            if (!(fb >> c & 1)) {
                x[c] = rr[c];
                v[c] = vv[c];
            }
    }
}

// 4 waves per SIMD: the registers of langevin_1's normals and coefficients
// held to 128.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
k_prop(const PropConst *__restrict__ pcg, BatchView bv, const double *cjk_all, const long long *cjk_off,
       const PropChunk *__restrict__ chunks, int nchunk, double *__restrict__ com, const uint32_t *step_base,
       uint32_t step_prev, uint32_t step, int flags) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double s_x[3][256], s_v[3][256];
    __shared__ int s_small[256];
    __shared__ double s_com[4][4];
    const PropConst &pc = *pcg;
    const int w = chunk_of_block(nchunk);
    if (w >= nchunk) return;  // whole block: uniform
    const PropChunk ch = chunks[w];
    const int t = ch.t, na = ch.na, nb = ch.nb;
    if (bv.done && bv.done[t]) return;  // frozen trajectory (whole block: uniform)
    const int N = bv.traj_N[t], P = bv.traj_P[t];
    const long long soff = bv.traj_soff[t];
    const long long aoff = bv.traj_aoff[t];
    const uint32_t tid = bv.traj_id[t];
    const double tsurf = bv.tsurf[t], tproj = bv.tproj[t];
    const double dt = pc.dt;
    const int lane = threadIdx.x, nthr = blockDim.x;
    if (step_base) {  // graph replays: step numbers are offsets from the device counter
        const uint32_t s0 = *step_base;
        step_prev += s0;
        step += s0;
    }
    double *C = (double *)smem_raw;  // P (P + 1), loaded where the chunk transforms
    const bool act = lane < na * nb;
    const int b = lane / na, a_ = lane - b * na;  // bead, atom of the chunk
    const int i = ch.i0 + a_;
    const long long xi = soff + (long long)b * 3 * N + i;             // component 0; + N per component
    const long long pi = soff / 3 + (long long)b * N + i;
    int ty = 0, algo = MDT_PROP_VERLET;
    uint8_t fb = 7;
    double mass = 1.0, dn = 0.0;
    double x[3] = {0.0, 0.0, 0.0}, v[3] = {0.0, 0.0, 0.0}, a[3] = {0.0, 0.0, 0.0}, v0[3] = {0.0, 0.0, 0.0};
    int bad_local = 0;
    if (act) {
        ty = bv.type[aoff + i];
        algo = pc.algo[ty];
        fb = bv.fixed[pi];
        mass = bv.mass[aoff + i];
        dn = bv.dens[pi];
        const bool ring = (flags & 4) && nb > 1;  // the spring forces and transforms read every bead's x
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            v0[c] = v[c] = bv.v[xi + (long long)c * N];
            if (ring || ((flags & 2) && !(fb >> c & 1))) x[c] = bv.x[xi + (long long)c * N];
            if ((flags & 3) && !(fb >> c & 1)) a[c] = bv.a[xi + (long long)c * N];
        }
    }
    const bool lan = act && algo == MDT_PROP_LANGEVIN;
    const double temp_k = pc.is_proj[ty] ? tproj : tsurf;
    LanCoef L;
    if (flags & 3) {
        if ((flags & 1) && lan) {
            int bad = 0;
            dn = ldfa(dn, mass, &bad);  // per bead (md_algo.f90:97)
            if (bad) bad_local |= MDT_ST_NEG_DENSITY;
            bv.dens[pi] = dn;
        }
        // the branch test of langevin_1 / langevin_2: every bead of the atom (md_algo.f90:176)
        bool big = lan_big(dn, dt);
        if (nb > 1) {
            if (lane < na) s_small[lane] = 0;
            __syncthreads();
            if (act && !big) s_small[a_] = 1;  // benign race: every writer stores 1
            __syncthreads();
            big = act && !s_small[a_];
        }
        if (lan) {
            const double temp = MDT_KB * nb * temp_k / mass;
            L = lan_coef(dn, dt, temp, big && temp > MDT_TOLERANCE);
        }
    }
    if ((flags & 1) && act) {  // propagate_2 of step step_prev
        if (lan) {
            const double w2 = lan_w(L);
#pragma unroll
            for (int c = 0; c < 3; ++c)  // the deviate of that step's langevin_1, kept by propagate_1
                v[c] = (fb >> c & 1) ? 0.0 : lan_v2(L, w2, v[c], a[c], bv.eta[xi + (long long)c * N]);
        } else {
#pragma unroll
            for (int c = 0; c < 3; ++c) v[c] = (fb >> c & 1) ? 0.0 : verlet_v(v[c], dt, a[c]);
        }
    }
    bool have_c = false;
    if (flags & 2) {  // propagate_1 of step step
        // pile_thermostat (md_algo.f90:440-502)
        if (pc.any_pile && nb == 1 && act && algo == MDT_PROP_PILE) {
            const double betaN = 1.0 / (MDT_KB * temp_k);
            const double c1 = exp(-0.5 * dt * (1 / pc.pile_tau));
            const double c2 = sqrt(1 - c1 * c1);
            for (int c = 0; c < 3; ++c) {
                const double z = mdt_normal(pc.seed, tid, step, MDT_STREAM_PILE, (uint32_t)(i * P), (uint32_t)c);
                const double np = c1 * (mass * v[c]) + sqrt(mass / betaN) * c2 * z;
                v[c] = (fb >> c & 1) ? 0.0 : np / mass;
            }
        }
        if (pc.any_pile && nb > 1) {
            const bool pile = act && algo == MDT_PROP_PILE;
            if (__syncthreads_or(pile)) {
                load_cjk(C, cjk_all + cjk_off[t], P, lane, nthr);
                have_c = true;
                const int k = b, ld = P + 1;
#pragma unroll
                for (int c = 0; c < 3; ++c) s_v[c][lane] = v[c];
                __syncthreads();
                double acc[3] = {0.0, 0.0, 0.0};
                if (pile) {
                    for (int j = 0; j < P; ++j) {
                        const double cj = C[j + ld * k];
#pragma unroll
                        for (int c = 0; c < 3; ++c) acc[c] = acc[c] + (mass * s_v[c][j * na + a_]) * cj;
                    }
                    const double betaN = 1.0 / (MDT_KB * temp_k * P);
                    double g;
                    if (k == 0) {
                        g = 1 / pc.pile_tau;
                    } else {
                        const double wn = 1 / betaN / MDT_HBAR;
                        const double wk = 2 * wn * sin(k * MDT_PI / P);
                        g = 2 * wk;
                    }
                    const double c1 = exp(-0.5 * dt * g);
                    const double c2 = sqrt(1 - c1 * c1);
                    double z[3];
                    mdt_normal3(pc.seed, tid, step, MDT_STREAM_PILE, (uint32_t)(i * P + k), z);
#pragma unroll
                    for (int c = 0; c < 3; ++c) acc[c] = c1 * acc[c] + sqrt(mass / betaN) * c2 * z[c];
                }
                __syncthreads();
#pragma unroll
                for (int c = 0; c < 3; ++c) s_v[c][lane] = acc[c];
                __syncthreads();
                if (pile) {
                    double ap[3] = {0.0, 0.0, 0.0};
                    for (int j = 0; j < P; ++j) {
                        const double cj = C[b + ld * j];
#pragma unroll
                        for (int c = 0; c < 3; ++c) ap[c] = ap[c] + s_v[c][j * na + a_] * cj;
                    }
#pragma unroll
                    for (int c = 0; c < 3; ++c) v[c] = (fb >> c & 1) ? 0.0 : ap[c] / mass;
                }
                __syncthreads();  // s_v is used again below
            }
        }
        if (lan) {
            if (fb != 7) {  // a fixed component uses no deviate
                double z[3];
                mdt_normal3(pc.seed, tid, step, MDT_STREAM_LANGEVIN, (uint32_t)(i * P + b), z);
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const double eta = z[c];
                    if (!(fb >> c & 1)) {
                        bv.eta[xi + (long long)c * N] = eta;  // langevin_2 of this step takes the same deviate
                        const double r = x[c], vo = v[c];
                        x[c] = lan_x1(L, dt, r, vo, a[c], eta);
                        v[c] = lan_v1(L, vo, a[c], eta);
                    } else {
                        v[c] = 0.0;
                    }
                }
            } else {
                v[0] = v[1] = v[2] = 0.0;
            }
        } else if (act && (algo == MDT_PROP_VERLET || algo == MDT_PROP_ANDERSEN || algo == MDT_PROP_PILE)) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const double vn = (fb >> c & 1) ? 0.0 : verlet_v(v[c], dt, a[c]);
                v[c] = vn;
                if (nb == 1 && !(fb >> c & 1)) x[c] = verlet_x(x[c], dt, vn);
            }
            if (algo == MDT_PROP_ANDERSEN) {
                const double sigma = sqrt(nb * MDT_KB * temp_k / mass);
                const double u = mdt_uniform(pc.seed, tid, step, MDT_STREAM_ANDERSEN_U, (uint32_t)(i * P + b), 0u);
                if (u < dt / pc.andersen_time) {
                    double z[3];
                    mdt_normal3(pc.seed, tid, step, MDT_STREAM_ANDERSEN_V, (uint32_t)(i * P + b), z);
#pragma unroll
                    for (int c = 0; c < 3; ++c)
                        if (!(fb >> c & 1)) v[c] = z[c] * sigma + 0.0;
                }
            }
        } else if (act) {
            bad_local |= MDT_ST_BAD_PROP;
        }
        if (flags & 8) {  // this chunk's part of remove_com_velocity's sums, in a fixed order
            double s[4];
#pragma unroll
            for (int c = 0; c < 3; ++c) s[c] = act ? v[c] * mass * (P / nb) : 0.0;  // classical: P identical beads
            s[3] = act && b == 0 ? mass : 0.0;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                for (int o = 32; o > 0; o >>= 1) s[c] += __shfl_xor(s[c], o, 64);
                if ((lane & 63) == 0) s_com[lane >> 6][c] = s[c];
            }
            __syncthreads();
            if (lane < 4) com[4 * (long long)w + lane] = s_com[0][lane] + s_com[1][lane] + s_com[2][lane] + s_com[3][lane];
        }
    }
    bool moved = (flags & 2) != 0;
    if (flags & 4) {
        double f[3] = {0.0, 0.0, 0.0};
        if (nb > 1) {
            const bool tr = act && !lan && !(flags & 8);
            __syncthreads();
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                s_x[c][lane] = x[c];
                s_v[c][lane] = v[c];
            }
            const bool any_tr = __syncthreads_or(tr);
            if (lan) {
                // the step is reverted; spring force with m(1) and Tproj (rpmd.f90:418-435)
                const double kt = MDT_KB * tproj * P / MDT_HBAR;
                const double prefactor = -1 * bv.mass[aoff + 0] * (kt * kt);
                const int pv = b == 0 ? P - 1 : b - 1, nx = b == P - 1 ? 0 : b + 1;
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    f[c] = prefactor * (2 * x[c] - s_x[c][pv * na + a_] - s_x[c][nx * na + a_]);
            }
            if (any_tr) {
                if (!have_c) {
                    load_cjk(C, cjk_all + cjk_off[t], P, lane, nthr);
                    __syncthreads();
                }
                ring_transform(s_x, s_v, C, tr, a_, b, na, P, mass, temp_k, dt, fb, x, v);
                moved = moved || tr;
            }
        }
        if (act)
#pragma unroll
            for (int c = 0; c < 3; ++c) bv.f[xi + (long long)c * N] = f[c];
    }
    if (act)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const bool fixc = fb >> c & 1;
            // a fixed component's v is written only when it was not 0 already
            if (((flags & 3) || moved) && (!fixc || v0[c] != v[c])) bv.v[xi + (long long)c * N] = v[c];
            if (moved && !fixc) bv.x[xi + (long long)c * N] = x[c];
        }
    if (bad_local) atomicOr(&bv.status[t], bad_local);
}

// remove_com_velocity (the closed form of its 1000 iterations) from the
// chunks' partial sums, then the transforms of the ring-polymer step.
__global__ void __launch_bounds__(256)
k_com_ring(const PropConst *__restrict__ pcg, BatchView bv, const double *cjk_all, const long long *cjk_off,
           const PropChunk *__restrict__ chunks, int nchunk, const double *__restrict__ com, int flags) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double s_x[3][256], s_v[3][256];
    const PropConst &pc = *pcg;
    const int w = chunk_of_block(nchunk);
    if (w >= nchunk) return;  // whole block: uniform
    const PropChunk ch = chunks[w];
    const int t = ch.t, na = ch.na, nb = ch.nb;
    if (bv.done && bv.done[t]) return;  // frozen trajectory (whole block: uniform)
    const int N = bv.traj_N[t], P = bv.traj_P[t];
    const long long soff = bv.traj_soff[t];
    const long long aoff = bv.traj_aoff[t];
    const int lane = threadIdx.x, nthr = blockDim.x;
    double *C = (double *)smem_raw;
    const bool act = lane < na * nb;
    const int b = lane / na, a_ = lane - b * na;
    const int i = ch.i0 + a_;
    const long long xi = soff + (long long)b * 3 * N + i;
    double x[3] = {0.0, 0.0, 0.0}, v[3] = {0.0, 0.0, 0.0};
    if (act)
#pragma unroll
        for (int c = 0; c < 3; ++c) v[c] = bv.v[xi + (long long)c * N];
    __shared__ double s_sub[3];
    if (lane < 64) {  // the trajectory's partial sums, in an order of its own chunks only
        double sum[4] = {0.0, 0.0, 0.0, 0.0};
        for (int q = lane; q < ch.count; q += 64)
#pragma unroll
            for (int c = 0; c < 4; ++c) sum[c] += com[4 * (long long)(ch.first + q) + c];
#pragma unroll
        for (int c = 0; c < 4; ++c)
            for (int o = 32; o > 0; o >>= 1) sum[c] += __shfl_xor(sum[c], o, 64);
        if (lane == 0) {
            const double fac = (1.0 - pow(1.0 - 1.0 / N, 1000.0)) / sum[3] / P;
#pragma unroll
            for (int c = 0; c < 3; ++c) s_sub[c] = sum[c] * fac;
        }
    }
    __syncthreads();
    if (act)
#pragma unroll
        for (int c = 0; c < 3; ++c) v[c] -= s_sub[c];
    const int ty = act ? bv.type[aoff + i] : 0;
    const bool tr = (flags & 4) && nb > 1 && act && pc.algo[ty] != MDT_PROP_LANGEVIN;
    if (__syncthreads_or(tr)) {
        load_cjk(C, cjk_all + cjk_off[t], P, lane, nthr);
        uint8_t fb = 7;
        double mass = 1.0;
        if (tr) {
            fb = bv.fixed[soff / 3 + (long long)b * N + i];
            mass = bv.mass[aoff + i];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                x[c] = bv.x[xi + (long long)c * N];
                s_x[c][lane] = x[c];
                s_v[c][lane] = v[c];
            }
        }
        __syncthreads();
        ring_transform(s_x, s_v, C, tr, a_, b, na, P, mass, pc.is_proj[ty] ? bv.tproj[t] : bv.tsurf[t], pc.dt, fb, x, v);
        if (tr)
#pragma unroll
            for (int c = 0; c < 3; ++c)
                if (!(fb >> c & 1)) bv.x[xi + (long long)c * N] = x[c];
    }
    if (act)
#pragma unroll
        for (int c = 0; c < 3; ++c) bv.v[xi + (long long)c * N] = v[c];
}

// traj_observe between propagate_2 and propagate_1 of k_prop, one workgroup
// per trajectory
__global__ void __launch_bounds__(256)
k_observe(const PropConst *__restrict__ pcg, BatchView bv, const uint32_t *step_base, uint32_t step_prev) {
    __shared__ int s_proj[MDT_MAXT];
    __shared__ double s_rmin[4];
    __shared__ int s_done;
    const PropConst &pc = *pcg;
    const int t = blockIdx.x;
    if (bv.done && bv.done[t]) return;  // frozen trajectory (whole block: uniform)
    if (step_base) step_prev += *step_base;
    for (int k = threadIdx.x; k < MDT_MAXT; k += blockDim.x) s_proj[k] = pc.is_proj[k];
    __syncthreads();
    traj_observe(pc, s_proj, bv, t, bv.traj_N[t], bv.traj_P[t], bv.traj_soff[t], bv.traj_aoff[t], threadIdx.x,
                 blockDim.x, step_prev, s_rmin, &s_done);
}

// ---------------------------------------------------------------------------
// k_traj_classical: the propagators of batches of classical trajectories
// (P = 1) with every atom on its own lane and no PILE or Andersen atoms (no
// COM removal): each lane keeps its atom's state in registers from
// propagate_2 through propagate_1 and the force reset, reading and writing
// each array once; the only barriers are the observer's, which runs inside.
// Same arithmetic, in the same order, as k_prop; a kernel of its own so that
// k_prop's ring-polymer code does not set its register budget.
__global__ void __launch_bounds__(256)
k_traj_classical(const PropConst *__restrict__ pcg, BatchView bv, const uint32_t *step_base, uint32_t step_prev,
                 uint32_t step, int flags, int t_base) {
    __shared__ int s_algo[MDT_MAXT], s_proj[MDT_MAXT];
    __shared__ double s_rmin[4];
    __shared__ int s_done;
    const PropConst &pc = *pcg;
    const int t = t_base + (int)blockIdx.x;  // trajectories t_base .. t_base + gridDim.x - 1
    if (bv.done && bv.done[t]) return;  // frozen trajectory (whole block: uniform)
    const int N = bv.traj_N[t];
    const long long soff = bv.traj_soff[t];
    const long long poff = soff / 3;
    const long long aoff = bv.traj_aoff[t];
    const uint32_t tid = bv.traj_id[t];
    const double tsurf = bv.tsurf[t], tproj = bv.tproj[t];
    const double dt = pc.dt;
    const int nthr = blockDim.x, lane = threadIdx.x;
    if (step_base) {  // graph replays: step numbers are offsets from the device counter
        const uint32_t s0 = *step_base;
        step_prev += s0;
        step += s0;
    }
    for (int k = lane; k < MDT_MAXT; k += nthr) {
        s_algo[k] = pc.algo[k];
        s_proj[k] = pc.is_proj[k];
    }
    int bad_local = 0;
#define XI(c, b, i) (soff + ((long long)(b) * 3 + (c)) * N + (i))
#define PI_(b, i) (poff + (long long)(b) * N + (i))
    __syncthreads();
    {
        const int i = lane;
        const bool act = i < N;
        double x[3] = {0.0, 0.0, 0.0}, v[3] = {0.0, 0.0, 0.0}, a[3] = {0.0, 0.0, 0.0};
        double dn = 0.0, mass = 1.0;
        int ty = 0, algo = MDT_PROP_VERLET;
        uint8_t fb = 0;
        // A fixed component keeps its position, gets v = 0 and uses no
        // deviate: its x, a and eta are not read, its x and eta not written,
        // and its v written only when it was not already 0 (the fixed bottom
        // layers are half the atoms of a slab).
        double v0[3] = {0.0, 0.0, 0.0};
        if (act) {
            ty = bv.type[aoff + i];
            algo = s_algo[ty];
            fb = bv.fixed[PI_(0, i)];
            mass = bv.mass[aoff + i];
            dn = bv.dens[PI_(0, i)];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                v0[c] = v[c] = bv.v[XI(c, 0, i)];
                if (!(fb >> c & 1)) {
                    x[c] = bv.x[XI(c, 0, i)];
                    a[c] = bv.a[XI(c, 0, i)];
                }
            }
        }
        const double temp = MDT_KB * (s_proj[ty] ? tproj : tsurf) / mass;
        LanCoef L;
        bool have = false;
        if ((flags & 1) && act) {  // propagate_2 of step step_prev
            if (algo == MDT_PROP_LANGEVIN) {
                int bad = 0;
                dn = ldfa(dn, mass, &bad);  // md_algo.f90:97
                if (bad) bad_local |= MDT_ST_NEG_DENSITY;
                bv.dens[PI_(0, i)] = dn;
                L = lan_coef(dn, dt, temp, lan_big(dn, dt) && temp > MDT_TOLERANCE);
                have = true;
                const double w = lan_w(L);
#pragma unroll
                for (int c = 0; c < 3; ++c) v[c] = (fb >> c & 1) ? 0.0 : lan_v2(L, w, v[c], a[c], bv.eta[XI(c, 0, i)]);
            } else {
#pragma unroll
                for (int c = 0; c < 3; ++c) v[c] = (fb >> c & 1) ? 0.0 : verlet_v(v[c], dt, a[c]);
            }
        }
        if ((flags & 1) && bv.obs) {
            if (i == 0)
                for (int c = 0; c < 3; ++c) bv.v[XI(c, 0, i)] = v[c];  // the observer reads the projectile's
            __syncthreads();
            if (traj_observe(pc, s_proj, bv, t, N, 1, soff, aoff, lane, nthr, step_prev, s_rmin, &s_done)) {
                // frozen: the state after this propagate_2 is the trajectory's last
                if (act)
                    for (int c = 0; c < 3; ++c)
                        if (!(fb >> c & 1) || v0[c] != 0.0) bv.v[XI(c, 0, i)] = v[c];
                if (bad_local) atomicOr(&bv.status[t], bad_local);
                return;
            }
        }
        if ((flags & 2) && act) {  // propagate_1 of step step
            if (algo == MDT_PROP_LANGEVIN) {
                if (!have) L = lan_coef(dn, dt, temp, lan_big(dn, dt) && temp > MDT_TOLERANCE);
                double z[3];
                mdt_normal3(pc.seed, tid, step, MDT_STREAM_LANGEVIN, (uint32_t)i, z);
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const double eta = z[c];
                    if (!(fb >> c & 1)) {
                        bv.eta[XI(c, 0, i)] = eta;  // langevin_2 of this step takes the same deviate
                        const double r = x[c], vo = v[c];
                        x[c] = lan_x1(L, dt, r, vo, a[c], eta);
                        v[c] = lan_v1(L, vo, a[c], eta);
                    } else {
                        v[c] = 0.0;
                    }
                }
            } else if (algo == MDT_PROP_VERLET) {
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const double vn = (fb >> c & 1) ? 0.0 : verlet_v(v[c], dt, a[c]);
                    v[c] = vn;
                    if (!(fb >> c & 1)) x[c] = verlet_x(x[c], dt, vn);
                }
            } else {
                bad_local |= MDT_ST_BAD_PROP;
            }
        }
        if (act) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const bool fixc = fb >> c & 1;
                if ((flags & 3) && (!fixc || v0[c] != 0.0)) bv.v[XI(c, 0, i)] = v[c];
                if ((flags & 2) && !fixc) bv.x[XI(c, 0, i)] = x[c];
                if (flags & 4) bv.f[XI(c, 0, i)] = 0.0;  // calc_force zeroes f (P == 1)
            }
        }
    }
#undef XI
#undef PI_
    if (bad_local) atomicOr(&bv.status[t], bad_local);
}

// ---------------------------------------------------------------------------
// k_mixed: calc_force of a mixed-bead trajectory (one workgroup, 512 lanes):
// atom 0 (the projectile) has P beads, atoms 1..N-1 are classical and kept
// in bead 0.  The potential of bead b is the EMT energy of the classical
// atoms with projectile bead b; the classical atoms feel the bead average
// of their forces (the force on a rigid P-bead copy divided by P).  Because
// the classical-classical pair geometry does not depend on the bead, the
// averaged force needs the pair passes once, with G replaced by its bead
// average, plus the projectile pairs of every bead:
//   1. owned half lists of the classical atoms (HBM), sigma^0 from their
//      pairs (pass A), per atom G^0, E^0, dens^0;
//   2. per bead b, 16 lanes: the classical atoms within the cut-off of the
//      projectile's bead b; its sigma, G_H(b), E_H(b); then per listed atom
//      a: sigma_a(b) = sigma_a^0 + its projectile term, G_a(b), E_a(b), the
//      pair force (+F to bead b, -F/P to atom a) and pair energy, and the
//      bead averages of G_a and dens_a (fixed point);
//   3. the classical pairs (pass B) with the averaged G.
// epot(b) = sum_a (E_a^0 - V pairs / 2) + sum_{a near b} (E_a(b) - E_a^0)
//           + E_H(b) - V_H(b) / 2.
// ---------------------------------------------------------------------------
#define MIX_CAPQ 192  // classical atoms within the cut-off of one projectile bead
#define MIX_G 16      // lanes per bead
#define MIX_BLOCK 512

// MAXB: 512, or 1024 for trajectories large enough that one 512-lane
// workgroup per CU leaves the classical passes short of waves (the extra
// lanes work the classical atoms; the bead groups stay in the first 512).
template <int TPA, int MAXB = 512>
__global__ void __launch_bounds__(MAXB, 2)
    k_mixed(const EmtConst *__restrict__ ecg, const PropConst *__restrict__ pcg, BatchView bv, int add_fin) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ LdsTables T;
    __shared__ double red[1];
    const int t = bv.rep_list ? bv.rep_list[blockIdx.x] : (int)blockIdx.x;  // trajectory list
    if (bv.done && bv.done[t]) return;  // frozen trajectory (whole block: uniform)
    const int N = bv.traj_N[t], P = bv.traj_P[t];
    const int Ns = N - 1;
    const int cap = bv.nbcap < Ns - 1 ? bv.nbcap : (Ns > 1 ? Ns - 1 : 1);
    const long long soff = bv.traj_soff[t];
    const long long poff = soff / 3;
    const long long aoff = bv.traj_aoff[t];
    const int nthr = blockDim.x, lane = threadIdx.x;
    CellRegs cell;
    load_cell(bv, t, cell);
    load_tables(T, ecg, pcg, cell, lane, nthr);

    // LDS: px py pz | A0 A1 A2 | G0 E0 D0 S0 | Gacc Dacc (classical atoms,
    // local index a = atom - 1) | per bead hx hy hz Eb | per
    // bead group GH EH DH | cnt cntf | group hcnt, hlist | typ (all atoms) |
    // tiny (classical atoms).  The words A0-A2 hold the fractional
    // coordinates in the scan, the sigma fixed point in pass A and the force
    // fixed point afterwards.  A classical atom's list holds its near entries
    // (within the near radius) from the front (cnt) and its far entries
    // (between the near radius and the cut-off) from the back (cntf); the far
    // entries are evaluated only for pairs with a tiny atom, one whose sigma
    // from its near pairs is below MDT_SIG_TINY.
    const int ngrp = MIX_BLOCK / MIX_G;
    double *px = (double *)smem_raw, *py = px + Ns, *pz = py + Ns;
    double *sx = pz + Ns, *sy = sx + Ns, *sz = sy + Ns;
    unsigned long long *shi = (unsigned long long *)sx, *smid = (unsigned long long *)sy,
                       *slo = (unsigned long long *)sz;
    unsigned long long *fxa = shi, *fya = smid, *fza = slo;
    double *G0 = sz + Ns, *E0 = G0 + Ns, *D0 = E0 + Ns, *S0 = D0 + Ns;
    unsigned long long *Gacc = (unsigned long long *)(S0 + Ns), *Dacc = Gacc + Ns;
    double *hx = (double *)(Dacc + Ns), *hy = hx + P, *hz = hy + P, *Eb = hz + P;
    double *GH = Eb + P, *EH = GH + ngrp, *DH = EH + ngrp;
    uint16_t *cnt = (uint16_t *)(DH + ngrp);
    uint16_t *cntf = cnt + Ns;
    uint16_t *hcnt = cntf + Ns;
    uint16_t *hlist = hcnt + ngrp;
    uint8_t *typ = (uint8_t *)(hlist + (size_t)ngrp * MIX_CAPQ);
    uint8_t *tiny = typ + N;
    __shared__ int s_anytiny;
    uint16_t *nbr = bv.nbr_global + (size_t)blockIdx.x * bv.nbr_stride;
    int bad_local = 0;
    // Verlet skin for the classical lists: built with cut-off + skin, reused
    // while no classical atom moved more than skin / 2 since the build.  The
    // positions keep the fold of the build, so the lists' image codes stay
    // valid; a cell narrower than 2 (cut-off + skin) rebuilds every launch.
    const long long slot = blockIdx.x;
    double wmin = 1e300;
    for (int q = 0; q < 3; ++q) {
        const double w = 1.0 / sqrt(cell.ih[q] * cell.ih[q] + cell.ih[q + 3] * cell.ih[q + 3] +
                                    cell.ih[q + 6] * cell.ih[q + 6]);
        wmin = w < wmin ? w : wmin;
    }
    const double skin = bv.mix_skin;
    const bool keep = skin > 0.0 && bv.mix_valid && 2.0 * (ecg->cutr + skin) < wmin;
    double *ref = keep ? bv.mix_ref + slot * 3 * bv.mix_ns : nullptr;
    double *fold = keep ? bv.mix_fold + slot * 3 * bv.mix_ns : nullptr;
    __shared__ int s_reuse;
    if (lane == 0) s_reuse = keep && bv.mix_valid[slot];
    __syncthreads();
    if (s_reuse) {  // every thread reads the flag before any clears it
        double dmax = 0.0;
        for (int a = lane; a < Ns; a += nthr) {
            const int i = a + 1;
            const double d0 = bv.x[soff + i] - ref[3 * a], d1 = bv.x[soff + N + i] - ref[3 * a + 1],
                         d2 = bv.x[soff + 2 * N + i] - ref[3 * a + 2];
            const double d2s = d0 * d0 + d1 * d1 + d2 * d2;
            dmax = d2s > dmax ? d2s : dmax;
        }
        __syncthreads();
        if (dmax > 0.25 * skin * skin) s_reuse = 0;  // benign race: every writer stores 0
    }
    __syncthreads();
    const bool reuse = s_reuse != 0;

    // ---- stage: classical atoms (bead 0) and the projectile's beads, folded ----
    for (int i = lane; i < N; i += nthr) typ[i] = (uint8_t)bv.type[aoff + i];
    for (int a = lane; a < Ns; a += nthr) {
        const int i = a + 1;
        const double r[3] = {bv.x[soff + i], bv.x[soff + N + i], bv.x[soff + 2 * N + i]};
        double f0 = cell.ih[0] * r[0] + cell.ih[3] * r[1] + cell.ih[6] * r[2];
        double f1 = cell.ih[1] * r[0] + cell.ih[4] * r[1] + cell.ih[7] * r[2];
        double f2 = cell.ih[2] * r[0] + cell.ih[5] * r[1] + cell.ih[8] * r[2];
        if (reuse) {  // the fold of the list build
            f0 -= fold[3 * a];
            f1 -= fold[3 * a + 1];
            f2 -= fold[3 * a + 2];
        } else {
            const double g0 = floor(f0), g1 = floor(f1), g2 = floor(f2);
            f0 -= g0;
            f1 -= g1;
            f2 -= g2;
            if (keep) {
                fold[3 * a] = g0;
                fold[3 * a + 1] = g1;
                fold[3 * a + 2] = g2;
                ref[3 * a] = r[0];
                ref[3 * a + 1] = r[1];
                ref[3 * a + 2] = r[2];
            }
        }
        sx[a] = f0;
        sy[a] = f1;
        sz[a] = f2;
        px[a] = cell.h[0] * f0 + cell.h[3] * f1 + cell.h[6] * f2;
        py[a] = cell.h[1] * f0 + cell.h[4] * f1 + cell.h[7] * f2;
        pz[a] = cell.h[2] * f0 + cell.h[5] * f1 + cell.h[8] * f2;
    }
    for (int b = lane; b < P; b += nthr) {
        const long long rb = soff + (long long)b * 3 * N;
        const double r[3] = {bv.x[rb], bv.x[rb + N], bv.x[rb + 2 * N]};
        double f0 = cell.ih[0] * r[0] + cell.ih[3] * r[1] + cell.ih[6] * r[2];
        double f1 = cell.ih[1] * r[0] + cell.ih[4] * r[1] + cell.ih[7] * r[2];
        double f2 = cell.ih[2] * r[0] + cell.ih[5] * r[1] + cell.ih[8] * r[2];
        f0 -= floor(f0);
        f1 -= floor(f1);
        f2 -= floor(f2);
        hx[b] = cell.h[0] * f0 + cell.h[3] * f1 + cell.h[6] * f2;
        hy[b] = cell.h[1] * f0 + cell.h[4] * f1 + cell.h[7] * f2;
        hz[b] = cell.h[2] * f0 + cell.h[5] * f1 + cell.h[8] * f2;
    }
    __syncthreads();
    const double acut = ecg->acut, rcut = ecg->rcut, cutr = ecg->cutr, cut2 = ecg->cut2hi;
    const int apb = nthr / TPA;
    const int wl = lane & 63;
    const unsigned long long below = (wl == 0) ? 0ull : ((~0ull) >> (64 - wl));
    const unsigned long long gmask = (TPA >= 64 ? ~0ull : ((1ull << TPA) - 1ull)) << ((wl / TPA) * TPA);
    const int tq = typ[0];

    // ---- 1a: owned half lists of the classical atoms ----
    // FP32 membership scan on float copies of the fractional coordinates (in
    // the G0/E0/D0 words, unused until pass A), r^2 bound widened by 1e-4;
    // both passes re-check r <= cutr in FP64, and half-cell ties take the
    // reference's image (tie_image)
    float *fx32 = (float *)G0, *fy32 = (float *)E0, *fz32 = (float *)D0;
    uint16_t *kcnt = keep ? bv.mix_cnt + slot * 2 * bv.mix_ns : nullptr;
    uint16_t *kcntf = keep ? kcnt + bv.mix_ns : nullptr;
    if (reuse)
        for (int a = lane; a < Ns; a += nthr) {
            cnt[a] = kcnt[a];
            cntf[a] = kcntf[a];
        }
    for (int a = lane; a < Ns; a += nthr) {
        fx32[a] = (float)sx[a];
        fy32[a] = (float)sy[a];
        fz32[a] = (float)sz[a];
    }
    __syncthreads();
    float hf[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) hf[q] = (float)cell.h[q];
    const double cutl = keep ? (ecg->cutr + skin) * (ecg->cutr + skin) : cut2;
    const float cut2f = (float)(cutl * (1.0 + 1e-4));
    const double rn = keep ? ecg->rnear + skin : ecg->rnear;  // near / far split (k_replica)
    const float near2f = (float)(rn * rn * (1.0 + 1e-4));
    const int mmax = Ns / 2 + 1;  // owned candidates only, in increasing index (as k_replica)
    for (int k0 = 0; k0 < (reuse ? 0 : Ns); k0 += apb) {
        const int k = k0 + lane / TPA;
        const int sub = lane % TPA;
        const bool act = k < Ns;
        const int tk = act ? typ[k + 1] : 0;
        const float fxk = act ? fx32[k] : 0.f, fyk = act ? fy32[k] : 0.f, fzk = act ? fz32[k] : 0.f;
        const int a_lo = (k + 1) >> 1;
        int c = 0, cf = 0;
        for (int m0 = 0; m0 < mmax; m0 += TPA) {
            const int mi = m0 + sub;
            const int n = mi < a_lo ? ((k + 1) & 1) + 2 * mi : k + 2 + 2 * (mi - a_lo);
            bool in = false, nr = false;
            int code = 0;
            if (act && n < Ns) {
                const int tn = typ[n + 1];
                if (T.pair_on[tk * MDT_MAXT + tn]) {
                    float d0 = fxk - fx32[n], d1 = fyk - fy32[n], d2 = fzk - fz32[n];
                    float m0 = rintf(d0), m1 = rintf(d1), m2 = rintf(d2);
                    const bool t0 = fabsf(fabsf(d0) - 0.5f) < 1e-4f, t1 = fabsf(fabsf(d1) - 0.5f) < 1e-4f,
                               t2 = fabsf(fabsf(d2) - 0.5f) < 1e-4f;
                    if (t0 | t1 | t2) {  // half-cell tie: the reference's image
                        const double *xr = bv.x + soff;
                        const double a0 = xr[k + 1], a1 = xr[N + k + 1], a2 = xr[2 * N + k + 1];
                        const double b0 = xr[n + 1], b1 = xr[N + n + 1], b2 = xr[2 * N + n + 1];
                        if (t0) m0 = (float)tie_image(cell.ih[0], cell.ih[3], cell.ih[6], a0, a1, a2, b0, b1, b2, sx[k] - sx[n]);
                        if (t1) m1 = (float)tie_image(cell.ih[1], cell.ih[4], cell.ih[7], a0, a1, a2, b0, b1, b2, sy[k] - sy[n]);
                        if (t2) m2 = (float)tie_image(cell.ih[2], cell.ih[5], cell.ih[8], a0, a1, a2, b0, b1, b2, sz[k] - sz[n]);
                    }
                    d0 -= m0;
                    d1 -= m1;
                    d2 -= m2;
                    const float ex = hf[0] * d0 + hf[3] * d1 + hf[6] * d2;
                    const float ey = hf[1] * d0 + hf[4] * d1 + hf[7] * d2;
                    const float ez = hf[2] * d0 + hf[5] * d1 + hf[8] * d2;
                    const float rr2 = ex * ex + ey * ey + ez * ez;
                    in = rr2 <= cut2f;
                    nr = rr2 <= near2f;
                    code = ((int)m0 + 1) + 3 * ((int)m1 + 1) + 9 * ((int)m2 + 1);
                }
            }
            const unsigned long long mall = __ballot(in) & gmask;
            const unsigned long long mn = __ballot(in && nr) & gmask;
            const unsigned long long mf = mall & ~mn;
            if (in) {  // near entries from the front, far entries from the back
                const int pos = nr ? c + __popcll(mn & below) : cf + __popcll(mf & below);
                if (pos < cap)
                    nbr[(size_t)k * cap + (nr ? pos : cap - 1 - pos)] = (uint16_t)(n | (code << MDT_NBR_IDX_BITS));
            }
            c += __popcll(mn);
            cf += __popcll(mf);
        }
        if (act && sub == 0) {
            if (c + cf > cap) bad_local |= MDT_ST_NBR_OVERFLOW;
            cnt[k] = (uint16_t)(c < cap ? c : cap);
            cntf[k] = (uint16_t)(cf < cap - cnt[k] ? cf : cap - cnt[k]);
            if (keep) {
                kcnt[k] = cnt[k];
                kcntf[k] = cntf[k];
            }
        }
    }
    __syncthreads();
    if (keep && !reuse && lane == 0) bv.mix_valid[slot] = 1;  // read by the next launch
    for (int a = lane; a < Ns; a += nthr) shi[a] = smid[a] = slo[a] = 0ull;
    __syncthreads();

    // ---- 1b: sigma^0 of the classical atoms (pass A over their pairs) ----
    // near entries; then, for the pairs with a tiny atom (sigma^0 from the
    // near pairs below MDT_SIG_TINY), the far entries too
    auto pair_a = [&](int k, int tk, double xk, double yk, double zk, int e, bool far, double &sig) {
        const unsigned q = nbr[(size_t)k * cap + e];
        const int n = q & MDT_NBR_IDX_MASK, code = q >> MDT_NBR_IDX_BITS;
        if (far && !(tiny[k] | tiny[n])) return;
        const int tn = typ[n + 1];
        const double dx = (xk - px[n]) - T.shift[3 * code];
        const double dy = (yk - py[n]) - T.shift[3 * code + 1];
        const double dz = (zk - pz[n]) - T.shift[3 * code + 2];
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double r = r2 * mdt_rsqrt(r2);
        if (r > cutr) return;
        const double e1 = mdt_exp(acut * (r - rcut), T.exptab);
        const double th = mdt_rcp(1 + e1);
        const double fsn = th * mdt_exp(-T.eta2[tn] * (r - T.bs0[tn]), T.exptab);
        const double fsk = (tn == tk) ? fsn : th * mdt_exp(-T.eta2[tk] * (r - T.bs0[tk]), T.exptab);
        sig += T.csig[tk * MDT_MAXT + tn] * fsn;
        sig_add_scaled(&shi[n], &smid[n], &slo[n], T.csig48[tn * MDT_MAXT + tk] * fsk, &bad_local);
    };
    for (int k0 = 0; k0 < Ns; k0 += apb) {
        const int k = k0 + lane / TPA;
        const int sub = lane % TPA;
        const bool act = k < Ns;
        double sig = 0.0;
        if (act) {
            const int tk = typ[k + 1];
            const double xk = px[k], yk = py[k], zk = pz[k];
            const int ck = cnt[k];
            for (int e = sub; e < ck; e += TPA) pair_a(k, tk, xk, yk, zk, e, false, sig);
        }
        sig = group_sum<TPA>(sig);
        if (act && sub == 0) G0[k] = sig;
    }
    if (lane == 0) s_anytiny = 0;
    __syncthreads();
    for (int a = lane; a < Ns; a += nthr) {
        const uint8_t ty = (T.owner[typ[a + 1]] && G0[a] + sig_value(shi[a], smid[a], slo[a]) < MDT_SIG_TINY) ? 1 : 0;
        tiny[a] = ty;
        if (ty) s_anytiny = 1;  // benign race: every writer stores 1
    }
    __syncthreads();
    const bool anytiny = s_anytiny != 0;
    if (anytiny) {
        for (int k0 = 0; k0 < Ns; k0 += apb) {
            const int k = k0 + lane / TPA;
            const int sub = lane % TPA;
            const bool act = k < Ns;
            double sig = 0.0;
            if (act) {
                const int tk = typ[k + 1];
                const double xk = px[k], yk = py[k], zk = pz[k];
                for (int e = cap - cntf[k] + sub; e < cap; e += TPA) pair_a(k, tk, xk, yk, zk, e, true, sig);
            }
            sig = group_sum<TPA>(sig);
            if (act && sub == 0) G0[k] += sig;
        }
        __syncthreads();
    }
    for (int a = lane; a < Ns; a += nthr) {
        const int ta = typ[a + 1];
        double g = 0.0, e = 0.0, dn = 0.0;
        const double s0 = G0[a] + sig_value(shi[a], smid[a], slo[a]);
        if (T.owner[ta]) emt_atom(T, ta, s0, &g, &e, &dn);
        S0[a] = s0;
        G0[a] = g;
        E0[a] = e;
        D0[a] = dn;
        Gacc[a] = Dacc[a] = 0ull;
    }
    __syncthreads();
    for (int a = lane; a < Ns; a += nthr) fxa[a] = fya[a] = fza[a] = 0ull;  // force words from here on
    __syncthreads();

    // ---- 2: the projectile's beads, MIX_G lanes each ----
    const int grp = lane / MIX_G, gsub = lane % MIX_G;
    const unsigned long long qmask = ((1ull << MIX_G) - 1ull) << ((wl / MIX_G) * MIX_G);
    const double invP = 1.0 / P;
    const int kn = tq * MDT_MAXT, kq = tq;
    for (int b0 = 0; b0 < P; b0 += ngrp) {
        const int b = b0 + grp;
        const bool bact = grp < ngrp && b < P;
        // 2a: classical atoms within the cut-off of bead b
        {
            int c = 0;
            const double xq = bact ? hx[b] : 0.0, yq = bact ? hy[b] : 0.0, zq = bact ? hz[b] : 0.0;
            for (int n0 = 0; n0 < Ns; n0 += MIX_G) {
                const int n = n0 + gsub;
                bool in = false;
                int code = 0;
                if (bact && n < Ns && T.pair_on[kn + typ[n + 1]]) {
                    // fractional difference from the folded cartesian positions (the
                    // fractional words hold sigma / force sums by now)
                    const double cx = xq - px[n], cy = yq - py[n], cz = zq - pz[n];
                    double d0 = cell.ih[0] * cx + cell.ih[3] * cy + cell.ih[6] * cz;
                    double d1 = cell.ih[1] * cx + cell.ih[4] * cy + cell.ih[7] * cz;
                    double d2 = cell.ih[2] * cx + cell.ih[5] * cy + cell.ih[8] * cz;
                    double m0 = rint(d0), m1 = rint(d1), m2 = rint(d2);
                    const bool t0 = fabs(fabs(d0) - 0.5) < 1e-4, t1 = fabs(fabs(d1) - 0.5) < 1e-4,
                               t2 = fabs(fabs(d2) - 0.5) < 1e-4;
                    if (t0 | t1 | t2) {  // half-cell tie: the reference's image (slab in bead 0)
                        const double *xh = bv.x + soff + (long long)b * 3 * N, *xs = bv.x + soff;
                        const double a0 = xh[0], a1 = xh[N], a2 = xh[2 * N];
                        const double b0 = xs[n + 1], b1 = xs[N + n + 1], b2 = xs[2 * N + n + 1];
                        if (t0) m0 = tie_image(cell.ih[0], cell.ih[3], cell.ih[6], a0, a1, a2, b0, b1, b2, d0);
                        if (t1) m1 = tie_image(cell.ih[1], cell.ih[4], cell.ih[7], a0, a1, a2, b0, b1, b2, d1);
                        if (t2) m2 = tie_image(cell.ih[2], cell.ih[5], cell.ih[8], a0, a1, a2, b0, b1, b2, d2);
                    }
                    d0 -= m0;
                    d1 -= m1;
                    d2 -= m2;
                    const double ex = cell.h[0] * d0 + cell.h[3] * d1 + cell.h[6] * d2;
                    const double ey = cell.h[1] * d0 + cell.h[4] * d1 + cell.h[7] * d2;
                    const double ez = cell.h[2] * d0 + cell.h[5] * d1 + cell.h[8] * d2;
                    in = (ex * ex + ey * ey + ez * ez) <= cut2;
                    code = ((int)m0 + 1) + 3 * ((int)m1 + 1) + 9 * ((int)m2 + 1);
                }
                const unsigned long long m = __ballot(in) & qmask;
                if (in) {
                    const int pos = c + __popcll(m & below);
                    if (pos < MIX_CAPQ)
                        hlist[(size_t)grp * MIX_CAPQ + pos] = (uint16_t)(n | (code << MDT_NBR_IDX_BITS));
                    else
                        bad_local |= MDT_ST_NBR_OVERFLOW;
                }
                c += __popcll(m);
            }
            if (gsub == 0 && grp < ngrp) hcnt[grp] = (uint16_t)(c < MIX_CAPQ ? c : MIX_CAPQ);
        }
        __syncthreads();
        // 2b: sigma of the projectile's bead b
        {
            double sig = 0.0;
            const int ch = bact ? hcnt[grp] : 0;
            for (int e = gsub; e < ch; e += MIX_G) {
                const unsigned q = hlist[(size_t)grp * MIX_CAPQ + e];
                const int n = q & MDT_NBR_IDX_MASK, code = q >> MDT_NBR_IDX_BITS;
                const int tn = typ[n + 1];
                const double dx = (hx[b] - px[n]) - T.shift[3 * code];
                const double dy = (hy[b] - py[n]) - T.shift[3 * code + 1];
                const double dz = (hz[b] - pz[n]) - T.shift[3 * code + 2];
                const double r2 = dx * dx + dy * dy + dz * dz;
                const double r = r2 * mdt_rsqrt(r2);
                if (r > cutr) continue;
                const double e1 = mdt_exp(acut * (r - rcut), T.exptab);
                const double th = mdt_rcp(1 + e1);
                sig += T.csig[kn + tn] * (th * mdt_exp(-T.eta2[tn] * (r - T.bs0[tn]), T.exptab));
            }
            sig = group_sum<MIX_G>(sig);
            if (bact && gsub == 0) {
                double g = 0.0, e = 0.0, dn = 0.0;
                if (T.owner[tq]) emt_atom(T, tq, sig, &g, &e, &dn);
                GH[grp] = g;
                EH[grp] = e;
                DH[grp] = dn;
            }
        }
        __syncthreads();
        // 2c: the listed atoms' sigma(b), G(b), E(b); pair forces and energies
        {
            double fx = 0.0, fy = 0.0, fz = 0.0, dE = 0.0, vs = 0.0;
            const int ch = bact ? hcnt[grp] : 0;
            const double Gq = bact ? GH[grp] : 0.0;
            for (int e = gsub; e < ch; e += MIX_G) {
                const unsigned q = hlist[(size_t)grp * MIX_CAPQ + e];
                const int n = q & MDT_NBR_IDX_MASK, code = q >> MDT_NBR_IDX_BITS;
                const int tn = typ[n + 1];
                const double dx = (hx[b] - px[n]) - T.shift[3 * code];
                const double dy = (hy[b] - py[n]) - T.shift[3 * code + 1];
                const double dz = (hz[b] - pz[n]) - T.shift[3 * code + 2];
                const double r2 = dx * dx + dy * dy + dz * dz;
                const double ri = mdt_rsqrt(r2);
                const double r = r2 * ri;
                if (r > cutr) continue;
                const double e1 = mdt_exp(acut * (r - rcut), T.exptab);
                const double th = mdt_rcp(1 + e1);
                const double rt1 = acut * e1 * th;
                const double fsn = th * mdt_exp(-T.eta2[tn] * (r - T.bs0[tn]), T.exptab);
                const double fvn = th * mdt_exp(-T.kdb[tn] * (r - T.bs0[tn]), T.exptab);
                double fsk = fsn, fvk = fvn;
                if (tn != tq) {
                    fsk = th * mdt_exp(-T.eta2[kq] * (r - T.bs0[kq]), T.exptab);
                    fvk = th * mdt_exp(-T.kdb[kq] * (r - T.bs0[kq]), T.exptab);
                }
                const int nk = tn * MDT_MAXT + tq;
                // the classical atom with this bead's projectile term
                double Gn = 0.0, En = 0.0, Dn = 0.0;
                if (T.owner[tn]) emt_atom(T, tn, S0[n] + T.csig[nk] * fsk, &Gn, &En, &Dn);
                dE += En - E0[n];
                fx_add(&Gacc[n], (Gn - G0[n]) * invP, MDT_F_SCALE, &bad_local);
                fx_add(&Dacc[n], (Dn - D0[n]) * invP, MDT_F_SCALE, &bad_local);
                const double c = Gq * T.csig[kn + tn] * ((T.etad[kn + tn] + rt1) * fsn) +
                                 Gn * T.csig[nk] * ((T.etad[nk] + rt1) * fsk) +
                                 0.5 * (T.wv[kn + tn] * ((T.kdb[tn] + rt1) * fvn) + T.wv[nk] * ((T.kdb[kq] + rt1) * fvk));
                vs += T.wv[kn + tn] * fvn + T.wv[nk] * fvk;
                const double cr = c * ri;
                fx -= cr * dx;
                fy -= cr * dy;
                fz -= cr * dz;
                fx_add(&fxa[n], cr * dx * invP, MDT_F_SCALE, &bad_local);
                fx_add(&fya[n], cr * dy * invP, MDT_F_SCALE, &bad_local);
                fx_add(&fza[n], cr * dz * invP, MDT_F_SCALE, &bad_local);
            }
            fx = group_sum<MIX_G>(fx);
            fy = group_sum<MIX_G>(fy);
            fz = group_sum<MIX_G>(fz);
            dE = group_sum<MIX_G>(dE);
            vs = group_sum<MIX_G>(vs);
            if (bact && gsub == 0) {
                const long long rb = soff + (long long)b * 3 * N;
                double F[3] = {T.owner[tq] ? fx : 0.0, T.owner[tq] ? fy : 0.0, T.owner[tq] ? fz : 0.0};
                if (add_fin) {
                    F[0] += bv.f[rb];
                    F[1] += bv.f[rb + N];
                    F[2] += bv.f[rb + 2 * N];
                }
                const uint8_t fb = bv.fixed[poff + (long long)b * N];
                const double mass = bv.mass[aoff];
                bv.f[rb] = F[0];
                bv.f[rb + N] = F[1];
                bv.f[rb + 2 * N] = F[2];
                bv.a[rb] = (fb & 1) ? 0.0 : F[0] / mass;
                bv.a[rb + N] = (fb & 2) ? 0.0 : F[1] / mass;
                bv.a[rb + 2 * N] = (fb & 4) ? 0.0 : F[2] / mass;
                bv.dens[poff + (long long)b * N] = DH[grp];
                Eb[b] = dE + EH[grp] - 0.5 * vs;  // bead part of the energy
            }
        }
        __syncthreads();
    }

    // ---- 3: classical pairs with the bead-averaged G (pass B) ----
    for (int a = lane; a < Ns; a += nthr)
        G0[a] += (double)(long long)Gacc[a] * MDT_F_ISCALE;  // G0 now holds the bead average
    __syncthreads();
    auto pair_b = [&](int k, int tk, double xk, double yk, double zk, double Gk, int e, bool far, double &fx,
                      double &fy, double &fz, double &ep) {
        const unsigned q = nbr[(size_t)k * cap + e];
        const int n = q & MDT_NBR_IDX_MASK, code = q >> MDT_NBR_IDX_BITS;
        if (far && !(tiny[k] | tiny[n])) return;
        const int tn = typ[n + 1];
        const double dx = (xk - px[n]) - T.shift[3 * code];
        const double dy = (yk - py[n]) - T.shift[3 * code + 1];
        const double dz = (zk - pz[n]) - T.shift[3 * code + 2];
        const double r2 = dx * dx + dy * dy + dz * dz;
        const double ri = mdt_rsqrt(r2);
        const double r = r2 * ri;
        if (r > cutr) return;
        const int ikn = tk * MDT_MAXT + tn, ink = tn * MDT_MAXT + tk;
        const double e1 = mdt_exp(acut * (r - rcut), T.exptab);
        const double th = mdt_rcp(1 + e1);
        const double rt1 = acut * e1 * th;
        const double fsn = th * mdt_exp(-T.eta2[tn] * (r - T.bs0[tn]), T.exptab);
        const double fvn = th * mdt_exp(-T.kdb[tn] * (r - T.bs0[tn]), T.exptab);
        double c;
        if (tn == tk) {  // one element: one set of pair constants (as in k_replica)
            c = T.csig[ikn] * ((T.etad[ikn] + rt1) * fsn) * (Gk + G0[n]) + T.wv[ikn] * ((T.kdb[tn] + rt1) * fvn);
            ep += 2.0 * T.wv[ikn] * fvn;
        } else {
            const double fsk = th * mdt_exp(-T.eta2[tk] * (r - T.bs0[tk]), T.exptab);
            const double fvk = th * mdt_exp(-T.kdb[tk] * (r - T.bs0[tk]), T.exptab);
            c = Gk * T.csig[ikn] * ((T.etad[ikn] + rt1) * fsn) + G0[n] * T.csig[ink] * ((T.etad[ink] + rt1) * fsk) +
                0.5 * (T.wv[ikn] * ((T.kdb[tn] + rt1) * fvn) + T.wv[ink] * ((T.kdb[tk] + rt1) * fvk));
            ep += T.wv[ikn] * fvn + T.wv[ink] * fvk;
        }
        const double crs = c * ri * MDT_F_SCALE;  // fixed-point units, as in k_replica
        const double gx = crs * dx, gy = crs * dy, gz = crs * dz;
        fx = fma(-crs, dx, fx);
        fy = fma(-crs, dy, fy);
        fz = fma(-crs, dz, fz);
        fx_add_scaled(&fxa[n], gx, &bad_local);
        fx_add_scaled(&fya[n], gy, &bad_local);
        fx_add_scaled(&fza[n], gz, &bad_local);
    };
    for (int k0 = 0; k0 < Ns; k0 += apb) {
        const int k = k0 + lane / TPA;
        const int sub = lane % TPA;
        const bool act = k < Ns;
        double fx = 0.0, fy = 0.0, fz = 0.0, ep = 0.0;
        if (act) {
            const int tk = typ[k + 1];
            const double xk = px[k], yk = py[k], zk = pz[k];
            const double Gk = G0[k];
            const int ck = cnt[k];
            for (int e = sub; e < ck; e += TPA) pair_b(k, tk, xk, yk, zk, Gk, e, false, fx, fy, fz, ep);
            if (anytiny)
                for (int e = cap - cntf[k] + sub; e < cap; e += TPA)
                    pair_b(k, tk, xk, yk, zk, Gk, e, true, fx, fy, fz, ep);
        }
        fx = group_sum<TPA>(fx);
        fy = group_sum<TPA>(fy);
        fz = group_sum<TPA>(fz);
        ep = group_sum<TPA>(ep);
        if (act && sub == 0) {
            fx_add_scaled(&fxa[k], fx, &bad_local);
            fx_add_scaled(&fya[k], fy, &bad_local);
            fx_add_scaled(&fza[k], fz, &bad_local);
            E0[k] -= 0.5 * ep;
        }
    }
    __syncthreads();

    // ---- outputs: classical atoms (bead 0), bead energies ----
    for (int a = lane; a < Ns; a += nthr) {
        const int i = a + 1;
        const int ta = typ[i];
        double F[3] = {(double)(long long)fxa[a] * MDT_F_ISCALE, (double)(long long)fya[a] * MDT_F_ISCALE,
                       (double)(long long)fza[a] * MDT_F_ISCALE};
        if (!T.owner[ta]) F[0] = F[1] = F[2] = 0.0;
        if (add_fin) {
            F[0] += bv.f[soff + i];
            F[1] += bv.f[soff + N + i];
            F[2] += bv.f[soff + 2 * N + i];
        }
        const uint8_t fb = bv.fixed[poff + i];
        const double mass = bv.mass[aoff + i];
        bv.f[soff + i] = F[0];
        bv.f[soff + N + i] = F[1];
        bv.f[soff + 2 * N + i] = F[2];
        bv.a[soff + i] = (fb & 1) ? 0.0 : F[0] / mass;
        bv.a[soff + N + i] = (fb & 2) ? 0.0 : F[1] / mass;
        bv.a[soff + 2 * N + i] = (fb & 4) ? 0.0 : F[2] / mass;
        if (T.owner[ta]) bv.dens[poff + i] = D0[a] + (double)(long long)Dacc[a] * MDT_F_ISCALE;
    }
    if (lane < 64) {
        double e = 0.0;
        for (int a = lane; a < Ns; a += 64) e += E0[a];
        for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
        if (lane == 0) red[0] = e;
    }
    __syncthreads();
    for (int b = lane; b < P; b += nthr) bv.epot[bv.traj_eoff[t] + b] = red[0] + Eb[b];
    if (bad_local) atomicOr(&bv.status[t], bad_local);
}

// ---------------------------------------------------------------------------
// Positions, velocities and forces between the device's layout [bead][component][atom]
// and the caller's (3, P, N): a workgroup takes a run of atoms with all their
// beads, contiguous in the caller's array and P * 3 runs in the device's, through
// LDS, so that both sides are read and written along cache lines.  Memory bound
// (4096 x 145 atoms: 14 MB, 12 us); done on the host it took 1.6 ms an array there and
// 2.5 ms for 64 x 385 atoms x 32 beads.  OUT: device to caller; in mixed bead mode a
// classical atom's bead 0 goes to every bead.
// ---------------------------------------------------------------------------
template <bool OUT>
__global__ void __launch_bounds__(256)
    k_relayout(const StateTile *__restrict__ tiles, const int *__restrict__ traj_N, const int *__restrict__ traj_P,
               const long long *__restrict__ traj_soff, int mixed, long long from, const double *__restrict__ src,
               double *__restrict__ dst) {
    __shared__ double s[3 * MDT_TILE];
    const StateTile w = tiles[blockIdx.x];
    const int N = traj_N[w.t], P3 = 3 * traj_P[w.t], n = P3 * w.na;
    const long long dev = traj_soff[w.t] + w.i0, ref = traj_soff[w.t] + (long long)P3 * w.i0 - from;
    const bool first = mixed && P3 > 3;
    if (OUT) {
        for (int q = threadIdx.x; q < n; q += 256) {
            const int bc = q / w.na, i = q - bc * w.na;
            s[i * P3 + bc] = src[dev + (long long)(first && w.i0 + i > 0 ? bc % 3 : bc) * N + i];
        }
        __syncthreads();
        for (int q = threadIdx.x; q < n; q += 256) dst[ref + q] = s[q];
    } else {
        for (int q = threadIdx.x; q < n; q += 256) s[q] = src[ref + q];
        __syncthreads();
        for (int q = threadIdx.x; q < n; q += 256) {
            const int bc = q / w.na, i = q - bc * w.na;
            dst[dev + (long long)bc * N + i] = s[i * P3 + bc];
        }
    }
}

// from: the first word of the caller's array that src (in) or dst (out) holds
hipError_t mdt_launch_relayout(bool out, int ntile, const StateTile *tiles, const BatchView &v, int mixed, long long from,
                               const double *src, double *dst, hipStream_t st) {
    if (out)
        hipLaunchKernelGGL((k_relayout<true>), dim3(ntile), dim3(256), 0, st, tiles, v.traj_N, v.traj_P, v.traj_soff,
                           mixed, from, src, dst);
    else
        hipLaunchKernelGGL((k_relayout<false>), dim3(ntile), dim3(256), 0, st, tiles, v.traj_N, v.traj_P, v.traj_soff,
                           mixed, from, src, dst);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// One universe's call (compute_emt, compute_nene): the batch arrays from one block of
// pinned host memory and the results into it, read and written over the host link
// by the kernels themselves.  A call is three launches and one wait (145 atoms x 16
// beads: 55 KB each way); with a copy or a fill per array and a wait after most of
// them it spent 170 of its 215 us on those.
//   in:  cell 9 | inverse 9 | r(3,P,N) | types (1-based, 4 bytes)
//   out: f(3,P,N) | epot(P) | dens(P,N) | status
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_call_in(const double *__restrict__ in, int N, int P, CallArrays a) {
    const int q = blockIdx.x * 256 + threadIdx.x, n3 = 3 * P * N;
    if (q < 9) a.cell[q] = in[q];
    if (q < 9) a.icell[q] = in[9 + q];
    if (q < n3) {
        const int i = q / (3 * P), bc = q - 3 * P * i;
        a.x[(long long)bc * N + i] = in[18 + q];
    }
    if (q < N) {
        a.type[q] = (uint8_t)(((const int32_t *)(in + 18 + n3))[q] - 1);
        a.mass[q] = 1.0;
    }
    if (q < P * N) a.fixed[q] = 0;
    if (q < P && a.nnkey) a.nnkey[q] = 0;  // new positions: kept lists are stale
    if (q == 0) *a.status = 0;
}

__global__ void __launch_bounds__(256) k_call_out(double *__restrict__ out, int N, int P, CallArrays a) {
    const int q = blockIdx.x * 256 + threadIdx.x, n3 = 3 * P * N;
    if (q < n3) {
        const int i = q / (3 * P), bc = q - 3 * P * i;
        out[q] = a.f[(long long)bc * N + i];
    }
    if (q < P) out[n3 + q] = a.epot[q];
    if (q < P * N) {
        const int i = q / P, b = q - P * i;
        out[n3 + P + q] = a.dens[(long long)b * N + i];
    }
    if (q == 0) *(int *)(out + n3 + P + P * N) = *a.status;
}

hipError_t mdt_launch_call(bool in, double *host, int N, int P, const CallArrays &a, hipStream_t st) {
    const dim3 g((3 * P * N + 255) / 256);
    if (in)
        hipLaunchKernelGGL(k_call_in, g, dim3(256), 0, st, host, N, P, a);
    else
        hipLaunchKernelGGL(k_call_out, g, dim3(256), 0, st, host, N, P, a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// host-side launchers (C++ linkage, used by mdt_api.hip)
// ---------------------------------------------------------------------------
// marks one slot in `period` invalid (launch-shape tuning)
__global__ void k_drop_lists(int2 *valid, int n, int period, int phase) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && i % period == phase) valid[i].x = 0;
}
hipError_t mdt_launch_drop_lists(int2 *valid, int n, int period, int phase, hipStream_t st) {
    hipLaunchKernelGGL(k_drop_lists, dim3((n + 256) / 256), dim3(256), 0, st, valid, n, period, phase);
    return hipGetLastError();
}

// k_replica's dynamic LDS, W2, W3, records, typ, tiny, and its HBM slot for a
// class: nrep replicas of up to N atoms, workgroups of `block` lanes, rows of up to
// cap entries; offsets in 4-byte words.  The stream's chunks of 64 pieces hold two
// entries a word, padded to their first piece's length, which is at most the
// last one's of the chunk before: 32 (longest + 1 a chunk) + half the entries -- 2
// more a chunk for lengths of 63 to 65, which are not told apart --, or, uncut, N
// rows of cap; and a row of slack.  The scanned rows go to LDS (scan < 0), if they fit
// into `lds`, where at most REP_FEW workgroups run, about two a CU, whose number
// LDS then does not limit, and where the rows serve one launch (once): they are
// then read from there, by the lanes that found them, without a cut.  The table
// holds N + block rows or pieces.
ReplicaLists mdt_replica_lists(int nrep, int N, int block, int cap, size_t lds, bool once) {
    ReplicaLists l;
    const long long chunks = (N + block) / 64 + 1;
    l.rows = 32 * (cap + 65 + 3 * chunks) + (N + 64LL) * (cap + 1) / 2 + 64;
    const size_t rows = 2 * (size_t)N * ((cap + 7) & ~7);
    l.smem = 58 * (size_t)N;
    const bool in_lds = (once || nrep <= REP_FEW) && l.smem + 8 + rows <= lds;
    if (in_lds && once) l.rows = 0;  // no stream
    l.chunk = l.rows + N + block;
    l.scan = (l.chunk + chunks + 3) & ~3LL;
    l.stride = l.scan;
    if (in_lds) {
        l.smem += 8 + rows;
        l.scan = -1;
    } else {
        l.stride += (long long)rows / 4;
    }
    return l;
}

template <bool M, int F, bool J>
static hipError_t launch_replica_t(dim3 g, dim3 blk, size_t smem, const EmtConst *ec, const BatchView &bv, int add_fin,
                                   hipStream_t st) {
    if (blk.x > 512)
        hipLaunchKernelGGL((k_replica<M, F, J, 1024>), g, blk, smem, st, ec, bv, add_fin);
    else
        hipLaunchKernelGGL((k_replica<M, F, J, 512>), g, blk, smem, st, ec, bv, add_fin);
    return hipGetLastError();
}

// calc_force on every replica; ec is a device pointer; tpa lanes per
// atom scan for the rows.  The judge (bv.judge_acc set) always runs the FP64
// arithmetic.
hipError_t mdt_launch_replica(int tpa, int nrep, int block, size_t smem, const EmtConst *ec, const BatchView &view,
                              int add_fin, hipStream_t st) {
    dim3 g(nrep), blk(block);
    BatchView bv = view;
    bv.tpa_shift = tpa == 8 ? 3 : tpa == 4 ? 2 : tpa == 2 ? 1 : 0;
    const bool m = bv.bulk < 0;
    if (bv.judge_acc)
        return m ? launch_replica_t<true, 0, true>(g, blk, smem, ec, bv, add_fin, st)
                 : launch_replica_t<false, 0, true>(g, blk, smem, ec, bv, add_fin, st);
    if (bv.precision == 1)
        return m ? launch_replica_t<true, 1, false>(g, blk, smem, ec, bv, add_fin, st)
                 : launch_replica_t<false, 1, false>(g, blk, smem, ec, bv, add_fin, st);
    if (bv.precision == 2)
        return m ? launch_replica_t<true, 2, false>(g, blk, smem, ec, bv, add_fin, st)
                 : launch_replica_t<false, 2, false>(g, blk, smem, ec, bv, add_fin, st);
    return m ? launch_replica_t<true, 0, false>(g, blk, smem, ec, bv, add_fin, st)
             : launch_replica_t<false, 0, false>(g, blk, smem, ec, bv, add_fin, st);
}

// LDS of k_mixed for trajectories of up to nmax atoms (one projectile) and
// pmax beads
size_t mdt_mixed_smem(int nmax, int pmax) {
    const size_t ns = (size_t)(nmax - 1), ngrp = MIX_BLOCK / MIX_G;
    return sizeof(double) * (12 * ns + 4 * (size_t)pmax + 3 * ngrp) +
           sizeof(uint16_t) * (2 * ns + ngrp + ngrp * MIX_CAPQ) + (size_t)nmax + ns + 16;
}

int mdt_mixed_block(void) { return MIX_BLOCK; }

// calc_force of the mixed-bead trajectories listed in bv.rep_list (ntraj of
// them); the classical atoms' owned half lists go to bv.nbr_global +
// list position x bv.nbr_stride
// block: MIX_BLOCK (512) or 1024 lanes
hipError_t mdt_launch_mixed(int tpa, int block, int ntraj, size_t smem, const EmtConst *ec, const PropConst *pc,
                            const BatchView &bv, int add_fin, hipStream_t st) {
    dim3 g(ntraj), blk(block);
    if (block == 1024) {
        switch (tpa) {
        case 2: hipLaunchKernelGGL((k_mixed<2, 1024>), g, blk, smem, st, ec, pc, bv, add_fin); break;
        case 4: hipLaunchKernelGGL((k_mixed<4, 1024>), g, blk, smem, st, ec, pc, bv, add_fin); break;
        case 8: hipLaunchKernelGGL((k_mixed<8, 1024>), g, blk, smem, st, ec, pc, bv, add_fin); break;
        default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    }
    if (block != MIX_BLOCK) return hipErrorInvalidValue;
    switch (tpa) {
    case 2: hipLaunchKernelGGL((k_mixed<2>), g, blk, smem, st, ec, pc, bv, add_fin); break;
    case 4: hipLaunchKernelGGL((k_mixed<4>), g, blk, smem, st, ec, pc, bv, add_fin); break;
    case 8: hipLaunchKernelGGL((k_mixed<8>), g, blk, smem, st, ec, pc, bv, add_fin); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// classical batches: every trajectory has P = 1 and at most `block` atoms,
// and no atom type uses PILE or Andersen (k_traj_classical)
hipError_t mdt_launch_traj_classical(int ntraj, const PropConst *pc, const BatchView &bv, const uint32_t *step_base,
                                     uint32_t step_prev, uint32_t step, int flags, int block, hipStream_t st,
                                     int t_base) {
    hipLaunchKernelGGL(k_traj_classical, dim3(ntraj), dim3(block), 0, st, pc, bv, step_base, step_prev, step, flags,
                       t_base);
    return hipGetLastError();
}

// the other batches, over the chunk table.  With observation the frozen
// trajectories are decided between propagate_2 and propagate_1; with COM
// removal (com_on) propagate_1 and the transforms are two launches.
hipError_t mdt_launch_prop(int ntraj, int maxP, const PropConst *pc, const BatchView &bv, const double *cjk,
                           const long long *cjk_off, const PropChunk *chunks, int nchunk, double *com, bool com_on,
                           const uint32_t *step_base, uint32_t step_prev, uint32_t step, int flags, hipStream_t st) {
    const size_t smem = maxP > 1 ? sizeof(double) * maxP * (maxP + 1) : 0;
    const dim3 g(((nchunk + 7) / 8) * 8), blk(256);
    if ((flags & 1) && bv.obs) {
        hipLaunchKernelGGL(k_prop, g, blk, smem, st, pc, bv, cjk, cjk_off, chunks, nchunk, com, step_base, step_prev,
                           step, 1);
        hipLaunchKernelGGL(k_observe, dim3(ntraj), blk, 0, st, pc, bv, step_base, step_prev);
        flags &= ~1;
    }
    if ((flags & 2) && com_on) flags |= 8;
    if (flags & 7)
        hipLaunchKernelGGL(k_prop, g, blk, smem, st, pc, bv, cjk, cjk_off, chunks, nchunk, com, step_base, step_prev,
                           step, flags);
    if (flags & 8)
        hipLaunchKernelGGL(k_com_ring, g, blk, smem, st, pc, bv, cjk, cjk_off, chunks, nchunk, com, flags);
    return hipGetLastError();
}

// the step counter of graph replays: one lane sets it (set != 0) or adds
// the chunk length
__global__ void k_advance(uint32_t *step_base, uint32_t n, int set) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *step_base = set ? n : *step_base + n;
}

hipError_t mdt_launch_advance(uint32_t *step_base, uint32_t n, int set, hipStream_t st) {
    hipLaunchKernelGGL(k_advance, dim3(1), dim3(64), 0, st, step_base, n, set);
    return hipGetLastError();
}
