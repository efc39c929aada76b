// ps_orbit.h -- the model rows (bright.c:14-126) of the J-free kernels by symmetry orbits of the facets,
// included by ps_fit2.h.
//
// The triangulated Gaussian image (trifac.c, period_search_BOINC.cpp:507-539) maps onto itself under
// rotations by 90 degrees about z and under inversion.  Its 8 nrows^2 facets fall into nrows^2 orbits of
// eight: the normals n_k = Rz(90k) (a, b, c), k = 0..3, and -n_k.  Two facts follow.
//  * Of n_k and -n_k at most one is turned to the observer, and mu of the other is -mu: four signed
//    evaluations of the scattering law serve all eight facets.
//  * A spherical harmonic takes the same value on all members up to sign and a swap of its cos/sin parts
//    ((-1)^l under inversion, a shift of m*90 degrees under rotation).  So the contraction
//    sum_f X_f Dsph_fk needs the representative's row only, applied to sums of the four signed X:
//    (l even: X, l odd: sign*X)  s = T0+T1+T2+T3 for m = 0 mod 4, r = T0-T1+T2-T3 for m = 2 mod 4 (one
//    multiply-add per coefficient and orbit), and d0 = T0-T2, d1 = T1-T3 for odd m (two).
// At Lmax = 6 an orbit takes 73 multiply-adds for the contraction instead of 8 x 49, and half the
// scattering evaluations.
//
// One lane owns one point: the orbit's constants (a, b, c and its row of 49) are the same for all lanes
// and are scalar operands of the multiply-adds, every sum over facets stays in the lane's registers, and
// nothing is reduced across lanes.  (FP64 MFMA and FP64 VALU have the same peak on gfx950 and share the
// issue slots, so the VALU form loses nothing.)  A pass of 128 rows is two groups of 64 points; the two
// waves of a group take alternate halves of the orbits and add their sums through the pass's LDS rows.
//
// What bounds it: FP64 issue.  Per orbit and 64 points 230 VALU instructions, 4 of them v_rcp_f64, replace the
// 8 x 2 x (73 VALU + 6 MFMA of 64 cycles) / 4 of the tile form (ps_fit2.h model_rows2): 920 cycles of issue
// instead of 2700.  Beside the other workgroup's wave on its SIMD a wave takes about 1650 cycles for them and
// 370 for the correction (42 % and 10 % of its time at 2400 points and 288 facets, 58 % and 13 % at 5000 and
// 512).  Measured when the form was made, 2560 fits of 50
// iterations: 2400 points and 288 facets 352 -> 207 ms, 5000 points and 512 facets 1006 -> 505 ms; with the
// steps since 178 and 484 ms (of these 189 -> 178 and 516 -> 484 by X's buffers on 16 bytes instead of 8
// past them).  Error of a Jacobian column against extended precision 3.8e-16 and 3.2e-16 rms of its largest
// entry (tile form 4.0e-16, 3.7e-16).
#pragma once

namespace psk {

// Coefficients of a layout for degree and order up to L, in the order the loop consumes them: even l
// (m = 0 mod 4, m = 2 mod 4, odd m), then odd l (m = 2 mod 4, m = 0 mod 4, odd m); within a class by m,
// then l; cos, then sin for m > 0.
constexpr int kOrbMaxL = 6;
constexpr int orb_ncoef(int L) { return (L + 1) * (L + 1); }

template <int L>
struct OrbLayout {
    static constexpr int N = orb_ncoef(L);
    int l[N] = {}, m[N] = {}, sn[N] = {};  // sn: 1 the sin part
    int neven = 0;                         // coefficients of even l (the first ones)
    constexpr OrbLayout() {
        int n = 0;
        for (int par = 0; par < 2; ++par) {
            for (int step = 0; step < 3; ++step) {
                const int cls = par == 0 ? step : (step == 0 ? 1 : step == 1 ? 0 : 2);  // 0: m%4==0, 1: m%4==2, 2: odd
                for (int mm = 0; mm <= L; ++mm) {
                    if ((mm % 2 ? 2 : mm % 4 ? 1 : 0) != cls) continue;
                    for (int ll = mm; ll <= L; ++ll) {
                        if (ll % 2 != par) continue;
                        for (int s = 0; s < (mm ? 2 : 1); ++s, ++n) {
                            l[n] = ll;
                            m[n] = mm;
                            sn[n] = s;
                        }
                    }
                }
            }
            if (par == 0) neven = n;
        }
    }
    // no cos/sin pair of odd m lies across position j (the loop's pieces of a row hold whole pairs)
    constexpr bool whole_at(int j) const { return j >= N || !(m[j] % 2 && sn[j]); }
};

constexpr int kOrbHead = 3;  // an orbit's row in the table: a, b, c, then the N coefficient values
constexpr int orb_stride(int L) { return (kOrbHead + orb_ncoef(L) + 3) & ~3; }

// Signs of T_k under the rotations, applied: the sums a coefficient class multiplies.
struct OrbSums {
    double s, r, d0, d1;
};

typedef double orb_d2 __attribute__((ext_vector_type(2)));

__device__ inline double orb_load(const double *p, int i) {  // a wave-uniform read through the scalar cache
    return reinterpret_cast<const __attribute__((address_space(4))) double *>(reinterpret_cast<unsigned long long>(p))[i];
}

__device__ inline unsigned hi_word(double x) { return unsigned(static_cast<unsigned long long>(__double_as_longlong(x)) >> 32); }
__device__ inline double flip_sign(double x, unsigned s) {  // x with its sign bit xor s (s = 0 or 1 << 31)
    const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(x));
    return __longlong_as_double(static_cast<long long>(b ^ (static_cast<unsigned long long>(s) << 32)));
}

// Correction of the folded contraction.  The tables of the eight members of an orbit differ from the
// symmetric ones by their own rounding, a few 1e-16 of a column's size, the same in every evaluation; left
// out, it steers the long fits away from those of the reference's tables (config3's 320 fits of 50
// iterations: 49 depart by more than 1e-9 in rms, against 33 for the reference's own FMA build).  The
// difference rows (member minus symmetric, exact) are contracted separately, sum_f X_f delta_fk: a term
// of 1e-16 of the result, so X and delta enter in bfloat16 (v_mfma_f32_32x32x16_bf16, 3 digits of the
// correction).  X of up to kSegOrbits orbits waits in the wave's share of the pass's row area; the
// MFMA's result tile (coefficient x point) turns into lane = point order with v_permlane32_swap.
constexpr int kSegOrbits = 14;                    // 14 KiB of X per wave: two waves fit a group's rows
constexpr int kXBytes = kSegOrbits * 64 * 16;
constexpr int orb_ctiles(int L) { return (orb_ncoef(L) + 31) / 32; }
typedef __bf16 orb_b8 __attribute__((ext_vector_type(8)));
typedef float orb_f16 __attribute__((ext_vector_type(16)));
typedef unsigned orb_u4 __attribute__((ext_vector_type(4)));

// The sums of one point over orbits: the N contraction sums (stream order), S = sum dbr/de, U = sum
// dbr/de0 and, with LS, the Lambert and Lommel-Seeliger sums.
template <int L, bool LS>
struct OrbAcc {
    static constexpr int N = orb_ncoef(L);
    double c[N];
    double S[3], U[3];
    double d1, d2;
    __device__ void clear() {
#pragma unroll
        for (int j = 0; j < N; ++j) c[j] = 0;
#pragma unroll
        for (int j = 0; j < 3; ++j) S[j] = U[j] = 0;
        d1 = d2 = 0;
    }
};

// Adds the orbits [o0, o1) to A; xl: the lane's place in the wave's buffer of X, 1 KiB per orbit.
template <int L, bool LS>
__device__ __forceinline__ void orbit_loop(const double *orb, int o0, int o1, const orb_d2 *tab, int zero_slot, double cls,
                                           const double e[3], const double e0[3], char *xl, OrbAcc<L, LS> &A) {
    constexpr OrbLayout<L> lay{};
    constexpr int N = orb_ncoef(L), ST = orb_stride(L);
    const char *tb = reinterpret_cast<const char *>(tab);
    const double *row = orb + size_t(o0) * ST;
    double a = orb_load(row, 0), b = orb_load(row, 1), c = orb_load(row, 2);
    // The orbit's row is read in three pieces so that at most two of them (64 scalar registers) are live.
    constexpr int C1 = N < 16 ? N : 16, C2 = N < 32 ? N : 32;
    static_assert(lay.whole_at(C1) && lay.whole_at(C2));
#pragma unroll 1
    for (int o = o0; o < o1; ++o, row += ST, xl += 1024) {
        double D[N];
#pragma unroll
        for (int j = 0; j < C2; ++j) D[j] = orb_load(row, kOrbHead + j);
        __builtin_amdgcn_sched_barrier(0);
        double mu[4], m0[4];
        {
            const double u = e[0] * a + e[1] * b, v = e[1] * a - e[0] * b, w = e[2] * c;
            const double u0 = e0[0] * a + e0[1] * b, v0 = e0[1] * a - e0[0] * b, w0 = e0[2] * c;
            mu[0] = w + u; mu[1] = w + v; mu[2] = w - u; mu[3] = w - v;
            m0[0] = w0 + u0; m0[1] = w0 + v0; m0[2] = w0 - u0; m0[3] = w0 - v0;
        }
        // the member of each pair that faces the observer, and its entry (Area*cl, Area*cls, negated for
        // the member -n_k): a point that does not see it lit takes a zero entry instead, so that every
        // term below vanishes without further tests
        unsigned sg[4];
        orb_d2 ar[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const unsigned h = hi_word(mu[k]);
            sg[k] = h & 0x80000000u;
            m0[k] = flip_sign(m0[k], sg[k]);
            mu[k] = fabs(mu[k]);
            const bool lit = mu[k] > kTiny && m0[k] > kTiny;
            const int off = lit ? int((h >> 31) << 4) + o * 128 : zero_slot;
            ar[k] = *reinterpret_cast<const orb_d2 *>(tb + off + 32 * k);
        }
        double rd[4], dn[4], er[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) dn[k] = fmax(mu[k] + m0[k], kTiny);
#pragma unroll
        for (int k = 0; k < 4; ++k) rd[k] = __builtin_amdgcn_rcp(dn[k]);
        // one step of third order, r + r (e + e^2) with e = 1 - d r: v_rcp_f64 is good to 2^-24, so the
        // error left is the last rounding's
#pragma unroll
        for (int k = 0; k < 4; ++k) er[k] = fma(-dn[k], rd[k], 1.0);
#pragma unroll
        for (int k = 0; k < 4; ++k) er[k] = fma(er[k], er[k], er[k]);
#pragma unroll
        for (int k = 0; k < 4; ++k) rd[k] = fma(rd[k], er[k], rd[k]);
        double X[4], Y[4], vs[4], vu[4];  // X = sign * Area*s, Y = Area*s
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const double mm = mu[k] * m0[k];
            if constexpr (LS) {
                // the entry holds (Area*cl, Area) here: d1 = sum Area*mm, d2 = sum Area*mm/(mu + mu0)
                const double am = fabs(mm * ar[k][1]);
                A.d1 += am;
                A.d2 += am * rd[k];
                ar[k][1] *= cls;
            }
            const double Ac = ar[k][0], t = ar[k][1] * rd[k];
            X[k] = mm * (t + Ac);
            const double h2 = t * rd[k];
            vs[k] = m0[k] * fma(h2, m0[k], Ac);
            vu[k] = mu[k] * fma(h2, mu[k], Ac);
            Y[k] = flip_sign(X[k], sg[k]);
        }
        {
            // X in bfloat16 at its member's place: the low half for n_k, the high half for -n_k
            orb_u4 w;
#pragma unroll
            for (int k = 0; k < 4; ++k) w[k] = (__float_as_uint(float(Y[k])) >> 16) << (sg[k] >> 27);
            *reinterpret_cast<orb_u4 *>(xl) = w;
        }
        {
            const double p = vs[0] - vs[2], q = vs[1] - vs[3], z = (vs[0] + vs[2]) + (vs[1] + vs[3]);
            A.S[0] = fma(-b, q, fma(a, p, A.S[0]));
            A.S[1] = fma(a, q, fma(b, p, A.S[1]));
            A.S[2] = fma(c, z, A.S[2]);
        }
        {
            const double p = vu[0] - vu[2], q = vu[1] - vu[3], z = (vu[0] + vu[2]) + (vu[1] + vu[3]);
            A.U[0] = fma(-b, q, fma(a, p, A.U[0]));
            A.U[1] = fma(a, q, fma(b, p, A.U[1]));
            A.U[2] = fma(c, z, A.U[2]);
        }
        OrbSums ev, od;
        {
            const double p = Y[0] + Y[2], q = Y[1] + Y[3];
            ev = {p + q, p - q, Y[0] - Y[2], Y[1] - Y[3]};
        }
        {
            const double p = X[0] + X[2], q = X[1] + X[3];
            od = {p + q, p - q, X[0] - X[2], X[1] - X[3]};
        }
        auto take = [&](int j0, int j1) {
#pragma unroll
            for (int j = 0; j < N; ++j) {
                if (j < j0 || j >= j1) continue;
                const OrbSums &t = j < lay.neven ? ev : od;
                const int m4 = lay.m[j] & 3;
                if (m4 == 0)
                    A.c[j] = fma(t.s, D[j], A.c[j]);
                else if (m4 == 2)
                    A.c[j] = fma(t.r, D[j], A.c[j]);
                else {
                    // cos part: d0 cos - sigma d1 sin; sin part: d0 sin + sigma d1 cos, sigma = sin(m pi/2)
                    const int o_cs = lay.sn[j] ? j - 1 : j + 1;
                    const bool neg = (m4 == 1) == (lay.sn[j] == 0);
                    A.c[j] = fma(t.d0, D[j], A.c[j]);
                    A.c[j] = fma(neg ? -t.d1 : t.d1, D[o_cs], A.c[j]);
                }
            }
        };
        take(0, C1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = C2; j < N; ++j) D[j] = orb_load(row, kOrbHead + j);
        a = orb_load(row, ST);  // the next orbit's normal (the table has one orbit more than the mesh)
        b = orb_load(row, ST + 1);
        c = orb_load(row, ST + 2);
        __builtin_amdgcn_sched_barrier(0);
        take(C1, C2);
        __builtin_amdgcn_sched_barrier(0);
        take(C2, N);
    }
}

// Adds the correction of cnt orbits from orbit o0 on (their X in the wave's buffer xw) to A.  corr: per
// 32 stream positions and orbit, 32 x 8 bfloat16 (position x member).
template <int L, bool LS>
__device__ __forceinline__ void orbit_correct(const orb_u4 *corr, int norb, int o0, int cnt, char *xw, OrbAcc<L, LS> &A) {
    constexpr int N = orb_ncoef(L);
    const int lane = threadIdx.x & 63, hi = lane >> 5, lo = lane & 31;
    // an odd orbit at the end: zeros beside it (the table has a zero orbit past the last one)
    if (cnt & 1) *reinterpret_cast<orb_u4 *>(xw + cnt * 1024 + lane * 16) = orb_u4{0, 0, 0, 0};
    wave_lds_fence();  // X of all lanes, before any lane reads another's
    const char *xr = xw + hi * 1024 + lo * 16;
#pragma unroll
    for (int t = 0; t < orb_ctiles(L); ++t) {
        const orb_u4 *cp = corr + (size_t(t) * (norb + 1) + o0 + hi) * 32 + lo;
        orb_f16 a0, a1;
#pragma unroll
        for (int r = 0; r < 16; ++r) a0[r] = a1[r] = 0;
        for (int k = 0; k < cnt; k += 2) {
            const orb_b8 d = __builtin_bit_cast(orb_b8, reinterpret_cast<const __attribute__((address_space(1))) orb_u4 *>(
                                                            reinterpret_cast<unsigned long long>(cp))[k * 32]);
            const orb_b8 x0 = *reinterpret_cast<const orb_b8 *>(xr + k * 1024);
            const orb_b8 x1 = *reinterpret_cast<const orb_b8 *>(xr + k * 1024 + 512);
            a0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(d, x0, a0, 0, 0, 0);
            a1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(d, x1, a1, 0, 0, 0);
        }
        // register r of lane l: position 8 (r / 4) + 4 (l / 32) + r % 4 of point l % 32 (a1: of point 32 + l % 32)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int j = 32 * t + 8 * (r / 4) + r % 4;
            if (j >= N) continue;
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(a0[r]), __float_as_uint(a1[r]), false, false);
            if (j > 0) A.c[j] += double(__uint_as_float(sw[0]));  // position 0 (c00) has no correction
            if (j + 4 < N) A.c[j + 4] += double(__uint_as_float(sw[1]));
        }
    }
    wave_lds_fence();  // the next piece's X overwrites what other lanes have read here
}

}  // namespace psk
