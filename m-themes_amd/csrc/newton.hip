// newton.hip -- per-voxel viscoplastic stress update (src/evolution.c:2-310)
// with the power-law rate of src/constitutive.c:5-67, in FP64, one voxel per
// lane, plus the block partial sums of the convergence norms and the stress
// averages that get_smacro needs (src/evolution.c:1415-1437, 473-497).
//
// The arithmetic follows the reference's: the same equations in the same
// basis, the NR_MODIFIED backtracking line search with its constants, branches
// and the TOLX rejection of small steps.  Rewritten, with the same
// mathematics:
//   * the Newton step: J step = -R with J = I + C0 (S + dt D) is solved as
//     K step = -S0 R with the symmetric positive definite K = S0 + S + dt D
//     (S0 = C0^-1) by an L D L^T factorisation -- the reference forms
//     LU_inv_66(J) with pivoting and multiplies; the slope of the merit
//     function along that step is -|R|^2;
//   * S = LU_inv_66(C_gr) is a per-orientation constant (read from a table,
//     upper triangle), and d(edot)/d(sigma) is symmetric, so only upper
//     triangles are formed;
//   * rates in the crystal axes, where the Schmid tensors are constants of the
//     phase (0, 1 and 2 of a scaled basis for the cubic family, scalar
//     registers otherwise), between two 5x5 rotations of the voxel;
//   * |x|^n by repeated squaring for integral n, 1/CRSS multiplied instead of
//     divided, fused multiply-adds.
// A K that is not positive definite returns status 35, the reference's
// singular-LU exit; one that only its rounded sums made so is factored
// another way first (rank1_solve).
//
// What bounds it: FP64 vector issue, two waves per SIMD (256 registers each).
// One voxel per lane; K0 = S0 + S, the rotation, the stress and the residual
// stay in registers (116 of them), what is read once per evaluation (1/CRSS,
// d, the tangent's weights) in LDS columns of the lane (15 KB per wave), the
// constants arrive by scalar loads.  The 12 Schmid tensors in sample axes, as
// an LDS slab of 30 KB per wave, held the kernel at one wave per SIMD, with
// 5 LDS reads per system and evaluation, and every iteration evaluated the
// accepted trial a second time.  Per launch, that form, this one with the
// Schmid constants from scalar registers, and this one with the sums of the
// cubic family: 583, 240 and 219 us at 128^3 with 2 % pores (iterations 1-200
// of an increment, n = 10), 81, 40 and 33 us at 64^3, 118, 74 and 64 us at 64^3
// under the dislocation-density law (a first increment; 111 us in its 16th, 94
// with the rates left out for the lanes that wait), 110, 37 and 33 us at 24^3 with a
// non-integral exponent (pow() of each system once per evaluation instead of
// twice, and one evaluation in three less).
#include <hip/hip_ext.h>

#include "linesearch.h"
#include "newton_common.h"

namespace {

// x^M for a compile-time M: the products of ipow with the bit tests folded
// (x^9 is three squarings and one product)
template <int M> __device__ __forceinline__ double ipowc(double x)
{
    double r = 1.0, b = x;
#pragma unroll
    for (int m = M; m; m >>= 1) {
        if (m & 1) r *= b;
        if (m > 1) b *= b;
    }
    return r;
}

// 1/d for a normal d: the hardware estimate refined by two Newton steps
// y += y (1 - d y) (the relative error e becomes e^2 per step)
__device__ __forceinline__ double rcp_refined(double d)
{
    double y = __builtin_amdgcn_rcp(d);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const double e = fma(-d, y, 1.0);
        y = fma(y, e, y);
    }
    return y;
}

// 1/c for a CRSS: 0 where it is infinite (the system is off), as the reference's
// division gives; the estimate's refinement alone is NaN there (inf 0).
__device__ __forceinline__ double rcp_crss(double c)
{
    return __builtin_amdgcn_div_fixup(rcp_refined(c), c, 1.0);
}

constexpr int NB_THREADS = 64; // one wave per block: the LDS columns are wave-private

// The kernel's NewtonParams (its first argument) in the kernel-argument
// segment: wave-uniform reads from it become scalar loads.  fresh() hides the
// address from the optimiser and ties it to a value the arithmetic before it
// produces, so that a block of constants is loaded about where it is used:
// hoisted they would not fit the scalar registers, and each use of a spilled
// one costs two lane reads.
typedef const __attribute__((address_space(4))) double *cdouble;

__device__ __forceinline__ cdouble params_at(size_t byte)
{
    return (cdouble)((const __attribute__((address_space(4))) char *)__builtin_amdgcn_kernarg_segment_ptr() + byte);
}

__device__ __forceinline__ cdouble fresh(cdouble p, const double &after)
{
    __asm__ volatile("" : "+s"(p) : "v"(after) : "memory");
    return p;
}

// the same after every one of n accumulators has been brought up to date (a
// sum left for later would keep its constants in scalar registers)
template <int N> __device__ __forceinline__ cdouble fresh_after(cdouble p, const double (&a)[N])
{
#pragma unroll
    for (int i = 0; i < N; i++) __asm__ volatile("" ::"v"(a[i]));
    return fresh(p, a[0]);
}

// n Schmid constants (5 per system) from m
template <int N> struct Consts {
    double c[N];
};
template <int N> __device__ __forceinline__ Consts<N> load_consts(cdouble m)
{
    Consts<N> o;
#pragma unroll
    for (int i = 0; i < N; i++) o.c[i] = m[i];
    return o;
}

// x^m of a wave-uniform or compile-time exponent, as the rate law needs it
template <int RM, int NE> __device__ __forceinline__ double rate_power(double a, int intn, double nrs)
{
    if (RM == RM_FAST) return NE > 0 ? ipowc<(NE > 0 ? NE - 1 : 0)>(a) : ipow5(a, intn - 1);
    if (RM == RM_LOOP) return ipow(a, intn - 1);
    return pow(a, nrs - 1.);
}

// The slip systems are handled SYS_GROUP at a time: their Schmid constants
// come in by scalar loads (5 doubles each) ahead of the group's arithmetic.
constexpr int SYS_GROUP = 2;

// StrainRate_eval (src/constitutive.c:5-67) at the stress s: edot (sample
// axes).  Resolved shears and rates are formed in the crystal axes, where the
// Schmid tensors are constants of the phase: Q (5x5, rotation of deviators
// crystal -> sample, row-major) takes the stress in and the rate out.  The
// derivative of each system's rate in its resolved shear, times dt, goes to
// the lane's LDS column w (tangent() reads it if a Newton step follows).
// it: LDS columns of 1/CRSS, forward then backward (RM_DISL: the passing
// stress, then 1/(tau_0 + tau_cut)).  GD: the slip rates are written.
//
// CUBIC: the phase's systems are the twelve of {111}<110> (or {110}<111>, whose
// symmetric Schmid tensors are the same) in any order and sign.  In the basis
// that cubic_basis() scales Q to, the resolved shears of the four systems of a
// cube axis are b + u + v, b - u - v, b + u - v and b - u + v, b one of R - P,
// R + P and 2 P and u, v two of the shears: 21 additions instead of 60 fused
// multiply-adds, 27 for the rate's five components and 40 instead of 240
// operations for the tangent, and no constants to load.  The LDS columns hold
// the systems in that order (P.cub_sys: the phase's own index of each).
template <int RM, bool CSYM, bool GD, int NE, bool CUBIC>
__device__ __forceinline__ void rates(const NewtonParams &P, int p, const double *it, double *w,
                                      const double *g0c, long long N, const double Q[25],
                                      const double s[6], double ed[5], double *gd, bool keep)
{
    const int ns = RM == RM_FAST || RM == RM_DISL ? EVPGPU_NSYSMX : P.nsys[p];
    const int intn = P.int_n[p];
    const double g0 = P.gam0[p][0], ndt = P.nrs[p][0] * P.dt;
    // the rate at the resolved shear r of system k (LDS columns in k's order)
    auto slip = [&](int k, double r) {
        const int sy = CUBIC ? P.cub_sys[p][k] : k; // the phase's index of it
        double g, d; // the rate and dt times its derivative in the resolved shear
        if (RM == RM_DISL) {
            // gam = gam_o sinh((|rss| - tau_pass)/(tau_0 + tau_cut)) sign(rss)
            // above the passing stress, 0 below (FORWARD_PLUS_BACKWARD)
            const double a = fabs(r), tp = it[k * NB_THREADS];
            const double itc = it[(EVPGPU_NSYSMX + k) * NB_THREADS];
            const double g0k = g0c[sy * N];
            g = d = 0.0;
            // (only for the lanes at work: a wave that waits for a few lanes'
            // line searches then skips the systems below their passing stress)
            if (keep && a > tp) {
                const double x = (a - tp) * itc;
                // sinh and cosh from one expm1: with m = e^x - 1 and
                // q = e^-x, sinh x = m (1 + q) / 2 (no cancellation at
                // small x) and cosh x = (1 + m + q) / 2
                const double em = expm1(x), q = rcp_refined(1.0 + em);
                g = copysign(g0k * (0.5 * em * (1.0 + q)), r);
                d = g0k * (0.5 * ((1.0 + em) + q)) * itc * P.dt;
            }
        } else {
            const double itau = CSYM ? it[k * NB_THREADS] : it[((r < 0 ? EVPGPU_NSYSMX : 0) + k) * NB_THREADS];
            const double x = r * itau, a = fabs(x);
            const double p1 = (RM == RM_FAST ? g0 : P.gam0[p][sy]) * rate_power<RM, NE>(a, intn, P.nrs[p][sy]);
            g = p1 * x;
            // n < 1: |x|^(n-1) has no value at x = 0, |x|^n has
            if (RM == RM_POW && P.nrs[p][sy] < 1.0)
                g = copysign(P.gam0[p][sy] * pow(a, P.nrs[p][sy]), x);
            d = (p1 * itau) * (RM == RM_FAST ? ndt : P.nrs[p][sy] * P.dt);
        }
        if (GD && keep) {
            gd[sy * N] = CUBIC && P.cub_neg[p][k] ? -g : g;
        }
        if (RM != RM_DISL || keep) w[k * NB_THREADS] = d;
        return g;
    };
    double sc[5], e[5];
#pragma unroll
    for (int j = 0; j < 5; j++) {
        double a = Q[j] * s[0];
#pragma unroll
        for (int i = 1; i < 5; i++) a = fma(Q[5 * i + j], s[i], a);
        sc[j] = a;
        e[j] = 0.0;
    }
    if (CUBIC) {
        // (sums of products: left to the compiler, some would be contracted
        // and some not, another choice in each variant of the kernel)
#pragma clang fp contract(off)
        // (the columns are read here each time: hoisted they would spill)
        __asm__ volatile("" ::: "memory");
        const double b[3] = {sc[1] - sc[0], sc[1] + sc[0], 2.0 * sc[0]};
        double G[3], U[3], V[3]; // per axis: sum of the rates, of the rates times the signs of u and v
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const double u = sc[CUB_U[a]], v = sc[CUB_V[a]], pl = u + v, mi = u - v;
            const double g0 = slip(4 * a, b[a] + pl), g1 = slip(4 * a + 1, b[a] - pl);
            const double g2 = slip(4 * a + 2, b[a] + mi), g3 = slip(4 * a + 3, b[a] - mi);
            const double x = g0 - g1, y = g2 - g3;
            G[a] = (g0 + g1) + (g2 + g3);
            U[a] = x + y;
            V[a] = x - y;
        }
        e[0] = fma(2.0, G[2], G[1] - G[0]);
        e[1] = G[0] + G[1];
        e[2] = V[1] + V[2];
        e[3] = U[0] + U[2];
        e[4] = V[0] + U[1];
    } else {
        cdouble mx = params_at(offsetof(NewtonParams, mx)) + p * (EVPGPU_NSYSMX * 5);
        Consts<5 * SYS_GROUP> next = load_consts<5 * SYS_GROUP>(fresh(mx, s[0]));
#pragma unroll
        for (int k0 = 0; k0 < EVPGPU_NSYSMX; k0 += SYS_GROUP) {
            const Consts<5 * SYS_GROUP> m = next;
            if (k0 + SYS_GROUP < EVPGPU_NSYSMX)
                next = load_consts<5 * SYS_GROUP>(fresh_after(mx, e) + 5 * (k0 + SYS_GROUP));
#pragma unroll
            for (int k = k0; k < k0 + SYS_GROUP; k++) {
                if (k >= ns) break;
                const double *mk = m.c + 5 * (k - k0);
                const double m0 = mk[0], m1 = mk[1], m2 = mk[2], m3 = mk[3], m4 = mk[4];
                double r = m0 * sc[0];
                r = fma(m1, sc[1], r);
                r = fma(m2, sc[2], r);
                r = fma(m3, sc[3], r);
                r = fma(m4, sc[4], r);
                const double g = slip(k, r);
                e[0] = fma(m0, g, e[0]);
                e[1] = fma(m1, g, e[1]);
                e[2] = fma(m2, g, e[2]);
                e[3] = fma(m3, g, e[3]);
                e[4] = fma(m4, g, e[4]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 5; i++) {
        double a = Q[5 * i] * e[0];
#pragma unroll
        for (int j = 1; j < 5; j++) a = fma(Q[5 * i + j], e[j], a);
        ed[i] = a;
    }
}

// K = K0 + dt d(edot)/d(sigma) (packed upper triangle) from the weights the
// last rates() left: D' = sum_k w_k m_k m_k^T in crystal axes, then Q D' Q^T.
template <bool CUBIC>
__device__ __forceinline__ void tangent(int ns, int p, const double *w, const double Q[25],
                                        const double K0[21], double K[21])
{
    double D[15]; // upper triangle, row by row
    if (CUBIC) {
        // per axis: the sum of the weights, and of the weights times the signs
        // of u, of v and of u v
        __asm__ volatile("" ::: "memory");
        double W[3], U[3], V[3], C[3];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            const double w0 = w[4 * a * NB_THREADS], w1 = w[(4 * a + 1) * NB_THREADS];
            const double w2 = w[(4 * a + 2) * NB_THREADS], w3 = w[(4 * a + 3) * NB_THREADS];
            const double pl = w0 + w1, mi = w2 + w3, x = w0 - w1, y = w2 - w3;
            W[a] = pl + mi;
            C[a] = pl - mi;
            U[a] = x + y;
            V[a] = x - y;
        }
        // the columns P R 12 02 01; axis 0 (-1 1 0 u v), 1 (1 1 v 0 u), 2 (2 0 v u 0)
        D[0] = fma(4.0, W[2], W[0] + W[1]);
        D[1] = W[1] - W[0];
        D[2] = fma(2.0, V[2], V[1]);
        D[3] = fma(2.0, U[2], -U[0]);
        D[4] = U[1] - V[0];
        D[5] = W[0] + W[1];
        D[6] = V[1];
        D[7] = U[0];
        D[8] = V[0] + U[1];
        D[9] = W[1] + W[2];
        D[10] = C[2];
        D[11] = C[1];
        D[12] = W[0] + W[2];
        D[13] = C[0];
        D[14] = W[0] + W[1];
    } else {
#pragma unroll
        for (int i = 0; i < 15; i++) D[i] = 0.0;
        cdouble mx = params_at(offsetof(NewtonParams, mx)) + p * (EVPGPU_NSYSMX * 5);
        Consts<5 * SYS_GROUP> next = load_consts<5 * SYS_GROUP>(fresh(mx, K0[0]));
#pragma unroll
        for (int k0 = 0; k0 < EVPGPU_NSYSMX; k0 += SYS_GROUP) {
            const Consts<5 * SYS_GROUP> mc = next;
            if (k0 + SYS_GROUP < EVPGPU_NSYSMX)
                next = load_consts<5 * SYS_GROUP>(fresh_after(mx, D) + 5 * (k0 + SYS_GROUP));
#pragma unroll
            for (int k = k0; k < k0 + SYS_GROUP; k++) {
                if (k >= ns) break;
                const double *m = mc.c - 5 * k0;
                const double wk = w[k * NB_THREADS];
                int c = 0;
#pragma unroll
                for (int i = 0; i < 5; i++) {
                    const double a = wk * m[5 * k + i];
#pragma unroll
                    for (int j = i; j < 5; j++, c++) D[c] = fma(a, m[5 * k + j], D[c]);
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 5; i++) {
        double t[5]; // row i of Q D'
#pragma unroll
        for (int j = 0; j < 5; j++) {
            double a = 0.0;
#pragma unroll
            for (int q = 0; q < 5; q++) {
                const int lo = q < j ? q : j, hi = q < j ? j : q;
                const double d = D[lo * 5 - lo * (lo - 1) / 2 + (hi - lo)];
                a = q == 0 ? Q[5 * i] * d : fma(Q[5 * i + q], d, a);
            }
            t[j] = a;
        }
#pragma unroll
        for (int j = i; j < 5; j++) {
            double a = K0[PK(i, j)];
#pragma unroll
            for (int q = 0; q < 5; q++) a = fma(t[q], Q[5 * j + q], a);
            K[PK(i, j)] = a;
        }
        K[PK(i, 5)] = K0[PK(i, 5)];
    }
    K[PK(5, 5)] = K0[PK(5, 5)];
}

// L D L^T of the packed symmetric 6x6 k (in place) and the solve k x = b (b
// overwritten).  Returns false if k is not positive definite.
__device__ __forceinline__ bool ldl6_solve(double k[21], double b[6])
{
    double inv[6];
    bool pd = true;
#pragma unroll
    for (int j = 0; j < 6; j++) {
        // column j of L scaled by its pivot stays in k; the update of the
        // columns after it takes L_ij from k_ij inv_j
        const double d = k[PK(j, j)];
        pd = pd && d > 0.0;
        inv[j] = rcp_refined(d);
#pragma unroll
        for (int i = j + 1; i < 6; i++) {
            const double l = k[PK(j, i)] * inv[j];
#pragma unroll
            for (int q = i; q < 6; q++) k[PK(i, q)] = fma(-l, k[PK(j, q)], k[PK(i, q)]);
            b[i] = fma(-l, b[j], b[i]);
        }
    }
#pragma unroll
    for (int i = 5; i >= 0; i--) {
        double s = b[i];
#pragma unroll
        for (int q = i + 1; q < 6; q++) s = fma(-k[PK(i, q)], b[q], s);
        b[i] = s * inv[i];
    }
    return pd;
}

// (K0 + sum_k w_k m_k m_k^T) x = b (b overwritten) by rank-one updates of K0's
// L D L^T (Gill, Golub, Murray and Saunders 1974, method C1), the Schmid
// vectors m_k in sample axes and the weights w those of tangent().  Every update
// raises the pivots, so the factors are positive definite wherever K0 is.
// The sums of tangent() round to 1e-16 of the largest weight.  The weights go as
// |x|^(n-1), and where that leaves fewer than five independent systems within
// 1e16 of the largest, the small pivots can round to below 0: with n of 45 and
// more, in a first iteration next to a pore, some voxels of 1e5 (none up to
// n = 40, at any overstress tried).  Taken there only: 12 updates of dependent
// operations.  (Registers held for it: 1 % of an iteration at n = 33, 0.4 % at
// n = 12.5 with unequal CRSS.)
__device__ __forceinline__ bool rank1_solve(const NewtonParams &P, int p, int ns, const double *w,
                                            const double Q[25], const double K0[21], double b[6])
{
    double k[21]; // D on the diagonal, L (unit) above it, transposed
    bool pd = true;
#pragma unroll
    for (int i = 0; i < 21; i++) k[i] = K0[i];
#pragma unroll
    for (int j = 0; j < 6; j++) {
        pd = pd && k[PK(j, j)] > 0.0;
        const double inv = rcp_refined(k[PK(j, j)]);
#pragma unroll
        for (int i = j + 1; i < 6; i++) {
            const double l = k[PK(j, i)] * inv;
#pragma unroll
            for (int q = i; q < 6; q++) k[PK(i, q)] = fma(-l, k[PK(j, q)], k[PK(i, q)]);
        }
#pragma unroll
        for (int i = j + 1; i < 6; i++) k[PK(j, i)] *= inv;
    }
#pragma unroll 1
    for (int s = 0; s < ns; s++) {
        const double *m = P.mx[p][s];
        double a = w[s * NB_THREADS], z[6];
#pragma unroll
        for (int i = 0; i < 5; i++) {
            z[i] = Q[5 * i] * m[0];
#pragma unroll
            for (int j = 1; j < 5; j++) z[i] = fma(Q[5 * i + j], m[j], z[i]);
        }
        z[5] = 0.0;
#pragma unroll
        for (int j = 0; j < 6; j++) {
            const double d = k[PK(j, j)], pj = z[j], dn = fma(a * pj, pj, d), inv = rcp_refined(dn);
            const double be = a * pj * inv;
            a *= d * inv;
            k[PK(j, j)] = dn;
#pragma unroll
            for (int r = j + 1; r < 6; r++) {
                z[r] = fma(-pj, k[PK(j, r)], z[r]);
                k[PK(j, r)] = fma(be, z[r], k[PK(j, r)]);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 6; j++) {
        pd = pd && k[PK(j, j)] > 0.0; // (not where a weight is not a number)
#pragma unroll
        for (int i = j + 1; i < 6; i++) b[i] = fma(-k[PK(j, i)], b[j], b[i]);
    }
#pragma unroll
    for (int i = 5; i >= 0; i--) {
        b[i] *= rcp_refined(k[PK(i, i)]);
#pragma unroll
        for (int q = i + 1; q < 6; q++) b[i] = fma(-k[PK(i, q)], b[q], b[i]);
    }
    return pd;
}

// y = A x for a packed symmetric 6x6 A of NewtonParams, added to y
__device__ __forceinline__ void sym6_mul_add(cdouble A, const double x[6], double y[6])
{
#pragma unroll
    for (int i = 0; i < 6; i++)
#pragma unroll
        for (int j = 0; j < 6; j++) y[i] = fma(A[PK(i, j)], x[j], y[i]);
}

// r = K0 s + dt edot + d (d: LDS columns)
__device__ __forceinline__ void scaled_residual(double dt, const double K0[21], const double *d,
                                                const double s[6], const double ed[5], double r[6])
{
#pragma unroll
    for (int i = 0; i < 6; i++) {
        double a = i < 5 ? fma(ed[i], dt, d[i * NB_THREADS]) : d[i * NB_THREADS];
#pragma unroll
        for (int j = 0; j < 6; j++) a = fma(K0[PK(i, j)], s[j], a);
        r[i] = a;
    }
}

__device__ __forceinline__ double norm2(const double v[6])
{
    double a = v[0] * v[0];
#pragma unroll
    for (int i = 1; i < 6; i++) a = fma(v[i], v[i], a);
    return a;
}

// The rotation of deviators, crystal -> sample, for the orientation T (3x3,
// row-major): column j of Q (5x5, row-major) is the 5-vector of T B_j T^T, from
// the products of T's columns.
__device__ __forceinline__ void rotation5(const double T[9], double Q[25])
{
    double dg[3][5]; // sqrt 2 times the 5-vectors of c_a c_a^T
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const double x = T[a], y = T[3 + a], z = T[6 + a];
        const double xx = x * x, yy = y * y, zz = z * z;
        dg[a][0] = yy - xx;
        dg[a][1] = (2.0 * zz - xx - yy) * RSQ3;
        dg[a][2] = 2.0 * (y * z);
        dg[a][3] = 2.0 * (x * z);
        dg[a][4] = 2.0 * (x * y);
    }
    // B_0 = (e1e1 - e0e0)/sqrt 2, B_1 = (2 e2e2 - e0e0 - e1e1)/sqrt 6
#pragma unroll
    for (int i = 0; i < 5; i++) {
        Q[5 * i] = 0.5 * (dg[1][i] - dg[0][i]);
        Q[5 * i + 1] = (0.5 * RSQ3) * (2.0 * dg[2][i] - dg[0][i] - dg[1][i]);
    }
    // B_2, B_3, B_4: sym(e1e2), sym(e0e2), sym(e0e1) times sqrt 2
    const int ca[3] = {1, 0, 0}, cb[3] = {2, 2, 1};
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const double x0 = T[ca[q]], y0 = T[3 + ca[q]], z0 = T[6 + ca[q]];
        const double x1 = T[cb[q]], y1 = T[3 + cb[q]], z1 = T[6 + cb[q]];
        const double xx = x0 * x1, yy = y0 * y1, zz = z0 * z1;
        Q[2 + q] = yy - xx;
        Q[7 + q] = (2.0 * zz - xx - yy) * RSQ3;
        Q[12 + q] = fma(y0, z1, z0 * y1);
        Q[17 + q] = fma(x0, z1, z0 * x1);
        Q[22 + q] = fma(x0, y1, y0 * x1);
    }
}

// Q to the basis of rates<CUBIC>: P, R and the three shears of the stress as
// the resolved shears hold them (1/sqrt 6 of n and b included), so that every
// Schmid component is 0, +-1 or +-2
__device__ __forceinline__ void cubic_basis(double Q[25])
{
#pragma unroll
    for (int i = 0; i < 5; i++)
#pragma unroll
        for (int j = 0; j < 5; j++) Q[5 * i + j] *= cub_scale(j);
}

// merit function of NR_MODIFIED: |R|^2 / 2 with R = C0 r
__device__ __forceinline__ double merit(const double r[6])
{
    double R[6] = {0., 0., 0., 0., 0., 0.};
    sym6_mul_add(fresh(params_at(offsetof(NewtonParams, c0p)), r[0]), r, R);
    return 0.5 * norm2(R);
}

// One lane per voxel.  Reads lambda from sig_in and writes the new stress to
// sig (the same buffer or another) and, with FAST off, edot and gamdot; block
// partials (NRED doubles per block) of err_s, err_e, Newton iterations, sum
// sig, sum sig over phase 1 and line-search trials.
//
// The update works on r = S0 R, R the reference's residual
// s - lambda + C0 (eps_p + dt edot(s) + S s - E): with K0 = S0 + S and
// d = eps_p - E - S0 lambda it is r = K0 s + dt edot(s) + d, the Newton step
// solves (K0 + dt D) step = -r, and R itself is needed only where the line
// search has to compare |R|^2.  An accepted trial's rates and residual are
// the next iteration's start, and its tangent is formed only if that
// iteration takes a step.
//
// FAST: an iteration whose step the reference's line search is certain to
// reject (TOLX) ends right after the residual.  Since D >= 0, K = S0 + S +
// dt D >= S0 + S, so |step|_inf <= |r|_2 / lambda_min(S0 + S); when that
// bound is below TOLX (P.kmin_tolx2 holds (0.99 TOLX lambda_min)^2, the
// minimum over all orientations) the reference's test
// max|step_i|/max(|s_i|,1) < TOLX holds and its first trial is rejected,
// leaving s, edot, the error norms and the counts exactly as computed here.
// Only gamdot (from the rejected trial point) differs; the loop repeats the
// last Newton launch of an increment with FAST off before edot or gamdot is
// used, so FAST launches write neither.
template <int RM, bool CSYM, bool FAST, int NE, bool CUBIC>
__global__ __launch_bounds__(NB_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_newton(
    NewtonParams P, long long N, int p, int lead, const int *__restrict__ phase,
    const int *__restrict__ orient, const double *__restrict__ sgr, const double *sig_in, double *sig,
    const double *__restrict__ E, const double *__restrict__ epsp, double *__restrict__ edot,
    const double *__restrict__ tran, const double *__restrict__ crss, double *__restrict__ gamdot,
    double *__restrict__ partials, int *__restrict__ status)
{
    if (P.skip && *P.skip) return;
    constexpr bool GD = !FAST;
    // LDS columns: 1/CRSS, the tangent's weights, d and (FAST off) edot
    constexpr int NIT = CSYM ? EVPGPU_NSYSMX : 2 * EVPGPU_NSYSMX, ND = NIT + EVPGPU_NSYSMX;
    __shared__ double slab[(ND + 6 + (FAST ? 0 : 5)) * NB_THREADS];
    const int lane = threadIdx.x;
    const long long v0 = (long long)blockIdx.x * NB_THREADS + lane;
    // a lane past the end takes the last voxel's inputs and drops the result
    const unsigned v = (unsigned)(v0 < N ? v0 : N - 1);
    const int ph = phase[v], ori = orient[v];
    const int pl = ph - 1 < 0 ? 0 : (ph - 1 > 1 ? 1 : ph - 1);
    const bool gas_l = pl == 0 ? P.is_gas[0] != 0 : P.is_gas[1] != 0;
    const bool mine = v0 < N && !gas_l && pl == p;
    double *red = slab + lane; // the lane's NRED sums, in its own columns at the end
    if (__any(mine)) {
        double *it = slab + lane, *w = slab + NIT * NB_THREADS + lane;
        double *dl = slab + ND * NB_THREADS + lane, *edl = slab + (ND + 6) * NB_THREADS + lane;
        double K0[21], Q[25], s[6], r[6];
        double sn2; // |lambda|_F^2 (src/evolution.c:92-96)
        {
            // every load of the voxel's inputs first, then the arithmetic
            double d[6], t[6], tp[6], te[6], T9[9], c1[EVPGPU_NSYSMX], c2[EVPGPU_NSYSMX];
#pragma unroll
            for (int c = 0; c < 6; c++) t[c] = sig_in[c * N + v];
#pragma unroll
            for (int c = 0; c < 6; c++) tp[c] = epsp[c * N + v];
#pragma unroll
            for (int c = 0; c < 6; c++) te[c] = E[c * N + v];
#pragma unroll
            for (int q = 0; q < 9; q++) T9[q] = tran[q * N + v];
            const long long S12 = (long long)EVPGPU_NSYSMX * N;
#pragma unroll
            for (int k = 0; k < EVPGPU_NSYSMX; k++) {
                const int sy = CUBIC ? P.cub_sys[p][k] : k; // column k's system
                if (RM == RM_DISL) {
                    // crss holds the increment's constants: passing stress,
                    // 1/(tau_0 + tau_cut), gam_o, the first call's passing stress
                    c1[k] = crss[(P.dd_first ? 3 * S12 : 0) + sy * N + v];
                    c2[k] = crss[S12 + sy * N + v];
                } else {
                    c1[k] = crss[(sy * 2) * N + v];
                    if (!CSYM) c2[k] = crss[(sy * 2 + 1) * N + v];
                }
            }
            const double *sv = sgr + 36LL * ori;
#pragma unroll
            for (int i = 0; i < 6; i++)
#pragma unroll
                for (int j = i; j < 6; j++) K0[PK(i, j)] = sv[i * 6 + j];
            sn2 = t[0] * t[0] + t[1] * t[1] + t[2] * t[2] + 2.0 * (t[3] * t[3] + t[4] * t[4] + t[5] * t[5]);
            sym_to_v6(t, s);
#pragma unroll
            for (int i = 0; i < 6; i++) te[i] = tp[i] - te[i];
            sym_to_v6(te, d);
            // d = eps_p - E - S0 lambda, K0 = S0 + S
            cdouble S0 = fresh(params_at(offsetof(NewtonParams, s0p)), s[0]);
#pragma unroll
            for (int i = 0; i < 6; i++)
#pragma unroll
                for (int j = 0; j < 6; j++) d[i] = fma(-S0[PK(i, j)], s[j], d[i]);
#pragma unroll
            for (int i = 0; i < 21; i++) K0[i] += S0[i];
#pragma unroll
            for (int i = 0; i < 6; i++) dl[i * NB_THREADS] = d[i];
            rotation5(T9, Q);
            if (CUBIC) cubic_basis(Q);
#pragma unroll
            for (int k = 0; k < EVPGPU_NSYSMX; k++) {
                if (RM == RM_DISL) {
                    it[k * NB_THREADS] = c1[k];
                    it[(EVPGPU_NSYSMX + k) * NB_THREADS] = c2[k];
                } else {
                    it[k * NB_THREADS] = rcp_crss(c1[k]);
                    if (!CSYM) it[(EVPGPU_NSYSMX + k) * NB_THREADS] = rcp_crss(c2[k]);
                }
            }
        }
        const double *g0c = crss + 2LL * EVPGPU_NSYSMX * N + v; // RM_DISL: gam_o
        double *gd = gamdot + v;
        const int ns = RM == RM_FAST || RM == RM_DISL ? EVPGPU_NSYSMX : P.nsys[p];
        // The loops below are wave-uniform: a lane that has finished runs
        // along with its state frozen (open false), which keeps the control
        // flow scalar and the registers of the two loops disjoint.
        bool open = mine, singular = false, uphill = false;
        int iterl = 0, trials = 0;
        {
            double ed[5];
            rates<RM, CSYM, GD, NE, CUBIC>(P, p, it, w, g0c, N, Q, s, ed, gd, open);
            scaled_residual(P.dt, K0, dl, s, ed, r);
            if (!FAST)
#pragma unroll
                for (int i = 0; i < 5; i++) edl[i * NB_THREADS] = ed[i];
        }
        if (RM == RM_DISL && P.dd_first) {
            // the first call used the previous call's mobile density; every
            // later one sees the density that call formed
#pragma unroll
            for (int k = 0; k < EVPGPU_NSYSMX; k++)
                it[k * NB_THREADS] = crss[(CUBIC ? P.cub_sys[p][k] : k) * N + v];
        }
        double y2 = norm2(r);
        bool moved = false; // the last step, accepted, ended the solve
        for (;;) {
            iterl += open;
            if (FAST) {
                const bool sk = open && y2 > 0.0 && y2 < P.kmin_tolx2;
                trials += sk; // the reference's one rejected trial
                open = open && !sk;
                if (!__any(open)) break;
            }
            double step[6];
            {
                double K[21];
                tangent<CUBIC>(ns, p, w, Q, K0, K);
#pragma unroll
                for (int i = 0; i < 6; i++) step[i] = -r[i];
                bool pd = ldl6_solve(K, step);
                // (steep rates are RM_LOOP's, or RM_POW's without CUBIC)
                if (!CUBIC && (RM == RM_POW || RM == RM_LOOP) && __builtin_expect(__any(open && !pd), 0)) {
                    double x[6];
#pragma unroll
                    for (int i = 0; i < 6; i++) x[i] = -r[i];
                    const bool ok = rank1_solve(P, p, ns, w, Q, K0, x);
#pragma unroll
                    for (int i = 0; i < 6; i++) step[i] = pd ? step[i] : x[i];
                    pd = pd || ok;
                }
                singular = singular || (open && !pd);
                // the slope of the merit function along the step is
                // -scale |R|^2: zero only where the residual is
                uphill = uphill || (open && pd && y2 == 0.0);
                open = open && pd && y2 != 0.0;
            }
            // stpmax = 10 (src/evolution.c:166-170)
            const double sum = norm2(step);
            double scale = 1.0;
            if (sum > 100.0) {
                scale = 10.0 / sqrt(sum);
#pragma unroll
                for (int i = 0; i < 6; i++) step[i] *= scale;
            }
            // a trial is rejected (TOLX) when alam max|step_i|/max(|s_i|,1) < TOLX
            auto rejected = [&](double alam) {
                bool far = false;
#pragma unroll
                for (int i = 0; i < 6; i++)
                    far = far || alam * fabs(step[i]) >= P.tolx * fmax(fabs(s[i]), 1.0);
                return !far;
            };
            double alam = 1.0;
            bool rej = rejected(alam);
            // A rejected first trial leaves the step undone whatever its
            // merit value; only gamdot (from the trial point) is affected,
            // which FAST launches do not form, so they skip the evaluation.
            if (FAST) {
                trials += open && rej;
                open = open && !rej;
                if (!__any(open)) break;
            }
            double alam2 = 0.0, f2 = 0.0, sn[6], en[5] = {0., 0., 0., 0., 0.}, rn[6], y2n;
            bool search = open;
            for (;;) {
#pragma unroll
                for (int i = 0; i < 6; i++) sn[i] = fma(alam, step[i], s[i]);
                // (a lane whose search is over repeats its last trial, with
                // RM_DISL from the rates that it kept)
                double et[5];
                rates<RM, CSYM, GD, NE, CUBIC>(P, p, it, w, g0c, N, Q, sn, et, gd, search);
#pragma unroll
                for (int i = 0; i < 5; i++) en[i] = RM != RM_DISL || search ? et[i] : en[i];
                scaled_residual(P.dt, K0, dl, sn, en, rn);
                trials += search;
                y2n = norm2(rn);
                // |C0 r|^2 lies between c0_lo2 |r|^2 and c0_hi2 |r|^2 (C0's
                // extreme eigenvalues squared): where that decides the descent
                // test, the merit functions are not formed
                search = search && !rej && !(P.c0_hi2 * y2n <= 0.9997 * P.c0_lo2 * y2);
                if (!__any(search)) break;
                if (search) {
                    const double fo = merit(r), fn = merit(rn), slope = -2.0 * scale * fo;
                    search = !(fn <= fo + 1.E-4 * alam * slope);
                    if (search) {
                        const double next = ls_backtrack(alam, alam2, fn, f2, fo, slope);
                        alam2 = alam;
                        f2 = fn; // the backtrack value the cubic step needs (Q18)
                        alam = next;
                        rej = rejected(alam);
                    }
                }
                if (!__any(search)) break;
            }
            open = open && !rej;
            double cn = 0.0;
#pragma unroll
            for (int i = 0; i < 6; i++) cn = fma(sn[i] - s[i], sn[i] - s[i], cn);
            // the relative step against the tolerance (|sn - s| / |lambda|)
            if (open && (iterl >= 500 || !(cn > P.nr_tol * P.nr_tol * sn2))) {
                // done: edot and err_e stay those of the iteration's start
#pragma unroll
                for (int i = 0; i < 6; i++) it[i * NB_THREADS] = sn[i];
                moved = true;
                open = false;
            }
            if (!__any(open)) break;
            if (open) {
#pragma unroll
                for (int i = 0; i < 6; i++) {
                    s[i] = sn[i];
                    r[i] = rn[i];
                    if (!FAST && i < 5) edl[i * NB_THREADS] = en[i];
                }
                y2 = y2n;
            }
        }
        if (singular || uphill) atomicCAS(status, 0, singular ? EVPGPU_ERR_SINGULAR : EVPGPU_ERR_LINESEARCH);
        if (mine && !singular && !uphill) {
            double lam[6], t[6], so[6];
#pragma unroll
            for (int c = 0; c < 6; c++) t[c] = sig_in[c * N + v];
            sym_to_v6(t, lam);
            // the strain mismatch eps_p + dt edot + S s - E = r - S0 (s - lambda)
            double ds[6], cs = 0.0;
#pragma unroll
            for (int i = 0; i < 6; i++) {
                ds[i] = lam[i] - s[i];
                so[i] = moved ? it[i * NB_THREADS] : s[i];
            }
            sym6_mul_add(fresh(params_at(offsetof(NewtonParams, s0p)), ds[0]), ds, r);
#pragma unroll
            for (int i = 0; i < 6; i++) cs = fma(so[i] - lam[i], so[i] - lam[i], cs);
            v6_to_sym(so, t);
#pragma unroll
            for (int c = 0; c < 6; c++) {
                sig[c * N + v] = t[c];
                red[(3 + c) * NB_THREADS] = t[c];
                red[(9 + c) * NB_THREADS] = pl == 0 ? t[c] : 0.0;
            }
            red[0] = sqrt(cs);
            red[NB_THREADS] = sqrt(norm2(r));
            red[2 * NB_THREADS] = (double)iterl;
            red[15 * NB_THREADS] = (double)trials;
            if (!FAST) {
                double e6[6];
#pragma unroll
                for (int i = 0; i < 6; i++) e6[i] = i < 5 ? edl[i * NB_THREADS] : 0.0;
                v6_to_sym(e6, t);
#pragma unroll
                for (int c = 0; c < 6; c++) edot[c * N + v] = t[c];
            }
        } else {
#pragma unroll
            for (int i = 0; i < NRED; i++) red[i * NB_THREADS] = 0.0;
        }
    } else {
#pragma unroll
        for (int i = 0; i < NRED; i++) red[i * NB_THREADS] = 0.0;
    }
    if (lead && gas_l && v0 < N) {
#pragma unroll
        for (int c = 0; c < 6; c++) {
            sig[c * N + v] = 0.0;
            if (!FAST) edot[c * N + v] = 0.0;
        }
    }
    // Block partial sums: value i is summed by lanes 4i..4i+3 over 16 entries
    // each (every value from its own start, so that the 64 lanes spread over
    // the banks), then across the four (a + b == b + a, so all four hold the
    // same sum): a fixed order at a quarter of the instructions of 16
    // butterfly reductions.
    static_assert(NB_THREADS == 64 && NRED * 4 == NB_THREADS && NRED <= 2 * EVPGPU_NSYSMX,
                  "one wave per block, 16 partial sums");
    __syncthreads();
    const int vi = lane >> 2, q = lane & 3;
    double sum = 0.0;
#pragma unroll
    for (int j = 0; j < 16; j++) sum += slab[vi * NB_THREADS + q * 16 + ((j + vi) & 15)];
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    if (q == 0) partials[(long long)blockIdx.x * NRED + vi] = sum;
}

// Deterministic two-stage sum of nblk rows of nval (<= 16) partials.
// Stage 1: workgroup g sums rows [g*per, (g+1)*per): thread t owns value
// t % 16 and rows t/16, t/16 + 16, ... (coalesced row-major reads), then the
// 16 row lanes of each value are summed in LDS in a fixed order.
// Stage 2: one workgroup sums the stage-1 rows the same way.
constexpr int RED_MAXV = 16;

// status (stage 2 only, may be null): the Newton status word, appended as
// out[nval] so that one copy brings back the sums and the status.  skip (may
// be null): the launch does nothing when *skip is set.
__global__ __launch_bounds__(256) void k_reduce_rows(const double *__restrict__ partials, int nblk,
                                                     int nval, int per, double *__restrict__ out,
                                                     const int *__restrict__ status,
                                                     const int *__restrict__ skip)
{
    if (skip && *skip) return;
    if (status && blockIdx.x == 0 && threadIdx.x == 0) out[nval] = (double)*status;
    __shared__ double sh[256];
    const int v = threadIdx.x % RED_MAXV, r0 = threadIdx.x / RED_MAXV;
    const long long b0 = (long long)blockIdx.x * per;
    const long long b1 = min((long long)nblk, b0 + per);
    double s = 0.0;
    if (v < nval) {
        // unrolled so that the loads go out together (the sum keeps its order)
#pragma unroll 4
        for (long long b = b0 + r0; b < b1; b += 256 / RED_MAXV) s += partials[b * nval + v];
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    if (threadIdx.x < RED_MAXV) {
        double t = 0.0;
        for (int r = 0; r < 256 / RED_MAXV; r++) t += sh[r * RED_MAXV + threadIdx.x];
        if (threadIdx.x < nval) out[(long long)blockIdx.x * nval + threadIdx.x] = t;
    }
}

} // namespace

int newton_rate_mode(const NewtonParams &P)
{
    // the integral-exponent variants need every crystal phase to have one;
    // the fast one also n <= 32, a full set of systems and one gam0
    bool intn = true, fastrm = true;
    for (int q = 0; q < 2; q++) {
        if (P.is_gas[q]) continue;
        if (P.int_n[q] == 0) intn = false;
        bool one = P.int_n[q] >= 1 && P.int_n[q] <= 32 && P.nsys[q] == EVPGPU_NSYSMX;
        for (int k = 0; k < P.nsys[q]; k++)
            if (P.gam0[q][k] != P.gam0[q][0] || P.nrs[q][k] != P.nrs[q][0]) one = false;
        if (!one) fastrm = false;
    }
    return !intn ? RM_POW : (fastrm ? RM_FAST : RM_LOOP);
}

int newton_launch(evpgpu_ctx *c, const NewtonParams &P, const double *sig_in, double *sig, const double *E,
                  const double *epsp, double *edot, const double *tran, const double *crss,
                  double *gamdot, const int *phase, const int *orient, const double *sgr,
                  long long n, double *partials, int *nblk_out, int *status, int fast, hipEvent_t ev_start,
                  hipEvent_t ev_stop)
{
    const int nblk = (int)((n + NB_THREADS - 1) / NB_THREADS);
    const int rm = newton_rate_mode(P);
    // the dislocation-density variant assumes 12 systems in every crystal phase
    if (P.dd)
        for (int q = 0; q < 2; q++)
            if (!P.is_gas[q] && P.nsys[q] != EVPGPU_NSYSMX) return EVPGPU_ERR_ARG;
    // One launch per crystal phase (two at most; nblk rows of partials each):
    // the phase is then an argument, its constants scalar loads.  The first
    // also clears the gas voxels; a grid of gas only takes one launch.
    int crystal[2], nc = 0;
    for (int q = 0; q < 2; q++)
        if (!P.is_gas[q]) crystal[nc++] = q;
    if (nc == 0) crystal[nc++] = 0;
    for (int q = 0; q < nc; q++) {
        const int p = crystal[q], lead = q == 0;
        double *part = partials + (long long)q * nblk * NRED;
        // compile-time exponents for the common n = 10 and n = 20, the sums of
        // the cubic family wherever a phase has its twelve systems (219 us
        // against 240 at 128^3) and the rate law is odd in the resolved shear
        // (a place may hold a system of the other sign): not for unequal
        // forward and backward CRSS.  RM_LOOP (n of 33 to 64) has no such
        // variant: no use of it is known.  RM_POW's is for n up to 32: above it
        // the general one, which has rank1_solve (128 us a 48^3 iteration
        // against 120 at n = 12.5).
        bool steep = false;
        for (int k = 0; k < P.nsys[p]; k++) steep = steep || P.nrs[p][k] > 32.0;
        const int ne = rm == RM_FAST && P.crss_sym && (P.int_n[p] == 10 || P.int_n[p] == 20) ? P.int_n[p] : 0;
        // the events (when given) take the kernel's own start and end times: no
        // marker packets between the launches
#define NEWTON_ARGS dim3(nblk), dim3(NB_THREADS), 0, c->stream, lead ? ev_start : nullptr,                  \
                    q == nc - 1 ? ev_stop : nullptr, 0, P, n, p, lead, phase, orient, sgr, sig_in, sig, E, epsp, \
                    edot, tran, crss, gamdot, part, status
#define LAUNCH(A, B, F, E, C) hipExtLaunchKernelGGL((k_newton<A, B, F, E, C>), NEWTON_ARGS)
#define LAUNCH_SYM(F, C)                                                                 \
    do { /* RM_FAST with equal forward and backward CRSS */                              \
        if (ne == 10) LAUNCH(RM_FAST, true, F, 10, C);                                   \
        else if (ne == 20) LAUNCH(RM_FAST, true, F, 20, C);                              \
        else LAUNCH(RM_FAST, true, F, 0, C);                                             \
    } while (0)
#define LAUNCH_RM(F)                                                                     \
    do {                                                                                 \
        if (P.dd && P.cubic[p]) LAUNCH(RM_DISL, false, F, 0, true);                      \
        else if (P.dd) LAUNCH(RM_DISL, false, F, 0, false);                              \
        else if (rm == RM_FAST && P.crss_sym && P.cubic[p]) LAUNCH_SYM(F, true);         \
        else if (rm == RM_FAST && P.crss_sym) LAUNCH_SYM(F, false);                      \
        else if (rm == RM_FAST) LAUNCH(RM_FAST, false, F, 0, false);                     \
        else if (rm == RM_LOOP && P.crss_sym) LAUNCH(RM_LOOP, true, F, 0, false);        \
        else if (rm == RM_LOOP) LAUNCH(RM_LOOP, false, F, 0, false);                     \
        else if (rm == RM_POW && P.crss_sym && P.cubic[p] && !steep) LAUNCH(RM_POW, true, F, 0, true); \
        else if (P.crss_sym) LAUNCH(RM_POW, true, F, 0, false);                          \
        else LAUNCH(RM_POW, false, F, 0, false);                                         \
    } while (0)
        if (fast) LAUNCH_RM(true);
        else LAUNCH_RM(false);
#undef LAUNCH_RM
#undef LAUNCH_SYM
#undef LAUNCH
#undef NEWTON_ARGS
    }
    if (nblk_out) *nblk_out = nc * nblk;
    return hipGetLastError() == hipSuccess ? EVPGPU_OK : EVPGPU_ERR_HIP;
}

// out[nval] = column sums of partials[nblk][nval]; uses c->red2 (REDUCE_G rows)
int reduce_partials(evpgpu_ctx *c, const double *partials, int nblk, int nval, double *out, const int *status)
{
    if (nval > RED_MAXV) return EVPGPU_ERR_ARG;
    // (up to REDUCE_G rows the first stage would only copy them)
    int g = nblk;
    if (nblk > REDUCE_G) {
        const int per = (nblk + REDUCE_G - 1) / REDUCE_G;
        g = (nblk + per - 1) / per;
        hipLaunchKernelGGL(k_reduce_rows, dim3(g), dim3(256), 0, c->stream, partials, nblk, nval, per, c->red2,
                           (const int *)nullptr, (const int *)nullptr);
        partials = c->red2;
    }
    hipLaunchKernelGGL(k_reduce_rows, dim3(1), dim3(256), 0, c->stream, partials, g, nval, g, out, status,
                       (const int *)nullptr);
    return hipGetLastError() == hipSuccess ? EVPGPU_OK : EVPGPU_ERR_HIP;
}

// the first stage of reduce_partials alone: c->red2 = g rows of nval sums
// (the second stage's input, summed the same way by the loop control)
int reduce_stage1(evpgpu_ctx *c, const double *partials, int nblk, int nval, const int *skip, int *g_out)
{
    if (nval > RED_MAXV) return EVPGPU_ERR_ARG;
    int g = nblk < REDUCE_G ? nblk : REDUCE_G;
    int per = (nblk + g - 1) / g;
    g = (nblk + per - 1) / per;
    hipLaunchKernelGGL(k_reduce_rows, dim3(g), dim3(256), 0, c->stream, partials, nblk, nval, per, c->red2,
                       (const int *)nullptr, skip);
    *g_out = g;
    return hipGetLastError() == hipSuccess ? EVPGPU_OK : EVPGPU_ERR_HIP;
}
