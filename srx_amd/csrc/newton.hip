// newton.hip -- CDNA4 (gfx950) Newton kernels of the EVP-FFT increment loop: the constitutive
// solve of UpdateStress (evolution.c:157-427), one voxel per lane in FP64, its fields read and
// written as raw buffer accesses (one 32-bit lane offset from a scalar base); the fixed-order
// reductions of its block partial sums (k_reduce, k_reduce_seg), so every sum is bitwise
// repeatable from run to run; the device-side outer-iteration control (k_control); the
// lockstep ensemble variants; and the recorder of training samples for the learned start.
#include "crystal_dev.hpp"
#include "mlp_dev.hpp"

#include <type_traits>

namespace srx {

// ---------------------------------------------------------------------------
// NR kernel: UpdateStress (evolution.c:157-427) in the crystal frame of the
// current orientation.  With Q the B-basis rotation, Sc = Q^T S066 Q,
// S' the grain compliance and D = d(edot)/d(sig):
//   Rt(sig) = Sc (sig - lam) + eps_p + edot(sig) dt + S' sig - eps_c  ( = S066 R )
//   K = Sc + S' + D dt  ( = S066 J, symmetric positive definite)
// so the Newton step K^-1 Rt equals the reference's J^-1 R; K is factored
// LDL^T in place.  Stopping rule, iteration cap and the pre-update iterate
// used for Edot and the errors are the reference's.
// ---------------------------------------------------------------------------
constexpr int NR_BLOCK = 64;
// Zero components of the 12 {111}<110> Schmid vectors in the crystal frame's B basis, bit i for
// component i, by system modulo 3 (the order of the reference's slip-mode file and interaction table):
// a system whose Burgers vector lies in the plane of two axes has no shear in that plane, and with the
// third axis normal to it (modulo 3: 2) no second normal component either.
constexpr int fcc_zero(int s) { return s % 3 == 0 ? 1 << 2 : s % 3 == 1 ? 1 << 3 : (1 << 4) | (1 << 1); }
bool nr_fcc(const DevConst &hc) {
    for (int p = 0; p < NPH; ++p) {
        if (!hc.ph[p].xtal) continue;
        if (p != 0 || hc.ph[p].nsys != NSYS) return false;
        for (int s = 0; s < NSYS; ++s)
            for (int i = 0; i < 5; ++i)
                if ((fcc_zero(s) >> i & 1) && hc.ph[p].p[s][i] != 0.0) return false;
    }
    return hc.ph[0].xtal;
}

struct NrResult {
    double cs, ce;
    double sig[6];
    int it;     // iterations of the solve that produced sig
    int itot;   // iterations executed (both attempts of a repeated solve)
    int bad;
};

// deviatoric stress block of A = Q^T S066 Q plus the compliance, packed
__device__ __forceinline__ void sc_rotate(const double *__restrict__ S, const double Q[5][5], double A[15]) {
    double T1[5][5];
#pragma unroll
    for (int i = 0; i < 5; ++i)
#pragma unroll
        for (int j = 0; j < 5; ++j) {
            double acc = 0.0;
#pragma unroll
            for (int k = 0; k < 5; ++k) acc += S[6 * i + k] * Q[k][j];
            T1[i][j] = acc;
        }
#pragma unroll
    for (int i = 0; i < 5; ++i)
#pragma unroll
        for (int j = i; j < 5; ++j) {
            double acc = 0.0;
#pragma unroll
            for (int k = 0; k < 5; ++k) acc += Q[k][i] * T1[k][j];
            A[ps(i, j)] = acc;
        }
}

// eps_c = (DisGrad + DisGrad^T) / 2 in the B basis (chg_basis opt 2), from the 9 row-major components
__device__ __forceinline__ void ec_from_dg(const double d[9], double ec[6]) {
    const double s00 = d[0], s11 = d[4], s22 = d[8];
    const double s12 = (d[5] + d[7]) / 2.0, s02 = (d[2] + d[6]) / 2.0, s01 = (d[1] + d[3]) / 2.0;
    ec[0] = s00 * (-SRX_R2) + s11 * SRX_R2;
    ec[1] = s00 * (-SRX_R6) + s11 * (-SRX_R6) + s22 * (2. * SRX_R6);
    ec[2] = s12 * SRX_R2 + s12 * SRX_R2;
    ec[3] = s02 * SRX_R2 + s02 * SRX_R2;
    ec[4] = s01 * SRX_R2 + s01 * SRX_R2;
    ec[5] = s00 * SRX_R3 + s11 * SRX_R3 + s22 * SRX_R3;
}

// The strain a Newton call is driven by, eps_c - eps_p in the B basis: f.ee, or formed from DisGrad and
// the plastic strain where the outer iterations advance DisGrad itself (uniform branch).
__device__ __forceinline__ void load_strain(const Fields &f, size_t N, unsigned o8, double e[6]) {
    if (f.ee) {
#pragma unroll
        for (int k = 0; k < 6; ++k) e[k] = ldc(f.ee + (size_t)k * N, N, o8);
    } else {
        double d[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) d[k] = ldc(f.dg + (size_t)k * N, N, o8);
        ec_from_dg(d, e);
#pragma unroll
        for (int k = 0; k < 5; ++k) e[k] -= ldc(f.eps + (size_t)k * N, N, o8);
    }
}

// LDS slots of the per-system constants (tau_pass * inv, inv, gamma_0 dt of 12 systems), also the
// component order of Fields::nrc
constexpr int NRC_TP = 0, NRC_INV = NSYS, NRC_G0 = 2 * NSYS, NRC_COMPS = 3 * NSYS;
// after them, the orientation quaternion of the block's voxels: 40 slots of 64 doubles, 20 KB, are
// exactly an eighth of a compute unit's LDS
constexpr int NRC_QUAT = NRC_COMPS;
// The later calls of mixed precision keep their FP32 constants and 14 of the 15 values of A as FP32
// (widened at each use): 12.5 KB, a twelfth of a compute unit's LDS, so that three wavefronts per
// SIMD fit where the FP64 layout allows two.
constexpr int NRF_A = NRC_COMPS, NRF_A_COMPS = 14, NRF_SLOTS = NRC_COMPS + NRF_A_COMPS;
typedef float __attribute__((may_alias)) float_alias;

// Per-voxel values every Newton call of an increment starts from, in the crystal frame of the
// current orientation: lam' = Q^T lam, the matrix A = Sc + S' (packed), r0 = Q^T (eps_p - eps_c -
// S066 lam) (= Q^T (eps_p - eps_c) - Sc lam', Q being orthogonal), the hydrostatic parts and
// 1/||lam||^2.
struct NrPro {
    double lam[5], r0[5], A[15];
    double lamh, qh, rsig2;
};
// An empty statement that takes x in a register: x is computed before it, and the statement stays
// in program order with the memory waits around it.
__device__ __forceinline__ void pin(double &x) { asm volatile("" : "+v"(x)); }
// A field's base pointer as an opaque value at this point: the epilogue's buffer descriptors are
// built after the Newton loop instead of being the prologue's identical ones, which the compiler
// would keep in scalar registers (spilled to vector lanes) across the loop.
template <typename T>
__device__ __forceinline__ T *fresh(T *p) {
    asm volatile("" : "+s"(p));
    return p;
}
// The prologue is formed while the copies issued before it are in flight, not after the wait for
// them (the compiler would otherwise sink the arithmetic to its first use).
__device__ __forceinline__ void pin_prologue(NrPro &p) {
#pragma unroll
    for (int i = 0; i < 5; ++i) { pin(p.lam[i]); pin(p.r0[i]); }
    pin(p.lamh); pin(p.qh); pin(p.rsig2);
}

// The inputs of a Newton call for one voxel: orientation, stress, the strain eps_c - eps_p and,
// after the first call of an increment, the increment's matrix A (packed).  The orientation is TranMat
// for the first call, and for the later ones its quaternion (in a[0..3] until nr_orient expands it)
// where the context keeps one: 32 B instead of 72, and the epilogue takes it from LDS instead of
// reading TranMat again, 112 of 545 B per voxel and launch in mixed precision.
struct NrIn {
    double a[9], lam6[6], e[6], A[15];
};
__device__ __forceinline__ void nr_orient(const Fields &f, NrIn &in) {
    if (f.quat) {
        const double q[4] = {in.a[0], in.a[1], in.a[2], in.a[3]};
        rot_from_quat(q, in.a);
    }
}
template <bool LOAD_A, bool F32>
__device__ __forceinline__ void nr_load(const Fields &f, size_t N, unsigned o8, NrIn &in) {
    if (LOAD_A && f.quat) {
#pragma unroll
        for (int k = 0; k < 4; ++k) in.a[k] = ldc(f.quat + (size_t)k * N, N, o8);
    } else {
#pragma unroll
        for (int k = 0; k < 9; ++k) in.a[k] = ldc(f.tran + (size_t)k * N, N, o8);
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) in.lam6[k] = ldc(f.sig + (size_t)k * N, N, o8);
    load_strain(f, N, o8, in.e);
    if (LOAD_A) {
        const size_t P = nrcf_pitch(N);
        if (F32) {
#pragma unroll
            for (int k = NRF_A_COMPS; k < 15; ++k) in.A[k] = (double)ldcf(f.acrf + (size_t)k * P, P, o8 / 2);
        } else if (f.acrf) {
#pragma unroll
            for (int k = 0; k < 15; ++k) in.A[k] = (double)ldcf(f.acrf + (size_t)k * P, P, o8 / 2);
        } else {
#pragma unroll
            for (int k = 0; k < 15; ++k) in.A[k] = ldc(f.acr + (size_t)k * N, N, o8);
        }
    }
}

// WS: Newton start 0 = lam (the reference), 1 = lam + the previous call's change (extrapolated),
// 2 = lam + the learned prediction `wsp` (crystal frame)
// Prologue of a Newton call from its inputs `in`.  FIRST (the increment's first call): A assembled
// from the orientations (Sc = Q^T S066 Q and the rotated grain compliance S') and stored in f.acr
// for the increment's later calls.  Otherwise A is in.A.
// KEEP_EC (warm starts): the strain is also stored in f.ecp where `store` is set, for the next
// call's learned-start features.
template <bool FIRST, bool ROT, int PH, bool KEEP_EC, bool F32>
__device__ __forceinline__ void nr_prologue(const DevConst *__restrict__ cst, const Fields &f, int v, size_t N,
                                            const NrIn &in, NrPro &pro, bool store = true) {
    const DevPhase &P = cst->ph[PH];
    const unsigned o8 = 8u * (unsigned)v;
    if (!FIRST) {
#pragma unroll
        for (int k = F32 ? NRF_A_COMPS : 0; k < 15; ++k) pro.A[k] = in.A[k];
    }
    const double *a = in.a;
    double Q[5][5];
    q5_from(a, Q);
    double lam6[6], w[5];
    {
#pragma unroll
        for (int k = 0; k < 6; ++k) lam6[k] = in.lam6[k];
        if (KEEP_EC && store && f.ecp) {
#pragma unroll
            for (int k = 0; k < 6; ++k) stcf(f.ecp + (size_t)k * N, N, 4u * (unsigned)v, (float)in.e[k]);
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) w[k] = -in.e[k];
        pro.qh = -in.e[5];
    }
    double sn = 0.0;
#pragma unroll
    for (int k = 0; k < 6; ++k) sn += lam6[k] * lam6[k];
    pro.rsig2 = 1.0 / sn;
    pro.lamh = lam6[5];
    // u = S066 lam (deviatoric block, sample frame)
    double u[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        double acc = 0.0;
#pragma unroll
        for (int k = 0; k < 5; ++k) acc += cst->S066[i][k] * lam6[k];
        u[i] = acc;
    }
    // crystal frame: lam' = Q^T lam, r0 = Q^T (w - u)
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        double al = 0.0, ar = 0.0;
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            al += Q[k][i] * lam6[k];
            ar += Q[k][i] * (w[k] - u[k]);
        }
        pro.lam[i] = al;
        pro.r0[i] = ar;
    }
    if (FIRST) {
        sc_rotate(&cst->S066[0][0], Q, pro.A);
        if (ROT) {
            double a0[9], Sp[15];
#pragma unroll
            for (int k = 0; k < 9; ++k) a0[k] = ldc(f.tran0 + (size_t)(k) * N, N, o8);
            sprime(a, a0, P.sinv, Sp);
#pragma unroll
            for (int k = 0; k < 15; ++k) pro.A[k] += Sp[k];
        } else {
#pragma unroll
            for (int i = 0; i < 5; ++i) pro.A[ps(i, i)] += P.sinv[i];
        }
        if (f.acrf) {
#pragma unroll
            for (int k = 0; k < 15; ++k) {
                const float a32 = (float)pro.A[k];
                pro.A[k] = (double)a32;
                stcf(f.acrf + (size_t)(k) * nrcf_pitch(N), nrcf_pitch(N), 4u * (unsigned)v, a32);
            }
        } else {
#pragma unroll
            for (int k = 0; k < 15; ++k) stc(f.acr + (size_t)(k) * N, N, o8, pro.A[k]);
        }
    }
}

// WS: Newton start 0 = lam (the reference), 1 = lam + the previous call's change (extrapolated),
// 2 = lam + the learned prediction `wsp` (crystal frame).  FIRST: the call computes its prologue
// and per-system constants and stores them for the increment; otherwise the caller has put the
// prologue in `pro` and the constants in the LDS slots NRC_*.
// F32: the FP32 LDS layout (later calls of mixed precision).  FCC: the Schmid vectors have fcc_zero's zeros,
// which leaves out 10 of about 70 instructions per active system.
template <bool FIRST, bool ROT, int PH, int WS, bool GND, bool F32, bool FCC>
__device__ __forceinline__ void nr_voxel(const DevConst *__restrict__ cst, const Fields &f, int v, size_t N,
                                         double *lds, NrPro &pro, const float *wsp, NrResult &res) {
    // compile-time phase index: every material constant is a scalar load at a fixed offset
    const DevPhase &P = cst->ph[PH];
    const double dt = cst->dt;
    const unsigned o8 = 8u * (unsigned)v;
    if (FIRST) {
        NrIn in;
        nr_load<false, false>(f, N, o8, in);
        nr_prologue<true, ROT, PH, (WS != 0), false>(cst, f, v, N, in, pro);
        if (f.quat) {
            double q[4];
            quat_from_rot(in.a, q);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                stc(f.quat + (size_t)k * N, N, o8, q[k]);
                lds[(NRC_QUAT + k) * NR_BLOCK + threadIdx.x] = q[k];
            }
        }
    }
    double (&lam)[5] = pro.lam;
    double (&A)[15] = pro.A;
    double (&r0)[5] = pro.r0;
    const double lamh = pro.lamh, qh = pro.qh, rsig2 = pro.rsig2;
    double ws[5] = {0, 0, 0, 0, 0}, wsh = 0.0;   // warm start: crystal-frame offset of the first iterate
    const double Shh = cst->S066[5][5];
    const double Ah = Shh + P.sinv[5];
    const double rAh = rcp(Ah);
    const double r0h = qh - Shh * lamh;

    // per-system constants, kept in LDS (lane-major, conflict free): tau_pass * inv, inv and
    // gamma_0 * dt (the slip rates enter the residual and the Jacobian times dt); the first call of
    // an increment computes them and stores them in f.nrc, from where the caller copies them into
    // LDS for the later calls.  Its own first iterate takes tau_pass with the lagged rho_m: those
    // values sit in the tau_pass slots for the first iteration, and the second reloads the
    // increment's from f.nrc (this lane's own stores).
    double *tp = lds + NRC_TP * NR_BLOCK + threadIdx.x, *inv = lds + NRC_INV * NR_BLOCK + threadIdx.x;
    double *g0 = lds + NRC_G0 * NR_BLOCK + threadIdx.x;
    const float_alias *ldf = reinterpret_cast<const float_alias *>(lds) + threadIdx.x;
    // value of LDS slot `slot` of this lane, and of A
    auto slot = [&](int k) { return F32 ? (double)ldf[k * NR_BLOCK] : lds[k * NR_BLOCK + threadIdx.x]; };
    auto Aat = [&](int k) { return F32 && k < NRF_A_COMPS ? (double)ldf[(NRF_A + k) * NR_BLOCK] : A[k]; };
    // mixed precision: the constants are stored in FP32 (f.nrcf), and this call iterates with the
    // rounded values too, so that every call of the increment solves with the same constants
    const size_t fpitch = nrcf_pitch(N);
    if (FIRST) {
        const int nsys = P.nsys;
        const bool f32 = f.nrcf != nullptr;
        double rs[NSYS];
#pragma unroll
        for (int s = 0; s < NSYS; ++s) rs[s] = ldc(f.rho_s + (size_t)(s) * N, N, o8);
#pragma unroll
        for (int s = 0; s < NSYS; ++s) {
            double ct, ci, cg;
            if (s < nsys) {
                double rP, rF;
                rho_pf(P, rs, s, rP, rF);
                if (GND) gnd_add(cst, s, N, v, rP, rF);
                const double rmn = rho_mobile(P, rP, rF);
                double t, iv, g;
                sys_const(P, rP, rF, rmn, rmn, t, iv, g);
                ct = t * iv;
                ci = iv;
                cg = g * dt;
                const double rmo = ldc(f.rho_m + (size_t)(s) * N, N, o8);
                tp[s * NR_BLOCK] = P.c1Gb3 * fsqrt(fabs(rP + rmo)) * iv;
                stc(f.rho_m_old + (size_t)(s) * N, N, o8, rmo);
                stc(f.rho_m + (size_t)(s) * N, N, o8, rmn);
            } else {
                // an inactive system: e = |rss| ci - ct stays negative (also as FP32's largest value)
                ct = 1e300; ci = 0.0; cg = 0.0;
                tp[s * NR_BLOCK] = 1e300;
            }
            if (f32) {
                ct = (double)(float)fmin(ct, 3.0e38);
                ci = (double)(float)ci;
                cg = (double)(float)cg;
            }
            inv[s * NR_BLOCK] = ci;
            g0[s * NR_BLOCK] = cg;
            if (f32) {
                stcf(f.nrcf + (size_t)(NRC_TP + s) * fpitch, fpitch, 4u * (unsigned)v, (float)ct);
                stcf(f.nrcf + (size_t)(NRC_INV + s) * fpitch, fpitch, 4u * (unsigned)v, (float)ci);
                stcf(f.nrcf + (size_t)(NRC_G0 + s) * fpitch, fpitch, 4u * (unsigned)v, (float)cg);
            } else {
                stc(f.nrc + (size_t)(NRC_TP + s) * nrc_pitch(N), nrc_pitch(N), o8, ct);
                stc(f.nrc + (size_t)(NRC_INV + s) * nrc_pitch(N), nrc_pitch(N), o8, ci);
                stc(f.nrc + (size_t)(NRC_G0 + s) * nrc_pitch(N), nrc_pitch(N), o8, cg);
            }
        }
    }

    if (!FIRST && WS != 0) {
        // extrapolated start (WS 1): lam + (lam - lam of the previous outer iteration), the change
        // kept in the crystal frame of this increment's orientation, loaded by the caller with
        // the other inputs; learned start (WS 2): the network's offset
#pragma unroll
        for (int i = 0; i < 5; ++i) ws[i] = (double)wsp[i];
        wsh = (double)wsp[5];
    }
    double sg[5], sh = lamh + wsh, pre[5], preh = sh, R[5];   // R: residual of the iterate `pre`
#pragma unroll
    for (int i = 0; i < 5; ++i) { sg[i] = lam[i] + ws[i]; pre[i] = sg[i]; R[i] = 0.0; }
    int it = 0, itot = 0;
    // stopping rule ||d sig|| / ||lam|| <= 1e-10, compared squared (no square root per iteration)
    double err2 = 1E-18, errp2 = 0.0;   // this and the previous step's
    bool again = false;
    // the last step without K (see below): not with the FP32 layout, where keeping the factors across
    // iterations spills (349 us at 128^3 instead of 322), nor in the one first call
    constexpr bool SHORT_LAST = !F32 && !FIRST;
    // K: the iteration's matrix, then its factors
    double K[15];
    // One iteration's residual R = r0 + A sg + sum_s p_s g_s (and K = A + sum_s g2_s p_s p_s^T).
    // Two systems per trip, under one wavefront-uniform branch: their slip-rate evaluations are
    // independent dependency chains the scheduler interleaves (an inactive system of the two
    // evaluates at 0 and adds exact zeros).  Zp: components of the Schmid vectors of both systems that are
    // exactly zero, left out of the sums.
    auto two_systems = [&](auto with_k, auto zero, int sa, int sb) {
        constexpr bool WK = decltype(with_k)::value;
        constexpr int Zp = decltype(zero)::value;
        double rss[2], ivs[2], e[2];
        bool act = false;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int sys = u ? sb : sa;
            const double *p = P.p[sys];
            double acc = 0.0;
            bool any = false;
#pragma unroll
            for (int i = 0; i < 5; ++i)
                if (!(Zp >> i & 1)) {
                    acc = any ? acc + p[i] * sg[i] : p[i] * sg[i];
                    any = true;
                }
            rss[u] = acc;
            ivs[u] = slot(NRC_INV + sys);
            e[u] = fma(fabs(rss[u]), ivs[u], -slot(NRC_TP + sys));
            act |= e[u] > 0.0;
        }
        if (!__any(act)) return;
        double g[2], g2dt[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int sys = u ? sb : sa;
            if (WK) slip_rate(rss[u], e[u], ivs[u], slot(NRC_G0 + sys), g[u], g2dt[u]);
            else g[u] = slip_rate_only(rss[u], e[u], slot(NRC_G0 + sys));
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const double *p = P.p[u ? sb : sa];
#pragma unroll
            for (int i = 0; i < 5; ++i) {
                if (Zp >> i & 1) continue;
                R[i] += p[i] * g[u];
                if (WK) {
                    const double gp = g2dt[u] * p[i];
#pragma unroll
                    for (int j = i; j < 5; ++j)
                        if (!(Zp >> j & 1)) K[ps(i, j)] += gp * p[j];
                }
            }
        }
    };
    auto residual = [&](auto with_k) {
        constexpr bool WK = decltype(with_k)::value;
        double M[15];
#pragma unroll
        for (int k = 0; k < 15; ++k) M[k] = Aat(k);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            double acc = r0[i];
#pragma unroll
            for (int j = 0; j < 5; ++j) acc += M[ps(i, j)] * sg[j];
            R[i] = acc;
        }
        if (WK) {
#pragma unroll
            for (int k = 0; k < 15; ++k) K[k] = M[k];
        }
        if constexpr (FCC) {
            // the systems of one residue modulo 3 share their zero components (fcc_zero)
#pragma unroll 1
            for (int h = 0; h < NSYS; h += 6) two_systems(with_k, std::integral_constant<int, fcc_zero(0)>{}, h, h + 3);
#pragma unroll 1
            for (int h = 1; h < NSYS; h += 6) two_systems(with_k, std::integral_constant<int, fcc_zero(1)>{}, h, h + 3);
#pragma unroll 1
            for (int h = 2; h < NSYS; h += 6) two_systems(with_k, std::integral_constant<int, fcc_zero(2)>{}, h, h + 3);
        } else {
#pragma unroll 1
            for (int s0 = 0; s0 < NSYS; s0 += 2) two_systems(with_k, std::integral_constant<int, 0>{}, s0, s0 + 1);
        }
    };
    // With the learned start (WS 2), a solve that does not converge (non-finite iterate, or 500
    // iterations) is repeated from lam, the reference's start; `itot` counts both attempts.  (The
    // extrapolated start has not needed it; the second attempt costs it registers.  The first call
    // of an increment starts from lam already.)
    for (int att = 0; att < ((WS == 2 && !FIRST) ? 2 : 1); ++att) {
    if (att == 1) {
        if (err2 <= 1E-20) break;
#pragma unroll
        for (int i = 0; i < 5; ++i) { sg[i] = lam[i]; pre[i] = sg[i]; }
        sh = lamh;
        preh = sh;
        it = 0;
        err2 = 1E-18;
        again = false;
    }
    while (it < 500 && err2 > 1E-20) {
        // A lane's last step: with two steps taken and the next one predicted from their quadratic
        // convergence, err (err / errp)^2, a decade below the tolerance, the previous iteration's factors
        // give it as well (they differ by the last step's size, 1e-5 or less, of a step near 1e-12).
        // When that holds for every lane still iterating, K and its factorisation are left out, a third
        // of the iteration's instructions; a lane whose step then is not its last (a slip system became
        // active) repeats the iteration with its own K, so the iterates are the full iteration's.
        const bool last = SHORT_LAST && !again && it >= 2 && err2 * err2 * err2 <= 1E-22 * (errp2 * errp2);
        ++it;
        ++itot;
        if (FIRST && it == 2) {
            if (f.nrcf) {
                const float *nc = fresh(f.nrcf);
#pragma unroll
                for (int s = 0; s < NSYS; ++s)
                    tp[s * NR_BLOCK] = (double)ldcf(nc + (size_t)(NRC_TP + s) * fpitch, fpitch, 4u * (unsigned)v);
            } else {
                const double *nc = fresh(f.nrc);
#pragma unroll
                for (int s = 0; s < NSYS; ++s)
                    tp[s * NR_BLOCK] = ldc(nc + (size_t)(NRC_TP + s) * nrc_pitch(N), nrc_pitch(N), o8);
            }
        }
        const bool full = !SHORT_LAST || __any(!last);
        if (full) {
            residual(std::true_type{});
            // LDL^T in place: K[ps(j,j)] <- 1/D_j, K[ps(i,j)] <- L_ij (i > j)
            double D[5];
#pragma unroll
            for (int j = 0; j < 5; ++j) {
                double dj = K[ps(j, j)];
#pragma unroll
                for (int k = 0; k < j; ++k) dj -= K[ps(j, k)] * K[ps(j, k)] * D[k];
                const double rj = rcp_step(dj);
#pragma unroll
                for (int i = j + 1; i < 5; ++i) {
                    double acc = K[ps(i, j)];
#pragma unroll
                    for (int k = 0; k < j; ++k) acc -= K[ps(i, k)] * K[ps(j, k)] * D[k];
                    K[ps(i, j)] = acc * rj;
                }
                D[j] = dj;
                K[ps(j, j)] = rj;
            }
        } else {
            residual(std::false_type{});
        }
        double y[5];
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            double acc = R[i];
#pragma unroll
            for (int k = 0; k < i; ++k) acc -= K[ps(i, k)] * y[k];
            y[i] = acc;
        }
#pragma unroll
        for (int i = 0; i < 5; ++i) y[i] *= K[ps(i, i)];
#pragma unroll
        for (int i = 4; i >= 0; --i) {
#pragma unroll
            for (int k = i + 1; k < 5; ++k) y[i] -= K[ps(k, i)] * y[k];
        }
        const double dh = (Ah * sh + r0h) * rAh;
        double cnr = dh * dh;
#pragma unroll
        for (int i = 0; i < 5; ++i) cnr += y[i] * y[i];
        const double errn = cnr * rsig2;
        if (SHORT_LAST) {
            again = !full && errn > 1E-20;
            if (again) {
                --it;
                --itot;
                continue;
            }
            errp2 = err2;
        }
        err2 = errn;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            pre[i] = sg[i];
            sg[i] -= y[i];
        }
        preh = sh;
        sh -= dh;
    }
    }
    if (WS) {
        // this call's stress change (crystal frame) for the next call's extrapolated start
#pragma unroll
        for (int i = 0; i < 5; ++i) stcf(f.dsig + (size_t)i * N, N, 4u * (unsigned)v, (float)(sg[i] - lam[i]));
        stcf(f.dsig + 5 * N, N, 4u * (unsigned)v, (float)(sh - lamh));
    }
    // errors of evolution.c:381-391 and the stress back in the sample frame.  The strain error at the
    // pre-update iterate, eps_p + edot dt + S' pre - eps_c, is R - Sc (pre - lam') (R the residual there),
    // in the sample frame Q R - S066 (Q pre - lam).  The orientation comes back from LDS, or from memory
    // where it does not fit beside the FP32 layout's three wavefronts (the registers that held it were
    // released for the Newton loop); so does lam.
    {
        double a[9], qu[4];
        if (f.quat) {
            const double *qp = fresh(f.quat);
#pragma unroll
            for (int k = 0; k < 4; ++k)
                qu[k] = F32 ? ldc(qp + (size_t)k * N, N, o8) : lds[(NRC_QUAT + k) * NR_BLOCK + threadIdx.x];
        }
        double l5[5];
        if (F32) {
            const double *sp = fresh(f.sig);
#pragma unroll
            for (int k = 0; k < 5; ++k) l5[k] = ldc(sp + (size_t)k * N, N, o8);
        }
        if (f.quat) {
            rot_from_quat(qu, a);
        } else {
            const double *tr = fresh(f.tran);
#pragma unroll
            for (int k = 0; k < 9; ++k) a[k] = ldc(tr + (size_t)(k) * N, N, o8);
        }
        double Q[5][5];
        q5_from(a, Q);
        double d[5], e[5], cs2 = (sh - lamh) * (sh - lamh);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            double as = 0.0, ad = 0.0, ar = 0.0;
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                as += Q[i][k] * sg[k];
                ad += Q[i][k] * (F32 ? pre[k] : pre[k] - lam[k]);
                ar += Q[i][k] * R[k];
            }
            res.sig[i] = as;
            d[i] = F32 ? ad - l5[i] : ad;
            e[i] = ar;
            const double ds = F32 ? as - l5[i] : sg[i] - lam[i];
            cs2 += ds * ds;
        }
        res.cs = sqrt(cs2);
        double ce2 = 0.0;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            double acc = e[i];
#pragma unroll
            for (int k = 0; k < 5; ++k) acc -= cst->S066[i][k] * d[k];
            ce2 += acc * acc;
        }
        const double eh = qh + P.sinv[5] * preh;
        ce2 += eh * eh;
        res.ce = sqrt(ce2);
    }
    res.sig[5] = sh;
#pragma unroll
    for (int k = 0; k < 5; ++k) stc(fresh(f.sig_pre) + (size_t)(k) * N, N, o8, pre[k]);
    res.it = it;
    res.itot = itot;
    bool bad = false;
#pragma unroll
    for (int k = 0; k < 6; ++k) bad |= !isfinite(res.sig[k]);
    res.bad = bad;
}

// Waves per SIMD the register allocator targets for the Newton kernel: a second wavefront per
// SIMD to issue from (measured 31% faster than one), which the LDS of the per-system constants and the
// quaternion (20 KB per 64-lane block; 12.5 KB and three in the FP32 layout) also allows; both the first call of an increment and the later ones
// fit two without spills.
#ifndef SRX_NR_WAVES_PER_EU
#define SRX_NR_WAVES_PER_EU 2
#endif
#ifndef SRX_NR_F32_WAVES_PER_EU
#define SRX_NR_F32_WAVES_PER_EU 3
#endif
#ifndef SRX_NR_FIRST_WAVES_PER_EU
#define SRX_NR_FIRST_WAVES_PER_EU 2
#endif

typedef __attribute__((address_space(3))) void lds_void;

// Asynchronous copies of the NC components of one field (component c at base + c P, the pitch P
// even, so that every component slice is 16-byte aligned) for the voxels [v0, v0 + 64) of this
// block into the LDS slots lds + 64 c, as raw buffer loads to LDS: the component's base in a buffer
// resource (scalar registers) and one 32-bit byte offset per lane.  One 16-byte load per lane moves
// two components (lanes 32-63 the second, at byte offset 8 P further; with an odd NC the slot after
// the last one receives a copy of it).  Lanes past the last voxel read the pitch's padding or
// re-read valid elements (the values are never used).  Every lane of the block must take part (a
// lane's copy fills other lanes' elements), and the caller waits for the copies (copy_wait).
template <int NC>
__device__ __forceinline__ void copy_field(const double *base, size_t P, double *lds, int blk) {
#if __HIP_DEVICE_COMPILE__
    const int lane = threadIdx.x;
    const int v0 = blk * NR_BLOCK;
    const unsigned pb = 8u * (unsigned)min((size_t)(v0 + 2 * (lane & 31)), P - 2);
    const unsigned hi = (lane >> 5) ? 8u * (unsigned)P : 0u;
#pragma unroll
    for (int c = 0; c < NC; c += 2) {
        const bool two = c + 1 < NC;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(comp_rsrc(base + (size_t)c * P, two ? 2 * P : P),
                                                 (lds_void *)(lds + c * NR_BLOCK), 16, pb + (two ? hi : 0u), 0, 0, 0);
    }
#endif
}
// The same for constants stored in FP32 at pitch P (a multiple of 4): one 16-byte load per lane moves
// four components (lanes 16 q .. 16 q + 15 component c + q, four voxels each) into the upper half of
// the NC FP64 slots: FP32 slot k at float offset (NC + k) 64 from their start; widen_slots then
// converts them in place.  (The FP32 layout copies to its own first slot SLOT0 and does not widen.)
template <int NC, int SLOT0 = NC>
__device__ __forceinline__ void copy_field_f32(const float *base, size_t P, double *lds, int blk) {
#if __HIP_DEVICE_COMPILE__
    const int lane = threadIdx.x;
    const int v0 = blk * NR_BLOCK;
    const unsigned pb = 4u * (unsigned)min((size_t)(v0 + 4 * (lane & 15)), P - 4);
    const unsigned q = 4u * (unsigned)P * (unsigned)(lane >> 4);
    float *half = reinterpret_cast<float *>(lds) + SLOT0 * NR_BLOCK;
#pragma unroll
    for (int c = 0; c < NC; c += 4) {
        if (c + 4 <= NC || lane < (NC - c) * 16)   // a remainder of components: their lanes only
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base + (size_t)c * P), (short)0,
                                                  rsrc_bytes((NC - c < 4 ? NC - c : 4) * P * 4u), 0x00020000),
                (lds_void *)(half + c * NR_BLOCK), 16, pb + q, 0, 0, 0);
    }
#endif
}
// After copy_field_f32 and copy_wait: FP32 slot k -> FP64 slot k of the lane's voxel.  Every FP32
// value of the lane is read before the first FP64 slot is written (the FP64 slots overlay the FP32
// ones; a block is one wavefront, whose LDS accesses complete in program order).
template <int NC>
__device__ __forceinline__ void widen_slots(double *lds) {
    static_assert(NR_BLOCK == 64, "one wavefront per block");
    const float_alias *half = reinterpret_cast<const float_alias *>(lds + NC / 2 * NR_BLOCK) + threadIdx.x;
    float x[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) x[c] = half[c * NR_BLOCK];
    asm volatile("" ::: "memory");
#pragma unroll
    for (int c = 0; c < NC; ++c) lds[c * NR_BLOCK + threadIdx.x] = (double)x[c];
}
__device__ __forceinline__ void copy_wait() {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
}

// Learned start of the wavefront's voxels (every lane calls; non-crystalline lanes get zero).
// Features from the Newton call's inputs (orientation, stress, strain), the previous change and
// rho_s.
__device__ __forceinline__ void nr_learned_start(const DevConst *__restrict__ cst, const Fields &f, size_t N, int v,
                                                 bool xt, const NrIn &in, float wsp[6]) {
    float xf[MLP_IN], nd = 0.0f;
    if (xt) {
        double lamc[6], de[6], dec[6], rho = 0.0;
        const double *a = in.a;
        float d[6];
        crystal_stress(a, in.lam6, lamc);
        // forcing: the strain now minus that of the previous call, crystal frame
#pragma unroll
        for (int k = 0; k < 6; ++k) de[k] = in.e[k] - (double)f.ecp[k * N + v];
        crystal_stress(a, de, dec);
#pragma unroll
        for (int k = 0; k < 6; ++k) d[k] = f.dsig[k * N + v];
#pragma unroll
        for (int k = 0; k < NSYS; ++k) rho += ldc(f.rho_s + (size_t)(k) * N, N, 8u * (unsigned)v);
        mlp_features(a, lamc, d, dec, rho / NSYS, xf, nd);
    } else {
#pragma unroll
        for (int k = 0; k < MLP_IN; ++k) xf[k] = 0.0f;
    }
    float u[MLP_OUT];
#pragma unroll
    for (int k = 0; k < MLP_OUT; ++k) u[k] = xf[4 + k];
    mlp_normalise(f.mlp, xf);
    float y[MLP_OUT];
    MlpAcc unused;
    mlp_forward_wave<false>(f.mlp, xf, y, unused);
    double w6[6] = {0, 0, 0, 0, 0, 0};
    if (xt) mlp_start(f.mlp, y, u, nd, w6);
#pragma unroll
    for (int k = 0; k < 6; ++k) wsp[k] = (float)w6[k];
}

// One 64-voxel block of the Newton kernel: block `blk` of the `nblk` blocks of a grid of nvox
// voxels (partials: NR_NPART x nblk block partial sums).
// PH2: the second phase is crystalline (else its voxels are gas and its Newton path is not compiled).
template <bool FIRST, bool ROT, int WS, bool GND, bool PH2, bool F32, bool FCC>
__device__ __forceinline__ void nr_block(const DevConst *__restrict__ cst, const Fields &f, int nvox,
                                         double *__restrict__ partials, const IterCtl *__restrict__ ctl, int blk,
                                         int nblk) {
    if (ctl && ctl->done) return;
    const int v = blk * NR_BLOCK + threadIdx.x;
    const size_t N = (size_t)nvox;
    const bool valid = v < nvox;
    const int ph = valid ? f.phase[v] : 0;
    // LDS: the 36 per-system constants of the block's 64 voxels (18 KB; the first call of an
    // increment computes them here, the later ones copy them from f.nrc) and the orientation (2 KB); the FP32
    // layout holds the constants and 14 values of A in 12.5 KB.
    static_assert(!(F32 && FIRST), "the first call computes its constants in the FP64 layout");
    constexpr int NSLOT = F32 ? NRF_SLOTS / 2 : NRC_COMPS + 4;
    __shared__ __align__(16) double lds[NSLOT * NR_BLOCK];
    NrPro pro;
    float wsp[6] = {0, 0, 0, 0, 0, 0};
    if constexpr (!FIRST) {
        // After the first call of an increment: the call's inputs and A are loaded into registers,
        // then the increment's per-system constants are copied into LDS by asynchronous buffer
        // loads, so both arrive in one round trip to HBM and the prologue is formed while the
        // constants are in flight.  Every lane forms a prologue (lanes past the last voxel from
        // the last one's inputs).
        const int vv = valid ? v : nvox - 1;
        NrIn in;
        nr_load<true, F32>(f, N, 8u * (unsigned)vv, in);
        if constexpr (WS == 1) {
#pragma unroll
            for (int k = 0; k < 6; ++k) wsp[k] = ldcf(f.dsig + (size_t)k * N, N, 4u * (unsigned)vv);
        }
        if constexpr (WS == 2) {
#pragma unroll
            for (int k = 0; k < 4; ++k) lds[(NRC_QUAT + k) * NR_BLOCK + threadIdx.x] = in.a[k];
            nr_orient(f, in);
            nr_learned_start(cst, f, N, v, valid && ph >= 1 && ph <= NPH && cst->ph[ph - 1].xtal, in, wsp);
        }
        const bool f32 = f.nrcf != nullptr;
        if constexpr (F32) {
            copy_field_f32<NRC_COMPS, 0>(f.nrcf, nrcf_pitch(N), lds, blk);
            copy_field_f32<NRF_A_COMPS, NRF_A>(f.acrf, nrcf_pitch(N), lds, blk);
        } else if (f32) {
            copy_field_f32<NRC_COMPS>(f.nrcf, nrcf_pitch(N), lds, blk);
        } else {
            copy_field<NRC_COMPS>(f.nrc, nrc_pitch(N), lds, blk);
        }
        if constexpr (WS != 2) {
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (!F32) lds[(NRC_QUAT + k) * NR_BLOCK + threadIdx.x] = in.a[k];
            nr_orient(f, in);
        }
        nr_prologue<false, ROT, 0, (WS != 0), F32>(cst, f, vv, N, in, pro, valid);
        pin_prologue(pro);
        copy_wait();
        if (f32 && !F32) widen_slots<NRC_COMPS>(lds);
    }
    NrResult r;
    r.cs = 0.0; r.ce = 0.0; r.it = 0; r.itot = 0; r.bad = 0;
#pragma unroll
    for (int k = 0; k < 6; ++k) r.sig[k] = 0.0;
    // one pass per distinct phase present in the wavefront, with the phase index uniform
    unsigned long long todo = __ballot(valid && ph >= 1 && ph <= NPH);
    while (todo) {
        const int first = __ffsll((unsigned long long)todo) - 1;
        const int pu = __builtin_amdgcn_readfirstlane(__shfl(ph, first, 64));
        const bool mine = valid && ph == pu;
        if (mine) {
            if (pu == 1) {
                if (cst->ph[0].xtal) nr_voxel<FIRST, ROT, 0, WS, GND, F32, FCC>(cst, f, v, N, lds, pro, wsp, r);
            } else if constexpr (PH2) {
                if (cst->ph[1].xtal) nr_voxel<FIRST, ROT, 1, WS, GND, F32, false>(cst, f, v, N, lds, pro, wsp, r);
            }
        }
        todo &= ~__ballot(mine);
    }
    if (valid) {
        const unsigned o8 = 8u * (unsigned)v;
        // gas voxels: Sig = Edot = 0 (evolution.c:418-423)
        double *sg = fresh(f.sig);
#pragma unroll
        for (int k = 0; k < 6; ++k) stc(sg + (size_t)(k) * N, N, o8, r.sig[k]);
        fresh(f.nr_it)[v] = r.it;
    }
    // block partials: conv_s, conv_e, sig6, sig6 of phase 1, nr_sum, nr_max, nan, wavefront nr_max
    const int lane = threadIdx.x & 63;
    double red[NR_NPART];
    red[0] = wave_sum(r.cs);
    red[1] = wave_sum(r.ce);
#pragma unroll
    for (int k = 0; k < 6; ++k) red[2 + k] = wave_sum(r.sig[k]);
    // when every voxel of the wavefront is phase 1 the phase-1 sums are the full sums
    if (__any(valid && ph != 1)) {
#pragma unroll
        for (int k = 0; k < 6; ++k) red[8 + k] = wave_sum((valid && ph == 1) ? r.sig[k] : 0.0);
    } else {
#pragma unroll
        for (int k = 0; k < 6; ++k) red[8 + k] = red[2 + k];
    }
    red[14] = wave_sum((double)r.itot);
    // the wavefront's largest iteration count (the lane-iterations it executed / 64)
    red[15] = wave_max((double)r.itot);
    red[16] = __any(r.bad) ? 1.0 : 0.0;
    red[17] = red[15];
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < NR_NPART; ++k) partials[(size_t)k * nblk + blk] = red[k];
    }
}

template <bool FIRST, bool ROT, int WS, bool GND, bool PH2, bool F32, bool FCC>
__global__ void __launch_bounds__(NR_BLOCK)
__attribute__((amdgpu_waves_per_eu(FIRST ? SRX_NR_FIRST_WAVES_PER_EU : F32 ? SRX_NR_F32_WAVES_PER_EU : SRX_NR_WAVES_PER_EU, 8)))
k_nr(const DevConst *__restrict__ cst, Fields f, int nvox, double *__restrict__ partials,
     const IterCtl *__restrict__ ctl) {
    nr_block<FIRST, ROT, WS, GND, PH2, F32, FCC>(cst, f, nvox, partials, ctl, blockIdx.x, gridDim.x);
}

// The Newton kernel over every member of an ensemble in one launch: member m owns the blocks
// [tab[m].blk0, tab[m].blk0 + tab[m].nblk) of the grid.
template <bool FIRST, bool ROT, int WS, bool GND, bool PH2, bool F32, bool FCC>
__global__ void __launch_bounds__(NR_BLOCK)
__attribute__((amdgpu_waves_per_eu(FIRST ? SRX_NR_FIRST_WAVES_PER_EU : F32 ? SRX_NR_F32_WAVES_PER_EU : SRX_NR_WAVES_PER_EU, 8)))
k_nr_ens(const EnsMember *__restrict__ tab, int nmem) {
    int m = 0;
    while (m + 1 < nmem && (int)blockIdx.x >= tab[m + 1].blk0) ++m;
    const EnsMember &e = tab[m];
    nr_block<FIRST, ROT, WS, GND, PH2, F32, FCC>(e.cst, e.f, e.nvox, e.partials, e.ctl, blockIdx.x - e.blk0, e.nblk);
}

// fixed-order reduction of block partials stored component-major:
// out[k] = sum over blocks of part[k][b] (max for k in maxmask); one block per k.  Each thread
// keeps eight independent accumulators over a fixed stride, combined in a fixed order, so the
// result is the same on every run.
constexpr int RED_BLOCK = 1024;
// value k of the block partials part[k][0 .. nblocks-1] into out[k]; sh: the kernel's RED_BLOCK doubles of LDS
__device__ __forceinline__ void reduce_value(const double *__restrict__ part, int nblocks, unsigned long long maxmask,
                                             double *__restrict__ out, unsigned k, double *sh) {
    const bool ismax = (maxmask >> k) & 1ull;
    const double *row = part + (size_t)k * nblocks;
    const double init = ismax ? -1e308 : 0.0;
    double acc[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[u] = init;
    for (int b0 = threadIdx.x; b0 < nblocks; b0 += 8 * RED_BLOCK) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int b = b0 + u * RED_BLOCK;
            if (b < nblocks) acc[u] = ismax ? fmax(acc[u], row[b]) : acc[u] + row[b];
        }
    }
    double a = acc[0];
#pragma unroll
    for (int u = 1; u < 8; ++u) a = ismax ? fmax(a, acc[u]) : a + acc[u];
    sh[threadIdx.x] = a;
    __syncthreads();
    for (int st = RED_BLOCK / 2; st > 0; st >>= 1) {
        if (threadIdx.x < st)
            sh[threadIdx.x] = ismax ? fmax(sh[threadIdx.x], sh[threadIdx.x + st]) : sh[threadIdx.x] + sh[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[k] = sh[0];
}

__global__ void __launch_bounds__(RED_BLOCK) k_reduce(const double *__restrict__ part, int nblocks, int nvals,
                                                      unsigned long long maxmask, double *__restrict__ out,
                                                      const IterCtl *__restrict__ ctl) {
    if (ctl && ctl->done) return;
    __shared__ double sh[RED_BLOCK];
    reduce_value(part, nblocks, maxmask, out, blockIdx.x, sh);
    (void)nvals;
}

// the end-of-increment partials of every member of a lockstep ensemble: block (k, m) reduces value
// k of member m into its `red`
__global__ void __launch_bounds__(RED_BLOCK) k_reduce_end_ens(const EnsIncr *__restrict__ tab) {
    const EnsIncr &e = tab[blockIdx.y];
    __shared__ double sh[RED_BLOCK];
    reduce_value(e.partials, e.nblk, 0ull, e.red, blockIdx.x, sh);
}

// First stage of the per-iteration reduction: block (k, sg) reduces value k over the sg-th of
// RED_SEGS contiguous ranges of block partials, in a fixed order (strided accumulators, then the
// wavefronts, then the four wavefront results), into seg[k * RED_SEGS + sg].  k_control finishes.
constexpr int RED_SEGS = 16, RED_SEG_BLOCK = 256;

static_assert(NR_RED_SEG_DOUBLES == NR_NPART * RED_SEGS, "segment buffer size");
__device__ __forceinline__ void reduce_seg_block(const double *__restrict__ part, int nblocks,
                                                 unsigned long long maxmask, double *__restrict__ seg,
                                                 const IterCtl *__restrict__ ctl, int k, int sg) {
    if (ctl && ctl->done) return;
    const bool ismax = (maxmask >> k) & 1ull;
    const int chunk = (nblocks + RED_SEGS - 1) / RED_SEGS;
    const int b1 = min(nblocks, (sg + 1) * chunk);
    const double *row = part + (size_t)k * nblocks;
    const double init = ismax ? -1e308 : 0.0;
    double acc[4] = {init, init, init, init};
    for (int b0 = sg * chunk + threadIdx.x; b0 < b1; b0 += 4 * RED_SEG_BLOCK) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int b = b0 + u * RED_SEG_BLOCK;
            if (b < b1) acc[u] = ismax ? fmax(acc[u], row[b]) : acc[u] + row[b];
        }
    }
    double a = ismax ? fmax(fmax(acc[0], acc[1]), fmax(acc[2], acc[3])) : (acc[0] + acc[1]) + (acc[2] + acc[3]);
    a = ismax ? wave_max(a) : wave_sum(a);
    __shared__ double sh[RED_SEG_BLOCK / 64];
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = a;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = sh[0];
        for (int w = 1; w < RED_SEG_BLOCK / 64; ++w) r = ismax ? fmax(r, sh[w]) : r + sh[w];
        seg[k * RED_SEGS + sg] = r;
    }
}

__global__ void __launch_bounds__(RED_SEG_BLOCK) k_reduce_seg(const double *__restrict__ part, int nblocks,
                                                              unsigned long long maxmask, double *__restrict__ seg,
                                                              const IterCtl *__restrict__ ctl) {
    reduce_seg_block(part, nblocks, maxmask, seg, ctl, blockIdx.x, blockIdx.y);
}

// the same for every member of an ensemble: grid (NR_NPART, RED_SEGS, members)
__global__ void __launch_bounds__(RED_SEG_BLOCK) k_reduce_seg_ens(const EnsMember *__restrict__ tab,
                                                                  unsigned long long maxmask) {
    const EnsMember &e = tab[blockIdx.z];
    if (e.nblk <= NR_RED_ONE) return;   // k_control_ens sums this member's partials itself
    reduce_seg_block(e.partials, e.nblk, maxmask, e.redseg, e.ctl, blockIdx.x, blockIdx.y);
}

// One outer iteration's bookkeeping on the device (the host loop of evolution.c:1150-1256): the
// dDisGradAvg this iteration's inverse-z pass applied joins the uniform part, the reduced sums give the
// errors and get_smacro's averages and correction, and `done` decides whether the next iteration runs.
// One block; the iteration's other kernels have finished (stream order).
// Bound by latency alone: the control block, the compliance S0 and the sums are fetched together, and
// the first wavefront works the algebra out one tensor component per lane, in LDS (5.6-7.5 us a
// launch when one thread did it with S0 in memory).  Up to NR_RED_ONE Newton blocks the kernel also sums
// their partials itself, which saves k_reduce_seg's launch (4.6 us); beyond, one block's loads would
// take longer than that.
constexpr int CTL_BLOCK = 1024;
// One wavefront's sum (and, for the last value, maximum too) of one value's partials, 8 loads per lane
// in flight.
__device__ __forceinline__ void sum_partials(const double *__restrict__ row, int nblocks, double &sum, double &mx) {
    constexpr int U = 8;
    double acc[U], m = -1e308;
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = 0.0;
    for (int b0 = threadIdx.x & 63; b0 < nblocks; b0 += U * 64) {
        double x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = row[min(b0 + u * 64, nblocks - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bool in = b0 + u * 64 < nblocks;
            acc[u] += in ? x[u] : 0.0;
            m = fmax(m, x[u]);
        }
    }
#pragma unroll
    for (int st = U / 2; st > 0; st >>= 1)
#pragma unroll
        for (int u = 0; u < st; ++u) acc[u] += acc[u + st];
    sum = wave_sum(acc[0]);
    mx = m;
}

// orders one wavefront's LDS writes before its lanes' reads of each other's values
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// the B basis as a table, [6][9], for lanes that hold one component each
#define SRX_BB(i) bbasis(i, 0, 0), bbasis(i, 0, 1), bbasis(i, 0, 2), bbasis(i, 1, 0), bbasis(i, 1, 1), bbasis(i, 1, 2), \
                  bbasis(i, 2, 0), bbasis(i, 2, 1), bbasis(i, 2, 2)
__constant__ double k_bbasis[54] = {SRX_BB(0), SRX_BB(1), SRX_BB(2), SRX_BB(3), SRX_BB(4), SRX_BB(5)};
#undef SRX_BB
// get_smacro (evolution.c:590-664) by the first wavefront, one component per lane: volume averages, the
// strain correction dDisGradAvg of the stress-controlled components (upper-triangle entries only), and
// the two von Mises measures (the first with the out-of-bounds SigDevAvg[3][3] term of evolution.c:648
// taken as svm_stray).
// bcol: column l mod 9 of the B basis (tensor entry l mod 9 of each basis tensor), brow: its row l.
__device__ __forceinline__ void smacro_wave(IterCtl &c, const double *S0, const double *sum6, const double *sum6_ph1,
                                            const double bcol[6], const double brow[9], double *sda, double *sda1) {
    constexpr int UP[6] = {0, 4, 8, 5, 2, 1};   // tensor entries of the six upper-triangle components
    const int l = threadIdx.x;
    if (l < 18) {   // the averages: tensor entries of the sums
        const int k = l < 9 ? l : l - 9;
        const double *v = l < 9 ? sum6 : sum6_ph1;
        double t = 0.0;
#pragma unroll
        for (int i = 0; i < 6; ++i) t += v[i] * bcol[i];
        if (l < 9) c.SigAvg[k] = t * c.wgt;
        else c.SigAvg1[k] = t * (c.wgt / c.wgt_ph1);
    }
    wave_sync();
    if (l < 9) c.ddg[l] = 0.0;   // (lower-triangle entries are never set)
    wave_sync();
    if (l < 6) {
        const int q = UP[l];
        double acc = 0.0;
        if (c.vbc[l] == 0) {
#pragma unroll
            for (int k = 0; k < 6; ++k) acc += S0[q * 9 + UP[k]] * c.sbc[k] * (c.Scauchy[UP[k]] - c.SigAvg[UP[k]]);
        }
        c.ddg[q] = acc;
    }
    // deviators of the two averages: tensor entries of their five deviatoric B-basis components
    if (l < 18) {
        const int k = l < 9 ? l : l - 9;
        const double *a = l < 9 ? c.SigAvg : c.SigAvg1;
        double t = 0.0;
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            double b = 0.0;
#pragma unroll
            for (int e = 0; e < 9; ++e) b += a[e] * bbasis(i, e / 3, e % 3);
            t += b * bcol[i];
        }
        (l < 9 ? sda : sda1)[k] = t;
    }
    wave_sync();
    if (l < 9) c.acum[l] += c.ddg[l];
    if (l < 6) {   // sym(dDisGradAvg) in the B basis
        double b = 0.0;
#pragma unroll
        for (int e = 0; e < 9; ++e) {
            const int i = e / 3, j = e % 3;
            b += 0.5 * (c.ddg[e] + c.ddg[3 * j + i]) * brow[e];
        }
        c.ddg6[l] = b;
    }
    if (l == 0) {
        const double tr = c.svm_mode == 1 ? (sda[0] + sda[4] + sda[8]) : (sda[4] + sda[8] + c.svm_stray);
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            const double x = sda[k];
            s += k % 4 ? x * x : (x - tr / 3.0) * (x - tr / 3.0);
        }
        c.s_vm = sqrt(3. / 2. * s);
    }
    if (l == 1) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 9; ++k) s += sda1[k] * sda1[k];
        c.s_vm1 = sqrt(3. / 2. * s);
    }
    wave_sync();
}

__device__ __forceinline__ void control_block(const DevConst *__restrict__ cst, const double *__restrict__ part,
                                              int nblocks, const double *__restrict__ seg, IterCtl *ctl) {
    static_assert(sizeof(IterCtl) % 8 == 0, "IterCtl is copied as 64-bit words");
    constexpr int NW = sizeof(IterCtl) / 8;
    static_assert(NW + 81 <= CTL_BLOCK, "one word per thread");
    __shared__ IterCtl c;
    __shared__ double S0[81], red[NR_NPART], sda[9], sda1[9];
    const int t = threadIdx.x, nt = blockDim.x;
    for (int i = t; i < NW; i += nt)
        reinterpret_cast<unsigned long long *>(&c)[i] = reinterpret_cast<const unsigned long long *>(ctl)[i];
    for (int i = t; i < 81; i += nt) S0[i] = cst->S0[i];
    double bcol[6], brow[9];
    if (t < 64) {
#pragma unroll
        for (int i = 0; i < 6; ++i) bcol[i] = k_bbasis[i * 9 + t % 9];
#pragma unroll
        for (int e = 0; e < 9; ++e) brow[e] = k_bbasis[t % 6 * 9 + e];
    }
    if (nblocks <= NR_RED_ONE) {
        // wavefront w: value w, the last two also 16 (a flag) and 17 (the sum of what 15 is the maximum of)
        static_assert(NR_NPART == 18 && CTL_BLOCK == 16 * 64, "18 values over 16 wavefronts");
        const int w = t >> 6;
        double r, m;
        sum_partials(part + (size_t)w * nblocks, nblocks, r, m);
        if (w == 15) m = wave_max(m);
        if ((t & 63) == 0) {
            red[w] = w == 15 ? m : r;
            if (w == 15) red[17] = r;
        }
        if (w == 14) {
            sum_partials(part + (size_t)16 * nblocks, nblocks, r, m);
            if ((t & 63) == 0) red[16] = r;
        }
    } else if (t < NR_NPART) {
        // second stage of the reduction: the RED_SEGS partial results of each value, in order
        double r = seg[t * RED_SEGS];
#pragma unroll
        for (int sg = 1; sg < RED_SEGS; ++sg) r = t == 15 ? fmax(r, seg[t * RED_SEGS + sg]) : r + seg[t * RED_SEGS + sg];
        red[t] = r;
    }
    __syncthreads();
    if (c.done) return;
    if (t < 64) {
        const bool bad = red[16] > 0;   // a non-finite stress (the reference asserts, constitutive.c:683)
        if (t < 9) c.uniform[t] += c.ddg[t];
        if (t < 6 && !bad) c.sig_sum6[t] = red[2 + t];
        wave_sync();
        if (!bad) smacro_wave(c, S0, red + 2, red + 8, bcol, brow, sda, sda1);
        if (t < 6 && !bad) {
            const double m = c.mixed ? red[2 + t] / c.nvox : 0.0;
            c.mean6[t] = m;
            c.dcs6[t] = c.mixed ? m * c.nvox : 0.0;
        }
        if (t == 0) {
            c.iter += 1;
            if (bad) {
                c.nan = 1;
                c.done = 1;
            } else {
                c.nrtot += (long long)red[14];
                c.nrmax = max(c.nrmax, (int)red[15]);
                c.nrwave += red[17];
                const double ee = red[1] * c.wgt;
                c.Err_e = fabs(c.e_vm_prev) < 1E-5 ? 0.0 : ee / c.e_vm_prev;
                c.Err_s = red[0] * c.wgt / c.s_vm;
                c.done = ctl_stop(c);
            }
            if (c.done && c.done_host) __hip_atomic_store(c.done_host, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    __syncthreads();
    for (int i = t; i < NW; i += nt)
        reinterpret_cast<unsigned long long *>(ctl)[i] = reinterpret_cast<const unsigned long long *>(&c)[i];
}

__global__ void __launch_bounds__(CTL_BLOCK) k_control(const DevConst *__restrict__ cst, const double *__restrict__ part,
                                                       int nblocks, const double *__restrict__ seg, IterCtl *ctl) {
    control_block(cst, part, nblocks, seg, ctl);
}

// the same for every member of an ensemble (one block each); done[m] receives the member's stop
// flag, the only value the host reads between batches of iterations
__global__ void __launch_bounds__(CTL_BLOCK) k_control_ens(const EnsMember *__restrict__ tab, int *__restrict__ done) {
    const EnsMember &e = tab[blockIdx.x];
    control_block(e.cst, e.partials, e.nblk, e.redseg, e.ctl);
    __syncthreads();
    if (threadIdx.x == 0) done[blockIdx.x] = e.ctl->done;
}

// ---------------------------------------------------------------------------
// Training samples for the learned Newton start: voxel j * stride (j < nsamp).  Before a Newton
// call: features and the scale |d| of the previous change, at slot *count + j.  After it: the
// target, this call's change over that scale minus the previous change's direction (the
// correction to the extrapolated start), and the count advanced by nsamp (recording stops when
// the buffer is full).
// ---------------------------------------------------------------------------
__global__ void k_mlp_rec_x(const DevConst *__restrict__ cst, Fields f, int nvox, int stride, int nsamp,
                            float *__restrict__ X, float *__restrict__ ND, const int *__restrict__ count, int cap,
                            const IterCtl *__restrict__ ctl) {
    if (ctl && ctl->done) return;
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int base = *count;
    if (j >= nsamp || base + nsamp > cap) return;
    const int v = j * stride;
    const size_t N = (size_t)nvox;
    const int ph = f.phase[v];
    float x[MLP_IN], nd = 0.0f;
    if (ph >= 1 && ph <= NPH && cst->ph[ph - 1].xtal) {
        double a[9], lam6[6], lamc[6], de[6], dec[6], rho = 0.0;
        float d[6];
        for (int k = 0; k < 9; ++k) a[k] = f.tran[k * N + v];
        for (int k = 0; k < 6; ++k) lam6[k] = f.sig[k * N + v];
        crystal_stress(a, lam6, lamc);
        load_strain(f, N, 8u * (unsigned)v, de);
        for (int k = 0; k < 6; ++k) de[k] -= (double)f.ecp[k * N + v];
        crystal_stress(a, de, dec);
        for (int k = 0; k < 6; ++k) d[k] = f.dsig[k * N + v];
        for (int k = 0; k < NSYS; ++k) rho += f.rho_s[k * N + v];
        mlp_features(a, lamc, d, dec, rho / NSYS, x, nd);
    } else {
        for (int k = 0; k < MLP_IN; ++k) x[k] = 0.0f;
    }
    for (int k = 0; k < MLP_IN; ++k) X[(size_t)(base + j) * MLP_IN + k] = x[k];
    ND[base + j] = nd;
}

__global__ void k_mlp_rec_t(Fields f, int nvox, int stride, int nsamp, const float *__restrict__ X,
                            float *__restrict__ T, const float *__restrict__ ND, const int *__restrict__ count, int cap,
                            const IterCtl *__restrict__ ctl) {
    if (ctl && ctl->done) return;
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    const int base = *count;
    if (j >= nsamp || base + nsamp > cap) return;
    const int v = j * stride;
    const size_t N = (size_t)nvox;
    const float nd = ND[base + j];
    const float *u = X + (size_t)(base + j) * MLP_IN + 4;
    for (int k = 0; k < MLP_OUT; ++k)
        T[(size_t)(base + j) * MLP_OUT + k] = nd > 0.0f ? f.dsig[k * N + v] / nd - u[k] : 0.0f;
}

__global__ void k_mlp_rec_adv(int *__restrict__ count, int cap, int nsamp, const IterCtl *__restrict__ ctl) {
    if (ctl && ctl->done) return;
    if (threadIdx.x == 0 && *count + nsamp <= cap) *count += nsamp;
}

// ---------------------------------------------------------------------------
// host launch wrappers
// ---------------------------------------------------------------------------
void launch_mlp_record(hipStream_t s, const DevConst *cst, const Fields &f, int nvox, int stride, int after,
                       float *X, float *T, float *ND, int *count, int cap, const IterCtl *ctl) {
    const int nsamp = (nvox + stride - 1) / stride;
    const dim3 g((nsamp + 255) / 256), b(256);
    if (!after) {
        hipLaunchKernelGGL(k_mlp_rec_x, g, b, 0, s, cst, f, nvox, stride, nsamp, X, ND, count, cap, ctl);
    } else {
        hipLaunchKernelGGL(k_mlp_rec_t, g, b, 0, s, f, nvox, stride, nsamp, X, T, ND, count, cap, ctl);
        hipLaunchKernelGGL(k_mlp_rec_adv, dim3(1), dim3(64), 0, s, count, cap, nsamp, ctl);
    }
    check_launch("mlp_record");
}

int nr_block_count(int nvox) { return (nvox + NR_BLOCK - 1) / NR_BLOCK; }

// Kernel variant of a Newton call: first call of an increment (F), rotated texture (R, which only the
// first call's matrix A depends on), Newton start (W: 0 reference, 1 extrapolated, 2 learned; the first call
// of an increment starts as 1), GND option (G, reference start only), crystalline second phase (P); for
// the later calls also the FP32 LDS layout of mixed precision (not with the learned start, whose
// matrix-core operands need the registers) and the FCC zeros (not with a second phase or the learned
// start; the first call, one in about sixty, goes without).
#define SRX_NR_VARIANTS(K, ARGS)                                                                           \
    do {                                                                                                 \
        const int ws_ = first_call && ws == 2 ? 1 : ws;                                                  \
        const bool v_ = !first_call && ws_ != 2;                                                         \
        const int code_ = (first_call ? 32 : 0) | (first_call && rotated ? 16 : 0) | (gnd ? 8 : 0) |     \
                          (ph2 ? 4 : 0) | (v_ && f32 ? 2 : 0) | (v_ && fcc && !ph2 ? 1 : 0);             \
        switch (code_ * 4 + ws_) {                                                                       \
        SRX_NR_FIRST(K, ARGS, 0, 0) SRX_NR_FIRST(K, ARGS, 0, 1) SRX_NR_FIRST(K, ARGS, 1, 0)              \
        SRX_NR_LATER(K, ARGS, 0, 0) SRX_NR_LATER(K, ARGS, 0, 1) SRX_NR_LATER(K, ARGS, 1, 0)              \
        SRX_NR_ONE(K, ARGS, 0, 0, 2, 0, 0, 0, 0) SRX_NR_ONE(K, ARGS, 0, 0, 2, 0, 1, 0, 0)                \
        default: break;                                                                                  \
        }                                                                                                \
    } while (0)
#define SRX_NR_ONE(K, ARGS, F, R, W, G, P, S, Z)                                                         \
    case ((F) * 32 + (R) * 16 + (G) * 8 + (P) * 4 + (S) * 2 + (Z)) * 4 + (W):                            \
        SRX_APPLY(SRX_LAUNCH, (K<(F) != 0, (R) != 0, (W), (G) != 0, (P) != 0, (S) != 0, (Z) != 0>),      \
                  SRX_UNPACK ARGS);                                                                      \
        break;
#define SRX_NR_FIRST(K, ARGS, G, W)                                                                      \
    SRX_NR_ONE(K, ARGS, 1, 0, W, G, 0, 0, 0) SRX_NR_ONE(K, ARGS, 1, 1, W, G, 0, 0, 0)                    \
    SRX_NR_ONE(K, ARGS, 1, 0, W, G, 1, 0, 0) SRX_NR_ONE(K, ARGS, 1, 1, W, G, 1, 0, 0)
#define SRX_NR_LATER(K, ARGS, G, W)                                                                      \
    SRX_NR_ONE(K, ARGS, 0, 0, W, G, 0, 0, 0) SRX_NR_ONE(K, ARGS, 0, 0, W, G, 0, 0, 1)                    \
    SRX_NR_ONE(K, ARGS, 0, 0, W, G, 0, 1, 0) SRX_NR_ONE(K, ARGS, 0, 0, W, G, 0, 1, 1)                    \
    SRX_NR_ONE(K, ARGS, 0, 0, W, G, 1, 0, 0) SRX_NR_ONE(K, ARGS, 0, 0, W, G, 1, 1, 0)
#define SRX_UNPACK(...) __VA_ARGS__
#define SRX_APPLY(M, ...) M(__VA_ARGS__)

void launch_nr(hipStream_t s, const DevConst *cst, const Fields &f, int nvox, int first_call, int rotated,
               double *partials, const IterCtl *ctl, int gnd, int ph2, int fcc) {
    const dim3 g(nr_block_count(nvox)), b(NR_BLOCK);
    // the learned start needs the network; with only the previous change it is the extrapolated one
    const int ws = gnd ? 0 : (f.dsig && f.mlp) ? 2 : f.dsig ? 1 : 0;
    const bool f32 = f.nrcf && f.quat;   // (without the quaternion the epilogue's orientation does not fit)
    SRX_NR_VARIANTS(k_nr, (g, b, 0, s, cst, f, nvox, partials, ctl));
    check_launch("nr");
}

void launch_reduce(hipStream_t s, const double *partials, int nblocks, int nvals, double *out, const IterCtl *ctl) {
    const unsigned long long mask = nvals == NR_NPART ? (1ull << 15) : 0ull;
    SRX_LAUNCH(k_reduce, dim3(nvals), dim3(RED_BLOCK), 0, s, partials, nblocks, nvals, mask, out, ctl);
    check_launch("reduce");
}

void launch_reduce_end_ens(hipStream_t s, const EnsIncr *tab, int nmem) {
    SRX_LAUNCH(k_reduce_end_ens, dim3(END_NPART, nmem), dim3(RED_BLOCK), 0, s, tab);
    check_launch("reduce_end_ens");
}

void launch_reduce_nr(hipStream_t s, const double *partials, int nblocks, double *seg, const IterCtl *ctl) {
    if (nblocks <= NR_RED_ONE) return;   // left to k_control
    SRX_LAUNCH(k_reduce_seg, dim3(NR_NPART, RED_SEGS), dim3(RED_SEG_BLOCK), 0, s, partials, nblocks, 1ull << 15, seg,
               ctl);
    check_launch("reduce");
}

void launch_nr_ens(hipStream_t s, const EnsMember *tab, int nmem, int nblocks, int first_call, int rotated, int ws,
                   int gnd, int ph2, int f32, int fcc) {
    const dim3 g(nblocks), b(NR_BLOCK);
    if (gnd) ws = 0;
    SRX_NR_VARIANTS(k_nr_ens, (g, b, 0, s, tab, nmem));
    check_launch("nr_ens");
}

void launch_reduce_nr_ens(hipStream_t s, const EnsMember *tab, int nmem) {
    SRX_LAUNCH(k_reduce_seg_ens, dim3(NR_NPART, RED_SEGS, nmem), dim3(RED_SEG_BLOCK), 0, s, tab, 1ull << 15);
    check_launch("reduce_ens");
}

void launch_control_ens(hipStream_t s, const EnsMember *tab, int nmem, int *done) {
    SRX_LAUNCH(k_control_ens, dim3(nmem), dim3(CTL_BLOCK), 0, s, tab, done);
    check_launch("control_ens");
}

void launch_control(hipStream_t s, const DevConst *cst, const double *partials, int nblocks, const double *seg,
                    IterCtl *ctl) {
    SRX_LAUNCH(k_control, dim3(1), dim3(nblocks <= NR_RED_ONE ? CTL_BLOCK : 256), 0, s, cst, partials, nblocks, seg, ctl);
    check_launch("control");
}

}  // namespace srx
