// fft.hip -- CDNA4 (gfx950) FFT and Green passes of the EVP-FFT increment loop
// (evolution.c:1157-1201 replaced): LDS-resident Stockham radix-2/3/4/5/8 transforms over
// batches of pencils, 256 threads per block, their global loads issued in chunks before the
// first wait.
//   fwd_z   real [c][x][y][z]      -> half spectrum B [c][kz][x][y]   (two real comps per complex FFT)
//   fft_y   B <-> C [c][kz][y][x]  (the y transform doubles as the pencil transpose)
//   green   C(6 stress comps) -> forward x -> Green operator -> inverse x -> C(6 strain comps, or DisGrad's 9:
//           strain_form), in place (k_green_wave: one wavefront per row, cross-lane butterflies, for x extents 64/128/256;
//           k_green_x: LDS transforms otherwise)
//   inv_z   B(6 or 9 comps) -> c2r along z, fused with the FP64 update of the strain or of DisGrad (Eq. 15)
//   plane   forward y, green and inverse y of small planes in one launch, layout B in place
// and, once per increment with the six components, DisGrad's rotation part (launch_rotation_part).
// Also here: the FFT-only test entry points and the streaming copy that measures the HBM ceiling.
#include "kern_common.hpp"

namespace srx {

// Events of the next launch (see SRX_LAUNCH).
thread_local hipEvent_t g_ev_start = nullptr, g_ev_stop = nullptr;
void set_launch_events(hipEvent_t a, hipEvent_t b) {
    g_ev_start = a;
    g_ev_stop = b;
}

// ---------------------------------------------------------------------------
// complex helpers
// ---------------------------------------------------------------------------
template <typename T>
struct cx {
    T x, y;
};
template <typename T>
__device__ __forceinline__ cx<T> operator+(cx<T> a, cx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ cx<T> operator-(cx<T> a, cx<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T>
__device__ __forceinline__ cx<T> cmul(cx<T> a, cx<T> b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
template <typename T>
__device__ __forceinline__ cx<T> cscale(cx<T> a, T s) { return {a.x * s, a.y * s}; }
// multiply by -i*sign ... helpers: i*a = (-a.y, a.x)
template <typename T>
__device__ __forceinline__ cx<T> mul_i(cx<T> a) { return {-a.y, a.x}; }
// two complex values (a pair of components loaded together)
template <typename T>
struct cx2 {
    cx<T> a, b;
};

// ---------------------------------------------------------------------------
// radix butterflies; sign = -1 forward (e^{-2 pi i/R}), +1 inverse
// ---------------------------------------------------------------------------
template <typename T, int R>
struct Dft;

template <typename T>
struct Dft<T, 2> {
    __device__ __forceinline__ static void run(cx<T> *v, int) {
        cx<T> a = v[0], b = v[1];
        v[0] = a + b;
        v[1] = a - b;
    }
};
template <typename T>
struct Dft<T, 3> {
    __device__ __forceinline__ static void run(cx<T> *v, int sign) {
        const T c = T(-0.5), s = T(0.86602540378443864676) * T(sign);
        cx<T> t1 = v[1] + v[2], t2 = v[1] - v[2];
        cx<T> a = v[0];
        cx<T> m = {a.x + c * t1.x, a.y + c * t1.y};
        cx<T> r = {-s * t2.y, s * t2.x};   // i*s*t2
        v[0] = a + t1;
        v[1] = m + r;
        v[2] = m - r;
    }
};
template <typename T>
struct Dft<T, 4> {
    __device__ __forceinline__ static void run(cx<T> *v, int sign) {
        cx<T> t0 = v[0] + v[2], t1 = v[0] - v[2], t2 = v[1] + v[3], d = v[1] - v[3];
        // t3 = sign*i*(b-d): forward -> -i(b-d)
        cx<T> t3 = sign < 0 ? cx<T>{d.y, -d.x} : cx<T>{-d.y, d.x};
        v[0] = t0 + t2;
        v[2] = t0 - t2;
        v[1] = t1 + t3;
        v[3] = t1 - t3;
    }
};
template <typename T>
struct Dft<T, 5> {
    __device__ __forceinline__ static void run(cx<T> *v, int sign) {
        const T c1 = T(0.30901699437494742410), c2 = T(-0.80901699437494742410);
        const T s1 = T(0.95105651629515357212) * T(sign), s2 = T(0.58778525229247312917) * T(sign);
        cx<T> a = v[0];
        cx<T> p1 = v[1] + v[4], m1 = v[1] - v[4], p2 = v[2] + v[3], m2 = v[2] - v[3];
        cx<T> r1 = {a.x + c1 * p1.x + c2 * p2.x, a.y + c1 * p1.y + c2 * p2.y};
        cx<T> r2 = {a.x + c2 * p1.x + c1 * p2.x, a.y + c2 * p1.y + c1 * p2.y};
        // i*(s1*m1 + s2*m2) and i*(s2*m1 - s1*m2)
        cx<T> q1 = {s1 * m1.x + s2 * m2.x, s1 * m1.y + s2 * m2.y};
        cx<T> q2 = {s2 * m1.x - s1 * m2.x, s2 * m1.y - s1 * m2.y};
        v[0] = a + p1 + p2;
        v[1] = r1 + mul_i(q1);
        v[4] = r1 - mul_i(q1);
        v[2] = r2 + mul_i(q2);
        v[3] = r2 - mul_i(q2);
    }
};

template <typename T>
struct Dft<T, 8> {
    // even/odd split into two radix-4 transforms
    __device__ __forceinline__ static void run(cx<T> *v, int sign) {
        cx<T> e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
        Dft<T, 4>::run(e, sign);
        Dft<T, 4>::run(o, sign);
        const T h = T(0.70710678118654752440);
        const T sh = T(sign) * h;
        const cx<T> o1 = cmul(o[1], cx<T>{h, sh});
        const cx<T> o2 = sign < 0 ? cx<T>{o[2].y, -o[2].x} : cx<T>{-o[2].y, o[2].x};
        const cx<T> o3 = cmul(o[3], cx<T>{-h, sh});
        v[0] = e[0] + o[0];
        v[4] = e[0] - o[0];
        v[1] = e[1] + o1;
        v[5] = e[1] - o1;
        v[2] = e[2] + o2;
        v[6] = e[2] - o2;
        v[3] = e[3] + o3;
        v[7] = e[3] - o3;
    }
};

constexpr int FFT_BLOCK = 256;

// n / d for 0 <= n with n * d < 2^32, as one high multiply by ceil(2^32 / d) (exact in that
// range); replaces the long integer-division sequence in the index arithmetic of the passes.  Built on
// the host and passed to the kernels: the multiplier is itself a division, and working out a handful of
// them per stage lengthened the passes' chains.  16^3: 50.5 -> 46.7 us an outer iteration, 96^3 in mixed
// precision 283 -> 272.
struct FastDiv {
    unsigned m;
    int d;
    FastDiv() = default;
    explicit FastDiv(int dd) : m(dd > 1 ? 0xFFFFFFFFu / (unsigned)dd + 1u : 0u), d(dd) {}
    __device__ __forceinline__ int div(int n) const { return d > 1 ? (int)__umulhi((unsigned)n, m) : n; }
};
// rows of a block's tile (the last tile of a pass may be short), times a row's length `per`
struct TileDiv {
    FastDiv full, last;
    TileDiv(int rows, int tile, int per) : full(tile * per), last((rows - (rows - 1) / tile * tile) * per) {}
    __device__ __forceinline__ FastDiv of(bool whole) const {
        FastDiv f;
        f.m = whole ? full.m : last.m;
        f.d = whole ? full.d : last.d;
        return f;
    }
};
// A plan with what each of its stages needs: radix, twiddle step and the divisors of its indices (dL: by the span)
struct FftStages {
    int n, nst;
    struct Stage {
        int R, tstep;
        FastDiv nb, dL;
    } st[MAX_RADIX_STAGES];
    explicit FftStages(const FftPlan &p) : n(p.n), nst(p.nst) {
        int L = 1;
        for (int i = 0; i < nst; ++i) {
            const int R = p.rad[i];
            st[i] = {R, n / (L * R), FastDiv(n / R), FastDiv(L)};
            L *= R;
        }
    }
};

// Element loop of a pass's global-memory side: elements [0, tot) dealt to the block's threads,
// taken in chunks of CH per thread whose loads ld(i) are all issued before the first store
// st(i, value) waits on them (one round trip to HBM per chunk, not per element).  Threads past the
// end load element tot - 1 again and store nothing.
constexpr int FFT_CHUNK = 8;
template <typename V, typename Ld, typename St>
__device__ __forceinline__ void chunked_copy(int tot, Ld ld, St st) {
    for (int b = 0; b < tot; b += FFT_CHUNK * FFT_BLOCK) {
        V v[FFT_CHUNK];
#pragma unroll
        for (int e = 0; e < FFT_CHUNK; ++e) v[e] = ld(min(b + e * FFT_BLOCK + (int)threadIdx.x, tot - 1));
#pragma unroll
        for (int e = 0; e < FFT_CHUNK; ++e) {
            const int i = b + e * FFT_BLOCK + (int)threadIdx.x;
            if (i < tot) st(i, v[e]);
        }
    }
}

// Position in LDS of element e of a pencil whose length is a multiple of 32: bits 0-4 of e XORed
// with b and 8b, b = bits 5-6 of e (a permutation within each aligned run of 32 elements).  A
// radix-8 first stage writes element 8j + r from butterfly j and a radix-4 second stage element
// 32 jl + k + 8 r (j = 8 jl + k); unswizzled, four lanes of a pencil share each LDS bank in both,
// swizzled the lanes of a pencil write distinct banks.  The passes' own LDS accesses use the same
// positions.
__device__ __forceinline__ int lds_swz(int e) {
    const int b = (e >> 5) & 3;
    return e ^ b ^ (b << 3);
}

// One Stockham stage (radix R, sub-transform span L) over `npen` pencils of
// length N stored pencil-major in LDS.  Every butterfly of the stage is held
// in registers between the load and the store, so the stage runs in place.
template <typename T, int R, int MAXB>
__device__ __forceinline__ void stockham_stage(cx<T> *buf, int npen, const FftStages::Stage &sg,
                                               const cx<T> *__restrict__ tw, int sign, int pitch) {
    const FastDiv dnb = sg.nb, dL = sg.dL;
    const int nb = dnb.d, L = dL.d, tstep = sg.tstep;
    const int total = npen * nb;
    cx<T> v[MAXB][R];
#pragma unroll
    for (int m = 0; m < MAXB; ++m) {
        const int t = threadIdx.x + m * FFT_BLOCK;
        if (t < total) {
            const int p = dnb.div(t), j = t - p * nb;
            const cx<T> *src = buf + p * pitch + j;
#pragma unroll
            for (int r = 0; r < R; ++r) v[m][r] = src[r * nb];
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MAXB; ++m) {
        const int t = threadIdx.x + m * FFT_BLOCK;
        if (t < total) {
            const int p = dnb.div(t), j = t - p * nb;
            const int jl = dL.div(j), k = j - jl * L;
            if (k) {
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    cx<T> w = tw[r * k * tstep];
                    if (sign > 0) w.y = -w.y;
                    v[m][r] = cmul(v[m][r], w);
                }
            }
            Dft<T, R>::run(v[m], sign);
            cx<T> *dst = buf + p * pitch + jl * L * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) dst[r * L] = v[m][r];
        }
    }
    __syncthreads();
}

// The same stage with the pencil length and span known at compile time (powers of two):
// the index arithmetic reduces to shifts and masks.
template <typename T, int R, int MAXB, int N, int L, bool SW>
__device__ __forceinline__ void stockham_stage_ct(cx<T> *buf, int npen, const cx<T> *__restrict__ tw, int sign,
                                                  int pitch) {
    constexpr int nb = N / R;
    constexpr int tstep = N / (L * R);
    const int total = npen * nb;
    cx<T> v[MAXB][R];
#pragma unroll
    for (int m = 0; m < MAXB; ++m) {
        const int t = threadIdx.x + m * FFT_BLOCK;
        if (t < total) {
            const int p = t / nb, j = t % nb;
            const cx<T> *src = buf + p * pitch + (SW ? 0 : j);
#pragma unroll
            for (int r = 0; r < R; ++r) v[m][r] = src[SW ? lds_swz(j + r * nb) : r * nb];
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MAXB; ++m) {
        const int t = threadIdx.x + m * FFT_BLOCK;
        if (t < total) {
            const int p = t / nb, j = t % nb;
            const int k = j % L;
            if (k) {
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    cx<T> w = tw[r * k * tstep];
                    if (sign > 0) w.y = -w.y;
                    v[m][r] = cmul(v[m][r], w);
                }
            }
            Dft<T, R>::run(v[m], sign);
            const int e0 = (j / L) * L * R + k;
            cx<T> *dst = buf + p * pitch + (SW ? 0 : e0);
#pragma unroll
            for (int r = 0; r < R; ++r) dst[SW ? lds_swz(e0 + r * L) : r * L] = v[m][r];
        }
    }
    __syncthreads();
}

// radix of stage st of a power-of-two length N, in the order make_plan chooses
// (radix 8 as often as possible without a radix-2 stage, then 4s, then a 2)
__host__ __device__ constexpr int pow2_radix(int N, int st) {
    int k2 = 0;
    while ((1 << k2) < N) ++k2;
    int n8 = k2 / 3, n4 = 0, n2 = 0;
    if (k2 % 3 == 1) { if (n8 > 0) { --n8; n4 = 2; } else { n2 = 1; } }
    else if (k2 % 3 == 2) n4 = 1;
    if (st < n8) return 8;
    if (st < n8 + n4) return 4;
    if (st < n8 + n4 + n2) return 2;
    return 0;
}

template <typename T, int MAXB, int N, int ST, int L, bool SW>
__device__ __forceinline__ void lds_fft_pow2(cx<T> *buf, int npen, const cx<T> *__restrict__ tw, int sign,
                                             int pitch) {
    constexpr int R = pow2_radix(N, ST);
    if constexpr (R != 0) {
        stockham_stage_ct<T, R, MAXB, N, L, SW>(buf, npen, tw, sign, pitch);
        lds_fft_pow2<T, MAXB, N, ST + 1, L * R, SW>(buf, npen, tw, sign, pitch);
    }
}

// whether plan pl is make_plan's schedule for the power-of-two length N (the one the compile-time
// stages run); a tuned or caller-set plan with other radices takes the runtime stages
template <int N>
__device__ __forceinline__ bool pow2_default(const FftStages &pl) {
    constexpr int ns = pow2_radix(N, 0) == 0 ? 0 : pow2_radix(N, 1) == 0 ? 1 : pow2_radix(N, 2) == 0 ? 2
                     : pow2_radix(N, 3) == 0 ? 3 : 4;
    bool same = pl.nst == ns;
#pragma unroll
    for (int st = 0; st < ns; ++st) same = same && pl.st[st].R == pow2_radix(N, st);
    return same;
}

// Full 1-D transform of npen LDS-resident pencils.  Caller guarantees
// npen*N/min_radix <= MAXB*FFT_BLOCK and a __syncthreads() before the call.  SWZ: the compile-time
// stages store the pencils swizzled (lds_swz), and the caller's own accesses must do the same.
// POW2: lengths 32..256 with make_plan's radices use the compile-time stages (measured faster in
// the x, y and z passes; in the z passes they cost an occupancy step, which the swizzled, conflict
// free stages more than repay).
template <typename T, int MAXB, bool POW2 = true, bool SWZ = true>
__device__ void lds_fft(cx<T> *buf, int npen, const FftStages &pl, const cx<T> *__restrict__ tw, int sign,
                        int pitch) {
    if constexpr (POW2) {
        switch (pl.n) {
        case 32: if (pow2_default<32>(pl)) { lds_fft_pow2<T, MAXB, 32, 0, 1, SWZ>(buf, npen, tw, sign, pitch); return; } break;
        case 64: if (pow2_default<64>(pl)) { lds_fft_pow2<T, MAXB, 64, 0, 1, SWZ>(buf, npen, tw, sign, pitch); return; } break;
        case 128: if (pow2_default<128>(pl)) { lds_fft_pow2<T, MAXB, 128, 0, 1, SWZ>(buf, npen, tw, sign, pitch); return; } break;
        case 256: if (pow2_default<256>(pl)) { lds_fft_pow2<T, MAXB, 256, 0, 1, SWZ>(buf, npen, tw, sign, pitch); return; } break;
        default: break;
        }
    }
    for (int st = 0; st < pl.nst; ++st) {
        const FftStages::Stage sg = pl.st[st];
        switch (sg.R) {
        case 8: stockham_stage<T, 8, MAXB>(buf, npen, sg, tw, sign, pitch); break;
        case 4: stockham_stage<T, 4, MAXB>(buf, npen, sg, tw, sign, pitch); break;
        case 2: stockham_stage<T, 2, MAXB>(buf, npen, sg, tw, sign, pitch); break;
        case 3: stockham_stage<T, 3, MAXB>(buf, npen, sg, tw, sign, pitch); break;
        default: stockham_stage<T, 5, MAXB>(buf, npen, sg, tw, sign, pitch); break;
        }
    }
}

// Waves per SIMD targeted for the z passes (0: the compiler's choice).
#ifndef SRX_ZPASS_WPE
#define SRX_ZPASS_WPE 0
#endif
#if SRX_ZPASS_WPE > 0
#define SRX_ZPASS_ATTR __attribute__((amdgpu_waves_per_eu(SRX_ZPASS_WPE, 8)))
#else
#define SRX_ZPASS_ATTR
#endif

// ---------------------------------------------------------------------------
// forward z: real comps -> half spectrum, layout B [c][kz][x][y].  A block takes TY consecutive
// z rows of the n0 n1 (row (x, y) at x n1 + y, in both layouts), so short z extents fill a block with
// more rows and a row range may cross x planes: at 256 x 256 x 1 a block of 16 rows had 16 elements
// to transform (28 us forward, 47 inverse); grid: (ceil(n0 n1 / TY), component pairs)
// ---------------------------------------------------------------------------
template <typename T, bool SW>
__global__ void __launch_bounds__(FFT_BLOCK) SRX_ZPASS_ATTR k_fwd_z(const double *__restrict__ in, cx<T> *__restrict__ specB,
                                                     int ncomp, int n0, int n1, int n2, FftStages pz,
                                                     FastDiv dn2, TileDiv dt, const cx<T> *__restrict__ tw, int TY,
                                                     const IterCtl *__restrict__ ctl) {
    if (ctl && ctl->done) return;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T> *buf = reinterpret_cast<cx<T> *>(smem_raw);
    // SW: the plan runs the compile-time stages, which store the pencils swizzled (lds_swz) at pitch
    // n2 + 2, and the accesses here do the same; else the runtime stages, plain, at pitch n2 + 1
    constexpr bool sw = SW;
    const int P = SW ? n2 + 2 : n2 + 1;   // padded pencil pitch: rows fall on different LDS banks
    cx<T> *stw = buf + TY * P;            // twiddle table staged in LDS
    const int rows = n0 * n1, row0 = blockIdx.x * TY;
    const int ty = min(TY, rows - row0);
    const int H = n2 / 2 + 1;
    const size_t N = (size_t)rows * n2;
    const size_t HS = (size_t)H * rows;
    const FastDiv dty = dt.of(ty == TY);
    for (int i = threadIdx.x; i < n2; i += FFT_BLOCK) stw[i] = tw[i];
    // one pair of components per block along grid y
    for (int ca = 2 * blockIdx.y; ca < ncomp && ca < 2 * blockIdx.y + 2; ca += 2) {
        const int cb = ca + 1;
        const bool two = cb < ncomp;
        const double ma = ctl && ca < 6 ? ctl->mean6[ca] : 0.0, mb = (ctl && two && cb < 6) ? ctl->mean6[cb] : 0.0;
        const double *ia = in + ca * N, *ib = in + (two ? cb : ca) * N;
        const size_t g0 = (size_t)row0 * n2;   // the block's rows are contiguous
        chunked_copy<cx<double>>(
            ty * n2, [&](int i) { return cx<double>{ia[g0 + i], ib[g0 + i]}; },
            [&](int i, cx<double> v) {
                const int yy = dn2.div(i), z = i - yy * n2;
                buf[yy * P + (sw ? lds_swz(z) : z)] = cx<T>{T(v.x - ma), T(two ? v.y - mb : 0.0)};
            });
        __syncthreads();
        if constexpr (SW) lds_fft<T, 2, true, true>(buf, ty, pz, stw, -1, P);
        else lds_fft<T, 2, false, false>(buf, ty, pz, stw, -1, P);
        for (int i = threadIdx.x; i < H * ty; i += FFT_BLOCK) {
            const int kz = dty.div(i), yy = i - kz * ty;
            const int e2 = kz == 0 ? 0 : n2 - kz;
            const cx<T> z1 = buf[yy * P + (sw ? lds_swz(kz) : kz)];
            const cx<T> z2 = buf[yy * P + (sw ? lds_swz(e2) : e2)];
            const size_t o = (size_t)kz * rows + row0 + yy;
            specB[ca * HS + o] = cx<T>{T(0.5) * (z1.x + z2.x), T(0.5) * (z1.y - z2.y)};
            if (two) specB[cb * HS + o] = cx<T>{T(0.5) * (z1.y + z2.y), T(-0.5) * (z1.x - z2.x)};
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// y transform with transpose.  b_to_c: B [c][kz][x][y] -> C [c][kz][y][x]
// (forward, sign -1); otherwise C -> B (inverse, sign +1).
// grid: (ceil(n0/TX), H, ncomp)
// ---------------------------------------------------------------------------
template <typename T, bool SW>
__global__ void __launch_bounds__(FFT_BLOCK) k_fft_y(const cx<T> *__restrict__ in, cx<T> *__restrict__ out,
                                                     int n0, int n1, int n2, int b_to_c, FftStages py,
                                                     FastDiv dn1, TileDiv dt,
                                                     const cx<T> *__restrict__ tw, int TX,
                                                     const IterCtl *__restrict__ ctl) {
    if (ctl && ctl->done) return;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T> *buf = reinterpret_cast<cx<T> *>(smem_raw);
    // SW: compile-time stages, swizzled pencils at pitch n1 + 2; else runtime stages, plain, n1 + 1
    constexpr bool sw = SW;
    const int P = SW ? n1 + 2 : n1 + 1;   // padded pencil pitch
    cx<T> *stw = buf + TX * P;
    for (int i = threadIdx.x; i < n1; i += FFT_BLOCK) stw[i] = tw[i];
    const int H = n2 / 2 + 1;
    const int x0 = blockIdx.x * TX;
    const int tx = min(TX, n0 - x0);
    const int kz = blockIdx.y;
    const int c = blockIdx.z;
    const size_t plane = (size_t)n0 * n1;
    const size_t base = ((size_t)c * H + kz) * plane;
    const FastDiv dtx = dt.of(tx == TX);
    if (b_to_c) {
        // the block's x rows are contiguous in B
        const cx<T> *src = in + base + (size_t)x0 * n1;
        chunked_copy<cx<T>>(tx * n1, [&](int i) { return src[i]; },
                            [&](int i, cx<T> v) {
                                const int xx = dn1.div(i), y = i - xx * n1;
                                buf[xx * P + (sw ? lds_swz(y) : y)] = v;
                            });
    } else {
        chunked_copy<cx<T>>(
            tx * n1,
            [&](int i) {
                const int y = dtx.div(i), xx = i - y * tx;
                return in[base + (size_t)y * n0 + x0 + xx];
            },
            [&](int i, cx<T> v) {
                const int y = dtx.div(i), xx = i - y * tx;
                buf[xx * P + (sw ? lds_swz(y) : y)] = v;
            });
    }
    __syncthreads();
    if constexpr (SW) lds_fft<T, 2, true, true>(buf, tx, py, stw, b_to_c ? -1 : +1, P);
    else lds_fft<T, 2, false, false>(buf, tx, py, stw, b_to_c ? -1 : +1, P);
    if (b_to_c) {
        for (int i = threadIdx.x; i < tx * n1; i += FFT_BLOCK) {
            const int y = dtx.div(i), xx = i - y * tx;
            out[base + (size_t)y * n0 + x0 + xx] = buf[xx * P + (sw ? lds_swz(y) : y)];
        }
    } else {
        for (int i = threadIdx.x; i < tx * n1; i += FFT_BLOCK) {
            const int xx = dn1.div(i), y = i - xx * n1;
            out[base + (size_t)(x0 + xx) * n1 + y] = buf[xx * P + (sw ? lds_swz(y) : y)];
        }
    }
}

// ---------------------------------------------------------------------------
// Green operator at one k point (init.c:542-592 with evolution.c:1169-1183):
//   Omega = (C0_ijkl n_j n_l)^-1,  du_ij = -Omega_ik (sig_kl n_l) n_j
// sig: 6 B-basis comps (complex) -> the strain increment sym(du), 6 B-basis comps.
// ---------------------------------------------------------------------------
template <typename A>
__device__ __forceinline__ void unit_k(int idx, int n, A &t) {
    A v = (A)idx * (A)(1.0 / n);
    v -= round(v);
    t = v * (A)6.28318530718;
}

// B-basis 6-vector -> symmetric tensor entries (00, 11, 22, 12, 02, 01)
template <typename A>
__device__ __forceinline__ void b6_to_sym(const A v[6], A t[6]) {
    t[0] = v[0] * A(-SRX_R2) + v[1] * A(-SRX_R6) + v[5] * A(SRX_R3);
    t[1] = v[0] * A(SRX_R2) + v[1] * A(-SRX_R6) + v[5] * A(SRX_R3);
    t[2] = v[1] * A(2. * SRX_R6) + v[5] * A(SRX_R3);
    t[3] = v[2] * A(SRX_R2);
    t[4] = v[3] * A(SRX_R2);
    t[5] = v[4] * A(SRX_R2);
}
__device__ __forceinline__ void sym_to_t9(const double t[6], double m[9]) {
    m[0] = t[0]; m[4] = t[1]; m[8] = t[2];
    m[5] = m[7] = t[3];
    m[2] = m[6] = t[4];
    m[1] = m[3] = t[5];
}

// Green operator at one k point from the symmetric contraction table G6:
//   A_ik = sum_jl C0_ijkl n_j n_l = sum_b G6[(ik)][b] m_b,  m = (n0^2, n1^2, n2^2, n1n2, n0n2, n0n1)
//   w = A^-1 (sig n)  (cofactors of the symmetric A, as M3Inverse, init.c:518-540)
// and du_ij = -w_i n_j  (init.c:585 with evolution.c:1169-1183).
template <typename A>
__device__ __forceinline__ void green_w6(const A *__restrict__ G6, const A n[3], const A sr[6], const A si[6],
                                         A wr[3], A wi[3]) {
    const A m[6] = {n[0] * n[0], n[1] * n[1], n[2] * n[2], n[1] * n[2], n[0] * n[2], n[0] * n[1]};
    A Am[6];
#pragma unroll
    for (int a = 0; a < 6; ++a) {
        A acc = A(0);
#pragma unroll
        for (int b = 0; b < 6; ++b) acc += G6[6 * a + b] * m[b];
        Am[a] = acc;
    }
    // A = [[A0, A5, A4], [A5, A1, A3], [A4, A3, A2]]
    const A c00 = Am[1] * Am[2] - Am[3] * Am[3], c11 = Am[0] * Am[2] - Am[4] * Am[4], c22 = Am[0] * Am[1] - Am[5] * Am[5];
    const A c01 = Am[4] * Am[3] - Am[5] * Am[2], c02 = Am[5] * Am[3] - Am[4] * Am[1], c12 = Am[5] * Am[4] - Am[0] * Am[3];
    const A rdet = A(1) / (Am[0] * c00 + Am[5] * c01 + Am[4] * c02);
    // t = sig n with sig = [[s0, s5, s4], [s5, s1, s3], [s4, s3, s2]]
    const A t0r = sr[0] * n[0] + sr[5] * n[1] + sr[4] * n[2], t0i = si[0] * n[0] + si[5] * n[1] + si[4] * n[2];
    const A t1r = sr[5] * n[0] + sr[1] * n[1] + sr[3] * n[2], t1i = si[5] * n[0] + si[1] * n[1] + si[3] * n[2];
    const A t2r = sr[4] * n[0] + sr[3] * n[1] + sr[2] * n[2], t2i = si[4] * n[0] + si[3] * n[1] + si[2] * n[2];
    wr[0] = (c00 * t0r + c01 * t1r + c02 * t2r) * rdet;
    wi[0] = (c00 * t0i + c01 * t1i + c02 * t2i) * rdet;
    wr[1] = (c01 * t0r + c11 * t1r + c12 * t2r) * rdet;
    wi[1] = (c01 * t0i + c11 * t1i + c12 * t2i) * rdet;
    wr[2] = (c02 * t0r + c12 * t1r + c22 * t2r) * rdet;
    wi[2] = (c02 * t0i + c12 * t1i + c22 * t2i) * rdet;
}

// Symmetric tensor entries (00, 11, 22, 12, 02, 01) -> B basis (chg_basis opt 2), the inverse of b6_to_sym.
template <typename A>
__device__ __forceinline__ void sym_to_b6(const A t[6], A v[6]) {
    v[0] = A(SRX_R2) * (t[1] - t[0]);
    v[1] = A(SRX_R6) * (A(2) * t[2] - t[0] - t[1]);
    v[2] = A(2. * SRX_R2) * t[3];
    v[3] = A(2. * SRX_R2) * t[4];
    v[4] = A(2. * SRX_R2) * t[5];
    v[5] = A(SRX_R3) * (t[0] + t[1] + t[2]);
}

// Unit wave vector of k point (kx, ky, kz) (k != 0).
template <typename A>
__device__ __forceinline__ void unit_wave(int kx, int ky, int kz, int n0, int n1, int n2, A n[3]) {
    unit_k(kx, n0, n[0]);
    unit_k(ky, n1, n[1]);
    unit_k(kz, n2, n[2]);
    const A rg = A(1) / sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
    n[0] *= rg; n[1] *= rg; n[2] *= rg;
}

// Nyquist accumulator (see green_point): points on a Nyquist plane, kz = n2 / 2 first, then ky = n1 / 2,
// then kx = n0 / 2; three complex values each, [plane][comp][row][col] with the faster index last.
__device__ __forceinline__ bool nyq_slot(int kx, int ky, int kz, int n0, int n1, int n2, size_t &at, size_t &pitch) {
    const int H = n2 / 2 + 1;
    if (n2 % 2 == 0 && kz == n2 / 2) {
        at = (size_t)ky * n0 + kx;
        pitch = (size_t)n0 * n1;
        return true;
    }
    if (n1 % 2 == 0 && ky == n1 / 2) {
        at = 3 * (size_t)n0 * n1 + (size_t)kz * n0 + kx;
        pitch = (size_t)H * n0;
        return true;
    }
    if (n0 % 2 == 0 && kx == n0 / 2) {
        at = 3 * ((size_t)n0 * n1 + (size_t)H * n0) + (size_t)kz * n1 + ky;
        pitch = (size_t)H * n1;
        return true;
    }
    return false;
}

// Green operator at one k point (kx, ky, kz): B-basis spectrum q[6] of the stress -> the strain
// increment sym(du) in the B basis, out[6], computed in the spectrum's precision T (FP32 in the
// mixed-precision path, whose convolution is FP32 throughout).  The outer iterations need only the
// strain: the rotation part of du follows from the accumulated strain at the end of the increment
// (rotation_point), except on the Nyquist planes, where it is summed over the iterations in `nyq`
// (FP64; null: not kept; `first`: the increment's first iteration stores instead of adding).
// k = 0: -S0 (sig + dc6) for ElastBC 0, else 0 (init.c:558-569); dc6 is the grid sum of sig that a
// mean-subtracted (mixed precision) spectrum lacks, B basis.
// EDGE false: a row away from k = 0 and from the y and z Nyquist planes (NX: nor the x one).
template <typename T, bool EDGE = true, bool NX = true>
__device__ __forceinline__ void green_point(const DevConst *__restrict__ cst, const double dc6[6], int kx, int ky,
                                            int kz, int n0, int n1, int n2, const cx<T> q[6], cx<T> out[6],
                                            cx<double> *__restrict__ nyq, bool first) {
    using A = T;
    const A *G6;
    if constexpr (sizeof(T) == 4) G6 = cst->G6f;
    else G6 = cst->G6;
    if (EDGE && kx == 0 && ky == 0 && kz == 0) {
        double sr[6], si[6], vr[6], vi[6], br[6] = {0, 0, 0, 0, 0, 0}, bi[6] = {0, 0, 0, 0, 0, 0};
        if (cst->elast_bc == 0) {
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                vr[c] = (double)q[c].x;
                vi[c] = (double)q[c].y;
            }
            b6_to_sym(vr, sr);
            b6_to_sym(vi, si);
            double dcs[6], t9r[9], t9i[9], d9[9], er[6], ei[6];
            b6_to_sym(dc6, dcs);
            sym_to_t9(sr, t9r);
            sym_to_t9(si, t9i);
            sym_to_t9(dcs, d9);
            const int row[6] = {0, 4, 8, 5, 2, 1};
#pragma unroll
            for (int e = 0; e < 6; ++e) {
                double accr = 0.0, acci = 0.0;
                for (int r = 0; r < 9; ++r) {
                    accr += -cst->S0[row[e] * 9 + r] * (t9r[r] + d9[r]);
                    acci += -cst->S0[row[e] * 9 + r] * t9i[r];
                }
                er[e] = accr;
                ei[e] = acci;
            }
            sym_to_b6(er, br);
            sym_to_b6(ei, bi);
        }
#pragma unroll
        for (int c = 0; c < 6; ++c) out[c] = cx<T>{T(br[c]), T(bi[c])};
        return;
    }
    A nv[3];
    unit_wave(kx, ky, kz, n0, n1, n2, nv);
    const bool nyz = EDGE && (n2 % 2 == 0) && (kz == n2 / 2);
    const bool nyx = NX && (n0 % 2 == 0) && (kx == n0 / 2);
    const bool nyy = EDGE && (n1 % 2 == 0) && (ky == n1 / 2);
    A sr[6], si[6];
    {
        A vr[6], vi[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            vr[c] = (A)q[c].x;
            vi[c] = (A)q[c].y;
        }
        b6_to_sym(vr, sr);
        b6_to_sym(vi, si);
    }
    A wr[3], wi[3], er[6], ei[6];
    green_w6(G6, nv, sr, si, wr, wi);
    if (!(nyx || nyy || nyz)) {
        // du_ij = -w_i n_j: entries of sym(du)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int i = a == 2 ? 0 : a == 1 ? 0 : 1, j = a == 2 ? 1 : 2;   // (1,2), (0,2), (0,1)
            er[a] = -wr[a] * nv[a];
            ei[a] = -wi[a] * nv[a];
            er[3 + a] = A(-0.5) * (wr[i] * nv[j] + wr[j] * nv[i]);
            ei[3 + a] = A(-0.5) * (wi[i] * nv[j] + wi[j] * nv[i]);
        }
    } else {
        // Taking Re() of the inverse transform (evolution.c:1197) keeps the Hermitian part of du; at
        // a Nyquist index that part averages Gamma(n) with Gamma(n') where n' has the Nyquist
        // components negated.
        const A np[3] = {nyx ? -nv[0] : nv[0], nyy ? -nv[1] : nv[1], nyz ? -nv[2] : nv[2]};
        A wr2[3], wi2[3];
        green_w6(G6, np, sr, si, wr2, wi2);
        size_t at = 0, pitch = 0;
        nyq_slot(kx, ky, kz, n0, n1, n2, at, pitch);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int i = a == 2 ? 0 : a == 1 ? 0 : 1, j = a == 2 ? 1 : 2;
            er[a] = A(-0.5) * (wr[a] * nv[a] + wr2[a] * np[a]);
            ei[a] = A(-0.5) * (wi[a] * nv[a] + wi2[a] * np[a]);
            const A rij = A(-0.5) * (wr[i] * nv[j] + wr2[i] * np[j]), rji = A(-0.5) * (wr[j] * nv[i] + wr2[j] * np[i]);
            const A iij = A(-0.5) * (wi[i] * nv[j] + wi2[i] * np[j]), iji = A(-0.5) * (wi[j] * nv[i] + wi2[j] * np[i]);
            er[3 + a] = A(0.5) * (rij + rji);
            ei[3 + a] = A(0.5) * (iij + iji);
            if (nyq) {
                // one thread owns the point, so the atomic only spares it the wait for the old sum
                cx<double> *o = nyq + at + a * pitch;
                const cx<double> s = {0.5 * ((double)rij - (double)rji), 0.5 * ((double)iij - (double)iji)};
                if (first) {
                    *o = s;
                } else {
                    atomicAdd(&o->x, s.x);
                    atomicAdd(&o->y, s.y);
                }
            }
        }
    }
    A br[6], bi[6];
    sym_to_b6(er, br);
    sym_to_b6(ei, bi);
#pragma unroll
    for (int c = 0; c < 6; ++c) out[c] = cx<T>{br[c], bi[c]};
}

// The nine-component form: mixed precision on grids whose extents are not all powers of two.  There
// the FP32 wave vector idx * (1/n) - round(..) of a negative index carries a relative error near
// n / 2^25, so the kz = 0 plane of the strain is Hermitian only to that (3e-6 at n = 96), and the six
// symmetric components, transformed in other pairs than the nine, differ from them by 1e-5 of the
// strain after a few increments (2e-7 where the wave vectors are exact).
// Green operator at one k point (kx, ky, kz): B-basis spectrum q[6] of the stress -> du[9]
// (row-major), computed in the spectrum's precision T (FP32 in the mixed-precision path, whose
// convolution is FP32 throughout).  k = 0: -S0 (sig + dc6) for ElastBC 0, else 0 (init.c:558-569);
// dc6 is the grid sum of sig that a mean-subtracted (mixed precision) spectrum lacks, B basis.
template <typename T>
__device__ __forceinline__ void green_point9(const DevConst *__restrict__ cst, const double dc6[6], int kx, int ky,
                                            int kz, int n0, int n1, int n2, const cx<T> q[6], cx<T> out[9]) {
    using A = T;
    const A *G6;
    if constexpr (sizeof(T) == 4) G6 = cst->G6f;
    else G6 = cst->G6;
    if (kx == 0 && ky == 0 && kz == 0) {
        double sr[6], si[6], vr[6], vi[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            vr[c] = (double)q[c].x;
            vi[c] = (double)q[c].y;
        }
        b6_to_sym(vr, sr);
        b6_to_sym(vi, si);
        double dr[9], di[9];
        if (cst->elast_bc == 0) {
            double dcs[6], t9r[9], t9i[9];
            b6_to_sym(dc6, dcs);
            sym_to_t9(sr, t9r);
            sym_to_t9(si, t9i);
            double d9[9];
            sym_to_t9(dcs, d9);
            for (int qq = 0; qq < 9; ++qq) {
                double accr = 0.0, acci = 0.0;
                for (int r = 0; r < 9; ++r) {
                    accr += -cst->S0[qq * 9 + r] * (t9r[r] + d9[r]);
                    acci += -cst->S0[qq * 9 + r] * t9i[r];
                }
                dr[qq] = accr;
                di[qq] = acci;
            }
        } else {
#pragma unroll
            for (int qq = 0; qq < 9; ++qq) dr[qq] = di[qq] = 0.0;
        }
#pragma unroll
        for (int qq = 0; qq < 9; ++qq) out[qq] = cx<T>{T(dr[qq]), T(di[qq])};
        return;
    }
    A tzv, tyv, txv;
    unit_k(kz, n2, tzv);
    unit_k(ky, n1, tyv);
    unit_k(kx, n0, txv);
    const bool nyz = (n2 % 2 == 0) && (kz == n2 / 2);
    const bool nyx = (n0 % 2 == 0) && (kx == n0 / 2);
    const bool nyy = (n1 % 2 == 0) && (ky == n1 / 2);
    A sr[6], si[6];
    {
        A vr[6], vi[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            vr[c] = (A)q[c].x;
            vi[c] = (A)q[c].y;
        }
        b6_to_sym(vr, sr);
        b6_to_sym(vi, si);
    }
    A nv[3] = {txv, tyv, tzv};
    const A rg = A(1) / sqrt(nv[0] * nv[0] + nv[1] * nv[1] + nv[2] * nv[2]);
    nv[0] *= rg; nv[1] *= rg; nv[2] *= rg;
    A wr[3], wi[3];
    green_w6(G6, nv, sr, si, wr, wi);
    if (!(nyx || nyy || nyz)) {
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int b = 0; b < 3; ++b) out[3 * a + b] = cx<T>{T(-wr[a] * nv[b]), T(-wi[a] * nv[b])};
    } else {
        // Taking Re() of the inverse transform (evolution.c:1197) keeps the Hermitian part of du; at
        // a Nyquist index that part averages Gamma(n) with Gamma(n') where n' has the Nyquist
        // components negated.
        const A np[3] = {nyx ? -nv[0] : nv[0], nyy ? -nv[1] : nv[1], nyz ? -nv[2] : nv[2]};
        A wr2[3], wi2[3];
        green_w6(G6, np, sr, si, wr2, wi2);
#pragma unroll
        for (int a = 0; a < 3; ++a)
#pragma unroll
            for (int b = 0; b < 3; ++b)
                out[3 * a + b] = cx<T>{T(A(0.5) * (-wr[a] * nv[b] - wr2[a] * np[b])),
                                       T(A(0.5) * (-wi[a] * nv[b] - wi2[a] * np[b]))};
    }
}

// The same operator in factored form along an x row, for rows with ky and kz both off their
// Nyquist indices and not both 0.  With t the unnormalised wave vector (unit_k), n = t / |t| and
// du_ij = -w_i n_j, the y and z columns are t_y Y_i and t_z Y_i with Y_i = -w_i / |t|, and t_y, t_z
// are constant along the row, so the row's inverse x transforms of those six components are
// t_y IFFT(Y_i) and t_z IFFT(Y_i).  X_i is the x column.  At the x Nyquist index the Hermitian
// average of green_point9 keeps this form: Y_i = -(w_i + w'_i) / (2 |t|), X_i = -(w_i - w'_i) n_x / 2.
template <typename T>
__device__ __forceinline__ void green_point_xy(const DevConst *__restrict__ cst, int kx, int ky, int kz, int n0,
                                               int n1, int n2, const cx<T> q[6], cx<T> X[3], cx<T> Y[3]) {
    using A = T;
    const A *G6;
    if constexpr (sizeof(T) == 4) G6 = cst->G6f;
    else G6 = cst->G6;
    A tzv, tyv, txv;
    unit_k(kz, n2, tzv);
    unit_k(ky, n1, tyv);
    unit_k(kx, n0, txv);
    const bool nyx = (n0 % 2 == 0) && (kx == n0 / 2);
    A sr[6], si[6];
    {
        A vr[6], vi[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            vr[c] = (A)q[c].x;
            vi[c] = (A)q[c].y;
        }
        b6_to_sym(vr, sr);
        b6_to_sym(vi, si);
    }
    A nv[3] = {txv, tyv, tzv};
    const A rg = A(1) / sqrt(nv[0] * nv[0] + nv[1] * nv[1] + nv[2] * nv[2]);
    nv[0] *= rg; nv[1] *= rg; nv[2] *= rg;
    A wr[3], wi[3];
    green_w6(G6, nv, sr, si, wr, wi);
    if (!nyx) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            X[a] = cx<T>{-wr[a] * nv[0], -wi[a] * nv[0]};
            Y[a] = cx<T>{-wr[a] * rg, -wi[a] * rg};
        }
    } else {
        const A np[3] = {-nv[0], nv[1], nv[2]};
        A wr2[3], wi2[3];
        green_w6(G6, np, sr, si, wr2, wi2);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            X[a] = cx<T>{A(0.5) * (-wr[a] + wr2[a]) * nv[0], A(0.5) * (-wi[a] + wi2[a]) * nv[0]};
            Y[a] = cx<T>{A(-0.5) * (wr[a] + wr2[a]) * rg, A(-0.5) * (wi[a] + wi2[a]) * rg};
        }
    }
}

// Rotation part of the displacement gradient at one k point from the accumulated strain e (B basis).
// Off the Nyquist planes every iteration's du is u_i n_j, so with g = e n the antisymmetric part
// (u_i n_j - u_j n_i) / 2 is g_i n_j - g_j n_i (the u.n parts cancel): entries (1,2), (0,2), (0,1).
// On the Nyquist planes it is the sum kept by green_point; at k = 0 there is none.
template <typename T>
__device__ __forceinline__ void rotation_point(int kx, int ky, int kz, int n0, int n1, int n2, const cx<T> q[6],
                                               const cx<double> *__restrict__ nyq, cx<T> om[3]) {
    size_t at, pitch;
    if (kx == 0 && ky == 0 && kz == 0) {
#pragma unroll
        for (int a = 0; a < 3; ++a) om[a] = cx<T>{T(0), T(0)};
        return;
    }
    if (nyq_slot(kx, ky, kz, n0, n1, n2, at, pitch)) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const cx<double> s = nyq[at + a * pitch];
            om[a] = cx<T>{T(s.x), T(s.y)};
        }
        return;
    }
    T n[3], vr[6], vi[6], sr[6], si[6], gr[3], gi[3];
    unit_wave(kx, ky, kz, n0, n1, n2, n);
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        vr[c] = q[c].x;
        vi[c] = q[c].y;
    }
    b6_to_sym(vr, sr);
    b6_to_sym(vi, si);
    gr[0] = sr[0] * n[0] + sr[5] * n[1] + sr[4] * n[2]; gi[0] = si[0] * n[0] + si[5] * n[1] + si[4] * n[2];
    gr[1] = sr[5] * n[0] + sr[1] * n[1] + sr[3] * n[2]; gi[1] = si[5] * n[0] + si[1] * n[1] + si[3] * n[2];
    gr[2] = sr[4] * n[0] + sr[3] * n[1] + sr[2] * n[2]; gi[2] = si[4] * n[0] + si[3] * n[1] + si[2] * n[2];
    om[0] = cx<T>{gr[1] * n[2] - gr[2] * n[1], gi[1] * n[2] - gi[2] * n[1]};
    om[1] = cx<T>{gr[0] * n[2] - gr[2] * n[0], gi[0] * n[2] - gi[2] * n[0]};
    om[2] = cx<T>{gr[0] * n[1] - gr[1] * n[0], gi[0] * n[1] - gi[1] * n[0]};
}

// x pass with the Green operator.  grid: (ceil(n1/TY), H).  LDS: CO slots of TY*n0 (modes 0 and 2: ncomp).
// mode 1: forward x of 6 comps, Green, inverse x of CO comps (the solver pass)
// mode 3: forward x of 6 strain comps, rotation_point, inverse x of 3 comps (end of increment)
// mode 0: forward x only (ncomp comps, testing)   mode 2: inverse x only (testing)
template <typename T, int MAXB, int CO>
__global__ void __launch_bounds__(FFT_BLOCK) k_green_x(cx<T> *__restrict__ spec, int n0, int n1, int n2, FftStages px,
                                                       FastDiv dn0, TileDiv dt,
                                                       const cx<T> *__restrict__ tw, int TY, int mode, int ncomp,
                                                       const DevConst *__restrict__ cst,
                                                       const IterCtl *__restrict__ ctl, cx<double> *__restrict__ nyq) {
    if (ctl && ctl->done) return;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T> *buf = reinterpret_cast<cx<T> *>(smem_raw);
    const int H = n2 / 2 + 1;
    const int y0 = blockIdx.x * TY;
    const int ty = min(TY, n1 - y0);
    const int kz = blockIdx.y;
    const size_t plane = (size_t)n0 * n1;
    const int slot = ty * n0;
    const int cin = mode & 1 ? 6 : ncomp;
    const int cout = mode == 1 ? CO : mode == 3 ? 3 : ncomp;
    const FastDiv dslot = dt.of(ty == TY);
    cx<T> *stw = buf + (mode & 1 ? CO : ncomp) * slot;
    for (int i = threadIdx.x; i < n0; i += FFT_BLOCK) stw[i] = tw[i];
    // the block's rows of one component are contiguous: y0 * n0 .. (y0 + ty) * n0 of plane kz
    chunked_copy<cx<T>>(
        cin * slot,
        [&](int i) {
            const int c = dslot.div(i), r = i - c * slot;
            return spec[((size_t)c * H + kz) * plane + (size_t)y0 * n0 + r];
        },
        [&](int i, cx<T> v) { buf[i] = v; });
    __syncthreads();
    if (mode != 2) lds_fft<T, MAXB, true, false>(buf, cin * ty, px, stw, -1, n0);
    if (mode == 1) {
        double dc6[6] = {0, 0, 0, 0, 0, 0};
        if (ctl)
            for (int k = 0; k < 6; ++k) dc6[k] = ctl->dcs6[k];
        const bool first = ctl && ctl->iter == 0;
        for (int i = threadIdx.x; i < slot; i += FFT_BLOCK) {
            const int yy = dn0.div(i), kx = i - yy * n0, ky = y0 + yy;
            cx<T> q[6], o[CO];
#pragma unroll
            for (int c = 0; c < 6; ++c) q[c] = buf[c * slot + i];
            if constexpr (CO == 9) green_point9(cst, dc6, kx, ky, kz, n0, n1, n2, q, o);
            else green_point<T>(cst, dc6, kx, ky, kz, n0, n1, n2, q, o, nyq, first);
#pragma unroll
            for (int c = 0; c < CO; ++c) buf[c * slot + i] = o[c];
        }
        __syncthreads();
    } else if (mode == 3) {
        for (int i = threadIdx.x; i < slot; i += FFT_BLOCK) {
            const int yy = dn0.div(i), kx = i - yy * n0, ky = y0 + yy;
            cx<T> q[6], o[3];
#pragma unroll
            for (int c = 0; c < 6; ++c) q[c] = buf[c * slot + i];
            rotation_point(kx, ky, kz, n0, n1, n2, q, nyq, o);
#pragma unroll
            for (int c = 0; c < 3; ++c) buf[c * slot + i] = o[c];
        }
        __syncthreads();
    }
    if (mode != 0) lds_fft<T, MAXB, true, false>(buf, cout * ty, px, stw, +1, n0);
    for (int i = threadIdx.x; i < cout * slot; i += FFT_BLOCK) {
        const int c = dslot.div(i), r = i - c * slot;
        spec[((size_t)c * H + kz) * plane + (size_t)y0 * n0 + r] = buf[i];
    }
}

// ---------------------------------------------------------------------------
// The solver's x pass with one wavefront per (ky, kz) row and no LDS or barriers, for
// n0 = 64 NPL.  Lane l holds points l + 64 r (r < NPL) of each component.  Forward transform as
// four steps: an in-lane NPL-point DFT, the twiddle w_N^(l k1), then a 64-point radix-2
// decimation-in-frequency transform across lanes (partners l ^ h, h = 32 .. 1), which leaves
// X[k1 + NPL bitrev6(l)] in lane l, register k1.  The Green operator is applied in that order and
// the inverse runs the conjugate-transposed stages in reverse (decimation in time), which returns
// natural order: an unnormalised inverse DFT, as lds_fft with sign +1.
// grid: (ceil(n1 / 4), H), 256 threads (four rows per block).
// ---------------------------------------------------------------------------
__device__ __forceinline__ int brev6(int l) { return (int)(__brev((unsigned)l) >> 26); }

// value of lane ^ H: DPP quad permutations for H = 1, 2 (no LDS traffic), ds_swizzle's xor mode
// within 32 lanes for H = 4, 8, 16, ds_bpermute for H = 32
template <int H>
__device__ __forceinline__ int xor_lane(int v) {
    if constexpr (H == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false);   // quad_perm 1,0,3,2
    else if constexpr (H == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false);   // quad_perm 2,3,0,1
    else if constexpr (H < 32) return __builtin_amdgcn_ds_swizzle(v, (H << 10) | 0x1F);
    else return __shfl_xor(v, 32, 64);
}
template <int H>
__device__ __forceinline__ float xor_lane(float v) { return __int_as_float(xor_lane<H>(__float_as_int(v))); }
template <int H>
__device__ __forceinline__ double xor_lane(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = xor_lane<H>((int)(b & 0xffffffffll)), hi = xor_lane<H>((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int H, typename T>
__device__ __forceinline__ cx<T> shfl_xor_cx(cx<T> v) {
    return cx<T>{xor_lane<H>(v.x), xor_lane<H>(v.y)};
}
template <typename T>
__device__ __forceinline__ cx<T> conj_cx(cx<T> a) { return cx<T>{a.x, -a.y}; }

// Cross-lane stage ST (partner lane ^ h, h = 32 >> ST) and the ones after it, for C components at
// once: all partner values of a stage are requested before any is used, so one wait covers them.
// Branch free: with s = +1 in the lower lane of a pair and -1 in the upper one, and the upper
// lane's twiddle w (the lower lane's is 1),
//   decimation in frequency: lower x_lo + x_hi, upper (x_lo - x_hi) w  =  (u + s v) w'
//   decimation in time:      lower x_lo + w x_hi, upper x_lo - w x_hi  =  m_partner + s m,
//                            m = w' v (each upper lane multiplies its own value before the exchange)
// (u the partner's value, v the lane's own, w' = w in the upper lane and 1 in the lower one; a
// product by exactly 1 returns its operand, so the results equal the two-sided forms').  The last
// DIF and first DIT stage (h = 1) has w = 1 in every lane and no product.
template <typename T>
__device__ __forceinline__ cx<T> pair_twiddle(const cx<T> w, bool hi) {
    return cx<T>{hi ? w.x : T(1), hi ? w.y : T(0)};
}
template <typename T, int NPL, int C, int ST>
__device__ __forceinline__ void wave_dif_stage(cx<T> (&v)[C][NPL], const cx<T> ws[6], int lane) {
    if constexpr (ST < 6) {
        constexpr int h = 32 >> ST;
        const bool hi = lane & h;
        const T s = hi ? T(-1) : T(1);
        const cx<T> w = pair_twiddle(ws[ST], hi);
        cx<T> u[C][NPL];
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < NPL; ++k) u[c][k] = shfl_xor_cx<h>(v[c][k]);
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < NPL; ++k) {
                const cx<T> t{fma(s, v[c][k].x, u[c][k].x), fma(s, v[c][k].y, u[c][k].y)};
                v[c][k] = h == 1 ? t : cmul(t, w);
            }
        wave_dif_stage<T, NPL, C, ST + 1>(v, ws, lane);
    }
}
template <typename T, int NPL, int C, int ST>
__device__ __forceinline__ void wave_dit_stage(cx<T> (&v)[C][NPL], const cx<T> ws[6], int lane) {
    if constexpr (ST >= 0) {
        constexpr int h = 32 >> ST;
        const bool hi = lane & h;
        const T s = hi ? T(-1) : T(1);
        if constexpr (h != 1) {
            const cx<T> w = pair_twiddle(conj_cx(ws[ST]), hi);
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int k = 0; k < NPL; ++k) v[c][k] = cmul(v[c][k], w);
        }
        cx<T> u[C][NPL];
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < NPL; ++k) u[c][k] = shfl_xor_cx<h>(v[c][k]);
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int k = 0; k < NPL; ++k) v[c][k] = cx<T>{fma(s, v[c][k].x, u[c][k].x), fma(s, v[c][k].y, u[c][k].y)};
        wave_dit_stage<T, NPL, C, ST - 1>(v, ws, lane);
    }
}

template <typename T, int NPL, int C>
__device__ __forceinline__ void wave_fft_fwd(cx<T> (&v)[C][NPL], const cx<T> wl[], const cx<T> ws[6], int lane) {
    if constexpr (NPL > 1) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
            Dft<T, NPL>::run(v[c], -1);
#pragma unroll
            for (int k = 1; k < NPL; ++k) v[c][k] = cmul(v[c][k], wl[k - 1]);
        }
    }
    wave_dif_stage<T, NPL, C, 0>(v, ws, lane);
}

template <typename T, int NPL, int C>
__device__ __forceinline__ void wave_fft_inv(cx<T> (&v)[C][NPL], const cx<T> wl[], const cx<T> ws[6], int lane) {
    wave_dit_stage<T, NPL, C, 5>(v, ws, lane);
    if constexpr (NPL > 1) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
#pragma unroll
            for (int k = 1; k < NPL; ++k) v[c][k] = cmul(v[c][k], conj_cx(wl[k - 1]));
            Dft<T, NPL>::run(v[c], +1);
        }
    }
}

// blocks of the wavefront Green kernel per compute unit the register allocator targets
#ifndef SRX_GREEN_MIN_BLOCKS
#define SRX_GREEN_MIN_BLOCKS 1
#endif
// CO = 6: stress -> strain increment; 9: stress -> displacement gradient increment; 3: the
// end-of-increment pass, strain -> rotation part (rotation_point).
template <typename T, int NPL, int CO>
__global__ void __launch_bounds__(256, SRX_GREEN_MIN_BLOCKS) k_green_wave(cx<T> *__restrict__ spec, int n1, int n2,
                                                    const cx<T> *__restrict__ tw, const DevConst *__restrict__ cst,
                                                    const IterCtl *__restrict__ ctl, cx<double> *__restrict__ nyq) {
    if (ctl && ctl->done) return;
    constexpr int N = 64 * NPL;
    const int lane = threadIdx.x & 63;
    const int ky = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int kz = blockIdx.y;
    if (ky >= n1) return;   // the whole wavefront: no barrier follows
    const int H = n2 / 2 + 1;
    const size_t plane = (size_t)N * n1;
    double dc6[6] = {0, 0, 0, 0, 0, 0};
    bool first = false;
    if (ctl) {
        for (int k = 0; k < 6; ++k) dc6[k] = ctl->dcs6[k];
        first = ctl->iter == 0;
    }
    // twiddles of this lane: w_N^(l k1) for the four-step split, and W_2h^(l mod h) = w_N^(..) of
    // each cross-lane stage
    cx<T> wl[NPL > 1 ? NPL - 1 : 1];
#pragma unroll
    for (int k = 1; k < NPL; ++k) wl[k - 1] = tw[lane * k];
    cx<T> ws[6];
#pragma unroll
    for (int st = 0; st < 6; ++st) {
        const int h = 32 >> st;
        ws[st] = tw[(lane & (h - 1)) * (32 / h) * NPL];
    }
    const size_t row = (size_t)kz * plane + (size_t)ky * N + lane;
    const size_t cstride = (size_t)H * plane;
    cx<T> q[6][NPL];
#pragma unroll
    for (int c = 0; c < 6; ++c)
#pragma unroll
        for (int r = 0; r < NPL; ++r) q[c][r] = spec[c * cstride + row + 64 * r];
    wave_fft_fwd<T, NPL, 6>(q, wl, ws, lane);
    const int kb = NPL * brev6(lane);
    if constexpr (CO == 9) {
        // the row's Green operator in factored form (6 inverse transforms) unless ky or kz is at its
        // Nyquist index or the row holds k = 0 (wavefront-uniform)
        const bool factored = !((n1 % 2 == 0 && ky == n1 / 2) || (n2 % 2 == 0 && kz == n2 / 2) || (ky == 0 && kz == 0));
        if (factored) {
            cx<T> o[6][NPL];   // X_0..2, Y_0..2
#pragma unroll
            for (int r = 0; r < NPL; ++r) {
                cx<T> qi[6], xi[3], yi[3];
#pragma unroll
                for (int c = 0; c < 6; ++c) qi[c] = q[c][r];
                green_point_xy(cst, r + kb, ky, kz, N, n1, n2, qi, xi, yi);
#pragma unroll
                for (int a = 0; a < 3; ++a) { o[a][r] = xi[a]; o[3 + a][r] = yi[a]; }
            }
            wave_fft_inv<T, NPL, 6>(o, wl, ws, lane);
            T ty, tz;
            unit_k(ky, n1, ty);
            unit_k(kz, n2, tz);
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int r = 0; r < NPL; ++r) {
                    const cx<T> y = o[3 + a][r];
                    spec[(3 * a) * cstride + row + 64 * r] = o[a][r];
                    spec[(3 * a + 1) * cstride + row + 64 * r] = cx<T>{ty * y.x, ty * y.y};
                    spec[(3 * a + 2) * cstride + row + 64 * r] = cx<T>{tz * y.x, tz * y.y};
                }
            return;
        }
    }
    cx<T> o[CO][NPL];
    // a row at the y or z Nyquist index or with k = 0 (wavefront-uniform), about 2% of them at 128^3;
    // in the others only the lane with kx = N / 2 (lane 1, register 0) takes the averaged form
    const bool edge = (n1 % 2 == 0 && ky == n1 / 2) || (n2 % 2 == 0 && kz == n2 / 2) || (ky == 0 && kz == 0);
    auto points = [&](auto point) {
#pragma unroll
        for (int r = 0; r < NPL; ++r) {
            cx<T> qi[6], oi[CO];
#pragma unroll
            for (int c = 0; c < 6; ++c) qi[c] = q[c][r];
            point(r, qi, oi);
#pragma unroll
            for (int c = 0; c < CO; ++c) o[c][r] = oi[c];
        }
    };
    if constexpr (CO == 9) {
        points([&](int r, const cx<T> *qi, cx<T> *oi) { green_point9(cst, dc6, r + kb, ky, kz, N, n1, n2, qi, oi); });
    } else if constexpr (CO == 3) {
        points([&](int r, const cx<T> *qi, cx<T> *oi) { rotation_point(r + kb, ky, kz, N, n1, n2, qi, nyq, oi); });
    } else if (edge) {
        points([&](int r, const cx<T> *qi, cx<T> *oi) {
            green_point<T>(cst, dc6, r + kb, ky, kz, N, n1, n2, qi, oi, nyq, first);
        });
    } else {
        points([&](int r, const cx<T> *qi, cx<T> *oi) {
            if (r == 0) green_point<T, false, true>(cst, dc6, r + kb, ky, kz, N, n1, n2, qi, oi, nyq, first);
            else green_point<T, false, false>(cst, dc6, r + kb, ky, kz, N, n1, n2, qi, oi, nyq, first);
        });
    }
    wave_fft_inv<T, NPL, CO>(o, wl, ws, lane);
#pragma unroll
    for (int c = 0; c < CO; ++c)
#pragma unroll
        for (int r = 0; r < NPL; ++r) spec[c * cstride + row + 64 * r] = o[c][r];
}

// ---------------------------------------------------------------------------
// The y, x and Green passes of small planes in one kernel: a block holds the whole plane kz of every
// component in LDS, laid out as the z passes' B ([x][y]), and runs the y transforms, the x transforms
// (elements a row apart), the Green operator and both inverses there, stage by stage as stockham_stage.
// grid: (H), PLANE_BLOCK threads.  LDS: CO slots of n0 rows of n1 | 1, then the two twiddle tables.
// Bound by the chain of one block's stages.  Against the three passes it saves two launches and the
// spectra's trips through memory, an outer iteration in FP64: 8^3 44.0 -> 37.7 us, 12^3 45.7 -> 41.6, 16^3
// 46.3 -> 43.6, 16 x 16 x 256 72.1 -> 63.0.  Long planes, whose x pass would be the wavefront Green pass:
// 64 x 1 x 4 39.1 -> 36.9, 64 x 4 x 64 46.2 -> 46.6, 128 x 2 x 64 49.0 -> 48.3, 256 x 1 x 128 59.0 -> 50.6,
// 4 x 64 x 64 51.0 -> 47.5 (the one slower by more than 1%: 64 x 4 x 8, 41.6 -> 42.9; in mixed
// precision all are faster).  Beyond 256 points a plane's chain is longer than the three
// launches (18^3 48.9 -> 50.9, 24^3 49.5 -> 53.4): PLANE_POINTS.
// ---------------------------------------------------------------------------
constexpr int PLANE_BLOCK = 512, PLANE_POINTS = 256;
// One stage of a plane's transforms along one axis: nc components of np pencils, pencil stride ps,
// element stride es.  In place like stockham_stage.
template <typename T, int R, int CO>
__device__ __forceinline__ void plane_stage(cx<T> *buf, int nc, FastDiv dnp, int slot, int ps, int es,
                                            const FftStages::Stage &sg, const cx<T> *__restrict__ tw, int sign) {
    constexpr int MB = (CO * PLANE_POINTS + PLANE_BLOCK * R - 1) / (PLANE_BLOCK * R);
    const FastDiv dnb = sg.nb, dL = sg.dL;
    const int nb = dnb.d, L = dL.d, tstep = sg.tstep, np = dnp.d;
    const int total = nc * np * nb;
    cx<T> v[MB][R];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        const int t = threadIdx.x + m * PLANE_BLOCK;
        if (t < total) {
            const int p = dnb.div(t), j = t - p * nb;
            const int c = dnp.div(p);
            const cx<T> *src = buf + c * slot + (p - c * np) * ps + j * es;
#pragma unroll
            for (int r = 0; r < R; ++r) v[m][r] = src[r * nb * es];
        }
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        const int t = threadIdx.x + m * PLANE_BLOCK;
        if (t < total) {
            const int p = dnb.div(t), j = t - p * nb;
            const int c = dnp.div(p);
            const int jl = dL.div(j), k = j - jl * L;
            if (k) {
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    cx<T> w = tw[r * k * tstep];
                    if (sign > 0) w.y = -w.y;
                    v[m][r] = cmul(v[m][r], w);
                }
            }
            Dft<T, R>::run(v[m], sign);
            cx<T> *dst = buf + c * slot + (p - c * np) * ps + (jl * L * R + k) * es;
#pragma unroll
            for (int r = 0; r < R; ++r) dst[r * L * es] = v[m][r];
        }
    }
    __syncthreads();
}
struct PlanePlans {
    FftStages ax[2];   // x, y
    FastDiv n[2], plane;
};
template <typename T, int CO>
__global__ void __launch_bounds__(PLANE_BLOCK) k_plane(cx<T> *__restrict__ spec, int n0, int n1, int n2, PlanePlans pl,
                                                       const cx<T> *__restrict__ twx, const cx<T> *__restrict__ twy,
                                                       const DevConst *__restrict__ cst,
                                                       const IterCtl *__restrict__ ctl, cx<double> *__restrict__ nyq) {
    if (ctl && ctl->done) return;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T> *buf = reinterpret_cast<cx<T> *>(smem_raw);
    const int P = n1 | 1, slot = n0 * P, plane = n0 * n1;
    cx<T> *stw = buf + CO * slot;
    const int H = n2 / 2 + 1, kz = blockIdx.x;
    const FastDiv dplane = pl.plane, dn1 = pl.n[1];
    for (int i = threadIdx.x; i < n0 + n1; i += PLANE_BLOCK) stw[i] = i < n0 ? twx[i] : twy[i - n0];
    auto at = [&](int c, int r) {   // LDS position of point r = x n1 + y
        const int x = dn1.div(r);
        return c * slot + x * P + (r - x * n1);
    };
    for (int i = threadIdx.x; i < 6 * plane; i += PLANE_BLOCK) {
        const int c = dplane.div(i), r = i - c * plane;
        buf[at(c, r)] = spec[((size_t)c * H + kz) * plane + r];
    }
    __syncthreads();
    // forward y and x, the Green operator, inverse x and y: one copy of the stages' code for the four
#pragma unroll 1
    for (int pass = 0; pass < 4; ++pass) {
        const int ax = pass == 0 || pass == 3, sign = pass < 2 ? -1 : 1;
        const int nc = pass < 2 ? 6 : CO, ps = ax ? P : 1, es = ax ? 1 : P;
        const FastDiv np = pl.n[1 - ax];
        const cx<T> *tw = stw + (ax ? n0 : 0);
        const FftStages &st = pl.ax[ax];
#pragma unroll 1
        for (int s = 0; s < st.nst; ++s) {
            const FftStages::Stage sg = st.st[s];
            switch (sg.R) {
            case 8: plane_stage<T, 8, CO>(buf, nc, np, slot, ps, es, sg, tw, sign); break;
            case 4: plane_stage<T, 4, CO>(buf, nc, np, slot, ps, es, sg, tw, sign); break;
            case 2: plane_stage<T, 2, CO>(buf, nc, np, slot, ps, es, sg, tw, sign); break;
            case 3: plane_stage<T, 3, CO>(buf, nc, np, slot, ps, es, sg, tw, sign); break;
            default: plane_stage<T, 5, CO>(buf, nc, np, slot, ps, es, sg, tw, sign); break;
            }
        }
        if (pass == 1) {
            double dc6[6] = {0, 0, 0, 0, 0, 0};
            if (ctl)
                for (int k = 0; k < 6; ++k) dc6[k] = ctl->dcs6[k];
            const bool first = ctl && ctl->iter == 0;
            for (int i = threadIdx.x; i < plane; i += PLANE_BLOCK) {
                const int kx = dn1.div(i), ky = i - kx * n1, b = kx * P + ky;
                cx<T> q[6], o[CO];
#pragma unroll
                for (int c = 0; c < 6; ++c) q[c] = buf[c * slot + b];
                if constexpr (CO == 9) green_point9(cst, dc6, kx, ky, kz, n0, n1, n2, q, o);
                else green_point<T>(cst, dc6, kx, ky, kz, n0, n1, n2, q, o, nyq, first);
#pragma unroll
                for (int c = 0; c < CO; ++c) buf[c * slot + b] = o[c];
            }
            __syncthreads();
        }
    }
    for (int i = threadIdx.x; i < CO * plane; i += PLANE_BLOCK) {
        const int c = dplane.div(i), r = i - c * plane;
        spec[((size_t)c * H + kz) * plane + r] = buf[at(c, r)];
    }
}

// ---------------------------------------------------------------------------
// inverse z (c2r) fused with Eq. 15: ee[c] += ddg6[c] + Re(IFFT)/Nxyz for the six strain components,
// or the same for the nine of DisGrad with ddg
// grid: (ceil(n0 n1 / TY), component pairs); `ee` is an output (scale mode) when accumulate=0
// ---------------------------------------------------------------------------
template <typename T, bool SW>
__global__ void __launch_bounds__(FFT_BLOCK) SRX_ZPASS_ATTR k_inv_z(const cx<T> *__restrict__ specB, double *__restrict__ ee,
                                                     int ncomp, int n0, int n1, int n2, FftStages pz,
                                                     FastDiv dn2, TileDiv dt, const cx<T> *__restrict__ tw, int TY, int accumulate,
                                                     double divisor, const IterCtl *__restrict__ ctl) {
    if (ctl && ctl->done) return;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    cx<T> *buf = reinterpret_cast<cx<T> *>(smem_raw);
    // SW: compile-time stages, swizzled pencils at pitch n2 + 2; else runtime stages, plain, n2 + 1
    constexpr bool sw = SW;
    const int P = SW ? n2 + 2 : n2 + 1;   // padded pencil pitch
    cx<T> *stw = buf + TY * P;
    for (int i = threadIdx.x; i < n2; i += FFT_BLOCK) stw[i] = tw[i];
    const int rows = n0 * n1, row0 = blockIdx.x * TY;
    const int ty = min(TY, rows - row0);
    const int H = n2 / 2 + 1;
    const size_t N = (size_t)rows * n2;
    const size_t HS = (size_t)H * rows;
    const double *add = ctl ? (ncomp == 9 ? ctl->ddg : ctl->ddg6) : nullptr;
    const FastDiv dty = dt.of(ty == TY);
    // 1/Nxyz: a power of two for the usual grids, where the product equals the division
    const double rdiv = 1.0 / divisor;
    // one pair of components per block along grid y
    for (int ca = 2 * blockIdx.y; ca < ncomp && ca < 2 * blockIdx.y + 2; ca += 2) {
        const int cb = ca + 1;
        const bool two = cb < ncomp;
        const cx<T> *sa = specB + ca * HS, *sb = specB + (two ? cb : ca) * HS;
        const double aa = add ? add[ca] : 0.0, ab = add && two ? add[cb] : 0.0;
        chunked_copy<cx2<T>>(
            H * ty,
            [&](int i) {
                const int kz = dty.div(i), yy = i - kz * ty;
                const size_t o = (size_t)kz * rows + row0 + yy;
                return cx2<T>{sa[o], sb[o]};
            },
            [&](int i, cx2<T> v) {
                const int kz = dty.div(i), yy = i - kz * ty;
                const cx<T> A = v.a;
                const cx<T> B = two ? v.b : cx<T>{T(0), T(0)};
                // The transform of a real row has no imaginary part at kz = 0 and n2 / 2.  What FP32 rounding left
                // there would pass into the pair's other component, and six components, unlike nine, hold
                // each shear once and average nothing: strain error at 64 x 64 x 1 in mixed precision
                // 4.1e-7 with it, 1.4e-7 without (nine components 3.7e-7).  (The nine, and a caller's spectra,
                // keep it; so does FP64, at 1e-16, where leaving it out cost 0.6 of 8.5 us at 45 x 60 x 50.)
                const bool end = sizeof(T) == 4 && accumulate && ncomp == 6 && (kz == 0 || 2 * kz == n2);
                buf[yy * P + (sw ? lds_swz(kz) : kz)] = end ? cx<T>{A.x, B.x} : cx<T>{A.x - B.y, A.y + B.x};
                if (kz >= 1 && kz <= n2 - H)
                    buf[yy * P + (sw ? lds_swz(n2 - kz) : n2 - kz)] = cx<T>{A.x + B.y, B.x - A.y};
            });
        // the strain of the block's rows (contiguous): the first chunk of each thread's values is
        // loaded before the transform, so its round trip to HBM overlaps the LDS work
        double *da = ee + ca * N, *db = ee + (two ? cb : ca) * N;
        const size_t g0 = (size_t)row0 * n2;
        const int tot = ty * n2;
        cx<double> pre[FFT_CHUNK];
        if (accumulate) {
#pragma unroll
            for (int e = 0; e < FFT_CHUNK; ++e) {
                const int i = min(e * FFT_BLOCK + (int)threadIdx.x, tot - 1);
                pre[e] = cx<double>{da[g0 + i], db[g0 + i]};
            }
        }
        __syncthreads();
        if constexpr (SW) lds_fft<T, 2, true, true>(buf, ty, pz, stw, +1, P);
        else lds_fft<T, 2, false, false>(buf, ty, pz, stw, +1, P);
        for (int b = 0; b < tot; b += FFT_CHUNK * FFT_BLOCK) {
            if (accumulate && b > 0) {
#pragma unroll
                for (int e = 0; e < FFT_CHUNK; ++e) {
                    const int i = min(b + e * FFT_BLOCK + (int)threadIdx.x, tot - 1);
                    pre[e] = cx<double>{da[g0 + i], db[g0 + i]};
                }
            }
#pragma unroll
            for (int e = 0; e < FFT_CHUNK; ++e) {
                const int i = b + e * FFT_BLOCK + (int)threadIdx.x;
                if (i < tot) {
                    const int yy = dn2.div(i), z = i - yy * n2;
                    const cx<T> v = buf[yy * P + (sw ? lds_swz(z) : z)];
                    if (accumulate) {
                        da[g0 + i] = pre[e].x + (aa + (double)v.x * rdiv);
                        if (two) db[g0 + i] = pre[e].y + (ab + (double)v.y * rdiv);
                    } else {
                        da[g0 + i] = (double)v.x * rdiv;
                        if (two) db[g0 + i] = (double)v.y * rdiv;
                    }
                }
            }
        }
        __syncthreads();
    }
}


// ---------------------------------------------------------------------------
// host launch wrappers
// ---------------------------------------------------------------------------
static int min_radix(const FftPlan &p) {
    int m = 1 << 30;
    for (int i = 0; i < p.nst; ++i) m = p.rad[i] < m ? p.rad[i] : m;
    return p.nst ? m : 1;
}

bool make_plan(int n, FftPlan &p) {
    p.n = n;
    p.nst = 0;
    int m = n;
    if (n < 1 || n > 1024) return false;
    // powers of two: as many radix-8 stages as possible without leaving a radix-2 stage
    // (2^7 = 8*4*4, 2^8 = 8*8*4), then radix 3 and 5
    int k2 = 0;
    while (m % 2 == 0) { ++k2; m /= 2; }
    int n8 = k2 / 3, n4 = 0, n2 = 0;
    if (k2 % 3 == 1) { if (n8 > 0) { --n8; n4 = 2; } else { n2 = 1; } }
    else if (k2 % 3 == 2) n4 = 1;
    for (int i = 0; i < n8; ++i) p.rad[p.nst++] = 8;
    for (int i = 0; i < n4; ++i) p.rad[p.nst++] = 4;
    for (int i = 0; i < n2; ++i) p.rad[p.nst++] = 2;
    while (m % 3 == 0) { p.rad[p.nst++] = 3; m /= 3; }
    while (m % 5 == 0) { p.rad[p.nst++] = 5; m /= 5; }
    if (p.nst > MAX_RADIX_STAGES) return false;
    return m == 1;
}

// Radix plans of length n the tuner may time: make_plan's first, then every split of the power of
// two into radix-8 and radix-4 stages with at most one radix-2 stage (more radix-2 stages only add
// passes over LDS), each in make_plan's order (8s, 4s, the 2, then 3s and 5s) and in the reverse
// order.  Returns the number written to out (at most cap); 0 when make_plan rejects n.
int plan_candidates(int n, FftPlan *out, int cap) {
    FftPlan d;
    if (cap < 1 || !make_plan(n, d)) return 0;
    int cnt = 0;
    auto add = [&](const FftPlan &p) {
        for (int i = 0; i < cnt; ++i) {
            bool same = out[i].nst == p.nst;
            for (int s = 0; same && s < p.nst; ++s) same = out[i].rad[s] == p.rad[s];
            if (same) return;
        }
        if (cnt < cap) out[cnt++] = p;
    };
    add(d);
    int m = n, k2 = 0, k3 = 0, k5 = 0;
    while (m % 2 == 0) { ++k2; m /= 2; }
    while (m % 3 == 0) { ++k3; m /= 3; }
    while (m % 5 == 0) { ++k5; m /= 5; }
    for (int n8 = k2 / 3; n8 >= 0; --n8)
        for (int n4 = (k2 - 3 * n8) / 2; n4 >= 0; --n4) {
            const int n2 = k2 - 3 * n8 - 2 * n4;
            if (n2 > 1 || n8 + n4 + n2 + k3 + k5 > MAX_RADIX_STAGES) continue;
            FftPlan p;
            p.n = n;
            p.nst = 0;
            for (int i = 0; i < n8; ++i) p.rad[p.nst++] = 8;
            for (int i = 0; i < n4; ++i) p.rad[p.nst++] = 4;
            for (int i = 0; i < n2; ++i) p.rad[p.nst++] = 2;
            for (int i = 0; i < k3; ++i) p.rad[p.nst++] = 3;
            for (int i = 0; i < k5; ++i) p.rad[p.nst++] = 5;
            add(p);
            FftPlan r = p;
            for (int s = 0; s < p.nst; ++s) r.rad[s] = p.rad[p.nst - 1 - s];
            add(r);
        }
    return cnt;
}

// LDS budget of one FFT block (bytes)
constexpr int FFT_LDS_MAX = 48 * 1024;

// LDS of a y or z pass: t pencils at the padded pitch (n + 2 swizzled, else n + 1), then the
// twiddle table
static size_t padded_lds(int t, int n, size_t csz, bool sw) { return ((size_t)t * (sw ? n + 2 : n + 1) + n) * csz; }

// Whether a z or y pass runs plan p with the compile-time stages and swizzled pencils (the kernels'
// SW = true instantiation): lengths 32..256 with make_plan's radices.  Other plans run the runtime
// stages on plain pencils (SW = false), a separate instantiation so that neither pays for the
// other's registers.
static bool plan_swizzled(const FftPlan &p) {
    if (p.n != 32 && p.n != 64 && p.n != 128 && p.n != 256) return false;
    FftPlan d;
    make_plan(p.n, d);
    if (d.nst != p.nst) return false;
    for (int s = 0; s < p.nst; ++s)
        if (d.rad[s] != p.rad[s]) return false;
    return true;
}

// largest tile count t with t*n/minrad <= maxb*FFT_BLOCK, t*comps*lds_pitch(n) complex values within
// FFT_LDS_MAX and t <= cap
static int tile_for(const FftPlan &p, int per_tile_comps, int maxb, int cap, int prec) {
    const int mr = min_radix(p);
    int t = (maxb * FFT_BLOCK * mr) / (p.n * per_tile_comps);
    const int csz = prec == 0 ? 16 : 8;
    const int tl = (FFT_LDS_MAX - p.n * csz) / (per_tile_comps * lds_pitch(p.n) * csz);
    if (t > tl) t = tl;
    if (t > cap) t = cap;
    if (t < 1) t = 1;
    return t;
}

// Rows (pencils) per block of a z or y pass: `tile` if it is valid, else the largest that fits, up to
// 16, or up to what makes 1024 elements of short rows (a wavefront's loads then move 64 of them, not a
// fraction of a row).
static int zy_tile(const FftPlan &p, int rows, int tile, int prec) {
    const int cap = p.n >= 64 ? 16 : 1024 / p.n;
    const int t = tile_for(p, 1, 2, rows < cap ? rows : cap, prec);
    return tile >= 1 && tile <= t ? tile : t;
}

// Largest valid tile of pass `pass` (0 forward z, 1 forward y, 2 Green x, 3 inverse y, 4 inverse
// z); p is the plan of the pass's axis.
int fft_tile_max(int pass, const int n[3], const FftPlan &p, int prec, int comps) {
    switch (pass) {
    case 0: case 4: return zy_tile(p, n[0] * n[1], 0, prec);
    case 1: case 3: return zy_tile(p, n[0], 0, prec);
    default: {   // Green x pass: `comps` slots of t rows, up to 4 butterflies per thread
        int t = (4 * FFT_BLOCK * min_radix(p)) / (comps * p.n);
        const int csz = prec == 0 ? 16 : 8;
        const int tl = (FFT_LDS_MAX / csz - p.n) / (comps * p.n);
        t = t < tl ? t : tl;
        t = t < n[1] ? t : n[1];
        return t < 1 ? 1 : (t > 4 ? 4 : t);
    }
    }
}

template <typename T>
static hipError_t launch_fwd_z(hipStream_t s, const double *in, void *specB, int ncomp, const int n[3], const FftPlan &pz,
                         const void *twz, const IterCtl *ctl, int tile, int prec) {
    const int rows = n[0] * n[1], TY = zy_tile(pz, rows, tile, prec);
    const bool sw = plan_swizzled(pz);
    const dim3 grid((rows + TY - 1) / TY, (ncomp + 1) / 2);
    const size_t sm = padded_lds(TY, n[2], sizeof(cx<T>), sw);
    if (sw)
        SRX_LAUNCH((k_fwd_z<T, true>), grid, dim3(FFT_BLOCK), sm, s, in, (cx<T> *)specB, ncomp, n[0], n[1], n[2], FftStages(pz),
                   FastDiv(n[2]), TileDiv(rows, TY, 1), (const cx<T> *)twz, TY, ctl);
    else
        SRX_LAUNCH((k_fwd_z<T, false>), grid, dim3(FFT_BLOCK), sm, s, in, (cx<T> *)specB, ncomp, n[0], n[1], n[2], FftStages(pz),
                   FastDiv(n[2]), TileDiv(rows, TY, 1), (const cx<T> *)twz, TY, ctl);
    return check_launch("fwd_z");
}

void launch_fft_fwd_z(hipStream_t s, int prec, const double *sig, void *specB, const int n[3], const FftPlan &pz,
                      const void *twz, const IterCtl *ctl, int tile) {
    if (prec == 0) launch_fwd_z<double>(s, sig, specB, 6, n, pz, twz, ctl, tile, prec);
    else launch_fwd_z<float>(s, sig, specB, 6, n, pz, twz, ctl, tile, prec);
}

hipError_t launch_fft_y(hipStream_t s, int prec, const void *in, void *out, int ncomp, int sign, int b_to_c, const int n[3],
                  const FftPlan &py, const void *twy, const IterCtl *ctl, int tile) {
    (void)sign;
    const int TX = zy_tile(py, n[0], tile, prec);
    const bool sw = plan_swizzled(py);
    const int H = n[2] / 2 + 1;
    dim3 grid((n[0] + TX - 1) / TX, H, ncomp);
    if (prec == 0) {
        size_t sm = padded_lds(TX, n[1], sizeof(cx<double>), sw);
        if (sw)
            SRX_LAUNCH((k_fft_y<double, true>), grid, dim3(FFT_BLOCK), sm, s, (const cx<double> *)in, (cx<double> *)out,
                           n[0], n[1], n[2], b_to_c, FftStages(py), FastDiv(n[1]), TileDiv(n[0], TX, 1), (const cx<double> *)twy, TX, ctl);
        else
            SRX_LAUNCH((k_fft_y<double, false>), grid, dim3(FFT_BLOCK), sm, s, (const cx<double> *)in, (cx<double> *)out,
                           n[0], n[1], n[2], b_to_c, FftStages(py), FastDiv(n[1]), TileDiv(n[0], TX, 1), (const cx<double> *)twy, TX, ctl);
    } else {
        size_t sm = padded_lds(TX, n[1], sizeof(cx<float>), sw);
        if (sw)
            SRX_LAUNCH((k_fft_y<float, true>), grid, dim3(FFT_BLOCK), sm, s, (const cx<float> *)in, (cx<float> *)out,
                           n[0], n[1], n[2], b_to_c, FftStages(py), FastDiv(n[1]), TileDiv(n[0], TX, 1), (const cx<float> *)twy, TX, ctl);
        else
            SRX_LAUNCH((k_fft_y<float, false>), grid, dim3(FFT_BLOCK), sm, s, (const cx<float> *)in, (cx<float> *)out,
                           n[0], n[1], n[2], b_to_c, FftStages(py), FastDiv(n[1]), TileDiv(n[0], TX, 1), (const cx<float> *)twy, TX, ctl);
    }
    return check_launch("fft_y");
}

template <typename T, int CO>
static hipError_t launch_green_generic(hipStream_t s, int prec, void *specC, const int n[3], const FftPlan &px,
                                 const void *twx, const DevConst *cst, int mode, int ncomp, const IterCtl *ctl,
                                 void *nyq, int tile = 0) {
    const int slots = mode & 1 ? CO : ncomp;
    int TY;
    bool wide;
    if (mode == 1 && tile >= 1 && tile <= fft_tile_max(2, n, px, prec, CO)) {
        TY = tile;
        wide = (long)slots * TY * n[0] / min_radix(px) > 2 * FFT_BLOCK;
    } else {
        // two butterflies per thread when one row of `slots` pencils allows it, four otherwise
        wide = (long)slots * n[0] / min_radix(px) > 2 * FFT_BLOCK;
        TY = tile_for(px, slots, wide ? 4 : 2, n[1] < 2 ? n[1] : 2, prec);
    }
    const int H = n[2] / 2 + 1;
    const dim3 grid((n[1] + TY - 1) / TY, H);
    cx<double> *ny = (cx<double> *)nyq;
    const size_t sm = (size_t)(slots * TY + 1) * n[0] * sizeof(cx<T>);
    if (wide)
        SRX_LAUNCH((k_green_x<T, 4, CO>), grid, dim3(FFT_BLOCK), sm, s, (cx<T> *)specC, n[0], n[1], n[2], FftStages(px),
                   FastDiv(n[0]), TileDiv(n[1], TY, n[0]), (const cx<T> *)twx, TY, mode, ncomp, cst, ctl, ny);
    else
        SRX_LAUNCH((k_green_x<T, 2, CO>), grid, dim3(FFT_BLOCK), sm, s, (cx<T> *)specC, n[0], n[1], n[2], FftStages(px),
                   FastDiv(n[0]), TileDiv(n[1], TY, n[0]), (const cx<T> *)twx, TY, mode, ncomp, cst, ctl, ny);
    return check_launch("green_x");
}

// The wavefront-per-row x pass serves n0 = 64, 128, 256 (tile -1, and the default tile 0 there);
// other extents, and tiles >= 1, use the LDS kernel.
bool green_wave_ok(const int n[3]) { return n[0] == 64 || n[0] == 128 || n[0] == 256; }

template <typename T, int CO>
static void launch_green_wave(hipStream_t s, void *specC, const int n[3], const void *twx, const DevConst *cst,
                              const IterCtl *ctl, void *nyq) {
    const dim3 grid((n[1] + 3) / 4, n[2] / 2 + 1), block(256);
    cx<T> *sp = (cx<T> *)specC;
    cx<double> *ny = (cx<double> *)nyq;
    const cx<T> *tw = (const cx<T> *)twx;
    if (n[0] == 64) SRX_LAUNCH((k_green_wave<T, 1, CO>), grid, block, 0, s, sp, n[1], n[2], tw, cst, ctl, ny);
    else if (n[0] == 128) SRX_LAUNCH((k_green_wave<T, 2, CO>), grid, block, 0, s, sp, n[1], n[2], tw, cst, ctl, ny);
    else SRX_LAUNCH((k_green_wave<T, 4, CO>), grid, block, 0, s, sp, n[1], n[2], tw, cst, ctl, ny);
}

size_t nyq_elems(const int n[3]) {
    const size_t H = n[2] / 2 + 1;
    return 3 * ((size_t)n[0] * n[1] + H * n[0] + H * n[1]);
}

// Whether the outer iterations carry the six strain components (else DisGrad's nine): always in FP64;
// in mixed precision where the FP32 wave vectors are exact, i.e. every extent is a power of two.
bool strain_form(const int n[3], int prec) {
    auto pow2 = [](int v) { return (v & (v - 1)) == 0; };
    return prec == 0 || (pow2(n[0]) && pow2(n[1]) && pow2(n[2]));
}

void launch_green_x(hipStream_t s, int prec, void *specC, const int n[3], const FftPlan &px, const void *twx,
                    const DevConst *cst, const IterCtl *ctl, void *nyq, int tile) {
    const bool six = strain_form(n, prec);
    if (green_wave_ok(n) && tile <= 0) {
        if (prec == 0) launch_green_wave<double, 6>(s, specC, n, twx, cst, ctl, nyq);
        else if (six) launch_green_wave<float, 6>(s, specC, n, twx, cst, ctl, nyq);
        else launch_green_wave<float, 9>(s, specC, n, twx, cst, ctl, nyq);
        check_launch("green_x");
        return;
    }
    if (prec == 0) launch_green_generic<double, 6>(s, prec, specC, n, px, twx, cst, 1, 6, ctl, nyq, tile);
    else if (six) launch_green_generic<float, 6>(s, prec, specC, n, px, twx, cst, 1, 6, ctl, nyq, tile);
    else launch_green_generic<float, 9>(s, prec, specC, n, px, twx, cst, 1, 9, ctl, nyq, tile);
}

// planes of up to 256 points, where one block's chain is shorter than three launches (k_plane's figures)
bool plane_pass_ok(const int n[3]) { return n[0] * n[1] <= PLANE_POINTS; }

template <typename T, int CO>
static void launch_plane_t(hipStream_t s, void *specB, const int n[3], const FftPlan pl[3], void *const tw[3],
                           const DevConst *cst, const IterCtl *ctl, void *nyq) {
    const PlanePlans pp = {{FftStages(pl[0]), FftStages(pl[1])}, {FastDiv(n[0]), FastDiv(n[1])}, FastDiv(n[0] * n[1])};
    const size_t sm = ((size_t)CO * n[0] * (n[1] | 1) + n[0] + n[1]) * sizeof(cx<T>);
    SRX_LAUNCH((k_plane<T, CO>), dim3(n[2] / 2 + 1), dim3(PLANE_BLOCK), sm, s, (cx<T> *)specB, n[0], n[1], n[2], pp,
               (const cx<T> *)tw[0], (const cx<T> *)tw[1], cst, ctl, (cx<double> *)nyq);
}
void launch_plane(hipStream_t s, int prec, void *specB, const int n[3], const FftPlan pl[3], void *const tw[3],
                  const DevConst *cst, const IterCtl *ctl, void *nyq) {
    if (prec == 0) launch_plane_t<double, 6>(s, specB, n, pl, tw, cst, ctl, nyq);
    else if (strain_form(n, prec)) launch_plane_t<float, 6>(s, specB, n, pl, tw, cst, ctl, nyq);
    else launch_plane_t<float, 9>(s, specB, n, pl, tw, cst, ctl, nyq);
    check_launch("plane");
}

template <typename T>
static hipError_t launch_inv_z(hipStream_t s, const void *specB, double *out, int ncomp, const int n[3], const FftPlan &pz,
                         const void *twz, int accumulate, double divisor, const IterCtl *ctl, int tile, int prec) {
    const int rows = n[0] * n[1], TY = zy_tile(pz, rows, tile, prec);
    const bool sw = plan_swizzled(pz);
    const dim3 grid((rows + TY - 1) / TY, (ncomp + 1) / 2);
    const size_t sm = padded_lds(TY, n[2], sizeof(cx<T>), sw);
    if (sw)
        SRX_LAUNCH((k_inv_z<T, true>), grid, dim3(FFT_BLOCK), sm, s, (const cx<T> *)specB, out, ncomp, n[0], n[1], n[2],
                   FftStages(pz), FastDiv(n[2]), TileDiv(rows, TY, 1), (const cx<T> *)twz, TY, accumulate, divisor, ctl);
    else
        SRX_LAUNCH((k_inv_z<T, false>), grid, dim3(FFT_BLOCK), sm, s, (const cx<T> *)specB, out, ncomp, n[0], n[1], n[2],
                   FftStages(pz), FastDiv(n[2]), TileDiv(rows, TY, 1), (const cx<T> *)twz, TY, accumulate, divisor, ctl);
    return check_launch("inv_z");
}

void launch_fft_inv_z_update(hipStream_t s, int prec, const void *specB, double *ee, const int n[3], const FftPlan &pz,
                             const void *twz, const IterCtl *ctl, double divisor, int tile) {
    const int nc = strain_form(n, prec) ? 6 : 9;
    if (prec == 0) launch_inv_z<double>(s, specB, ee, nc, n, pz, twz, 1, divisor, ctl, tile, prec);
    else launch_inv_z<float>(s, specB, ee, nc, n, pz, twz, 1, divisor, ctl, tile, prec);
}

// The rotation part of the increment's displacement gradient from its accumulated strain (in [6][N],
// B basis), into out [3][N] (entries (1,2), (0,2), (0,1)): forward transforms of the six strain
// components, rotation_point, inverse transforms of three.  In FP64 in mixed precision too: the strain is a
// sum of FP32 increments that is kept in FP64, and casting that sum to FP32 for one more pair of
// transforms added 1.3e-7 of the rotation to its error (0.18 ms an increment at 128^3 instead of 0.15).
// specB, specC: 6 FP64 half spectra each; tw: FP64 twiddles; tiles: the solver passes' (launch shapes only).
void launch_rotation_part(hipStream_t s, const double *in, double *out, void *specB, void *specC, const int n[3],
                          const FftPlan pl[3], void *const tw[3], const DevConst *cst, void *nyq, const int tiles[5]) {
    launch_fft_fwd_z(s, 0, in, specB, n, pl[2], tw[2], nullptr, tiles[0]);
    launch_fft_y(s, 0, specB, specC, 6, -1, 1, n, pl[1], tw[1], nullptr, tiles[1]);
    if (green_wave_ok(n)) {
        launch_green_wave<double, 3>(s, specC, n, tw[0], cst, nullptr, nyq);
        check_launch("rotation_x");
    } else {
        launch_green_generic<double, 6>(s, 0, specC, n, pl[0], tw[0], cst, 3, 3, nullptr, nyq);
    }
    launch_fft_y(s, 0, specC, specB, 3, +1, 0, n, pl[1], tw[1], nullptr, tiles[3]);
    launch_inv_z<double>(s, specB, out, 3, n, pl[2], tw[2], 0, (double)n[0] * n[1] * n[2], nullptr, tiles[4], 0);
}

// forward FFT of ncomp real comps to layout C (x pass done), no Green: the entry points' transforms
hipError_t launch_fft_real_forward_test(hipStream_t s, int prec, const double *in, int ncomp, void *specB, void *specC,
                                        const int n[3], const FftPlan *pl, void *const *tw) {
    hipError_t e;
    if (prec == 0) e = launch_fwd_z<double>(s, in, specB, ncomp, n, pl[2], tw[2], nullptr, 0, prec);
    else e = launch_fwd_z<float>(s, in, specB, ncomp, n, pl[2], tw[2], nullptr, 0, prec);
    if (e == hipSuccess) e = launch_fft_y(s, prec, specB, specC, ncomp, -1, 1, n, pl[1], tw[1], nullptr);
    if (e != hipSuccess) return e;
    if (prec == 0) return launch_green_generic<double, 6>(s, prec, specC, n, pl[0], tw[0], nullptr, 0, ncomp, nullptr, nullptr);
    return launch_green_generic<float, 6>(s, prec, specC, n, pl[0], tw[0], nullptr, 0, ncomp, nullptr, nullptr);
}

// inverse of the above for ncomp comps (layout C in, real out = IFFT * 1/divisor)
hipError_t launch_fft_real_inverse_test(hipStream_t s, int prec, void *specC, void *specB, int ncomp, double *out,
                                        const int n[3], const FftPlan *pl, void *const *tw, double divisor) {
    hipError_t e;
    if (prec == 0) e = launch_green_generic<double, 6>(s, prec, specC, n, pl[0], tw[0], nullptr, 2, ncomp, nullptr, nullptr);
    else e = launch_green_generic<float, 6>(s, prec, specC, n, pl[0], tw[0], nullptr, 2, ncomp, nullptr, nullptr);
    if (e == hipSuccess) e = launch_fft_y(s, prec, specC, specB, ncomp, +1, 0, n, pl[1], tw[1], nullptr);
    if (e != hipSuccess) return e;
    if (prec == 0) return launch_inv_z<double>(s, specB, out, ncomp, n, pl[2], tw[2], 0, divisor, nullptr, 0, prec);
    return launch_inv_z<float>(s, specB, out, ncomp, n, pl[2], tw[2], 0, divisor, nullptr, 0, prec);
}

// ---------------------------------------------------------------------------
// HBM ceiling: a plain streaming copy, 16 bytes per lane per access, U independent accesses in
// flight per lane, grid-stride over the buffer.  The measured rate is the ceiling the HBM-bound
// passes above are compared with.
// ---------------------------------------------------------------------------
typedef double dvec2 __attribute__((ext_vector_type(2)));
template <int U>
__global__ void __launch_bounds__(256) k_stream_copy(const dvec2 *__restrict__ in, dvec2 *__restrict__ out,
                                                      size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    for (; i + (U - 1) * stride < n; i += U * stride) {
        dvec2 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(in + i + u * stride);
#pragma unroll
        for (int u = 0; u < U; ++u) __builtin_nontemporal_store(v[u], out + i + u * stride);
    }
    for (; i < n; i += stride) out[i] = in[i];
}

void launch_stream_copy(hipStream_t s, const void *in, void *out, size_t n16, int unroll, int blocks) {
    const dim3 grid(blocks), block(256);
    if (unroll == 4)
        hipLaunchKernelGGL(k_stream_copy<4>, grid, block, 0, s, (const dvec2 *)in, (dvec2 *)out, n16);
    else if (unroll == 2)
        hipLaunchKernelGGL(k_stream_copy<2>, grid, block, 0, s, (const dvec2 *)in, (dvec2 *)out, n16);
    else
        hipLaunchKernelGGL(k_stream_copy<1>, grid, block, 0, s, (const dvec2 *)in, (dvec2 *)out, n16);
    check_launch("stream_copy");
}

}  // namespace srx
