// qk_oneint.hip -- one-electron integrals and their nuclear-gradient terms on
// the device (gfx950).
//
// Replaces QUICK's get1e (kinetic get1eO and nuclear attraction attrashell,
// quick_one_electron_integral.f90:1633-1925) and the one-electron part of
// hfgrad (gradient.f90:40-250: nuclear repulsion, -2 W dS/dR + 2 D dT/dR, and
// attrashellopt's D dV/dR, shell.f90:1747-1860).
//
// A lane takes primitive pairs of one pair of shells (single angular momentum,
// one kernel per class, LA >= LB) and loops over the nuclei.  The work that
// grows with the nuclei is then the Boys functions and the Hermite Coulomb
// integrals R_tuv alone (McMurchie-Davidson), once per primitive pair for all
// functions of the shells: the attraction integrals need only
// V_tuv = sum_C -Z_C R_tuv(P - C), contracted with the Hermite expansion
// coefficients E^{ij}_t after the loop.  For the gradient the density is
// contracted first: with h_tuv = sum_ab D_ab E^x_t E^y_u E^z_v the force on
// nucleus C is Z_C sum h_tuv R_{tuv + 1}, minus their sum the derivative with
// respect to P, and the part of d/dA at fixed P contracts with V_tuv (d/dB is
// what translational invariance leaves).  Bound by FP64 issue and the latency
// of one lane's chain (Boys -> R -> sums).  One thread per pair of functions,
// with 12 contractions per nucleus and 64 lanes adding to one LDS word, had
// taken 23 ms for the integrals and gradient of (H2O)32; the twelve kernels here
// take 2.4 ms one after another, 0.9 ms on four streams.
//
// The order asked of the Boys fit is Qfinal(I) + Qfinal(J) (+ 2 for the
// gradient), as the reference asks it.  A shell pair's matrix elements are
// summed over a fixed group of lanes and written once, without atomics; the
// gradient goes to a per-block int64 fixed-point copy in LDS (2^-44 units) and
// then to the global accumulator, so both are bitwise reproducible.
#include <utility>

#include "qk_kernels.h"

namespace qk {

// f(0), ..., f(N - 1) with compile-time arguments, so that every table index
// below is a constant and the tables stay in registers
template <class F, int... I>
__device__ __forceinline__ void sfor_(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void sfor(F&& f) {
    sfor_(f, std::make_integer_sequence<int, N>{});
}

// power of direction d in component k of a shell of angular momentum l: x powers
// falling, then y powers falling (the order of a shell's slots)
__host__ __device__ constexpr int cart(int l, int k, int d) {
    for (int x = l; x >= 0; --x)
        for (int y = l - x; y >= 0; --y, --k)
            if (k == 0) return d == 0 ? x : (d == 1 ? y : l - x - y);
    return 0;
}

// (t, u, v) with t + u + v <= L in one tetrahedral array: the shells of equal
// t + u + v one after another, within a shell by u + v, then v
constexpr int tet_size(int L) { return (L + 1) * (L + 2) * (L + 3) / 6; }
constexpr int tet(int t, int u, int v) {
    return (t + u + v) * (t + u + v + 1) * (t + u + v + 2) / 6 + (u + v) * (u + v + 1) / 2 + v;
}

// Hermite Coulomb integrals R^{(0)}_tuv for t + u + v <= L: R^{(n)}_000 =
// (-2p)^n F_n, raised one index at a time (t first, then u, then v), level n
// holding t + u + v <= L - n; all indices compile-time, so the table stays in
// registers
template <int L>
__device__ __forceinline__ void hermite_r_u(double p, const double* PC, const double* F, double* R0) {
    double R[L + 1][tet_size(L)];
    double pw = 1.0;
#pragma unroll
    for (int n = 0; n <= L; ++n) {
        R[n][0] = pw * F[n];
        pw *= -2.0 * p;
    }
#pragma unroll
    for (int n = L - 1; n >= 0; --n)
#pragma unroll
        for (int s = 1; s <= L - n; ++s)
#pragma unroll
            for (int r = 0; r <= s; ++r)
#pragma unroll
                for (int v = 0; v <= r; ++v) {
                    const int u = r - v, t = s - r;
                    double x;
                    if (t > 0)
                        x = (t > 1 ? (t - 1) * R[n + 1][tet(t - 2, u, v)] : 0.0) + PC[0] * R[n + 1][tet(t - 1, u, v)];
                    else if (u > 0)
                        x = (u > 1 ? (u - 1) * R[n + 1][tet(t, u - 2, v)] : 0.0) + PC[1] * R[n + 1][tet(t, u - 1, v)];
                    else
                        x = (v > 1 ? (v - 1) * R[n + 1][tet(t, u, v - 2)] : 0.0) + PC[2] * R[n + 1][tet(t, u, v - 1)];
                    R[n][tet(t, u, v)] = x;
                }
#pragma unroll
    for (int k = 0; k < tet_size(L); ++k) R0[k] = R[0][k];
}

// E^{ij}_t of one direction for i <= LA, j <= LB, t <= i + j: E^{00}_0 = 1,
// E^{i+1,j}_t = E^{ij}_{t-1} / 2p + PA E^{ij}_t + (t + 1) E^{ij}_{t+1}, in j with PB
template <int LA, int LB>
struct HermE {
    double e[LA + 1][LB + 1][LA + LB + 1];
    __device__ __forceinline__ void make(double PA, double PB, double oo2p) {
        e[0][0][0] = 1.0;
        sfor<LA>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            raise<i + 1>(e[i + 1][0], e[i][0], PA, oo2p);
        });
        sfor<LA + 1>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            sfor<LB>([&](auto j_) {
                constexpr int j = decltype(j_)::value;
                raise<i + j + 1>(e[i][j + 1], e[i][j], PB, oo2p);
            });
        });
    }
    // T_t, t = 0..N from E_t, t = 0..N - 1
    template <int N>
    static __device__ __forceinline__ void raise(double* T, const double* E, double X, double oo2p) {
        sfor<N + 1>([&](auto t_) {
            constexpr int t = decltype(t_)::value;
            double v = 0.0;
            if constexpr (t > 0) v = oo2p * E[t - 1];
            if constexpr (t < N) v += X * E[t];
            if constexpr (t + 1 < N) v += double(t + 1) * E[t + 1];
            T[t] = v;
        });
    }
};

// overlap and kinetic factors of one direction in units of sqrt(pi/p), i <= LA,
// j <= LB: s_ij = E^{ij}_0, and -1/2 d^2/dx^2 on the second function,
// t_ij = b(2j+1) s_ij - 2 b^2 s_i,j+2 - j(j-1)/2 s_i,j-2
template <int LA, int LB>
struct Factors {
    double s[LA + 1][LB + 3];
    __device__ __forceinline__ void make(double PA, double PB, double oo2p) {
        s[0][0] = 1.0;
        sfor<LA>([&](auto i_) {
            constexpr int i = decltype(i_)::value;
            double v = PA * s[i][0];
            if constexpr (i > 0) v += oo2p * double(i) * s[i - 1][0];
            s[i + 1][0] = v;
        });
        sfor<LB + 2>([&](auto j_) {
            constexpr int j = decltype(j_)::value;
            sfor<LA + 1>([&](auto i_) {
                constexpr int i = decltype(i_)::value;
                double v = PB * s[i][j];
                if constexpr (i > 0) v += oo2p * double(i) * s[i - 1][j];
                if constexpr (j > 0) v += oo2p * double(j) * s[i][j - 1];
                s[i][j + 1] = v;
            });
        });
    }
    template <int i, int j>
    __device__ __forceinline__ double kin(double b) const {
        double t = b * (2 * j + 1) * s[i][j] - 2.0 * b * b * s[i][j + 2];
        if constexpr (j >= 2) t -= 0.5 * j * (j - 1) * s[i][j - 2];
        return t;
    }
};

constexpr double kPi = 3.14159265358979323846;
// primitive pairs whose Gaussian-product prefactor lies below this contribute
// less than 1e-24 to any element and are skipped
constexpr double k1eKabCut = 1e-24;

// A lane's pair of shells and its walk over their primitive pairs.  A lane beyond
// the batch's pairs walks none, but it runs the same code up to the wavefront's
// sums: it holds the batch's first pair, so that what it reads belongs to that pair.
struct OnePair {
    bool have;        // whether the lane has a pair
    int fA, fB;       // first slots
    int nB, npp;      // primitives of B, primitive pairs
    int atA, atB;
    double A[3], B[3], AB2;
    int next;         // next primitive pair to look at
    __device__ __forceinline__ void load(const OneFuncs& f, const OneSys& sys, const int2* pairs, long long k, bool in,
                                         int first) {
        have = in;
        const int2 pr = pairs[in ? k : 0];
        fA = pr.x; fB = pr.y;
        nB = f.np[fB];
        npp = in ? f.np[fA] * nB : 0;
        atA = f.atom[fA]; atB = f.atom[fB];
        AB2 = 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            A[d] = sys.xyz[3 * atA + d];
            B[d] = sys.xyz[3 * atB + d];
        }
        AB2 = (A[0] - B[0]) * (A[0] - B[0]) + (A[1] - B[1]) * (A[1] - B[1]) + (A[2] - B[2]) * (A[2] - B[2]);
        next = first;
    }
};
// One primitive pair; a lane that has none left keeps a harmless one with K = 0
struct OnePrim {
    int ci, cj;
    double a, b, p, oop, oo2p, K, P[3], PA[3], PB[3];
    // the lane's next pair above k1eKabCut, step apart; whether there is one
    __device__ __forceinline__ bool seek(const OneFuncs& f, OnePair& q, int step) {
        bool found = false;
        ci = cj = 0;
        a = b = 1.0;
        oop = 0.5;
        K = 0.0;
        while (!found && q.next < q.npp) {
            ci = q.next / q.nB;
            cj = q.next - ci * q.nB;
            q.next += step;
            a = f.a[k1eMaxPrim * q.fA + ci];
            b = f.a[k1eMaxPrim * q.fB + cj];
            oop = 1.0 / (a + b);
            K = exp(-a * b * oop * q.AB2);
            found = !(K < k1eKabCut);
        }
        if (!found) K = 0.0;
        p = a + b;
        oo2p = 0.5 * oop;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            P[d] = (a * q.A[d] + b * q.B[d]) * oop;
            PA[d] = P[d] - q.A[d];
            PB[d] = P[d] - q.B[d];
        }
        return found;
    }
    // makes the compiler compute what follows from PA, PB here and not before the
    // loop over the nuclei, through which it would keep the tables in registers
    __device__ __forceinline__ void after_nuclei() {
#pragma unroll
        for (int d = 0; d < 3; ++d) asm volatile("" : "+v"(PA[d]), "+v"(PB[d]));
    }
    // of two slots
    __device__ __forceinline__ double coef(const OneFuncs& f, int sA, int sB) const {
        return f.c[k1eMaxPrim * sA + ci] * f.c[k1eMaxPrim * sB + cj];
    }
};

// QUICK's fit, with exp(-T) for any T: a nucleus may lie farther away than exp_neg
// can carry (exp(-T) is zero from T = 746 on)
template <int L>
__device__ __forceinline__ void boys_one(double T, int M, const double* __restrict__ tab, double* F) {
    const double E = exp_neg(fmin(T, 800.0));
    boys_fit_main<L>(T, E, tab, F);
    if (!boys_fit_up(T, M)) boys_fit_near0<L>(T, E, M, F);
}

// The pair list of a class holds first the pairs of many primitives, 2^kOneLog[0]
// lanes each, then those of fewer: a lane walks at most about four primitive
// pairs.  Calls use(first pair, pairs, lanes per pair log2) for the wavefront's
// batch, which has at least one pair.
template <class F>
__device__ __forceinline__ void one_batches(const OnePairs& w, F&& use) {
    const long long wave0 = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    const long long nwaves = (long long)gridDim.x * (blockDim.x >> 6);
    long long w0 = 0, k0 = 0;   // first wavefront and first pair of the bucket
    long long t = wave0;
    for (int b = 0; b < kOneBuckets; ++b) {
        const int lg = kOneLog[b], per = 64 >> lg;
        const long long nw = (w.n[b] + per - 1) / per;
        for (; t < w0 + nw; t += nwaves) use(w.pairs + k0 + (t - w0) * per, w.n[b] - (t - w0) * per, lg);
        w0 += nw;
        k0 += w.n[b];
    }
}

// S and H = T + V (n x n, column-major, both triangles) for the shell pairs of
// one class
template <int LA, int LB>
__global__ void __launch_bounds__(256, LA + LB >= 2 && LA * LB > 0 ? 1 : 2)
    oneint_kernel(const OneFuncs f, const OneSys sys, const OnePairs w, double* __restrict__ S, double* __restrict__ H) {
    constexpr int L = LA + LB, NA = ncart(LA), NB = ncart(LB), NT = tet_size(L);
    __shared__ double s_boys[kBoysFitRegions * kBoysFitTerms];
    for (int k = threadIdx.x; k < kBoysFitRegions * kBoysFitTerms; k += blockDim.x) s_boys[k] = kBoysFit[k];
    __syncthreads();
    const int lane = threadIdx.x & 63;
    one_batches(w, [&](const int2* pairs, long long left, int lg) {
        const int G = 1 << lg, sub = lane & (G - 1);
        OnePair q;
        q.load(f, sys, pairs, lane >> lg, (lane >> lg) < left, sub);
        const int M = max(f.qf[q.fA] + f.qf[q.fB], L);
        double so[NA * NB], ho[NA * NB];
#pragma unroll
        for (int k = 0; k < NA * NB; ++k) so[k] = ho[k] = 0.0;
        for (;;) {
            OnePrim o;
            const bool got = o.seek(f, q, G);
            if (!__any(got)) break;
            double V[NT];
#pragma unroll
            for (int k = 0; k < NT; ++k) V[k] = 0.0;
            if (H)
                for (int C = 0; C < sys.natom; ++C) {
                    const double PC[3] = {o.P[0] - sys.xyz[3 * C], o.P[1] - sys.xyz[3 * C + 1],
                                          o.P[2] - sys.xyz[3 * C + 2]};
                    double F[L + 1], R0[NT];
                    boys_one<L>(o.p * (PC[0] * PC[0] + PC[1] * PC[1] + PC[2] * PC[2]), M, s_boys, F);
                    hermite_r_u<L>(o.p, PC, F, R0);
                    const double z = -sys.chg[C];
#pragma unroll
                    for (int k = 0; k < NT; ++k) V[k] += z * R0[k];
                }
            o.after_nuclei();
            HermE<LA, LB> E[3];
            Factors<LA, LB> t[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                E[d].make(o.PA[d], o.PB[d], o.oo2p);
                t[d].make(o.PA[d], o.PB[d], o.oo2p);
            }
            const double s0 = o.K * kPi * o.oop * sqrt(kPi * o.oop);   // (pi/p)^{3/2} K_ab
            const double v0 = 2.0 * kPi * o.oop * o.K;
            sfor<NA>([&](auto ia_) {
                constexpr int ia = decltype(ia_)::value;
                sfor<NB>([&](auto ib_) {
                    constexpr int ib = decltype(ib_)::value;
                    constexpr int ax = cart(LA, ia, 0), ay = cart(LA, ia, 1), az = cart(LA, ia, 2);
                    constexpr int bx = cart(LB, ib, 0), by = cart(LB, ib, 1), bz = cart(LB, ib, 2);
                    const double cc = o.coef(f, q.fA + ia, q.fB + ib);
                    const double sx = t[0].s[ax][bx], sy = t[1].s[ay][by], sz = t[2].s[az][bz];
                    const double kx = t[0].template kin<ax, bx>(o.b), ky = t[1].template kin<ay, by>(o.b),
                                 kz = t[2].template kin<az, bz>(o.b);
                    double v = 0.0;
                    sfor<ax + bx + 1>([&](auto t_) {
                        constexpr int tt = decltype(t_)::value;
                        double su = 0.0;
                        sfor<ay + by + 1>([&](auto u_) {
                            constexpr int uu = decltype(u_)::value;
                            double sv = 0.0;
                            sfor<az + bz + 1>([&](auto v_) {
                                constexpr int vv = decltype(v_)::value;
                                sv += E[2].e[az][bz][vv] * V[tet(tt, uu, vv)];
                            });
                            su += E[1].e[ay][by][uu] * sv;
                        });
                        v += E[0].e[ax][bx][tt] * su;
                    });
                    so[ia * NB + ib] += cc * s0 * sx * sy * sz;
                    ho[ia * NB + ib] += cc * (s0 * (kx * sy * sz + sx * ky * sz + sx * sy * kz) + v0 * v);
                });
            });
        }
        for (int off = G >> 1; off >= 1; off >>= 1)
#pragma unroll
            for (int k = 0; k < NA * NB; ++k) {
                so[k] += __shfl_xor(so[k], off, 64);
                ho[k] += __shfl_xor(ho[k], off, 64);
            }
        if (q.have && sub == 0)
#pragma unroll
            for (int k = 0; k < NA * NB; ++k) {
                if (q.fA == q.fB && k % NB < k / NB) continue;   // one shell: its lower half by symmetry
                const int I = f.out[q.fA + k / NB], J = f.out[q.fB + k % NB];
                if (I < 0 || J < 0) continue;   // an empty component
                const long long o1 = (long long)I * sys.n + J, o2 = (long long)J * sys.n + I;
                if (S) S[o1] = S[o2] = so[k];
                if (H) H[o1] = H[o2] = ho[k];
            }
    });
}

// sum over the 64 lanes, in lane 63 (row shifts, then the rows' last lanes
// broadcast to the next row; always the same order)
__device__ __forceinline__ double wave_sum(double v) {
    auto step = [&](auto ctl, auto mask) {
        const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), decltype(ctl)::value, decltype(mask)::value, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), decltype(ctl)::value, decltype(mask)::value, 0xf, false);
        v += __hiloint2double(hi, lo);
    };
    using std::integral_constant;
    step(integral_constant<int, 0x111>{}, integral_constant<int, 0xf>{});   // row_shr:1
    step(integral_constant<int, 0x112>{}, integral_constant<int, 0xf>{});   // row_shr:2
    step(integral_constant<int, 0x114>{}, integral_constant<int, 0xf>{});   // row_shr:4
    step(integral_constant<int, 0x118>{}, integral_constant<int, 0xf>{});   // row_shr:8
    step(integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});   // row_bcast:15
    step(integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});   // row_bcast:31
    return v;
}

__device__ __forceinline__ void lds_gadd(unsigned long long* g, int i, double v) {
    const long long iv = __double2ll_rn(v * 0x1p44);
    if (iv) atomicAdd(g + i, (unsigned long long)iv);
}

// grad += sum over the shell pairs of one class of D dH/dR - W dS/dR (3 x natom,
// 2^-44 units, accumulated per block in LDS: dynamic LDS of 3 natom int64).  The
// blocks of row y take the y-th part of the nuclei (everything is linear in them;
// row 0 adds overlap and kinetic energy).
template <int LA, int LB>
__global__ void __launch_bounds__(256, LA + LB >= 2 ? 1 : 2)
    oneint_grad_kernel(const OneFuncs f, const OneSys sys, const OnePairs w, const double* __restrict__ Dm,
                       const double* __restrict__ Wm, unsigned long long* __restrict__ Gacc) {
    constexpr int L = LA + LB, NA = ncart(LA), NB = ncart(LB), NT = tet_size(L);
    extern __shared__ unsigned long long s_g[];
    __shared__ double s_boys[kBoysFitRegions * kBoysFitTerms];
    const int m3 = 3 * sys.natom;
    const int C0 = (long long)sys.natom * blockIdx.y / gridDim.y,
              C1 = (long long)sys.natom * (blockIdx.y + 1) / gridDim.y;
    for (int i = threadIdx.x; i < m3; i += blockDim.x) s_g[i] = 0ull;
    for (int k = threadIdx.x; k < kBoysFitRegions * kBoysFitTerms; k += blockDim.x) s_boys[k] = kBoysFit[k];
    __syncthreads();
    const int lane = threadIdx.x & 63;
    one_batches(w, [&](const int2* pairs, long long left, int lg) {
        const int G = 1 << lg;
        OnePair q;
        q.load(f, sys, pairs, lane >> lg, (lane >> lg) < left, lane & (G - 1));
        const int M = max(f.qf[q.fA] + f.qf[q.fB] + 2, L + 1);
        const double wt = q.fA == q.fB ? 1.0 : 2.0;   // every pair of functions twice, (I, J) and (J, I)
        auto elem = [&](const double* X, int I, int J) {
            return X[I < J ? (long long)I * sys.n + J : (long long)J * sys.n + I];
        };
        double gA[3] = {0.0, 0.0, 0.0}, gB[3] = {0.0, 0.0, 0.0};
        for (;;) {
            OnePrim o;
            const bool got = o.seek(f, q, G);
            if (!__any(got)) break;
            HermE<LA, LB> E[3];
            double h[NT], V[NT];
#pragma unroll
            for (int d = 0; d < 3; ++d) E[d].make(o.PA[d], o.PB[d], o.oo2p);
#pragma unroll
            for (int k = 0; k < NT; ++k) h[k] = V[k] = 0.0;
            const double v0 = wt * 2.0 * kPi * o.oop * o.K;
            sfor<NA>([&](auto ia_) {
                constexpr int ia = decltype(ia_)::value;
                sfor<NB>([&](auto ib_) {
                    constexpr int ib = decltype(ib_)::value;
                    constexpr int ax = cart(LA, ia, 0), ay = cart(LA, ia, 1), az = cart(LA, ia, 2);
                    constexpr int bx = cart(LB, ib, 0), by = cart(LB, ib, 1), bz = cart(LB, ib, 2);
                    const int I = f.fn[q.fA + ia], J = f.fn[q.fB + ib];
                    const double c = o.coef(f, q.fA + ia, q.fB + ib) * v0 * elem(Dm, I, J);
                    sfor<ax + bx + 1>([&](auto t_) {
                        constexpr int tt = decltype(t_)::value;
                        const double ct = c * E[0].e[ax][bx][tt];
                        sfor<ay + by + 1>([&](auto u_) {
                            constexpr int uu = decltype(u_)::value;
                            const double cu = ct * E[1].e[ay][by][uu];
                            sfor<az + bz + 1>([&](auto v_) {
                                constexpr int vv = decltype(v_)::value;
                                h[tet(tt, uu, vv)] += cu * E[2].e[az][bz][vv];
                            });
                        });
                    });
                });
            });
            double dP[3] = {0.0, 0.0, 0.0};
            for (int C = C0; C < C1; ++C) {
                const double PC[3] = {o.P[0] - sys.xyz[3 * C], o.P[1] - sys.xyz[3 * C + 1], o.P[2] - sys.xyz[3 * C + 2]};
                double F[L + 2], R0[tet_size(L + 1)];
                boys_one<L + 1>(o.p * (PC[0] * PC[0] + PC[1] * PC[1] + PC[2] * PC[2]), M, s_boys, F);
                hermite_r_u<L + 1>(o.p, PC, F, R0);
                // one-centre terms add up to zero
                const double z = q.atA == C && q.atB == C ? 0.0 : -sys.chg[C];
                double g[3] = {0.0, 0.0, 0.0};
                sfor<L + 1>([&](auto t_) {
                    constexpr int tt = decltype(t_)::value;
                    sfor<L + 1 - tt>([&](auto u_) {
                        constexpr int uu = decltype(u_)::value;
                        sfor<L + 1 - tt - uu>([&](auto v_) {
                            constexpr int vv = decltype(v_)::value;
                            constexpr int k = tet(tt, uu, vv);
                            V[k] += z * R0[k];
                            g[0] += h[k] * R0[tet(tt + 1, uu, vv)];
                            g[1] += h[k] * R0[tet(tt, uu + 1, vv)];
                            g[2] += h[k] * R0[tet(tt, uu, vv + 1)];
                        });
                    });
                });
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    g[x] *= z;
                    dP[x] += g[x];
                    // the force on C: one LDS add per wavefront
                    const double gw = wave_sum(g[x]);
                    if (lane == 63) lds_gadd(s_g, 3 * C + x, -gw);
                }
            }
            // d/dA = (a/p) d/dP + the change at fixed P, whose coefficients are
            // 2a (PA E^{ij}_t + (t+1) E^{ij}_{t+1}) - i E^{i-1,j}_t, t <= i + j;
            // overlap and kinetic: two-centre, zero on one atom
            o.after_nuclei();
            Factors<LA + 1, LB> t[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                E[d].make(o.PA[d], o.PB[d], o.oo2p);
                t[d].make(o.PA[d], o.PB[d], o.oo2p);
            }
            const double s0 = q.atA != q.atB && blockIdx.y == 0 ? wt * o.K * kPi * o.oop * sqrt(kPi * o.oop) : 0.0;
            double rel[3] = {0.0, 0.0, 0.0}, st[3] = {0.0, 0.0, 0.0};
            sfor<NA>([&](auto ia_) {
                constexpr int ia = decltype(ia_)::value;
                sfor<NB>([&](auto ib_) {
                    constexpr int ib = decltype(ib_)::value;
                    constexpr int la[3] = {cart(LA, ia, 0), cart(LA, ia, 1), cart(LA, ia, 2)};
                    constexpr int lb[3] = {cart(LB, ib, 0), cart(LB, ib, 1), cart(LB, ib, 2)};
                    const int I = f.fn[q.fA + ia], J = f.fn[q.fB + ib];
                    const double cc = o.coef(f, q.fA + ia, q.fB + ib);
                    const double d = cc * elem(Dm, I, J), wv = cc * elem(Wm, I, J);
                    double sd[3], kd[3], dsd[3], dkd[3];
                    sfor<3>([&](auto d_) {
                        constexpr int x = decltype(d_)::value, i = la[x], j = lb[x];
                        sd[x] = t[x].s[i][j];
                        kd[x] = t[x].template kin<i, j>(o.b);
                        dsd[x] = 2.0 * o.a * t[x].s[i + 1][j];
                        dkd[x] = 2.0 * o.a * t[x].template kin<i + 1, j>(o.b);
                        if constexpr (i > 0) {
                            dsd[x] -= double(i) * t[x].s[i - 1][j];
                            dkd[x] -= double(i) * t[x].template kin<i - 1, j>(o.b);
                        }
                    });
                    st[0] += d * (dkd[0] * sd[1] * sd[2] + dsd[0] * (kd[1] * sd[2] + sd[1] * kd[2])) -
                             wv * dsd[0] * sd[1] * sd[2];
                    st[1] += d * (dkd[1] * sd[0] * sd[2] + dsd[1] * (kd[0] * sd[2] + sd[0] * kd[2])) -
                             wv * dsd[1] * sd[0] * sd[2];
                    st[2] += d * (dkd[2] * sd[0] * sd[1] + dsd[2] * (kd[0] * sd[1] + sd[0] * kd[1])) -
                             wv * dsd[2] * sd[0] * sd[1];
                    // e[x][t] of the three directions and the change of each
                    double r[3] = {0.0, 0.0, 0.0};
                    double dx[la[0] + lb[0] + 1], dy[la[1] + lb[1] + 1], dz[la[2] + lb[2] + 1];
                    auto change = [&](auto d_, double* out) {
                        constexpr int x = decltype(d_)::value, i = la[x], j = lb[x];
                        sfor<i + j + 1>([&](auto t_) {
                            constexpr int tt = decltype(t_)::value;
                            double v = o.PA[x] * E[x].e[i][j][tt];
                            if constexpr (tt < i + j) v += double(tt + 1) * E[x].e[i][j][tt + 1];
                            v *= 2.0 * o.a;
                            if constexpr (i > 0 && tt < i + j) v -= double(i) * E[x].e[i - 1][j][tt];
                            out[tt] = v;
                        });
                    };
                    change(std::integral_constant<int, 0>{}, dx);
                    change(std::integral_constant<int, 1>{}, dy);
                    change(std::integral_constant<int, 2>{}, dz);
                    sfor<la[0] + lb[0] + 1>([&](auto t_) {
                        constexpr int tt = decltype(t_)::value;
                        double s00 = 0.0, s10 = 0.0, s01 = 0.0;
                        sfor<la[1] + lb[1] + 1>([&](auto u_) {
                            constexpr int uu = decltype(u_)::value;
                            double v0_ = 0.0, v1_ = 0.0;
                            sfor<la[2] + lb[2] + 1>([&](auto v_) {
                                constexpr int vv = decltype(v_)::value;
                                v0_ += E[2].e[la[2]][lb[2]][vv] * V[tet(tt, uu, vv)];
                                v1_ += dz[vv] * V[tet(tt, uu, vv)];
                            });
                            s00 += E[1].e[la[1]][lb[1]][uu] * v0_;
                            s10 += dy[uu] * v0_;
                            s01 += E[1].e[la[1]][lb[1]][uu] * v1_;
                        });
                        r[0] += dx[tt] * s00;
                        r[1] += E[0].e[la[0]][lb[0]][tt] * s10;
                        r[2] += E[0].e[la[0]][lb[0]][tt] * s01;
                    });
#pragma unroll
                    for (int x = 0; x < 3; ++x) rel[x] += d * r[x];
                });
            });
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                const double va = o.a * o.oop * dP[x] + v0 * rel[x], sa = s0 * st[x];
                gA[x] += va + sa;
                gB[x] += dP[x] - va - sa;
            }
        }
        if (q.have)
#pragma unroll
            for (int x = 0; x < 3; ++x) {
                lds_gadd(s_g, 3 * q.atA + x, gA[x]);
                lds_gadd(s_g, 3 * q.atB + x, gB[x]);
            }
    });
    __syncthreads();
    for (int i = threadIdx.x; i < m3; i += blockDim.x)
        if (s_g[i]) atomicAdd(Gacc + i, s_g[i]);
}

// nuclear repulsion gradient: one thread per atom (2^-44 units)
__global__ void nuclear_grad_kernel(const OneSys sys, unsigned long long* __restrict__ G) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= sys.natom) return;
    double g[3] = {0.0, 0.0, 0.0};
    for (int j = 0; j < sys.natom; ++j) {
        if (j == i) continue;
        double d[3], r2 = 0.0;
        for (int x = 0; x < 3; ++x) {
            d[x] = sys.xyz[3 * j + x] - sys.xyz[3 * i + x];
            r2 += d[x] * d[x];
        }
        const double c = sys.chg[i] * sys.chg[j] / (r2 * sqrt(r2));
        for (int x = 0; x < 3; ++x) g[x] += d[x] * c;
    }
    for (int x = 0; x < 3; ++x) {
        const long long iv = __double2ll_rn(g[x] * 0x1p44);
        if (iv) atomicAdd(G + 3 * i + x, (unsigned long long)iv);
    }
}

// one launch per class of shell pairs (lists built on the host once per system)
static int one_grid(const OnePairs& w, long long per_cu = 8) {
    long long waves = 0;
    for (int b = 0; b < kOneBuckets; ++b) waves += (w.n[b] + (64 >> kOneLog[b]) - 1) / (64 >> kOneLog[b]);
    return (int)std::min((waves + 3) / 4, 256LL * per_cu);
}

#define QK_1E_CLASSES(X) X(0, 0, 0) X(1, 1, 0) X(2, 1, 1) X(3, 2, 0) X(4, 2, 1) X(5, 2, 2)

// s[k]: the stream of class k
void launch_oneint(const OneFuncs& f, const OneSys& sys, const OnePairs* w, double* S, double* H,
                   const hipStream_t* s) {
#define QK_1E(k, la, lb)                  \
    if (const int grid = one_grid(w[k])) \
        hipLaunchKernelGGL((oneint_kernel<la, lb>), dim3(grid), dim3(256), 0, s[k], f, sys, w[k], S, H);
    QK_1E_CLASSES(QK_1E)
#undef QK_1E
}

// Rows of blocks, each with a part of the nuclei: where a class has too few
// wavefronts to fill the GPU (512 blocks are taken as full), up to eight, of at
// least eight nuclei (a row repeats the density contraction of each primitive
// pair).  Measured on (H2O)32: (d|d) 277 -> 87 us, (d|s) 228 -> 93 us.
static int one_rows(int grid, int natom) { return std::max(1, std::min({8, 512 / grid, natom / 8})); }

// (d|d) is the one class here that spills; it takes one block per CU, and its grid,
// rows and all, keeps its scratch backing under the bound
void launch_oneint_grad(const OneFuncs& f, const OneSys& sys, const OnePairs* w, const double* D, const double* W,
                        unsigned long long* G, const hipStream_t* s) {
    const size_t lds = sizeof(unsigned long long) * 3 * (size_t)sys.natom;
#define QK_1E(k, la, lb)                                                                                      \
    if (int grid = one_grid(w[k], la + lb == 4 ? 1 : 8)) {                                                    \
        static const long long cap =                                                                          \
            scratch_grid_cap(kernel_scratch(reinterpret_cast<const void*>(&oneint_grad_kernel<la, lb>)), 4);  \
        grid = (int)std::min<long long>(grid, cap);                                                           \
        const int rows = (int)std::min<long long>(one_rows(grid, sys.natom), cap / grid);                     \
        hipLaunchKernelGGL((oneint_grad_kernel<la, lb>), dim3(grid, rows), dim3(256), lds, s[k], f, sys, w[k], D, W, \
                           G);                                                                                \
    }
    QK_1E_CLASSES(QK_1E)
#undef QK_1E
    hipLaunchKernelGGL(nuclear_grad_kernel, dim3((sys.natom + 255) / 256), dim3(256), 0, s[0], sys, G);
}

}  // namespace qk
