// Register-direct complex FFT of compile-time length for gfx950 (FP64).
//
// The Stockham transform of fft_ct.h keeps a tile in LDS from the load to the
// store: every stage, the staging of the input and the real/halfcomplex
// conversion are LDS round trips.  Here the first stage takes its inputs
// straight from memory and the last one hands its outputs straight to memory,
// so a transform of S stages makes S - 1 LDS round trips.
//
// The real/halfcomplex conversion needs elements t and N - t together.  The
// last stage of radix R (m = N/R butterflies) yields elements j + q m, and the
// first one reads elements j + r m: element N - (j + q m) belongs to butterfly
// m - j, so a thread that runs butterflies p and m - p holds every pair.
// Pairs are p = 0 .. m/2: p = 0 runs butterfly 0 twice, the second time with
// its outputs turned by one (its twiddles are those of k = m), so the pairing
// needs no special case; p = m/2 (m even) runs its butterfly twice.
#pragma once

#include <hip/hip_runtime.h>

#include "fft_ct.h"

namespace dnsp {

// ---------------------------------------------------------------------------
// radix plan
// ---------------------------------------------------------------------------
constexpr int kRgMaxStages = 4;
struct RgPlan {
    int nf;
    int r[kRgMaxStages];
};

// Instructions per element of a radix, roughly (0: not a radix).
constexpr int rg_radix_cost(int r) {
    constexpr int c[17] = {0, 0, 2, 5, 4, 8, 7, 15, 6, 10, 10, 23, 9, 27, 0, 13, 8};
    return r <= 16 ? c[r] : 0;
}
// Extra cost of a radix by the registers its butterflies take: 4 VGPRs per
// complex value, twice the values in the paired stage.
constexpr int rg_reg_cost(int r, bool paired) {
    return paired ? (r > 8 ? 6 * (r - 8) : 0) : (r > 12 ? 2 * (r - 12) : 0);
}
constexpr int kRgExchangeCost = 30;  // an LDS round trip with its barriers

// The cheapest split of n into at most kRgMaxStages radices; the paired stage
// is the last one (forward) or the first one (inverse).  nf = 0: none.
constexpr RgPlan rg_plan(int n, bool inv) {
    RgPlan best{0, {0, 0, 0, 0}};
    int bc = 1 << 30;
    for (int a = 2; a <= 16; ++a) {
        if (n % a || !rg_radix_cost(a)) continue;
        for (int b = 1; b <= 16; ++b) {
            if ((n / a) % b || (b > 1 && !rg_radix_cost(b))) continue;
            for (int c = 1; c <= 16; ++c) {
                if ((n / a / b) % c || (c > 1 && (b == 1 || !rg_radix_cost(c)))) continue;
                const int d = n / a / b / c;
                if (d > 16 || (d > 1 && (c == 1 || !rg_radix_cost(d)))) continue;
                const int nf = 1 + (b > 1) + (c > 1) + (d > 1);
                if (nf < 2) continue;  // one exchange at least: first and last stage differ
                const int r[4] = {a, b, c, d};
                int cost = kRgExchangeCost * (nf - 1);
                for (int s = 0; s < nf; ++s) {
                    const bool paired = s == (inv ? 0 : nf - 1);
                    cost += rg_radix_cost(r[s]) + rg_reg_cost(r[s], paired);
                }
                if (cost < bc) {
                    bc = cost;
                    best = RgPlan{nf, {a, b, c, d}};
                }
            }
        }
    }
    return best;
}

template <int N, bool INV>
struct Rg {
    static constexpr RgPlan plan = rg_plan(N, INV);
    static constexpr int nf = plan.nf;
    static constexpr int r0 = plan.r[0];
    static constexpr int rl = plan.r[nf > 0 ? nf - 1 : 0];
    static constexpr int radix(int s) { return plan.r[s]; }
    static constexpr int ns(int s) {
        int v = 1;
        for (int i = 0; i < s; ++i) v *= plan.r[i];
        return v;
    }
    // paired items of one line
    static constexpr int mp = N / (INV ? r0 : rl);
    static constexpr int pairs = mp / 2 + 1;
};

// ---------------------------------------------------------------------------
// radices
// ---------------------------------------------------------------------------
// Odd prime R: sums and differences of v[r], v[R - r] against real cosines and
// sines (ceil-half of the products of the plain sum).
template <int R, bool INV, typename V>
__device__ __forceinline__ void dft_odd(V* v, const double (&co)[R / 2 + 1], const double (&si)[R / 2 + 1]) {
    using T = decltype(v[0].x);
    constexpr int H = R / 2;
    V t[H + 1], d[H + 1];
    V s = v[0];
#pragma unroll
    for (int r = 1; r <= H; ++r) {
        t[r] = cadd(v[r], v[R - r]);
        d[r] = csub(v[r], v[R - r]);
        s = cadd(s, t[r]);
    }
#pragma unroll
    for (int q = 1; q <= H; ++q) {
        V m = v[0], e;
        e.x = e.y = T(0);
#pragma unroll
        for (int r = 1; r <= H; ++r) {
            const int i = (q * r) % R;
            const T c = T(i <= H ? co[i] : co[R - i]);
            const T w = T(i <= H ? si[i] : -si[R - i]);
            m.x += c * t[r].x;
            m.y += c * t[r].y;
            e.x += w * d[r].x;
            e.y += w * d[r].y;
        }
        e = rot<INV>(e);
        v[q] = cadd(m, e);  // v[1..H] is no longer read (t, d hold it)
        v[R - q] = csub(m, e);
    }
    v[0] = s;
}

template <bool INV, typename V>
__device__ __forceinline__ void dft7(V* v) {
    constexpr double c[4] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
    constexpr double s[4] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
    dft_odd<7, INV>(v, c, s);
}
template <bool INV, typename V>
__device__ __forceinline__ void dft11(V* v) {
    constexpr double c[6] = {1.0, 0.84125353283118116886, 0.41541501300188642553, -0.14231483827328514044,
                             -0.65486073394528506406, -0.95949297361449738989};
    constexpr double s[6] = {0.0, 0.54064081745559758211, 0.90963199535451837141, 0.98982144188093273238,
                             0.75574957435425828377, 0.28173255684142969771};
    dft_odd<11, INV>(v, c, s);
}
template <bool INV, typename V>
__device__ __forceinline__ void dft13(V* v) {
    constexpr double c[7] = {1.0, 0.88545602565320989590, 0.56806474673115580251, 0.12053668025532305335,
                             -0.35460488704253562597, -0.74851074817110109863, -0.97094181742605202716};
    constexpr double s[7] = {0.0, 0.46472317204376854566, 0.82298386589365639458, 0.99270887409805399280,
                             0.93501624268541482344, 0.66312265824079520238, 0.23931566428755776715};
    dft_odd<13, INV>(v, c, s);
}

template <int R, bool INV, typename V>
__device__ __forceinline__ void rg_dft(V* v);

// R = A B with A, B coprime (Good-Thomas): no twiddles between the two.
template <int A, int B, bool INV, typename V>
__device__ __forceinline__ void dft_pfa(V* v) {
    constexpr int R = A * B;
    constexpr auto inv_mod = [](int x, int m) {
        for (int i = 1; i < m; ++i)
            if ((x * i) % m == 1) return i;
        return 0;
    };
    constexpr int ea = B * inv_mod(B % A, A), eb = A * inv_mod(A % B, B);  // = 1 mod A / 0 mod B and the reverse
    V w[A][B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        V c[A];
#pragma unroll
        for (int a = 0; a < A; ++a) c[a] = v[(B * a + A * b) % R];
        rg_dft<A, INV>(c);
#pragma unroll
        for (int a = 0; a < A; ++a) w[a][b] = c[a];
    }
#pragma unroll
    for (int a = 0; a < A; ++a) {
        rg_dft<B, INV>(w[a]);
#pragma unroll
        for (int b = 0; b < B; ++b) v[(a * ea + b * eb) % R] = w[a][b];
    }
}

// R = A B with twiddles exp(-2 pi i a b / R) = (co[a b], -si[a b]).
template <int A, int B, bool INV, typename V, int L>
__device__ __forceinline__ void dft_ab(V* v, const double (&co)[L], const double (&si)[L]) {
    using T = decltype(v[0].x);
    V w[A][B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        V c[A];
#pragma unroll
        for (int a = 0; a < A; ++a) c[a] = v[B * a + b];
        rg_dft<A, INV>(c);
#pragma unroll
        for (int a = 0; a < A; ++a) {
            V t;
            t.x = T(co[a * b]);
            t.y = T(-si[a * b]);
            w[a][b] = a * b == 0 ? c[a] : (INV ? cmulc(c[a], t) : cmul(c[a], t));
        }
    }
#pragma unroll
    for (int a = 0; a < A; ++a) {
        rg_dft<B, INV>(w[a]);
#pragma unroll
        for (int b = 0; b < B; ++b) v[a + A * b] = w[a][b];
    }
}

template <bool INV, typename V>
__device__ __forceinline__ void dft9(V* v) {
    constexpr double c[5] = {1.0, 0.76604444311897803520, 0.17364817766693034885, -0.5, -0.93969262078590838405};
    constexpr double s[5] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676,
                             0.34202014332566873304};
    dft_ab<3, 3, INV>(v, c, s);
}
template <bool INV, typename V>
__device__ __forceinline__ void dft16(V* v) {
    constexpr double h = 0.70710678118654752440, c1 = 0.92387953251128675613, s1 = 0.38268343236508977173;
    constexpr double c[10] = {1.0, c1, h, s1, 0.0, -s1, -h, -c1, -1.0, -c1};
    constexpr double s[10] = {0.0, s1, h, c1, 1.0, c1, h, s1, 0.0, -s1};
    dft_ab<4, 4, INV>(v, c, s);
}

template <int R, bool INV, typename V>
__device__ __forceinline__ void rg_dft(V* v) {
    if constexpr (R == 2) dft2<INV>(v);
    else if constexpr (R == 3) dft3<INV>(v);
    else if constexpr (R == 4) dft4<INV>(v);
    else if constexpr (R == 5) dft5<INV>(v);
    else if constexpr (R == 6) dft_pfa<2, 3, INV>(v);
    else if constexpr (R == 7) dft7<INV>(v);
    else if constexpr (R == 8) dft8<INV>(v);
    else if constexpr (R == 9) dft9<INV>(v);
    else if constexpr (R == 10) dft_pfa<2, 5, INV>(v);
    else if constexpr (R == 11) dft11<INV>(v);
    else if constexpr (R == 12) dft_pfa<4, 3, INV>(v);
    else if constexpr (R == 13) dft13<INV>(v);
    else if constexpr (R == 15) dft_pfa<3, 5, INV>(v);
    else if constexpr (R == 16) dft16<INV>(v);
    else static_assert(R == 1, "radix");
}

// ---------------------------------------------------------------------------
// transforms of G lines by NT threads, line g at buf[g LP + ct_pad(element)]
// ---------------------------------------------------------------------------
// Item idx of `per` items a line -> (line, item); LF: the line index runs
// fastest (z: adjacent columns are adjacent in memory).
template <int G, bool LF>
__device__ __forceinline__ void rg_item(int idx, int per, int& g, int& j) {
    if constexpr (LF) {
        j = idx / G;
        g = idx - j * G;
    } else {
        g = idx / per;
        j = idx - g * per;
    }
}

// Stage s, neither first nor last: LDS to LDS.
template <int N, bool INV, int S, int G, int NT, int LP>
__device__ __forceinline__ void rg_mid(double2* buf, const double2* __restrict__ tw) {
    constexpr int R = Rg<N, INV>::radix(S), NS = Rg<N, INV>::ns(S), m = N / R, tstep = N / (NS * R);
    constexpr int tot = G * m, NB = (tot + NT - 1) / NT;
    double2 v[NB][R];
    int base[NB];
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        int idx = (int)threadIdx.x + q * NT;
        idx = (tot % NT == 0 || idx < tot) ? idx : 0;
        const int g = idx / m, j = idx - g * m, k = j % NS;
#pragma unroll
        for (int r = 0; r < R; ++r) v[q][r] = buf[g * LP + ct_pad(j + r * m)];
#pragma unroll
        for (int r = 1; r < R; ++r) {
            const double2 w = tw[r * k * tstep];
            v[q][r] = INV ? cmulc(v[q][r], w) : cmul(v[q][r], w);
        }
        base[q] = g * LP;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        const int idx = (int)threadIdx.x + q * NT;
        rg_dft<R, INV>(v[q]);
        if (tot % NT == 0 || idx < tot) {
            const int j = idx - (idx / m) * m, k = j % NS, dst = (j / NS) * NS * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) buf[base[q] + ct_pad(dst + r * NS)] = v[q][r];
        }
    }
    __syncthreads();
}

template <int N, bool INV, int S, int G, int NT, int LP>
__device__ __forceinline__ void rg_mids(double2* buf, const double2* __restrict__ tw) {
    if constexpr (S < Rg<N, INV>::nf - 1) {
        rg_mid<N, INV, S, G, NT, LP>(buf, tw);
        rg_mids<N, INV, S + 1, G, NT, LP>(buf, tw);
    }
}

// Whether element p + r m of the paired stage is 0 or N/2 (m R = N), the two
// without a mirror image: N/2 is (R/2) m for even R and m/2 + (R/2) m for odd R.
template <int R>
__device__ __forceinline__ bool rg_single(int r, int p, int m) {
    if (r == 0 || 2 * r == R) return p == 0;
    return 2 * r + 1 == R && 2 * p == m;
}

// Forward transform of G pairs of real lines (u, v): ld(g, j, m, v) loads
// elements j + r m of pair g as v[r] = (u, v); st(g, lo, hi, both, L, H) gets
// the halfcomplex entries lo <= N/2 as L = (u_lo, v_lo) and, when both, hi = N
// - lo as H.
template <int N, int G, int NT, int LP, bool LF, class LD, class ST>
__device__ __forceinline__ void rg_forward(double2* buf, const double2* __restrict__ tw, const LD& ld, const ST& st) {
    using P = Rg<N, false>;
    {
        constexpr int R = P::r0, m = N / R, tot = G * m, NB = (tot + NT - 1) / NT;
        double2 v[NB][R];
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            int idx = (int)threadIdx.x + q * NT, g, j;
            idx = (tot % NT == 0 || idx < tot) ? idx : 0;
            rg_item<G, LF>(idx, m, g, j);
            ld(g, j, m, v[q]);
        }
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            const int idx = (int)threadIdx.x + q * NT;
            rg_dft<R, false>(v[q]);
            if (tot % NT == 0 || idx < tot) {
                int g, j;
                rg_item<G, LF>(idx, m, g, j);
#pragma unroll
                for (int r = 0; r < R; ++r) buf[g * LP + ct_pad(j * R + r)] = v[q][r];
            }
        }
    }
    __syncthreads();
    rg_mids<N, false, 1, G, NT, LP>(buf, tw);
    constexpr int R = P::rl, m = N / R, tot = G * P::pairs, NB = (tot + NT - 1) / NT;
#pragma unroll 1
    for (int q = 0; q < NB; ++q) {
        const int idx = (int)threadIdx.x + q * NT;
        if (tot % NT == 0 || idx < tot) {
            int g, p;
            rg_item<G, LF>(idx, P::pairs, g, p);
            const int j2 = p == 0 ? 0 : m - p, k2 = m - p;
            double2 a[R], b[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                a[r] = buf[g * LP + ct_pad(p + r * m)];
                b[r] = buf[g * LP + ct_pad(j2 + r * m)];
            }
#pragma unroll
            for (int r = 1; r < R; ++r) {
                a[r] = cmul(a[r], tw[r * p]);
                b[r] = cmul(b[r], tw[r * k2]);
            }
            rg_dft<R, false>(a);
            rg_dft<R, false>(b);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                // elements t = p + r m (a) and N - t (b); t <= N/2 exactly when 2 r < R
                const bool lo = 2 * r < R;
                const double2 C = lo ? a[r] : b[R - 1 - r], D = lo ? b[R - 1 - r] : a[r];
                const int t = p + r * m, l = lo ? t : N - t;
                // hi = N - l exists unless l is 0 or N/2
                const bool both = !rg_single<R>(r, p, m);
                st(g, l, N - l, both, make_double2(0.5 * (C.x + D.x), 0.5 * (C.y + D.y)),
                   make_double2(0.5 * (C.y - D.y), 0.5 * (D.x - C.x)));
            }
        }
    }
}

// Inverse transform of G pairs of halfcomplex lines: ld(g, lo, hi, A, B)
// loads A = (u_lo, v_lo), B = (u_hi, v_hi) (hi clamped to lo where there is no
// such entry: B is then ignored); st(g, j, m, v) stores elements j + q m.
template <int N, int G, int NT, int LP, bool LF, class LD, class ST>
__device__ __forceinline__ void rg_inverse(double2* buf, const double2* __restrict__ tw, const LD& ld, const ST& st) {
    using P = Rg<N, true>;
    {
        constexpr int R = P::r0, m = N / R, tot = G * P::pairs, NB = (tot + NT - 1) / NT;
        double2 A[NB][R], B[NB][R];
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            int idx = (int)threadIdx.x + q * NT, g, p;
            idx = (tot % NT == 0 || idx < tot) ? idx : 0;
            rg_item<G, LF>(idx, P::pairs, g, p);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int t = p + r * m, lo = 2 * r < R ? t : N - t;
                int hi = N - lo;
                if (r == 0) hi = p == 0 ? 0 : hi;
                ld(g, lo, hi, A[q][r], B[q][r]);
            }
        }
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            const int idx = (int)threadIdx.x + q * NT;
            int g, p;
            rg_item<G, LF>(idx, P::pairs, g, p);
            double2 a[R], b[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const bool lo = 2 * r < R;
                double2 u = A[q][r], w = B[q][r];  // (ur, vr), (ui, vi)
                if (rg_single<R>(r, p, m)) w = make_double2(0.0, 0.0);
                const double2 L = make_double2(u.x - w.y, w.x + u.y), H = make_double2(u.x + w.y, u.y - w.x);
                a[r] = lo ? L : H;
                b[R - 1 - r] = lo ? H : L;
            }
            rg_dft<R, true>(a);
            rg_dft<R, true>(b);
            if (tot % NT == 0 || idx < tot) {
#pragma unroll
                for (int r = 0; r < R; ++r) buf[g * LP + ct_pad(p * R + r)] = a[r];
                if (p != 0 && 2 * p != m) {
#pragma unroll
                    for (int r = 0; r < R; ++r) buf[g * LP + ct_pad((m - p) * R + r)] = b[r];
                }
            }
        }
    }
    __syncthreads();
    rg_mids<N, true, 1, G, NT, LP>(buf, tw);
    constexpr int R = P::rl, m = N / R, tot = G * m, NB = (tot + NT - 1) / NT;
#pragma unroll 1
    for (int q = 0; q < NB; ++q) {
        const int idx = (int)threadIdx.x + q * NT;
        if (tot % NT == 0 || idx < tot) {
            int g, j;
            rg_item<G, LF>(idx, m, g, j);
            double2 v[R];
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = buf[g * LP + ct_pad(j + r * m)];
#pragma unroll
            for (int r = 1; r < R; ++r) v[r] = cmulc(v[r], tw[r * j]);
            rg_dft<R, true>(v);
            st(g, j, m, v);
        }
    }
}

}  // namespace dnsp
