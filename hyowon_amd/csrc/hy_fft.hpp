// Pencil FFT building blocks for the PM Poisson solve (gfx950).
//
// A row of LEN complex values is transformed in two levels of register DFTs
// (lengths A and B, LEN = A * B) with one exchange through LDS between them;
// a workgroup holds ROWS rows.  LEN = 2^a or 3*2^a.
//
// Twiddles come from one table tw[m] = exp(-2*pi*i*m/NT) (NT = mesh size),
// evaluated in binary64 on the host, read with a stride NT/LEN.
//
// Conventions follow the reference FFT backend (src/mesh/fft_backend.cpp:
// 1088-1145): forward transforms are unnormalized, the inverse is the
// unnormalized backward DFT; the 1/N^3 factor is folded into the Green
// multiply of the x pass.
#pragma once

#include "hy_device.hpp"

namespace hy {

// ---------------------------------------------------------------------------
// Complex helpers
// ---------------------------------------------------------------------------
template <typename C>
HY_HD C cadd(C a, C b) { return {a.x + b.x, a.y + b.y}; }
template <typename C>
HY_HD C csub(C a, C b) { return {a.x - b.x, a.y - b.y}; }
template <typename C>
HY_HD C cmul(C a, C b) {
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename C>
HY_HD C cconj(C a) { return {a.x, -a.y}; }
// multiply by s*i, s = +1 or -1
template <int S, typename C>
HY_HD C cmuli(C a) {
    if constexpr (S > 0) return {-a.y, a.x};
    else return {a.y, -a.x};
}

// In-register DFTs of radix 2, 3, 4, 8.  S = -1 forward, +1 backward.
template <int S, typename C>
HY_HD void dft2(C* u) {
    const C a = u[0], b = u[1];
    u[0] = cadd(a, b);
    u[1] = csub(a, b);
}

template <int S, typename C>
HY_HD void dft3(C* u) {
    using T = decltype(u[0].x);
    const T h = (T)0.86602540378443864676;  // sqrt(3)/2
    const C t1 = cadd(u[1], u[2]);
    const C t2 = {u[0].x - (T)0.5 * t1.x, u[0].y - (T)0.5 * t1.y};
    const C d0 = csub(u[1], u[2]);
    const C d = {(T)S * h * d0.x, (T)S * h * d0.y};
    const C id = {-d.y, d.x};
    u[0] = cadd(u[0], t1);
    u[1] = cadd(t2, id);
    u[2] = csub(t2, id);
}

template <int S, typename C>
HY_HD void dft4(C* u) {
    const C t0 = cadd(u[0], u[2]);
    const C t1 = csub(u[0], u[2]);
    const C t2 = cadd(u[1], u[3]);
    const C t3 = cmuli<S>(csub(u[1], u[3]));
    u[0] = cadd(t0, t2);
    u[2] = csub(t0, t2);
    u[1] = cadd(t1, t3);
    u[3] = csub(t1, t3);
}

template <int S, typename C>
HY_HD void dft8(C* u) {
    using T = decltype(u[0].x);
    C e[4] = {u[0], u[2], u[4], u[6]};
    C o[4] = {u[1], u[3], u[5], u[7]};
    dft4<S>(e);
    dft4<S>(o);
    const T r = (T)0.70710678118654752440;
    // w8^q for q = 1, 2, 3 with w8 = exp(S*2*pi*i/8)
    const C o1 = {r * (o[1].x - (T)S * o[1].y), r * ((T)S * o[1].x + o[1].y)};
    const C o2 = cmuli<S>(o[2]);
    const C o3 = {r * (-o[3].x - (T)S * o[3].y), r * ((T)S * o[3].x - o[3].y)};
    u[0] = cadd(e[0], o[0]);
    u[4] = csub(e[0], o[0]);
    u[1] = cadd(e[1], o1);
    u[5] = csub(e[1], o1);
    u[2] = cadd(e[2], o2);
    u[6] = csub(e[2], o2);
    u[3] = cadd(e[3], o3);
    u[7] = csub(e[3], o3);
}

template <int R, int S, typename C>
HY_HD void dftR(C* u) {
    if constexpr (R == 2) dft2<S>(u);
    else if constexpr (R == 3) dft3<S>(u);
    else if constexpr (R == 4) dft4<S>(u);
    else dft8<S>(u);
}

// ---------------------------------------------------------------------------
// Register DFTs of length 2..32 (natural order in and out) and the two-level
// row FFT built on them.
// ---------------------------------------------------------------------------
// cos(2 pi m / 32) over the first quarter turn, correctly rounded; the other
// quadrants and the sines are these values mirrored.
constexpr double kCos32[9] = {1.0, 0.98078528040323043, 0.92387953251128674, 0.83146961230254524,
                              0.70710678118654757, 0.55557023301960218, 0.38268343236508978,
                              0.19509032201612828, 0.0};

HY_HD constexpr double cos32(int m) {
    int q = m & 31;
    if (q > 16) q = 32 - q;
    return q > 8 ? -kCos32[16 - q] : kCos32[q];
}

// exp(S 2 pi i m / R) for R | 32, as a complex constant of type C.
template <int R, int S, typename C>
HY_HD C wconst(int m) {
    using T = decltype(C{}.x);
    const int q = m * (32 / R);
    return C{(T)cos32(q), (T)(S * cos32(q - 8))};
}

// In-register DFT of length R (2^a <= 32, or 3 * 2^a <= 24), natural order in
// and out, in place.
//   R = 3 M: the prime-factor algorithm (Good, Thomas), a 3 x M transform
//     without twiddles: input M n1 + 3 n2 and output k with k = k1 mod 3, k = k2 mod M
//     (compile-time permutations of registers).  With twiddles exp(2 pi i m / 24)
//     instead the row transforms of 24 and 48 were 4 and 2% less accurate.
//   else R = 4 B: a length-4 DFT over each stride-B column, the twiddle
//     exp(S 2 pi i n2 k1 / R), then a length-B DFT over each row.
template <int R, int S, typename C>
HY_HD void dft_reg(C* u) {
    if constexpr (R == 2 || R == 3 || R == 4 || R == 8) {
        dftR<R, S>(u);
    } else if constexpr (R % 3 == 0) {
        constexpr int M = R / 3;
        // M (M^-1 mod 3) = M^2 as 2^-1 = 2 mod 3; 3 (3^-1 mod M) = 3, 9 and 9 for M = 2, 4, 8
        constexpr int e1 = M * M % R, e2 = (M == 2 ? 3 : 9) % R;
        static_assert(e1 % 3 == 1 && e1 % M == 0 && e2 % 3 == 0 && e2 % M == 1, "Chinese remainders");
        C y[R];
#pragma unroll
        for (int n1 = 0; n1 < 3; ++n1) {
#pragma unroll
            for (int n2 = 0; n2 < M; ++n2) y[n1 * M + n2] = u[(M * n1 + 3 * n2) % R];
            dftR<M, S>(y + n1 * M);
        }
#pragma unroll
        for (int k2 = 0; k2 < M; ++k2) {
            C col[3] = {y[k2], y[M + k2], y[2 * M + k2]};
            dft3<S>(col);
#pragma unroll
            for (int k1 = 0; k1 < 3; ++k1) u[(e1 * k1 + e2 * k2) % R] = col[k1];
        }
    } else {
        constexpr int A = 4, B = R / A;
        C y[R];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) {
            C col[A];
#pragma unroll
            for (int n1 = 0; n1 < A; ++n1) col[n1] = u[B * n1 + n2];
            dft4<S>(col);
#pragma unroll
            for (int k1 = 0; k1 < A; ++k1)
                y[k1 * B + n2] = (k1 * n2 == 0) ? col[k1] : cmul(col[k1], wconst<R, S, C>(k1 * n2));
        }
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) {
            C row[B];
#pragma unroll
            for (int n2 = 0; n2 < B; ++n2) row[n2] = y[k1 * B + n2];
            dftR<B, S>(row);
#pragma unroll
            for (int k2 = 0; k2 < B; ++k2) u[k1 + A * k2] = row[k2];
        }
    }
}

// Two-level row FFT of length LEN = A * B (A <= B <= 32; 2^a from 4 to 1024 or
// 3 * 2^a from 6 to 384; A and B as near each other as the length allows):
//   level 1: thread n2 < B holds the stride-B column x[n2 + B n1] (n1 < A),
//            transforms it (length A) and multiplies by W_LEN^(n2 k1);
//   exchange: Y[k1][n2] through LDS (row stride B + 1);
//   level 2: thread k1 < A holds row Y[k1][*], transforms it (length B) and
//            then holds X[k1 + A k2], k2 < B.
// The inverse of a spectrum held as in level 2 is the same procedure with
// A and B exchanged.
template <int LEN>
struct TwoLevel {
    static constexpr int lg(int v) { return v <= 1 ? 0 : 1 + lg(v / 2); }
    static constexpr bool has3 = LEN % 3 == 0;
    static constexpr int K = lg(has3 ? LEN / 3 : LEN);
    static constexpr int A = !has3 ? 1 << (K / 2) : (K % 2 ? 1 << ((K + 1) / 2) : 3 << (K / 2 - 1));
    static constexpr int B = LEN / A;
    static constexpr int TPR = A > B ? A : B;
    static constexpr int EMAX = A > B ? A : B;
    // exchange region per row (complex): A rows of B+1 or B rows of A+1
    static constexpr int XS0 = (A * (B + 1) > B * (A + 1) ? A * (B + 1) : B * (A + 1));
    static constexpr int XS = XS0 % 2 == 0 ? XS0 + 1 : XS0;
    static_assert(A * B == LEN && A <= 32 && B <= 32 && A >= 2, "two-level FFT length");
};

// Level-1 twiddle: v[k1] *= W_LEN^(S col k1), twiddles from the table
// tw[m * stride] = exp(-2 pi i m / LEN).
// Level-1 twiddles split into the loads, issued with a pass's row loads so
// their latency hides under the row fetch, and the multiplies, which match
// tl_twiddle's arithmetic.
template <int A, int LEN, typename C>
HY_HD void tl_twiddle_load(C* w, int col, const C* tw, int stride) {
#pragma unroll
    for (int k1 = 1; k1 < A; ++k1) w[k1] = tw[((col * k1) % LEN) * stride];
}

template <int A, int S, typename C>
HY_HD void tl_twiddle_apply(C* v, const C* w) {
#pragma unroll
    for (int k1 = 1; k1 < A; ++k1) {
        C x = w[k1];
        if constexpr (S > 0) x.y = -x.y;
        v[k1] = cmul(v[k1], x);
    }
}

// Level-1 twiddles W^(col k1), k1 = 1 .. A-1, as the products
// W^(col j) W^(col L h) (k1 = j + L h) of L - 1 + H - 1 table entries instead
// of A - 1: for A = 32 a row holds 10 complex factors in registers rather
// than 31 (the registers that bound the passes' occupancy), at one rounding
// more per twiddle.
template <int A>
struct TwSplit {
    static constexpr int L = A >= 16 ? 8 : A;
    static constexpr int H = (A + L - 1) / L;
};

template <int A, int LEN, typename C>
HY_HD void tl_twiddle_load_split(C* lo, C* hi, int col, const C* tw, int stride) {
    constexpr int L = TwSplit<A>::L, H = TwSplit<A>::H;
#pragma unroll
    for (int j = 1; j < L; ++j) lo[j] = tw[((col * j) % LEN) * stride];
#pragma unroll
    for (int h = 1; h < H; ++h) hi[h] = tw[((col * L * h) % LEN) * stride];
}

template <int A, int S, typename C>
HY_HD void tl_twiddle_apply_split(C* v, const C* lo, const C* hi) {
    constexpr int L = TwSplit<A>::L;
#pragma unroll
    for (int k1 = 1; k1 < A; ++k1) {
        const int j = k1 % L, h = k1 / L;
        C x = h == 0 ? lo[j] : (j == 0 ? hi[h] : cmul(lo[j], hi[h]));
        if constexpr (S > 0) x.y = -x.y;
        v[k1] = cmul(v[k1], x);
    }
}

// The table loads go out in batches of TB ahead of their multiplies (a
// scheduling barrier keeps the compiler from interleaving them with the
// uses), so a row pays (A - 1) / TB memory round trips for its twiddles rather
// than up to one per twiddle.
template <int A, int LEN, int S, int TB = 16, typename C>
HY_HD void tl_twiddle(C* v, int col, const C* tw, int stride) {
#pragma unroll
    for (int k0 = 1; k0 < A; k0 += TB) {
        C w[TB];
#pragma unroll
        for (int j = 0; j < TB; ++j) {
            if (k0 + j < A) w[j] = tw[((col * (k0 + j)) % LEN) * stride];
        }
#ifdef __HIP_DEVICE_COMPILE__
        __builtin_amdgcn_sched_barrier(0);
#endif
#pragma unroll
        for (int j = 0; j < TB; ++j) {
            if (k0 + j < A) {
                C x = w[j];
                if constexpr (S > 0) x.y = -x.y;
                v[k0 + j] = cmul(v[k0 + j], x);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Per-pass launch geometry
// ---------------------------------------------------------------------------
// Launch variants of every pass (chosen per pass by the autotuner): an LDS
// budget per workgroup, which sets the rows per workgroup and therefore the
// workgroups resident per CU (160 KB of LDS each) and the length of the
// contiguous runs of the transposing stores.
constexpr int kFftVariants = 4;
constexpr int fft_lds_budget(int v) {
    return v == 0 ? 80 * 1024 : v == 1 ? 40 * 1024 : v == 2 ? 136 * 1024 : 20 * 1024;
}
// Rows shorter than 64, and the y and x rows of a 64^3 mesh: 128 threads, so
// that a small mesh still makes a workgroup or two per CU (a 64^3 mesh: 132 per
// y pass, 16 rows each; 4.8 -> 3.2 us against one workgroup of 64 rows).  The
// z rows of a 128^3 mesh (LEN 64) keep 64 rows: 16 of them read 128-byte runs,
// 0.29 against 0.20 ms for 64 boxes.
constexpr int fft_thread_cap(int v, int len, int dim) {
    return len < 64 || (len == 64 && dim != 128) ? 128 : v == 2 ? 1024 : 512;
}

constexpr int pow2_floor(int v) {
    int p = 1;
    while (p * 2 <= v) p *= 2;
    return p;
}

// Launch geometry of the two-level passes: ROWS rows per workgroup, TPR
// threads per row; the LDS holds either the per-row exchange (XS complex per
// row), a natural-order copy of the rows (LEN + 1 per row) or the transposed
// tile of the y passes (LEN x (ROWS + 1)).
template <typename T, int LEN, int DIM, int V = 0>
struct TLCfg {
    using C = cplx<T>;
    using TL = TwoLevel<LEN>;
    static constexpr int TPR = TL::TPR;
    static constexpr int PER_ROW = (TL::XS > LEN + 1 ? TL::XS : LEN + 1) + LEN / 8 + 1;
    static constexpr int by_threads = fft_thread_cap(V, LEN, DIM) / TPR;
    static constexpr int by_lds = fft_lds_budget(V) / (PER_ROW * (int)sizeof(C));
    static constexpr int cap = by_threads < by_lds ? by_threads : by_lds;
    static constexpr int dim_pow2 = (DIM & (-DIM));
    static constexpr int ROWS0 = pow2_floor(cap < 1 ? 1 : cap);
    static constexpr int ROWS = ROWS0 < dim_pow2 ? ROWS0 : dim_pow2;
    static constexpr int THREADS = ROWS * TPR;
    static constexpr int NAT = LEN + 1;  // natural-order row stride (odd)
    static constexpr int TS = ROWS + 1;  // transposed tile row stride
    static constexpr int ELEMS = (ROWS * TL::XS > ROWS * NAT ? ROWS * TL::XS : ROWS * NAT) > LEN * TS
                                     ? (ROWS * TL::XS > ROWS * NAT ? ROWS * TL::XS : ROWS * NAT)
                                     : LEN * TS;
    static constexpr int LDS_BYTES = ELEMS * (int)sizeof(C);
    // the x passes use only the per-row exchange regions (no transposed tile)
    static constexpr int X_LDS_BYTES = ROWS * TL::XS * (int)sizeof(C);
    static_assert(LDS_BYTES <= 160 * 1024, "LDS per workgroup");
};

}  // namespace hy
