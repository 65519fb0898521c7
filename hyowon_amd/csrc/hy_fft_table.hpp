// Table of the compiled FFT pass kernels: per mesh size, per pass, per launch
// variant.  The instantiations live in hy_fft_f32.hip and hy_fft_f64.hip so
// the two precisions compile in parallel.
#pragma once

#include "hy_fft_passes.hpp"

// Supported mesh sizes (compile-time FFT plans).
#define HY_MESH_SIZES(X) X(8) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512) X(1024)

namespace hy {

enum { FFT_Z_R2C = 0, FFT_Y_FWD, FFT_X_GREEN, FFT_Y_BWD, FFT_Z_C2R, FFT_PASSES };

template <typename T>
struct FftPass {
    void (*fn)(FftArgs<T>) = nullptr;
    int rows = 0, threads = 0, lds = 0;
};

template <typename T>
struct FftKernels {
    FftPass<T> pass[FFT_PASSES][kFftVariants];
    FftPass<T> x_fwd;  // forward-only x pass of the spectral estimators (in place on B)
    FftPass<T> z_fwd;  // z r2c pass of the spectral estimators (stores kz <= mode_limit only)
    FftPass<T> x_inv;  // inverse-only x pass of the IC displacements (in place on B)
    FftPass<T> sg[3];  // spectral-gradient x (fft_x_variant), y^-1 and z^-1 passes (variant 0; TreePM long range)
    bool sg_x_dual = false;  // sg[0] writes the -i k_x and the plain inverse from one read of B
    FftPass<T> sg_y_dual;    // y^-1 pass writing the -i k_y and the plain inverse from one read of B (or none)
    int variants = 0;  // launch variants compiled for this size
    int plan[FFT_PASSES] = {0, 0, 0, 0, 0};  // variants a context starts with (hy_pm_autotune refines them)
};

// Sizes below this have one launch variant (their passes are latency-bound and
// the variants collapse onto the same row counts).
constexpr int kFftTunedFrom = 192;

// Defined in hy_fft_f32.hip / hy_fft_f64.hip; false for an unsupported size.
bool lookup_fft(int N, FftKernels<float>& out);
bool lookup_fft(int N, FftKernels<double>& out);

#ifdef HY_FFT_INSTANTIATE
// Variant of the x passes with a Green multiply (the others of theirs are the
// autotuner's): they need LDS for the exchange only, so small workgroups keep more
// of them resident: 20 KB on 2^a meshes, as long as that makes a whole wave (at
// 1024 in binary64 it holds one row, 32 threads: 5.79 ms, the spectral gradient
// 11.0), else 40 KB.  Against 80 KB: 512^3 binary32 0.39 -> 0.28 ms, binary64
// 0.71 -> 0.60; 1024^3 binary32 1.91 -> 1.61, binary64 3.77 -> 3.41, its spectral
// gradient 6.48 -> 6.40; 384^3 binary32 0.126 -> 0.107, its spectral gradient 0.28 ->
// 0.19, binary64 0.34 and 0.34.
template <typename T, int N>
constexpr int fft_x_variant() {
    if (N < kFftTunedFrom) return 0;
    return (N & (N - 1)) == 0 && TLCfg<T, N, (N / 2 + 1) * N, 3>::THREADS >= 64 ? 3 : 1;
}

// ... and of the forward or inverse x passes, one transform each, which hold half the
// registers: 20 KB also where that is half a wave (1024^3 binary64 3.23 ms, 3.41 with
// 80 KB), but 80 KB on the large binary32 meshes (1024^3 1.45 ms, 1.52 with 20 KB).
template <typename T, int N>
constexpr int fft_x_dft_variant() {
    if (N < kFftTunedFrom || (N >= 512 && sizeof(T) == 4)) return 0;
    return (N & (N - 1)) == 0 ? 3 : 1;
}

template <typename T, int N, int V>
void fill_variant(FftKernels<T>& k) {
    using RZ = TLCfg<T, N / 2, N, V>;
    using RY = TLCfg<T, N, N, V>;
    using RX = TLCfg<T, N, (N / 2 + 1) * N, V>;
    k.pass[FFT_Z_R2C][V] = {k_tl_z_r2c<T, N, V>, RZ::ROWS, RZ::THREADS, RZ::LDS_BYTES};
    k.pass[FFT_Y_FWD][V] = {k_tl_y_fwd<T, N, V>, RY::ROWS, RY::THREADS, RY::LDS_BYTES};
    k.pass[FFT_X_GREEN][V] = {k_tl_x_green<T, N, V>, RX::ROWS, RX::THREADS, RX::X_LDS_BYTES};
    k.pass[FFT_Y_BWD][V] = {k_tl_y_bwd<T, N, V>, RY::ROWS, RY::THREADS, RY::LDS_BYTES};
    k.pass[FFT_Z_C2R][V] = {k_tl_z_c2r<T, N, V>, RZ::ROWS, RZ::THREADS, RZ::LDS_BYTES};
    if constexpr (V == fft_x_dft_variant<T, N>()) {
        k.x_fwd = {k_tl_x_dft<T, N, V, -1>, RX::ROWS, RX::THREADS, RX::X_LDS_BYTES};
        k.x_inv = {k_tl_x_dft<T, N, V, +1>, RX::ROWS, RX::THREADS, RX::X_LDS_BYTES};
    }
    if constexpr (V == fft_x_variant<T, N>()) {
        if constexpr (sizeof(T) == 4) {
            // binary32: the second held column fits the register file
            k.sg[0] = {k_tl_x_green_dual<T, N, V>, RX::ROWS, RX::THREADS, RX::X_LDS_BYTES};
            k.sg_x_dual = true;
        } else {
            k.sg[0] = {k_tl_x_green<T, N, V, 1>, RX::ROWS, RX::THREADS, RX::X_LDS_BYTES};
        }
    }
    if constexpr (V == 0) {
        k.z_fwd = {k_tl_z_r2c<T, N, V, true>, RZ::ROWS, RZ::THREADS, RZ::LDS_BYTES};
        if constexpr (sizeof(T) == 4)
            k.sg_y_dual = {k_tl_y_bwd<T, N, V, 2>, RY::ROWS, RY::THREADS, RY::LDS_BYTES};
        k.sg[1] = {k_tl_y_bwd<T, N, V, 1>, RY::ROWS, RY::THREADS, RY::LDS_BYTES};
        k.sg[2] = {k_tl_z_c2r<T, N, V, 1>, RZ::ROWS, RZ::THREADS, RZ::LDS_BYTES};
    }
}

// Variants a context starts with, from the measured times of all four:
//   x + Green: fft_x_variant;
//   256^3 y and y^-1: 40 KB (0.025 -> 0.021 ms);
//   192^3 z c2r: 64 rows in binary32 (one box 0.0165 -> 0.0152 ms, 64 boxes 1.06 ->
//     0.70), and 16 in binary64 with z r2c (one box 0.022 -> 0.017 and 0.022 ->
//     0.019 ms, 64 boxes 1.28 -> 1.27 and 1.27 -> 1.23).
template <typename T, int N>
constexpr int fft_plan(int pass) {
    if (N < kFftTunedFrom) return 0;
    if (pass == FFT_X_GREEN) return fft_x_variant<T, N>();
    if (N == 256 && (pass == FFT_Y_FWD || pass == FFT_Y_BWD)) return 1;
    if (N == 192 && sizeof(T) == 4 && pass == FFT_Z_C2R) return 2;
    if (N == 192 && sizeof(T) == 8 && (pass == FFT_Z_R2C || pass == FFT_Z_C2R)) return 1;
    return 0;
}

template <typename T, int N>
FftKernels<T> make_fft() {
    FftKernels<T> k{};
    fill_variant<T, N, 0>(k);
    k.variants = 1;
    if constexpr (N >= kFftTunedFrom) {
        fill_variant<T, N, 1>(k);
        fill_variant<T, N, 2>(k);
        fill_variant<T, N, 3>(k);
        k.variants = kFftVariants;
    }
    for (int p = 0; p < FFT_PASSES; ++p) k.plan[p] = fft_plan<T, N>(p);
    return k;
}

template <typename T>
bool lookup_fft_impl(int N, FftKernels<T>& out) {
    switch (N) {
#define HY_CASE(n) \
    case n: out = make_fft<T, n>(); return true;
        HY_MESH_SIZES(HY_CASE)
#undef HY_CASE
        default: return false;
    }
}
#endif

}  // namespace hy
