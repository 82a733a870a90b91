// erf_poly.hpp - polynomials for the GELU's erf on |z| < 3, for host and device code.
//
// The canonical erf is the Maclaurin series in double (device_common.hpp), rounded to
// float. On [0, 3) these polynomials round to the same float for every float argument
// (all 1,078 million checked against the series; the largest relative difference before
// rounding is 1.1e-15, 2.3e-15 and 1.3e-13 on the three intervals, the last one the
// series' own cancellation). From 3 on that cancellation reaches float boundaries (8 of
// the 2 million floats in [3, 3.5) differ), so [3, 4) keeps the series.
// Chebyshev fits of erf(sqrt(t)) / sqrt(t) on t in [0, 1], erf on [1, 2] about 1.5 and on
// [2, 3] about 2.5, highest power first, truncation below 3e-17.
#pragma once

namespace mtg {

constexpr double kErfPoly0[12] = {
    -0x1.ac9585a44fe29p-31, 0x1.d76af6ca49787p-27, -0x1.5c131500d3f88p-23, 0x1.b981d78881a5dp-20,
    -0x1.f4ca838adb73bp-17, 0x1.f9a2be4f731a1p-14, -0x1.c02db0665e53dp-11, 0x1.565bccfa44156p-8,
    -0x1.b82ce31203772p-6, 0x1.ce2f21a040f66p-4, -0x1.812746b0379c1p-2, 0x1.20dd750429b6dp+0};
constexpr double kErfPoly1[18] = {
    -0x1.305d37a851c9dp-22, 0x1.7c67db8e155e0p-20, 0x1.32b587a24f780p-21, -0x1.d70efbc5f9ed6p-17,
    0x1.2d574ba32d17bp-16, 0x1.45cc7994de082p-14, -0x1.0acf353ecb714p-12, -0x1.85b3d151e9cfdp-14,
    0x1.c0380d88e655ap-10, -0x1.35ae4fb43b234p-9, -0x1.36d73a65ecb0ap-8, 0x1.3ca3d72e94d2cp-6,
    -0x1.e723726b75a2bp-7, -0x1.6d5a95d0a8e2dp-5, 0x1.1c2a02beb6a99p-3, -0x1.6d5a95d0a1b3ap-3,
    0x1.e723726b824a9p-4, 0x1.eea5557137ae0p-1};
constexpr double kErfPoly2[17] = {
    0x1.4c5c2e28918dep-23, -0x1.4c8310c1df6c5p-21, 0x1.9c3a8df6aef99p-23, 0x1.3a22b06c6c19ap-18,
    -0x1.d887680497104p-17, 0x1.58e57ffcb4c61p-18, 0x1.4a84a0f850127p-14, -0x1.06718e6162745p-12,
    0x1.11551c4ad2affp-12, 0x1.1c610c9c3b183p-11, -0x1.6ecdbf65adc1dp-9, 0x1.90e81282f02d9p-8,
    -0x1.1a89b97ced2f0p-7, 0x1.119da0c46f2d8p-7, -0x1.64e3dcd3af454p-8, 0x1.1d83170fbf630p-9,
    0x1.ffcaa8f4c9beap-1};

}  // namespace mtg
