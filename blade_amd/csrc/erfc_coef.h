// Generated by fit_erfc.py: erfcx(x) ~ sum_k C[k] t^k, t = 1/(1+P x),
// x in [0,4.0], max relative error of the fit 7.20e-09 (exact arithmetic).
#pragma once
#define BM_ERFC_XMAX 4.0f
#define BM_ERFC_P 0.4f
#define BM_ERFC_DEG 9
static constexpr float bm_erfc_c[BM_ERFC_DEG + 1] = {
    5.551869645e-04f,
    2.167838891e-01f,
    2.884817546e-01f,
    -4.878207972e-02f,
    8.359773553e-01f,
    -1.002798473e+00f,
    1.285446394e+00f,
    -7.541636032e-01f,
    1.963993090e-01f,
    -1.789973063e-02f};
