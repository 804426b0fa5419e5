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
// FP64: erfcx(x) ~ sum_k C[k] y^k, y = (x-A)/(x+A), x in [0,6.0], max relative
// error 6.7e-15 (FP64 arithmetic).
#define BM_ERFCD_XMAX 6.0
#define BM_ERFCD_A 3.0
#define BM_ERFCD_DEG 16
#define BM_ERFCD_COEF \
    1.79001151181390872e-01, \
    -3.26233560043039272e-01, \
    2.45603801712036413e-01, \
    -1.50115936500831354e-01, \
    7.16658372168390706e-02, \
    -2.43924992961200258e-02, \
    4.26913586564995565e-03, \
    7.07745462217680222e-04, \
    -5.97056950633524696e-04, \
    4.52717610492041735e-05, \
    6.40421707963862650e-05, \
    -1.29758169943538768e-05, \
    -8.08943775972313603e-06, \
    2.32818819053842469e-06, \
    1.85299232560947820e-06, \
    2.94872028627263940e-07, \
    -6.12414622653418494e-09
