// Launcher of the K-range tile GEMM (b1_tile_gemm.h): which tile and how
// many K ranges a shape runs with.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "b1_device.h"
#include "b1_internal.h"

namespace b1 {
namespace {

#include "b1_tile_gemm.h"

// The tiles, by number of K ranges: BM x WN per wave, NWN waves along N, KG
// ranges, KS per stage, R stages in the ring, and whether the packed-output
// epilogue can use them (whole 32-column blocks; 64 for SwiGLU pairs).
//                 BM  WN NWN KG  KS  R
using T8s = TileCfg<32, 48, 1, 8, 64, 3>;
using T8 = TileCfg<64, 48, 1, 8, 64, 2>;
using T8sp = TileCfg<32, 64, 1, 8, 64, 3>;
using T8p = TileCfg<64, 64, 1, 8, 64, 2>;
using T4s = TileCfg<32, 48, 2, 4, 64, 4>;
using T4 = TileCfg<64, 48, 2, 4, 64, 4>;
using T4p = TileCfg<64, 64, 2, 4, 64, 3>;
using T2s = TileCfg<64, 48, 2, 2, 64, 4>;
using T2sp = TileCfg<64, 64, 2, 2, 64, 3>;
using T2 = TileCfg<64, 48, 4, 2, 64, 4>;
using T1s = TileCfg<32, 48, 4, 1, 64, 4>;
using T1 = TileCfg<64, 48, 4, 1, 128, 3>;
using T1b = TileCfg<128, 48, 4, 1, 64, 3>;

// Time model of a launch, in microseconds, from launches of 0.7 to 116
// GFLOP on 256 CUs (within ~15 % of each): 2 + q (e + c b), q tiles per CU
// (rounded up) of b = K / 32 / KG blocks per wave group each; a lone tile
// of a configuration that shares a CU runs slower than one of two (c1).
struct TileCost {
    double e, c, c1;
};
template <class C>
constexpr TileCost tile_cost() {
    if (C::KG == 8) return C::BM == 32 ? TileCost{0.8, 0.40, 0.40} : TileCost{2.2, 0.56, 0.56};
    if (C::KG == 4) return C::BM == 32 ? TileCost{1.9, 0.34, 0.34} : TileCost{2.8, 0.48, 0.48};
    if (C::KG == 2) return C::BN == 192 ? TileCost{3.0, 0.38, 0.38} : TileCost{1.5, 0.23, 0.26};
    if (C::BM == 32) return TileCost{0.8, 0.14, 0.20};
    return C::BM == 64 ? TileCost{0.6, 0.19, 0.24} : TileCost{1.5, 0.335, 0.35};
}
template <class C>
double tile_us(int M, int K, int N, int num_cus) {
    const TileCost t = tile_cost<C>();
    const int64_t tiles = (int64_t)((M + C::BM - 1) / C::BM) * ((N + C::BN - 1) / C::BN);
    const double q = (double)((tiles + num_cus - 1) / num_cus), b = (double)(K / 32) / C::KG;
    return 2.0 + q * (t.e + (q > 1 ? t.c : t.c1) * b);
}

template <class C, int EPI>
hipError_t launch_tile(const void *packed, const uint8_t *w, int K, int N, int M, float *out, int64_t ldo,
                       int32_t *nonfinite, const GemmEpi &epi, hipStream_t s) {
    auto kernel = &b1_tile_gemm_kernel<C, EPI>;
    static std::once_flag attr_once;
    static hipError_t attr_err = hipSuccess;
    std::call_once(attr_once, [kernel] {
        attr_err = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
    });
    if (attr_err != hipSuccess) return attr_err;
    auto al16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    bool vec = al16(out) && ldo % 4 == 0;
    if (EPI == 1) vec = vec && al16(epi.res) && al16(epi.gate) && epi.ldr % 4 == 0;
    const int tiles_m = (M + C::BM - 1) / C::BM, tiles_n = (N + C::BN - 1) / C::BN;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((int64_t)tiles_m * tiles_n)), dim3(C::NT), C::LDS, s,
                       static_cast<const uint16_t *>(packed), w, K, N, M, out, ldo, nonfinite, tiles_m, tiles_n,
                       (int)vec, epi);
    return hipGetLastError();
}

} // namespace

int gemm_kranges(int M, int K, int N, int num_cus) {
    if (num_cus <= 0) num_cus = 256;
    const int64_t mt = (M + 63) / 64;
    auto tiles = [&](int bn) { return mt * ((N + bn - 1) / bn); };
    int kg = 1;
    if (4 * tiles(192) < 5 * (int64_t)num_cus) kg = tiles(48) <= num_cus ? 8 : tiles(96) <= num_cus ? 4 : 2;
    while (kg > 1 && kg * 384 > K) kg /= 2;
    return kg;
}

double tile_gemm_us(int M, int K, int N, int num_cus) {
    return std::min({tile_us<T1s>(M, K, N, num_cus), tile_us<T1>(M, K, N, num_cus), tile_us<T1b>(M, K, N, num_cus)});
}

template <int EPI>
static hipError_t tile_gemm_t(const void *packed, const uint8_t *w, int K, int N, int M, float *out, int64_t ldo,
                              int32_t *nonfinite, int num_cus, int kranges, const GemmEpi &epi, hipStream_t s) {
    const int cus = num_cus > 0 ? num_cus : 256;
#define B1_TILE(C) launch_tile<C, EPI>(packed, w, K, N, M, out, ldo, nonfinite, epi, s)
#define B1_LESS(A, B) (tile_us<A>(M, K, N, cus) < tile_us<B>(M, K, N, cus))
    // (the packed output takes tiles of whole 64-column blocks)
    if constexpr (EPI == 3) {
        switch (kranges) {
        case 8: return B1_LESS(T8sp, T8p) ? B1_TILE(T8sp) : B1_TILE(T8p);
        case 4: return B1_TILE(T4p);
        case 2: return B1_LESS(T2sp, T2) ? B1_TILE(T2sp) : B1_TILE(T2);
        default: break;
        }
    } else {
        switch (kranges) {
        case 8: return B1_LESS(T8s, T8) ? B1_TILE(T8s) : B1_TILE(T8);
        case 4: return B1_LESS(T4s, T4) ? B1_TILE(T4s) : B1_TILE(T4);
        case 2: return B1_LESS(T2s, T2) ? B1_TILE(T2s) : B1_TILE(T2);
        default: break;
        }
    }
    if (B1_LESS(T1s, T1) && B1_LESS(T1s, T1b)) return B1_TILE(T1s);
    return B1_LESS(T1, T1b) ? B1_TILE(T1) : B1_TILE(T1b);
#undef B1_TILE
#undef B1_LESS
}

hipError_t launch_tile_gemm(const void *packed, const uint8_t *w, int K, int N, int M, float *out, int64_t ldo,
                            int32_t *nonfinite, int num_cus, int kranges, int kind, const GemmEpi &epi,
                            hipStream_t s) {
    switch (kind) {
    case 0: return tile_gemm_t<0>(packed, w, K, N, M, out, ldo, nonfinite, num_cus, kranges, epi, s);
    case 1: return tile_gemm_t<1>(packed, w, K, N, M, out, ldo, nonfinite, num_cus, kranges, epi, s);
    case 2: return tile_gemm_t<2>(packed, w, K, N, M, out, ldo, nonfinite, num_cus, kranges, epi, s);
    case 3: return tile_gemm_t<3>(packed, w, K, N, M, out, ldo, nonfinite, num_cus, kranges, epi, s);
    default: return hipErrorInvalidValue;
    }
}

} // namespace b1
