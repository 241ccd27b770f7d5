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
// ranges, KS per stage, R stages in the ring, L pairs of a column a load, and whether the packed-output
// epilogue can use them (whole 32-column blocks; 64 for SwiGLU pairs).
//                 BM  WN NWN KG  KS  R  L
using T8s = TileCfg<32, 48, 1, 8, 64, 2, 4>;
using T8 = TileCfg<64, 48, 1, 8, 64, 2, 1>;
using T8sp = TileCfg<32, 64, 1, 8, 64, 3, 2>;
using T8p = TileCfg<64, 64, 1, 8, 64, 2, 1>;
using T4s = TileCfg<32, 48, 2, 4, 64, 4, 4>;
using T4 = TileCfg<64, 48, 2, 4, 64, 2, 4>;
using T4p = TileCfg<64, 64, 2, 4, 64, 3, 2>;
using T2s = TileCfg<64, 48, 2, 2, 64, 2, 2>;
using T2sp = TileCfg<64, 64, 2, 2, 64, 2, 2>;
using T2 = TileCfg<64, 48, 4, 2, 64, 4, 4>;
using T1s = TileCfg<32, 48, 4, 1, 64, 4, 4>;
using T1 = TileCfg<64, 48, 4, 1, 64, 2, 4>;
using T1b = TileCfg<128, 48, 4, 1, 64, 2, 4>;

// Time model of a launch, in microseconds, from launches of every tile over
// 32 to 2048 tokens, K 1536 to 9216, N 3072 to 18432 on 256 CUs (most within
// 10 %; up to 4608 tokens the 128-row tile takes up to 13 % more than modelled,
// M=4592 N=12288 307 us for 285, 23 % at K = 768): a CU runs q tiles (rounded
// up), `occ` at a time; each adds e + c b to a busy CU, b = K / 32 / KG blocks
// per range, and what is left at the end takes e1 + c1 b at least, a tile's
// time alone.
struct TileCost {
    int occ;
    double e, c, e1, c1;
};
template <class C>
constexpr TileCost tile_cost() {
    constexpr double wide = C::WN / 48.0; // 64-column waves, by their columns
    if (C::KG == 8) return C::BM == 32 ? TileCost{1, 1.2, 0.34 * wide, 2.0, 0.34 * wide} : TileCost{1, 2.5, 0.50 * wide, 2.5, 0.50 * wide};
    if (C::KG == 4) return C::BM == 32 ? TileCost{1, 2.9, 0.25 * wide, 2.9, 0.25 * wide} : TileCost{1, 2.5, 0.41 * wide, 2.5, 0.41 * wide};
    if (C::KG == 2)
        return C::NWN == 4 ? TileCost{1, 4.0, 0.375, 4.0, 0.375}
                           : TileCost{C::WN == 48 ? 3 : 2, 1.0, 0.195 * wide, 0.9, 0.31 * wide};
    if (C::BM == 32) return TileCost{3, 0.9, 0.115, 1.1, 0.207};
    return C::BM == 64 ? TileCost{3, 0.9, 0.18, 3.4, 0.25} : TileCost{2, 1.0, 0.305, 4.7, 0.365};
}
// `more`: us a tile's epilogue takes beyond a plain one's.
template <class C>
double tile_us(int M, int K, int N, int num_cus, double more = 0.0) {
    TileCost t = tile_cost<C>();
    t.e += more, t.e1 += more;
    const int64_t tiles = (int64_t)((M + C::BM - 1) / C::BM) * ((N + C::BN - 1) / C::BN);
    const int64_t q = (tiles + num_cus - 1) / num_cus, rest = q % t.occ;
    const double b = (double)(K / 32) / C::KG, add = t.e + t.c * b, alone = t.e1 + t.c1 * b;
    return 3.3 + (double)(q - rest) * add + (rest ? std::max(alone, (double)rest * add) : 0.0);
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

double tile_gemm_us(int M, int K, int N, int num_cus, int kranges) {
    const int cus = num_cus > 0 ? num_cus : 256;
    auto us = [&](auto a, auto b) { return std::min(tile_us<decltype(a)>(M, K, N, cus), tile_us<decltype(b)>(M, K, N, cus)); };
    switch (kranges) {
    case 8: return us(T8s{}, T8{});
    case 4: return us(T4s{}, T4{});
    case 2: return us(T2s{}, T2{});
    default: return std::min(us(T1s{}, T1{}), tile_us<T1b>(M, K, N, cus));
    }
}

// The fewest microseconds by the models of the tiles and, for one range, of
// the persistent kernels; a range has at least 384 of K.  One range from 1.25
// tiles of 64 x 192 a CU on: there a row's bits do not depend on how many rows
// come with it, and a second range saves little (M=1500 K=3072 N=3072: 39 and
// 37 us; below, M=300 N=9216: 32 and 25).
int gemm_kranges(int M, int K, int N, int num_cus) {
    int best = 1;
    double best_us = std::min(tile_gemm_us(M, K, N, num_cus, 1), persistent_gemm_us(M, K, N, num_cus));
    const int64_t tiles = (int64_t)((M + 63) / 64) * ((N + 191) / 192);
    if (4 * tiles >= 5 * (int64_t)(num_cus > 0 ? num_cus : 256)) return 1;
    for (int kg = 2; kg <= 8 && kg * 384 <= K; kg *= 2) {
        const double us = tile_gemm_us(M, K, N, num_cus, kg);
        if (us < best_us) {
            best_us = us;
            best = kg;
        }
    }
    return best;
}

// run(tile) with the tile a GEMM of `kranges` K ranges takes (PACKED: with the
// packed-output epilogue, which needs whole 64-column blocks).
template <bool PACKED, class Run>
static auto with_tile(int M, int K, int N, int num_cus, int kranges, Run run) {
    const int cus = num_cus > 0 ? num_cus : 256;
#define B1_LESS(A, B) (tile_us<A>(M, K, N, cus) < tile_us<B>(M, K, N, cus))
    if constexpr (PACKED) {
        switch (kranges) {
        case 8: return B1_LESS(T8sp, T8p) ? run(T8sp{}) : run(T8p{});
        case 4: return run(T4p{});
        case 2: return B1_LESS(T2sp, T2) ? run(T2sp{}) : run(T2{});
        default: break;
        }
    } else {
        switch (kranges) {
        case 8: return B1_LESS(T8s, T8) ? run(T8s{}) : run(T8{});
        case 4: return B1_LESS(T4s, T4) ? run(T4s{}) : run(T4{});
        case 2: return B1_LESS(T2s, T2) ? run(T2s{}) : run(T2{});
        default: break;
        }
    }
    if (B1_LESS(T1s, T1) && B1_LESS(T1s, T1b)) return run(T1s{});
    return B1_LESS(T1, T1b) ? run(T1{}) : run(T1b{});
#undef B1_LESS
}

// A packed output's epilogue (fp16 pairs, GELU) counts 1 us more than a plain
// one's in a 64-row tile and 2 in a 128-row one, with SwiGLU 1.5 and 5, from
// 713 launches of each over 300 to 4608 tokens: fewer work-groups a CU leave
// more of it bare (M=1024 K=3072 N=18432, six 64-row or three 128-row tiles a
// CU: plain 114 and 111 us, packed SwiGLU 118 and 119).
double packed_tile_us(int M, int K, int N, int num_cus, bool swiglu) {
    const int cus = num_cus > 0 ? num_cus : 256;
    return with_tile<true>(M, K, N, cus, 1, [&](auto tile) {
        using C = decltype(tile);
        return tile_us<C>(M, K, N, cus, C::BM == 128 ? (swiglu ? 5.0 : 2.0) : swiglu ? 1.5 : 1.0);
    });
}

TileShape tile_shape(int M, int K, int N, int num_cus, int kranges, bool packed_out) {
    auto shape = [](auto tile) {
        using C = decltype(tile);
        return TileShape{C::KG, C::BM, C::BN};
    };
    return packed_out ? with_tile<true>(M, K, N, num_cus, kranges, shape)
                      : with_tile<false>(M, K, N, num_cus, kranges, shape);
}

template <int EPI>
static hipError_t tile_gemm_t(const void *packed, const uint8_t *w, int K, int N, int M, float *out, int64_t ldo,
                              int32_t *nonfinite, int num_cus, int kranges, const GemmEpi &epi, hipStream_t s) {
    return with_tile<EPI == 3>(M, K, N, num_cus, kranges, [&](auto tile) {
        return launch_tile<decltype(tile), EPI>(packed, w, K, N, M, out, ldo, nonfinite, epi, s);
    });
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
