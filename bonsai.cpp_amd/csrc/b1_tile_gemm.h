// ------------------------------------------------------------ tile gemm --
//
// The packed GEMM for shapes whose 128 x 512 (or x 384) tiles would leave
// CUs idle: smaller tiles, and the work-group's waves split along K as well
// as along N.  A work-group computes a BM x BN tile; its waves form KG
// groups, group k taking the k-th contiguous range of K, NWN waves of WN
// columns in a group.  Each group runs BM x BN over its own range with its
// own stages, and the KG partial tiles meet in LDS, added in range order, so
// a tile is written once, with any epilogue, and no partial product goes to
// memory.  BM and BN need not divide M and N: rows and columns past the
// matrix read its last ones and are not stored.
//
// What bounds it: at M=512 K=9216 N=3072 (64 x 96 tiles, 4 ranges, 256
// work-groups) the loads alone take 34 us, the work on them alone 31, both
// 41: a CU's LDS-DMA moves ~40 bytes a cycle of activations, and a weight
// column's 12 bytes cost ~2 cycles, however few they are.  Hence many
// columns per activation row in the wide tiles and several ranges in the
// small ones, where eight waves would otherwise have nothing to share.
// Two stages read ahead into registers measured no faster, nor did weights
// loaded 48 bytes a column at a time (fewer accesses, more LDS).
//
// Against 128 x 512 tiles with K split over work-groups and summed by a
// second launch (both sides GPU time, us, pack excluded): M=77 K=3072
// N=3072 33 -> 7.3, M=256 25 -> 11.3; against the same tiles unsplit, what
// the epilogues ran: M=512 K=3072 N=3072 58 -> 17.4, M=512 K=9216 N=3072
// 157 -> 42, M=1024 K=9216 N=3072 158 -> 64, and with one range M=1024
// K=3072 N=18432 131 -> 106.
//
// MFMA 16x16x32, operands, K order and LDS staging as in b1_gemm16_kernel:
// weights are the A operand (16 columns), tokens the B operand, lane (li, g)
// holding 16-byte chunk g of a 32-element block.  With KG = 1 the outputs
// are those of the other packed kernels bit for bit.  A stage is KS of K:
// rows of 2 KS bytes whose 16-byte chunks sit at c ^ row (256-byte rows) or
// c ^ row / 2 (128-byte rows), so that 16 lanes of a fragment read (rows li,
// one chunk) cover all 64 banks; weights 12 bytes per column and 64 K at a
// 16-byte stride, loaded and read by the same wave.
template <int BM_, int WN_, int NWN_, int KG_, int KS_, int R_>
struct TileCfg {
    static constexpr int BM = BM_, WN = WN_, NWN = NWN_, KG = KG_, KS = KS_, R = R_;
    static constexpr int NW = NWN * KG, NT = NW * 64, BN = WN * NWN;
    static constexpr int MT = BM / 16, NTL = WN / 16;
    static constexpr int ROWB = KS * 2, CPR = ROWB / 16, RPI = 64 / CPR;
    static constexpr int AGRP = BM * ROWB;             // activation bytes of one K range's stage
    static constexpr int AW = AGRP / 1024 / NWN;       // 1 KB activation loads per wave
    static constexpr int BP = KS / 64;                 // 12-byte weight pairs (2 blocks) per column and stage
    static constexpr int CG = (WN + 63) / 64;          // 64-column weight load groups per wave
    static constexpr int BWAVE = BP * WN * 16;         // weight bytes per wave and stage
    static constexpr int ASZ = KG * AGRP, SLOT = ASZ + NW * BWAVE;
    static constexpr int LOADS = AW + BP * CG;         // loads per wave and stage
    static constexpr int RST = BN + 4;                 // floats per partial row in LDS
    static constexpr int fit_rows() {
        int r = BM;
        while (r > 16 && KG * r * RST * 4 > R * SLOT) r /= 2;
        return r;
    }
    static constexpr int RCH = fit_rows(); // rows per epilogue pass
    static constexpr int RED = KG * RCH * RST * 4;
    static constexpr int LDS = R * SLOT > RED ? R * SLOT : RED;
    static_assert(BM % 16 == 0 && WN % 16 == 0 && (KS == 64 || KS == 128), "tile shape");
    static_assert(AGRP % (1024 * NWN) == 0, "activation loads split evenly over a range's waves");
    static_assert(LDS <= 160 * 1024, "gfx950 LDS");
    static_assert(BM % RCH == 0 && RCH % 16 == 0, "epilogue passes");
    static_assert((R - 2) * LOADS < 64, "vmcnt holds 6 bits");
};

// Waits until at most `later` stages' loads are outstanding (later <= MAXL).
template <int LOADS, int MAXL>
__device__ __forceinline__ void wait_stages(int later) {
    if constexpr (MAXL == 0) {
        wait_vmcnt<0>();
    } else {
        if (later >= MAXL)
            wait_vmcnt<LOADS * MAXL>();
        else
            wait_stages<LOADS, MAXL - 1>(later);
    }
}

template <class C, int EPI>
__global__ __launch_bounds__(C::NT, 2) void b1_tile_gemm_kernel(const uint16_t *__restrict__ ah,
                                                                  const uint8_t *__restrict__ w, int K, int N, int M,
                                                                  float *out, int64_t ldo, int32_t *nonfinite,
                                                                  int tiles_m, int tiles_n, int vec_store,
                                                                  GemmEpi epi) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, g = lane >> 4;
    const int grp = wave / C::NWN, wn = wave - grp * C::NWN;
    const uint32_t rs = (uint32_t)(K / 32) * 6;

    // tile of this work-group: contiguous runs per XCD, groups of 8 tile
    // rows, rows fastest
    const int t = xcd_tile(blockIdx.x, tiles_m * tiles_n);
    constexpr int GM = 8;
    const int tg = t / (GM * tiles_n), first_m = tg * GM;
    const int gsize = min(GM, tiles_m - first_m);
    const int tin = t - first_m * tiles_n;
    const int m0 = (first_m + tin % gsize) * C::BM, n0 = (tin / gsize) * C::BN;

    // the K range of this wave's group, in stages of KS
    const int units = K / C::KS;
    const int u0 = grp * units / C::KG, n = (grp + 1) * units / C::KG - u0;
    const int nmax = (units + C::KG - 1) / C::KG;

    auto swz = [](int row) { return C::CPR == 16 ? (row & 15) : ((row >> 1) & 7); };
    uint32_t aoff[C::AW], boff[C::CG];
#pragma unroll
    for (int i = 0; i < C::AW; ++i) {
        const int row = C::RPI * (wn * C::AW + i) + lane / C::CPR;
        const int c = (lane % C::CPR) ^ swz(row);
        aoff[i] = ((uint32_t)min(m0 + row, M - 1) * (uint32_t)K + (uint32_t)c * 8) * 2;
    }
    // the weight row of a tile column
    auto weight_row = [&](int tc) {
        int row = min(n0 + tc, N - 1);
        if constexpr (EPI == 2) {
            // the tile's left half gates, its right half their values
            const int j = min((n0 >> 1) + (tc < C::BN / 2 ? tc : tc - C::BN / 2), epi.glu_h - 1);
            row = (tc < C::BN / 2 ? 0 : epi.glu_h) + j;
        }
        if constexpr (EPI == 3) {
            if (epi.act == 2 && row >= epi.split) {
                const int b = (row - epi.split) >> 6, within = (row - epi.split) & 63;
                row = epi.split + (within < 32 ? 32 * b + within : epi.glu_h + 32 * b + (within - 32));
            }
        }
        return row;
    };
#pragma unroll
    for (int cg = 0; cg < C::CG; ++cg)
        boff[cg] = (uint32_t)weight_row(wn * C::WN + min(cg * 64 + lane, C::WN - 1)) * rs;
    const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(ah), (short)0, (int)((uint32_t)M * (uint32_t)K * 2u), kBufferFlags);
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(w), (short)0, (int)((uint32_t)N * rs), kBufferFlags);
    auto issue = [&](int s, int slot) {
        uint8_t *sa = smem + slot + grp * C::AGRP + wn * C::AW * 1024;
        uint8_t *sw = smem + slot + C::ASZ + wave * C::BWAVE;
        const uint32_t aso = (uint32_t)(u0 + s) * C::ROWB, wso = (uint32_t)(u0 + s) * (C::BP * 12);
#pragma unroll
        for (int i = 0; i < C::AW; ++i) dma_buf_lds16s(ars, sa + i * 1024, aoff[i], aso);
#pragma unroll
        for (int cg = 0; cg < C::CG; ++cg) {
            if (cg * 64 + lane < C::WN) {
#pragma unroll
                for (int bp = 0; bp < C::BP; ++bp)
                    dma_buf_lds12s(wrs, sw + (bp * C::WN + cg * 64) * 16, boff[cg], wso + 12 * bp);
            }
        }
    };

    typedef __attribute__((address_space(3))) uint8_t lds_u8;
    typedef const __attribute__((address_space(3))) uint32_t lds_u32;
    typedef __attribute__((address_space(3))) half8 lds_half8;
    typedef __attribute__((address_space(3))) floatx4 lds_f4;
    lds_u8 *const lbase = (lds_u8 *)smem;
    lds_u8 *fa[C::KS / 32];
#pragma unroll
    for (int j = 0; j < C::KS / 32; ++j)
        fa[j] = lbase + grp * C::AGRP + li * C::ROWB + (((4 * j + g) ^ swz(li)) * 16);
    lds_u8 *const qw = lbase + C::ASZ + wave * C::BWAVE + li * 16;

    floatx4 acc[C::MT][C::NTL];
#pragma unroll
    for (int i = 0; i < C::MT; ++i)
#pragma unroll
        for (int j = 0; j < C::NTL; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    auto compute = [&](int slot) {
        // the stage's packed weight words and activation fragments
        uint32_t d[C::BP][C::NTL][3];
        half8 af[C::KS / 32][C::MT];
#pragma unroll
        for (int bp = 0; bp < C::BP; ++bp)
#pragma unroll
            for (int nt = 0; nt < C::NTL; ++nt) {
                lds_u32 *q = (lds_u32 *)(qw + slot + (bp * C::WN + nt * 16) * 16);
                d[bp][nt][0] = q[0];
                d[bp][nt][1] = q[1];
                d[bp][nt][2] = q[2];
            }
#pragma unroll
        for (int b = 0; b < C::KS / 32; ++b)
#pragma unroll
            for (int mt = 0; mt < C::MT; ++mt) af[b][mt] = *(const lds_half8 *)(fa[b] + slot + mt * 16 * C::ROWB);
#pragma unroll
        for (int b = 0; b < C::KS / 32; ++b) {
#pragma unroll
            for (int nt = 0; nt < C::NTL; ++nt) {
                const uint32_t *dd = d[b >> 1][nt];
                uint32_t s2, wg;
                if ((b & 1) == 0) {
                    s2 = dup_lo16(dd[0]);
                    wg = __builtin_amdgcn_alignbit(dd[1], dd[0], 16 + 4 * g);
                } else {
                    s2 = dup_hi16(dd[1]);
                    wg = dd[2] >> (4 * g);
                }
                u32x4 bo;
#pragma unroll
                for (int q = 0; q < 4; ++q) bo[q] = wpair(wg, 15 - q, s2);
#pragma unroll
                for (int mt = 0; mt < C::MT; ++mt)
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, bo), af[b][mt],
                                                                         acc[mt][nt], 0, 0, 0);
            }
        }
    };
    // Every wave's part of the stage is in LDS and its reads of the previous
    // stage are done; a group of one wave shares its stages with no other.
    auto publish = [&]() {
        wait_lgkmcnt0();
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (C::NWN > 1) lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto next = [&](int slot) { return slot + C::SLOT == C::R * C::SLOT ? 0 : slot + C::SLOT; };

#pragma unroll
    for (int s = 0; s < C::R - 1; ++s)
        if (s < n) issue(s, s * C::SLOT);
    int slot = 0, fill = (C::R - 1) * C::SLOT, s = 0;
    for (; s + C::R - 1 < n; ++s) {
        wait_vmcnt<(C::R - 2) * C::LOADS>();
        publish();
        issue(s + C::R - 1, fill);
        compute(slot);
        fill = slot;
        slot = next(slot);
    }
    for (; s < n; ++s) {
        wait_stages<C::LOADS, C::R - 2>(n - 1 - s);
        publish();
        compute(slot);
        slot = next(slot);
    }
    for (; s < nmax; ++s) publish();

    // ---- epilogue: the ranges' partial tiles through LDS, summed in range
    // order, RCH rows at a time
    int bad = 0;
    const bool cnt = nonfinite != nullptr;
#pragma unroll
    for (int ch = 0; ch < C::BM / C::RCH; ++ch) {
        wait_vmcnt<0>();
        wait_lgkmcnt0();
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
#pragma unroll
        for (int mr = 0; mr < C::RCH / 16; ++mr)
#pragma unroll
            for (int nt = 0; nt < C::NTL; ++nt)
                *(lds_f4 *)(lbase + ((grp * C::RCH + mr * 16 + li) * C::RST + wn * C::WN + nt * 16 + 4 * g) * 4) =
                    acc[ch * (C::RCH / 16) + mr][nt];
        wait_lgkmcnt0();
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
        const int mb = m0 + ch * C::RCH;
        // y of tile row r (of this pass), columns c .. c + 3
        auto y4 = [&](int r, int c, float sc) {
            const lds_u8 *p = lbase + (r * C::RST + c) * 4;
            floatx4 v = *(const lds_f4 *)p;
#pragma unroll
            for (int k = 1; k < C::KG; ++k) {
                const floatx4 x = *(const lds_f4 *)(p + k * C::RCH * C::RST * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] += x[e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] *= sc;
            return v;
        };
        auto count4 = [&](const floatx4 &v) {
#pragma unroll
            for (int e = 0; e < 4; ++e) bad += !__builtin_isfinite(v[e]);
        };
        if constexpr (EPI == 0 || EPI == 1) {
            constexpr int Q = C::BN / 4;
            for (int u = tid; u < C::RCH * Q; u += C::NT) {
                const int r = u / Q, c = (u - r * Q) * 4;
                const int m = mb + r, col = n0 + c;
                if (m >= M || col >= N) continue;
                floatx4 v = y4(r, c, epi.rsc ? epi.rsc[m] : 1.0f);
                float *o = out + (size_t)m * ldo + col;
                if (vec_store && col + 4 <= N) {
                    if (cnt) count4(v);
                    if constexpr (EPI == 1) {
                        const floatx4 gq = *reinterpret_cast<const floatx4 *>(epi.gate + col);
                        const floatx4 rq = *reinterpret_cast<const floatx4 *>(epi.res + (size_t)m * epi.ldr + col);
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = gate_residual(rq[e], gq[e], v[e]);
                    }
                    *reinterpret_cast<floatx4 *>(o) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (col + e < N) {
                            float y = v[e];
                            bad += cnt && !__builtin_isfinite(y);
                            if constexpr (EPI == 1)
                                y = gate_residual(epi.res[(size_t)m * epi.ldr + col + e], epi.gate[col + e], y);
                            o[e] = y;
                        }
                }
            }
        } else if constexpr (EPI == 2) {
            constexpr int Q = C::BN / 8;
            for (int u = tid; u < C::RCH * Q; u += C::NT) {
                const int r = u / Q, c = (u - r * Q) * 4;
                const int m = mb + r, j = (n0 >> 1) + c;
                if (m >= M || j >= epi.glu_h) continue;
                const float sc = epi.rsc ? epi.rsc[m] : 1.0f;
                const floatx4 gt = y4(r, c, sc), vl = y4(r, C::BN / 2 + c, sc);
                if (cnt) {
                    count4(gt);
                    count4(vl);
                }
                floatx4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = mul_f32(silu_f32(gt[e]), vl[e]);
                float *o = out + (size_t)m * ldo + j;
                if (vec_store) {
                    *reinterpret_cast<floatx4 *>(o) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = v[e];
                }
            }
        } else {
            // (row, 32-column block, quad of 4 dwords)
            constexpr int Q = C::BN / 8;
            for (int u = tid; u < C::RCH * Q; u += C::NT) {
                const int r = u / Q, q = u - r * Q, jb = q >> 2, dq = (q & 3) * 4;
                const int m = mb + r, cb = n0 + 32 * jb;
                if (m >= M || cb >= N) continue;
                const float sc = epi.rsc ? epi.rsc[m] : 1.0f;
                const bool pcol = cb >= epi.split;
                if (pcol && epi.act == 2 && ((cb - epi.split) & 32)) continue; // the pair's value block
                floatx4 lo = y4(r, 32 * jb + dq, sc), hi = y4(r, 32 * jb + dq + 16, sc);
                if (cnt) {
                    count4(lo);
                    count4(hi);
                }
                if (!pcol) {
                    float *o = out + (size_t)m * ldo + cb + dq;
                    *reinterpret_cast<floatx4 *>(o) = lo;
                    *reinterpret_cast<floatx4 *>(o + 16) = hi;
                    continue;
                }
                int blk = (cb - epi.split) >> 5;
                if (epi.act == 2) {
                    blk >>= 1;
                    const floatx4 vlo = y4(r, 32 * jb + 32 + dq, sc), vhi = y4(r, 32 * jb + 48 + dq, sc);
                    if (cnt) {
                        count4(vlo);
                        count4(vhi);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        lo[e] = mul_f32(silu_f32(lo[e]), vlo[e]);
                        hi[e] = mul_f32(silu_f32(hi[e]), vhi[e]);
                    }
                } else if (epi.act == 1) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        lo[e] = gelu_tanh(lo[e]);
                        hi[e] = gelu_tanh(hi[e]);
                    }
                }
                u32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = pack_f16_rounded(lo[e], hi[e]);
                *reinterpret_cast<u32x4 *>(epi.pk + (size_t)m * epi.ldpw + blk * 16 + dq) = v;
            }
        }
    }
    count_nonfinite(nonfinite, bad);
}
