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
// What bounds it: matrix and vector work of a SIMD's waves overlap little (12
// MFMAs of one wave and 48 shifts of another, 98 and 105 ns alone, take 148
// together), and a block's weights cost ~30 vector operations a wave whatever
// its rows; beside that the loads.  A CU's LDS-DMA moves ~40 bytes a cycle of
// activations, and a weight load costs a request a column and line, since a
// row's next 12 bytes have left L1 by the next stage.  So a wave loads L
// consecutive 64-K pairs of a column with L adjacent lanes, WN / L columns a
// load, a slice of the group a pair ahead of its use: a quarter (L = 4) of
// the requests with as many loads.  us with L = 1 -> now: M=512 K=9216 N=3072
// 42.4 -> 38, M=1024 N=3072 68.5 -> 62, M=1024 K=3072 N=18432 124 -> 113
// (all columns in one line, the limit: 33, 54 and 99).  Shallower rings that
// let three work-groups of 64 x 192 on a CU: M=512 K=3072 N=18432 69 -> 62.
// A block's fragments are read from LDS while the one before is multiplied.
//
// Against 128 x 512 tiles with K split over work-groups and summed by a
// second launch (both sides GPU time, us, pack excluded): M=77 K=3072
// N=3072 33 -> 7.3, M=256 25 -> 11.3; against the same tiles unsplit, what
// the epilogues ran: M=512 K=3072 N=3072 58 -> 17, M=512 K=9216 N=3072
// 157 -> 37, M=1024 K=9216 N=3072 158 -> 63, and with one range M=1024
// K=3072 N=18432 131 -> 107 (plain).
//
// MFMA 16x16x32, operands, K order and LDS staging as in b1_gemm16_kernel:
// weights are the A operand (16 columns), tokens the B operand, lane (li, g)
// holding 16-byte chunk g of a 32-element block.  With KG = 1 the outputs
// are those of the other packed kernels bit for bit.  A stage is KS of K:
// rows of 2 KS bytes whose 16-byte chunks sit at c ^ row (256-byte rows) or
// c ^ row / 2 (128-byte rows), so that 16 lanes of a fragment read (rows li,
// one chunk) cover all 64 banks; weights 12 bytes per column and 64 K at a
// 16-byte stride, a group of L pairs of every column together, loaded and
// read by the same wave.
template <int BM_, int WN_, int NWN_, int KG_, int KS_, int R_, int L_>
struct TileCfg {
    static constexpr int BM = BM_, WN = WN_, NWN = NWN_, KG = KG_, KS = KS_, R = R_, L = L_;
    static constexpr int NW = NWN * KG, NT = NW * 64, BN = WN * NWN;
    static constexpr int MT = BM / 16, NTL = WN / 16;
    static constexpr int ROWB = KS * 2, CPR = ROWB / 16, RPI = 64 / CPR;
    static constexpr int AGRP = BM * ROWB;             // activation bytes of one K range's stage
    static constexpr int AW = AGRP / 1024 / NWN;       // 1 KB activation loads per wave
    static constexpr int ASZ = KG * AGRP;              // activation bytes of a stage
    static constexpr int BP = KS / 64;                 // 12-byte weight pairs (2 blocks) per column and stage
    static constexpr int WSL = WN * 16;                // a slice: WN / L columns x L pairs
    static constexpr int WGRP = L * WSL;               // a wave's weight group, L pairs of every column
    // groups kept: stage s + R's loads fill slices of group (s + R) BP / L + 1
    // while stage s + 1 of this and every later group is still to be read
    static constexpr int groups() {
        int g = 0;
        for (int s = 0; s < 4 * L; ++s) {
            const int d = ((s + R) * BP + BP - 1) / L + 1 - (s + 1) * BP / L;
            if (d > g) g = d;
        }
        return g + 1;
    }
    static constexpr int RW = groups();
    static constexpr int WBASE = R * ASZ;              // the weight groups follow the stages
    static constexpr int STAGED = WBASE + NW * RW * WGRP;
    static constexpr int LOADS = AW + BP;              // loads per wave and stage
    static constexpr int RST = BN + 4;                 // floats per partial row in LDS
    static constexpr int fit_rows() {
        int r = BM;
        while (r > 16 && KG * r * RST * 4 > STAGED) r /= 2;
        return r;
    }
    static constexpr int RCH = fit_rows(); // rows per epilogue pass
    static constexpr int RED = KG * RCH * RST * 4;
    static constexpr int LDS = STAGED > RED ? STAGED : RED;
    static_assert(BM % 16 == 0 && WN % 16 == 0 && (KS == 64 || KS == 128), "tile shape");
    static_assert(WN <= 64 && (L == 1 || L == 2 || L == 4) && WN % L == 0 && L % BP == 0, "weight slices");
    static_assert(AGRP % (1024 * NWN) == 0, "activation loads split evenly over a range's waves");
    static_assert(LDS <= 160 * 1024, "gfx950 LDS");
    static_assert(BM % RCH == 0 && RCH % 16 == 0, "epilogue passes");
    static_assert((R - 1) * LOADS < 64, "vmcnt holds 6 bits");
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
    uint32_t aoff[C::AW], boff[C::L];
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
    // Slice i of a weight group: columns i WN / L .. + WN / L - 1, lane
    // (column, pair), the pairs of column c in the order pair ^ swl(c) so that
    // the 16 columns of a fragment read lie in distinct banks.
    auto swl = [](int c) { return C::L == 4 ? (c >> 2) & 3 : C::L == 2 ? (c >> 3) & 1 : 0; };
#pragma unroll
    for (int i = 0; i < C::L; ++i) {
        const int c = min(i * (C::WN / C::L) + lane / C::L, C::WN - 1);
        boff[i] = (uint32_t)weight_row(wn * C::WN + c) * rs + 12u * (uint32_t)((lane % C::L) ^ swl(c));
    }
    const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(ah), (short)0, (int)((uint32_t)M * (uint32_t)K * 2u), kBufferFlags);
    const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(w), (short)0, (int)((uint32_t)N * rs), kBufferFlags);
    // Pair q of the range goes with slice q % L of the next weight group (one
    // load a pair; group 0 is loaded before the first stage; past the last
    // group, that one again).  A group's pairs past the range are loaded too
    // (past the buffer: zeros) and never used.
    const int last_group = (n * C::BP - 1) / C::L;
    uint8_t *const sw0 = smem + C::WBASE + wave * (C::RW * C::WGRP);
    int wfill = C::WGRP;
    auto load_slice = [&](int at, int group) {
        if (lane < C::WN)
            dma_buf_lds12s(wrs, sw0 + at, boff[0], (uint32_t)((u0 * C::BP + min(group, last_group) * C::L) * 12));
        const uint32_t b0 = boff[0];
#pragma unroll
        for (int i = 0; i + 1 < C::L; ++i) boff[i] = boff[i + 1];
        boff[C::L - 1] = b0;
    };
    auto issue = [&](int s, int slot) {
        uint8_t *sa = smem + slot + grp * C::AGRP + wn * C::AW * 1024;
        const uint32_t aso = (uint32_t)(u0 + s) * C::ROWB;
#pragma unroll
        for (int i = 0; i < C::AW; ++i) dma_buf_lds16s(ars, sa + i * 1024, aoff[i], aso);
#pragma unroll
        for (int bp = 0; bp < C::BP; ++bp) {
            load_slice(wfill, (s * C::BP + bp) / C::L + 1);
            wfill = wfill + C::WSL == C::RW * C::WGRP ? 0 : wfill + C::WSL;
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
    // the pair to read next: its group's place and its lane offset
    lds_u8 *const qw = lbase + C::WBASE + wave * (C::RW * C::WGRP) + li * (C::L * 16);
    const int qsw = swl(li) * 16;
    int rgrp = 0, rsub = 0;

    floatx4 acc[C::MT][C::NTL];
#pragma unroll
    for (int i = 0; i < C::MT; ++i)
#pragma unroll
        for (int j = 0; j < C::NTL; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // Blocks are software-pipelined: a block's fragments (one of two sets) and
    // a pair's packed weight words are read from LDS while the MFMAs of the
    // block before it run, across stages too.
    constexpr int J = C::KS / 32;
    static_assert(J % 2 == 0, "a stage starts with fragment set 0");
    uint32_t d[C::NTL][3], s2[C::NTL], wg[C::NTL];
    half8 af[2][C::MT];
    auto read = [&](int slot, int j) {
        if (j % 2 == 0) {
            lds_u8 *const qp = qw + rgrp + (rsub ^ qsw);
            rsub += 16;
            if (rsub == 16 * C::L) {
                rsub = 0;
                rgrp = rgrp + C::WGRP == C::RW * C::WGRP ? 0 : rgrp + C::WGRP;
            }
#pragma unroll
            for (int nt = 0; nt < C::NTL; ++nt) {
                lds_u32 *q = (lds_u32 *)(qp + nt * (C::L * 256));
                d[nt][0] = q[0];
                d[nt][1] = q[1];
                d[nt][2] = q[2];
            }
        }
#pragma unroll
        for (int mt = 0; mt < C::MT; ++mt) af[j & 1][mt] = *(const lds_half8 *)(fa[j] + slot + mt * 16 * C::ROWB);
    };
    // the scale pair and the sign word of block j, the lane's last pair at the
    // sign bits, from the pair's words
    auto scales = [&](int j) {
#pragma unroll
        for (int nt = 0; nt < C::NTL; ++nt) {
            if ((j & 1) == 0) {
                s2[nt] = dup_lo16(d[nt][0]);
                wg[nt] = __builtin_amdgcn_alignbit(d[nt][1], d[nt][0], 4 + 4 * g);
            } else {
                s2[nt] = dup_hi16(d[nt][1]);
                wg[nt] = d[nt][2] << (12 - 4 * g);
            }
        }
    };
    auto mma = [&](int set) {
#pragma unroll
        for (int nt = 0; nt < C::NTL; ++nt) {
            const u32x4 bo = wpair4(wg[nt], s2[nt]);
#pragma unroll
            for (int mt = 0; mt < C::MT; ++mt)
                acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, bo), af[set][mt],
                                                                     acc[mt][nt], 0, 0, 0);
        }
    };
    // Every wave's part of the next stage is in LDS (its loads waited for
    // before) and this one's reads are done, so that its slot can be filled;
    // a group of one wave shares its stages with no other.
    auto publish = [&]() {
        wait_lgkmcnt0();
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (C::NWN > 1) lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto next = [&](int slot) { return slot + C::ASZ == C::R * C::ASZ ? 0 : slot + C::ASZ; };
    // the stage in `slot`; `advance` makes the next one readable
    auto stage = [&](int slot, auto &&advance, bool more) {
#pragma unroll
        for (int j = 0; j < J; ++j) {
            scales(j);
            if (j + 1 < J) {
                read(slot, j + 1);
            } else if (more) {
                advance();
                read(next(slot), 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            mma(j & 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

#pragma unroll
    for (int i = 0; i < C::L; ++i) load_slice(i * C::WSL, 0);
#pragma unroll
    for (int s = 0; s < C::R; ++s)
        if (s < n) issue(s, s * C::ASZ);
    wait_stages<C::LOADS, C::R - 1>(n - 1);
    publish();
    read(0, 0);
    int slot = 0, s = 0;
    for (; s + C::R < n; ++s) {
        stage(slot, [&]() {
            wait_vmcnt<(C::R - 2) * C::LOADS>();
            publish();
            issue(s + C::R, slot);
        }, true);
        slot = next(slot);
    }
    for (; s + 1 < n; ++s) {
        stage(slot, [&]() {
            wait_stages<C::LOADS, C::R - 2>(n - 2 - s);
            publish();
        }, true);
        slot = next(slot);
    }
    stage(slot, []() {}, false);
    for (s = n; s < nmax; ++s) publish();

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
