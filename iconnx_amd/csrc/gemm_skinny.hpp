// MatMulInteger for products with too few output tiles to fill the chip (a batch of pooled
// rows, one short text): included by gemm.hip, whose operand handling (zero-point algebra,
// packed weights, chains, segmented outputs) it shares.
//
// What bounds such a product is the latency of one K walk, not bandwidth or the matrix
// cores: a 64x64-tile block on each of 12 CUs walks K = 768 in 12 dependent LDS stages, the
// persistent kernel's 6 blocks K = 3072 in 48.  Here a block owns a small tile, 16 TI x 16 TJ,
// and its W waves split K among them, so each wave has only a few 64-wide steps; fragments
// come straight from memory in the MFMA operand layout (no LDS stage, no barrier), with the
// loads of four steps in flight at once, and one LDS pass adds the waves' partial sums
// (integers: the same result in any order).
#pragma once

__device__ __forceinline__ v4i as_v4i(uint4 v) { return v4i{(int)v.x, (int)v.y, (int)v.z, (int)v.w}; }

// v_mfma_i32_16x16x64_i8: A lane l = row l % 16, bytes 16 (l / 16) .. +15 of the 64-wide step,
// B likewise by column; D register r of lane l = row 4 (l / 16) + r, column l % 16.
// AQ: A is the f32 input of the DynamicQuantizeLinear (g.xin, K % 64 == 0), whose producer
// left its range as g.n_xpart partials: every block folds them as the DQL launch does and
// quantizes the values it multiplies itself, the same bytes (dql_core.hpp), instead of a
// launch that writes them (4.6 us and a launch gap for one text) and another that reads them.
// The row sums of a' that a weight zero point multiplies are formed here (g.self_rowsum), as
// the product with a column of ones, when no DQL left them, and the column sums of b' likewise
// when the weight was packed for this call (g.colsum null): no launch for either.
template <int TI, int TJ, int W, bool VEC, int OUT, int CH, bool AQ = false>
__global__ void __launch_bounds__(64 * W) gemm_i8_skinny_kernel(GemmArgs g) {
    constexpr int BM = 16 * TI, BN = 16 * TJ, NT = 64 * W, TILES = TI * TJ;
    constexpr int U = AQ ? 3 : 4;  // K steps in flight per wave
    constexpr bool OPS = OUT == OUT_F32 && CH != CH_GENERAL;
    constexpr int MODE = CH == CH_COL_EXT ? 2 : 0;
    static_assert(W >= TILES && NT >= ICX_MAX_CHAIN * BN, "a wave per tile in the epilogue; a lane per operand");
    __shared__ v4i part[W][TILES][64];
    __shared__ v4i rpart[W][TI][64];
    __shared__ int cpart[W][TJ][64];
    __shared__ float sop[ICX_MAX_CHAIN][BN];

    // the row tiles of one column tile on one XCD (block i runs on XCD i % 8): they read the
    // same weight columns
    int tm, tn;
    if ((g.tiles_n & 7) == 0) {
        const int y = blockIdx.x >> 3;
        tn = (blockIdx.x & 7) + 8 * (y / g.tiles_m);
        tm = y % g.tiles_m;
    } else {
        tn = blockIdx.x / g.tiles_m;
        tm = blockIdx.x % g.tiles_m;
    }
    const int m0 = tm * BM, n0 = tn * BN;
    const int t = threadIdx.x, lane = t & 63;
    const int wid = __builtin_amdgcn_readfirstlane(t >> 6);
    const int lr = lane & 15, lk = (lane >> 4) * 16;
    const bool self = !AQ && g.self_rowsum, selfc = !AQ && g.colsum == nullptr;

    // the range partials first: they are folded while the first x and weight loads arrive
    constexpr int PN = (icx::kMaxRangeParts + NT - 1) / NT;
    float2 xp[AQ ? PN : 1];
    if constexpr (AQ) {
#pragma unroll
        for (int u = 0; u < PN; ++u) xp[u] = g.xpart[min(t + u * NT, g.n_xpart - 1)];
    }

    // epilogue operands: one chain operand per lane, and the column terms of the lane's column
    float f0 = 1.0f, f1 = 1.0f;
    const int ok = t / BN, oc = t % BN;
    if constexpr (OPS) {
        if (ok < g.chain.n_ops && icx::op_takes_operand(g.chain.ops[ok].op)) {
            const icx_chain_op& op = g.chain.ops[ok];
            const int c = min(n0 + oc, g.N - 1);
            f0 = op.p0[op.kind0 == ICX_BCAST_SCALAR ? 0 : c];
            if (op.p1) f1 = op.p1[op.kind1 == ICX_BCAST_SCALAR ? 0 : c];
        }
    }
    const int ti = wid / TJ, tj = wid % TJ;  // this wave's tile in the epilogue (wid < TILES)
    const int col = n0 + tj * 16 + lr, ccol = min(col, g.N - 1);
    const int row0 = m0 + ti * 16 + 4 * (lane >> 4);
    int azp = 0, bzp = 0;
    uint32_t csum = 0, rs[4] = {0, 0, 0, 0};
    if (wid < TILES) {
        azp = load_zp(g.a_zp, g.a_zp_u8, 0);
        bzp = load_zp(g.b_zp, g.b_zp_u8, g.b_zp_len == 1 ? 0 : ccol);
        if (!selfc) csum = (uint32_t)g.colsum[ccol];
        if (g.rowsum_raw) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                rs[r] = (uint32_t)g.rowsum_raw[min(row0 + r, g.M - 1)] - (uint32_t)g.alpha * (uint32_t)g.K;
        }
    }

    v4i acc[TI][TJ], racc[TI], cacc[TJ];
#pragma unroll
    for (int j = 0; j < TJ; ++j) cacc[j] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        racc[i] = v4i{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    }
    const int8_t* pa[TI];
    const float* px[TI];
    const int8_t* pb[TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i) {
        const size_t row = (size_t)min(m0 + 16 * i + lr, g.M - 1) * g.K;
        px[i] = g.xin + row;  // (AQ)
        pa[i] = g.A + row;
    }
#pragma unroll
    for (int j = 0; j < TJ; ++j) pb[j] = g.Bp + (size_t)min(n0 + 16 * j + lr, g.N - 1) * g.K;
    const v4i ones = v4i{0x01010101, 0x01010101, 0x01010101, 0x01010101};
    const int axr = (int)g.a_xor;
    auto step = [&](const v4i (&a)[TI], const v4i (&b)[TJ]) {
#pragma unroll
        for (int i = 0; i < TI; ++i) {
#pragma unroll
            for (int j = 0; j < TJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i], b[j], acc[i][j], 0, 0, 0);
            if (self) racc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i], ones, racc[i], 0, 0, 0);
        }
        if (selfc) {
#pragma unroll
            for (int j = 0; j < TJ; ++j) cacc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, b[j], cacc[j], 0, 0, 0);
        }
    };
    // wave `wid` walks steps [s0, e) of the whole ones, and the last wave with any takes the
    // partial one (K % 64 != 0)
    const int full = g.K / 64, steps = (g.K + 63) / 64;
    const int per = (steps + W - 1) / W;
    const int s0 = wid * per, e = min(s0 + per, full);
    icx::dql::DqlParams prm;
    if constexpr (AQ) {
        float4 xv[U][TI][4];
        uint4 rb[U][TJ];
        auto load = [&](int s) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = max(0, min(s + u, e - 1)) * 64 + lk;  // past the end: not used
#pragma unroll
                for (int i = 0; i < TI; ++i)
#pragma unroll
                    for (int c = 0; c < 4; ++c) xv[u][i][c] = *reinterpret_cast<const float4*>(px[i] + k + 4 * c);
#pragma unroll
                for (int j = 0; j < TJ; ++j) rb[u][j] = ld16<true>(pb[j] + k);
            }
        };
        load(s0);
        __builtin_amdgcn_sched_barrier(0);
        float qmn = 0.0f, qmx = 0.0f;
#pragma unroll
        for (int u = 0; u < PN; ++u) {
            icx::dql::acc_minmax(xp[u].x, qmn, qmx);
            icx::dql::acc_minmax(xp[u].y, qmn, qmx);
        }
        icx::dql::block_minmax<NT>(qmn, qmx);
        prm = icx::dql::make_params(qmn, qmx);
        azp = prm.zp;
        for (int s = s0; s < e; s += U) {
            if (s != s0) load(s);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (s + u >= e) break;
                v4i a[TI], b[TJ];
#pragma unroll
                for (int i = 0; i < TI; ++i)
#pragma unroll
                    for (int c = 0; c < 4; ++c) a[i][c] = (int)icx::dql::quant4(xv[u][i][c], prm) ^ axr;
#pragma unroll
                for (int j = 0; j < TJ; ++j) b[j] = as_v4i(rb[u][j]);
                step(a, b);
            }
        }
    } else {
        for (int s = s0; s < e; s += U) {
            uint4 ra[U][TI], rb[U][TJ];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int k = min(s + u, e - 1) * 64 + lk;  // past the end: the last step again, not used
#pragma unroll
                for (int i = 0; i < TI; ++i) ra[u][i] = ld16<VEC>(pa[i] + k);
#pragma unroll
                for (int j = 0; j < TJ; ++j) rb[u][j] = ld16<VEC>(pb[j] + k);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (s + u >= e) break;
                v4i a[TI], b[TJ];
#pragma unroll
                for (int i = 0; i < TI; ++i) a[i] = as_v4i(ra[u][i]) ^ axr;
#pragma unroll
                for (int j = 0; j < TJ; ++j) b[j] = as_v4i(rb[u][j]);
                step(a, b);
            }
        }
    }
    if (!AQ && steps > full && steps - 1 >= s0 && steps - 1 < s0 + per) {
        const int k = full * 64 + lk;
        v4i a[TI], b[TJ];
#pragma unroll
        for (int i = 0; i < TI; ++i) a[i] = as_v4i(ld16_tail<VEC>(pa[i], k, g.K, g.a_xor));
#pragma unroll
        for (int j = 0; j < TJ; ++j) b[j] = as_v4i(ld16_tail<VEC>(pb[j], k, g.K, 0u));
        step(a, b);
    }

#pragma unroll
    for (int i = 0; i < TI; ++i) {
#pragma unroll
        for (int j = 0; j < TJ; ++j) part[wid][i * TJ + j][lane] = acc[i][j];
        if (self) rpart[wid][i][lane] = racc[i];
    }
    if (selfc) {
#pragma unroll
        for (int j = 0; j < TJ; ++j) cpart[wid][j][lane] = cacc[j][0];  // every row holds the column's sum
    }
    if constexpr (OPS) {
        if (ok < ICX_MAX_CHAIN) {
            if constexpr (AQ) {  // the activation's scale, just computed (scalar: the host checks)
                if (ok < g.chain.n_ops && icx::op_takes_operand(g.chain.ops[ok].op)) {
                    if (g.chain.ops[ok].p0 == g.q_scale) f0 = (float)prm.s;
                    if (g.chain.ops[ok].p1 == g.q_scale) f1 = (float)prm.s;
                }
            }
            const float a = __fmul_rn(f0, f1);  // f1 == 1 without a second factor: f0 itself
            sop[ok][oc] = icx::div_feeds_erf(g.chain, ok) ? __fdiv_rn(1.0f, a) : a;
        }
    }
    __syncthreads();

    float mn = 0.0f, mx = 0.0f;  // DQL range of the output (when g.part is given)
    if (wid < TILES) {
        v4i sum = part[0][wid][lane];
#pragma unroll
        for (int w = 1; w < W; ++w) sum += part[w][wid][lane];
        if (self) {
            v4i r = rpart[0][ti][lane];
#pragma unroll
            for (int w = 1; w < W; ++w) r += rpart[w][ti][lane];
#pragma unroll
            for (int q = 0; q < 4; ++q) rs[q] = (uint32_t)r[q];
        }
        if (selfc) {
#pragma unroll
            for (int w = 0; w < W; ++w) csum += (uint32_t)cpart[w][tj][lane];
        }
        const uint32_t amz = (uint32_t)(g.alpha - azp), colfac = (uint32_t)(g.beta - bzp);
        const uint32_t colterm = amz * csum + (uint32_t)g.K * amz * colfac;
        const OutView ov = out_view(g, n0);
        float4 v[1];
        float* w = reinterpret_cast<float*>(v);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t x = (uint32_t)sum[r] + colterm + colfac * rs[r];
            w[r] = OUT == OUT_I32 ? __int_as_float((int32_t)x) : (float)(int32_t)x;  // Cast: RNE
        }
        if constexpr (OPS) {
            icx::run_chain4<MODE>(g.codes, g.chain.n_ops, v, [&](int k) {
                const float o = sop[k][tj * 16 + lr];
                return make_float4(o, o, o, o);
            });
        } else if constexpr (OUT == OUT_F32) {
#pragma unroll
            for (int r = 0; r < 4; ++r) w[r] = icx::apply_chain(g.chain, w[r], min(row0 + r, g.M - 1), ccol, g.N);
        }
        if (col < g.N) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (row0 + r >= g.M) continue;
                ov.base[(size_t)(row0 + r) * ov.ld + (col - ov.c0)] = w[r];
                if (OUT == OUT_F32 && g.part) icx::range_acc(w[r], mn, mx);
            }
        }
    }
    if (OUT == OUT_F32 && g.part) icx::block_range_store<NT>(mn, mx, g.part);
}
