// GEMM of BF16 / F16 weights (unquantized model files) over many fp32 activation rows on the 16-bit
// matrix cores: Y[b, r] = sum_c W[r, c] * x[b, c] (+ bias, residual or SwiGLU epilogue).
//
// Reference semantics: the F32-accumulated product of runtime/vault3.c:499-535 over a block of rows.
//
// Exactness.  The activations enter as three bf16 pieces cut from the fp32 mantissa by truncation (8 + 8 + 8
// bits, each element under its own exponent: every product is exact and the pieces add up to the activation,
// but for pieces below bf16's normal range).  BF16 weights enter as they are, F16 weights as two bf16 pieces
// (8 + 3 bits, exact over fp16's whole range), widened from the staged tile.  All pieces of a block accumulate
// into one fp32 accumulator.
//
// What bounds it: at chunk sizes the matrix cores at three (F16: six) times the product's operations (gate/up
// 2 x 8960 x 1536 over 1024 rows: 184 us, 306 TFLOP/s of the product, 920 of the pieces, against 1200 of
// a large library product), below about 100 rows the weights' HBM stream (55 MB, 25 us) and the padding
// of the 64-row tile.  The fp32 MFMA that f32gemm_tile_kernel runs has 1/16 of the 16-bit rate (gate/up
// 591 us at 95 TFLOP/s; down 1536 x 8960, 384 workgroups of 64 x 64 whose chain of 280 blocks is not split: 467
// us against 107).
#pragma once

namespace {

constexpr int kPlanes = 3;
constexpr int kWgTM = 256, kWgTN = 64;     // weight rows x activation rows of a tile

// Three bf16 planes of the activations, natural order: plane p of row b at xs + p * pstride + b * cols.
// One thread per four elements.
__global__ __launch_bounds__(256) void xsplit_bf16x3_kernel(const float *__restrict__ x, int64_t ldx, int cols,
                                                             int64_t n4, uint16_t *__restrict__ xs, int64_t pstride) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    const int64_t b = i / (cols / 4);
    const int c = (int)(i - b * (cols / 4)) * 4;
    const float *xp = x + b * ldx + c;
    float e[4];
    if (((uintptr_t)xp & 15) == 0) {
        const float4 v = *reinterpret_cast<const float4 *>(xp);
        e[0] = v.x; e[1] = v.y; e[2] = v.z; e[3] = v.w;
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) e[k] = xp[k];
    }
    uint32_t h[4], m[4], l[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        h[k] = __float_as_uint(e[k]) & 0xFFFF0000u;
        const float r = e[k] - __uint_as_float(h[k]);               // exact: the low 16 mantissa bits
        m[k] = __float_as_uint(r) & 0xFFFF0000u;
        l[k] = __float_as_uint(r - __uint_as_float(m[k]));          // exact: at most 8 bits
    }
    const auto put = [&](int p, const uint32_t (&v)[4]) {
        *reinterpret_cast<uint2 *>(xs + p * pstride + b * cols + c) =
            make_uint2(v[0] >> 16 | (v[1] & 0xFFFF0000u), v[2] >> 16 | (v[3] & 0xFFFF0000u));
    };
    put(0, h);
    put(1, m);
    put(2, l);
}

// Eight fp16 weights as bf16 pieces: hi the leading 8 bits of the significand, lo the other 3.
__device__ __forceinline__ void widen_f16x8(uint4 h, uint4 &hi, uint4 &lo) {
    const uint32_t w[4] = {h.x, h.y, h.z, h.w};
    uint32_t hv[4], lv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = half_bits_to_float(w[i]), b = half_bits_to_float(w[i] >> 16);
        const uint32_t ha = __float_as_uint(a) & 0xFFFF0000u, hb = __float_as_uint(b) & 0xFFFF0000u;
        hv[i] = ha >> 16 | hb;
        lv[i] = __float_as_uint(a - __uint_as_float(ha)) >> 16 | (__float_as_uint(b - __uint_as_float(hb)) & 0xFFFF0000u);
    }
    hi = make_uint4(hv[0], hv[1], hv[2], hv[3]);
    lo = make_uint4(lv[0], lv[1], lv[2], lv[3]);
}

// One output of blocks blk_lo .. blk_hi - 1 from the operands as they are, for the outputs that the pieces make
// NaN: an infinite weight or activation meets a piece that is zero (or the rest of an infinity), where the product
// itself is an infinity or NaN as the other factor says.
template <int WDT>
__device__ float wgemm_plain_dot(const uint8_t *__restrict__ W, int nblk, int64_t row, int blk_lo, int blk_hi,
                                 const float *__restrict__ xr) {
    const uint16_t *wr = reinterpret_cast<const uint16_t *>(W) + ((row >> 2) * nblk * 4 + (row & 3)) * QK;
    float s = 0.0f;
#pragma unroll 1
    for (int blk = blk_lo; blk < blk_hi; ++blk)
#pragma unroll 4
        for (int j = 0; j < QK; ++j) {
            const uint32_t w = wr[(int64_t)blk * 4 * QK + j];
            s = fmaf(WDT == VGX_BF16 ? bf16_bits_to_float(w) : half_bits_to_float(w), xr[blk * QK + j], s);
        }
    return s;
}

// Tile of 256 weight rows x 64 activation rows, a wave 64 x 64.  Two stages of one 32-wide K block of the weights
// and of every activation plane are filled by LDS DMA: the loads of block k + 1 leave behind the barrier of
// block k (past the range they read zeros).  Rows of a stage are 64 bytes (one block), their 16-byte
// pieces swizzled by (row >> 2) & 3 against bank conflicts of the MFMA operand reads.  M0 is written by
// the DMA alone (checked in the compiled code, as dma16 asks).
// Tiles measured (BF16, gate/up | down over 333 and 1024 rows, us): 256 x 64 with two stages 76, 184 | 53,
// 107; 128 x 128 78, 187 | 53, 108; 256 x 64 with three stages (one workgroup per CU) 94, 222 | 58, 115;
// 256 x 128 of eight waves with two stages 83, 176 | 65, 105, with three 93, 203 | 71, 114.
template <int WDT, int EPI, bool SPLIT>
__global__ __launch_bounds__(256, 2) void wgemm_tile_kernel(
    const uint8_t *__restrict__ W, int64_t n_rq, int nblk, int64_t rows_out, const uint16_t *__restrict__ xs,
    int64_t pstride, const float *__restrict__ x, int64_t ldx, int64_t batch, const float *__restrict__ bias,
    float *__restrict__ y, int64_t ldy, float *__restrict__ part, int kper) {
    constexpr int NP = kPlanes;
    constexpr int NW = WDT == VGX_F16 ? 2 : 1;         // bf16 pieces of a weight
    constexpr int TM = kWgTM, TN = kWgTN, NWAVE = TM / 64, NT = 64 * NWAVE;
    constexpr int A_B = TM * QK * 2, BH_B = TN * QK * 2;
    constexpr int STAGE_B = A_B + NP * BH_B;
    constexpr int NJ = STAGE_B / 1024;                 // wave-loads per block
    constexpr int NPW = NJ / NWAVE;
    static_assert(NJ % NWAVE == 0, "every wave issues the same loads");
    constexpr int kERow = 64 + 4;
    constexpr int EPI_B = TN * kERow * 4;
    __shared__ __align__(16) uint8_t smem[2 * STAGE_B > EPI_B ? 2 * STAGE_B : EPI_B];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lg = lane >> 4;
    const int cols = nblk * QK;
    // XCD-aware tile order, as qgemm_tile_dma_kernel's
    int tr = blockIdx.x, tt = blockIdx.y;
    {
        const int64_t G = gridDim.x, total = G * gridDim.y, id = blockIdx.x + G * blockIdx.y;
        if (total % 8 == 0) {
            const int64_t s = (id % 8) * (total / 8) + id / 8;
            tt = (int)(s / G);
            tr = (int)(s - (int64_t)tt * G);
        }
    }
    const int64_t rq0 = (int64_t)tr * (TM / 4);
    const int64_t b0 = (int64_t)tt * TN;
    const int blk_lo = SPLIT ? (int)blockIdx.z * kper : 0;
    const int blk_hi = SPLIT ? min(nblk, blk_lo + kper) : nblk;

    const dma_rsrc_t wrs = dma_rsrc(W, (uint32_t)(n_rq * nblk * 4 * QK * 2));
    const dma_rsrc_t xrs = dma_rsrc(xs, (uint32_t)(((NP - 1) * pstride + batch * cols) * 2));
    // byte offsets of this lane's 16-byte pieces at block 0 (kDmaPast: rows past the operand)
    uint32_t off[NPW];
#pragma unroll
    for (int i = 0; i < NPW; ++i) {
        const int j = i * NWAVE + wave;
        const int row = (j < A_B / 1024 ? j : (j - A_B / 1024) % (BH_B / 1024)) * 16 + (lane >> 2);
        const int piece = (lane & 3) ^ ((row >> 2) & 3);
        if (j < A_B / 1024) {
            const int64_t rq = rq0 + (row >> 2);
            off[i] = rq < n_rq ? (uint32_t)(((rq * nblk) * 4 + (row & 3)) * QK * 2 + piece * 16) : kDmaPast;
        } else {
            const int64_t b = b0 + row, p = (j - A_B / 1024) / (BH_B / 1024);
            off[i] = b < batch ? (uint32_t)((p * pstride + b * cols) * 2 + piece * 16) : kDmaPast;
        }
    }
    auto issue = [&](int blk, int buf) {
        const bool in = blk < blk_hi;
#pragma unroll
        for (int i = 0; i < NPW; ++i) {
            const int j = i * NWAVE + wave;
            const bool isw = j < A_B / 1024;
            const uint32_t o = in && off[i] != kDmaPast ? off[i] + (uint32_t)blk * (isw ? 4 * QK * 2 : QK * 2) : kDmaPast;
            dma16(isw ? wrs : xrs, o, smem + buf * STAGE_B + j * 1024);
        }
    };
    f32x4_t acc[4][4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[t][c] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto frag = [&](int base, int row) {
        return *reinterpret_cast<const uint4 *>(smem + base + row * 64 + 16 * (lg ^ ((row >> 2) & 3)));
    };
    auto compute = [&](int buf) {
        const int s0 = buf * STAGE_B;
        uint4 af[NW][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            af[0][t] = frag(s0, wave * 64 + 16 * t + l16);
            if constexpr (WDT == VGX_F16) widen_f16x8(af[0][t], af[0][t], af[NW - 1][t]);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                const uint4 bf = frag(s0 + A_B + p * BH_B, 16 * c + l16);
#pragma unroll
                for (int w = 0; w < NW; ++w)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, af[w][t]),
                                                                             __builtin_bit_cast(bf16x8_t, bf), acc[t][c],
                                                                             0, 0, 0);
            }
        }
    };

    const int nb = blk_hi - blk_lo;
    issue(blk_lo, 0);
    int cur = 0;
    for (int k = 0; k < nb; ++k) {
        // block k of this wave has landed and its reads of block k - 1 are done; the barrier extends both
        // to the workgroup, so block k is complete and the stage of block k - 1 is free
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        issue(blk_lo + k + 1, cur ^ 1);
        compute(cur);
        cur ^= 1;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");   // the stages are free for the epilogue

    auto any_nan = [](float4 v) { return !(v.x == v.x && v.y == v.y && v.z == v.z && v.w == v.w); };
    // this lane's NaN sums, four rows at at(t, b, crq, c), computed again
    auto repair = [&](auto at) {
#pragma unroll 1
        for (int e = 0; e < 16; ++e) {
            const int c = e >> 2, t = e & 3;
            const int64_t b = b0 + 16 * c + l16, crq = rq0 + wave * 16 + 4 * t + lg;
            if (b >= batch || crq >= n_rq) continue;
            float *v = at(t, b, crq, c);
#pragma unroll 1
            for (int i = 0; i < 4; ++i)
                if (__builtin_isnan(v[i])) v[i] = wgemm_plain_dot<WDT>(W, nblk, crq * 4 + i, blk_lo, blk_hi, x + b * ldx);
        }
    };
    if constexpr (SPLIT) {
        bool bad = false;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int64_t b = b0 + 16 * c + l16;
            if (b >= batch) continue;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int64_t crq = rq0 + wave * 16 + 4 * t + lg;
                if (crq >= n_rq) continue;
                float4 v;
                v.x = acc[t][c][0]; v.y = acc[t][c][1]; v.z = acc[t][c][2]; v.w = acc[t][c][3];
                *reinterpret_cast<float4 *>(part + ((int64_t)blockIdx.z * batch + b) * (n_rq * 4) + crq * 4) = v;
                bad |= any_nan(v);
            }
        }
        if (bad)
            repair([&](int, int64_t b, int64_t crq, int) {
                return part + ((int64_t)blockIdx.z * batch + b) * (n_rq * 4) + crq * 4;
            });
        return;
    }
    // through LDS in TM / 64 passes of 64 weight rows, so that consecutive threads store consecutive outputs
    float *et = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int half = 0; half < TM / 64; ++half) {
        if (wave == half) {
            bool bad = false;
            auto at = [&](int t, int c) { return et + (16 * c + l16) * kERow + 16 * t + 4 * lg; };
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    float4 v;
                    v.x = acc[t][c][0]; v.y = acc[t][c][1]; v.z = acc[t][c][2]; v.w = acc[t][c][3];
                    *reinterpret_cast<float4 *>(at(t, c)) = v;
                    bad |= any_nan(v);
                }
            if (bad) repair([&](int t, int64_t, int64_t, int c) { return at(t, c); });
        }
        __syncthreads();
        const int64_t r0 = (rq0 + half * 16) * 4;
        if constexpr (EPI == EPI_SWIGLU) {
            // packed row-quad q: rows (gate 2q, gate 2q + 1, up 2q, up 2q + 1) -> outputs 2q, 2q + 1
            for (int i = tid; i < TN * 32; i += NT) {
                const int bl_ = i >> 5, o = i & 31;
                const int64_t b = b0 + bl_, oo = r0 / 2 + o;
                if (b >= batch || oo >= rows_out) continue;
                const float *er = et + bl_ * kERow + (o >> 1) * 4 + (o & 1);
                const float g = er[0], u = er[2];
                y[b * ldy + oo] = g / (1.0f + __expf(-g)) * u;
            }
        } else {
            for (int i = tid; i < TN * 64; i += NT) {
                const int bl_ = i >> 6, rr = i & 63;
                const int64_t b = b0 + bl_, row = r0 + rr;
                if (b >= batch || row >= rows_out) continue;
                float v = et[bl_ * kERow + rr];
                if (bias) v += bias[row];
                if constexpr (EPI == EPI_ACCUM) v += y[b * ldy + row];
                y[b * ldy + row] = v;
            }
        }
        __syncthreads();
    }
}

}  // namespace
