// hx_gemm_impl.hpp -- EXL3 quantized linear for M > 16 on MFMA (gfx950): quarter-operand MFMA tiles
// (hx_mfma.hpp) over the transformed input, split over K where the tiles leave the chip idle, with the
// output Hadamard + svh epilogue fused.  One translation unit per bit width (hx_gemm_b<bits>.hip).
// Reference semantics: src/cuda/quant/exl3_gemm_kernel.cuh:8-80, exl3_gemm_inner.cuh:456-480.
#pragma once
#include "hx_mfma.hpp"
#include "hx_kernels.hpp"

namespace hx {

struct MfmaGemmArgs {
    const _Float16* a;        // M x K transformed input
    const float* rs;          // M x K/128 sums of a's 128-wide blocks (null: the tile sums a itself)
    const uint32_t* trellis;
    const _Float16* svh;
    void* y;
    int M, K, N;
    bool y_fp32;
    int splits;               // K splits (> 1: partial and counter are used, rs is not null)
    int frags;                // accumulator fragments stored per (tile, split), 2 per 16 rows
    hx_f4* partial;           // [tile][split][frags][256] raw accumulators
    int* counter;             // [tile]
};

// 128-point Sylvester transform of a row held by 4 consecutive lanes: value v[8 m + i] of lane p is
// column 32 m + 8 p + i.  Column bits 0-2 and 5-6 are butterflies in registers, bits 3-4 lane
// exchanges within a quad (DPP); scaled by 1/sqrt(128).
HX_INLINE void had128_quad(float (&v)[32])
{
    auto bfly = [&](int h) {
#pragma unroll
        for (int j = 0; j < 32; ++j)
            if (!(j & h)) {
                const float a = v[j], b = v[j + h];
                v[j] = a + b;
                v[j + h] = a - b;
            }
    };
    bfly(1);
    bfly(2);
    bfly(4);
    bfly(8);
    bfly(16);
    const int p = threadIdx.x & 3;
    const float s0 = (p & 1) ? -1.0f : 1.0f, s1 = (p & 2) ? -1.0f : 1.0f;
#pragma unroll
    for (int j = 0; j < 32; ++j)  // lane p ^ 1, then p ^ 2 (quad_perm); fma by +-1 is one rounding of the sum
        v[j] = fmaf(v[j], s0, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v[j]), 0xB1,
                                                                                0xf, 0xf, false)));
#pragma unroll
    for (int j = 0; j < 32; ++j)
        v[j] = fmaf(v[j], s1, __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v[j]), 0x4E,
                                                                                0xf, 0xf, false))) * HX_RSQRT128;
}

// y[row][cg*128 + c] = svh . H128(C[row][:]) for the tile's rows: the accumulators staged in LDS 64 rows at a
// time, 4 lanes per row.  (One wave per row, two columns per lane and 6 shuffle stages took 1900 VALU
// instructions per wave and 128-row tile, a sixth of the tile's work at K = 4096; this takes 700.)
template <int CB, int BM, class Smem>
__device__ __forceinline__ void linear_tile_store(const hx_f4 (&acc)[BM / 16][2], Smem& sm, const MfmaGemmArgs& g,
                                                  int m0, int rows, int cg)
{
    const int r = threadIdx.x >> 2, c = cg * 128 + 8 * (threadIdx.x & 3);
    hx_h8 sv[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) sv[m] = *reinterpret_cast<const hx_h8u*>(g.svh + c + 32 * m);
#pragma unroll
    for (int half = 0; half < (BM + 63) / 64; ++half) {
        if (half) __syncthreads();
        qt_stage_c_half<BM>(acc, half, sm);
        __syncthreads();
        const int row = 64 * half + r;
        float v[32];
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const hx_f4 q = *reinterpret_cast<const hx_f4*>(&sm.c[r * MF_LDC + 32 * m + 8 * (threadIdx.x & 3) + 4 * e]);
#pragma unroll
                for (int i = 0; i < 4; ++i) v[8 * m + 4 * e + i] = q[i];
            }
        if constexpr (CB == 2) {
            const float b = CB2_BIAS * sm.rowsum[min(row, MF_BM - 1)];
#pragma unroll
            for (int j = 0; j < 32; ++j) v[j] = fmaf(v[j], CB2_SCALE, b);
        }
        had128_quad(v);
        if (row >= rows) continue;
        const size_t o = (size_t)(m0 + row) * g.N + c;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            if (g.y_fp32) {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    hx_f4 q;
#pragma unroll
                    for (int i = 0; i < 4; ++i) q[i] = v[8 * m + 4 * e + i] * (float)sv[m][4 * e + i];
                    *reinterpret_cast<hx_f4u*>(static_cast<float*>(g.y) + o + 32 * m + 4 * e) = q;
                }
            } else {
                hx_h8 h;
#pragma unroll
                for (int i = 0; i < 8; ++i) h[i] = (_Float16)v[8 * m + i];
                *reinterpret_cast<hx_h8u*>(static_cast<_Float16*>(g.y) + o + 32 * m) = h * sv[m];
            }
        }
    }
}

// One (row tile, column group, K split).  A split stores its raw accumulators (device-coherent 16-byte
// stores, each lane its own), and the last split of the tile to arrive adds them in split order
// (deterministic) in the same lanes.  EXT: the row sums of a are given, and a goes to LDS by buffer loads; else (never
// split) codebook 2 sums its rows from a on its way through registers.
template <int BITS, int CB, int BM, bool EXT>
__device__ __forceinline__ void linear_tile(const MfmaGemmArgs& g, int mt, int cg, int s, MfmaSmemQ& sm)
{
    const int m0 = mt * MF_BM, rows = min(MF_BM, g.M - m0), t = threadIdx.x;
    const int nk = g.K / MF_BK, nblk = g.K >> 7;
    const int c0 = s * nk / g.splits, c1 = (s + 1) * nk / g.splits;
    hx_f4 acc[BM / 16][2];
    const float* rs = EXT && CB == 2 ? g.rs + (size_t)m0 * nblk : nullptr;
    mfma_tile_q<BITS, CB, BM, EXT>(g.a + (size_t)m0 * g.K + c0 * MF_BK, g.K, rows,
                                          g.trellis + (size_t)(c0 * (MF_BK / 16)) * (g.N >> 4) * (8 * BITS),
                                          (c1 - c0) * MF_BK, g.N, cg * 8, sm, acc, rs, g.splits > 1 ? 0 : nblk);
    if constexpr (EXT) {
        if (g.splits > 1) {
            const int tile = mt * (g.N >> 7) + cg;
            constexpr int NF = BM / 16 * 2;
            const __amdgpu_buffer_rsrc_t rp = mf_rsrc(g.partial + (size_t)tile * g.splits * g.frags * MF_THREADS,
                                                      (size_t)g.splits * g.frags * MF_THREADS * sizeof(hx_f4));
            auto off = [&](int sp, int f) { return ((sp * g.frags + f) * MF_THREADS + t) * (int)sizeof(hx_f4); };
            const int nf = (rows + 15) / 16 * 2;  // fragments that hold rows
#pragma unroll
            for (int f = 0; f < NF; ++f)
                if (f < nf) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(hx_u4v, acc[f >> 1][f & 1]), rp, off(s, f), 0, HX_BUF_SC1);
            if (!arrive_last(&g.counter[tile], g.splits)) return;
#pragma unroll
            for (int f = 0; f < NF; ++f) acc[f >> 1][f & 1] = hx_f4{0.f, 0.f, 0.f, 0.f};
            constexpr int SB = NF <= 4 ? 4 : NF <= 8 ? 2 : 1;  // splits read together (64 registers)
            for (int s0 = 0; s0 < g.splits; s0 += SB) {
                hx_f4 p[SB][NF];
#pragma unroll
                for (int j = 0; j < SB; ++j)
#pragma unroll
                    for (int f = 0; f < NF; ++f)
                        if (f < nf) p[j][f] = __builtin_bit_cast(hx_f4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                rp, off(min(s0 + j, g.splits - 1), f), 0, HX_BUF_SC1));
#pragma unroll
                for (int j = 0; j < SB; ++j)
                    if (s0 + j < g.splits)
#pragma unroll
                        for (int f = 0; f < NF; ++f)
                            if (f < nf) acc[f >> 1][f & 1] += p[j][f];
            }
            if constexpr (CB == 2) {
                if (t < BM) {
                    float v = 0.0f;
                    if (t < rows)
                        for (int b0 = 0; b0 < nblk; b0 += 32) {
                            float q[32];
#pragma unroll
                            for (int j = 0; j < 32; ++j) q[j] = b0 + j < nblk ? rs[(size_t)t * nblk + b0 + j] : 0.0f;
#pragma unroll
                            for (int j = 0; j < 32; ++j) v += q[j];
                        }
                    sm.rowsum[t] = v;
                }
                __syncthreads();
            }
        }
    }
    linear_tile_store<CB, BM>(acc, sm, g, m0, rows, cg);
}

// Quarter-operand tiles of 128 rows, the last row tile 32, 64 or 96 rows tall if that holds its rows;
// three workgroups per CU.
template <int BITS, int CB, bool EXT>
__global__ __launch_bounds__(MF_THREADS, qt_occ<CB>()) void linear_mfma_kernel(MfmaGemmArgs g)
{
    __shared__ MfmaSmemQ sm;
    // the row tiles of a (column group, split) on one XCD: its trellis words come from memory once and the
    // other row tiles read them from that XCD's L2
    int mt, cs;
    if (!xcd_group_index(blockIdx.x + blockIdx.y * gridDim.x, gridDim.y, gridDim.x, mt, cs)) return;
    const int groups = g.N >> 7, cg = cs % groups, s = cs / groups;
    const int rows = g.M - mt * MF_BM;
    if (rows <= 32) return linear_tile<BITS, CB, 32, EXT>(g, mt, cg, s, sm);
    if (rows <= 64) return linear_tile<BITS, CB, 64, EXT>(g, mt, cg, s, sm);
    if (rows <= 96) return linear_tile<BITS, CB, 96, EXT>(g, mt, cg, s, sm);
    linear_tile<BITS, CB, MF_BM, EXT>(g, mt, cg, s, sm);
}

template <int BITS>
hipError_t launch_mfma_b(int cb, const MfmaGemmArgs& g, hipStream_t st)
{
    const dim3 grid(g.N / 128 * g.splits, (g.M + MF_BM - 1) / MF_BM);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(MF_THREADS), 0, st, g);
        return hipGetLastError();
    };
    if (g.rs) {
        switch (cb) {
            case 0: return go(linear_mfma_kernel<BITS, 0, true>);
            case 1: return go(linear_mfma_kernel<BITS, 1, true>);
            default: return go(linear_mfma_kernel<BITS, 2, true>);
        }
    }
    switch (cb) {
        case 0: return go(linear_mfma_kernel<BITS, 0, false>);
        case 1: return go(linear_mfma_kernel<BITS, 1, false>);
        default: return go(linear_mfma_kernel<BITS, 2, false>);
    }
}

}  // namespace hx
