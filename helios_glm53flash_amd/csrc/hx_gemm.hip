// hx_gemm.hip -- EXL3 quantized linear for M > 16 on MFMA (gfx950): the input transform kernel, the plan and
// the dispatch (tile kernels in hx_gemm_impl.hpp, one translation unit per bit width: hx_gemm_b<bits>.hip).
#include "hx_gemm_impl.hpp"

namespace hx {

template <int BITS>
hipError_t launch_mfma_b(int cb, const MfmaGemmArgs& g, hipStream_t st);  // hx_gemm_b*.hip

// a = fp16(H128(fp16(x . suh))) row-wise (had_hf_r_128_inner<true,false>) and, with RS, the fp32 sum of each
// 128-wide block of a.  One wave per 16 consecutive blocks on the matrix cores (hx_gemv.hpp), the
// results stored 16 bytes per lane through LDS.  Bound: memory; M = 2000, K = 4096 (33 MB) 15.6 us with
// one block per wave and a shuffle butterfly.  Few rows: latency, so the column of a block comes from a 32-bit
// remainder (a 64-bit one is a hundred instructions ahead of the first load) and sums nobody reads are not made.
constexpr int HAD_LD = 128 + 8;  // halves per staged block
template <bool RS>
__global__ __launch_bounds__(256) void input_had_kernel(const _Float16* x, const _Float16* suh, _Float16* a, float* rs,
                                                        uint32_t blocks, uint32_t nblk)
{
    __shared__ _Float16 stage[4][16 * HAD_LD];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t b0 = (blockIdx.x * 4 + wave) * 16;
    if (b0 >= blocks) return;
    const uint32_t g = lane >> 4;
    const uint32_t b = min(b0 + (lane & 15), blocks - 1);
    const _Float16* xb = x + (size_t)b * 128 + 8 * g;
    const _Float16* sb = suh + (b % nblk) * 128 + 8 * g;
    InputRegs r;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) r.x[kk] = *reinterpret_cast<const hx_h8u*>(xb + 32 * kk);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) r.s[kk] = *reinterpret_cast<const hx_h8u*>(sb + 32 * kk);
    _Float16* sw = stage[wave];
    input_store(reinterpret_cast<uint32_t*>(sw), r, 16, 0, HAD_LD);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
        const uint32_t j = 4 * q + g, c8 = 8 * (lane & 15);
        const hx_h8 v = *reinterpret_cast<const hx_h8*>(sw + j * HAD_LD + c8);
        if (b0 + j < blocks) *reinterpret_cast<hx_h8u*>(a + (size_t)(b0 + j) * 128 + c8) = v;
        if constexpr (RS) {
            float s = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) s += (float)v[i];
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) s += __shfl_xor(s, o, 64);
            if (b0 + j < blocks && (lane & 15) == 0) rs[b0 + j] = s;
        }
    }
}

hipError_t launch_input_had(const _Float16* x, const _Float16* suh, _Float16* a, float* rs, long rows, int K,
                            hipStream_t st)
{
    const long blocks = rows * (K / 128);  // of 128 fp16: 2^32 of them would be 1 TiB
    if (blocks == 0) return hipSuccess;
    if (blocks > 0xffffffffl - 64) return hipErrorInvalidValue;
    hipLaunchKernelGGL((rs ? input_had_kernel<true> : input_had_kernel<false>), dim3((unsigned)((blocks + 63) / 64)),
                       dim3(256), 0, st, x, suh, a, rs, (uint32_t)blocks, (uint32_t)(K / 128));
    return hipGetLastError();
}

// K splits: tiles that leave more than half of the 768 resident workgroups (3 on each of 256 CUs) empty are split,
// with at least 8 chunks of 64 k each.  A split costs its accumulators a trip through memory (written, then
// read by the last to arrive), so past 5 splits only up to 2 workgroups per CU.  4096 -> 12288 4-bit (96 row x
// column tiles) at M = 45 / 128: 58 / 67 us unsplit, 35.0 / 49.4 with 2, 28.8 / 42.6 with 4, 27.3 / 41.1 with 5,
// 28.9 / 49.4 with 8; 24576 columns (192 tiles) at M = 45: 44.6 with 2, 36.5 with 4; 8192 -> 8192 (64 tiles): 63.0
// with 2, 42.3 with 5, 37.1 with 8 (graphs of 10 calls, input transform included).
// Where tiles alone reach more than half of the CUs a split saves less of a chunk's time, so it has to be longer to
// be worth its trip: 16 chunks (12 at up to 32 rows, whose accumulators are few), and 24 with more tiles than CUs.
// 4-bit, 126 rows, 17792 columns (139 tiles), unsplit / 2 splits: K = 1024 25.4 / 30.6 us, K = 1280 29.1 / 32.9,
// K = 1536 32.8 / 35.6, K = 2048 40.8 / 40.4; 200 rows (278 tiles): K = 1024 28.9 / 36.5, K = 2048 49.5 / 48.4, K = 3072
// 69.0 / 60.1.  (512 to 24576 columns, K = 512 to 8192, 17 to 512 rows, 2, 4 and 6 bits: no shape more than 2 %
// slower than unsplit; with 8 chunks everywhere up to 30 %.)
static int mfma_splits(int M, int K, int N)
{
    const long tiles = (long)((M + MF_BM - 1) / MF_BM) * (N / 128), nk = K / MF_BK;
    auto least = [](long a, long b) { return a < b ? a : b; };
    const long two = 2 * GEMV_CUS / tiles;
    const long chunks = tiles <= GEMV_CUS / 2 ? 8 : tiles > GEMV_CUS ? 24 : M <= 32 ? 12 : 16;
    const long s = least(least(3 * GEMV_CUS / tiles, two > 5 ? two : 5), least(nk / chunks, 8));
    return s > 1 ? (int)s : 1;
}

static size_t al256(size_t v) { return (v + 255) & ~(size_t)255; }

// 16-column fragments of accumulators that a split of the tallest row tile stores.
static int mfma_frags(int M) { return ((M < MF_BM ? M : MF_BM) + 15) / 16 * 2; }

// A function of the shape alone, so that a shape takes the same path (and rounds alike) wherever MFMA_EXTRA_BYTES are
// there: what does not fit those is left out even if the caller has more.
MfmaExtra mfma_extra(int M, int K, int N)
{
    MfmaExtra e{al256((size_t)M * (K / 128) * sizeof(float)), 0, 1};
    if (e.rs > MFMA_EXTRA_BYTES) return MfmaExtra{0, 0, 1};
    const size_t one = (size_t)((M + MF_BM - 1) / MF_BM) * (N / 128) * mfma_frags(M) * MF_THREADS * sizeof(hx_f4);
    int s = mfma_splits(M, K, N);
    while (s > 1 && e.rs + s * one > MFMA_EXTRA_BYTES) --s;
    if (s > 1) {
        e.partial = s * one;
        e.splits = s;
    }
    return e;
}

hipError_t launch_linear_mfma(const _Float16* a_had, const float* rs, const uint16_t* trellis, const _Float16* svh,
                              void* y, int M, int K, int N, int bits, int cb, bool y_fp32, int splits, void* partial,
                              int* counter, hipStream_t st)
{
    MfmaGemmArgs g{a_had, rs, reinterpret_cast<const uint32_t*>(trellis), svh, y, M, K, N, y_fp32,
                   splits, mfma_frags(M), static_cast<hx_f4*>(partial), counter};
    switch (bits) {
        case 1: return launch_mfma_b<1>(cb, g, st);
        case 2: return launch_mfma_b<2>(cb, g, st);
        case 3: return launch_mfma_b<3>(cb, g, st);
        case 4: return launch_mfma_b<4>(cb, g, st);
        case 5: return launch_mfma_b<5>(cb, g, st);
        case 6: return launch_mfma_b<6>(cb, g, st);
        case 7: return launch_mfma_b<7>(cb, g, st);
        case 8: return launch_mfma_b<8>(cb, g, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace hx
