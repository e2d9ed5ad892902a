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

// K splits: row x column tiles that leave more than half of the 768 resident workgroups (3 on each of 256 CUs) empty,
// split where that is faster than the unsplit tile, which sums its input itself (2, 4, 5, 6 and 8 bits, 512 to 40960
// columns, K = 512 to 8192, 17 to 2000 rows: 4378 shapes, against the unsplit call 0.823 in the geometric mean, 2 %
// slower or more at 9 of them; the best split of each shape would give 0.819).
// A split costs row sums ahead of it, and its accumulators a trip through memory (written, then read by the last to
// arrive).  The more CUs the tiles fill by themselves, the less a split saves, so K has to be the longer: in chunks
// of 64, tiles / 4 up to 128 tiles (half of the CUs; never under 20), tiles / 3 beyond.  4-bit, M = 100: 64
// tiles (8192 columns) K = 1024 22.0 us unsplit, 22.3 with 2 splits, K = 1280 24.9 / 22.4 with 3, K = 2048 33.0 / 26.6 with 4;
// 139 tiles (17792 columns) K = 2048 33.8 / 36.1 with 3, K = 2560 39.5 / 39.2, K = 3072 45.0 / 41.4 with 5.
// One workgroup per CU where 4 splits or more reach that, two if K is 6144 or longer; else at most 5.  48 tiles,
// 8-bit, K = 3072, M = 100: 45.8 us unsplit, 30.4 with 5, 36.6 with 8.
static int mfma_splits(int M, int K, int N)
{
    const long tiles = (long)((M + MF_BM - 1) / MF_BM) * (N / 128), nk = K / MF_BK;
    auto least = [](long a, long b) { return a < b ? a : b; };
    const long from = tiles <= GEMV_CUS / 2 ? (tiles + 3) / 4 : (tiles + 2) / 3;
    if (nk < (from > 20 ? from : 20)) return 1;
    const long round = (nk >= 96 ? 2 : 1) * GEMV_CUS / tiles;
    const long s = least(least(3 * GEMV_CUS / tiles, round >= 4 ? round : 5), least(nk / (tiles <= 64 ? 6 : 8), 8));
    return s > 1 ? (int)s : 1;
}

static size_t al256(size_t v) { return (v + 255) & ~(size_t)255; }

// 16-column fragments of accumulators that a split of the tallest row tile stores.
static int mfma_frags(int M) { return ((M < MF_BM ? M : MF_BM) + 15) / 16 * 2; }

// Unsplit calls with row sums made ahead of the tiles (whose input then goes to LDS by buffer loads): codebook 2 at up
// to 4 bits.  It saves VALU work, which pays while 3 workgroups share a CU, but a chunk then takes longer for a
// workgroup that has its CU almost to itself.  So the last round of tiles decides (768 a round), the less the more
// full rounds there are.  Sustained, sums ahead over sums in the tile, 4-bit, K = 4096, M = 512: 384 tiles 1.09, 512 1.03,
// 544 0.97, 768 0.98; 784 1.08, 960 1.04, 1088 1.01, 1152 1.00, 1280 0.99, 1536 0.98; 1568 1.02, 1632 1.00, 1728 0.97; 2304 and
// more 0.97-0.99 (the same within 0.03 at 2 and 3 bits, K = 2048 and 8192, M = 256 and 1024).  More bits (two loads of
// trellis words a chunk): 5-bit 4096 -> 151552, M = 512 1.02, 4096 -> 24576, M = 2000 1.02, 8-bit 8192 -> 40960, M = 1500 1.05.
static bool sums_ahead(long tiles, int bits)
{
    constexpr long ROUND = 3 * GEMV_CUS;
    const long full = tiles / ROUND, last = tiles % ROUND;
    return bits <= 4 && (last == 0 || last > (full == 0 ? 512 : full == 1 ? 383 : full == 2 ? 111 : 0));
}

// A function of shape, width and codebook alone, so that a call takes the same path (and rounds alike) wherever
// MFMA_EXTRA_BYTES are there: what does not fit those is left out even if the caller has more.
MfmaExtra mfma_extra(int M, int K, int N, int bits, int cb)
{
    const size_t rs = al256((size_t)M * (K / 128) * sizeof(float));
    const long tiles = (long)((M + MF_BM - 1) / MF_BM) * (N / 128);
    const size_t one = (size_t)tiles * mfma_frags(M) * MF_THREADS * sizeof(hx_f4);
    int s = mfma_splits(M, K, N);
    while (s > 1 && rs + s * one > MFMA_EXTRA_BYTES) --s;
    if (s > 1) return MfmaExtra{rs, s * one, s};
    const bool ahead = cb == 2 && sums_ahead(tiles, bits) && rs <= MFMA_EXTRA_BYTES;
    return MfmaExtra{ahead ? rs : 0, 0, 1};
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
