// hx_router.hip -- dense fp16 NT GEMM y[m][n] = sum_k x[m][k] * w[n][k] (w row-major [N][K], fp32
// accumulate), the router-logits front end of the MoE layer on gfx950.  Reference semantics:
// helios::glue::gemm_nt_f16 / gemv_nt_f16 (src/engine/glue2.cu:9-65,165-182): fp16 output rounded
// once from the fp32 sum, or fp32 output (optionally added to y).
//
//   M <= 8   gemv: one workgroup per output column n; its 4 waves split K, each lane takes 8
//            consecutive k per step (16-byte loads of w and x), v_dot2_f32_f16 accumulation, the
//            wave sums added in wave order.
//   M > 8    MFMA, the waves of a workgroup split K (gemm_nt_split_kernel): each streams both operands of
//            its k range through LDS by itself, and the waves' sums are added at the end.
#include "hx_mfma.hpp"
#include "hx_kernels.hpp"

namespace hx {

namespace {

typedef uint32_t u4v __attribute__((ext_vector_type(4)));

HX_INLINE float dot8(u4v a, u4v b, float acc)
{
    acc = __builtin_amdgcn_fdot2(u32_as_h2(a.x), u32_as_h2(b.x), acc, false);
    acc = __builtin_amdgcn_fdot2(u32_as_h2(a.y), u32_as_h2(b.y), acc, false);
    acc = __builtin_amdgcn_fdot2(u32_as_h2(a.z), u32_as_h2(b.z), acc, false);
    acc = __builtin_amdgcn_fdot2(u32_as_h2(a.w), u32_as_h2(b.w), acc, false);
    return acc;
}

HX_INLINE void store_out(void* y, size_t idx, float v, bool y_fp32, bool add)
{
    if (y_fp32) {
        float* yf = static_cast<float*>(y);
        yf[idx] = add ? yf[idx] + v : v;
    } else {
        static_cast<_Float16*>(y)[idx] = (_Float16)v;
    }
}

}  // namespace

template <int MT>
__global__ __launch_bounds__(256) void gemv_nt_kernel(const _Float16* x, const _Float16* w, void* y, int M, int N,
                                                      int K, bool y_fp32, bool add)
{
    __shared__ float part[4][MT];
    const int n = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int kq = (K / 4 + 7) & ~7;  // k range of a wave, a multiple of 8
    const int k0 = wave * kq, k1 = min(K, k0 + kq);
    const _Float16* wr = w + (size_t)n * K;
    float acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = 0.0f;
    for (int k = k0 + 8 * lane; k < k1; k += 512) {
        const u4v wv = *reinterpret_cast<const u4v*>(wr + k);
#pragma unroll
        for (int m = 0; m < MT; ++m)
            if (m < M) acc[m] = dot8(*reinterpret_cast<const u4v*>(x + (size_t)m * K + k), wv, acc[m]);
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        float v = acc[m];
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) part[wave][m] = v;
    }
    __syncthreads();
    if (threadIdx.x < M) {
        const int m = threadIdx.x;
        const float v = ((part[0][m] + part[1][m]) + part[2][m]) + part[3][m];
        store_out(y, (size_t)m * N + n, v, y_fp32, add);
    }
}

// One workgroup: rows 16 RB * bx + .., columns 16 CB * by + ..; its KS waves take equal k ranges of the
// same tile, and their fp32 sums are added pairwise through LDS (wave w + wave w + h, h = KS/2, .., 1: a
// fixed order).  N is small here (a router's 64-288 experts), so tiles alone leave the chip idle, and one
// wave per 32 x 32 block over all of K waited a round trip of latency every few steps (115 us at
// 4096 x 288 x 4096, 27 us at M = 16).  A wave has NB chunks of 64 k in LDS buffers of its own, filled
// by buffer loads with an LDS destination (8 rows x 128 bytes each): no barrier, only its own loads to
// wait for.  What bounds it is these loads: 24.9 us at 4096 x 288 x 4096, 22.0 without the MFMAs, 24.1 without the
// LDS reads, 21.7 with neither (251 MB through 192 CUs, 60 GB/s each; at M = 512 8.4 / 7.9 / 8.0 / 7.7, and nothing at
// 64 experts).  In whole 128-byte lines a CU reads up to 115 GB/s from L2, in the 64-byte halves that fragments loaded
// straight into MFMA layout touch 37 GB/s (that variant of this kernel: 45 us at M = 4096, 17 us at M = 33-512).
// LDS rows are 64 halves with the 16-byte chunks of row r permuted by mf_swz(r) (hx_mfma.hpp).
// DMA false: x or w is not 16-byte aligned, which the buffer loads into LDS ask for; the chunks go through
// registers (global loads take any address), without loads in flight across chunks.
template <int RB, int CB, int KS, int NB, bool DMA>
__device__ __forceinline__ void gemm_nt_split(const _Float16* x, const _Float16* w, void* y, int M, int N, int K,
                                              bool y_fp32, bool add)
{
    constexpr int ROWS = 16 * (RB + CB), NL = ROWS / 8;  // LDS rows and loads per chunk
    static_assert(sizeof(hx_f4) * 64 * RB * CB * (KS / 2) <= sizeof(_Float16) * KS * NB * ROWS * 64, "sums fit the buffers");
    extern __shared__ _Float16 buf[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r0 = 16 * RB * blockIdx.x, c0 = 16 * CB * blockIdx.y;
    const int nk = (K + 63) / 64, kq = (nk + KS - 1) / KS;  // chunks in all, per wave
    const int q0 = wave * kq, n = min(nk, q0 + kq) - q0;
    _Float16* wb = buf + (size_t)wave * NB * ROWS * 64;
    const __amdgpu_buffer_rsrc_t rx = mf_rsrc(x + (size_t)r0 * K, (size_t)(M - r0) * K * sizeof(_Float16));
    const __amdgpu_buffer_rsrc_t rw = mf_rsrc(w + (size_t)c0 * K, (size_t)(N - c0) * K * sizeof(_Float16));
    // lane l of load i fetches, for LDS row r = 8i + l/8, the chunk that the permutation puts in slot l % 8;
    // rows past the end (clamped) are computed but not stored; a chunk past K reads the next row's k or,
    // past the end, zeros, and its MFMAs are skipped below
    int voff[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int r = 8 * i + (lane >> 3), rr = i < 2 * RB ? min(r, M - r0 - 1) : min(r - 16 * RB, N - c0 - 1);
        voff[i] = (int)(((size_t)rr * K + 8 * ((lane & 7) ^ mf_swz(r))) * sizeof(_Float16));
    }
    auto load = [&](int p) {
        const int q = q0 + p;
        _Float16* d = wb + p % NB * ROWS * 64;
        if constexpr (DMA) {
#pragma unroll
            for (int i = 0; i < NL; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(i < 2 * RB ? rx : rw,
                                                         (__attribute__((address_space(3))) void*)(d + 512 * i), 16,
                                                         voff[i], q * 128, 0, 0);
        } else {
            typedef _Float16 h8a2 __attribute__((ext_vector_type(8), aligned(2)));
            hx_h8 v[NL];
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const _Float16* s = (i < 2 * RB ? x + (size_t)r0 * K : w + (size_t)c0 * K) + voff[i] / 2 + 64 * q;
                v[i] = hx_h8{};
                if (64 * q + 8 * ((lane & 7) ^ mf_swz(8 * i + (lane >> 3))) < K) v[i] = *reinterpret_cast<const h8a2*>(s);
            }
#pragma unroll
            for (int i = 0; i < NL; ++i) *reinterpret_cast<hx_h8*>(d + 512 * i + 8 * lane) = v[i];
        }
    };
    hx_f4 acc[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i][j] = hx_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < NB; ++p) {
        if (p < n) load(p);
        asm volatile("" ::: "memory");  // the waits below count whole chunks: their loads stay apart
    }
    for (int p = 0; p < n; ++p) {
        // chunk p has arrived once at most the loads of the later chunks in flight are outstanding
        asm volatile("" ::: "memory");
        if (n - p >= NB) __builtin_amdgcn_s_waitcnt(qt_vmcnt((NB - 1) * NL));
        else __builtin_amdgcn_s_waitcnt(qt_vmcnt(0));
        asm volatile("" ::: "memory");
        const int q = q0 + p;
        const _Float16* s = wb + p % NB * ROWS * 64;
        hx_h8 f[2][RB + CB];
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int i = 0; i < RB + CB; ++i)
                f[kk][i] = *reinterpret_cast<const hx_h8*>(s + mf_off(16 * i + (lane & 15), 4 * kk + (lane >> 4)));
        // every fragment is in registers before the buffer is refilled
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        asm volatile("" ::: "memory");
        if (p + NB < n) load(p + NB);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
            if (kk == 0 || 64 * q + 32 < K) {  // K is a multiple of 32
#pragma unroll
                for (int i = 0; i < RB; ++i)
#pragma unroll
                    for (int j = 0; j < CB; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[kk][i], f[kk][RB + j], acc[i][j], 0, 0, 0);
            }
    }
    hx_f4* part = reinterpret_cast<hx_f4*>(buf);  // [KS / 2][RB * CB][64]
    __syncthreads();                              // every wave is done with its buffers
#pragma unroll
    for (int h = KS / 2; h >= 1; h >>= 1) {
        if (wave >= h && wave < 2 * h) {
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j) part[((wave - h) * RB * CB + i * CB + j) * 64 + lane] = acc[i][j];
        }
        __syncthreads();
        if (wave < h) {
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j) acc[i][j] += part[(wave * RB * CB + i * CB + j) * 64 + lane];
        }
        if (h > 1) __syncthreads();
    }
    if (wave != 0) return;
    // C: lane holds column lane % 16, rows 4 * (lane / 16) + r of each 16 x 16 block
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = r0 + 16 * i + 4 * (lane >> 4) + r, n = c0 + 16 * j + (lane & 15);
                if (m < M && n < N) store_out(y, (size_t)m * N + n, acc[i][j][r], y_fp32, add);
            }
}

template <int RB, int CB, int KS, int NB, bool DMA>
__global__ __launch_bounds__(64 * KS) void gemm_nt_split_kernel(const _Float16* x, const _Float16* w, void* y, int M,
                                                                int N, int K, bool y_fp32, bool add)
{
    gemm_nt_split<RB, CB, KS, NB, DMA>(x, w, y, M, N, K, y_fp32, add);
}

struct NtCall {
    const _Float16 *x, *w;
    void* y;
    int M, N, K;
    bool y_fp32, add;
};

// Rounds of workgroups (one per CU, by LDS) times the rows of x and w that a workgroup reads.
template <int RB, int CB>
static long nt_cost(const NtCall& c)
{
    const long wgs = (long)((c.M + 16 * RB - 1) / (16 * RB)) * ((c.N + 16 * CB - 1) / (16 * CB));
    return (wgs + 255) / 256 * (RB + CB);
}

template <int RB, int CB, int KS, int NB, bool DMA = true>
static hipError_t nt_launch(const NtCall& c, hipStream_t st)
{
    constexpr size_t lds = sizeof(_Float16) * KS * NB * 16 * (RB + CB) * 64;
    hipLaunchKernelGGL((gemm_nt_split_kernel<RB, CB, KS, NB, DMA>),
                       dim3((c.M + 16 * RB - 1) / (16 * RB), (c.N + 16 * CB - 1) / (16 * CB)), dim3(64 * KS), lds, st,
                       c.x, c.w, c.y, c.M, c.N, c.K, c.y_fp32, c.add);
    return hipGetLastError();
}

hipError_t launch_gemm_nt_f16(const _Float16* x, const _Float16* w, void* y, int M, int N, int K, bool y_fp32,
                              bool add, hipStream_t st)
{
    if (M <= 0 || N <= 0) return hipSuccess;
    if (M <= 8) {
        if (M <= 1)
            hipLaunchKernelGGL((gemv_nt_kernel<1>), dim3(N), dim3(256), 0, st, x, w, y, M, N, K, y_fp32, add);
        else
            hipLaunchKernelGGL((gemv_nt_kernel<8>), dim3(N), dim3(256), 0, st, x, w, y, M, N, K, y_fp32, add);
    } else {
        // The tile with the least reading on the busiest CU; equal costs go to the larger tile (fewer bytes
        // in all).
        const NtCall c{x, w, y, M, N, K, y_fp32, add};
        if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) return nt_launch<2, 2, 8, 2, false>(c, st);
        const long cost[5] = {nt_cost<4, 6>(c), nt_cost<4, 4>(c), nt_cost<2, 3>(c), nt_cost<2, 2>(c), nt_cost<1, 1>(c)};
        int best = 0;
        for (int i = 1; i < 5; ++i)
            if (cost[i] < cost[best]) best = i;
        switch (best) {
            case 0: return nt_launch<4, 6, 4, 2>(c, st);
            case 1: return nt_launch<4, 4, 4, 2>(c, st);
            case 2: return nt_launch<2, 3, 8, 2>(c, st);
            case 3: return nt_launch<2, 2, 8, 2>(c, st);
            default: return nt_launch<1, 1, 16, 2>(c, st);
        }
    }
    return hipGetLastError();
}

}  // namespace hx
