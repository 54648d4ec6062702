// Trellis -> fp16 weight reconstruction for gfx950.
//
//   reconstruct      W_hat (k, n) in the Hadamard basis        (quant/reconstruct.cu:14-98)
//   reconstruct_had  W = diag(suh) H W_hat H diag(svh) per 128x128 block, original basis,
//                    with the reference's fp16 rounding points  (quant/reconstruct.cu:212-364)
//
// Both are bit-exact restatements: the decode is the codebook arithmetic of exl3_common.cuh,
// and every fp16 operation of the fused form is issued in the reference's order (the column
// pass rounds after each add / sub and after the 1/sqrt(128) multiply; the row pass runs its
// first two butterfly stages in fp32, then fp16).
#include "exl3_common.cuh"
#include "exl3_kernels.h"

using namespace exl3;

namespace {

// Load this lane's K words of the 8-tile chunk; ring_prev supplies the word before them.
template <int K>
__device__ __forceinline__ void load_lane_words(const uint32_t* __restrict__ p, uint32_t* w)
{
    if constexpr (K % 4 == 0)
    {
        #pragma unroll
        for (int i = 0; i < K / 4; ++i)
        {
            u32x4 v = __builtin_nontemporal_load((const u32x4*) p + i);
            w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
        }
    }
    else if constexpr (K % 2 == 0)
    {
        #pragma unroll
        for (int i = 0; i < K / 2; ++i)
        {
            u32x2 v = __builtin_nontemporal_load((const u32x2*) p + i);
            w[2 * i] = v.x; w[2 * i + 1] = v.y;
        }
    }
    else
    {
        #pragma unroll
        for (int i = 0; i < K; ++i) w[i] = __builtin_nontemporal_load(p + i);
    }
}

// Decode one k-slice x 128-column chunk per wave: returns the 16 packed pairs of this lane.
template <int K, int CB>
__device__ __forceinline__ void decode_slice(const uint16_t* __restrict__ trellis, int tiles_n,
                                             int kt, int nt0, int lane, uint32_t* pairs,
                                             const DecodeRegs& r)
{
    constexpr int KB = kbits(K);
    uint32_t wv[KB + 1];
    if constexpr (khalf(K))
    {
        const uint32_t* tile = (const uint32_t*) trellis
                             + ((size_t) kt * tiles_n + nt0 + (lane >> 3)) * tile_words(K);
        load_frame_half<K>(tile, lane & 7, wv);
    }
    else
    {
        const uint32_t* base = (const uint32_t*) trellis
                             + ((size_t) kt * tiles_n + nt0) * (8 * K) + (size_t) lane * K;
        load_lane_words<K>(base, wv + 1);
        wv[0] = ring_prev(wv[K], lane);
    }
    decode_lane32<K, CB>(wv, pairs, r);
}

// ------------------------------------------------------------------------------ reconstruct
// Grid (n / 128, ceil(k / 64)), 256 threads: wave w decodes k-slice 4*blockIdx.y + w of the
// 128-column chunk, transposes through LDS and writes 16 coalesced 256-byte rows.
template <int K, int CB>
__global__ __launch_bounds__(256)
void reconstruct_kernel(uint16_t* __restrict__ W, const uint16_t* __restrict__ trellis,
                        int k, int n, int tiles_n, int nt_off)
{
    __shared__ __align__(16) uint32_t sh[4][16][64 + 4];     // per wave: 16 rows x 128 halves (+pad)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int kt = blockIdx.y * 4 + wave;
    const int chunk = blockIdx.x;
    if (kt >= k / 16) return;
    const DecodeRegs r = make_decode_regs<CB>();

    uint32_t pairs[16];
    decode_slice<K, CB>(trellis, tiles_n, kt, nt_off + chunk * 8, lane, pairs, r);

    uint16_t* s16 = (uint16_t*) &sh[wave][0][0];
    const int j = lane & 7, tcol = (lane >> 3) * 16;
    #pragma unroll
    for (int q = 0; q < 16; ++q)
    {
        const int c = tcol + pair_col(j, q), row = pair_row(q);
        s16[row * 136 + c] = (uint16_t) pairs[q];
        s16[(row + 1) * 136 + c] = (uint16_t)(pairs[q] >> 16);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    // 4 stores of 64 lanes x 16 bytes: lane -> row (4i + lane/16), 8 halves at (lane%16)*8
    #pragma unroll
    for (int i = 0; i < 4; ++i)
    {
        const int row = 4 * i + (lane >> 4), c8 = (lane & 15) * 8;
        u32x4 v = *(const u32x4*) (s16 + row * 136 + c8);
        *(u32x4*) (W + (size_t) (kt * 16 + row) * n + chunk * 128 + c8) = v;
    }
}

// ---------------------------------------------------------------------------- reconstruct_t
// W_hat transposed, (n, k) row-major: the layout the recon GEMM reads fastest (both operands
// k-contiguous).  Same grid as reconstruct_kernel: wave w decodes k-slice 4 blockIdx.y + w of the
// chunk; lane (tile t, j) holds the 16 rows of columns j and j + 8 of its tile, i.e. 32-byte runs
// of two transposed rows.  The workgroup's 128 columns x 64 k meet in LDS and leave as whole
// 128-byte lines (8 threads per transposed row).
//
// With svh (the rotated branch of the recon GEMM), every k row of the tile is then rotated
// across its 128 columns and scaled: W' = W_hat H128 diag(svh) / sqrt(128), fp32 butterflies from
// the fp16 weights, one fp16 rounding.  y = had(x o suh) @ W' then needs no output rotation.
template <int K, int CB>
__global__ __launch_bounds__(256)
void reconstruct_t_kernel(uint16_t* __restrict__ WT, const uint16_t* __restrict__ trellis,
                          int k, int tiles_n, int nt_off, const uint16_t* __restrict__ svh, int slabs)
{
    __shared__ __align__(16) uint32_t sh[128][32 + 4];    // [column][64 k as 32 pairs] (+pad)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int kt = blockIdx.y * 4 + wave;
    const int chunk = blockIdx.x;
    const int nks = min(4, k / 16 - blockIdx.y * 4);     // k-slices of this workgroup
    if (wave < nks)
    {
        const DecodeRegs r = make_decode_regs<CB>();
        uint32_t p[16];
        decode_slice<K, CB>(trellis, tiles_n, kt, nt_off + chunk * 8, lane, p, r);
        // pair q holds rows pair_row(q), +1 of column pair_col(j, q): column j = pairs 0,4,8,12
        // (rows 0-7) and 1,5,9,13 (rows 8-15); column j + 8 = pairs 2,6,10,14 and 3,7,11,15
        const int ca = (lane >> 3) * 16 + (lane & 7);
        *(u32x4*) &sh[ca][8 * wave] = (u32x4) { p[0], p[4], p[8], p[12] };
        *(u32x4*) &sh[ca][8 * wave + 4] = (u32x4) { p[1], p[5], p[9], p[13] };
        *(u32x4*) &sh[ca + 8][8 * wave] = (u32x4) { p[2], p[6], p[10], p[14] };
        *(u32x4*) &sh[ca + 8][8 * wave + 4] = (u32x4) { p[3], p[7], p[11], p[15] };
    }
    __syncthreads();
    if (svh)
    {
        // wave w: k pairs 8 w .. 8 w + 7; lane l holds columns 2 l, 2 l + 1 (the GEMV output layout)
        const f16x2 sv = as_h2(*to_global((const uint32_t*) (svh + chunk * 128 + 2 * lane)));
        const float s0 = (float) sv.x * EXL3_HAD_RSCALE, s1 = (float) sv.y * EXL3_HAD_RSCALE;
        #pragma unroll 2
        for (int q = 0; q < 8; ++q)
        {
            const int pr = 8 * wave + q;
            const f16x2 a = as_h2(sh[2 * lane][pr]), b = as_h2(sh[2 * lane + 1][pr]);
            float a0 = (float) a.x, b0 = (float) b.x, a1 = (float) a.y, b1 = (float) b.y;
            fwht128_wave(a0, b0, lane);
            fwht128_wave(a1, b1, lane);
            sh[2 * lane][pr] = as_u32((f16x2) { (f16) (a0 * s0), (f16) (a1 * s0) });
            sh[2 * lane + 1][pr] = as_u32((f16x2) { (f16) (b0 * s1), (f16) (b1 * s1) });
        }
        __syncthreads();
    }
    // 128 rows x (nks x 32 bytes): thread t writes 16-byte piece t % 8 of rows t / 8 + 32 i
    const int piece = threadIdx.x & 7;
    if (piece < 2 * nks)
    {
        #pragma unroll
        for (int i = 0; i < 4; ++i)
        {
            const int row = (threadIdx.x >> 3) + 32 * i;
            const u32x4 v = *(const u32x4*) &sh[row][4 * piece];
            const int kk = blockIdx.y * 64 + 8 * piece;
            // k slabs ([k / 32][n][32], n = gridDim.x * 128) or row-major (n, k)
            const size_t o = slabs ? (size_t) (kk >> 5) * gridDim.x * 128 * 32 + (size_t) (chunk * 128 + row) * 32 + (kk & 31)
                                   : (size_t) (chunk * 128 + row) * k + kk;
            *to_global_w((u32x4*) (WT + o)) = v;
        }
    }
}

// -------------------------------------------------------------------------- reconstruct_had
// One 128x128 block per workgroup.  LDS holds the block as 128 rows x 64 dwords with the
// dword index of (row R, column pair cp) swizzled to cp ^ (2 * ((R >> 2) & 31)): conflict-free
// for the column pass (16 column pairs x 4 rows, 32 apart) and 8-byte aligned and conflict-free for
// the row pass (rows 4 apart x 4 column ranges).
//
// VALU- and LDS-bound (the 2.5 bytes a weight read and written would take 115 us at 8192 x 28672, 4 bits).  A lane holds 32 values of its column pair or row, so that three of the five fp16 stages
// stay in its registers and two are quad DPP; with 4 values a lane all five went through the LDS
// crossbar: 216 -> 182 us at that size (whole 2048-row product 1007 -> 980).
__device__ __forceinline__ int rh_dw(int R, int cp) { return R * 64 + (cp ^ (((R >> 2) & 31) << 1)); }


// fp16 stage between quad lanes xor M (1, 2): lower lane a + b, upper a - b, as one v_pk_fma_f16 with a
// +-1 factor (exactly v + p or p - v, one rounding).
template <int M>
__device__ __forceinline__ f16x2 had_h2_quad(f16x2 v, int lane)
{
    const f16x2 p = as_h2(__builtin_bit_cast(uint32_t, xor_partner<M>(__builtin_bit_cast(float, as_u32(v)), lane)));
    const f16 sg = (lane & M) ? (f16) -1.0f : (f16) 1.0f;
    const f16x2 sg2 = { sg, sg };
    return __builtin_elementwise_fma(v, sg2, p);
}

// fp16 stage between elements i and i + W of N, in place.
template <int W, int N>
__device__ __forceinline__ void had_h2_inlane(f16x2 (&v)[N])
{
    #pragma unroll
    for (int i = 0; i < N; ++i)
    {
        if (i & W) continue;
        const f16x2 a = v[i], b = v[i + W];
        v[i] = a + b;
        v[i + W] = a - b;
    }
}

// TR: write the block transposed, WT (n, k) row-major (the layout the recon route's dense GEMM
// reads): the row pass leaves its fp16 results in LDS, then each wave stores whole 128-element
// columns.  The values are those of the (k, n) form, bit for bit.
template <int K, int CB, bool TR>
__global__ __launch_bounds__(256)
void reconstruct_had_kernel(uint16_t* __restrict__ W, const uint16_t* __restrict__ trellis,
                            const uint16_t* __restrict__ suh, const uint16_t* __restrict__ svh,
                            int n, int tiles_n, int nt_off, int k, int slabs)
{
    __shared__ __align__(16) uint32_t blk[128 * 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nb = blockIdx.x, kb = blockIdx.y;
    const DecodeRegs r = make_decode_regs<CB>();
    uint16_t* b16 = (uint16_t*) blk;

    // 1. decode 8 k-slices x 8 tiles (wave w: slices w, w + 4)
    #pragma unroll
    for (int it = 0; it < 2; ++it)
    {
        const int js = wave + 4 * it;
        uint32_t pairs[16];
        decode_slice<K, CB>(trellis, tiles_n, kb * 8 + js, nt_off + nb * 8, lane, pairs, r);
        const int j = lane & 7, tcol = (lane >> 3) * 16;
        #pragma unroll
        for (int q = 0; q < 16; ++q)
        {
            const int c = tcol + pair_col(j, q), R = js * 16 + pair_row(q);
            b16[rh_dw(R, c >> 1) * 2 + (c & 1)] = (uint16_t) pairs[q];
            b16[rh_dw(R + 1, c >> 1) * 2 + (c & 1)] = (uint16_t)(pairs[q] >> 16);
        }
    }
    __syncthreads();

    const f16x2 rs2 = { (f16) 0.08838834764831845f, (f16) 0.08838834764831845f };
    const int qd = lane & 3, q16 = lane >> 2;

    // 2. column pass (reconstruct.cu:290-325): rows 32 qd .. + 31 of column pair 16 wave + q16 in a lane, so
    //    that three of the five fp16 stages (strides 4 .. 64 rows) stay in the lane and the last two are
    //    quad DPP; fp16 4-point stage, times rs, fp16 stages.  The swizzle spreads the wave's reads of a
    //    row offset over all banks.
    {
        const int cp = 16 * wave + q16;
        f16x2 v[32];
        #pragma unroll
        for (int i = 0; i < 32; ++i) v[i] = as_h2(blk[rh_dw(32 * qd + i, cp)]);
        #pragma unroll
        for (int i = 0; i < 32; i += 4)
        {
            const f16x2 s0 = v[i] + v[i + 1], d0 = v[i] - v[i + 1];
            const f16x2 s1 = v[i + 2] + v[i + 3], d1 = v[i + 2] - v[i + 3];
            v[i] = (s0 + s1) * rs2;
            v[i + 1] = (d0 + d1) * rs2;
            v[i + 2] = (s0 - s1) * rs2;
            v[i + 3] = (d0 - d1) * rs2;
        }
        had_h2_inlane<4>(v);
        had_h2_inlane<8>(v);
        had_h2_inlane<16>(v);
        #pragma unroll
        for (int i = 0; i < 32; ++i) v[i] = had_h2_quad<1>(v[i], lane);
        #pragma unroll
        for (int i = 0; i < 32; ++i) v[i] = had_h2_quad<2>(v[i], lane);
        #pragma unroll
        for (int i = 0; i < 32; ++i) blk[rh_dw(32 * qd + i, cp)] = as_u32(v[i]);
    }
    __syncthreads();

    // 3. row pass (reconstruct.cu:331-357): columns 32 qd .. + 31 of row 64 it + 4 q16 + wave in a lane (as
    //    above; rows 4 apart, for the banks); fp32 4-point stage, round, times rs in fp16, fp16 stages,
    //    * suh * svh, back in place
    uint32_t sv[16];
    #pragma unroll
    for (int j = 0; j < 16; ++j) sv[j] = ((const uint32_t*) svh)[nb * 64 + 16 * qd + j];
    #pragma unroll
    for (int it = 0; it < 2; ++it)
    {
        const int R = 64 * it + 4 * q16 + wave;
        f16x2 h[16];
        #pragma unroll
        for (int j = 0; j < 16; j += 2)
        {
            const u32x2 w = *(const u32x2*) &blk[rh_dw(R, 16 * qd + j)];
            const f16x2 a = as_h2(w.x), b = as_h2(w.y);
            float v0 = (float) a.x, v1 = (float) a.y, v2 = (float) b.x, v3 = (float) b.y;
            float s0 = v0 + v1, d0 = v0 - v1, s1 = v2 + v3, d1 = v2 - v3;
            f16x2 h01 = { (f16) (s0 + s1), (f16) (d0 + d1) };
            f16x2 h23 = { (f16) (s0 - s1), (f16) (d0 - d1) };
            h[j] = h01 * rs2;
            h[j + 1] = h23 * rs2;
        }
        had_h2_inlane<2>(h);
        had_h2_inlane<4>(h);
        had_h2_inlane<8>(h);
        #pragma unroll
        for (int j = 0; j < 16; ++j) h[j] = had_h2_quad<1>(h[j], lane);
        #pragma unroll
        for (int j = 0; j < 16; ++j) h[j] = had_h2_quad<2>(h[j], lane);
        const f16 su = as_h(suh[kb * 128 + R]);
        const f16x2 su2 = { su, su };
        #pragma unroll
        for (int j = 0; j < 16; j += 2)
        {
            const f16x2 h01 = (h[j] * su2) * as_h2(sv[j]), h23 = (h[j + 1] * su2) * as_h2(sv[j + 1]);
            *(u32x2*) &blk[rh_dw(R, 16 * qd + j)] = (u32x2) { as_u32(h01), as_u32(h23) };   // this lane's own words
        }
    }
    __syncthreads();
    if constexpr (!TR)
    {
        // 4. store: a half wave per row
        const int t = lane & 31, half = lane >> 5;
        #pragma unroll 4
        for (int it = 0; it < 16; ++it)
        {
            const int R = (wave * 16 + it) * 2 + half;
            *(u32x2*) (W + (size_t) (kb * 128 + R) * n + nb * 128 + 4 * t) = *(const u32x2*) &blk[rh_dw(R, 2 * t)];
        }
    }
    if constexpr (TR)
    {
        // 4. transposed store.  Unit (column quad q, row group g) = columns 4 q .. 4 q + 3 at k rows
        //    8 g .. 8 g + 7 of the block: eight ds_read_b64 (the quad's two column-pair dwords of a
        //    row sit side by side: the swizzle flips even bits only), repacked by v_perm into four
        //    16-byte runs of 8 k, one per column.  Thread t takes units t and t + 256 (g = unit % 16,
        //    so 16 consecutive lanes store one column's 128 k contiguously; with slabs, 4 x 64 bytes).
        #pragma unroll
        for (int u = 0; u < 2; ++u)
        {
            const int unit = threadIdx.x + 256 * u;
            const int q = unit >> 4, g = unit & 15;
            uint32_t lo[8], hi[8];
            #pragma unroll
            for (int i = 0; i < 8; ++i)
            {
                const u32x2 v = *(const u32x2*) &blk[rh_dw(8 * g + i, 2 * q)];
                lo[i] = v.x;                                   // columns 4 q, 4 q + 1
                hi[i] = v.y;                                   // columns 4 q + 2, 4 q + 3
            }
            const int kk = kb * 128 + 8 * g;
            #pragma unroll
            for (int j = 0; j < 4; ++j)
            {
                const uint32_t* src = j < 2 ? lo : hi;
                const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;   // high or low halves
                const u32x4 o = { __builtin_amdgcn_perm(src[1], src[0], sel), __builtin_amdgcn_perm(src[3], src[2], sel),
                                  __builtin_amdgcn_perm(src[5], src[4], sel), __builtin_amdgcn_perm(src[7], src[6], sel) };
                const int c = nb * 128 + 4 * q + j;
                const size_t off = slabs ? (size_t) (kk >> 5) * n * 32 + (size_t) c * 32 + (kk & 31)
                                         : (size_t) c * k + kk;
                *(u32x4*) (W + off) = o;
            }
        }
    }
}

template <int K, int CB>
int launch_reconstruct_t(uint16_t* W, const uint16_t* trellis, int k, int n, int tiles_n,
                         int nt_off, hipStream_t s)
{
    dim3 grid(n / 128, (k / 16 + 3) / 4);
    hipLaunchKernelGGL((reconstruct_kernel<K, CB>), grid, dim3(256), 0, s, W, trellis, k, n, tiles_n, nt_off);
    return (int) hipGetLastError();
}

template <int K, int CB>
int launch_reconstruct_tr(uint16_t* WT, const uint16_t* trellis, int k, int n, int tiles_n,
                          int nt_off, const uint16_t* svh, int slabs, hipStream_t s)
{
    dim3 grid(n / 128, (k / 16 + 3) / 4);
    hipLaunchKernelGGL((reconstruct_t_kernel<K, CB>), grid, dim3(256), 0, s, WT, trellis, k, tiles_n, nt_off, svh, slabs);
    return (int) hipGetLastError();
}

template <int K, int CB>
int launch_reconstruct_had_t(uint16_t* W, const uint16_t* trellis, const uint16_t* suh,
                             const uint16_t* svh, int k, int n, int tiles_n, int nt_off,
                             hipStream_t s)
{
    dim3 grid(n / 128, k / 128);
    hipLaunchKernelGGL((reconstruct_had_kernel<K, CB, false>), grid, dim3(256), 0, s, W, trellis, suh, svh, n, tiles_n,
                       nt_off, k, 0);
    return (int) hipGetLastError();
}

template <int K, int CB>
int launch_reconstruct_had_tr(uint16_t* WT, const uint16_t* trellis, const uint16_t* suh,
                              const uint16_t* svh, int k, int n, int tiles_n, int nt_off,
                              int slabs, hipStream_t s)
{
    dim3 grid(n / 128, k / 128);
    hipLaunchKernelGGL((reconstruct_had_kernel<K, CB, true>), grid, dim3(256), 0, s, WT, trellis, suh, svh, n, tiles_n,
                       nt_off, k, slabs);
    return (int) hipGetLastError();
}

}  // namespace

#define EXL3_DISPATCH_K_CB(K, CB, FN, ...)                                        \
    switch (CB * 32 + K)                                                          \
    {                                                                             \
        case 2 * 32 + 17: return FN<17, 2>(__VA_ARGS__);                          \
        case 2 * 32 + 18: return FN<18, 2>(__VA_ARGS__);                          \
        case 2 * 32 + 19: return FN<19, 2>(__VA_ARGS__);                          \
        case 0 * 32 + 1: return FN<1, 0>(__VA_ARGS__);                            \
        case 0 * 32 + 2: return FN<2, 0>(__VA_ARGS__);                            \
        case 0 * 32 + 3: return FN<3, 0>(__VA_ARGS__);                            \
        case 0 * 32 + 4: return FN<4, 0>(__VA_ARGS__);                            \
        case 0 * 32 + 5: return FN<5, 0>(__VA_ARGS__);                            \
        case 0 * 32 + 6: return FN<6, 0>(__VA_ARGS__);                            \
        case 0 * 32 + 7: return FN<7, 0>(__VA_ARGS__);                            \
        case 0 * 32 + 8: return FN<8, 0>(__VA_ARGS__);                            \
        case 1 * 32 + 1: return FN<1, 1>(__VA_ARGS__);                            \
        case 1 * 32 + 2: return FN<2, 1>(__VA_ARGS__);                            \
        case 1 * 32 + 3: return FN<3, 1>(__VA_ARGS__);                            \
        case 1 * 32 + 4: return FN<4, 1>(__VA_ARGS__);                            \
        case 1 * 32 + 5: return FN<5, 1>(__VA_ARGS__);                            \
        case 1 * 32 + 6: return FN<6, 1>(__VA_ARGS__);                            \
        case 1 * 32 + 7: return FN<7, 1>(__VA_ARGS__);                            \
        case 1 * 32 + 8: return FN<8, 1>(__VA_ARGS__);                            \
        case 2 * 32 + 1: return FN<1, 2>(__VA_ARGS__);                            \
        case 2 * 32 + 2: return FN<2, 2>(__VA_ARGS__);                            \
        case 2 * 32 + 3: return FN<3, 2>(__VA_ARGS__);                            \
        case 2 * 32 + 4: return FN<4, 2>(__VA_ARGS__);                            \
        case 2 * 32 + 5: return FN<5, 2>(__VA_ARGS__);                            \
        case 2 * 32 + 6: return FN<6, 2>(__VA_ARGS__);                            \
        case 2 * 32 + 7: return FN<7, 2>(__VA_ARGS__);                            \
        case 2 * 32 + 8: return FN<8, 2>(__VA_ARGS__);                            \
    }                                                                             \
    return -1;

int exl3k_reconstruct(uint16_t* W, const uint16_t* trellis, int k, int n, int tiles_n,
                      int nt_off, int K, int cb, hipStream_t s)
{
    EXL3_DISPATCH_K_CB(K, cb, launch_reconstruct_t, W, trellis, k, n, tiles_n, nt_off, s)
}

int exl3k_reconstruct_had(uint16_t* W, const uint16_t* trellis, const uint16_t* suh,
                          const uint16_t* svh, int k, int n, int tiles_n, int nt_off,
                          int K, int cb, hipStream_t s)
{
    EXL3_DISPATCH_K_CB(K, cb, launch_reconstruct_had_t, W, trellis, suh, svh, k, n, tiles_n, nt_off, s)
}

int exl3k_reconstruct_tr(uint16_t* WT, const uint16_t* trellis, int k, int n, int tiles_n,
                         int nt_off, int K, int cb, const uint16_t* svh, int slabs, hipStream_t s)
{
    EXL3_DISPATCH_K_CB(K, cb, launch_reconstruct_tr, WT, trellis, k, n, tiles_n, nt_off, svh, slabs, s)
}

int exl3k_reconstruct_had_tr(uint16_t* WT, const uint16_t* trellis, const uint16_t* suh,
                             const uint16_t* svh, int k, int n, int tiles_n, int nt_off,
                             int K, int cb, int slabs, hipStream_t s)
{
    EXL3_DISPATCH_K_CB(K, cb, launch_reconstruct_had_tr, WT, trellis, suh, svh, k, n, tiles_n, nt_off, slabs, s)
}
