// Row-tile trellis GEMM for gfx950: C = had(A_rot @ W_hat) o svh for 9 rows up to a few hundred.
//
// Between the GEMV (up to 16 rows, dots of one column per lane) and the 256 x 256 tiles of
// gemm_dma_kernel (which compute 256 rows whatever m is, two waves per SIMD in step) lies the
// batch of a serving engine: tens of rows.  There the decode of the weights (VALU) is the work,
// so each weight is decoded once per row tile of 16 R rows, straight into the registers of a
// matrix operand, and only the row groups that exist are multiplied (there is no instance of 7
// groups: 97 to 112 rows of a tile run as 8).
//
// Work split.  A workgroup owns one 128-column chunk, one row tile and one range of k (split k:
// S ranges per chunk); its 8 waves are 4 column pairs (two 16-column tiles each) x 2 halves of
// the k range.  A unit of work is 64 k x 32 columns per wave: 8 trellis tiles, one per 8 lanes,
// decoded as in the GEMV into 16 packed fp16 pairs per lane (pair q: rows 2 (q >> 2) + 8 (q & 1)
// and the next, column half (q >> 1) & 1).  Matrix operand A (16 columns x 32 k) for column half c
// and row half h is pairs { h, 4 + h, 8 + h, 12 + h } + 2 c; operand B (32 k x 16 rows) is 16
// contiguous bytes of an input row: k 64 u + 16 (lane / 16) + 8 h .. + 7, from LDS.
//
// The rotated rows go from L2 into LDS with buffer_load_dwordx4 ... lds, ROWS_XD units ahead, 8 rows x
// 128 bytes (whole lines) per instruction; lane -> chunk is permuted so that the operand reads
// are conflict-free.  One barrier per unit: it publishes unit u's rows and frees unit u - 1's.
//
// Numerics are the tiled GEMM's: the reference's fp16 weights (3INST / MCG: lo + hi, MUL1: one fma,
// one rounding each), fp32 accumulation, output rotation in fp32.
//
// What bounds it: the decode's VALU instructions (~134 a unit) and the MFMAs, which add up on a SIMD: on
// gfx950 a 16x16x32 MFMA holds the VALU for about two issue slots, from whichever wave.  Of the kernel's
// cycles, fill, reduction and last arrival included, 45 % issue VALU and 14 % are in MFMAs at 33 rows of 17408 ->
// 5120, 36 and 22 % at 100 rows of 4096 -> 14336 (one workgroup a CU: nothing covers its ends).  Hence one
// decode per tile and few spare row groups; interleaving MFMAs with the decode or 4 k quarters per
// workgroup gained nothing.  The trellis loads of two units and the row DMAs of two stay in flight across the
// barrier: the DMAs go through a buffer resource, LDS is one array and half-rate words are shifted when
// used.  With global_load_lds, a second LDS variable and a shift at the load the compiler waited for every
// load once or twice a turn of the buffers.  MI355X, whole calls before / after, us: 32 rows of 17408 ->
// 5120 at 4 / 3.5 bits 34.7 / 28.3 and 35.8 / 27.9, 9 rows of 8192 -> 28672 at 4 bits 66.4 / 48.0 (the GEMV of
// 16-row groups: 62 to 67), 64 rows of 14336 -> 4096 31.8 / 27.8, 96 rows of 4096 -> 14336 34.9 / 31.6.
// gemm_dma_kernel with its split k: 65 us for 33 rows of 17408 -> 5120, 57 for 100 rows of 4096 -> 14336.
//
// Split k: each range stores its fp32 partial rows; the last arrival of a chunk (XCD-local
// hand-off, exl3_xcd.cuh) adds them in k order, four rows in flight per wave, rotates and stores.
// Without the hand-off exl3k_rows_finish does the same in a second launch.
#include "exl3_common.cuh"
#include "exl3_gemv_core.cuh"
#include "exl3_kernels.h"
#include "exl3_xcd.cuh"

#ifndef EXL3_INST_K
#define EXL3_INST_K 4
#endif

using namespace exl3;

namespace {

typedef _Float16 h8v __attribute__((ext_vector_type(8)));

constexpr int ROWS_KW = 2;                     // k halves of a workgroup
constexpr int ROWS_THREADS = 256 * ROWS_KW;
constexpr int ROWS_XNB = 4, ROWS_XD = ROWS_XNB - 1;   // row buffers (units) per k half, units in flight
constexpr int ROWS_PF = 2;                     // trellis units in flight per wave
constexpr int ROWS_RS = 132;                   // fp32 row stride of the reduction buffer

template <int R> struct RowsLds
{
    static constexpr int RT = 16 * R;                             // rows per tile
    static constexpr int X = ROWS_KW * ROWS_XNB * RT * 32;        // staged rows, u32
    static constexpr int RED = (ROWS_KW - 1) * RT * ROWS_RS;
    static constexpr int TOTAL = X > RED ? X : RED;
};

// The lane's 32 windows as 16 packed pairs, eight windows at a time (bounded registers).
template <int K, int CB>
__device__ __forceinline__ void decode_pairs(const uint32_t* wv, uint32_t* pk, uint32_t a3, uint32_t b3)
{
    static_for<0, 4>([&](auto g) {
        constexpr int G = g;
        if constexpr (CB == 2)
        {
            const f16x2 kinv = { as_h(0x1eee), as_h(0x1eee) }, bias = { as_h(0xc931), as_h(0xc931) };
            const uint32_t h[4] = { mul1_pair<K, 4 * G>(wv), mul1_pair<K, 4 * G + 1>(wv), mul1_pair<K, 4 * G + 2>(wv),
                                    mul1_pair<K, 4 * G + 3>(wv) };
            #pragma unroll
            for (int i = 0; i < 4; ++i) pk[4 * G + i] = as_u32(__builtin_elementwise_fma(as_h2(h[i]), kinv, bias));
        }
        else
        {
            uint32_t raw[32];
            raw8<K, CB, 8 * G>(wv, raw, a3, b3);
            sum_pairs4(raw + 8 * G, pk + 4 * G);
        }
        __builtin_amdgcn_sched_barrier(0);
    });
}

// rows_kernel's body (a device function: the host pass knows no buffer resources).
template <int K, int CB, int R>
__device__ __forceinline__ void rows_body(const RowsArgs& g, uint32_t* lds)
{
    using LD = RowsLds<R>;
    constexpr int TWD = tile_words(K), KB = kbits(K), RT = LD::RT, XBUF = RT * 32;
    int* flag = (int*) (lds + LD::TOTAL);
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int cw = wave & 3, kg = wave >> 2;              // column pair, k half
    const int k = g.k, n = g.n, S = g.splits;
    const int blocks = k / 128, tiles_n = n / 16;
    const uint32_t a3 = sconst(89226354u), b3 = vconst(64248484u);
    int chunk, slot;
    gemv_block_coords(g.xcd, S, (int) blockIdx.x, chunk, slot);
    const int row0 = blockIdx.y * RT, M = min(RT, g.m - row0);
    // this range's 128-k blocks [b0, b1): b1 - b0 units of 64 k per k half
    const int b0 = (int) ((long) blocks * slot / S), b1 = (int) ((long) blocks * (slot + 1) / S);
    const int units = b1 - b0, u00 = 2 * b0 + kg * units;
    const uint16_t* A = g.A_rot + (size_t) row0 * k + (size_t) u00 * 64;
    const int jt = lane & 7;
    const uint32_t* tile0 = (const uint32_t*) g.trellis
                          + ((size_t) (u00 * 4 + (lane >> 4)) * tiles_n + chunk * 8 + 2 * cw + ((lane >> 3) & 1)) * TWD;
    const size_t ustride = (size_t) 4 * tiles_n * TWD;
    const int prev_off = jt == 0 ? 8 * KB - 1 : -1;
    uint32_t ring[ROWS_PF][RING_WORDS<K>];

    // Row staging: a unit is 2 R blocks of 8 rows x 128 bytes; wave cw of the k half fills blocks
    // cw, cw + 4, ... (past the last one: the same bytes to the same place, so that every wave
    // issues the same number).  Rows past m repeat row m - 1; their products are never stored.
    // 16-byte chunk c of row r sits at chunk c ^ s(r % 16), s(q) = (q ^ (q >> 3)) & 7 (moeg_kernel's).
    constexpr int ND = (2 * R + 3) / 4;
    uint32_t* xs = lds + kg * (ROWS_XNB * XBUF);
    const __amdgpu_buffer_rsrc_t rows = buffer_of(A, (uint32_t) (2 * ((M - 1) * k + units * 64)));
    uint32_t xoff[ND];
    #pragma unroll
    for (int i = 0; i < ND; ++i)
    {
        const int q = min(cw + 4 * i, 2 * R - 1), row = 8 * q + (lane >> 3), rr = row & 15;
        xoff[i] = (uint32_t) (2 * (min(row, M - 1) * k + 8 * ((lane & 7) ^ ((rr ^ (rr >> 3)) & 7))));
    }
    auto xissue = [&](int u) {
        #pragma unroll
        for (int i = 0; i < ND; ++i)
        {
            const int q = min(cw + 4 * i, 2 * R - 1);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (lds_ptr_t) (xs + (u % ROWS_XNB) * XBUF + 256 * q), 16, xoff[i],
                                                     (uint32_t) (min(u, units - 1) * 128), 0, 0);
        }
    };
    // issue order: rows(0), trellis(0), rows(1), trellis(1), rows(2); then per unit trellis(u + PF), rows(u + XD)
    static_for<0, ROWS_XD>([&](auto d) {
        xissue(d);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (d < ROWS_PF) load_tile_ring<K>(tile0 + (size_t) min((int) d, units - 1) * ustride, jt, prev_off, ring[d]);
        __builtin_amdgcn_sched_barrier(0);
    });

    f32x4 acc[2][R];
    #pragma unroll
    for (int r = 0; r < R; ++r) { acc[0][r] = (f32x4) { }; acc[1][r] = (f32x4) { }; }
    const int xb0 = (lane & 15) * 32 + 4 * ((2 * (lane >> 4)) ^ (((lane & 15) ^ ((lane & 15) >> 3)) & 7));
    for (int u0 = 0; u0 < units; u0 += ROWS_XNB)
    {
        #pragma unroll
        for (int d = 0; d < ROWS_XNB; ++d)
        {
            const int u = u0 + d;
            if (u >= units) break;
            uint32_t pk[16];
            ring_words<K>(ring[d % ROWS_PF], jt);
            decode_pairs<K, CB>(ring[d % ROWS_PF], pk, a3, b3);
            load_tile_ring<K>(tile0 + (size_t) min(u + ROWS_PF, units - 1) * ustride, jt, prev_off, ring[d % ROWS_PF]);
            __builtin_amdgcn_sched_barrier(0);
            // unit u's rows have landed when all but the row loads of units u + 1, u + 2 and the trellis
            // loads issued after unit u's rows are done (loads complete in issue order)
            constexpr int VN = (ROWS_XD - 1) * ND + ROWS_XD * tile_lane_loads(K);
            static_assert(ROWS_PF <= ROWS_XD, "the wait assumes a trellis load between any two units' row loads");
            EXL3_WAIT_VM_LGKM0(VN < 60 ? VN : 60);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            xissue(u + ROWS_XD);                          // into unit u - 1's buffer: every wave is past it
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t* xb = xs + d * XBUF;
            h8v bx[2][R];
            #pragma unroll
            for (int h = 0; h < 2; ++h)
            {
                #pragma unroll
                for (int r = 0; r < R; ++r) bx[h][r] = __builtin_bit_cast(h8v, *(const u32x4*) (xb + 512 * r + (xb0 ^ (4 * h))));
            }
            #pragma unroll
            for (int h = 0; h < 2; ++h)
            {
                #pragma unroll
                for (int r = 0; r < R; ++r)
                {
                    #pragma unroll
                    for (int c = 0; c < 2; ++c)
                    {
                        const u32x4 a = { pk[h + 2 * c], pk[4 + h + 2 * c], pk[8 + h + 2 * c], pk[12 + h + 2 * c] };
                        acc[c][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8v, a), bx[h][r], acc[c][r], 0, 0, 0);
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    EXL3_WAIT_VM_LGKM0(0);                                     // the past-the-end row loads still write LDS
    // the past-the-end trellis loads have to stay: the row waits count them
    #pragma unroll
    for (int d = 0; d < ROWS_PF; ++d)
    {
        #pragma unroll
        for (int w = 0; w < RING_WORDS<K>; ++w) asm volatile("" :: "v"(ring[d][w]));
    }
    __syncthreads();

    // the k halves meet in LDS: D[i][nn] of acc[c][r] (lane: i = 4 (lane / 16) + e, nn = lane % 16) is
    // column 32 cw + 16 (i / 8) + i % 8 + 8 c, row 16 r + nn
    float* red = (float*) lds;
    const int nn = lane & 15, q4 = lane >> 4;
    float* rp = red + nn * ROWS_RS + 32 * cw + 16 * (q4 >> 1) + 4 * (q4 & 1);
    if (kg == 1)
    {
        #pragma unroll
        for (int r = 0; r < R; ++r)
        {
            *(f32x4*) (rp + 16 * r * ROWS_RS) = acc[0][r];
            *(f32x4*) (rp + 16 * r * ROWS_RS + 8) = acc[1][r];
        }
    }
    __syncthreads();
    if (kg == 0)
    {
        #pragma unroll
        for (int r = 0; r < R; ++r)
        {
            #pragma unroll
            for (int c = 0; c < 2; ++c)
            {
                float* p = rp + 16 * r * ROWS_RS + 8 * c;
                *(f32x4*) p = acc[c][r] + *(const f32x4*) p;
            }
        }
    }
    __syncthreads();

    const uint32_t svp = *to_global((const uint32_t*) ((g.svh ? g.svh + chunk * 128 : g.A_rot) + 2 * lane));
    const bool has_svh = g.svh != nullptr;
    const size_t c0 = (size_t) row0 * n + chunk * 128 + 2 * lane;
    constexpr int RW = 4 * ROWS_KW;                       // waves: rows r, r + RW, ... each, 4 in flight
    if (S == 1)
    {
        for (int r0 = wave; r0 < M; r0 += 4 * RW)
        {
            f32x2 v[4];
            #pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = *(const f32x2*) (red + min(r0 + RW * i, M - 1) * ROWS_RS + 2 * lane);
            #pragma unroll
            for (int i = 0; i < 4; ++i)
                if (r0 + RW * i < M) gemm_store(v[i].x, v[i].y, g.C, g.c_fp32, has_svh, svp, c0 + (size_t) (r0 + RW * i) * n, lane);
        }
        return;
    }
    const size_t tile = (size_t) blockIdx.y * (n / 128) + chunk;
    float* pb = g.part + tile * S * (RT * 128);
    for (int e = t; e < M * 32; e += ROWS_THREADS)
        *to_global_w((f32x4*) (pb + (size_t) slot * (RT * 128) + 4 * e)) = *(const f32x4*) (red + (e >> 5) * ROWS_RS + 4 * (e & 31));
    if (!g.xcd) return;                                   // exl3k_rows_finish sums the ranges
    // the stores reach the XCD's L2 before the counter moves (exl3_xcd.cuh; arrive_last of the GEMV)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    if (t == 0) *flag = xcd_arrive(g.xg, g.ctr + tile * 32, S);
    __syncthreads();
    if (!*flag) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    for (int r0 = wave; r0 < M; r0 += 4 * RW)
    {
        float s0[4] = { 0.0f, 0.0f, 0.0f, 0.0f }, s1[4] = { 0.0f, 0.0f, 0.0f, 0.0f };
        for (int p0 = 0; p0 < S; p0 += 4)
        {
            f32x2 v[4][4];
            #pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                #pragma unroll
                for (int q = 0; q < 4; ++q)
                    v[i][q] = load_l2_f32x2(pb + (size_t) min(p0 + q, S - 1) * (RT * 128) + min(r0 + RW * i, M - 1) * 128 + 2 * lane);
            }
            #pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                #pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (p0 + q < S) { s0[i] += v[i][q].x; s1[i] += v[i][q].y; }
            }
        }
        #pragma unroll
        for (int i = 0; i < 4; ++i)
            if (r0 + RW * i < M) gemm_store(s0[i], s1[i], g.C, g.c_fp32, has_svh, svp, c0 + (size_t) (r0 + RW * i) * n, lane);
    }
}

template <int K, int CB, int R>
__global__ __launch_bounds__(ROWS_THREADS)
__attribute__((amdgpu_waves_per_eu(R <= 4 ? 4 : 2, R <= 4 ? 4 : 2)))
void rows_kernel(const RowsArgs g)
{
    // one array: with a second LDS variable in the kernel the compiler tracks the DMAs into this one and waits
    // for all of them (vmcnt(0)) before any read of it; the unit loop's own waits are what orders them
    __shared__ __align__(16) uint32_t lds[RowsLds<R>::TOTAL + 4];
    rows_body<K, CB, R>(g, lds);
}

template <int K, int CB, int R>
int launch_rows_r(const RowsArgs& g, hipStream_t s)
{
    const int nt = (g.m + 16 * R - 1) / (16 * R);
    hipLaunchKernelGGL((rows_kernel<K, CB, R>), dim3(g.splits * (g.n / 128), nt), dim3(ROWS_THREADS), 0, s, g);
    if (int rc = (int) hipGetLastError()) return rc;
    return g.splits > 1 && !g.xcd ? exl3k_rows_finish(g, s) : 0;
}

template <int K, int CB>
int launch_rows(const RowsArgs& g, hipStream_t s)
{
    switch (g.groups)
    {
        case 1: return launch_rows_r<K, CB, 1>(g, s);
        case 2: return launch_rows_r<K, CB, 2>(g, s);
        case 3: return launch_rows_r<K, CB, 3>(g, s);
        case 4: return launch_rows_r<K, CB, 4>(g, s);
        case 5: return launch_rows_r<K, CB, 5>(g, s);
        case 6: return launch_rows_r<K, CB, 6>(g, s);
        case 8: return launch_rows_r<K, CB, 8>(g, s);
    }
    return -1;
}

}  // namespace

#define EXL3_CAT2(a, b) a##b
#define EXL3_CAT(a, b) EXL3_CAT2(a, b)

int EXL3_CAT(exl3k_rows_k, EXL3_INST_K)(const RowsArgs& g, int cb, hipStream_t s)
{
#if EXL3_INST_K >= 16
    return cb == 2 ? launch_rows<EXL3_INST_K, 2>(g, s) : -1;       // half rates: mul1 only
#else
    switch (cb)
    {
        case 0: return launch_rows<EXL3_INST_K, 0>(g, s);
        case 1: return launch_rows<EXL3_INST_K, 1>(g, s);
        case 2: return launch_rows<EXL3_INST_K, 2>(g, s);
    }
    return -1;
#endif
}
