// Register-decode grouped GEMM of the token-sorted MoE (exl3_moe_sorted.hip): one launch per phase
// runs the row tiles of every expert at every bitrate.
//
// The row tiles hold few rows (T * topk / experts: 16 at T = 512, 64 at T = 2048), so the weight
// decode, not the matrix pipe, bounds these GEMMs.  Here every weight is decoded once per row tile
// straight into MFMA operand registers (no LDS round trip and no barrier for the weights), and each
// decoded fragment feeds one v_mfma_f32_16x16x32_f16 per 16-row group of the tile.
//
// Work item = (row tile, matrix, 128-column chunk); a workgroup of 4 waves owns the chunk, wave w
// the column tiles 2w, 2w+1.  Per unit of 4 k-tiles (64 k) lane l decodes tile (k-tile l/16,
// column tile 2w + (l%16)/8) at position j = l%8 -- columns j and j+8, all 16 rows -- into 16
// packed fp16 pairs (pair q: rows 2(q>>2) + 8(q&1) + {0,1}, column half (q>>1)&1).  Operand A
// (16 columns x 32 k) for column half c and row half h is lane l's rows 8h..8h+7 of its column,
// pairs {h+2c, 4+h+2c, 8+h+2c, 12+h+2c}, in natural k order; operand B (32 k x 16 rows) is, for
// lane l, row l%16 of the group at k = 64u + 16(l/16) + 8h .. +7: 16 contiguous bytes in LDS.
//
// MUL1 weights enter as h = 1024 + byte sum, the decode's exact fp16 value, and the codebook's
// affine map is applied to the sums: y = kinv sum(h x) + bias sum(x) (codebook.cuh:78-84), with
// sum(x) from the 128-chunk sums the staging kernels write beside the rows (psum, added in a
// fixed order).  MCG weights are the reference's fp16 lo + hi (one rounding).
//
// The rows go from L2 into LDS with buffer_load_dwordx4 ... lds, MG_XD units ahead; one barrier per
// unit publishes its rows and frees the previous unit's.
//
// One launch takes every bitrate: the item finds its list (and so its rate) on the device, and the
// body is a switch over the rates.  Items run persistently and XCD-aware: the workgroups of XCD x
// (blockIdx % 8) take the (row tile, matrix) entries e with e % 8 == x, so all chunks of an entry
// share one L2.  Measured on MI355X against one launch per possible bitrate (8 with rate tables, most
// of them without an entry, each with a tail of its own), mul1 at 2, 3 and 4 bits, whole calls: 16
// experts 3072 -> 1024, 300 tokens, top-2: 210 -> 91 us; 64 experts 2048 -> 1536, 512 tokens, top-4: 269 ->
// 158; 128 experts 2048 -> 768, 4096 tokens, top-8: 989 -> 750; 256 experts 4096 -> 2048, top-8:
// 2048 tokens 1806 -> 1462, 1024 tokens 1244 -> 1067, 512 tokens 985 -> 931.  At one rate, where that was
// one launch too: 64 experts 2048 -> 1536, 512 tokens, at 4 / 2.5 bits 173 -> 160 / 171 -> 157.
//
// The trellis loads of two units and the row DMAs of two stay in flight across the barrier.  That takes DMAs
// through a buffer resource, a single LDS array and half-rate words that are shifted when they are used;
// with global_load_lds, several LDS variables and a shift at the load the compiler waited for everything
// once a unit, and at one rate the calls took 8 to 28 % longer at 2.5 bits, up to 34 % with few experts.
//
// What bounds it: the issue slots.  A unit is 96 VALU instructions of decode (bfe, mul, sad a weight)
// per 10 MFMAs at 40 rows; of the cycles 81 % issue VALU and 17 % are in MFMAs at 512 tokens (256 experts 4096 ->
// 2048, 32-row tiles), 67 and 41 % at 2048 (96-row tiles), and the two mostly add up.  So the products are
// made for the row groups that exist only (all four groups of a 64-row tile always: 1.40 against 1.26 ms
// at 1024 tokens, before the waits above).
#include "exl3_common.cuh"
#include "exl3_gemv_core.cuh"
#include "exl3_kernels.h"

#ifndef EXL3_MOEG_CB
#define EXL3_MOEG_CB 2
#endif
#ifndef EXL3_MOEG_R
#define EXL3_MOEG_R 4
#endif

using namespace exl3;

namespace {

typedef _Float16 h8v __attribute__((ext_vector_type(8)));

constexpr int MG_PF = 2;                       // trellis ring depth (units)
constexpr int MG_XNB = 4, MG_XD = MG_XNB - 1;  // row buffers (units), units in flight
constexpr int MG_THREADS = 256;

template <int R> struct MgLds
{
    static constexpr int RT = 16 * R;                   // rows per tile
    static constexpr int XBUF = RT * 32;                // staged rows of one unit
    static constexpr int TOTAL = MG_XNB * XBUF;         // also holds the item's RT x 128 fp32 sums
};

// Waves per SIMD of an instance, which is also its workgroups per CU.
constexpr int moeg_waves(int R) { return R <= 2 ? 5 : (R <= 4 ? 4 : (R <= 6 ? 3 : 2)); }

// The pairs of row half H: pk[4 c + i] is pair 4 i + H + 2 c (four at a time: bounded registers).
template <int K, int CB, int H>
__device__ __forceinline__ void moeg_pairs(const uint32_t* wv, uint32_t* pk)
{
    static_for<0, 2>([&](auto c) {
        constexpr int Q = H + 2 * c;
        if constexpr (CB == 2) static_for<0, 4>([&](auto i) { pk[4 * c + i] = mul1_pair<K, 4 * i + Q>(wv); });
        else
        {
            uint32_t raw[8];
            static_for<0, 4>([&](auto i) {
                raw[2 * i] = raw_at<K, CB, 2 * (4 * i + Q)>(wv);
                raw[2 * i + 1] = raw_at<K, CB, 2 * (4 * i + Q) + 1>(wv);
            });
            sum_pairs4(raw, pk + 4 * c);
        }
        __builtin_amdgcn_sched_barrier(0);
    });
}

// The sums of one item (M rows of A at row stride k, one 128-column chunk of a trellis with tiles_n
// column tiles) into LDS: RT rows x 128 columns, 4-column group c of row r at group c ^ (r % 16).  They leave
// the registers here: accumulators that live on past the switch over the rates cost copies and spills.
// G: the 16-row groups that are staged and multiplied, at least the item's.
template <int K, int CB, int R, int G>
__device__ __forceinline__ void moeg_sums(const uint16_t* A, int M, int k, int tiles_n, const uint32_t* trellis,
                                          int chunk, uint32_t* lds)
{
    constexpr int TWD = tile_words(K), KB = kbits(K), XBUF = MgLds<R>::XBUF, PF = MG_PF;
    // opaque: the rates' offsets are worked out per item, not all kept across the item loop
    int t = threadIdx.x;
    asm volatile("" : "+v"(t), "+s"(k), "+s"(tiles_n));
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int units = k / 64;
    const int jt = lane & 7;
    const uint32_t* tile0 = trellis + ((size_t) (lane >> 4) * tiles_n + chunk * 8 + 2 * wave + ((lane >> 3) & 1)) * TWD;
    const size_t ustride = (size_t) 4 * tiles_n * TWD;
    const int prev_off = jt == 0 ? 8 * KB - 1 : -1;
    uint32_t ring[PF][RING_WORDS<K>];

    // Row staging: a unit is 2 G blocks of 8 rows x 128 bytes; wave w fills blocks w, w + 4, ... (past the
    // last one: the same bytes to the same place, so that every wave issues the same number).  Rows
    // past M repeat row M - 1; their products are never stored.  16-byte chunk c of row r sits at
    // chunk c ^ s(r % 16), s(q) = (q ^ (q >> 3)) & 7: no bank conflicts for the operand reads.
    constexpr int ND = (2 * G + 3) / 4;
    const __amdgpu_buffer_rsrc_t rows = buffer_of(A, (uint32_t) (M * k * 2));
    uint32_t xoff[ND];
    #pragma unroll
    for (int i = 0; i < ND; ++i)
    {
        const int q = min(wave + 4 * i, 2 * G - 1), row = 8 * q + (lane >> 3), rr = row & 15;
        xoff[i] = (uint32_t) (2 * (min(row, M - 1) * k + 8 * ((lane & 7) ^ ((rr ^ (rr >> 3)) & 7))));
    }
    auto xissue = [&](int u) {
        #pragma unroll
        for (int i = 0; i < ND; ++i)
        {
            const int q = min(wave + 4 * i, 2 * G - 1);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (lds_ptr_t) (lds + (u % MG_XNB) * XBUF + 256 * q), 16, xoff[i],
                                                     (uint32_t) (min(u, units - 1) * 128), 0, 0);
        }
    };
    // issue order: rows(0), trellis(0), rows(1), trellis(1), ...; then per unit rows(u + XD), trellis(u + PF)
    static_for<0, (PF > MG_XD ? PF : MG_XD)>([&](auto d) {
        if constexpr (d < MG_XD) xissue(d);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (d < PF) load_tile_ring<K>(tile0 + (size_t) min((int) d, units - 1) * ustride, jt, prev_off, ring[d]);
        __builtin_amdgcn_sched_barrier(0);
    });
    f32x4 acc[2][G];
    #pragma unroll
    for (int r = 0; r < G; ++r) { acc[0][r] = (f32x4) { }; acc[1][r] = (f32x4) { }; }
    const int xb0 = (lane & 15) * 32 + 4 * ((2 * (lane >> 4)) ^ (((lane & 15) ^ ((lane & 15) >> 3)) & 7));
    // unit u, u % 4 = d
    auto unit = [&](int u, auto dd) {
        constexpr int d = dd;
        // unit u's rows have landed when all but the row loads of units u + 1, u + 2 and the trellis
        // loads issued after unit u's rows, min(PF, XD) or more, are done (loads complete in issue order)
        constexpr int VN = (MG_XD - 1) * ND + (PF < MG_XD ? PF : MG_XD) * tile_lane_loads(K);
        EXL3_WAIT_VM_LGKM0(VN < 60 ? VN : 60);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        xissue(u + MG_XD);                            // into unit u - 1's buffer: every wave is past it
        // a row half at a time (registers): its row operands first (their LDS latency hides behind the
        // decode), its pairs, its products
        const uint32_t* xs = lds + d * XBUF;
        ring_words<K>(ring[d % PF], jt);
        static_for<0, 2>([&](auto hh) {
            constexpr int h = hh;
            h8v bx[G];
            #pragma unroll
            for (int r = 0; r < G; ++r) bx[r] = __builtin_bit_cast(h8v, *(const u32x4*) (xs + 512 * r + (xb0 ^ (4 * h))));
            __builtin_amdgcn_sched_barrier(0);
            uint32_t pk[8];
            moeg_pairs<K, CB, h>(ring[d % PF], pk);
            if constexpr (h == 1)
                load_tile_ring<K>(tile0 + (size_t) min(u + PF, units - 1) * ustride, jt, prev_off, ring[d % PF]);
            __builtin_amdgcn_sched_barrier(0);
            #pragma unroll
            for (int r = 0; r < G; ++r)
            {
                #pragma unroll
                for (int c = 0; c < 2; ++c)
                {
                    const u32x4 a = { pk[4 * c], pk[4 * c + 1], pk[4 * c + 2], pk[4 * c + 3] };
                    acc[c][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8v, a), bx[r], acc[c][r], 0, 0, 0);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    static_assert(MG_XNB == 4 && 4 % PF == 0, "buffer and ring slots are compile-time functions of d");
    int u = 0;
    for (; u + 4 <= units; u += 4) static_for<0, 4>([&](auto d) { unit(u + d, d); });
    if (u < units) static_for<0, 2>([&](auto d) { unit(u + d, d); });      // (units is even)
    EXL3_WAIT_VM_LGKM0(0);                                // the past-the-end row loads still write LDS
    // the past-the-end trellis loads have to stay: the row waits count them
    #pragma unroll
    for (int d = 0; d < PF; ++d)
    {
        #pragma unroll
        for (int w = 0; w < RING_WORDS<K>; ++w) asm volatile("" :: "v"(ring[d][w]));
    }
    __syncthreads();
    // D[i][nn] of acc[c][r] (lane: i = 4 (lane / 16) + e, nn = lane % 16) is column
    // 32 w + 16 (i / 8) + i % 8 + 8 c, row 16 r + nn
    const int nn = lane & 15, cg = 8 * wave + 4 * (lane >> 5) + ((lane >> 4) & 1);
    #pragma unroll
    for (int r = 0; r < G; ++r)
    {
        #pragma unroll
        for (int c = 0; c < 2; ++c) *(f32x4*) (lds + (16 * r + nn) * 128 + 4 * ((cg + 2 * c) ^ nn)) = acc[c][r];
    }
}

// The instance for the item's row groups: 1, 2 of 2; 2, 3, 4 of 4; 4, 6 of 6; 6, 8 of 8 (each is a copy of the
// loop, and a product costs two VALU slots where a unit's decode costs about 100).
template <int K, int CB, int R>
__device__ __forceinline__ void moeg_sums_rows(const uint16_t* A, int M, int k, int tiles_n, const uint32_t* trellis,
                                               int chunk, uint32_t* lds)
{
    constexpr int G0 = R == 2 ? 1 : (R == 4 ? 2 : R - 2);
    if (M <= 16 * G0) moeg_sums<K, CB, R, G0>(A, M, k, tiles_n, trellis, chunk, lds);
    else if (R == 4 && M <= 48) moeg_sums<K, CB, R, (R == 4 ? 3 : R)>(A, M, k, tiles_n, trellis, chunk, lds);
    else moeg_sums<K, CB, R, R>(A, M, k, tiles_n, trellis, chunk, lds);
}

template <int CB, int R>
__global__ __launch_bounds__(MG_THREADS)
__attribute__((amdgpu_waves_per_eu(moeg_waves(R), moeg_waves(R))))
void moeg_kernel(const MoegArgs g)
{
    using LD = MgLds<R>;
    // one array: with a second LDS variable in the kernel the compiler tracks the DMAs into this one and waits
    // for all of them (vmcnt(0)) before any read of it; the unit loop's own waits are what orders them
    __shared__ __align__(16) uint32_t lds[LD::TOTAL + 64 + LD::RT];
    int* ends = (int*) (lds + LD::TOTAL);
    float* sumx = (float*) (lds + LD::TOTAL + 64);
    const int t = threadIdx.x, lane = t & 63;
    const int k = g.k, n = g.n;
    const int nch = n / 128;
    // ends[32 m + s]: entries of matrix m in the lists of slots slots - 1 .. slots - 1 - s
    if (t < 64)
    {
        const int m = t >> 5, s = t & 31;
        int v = 0;
        if (m < g.mats && s < g.slots) v = *to_global((m ? g.count[1] : g.count[0]) + (g.slots - 1 - s));
        #pragma unroll
        for (int o = 1; o < 16; o <<= 1)
        {
            const int u = __shfl_up(v, o, 32);
            if (s >= o) v += u;
        }
        ends[t] = v;
    }
    __syncthreads();
    const int tot0 = __builtin_amdgcn_readfirstlane(ends[15]), tot1 = __builtin_amdgcn_readfirstlane(ends[47]);
    const int ents = max(tot0, tot1) * g.mats;
    const int xcd = blockIdx.x & 7, lb = blockIdx.x >> 3, nlb = gridDim.x >> 3;
    const int per_xcd = ents > xcd ? (ents - xcd + 7) / 8 : 0;

    for (int it = lb; it < per_xcd * nch; it += nlb)
    {
        const int ent = xcd + 8 * (it / nch), chunk = it % nch;
        const int mat = ent % g.mats, pos = ent / g.mats;
        if (pos >= (mat ? tot1 : tot0)) continue;
        // the list that holds entry pos: the number of lists that end at or before it
        const uint64_t before = __ballot(ends[lane] <= pos) & (0xffffull << (32 * mat));
        const int s = __builtin_popcountll(before), slot = g.slots - 1 - s;
        const int li = pos - (s ? __builtin_amdgcn_readfirstlane(ends[32 * mat + s - 1]) : 0);
        const int tid = *to_global((mat ? g.list[1] : g.list[0]) + (size_t) slot * g.list_stride + li);
        const int e = *to_global(g.rt + 3 * tid);
        const int row0 = __builtin_amdgcn_readfirstlane(*to_global(g.rt + 3 * tid + 1));
        const int M = __builtin_amdgcn_readfirstlane(*to_global(g.rt + 3 * tid + 2));
        const uint16_t* A = (mat ? g.A[1] : g.A[0]) + (size_t) row0 * k;
        uint16_t* C = (mat ? g.C[1] : g.C[0]) + (size_t) row0 * n + chunk * 128;
        const uint32_t* trellis = (const uint32_t*) *to_global((mat ? g.tab[1] : g.tab[0]) + e);
        if constexpr (CB == 2)
        {
            // sum(x) of every row from its 128-chunk sums: 4 lanes a row, lane q adds chunks q, q + 4, ...,
            // then 0 + 1 and 2 + 3, then the pairs
            const int kc = k / 128, q4 = t & 3;
            const float* ps = (mat ? g.psum[1] : g.psum[0]) + (size_t) row0 * kc;
            for (int r = t >> 2; r < M; r += MG_THREADS / 4)
            {
                const float* pr = ps + (size_t) r * kc;
                float sx = 0.0f;
                for (int c0 = 0; c0 < kc; c0 += 32)
                {
                    float v[8];
                    #pragma unroll
                    for (int i = 0; i < 8; ++i) v[i] = *to_global(pr + min(c0 + 4 * i + q4, kc - 1));
                    #pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (c0 + 4 * i + q4 < kc) sx += v[i];
                }
                sx += __shfl_xor(sx, 1, 64);
                sx += __shfl_xor(sx, 2, 64);
                if (q4 == 0) sumx[r] = sx * (float) as_h(0xc931);
            }
        }
#define EXL3_MOEG_RATE(K) moeg_sums_rows<K, CB, R>(A, M, k, n / 16, trellis, chunk, lds)
        switch (slot)
        {
            case 0: EXL3_MOEG_RATE(1); break;
            case 1: EXL3_MOEG_RATE(2); break;
            case 2: EXL3_MOEG_RATE(3); break;
            case 3: EXL3_MOEG_RATE(4); break;
            case 4: EXL3_MOEG_RATE(5); break;
            case 5: EXL3_MOEG_RATE(6); break;
            case 6: EXL3_MOEG_RATE(7); break;
            case 7: EXL3_MOEG_RATE(8); break;
            default:
                if constexpr (CB == 2)                    // the half rates exist for mul1 only
                {
                    if (slot == 8) EXL3_MOEG_RATE(17);
                    else if (slot == 9) EXL3_MOEG_RATE(18);
                    else EXL3_MOEG_RATE(19);
                }
        }
#undef EXL3_MOEG_RATE
        __syncthreads();

        for (int q = t; q < M * 16; q += MG_THREADS)
        {
            const int row = q >> 4, part = q & 15;
            const float* p = (const float*) lds + row * 128;
            const f32x4 v0 = *(const f32x4*) (p + 4 * ((2 * part) ^ (row & 15)));
            const f32x4 v1 = *(const f32x4*) (p + 4 * ((2 * part + 1) ^ (row & 15)));
            const float sx = CB == 2 ? sumx[row] : 0.0f;
            uint32_t o[4];
            #pragma unroll
            for (int i = 0; i < 4; ++i)
            {
                float e0 = i < 2 ? v0[2 * i] : v1[2 * i - 4], e1 = i < 2 ? v0[2 * i + 1] : v1[2 * i - 3];
                if (CB == 2)
                {
                    e0 = e0 * (float) as_h(0x1eee) + sx;
                    e1 = e1 * (float) as_h(0x1eee) + sx;
                }
                o[i] = as_u32((f16x2) { (f16) e0, (f16) e1 });
            }
            *to_global_w((u32x4*) (C + (size_t) row * n + part * 8)) = (u32x4) { o[0], o[1], o[2], o[3] };
        }
        EXL3_WAIT_VM_LGKM0(0);                            // the next item counts its own loads only
        __syncthreads();
    }
}
}  // namespace

#define EXL3_CAT4(a, b, c, d) a##b##c##d
#define EXL3_MOEG_FN(cb, r) EXL3_CAT4(exl3k_moeg_cb, cb, _r, r)

int EXL3_MOEG_FN(EXL3_MOEG_CB, EXL3_MOEG_R)(const MoegArgs& g, int cus, hipStream_t s)
{
    const long items = (long) g.nrt * g.mats * (g.n / 128);
    if (items <= 0) return 0;
    long grid = (long) cus * moeg_waves(EXL3_MOEG_R);
    if (grid > items) grid = items;
    grid = (grid + 7) / 8 * 8;
    hipLaunchKernelGGL((moeg_kernel<EXL3_MOEG_CB, EXL3_MOEG_R>), dim3((unsigned) grid), dim3(MG_THREADS), 0, s, g);
    return (int) hipGetLastError();
}
