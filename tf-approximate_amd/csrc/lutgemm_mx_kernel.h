// Dense LUT-GEMM whose sums are made by the matrix cores (gfx950), out of pre-expanded rows or
// of rows that it makes itself (EXPAND).
//
// Every product is a lookup in the truth table, as in the other kernels: per activation code a 256-byte row of LDS
// holds the table entries of 128 slots (16 filter elements x 8 columns), and a lane fetches eight of them with one
// ds_read_b128.  What differs is who adds them up.  The vector ALUs need six instructions per such read (0.75 per
// entry), which kept the SIMDs at 38.8 cycles per read where the LDS alone takes 16; here one
// v_smfmac_i32_16x16x128_i8 per TWO reads adds them, with a constant operand of ones and zeros that only says which
// byte belongs to which sum (gen_lookup_mx.py).  The sparse form reads 32 bytes of looked-up data per lane where the
// dense one reads 16, in the same 16 cycles and for less power: under a full stream of lookups the chip is bound by
// power (a loop of nothing but lookups and dense instructions runs at 1.85-2.1 GHz and 49-56 T entries/s, with sparse
// ones at 2.2 GHz and 66 T; with the rows' and activations' traffic 42-47 and 55 T; the vector-ALU loop 32 T).
//
//   E[column tile][fill][phys_row(a)][slot]  = T[a][filter code of slot] ^ 0x8080
//   slot = filter element in the fill * 8 + column;  256 rows x 128 slots x uint16 = 64 KiB
//
// A fill covers 16 consecutive filter elements (four channel quads, which may belong to different taps: every lane
// walks the taps on its own).  The input is read through a copy of its codes with the padding written out (XqLayout),
// so that no tap is ever outside and four neighbouring pixels of an output row are one 16-byte load.
//
// One workgroup of four wavefronts per CU, each alone on its SIMD with all its 512 registers: up to 25 units of 64
// pixels x 8 columns of int32 sums (two per entry: low and high bytes add up separately and are joined at the end).
// A tile of 100 units reads a fill of 64 KiB for 6 400 pixels; fewer pixels per fill cost power and L2 bandwidth.
//
// Restates ApproxConvIm2ColKernel + ApproxConvGEMMKernel (tf2/src/approx_nn_conv_kernels.cpp:215-296); int32 sums and
// float outputs are bit-identical to the other kernels'.
#pragma once
#include "lutgemm_tile.h"
#include "px_expand.h"
#include "lookup_mx.inc"

namespace axc {

extern __shared__ __align__(16) unsigned char lds_mx[];

// Control block in LDS behind the two fill buffers: EVENTS[0], EVENTS[1], ABORT (see gen_lookup_mx.py).  EVENTS[b] only
// grows, by one per wavefront and event: four arrivals of the buffer's fill j, then its four readers, then the
// arrivals of fill j + 1, ...
constexpr uint32_t kMxCb = 2 * kPxFillBytes;
// Behind that the values the wavefronts' pixels add (patch sums, or the zero-point terms of integer outputs): a dword per
// pixel of the tile, 256 bytes per unit.
constexpr uint32_t kMxPixelValues = kMxCb + 32;
// ... and behind those the smallest and the largest output of every lane so far, for launches that report them.
constexpr uint32_t mx_range_at(const int units) { return kMxPixelValues + (uint32_t)(kMxWaves * units) * 256u; }
constexpr int mx_lds_bytes(const int units, const bool range = false) { return (int)mx_range_at(units) + (range ? kMxThreads * 8 : 0); }
constexpr uint32_t kMxWaveBytes = kPxFillBytes / kMxWaves;   // a wavefront's share of a fill
constexpr int kMxBlockCols = 8;   // column tiles (of 8) that the workgroups of an XCD walk side by side

__device__ __forceinline__ uint32_t mx_whole(const uint32_t gf) { return kMxWaves * (2u * (gf >> 1) + 1u); }
__device__ __forceinline__ uint32_t mx_free(const uint32_t gf) { return kMxWaves * (2u * (gf >> 1) + 2u); }

// n / d for n < 2^31 (MxDiv made by mx_div)
__device__ __forceinline__ uint32_t mx_quotient(const uint32_t n, const MxDiv &d)
{
    return d.mul ? __umulhi(n, d.mul) >> d.shift : n;
}

// The lane's index, recomputed where it is needed: behind the fill loop no vector register is free to have kept it.
__device__ __forceinline__ int mx_lane()
{
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(lane));
    return lane;
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) f32x2 *mx_lds_range;
typedef __attribute__((address_space(3))) uint32_t *mx_lds_u32;   // from an LDS address (dynamic LDS starts at 0)
typedef int32_t i32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t mx_u32x4 __attribute__((ext_vector_type(4)));

struct MxKStep {   // how a lane's filter position moves on by four quads (scalar operands of the fill loop)
    uint32_t dq, dkw, doff, c4, qoff, kwn, kwoff, pitch[3];
};

template <int U, bool VEC>
__device__ __forceinline__ void mx_fills(i32x16 (&acc)[U], uint32_t &ch0, uint32_t &ch1, uint32_t &koff, uint32_t &ql,
                                         uint32_t &kwl, uint32_t &cinit, uint32_t &l16, uint32_t &cbcur, uint32_t &cboth,
                                         uint32_t &edst, uint32_t &gf, uint32_t &left, uint32_t &free_at, uint32_t &whole, uint32_t &eoff,
                                         uint32_t &fail, const mx_u32x4 aop, const uint32_t idx,
                                         const uint32_t (&sel)[4], const uint32_t (&base)[U], const rsrc_t xq,
                                         const rsrc_t erc, const uint32_t enext, const uint32_t spin, const uint32_t whole0,
                                         const MxKStep &ks)
{
    uint32_t tmp, ev;
#define AXC_MX_CASE(N)                                                                                                  \
    if constexpr (U == N && VEC)                                                                                        \
        MX_FILLS_U##N##_V(acc, ch0, ch1, koff, ql, kwl, cinit, l16, cbcur, cboth, edst, gf, left, free_at, whole, eoff, fail, \
                          tmp, ev, aop, idx, sel, base, xq, erc, enext, kMxCb, spin, whole0, ks);                      \
    if constexpr (U == N && !VEC)                                                                                       \
        MX_FILLS_U##N##_S(acc, ch0, ch1, koff, ql, kwl, cinit, l16, cbcur, cboth, edst, gf, left, free_at, whole, eoff, fail, \
                          tmp, ev, aop, idx, sel, base, xq, erc, enext, kMxCb, spin, whole0, ks);
    AXC_MX_CASE(2)
    AXC_MX_CASE(3)
    AXC_MX_CASE(4)
    AXC_MX_CASE(6)
    AXC_MX_CASE(8)
    AXC_MX_CASE(10)
    AXC_MX_CASE(13)
    AXC_MX_CASE(16)
    AXC_MX_CASE(20)
    AXC_MX_CASE(25)
#undef AXC_MX_CASE
    (void)tmp;
    (void)ev;
}

// The same for the expanding form: codes of the fill that is expanded next, where the lane's chunks go in the other buffer,
// the lane's offset into a table row, and the entries of the fill stored next.
template <int U, bool VEC>
__device__ __forceinline__ void mx_xfills(i32x16 (&acc)[U], uint32_t &ch0, uint32_t &ch1, uint32_t &koff, uint32_t &ql,
                                          uint32_t &kwl, uint32_t &cinit, uint32_t &l16, uint32_t &cbcur, uint32_t &cboth,
                                          uint32_t &gf, uint32_t &left, uint32_t &free_at, uint32_t &whole, uint32_t &eoff,
                                          uint32_t &fail, const mx_u32x4 aop, const uint32_t idx,
                                          const uint32_t (&sel)[4], const uint32_t (&base)[U], const rsrc_t xq,
                                          const rsrc_t erc, const uint32_t enext, const uint32_t spin, const uint32_t whole0,
                                          const MxKStep &ks, const rsrc_t wrc, mx_u32x4 &codes, uint32_t &ldst,
                                          const uint32_t toff, i32x16 (&land)[4])
{
    uint32_t tmp, ev;
#define AXC_MX_CASE(N)                                                                                                  \
    if constexpr (U == N && VEC)                                                                                        \
        MX_XFILLS_U##N##_V(acc, ch0, ch1, koff, ql, kwl, cinit, l16, cbcur, cboth, gf, left, free_at, whole, eoff, fail, \
                           tmp, ev, aop, idx, sel, base, xq, erc, enext, kMxCb, spin, whole0, ks, wrc, codes, ldst, toff, land); \
    if constexpr (U == N && !VEC)                                                                                       \
        MX_XFILLS_U##N##_S(acc, ch0, ch1, koff, ql, kwl, cinit, l16, cbcur, cboth, gf, left, free_at, whole, eoff, fail, \
                           tmp, ev, aop, idx, sel, base, xq, erc, enext, kMxCb, spin, whole0, ks, wrc, codes, ldst, toff, land);
    AXC_MX_CASE(2)
    AXC_MX_CASE(3)
    AXC_MX_CASE(4)
    AXC_MX_CASE(6)
    AXC_MX_CASE(8)
    AXC_MX_CASE(10)
    AXC_MX_CASE(12)
    AXC_MX_CASE(13)
    AXC_MX_CASE(14)
    AXC_MX_CASE(16)
    AXC_MX_CASE(18)
#undef AXC_MX_CASE
    (void)tmp;
    (void)ev;
}

// Where lane (s, c) of a wavefront of the expanding form reads a table row and writes its chunks (gen_lookup_mx.py).
__device__ __forceinline__ uint32_t mx_x_element(const uint32_t lane) { return (lane >> 1) & 15u; }
__device__ __forceinline__ uint32_t mx_x_codes(const uint32_t lane) { return (lane & 1u) | ((lane >> 5) << 1); }

// The entries of a fill that this lane turns: quadruple 8 b + j for block b and column j.
__device__ __forceinline__ void mx_x_entries(const rsrc_t trc, const mx_u32x4 codes, const uint32_t toff, i32x16 (&land)[4])
{
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int j = i & 7;
        const uint32_t code = (j & 1) ? codes[j >> 1] >> 16 : codes[j >> 1] & 0xffffu;
        const mx_u32x4 row = __builtin_bit_cast(
            mx_u32x4, __builtin_amdgcn_raw_buffer_load_b128(trc, (int)(code * 512u + toff + 64u * (i >> 3)), 0, 0));
#pragma unroll
        for (int k = 0; k < 4; ++k)
            land[i >> 2][(i & 3) * 4 + k] = (int32_t)row[k];
    }
}

// ... turned and stored as chunks of rows: the very first fill of a workgroup.
__device__ __forceinline__ void mx_x_store(const i32x16 (&land)[4], const uint32_t ldst)
{
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        auto row = [&](const int j, const int k) __attribute__((always_inline)) {
            return (uint32_t)land[2 * b + (j >> 2)][(j & 3) * 4 + k];
        };
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            mx_u32x4 d;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                d[k] = __builtin_amdgcn_perm(row(2 * k + 1, e >> 1), row(2 * k, e >> 1), (e & 1) ? 0x07060302u : 0x05040100u);
            *(__attribute__((address_space(3))) mx_u32x4 *)(uintptr_t)(ldst + (e >> 2) * 256u + (e & 3) * 16384u + b * 2048u) = d;
        }
    }
}

// The smallest and the largest of the wavefront's outputs, where the next layer's call looks for them.
__device__ __forceinline__ void mx_store_range(float *const to, const mx_lds_range range, const int wave)
{
    f32x2 r = *range;
#pragma unroll
    for (int step = 32; step > 0; step >>= 1) {
        r[0] = fminf(r[0], __shfl_xor(r[0], step));
        r[1] = fmaxf(r[1], __shfl_xor(r[1], step));
    }
    *(f32x2 *)(to + 2 * (blockIdx.x * kMxWaves + wave)) = r;   // (by every lane the same)
}

// SIMPLE: output rows of whole groups of four pixels (p.linear) and columns in fours.  Its stores need no branch: their
// descriptor ends behind the tile's last unit, and lanes beyond the last column start at an offset that no descriptor
// reaches (2^31; 24 * 256 pixels of at most 2^18 bytes stay below 2^32).  An instantiation of its own, because the sums
// leave no registers for both forms side by side (of U = 2, whose stores are few, the compiler makes none).
// RANGE: the launch reports the smallest and the largest of its float outputs (p.range); an instantiation of its own, because
// with these stores beside the others the compiler spills.
// ADD: a tensor like the output is added before the activation (p.addend), in an instantiation of its own for the same reason.
template <int U, bool VEC, bool SIMPLE, bool EXPAND, bool RANGE = false, bool ADD = false>
__global__ void __launch_bounds__(kMxThreads, 1) lutgemm_mx_kernel(const MxParams p)
{
    fetch_arguments<sizeof(MxParams)>();
    const bool linear = SIMPLE || p.linear;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);

    if (threadIdx.x < 8)
        ((mx_lds_u32)(lds_mx + kMxCb))[threadIdx.x] = 0u;
    // (the lane's place is worked out again wherever it is needed: the fill loop leaves no register for it)
    const auto range_of = [&]() __attribute__((always_inline)) { return (mx_lds_range)(uintptr_t)mx_range_at(U) + (wave * 64 + mx_lane()); };
    if constexpr (RANGE) {
        *range_of() = f32x2{__builtin_inff(), -__builtin_inff()};
        // pairs that no wavefront of the grid writes below
        if (blockIdx.x == 0)
            for (int i = (int)(gridDim.x * kMxWaves + threadIdx.x); i < kRangePairs; i += kMxThreads)
                *(f32x2 *)(p.range + 2 * i) = f32x2{__builtin_inff(), -__builtin_inff()};
    }
    __syncthreads();   // the only barrier of the kernel

    const int n_col = p.plan.n_col_tiles * p.plan.k_splits, n_row = p.plan.n_row_tiles;
    const int ntiles = n_row * n_col;
    const int F = p.plan.fills;
    const int Fs = p.plan.k_splits > 1 ? p.plan.fills_per_split : F;
    const rsrc_t xq_rsrc = make_rsrc(p.xq, p.xq_bytes);
    // rows: pre-expanded ones, or the truth table's; the packed filter codes that name the latter
    const rsrc_t e_rsrc = EXPAND ? make_rsrc(p.tableF, kTableAllocBytes) : make_rsrc(p.rows, p.rows_bytes);
    const rsrc_t w_rsrc = make_rsrc(p.wq, EXPAND ? p.wq_bytes : 0u);
    constexpr uint32_t kStep = EXPAND ? kMxCodeBytes : (uint32_t)kPxFillBytes;   // bytes per fill of what is streamed

    // Tiles in blocks of kMxBlockCols column tiles, row tile after row tile inside a block; each XCD gets a contiguous
    // eighth of that order, which its workgroups walk side by side: the same few column tiles (same rows) of a few row
    // tiles (same activations) at a time.
    auto decode = [&](const int tile, int &rt, int &ct) __attribute__((always_inline)) {
        const int per_block = n_row * kMxBlockCols;
        const int cb = tile / per_block;
        const int in_block = tile - cb * per_block;
        const int left = n_col - cb * kMxBlockCols;
        const int w = left < kMxBlockCols ? left : kMxBlockCols;
        rt = in_block / w;
        ct = cb * kMxBlockCols + in_block - rt * w;
    };
    const int G = (int)gridDim.x;
    int tile_first, tile_end, tile_step;
    if ((G & 7) == 0) {
        const int xcd = (int)blockIdx.x & 7, i = (int)blockIdx.x >> 3;
        tile_first = (int)((int64_t)ntiles * xcd / 8) + i;
        tile_end = (int)((int64_t)ntiles * (xcd + 1) / 8);
        tile_step = G >> 3;
    } else {
        tile_first = (int)blockIdx.x;
        tile_end = ntiles;
        tile_step = G;
    }
    if (tile_first >= tile_end) {
        if constexpr (RANGE)
            mx_store_range(p.range, range_of(), wave);
        return;
    }
    const uint32_t wofs = EXPAND ? 0u : (uint32_t)wave * kMxWaveBytes;
    // expanding: this lane's filter codes of the fill whose entries are loaded next; and those of the fill stored next
    constexpr uint32_t kCodesAhead = 3;   // fills by which the loop loads filter codes ahead
    mx_u32x4 codes = {0u, 0u, 0u, 0u};
    i32x16 land[4];
    auto first_fill_of = [&](const int ctv) __attribute__((always_inline)) {
        const int ksi = ctv / p.plan.n_col_tiles;
        return (uint32_t)((ctv - ksi * p.plan.n_col_tiles) * F + ksi * Fs);
    };
    uint32_t gf = 0;   // fills this workgroup has begun, over all its tiles: fill gf lies in buffer gf & 1
    {
        int rt0, ct0;
        decode(tile_first, rt0, ct0);
        const uint32_t eoff = first_fill_of(ct0) * kStep + wofs;
        const uint32_t lane = threadIdx.x & 63u;
        // LDS addresses as integers: the kernel's dynamic LDS starts at 0 (checked at launch)
        if constexpr (EXPAND) {
            const uint32_t s16 = mx_x_element(lane) * 16u, c = mx_x_codes(lane);
            auto load = [&](const uint32_t at) __attribute__((always_inline)) {
                return __builtin_bit_cast(mx_u32x4, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (int)s16, (int)at, 0));
            };
            const mx_u32x4 first = load(eoff);
            codes = load(eoff + kStep);   // (a tile has kCodesAhead fills or more)
            const uint32_t toff = ((uint32_t)wave * 64u + c * 8u) * 2u;
            mx_x_entries(e_rsrc, first, toff, land);
            mx_x_store(land, ((uint32_t)wave * 16u + c * 2u) * 256u + s16);
            mx_x_entries(e_rsrc, codes, toff, land);
            codes = load(eoff + 2u * kStep);
        } else {
#pragma unroll
            for (int j = 0; j < (int)kMxWaveBytes / 1024; ++j)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(e_rsrc, (__attribute__((address_space(3))) void *)(uintptr_t)(wofs + j * 1024u),
                                                         16, (int)(lane * 16u), (int)(eoff + j * 1024u), 0, 0);
        }
    }
    bool first_tile = true;
    for (int tile = tile_first; tile < tile_end; tile += tile_step) {
        int rt, ctv;
        decode(tile, rt, ctv);
        const bool has_next = tile + tile_step < tile_end;
        // rows to fetch behind this tile's last fill: the next tile's first fill, or none (bit 31: the fill loop's loads then
        // lie behind the descriptor's end, and nothing moves)
        uint32_t enext = 0x80000000u;
        if (has_next) {
            int rt_next, ctv_next;
            decode(tile + tile_step, rt_next, ctv_next);
            enext = first_fill_of(ctv_next) * kStep + wofs;
        }
        const int ksi = ctv / p.plan.n_col_tiles;           // K split of this tile
        const int ct = ctv - ksi * p.plan.n_col_tiles;
        const int f0 = ksi * Fs;                            // its fills: [f0, f0 + Ft)
        const int Ft = F - f0 < Fs ? F - f0 : Fs;
        const int unit0 = rt * p.plan.units_per_tile;

        // What every pixel adds, fetched into LDS under the lookups, 64 pixels of this wavefront per instruction.  Loaded
        // by the epilogue instead, a batch of them waited for the stores of the batch before (the vector-memory counter
        // goes down in order), a round trip through the stores' queue for every six units: 5.3 us a tile of 25 (whole op,
        // us: 1x1 256->1024 @56x56x32 682 -> 640, 3x3 64->64 @56x56x64 184 -> 181).  A pixel that does not exist fetches the
        // tile's first one's.
        struct Pixels {   // the tile's first pixel, its output row and the pixels of that row before it (not linear), and how
            uint32_t row_first, before, count;   // many pixels the layer has from the first one on
            int64_t m_first;
        };
        auto tile_pixels_of = [&](const int unit) __attribute__((always_inline)) {
            Pixels t;
            const uint32_t grp = (uint32_t)unit * 16u;
            t.row_first = linear ? 0u : mx_quotient(grp, p.div_groups);
            t.before = linear ? 0u : (grp - t.row_first * (uint32_t)p.groups_per_row) * 4u;
            t.m_first = linear ? (int64_t)unit * 64 : (int64_t)t.row_first * p.ow + t.before;
            t.count = (uint32_t)(p.M - t.m_first < 1 << 20 ? p.M - t.m_first : 1 << 20);
            return t;
        };
        const uint32_t values_at = kMxPixelValues + (uint32_t)wave * (U * 256u);
        if (p.out_i == nullptr || (p.column_term != nullptr && ksi == 0)) {
            const Pixels t = tile_pixels_of(unit0);
            const uint32_t row_first = t.row_first, before = t.before, tile_pixels = t.count;
            const void *const per_pixel = p.out_i ? static_cast<const void *>(p.pixel_term + t.m_first) : p.psum + t.m_first;
            const rsrc_t pp_rsrc = make_rsrc(per_pixel, tile_pixels * 4u);
            const uint32_t lane = (uint32_t)mx_lane();
#pragma unroll
            for (int u = 0; u < U; ++u) {
                uint32_t at;
                if (linear) {
                    at = (uint32_t)(wave + u * kMxWaves) * 64u + lane;
                    at = at < tile_pixels ? at : 0u;
                } else {
                    const uint32_t grp = (uint32_t)(unit0 + wave + u * kMxWaves) * 16u + (lane >> 2);
                    const uint32_t row = mx_quotient(grp, p.div_groups);
                    const uint32_t ow = (grp - row * (uint32_t)p.groups_per_row) * 4u + (lane & 3u);
                    at = (row - row_first) * (uint32_t)p.ow + ow - before;
                    at = ow < (uint32_t)p.ow && at < tile_pixels ? at : 0u;
                }
                __builtin_amdgcn_raw_ptr_buffer_load_lds(pp_rsrc, (__attribute__((address_space(3))) void *)(uintptr_t)(values_at + u * 256u),
                                                         4, (int)(at * 4u), 0, 0, 0);
            }
        }

        i32x16 acc[U];
        uint32_t fail;
        {
            const int lane = mx_lane();
            const uint32_t q = (uint32_t)lane >> 4, i = (uint32_t)lane & 15u, ilo = i & 3u;
            const uint32_t plane = (i >> 2) ^ (q == 0u ? 0u : q == 1u ? 3u : q - 1u);
            // the constant operand of the matrix instruction: row i of it selects byte i of both 16-byte halves.  Stored
            // two of every four (sparse): byte i & 3 of its group in the first slot, or 3 in the second.
            uint32_t idx = 0xccccccccu;   // slots hold elements 0 and 3
            uint32_t one = 0x100u;
            if (ilo < 3u) {
                const uint32_t sh = 4u * (i >> 2);
                idx = (idx & ~(3u << sh) & ~(3u << (sh + 16u))) | (ilo << sh) | (ilo << (sh + 16u));
                one = 1u;
            }
            one <<= (i & 4u) ? 16 : 0;
            const mx_u32x4 aop = {i < 8u ? one : 0u, i < 8u ? 0u : one, i < 8u ? one : 0u, i < 8u ? 0u : one};
            const uint32_t buf = (gf & 1u) << 24;
            uint32_t sel[4], chunk[4];
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) {
                sel[c] = 0x0c030000u | ((4u + (ilo ^ c)) << 8) | (c < 3u ? c : 0u);
                chunk[c] = (plane * 4u + (ilo ^ c)) << 4;
            }
            uint32_t ch0 = chunk[0] | (chunk[1] << 8) | (chunk[2] << 16) | buf, ch1 = chunk[3] | buf;
            // where the lane's filter position starts: quad f0 * 4 + plane of the K order (tap row, tap column, quad)
            uint32_t ql, kwl, koff;
            {
                const uint32_t quad = (uint32_t)f0 * 4u + plane, tap = mx_quotient(quad, p.div_c4);
                ql = quad - tap * (uint32_t)p.c4;
                const uint32_t kh = mx_quotient(tap, p.div_kw);
                kwl = tap - kh * (uint32_t)p.kw;
                koff = kh * p.kh_step + kwl * p.kw_step + ql * p.quad_step;
            }
            uint32_t base[U];
            {   // unit 0 by division, the others from it: 64 groups on are p.step_* (images, rows, groups), with carries
                const uint32_t grp = (uint32_t)(unit0 + wave) * 16u + i;
                const uint32_t row = mx_quotient(grp, p.div_groups), n = mx_quotient(row, p.div_oh);
                uint32_t gw = grp - row * (uint32_t)p.groups_per_row, oh = row - n * (uint32_t)p.oh;
                uint32_t b = p.origin + n * p.img_step + oh * p.orow_step + gw * p.group_step;
#pragma unroll
                for (int u = 0; u < U; ++u) {   // (a unit that does not exist reads what lies behind the layer's input, or nothing)
                    base[u] = b;
                    gw += p.step_groups;
                    const bool c1 = gw >= (uint32_t)p.groups_per_row;
                    gw -= c1 ? (uint32_t)p.groups_per_row : 0u;
                    oh += p.step_rows + (c1 ? 1u : 0u);
                    const bool c2 = oh >= (uint32_t)p.oh;
                    oh -= c2 ? (uint32_t)p.oh : 0u;
                    b += p.step_bytes + (c1 ? p.carry_row : 0u) + (c2 ? p.carry_img : 0u);
                }
            }
            const MxKStep ks = {(uint32_t)p.dq, (uint32_t)p.dkw, p.doff, (uint32_t)p.c4, p.qoff, (uint32_t)p.kw, p.kwoff,
                                {p.pitch, 2u * p.pitch, 3u * p.pitch}};
            if (first_tile) {   // this wavefront's share of the workgroup's very first fill has arrived (LDS stores: in order)
                if (!EXPAND)
                    __builtin_amdgcn_s_waitcnt(0x0F70);
                if (lane == 0)
                    asm volatile("ds_add_u32 %0, %1" : : "v"(kMxCb), "v"(1u) : "memory");
                first_tile = false;
            }
            const uint32_t other = (gf & 1u) ^ 1u;
            uint32_t cinit = 32896u * 16u * (uint32_t)Ft;   // what flipping the top bits took from every sum
            uint32_t cbcur = kMxCb + 4u * (gf & 1u), cboth = kMxCb + 4u * other, edst = wofs + other * (uint32_t)kPxFillBytes;
            uint32_t left = (uint32_t)Ft;
            // the other buffer is free once fill gf - 1 is read (fill 1 goes into a buffer never used)
            uint32_t free_at = gf == 0u ? 0u : mx_free(gf - 1u), whole = Ft > 1 ? mx_whole(gf + 1u) : 0u;
            const uint32_t whole0 = mx_whole(gf);
            if constexpr (EXPAND) {   // filter codes are loaded three fills ahead
                const uint32_t after = Ft > (int)kCodesAhead ? ((uint32_t)(ct * F + f0) + kCodesAhead) * kStep : enext;
                const uint32_t s16 = mx_x_element((uint32_t)lane) * 16u, c = mx_x_codes((uint32_t)lane);
                uint32_t eoff = after & 0x7fffffffu, l16 = s16 | (after & 0x80000000u);
                uint32_t ldst = ((uint32_t)wave * 16u + c * 2u) * 256u + s16 + other * (uint32_t)kPxFillBytes;
                mx_xfills<U, VEC>(acc, ch0, ch1, koff, ql, kwl, cinit, l16, cbcur, cboth, gf, left, free_at, whole, eoff, fail,
                                  aop, idx, sel, base, xq_rsrc, e_rsrc, enext, p.spin_limit, whole0, ks, w_rsrc, codes, ldst,
                                  ((uint32_t)wave * 64u + c * 8u) * 2u, land);
            } else {
                const uint32_t after = Ft > 1 ? ((uint32_t)(ct * F + f0) + 1u) * kStep + wofs : enext;
                uint32_t eoff = after & 0x7fffffffu, l16 = (uint32_t)lane * 16u | (after & 0x80000000u);
                mx_fills<U, VEC>(acc, ch0, ch1, koff, ql, kwl, cinit, l16, cbcur, cboth, edst, gf, left, free_at, whole, eoff, fail,
                                 aop, idx, sel, base, xq_rsrc, e_rsrc, enext, p.spin_limit, whole0, ks);
            }
        }
        if (fail) {   // a wait that ran out: tell the host and the other wavefronts, and leave
            if (mx_lane() == 0) {
                *(mx_lds_u32)(uintptr_t)(kMxCb + 8u) = 1u;
                if (p.wait_error)
                    __hip_atomic_store(p.wait_error, fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
            return;
        }

        // ---- epilogue: join low and high bytes, zero-point correction + dequantize (approx_nn_conv_kernels.cpp:250-253),
        // bias and activation of the layer entry, store ----
        // Lane (g, i) holds columns 2 g and 2 g + 1 of pixels 4 i .. 4 i + 3.  Swapping 16-lane rows between an even and
        // an odd pixel leaves it with four consecutive columns of one pixel: 16-byte stores, through a buffer descriptor
        // that begins at the tile's first pixel, so that a unit's address is one addition and what lies outside the layer
        // (beyond the last pixel: the descriptor's end; beyond a row or the last column: an offset that no descriptor
        // reaches) is not stored.  A tile has at most 6 400 pixels of at most 2^18 bytes: offsets stay below 2^31.
        const int lane = mx_lane();
        const uint32_t g = (uint32_t)lane >> 4, i = (uint32_t)lane & 15u;
        const int col0 = ct * 8 + (int)(g >> 1) * 4;
        const bool ints = p.out_i != nullptr, terms = ints && p.column_term != nullptr && ksi == 0;
        int unit_first = unit0;
        asm volatile("" : "+s"(unit_first));   // worked out again, not kept: the fill loop leaves few scalar registers
        const Pixels tile_px = tile_pixels_of(unit_first);
        const uint32_t row_first = tile_px.row_first, before = tile_px.before, tile_pixels = tile_px.count;
        const int64_t m_first = tile_px.m_first;
        const uint32_t pixel_bytes = (uint32_t)p.Co * 4u;
        uint32_t *const out = (ints ? reinterpret_cast<uint32_t *>(p.out_i) + (int64_t)ksi * p.M * p.Co
                                    : reinterpret_cast<uint32_t *>(p.out_f)) + m_first * p.Co;
        const uint32_t own_pixels = (uint32_t)p.plan.units_per_tile * 64u;
        const uint64_t out_bytes = (uint64_t)(SIMPLE && own_pixels < tile_pixels ? own_pixels : tile_pixels) * pixel_bytes;
        const rsrc_t out_rsrc = make_rsrc(out, out_bytes < 0x80000000u ? (uint32_t)out_bytes : 0x80000000u);
        constexpr uint32_t kNowhere = 0x80000000u;
        // This lane's pixels of the wavefront's unit u (in each pair of neighbours the even or the odd one), counted from
        // the tile's first pixel: px[jp]; kNowhere where there is none.  Where output rows are whole groups of four,
        // pixels follow each other (those beyond the layer's last are left to the descriptors).
        const uint32_t j0 = g & 1u, px0 = ((uint32_t)wave * 16u + i) * 4u + j0;
        auto pixels_of = [&](const int u, uint32_t (&px)[2]) __attribute__((always_inline)) {
            if (linear) {
                px[0] = px0 + (uint32_t)u * (kMxWaves * 64u);
                px[1] = px[0] + 2u;
            } else {
                const uint32_t grp = (uint32_t)(unit_first + wave + u * kMxWaves) * 16u + i;
                const uint32_t row = mx_quotient(grp, p.div_groups), ow = (grp - row * (uint32_t)p.groups_per_row) * 4u + j0;
                const uint32_t at = (row - row_first) * (uint32_t)p.ow + ow - before;
                px[0] = ow < (uint32_t)p.ow && at < tile_pixels ? at : kNowhere;
                px[1] = ow + 2u < (uint32_t)p.ow && at + 2u < tile_pixels ? at + 2u : kNowhere;
            }
        };
        const uint32_t at0 = SIMPLE && col0 >= p.Co ? kNowhere : px0 * pixel_bytes + (uint32_t)col0 * 4u;   // bytes of px0 (linear)
        // Four columns leave as one 16-byte store, which needs no more than the alignment of a dword, and only those of an
        // incomplete last group one by one (all of them, where columns do not come in fours: 1x1 16->342 @38x38x38 88.9 us).
        const bool tail = !SIMPLE && (p.Co & 3) != 0 && ct * 8 + 8 > p.Co;
        const bool whole = col0 + 4 <= p.Co;
        const float e_s1xs2 = p.lq_dev ? p.lq_dev->s1xs2 : p.s1xs2, e_m1 = p.lq_dev ? p.lq_dev->m1 : p.m1;
        const float e_m2 = p.lq_dev ? p.lq_dev->m2 : p.m2, e_km = p.lq_dev ? p.lq_dev->k_m1xm2 : p.k_m1xm2;
        float t3[4], bias[4];   // no bias: -0.0f, which changes no value
        uint32_t term[4];       // integer outputs: what the column adds
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = col0 + e < p.Co ? col0 + e : p.Co - 1;
            t3[e] = ints ? 0.0f : __fmul_rn(e_m1, p.fsum[c]);
            bias[e] = (!ints && p.bias) ? p.bias[c] : -0.0f;
            term[e] = terms ? (uint32_t)p.column_term[c] : 0u;
        }
        // the values fetched before the lookups, of this lane's pixels of unit 0 (integer outputs without terms: masked out)
        const mx_lds_u32 values = (mx_lds_u32)(uintptr_t)(values_at + i * 16u + j0 * 4u);
        const uint32_t value_mask = ints && !terms ? 0u : 0xffffffffu;
        auto join = [&](const int32_t lo, const int32_t hi) __attribute__((always_inline)) {
            return (uint32_t)lo + ((uint32_t)hi << 8);
        };
        // kInts: int32 sums; kRelu: the activation
        auto store_tile = [&](auto ints_t, auto relu_t) __attribute__((always_inline)) {
            constexpr bool kInts = decltype(ints_t)::value, kRelu = decltype(relu_t)::value;
            float lo = __builtin_inff(), hi = -__builtin_inff();
            const bool relu = p.relu != 0;
            constexpr int kAhead = 6;   // units whose values are read together
            // What is added is loaded a batch of units ahead of its use: the vector-memory counter goes down in order, so a load
            // waits for the stores before it, here those of two batches ago.  Bound by memory (1x1 64->256 @56x56x64, 205 MB in
            // and out, on top of the 145 us that the layer takes: batches of 4 units 72 us, of 6 93, a window of 6 units that
            // moves on by one 81, by two 77; an elementwise pass took 118).
            constexpr int kBatch = 4;
            const rsrc_t add_rsrc = make_rsrc(ADD ? p.addend + m_first * p.Co : nullptr, ADD ? (uint32_t)out_bytes : 0u);
            const float floor = relu ? 0.0f : -__builtin_inff();
            mx_u32x4 added[ADD ? U : 1][2];
            auto load_added = [&](const int from, const int to) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (u >= from && u < to) {
                        const uint32_t at = at0 + (uint32_t)u * (kMxWaves * 64u) * pixel_bytes;
                        added[u][0] = __builtin_amdgcn_raw_buffer_load_b128(add_rsrc, (int)at, 0, 0);
                        added[u][1] = __builtin_amdgcn_raw_buffer_load_b128(add_rsrc, (int)(at + 2u * pixel_bytes), 0, 0);
                    }
            };
            if constexpr (ADD)
                load_added(0, kBatch);
#pragma unroll
            for (int u0 = 0; u0 < U; u0 += kAhead) {
                uint32_t ps[kAhead][2];
#pragma unroll
                for (int k = 0; k < kAhead; ++k)
                    if (u0 + k < U) {
                        ps[k][0] = values[(u0 + k) * 64] & value_mask;
                        ps[k][1] = values[(u0 + k) * 64 + 2] & value_mask;
                    }
#pragma unroll
                for (int k = 0; k < kAhead; ++k) {
                    const int u = u0 + k;
                    if constexpr ((RANGE && U > 20) || ADD)   // (or the scheduler joins the sums of many units ahead of their turn, and spills)
                        __builtin_amdgcn_sched_barrier(0);
                    if (u >= U || (!SIMPLE && u * kMxWaves + wave >= p.plan.units_per_tile))
                        continue;
                    if constexpr (ADD)
                        if (u % kBatch == 0)
                            load_added(u + kBatch, u + 2 * kBatch);
                    const i32x16 &a = acc[u < U ? u : 0];
                    uint32_t at[2] = {at0 + (uint32_t)u * (kMxWaves * 64u) * pixel_bytes, 0u};
                    at[1] = at[0] + 2u * pixel_bytes;
                    if (!linear) {
                        uint32_t px[2];
                        pixels_of(u, px);
                        at[0] = px[0] == kNowhere ? kNowhere : px[0] * pixel_bytes + (uint32_t)col0 * 4u;
                        at[1] = px[1] == kNowhere ? kNowhere : px[1] * pixel_bytes + (uint32_t)col0 * 4u;
                    }
#pragma unroll
                    for (int jp = 0; jp < 2; ++jp) {
                        const auto s0 = __builtin_amdgcn_permlane16_swap(join(a[8 * jp], a[8 * jp + 1]),
                                                                         join(a[8 * jp + 4], a[8 * jp + 5]), false, false);
                        const auto s1 = __builtin_amdgcn_permlane16_swap(join(a[8 * jp + 2], a[8 * jp + 3]),
                                                                         join(a[8 * jp + 6], a[8 * jp + 7]), false, false);
                        mx_u32x4 d = {s0[0], s1[0], s0[1], s1[1]};
                        if (kInts) {
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                d[e] += ps[k][jp] + term[e];
                        } else {
                            const float t1 = __fmul_rn(e_m2, __uint_as_float(ps[k][jp]));
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                float v = __fadd_rn(__fmul_rn((float)(int32_t)d[e], e_s1xs2), t1);
                                v = __fadd_rn(__fsub_rn(__fadd_rn(v, t3[e]), e_km), bias[e]);
                                if constexpr (ADD) {   // (as the elementwise pass has it: NaN stays, and no sum of -0 does)
                                    v = __fadd_rn(v, __uint_as_float(added[u < U ? u : 0][jp][e]));
                                    d[e] = __float_as_uint(!(v <= floor) ? v : floor);
                                } else if constexpr (RANGE)   // (one form: of two side by side the compiler joins all sums first, and spills)
                                    d[e] = __float_as_uint(relu ? fmaxf(v, 0.0f) : v);
                                else
                                    d[e] = __float_as_uint(kRelu ? fmaxf(v, 0.0f) : v);
                            }
                            if constexpr (RANGE) {   // what is not stored counts as NaN: as nothing
                                const bool there = at[jp] < (uint32_t)out_bytes;
#pragma unroll
                                for (int e = 0; e < 4; ++e) {
                                    const float v = there && (SIMPLE || whole || col0 + e < p.Co) ? __uint_as_float(d[e]) : __builtin_nanf("");
                                    lo = fminf(lo, v);
                                    hi = fmaxf(hi, v);
                                }
                            }
                        }
                        if (SIMPLE) {
                            __builtin_amdgcn_raw_buffer_store_b128(d, out_rsrc, (int)at[jp], 0, 0);
                        } else {
                            __builtin_amdgcn_raw_buffer_store_b128(d, out_rsrc, (int)(whole ? at[jp] : kNowhere), 0, 0);
                            if (tail) {
#pragma unroll
                                for (int e = 0; e < 3; ++e)
                                    __builtin_amdgcn_raw_buffer_store_b32(d[e], out_rsrc, (int)(!whole && col0 + e < p.Co ? at[jp] + 4u * e : kNowhere), 0, 0);
                            }
                        }
                    }
                }
            }
            if constexpr (RANGE) {
                const mx_lds_range range = range_of();
                const f32x2 r = *range;
                *range = f32x2{fminf(r[0], lo), fmaxf(r[1], hi)};
            }
        };
        using yes = std::true_type;
        using no = std::false_type;
        if (!RANGE && !ADD && ints)
            store_tile(yes(), no());
        else if (!RANGE && !ADD && p.relu)
            store_tile(no(), yes());
        else
            store_tile(no(), no());
        asm volatile("" ::: "memory");   // the values are read before the next tile's are fetched into their place
    }
    if constexpr (RANGE)
        mx_store_range(p.range, range_of(), wave);
}

template <int U, bool VEC, bool SIMPLE, bool EXPAND, bool RANGE = false, bool ADD = false>
static hipError_t launch_mx_one(const MxParams &p, hipStream_t stream)
{
    auto kernel = lutgemm_mx_kernel<U, VEC, SIMPLE, EXPAND, RANGE, ADD>;
    const hipError_t e = set_max_dynamic_lds_once(reinterpret_cast<const void *>(kernel), mx_lds_bytes(U, RANGE), true);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(kernel, dim3(p.plan.grid), dim3(kMxThreads), mx_lds_bytes(U, RANGE), stream, p);
    return hipGetLastError();
}

template <int U, bool EXPAND>
static hipError_t launch_mx_units(const MxParams &p, hipStream_t stream)
{
    const bool vec = p.pitch == 4, simple = p.linear && (p.Co & 3) == 0;
    if (p.addend)       // (where mx_adds says so)
        return launch_mx_one<U, true, true, EXPAND, false, true>(p, stream);
    if constexpr (U >= kMxRangeUnits) {
        if (p.range)   // (where mx_reports_range says so)
            return vec ? launch_mx_one<U, true, true, EXPAND, true>(p, stream) : launch_mx_one<U, false, true, EXPAND, true>(p, stream);
    }
    if constexpr (U > 2) {
        if (simple)
            return vec ? launch_mx_one<U, true, true, EXPAND>(p, stream) : launch_mx_one<U, false, true, EXPAND>(p, stream);
    }
    return vec ? launch_mx_one<U, true, false, EXPAND>(p, stream) : launch_mx_one<U, false, false, EXPAND>(p, stream);
}

} // namespace axc
