// A whole dense layer in one launch, for layers of few lookups (gfx950).
//
// The LUT-GEMM kernels want tables turned into expanded rows, packed operands and sums made beforehand: three dependent
// launches of 4 to 16 us each before the last output of even the smallest layer is there.  Here every workgroup holds the
// whole truth table in LDS (128 KiB of its 160) and takes a tile of output pixels x columns from the raw tensors to the
// finished outputs: it quantizes its pixels' patches and its columns' weights, sums both in the reference's order, looks
// every product up by itself and applies the epilogue.
//
// What bounds it: single lookups of two bytes.  Lanes 0-31 and lanes 32-63 of a ds_read_u16 each look up one weight, so
// that their entries lie in one row of 512 bytes, whose 128 dwords lie two to a bank.  Everything else - loads,
// quantization, and the chains of dependent adds that the reference's order asks for - runs beside that on wavefronts of
// its own: of sixteen, two add (pixels, columns), six load and convert the next chunk of the filter elements, eight look up.
//
// Restates ApproxConvIm2ColKernel + ApproxFilterCorrCoeff + ApproxConvGEMMKernel (tf2/src/approx_nn_conv_kernels.cpp:215-306);
// sums and outputs are bit-identical to the other kernels'.
#include "lutgemm_tile.h"

namespace axc {

extern __shared__ __align__(16) unsigned char lds_direct[];

typedef uint32_t dk_u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) uint32_t *dk_lds_u32;
typedef __attribute__((address_space(3))) float *dk_lds_f32;
typedef __attribute__((address_space(3))) dk_u32x4 *dk_lds_u32x4;
typedef __attribute__((address_space(3))) uint64_t *dk_lds_u64;
typedef __attribute__((address_space(3))) uint16_t *dk_lds_u16;

// n / d for n < 2^31, without a branch
__device__ __forceinline__ uint32_t dk_quotient(const uint32_t n, const __attribute__((address_space(4))) DirectDiv &d)
{
    return (__umulhi(n, d.mul) >> d.shift) + (n & d.whole);
}

// The launch's arguments, fetched anew where they are used: all of them at once are more than there are scalar registers,
// and kept they are spilled.
typedef const __attribute__((address_space(4))) DirectParams *dk_args;
__device__ __forceinline__ dk_args dk_arguments()
{
    dk_args a = (dk_args)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return a;
}

// What quantizes a tensor, in vector registers.
struct DkQuant {
    float offset, inv_scale, scale, nudged_max;
    uint32_t fq;
};
__device__ __forceinline__ void dk_hold(DkQuant &q)
{
    asm volatile("" : "+v"(q.offset), "+v"(q.inv_scale), "+v"(q.scale), "+v"(q.nudged_max), "+v"(q.fq));
}
__device__ __forceinline__ float dk_fake_quant(const float v, const DkQuant &q)
{
    return fake_quant_value(v, TensorQuant{q.offset, q.inv_scale, q.scale, q.nudged_max, 1u, 0u});
}

// LDS behind the table: per pixel of the tile the offset and coordinates of its patch, both kinds of sums, then the two
// buffers of a chunk's floats and codes, which the tile's int32 sums take over in the end.
constexpr uint32_t kDkGeom = kTableBytes;                        // [3][64] dwords
constexpr uint32_t kDkSums = kDkGeom + 3 * 64 * 4;               // [2][64] floats
constexpr uint32_t kDkBuffers = kDkSums + 2 * 64 * 4;
constexpr int kDkItems = kDirectItems;
constexpr int kDkFirstGather = kDirectWaves - kDirectGatherWaves;   // wavefront 0: patch sums, 1: filter sums, then copies

// All wavefronts of the workgroup meet here, from wherever their part of the work has them: what they wrote to LDS is there.
// (Loads into registers stay in flight.)
__device__ __forceinline__ void dk_meet()
{
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int PT, int NCW, bool VEC>
__global__ void __launch_bounds__(kDirectThreads, 1) direct_kernel(const DirectParams)
{
    fetch_arguments<sizeof(DirectParams) <= 384 ? sizeof(DirectParams) : 384>();
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lane = (int)threadIdx.x & 63;
    const bool gathers = wave >= kDkFirstGather, copies = wave >= 2 && !gathers;

    DkQuant qi, qf;
    uint32_t CT, kc, chunks, buffer_bytes;
    int n_row_tiles, ntiles;
    {
        const dk_args a = dk_arguments();
        CT = (uint32_t)a->plan.ct;
        kc = (uint32_t)a->plan.kc;
        chunks = (uint32_t)a->plan.chunks;
        buffer_bytes = (uint32_t)a->plan.buffer_bytes;
        n_row_tiles = a->plan.n_row_tiles;
        ntiles = n_row_tiles * a->plan.n_col_tiles;
        const LayerQuant *const lq = a->lq_dev;
        if (lq) {
            qi = {lq->in.offset, lq->in.inv_scale, lq->in.scale, lq->in.nudged_max, lq->in.fq};
            qf = {lq->flt.offset, lq->flt.inv_scale, lq->flt.scale, lq->flt.nudged_max, lq->flt.fq};
        } else {
            qi = {a->in_q.offset, a->in_q.inv_scale, 0.0f, 0.0f, 0u};
            qf = {a->flt_q.offset, a->flt_q.inv_scale, 0.0f, 0.0f, 0u};
        }
        dk_hold(qi);
        dk_hold(qf);
    }
    const bool fq = __builtin_amdgcn_readfirstlane((int)qi.fq) != 0;   // of both tensors or of neither
    // rows of a buffer: pixels' floats, columns' floats, pixels' codes (two bytes each, see below), columns' codes; odd counts of
    // 16 bytes and of 8
    const uint32_t float_pitch = kc * 4u + 16u, a_pitch = kc * 2u + ((kc >> 3 & 1u) ? 0u : 16u), b_pitch = kc + ((kc >> 3 & 1u) ? 0u : 8u);
    const uint32_t fb0 = PT * float_pitch, ca0 = fb0 + CT * float_pitch, cb0 = ca0 + PT * a_pitch;
    const uint32_t kq = kc >> 2, px_items = PT * kq, col_items = CT * kq;

    // Row tiles fastest; an XCD's workgroups take a contiguous piece of that order: few columns of the filter each.
    int tile = (int)blockIdx.x, tile_end = ntiles, tile_step = (int)gridDim.x;
    if ((tile_step & 7) == 0) {
        const int xcd = tile & 7;
        tile_step >>= 3;
        tile_end = (int)((int64_t)ntiles * (xcd + 1) / 8);
        tile = (int)((int64_t)ntiles * xcd / 8) + (tile >> 3);
    }
    bool has_table = false;
    for (; tile < tile_end; tile += (tile_step)) {
        const int ct = tile / n_row_tiles, rt = tile - ct * n_row_tiles;
        const uint32_t m0 = (uint32_t)rt * PT, col0 = (uint32_t)ct * CT;

        if (threadIdx.x < PT) {   // a pixel beyond the last one is the last one, and not stored
            const dk_args p = dk_arguments();
            const uint32_t m = m0 + threadIdx.x < (uint32_t)p->M ? m0 + threadIdx.x : (uint32_t)p->M - 1u;
            const uint32_t row = dk_quotient(m, p->div_ow), n = dk_quotient(row, p->div_oh);
            const int ih = (int)(row - n * (uint32_t)p->OH) * p->sh - p->ph, iw = (int)(m - row * (uint32_t)p->OW) * p->sw - p->pw;
            const dk_lds_u32 geom = (dk_lds_u32)(uintptr_t)kDkGeom;
            geom[threadIdx.x] = (uint32_t)((((int)n * p->H + ih) * p->W + iw) * p->C);
            geom[64 + threadIdx.x] = (uint32_t)ih;
            geom[128 + threadIdx.x] = (uint32_t)iw;
        }
        dk_meet();

        // Filter elements come in by items, four of a pixel or of a column: fetched by one function, converted by another -
        // floats for the sums, codes for the lookups.  Elements beyond K add 0.0f to the sums and look up entry (0, 0), which
        // the end takes off again.  A thread has up to kDkItems items of either kind at a time, `threads` apart.
        struct Item {
            uint32_t in;          // bit e: element e exists and lies inside the image
            float v[4];
        };
        struct PxPlace {          // of an item: the pixel's patch, the first element in the chunk, where it goes in a buffer
            int off, ih0, iw0;
            uint32_t k, floats, codes;
        };
        struct ColPlace {
            uint32_t column, k, floats, codes;
        };
        struct Shape {            // of the layer, as far as items need it: in vector registers, scalar ones are short
            uint32_t K, C, KW, H, W, Co;
            int dh, dw;
        };
        auto shape_of = [&]() __attribute__((always_inline)) {
            const dk_args p = dk_arguments();
            Shape s = {(uint32_t)p->K, (uint32_t)p->C, (uint32_t)p->KW, (uint32_t)p->H, (uint32_t)p->W, (uint32_t)p->Co, p->dh, p->dw};
            return s;
        };
        auto some = [](const uint32_t i, const uint32_t n) __attribute__((always_inline)) {   // in this wavefront
            return (uint32_t)__builtin_amdgcn_readfirstlane((int)i) < n;
        };
        auto px_place = [&](const uint32_t i) __attribute__((always_inline)) {
            const dk_args p = dk_arguments();
            const uint32_t px = dk_quotient(i, p->div_kq), j = i - px * kq, at = px & (PT - 1);
            const dk_lds_u32 geom = (dk_lds_u32)(uintptr_t)kDkGeom;
            // (an item that does not exist: beyond K)
            return PxPlace{(int)geom[at], (int)geom[64 + at], (int)geom[128 + at], i < px_items ? 4u * j : 0x40000000u,
                           px * float_pitch + j * 16u, ca0 + px * a_pitch + j * 8u};
        };
        auto col_place = [&](const uint32_t i) __attribute__((always_inline)) {
            const uint32_t j = dk_quotient(i, dk_arguments()->div_ct), col = i - j * CT;
            return ColPlace{col0 + col, i < col_items ? 4u * j : 0x40000000u, fb0 + col * float_pitch + j * 16u, cb0 + col * b_pitch + j * 4u};
        };
        auto px_fetch = [&](Item &item, const PxPlace &at, const uint32_t k_base, const rsrc_t x_rsrc, const Shape &s,
                            const DirectDiv &div_c, const DirectDiv &div_kw) __attribute__((always_inline)) {
            const uint32_t k = k_base + at.k;
            const uint32_t tap = (__umulhi(k, div_c.mul) >> div_c.shift) + (k & div_c.whole);
            uint32_t c = k - tap * s.C, kh = (__umulhi(tap, div_kw.mul) >> div_kw.shift) + (tap & div_kw.whole), kw = tap - kh * s.KW;
            if (VEC) {   // four channels of one tap
                const int dh = (int)kh * s.dh, dw = (int)kw * s.dw;
                const bool inside = (k < s.K) & ((uint32_t)(at.ih0 + dh) < s.H) & ((uint32_t)(at.iw0 + dw) < s.W);
                const uint32_t byte = (uint32_t)(at.off + (dh * (int)s.W + dw) * (int)s.C + (int)c) * 4u;
                const dk_u32x4 d = __builtin_bit_cast(dk_u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                    x_rsrc, (int)(inside ? byte : 0x80000000u), 0, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    item.v[e] = __uint_as_float(d[e]);
                item.in = inside ? 15u : 0u;
            } else {
                item.in = 0u;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int dh = (int)kh * s.dh, dw = (int)kw * s.dw;
                    const bool inside = (k + e < s.K) & ((uint32_t)(at.ih0 + dh) < s.H) & ((uint32_t)(at.iw0 + dw) < s.W);
                    const uint32_t byte = (uint32_t)(at.off + (dh * (int)s.W + dw) * (int)s.C + (int)c) * 4u;
                    item.in |= inside ? 1u << e : 0u;
                    item.v[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(x_rsrc, (int)(inside ? byte : 0x80000000u), 0, 0));
                    const uint32_t next_tap = ++c == s.C ? 1u : 0u;
                    c = next_tap ? 0u : c;
                    kw += next_tap;
                    const uint32_t next_row = kw == s.KW ? 1u : 0u;
                    kw = next_row ? 0u : kw;
                    kh += next_row;
                }
            }
        };
        auto col_fetch = [&](Item &item, const ColPlace &at, const uint32_t k_base, const rsrc_t f_rsrc, const Shape &s) __attribute__((always_inline)) {
            const uint32_t k = k_base + at.k;
            uint32_t byte = (k * s.Co + at.column) * 4u;
            item.in = 0u;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const bool there = (k + e < s.K) & (at.column < s.Co);
                item.in |= there ? 1u << e : 0u;
                item.v[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(f_rsrc, (int)(there ? byte : 0x80000000u), 0, 0));
                byte += s.Co * 4u;
            }
        };
        // `left`: elements from the chunk's first on
        auto convert = [&](const Item &item, const uint32_t k, const uint32_t floats, const uint32_t codes, const uint32_t left,
                           const DkQuant &qt, const bool column) __attribute__((always_inline)) {
            uint32_t code[4];
            dk_u32x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float f = item.v[e];
                if (fq)
                    f = (item.in >> e & 1u) ? dk_fake_quant(f, qt) : 0.0f;
                w[e] = __float_as_uint(f);
                code[e] = quantize_code(f, qt.offset, qt.inv_scale);
            }
            if (left < kc) {   // (the last chunk only)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    code[e] = k + e < left ? code[e] : 0u;
            }
            if (k >= kc)       // (an item that does not exist)
                return;
            *(dk_lds_u32x4)(uintptr_t)floats = w;
            if (column)
                *(dk_lds_u32)(uintptr_t)codes = code[0] | (code[1] << 8) | (code[2] << 16) | (code[3] << 24);
            else
                *(dk_lds_u64)(uintptr_t)codes = (uint64_t)(code[0] << 1 | code[1] << 17) | (uint64_t)(code[2] << 1 | code[3] << 17) << 32;
        };

        // The first chunk is everybody's, or of those that do not fetch the table.
        if (has_table || !gathers) {
            const uint32_t threads = has_table ? kDirectThreads : kDkFirstGather * 64;
            const dk_args p = dk_arguments();
            const rsrc_t x_rsrc = make_rsrc(p->x, p->x_bytes), f_rsrc = make_rsrc(p->f, p->f_bytes);
            const DirectDiv div_c = {p->div_c.mul, p->div_c.shift, p->div_c.whole}, div_kw = {p->div_kw.mul, p->div_kw.shift, p->div_kw.whole};
            const Shape s = shape_of();
            for (uint32_t first = threadIdx.x; some(first, px_items) || some(first, col_items); first += kDkItems * threads) {
                Item px[kDkItems], col[kDkItems];
                PxPlace px_at[kDkItems];
                ColPlace col_at[kDkItems];
#pragma unroll
                for (int b = 0; b < kDkItems; ++b) {
                    px_at[b] = px_place(first + b * threads);
                    px_fetch(px[b], px_at[b], 0u, x_rsrc, s, div_c, div_kw);
                }
#pragma unroll
                for (int b = 0; b < kDkItems; ++b) {
                    col_at[b] = col_place(first + b * threads);
                    col_fetch(col[b], col_at[b], 0u, f_rsrc, s);
                }
#pragma unroll
                for (int b = 0; b < kDkItems; ++b)
                    if (some(first + b * threads, px_items))
                        convert(px[b], px_at[b].k, kDkBuffers + px_at[b].floats, kDkBuffers + px_at[b].codes, s.K, qi, false);
#pragma unroll
                for (int b = 0; b < kDkItems; ++b)
                    if (some(first + b * threads, col_items))
                        convert(col[b], col_at[b].k, kDkBuffers + col_at[b].floats, kDkBuffers + col_at[b].codes, s.K, qf, true);
            }
        } else {   // 16 KiB per wavefront
            const rsrc_t t_rsrc = make_rsrc(dk_arguments()->tableT, kTableBytes);
            constexpr int kLoads = kTableBytes / kDirectGatherWaves / 1024;
            // row b's entries 0-127 to b * 256, 128-255 to 65536 + b * 256: an instruction's 1 KiB holds two rows
            const uint32_t at = (uint32_t)(wave - kDkFirstGather) * (kLoads * 1024u) + (uint32_t)lane * 16u;
            const uint32_t to = (at >> 9 << 8) | (at & 255u) | (at >> 8 & 1u) << 16;
            dk_u32x4 w[kLoads];
#pragma unroll
            for (int i = 0; i < kLoads; ++i)
                w[i] = __builtin_bit_cast(dk_u32x4, __builtin_amdgcn_raw_buffer_load_b128(t_rsrc, (int)at, i * 1024, 0));
#pragma unroll
            for (int i = 0; i < kLoads; ++i)
                *(dk_lds_u32x4)(uintptr_t)(to + i * 512u) = w[i];
        }
        has_table = true;
        dk_meet();

        uint32_t acc[NCW];
        float sum = 0.0f;   // wavefronts 0 and 1: of this lane's pixel or column
#pragma unroll
        for (int c = 0; c < NCW; ++c)
            acc[c] = 0u;
        const uint32_t gw = (uint32_t)(wave - kDkFirstGather), px = (uint32_t)lane & (PT - 1);
        const uint32_t wc = gw & (uint32_t)(dk_arguments()->plan.wc - 1), wk = gw >> dk_arguments()->plan.wc_log;
        if (gathers) {
            // Wavefront (wc, wk) of the eight has NCW columns and a share of the chunk, lanes beyond PT a further one.  The
            // address of entry (weight b, input a) is a's low byte, b and a's high byte, a being twice the code.  The next
            // eight filter elements' codes are read behind the lookups of the last.
            const uint32_t kl = (uint32_t)dk_arguments()->plan.kl, k0 = (wk * (64 / PT) + (uint32_t)lane / PT) * kl;
            const uint32_t a_in = ca0 + px * a_pitch + k0 * 2u, b_in = cb0 + wc * (NCW * b_pitch) + k0;
            for (uint32_t q = 0; q < chunks; ++q) {
                const uint32_t buf = kDkBuffers + (q & 1u) * buffer_bytes;
                const uint32_t a_at = buf + a_in, b_at = buf + b_in;
                dk_u32x4 a_next = *(dk_lds_u32x4)(uintptr_t)a_at;
                uint64_t b_next[NCW];
#pragma unroll
                for (int c = 0; c < NCW; ++c)
                    b_next[c] = *(dk_lds_u64)(uintptr_t)(b_at + c * b_pitch);
                for (uint32_t kk = 0; kk < kl; kk += 8) {
                    const dk_u32x4 a = a_next;
                    uint32_t b[NCW][2];
#pragma unroll
                    for (int c = 0; c < NCW; ++c) {
                        b[c][0] = (uint32_t)b_next[c];
                        b[c][1] = (uint32_t)(b_next[c] >> 32);
                    }
                    const uint32_t next = kk + 8 < kl ? kk + 8 : kk;
                    a_next = *(dk_lds_u32x4)(uintptr_t)(a_at + next * 2u);
#pragma unroll
                    for (int c = 0; c < NCW; ++c)
                        b_next[c] = *(dk_lds_u64)(uintptr_t)(b_at + next + c * b_pitch);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int c = 0; c < NCW; ++c) {
                        uint32_t t[8];
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            // bytes 0-3 of the selector's operands are a's dword, 4-7 b's; 12 is zero
                            const uint32_t sel = 0x0c000000u | (2u * (e & 1) + 1u) << 16 | (4u + (e & 3)) << 8 | 2u * (e & 1);
                            t[e] = *(dk_lds_u16)(uintptr_t)__builtin_amdgcn_perm(b[c][e >> 2], a[e >> 1], sel);
                        }
#pragma unroll
                        for (int e = 0; e < 8; e += 2)
                            acc[c] += t[e] + t[e + 1];
                    }
                    // (opaque, or the compiler makes them reads of the next round)
                    asm volatile("" : "+v"(a_next));
#pragma unroll
                    for (int c = 0; c < NCW; ++c)
                        asm volatile("" : "+v"(b_next[c]));
                }
                dk_meet();
            }
        } else if (copies) {
            // chunk q + 2 on its way into registers while chunk q is used and chunk q + 1 converted
            constexpr uint32_t kCopiers = (kDkFirstGather - 2) * 64;
            const uint32_t first = threadIdx.x - 128u;
            const dk_args p = dk_arguments();
            const rsrc_t x_rsrc = make_rsrc(p->x, p->x_bytes), f_rsrc = make_rsrc(p->f, p->f_bytes);
            const DirectDiv div_c = {p->div_c.mul, p->div_c.shift, p->div_c.whole}, div_kw = {p->div_kw.mul, p->div_kw.shift, p->div_kw.whole};
            const Shape s = shape_of();
            Item px[kDkItems], col[kDkItems];
            PxPlace px_at[kDkItems];
            ColPlace col_at[kDkItems];
            bool has_px[kDkItems], has_col[kDkItems];
#pragma unroll
            for (int b = 0; b < kDkItems; ++b) {
                px_at[b] = px_place(first + b * kCopiers);
                col_at[b] = col_place(first + b * kCopiers);
                has_px[b] = some(first + b * kCopiers, px_items);
                has_col[b] = some(first + b * kCopiers, col_items);
            }
            for (uint32_t q = 0; q <= chunks; ++q) {   // (the first time round nothing has been fetched)
                if (q != 0u) {
                    if (q < chunks) {
                        const uint32_t buf = kDkBuffers + (q & 1u) * buffer_bytes, left = s.K - q * kc;
#pragma unroll
                        for (int b = 0; b < kDkItems; ++b)
                            if (has_px[b])
                                convert(px[b], px_at[b].k, buf + px_at[b].floats, buf + px_at[b].codes, left, qi, false);
#pragma unroll
                        for (int b = 0; b < kDkItems; ++b)
                            if (has_col[b])
                                convert(col[b], col_at[b].k, buf + col_at[b].floats, buf + col_at[b].codes, left, qf, true);
                    }
                }
                if (q + 1u < chunks) {
                    const uint32_t k_base = (q + 1u) * kc;
                    __builtin_amdgcn_s_waitcnt(0x0F70);   // nothing is in flight here; the compiler would wait for each register anew
#pragma unroll
                    for (int b = 0; b < kDkItems; ++b)
                        if (has_px[b])
                            px_fetch(px[b], px_at[b], k_base, x_rsrc, s, div_c, div_kw);
#pragma unroll
                    for (int b = 0; b < kDkItems; ++b)
                        if (has_col[b])
                            col_fetch(col[b], col_at[b], k_base, f_rsrc, s);
                }
                if (q != 0u)
                    dk_meet();
            }
        } else {
            // Dependent adds, sixteen at a time, the reads of the next four quads in front of them (behind a row's end lie other
            // rows).  A dependent add takes 6.6 cycles and any other instruction between two of them 2.2 more: eight at a time
            // took 15 cycles an add.
            const bool sums = dk_arguments()->out_f != nullptr;
            const uint32_t own = wave == 0 ? ((uint32_t)lane < PT ? (uint32_t)lane : PT - 1) : ((uint32_t)lane < CT ? (uint32_t)lane : CT - 1u);
            const uint32_t floats = (wave == 0 ? 0u : fb0) + own * float_pitch;
            __builtin_amdgcn_s_setprio(3);
            for (uint32_t q = 0; q < chunks; ++q) {
                if (sums) {
                    uint32_t at = kDkBuffers + (q & 1u) * buffer_bytes + floats;
                    dk_u32x4 w[4];
                    auto read = [&]() __attribute__((always_inline)) {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            w[i] = *(dk_lds_u32x4)(uintptr_t)(at + i * 16u);
                    };
                    auto add = [&](const dk_u32x4 v) __attribute__((always_inline)) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            sum = __fadd_rn(sum, __uint_as_float(v[e]));
                    };
                    read();
                    for (uint32_t b = kq >> 2; b != 0u; --b) {
                        const dk_u32x4 v0 = w[0], v1 = w[1], v2 = w[2], v3 = w[3];
                        at += 64u;
                        read();
                        __builtin_amdgcn_sched_barrier(0);
                        add(v0);
                        add(v1);
                        add(v2);
                        add(v3);
                        asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]));
                    }
                    if (kq & 2u) {
                        add(w[0]);
                        add(w[1]);
                    }
                }
                dk_meet();
            }
            __builtin_amdgcn_s_setprio(0);
        }

        // the shares of the filter elements meet in LDS, where the buffers were
        const dk_lds_u32 total = (dk_lds_u32)(uintptr_t)kDkBuffers;
        const uint32_t outputs = PT * CT;
        for (uint32_t i = threadIdx.x; i < outputs; i += kDirectThreads)
            total[i] = 0u;
        if (wave < 2)
            ((dk_lds_f32)(uintptr_t)kDkSums)[wave * 64 + lane] = sum;
        dk_meet();
        if (gathers) {
#pragma unroll
            for (int c = 0; c < NCW; ++c)
                __hip_atomic_fetch_add(total + px * CT + wc * NCW + c, acc[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
        dk_meet();
        const dk_args p = dk_arguments();
        const float *const bias = p->bias, *const addend = p->addend;
        const LayerQuant *const lq = p->lq_dev;
        float s1xs2 = p->s1xs2, m1 = p->m1, m2 = p->m2, k_m1xm2 = p->k_m1xm2;
        if (lq) {
            s1xs2 = lq->s1xs2;
            m1 = lq->m1;
            m2 = lq->m2;
            k_m1xm2 = lq->k_m1xm2;
        }
        const uint32_t surplus = (chunks * kc - (uint32_t)p->K) * (uint32_t)*(dk_lds_u16)(uintptr_t)0;
        const dk_lds_f32 psum = (dk_lds_f32)(uintptr_t)kDkSums, fsum = psum + 64;
        for (uint32_t i = threadIdx.x; i < outputs; i += kDirectThreads) {
            const uint32_t pixel = dk_quotient(i, p->div_ct), c = i - pixel * CT;
            const uint32_t m = m0 + pixel, col = col0 + c;
            if (m >= (uint32_t)p->M || col >= (uint32_t)p->Co)
                continue;
            const int32_t s = (int32_t)(total[i] - surplus);
            const int64_t at = (int64_t)m * p->Co + col;
            if (p->out_i) {
                p->out_i[at] = s;
                continue;
            }
            // approx_nn_conv_kernels.cpp:250-253, then bias and activation of the layer entry
            float v = __fadd_rn(__fmul_rn((float)s, s1xs2), __fmul_rn(m2, psum[pixel]));
            v = __fsub_rn(__fadd_rn(v, __fmul_rn(m1, fsum[c])), k_m1xm2);
            v = __fadd_rn(v, bias ? bias[col] : -0.0f);   // no bias: -0.0f, which changes no value
            if (addend)
                p->out_f[at] = sum_activation(__fadd_rn(v, addend[at]), p->relu);
            else
                p->out_f[at] = p->relu ? fmaxf(v, 0.0f) : v;
        }
        dk_meet();   // the next tile's geometry and chunks
    }
}

template <int PT, int NCW>
static hipError_t launch_direct_one(const DirectParams &p, hipStream_t stream)
{
    auto kernel = (p.C & 3) == 0 ? direct_kernel<PT, NCW, true> : direct_kernel<PT, NCW, false>;
    const hipError_t e = set_max_dynamic_lds_once(reinterpret_cast<const void *>(kernel), kDirectLdsBytes, true);
    if (e != hipSuccess)
        return e;
    hipLaunchKernelGGL(kernel, dim3(p.plan.grid), dim3(kDirectThreads), kDirectLdsBytes, stream, p);
    return hipGetLastError();
}

template <int PT>
static hipError_t launch_direct_pixels(const DirectParams &p, hipStream_t stream)
{
    switch (p.plan.ncw) {
    case 1: return launch_direct_one<PT, 1>(p, stream);
    case 2: return launch_direct_one<PT, 2>(p, stream);
    case 3: return launch_direct_one<PT, 3>(p, stream);
    case 4: return launch_direct_one<PT, 4>(p, stream);
    case 6: return launch_direct_one<PT, 6>(p, stream);
    case 8: return launch_direct_one<PT, 8>(p, stream);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_direct(const DirectParams &p, hipStream_t stream)
{
    switch (p.plan.pt) {
    case 16: return launch_direct_pixels<16>(p, stream);
    case 32: return launch_direct_pixels<32>(p, stream);
    case 64: return launch_direct_pixels<64>(p, stream);
    }
    return hipErrorInvalidValue;
}

} // namespace axc
