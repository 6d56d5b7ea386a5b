// Internal declarations shared by the HIP translation units of libaxconv_hip.so.
#pragma once

#include <hip/hip_runtime.h>
#include <map>
#include <mutex>
#include <utility>
#include <stdint.h>
#include <stddef.h>

#include "axconv.h"

namespace axc {

constexpr int kTableBytes = 131072;            // 256 x 256 uint16, weight-code major
constexpr int kTableRows = 257;                // row 256 is all zeros: the row of the null weight
constexpr int kTableAllocBytes = kTableRows * 512;
constexpr int kExpandBytes = 32768;            // one expanded-row buffer: 256 activation rows x 64 slots x uint16
constexpr int kDenseLdsBytes = 4 * kExpandBytes; // dense kernel: 2 buffers of expanded rows + 2 of staged table rows
constexpr int kDenseThreads = 512;             // dense kernel: 8 wavefronts x 256 VGPRs, one workgroup per CU
constexpr int kDenseWaves = kDenseThreads / 64;
constexpr int kDenseParkBytes = 16 * 4 * kDenseThreads; // per-thread pixel geometry parked behind the buffers
constexpr int kPxMaxTileWaveRows = 8 * kDenseWaves - 1;  // lutgemm_pxf_kernel: the last wavefront's last pixel slot holds
                                                         // the kernel's wait counters instead of geometry
constexpr int kBlockThreads = 1024;            // depthwise kernel / LDS probe: 16 wavefronts per CU
constexpr int kWaves = kBlockThreads / 64;
// Accumulate instruction mix of the dense kernel's generated phase body (gen_lookup_asm.py emits the same):
// 0 = one VALU add per table entry (v_add_u32 of a whole dword + v_add_u32_sdwa of its high half);
// 1 = three per four entries (two dwords of one column pair folded by one v_add3_u32, the high halves by SDWA adds).
constexpr int kDenseAccumulateMix = 1;   // what the 16- and 32-column tiles run (64-column tiles: mix 0)
constexpr uint16_t kNullWeight = 256;          // slot that contributes nothing (padding channel / column)

// Geometry of one dense layer after validation.
struct ConvGeom {
    int N, H, W, C;        // input NHWC
    int KH, KW, Co;        // filter HWIO (in depth == C)
    int OH, OW;
    int sh, sw, dh, dw, ph, pw;
    int C4;                // ceil(C / 4): channel quads in the quantized activation layout
    int64_t M;             // N * OH * OW
    int K;                 // KH * KW * C
};

// How the dense LUT-GEMM is cut into workgroup tiles.
struct DensePlan {
    int nt;                // columns per tile: 16, 32 or 64
    int rows_per_tile;     // multiple of 64, <= 1024 * (64 / nt)
    int n_row_tiles, n_col_tiles;
    int fills;             // expanded-row refills over the whole K: KH*KW * C4 * (4 / (64/nt))
    int k_splits;          // tiles along K: each computes fills_per_split fills into its own int32 partial sums
    int fills_per_split;
    int grid;
    int px;                // 1: the layer suits the kernel that reads pre-expanded rows (lutgemm_px_kernel.hip)
    float cost;            // what the planner's model expects of the LUT-GEMM launches, in cycles
};

// Quantization of one tensor as the pre-pass kernels see it.
struct TensorQuant {
    float offset;       // nudged minimum
    float inv_scale;
    float scale;
    float nudged_max;
    uint32_t fq;        // 1: snap every value to the 8-bit grid first (the Keras layer's fake quantization)
    uint32_t zp4;       // row-permuted code of 0.0f, replicated in all four bytes (input tensor only)
};

// Everything the kernels need to know about a layer's quantization.  The op entry points pass it by value
// (min/max are host scalars there); the layer entry point computes it on the device from the tensors' own
// min/max, so kernels take both a value and a device pointer and use the pointer when it is not null.
struct LayerQuant {
    TensorQuant in, flt;
    float s1xs2, m1, m2, k_m1xm2;
};

// fake_quant_with_min_max_vars on one value (clamp to the nudged range, round half up to the grid), in the
// float32 operations of TensorFlow's functor; identity unless q.fq.
__device__ inline float fake_quant_value(float v, const TensorQuant &q)
{
    if (!q.fq)
        return v;
    if (q.scale == 0.0f)
        return 0.0f;                       // min == max == 0: the whole tensor quantizes to 0
    const float c = fmaxf(fminf(v, q.nudged_max), q.offset);
    const float t = floorf(__fadd_rn(__fmul_rn(__fsub_rn(c, q.offset), q.inv_scale), 0.5f));
    return __fadd_rn(__fmul_rn(t, q.scale), q.offset);
}

struct DenseParams {
    ConvGeom g;
    DensePlan plan;
    const uint32_t *xq;     // [N][H][C4][W] dwords of 4 row-permuted activation codes, then one more
                            // [C4][W] row holding the zero-point code (read by taps outside the image)
    const float *psum;      // [M] sum of the raw input over each output pixel's patch (float epilogue only)
    const uint16_t *wq;     // [n_col_tiles][fills][64] packed filter codes (kNullWeight = none)
    const float *fsum;      // [Co] sum over (h, w, c) of the raw filter
    const uint16_t *tableT; // [257 filter code (256 = null)][256 input code]
    float *out_f;
    int32_t *out_i;         // with k_splits > 1: [k_splits][M][Co] partial sums, reduced by launch_splitk_epilogue
    float s1xs2, m1, m2, k_m1xm2; // epilogue constants; k_m1xm2 = float(K) * m1xM2
    uint32_t zp4;           // row-permuted zero code replicated in all four bytes
    uint32_t xq_bytes, wq_bytes; // sizes of the two streams (buffer-descriptor bounds)
    int step_n, step_oh, step_ow; // 64 * kDenseWaves / 2 output pixels (the distance between a lane's pixels) as
                                  // images, output rows and output columns
    const LayerQuant *lq_dev;    // not null: epilogue constants come from here instead of the four floats above
    const float *bias;           // not null: added to every output column after the epilogue
    const float *addend;         // not null: a tensor like the output, added before the activation, by the epilogues of split sums
    int relu;                    // 1: max(x, 0) last
    int stagger_sleeps;          // s_sleep(127) periods by which group g of the workgroups starts late, times g (0: none)
    int stagger_groups;          // g = 0 .. stagger_groups - 1 in turn (2: every second group, the only form lutgemm_expand has)
    const uint16_t *px_rows;     // pre-expanded rows [n_col_tiles][fills / 2][256][128] (lutgemm_px_kernel only)
    uint32_t px_bytes;
    // Addressing of xq.  Usual layout: dwords of four channels, [N][H][C4][W].  Flat layout (channel counts that are
    // no multiple of four, see prepare_dense): bytes, [N][H][row], a row = the pixels' channels one after the other
    // with the horizontal padding written out; g then describes a filter of KH taps whose "channels" are the
    // KW * C bytes a filter row covers.
    int row_step;                // between input rows, in address units
    int addr_unit;               // bytes per address unit: 4 (dwords) or 1 (flat)
    uint32_t quad_bytes;         // between the channel quads that one tap of a pixel reads
    uint32_t zp_tail_bytes;      // size of the zero-point row behind xq
    int flat_col_bytes;          // flat: bytes between horizontally neighbouring output pixels (sw * C); 0 = usual layout
    // lutgemm_pxf_kernel: its wavefronts wait for each other through counters in LDS, every wait a bounded number of
    // polls.  A wait that runs out writes a nonzero word to *wait_error (host-visible memory) and the wavefront leaves
    // the kernel; so do the others at their next wait.
    uint32_t spin_limit;
    uint32_t *wait_error;
};

constexpr int kRangePairs = AXC_RANGE_BYTES / 8; // (smallest, largest) of a tensor as one call leaves them to the next

// ---- lutgemm_mx_kernel.hip: lookups summed by the matrix cores ----
constexpr int kMxThreads = 256;                // four wavefronts, one per SIMD, 512 registers each
constexpr int kMxWaves = kMxThreads / 64;
constexpr int kMxCols = 8;                     // columns per tile
constexpr int kMxFillQuads = 4;                // channel quads (of any taps) per fill
constexpr int kMxUnits[] = {2, 3, 4, 6, 8, 10, 13, 16, 20, 25};   // 64-pixel units per wavefront: the kernel's variants
constexpr int kMxExpandUnits[] = {2, 3, 4, 6, 8, 10, 12, 13, 14, 16, 18};   // the same where it makes its rows itself
constexpr int kMxMinExpandFills = 3;           // ... and the fewest fills of its tiles (it loads that far ahead)
constexpr int kMxCodeBytes = 256;              // packed filter codes of a fill: 16 filter elements x 8 columns x uint16

struct MxPlan {
    int units;             // units per wavefront, one of kMxUnits
    int units_per_tile;    // units in a tile, at most kMxWaves * units
    int n_row_tiles, n_col_tiles;
    int fills;             // fills of kMxFillQuads quads over the whole K
    int k_splits, fills_per_split;
    int grid;
    int expand;            // 1: the kernel makes its rows itself, out of packed filter codes and the table
    int swap;              // 1 (with expand): operands exchanged, see SwapPack
    float cost;            // cycles the planner's model expects
};

// Quantized input with its padding written out, as lutgemm_mx_kernel reads it: dwords [n][Hp][C4][Wp], pixel (h, w) in
// row h + row0, column w + col0.  The rows and columns in front of an image double as those behind the one before it,
// so row0 and col0 are the larger of the two paddings (or one column more: padded_layout); behind the last image follow row0
// more rows and, where there is column padding too, one for the columns behind the last of those.  Without padding (and always for the other kernels)
// Hp = H, Wp = W, row0 = col0 = 0, and one row follows the last image.
struct XqLayout {
    int Hp, Wp, row0, col0;
    __host__ __device__ int tail_rows() const { return row0 == 0 ? 1 : row0 + (col0 > 0 ? 1 : 0); }
};

// Few output pixels under many weights: lutgemm_mx_kernel with its operands exchanged.  A fill costs what it costs
// however few pixels look it up, so the operand with the fewer rows makes the fills: output pixels stand where columns
// stood (8 to a tile, the codes of their patches packed as filter codes are), and the filter's columns where pixels stood,
// an image of one row, Co pixels and K channels.  The table is taken the other way round, sums come out as [Co][M].
struct SwapPack {
    int K, quads, fills;   // filter elements, ceil(K / 4), ceil(quads / 4)
    int cols, pitch;       // Co, and Co rounded up to fours
    int tiles;             // ceil(M / 8)
    __host__ __device__ int64_t filter_units() const { return (int64_t)quads * (pitch / 4); }
    __host__ __device__ int64_t units() const { return filter_units() + (int64_t)tiles * fills * 16; }
};
inline SwapPack swap_pack_of(const ConvGeom &g)
{
    const int quads = (g.K + 3) / 4;
    return {g.K, quads, (quads + 3) / 4, g.Co, (g.Co + 3) & ~3, (int)((g.M + 7) / 8)};
}

struct MxDiv {             // division by a constant for 31-bit numbers: mulhi(n, mul) >> shift; mul = 0: n itself
    uint32_t mul, shift;
};

struct MxParams {
    MxPlan plan;
    const void *xq;
    uint32_t xq_bytes;
    const uint16_t *rows;  // pre-expanded ones
    uint32_t rows_bytes;
    const float *psum, *fsum, *bias;
    const int32_t *pixel_term, *column_term;   // not null (tf1 op): added to the integer outputs, by the first K split
    float *out_f;
    int32_t *out_i;        // with k_splits > 1: [k_splits][M][Co] partial sums
    const LayerQuant *lq_dev;
    float s1xs2, m1, m2, k_m1xm2;
    int relu;
    int64_t M;
    int Co, oh, ow;
    int groups_per_row;            // groups of four neighbouring pixels per output row
    int linear;                    // output rows are whole groups: pixel = 4 * group + position
    MxDiv div_groups, div_oh, div_c4, div_kw;
    // bytes in xq: of output pixel 0's tap (0, 0); between images, output rows, pixel groups, pixels of a group; between
    // tap rows, tap columns and quads
    uint32_t origin, img_step, orow_step, group_step, pitch, kh_step, kw_step, quad_step;
    int c4, kw;                    // quads per tap, taps per filter row
    int dq, dkw;                   // four quads on: quads and taps to add, and the bytes they are; then what a carry
    uint32_t doff, qoff, kwoff;    // of the quad into the tap and of the tap into the tap row adds
    // 64 groups on (a wavefront's next unit): output rows and groups to add (and images), the bytes they are; what a carry
    // of the groups into the row and of the rows into the image adds to those
    uint32_t step_rows, step_groups, step_bytes, carry_row, carry_img;
    uint32_t spin_limit;
    uint32_t *wait_error;
    const uint16_t *wq;    // plan.expand: filter codes [column tile][fill][filter element 0..15][column 0..7], and the table
    const uint16_t *tableF;  // with the top bit of every byte flipped, filter-code major
    uint32_t wq_bytes;
    float *range;          // not null (mx_reports_range): kRangePairs pairs, smallest and largest output
    const float *addend;   // not null (mx_adds): a tensor like the output, added before the activation
};
// Launches that can add a tensor to their outputs: the simple store form, activations by one load.
inline bool mx_adds(const MxPlan &plan, const bool linear, const uint32_t pitch, const int co)
{
    return !plan.swap && plan.k_splits == 1 && linear && pitch == 4 && (co & 3) == 0;
}
// Launches that can report the range of their outputs: tall tiles, which layers of many outputs have, in the simple store form.
constexpr int kMxRangeUnits = 10;
inline bool mx_reports_range(const MxPlan &plan, const bool linear, const int co)
{
    return plan.units >= kMxRangeUnits && !plan.swap && plan.k_splits == 1 && linear && (co & 3) == 0;
}

// ---- direct_kernel.hip: a whole layer of few lookups in one launch ----
constexpr int kDirectThreads = 1024, kDirectWaves = kDirectThreads / 64;
constexpr int kDirectGatherWaves = 8;          // of which this many look up
constexpr int kDirectItems = 2;                // quads of filter elements of pixels, and of columns, a thread fetches at a time
constexpr int kDirectMaxItems = kDirectItems * (kDirectWaves - kDirectGatherWaves - 2) * 64;   // of a chunk that is not the only one
constexpr int kDirectLdsBytes = 163840;        // the table and 32 KiB for everything else
constexpr int kDirectBufferBytes = kDirectLdsBytes - kTableBytes - 3 * 64 * 4 - 2 * 64 * 4;   // both buffers of a chunk
constexpr int kDirectPixels[] = {16, 32, 64};  // pixels of a tile
constexpr int kDirectMaxColumns = 64;
constexpr int kDirectColumns[] = {1, 2, 3, 4, 6, 8};   // columns of a wavefront: the kernel's variants

struct DirectPlan {
    int pt, ct;            // pixels and columns of a tile
    int ncw, wc, wc_log;   // columns of a wavefront that looks up, and how many wavefronts side by side make the tile's
    int kc, kl, chunks;    // filter elements of a chunk and of a lane in it; chunks over the whole K
    int buffer_bytes;
    int n_row_tiles, n_col_tiles, grid;
    float us;              // what the planner's model expects of the launch; 0: the layer does not suit the kernel
};

struct DirectDiv {         // as MxDiv, but whole = 2^32 - 1 and mul = 0 where the divisor is one
    uint32_t mul, shift, whole;
};

struct DirectParams {
    DirectPlan plan;
    const float *x, *f, *bias;
    const uint16_t *tableT;
    float *out_f;
    int32_t *out_i;
    const float *addend;
    const LayerQuant *lq_dev;
    TensorQuant in_q, flt_q;
    float s1xs2, m1, m2, k_m1xm2;
    int relu;
    uint32_t x_bytes, f_bytes;
    int M, K, H, W, C, KW, Co, OH, OW, sh, sw, dh, dw, ph, pw;
    DirectDiv div_ow, div_oh, div_c, div_kw, div_kq, div_ct;   // kq: quads of a chunk
};

struct DepthwiseParams {
    int N, H, W, C, KH, KW, OH, OW, sh, sw, dh, dw, ph, pw;
    int64_t M;
    const float *x;         // NHWC raw input
    const uint8_t *wcodes;  // [KH*KW][C] filter codes
    const float *fsum;      // [C]
    const uint16_t *tableT;
    float *out_f;
    int32_t *out_i;
    TensorQuant in_q;            // quantization of the input (op entry points: from the host scalars)
    float s1xs2, m1, m2, k_m1xm2;
    const LayerQuant *lq_dev;    // not null (layer entry point): input quantization and epilogue constants from here
    const float *bias;           // not null: added per channel after the epilogue
    int relu;                    // 1: max(x, 0) last
    int stagger_sleeps;          // s_sleep(127) periods by which every second group of workgroups starts late (0: none)
    float *range;                // not null (depthwise_reports_range): kRangePairs pairs, smallest and largest output
};
bool depthwise_reports_range(const DepthwiseParams &p);

// Row permutation of the expanded table: logical activation code a lives in physical row
// (a >> 2) | ((a & 3) << 6), so that the four codes one lane transposes land in rows of
// alternating bank parity.
__host__ __device__ inline uint32_t phys_row(uint32_t a) { return (a >> 2) | ((a & 3u) << 6); }

// Device-side quantize: three separately rounded fp32 operations, truncation, clamp.
__device__ inline uint32_t quantize_code(float v, float offset, float inv_scale)
{
    float t = __fadd_rn(__fmul_rn(__fsub_rn(v, offset), inv_scale), 0.5f);
    t = t > 0.0f ? t : 0.0f;          // also maps NaN to 0
    t = t < 255.0f ? t : 255.0f;      // truncation of [255,256) is 255 as well
    return (uint32_t)t;
}

// Function attributes belong to a (kernel, device) pair and never change here: they are set on first use instead
// of before every launch (the runtime calls cost a few microseconds of host time each).
inline hipError_t set_max_dynamic_lds_once(const void *kernel, int bytes, bool require_no_static_lds = false)
{
    static std::mutex mu;
    static std::map<std::pair<const void *, int>, int> done;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return e;
    const std::pair<const void *, int> key(kernel, dev);
    {
        std::lock_guard<std::mutex> lock(mu);
        auto it = done.find(key);
        if (it != done.end() && it->second >= bytes)
            return hipSuccess;
    }
    if (require_no_static_lds) {
        hipFuncAttributes attr;
        e = hipFuncGetAttributes(&attr, kernel);
        if (e != hipSuccess)
            return e;
        if (attr.sharedSizeBytes != 0)
            return hipErrorInvalidConfiguration;
    }
    e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess)
        return e;
    std::lock_guard<std::mutex> lock(mu);
    done[key] = bytes;
    return hipSuccess;
}

// Brings a kernel's arguments (BYTES of them, at most six lines of 64) into the scalar cache at once.  They lie in host-visible
// memory, and used as the code comes to them every line is a round trip of its own, one after the other: LUT-GEMM launches of
// small layers 15.1 -> 14.6 us, 13.5 -> 13.1.
template <int BYTES>
__device__ __forceinline__ void fetch_arguments()
{
    constexpr int kLines = (BYTES + 63) / 64;
    static_assert(kLines >= 1 && kLines <= 6, "lines");
    const auto args = __builtin_amdgcn_kernarg_segment_ptr();
    uint32_t t[6];
    asm volatile("s_load_dword %0, %6, 0\n\ts_load_dword %1, %6, %7\n\ts_load_dword %2, %6, %8\n\t"
                 "s_load_dword %3, %6, %9\n\ts_load_dword %4, %6, %10\n\ts_load_dword %5, %6, %11\n\ts_waitcnt lgkmcnt(0)"
                 : "=&s"(t[0]), "=&s"(t[1]), "=&s"(t[2]), "=&s"(t[3]), "=&s"(t[4]), "=&s"(t[5])
                 : "s"(args), "n"((kLines > 1 ? 1 : 0) * 64), "n"((kLines > 2 ? 2 : 0) * 64), "n"((kLines > 3 ? 3 : 0) * 64),
                   "n"((kLines > 4 ? 4 : 0) * 64), "n"((kLines > 5 ? 5 : 0) * 64));
}

int device_cus();   // compute units of the current device (cached)
int device_lds_bytes();    // LDS one workgroup may take on the current device (cached)
double device_clock_hz();  // shader clock of the current device (cached)

// ---- launchers (each enqueues on `stream`; returns hipError_t of the launch) -----------------
hipError_t launch_quantize_relayout(const float *x, const ConvGeom &g, const TensorQuant &tq, const LayerQuant *lq_dev,
                                    const XqLayout &lay, uint32_t *xq, float *chsum, hipStream_t stream);
// With xq_fused / fused given, 1x1 stride-1 layers also get their quantized activations from this pass
// (*fused = true); the caller then skips launch_quantize_relayout.
// The filter pre-pass of the same layer (what launch_filter_pack would do), for a launch that can take it along.
struct FilterJob {
    const float *filter;
    const uint8_t *filter_codes;
    const DensePlan *plan;
    TensorQuant tq;
    uint16_t *wq;
    float *fsum;
    const uint16_t *tableT;   // with px_rows: the transposed table the pre-expanded rows are built from
    uint16_t *px_rows;        // nullptr: the layer does not run out of pre-expanded rows
    const MxPlan *mx;         // not null: the layer runs lutgemm_mx_kernel, whose rows those are
    uint32_t *swap_xq;        // mx->swap: the filter's codes as that kernel's input (wq: those of the patches)
};
// xq_fused / fused: the launch may also quantize the input into xq (then *fused is set);
// filter_job / filter_done: it may also do the filter pre-pass (then *filter_done is set), and with it build the
// pre-expanded rows that filter_job names (then *px_done is set).
hipError_t launch_patch_sums(const float *x, const ConvGeom &g, const TensorQuant &tq, const LayerQuant *lq_dev,
                             float *psum, hipStream_t stream, const XqLayout &lay, uint32_t *xq_fused = nullptr,
                             bool *fused = nullptr,
                             const FilterJob *filter_job = nullptr, bool *filter_done = nullptr,
                             int flat_row_bytes = 0,   // > 0: a fused xq is written in the flat layout
                             bool *px_done = nullptr);
// input_range: kRangePairs (smallest, largest) pairs of the input, which then is not read
hipError_t launch_layer_quant(const float *input, int64_t n_input, const float *filter, int64_t n_filter, int K,
                              float *partials, LayerQuant *lq_dev, hipStream_t stream, const float *input_range = nullptr);
constexpr int kMinMaxBlocks = 2048;   // partial (min, max) pairs per tensor in launch_layer_quant's scratch
// out[n][oh][ow][:] = in[n][oh * sh][ow * sw][:] for tensors of element_bytes-wide elements (C per pixel)
hipError_t launch_subsample(const void *in, int element_bytes, int N, int H, int W, int C, int sh, int sw, int OH, int OW,
                            void *out, hipStream_t stream);
hipError_t launch_codes_relayout(const uint8_t *codes, const ConvGeom &g, const XqLayout &lay, uint32_t zp4, uint32_t *xq,
                                 hipStream_t stream);
// Flat layout of xq: rows of row_bytes bytes, pad_left pixels of the zero-point code, the W pixels' codes, zero-point
// codes up to the end of the row; one more row of zero-point codes behind the last image.  From floats (x) or codes.
hipError_t launch_quantize_flat_rows(const float *x, const uint8_t *codes, const ConvGeom &g, const XqLayout &lay,
                                     int pad_left, int row_bytes, const TensorQuant &tq, const LayerQuant *lq_dev, uint8_t *xq,
                                     hipStream_t stream);
// tableT / px_rows / px_done: the launch may also build the pre-expanded rows of the layer (then *px_done is set)
hipError_t launch_filter_pack(const float *filter, const uint8_t *filter_codes, const ConvGeom &g,
                              const DensePlan &plan, const MxPlan *mx, const TensorQuant &tq, const LayerQuant *lq_dev,
                              uint16_t *wq, float *fsum, hipStream_t stream, const uint16_t *tableT = nullptr,
                              uint16_t *px_rows = nullptr, bool *px_done = nullptr);
hipError_t launch_quantize_flat(const float *v, int64_t n, float offset, float inv_scale, uint8_t *codes,
                                hipStream_t stream);
hipError_t launch_dense(const DenseParams &p, bool out_i32, hipStream_t stream);
// the same layer out of pre-expanded rows: launch_px_expand_rows builds p.px_rows from the packed filter codes
hipError_t launch_px_expand_rows(const uint16_t *wq, const uint16_t *tableT, const DensePlan &plan, uint16_t *rows,
                                 hipStream_t stream);
hipError_t launch_dense_px(const DenseParams &p, bool out_i32, hipStream_t stream);
bool px_free_running(const DensePlan &plan, int taps);   // the plan runs lutgemm_pxf_kernel (no barrier between fills)
hipError_t launch_mx_expand_rows(const float *filter, const uint8_t *filter_codes, const ConvGeom &g, const MxPlan &plan,
                                 const TensorQuant &tq, const LayerQuant *lq_dev, const uint16_t *tableT, uint16_t *rows,
                                 hipStream_t stream);
// xq by tap columns, [image row][tap column][quad][output column], for lutgemm_mx_kernel at a stride
hipError_t launch_split_columns(const uint32_t *xq, const ConvGeom &g, const XqLayout &lay, uint32_t *planes, hipStream_t stream);
// mx->swap, where no other launch has done it: both operands packed, from floats or codes; and the pass behind the LUT-GEMM,
// which adds the K splits' [Co][M] sums (rows of m_pitch), turns them and applies the op's epilogue
hipError_t launch_swap_pack(const float *x, const uint8_t *codes, const float *filter, const uint8_t *filter_codes,
                            const ConvGeom &g, const TensorQuant &tq_in, const TensorQuant &tq_f, const LayerQuant *lq_dev,
                            uint32_t *xq, uint16_t *wq, hipStream_t stream);
// out = activation(out + addend), n values
hipError_t launch_add(float *out, const float *addend, int64_t n, bool relu, hipStream_t stream);
// max(s, 0) as the networks' residual sums have it: NaN stays, and -0 becomes 0
__device__ __forceinline__ float sum_activation(const float s, const int relu)
{
    return relu && s <= 0.0f ? 0.0f : s;
}
hipError_t launch_swap_epilogue(const DenseParams &p, const int32_t *partials, int k_splits, int m_pitch, float *out_f,
                                int32_t *out_i, hipStream_t stream);
hipError_t launch_dense_mx(const MxParams &p, hipStream_t stream);          // out of pre-expanded rows
hipError_t launch_dense_mx_expand(const MxParams &p, hipStream_t stream);   // plan.expand
hipError_t launch_direct(const DirectParams &p, hipStream_t stream);
hipError_t launch_splitk_epilogue(const DenseParams &p, const int32_t *partials, float *out_f, int32_t *out_i,
                                  hipStream_t stream);
// tf1 AxConv2D: what the zero points add to the sums of products, per output pixel and per output column; and the pass
// that adds them to finished sums (lutgemm_mx_kernel does so as it stores)
hipError_t launch_axconv_terms(const uint8_t *codes, const uint8_t *fcodes, const ConvGeom &g, int offset_input,
                               int offset_filter, int32_t *pixel_term, int32_t *column_term, hipStream_t stream);
// All three at once for lutgemm_mx_kernel's layers given as codes (*done = false: not for this one; nothing was launched):
// relayout, filter packing or rows, and with `terms` those of the zero points.
hipError_t launch_codes_prep(const uint8_t *codes, const uint8_t *fcodes, const ConvGeom &g, const XqLayout &lay, uint32_t zp4,
                             uint32_t *xq, const MxPlan &mx, uint16_t *wq, const uint16_t *tableT, uint16_t *rows, bool terms,
                             int offset_input, int offset_filter, int32_t *pixel_term, int32_t *column_term, hipStream_t stream,
                             bool *done);
hipError_t launch_axconv_correction(const ConvGeom &g, const int32_t *pixel_term, const int32_t *column_term, int32_t *out,
                                    hipStream_t stream);
hipError_t launch_fill_u32(uint32_t *dst, int64_t n, uint32_t value, hipStream_t stream);
hipError_t launch_depthwise_filter(const float *filter, int taps, int C, const TensorQuant &tq,
                                   const LayerQuant *lq_dev, uint8_t *wcodes, float *fsum, hipStream_t stream);
hipError_t launch_depthwise(const DepthwiseParams &p, bool out_i32, int grid, hipStream_t stream);
hipError_t run_lds_gather_peak(double *lookups_per_second, hipStream_t stream, bool stream_b128);
hipError_t run_valu_issue_peak(double *lane_ops_per_second, int mix, hipStream_t stream);
hipError_t run_lookup_mix_peak(double *lookups_per_second, hipStream_t stream);

} // namespace axc
