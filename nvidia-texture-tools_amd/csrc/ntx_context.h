// ntx_context.h -- internal: the context behind the C ABI handle and the
// helpers shared by the translation units of libntx_hip (ntx_api.cpp,
// batch_api.cpp).  Not installed; the public interface is include/ntx_hip.h.
#pragma once

#include <map>
#include <string>
#include <tuple>
#include <vector>

#include "ntx_common.h"

namespace ntx {
hipError_t launch_bc1(const Bc1Target *images, int n, int alpha_mode, const float *cw, const Tables *d_tab,
                      hipStream_t stream, bool urgent = false, int level = 8);
// icbc Level8 in two passes, one block per lane (large images); d_counts:
// bucket scratch of bc1_scratch_ints(blocks) ints with zero tallies.
hipError_t launch_bc1_classify(const float *d_src, int w, int h, int alpha_mode, const Tables *d_tab, void *d_out,
                               int16_t *d_nm, int *d_counts, int *d_lists, hipStream_t stream, bool urgent);
hipError_t launch_bc1_list(const float *d_src, int w, int h, int alpha_mode, const float *cw, const Tables *d_tab,
                           void *d_out, const int *d_list, const int *d_count, int cap, int max_groups,
                           hipStream_t stream);
hipError_t launch_bc1_search(const float *d_src, int w, int h, int alpha_mode, const float *cw, const Tables *d_tab,
                             void *d_out, int16_t *d_nm, int *d_counts, const int *d_lists, int cap, int cus,
                             hipStream_t stream);
// The multi-image two-pass BC1 encoder (Level8) over a table of images:
// at most bc1_multi_max_images() images of at most bc1_multi_max_blocks()
// blocks; d_map: (image, first block) per 256-block chunk.
int bc1_multi_max_images();
int bc1_multi_max_blocks();
hipError_t launch_bc1_classify_multi(const Bc1Image *d_imgs, const void *d_map, int nchunks, const Tables *d_tab,
                                     int *d_counts, int *d_lists, int cap, hipStream_t stream);
hipError_t launch_bc1_search_multi(const Bc1Image *d_imgs, int nimgs, const Tables *d_tab, int *d_counts,
                                   const int *d_lists, int cap, int cus, hipStream_t stream);
// Workgroups (four wavefronts each) per compute unit for the OptimalCompress
// searches: a grid-stride loop over the blocks.
constexpr int kOptimalGroupsPerCU = 8;
int bc1_scratch_ints(int nblocks);
// Zeros n ints at p.
hipError_t launch_batch_reset(int *p, int n, hipStream_t stream);
hipError_t launch_bc1_classify_set(const Bc1Target *images, int n, int alpha_mode, const float *cw, const Tables *d_tab,
                                   int *d_counts, int cap, hipStream_t stream);
hipError_t launch_bc1_search_set(const Bc1Target *images, int n, int alpha_mode, const float *cw, const Tables *d_tab,
                                 int *d_counts, int cap, int cus, hipStream_t stream);
hipError_t launch_channels(const float *d_src, int w, int h, int format, void *d_out, hipStream_t stream,
                           bool urgent = false);
hipError_t launch_bc3_front(const float *d_src, int w, int h, const Tables *d_tab, void *d_out, int *d_counts,
                            int *d_lists, int cap, int weight_by_alpha, uint32_t *d_packed, bool urgent,
                            hipStream_t stream, bool normal = false);
hipError_t launch_bc3_clear_counts(int *d_counts, hipStream_t stream);
hipError_t launch_bc1a(const float *d_src, int w, int h, int weight_by_alpha, const float *cw, const Tables *d_tab,
                       void *d_out, int *d_counts, int *d_lists, int cap, uint32_t *d_packed, hipStream_t stream);
hipError_t launch_optimal_channels(const float *d_src, int w, int h, int format, void *d_out, int groups,
                                   hipStream_t stream);
hipError_t launch_optimal_green(const float *d_src, int w, int h, const Tables *d_tab, void *d_out, int groups,
                                hipStream_t stream);
hipError_t launch_bc3_fast(const float *d_src, int w, int h, bool normal, const Tables *d_tab, void *d_out,
                           hipStream_t stream);
hipError_t launch_bc3_search(const uint32_t *d_packed, int w, int h, int weight_by_alpha, const float *cw, void *d_out,
                             int *d_counts, const int *d_lists, int cap, const Tables *d_tab, int lpb_shift,
                             bool urgent, hipStream_t stream);
int bc3_scratch_ints(int nblocks);
int bc3_lists_offset();
int bc3_packed_offset(int nblocks);
hipError_t launch_box(const float *d_src, int W, int H, float *d_dst, hipStream_t stream);
hipError_t launch_poly_x(const float *d_src, int W, int H, float *d_tmp, const float *d_kx, const int *d_lx, int wx, int wrap,
                         hipStream_t stream);
hipError_t launch_poly_y(const float *d_tmp, int W, int H, float *d_dst, const float *d_ky, const int *d_ly, int wy, int wrap,
                         hipStream_t stream);
hipError_t launch_mip_tail(const float *d_src, const MipTail &tail, int wrap, hipStream_t stream);
// Exact halving with the same taps for every output (PolyDev::uniform) in
// both directions, an odd window of 3 to 15 taps: host weights kx, ky,
// first taps lx0, ly0 of output 0, strips of `rows` output rows
// (poly_slide_rows: 0 when the tiled kernel suits the size better).
int poly_slide_rows(int W, int H, int cus);
hipError_t launch_poly_slide(const float *d_src, int W, int H, float *d_dst, const float *kx, int lx0, const float *ky,
                             int ly0, int win, int wrap, int rows, hipStream_t stream);
hipError_t launch_poly_fused(const float *d_src, int W, int H, float *d_dst, const float *d_kx, const int *d_lx, int wx,
                             bool pair_x, const float *d_ky, const int *d_ly, int wy, int wrap, hipStream_t stream);
bool poly_fused_fits(int max_sw, int max_sh, int wx, int wy);
// The fused kernel without tables, for exact halving with uniform taps
// (PolyDev::uniform) of a window poly_fused_uniform_window accepts.
bool poly_fused_uniform_window(int win);
hipError_t launch_poly_fused_uniform(const float *d_src, int W, int H, float *d_dst, const float *kx, int lx0,
                                     const float *ky, int ly0, int win, int wrap, hipStream_t stream);

int poly_tile_x();
int poly_tile_y();
hipError_t launch_srgb(float *d, size_t n, const float *d_lut, hipStream_t stream);
// d_srgb_lut: NULL, or the 256-entry sRGB->linear table to convert R, G, B as well.
hipError_t launch_unpack(const uint8_t *d_bgra, size_t n, float *d_dst, const float *d_srgb_lut, hipStream_t stream);
// Levels for one gamma launch: texels[l] = w * h of level l; start[] is
// filled by launch_gamma.
constexpr int kMaxGammaLevels = 16;
struct GammaJob {
    const float *src[kMaxGammaLevels];
    float *dst[kMaxGammaLevels];
    unsigned long long texels[kMaxGammaLevels];
    unsigned long long start[kMaxGammaLevels + 1];
    int levels;
};
// mode 0: gamma 2.2 -> linear (table form), 1: linear -> gamma 2.2 (table
// form), 2: powf(max(0, x), power).
hipError_t launch_gamma(const GammaJob &job, int mode, float power, const Tables *d_tab, hipStream_t stream);
// [expandNormals +] normalizeNormalMap [+ packNormals] on the R, G, B planes of n texels.
hipError_t launch_normals(float *d_rgba, size_t n, bool expand_pack, hipStream_t stream);
hipError_t launch_bc1_sse(const float *d_src, int w, int h, const void *d_blocks, double *d_partial, double *d_out,
                          hipStream_t stream);
int bc1_sse_partials(int w, int h);
hipError_t launch_decode(int format, int d3d9, const void *d_blocks, int w, int h, float *d_dst, hipStream_t stream);
int rms_partials();
hipError_t launch_rms(const float *d_ref, const float *d_img, size_t n, int mode, double *d_partial, double *d_out,
                      hipStream_t stream);

struct DevBuf {
    void *ptr = nullptr;
    size_t cap = 0;
};

struct PolyDev {
    float *weights = nullptr;
    int *left = nullptr;
    int window = 0;
    int span_x = 0;  // largest source span of a run of poly_tile_x() outputs
    int span_y = 0;  // same for poly_tile_y() outputs
    bool stride2 = false;  // left[i] == left[0] + 2 i for every output i
    // stride2 and every output's weights equal output 0's (bit for bit):
    // exact halving, whose taps left0, w0[0 .. window) the sliding-window
    // kernel takes as arguments.
    bool uniform = false;
    int left0 = 0;
    float w0[16] = {};
    // Host copies of the weights and first taps (the tail's packed taps).
    std::vector<float> host_weights;
    std::vector<int> host_left;
};

using PolyKey = std::tuple<int, uint32_t, uint32_t, uint32_t, int, int>;
// Tail taps: filter, width, alpha, stretch bits, source W, H, levels, wrap.
using TailKey = std::tuple<int, uint32_t, uint32_t, uint32_t, int, int, int, int>;
struct TailTaps {
    float *packed = nullptr;  // device, 2 floats per tap
    int count = 0;
};

}  // namespace ntx

struct ntx_hip_context {
    int device = 0;
    int cus = 256;  // compute units of the device
    hipStream_t stream = nullptr;
    ntx::Tables *d_tab = nullptr;
    float *d_srgb = nullptr;
    // 8-bit -> linear table of ntx_hip_unpack_bgra8_gamma_device for the
    // gamma whose float bits are gamma_lut_key (valid when d_gamma_lut set).
    float *d_gamma_lut = nullptr;
    uint32_t gamma_lut_key = 0;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    ntx::DevBuf in, out, tmp, dst, bucket, metric;
    void *host_result = nullptr;  // pinned, see host_result() below
    // Bytes of the DevBuf scratch above (and `chain`) now allocated, and the
    // cap set by ntx_hip_set_scratch_limit (0: none).
    size_t scratch_bytes = 0, scratch_limit = 0;
    // BC1 images of at least this many blocks take the two-pass encoder.
    static constexpr int kBc1LanesMinDefault = 1 << 17;
    int bc1_lanes_min = kBc1LanesMinDefault;
    // Unless that threshold was set: an image of fewer blocks, but at least
    // this many, or a set of images of at least that many together, takes the
    // two-pass encoder too where its scratch is free to be had
    // (optional_bc1_bucket), and the one-pass one otherwise.  Which is faster
    // lies with the content, which the host does not know: the lines are where
    // no content measured takes more than 1.02 times what images of their own
    // launches took before there was a choice.  One-pass and two-pass calls in
    // us, noise with rectangles, random texels, gradients, four colours a
    // block, dark texels: 65,536 blocks 198 and 148, 224 and 266, 202 and 225,
    // 76 and 74, 184 and 193; 82,944 blocks 221 and 212, 282 and 326, 253 and
    // 246, 97 and 80, 240 and 303; 102,400 blocks 259 and 199, 339 and 356, 304
    // and 285, 115 and 85, 285 and 302; 131,044 blocks 291 and 212, 429 and 363,
    // 386 and 322, 148 and 100, 363 and 374.  Chains of 74,261 blocks, one
    // launch either way: 191 and 174, 257 and 299, 231 and 246, 105 and 85, 220
    // and 283; of 87,383: 265 and 205, 302 and 331, 272 and 258, 122 and 84, 257
    // and 311.
    static constexpr int kBc1LanesOptional = 96 << 10, kBc1LanesOptionalSet = 80 << 10;
    // The BC3 tallies at the start of `bucket` are zero: set after a complete
    // front + search sequence (the search clears them), cleared before one.
    bool bc3_counts_zero = false;
    // The optional two-pass encoder's scratch and whether its tallies are
    // zero.  Apart from the buffers above, so that a call that does without it
    // neither moves memory that a recorded graph holds nor counts towards a
    // scratch limit set later, which also gives it back.
    ntx::DevBuf optional;
    bool optional_counts_zero = false;
    // Concurrent compression of several images (mip chains, image sets):
    // the side streams, fork/join events, and per-image BC3 scratch (every
    // region's tallies zero when chain_counts_zero).
    static constexpr int kSideStreams = 2;
    hipStream_t side[kSideStreams] = {};
    std::vector<hipEvent_t> sync_events;
    ntx::DevBuf chain;
    bool chain_counts_zero = false;
    std::vector<size_t> chain_layout;  // offsets (ints) of the regions with tallies in the last complete run
    std::map<ntx::PolyKey, ntx::PolyDev> poly;
    std::map<ntx::TailKey, ntx::TailTaps> tail_taps;
    std::map<std::string, ntx_batch_tuning> batch_tuning;  // autotuned, keyed by batch shape list
    std::string err;
    // per-kernel event timing (ntx_hip_profile_*)
    bool profiling = false;
    struct Mark { int kernel; hipEvent_t start, stop; };
    std::vector<Mark> marks;
    std::vector<hipEvent_t> spare;
};

namespace ntx {

ntx_status fail(ntx_hip_context *ctx, hipError_t e, const char *what);
ntx_status bind(ntx_hip_context *ctx);
ntx_status ensure(ntx_hip_context *ctx, DevBuf &b, size_t bytes);
// The context's pinned memory for what a call's last kernel hands to the host,
// kHostResultBytes of it, written after the call's work on the stream and read
// after its one wait: a copy into the caller's pageable memory takes 10 to
// 18 us for a few bytes.
constexpr size_t kHostResultBytes = 64 << 10;
ntx_status host_result(ntx_hip_context *ctx, void **p);
// Frees a buffer ensure() allocated (and takes it off the scratch count).
void release(ntx_hip_context *ctx, DevBuf &b);
hipEvent_t take_event(ntx_hip_context *ctx);
// Quality levels handled exactly by the kernels.
bool supported(int format, int quality);
// icbc quality level of a BC1 nvtt quality (1, 8 or 9).
int bc1_level(int quality);
// BC1 at this quality and size takes the two-pass (lane per block) encoder.
bool bc1_two_pass(const ntx_hip_context *ctx, int quality, int w, int h);
// Bucket scratch (ints) one image's compression needs: BC3, two-pass BC1.
size_t scratch_ints(const ntx_hip_context *ctx, int format, int quality, int w, int h);
// One image's compression on the context's stream with the given bucket
// scratch (null: BC1 takes its one-pass encoder); the tallies are cleared by
// a fill kernel first.
ntx_status side_stream_after(ntx_hip_context *ctx, int i, hipStream_t *out);
ntx_status side_stream_done(ntx_hip_context *ctx, int i, hipEvent_t *out);
ntx_status side_plain_bc1(ntx_hip_context *ctx, int n, const float *const *d_in, const int *w, const int *h,
                          void *const *d_out, hipEvent_t *join);
hipError_t compress_scratch(ntx_hip_context *ctx, int format, int quality, int alpha_mode, const float *cw,
                            const float *d_rgba, int w, int h, void *d_out, int *bucket);
// Looks up the device address of the no-allocation entry point's scratch
// array on the context's (current) device; once per device.
ntx_status noalloc_init(ntx_hip_context *ctx);
// Polyphase weights and first-tap indices for src -> dst samples, cached per context.
ntx_status poly_tables(ntx_hip_context *ctx, int filter, float width, const float *params, int src, int dst, PolyDev **out);

// Runs one launch; brackets it with events when the context is profiling.
// Runs `launch` (which enqueues on `stream`), bracketed by profiling events
// on that stream when profiling is on.
template <typename F>
hipError_t timed_on(ntx_hip_context *ctx, hipStream_t stream, int kernel, F &&launch)
{
    if (!ctx->profiling) return launch();
    hipEvent_t a = take_event(ctx), b = take_event(ctx);
    if (!a || !b) return hipErrorOutOfMemory;
    hipError_t e = hipEventRecord(a, stream);
    if (e == hipSuccess) e = launch();
    if (e == hipSuccess) e = hipEventRecord(b, stream);
    ctx->marks.push_back({ kernel, a, b });
    return e;
}

template <typename F>
hipError_t timed(ntx_hip_context *ctx, int kernel, F &&launch)
{
    return timed_on(ctx, ctx->stream, kernel, static_cast<F &&>(launch));
}

}  // namespace ntx

#define NTX_HIP(ctx, call)                                      \
    do {                                                        \
        hipError_t e_ = (call);                                 \
        if (e_ != hipSuccess) return ntx::fail(ctx, e_, #call); \
    } while (0)
