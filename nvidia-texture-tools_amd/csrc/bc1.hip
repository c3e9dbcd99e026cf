// bc1.hip -- BC1 encoder for gfx950, bit-exact with NVTT's CPU path
// (icbc v1.05 compress_dxt1 at Quality_Level8; Level9 for Quality_Production,
// Level1 for Quality_Fastest), icbc.h:3485-3559.
//
// Two mappings:
//  * bc1_kernel: 16-lane groups, sixteen per 256-thread workgroup
//    (bc1_block.hpp), one or more per 4x4 block; used for small images, the
//    other quality levels and as the reference form.
//  * bc1_classify_kernel + bc1_search_kernel (Level8): 1 to 8 lanes per
//    block.  The classify pass reduces each block's colours, finishes blocks
//    of 0 or 1 colours and appends the others to the list of their colour
//    count n; the search pass takes whole wavefronts from one list, so every
//    lane runs the same loops over the partitions (bc1_lane.hpp) with scalar
//    loop control and, for unit-weight blocks, the candidates' weight terms
//    from tables.  Over one image, or over the images of a table.
#include "bc1_lane.hpp"
#include "bucket.hpp"

namespace {

using namespace ntx_bc1;

// One image of a bc1_kernel launch: its blocks start at workgroup `first`,
// each on `parts` 16-lane groups.
struct Bc1Job {
    const float *src;
    uint2 *out;
    short2 *nm;
    int w, h, bw, blocks, first, parts;
};
struct Bc1Jobs {
    int n;
    Bc1Job job[ntx::kBc1MaxImages];
};
// The image of a workgroup.
__device__ __forceinline__ const Bc1Job &job_of(const Bc1Job &job, int) { return job; }
__device__ __forceinline__ const Bc1Job &job_of(const Bc1Jobs &jobs, int group)
{
    int j = 0;
    while (j + 1 < jobs.n && group >= jobs.job[j + 1].first) j++;
    return jobs.job[j];
}

// Jobs: Bc1Job, one image, whose fields are loaded together at the start, or
// Bc1Jobs.
//
// Level 9 is held to eight wavefronts a SIMD (64 registers, without spills);
// left to itself the compiler takes 84 for one image and 64 to 66 for several,
// with every size slower: Production of 700 x 300, 2048^2 and 4096^2 136,
// 1,242 and 4,120 us with 84 of them, 128, 1,178 and 3,775 us so.  Level 8 has
// the LDS of its term tables for four; Level 1 is left alone (held to eight
// 8192^2 takes 1,645 us, not 1,600).
template <int LEVEL, class Jobs>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(LEVEL == 9 ? 8 : LEVEL == 8 ? 4 : 1)))
void bc1_kernel(Jobs jobs, int alpha_mode, float cwx, float cwy, float cwz,
                                                  const ntx::Tables *__restrict__ tab, int urgent)
{
    if (urgent) __builtin_amdgcn_s_setprio(3);
    __shared__ Bc1Shared sh;
    __shared__ TermTables s_terms;
    const Bc1Job &im = job_of(jobs, int(blockIdx.x));
    const int g = threadIdx.x >> 4;
    const int lane = threadIdx.x & 15;
    const int parts = LEVEL == 8 ? im.parts : 1;
    // A block on a whole workgroup searches in five trips: fewer than the
    // term tables' 18 KB are worth.  Level 9 spends its time in the refinement
    // and wants the wavefronts that the tables would cost it.
    const bool use_terms = LEVEL == 8 && parts < kBlocksPerWG;
    load_shared_tables(sh, tab, threadIdx.x, blockDim.x);
    if (use_terms) load_term_tables(s_terms, tab, threadIdx.x, blockDim.x);
    __syncthreads();

    const int blk = ((int(blockIdx.x) - im.first) * kBlocksPerWG + g) >> __builtin_ctz(parts);  // 1, 4 or 16
    if (blk >= im.blocks) return;  // every group of a block leaves together
    const Parts ps{ g & (parts - 1), parts };
    int n, m;
    const uint2 result = encode_block<LEVEL>(sh, im.src, im.w, im.h, blk % im.bw, blk / im.bw, alpha_mode, cwx, cwy, cwz,
                                             tab, g, lane, &n, &m, true, ps, use_terms ? &s_terms : nullptr);
    if (lane == 0 && ps.part == 0) {
        im.out[blk] = result;
        if (im.nm) im.nm[blk] = make_short2(short(n), short(m));
    }
}

// The blocks listed in list[0, min(*count, cap)) (indices below cap), one
// per 16-lane group as bc1_kernel encodes them, the groups striding over the
// list.  The encoder synchronises only within a wavefront, so groups may
// finish their strides at different times.  For short lists (the learned
// form's fallback blocks) this has a group's latency, where the one-block-
// per-lane search pass has a whole block's search per lane.
template <int LEVEL>
__global__ __launch_bounds__(256) void bc1_list_kernel(const float *__restrict__ src, int w, int h, int bw,
                                                       const int *__restrict__ list, const int *__restrict__ count,
                                                       int cap, int alpha_mode, float cwx, float cwy, float cwz,
                                                       const ntx::Tables *__restrict__ tab, uint2 *__restrict__ out)
{
    __shared__ Bc1Shared sh;
    load_shared_tables(sh, tab, threadIdx.x, blockDim.x);
    __syncthreads();
    const int g = threadIdx.x >> 4;
    const int lane = threadIdx.x & 15;
    const int items = min(*count, cap);
    for (int item = blockIdx.x * kBlocksPerWG + g; item < items; item += gridDim.x * kBlocksPerWG) {
        const int blk = list[item];
        if (unsigned(blk) >= unsigned(cap)) continue;  // the whole group skips it
        int n, m;
        const uint2 result =
            encode_block<LEVEL>(sh, src, w, h, blk % bw, blk / bw, alpha_mode, cwx, cwy, cwz, tab, g, lane, &n, &m);
        if (lane == 0) out[blk] = result;
    }
}

// LDS of a classify workgroup (four wavefronts).
struct ClassifyShared {
    float4 rows[4][16][64];
    int cnt[ntx_bucket::kCountSlots], base[ntx_bucket::kCountSlots];
};

// One block of a classify pass per thread; the whole workgroup calls it.
__device__ __forceinline__ void classify_chunk(const float *__restrict__ src, int w, int h, int bw, int nblocks,
                                               int alpha_mode, const ntx::Tables *__restrict__ tab,
                                               uint2 *__restrict__ out, short2 *__restrict__ nm,
                                               int *__restrict__ counts, int *__restrict__ lists, int cap, int rows16,
                                               ClassifyShared &sh, int blk, int tag = 0)
{
    using namespace ntx_bucket;
    const int t = threadIdx.x, lane = t & 63;
    if (t < kCountSlots) sh.cnt[t] = 0;
    __syncthreads();
    int k = 0, local = -1;
    if (blk < nblocks) {
        LaneRows rows = sh.rows[t >> 6];
        const int n = classify_reduce(rows, lane, BlockTexels(src, w, h, blk % bw, blk / bw, alpha_mode, rows16 != 0));
        if (n <= 1) {
            uint2 r = make_uint2(0u, 0u);
            if (n == 1) {
                const float4 c = rows[0][lane];
                r = single_color_block(tab, c.x, c.y, c.z);
            }
            out[blk] = r;
            if (nm) nm[blk] = make_short2(short(n), short(-1));
        } else {
            k = n;
            local = atomicAdd(&sh.cnt[n], 1);
        }
    }
    append_to_lists(sh.cnt, sh.base, counts, lists, cap, k, local, tag | blk);
}

// Level8 pass 1, one block per lane: FloatColorCompressor's gather and
// reduce_colors; a block of no colour (every weight 0) is the zero block, a
// block of one colour compress_dxt1_single_color_optimal (icbc.h:3515-3525),
// every other block goes to list n.  The clusters live in LDS only while
// they are counted.  (Clusters as three columns without weights, 48 KB a
// workgroup and three wavefronts a SIMD, took 510 us at 8192^2 where this took
// 460, and takes 482: the LDS reads, one of 16 bytes here, are what it waits
// for.)
__global__ __launch_bounds__(256) void bc1_classify_kernel(const float *__restrict__ src, int w, int h, int bw, int nblocks,
                                                           int alpha_mode, const ntx::Tables *__restrict__ tab,
                                                           uint2 *__restrict__ out, short2 *__restrict__ nm,
                                                           int *__restrict__ counts, int *__restrict__ lists, int rows16,
                                                           int urgent)
{
    if (urgent) __builtin_amdgcn_s_setprio(3);
    __shared__ ClassifyShared sh;
    classify_chunk(src, w, h, bw, nblocks, alpha_mode, tab, out, nm, counts, lists, nblocks, rows16, sh,
                   blockIdx.x * 256 + threadIdx.x);
}

// The image a search lane encodes a block of: the single image of a launch
// (the same in every lane) or the image its list entry names.
struct LaneImage {
    const float *src;
    uint2 *out;
    int w, h, bw, alpha_mode, rows16;
    float cwx, cwy, cwz;
};

// Block blk of image im, of k colours, by the S lanes of column col (sub:
// this lane's number among them) of a wavefront whose blocks all have k
// colours; written when live (lanes past the end of their list encode the
// wave's first block again, with the same count and valid weights, and
// discard it).
__device__ __forceinline__ void search_lane(const LaneImage &im, int blk, bool live,
                                            const ntx::Tables *__restrict__ tab, short2 *__restrict__ nm,
                                            LaneRows rows, int col, int sub, int S, int k, const SearchTables &st)
{
    const BlockTexels texels(im.src, im.w, im.h, blk % im.bw, blk / im.bw, im.alpha_mode, im.rows16 != 0);
    Reduced red = lane_reduce(rows, col, texels, k);
    const int n = red.n;  // == k in live lanes
    const float mx = im.cwx * im.cwx, my = im.cwy * im.cwy, mz = im.cwz * im.cwz;
    // What holds for every live lane of the wavefront: values whose errors
    // are finite (metric included), and of those, texels that all weigh 1
    // (so that the cluster weights are integer counts) under the metric 1.
    const bool tame = __builtin_amdgcn_ballot_w64(live && !(red.tame && mx <= 1e15f && my <= 1e15f && mz <= 1e15f)) == 0;
    const bool units = tame && __builtin_amdgcn_ballot_w64(live && !(red.unit && mx == 1.0f && my == 1.0f && mz == 1.0f)) == 0;
    const bool rebuild = red.any_black && lane_has_black_cluster(rows, col, n);
    const float *mid5 = st.mid5, *mid6 = st.mid6, *div255 = st.div255;

    // Four colours over the block's clusters, then three colours over the
    // same or the non-black ones.
    uint2 result = make_uint2(0u, 0u);
    float best = FLT_MAX;
    int m = n;
    float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    bool run3 = true;
#pragma unroll 1
    for (int pass = 0; pass < 2; pass++) {
        if (pass == 1 && rebuild) {
            lane_reduce(rows, col, texels, k);
            m = lane_skip_blacks(rows, col, n);
            run3 = m > 0;
        }
        if ((pass == 0 || rebuild) && m > 0) sum = lane_sat(rows, col, m, tame);
        uint2 r;
        float e;
        if (pass == 0) {
            Best b;
            if (tame) {
                TameBest tb;
                if (S == 1 && units && k == 16)
                    search4<true, Terms::kScalar>(rows, col, 0, 1, 16, sum, mx, my, mz,
                                                  reinterpret_cast<const float4 *>(tab->bc1h4), tb);
                else if (S == 1 && units)
                    search4<true, Terms::kTable>(rows, col, 0, 1, k, sum, mx, my, mz, st.terms.four, tb);
                else if (units)
                    search4<false, Terms::kTable>(rows, col, sub, S, k, sum, mx, my, mz, st.terms.four, tb);
                else
                    search4<false, Terms::kComputed>(rows, col, sub, S, k, sum, mx, my, mz, st.terms.four, tb);
                tb.combine(S);
                offer_past_end(terms_c(k + 1) - 1, tb);
                b = tb.best();
            } else {
                b = search4_any(rows, col, k, sum, mx, my, mz);
            }
            e = lane_output<true>(lane_winner<true>(rows, col, b, sum, mx, my, mz, st), texels, im.cwx, im.cwy,
                                  im.cwz, mid5, mid6, div255, &r);
        } else {
            const bool units3 = units && __builtin_amdgcn_ballot_w64(live && run3 && sum.w != 16.0f) == 0;
            if (!run3) break;
            Best b;
            if (tame) {
                TameBest tb;
                if (units3)
                    search3<false, Terms::kTable>(rows, col, sub, S, m, sum, mx, my, mz, st.terms.three, tb);
                else
                    search3<false, Terms::kComputed>(rows, col, sub, S, m, sum, mx, my, mz, st.terms.three, tb);
                tb.combine(S);
                offer_past_end((m + 1) * (m + 2) / 2 - 1, tb);
                b = tb.best();
            } else {
                b = search3_any(rows, col, m, sum, mx, my, mz);
            }
            e = lane_output<false>(lane_winner<false>(rows, col, b, sum, mx, my, mz, st), texels, im.cwx, im.cwy,
                                   im.cwz, mid5, mid6, div255, &r);
        }
        if (pass == 0 || e < best) { best = e; result = r; }
    }
    if (!(best < FLT_MAX)) result = make_uint2(0u, 0u);
    if (live && sub == 0) {
        im.out[blk] = result;
        if (nm) nm[blk] = make_short2(short(n), short(run3 ? m : -1));
    }
}

// Wavefronts of a search workgroup: with the term tables they fill a compute
// unit's LDS (two wavefronts a SIMD, at their registers the most there are).
constexpr int kSearchWaves = 8;

// A search's lists cut into wavefronts: of each list the first entries into
// wavefronts of 64 >> s blocks, the others into finer ones.  The lists are
// walked from count 16 down, first the coarse wavefronts, whole rounds of the
// grid's, then the finer ones: one long wavefront too many would take as long
// as a round, short ones fill in (blocks of 16 random texels, 65,536 and
// 262,144 of them: 339 and 889 us with one cut for all, 266 and 716 so).
//
// Runs 0 to 14 are the coarse wavefronts of lists 16 to 2, 15 to 29 the finer
// ones.
constexpr int kRuns = 30;
struct ListRuns {
    int start[32];  // first wavefront
    int first[32];  // first entry
    int list[32];   // list | s << 8
    int count[32];  // entries of the list
    int total;      // wavefronts
    float end[32];
};

// How long a wavefront of list n at 1 << s lanes per block takes, in trips of
// a candidate: both fits' and the set-up.
constexpr int wave_trips(int n, int s)
{
    int t = 120;
    for (int b = 0; b <= n; b++) t += ((b >> s) + 1) * (n - (b > 1 ? b : 1) + 1 + (b > 0 ? 1 : 0));
    return t;
}
struct TripTable {
    uint16_t t[17][4] = {};
};
constexpr TripTable trip_table()
{
    TripTable r;
    for (int n = 2; n <= 16; n++)
        for (int s = 0; s < 4; s++) r.t[n][s] = uint16_t(wave_trips(n, s));
    return r;
}
__device__ constexpr TripTable kTrips = trip_table();

// The value of the lane N places before in the row of 16 (DPP row_shr), 0 in
// the first N.
template <int N, class V>
__device__ __forceinline__ V row_before(V v)
{
    const int x = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x110 + N, 0xf, 0xf, false);
    return __builtin_bit_cast(V, x);
}
__device__ __forceinline__ int row_before_sum(int v)  // of the lanes before
{
    const int own = v;
    v += row_before<1>(v);
    v += row_before<2>(v);
    v += row_before<4>(v);
    v += row_before<8>(v);
    return v - own;
}
template <class V, class F>
__device__ __forceinline__ V row_all(V v, F f)
{
    v = f(v, gror<8>(v));
    v = f(v, gror<4>(v));
    v = f(v, gror<2>(v));
    return f(v, gror<1>(v));
}

// The runs that should end first on a grid of `slots` wavefronts, two a SIMD,
// the same in every workgroup; the whole workgroup of eight wavefronts calls
// it, a row of 16 lanes a way to cut, a lane a list.  A way: the candidates
// that a lane of a coarse wavefront walks at most, C(n + 3, 3) over its
// block's lanes (eight at most), and the finer wavefronts' least lanes.
//
// A trip takes the same 0.24 us however many wavefronts a SIMD has, one or
// two, and however many lanes a block: scheduling wavefronts of wave_trips so
// comes within 8% of the measured times of five contents (noise with
// rectangles, random texels, gradients, four colours a block, dark texels) at
// 13 sizes and seven cuts each, and the estimate of the end below chooses as
// that schedule would.  (A rule fitted to the first of these contents chose
// cuts up to 1.2 times as long for the others.)
__device__ __forceinline__ void choose_runs(ListRuns &runs, const int *__restrict__ counts, int cap, int slots)
{
    static_assert(kSearchWaves == 8, "32 rows, a way each");
    const int t = threadIdx.x, way = t >> 4, l = t & 15, n = 16 - l, m = way >> 2;
    const int c = n >= 2 ? min(counts[n], cap) : 0;
    const int most = m == 0 ? 1 << 20 : m == 1 ? 700 : m == 2 ? 500 : m == 3 ? 350 : m == 4 ? 250 : m == 5 ? 180 : 130;
    const int each = (n + 1) * (n + 2) * (n + 3) / 6;
    const int s = (each > most ? 1 : 0) + (each > 2 * most ? 1 : 0) + (each > 4 * most ? 1 : 0), f = max(s, way & 3);
    const float trips = float(kTrips.t[n][s]), fine_trips = float(kTrips.t[n][f]);
    const auto add = [](auto a, auto b) { return a + b; };
    const auto greater = [](float a, float b) { return fmaxf(a, b); };

    const int waves = (c + (64 >> s) - 1) >> (6 - s);
    const int rounds = row_all(waves, add) / slots, coarse = rounds * slots;
    const int before = min(row_before_sum(waves), coarse), k = min(waves, coarse - before);
    const int done = min(k << (6 - s), c);
    const int r = (c - done + (64 >> f) - 1) >> (6 - f);
    const int rest = row_all(r, add);
    const float sum = row_all(float(k) * trips, add), rest_sum = row_all(float(r) * fine_trips, add);
    const float longest = row_all(k > 0 ? trips : 0.0f, greater), rest_longest = row_all(r > 0 ? fine_trips : 0.0f, greater);
    // The first and the last wavefront of the last coarse round.
    const float top = row_all(before <= coarse - slots && coarse - slots < before + k ? trips : 0.0f, greater);
    const float last = row_all(k > 0 && before + k == coarse ? trips : 0.0f, greater);
    const float per = 1.0f / float(slots), spread = fmaxf(top - last, 0.0f);
    float end;
    if (rounds == 0) {
        end = rest <= slots ? fmaxf(rest_longest, rest_sum * per) : FLT_MAX;
    } else if (rest == 0) {
        end = fmaxf(longest, sum * per + (rounds > 1 ? 0.5f * spread : 0.0f));
    } else {
        // After coarse wavefronts that end together the finer ones take whole
        // rounds; they fill in between those that end apart.
        const float u = fminf(1.0f, spread / rest_longest);
        const float whole = float((rest + slots - 1) / slots) * rest_longest;
        end = fmaxf(longest, (sum + rest_sum) * per + (1.0f - u) * (whole - rest_sum * per) + u * 0.5f * rest_longest);
    }
    if (l == 0) runs.end[way] = way < 28 ? end : FLT_MAX;
    __syncthreads();
    const float own = runs.end[t & 31];
    float least = own;
#pragma unroll
    for (int x = 1; x < 32; x <<= 1) least = fminf(least, __shfl_xor(least, x));
    const int pick = __builtin_ctzll(__builtin_amdgcn_ballot_w64(own == least));
    if (way == pick && l < 15) {
        runs.start[l] = before;
        runs.first[l] = 0;
        runs.list[l] = n | s << 8;
        runs.start[15 + l] = coarse + row_before_sum(r);
        runs.first[15 + l] = done;
        runs.list[15 + l] = n | f << 8;
        runs.count[l] = runs.count[15 + l] = c;
        if (l == 0) runs.total = coarse + rest;
    }
    __syncthreads();
}

// Wavefront `wave` of the runs: entries first .. of list k's cnt, 64 >> shift
// of them.  False past the last wavefront.
__device__ __forceinline__ bool list_wave(const ListRuns &runs, int wave, int lane, int &k, int &first, int &cnt, int &shift)
{
    if (wave >= __builtin_amdgcn_readfirstlane(runs.total)) return false;
    // The last run that starts no later: those after it without wavefronts start later.
    const int at = runs.start[lane & 31];
    const int j = 63 - __builtin_clzll(__builtin_amdgcn_ballot_w64(lane < kRuns && at <= wave));
    const int list = __builtin_amdgcn_readfirstlane(runs.list[j]);
    k = list & 0xff;
    shift = list >> 8;
    cnt = __builtin_amdgcn_readfirstlane(runs.count[j]);
    first = __builtin_amdgcn_readfirstlane(runs.first[j]) +
            ((wave - __builtin_amdgcn_readfirstlane(runs.start[j])) << (6 - shift));
    return true;
}

// Images of a search launch: `get` gives the image and block of a list
// entry; false for an entry that names none.  Shared: what a workgroup keeps
// of them in LDS, filled by `load`.
struct OneImage {
    struct Shared {};
    LaneImage im;
    int blocks;
    __device__ __forceinline__ void load(Shared &) const {}
    __device__ __forceinline__ bool get(const Shared &, int entry, LaneImage &out, int &blk) const
    {
        out = im;
        blk = entry;
        return unsigned(entry) < unsigned(blocks);
    }
};

// List entries of a launch over several images: image << kImageShift | block.
constexpr int kImageShift = 20;

__device__ __forceinline__ bool named_image(const ntx::Bc1Image *imgs, int n, int entry, LaneImage &out, int &blk)
{
    const int img = int(unsigned(entry) >> kImageShift);
    const ntx::Bc1Image d = imgs[img < n ? img : 0];
    out = { d.src, reinterpret_cast<uint2 *>(d.out), d.w, d.h, (d.w + 3) / 4, d.alpha_mode, d.rows16, d.cw[0], d.cw[1],
            d.cw[2] };
    blk = entry & ((1 << kImageShift) - 1);
    return img < n && blk < out.bw * ((d.h + 3) / 4);
}

// Images of a table in device memory.
struct ImageTable {
    struct Shared {};
    const ntx::Bc1Image *imgs;
    int n;
    __device__ __forceinline__ void load(Shared &) const {}
    __device__ __forceinline__ bool get(const Shared &, int entry, LaneImage &out, int &blk) const
    {
        return named_image(imgs, n, entry, out, blk);
    }
};

// Images that come with the launch (a mip chain); image i's 256-block chunks
// start at `first[i]`.
struct ImageSet {
    struct Shared {
        ntx::Bc1Image imgs[ntx::kBc1MaxImages];
    };
    ntx::Bc1Image imgs[ntx::kBc1MaxImages];
    int first[ntx::kBc1MaxImages];
    int n;
    __device__ __forceinline__ void load(Shared &sh) const
    {
#pragma unroll
        for (int i = 0; i < ntx::kBc1MaxImages; i++)
            if (threadIdx.x == 0) sh.imgs[i] = imgs[i];
    }
    __device__ __forceinline__ bool get(const Shared &sh, int entry, LaneImage &out, int &blk) const
    {
        return named_image(sh.imgs, n, entry, out, blk);
    }
};


// Level8 pass 2 (icbc.h:3292-3326 + :3543-3550).  The lists are cut into
// wavefronts of consecutive entries, 1 to 8 lanes a block by list, and walked
// from n = 16 down: the grid's wavefronts take the first, then the next from
// a queue, so that the longest start first and the short ones fill in.  Lanes
// past the end of their list repeat its first block and write nothing.  The
// block is gathered and reduced again (the same n), its prefix-sum table
// built in LDS, the four-colour fit searched, then (after skip_blacks when
// some cluster is black) the three-colour fit, and the better block kept.
// The last workgroup clears the tallies and the queue.
template <class Images>
__global__ __launch_bounds__(64 * kSearchWaves, 2) void bc1_search_kernel(Images images,
                                                                          const ntx::Tables *__restrict__ tab,
                                                                          short2 *__restrict__ nm,
                                                                          int *__restrict__ counts,
                                                                          const int *__restrict__ lists, int cap)
{
    using namespace ntx_bucket;
    __shared__ float4 s_rows[kSearchWaves][17][64];
    __shared__ SearchTables s_tables;
    __shared__ typename Images::Shared s_images;
    __shared__ ListRuns s_runs;
    load_search_tables(s_tables, tab, threadIdx.x, 64 * kSearchWaves);
    images.load(s_images);
    choose_runs(s_runs, counts, cap, int(gridDim.x) * kSearchWaves);
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
    for (int wave = blockIdx.x + gridDim.x * wv;;) {
        int k = 0, first = 0, cnt = 0, shift = 0;
        if (!list_wave(s_runs, wave, lane, k, first, cnt, shift)) break;
        const int cols = 64 >> shift;
        const int item = first + (lane & (cols - 1));
        bool live = item < cnt;
        // Every caller's lists hold blocks of its images; anything else is
        // written nowhere.
        LaneImage im;
        int blk;
        if (!images.get(s_images, lists[size_t(k) * cap + (live ? item : first)], im, blk)) {
            blk = 0;
            live = false;
        }
        search_lane(im, blk, live, tab, nm, s_rows[wv], lane & (cols - 1), lane >> (6 - shift), 1 << shift, k, s_tables);
        int next = 0;
        if (lane == 0) next = atomicAdd(&counts[kQueueSlot], 1);
        wave = int(gridDim.x) * kSearchWaves + __builtin_amdgcn_readfirstlane(next);
    }
    // Every wavefront has read the tallies for the last time.
    __syncthreads();
    release_counts(counts);
}

// Pass 1 over several images: one workgroup per chunk of 256 blocks of one
// image.
__global__ __launch_bounds__(256) void bc1_classify_multi_kernel(const ntx::Bc1Image *__restrict__ imgs,
                                                                 const int2 *__restrict__ map,
                                                                 const ntx::Tables *__restrict__ tab,
                                                                 int *__restrict__ counts, int *__restrict__ lists,
                                                                 int cap)
{
    __shared__ ClassifyShared sh;
    const int2 m = map[blockIdx.x];
    const ntx::Bc1Image im = imgs[m.x];
    const int bw = (im.w + 3) / 4;
    const int blocks = bw * ((im.h + 3) / 4);
    classify_chunk(im.src, im.w, im.h, bw, blocks, im.alpha_mode, tab, reinterpret_cast<uint2 *>(im.out), nullptr, counts,
                   lists, cap, im.rows16, sh, m.y + int(threadIdx.x), m.x << kImageShift);
}

__global__ __launch_bounds__(256) void bc1_classify_set_kernel(ImageSet set, const ntx::Tables *__restrict__ tab,
                                                               int *__restrict__ counts, int *__restrict__ lists, int cap)
{
    __shared__ ClassifyShared sh;
    int j = 0;
    while (j + 1 < set.n && int(blockIdx.x) >= set.first[j + 1]) j++;
    const ntx::Bc1Image &im = set.imgs[j];
    const int bw = (im.w + 3) / 4;
    const int blocks = bw * ((im.h + 3) / 4);
    classify_chunk(im.src, im.w, im.h, bw, blocks, im.alpha_mode, tab, reinterpret_cast<uint2 *>(im.out), nullptr, counts,
                   lists, cap, im.rows16, sh, (int(blockIdx.x) - set.first[j]) * 256 + int(threadIdx.x), j << kImageShift);
}

}  // namespace

namespace ntx {

// Groups per block of an image of `blocks` blocks: a block on one group
// searches up to 61 runs of partitions one after another (about 37 us), which
// an image that leaves SIMDs idle should not wait for.  Every group of a block
// prepares it again, so the lines are where blocks of few colours, which have
// next to nothing to search, lose no more than 2 us.  On 1, 4 and 16 groups,
// noise with rectangles and blocks of four colours: 256 blocks 34.5, 18.1 and
// 14.2 us, 13.8, 12.9 and 13.0; 400 blocks 35.6, 18.3 and 15.9, 14.1, 12.9 and
// 14.8; 784 blocks 35.2, 18.3 and 21.0, 14.0, 13.1 and 21.0; 2,025 blocks 35.5,
// 19.9 and 38.8, 13.5, 15.0 and 37.0; 4,096 blocks 35.4, 30.3 and 71.2, 13.6,
// 21.7 and 68.1.
static int bc1_parts(int blocks)
{
    return blocks <= 512 ? 16 : blocks <= 2048 ? 4 : 1;
}

// Up to kBc1MaxImages images in one launch, in the order given (the largest
// first, so that the small ones' workgroups fill in behind it).  urgent: the
// waves raise their issue priority (s_setprio), for small latency-bound
// images compressed beside large ones; level: icbc quality level 8 (nvtt
// Normal / Highest), 9 (Production) or 1 (Fastest).
hipError_t launch_bc1(const Bc1Target *images, int n, int alpha_mode, const float *cw, const Tables *d_tab,
                      hipStream_t stream, bool urgent, int level)
{
    Bc1Jobs jobs{};
    int grid = 0;
    for (int k = 0; k < n && jobs.n < kBc1MaxImages; k++) {
        const Bc1Target &t = images[k];
        Bc1Job &job = jobs.job[jobs.n];
        job.src = t.src;
        job.out = static_cast<uint2 *>(t.out);
        job.nm = reinterpret_cast<short2 *>(t.nm);
        job.w = t.w;
        job.h = t.h;
        job.bw = (t.w + 3) / 4;
        job.blocks = job.bw * ((t.h + 3) / 4);
        if (job.blocks == 0) continue;
        job.parts = level == 8 ? bc1_parts(job.blocks) : 1;
        job.first = grid;
        const int each = kBlocksPerWG / job.parts;
        grid += (job.blocks + each - 1) / each;
        jobs.n++;
    }
    if (jobs.n == 0) return hipSuccess;
    auto launch = [&](auto kernel, const auto &args) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlocksPerWG * kGroup), 0, stream, args, alpha_mode, cw[0], cw[1],
                           cw[2], d_tab, urgent ? 1 : 0);
    };
    if (jobs.n == 1)
        launch(level == 1 ? bc1_kernel<1, Bc1Job> : level == 9 ? bc1_kernel<9, Bc1Job> : bc1_kernel<8, Bc1Job>, jobs.job[0]);
    else
        launch(level == 1 ? bc1_kernel<1, Bc1Jobs> : level == 9 ? bc1_kernel<9, Bc1Jobs> : bc1_kernel<8, Bc1Jobs>, jobs);
    return hipGetLastError();
}

// Level8 pass 1 into the block lists in `counts` / `lists` (zero tallies on
// entry; lists: 17 x the image's blocks).
hipError_t launch_bc1_classify(const float *d_src, int w, int h, int alpha_mode, const Tables *d_tab, void *d_out,
                               int16_t *d_nm, int *d_counts, int *d_lists, hipStream_t stream, bool urgent)
{
    const int bw = (w + 3) / 4, bh = (h + 3) / 4, nblocks = bw * bh;
    if (nblocks == 0) return hipSuccess;
    const int rows16 = (reinterpret_cast<uintptr_t>(d_src) & 15) == 0 && (w & 3) == 0;
    hipLaunchKernelGGL(bc1_classify_kernel, dim3((nblocks + 255) / 256), dim3(256), 0, stream, d_src, w, h, bw, nblocks, alpha_mode,
                       d_tab, reinterpret_cast<uint2 *>(d_out), reinterpret_cast<short2 *>(d_nm), d_counts, d_lists, rows16,
                       urgent ? 1 : 0);
    return hipGetLastError();
}

template <class Images>
static hipError_t launch_search(const Images &images, const Tables *d_tab, int16_t *d_nm, int *d_counts,
                                const int *d_lists, int cap, int cus, hipStream_t stream)
{
    // At most eight lanes a block.
    const int groups = (cap + 8 * kSearchWaves - 1) / (8 * kSearchWaves);
    hipLaunchKernelGGL(bc1_search_kernel<Images>, dim3(groups < cus ? groups : cus), dim3(64 * kSearchWaves), 0, stream,
                       images, d_tab, reinterpret_cast<short2 *>(d_nm), d_counts, d_lists, cap);
    return hipGetLastError();
}

// Level8 pass 2 over the lists pass 1 filled (at most `cap` blocks in all);
// leaves the tallies zero.  cus: the device's compute units.
hipError_t launch_bc1_search(const float *d_src, int w, int h, int alpha_mode, const float *cw, const Tables *d_tab,
                             void *d_out, int16_t *d_nm, int *d_counts, const int *d_lists, int cap, int cus,
                             hipStream_t stream)
{
    if (cap == 0) return hipSuccess;
    const int rows16 = (reinterpret_cast<uintptr_t>(d_src) & 15) == 0 && (w & 3) == 0;
    const OneImage one{ { d_src, reinterpret_cast<uint2 *>(d_out), w, h, (w + 3) / 4, alpha_mode, rows16, cw[0], cw[1],
                          cw[2] },
                        cap };
    return launch_search(one, d_tab, d_nm, d_counts, d_lists, cap, cus, stream);
}

int bc1_scratch_ints(int nblocks) { return ntx_bucket::kListsOffset + ntx_bucket::kCountSlots * nblocks; }

int bc1_multi_max_images() { return 1 << (31 - kImageShift); }
int bc1_multi_max_blocks() { return 1 << kImageShift; }

// Pass 1 of the multi-image form: d_map holds nchunks (image, first block)
// pairs, one per workgroup of 256 blocks; the lists (zero tallies on entry)
// take up to cap entries each, cap >= all the images' blocks.
hipError_t launch_bc1_classify_multi(const Bc1Image *d_imgs, const void *d_map, int nchunks, const Tables *d_tab,
                                     int *d_counts, int *d_lists, int cap, hipStream_t stream)
{
    if (nchunks == 0) return hipSuccess;
    hipLaunchKernelGGL(bc1_classify_multi_kernel, dim3(nchunks), dim3(256), 0, stream, d_imgs,
                       static_cast<const int2 *>(d_map), d_tab, d_counts, d_lists, cap);
    return hipGetLastError();
}

// Pass 2 of the multi-image form over the lists pass 1 filled; leaves the
// tallies zero.
hipError_t launch_bc1_search_multi(const Bc1Image *d_imgs, int nimgs, const Tables *d_tab, int *d_counts,
                                   const int *d_lists, int cap, int cus, hipStream_t stream)
{
    if (cap == 0) return hipSuccess;
    const ImageTable table{ d_imgs, nimgs };
    return launch_search(table, d_tab, nullptr, d_counts, d_lists, cap, cus, stream);
}

static ImageSet image_set(const Bc1Target *images, int n, int alpha_mode, const float *cw, int *chunks)
{
    ImageSet set{};
    *chunks = 0;
    for (int k = 0; k < n && k < kBc1MaxImages; k++) {
        const Bc1Target &t = images[k];
        Bc1Image &im = set.imgs[k];
        im.src = t.src;
        im.out = t.out;
        im.w = t.w;
        im.h = t.h;
        im.alpha_mode = alpha_mode;
        im.rows16 = (reinterpret_cast<uintptr_t>(t.src) & 15) == 0 && (t.w & 3) == 0;
        for (int c = 0; c < 3; c++) im.cw[c] = cw[c];
        set.first[k] = *chunks;
        *chunks += (((t.w + 3) / 4) * ((t.h + 3) / 4) + 255) / 256;
        set.n = k + 1;
    }
    return set;
}

// The two passes over up to kBc1MaxImages images of at most
// bc1_multi_max_blocks() blocks each, together `cap` blocks, in a launch
// each; d_counts: bucket scratch of bc1_scratch_ints(cap) ints with zero
// tallies, which are zero again after the second.
hipError_t launch_bc1_classify_set(const Bc1Target *images, int n, int alpha_mode, const float *cw, const Tables *d_tab,
                                   int *d_counts, int cap, hipStream_t stream)
{
    int chunks = 0;
    const ImageSet set = image_set(images, n, alpha_mode, cw, &chunks);
    if (chunks == 0) return hipSuccess;
    int *d_lists = d_counts + ntx_bucket::kListsOffset;
    hipLaunchKernelGGL(bc1_classify_set_kernel, dim3(chunks), dim3(256), 0, stream, set, d_tab, d_counts, d_lists, cap);
    return hipGetLastError();
}

hipError_t launch_bc1_search_set(const Bc1Target *images, int n, int alpha_mode, const float *cw, const Tables *d_tab,
                                 int *d_counts, int cap, int cus, hipStream_t stream)
{
    int chunks = 0;
    const ImageSet set = image_set(images, n, alpha_mode, cw, &chunks);
    if (chunks == 0) return hipSuccess;
    return launch_search(set, d_tab, nullptr, d_counts, d_counts + ntx_bucket::kListsOffset, cap, cus, stream);
}

// icbc Level8 of the *d_count blocks listed in d_list (at most cap, each
// below cap, cap = the image's block count), at most max_groups workgroups.
hipError_t launch_bc1_list(const float *d_src, int w, int h, int alpha_mode, const float *cw, const Tables *d_tab,
                           void *d_out, const int *d_list, const int *d_count, int cap, int max_groups,
                           hipStream_t stream)
{
    if (cap == 0) return hipSuccess;
    const int bw = (w + 3) / 4;
    int grid = (cap + kBlocksPerWG - 1) / kBlocksPerWG;
    if (max_groups > 0 && grid > max_groups) grid = max_groups;
    hipLaunchKernelGGL(bc1_list_kernel<8>, dim3(grid), dim3(kBlocksPerWG * kGroup), 0, stream, d_src, w, h, bw, d_list,
                       d_count, cap, alpha_mode, cw[0], cw[1], cw[2], d_tab, reinterpret_cast<uint2 *>(d_out));
    return hipGetLastError();
}

}  // namespace ntx
