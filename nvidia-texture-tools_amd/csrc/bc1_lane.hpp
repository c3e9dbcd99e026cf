// bc1_lane.hpp -- icbc v1.05 compress_dxt1 at Quality_Level8 (icbc.h:3485-3559,
// the SSE4.1 build: no FMA, exact division, round-half-even, 4-lane
// tie-break) with S lanes per 4x4 block (1, 2, 4 or 8), for the two-pass BC1
// encoder (bc1.hip: bc1_classify_kernel, bc1_search_kernel).
//
// A wavefront's 64 / S blocks each have a column of a [17][64] float4 LDS
// array for their clusters, then their prefix-sum table: lane l works on
// column l % (64 / S), so the lanes that read row r read consecutive entries
// (the S lanes of a block the same one) without bank conflicts.  The S lanes
// of a block prepare it alike (the same stores to the same places) and split
// the partition search.
//
// The cluster tables (icbc.h:1906-2012) list, for t = 1..16, the new
// prefix triples c0 <= c1 <= c2 = t in (c0, c1) order, and the pairs
// c0 <= c1 = t in c0 order; the table of a colour count n is the first
// C(n+3,3)-1 (C(n+2,2)-1) entries.  The winner is the SSE build's: the least
// (error, p & 3, p >> 2) over the table index p, so the candidates may be
// visited in any order that knows their p.
#pragma once

#include "bc1_block.hpp"

namespace ntx_bc1 {

using LaneRows = float4 (*)[64];

__device__ __forceinline__ bool is_black(float r, float g, float b)
{
    // icbc.h:1628-1635.
    return r < 1.0f / 8 && g < 1.0f / 8 && b < 1.0f / 8;
}

// The set-up of a block below runs once per block beside some hundred
// candidates per lane, so what it costs is mostly fetching its instructions:
// it is kept in loops over rows of four texels or over clusters, with one
// instance of each part for both fits: a third of the code that the loops
// unrolled took (10,000 vector instructions a kernel of 18,000 before), and
// the search of an 8192^2 image 4.8 -> 4.1 ms together with the branches
// below.

// A block's texels, by row.
struct BlockTexels {
    const float *src;
    size_t plane;
    int w, h, x, y;
    bool transparency, whole;

    // rows16: every row of every plane starts 16-byte aligned, so an inner
    // block reads each row of each plane with one 16-byte load.
    __device__ __forceinline__ BlockTexels(const float *src_, int w_, int h_, int bx, int by, int alpha_mode, bool rows16)
        : src(src_), plane(size_t(w_) * size_t(h_)), w(w_), h(h_), x(4 * bx), y(4 * by),
          transparency(alpha_mode == NTX_ALPHA_TRANSPARENCY), whole(rows16 && 4 * bx + 4 <= w_ && 4 * by + 4 <= h_)
    {
    }

    // FloatColorCompressor's gather (BlockCompressor.cpp:116-166) of row r:
    // texel i = (r, g, b, weight); outside the image colour 0, weight 0;
    // weight = saturate(alpha) for Transparency, else 1.
    __device__ __forceinline__ void row(int r, float4 (&t)[4]) const
    {
        if (whole) whole_row(r, t);
        else edge_row(r, t);
    }
    // All rows, 4 r + i: one branch, so that every row's loads are in flight
    // together (a branch a row, with a wait at its end: 8192^2 classified in
    // 516 us, 482 so).
    __device__ __forceinline__ void all(float4 (&t)[16]) const
    {
        if (whole) {
#pragma unroll
            for (int r = 0; r < 4; r++) whole_row(r, t + 4 * r);
            return;
        }
#pragma unroll
        for (int r = 0; r < 4; r++) edge_row(r, t + 4 * r);
    }

private:
    __device__ __forceinline__ void whole_row(int r, float4 *t) const
    {
        const float *p = src + (size_t(y) * size_t(w) + size_t(x)) + size_t(r) * size_t(w);  // r w: scalar
        const float4 vr = *reinterpret_cast<const float4 *>(p);
        const float4 vg = *reinterpret_cast<const float4 *>(p + plane);
        const float4 vb = *reinterpret_cast<const float4 *>(p + 2 * plane);
        float4 wt = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
        if (transparency) {
            const float4 va = *reinterpret_cast<const float4 *>(p + 3 * plane);
            wt = make_float4(icbc_saturate(va.x), icbc_saturate(va.y), icbc_saturate(va.z), icbc_saturate(va.w));
        }
        t[0] = make_float4(vr.x, vg.x, vb.x, wt.x);
        t[1] = make_float4(vr.y, vg.y, vb.y, wt.y);
        t[2] = make_float4(vr.z, vg.z, vb.z, wt.z);
        t[3] = make_float4(vr.w, vg.w, vb.w, wt.w);
    }
    __device__ __forceinline__ void edge_row(int r, float4 *t) const
    {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (x + i < w && y + r < h) {
                const size_t o = size_t(y + r) * size_t(w) + size_t(x + i);
                v.x = src[o];
                v.y = src[o + plane];
                v.z = src[o + 2 * plane];
                v.w = transparency ? icbc_saturate(src[o + 3 * plane]) : 1.0f;
            }
            t[i] = v;
        }
    }
};

// What reduce_colors saw of a block.
struct Reduced {
    int n = 0;               // clusters
    bool any_black = false;  // some texel of positive weight is black (is_black)
    bool unit = true;        // every texel weighs 1
    bool tame = true;        // every component is 0 or of magnitude 1e-18 to 1e18
};

// reduce_colors (icbc.h:1638-1683): texels of positive weight merge, in
// texel order, into the first earlier cluster within 1/256 in every channel
// (weighted running mean), or open a new one.  Leaves clusters 0..n-1 as
// (r, g, b, weight) in rows[0..n-1].  Tame texels, with weights of at most 1,
// keep every sum and error of the searches finite, and those of unit weights
// normal (or an exact zero) too; the principal axis, which squares its
// covariances, they do not (lane_sat).  k: the block's known cluster count
// (every texel of 16 clusters opens one).
__device__ __forceinline__ Reduced lane_reduce(LaneRows rows, int lane, const BlockTexels &texels, int k)
{
    const float thr = 1.0f / 256;
    Reduced out;
    uint32_t largest = 0, least = 0xffffffffu;
    float4 t[4], next[4];
    texels.row(0, next);
#pragma unroll 1
    for (int r = 0; r < 4; r++) {
#pragma unroll
        for (int i = 0; i < 4; i++) t[i] = next[i];
        if (r < 3) texels.row(r + 1, next);
#pragma unroll 1
        for (int i = 0; i < 4; i++) {
            const float4 ci = t[0];
            t[0] = t[1];
            t[1] = t[2];
            t[2] = t[3];
            const float c[3] = { ci.x, ci.y, ci.z };
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const uint32_t u = uint32_t(__float_as_int(c[k])) << 1;
                largest = max(largest, u);
                least = min(least, u - 1);  // zero wraps to the largest
            }
            out.unit = out.unit && ci.w == 1.0f;
            if (ci.w > 0) {
                // First matching cluster: two a trip until every lane has
                // found one or passed its last (at most 15 here).
                int jm = -1;
                for (int j = 0; k < 16 && __builtin_amdgcn_ballot_w64(jm < 0 && j < out.n) != 0; j += 2) {
                    const float4 k0 = rows[j][lane], k1 = rows[j + 1][lane];
                    const bool m0 = fabsf(k0.x - ci.x) < thr && fabsf(k0.y - ci.y) < thr && fabsf(k0.z - ci.z) < thr;
                    const bool m1 = fabsf(k1.x - ci.x) < thr && fabsf(k1.y - ci.y) < thr && fabsf(k1.z - ci.z) < thr;
                    if (jm < 0 && j < out.n && m0) jm = j;
                    if (jm < 0 && j + 1 < out.n && m1) jm = j + 1;
                }
                if (jm >= 0) {
                    const float4 k = rows[jm][lane];
                    const float s = k.w + ci.w;
                    const float nr = k.x * k.w + ci.x * ci.w, ng = k.y * k.w + ci.y * ci.w, nb = k.z * k.w + ci.z * ci.w;
                    rows[jm][lane] = make_float4(nr / s, ng / s, nb / s, s);
                } else {
                    rows[out.n][lane] = ci;
                    out.n++;
                }
                if (is_black(ci.x, ci.y, ci.z)) out.any_black = true;
            }
        }
    }
    out.tame = largest <= uint32_t(__float_as_int(1e18f)) << 1 && least >= (uint32_t(__float_as_int(1e-18f)) << 1) - 1;
    return out;
}

// reduce_colors alone, for the classify pass, which is all of it: the same
// loops unrolled (16 texels against up to 15 clusters).  Returns the number
// of clusters, left in rows.
__device__ __forceinline__ int classify_reduce(LaneRows rows, int lane, const BlockTexels &texels)
{
    const float thr = 1.0f / 256;
    float4 t[16];
    texels.all(t);
    int n = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const float4 ci = t[i];
        if (ci.w > 0) {
            // First matching cluster: clusters j < n (n <= i here).
            int jm = -1;
#pragma unroll
            for (int j = i - 1; j >= 0; j--) {
                const float4 k = rows[j][lane];
                if (j < n && fabsf(k.x - ci.x) < thr && fabsf(k.y - ci.y) < thr && fabsf(k.z - ci.z) < thr) jm = j;
            }
            if (jm >= 0) {
                const float4 k = rows[jm][lane];
                const float s = k.w + ci.w;
                const float nr = k.x * k.w + ci.x * ci.w, ng = k.y * k.w + ci.y * ci.w, nb = k.z * k.w + ci.z * ci.w;
                rows[jm][lane] = make_float4(nr / s, ng / s, nb / s, s);
            } else {
                rows[n][lane] = ci;
                n++;
            }
        }
    }
    return n;
}

// skip_blacks (icbc.h:1685-1703) in place: keeps the clusters that are not
// black, in order; returns their count.
__device__ __forceinline__ int lane_skip_blacks(LaneRows rows, int lane, int n)
{
    int m = 0;
#pragma unroll 1
    for (int j = 0; j < n; j++) {
        const float4 k = rows[j][lane];
        if (!is_black(k.x, k.y, k.z)) {
            rows[m][lane] = k;
            m++;
        }
    }
    return m;
}

// True if some cluster 0..n-1 is black (skip_blacks would drop it).
__device__ __forceinline__ bool lane_has_black_cluster(LaneRows rows, int lane, int n)
{
    bool any = false;
#pragma unroll 1
    for (int j = 0; j < n; j++) {
        const float4 k = rows[j][lane];
        any = any || is_black(k.x, k.y, k.z);
    }
    return any;
}

__device__ __forceinline__ void min_max_f64(double &a, double &b)
{
    double lo, hi;
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo;
    b = hi;
}

// compute_sat (icbc.h:1796-1882) of the n >= 1 clusters in rows[0..n-1]:
// weighted PCA by the power method, the stable insertion sort by projection,
// and the prefix sums in sorted order.  Leaves row 0 zero, rows 1..n the
// prefix sums (r*w, g*w, b*w, w) and rows n+1..16 FLT_MAX (the entries the
// SSE build reads past the count), and returns row n.  tame: the same in
// every lane of the wave.
__device__ __forceinline__ float4 lane_sat(LaneRows rows, int lane, int n, bool tame)
{
    // computeCentroid: sequential sums over clusters 0..n-1.
    float total = 0.0f, cr = 0.0f, cg = 0.0f, cb = 0.0f;
#pragma unroll 4
    for (int j = 0; j < 16; j++) {
        const float4 c = rows[j][lane];
        if (j < n) {
            total += c.w;
            cr += c.x * c.w;
            cg += c.y * c.w;
            cb += c.z * c.w;
        }
    }
    const float inv = 1.0f / total;
    cr *= inv; cg *= inv; cb *= inv;
    // computeCovariance.
    float m0 = 0.0f, m1 = 0.0f, m2 = 0.0f, m3 = 0.0f, m4 = 0.0f, m5 = 0.0f;
#pragma unroll 4
    for (int j = 0; j < 16; j++) {
        const float4 c = rows[j][lane];
        if (j < n) {
            const float ar = c.x - cr, ag = c.y - cg, ab = c.z - cb;
            const float br = ar * c.w, bg = ag * c.w, bb = ab * c.w;
            m0 += ar * br; m1 += ar * bg; m2 += ar * bb;
            m3 += ag * bg; m4 += ag * bb; m5 += ab * bb;
        }
    }
    // firstEigenVector_PowerMethod (icbc.h:1767-1791).
    float vx = 0.0f, vy = 0.0f, vz = 0.0f;
    if (!(m0 == 0 && m3 == 0 && m5 == 0)) {
        const float r0 = m0 * m0 + m1 * m1 + m2 * m2;
        const float r1 = m1 * m1 + m3 * m3 + m4 * m4;
        const float r2 = m2 * m2 + m4 * m4 + m5 * m5;
        if (r0 > r1 && r0 > r2) { vx = m0; vy = m1; vz = m2; }
        else if (r1 > r2) { vx = m1; vy = m3; vz = m4; }
        else { vx = m2; vy = m4; vz = m5; }
#pragma unroll 1
        for (int it = 0; it < 8; it++) {
            const float x = vx * m0 + vy * m1 + vz * m2;
            const float y = vx * m1 + vy * m3 + vz * m4;
            const float z = vx * m2 + vy * m4 + vz * m5;
            float norm = (y < x) ? x : y;  // icbc max(a,b) = (b<a)?a:b
            norm = (z < norm) ? norm : z;
            const float iv = 1.0f / norm;
            vx = x * iv; vy = y * iv; vz = z * iv;
        }
    }
    // The stable order by projection: ord[r], the cluster at rank r, in four
    // bits each.  The keys below order numbers only, and tame texels have none
    // where the axis squares covariances beyond the range of floats:
    // components that lie 4e9 apart or more, weights of 1e-17 or less.
    const bool axis = fabsf(vx) <= 1e18f && fabsf(vy) <= 1e18f && fabsf(vz) <= 1e18f;
    uint64_t ord = 0;
    if (tame && __builtin_amdgcn_ballot_w64(!axis) == 0) {
        // (projection, cluster) as doubles (TameBest; + 0 makes a -0 the 0
        // that the comparisons take it for), through an odd-even merge sort:
        // two instructions a comparator.  Ranks past n sort last.
        double key[16];
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const float4 c = rows[j][lane];
            const float dp = (c.x * vx + c.y * vy + c.z * vz) + 0.0f;
            const int hi = j < n ? __float_as_int(dp) : __float_as_int(FLT_MAX);
            key[j] = __hiloint2double(hi, j ^ (hi >> 31));
        }
#pragma unroll
        for (int p = 1; p < 16; p <<= 1)
#pragma unroll
            for (int k = p; k >= 1; k >>= 1)
#pragma unroll
                for (int j = k % p; j <= 15 - k; j += 2 * k)
#pragma unroll
                    for (int i = 0; i < k; i++)
                        if (i + j + k < 16 && (i + j) / (2 * p) == (i + j + k) / (2 * p)) min_max_f64(key[i + j], key[i + j + k]);
#pragma unroll
        for (int r = 0; r < 16; r++) ord |= uint64_t(uint32_t(__double2loint(key[r]) ^ (__double2hiint(key[r]) >> 31)) & 15u) << (4 * r);
    } else {
        // The insertion sort itself: a NaN stops an element where it stops
        // the reference's loop.
        float dps[16];
        int at[16];
#pragma unroll 1
        for (int j = 0; j < n; j++) {
            const float4 c = rows[j][lane];
            dps[j] = c.x * vx + c.y * vy + c.z * vz;
            at[j] = j;
        }
#pragma unroll 1
        for (int i = 1; i < n; i++)
#pragma unroll 1
            for (int j = i; j > 0 && dps[j] < dps[j - 1]; j--) {
                const float td = dps[j]; dps[j] = dps[j - 1]; dps[j - 1] = td;
                const int to = at[j]; at[j] = at[j - 1]; at[j - 1] = to;
            }
#pragma unroll 1
        for (int r = 0; r < n; r++) ord |= uint64_t(at[r]) << (4 * r);
    }
    // The clusters in sorted order (all read before any row is rewritten).
    float4 s[16];
#pragma unroll
    for (int r = 0; r < 16; r++) s[r] = rows[int(ord >> (4 * r)) & 15][lane];
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f), sum = acc;
    rows[0][lane] = acc;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const float wgt = s[r].w;
        const float4 v = make_float4(s[r].x * wgt, s[r].y * wgt, s[r].z * wgt, wgt);
        if (r == 0) acc = v;
        else acc = make_float4(acc.x + v.x, acc.y + v.y, acc.z + v.z, acc.w + v.w);
        // By component: a choice between two float4 goes through memory.
        rows[r + 1][lane] = make_float4(r < n ? acc.x : FLT_MAX, r < n ? acc.y : FLT_MAX, r < n ? acc.z : FLT_MAX,
                                        r < n ? acc.w : FLT_MAX);
        if (r == n - 1) sum = acc;
    }
    return sum;
}

// The order among candidates of equal error, (p & 3, p >> 2), as one word
// (shifts that the scalar unit has, for the loops where p is the same in
// every lane).
__device__ __forceinline__ uint32_t tie_key(int p) { return uint32_t(p & 3) << 16 | uint32_t(p) >> 2; }
__device__ __forceinline__ int tie_index(uint32_t key) { return int((key & 0xffffu) << 2 | key >> 16); }

// Best-candidate bookkeeping of the general path: any floats, NaN never wins.
struct Best {
    float e = FLT_MAX;
    uint32_t key = 0;
    __device__ __forceinline__ void offer(float err, int p)
    {
        const uint32_t k = tie_key(p);
        if (err < e || (err == e && k < key)) { e = err; key = k; }
    }
    __device__ __forceinline__ int index() const { return tie_index(key); }
};

// The same for finite errors none of which is -0, in one minimum: (error,
// key) as a double whose high word is the error's bits and whose low word is
// the key, inverted where the sign makes larger words smaller doubles.  Two
// instructions and the minimum (double precision issues at the single rate
// here), where compares and selects take six.
struct TameBest {
    double v = __hiloint2double(__float_as_int(FLT_MAX), 0);
    __device__ __forceinline__ void take(double d) { asm("v_min_f64 %0, %0, %1" : "+v"(v) : "v"(d)); }
    __device__ __forceinline__ void offer(float err, uint32_t key)
    {
        const int hi = __float_as_int(err);
        take(__hiloint2double(hi, int(key ^ uint32_t(hi >> 31))));
    }
    // The least of the S lanes of a block, in each of them.
    __device__ __forceinline__ void combine(int S)
    {
        for (int x = 64 / S; x < 64; x <<= 1)
            take(__hiloint2double(__shfl_xor(__double2hiint(v), x), __shfl_xor(__double2loint(v), x)));
    }
    __device__ __forceinline__ Best best() const
    {
        const int hi = __double2hiint(v);
        return { __int_as_float(hi), uint32_t(__double2loint(v)) ^ uint32_t(hi >> 31) };
    }
};

// Where a candidate's weight terms come from: kScalar, 16 clusters of weight
// 1, so that the terms are the same in every lane and come by scalar loads;
// kTable, cluster weights that are integers summing to 16; kComputed, any.
enum class Terms { kScalar, kTable, kComputed };

// Index of the prefix weights a <= b <= c (integers up to 16) in the tables
// Tables::bc1h4 and bc1h3: C(c + 2, 3) + C(b + 1, 2) + a.
__device__ __forceinline__ constexpr int terms_c(int c) { return c * (c + 1) * (c + 2) / 6; }
__device__ __forceinline__ constexpr int terms_b(int b) { return b * (b + 1) / 2; }

// cluster_fit_four (icbc.h:2250-2549) over the table of a block with n
// clusters (the same n in every lane); sub: this lane's number among the
// block's S (WHOLE: S is 1, and c0 the same in every lane).  VALU issue bound, so the loops are ordered for what they can
// share with every rounding kept: the middle prefix c1 outermost, whose
// (x2 - x1) / 3 for every c2 stay in registers (hence the unrolled c2 loop);
// then c0, split over the S lanes (a lane past the end repeats the last,
// which offers the same candidate again), with (x1 - x0) 2/3 + x0; a
// candidate's weighted sum is then one addition per channel.  That, the
// halved error and TameBest make 88 instructions a candidate of the 109 that
// the (c2, c0, c1) order took: an 8192^2 noise and rectangles image 6.13 ->
// 4.78 ms a call, of which 4.1 are bc1_search_kernel.
template <bool WHOLE, Terms T>
__device__ __forceinline__ void search4(LaneRows rows, int col, int sub, int S, int n, float4 sum, float mx, float my,
                                        float mz, const float4 *terms, TameBest &best)
{
    // Per c2: kTable the byte offset of its terms, kComputed its weight.
    float xw[17];
#pragma unroll
    for (int c = 1; c <= 16; c++) {
        xw[c] = 0.0f;
        if (T != Terms::kScalar && c <= n) {
            const float w = rows[c][col].w;
            xw[c] = T == Terms::kTable ? __int_as_float(terms_c(int(w)) * 16) : w;
        }
    }
    for (int b = 0; b <= n; b++) {
        const float4 x1 = rows[b][col];
        // Bit c: c2 = c is one of this c1's, max(b, 1) to n.
        const uint32_t span = (2u << n) - (2u << max(b - 1, 0));
        float ux[17], uy[17], uz[17];
#pragma unroll
        for (int c = 1; c <= 16; c++) {
            if (span >> c & 1) {
                const float4 x2 = rows[c][col];
                ux[c] = (x2.x - x1.x) * (1.0f / 3.0f);
                uy[c] = (x2.y - x1.y) * (1.0f / 3.0f);
                uz[c] = (x2.z - x1.z) * (1.0f / 3.0f);
            }
        }
        const int wb = T == Terms::kScalar ? terms_b(b) : T == Terms::kTable ? terms_b(int(x1.w)) : 0;
        for (int a0 = 0; a0 <= b; a0 += WHOLE ? 1 : S) {
            const int a = WHOLE ? a0 : min(a0 + sub, b);
            const float4 x0 = rows[a][col];
            const float vx = (x1.x - x0.x) * (2.0f / 3.0f) + x0.x;
            const float vy = (x1.y - x0.y) * (2.0f / 3.0f) + x0.y;
            const float vz = (x1.z - x0.z) * (2.0f / 3.0f) + x0.z;
            const float4 *ta = terms + wb + (T == Terms::kScalar ? a : T == Terms::kTable ? int(x0.w) : 0);
            // Table index of (a, b, c): C(c + 2, 3) - 1 + a c + b - a (a - 1) / 2.
            const int pa = b - a * (a - 1) / 2 - 1;
#pragma unroll
            for (int c = 1; c <= 16; c++) {
                if (!(span >> c & 1)) continue;
                const float axr = ux[c] + vx, axg = uy[c] + vy, axb = uz[c] + vz;
                const uint32_t key = tie_key(terms_c(c) + pa + a * c);
                float e;
                if constexpr (T == Terms::kComputed) {
                    float4 x2 = x1;
                    x2.w = xw[c];
                    // + 0: no error is -0 (TameBest).
                    e = eval_from_sum(axr, axg, axb, sum, cluster_terms<true>(x0, x1, x2, sum.w), mx, my, mz, nullptr) + 0.0f;
                } else {
                    const float4 h = T == Terms::kScalar ? ta[terms_c(c)]
                                                         : *reinterpret_cast<const float4 *>(
                                                               reinterpret_cast<const char *>(ta) + __float_as_int(xw[c]));
                    e = half_error_from_sum(axr, axg, axb, sum, h);
                }
                best.offer(e, key);
            }
        }
    }
}

// cluster_fit_three (icbc.h:2016-2247), the same way: pairs (c0, c1 = t) for
// t = 1..m.  m need not be the same in every lane.
template <bool WHOLE, Terms T>
__device__ __forceinline__ void search3(LaneRows rows, int col, int sub, int S, int m, float4 sum, float mx, float my,
                                        float mz, const float4 *terms, TameBest &best)
{
    for (int b = 1; b <= m; b++) {
        const float4 x1 = rows[b][col];
        const float4 *tb = terms + (T == Terms::kScalar ? terms_b(b) : T == Terms::kTable ? terms_b(int(x1.w)) : 0);
        const int pb = b * (b + 1) / 2 - 1;
        for (int a0 = 0; a0 <= b; a0 += WHOLE ? 1 : S) {
            const int a = WHOLE ? a0 : min(a0 + sub, b);
            const float4 x0 = rows[a][col];
            const float axr = x0.x + (x1.x - x0.x) * 0.5f;
            const float axg = x0.y + (x1.y - x0.y) * 0.5f;
            const float axb = x0.z + (x1.z - x0.z) * 0.5f;
            float e;
            if constexpr (T == Terms::kComputed)
                e = eval_from_sum(axr, axg, axb, sum, cluster_terms<false>(x0, x1, x1, sum.w), mx, my, mz, nullptr) + 0.0f;
            else
                e = half_error_from_sum(axr, axg, axb, sum, tb[T == Terms::kScalar ? a : int(x0.w)]);
            best.offer(e, tie_key(pb + a));
        }
    }
}

// The entries that the SSE build's four-wide loops read past the table of
// `count` entries: prefixes (0, q, n + 1), whose row n + 1 is FLT_MAX.  Over
// tame texels their endpoints come out as 0 (every product overflows to an
// infinity or a NaN, which saturates to 0) with an error of 0.
__device__ __forceinline__ void offer_past_end(int count, TameBest &best)
{
    for (int p = count; p & 3; p++) best.offer(0.0f, tie_key(p));
}

// Both searches over any floats, in the order of the tables, as the SSE
// build evaluates them (every lane of a block alike).
__device__ __forceinline__ Best search4_any(LaneRows rows, int col, int n, float4 sum, float mx, float my, float mz)
{
    Best best;
    int p = 0;
    for (int c = 1; c <= n; c++) {
        const float4 x2 = rows[c][col];
        for (int a = 0; a <= c; a++) {
            const float4 x0 = rows[a][col];
            for (int b = a; b <= c; b++, p++) {
                const float4 x1 = rows[b][col];
                best.offer(eval_terms<true>(x0, x1, x2, sum, cluster_terms<true>(x0, x1, x2, sum.w), mx, my, mz, nullptr),
                           p);
            }
        }
    }
    const float4 x0 = rows[0][col], x2 = rows[n + (n < 16 ? 1 : 0)][col];
    for (int q = 0; p & 3; q++, p++) {
        const float4 x1 = rows[q][col];
        best.offer(eval_terms<true>(x0, x1, x2, sum, cluster_terms<true>(x0, x1, x2, sum.w), mx, my, mz, nullptr), p);
    }
    return best;
}

__device__ __forceinline__ Best search3_any(LaneRows rows, int col, int m, float4 sum, float mx, float my, float mz)
{
    Best best;
    int p = 0;
    for (int b = 1; b <= m; b++) {
        const float4 x1 = rows[b][col];
        for (int a = 0; a <= b; a++, p++) {
            const float4 x0 = rows[a][col];
            best.offer(eval_terms<false>(x0, x1, x1, sum, cluster_terms<false>(x0, x1, x1, sum.w), mx, my, mz, nullptr), p);
        }
    }
    const float4 x1 = rows[m + (m < 16 ? 1 : 0)][col];
    for (int q = 0; p & 3; q++, p++) {
        const float4 x0 = rows[q][col];
        best.offer(eval_terms<false>(x0, x1, x1, sum, cluster_terms<false>(x0, x1, x1, sum.w), mx, my, mz, nullptr), p);
    }
    return best;
}

// What a search workgroup keeps in LDS beside its rows: the weight terms, the
// cluster tables (five bits a prefix), and the tables that the endpoints and
// the palette look up (a chain of gathers from memory after every search
// otherwise).
struct SearchTables {
    TermTables terms;
    uint16_t four[976], three[160];
    float mid5[32], mid6[64], div255[256];
};
__device__ __forceinline__ uint16_t pack_prefixes(uint32_t c) { return uint16_t((c & 31) | (c >> 8 & 31) << 5 | (c >> 16 & 31) << 10); }
__device__ __forceinline__ void load_search_tables(SearchTables &st, const ntx::Tables *tab, int t, int nthreads)
{
    load_term_tables(st.terms, tab, t, nthreads);
    for (int i = t; i < 976; i += nthreads) st.four[i] = pack_prefixes(tab->four[i]);
    for (int i = t; i < 160; i += nthreads) st.three[i] = pack_prefixes(tab->three[i]);
    for (int i = t; i < 256; i += nthreads) st.div255[i] = tab->div255[i];
    if (t < 64) st.mid6[t] = tab->mid6[t];
    if (t < 32) st.mid5[t] = tab->mid5[t];
}

// The winning candidate's endpoints (the SSE build keeps lane 0's zeros when
// no candidate beat FLT_MAX).
template <bool FOUR>
__device__ __forceinline__ Cand lane_winner(LaneRows rows, int col, const Best &best, float4 sum, float mx, float my,
                                           float mz, const SearchTables &st)
{
    Cand c = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f };
    if (!(best.e < FLT_MAX)) return c;
    const uint32_t packed = FOUR ? st.four[best.index()] : st.three[best.index()];
    const float4 x0 = rows[packed & 31][col];
    const float4 x1 = rows[(packed >> 5) & 31][col];
    const float4 x2 = FOUR ? rows[packed >> 10][col] : x1;
    eval_terms<FOUR>(x0, x1, x2, sum, cluster_terms<FOUR>(x0, x1, x2, sum.w), mx, my, mz, &c);
    return c;
}

// output_block4 / output_block3 (icbc.h:2944-2980) for one lane's block:
// 5:6:5 endpoints (vector3_to_color16), order, the D3D10 palette, each
// texel's index (compute_indices4 / compute_indices3 with transparent
// black), and evaluate_mse summed in texel order.
template <bool FOUR>
__device__ __forceinline__ float lane_output(const Cand &c, const BlockTexels &texels, float cwx, float cwy, float cwz,
                                             const float *mid5, const float *mid6, const float *div255, uint2 *blk)
{
    float4 next[4];
    texels.row(0, next);
    uint32_t c0 = to565(c.ax, c.ay, c.az, mid5, mid6);
    uint32_t c1 = to565(c.bx, c.by, c.bz, mid5, mid6);
    if (FOUR ? (c0 < c1) : (c0 > c1)) { const uint32_t tmp = c0; c0 = c1; c1 = tmp; }
    float p[4][3];
    palette(c0, c1, p, div255);
    float pw[4][3];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        pw[k][0] = p[k][0] * cwx;
        pw[k][1] = p[k][1] * cwy;
        pw[k][2] = p[k][2] * cwz;
    }
    float err = 0.0f;
    uint32_t bits = 0;
#pragma unroll 1
    for (int r = 0; r < 4; r++) {
        float4 t[4];
#pragma unroll
        for (int i = 0; i < 4; i++) t[i] = next[i];
        if (r < 3) texels.row(r + 1, next);
        uint32_t four = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float tr = t[i].x, tg = t[i].y, tb = t[i].z, tw = t[i].w;
            const float vr = tr * cwx, vg = tg * cwy, vb = tb * cwz;
            float d[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                float dr, dg, db;
                if (FOUR) { dr = vr - pw[k][0]; dg = vg - pw[k][1]; db = vb - pw[k][2]; }
                else { dr = pw[k][0] - vr; dg = pw[k][1] - vg; db = pw[k][2] - vb; }
                d[k] = dr * dr + dg * dg + db * db;
            }
            uint32_t idx;
            if (FOUR) {
                // compute_indices4 (icbc.h:2803-2825).
                const bool x0 = ((d[1] > d[2]) && (d[0] > d[2])) || ((d[0] > d[3]) && (d[1] > d[3]));
                const bool x1 = (d[0] > d[3]) && (d[2] > d[3]);
                idx = (x1 ? 1u : 0u) | (x0 ? 2u : 0u);
            } else {
                // compute_indices3 with allow_transparent_black (icbc.h:2836-2856).
                const float d3 = vr * vr + vg * vg + vb * vb;
                const bool i1 = d[1] < d[2];
                const bool i2 = (d[2] <= d[0]) && (d[2] <= d[1]);
                const bool i3 = (d3 <= d[0]) && (d3 <= d[1]) && (d3 <= d[2]);
                idx = ((i1 || i3) ? 1u : 0u) | ((i2 || i3) ? 2u : 0u);
            }
            // evaluate_mse (icbc.h:2738-2749) term of this texel.
            const float qr = idx == 0 ? p[0][0] : idx == 1 ? p[1][0] : idx == 2 ? p[2][0] : p[3][0];
            const float qg = idx == 0 ? p[0][1] : idx == 1 ? p[1][1] : idx == 2 ? p[2][1] : p[3][1];
            const float qb = idx == 0 ? p[0][2] : idx == 1 ? p[1][2] : idx == 2 ? p[2][2] : p[3][2];
            const float er = ((qr - tr) * cwx) * 255.0f;
            const float eg = ((qg - tg) * cwy) * 255.0f;
            const float eb = ((qb - tb) * cwz) * 255.0f;
            err += tw * (er * er + eg * eg + eb * eb);
            four |= idx << (2 * i);
        }
        bits |= four << (8 * r);
    }
    blk->x = c0 | (c1 << 16);
    blk->y = bits;
    return err;
}

}  // namespace ntx_bc1
