// device.h -- the per-column device stages shared by libgudni_hip's kernels:
// threshold generation, the per-column sort, the coverage / compositing sweep
// and the work-unit driver (see raster.hip for the launch structure).
//
// Numerics: compiled with -ffp-contract=off and correctly rounded FP32
// division, and every FP32 expression is evaluated in the order the
// reference writes it, so records, their order and the coverage sums are
// bit-identical to a strict (non-relaxed) evaluation of Kernels.cl.
// min/max are the OpenCL definitions: max(x,y) = x < y ? y : x,
// min(x,y) = y < x ? y : x.
#pragma once
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <cstdint>

#include "gudni_hip.h"
#include "internal.h"

namespace gudni {
namespace dev {

constexpr uint32_t kPositiveSlope = 0x80000000u;
constexpr uint32_t kPersist = 0x40000000u;
constexpr uint32_t kPersistAndSlope = 0xC0000000u;
constexpr uint32_t kPersistTop = 0xC0000000u;
constexpr uint32_t kPersistBottom = 0x40000000u;
constexpr uint32_t kUnpersist = 0xBFFFFFFFu;
constexpr uint32_t kShapeBitMask = 0x0FFFFFFFu;
// Shape labels are below 128 (maxShapes <= 127), so only the low seven bits
// of the shape-bit field carry them; the adjoint keeps a record's origin in
// the bits above.
constexpr uint32_t kLabelMask = 0x7Fu;
// Fill rule (extension): records of a nonzero-fill shape carry kNonzero, and
// kReversed when their strand runs against the outline (bits 29 and 28,
// which the reference leaves clear: its bit 29 "enable" is unused on this
// path and its shape bits never exceed 127).
constexpr uint32_t kNonzero = 0x20000000u;
constexpr uint32_t kReversed = 0x10000000u;
// Per-lane words of the shape scratch: [0, 128) shape indices of a general
// tile's bits, [128, 256) winding numbers of nonzero-fill shapes by label.
constexpr int kSidxWords = 256;
constexpr int kWindOffset = 128;
constexpr int kOriginShift = 7;
constexpr uint32_t kOriginMask = 0x3FFFFFu;   // 22 bits: bits 7..28
constexpr float kMinCrop = 0.2f;          // MINCROP (Kernels.cl:47)
constexpr float kFlatness = 0.25f;        // TAXICAB_FLATNESS (Kernels.cl:250)

constexpr uint64_t kTagTypeMask = 0xC000000000000000ull;
constexpr uint64_t kTagSolid = 0x8000000000000000ull;
constexpr uint64_t kTagCompoundMask = 0x3000000000000000ull;
constexpr uint64_t kTagContinue = 0x1000000000000000ull;
constexpr uint64_t kTagAdd = 0x2000000000000000ull;
constexpr uint64_t kTagIdMask = 0x07FFFFFFFFFFFFFFull;   // bit 59 is the fill rule
constexpr uint64_t kTagNonzero = GUDNI_TAG_NONZERO;
// Both type bits set: a gradient substance (an extension; the reference
// knows solids and pictures only).
constexpr uint64_t kTagGradient = 0xC000000000000000ull;

constexpr int kWave = 64;
constexpr int kFastCapLog2 = 7;           // 128-record rings in the fast pass
constexpr long kSectionGuard = 1L << 22;  // sweep-length bound per column: the
                                          // longest legitimate sweep is 256 rows
                                          // x (2*4096+1) sections = 2.1M
constexpr int kRadixMaxBits = 5;          // widest digit of the sort's radix pass
constexpr int kMaxBisect = 64;            // bifurcation bound per intersection

// status codes a lane can raise (bit flags in the launch's status word)
// Control words of a launch: per-part work counters of the fast pass, the
// retry pass's counter, the status word, the retry list (count, units).
constexpr int kParts = 8;                  // one work range per XCD
constexpr int kCtlFast = 0, kCtlSlow = kParts, kCtlStatus = kParts + 1, kCtlRetry = kParts + 2;
constexpr int kCtlWords = kCtlRetry + 1;   // words before the retry entries
constexpr uint32_t kStatusOverflow = 1u;   // live queue > maxThresholds
constexpr uint32_t kStatusGuard = 2u;      // section guard hit

struct Thr { float top, bottom, left, right; };

// The scene buffers are read-only for the whole launch.  Reading them through
// the constant address space says so, which lets wave-uniform reads (the
// shape records and strand headers every lane walks) go to the scalar unit.
#define GUDNI_CONST __attribute__((address_space(4)))
template <typename T>
__device__ __forceinline__ const GUDNI_CONST T *ro(const T *p)
{
    return (const GUDNI_CONST T *)(p);
}
__device__ __forceinline__ float4 ld4(const GUDNI_CONST uint8_t *p)
{
    const GUDNI_CONST float *q = reinterpret_cast<const GUDNI_CONST float *>(p);
    return make_float4(q[0], q[1], q[2], q[3]);
}
__device__ __forceinline__ float2 ld2(const GUDNI_CONST uint8_t *p)
{
    const GUDNI_CONST float *q = reinterpret_cast<const GUDNI_CONST float *>(p);
    return make_float2(q[0], q[1]);
}

__device__ __forceinline__ float cl_max(float x, float y) { return x < y ? y : x; }
__device__ __forceinline__ float cl_min(float x, float y) { return y < x ? y : x; }

__device__ __forceinline__ bool hdr_pos(uint32_t h) { return (h & kPositiveSlope) != 0u; }
__device__ __forceinline__ bool hdr_persist(uint32_t h) { return (h & kPersist) != 0u; }
__device__ __forceinline__ bool hdr_persist_top(uint32_t h) { return (h & kPersistAndSlope) == kPersistTop; }
__device__ __forceinline__ bool hdr_persist_bottom(uint32_t h) { return (h & kPersistAndSlope) == kPersistBottom; }

// thresholdInvertedSlope (Kernels.cl:240-246)
__device__ __forceinline__ float inv_slope(uint32_t h, const Thr &t)
{
    const float sgn = hdr_pos(h) ? 1.0f : -1.0f;
    return (t.top == t.bottom) ? FLT_MAX : (t.right - t.left) / (t.bottom - t.top) * sgn;
}
__device__ __forceinline__ float top_x(uint32_t h, const Thr &t) { return hdr_pos(h) ? t.left : t.right; }

// thresholdIntersectX (Kernels.cl:900-913)
__device__ __forceinline__ float intersect_x(uint32_t h, const Thr &t, float y)
{
    if (t.left == t.right) return t.left;
    const float sy = hdr_pos(h) ? t.top : t.bottom;
    return ((y - sy) * inv_slope(h, t)) + t.left;
}

// thresholdIsBelow (Kernels.cl:1079-1094): a sorts after b
__device__ __forceinline__ bool is_below(uint32_t ah, const Thr &a, uint32_t bh, const Thr &b)
{
    if (a.top > b.top) return true;
    if (a.top == b.top) {
        const float ax = top_x(ah, a), bx = top_x(bh, b);
        if (ax > bx) return true;
        if (ax == bx && inv_slope(ah, a) > inv_slope(bh, b)) return true;
    }
    return false;
}

// Launch-wide read-only inputs.
// One scene: its read-only buffers and its frame.
struct alignas(16) SceneDesc {
    const uint8_t *geo;           // strand heap
    const ShapeRec *shapes;       // shape references (tile shape_start indexes here)
    const float4 *bounds;         // per reference: strand extent (xmin, ymin, xmax, ymax)
    const float4 *substances;
    const uint8_t *pict;
    const PictUse *uses;
    uint32_t *out;                // BGRA words
    float4 *out_f32;              // optional pre-quantisation colours
    const float4 *grads;          // gradient records, 7 float4 each
    float bg[4];                  // background RGBA
    int32_t width, height;
    int32_t filter;               // picture sampling: 0 nearest, 1 bilinear
    int32_t sort_bits;            // radix digit width of the record sort (0: insertion only)
};

struct Frame {
    const SceneDesc *scenes;      // scene table (one entry for a single frame)
    const int32_t *tile_scene;    // scene of each tile (null: all scene 0)
    unsigned long long *scene_done; // wall clock when a scene's last unit ended
    const TileRec *tiles;         // tile records, shape_start absolute
    const int32_t *tile_job;      // job index per tile
    const uint32_t *work;         // work units: tile << 2 | quarter
    int32_t n_work;
    const float *random;
    int32_t compute_depth, max_shapes, max_thresholds, random_mask;
    float stochastic;
    int32_t coverage_mode;
    int32_t out_rgba;             // pixel words in R,G,B,A byte order, else the reference's B,G,R,A
    // scratch
    float4 *q_thr;                // [slots][64][cap]
    uint32_t *q_hdr;              // [slots][64][cap]
    int32_t *shape_idx;           // [slots][max_shapes][64]
    int32_t cap_log2, slot_log2;  // records of a lane's ring; of a wave slot's rings
    int32_t split;                // a unit's 64 columns are run by 2^split waves, 64 >> split lanes each
    // control
    uint32_t *counter;            // work counters of this pass, one per part
    int32_t n_parts;              // parts the work list is cut into
    uint32_t *status;             // OR of lane status flags
    uint32_t *retry;              // [0] = count, [1..] = abandoned parts of work units (unit index << split | part)
    int32_t retry_capacity;
    // dump hooks (Level-1 test path), null in normal runs
    float4 *dump_pre_thr; uint32_t *dump_pre_hdr;
    float4 *dump_thr; uint32_t *dump_hdr;
    int32_t *dump_qlen; uint32_t *dump_bits; uint64_t *dump_stack; int32_t *dump_sidx;
    int32_t dump_cap, threads_per_tile;
    // stage cycle counters (null unless timing): [0] generate [1] sort
    // [2] render [3] work units, summed over waves
    unsigned long long *stage_cycles;
};

// A lane's threshold queue: a ring of its own in the wave slot's scratch.
// Logical element 0 is the front of the reference's ThresholdQueue
// (qSlice.sStart).  A ring's records are contiguous, so the few records at
// the front of a queue, which the sweep reads again and again, share cache
// lines (with the rings of a wave interleaved record by record, as the
// reference interleaves its threshold columns, the 4096^2 frame took 3.6%
// longer).
struct Queue {
    float4 *thr;      // the lane's ring (cap records)
    uint32_t *hdr;
    int head, len, mask, maxt;
    // The sweep keeps a span's active records apart from the waiting ones, in
    // the ring's rows from its end on: the end never moves (records come and
    // go at the front), so a waiting record is inserted and removed without
    // the active ones being moved.
    int n_active;
    bool spilled;     // ring too small: abandon the unit
    bool overflow;    // live queue > maxThresholds (reference would corrupt)

    __device__ __forceinline__ void reset()
    {
        head = len = n_active = 0;
        spilled = overflow = false;
    }
    __device__ __forceinline__ int row(int i) const { return (head + i) & mask; }
    __device__ __forceinline__ Thr active(int i) const { return get(len + i); }
    __device__ __forceinline__ uint32_t active_h(int i) const { return get_h(len + i); }
    __device__ __forceinline__ void set_active(int i, uint32_t h, const Thr &t) { set(len + i, h, t); }
    __device__ __forceinline__ Thr get(int i) const
    {
        const float4 v = thr[row(i)];
        return Thr{v.x, v.y, v.z, v.w};
    }
    __device__ __forceinline__ uint32_t get_h(int i) const { return hdr[row(i)]; }
    __device__ __forceinline__ void set(int i, uint32_t h, const Thr &t)
    {
        const int r = row(i);
        thr[r] = make_float4(t.top, t.bottom, t.left, t.right);
        hdr[r] = h;
    }
    // pushTopSlot (Kernels.cl:402-405)
    __device__ __forceinline__ bool push_slot()
    {
        if (len + n_active + 1 > maxt) { overflow = true; return false; }
        if (len + n_active > mask) { spilled = true; return false; }
        head = (head - 1) & mask;
        ++len;
        return true;
    }
    __device__ __forceinline__ void pop() { head = (head + 1) & mask; --len; }
};

// Work claiming.  The list is cut into n_parts contiguous ranges; block b
// starts on range b % n_parts.  Workgroups are dispatched to the XCDs round
// robin, so with one range per XCD a wave first drains the range its own
// XCD owns -- neighbouring tiles share shapes, whose records and strands are
// then read through one L2 -- and afterwards helps with the others.  Every
// wave visits every range, so the grid drains completely.
struct Claimer {
    uint32_t *counters;
    int parts, n_work, part0, k, begin, end;
    __device__ void init(uint32_t *c, int n_parts, int n, int first)
    {
        counters = c;
        parts = n_parts;
        n_work = n;
        part0 = first % n_parts;
        k = 0;
        range();
    }
    __device__ void range()
    {
        const int part = (part0 + k) % parts;
        begin = (int)(((long long)n_work * part) / parts);
        end = (int)(((long long)n_work * (part + 1)) / parts);
    }
    // next work index (wave-uniform), or -1 once every range is drained
    __device__ int next(int lane)
    {
        while (k < parts) {
            uint32_t w = 0;
            if (lane == 0) w = atomicAdd(counters + (part0 + k) % parts, 1u);
            w = __builtin_amdgcn_readfirstlane(w);
            if ((int)w < end - begin) return begin + (int)w;
            if (++k < parts) range();
        }
        return -1;
    }
};

struct Column {
    int dx, dy;                   // threadDelta
    int int_height;
    float float_height;
    uint32_t unique;              // threadUnique (random field seed)
    int shape_start, num_shapes;
};

struct Trav { float2 right, left, ctl; float xpos; int index; };

__device__ __forceinline__ float2 mid_point(float2 a, float2 b)
{   // (1-T)*a + T*b with T = 0.5f (Kernels.cl:864-866)
    return make_float2(0.5f * a.x + 0.5f * b.x, 0.5f * a.y + 0.5f * b.y);
}

// bifurcateCurve + intersectCurve (Kernels.cl:1226-1258) + yIntercept (:818-820)
__device__ float intersect_curve(Trav t)
{
    if (!(t.left.x == t.ctl.x && t.left.y == t.ctl.y)) {
        // at most kMaxBisect halvings: a curve inside a 2^30-pixel canvas is
        // flat after ~35; beyond that FP32 can reach a fixed point where an
        // unbounded loop would never end
        for (int it = 0; it < kMaxBisect; ++it) {
            const float2 lm = mid_point(t.left, t.ctl);
            const float2 rm = mid_point(t.ctl, t.right);
            const float2 on = mid_point(lm, rm);
            const float flat = fabsf(t.ctl.x - on.x) + fabsf(t.ctl.y - on.y);
            if (!(flat > kFlatness)) break;
            if (t.xpos < on.x) { t.ctl = lm; t.right = on; }
            else { t.left = on; t.ctl = rm; }
        }
    }
    if (t.left.x == t.right.x) return cl_min(t.left.y, t.right.y);
    return (((t.right.y - t.left.y) / (t.right.x - t.left.x)) * (t.xpos - t.left.x)) + t.left.y;
}

// addThreshold + trimThresholdTop (Kernels.cl:982-1005, 1175-1220)
__device__ __forceinline__ void add_threshold(Queue &q, const Column &c, uint32_t h, Thr t,
                                              bool &added, bool &enclosed)
{
    const bool keep = hdr_persist(h) || ((t.bottom - t.top) >= kMinCrop);
    if (!keep) return;
    enclosed = enclosed || ((t.top <= 0.0f) && hdr_persist_top(h)) ||
               ((t.bottom <= 0.0f) && hdr_persist_bottom(h));
    if (t.top < c.float_height && t.bottom > 0.0f && t.left < 1.0f) {
        if (t.top <= 0.0f) {
            const float sx = intersect_x(h, t, 0.0f);
            if (hdr_pos(h)) { t = Thr{0.0f, t.bottom, sx, t.right}; h &= kUnpersist; }
            else { t = Thr{0.0f, t.bottom, t.left, sx}; }
        }
        if (t.right <= 0.0f) {
            enclosed = true;
        } else {
            added = true;
            if (q.push_slot()) q.set(0, h, t);
        }
    }
}

// addLineSegment (Kernels.cl:1131-1173)
__device__ __forceinline__ void add_line(Queue &q, const Column &c, float2 l, float2 r,
                                         uint32_t bit, bool &added, bool &enclosed)
{
    const Thr t{cl_min(l.y, r.y), cl_max(l.y, r.y), l.x, r.x};
    const bool pos = l.y <= r.y;
    const bool persistent = (l.x != r.x) && (l.x == 0.0f);
    const uint32_t h = (pos ? kPositiveSlope : 0u) | (persistent ? kPersist : 0u) | bit;
    add_threshold(q, c, h, t, added, enclosed);
}

// spawnThresholds (Kernels.cl:1264-1333)
__device__ void spawn(Queue &q, const Column &c, uint32_t bit, const Trav &l, const Trav &r,
                      bool &added, bool &enclosed)
{
    const float yl = (l.left.x >= 0.0f) ? l.left.y : intersect_curve(l);
    bool lw = false, rw = false;
    if ((l.right.x < 1.0f) && (l.right.x > 0.0f)) {
        add_line(q, c, make_float2(l.xpos, yl), l.right, bit, added, enclosed);
        lw = true;
    }
    const float yr = (r.right.x <= 1.0f) ? r.right.y : intersect_curve(r);
    if ((r.left.x > 0.0f) && (r.left.x < 1.0f) && (l.index != r.index)) {
        add_line(q, c, r.left, make_float2(r.xpos, yr), bit, added, enclosed);
        rw = true;
    }
    if (l.right.x < r.left.x || (!lw && !rw)) {
        const float2 bl = (lw || (l.left.x == l.right.x)) ? l.right : make_float2(l.xpos, yl);
        const float2 br = (rw || (r.left.x == r.right.x)) ? r.left : make_float2(r.xpos, yr);
        add_line(q, c, bl, br, bit, added, enclosed);
    }
}


// searchTree (Kernels.cl:1337-1357) over the strand's Eytzinger tree, for
// the column's left border (l, which also takes a node at its x) and right
// border (r) in one loop: the two descents are independent, so their node
// reads are issued together (the 4096^2 frame: 43.5 -> 42.8 ms).
__device__ __forceinline__ void search_pair(Trav &l, Trav &r, const GUDNI_CONST uint8_t *tree, int tree_size,
                                            float dx, float dy)
{
    l.index = 0;
    r.index = 0;
    while (l.index < tree_size || r.index < tree_size) {
        const bool ml = l.index < tree_size, mr = r.index < tree_size;
        const float4 nl = ld4(tree + 16 * (ml ? l.index : 0));
        const float4 nr = ld4(tree + 16 * (mr ? r.index : 0));
        if (ml) {
            const float px = nl.x - dx, py = nl.y - dy, cx = nl.z - dx, cy = nl.w - dy;
            if ((l.xpos < px) || (l.xpos == px)) {
                l.right = make_float2(px, py);
                l.index = (l.index << 1) + 1;
            } else {
                l.left = make_float2(px, py);
                l.ctl = make_float2(cx, cy);
                l.index = (l.index << 1) + 2;
            }
        }
        if (mr) {
            const float px = nr.x - dx, py = nr.y - dy, cx = nr.z - dx, cy = nr.w - dy;
            if (r.xpos < px) {
                r.right = make_float2(px, py);
                r.index = (r.index << 1) + 1;
            } else {
                r.left = make_float2(px, py);
                r.ctl = make_float2(cx, cy);
                r.index = (r.index << 1) + 2;
            }
        }
    }
}

__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A wave's list of sections waiting for their colours: per section its area
// (adj) and the stack it lies under, which the colour pass replaces by colour
// x area.  info: the lane that swept it (bits 0..5), its pixel's row in that
// lane's segment (6..18), whether it is its pixel's last (kSecEnd), and the
// lane's next section in the list (24..31, kSecNone: none).
constexpr int kSections = 192;             // three full waves of colours
constexpr uint32_t kSecEnd = 1u << 19, kSecNone = 0xFFu;
struct SectionList {
    float4 val[kSections];
    float adj[kSections];
    uint32_t info[kSections];
};

// A wave's list of strands that generation walks: extents (left x, right x,
// top, bottom) and the strand's place in the heap (16-byte units) and meta
// word (size in 8-byte units, the shape's index in its group of 64 << 16,
// kStrandNonzero, kStrandReversed, kStrandFar: not to be judged by extents).
constexpr int kStrands = 192;
constexpr uint32_t kStrandNonzero = 1u << 22, kStrandReversed = 1u << 23, kStrandFar = 1u << 24;
struct StrandList {
    float4 box[kStrands];
    uint2 ref[kStrands];
    uint32_t rows[32 * 8];   // rows of 32 of them in a wave's columns, at most 8 (pack_rows)
};

// Per-wave LDS table of a compact tile's shapes by tile-local index: tag,
// and the solid colour (in the coverage mode's form) or, for a picture or
// gradient, the substance record itself.
struct TileTable {
    uint64_t tag[128];
    float4 color[128];
    union {
        SectionList sec;       // the sweep's sections
        StrandList strands;    // generation's strands
        uint16_t hist[(1 << kRadixMaxBits) * kWave];   // the sort's histogram
    };
    int mixed;             // some shape is a picture or gradient (adjoint)
    uint64_t lookup[2];    // shapes that are pictures or gradients (grouped colours)
    int grouped;           // the tile qualifies for grouped colours
    // colour group g holds tile-local shapes [g gq, (g+1) gq), gq = ceil(n / 4)
    // for a tile of n shapes
    uint32_t gq;
};
// traverseTree (Kernels.cl:1378-1408)'s column-relative view of a strand.
__device__ __forceinline__ Trav strand_view(const GUDNI_CONST uint8_t *strand, float dx, float dy)
{
    const float2 right = ld2(strand + 8);
    const float4 lc = ld4(strand + 16);
    Trav t;
    t.right = make_float2(right.x - dx, right.y - dy);
    t.left = make_float2(lc.x - dx, lc.y - dy);
    t.ctl = make_float2(lc.z - dx, lc.w - dy);
    t.xpos = 0.0f;
    t.index = 0;
    return t;
}

// Bounds (lo, hi) on the y of an x-monotone curve over [x0, x1]: the hull of
// the piece between the parameters of x0 and x1 (the roots of its x
// polynomial, by hardware reciprocal and square root: what is off is covered
// by the caller's margin).  False where the parameters are not well defined.
__device__ __forceinline__ bool curve_bounds(const Trav &t, float x0, float x1, float &lo, float &hi)
{
    const float a = (t.left.x - t.ctl.x) + (t.right.x - t.ctl.x), b = t.ctl.x - t.left.x;
    const float b2 = b * b;
    const float d0 = b + __builtin_amdgcn_sqrtf(fmaxf(b2 - a * (t.left.x - x0), 0.0f));
    const float d1 = b + __builtin_amdgcn_sqrtf(fmaxf(b2 - a * (t.left.x - x1), 0.0f));
    const float t0 = fminf(fmaxf((x0 - t.left.x) * __builtin_amdgcn_rcpf(d0), 0.0f), 1.0f);
    const float t1 = fminf(fmaxf((x1 - t.left.x) * __builtin_amdgcn_rcpf(d1), 0.0f), 1.0f);
    // blossom of the y polynomial: (t0,t0), (t0,t1), (t1,t1)
    const float u0 = t.left.y + (t.ctl.y - t.left.y) * t0, v0 = t.ctl.y + (t.right.y - t.ctl.y) * t0;
    const float u1 = t.left.y + (t.ctl.y - t.left.y) * t1, v1 = t.ctl.y + (t.right.y - t.ctl.y) * t1;
    const float ya = u0 + (v0 - u0) * t0, yb = u0 + (v0 - u0) * t1, yc = u1 + (v1 - u1) * t1;
    lo = fminf(lo, fminf(ya, fminf(yb, yc)));
    hi = fmaxf(hi, fmaxf(ya, fmaxf(yb, yc)));
    return d0 > 1e-3f && d1 > 1e-3f;
}

// Bounds (lo, hi), with their margin, on the y of a strand that covers the
// column at dx, relative to dy; false where it has none.  spawn's lines run
// between points of the curve under the left border, of the one under the
// right border, and from one curve to the other.  A border's y is a chord's,
// and a flat chord lies within 0.25 (in x plus y) of its curve; so all of them
// lie within the bounds of both curves over the column widened by half a
// pixel, and the margin: a pixel and 1/256 of the curves' extent.
__device__ __forceinline__ bool strand_bounds(const SceneDesc &s, uint2 ref, float dx, float dy, float &lo, float &hi)
{
    if (ref.y & kStrandFar) return false;
    const GUDNI_CONST uint8_t *strand = ro(s.geo) + 16ull * ref.x;
    Trav l = strand_view(strand, dx, dy), r = l;
    l.xpos = cl_max(0.0f, l.left.x);
    r.xpos = cl_min(1.0f, l.right.x);
    search_pair(l, r, strand + 32, ((int)(ref.y & 0xFFFFu) - 4) / 2, dx, dy);
    lo = FLT_MAX;
    hi = -FLT_MAX;
    bool known = curve_bounds(l, fmaxf(l.left.x, -0.5f), fminf(1.5f, l.right.x), lo, hi);
    float extent = (l.right.x - l.left.x) + fabsf(l.ctl.y - l.left.y) + fabsf(l.right.y - l.ctl.y);
    if (l.index != r.index) {
        known = curve_bounds(r, fmaxf(r.left.x, -0.5f), fminf(1.5f, r.right.x), lo, hi) && known;
        extent = fmaxf(extent, (r.right.x - r.left.x) + fabsf(r.ctl.y - r.left.y) + fabsf(r.right.y - r.ctl.y));
    }
    const float margin = 1.0f + extent * (1.0f / 256.0f);
    lo -= margin;
    hi += margin;
    return known;
}

// Whether a strand that covers the column passes wholly above its segment
// (-1), wholly below (1) or may meet it (0).
__device__ __forceinline__ int strand_side(const SceneDesc &s, uint2 ref, float dx, float dy, float height)
{
    float lo, hi;
    if (!strand_bounds(s, ref, dx, dy, lo, hi)) return 0;
    return hi <= 0.0f ? -1 : (lo >= height ? 1 : 0);
}

// Rows [lo, hi) as 15 and 16 bits (rounded outwards, held to +-kRowMax, which
// the segments' rows stay below), and whether the strand covers the column's
// left border.
constexpr float kRowMax = 16000.0f;
__device__ __forceinline__ uint32_t pack_rows(float lo, float hi, bool border)
{
    const int a = (int)floorf(fminf(fmaxf(lo, -kRowMax), kRowMax)), b = (int)ceilf(fminf(fmaxf(hi, -kRowMax), kRowMax));
    return ((uint32_t)b << 16) | (((uint32_t)a & 0x7FFFu) << 1) | (border ? 1u : 0u);
}
__device__ __forceinline__ int rows_lo(uint32_t w) { return (int)(w << 16) >> 17; }
__device__ __forceinline__ int rows_hi(uint32_t w) { return (int)w >> 16; }
// log2 of a wave's columns (a power of two) where they are at most 8, else -1.
__device__ __forceinline__ int columns_log2(int n) { return n <= 8 ? __ffs(n) - 1 : -1; }

// buildThresholdArray (Kernels.cl:1540-1595): every column of the wave takes
// the strands of its tile's shapes in order and emits their thresholds.
//
// The walk is a lane's own.  Per group of 64 shapes the wave lists the
// strands of those that reach its columns, with their extents; each lane then
// marks the strands that cross its own segment and runs only those, one a
// step, so a step serves a different strand in every lane and there are as
// many steps as the busiest lane has crossing strands (walking strand by
// strand, the wave ran every strand that crossed any of its 64 columns).  A
// wave of at most 8 columns bounds each strand once a column, as many at a
// time as fill its lanes, for all the column's segments; wider ones a lane.
// What the other strands do to a column follows from their extents:
//  * left of or right of the column (the reference's own range test): nothing;
//  * wholly below the segment, by a pixel or more: no threshold, and none that
//    starts at or above its top;
//  * wholly above it, by a pixel or more: no threshold either, but a strand
//    that covers the column's left border has a persistent threshold there,
//    which ends above the top: the segment's enclosure flips (checkInRange
//    holds and xpos is 0, so the first line starts on the border).
// A strand with a coordinate at or beyond 2^20 (whose rounding the pixel does
// not cover) or NaN is always run.  Strands are then bounded within the very
// column (strand_bounds): on the 4096^2 frame a wave lists 510 strands, 200
// reach some of its columns, 57 of them a lane's segment by their extents, and
// a column takes 5.5 records.
// Generation of that frame took 95e9 wave cycles when every strand that crosses
// some column was run, 60e9 with the choice made a lane, and 36e9 with it made
// a column; 512^2 scribbles 51e9, 31e9 and 22e9.  What is left is bound by its
// busiest lane's strands and, a third of it, by listing: a strand's place is
// known when the one before it is read, one read's latency a strand.
//
// kCompact (a tile of at most maxShapes shapes, i.e. every tile above the
// 8-pixel floor): the 127-shape cap cannot bind, and the column's shape bit
// b is a monotone relabelling of the tile-local shape index n (b = number of
// contributing shapes before n).  Labelling headers and the stack by n
// instead visits the same shapes in the same order everywhere, and lets the
// compositing walk read tags and colours from a per-tile table in LDS
// instead of chasing shapeIndices[b] -> shape record -> substance in memory.
// `contrib` records which n contributed, so the reference's labels can be
// recovered (dump path).
// emit(place, meta, label and rule bits, added, enclosed) runs one strand.
template <bool kCompact, class Emit>
__device__ __forceinline__ void walk_strands(const Frame &f, const SceneDesc &s, const Queue &q, const Column &c,
                                             bool active, int lane, float span0, float span1, int32_t *sidx,
                                             StrandList &list, int cols_log2, uint32_t &shape_bits, uint64_t &stack0,
                                             uint64_t &stack1, uint64_t &contrib0, uint64_t &contrib1,
                                             bool &any_nonzero, Emit &&emit)
{
    const float dx = (float)c.dx, dy = (float)c.dy;
    const uint32_t max_shapes = (uint32_t)f.max_shapes;
    const int num_shapes = (int)__builtin_amdgcn_readfirstlane(c.num_shapes);
    const int shape_start = (int)__builtin_amdgcn_readfirstlane(c.shape_start);
    float highest = active ? dy : FLT_MAX;
    for (int o = 32; o > 0; o >>= 1) highest = fminf(highest, __shfl_xor(highest, o));
    const float ux = span0 + 1.0f;
    const int my_col = (int)(dx - ux), my_row = (int)(dy - highest), my_end = my_row + c.int_height;
    if (__any(active && (float)my_end >= kRowMax)) cols_log2 = -1;
    const int cmask = (1 << (cols_log2 & 3)) - 1;
    const float below = dy + c.float_height + 1.0f, above = dy - 1.0f;
    float lowest = active ? below : -FLT_MAX;   // nothing below it reaches the wave
    for (int o = 32; o > 0; o >>= 1) lowest = fmaxf(lowest, __shfl_xor(lowest, o));
    bool alive = active;
    for (int base = 0; base < num_shapes; base += kWave) {
        alive = alive && shape_bits < max_shapes && !q.spilled && !q.overflow;
        if (!__any(alive)) break;
        // a shape none of whose strands reaches a column adds no threshold
        // and no enclosure there: those that miss [span0, span1] (the wave's
        // columns widened by a pixel) are left out
        const int ni = base + lane;
        uint32_t ns = 0, place = 0, rule = 0;
        float shape_top = 0.0f;
        if (ni < num_shapes) {
            const float4 b = s.bounds[shape_start + ni];
            shape_top = b.y;
            if (b.x <= span1 && b.z > span0 && !(b.y >= lowest)) {
                const ShapeRec r = s.shapes[shape_start + ni];
                ns = r.num_strands;
                place = r.geo_start;
                rule = (r.tag & kTagNonzero) ? kStrandNonzero : 0u;
            }
        }
        uint32_t start = ns;
        for (int o = 1; o < kWave; o <<= 1) {
            const uint32_t t = __shfl_up(start, (unsigned)o);
            if (lane >= o) start += t;
        }
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)start, kWave - 1);
        start -= ns;
        uint64_t enc = 0, add = 0;   // shapes of the group that enclose the corner; that added records
        int cur = -1;                // the nonzero-fill shape whose winding number w is being summed
        int32_t w = 0;
        auto label_of = [&](int k) -> uint32_t {
            return kCompact ? (uint32_t)(base + k)
                            : shape_bits + (uint32_t)__popcll((enc | add) & ((1ull << k) - 1ull));
        };
        auto close_winding = [&]() {
            if (cur < 0) return;
            if (w != 0) enc |= 1ull << cur;
            const uint32_t label = label_of(cur);
            if ((((enc | add) >> cur) & 1ull) && label < max_shapes) sidx[(kWindOffset + (int)label) * kWave] = w;
            cur = -1;
        };
        uint32_t listed = 0;         // strands of this lane's shape listed so far
        uint32_t n = 0;              // strands in the list
        for (uint32_t w0 = 0; w0 < total;) {
            const uint32_t w1 = min(total, w0 + (uint32_t)kStrands - n);
            wave_sync();
            if (listed < ns && start + listed < w1) {
                // the next strand's head and first curve come with this
                // one's curves
                const GUDNI_CONST uint8_t *p = ro(s.geo) + 16ull * place;
                float4 h = ld4(p);
                for (bool more = true; more;) {
                    const uint32_t head = __float_as_uint(h.x), size = head & 0xFFFFu;
                    const int m = (int)size / 2;   // float4s of the strand
                    const uint32_t e = n + start + listed - w0;
                    ++listed;
                    more = listed < ns && start + listed < w1;
                    const GUDNI_CONST uint8_t *next = p + 16 * m;
                    const float4 first = ld4(p + 16), nh = ld4(more ? next : p);
                    float4 v = m > 2 ? ld4(p + 32) : first;
                    float lo = fminf(h.w, fminf(first.y, first.w)), hi = fmaxf(h.w, fmaxf(first.y, first.w));
                    // the largest magnitude, as bits: those of a NaN exceed all
                    auto mag = [](float x) { return __float_as_uint(x) & 0x7FFFFFFFu; };
                    auto mag4 = [&](float4 x) { return max(max(mag(x.x), mag(x.y)), max(mag(x.z), mag(x.w))); };
                    uint32_t far = max(max(mag(h.z), mag(h.w)), mag4(first));
                    for (int i = 2; i < m;) {
                        lo = fminf(lo, fminf(v.y, v.w));
                        hi = fmaxf(hi, fmaxf(v.y, v.w));
                        far = max(far, mag4(v));
                        if (++i < m) v = ld4(p + 16 * i);
                    }
                    const bool wild = far >= __float_as_uint(1048576.0f);
                    if (wild) {
                        lo = shape_top;
                        hi = INFINITY;
                    }
                    list.box[e] = make_float4(first.x, h.z, lo, hi);
                    list.ref[e] = make_uint2(place, size | ((uint32_t)lane << 16) | rule | (wild ? kStrandFar : 0u) |
                                                        (rule && ((head >> 16) & GUDNI_STRAND_REVERSED) ? kStrandReversed : 0u));
                    place += size / 2;
                    p = next;
                    h = nh;
                }
            }
            wave_sync();
            // of these, the list keeps those that reach the wave's columns
            const uint32_t end = n + (w1 - w0);
            for (uint32_t e0 = n; e0 < end; e0 += kWave) {
                const uint32_t e = e0 + (uint32_t)lane;
                float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
                uint2 ref = make_uint2(0u, 0u);
                if (e < end) {
                    b = list.box[e];
                    ref = list.ref[e];
                }
                const bool keep = e < end && b.x <= span1 && b.y > span0 && !(b.z >= lowest);
                const uint64_t mask = __ballot(keep);
                if (keep) {
                    const uint32_t at = n + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                                      __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
                    list.box[at] = b;
                    list.ref[at] = ref;
                }
                n += (uint32_t)__popcll(mask);
            }
            w0 = w1;
            if (w0 < total && n <= (uint32_t)kStrands / 2) continue;   // room for more
            wave_sync();
            uint32_t todo[kStrands / 32];   // strands that this lane runs
#pragma unroll
            for (int g = 0; g < kStrands / 32; ++g) todo[g] = 0u;
            // rolled, the word chosen by selects: the body is long
#pragma unroll 1
            for (int e0 = 0; e0 < (int)n; e0 += 32) {
                uint32_t run = 0;
                const int e1 = min(e0 + 32, (int)n);
                if (cols_log2 >= 0) {
                    wave_sync();
                    for (int i = lane; i < (e1 - e0) << cols_log2; i += kWave) {
                        const float4 b = list.box[e0 + (i >> cols_log2)];
                        const uint2 ref = list.ref[e0 + (i >> cols_log2)];
                        const float cx = ux + (float)(i & cmask), cy = highest;
                        const float lx = b.x - cx;
                        uint32_t rows = pack_rows(kRowMax, kRowMax, false);   // does not cover the column
                        if (lx <= 1.0f && b.y - cx > 0.0f) {
                            float lo, hi;
                            if (!strand_bounds(s, ref, cx, cy, lo, hi)) {
                                lo = b.z - cy - 1.0f;
                                hi = b.w - cy + 1.0f;
                            }
                            rows = pack_rows(lo, hi, lx <= 0.0f);
                        }
                        list.rows[i] = rows;
                    }
                    wave_sync();
                    for (int e = e0; e < e1; ++e) {
                        const uint32_t rows = list.rows[((e - e0) << cols_log2) + (my_col & cmask)];
                        const uint32_t meta = __builtin_amdgcn_readfirstlane(list.ref[e].y);
                        const bool over = rows_hi(rows) <= my_row && !(meta & kStrandNonzero);
                        if (!over && rows_lo(rows) < my_end) run |= 1u << (e - e0);
                        if (over && (rows & 1u)) enc ^= 1ull << ((meta >> 16) & 63u);
                    }
                    run = alive ? run : 0u;
                } else {
                    uint32_t m = 0;
                    for (int e = e0; e < e1; ++e) {
                        const float4 b = list.box[e];
                        const uint32_t meta = __builtin_amdgcn_readfirstlane(list.ref[e].y);
                        const float lx = b.x - dx;
                        const bool in = lx <= 1.0f && b.y - dx > 0.0f;
                        const bool over = b.w <= above && !(meta & kStrandNonzero);
                        if (in && !over && !(b.z >= below)) m |= 1u << (e - e0);
                        if (in && over && lx <= 0.0f) enc ^= 1ull << ((meta >> 16) & 63u);
                    }
                    m = alive ? m : 0u;
                    // of those, the ones whose curves come near the segment in
                    // this very column
                    while (__any(m != 0u)) {
                        if (m) {
                            const uint32_t bit = m & (0u - m);
                            m ^= bit;
                            const int e = e0 + __ffs((int)bit) - 1;
                            const uint2 ref = list.ref[e];
                            const int side = strand_side(s, ref, dx, dy, c.float_height);
                            if (side == 0 || (side < 0 && (ref.y & kStrandNonzero))) run |= bit;
                            else if (side < 0 && list.box[e].x - dx <= 0.0f) enc ^= 1ull << ((ref.y >> 16) & 63u);
                        }
                    }
                }
#pragma unroll
                for (int g = 0; g < kStrands / 32; ++g) todo[g] = e0 == 32 * g ? run : todo[g];
            }
            for (;;) {
                int e = -1;
#pragma unroll
                for (int g = 0; g < kStrands / 32; ++g)
                    if (e < 0 && todo[g]) {
                        e = 32 * g + __ffs((int)todo[g]) - 1;
                        todo[g] &= todo[g] - 1u;
                    }
                if (!__any(e >= 0)) break;
                if (e < 0) continue;
                const uint2 ref = list.ref[e];
                const int k = (int)((ref.y >> 16) & 63u);
                const bool nonzero = (ref.y & kStrandNonzero) != 0u;
                if (k != cur) close_winding();
                const uint32_t label = label_of(k);
                if ((!kCompact && label >= max_shapes) || q.spilled || q.overflow) continue;
                const bool reversed = (ref.y & kStrandReversed) != 0u;
                bool added = false, enclosed = false;
                emit(ref.x, ref.y, label | (nonzero ? (kNonzero | (reversed ? kReversed : 0u)) : 0u), added, enclosed);
                if (added) add |= 1ull << k;
                if (nonzero) {
                    // a strand crossing the left border above the segment
                    // adds the sign of its original x direction
                    any_nonzero = true;
                    if (cur < 0) { cur = k; w = 0; }
                    if (enclosed) w += reversed ? -1 : 1;
                } else if (enclosed) {
                    enc ^= 1ull << k;
                }
            }
            n = 0;
        }
        close_winding();
        if (!alive) enc = 0;
        uint64_t both = enc | add;
        if (kCompact) {
            if (base == 0) { stack0 = enc; contrib0 = both; }
            else { stack1 = enc; contrib1 = both; }
            shape_bits += (uint32_t)__popcll(both);
        } else {
            while (both && shape_bits < max_shapes) {
                const int k = __ffsll((long long)both) - 1;
                both &= both - 1;
                sidx[(int)shape_bits * kWave] = shape_start + base + k;
                if ((enc >> k) & 1ull) {
                    if (shape_bits < 64u) stack0 |= 1ull << shape_bits;
                    else stack1 |= 1ull << (shape_bits - 64u);
                }
                ++shape_bits;
            }
        }
    }
    wave_sync();
}

template <bool kCompact>
__device__ __forceinline__ void generate(const Frame &f, const SceneDesc &s, Queue &q, const Column &c, bool active, int lane,
                         float span0, float span1, int32_t *sidx, TileTable *tt, int cols_log2,
                         uint32_t &shape_bits, uint64_t &stack0, uint64_t &stack1,
                         uint64_t &contrib0, uint64_t &contrib1, bool &any_nonzero)
{
    const float dx = (float)c.dx, dy = (float)c.dy;
    walk_strands<kCompact>(f, s, q, c, active, lane, span0, span1, sidx, tt->strands, cols_log2, shape_bits, stack0,
                           stack1, contrib0, contrib1, any_nonzero,
                           [&](uint32_t place, uint32_t meta, uint32_t bit, bool &added, bool &enclosed) {
                               const GUDNI_CONST uint8_t *strand = ro(s.geo) + 16ull * place;
                               Trav l = strand_view(strand, dx, dy), r = l;
                               l.xpos = cl_max(0.0f, l.left.x);
                               r.xpos = cl_min(1.0f, l.right.x);
                               search_pair(l, r, strand + 32, ((int)(meta & 0xFFFFu) - 4) / 2, dx, dy);
                               spawn(q, c, bit, l, r, added, enclosed);
                           });
}

// Stable insertion sort by thresholdIsBelow: the same permutation as the
// reference's bubble sort (Kernels.cl:1962-1976), which never swaps equal
// keys.
__device__ void sort_queue(Queue &q)
{
    for (int i = 1; i < q.len; ++i) {
        const Thr x = q.get(i);
        const uint32_t xh = q.get_h(i);
        int j = i - 1;
        while (j >= 0) {
            const Thr y = q.get(j);
            const uint32_t yh = q.get_h(j);
            if (!is_below(yh, y, xh, x)) break;
            q.set(j + 1, yh, y);
            --j;
        }
        if (j + 1 != i) q.set(j + 1, xh, x);
    }
}

// Stage (b) with a radix pass first.  The records' top digit is a
// monotone key prefix: floor(top * 2^bits / h2), h2 the column segment's
// height rounded up to a power of two (an exact scaling), so bucket order
// never contradicts thresholdIsBelow and equal tops share a bucket.  A
// counting pass (per-lane histogram in LDS), an exclusive scan and a stable
// scatter into the ring's free half order the records by digit; the
// insertion sort then only meets inversions inside a bucket.  Both steps
// are stable, so the permutation is the stable sort's, i.e. the reference's
// bubble sort's.  The 64 lanes of a wave sort their 64 columns in lockstep;
// `hist` is the lane's column of a [32][64] u16 table (the tile table's, in
// the place of generation's strands and the sweep's sections).  Columns with
// fewer than kRadixMin records, or more than half a ring, take the insertion
// sort alone.
constexpr int kRadixMin = 8;

__device__ __forceinline__ int top_digit(float top, float scale, int nb)
{
    const int d = (int)(top * scale);
    return d < 0 ? 0 : (d >= nb ? nb - 1 : d);
}

__device__ void radix_sort_queue(Queue &q, uint16_t *hist, int bits, float height)
{
    const int n = q.len;
    if (bits > 0 && n >= kRadixMin && 2 * n <= q.mask + 1) {
        const int nb = 1 << bits;
        float h2 = 1.0f;
        while (h2 < height) h2 *= 2.0f;
        const float scale = (float)nb / h2;
        for (int b = 0; b < nb; ++b) hist[b * kWave] = 0;
        for (int i = 0; i < n; ++i) {
            const int d = top_digit(q.thr[q.row(i)].x, scale, nb);
            hist[d * kWave] = (uint16_t)(hist[d * kWave] + 1);
        }
        uint32_t sum = 0;
        for (int b = 0; b < nb; ++b) {
            const uint32_t c = hist[b * kWave];
            hist[b * kWave] = (uint16_t)sum;
            sum += c;
        }
        for (int i = 0; i < n; ++i) {
            const Thr t = q.get(i);
            const uint32_t h = q.get_h(i);
            const int d = top_digit(t.top, scale, nb);
            const int pos = hist[d * kWave];
            hist[d * kWave] = (uint16_t)(pos + 1);
            q.set(n + pos, h, t);
        }
        q.head = (q.head + n) & q.mask;
    }
    sort_queue(q);
}

// insertThreshold (Kernels.cl:1105-1124)
__device__ void insert_threshold(Queue &q, uint32_t h, const Thr &t)
{
    if (!q.push_slot()) return;
    int cur = 0;
    while (cur < q.len - 1) {
        const uint32_t oh = q.get_h(cur + 1);
        const Thr o = q.get(cur + 1);
        if (!is_below(h, t, oh, o)) break;
        q.set(cur, oh, o);
        ++cur;
    }
    q.set(cur, h, t);
}

struct Sweep {
    int current;
    float sx0, sy0, sx1, sy1;     // sectionStart / sectionEnd
    float pixel_y;
    uint32_t rnd;
    float active_bottom;          // where the active records end
    // the stack at the column's left border in the current span, and below
    // its active records' ends there
    uint64_t left0, left1, below0, below1;
};

// How a crossing of a record moves through it (the fill rule's sign):
// kCrossRight moving right (horizontalAdvance), kCrossLeft moving back to
// the column's left border (the start of verticalAdvance), kCrossDown moving
// down that border through a persistent record's end there.
enum Cross { kCrossRight, kCrossLeft, kCrossDown };

struct Stack {
    uint64_t s0, s1;
    __device__ __forceinline__ void flip(uint32_t h)
    {
        const uint32_t b = h & kLabelMask;
        if (b < 64u) s0 ^= 1ull << b;
        else s1 ^= 1ull << (b - 64u);
    }
    // Crossing record h: an even-odd shape flips its bit (passHeader,
    // Kernels.cl:298-304).  A nonzero-fill shape adds the crossing's winding
    // change, sign(e.x m.y - e.y m.x) for an edge of original direction e
    // crossed by a move m, to its counter (wind[label * 64], this lane's) and
    // its bit becomes counter != 0.
    // any: some record may carry kNonzero (else this is flip).
    template <Cross kHow>
    __device__ __forceinline__ void cross(uint32_t h, int32_t *wind, bool any)
    {
        if (!any || !(h & kNonzero)) {
            flip(h);
            return;
        }
        const bool rev = (h & kReversed) != 0u;
        int d;
        if (kHow == kCrossDown) {
            d = rev ? -1 : 1;
        } else {
            d = (rev != ((h & kPositiveSlope) != 0u)) ? -1 : 1;
            if (kHow == kCrossLeft) d = -d;
        }
        const uint32_t b = h & kLabelMask;
        int32_t *w = wind + (int)b * kWave;
        const int32_t v = *w + d;
        *w = v;
        const uint64_t m = 1ull << (b & 63u);
        uint64_t &word = b < 64u ? s0 : s1;
        word = v != 0 ? (word | m) : (word & ~m);
    }
};

// splitNext = countActive + nextSlicePoint + sliceActive (Kernels.cl:1007-1077)
// and the rest of verticalAdvance's opening of a span (Kernels.cl:1790-1815):
// the waiting records with the front's top become active, cut at the height
// where the first of them ends or the next record starts, their lower parts
// go back to the waiting records, records without height drop out, and the
// stack passes the ends that lie on the column's left border.  Each record is
// read once into the active rows and once there: the passes the reference
// makes over the active records one after the other (and, in the previous
// form here, the moves of all of them at every insertion) are one.
__device__ float open_span(Queue &q, Sweep &p, Stack &st, int32_t *wind, bool nz)
{
    float slice = FLT_MAX, ends = FLT_MAX;
    Thr t = q.get(0);
    const float top = t.top;
    int n = 0;
    for (;;) {
        if (top < t.bottom) ends = cl_min(ends, t.bottom);
        const uint32_t h = q.get_h(0);
        // the record leaves the front and joins the active rows, whose place
        // does not depend on the front
        q.pop();
        q.set_active(n, h, t);
        ++n;
        if (q.len == 0) break;
        t = q.get(0);
        if (t.top > top) { slice = t.top; break; }
    }
    q.n_active = n;
    slice = cl_min(slice, ends);
    int kept = 0;
    float first_bottom = 0.0f;
    uint64_t b0 = 0, b1 = 0;   // labels whose bottom end lies on the left border
    for (int i = 0; i < n; ++i) {
        uint32_t h = q.active_h(i);
        t = q.active(i);
        bool write = kept != i;
        if (t.top < slice && slice < t.bottom) {
            // splitThreshold + divideThreshold (Kernels.cl:928-979)
            const float sx = intersect_x(h, t, slice);
            uint32_t bh;
            Thr b;
            if (hdr_pos(h)) {
                b = Thr{slice, t.bottom, sx, t.right};
                t = Thr{t.top, slice, t.left, sx};
                bh = h & kUnpersist;
            } else {
                b = Thr{slice, t.bottom, t.left, sx};
                t = Thr{t.top, slice, sx, t.right};
                bh = h;
                h &= kUnpersist;
            }
            write = true;
            if (hdr_persist(bh) || ((b.bottom - b.top) >= kMinCrop)) {
                insert_threshold(q, bh, b);
                if (q.spilled || q.overflow) return slice;
            }
        }
        if (kept == 0) {
            if (t.top == t.bottom) {   // before every record with height: dropped
                if (hdr_persist_top(h)) st.cross<kCrossDown>(h, wind, nz);
                continue;
            }
            first_bottom = t.bottom;
        }
        if (t.top > 0.0f && hdr_persist_top(h)) st.cross<kCrossDown>(h, wind, nz);
        if (hdr_persist_bottom(h)) {
            const uint32_t b = h & kLabelMask;
            if (b < 64u) b0 ^= 1ull << b;
            else b1 ^= 1ull << (b - 64u);
        }
        if (write) q.set_active(kept, h, t);
        ++kept;
    }
    q.n_active = kept;
    p.active_bottom = first_bottom;
    p.below0 = st.s0 ^ b0;
    p.below1 = st.s1 ^ b1;
    return slice;
}

// verticalAdvance (Kernels.cl:1744-1824), for a lane whose section reached the
// right border (sx1 == 1).  nz: some record may belong to a nonzero-fill
// shape, whose winding counters (wind, this lane's) the crossings step; the
// stack alone is put back from what it was at the left border.
__device__ void vertical_advance(Queue &q, const Column &c, Sweep &p, Stack &st, int32_t *wind = nullptr,
                                 bool nz = false)
{
    if (nz) {
        for (int i = 0; i < q.n_active; ++i) st.cross<kCrossLeft>(q.active_h(i), wind, nz);
    } else {
        st.s0 = p.left0;
        st.s1 = p.left1;
    }
    const float next_break = cl_min(c.float_height, p.pixel_y);
    if (q.n_active > 0 && p.active_bottom == p.sy1) {
        if (nz) {
            for (int i = 0; i < q.n_active; ++i) {
                const uint32_t h = q.active_h(i);
                if (hdr_persist_bottom(h)) st.cross<kCrossDown>(h, wind, nz);
            }
        } else {
            st.s0 = p.below0;
            st.s1 = p.below1;
        }
        q.n_active = 0;
    }
    float next_bottom;
    if (q.n_active > 0) {
        next_bottom = cl_min(p.active_bottom, next_break);
    } else {
        const float next_top = q.len > 0 ? q.get(0).top : FLT_MAX;
        if (next_top > p.sy1) {
            next_bottom = cl_min(next_break, next_top);
        } else {
            next_bottom = cl_min(next_break, open_span(q, p, st, wind, nz));
            if (q.spilled || q.overflow) return;
        }
    }
    p.left0 = st.s0;
    p.left1 = st.s1;
    p.sy0 = p.sy1;
    p.sy1 = next_bottom;
    p.sx0 = p.sx1 = 0.0f;
    p.current = 0;
}

__device__ __forceinline__ float4 composite(const float4 fg, const float4 bg)
{   // composite (Kernels.cl:878-887)
    const float a = fg.w + bg.w * (1.0f - fg.w);
    if (a > 0.0f) {
        const float k = 1.0f - fg.w;
        return make_float4(((fg.x * fg.w) + (bg.x * bg.w * k)) / a,
                           ((fg.y * fg.w) + (bg.y * bg.w * k)) / a,
                           ((fg.z * fg.w) + (bg.z * bg.w * k)) / a, a);
    }
    return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

__device__ __forceinline__ int f2i_rtz(float v)
{
    if (!(v == v)) return 0;
    if (v >= 2147483647.0f) return 2147483647;
    if (v <= -2147483648.0f) return (-2147483647 - 1);
    return (int)v;
}

__device__ __forceinline__ int f2i_floor(float v)
{
    if (!(v == v)) return 0;
    if (v >= 2147483647.0f) return 2147483647;
    if (v <= -2147483648.0f) return (-2147483647 - 1);
    return (int)floorf(v);
}

// b / 255 for a byte b, correctly rounded: 1/255 as a sum of two floats, which
// equals the IEEE division for every one of the 256 bytes.
__device__ __forceinline__ float unit_byte(uint32_t b)
{
    const float x = (float)b;
    return fmaf(x, 0x1.010102p-8f, x * -0x1.fdfdfep-33f);
}
__device__ __forceinline__ float4 unit_bytes(uint32_t v)
{
    return make_float4(unit_byte(v & 0xFFu), unit_byte((v >> 8) & 0xFFu), unit_byte((v >> 16) & 0xFFu),
                       unit_byte(v >> 24));
}

// Two texels of a row (4-byte aligned, read as one).
struct TexelPair {
    uint32_t left, right;
};

// Texel (x, y) of a picture use, transparent black outside it.  The
// coordinates are taken as unsigned, so a negative one is outside too; a
// texel's byte offset fits in 31 bits (validate_uses).
__device__ __forceinline__ float4 texel(const SceneDesc &s, const PictUse &u, uint32_t x, uint32_t y)
{
    if (x >= (uint32_t)u.w || y >= (uint32_t)u.h) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const uint32_t off = (uint32_t)u.mem_offset + 4u * (y * (uint32_t)u.w + x);
    return unit_bytes(*reinterpret_cast<const uint32_t *>(s.pict + off));
}

// Gradient substance at the pixel's integer position (where pictures are
// sampled too): linear from (x0,y0) to (x1,y1) or radial around (x0,y0) with
// radius x1, stops interpolated piecewise linearly.  Where the wave asks for one
// gradient (kUniform) the whole record is read at once, by scalar loads, and a
// lane's stops are selects; else they are a second, dependent read, which
// takes fewer registers.
template <bool kUniform>
__device__ __forceinline__ float4 eval_gradient(const GUDNI_CONST uint8_t *g, int ax, int ay)
{
    const float4 h0 = ld4(g), h1 = ld4(g + 16), off = ld4(g + 32);
    float4 c0, c1, c2, c3;
    if (kUniform) {
        c0 = ld4(g + 48);
        c1 = ld4(g + 64);
        c2 = ld4(g + 80);
        c3 = ld4(g + 96);
    }
    const int kind = (int)__float_as_uint(h0.x);
    int n = (int)__float_as_uint(h0.y);
    const float x0 = h0.z, y0 = h0.w, x1 = h1.x, y1 = h1.y;
    const float px = (float)ax, py = (float)ay;
    // radial: |p - c| / radius; linear: (p - a).(b - a) / |b - a|^2 -- one
    // division for both, so a wave with both kinds divides once
    float num, den;
    if (kind == 1) {
        const float ex = px - x0, ey = py - y0;
        num = sqrtf((ex * ex) + (ey * ey));
        den = x1;
    } else {
        const float dx = x1 - x0, dy = y1 - y0;
        num = ((px - x0) * dx) + ((py - y0) * dy);
        den = (dx * dx) + (dy * dy);
    }
    float t = den > 0.0f ? num / den : 0.0f;
    t = cl_min(cl_max(t, 0.0f), 1.0f);
    n = n < 1 ? 1 : (n > 4 ? 4 : n);
    // the stops (a, b) that t lies between; past the last one, b is it
    float4 a, b;
    float lo = off.x, hi = off.y;
    bool past = n == 1;
    if (kUniform) {
        a = c0;
        b = n > 1 ? c1 : c0;
        if (n > 1 && t > off.y) {
            past = n == 2;
            a = c1;
            b = n > 2 ? c2 : c1;
            lo = off.y;
            hi = off.z;
            if (n > 2 && t > off.z) {
                past = n == 3;
                a = c2;
                b = n > 3 ? c3 : c2;
                lo = off.z;
                hi = off.w;
                if (n > 3 && t > off.w) {
                    past = true;
                    b = c3;
                }
            }
        }
        if (!(t > off.x)) return c0;
    } else {
        if (!(t > off.x)) return ld4(g + 48);
        const float o[4] = {off.x, off.y, off.z, off.w};
        int i = 1;
        while (i < n && t > o[i]) ++i;
        past = i == n;
        b = ld4(g + 48 + 16 * (past ? n - 1 : i));
        if (past) return b;
        a = ld4(g + 32 + 16 * i);
        lo = o[i - 1];
        hi = o[i];
    }
    if (past) return b;
    const float span = hi - lo;
    const float f = span > 0.0f ? (t - lo) / span : 0.0f;
    return make_float4(a.x + ((b.x - a.x) * f), a.y + ((b.y - a.y) * f), a.z + ((b.z - a.z) * f),
                       a.w + ((b.w - a.w) * f));
}

// readColor (Kernels.cl:1411-1442): solid colour, picture texel (nearest, as
// the reference samples, or bilinear) or gradient, from the shape's
// substance record `sub`.  A picture at its own scale needs no division.
// kUniform: the wave asks for one substance; four texels inside its picture are
// two reads of a pair, without tests.  Pictures and gradients are 3 in 10 of the
// substances that the 4096^2 frame's colours evaluate; with their records read
// whole by scalar loads it takes 19.0 ms against 20.7.
template <bool kUniform = false>
__device__ __forceinline__ float4 read_color_sub(const SceneDesc &s, uint64_t tag, float4 sub, int ax, int ay)
{
    const uint64_t type = tag & kTagTypeMask;
    if (type == kTagSolid) return sub;
    const uint32_t id = __float_as_uint(sub.x);
    if (type == kTagGradient) return eval_gradient<kUniform>(ro((const uint8_t *)s.grads) + 112 * (size_t)id, ax, ay);
    const GUDNI_CONST PictUse *use = ro(s.uses) + id;
    const PictUse u{use->tx, use->ty, use->w, use->h, use->mem_offset, use->scale};
    float sx = (float)ax, sy = (float)ay;
    if (u.scale != 1.0f) {
        const float scale = u.scale < 0.0000001f ? 0.0000001f : u.scale;
        sx = sx / scale;
        sy = sy / scale;
    }
    sx = sx - u.tx;
    sy = sy - u.ty;
    if (s.filter == 1) {
        const float fx = sx - 0.5f, fy = sy - 0.5f;
        const int ix = f2i_floor(fx), iy = f2i_floor(fy);
        const float wx = fx - (float)ix, wy = fy - (float)iy;
        const uint32_t x0 = (uint32_t)ix, y0 = (uint32_t)iy;
        float4 t0, t1, t2, t3;
        if (kUniform && max(x0, x0 + 1u) < (uint32_t)u.w && max(y0, y0 + 1u) < (uint32_t)u.h) {
            const uint32_t off = (uint32_t)u.mem_offset + 4u * (y0 * (uint32_t)u.w + x0);
            const TexelPair p = *reinterpret_cast<const TexelPair *>(s.pict + off);
            const TexelPair q = *reinterpret_cast<const TexelPair *>(s.pict + (off + 4u * (uint32_t)u.w));
            t0 = unit_bytes(p.left);
            t1 = unit_bytes(p.right);
            t2 = unit_bytes(q.left);
            t3 = unit_bytes(q.right);
        } else {
            t0 = texel(s, u, x0, y0);
            t1 = texel(s, u, x0 + 1u, y0);
            t2 = texel(s, u, x0, y0 + 1u);
            t3 = texel(s, u, x0 + 1u, y0 + 1u);
        }
        const float ax0 = 1.0f - wx, ay0 = 1.0f - wy;
        float4 r;
        r.x = (((t0.x * ax0) + (t1.x * wx)) * ay0) + (((t2.x * ax0) + (t3.x * wx)) * wy);
        r.y = (((t0.y * ax0) + (t1.y * wx)) * ay0) + (((t2.y * ax0) + (t3.y * wx)) * wy);
        r.z = (((t0.z * ax0) + (t1.z * wx)) * ay0) + (((t2.z * ax0) + (t3.z * wx)) * wy);
        r.w = (((t0.w * ax0) + (t1.w * wx)) * ay0) + (((t2.w * ax0) + (t3.w * wx)) * wy);
        return r;
    }
    return texel(s, u, (uint32_t)f2i_rtz(sx), (uint32_t)f2i_rtz(sy));
}

__device__ __forceinline__ float4 read_color(const SceneDesc &s, uint64_t tag, int ax, int ay)
{
    return read_color_sub(s, tag, s.substances[tag & kTagIdMask], ax, ay);
}

// Bits [start, start + q) of the 128-bit set (s1:s0), q <= 32, start < 128;
// bits past 127 read as 0.
__device__ __forceinline__ uint32_t group_bits(uint64_t s0, uint64_t s1, uint32_t start, uint32_t q)
{
    uint64_t v;
    if (start >= 64u) v = s1 >> (start - 64u);
    else if (start == 0u) v = s0;
    else v = (s0 >> start) | (s1 << (64u - start));
    return (uint32_t)v & (q >= 32u ? 0xFFFFFFFFu : ((1u << q) - 1u));
}

__device__ __forceinline__ uint64_t wave_uniform64(uint64_t v)
{
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    return ((uint64_t)hi << 32) | lo;
}

// OR of a word over the wave's 64 lanes (all of them active).
__device__ __forceinline__ uint32_t wave_or(uint32_t v)
{
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true);   // row_shr:1
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, true);   // row_shr:2
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, true);   // row_shr:4
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, true);   // row_shr:8
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, true);   // row_bcast:15
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, true);   // row_bcast:31
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Composite of one group's set shapes (word: this lane's bits, 0 for a lane
// that takes no part), top-down, premultiplied.  Once the alpha is exactly 1
// every later layer adds its colour times 0, so a lane stops there with the
// same result.  The wave walks the shapes some lane holds together, from the
// top: each shape is composited by the lanes that hold it.  A lane meets its
// own shapes in its own order, as a walk of its bits alone would, but the
// wave evaluates one substance at a time, whose record every lane reads alike.
// lookup: the group's pictures and gradients, the only ones whose tags are
// read (the 4096^2 frame 19.0 -> 18.4 ms).  Reading the next shape's colour
// ahead cost 16 bytes of scratch a lane and 2%.  Every lane of the wave calls
// it.
__device__ __forceinline__ float4 group_composite(const SceneDesc &s, const TileTable *tt,
                                                  uint32_t word, uint32_t lookup, int n0, int ax, int ay)
{
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    uint32_t cand = wave_or(word);
    while (cand) {
        if (!__any(word != 0u)) break;
        const int b = 31 - __clz((int)cand);
        cand &= ~(1u << b);
        if ((word >> b) & 1u) {
            word &= ~(1u << b);
            const int n = n0 + b;
            float4 pm = tt->color[n];
            if ((lookup >> b) & 1u) {
                const uint64_t tag = wave_uniform64(tt->tag[n]);
                pm.x = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(pm.x)));
                const float4 c = read_color_sub<true>(s, tag, pm, ax, ay);
                pm = make_float4(c.x * c.w, c.y * c.w, c.z * c.w, c.w);
            }
            const float t = 1.0f - acc.w;
            acc.x = acc.x + pm.x * t;
            acc.y = acc.y + pm.y * t;
            acc.z = acc.z + pm.z * t;
            acc.w = acc.w + pm.w * t;
            if (acc.w == 1.0f) word = 0u;
        }
    }
    return acc;
}

// Accurate-mode colour of a grouped tile under the stack (s0, s1):
// over(group 3 .. group 0, background).  Groups under an alpha of exactly 1
// add nothing (their colour times 0) and are not walked.  Every lane of the
// wave calls it, with valid false where it holds no section.
__device__ __forceinline__ float4 grouped_color(const SceneDesc &s, const TileTable *tt, uint64_t s0, uint64_t s1,
                                                bool valid, int ax, int ay)
{
    const uint32_t q = __builtin_amdgcn_readfirstlane(tt->gq);
    const uint64_t l0 = wave_uniform64(tt->lookup[0]), l1 = wave_uniform64(tt->lookup[1]);
    float P0 = 0.f, P1 = 0.f, P2 = 0.f, A = 0.f;
#pragma unroll 1
    for (int g = 3; g >= 0; --g) {
        const bool open = valid && A != 1.0f;
        const uint32_t word = open ? group_bits(s0, s1, (uint32_t)g * q, q) : 0u;
        const float4 gcol = group_composite(s, tt, word, group_bits(l0, l1, (uint32_t)g * q, q), (int)(g * q), ax, ay);
        if (open) {
            const float t = 1.0f - A;
            P0 = P0 + gcol.x * t;
            P1 = P1 + gcol.y * t;
            P2 = P2 + gcol.z * t;
            A = A + gcol.w * t;
        }
    }
    {
        const float4 pm = make_float4(s.bg[0] * s.bg[3], s.bg[1] * s.bg[3], s.bg[2] * s.bg[3], s.bg[3]);
        const float t = 1.0f - A;
        P0 = P0 + pm.x * t;
        P1 = P1 + pm.y * t;
        P2 = P2 + pm.z * t;
        A = A + pm.w * t;
    }
    if (A > 0.0f) return make_float4(P0 / A, P1 / A, P2 / A, A);
    return make_float4(0.f, 0.f, 0.f, 0.f);
}

// determineColor (Kernels.cl:1447-1513).  kCompact: the stack is labelled by
// tile-local shape index and tags/colours come from the LDS table.
template <bool kCompact>
__device__ float4 determine_color(const Frame &f, const SceneDesc &s, const Stack &st, const int32_t *sidx,
                                  const TileTable *tt, int ax, int ay)
{
    // The walk visits set stack bits from the top (findTop with a falling
    // ignoreAbove, Kernels.cl:281-292): pop the highest bit of a working copy.
    // Bits at or above maxShapes are never set.
    uint64_t w0 = st.s0, w1 = st.s1;
    float4 base = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float4 next = base;      // REFERENCE: colour; ACCURATE: premultiplied colour
    uint64_t last_id = ~0ull;
    bool last_is_continue = true, last_is_set = false;
    const bool ref_mode = f.coverage_mode == GUDNI_COVERAGE_REFERENCE;
    for (;;) {
        bool should_composite = true;
        bool done = false;
        int top_bit;
        if (w1) { top_bit = 127 - __clzll((long long)w1); w1 &= ~(1ull << (top_bit - 64)); }
        else if (w0) { top_bit = 63 - __clzll((long long)w0); w0 &= ~(1ull << top_bit); }
        else top_bit = -1;
        if (top_bit < 0) {
            next = make_float4(s.bg[0], s.bg[1], s.bg[2], s.bg[3]);
            if (!ref_mode) next = make_float4(next.x * next.w, next.y * next.w, next.z * next.w, next.w);
            done = true;
            last_is_set = true;
        } else {
            uint64_t tag;
            if (kCompact) tag = tt->tag[top_bit];
            else tag = s.shapes[sidx[top_bit * kWave]].tag;
            const uint64_t sid = tag & kTagIdMask;
            const bool is_cont = (tag & kTagCompoundMask) == kTagContinue;
            const bool is_add = (tag & kTagCompoundMask) == kTagAdd;
            if (sid == last_id) {
                if (last_is_continue) {
                    if (!is_cont) { last_is_set = is_add; last_is_continue = false; }
                    else last_is_set = !last_is_set;
                }
                should_composite = false;
            } else {
                const bool solid = (tag & kTagTypeMask) == kTagSolid;
                if (kCompact && solid) {
                    next = tt->color[top_bit];          // already in the mode's form
                } else {
                    if (kCompact) next = read_color_sub(s, tag, tt->color[top_bit], ax, ay);
                    else next = read_color(s, tag, ax, ay);
                    if (!ref_mode)
                        next = make_float4(next.x * next.w, next.y * next.w, next.z * next.w, next.w);
                }
                last_is_set = is_add || is_cont;
            }
            last_id = sid;
        }
        if (should_composite && last_is_set) {
            if (ref_mode) {
                base = composite(base, next);
            } else {
                // premultiplied: base.xyz = P, base.w = A; the alpha update is
                // the reference's alphaOut expression, so A == 1 terminates at
                // the same shape
                const float t = 1.0f - base.w;
                base.x = base.x + next.x * t;
                base.y = base.y + next.y * t;
                base.z = base.z + next.z * t;
                base.w = base.w + next.w * t;
            }
            if (base.w == 1.0f) done = true;
        }
        if (done) break;
    }
    if (!ref_mode) {
        if (base.w > 0.0f) {
            base.x = base.x / base.w;
            base.y = base.y / base.w;
            base.z = base.z / base.w;
        } else {
            base = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    }
    return base;
}

__device__ __forceinline__ uint32_t pixel_word(float4 c, bool rgba)
{   // colorToSolidPixel_Word32_BGRA (Kernels.cl:842-844): rtz, alpha 255; the
    // same bytes in R,G,B,A memory order when `rgba`
    const float ch[3] = {c.z * 255.0f, c.y * 255.0f, c.x * 255.0f};
    uint32_t w = 0xFF000000u;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float v = ch[i];
        const uint32_t u = (v == v) ? (v >= 255.0f ? 255u : (v <= 0.0f ? 0u : (uint32_t)v)) : 0u;
        w |= u << (8 * (rgba ? 2 - i : i));
    }
    return w;
}

__device__ __forceinline__ void write_pixel(const Frame &f, const SceneDesc &s, int x, int y, float4 color)
{
    const long long pix = (long long)y * s.width + x;
    s.out[pix] = pixel_word(color, f.out_rgba != 0);
    if (s.out_f32) s.out_f32[pix] = color;
}

// The colours of the `count` listed sections, a section a lane, whichever
// lanes swept them; then every sweeping lane adds its sections' colour x area
// in their order (head: its first), and the pixels that ended are written
// (writePixelGlobal, Kernels.cl:1853-1862: the area-weighted mean).
template <bool kCompact>
__device__ __forceinline__ void color_sections(const Frame &f, const SceneDesc &s, const Column &c,
                                               const int32_t *sidx, TileTable *tt, bool grouped, int lane, int count,
                                               uint32_t head, float4 &acc, float &area_sum)
{
    SectionList &L = tt->sec;
    wave_sync();
    for (int e0 = 0; e0 < count; e0 += kWave) {
        const int e = e0 + lane;
        const bool valid = e < count;
        const uint32_t info = valid ? L.info[e] : 0u;
        const float4 bits = L.val[valid ? e : 0];
        const int owner = (int)(info & 63u);
        const int ax = __shfl(c.dx, owner), ay = __shfl(c.dy, owner) + (int)((info >> 6) & 0x1FFFu);
        const uint64_t s0 = ((uint64_t)__float_as_uint(bits.y) << 32) | __float_as_uint(bits.x);
        const uint64_t s1 = ((uint64_t)__float_as_uint(bits.w) << 32) | __float_as_uint(bits.z);
        float4 col;
        if (grouped) {
            col = grouped_color(s, tt, s0, s1, valid, ax, ay);
        } else {
            if (valid) col = determine_color<kCompact>(f, s, Stack{s0, s1}, sidx - lane + owner, tt, ax, ay);
        }
        if (valid) {
            const float adj = L.adj[e];
            L.val[e] = make_float4(col.x * adj, col.y * adj, col.z * adj, col.w * adj);
        }
    }
    wave_sync();
    for (uint32_t e = head; e != kSecNone;) {
        const float4 v = L.val[e];
        const uint32_t info = L.info[e];
        acc.x += v.x;
        acc.y += v.y;
        acc.z += v.z;
        acc.w += v.w;
        area_sum += L.adj[e];
        if (info & kSecEnd) {
            L.val[e] = acc;
            L.adj[e] = area_sum;
            acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            area_sum = 0.0f;
        }
        e = info >> 24;
    }
    wave_sync();
    for (int e0 = 0; e0 < count; e0 += kWave) {
        const int e = e0 + lane;
        const uint32_t info = e < count ? L.info[e] : 0u;
        const int owner = (int)(info & 63u);
        const int ax = __shfl(c.dx, owner), ay = __shfl(c.dy, owner) + (int)((info >> 6) & 0x1FFFu);
        if (info & kSecEnd) {
            const float4 a = L.val[e];
            const float w = L.adj[e];
            write_pixel(f, s, ax, ay, make_float4(a.x / w, a.y / w, a.z / w, a.w / w));
        }
    }
    wave_sync();
}

// renderThresholdArray + calculatePixel + horizontalAdvance + sectionColor
// (Kernels.cl:1724-1742, 1826-1851, 1881-1916, 1978-2028).  The reference
// loops over a column's pixels and, inside, over each pixel's sections; here
// one loop steps a section of every lane that has one left, whatever its
// pixel, so lanes only wait for each other at the end of their columns (the
// 4096^2 frame: 57.4 -> 51.9 ms).
// The loop only sweeps: it appends each section, its area and the stack it
// lies under to a list in LDS, and when 192 are listed the whole wave gives
// them their colours, a section a lane (color_sections).  A step of the sweep
// has ~21 of 64 lanes in a section; colouring them there kept the colour
// walks, half of the frame's vector instructions, at that occupancy, and a
// lone busy column waited for each of its colours.  The 4096^2 frame went
// from 43.5 to 35.2 ms (1.34e10 vector instructions against 1.75e10) and an
// 800x600 frame of 256-px tiles, 250 waves in all, from 45 to 27.  A list of
// 171 entries took 35.6 ms; of the frame's 176e9 wave cycles then left (20.7
// ms) colours took 89e9, span starts 33e9, other steps 37e9, generation 36e9.
// A section costs little beside the start of a span (vertical_advance), so
// lanes take sections at their own pace within a span but start spans
// together: on the 4096^2 frame a wave then starts spans half as often, for 24
// lanes instead of 9.  With the active records read once at their start
// (open_span) the frame takes 23.3 ms against 33.4; waiting for 1/8, 1/4, 1/2
// and 3/4 of the lanes only took 28.3, 27.2, 25.3 and 24.2.
// Every lane of the wave calls it; ok: the lane has a column to sweep.
template <bool kCompact>
__device__ __forceinline__ uint32_t render(const Frame &f, const SceneDesc &s, Queue &q, const Column &c, Stack st,
                           int32_t *sidx, TileTable *tt, bool nz, bool ok)
{
    int32_t *const wind = sidx + kWindOffset * kWave;
    SectionList &L = tt->sec;
    Sweep p;
    p.current = 0;
    p.left0 = st.s0; p.left1 = st.s1;
    p.active_bottom = 0.0f;
    p.below0 = p.below1 = 0;
    p.sx0 = 0.0f; p.sy0 = 0.0f; p.sx1 = 1.0f; p.sy1 = 0.0f;
    const bool stochastic = f.stochastic != 0.0f;
    p.rnd = 0;
    if (stochastic && ok) {   // initRandomField (Kernels.cl:1597-1606)
        const uint32_t start = c.unique & (uint32_t)f.random_mask;
        p.rnd = __float_as_uint(f.random[start]) & (uint32_t)f.random_mask;
    }
    uint32_t status = 0;
    int guard = (int)kSectionGuard;
    uint32_t row = 0;
    const int lane = threadIdx.x & (kWave - 1);
    const bool grouped = kCompact && __builtin_amdgcn_readfirstlane((uint32_t)tt->grouped) != 0u;
    p.pixel_y = 1.0f;
    bool alive = ok && p.pixel_y <= c.float_height;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float area_sum = 0.0f;
    int count = 0;                              // listed sections (wave-uniform)
    uint32_t head = kSecNone, last = kSecNone;  // this lane's first and last
    for (;;) {
        const bool running = __any(alive);
        bool have = false, end = false;
        float adj = 0.0f;
        uint64_t s0 = 0, s1 = 0;
        const uint32_t at_row = row;
        // lanes whose section reached the right border wait for the others
        // to get there, and all start their next spans together
        const bool advance = !__any(alive && p.sx1 != 1.0f);
        if (alive && (advance || p.sx1 != 1.0f)) {
            bool done = !((p.sx1 < 1.0f) || (p.sy1 < p.pixel_y));
            if (done) {
                // a pixel without sections (its records hold NaN): 0 / 0
                const float nan = __int_as_float(0x7FC00000);
                write_pixel(f, s, c.dx, c.dy + (int)row, make_float4(nan, nan, nan, nan));
            } else if (--guard < 0) {
                status = kStatusGuard;
                alive = false;
            } else {
                if (p.sx1 == 1.0f) vertical_advance(q, c, p, st, wind, nz);
                if (q.spilled || q.overflow) {
                    alive = false;
                } else {
                    // horizontalAdvance with thresholdMidXLow (Kernels.cl:916-926)
                    float nx = 1.0f;
                    uint32_t h = 0;
                    const bool crossing = p.current < q.n_active;
                    if (crossing) {
                        const Thr t = q.active(p.current);
                        h = q.active_h(p.current);
                        float x;
                        if (f.coverage_mode == GUDNI_COVERAGE_REFERENCE) {
                            const float ymid = p.sy0 + ((p.sy1 - p.sy0) * 0.5f);
                            x = intersect_x(h, t, ymid);
                        } else if (t.left == t.right) {
                            x = t.left;
                        } else {
                            // the same mid point, relative to the threshold's start
                            const float sy = hdr_pos(h) ? t.top : t.bottom;
                            const float d = (p.sy0 - sy) + ((p.sy1 - p.sy0) * 0.5f);
                            x = (d * inv_slope(h, t)) + t.left;
                        }
                        nx = (x >= 1.0f) ? 0.0f : cl_max(0.0f, x);
                    }
                    p.sx0 = p.sx1;
                    p.sx1 = nx;
                    const float area = (p.sx1 - p.sx0) * (p.sy1 - p.sy0);
                    adj = area;
                    if (stochastic) {   // getRandom (Kernels.cl:1608-1613)
                        p.rnd = (p.rnd + 1u) & (uint32_t)f.random_mask;
                        adj = area + (area * f.random[p.rnd] * f.stochastic);
                    }
                    have = true;
                    s0 = st.s0;
                    s1 = st.s1;
                    if (crossing) st.cross<kCrossRight>(h, wind, nz);
                    ++p.current;
                    done = end = !((p.sx1 < 1.0f) || (p.sy1 < p.pixel_y));
                }
            }
            if (done) {   // the next pixel
                p.sx0 = 0.0f;
                p.sy0 = p.pixel_y;
                ++row;
                p.pixel_y += 1.0f;
                alive = p.pixel_y <= c.float_height;
            }
        }
        const uint64_t mask = __ballot(have);
        const int n = __popcll(mask);
        if (count + n > kSections || !running) {
            color_sections<kCompact>(f, s, c, sidx, tt, grouped, lane, count, head, acc, area_sum);
            count = 0;
            head = last = kSecNone;
            if (!running) break;
        }
        if (have) {
            const uint32_t e = (uint32_t)count + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                                           __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
            L.val[e] = make_float4(__uint_as_float((uint32_t)s0), __uint_as_float((uint32_t)(s0 >> 32)),
                                   __uint_as_float((uint32_t)s1), __uint_as_float((uint32_t)(s1 >> 32)));
            L.adj[e] = adj;
            L.info[e] = (uint32_t)lane | (at_row << 6) | (end ? kSecEnd : 0u) | (kSecNone << 24);
            if (last == kSecNone) head = e;
            else reinterpret_cast<uint8_t *>(&L.info[last])[3] = (uint8_t)e;
            last = e;
        }
        count += n;
    }
    return status;
}

// initTileState / isActiveThread (Kernels.cl:1692-1722)
__device__ __forceinline__ bool init_column(const Frame &f, const SceneDesc &s, const TileRec &t, int job, int column,
                                            Column &c)
{
    const int hd = t.hdepth, vd = t.vdepth, cd = f.compute_depth;
    const int dd = max(0, vd - (cd - hd));
    const int ix = ((1 << hd) - 1) & column;
    const int iy = (column >> hd) << dd;
    c.dx = ix + t.box[0];
    c.dy = iy + t.box[1];
    c.unique = ((uint32_t)t.column_allocation + (1u << cd) + (uint32_t)job * (1u << (2 * cd))) * 7919u;
    c.int_height = min(1 << dd, s.height - c.dy);
    c.float_height = (float)c.int_height;
    c.shape_start = t.shape_start;
    c.num_shapes = t.shape_count;
    return (iy < t.box[3] - t.box[1]) && (c.dx < s.width) && (c.dy < s.height);
}

__device__ __forceinline__ uint32_t wave_uniform(uint32_t v)
{
    return __builtin_amdgcn_readfirstlane(v);
}

// Number of contributing shapes with tile-local index below n: the
// reference's shape bit of shape n in a compact tile.
__device__ __forceinline__ uint32_t bit_of(uint64_t c0, uint64_t c1, uint32_t n)
{
    if (n < 64u) return (uint32_t)__popcll(c0 & ((1ull << n) - 1ull));
    return (uint32_t)(__popcll(c0) + __popcll(c1 & ((1ull << (n - 64u)) - 1ull)));
}

__device__ __forceinline__ uint32_t relabel(uint32_t h, uint64_t c0, uint64_t c1)
{
    return (h & ~kShapeBitMask) | bit_of(c0, c1, h & kShapeBitMask);
}

// Copy the queue into the dump buffers, in the reference's labels.
template <bool kCompact>
__device__ void dump_queue(const Frame &f, const Queue &q, int dslot, bool pre, uint64_t c0,
                           uint64_t c1)
{
    const int k = min(q.len, f.dump_cap);
    float4 *thr = pre ? f.dump_pre_thr : f.dump_thr;
    uint32_t *hdr = pre ? f.dump_pre_hdr : f.dump_hdr;
    for (int i = 0; i < k; ++i) {
        const Thr x = q.get(i);
        const uint32_t h = q.get_h(i);
        thr[(size_t)dslot * f.dump_cap + i] = make_float4(x.top, x.bottom, x.left, x.right);
        hdr[(size_t)dslot * f.dump_cap + i] = kCompact ? relabel(h, c0, c1) : h;
    }
}

// One work unit: 64 columns of one tile, generate -> sort -> render per lane,
// with wave-uniform boundaries between the stages so the optional stage
// clocks bracket whole stages of the wave.
template <bool kCompact>
__device__ __forceinline__ void run_unit(const Frame &f, const SceneDesc &s, int lane, uint32_t unit, int part, Queue &q, int32_t *sidx,
                         TileTable *tt, uint32_t &status)
{
    const int tile = (int)(unit >> 2), quarter = (int)(unit & 3u);
    const TileRec t = f.tiles[tile];
    const int job = f.tile_job ? f.tile_job[tile] : 0;
    const int column = unit_column(t.hdepth, f.compute_depth, quarter, lane);
    Column c;
    const bool mine = (lane >> (6 - f.split)) == part;   // a lane of this wave's part of the unit
    const bool active = init_column(f, s, t, job, column, c) && mine;
    const int dslot = tile * f.threads_per_tile + column;
    const bool timed = f.stage_cycles != nullptr;
    const long long t0 = timed ? clock64() : 0;
    if (kCompact) {
        // the tile's tags and solid colours, by tile-local index
        const bool premultiply = f.coverage_mode != GUDNI_COVERAGE_REFERENCE;
        bool all_add = true;
        for (int n = lane; n < c.num_shapes; n += kWave) {
            const uint64_t tag = s.shapes[c.shape_start + n].tag;
            tt->tag[n] = tag;
            float4 col = s.substances[tag & kTagIdMask];
            if ((tag & kTagTypeMask) == kTagSolid && premultiply)
                col = make_float4(col.x * col.w, col.y * col.w, col.z * col.w, col.w);
            tt->color[n] = col;
            all_add = all_add && (tag & kTagCompoundMask) == kTagAdd;
            const uint64_t lookup = __ballot((tag & kTagTypeMask) != kTagSolid);
            if (lane == 0) tt->lookup[n >> 6] = lookup;
        }
        wave_sync();
        // grouped colours need every shape added with its own substance
        bool distinct = true;
        for (int n = lane; n < c.num_shapes; n += kWave) {
            const uint64_t sid = tt->tag[n] & kTagIdMask;
            for (int m = n + 1; m < c.num_shapes && distinct; ++m)
                distinct = (tt->tag[m] & kTagIdMask) != sid;
        }
        const bool grouped_tile = premultiply && __all(all_add && distinct);
        if (lane == 0) {
            tt->grouped = grouped_tile ? 1 : 0;
            const uint32_t gq = c.num_shapes > 4 ? (uint32_t)(c.num_shapes + 3) / 4u : 1u;
            tt->gq = gq;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    uint32_t bits = 0;
    uint64_t s0 = 0, s1 = 0, c0 = 0, c1 = 0;
    bool any_nonzero = false;
    {
        // x extent of this unit's columns (isActiveThread's internalX)
        int x0 = t.box[0] + unit_x0(t.hdepth, f.compute_depth, quarter);
        const int uw = unit_width(t.hdepth, f.compute_depth), lanes = kWave >> f.split;
        if (lanes < uw) x0 += (part * lanes) & (uw - 1);
        const int x1 = x0 + min(uw, lanes);
        generate<kCompact>(f, s, q, c, active, lane, (float)x0 - 1.0f, (float)x1 + 1.0f, sidx, tt,
                           columns_log2(x1 - x0), bits,
                           s0, s1, c0, c1, any_nonzero);
    }
    const bool ok = active && !q.spilled && !q.overflow;
    const long long t1 = timed ? clock64() : 0;
    if (ok && f.dump_qlen) dump_queue<kCompact>(f, q, dslot, true, c0, c1);
    if (ok) radix_sort_queue(q, tt->hist + lane, s.sort_bits,
                             c.float_height);
    if (ok && f.dump_qlen) {
        dump_queue<kCompact>(f, q, dslot, false, c0, c1);
        f.dump_qlen[dslot] = q.len;
        f.dump_bits[dslot] = bits;
        uint64_t r0 = s0, r1 = s1;
        if (kCompact) {     // the initial stack in the reference's labels
            r0 = r1 = 0;
            for (uint32_t n = 0; n < 128u; ++n) {
                const bool on = n < 64u ? ((s0 >> n) & 1ull) : ((s1 >> (n - 64u)) & 1ull);
                if (on) {
                    const uint32_t b = bit_of(c0, c1, n);
                    if (b < 64u) r0 |= 1ull << b; else r1 |= 1ull << (b - 64u);
                }
            }
        }
        f.dump_stack[2 * (size_t)dslot] = r0;
        f.dump_stack[2 * (size_t)dslot + 1] = r1;
        int b = 0;
        for (int i = 0; i < f.max_shapes; ++i) f.dump_sidx[(size_t)dslot * f.max_shapes + i] = 0;
        if (kCompact) {
            for (int n = 0; n < 128; ++n) {
                const bool on = n < 64 ? ((c0 >> n) & 1ull) : ((c1 >> (n - 64)) & 1ull);
                if (on && b < f.max_shapes) f.dump_sidx[(size_t)dslot * f.max_shapes + b++] = c.shape_start + n;
            }
        } else {
            for (int i = 0; i < (int)bits && i < f.max_shapes; ++i)
                f.dump_sidx[(size_t)dslot * f.max_shapes + i] = sidx[i * kWave];
        }
    }
    const long long t2 = timed ? clock64() : 0;
    // only a lane that walked a nonzero-fill shape keeps winding counters
    status = render<kCompact>(f, s, q, c, Stack{s0, s1}, sidx, tt, any_nonzero, ok);
    if (active && q.overflow) status |= kStatusOverflow;
    if (mine && !active && f.dump_qlen) f.dump_qlen[dslot] = -1;
    if (timed) {
        const long long t3 = clock64();
        if (lane == 0) {
            atomicAdd(f.stage_cycles + 0, (unsigned long long)(t1 - t0));
            atomicAdd(f.stage_cycles + 1, (unsigned long long)(t2 - t1));
            atomicAdd(f.stage_cycles + 2, (unsigned long long)(t3 - t2));
            atomicAdd(f.stage_cycles + 3, 1ull);   // parts; units once read (gudni_frame_check)
        }
    }
}

} // namespace dev
} // namespace gudni
