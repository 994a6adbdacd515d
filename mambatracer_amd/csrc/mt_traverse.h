// Per-ray BVH traversal (device code) shared by the traversal entry points
// (mt_trace.hip) and the bounce loop's fused kernels (mt_render.hip):
// intersectMesh / testOcclusion (src/cl/kernel/NormalBVH.cl:14-92,
// 235-317) over the reference arrays and over the packed layout, in the
// reference's visiting order (see mt_trace.hip for the layouts).
#pragma once
#include "mt_devmath.h"
#include "mt_internal.h"

namespace {

struct RayT {
    v3 o, d, inv;
    int sx, sy, sz;
    float tmin, tmax;
};

__device__ __forceinline__ void ray_init(RayT& r, float4 a, float4 b)
{ // initGlobalRay, Util.cl:577-600
    r.o = mk3(a.x, a.y, a.z);
    r.d = mk3(b.x, b.y, b.z);
    r.inv = mk3(1.0f / b.x, 1.0f / b.y, 1.0f / b.z);
    r.sx = r.inv.x < 0.0f;
    r.sy = r.inv.y < 0.0f;
    r.sz = r.inv.z < 0.0f;
    r.tmin = a.w;
    r.tmax = b.w;
}

// intersectBoundT, Util.cl:707-732.  Conditional assignments (not fminf/fmaxf)
// keep the reference's NaN behaviour.  The reference's two early returns
// become terms of one conjunction (all six slab distances are computed
// either way), so the test has no branches: a wave's lanes never split
// inside it, and the node's loads all issue before the first compare.
__device__ __forceinline__ bool box_hit(const RayT& r, float mnx, float mny, float mnz,
                                        float mxx, float mxy, float mxz, float& tnear)
{
    const float tmin = ((r.sx ? mxx : mnx) - r.o.x) * r.inv.x;
    const float tmax = ((r.sx ? mnx : mxx) - r.o.x) * r.inv.x;
    const float tymin = ((r.sy ? mxy : mny) - r.o.y) * r.inv.y;
    const float tymax = ((r.sy ? mny : mxy) - r.o.y) * r.inv.y;
    const float tzmin = ((r.sz ? mxz : mnz) - r.o.z) * r.inv.z;
    const float tzmax = ((r.sz ? mnz : mxz) - r.o.z) * r.inv.z;
    const bool xy = !((tmin > tymax) | (tymin > tmax));
    const float t1 = tymin > tmin ? tymin : tmin;
    const float u1 = tymax < tmax ? tymax : tmax;
    const bool xyz = !((t1 > tzmax) | (tzmin > u1));
    const float t2 = tzmin > t1 ? tzmin : t1;
    const float u2 = (tzmax < u1 ? tzmax : u1) * 1.00000024f;
    tnear = t2;
    return xy & xyz & (t2 < r.tmax) & (u2 > r.tmin);
}

// fastTriangleIntersection, Primitive.cl:3-29, on p1 and the two edges.
// Both early returns of the reference give tMax; here every quantity is
// computed and one select picks t or tMax, so p1 is fetched with the edges
// instead of after the determinant test.
__device__ __forceinline__ float tri_hit(const RayT& r, v3 p1, v3 e1, v3 e2)
{
    const v3 h = cross3(r.d, e2);
    const float a = dot3(e1, h);
    // :13 compares a with the double 0.0000001; 0x33d6bf94 (9.9999994e-8) is
    // the largest float below it, so in floats the test is |a| <= that
    const bool parallel = fabsf(a) <= __int_as_float(0x33d6bf94);
    const float f = 1.0f / a;
    const v3 s = sub3(r.o, p1);
    const float b1 = f * dot3(s, h);
    const v3 q = cross3(s, e1);
    const float b2 = f * dot3(r.d, q);
    const float t = f * dot3(e2, q);
    const bool out = (b1 < 0.0f) | (b1 > 1.0f) | (b2 < 0.0f) | (b1 + b2 > 1.0f) | (t < 0.0f) | (t > r.tmax);
    return (parallel | out) ? r.tmax : t;
}

struct BitStack {
    uint64_t lo, hi;
    __device__ __forceinline__ void push0()
    {
        hi = (hi << 1) | (lo >> 63);
        lo <<= 1;
    }
    __device__ __forceinline__ void pop()
    {
        lo = (lo >> 1) | (hi << 63);
        hi >>= 1;
    }
    __device__ __forceinline__ bool empty() const { return (lo | hi) == 0; }
    // zero bits above the lowest set bit (the pops the reference performs)
    __device__ __forceinline__ int ctz() const
    {
        return lo ? __builtin_ctzll(lo) : 64 + __builtin_ctzll(hi);
    }
    __device__ __forceinline__ void shr(int z)
    {
        if (z == 0) return;
        if (z < 64) {
            lo = (lo >> z) | (hi << (64 - z));
            hi >>= z;
        } else {
            lo = hi >> (z - 64);
            hi = 0;
        }
    }
};

// Short stack of postponed far children, newest first.  Each 1 bit of the
// bitstack is a both-children-hit decision whose far child is still to be
// visited; the stack holds the most recent MT_SHORT_STACK of them.  Reaching
// the next pending far child then costs no memory access: the reference's
// pops (walking parent links up to the lowest 1 bit) are counted as
// ctz(bitstack) without being fetched.  When older entries have been
// dropped, the parent walk finds them exactly as the reference does, reading
// parent and sibling links from the current node's record (an interior
// record's last word pair, a leaf triangle's spare words), so no links are
// carried in registers while descending.  Depth N is a trade: each push
// and pop moves N registers, and a deeper stack saves parent walks on deep
// trees.
#ifndef MT_SHORT_STACK
#define MT_SHORT_STACK 8
#endif
template <int N>
struct ShortStackN {
    int ref[N];
    int n;
    __device__ __forceinline__ void push(int r)
    {
#pragma unroll
        for (int k = N - 1; k > 0; k--) ref[k] = ref[k - 1];
        ref[0] = r;
        n = n < N ? n + 1 : N;
    }
    __device__ __forceinline__ int pop()
    {
        const int r = ref[0];
#pragma unroll
        for (int k = 0; k < N - 1; k++) ref[k] = ref[k + 1];
        n--;
        return r;
    }
};
using ShortStack = ShortStackN<MT_SHORT_STACK>;

// -------------------------------------------------------------------------
// Reference layout: NormalBVH.cl:14-92 over nodes[7], bounds[8], faces[10].
// -------------------------------------------------------------------------
template <bool ANY, bool STATS>
__device__ __forceinline__ int trace_reference(const int* __restrict__ nodes,
                                               const float* __restrict__ bounds,
                                               const int* __restrict__ faces,
                                               const float4* __restrict__ points, RayT& r,
                                               int& child, int* st)
{
    int hit = 0;
    int node_id = 0;
    BitStack bs{0, 0};
    int parent_id = 0, sibling_id = 0;
    for (;;) {
        while (!nodes[7 * node_id + 5]) {
            const int* n = nodes + 7 * node_id;
            parent_id = n[4];
            sibling_id = n[1];
            int left = n[2], right = n[3];
            const float* lb = bounds + 8 * nodes[7 * left];
            const float* rb = bounds + 8 * nodes[7 * right];
            float lt, rt;
            bool lh = box_hit(r, lb[0], lb[1], lb[2], lb[4], lb[5], lb[6], lt);
            bool rh = box_hit(r, rb[0], rb[1], rb[2], rb[4], rb[5], rb[6], rt);
            if (STATS) st[0]++;
            if (!lh && !rh) break;
            bs.push0();
            if (lh && rh) {
                node_id = (rt < lt) ? right : left;
                bs.lo |= 1;
            } else {
                node_id = lh ? left : right;
            }
        }
        if (nodes[7 * node_id + 5]) {
            const int* n = nodes + 7 * node_id;
            if (STATS) st[1]++;
            int c = n[6];
            const int* F = faces + 10 * c;
            v3 p1 = xyz(points[F[0]]);
            v3 p2 = xyz(points[F[1]]);
            v3 p3 = xyz(points[F[2]]);
            float t = tri_hit(r, p1, sub3(p2, p1), sub3(p3, p1));
            if ((r.tmin < t) && (t < r.tmax)) {
                if (ANY) return 1;
                hit = 1;
                r.tmax = t;
                child = c;
            }
            parent_id = n[4];
            sibling_id = n[1];
        }
        while ((bs.lo & 1) == 0) {
            if (bs.empty()) return hit;
            node_id = parent_id;
            const int* n = nodes + 7 * node_id;
            parent_id = n[4];
            sibling_id = n[1];
            bs.pop();
            if (STATS) st[2]++;
        }
        node_id = sibling_id;
        bs.lo ^= 1;
    }
}

// -------------------------------------------------------------------------
// Packed layout, same visiting order.  cur >= 0: interior node record;
// cur < 0: leaf ~rank.  parent/sib track the current node's links, which the
// reference reads from the node records (leaves are not records here).
// -------------------------------------------------------------------------
// Parent and sibling references of node `cur`: an interior record's last
// word pair, or the spare words of a leaf's triangle record.
__device__ __forceinline__ int2 node_links(const float4* __restrict__ pn, const float4* __restrict__ pt, int cur)
{
    const float4 w = cur >= 0 ? pn[4 * (size_t)cur + 3] : pt[3 * (size_t)(~cur) + 2];
    return make_int2(__float_as_int(w.z), __float_as_int(w.w));
}

// The reference's backtracking (NormalBVH.cl:80-90): climb parent links
// while the lowest bitstack bit is 0, then cross to the sibling and flip the
// bit.  Returns false when the bitstack empties (the ray is finished).
template <bool STATS>
__device__ __forceinline__ bool parent_walk(const float4* __restrict__ pn, const float4* __restrict__ pt, int& cur,
                                            BitStack& bs, int* st)
{
    int2 l = node_links(pn, pt, cur); // (parent, sibling) of cur
    while ((bs.lo & 1) == 0) {
        if (bs.empty()) return false;
        cur = l.x;
        l = node_links(pn, pt, cur);
        bs.pop();
        if (STATS) st[2]++;
    }
    cur = l.y;
    bs.lo ^= 1;
    return true;
}

// Work-groups go to the 8 XCDs in turn (group b on XCD b mod 8), each XCD
// with its own L2.  Where neighbouring work-groups trace rays that walk the
// same subtrees, renumbering the groups so that each XCD takes runs of
// neighbouring work keeps each L2 on its own region's nodes instead of all
// eight caching the same ones, while the XCDs taking the runs in turn keeps
// work that varies across the range balanced between them.
//
// Runs of `chunk` consecutive numbers per XCD (XCD x takes runs x, x + 8,
// x + 16, ...); groups past the last whole round of 8 runs keep their own
// number.  A bijection of [0, groups).
__device__ __forceinline__ unsigned xcd_chunked_group(unsigned b, unsigned groups, unsigned chunk)
{
    const unsigned round = 8u * chunk;
    if (b >= (groups / round) * round) return b;
    const unsigned x = b & 7u, k = b >> 3;
    return ((k / chunk) * 8u + x) * chunk + k % chunk;
}

// Run length of the renumbered kernels (camera rays: 16K paths, a compact
// patch of pixels; binned order: 128K rays, 64 neighbouring origin cells of
// a uniform batch).  Measured: a 1920x1080 x 16 spp render of 1M triangles
// 9.69 -> 9.63 ms with the camera traversal renumbered (runs of 256 or
// 1024: the same); 64M random rays through 4M triangles,
// closest / any hit with the sorted order renumbered 48.4 / 34.0 -> 47.6 /
// 33.1 ms (runs of 16: 47.8 / 33.1; 32: 47.5 / 33.0; 256 or contiguous
// eighths of the order: 48.2 / 33.4-33.6).
constexpr unsigned XCD_RUN = 64;

// Work-group number v of a sweep over a segmented queue: group v takes
// segment v mod nseg from chunk v / nseg (the grid a multiple of nseg).  The
// bounce loop's shading appends work-group b's paths to segment b mod 1024,
// so consecutive segments hold neighbouring pixel blocks; runs of XCD_RUN
// consecutive numbers per XCD keep each XCD's L2 on the nodes of a compact
// stretch of the image (the traversal sweeps: the 1080p x 16 spp render
// 9.56 -> 9.49 ms; the shading sweeps, which read per-path state rather than nodes,
// lost 0.4% with it and keep v = b), and with 1024 segments every group of
// one segment runs on the same XCD.
__device__ __forceinline__ unsigned seg_sweep_group()
{
    return xcd_chunked_group(blockIdx.x, gridDim.x, XCD_RUN);
}

// ---------------------------------------------------------------------------
// Wave traversal: one ray per lane of a wave, every ray in the reference's
// visiting order (the packed layout of trace_packed below).
//
// What bounds it on gfx950: the vector memory path and vector issue between
// them, with latency in the gaps; neither is full by itself.  Per wave64
// instruction and SIMD, f32 add / mul / FMA, moves, integer add and logic take
// 2.1-2.4 cycles; compares, selects, min / max (also of three), DPP, shift-adds
// and whatever reads a scalar register 4.1, unless they alternate with the
// first kind (max + add: 4.2 the pair).  The L1 looks one 64-byte piece up per
// cycle, and four 16-byte loads of a node by lanes that hold different nodes
// are four pieces per lane.  Measured per CU: camera rays (direct) 3.9 cycles
// per VALU instruction and SIMD, 0.81 pieces per cycle, the data return busy
// 0.86 of the time; bounces (staged) 7.5, 0.46, 0.89 and LDS 0.21 (0.09 of it
// bank conflicts); a sorted random batch (staged, deep) 6.3, 0.55, 0.93, 0.22.
// So:
//  * a lane's pending subtrees are a plain stack of references in LDS (one
//    write and one read per step, both unconditional) instead of a register
//    queue moved on every push and pop and a 128-bit bitstack; entries past
//    the LDS rows go to scratch memory, which only deep trees reach;
//  * a step has no branches: lanes without an interior node run along and
//    keep their state by selects;
//  * the slab test is max3 / min3 (20 instead of 30 instructions per box)
//    wherever no NaN can arise, intersectBoundT's chain otherwise (slab);
//  * leaves wait until a quarter of the wave's rays are at one, or done
//    (tried: an eighth to a half), so the triangle test runs for many lanes
//    instead of interrupting the walk for one or two;
//  * lanes whose ray has ended take the next of the wave's run together.
// Node records reach the lanes in one of two ways (WaveForm):
//  * direct: each lane loads its own record (four loads); near and far planes
//    picked by selects.  8 waves per SIMD.  Best where neighbouring lanes hold the
//    same node (camera rays, shadow rays) or rays are short.
//  * staged: the four lanes of a quad load each of their four records
//    together, 16 bytes per lane, straight into LDS
//    (global_load_lds_dwordx4), so a record is one L1 piece instead of
//    four; every lane then reads its near and its far planes from LDS with
//    addresses that hold its ray's signs, so nothing is selected.  LDS limits it to 6 waves
//    per SIMD, 5 with a deeper stack.  Best on incoherent rays with long walks.
// Measured, start of this design (register queue and bitstack, leaf tests
// mixed into every step) against now: closest hit of 16M random rays sorted by
// origin through 4M triangles 12.9 -> 8.6 ms (staged; VALU instructions
// 8.9 -> 3.6 G, active lanes 25 -> 46 of 64, L1 pieces 6.2 -> 2.7 G);
// 1920x1080 x 16 spp camera rays through 1M triangles 1.34 -> 1.24 ms (direct;
// staged 1.54), the 16M shadow rays of its first hits 1.65 -> 1.44 ms (direct;
// staged 1.81); first bounce of 993K rays in a soup of 150K triangles
// 0.98 -> 0.61 ms (staged; direct 0.65).
// ---------------------------------------------------------------------------
constexpr int WT_NONE = (int)0x80000000; // no node (never a leaf reference: ranks stay below 2^30)
constexpr int WT_SLOT = 1040;            // bytes between a wave's four load slots: 16 past 1024, so
                                         // that a quad's records lie in different LDS banks
constexpr int WT_REFILL = 16;            // idle lanes a wave waits for before starting new rays
constexpr int WT_REFILL_ANY = 32;        // the same for shadow rays, whose end costs more (any of 16 .. 48: within 1%)
constexpr int WT_REFILL_CAMERA = 64;     // camera rays start and end together; making one costs ~200 instructions
constexpr int WT_OVF = 128;              // stack entries in scratch memory: trees are at most 128 deep, a pending
                                         // subtree per level at most
constexpr int WT_MIN_RUN = 16;           // rays per wave, at least, and
constexpr int WT_MAX_RUN = 256;          //   at most while that fills the GPU's wave slots
constexpr int WT_BINNED_RUN = 512;       // rays per wave of a sorted batch: neighbours share nodes

enum WaveForm { WT_DIRECT, WT_STAGED, WT_STAGED_DEEP };

// Aligned for the 16-byte loads into `node` and the 8-byte reads of it, wherever
// the compiler places a kernel's LDS objects.
template <WaveForm F>
struct alignas(16) WaveLds {
    static constexpr int ROWS = F == WT_DIRECT ? 12 : F == WT_STAGED ? 9 : 14; // pending subtrees per lane
    static constexpr int WAVES = F == WT_DIRECT ? 8 : F == WT_STAGED ? 6 : 5;  // per SIMD
    static constexpr int SLOTS = 1024 * WAVES; // waves that the GPU's 1024 SIMDs hold at once
    char node[F == WT_DIRECT ? 256 : 4 * WT_SLOT]; // direct: only the row under the stack, which idle lanes read
    int stack[ROWS + 1][64];                       // row 0: WT_NONE under the bottom
};
template <WaveForm F>
constexpr bool wave_lds_aligned = alignof(WaveLds<F>) == 16 && offsetof(WaveLds<F>, node) == 0 && WT_SLOT % 16 == 0;
static_assert(wave_lds_aligned<WT_DIRECT> && wave_lds_aligned<WT_STAGED> && wave_lds_aligned<WT_STAGED_DEEP>,
              "load slots on 16 bytes");
typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) int lds_int;
typedef float vf2 __attribute__((ext_vector_type(2)));
typedef int vi2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ vf2 lds_pair(int addr) { return *(__attribute__((address_space(3))) vf2*)addr; }
__device__ __forceinline__ lds_int& lds_word(int addr) { return *(lds_int*)addr; }

// Lane J's value of each quad, in all four lanes.
template <int J>
__device__ __forceinline__ int quad_bcast(int v)
{
    return __builtin_amdgcn_mov_dpp(v, J * 0x55, 0xf, 0xf, true);
}

struct WaveRay {
    v3 o, d, inv;
    float tmin, tmax;
    int cur;        // node to visit: >= 0 interior, < 0 leaf ~rank, WT_NONE
    int child;      // leaf of the closest hit so far, WT_NONE: none
    int sp;         // LDS address of the row above the newest pending subtree
    int nx, ny, nz; // staged: LDS address of the near planes' pair per axis (less 16 per axis);
    int fx, fy, fz; //   and of the far planes'.  Direct: nx .. nz nonzero where inv < 0
};

// Whether max3 / min3 give intersectBoundT's result for this ray in a plain
// scene (mt_scene::plain): no product can be NaN (inv finite and not 0, origin and
// planes within 1e30) and the sign words say what inv does, so that per axis
// near <= far.
__device__ __forceinline__ bool ray_plain(const RayT& r)
{
    auto ok = [](float inv, float o, int s) {
        const float a = fabsf(inv);
        return a > 0.0f && a < INFINITY && fabsf(o) < 1e30f && (s != 0) == (inv < 0.0f);
    };
    return ok(r.inv.x, r.o.x, r.sx) && ok(r.inv.y, r.o.y, r.sy) && ok(r.inv.z, r.o.z, r.sz);
}

__device__ __forceinline__ void wave_ray_start(WaveRay& R, const RayT& r, int slot, int col, int root)
{
    R.o = r.o;
    R.d = r.d;
    R.inv = r.inv;
    R.tmin = r.tmin;
    R.tmax = r.tmax;
    R.cur = root;
    R.child = WT_NONE;
    // the last ray's last pop left sp at this row, and until the lane takes a
    // ray again the steps of the other lanes write there
    lds_word(col) = WT_NONE;
    R.sp = col + 256;
    const int sx = r.sx ? 8 : 0, sy = r.sy ? 8 : 0, sz = r.sz ? 8 : 0;
    R.nx = slot + sx;
    R.ny = slot + sy;
    R.nz = slot + sz;
    R.fx = slot + 8 - sx;
    R.fy = slot + 8 - sy;
    R.fz = slot + 8 - sz;
}

// intersectBoundT (Util.cl:707-732) on near and far planes.  EXACT: the
// reference's chain of conditional assignments, as box_hit.  Otherwise, for
// plain rays: the conjunction of its early outs is max(near) <= min(far) (the
// same-axis pairs hold by themselves), and its t is max(near).
template <bool EXACT>
__device__ __forceinline__ bool slab(const WaveRay& R, float nx, float ny, float nz, float fx, float fy, float fz,
                                     float& tnear)
{
    const float tmin = (nx - R.o.x) * R.inv.x, tmax = (fx - R.o.x) * R.inv.x;
    const float tymin = (ny - R.o.y) * R.inv.y, tymax = (fy - R.o.y) * R.inv.y;
    const float tzmin = (nz - R.o.z) * R.inv.z, tzmax = (fz - R.o.z) * R.inv.z;
    if (EXACT) {
        const bool xy = !((tmin > tymax) | (tymin > tmax));
        const float t1 = tymin > tmin ? tymin : tmin;
        const float u1 = tymax < tmax ? tymax : tmax;
        const bool xyz = !((t1 > tzmax) | (tzmin > u1));
        const float t2 = tzmin > t1 ? tzmin : t1;
        const float u2 = (tzmax < u1 ? tzmax : u1) * 1.00000024f;
        tnear = t2;
        return xy & xyz & (t2 < R.tmax) & (u2 > R.tmin);
    }
    const float t2 = fmaxf(fmaxf(tmin, tymin), tzmin), u = fminf(fminf(tmax, tymax), tzmax);
    tnear = t2;
    return (t2 <= u) & (t2 < R.tmax) & (u * 1.00000024f > R.tmin);
}

// A lane's pending subtrees lie in its column of the LDS stack, oldest first,
// above a row that holds WT_NONE (popped when none is left); those past the
// column's last row lie in `ovf`.  sp is the address of the row above the newest
// (256 bytes per row), `last` the address past the column.
__device__ __forceinline__ int wave_top(int sp, int last, const int* ovf)
{
    if (__any(sp > last)) { // rare
        if (sp > last) return ovf[(((sp - last) >> 8) - 1) & (WT_OVF - 1)];
    }
    return lds_word(sp - 256);
}

// One interior node for every lane that holds one.  Called with the whole
// wave active.
template <bool EXACT, bool WIDE, bool STAGED>
__device__ __forceinline__ void wave_step(const char* __restrict__ nodes, lds_char* slots, int last, int c16,
                                          int slot, WaveRay& R, int* ovf)
{
    const bool inner = R.cur >= 0;
    const int node = inner ? R.cur : 0; // the other lanes load the root's record
    vf2 nx, ny, nz, fx, fy, fz;
    vi2 ref;
    float4 px, py, pz;
    if (STAGED) {
        int alo, ahi = 0;
        if (WIDE) { // 64-bit address of this lane's node
            const uint64_t a = reinterpret_cast<uint64_t>(nodes) + ((uint64_t)(uint32_t)node << 6);
            alo = (int)(uint32_t)a;
            ahi = (int)(uint32_t)(a >> 32);
        } else {
            alo = node << 6; // byte offset into the scene's records
        }
#define WT_LOAD(J)                                                                                                   \
    {                                                                                                                \
        const char* a_;                                                                                              \
        if (WIDE)                                                                                                    \
            a_ = reinterpret_cast<const char*>(((uint64_t)(uint32_t)quad_bcast<J>(ahi) << 32) |                      \
                                               (uint32_t)quad_bcast<J>(alo)) + c16;                                  \
        else a_ = nodes + (uint32_t)(quad_bcast<J>(alo) + c16);                                                      \
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)a_,                          \
                                         (__attribute__((address_space(3))) void*)(slots + J * WT_SLOT), 16, 0, 0); \
    }
        WT_LOAD(0)
        WT_LOAD(1)
        WT_LOAD(2)
        WT_LOAD(3)
#undef WT_LOAD
    } else {
        const char* N = WIDE ? nodes + ((uint64_t)(uint32_t)node << 6) : nodes + (uint32_t)(node << 6);
        px = *reinterpret_cast<const float4*>(N);
        py = *reinterpret_cast<const float4*>(N + 16);
        pz = *reinterpret_cast<const float4*>(N + 32);
        ref = *reinterpret_cast<const vi2*>(N + 48);
    }
    const bool deep = __any(R.sp >= last); // rare
    int top;
    if (deep && R.sp > last) top = ovf[(((R.sp - last) >> 8) - 1) & (WT_OVF - 1)];
    else top = lds_word(R.sp - 256);
    if (STAGED) {
        __builtin_amdgcn_s_waitcnt(0x0f70); // vmcnt(0): the records are in LDS
        nx = lds_pair(R.nx), fx = lds_pair(R.fx);
        ny = lds_pair(R.ny + 16), fy = lds_pair(R.fy + 16);
        nz = lds_pair(R.nz + 32), fz = lds_pair(R.fz + 32);
        ref = *(__attribute__((address_space(3))) vi2*)(slot + 48);
    } else {
        auto pick = [](int neg, float4 p, vf2& n, vf2& f) {
            n.x = neg ? p.z : p.x, n.y = neg ? p.w : p.y;
            f.x = neg ? p.x : p.z, f.y = neg ? p.y : p.w;
        };
        pick(R.nx, px, nx, fx);
        pick(R.ny, py, ny, fy);
        pick(R.nz, pz, nz, fz);
    }
    float lt, rt;
    const bool lh = inner && slab<EXACT>(R, nx.x, ny.x, nz.x, fx.x, fy.x, fz.x, lt);
    const bool rh = inner && slab<EXACT>(R, nx.y, ny.y, nz.y, fx.y, fy.y, fz.y, rt);
    const bool both = lh && rh;
    const bool right = rh && (!lh || rt < lt); // nearer child first, ties to the left
    const bool pop = inner && !lh && !rh;
    const int near = right ? ref.y : ref.x, far = right ? ref.x : ref.y;
    if (deep) {
        if (both && R.sp >= last) ovf[((R.sp - last) >> 8) & (WT_OVF - 1)] = far;
        else if (both) lds_word(R.sp) = far;
    } else {
        lds_word(R.sp) = far; // above the top: kept only where both were hit
    }
    R.cur = pop ? top : (inner ? near : R.cur);
    R.sp += both ? 256 : 0;
    R.sp -= pop ? 256 : 0;
}

// What a wave's lanes need besides their rays.
template <WaveForm F>
struct WaveLane {
    lds_char* slots;
    int slot, col, last, c16;
    __device__ __forceinline__ WaveLane(WaveLds<F>* wave_lds)
    {
        const int lane = __lane_id();
        WaveLds<F>* lds = wave_lds + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        slots = (lds_char*)lds->node;
        slot = F != WT_DIRECT ? (int)(uintptr_t)slots + (lane & 3) * WT_SLOT + (lane >> 2) * 64 : 0;
        col = (int)(uintptr_t)(lds_int*)&lds->stack[0][lane];
        last = col + 256 * (WaveLds<F>::ROWS + 1);
        c16 = (lane & 3) << 4;
    }
    __device__ __forceinline__ void idle(WaveRay& R) const
    { // a lane that has had no ray yet
        R.cur = WT_NONE;
        R.sp = col + 256;
        R.nx = R.ny = R.nz = R.fx = R.fy = R.fz = slot;
    }
};

// Takes the wave's rays (lanes with `active`) on until leaves have been tested once:
// interior nodes while more than three quarters of the rays are at one, then the
// leaves that have been reached.  Clears `active` where a ray has ended.
// exact: some active ray needs intersectBoundT's chain.  Called with the whole
// wave active.
template <bool ANY, bool WIDE, WaveForm F>
__device__ __forceinline__ void wave_walk(const WaveLane<F>& W, MtSceneRef sc, bool exact, WaveRay& R, bool& active,
                                          int* ovf)
{
    constexpr bool STAGED = F != WT_DIRECT;
    const int thr = (int)__popcll(__ballot(active)) * 3 / 4;
    const char* nodes = reinterpret_cast<const char*>(sc.pn);
    if (exact) {
        while ((int)__popcll(__ballot(R.cur >= 0)) > thr)
            wave_step<true, WIDE, STAGED>(nodes, W.slots, W.last, W.c16, W.slot, R, ovf);
    } else {
        while ((int)__popcll(__ballot(R.cur >= 0)) > thr)
            wave_step<false, WIDE, STAGED>(nodes, W.slots, W.last, W.c16, W.slot, R, ovf);
    }
    if (R.cur < 0 && R.cur != WT_NONE) {
        const float4* T = sc.pt + 3 * (size_t)(~R.cur);
        const float4 t0 = T[0], t1 = T[1];
        const float e2z = T[2].x;
        RayT r;
        r.o = R.o;
        r.d = R.d;
        r.tmax = R.tmax;
        const float t = tri_hit(r, mk3(t0.x, t0.y, t0.z), mk3(t0.w, t1.x, t1.y), mk3(t1.z, t1.w, e2z));
        if ((R.tmin < t) && (t < R.tmax)) {
            R.child = R.cur;
            if (ANY) R.sp = W.col + 256; // found: nothing is pending any more
            else R.tmax = t;
        }
        R.cur = wave_top(R.sp, W.last, ovf);
        R.sp -= 256;
    }
    if (R.cur == WT_NONE) active = false;
}

// Traces the rays of entries [next, end) (wave-uniform).  load(id, r, sc)
// fills entry id's ray (WIDE: and may set the lane's scene, whose records are then
// addressed with 64 bits); done(fin, id, t, child, sc) is called with the whole
// wave active, fin set on the lanes whose ray has ended (t: its tMax after the
// walk, child: the leaf hit or WT_NONE).  `wave_lds`: one per wave of the
// work-group.
template <bool ANY, bool WIDE, int REFILL, WaveForm F, class Load, class Done>
__device__ __forceinline__ void wave_trace(WaveLds<F>* wave_lds, MtSceneRef scene, int next, int end, Load&& load,
                                           Done&& done)
{
    const WaveLane<F> W(wave_lds);
    int ovf[WT_OVF];
    bool active = false, ended = false, plain = true;
    int id = 0;
    MtSceneRef sc = scene; // this lane's scene
    WaveRay R;
    W.idle(R);
    for (;;) {
        const uint64_t idle = __ballot(!active);
        const int nidle = (int)__popcll(idle);
        if (nidle == 64 || (next < end && nidle >= REFILL)) {
            ended = ended && !active;
            if (__any(ended)) done(ended, id, R.tmax, R.child, sc);
            ended = false;
            if (next >= end) break; // run drained, every lane done
            const int avail = end - next;
            const int n = avail < nidle ? avail : nidle;
            const int rk = (int)lane_rank(idle);
            if (!active && rk < n) {
                id = next + rk;
                RayT r;
                load(id, r, sc);
                wave_ray_start(R, r, W.slot, W.col, sc.root);
                plain = ray_plain(r) && sc.plain;
                active = true;
            }
            next += n;
        }
        ended |= active;
        wave_walk<ANY, WIDE>(W, WIDE ? sc : scene, __any(active && !plain), R, active, ovf);
    }
}

// Primitive of a leaf, -1 for none.
__device__ __forceinline__ int leaf_prim(const float4* __restrict__ pt, int child)
{
    return child != WT_NONE ? __float_as_int(pt[3 * (size_t)(~child) + 2].y) : -1;
}

// How a launch is split into waves: a wave takes `run` consecutive rays, so
// many that the launch just fills the GPU's wave slots (`slots`, of the
// kernel's form) where there are few rays, WT_MAX_RUN where there are many (a
// wave's start and drain, with few lanes busy, then weigh little).  993K soup
// rays per bounce: filling exactly the staged form's 6144 slots instead of
// 8192 waves took a whole render from 5.49 to 5.07 ms (the last third of a
// second round of waves is gone); 957K short rays in runs of 30 instead of
// 128: 0.29 -> 0.73 ms.

// Rays per wave of a plain queue of up to n entries.  Below WT_MIN_RUN rays for
// each of two waves per SIMD they are spread thinner: a wave lasts as long as
// its lanes together need, but a wave of few lanes costs the SIMD as much as
// a full one (with launch and read-back, 4096 camera rays in waves of 16: 278
// us, of 4: 251; 30000 in waves of 16: 303, of 4: 391).
__host__ __device__ inline int wave_run(int n, int slots)
{
    const int r = (n / slots + 15) & ~15, few = (n / 2048 + 4) & ~3;
    if (r <= WT_MIN_RUN) return few < WT_MIN_RUN ? few : WT_MIN_RUN;
    return r > WT_MAX_RUN ? WT_MAX_RUN : r;
}

// Waves of a launch over a plain queue of up to n entries whose length only the
// device knows: as many as a full queue takes, and enough to fill the slots
// with fewer entries.
inline int64_t wave_count(int n, int slots)
{
    const int64_t full = ((int64_t)n + wave_run(n, slots) - 1) / wave_run(n, slots);
    const int64_t few = ((int64_t)n + WT_MIN_RUN - 1) / WT_MIN_RUN;
    const int64_t fill = few < slots ? few : slots;
    return full > fill ? full : fill;
}

// The run of this wave in a plain queue of `count` entries (at least 0): lengths
// by the count, not by the capacity (the drain of 24 jobs through a queue of 2M:
// 300K entries in runs of 256 left four of five wave slots empty; an iteration's
// closest hits 0.36 -> 0.2 ms.  20000 random rays in a queue of 2M, closest hit:
// 257 -> 118 us, staged 251 -> 122; 100000: 258 -> 189, 254 -> 158; 1M: 515 ->
// 557, 380 -> 383, what a queue of that capacity takes).
__device__ __forceinline__ void plain_run(int count, int slots, int& next, int& end)
{
    const unsigned waves = gridDim.x * 4; // at most 2^31 / 4 (wave_count)
    int run = wave_run(count, slots);
    if ((int64_t)run * waves < count) run = (int)(((unsigned)count + waves - 1) / waves); // the grid covers the queue
    const int64_t first = (int64_t)(blockIdx.x * 4 + (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * run;
    next = first < count ? (int)first : count;
    end = count - next < run ? count : next + run;
}

// Work-groups per segment of a queue of nseg segments.
inline int wave_seg_groups(int seg_cap, int nseg, int slots)
{
    const int want = slots / 4 / nseg;
    const int full = (seg_cap + 4 * WT_MAX_RUN - 1) / (4 * WT_MAX_RUN);
    const int most = (seg_cap + 4 * WT_MIN_RUN - 1) / (4 * WT_MIN_RUN);
    return full > want ? full : (want < most ? want : most);
}

// The run of this wave in a queue of nseg segments of seg_cap entries,
// counts[p] live in segment p: work-group v (seg_sweep_group) belongs to
// segment v mod nseg.  Lengths as above, from the segment's count.
__device__ __forceinline__ void seg_run(const int* __restrict__ counts, int nseg, int seg_cap, int slots, int& next,
                                        int& end)
{
    const unsigned v = seg_sweep_group();
    const int p = (int)(v % (unsigned)nseg), c = (int)(v / (unsigned)nseg);
    const int waves = (int)(gridDim.x / (unsigned)nseg) * 4;
    int cnt = counts[p];
    cnt = cnt < seg_cap ? cnt : seg_cap;
    const int want = slots / nseg;
    int run = (cnt + want - 1) / want;
    run = run < WT_MIN_RUN ? WT_MIN_RUN : (run > WT_MAX_RUN ? WT_MAX_RUN : run);
    if (run < (cnt + waves - 1) / waves) run = (cnt + waves - 1) / waves; // the grid covers the segment
    const int off = (c * 4 + (int)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * run;
    next = p * seg_cap + off;
    end = p * seg_cap + (cnt < off + run ? cnt : off + run);
}

// Whether node records lie beyond a 32-bit byte offset.
inline bool scene_wide(const mt_scene* sc) { return sc->num_interior > (1 << 26); }

template <bool ANY, bool STATS, bool SHORT_STACK>
__device__ __forceinline__ int trace_packed(const float4* __restrict__ pn,
                                            const float4* __restrict__ pt, int root, RayT& r,
                                            int& child, int* st)
{
    int hit = 0;
    int cur = root;
    BitStack bs{0, 0};
    ShortStack ss;
    ss.n = 0;
    for (;;) {
        while (cur >= 0) {
            const float4* N = pn + 4 * (size_t)cur;
            float4 a = N[0], b = N[1], c = N[2];
            int4 d = *reinterpret_cast<const int4*>(N + 3);
            float lt, rt;
            bool lh = box_hit(r, a.x, b.x, c.x, a.z, b.z, c.z, lt);
            bool rh = box_hit(r, a.y, b.y, c.y, a.w, b.w, c.w, rt);
            if (STATS) st[0]++;
            if (!lh && !rh) break;
            bs.push0();
            int nxt;
            if (lh && rh) {
                bool right_first = rt < lt;
                nxt = right_first ? d.y : d.x;
                if (SHORT_STACK) ss.push(right_first ? d.x : d.y);
                bs.lo |= 1;
            } else {
                nxt = lh ? d.x : d.y;
            }
            cur = nxt;
        }
        if (cur < 0) {
            if (STATS) st[1]++;
            const float4* T = pt + 3 * (size_t)(~cur);
            float4 t0 = T[0], t1 = T[1], t2 = T[2];
            float t = tri_hit(r, mk3(t0.x, t0.y, t0.z), mk3(t0.w, t1.x, t1.y), mk3(t1.z, t1.w, t2.x));
            if ((r.tmin < t) && (t < r.tmax)) {
                if (ANY) return 1;
                hit = 1;
                r.tmax = t;
                child = __float_as_int(t2.y);
            }
        }
        if (bs.empty()) return hit;
        if (SHORT_STACK && ss.n > 0) {
            // the lowest 1 bit's far child is on top of the short stack
            int z = bs.ctz();
            if (STATS) st[2] += z;
            bs.shr(z);
            bs.lo ^= 1;
            cur = ss.pop();
            continue;
        }
        if (!parent_walk<STATS>(pn, pt, cur, bs, st)) return hit;
    }
}

} // namespace
