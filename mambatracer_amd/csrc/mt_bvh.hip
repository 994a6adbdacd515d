// Device BVH builder: CNormalBVH.build/subdivide (src/cl/scene/
// CNormalBVH.java:45-148) on the GPU, producing the same nodes and bounds as
// the host builder mt_bvh_build (same node numbering, same primitive order
// in the leaves, bounds equal up to the sign of zero).
//
// The reference recurses depth first.  Here the nodes of more than SUB
// primitives grow one level per round, every node of a level at once, and
// each subtree of at most SUB primitives is then built by one work-group in
// LDS (k_subtrees).  A round:
//   1. k_bounds: each wave takes WIN positions of the object order and reduces
//      the boxes and centroids of every node's run in them (positions of one
//      node are contiguous) to one partial result per run: a window holds at
//      most a run that began before it, a whole node, and a run that goes on;
//   2. k_node: a work-group per node combines its windows' partials: bounds,
//      split axis (largest centroid extent), centroid midpoint;
//   3. k_flag_scan: right = centroid[axis] >= split per position, and in the
//      same pass (decoupled look-back) the exclusive scan of these flags;
//   4. k_pair: mid = start + lefts (or the midpoint index when one side is
//      empty), child numbering from the depth-first counter formula (left child
//      `base`, right `base + 1`, left subtree from `base + 2`, right subtree
//      from `base + 2 * lefts`), child records; and the two-pointer
//      partition's pairs: the k-th right element from the left of [start, mid)
//      trades places with the k-th left element from the right of [mid, end),
//      exactly the swaps the sequential partition performs;
//   5. k_scatter: the swaps, in place; each element takes its child's id.
// Counts stay on the device; the host enqueues the rounds that every tree of
// this size needs and then looks every few rounds.
//
// What bounded the first version, one level per round to the leaves with a
// read-back each (1.05M triangles of 256 spheres: 6.7 ms, 30 rounds of nine
// launches): atomics of all waves on the root's twelve keys (174 us) and, at
// the leaves, on one or two primitives' keys per run (up to 198 us per round),
// an idle gap of 45 us per read-back, and about 1 ms of allocating and freeing
// the state.  Now 1.78 ms: a round of large nodes 60 us (k_bounds 16-21,
// k_flag_scan 22, the rest 5-10 each), the subtrees 345 us.
#include "mt_lookback.h"

namespace {

constexpr int BB = 256;
constexpr int SUB = 256; // primitives of a subtree that one work-group finishes (a lane each)
constexpr int WIN = 512; // positions per wave of k_bounds; < 2 (SUB + 1): at most one whole node inside
static_assert(WIN < 2 * (SUB + 1) && BB == SUB, "k_bounds: one whole node per window");
constexpr int FLAG_ROWS = 8; // rows of BB positions per tile of k_flag_scan
constexpr int FLAG_TILE = BB * FLAG_ROWS;

__device__ __forceinline__ int fkey(float f)
{ // order-preserving int key of a float (min/max on keys = min/max on floats)
    int b = __float_as_int(f);
    return b >= 0 ? b : b ^ 0x7FFFFFFF;
}
__device__ __forceinline__ float fval(int k) { return __int_as_float(k >= 0 ? k : k ^ 0x7FFFFFFF); }

// Twelve keys of a set of primitives: box min xyz, box max xyz, centroid min
// xyz, centroid max xyz.
struct Keys {
    int v[12];
};
__device__ __forceinline__ bool key_is_max(int k) { return ((k / 3) & 1) != 0; }
__device__ __forceinline__ int kcomb(int k, int x, int y)
{
    return key_is_max(k) ? (x > y ? x : y) : (x < y ? x : y);
}
__device__ __forceinline__ int key_none(int k) { return key_is_max(k) ? fkey(-INFINITY) : fkey(INFINITY); }
__device__ __forceinline__ Keys prim_keys(float4 a, float4 b, float4 c)
{ // box min, box max, centroid
    auto mn = [](int x, int y) { return x < y ? x : y; };
    auto mx = [](int x, int y) { return x > y ? x : y; };
    Keys K;
    const float A[3] = {a.x, a.y, a.z}, B[3] = {b.x, b.y, b.z}, C[3] = {c.x, c.y, c.z};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        K.v[d] = mn(fkey(A[d]), fkey(B[d]));
        K.v[3 + d] = mx(fkey(A[d]), fkey(B[d]));
        K.v[6 + d] = K.v[9 + d] = fkey(C[d]);
    }
    return K;
}

// Split axis and position of a node (subdivide, CNormalBVH.java:100-132).
__device__ __forceinline__ void node_split(const int* K, int& axis, float& split)
{
    const float cmn[3] = {fval(K[6]), fval(K[7]), fval(K[8])}, cmx[3] = {fval(K[9]), fval(K[10]), fval(K[11])};
    const float dx = cmx[0] - cmn[0], dy = cmx[1] - cmn[1], dz = cmx[2] - cmn[2];
    axis = (dx > dy && dx > dz) ? 0 : (dy > dz ? 1 : 2);
    split = axis == 0 ? 0.5f * (cmn[0] + cmx[0]) : (axis == 1 ? 0.5f * (cmn[1] + cmx[1]) : 0.5f * (cmn[2] + cmx[2]));
}

__device__ __forceinline__ void write_bounds(float* pb, const int* K)
{
    pb[0] = fval(K[0]);
    pb[1] = fval(K[1]);
    pb[2] = fval(K[2]);
    pb[3] = 0.0f;
    pb[4] = fval(K[3]);
    pb[5] = fval(K[4]);
    pb[6] = fval(K[5]);
    pb[7] = 0.0f;
}

// cnt: node counts of the rounds' lists (round r: word r mod 4), then
constexpr int CNT_SMALL = 4; // subtrees handed to k_subtrees
constexpr int CNT_DEPTH = 5; // deepest leaf
constexpr int CNT_WORDS = 8;

struct BuildState {
    int n;
    float4 *pmn, *pmx, *cen; // per primitive
    int* obj;                // object order
    int* seg;                // node id of each position, -1 once in a subtree of at most SUB
    int* scan;               // exclusive scan of the right flags, [n] = total
    int* table;              // pairing table, indexed start + k
    int* part;               // k_bounds: per window 3 x 12 keys
    // per node
    int *nstart, *nend, *nbase;
    int* nmid;               // split position; ~mid for a node without swaps (one side was empty)
    int* naxis;
    float* nsplit;
    int* list[2];            // this round's nodes, the next round's
    int2* small;             // (node, level) of the subtrees
    int* cnt;
    int* nodes;
    float* bounds;
};

__global__ void k_prims(BuildState S, const float4* __restrict__ points, const int* __restrict__ faces)
{ // CMesh.getBound (CMesh.java:64-71) and the box centre per primitive
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) { // the root
        S.nstart[0] = 0;
        S.nend[0] = S.n;
        S.nbase[0] = 1;
        for (int k = 0; k < 7; k++) S.nodes[k] = 0;
        for (int k = 0; k < CNT_WORDS; k++) S.cnt[k] = 0;
        S.cnt[S.n > SUB ? 0 : CNT_SMALL] = 1;
        S.list[0][0] = 0;
        S.small[0] = make_int2(0, 0);
    }
    if (i >= S.n) return;
    float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int k = 0; k < 3; k++) {
        float4 p = points[faces[10 * (size_t)i + k]];
        float c[3] = {p.x, p.y, p.z};
        for (int a = 0; a < 3; a++) { // CBound.include, CBound.java:54-70
            if (c[a] < mn[a]) mn[a] = c[a];
            if (c[a] > mx[a]) mx[a] = c[a];
        }
    }
    S.pmn[i] = make_float4(mn[0], mn[1], mn[2], 0.0f);
    S.pmx[i] = make_float4(mx[0], mx[1], mx[2], 0.0f);
    S.cen[i] = make_float4(0.5f * (mn[0] + mx[0]), 0.5f * (mn[1] + mx[1]), 0.5f * (mn[2] + mx[2]), 0.0f);
    S.obj[i] = i;
    S.seg[i] = 0;
}

// Wave-wide result of a run, stored by lane 0: partial 0 of the window for a
// run that began before it, 2 for a whole node, 1 for a run that goes on.
__device__ __forceinline__ void flush_run(const BuildState& S, int s, const Keys& acc, int base)
{
    int* P = S.part + 36 * (size_t)(base / WIN);
    const int start = S.nstart[s];
    P += 12 * (start < base ? 0 : (S.nend[s] <= base + WIN ? 2 : 1));
#pragma unroll
    for (int k = 0; k < 12; k++) {
        int v = acc.v[k];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v = kcomb(k, v, __shfl_xor(v, o));
        if (__lane_id() == 0) P[k] = v;
    }
}

// Bound by the gather of 48 bytes per primitive and the few waves a level
// has; a run's lanes accumulate on their own and are combined once at its
// end.  1.05M positions: 174 us (root, atomics) and 41 us (most rounds) before.
__global__ __launch_bounds__(BB) void k_bounds(BuildState S, const int* __restrict__ count)
{
    if (*count == 0) return;
    const int lane = __lane_id();
    const int64_t base = (((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6) * WIN;
    if (base >= S.n) return; // wave-uniform
    int cs = -1;             // node of the open run (wave-uniform)
    Keys acc;
    for (int row = 0; row < WIN; row += 64) {
        const int64_t i = base + row + lane;
        if (base + row >= S.n) break; // wave-uniform
        const int s = i < S.n ? S.seg[i] : -1;
        Keys K;
        if (s >= 0) {
            const int p = S.obj[i];
            K = prim_keys(S.pmn[p], S.pmx[p], S.cen[p]);
        }
        uint64_t left = __ballot(true);
        while (left) { // one pass per node that the row holds
            const int sl = __shfl(s, (int)__builtin_ctzll(left));
            const uint64_t run = __ballot(s == sl) & left;
            if (sl != cs) {
                if (cs >= 0) flush_run(S, cs, acc, (int)base);
                cs = sl;
#pragma unroll
                for (int k = 0; k < 12; k++) acc.v[k] = key_none(k);
            }
            if (sl >= 0 && ((run >> lane) & 1ull)) {
#pragma unroll
                for (int k = 0; k < 12; k++) acc.v[k] = kcomb(k, acc.v[k], K.v[k]);
            }
            left &= ~run;
        }
    }
    if (cs >= 0) flush_run(S, cs, acc, (int)base);
}

// A work-group per node of the round's list.  Work-group 0 also readies the
// look-back of k_flag_scan and the list count of the round after next.
__global__ __launch_bounds__(BB) void k_node(BuildState S, const int* __restrict__ list,
                                             const int* __restrict__ count, int* __restrict__ zero, ScanWork W)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *zero = 0;
        W.ticket[0] = 0u;
        const uint32_t e = (W.ticket[2] + 1u) & 0x3FFFFFFFu; // epoch 0 is never current
        W.ticket[2] = e ? e : 1u;
    }
    if ((int)blockIdx.x >= *count) return;
    __shared__ int s_k[BB / 64][12];
    const int s = list[blockIdx.x];
    const int start = S.nstart[s], end = S.nend[s];
    const int w0 = start / WIN, w1 = (end - 1) / WIN;
    int v[12];
#pragma unroll
    for (int k = 0; k < 12; k++) v[k] = key_none(k);
    for (int w = w0 + (int)threadIdx.x; w <= w1; w += BB) {
        const int* P = S.part + 36 * (size_t)w + 12 * (w > w0 ? 0 : (w0 == w1 ? 2 : 1));
#pragma unroll
        for (int k = 0; k < 12; k++) v[k] = kcomb(k, v[k], P[k]);
    }
#pragma unroll
    for (int k = 0; k < 12; k++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v[k] = kcomb(k, v[k], __shfl_xor(v[k], o));
        if (__lane_id() == 0) s_k[threadIdx.x >> 6][k] = v[k];
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
#pragma unroll
    for (int k = 0; k < 12; k++)
        for (int w = 1; w < BB / 64; w++) v[k] = kcomb(k, v[k], s_k[w][k]);
    write_bounds(S.bounds + 8 * (size_t)s, v);
    S.nodes[7 * (size_t)s] = s;
    node_split(v, S.naxis[s], S.nsplit[s]);
}

// Right flags and their exclusive scan in one pass (1.05M positions: 26 + 19
// us as two kernels and a reset before).
__global__ __launch_bounds__(BB) void k_flag_scan(BuildState S, const int* __restrict__ count, ScanWork W)
{
    __shared__ int s_tile;
    __shared__ uint32_t s_wave[FLAG_ROWS][BB / 64];
    __shared__ uint32_t s_prefix;
    if (*count == 0) return;
    const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6;
    const uint32_t epoch = W.ticket[2];
    if (tid == 0) s_tile = (int)atomicAdd(&W.ticket[0], 1u);
    __syncthreads();
    const int64_t base = (int64_t)s_tile * FLAG_TILE;
    uint64_t mask[FLAG_ROWS];
#pragma unroll
    for (int k = 0; k < FLAG_ROWS; k++) {
        const int64_t i = base + k * BB + tid;
        bool right = false;
        if (i < S.n) {
            const int s = S.seg[i];
            if (s >= 0) {
                const float4 c = S.cen[S.obj[i]];
                const int dim = S.naxis[s];
                const float v = dim == 0 ? c.x : (dim == 1 ? c.y : c.z);
                right = !(v < S.nsplit[s]); // the partition keeps centroid < split on the left
            }
        }
        mask[k] = __ballot(right);
        if (lane == 0) s_wave[k][wave] = (uint32_t)__popcll(mask[k]);
    }
    __syncthreads();
    if (tid == 0) {
        uint32_t run = 0;
        for (int k = 0; k < FLAG_ROWS; k++)
            for (int w = 0; w < BB / 64; w++) {
                const uint32_t t = s_wave[k][w];
                s_wave[k][w] = run;
                run += t;
            }
        s_prefix = run;
    }
    __syncthreads();
    if (wave == 0) {
        const uint32_t agg = s_prefix;
        const uint32_t pre = look_back(W, s_tile, agg, epoch);
        if (lane == 0) {
            s_prefix = pre;
            if (base + FLAG_TILE >= S.n) S.scan[S.n] = (int)(pre + agg);
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < FLAG_ROWS; k++) {
        const int64_t i = base + k * BB + tid;
        if (i < S.n) S.scan[i] = (int)(s_prefix + s_wave[k][wave] + lane_rank(mask[k]));
    }
}

// Split position of a node of [start, end) with `rights` right elements;
// swaps: whether both sides have elements.
__device__ __forceinline__ int node_mid(int start, int end, int rights, bool& swaps)
{
    const int mid = end - rights;
    swaps = mid != start && mid != end;
    return swaps ? mid : start + (end - start) / 2; // one side empty: the range in half
}

// Records of both children: own id, sibling, parent.
__device__ __forceinline__ void child_records(int* nodes, int parent, int li)
{
    int* pn = nodes + 7 * (size_t)parent;
    pn[2] = li;
    pn[3] = li + 1;
    int* c = nodes + 7 * (size_t)li;
    for (int k = 0; k < 14; k++) c[k] = 0;
    c[1] = li + 1;
    c[4] = parent;
    c[7 + 1] = li;
    c[7 + 4] = parent;
}

// A node's first position makes its children; positions of the right part
// register the k-th left element counted from the right at table[start + k].
__global__ __launch_bounds__(BB) void k_pair(BuildState S, const int* __restrict__ count, int* __restrict__ next,
                                             int* __restrict__ next_count, int level)
{
    if (*count == 0) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= S.n) return;
    const int s = S.seg[i];
    if (s < 0) return;
    const int start = S.nstart[s], end = S.nend[s], send = S.scan[end];
    bool swaps;
    const int mid = node_mid(start, end, send - S.scan[start], swaps);
    if (i == start) {
        const int base = S.nbase[s];
        S.nmid[s] = swaps ? mid : ~mid;
        child_records(S.nodes, s, base);
        for (int c = 0; c < 2; c++) {
            const int id = base + c, a = c ? mid : start, b = c ? end : mid;
            S.nstart[id] = a;
            S.nend[id] = b;
            S.nbase[id] = c ? base + 2 * (mid - start) : base + 2;
            if (b - a > SUB) next[atomicAdd(next_count, 1)] = id;
            else S.small[atomicAdd(&S.cnt[CNT_SMALL], 1)] = make_int2(id, level + 1);
        }
    }
    if (!swaps || i < mid) return;
    const int after = S.scan[i + 1];
    if (after != S.scan[i]) return;                  // a right element
    const int k = (end - 1 - i) - (send - after);    // left elements in (i, end)
    S.table[start + k] = i;
}

// The partition's swaps, and the next round's node ids.
__global__ __launch_bounds__(BB) void k_scatter(BuildState S, const int* __restrict__ count)
{
    if (*count == 0) return;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= S.n) return;
    const int s = S.seg[i];
    if (s < 0) return;
    const int m = S.nmid[s], start = S.nstart[s];
    const int mid = m < 0 ? ~m : m;
    const int at = S.scan[i];
    if (m >= 0 && i < mid && S.scan[i + 1] != at) {
        const int q = S.table[start + (at - S.scan[start])]; // right elements in [start, i)
        const int x = S.obj[i];
        S.obj[i] = S.obj[q]; // nobody else touches i or q
        S.obj[q] = x;
    }
    const bool right = i >= mid;
    const int len = right ? S.nend[s] - mid : mid - start;
    S.seg[i] = len > SUB ? S.nbase[s] + (right ? 1 : 0) : -1;
}

// One subtree of at most SUB primitives, level by level in LDS: lane t is
// position t, node j of the subtree is created by the level above and handled by
// lane j - lo.  Same steps as a round.  Bound by its barriers (seven per
// level) and LDS atomics: 1.05M primitives in 6,200 subtrees 345 us, the
// last thirteen of 30 rounds before (2.2 ms).
__global__ __launch_bounds__(SUB, 3) void k_subtrees(BuildState S)
{
    __shared__ float s_c[3][SUB];               // centroids, by initial position
    __shared__ int s_obj[SUB];                  // primitive ids, by initial position
    __shared__ short s_ord[SUB];                // position -> initial position
    __shared__ short s_tab[SUB];
    __shared__ short s_scan[SUB + 1];
    __shared__ int s_wave[SUB / 64];
    __shared__ int s_key[2 * SUB][12];
    __shared__ short s_start[2 * SUB], s_end[2 * SUB], s_mid[2 * SUB];
    __shared__ int s_id[2 * SUB], s_base[2 * SUB];
    __shared__ signed char s_axis[2 * SUB];     // 0 .. 2, -1: leaf
    __shared__ float s_split[2 * SUB];
    __shared__ short s_child[2 * SUB];          // local index of the left child
    __shared__ int s_n;
    const int2 sub = S.small[blockIdx.x];
    const int first = S.nstart[sub.x], m = S.nend[sub.x] - first;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    Keys K;
    int p0 = 0; // this position's node, -1 once in a leaf
    if (t < m) {
        const int p = S.obj[first + t];
        s_obj[t] = p;
        s_ord[t] = (short)t;
        const float4 c = S.cen[p];
        s_c[0][t] = c.x;
        s_c[1][t] = c.y;
        s_c[2][t] = c.z;
        K = prim_keys(S.pmn[p], S.pmx[p], c);
    } else {
        p0 = -1;
    }
    // lane t keeps the keys of the primitive at initial position t; `own` is
    // the position where that primitive is now
    if (t == 0) {
        s_start[0] = 0;
        s_end[0] = (short)m;
        s_id[0] = sub.x;
        s_base[0] = S.nbase[sub.x];
        s_n = 1;
    }
    if (t < 12) s_key[0][t] = key_none(t);
    __shared__ short s_node[SUB];               // node of each position
    s_node[t] = (short)p0;
    __shared__ short s_own[SUB];                // initial position -> position
    s_own[t] = (short)t;
    int lo = 0, hi = 1, level = sub.y;
    __syncthreads();
    for (;;) {
        // bounds: every primitive adds its keys to its node's
        const int mine = t < m ? s_node[s_own[t]] : -1;
        if (mine >= 0) {
#pragma unroll
            for (int k = 0; k < 12; k++) {
                if (key_is_max(k)) atomicMax(&s_key[mine][k], K.v[k]);
                else atomicMin(&s_key[mine][k], K.v[k]);
            }
        }
        __syncthreads();
        const int j = lo + t; // this lane's node of the level
        if (j < hi) {
            const int id = s_id[j];
            write_bounds(S.bounds + 8 * (size_t)id, s_key[j]);
            int* pn = S.nodes + 7 * (size_t)id;
            pn[0] = id;
            if (s_end[j] - s_start[j] < 2) {
                pn[6] = s_obj[s_ord[s_start[j]]];
                pn[5] = 1;
                s_axis[j] = -1;
            } else {
                int axis;
                node_split(s_key[j], axis, s_split[j]);
                s_axis[j] = (signed char)axis;
            }
        }
        __syncthreads();
        // flags and their scan
        const int s = s_node[t];
        bool right = false;
        if (s >= 0) {
            const int axis = s_axis[s];
            if (axis < 0) s_node[t] = -1;
            else right = !(s_c[axis][s_ord[t]] < s_split[s]);
        }
        const uint64_t mask = __ballot(right);
        if (lane == 0) s_wave[wave] = (int)__popcll(mask);
        __syncthreads();
        int at = (int)lane_rank(mask);
        for (int w = 0; w < wave; w++) at += s_wave[w];
        s_scan[t] = (short)at;
        if (t == SUB - 1) s_scan[SUB] = (short)(at + (right ? 1 : 0));
        __syncthreads();
        // children
        if (j < hi && s_axis[j] >= 0) {
            const int a = s_start[j], b = s_end[j];
            bool swaps;
            const int mid = node_mid(a, b, s_scan[b] - s_scan[a], swaps);
            s_mid[j] = (short)(swaps ? mid : ~mid);
            const int base = s_base[j];
            child_records(S.nodes, s_id[j], base);
            const int c = atomicAdd(&s_n, 2);
            s_child[j] = (short)c;
            s_start[c] = (short)a;
            s_end[c] = s_start[c + 1] = (short)mid;
            s_end[c + 1] = (short)b;
            s_id[c] = base;
            s_id[c + 1] = base + 1;
            s_base[c] = base + 2;
            s_base[c + 1] = base + 2 * (mid - a);
            for (int k = 0; k < 12; k++) s_key[c][k] = s_key[c + 1][k] = key_none(k);
        }
        __syncthreads();
        lo = hi;
        hi = s_n;
        if (lo == hi) break; // every node of the level was a leaf
        level++;
        // pairs
        int mid = 0, start = 0;
        bool swaps = false;
        if (s >= 0 && s_axis[s] >= 0) {
            mid = s_mid[s];
            swaps = mid >= 0;
            mid = swaps ? mid : ~mid;
            start = s_start[s];
            const int end = s_end[s];
            if (swaps && t >= mid && !right) s_tab[start + (end - 1 - t) - (s_scan[end] - s_scan[t + 1])] = (short)t;
        }
        __syncthreads();
        // swaps, next nodes
        if (s >= 0 && s_axis[s] >= 0) {
            if (swaps && t < mid && right) {
                const int q = s_tab[start + (at - s_scan[start])];
                const short x = s_ord[t], y = s_ord[q];
                s_ord[t] = y;
                s_ord[q] = x;
                s_own[y] = (short)t;
                s_own[x] = (short)q;
            }
            s_node[t] = (short)(s_child[s] + (t >= mid ? 1 : 0));
        }
        __syncthreads();
    }
    if (t == 0) atomicMax(&S.cnt[CNT_DEPTH], level);
}

// The build state (120 bytes per primitive).  Up to BUILD_KEEP it lives in the
// context's workspace, which the context keeps: allocating and freeing it would
// cost a small build dear (0.4 ms at 4.6M primitives).  A larger one is given
// back by the call, unless the workspace is that large already: 4.6M
// primitives 8.07 ms kept, 8.48 given back; 16M 27.4, 28.2, and 1.8 GB.
constexpr size_t BUILD_KEEP = (size_t)512 << 20; // 4.4M primitives
struct BuildMem {
    mt_context* ctx;
    void *p = nullptr, *own = nullptr;
    explicit BuildMem(mt_context* c) : ctx(c) {}
    BuildMem(const BuildMem&) = delete;
    ~BuildMem()
    {
        if (!own) return;
        (void)hipStreamSynchronize(ctx->stream); // also after an error: launches may still use it
        (void)hipFree(own);
    }
    int32_t take(size_t bytes)
    {
        if (bytes <= BUILD_KEEP || bytes <= ctx->temp_bytes) return mt_ctx_temp(ctx, bytes, &p);
        if (hipMalloc(&own, bytes) != hipSuccess) {
            own = nullptr;
            mt_set_error("mt_bvh_build_device: cannot allocate %.2f GB of build state", bytes / 1e9);
            return MT_ERR_ALLOC;
        }
        p = own;
        return MT_OK;
    }
};

} // namespace

extern "C" int32_t mt_bvh_build_device(mt_context* ctx, int32_t ntris, const float* points, const int32_t* faces,
                                       int32_t* nodes, float* bounds, int32_t* max_depth)
{
    MT_ARG_CHECK(ctx && points && faces && nodes && bounds, "mt_bvh_build_device: NULL argument");
    MT_ARG_CHECK(ntris >= 1 && ntris <= (1 << 30), "mt_bvh_build_device: ntris %d", ntris);
    const size_t n = (size_t)ntris, m = 2 * n - 1, big = n / (SUB + 1) + 1; // nodes of more than SUB per round
    const int nwin = (int)((n + WIN - 1) / WIN);
    size_t bytes = 0;
    auto take = [&](size_t b) { size_t off = bytes; bytes += (b + 255) & ~(size_t)255; return off; };
    size_t oMn = take(16 * n), oMx = take(16 * n), oCen = take(16 * n);
    size_t oObj = take(4 * n), oSeg = take(4 * n), oScan = take(4 * (n + 1)), oTab = take(4 * n);
    size_t oPart = take(4 * 36 * (size_t)nwin);
    size_t oStart = take(4 * m), oEnd = take(4 * m), oBase = take(4 * m), oMid = take(4 * m), oAxis = take(4 * m);
    size_t oSplit = take(4 * m);
    size_t oList0 = take(4 * big), oList1 = take(4 * big), oSmall = take(8 * n), oCnt = take(4 * CNT_WORDS);
    BuildMem mem(ctx);
    int32_t rc = mem.take(bytes);
    if (rc) return rc;
    ScanWork W;
    const int64_t ntiles = ((int64_t)n + FLAG_TILE - 1) / FLAG_TILE;
    rc = scan_workspace_tiles(ctx, ntiles, W);
    if (rc) return rc;
    char* at = reinterpret_cast<char*>(mem.p);
    auto I = [&](size_t o) { return reinterpret_cast<int*>(at + o); };
    BuildState S;
    S.n = ntris;
    S.pmn = reinterpret_cast<float4*>(at + oMn);
    S.pmx = reinterpret_cast<float4*>(at + oMx);
    S.cen = reinterpret_cast<float4*>(at + oCen);
    S.obj = I(oObj);
    S.seg = I(oSeg);
    S.scan = I(oScan);
    S.table = I(oTab);
    S.part = I(oPart);
    S.nstart = I(oStart);
    S.nend = I(oEnd);
    S.nbase = I(oBase);
    S.nmid = I(oMid);
    S.naxis = I(oAxis);
    S.nsplit = reinterpret_cast<float*>(at + oSplit);
    S.list[0] = I(oList0);
    S.list[1] = I(oList1);
    S.small = reinterpret_cast<int2*>(at + oSmall);
    S.cnt = I(oCnt);
    S.nodes = nodes;
    S.bounds = bounds;
    hipStream_t st = ctx->stream;
    const int grid = mt_blocks((int64_t)n, BB);
    int host[CNT_WORDS];
    auto read_counts = [&]() -> int32_t {
        if (hipGetLastError() != hipSuccess ||
            hipMemcpyAsync(host, S.cnt, sizeof(host), hipMemcpyDeviceToHost, st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess) {
            mt_set_error("mt_bvh_build_device: launch or read-back failed");
            return MT_ERR_HIP;
        }
        return MT_OK;
    };
    k_prims<<<grid, BB, 0, st>>>(S, reinterpret_cast<const float4*>(points), faces);
    // a tree of n > SUB primitives has nodes of more than SUB in at least
    // log2(n / SUB) rounds; past those, a look every three rounds (an empty
    // round costs five launches that leave at once, a look a 40 us gap)
    int ahead = 0;
    while (((int64_t)SUB << ahead) < (int64_t)n) ahead++;
    int level = 0;
    host[0] = n > SUB ? 1 : 0;
    while (host[level & 3] > 0) {
        for (int r = 0; r < ahead; r++, level++) {
            int* count = S.cnt + (level & 3);
            int* next_count = S.cnt + ((level + 1) & 3);
            k_bounds<<<mt_blocks((int64_t)nwin * 64, BB), BB, 0, st>>>(S, count);
            k_node<<<(unsigned)big, BB, 0, st>>>(S, S.list[level & 1], count, S.cnt + ((level + 2) & 3), W);
            k_flag_scan<<<(unsigned)ntiles, BB, 0, st>>>(S, count, W);
            k_pair<<<grid, BB, 0, st>>>(S, count, S.list[1 - (level & 1)], next_count, level);
            k_scatter<<<grid, BB, 0, st>>>(S, count);
        }
        if ((rc = read_counts())) return rc;
        ahead = 3;
    }
    if (n <= SUB) host[CNT_SMALL] = 1;
    k_subtrees<<<(unsigned)host[CNT_SMALL], SUB, 0, st>>>(S);
    if ((rc = read_counts())) return rc;
    if (max_depth) *max_depth = host[CNT_DEPTH];
    return mt_scan_check(ctx);
}
