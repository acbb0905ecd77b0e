// Warp-field maintenance kernels (include/mvdr/warpfield.h): node graph,
// skinning, forward and inverse warps.
//
// The two searches scan the canonical nodes in index order (the slots of a
// result record the order of the insertions, so the order is part of it).
// Both skip most of them by boxes around 8 consecutive nodes (built by every
// workgroup): a box no nearer than the farthest result slot holds nothing that
// could be inserted.
//   vertices  : a thread per vertex.  A wave tests 64 boxes at a time against the
//               box of its vertices, a lane per box; the nodes of a box pass through
//               scalar registers (every lane looks at the same node; from LDS the
//               reads alone took as long as the arithmetic), asked for one box ahead.
//   nodes     : lanes of its own to a node, a lane per box and then per node of the
//               next near boxes; the few that beat the worst slot are inserted one after
//               another.  (A thread per node filled 16 workgroups of 256.)  The lanes of
//               a node repeat its insertions, so the more nodes, the fewer lanes each:
//               a wave or a row of 16 in the graph, a row or a thread, as the vertices,
//               in the skinning.
// Bound by the chain of insertions and the arithmetic around it (the memory traffic
// is 8 MB).  How many there are depends on the order of the nodes; the most are
// on a line that comes nearer, all of them.  us of a call, a thread per point -> here:
//   body scene, 159k surfels, 4018 nodes: skinning 431 -> 185, graph 796 -> 88
//     surfels in no order (their boxes exclude nothing) 533 -> 454, nodes in no order
//     364 -> 154 and 757 -> 53, both 368 -> 262
//   281k surfels in no order, 7500 nodes: skinning 1099 -> 1052
//   20k points in no order and nodes on a line, 600 / 1000 / 2000 / 4000 / 8192 / 65535 nodes:
//     skinning 87 / 143 / 284 / 556 / 1146 / 8988 -> 52 / 82 / 157 / 330 / 772 / 5931
//     graph 161 / 274 / 531 / 1069 / 2226 / 17970 -> 67 / 107 / 210 / 486 / 1345 / 17427
//
// The warps are streaming passes bound by HBM (a 16-32 B read and write per point plus
// the L2-resident warp-field gathers).
//
// Distances are evaluated without contraction except where the reference
// fuses explicitly (the skinning distance), so that they round like the
// oracle's.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "../../include/mvdr/warpfield.h"
#include "common.h"
#include "device_util.h"

namespace mvdr {
namespace {

constexpr uint32_t kBoxNodes = 8;       // nodes per box
constexpr uint32_t kBoxes = 512;        // boxes in LDS at a time (4096 nodes, 16 KB)
constexpr int kGraphNeighbours = 8;     // nodesGraphNeigboursNum
constexpr uint32_t graph_threads(uint32_t lanes) { return lanes == 64 ? 512 : 256; }  // per workgroup of the graph search

// Squared distances are compared by their bits: at least +0, they are ordered alike (a
// not-a-number comes last), and integer minima and maxima need no canonical operands.
__device__ inline uint32_t bits(float d) { return __float_as_uint(d); }

// The reference's 4-slot heap update (brute_foce_knn.cuh:17-39): slot x holds
// the current worst; a closer node replaces it and sifts once.  Minima, maxima and
// selects, no branches: the slots always form a heap (0 over 1 and 2, 1 over 3), so a
// node that is not closer leaves them as they are.
__device__ inline void heap_update(uint32_t d[4], uint32_t id[4], uint32_t idx, uint32_t dist) {
    const uint32_t m = dist < d[0] ? idx : id[0], n = min(dist, d[0]);
    const bool right = d[1] < d[2];
    const uint32_t c = max(d[1], d[2]), ic = right ? id[2] : id[1];
    const bool sift = n < c, to2 = sift & right, to1 = sift & !right;
    const uint32_t e = to1 ? n : d[1], ie = to1 ? m : id[1];  // at slot 1 before the look at slot 3
    const bool to3 = e < d[3];
    d[0] = max(n, c);
    id[0] = sift ? ic : m;
    d[2] = to2 ? n : d[2];
    id[2] = to2 ? m : id[2];
    d[1] = max(e, d[3]);
    id[1] = to3 ? id[3] : ie;
    d[3] = min(e, d[3]);
    id[3] = to3 ? ie : id[3];
}

// Maximum over each eight lanes, and over the wave (from lane 63, without LDS).
template <int kCtrl, int kRows = 0xF>
__device__ inline float dpp(float v) {
    return __uint_as_float(lane_dpp<kCtrl, kRows>(__float_as_uint(v), __float_as_uint(v)));
}
__device__ inline float wave_max(float v) {
    v = fmaxf(v, dpp<0xB1>(v));        // lane ^ 1
    v = fmaxf(v, dpp<0x4E>(v));        // lane ^ 2
    v = fmaxf(v, dpp<0x141>(v));       // the other four of eight
    v = fmaxf(v, dpp<0x140>(v));       // the other eight of a row
    v = fmaxf(v, dpp<0x142, 0xA>(v));  // rows 1 and 3: lane 15 of the row before
    v = fmaxf(v, dpp<0x143, 0xC>(v));  // rows 2 and 3: lane 31
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// The same for the bits of squared distances (one instruction a step).
template <int kCtrl, int kRows = 0xF>
__device__ inline uint32_t max_dpp(uint32_t v) {
    return max(v, lane_dpp<kCtrl, kRows>(v));
}
__device__ inline uint32_t eight_max(uint32_t v) { return max_dpp<0x141>(max_dpp<0x4E>(max_dpp<0xB1>(v))); }
__device__ inline uint32_t wave_max(uint32_t v) {
    v = max_dpp<0x143, 0xC>(max_dpp<0x142, 0xA>(max_dpp<0x140>(eight_max(v))));
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The boxes of nodes [base, base + n), n <= kBoxes * kBoxNodes, by the workgroup.
struct NodeBoxes {
    float4 lo[kBoxes], hi[kBoxes];
    __device__ void put(uint32_t, float4) {}
};
// The same of kTileNodes nodes at a time, and the nodes.
constexpr uint32_t kTileNodes = 1024;
struct NodeTile {
    float4 lo[kTileNodes / kBoxNodes], hi[kTileNodes / kBoxNodes], node[kTileNodes];
    __device__ void put(uint32_t k, float4 q) { node[k] = q; }
};
template <class Boxes>
__device__ inline uint32_t build_boxes(const float4* __restrict__ nodes, uint32_t base, uint32_t n, Boxes& x) {
    const uint32_t boxes = (n + kBoxNodes - 1) / kBoxNodes;
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < 2 * boxes; t += blockDim.x) {  // two lanes per box, four nodes each
        float4 l, h;
#pragma unroll
        for (uint32_t j = 0; j < kBoxNodes / 2; ++j) {
            const float4 q = nodes[base + min(t * (kBoxNodes / 2) + j, n - 1)];  // the last node repeats past the end
            x.put(t * (kBoxNodes / 2) + j, q);
            l = j == 0 ? q : make_float4(fminf(l.x, q.x), fminf(l.y, q.y), fminf(l.z, q.z), 0.f);
            h = j == 0 ? q : make_float4(fmaxf(h.x, q.x), fmaxf(h.y, q.y), fmaxf(h.z, q.z), 0.f);
        }
        l = make_float4(fminf(l.x, dpp<0xB1>(l.x)), fminf(l.y, dpp<0xB1>(l.y)), fminf(l.z, dpp<0xB1>(l.z)), 0.f);
        h = make_float4(fmaxf(h.x, dpp<0xB1>(h.x)), fmaxf(h.y, dpp<0xB1>(h.y)), fmaxf(h.z, dpp<0xB1>(h.z)), 0.f);
        if (t % 2 == 0)
            x.lo[t / 2] = l;
        else
            x.hi[t / 2] = h;
    }
    __syncthreads();
    return boxes;
}

// Eight nodes at a wave-uniform index in scalar registers (nothing writes the nodes
// during the call, so the constant address space may serve them).  Volatile: the
// compiler would move the loads down to their first use, and the wave would wait there.
typedef float float16 __attribute__((ext_vector_type(16), aligned(16)));
struct NodeGroup {
    float16 q[2];
    __device__ void load(const float4* nodes, uint32_t k) {
#if __HIP_DEVICE_COMPILE__
        const auto* p = (const volatile __attribute__((address_space(4))) float16*)(nodes + k);
        q[0] = p[0];
        q[1] = p[1];
#endif
    }
    __device__ float4 node(uint32_t j) const {
        const float16& h = q[j / 4];
        return make_float4(h[j % 4 * 4], h[j % 4 * 4 + 1], h[j % 4 * 4 + 2], 0.f);
    }
};

__device__ inline float skin_distance(float4 pt, float4 q) {
    const float dx = pt.x - q.x, dy = pt.y - q.y, dz = pt.z - q.z;
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}

// Squared distance of two boxes (a point is a box of no extent).
__device__ inline float box_distance(float4 alo, float4 ahi, float4 lo, float4 hi) {
    const float dx = fmaxf(fmaxf(lo.x - ahi.x, alo.x - hi.x), 0.f);
    const float dy = fmaxf(fmaxf(lo.y - ahi.y, alo.y - hi.y), 0.f);
    const float dz = fmaxf(fmaxf(lo.z - ahi.z, alo.z - hi.z), 0.f);
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}

// Whether a distance below d0 may hide behind a box distance.  Box distances and
// distances carry at most 5 roundings each way; 2e-6 below a box distance no
// distance can fall (above the denormal range).  Not-a-number answers true.
__device__ inline bool may_be_nearer(float box, float d0) { return !(box * 0.999998f >= d0 && box > 1e-30f); }

// Passes the nodes that may enter the slots of one point `me` (the wave's), in index
// order: a lane per box, then per node of the next eight near boxes.
//   slots.bound()             the farthest slot
//   slots.distance(me, q)     slots.wants(d): whether a distance may be inserted
//   slots.insert(k, d)        one node, k and d wave-uniform
template <class Slots>
__device__ inline void scan_for_point(const float4* __restrict__ nodes, uint32_t num_nodes, float4 me, NodeBoxes& box,
                                      Slots& slots) {
    const uint32_t lane = threadIdx.x & 63, part = lane / kBoxNodes;
    for (uint32_t base = 0; base < num_nodes; base += kBoxes * kBoxNodes) {
        const uint32_t boxes = build_boxes(nodes, base, min(kBoxes * kBoxNodes, num_nodes - base), box);
        for (uint32_t b0 = 0; b0 < boxes; b0 += 64) {
            const uint32_t mine = min(b0 + lane, boxes - 1);
            const float away = box_distance(me, me, box.lo[mine], box.hi[mine]);
            uint64_t left = b0 + 64 <= boxes ? ~0ull : (1ull << (boxes - b0)) - 1;  // boxes not yet passed
            for (;;) {
                // the next eight near boxes, one to eight lanes (a box passed over
                // is no nearer than the farthest slot, which only gets nearer)
                uint64_t near = left & __ballot(may_be_nearer(away, slots.bound()));
                if (!near) break;
                uint32_t x = 0xFFFFFFFFu, last = 0;
#pragma unroll
                for (uint32_t r = 0; r < 64 / kBoxNodes; ++r) {
                    if (near) {
                        last = (uint32_t)__builtin_ctzll(near);
                        near &= near - 1;
                        if (part == r) x = last;
                    }
                }
                left = last == 63 ? 0 : left & (~0ull << (last + 1));
                const uint32_t k = base + (b0 + x) * kBoxNodes + lane % kBoxNodes;
                const bool live = x != 0xFFFFFFFFu && k < num_nodes;
                const float d = slots.distance(me, nodes[live ? k : 0]);
                uint64_t hits = __ballot(live && slots.wants(d));
                while (hits) {
                    const int l = __builtin_ctzll(hits);
                    slots.insert((uint32_t)__builtin_amdgcn_readlane((int)k, l),
                                 __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d), l)));
                    // later hits that still beat the farthest slot
                    hits &= __ballot(d < slots.bound()) & (l == 63 ? 0ull : ~0ull << (l + 1));
                }
            }
        }
    }
}

// The value of lane j of each row of 16 lanes, in all of them, and their bits of a ballot.
template <uint32_t j>
__device__ inline float row_lane(float v) { return dpp<0x150 + j>(v); }
__device__ inline uint32_t row_bits(bool p) { return (uint32_t)(__ballot(p) >> (threadIdx.x & 48)) & 0xFFFFu; }

// Inserts where a row may have a hit: lane j's node is first + j for j < 8, second + j - 8 after.
template <uint32_t j = 0, class Slots>
__device__ inline void insert_hits(Slots& slots, uint32_t hits, uint32_t first, uint32_t second, float d) {
    if (hits & (1u << j)) slots.insert(j < kBoxNodes ? first + j : second + j - kBoxNodes, row_lane<j>(d));
    if constexpr (j < 15) insert_hits<j + 1>(slots, hits, first, second, d);
}

// Passes the nodes that may enter the slots of four points, one to each row of 16 lanes
// (`me`), in index order: a lane per box, then per node of the point's next two near boxes.
//   slots.bound()             the farthest slot
//   slots.distance(me, q)     slots.wants(d): whether a distance may be inserted
//   slots.insert(k, d)        node k at distance d, where wanted; equal in the row
template <class Slots>
__device__ inline void scan_for_row(const float4* __restrict__ nodes, uint32_t num_nodes, float4 me, NodeTile& tile,
                                    Slots& slots) {
    const uint32_t lane = threadIdx.x & 15;
    for (uint32_t base = 0; base < num_nodes; base += kTileNodes) {
        const uint32_t n = min(kTileNodes, num_nodes - base), boxes = build_boxes(nodes, base, n, tile);
        float4 lo = tile.lo[min(lane, boxes - 1)], hi = tile.hi[min(lane, boxes - 1)];
        for (uint32_t b0 = 0; b0 < boxes; b0 += 16) {
            const float away = box_distance(me, me, lo, hi);
            uint32_t near = row_bits(b0 + lane < boxes && may_be_nearer(away, slots.bound()));
            const uint32_t mine = min(b0 + 16 + lane, boxes - 1);  // the next step's box loads meanwhile
            lo = tile.lo[mine];
            hi = tile.hi[mine];
            while (__any(near != 0)) {
                const uint32_t rest = near & (near - 1);
                const uint32_t first = (b0 + (near ? (uint32_t)__builtin_ctz(near) : 0u)) * kBoxNodes;
                const uint32_t second = (b0 + (rest ? (uint32_t)__builtin_ctz(rest) : 0u)) * kBoxNodes;
                const uint32_t k = (lane < kBoxNodes ? first : second) + lane % kBoxNodes;
                const bool live = (lane < kBoxNodes ? near : rest) != 0 && k < n;
                near = rest & (rest - 1);
                const float4 q = tile.node[k];
                const float d = live ? slots.distance(me, q) : __int_as_float(0x7f800000);
                uint64_t hits = __ballot(slots.wants(d));
                if (!hits) continue;
                hits |= hits >> 32;
                hits |= hits >> 16;
                insert_hits(slots, (uint32_t)hits, base + first, base + second, d);
                // a box passed over is no nearer than the farthest slot, which only gets nearer
                near &= row_bits(may_be_nearer(away, slots.bound()));
            }
        }
    }
}

struct SkinSlots {
    uint32_t d[4], id[4] = {0, 0, 0, 0};
    __device__ SkinSlots() { d[0] = d[1] = d[2] = d[3] = bits(1e6f); }
    __device__ float bound() const { return __uint_as_float(d[0]); }
    __device__ static float distance(float4 pt, float4 q) { return skin_distance(pt, q); }
    __device__ bool wants(float dist) const { return bits(dist) < d[0]; }
    __device__ void insert(uint32_t k, float dist) { heap_update(d, id, k, bits(dist)); }
    // nodes k .. k + 8, each lane's point its own; whether any entered
    __device__ bool pass(float4 pt, const NodeGroup& g, uint32_t k) {
        uint32_t dist[kBoxNodes], nearest;
#pragma unroll
        for (uint32_t j = 0; j < kBoxNodes; ++j) {
            dist[j] = bits(skin_distance(pt, g.node(j)));
            nearest = j == 0 ? dist[0] : min(nearest, dist[j]);
        }
        if (!__any(nearest < d[0])) return false;
#pragma unroll
        for (uint32_t j = 0; j < kBoxNodes; ++j)
            if (__any(dist[j] < d[0])) heap_update(d, id, k + j, dist[j]);
        return true;
    }
};

// Weights of the four slots (skinningVertexAndNodeKernel).
__device__ inline void put_skin(float4 pt, const SkinSlots& slots, const float4* __restrict__ nodes, float radius,
                                ushort4* __restrict__ knn, float4* __restrict__ weight) {
    float w[4];
    const float den = (2.0f * radius) * radius;
    for (int s = 0; s < 4; ++s) {
        const float4 q = nodes[slots.id[s]];
        const float dx = pt.x - q.x, dy = pt.y - q.y, dz = pt.z - q.z;
        w[s] = expf(-(dx * dx + dy * dy + dz * dz) / den);
    }
    const float inv = 1.0f / (fabsf(w[0]) + fabsf(w[1]) + fabsf(w[2]) + fabsf(w[3]));
    *knn = make_ushort4(slots.id[0], slots.id[1], slots.id[2], slots.id[3]);
    *weight = make_float4(w[0] * inv, w[1] * inv, w[2] * inv, w[3] * inv);
}

constexpr uint32_t kSkinWaves = 4;  // waves per workgroup of the skinning

// 16 lanes to a node up to kSkinRowNodes, a thread above: 64 nodes in a row lie too far
// apart for boxes common to them, so lanes of its own serve a node better, until the
// insertions of all nodes fill the chip.  us; listed order / a line that comes nearer:
//   600 nodes   16 lanes  40 /   51, thread  54 /   60, wave  40 /   85
//   2000                 100 /  154,        121 /  183,      102 /  327
//   4000                 186 /  326,        194 /  361,      188 /  888
//   7500, 8192           312 /  766,        336 /  743,      323 / 2914
//   12000 (no order)     455 / 1285,        468 / 1073,      468 / 5842
constexpr uint32_t kNodeRow = 16, kNodeThread = 1;
constexpr uint32_t kSkinRowNodes = 8192;

// Workgroups of 256 vertices, then of nodes with lanes of their own; nodes by threads
// come first, as the longest waves (4018 nodes 202 us, last 216).
template <uint32_t kNodeLanes>
__global__ void __launch_bounds__(64 * kSkinWaves)
    skin_kernel(const float4* vertices, uint32_t num_vertices, const float4* nodes, uint32_t num_nodes, float radius,
                ushort4* vknn, float4* vw, ushort4* nknn, float4* nw) {
    __shared__ union {
        NodeBoxes box;
        NodeTile tile;
    } shared;
    NodeBoxes& box = shared.box;
    SkinSlots slots;
    const uint32_t vertex_blocks = (num_vertices + blockDim.x - 1) / blockDim.x, lane = threadIdx.x & 63;
    const uint32_t node_blocks = gridDim.x - vertex_blocks;
    const bool is_node = kNodeLanes == kNodeThread ? blockIdx.x < node_blocks : blockIdx.x >= vertex_blocks;
    uint32_t block = blockIdx.x;
    if (is_node != (kNodeLanes == kNodeThread)) block -= is_node ? vertex_blocks : node_blocks;
    if (kNodeLanes != kNodeThread && is_node) {
        const uint32_t i = (block * blockDim.x + threadIdx.x) / kNodeLanes;
        const float4 me = nodes[min(i, num_nodes - 1)];
        scan_for_row(nodes, num_nodes, me, shared.tile, slots);
        if (i < num_nodes && threadIdx.x % kNodeLanes == 0) put_skin(me, slots, nodes, radius, nknn + i, nw + i);
        return;
    }
    if (is_node) {  // as the vertices are
        vertices = nodes;
        num_vertices = num_nodes;
        vknn = nknn;
        vw = nw;
    }
    const uint32_t p = block * blockDim.x + threadIdx.x;
    const float4 pt = vertices[min(p, num_vertices - 1)];  // idle lanes repeat the last vertex
    const float4 whi = make_float4(wave_max(pt.x), wave_max(pt.y), wave_max(pt.z), 0.f);
    const float4 wlo = make_float4(-wave_max(-pt.x), -wave_max(-pt.y), -wave_max(-pt.z), 0.f);
    for (uint32_t base = 0; base < num_nodes; base += kBoxes * kBoxNodes) {
        const uint32_t n = min(kBoxes * kBoxNodes, num_nodes - base);
        build_boxes(nodes, base, n, box);
        const uint32_t whole = n / kBoxNodes;  // whole boxes; the rest comes last in any case
        for (uint32_t b0 = 0; b0 < whole; b0 += 64) {
            const uint32_t mine = min(b0 + lane, whole - 1);
            const float coarse = box_distance(wlo, whi, box.lo[mine], box.hi[mine]);
            uint64_t left = b0 + 64 <= whole ? ~0ull : (1ull << (whole - b0)) - 1;  // boxes not yet passed
            float worst = __uint_as_float(wave_max(slots.d[0]));  // the farthest fourth neighbour of the wave's points
            uint64_t near = left & __ballot(may_be_nearer(coarse, worst));
            if (!near) continue;
            uint32_t vain = 0;  // last looks at the boxes that excluded none
            const float4* first = nodes + base + b0 * kBoxNodes;
            uint32_t x = (uint32_t)__builtin_ctzll(near);
            NodeGroup here, next;
            here.load(first, x * kBoxNodes);
            for (;;) {
                // the next box's nodes are asked for before this one's are worked on
                left &= ~((2ull << x) - 1);
                near &= left;
                const uint32_t y = near ? (uint32_t)__builtin_ctzll(near) : x;
                next.load(first, y * kBoxNodes);
                if (slots.pass(pt, here, base + (b0 + x) * kBoxNodes) && vain < 4) {
                    // looked at again while that excludes boxes (points in no order: 1125 -> 1047 us)
                    worst = __uint_as_float(wave_max(slots.d[0]));
                    const uint64_t again = near & __ballot(may_be_nearer(coarse, worst));
                    vain = again == near ? vain + 1 : 0;
                    near = again;
                }
                if (y == x) break;
                x = y;
                here = next;
            }
        }
        for (uint32_t k = base + whole * kBoxNodes; k < base + n; ++k) slots.insert(k, skin_distance(pt, nodes[k]));
    }
    if (p < num_vertices) put_skin(pt, slots, nodes, radius, vknn + p, vw + p);
}

// BuildNodesGraphKernel: 8 slots, the worst replaced (WarpField.cu:15-59).  Lane j of
// the node's wave or row of 16 lanes holds slot j; the lanes from 8 on hold none.
template <uint32_t kLanes>
struct GraphSlots {
    float dist = threadIdx.x % kLanes < kGraphNeighbours ? 1e5f : 0.f;
    int idx = -1;
    float worst_d = 1e5f;
    uint32_t worst = 0;
    __device__ float bound() const { return worst_d; }
    __device__ static float distance(float4 me, float4 q) {
        return (me.x - q.x) * (me.x - q.x) + (me.y - q.y) * (me.y - q.y) + (me.z - q.z) * (me.z - q.z);
    }
    __device__ bool wants(float d) const { return d > 1e-6f && d < worst_d; }
    __device__ void insert(uint32_t k, float d) {
        // (the scan of a wave passes only wanted ones)
        if ((kLanes == 64 || wants(d)) && threadIdx.x % kLanes == worst) {
            dist = d;
            idx = (int)k;
        }
        // the new worst slot: the first of the largest
        const float m = __uint_as_float(eight_max(bits(dist)));
        if constexpr (kLanes == 64) {
            worst_d = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(m)));
            worst = (uint32_t)__builtin_ctzll(__ballot(dist == worst_d));
        } else {
            worst_d = row_lane<0>(m);
            worst = (uint32_t)__builtin_ctz(row_bits(dist == worst_d));
        }
    }
};

// A wave per node up to kGraphWaveNodes, 16 lanes above.  us; random order / a line that
// comes nearer: 4000 nodes 57 / 492 and 89 / 342, 8192 165 / 1379 and 161 / 740, 12000
// 317 / 2555 and 239 / 1172, 65535 7106 / 54884 and 3671 / 17515 (listed order: 7500
// nodes 161 and 204).  Workgroups of four waves with rows (of eight 159 / 779 at 8192).
constexpr uint32_t kGraphWaveNodes = 8192;
template <uint32_t kLanes>
__global__ void __launch_bounds__(graph_threads(kLanes))
    node_graph_kernel(const float4* __restrict__ nodes, uint32_t num_nodes, ushort2* __restrict__ graph) {
    const uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) / kLanes, lane = threadIdx.x % kLanes;
    const float4 me = nodes[min(i, num_nodes - 1)];
    GraphSlots<kLanes> slots;
    if constexpr (kLanes == 64) {
        __shared__ NodeBoxes box;
        scan_for_point(nodes, num_nodes, me, box, slots);
    } else {
        __shared__ NodeTile tile;
        scan_for_row(nodes, num_nodes, me, tile, slots);
    }
    if (i < num_nodes && lane < (uint32_t)kGraphNeighbours)
        graph[(size_t)i * kGraphNeighbours + lane] = make_ushort2((uint16_t)i, (uint16_t)slots.idx);
}

__device__ inline bool knn_in_range(ushort4 k, uint32_t n) { return k.x < n && k.y < n && k.z < n && k.w < n; }

// forwardWarpVertexAndNodeKernel: surfels (vertex, normal), then nodes.  A
// point whose knn names a node outside the field is copied unwarped.
__global__ void __launch_bounds__(256) forward_warp_kernel(const DQ* __restrict__ field, const float4* __restrict__ cv,
                                                           const float4* __restrict__ cn, const ushort4* __restrict__ vknn,
                                                           const float4* __restrict__ vw, uint32_t num_vertices,
                                                           const float4* __restrict__ nodes,
                                                           const ushort4* __restrict__ nknn,
                                                           const float4* __restrict__ nw, uint32_t num_nodes,
                                                           float4* __restrict__ lv, float4* __restrict__ ln,
                                                           float4* __restrict__ lnodes) {
    const uint32_t total = num_vertices + num_nodes;
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < total; p += gridDim.x * blockDim.x) {
        const bool is_vertex = p < num_vertices;
        const uint32_t o = is_vertex ? p : p - num_vertices;
        const float4 v = is_vertex ? cv[o] : nodes[o];
        const ushort4 k = is_vertex ? vknn[o] : nknn[o];
        const float4 w = is_vertex ? vw[o] : nw[o];
        float4 vo = v, no = is_vertex ? cn[o] : make_float4(0.f, 0.f, 0.f, 0.f);
        if (knn_in_range(k, num_nodes)) {
            const Mat34 T = se3_of(blend4(field, k, w));
            const f3 pv = T.apply(xyz(v));
            vo = make_float4(pv.x, pv.y, pv.z, v.w);
            if (is_vertex) {
                const f3 nv = T.rot(xyz(no));
                no = make_float4(nv.x, nv.y, nv.z, no.w);
            }
        }
        if (is_vertex) {
            lv[o] = vo;
            ln[o] = no;
        } else {
            lnodes[o] = vo;
        }
    }
}

// inverseWarpVertexNormalKernel (without the correction transform).
__global__ void __launch_bounds__(256) inverse_warp_kernel(const DQ* __restrict__ field, uint32_t field_nodes,
                                                           const float4* __restrict__ lv, const float4* __restrict__ ln,
                                                           const ushort4* __restrict__ vknn,
                                                           const float4* __restrict__ vw, uint32_t num_vertices,
                                                           float4* __restrict__ rv, float4* __restrict__ rn) {
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < num_vertices; p += gridDim.x * blockDim.x) {
        const float4 v = lv[p], n = ln[p];
        float4 vo = v, no = n;
        const ushort4 k = vknn[p];
        if (knn_in_range(k, field_nodes)) {
            const Mat34 T = se3_of(blend4(field, k, vw[p]));
            const f3 a = T.rot_t(mk(v.x - T.t.x, v.y - T.t.y, v.z - T.t.z));
            const f3 b = T.rot_t(xyz(n));
            vo = make_float4(a.x, a.y, a.z, v.w);
            no = make_float4(b.x, b.y, b.z, n.w);
        }
        rv[p] = vo;
        rn[p] = no;
    }
}

// --------------------------------------------- large-error node correction
constexpr uint32_t kCorrHalfWindow = 2;  // CorrSearchWindowHalfSize (NonRigidSolver.h:41)
constexpr float kNodeRadius = 0.025f;    // NODE_RADIUS (GlobalConfigs.h:85)

struct CorrViews {
    uint32_t V, W, H;
    float fx[kMaxViews], fy[kMaxViews], cx[kMaxViews], cy[kMaxViews];
    Mat34 w2c[kMaxViews], w2c_inv[kMaxViews], init[kMaxViews], init_inv[kMaxViews];
    const float4* prev[kMaxViews];
    const float* guided[kMaxViews];  // 12 floats per pixel: rotation columns, translation
    const uint8_t* valid[kMaxViews];
};

// mat34::operator* (MatUtils.h:449-455): a * b
__device__ inline Mat34 compose(const Mat34& a, const Mat34& b) {
    Mat34 o;
    o.c0 = a.rot(b.c0);
    o.c1 = a.rot(b.c1);
    o.c2 = a.rot(b.c2);
    o.t = a.rot(b.t) + a.t;
    return o;
}

__device__ inline Mat34 identity34() {
    Mat34 m;
    m.c0 = mk(1.f, 0.f, 0.f);
    m.c1 = mk(0.f, 1.f, 0.f);
    m.c2 = mk(0.f, 0.f, 1.f);
    m.t = mk(0.f, 0.f, 0.f);
    return m;
}

// decodeNodesCameraView (CommonUtils.h:110-117): v with v < w <= v + 1.
__device__ inline uint32_t node_view(float w) {
    for (uint32_t v = 0; v < (uint32_t)kMaxViews; ++v)
        if ((float)v < w && w <= (float)(v + 1)) return v;
    return 0xFFFFFFFFu;
}

// The pixel coordinate of the reference's projection: the expression is
// evaluated in double (its 1e-10 literal), converted to float and rounded to
// the nearest integer (ties to even); negative values give 0.
__device__ inline uint32_t pixel_of(float x, float z, float f, float c) {
    const float p = (float)(((double)x / ((double)z + 1e-10)) * (double)f + (double)c);
    if (!(p > 0.f)) return 0u;
    if (p >= 4294967040.f) return 0xFFFFFFFFu;
    return (uint32_t)rintf(p);
}

__device__ inline float4 qconj(float4 q) { return make_float4(-q.x, -q.y, -q.z, q.w); }

// Quaternion::pow (Quaternion.h:235-249)
__device__ inline float4 qpow(float4 q, float t) {
    const float n = sqrtf(q.x * q.x + q.y * q.y + q.z * q.z);
    const float nt = atan2f(n, q.w) * t;
    if (fabsf(n) < 1e-6f) return make_float4(0.f, 0.f, 0.f, cosf(nt));
    const float sc = sinf(nt) / n;
    return make_float4(q.x * sc, q.y * sc, q.z * sc, cosf(nt));
}

// DualQuaternion::operator*(float) (DualQuaternion.h:165-178): the screw
// scaled by t in [1e-10, 1].
__device__ inline DQ dq_scale(const DQ& d, float ratio) {
    float t = ratio;
    if (t > 1.0f) t = 1.0f;
    else if (t < 1e-10f) t = 1e-10f;
    const float4 r = qmul(d.q1, qconj(d.q0));
    const float4 q0s = qpow(d.q0, t);
    return DQ{q0s, qmul(make_float4(t * r.x, t * r.y, t * r.z, t * r.w), q0s)};
}

// DualQuaternion::operator*(DualQuaternion) (DualQuaternion.h:152-157)
__device__ inline DQ dq_mul(const DQ& a, const DQ& b) {
    const float4 u = qmul(a.q1, b.q0), v = qmul(a.q0, b.q1);
    return DQ{qmul(a.q0, b.q0), make_float4(u.x + v.x, u.y + v.y, u.z + v.z, u.w + v.w)};
}

// computeCorrespondenceGuidedNodesSE3 with computeSuitableCorrespondenceGuidedSe3
// (NonRigidSolver.cu:100-138, :155-167): 16 lanes per node for the 25 pixels of its 5 x 5
// window (columns outer); the nearest of the suitable pixels wins, the first of equals.
// Few nodes are bound by dependent reads (maps, transforms near enough, the winner's
// transform), many by the motion's arithmetic, which every lane of a node repeats.
// 100 / 4018 / 16000 / 65535 nodes 7.2 / 7.0 / 10.8 / 28.3 us; with 32 lanes 6.7 / 7.5 /
// 14.9 / 43.3, with 8 lanes 7.7 / 8.5 / 10.2 / 21.7; a thread per node 22.7 / 27.5 /
// 25.6 / 28.5.
constexpr uint32_t kCorrLanes = 16;
__global__ void __launch_bounds__(256) correction_kernel(CorrViews r, const float4* __restrict__ nodes,
                                                         const float* __restrict__ error, uint32_t num_nodes,
                                                         DQ* __restrict__ correction) {
    constexpr uint32_t kSide = 2 * kCorrHalfWindow + 1, kPixels = kSide * kSide;
    constexpr uint32_t kRounds = (kPixels + kCorrLanes - 1) / kCorrLanes;
    const uint32_t lane = threadIdx.x % kCorrLanes;
    for (uint32_t n = (blockIdx.x * blockDim.x + threadIdx.x) / kCorrLanes; n < num_nodes;
         n += gridDim.x * blockDim.x / kCorrLanes) {
        const float e = error[n];
        DQ out;
        out.q0 = make_float4(0.f, 0.f, 0.f, 1.f);
        out.q1 = make_float4(0.f, 0.f, 0.f, 0.f);
        const float4 node = nodes[n];
        const uint32_t v = node_view(node.w);
        if (e > 0.2f && v < r.V) {
            Mat34 sel = identity34();
            const f3 c = r.init_inv[v].apply(r.w2c[v].apply(xyz(node)));
            const uint32_t u = pixel_of(c.x, c.z, r.fx[v], r.cx[v]);
            const uint32_t y = pixel_of(c.y, c.z, r.fy[v], r.cy[v]);
            const bool room = r.W > 2 * kCorrHalfWindow && r.H > 2 * kCorrHalfWindow;  // the window fits the map
            if (room && !(u >= r.W - kCorrHalfWindow || u < kCorrHalfWindow || y >= r.H - kCorrHalfWindow ||
                          y < kCorrHalfWindow)) {
                // window pixel w is column w / 5, row w % 5
                auto offset = [&](uint32_t w) {
                    return (size_t)(y - kCorrHalfWindow + w % kSide) * r.W + (u - kCorrHalfWindow + w / kSide);
                };
                auto transform = [&](uint32_t w) {
                    const float* g = r.guided[v] + 12 * offset(w);
                    Mat34 G;
                    G.c0 = mk(g[0], g[1], g[2]);
                    G.c1 = mk(g[3], g[4], g[5]);
                    G.c2 = mk(g[6], g[7], g[8]);
                    G.t = mk(g[9], g[10], g[11]);
                    return G;
                };
                float4 pv[kRounds];
                uint8_t valid[kRounds];
#pragma unroll
                for (uint32_t k = 0; k < kRounds; ++k) {
                    const uint32_t w = min(lane + kCorrLanes * k, kPixels - 1);
                    pv[k] = r.prev[v][offset(w)];
                    valid[k] = lane + kCorrLanes * k < kPixels ? r.valid[v][offset(w)] : 0;
                }
                uint32_t best = 0xFFFFFFFFu, at = kPixels;  // squared distance (its bits) and place of a suitable pixel
#pragma unroll
                for (uint32_t k = 0; k < kRounds; ++k) {
                    const f3 d = c - xyz(pv[k]);
                    const float d2 = dot3(d, d);
                    if (valid[k] != 1 || is_zero_vertex(pv[k]) || !(d2 < 1e-4f)) continue;
                    const f3 m = transform(lane + kCorrLanes * k).apply(c) - c;
                    if (dot3(m, m) < 4 * (kNodeRadius * kNodeRadius) && __float_as_uint(d2) < best) {
                        best = __float_as_uint(d2);
                        at = lane + kCorrLanes * k;
                    }
                }
#pragma unroll
                for (uint32_t s = 1; s < kCorrLanes; s *= 2) {
                    const uint32_t d = (uint32_t)__shfl_xor((int)best, s, 64), w = (uint32_t)__shfl_xor((int)at, s, 64);
                    const bool take = d < best || (d == best && w < at);
                    best = take ? d : best;
                    at = take ? w : at;
                }
                if (at < kPixels) sel = transform(at);
                sel = compose(compose(compose(compose(r.w2c_inv[v], r.init[v]), sel), r.init_inv[v]), r.w2c[v]);
            }
            out = dq_scale(dq_from_mat34(sel), e);
        }
        if (lane == 0) correction[n] = out;
    }
}

// CorrectWarpVertexAndNodeKernel (NonRigidSolver.cu:170-216): surfels
// [0, S), then nodes; in place.
__global__ void __launch_bounds__(256) apply_correction_kernel(const DQ* __restrict__ correction, uint32_t num_nodes,
                                                               float4* __restrict__ lv, float4* __restrict__ ln,
                                                               const ushort4* __restrict__ sknn,
                                                               const float4* __restrict__ sw, uint32_t num_surfels,
                                                               float4* __restrict__ lnodes, DQ* __restrict__ node_se3,
                                                               const ushort4* __restrict__ nknn,
                                                               const float4* __restrict__ nw) {
    const uint32_t total = num_surfels + num_nodes;
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < total; p += gridDim.x * blockDim.x) {
        const bool surfel = p < num_surfels;
        const uint32_t o = surfel ? p : p - num_surfels;
        const ushort4 k = surfel ? sknn[o] : nknn[o];
        if (!knn_in_range(k, num_nodes)) continue;
        const DQ avg = blend4(correction, k, surfel ? sw[o] : nw[o]);
        const Mat34 T = se3_of(avg);
        const float4 v = surfel ? lv[o] : lnodes[o];
        const f3 pv = T.apply(xyz(v));
        if (surfel) {
            const float4 n = ln[o];
            const f3 pn = T.rot(xyz(n));
            lv[o] = make_float4(pv.x, pv.y, pv.z, v.w);
            ln[o] = make_float4(pn.x, pn.y, pn.z, n.w);
        } else {
            lnodes[o] = make_float4(pv.x, pv.y, pv.z, v.w);
            node_se3[o] = dq_mul(avg, node_se3[o]);
        }
    }
}

uint32_t stream_grid(uint32_t n) { return std::max<uint32_t>(1, std::min<uint32_t>((n + 255) / 256, 4096u)); }

}  // namespace
}  // namespace mvdr

using namespace mvdr;

extern "C" {

mvdr_status mvdr_warp_build_node_graph(const void* nodes, uint32_t num_nodes, void* graph, void* stream) {
    if (num_nodes == 0) return MVDR_OK;
    if (!nodes || !graph) return MVDR_E_INVALID;
    if (num_nodes > 65535) return MVDR_E_SHAPE;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const float4* n = static_cast<const float4*>(nodes);
    ushort2* g = static_cast<ushort2*>(graph);
    const uint32_t lanes = num_nodes <= kGraphWaveNodes ? 64 : 16, threads = graph_threads(lanes);
    const dim3 grid((num_nodes + threads / lanes - 1) / (threads / lanes)), wg(threads);
    if (lanes == 64) hipLaunchKernelGGL(node_graph_kernel<64>, grid, wg, 0, st, n, num_nodes, g);
    else hipLaunchKernelGGL(node_graph_kernel<16>, grid, wg, 0, st, n, num_nodes, g);
    return hipGetLastError() == hipSuccess ? MVDR_OK : MVDR_E_HIP;
}

mvdr_status mvdr_warp_skin(const void* vertices, uint32_t num_vertices, const void* nodes, uint32_t num_nodes,
                           float node_radius, void* vknn, void* vw, void* nknn, void* nw, void* stream) {
    if (num_nodes == 0 || !nodes || !(node_radius > 0.f)) return MVDR_E_INVALID;
    if (num_nodes > 65535) return MVDR_E_SHAPE;
    if (num_vertices && (!vertices || !vknn || !vw)) return MVDR_E_INVALID;
    if (!nknn || !nw) return MVDR_E_INVALID;
    const uint64_t total = (uint64_t)num_vertices + num_nodes;
    if (total > 0xFFFFFFFFull - 255) return MVDR_E_SHAPE;
    constexpr uint32_t kSkinThreads = 64 * kSkinWaves;
    const bool row = num_nodes <= kSkinRowNodes;
    const uint32_t per = kSkinThreads / (row ? kNodeRow : kNodeThread);  // nodes per workgroup
    const dim3 grid((num_vertices + kSkinThreads - 1) / kSkinThreads + (num_nodes + per - 1) / per);
    auto* kernel = row ? skin_kernel<kNodeRow> : skin_kernel<kNodeThread>;
    hipLaunchKernelGGL(kernel, grid, dim3(kSkinThreads), 0, static_cast<hipStream_t>(stream),
                       static_cast<const float4*>(vertices), num_vertices, static_cast<const float4*>(nodes), num_nodes,
                       node_radius, static_cast<ushort4*>(vknn), static_cast<float4*>(vw), static_cast<ushort4*>(nknn),
                       static_cast<float4*>(nw));
    return hipGetLastError() == hipSuccess ? MVDR_OK : MVDR_E_HIP;
}

mvdr_status mvdr_warp_forward(const void* node_se3, const void* cv, const void* cn, const void* vknn, const void* vw,
                              uint32_t num_vertices, const void* nodes, const void* nknn, const void* nw,
                              uint32_t num_nodes, void* lv, void* ln, void* lnodes, void* stream) {
    if (!node_se3 || num_nodes == 0) return MVDR_E_INVALID;
    if (num_vertices && (!cv || !cn || !vknn || !vw || !lv || !ln)) return MVDR_E_INVALID;
    if (!nodes || !nknn || !nw || !lnodes) return MVDR_E_INVALID;
    if (num_nodes > 65535) return MVDR_E_SHAPE;
    const uint64_t total = (uint64_t)num_vertices + num_nodes;
    if (total > 0xFFFFFFFFull) return MVDR_E_SHAPE;
    hipLaunchKernelGGL(forward_warp_kernel, dim3(stream_grid((uint32_t)total)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), static_cast<const DQ*>(node_se3),
                       static_cast<const float4*>(cv), static_cast<const float4*>(cn), static_cast<const ushort4*>(vknn),
                       static_cast<const float4*>(vw), num_vertices, static_cast<const float4*>(nodes),
                       static_cast<const ushort4*>(nknn), static_cast<const float4*>(nw), num_nodes,
                       static_cast<float4*>(lv), static_cast<float4*>(ln), static_cast<float4*>(lnodes));
    return hipGetLastError() == hipSuccess ? MVDR_OK : MVDR_E_HIP;
}

mvdr_status mvdr_warp_inverse(const void* node_se3, uint32_t num_nodes, const void* lv, const void* ln,
                              const void* vknn, const void* vw, uint32_t num_vertices, void* rv, void* rn,
                              void* stream) {
    if (num_vertices == 0) return MVDR_OK;
    if (!node_se3 || num_nodes == 0 || !lv || !ln || !vknn || !vw || !rv || !rn) return MVDR_E_INVALID;
    if (num_nodes > 65535) return MVDR_E_SHAPE;
    hipLaunchKernelGGL(inverse_warp_kernel, dim3(stream_grid(num_vertices)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), static_cast<const DQ*>(node_se3), num_nodes,
                       static_cast<const float4*>(lv), static_cast<const float4*>(ln),
                       static_cast<const ushort4*>(vknn), static_cast<const float4*>(vw), num_vertices,
                       static_cast<float4*>(rv), static_cast<float4*>(rn));
    return hipGetLastError() == hipSuccess ? MVDR_OK : MVDR_E_HIP;
}

mvdr_status mvdr_warp_correct_nodes(const mvdr_node_correction* in, void* stream) {
    if (!in) return MVDR_E_INVALID;
    if (in->num_views < 1 || in->num_views > MVDR_MAX_VIEWS || in->width < 1 || in->height < 1 ||
        in->width > 65535 || in->height > 65535 || in->num_nodes > 65535)
        return MVDR_E_SHAPE;
    if (in->num_nodes == 0) return MVDR_OK;
    if (!in->node_error || !in->live_nodes || !in->node_se3 || !in->node_knn || !in->node_knn_weight || !in->correction)
        return MVDR_E_INVALID;
    if (in->num_surfels && (!in->live_vertex || !in->live_normal || !in->surfel_knn || !in->surfel_knn_weight))
        return MVDR_E_INVALID;
    if ((uint64_t)in->num_surfels + in->num_nodes > 0xFFFFFFFFull) return MVDR_E_SHAPE;
    CorrViews r;
    std::memset(&r, 0, sizeof(r));
    r.V = in->num_views;
    r.W = in->width;
    r.H = in->height;
    for (uint32_t v = 0; v < r.V; ++v) {
        if (!in->previous_vertex[v] || !in->guided_se3[v] || !in->guided_valid[v]) return MVDR_E_INVALID;
        r.fx[v] = in->intrinsic[v].fx;
        r.fy[v] = in->intrinsic[v].fy;
        r.cx[v] = in->intrinsic[v].cx;
        r.cy[v] = in->intrinsic[v].cy;
        r.w2c[v] = to_mat34(in->world2camera[v]);
        r.init[v] = to_mat34(in->initial_camera_se3[v]);
        r.w2c_inv[v] = inverse(r.w2c[v]);
        r.init_inv[v] = inverse(r.init[v]);
        r.prev[v] = static_cast<const float4*>(in->previous_vertex[v]);
        r.guided[v] = static_cast<const float*>(in->guided_se3[v]);
        r.valid[v] = static_cast<const uint8_t*>(in->guided_valid[v]);
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    constexpr uint32_t kCorrNodes = 256 / kCorrLanes;  // per workgroup
    hipLaunchKernelGGL(correction_kernel, dim3((in->num_nodes + kCorrNodes - 1) / kCorrNodes), dim3(256), 0, st, r,
                       static_cast<const float4*>(in->live_nodes), static_cast<const float*>(in->node_error),
                       in->num_nodes, static_cast<DQ*>(in->correction));
    hipLaunchKernelGGL(apply_correction_kernel, dim3(stream_grid(in->num_surfels + in->num_nodes)), dim3(256), 0, st,
                       static_cast<const DQ*>(in->correction), in->num_nodes, static_cast<float4*>(in->live_vertex),
                       static_cast<float4*>(in->live_normal), static_cast<const ushort4*>(in->surfel_knn),
                       static_cast<const float4*>(in->surfel_knn_weight), in->num_surfels,
                       static_cast<float4*>(in->live_nodes), static_cast<DQ*>(in->node_se3),
                       static_cast<const ushort4*>(in->node_knn), static_cast<const float4*>(in->node_knn_weight));
    return hipGetLastError() == hipSuccess ? MVDR_OK : MVDR_E_HIP;
}

}  // extern "C"
