// Cross-view edge pair production (include/mvdr/crossview.h): candidates by a
// windowed nearest-vertex search into the neighbouring views, one-to-one
// pairs by a per-target minimum, the back-traced subset, and in-order
// compaction of the three lists.  Reconstructs
// core/CrossViewEdgeCorrespondence/CrossViewEdgeCorrespondence.h:21-224
// (header only in the reference).
//
// Edge pixels are ~1 % of the V x H x W grid and each looks at a few hundred
// window taps in two views.  A first pass streams the edge masks (one byte per
// pixel, the only array read whole) and appends the edge pixels to a list; then
// a wave takes one listed pixel at a time, its lanes the window's taps (the
// nearest tap by a minimum of (squared-distance bits, scan position), which is
// the first strict minimum of the scan).  With one thread per pixel the few
// edge pixels of a wave walked 2 x 441 taps each in a chain, at one or two
// active lanes: 493 us for three 640x480 views, 17 us now (all passes 525 -> 49 us).
// With many edges the taps' arithmetic bounds it: the pixel and its views are the
// wave's (scalars), a tap's place follows from the last one's by additions, and a
// window inside the image needs no bounds.  A frame of almost nothing but edge pixels
// takes a thread per pixel again.  All passes, 2 / 10 / 50 / 100 % edge pixels of three
// 640x480 views, every second tap: 70 / 192 / 780 / 909 us (by waves alone 1560); a
// division per tap and addresses per lane 87 / 297 / 1291 / 2442; a thread per pixel
// throughout 636 / 1135 / 1485 / 1433.
// The list's order is arbitrary and no result depends on it: candidates and the
// per-target 64-bit minimum (squared-distance bits << 32 | source pixel) are kept
// per pixel, and the three lists are compacted in pixel order.
//
// Selection arithmetic (transforms, projection, distances) is evaluated
// without FMA contraction so that it rounds exactly like the oracle's.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <type_traits>

#include "../../include/mvdr/crossview.h"
#include "common.h"
#include "crossview_tiles.h"
#include "device_util.h"

namespace mvdr {
namespace {

constexpr uint32_t kCvWaves = kCvThreads / 64;
constexpr uint32_t kCvLists = 3;
constexpr uint32_t kNoCandidate = 0xFFFFFFFFu;

struct CvFrame {
    uint32_t V, W, H;
    float fx[kMaxViews], fy[kMaxViews], cx[kMaxViews], cy[kMaxViews];
    Mat34 init[kMaxViews], init_inv[kMaxViews];
    const float4* vertex[kMaxViews];
    const uint8_t* edge[kMaxViews];
    const ushort4* corr[kMaxViews];
};

struct CvBuffers {
    // cand and best are kept (cleared, written, read) at edge pixels alone
    uint2* cand;                 // per source pixel: (x2 | y2 << 16, view2) or (kNoCandidate, 0)
    unsigned long long* best;    // per target pixel: min (dist2 bits << 32 | source pixel)
    uint32_t* edges;             // the edge pixels, in any order
    uint32_t* num_edges;         // zero between calls
    uint32_t cap_edges;          // pixels the buffers were sized for
    uint8_t* flags;              // per source pixel: 1 candidate, 2 unique, 4 back-traced
    uint32_t* tile_count;        // kCvLists x tiles
    uint32_t* tile_offset;       // kCvLists x tiles
    uint32_t* counts;            // kCvLists totals (untruncated), in host memory
    mvdr_cross_pair* out[kCvLists];
    uint32_t max_pairs;
    int radius, step, track;
    float max_d2;
};

__device__ inline bool zero_vertex(float4 v) { return fabsf(v.x) < 1e-3f && fabsf(v.y) < 1e-3f && fabsf(v.z) < 1e-3f; }

// Edge pixel (x, y) of view v with a vertex there (in bounds by the caller).
__device__ inline bool edge_vertex(const CvFrame& f, uint32_t v, uint32_t o, float4& vert) {
    vert = f.vertex[v][o];
    return !zero_vertex(vert);
}

// The edge-mask bytes of the calling thread's kCvRounds pixels of a tile.
__device__ inline void tile_edges(const CvFrame& f, uint32_t base, uint8_t (&e)[kCvRounds]) {
    const uint32_t plane = f.W * f.H, pixels = f.V * plane;
#pragma unroll
    for (uint32_t k = 0; k < kCvRounds; ++k) {
        const uint32_t p = base + k * kCvThreads + threadIdx.x;
        e[k] = 0;
        if (p < pixels) {
            const uint32_t v = p / plane;
            e[k] = f.edge[v][p - v * plane];
        }
    }
}

// The listed edge pixels with their candidates and minima cleared, and the flags
// and tile counts of all pixels; one counter update per workgroup (one per wave and
// round took 50 us, all on one address).
__global__ void __launch_bounds__(kCvThreads) cv_edges_kernel(CvFrame f, CvBuffers b, uint32_t tiles) {
    const uint32_t pixels = f.V * f.W * f.H, base = blockIdx.x * kCvTile;
    const uint32_t wave = threadIdx.x >> 6;
    uint8_t e[kCvRounds];
    tile_edges(f, base, e);
    if (threadIdx.x < kCvLists) b.tile_count[threadIdx.x * tiles + blockIdx.x] = 0;
#pragma unroll
    for (uint32_t k = 0; k < kCvRounds; ++k) {
        const uint32_t p = base + k * kCvThreads + threadIdx.x;
        if (p < pixels) b.flags[p] = 0;
    }
    __shared__ uint32_t wave_cnt[kCvWaves], first;
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t k = 0; k < kCvRounds; ++k) mine += (uint32_t)__popcll(__ballot(e[k] == 1));
    if ((threadIdx.x & 63) == 0) wave_cnt[wave] = mine;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t total = 0;
        for (uint32_t w = 0; w < kCvWaves; ++w) total += wave_cnt[w];
        first = total ? atomicAdd(b.num_edges, total) : 0u;
    }
    __syncthreads();
    uint32_t at = first;
    for (uint32_t w = 0; w < wave; ++w) at += wave_cnt[w];
#pragma unroll
    for (uint32_t k = 0; k < kCvRounds; ++k) {
        const uint64_t mask = __ballot(e[k] == 1);
        if (e[k] == 1) {
            const uint32_t p = base + k * kCvThreads + threadIdx.x, i = at + lane_prefix(mask);
            if (i < b.cap_edges) b.edges[i] = p;
            b.cand[p] = make_uint2(kNoCandidate, 0u);
            b.best[p] = ~0ull;
        }
        at += (uint32_t)__popcll(mask);
    }
}

// Nearest edge vertex of view n to camera-n point q in the sampled window
// around q's projection, over the wave: its squared distance (or +inf) and
// pixel, in every lane.
__device__ inline float nearest_in_view(const CvFrame& f, const CvBuffers& b, uint32_t n, f3 q, uint32_t& bx, uint32_t& by) {
    const float inf = __int_as_float(0x7f800000);
    float best = inf;
    uint32_t at = 0xFFFFFFFFu;
    bx = by = 0;
    if (!(q.z > 0.f)) return best;
    const uint32_t side = 2 * (uint32_t)b.radius / (uint32_t)b.step + 1, taps = side * side;
    const uint32_t x0 = (uint32_t)project_round<float>(q.x, q.z, f.fx[n], f.cx[n]) - (uint32_t)b.radius;
    const uint32_t y0 = (uint32_t)project_round<float>(q.y, q.z, f.fy[n], f.cy[n]) - (uint32_t)b.radius;
    const uint32_t lane = threadIdx.x & 63;
    // tap t is the window's (t / side, t % side); 64 taps on by two additions
    const uint32_t rows = 64 / side, columns = 64 - rows * side;
    uint32_t iy = lane / side, ix = lane - iy * side;
    constexpr uint32_t kTaps = 4;  // a lane's taps in flight
    const uint8_t* edge = f.edge[n];
    const float4* vertex = f.vertex[n];
    auto scan = [&](auto inside) {
        for (uint32_t t0 = lane; t0 < taps; t0 += 64 * kTaps) {
            uint32_t o[kTaps];
            uint8_t e[kTaps];
            float4 v[kTaps];
#pragma unroll
            for (uint32_t k = 0; k < kTaps; ++k) {
                const uint32_t x = x0 + ix * (uint32_t)b.step, y = y0 + iy * (uint32_t)b.step;
                // negative coordinates wrap above both sizes
                const bool in = t0 + 64 * k < taps && (decltype(inside)::value || (x < f.W && y < f.H));
                o[k] = in ? y * f.W + x : 0u;
                e[k] = in ? edge[o[k]] : 0;
                const uint32_t next = ix + columns;
                ix = next < side ? next : next - side;
                iy += next < side ? rows : rows + 1;
            }
#pragma unroll
            for (uint32_t k = 0; k < kTaps; ++k) {
                v[k] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (e[k] == 1) v[k] = vertex[o[k]];
            }
#pragma unroll
            for (uint32_t k = 0; k < kTaps; ++k) {
                const float dx = v[k].x - q.x, dy = v[k].y - q.y, dz = v[k].z - q.z;
                const float d2 = dx * dx + dy * dy + dz * dz;
                const bool nearer = !zero_vertex(v[k]) && d2 < best;
                best = nearer ? d2 : best;
                at = nearer ? t0 + 64 * k : at;
            }
        }
    };
    const uint32_t last = (side - 1) * (uint32_t)b.step;
    if (x0 < f.W && y0 < f.H && last < f.W - x0 && last < f.H - y0) scan(std::true_type{});
    else scan(std::false_type{});
    // the smallest distance, and of equal ones the first in the scan
    unsigned long long key = ((unsigned long long)__float_as_uint(best) << 32) | at;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const unsigned long long u = __shfl_xor(key, s, 64);
        key = u < key ? u : key;
    }
    best = __uint_as_float((uint32_t)(key >> 32));
    at = (uint32_t)key;
    if (at != 0xFFFFFFFFu) {
        const uint32_t row = at / side;
        bx = x0 + (at - row * side) * (uint32_t)b.step;
        by = y0 + row * (uint32_t)b.step;
    }
    return best;
}

// The same by one thread for a frame of mostly edge pixels: the taps of neighbouring
// threads lie side by side, a wave's taps `step` apart.
__device__ inline float nearest_by_thread(const CvFrame& f, const CvBuffers& b, uint32_t n, f3 q, uint32_t& bx, uint32_t& by) {
    float best = __int_as_float(0x7f800000);
    bx = by = 0;
    if (!(q.z > 0.f)) return best;
    const uint32_t side = 2 * (uint32_t)b.radius / (uint32_t)b.step + 1;
    const uint32_t x0 = (uint32_t)project_round<float>(q.x, q.z, f.fx[n], f.cx[n]) - (uint32_t)b.radius;
    const uint32_t y0 = (uint32_t)project_round<float>(q.y, q.z, f.fy[n], f.cy[n]) - (uint32_t)b.radius;
    const uint8_t* edge = f.edge[n];
    const float4* vertex = f.vertex[n];
    for (uint32_t iy = 0, y = y0; iy < side; ++iy, y += (uint32_t)b.step)
        for (uint32_t ix = 0, x = x0; ix < side; ++ix, x += (uint32_t)b.step) {
            if (x >= f.W || y >= f.H || edge[y * f.W + x] != 1) continue;  // negative coordinates wrap above both sizes
            const float4 v = vertex[y * f.W + x];
            if (zero_vertex(v)) continue;
            const float dx = v.x - q.x, dy = v.y - q.y, dz = v.z - q.z;
            const float d2 = dx * dx + dy * dy + dz * dz;
            if (d2 < best) {
                best = d2;
                bx = x;
                by = y;
            }
        }
    return best;
}

// The candidate of source pixel p (at vertex src of view v) and the per-target minimum.
template <bool kWave>
__device__ inline void find_candidate(const CvFrame& f, const CvBuffers& b, uint32_t p) {
    const uint32_t plane = f.W * f.H, v = p / plane;
    float4 src;
    if (f.V < 2 || v >= f.V || !edge_vertex(f, v, p - v * plane, src)) return;
    const f3 world = f.init[v].apply(xyz(src));
    float best = __int_as_float(0x7f800000);
    uint2 cand = make_uint2(kNoCandidate, 0u);
    const uint32_t next = (v + 1) % f.V, last = (v + f.V - 1) % f.V;
    for (int k = 0; k < 2; ++k) {
        const uint32_t n = k == 0 ? next : last;
        if (k == 1 && last == next) break;
        uint32_t bx, by;
        const f3 q = f.init_inv[n].apply(world);
        const float d2 = kWave ? nearest_in_view(f, b, n, q, bx, by) : nearest_by_thread(f, b, n, q, bx, by);
        if (d2 < best) {
            best = d2;
            cand = make_uint2(bx | (by << 16), n);
        }
    }
    if (!(best < b.max_d2)) return;
    if (!kWave || (threadIdx.x & 63) == 0) {
        b.cand[p] = cand;
        const uint32_t t = cand.y * plane + (cand.x >> 16) * f.W + (cand.x & 0xFFFF);
        atomicMin(&b.best[t], ((unsigned long long)__float_as_uint(best) << 32) | p);
    }
}

// Stage 1: one candidate per edge pixel, one wave each from the list; where more than
// 7/8 of the pixels are edges, a thread per pixel of the frame (100 %: 909 us against
// 1560 with every second tap, 3230 against 3773 with every tap, where the two meet at
// about 85 %; 70 % by waves 1080 and 2640).  Eight waves to a SIMD: left to itself the
// compiler gives the two paths other registers, and 2 % edges take 75 us in place of 70.
__global__ void __launch_bounds__(kCvThreads, 8) cv_candidates_kernel(CvFrame f, CvBuffers b) {
    const uint32_t count = min(*b.num_edges, b.cap_edges), pixels = f.V * f.W * f.H;
    if (count > pixels - pixels / 8) {
        uint32_t p = blockIdx.x * kCvThreads + threadIdx.x;
        if (p >= pixels) return;
        do {
            const uint32_t v = p / (f.W * f.H);
            if (f.edge[v][p - v * (f.W * f.H)] == 1) find_candidate<false>(f, b, p);
        } while (cv_step(p, gridDim.x * kCvThreads, pixels));
        return;
    }
    const uint32_t waves = gridDim.x * (kCvThreads / 64);
    uint32_t w = blockIdx.x * (kCvThreads / 64) + (threadIdx.x >> 6);
    if (w >= count) return;
    do {
        find_candidate<true>(f, b, (uint32_t)__builtin_amdgcn_readfirstlane((int)b.edges[w]));
    } while (cv_step(w, waves, count));
}

__device__ inline uint32_t target_of(const CvFrame& f, uint2 c) {
    return c.y * f.W * f.H + (c.x >> 16) * f.W + (c.x & 0xFFFF);
}

// An optical-flow correspondence ends within the track window around (x, y).
__device__ inline bool traceable(const CvFrame& f, const CvBuffers& b, uint32_t v, int x, int y) {
    const ushort4* m = f.corr[v];
    if (!m) return false;
    for (int yy = y - b.track; yy <= y + b.track; ++yy)
        for (int xx = x - b.track; xx <= x + b.track; ++xx) {
            if (xx < 0 || yy < 0 || xx >= (int)f.W || yy >= (int)f.H) continue;
            const ushort4 e = m[(size_t)yy * f.W + xx];
            if (e.z == (uint32_t)xx && e.w == (uint32_t)yy) return true;
        }
    return false;
}

// Stage 2 + 3 flags of source pixel p with candidate c.
__device__ inline uint32_t pair_flags(const CvFrame& f, const CvBuffers& b, uint32_t p, uint2 c) {
    if (c.x == kNoCandidate) return 0;
    const uint32_t t = target_of(f, c);
    bool unique = (uint32_t)(b.best[t] & 0xFFFFFFFFull) == p;
    if (unique && t < p) {
        // the reverse pair t -> p kept as well: it stays from the lower source pixel
        const uint2 r = b.cand[t];
        if (r.x != kNoCandidate && target_of(f, r) == p && (uint32_t)(b.best[p] & 0xFFFFFFFFull) == t) unique = false;
    }
    if (!unique) return 1;
    const uint32_t plane = f.W * f.H, v = p / plane, o = p - v * plane;
    if (traceable(f, b, v, (int)(o % f.W), (int)(o / f.W)) && traceable(f, b, c.y, (int)(c.x & 0xFFFF), (int)(c.x >> 16)))
        return 7;
    return 3;
}

// Flags of the listed edge pixels, and the tiles' counts of the three lists: a
// wave's pixels mostly share a tile, so it adds once per tile it meets.
__global__ void __launch_bounds__(kCvThreads) cv_flags_kernel(CvFrame f, CvBuffers b, uint32_t tiles) {
    const uint32_t count = min(*b.num_edges, b.cap_edges), pixels = f.V * f.W * f.H;
    uint32_t base = blockIdx.x * kCvThreads;
    if (base >= count) return;
    do {
        const uint32_t i = base + threadIdx.x;
        uint32_t tile = 0xFFFFFFFFu, flag = 0;
        const uint32_t p = i < count ? b.edges[i] : pixels;
        if (p < pixels) {
            flag = pair_flags(f, b, p, b.cand[p]);
            b.flags[p] = (uint8_t)flag;
            tile = p / kCvTile;
        }
        uint64_t left = __ballot(flag != 0);
        while (left) {
            const int leader = __builtin_ctzll(left);
            const uint32_t t = (uint32_t)__shfl((int)tile, leader, 64);
            const bool mine = flag != 0 && tile == t;
#pragma unroll
            for (uint32_t l = 0; l < kCvLists; ++l) {
                const uint32_t n = (uint32_t)__popcll(__ballot(mine && ((flag >> l) & 1u)));
                if ((int)(threadIdx.x & 63) == leader && n) atomicAdd(&b.tile_count[l * tiles + t], n);
            }
            left &= ~__ballot(mine);
        }
    } while (cv_step(base, gridDim.x * kCvThreads, count));
}

__global__ void __launch_bounds__(1024) cv_scan_kernel(CvBuffers b, uint32_t tiles) {
    for (uint32_t l = 0; l < kCvLists; ++l) {
        const uint32_t total = block_exclusive_scan_1024(b.tile_count + l * tiles, b.tile_offset + l * tiles, tiles);
        if (threadIdx.x == 0) b.counts[l] = total;
    }
    if (threadIdx.x == 0) *b.num_edges = 0;  // the next call's list starts empty
}

// The lists in source-pixel order: a tile's rounds in turn, waves and lanes
// within a round; every round's positions from one exchange of counts.
__global__ void __launch_bounds__(kCvThreads) cv_scatter_kernel(CvFrame f, CvBuffers b, uint32_t tiles) {
    const uint32_t plane = f.W * f.H, pixels = f.V * plane, base = blockIdx.x * kCvTile;
    const uint32_t wave = threadIdx.x >> 6;
    uint32_t flag[kCvRounds];
#pragma unroll
    for (uint32_t k = 0; k < kCvRounds; ++k) {
        const uint32_t p = base + k * kCvThreads + threadIdx.x;
        flag[k] = p < pixels ? b.flags[p] : 0u;
    }
    __shared__ uint32_t wave_cnt[kCvRounds][kCvLists][kCvWaves];
#pragma unroll
    for (uint32_t k = 0; k < kCvRounds; ++k)
#pragma unroll
        for (uint32_t l = 0; l < kCvLists; ++l) {
            const uint64_t mask = __ballot((flag[k] >> l) & 1u);
            if ((threadIdx.x & 63) == 0) wave_cnt[k][l][wave] = (uint32_t)__popcll(mask);
        }
    __syncthreads();
    uint32_t dst[kCvLists];
#pragma unroll
    for (uint32_t l = 0; l < kCvLists; ++l) dst[l] = b.tile_offset[l * tiles + blockIdx.x];
#pragma unroll
    for (uint32_t k = 0; k < kCvRounds; ++k) {
        const uint32_t p = base + k * kCvThreads + threadIdx.x;
        mvdr_cross_pair rec;
        if (flag[k]) {
            const uint2 c = b.cand[p];
            const uint32_t v = p / plane, o = p - v * plane;
            rec.pixel[0] = (uint16_t)(o % f.W);
            rec.pixel[1] = (uint16_t)(o / f.W);
            rec.pixel[2] = (uint16_t)(c.x & 0xFFFF);
            rec.pixel[3] = (uint16_t)(c.x >> 16);
            rec.view[0] = (uint16_t)v;
            rec.view[1] = (uint16_t)c.y;
        }
#pragma unroll
        for (uint32_t l = 0; l < kCvLists; ++l) {
            const bool in = (flag[k] >> l) & 1u;
            uint32_t at = dst[l] + lane_prefix(__ballot(in));
#pragma unroll
            for (uint32_t w = 0; w < kCvWaves; ++w) {
                const uint32_t n = wave_cnt[k][l][w];
                at += w < wave ? n : 0u;
                dst[l] += n;
            }
            if (in && at < b.max_pairs) b.out[l][at] = rec;
        }
    }
}

}  // namespace
}  // namespace mvdr

using namespace mvdr;

struct mvdr_crossview {
    mvdr_crossview_config cfg{};
    CvBuffers b{};
    uint32_t tiles = 0;
    void* block = nullptr;
    hipEvent_t done = nullptr;
    bool found = false;
    ~mvdr_crossview() {
        if (done) (void)hipEventDestroy(done);
        if (b.counts) (void)hipHostFree(b.counts);
        if (block) (void)hipFree(block);
    }
};

extern "C" {

void mvdr_crossview_default_config(mvdr_crossview_config* c) {
    if (!c) return;
    std::memset(c, 0, sizeof(*c));
    c->max_views = MVDR_MAX_VIEWS;
    c->max_width = 640;
    c->max_height = 480;
    c->max_pairs = 16384;
    c->search_radius = 20;
    c->search_step = 2;
    c->track_radius = 1;
    c->max_distance2 = 1e-4f;  // 1 cm
}

mvdr_status mvdr_crossview_create(const mvdr_crossview_config* config, mvdr_crossview** out) {
    if (!config || !out) return MVDR_E_INVALID;
    *out = nullptr;
    const mvdr_crossview_config& c = *config;
    if (c.max_views < 1 || c.max_views > MVDR_MAX_VIEWS || c.max_width < 1 || c.max_height < 1 ||
        c.max_width > 65535 || c.max_height > 65535 || c.max_pairs < 1 || c.search_step < 1 || c.search_radius > 1024 ||
        c.track_radius > 16 || !(c.max_distance2 >= 0.f))
        return MVDR_E_SHAPE;
    const uint64_t pixels = (uint64_t)c.max_views * c.max_width * c.max_height;
    if (pixels >= 0xFFFFFFFFull) return MVDR_E_SHAPE;
    auto* h = new mvdr_crossview();
    h->cfg = c;
    h->tiles = cv_tiles((uint32_t)pixels);
    size_t off = 0;
    auto carve = [&](auto*& p, size_t n, char* base) {
        using T = std::remove_reference_t<decltype(*p)>;
        off = (off + 255) & ~(size_t)255;
        p = base ? reinterpret_cast<T*>(base + off) : nullptr;
        off += std::max<size_t>(n, 1) * sizeof(T);
    };
    auto lay = [&](char* base) {
        off = 0;
        carve(h->b.cand, pixels, base);
        carve(h->b.best, pixels, base);
        carve(h->b.edges, pixels, base);
        carve(h->b.num_edges, 1, base);
        carve(h->b.flags, pixels, base);
        carve(h->b.tile_count, (size_t)kCvLists * h->tiles, base);
        carve(h->b.tile_offset, (size_t)kCvLists * h->tiles, base);
        for (uint32_t l = 0; l < kCvLists; ++l) carve(h->b.out[l], c.max_pairs, base);
        return off;
    };
    const size_t bytes = lay(nullptr);
    hipError_t e = hipMalloc(&h->block, bytes);
    if (e == hipSuccess) {
        lay(static_cast<char*>(h->block));
        e = hipMemset(h->b.num_edges, 0, sizeof(uint32_t));
        // the fill is done before a call on a stream that does not wait for the null stream
        if (e == hipSuccess) e = hipStreamSynchronize(nullptr);
    }
    // the getters read the totals without a copy (~10 us each)
    if (e == hipSuccess)
        e = hipHostMalloc(reinterpret_cast<void**>(&h->b.counts), kCvLists * sizeof(uint32_t), hipHostMallocDefault);
    if (e == hipSuccess) std::memset(h->b.counts, 0, kCvLists * sizeof(uint32_t));
    if (e == hipSuccess) e = hipEventCreateWithFlags(&h->done, hipEventDisableTiming);
    if (e != hipSuccess) {
        delete h;
        return MVDR_E_HIP;
    }
    h->b.max_pairs = c.max_pairs;
    h->b.cap_edges = (uint32_t)pixels;
    h->b.radius = (int)c.search_radius;
    h->b.step = (int)c.search_step;
    h->b.track = (int)c.track_radius;
    h->b.max_d2 = c.max_distance2;
    *out = h;
    return MVDR_OK;
}

void mvdr_crossview_destroy(mvdr_crossview* h) {
    if (!h) return;
    if (h->done) (void)hipEventSynchronize(h->done);
    delete h;
}

mvdr_status mvdr_crossview_find(mvdr_crossview* h, const mvdr_crossview_input* in, void* stream) {
    if (!h || !in) return MVDR_E_INVALID;
    const mvdr_crossview_config& c = h->cfg;
    if (in->num_views < 1 || in->num_views > c.max_views || in->width < 1 || in->height < 1 ||
        in->width > c.max_width || in->height > c.max_height)
        return MVDR_E_SHAPE;
    CvFrame f;
    std::memset(&f, 0, sizeof(f));
    f.V = in->num_views;
    f.W = in->width;
    f.H = in->height;
    for (uint32_t v = 0; v < f.V; ++v) {
        if (!in->vertex[v] || !in->edge_mask[v]) return MVDR_E_INVALID;
        f.fx[v] = in->intrinsic[v].fx;
        f.fy[v] = in->intrinsic[v].fy;
        f.cx[v] = in->intrinsic[v].cx;
        f.cy[v] = in->intrinsic[v].cy;
        f.init[v] = to_mat34(in->initial_camera_se3[v]);
        f.init_inv[v] = inverse(f.init[v]);
        f.vertex[v] = static_cast<const float4*>(in->vertex[v]);
        f.edge[v] = static_cast<const uint8_t*>(in->edge_mask[v]);
        f.corr[v] = static_cast<const ushort4*>(in->corr_map[v]);
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint32_t pixels = f.V * f.W * f.H;
    const uint32_t tiles = cv_tiles(pixels);
    // candidates and flags loop over the edge list (its length is known on the
    // device alone)
    hipLaunchKernelGGL(cv_edges_kernel, dim3(tiles), dim3(kCvThreads), 0, st, f, h->b, tiles);
    hipLaunchKernelGGL(cv_candidates_kernel, dim3(2048), dim3(256), 0, st, f, h->b);
    hipLaunchKernelGGL(cv_flags_kernel, dim3(std::min<uint32_t>(tiles, 512u)), dim3(kCvThreads), 0, st, f, h->b, tiles);
    hipLaunchKernelGGL(cv_scan_kernel, dim3(1), dim3(1024), 0, st, h->b, tiles);
    hipLaunchKernelGGL(cv_scatter_kernel, dim3(tiles), dim3(kCvThreads), 0, st, f, h->b, tiles);
    if (hipGetLastError() != hipSuccess) return MVDR_E_HIP;
    if (hipEventRecord(h->done, st) != hipSuccess) return MVDR_E_HIP;
    h->found = true;
    return MVDR_OK;
}

mvdr_status mvdr_crossview_get_pairs(mvdr_crossview* h, int list, const void** pairs, uint32_t* count) {
    if (!h || !pairs || !count || list < 0 || list >= (int)kCvLists) return MVDR_E_INVALID;
    if (!h->found) return MVDR_E_STATE;
    if (hipEventSynchronize(h->done) != hipSuccess) return MVDR_E_HIP;
    if (hipStreamSynchronize(nullptr) != hipSuccess) return MVDR_E_HIP;  // as a copy on it would
    const uint32_t n = *static_cast<volatile const uint32_t*>(h->b.counts + list);
    *pairs = h->b.out[list];
    *count = std::min(n, h->cfg.max_pairs);
    return n > h->cfg.max_pairs ? MVDR_E_CAPACITY : MVDR_OK;
}

}  // extern "C"
