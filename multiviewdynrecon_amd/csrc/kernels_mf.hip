// Matrix-free J^T J apply (applyJtJDotWithIndexKernel,
// ApplyJtJMatrixFreeIndexed.cu:29-349) and the block-Jacobi PCG around it.
//
// y = sum_t J_t^T (J_t v) + damping v without the J^T J blocks, in the
// node-centred coordinates of the rest of the solve (rows J'_n = w_n J T_n):
//   terms  : one thread per term, u_t = lambda^2 J_t (sum_k w_k T_k v_k) over
//            the term's knn slots (graph edges: both ends' own rows) -- the
//            Jacobians are recomputed from the term records every apply;
//   gather : a row group per node over its Node2Term list,
//            y_i = sum_(i,t) J'_i(t)^T u_t + 1e-2 T_i^T T_i v_i.
// A node named by m > 1 knn slots of one term (the reference's pair
// multiplicity) appears m times in its Node2Term list; each entry subtracts
// (m - 1) lambda^2 J'^T J' v_i, so the apply equals the materialized J^T J of
// the index-driven assembly exactly, damping and cross-view term included
// (the reference's matrix-free path leaves both out).
#include "common.h"
#include "device_util.h"
#include "eval.h"
#include "pcg_util.h"
#include "terms.h"

namespace mvdr {

enum : int { kSrcDir = 0, kSrcX = 1, kSrcZ = 2 };        // the vector v applied to
enum : int { kEpiSpmv = 0, kEpiResidual = 1, kEpiCurvature = 2 };

// Node-centred twist -> reference twist: (w, v + g x w).
__device__ inline void node_to_ref(const float4 g, const float x[6], float y[6]) {
    y[0] = x[0];
    y[1] = x[1];
    y[2] = x[2];
    y[3] = x[3] + (g.y * x[2] - g.z * x[1]);
    y[4] = x[4] + (g.z * x[0] - g.x * x[2]);
    y[5] = x[5] + (g.x * x[1] - g.y * x[0]);
}

__device__ inline float dot6(const float a[6], const float b[6]) {
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2] + a[3] * b[3] + a[4] * b[4] + a[5] * b[5];
}

struct MfLambda2 {
    float smooth, density, foreground, feature, cross;
};

__device__ inline MfLambda2 mf_lambda2(const Penalty& p) {
    return MfLambda2{p.smooth * p.smooth, p.density * p.density, p.foreground * p.foreground, p.feature * p.feature,
                     p.cross * p.cross};
}

// Term pass: u_t for every term.  kSrcDir forms the PCG direction
// d = s + beta d_prev (beta from the previous launches' partials) on the fly
// and stores it for the gather and the update.
template <int kSrc>
__global__ void __launch_bounds__(256) mf_terms_kernel(const Buffers* __restrict__ bs, uint32_t k, uint32_t cur, Penalty pen) {
    const Buffers b = frame_buffers(bs);
    const FrameDev& f = *b.frame;
    const Counts& c = *b.counts;
    float beta = 0;
    if (kSrc == kSrcDir && k > 0) {
        float num, den;
        reduce_partials2<float>(slot_ptr(b, kSlotDelta + k), kVecBlocks, slot_ptr(b, kSlotDelta + k - 1), kVecBlocks, num, den);
        beta = den != (float)0 ? num / den : (float)0;
    }
    if (c.error) return;
    const float* __restrict__ prev = cur ? b.d1 : b.d0;
    float* __restrict__ dout = cur ? b.d0 : b.d1;
    const float* __restrict__ vec = kSrc == kSrcX ? b.x : b.d1;
    auto source = [&](uint32_t n, float v[6]) {
#pragma unroll
        for (int a = 0; a < 6; ++a) {
            if (kSrc == kSrcDir) {
                const float p = prev[6 * n + a];
                v[a] = k > 0 ? (float)((float)b.s[6 * n + a] + beta * (float)p) : p;
            } else {
                v[a] = vec[6 * n + a];
            }
        }
    };
    const TermBounds tb(c);
    const MfLambda2 l2 = mf_lambda2(pen);
    const bool density = b.density && pen.density != 0.f;
    const uint32_t total = c.off[4];
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < total; t += stride) {
        uint32_t kk;
        const int type = type_of(tb, t, kk);
        float u[3] = {0.f, 0.f, 0.f};
        if (type == kSmooth) {
            const SmoothRec sm = b.smooth[kk];
            const uint32_t n1 = sm.ij & 0xFFFF, n2 = sm.ij >> 16;
            float J1[3][6], J2[3][6], res[3], v[6], w1[6], w2[6];
            smooth_rows(sm, true, J1, res);
            smooth_rows(sm, n2 == n1, J2, res);
            source(n1, v);
            node_to_ref(f.nodes[n1], v, w1);
            source(n2, v);
            node_to_ref(f.nodes[n2], v, w2);
#pragma unroll
            for (int r = 0; r < 3; ++r) u[r] = l2.smooth * (dot6(J1[r], w1) + dot6(J2[r], w2));
        } else {
            ushort4 knn;
            float4 wk;
            float J[3][6], res[3];
            int rows = 3;
            float lam[3];
            if (type == kDense || type == kForeground) {
                const ScalarRec& rec = type == kDense ? b.dense[kk] : b.fg[kk];
                knn = rec.knn;
                wk = rec.w;
#pragma unroll
                for (int q = 0; q < 6; ++q) J[0][q] = rec.J[q];
                lam[0] = type == kDense ? 1.f : l2.foreground;
                rows = 1;
                if (type == kDense && density) {
                    const ScalarRec& d = b.density[kk];
#pragma unroll
                    for (int q = 0; q < 6; ++q) J[1][q] = d.J[q];
                    lam[1] = l2.density;
                    rows = 2;
                }
            } else {
                const P2PRec& rec = type == kFeature ? b.feat[kk] : b.cross[kk];
                knn = rec.knn;
                wk = rec.w;
                p2p_rows(rec, J, res);
                const uint32_t mask = type == kFeature ? 0xFFFFFFFFu : 0u;
                lam[0] = lam[1] = lam[2] =
                    __uint_as_float((__float_as_uint(l2.feature) & mask) | (__float_as_uint(l2.cross) & ~mask));
            }
            // sum_k w_k T_k v_k over the knn slots (slot-rule weights)
            float V[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            const uint32_t n[4] = {knn.x, knn.y, knn.z, knn.w};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float v[6], w6[6];
                source(n[q], v);
                node_to_ref(f.nodes[n[q]], v, w6);
                const float ws = slot_weight(knn, wk, n[q]);
#pragma unroll
                for (int a = 0; a < 6; ++a) V[a] += ws * w6[a];
            }
#pragma unroll
            for (int r = 0; r < 3; ++r)
                if (r < rows) u[r] = lam[r] * dot6(J[r], V);
        }
        b.mf_u[t] = make_float4(u[0], u[1], u[2], 0.f);
    }
    if (kSrc == kSrcDir) {
        for (uint32_t n = blockIdx.x * blockDim.x + threadIdx.x; n < f.N; n += stride) {
            float v[6];
            source(n, v);
#pragma unroll
            for (int a = 0; a < 6; ++a) dout[6 * n + a] = v[a];
        }
    }
}

// Gather pass: y_i over the Node2Term list of row i (kRowLanes lanes per row),
// then the epilogue of the PCG step it serves.
template <int kEpi>
__global__ void __launch_bounds__(256) mf_gather_kernel(const Buffers* __restrict__ bs, uint32_t k, uint32_t cur, Penalty pen) {
    const Buffers b = frame_buffers(bs);
    const FrameDev& f = *b.frame;
    const Counts& c = *b.counts;
    const uint32_t sub = threadIdx.x % kRowLanes;
    const float* __restrict__ vec = kEpi == kEpiSpmv ? (cur ? b.d0 : b.d1) : (kEpi == kEpiResidual ? b.x : b.d1);
    float acc = 0;
    if (!c.error) {
        const TermBounds tb(c);
        const MfLambda2 l2 = mf_lambda2(pen);
        const bool density = b.density && pen.density != 0.f;
        const uint32_t groups = gridDim.x * kRowsPerBlock;
        for (uint32_t base = blockIdx.x * kRowsPerBlock; base < f.N; base += groups) {
            const uint32_t i = base + threadIdx.x / kRowLanes;
            float y[6] = {0, 0, 0, 0, 0, 0};
            float vi[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (i < f.N) {
                const float4 g = f.nodes[i];
#pragma unroll
                for (int a = 0; a < 6; ++a) vi[a] = vec[6 * i + a];
                const uint32_t beg = b.n2t_offset[i], end = b.n2t_offset[i + 1];
                for (uint32_t e = beg + sub; e < end; e += kRowLanes) {
                    const uint32_t t = b.n2t_index[e];
                    uint32_t kk;
                    const int type = type_of(tb, t, kk);
                    float J[3][6], res[3], lam[3];
                    int rows = 3;
                    float wi = 1.f;
                    uint32_t mult = 1;
                    if (type == kSmooth) {
                        const SmoothRec sm = b.smooth[kk];
                        const uint32_t n1 = sm.ij & 0xFFFF, n2 = sm.ij >> 16;
                        smooth_rows(sm, i == n1, J, res);
                        lam[0] = lam[1] = lam[2] = l2.smooth;
                        mult = (n1 == i ? 1u : 0u) + (n2 == i ? 1u : 0u);
                    } else {
                        ushort4 knn;
                        float4 wk;
                        if (type == kDense || type == kForeground) {
                            const ScalarRec& rec = type == kDense ? b.dense[kk] : b.fg[kk];
                            knn = rec.knn;
                            wk = rec.w;
#pragma unroll
                            for (int q = 0; q < 6; ++q) J[0][q] = rec.J[q];
                            lam[0] = type == kDense ? 1.f : l2.foreground;
                            rows = 1;
                            if (type == kDense && density) {
                                const ScalarRec& d = b.density[kk];
#pragma unroll
                                for (int q = 0; q < 6; ++q) J[1][q] = d.J[q];
                                lam[1] = l2.density;
                                rows = 2;
                            }
                        } else {
                            const P2PRec& rec = type == kFeature ? b.feat[kk] : b.cross[kk];
                            knn = rec.knn;
                            wk = rec.w;
                            p2p_rows(rec, J, res);
                            const uint32_t mask = type == kFeature ? 0xFFFFFFFFu : 0u;
                            lam[0] = lam[1] = lam[2] = __uint_as_float((__float_as_uint(l2.feature) & mask) |
                                                                       (__float_as_uint(l2.cross) & ~mask));
                        }
                        wi = slot_weight(knn, wk, i);
                        mult = (knn.x == i) + (knn.y == i) + (knn.z == i) + (knn.w == i);
                    }
                    const float4 ut = b.mf_u[t];
                    const float u[3] = {ut.x, ut.y, ut.z};
#pragma unroll
                    for (int r = 0; r < 3; ++r) {
                        if (r < rows) {
                            to_node_frame(J[r], g);
                            float s = wi * u[r];
                            if (mult > 1) s -= (float)(mult - 1) * lam[r] * wi * wi * dot6(J[r], vi);
#pragma unroll
                            for (int a = 0; a < 6; ++a) y[a] += (float)(s * J[r][a]);
                        }
                    }
                }
                if (sub == 0) {
                    // damping 1e-2 T^T T v: T v = (w, v + g x w), T^T (a, b) = (a + b x g, b)
                    float tv[6];
                    node_to_ref(g, vi, tv);
                    const float bx = tv[4] * g.z - tv[5] * g.y, by = tv[5] * g.x - tv[3] * g.z,
                                bz = tv[3] * g.y - tv[4] * g.x;
                    const float damp[6] = {tv[0] + bx, tv[1] + by, tv[2] + bz, tv[3], tv[4], tv[5]};
#pragma unroll
                    for (int a = 0; a < 6; ++a) y[a] += (float)(1e-2f * damp[a]);
                }
            }
#pragma unroll
            for (int a = 0; a < 6; ++a) y[a] = lanes_sum<kRowLanes>(y[a]);
            if (i < f.N && sub == 0) {
                if (kEpi == kEpiSpmv) {
#pragma unroll
                    for (int a = 0; a < 6; ++a) {
                        b.q[6 * i + a] = (float)y[a];
                        acc += (float)vi[a] * y[a];
                    }
                } else if (kEpi == kEpiResidual) {
                    float rr[6], z[6];
#pragma unroll
                    for (int a = 0; a < 6; ++a) {
                        rr[a] = (float)((float)b.jtr[6 * i + a] - y[a]);
                        b.r[6 * i + a] = rr[a];
                    }
                    apply_minv<float>(b, i, rr, z);
#pragma unroll
                    for (int a = 0; a < 6; ++a) {
                        b.d1[6 * i + a] = z[a];
                        acc += (float)rr[a] * (float)z[a];
                    }
                } else {
#pragma unroll
                    for (int a = 0; a < 6; ++a) acc += (float)vi[a] * y[a];
                }
            }
        }
    }
    write_partial<float>(b, kEpi == kEpiSpmv ? kSlotDQ + k : (kEpi == kEpiResidual ? kSlotRefNum : kSlotRefDen), acc);
}

// ------------------------------------------ matrix-free apply, J recomputed
// MVDR_JTJ_RECOMPUTE: the operator above with every Jacobian re-evaluated
// inside each apply from the solver / observation maps and the current warp
// se3[which] (eval.h), the way the evaluation pass computes it; from the term
// records only the index's knn and weights and the feature targets are read.
//   terms  : one thread per term: J_t, u_t = J_t V_t with V_t the knn blend
//            of the source vector, and g_t = sum_r lambda_r^2 u_tr J_tr
//            (6 floats; an edge term keeps lambda^2 u_t, 3 floats);
//   gather : y_i = T_i^T sum_(i,t) w_i(t) g_t + damping, an edge term's rows
//            re-evaluated from its two node transforms, and a knn term's J
//            re-evaluated when the term names node i in m > 1 slots (the
//            multiplicity correction of the stored-J apply).
// Debug forms (unit term weights): kSrcRows takes u_t from mf_u, kOutRows
// writes u_t = J_t V_t to mf_u (J x), and kEpiAdjoint writes the gather's sum
// without damping or correction to q (J^T y, the exact adjoint of J x: the
// slot weight of node i depends on i alone, so each of its m entries carries
// it once).
enum : int { kSrcRows = 3 };
enum : int { kOutG = 0, kOutRows = 1 };
enum : int { kEpiAdjoint = 3 };

// Knn and weights of a knn term (fixed by the index build).
__device__ inline void term_knn(const Buffers& b, int type, uint32_t kk, ushort4& knn, float4& w) {
    if (type == kDense || type == kForeground) {
        const ScalarRec& r = type == kDense ? b.dense[kk] : b.fg[kk];
        knn = r.knn;
        w = r.w;
    } else {
        const P2PRec& r = type == kFeature ? b.feat[kk] : b.cross[kk];
        knn = r.knn;
        w = r.w;
    }
}

// J rows and lambda^2 of a knn term (dense depth + density, foreground,
// feature, cross view) evaluated at the warp se3.
template <typename R>
__device__ inline int knn_term_rows(const Buffers& b, const FrameDev& f, const DQ* se3, int type, uint32_t kk,
                                    const MfLambda2& l2, bool density, float J[3][6], float lam[3]) {
    if (type == kDense || type == kForeground) {
        ScalarRec rec;
        term_knn(b, type, kk, rec.knn, rec.w);
        const ushort4 px = type == kDense ? b.dense_px[kk] : b.fg_px[kk];
        if (type == kDense) eval_dense<R>(f, se3, px, rec);
        else eval_image<R>(f, se3, px, false, rec);
#pragma unroll
        for (int q = 0; q < 6; ++q) J[0][q] = rec.J[q];
        lam[0] = type == kDense ? 1.f : l2.foreground;
        if (type == kDense && density) {
            eval_image<R>(f, se3, px, true, rec);
#pragma unroll
            for (int q = 0; q < 6; ++q) J[1][q] = rec.J[q];
            lam[1] = l2.density;
            return 2;
        }
        return 1;
    }
    const bool cross = type == kCross;
    const P2PRec& src = cross ? b.cross[kk] : b.feat[kk];
    P2PRec rec;
    rec.knn = src.knn;
    rec.w = src.w;
    rec.target = src.target;
    rec.warped = eval_warped<R>(se3, rec.knn, rec.w, cross ? b.cross_canon[kk] : b.feat_canon[kk]);
    float res[3];
    p2p_rows(rec, J, res);
    lam[0] = lam[1] = lam[2] = cross ? l2.cross : l2.feature;
    return 3;
}

// The weight of each Node2Term entry's node, fixed by the index build: the
// slot weight of node i in the term's knn, its sign bit set when the term
// names i in more than one slot (the rare entries whose apply needs the
// multiplicity correction).  Graph-edge entries are not read through it.
__global__ void __launch_bounds__(256) mf_entry_weights_kernel(const Buffers* __restrict__ bs) {
    const Buffers b = frame_buffers(bs);
    const FrameDev& f = *b.frame;
    const Counts& c = *b.counts;
    if (c.error) return;
    const TermBounds tb(c);
    const uint32_t sub = threadIdx.x % kRowLanes;
    const uint32_t groups = gridDim.x * kRowsPerBlock;
    for (uint32_t base = blockIdx.x * kRowsPerBlock; base < f.N; base += groups) {
        const uint32_t i = base + threadIdx.x / kRowLanes;
        if (i >= f.N) continue;
        const uint32_t beg = b.n2t_offset[i], end = b.n2t_offset[i + 1];
        for (uint32_t e = beg + sub; e < end; e += kRowLanes) {
            uint32_t kk;
            const int type = type_of(tb, b.n2t_index[e], kk);
            if (type == kSmooth) continue;
            ushort4 knn;
            float4 wk;
            term_knn(b, type, kk, knn, wk);
            const uint32_t mult = (knn.x == i) + (knn.y == i) + (knn.z == i) + (knn.w == i);
            const float wi = slot_weight(knn, wk, i);
            b.n2t_w[e] = mult > 1 ? copysignf(fabsf(wi), -1.0f) : fabsf(wi);
        }
    }
}

template <int kSrc, int kOut>
__global__ void __launch_bounds__(256) mfr_terms_kernel(const Buffers* __restrict__ bs, uint32_t k, uint32_t cur, Penalty pen,
                                                        uint32_t which) {
    const Buffers b = frame_buffers(bs);
    const FrameDev& f = *b.frame;
    const Counts& c = *b.counts;
    const DQ* __restrict__ se3 = which ? b.se3[1] : b.se3[0];
    float beta = 0;
    if (kSrc == kSrcDir && k > 0) {
        float num, den;
        reduce_partials2<float>(slot_ptr(b, kSlotDelta + k), kVecBlocks, slot_ptr(b, kSlotDelta + k - 1), kVecBlocks, num, den);
        beta = den != (float)0 ? num / den : (float)0;
    }
    if (c.error) return;
    const float* __restrict__ prev = cur ? b.d1 : b.d0;
    float* __restrict__ dout = cur ? b.d0 : b.d1;
    const float* __restrict__ vec = kSrc == kSrcX ? b.x : b.d1;
    auto source = [&](uint32_t n, float v[6]) {
#pragma unroll
        for (int a = 0; a < 6; ++a) {
            if (kSrc == kSrcDir) {
                const float p = prev[6 * n + a];
                v[a] = k > 0 ? (float)((float)b.s[6 * n + a] + beta * (float)p) : p;
            } else {
                v[a] = vec[6 * n + a];
            }
        }
    };
    const TermBounds tb(c);
    const MfLambda2 l2 = mf_lambda2(pen);
    const bool density = b.density && pen.density != 0.f;
    const uint32_t total = c.off[4];
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < total; t += stride) {
        uint32_t kk;
        const int type = type_of(tb, t, kk);
        float u[3] = {0.f, 0.f, 0.f};
        float g[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (kSrc == kSrcRows) {
            const float4 ut = b.mf_u[t];
            u[0] = ut.x;
            u[1] = ut.y;
            u[2] = ut.z;
        }
        if (type == kSmooth) {
            if (kSrc != kSrcRows) {
                const SmoothRec sm = eval_smooth<float>(f, se3, kk);
                const uint32_t n1 = sm.ij & 0xFFFF, n2 = sm.ij >> 16;
                float J1[3][6], J2[3][6], res[3], v[6], w1[6], w2[6];
                smooth_rows(sm, true, J1, res);
                smooth_rows(sm, n2 == n1, J2, res);
                source(n1, v);
                node_to_ref(f.nodes[n1], v, w1);
                source(n2, v);
                node_to_ref(f.nodes[n2], v, w2);
#pragma unroll
                for (int r = 0; r < 3; ++r) u[r] = dot6(J1[r], w1) + dot6(J2[r], w2);
            }
            const float l = kSrc == kSrcRows ? 1.f : l2.smooth;
#pragma unroll
            for (int r = 0; r < 3; ++r) g[r] = l * u[r];
        } else {
            float J[3][6], lam[3];
            const int rows = knn_term_rows<float>(b, f, se3, type, kk, l2, density, J, lam);
            if (kSrc != kSrcRows) {
                ushort4 knn;
                float4 wk;
                term_knn(b, type, kk, knn, wk);
                float V[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                const uint32_t n[4] = {knn.x, knn.y, knn.z, knn.w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float v[6], w6[6];
                    source(n[q], v);
                    node_to_ref(f.nodes[n[q]], v, w6);
                    const float ws = slot_weight(knn, wk, n[q]);
#pragma unroll
                    for (int a = 0; a < 6; ++a) V[a] += ws * w6[a];
                }
#pragma unroll
                for (int r = 0; r < 3; ++r) u[r] = r < rows ? dot6(J[r], V) : 0.f;
            }
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                if (r < rows) {
                    const float s = (kSrc == kSrcRows ? 1.f : lam[r]) * u[r];
#pragma unroll
                    for (int a = 0; a < 6; ++a) g[a] += s * J[r][a];
                }
            }
        }
        if (kOut == kOutRows) {
            b.mf_u[t] = make_float4(u[0], u[1], u[2], 0.f);
        } else {
            b.mf_g[2 * (size_t)t] = make_float4(g[0], g[1], g[2], g[3]);
            b.mf_g[2 * (size_t)t + 1] = make_float4(g[4], g[5], 0.f, 0.f);
        }
    }
    if (kSrc == kSrcDir) {
        for (uint32_t n = blockIdx.x * blockDim.x + threadIdx.x; n < f.N; n += stride) {
            float v[6];
            source(n, v);
#pragma unroll
            for (int a = 0; a < 6; ++a) dout[6 * n + a] = v[a];
        }
    }
}

template <int kEpi>
__global__ void __launch_bounds__(256) mfr_gather_kernel(const Buffers* __restrict__ bs, uint32_t k, uint32_t cur, Penalty pen,
                                                         uint32_t which) {
    const Buffers b = frame_buffers(bs);
    const FrameDev& f = *b.frame;
    const Counts& c = *b.counts;
    const DQ* __restrict__ se3 = which ? b.se3[1] : b.se3[0];
    const uint32_t sub = threadIdx.x % kRowLanes;
    const float* __restrict__ vec = kEpi == kEpiSpmv ? (cur ? b.d0 : b.d1) : (kEpi == kEpiResidual ? b.x : b.d1);
    constexpr bool correct = kEpi != kEpiAdjoint;
    float acc = 0;
    if (!c.error) {
        const TermBounds tb(c);
        const MfLambda2 l2 = mf_lambda2(pen);
        const bool density = b.density && pen.density != 0.f;
        const uint32_t groups = gridDim.x * kRowsPerBlock;
        for (uint32_t base = blockIdx.x * kRowsPerBlock; base < f.N; base += groups) {
            const uint32_t i = base + threadIdx.x / kRowLanes;
            float y[6] = {0, 0, 0, 0, 0, 0};   // reference coordinates until the row is complete
            float vi[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            float4 gi = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i < f.N) {
                gi = f.nodes[i];
                float tvi[6];
                if (correct) {
#pragma unroll
                    for (int a = 0; a < 6; ++a) vi[a] = vec[6 * i + a];
                }
                node_to_ref(gi, vi, tvi);
                const uint32_t beg = b.n2t_offset[i], end = b.n2t_offset[i + 1];
                for (uint32_t e = beg + sub; e < end; e += kRowLanes) {
                    const uint32_t t = b.n2t_index[e];
                    uint32_t kk;
                    const int type = type_of(tb, t, kk);
                    const float4 g0 = b.mf_g[2 * (size_t)t];
                    if (type == kSmooth) {
                        const SmoothRec sm = eval_smooth<float>(f, se3, kk);
                        const uint32_t n1 = sm.ij & 0xFFFF, n2 = sm.ij >> 16;
                        float J[3][6], res[3];
                        smooth_rows(sm, i == n1, J, res);
                        const uint32_t mult = (n1 == i ? 1u : 0u) + (n2 == i ? 1u : 0u);
                        const float u[3] = {g0.x, g0.y, g0.z};
#pragma unroll
                        for (int r = 0; r < 3; ++r) {
                            float s = u[r];
                            if (correct && mult > 1) s -= (float)(mult - 1) * l2.smooth * dot6(J[r], tvi);
#pragma unroll
                            for (int a = 0; a < 6; ++a) y[a] += (float)(s * J[r][a]);
                        }
                    } else {
                        const float4 g1 = b.mf_g[2 * (size_t)t + 1];
                        const float ws = b.n2t_w[e];
                        const float wi = fabsf(ws);
                        const float gv[6] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y};
#pragma unroll
                        for (int a = 0; a < 6; ++a) y[a] += (float)(wi * gv[a]);
                        if (correct && signbit(ws)) {
                            ushort4 knn;
                            float4 wk;
                            term_knn(b, type, kk, knn, wk);
                            const uint32_t mult = (knn.x == i) + (knn.y == i) + (knn.z == i) + (knn.w == i);
                            float J[3][6], lam[3];
                            const int rows = knn_term_rows<float>(b, f, se3, type, kk, l2, density, J, lam);
                            for (int r = 0; r < rows; ++r) {
                                const float s = -(float)(mult - 1) * lam[r] * wi * wi * dot6(J[r], tvi);
#pragma unroll
                                for (int a = 0; a < 6; ++a) y[a] += (float)(s * J[r][a]);
                            }
                        }
                    }
                }
            }
#pragma unroll
            for (int a = 0; a < 6; ++a) y[a] = lanes_sum<kRowLanes>(y[a]);
            if (i < f.N && sub == 0) {
                // to node-centred coordinates: T^T (a, b) = (a + b x g, b)
                y[0] += y[4] * (float)gi.z - y[5] * (float)gi.y;
                y[1] += y[5] * (float)gi.x - y[3] * (float)gi.z;
                y[2] += y[3] * (float)gi.y - y[4] * (float)gi.x;
                if (kEpi == kEpiAdjoint) {
#pragma unroll
                    for (int a = 0; a < 6; ++a) b.q[6 * i + a] = (float)y[a];
                    continue;
                }
                // damping 1e-2 T^T T v
                float tv[6];
                node_to_ref(gi, vi, tv);
                const float bx = tv[4] * gi.z - tv[5] * gi.y, by = tv[5] * gi.x - tv[3] * gi.z,
                            bz = tv[3] * gi.y - tv[4] * gi.x;
                const float damp[6] = {tv[0] + bx, tv[1] + by, tv[2] + bz, tv[3], tv[4], tv[5]};
#pragma unroll
                for (int a = 0; a < 6; ++a) y[a] += (float)(1e-2f * damp[a]);
                if (kEpi == kEpiSpmv) {
#pragma unroll
                    for (int a = 0; a < 6; ++a) {
                        b.q[6 * i + a] = (float)y[a];
                        acc += (float)vi[a] * y[a];
                    }
                } else if (kEpi == kEpiResidual) {
                    float rr[6], z[6];
#pragma unroll
                    for (int a = 0; a < 6; ++a) {
                        rr[a] = (float)((float)b.jtr[6 * i + a] - y[a]);
                        b.r[6 * i + a] = rr[a];
                    }
                    apply_minv<float>(b, i, rr, z);
#pragma unroll
                    for (int a = 0; a < 6; ++a) {
                        b.d1[6 * i + a] = z[a];
                        acc += (float)rr[a] * (float)z[a];
                    }
                } else {
#pragma unroll
                    for (int a = 0; a < 6; ++a) acc += (float)vi[a] * y[a];
                }
            }
        }
    }
    if (kEpi != kEpiAdjoint)
        write_partial<float>(b, kEpi == kEpiSpmv ? kSlotDQ + k : (kEpi == kEpiResidual ? kSlotRefNum : kSlotRefDen), acc);
}

// Node-centred <-> reference coordinates of the debug products, in place on
// q: to_ref 1: T^-T y (a J^T result), 0 on d1: T^-1 x (a twist).
__global__ void __launch_bounds__(256) mfr_coords_kernel(const Buffers* __restrict__ bs, int jt_result) {
    const Buffers b = frame_buffers(bs);
    const FrameDev& f = *b.frame;
    float* v = jt_result ? b.q : b.d1;
    for (uint32_t n = blockIdx.x * blockDim.x + threadIdx.x; n < f.N; n += gridDim.x * blockDim.x) {
        const float4 g = f.nodes[n];
        float a[3] = {v[6 * n], v[6 * n + 1], v[6 * n + 2]};
        const float c[3] = {v[6 * n + 3], v[6 * n + 4], v[6 * n + 5]};
        if (jt_result) {
            // (a, c) -> (a - c x g, c)
            a[0] -= c[1] * g.z - c[2] * g.y;
            a[1] -= c[2] * g.x - c[0] * g.z;
            a[2] -= c[0] * g.y - c[1] * g.x;
#pragma unroll
            for (int q = 0; q < 3; ++q) v[6 * n + q] = a[q];
        } else {
            // (a, c) -> (a, c - g x a)
            v[6 * n + 3] = c[0] - (g.y * a[2] - g.z * a[1]);
            v[6 * n + 4] = c[1] - (g.z * a[0] - g.x * a[2]);
            v[6 * n + 5] = c[2] - (g.x * a[1] - g.y * a[0]);
        }
    }
}

// ------------------------------------------------------------- mixed mode
// The same PCG with FP64 sums, three launches per iteration: terms, gather,
// update.  What bounds them is gathers of a few words per lane, so the data is
// laid out for wide loads:
//   terms  : a knn slot's source is one 64-byte record (s, d_prev, node) -- four
//            16-byte loads where separate arrays took 13 dwords -- and the
//            direction is formed from it as before;
//   gather : one wave per node over its Node2Term list, an entry being one 8-byte
//            record (term, sign bit set when the term names the node in several
//            slots, and the slot weight) and the term's J and u (stored J) or
//            g_t (recomputed J); the six sums of a row by a reduce-scatter.  With
//            16 lanes a row of 450 entries was 28 dependent rounds on 125
//            workgroups;
//   update : eight lanes per node, a lane reading its row of M^-1 (48 contiguous
//            bytes) where a thread per node read 288 on 64 workgroups.
// Every 32-bit value (d, q, x, r, s, and a term's u, g and products) is rounded
// where it was, and only FP64 sums are reordered, so the iterates keep their bits.
// 2k nodes, 220k terms, stored J: gather 127 -> 22 us, terms 14 -> 9, update 8.9 ->
// 4.8 (10 PCG x 5 GN: 8.2 -> 2.55 ms a frame); 8k nodes, 163k terms, recomputed J:
// gather 28 -> 14 us, terms 27 -> 20, update 8.9 -> 5.1 (15 x 5: 5.3 -> 3.45 ms).
// The FP32 mode keeps the kernels above: its sums are 32-bit, their order is part
// of its results.
constexpr uint32_t kMfWaves = 8;                      // rows (waves) per gather workgroup
constexpr uint32_t kMfGroups = kPartialStride;        // partial sums of the gather, at most
constexpr uint32_t kMfLanes = 8;                      // lanes per node in the update
constexpr uint32_t kMfNodes = 256 / kMfLanes;         // nodes per update workgroup
constexpr uint32_t kManySlots = 0x80000000u;

// Partial sums of a frame of N nodes, functions of N alone (a member of a batch
// sums as it does alone): one per gather workgroup of kMfWaves rows, the rows
// past kMfGroups of them wrapping around, and one per update workgroup.
__host__ __device__ inline uint32_t mf_partials(uint32_t nodes) {
    const uint32_t g = (nodes + kMfWaves - 1) / kMfWaves;
    return g < kMfGroups ? g : kMfGroups;
}
__host__ __device__ inline uint32_t mf_delta_partials(uint32_t nodes) { return (nodes + kMfNodes - 1) / kMfNodes; }

// Value a (lanes 8 k + a, a < 6) of one node's 6-vector, seen by its lanes.
__device__ inline double node_lane(double v, uint32_t a) { return __shfl(v, (int)((threadIdx.x & 56u) + a), 64); }

// Lane a's component of M^-1 v for the 32-bit vector v.
__device__ inline float lane_minv(const Buffers& b, uint32_t n, float v, uint32_t a) {
    const double* M = b.diag_inv64 + 36 * (size_t)n + 6 * (a < 6 ? a : 0);
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 6; ++k) s += M[k] * node_lane(v, k);
    return (float)s;
}

// The node records read by the terms of iteration k (k & 1): s 0..5, d_{k-1}
// 6..11, node 12..14; the other set receives d_k and s_{k+1}.
constexpr uint32_t kNodeRec = 16;
__device__ inline float* node_recs(const Buffers& b, uint32_t set) { return set & 1 ? b.mf_rec[1] : b.mf_rec[0]; }

// kStart: r = b, d_0 = M^-1 b, x = 0, delta_0.  Otherwise iteration k:
// alpha = delta_k / dot(d, q); x += alpha d; r -= alpha q; s = M^-1 r; delta_{k+1}.
template <bool kStart>
__global__ void __launch_bounds__(256) mf_update_kernel(const Buffers* __restrict__ bs, uint32_t k) {
    const Buffers b = frame_buffers(bs);
    const FrameDev& f = *b.frame;
    double alpha = 0.0;
    if (!kStart) {
        double delta, dq;
        reduce_partials2<double>(slot_ptr(b, kSlotDelta + k), mf_delta_partials(f.N), slot_ptr(b, kSlotDQ + k),
                                 mf_partials(f.N), delta, dq);
        alpha = dq != 0.0 ? delta / dq : 0.0;
    }
    const uint32_t first = blockIdx.x * kMfNodes;
    if (b.counts->error || first >= f.N) return;
    const uint32_t a = threadIdx.x % kMfLanes, n = first + threadIdx.x / kMfLanes;
    const bool own = n < f.N && a < 6;
    const uint32_t nn = n < f.N ? n : f.N - 1;
    const size_t i = 6 * (size_t)nn + (a < 6 ? a : 0);
    float t;
    if (kStart) {
        t = b.jtr[i];
        if (own) b.x[i] = 0.f;
    } else {
        const float x = (float)((double)b.x[i] + alpha * (double)b.d1[i]);
        t = (float)((double)b.r[i] - alpha * (double)b.q[i]);
        if (own) b.x[i] = x;
    }
    const float s = lane_minv(b, nn, t, a);
    if (own) {
        b.r[i] = t;
        if (kStart) {
            node_recs(b, 0)[kNodeRec * (size_t)nn + 6 + a] = s;
            if (a < 3) {
                const float4 g = f.nodes[nn];
                const float ga = a == 0 ? g.x : a == 1 ? g.y : g.z;
                node_recs(b, 0)[kNodeRec * (size_t)nn + 12 + a] = ga;
                node_recs(b, 1)[kNodeRec * (size_t)nn + 12 + a] = ga;
            }
        } else {
            node_recs(b, k + 1)[kNodeRec * (size_t)nn + a] = s;
        }
    }
    write_partial<double>(b, kStart ? kSlotDelta : kSlotDelta + k + 1, own ? (double)t * (double)s : 0.0);
}

// x += (num / den) z of a refinement step.
__global__ void __launch_bounds__(256) mf_refine_step_kernel(const Buffers* __restrict__ bs) {
    const Buffers b = frame_buffers(bs);
    const FrameDev& f = *b.frame;
    double num, den;
    const uint32_t parts = mf_partials(f.N);
    reduce_partials2<double>(slot_ptr(b, kSlotRefNum), parts, slot_ptr(b, kSlotRefDen), parts, num, den);
    if (b.counts->error) return;
    const double a = den > 0.0 ? num / den : 0.0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < 6 * f.N; i += gridDim.x * blockDim.x)
        b.x[i] = (float)((double)b.x[i] + a * (double)b.d1[i]);
}

// Node2Term entries as (term | kManySlots, slot weight of the entry's node; an
// edge's entries 1 at its first node, 0 at its second).
__global__ void __launch_bounds__(256) mf_entries_kernel(const Buffers* __restrict__ bs) {
    const Buffers b = frame_buffers(bs);
    const FrameDev& f = *b.frame;
    const Counts& c = *b.counts;
    if (c.error) return;
    const TermBounds tb(c);
    const uint32_t lane = threadIdx.x & 63, waves = gridDim.x * (blockDim.x / 64);
    for (uint32_t i = blockIdx.x * (blockDim.x / 64) + (threadIdx.x >> 6); i < f.N; i += waves) {
        const uint32_t beg = b.n2t_offset[i], end = b.n2t_offset[i + 1];
        for (uint32_t e = beg + lane; e < end; e += 64) {
            const uint32_t t = b.n2t_index[e];
            uint32_t kk, many;
            float wi;
            const int type = type_of(tb, t, kk);
            if (type == kSmooth) {
                const ushort2 ij = f.graph[kk];
                wi = ij.x == i ? 1.f : 0.f;
                many = ij.x == ij.y ? kManySlots : 0u;
            } else {
                ushort4 knn;
                float4 wk;
                term_knn(b, type, kk, knn, wk);
                wi = slot_weight(knn, wk, i);
                many = (knn.x == i) + (knn.y == i) + (knn.z == i) + (knn.w == i) > 1 ? kManySlots : 0u;
            }
            b.mf_ent[e] = make_uint2(t | many, __float_as_uint(wi));
        }
    }
}

// J rows and lambda^2 of a knn term from its record.
__device__ inline int stored_rows(const Buffers& b, int type, uint32_t kk, const MfLambda2& l2, bool density, float J[3][6],
                                  float lam[3]) {
    if (type == kDense || type == kForeground) {
        const ScalarRec& rec = type == kDense ? b.dense[kk] : b.fg[kk];
#pragma unroll
        for (int q = 0; q < 6; ++q) J[0][q] = rec.J[q];
        lam[0] = type == kDense ? 1.f : l2.foreground;
        if (type == kDense && density) {
            const ScalarRec& d = b.density[kk];
#pragma unroll
            for (int q = 0; q < 6; ++q) J[1][q] = d.J[q];
            lam[1] = l2.density;
            return 2;
        }
        return 1;
    }
    const P2PRec& rec = type == kFeature ? b.feat[kk] : b.cross[kk];
    float res[3];
    p2p_rows(rec, J, res);
    const uint32_t mask = type == kFeature ? 0xFFFFFFFFu : 0u;
    lam[0] = lam[1] = lam[2] = __uint_as_float((__float_as_uint(l2.feature) & mask) | (__float_as_uint(l2.cross) & ~mask));
    return 3;
}

// kSrc kSrcDir: V from the direction of iteration k, also stored (d1, and the
// records of the next iteration); kSrcX, kSrcZ: from x or d1; kSrcRows: u_t from
// mf_u (debug).  Stored J: u_t to mf_u.  Recomputed J: kOutG g_t, kOutRows u_t.
// An edge of the recomputing apply leaves lambda^2 u and its two lever arms
// (zero when it is not valid) for the gather: mf_g = (u, valid; a), mf_edge = b.
template <bool kRecompute, int kSrc, int kOut>
__global__ void __launch_bounds__(256) mf_apply_terms_kernel(const Buffers* __restrict__ bs, uint32_t k, Penalty pen,
                                                             uint32_t which) {
    const Buffers b = frame_buffers(bs);
    const FrameDev& f = *b.frame;
    const Counts& c = *b.counts;
    if (c.error) return;
    double beta = 0.0, num = 0.0, den = 0.0;
    if (kSrc == kSrcDir && k > 0) {
        const uint32_t parts = mf_delta_partials(f.N);
        partials_sum2<double>(slot_ptr(b, kSlotDelta + k), parts, slot_ptr(b, kSlotDelta + k - 1), parts, num, den);
    }
    const DQ* __restrict__ se3 = which ? b.se3[1] : b.se3[0];
    const float4* __restrict__ recs = reinterpret_cast<const float4*>(node_recs(b, k));
    const float* __restrict__ vec = kSrc == kSrcX ? b.x : b.d1;
    // the source vector at node n, node-centred
    auto source = [&](uint32_t n, float v[6], float4& g) {
        if (kSrc == kSrcDir) {
            const float4 q0 = recs[4 * (size_t)n], q1 = recs[4 * (size_t)n + 1], q2 = recs[4 * (size_t)n + 2];
            g = recs[4 * (size_t)n + 3];
            const float sv[6] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y};
            const float pv[6] = {q1.z, q1.w, q2.x, q2.y, q2.z, q2.w};
#pragma unroll
            for (int a = 0; a < 6; ++a) v[a] = k > 0 ? (float)((double)sv[a] + beta * (double)pv[a]) : pv[a];
        } else {
            g = f.nodes[n];
            const float2* p = reinterpret_cast<const float2*>(vec + 6 * (size_t)n);
            const float2 p0 = p[0], p1 = p[1], p2 = p[2];
            v[0] = p0.x; v[1] = p0.y; v[2] = p1.x; v[3] = p1.y; v[4] = p2.x; v[5] = p2.y;
        }
    };
    const TermBounds tb(c);
    const MfLambda2 l2 = mf_lambda2(pen);
    const bool density = b.density && pen.density != 0.f;
    const uint32_t total = c.off[4];
    const uint32_t stride = gridDim.x * blockDim.x;
    // a term's rows, which do not depend on the source ...
    struct Rows {
        int type, rows;
        uint32_t kk;
        ushort4 knn;
        float4 wk;
        float J[3][6], lam[3];
        SmoothRec sm;
    };
    auto rows_of = [&](uint32_t t, Rows& r) {
        r.type = type_of(tb, t, r.kk);
        if (r.type == kSmooth) {
            r.sm = kRecompute ? eval_smooth<double>(f, se3, r.kk) : b.smooth[r.kk];
        } else {
            term_knn(b, r.type, r.kk, r.knn, r.wk);
            r.rows = kRecompute ? knn_term_rows<double>(b, f, se3, r.type, r.kk, l2, density, r.J, r.lam)
                                : stored_rows(b, r.type, r.kk, l2, density, r.J, r.lam);
        }
    };
    // ... and their product with it
    auto apply_rows = [&](uint32_t t, const Rows& r) {
        float u[3] = {0.f, 0.f, 0.f};
        float4 g0 = make_float4(0.f, 0.f, 0.f, 0.f), g1 = g0;
        if (kSrc == kSrcRows) {
            const float4 ut = b.mf_u[t];
            u[0] = ut.x;
            u[1] = ut.y;
            u[2] = ut.z;
        }
        if (r.type == kSmooth) {
            const SmoothRec& sm = r.sm;
            const float l = kSrc == kSrcRows ? 1.f : l2.smooth;
            if (kSrc != kSrcRows) {
                const uint32_t n1 = sm.ij & 0xFFFF, n2 = sm.ij >> 16;
                float J1[3][6], J2[3][6], res[3], v[6], w1[6], w2[6];
                float4 g;
                smooth_rows(sm, true, J1, res);
                smooth_rows(sm, n2 == n1, J2, res);
                source(n1, v, g);
                node_to_ref(g, v, w1);
                source(n2, v, g);
                node_to_ref(g, v, w2);
                if (kRecompute) {
#pragma unroll
                    for (int q = 0; q < 3; ++q) u[q] = dot6(J1[q], w1) + dot6(J2[q], w2);
                } else {
#pragma unroll
                    for (int q = 0; q < 3; ++q) u[q] = l * (dot6(J1[q], w1) + dot6(J2[q], w2));
                }
            }
            if (kRecompute && kOut == kOutG) {
                const float on = sm.valid ? 1.f : 0.f;
                g0 = make_float4(l * u[0], l * u[1], l * u[2], on);
                g1 = make_float4(on * sm.Ti_xj[0], on * sm.Ti_xj[1], on * sm.Ti_xj[2], 0.f);
                b.mf_edge[r.kk] = make_float4(on * (sm.Ti_xj[0] - sm.r[0]), on * (sm.Ti_xj[1] - sm.r[1]),
                                              on * (sm.Ti_xj[2] - sm.r[2]), 0.f);
            }
        } else {
            if (kSrc != kSrcRows) {
                // sum_k w_k T_k v_k over the knn slots (slot-rule weights)
                float V[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                const uint32_t n[4] = {r.knn.x, r.knn.y, r.knn.z, r.knn.w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float v[6], w6[6];
                    float4 g;
                    source(n[q], v, g);
                    node_to_ref(g, v, w6);
                    const float ws = slot_weight(r.knn, r.wk, n[q]);
#pragma unroll
                    for (int a = 0; a < 6; ++a) V[a] += ws * w6[a];
                }
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    if (q < r.rows) u[q] = kRecompute ? dot6(r.J[q], V) : r.lam[q] * dot6(r.J[q], V);
            }
            if (kRecompute && kOut == kOutG) {
                float g[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    if (q < r.rows) {
                        const float s = (kSrc == kSrcRows ? 1.f : r.lam[q]) * u[q];
#pragma unroll
                        for (int a = 0; a < 6; ++a) g[a] += s * r.J[q][a];
                    }
                }
                g0 = make_float4(g[0], g[1], g[2], g[3]);
                g1 = make_float4(g[4], g[5], 0.f, 0.f);
            }
        }
        if (kRecompute && kOut == kOutG) {
            b.mf_g[2 * (size_t)t] = g0;
            b.mf_g[2 * (size_t)t + 1] = g1;
        } else {
            b.mf_u[t] = make_float4(u[0], u[1], u[2], 0.f);
        }
    };
    uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    Rows rows;
    if (t < total) rows_of(t, rows);  // the first term's rows overlap the reduction
    if (kSrc == kSrcDir && k > 0) {
        double s0, s1;
        partials_finish2<double>(num, den, s0, s1);
        beta = s1 != 0.0 ? s0 / s1 : 0.0;
    }
    while (t < total) {
        apply_rows(t, rows);
        t += stride;
        if (t < total) rows_of(t, rows);
    }
    if (kSrc == kSrcDir) {
        float* next = node_recs(b, k + 1);
        for (uint32_t n = blockIdx.x * blockDim.x + threadIdx.x; n < f.N; n += stride) {
            float v[6];
            float4 g;
            source(n, v, g);
#pragma unroll
            for (int a = 0; a < 6; ++a) {
                b.d1[6 * (size_t)n + a] = v[a];
                next[kNodeRec * (size_t)n + 6 + a] = v[a];
            }
        }
    }
}

// y_i over the Node2Term list of row i, then the epilogue: kEpiSpmv (v = d):
// q and dot(d, q) of iteration k; kEpiResidual (v = x): r = b - A x, z = M^-1 r to
// d1, (r, z); kEpiCurvature (v = z): (z, A z); kEpiAdjoint: the gather's sum to q.
template <bool kRecompute, int kEpi>
__global__ void __launch_bounds__(64 * kMfWaves) mf_apply_gather_kernel(const Buffers* __restrict__ bs, uint32_t k, Penalty pen) {
    const Buffers b = frame_buffers(bs);
    const FrameDev& f = *b.frame;
    const Counts& c = *b.counts;
    // XCD-aware rows: neighbouring rows share terms and stay in one L2
    const uint32_t group = xcd_remap(blockIdx.x, gridDim.x, mf_partials(f.N));
    if (c.error || group == 0xFFFFFFFFu) return;
    const uint32_t lane = threadIdx.x & 63, a = threadIdx.x % kMfLanes;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const float* __restrict__ vec = kEpi == kEpiResidual ? b.x : b.d1;
    constexpr bool correct = kEpi != kEpiAdjoint;
    const TermBounds tb(c);
    const MfLambda2 l2 = mf_lambda2(pen);
    const bool density = b.density && pen.density != 0.f;
    double acc = 0.0;
    for (uint32_t i = group * kMfWaves + wave; i < f.N; i += kMfGroups * kMfWaves) {
        const uint32_t beg = b.n2t_offset[i], end = b.n2t_offset[i + 1];
        const float4 g = f.nodes[i];
        float vi[6], tv[6];
#pragma unroll
        for (int q = 0; q < 6; ++q) vi[q] = correct ? vec[6 * (size_t)i + q] : 0.f;
        node_to_ref(g, vi, tv);
        double y[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // kRecompute: in reference coordinates until the row is complete
        // the next round's entries load while this round's terms do
        uint2 next = beg + lane < end ? b.mf_ent[beg + lane] : make_uint2(0u, 0u);
        for (uint32_t e = beg + lane; e < end; e += 64) {
            const uint2 ent = next;
            if (e + 64 < end) next = b.mf_ent[e + 64];
            const uint32_t t = ent.x & ~kManySlots;
            const bool many = (ent.x & kManySlots) != 0;
            const float wi = __uint_as_float(ent.y);
            uint32_t kk;
            const int type = type_of(tb, t, kk);
            if (kRecompute) {
                const float4 g0 = b.mf_g[2 * (size_t)t], g1 = b.mf_g[2 * (size_t)t + 1];
                if (type == kSmooth) {
                    // J^T u of one end: rotation p x u, translation u, opposite signs
                    const bool first = wi != 0.f;
                    const float4 p = first ? g1 : b.mf_edge[kk];
                    const float sg = first ? 1.f : -1.f;
                    const float J[3][6] = {{0.f, sg * p.z, -sg * p.y, g0.w * sg, 0.f, 0.f},
                                           {-sg * p.z, 0.f, sg * p.x, 0.f, g0.w * sg, 0.f},
                                           {sg * p.y, -sg * p.x, 0.f, 0.f, 0.f, g0.w * sg}};
                    const float u[3] = {g0.x, g0.y, g0.z};
#pragma unroll
                    for (int r = 0; r < 3; ++r) {
                        float s = u[r];
                        if (correct && many) s -= l2.smooth * dot6(J[r], tv);
#pragma unroll
                        for (int q = 0; q < 6; ++q) y[q] += (double)(s * J[r][q]);
                    }
                } else {
                    const float gv[6] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y};
#pragma unroll
                    for (int q = 0; q < 6; ++q) y[q] += (double)(wi * gv[q]);
                    if (correct && many) {
                        // (m - 1) w^2 J^T J v less, J as the evaluation pass stored it
                        ushort4 knn;
                        float4 wk;
                        term_knn(b, type, kk, knn, wk);
                        const uint32_t mult = (knn.x == i) + (knn.y == i) + (knn.z == i) + (knn.w == i);
                        float J[3][6], lam[3];
                        const int rows = stored_rows(b, type, kk, l2, density, J, lam);
#pragma unroll
                        for (int r = 0; r < 3; ++r) {
                            if (r < rows) {
                                const float s = -(float)(mult - 1) * lam[r] * wi * wi * dot6(J[r], tv);
#pragma unroll
                                for (int q = 0; q < 6; ++q) y[q] += (double)(s * J[r][q]);
                            }
                        }
                    }
                }
            } else {
                const float4 ut = b.mf_u[t];
                const float u[3] = {ut.x, ut.y, ut.z};
                float J[3][6], lam[3], w = 1.f;
                uint32_t mult = 1;
                int rows = 3;
                if (type == kSmooth) {
                    float res[3];
                    smooth_rows(b.smooth[kk], wi != 0.f, J, res);
                    lam[0] = lam[1] = lam[2] = l2.smooth;
                    if (many) mult = 2;
                } else {
                    rows = stored_rows(b, type, kk, l2, density, J, lam);
                    w = wi;
                    if (many) {
                        ushort4 knn;
                        float4 wk;
                        term_knn(b, type, kk, knn, wk);
                        mult = (knn.x == i) + (knn.y == i) + (knn.z == i) + (knn.w == i);
                    }
                }
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    if (r < rows) {
                        to_node_frame(J[r], g);
                        float s = w * u[r];
                        if (mult > 1) s -= (float)(mult - 1) * lam[r] * w * w * dot6(J[r], vi);
#pragma unroll
                        for (int q = 0; q < 6; ++q) y[q] += (double)(s * J[r][q]);
                    }
                }
            }
        }
        reduce_half<4>(y);
        reduce_half<2>(y);
        reduce_half<1>(y);
        double ya = y[0];  // component a over the lanes 8 k + a
        ya += lane_xor<8>(ya);
        ya += lane_xor<16>(ya);
        ya += lane_xor<32>(ya);
        if (kRecompute) {
            // to node-centred coordinates: T^T (r, t) = (r + t x g, t)
            const double t0 = node_lane(ya, 3), t1 = node_lane(ya, 4), t2 = node_lane(ya, 5);
            ya += a == 0 ? t1 * g.z - t2 * g.y : a == 1 ? t2 * g.x - t0 * g.z : a == 2 ? t0 * g.y - t1 * g.x : 0.0;
        }
        if (correct) {
            // damping 1e-2 T^T T v: T v = (w, v + g x w), T^T (a, b) = (a + b x g, b)
            const float bx = tv[4] * g.z - tv[5] * g.y, by = tv[5] * g.x - tv[3] * g.z, bz = tv[3] * g.y - tv[4] * g.x;
            const float damp[6] = {tv[0] + bx, tv[1] + by, tv[2] + bz, tv[3], tv[4], tv[5]};
            const float da = a == 0 ? damp[0] : a == 1 ? damp[1] : a == 2 ? damp[2] : a == 3 ? damp[3] : a == 4 ? damp[4] : damp[5];
            ya += (double)(1e-2f * da);
        }
        const float va = a == 0 ? vi[0] : a == 1 ? vi[1] : a == 2 ? vi[2] : a == 3 ? vi[3] : a == 4 ? vi[4] : vi[5];
        const size_t ka = 6 * (size_t)i + (a < 6 ? a : 0);
        const bool own = lane < 6;
        if (kEpi == kEpiSpmv || kEpi == kEpiAdjoint) {
            if (own) b.q[ka] = (float)ya;
            acc += own ? (double)va * ya : 0.0;
        } else if (kEpi == kEpiResidual) {
            const float rr = (float)((double)b.jtr[ka] - ya), z = lane_minv(b, i, rr, a);
            if (own) {
                b.r[ka] = rr;
                b.d1[ka] = z;
            }
            acc += own ? (double)rr * (double)z : 0.0;
        } else {
            acc += own ? (double)va * ya : 0.0;
        }
    }
    if (kEpi == kEpiAdjoint) return;
    // the waves' sums in order
    __shared__ double part[kMfWaves];
    acc = wave_sum(acc);
    if (lane == 0) part[wave] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < (int)kMfWaves; ++w) s += part[w];
        slot_ptr(b, kEpi == kEpiSpmv ? kSlotDQ + k : kEpi == kEpiResidual ? kSlotRefNum : kSlotRefDen)[group] = s;
    }
}

// ------------------------------------------------------------- host launch
void launch_pcg_init(const Batch& B, hipStream_t stream);
void launch_pcg_update(const Batch& B, uint32_t k, uint32_t spmv_blocks, uint32_t dsel, hipStream_t stream);
void launch_refine_step(const Batch& B, uint32_t spmv_blocks, hipStream_t stream);
uint32_t row_group_grid(uint32_t nodes);

static uint32_t term_grid(const Batch& B) { return std::min<uint32_t>(std::max<uint32_t>(64 * B.nodes / 256, 64), 2048); }
// Gather workgroups: one per partial of the largest frame, a multiple of the XCD count.
static uint32_t gather_grid(const Batch& B) { return (mf_partials(B.nodes) + kXcds - 1) / kXcds * kXcds; }

// ------------------------------------------------ FP32 mode
static void mf_apply(const Batch& B, int src_epi, uint32_t k, uint32_t cur, const Penalty& pen, hipStream_t stream) {
    const dim3 tg(term_grid(B), B.frames), sg(row_group_grid(B.nodes), B.frames), wg(256);
    if (src_epi == 0) {
        hipLaunchKernelGGL((mf_terms_kernel<kSrcDir>), tg, wg, 0, stream, B.dev, k, cur, pen);
        hipLaunchKernelGGL((mf_gather_kernel<kEpiSpmv>), sg, wg, 0, stream, B.dev, k, cur, pen);
    } else if (src_epi == 1) {
        hipLaunchKernelGGL((mf_terms_kernel<kSrcX>), tg, wg, 0, stream, B.dev, k, cur, pen);
        hipLaunchKernelGGL((mf_gather_kernel<kEpiResidual>), sg, wg, 0, stream, B.dev, k, cur, pen);
    } else {
        hipLaunchKernelGGL((mf_terms_kernel<kSrcZ>), tg, wg, 0, stream, B.dev, k, cur, pen);
        hipLaunchKernelGGL((mf_gather_kernel<kEpiCurvature>), sg, wg, 0, stream, B.dev, k, cur, pen);
    }
}

static void mfr_apply(const Batch& B, int src_epi, uint32_t k, uint32_t cur, const Penalty& pen, uint32_t which,
                      hipStream_t stream) {
    const dim3 tg(term_grid(B), B.frames), sg(row_group_grid(B.nodes), B.frames), wg(256);
    if (src_epi == 0) {
        hipLaunchKernelGGL((mfr_terms_kernel<kSrcDir, kOutG>), tg, wg, 0, stream, B.dev, k, cur, pen, which);
        hipLaunchKernelGGL((mfr_gather_kernel<kEpiSpmv>), sg, wg, 0, stream, B.dev, k, cur, pen, which);
    } else if (src_epi == 1) {
        hipLaunchKernelGGL((mfr_terms_kernel<kSrcX, kOutG>), tg, wg, 0, stream, B.dev, k, cur, pen, which);
        hipLaunchKernelGGL((mfr_gather_kernel<kEpiResidual>), sg, wg, 0, stream, B.dev, k, cur, pen, which);
    } else {
        hipLaunchKernelGGL((mfr_terms_kernel<kSrcZ, kOutG>), tg, wg, 0, stream, B.dev, k, cur, pen, which);
        hipLaunchKernelGGL((mfr_gather_kernel<kEpiCurvature>), sg, wg, 0, stream, B.dev, k, cur, pen, which);
    }
}

static void apply_fp32(const Batch& B, bool recompute, int src_epi, uint32_t k, uint32_t cur, const Penalty& pen,
                       uint32_t which, hipStream_t stream) {
    if (recompute) mfr_apply(B, src_epi, k, cur, pen, which, stream);
    else mf_apply(B, src_epi, k, cur, pen, stream);
}

// ------------------------------------------------ mixed mode
// Workgroups of a term launch over all frames, six to a CU, shared by the frames of a
// batch: a workgroup forms the iteration's scalars from all partials before its terms,
// and a frame's 160k terms fill a few hundred of them.  A lone frame takes
// 1024 (a term or two a thread: 300 nodes 1090 us a solve, 75 workgroups 1143).  Batches
// with 1024 a frame, and with their share (stored / recomputed J, ms a solve, two
// 320x240 views, 3 GN x 10 PCG): 32 frames of 600 nodes 5.12 / 6.28 and 4.15 / 4.79, 16 of
// 2000 3.44 / 4.06 and 2.95 / 3.41, 4 of 8000 2.36 / 2.59 and 2.19 / 2.28.
constexpr uint32_t kTermWorkgroups = 6 * 256;
static uint32_t mixed_term_grid(const Batch& B) {
    return std::max<uint32_t>(64, std::min<uint32_t>(1024, kTermWorkgroups / B.frames));
}
template <int kSrc, int kEpi>
static void apply_mixed(const Batch& B, bool recompute, uint32_t k, const Penalty& pen, uint32_t which,
                        hipStream_t stream) {
    const dim3 tg(mixed_term_grid(B), B.frames), gg(gather_grid(B), B.frames), wg(256), ww(64 * kMfWaves);
    if (recompute) {
        hipLaunchKernelGGL((mf_apply_terms_kernel<true, kSrc, kOutG>), tg, wg, 0, stream, B.dev, k, pen, which);
        hipLaunchKernelGGL((mf_apply_gather_kernel<true, kEpi>), gg, ww, 0, stream, B.dev, k, pen);
    } else {
        hipLaunchKernelGGL((mf_apply_terms_kernel<false, kSrc, kOutG>), tg, wg, 0, stream, B.dev, k, pen, which);
        hipLaunchKernelGGL((mf_apply_gather_kernel<false, kEpi>), gg, ww, 0, stream, B.dev, k, pen);
    }
}

// Block-Jacobi PCG with the matrix-free apply.
void launch_pcg_matrix_free(const Batch& B, uint32_t iters, uint32_t refine, bool fp64, const Penalty& pen,
                            bool recompute, uint32_t which, hipStream_t stream) {
    iters = std::min(iters, kMaxIters);
    if (fp64) {
        const dim3 ug(mf_delta_partials(B.nodes), B.frames);
        hipLaunchKernelGGL(mf_update_kernel<true>, ug, dim3(256), 0, stream, B.dev, 0u);
        for (uint32_t k = 0; k < iters; ++k) {
            apply_mixed<kSrcDir, kEpiSpmv>(B, recompute, k, pen, which, stream);
            hipLaunchKernelGGL(mf_update_kernel<false>, ug, dim3(256), 0, stream, B.dev, k);
        }
        for (uint32_t r = 0; r < refine; ++r) {
            apply_mixed<kSrcX, kEpiResidual>(B, recompute, 0, pen, which, stream);
            apply_mixed<kSrcZ, kEpiCurvature>(B, recompute, 0, pen, which, stream);
            hipLaunchKernelGGL(mf_refine_step_kernel, dim3(kVecBlocks, B.frames), dim3(256), 0, stream, B.dev);
        }
        return;
    }
    // FP32: per iteration the term pass, the gather (q = A d, dot(d, q)) and
    // the update of the materialized path
    const uint32_t sg = row_group_grid(B.nodes);
    launch_pcg_init(B, stream);
    uint32_t cur = 0;
    for (uint32_t k = 0; k < iters; ++k) {
        apply_fp32(B, recompute, 0, k, cur, pen, which, stream);
        cur ^= 1;
        launch_pcg_update(B, k, sg, cur, stream);
    }
    for (uint32_t r = 0; r < refine; ++r) {
        apply_fp32(B, recompute, 1, 0, 0, pen, which, stream);
        apply_fp32(B, recompute, 2, 0, 0, pen, which, stream);
        launch_refine_step(B, sg, stream);
    }
}

// One matrix-free apply q = A d (stage timing), d as the last PCG left it.
void launch_mf_apply_once(const Batch& B, bool fp64, const Penalty& pen, bool recompute, uint32_t which,
                          hipStream_t stream) {
    if (fp64) apply_mixed<kSrcDir, kEpiSpmv>(B, recompute, 0, pen, which, stream);
    else apply_fp32(B, recompute, 0, 0, 0, pen, which, stream);
}

// One PCG update of the mixed matrix-free solve (stage timing).
void launch_mf_update_once(const Batch& B, hipStream_t stream) {
    hipLaunchKernelGGL(mf_update_kernel<false>, dim3(mf_delta_partials(B.nodes), B.frames), dim3(256), 0, stream, B.dev, 0u);
}

// The entry weights the matrix-free applies read (fixed by the index build).
void launch_mf_entries(const Batch& B, bool fp64, bool recompute, hipStream_t stream) {
    const dim3 sg(row_group_grid(B.nodes), B.frames);
    if (fp64) hipLaunchKernelGGL(mf_entries_kernel, dim3((B.nodes + 3) / 4, B.frames), dim3(256), 0, stream, B.dev);
    else if (recompute) hipLaunchKernelGGL(mf_entry_weights_kernel, sg, dim3(256), 0, stream, B.dev);
}

// The term Jacobian at se3[which] with unit weights, recomputed from the maps:
// transpose 0: mf_u = J x for x (reference twists) in d1 (d1 is overwritten);
// transpose 1: q = J^T y (reference twists) for y in mf_u.
void launch_debug_jacobian(const Batch& B, bool fp64, bool transpose, uint32_t which, hipStream_t stream) {
    const Penalty unit{1.f, 1.f, 1.f, 1.f, 1.f};
    const dim3 tg(term_grid(B), B.frames), sg(row_group_grid(B.nodes), B.frames), vg((B.nodes + 255) / 256, B.frames), wg(256);
    if (fp64) {
        if (!transpose) {
            hipLaunchKernelGGL(mfr_coords_kernel, vg, wg, 0, stream, B.dev, 0);
            hipLaunchKernelGGL((mf_apply_terms_kernel<true, kSrcZ, kOutRows>), tg, wg, 0, stream, B.dev, 0u, unit, which);
        } else {
            hipLaunchKernelGGL((mf_apply_terms_kernel<true, kSrcRows, kOutG>), tg, wg, 0, stream, B.dev, 0u, unit, which);
            hipLaunchKernelGGL((mf_apply_gather_kernel<true, kEpiAdjoint>), dim3(gather_grid(B), B.frames),
                               dim3(64 * kMfWaves), 0, stream, B.dev, 0u, unit);
            hipLaunchKernelGGL(mfr_coords_kernel, vg, wg, 0, stream, B.dev, 1);
        }
        return;
    }
    if (!transpose) {
        hipLaunchKernelGGL(mfr_coords_kernel, vg, wg, 0, stream, B.dev, 0);
        hipLaunchKernelGGL((mfr_terms_kernel<kSrcZ, kOutRows>), tg, wg, 0, stream, B.dev, 0u, 0u, unit, which);
        return;
    }
    hipLaunchKernelGGL((mfr_terms_kernel<kSrcRows, kOutG>), tg, wg, 0, stream, B.dev, 0u, 0u, unit, which);
    hipLaunchKernelGGL((mfr_gather_kernel<kEpiAdjoint>), sg, wg, 0, stream, B.dev, 0u, 0u, unit, which);
    hipLaunchKernelGGL(mfr_coords_kernel, vg, wg, 0, stream, B.dev, 1);
}

}  // namespace mvdr
