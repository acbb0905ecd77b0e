// Evaluated records to memory, whole lines at a time.  The including file supplies the
// record type and the wave primitives (common.h, device_util.h).
#pragma once

namespace mvdr {

// A wave's 64 evaluated records, whole lines of 1 KB a store: through LDS, where the
// weights wait as well.  (Each lane storing r and J of its own record touched 64 lines in
// part with every dword.  The evaluation moves ~440 MB a launch of 16 frames, 64 bytes
// read and written per record; 148.6 -> 142 us, a lone frame of 190k terms 13.1 -> 11.9.)
struct RecordStage {
    float4 q[4][64 * 4];
};
__device__ inline float4* staged(RecordStage& stage, uint32_t r, uint32_t chunk) {
    return stage.q[threadIdx.x >> 6] + 4 * r + (chunk + (r >> 1)) % 4;  // rotated: fewer bank conflicts
}
__device__ inline void stage_weights(RecordStage& stage, const ScalarRec& rec) { *staged(stage, threadIdx.x & 63, 1) = rec.w; }
// out: the wave's first record, n of them in the list; a wave that is not all dense
// terms stores its records lane by lane.  The staged path is taken by whole waves; it
// ends with every lane's reads done, so the rows may be staged again.
__device__ inline void store_records(RecordStage& stage, ScalarRec* __restrict__ out, uint32_t n, const ScalarRec& rec) {
    const uint32_t lane = threadIdx.x & 63;
    if (n < 64) {
        out[lane].r = rec.r;
#pragma unroll
        for (int k = 0; k < 6; ++k) out[lane].J[k] = rec.J[k];
        return;
    }
    *staged(stage, lane, 0) = make_float4(__uint_as_float((uint32_t)rec.knn.x | ((uint32_t)rec.knn.y << 16)),
                                          __uint_as_float((uint32_t)rec.knn.z | ((uint32_t)rec.knn.w << 16)), rec.r, 0.f);
    *staged(stage, lane, 2) = make_float4(rec.J[0], rec.J[1], rec.J[2], rec.J[3]);
    *staged(stage, lane, 3) = make_float4(rec.J[4], rec.J[5], 0.f, 0.f);
    wave_lds_sync();  // a lane reads what other lanes staged
#pragma unroll
    for (uint32_t s = 0; s < 4; ++s)
        reinterpret_cast<float4*>(out)[64 * s + lane] = *staged(stage, 16 * s + (lane >> 2), lane & 3);
    wave_lds_sync();  // ... before any lane stages its next record
}

}  // namespace mvdr
