// csrc/record_stage.h on the host: the lanes of a wave run one after another from one
// wave_lds_sync() to the next, in ascending or descending order, which is the least
// that the device promises about them.  A lane that reads what another lane has not
// staged yet, or stages over what another has not read, stores a wrong record.
#include <cstdint>
#include <cstring>
#include <condition_variable>
#include <cstdio>
#include <mutex>
#include <thread>
#include <vector>

#define __device__
struct float4 { float x, y, z, w; };
struct ushort4 { uint16_t x, y, z, w; };
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }
inline float __uint_as_float(uint32_t u) { float f; std::memcpy(&f, &u, 4); return f; }
struct Index { uint32_t x; };
static thread_local Index threadIdx;

// The token goes to the lanes in turn, once round per phase.
static std::mutex m;
static std::condition_variable turn;
static long token;
static thread_local long place, phase;
static void wait_turn() {
    std::unique_lock<std::mutex> lock(m);
    turn.wait(lock, [] { return token == phase * 64 + place; });
}
static void pass_turn() {
    {
        std::lock_guard<std::mutex> lock(m);
        ++token;
    }
    turn.notify_all();
}
inline void wave_lds_sync() {
    pass_turn();
    ++phase;
    wait_turn();
}

namespace mvdr {
struct ScalarRec { ushort4 knn; float r; uint32_t pad0; float4 w; float J[6]; float pad1[2]; };
static_assert(sizeof(ScalarRec) == 64, "as in common.h");
}  // namespace mvdr
#include "../multiviewdynrecon_amd/csrc/record_stage.h"

using namespace mvdr;

static ScalarRec record(uint32_t t, int kind) {
    ScalarRec r{};
    r.knn = {(uint16_t)(4 * t), (uint16_t)(4 * t + 1), (uint16_t)(4 * t + 2), (uint16_t)(4 * t + 3)};
    r.w = {t + 0.1f, t + 0.2f, t + 0.3f, t + 0.4f};
    r.r = 1000.f * kind + t;
    for (int k = 0; k < 6; ++k) r.J[k] = 10000.f * kind + 8 * t + k;
    return r;
}

int main() {
    constexpr uint32_t kTerms = 192 + 7;  // three whole waves of terms and a part of one
    for (int descending = 0; descending < 2; ++descending) {
        std::vector<ScalarRec> dense(kTerms), density(kTerms);
        for (uint32_t t = 0; t < kTerms; ++t) {
            dense[t].knn = density[t].knn = record(t, 0).knn;  // the index build's fields
            dense[t].w = density[t].w = record(t, 0).w;
        }
        RecordStage stage;
        std::memset(&stage, 0xEE, sizeof(stage));
        token = 0;
        std::vector<std::thread> lanes;
        for (uint32_t lane = 0; lane < 64; ++lane)
            lanes.emplace_back([&, lane] {
                threadIdx.x = 64 + lane;  // the second wave of its workgroup
                place = descending ? 63 - lane : lane;
                phase = 0;
                wait_turn();
                for (uint32_t t = lane; t < kTerms; t += 64) {  // as the evaluation kernel goes through its terms
                    const uint32_t t0 = t - lane;
                    ScalarRec rec = record(t, 1);
                    stage_weights(stage, rec);
                    store_records(stage, dense.data() + t0, kTerms - t0, rec);
                    rec = record(t, 2);
                    store_records(stage, density.data() + t0, kTerms - t0, rec);
                }
                pass_turn();
            });
        for (std::thread& l : lanes) l.join();
        for (uint32_t t = 0; t < kTerms; ++t) {
            const ScalarRec a = record(t, 1), b = record(t, 2);
            if (std::memcmp(&dense[t], &a, sizeof(a)) || std::memcmp(&density[t], &b, sizeof(b))) {
                std::printf("record %u of %u differs, lanes %s\n", t, kTerms, descending ? "descending" : "ascending");
                return 1;
            }
        }
    }
    return 0;
}
