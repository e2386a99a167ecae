// Host-side check of the chunk queue (ataraxia_amd/csrc/wavefront.h): the
// counters' chunks and the waves' first ones are all chunks, each once; the
// jobs per chunk chosen per launch (launch_chunk_px); the counter lines' sums.
// Built host-only (hipcc --offload-host-only) by tests/test_queue_host.py.
#include <cstdio>
#include <vector>

#include "device_types.h"
#include "wavefront_host.h"

using namespace atx;

int main()
{
    int bad = 0;
    for (uint32_t waves : {4u, 12u, 5120u})
        for (uint32_t chunks : {1u, 4u, 13u, 5119u, 5120u, 5121u, 5140u, 20000u}) {
            std::vector<int> seen(chunks, 0);
            for (uint32_t w = 0; w < waves && w < chunks; ++w)
                seen[w]++;
            for (uint32_t k = 0; k < kQueueShards; ++k)
                for (uint32_t i = 0; queue_chunk(k, i, waves) < chunks; ++i)
                    seen[queue_chunk(k, i, waves)]++;
            for (int s : seen)
                bad += s != 1;
        }
    // 1280 workgroups: 5120 waves
    const struct { uint64_t jobs; bool flat; uint32_t px; } rule[] = {
        {0, false, 64},  {5120 * 512 - 1, false, 64}, {5120 * 512, false, 128}, {5120 * 4000, false, 256},
        {5120 * 5000, false, 512}, {5120 * 16 - 1, true, 64}, {5120 * 16, true, 128}, {5120 * 64, true, 256},
        {5120 * 256, true, 512}, {1ull << 31, true, 512}};
    for (const auto& r : rule)
        bad += launch_chunk_px(r.jobs, 1280, r.flat) != r.px;
    bad += launch_chunk_px(1, 0, false) != 64;
    std::vector<unsigned long long> lines(kCounterWords, 0);
    for (uint32_t i = 0; i < kCounterLines; ++i)
        lines[i * kCounterStride + kCtrBoxes] = 1ull << (2 * i + 20);
    bad += counter_sum(lines.data(), kCtrBoxes) != 0x5555555500000ull || counter_sum(lines.data(), kCtrRays) != 0;
    std::printf(bad ? "%d checks failed\n" : "all checks passed\n", bad);
    return bad != 0;
}
