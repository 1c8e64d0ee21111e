// WaveQueue (bg_device.h) on the device: every schedule position goes to exactly
// one lane, with the instance that the schedule names for it, and a lane that
// does not ask keeps its position while others are served.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../bacon_amd/csrc/bg_device.h"

// The lanes of a wave ask at times of their own: lane l is busy for
// 1 + (position * 7 + l) mod 5 rounds with each position.
__global__ void __launch_bounds__(256)
    queue_kernel(uint32_t *counter, uint32_t n, const int32_t *order, uint32_t *taken,
                 int32_t *instance, uint32_t *moved) {
    bg::WaveQueue queue(counter);
    const uint32_t lane = threadIdx.x & 63;
    uint32_t pos = blockIdx.x * blockDim.x + threadIdx.x;
    int64_t inst = queue.start(n, order);
    uint32_t mine = pos, busy = 0;
    bool take = inst >= 0;
    for (;;) {
        if (take) {
            mine = pos;
            busy = 1 + (pos * 7 + lane) % 5;
            atomicAdd(&taken[pos], 1u);
            instance[pos] = (int32_t)inst;
        }
        if (bg::ballot(inst >= 0) == 0) break;
        if (inst >= 0) --busy;
        const bool want = inst >= 0 && busy == 0;
        queue.ticks += 40;  // runs of several lengths
        if (queue.drained()) {
            if (want) inst = -1;
            take = false;
            continue;
        }
        const int64_t got = queue.next(counter, n, order, want, pos);
        if (want) inst = got;
        else if (inst >= 0 && pos != mine) atomicAdd(moved, 1u);
        take = want && inst >= 0;
    }
}

#define CHECK(x)                                                       \
    if ((x) != hipSuccess) {                                           \
        printf("%s: %s\n", #x, hipGetErrorString(hipGetLastError()));  \
        exit(2);                                                       \
    }

int main() {
    int bad = 0;
    for (const bool ordered : {false, true})
        for (const uint32_t n : {1u, 63u, 1024u, 1025u, 1100u, 5000u, 70001u}) {
            const uint32_t blocks = 4, block = 256, lanes = blocks * block;
            std::vector<int32_t> order(n);
            for (uint32_t k = 0; k < n; ++k) order[k] = (int32_t)(n - 1 - k);
            uint32_t *counter, *taken, *moved;
            int32_t *dorder, *instance;
            CHECK(hipMalloc(&counter, 256));
            CHECK(hipMalloc(&moved, 256));
            CHECK(hipMalloc(&taken, n * 4));
            CHECK(hipMalloc(&dorder, n * 4));
            CHECK(hipMalloc(&instance, n * 4));
            CHECK(hipMemcpy(counter, &lanes, 4, hipMemcpyHostToDevice));
            CHECK(hipMemset(moved, 0, 4));
            CHECK(hipMemset(taken, 0, n * 4));
            CHECK(hipMemcpy(dorder, order.data(), n * 4, hipMemcpyHostToDevice));
            queue_kernel<<<blocks, block>>>(n > lanes ? counter : nullptr, n,
                                            ordered ? dorder : nullptr, taken, instance, moved);
            CHECK(hipGetLastError());
            CHECK(hipDeviceSynchronize());
            std::vector<uint32_t> t(n);
            std::vector<int32_t> who(n);
            uint32_t m = 0;
            CHECK(hipMemcpy(t.data(), taken, n * 4, hipMemcpyDeviceToHost));
            CHECK(hipMemcpy(who.data(), instance, n * 4, hipMemcpyDeviceToHost));
            CHECK(hipMemcpy(&m, moved, 4, hipMemcpyDeviceToHost));
            uint32_t wrong = 0;
            for (uint32_t k = 0; k < n; ++k)
                wrong += t[k] != 1 || who[k] != (ordered ? order[k] : (int32_t)k);
            printf("n %u ordered %d: %u positions wrong, %u moved under a busy lane\n", n,
                   (int)ordered, wrong, m);
            bad += wrong != 0 || m != 0;
            CHECK(hipFree(counter));
            CHECK(hipFree(moved));
            CHECK(hipFree(taken));
            CHECK(hipFree(dorder));
            CHECK(hipFree(instance));
        }
    return bad ? 1 : 0;
}
