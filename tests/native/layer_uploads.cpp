// New batches through the C++ layer class without a GPU (host_stub.c preloaded): pinned memory, a staging copy and threads
// are made for the second batch, and where they cannot be had every batch is copied as it is; batches from two threads.
#include <cassert>
#include <thread>
#include <vector>

#include "../../tcbnn_amd/host/tcbnn_layers.hpp"

extern "C" {
extern int stub_host_mallocs_left, stub_mallocs_left, stub_threads_left, stub_allocations;
}

static const int kBatch = 8, kSize = 224, kFloats = kBatch * 3 * kSize * kSize;

static std::vector<float> batch(int seed) {
    std::vector<float> v(kFloats);
    for (int i = 0; i < kFloats; ++i) v[i] = (float)((i * 7919 + seed * 104729) % 1000) / 1000.0f - 0.5f;
    return v;
}

int main() {
    int* const knobs[] = {nullptr, &stub_host_mallocs_left, &stub_mallocs_left, &stub_threads_left};
    for (int save = 0; save < 2; ++save)
        for (int* knob : knobs) {
            InConv128LayerParam layer("Conv1", kSize, kSize, 3, 3, 3, 64, kBatch, 1, 1, true, 1, 1, save != 0);
            SAFE_ALOC_GPU(layer.input_gpu, layer.input_bytes());
            SAFE_ALOC_GPU(layer.output_residual_gpu, 4);
            layer.residual_info = tcbnn_host::make_residual_info(64, 2000, kBatch);
            const int before = stub_allocations;
            std::vector<float> x = batch(1);
            layer.set_input(x.data());
            assert(memcmp(layer.input_gpu, x.data(), 4 * (size_t)kFloats) == 0 && stub_allocations == before);
            if (knob != nullptr) *knob = 0;
            for (int k = 2; k < 5; ++k) {
                x = batch(k);
                layer.set_input(x.data());
                assert(memcmp(layer.input_gpu, x.data(), 4 * (size_t)kFloats) == 0);
            }
            if (knob != nullptr) *knob = -1;
            std::vector<float> a = batch(10), b = batch(11);
            std::thread t([&] {
                for (int k = 0; k < 20; ++k) layer.set_input(a.data());
            });
            for (int k = 0; k < 20; ++k) layer.set_input(b.data());
            t.join();
            assert(memcmp(layer.input_gpu, a.data(), 4 * (size_t)kFloats) == 0 || memcmp(layer.input_gpu, b.data(), 4 * (size_t)kFloats) == 0);
        }
    puts("done");
    return 0;
}
