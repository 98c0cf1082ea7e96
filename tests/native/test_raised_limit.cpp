// Two threads raise the limit of one device to different values at the same time; the setter of the smaller value
// takes until the other thread has had every chance to set the larger one.  Prints the limit that is left.
#include "../../mhc.cu_amd/csrc/raised_limit.h"

#include <chrono>
#include <cstdio>
#include <thread>

int main() {
    for (int device : {0, 63, 64}) {
        mhc::RaisedLimit limit;
        std::atomic<int> attribute{0}, calls{0};
        std::atomic<bool> small_inside{false}, large_set{false};
        std::thread small([&] {
            limit.raise(device, 80, [&](int value) {
                small_inside = true;
                for (int i = 0; i < 50 && !large_set; i++) std::this_thread::sleep_for(std::chrono::milliseconds(2));
                attribute = value;
                return calls++ * 0;
            });
        });
        while (!small_inside) std::this_thread::yield();
        std::thread large([&] {
            limit.raise(device, 100, [&](int value) {
                attribute = value;
                large_set = true;
                return calls++ * 0;
            });
        });
        small.join();
        large.join();
        // from here on neither size is set again on a known device, and never a smaller one
        auto set = [&](int value) { attribute = value; return calls++ * 0; };
        limit.raise(device, 100, set);
        limit.raise(device, 80, set);
        if (attribute != 100 || (device < 64 && calls != 2)) {
            std::printf("device %d: limit %d after %d calls\n", device, attribute.load(), calls.load());
            return 1;
        }
        // a setter that fails is asked again
        if (limit.raise(device, 120, [](int) { return 1; }) != 1 || limit.raise(device, 120, set) != 0 || attribute != 120) return 2;
    }
    std::printf("ok\n");
    return 0;
}
