// LdsGrant (xnor_nn_amd/csrc/plan.hpp) with stand-ins for the two runtime calls it makes: two
// threads ask for different sizes, and the one with more is held up after its size has been set
// until the other one is through, or cannot get through.
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <thread>

#include "plan.hpp"

namespace {
constexpr size_t MORE = 100 << 10, LESS = 80 << 10;
std::mutex mu;
std::condition_variable change;
bool more_set = false, less_asked = false;
size_t attribute = 0;
} // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int value) {
    std::unique_lock<std::mutex> l(mu);
    attribute = (size_t)value;
    if (attribute == MORE) {
        more_set = true;
        change.notify_all();
        change.wait_for(l, std::chrono::milliseconds(300), [] { return less_asked; });
    }
    return hipSuccess;
}
}

int main() {
    static xnor_hip::LdsGrant grant;
    std::thread other([] {
        {
            std::unique_lock<std::mutex> l(mu);
            change.wait(l, [] { return more_set; });
        }
        (void)grant.ask(nullptr, LESS);
        std::lock_guard<std::mutex> l(mu);
        less_asked = true;
        change.notify_all();
    });
    (void)grant.ask(nullptr, MORE);
    other.join();
    // a size that has been granted has to be had
    (void)grant.ask(nullptr, MORE);
    if (attribute < MORE) {
        printf("granted %zu, set %zu\n", MORE, attribute);
        return 1;
    }
    printf("ok\n");
    return 0;
}
