// read_back of memory that work queued on the caller's stream fills: the bytes
// that are still the old ones.  Arguments: bytes, and 1 for hipStreamPerThread.
#include <cstdio>
#include <vector>

#include "rbhip_readback.h"

int main(int, char** argv) {
    const size_t n = std::strtoul(argv[1], nullptr, 10);
    std::vector<unsigned char> device(n, 0), host(n, 0xee);
    FakeStream plain;
    hipStream_t s = argv[2][0] == '1' ? hipStreamPerThread : &plain;
    auto value = [](size_t i) { return (unsigned char)(1 + i % 251); };
    fake_queue(s, [&] {
        for (size_t i = 0; i < n; i++) device[i] = value(i);
    });
    if (rbhip::read_back(host.data(), device.data(), n, 0, s) != hipSuccess) return 1;
    size_t stale = 0;
    for (size_t i = 0; i < n; i++) stale += host[i] != value(i);
    std::printf("%zu\n", stale);
}
