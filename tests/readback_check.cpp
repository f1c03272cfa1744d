// Checks of lfh::Readback on the CPU, over the stand-in HIP runtime of
// tests/fake_hip.  Prints each check before it runs; exits with 1 at the first
// that fails.
#include <chrono>
#include <cstdio>
#include <vector>

#include "../lavaframe_amd/csrc/readback.h"

#define CHECK(x)                                            \
    do {                                                    \
        if (!(x)) {                                         \
            std::printf("line %d: %s\n", __LINE__, #x);     \
            std::fflush(stdout);                            \
            std::_Exit(1);                                  \
        }                                                   \
    } while (0)

namespace {

constexpr size_t kMiB = (size_t)1 << 20;

std::vector<unsigned char> image(size_t n, unsigned seed) {
    std::vector<unsigned char> v(n);
    unsigned x = seed * 2654435761u + 1u;
    for (auto& b : v) b = (unsigned char)((x = x * 1664525u + 1013904223u) >> 24);
    return v;
}

// Bytes and flag of an image, with and without the flag; one byte past the image stays as it was.
void whole(lfh::Readback& rb, size_t n, unsigned seed) {
    const auto src = image(n, seed);
    for (int with_flag = 0; with_flag < 2; ++with_flag) {
        std::vector<unsigned char> dst(n + 1, 0xA5);
        const int d_flag = 7 + (int)seed;
        int flag = 0;
        CHECK(rb.read(dst.data(), src.data(), n, with_flag ? &d_flag : nullptr, &flag, 0, 0) == hipSuccess);
        CHECK(std::memcmp(dst.data(), src.data(), n) == 0 && dst[n] == 0xA5);
        CHECK(flag == (with_flag ? d_flag : 0));
    }
}

void begin(const char* what) {
    std::printf("%s\n", what);
    std::fflush(stdout);
}

}  // namespace

int main() {
    std::thread gpu(fake::work);
    fake::open(true);
    {
        lfh::Readback rb;
        begin("sizes around a piece and around the pinned buffer");
        const size_t sizes[] = {1, 12, kMiB - 1, kMiB, kMiB + 1, 2 * kMiB, 3 * kMiB + 77, 32 * kMiB, 32 * kMiB + 1, 65 * kMiB + 5};
        unsigned seed = 1;
        for (size_t n : sizes) whole(rb, n, seed++);
        for (size_t n : {5 * kMiB, (size_t)100, kMiB + 9}) whole(rb, n, seed++);   // smaller after larger

        begin("one thread waits for the frame, helpers start with its first piece");
        fake::open(false);
        const auto src = image(8 * kMiB + 3, 99);
        std::vector<unsigned char> dst(src.size());
        const int d_flag = 5;
        int flag = 0;
        fake::helpers = fake::most_waiting = 0;
        hipError_t r = hipErrorUnknown;
        std::thread caller([&] { r = rb.read(dst.data(), src.data(), src.size(), &d_flag, &flag, 0, 0); });
        std::this_thread::sleep_for(std::chrono::milliseconds(300));
        {
            std::lock_guard<std::mutex> lk(fake::mu);
            CHECK(fake::helpers == 0);
            CHECK(fake::most_waiting == 1);
        }
        fake::open(true);
        caller.join();
        CHECK(r == hipSuccess && flag == 5 && dst == src);
        CHECK(fake::helpers == 3);

        begin("pinned memory of the caller: one transfer and the flag's, no helpers");
        fake::known = dst.data();
        fake::copies = fake::helpers = 0;
        std::fill(dst.begin(), dst.end(), (unsigned char)0);
        flag = 0;
        CHECK(rb.read(dst.data(), src.data(), src.size(), &d_flag, &flag, 0, 0) == hipSuccess);
        CHECK(flag == 5 && dst == src && fake::copies == 2 && fake::helpers == 0);
        fake::known = nullptr;

        begin("a failed copy or wait is reported and leaves nothing behind");
        for (int k = 0; k < 12; ++k) {
            fake::fail_copy = k;
            const hipError_t e = rb.read(dst.data(), src.data(), src.size(), &d_flag, &flag, 0, 0);
            CHECK((e == hipSuccess) == (fake::fail_copy >= 0));
            fake::fail_copy = -1;
            CHECK(fake::queue.empty());
            fake::fail_sync = k;
            const hipError_t w = rb.read(dst.data(), src.data(), src.size(), nullptr, nullptr, 0, 0);
            CHECK((w == hipSuccess) == (fake::fail_sync >= 0));
            fake::fail_sync = -1;
            CHECK(fake::queue.empty());
        }
        whole(rb, 6 * kMiB + 1, 1234);
    }
    CHECK(fake::pinned == 0 && fake::events == 0);

    begin("without pinned memory");
    fake::no_pinned = true;
    {
        lfh::Readback rb;
        for (size_t n : {(size_t)100, kMiB, 3 * kMiB + 1}) whole(rb, n, (unsigned)n);
    }
    {
        std::lock_guard<std::mutex> lk(fake::mu);
        fake::quit = true;
        fake::cv.notify_all();
    }
    gpu.join();
    begin("ok");
    return 0;
}
