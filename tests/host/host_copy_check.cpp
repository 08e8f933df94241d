// csrc/host_copy.hip on the host, over the fake runtime of fake_hip: bytes of copies
// both ways (below and above the ring's threshold, tails, several segments), a stream
// of another device than the current one, a copy that fails, and the CPU time spent
// while the stream's earlier work runs.  Exit status 1 and a line per failure.
#include <cstdio>
#include <ctime>
#include <random>
#include <vector>

#include "host_copy.hpp"

static int bad = 0;
static void expect(bool ok, const char* what)
{
    if (!ok) {
        std::printf("FAILED: %s\n", what);
        bad = 1;
    }
}
static double cpu_seconds()
{
    timespec t;
    clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t);
    return (double)t.tv_sec + 1e-9 * (double)t.tv_nsec;
}

int main()
{
    FakeStream s;
    std::mt19937_64 rng(1);
    for (size_t total : {size_t(1000), (size_t(32) << 20) - 8, size_t(32) << 20, (size_t(33) << 20) + 8, (size_t(90) << 20) + 12344})
        for (int n : {1, 3}) {
            std::vector<unsigned char> h(total), d(total, 0), back(total, 0);
            for (size_t i = 0; i < total; i += 8) h[i] = (unsigned char)rng();
            std::vector<gkm::CopySeg> up, down;
            for (int k = 0; k < n; k++) {
                const size_t a = total * k / n, b = total * (k + 1) / n;
                up.push_back({h.data() + a, d.data() + a, b - a});
                down.push_back({back.data() + a, d.data() + a, b - a});
            }
            gkm::HostPipe p;
            expect(p.to_device(up.data(), n, &s) == hipSuccess && d == h, "bytes up");
            expect(p.to_host(down.data(), n, &s) == hipSuccess && back == h, "bytes down");
            p.release();
            expect(fake::live == 0, "everything given back");
        }
    const size_t big = size_t(64) << 20;
    std::vector<unsigned char> h(big, 7), d(big, 9);
    gkm::CopySeg seg{h.data(), d.data(), big};
    {
        FakeStream other;
        other.device = 1;
        gkm::HostPipe p;
        expect(p.to_host(&seg, 1, &other) == hipSuccess && h == d, "a stream of another device than the current one");
        expect(fake::current == 0, "the caller's device is current again");
        p.release();
    }
    for (int at : {0, 1, 5}) {
        gkm::HostPipe p;
        fake::fail_at = fake::copies + at;
        expect(p.to_host(&seg, 1, &s) != hipSuccess, "a failing copy down is reported");
        fake::fail_at = fake::copies + at;
        expect(p.to_device(&seg, 1, &s) != hipSuccess, "a failing copy up is reported");
        fake::fail_at = -1;
        p.release();
    }
    for (bool down : {true, false}) {
        gkm::HostPipe p;
        expect(p.to_host(&seg, 1, &s) == hipSuccess, "a first copy");
        const int ring = fake::pinned;
        s.busy = 0.5;
        const double t = cpu_seconds();
        expect((down ? p.to_host(&seg, 1, &s) : p.to_device(&seg, 1, &s)) == hipSuccess, "a copy behind other work");
        const double used = cpu_seconds() - t;
        std::printf("%s behind 0.5 s of other work: %.3f s of CPU\n", down ? "down" : "up", used);
        expect(used < 0.25, "no CPU time while the stream's earlier work runs");
        expect(fake::pinned == ring, "the ring is kept");
        p.release();
    }
    std::printf("%s\n", bad ? "wrong" : "all right");
    return bad;
}
