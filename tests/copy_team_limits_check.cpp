// CPU checks of CopyTeam (vship_amd/csrc/parallel_copy.hpp) where a machine is
// short of something; prints "ok" and exits 0 on success.
//
//   asleep   while the next chunk is not open, the helpers use no CPU time
//   threads  a team whose threads the system refuses copies with those it has
//   taken    taken() says whether a copy has the helpers
#include <dlfcn.h>
#include <pthread.h>
#include <sys/resource.h>

#include <atomic>
#include <cerrno>
#include <cstdio>
#include <string>

#include "../vship_amd/csrc/parallel_copy.hpp"

using vship::CopyTeam;

// Threads that may still be started; -1: any number. The library's
// std::thread starts its threads through this one.
static std::atomic<int> g_threads{-1};
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) noexcept {
    using Fn = int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
    static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
    if (g_threads.load() == 0) return EAGAIN;
    if (g_threads.load() > 0) g_threads--;
    return real(t, a, f, arg);
}

static std::vector<uint8_t> src(2 << 20), dst(2 << 20);

// eight pieces in two chunks
static std::vector<CopyTeam::Piece> pieces() {
    std::vector<CopyTeam::Piece> p;
    for (int i = 0; i < 8; i++) {
        const size_t o = (size_t)i << 18;
        p.push_back({dst.data() + o, src.data() + o, (size_t)1 << 18, i / 4});
    }
    return p;
}

static bool copied() {
    const bool same = std::memcmp(dst.data(), src.data(), src.size()) == 0;
    std::fill(dst.begin(), dst.end(), 0);
    return same;
}

static double cpu_seconds() {
    rusage u;
    getrusage(RUSAGE_SELF, &u);
    return (double)(u.ru_utime.tv_sec + u.ru_stime.tv_sec) + 1e-6 * (double)(u.ru_utime.tv_usec + u.ru_stime.tv_usec);
}

static int asleep() {
    CopyTeam team(3);
    const double t0 = cpu_seconds();
    team.run(
        pieces(), 2, 2,
        [](int c, bool wait) {
            if (c == 0) return true;
            if (!wait) return false;
            std::this_thread::sleep_for(std::chrono::milliseconds(500));
            return true;
        },
        [](int) {});
    const double used = cpu_seconds() - t0;
    // 2 MiB take about a millisecond; one helper that does not sleep uses the 500
    std::printf("%.3f s of CPU time\n", used);
    return copied() && used < 0.1 ? 0 : 1;
}

static int threads() {
    for (int given = 0; given < 4; given++) {
        g_threads = given;
        CopyTeam team(3);
        g_threads = -1;
        for (int rep = 0; rep < 20; rep++) {
            team.run(pieces(), 2, 2, [](int, bool) { return true; }, [](int) {});
            if (!copied()) return 1;
        }
    }
    return 0;
}

static int taken() {
    CopyTeam team(2), nobody(0);
    std::atomic<int> bad{0};
    if (team.taken()) bad++;
    team.run(
        pieces(), 2, 2, [](int, bool) { return true; },
        [&](int) {
            std::thread([&] {
                if (!team.taken()) bad++;
            }).join();
        });
    if (team.taken() || !copied()) bad++;
    nobody.run(
        pieces(), 2, 2, [](int, bool) { return true; },
        [&](int) {
            std::thread([&] {
                if (nobody.taken()) bad++;  // a copy has nothing that another could want
            }).join();
        });
    return bad ? 1 : 0;
}

int main(int argc, char** argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    for (size_t i = 0; i < src.size(); i++) src[i] = (uint8_t)(i * 2654435761u >> 24);
    const int rc = what == "asleep" ? asleep() : what == "threads" ? threads() : what == "taken" ? taken() : 2;
    if (rc == 0) std::printf("ok\n");
    return rc;
}
