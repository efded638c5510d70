// CPU check of CopyTeam (vship_amd/csrc/parallel_copy.hpp): random copies in
// chunks, with and without row strides, equal memcpy; chunks are opened only
// while fewer than `depth` are ahead of the last one done, done follows in
// order; an exception from a callback ends the copy and reaches the caller; and
// callers on several threads may share one team.
// Prints "ok" and exits 0 on success.
#include <atomic>
#include <cstdio>
#include <random>

#include "../vship_amd/csrc/parallel_copy.hpp"

using vship::CopyTeam;

int main() {
    std::mt19937_64 rng(3);
    std::vector<uint8_t> src(24 << 20), dst(src.size());
    for (auto& v : src) v = (uint8_t)rng();
    for (int helpers = 0; helpers < 5; helpers++) {
        CopyTeam team(helpers);
        for (int rep = 0; rep < 200; rep++) {
            const int chunks = 1 + (int)(rng() % 20), depth = 1 + (int)(rng() % 4);
            std::vector<CopyTeam::Piece> p;
            size_t off = 0;
            for (int c = 0; c < chunks; c++)
                for (int k = 1 + (int)(rng() % 4); k > 0; k--) {
                    const size_t n = 1 + rng() % 200000;
                    CopyTeam::Piece q{dst.data() + off, src.data() + off, n, c};
                    if (n % 3 == 0) {  // the same bytes as three rows
                        q.bytes = n / 3;
                        q.rows = 3;
                        q.dst_stride = q.src_stride = (int64_t)(n / 3);
                    }
                    p.push_back(q);
                    off += n;
                }
            std::fill(dst.begin(), dst.begin() + (long)off + 64, 0);
            const bool fail = rep % 10 == 9;
            std::vector<int> opened(chunks, 0);
            int last = -1, polls = 0;
            bool bad = false, caught = false;
            try {
                team.run(
                    p, chunks, depth,
                    [&](int c, bool wait) {
                        if (c > last + depth) bad = true;
                        if (!wait && ++polls % 3) return false;
                        opened[c] = 1;
                        return true;
                    },
                    [&](int c) {
                        if (c != last + 1 || !opened[c]) bad = true;
                        last = c;
                        if (fail && c == chunks / 2) throw 1;
                    });
            } catch (int) {
                caught = true;
            }
            if (caught != fail || bad || (!fail && std::memcmp(dst.data(), src.data(), off) != 0) ||
                dst[off] != 0) {
                std::printf("helpers %d repetition %d\n", helpers, rep);
                return 1;
            }
        }
    }
    CopyTeam team(3);
    std::atomic<int> bad{0};
    std::vector<std::thread> callers;
    for (int k = 0; k < 6; k++)
        callers.emplace_back([&, k] {
            std::vector<uint8_t> out(4 << 20);
            for (int rep = 0; rep < 50; rep++) {
                std::vector<CopyTeam::Piece> p;
                for (int i = 0; i < 16; i++) {
                    const size_t o = (size_t)i << 18;
                    p.push_back({out.data() + o, src.data() + 1000 * k + o, (size_t)1 << 18, i / 2});
                }
                team.run(p, 8, 4, [](int, bool) { return true; }, [](int) {});
                if (std::memcmp(out.data(), src.data() + 1000 * k, out.size()) != 0) bad++;
            }
        });
    for (auto& t : callers) t.join();
    if (bad) return 1;
    std::printf("ok\n");
    return 0;
}
