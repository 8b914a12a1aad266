// Checks of ornithology_amd/csrc/oh_pool.h over a made-up device: one check per
// run, named by the first argument (tests/test_pool.py builds and runs them).
#include "oh_pool.h"

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <atomic>
#include <map>
#include <mutex>
#include <set>
#include <thread>
#include <vector>

namespace {

constexpr size_t MiB = (size_t)1 << 20, GiB = (size_t)1 << 30;
size_t capacity = 288 * GiB, used = 0;
uintptr_t next_addr = 0x1000;
std::map<void *, size_t> live;
std::mutex dev_mu;

int dev_alloc(void **p, size_t n) {
    std::lock_guard<std::mutex> lk(dev_mu);
    if (used + n > capacity) return 2;
    *p = (void *)next_addr;
    next_addr += n + 256;
    live[*p] = n;
    used += n;
    return 0;
}
void dev_release(void *p) {
    std::lock_guard<std::mutex> lk(dev_mu);
    auto it = live.find(p);
    if (it == live.end()) {
        printf("a block that is not live was released\n");
        exit(1);
    }
    used -= it->second;
    live.erase(it);
}
int asked = 0;
size_t dev_unused(int) {
    std::lock_guard<std::mutex> lk(dev_mu);
    asked++;
    return capacity - used;
}
const DevMem kMem = {dev_alloc, dev_release, dev_unused};

#define CHECK(x)                                                     \
    do {                                                             \
        if (!(x)) {                                                  \
            printf("%s:%d: %s\n", __FILE__, __LINE__, #x);           \
            return 1;                                                \
        }                                                            \
    } while (0)

DevBlock get(DevPool &p, size_t n) {
    DevBlock b;
    if (p.get(n, &b) != 0) {
        printf("no block of %zu bytes\n", n);
        exit(1);
    }
    return b;
}

// a block serves sizes down to two thirds of it (and 1 MiB), the smallest such one
int fit() {
    DevPool p(kMem, 0);
    const DevBlock a = get(p, 300 * MiB), b = get(p, 290 * MiB);
    p.put(a);
    p.put(b);
    CHECK(get(p, 301 * MiB).p != a.p);
    const DevBlock c = get(p, 250 * MiB);
    CHECK(c.p == b.p && c.n == b.n);
    CHECK(get(p, 150 * MiB).p != a.p);
    CHECK(get(p, 200 * MiB).p == a.p);
    return 0;
}

// sizes that no longer occur do not keep those that do out of the pool
int unusable_bytes() {
    DevPool p(kMem, 0);
    DevBlock b[4];
    for (int i = 0; i < 4; i++) b[i] = get(p, (size_t)(10 + i) * GiB / 13);
    for (const DevBlock &x : b) p.put(x);
    const DevBlock s = get(p, 2 * GiB);
    p.put(s);
    CHECK(get(p, 2 * GiB).p == s.p);
    CHECK(used <= 6 * GiB);
    return 0;
}
int unusable_blocks() {
    DevPool p(kMem, 0);
    DevBlock b[3 * DevPool::kBlocks];
    for (int i = 0; i < 3 * DevPool::kBlocks; i++) b[i] = get(p, 4096 + 256 * i);
    for (const DevBlock &x : b) p.put(x);
    CHECK((int)live.size() == DevPool::kBlocks);
    const DevBlock s = get(p, 64 * MiB);
    p.put(s);
    CHECK((int)live.size() == DevPool::kBlocks);
    CHECK(get(p, 64 * MiB).p == s.p);
    return 0;
}

// the pool never holds more than its bounds, and gives the oldest back first
int bounds() {
    DevPool p(kMem, 0);
    DevBlock b[8];
    for (int i = 0; i < 8; i++) b[i] = get(p, GiB);
    for (const DevBlock &x : b) {
        p.put(x);
        CHECK(live.count(x.p) == 1);
    }
    CHECK(used == DevPool::kBytes);
    for (int i = 0; i < 8; i++) CHECK(live.count(b[i].p) == (i >= 4 ? 1u : 0u));
    const DevBlock big = get(p, DevPool::kBytes + 1);
    p.put(big);
    CHECK(live.count(big.p) == 0 && used == DevPool::kBytes);
    CHECK(p.trim() == DevPool::kBytes && used == 0 && p.trim() == 0);
    return 0;
}

// on a device that is nearly full the pool keeps a sixteenth of the rest
int share() {
    DevPool p(kMem, 0);
    capacity = 100 * GiB;
    const DevBlock a = get(p, 2 * GiB), s = get(p, 100 * MiB);
    p.put(a);
    const DevBlock rest = get(p, 93 * GiB);
    CHECK(live.count(a.p) == 1);
    p.put(s);                              // 7 GiB without it and a: room for 448 MiB
    CHECK(live.count(a.p) == 0 && live.count(s.p) == 1);
    const DevBlock c = get(p, GiB);
    p.put(c);
    CHECK(live.count(c.p) == 0 && live.count(s.p) == 1);
    p.put(get(p, 300 * MiB));
    CHECK(live.count(s.p) == 1 && used == rest.n + 400 * MiB);
    return 0;
}

// blocks that come and go do not ask the device each time, and one that another
// user filled is noticed all the same
int asking() {
    DevPool p(kMem, 0);
    p.put(get(p, 100 * MiB));
    asked = 0;
    for (int i = 0; i < DevPool::kAsk - 1; i++) p.put(get(p, 100 * MiB));
    CHECK(asked == 0 && used == 100 * MiB);
    capacity = 1 * GiB;
    p.put(get(p, 100 * MiB));
    CHECK(asked == 1 && used == 0);
    return 0;
}

// several threads: every block is in one place, none is lost, the bounds hold
int threads() {
    DevPool p(kMem, 0);
    std::vector<std::thread> ts;
    std::atomic<int> bad{0};
    std::mutex mu;
    std::set<void *> out;
    for (int t = 0; t < 8; t++)
        ts.emplace_back([&, t]() {
            unsigned r = 17u * (unsigned)t + 1;
            for (int i = 0; i < 2000; i++) {
                r = r * 1664525u + 1013904223u;
                DevBlock b;
                if (p.get((1 + (r >> 8) % 200) * MiB, &b) != 0) bad++;
                {
                    std::lock_guard<std::mutex> lk(mu);
                    if (!out.insert(b.p).second) bad++;
                }
                {
                    std::lock_guard<std::mutex> lk(mu);
                    out.erase(b.p);
                }
                p.put(b);
                if (r % 97 == 0) p.trim();
            }
        });
    for (std::thread &t : ts) t.join();
    CHECK(bad == 0 && used <= DevPool::kBytes && (int)live.size() <= DevPool::kBlocks);
    p.trim();
    CHECK(used == 0 && live.empty());
    return 0;
}

// the end of one user leaves the blocks that served others
int owners() {
    DevPool p(kMem, 0);
    int one, two;
    DevBlock a = get(p, 10 * MiB), b = get(p, 20 * MiB), c = get(p, 40 * MiB), d = get(p, 80 * MiB);
    a.owner = c.owner = &one;
    b.owner = &two;
    for (const DevBlock &x : {a, b, c, d}) p.put(x);
    CHECK(p.trim(&one) == 50 * MiB);
    CHECK(live.count(a.p) == 0 && live.count(c.p) == 0 && live.count(b.p) == 1 && live.count(d.p) == 1);
    DevBlock e = get(p, 20 * MiB);
    CHECK(e.p == b.p);
    e.owner = &one;                       // now it serves the other one
    p.put(e);
    CHECK(p.trim(&two) == 0 && p.trim(&one) == 20 * MiB && p.trim() == 80 * MiB);
    return 0;
}

// an allocation that fails is tried again without the pool's blocks
int retry() {
    DevPool p(kMem, 0);
    const DevBlock a = get(p, 3 * GiB);
    p.put(a);
    CHECK(used == 3 * GiB);
    capacity = 8 * GiB;
    void *q = nullptr;
    CHECK(p.alloc(&q, 6 * GiB) == 0 && used == 6 * GiB && live.count(a.p) == 0);
    CHECK(p.alloc(&q, 3 * GiB) == 2 && used == 6 * GiB);
    return 0;
}

// ... and without those of the device's other pools; another device's stay
int other_pools() {
    DevPool p(kMem, 0), other(kMem, 1);
    auto *q = new DevPool(kMem, 0);
    const DevBlock a = get(p, GiB), b = get(*q, 2 * GiB), c = get(other, GiB);
    p.put(a);
    q->put(b);
    other.put(c);
    capacity = 8 * GiB;
    void *x = nullptr;
    CHECK(p.alloc(&x, 6 * GiB) == 0);
    CHECK(live.count(a.p) == 0 && live.count(b.p) == 0 && live.count(c.p) == 1);
    delete q;
    CHECK(p.alloc(&x, 2 * GiB) == 2 && live.count(c.p) == 1);
    return 0;
}

const struct { const char *name; int (*run)(); } kChecks[] = {
    {"fit", fit}, {"unusable_bytes", unusable_bytes}, {"unusable_blocks", unusable_blocks},
    {"bounds", bounds}, {"share", share}, {"asking", asking}, {"owners", owners}, {"threads", threads}, {"retry", retry}, {"other_pools", other_pools},
};

} // namespace

int main(int argc, char **argv) {
    for (const auto &c : kChecks)
        if (argc > 1 && strcmp(argv[1], c.name) == 0) return c.run();
    printf("no such check\n");
    return 2;
}
