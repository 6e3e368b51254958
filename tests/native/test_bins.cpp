// Host tests of axiomr_amd/csrc/bins.hpp, the functions that the kernels use:
// where a bin's entries and its counter lie, and the order in which waves
// store entries whose levels other waves open.  Built and run by
// tests/test_bin_layout.py.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <random>
#include <thread>
#include <vector>
#include "../../axiomr_amd/csrc/bins.hpp"

using namespace axr;

#define CHECK(c)                                                                  \
    do {                                                                          \
        if (!(c)) {                                                               \
            std::fprintf(stderr, "%s:%d: CHECK failed: %s\n", __FILE__, __LINE__, #c); \
            std::exit(1);                                                         \
        }                                                                         \
    } while (0)

static void test_levels() {
    for (uint32_t shift : {BIN0_LEAN_SHIFT, BIN0_MIN_SHIFT, 9u, BIN0_MAX_SHIFT}) {
        uint32_t level = 0, offset = 0;   // consecutive slots fill each level in turn
        for (uint32_t s = 0; s < (1u << 20); ++s) {
            const BinSlot b = bin_slot(shift, s);
            CHECK(b.level == level && b.offset == offset);
            if (++offset == 1u << (shift + level)) {
                offset = 0;
                ++level;
            }
        }
        // the ends of every level that the chunk table has
        for (uint32_t k = 0; k < BIN_LEVELS && shift + k < 31u; ++k) {
            const uint64_t first = ((1ull << k) - 1) << shift, last = first + (1ull << (shift + k)) - 1;
            if (last > 0xFFFFFFFFull) break;
            CHECK(bin_slot(shift, (uint32_t)first).level == k && bin_slot(shift, (uint32_t)first).offset == 0u);
            CHECK(bin_slot(shift, (uint32_t)last).level == k && bin_slot(shift, (uint32_t)last).offset == (uint32_t)(last - first));
        }
        // 2^31 - 16 entries stay within the table
        CHECK(bin_slot(shift, 0x7FFFFFFFu - 16u).level < BIN_LEVELS);
    }
}

static void test_count_words() {
    const uint32_t n = 3 * COUNT_BLOCK;
    std::vector<bool> seen(n);
    for (uint32_t t = 0; t < n; ++t) {
        const uint32_t w = count_word(t);
        CHECK(w / COUNT_BLOCK == t / COUNT_BLOCK && !seen[w]);   // each block onto itself, one to one
        seen[w] = true;
        if (t % 4) CHECK(w == count_word(t - 1) + 1u);                 // runs of four together,
        else if (t) CHECK(w / 32 != count_word(t - 4) / 32);           // neighbouring ones in other lines
    }
}

// ---- waves that store entries at the same time ------------------------------

constexpr uint32_t Q = 4, SHIFT = BIN0_LEAN_SHIFT;

struct Entry {
    bool act = false;
    uint32_t bin = 0, slot = 0, ref = 0;
};

struct Bins {
    uint32_t nbins;
    std::vector<uint32_t> first, pool;
    std::unique_ptr<std::atomic<uint32_t>[]> cells;   // 0: not published
    std::atomic<uint32_t> next{0};
    std::atomic<bool> stuck{false};
    Bins(uint32_t n, uint32_t pool_entries)
        : nbins(n), first(n << SHIFT, ~0u), pool(pool_entries, ~0u), cells(new std::atomic<uint32_t>[n * BIN_LEVELS]) {
        for (uint32_t i = 0; i < n * BIN_LEVELS; ++i) cells[i] = 0u;
    }
    uint32_t at(uint32_t bin, uint32_t slot) const {
        const BinSlot b = bin_slot(SHIFT, slot);
        return b.level ? pool[cells[bin * BIN_LEVELS + b.level] - 1u + b.offset] : first[(bin << SHIFT) + slot];
    }
};

// One wave: Q entries of every lane, all slots taken.
struct Wave {
    std::vector<Entry> e[Q];
};
struct WaveStore {
    Bins& bins;
    const std::vector<Entry> (&e)[Q];
    bool near(uint32_t q) {
        bool far = false;
        for (const Entry& x : e[q]) {
            const bool first = bin_slot(SHIFT, x.slot).level == 0u;
            if (x.act && first) bins.first[(x.bin << SHIFT) + x.slot] = x.ref;
            far |= x.act && !first;
        }
        return far;
    }
    bool any(bool far) const { return far; }
    void open(uint32_t q) {
        for (const Entry& x : e[q]) {
            const BinSlot b = bin_slot(SHIFT, x.slot);
            if (x.act && b.level != 0u && b.offset == 0u) {
                const uint32_t o = bins.next.fetch_add(1u << (SHIFT + b.level));
                bins.cells[x.bin * BIN_LEVELS + b.level].store(o + 1u, std::memory_order_relaxed);
            }
        }
    }
    void fill(uint32_t q) {
        const auto until = std::chrono::steady_clock::now() + std::chrono::seconds(5);
        for (const Entry& x : e[q]) {
            const BinSlot b = bin_slot(SHIFT, x.slot);
            if (!x.act || b.level == 0u) continue;
            uint32_t at;
            while ((at = bins.cells[x.bin * BIN_LEVELS + b.level].load(std::memory_order_relaxed)) == 0u) {
                if (std::chrono::steady_clock::now() > until) {
                    bins.stuck = true;
                    return;
                }
                std::this_thread::yield();
            }
            bins.pool[at - 1u + b.offset] = x.ref;
        }
    }
};

static void run(Bins& bins, std::vector<Wave>& waves) {
    std::vector<std::thread> ts;
    for (const Wave& w : waves)
        ts.emplace_back([&bins, &w] {
            WaveStore s{bins, w.e};
            place_entries<Q>(s);
        });
    for (auto& t : ts) t.join();
    CHECK(!bins.stuck);   // every wait ended
}

// Wave A's first entry lies in a level that wave B's second one opens, and the
// other way round: what atomics on two words, in flight together, may give.
static void test_crossed_levels() {
    Bins bins(2, 1u << 10);
    std::vector<Wave> waves(2);
    const uint32_t opens = 1u << SHIFT;   // level 1's first slot
    for (uint32_t w = 0; w < 2; ++w) {
        auto& e = waves[w].e;
        e[0] = {Entry{true, w, opens + 1u, 10u + w}};
        e[1] = {Entry{true, 1u - w, opens, 20u + w}};
        e[2] = e[3] = {Entry{}};
    }
    run(bins, waves);
    for (uint32_t w = 0; w < 2; ++w) CHECK(bins.at(w, opens + 1u) == 10u + w && bins.at(1u - w, opens) == 20u + w);
}

// The slots of several waves' entries handed out in any order.
static void test_any_order(uint32_t seed) {
    std::mt19937 rng(seed);
    const uint32_t nwaves = 8, lanes = 64, nbins = 1u + rng() % 12u;
    std::vector<Wave> waves(nwaves);
    std::vector<Entry*> order;
    uint32_t ref = 0;
    for (Wave& w : waves) {
        for (auto& entries : w.e) {
            entries.resize(lanes);
            for (Entry& x : entries) {
                x.act = rng() % 8u != 0u;
                x.bin = rng() % nbins;
                x.ref = ref++;
                if (x.act) order.push_back(&x);
            }
        }
    }
    std::shuffle(order.begin(), order.end(), rng);
    std::vector<uint32_t> count(nbins);
    for (Entry* x : order) x->slot = count[x->bin]++;
    Bins bins(nbins, 1u << 16);
    run(bins, waves);
    CHECK(bins.next <= bins.pool.size());
    for (const Entry* x : order) CHECK(bins.at(x->bin, x->slot) == x->ref);
}

int main() {
    test_levels();
    test_count_words();
    test_crossed_levels();
    for (uint32_t seed = 0; seed < 200; ++seed) test_any_order(seed);
    std::puts("ALL OK");
    return 0;
}
