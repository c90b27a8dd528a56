// Admission of solves to a GPU (cuev_amd/csrc/residency.hpp): the workgroups of every admitted mix find
// a CU each, and claims are served in order, never above the budget, to the end.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>

#include "../../cuev_amd/csrc/residency.hpp"

using namespace cuev;

#define CHECK(c)                                              \
    do {                                                      \
        if (!(c)) {                                           \
            std::printf("line %d: %s\n", __LINE__, #c);       \
            return 1;                                         \
        }                                                     \
    } while (0)

// a grid's workgroups, dealt out in turn to 8 XCDs and in each to 4 shader engines of 8 CUs
static void place(int (&load)[8][4], int wgs) {
    for (int i = 0; i < wgs; ++i) ++load[i % 8][i / 8 % 4];
}

static int mixes() {
    const int cus = 256, ns[] = {65, 300, 1000, 2048, 2049, 2500, 4096, 4097, 6000, 8192, 12000, 16384};
    const int bs[] = {16, 32, 64};
    std::vector<std::pair<int, int>> kinds; // (shares, widest grid)
    for (int n : ns)
        for (int b : bs) {
            const int hops = (n - 2) / b + 1, panel = (n + 63) / 64, wgs = hops > panel ? hops : panel;
            if (wgs > cus) continue; // more hops than CUs: below
            kinds.push_back({cu_shares(n, b, cus), wgs});
        }
    long admitted = 0;
    // every admitted mix of up to four kinds: no shader engine gets more than its 8 CUs
    for (size_t i = 0; i < kinds.size(); ++i)
        for (size_t j = i; j < kinds.size(); ++j)
            for (size_t k = j; k < kinds.size(); ++k)
                for (size_t l = k; l < kinds.size(); ++l) {
                    int load[8][4] = {}, used = 0;
                    for (size_t q : {i, j, k, l})
                        if (used + kinds[q].first <= kCuShares) {
                            used += kinds[q].first;
                            place(load, kinds[q].second);
                        }
                    for (auto &x : load)
                        for (int v : x) CHECK(v <= 8);
                    ++admitted;
                }
    CHECK(admitted > 1000);
    // the mixes that could block each other when only solves above n = 4096 took turns
    CHECK(cu_shares(16384, 64, cus) + cu_shares(1000, 64, cus) > kCuShares);
    CHECK(cu_shares(8192, 64, cus) + 3 * cu_shares(4096, 64, cus) > kCuShares);
    // and what goes on side by side
    CHECK(6 * cu_shares(1000, 64, cus) <= kCuShares && 4 * cu_shares(4096, 64, cus) <= kCuShares);
    // one workgroup waits for nobody; the largest take the whole GPU, whatever its size
    CHECK(cu_shares(1, 16, cus) == 0 && cu_shares(64, 64, cus) == 0 && cu_shares(65, 64, cus) == 1);
    CHECK(cu_shares(49152, 64, cus) == kCuShares && cu_shares(2000000000, 16, cus) == kCuShares);
    CHECK(cu_shares(4096, 64, 32) == kCuShares && cu_shares(256, 64, 32) == 1 && cu_shares(1000, 64, 4) == kCuShares);
    return 0;
}

static int threads() {
    CuBudget budget;
    std::atomic<int> used{0}, worst{0}, finished{0};
    std::vector<std::thread> pool;
    for (int t = 0; t < 12; ++t)
        pool.emplace_back([&, t] {
            for (int r = 0; r < 300; ++r) {
                const int k = 1 + (t * 7 + r * 3) % kCuShares;
                budget.take(k);
                const int now = used += k;
                for (int w = worst; now > w && !worst.compare_exchange_weak(w, now);) {}
                std::this_thread::yield();
                used -= k;
                budget.give(k);
            }
            ++finished;
        });
    for (auto &x : pool) x.join();
    CHECK(finished == 12 && used == 0 && worst <= kCuShares && worst > 1);
    // in order: a small claim behind a large one that waits does not pass it
    budget.take(4);
    std::atomic<int> order{0}, large{0}, small{0};
    std::thread a([&] {
        budget.take(8);
        large = ++order;
        budget.give(8);
    });
    std::this_thread::sleep_for(std::chrono::milliseconds(200));
    std::thread b([&] {
        budget.take(1);
        small = ++order;
        budget.give(1);
    });
    std::this_thread::sleep_for(std::chrono::milliseconds(200));
    CHECK(large == 0 && small == 0);
    budget.give(4);
    a.join();
    b.join();
    CHECK(large == 1 && small == 2);
    return 0;
}

int main() {
    if (mixes() || threads()) return 1;
    std::puts("residency ok");
    return 0;
}
