// Checks the bookkeeping of the second buffers with host memory in the
// device's place.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <thread>

#include "second_buffers.hpp"

using namespace lbm;

static int fails = 0;
#define CHECK(c)                                               \
    do {                                                       \
        if (!(c)) {                                            \
            if (++fails < 20) printf("FAIL %d: %s\n", __LINE__, #c); \
        }                                                      \
    } while (0)

struct HostMemory : SecondMemory {
    std::atomic<int> blocks{0}, drains{0}, asked{0};
    bool full = false;
    void *allocate(int, size_t bytes) override {
        ++asked;
        if (full) return nullptr;
        ++blocks;
        return malloc(bytes);
    }
    void release(void *p) override {
        --blocks;
        free(p);
    }
    void drain(int) override { ++drains; }
};

struct Solver {
    std::atomic<unsigned> version{0};
    SecondBuffer second;
    explicit Solver(size_t bytes, int device = 0) {
        second.version = &version;
        second.bytes = bytes;
        second.device = device;
    }
};

// A solver goes away on its own thread while another thread's failed allocation
// takes its buffer: after give() nothing of it may be written any more.
static void destroyed_while_taken_away() {
    HostMemory mem;
    SecondBuffers sb(mem);
    std::atomic<bool> stop{false};
    std::thread short_of_memory([&] {
        while (!stop) sb.give_all(0);
    });
    SecondBlock *const other = (SecondBlock *)0x10;
    for (int k = 0; k < 3000 && !fails; ++k) {
        Solver *s = new Solver(1000);
        CHECK(sb.take({&s->second}));
        while (s->second.at) {
        }
        sb.give(s->second);
        s->second.block = other;  // the solver's memory is someone else's now
        const unsigned v = s->version;
        const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(20);
        while (std::chrono::steady_clock::now() < until) {
        }
        CHECK(s->second.block == other && s->version == v);
        delete s;
    }
    stop = true;
    short_of_memory.join();
}

// While one thread enqueues a long sequence, another takes and gives back
// buffers without waiting for it; taking them away waits for the sequence, and
// does not wait for sequences that begin later.
static void launches_keep_nobody_waiting() {
    HostMemory mem;
    SecondBuffers sb(mem);
    auto within = [](std::atomic<bool> &done) {
        for (int k = 0; k < 5000 && !done; ++k) std::this_thread::sleep_for(std::chrono::milliseconds(1));
        return done.load();
    };
    Solver a(1000);
    CHECK(sb.take({&a.second}));
    std::atomic<bool> stepped{false}, taken{false}, stop{false};
    std::thread second, short_of_memory;
    {
        const auto enqueuing = sb.in_use();
        second = std::thread([&] {
            Solver b(1000);
            for (int k = 0; k < 2; ++k) {
                CHECK(sb.take({&b.second}));
                const auto lock = sb.in_use();
                CHECK(b.second.at);
            }
            sb.give(b.second);
            stepped = true;
        });
        CHECK(within(stepped));
        short_of_memory = std::thread([&] {
            sb.give_all(0);
            taken = true;
        });
        std::this_thread::sleep_for(std::chrono::milliseconds(50));
        CHECK(!taken && a.second.at);
    }
    second.join();
    std::vector<std::thread> busy;  // sequences that overlap without end
    for (int t = 0; t < 2; ++t)
        busy.emplace_back([&] {
            while (!stop) {
                const auto lock = sb.in_use();
                std::this_thread::sleep_for(std::chrono::milliseconds(2));
            }
        });
    CHECK(within(taken) && !a.second.at);
    taken = false;
    std::thread again([&] {
        Solver c(100);
        CHECK(sb.take({&c.second}) && sb.give_all(0));
        taken = true;
    });
    CHECK(within(taken));
    stop = true;
    for (std::thread &t : busy) t.join();
    short_of_memory.join();
    again.join();
}

static void blocks_and_spares() {
    HostMemory mem;
    SecondBuffers sb(mem);
    {
        Solver a(1000), b(200), c(500, 1);
        CHECK(sb.take({&a.second, &b.second}));
        CHECK(mem.blocks == 1 && (char *)b.second.at.load() - (char *)a.second.at.load() == 1024);
        CHECK(a.version == 1 && b.version == 1);
        CHECK(sb.take({&a.second, &b.second}) && mem.blocks == 1 && a.version == 1);
        CHECK(sb.take({&c.second}) && mem.blocks == 2);
        CHECK(sb.give_all(0) && mem.drains == 1);
        CHECK(!a.second.at && !b.second.at && c.second.at && a.version == 2 && mem.blocks == 1);
        CHECK(sb.take({&a.second}) && mem.blocks == 2);
        sb.give(a.second);
        CHECK(mem.blocks == 2);  // kept for the next solver
        CHECK(sb.take({&b.second}) && mem.blocks == 3);  // far too large for this one
        sb.give(b.second);
        sb.give(c.second);
        sb.give(c.second);
    }
    Solver d(900), far(300, 1), large(40000);
    CHECK(sb.has_spare({&d.second}) && sb.has_spare({&far.second}) && !sb.has_spare({&large.second}));
    CHECK(!sb.has_spare({&d.second, &large.second}) && !sb.has_spare({}));
    CHECK(sb.take({&d.second}) && mem.blocks == 3);
    sb.give(d.second);
    {
        std::vector<std::unique_ptr<Solver>> many;
        for (int k = 0; k < 30; ++k) {
            many.emplace_back(new Solver(5000 + 4000 * (size_t)k));
            CHECK(sb.take({&many.back()->second}));
        }
        for (auto &s : many) sb.give(s->second);
        CHECK(mem.blocks == (int)SecondBuffers::kSpares);
    }
    sb.give_all(0);
    CHECK(mem.blocks == 0 && !sb.give_all(0));
    {
        Solver e(100);
        CHECK(sb.take({&e.second}) && mem.blocks == 1);
        sb.give(e.second);
        CHECK(mem.blocks == 1);
        sb.release_spares();
        CHECK(mem.blocks == 0);
    }
}

// While a thread allocates, another one's question about the spares is answered at once.
static void asking_does_not_wait() {
    struct Slow : HostMemory {
        std::atomic<bool> within{false}, go{false};
        void *allocate(int device, size_t bytes) override {
            within = true;
            for (int k = 0; k < 5000 && !go; ++k) std::this_thread::sleep_for(std::chrono::milliseconds(1));
            return HostMemory::allocate(device, bytes);
        }
    } mem;
    SecondBuffers sb(mem);
    Solver a(1000), b(1000);
    std::thread t([&] { CHECK(sb.take({&a.second})); });
    while (!mem.within) std::this_thread::yield();
    CHECK(!sb.has_spare({&b.second}) && !a.second.at);
    mem.go = true;
    t.join();
    sb.give(a.second);
    CHECK(sb.has_spare({&b.second}));
    sb.give_all(0);
}

// A refusal holds for what was asked for, and for some sequences.
static void refused_for_a_while() {
    HostMemory mem;
    SecondBuffers sb(mem);
    Solver a(1000), b(5000), c(400);
    mem.full = true;
    CHECK(!sb.take({&a.second, &b.second}) && mem.asked == 1 && !a.second.at && !b.second.at);
    mem.full = false;  // as when another library has given its memory back
    CHECK(sb.take({&a.second}) && mem.asked == 2);  // less than was refused
    CHECK(sb.take({&b.second, &c.second}) && mem.asked == 3);
    Solver d(7000);
    mem.full = true;
    CHECK(!sb.take({&d.second}) && mem.asked == 4);
    mem.full = false;
    for (int k = 0; k < SecondBuffers::kWait; ++k) CHECK(!sb.take({&d.second}));
    CHECK(mem.asked == 4);
    CHECK(sb.take({&d.second}) && mem.asked == 5 && d.second.at);
    for (Solver *s : {&a, &b, &c, &d}) sb.give(s->second);
    mem.full = true;
    Solver e(100000);
    CHECK(!sb.take({&e.second}) && !e.second.at);
    sb.give(e.second);
}

int main() {
    blocks_and_spares();
    asking_does_not_wait();
    refused_for_a_while();
    launches_keep_nobody_waiting();
    destroyed_while_taken_away();
    if (fails) {
        printf("%d failures\n", fails);
        return 1;
    }
    printf("second buffers: ok\n");
    return 0;
}
