// The steps of a staged host copy (m3.c_amd/csrc/hip/m3_staging.h) on the
// CPU, over a stream that runs nothing until it is waited for: what arrives,
// and that a step that fails never hands the staging memory on while a
// queued copy could still touch it.
#include "m3_staging.h"

#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>

static int failures = 0;

static void expect(bool ok, const char *what, size_t a = 0, size_t b = 0)
{
    if (!ok) {
        std::printf("FAIL: %s (%zu, %zu)\n", what, a, b);
        ++failures;
    }
}

// Copies run when the stream is waited for, in order; queue call number
// `fail_queue` and wait call number `fail_wait` (from 1) fail, the former
// with its copy queued when `half` is set.
struct fake_stream {
    struct entry {
        uint8_t *destination;
        const uint8_t *source;
        size_t bytes;
    };
    std::vector<entry> queued;
    uint32_t sequence = 0xfffffffeU; // wraps
    size_t ran = 0;
    size_t queues = 0;
    size_t waits = 0;
    size_t fail_queue = 0;
    size_t fail_wait = 0;
    bool half = false;
    bool dead = false; // drain fails

    void run_to(size_t end)
    {
        for (; ran < end && ran < queued.size(); ++ran) {
            std::memcpy(queued[ran].destination, queued[ran].source,
                        queued[ran].bytes);
        }
    }
    int queue(uint8_t *destination, const uint8_t *source, size_t bytes,
              uint32_t *number)
    {
        const bool fails = ++queues == fail_queue;

        if (!fails || half) {
            queued.push_back({destination, source, bytes});
        }
        if (fails) {
            return 4;
        }
        *number = ++sequence;
        return 0;
    }
    int wait(uint32_t number)
    {
        if (++waits == fail_wait) {
            return 4;
        }
        run_to(queued.size() - (sequence - number));
        return 0;
    }
    bool drain()
    {
        if (dead) {
            return false;
        }
        run_to(queued.size());
        return true;
    }
};

static void check_steps()
{
    const size_t most = 4096;
    std::vector<uint8_t> source(5 * most + 7), target(source.size()),
        buffer(source.size());

    for (size_t i = 0; i < source.size(); ++i) {
        source[i] = (uint8_t)(i * 7 + i / 251);
    }
    for (size_t bytes : {(size_t)1, most - 1, most, most + 1, 3 * most,
                         source.size()}) {
        for (int down = 0; down < 2; ++down) {
            const size_t chunks = down ? (bytes + most - 1) / most : 1;

            // failing step 0: none; then every queue (without and with its
            // copy queued), then every wait
            for (size_t step = 0; step <= 3 * chunks; ++step) {
                for (int dead = 0; dead < 2; ++dead) {
                    fake_stream stream;
                    bool reusable = false;
                    int code;

                    stream.fail_queue = step <= chunks ? step
                                        : step <= 2 * chunks ? step - chunks
                                                             : 0;
                    stream.half = step > chunks;
                    stream.fail_wait =
                        step > 2 * chunks ? step - 2 * chunks : 0;
                    stream.dead = dead != 0;
                    std::fill(target.begin(), target.end(), 0);
                    code = down ? m3_stage_read(stream, buffer.data(),
                                                target.data(), source.data(),
                                                bytes, most, &reusable)
                                : m3_stage_write(stream, buffer.data(),
                                                 target.data(),
                                                 source.data(), bytes,
                                                 &reusable);
                    expect((code != 0) == (step != 0), "code", bytes, step);
                    expect(!reusable || stream.ran == stream.queued.size(),
                           "memory handed on with a copy on its way", bytes,
                           step);
                    expect(reusable == (step == 0 || !dead), "reusable",
                           bytes, step);
                    if (step == 0) {
                        expect(std::equal(source.begin(),
                                          source.begin() + (long)bytes,
                                          target.begin()),
                               "bytes", bytes, step);
                    }
                }
            }
        }
    }
}

// The pool: one owner per set, no allocation once a set is idle, the bound,
// a refused allocation, lost sets, and what closing gives back.
static void check_pool()
{
    static m3_stage_pool<2, 3> pool;
    static std::atomic<int> live{0}, made{0};
    static std::atomic<bool> refuse{false};
    auto allocate = [] {
        if (refuse.load()) {
            return (uint8_t *)nullptr;
        }
        ++live;
        ++made;
        return new uint8_t[64]();
    };
    auto release = [](uint8_t *memory) {
        --live;
        delete[] memory;
    };

    expect(pool.take(-1, allocate) == nullptr &&
               pool.take(2, allocate) == nullptr,
           "unknown ordinals have no sets");
    // sessions one after the other: one allocation, the second on
    for (int session = 0; session < 5; ++session) {
        pool.open(0);
        for (int copy = 0; copy < 3; ++copy) {
            m3_stage_set *set = pool.take(0, allocate);

            expect(set != nullptr, "a set for a lone copy");
            pool.give(0, set, true);
        }
        pool.close(0, release);
        expect(made.load() == 1 && live.load() == 1, "one set, kept");
    }
    // handles at once share sets; the bound; another GPU is apart
    pool.open(0);
    pool.open(0);
    pool.open(1);
    m3_stage_set *sets[3];

    for (m3_stage_set *&set : sets) {
        set = pool.take(0, allocate);
    }
    expect(sets[0] != sets[1] && sets[1] != sets[2] && sets[0] != sets[2],
           "a set has one owner");
    expect(pool.take(0, allocate) == nullptr, "no more sets than the bound");
    m3_stage_set *other = pool.take(1, allocate);

    expect(other != nullptr && made.load() == 4, "each GPU has its own");
    pool.give(1, other, true);
    for (m3_stage_set *set : sets) {
        pool.give(0, set, true);
    }
    pool.close(0, release);
    expect(live.load() == 4, "sets stay while a handle is open");
    pool.close(0, release);
    expect(live.load() == 2, "the last handle gives back all but one");
    // a lifetime of handles without a copy gives back that one too
    pool.open(0);
    pool.close(0, release);
    expect(live.load() == 1, "an unused set is given back");
    pool.close(1, release);
    pool.open(1);
    pool.close(1, release);
    expect(live.load() == 0, "and on the other GPU");
    // a refused allocation is not tried again until the handles closed
    refuse = true;
    pool.open(0);
    expect(pool.take(0, allocate) == nullptr, "refused");
    refuse = false;
    expect(pool.take(0, allocate) == nullptr, "not tried again");
    pool.close(0, release);
    pool.open(0);
    sets[0] = pool.take(0, allocate);
    expect(sets[0] != nullptr, "tried again by later handles");
    // a set that queued work may touch is neither lent again nor freed
    pool.give(0, sets[0], false);
    sets[1] = pool.take(0, allocate);
    expect(sets[1] != nullptr && sets[1] != sets[0], "a lost set stays out");
    pool.give(0, sets[1], true);
    pool.close(0, release);
    pool.open(0);
    pool.close(0, release);
    expect(live.load() == 1, "only the lost set is left");
    delete[] sets[0]->memory;

    // many threads, each owner alone with its set
    static std::atomic<int> shared{0}, lent{0};
    static m3_stage_pool<1, 3> busy;
    std::vector<std::thread> threads;

    for (int t = 0; t < 6; ++t) {
        threads.emplace_back([&] {
            for (int k = 0; k < 20000; ++k) {
                busy.open(0);
                m3_stage_set *set = busy.take(0, allocate);

                if (set != nullptr) {
                    lent += 1;
                    if (set->memory[1]++ != 0U) {
                        shared += 1;
                    }
                    set->memory[1] -= 1U;
                    busy.give(0, set, true);
                }
                busy.close(0, release);
            }
        });
    }
    for (std::thread &thread : threads) {
        thread.join();
    }
    expect(shared.load() == 0, "two owners of one set");
    expect(lent.load() > 0, "sets were lent");
    busy.open(0);
    busy.close(0, release);
    busy.open(0);
    busy.close(0, release);
    expect(live.load() == 1, "all given back"); // the lost set, counted above
}

int main()
{
    check_steps();
    check_pool();
    std::printf("failures %d\n", failures);
    return failures == 0 ? 0 : 1;
}
