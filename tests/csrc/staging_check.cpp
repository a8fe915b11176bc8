// The steps of a staged host copy (m3.c_amd/csrc/hip/m3_staging.h) on the
// CPU, over a stream that runs nothing until it is waited for: what arrives,
// and that a step that fails never hands the staging memory on while a
// queued copy could still touch it.
#include "m3_staging.h"

#include <cstdio>
#include <functional>
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

int main()
{
    const size_t most = 4096;
    std::vector<uint8_t> source(5 * most + 7), target(source.size()),
        buffer(source.size() + 64);

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
    std::printf("failures %d\n", failures);
    return failures == 0 ? 0 : 1;
}
