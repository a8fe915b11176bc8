/*
 * m3_staging.h - the order of the steps of a host copy that goes through
 * pinned staging memory, and the memory's owner (m3_hip_runtime.hip). Plain
 * C++ (no HIP), so that the CPU tests can compile it on its own and make its
 * steps fail.
 *
 * `Ops` is the stream:
 *   int queue(destination, source, bytes, sequence)  queues the copy of one
 *       chunk and, behind it, the completion number *sequence; on failure
 *       the copy may have been queued all the same
 *   int wait(sequence)  waits until that number has arrived
 *   bool drain()        waits for everything queued; false when it cannot
 * Codes are 0 for success. A step that fails leaves kernels that may still
 * read or write the staging memory, so the memory is handed on (*reusable)
 * only after a drain.
 */
#ifndef M3_STAGING_H
#define M3_STAGING_H

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <mutex>

/* After a copy that ended with `code`: what of it is still on its way. */
template <typename Ops>
int m3_stage_settle(Ops &ops, int code, bool *reusable)
{
    *reusable = code == 0 || ops.drain();
    return code;
}

/* Host to device through `buffer`, in one piece; the device has the bytes
 * when it returns 0. */
template <typename Ops>
int m3_stage_write(Ops &ops, uint8_t *buffer, uint8_t *destination,
                   const uint8_t *source, size_t bytes, bool *reusable)
{
    uint32_t sequence = 0U;
    int code;

    std::memcpy(buffer, source, bytes);
    code = ops.queue(destination, buffer, bytes, &sequence);
    if (code == 0) {
        code = ops.wait(sequence);
    }
    return m3_stage_settle(ops, code, reusable);
}

/* Device to host through `buffer`, which holds kStageChunks chunks of `most`
 * bytes, used in turn: the host copies a chunk out while the next one
 * arrives. */
constexpr size_t kStageChunks = 2U;

template <typename Ops>
int m3_stage_read(Ops &ops, uint8_t *buffer, uint8_t *destination,
                  const uint8_t *source, size_t bytes, size_t most,
                  bool *reusable)
{
    const size_t chunks = (bytes + most - 1U) / most;
    uint32_t numbers[kStageChunks] = {};
    size_t queued = 0U;
    int code = 0;

    for (size_t c = 0U; code == 0 && c < chunks; ++c) {
        for (; code == 0 && queued < chunks && queued < c + kStageChunks;
             ++queued) {
            code = ops.queue(buffer + (queued % kStageChunks) * most,
                             source + queued * most,
                             std::min(bytes - queued * most, most),
                             &numbers[queued % kStageChunks]);
        }
        if (code == 0) {
            code = ops.wait(numbers[c % kStageChunks]);
        }
        if (code == 0) {
            std::memcpy(destination + c * most,
                        buffer + (c % kStageChunks) * most,
                        std::min(bytes - c * most, most));
        }
    }
    return m3_stage_settle(ops, code, reusable);
}

/* The process's staging memory: at most SETS sets per GPU, lent to one copy
 * at a time. A copy is complete when its call returns, so a set belongs to
 * nobody between calls, and all handles and threads on a GPU share the few
 * there are: a session neither allocates nor frees staging memory unless
 * more copies run at once than ever before. When the last handle on a GPU
 * closes, its sets are freed but for one, and that one too when no copy
 * used it since the last handle closed before; so a program that opens one
 * session after another keeps a set, and one that stopped copying does not.
 * Copies that find no set (SETS of them lent, or an allocation that failed,
 * which is not tried again while the handles of that time are open) go
 * through the runtime instead. */
struct m3_stage_set {
    uint8_t *memory;   /* null: not allocated */
    uint32_t index;    /* among its GPU's sets */
    uint32_t sequence; /* the last completion number queued for it */
    bool lent;         /* or lost: queued work may still touch it */
    bool used;         /* since the last handle closed before */
};

template <int ORDINALS, int SETS>
class m3_stage_pool {
public:
    void open(int ordinal)
    {
        if (known(ordinal)) {
            const std::lock_guard<std::mutex> guard(gpus_[ordinal].lock);

            gpus_[ordinal].handles += 1U;
        }
    }

    template <typename Free>
    void close(int ordinal, Free free)
    {
        if (!known(ordinal)) {
            return;
        }
        gpu &g = gpus_[ordinal];
        const std::lock_guard<std::mutex> guard(g.lock);
        bool kept = false;

        g.handles -= 1U;
        if (g.handles != 0U) {
            return;
        }
        g.refused = false;
        for (m3_stage_set &set : g.sets) {
            if (set.memory == nullptr || set.lent) {
                continue;
            }
            if (!kept && set.used) {
                kept = true;
                set.used = false;
                continue;
            }
            free(set.memory);
            set = m3_stage_set();
        }
    }

    /* A set for one copy, or null. */
    template <typename Allocate>
    m3_stage_set *take(int ordinal, Allocate allocate)
    {
        if (!known(ordinal)) {
            return nullptr;
        }
        gpu &g = gpus_[ordinal];
        const std::lock_guard<std::mutex> guard(g.lock);

        m3_stage_set *found = nullptr;

        for (m3_stage_set &set : g.sets) {
            if (!set.lent && (found == nullptr || found->memory == nullptr)) {
                found = &set; /* an allocated one before others */
            }
        }
        if (found != nullptr && found->memory == nullptr && !g.refused) {
            found->memory = allocate();
            found->index = (uint32_t)(found - g.sets);
            g.refused = found->memory == nullptr;
        }
        if (found == nullptr || found->memory == nullptr) {
            return nullptr;
        }
        found->lent = true;
        found->used = true;
        return found;
    }

    /* Ends the loan; a set that is not reusable is never lent again. */
    void give(int ordinal, m3_stage_set *set, bool reusable)
    {
        if (reusable) {
            const std::lock_guard<std::mutex> guard(gpus_[ordinal].lock);

            set->lent = false;
        }
    }

private:
    struct gpu {
        std::mutex lock;
        uint32_t handles = 0U;
        bool refused = false; /* an allocation failed */
        m3_stage_set sets[SETS] = {};
    };

    static bool known(int ordinal)
    {
        return ordinal >= 0 && ordinal < ORDINALS;
    }

    gpu gpus_[ORDINALS];
};

#endif
