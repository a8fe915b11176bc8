/*
 * m3_staging.h - the order of the steps of a host copy that goes through
 * pinned staging memory (m3_hip_runtime.hip). Plain C++ (no HIP), so that
 * the CPU tests can compile it on its own and make its steps fail.
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

/* Device to host through `buffer`, which holds `bytes` bytes, in chunks of
 * `most` bytes: the host copies a chunk out while the next ones arrive. */
template <typename Ops>
int m3_stage_read(Ops &ops, uint8_t *buffer, uint8_t *destination,
                  const uint8_t *source, size_t bytes, size_t most,
                  bool *reusable)
{
    uint32_t first = 0U;
    int code = 0;

    for (size_t done = 0U; code == 0 && done < bytes; done += most) {
        uint32_t sequence = 0U;

        code = ops.queue(buffer + done, source + done,
                         std::min(bytes - done, most), &sequence);
        first = done == 0U ? sequence : first;
    }
    for (size_t done = 0U; code == 0 && done < bytes; done += most) {
        code = ops.wait(first + (uint32_t)(done / most));
        if (code == 0) {
            std::memcpy(destination + done, buffer + done,
                        std::min(bytes - done, most));
        }
    }
    return m3_stage_settle(ops, code, reusable);
}

#endif
