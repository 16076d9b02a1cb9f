// Large copies between a caller's pageable memory and the device.
#pragma once
#include <thread>
#include "runtime.hpp"

namespace bte {

struct StageThread {
    std::thread t;
    ~StageThread() {
        if (t.joinable()) t.join();
    }
};

// Copies through pinned chunks that two host threads fill or empty while
// the chunks before them are on the bus. A plain hipMemcpy of pageable memory
// has one thread do both the copy into its own staging buffer and, for memory
// that was never written (the caller's zero pages), the page faults: 128 MB
// took 4.6 ms up and 13 ms down into fresh memory, now 3.0 ms each way
// (43 GB/s). Chunks of 4 MB: 2 MB with 2 to 8 threads took 3.4 ms each way,
// 1 MB 4.4 ms, as each copy costs the bus about 16 us more.
// The pinned chunks (BYTES of them in all) are kept by the context, as their
// own first touch costs 0.4 ms per MB, and serve one call at a time: a call
// that finds them in use by another thread copies the plain way, as does one
// that gets no pinned memory; threads that cannot be started are done without.
//
// Copies below STAGE_MIN bytes, and from or to memory that the runtime knows
// (pinned, managed or device memory), are plain: a build's time outside the
// device is 1.5 ms either way with 10 to 13 MB each way and 4.0 (plain) or
// 3.5 ms (staged) with 32 MB; with 8 MB in BF16 it is 1.4 or 2.3 ms.
class Staging {
public:
    static constexpr size_t STAGE_MIN = (size_t)16 << 20;
    explicit Staging(Ctx* ctx) : c(ctx) {}
    ~Staging();
    Staging(const Staging&) = delete;
    Staging& operator=(const Staging&) = delete;
    // src has been read when upload returns; the copy is ordered on the
    // context's stream
    void upload(void* dst, const void* src, size_t bytes);
    // asks for dst's pages, from a thread beside the device's work, without
    // changing what they hold; ends before download begins
    void prefault(void* dst, size_t bytes);
    // after all work on the context's stream; dst is complete on return
    void download(void* dst, const void* src, size_t bytes);

private:
    static constexpr size_t CHUNK = (size_t)4 << 20;
    static constexpr int THREADS = 2, SLOTS = 2;
    static constexpr size_t BYTES = CHUNK * THREADS * SLOTS;
    Ctx* c;
    bool mine = false;  // the context's chunks are this object's
    StageThread bg;
    bool ready(const void* user, size_t bytes);
};

}  // namespace bte
