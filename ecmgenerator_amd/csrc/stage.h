// stage.h -- host batches through page-locked memory on their way to the
// device, apart from the device calls themselves.
#pragma once

#include <stddef.h>
#include <string.h>

#include <algorithm>

namespace ecm {

// Whether a host call of `rows` rows goes through page-locked memory, which its
// handle keeps from then on.  Not a handle's first call with few rows:
// allocating 4 MiB of it takes some 80 us (256 KiB 60, and 1.5 MiB, below the
// runtime's large pages, 300), and such a call gains 20-30 from it.  A first
// forward of 1 row takes 42 us without and 97 with it, of 300 rows 71 and 140,
// of 1,000 rows 250 and 165.
constexpr size_t kFirstCallRows = 512;
inline bool stage_page_locked(bool first_call, size_t rows) { return !first_call || rows > kFirstCallRows; }

// Pieces of one call's host data: each piece's copy runs while the next is
// filled.  Pageable buffers are copied by the runtime into memory of its own
// first, piece by piece with waits between.
//
// Queue is the device's side: copy(dst, src, bytes) queues a copy to the
// device and wait() waits for everything queued, both 0 on success.  The
// pieces belong to the handle, so no call may end with copies in flight: the
// next one would fill the same memory.  A call that waits for the queue
// itself says so (waited); any other return, with an error from a launch say,
// waits in the destructor.
template <typename Queue>
class Stager {
public:
    Stager(Queue& q, unsigned char* mem, size_t piece_bytes, size_t pieces)
        : q_(q), mem_(mem), bytes_(piece_bytes), pieces_(pieces) {}
    Stager(const Stager&) = delete;
    Stager& operator=(const Stager&) = delete;
    ~Stager() {
        if (in_flight_) (void)q_.wait();
    }
    // fill(to, at, len) writes bytes [at, at + len) of the data
    template <typename F>
    int put(void* dst, size_t bytes, F&& fill) {
        for (size_t at = 0; at < bytes; at += bytes_, ++next_) {
            if (next_ == pieces_) {                  // their memory is used again
                if (int rc = q_.wait()) return rc;
                next_ = 0;
            }
            unsigned char* to = mem_ + next_ * bytes_;
            const size_t len = std::min(bytes_, bytes - at);
            fill(to, at, len);
            in_flight_ = true;
            if (int rc = q_.copy((unsigned char*)dst + at, to, len)) return rc;
        }
        return 0;
    }
    int put(void* dst, const void* src, size_t bytes) {
        return put(dst, bytes, [&](void* to, size_t at, size_t len) { memcpy(to, (const unsigned char*)src + at, len); });
    }
    void waited() { in_flight_ = false; }

private:
    Queue& q_;
    unsigned char* mem_;
    size_t bytes_, pieces_, next_ = 0;
    bool in_flight_ = false;
};

}  // namespace ecm
