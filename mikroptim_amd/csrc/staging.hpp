// Host-device transfers of the host layer.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <initializer_list>
#include <stdexcept>
#include <string>
#include <vector>

namespace mko_host {

struct DeviceError : std::runtime_error {
    using std::runtime_error::runtime_error;
};

inline void hip_check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw DeviceError(std::string(what) + ": " + hipGetErrorString(e));
}

// Transfers between host arrays and device memory through pinned slots, ordered on the null stream.
// A copy of pageable memory stops the host at each array (11.5 us for the smallest) and runs at
// 12 ... 40 GB/s; a pinned one takes 2.5 us to issue and runs at 53 GB/s, and the host's copies in
// and out of the slots overlap it (11.5 MB to the host: 710 us pageable, 430 us this way, 210 us of
// it the copy). kSlots slots of 1 MiB (a copy costs some 20 us of its own: 256 KB slots take twice
// as long), each allocated at its first use, belong to one engine: its calls are not concurrent. A
// slot in flight is waited for before it is filled again.
class Staging {
public:
    struct Piece {
        void* host;
        const void* dev;
        size_t bytes;
        bool joined = false; // follows the piece before it in the same allocation
    };
    Staging() = default;
    Staging(const Staging&) = delete;
    Staging& operator=(const Staging&) = delete;
    ~Staging() {
        for (Slot& s : slots_) {
            if (s.done) {
                (void)hipEventSynchronize(s.done);
                (void)hipEventDestroy(s.done);
            }
            if (s.ptr) (void)hipHostFree(s.ptr);
        }
    }
    // Host to device; the source may change once this returns.
    void in(void* dev, const void* host, size_t bytes) {
        fill(dev, host, bytes);
        push();
    }
    // The same for several arrays of one allocation: adjacent ones go in one copy, the last of which
    // push() issues. An array of 2 MiB or more goes without a slot, as long as the source stays
    // until the null stream has passed the copy: 4 MiB take 135 us that way, through slots 82 us and
    // 64 of the host's copies.
    void stage(void* dev, const void* host, size_t bytes) {
        if (bytes >= 2 * kSlot) {
            push();
            hip_check(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, nullptr), "upload");
            return;
        }
        fill(dev, host, bytes);
    }
    void push() {
        const size_t n = run_bytes_;
        run_bytes_ = 0;
        used_ = std::min(kSlot, (used_ + 255) & ~size_t(255));
        if (n > 0)
            hip_check(hipMemcpyAsync(run_dev_, run_host_, n, hipMemcpyHostToDevice, nullptr),
                      "upload");
    }
    // Device to host; the pieces' host arrays hold the data when this returns. Joined pieces go in
    // one copy. On an error nothing is left in flight.
    void out(std::initializer_list<Piece> pieces) {
        size_t total = 0;
        for (const Piece& p : pieces) total += p.bytes;
        if (total == 0) return;
        try {
            const char* run = nullptr; // copy to the current slot that is not issued yet
            size_t run_bytes = 0;
            const auto issue = [&] {
                const size_t n = run_bytes;
                run_bytes = 0;
                if (n == 0) return;
                hip_check(hipMemcpyAsync(slots_[cur_].ptr + used_, run, n, hipMemcpyDeviceToHost,
                                         nullptr),
                          "download");
                used_ = std::min(kSlot, (used_ + n + 255) & ~size_t(255));
            };
            for (const Piece& p : pieces) {
                char* h = static_cast<char*>(p.host);
                const char* d = static_cast<const char*>(p.dev);
                if (!p.joined) issue();
                for (size_t left = p.bytes; left > 0;) {
                    if (room() == run_bytes) { // the slot is full
                        issue();
                        advance();
                    }
                    const size_t n = std::min(left, room() - run_bytes);
                    if (run_bytes == 0) run = d;
                    slots_[cur_].back.push_back({h, slots_[cur_].ptr + used_ + run_bytes, n});
                    run_bytes += n;
                    h += n;
                    d += n;
                    left -= n;
                }
            }
            issue();
            hip_check(hipEventRecord(slots_[cur_].done, nullptr), "download");
            slots_[cur_].busy = true;
            for (int i = 1; i <= kSlots; ++i) settle(slots_[(cur_ + i) % kSlots]);
        } catch (...) {
            (void)hipDeviceSynchronize();
            for (Slot& s : slots_) {
                s.back.clear();
                s.busy = false;
            }
            used_ = 0;
            throw;
        }
        used_ = 0; // the null stream has passed everything before the last event
    }

private:
    static constexpr size_t kSlot = size_t(1) << 20;
    static constexpr int kSlots = 8;
    struct Back {
        void* host;
        const char* slot;
        size_t bytes;
    };
    struct Slot {
        char* ptr = nullptr;
        hipEvent_t done = nullptr;
        bool busy = false;      // `done` is recorded behind the slot's last copy
        std::vector<Back> back; // to be copied to the host arrays after `done`
    };
    Slot slots_[kSlots];
    int cur_ = 0;
    size_t used_ = 0;
    char* run_dev_ = nullptr; // copy to the device being staged, at the end of the current slot
    const char* run_host_ = nullptr;
    size_t run_bytes_ = 0;

    // Copies the array into slots, behind what is staged already where that is adjacent.
    void fill(void* dev, const void* host, size_t bytes) {
        char* d = static_cast<char*>(dev);
        const char* h = static_cast<const char*>(host);
        while (bytes > 0) {
            try {
                if (run_bytes_ > 0 && d != run_dev_ + run_bytes_) push();
                if (room() == 0) advance();
            } catch (...) {
                run_bytes_ = 0; // a later call must not issue it
                throw;
            }
            const size_t n = std::min(bytes, room());
            char* slot = slots_[cur_].ptr + used_;
            if (run_bytes_ == 0) {
                run_dev_ = d;
                run_host_ = slot;
            }
            std::memcpy(slot, h, n);
            used_ += n;
            run_bytes_ += n;
            d += n;
            h += n;
            bytes -= n;
        }
    }
    size_t room() {
        Slot& s = slots_[cur_];
        if (!s.ptr) {
            if (!s.done)
                hip_check(hipEventCreateWithFlags(&s.done, hipEventDisableTiming), "staging");
            hip_check(hipHostMalloc(reinterpret_cast<void**>(&s.ptr), kSlot, hipHostMallocDefault),
                      "staging");
        }
        return kSlot - used_;
    }
    void settle(Slot& s) {
        if (s.busy) hip_check(hipEventSynchronize(s.done), "staging");
        s.busy = false;
        for (const Back& b : s.back) std::memcpy(b.host, b.slot, b.bytes);
        s.back.clear();
    }
    void advance() {
        push();
        hip_check(hipEventRecord(slots_[cur_].done, nullptr), "staging");
        slots_[cur_].busy = true;
        cur_ = (cur_ + 1) % kSlots;
        used_ = 0;
        settle(slots_[cur_]);
    }
};

} // namespace mko_host
