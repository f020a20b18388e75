// Device memory that the engine keeps between calls, for one device and under the engine's mutex.
// hipMalloc + hipFree cost an SPI call and a wait for the device (quantMatvec + release in a loop 14.9 -> 5.1 us
// a call without them; a token of ten calls, whose downloads wait anyhow, 66.4 -> 62.9);
// hipMallocAsync + hipFreeAsync cost a call with a workspace ~15 us and, on this runtime, a wait for the
// work before it (two launches of 50 us each: the host returns after 106 us with them, after 6 without).
//  - Blocks of released F32 / BF16 / I8 buffers, in powers of two from 256 bytes to 4 MiB, at
//    most 64 MiB in all: work on such a buffer runs on the engine stream alone, so its block may
//    be written again behind it with no wait. A buffer whose address left the engine
//    (j4q_buffer_info) can be in use on other streams and goes back with hipFree, which waits.
//  - Workspaces of up to 256 MiB each, 512 MiB in all. One serves the calls on the engine stream, which
//    run one after another. The others serve any stream of a caller's: an event that the last launch of a
//    call completes guards them, and the next call's stream waits for it, so nothing rests on which
//    stream a handle names. The wait costs nothing on the stream that used it last, and the event none of
//    the GPU's time (without a system fence; with one 1.9 us a call, recorded by itself 1.1).
//  - None of it serves a call under stream capture: a graph keeps the addresses it recorded, its operands'
//    too, and may be launched on any stream. Those buffers go back with hipFree as well.
// All of it is given back when the last buffer is released or memory is short.
#pragma once

#include <stdint.h>

#include <vector>

#include "j4q_common.h"

namespace j4q {

inline bool capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return st != hipStreamCaptureStatusNone;
}

// Another stream may be under capture, where only a relaxed thread may allocate, free or query.
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

class BlockCache {
public:
    static constexpr uint64_t kMaxBlock = 4ull << 20, kMaxBytes = 64ull << 20;
    static int slot(uint64_t n) {
        int k = 8;
        while ((1ull << k) < n) k++;
        return k;
    }
    void *take(int k) {
        if (free_[k].empty()) return nullptr;
        void *p = free_[k].back();
        free_[k].pop_back();
        bytes_ -= 1ull << k;
        return p;
    }
    bool give(void *p, int k) {
        if (bytes_ + (1ull << k) > kMaxBytes) return false;
        free_[k].push_back(p);
        bytes_ += 1ull << k;
        return true;
    }
    uint64_t bytes() const { return bytes_; }
    void clear() {
        const RelaxedCapture relaxed;
        for (auto &v : free_) {
            for (void *p : v) (void)hipFree(p);
            v.clear();
        }
        bytes_ = 0;
    }

private:
    std::vector<void *> free_[23];  // by log2 of the block size
    uint64_t bytes_ = 0;
};

class Workspaces {
public:
    static constexpr uint64_t kMaxOne = 256ull << 20, kMaxAll = 512ull << 20;

    // `blocks` are given back too where memory is short.
    explicit Workspaces(BlockCache &blocks) : blocks_(blocks) {}

    uint64_t bytes() const { return bytes_; }

    // A workspace of `bytes` for the work that the caller enqueues on `s` before it calls end(). The last
    // launch that uses it completes ws->done, if there is one.
    hipError_t begin(hipStream_t s, hipStream_t engine, uint64_t bytes, Workspace *ws) {
        *ws = Workspace();
        const bool captured = capturing(s);
        if (bytes <= kMaxOne && !captured) {
            const Slot *t = s == engine ? engine_slot(engine, bytes) : shared_slot(s, bytes);
            if (t && (!t->done || hipStreamWaitEvent(s, t->done, 0) == hipSuccess)) {
                ws->ptr = (float *)t->ptr;
                ws->bytes = bytes;
                ws->done = t->done;
                return hipSuccess;
            }
            (void)hipGetLastError();
        }
        void *p = nullptr;
        hipError_t e = hipMallocAsync(&p, bytes, s);
        if (e == hipErrorOutOfMemory && !captured && (bytes_ || blocks_.bytes())) {
            (void)hipGetLastError();
            give_back();
            e = hipMallocAsync(&p, bytes, s);
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();  // a launch checks for errors by the last one
            return e;
        }
        ws->ptr = (float *)p;
        ws->bytes = bytes;
        ws->stream_ordered = true;
        return hipSuccess;
    }

    // launched: whether every launch went out (else ws.done may not have been handed to one).
    void end(hipStream_t s, const Workspace &ws, bool launched) {
        if (ws.stream_ordered) (void)hipFreeAsync(ws.ptr, s);
        else if (ws.done && !launched) (void)hipEventRecord(ws.done, s);
    }

    // Everything kept, the blocks too; waits for the device.
    void give_back() {
        blocks_.clear();
        const RelaxedCapture relaxed;
        for (const Slot &t : shared_) drop(t);
        shared_.clear();
        drop(engine_);
        engine_ = Slot();
        bytes_ = 0;
    }

private:
    struct Slot {
        void *ptr = nullptr;
        uint64_t bytes = 0;
        hipEvent_t done = nullptr;   // none: the engine stream's
        hipStream_t last = nullptr;  // where it was used last: a first guess at what is free, no more
    };
    BlockCache &blocks_;
    Slot engine_;
    std::vector<Slot> shared_;
    uint64_t bytes_ = 0;

    static void drop(const Slot &t) {
        if (t.ptr) (void)hipFree(t.ptr);
        if (t.done) (void)hipEventDestroy(t.done);
    }
    static bool idle(const Slot &t) {
        const bool is = hipEventQuery(t.done) == hipSuccess;
        (void)hipGetLastError();
        return is;
    }
    static hipEvent_t new_event() {
        hipEvent_t e = nullptr;
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming | hipEventDisableSystemFence) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        return e;
    }
    // Memory for a workspace of `bytes`, in powers of two so that growing calls grow it rarely.
    bool alloc(uint64_t bytes, Slot *t) {
        const RelaxedCapture relaxed;
        uint64_t want = 1ull << 20;
        while (want < bytes) want *= 2;
        if (bytes_ + want > kMaxAll)  // what no call uses any more (hipFree waits for the device)
            for (size_t i = shared_.size(); i-- > 0;)
                if (idle(shared_[i])) {
                    drop(shared_[i]);
                    bytes_ -= shared_[i].bytes;
                    shared_.erase(shared_.begin() + (long)i);
                }
        for (int attempt = 0; attempt < 3; attempt++) {
            if (attempt == 1) want = bytes;  // no more than is needed
            if (attempt == 2) {
                if (!blocks_.bytes()) return false;
                blocks_.clear();
            }
            if (bytes_ + want > kMaxAll) continue;
            if (hipMalloc(&t->ptr, want) == hipSuccess) {
                t->bytes = want;
                bytes_ += want;
                return true;
            }
            (void)hipGetLastError();
        }
        t->ptr = nullptr;
        return false;
    }
    const Slot *engine_slot(hipStream_t engine, uint64_t bytes) {
        if (bytes <= engine_.bytes) return &engine_;
        Slot t;
        if (!alloc(bytes, &t)) return nullptr;
        const RelaxedCapture relaxed;
        if (engine_.ptr) {  // its calls may still run: any stream's once they are done
            engine_.done = new_event();
            if (engine_.done && hipEventRecord(engine_.done, engine) == hipSuccess) {
                shared_.push_back(engine_);
            } else {
                (void)hipGetLastError();
                bytes_ -= engine_.bytes;
                drop(engine_);
            }
        }
        engine_ = t;
        return &engine_;
    }
    const Slot *shared_slot(hipStream_t s, uint64_t bytes) {
        Slot *best = nullptr;
        for (Slot &t : shared_)
            if (t.bytes >= bytes && t.last == s) best = &t;
        if (!best) {
            const RelaxedCapture relaxed;
            for (Slot &t : shared_)
                if (!best && t.bytes >= bytes && idle(t)) best = &t;
        }
        if (!best) {
            Slot t;
            t.done = new_event();
            if (!t.done) return nullptr;
            if (!alloc(bytes, &t)) {
                (void)hipEventDestroy(t.done);
                return nullptr;
            }
            shared_.push_back(t);
            best = &shared_.back();
        }
        best->last = s;
        return best;
    }
};

}  // namespace j4q
