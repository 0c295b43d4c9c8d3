// Staged copies between the device and pageable host memory (transfer.h).
#include "transfer.h"
#include <algorithm>
#include <cstring>
#include <system_error>
#include "core.h"

namespace rm {

namespace {

// Measured on copies into fresh memory of 2 MB pages: one thread takes 2.4 ms
// for 33 MB, 4 take 0.84, 8 0.62, 12 0.57-0.67 (the DMA: 0.6); of 4 KB pages
// 7.0, 2.5, 1.5 and 1.2 ms.
constexpr unsigned kWorkers = 8;
// A DMA and its event cost some 25 us beside the transfer, so a block is far
// larger than a worker's chunk.  A 1920x1080 RGBA image read in slots of 8 MB
// and chunks of 1 MB takes 1.32 ms (plain 2.33), in slots of 2 MB 1.45, 4 MB
// 1.37, 16 MB 1.34, in chunks of 512 KB 1.49 and 2 MB 1.33; 1M rays to the
// device and their hits back 1.92 (plain 3.07), 2.25, 2.03, 2.07, 2.14, 1.98.
constexpr size_t kChunkBytes = (size_t)1 << 20;
constexpr size_t kSlotBytes = (size_t)8 << 20;
constexpr size_t kSlots = 4;
// Slots on the way to the device while the workers fill the others.
constexpr size_t kInFlight = 2;
// Smaller copies are left to the runtime's own staging: 2.7 MB to the host
// take 0.20 ms either way, 4.2 MB 0.23 (plain 0.31), 6.6 MB 0.18 (0.23); 2 MB
// to the device and 1.3 MB back take 0.06 ms more staged.
constexpr size_t kStagedMin = (size_t)3 << 20;

}  // namespace

HostCopies::~HostCopies() {
    {
        std::lock_guard<std::mutex> l(mutex_);
        stop_ = true;
    }
    wake_.notify_all();
    for (std::thread& t : workers_) t.join();
    for (size_t i = 0; i < events_.size(); i++) {
        if (pending_[i]) (void)hipEventSynchronize(events_[i]);
        (void)hipEventDestroy(events_[i]);
    }
    if (slots_) (void)hipHostFree(slots_);
}

// Slots, events and workers on first use.  False when they cannot be had: the
// copies then go the plain way.
bool HostCopies::prepare() {
    if (prepared_) return usable_;
    prepared_ = true;
    // allocating must not end a capture that another thread has under way
    struct Relaxed {
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
        ~Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    } relaxed;
    // the events belong to the streams' device, whichever is current
    struct Current {
        int device = 0;
        bool set;
        explicit Current(int ordinal) { set = hipGetDevice(&device) == hipSuccess && hipSetDevice(ordinal) == hipSuccess; }
        ~Current() {
            if (set) (void)hipSetDevice(device);
        }
    } current(ordinal_);
    if (!current.set) return false;
    if (hipHostMalloc(reinterpret_cast<void**>(&slots_), kSlots * kSlotBytes, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        slots_ = nullptr;
        return false;
    }
    pending_.assign(kSlots, 0);
    for (size_t i = 0; i < kSlots; i++) {
        hipEvent_t e;
        if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        events_.push_back(e);
    }
    const unsigned n = std::min(kWorkers, std::max(2u, std::thread::hardware_concurrency() / 2));
    try {
        for (unsigned i = 0; i < n; i++) workers_.emplace_back([this] { work(); });
    } catch (const std::system_error&) {
        if (workers_.empty()) return false;
    }
    return usable_ = true;
}

// Whether the pieces are worth staging: enough bytes, and ordinary host
// memory that does not overlap (memory the runtime knows, pinned or of a
// device, is left to it).
bool HostCopies::staged(const std::vector<CopyPiece>& pieces) const {
    size_t bytes = 0;
    for (const CopyPiece& p : pieces) bytes += p.bytes;
    if (bytes < kStagedMin) return false;
    for (size_t i = 0; i < pieces.size(); i++) {
        const CopyPiece& p = pieces[i];
        hipPointerAttribute_t at{};
        if (hipPointerGetAttributes(&at, p.host) != hipSuccess) (void)hipGetLastError();
        else if (at.type != hipMemoryTypeUnregistered) return false;
        for (size_t j = 0; j < i; j++) {
            const char *a = static_cast<const char*>(p.host), *b = static_cast<const char*>(pieces[j].host);
            if (a < b + pieces[j].bytes && b < a + p.bytes) return false;
        }
    }
    return true;
}

// Chunks end at multiples of their size in the host's address space.
void HostCopies::cut(const std::vector<CopyPiece>& pieces) {
    parts_.clear();
    chunks_.clear();
    blocks_.clear();
    size_t off = 0;  // in the open block's slot
    auto close = [&] {
        blocks_.push_back(Block{parts_.size(), chunks_.size()});
        off = 0;
    };
    for (const CopyPiece& p : pieces) {
        char* h = static_cast<char*>(p.host);
        char* d = static_cast<char*>(p.device);
        for (size_t left = p.bytes; left;) {
            const size_t part = std::min(left, kSlotBytes - off);
            parts_.push_back(Part{off, d, part});
            for (size_t done = 0; done < part;) {
                const size_t n = std::min(part - done, kChunkBytes - (size_t)(reinterpret_cast<uintptr_t>(h) % kChunkBytes));
                chunks_.push_back(Chunk{blocks_.size(), off + done, h, n});
                h += n;
                done += n;
            }
            d += part;
            left -= part;
            off = (off + part + 255) & ~(size_t)255;
            if (off >= kSlotBytes) close();
        }
    }
    if (off) close();
}

void HostCopies::begin(const std::vector<CopyPiece>& pieces, bool to_host) {
    std::lock_guard<std::mutex> l(mutex_);
    cut(pieces);
    unfinished_.clear();
    for (size_t b = 0, first = 0; b < blocks_.size(); first = blocks_[b++].chunks_end)
        unfinished_.push_back(blocks_[b].chunks_end - first);
    released_ = claimed_ = finished_count_ = 0;
    to_host_ = to_host;
}

// Enqueues a block's DMA.
void HostCopies::transfer(size_t block, hipStream_t st) {
    const size_t slot = block % kSlots;
    for (size_t i = block ? blocks_[block - 1].parts_end : 0; i < blocks_[block].parts_end; i++) {
        const Part& p = parts_[i];
        char* h = slots_ + slot * kSlotBytes + p.slot_offset;
        RM_HIP(to_host_ ? hipMemcpyAsync(h, p.device, p.bytes, hipMemcpyDeviceToHost, st)
                        : hipMemcpyAsync(p.device, h, p.bytes, hipMemcpyHostToDevice, st));
    }
    RM_HIP(hipEventRecord(events_[slot], st));
    pending_[slot] = 1;
}

void HostCopies::release_block(size_t block) {
    {
        std::lock_guard<std::mutex> l(mutex_);
        released_ = blocks_[block].chunks_end;
    }
    wake_.notify_all();
}

// Until the workers have finished every released chunk: the caller's memory
// and the slots are theirs no longer, and the lists may go.
void HostCopies::drain() {
    std::unique_lock<std::mutex> l(mutex_);
    finished_cv_.wait(l, [&] { return finished_count_ == released_; });
    released_ = claimed_ = finished_count_ = 0;
}

void HostCopies::wait_finished(size_t block) {
    std::unique_lock<std::mutex> l(mutex_);
    finished_cv_.wait(l, [&] { return unfinished_[block] == 0; });
}

bool HostCopies::is_finished(size_t block) {
    std::lock_guard<std::mutex> l(mutex_);
    return unfinished_[block] == 0;
}

void HostCopies::wait_slot(size_t slot) {
    if (!pending_[slot]) return;
    RM_HIP(hipEventSynchronize(events_[slot]));
    pending_[slot] = 0;
}

void HostCopies::work() {
    std::unique_lock<std::mutex> l(mutex_);
    for (;;) {
        wake_.wait(l, [&] { return stop_ || claimed_ < released_; });
        if (stop_) return;
        const Chunk c = chunks_[claimed_++];
        char* slot = slots_ + (c.block % kSlots) * kSlotBytes + c.slot_offset;
        const bool down = to_host_;
        l.unlock();
        std::memcpy(down ? c.host : slot, down ? slot : c.host, c.bytes);
        l.lock();
        finished_count_++;
        if (--unfinished_[c.block] == 0) finished_cv_.notify_one();
    }
}

void HostCopies::to_host(const std::vector<CopyPiece>& pieces, hipStream_t st) {
    std::unique_lock<std::mutex> use(in_use_, std::defer_lock);
    if (!staged(pieces) || !use.try_lock() || !prepare()) {
        for (const CopyPiece& p : pieces)
            if (p.bytes) RM_HIP(hipMemcpyAsync(p.host, p.device, p.bytes, hipMemcpyDeviceToHost, st));
        RM_HIP(hipStreamSynchronize(st));
        return;
    }
    begin(pieces, true);
    struct Drain {
        HostCopies* h;
        ~Drain() { h->drain(); }
    } drained{this};
    size_t issued = 0;
    for (size_t next = 0; next < blocks_.size(); next++) {
        for (; issued < blocks_.size() && issued < next + kSlots; issued++) {
            if (issued >= kSlots) {
                // a slot that the workers still read waits, unless no DMA is ahead
                if (issued == next) wait_finished(issued - kSlots);
                else if (!is_finished(issued - kSlots)) break;
            } else {
                wait_slot(issued % kSlots);
            }
            transfer(issued, st);
        }
        wait_slot(next % kSlots);
        release_block(next);
    }
}

void HostCopies::to_device(void* device, const void* host, size_t bytes, hipStream_t st) {
    if (bytes == 0) return;
    const std::vector<CopyPiece> pieces{CopyPiece{const_cast<void*>(host), device, bytes}};
    std::unique_lock<std::mutex> use(in_use_, std::defer_lock);
    if (!staged(pieces) || !use.try_lock() || !prepare()) {
        RM_HIP(hipMemcpyAsync(device, host, bytes, hipMemcpyHostToDevice, st));
        return;
    }
    begin(pieces, false);
    struct Drain {
        HostCopies* h;
        ~Drain() { h->drain(); }
    } drained{this};
    size_t released = 0;
    for (size_t next = 0; next < blocks_.size(); next++) {
        for (; released < blocks_.size() && released < next + kSlots - kInFlight; released++) {
            wait_slot(released % kSlots);
            release_block(released);
        }
        wait_finished(next);
        transfer(next, st);
    }
}

}  // namespace rm
