// Copies between the device and pageable host memory of the caller.
//
// A plain hipMemcpyAsync into memory that the caller has just allocated is
// bound by one thread's page faults and memcpy: 33 MB take 2.4 ms, four times
// the DMA's 0.6 ms.  HostCopies moves such copies in blocks through a ring of
// pinned slots, where the DMA of one block overlaps the memcpy of others by a
// few worker threads.
//
// The first copy of 3 MB or more sets this up: 32 MB of pinned slots, four
// events, up to eight threads, kept until the device is destroyed.  Reading a
// 1920x1080 image takes 10.2-10.8 ms the first time in a process and 1.3-1.45
// later; plain copies, whose own staging the runtime sets up, took 15.8-16.2
// and 2.5.
#pragma once
#include <hip/hip_runtime.h>
#include <condition_variable>
#include <cstdint>
#include <mutex>
#include <thread>
#include <vector>

namespace rm {

// Arrays of at most this size together go in one copy, with a memcpy on the
// host: a copy costs some 10 us beside its bytes.  Closest hits of one ray take
// 32 us with one copy back and 64 with four, of 52000 rays (1 MB) 207 either
// way, of 80000 305 against 271; a training step of one row takes 60 us with one
// copy there and 73-85 with two, of 17000 rows (1 MB) 247 against 252, of 30000
// 418 against 389.
constexpr size_t kOneCopyMax = (size_t)1 << 20;

struct CopyPiece {
    void* host;
    void* device;
    size_t bytes;
};

class HostCopies {
public:
    explicit HostCopies(int ordinal) : ordinal_(ordinal) {}
    HostCopies(const HostCopies&) = delete;
    HostCopies& operator=(const HostCopies&) = delete;
    ~HostCopies();

    // Copies in the stream's order; returns when the host has the data.
    void to_host(const std::vector<CopyPiece>& pieces, hipStream_t st);
    // Copies in the stream's order; returns when the host memory may change.
    void to_device(void* device, const void* host, size_t bytes, hipStream_t st);

private:
    // a DMA's worth of the copy, one slot: one transfer per piece in it
    struct Part {
        size_t slot_offset;
        char* device;
        size_t bytes;
    };
    struct Block {
        size_t parts_end, chunks_end;  // in parts_, chunks_
    };
    // one worker's memcpy
    struct Chunk {
        size_t block, slot_offset;
        char* host;
        size_t bytes;
    };
    bool staged(const std::vector<CopyPiece>& pieces) const;
    bool prepare();
    void cut(const std::vector<CopyPiece>& pieces);
    void begin(const std::vector<CopyPiece>& pieces, bool to_host);
    void transfer(size_t block, hipStream_t st);
    void release_block(size_t block);
    void drain();
    void wait_finished(size_t block);
    bool is_finished(size_t block);
    void wait_slot(size_t slot);
    void work();

    const int ordinal_;
    std::mutex in_use_;  // one staged copy at a time
    bool prepared_ = false, usable_ = false;
    char* slots_ = nullptr;
    std::vector<hipEvent_t> events_;
    std::vector<uint8_t> pending_;  // the slot's DMA has been enqueued and not waited for
    std::vector<std::thread> workers_;

    // the copy in hand, shared with the workers
    std::mutex mutex_;
    std::condition_variable wake_, finished_cv_;
    std::vector<Part> parts_;
    std::vector<Chunk> chunks_;
    std::vector<Block> blocks_;
    std::vector<size_t> unfinished_;  // per block: chunks not yet copied
    size_t released_ = 0, claimed_ = 0, finished_count_ = 0;
    bool to_host_ = false, stop_ = false;
};

}  // namespace rm
