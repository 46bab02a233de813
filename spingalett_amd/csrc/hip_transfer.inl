// hip_transfer.inl — large transfers between ordinary (pageable) host memory and the device.  Part of hip_forward.hip's
// translation unit.
//
// Array by array each transfer begins when the one before has ended: the arrays of a training of 784-512-1000-10, 26 MB there
// and back in 42 calls of the runtime's, took 1.9 ms; 0.77 here with the launches of one epoch.  A few threads copy between the
// caller's memory and a ring of pinned chunks while other chunks are on the bus (54 GB/s): the bus is the bound as long as the
// host's copies keep up, which four threads do (55 GB/s; one thread 31, eight no more than four).  The helpers start once per call,
// take parts of chunks in order and sleep while there is none.  The first chunks are small, so that the bus does not wait for a whole
// one to be filled, nor the host for a whole one to arrive.

namespace {

constexpr size_t kStageChunk = 8u << 20, kFirstChunk = 512u << 10, kStagePart = 256u << 10;
// Single arrays below these sizes are left to the runtime, which has the bus read the caller's pages up to 8 MB (2 / 5.5 / 8 /
// 15 / 31 MiB up 81 / 174 / 253 / 553 / 795 us, the last two copied into 8 MB chunks by four threads, against 105 / 202 / 278 /
// 408 / 739 here; 2 MB down 107 against 96, for which the ring is not worth its pinned memory).
constexpr size_t kStagedUp = 10u << 20, kStagedDown = 4u << 20, kHelperLeast = 1u << 20;
constexpr uint32_t kStageSlots = 4, kStageHelpers = 3, kIdleLooks = 1000;
constexpr uint32_t kInFlight = 8;              // chunks in the slots at once: six at most (slot_of)

// One ring for each direction: a download holds its own until all before it on the stream is done, which must not keep another
// thread's upload from filling chunks.  Three slots up: with a fourth, the slots and an array that is sent again and again no longer
// fit the host's cache together (32 MB 870 us, 805 with three; new arrays 751 and 750).
struct StageRing {
    const size_t chunk;                            // the longest
    const uint32_t slots;                          // kStageSlots at most
    void *buf[kStageSlots] = {};
    hipEvent_t ev[kStageSlots] = {}, start = nullptr;
    hipStream_t side = nullptr;                    // (with start: up only)
    bool ready = false;
    std::mutex mu;
    StageRing(size_t bytes, uint32_t count) : chunk(bytes), slots(count) {}
} g_up{kStageChunk, 3u}, g_down{4u * kFirstChunk, 4u};

// a contiguous part of a transfer; a transfer is its segments in a row, each beginning at a multiple of 64 bytes of it
struct Segment {
    char *host;
    char *dev;
    size_t bytes;
};

struct PieceArgs {
    struct { float *dev; uint32_t at, n; } p[16];   // at: first float in the chunk
    float *pin;
    int to_host;
};

// pieces of several arrays between their places and a pinned chunk, one per grid y
__global__ __launch_bounds__(256) void sp_move_pieces(const PieceArgs a)
{
    float *const dev = a.p[blockIdx.y].dev, *const pin = a.pin + a.p[blockIdx.y].at;
    const uint32_t n = a.p[blockIdx.y].n, quads = (reinterpret_cast<uintptr_t>(dev) & 15u) == 0 ? n / 4u : 0u;
    const float *const src = a.to_host ? dev : pin;
    float *const dst = a.to_host ? pin : dev;
    const uint32_t t = blockIdx.x * 256u + threadIdx.x, step = gridDim.x * 256u;
    for (uint32_t i = t; i < quads; i += step) reinterpret_cast<float4 *>(dst)[i] = reinterpret_cast<const float4 *>(src)[i];
    for (uint32_t i = 4u * quads + t; i < n; i += step) dst[i] = src[i];
}

class StagedTransfer {
public:
    StagedTransfer(const Segment *segments, uint32_t count, bool to_host)
        : seg_(segments), count_(count), to_host_(to_host), ring_(to_host ? g_down : g_up)
    {
        for (uint32_t i = 0; i < count; ++i) total_ += padded(segments[i].bytes);
        chunks_ = 0;
        while (chunk_at(chunks_) < total_) ++chunks_;
    }

    // The caller holds its ring's lock.  landed: see upload_from_host.
    int run(hipStream_t stream, const std::function<int(size_t)> &landed)
    {
        std::thread helpers[kStageHelpers];
        uint32_t started = 0, wanted = total_ / kHelperLeast < kStageHelpers ? (uint32_t)(total_ / kHelperLeast) : kStageHelpers;
        const int rc = pump(stream, landed, [&] {
            // (down: when the first chunk is here, which may be long after the call, behind everything the stream still does)
            try {
                for (; started < wanted; ++started) helpers[started] = std::thread([this] { help(); });
            } catch (...) {
                wanted = started;                       // no more threads to be had: fewer helpers
            }
        });
        {
            std::lock_guard<std::mutex> lock(mu_);
            stop_.store(true);
        }
        more_.notify_all();
        for (uint32_t t = 0; t < started; ++t) helpers[t].join();
        return rc;
    }

private:
    static size_t padded(size_t bytes) { return (bytes + 63u) & ~(size_t)63u; }

    // Where a chunk begins.  Up: at 0, 0.5, 1.5, 3.5, 8 MB and then every 8 (the bus rests for 9 us between two), so that what
    // runs over the first 8 MB that have landed need not wait for the next.  Down: at 0, 0.5, 1.5 MB and then every 2: the last
    // one's copy has nothing beside it.
    size_t chunk_at(uint32_t c) const
    {
        if (to_host_) return c < 3u ? kFirstChunk * ((1u << c) - 1u) : kFirstChunk * (3u + 4u * (size_t)(c - 2u));
        return c < 4u ? kFirstChunk * ((1u << c) - 1u) : (size_t)(c - 3u) * kStageChunk;
    }
    size_t chunk_end(uint32_t c) const { return std::min(chunk_at(c + 1u), total_); }

    // The slot a chunk lies in, and whether it is the first one there.  Up: the four that make 8 MB share one, so that the slots hold
    // 24 MB of a transfer that has to wait for the stream, and the call need not.
    uint32_t slot_of(uint32_t c) const { return (to_host_ ? c : c < 4u ? 0u : c - 3u) % ring_.slots; }
    bool begins_slot(uint32_t c) const { return to_host_ || c == 0u || c >= 4u; }
    char *chunk_pin(uint32_t c) const { return static_cast<char *>(ring_.buf[slot_of(c)]) + (begins_slot(c) ? 0u : chunk_at(c)); }

    // f(segment, offset in it, offset from `from`, bytes) for what lies in [from, to) of the transfer
    template <class F>
    void each(size_t from, size_t to, F &&f) const
    {
        size_t at = 0;
        for (uint32_t i = 0; i < count_; ++i) {
            const size_t lo = std::max(from, at), hi = std::min(to, at + seg_[i].bytes);
            if (lo < hi) f(seg_[i], lo - at, lo - from, hi - lo);
            at += padded(seg_[i].bytes);
            if (at >= to) break;
        }
    }

    // Copies the next part of an open chunk; false if there is none just now.  Parts are small: the calling thread is back at
    // the bus after each one, and a chunk that is full does not wait for it.
    bool copy_one()
    {
        size_t from = next_.load(std::memory_order_relaxed);
        do {
            if (from >= open_.load(std::memory_order_acquire)) return false;
        } while (!next_.compare_exchange_weak(from, from + kStagePart, std::memory_order_relaxed));
        uint32_t c = 0;
        while (chunk_at(c + 1u) <= from) ++c;
        const size_t to = std::min(from + kStagePart, total_);
        char *const pin = chunk_pin(c) + (from - chunk_at(c));
        each(from, to, [&](const Segment &s, size_t at, size_t in, size_t n) {
            if (to_host_) memcpy(s.host + at, pin + in, n);
            else memcpy(pin + in, s.host + at, n);
        });
        done_[c % kInFlight].fetch_add(1u, std::memory_order_release);
        return true;
    }

    // A helper looks for the next part for some 0.2 ms, longer than a chunk takes, and then sleeps: the next chunk may be behind everything
    // that the stream still does, for as long as that takes.
    void help()
    {
        for (uint32_t idle = 0; !stop_.load(std::memory_order_relaxed);) {
            if (copy_one()) {
                idle = 0;
            } else if (++idle < kIdleLooks) {
                std::this_thread::yield();
            } else {
                std::unique_lock<std::mutex> lock(mu_);
                more_.wait(lock, [this] { return stop_.load() || next_.load() < open_.load(); });
                idle = 0;
            }
        }
    }

    int submit(uint32_t c, hipStream_t stream)
    {
        char *const pin = chunk_pin(c);
        if (count_ == 1u) {
            const size_t at = chunk_at(c), n = std::min(chunk_end(c), seg_[0].bytes) - at;
            HCHECK(to_host_ ? hipMemcpyAsync(pin, seg_[0].dev + at, n, hipMemcpyDeviceToHost, stream)
                            : hipMemcpyAsync(seg_[0].dev + at, pin, n, hipMemcpyHostToDevice, stream));
        } else {
            PieceArgs a{};
            uint32_t pieces = 0, longest = 0;
            a.pin = reinterpret_cast<float *>(pin);
            a.to_host = to_host_;
            auto flush = [&] {
                if (!pieces) return;
                sp_move_pieces<<<dim3(std::min((longest / 4u + 255u) / 256u + 1u, 512u), pieces), 256, 0, stream>>>(a);
                pieces = longest = 0;
            };
            each(chunk_at(c), chunk_end(c), [&](const Segment &s, size_t at, size_t in, size_t n) {
                a.p[pieces] = {reinterpret_cast<float *>(s.dev + at), (uint32_t)(in / 4u), (uint32_t)(n / 4u)};
                longest = std::max(longest, (uint32_t)(n / 4u));
                if (++pieces == 16u) flush();
            });
            flush();
            HCHECK(hipGetLastError());
        }
        HCHECK(hipEventRecord(ring_.ev[slot_of(c)], stream));
        return 0;
    }

    // 0: the slot's last transfer has ended, 1: not yet, -1: an error
    int slot_busy(uint32_t slot) const
    {
        const hipError_t e = hipEventQuery(ring_.ev[slot]);
        if (e == hipSuccess) return 0;
        (void)hipGetLastError();
        if (e == hipErrorNotReady) return 1;
        (void)fail_hip("hipEventQuery", e);
        return -1;
    }

    template <class Start>
    int pump(hipStream_t stream, const std::function<int(size_t)> &landed, Start &&start_helpers)
    {
        uint32_t idle = 0, open = 0, sent = 0, freed = 0;        // chunks that may be copied, are on the bus or past it, (down) have been copied
        auto open_next = [&] {
            if (!to_host_) done_[open % kInFlight].store(0u, std::memory_order_relaxed);
            {
                std::lock_guard<std::mutex> lock(mu_);
                open_.store(chunk_end(open++), std::memory_order_release);
            }
            if (open == 1u) start_helpers();
            else more_.notify_all();
        };
        auto copied = [&](uint32_t c) { return done_[c % kInFlight].load(std::memory_order_acquire) == (chunk_end(c) - chunk_at(c) + kStagePart - 1u) / kStagePart; };
        while (to_host_ ? freed < chunks_ : sent < chunks_) {
            bool moved = false;
            if (to_host_) {
                for (; sent < chunks_ && sent < freed + ring_.slots; ++sent, moved = true) {
                    done_[sent % kInFlight].store(0u, std::memory_order_relaxed);
                    if (submit(sent, stream)) return 1;
                }
                // (everything the stream does before the first chunk: waited for, not polled)
                if (open == 0u) HCHECK(hipEventSynchronize(ring_.ev[0]));
                for (; open < sent; moved = true) {
                    const int busy = slot_busy(slot_of(open));
                    if (busy < 0) return 1;
                    if (busy) break;
                    open_next();
                }
                for (; freed < open && copied(freed); moved = true) ++freed;
            } else {
                // (a slot's last transfer may be one of the call before)
                for (; open < chunks_ && (open < 3u + ring_.slots || open < sent + ring_.slots); moved = true) {
                    const int busy = begins_slot(open) ? slot_busy(slot_of(open)) : 0;
                    if (busy < 0) return 1;
                    if (busy) break;
                    open_next();
                }
                for (; sent < open && copied(sent); moved = true) {
                    if (submit(sent, stream)) return 1;
                    ++sent;
                    if (landed) {
                        HCHECK(hipStreamWaitEvent(g_stream, ring_.ev[slot_of(sent - 1u)], 0));
                        if (landed(std::min(chunk_end(sent - 1u), seg_[0].bytes))) return 1;
                    }
                }
            }
            if (copy_one() || moved) {
                idle = 0;
                continue;
            }
            // Nothing to copy, to send or to hand out.  Where it is a chunk on the bus that is missing, and for long, the runtime waits for
            // it; else the helpers' copies are under way.
            if (++idle >= kIdleLooks && (to_host_ ? freed == open : sent == open)) HCHECK(hipEventSynchronize(ring_.ev[slot_of(open)]));
            else std::this_thread::yield();
        }
        return 0;
    }

    const Segment *seg_;
    uint32_t count_, chunks_ = 0;
    bool to_host_;
    StageRing &ring_;
    size_t total_ = 0;
    std::atomic<size_t> next_{0}, open_{0};        // bytes of the transfer that have been taken, that may be taken
    std::atomic<uint32_t> done_[kInFlight] = {};   // parts of a chunk that have been copied
    std::atomic<bool> stop_{false};
    std::mutex mu_;                                // open_ and stop_ change with it held, so that no helper sleeps through it
    std::condition_variable more_;
};

// a ring's buffers, with its lock held
int ring_ready(StageRing &r)
{
    if (r.ready) return 0;
    for (uint32_t i = 0; i < r.slots; ++i) {
        if (!r.buf[i]) HCHECK(hipHostMalloc(&r.buf[i], r.chunk, hipHostMallocDefault));
        if (!r.ev[i]) HCHECK(hipEventCreateWithFlags(&r.ev[i], hipEventDisableTiming));
    }
    if (&r == &g_up) {
        if (!r.start) HCHECK(hipEventCreateWithFlags(&r.start, hipEventDisableTiming));
        if (!r.side) HCHECK(hipStreamCreateWithFlags(&r.side, hipStreamNonBlocking));
    }
    r.ready = true;
    return 0;
}

// host memory that the copy engine reads as it is
bool host_registered(const void *src)
{
    hipPointerAttribute_t attr{};
    if (hipPointerGetAttributes(&attr, src) == hipSuccess && attr.type != hipMemoryTypeUnregistered) return true;
    (void)hipGetLastError();                                   // an unknown pointer leaves an error behind
    return false;
}

// Like hipMemcpyAsync from pageable memory, the call returns when all of src has been read; the transfers themselves are
// ordered on g_stream.
//
// With a `landed`, the transfers run on a stream of their own, and landed(upto) is called after each chunk: what it
// enqueues on g_stream may read the first upto bytes of dst and runs beside the transfers that follow.  The ways without a
// ring call it once.
int upload_from_host(void *dst, const void *src, size_t bytes, const std::function<int(size_t)> &landed = {})
{
    if (bytes < kStagedUp || host_registered(src)) {
        HCHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, g_stream));
        return landed ? landed(bytes) : 0;
    }
    std::lock_guard<std::mutex> lock(g_up.mu);
    if (ring_ready(g_up)) return 1;
    const hipStream_t stream = landed ? g_up.side : g_stream;
    if (landed) {
        HCHECK(hipEventRecord(g_up.start, g_stream));       // what is still reading dst
        HCHECK(hipStreamWaitEvent(stream, g_up.start, 0));
    }
    const Segment one{const_cast<char *>(static_cast<const char *>(src)), static_cast<char *>(dst), bytes};
    const int rc = StagedTransfer(&one, 1u, false).run(stream, landed);
    if (rc) (void)hipStreamSynchronize(stream);
    return rc;
}

// src to pageable host memory behind everything on g_stream; dst holds it when the call returns
int download_to_host(void *dst, const void *src, size_t bytes)
{
    if (bytes < kStagedDown || host_registered(dst)) {
        HCHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g_stream));
        HCHECK(hipStreamSynchronize(g_stream));
        return 0;
    }
    std::lock_guard<std::mutex> lock(g_down.mu);
    if (ring_ready(g_down)) return 1;
    const Segment one{static_cast<char *>(dst), const_cast<char *>(static_cast<const char *>(src)), bytes};
    const int rc = StagedTransfer(&one, 1u, true).run(g_stream, {});
    if (rc) (void)hipStreamSynchronize(g_stream);
    return rc;
}

// several arrays of whole floats at once, up (ordered on g_stream, the host arrays read when the call returns) or down
int move_arrays(const Segment *segments, uint32_t count, bool to_host)
{
    StageRing &ring = to_host ? g_down : g_up;
    std::lock_guard<std::mutex> lock(ring.mu);
    if (ring_ready(ring)) return 1;
    const int rc = StagedTransfer(segments, count, to_host).run(g_stream, {});
    if (rc) (void)hipStreamSynchronize(g_stream);
    return rc;
}

}  // namespace
