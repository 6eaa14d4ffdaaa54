// Cell data between host arrays and the device, in chunks through pinned memory.
//
// A copy between pageable host memory and the device runs at 9 (down) and 17 GB/s
// (up) here: the runtime stages it through its own pinned buffer and copies on one
// thread, which also takes the page faults of a fresh array. A chunk here is a
// run of cells whose kernel reads or writes a pinned slot directly over the bus
// (57 GB/s), and several host threads, each chunk with a slot and a stream, move the
// chunks between slots and the caller's arrays: the populations of 128^3 FP64
// cells (319 MB) come down in 7.4 ms instead of 34.8 and go up in 6.0 instead of
// 19.1, their density and velocity (67 MB) in 2.0 instead of 7.8. Only uploads of
// 0.75 to 72 MB take memory on the device (kCopiedUploadMin).
#ifndef PALABOS_AMD_HOSTIO_H
#define PALABOS_AMD_HOSTIO_H

#include <emmintrin.h>

#include <atomic>
#include <condition_variable>
#include <new>
#include <optional>
#include <thread>

#include "engine.h"

namespace plbamd {

// The slots and streams of one device: shared by its lattices, made by the first
// transfer, freed with the last lattice. A transfer takes a slot for each of its
// chunks, and who waits longest gets the next one: a small read does not wait for
// another lattice's gigabytes, but for one of their chunks.
struct HostSlots {
    static constexpr int kSlots = 8;
    static constexpr size_t kBytes = 4u << 20;
    int device = -1;
    char* pinned = nullptr;
    hipStream_t stream[kSlots] = {};
    ~HostSlots();
    char* slot(int k) { return pinned + (size_t)k * kBytes; }
    // a free slot for one chunk, in the order of asking
    struct Use {
        HostSlots& s;
        int k;
        explicit Use(HostSlots& slots) : s(slots) {
            std::unique_lock<std::mutex> lock(s.mutex);
            const uint64_t ticket = s.asked++;
            s.freed.wait(lock, [&] { return ticket == s.served && s.nFree > 0; });
            ++s.served;
            k = s.freeSlot[--s.nFree];
            if (s.served != s.asked && s.nFree > 0) s.freed.notify_all();
        }
        ~Use() {
            std::lock_guard<std::mutex> lock(s.mutex);
            s.freeSlot[s.nFree++] = k;
            if (s.served != s.asked) s.freed.notify_all();
        }
        Use(const Use&) = delete;
        Use& operator=(const Use&) = delete;
    };

private:
    std::mutex mutex;
    std::condition_variable freed;
    uint64_t asked = 0, served = 0;
    int freeSlot[kSlots] = {7, 6, 5, 4, 3, 2, 1, 0}, nFree = kSlots;
};
// Null when the pinned memory cannot be had.
std::shared_ptr<HostSlots> hostSlots(Lattice& L);

// Uploads between these sizes go in one pageable copy per array to device memory, and
// smaller ones in chunks on the calling thread: helper threads take the arrays' lines
// into other cores' caches, and a program that writes them anew pays for it (density and
// velocity rewritten, then uploaded, us: 8.4 MB copied 390, by eight threads 520-870; 16.8 MB
// 690, 1490-1670; 67 MB 4190, 4530-5300; from new arrays each time 2.1 MB 335, 530-800, 16.8
// MB 2000, 4930). Below, a chunk is the faster way (populations of 0.6 / 1.2 / 2.5 MB
// copied 51 / 87 / 151, in chunks 46 / 95 / 168). Above, the threads win (populations of 80 /
// 319 / 638 MB left as they are 3280 -> 1590, 11.3 -> 5.8 ms, 22.0 -> 11.5; rewritten in place
// 5300 -> 4800-6250, 19.8 -> 17-19 ms, 39 -> 33).
constexpr uint64_t kCopiedUploadMin = 768u << 10, kCopiedUploadMax = 72u << 20;

// One host array over a box, `perCell` bytes a cell in C order (host null: none).
struct HostPart {
    char* host;
    size_t perCell;
};

// A copy from another thread's array to a slot that the device reads, leaving neither
// in the caches of the core that makes it. (With memcpy the owner of the array, writing
// it anew, fetched its lines back from there: populations of 80 MB rewritten and uploaded
// 8.1-8.9 ms instead of 4.8-6.3.)
inline void copyPast(void* to, const void* from, size_t n) {
    char* d = static_cast<char*>(to);
    const char* s = static_cast<const char*>(from);
    for (; n >= 64; n -= 64, d += 64, s += 64) {
        _mm_prefetch(s + 1024, _MM_HINT_NTA);
        const __m128i a = _mm_loadu_si128((const __m128i*)s), b = _mm_loadu_si128((const __m128i*)(s + 16)),
                      c = _mm_loadu_si128((const __m128i*)(s + 32)), e = _mm_loadu_si128((const __m128i*)(s + 48));
        _mm_stream_si128((__m128i*)d, a);
        _mm_stream_si128((__m128i*)(d + 16), b);
        _mm_stream_si128((__m128i*)(d + 32), c);
        _mm_stream_si128((__m128i*)(d + 48), e);
    }
    _mm_sfence();
    std::memcpy(d, s, n);
}

inline void copyPlain(void* to, const void* from, size_t n) { std::memcpy(to, from, n); }

// Moves `parts` over box b: launch(chunk, staged, stream) queues the kernels that
// read (up) or write (down) the chunk's values at staged[part], C order over the
// chunk. The lattice's own stream must be idle. Returns when all is done.
template<typename Launch>
int hostTransfer(Lattice& L, const plbamd_box& b, const HostPart* parts, int nParts, bool up, Launch launch) {
    size_t perCell = 0;
    for (int p = 0; p < nParts; ++p) perCell += parts[p].host ? parts[p].perCell : 0;
    // runs of cells that are contiguous in the arrays: whole x planes, else rows of
    // one plane, else cells of one row
    const uint64_t ly = b.y1 - b.y0 + 1, lz = b.z1 - b.z0 + 1;
    const uint64_t lx = b.x1 - b.x0 + 1;
    const uint64_t total = boxCells(b) * perCell;
    if (up && total > kCopiedUploadMin && total < kCopiedUploadMax) {
        DeviceBuffers buf;
        void* dev[4] = {};
        auto padded = [&](int p) { return parts[p].host ? (boxCells(b) * parts[p].perCell + 15) / 16 * 16 : 0; };
        size_t bytes = 0;
        for (int p = 0; p < nParts; ++p) bytes += padded(p);
        // one allocation (each costs 30 us and more) and no larger than the arrays (64 MiB
        // and some bytes take 270 us longer than 64 MiB)
        if (char* at = static_cast<char*>(buf.get(bytes))) {
            for (int p = 0; p < nParts; ++p) {
                dev[p] = parts[p].host ? at : nullptr;
                at += padded(p);
            }
            hipError_t err = hipSuccess;
            for (int p = 0; p < nParts && err == hipSuccess; ++p)
                if (parts[p].host)
                    err = hipMemcpyAsync(dev[p], parts[p].host, boxCells(b) * parts[p].perCell, hipMemcpyHostToDevice, L.stream);
            if (err == hipSuccess) err = launch(b, dev, L.stream);
            const hipError_t end = hipStreamSynchronize(L.stream);   // before the buffers go, on every path
            if (err == hipSuccess) err = end;
            if (err != hipSuccess) return fail(PLBAMD_EHIP, std::string("transfer: ") + hipGetErrorString(err));
            ++L.pageableTransfers;
            return PLBAMD_OK;
        }
    }
    // chunks of an eighth of the whole, between 1 MB (a launch and its wait cost about
    // 10 us, a thread 20: 623 KB of populations up 79 us in chunks of 256 KB, 46 in one)
    // and a slot
    const size_t chunkBytes = std::min<uint64_t>(HostSlots::kBytes, std::max<uint64_t>(1u << 20, total / HostSlots::kSlots + 4096));
    const uint64_t fit = chunkBytes / perCell - 8;    // 8: the parts' alignment
    const uint64_t sx = std::min(lx, std::max<uint64_t>(1, fit / (ly * lz)));
    const uint64_t sy = ly * lz <= fit ? ly : std::min(ly, std::max<uint64_t>(1, fit / lz));
    const uint64_t sz = lz <= fit ? lz : fit;
    const uint64_t nX = (lx + sx - 1) / sx, nY = (ly + sy - 1) / sy, nZ = (lz + sz - 1) / sz;
    const uint64_t chunks = nX * nY * nZ;
    std::shared_ptr<HostSlots> slots = hostSlots(L);
    std::unique_ptr<char[]> pageable;   // without pinned memory: through ordinary memory and a device chunk
    DeviceBuffers buf;
    char* onDevice = nullptr;
    if (slots) {
        ++L.pinnedTransfers;
    } else {
        ++L.pageableTransfers;
        pageable.reset(new (std::nothrow) char[chunkBytes]);
        if (!pageable) return fail(PLBAMD_ENOMEM, "transfer: out of host memory");
        onDevice = static_cast<char*>(buf.get(chunkBytes));
        if (!onDevice) return fail(PLBAMD_ENOMEM, "transfer: cannot allocate a staging buffer");
    }
    const int want = !slots || (up && total <= kCopiedUploadMin) ? 1 : (int)std::min<uint64_t>(HostSlots::kSlots, chunks);
    std::atomic<uint64_t> next{0};
    std::atomic<int> error{(int)hipSuccess};
    auto work = [&]() {
        for (uint64_t c; error.load() == (int)hipSuccess && (c = next.fetch_add(1)) < chunks;) {
            std::optional<HostSlots::Use> use;
            if (slots) use.emplace(*slots);
            char* const slot = slots ? slots->slot(use->k) : pageable.get();
            hipStream_t stream = L.stream;
            if (slots) {
                // a slot's stream comes with its first use
                hipStream_t& own = slots->stream[use->k];
                const hipError_t made = own ? hipSuccess : hipStreamCreateWithFlags(&own, hipStreamNonBlocking);
                if (made != hipSuccess) { error.store((int)made); return; }
                stream = own;
            }
            const uint64_t ix = c / (nY * nZ), iy = c / nZ % nY, iz = c % nZ;
            plbamd_box k;
            k.x0 = b.x0 + (int)(ix * sx); k.x1 = std::min<int>(b.x1, k.x0 + (int)sx - 1);
            k.y0 = b.y0 + (int)(iy * sy); k.y1 = std::min<int>(b.y1, k.y0 + (int)sy - 1);
            k.z0 = b.z0 + (int)(iz * sz); k.z1 = std::min<int>(b.z1, k.z0 + (int)sz - 1);
            const uint64_t cells = boxCells(k);
            const uint64_t first = ((uint64_t)(k.x0 - b.x0) * ly + (uint64_t)(k.y0 - b.y0)) * lz + (uint64_t)(k.z0 - b.z0);
            void* staged[4] = {};
            size_t at = 0;
            for (int p = 0; p < nParts; ++p) {
                if (!parts[p].host) continue;
                staged[p] = slot + at;
                at = (at + cells * parts[p].perCell + 15) / 16 * 16;
                if (up) (want > 1 ? copyPast : copyPlain)(staged[p], parts[p].host + first * parts[p].perCell, cells * parts[p].perCell);
            }
            void* dev[4] = {};
            hipError_t err = hipSuccess;
            for (int p = 0; p < nParts; ++p) dev[p] = !staged[p] || !onDevice ? staged[p] : onDevice + ((char*)staged[p] - slot);
            if (onDevice && up) err = hipMemcpyAsync(onDevice, slot, at, hipMemcpyHostToDevice, stream);
            if (err == hipSuccess) err = launch(k, dev, stream);
            if (onDevice && !up && err == hipSuccess) err = hipMemcpyAsync(slot, onDevice, at, hipMemcpyDeviceToHost, stream);
            if (err == hipSuccess) err = hipStreamSynchronize(stream);
            if (err != hipSuccess) { error.store((int)err); return; }
            if (!up)
                for (int p = 0; p < nParts; ++p)
                    if (parts[p].host)
                        std::memcpy(parts[p].host + first * parts[p].perCell, staged[p], cells * parts[p].perCell);
        }
    };
    std::vector<std::thread> helpers;
    for (int k = 1; k < want; ++k) {
        try {
            helpers.emplace_back([&] {
                const hipError_t err = hipSetDevice(L.device);
                if (err == hipSuccess) work();
                else error.store((int)err);
            });
        } catch (...) {
            break;   // no more threads to be had: those there are do the work
        }
    }
    work();
    for (std::thread& t : helpers) t.join();
    if (error.load() != (int)hipSuccess)
        return fail(PLBAMD_EHIP, std::string("transfer: ") + hipGetErrorString((hipError_t)error.load()));
    return PLBAMD_OK;
}

}  // namespace plbamd

#endif
