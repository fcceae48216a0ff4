// Copies between device memory and the host's own (pageable) arrays through pinned buffers.
//
// The runtime's copies to pageable memory reach 17 GB/s down and 28 GB/s up, of the link's 57: one
// thread moves the data between the runtime's pinned buffers and the caller's pages.  Here up to
// HC_THREADS host threads take turns at pieces of HC_PIECE bytes, each with two pinned buffers, so
// that a thread's memcpy of one piece runs beside the link's copy of its next.  Reading 1.96 GB of
// state and history in 16 blocks took 111 ms through the runtime, now 52 ms; pieces of 0.5, 1, 4
// and 8 MB 96, 66, 48 and 46 ms, eight threads the same.  Setting a 78 MB state 2.7 ms, now 2.2 ms.
#pragma once
#include <algorithm>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

constexpr size_t HC_PIECE = (size_t)2 << 20;
constexpr int HC_THREADS = 4;
constexpr size_t HC_MIN = (size_t)128 << 10;  // below, the runtime's own copies

// A pinned buffer and the event of its last copy, both of device `dev`.
struct PinBuf {
    char* p = nullptr;
    hipEvent_t ev = nullptr;
    int dev = 0;
};

// The process's pinned buffers: at most HC_POOL are kept, shared by all contexts and threads,
// each taken by one transfer at a time; the last context to go gives them back.
constexpr int HC_POOL = 32;
struct PinPool {
    std::mutex m;
    std::vector<PinBuf> idle;
    int users = 0;

    static void drop(const PinBuf& b)
    {
        if (b.ev) (void)hipEventDestroy(b.ev);
        if (b.p) (void)hipHostFree(b.p);
    }
    void attach()
    {
        std::lock_guard<std::mutex> g(m);
        users++;
    }
    void detach()
    {
        std::lock_guard<std::mutex> g(m);
        if (--users > 0) return;
        for (const PinBuf& b : idle) drop(b);
        idle.clear();
    }
    // A buffer for device dev; false when there is no more pinned memory.
    bool take(int dev, PinBuf& out)
    {
        {
            std::lock_guard<std::mutex> g(m);
            for (size_t q = 0; q < idle.size(); q++)
                if (idle[q].dev == dev) {
                    out = idle[q];
                    idle.erase(idle.begin() + (long)q);
                    return true;
                }
        }
        out = PinBuf{};
        out.dev = dev;
        if (hipHostMalloc((void**)&out.p, HC_PIECE, hipHostMallocDefault) != hipSuccess) out.p = nullptr;
        if (out.p && hipEventCreateWithFlags(&out.ev, hipEventDisableTiming) != hipSuccess) out.ev = nullptr;
        if (out.p && out.ev) return true;
        drop(out);
        (void)hipGetLastError();
        return false;
    }
    void give(const PinBuf& b)
    {
        {
            std::lock_guard<std::mutex> g(m);
            if (users > 0 && (int)idle.size() < HC_POOL) {
                try {
                    idle.push_back(b);
                    return;
                } catch (const std::bad_alloc&) {  // not kept
                }
            }
        }
        drop(b);
    }
};
static PinPool g_pins;

// One contiguous copy.
struct HostCopy {
    char* host;
    char* dev;
    size_t bytes;
};

// `bytes` bytes of device memory from byte `off` of copy `q` on; they may run on into the copies
// that follow, where those lie behind each other on the device.
struct HostPiece {
    size_t q, off, bytes;
};

// fn(host address, bytes, offset in the piece) for the parts of a piece
template <typename F>
static void piece_parts(const std::vector<HostCopy>& list, const HostPiece& p, F fn)
{
    size_t q = p.q, off = p.off;
    for (size_t o = 0; o < p.bytes; q++, off = 0) {
        const size_t n = std::min(list[q].bytes - off, p.bytes - o);
        fn(list[q].host + off, n, o);
        o += n;
    }
}

static std::vector<HostPiece> host_pieces(const std::vector<HostCopy>& list)
{
    std::vector<HostPiece> out;
    const char* end = nullptr;  // of the last piece on the device
    for (size_t q = 0; q < list.size(); q++)
        for (size_t o = 0; o < list[q].bytes;) {
            size_t n = list[q].bytes - o;
            if (!out.empty() && list[q].dev + o == end && out.back().bytes < HC_PIECE) {
                n = std::min(n, HC_PIECE - out.back().bytes);
                out.back().bytes += n;
            } else {
                n = std::min(n, HC_PIECE);
                out.push_back(HostPiece{q, o, n});
            }
            o += n;
            end = list[q].dev + o;
        }
    return out;
}

// The pieces t, t + nt, ... of a transfer by one thread.
static hipError_t host_copy_pieces(const std::vector<HostCopy>& list, const std::vector<HostPiece>& pieces, int t,
                                   int nt, bool upload, int dev, hipStream_t stream, PinBuf buf[2])
{
    hipError_t e = hipSetDevice(dev);
    if (e != hipSuccess) return e;
    const HostPiece* in[2] = {nullptr, nullptr};  // the piece on its way through a buffer
    auto drain = [&](int s) -> hipError_t {
        if (!in[s]) return hipSuccess;
        const HostPiece& p = *in[s];
        in[s] = nullptr;
        const hipError_t r = hipEventSynchronize(buf[s].ev);
        if (r == hipSuccess && !upload)
            piece_parts(list, p, [&](char* h, size_t n, size_t o) { std::memcpy(h, buf[s].p + o, n); });
        return r;
    };
    int turn = 0;
    for (size_t q = (size_t)t; q < pieces.size(); q += (size_t)nt, turn ^= 1) {
        const HostPiece& p = pieces[q];
        char* const d = list[p.q].dev + p.off;
        if ((e = drain(turn)) != hipSuccess) break;
        if (upload) piece_parts(list, p, [&](char* h, size_t n, size_t o) { std::memcpy(buf[turn].p + o, h, n); });
        e = upload ? hipMemcpyAsync(d, buf[turn].p, p.bytes, hipMemcpyHostToDevice, stream)
                   : hipMemcpyAsync(buf[turn].p, d, p.bytes, hipMemcpyDeviceToHost, stream);
        if (e != hipSuccess || (e = hipEventRecord(buf[turn].ev, stream)) != hipSuccess) {
            (void)hipStreamSynchronize(stream);  // nothing may use the buffer when it is given back
            break;
        }
        in[turn] = &p;
    }
    for (int s = 0; s < 2; s++) {
        const hipError_t r = drain(turn ^ s);
        if (e == hipSuccess) e = r;
    }
    return e;
}

// The copies, after the stream's work so far.  Downloads are complete on return, uploads are queued
// on the stream and no longer read the host's memory.  (May throw std::bad_alloc, with no
// buffer kept and no thread running.)
static hipError_t host_copies(const std::vector<HostCopy>& list, bool upload, hipStream_t stream)
{
    size_t total = 0;
    for (const HostCopy& c : list) total += c.bytes;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    std::vector<HostPiece> pieces;
    std::vector<PinBuf> bufs;
    if (total >= HC_MIN) {
        pieces = host_pieces(list);
        const int want = 2 * (int)std::min<size_t>(HC_THREADS, pieces.size());
        bufs.reserve((size_t)want);
        PinBuf b;
        while ((int)bufs.size() < want && g_pins.take(dev, b)) bufs.push_back(b);
    }
    const int nt = (int)bufs.size() / 2;
    std::vector<std::thread> th;
    std::vector<hipError_t> er;
    try {
        th.reserve((size_t)nt);
        er.resize((size_t)nt, hipSuccess);
    } catch (const std::bad_alloc&) {
        for (const PinBuf& b : bufs) g_pins.give(b);
        throw;
    }
    if (nt == 0) {
        for (const HostCopy& c : list) {
            e = upload ? hipMemcpyAsync(c.dev, c.host, c.bytes, hipMemcpyHostToDevice, stream)
                       : hipMemcpyAsync(c.host, c.dev, c.bytes, hipMemcpyDeviceToHost, stream);
            if (e != hipSuccess) break;
        }
        const hipError_t r = hipStreamSynchronize(stream);
        if (e == hipSuccess) e = r;
    } else {
        int started = 1;
        try {
            for (; started < nt; started++)
                th.emplace_back([&, t = started] {
                    er[(size_t)t] = host_copy_pieces(list, pieces, t, nt, upload, dev, stream, &bufs[2 * (size_t)t]);
                });
        } catch (const std::exception&) {  // no more threads, or no memory for one: the caller does their pieces
        }
        er[0] = host_copy_pieces(list, pieces, 0, nt, upload, dev, stream, &bufs[0]);
        for (int t = started; t < nt; t++)
            er[(size_t)t] = host_copy_pieces(list, pieces, t, nt, upload, dev, stream, &bufs[2 * (size_t)t]);
        for (std::thread& t : th) t.join();
        for (hipError_t r : er)
            if (e == hipSuccess) e = r;
    }
    for (const PinBuf& b : bufs) g_pins.give(b);
    return e;
}
