// A large copy from device to pageable host memory by several host threads.
// No HIP types here: Api supplies the device side, so that the control flow
// (refused pinned memory, refused threads, a failing piece) runs on the host.
#pragma once
#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <thread>

namespace spd {

// Threads of a large download, each with a pinned slot, and the bytes of a slot
struct CopyShape
{
    static constexpr int threads = 4;
    static constexpr size_t slot = 4u << 20;
};

enum class Copied { all, failed, no_slots };

// Copies `bytes` to host: thread t of CopyShape::threads (0 is the caller's)
// moves every threads-th piece, Api::fetch(t, off, n) bringing the n bytes from
// offset off into slot(t).  The DMA engine runs at its pinned rate (55 GB/s)
// while the other threads copy from their slots to the caller's memory, which
// one pageable hipMemcpyAsync does in turn (17 GB/s).  Two pieces a thread where that
// makes them 1 to 4 MiB: every piece costs some 30 us of calls (20.5 MB in
// 512 KiB pieces 1030 us, in 2 MiB ones 650).  The pieces of a thread that cannot
// be had are copied here, in turn.
// failed: a fetch did (Api keeps the reason).  no_slots: Api::slots() has none to
// offer, nothing was copied and the caller takes another way.  Api::enter() sets up
// a helper thread (its device) and is not called in the caller's.
template <class Thread = std::thread, class Api>
Copied copy_in_pieces(Api& api, char* host, size_t bytes)
{
    if (!api.slots()) return Copied::no_slots;
    constexpr int T = CopyShape::threads;
    const size_t piece = std::min(CopyShape::slot, std::max<size_t>(1u << 20, ((bytes/(2*T) + 65535) >> 16) << 16));
    std::atomic<bool> failed{false};
    const std::thread::id caller = std::this_thread::get_id();
    auto work = [&](int t) noexcept
    {
        if (std::this_thread::get_id() != caller && !api.enter()) { failed = true; return; }
        for (size_t off = t*piece; off < bytes && !failed; off += T*piece)
        {
            const size_t n = std::min(piece, bytes - off);
            if (!api.fetch(t, off, n)) { failed = true; return; }
            std::memcpy(host + off, api.slot(t), n);
        }
    };
    Thread helper[T - 1];
    for (int t = 1; t < T; ++t)
    {
        // whatever refuses a thread (resources, memory), the ones that run must be joined
        try { helper[t - 1] = Thread([&, t] { work(t); }); }
        catch (...) { work(t); }
    }
    work(0);
    for (auto& h : helper) if (h.joinable()) h.join();
    return failed ? Copied::failed : Copied::all;
}

} // namespace spd
