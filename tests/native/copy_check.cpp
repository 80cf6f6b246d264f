// Host check of the large downloads' control flow (host_copy.hpp) on a device
// that is a host buffer.  argv: scenario, bytes; prints
// "result bytes_equal pieces entered callers", the threads that entered the device
// and whether the caller's is one of them.
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <new>
#include <string>
#include <system_error>
#include <vector>
#include "../../spade_amd/csrc/host_copy.hpp"

static int threads_left = 1 << 30;
static bool refuse_with_bad_alloc = false;

// std::thread that is refused after threads_left of them
struct FewThreads
{
    std::thread t;
    FewThreads() = default;
    template <class F> explicit FewThreads(F f)
    {
        if (threads_left-- <= 0)
        {
            if (refuse_with_bad_alloc) throw std::bad_alloc();
            throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
        }
        t = std::thread(f);
    }
    bool joinable() const { return t.joinable(); }
    void join() { t.join(); }
};

struct Fake
{
    std::vector<char> dev;
    std::vector<std::vector<char>> mem{(size_t)spd::CopyShape::threads};
    std::atomic<int> pieces{0};
    long fail_at = -1;
    bool have_slots = true;
    bool slots() const { return have_slots; }
    std::mutex mu;
    std::vector<std::thread::id> entered;
    bool enter() { std::lock_guard<std::mutex> l(mu); entered.push_back(std::this_thread::get_id()); return true; }
    const char* slot(int t) const { return mem[t].data(); }
    bool fetch(int t, size_t off, size_t n)
    {
        if (n > spd::CopyShape::slot || pieces++ == fail_at) return false;
        mem[t].assign(dev.begin() + off, dev.begin() + off + n);
        return true;
    }
};

int main(int, char** argv)
{
    const std::string scenario = argv[1];
    const size_t bytes = std::strtoull(argv[2], nullptr, 10);
    Fake f;
    f.dev.resize(bytes);
    for (size_t n = 0; n < bytes; ++n) f.dev[n] = (char)(n*2654435761u >> 13);
    if (scenario == "no_thread") threads_left = 0;
    if (scenario == "one_thread") threads_left = 1;
    if (scenario == "no_memory") { threads_left = 1; refuse_with_bad_alloc = true; }
    if (scenario == "failing_piece") f.fail_at = 2;
    if (scenario == "no_slots") f.have_slots = false;
    std::vector<char> host(bytes);
    const spd::Copied r = spd::copy_in_pieces<FewThreads>(f, host.data(), bytes);
    const char* name = r == spd::Copied::all ? "all" : r == spd::Copied::failed ? "failed" : "no_slots";
    const bool callers = std::count(f.entered.begin(), f.entered.end(), std::this_thread::get_id()) > 0;
    std::printf("%s %d %d %zu %d\n", name, (int)(host == f.dev), (int)f.pieces, f.entered.size(), (int)callers);
    return 0;
}
