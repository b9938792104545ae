#include "hostcopy.h"

#include <string.h>
#include <unistd.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>

namespace ncnn {

namespace {

// one core copies at about 24 GB/s, PCIe takes 56: four keep ahead of it with room for slow cores
const int HELPERS = 3;
const size_t PIECE = 256 * 1024;
// a helper that has finished looks for the next chunk of the same upload for this many turns (about 100 us) before it sleeps
const int SPINS = 2000;

// Never destroyed: a child of fork() has the object but none of its threads, and there the destructor of the condition
// variable would wait for sleepers that do not exist; and another thread may still be copying when the process exits.
class CopyPool
{
public:
    CopyPool() : count(0), owner(getpid()), generation(0), stop(false), open(false), next(0), active(0), dst(0), src(0), bytes(0)
    {
        if (std::thread::hardware_concurrency() <= (unsigned)HELPERS) return;
        try
        {
            while (count < HELPERS)
            {
                threads[count] = std::thread(&CopyPool::help, this);
                count++;
            }
        }
        catch (const std::system_error&) // the process may have no more threads: with those there are, or with none
        {
        }
    }
    // The end of the process, or of the library in it: ends the helpers.  Whoever copies afterwards copies alone (user stays
    // locked), and so does whoever copies just now: the helpers then sleep on until the process is gone.
    void retire()
    {
        if (getpid() != owner || !user.try_lock()) return;
        {
            std::lock_guard<std::mutex> g(lock);
            stop = true;
            generation.fetch_add(1);
        }
        wake.notify_all();
        for (int i = 0; i < count; i++) threads[i].join();
    }

    bool copy(void* _dst, const void* _src, size_t _bytes)
    {
        if (!count || getpid() != owner || !user.try_lock()) return false;
        {
            std::lock_guard<std::mutex> g(lock);
            dst = (unsigned char*)_dst;
            src = (const unsigned char*)_src;
            bytes = _bytes;
            next.store(0);
            open = true;
            generation.fetch_add(1);
        }
        wake.notify_all();
        work();
        {
            std::lock_guard<std::mutex> g(lock);
            open = false; // a helper that wakes up only now has nothing to do here
        }
        while (active.load(std::memory_order_acquire) != 0) __builtin_ia32_pause();
        user.unlock();
        return true;
    }

private:
    void work()
    {
        for (;;)
        {
            const size_t at = next.fetch_add(PIECE);
            if (at >= bytes) return;
            memcpy(dst + at, src + at, bytes - at < PIECE ? bytes - at : PIECE);
        }
    }
    void help()
    {
        unsigned long long seen = 0;
        for (;;)
        {
            for (int i = 0; i < SPINS && generation.load(std::memory_order_acquire) == seen; i++) __builtin_ia32_pause();
            bool join;
            {
                std::unique_lock<std::mutex> g(lock);
                while (generation.load() == seen) wake.wait(g);
                seen = generation.load();
                if (stop) return;
                join = open;
                if (join) active.fetch_add(1);
            }
            if (!join) continue;
            work();
            active.fetch_sub(1, std::memory_order_release);
        }
    }

    std::thread threads[HELPERS];
    int count;
    const pid_t owner;
    std::mutex user; // one copy at a time
    std::mutex lock;
    std::condition_variable wake;
    std::atomic<unsigned long long> generation;
    bool stop;
    bool open; // the current job still takes helpers
    std::atomic<size_t> next;
    std::atomic<int> active; // helpers inside the current job
    unsigned char* dst;
    const unsigned char* src;
    size_t bytes;
};

} // namespace

void parallel_copy(void* dst, const void* src, size_t bytes)
{
    // below 1 MB (40 us) one thread is done before the others are awake
    if (bytes >= 4 * PIECE)
    {
        static CopyPool* const pool = new (std::nothrow) CopyPool;
        static const struct AtExit
        {
            ~AtExit()
            {
                if (pool) pool->retire();
            }
        } at_exit;
        (void)at_exit;
        if (pool && pool->copy(dst, src, bytes)) return;
    }
    memcpy(dst, src, bytes);
}

} // namespace ncnn
