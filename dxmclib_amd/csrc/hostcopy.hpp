// Host-side copies of the staged transfers, free of HIP so that they build
// and are tested on any host.
//
// CopyHelpers: persistent helper threads that copy parts of one block while
// the calling thread copies the first part. One core copies 27-30 GB/s out of
// page-locked memory on the MI355X host, four 80-100 GB/s, while the
// device-to-host DMA of a staging chunk runs at 53-57 GB/s; but result arrays
// are mostly fresh memory, whose pages are cleared at the first touch, and
// four threads then keep up with 31 GB/s, eight with 44. A chunk that holds
// several arrays is one copy: a wake-up of the helpers for each cost more than
// they saved (three arrays of 1.3 MiB in all down 0.108 ms, 0.085 as one copy;
// 2.5 MiB 0.149 and 0.120). Copies from 512 KiB on go to the helpers (an array
// of 1.6 MiB down 0.073 ms, from 2 MiB on 0.100). A context starts
// its helpers with its staging chunks and stops them with them; its lock
// keeps one copy at a time. When the threads cannot start, every copy runs
// on the calling thread.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <thread>

namespace dxmc_backend {

class CopyHelpers {
public:
    static constexpr int PARTS = 8;
    // copies below this are made by the calling thread alone
    static constexpr std::size_t PART_MIN = std::size_t { 1 } << 19;

    CopyHelpers() = default;
    CopyHelpers(const CopyHelpers&) = delete;
    CopyHelpers& operator=(const CopyHelpers&) = delete;
    ~CopyHelpers() { stop(); }

    // starts the helper threads; false (and no helpers) if one cannot start
    bool start()
    {
        if (m_running)
            return true;
        m_quit = false;
        for (int k = 1; k < PARTS; ++k) {
            try {
                m_threads[k - 1] = std::thread([this, k] { work(k); });
            } catch (...) {
                stop();
                return false;
            }
        }
        m_running = true;
        return true;
    }

    void stop()
    {
        {
            std::lock_guard lock(m_mutex);
            m_quit = true;
        }
        m_wake.notify_all();
        for (auto& t : m_threads)
            if (t.joinable())
                t.join();
        m_running = false;
    }

    bool running() const { return m_running; }

    // one of the blocks of a copy: dst[0, len) = src[0, len)
    struct Block {
        char* dst;
        const char* src;
        std::size_t len;
    };

    // copies the blocks; with the helpers running and PART_MIN bytes or more
    // in all, in PARTS parts of their joined bytes on PARTS threads (one
    // wake-up a copy, also where it ends one array and starts the next)
    void copy(const Block* list, int count)
    {
        std::size_t total = 0;
        for (int i = 0; i < count; ++i)
            total += list[i].len;
        if (!m_running || total < PART_MIN) {
            for (int i = 0; i < count; ++i)
                if (list[i].len)
                    std::memcpy(list[i].dst, list[i].src, list[i].len);
            return;
        }
        {
            std::lock_guard lock(m_mutex);
            m_list = list;
            m_count = count;
            m_per = (total + PARTS - 1) / PARTS;
            m_pending = PARTS - 1;
            ++m_generation;
        }
        m_wake.notify_all();
        part(0);
        std::unique_lock lock(m_mutex);
        m_finished.wait(lock, [this] { return m_pending == 0; });
    }
    void copy(void* dst, const void* src, std::size_t len)
    {
        const Block b { static_cast<char*>(dst), static_cast<const char*>(src), len };
        copy(&b, 1);
    }

private:
    // bytes [k * m_per, (k + 1) * m_per) of the joined blocks
    void part(int k) const
    {
        std::size_t skip = k * m_per, left = m_per;
        for (int i = 0; i < m_count && left; ++i) {
            const Block& x = m_list[i];
            const std::size_t from = std::min(skip, x.len), len = std::min(left, x.len - from);
            if (len)
                std::memcpy(x.dst + from, x.src + from, len);
            skip -= from;
            left -= len;
        }
    }

    void work(int k)
    {
        unsigned seen = 0;
        for (;;) {
            {
                std::unique_lock lock(m_mutex);
                m_wake.wait(lock, [&] { return m_quit || m_generation != seen; });
                if (m_quit)
                    return;
                seen = m_generation;
            }
            part(k);
            bool last = false;
            {
                std::lock_guard lock(m_mutex);
                last = --m_pending == 0;
            }
            if (last)
                m_finished.notify_one();
        }
    }

    std::thread m_threads[PARTS - 1];
    bool m_running = false;
    std::mutex m_mutex;
    std::condition_variable m_wake, m_finished;
    bool m_quit = false;
    unsigned m_generation = 0;
    int m_pending = 0;
    const Block* m_list = nullptr;
    int m_count = 0;
    std::size_t m_per = 0;
};

}
