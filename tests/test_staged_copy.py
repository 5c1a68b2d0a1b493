"""The staged device-to-host copy (staged_copy.h) against a stand-in HIP runtime whose copies run later, on a thread of
their own, and whose calls can be made to fail."""
import os
import subprocess

import pytest

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "clode_amd", "csrc", "runtime",
                      "staged_copy.h")

FAKE_HIP = r"""
#pragma once
#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <thread>
enum hipError_t { hipSuccess = 0, hipErrorUnknown = 999 };
enum { hipMemcpyDeviceToHost, hipHostMallocPortable, hipEventDisableTiming };
struct Queue {
    std::mutex mu;
    std::condition_variable cv;
    std::deque<std::function<void()>> q;
    size_t done = 0, queued = 0;
    bool stop = false;
    std::thread t{[this] {
        for (;;) {
            std::function<void()> f;
            {
                std::unique_lock<std::mutex> lk(mu);
                cv.wait(lk, [this] { return stop || !q.empty(); });
                if (q.empty())
                    return;
                f = q.front();
                q.pop_front();
            }
            std::this_thread::sleep_for(std::chrono::milliseconds(1));
            f();
            std::lock_guard<std::mutex> lk(mu);
            ++done;
            cv.notify_all();
        }
    }};
    size_t put(std::function<void()> f)
    {
        std::lock_guard<std::mutex> lk(mu);
        q.push_back(f);
        cv.notify_all();
        return ++queued;
    }
    void wait(size_t k)
    {
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [&] { return done >= k; });
    }
    ~Queue()
    {
        {
            std::lock_guard<std::mutex> lk(mu);
            stop = true;
            cv.notify_all();
        }
        t.join();
    }
};
typedef Queue *hipStream_t;
struct Event { Queue *q = nullptr; size_t k = 0; };
typedef Event *hipEvent_t;
inline int records_left = -1;  // calls of hipEventRecord until one fails
inline std::mutex records_mu;
inline bool no_pinned = false;
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, int)
{
    *p = no_pinned ? nullptr : std::malloc(n);
    return *p ? hipSuccess : hipErrorUnknown;
}
inline hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, int, hipStream_t q)
{
    q->put([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t q) { q->wait(q->queued); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, int) { *e = new Event; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t q)
{
    {
        std::lock_guard<std::mutex> lk(records_mu);
        if (records_left == 0)
            return hipErrorUnknown;
        if (records_left > 0)
            --records_left;
    }
    e->k = q->put([] {});
    e->q = q;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) { e->q->wait(e->k); return hipSuccess; }
"""

MAIN = r"""
#include "%s"
#include <cstdio>
int main(int argc, char **argv)
{
    const size_t bytes = std::strtoull(argv[1], nullptr, 10);
    records_left = std::atoi(argv[2]);
    no_pinned = std::atoi(argv[3]) != 0;
    std::vector<char> src(bytes), dst(bytes, 1);
    for (size_t i = 0; i < bytes; ++i)
        src[i] = (char)(i * 2654435761u >> 13);
    Queue q;
    const hipError_t e = clode::StagedCopy::get()->toHost(0, dst.data(), src.data(), bytes, &q);
    size_t waiting;
    {
        std::lock_guard<std::mutex> lk(q.mu);
        waiting = q.queued - q.done;
    }
    std::printf("%%d %%d %%zu\n", (int)e, (int)(src == dst), waiting);
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("staged")
    (d / "hip").mkdir()
    (d / "hip" / "hip_runtime.h").write_text(FAKE_HIP)
    (d / "main.cpp").write_text(MAIN % HEADER)
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", str(d), str(d / "main.cpp"), "-o", str(d / "main")],
                   check=True)
    return str(d / "main")


def _run(program, bytes, records=-1, no_pinned=0):
    out = subprocess.run([program, str(bytes), str(records), str(no_pinned)], capture_output=True, text=True,
                         check=True, timeout=60).stdout
    return [int(v) for v in out.split()]


@pytest.mark.parametrize("bytes", [1, (8 << 20) - 1, 8 << 20, (8 << 20) + 1, (31 << 20) + 12345])
@pytest.mark.parametrize("no_pinned", [0, 1])
def test_copies_every_byte(program, bytes, no_pinned):
    assert _run(program, bytes, no_pinned=no_pinned) == [0, 1, 0]


@pytest.mark.parametrize("records", [0, 3, 9])
def test_nothing_is_in_flight_after_an_error(program, records):
    """A failing call is reported, and no copy into the shared blocks is still queued when it is."""
    error, same, waiting = _run(program, 31 << 20, records=records)
    assert error != 0 and not same and waiting == 0
