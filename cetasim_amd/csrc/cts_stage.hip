// cts_stage.hip -- the particle state on its way to the host.
//
// A copy into pageable memory is bound by the host: the runtime moves one
// array after the other, and the pages of a result array that is new to the
// process are faulted in one by one under it (480 000 macroparticles, 25 MB:
// 1.3 ms into pages that exist, 5.6 ms into new ones).  Here a kernel writes
// stretches of 65 536 macroparticles of all arrays into a small ring of pinned
// memory over the bus, loss codes widened on the way, and a few threads copy
// the stretches that have arrived to their arrays and take the page faults
// side by side: 1.4 ms into new pages (with stretches of 32 768 2.0, of 8192
// 3.3: threads wait for each other at the end of each); 20 000 macroparticles
// 0.5 -> 0.07 ms, where the seven calls counted.  The ring (6.8 MB at most)
// belongs to the handle and goes with it; the threads live as long as the call.
#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "cts_internal.hpp"

namespace cts {

// rows [i0, i0 + n) of every wanted array to out[q][rows] (loss codes as
// int32 after the six coordinates)
__global__ void __launch_bounds__(kBlock) k_stage(StageParams P)
{
    const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (k >= P.n) return;
    const int64_t i = P.i0 + k;
    double v[6];
#pragma unroll
    for (int q = 0; q < 6; q++) v[q] = ((P.want >> q) & 1u) ? P.src[q][i] : 0.0;
    const int32_t f = ((P.want >> 6) & 1u) ? P.flag[i] & 3 : 0;
#pragma unroll
    for (int q = 0; q < 6; q++)
        if ((P.want >> q) & 1u) P.out[(int64_t)q * P.rows + k] = v[q];
    if ((P.want >> 6) & 1u) reinterpret_cast<int32_t *>(P.out + 6 * P.rows)[k] = f;
}

void stage_free(Stage &S)
{
    for (hipEvent_t &e : S.ev)
        if (e) (void)hipEventDestroy(e);
    if (S.host) (void)hipHostFree(S.host);
    S = Stage{};
}

// room for n rows, or as many as a ring of kStageSlots stretches holds
// (made by the first call: a program that reads nothing back pays nothing);
// false: no pinned memory to be had, the caller copies directly
static bool stage_room(Stage &S, int64_t n)
{
    const int64_t rows = std::min((n + kBlock - 1) / kBlock * kBlock, kStageRows);
    const int slots = (int)std::min<int64_t>(kStageSlots, (n + rows - 1) / rows);
    if (S.host && S.rows >= rows && S.slots >= slots) return true;
    stage_free(S);
    const size_t slot = (size_t)rows * (6 * sizeof(double) + sizeof(int32_t));
    if (hipHostMalloc(&S.host, slot * slots, hipHostMallocDefault) != hipSuccess ||
        hipHostGetDevicePointer(&S.dev, S.host, 0) != hipSuccess) {
        (void)hipGetLastError();
        stage_free(S);
        return false;
    }
    for (int s = 0; s < slots; s++)
        if (hipEventCreateWithFlags(&S.ev[s], hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            stage_free(S);
            return false;
        }
    S.rows = rows;
    S.slots = slots;
    return true;
}

namespace {

struct Job {
    char *dst[7];
    const char *ring;
    int64_t n, rows;
    int slots, narr, arr[7];
    std::mutex m;
    std::condition_variable cv;
    int64_t ready = 0, next = 0;  // pieces (an array's part of a stretch) arrived, taken
    int left[kStageSlots] = {};   // pieces of a slot's stretch not yet copied
    bool stop = false;

    void copy(int64_t p)
    {
        const int64_t r = p / narr, i0 = r * rows, len = std::min(rows, n - i0);
        const int q = arr[p % narr];
        const size_t w = q < 6 ? sizeof(double) : sizeof(int32_t);
        const char *slot = ring + (size_t)(r % slots) * rows * (6 * sizeof(double) + sizeof(int32_t));
        std::memcpy(dst[q] + i0 * w, slot + (size_t)q * rows * sizeof(double), len * w);
    }
    // copy pieces that have arrived; wait: for more of them, until stop
    void work(bool wait)
    {
        std::unique_lock<std::mutex> l(m);
        for (;;) {
            if (wait) cv.wait(l, [&] { return next < ready || stop; });
            if (next >= ready) return;
            const int64_t p = next++;
            l.unlock();
            copy(p);
            l.lock();
            if (--left[p / narr % slots] == 0) cv.notify_all();
        }
    }
};

}  // namespace

hipError_t stage_download(Stage &S, StageParams P, int64_t n, double *const coord[6], int32_t *lost, hipStream_t st,
                          bool &done)
{
    done = false;
    Job J;
    J.narr = 0;
    P.want = 0;
    size_t width = 0;
    for (int q = 0; q < 7; q++) {
        J.dst[q] = q < 6 ? reinterpret_cast<char *>(coord[q]) : reinterpret_cast<char *>(lost);
        if (!J.dst[q]) continue;
        P.want |= 1u << q;
        J.arr[J.narr++] = q;
        width += q < 6 ? sizeof(double) : sizeof(int32_t);
    }
    // Nothing to copy (the caller waits for the stream), and one or two arrays
    // of more macroparticles than the ring holds at once: a stretch then has too
    // few pieces for the threads, and direct copies are faster.  Direct / ring in
    // us, into pages that exist: one array of 2e5 98 / 134, of 2e6 967 / 2004;
    // two of 2e5 195 / 180, of 5e5 485 / 592; three of 2e6 2859 / 2099; loss
    // codes alone of 2e5 32 / 74, of 2e6 247 / 1575.  (Below, the runtime's copy
    // takes 30 us of 6e4 values, but 200 where copies are rare; the ring 33.)
    const int64_t whole = kStageSlots * kStageRows;
    if (n == 0 || J.narr == 0 || (J.narr == 1 && n > whole) || (J.narr == 2 && n > 2 * whole)) return hipSuccess;
    if (!stage_room(S, n)) return hipSuccess;
    J.n = n;
    J.rows = S.rows;
    J.slots = S.slots;
    J.ring = static_cast<const char *>(S.host);
    done = true;
    const int64_t rounds = (n + S.rows - 1) / S.rows;
    const auto launch = [&](int64_t r) -> hipError_t {
        P.i0 = r * S.rows;
        P.n = std::min(S.rows, n - P.i0);
        P.rows = S.rows;
        P.out = reinterpret_cast<double *>(static_cast<char *>(S.dev) +
                                           (size_t)(r % S.slots) * S.rows * (6 * sizeof(double) + sizeof(int32_t)));
        hipLaunchKernelGGL(k_stage, dim3((unsigned)((P.n + kBlock - 1) / kBlock)), dim3(kBlock), 0, st, P);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipEventRecord(S.ev[r % S.slots], st);
        return e;
    };
    hipError_t err = hipSuccess;
    for (int64_t r = 0; r < std::min<int64_t>(S.slots, rounds) && err == hipSuccess; r++) err = launch(r);
    // a thread per megabyte: starting one costs about what it copies of that
    std::vector<std::thread> crew;
    const int extra = (int)std::min<size_t>(kStageThreads - 1, width * n >> 20);
    try {
        crew.reserve(extra);
        for (int t = 0; t < extra && err == hipSuccess; t++) crew.emplace_back([&J] { J.work(true); });
    } catch (const std::exception &) {
        // fewer threads: this one copies what they leave
    }
    for (int64_t r = 0; r < rounds && err == hipSuccess; r++) {
        const int slot = (int)(r % S.slots);
        if ((err = hipEventSynchronize(S.ev[slot])) != hipSuccess) break;
        {
            std::lock_guard<std::mutex> l(J.m);
            J.left[slot] = J.narr;
            J.ready = (r + 1) * J.narr;
        }
        J.cv.notify_all();
        J.work(false);
        // the slot's next stretch, or the end: its pieces are copied
        if (r + S.slots < rounds) {
            {
                std::unique_lock<std::mutex> l(J.m);
                J.cv.wait(l, [&] { return J.left[slot] == 0; });
            }
            err = launch(r + S.slots);
        }
    }
    {
        std::lock_guard<std::mutex> l(J.m);
        J.stop = true;
    }
    J.cv.notify_all();
    for (std::thread &t : crew) t.join();
    if (err != hipSuccess) (void)hipStreamSynchronize(st);
    return err;
}

}  // namespace cts
