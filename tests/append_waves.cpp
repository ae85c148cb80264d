// The block's append buffer (csrc/c3d_append.h) on the host: one thread per wave, a barrier that
// reports a wave that never arrives, and waves that are late after every barrier.  Prints "ok" if
// every pushed cell is listed exactly once, in its own list.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <thread>
#include <vector>

#define __device__
#define __forceinline__ inline
#define __shared__ static

constexpr int kWaves = 4;
static thread_local struct {
    unsigned x;
} threadIdx;
static struct {
    unsigned x;
} blockDim{kWaves};
static unsigned late;  // bit w: wave w is late after a barrier

static void __syncthreads()
{
    static std::mutex m;
    static std::condition_variable cv;
    static int arrived = 0, generation = 0;
    {
        std::unique_lock<std::mutex> lk(m);
        const int g = generation;
        if (++arrived == kWaves) {
            arrived = 0;
            ++generation;
            cv.notify_all();
        } else if (!cv.wait_for(lk, std::chrono::seconds(5), [&] { return g != generation; })) {
            std::puts("a wave waits at a barrier that the others do not reach");
            std::fflush(stdout);
            std::_Exit(2);
        }
    }
    if (late >> threadIdx.x & 1)
        std::this_thread::sleep_for(std::chrono::milliseconds(2));
}
static int atomicAdd(int *p, int v) { return __atomic_fetch_add(p, v, __ATOMIC_RELAXED); }

#include "c3d_append.h"

using namespace c3d;
static int buf[2 * kAggCap], cnt[2], base[2];

// rounds of perRound cells, the first `pushers` waves taking them in turn; every `every`th cell is
// of the mixed list
static int run(int perRound, int rounds, int pushers, int every)
{
    const int n = perRound * rounds;
    std::vector<int> wm(n + 2 * kAggCap, -1), wf(n + 2 * kAggCap, -1);
    int nm = 5, nf = 5;  // other blocks' cells come first
    base[0] = base[1] = 0;
    const Lists L{wm.data(), wf.data(), &nm, &nf};
    std::vector<std::thread> waves;
    for (int w = 0; w < kWaves; ++w)
        waves.emplace_back([&, w] {
            threadIdx.x = w;
            BlockAppender app{buf, cnt, base};
            app.init();
            for (int r = 0; r < rounds; ++r) {
                for (int i = 0; i < perRound; ++i)
                    if (i % pushers == w)
                        app.push((r * perRound + i) % every == 0, r * perRound + i);
                app.flush(L, r + 1 == rounds, perRound);
            }
        });
    for (auto &t : waves)
        t.join();
    std::vector<int> seen(n, 0);
    for (int i = 5; i < nm; ++i)
        if (wm[i] < 0 || wm[i] >= n || wm[i] % every != 0 || seen[wm[i]]++)
            return 1;
    for (int i = 5; i < nf; ++i)
        if (wf[i] < 0 || wf[i] >= n || wf[i] % every == 0 || seen[wf[i]]++)
            return 1;
    return nm + nf == n + 10 ? 0 : 1;
}

int main(int argc, char **argv)
{
    if (argc != 6)
        return 3;
    late = (unsigned)std::atoi(argv[5]);
    if (run(std::atoi(argv[1]), std::atoi(argv[2]), std::atoi(argv[3]), std::atoi(argv[4]))) {
        std::puts("lost, repeated or misplaced cells");
        return 1;
    }
    std::puts("ok");
}
