// WarpSpecSession on the emulated runtime: its queue, and whom a destroyed
// session leaves it to.  One scenario per run, named on the command line;
// "pass" and status 0, or what went wrong and status 3.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <future>
#include <memory>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "emu.h"
#include "gfd/hip_shim.h"
#include "gfd/warp_spec_session.h"

// Host memory runs out while this is set.
static bool g_no_memory = false;
void* operator new(size_t n) {
    void* p = g_no_memory ? nullptr : std::malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

namespace {

using gfd::WarpSpecConfig;
using gfd::WarpSpecSession;

std::vector<char> g_src(1 << 16), g_dst(1 << 16);

WarpSpecConfig config(uint32_t tokens = 64) {
    WarpSpecConfig c;
    c.total_tokens = tokens;
    c.token_size = 64;
    c.tokens_per_tile = 16;
    c.tokens_per_chunk = 8;
    c.cpu_src = g_src.data();
    c.gpu_dst = g_dst.data();
    return c;
}

#define REQUIRE(cond)                                                            \
    do {                                                                         \
        if (!(cond)) {                                                           \
            std::fprintf(stderr, "sessions: line %d: %s\n", __LINE__, #cond);    \
            return 3;                                                            \
        }                                                                        \
    } while (0)

// A kernel that the caller launched on device 0's queue, not synchronised,
// while the session is destroyed with device 1 current.
int run_owner_device() {
    emu::set_device_count(2);
    auto* a = new WarpSpecSession(config());
    REQUIRE(a->ok());
    const void* queue = a->get_launch_params().tq;
    emu::start_kernel(0);
    emu::start_kernel(1);
    REQUIRE(gfd_hip_set_device(1) == 0);
    delete a;
    REQUIRE(!emu::kernel_runs(0));  // waited for: nobody writes the queue any more
    REQUIRE(emu::kernel_runs(1));   // and only for its own device
    int dev = -1;
    REQUIRE(gfd_hip_get_device(&dev) == 0 && dev == 1);
    {
        WarpSpecSession other(config());
        REQUIRE(other.ok() && other.get_launch_params().tq != queue);
    }
    REQUIRE(gfd_hip_set_device(0) == 0);
    WarpSpecSession b(config());
    REQUIRE(b.ok() && b.get_launch_params().tq == queue);
    return 0;
}

// A kernel that the caller launched itself, or whose read-back launch failed:
// synchronize() copies the counters and the progress back, and the session is
// destroyed, without host memory to allocate (both are reached from C entries,
// where an exception would end the program).
int run_no_memory() {
    auto* s = new WarpSpecSession(config());
    REQUIRE(s->ok());
    gfd::TiledQueue* tq = s->get_launch_params().tq;
    s->before_launch(nullptr);
    // The kernel's writes: four tiles of 16 tokens landed.
    for (int t = 0; t < 4; t++) tq->d_tile_chunk_done[t] = 16;
    auto* c = reinterpret_cast<gfd::TileDeviceCounters*>(tq->d_tile_chunk_done + gfd::MAX_TILES);
    c->next_tile = 5;
    c->tiles_done = 4;
    g_no_memory = true;
    const bool done = s->synchronize();
    g_no_memory = false;
    REQUIRE(done && s->tiles_done() == 4 && s->error_bits() == 0 && tq->scheduler.next_tile == 4);
    for (int t = 0; t < 5; t++) REQUIRE(tq->tile_chunk_done[t] == (t < 4 ? 16u : 0u));
    g_no_memory = true;
    delete s;
    g_no_memory = false;
    return 0;
}

// Sessions destroyed, then hipDeviceReset(): the queues they left are gone, and
// sessions after it get new ones, each its own.
int run_device_reset() {
    emu::set_device_count(2);
    REQUIRE(gfd_hip_set_device(1) == 0);
    auto* other = new WarpSpecSession(config());
    const void* kept = other->get_launch_params().tq;
    delete other;
    REQUIRE(gfd_hip_set_device(0) == 0);
    {
        WarpSpecSession a(config()), b(config()), c(config());
        REQUIRE(a.ok() && b.ok() && c.ok());
    }
    emu::device_reset();
    std::vector<WarpSpecSession*> live;
    for (int i = 0; i < 6; i++) {
        live.push_back(new WarpSpecSession(config()));
        REQUIRE(live[i]->ok() && live[i]->get_launch_params().tq->scheduler.total_tiles == 4);
        for (int j = 0; j < i; j++)
            REQUIRE(live[i]->get_launch_params().tq != live[j]->get_launch_params().tq &&
                    live[i]->get_launch_params().tq->d_tile_chunk_done != live[j]->get_launch_params().tq->d_tile_chunk_done);
    }
    for (WarpSpecSession* s : live) delete s;
    REQUIRE(gfd_hip_set_device(1) == 0);  // the other device's queue is still there
    WarpSpecSession d(config());
    REQUIRE(d.ok() && d.get_launch_params().tq == kept);
    return 0;
}

// release_spare_queues() waits in a free for a kernel that ends only once
// another thread has made a session.
bool g_made = false;
std::thread g_other;
void make_session_elsewhere() {
    emu::set_free_hook(nullptr);
    auto made = std::make_shared<std::promise<bool>>();
    std::future<bool> f = made->get_future();
    g_other = std::thread([made] {
        WarpSpecSession s(config());
        made->set_value(s.ok());
    });
    g_made = f.wait_for(std::chrono::seconds(5)) == std::future_status::ready && f.get();
}
int run_release() {
    { WarpSpecSession a(config()); }
    emu::set_free_hook(make_session_elsewhere);
    WarpSpecSession::release_spare_queues();
    if (g_other.joinable()) g_other.join();
    REQUIRE(g_made);
    return 0;
}

}  // namespace

int main(int argc, char** argv) {
    setvbuf(stdout, nullptr, _IOLBF, 0);
    const std::string what = argc > 1 ? argv[1] : "";
    int rc = 4;
    if (what == "owner_device") rc = run_owner_device();
    if (what == "no_memory") rc = run_no_memory();
    if (what == "device_reset") rc = run_device_reset();
    if (what == "release") rc = run_release();
    WarpSpecSession::release_spare_queues();
    if (rc == 0) std::printf("%s: pass\n", what.c_str());
    if (rc == 4) std::fprintf(stderr, "usage: sessions_emu owner_device | no_memory | device_reset | release\n");
    return rc;
}
