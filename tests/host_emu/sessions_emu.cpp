// WarpSpecSession on the emulated runtime: its queue, and whom a destroyed
// session leaves it to.  One scenario per run, named on the command line;
// "pass" and status 0, or what went wrong and status 3.
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "emu.h"
#include "gfd/hip_shim.h"
#include "gfd/warp_spec_session.h"

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

}  // namespace

int main(int argc, char** argv) {
    setvbuf(stdout, nullptr, _IOLBF, 0);
    const std::string what = argc > 1 ? argv[1] : "";
    int rc = 4;
    if (what == "owner_device") rc = run_owner_device();
    WarpSpecSession::release_spare_queues();
    if (rc == 0) std::printf("%s: pass\n", what.c_str());
    if (rc == 4) std::fprintf(stderr, "usage: sessions_emu owner_device\n");
    return rc;
}
