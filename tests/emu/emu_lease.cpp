// The query workspaces' leases (taken from tl_runtime.cpp as they are) over a
// device that is played here: two threads, and a growth that waits for the
// workspace's last user.  Prints one line a check; exits 1 if one fails.
#include "hip/hip_runtime.h"
#include <condition_variable>
#include <cstdio>
#include <map>
#include <mutex>
#include <thread>

static std::mutex m;
static std::condition_variable cv;
static bool hold = false, waiting = false;   // the device is busy; a thread waits for it
static size_t limit = ~(size_t)0, used = 0;
static std::map<void *, size_t> blocks;

static hipError_t dev_sync(hipEvent_t) {
    std::unique_lock<std::mutex> lk(m);
    waiting = true;
    cv.notify_all();
    const bool ok = cv.wait_for(lk, std::chrono::seconds(20), [] { return !hold; });
    return ok ? hipSuccess : hipErrorUnknown;
}
static hipError_t dev_malloc(void **p, size_t n) {
    if (used + n > limit) return hipErrorUnknown;
    *p = malloc(1);
    blocks[*p] = n;
    used += n;
    return hipSuccess;
}
static hipError_t dev_free(void *p) {
    used -= blocks[p];
    blocks.erase(p);
    free(p);
    return hipSuccess;
}
typedef enum { hipStreamCaptureModeRelaxed = 2 } hipStreamCaptureMode;
static hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
#define hipEventSynchronize dev_sync
#define hipMalloc dev_malloc
#define hipFree dev_free
#include "src/tl_internal.hpp"
namespace tl {
#include "emu_lease_code.hpp"
}
using namespace tl;

static int bad = 0;
static void check(const char *what, bool ok) {
    printf("[emu-lease] %s: %s\n", what, ok ? "right" : "WRONG");
    bad += !ok;
}

int main() {
    Ctx c;
    c.device = 0;
    const hipStream_t s1 = (hipStream_t)1, s2 = (hipStream_t)2;
    Lease *a = lease_take(&c, 1000, s1);
    check("a lease has the bytes", a && a->mem && a->bytes >= 1000);
    Lease *b = lease_take(&c, 500, s2);
    check("two calls have a lease each", b && b != a);
    check("a third does without", !lease_take(&c, 10, (hipStream_t)3));
    lease_give(a, s1);
    lease_give(b, s2);
    void *mem = a->mem;
    a = lease_take(&c, 1100, s1);
    check("a somewhat larger batch needs no new memory", a && a->mem == mem);
    lease_give(a, s1);

    // s1's workspace grows while its last user runs: s2's call does not wait
    hold = true;
    Lease *grown = nullptr;
    std::thread t([&] { grown = lease_take(&c, 5000, s1); });
    {
        std::unique_lock<std::mutex> lk(m);
        cv.wait(lk, [] { return waiting; });
    }
    Lease *other = nullptr;
    bool done = false;
    std::thread u([&] {
        Lease *l = lease_take(&c, 400, s2);
        std::lock_guard<std::mutex> lk(m);
        other = l;
        done = true;
        cv.notify_all();
    });
    {
        std::unique_lock<std::mutex> lk(m);
        cv.wait_for(lk, std::chrono::seconds(5), [&] { return done; });
        check("a growing lease holds no other call up", done && other);
        hold = false;
        cv.notify_all();
    }
    t.join();
    u.join();
    check("it has grown", grown && grown->bytes >= 5000 && grown != other);
    leases_release(&c);
    check("leases in use are not released", used == grown->bytes + other->bytes);
    lease_give(grown, s1);
    leases_release(&c);
    check("idle ones are", used == other->bytes);
    lease_give(other, s2);
    leases_release(&c);
    check("all of them", used == 0);
    limit = 1100;
    a = lease_take(&c, 1000, s1);
    check("the bytes asked where a quarter more is not to be had", a && a->bytes == 1000);
    lease_give(a, s1);
    check("none where memory is short", !lease_take(&c, 2000, s1));
    limit = 4000;
    a = lease_take(&c, 2000, s1);
    check("and one when it is there again", a && a->bytes >= 2000);
    lease_give(a, s1);
    fflush(stdout);
    return bad ? 1 : 0;
}
