// Drives HostLink (softmold_amd/csrc/sm_transfer.hpp) without a GPU: the HIP calls it makes and
// the kernels it launches are played here on host memory, with a device to a stream, an event
// and an allocation.  Usage: transfer_harness SCENARIO; exit code 0 if it held.
#include "sm_transfer.hpp"

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <ctime>
#include <string>

namespace {

struct FakeStream { int device; };
struct FakeEvent { int device; };

int g_device = 0;                          // the current device
int g_allocations = 0, g_events = 0;       // made so far
int g_buffer_device = -1;                  // current at the last pinned allocation
size_t g_largest = 0;                      // pinned allocation, bytes
std::atomic<int> g_bad_wait{-1};           // the wait for an event that fails, counted down
std::atomic<int> g_busy_ms{0};             // the GPU's queued work: the next wait lasts so long
thread_local int g_bad_new = -1;           // this thread's allocation that fails, counted down

#define EXPECT(cond)                                                       \
    do {                                                                   \
        if (!(cond)) {                                                     \
            std::fprintf(stderr, "line %d: %s\n", __LINE__, #cond);        \
            std::exit(1);                                                  \
        }                                                                  \
    } while (0)

}  // namespace

thread_local std::string smapi::g_err;

void *operator new(size_t bytes)
{
    if (g_bad_new >= 0 && g_bad_new-- == 0) throw std::bad_alloc();
    if (void *p = std::malloc(bytes ? bytes : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipGetDevice(int *d) { *d = g_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { g_device = d; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorName(hipError_t e) { return e == hipSuccess ? "hipSuccess" : "hipError"; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    g_events++;
    *e = reinterpret_cast<hipEvent_t>(new FakeEvent{g_device});
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<FakeEvent *>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st)
{
    return reinterpret_cast<FakeEvent *>(e)->device == reinterpret_cast<FakeStream *>(st)->device ? hipSuccess
                                                                                                  : hipErrorInvalidHandle;
}
hipError_t hipEventSynchronize(hipEvent_t)
{
    std::this_thread::sleep_for(std::chrono::milliseconds(g_busy_ms.exchange(0)));
    return g_bad_wait >= 0 && g_bad_wait-- == 0 ? hipErrorUnknown : hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned)
{
    g_allocations++;
    g_buffer_device = g_device;
    g_largest = std::max(g_largest, bytes);
    *p = std::malloc(bytes);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
}

namespace smdev {
void launch_post(hipStream_t, const double *src, size_t count, const DevGlobal *glob, double *head)
{
    std::memcpy(head, (const void *)glob, sizeof(long long));
    for (size_t i = 0; i < count; i++) head[1 + i] = src[i];
}
void launch_pack(hipStream_t, int first, int count, const PackSrc &src, double *out, const DevRep *reps, int nrep,
                 const DevGlobal *glob, double *head)
{
    if (head) {
        std::memcpy(head, (const void *)glob, sizeof(long long));
        for (int i = 0; i < 3 * nrep; i++) head[1 + i] = reps[i / 3].L[i % 3];
    }
    float *f = reinterpret_cast<float *>(out + (src.beads ? 3 * (size_t)count : 0));
    for (int e = 0; e < 3 * count; e++) {
        const int i = first + e / 3, c = e % 3;
        if (src.beads) out[e] = (&src.beads[i].x)[c];
        if (src.a) f[e] = (&src.a[i].x)[c];
        if (src.b) f[(src.a ? 3 * (size_t)count : 0) + e] = (&src.b[i].x)[c];
    }
}
void launch_set_scale(hipStream_t, DevRep *reps, int nrep, const double *scale)
{
    for (int i = 0; i < 3 * nrep; i++) reps[i / 3].scale[i % 3] = scale[i];
}
void launch_set_positions(hipStream_t, int first, int count, const double *pos, Bead *beads)
{
    for (int e = 0; e < 3 * count; e++) (&beads[first + e / 3].x)[e % 3] = pos[e];
}
}  // namespace smdev

using namespace smdev;

namespace {

// A context's state: n beads of R replicas on device `device`.
struct State {
    int n, R;
    FakeStream stream;
    std::vector<Bead> beads;
    std::vector<float4> vel;
    std::vector<DevRep> reps;
    DevGlobal glob{};
    State(int n_, int r_, int device) : n(n_), R(r_), stream{device}, beads(n_), vel(n_), reps(r_)
    {
        for (int i = 0; i < n; i++) {
            beads[i].x = 0.5 + i, beads[i].y = 2.0 * i, beads[i].z = -1.0 * i;
            vel[i].x = 0.25f * i, vel[i].y = 1.0f, vel[i].z = -0.5f * i;
        }
        for (int r = 0; r < R; r++)
            for (int d = 0; d < 3; d++) reps[r].L[d] = 10.0 * r + d;
        glob.flags = 5, glob.fallbacks = 9;
    }
    hipStream_t st() { return reinterpret_cast<hipStream_t>(&stream); }
    PackSrc src() { return PackSrc{beads.data(), vel.data(), nullptr}; }
};

void check_download(State &s, HostLink &link)
{
    std::vector<double> pos(3 * (size_t)s.n, 7.0), vel(pos), box(3 * (size_t)s.R);
    EXPECT(link.fetch_beads(s.st(), s.n, s.src(), pos.data(), vel.data(), nullptr, &s.glob, s.reps.data(), s.R, box.data()) == 5);
    for (int i = 0; i < s.n; i++)
        for (int c = 0; c < 3; c++) {
            EXPECT(pos[3 * (size_t)i + c] == (&s.beads[i].x)[c]);
            EXPECT(vel[3 * (size_t)i + c] == (&s.vel[i].x)[c]);
        }
    for (int i = 0; i < 3 * s.R; i++) EXPECT(box[i] == s.reps[i / 3].L[i % 3]);
    EXPECT(link.fallbacks() == 9);
}

// Calls made while another device is current than the context's.
int other_device()
{
    State s(200001, 3, 1);
    HostLink link;
    g_device = 1;
    link.create(s.R);
    g_device = 0;
    std::vector<double> res(4 * (size_t)s.R, 3.25), got(res.size()), box(3 * (size_t)s.R);
    EXPECT(link.fetch(s.st(), &s.glob, res.data(), res.size(), got.data()) == 5 && got == res);
    EXPECT(link.fetch_boxes(s.st(), &s.glob, s.reps.data(), s.R, box.data()) == 5 && box[4] == 11.0);
    check_download(s, link);
    EXPECT(g_buffer_device == 1 && g_device == 0);
    std::vector<double> pos(3 * (size_t)s.n);
    for (size_t e = 0; e < pos.size(); e++) pos[e] = 0.125 * e;
    link.send_positions(s.st(), s.n, pos.data(), s.beads.data());
    for (int i = 0; i < s.n; i++) EXPECT(s.beads[i].y == pos[3 * (size_t)i + 1]);
    link.send_scale(s.st(), s.reps.data(), s.R, pos.data());
    EXPECT(s.reps[2].scale[1] == pos[7]);
    link.destroy();
    return 0;
}

// The first result of a new context, and the largest.
int no_allocation()
{
    State s(10, 5, 0);
    HostLink link;
    link.create(s.R);
    const int made = g_allocations + g_events;
    std::vector<double> res(4 * (size_t)s.R, -2.0), got(res.size());
    for (size_t count : {(size_t)s.R, res.size(), (size_t)0}) link.fetch(s.st(), &s.glob, res.data(), count, got.data());
    EXPECT(got == res);
    link.fetch_boxes(s.st(), &s.glob, s.reps.data(), s.R, got.data());
    EXPECT(g_allocations + g_events == made);
    link.destroy();
    return 0;
}

// The pinned buffers of a first download: none of the length whose allocation costs more than
// the download of a few chunks saves.
int first_buffers()
{
    for (int n : {1, 32768, 32769, 72000, 196608, 196609, 500000}) {
        State s(n, 1, 0);
        HostLink link;
        link.create(s.R);
        g_largest = 0;
        check_download(s, link);
        if (n <= 196608) EXPECT(g_largest <= 2u << 20);
        link.destroy();
    }
    return 0;
}

// Downloads whose workers cannot all be started, and downloads that fail under way.
int troubled_team()
{
    State s(300000, 1, 0);
    HostLink link;
    link.create(s.R);
    check_download(s, link);
    std::vector<double> pos(3 * (size_t)s.n), box(3);
    for (int k = 0; k < 8; k++) {   // the k-th allocation of the call: the team's room, then a worker each
        std::fill(pos.begin(), pos.end(), 7.0);
        g_bad_new = k;
        EXPECT(link.fetch_beads(s.st(), s.n, s.src(), pos.data(), nullptr, nullptr, &s.glob, s.reps.data(), 1, box.data()) == 5);
        g_bad_new = -1;
        for (int i = 0; i < s.n; i++) EXPECT(pos[3 * (size_t)i + 2] == s.beads[i].z);
    }
    for (int k = 0; k < 5; k++)
        for (int rep = 0; rep < 20; rep++) {
            bool thrown = false;
            g_bad_wait = k;
            try {
                link.fetch_beads(s.st(), s.n, s.src(), pos.data(), nullptr, nullptr, &s.glob, s.reps.data(), 1, box.data());
            } catch (const smapi::ApiError &) {
                thrown = true;
            }
            g_bad_wait = -1;
            EXPECT(thrown);
        }
    link.destroy();
    return 0;
}

// A download behind 600 ms of the GPU's work: the host's threads sleep meanwhile.
int behind_work()
{
    State s(300000, 1, 0);
    HostLink link;
    link.create(s.R);
    check_download(s, link);
    const std::clock_t idle = std::clock();
    check_download(s, link);
    const std::clock_t start = std::clock();
    g_busy_ms = 600;
    check_download(s, link);
    const double plain = double(start - idle) / CLOCKS_PER_SEC, behind = double(std::clock() - start) / CLOCKS_PER_SEC;
    std::fprintf(stderr, "CPU seconds: %.3f alone, %.3f behind the work\n", plain, behind);
    EXPECT(behind < plain + 0.3);
    link.destroy();
    return 0;
}

}  // namespace

int main(int argc, char **argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    try {
        if (what == "other_device") return other_device();
        if (what == "no_allocation") return no_allocation();
        if (what == "first_buffers") return first_buffers();
        if (what == "troubled_team") return troubled_team();
        if (what == "behind_work") return behind_work();
    } catch (const std::exception &e) {
        std::fprintf(stderr, "%s: %s\n", what.c_str(), e.what());
        return 1;
    }
    std::fprintf(stderr, "unknown scenario\n");
    return 2;
}
