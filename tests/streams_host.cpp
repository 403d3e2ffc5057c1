// The adjoint driver's stage DAG and the side streams on a HIP of bookkeeping:
// every launch keeps the set of launches that are ordered before it.  Built and
// run by test_streams_host.py.
#include "../pytential_amd/csrc/qbx_internal.h"

#include <atomic>
#include <chrono>
#include <cstdarg>
#include <cstdlib>
#include <map>
#include <set>
#include <thread>

using std::set;

struct Launch {
    hipStream_t s;
    int stage;
    set<int> before;
};
static std::vector<Launch> launches;
static std::map<void *, set<int>> known;                    // stream or event
static std::map<void *, unsigned long long> capture;        // stream -> capture id
static std::map<void *, bool> made;
static long handles = 1000;

static hipStream_t stream() { return (hipStream_t)(handles += 8); }

extern "C" {
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = stream(); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = (hipEvent_t)(handles += 8);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { known[e] = known[s]; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    known[s].insert(known[e].begin(), known[e].end());
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c)
{
    *c = capture.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamGetCaptureInfo(hipStream_t s, hipStreamCaptureStatus *c,
                                   unsigned long long *id)
{
    *id = capture.count(s) ? capture[s] : 0;
    return hipStreamIsCapturing(s, c);
}
hipError_t hipFree(void *) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }
}

namespace qbx {
void set_error(const char *, ...) {}
}
using namespace qbx;

#define REQUIRE(c)                                                          \
    do {                                                                    \
        if (!(c)) {                                                         \
            printf("line %d: %s\n", __LINE__, #c);                          \
            exit(1);                                                        \
        }                                                                   \
    } while (0)

// arrays: 0 Pa 1 Qa 2 La 3 Ma 4 str_adj; r reads, a adds by atomics, w anything else
struct Use {
    int stage;
    const char *how[5];
};
static const Use USES[] = {
    {QBX_ADJ_QBXL2P, {"r", "w", "", "", ""}}, {QBX_ADJ_L2QBXL, {"", "r", "w", "", ""}},
    {QBX_ADJ_L2P, {"r", "", "w", "", ""}},    {QBX_ADJ_L2L, {"", "", "w", "", ""}},
    {QBX_ADJ_M2L, {"", "", "r", "a", ""}},    {QBX_ADJ_M2QBXL, {"", "r", "", "a", ""}},
    {QBX_ADJ_M2P, {"r", "", "", "a", ""}},    {QBX_ADJ_P2L, {"", "", "r", "", "a"}},
    {QBX_ADJ_P2QBXL, {"", "r", "", "", "a"}}, {QBX_ADJ_P2P, {"r", "", "", "", "a"}},
    {QBX_ADJ_M2M, {"", "", "", "w", ""}},     {QBX_ADJ_P2M, {"", "", "", "r", "w"}},
};

static const Use &use_of(int stage)
{
    for (const Use &u : USES)
        if (u.stage == stage) return u;
    abort();
}

static int dag(qbx_ctx *ctx, hipStream_t st, int fail, set<hipStream_t> *used = nullptr)
{
    launches.clear();
    known.clear();
    return adjoint_dag(
        ctx, st,
        [&](hipStream_t s, int stage, const double *, double *) {
            if (stage == fail) return (int)QBX_ERR_INVALID;
            if (used) used->insert(s);
            launches.push_back({s, stage, known[s]});
            known[s].insert((int)launches.size() - 1);
            return (int)QBX_OK;
        },
        nullptr, nullptr, nullptr, nullptr, nullptr);
}

int main()
{
    qbx_ctx ctx;
    hipStream_t st = stream();
    // every pair of stages that share an array is ordered, but for readers
    // together and atomic additions together
    for (int tune : {4, 1}) {
        ctx.tune[QBX_TUNE_DRIVE_STREAMS] = tune;
        REQUIRE(dag(&ctx, st, -1) == QBX_OK && launches.size() == 12);
        for (size_t j = 0; j < launches.size(); ++j)
            for (size_t i = 0; i < j; ++i)
                for (int a = 0; a < 5; ++a) {
                    const std::string x = use_of(launches[i].stage).how[a],
                                      y = use_of(launches[j].stage).how[a];
                    if (x.empty() || y.empty() || (x == y && x != "w")) continue;
                    REQUIRE(launches[j].before.count((int)i));
                }
        // whatever stage fails, all that was launched is before what st does next
        for (const Use &u : USES) {
            REQUIRE(dag(&ctx, st, u.stage) == QBX_ERR_INVALID);
            REQUIRE(known[st].size() == launches.size());
        }
    }
    ctx.tune[QBX_TUNE_DRIVE_STREAMS] = 4;
    // calls one after another, also after an error, take the same two streams,
    // those of the forward
    hipStream_t fwd[3];
    REQUIRE(side_streams(0, fwd) == QBX_OK);
    set<hipStream_t> a, b;
    dag(&ctx, st, -1, &a);
    dag(&ctx, st, -1, &b);
    REQUIRE(a == b && (a == set<hipStream_t>{st, fwd[0], fwd[1]}));
    auto apart = [](const side_pair *x, const hipStream_t *y) {
        for (int i = 0; i < 3; ++i)
            if (x->s[0] == y[i] || x->s[1] == y[i]) return false;
        return true;
    };
    // a call while another has them takes others
    side_pair *p = nullptr, *q = nullptr;
    REQUIRE(side_pair_hold(0, st, &p) == QBX_OK && p && p->s[0] == fwd[0]);
    b.clear();
    dag(&ctx, st, -1, &b);
    REQUIRE(b.size() == 3 && !b.count(p->s[0]) && !b.count(p->s[1]));
    // a forward's capture waits for the one that has them
    hipStream_t c1 = stream(), c2 = stream();
    capture[c1] = 7;
    capture[c2] = 8;
    std::atomic<bool> in{false};
    std::thread th([&] {
        side_pair *f = nullptr;
        REQUIRE(side_streams_capture(0, c1, &f) == QBX_OK && f == p);
        in = true;
    });
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    REQUIRE(!in);
    side_pair_release(p);
    th.join();
    // and no adjoint begins on them until it is through, nor, forked into its
    // capture, until that ends
    for (int forked = 0; forked < 2; ++forked) {
        REQUIRE(side_pair_hold(0, st, &q) == QBX_OK && q && apart(q, fwd));
        side_pair_release(q);
        if (forked) break;
        capture[fwd[0]] = capture[fwd[1]] = capture[fwd[2]] = 7;
        side_pair_release(p);
    }
    for (hipStream_t x : fwd) capture.erase(x);
    REQUIRE(side_streams_capture(0, st, &q) == QBX_OK && !q);
    // an adjoint in a capture has its own pair, and keeps it until the capture
    // ends: not for eager calls, nor for another capture, but for the same one
    REQUIRE(side_pair_hold(0, c1, &p) == QBX_OK && p && apart(p, fwd));
    side_pair_release(p);
    capture[p->s[0]] = capture[p->s[1]] = 7;
    REQUIRE(side_pair_hold(0, c2, &q) == QBX_OK && q && q != p && apart(q, fwd));
    side_pair_release(q);
    side_pair *first = nullptr;
    REQUIRE(side_pair_hold(0, st, &first) == QBX_OK && first->s[0] == fwd[0]);
    REQUIRE(side_pair_hold(0, st, &q) == QBX_OK && q && q != p);
    side_pair_release(q);
    REQUIRE(side_pair_hold(0, c1, &q) == QBX_OK && q == p);
    // the pool is bounded; with all pairs taken a call runs on its own stream
    std::vector<side_pair *> held{first, q};
    while (true) {
        REQUIRE(side_pair_hold(0, st, &q) == QBX_OK);
        if (!q) break;
        held.push_back(q);
    }
    REQUIRE(held.size() == 1 + SIDE_PAIRS);
    b.clear();
    REQUIRE(dag(&ctx, st, -1, &b) == QBX_OK && b == set<hipStream_t>{st});
    // another device has its own
    REQUIRE(side_pair_hold(1, st, &q) == QBX_OK && q);
    for (side_pair *x : held) REQUIRE(x != q);
    printf("ok\n");
    return 0;
}
