// Side streams of the fused drivers: host code only.
#include "qbx_internal.h"

#include <array>
#include <condition_variable>
#include <map>
#include <memory>
#include <mutex>

namespace qbx {

int side_streams(int device, hipStream_t out[3])
{
    static std::mutex mu;
    static std::map<int, std::array<hipStream_t, 3>> pool;
    std::lock_guard<std::mutex> lock(mu);
    auto it = pool.find(device);
    if (it == pool.end()) {
        std::array<hipStream_t, 3> s{};
        for (hipStream_t &x : s) QBX_HIP(hipStreamCreateWithFlags(&x, hipStreamNonBlocking));
        it = pool.emplace(device, s).first;
    }
    for (int i = 0; i < 3; ++i) out[i] = it->second[i];
    return QBX_OK;
}

int ctx_events(qbx_ctx *ctx)
{
    for (hipEvent_t &e : ctx->ev)
        if (!e) QBX_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    return QBX_OK;
}

static std::mutex pair_mu;
static std::condition_variable pair_free;

using pair_list = std::vector<std::unique_ptr<side_pair>>;

// the device's pairs, the shared one first; pair_mu held
static int pairs_of(int device, pair_list **out)
{
    static std::map<int, pair_list> pool;
    pair_list &l = pool[device];
    *out = &l;
    if (!l.empty()) return QBX_OK;
    hipStream_t s[3];
    QBX_TRY(side_streams(device, s));
    l.emplace_back(new side_pair);
    l[0]->s[0] = s[0];
    l[0]->s[1] = s[1];
    return QBX_OK;
}

// the capture st is part of (its id + 1), 0 for none
static int capture_of(hipStream_t st, unsigned long long *id)
{
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    *id = 0;
    QBX_HIP(hipStreamIsCapturing(st, &cs));
    if (cs == hipStreamCaptureStatusNone) return QBX_OK;
    QBX_HIP(hipStreamGetCaptureInfo(st, &cs, id));
    ++*id;
    return QBX_OK;
}

int side_pair_hold(int device, hipStream_t st, side_pair **out)
{
    *out = nullptr;
    unsigned long long id, other;
    QBX_TRY(capture_of(st, &id));
    std::lock_guard<std::mutex> lock(pair_mu);
    pair_list *pairs;
    QBX_TRY(pairs_of(device, &pairs));
    for (size_t k = id == 0 ? 0 : 1; k < pairs->size(); ++k) {
        side_pair *p = (*pairs)[k].get();
        bool free = !p->held;
        for (int i = 0; free && i < 2; ++i) {
            QBX_TRY(capture_of(p->s[i], &other));
            free = other == 0 || other == id;
        }
        if (!free) continue;
        p->held = true;
        *out = p;
        return QBX_OK;
    }
    if (pairs->size() == 1 + SIDE_PAIRS) return QBX_OK;
    std::unique_ptr<side_pair> p(new side_pair);
    for (hipStream_t &x : p->s) QBX_HIP(hipStreamCreateWithFlags(&x, hipStreamNonBlocking));
    p->held = true;
    *out = p.get();
    pairs->push_back(std::move(p));
    return QBX_OK;
}

int side_streams_capture(int device, hipStream_t st, side_pair **out)
{
    *out = nullptr;
    unsigned long long id;
    QBX_TRY(capture_of(st, &id));
    if (id == 0) return QBX_OK;
    std::unique_lock<std::mutex> lock(pair_mu);
    pair_list *pairs;
    QBX_TRY(pairs_of(device, &pairs));
    side_pair *p = (*pairs)[0].get();
    pair_free.wait(lock, [&] { return !p->held; });
    p->held = true;
    *out = p;
    return QBX_OK;
}

void side_pair_release(side_pair *p)
{
    if (!p) return;
    {
        std::lock_guard<std::mutex> lock(pair_mu);
        p->held = false;
    }
    pair_free.notify_all();
}

}  // namespace qbx
