// Side streams of the fused drivers: host code only.
#include "qbx_internal.h"

#include <array>
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
    static std::map<int, std::vector<std::unique_ptr<side_pair>>> pool;
    *out = nullptr;
    unsigned long long id, other;
    QBX_TRY(capture_of(st, &id));
    std::lock_guard<std::mutex> lock(pair_mu);
    auto &pairs = pool[device];
    for (auto &p : pairs) {
        bool free = !p->held;
        for (int i = 0; free && i < 2; ++i) {
            QBX_TRY(capture_of(p->s[i], &other));
            free = other == 0 || other == id;
        }
        if (!free) continue;
        p->held = true;
        *out = p.get();
        return QBX_OK;
    }
    if (pairs.size() == SIDE_PAIRS) return QBX_OK;
    std::unique_ptr<side_pair> p(new side_pair);
    for (hipStream_t &x : p->s) QBX_HIP(hipStreamCreateWithFlags(&x, hipStreamNonBlocking));
    p->held = true;
    *out = p.get();
    pairs.push_back(std::move(p));
    return QBX_OK;
}

void side_pair_release(side_pair *p)
{
    std::lock_guard<std::mutex> lock(pair_mu);
    p->held = false;
}

}  // namespace qbx
