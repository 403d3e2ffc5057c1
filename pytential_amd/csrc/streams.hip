// Side streams of the fused drivers: host code only.
#include "qbx_internal.h"

#include <array>
#include <map>
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

}  // namespace qbx
