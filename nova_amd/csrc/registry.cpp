// nova-mi355x: the ownership registry declared in nova_common.h.
#include <mutex>
#include <unordered_map>

#include "nova_common.h"

namespace nova_amd {

namespace {
std::mutex g_mu;
struct Owned {
    size_t bytes;      // 0: not recorded
    int device;
};
std::unordered_map<const void *, Owned> &owned()
{
    static std::unordered_map<const void *, Owned> map;
    return map;
}
} // namespace

void registry_track(const void *p, size_t bytes, int device)
{
    if (p == nullptr)
        return;
    std::lock_guard<std::mutex> lk(g_mu);
    owned()[p] = Owned{bytes, device};
}

bool registry_holds(const void *p, size_t bytes, int device)
{
    if (p == nullptr || bytes == 0)
        return false;
    std::lock_guard<std::mutex> lk(g_mu);
    const auto it = owned().find(p);
    return it != owned().end() && it->second.bytes == bytes && it->second.device == device;
}

bool registry_untrack(const void *p)
{
    std::lock_guard<std::mutex> lk(g_mu);
    return owned().erase(p) > 0;
}

} // namespace nova_amd
