// The pool of pinned staging buffers (see hostcopy.h).
#include <mutex>
#include <vector>

#include "hostcopy.h"

namespace tags {

namespace {
// never destroyed: nothing of the HIP runtime is called while the process ends
struct Pool {
    std::mutex mu;
    std::vector<PinnedStage*> idle;
};
Pool& pool()
{
    static Pool* p = new Pool();
    return *p;
}
void destroy(PinnedStage* s)
{
    for (int i = 0; i < 2; i++) {
        (void)s->wait(i);
        if (s->p[i]) (void)hipHostFree(s->p[i]);
        if (s->ev[i]) (void)hipEventDestroy(s->ev[i]);
    }
    delete s;
}
}  // namespace

PinnedStage* stage_get()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    {
        Pool& q = pool();
        std::lock_guard<std::mutex> lock(q.mu);
        for (size_t i = q.idle.size(); i-- > 0;)
            if (q.idle[i]->dev == dev) {
                PinnedStage* s = q.idle[i];
                q.idle.erase(q.idle.begin() + (long)i);
                return s;
            }
    }
    PinnedStage* s = new PinnedStage();
    s->dev = dev;
    for (int i = 0; i < 2; i++)
        if (hipHostMalloc(&s->p[i], PinnedStage::kChunk, 0) != hipSuccess ||
            hipEventCreateWithFlags(&s->ev[i], hipEventDisableTiming) != hipSuccess) {
            destroy(s);
            return nullptr;
        }
    return s;
}

void stage_put(PinnedStage* s)
{
    {
        Pool& q = pool();
        std::lock_guard<std::mutex> lock(q.mu);
        if ((int)q.idle.size() < kStageIdle) {
            q.idle.push_back(s);
            return;
        }
    }
    destroy(s);
}

void stage_release()
{
    std::vector<PinnedStage*> out;
    {
        Pool& q = pool();
        std::lock_guard<std::mutex> lock(q.mu);
        out.swap(q.idle);
    }
    for (PinnedStage* s : out) destroy(s);
}

}  // namespace tags

extern "C" void tags_release_staging(void) { tags::stage_release(); }
