// mesh_scratch.cpp -- the store of mesh_scratch.h.
#include "mesh_scratch.h"

#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "../../include/cvt.h"
#include "cvt_engine.h"

namespace cvt {

namespace {

// Between two calls a program may reset the device, which frees what lies in the
// store, and the addresses may then hold allocations of its own.  Each
// allocation has an id that no other of the process ever gets, so a block is
// used, and freed, only while its ids still stand for its addresses (0.06 us
// an id).
struct Block {
    int device;
    char *dev;
    size_t bytes;
    int *pinned;
    uint64_t dev_id, pinned_id;
};

// the id of the allocation at p, 0 where there is none
uint64_t allocation_id(void *p)
{
    uint64_t id = 0;
    if (hipPointerGetAttribute(&id, HIP_POINTER_ATTRIBUTE_BUFFER_ID, p) == hipSuccess) return id;
    (void)hipGetLastError();
    return 0;
}
bool holds(void *p, uint64_t id) { return id && allocation_id(p) == id; }
bool whole(const Block &b) { return holds(b.dev, b.dev_id) && holds(b.pinned, b.pinned_id); }

std::mutex g_mutex;
std::vector<Block> &store()
{
    // never destroyed: the runtime may be gone before a static's destructor
    static std::vector<Block> *s = new std::vector<Block>();
    return *s;
}

// frees a block that has lain in the store
void drop(const Block &b)
{
    if (holds(b.dev, b.dev_id)) (void)hipFree(b.dev);
    if (holds(b.pinned, b.pinned_id)) (void)hipHostFree(b.pinned);
}

}  // namespace

void release_scratch()
{
    std::vector<Block> all;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        all.swap(store());
    }
    for (const Block &b : all) drop(b);
}

hipError_t MeshScratch::take(size_t bytes)
{
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return e;
    for (;;) {
        Block b;
        {
            std::lock_guard<std::mutex> lock(g_mutex);
            std::vector<Block> &s = store();
            auto best = s.end();
            for (auto i = s.begin(); i != s.end(); ++i)
                if (i->device == device && i->bytes >= bytes && (best == s.end() || i->bytes < best->bytes))
                    best = i;
            if (best == s.end()) break;
            b = *best;
            s.erase(best);
        }
        if (whole(b)) {
            device_ = device;
            dev_ = b.dev;
            bytes_ = b.bytes;
            pinned_ = b.pinned;
            return hipSuccess;
        }
        drop(b);
    }
    // whole megabytes, so that a slightly larger mesh fits the same block
    const size_t mb = (size_t)1 << 20, want = std::max(mb, (bytes + mb - 1) / mb * mb);
    void *p = nullptr, *h = nullptr;
    e = hipMalloc(&p, want);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        release_scratch();
        e = hipMalloc(&p, want);
        if (e != hipSuccess) return e;
    }
    e = hipHostMalloc(&h, sizeof(int) * kStatusWords, hipHostMallocDefault);
    if (e != hipSuccess) {
        (void)hipFree(p);
        return e;
    }
    device_ = device;
    dev_ = static_cast<char *>(p);
    bytes_ = want;
    pinned_ = static_cast<int *>(h);
    return hipSuccess;
}

MeshScratch::~MeshScratch()
{
    if (!dev_) return;
    if (!idle_) (void)hipStreamSynchronize(nullptr);
    Block b{device_, dev_, bytes_, pinned_, allocation_id(dev_), allocation_id(pinned_)};
    if (!b.dev_id || !b.pinned_id) {               // could not be told from another's later
        (void)hipFree(dev_);
        (void)hipHostFree(pinned_);
        return;
    }
    // the newest block stays, for the next call like this one, and the oldest
    // leave until the others fit beside it (were this one to leave, a mesh that
    // has grown past half the bound would be allocated anew on every call)
    if (bytes_ > kScratchBytes) {
        drop(b);
        return;
    }
    try {
        std::lock_guard<std::mutex> lock(g_mutex);
        store().push_back(b);
    } catch (...) {
        drop(b);
        return;
    }
    for (;;) {
        Block out{};
        {
            std::lock_guard<std::mutex> lock(g_mutex);
            std::vector<Block> &s = store();
            size_t held = 0, count = 0;
            auto oldest = s.end();
            for (auto i = s.begin(); i != s.end(); ++i)
                if (i->device == device_) {
                    held += i->bytes;
                    ++count;
                    if (oldest == s.end()) oldest = i;
                }
            if (held <= kScratchBytes && count <= (size_t)kScratchBlocks) return;
            out = *oldest;
            s.erase(oldest);
        }
        drop(out);
    }
}

bool in_place(const void *p, size_t align)
{
    if (!p || (uintptr_t)p % align) return false;
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    int device = 0;
    return hipGetDevice(&device) == hipSuccess && a.type == hipMemoryTypeDevice && a.device == device;
}

}  // namespace cvt

extern "C" int cvt_release_scratch(void)
{
    cvt::clear_error();
    cvt::release_scratch();
    return CVT_OK;
}
