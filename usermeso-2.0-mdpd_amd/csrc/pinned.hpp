// Page-locked staging buffers of one pool (asynchronous copies need them),
// reused by size class and freed with the pool.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <iterator>
#include <map>

namespace mdpd {

// A block's size is its class: the power of two, from 1 MiB up, that holds the
// request.  Requests take blocks of their own class only, so a small job's
// block is never a large job's; below 1 MiB inputs and results share a class,
// so that a first batch's results reuse its input blocks (classes from 64 KiB
// up: 256 more allocations in the first batch of 256 droplets, 20 ms).
struct PinnedCache {
    static constexpr size_t MIN_BLOCK = (size_t)1 << 20;
    // blocks held by inputs packed ahead of their admission, 512 of the
    // smallest; beyond this (or where page-locked memory runs out) inputs wait
    // in pageable memory, which costs each a copy (256 droplets of 2,000 to
    // 40,000 particles hold 260 MiB)
    static constexpr size_t MAX_STAGED = (size_t)1 << 29;
    // free blocks kept (a full hold of results, the inputs that wait and as
    // much again): a request that finds none of its class first gives back the
    // largest of more than this, so that sizes that drift from class to class
    // do not each leave their most behind
    static constexpr size_t MAX_FREE = (size_t)1 << 31;
    std::multimap<size_t, void *> free_;
    size_t staged = 0, free_bytes = 0;

    ~PinnedCache() { trim(0); }
    void trim(size_t keep)
    {
        while (free_bytes > keep) {
            auto it = std::prev(free_.end());
            (void)hipHostFree(it->second);
            free_bytes -= it->first;
            free_.erase(it);
        }
    }
    static size_t size_class(size_t bytes)
    {
        size_t sz = MIN_BLOCK;
        while (sz < bytes) sz <<= 1;
        return sz;
    }
    hipError_t get(size_t bytes, void **p, size_t &got)
    {
        got = size_class(bytes);
        auto it = free_.find(got);
        if (it == free_.end()) {
            trim(MAX_FREE);
            const hipError_t e = hipHostMalloc(p, got, hipHostMallocDefault);
            if (e == hipSuccess || free_.empty()) return e;
            (void)hipGetLastError();
            trim(0);                          // what other classes hold may be what is missing
            return hipHostMalloc(p, got, hipHostMallocDefault);
        }
        *p = it->second;
        free_bytes -= got;
        free_.erase(it);
        return hipSuccess;
    }
    void put(void *p, size_t sz)
    {
        free_.emplace(sz, p);
        free_bytes += sz;
    }

    // a block for an input that waits; false: none to be had
    bool stage(size_t bytes, void **p, size_t &got)
    {
        if (staged + size_class(bytes) > MAX_STAGED) return false;
        if (get(bytes, p, got) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        staged += got;
        return true;
    }
    // the input has gone to the device (its block is put back once read)
    void unstage(size_t got) { staged -= got; }
};

}  // namespace mdpd
