// work_pool.h -- work buffers of single calls, kept between calls.
#pragma once

#include <cstddef>
#include <mutex>
#include <vector>

namespace polyeri {

// Work buffers of single calls (MP2, CC, gradient, k-point SCF), kept between
// calls: mapping and unmapping gigabytes on each call took longer than the
// call ((H2O)8 cc-pVDZ MP2: 17 ms of kernels, 130 to 270 ms with hipMalloc and
// hipFree of its 9 GB in a process that holds other allocations).  A block is
// handed out only while it is in use by nobody (mutex; the caller waits for
// its streams before it gives a block back), and only for a request of nearly
// its size, so that a call never holds noticeably more than it asked for.  At
// most a quarter of a device's memory is kept idle ((H2O)12 cc-pVDZ MP2 works
// in 46 GB), the oldest blocks making room for new ones; all of a device's
// idle blocks go back when its last context ends, when an allocation of the
// library fails (get, alloc; release for those that rocBLAS and rocSOLVER
// make) and when the caller asks for it (polyeri_release_work), who alone
// knows what others in the process or on the device need.
//
// Mem: the device's allocator, with static functions
//   int device()                     the current device, negative on error
//   int alloc(void** p, size_t n)    0, or an error code, on the current device
//   void free(void* p)
//   size_t total(int device)         the memory of a device, 0 if unknown
template <typename Mem>
class WorkPool {
    struct Block {
        void* p;
        size_t bytes;
        int device;
    };
    std::mutex mu;
    std::vector<Block> idle, used;        // idle: oldest first
    std::vector<int> contexts;            // live contexts per device

    // How much larger than a request its block may be: up to 64 KB more than
    // twice the request for small buffers, never over 1 MB.
    static size_t slack(size_t bytes) {
        const size_t s = bytes + 65536;
        return s < (1u << 20) ? s : (1u << 20);
    }
    size_t idle_sum(int device) const {
        size_t n = 0;
        for (const Block& b : idle) n += b.device == device ? b.bytes : 0;
        return n;
    }
    size_t drop(int device) {
        size_t n = 0;
        for (size_t i = idle.size(); i-- > 0;)
            if (idle[i].device == device) {
                n += idle[i].bytes;
                Mem::free(idle[i].p);
                idle.erase(idle.begin() + i);
            }
        return n;
    }
    int alloc_locked(int device, void** p, size_t bytes) {
        int e = Mem::alloc(p, bytes);
        if (e && drop(device)) e = Mem::alloc(p, bytes);
        return e;
    }

  public:
    // A block of the current device.
    int get(void** p, size_t bytes) {
        const int device = Mem::device();
        if (device < 0) return -device;
        std::lock_guard<std::mutex> lk(mu);
        size_t best = idle.size();        // the smallest idle block that holds it
        for (size_t i = 0; i < idle.size(); ++i)
            if (idle[i].device == device && idle[i].bytes >= bytes && idle[i].bytes - bytes <= slack(bytes) &&
                (best == idle.size() || idle[i].bytes < idle[best].bytes))
                best = i;
        if (best < idle.size()) {
            used.push_back(idle[best]);
            idle.erase(idle.begin() + best);
        } else {
            void* q = nullptr;
            if (int e = alloc_locked(device, &q, bytes)) return e;
            used.push_back({q, bytes, device});
        }
        *p = used.back().p;
        return 0;
    }
    // Its return, once no stream uses it.
    void put(void* p) {
        std::lock_guard<std::mutex> lk(mu);
        for (size_t i = 0; i < used.size(); ++i) {
            if (used[i].p != p) continue;
            const Block b = used[i];
            used.erase(used.begin() + i);
            const size_t limit = Mem::total(b.device) / 4;
            if (b.bytes > limit) {
                Mem::free(b.p);
                return;
            }
            size_t sum = idle_sum(b.device);
            for (size_t k = 0; k < idle.size() && sum + b.bytes > limit;) {
                if (idle[k].device != b.device) { ++k; continue; }
                sum -= idle[k].bytes;
                Mem::free(idle[k].p);
                idle.erase(idle.begin() + k);
            }
            idle.push_back(b);
            return;
        }
    }
    // An allocation that is not the pool's, on the current device: where it
    // fails, idle blocks may be in the way and are given back first.
    int alloc(void** p, size_t bytes) {
        int e = Mem::alloc(p, bytes);
        if (!e) return 0;
        const int device = Mem::device();
        if (device < 0) return e;
        std::lock_guard<std::mutex> lk(mu);
        drop(device);                     // another thread may have done so: tried again all the same
        return Mem::alloc(p, bytes);
    }
    // Gives a device's idle blocks back; their bytes.
    size_t release(int device) {
        std::lock_guard<std::mutex> lk(mu);
        return drop(device);
    }
    size_t idle_bytes(int device) {
        std::lock_guard<std::mutex> lk(mu);
        return idle_sum(device);
    }
    // A context of the device begins (+1) or ends (-1).
    void context(int device, int step) {
        std::lock_guard<std::mutex> lk(mu);
        if ((int)contexts.size() <= device) contexts.resize(device + 1, 0);
        contexts[device] += step;
        if (contexts[device] <= 0) drop(device);
    }
};

}  // namespace polyeri
