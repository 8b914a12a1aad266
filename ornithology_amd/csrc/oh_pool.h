// oh_pool.h - device memory blocks kept between their users. The device's
// memory calls are passed in, so this header holds no HIP.
//
// A session's buffers are parts of two or three blocks, and a closed session's
// blocks serve the next session: a block of up to half again the size asked
// for (and 1 MiB) is taken. Opening and closing a session allocated and freed
// about 200 buffers before: a 4096-token request on 40 layers 131.5 -> 101.8 ms
// with the pool, 1003 tokens on four layers 11.3 -> 4.1 ms.
#pragma once
#include <cstddef>
#include <mutex>

struct DevBlock {
    void *p = nullptr;
    size_t n = 0;
    const void *owner = nullptr;          // whom it served last (a model; null: none in particular)
};

// The memory calls of a device.
struct DevMem {
    int (*alloc)(void **p, size_t n);     // 0, or the runtime's status
    void (*release)(void *p);
    size_t (*unused)(int device);         // bytes of the device that nobody holds
};

class DevPool {
public:
    // What a pool holds at most (a 4096-token prompt's buffers of the 35B shape
    // take 1.5 GB), and at most this share of the memory that is not in use
    // otherwise: other users of the device see what is held as taken. Beyond it
    // the blocks unused for longest are given back: sizes that no longer occur
    // make room for those that do. The device is asked when the pool would grow
    // past what the last answer allowed, after an allocation of the pool's own
    // and every kAsk blocks: asking each time took 12 us a block (a small encode
    // 117 -> 130 us).
    static constexpr size_t kBytes = (size_t)4 << 30, kShare = 16;
    static constexpr int kBlocks = 64, kAsk = 64;

    DevPool(const DevMem &mem, int device) : mem_(mem), device_(device) {
        std::lock_guard<std::mutex> lk(all_mu());
        next_ = all();
        all() = this;
    }
    ~DevPool() {
        {
            std::lock_guard<std::mutex> lk(all_mu());
            DevPool **p = &all();
            while (*p != this) p = &(*p)->next_;
            *p = next_;
        }
        trim();
    }
    DevPool(const DevPool &) = delete;
    DevPool &operator=(const DevPool &) = delete;

    // n bytes of device memory; when the device is out of it, once more after
    // the blocks of all of the device's pools are given back
    int alloc(void **p, size_t n) {
        int e = mem_.alloc(p, n);
        if (e != 0) {
            {
                std::lock_guard<std::mutex> lk(all_mu());
                for (DevPool *q = all(); q; q = q->next_)
                    if (q->device_ == device_) q->trim();
            }
            e = mem_.alloc(p, n);
        }
        std::lock_guard<std::mutex> lk(mu_);
        stale_ = true;                        // there is less now
        return e;
    }
    // a block of at least n bytes (contents undefined) from the pool or the device
    int get(size_t n, DevBlock *b) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            int best = -1;
            for (int i = 0; i < count_; i++) {
                const size_t z = held_[i].n;
                if (z >= n && z - n <= n / 2 + ((size_t)1 << 20) && (best < 0 || z < held_[best].n)) best = i;
            }
            if (best >= 0) {
                *b = take(best);
                return 0;
            }
        }
        b->n = n;
        return alloc(&b->p, n);
    }
    // the block back to the pool, or to the device when the pool may not be
    // that large
    void put(const DevBlock &b) {
        DevBlock old[kBlocks + 1];
        int n = 0;
        bool ask;
        {
            std::lock_guard<std::mutex> lk(mu_);
            ask = stale_ || bytes_ + b.n > most_ || ++puts_ >= kAsk;
        }
        const size_t unused = ask ? mem_.unused(device_) : 0;
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (ask) {
                const size_t share = (unused + bytes_ + b.n) / kShare;
                most_ = share < kBytes ? share : kBytes;
                puts_ = 0;
                stale_ = false;
            }
            const bool keep = b.n <= most_;
            while ((keep && count_ == kBlocks) || (count_ > 0 && bytes_ + (keep ? b.n : 0) > most_)) old[n++] = take(0);
            if (keep) {
                held_[count_++] = b;
                bytes_ += b.n;
            } else {
                old[n++] = b;
            }
        }
        for (int i = 0; i < n; i++) mem_.release(old[i].p);
    }
    // all blocks back to the device, or those that served owner last; the bytes
    // they held
    size_t trim(const void *owner = nullptr) {
        DevBlock old[kBlocks];
        int n = 0;
        size_t bytes = 0;
        {
            std::lock_guard<std::mutex> lk(mu_);
            for (int i = count_ - 1; i >= 0; i--)
                if (!owner || held_[i].owner == owner) old[n++] = take(i);
        }
        for (int i = 0; i < n; i++) {
            bytes += old[i].n;
            mem_.release(old[i].p);
        }
        return bytes;
    }

private:
    // the process's pools
    static DevPool *&all() { static DevPool *head = nullptr; return head; }
    static std::mutex &all_mu() { static std::mutex m; return m; }

    // held_[i] out of the pool (mu_ held)
    DevBlock take(int i) {
        const DevBlock b = held_[i];
        bytes_ -= b.n;
        for (count_--; i < count_; i++) held_[i] = held_[i + 1];
        return b;
    }

    DevMem mem_;
    int device_;
    DevPool *next_ = nullptr;
    std::mutex mu_;
    DevBlock held_[kBlocks];              // unused for longest first
    int count_ = 0;
    size_t bytes_ = 0;
    size_t most_ = 0;                     // what bytes_ may be, by the device's last answer
    bool stale_ = true;                   // it has to be asked again
    int puts_ = 0;                        // blocks returned since
};
