// Messages from the GPU to the host inside a loop: a few values in pinned host
// memory, then the number of the message.  The host reads a message as soon as
// its number arrives, where a copy and a stream synchronisation would leave
// the GPU idle until the host has woken up and launched the next work.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>

namespace bx {

struct Mail
{
    double             v[4];
    unsigned long long seq;
};

// Message `seq` goes to slot seq % MAIL_SLOTS, so a message stays readable
// while the next MAIL_SLOTS - 1 are posted.
constexpr int MAIL_SLOTS = 16;

__device__ __forceinline__ void mail_post(Mail *slots, unsigned long long seq, double v0,
                                          double v1 = 0.0)
{
    Mail &m = slots[seq % MAIL_SLOTS];
    m.v[0]  = v0;
    m.v[1]  = v1;
    __threadfence_system();
    __hip_atomic_store(&m.seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The host's side: pinned slots and their device address.
struct MailBox
{
    Mail              *slots = nullptr, *dev = nullptr;
    unsigned long long seq = 0; // the last message asked for

    hipError_t open()
    {
        hipError_t e = hipHostMalloc((void **)&slots, sizeof(Mail) * MAIL_SLOTS,
                                     hipHostMallocMapped | hipHostMallocCoherent);
        if (e != hipSuccess)
        {
            slots = nullptr;
            return e;
        }
        for (int k = 0; k < MAIL_SLOTS; ++k)
            slots[k] = Mail();
        e = hipHostGetDevicePointer((void **)&dev, slots, 0);
        if (e != hipSuccess)
            close(); // open or closed, nothing between: kernels post to dev
        return e;
    }
    void close()
    {
        if (slots)
            (void)hipHostFree(slots);
        slots = dev = nullptr;
    }
    bool arrived(unsigned long long n) const
    {
        const volatile unsigned long long *p = &slots[n % MAIL_SLOTS].seq;
        if (*p != n)
            return false;
        std::atomic_thread_fence(std::memory_order_acquire);
        return true;
    }
    const Mail &operator[](unsigned long long n) const { return slots[n % MAIL_SLOTS]; }

    // Waits for message n, posted by a kernel already launched on s: a
    // bounded spin, then the stream's synchronisation, which also reports a
    // failed launch or kernel.  Work launched on s before the kernel that
    // posts the message has completed when it arrives.
    hipError_t wait(unsigned long long n, hipStream_t s) const
    {
        hipError_t e = hipGetLastError();
        if (e != hipSuccess)
            return e;
        const auto t0 = std::chrono::steady_clock::now();
        while (!arrived(n))
        {
            for (int k = 0; k < 64 && !arrived(n); ++k)
                __builtin_ia32_pause();
            if (std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(50))
            {
                if ((e = hipStreamSynchronize(s)) != hipSuccess)
                    return e;
                return arrived(n) ? hipSuccess : hipErrorUnknown;
            }
        }
        return hipSuccess;
    }
};

} // namespace bx
