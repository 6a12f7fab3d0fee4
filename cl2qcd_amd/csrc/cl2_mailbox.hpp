// Scalars on their way to the host through pinned memory that a kernel writes (cl2_scalar_get).  Host code only.
#pragma once

#include <chrono>
#include <cstdint>
#include <cstring>
#include <mutex>

/* the values, then the number of the transfer they belong to */
struct cl2_mailbox {
    static constexpr int SIZE = 64;
    double value[SIZE];
    uint64_t number;
};

/* The host's end.  Transfers are numbered here and not from what the box holds: after a wait that failed the box may
 * still get that transfer, which must not pass for the next one. */
class cl2_mail_reader {
  public:
    cl2_mailbox* box = nullptr;

    /* the box, from allocate() at the first call that gets one; false without one */
    template<typename Allocate>
    bool open(Allocate&& allocate)
    {
        std::lock_guard<std::mutex> one_at_a_time(mutex_);
        if (!box) box = allocate();
        return box != nullptr;
    }

    /* n <= SIZE values into host: send(number) enqueues the transfer, and where it has not come within a millisecond
     * wait() waits for everything enqueued; both return 0 or an error, which ends the read */
    template<typename Send, typename Wait>
    auto read(double* host, int n, Send&& send, Wait&& wait) -> decltype(wait())
    {
        std::lock_guard<std::mutex> one_at_a_time(mutex_);
        const uint64_t number = ++last_;
        if (auto e = send(number)) return e;
        const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
        while (__atomic_load_n(&box->number, __ATOMIC_ACQUIRE) != number)
            if (std::chrono::steady_clock::now() > until) {
                if (auto e = wait()) return e;
                break;
            }
        std::memcpy(host, box->value, n * sizeof(double));
        return decltype(wait())(0);
    }

  private:
    uint64_t last_ = 0;
    std::mutex mutex_;
};
