/*
 * stc_wait.h — waiting for what arrives within microseconds. Host code alone,
 * without HIP.
 */
#ifndef STC_WAIT_H_
#define STC_WAIT_H_

#include <chrono>
#include <sched.h>

/* Looks for `there` (a bool()) for at most so long: every few tens of nanoseconds, and the core is offered to another
 * thread every ten microseconds or so. Without the offer the threads of a batch of streams that wait would keep off the
 * core those that have something to launch, where there are fewer cores than threads (16 streams on one core: 5.2 ms,
 * 4.1 to 4.9 so; on four 3.1 and 2.9; on 16 the same). */
template <class F>
inline bool look_for(F there, std::chrono::microseconds most) {
    const auto until = std::chrono::steady_clock::now() + most;
    do {
        for (int k = 0; k < 256; k++) {
            if (there()) return true;
            __builtin_ia32_pause();
        }
        sched_yield();
    } while (std::chrono::steady_clock::now() < until);
    return false;
}

#endif /* STC_WAIT_H_ */
