/*
 * stc_serve.h — the state that query batches read while steps go on, and the
 * leases on it. Host code alone, without HIP.
 *
 * A batch takes a lease: a copy of the published state, whose arrays stay as
 * they are until the lease is given back. The stepping thread overwrites and
 * frees arrays that a published state may name (the meeting arrays, the
 * memtable, the runs). The one order that is safe, whenever a batch comes:
 *   1. the published state stops naming the array (publish, amend, clear),
 *   2. the leases taken before that end,
 *   3. the array is overwritten or freed.
 * Waiting first and publishing afterwards leaves a gap in which a new lease
 * names what is about to go.
 */
#ifndef STC_SERVE_H_
#define STC_SERVE_H_

#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <utility>
#include <vector>

template <class State>
class Published {
  public:
    struct Lease {
        State state;
        int meet = 0;               /* the meeting array it reads */
        uint32_t epoch = 0;         /* the memtable epoch: +1 at every flush */
        uint64_t version = 0;
    };

    /* false: nothing is published */
    bool take(Lease *l) {
        std::lock_guard<std::mutex> lk(mu);
        if (!valid) return false;
        *l = now;
        open.push_back(OpenLease{now.version, now.meet, now.epoch});
        return true;
    }
    void give_back(const Lease &l) {
        {
            std::lock_guard<std::mutex> lk(mu);
            for (size_t i = 0; i < open.size(); i++)
                if (open[i].version == l.version) {
                    open[i] = open.back();
                    open.pop_back();
                    break;
                }
        }
        ended.notify_all();
    }

    void publish(State st, int meet, uint32_t epoch, bool any) {
        std::lock_guard<std::mutex> lk(mu);
        now = Lease{std::move(st), meet, epoch, now.version + 1};
        valid = any;
    }

    /* f(State &) on the state of the leases from now on, then (once those taken before have ended) gone() */
    template <class F, class G>
    void replace(F f, G gone) {
        {
            std::lock_guard<std::mutex> lk(mu);
            now.version++;
            f(now.state);
        }
        wait_earlier();
        gone();
    }

    /* meeting array `meet` is about to be overwritten or freed and, with `memtable`, the records of an epoch before
     * `epoch` are: no lease reads them when this returns, and none will until the next publish. A state that still
     * names them (its step's successor failed half way) is withdrawn. */
    void clear(int meet, bool memtable, uint32_t epoch) {
        std::unique_lock<std::mutex> lk(mu);
        if (now.meet == meet || (memtable && now.epoch != epoch)) valid = false;
        ended.wait(lk, [&] {
            for (const OpenLease &l : open)
                if (l.meet == meet || (memtable && l.epoch != epoch)) return false;
            return true;
        });
    }

    /* until the leases on states before the present one have ended */
    void wait_earlier() {
        std::unique_lock<std::mutex> lk(mu);
        const uint64_t v = now.version;
        ended.wait(lk, [&] {
            for (const OpenLease &l : open)
                if (l.version < v) return false;
            return true;
        });
    }
    /* until no lease is open */
    void wait_all() {
        std::unique_lock<std::mutex> lk(mu);
        ended.wait(lk, [&] { return open.empty(); });
    }

    /* for the thread that publishes alone */
    const State &state() const { return now.state; }

  private:
    struct OpenLease { uint64_t version; int meet; uint32_t epoch; };
    std::mutex mu;
    std::condition_variable ended;
    Lease now;
    bool valid = false;
    std::vector<OpenLease> open;
};

#endif /* STC_SERVE_H_ */
