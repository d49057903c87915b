// Internal: the object behind HEaaN::Context (parameters, per-level scales, encoding tables and the
// device-buffer pool).  Not part of the public surface.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <condition_variable>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "../../../include/hemm.h"
#include "HEaaN/HEaaN.hpp"

namespace HEaaN {

// A device buffer that was given up, with the readings of Recordings::now() when it was handed out and when it was given up.
struct Freed {
    size_t words;
    u64 *ptr, born, freed;
};
// Recorded sequences (hellm_graph_begin / _end) replay on the addresses they were recorded with: masks, tables and keys that were there
// already, whoever holds them and on whichever context they were made.  A buffer that was there while a recording was open may be one
// of its addresses; once given up it is kept from reuse for as long as that recording lives.
class Recordings {
public:
    static Recordings &all() {
        static Recordings *r = new Recordings;   // (outlives every buffer, static ones among them)
        return *r;
    }
    u64 now() const { return now_; }   // counts openings and closings
    u64 open() {
        std::lock_guard<std::mutex> lk(mu_);
        const u64 id = ++now_;
        closed_[id] = ~u64(0);
        living_ = closed_.size();
        return id;
    }
    void close(u64 id) {
        std::lock_guard<std::mutex> lk(mu_);
        closed_[id] = ++now_;
    }
    void drop(u64 id) {
        std::vector<Freed> rest;
        {
            std::lock_guard<std::mutex> lk(mu_);
            closed_.erase(id);
            living_ = closed_.size();
            rest.swap(orphans_);
            dropped_++;
        }
        for (const Freed &f : rest) leave(f);
    }
    u64 dropped() const { return dropped_; }
    bool need(const Freed &f) {
        if (living_ == 0) return false;
        std::lock_guard<std::mutex> lk(mu_);
        return needLocked(f);
    }
    // memory whose context is gone
    void leave(const Freed &f) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (needLocked(f)) {
                orphans_.push_back(f);
                return;
            }
        }
        (void)hipFree(f.ptr);
    }

private:
    bool needLocked(const Freed &f) const {
        for (const auto &r : closed_)
            if (r.first <= f.freed && r.second > f.born) return true;
        return false;
    }
    std::mutex mu_;
    std::map<u64, u64> closed_;   // living recordings: when opened -> when closed
    std::vector<Freed> orphans_;
    std::atomic<u64> now_{0}, dropped_{0};
    std::atomic<size_t> living_{0};
};

struct ContextContent {
    hemm_context *dev = nullptr;
    u64 logN = 0, N = 0, nQ = 0, nP = 0, dnum = 0, alpha = 0, log_scale = 42;
    std::vector<u64> q, p;
    std::vector<Real> delta;             // fixed scale of each level
    std::vector<u64> rot_group;          // 5^j mod 2N
    std::vector<double> ksi_re, ksi_im;  // exp(2 pi i k / 2N)
    // Freed buffers are kept by size and handed out again: kernels run on the default stream, so reuse is
    // ordered after the last use without any synchronisation.  The one exception is a side chain (forkSide /
    // joinSide below): while it is open, freed buffers are parked and only return to the pool at the join.
    std::multimap<size_t, u64 *> pool;
    std::vector<Freed> parked;
    std::vector<Freed> held;   // released, but a recording may replay on them
    u64 held_since = 0;        // Recordings::dropped() when they were last looked at
    std::mutex mu;
    size_t pool_bytes = 0;
    hipStream_t side = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr, ev_main = nullptr, ev_side = nullptr;
    bool side_open = false;
    // the stream the host layer queues on: the device context's (hemm_context_set_stream), by default the legacy
    // default stream; on(s) resolves a stream argument whose null value means that stream
    hipStream_t stream() const { return (hipStream_t)hemm_context_stream(dev); }
    hipStream_t on(hipStream_t s) const { return s != nullptr ? s : stream(); }

    // Opens a side chain: work given to the returned stream starts after everything queued on the default stream
    // so far and runs beside what the default stream is given next.  The stream does not synchronise implicitly
    // with the default stream; joinSide() makes the default stream wait for it.  Default priority.
    hipStream_t forkSide() {
        if (side_open) throw RuntimeException("side chain already open");
        auto ok = [](hipError_t e, const char *what) {
            if (e != hipSuccess) throw RuntimeException(std::string(what) + ": " + hipGetErrorString(e));
        };
        if (!side) {
            ok(hipStreamCreateWithFlags(&side, hipStreamNonBlocking), "hipStreamCreateWithFlags");
            ok(hipEventCreateWithFlags(&ev_fork, hipEventDisableTiming), "hipEventCreateWithFlags");
            ok(hipEventCreateWithFlags(&ev_join, hipEventDisableTiming), "hipEventCreateWithFlags");
            ok(hipEventCreateWithFlags(&ev_main, hipEventDisableTiming), "hipEventCreateWithFlags");
            ok(hipEventCreateWithFlags(&ev_side, hipEventDisableTiming), "hipEventCreateWithFlags");
        }
        ok(hipEventRecord(ev_fork, stream()), "hipEventRecord");
        ok(hipStreamWaitEvent(side, ev_fork, 0), "hipStreamWaitEvent");
        std::lock_guard<std::mutex> lk(mu);
        side_open = true;
        return side;
    }
    // While a side chain is open, the two streams can also wait for each other half way without closing it:
    // sideWaitsForMain() orders what the side stream is given next after everything queued on the default stream so
    // far; markSide() notes the side stream's position and waitSideMark() makes the default stream wait for the last
    // such note (work queued on the side stream after the note is not waited for).
    void sideWaitsForMain() {
        if (!side_open) throw RuntimeException("no side chain open");
        (void)hipEventRecord(ev_main, stream());
        (void)hipStreamWaitEvent(side, ev_main, 0);
    }
    void markSide() {
        if (!side_open) throw RuntimeException("no side chain open");
        (void)hipEventRecord(ev_side, side);
    }
    void waitSideMark() {
        if (!side_open) throw RuntimeException("no side chain open");
        (void)hipStreamWaitEvent(stream(), ev_side, 0);
    }
    void joinSide() {
        if (!side_open) return;
        (void)hipEventRecord(ev_join, side);
        (void)hipStreamWaitEvent(stream(), ev_join, 0);
        std::lock_guard<std::mutex> lk(mu);
        side_open = false;
        for (const Freed &f : parked) reuse(f);
        parked.clear();
    }

    // Optional phase trace of the batched products: while it is on, mark() records an event on the default stream at
    // a named point of the schedule; the report gives the time between consecutive marks.
    bool trace_on = false;
    std::vector<std::pair<std::string, hipEvent_t>> trace_marks;
    void mark(const char *name) {
        if (!trace_on) return;
        hipEvent_t e = nullptr;
        if (hipEventCreate(&e) != hipSuccess) return;
        (void)hipEventRecord(e, stream());
        trace_marks.emplace_back(name, e);
    }
    void traceClear() {
        for (auto &m : trace_marks) (void)hipEventDestroy(m.second);
        trace_marks.clear();
    }

    // Pinned host memory for the values of STAGES messages ([N/2] doubles each), which kernels read and write in place: a
    // transfer needs no copy command and no pageable staging.  One allocation on first use (it costs what one for a single message
    // does), kept for the context's life.  A user holds a stage from takeStage() to giveStage(); `queued` says that work on
    // `stream` still reads it, which the next user waits for: a queue of messages waits for the GPU once it holds STAGES of them.
    struct Stage {
        double *values = nullptr;
        hipEvent_t done = nullptr;
        bool pending = false;
    };
    static constexpr size_t STAGES = 8;
    double *stage_memory = nullptr;
    std::vector<Stage> stages;          // free ones, the longest unused first
    std::condition_variable stage_free;
    Stage takeStage() {
        std::unique_lock<std::mutex> lk(mu);
        if (stage_memory == nullptr) {
            std::vector<Stage> made(STAGES);
            bool ok = hipHostMalloc((void **)&stage_memory, STAGES * (N / 2) * sizeof(double)) == hipSuccess;
            for (size_t i = 0; ok && i < STAGES; i++) {
                made[i].values = stage_memory + i * (N / 2);
                ok = hipEventCreateWithFlags(&made[i].done, hipEventDisableTiming) == hipSuccess;
            }
            if (!ok) {
                for (Stage &s : made)
                    if (s.done) (void)hipEventDestroy(s.done);
                if (stage_memory) (void)hipHostFree(stage_memory);
                stage_memory = nullptr;
                throw RuntimeException("no pinned memory for the values of messages");
            }
            stages = std::move(made);
        }
        stage_free.wait(lk, [&] { return !stages.empty(); });
        Stage s = stages.front();
        stages.erase(stages.begin());
        lk.unlock();
        if (s.pending && hipEventQuery(s.done) != hipSuccess) {   // (a query of one long since reached is cheaper than a wait)
            (void)hipGetLastError();   // "not ready" is an answer here, not an error for the next launch to report
            (void)hipEventSynchronize(s.done);
        }
        s.pending = false;
        return s;
    }
    void giveStage(Stage s, bool queued) {
        if (queued && !(s.pending = hipEventRecord(s.done, stream()) == hipSuccess)) (void)hipStreamSynchronize(stream());
        {
            std::lock_guard<std::mutex> lk(mu);
            stages.push_back(s);
        }
        stage_free.notify_one();
    }

    u64 prime(size_t i) const { return i < nQ ? q[i] : p[i - nQ]; }
    u64 *alloc(size_t words) {
        {
            std::lock_guard<std::mutex> lk(mu);
            if (!held.empty() && held_since != Recordings::all().dropped()) {
                std::vector<Freed> all;
                all.swap(held);
                held_since = Recordings::all().dropped();
                for (const Freed &f : all) reuse(f);
            }
            auto it = pool.find(words);
            if (it != pool.end()) {
                u64 *r = it->second;
                pool.erase(it);
                return r;
            }
        }
        u64 *d = nullptr;
        hipError_t e = hipMalloc((void **)&d, words * sizeof(u64));
        if (e != hipSuccess) throw RuntimeException(std::string("hipMalloc: ") + hipGetErrorString(e));
        pool_bytes += words * 8;
        return d;
    }
    // Stream capture of a sequence of calls (hellm_graph_begin / _end): a buffer released while the capture is open
    // stays with the graph being recorded -- its replays write that memory -- and returns to the pool when the graph
    // is destroyed.
    bool capture_open = false;
    std::vector<Freed> captured;
    void release(u64 *ptr, size_t words, u64 born) {
        std::lock_guard<std::mutex> lk(mu);
        const Freed f{words, ptr, born, Recordings::all().now()};
        if (capture_open)
            captured.push_back(f);
        else if (side_open)
            parked.push_back(f);
        else
            reuse(f);
    }
    void reuse(const Freed &f) {   // (with mu held)
        if (Recordings::all().need(f))
            held.push_back(f);
        else
            pool.emplace(f.words, f.ptr);
    }
    ~ContextContent() {
        (void)hipDeviceSynchronize();
        traceClear();
        for (auto &kv : pool) (void)hipFree(kv.second);
        for (const std::vector<Freed> *l : {&parked, &held, &captured})
            for (const Freed &f : *l) Recordings::all().leave(f);
        for (auto &st : stages) (void)hipEventDestroy(st.done);
        if (stage_memory) (void)hipHostFree(stage_memory);
        if (side) (void)hipStreamDestroy(side);
        if (ev_fork) (void)hipEventDestroy(ev_fork);
        if (ev_join) (void)hipEventDestroy(ev_join);
        if (ev_main) (void)hipEventDestroy(ev_main);
        if (ev_side) (void)hipEventDestroy(ev_side);
        if (dev) hemm_context_destroy(dev);
    }
};

// a stage for as long as the object lives; read(): queued work reads it, so the next user has to wait for that
class HostStage {
  public:
    explicit HostStage(const Context &c) : c_(c), s_(c->takeStage()) {}
    ~HostStage() { c_->giveStage(s_, queued_); }
    HostStage(const HostStage &) = delete;
    HostStage &operator=(const HostStage &) = delete;
    double *values() const { return s_.values; }
    void read() { queued_ = true; }

  private:
    Context c_;
    ContextContent::Stage s_;
    bool queued_ = false;
};
// whether messages of this context go through a stage (a sequence being recorded reads its own copy: a replay would find
// another message in the stage)
inline bool stageable(const Context &c) { return c->logN >= 10 && !c->capture_open; }

}  // namespace HEaaN
