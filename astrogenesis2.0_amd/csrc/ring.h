// A flat block that travels between the caller's arrays and a device piece by
// piece through a ring of staging slots, host threads moving the pieces
// between slots and arrays while the next ones are under way.  Host code only
// (transfer.hip supplies the device, the CPU build one of memory copies).
#pragma once

#include <atomic>
#include <chrono>
#include <cstddef>
#include <cstring>
#include <functional>
#include <thread>
#include <vector>

namespace ag2 {

// The caller's side of a flat block: consecutive runs of bytes.
struct Run {
    char *host;
    size_t bytes;
};

// Copies [at, at + len) of the block between `buf` and the runs.
inline void move_runs(const std::vector<Run> &runs, size_t at, size_t len, char *buf, bool to_runs) {
    size_t lo = 0;
    for (const Run &r : runs) {
        const size_t hi = lo + r.bytes;
        if (hi > at && lo < at + len) {
            const size_t a = lo > at ? lo : at, b = hi < at + len ? hi : at + len;
            if (to_runs) std::memcpy(r.host + (a - lo), buf + (a - at), b - a);
            else std::memcpy(buf + (a - at), r.host + (a - lo), b - a);
        }
        lo = hi;
        if (lo >= at + len) break;
    }
}

// A staging buffer, taken for a transfer and given back after it.  A transfer
// that ends early (no call of whole()) may leave copies under way in the
// buffer: those are waited for, and the buffer is not kept for others.
//   take()      a buffer (may throw)
//   drain()     wait for the copies queued so far, whatever became of them
//   keep(b)     keep it for a later transfer, if there is room
//   destroy(b)
template <class Buffer, class Ops>
class Lease {
  public:
    explicit Lease(Ops ops) : ops_(ops), buffer(ops_.take()) {}
    ~Lease() {
        if (!whole_) ops_.drain();
        if (!whole_ || !ops_.keep(buffer)) ops_.destroy(buffer);
    }
    void whole() { whole_ = true; }   // every copy of the transfer has completed
    Lease(const Lease &) = delete;
    Lease &operator=(const Lease &) = delete;

  private:
    Ops ops_;
    bool whole_ = false;

  public:
    Buffer buffer;
};

// The device's side, called by the caller's thread alone; each may throw.
//   issue(p)  queue the copy of piece p between the block and its slot
//   wait(p)   return when it has completed
//   left(p)   has it completed?
// The caller's thread takes host-side pieces itself where it would wait for a
// helper.  Helpers sleep while there is no piece to take (a spinning one would
// compete with the caller's program for its share of the host).  The caller
// alone is enough: where a thread cannot be had, those that were do.  An error
// of the device goes up from run(), and the destructor then stops the helpers.
template <class Device>
class Ring {
  public:
    // start(f): a thread that runs f (throws where there is none to be had)
    Ring(Device &device, char *slots, int n_slots, size_t piece, const std::vector<Run> &r, size_t total,
         bool to_host, int helpers,
         const std::function<std::thread(std::function<void()>)> &start =
             [](std::function<void()> f) { return std::thread(std::move(f)); })
        : dev_(device), slots_(slots), ring_(n_slots), piece_(piece), runs_(r), bytes_(total), down_(to_host),
          pieces_((int)((total + piece - 1) / piece)), done_((size_t)pieces_) {
        open_ = down_ ? 0 : (pieces_ < ring_ ? pieces_ : ring_);
        try {
            th_.reserve((size_t)helpers);
            for (int k = 0; k < helpers; k++) th_.push_back(start([this] { help(); }));
        } catch (...) {
        }
    }
    ~Ring() {
        if (next_ < pieces_) bad_ = 1;   // left by an error
        for (auto &t : th_) t.join();
    }
    Ring(const Ring &) = delete;
    Ring &operator=(const Ring &) = delete;
    size_t off(int p) const { return (size_t)p * piece_; }
    size_t len(int p) const { return bytes_ - off(p) < piece_ ? bytes_ - off(p) : piece_; }
    char *slot(int p) const { return slots_ + (size_t)(p % ring_) * piece_; }
    int helpers() const { return (int)th_.size(); }

    void run() {
        int issued = 0, landed = 0;
        if (down_) {
            while (landed < pieces_) {
                while (issued < pieces_ && (issued < ring_ || done_[(size_t)(issued - ring_)])) dev_.issue(issued++);
                if (landed < issued) {
                    dev_.wait(landed);
                    open_ = ++landed;
                } else {
                    take_or_pause();
                }
            }
        } else {
            while (issued < pieces_) {
                if (done_[(size_t)issued]) dev_.issue(issued++);
                else take_or_pause();
                // slots whose copy has left are open again
                while (landed < issued && dev_.left(landed)) landed++;
                const int o = landed + ring_ < pieces_ ? landed + ring_ : pieces_;
                if (o > open_) open_ = o;
            }
        }
        while (next_ < pieces_) take_or_pause();
        for (auto &t : th_) t.join();
        th_.clear();
    }

  private:
    // The host side of one open piece, if there is one to take.
    bool take() {
        int p = next_;
        while (p < open_)
            if (next_.compare_exchange_weak(p, p + 1)) {
                move_runs(runs_, off(p), len(p), slot(p), down_);
                done_[(size_t)p] = 1;
                return true;
            }
        return false;
    }
    void help() {
        while (!bad_ && next_ < pieces_)
            if (!take()) std::this_thread::sleep_for(std::chrono::microseconds(20));
    }
    void take_or_pause() {
        if (!take()) __builtin_ia32_pause();
    }

    Device &dev_;
    char *slots_;
    const int ring_;
    const size_t piece_;
    const std::vector<Run> &runs_;
    const size_t bytes_;
    const bool down_;
    const int pieces_;
    std::vector<std::atomic<int>> done_;   // the host side of the piece is finished
    std::atomic<int> next_{0};             // pieces taken for their host side
    std::atomic<int> open_{0};             // pieces whose host side may start
    std::atomic<int> bad_{0};
    std::vector<std::thread> th_;
};

}  // namespace ag2
