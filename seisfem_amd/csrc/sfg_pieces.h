// Pieces of a transfer, moved by several threads (plain C++: the transfer itself is
// behind PiecePort).
#pragma once
#include <atomic>
#include <cstddef>
#include <exception>
#include <thread>

namespace sfg {

// One thread's side of a transfer.  Each thread has two buffers; piece p is queued into
// one of them, waited for, and taken out of it.  Calls return 0 or an error code.
struct PiecePort {
    virtual ~PiecePort() = default;
    virtual int open(int thread) = 0;                            // on the thread, before its pieces
    virtual int issue(int thread, int buffer, size_t piece) = 0; // queues the piece
    virtual int wait(int thread, int buffer) = 0;                // until the piece has arrived
    virtual void take(int thread, int buffer, size_t piece) = 0; // copies it to its place
    virtual void close(int thread) = 0;                          // after its pieces, whatever open returned
};

// Moves pieces 0 .. pieces - 1 with up to `threads` threads, the caller among them; a
// thread has one piece on its way while it copies another.  Returns 0 when every piece has
// been taken, else the first error that any call returned: from then on no thread queues
// another piece.
inline int deliver(PiecePort &port, size_t pieces, int threads)
{
    constexpr int MOST = 16;
    std::atomic<size_t> next{0};
    std::atomic<int> error{0};
    auto failed = [&](int e) {
        int none = 0;
        if (e) error.compare_exchange_strong(none, e);
        return e != 0;
    };
    auto work = [&](int q) {
        size_t piece[2] = {0, 0};
        bool have[2] = {false, false};           // on its way in each buffer
        auto issue = [&](int b) {
            have[b] = false;
            if (error.load()) return;
            piece[b] = next++;
            if (piece[b] < pieces) have[b] = !failed(port.issue(q, b, piece[b]));
        };
        if (!failed(port.open(q))) {
            issue(0);
            issue(1);
            for (int b = 0; have[0] || have[1]; b ^= 1) {
                if (!have[b]) continue;
                if (failed(port.wait(q, b))) break;
                port.take(q, b, piece[b]);
                issue(b);
            }
        }
        port.close(q);
    };
    std::thread th[MOST];
    int started = 1;
    try {
        for (; started < threads && started < MOST; ++started) th[started] = std::thread(work, started);
    } catch (const std::exception &) {
        // fewer helpers: the pieces are handed out as they are asked for
    }
    work(0);
    for (int q = 1; q < started; ++q) th[q].join();
    return error.load();
}

} // namespace sfg
