// Downloads of large results (see sfg_copy.h).
#include "sfg_copy.h"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <vector>

#include "sfg_pieces.h"

namespace sfg {

namespace {
constexpr int kThreads = 8;
constexpr size_t kPiece = (size_t)1 << 20;   // bytes of one transfer; two buffers per thread
// Downloads that have pinned buffers at a time (16 MB each, allocated when so many overlap);
// others are copied directly.  Threads that read back at the same time run side by side:
// with one set they took turns, and a small result waited for the largest (4.5 MB beside
// 131 MB 4.7 ms, with sets of their own 0.9; four threads of 131 MB each 17 ms, 15).
constexpr int kSets = 4;
// Results below kDirect are copied directly; those below kOne by the caller's thread alone,
// through a set if there is one (a new one costs its allocation, 20 us to a millisecond, and a
// page fault per 4 KB); larger ones by all threads.  us into memory in use / fresh memory,
// copied directly, through a set by one thread, by 8 threads: 16 KB 18 / 15, 12 / 14, 67 /
// 93; 128 KB 62 / 31, 14 / 30, 103 / 100; 1 MB 67 / 252, 61 / 244, 110 / 361; 4 MB 243 / 990,
// 220 / 940, 254 / 736; 16 MB 927 / 3699, 823 / 3557, 645 / 1185.
constexpr size_t kDirect = (size_t)64 << 10;
constexpr size_t kOne = (size_t)4 << 20;
std::mutex g_mu;
std::weak_ptr<Staging> g_staging;
} // namespace

// Sets of pinned buffers, each used by one download at a time
struct Staging {
    struct Set {
        std::mutex mu;                       // held by the download that uses it
        char *buf = nullptr;
        bool tried = false;
        // the buffers, locked by lk until the download ends; null: in use, no memory, or (make
        // false) not allocated yet
        char *take(std::unique_lock<std::mutex> &lk, bool make)
        {
            lk = std::unique_lock<std::mutex>(mu, std::try_to_lock);
            if (!lk.owns_lock()) return nullptr;
            if (make && !tried) {
                tried = true;
                if (hipHostMalloc((void **)&buf, 2 * kThreads * kPiece, hipHostMallocPortable) != hipSuccess) {
                    (void)hipGetLastError();
                    buf = nullptr;
                }
            }
            return buf;
        }
    } sets[kSets];
    // pinned memory for a result of so many bytes (null: none)
    char *get(std::unique_lock<std::mutex> &lk, size_t bytes)
    {
        if (bytes < kDirect) return nullptr;
        for (Set &x : sets)
            if (char *b = x.take(lk, bytes >= kOne)) return b;
        return nullptr;
    }
    ~Staging()
    {
        for (Set &x : sets)
            if (x.buf) (void)hipHostFree(x.buf);
    }
};

std::shared_ptr<Staging> staging()
{
    std::lock_guard<std::mutex> lk(g_mu);
    std::shared_ptr<Staging> s = g_staging.lock();
    if (!s) {
        s = std::make_shared<Staging>();
        g_staging = s;
    }
    return s;
}

// One transfer, whatever the number of rows: rows in a pitch come over with what lies
// between them and are copied apart here (a 2D copy into pageable memory moves row by row,
// 7 us each: 1024 rows of 52 bytes 7.0 ms against 0.04).  buf: pinned memory of that size, or null.
static hipError_t in_one(char *dst, const char *src, size_t pitch, size_t width, size_t rows, const int *map,
                         hipStream_t st, char *buf, std::vector<char> *scratch)
{
    const size_t bytes = (rows - 1) * pitch + width;
    const bool apart = map || pitch != width;
    std::vector<char> own;
    if (apart && !buf) {
        std::vector<char> &v = scratch ? *scratch : own;
        if (v.size() < bytes) v.resize(bytes);
        buf = v.data();
    }
    const hipError_t e = hipMemcpyWithStream(buf ? buf : dst, src, bytes, hipMemcpyDeviceToHost, st);
    if (e != hipSuccess) return e;
    if (!apart && buf) std::memcpy(dst, buf, bytes);
    for (size_t i = 0; apart && i < rows; ++i) std::memcpy(dst + (map ? (size_t)map[i] : i) * width, buf + i * pitch, width);
    return hipSuccess;
}

// The pieces of one download: parts of a row, or several whole rows
struct Download : PiecePort {
    hipDevice_t device = 0;
    hipStream_t st = nullptr;
    char *buf = nullptr, *to = nullptr;
    const char *from = nullptr;
    size_t pitch = 0, width = 0, rows = 0, per_row = 0, per_piece = 0;
    const int *map = nullptr;
    hipEvent_t done[kThreads][2] = {};

    char *buffer(int q, int b) const { return buf + (size_t)(2 * q + b) * kPiece; }
    size_t rows_of(size_t piece) const { return std::min(per_piece, rows - piece * per_piece); }
    size_t bytes_of(size_t piece) const { return std::min(kPiece, width - piece % per_row * kPiece); }

    int open(int q) override
    {
        hipError_t e = hipSetDevice(device);
        for (int b = 0; b < 2 && e == hipSuccess; ++b) e = hipEventCreateWithFlags(&done[q][b], hipEventDisableTiming);
        return e;
    }
    int issue(int q, int b, size_t piece) override
    {
        hipError_t e;
        if (per_row > 1)
            e = hipMemcpyAsync(buffer(q, b), from + piece / per_row * pitch + piece % per_row * kPiece, bytes_of(piece),
                               hipMemcpyDeviceToHost, st);
        else if (pitch == width)
            e = hipMemcpyAsync(buffer(q, b), from + piece * per_piece * pitch, rows_of(piece) * width,
                               hipMemcpyDeviceToHost, st);
        else
            e = hipMemcpy2DAsync(buffer(q, b), width, from + piece * per_piece * pitch, pitch, width, rows_of(piece),
                                 hipMemcpyDeviceToHost, st);
        return e == hipSuccess ? hipEventRecord(done[q][b], st) : e;
    }
    int wait(int q, int b) override { return hipEventSynchronize(done[q][b]); }
    void take(int q, int b, size_t piece) override
    {
        const char *src = buffer(q, b);
        auto place = [&](size_t row) { return to + (map ? (size_t)map[row] : row) * width; };
        if (per_row > 1) {
            std::memcpy(place(piece / per_row) + piece % per_row * kPiece, src, bytes_of(piece));
        } else if (!map) {
            std::memcpy(place(piece * per_piece), src, rows_of(piece) * width);
        } else {
            for (size_t r = 0; r < rows_of(piece); ++r) std::memcpy(place(piece * per_piece + r), src + r * width, width);
        }
    }
    void close(int q) override
    {
        for (hipEvent_t &x : done[q])
            if (x) (void)hipEventDestroy(x);
    }
};

hipError_t download(const std::shared_ptr<Staging> &staging, void *dst, const void *src, size_t pitch, size_t width,
                    size_t rows, const int *map, hipStream_t st, std::vector<char> *scratch)
{
    if (width == 0 || rows == 0) return hipStreamSynchronize(st);
    char *to = (char *)dst;
    const char *from = (const char *)src;
    const size_t bytes = (rows - 1) * pitch + width;
    std::unique_lock<std::mutex> lk;
    char *buf = staging ? staging->get(lk, bytes) : nullptr;
    if (!buf || bytes < kOne) return in_one(to, from, pitch, width, rows, map, st, buf, scratch);
    // the stream's device, which need not be the caller's
    hipDevice_t device = 0;
    int callers = 0;
    if (hipStreamGetDevice(st, &device) != hipSuccess || hipGetDevice(&callers) != hipSuccess) {
        (void)hipGetLastError();
        return in_one(to, from, pitch, width, rows, map, st, nullptr, scratch);
    }

    Download d;
    d.device = device;
    d.st = st;
    d.buf = buf;
    d.to = to;
    d.from = from;
    d.pitch = pitch;
    d.width = width;
    d.rows = rows;
    d.map = map;
    d.per_row = (width + kPiece - 1) / kPiece;
    d.per_piece = d.per_row > 1 ? 1 : kPiece / width;
    const size_t pieces = d.per_row > 1 ? rows * d.per_row : (rows + d.per_piece - 1) / d.per_piece;
    const hipError_t e = (hipError_t)deliver(d, pieces, kThreads);
    if (callers != device) (void)hipSetDevice(callers);
    const hipError_t e2 = hipStreamSynchronize(st);   // (nothing is left in flight to the buffers)
    return e != hipSuccess ? e : e2;
}

} // namespace sfg
