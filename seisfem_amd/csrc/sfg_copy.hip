// Downloads of large results (see sfg_copy.h).
#include "sfg_copy.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace sfg {

namespace {
constexpr int kThreads = 8;
constexpr size_t kPiece = (size_t)1 << 20;   // bytes of one transfer; two buffers per thread
constexpr size_t kDirect = (size_t)4 << 20;  // smaller results are copied directly
std::mutex g_mu;
std::weak_ptr<Staging> g_staging;
} // namespace

struct Staging {
    std::mutex mu;                           // one download at a time
    char *buf = nullptr;
    bool tried = false;
    char *get()
    {
        if (!tried) {
            tried = true;
            if (hipHostMalloc((void **)&buf, 2 * kThreads * kPiece, hipHostMallocPortable) != hipSuccess) {
                (void)hipGetLastError();
                buf = nullptr;
            }
        }
        return buf;
    }
    ~Staging()
    {
        if (buf) (void)hipHostFree(buf);
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

static hipError_t direct(char *dst, const char *src, size_t pitch, size_t width, size_t rows, const int *map,
                         hipStream_t st)
{
    hipError_t e;
    std::vector<char> rowsv;
    if (map) rowsv.resize(width * rows);     // one transfer, whatever the number of rows
    char *to = map ? rowsv.data() : dst;
    if (pitch == width)
        e = hipMemcpyAsync(to, src, width * rows, hipMemcpyDeviceToHost, st);
    else
        e = hipMemcpy2DAsync(to, width, src, pitch, width, rows, hipMemcpyDeviceToHost, st);
    const hipError_t e2 = hipStreamSynchronize(st);
    if (map && e == hipSuccess && e2 == hipSuccess)
        for (size_t i = 0; i < rows; ++i) std::memcpy(dst + (size_t)map[i] * width, to + i * width, width);
    return e != hipSuccess ? e : e2;
}

hipError_t download(const std::shared_ptr<Staging> &staging, void *dst, const void *src, size_t pitch, size_t width,
                    size_t rows, const int *map, hipStream_t st)
{
    if (width == 0 || rows == 0) return hipStreamSynchronize(st);
    char *to = (char *)dst;
    const char *from = (const char *)src;
    if (!staging || width * rows < kDirect) return direct(to, from, pitch, width, rows, map, st);
    std::lock_guard<std::mutex> lk(staging->mu);
    char *buf = staging->get();
    // the stream's device, which need not be the caller's
    hipDevice_t device = 0;
    int callers = 0;
    if (!buf || hipStreamGetDevice(st, &device) != hipSuccess || hipGetDevice(&callers) != hipSuccess) {
        (void)hipGetLastError();
        return direct(to, from, pitch, width, rows, map, st);
    }

    // pieces: parts of a row, or several whole rows
    const size_t per_row = (width + kPiece - 1) / kPiece, per_piece = per_row > 1 ? 1 : kPiece / width;
    const size_t pieces = per_row > 1 ? rows * per_row : (rows + per_piece - 1) / per_piece;
    std::atomic<size_t> next{0};
    std::atomic<int> error{hipSuccess};
    auto work = [&](int q) {
        hipError_t e = hipSetDevice(device);
        hipEvent_t done[2] = {nullptr, nullptr};
        for (int k = 0; k < 2 && e == hipSuccess; ++k) e = hipEventCreateWithFlags(&done[k], hipEventDisableTiming);
        size_t row[2], off[2], len[2];           // the piece on its way in each buffer
        bool have[2] = {false, false};
        auto issue = [&](int k) {
            have[k] = false;
            const size_t i = next++;
            if (i >= pieces || e != hipSuccess || error.load() != hipSuccess) return;
            char *b = buf + (size_t)(2 * q + k) * kPiece;
            if (per_row > 1) {
                row[k] = i / per_row;
                off[k] = i % per_row * kPiece;
                len[k] = std::min(kPiece, width - off[k]);
                e = hipMemcpyAsync(b, from + row[k] * pitch + off[k], len[k], hipMemcpyDeviceToHost, st);
            } else {
                row[k] = i * per_piece;
                off[k] = 0;
                const size_t nr = std::min(per_piece, rows - row[k]);
                len[k] = nr * width;
                e = pitch == width ? hipMemcpyAsync(b, from + row[k] * pitch, len[k], hipMemcpyDeviceToHost, st)
                                   : hipMemcpy2DAsync(b, width, from + row[k] * pitch, pitch, width, nr,
                                                      hipMemcpyDeviceToHost, st);
            }
            if (e == hipSuccess) e = hipEventRecord(done[k], st);
            have[k] = e == hipSuccess;
        };
        issue(0);
        issue(1);
        for (int k = 0; have[k]; k ^= 1) {
            e = hipEventSynchronize(done[k]);
            if (e != hipSuccess) break;
            const char *b = buf + (size_t)(2 * q + k) * kPiece;
            if (per_row > 1 || !map) {
                std::memcpy(to + (map ? (size_t)map[row[k]] : row[k]) * width + off[k], b, len[k]);
            } else {
                for (size_t r = 0; r < len[k] / width; ++r)
                    std::memcpy(to + (size_t)map[row[k] + r] * width, b + r * width, width);
            }
            issue(k);
        }
        for (hipEvent_t &x : done)
            if (x) (void)hipEventDestroy(x);
        if (e != hipSuccess) error.store(e);
    };
    std::thread th[kThreads];
    int started = 1;
    try {
        for (; started < kThreads; ++started) th[started] = std::thread(work, started);
    } catch (const std::exception &) {
        // fewer helpers: the pieces are handed out as they are asked for
    }
    work(0);
    for (int q = 1; q < started; ++q) th[q].join();
    if (callers != device) (void)hipSetDevice(callers);
    const hipError_t e2 = hipStreamSynchronize(st);
    const hipError_t e = (hipError_t)error.load();
    return e != hipSuccess ? e : e2;
}

} // namespace sfg
