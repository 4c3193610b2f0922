// transfer.hip -- device fields to the caller's pageable host arrays.
//
// The host layouts are compact (and the velocity interleaved), the device ones
// padded: a kernel packs a chunk of the host layout straight into pinned staging
// memory, and threads copy it on into the caller's array while the next chunk is
// packed into the other half.  Nothing of the context is written.  The link takes
// 57 GB/s, one thread copies into fresh pages at 10-14; a pageable 2-D copy moves
// 3.2 GB/s here (135 MB in 41 ms; the velocity of 4096^2 cells, interleaved by one
// thread, in 143 ms).  c and v of 64^2 cells take 14 and 15 us, of 1024^2 0.32 and
// 0.47 ms, of 4096^2 2.7 and 5.3 ms; packed into device memory and copied from
// there 30 and 52 us, 0.39 and 0.56 ms, 3.0 and 5.7 ms.  Where there is no pinned
// memory to be had, or none free, the pageable copies serve.
#include "impec_device.h"
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace impec {

// element k of the host layout: row k / cols, column k % cols; the velocity has
// two components per column
__global__ void __launch_bounds__(256) k_pack(const double *__restrict__ a, const double *__restrict__ b, int ld,
                                              unsigned long long cols, unsigned long long k0, unsigned long long n,
                                              double *__restrict__ out) {
    const unsigned long long k = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const unsigned long long e = k0 + k;
    unsigned long long cell = b ? e >> 1 : e, row, col;
    if (cell < (1ull << 32) && cols < (1ull << 32)) {   // 32-bit division where it suffices
        row = (unsigned)cell / (unsigned)cols;
        col = (unsigned)cell - (unsigned)row * (unsigned)cols;
    } else {
        row = cell / cols;
        col = cell - row * cols;
    }
    const double *p = b && (e & 1) ? b : a;
    out[k] = p[row * ld + col];
}

namespace {

constexpr size_t STAGE_BYTES = 8u << 20;   // one half of a stage
constexpr int STAGES_MAX = 8;              // stages of the process (128 MiB)
constexpr int COPY_THREADS = 8;
constexpr size_t THREADS_FROM = 4u << 20;  // bytes from which several threads copy

// Pinned staging memory, shared by all contexts of the process: a call takes a
// stage for itself and gives it back.  Stages are allocated as calls overlap and
// kept while contexts exist, since allocating 16 MiB of pinned memory takes longer
// than most reads (a limit of two kept ones made twelve threads allocate 80 times
// in 288 reads); a call that finds all STAGES_MAX taken goes without one.
struct Stage {
    double *half[2], *dev[2];   // on the host, and as the device sees them
};
std::mutex stage_lock;
Stage stage_idle[STAGES_MAX];
int stage_nidle = 0, stage_count = 0, stage_users = 0;

bool stage_take(Stage &s) {
    {
        std::lock_guard<std::mutex> g(stage_lock);
        if (stage_nidle > 0) {
            s = stage_idle[--stage_nidle];
            return true;
        }
        if (stage_count == STAGES_MAX) return false;
        stage_count++;
    }
    s.half[0] = nullptr;
    // coherent: a kernel writes it, and the host reads it when the event has passed
    const unsigned flags = hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent;
    if (hipHostMalloc((void **)&s.half[0], 2 * STAGE_BYTES, flags) != hipSuccess ||
        hipHostGetDevicePointer((void **)&s.dev[0], s.half[0], 0) != hipSuccess) {
        (void)hipGetLastError();
        if (s.half[0]) hipHostFree(s.half[0]);
        std::lock_guard<std::mutex> g(stage_lock);
        stage_count--;
        return false;
    }
    s.half[1] = s.half[0] + STAGE_BYTES / sizeof(double);
    s.dev[1] = s.dev[0] + STAGE_BYTES / sizeof(double);
    return true;
}

// a stage that comes back belongs to a call on a context, so stage_users > 0
void stage_give(const Stage &s) {
    std::lock_guard<std::mutex> g(stage_lock);
    stage_idle[stage_nidle++] = s;
}

// Slices of consecutive chunks copied by `n` threads, the caller among them:
// copy() hands out a chunk, copies the caller's share and waits for the others'.
// Between chunks the threads look for the next one SPINS times, about as long as
// a chunk that is due takes, then sleep: where the caller copies slower than the
// link brings chunks they hardly ever do.
struct Copiers {
    static constexpr int SPINS = 64;
    std::mutex m;
    std::condition_variable go;
    std::atomic<int> chunk{0}, left{0};
    std::atomic<bool> stop{false};
    char *dst = nullptr;
    const char *src = nullptr;
    size_t bytes = 0;
    int n = 1;
    std::vector<std::thread> threads;

    void share(int k) {
        const size_t per = ((bytes + n - 1) / n + 63) & ~size_t(63), at = per * k;
        if (at < bytes) memcpy(dst + at, src + at, per < bytes - at ? per : bytes - at);
    }
    void worker(int k) {
        int seen = 0;
        for (;;) {
            for (int spin = 0; chunk.load(std::memory_order_acquire) == seen; spin++) {
                if (stop.load(std::memory_order_acquire)) return;
                if (spin < SPINS) {
                    std::this_thread::yield();
                } else {
                    std::unique_lock<std::mutex> l(m);
                    go.wait(l, [&] { return chunk.load() != seen || stop.load(); });
                }
            }
            seen++;
            share(k);
            left.fetch_sub(1, std::memory_order_release);
        }
    }
    explicit Copiers(int want) {
        threads.reserve(want);
        // the share of thread k exists only once the thread does
        for (int k = 1; k < want; k++) {
            try {
                threads.emplace_back(&Copiers::worker, this, k);
            } catch (...) {
                break;
            }
        }
        n = 1 + (int)threads.size();
    }
    void copy(char *d, const char *s, size_t b) {
        dst = d;
        src = s;
        bytes = b;
        left.store(n - 1, std::memory_order_relaxed);
        {
            std::lock_guard<std::mutex> l(m);
            chunk.fetch_add(1, std::memory_order_release);
        }
        go.notify_all();
        share(0);
        while (left.load(std::memory_order_acquire) > 0) std::this_thread::yield();
    }
    ~Copiers() {
        {
            std::lock_guard<std::mutex> l(m);
            stop.store(true, std::memory_order_release);
        }
        go.notify_all();
        for (std::thread &t : threads) t.join();
    }
};

int copy_threads(size_t bytes) {
    if (bytes < THREADS_FROM) return 1;
    const unsigned hw = std::thread::hardware_concurrency();
    return hw == 0 ? 1 : (hw / 2 < (unsigned)COPY_THREADS ? (hw / 2 ? (int)(hw / 2) : 1) : COPY_THREADS);
}

}  // namespace

void transfer_attach() {
    std::lock_guard<std::mutex> g(stage_lock);
    stage_users++;
}

void transfer_detach() {
    std::lock_guard<std::mutex> g(stage_lock);
    if (--stage_users > 0) return;
    while (stage_nidle > 0) {
        hipHostFree(stage_idle[--stage_nidle].half[0]);
        stage_count--;
    }
}

// rows x cols of the device array a (pitch ld), or of a and b interleaved, into dst
static int get_chunks(impec_ctx *ctx, const Stage &st, double *dst, const double *a, const double *b, int ld, int rows,
                      int cols) {
    const size_t total = (size_t)rows * cols * (b ? 2 : 1);
    const size_t per = STAGE_BYTES / sizeof(double), chunks = (total + per - 1) / per;
    auto queue = [&](size_t c) -> int {
        const size_t at = c * per, n = per < total - at ? per : total - at;
        hipLaunchKernelGGL(k_pack, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, a, b, ld,
                           (unsigned long long)cols, (unsigned long long)at, (unsigned long long)n, st.dev[c & 1]);
        IMPEC_HIP_CHECK(ctx, hipGetLastError());
        IMPEC_HIP_CHECK(ctx, hipEventRecord(ctx->ev_get[c & 1], ctx->stream));
        return IMPEC_OK;
    };
    const int nthreads = copy_threads(total * sizeof(double));
    // the copying threads start when the stream has come to the read
    if (nthreads > 1) IMPEC_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    if (int e = queue(0)) return e;
    Copiers pool(nthreads);
    for (size_t c = 0; c < chunks; c++) {
        if (c + 1 < chunks)   // its half was emptied in the previous round
            if (int e = queue(c + 1)) return e;
        IMPEC_HIP_CHECK(ctx, hipEventSynchronize(ctx->ev_get[c & 1]));
        const size_t at = c * per, n = per < total - at ? per : total - at;
        pool.copy((char *)(dst + at), (const char *)st.half[c & 1], n * sizeof(double));
    }
    return IMPEC_OK;
}

// the same without staging memory: pageable 2-D copies, the velocity's components
// interleaved on the host
static int get_plain(impec_ctx *ctx, double *dst, const double *a, const double *b, int ld, int rows, int cols) {
    auto get2d = [&](double *to, const double *from) -> int {
        IMPEC_HIP_CHECK(ctx, hipMemcpy2DAsync(to, sizeof(double) * cols, from, sizeof(double) * ld, sizeof(double) * cols,
                                              rows, hipMemcpyDeviceToHost, ctx->stream));
        IMPEC_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
        return IMPEC_OK;
    };
    if (!b) return get2d(dst, a);
    std::vector<double> u((size_t)rows * cols), v((size_t)rows * cols);
    int e = get2d(u.data(), a);
    if (!e) e = get2d(v.data(), b);
    for (size_t k = 0; !e && k < u.size(); k++) {
        dst[2 * k] = u[k];
        dst[2 * k + 1] = v[k];
    }
    return e;
}

int get_field(impec_ctx *ctx, double *dst, const double *a, const double *b, int ld, int rows, int cols) {
    Stage st;
    const bool staged = stage_take(st);
    int e;
    try {
        if (staged)
            e = get_chunks(ctx, st, dst, a, b, ld, rows, cols);
        else
            e = get_plain(ctx, dst, a, b, ld, rows, cols);
    } catch (const std::bad_alloc &) {
        e = set_error(ctx, IMPEC_ENOMEM, "host memory");
    }
    if (!staged) return e;
    if (e) hipStreamSynchronize(ctx->stream);   // no copy into the stage is left in flight
    stage_give(st);
    return e;
}

}  // namespace impec
