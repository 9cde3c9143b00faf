// transfer.hip -- host <-> device state transfers (transfer.hpp), gfx950.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>

#include "transfer.hpp"

namespace {

// Layout change on the device: element-major rows (e, v) of M3 doubles to
// variable-major ones or back.  HBM-bound: a thread moves one double, a
// wavefront 512 consecutive bytes on the element-major side and whole rows on
// the other, so both sides coalesce.  It takes the place of a second host
// array as large as the state and a row-by-row memcpy on one host thread: a
// download of 262 144 elements of 5 x 64 (671 MB) took 205 ms with them and
// takes 15 to 17 ms now, with the staging below.
template <int V, int M3, bool TO_HOST>
__global__ __launch_bounds__(256) void layout_kernel(const double* __restrict__ src, double* __restrict__ dst,
                                                     long long stride, long long off, long long ne) {
    const long long n = ne * V * M3;
    for (long long i = blockIdx.x * 256ll + threadIdx.x; i < n; i += gridDim.x * 256ll) {
        const long long row = i / M3;  // e * V + v
        const int node = int(i - row * M3);
        const long long e = row / V;
        const int v = int(row - e * V);
        const long long d = (v * stride + off + e) * M3 + node;
        if constexpr (TO_HOST)
            dst[i] = src[d];
        else
            dst[d] = src[i];
    }
}

// Returns the launch's own error: the thread's last error may be an earlier
// call's (a failed allocation, another library's), which is no reason to refuse
// a transfer.
template <bool TO_HOST>
hipError_t launch_layout(hipStream_t stream, const double* src, double* dst, long long stride, long long off,
                         long long ne, int V, int M3) {
    const long long n = ne * V * M3;
    const dim3 grid{unsigned(std::min<long long>((n + 255) / 256, 1 << 20))}, block{256};
    void* args[] = {&src, &dst, &stride, &off, &ne};
#define NEMO_LAYOUT(V_, M3_)   \
    if (V == V_ && M3 == M3_)  \
        return hipLaunchKernel(reinterpret_cast<const void*>(&layout_kernel<V_, M3_, TO_HOST>), grid, block, args, 0, \
                               stream);
    NEMO_LAYOUT(5, 27)
    NEMO_LAYOUT(5, 64)
    NEMO_LAYOUT(5, 125)
    NEMO_LAYOUT(9, 27)
    NEMO_LAYOUT(9, 64)
    NEMO_LAYOUT(9, 125)
#undef NEMO_LAYOUT
    return hipErrorInvalidValue;
}

// Pinned staging of the copies over the host link.  A copy to or from
// pageable memory runs at 10 GB/s into fresh pages (one thread of the runtime
// copies and takes the page faults); four threads that each pipeline their
// own two pinned chunks reach 45 to 51 GB/s both ways (671 MB).  ms per
// transfer, plain copy -> staged:
//   download into fresh pages    6 MB 0.82 -> 0.39, 13 MB 1.6 -> 0.65, 26 MB 2.7 -> 0.93, 49 MB 5.0 -> 1.5
//   into pages touched before    6 MB 0.33 -> 0.22, 13 MB 0.75 -> 0.37, 26 MB 1.4 -> 0.60, 49 MB 4.7 -> 1.0
//   upload                       6 MB 0.25 -> 0.26, 13 MB 0.49 -> 0.43, 20 MB 0.74 -> 0.58, 26 MB 0.95 -> 0.69
// and at 1.3 MB a download 0.09 -> 0.21: so downloads are staged from 4 MB on,
// uploads, whose pages have always been touched, from 8 MB on.  A chunk costs a
// gap of 8 us on the link: 2 MB (upload of 671 MB on one stream 21.5 ms with
// 1 MB, 16.8 with 2); short downloads take smaller ones, so that all threads
// have a share of the page faults.
//
// Half of the threads copy on the caller's stream, half on a second one, which
// fills the gaps (16.8 -> 13.0 ms).  More streams gain nothing, and the first
// copies on each set up a hardware queue: with one for every thread the first
// transfers of a process took 28 to 35 ms longer, with two 13 to 20.
//
// The calling thread and three helpers claim chunks one by one.  The caller
// waits only for helpers that have claimed one, so a helper that the host's
// scheduler keeps back (all cores busy, for instance with the spinning
// threads of an OpenMP program) costs nothing: with threads of fixed shares,
// started for each call, 40 downloads of 9 MB on average between such sections
// took 38 ms longer.  A helper that loses its core after it has claimed one is
// waited for: right after such a section a download of 6 MB takes 0.6 ms (plain
// copy 0.4), of 13 MB 0.7 (0.8), of 49 MB 2.8 (5.6).
constexpr int NT = 4, NBUF = 2 * NT;
constexpr size_t MB = size_t(1) << 20, CHUNK = 2 * MB;
constexpr size_t MIN_DOWNLOAD = 4 * MB, MIN_UPLOAD = 8 * MB;

size_t chunk_for(size_t bytes, bool to_host) {
    return !to_host || bytes >= 16 * MB ? CHUNK : (bytes < 8 * MB ? CHUNK / 4 : CHUNK / 2);
}

// One transfer: chunks [0, nc) of `chunk` bytes between dev and host; thread k
// copies on stream[k & 1].
struct Job {
    hipStream_t stream[2];
    char* dev;
    char* host;
    size_t bytes, chunk, nc;
    bool to_host;
    std::atomic<size_t> next{0};
    std::atomic<int> err{int(hipSuccess)};
};

class Staging {
public:
    // nullptr if a part of it cannot be had
    static Staging* create(int device) {
        Staging* s = new (std::nothrow) Staging();
        if (!s) return nullptr;
        bool ok = hipHostMalloc(reinterpret_cast<void**>(&s->pinned_), NBUF * CHUNK, hipHostMallocDefault) == hipSuccess;
        for (auto& x : s->done_) ok = ok && hipEventCreateWithFlags(&x, hipEventDisableTiming) == hipSuccess;
        ok = ok && hipStreamCreateWithFlags(&s->second_, hipStreamNonBlocking) == hipSuccess;
        ok = ok && hipEventCreateWithFlags(&s->start_, hipEventDisableTiming) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            delete s;
            return nullptr;
        }
        for (int k = 1; k < NT; ++k) {
            try {
                s->helper_[k] = std::thread([s, k, device] { s->help(k, device); });
            } catch (const std::system_error&) {
                break;  // fewer helpers
            }
        }
        return s;
    }
    ~Staging() {
        {
            std::lock_guard<std::mutex> l(mu_);
            stop_ = true;
        }
        wake_.notify_all();
        for (auto& t : helper_)
            if (t.joinable()) t.join();
        if (second_) (void)hipStreamDestroy(second_);
        for (auto& x : done_)
            if (x) (void)hipEventDestroy(x);
        if (start_) (void)hipEventDestroy(start_);
        if (pinned_) (void)hipHostFree(pinned_);
    }

    // The whole transfer, after the work already on `stream`; one at a time.
    hipError_t copy(hipStream_t stream, Job& job) {
        hipError_t rc = hipEventRecord(start_, stream);
        if (rc == hipSuccess) rc = hipStreamWaitEvent(second_, start_, 0);
        if (rc != hipSuccess) return rc;
        job.stream[0] = stream;
        job.stream[1] = second_;
        {
            std::lock_guard<std::mutex> l(mu_);
            job_ = &job;
            ++generation_;
        }
        wake_.notify_all();
        work(0, job);
        std::unique_lock<std::mutex> l(mu_);
        job_ = nullptr;  // helpers that wake from here on find nothing
        idle_.wait(l, [this] { return active_ == 0; });
        return hipError_t(job.err.load());
    }

private:
    void help(int k, int device) {
        (void)hipSetDevice(device);
        unsigned long long seen = 0;
        std::unique_lock<std::mutex> l(mu_);
        for (;;) {
            wake_.wait(l, [&] { return stop_ || (job_ && generation_ != seen); });
            if (stop_) return;
            seen = generation_;
            Job* job = job_;
            ++active_;
            l.unlock();
            work(k, *job);
            l.lock();
            if (--active_ == 0) idle_.notify_all();
        }
    }

    // Claims chunks and moves them through buffers 2k and 2k + 1: while one is
    // copied on the host the other is on the link.
    void work(int k, Job& j) {
        char* const buf[2] = {pinned_ + size_t(2 * k) * CHUNK, pinned_ + size_t(2 * k + 1) * CHUNK};
        hipEvent_t* const done = done_ + 2 * k;
        const hipStream_t stream = j.stream[k & 1];
        hipError_t e = hipSuccess;
        auto len = [&](size_t c) { return std::min(j.chunk, j.bytes - c * j.chunk); };
        auto claim = [&] { return j.next.fetch_add(1); };
        auto link = [&](size_t c, int b) {
            char* const d = j.dev + c * j.chunk;
            e = j.to_host ? hipMemcpyAsync(buf[b], d, len(c), hipMemcpyDeviceToHost, stream)
                          : hipMemcpyAsync(d, buf[b], len(c), hipMemcpyHostToDevice, stream);
            if (e == hipSuccess) e = hipEventRecord(done[b], stream);
        };
        int b = 0;
        if (j.to_host) {
            size_t c = claim();
            if (c < j.nc) link(c, 0);
            while (c < j.nc && e == hipSuccess) {
                const size_t ahead = claim();
                if (ahead < j.nc) link(ahead, b ^ 1);
                if (e == hipSuccess) e = hipEventSynchronize(done[b]);
                if (e == hipSuccess) std::memcpy(j.host + c * j.chunk, buf[b], len(c));
                c = ahead;
                b ^= 1;
            }
        } else {
            int used = 0;
            for (size_t c = claim(); c < j.nc && e == hipSuccess; c = claim(), b ^= 1) {
                if (used >= 2) e = hipEventSynchronize(done[b]);
                if (e != hipSuccess) break;
                std::memcpy(buf[b], j.host + c * j.chunk, len(c));
                link(c, b);
                ++used;
            }
            // (the last copy of either buffer; downloads have waited for theirs)
            for (int q = 0; q < 2 && q < used && e == hipSuccess; ++q) e = hipEventSynchronize(done[q]);
        }
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(stream);  // nothing is left in flight
            j.err.store(int(e));
            j.next.store(j.nc);
        }
    }

    char* pinned_ = nullptr;  // NBUF chunks of CHUNK bytes
    hipStream_t second_ = nullptr;
    hipEvent_t done_[NBUF] = {};
    hipEvent_t start_ = nullptr;
    std::thread helper_[NT];
    std::mutex mu_;
    std::condition_variable wake_, idle_;
    Job* job_ = nullptr;
    unsigned long long generation_ = 0;
    int active_ = 0;
    bool stop_ = false;
};

// One per device, made by the first transfer that needs it and freed with the
// last handle (never by a static destructor: a program may end with handles).
constexpr int kMaxDevices = 64;
std::mutex staging_mu[kMaxDevices];  // held for the length of a transfer
Staging* staging[kMaxDevices] = {};
std::mutex refs_mu;
int refs = 0;

// Copies `bytes` between `dev` and `host` through the staging buffers, after
// the work already on `stream`; false if they are not available (another
// transfer on this device holds them, or they could not be made), in which
// case nothing has been copied.
bool staged_copy(hipStream_t stream, double* dev, double* host, size_t bytes, bool to_host, hipError_t* err) {
    int device = 0, of_stream = 0;
    if (hipGetDevice(&device) != hipSuccess || hipStreamGetDevice(stream, &of_stream) != hipSuccess) return false;
    if (device != of_stream || device < 0 || device >= kMaxDevices) return false;
    std::unique_lock<std::mutex> lock(staging_mu[device], std::try_to_lock);
    if (!lock.owns_lock()) return false;
    if (!staging[device]) staging[device] = Staging::create(device);
    if (!staging[device]) return false;
    Job job;
    job.dev = reinterpret_cast<char*>(dev);
    job.host = reinterpret_cast<char*>(host);
    job.bytes = bytes;
    job.chunk = chunk_for(bytes, to_host);
    job.nc = (bytes + job.chunk - 1) / job.chunk;
    job.to_host = to_host;
    *err = staging[device]->copy(stream, job);
    return true;
}

}  // namespace

namespace nemo_host {

// The reports of up to 64 handles share one pinned page, which stays until the
// process ends: a pinned allocation takes longer than the rest of a handle's
// creation.  Further handles allocate their own.
namespace {
constexpr size_t REPORT_BYTES = 64, REPORT_SLOTS = 64;
std::mutex report_mu;
char* report_page = nullptr;
uint64_t report_used = 0;
}  // namespace

void* report_get() {
    std::lock_guard<std::mutex> lock(report_mu);
    if (!report_page && hipHostMalloc(reinterpret_cast<void**>(&report_page), REPORT_BYTES * REPORT_SLOTS,
                                      hipHostMallocPortable) != hipSuccess)
        report_page = nullptr;
    if (report_page && ~report_used) {
        const int k = __builtin_ctzll(~report_used);
        report_used |= uint64_t(1) << k;
        return report_page + REPORT_BYTES * size_t(k);
    }
    void* p = nullptr;
    return hipHostMalloc(&p, REPORT_BYTES, hipHostMallocPortable) == hipSuccess ? p : nullptr;
}

void report_put(void* p) {
    if (!p) return;
    std::lock_guard<std::mutex> lock(report_mu);
    const size_t at = size_t(static_cast<char*>(p) - report_page);
    if (report_page && static_cast<char*>(p) >= report_page && at < REPORT_BYTES * REPORT_SLOTS)
        report_used &= ~(uint64_t(1) << (at / REPORT_BYTES));
    else
        (void)hipHostFree(p);
}

void staging_retain() {
    std::lock_guard<std::mutex> lock(refs_mu);
    ++refs;
}

void staging_release() {
    std::lock_guard<std::mutex> lock(refs_mu);
    if (--refs > 0) return;
    for (int d = 0; d < kMaxDevices; ++d) {
        std::lock_guard<std::mutex> l(staging_mu[d]);
        delete staging[d];
        staging[d] = nullptr;
    }
}

hipError_t state_to_host(hipStream_t stream, const double* dev, long long stride, long long off, long long ne, int V,
                         int M3, double* scratch, double* host) {
    const size_t bytes = size_t(ne) * V * M3 * sizeof(double);
    hipError_t e = launch_layout<true>(stream, dev, scratch, stride, off, ne, V, M3);
    if (e != hipSuccess) return e;
    if (bytes >= MIN_DOWNLOAD && staged_copy(stream, scratch, host, bytes, true, &e)) return e;
    e = hipMemcpyAsync(host, scratch, bytes, hipMemcpyDeviceToHost, stream);
    return e != hipSuccess ? e : hipStreamSynchronize(stream);
}

hipError_t state_to_device(hipStream_t stream, const double* host, double* scratch, double* dev, long long stride,
                           long long off, long long ne, int V, int M3) {
    const size_t bytes = size_t(ne) * V * M3 * sizeof(double);
    hipError_t e = hipSuccess;
    if (bytes < MIN_UPLOAD || !staged_copy(stream, scratch, const_cast<double*>(host), bytes, false, &e)) {
        e = hipMemcpyAsync(scratch, host, bytes, hipMemcpyHostToDevice, stream);
        // the host array is the caller's again on return
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
    }
    if (e != hipSuccess) return e;
    return launch_layout<false>(stream, scratch, dev, stride, off, ne, V, M3);
}

}  // namespace nemo_host
