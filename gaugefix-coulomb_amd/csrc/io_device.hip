// io_device.hip -- configurations and gauge transformations streamed between
// HBM and files or host arrays.
//
// The file formats are those of host_io.c (src/fields_io.c of the reference):
// a configuration is the raw image of 4V matrices of 18 reals of 4 or 8
// bytes, optionally byte-swapped; a gauge transformation is the native-endian
// FP64 image of V matrices.  Here a file moves through two pinned host
// blocks: host threads read (or write) one block with pread (pwrite) while the
// DMA engine copies the other, and the byte swap and the FP32 <-> FP64
// conversions run on the device.  No full-size host image is made.
//
// Host arrays (gfc_job_upload_config, gfc_job_download_*, the server's inputs
// and results) are pageable memory that the copy engine cannot read by itself:
// a plain hipMemcpy moves them through one thread at 10 GB/s.  copy_to_host and
// copy_from_host move them through a ring of pinned slots, with host threads
// copying between the slots and the array while the engine moves others.
#include <fcntl.h>
#include <hip/hip_runtime.h>
#include <sys/stat.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstring>
#include <exception>
#include <memory>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "internal.hpp"

using gfc::cplx;
using gfc::kBlock;
using gfcx::fail;
using gfcx::nblocks;

namespace {

constexpr size_t kIoBlock = 16u << 20;  // bytes per pinned block
constexpr int kIoThreads = 4;           // host threads per block

__global__ __launch_bounds__(kBlock) void k_bswap64(uint64_t *__restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) p[i] = __builtin_bswap64(p[i]);
}

// FP32 reals (optionally byte-swapped) -> FP64.
__global__ __launch_bounds__(kBlock) void k_f32raw_to_f64(const uint32_t *__restrict__ in,
                                                          double *__restrict__ out, int64_t n,
                                                          int swap) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    uint32_t v = in[i];
    if (swap) v = __builtin_bswap32(v);
    out[i] = (double)__uint_as_float(v);
}

// FP64 reals [0, n) -> out as FP64 or FP32, optionally byte-swapped.
__global__ __launch_bounds__(kBlock) void k_f64_to_raw(const double *__restrict__ in,
                                                       void *__restrict__ out, int64_t n,
                                                       int prec, int swap) {
    const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    if (prec == 8) {
        uint64_t v = (uint64_t)__double_as_longlong(in[i]);
        static_cast<uint64_t *>(out)[i] = swap ? __builtin_bswap64(v) : v;
    } else {
        uint32_t v = __float_as_uint((float)in[i]);
        static_cast<uint32_t *>(out)[i] = swap ? __builtin_bswap32(v) : v;
    }
}

// pread / pwrite of n bytes at off, split over kIoThreads threads; false on a
// short transfer or an error.
bool par_io(int fd, char *buf, size_t n, off_t off, bool write) {
    std::vector<std::thread> th;
    std::vector<char> ok(kIoThreads, 1);
    const size_t part = (n + kIoThreads - 1) / kIoThreads;
    for (int t = 0; t < kIoThreads; t++) {
        const size_t a = std::min(n, t * part), b = std::min(n, a + part);
        if (a >= b) break;
        th.emplace_back([=, &ok] {
            size_t done = a;
            while (done < b) {
                const ssize_t r = write ? pwrite(fd, buf + done, b - done, off + done)
                                        : pread(fd, buf + done, b - done, off + done);
                if (r <= 0) {
                    ok[t] = 0;
                    return;
                }
                done += (size_t)r;
            }
        });
    }
    for (auto &x : th) x.join();
    for (char c : ok)
        if (!c) return false;
    return true;
}

// Two pinned blocks of the context, allocated on first use.  The caller holds
// c->pin_mu from here until its last use of them.
int pinned_blocks(gfc_ctx *c) {
    for (int k = 0; k < 2; k++) {
        if (c->pin[k] == nullptr)
            HIP_TRY(hipHostMalloc(&c->pin[k], kIoBlock, hipHostMallocDefault));
        if (c->pin_ev[k] == nullptr)
            HIP_TRY(hipEventCreateWithFlags(&c->pin_ev[k], hipEventDisableTiming));
    }
    return GFC_OK;
}

// The ring of pinned slots for host arrays, and the pieces of a slot that host
// threads copy.
// 1.53 GB to a host array takes 42 ms in slots of 8 MiB, 50 ms in slots of
// 4 MiB, 74 ms of 2 MiB, 85 ms of 1 MiB (each copy call costs some 20 us) and
// 38 ms in three of 16 MiB; 12 threads gain nothing over 8.
constexpr int kSlots = gfc_ctx::kSlots;
constexpr size_t kSlot = 8u << 20;
constexpr size_t kPiece = 256u << 10;
constexpr int kCopyThreads = 8;
// Below this a plain copy is as fast (19 MB: 1.4 ms either way; 46 MB: 4.5
// against 2.8 ms); and for a context without a ring yet, whose allocation takes
// some 3 ms, below kRingNew (plain copies move 10 to 14 GB/s).
constexpr size_t kRingMin = 24u << 20, kRingNew = 64u << 20;

// Whether `total` bytes of the host array `host` go through the ring.  Memory
// that HIP knows (pinned by the caller, managed) is read by the copy engine
// itself, at 56 GB/s in one plain copy: 32^3 x 64, ring / plain, G 6.1 / 5.4 ms,
// U 23.5 / 21.1 ms.
bool use_ring(gfc_ctx *c, const void *host, size_t total) {
    {
        std::lock_guard<std::mutex> lk(c->pin_mu);
        if (total < (c->ring ? kRingMin : kRingNew)) return false;
    }
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, host) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();  // memory unknown to HIP, in older versions
    return true;
}

char *slot(gfc_ctx *c, int k) { return c->ring + (size_t)k * kSlot; }

// The ring of the context, allocated on first use, with no copy of an earlier
// call still running in it.  The caller holds c->pin_mu.
int make_ring(gfc_ctx *c) {
    if (c->ring == nullptr) {
        void *p = nullptr;
        HIP_TRY(hipHostMalloc(&p, kSlots * kSlot, hipHostMallocDefault));
        c->ring = static_cast<char *>(p);
    }
    for (hipEvent_t &e : c->slot_ev) {
        if (e == nullptr) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        HIP_TRY(hipEventSynchronize(e));
    }
    return GFC_OK;
}

// Whether the context has its ring.  When it cannot have one the caller takes
// another way, so the failed request must not be reported by the next launch
// check (HIP keeps an error until it is read) nor by gfc_last_error.
bool ring(gfc_ctx *c) {
    std::string message;
    message.swap(gfcx::last_error);
    const bool have = make_ring(c) == GFC_OK;
    if (!have) (void)hipGetLastError();
    gfcx::last_error.swap(message);
    return have;
}

// Host threads that take the pieces of a transfer in turn and copy each once
// its block is open, i.e. below `open`.  done[b] counts the pieces of block b
// that are copied.  They end when every piece is taken or `stop` is set, and
// are joined by the destructor.  Nothing here throws: the callers are C entries.
struct Copiers {
    std::atomic<size_t> open{0}, next{0};
    std::atomic<bool> stop{false};
    std::unique_ptr<std::atomic<size_t>[]> done;
    std::vector<std::thread> th;

    explicit Copiers(size_t blocks) : done(new (std::nothrow) std::atomic<size_t>[blocks]()) {}
    // copy(block, offset, n) for every piece; false if no thread could start.
    template <typename Copy>
    bool start(size_t total, Copy copy) {
        if (!done) return false;
        const size_t pieces = (total + kPiece - 1) / kPiece;
        const int nth = (int)std::min<size_t>(
            kCopyThreads, std::max(1u, std::thread::hardware_concurrency()));
        try {
            for (int t = 0; t < nth; t++)
                th.emplace_back([this, total, pieces, copy] {
                    for (;;) {
                        const size_t i = next.fetch_add(1, std::memory_order_relaxed);
                        if (i >= pieces) return;
                        const size_t off = i * kPiece, b = off / kSlot;
                        while (open.load(std::memory_order_acquire) <= b) {
                            if (stop.load(std::memory_order_relaxed)) return;
                            std::this_thread::yield();
                        }
                        copy(b, off, std::min(kPiece, total - off));
                        done[b].fetch_add(1, std::memory_order_release);
                    }
                });
        } catch (const std::exception &) {  // no memory, or no thread
            return !th.empty();             // fewer threads do the same work
        }
        return true;
    }
    // Waits until the pieces of block b of a transfer of `total` bytes are copied.
    void wait(size_t b, size_t total) const {
        const size_t n = std::min(kSlot, total - b * kSlot), pieces = (n + kPiece - 1) / kPiece;
        while (done[b].load(std::memory_order_acquire) < pieces) std::this_thread::yield();
    }
    ~Copiers() {
        stop.store(true, std::memory_order_relaxed);
        for (auto &t : th) t.join();
    }
};

// File bytes [0, total) -> device bytes dst[0, total), block by block.
int stream_in(gfc_ctx *c, int fd, char *dst, size_t total) {
    std::lock_guard<std::mutex> lk(c->pin_mu);
    RC_TRY(pinned_blocks(c));
    int k = 0;
    for (size_t off = 0; off < total; off += kIoBlock, k ^= 1) {
        const size_t n = std::min(kIoBlock, total - off);
        HIP_TRY(hipEventSynchronize(c->pin_ev[k]));  // the copy that used this block
        if (!par_io(fd, static_cast<char *>(c->pin[k]), n, (off_t)off, false)) {
            hipStreamSynchronize(c->stream);
            return -2;
        }
        HIP_TRY(hipMemcpyAsync(dst + off, c->pin[k], n, hipMemcpyHostToDevice, c->stream));
        HIP_TRY(hipEventRecord(c->pin_ev[k], c->stream));
    }
    HIP_TRY(hipStreamSynchronize(c->stream));
    return GFC_OK;
}

// Device bytes src[0, total) -> file bytes [0, total), block by block: the
// copy of block b+1 runs while block b is written.
int stream_out(gfc_ctx *c, int fd, const char *src, size_t total) {
    std::lock_guard<std::mutex> lk(c->pin_mu);
    RC_TRY(pinned_blocks(c));
    const size_t nb = (total + kIoBlock - 1) / kIoBlock;
    auto issue = [&](size_t b) -> int {
        const size_t off = b * kIoBlock, n = std::min(kIoBlock, total - off);
        HIP_TRY(hipMemcpyAsync(c->pin[b & 1], src + off, n, hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(hipEventRecord(c->pin_ev[b & 1], c->stream));
        return GFC_OK;
    };
    if (nb) RC_TRY(issue(0));
    for (size_t b = 0; b < nb; b++) {
        HIP_TRY(hipEventSynchronize(c->pin_ev[b & 1]));
        if (b + 1 < nb) RC_TRY(issue(b + 1));
        const size_t off = b * kIoBlock, n = std::min(kIoBlock, total - off);
        if (!par_io(fd, static_cast<char *>(c->pin[b & 1]), n, (off_t)off, true)) {
            hipStreamSynchronize(c->stream);
            return -2;
        }
    }
    return GFC_OK;
}

// copy_to_host and copy_from_host through the ring; > 0 if it is not to be had.
int ring_to_host(gfc_ctx *c, hipStream_t s, char *dst, const char *src, size_t total) {
    std::lock_guard<std::mutex> lk(c->pin_mu);
    if (!ring(c)) return 1;
    const size_t nb = (total + kSlot - 1) / kSlot;
    Copiers cp(nb);
    if (!cp.start(total, [=](size_t b, size_t off, size_t n) {
            std::memcpy(dst + off, slot(c, (int)(b % kSlots)) + (off - b * kSlot), n);
        }))
        return 1;
    size_t issued = 0;
    for (size_t b = 0; b < nb; b++) {
        for (; issued < nb && issued < b + kSlots; issued++) {
            if (issued >= kSlots) cp.wait(issued - kSlots, total);
            const size_t off = issued * kSlot, n = std::min(kSlot, total - off);
            const int k = (int)(issued % kSlots);
            HIP_TRY(hipMemcpyAsync(slot(c, k), src + off, n, hipMemcpyDeviceToHost, s));
            HIP_TRY(hipEventRecord(c->slot_ev[k], s));
        }
        HIP_TRY(hipEventSynchronize(c->slot_ev[b % kSlots]));
        cp.open.store(b + 1, std::memory_order_release);
    }
    for (size_t b = nb < (size_t)kSlots ? 0 : nb - kSlots; b < nb; b++) cp.wait(b, total);
    return GFC_OK;
}

int ring_from_host(gfc_ctx *c, hipStream_t s, char *dst, const char *src, size_t total) {
    std::lock_guard<std::mutex> lk(c->pin_mu);
    if (!ring(c)) return 1;
    const size_t nb = (total + kSlot - 1) / kSlot;
    Copiers cp(nb);
    cp.open.store(kSlots, std::memory_order_relaxed);  // every slot is free
    if (!cp.start(total, [=](size_t b, size_t off, size_t n) {
            std::memcpy(slot(c, (int)(b % kSlots)) + (off - b * kSlot), src + off, n);
        }))
        return 1;
    for (size_t b = 0; b < nb; b++) {
        cp.wait(b, total);
        const size_t off = b * kSlot, n = std::min(kSlot, total - off);
        const int k = (int)(b % kSlots);
        HIP_TRY(hipMemcpyAsync(dst + off, slot(c, k), n, hipMemcpyHostToDevice, s));
        HIP_TRY(hipEventRecord(c->slot_ev[k], s));
        if (b > 0) {
            HIP_TRY(hipEventSynchronize(c->slot_ev[(b - 1) % kSlots]));
            cp.open.store(b + kSlots, std::memory_order_release);
        }
    }
    return GFC_OK;
}

}  // namespace

// Device bytes src[0, total) -> host array dst, complete on return.  48^3 x 96:
// G (1.53 GB) 144 -> 43 ms, U (6.1 GB) 574 -> 170 ms.
int gfcx::copy_to_host(gfc_ctx *c, hipStream_t s, void *dst, const void *src, size_t total) {
    if (use_ring(c, dst, total)) {
        const int rc = ring_to_host(c, s, static_cast<char *>(dst), static_cast<const char *>(src),
                                    total);
        if (rc <= 0) return rc;
    }
    HIP_TRY(hipMemcpyAsync(dst, src, total, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    return GFC_OK;
}

// Host array src -> device bytes dst[0, total); pageable memory is read on
// return (the last copies to the device may still be running on s), pinned
// memory once s has got there.  48^3 x 96, an FP32
// configuration (3.06 GB): 103 -> 62 ms.
int gfcx::copy_from_host(gfc_ctx *c, hipStream_t s, void *dst, const void *src, size_t total) {
    if (use_ring(c, src, total)) {
        const int rc = ring_from_host(c, s, static_cast<char *>(dst),
                                      static_cast<const char *>(src), total);
        if (rc <= 0) return rc;
    }
    HIP_TRY(hipMemcpyAsync(dst, src, total, hipMemcpyHostToDevice, s));
    return GFC_OK;
}

// Host array src -> host array dst, the server's own copy of an input (new
// memory: most of its time is the first touch of its pages).
void gfcx::copy_host(void *dst, const void *src, size_t total) {
    const size_t blocks = (total + kSlot - 1) / kSlot;
    Copiers cp(blocks);
    cp.open.store(blocks, std::memory_order_relaxed);
    char *d = static_cast<char *>(dst);
    const char *f = static_cast<const char *>(src);
    if (total < kRingMin ||
        !cp.start(total, [=](size_t, size_t off, size_t n) { std::memcpy(d + off, f + off, n); })) {
        std::memcpy(d, f, total);
        return;
    }
    for (size_t b = 0; b < blocks; b++) cp.wait(b, total);
}

extern "C" int gfc_job_load_config(gfc_job *j, const char *path, int in_precision,
                                   int byte_swap) {
    if (in_precision != 4 && in_precision != 8) return -4;
    if (j == nullptr || path == nullptr) return fail(GFC_EINVAL, "gfc_job_load_config: NULL");
    HIP_TRY(hipSetDevice(j->ctx->device));
    const int fd = open(path, O_RDONLY);
    if (fd < 0) {
        fprintf(stderr, "Error: Problem opening config file %s.\n", path);
        return -1;
    }
    struct stat sb;
    const size_t nreal = (size_t)j->V * 4 * 18;
    const size_t total = nreal * (size_t)in_precision;
    if (fstat(fd, &sb) != 0 || (size_t)sb.st_size < total) {
        fprintf(stderr, "Error: Reading from file %s.\n", path);
        close(fd);
        return -2;
    }
    if ((size_t)sb.st_size > total) {
        fprintf(stderr, "Error: File has not been read till the end.\n Check lattice sizes.\n");
        close(fd);
        return -3;
    }
    gfc_ctx *c = j->ctx;
    // FP64 lands in place; FP32 is staged in the u0 fields (288V bytes, the
    // size of an FP32 configuration), which the next fix rebuilds anyway
    char *dst = in_precision == 8 ? reinterpret_cast<char *>(j->cfg)
                                  : reinterpret_cast<char *>(j->u0);
    int rc = stream_in(c, fd, dst, total);
    close(fd);
    if (rc == -2) fprintf(stderr, "Error: Reading from file %s.\n", path);
    if (rc) return rc;
    if (in_precision == 8) {
        if (byte_swap) {
            hipLaunchKernelGGL(k_bswap64, dim3(nblocks(nreal)), dim3(kBlock), 0, c->stream,
                               reinterpret_cast<uint64_t *>(j->cfg), (int64_t)nreal);
            LAUNCH_CHECK();
        }
    } else {
        hipLaunchKernelGGL(k_f32raw_to_f64, dim3(nblocks(nreal)), dim3(kBlock), 0, c->stream,
                           reinterpret_cast<const uint32_t *>(j->u0),
                           reinterpret_cast<double *>(j->cfg), (int64_t)nreal, byte_swap);
        LAUNCH_CHECK();
    }
    RC_TRY(gfcx::set_identity(j));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return GFC_OK;
}

extern "C" int gfc_job_write_gauge_transf(gfc_job *j, const char *path) {
    if (j == nullptr || path == nullptr)
        return fail(GFC_EINVAL, "gfc_job_write_gauge_transf: NULL");
    HIP_TRY(hipSetDevice(j->ctx->device));
    gfc_ctx *c = j->ctx;
    // AoS image of G staged in the u0 fields (144V bytes)
    cplx<double> *stage = j->u0;
    hipLaunchKernelGGL(gfc::k_g_to_aos, dim3(nblocks(j->V)), dim3(kBlock), 0, c->stream, j->g,
                       stage, j->geom.ns, j->Vh);
    LAUNCH_CHECK();
    const int fd = open(path, O_WRONLY | O_CREAT | O_TRUNC, 0644);
    if (fd < 0) {
        hipStreamSynchronize(c->stream);
        return -1;
    }
    int rc = stream_out(c, fd, reinterpret_cast<const char *>(stage),
                        (size_t)j->V * 18 * sizeof(double));
    if (close(fd) != 0 && rc == GFC_OK) rc = -2;
    return rc;
}

extern "C" int gfc_job_write_config(gfc_job *j, const char *path, int out_precision,
                                    int byte_swap) {
    if (out_precision != 4 && out_precision != 8) return -4;
    if (j == nullptr || path == nullptr) return fail(GFC_EINVAL, "gfc_job_write_config: NULL");
    HIP_TRY(hipSetDevice(j->ctx->device));
    gfc_ctx *c = j->ctx;
    const int64_t nreal = j->V * 4 * 18;
    const size_t total = (size_t)nreal * (size_t)out_precision;
    // the output image, staged in the u0 fields (FP32: 288V bytes) or, for
    // FP64, converted in place only when it has to be swapped
    const char *src = reinterpret_cast<const char *>(j->cfg);
    void *tmp = nullptr;
    if (out_precision == 4 || byte_swap) {
        void *stage = j->u0;
        if (out_precision == 8) {
            hipError_t e = hipMalloc(&tmp, total);
            if (e != hipSuccess)
                return fail(GFC_ENOMEM, std::string("gfc_job_write_config: ") +
                                            hipGetErrorString(e));
            stage = tmp;
        }
        hipLaunchKernelGGL(k_f64_to_raw, dim3(nblocks(nreal)), dim3(kBlock), 0, c->stream,
                           reinterpret_cast<const double *>(j->cfg), stage, nreal, out_precision,
                           byte_swap);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            hipFree(tmp);
            return fail(GFC_EDEVICE, hipGetErrorString(e));
        }
        src = static_cast<const char *>(stage);
    }
    const int fd = open(path, O_WRONLY | O_CREAT | O_TRUNC, 0644);
    int rc = -1;
    if (fd >= 0) {
        rc = stream_out(c, fd, src, total);
        if (close(fd) != 0 && rc == GFC_OK) rc = -2;
    } else {
        fprintf(stderr, "Error: Problem creating file %s for config.\n", path);
        hipStreamSynchronize(c->stream);
    }
    hipFree(tmp);
    return rc;
}
