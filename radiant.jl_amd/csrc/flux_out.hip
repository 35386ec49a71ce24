// flux_out.hip -- flux moments from the device into the caller's (pageable) memory.
//
// The flux lies [group][moment][cell] on the device and leaves as Radiant's [cell][moment][group].
// Cells are outermost there, so a range of cells is one contiguous piece of the output.  Pieces go
// through a ring of pinned host memory, from which host threads copy them into the caller's memory, whose
// pages are usually touched there for the first time.  Small pieces keep the link and the threads
// busy at once.  They reach the ring in one of two ways:
//  - With nothing else running on the device, the kernel that rearranges a piece writes it straight
//    into the ring: the link's speed without a staging copy.  Bound by the link (57 GB/s measured into
//    pinned memory).  With two 64 MiB staging buffers and threads made for each: 1.41 GB of a 64^3
//    solve 36 ms, 119 MB 4.4 ms, twelve fluxes of 45 MB 23.5 ms; here 27.8 (51 GB/s), 2.9 and 16.5 ms.
//  - Beside other solves those kernels wait, piece by piece, behind the others' on the process's four
//    hardware queues, and hold the queue and their CUs for as long as their stores cross the link:
//    4.03 GB beside six solving threads took 196-206 ms and the solves fell from 122 to 82 a second
//    (two staging buffers: 126-190 ms, 95-110 a second).  There the device rearranges 64 MiB at a
//    time into device memory and the copy engines move the pieces: 135 ms, 119-123 solves a second.  From a
//    server with eight requests in flight 4.03, 3.58 and 0.49 GB took 167-230, 156-227 and 23-41 ms (medians of
//    runs; staging buffers 142-209, 107-176 and 20-38), now 148-155, 134-142 and 27-31.  Alone on the
//    device this way is the slower one: 134 against 74 ms, as the copy engines reach 30 GB/s here.
#include "flux_out.hpp"
#include "engine.hpp"

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <deque>
#include <mutex>
#include <stdexcept>
#include <string>
#include <system_error>
#include <thread>
#include <vector>

namespace rt {

#define RT_HIP(x)                                                                                 \
    do {                                                                                          \
        hipError_t e_ = (x);                                                                      \
        if (e_ != hipSuccess) throw std::runtime_error(std::string("HIP error: ") + hipGetErrorString(e_) + \
                                                       " at " + __FILE__ + ":" + std::to_string(__LINE__)); \
    } while (0)

namespace {

constexpr int TILE = 64;

// dst[(g + G p) + G Np (c - c0)] = src[(g Np + p) Nc + c]: tiles of 64 output rows x 64 cells through
// LDS, so that both sides move 512 contiguous bytes per wave.
__global__ __launch_bounds__(256) void flux_rows_kernel(double* __restrict__ dst, const double* __restrict__ src, int G, int Np,
                                                        int Nc, int c0, int nc) {
    __shared__ double s[TILE][TILE + 1];
    const int R = G * Np, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int j0 = blockIdx.x * TILE, b0 = blockIdx.y * TILE;
    for (int r = wv; r < TILE; r += 4) {
        const int j = j0 + r;  // output row g + G p
        if (j < R && b0 + lane < nc) {
            const int p = j / G, g = j - p * G;
            s[r][lane] = src[((size_t)g * Np + p) * Nc + c0 + b0 + lane];
        }
    }
    __syncthreads();
    for (int c = wv; c < TILE; c += 4)
        if (j0 + lane < R && b0 + c < nc) dst[(size_t)(b0 + c) * R + j0 + lane] = s[lane][c];
}

constexpr size_t HUGE_PAGE = (size_t)2 << 20;
constexpr size_t RING = (size_t)12 << 20;    // doubles of the ring (96 MiB pinned, held by the process)
constexpr size_t PIECE_MAX = RING / 12;      // doubles of a piece at most (8 MiB)
constexpr int SLOTS_MAX = 48;
// Pieces alternate between two streams, so that one drains while the next runs.  Four were no faster for
// the copy engines, and two more streams in the process moved a lockstep batch's own streams to other
// hardware queues (41.1 -> 44.5 ms).
constexpr int STREAMS = 2;
// A chunk that the copy engines empty while the next one is filled, in the scratch that the caller lends:
// 32 MiB does not cover the wait of the rearranging kernel behind others' (145-172 ms where 64 MiB took
// 135; 0.49 GB in chunks of 20 MiB 28-47 ms, of 41 MiB 30-31), 128 MiB is no faster.
constexpr size_t CHUNK_MAX = (size_t)8 << 20;    // doubles
constexpr size_t CHUNK_MIN = PIECE_MAX / 8;      // below 1 MiB the copies' own cost counts

// Doubles per piece: large ones keep the link busiest (2 MiB 49, 4 MiB 53, 8 MiB 55 GB/s of 57), small
// ones let a small flux overlap its transfer with its copies.
size_t piece_size(size_t total) {
    const size_t mib = (size_t)1 << 17;
    return total >= 256 * mib ? 8 * mib : (total >= 64 * mib ? 4 * mib : 2 * mib);
}

// The ring and its copying threads: one copy-out at a time, the threads asleep between them.
struct Ring {
    std::mutex use;  // held by the copy-out that runs
    double* buf = nullptr;
    hipEvent_t ev[SLOTS_MAX] = {}, ready_ev = nullptr, chunk_ev[2] = {};
    hipStream_t st[STREAMS] = {};
    bool tried = false;
    std::mutex mu;
    std::condition_variable work, done;
    struct Job { double* dst; const double* src; size_t n; int slot; };
    std::deque<Job> jobs;
    int busy[SLOTS_MAX] = {};  // copies of a slot's piece under way
    int threads = 0;

    bool ready() {  // false: no pinned memory
        if (tried) return buf != nullptr;
        tried = true;
        bool ok = hipHostMalloc((void**)&buf, RING * sizeof(double), hipHostMallocDefault) == hipSuccess;
        for (auto& q : st) ok = ok && hipStreamCreateWithFlags(&q, hipStreamNonBlocking) == hipSuccess;
        for (auto& e : ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
        for (auto& e : chunk_ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
        ok = ok && hipEventCreateWithFlags(&ready_ev, hipEventDisableTiming) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            if (buf) (void)hipHostFree(buf);
            buf = nullptr;
            return false;
        }
        const unsigned hc = std::thread::hardware_concurrency();
        const int want = hc >= 16 ? 10 : (hc > 2 ? (int)hc - 1 : 1);
        for (; threads < want; ++threads) {
            try {
                std::thread([this] { loop(); }).detach();
            } catch (const std::system_error&) {
                break;
            }
        }
        if (threads == 0) {
            (void)hipHostFree(buf);
            buf = nullptr;
            return false;
        }
        return true;
    }
    void loop() {
        for (;;) {
            Job j;
            {
                std::unique_lock<std::mutex> lk(mu);
                work.wait(lk, [&] { return !jobs.empty(); });
                j = jobs.front();
                jobs.pop_front();
            }
            std::memcpy(j.dst, j.src, j.n * sizeof(double));
            bool last;
            {
                std::lock_guard<std::mutex> lk(mu);
                last = --busy[j.slot] == 0;
            }
            if (last) done.notify_all();
        }
    }
    void wait_slot(int s) {
        std::unique_lock<std::mutex> lk(mu);
        done.wait(lk, [&] { return busy[s] == 0; });
    }
    void wait_all() {
        for (int s = 0; s < SLOTS_MAX; ++s) wait_slot(s);
    }
    // A finished piece in parts that end at huge-page boundaries of the destination: each page is
    // then touched first, and cleared by the kernel, on one thread.
    void push(double* dst, const double* src, size_t n, int slot) {
        {
            std::lock_guard<std::mutex> lk(mu);
            while (n > 0) {
                const size_t to_page = (HUGE_PAGE - ((uintptr_t)dst & (HUGE_PAGE - 1)) + sizeof(double) - 1) / sizeof(double);
                size_t m = std::min(n, to_page);
                if (n - m < HUGE_PAGE / sizeof(double) / 8) m = n;  // no small remainder on its own
                jobs.push_back({dst, src, m, slot});
                ++busy[slot];
                dst += m; src += m; n -= m;
            }
        }
        work.notify_all();
    }
};
// Never destroyed: its threads may outlive the static objects of the process.
Ring& ring() {
    static Ring* r = new Ring;
    return *r;
}

void launch_rows(double* dst, const double* src, int G, int Np, int Nc, size_t c0, size_t nc, hipStream_t st) {
    constexpr size_t CELLS_MAX = (size_t)TILE << 15;  // a grid holds 65535 tiles along y
    for (size_t a = 0; a < nc; a += CELLS_MAX) {
        const size_t n = std::min(CELLS_MAX, nc - a);
        hipLaunchKernelGGL(flux_rows_kernel, dim3((unsigned)((G * Np + TILE - 1) / TILE), (unsigned)((n + TILE - 1) / TILE)),
                           dim3(256), 0, st, dst + a * G * Np, src, G, Np, Nc, (int)(c0 + a), (int)n);
    }
    RT_HIP(hipGetLastError());
}

// Without pinned memory, or with one cell's moments beyond a piece: staged on the device and copied
// into the caller's memory.
void direct_out(double* out, const double* phi, int G, int Np, int Nc, hipStream_t st) {
    const size_t per = (size_t)G * Np, cells = std::max<size_t>(1, std::min<size_t>(Nc, 4 * PIECE_MAX / per));
    double* tmp = (double*)dev_alloc(cells * per * sizeof(double));
    try {
        for (size_t c0 = 0; c0 < (size_t)Nc; c0 += cells) {
            const size_t nc = std::min(cells, (size_t)Nc - c0);
            launch_rows(tmp, phi, G, Np, Nc, c0, nc, st);
            RT_HIP(hipMemcpyAsync(out + c0 * per, tmp, nc * per * sizeof(double), hipMemcpyDeviceToHost, st));
        }
        RT_HIP(hipStreamSynchronize(st));
    } catch (...) {
        (void)hipStreamSynchronize(st);
        dev_free(tmp);
        throw;
    }
    dev_free(tmp);
}

// The kernels write the ring.
void link_out(Ring& r, double* out, const double* phi, int G, int Np, int Nc, size_t piece, hipStream_t st) {
    const size_t per = (size_t)G * Np;
    const size_t cells = std::min<size_t>(Nc, piece / per), np = (Nc + cells - 1) / cells;
    // a third of the ring is asked of the device ahead, the rest is being copied
    const size_t slots = std::min<size_t>(SLOTS_MAX, RING / piece), ahead = slots / 3;
    size_t issued = 0;
    RT_HIP(hipEventRecord(r.ready_ev, st));
    for (int q = 0; q < STREAMS; ++q) RT_HIP(hipStreamWaitEvent(r.st[q], r.ready_ev, 0));
    for (size_t k = 0; k < np; ++k) {
        // each once its slot's last piece, slots - ahead before the one waited for, is copied out
        for (; issued < np && issued < k + ahead; ++issued) {
            const int s = (int)(issued % slots);
            r.wait_slot(s);
            const size_t c0 = issued * cells;
            hipStream_t q = r.st[issued % STREAMS];
            launch_rows(r.buf + s * piece, phi, G, Np, Nc, c0, std::min(cells, (size_t)Nc - c0), q);
            RT_HIP(hipEventRecord(r.ev[s], q));
        }
        const int s = (int)(k % slots);
        RT_HIP(hipEventSynchronize(r.ev[s]));
        const size_t c0 = k * cells, n = std::min(cells, (size_t)Nc - c0) * per;
        if (np == 1 && n <= HUGE_PAGE / 4 / sizeof(double)) std::memcpy(out, r.buf + s * piece, n * sizeof(double));
        else r.push(out + c0 * per, r.buf + s * piece, n, s);
    }
    r.wait_all();
}

// The copy engines write the ring, from chunks of whole pieces rearranged on the device (two of at most
// chunk doubles, in the scratch).  Nothing that waits for a copy goes onto a stream, where it would hold up
// the others of its hardware queue: a piece is waited for on its stream, which nothing else uses, instead
// of by an event behind it (with events 4.03 GB took 167-202 ms from the server and 191 beside the
// threads), and a chunk's kernel is launched once the host has seen the chunk before the last emptied.
void engine_out(Ring& r, double* out, const double* phi, int G, int Np, int Nc, size_t piece, const FluxScratch& tmp,
                size_t chunk, hipStream_t st) {
    const size_t per = (size_t)G * Np;
    const size_t cells = std::min<size_t>(Nc, piece / per), np = (Nc + cells - 1) / cells;
    const size_t slots = std::min<size_t>(SLOTS_MAX, RING / piece);
    const size_t cp = chunk / piece, nch = (np + cp - 1) / cp;  // pieces per chunk, chunks
    size_t launched = 0, issued = 0;
    auto rearrange = [&] {  // the next chunk
        const size_t c0 = launched * cp * cells, c1 = std::min<size_t>(Nc, c0 + cp * cells);
        launch_rows(tmp.p[launched & 1], phi, G, Np, Nc, c0, c1 - c0, st);
        RT_HIP(hipEventRecord(r.chunk_ev[launched & 1], st));
        ++launched;
    };
    rearrange();
    if (nch > 1) rearrange();
    for (size_t k = 0; k < np; ++k) {
        for (; issued < std::min(np, launched * cp) && issued < k + STREAMS; ++issued) {
            const size_t c = issued / cp;
            if (issued == c * cp) RT_HIP(hipEventSynchronize(r.chunk_ev[c & 1]));
            const int s = (int)(issued % slots);
            r.wait_slot(s);
            const size_t n = std::min(cells, (size_t)Nc - issued * cells) * per;
            RT_HIP(hipMemcpyAsync(r.buf + s * piece, tmp.p[c & 1] + (issued - c * cp) * cells * per,
                                  n * sizeof(double), hipMemcpyDeviceToHost, r.st[issued % STREAMS]));
        }
        RT_HIP(hipStreamSynchronize(r.st[k % STREAMS]));
        const int s = (int)(k % slots);
        const size_t c0 = k * cells, n = std::min(cells, (size_t)Nc - c0) * per;
        r.push(out + c0 * per, r.buf + s * piece, n, s);
        if ((k + 1) % cp == 0 && launched < nch) rearrange();  // chunk (k + 1) / cp - 1 is empty
    }
    r.wait_all();
}

}  // namespace

void flux_to_host(double* out, const double* phi, int G, int Np, int Nc, FluxWay way, const FluxScratch& scratch,
                  hipStream_t st) {
    const size_t per = (size_t)G * Np, total = per * Nc;
    Ring& r = ring();
    std::unique_lock<std::mutex> lk(r.use);  // held to the end: the calls on one problem share its scratch
    // beside other work one launch for what fits a piece, as each waits its turn; chunks where the
    // scratch holds them
    const size_t chunk = std::min(CHUNK_MAX, scratch.n);
    const bool engine = way == FLUX_ENGINE && total > PIECE_MAX && chunk >= std::max(CHUNK_MIN, per);
    const size_t piece = engine ? std::min(PIECE_MAX, chunk)
                                : std::max(way == FLUX_ENGINE ? PIECE_MAX : piece_size(total), std::min(per, PIECE_MAX));
    if (way == FLUX_DIRECT || per > piece || !r.ready()) {
        lk.unlock();
        direct_out(out, phi, G, Np, Nc, st);
        return;
    }
    try {
        if (engine) engine_out(r, out, phi, G, Np, Nc, piece, scratch, chunk, st);
        else link_out(r, out, phi, G, Np, Nc, piece, st);
    } catch (...) {
        (void)hipStreamSynchronize(st);
        for (auto q : r.st) (void)hipStreamSynchronize(q);
        r.wait_all();
        throw;
    }
}

void test_flux_out(int way, int G, int Np, int Nc, const double* phi, size_t chunk, double* out) {
    const size_t bytes = (size_t)G * Np * Nc * sizeof(double);
    double* d = (double*)dev_alloc(bytes);
    FluxScratch s{{nullptr, nullptr}, chunk};
    auto free_all = [&] {
        for (double* p : s.p) dev_free(p);
        dev_free(d);
    };
    try {
        if (chunk > 0)
            for (double*& p : s.p) p = (double*)dev_alloc(chunk * sizeof(double));
        RT_HIP(hipMemcpy(d, phi, bytes, hipMemcpyHostToDevice));
        flux_to_host(out, d, G, Np, Nc, (FluxWay)way, s, nullptr);
    } catch (...) {
        free_all();
        throw;
    }
    free_all();
}

}  // namespace rt
