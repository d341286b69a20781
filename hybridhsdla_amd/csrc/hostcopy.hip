// Copies between device memory and pageable host memory.
//
// The runtime's own copies from and to pageable memory reach 10 (fresh pages)
// and 23 GB/s here, pinned ones 56.  So everything goes through a ring of
// pinned slots: a small copy kernel per slot on the one side, several threads on
// the other, the calling thread in between, which launches the kernel of a slot
// when it may be overwritten (or has been filled) and hands it on when it has
// landed.
// Why a kernel: hipMemcpyAsync and an event per slot cost 8 to 10 us beside the
// bytes (43 GB/s in slots of 2 MiB, 48 in 4, 51 in 8), and a lower triangle is a
// rectangle to it; the kernel takes each column from its diagonal on and says
// itself, in pinned memory, when a slot has landed.  To the host three slots per
// launch (62 MB in 1230 us; one: 1370); from it a slot as soon as it is filled.
// Few workgroups: the link takes slots of 4 MiB at 52 GB/s to the host and 53 from
// it with 24, 51 and 48 with 64, 44 and 34 with 256.
// Threads matter most where the host pages are fresh: one thread writes them at
// 15 GB/s, eight at 65, more not faster.  The last slot's host side overlaps
// nothing, so slots are small.
// Measured, whole calls, the runtime's copies before: A and B of 16 atoms at
// N_G 1500 (62 MB) 5.0-5.8 -> 1.3-1.7 ms (over boards); H and S at N_G 1201 (46 MB, both triangles)
// 2.87 -> 1.45 ms; the contraction of given coefficients at N_G 1500 (62 MB in,
// two lower triangles out) 7.7 -> 4.9 ms, 3.4 with M built on the GPU and S's copy
// beside H.
#include <sys/mman.h>

#include <algorithm>
#include <cstring>
#include <thread>

#include "hsgen_host.h"

namespace hsgen {

namespace {

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23
#endif

constexpr size_t kSlotBytes = (size_t)4 << 20;
constexpr size_t kPieceBytes = (size_t)256 << 10;    // what a thread copies at a time
constexpr size_t kThreadBytes = (size_t)512 << 10;   // one more thread per so many bytes
constexpr size_t kFlagBytes = 64 * (kRingSlots + 1); // one line per slot, after the slots, and one for the start
constexpr size_t kGrid = 24;                         // workgroups of a copy kernel
constexpr int kGroup = kRingSlots / 2;               // slots of one launch
constexpr size_t kRange = (size_t)2 << 20;           // memory that Prefault maps at a time

// What one slot holds and one kernel moves: `height` columns of `width` bytes,
// column c from byte 16 c * lower on.
struct Block {
    char* dev;
    size_t width, dpitch;
    int height, lower;
    int npieces;
};

// A block's kernel.  Bound by the link; 16 bytes per lane and access, four in
// flight.  The last workgroup to finish tells the host.
struct SlotCopy {
    char* dev;
    char* slot;
    size_t width, dpitch;
    int32_t height, lower;
    uint32_t* left;         // workgroups that finished, zero between launches
    uint64_t* flag;         // pinned: takes seq
    uint64_t seq;
};

typedef double v2d __attribute__((ext_vector_type(2)));

struct SlotGroup {
    SlotCopy c[kGroup];
    uint64_t* begun;        // pinned: takes the first block's seq as the kernel starts
    int32_t n;
};

// units of 16 bytes [first, n) of one column, `stride` lanes side by side
__device__ __forceinline__ void copy_units(const char* src, char* dst, uint32_t first, uint32_t n, uint32_t stride)
{
    const v2d* s = (const v2d*)src;
    v2d* d = (v2d*)dst;
    for (uint32_t u0 = first; u0 < n; u0 += 4 * stride) {
        v2d v[4];
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            if (u0 + i * stride < n) v[i] = s[u0 + i * stride];
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            if (u0 + i * stride < n) d[u0 + i * stride] = v[i];
    }
}

template <bool kToHost>
__global__ __launch_bounds__(256) void k_slot_copy(SlotGroup g)
{
    if (blockIdx.x == 0 && threadIdx.x == 0)
        __hip_atomic_store(g.begun, g.c[0].seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    for (int b = 0; b < g.n; ++b) {
        const SlotCopy& p = g.c[b];
        const uint32_t w = (uint32_t)(p.width / 16);
        if (p.height == 1) {             // a run: all workgroups side by side
            copy_units(kToHost ? p.dev : p.slot, kToHost ? p.slot : p.dev, blockIdx.x * 256 + threadIdx.x, w,
                       gridDim.x * 256);
            if (p.width % 16 && blockIdx.x == 0 && threadIdx.x == 0) {     // a multiple of 8 bytes
                const size_t o = p.width - 8;
                if (kToHost) *(double*)(p.slot + o) = *(const double*)(p.dev + o);
                else *(double*)(p.dev + o) = *(const double*)(p.slot + o);
            }
        } else {
            for (int c = blockIdx.x; c < p.height; c += gridDim.x) {
                char* d = p.dev + c * p.dpitch;
                char* s = p.slot + c * p.width;
                copy_units(kToHost ? d : s, kToHost ? s : d, (p.lower ? c : 0) + threadIdx.x, w, 256);
            }
        }
        __threadfence_system();
        __syncthreads();
        if (threadIdx.x == 0 && atomicAdd(p.left, 1u) == gridDim.x - 1) {
            *p.left = 0;
            __hip_atomic_store(p.flag, p.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

// What a thread copies at a time: `cols` columns of a slot, column c from byte
// c * skip on.
struct Piece {
    int block;
    char* host;
    size_t at;                        // of its first byte in the slot
    size_t width, spitch, hpitch;     // spitch, hpitch: of the slot's and the host's columns
    int cols, skip;
    size_t lead;                      // bytes above the first column's part
    bool clear;                       // and whether they (and skipped ones) become zero
};

void copy_piece(const Piece& p, char* slot, bool to_host)
{
    for (int c = 0; c < p.cols; ++c) {
        const size_t off = (size_t)c * p.skip;
        char* h = p.host + c * p.hpitch + off;
        char* s = slot + p.at + c * p.spitch + off;
        if (p.clear) std::memset(h - p.lead - off, 0, p.lead + off);
        if (to_host) std::memcpy(h, s, p.width - off);
        else std::memcpy(s, h, p.width - off);
    }
}

struct Plan {
    std::vector<Block> blocks;
    std::vector<Piece> pieces;
    size_t bytes = 0;

    // one run of memory; it shares a block with the run before it on the device
    void add_run(char* dev, char* host, size_t n)
    {
        bytes += n;
        while (n > 0) {
            Block* b = blocks.empty() ? nullptr : &blocks.back();
            size_t at = 0;
            if (b && b->height == 1 && dev == b->dev + b->width && b->width % 16 == 0 && b->width < kSlotBytes) {
                at = b->width;
            } else {
                blocks.push_back(Block{dev, 0, 0, 1, 0, 0});
                b = &blocks.back();
            }
            const size_t m = std::min(std::min(n, kPieceBytes), kSlotBytes - at);
            pieces.push_back(Piece{(int)blocks.size() - 1, host, at, m, 0, 0, 1, 0, 0, false});
            b->width = at + m;
            ++b->npieces;
            dev += m;
            host += m;
            n -= m;
        }
    }

    void add(const HostCopy& h)
    {
        if (h.rows == 0 || h.cols == 0) return;
        if (!h.lower && ((h.ldd == h.rows && h.ldh == h.rows) || h.cols == 1)) {
            add_run(h.dev, h.host, h.rows * h.cols);
            return;
        }
        const size_t e = sizeof(double2);
        for (size_t j = 0; j < h.cols;) {
            const size_t i0 = h.lower ? j * e : 0, width = h.rows - i0;
            char* dev = h.dev + j * h.ldd + i0;
            char* host = h.host + j * h.ldh + i0;
            if (width > kSlotBytes) {
                if (h.lower && h.clear) std::memset(host - i0, 0, i0);
                add_run(dev, host, width);
                ++j;
                continue;
            }
            const int height = (int)std::min(h.cols - j, kSlotBytes / width);
            blocks.push_back(Block{dev, width, h.ldd, height, h.lower, 0});
            const int step = (int)std::max<size_t>(1, kPieceBytes / width);
            for (int c = 0; c < height; c += step) {
                const size_t off = h.lower ? c * e : 0;
                pieces.push_back(Piece{(int)blocks.size() - 1, host + c * h.ldh + off, c * width + off, width - off, width,
                                       h.ldh, std::min(step, height - c), h.lower ? (int)e : 0,
                                       i0 + off, h.lower && h.clear});
                ++blocks.back().npieces;
            }
            bytes += width * height;
            j += height;
        }
    }
};

// memory [p, p + n) in ranges of whole pages
void add_range(std::vector<std::pair<char*, size_t>>& out, char* p, size_t n)
{
    const uintptr_t page = 4096;
    uintptr_t a = (uintptr_t)p & ~(page - 1);
    const uintptr_t e = ((uintptr_t)p + n + page - 1) & ~(page - 1);
    for (; a < e; a += kRange) out.emplace_back((char*)a, std::min<size_t>(kRange, e - a));
}

}  // namespace

// ---------------------------------------------------------------------------
// Threads
// ---------------------------------------------------------------------------
// the context's threads; null: the calling thread works alone
static HostPool* pool(hsgen_ctx* ctx, size_t bytes)
{
    if (bytes < kThreadBytes) return nullptr;
    if (!ctx->pool) ctx->pool.reset(new HostPool);
    return ctx->pool->size() > 0 ? ctx->pool.get() : nullptr;
}

// Maps the pages of host results while the GPU computes them: fresh memory is
// zeroed by the first access, at 35 GB/s per thread and at most 60 in all
// (four threads), about the rate of the copy that would wait for it.  No byte
// changes.
Prefault::Prefault(hsgen_ctx* ctx, const std::vector<HostCopy>& list) : ctx_(ctx)
{
    if (ctx->prefault) return;           // the caller's works on the same memory
    size_t bytes = 0;
    for (const HostCopy& h : list) {
        // columns with little above their diagonal as one piece of memory
        const size_t step = h.lower && !h.clear ? ((size_t)64 << 10) / sizeof(double2) : h.cols;
        for (size_t j = 0; j < h.cols;) {
            const size_t i0 = h.lower && !h.clear ? j * sizeof(double2) : 0;
            const size_t m = j < step ? std::min(step, h.cols) : 1;
            add_range(ranges_, h.host + j * h.ldh + i0, (m - 1) * h.ldh + h.rows - i0);
            j += m;
        }
        bytes += h.rows * h.cols;
    }
    pool_ = bytes < kSlotBytes ? nullptr : pool(ctx, bytes);
    if (!pool_) return;
    ctx->prefault = this;
    pool_->post(
        this,
        [this] {
            while (!stop_.load(std::memory_order_relaxed)) {
                const size_t i = next_.fetch_add(1, std::memory_order_relaxed);
                if (i >= ranges_.size() || madvise(ranges_[i].first, ranges_[i].second, MADV_POPULATE_WRITE)) return;
            }
        },
        4);
}

Prefault::~Prefault()
{
    if (!pool_) return;
    stop();
    pool_->finish(this);
    ctx_->prefault = nullptr;
}

hsgen_status host_copy(hsgen_ctx* ctx, const std::vector<HostCopy>& list, bool to_host, hipStream_t stream, bool computed)
{
    constexpr int kN = kRingSlots;
    Plan plan;
    for (const HostCopy& h : list) plan.add(h);
    const std::vector<Block>& blocks = plan.blocks;
    const std::vector<Piece>& pieces = plan.pieces;
    const int n = (int)blocks.size();
    if (n == 0) return HSGEN_OK;
    if (!ctx->ring) {
        void* p = nullptr;
        hipError_t e = hipHostMalloc(&p, kSlotBytes * kN + kFlagBytes, hipHostMallocDefault);
        if (e == hipSuccess) e = hipHostGetDevicePointer(&ctx->ring_dev, p, 0);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            if (p) (void)hipHostFree(p);
            return fail(ctx, HSGEN_ERR_NOMEM, "hipHostMalloc(%zu bytes) failed: %s", kSlotBytes * kN + kFlagBytes,
                        hipGetErrorString(e));
        }
        std::memset((char*)p + kSlotBytes * kN, 0, kFlagBytes);
        ctx->ring = (char*)p;
    }
    if (!ctx->ring_left.p) {
        const hsgen_status st = ensure(ctx, ctx->ring_left, sizeof(uint32_t) * kN, true);
        if (st) return st;
        HIPCHK(hipStreamSynchronize(ctx->stream));
    }
    // an earlier copy to the device may still read the slots
    if (!to_host) HIPCHK(hipStreamSynchronize(stream));

    auto slot = [&](int b) { return ctx->ring + kSlotBytes * (size_t)(b % kN); };
    std::unique_ptr<std::atomic<int>[]> done(new std::atomic<int>[n]);    // pieces of a block that are copied
    for (int b = 0; b < n; ++b) done[b].store(0, std::memory_order_relaxed);
    std::atomic<size_t> next{0};        // piece to take
    std::atomic<int> ready{0};          // blocks whose slots the host side may touch
    std::atomic<bool> stop{false};
    auto take = [&](size_t i) {
        const Piece& p = pieces[i];
        copy_piece(p, slot(p.block), to_host);
        done[p.block].fetch_add(1, std::memory_order_release);
    };
    auto worker = [&] {
        for (;;) {
            const size_t i = next.fetch_add(1, std::memory_order_relaxed);
            if (i >= pieces.size()) return;
            while (ready.load(std::memory_order_acquire) <= pieces[i].block) {
                if (stop.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            take(i);
        }
    };
    auto copied = [&](int b) { return done[b].load(std::memory_order_acquire) == blocks[b].npieces; };
    // sequence numbers of the blocks' kernels: never used twice on a context
    const uint64_t seq0 = ctx->ring_seq + 1;
    ctx->ring_seq += n;
    // launches the kernel of blocks b .. b + m - 1
    auto move = [&](int b, int m) {
        SlotGroup g{};
        g.begun = (uint64_t*)((char*)ctx->ring_dev + kSlotBytes * kN + 64 * kN);
        size_t most = 0;
        for (g.n = 0; g.n < m; ++g.n) {
            const Block& k = blocks[b + g.n];
            const int i = (b + g.n) % kN;
            g.c[g.n] = SlotCopy{k.dev, (char*)ctx->ring_dev + kSlotBytes * i, k.width, k.dpitch, k.height, k.lower,
                                (uint32_t*)ctx->ring_left.p + i,
                                (uint64_t*)((char*)ctx->ring_dev + kSlotBytes * kN + 64 * i), seq0 + b + g.n};
            most = std::max(most, k.width * k.height);
        }
        const dim3 grid((unsigned)std::min<size_t>(kGrid, most / 16384 + 1));

        if (to_host) hipLaunchKernelGGL(k_slot_copy<true>, grid, dim3(256), 0, stream, g);
        else hipLaunchKernelGGL(k_slot_copy<false>, grid, dim3(256), 0, stream, g);
        return hipGetLastError();
    };
    auto flag = [&](int i) {
        return __atomic_load_n((const uint64_t*)(ctx->ring + kSlotBytes * kN + 64 * i), __ATOMIC_ACQUIRE);
    };
    auto landed = [&](int b) { return flag(b % kN) >= seq0 + b; };

    // While the stream still computes what is to be copied the threads sleep until
    // the first kernel starts: they would spin meanwhile.  Where it is done they
    // start at once, with the kernel's launch (H and S at N_G 1201: 1.44 ms, 1.51
    // with the kernel's start).
    hipError_t e = hipSuccess;
    int issued = 0, nready = 0, freed = 0;
    unsigned idle = 0;
    // to the host: whole groups, the rest at the end
    auto send = [&] {
        for (int m; e == hipSuccess && issued < n; issued += m) {
            m = std::min(kGroup, n - issued);
            if (issued + m > freed + kN) return;
            e = move(issued, m);
        }
    };
    if (to_host) {
        send();
    } else {
        nready = std::min(n, kN);
        ready.store(nready, std::memory_order_release);
    }
    HostPool* threads = pool(ctx, plan.bytes);
    bool posted = false;
    while (e == hipSuccess && (to_host ? freed < n : issued < n)) {
        if (!posted && (!to_host || computed || flag(kN) >= seq0 || landed(0))) {
            if (to_host && ctx->prefault) ctx->prefault->stop();
            if (threads) threads->post(&plan, worker, std::min(threads->size(), plan.bytes / kThreadBytes));
            posted = true;
        }
        if (to_host) {
            send();
        } else {
            while (e == hipSuccess && issued < n && copied(issued)) e = move(issued++, 1);
        }
        if (e != hipSuccess) break;
        // the oldest kernel: when it is done its block is copied out, or its slot filled again
        const int oldest = to_host ? nready : nready - kN;
        if (nready < n && oldest < issued) {
            if (landed(oldest)) {
                ready.store(++nready, std::memory_order_release);
                idle = 0;
            } else if (++idle % 4096 == 0) {
                // a stream that failed, or is done without the flag, ends the wait
                const hipError_t q = hipStreamQuery(stream);
                if (q == hipErrorNotReady) (void)hipGetLastError();
                else if (q != hipSuccess) e = q;
                else if (!landed(oldest)) e = hipErrorUnknown;
            }
        }
        // alone, or with a small copy's blocks all on their way, this thread copies
        // too (in a large one it hands on what lands: 1.45 ms at N_G 1201, 1.55 helping)
        if (!threads || (to_host && issued == n && plan.bytes <= 2 * kSlotBytes)) {
            size_t i = next.load(std::memory_order_relaxed);
            if (i < pieces.size() && pieces[i].block < nready && next.compare_exchange_strong(i, i + 1)) take(i);
        }
        while (to_host && freed < nready && copied(freed)) ++freed;
    }
    stop.store(true);
    if (threads) threads->finish(&plan);
    if (e != hipSuccess) (void)hipStreamSynchronize(stream);
    HIPCHK(e);
    return HSGEN_OK;
}

}  // namespace hsgen
