// Host-to-device uploads through a ring of page-locked chunks (HostStager).
#include "host_stage.hpp"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <thread>

#include "engine.hpp"

namespace vship {

HostMem host_memory_kind(const void* p, size_t bytes) {
    if (!p || bytes == 0) return HostMem::Pageable;
    const uint8_t* b = static_cast<const uint8_t*>(p);
    bool locked = true;
    for (const uint8_t* q : {b, b + bytes - 1}) {
        hipPointerAttribute_t attr;
        if (hipPointerGetAttributes(&attr, q) != hipSuccess) {
            (void)hipGetLastError();  // pageable memory: the query fails and leaves its error behind
            locked = false;
            continue;
        }
        if (q == b && attr.type == hipMemoryTypeDevice) return HostMem::Device;
        if (attr.type != hipMemoryTypeHost) locked = false;
    }
    return locked ? HostMem::PageLocked : HostMem::Pageable;
}

UploadPlan plan_upload(const uint8_t* const* src, const size_t* bytes, int n) {
    constexpr size_t kAlign = 256, kMaxGap = 64 << 10;
    UploadPlan P;
    P.off.resize(n);
    size_t total = 0;
    for (int i = 0; i < n;) {
        if (!src[i] || bytes[i] == 0) VSHIP_THROW(E_BadPointer);
        const HostMem kind = host_memory_kind(src[i], bytes[i]);
        if (kind == HostMem::Device) VSHIP_THROW(E_BadPointer);
        UploadPlan::Run r{src[i], bytes[i], (total + kAlign - 1) / kAlign * kAlign, kind == HostMem::PageLocked};
        P.off[i] = r.off;
        int j = i + 1;
        if (r.locked) {
            hipDeviceptr_t base = nullptr;
            size_t size = 0;
            if (hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)src[i]) != hipSuccess) {
                (void)hipGetLastError();
                size = 0;
            }
            const uint8_t* lo = static_cast<const uint8_t*>(base);
            const uint8_t* hi = lo + size;
            if (size == 0 || r.src < lo || r.src + r.bytes > hi) hi = lo = nullptr;
            for (; lo && j < n; j++) {
                const uint8_t* s = src[j];
                const uint8_t* prev_end = r.src + r.bytes;
                if (!s || bytes[j] == 0 || s < prev_end || (size_t)(s - prev_end) > kMaxGap ||
                    (size_t)(s - r.src) % kAlign != 0 || s + bytes[j] > hi)
                    break;
                P.off[j] = r.off + (size_t)(s - r.src);
                r.bytes = (size_t)(s + bytes[j] - r.src);
            }
        }
        P.runs.push_back(r);
        total = r.off + r.bytes;
        i = j;
    }
    P.total = total;
    return P;
}

namespace {

// The helpers of the stagers without threads of their own. Three beside the
// caller saturate PCIe from pageable memory (a CPU thread copies about 25 GB/s of its
// 57), and as there is one team, many handles on many threads still make only
// three extra threads: one upload has them, the others copy alone.
std::shared_ptr<CopyTeam> shared_team() {
    static std::mutex mu;
    static std::weak_ptr<CopyTeam> team;
    std::lock_guard<std::mutex> lk(mu);
    std::shared_ptr<CopyTeam> t = team.lock();
    if (!t) {
        const int cpus = (int)std::thread::hardware_concurrency();
        t = std::make_shared<CopyTeam>(std::min(3, std::max(0, cpus - 1)));
        team = t;
    }
    return t;
}

// Bytes between a chunk of the ring and device memory, by a kernel in the
// stream itself: a DMA and its hand-over to the kernels behind it cost about
// 20 us each besides the bytes (measured at 1, 2 and 4 MiB), more than a small
// picture's whole upload. Bound by PCIe; 64 workgroups keep 256 KiB of 16-byte
// accesses in flight, several times what the link's latency needs. Where several
// Butteraugli handles work at once, one that finds the helpers taken, as most do,
// uses the DMA engines instead: the link is never idle there, and the kernel would
// wait for CUs behind the other handles' stages (300 us of them per 1080p pair)
// and hold them up. 1920 x 1080 float pairs with maps, per call: one handle
// 1,765 us by the kernel and 1,975 by DMA, eight handles on eight threads 1,150
// and 1,025. SSIMULACRA2's kernels are done in 75 us: eight threads 923 by the
// kernel and 904 by DMA, but eight streams of the video filter 940 and 910 pairs/s,
// so its handles stay with the kernel.
constexpr int kMoveGroups = 64;
__global__ __launch_bounds__(256) void move_kernel(uint8_t* __restrict__ dst, const uint8_t* __restrict__ src,
                                                   size_t bytes) {
    const size_t n16 = bytes / 16, step = (size_t)gridDim.x * 256, t = (size_t)blockIdx.x * 256 + threadIdx.x;
    for (size_t i = t; i < n16; i += step)
        reinterpret_cast<uint4*>(dst)[i] = reinterpret_cast<const uint4*>(src)[i];
    for (size_t i = 16 * n16 + t; i < bytes; i += step) dst[i] = src[i];
}

// dst and src 16-byte aligned, one of them in page-locked memory
void move_chunk(void* dst, const void* src, size_t bytes, hipStream_t st) {
    const int groups = (int)std::min<size_t>(kMoveGroups, (bytes / 16 + 255) / 256 + 1);
    move_kernel<<<groups, 256, 0, st>>>(static_cast<uint8_t*>(dst), static_cast<const uint8_t*>(src), bytes);
    HIP_OR_THROW(hipGetLastError(), E_BadDeviceCode);
}

constexpr size_t kPiece = 256 << 10;     // bytes a thread copies at a time
constexpr size_t kSharedMin = 1 << 20;   // below it, waking the helpers costs more than it saves

}  // namespace

HostStager::HostStager(int device, size_t chunk_bytes, int slots, int threads, bool dma_when_taken)
    : shared_(threads == 0), dma_when_taken_(dma_when_taken) {
    HIP_OR_THROW(hipSetDevice(device), E_BadDeviceArgument);
    chunk_ = std::max<size_t>(chunk_bytes / 4096 * 4096, 4096);
    slots = std::max(slots, 2);
    try {
        for (int i = 0; i < slots; i++) {
            void* p = nullptr;
            HIP_OR_THROW(hipHostMalloc(&p, chunk_, hipHostMallocDefault), E_OutOfRAM);
            ring_.push_back(static_cast<uint8_t*>(p));
            hipEvent_t e = nullptr;
            HIP_OR_THROW(hipEventCreateWithFlags(&e, hipEventDisableTiming), E_OutOfRAM);
            ev_.push_back(e);
        }
        if (threads > 1) pool_ = new ParallelCopy(threads);
    } catch (...) {
        release();
        throw;
    }
}

HostStager::~HostStager() { release(); }

void HostStager::release() {
    for (hipEvent_t e : ev_) {
        (void)hipEventSynchronize(e);
        (void)hipEventDestroy(e);
    }
    for (uint8_t* p : ring_) (void)hipHostFree(p);
    ev_.clear();
    ring_.clear();
    delete pool_;
    pool_ = nullptr;
}

void HostStager::upload(uint8_t* dst_base, const UploadPlan& plan, hipStream_t st) {
    if (!dst_base) VSHIP_THROW(E_BadPointer);
    if (shared_) return upload_shared(dst_base, plan, st);
    // the open chunk: slot k holds device bytes [c0, c0 + fill)
    int k = -1;
    size_t c0 = 0, fill = 0;
    std::vector<CopySeg> segs;
    auto flush = [&] {
        if (k < 0) return;
        if (pool_)
            pool_->copy(segs.data(), (int)segs.size());
        else
            copy_seg_range(segs.data(), (int)segs.size(), 0, SIZE_MAX);
        HIP_OR_THROW(hipMemcpyAsync(dst_base + c0, ring_[k], fill, hipMemcpyHostToDevice, st), E_BadPointer);
        HIP_OR_THROW(hipEventRecord(ev_[k], st), E_BadDeviceCode);
        k = -1;
        segs.clear();
    };
    for (const UploadPlan::Run& r : plan.runs) {
        if (r.locked) {
            flush();
            HIP_OR_THROW(hipMemcpyAsync(dst_base + r.off, r.src, r.bytes, hipMemcpyHostToDevice, st), E_BadPointer);
            direct_bytes_ += r.bytes;
            continue;
        }
        for (size_t done = 0; done < r.bytes;) {
            const size_t dpos = r.off + done;
            if (k >= 0 && dpos >= c0 + chunk_) flush();
            if (k < 0) {
                k = next_;
                next_ = (next_ + 1) % (int)ring_.size();
                // the slot's previous DMA has to have read it before it is refilled
                HIP_OR_THROW(hipEventSynchronize(ev_[k]), E_BadDeviceCode);
                c0 = dpos;
                fill = 0;
            }
            const size_t n = std::min(r.bytes - done, c0 + chunk_ - dpos);
            segs.push_back({ring_[k] + (dpos - c0), r.src + done, n});
            fill = dpos - c0 + n;
            done += n;
            if (fill == chunk_) flush();
        }
        pageable_bytes_ += r.bytes;
    }
    flush();
}

CopyTeam& HostStager::team_for(size_t bytes) {
    static CopyTeam nobody(0);
    if (!shared_ || bytes < kSharedMin) return nobody;
    if (!team_) team_ = shared_team();
    return *team_;
}

void HostStager::upload_shared(uint8_t* dst_base, const UploadPlan& plan, hipStream_t st) {
    // chunks of the ring, each a device range of whole or partial runs
    struct Chunk {
        size_t off, bytes;
    };
    std::vector<Chunk> chunks;
    std::vector<CopyTeam::Piece> pieces;
    bool open = false;  // the last chunk may take the next run (no page-locked run lies between)
    for (const UploadPlan::Run& r : plan.runs) {
        if (r.locked) {
            HIP_OR_THROW(hipMemcpyAsync(dst_base + r.off, r.src, r.bytes, hipMemcpyHostToDevice, st), E_BadPointer);
            direct_bytes_ += r.bytes;
            open = false;
            continue;
        }
        for (size_t done = 0; done < r.bytes;) {
            const size_t dpos = r.off + done;
            if (!open || dpos >= chunks.back().off + chunk_) chunks.push_back({dpos, 0});
            open = true;
            Chunk& c = chunks.back();
            const size_t n = std::min({r.bytes - done, c.off + chunk_ - dpos, kPiece});
            const int slot = (next_ + (int)chunks.size() - 1) % (int)ring_.size();
            pieces.push_back({ring_[slot] + (dpos - c.off), r.src + done, n, (int)chunks.size() - 1});
            c.bytes = dpos - c.off + n;
            done += n;
        }
        pageable_bytes_ += r.bytes;
    }
    if (chunks.empty()) return;
    const int nslots = (int)ring_.size(), n = (int)chunks.size(), first = next_;
    next_ = (first + n) % nslots;
    CopyTeam& team = team_for(plan.total);
    const bool dma = dma_when_taken_ && team.taken();
    team.run(
        pieces, n, nslots,
        [&](int c, bool wait) {
            // the slot's previous move has to have read it before it is refilled
            hipEvent_t e = ev_[(first + c) % nslots];
            if (!wait) return hipEventQuery(e) == hipSuccess;
            HIP_OR_THROW(hipEventSynchronize(e), E_BadDeviceCode);
            return true;
        },
        [&](int c) {
            const int k = (first + c) % nslots;
            void* to = dst_base + chunks[c].off;
            if (dma)
                HIP_OR_THROW(hipMemcpyAsync(to, ring_[k], chunks[c].bytes, hipMemcpyHostToDevice, st), E_BadPointer);
            else
                move_chunk(to, ring_[k], chunks[c].bytes, st);
            HIP_OR_THROW(hipEventRecord(ev_[k], st), E_BadDeviceCode);
        });
}

void HostStager::download_rows(void* dst, int64_t dst_stride, const void* src, int64_t src_stride,
                               size_t row_bytes, int rows, hipStream_t st) {
    if (rows < 1 || row_bytes == 0) return;
    if (!dst || !src || dst_stride < (int64_t)row_bytes || src_stride < (int64_t)row_bytes)
        VSHIP_THROW(E_BadPointer);
    uint8_t* d = static_cast<uint8_t*>(dst);
    const uint8_t* s = static_cast<const uint8_t*>(src);
    const HostMem kind = host_memory_kind(d, (size_t)dst_stride * (rows - 1) + row_bytes);
    if (kind == HostMem::Device) VSHIP_THROW(E_BadPointer);
    if (kind == HostMem::PageLocked) {
        HIP_OR_THROW(hipMemcpy2DAsync(d, dst_stride, s, src_stride, row_bytes, rows, hipMemcpyDeviceToHost, st),
                     E_BadPointer);
        HIP_OR_THROW(hipStreamSynchronize(st), E_BadPointer);
        direct_bytes_ += row_bytes * rows;
        return;
    }
    if (row_bytes > chunk_) {  // a row of over half a million samples
        HIP_OR_THROW(hipStreamSynchronize(st), E_BadPointer);
        HIP_OR_THROW(hipMemcpy2D(d, dst_stride, s, src_stride, row_bytes, rows, hipMemcpyDeviceToHost), E_BadPointer);
        pageable_bytes_ += row_bytes * rows;
        return;
    }
    const int per = (int)std::min<size_t>(chunk_ / row_bytes, (size_t)rows);
    const int nchunks = (rows + per - 1) / per;
    const int nslots = (int)ring_.size();
    CopyTeam& team = team_for(row_bytes * rows);
    const bool dma = !shared_ || (dma_when_taken_ && team.taken());
    // chunk c goes through slot (next_ + c) % nslots; up to nslots ahead
    auto enqueue = [&](int c) {
        const int k = (next_ + c) % nslots;
        const int r0 = c * per, n = std::min(per, rows - r0);
        HIP_OR_THROW(hipEventSynchronize(ev_[k]), E_BadDeviceCode);
        const uint8_t* from = s + (int64_t)r0 * src_stride;
        if (!dma && src_stride == (int64_t)row_bytes && reinterpret_cast<uintptr_t>(from) % 16 == 0)
            move_chunk(ring_[k], from, row_bytes * n, st);
        else
            HIP_OR_THROW(hipMemcpy2DAsync(ring_[k], row_bytes, from, src_stride, row_bytes, n, hipMemcpyDeviceToHost, st),
                         E_BadPointer);
        HIP_OR_THROW(hipEventRecord(ev_[k], st), E_BadDeviceCode);
    };
    for (int c = 0; c < std::min(nchunks, nslots); c++) enqueue(c);
    // pieces of whole rows, copied out of a chunk once it has arrived
    std::vector<CopyTeam::Piece> pieces;
    const int piece_rows = std::max(1, (int)(kPiece / row_bytes));
    for (int c = 0; c < nchunks; c++)
        for (int r = c * per; r < std::min(rows, (c + 1) * per); r += piece_rows) {
            const int n = std::min(piece_rows, std::min(rows, (c + 1) * per) - r);
            CopyTeam::Piece p{d + (int64_t)r * dst_stride, ring_[(next_ + c) % nslots] + row_bytes * (r - c * per),
                              row_bytes, c};
            if (dst_stride == (int64_t)row_bytes) {
                p.bytes = row_bytes * n;
            } else {
                p.rows = n;
                p.dst_stride = dst_stride;
                p.src_stride = (int64_t)row_bytes;
            }
            pieces.push_back(p);
        }
    auto arrived = [&](int c, bool wait) {
        hipEvent_t e = ev_[(next_ + c) % nslots];
        if (!wait) return hipEventQuery(e) == hipSuccess;
        HIP_OR_THROW(hipEventSynchronize(e), E_BadDeviceCode);
        return true;
    };
    auto copied = [&](int c) {
        if (c + nslots < nchunks) enqueue(c + nslots);
    };
    team.run(pieces, nchunks, nslots, arrived, copied);
    next_ = (next_ + nchunks) % nslots;
    pageable_bytes_ += row_bytes * rows;
}

}  // namespace vship
