// Internal definitions shared by the backend's translation units: the opaque
// C ABI objects, device buffers, error handling and the table builder.
#pragma once
#include "device/physics.hpp"
#include "dxmc_hip.h"
#include "hostcopy.hpp"

#include <hip/hip_runtime.h>
#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <tuple>
#include <cmath>
#include <type_traits>
#include <vector>

namespace dxmc_backend {
// page-locked blocks from dxmc_hip_host_alloc; pinnedHost: whether
// [p, p + bytes) lies in one of them
void registerPinned(const void* p, size_t bytes);
bool unregisterPinned(const void* p);
bool pinnedHost(const void* p, size_t bytes);
}

struct dxmc_ctx;

namespace dxmc_backend {
// the calling thread's last failure message per context: with several
// threads on one context, each reads its own error
std::map<const dxmc_ctx*, std::string>& threadErrors();
}

struct dxmc_ctx {
    int device = 0;
    int numCU = 256;
    std::string arch;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    void* historyCounter = nullptr; // u64 work counter of the persistent kernel
    void* scratch = nullptr; // device address of the no-allocation run's scratch array (null: unavailable)
    // autotuner results per (world, tables, precision, low energy correction,
    // whether the world had codes)
    std::map<std::tuple<const void*, const void*, int, int, bool>, dxmc_run_cfg> tuned;
    // Held by every entry point for the whole call: the staging chunks, the
    // work counter, the autotuner map and the stream's order of a call's
    // steps are per context, so calls from several threads on one context
    // run one after the other (device work on the stream is ordered anyway).
    // Recursive: entry points call one another.
    std::recursive_mutex lock;

    int fail(int status, const std::string& msg)
    {
        dxmc_backend::threadErrors()[this] = msg;
        return status;
    }
    // records a HIP error, returns non-zero on failure
    int check(hipError_t e)
    {
        if (e == hipSuccess)
            return 0;
        return fail(DXMC_ERR_DEVICE, std::string("HIP error: ") + hipGetErrorString(e));
    }
    // Device memory is stream-ordered (hipMallocAsync / hipFreeAsync on the
    // context's stream, from the device's pool, which keeps freed blocks):
    // unlike hipFree, releasing memory then does not wait for the kernels
    // other contexts run on the same device.
    template <typename P>
    int alloc(P** p, size_t bytes)
    {
        void* q = nullptr;
        const hipError_t e = hipMallocAsync(&q, bytes ? bytes : 1, stream);
        if (e != hipSuccess) {
            hipGetLastError();
            return fail(DXMC_ERR_MEMORY, "device allocation of " + std::to_string(bytes) + " bytes failed");
        }
        *p = static_cast<P*>(q);
        return DXMC_OK;
    }
    void release(void* p)
    {
        if (p)
            hipFreeAsync(p, stream);
    }
    // Host transfers go through page-locked memory; from pageable memory the
    // runtime's own staging reaches a fraction of the link rate, and each
    // call of it waits. Small ones take turns in a ring that the context
    // holds from its creation: an upload returns once its bytes are in the
    // ring (a copy and a launch later the device has them), a download waits
    // once. Large ones go through two chunks, so the DMA of one overlaps the
    // host copy of the other; they are allocated at the context's first large
    // transfer. Chunks of 16 MiB copied by 8 threads bring 134 M voxels'
    // results (2.7 GB) to fresh host memory in 62 ms, 8 MiB by 4 threads in
    // 87; the link alone takes 49.
    static constexpr size_t RING_BYTES = size_t { 1 } << 20;
    static constexpr size_t STAGE_CHUNK = size_t { 16 } << 20;
    // bytes of a chunk in a transfer of 'total': below 22 MiB half chunks, so
    // that DMA and host copy still overlap (one array of 12 MiB down 0.36 ms
    // in one chunk, 0.31 in two; 15.9 MiB 0.46 and 0.41; three arrays of 20
    // MiB 0.54 as 16 + 4, 0.48 in three; of 24 MiB 0.58 and 0.62)
    static constexpr size_t chunkOf(size_t total) { return 8 * total < 11 * STAGE_CHUNK ? STAGE_CHUNK / 2 : STAGE_CHUNK; }
    unsigned char* ring = nullptr;
    size_t ringNext = 0;
    void* stage[2] = { nullptr, nullptr };
    hipEvent_t stageDone[2] = { nullptr, nullptr };
    // copy a chunk into or out of the staging memory on several host threads
    dxmc_backend::CopyHelpers helpers;

    bool staging()
    {
        if (stage[0])
            return true;
        for (int i = 0; i < 2; ++i)
            if (hipHostMalloc(&stage[i], STAGE_CHUNK, hipHostMallocDefault) != hipSuccess
                || hipEventCreateWithFlags(&stageDone[i], hipEventDisableTiming) != hipSuccess) {
                hipGetLastError();
                releaseStaging();
                return false;
            }
        helpers.start(); // without helpers the copies run on the calling thread
        return true;
    }
    void releaseStaging()
    {
        helpers.stop();
        for (int i = 0; i < 2; ++i) {
            if (stage[i])
                hipHostFree(stage[i]);
            if (stageDone[i])
                hipEventDestroy(stageDone[i]);
            stage[i] = nullptr;
            stageDone[i] = nullptr;
        }
    }
    // 'bytes' of the ring, free of transfers in flight; null when it has no
    // room for them at all (or could not be allocated)
    unsigned char* ringSpace(size_t bytes)
    {
        if (!ring || bytes > RING_BYTES)
            return nullptr;
        if (ringNext + bytes > RING_BYTES) {
            if (hipStreamSynchronize(stream) != hipSuccess)
                return nullptr; // (the transfer that follows reports it)
            ringNext = 0;
        }
        unsigned char* p = ring + ringNext;
        ringNext += (bytes + 63) & ~size_t { 63 };
        return p;
    }
    // host -> device on the stream; the host array may be freed on return
    int copy(void* dst, const void* src, size_t bytes)
    {
        if (bytes == 0)
            return DXMC_OK;
        if (unsigned char* p = ringSpace(bytes)) {
            std::memcpy(p, src, bytes);
            return check(hipMemcpyAsync(dst, p, bytes, hipMemcpyHostToDevice, stream));
        }
        if (dxmc_backend::pinnedHost(src, bytes) || !staging()) {
            if (int st = check(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream)))
                return st;
            return check(hipStreamSynchronize(stream));
        }
        const auto* from = static_cast<const char*>(src);
        auto* to = static_cast<char*>(dst);
        const size_t chunk = chunkOf(bytes);
        for (size_t off = 0, i = 0; off < bytes; off += chunk, ++i) {
            const int b = static_cast<int>(i & 1);
            const size_t len = std::min(chunk, bytes - off);
            // the chunk's previous DMA (two chunks back) has to be done
            if (i >= 2)
                if (int st = check(hipEventSynchronize(stageDone[b])))
                    return st;
            helpers.copy(stage[b], from + off, len);
            if (int st = check(hipMemcpyAsync(to + off, stage[b], len, hipMemcpyHostToDevice, stream)))
                return st;
            if (int st = check(hipEventRecord(stageDone[b], stream)))
                return st;
        }
        return check(hipStreamSynchronize(stream));
    }
    // one array of a download
    struct Fetch {
        void* dst;
        const void* src;
        size_t bytes;
    };
    // device -> host, complete on return. Arrays that fit the ring together go
    // through it; of others those in the caller's page-locked memory go direct,
    // each by itself, and the pageable ones as one stream of bytes.
    int download(const Fetch* list, int count)
    {
        size_t total = 0;
        for (int k = 0; k < count; ++k)
            total += list[k].bytes;
        if (total == 0)
            return DXMC_OK;
        if (unsigned char* p = ringSpace(total))
            return downloadRing(p, list, count);
        std::vector<Fetch> pageable;
        size_t pageableBytes = 0;
        for (int k = 0; k < count; ++k) {
            if (list[k].bytes && !dxmc_backend::pinnedHost(list[k].dst, list[k].bytes)) {
                pageable.push_back(list[k]);
                pageableBytes += list[k].bytes;
            } else if (int st = downloadDirect(list[k])) {
                return st;
            }
        }
        const int left = static_cast<int>(pageable.size());
        if (unsigned char* p = left ? ringSpace(pageableBytes) : nullptr)
            return downloadRing(p, pageable.data(), left); // waits for the direct ones too
        if (left && staging()) {
            if (int st = downloadChunks(pageable.data(), left, chunkOf(pageableBytes)))
                return st;
        } else {
            for (const Fetch& f : pageable)
                if (int st = downloadDirect(f))
                    return st;
        }
        return check(hipStreamSynchronize(stream));
    }
    // one array straight to its destination (on the stream, without a wait)
    int downloadDirect(const Fetch& f)
    {
        return f.bytes ? check(hipMemcpyAsync(f.dst, f.src, f.bytes, hipMemcpyDeviceToHost, stream)) : DXMC_OK;
    }
    // the arrays through 'p' in the ring
    int downloadRing(unsigned char* p, const Fetch* list, int count)
    {
        size_t off = 0;
        for (int k = 0; k < count; off += list[k++].bytes)
            if (int st = downloadDirect({ p + off, list[k].src, list[k].bytes }))
                return st;
        if (int st = check(hipStreamSynchronize(stream)))
            return st;
        off = 0;
        for (int k = 0; k < count; off += list[k++].bytes)
            if (list[k].bytes)
                std::memcpy(list[k].dst, p + off, list[k].bytes);
        return DXMC_OK;
    }
    // the arrays as one stream of bytes through the staging chunks
    int downloadChunks(const Fetch* list, int count, size_t chunk)
    {
        // chunks across the arrays: a chunk holds the end of one and the
        // start of the next
        std::vector<dxmc_backend::CopyHelpers::Block> parts[2];
        auto drain = [&](int b) {
            if (int st = check(hipEventSynchronize(stageDone[b])))
                return st;
            helpers.copy(parts[b].data(), static_cast<int>(parts[b].size()));
            parts[b].clear();
            return 0;
        };
        int array = 0;
        size_t done = 0; // of the current array
        for (int b = 0; array < count; b ^= 1) {
            size_t used = 0;
            while (array < count && used < chunk) {
                const Fetch& f = list[array];
                const size_t len = std::min(chunk - used, f.bytes - done);
                if (len) {
                    if (int st = check(hipMemcpyAsync(static_cast<char*>(stage[b]) + used, static_cast<const char*>(f.src) + done, len,
                            hipMemcpyDeviceToHost, stream)))
                        return st;
                    parts[b].push_back({ static_cast<char*>(f.dst) + done, static_cast<char*>(stage[b]) + used, len });
                }
                used += len;
                done += len;
                if (done == f.bytes) {
                    ++array;
                    done = 0;
                }
            }
            if (int st = check(hipEventRecord(stageDone[b], stream)))
                return st;
            // copy out the previous chunk while this one is in flight
            if (!parts[b ^ 1].empty())
                if (int st = drain(b ^ 1))
                    return st;
        }
        for (int b = 0; b < 2; ++b)
            if (!parts[b].empty())
                if (int st = drain(b))
                    return st;
        return DXMC_OK;
    }
    int download(void* dst, const void* src, size_t bytes)
    {
        const Fetch f { dst, src, bytes };
        return download(&f, 1);
    }
};

// serialises the calls on one context (see dxmc_ctx::lock)
#define DXMC_LOCK(ctx) std::lock_guard<std::recursive_mutex> dxmc_lock_((ctx)->lock)

#define DXMC_CHECK(ctx, expr)                      \
    do {                                           \
        if (int dxmc_st_ = (ctx)->check((expr))) \
            return dxmc_st_;                       \
    } while (0)

struct dxmc_world {
    dxmc_ctx* ctx = nullptr;
    uint64_t n = 0;
    uint32_t dims[3] = { 0, 0, 0 };
    double spacing[3] = { 0, 0, 0 };
    double extent[6] = { 0, 0, 0, 0, 0, 0 };
    uint32_t nMaterials = 0;
    bool hasMeasurement = false;
    std::vector<double> maxDensity; // per material, host copy
    void* material = nullptr; // u8[n]
    void* density = nullptr; // f64[n]
    void* measurement = nullptr; // u8[n] or null
    void* voxels = nullptr; // FP32 path: palette index (u8/u16) or uint2 record per voxel
    void* palette = nullptr; // uint2[nPalette] FP32 records, null for 8-byte voxels
    uint32_t voxelBytes = 8;
    uint32_t nPalette = 0;
    // Bounded-density code per voxel (u8/u16) and the interval of each code
    // (DensityBound[nCodes]); codeBytes 0: none. 8-byte-record worlds get
    // them at upload, palette worlds by a run, once runs pay for them (under
    // the context's lock, hence mutable).
    mutable void* codes = nullptr;
    mutable void* bounds = nullptr;
    mutable uint32_t codeBytes = 0;
    mutable uint32_t nCodes = 0;
    mutable bool codesTried = false; // palette worlds: the run-time build was done (or failed)
    mutable uint64_t codeHistories = 0; // palette worlds: histories of the large runs that could use codes
    // 1-byte code worlds: a 2-byte code per block of voxels (smallest |
    // largest code << 8 of a one-material block, else BLOCK_MIXED)
    mutable void* blocks = nullptr;
    mutable uint32_t blockDims[3] = { 0, 0, 0 };
    mutable uint32_t blockShift = 0; // block edge 2^blockShift voxels
    mutable uint32_t codeMul = 0; // 1-byte codes: (code * codeMul) >> CODE_MUL_SHIFT is the code's material
    // device bytes; read by dxmc_hip_world_bytes without the lock, while a
    // run on another thread may add a palette world's codes
    mutable std::atomic<uint64_t> bytes { 0 };
};

struct dxmc_tables {
    dxmc_ctx* ctx = nullptr;
    uint32_t nMaterials = 0, nSpectra = 0, nHeel = 0, nBowtie = 0;
    dxmc_dev::Tables<double> f64 {};
    dxmc_dev::Tables<float> f32 {};
    std::vector<void*> allocations;
};

struct dxmc_tally {
    dxmc_ctx* ctx = nullptr;
    uint64_t n = 0;
    // the transport accumulates into scores (VoxelScore[n]); normalisation
    // and download fill the per-voxel arrays from them
    void* scores = nullptr;
    void* dose = nullptr;
    void* nEvents = nullptr;
    void* variance = nullptr;
    // the arrays hold the scores (raw or normalised) since the last run or
    // reset
    mutable bool arraysCurrent = false;
};

namespace dxmc_backend {

void setGlobalError(const std::string& s);
const char* globalError();

// RAII device buffer for temporaries
struct DeviceBuffer {
    dxmc_ctx* c;
    void* p = nullptr;
    explicit DeviceBuffer(dxmc_ctx* ctx)
        : c(ctx)
    {
    }
    ~DeviceBuffer() { c->release(p); }
    DeviceBuffer(const DeviceBuffer&) = delete;
    DeviceBuffer& operator=(const DeviceBuffer&) = delete;
    int alloc(size_t bytes)
    {
        c->release(p);
        p = nullptr;
        return c->alloc(&p, bytes);
    }
    int upload(const void* src, size_t bytes)
    {
        if (int st = alloc(bytes))
            return st;
        return c->copy(p, src, bytes);
    }
    int zeros(size_t bytes)
    {
        if (int st = alloc(bytes))
            return st;
        return c->check(hipMemsetAsync(p, 0, bytes, c->stream));
    }
};

// a run's device inputs in one allocation: exposure records of the run's
// precision, history prefix sums, step/event counters
struct RunBuffers {
    DeviceBuffer block;
    size_t startAt = 0, countersAt = 0;
    std::vector<uint64_t> start;
    uint64_t totalHistories = 0;
    explicit RunBuffers(dxmc_ctx* c)
        : block(c)
    {
    }
    template <typename T>
    T* at(size_t offset) const { return reinterpret_cast<T*>(static_cast<unsigned char*>(block.p) + offset); }
};

// the linear voxel index fits 24-bit products (World::index24)
inline bool hasIndex24(const dxmc_world* w)
{
    const uint64_t slice = uint64_t(w->dims[0]) * w->dims[1];
    return slice < (uint64_t(1) << 24) && w->dims[2] < (uint32_t(1) << 24) && slice * w->dims[2] < (uint64_t(1) << 32);
}

template <typename T>
inline dxmc_dev::World<T> deviceWorld(const dxmc_world* w)
{
    dxmc_dev::World<T> d {};
    d.nx = w->dims[0];
    d.ny = w->dims[1];
    d.nz = w->dims[2];
    for (int i = 0; i < 3; ++i)
        d.spacing[i] = static_cast<T>(w->spacing[i]);
    if constexpr (std::is_same_v<T, double>) {
        for (int i = 0; i < 6; ++i)
            d.extent[i] = w->extent[i];
    } else {
        // the safe extent one ulp inside the grid, formed in T from the grid
        // bounds as World<T>::updateMatrixExtent does (world.hpp:55-67), so
        // that a position on a voxel face indexes the voxel below it
        for (int i = 0; i < 3; ++i) {
            const T lower = static_cast<T>(std::nextafter(w->extent[2 * i], -HUGE_VAL));
            const T upper = static_cast<T>(std::nextafter(w->extent[2 * i + 1], HUGE_VAL));
            d.extent[2 * i] = std::nextafter(lower, upper);
            d.extent[2 * i + 1] = std::nextafter(upper, lower);
        }
    }
    d.material = static_cast<const uint8_t*>(w->material);
    d.density = static_cast<const double*>(w->density);
    d.measurement = static_cast<const uint8_t*>(w->measurement);
    d.voxels = w->voxels;
    d.palette = static_cast<const uint2*>(w->palette);
    d.codes = w->codes;
    d.bounds = static_cast<const dxmc_dev::DensityBound*>(w->bounds);
    d.codeBytes = w->codeBytes;
    d.index24 = hasIndex24(w);
    d.nxy = d.index24 ? d.nx * d.ny : 0;
    d.blocks = static_cast<const uint16_t*>(w->blocks);
    d.bnx = w->blockDims[0];
    d.bnxy = w->blockDims[0] * w->blockDims[1];
    d.blockShift = w->blockShift;
    d.codeMul = w->codeMul;
    d.voxelBytes = w->voxelBytes;
    if constexpr (std::is_same_v<T, float>)
        for (int i = 0; i < 3; ++i)
            d.facesRound |= dxmc_dev::coordinateReaches(d.extent[2 * i], d.extent[2 * i + 1], 1.0f / d.spacing[i], w->dims[i]) ? 1u : 0u;
    return d;
}

// block reduction of the step / event counters into the global counters
__device__ inline void accumulateCounters(dxmc_dev::Counters* ctr, uint32_t steps, uint32_t events)
{
    __shared__ unsigned long long s[2];
    if (threadIdx.x == 0) {
        s[0] = 0;
        s[1] = 0;
    }
    __syncthreads();
    if (steps)
        atomicAdd(&s[0], static_cast<unsigned long long>(steps));
    if (events)
        atomicAdd(&s[1], static_cast<unsigned long long>(events));
    __syncthreads();
    if (threadIdx.x == 0) {
        if (s[0])
            atomicAdd(&ctr->steps, s[0]);
        if (s[1])
            atomicAdd(&ctr->events, s[1]);
    }
}

bool validateTables(const dxmc_tables_desc& d, std::string& why);
int buildDeviceTables(dxmc_ctx* c, const dxmc_tables_desc& d, dxmc_tables& t);
int uploadExposures(dxmc_ctx* c, const dxmc_exposure* x, uint64_t nExp, int precision, RunBuffers& rb);
// argument checks shared by dxmc_hip_run and dxmc_hip_autotune (tally may be null)
int validateRun(dxmc_ctx* c, const dxmc_world* w, const dxmc_tables* t, const dxmc_exposure* x, uint64_t nExp, const dxmc_run_cfg* cfg,
    const dxmc_tally* tally);
inline std::tuple<const void*, const void*, int, int, bool> tuneKey(const dxmc_world* w, const dxmc_tables* t, const dxmc_run_cfg& cfg)
{
    return { w, t, cfg.precision, cfg.low_energy_correction, w->codeBytes != 0 };
}
// autotune.hip
int autotune(dxmc_ctx* c, const dxmc_world* w, const dxmc_tables* t, const dxmc_exposure* x, uint64_t nExp, const dxmc_run_cfg& base,
    uint64_t trialHistories, dxmc_run_cfg& best, dxmc_tune_report* report);
// codes of a palette world, once its runs and this one pay for them
// (world.hip). counts: the run takes place (else it is only being tuned for)
int preparePaletteCodes(dxmc_ctx* c, const dxmc_world* w, const dxmc_tables* t, const dxmc_exposure* x, uint64_t nExp, const dxmc_run_cfg& cfg, bool counts);
// whether a run on a world of such voxels with these tables uses 1-byte codes
bool usesCodesFp32(const dxmc_run_cfg& cfg, const dxmc_dev::Tables<float>& t, uint32_t voxelBytes, uint64_t voxels, bool pencil);
bool usesCodesFp64(const dxmc_run_cfg& cfg, const dxmc_dev::Tables<double>& t, uint32_t voxelBytes, uint64_t voxels, bool pencil);
int runTransport(dxmc_ctx* c, const dxmc_world* w, const dxmc_tables* t, const dxmc_exposure* x, uint64_t nExp, const dxmc_run_cfg& cfg,
    dxmc_tally* tally, const dxmc_run_monitor* monitor, dxmc_run_stats* stats);
// device inputs of a run's launches: exposure records of the run's precision
// (of both in the run without allocation),
// history prefix sums (device; host copy for progress, may be null), total
// histories, step/event counters (may be null) and the FP32 kernel's work
// counter
struct RunInputs {
    const dxmc_dev::Exposure<double>* exp64;
    const dxmc_dev::Exposure<float>* exp32;
    const uint64_t* startDev;
    const uint64_t* startHost;
    uint64_t total;
    dxmc_dev::Counters* ctr;
    unsigned long long* historyCounter;
    bool pencil; // every exposure is a pencil beam
};
// whether every exposure is a pencil beam (one direction)
inline bool pencilBeams(const dxmc_exposure* x, uint64_t nExp)
{
    for (uint64_t i = 0; i < nExp; ++i)
        if (x[i].collimation_angles[0] != x[i].collimation_angles[1] || x[i].collimation_angles[2] != x[i].collimation_angles[3])
            return false;
    return true;
}
// the launch loop of a run on prepared inputs (cancel, progress and preview
// through the monitor, which may be null)
int runLaunches(dxmc_ctx* c, const dxmc_world* w, const dxmc_tables* t, uint64_t nExp, const dxmc_run_cfg& cfg, dxmc_tally* tally,
    const RunInputs& in, const dxmc_run_monitor* monitor, double& kernelMs, uint64_t& launches);
// maximum intensity projection of the tally's dose along axis into a device
// image (launch only, on the context's stream); width and height returned
int launchTallyMip(dxmc_ctx* c, const dxmc_tally* tally, const dxmc_world* w, int axis, float* image, uint64_t& width, uint64_t& height);
// fills the tally's result arrays from its voxel scores: normalised for an
// output mode, the sums as they stand for mode -1
int launchNormalize(dxmc_ctx* c, const dxmc_tally* t, const dxmc_world* w, int mode, uint64_t nHist, double calibration);
// device address of the no-allocation run's scratch array on the current
// device (noalloc.hip), taken once per device
int noallocScratch(int device, void** out);
// FP32 transport launch (transport_fp32.hip)
void launchFp32(dxmc_ctx* c, const dxmc_run_cfg& cfg, const dxmc_dev::World<float>& w, const dxmc_dev::Tables<float>& t,
    const dxmc_dev::Exposure<float>* exps, const uint64_t* expStart, uint32_t nExp, uint64_t hb, uint64_t he, const dxmc_dev::Tally& tally,
    dxmc_dev::Counters* ctr, unsigned long long* historyCounter, bool pencilBeam);
// FP64 transport launch (transport_fp64.hip); t32: the FP32 copy of the tables,
// whose attenuation bounds and coefficients filter the FP64 decisions
void launchFp64(dxmc_ctx* c, const dxmc_run_cfg& cfg, const dxmc_dev::World<double>& w, const dxmc_dev::Tables<double>& t,
    const dxmc_dev::Tables<float>& t32, const dxmc_dev::Exposure<double>* exps, const uint64_t* expStart, uint32_t nExp, uint64_t hb, uint64_t he,
    const dxmc_dev::Tally& tally, dxmc_dev::Counters* ctr, unsigned long long* historyCounter, bool pencilBeam);
// Histories a wave of a persistent kernel claims per atomic on the launch's
// counter: 512, less in launches where that leaves waves without work while
// others run long (two claims a wave; at least a wave's 64 lanes, from 2^18
// histories on 128, with which a wave refills its lanes once). ms at 64, 128,
// 256, 512: FP32 DX 128x128x64, 2e4 histories 0.28 0.31 0.38 0.54, 1e6 0.66
// 0.58 0.59 0.70, 1e7 3.15 2.71 2.65 2.59; FP64 2e4 0.50 0.54 0.67 0.93, 1e6
// 1.16 1.12 1.10 1.17.
inline uint32_t historiesPerClaim(uint64_t histories, uint64_t waves)
{
    const uint64_t two = (histories / (2 * std::max<uint64_t>(waves, 1)) + 63) / 64 * 64;
    return static_cast<uint32_t>(std::clamp<uint64_t>(two, histories < (uint64_t(1) << 18) ? 64 : 128, 512));
}
}
