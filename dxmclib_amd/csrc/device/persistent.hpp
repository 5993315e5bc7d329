// Pieces shared by the two persistent transport kernels (transport_fp32.hip,
// transport_fp64.hip): world kinds, ranks among lanes, table access by 32-bit
// offsets, the copy of tables into LDS and the plan of a block's LDS, claims of
// histories, and the scores of a wave and of a pencil beam's block.
#pragma once
#include "physics.hpp"

namespace dxmc_dev {

// World kinds the persistent kernels are compiled for: the two common layouts
// get their code width, record width, 24-bit index and bounds table fixed at
// compile time, so a flight carries no branches on them
//   WORLD_CODES8    1-byte bounded-density codes (and their block codes
//                   when the run uses them), records of any width, the
//                   attenuation bounds table, 24-bit index
//   WORLD_PALETTE8  1-byte palette indices, no codes, no measurement flags,
//                   24-bit index
//   WORLD_PALETTE8_MEASURED  the same with measurement flags (forced events)
//   WORLD_ANY       every other world (branches at run time)
enum : uint32_t { WORLD_ANY = 0, WORLD_CODES8 = 1, WORLD_PALETTE8 = 2, WORLD_PALETTE8_MEASURED = 3 };
// kinds whose voxels may carry a measurement flag
__host__ __device__ constexpr bool kindForces(uint32_t kind) { return kind == WORLD_ANY || kind == WORLD_PALETTE8_MEASURED; }
__host__ __device__ constexpr bool kindPalette8(uint32_t kind) { return kind == WORLD_PALETTE8 || kind == WORLD_PALETTE8_MEASURED; }

__device__ inline uint32_t rankBelow(uint64_t mask)
{
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0u));
}

// inside the safe extent, without short-circuit branches
template <typename T>
__device__ inline bool insideFast(const World<T>& w, const T* pos)
{
    return (pos[0] > w.extent[0]) & (pos[0] < w.extent[1]) & (pos[1] > w.extent[2]) & (pos[1] < w.extent[3]) & (pos[2] > w.extent[4])
        & (pos[2] < w.extent[5]);
}

// linear voxel index; with 24-bit products where the grid allows (the
// compiler turns a 24-bit multiply-add into a 64-bit one, so the three terms
// are summed instead)
template <typename T>
__device__ inline uint64_t voxelIndexFast(const World<T>& w, uint3 v, bool index24)
{
    if (index24)
        return __umul24(v.z, w.nxy) + __umul24(v.y, w.nx) + v.x;
    return (static_cast<uint64_t>(v.z) * w.ny + v.y) * w.nx + v.x;
}

// element 'index' of a table addressed by a 32-bit byte offset from its
// base (tables below 4 GiB): the load takes the base from scalar registers
// and the offset from one vector register, with no 64-bit address
// arithmetic per lane
template <typename T>
__device__ inline T loadAt(const T* base, uint32_t index)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const unsigned char*>(base) + index * static_cast<uint32_t>(sizeof(T)));
}

// Whether q, a coordinate times the reciprocal spacing, is so near a whole
// number that the rounded quotient may truncate differently: the product is
// within 2^-51 q of it.
__host__ __device__ inline bool nearWhole(double q) { return fabs(q - rint(q)) <= fabs(q) * 0x1p-50; }

// block of a voxel (1-byte code worlds: 24-bit products hold)
template <typename T>
__device__ inline uint32_t blockIndexFast(const World<T>& w, uint3 v)
{
    return __umul24(v.z >> w.blockShift, w.bnxy) + __umul24(v.y >> w.blockShift, w.bnx) + (v.x >> w.blockShift);
}

// ------------------------------------------------------ LDS-staged tables
// The tables the samplers read with data-dependent indices (RITA, spline,
// shells, spectrum alias tables, heel and bowtie filters, the majorant and
// the segment bounds or nodes, optionally the attenuation coefficients) are copied
// into LDS at kernel start, one copy per block: their lookups then cost LDS
// latency instead of L2 latency, also while the world gathers keep evicting
// them from L1. Staging level: 1 none, 2 all but the attenuation
// coefficients, 3 all. Of the interaction tables only those of the run's
// low-energy model are staged (RITA for L >= 1, the scatter-function spline
// for L = 1, the shells for L = 2).
enum : uint32_t { STAGE_NONE = 1, STAGE_SMALL = 2, STAGE_ALL = 3 };

__host__ __device__ constexpr uint64_t ldsAlign(uint64_t bytes) { return (bytes + 15) & ~uint64_t(15); }

// bytes of LDS a staging level needs for low-energy model L (the same walk
// as stageTables)
template <typename T>
__host__ __device__ inline uint64_t ldsBytes(const Tables<T>& t, uint32_t level, int L)
{
    if (level <= STAGE_NONE)
        return 0;
    uint64_t b = 0;
    if (L >= 1)
        b += ldsAlign(uint64_t(t.nMaterials) * 4 * 56 * sizeof(T));
    if (L == 1)
        b += ldsAlign(uint64_t(t.nMaterials) * 63 * sizeof(T));
    if (L == 2)
        b += ldsAlign(uint64_t(t.nMaterials) * 12 * sizeof(Shell<T>));
    b += ldsAlign(uint64_t(t.lutNodes) * 2 * sizeof(T));
    b += sizeof(T) == 4 ? 2 * ldsAlign(uint64_t(t.lutNodes) * sizeof(float)) : ldsAlign(uint64_t(t.lutNodes) * sizeof(double));
    b += ldsAlign(uint64_t(t.nSpectra + 1) * sizeof(uint32_t));
    b += ldsAlign(uint64_t(t.nSpectra ? t.nSpectra : 1) * sizeof(uint32_t));
    b += 2 * ldsAlign(uint64_t(t.specTotal) * sizeof(T)) + ldsAlign(uint64_t(t.specTotal) * sizeof(uint32_t));
    b += ldsAlign(uint64_t(t.nHeel) * sizeof(Heel<T>)) + ldsAlign(uint64_t(t.heelWeightTotal) * sizeof(T));
    b += ldsAlign(uint64_t(t.nBowtie + 1) * sizeof(uint32_t)) + 2 * ldsAlign(uint64_t(t.bowtieTotal) * sizeof(T));
    if (level >= STAGE_ALL)
        b += ldsAlign(uint64_t(t.nMaterials) * t.lutNodes * 6 * sizeof(T));
    return b;
}

// LDS of the density intervals and attenuation bounds a staged code world
// adds: a flight reads them after the block code (and the voxel code); from
// LDS instead of L1 they took the CT spiral from 201 to 180 ms
template <typename T>
__host__ __device__ inline uint64_t boundsBytes(const Tables<T>& t)
{
    return ldsAlign(uint64_t(t.nMaterials) * t.lutNodes * sizeof(float2)) + 256 * sizeof(float2);
}

// a table's copy in LDS at the cursor, made by all threads of the block
template <typename T>
__device__ inline const T* stageArray(const T* src, uint64_t count, unsigned char*& cursor)
{
    static_assert(sizeof(T) % 4 == 0);
    T* dst = reinterpret_cast<T*>(cursor);
    const uint64_t words = count * sizeof(T) / 4;
    const uint32_t* s = reinterpret_cast<const uint32_t*>(src);
    uint32_t* d = reinterpret_cast<uint32_t*>(dst);
    for (uint64_t i = threadIdx.x; i < words; i += blockDim.x)
        d[i] = s[i];
    cursor += ldsAlign(count * sizeof(T));
    return dst;
}

// copies the tables into LDS and points t at the copies (all threads of the
// block call it; ends with a barrier). The level is a template parameter so
// that the compiler sees which pointers address LDS.
template <typename T, uint32_t level, int L>
__device__ inline void stageTables(Tables<T>& t, unsigned char* lds)
{
    if constexpr (level <= STAGE_NONE)
        return;
    unsigned char* c = lds;
    if constexpr (L >= 1)
        t.rita = stageArray(t.rita, uint64_t(t.nMaterials) * 4 * 56, c);
    if constexpr (L == 1)
        t.spline = stageArray(t.spline, uint64_t(t.nMaterials) * 63, c);
    if constexpr (L == 2)
        t.shells = stageArray(t.shells, uint64_t(t.nMaterials) * 12, c);
    t.lutMajorant = stageArray(t.lutMajorant, uint64_t(t.lutNodes) * 2, c);
    if constexpr (sizeof(T) == 4) {
        t.lutBoundUp = stageArray(t.lutBoundUp, t.lutNodes, c);
        t.lutAnchor = stageArray(t.lutAnchor, t.lutNodes, c);
    } else {
        t.lutGrid = stageArray(t.lutGrid, t.lutNodes, c);
    }
    t.specOffset = stageArray(t.specOffset, t.nSpectra + 1, c);
    t.specThreshold = stageArray(t.specThreshold, t.nSpectra ? t.nSpectra : 1, c);
    t.specProb = stageArray(t.specProb, t.specTotal, c);
    t.specEnergy = stageArray(t.specEnergy, t.specTotal, c);
    t.specAlias = stageArray(t.specAlias, t.specTotal, c);
    t.heel = stageArray(t.heel, t.nHeel, c);
    t.heelWeight = stageArray(t.heelWeight, t.heelWeightTotal, c);
    t.bowtieOffset = stageArray(t.bowtieOffset, t.nBowtie + 1, c);
    t.bowtieAngle = stageArray(t.bowtieAngle, t.bowtieTotal, c);
    t.bowtieWeight = stageArray(t.bowtieWeight, t.bowtieTotal, c);
    if constexpr (level >= STAGE_ALL)
        t.lutCoef = stageArray(t.lutCoef, uint64_t(t.nMaterials) * t.lutNodes * 6, c);
    __syncthreads();
}

// The wave's next histories from the launch's global counter: 'pool' at a
// time, one atomic by lane 0. False when the launch has none left. The
// bounds are wave-uniform and live in scalar registers.
__device__ inline bool claimHistories(unsigned long long* next, uint32_t pool, uint64_t span, uint64_t hBegin, uint32_t lane, uint64_t& poolNext,
    uint64_t& poolEnd)
{
    unsigned long long base = 0;
    if (lane == 0)
        base = atomicAdd(next, static_cast<unsigned long long>(pool));
    base = __shfl(base, 0);
    base = (static_cast<unsigned long long>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(base >> 32))) << 32)
        | __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(base));
    if (base >= span)
        return false;
    poolNext = hBegin + base;
    poolEnd = hBegin + (base + pool < span ? base + pool : span);
    return true;
}

// Adds one score per lane that has one to the tally; the whole wave calls it.
// Atomics cost a request per cache line, so the scores are packed into the
// wave's first lanes (one permutation) and added 16 at a time, the four lanes
// of a group to the dose, the variance and the event count of one voxel.
// wide: voxel indices may exceed 32 bits.
template <typename T>
__device__ inline void scoreWave(const Tally& tally, bool has, uint64_t idx, T e, bool wide)
{
    const uint64_t mask = __ballot(has);
    const uint32_t n = __popcll(mask);
    if (n == 0)
        return;
    const uint32_t lane = __lane_id();
    const int to = static_cast<int>(4 * (has ? rankBelow(mask) : n + rankBelow(~mask)));
    auto move = [&](uint32_t v) { return __builtin_amdgcn_ds_permute(to, static_cast<int>(v)); };
    const int lo = move(static_cast<uint32_t>(idx));
    const int hi = wide ? move(static_cast<uint32_t>(idx >> 32)) : 0;
    int e0, e1 = 0;
    if constexpr (sizeof(T) == 4) {
        e0 = move(__float_as_uint(e));
    } else {
        e0 = move(static_cast<uint32_t>(__double2loint(e)));
        e1 = move(static_cast<uint32_t>(__double2hiint(e)));
    }
    const uint32_t field = lane & 3u;
    for (uint32_t base = 0; base < n; base += 16) {
        const uint32_t slot = base + lane / 4;
        const int from = static_cast<int>(4 * slot);
        const uint32_t vLo = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(from, lo));
        const uint32_t vHi = wide ? static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(from, hi)) : 0u;
        double v;
        if constexpr (sizeof(T) == 4)
            v = static_cast<double>(__uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(from, e0))));
        else
            v = __hiloint2double(__builtin_amdgcn_ds_bpermute(from, e1), __builtin_amdgcn_ds_bpermute(from, e0));
        const double add = field == 0 ? v : field == 1 ? v * v : 1.0;
        if (slot < n && field < 3)
            unsafeAtomicAdd(reinterpret_cast<double*>(tally.voxels + (static_cast<uint64_t>(vHi) << 32 | vLo)) + field, add);
    }
}

// Scores of pencil beams. Their photons interact on one line of voxels, whose
// cache lines all XCDs then change in turn (a line's score of three atomics
// takes 95 ns when all XCDs add to it, 12 ns when one does), so a block keeps the sums of up to 256 voxels in LDS,
// first come, first served, and adds them to the tally once, at its end. Runs
// of other beams score all over the world and would only fill it.
constexpr uint32_t SCORE_CACHE_ENTRIES = 256;
constexpr uint32_t SCORE_CACHE_BYTES = SCORE_CACHE_ENTRIES * (3 * sizeof(double) + sizeof(uint32_t));

// Slots of a wave's photon pool: sampling leaves POOL_RESERVE for photons that
// become pending, and a wave uses at most POOL_MAX.
constexpr uint32_t POOL_RESERVE = 16;
constexpr uint32_t POOL_MAX = 128;

// Orders a wave's accesses to its pool: a slot that one lane writes is read by
// another. The LDS unit keeps a wave's order, so this costs no instruction; it
// keeps the compiler from moving one lane's accesses across another's.
__device__ inline void poolFence()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

// What a block holds in LDS ahead of its waves' pools: tables of a staging
// level, on worlds of 1-byte codes also the density and attenuation bounds, in
// a run of pencil beams the score cache.
struct LdsPlan {
    uint32_t stage;
    bool bounds;
    uint32_t bytes;
    uint32_t block, slotBytes;
    // slots of each wave's pool in a block of so many waves
    uint32_t slots(uint32_t waves) const { return block <= bytes ? 0u : least(POOL_MAX, (block - bytes) / waves / slotBytes); }
    static constexpr uint32_t least(uint32_t a, uint32_t b) { return b < a ? b : a; }
};

// The plan of a launch whose blocks have 'block' bytes of LDS and 'waves'
// waves: of the requested level, or what of it leaves each pool 'poolMin' slots
// (set where a fuller pool is worth more than the tables, measured in each
// kernel's file). The bounds go first: they and the sampling tables take 1.1 KB
// a material each (FP32; FP64 2.2 KB of tables), so the tables alone fit with
// about twice the materials. Dropped together, code worlds of 20 and more
// materials read everything from global memory (20 materials, 192x160x120, 2e7
// histories FP32, L = 1: 3.85 ms; with the tables 3.35; L = 2, 24 materials
// 7.45 and 6.35).
template <typename T>
inline LdsPlan planLds(const Tables<T>& t, uint32_t level, int L, bool codes8, bool pencil, uint32_t block, uint32_t waves, uint32_t slotBytes,
    uint32_t poolMin)
{
    const uint64_t pools = uint64_t(waves) * poolMin * slotBytes;
    for (;; --level) {
        const uint64_t tables = ldsBytes(t, level, L) + (pencil ? SCORE_CACHE_BYTES : 0u);
        if (level <= STAGE_NONE)
            return { STAGE_NONE, false, static_cast<uint32_t>(tables), block, slotBytes };
        if (codes8 && tables + boundsBytes(t) + pools <= block)
            return { level, true, static_cast<uint32_t>(tables + boundsBytes(t)), block, slotBytes };
        // (without the bounds, code worlds have a kernel at level 2 only)
        if (!(codes8 && level >= STAGE_ALL) && tables + pools <= block)
            return { level, false, static_cast<uint32_t>(tables), block, slotBytes };
    }
}

// Whether a run with this plan uses a world's codes (one that sets block_bounds
// does in any case). Worlds of 8-byte records always do. A palette's records can be as fast where the bounds are not in
// LDS (18 and more materials): FP64 drew or lost up to 7 % with codes (30
// materials, 1e6 to 6.7e7 voxels, 5e6 histories: 3.45 ms with records, 3.57
// with codes). FP32 gains 5 to 59 % on palettes of more than 256 records
// (CT numbers); on smaller ones it loses 2 to 7 % (30 materials, 3.7e6 voxels,
// 2e7 histories: 3.44 ms with records, 3.63 with codes) up to 2e7 voxels, at
// L = 0 below 3.7e6, and gains 3 to 14 % beyond.
template <typename T>
inline bool codesPay(const LdsPlan& plan, uint32_t voxelBytes, uint64_t voxels, int L)
{
    if (voxelBytes == 8 || plan.bounds)
        return true;
    if (sizeof(T) == 8)
        return false;
    return voxelBytes == 2 || voxels >= (uint64_t(1) << (L == 0 ? 22 : 25));
}

struct ScoreCache {
    static constexpr uint32_t FREE = 0xffffffffu; // no voxel index where indices fit 24-bit products
    double* sums; // dose, variance, events of each entry
    uint32_t* voxel;

    // the cache in LDS, empty (all threads of the block call it)
    __device__ explicit ScoreCache(unsigned char* lds)
        : sums(reinterpret_cast<double*>(lds))
        , voxel(reinterpret_cast<uint32_t*>(lds + SCORE_CACHE_ENTRIES * 3 * sizeof(double)))
    {
    }
    __device__ inline void clear() const
    {
        for (uint32_t i = threadIdx.x; i < SCORE_CACHE_ENTRIES; i += blockDim.x)
            voxel[i] = FREE;
        for (uint32_t i = threadIdx.x; i < 3 * SCORE_CACHE_ENTRIES; i += blockDim.x)
            sums[i] = 0.0;
        __syncthreads();
    }
    // takes the score of a lane that has one; false when its entry is another voxel's
    __device__ inline bool add(uint32_t idx, double e) const
    {
        const uint32_t k = (idx * 2654435761u) >> 24;
        const uint32_t was = atomicCAS(&voxel[k], FREE, idx);
        if (was != FREE && was != idx)
            return false;
        const double v[3] = { e, e * e, 1.0 };
        for (int f = 0; f < 3; ++f)
            __hip_atomic_fetch_add(&sums[3 * k + f], v[f], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return true;
    }
    // adds the sums to the tally (all threads of the block call it)
    __device__ inline void flush(const Tally& tally) const
    {
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < 4 * SCORE_CACHE_ENTRIES; i += blockDim.x)
            if ((i & 3u) < 3 && voxel[i / 4] != FREE)
                unsafeAtomicAdd(reinterpret_cast<double*>(tally.voxels + voxel[i / 4]) + (i & 3u), sums[3 * (i / 4) + (i & 3u)]);
    }
};
}
