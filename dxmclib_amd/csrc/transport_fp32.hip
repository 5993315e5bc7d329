// FP32 photon transport: persistent kernel with per-wave photon pools.
//
// Each lane flies one photon (position, direction, energy, weight, majorant,
// PCG state) in registers; a wave keeps further photons in a pool in LDS,
// some ready to fly, others with an interaction due. The wave runs three
// kinds of work, each with many lanes:
//   flights       Woodcock flights of the lanes (distance under the majorant,
//                 real-or-virtual decision from density and attenuation
//                 bounds, roulette), until 'regeneration_threshold' lanes
//                 have lost their photon or are due to interact; due photons
//                 then go to the pool and ready ones take their lanes
//   interactions  once 'interaction_threshold' photons are due, they come to
//                 the lanes, in exchange for the photons flying there, and
//                 run the samplers (Compton/Rayleigh rejection loops,
//                 fluorescence) together; the survivors fly on
//   sampling      when too few photons are ready, the whole wave samples new
//                 histories into the pool (from a wave-private range of
//                 history indices, which one lane refills with an atomic on
//                 the launch's counter)
// Without the pool, due photons waited on their lanes: 51 of 64 lanes flew
// and 21 interacted (126 vector instructions a history on the CT spiral
// workload, 91 with it).
//
// What bounds it: vector issue (CT spiral: busy 94 % of the cycles, with 58 %
// of the lanes at work; 75 % before the bounds moved to LDS, when flights
// waited on them). CT spiral 512x512x300, 1e9 histories: 228 ms
// with due photons on their lanes and 7 waves a SIMD, 197 with pools and 6
// waves, 180 with density intervals and attenuation bounds in LDS; axial
// 1024x1024x128, 4e8: 77, 69, 60 ms; impulse approximation, 401x333x151,
// 1.5e8: 48.4, 42.7, 38.9 ms (4 waves).
//
// Each history keeps its own PCG stream and consumes it in the reference's
// order (flight, decision, interaction, roulette), so delaying an interaction
// changes nothing but timing: results depend neither on the lane or wave that
// ran a history nor on the grid size or thresholds.
//
// Arithmetic is FP32 (base-2 anchored LUT, FP32 transcendentals, voxel index
// by multiplication with the reciprocal spacing, FP32 denormals flushed);
// each scoring event is added to the FP64 tallies with hardware FP64
// atomics. The kernel is compiled per low-energy model, register budget
// (4 or 6 waves per SIMD), LDS staging and world kind.
#include "device/persistent.hpp"
#include "internal.hpp"

using namespace dxmc_dev;

namespace {

// voxel coordinates, with the reciprocal spacing, of a position inside the
// extent. Kept inside the grid where rounding can reach its far end
// (facesRound, known per world).
__device__ inline uint3 voxelCoordsFast(const World<float>& w, const float* pos, const float* inv)
{
    uint3 v = make_uint3(static_cast<uint32_t>((pos[0] - w.extent[0]) * inv[0]), static_cast<uint32_t>((pos[1] - w.extent[2]) * inv[1]),
        static_cast<uint32_t>((pos[2] - w.extent[4]) * inv[2]));
    if (w.facesRound) {
        v.x = min(v.x, w.nx - 1);
        v.y = min(v.y, w.ny - 1);
        v.z = min(v.z, w.nz - 1);
    }
    return v;
}

constexpr float LN2F = 0.693147180559945309f;

// A wave's pool of photons in LDS: a ring of slots whose first 'ready' ones
// hold photons to fly and the next 'pending' ones photons with an interaction
// due. One record of 13 words a photon (an odd stride: lanes reading the same
// word of consecutive slots hit different banks): position, direction,
// energy, weight, PCG state, the history's offset in the launch (its PCG
// increment is 2 (first history + launch begin + offset) + 1), LUT segment |
// material << 20 | measurement flag << 28, and the history's steps so far.
// What follows from these (the LUT offset, the majorant, the voxel) is
// computed again when a lane takes the photon.
constexpr uint32_t SLOT_WORDS = 13;
constexpr uint32_t SLOT_BYTES = SLOT_WORDS * 4;
constexpr uint32_t FLIGHTS_PER_LOOP = 64; // most flights before the outer loop runs

// Waves of a block: two blocks fill a CU's 4 W waves, so the staged tables
// are held twice a CU and the LDS left is the waves' pools.
__host__ __device__ constexpr uint32_t blockWaves(uint32_t W) { return 2 * W; }

// Russian roulette after a step that left the photon alive (transport.hpp:684-694)
__device__ inline bool roulette(Particle<float>& p, Rng& rng)
{
    if (p.energy * p.weight < 5.0f) {
        if (rng.uniform<float>() < 0.8f)
            return false;
        p.weight *= 1.0f / (1.0f - 0.8f);
    }
    return true;
}

// W: resident waves per SIMD the register allocation must allow, 6 (at most 80
// VGPRs, spill-free at L = 0, 1 but for few lanes' values of kind any) or 4
// (128 VGPRs; CT spiral 206 ms, 6: 180). Blocks of 10 or 14 waves load the
// SIMDs unevenly, so that a CU holds one instead of two (340 ms); 16 waves
// with 64 VGPRs spill (282 ms).
// S: LDS staging level. K: world kind. BOUNDS_LDS: density intervals and
// attenuation bounds of a code world in LDS too. The autotuner picks among the
// register budgets and staging levels.
template <int L, int W, uint32_t S, uint32_t K, bool BOUNDS_LDS>
__global__ __launch_bounds__(64 * blockWaves(W)) __attribute__((amdgpu_waves_per_eu(W, 8))) void transportPersistent(World<float> w, Tables<float> tg, const Exposure<float>* exps, const uint64_t* expStart,
    uint32_t nExp, uint64_t hBegin, uint64_t hEnd, uint64_t seed, uint64_t firstHistory, Tally tally, Counters* ctr, unsigned long long* next,
    uint32_t refillThreshold, uint32_t interactThreshold, uint32_t poolSize, uint32_t slots, bool pencil)
{
    extern __shared__ __align__(16) unsigned char lds[];
    Tables<float> t = tg;
    stageTables<float, S, L>(t, lds);
    const float2* bounds = nullptr; // staged: density interval of each code
    if constexpr (BOUNDS_LDS) {
        unsigned char* c = lds + ldsBytes(tg, S, L);
        t.lutSumBound = stageArray(t.lutSumBound, uint64_t(t.nMaterials) * t.lutNodes, c);
        float2* d = reinterpret_cast<float2*>(c);
        for (uint32_t i = threadIdx.x; i < 256; i += blockDim.x)
            d[i] = make_float2(w.bounds[i].lo, w.bounds[i].hi);
        bounds = d;
        __syncthreads();
    }
    Particle<float> p;
    Rng rng { 0, 1 };
    float majInv = 0;
    bool flying = false, due = false; // neither: the lane holds no photon
    // the wave's claimed, not yet started histories [poolNext, poolEnd)
    const uint64_t span = hEnd - hBegin;
    uint64_t poolNext = 0, poolEnd = 0;
    uint32_t poolExp = 0;
    bool claimedAll = span == 0;
    uint32_t events = 0; // scoring events of the lane's interactions
    uint32_t steps = 0; // in-world steps of the histories that ended on this lane
    uint32_t historySteps = 0; // of its current one
    // material | measurement flag << 24 of the voxel reached (one register;
    // the LUT row products are 24-bit and ignore the flag)
    uint32_t matMeas = 0;
    // the photon's place in the LUT; changes only with its energy
    LutPoint<float> lp { 0, 0.0f };
    const float inv[3] = { 1.0f / w.spacing[0], 1.0f / w.spacing[1], 1.0f / w.spacing[2] };
    // the world's layout, fixed by K where it can be
    const uint32_t codeBytes = K == WORLD_CODES8 ? 1u : kindPalette8(K) ? 0u : w.codeBytes;
    const uint32_t voxelBytes = kindPalette8(K) ? 1u : w.voxelBytes; // (kinds without codes)
    const bool index24 = K != WORLD_ANY || w.index24 != 0;
    const bool sumBounds = K == WORLD_CODES8 || (K == WORLD_ANY && t.lutSumBound != nullptr);
    // global index of the launch's first history (PCG increments of pooled photons)
    const uint64_t launchFirst = firstHistory + hBegin;
    const uint32_t lane = __lane_id();

    uint32_t poolAt = static_cast<uint32_t>(ldsBytes(tg, S, L) + (BOUNDS_LDS ? boundsBytes(tg) : 0u));
    const ScoreCache cache(lds + poolAt);
    if (pencil) {
        poolAt += SCORE_CACHE_BYTES;
        cache.clear();
    }
    uint32_t* pool = reinterpret_cast<uint32_t*>(lds + poolAt + (threadIdx.x / 64) * (slots * SLOT_BYTES));
    uint32_t first = 0, ready = 0, pending = 0; // the ring's window (wave-uniform)
    // slot 'offset' from the start of the window
    auto slotAt = [&](uint32_t offset) {
        const uint32_t k = first + offset;
        return pool + (k >= slots ? k - slots : k) * SLOT_WORDS;
    };
    auto packSegment = [&]() { return lp.k | (matMeas & 0xffu) << 20 | (kindForces(K) ? (matMeas >> 24 != 0 ? 1u << 28 : 0u) : 0u); };
    auto store = [&](uint32_t* q) {
        for (int i = 0; i < 3; ++i) {
            q[i] = __float_as_uint(p.pos[i]);
            q[3 + i] = __float_as_uint(p.dir[i]);
        }
        q[6] = __float_as_uint(p.energy);
        q[7] = __float_as_uint(p.weight);
        q[8] = static_cast<uint32_t>(rng.s);
        q[9] = static_cast<uint32_t>(rng.s >> 32);
        q[10] = static_cast<uint32_t>(rng.inc >> 1) - static_cast<uint32_t>(launchFirst);
        q[11] = packSegment();
        q[12] = historySteps;
    };
    // takes the photon out of a slot; what it leaves out is set by derive()
    auto load = [&](const uint32_t* q) {
        for (int i = 0; i < 3; ++i) {
            p.pos[i] = __uint_as_float(q[i]);
            p.dir[i] = __uint_as_float(q[3 + i]);
        }
        p.energy = __uint_as_float(q[6]);
        p.weight = __uint_as_float(q[7]);
        rng.s = static_cast<uint64_t>(q[9]) << 32 | q[8];
        rng.inc = 2 * (launchFirst + q[10]) + 1;
        const uint32_t segment = q[11];
        lp.k = segment & 0xfffffu;
        matMeas = (segment >> 20 & 0xffu) | (kindForces(K) ? segment >> 28 << 24 : 0u);
        historySteps = q[12];
    };
    // the LUT point lutPoint() gives, from the known segment, and the majorant
    auto derive = [&]() {
        lp.x = __builtin_amdgcn_logf(p.energy) - t.lutAnchor[lp.k];
        majInv = majorantInverseAt(t, lp);
    };

    for (;;) {
        const uint64_t dueMask = __ballot(due);
        uint64_t flyMask = __ballot(flying);
        const uint32_t nDue = __popcll(dueMask);
        const uint32_t nFly = __popcll(flyMask);
        const uint32_t room = slots - ready - pending;
        const bool work = poolNext < poolEnd || !claimedAll;
        const bool canSample = work && room > POOL_RESERVE;
        // Interactions run once enough photons wait for one (on lanes and in
        // the pool), when the pool cannot take the lanes' due photons, or when
        // there is little else left to do.
        const uint32_t waiting = nDue + pending;
        if (waiting != 0
            && (waiting >= interactThreshold || nDue > room || (!work && ready == 0 && waiting >= nFly) || (nFly == 0 && ready == 0 && !canSample))) {
            // The pool's pending photons come to the lanes: to lanes without
            // a photon from the end of the window, and to flying lanes from
            // its front in exchange for their photon, whose slot then joins
            // the ready ones.
            const uint64_t emptyMask = ~(dueMask | flyMask);
            const uint32_t back = min(64u - nDue - nFly, pending);
            const uint32_t front = min(nFly, pending - back);
            const bool taken = !due && !flying && rankBelow(emptyMask) < back;
            const bool exchanged = flying && rankBelow(flyMask) < front;
            if (taken || exchanged) {
                uint32_t* q = slotAt(taken ? ready + pending - 1 - rankBelow(emptyMask) : ready + rankBelow(flyMask));
                if (exchanged) {
                    uint32_t v[SLOT_WORDS];
                    for (uint32_t f = 0; f < SLOT_WORDS; ++f)
                        v[f] = q[f];
                    store(q);
                    load(v);
                } else {
                    steps += historySteps;
                    load(q);
                }
                derive();
                due = true;
                flying = false;
            }
            pending -= back + front;
            ready += front;
            Deposits<float> deposits;
            uint64_t idx = 0;
            if (due) {
                const uint32_t mat = matMeas & 0xffu;
                idx = voxelIndexFast(w, voxelCoordsFast(w, p.pos, inv), index24); // the voxel the flight ended in
                bool update = false;
                float att[3];
                attenuationAt(t, mat, lp, att);
                bool alive;
                if (kindForces(K) && matMeas > 0xffffffu) { // forced event (measurement voxel)
                    float density;
                    uint32_t tag;
                    readVoxelPacked(w, voxelBytes, idx, tag, density);
                    const float prob = ((att[0] + att[1]) + att[2]) * density * majInv;
                    alive = computeInteractionsForced<float, L>(t, prob, att, p, mat, deposits, rng, update);
                } else {
                    alive = computeInteractions<float, L>(t, att, p, mat, deposits, rng, update);
                }
                if (alive)
                    alive = roulette(p, rng);
                if (alive && update) { // new energy: its LUT segment and majorant
                    lp = lutPoint(t, p.energy);
                    majInv = majorantInverseAt(t, lp);
                }
                flying = alive;
                due = false;
            }
            events += deposits.n;
            bool scores = deposits.n > 0;
            if (pencil && scores)
                scores = !cache.add(static_cast<uint32_t>(idx), static_cast<double>(deposits.first));
            scoreWave(tally, scores, idx, deposits.first, !index24);
            if (kindForces(K) && __ballot(deposits.n > 1) != 0) // forced events with a Compton event
                scoreWave(tally, deposits.n > 1, idx, deposits.second, !index24);
        } else if (nDue != 0) {
            // photons with an interaction due wait in the pool
            if (due) {
                store(slotAt(ready + pending + rankBelow(dueMask)));
                historySteps = 0;
                due = false;
            }
            pending += nDue;
        }
        flyMask = __ballot(flying);
        const uint32_t nEmpty = 64u - __popcll(flyMask);
        if (work && ready < nEmpty && slots - ready - pending > POOL_RESERVE) {
            // sample new histories with the whole wave: lanes 0 .. want-1
            // take the next histories of the wave's pool (refilled from the
            // global counter as needed), photons that enter the world join
            // the ready ones
            const uint32_t want = min(64u, slots - ready - pending - POOL_RESERVE);
            uint32_t assigned = 0;
            bool sampled = false;
            Particle<float> np;
            Rng nr { 0, 1 };
            uint32_t nOffset = 0;
            while (assigned < want) {
                if (poolNext >= poolEnd) {
                    if (claimedAll)
                        break;
                    if (!claimHistories(next, poolSize, span, hBegin, lane, poolNext, poolEnd)) {
                        claimedAll = true;
                        break;
                    }
                    if (poolEnd == hEnd)
                        claimedAll = true;
                    poolExp = upperBound(expStart, nExp + 1, poolNext) - 1;
                }
                const uint64_t avail = poolEnd - poolNext;
                const uint32_t take = avail < want - assigned ? static_cast<uint32_t>(avail) : want - assigned;
                if (lane >= assigned && lane < assigned + take) {
                    const uint64_t h = poolNext + (lane - assigned);
                    uint32_t e = poolExp;
                    while (h >= expStart[e + 1])
                        ++e;
                    nr = Rng::forHistory(seed, firstHistory + h);
                    nOffset = static_cast<uint32_t>(h - hBegin);
                    sampleParticle(exps[e], t, nr, np);
                    sampled = transportToWorld(w, np);
                }
                poolNext += take;
                assigned += take;
            }
            const uint64_t entered = __ballot(sampled);
            const uint32_t n = __popcll(entered);
            first = first >= n ? first - n : first + slots - n; // ahead of the ready ones
            ready += n;
            if (sampled) {
                uint32_t* q = slotAt(rankBelow(entered));
                for (int i = 0; i < 3; ++i) {
                    q[i] = __float_as_uint(np.pos[i]);
                    q[3 + i] = __float_as_uint(np.dir[i]);
                }
                q[6] = __float_as_uint(np.energy);
                q[7] = __float_as_uint(np.weight);
                q[8] = static_cast<uint32_t>(nr.s);
                q[9] = static_cast<uint32_t>(nr.s >> 32);
                q[10] = nOffset;
                q[11] = lutPoint(t, np.energy).k;
                q[12] = 0;
            }
        }
        poolFence(); // slots written above, read below by other lanes
        // lanes without a photon take ready ones from the front of the window
        const uint32_t take = min(nEmpty, ready);
        if (take != 0) {
            const uint32_t r = rankBelow(~flyMask);
            if (!flying && r < take) {
                steps += historySteps;
                load(slotAt(r));
                derive();
                flying = true;
            }
            first += take;
            first = first >= slots ? first - slots : first;
            ready -= take;
        }
        poolFence(); // slots read above, written next by other lanes
        const bool more = poolNext < poolEnd || !claimedAll || ready != 0;
        if (__ballot(flying) == 0) {
            if (!more && pending == 0)
                break;
            continue;
        }
        // Woodcock flights of the flying lanes until enough lanes wait for
        // another photon (or, near the end, for interactions). Only the
        // flight's own values are live in this loop. Lanes whose photon may be
        // below the roulette limit (a flight only raises a weight) or within
        // the loop's flights of the step cap are known as wave masks, so that
        // the other flights test neither.
        const uint32_t limit = more ? refillThreshold : 64u;
        const uint64_t faintMask = __ballot(p.energy * p.weight < 5.0f);
        const bool nearCap = __ballot(flying && historySteps >= MAX_STEPS - FLIGHTS_PER_LOOP) != 0;
        for (uint32_t n = 0; n < FLIGHTS_PER_LOOP; ++n) {
            if (flying) {
                // one Woodcock flight (woodcockParticleTracking, transport.hpp:
                // 650-699)
                const float u1 = rng.uniform<float>();
                const float step = -__builtin_amdgcn_logf(u1) * (LN2F * 10.0f) * majInv; // cm -> mm
                for (int i = 0; i < 3; ++i)
                    p.pos[i] += p.dir[i] * step;
                flying = insideFast(w, p.pos);
                if (flying) {
                    const uint3 vc = voxelCoordsFast(w, p.pos, inv);
                    Rng r2 = rng;
                    const float u2 = r2.uniform<float>();
                    // The acceptance probability (Σμ·ρ)·(1/μ̂) is monotone in Σμ and
                    // in ρ. Bounds of both settle most draws exactly as the values
                    // would: u2 < p(lower bounds) accepts, u2 >= p(upper bounds)
                    // rejects. Σμ is bounded over the photon's LUT segment; ρ by the
                    // voxel's block when the block holds one material, else by the
                    // voxel's code when the world has codes, else read exactly. Only
                    // a draw between the bounds evaluates the attenuation (and reads
                    // the record).
                    float prob = 0.0f;
                    bool settled = false;
                    // (the L = 2 kernel also runs without block codes: a run
                    // switch there costs no occupancy; at L = 0, 1 a world
                    // without them runs the K = any kernel)
                    if (K == WORLD_CODES8 && (L < 2 || w.blocks != nullptr)) {
                        const uint32_t bc = loadAt(w.blocks, blockIndexFast(w, vc));
                        // the material from the largest code by arithmetic, so
                        // the intervals and the segment bounds load together
                        const uint32_t bm = __umul24(bc >> 8, w.codeMul) >> CODE_MUL_SHIFT;
                        const float bLo = BOUNDS_LDS ? bounds[bc & 0xffu].x : w.bounds[bc & 0xffu].lo;
                        const float bHi = BOUNDS_LDS ? bounds[bc >> 8].y : w.bounds[bc >> 8].hi;
                        const float2 sb = BOUNDS_LDS ? t.lutSumBound[__umul24(bm, t.lutNodes) + lp.k] : loadAt(t.lutSumBound, __umul24(bm, t.lutNodes) + lp.k);
                        const float lo = sb.x * bLo * majInv;
                        const float hi = sb.y * bHi * majInv;
                        settled = (bc != BLOCK_MIXED) & ((u2 < lo) | (u2 >= hi));
                        matMeas = bm;
                        prob = lo;
                    }
                    if (!settled) {
                        const uint64_t idx = voxelIndexFast(w, vc, index24);
                        float density, dLo, dHi;
                        if (K == WORLD_CODES8) {
                            // material by arithmetic, interval and segment bounds
                            // loaded together (code worlds carry no measurement flags)
                            // (1-byte codes: below 2^32 voxels, a 32-bit offset)
                            const uint32_t code = loadAt(static_cast<const uint8_t*>(w.codes), static_cast<uint32_t>(idx));
                            matMeas = __umul24(code, w.codeMul) >> CODE_MUL_SHIFT;
                            if constexpr (BOUNDS_LDS) {
                                const float2 b = bounds[code];
                                dLo = b.x;
                                dHi = b.y;
                            } else {
                                const uint2 b = *reinterpret_cast<const uint2*>(w.bounds + code);
                                dLo = __uint_as_float(b.x);
                                dHi = __uint_as_float(b.y);
                            }
                            density = dLo;
                        } else if (codeBytes != 0) {
                            const uint32_t code = codeBytes == 1 ? static_cast<const uint8_t*>(w.codes)[idx] : static_cast<const uint16_t*>(w.codes)[idx];
                            // the interval as one 16-byte load (read field by field,
                            // the compiler splits it into two loads on the chain)
                            const uint4 b = *reinterpret_cast<const uint4*>(w.bounds + code);
                            matMeas = b.z; // material; code worlds carry no measurement flags
                            dLo = __uint_as_float(b.x);
                            dHi = __uint_as_float(b.y);
                            density = dLo;
                        } else {
                            readVoxelPacked(w, voxelBytes, idx, matMeas, density);
                            dLo = density;
                            dHi = density;
                        }
                        if (sumBounds) {
                            const float2 sb = BOUNDS_LDS ? t.lutSumBound[__umul24(matMeas, t.lutNodes) + lp.k] : loadAt(t.lutSumBound, __umul24(matMeas, t.lutNodes) + lp.k);
                            const float lo = sb.x * dLo * majInv;
                            const float hi = sb.y * dHi * majInv;
                            settled = (u2 < lo) | (u2 >= hi);
                            prob = lo;
                        }
                        if (!settled) {
                            // the record's density, from the FP64 array it was
                            // rounded from (one layout for all code worlds); a
                            // code of one density names it
                            if (codeBytes != 0 && dLo != dHi)
                                density = static_cast<float>(w.density[idx]);
                            float att[3];
                            attenuationAt(t, matMeas, lp, att); // 24-bit row product: flag ignored
                            prob = ((att[0] + att[1]) + att[2]) * density * majInv;
                        }
                    }
                    // a forced event draws no decision
                    const bool measured = kindForces(K) && matMeas > 0xffffffu;
                    rng.s = measured ? rng.s : r2.s;
                    due = measured | (u2 < prob);
                    flying = !due;
                    if (flying & __builtin_amdgcn_inverse_ballot_w64(faintMask))
                        flying = roulette(p, rng);
                    ++historySteps;
                    if (nearCap && historySteps >= MAX_STEPS) {
                        flying = false;
                        due = false;
                    }
                }
            }
            const uint32_t flyNow = __popcll(__ballot(flying));
            if (flyNow == 0 || 64u - flyNow >= limit || (!more && __popcll(__ballot(due)) + pending >= flyNow))
                break;
        }
    }
    if (pencil)
        cache.flush(tally);
    if (ctr)
        dxmc_backend::accumulateCounters(ctr, steps + historySteps, events);
}

}

namespace dxmc_backend {

namespace {

__global__ void clearCounter(unsigned long long* counter) { *counter = 0; }

using KernelFn = void (*)(World<float>, Tables<float>, const Exposure<float>*, const uint64_t*, uint32_t, uint64_t, uint64_t, uint64_t, uint64_t,
    Tally, Counters*, unsigned long long*, uint32_t, uint32_t, uint32_t, uint32_t, bool);

// waves: resolved by wavesFp32
template <int L, uint32_t S, uint32_t K, bool B>
KernelFn variant(uint32_t waves)
{
    return waves >= 6 ? transportPersistent<L, 6, S, K, B> : transportPersistent<L, 4, S, K, B>;
}

template <int L, uint32_t K>
KernelFn variant(uint32_t waves, const LdsPlan& plan)
{
    constexpr bool B = K == WORLD_CODES8;
    if (plan.stage >= STAGE_ALL)
        return variant<L, STAGE_ALL, K, B>(waves);
    if (plan.stage < STAGE_SMALL)
        return variant<L, STAGE_NONE, K, false>(waves);
    return B && plan.bounds ? variant<L, STAGE_SMALL, K, B>(waves) : variant<L, STAGE_SMALL, K, false>(waves);
}

template <int L>
KernelFn variant(uint32_t waves, const LdsPlan& plan, uint32_t kind)
{
    return kind == WORLD_CODES8 ? variant<L, WORLD_CODES8>(waves, plan)
        : kind == WORLD_PALETTE8          ? variant<L, WORLD_PALETTE8>(waves, plan)
        : kind == WORLD_PALETTE8_MEASURED ? variant<L, WORLD_PALETTE8_MEASURED>(waves, plan)
                                          : variant<L, WORLD_ANY>(waves, plan);
}

KernelFn kernelFor(int L, uint32_t waves, const LdsPlan& plan, uint32_t kind)
{
    return L == 0 ? variant<0>(waves, plan, kind) : L == 1 ? variant<1>(waves, plan, kind) : variant<2>(waves, plan, kind);
}

// the kind a world and its tables run as (after launchFp32 has dropped the
// codes and bounds where they do not pay)
uint32_t worldKind(const World<float>& w, const Tables<float>& t)
{
    if (!w.index24)
        return WORLD_ANY;
    if (w.codeBytes == 1 && t.lutSumBound)
        return WORLD_CODES8;
    if (w.codeBytes == 0 && w.voxelBytes == 1 && !t.lutSumBound)
        return w.measurement ? WORLD_PALETTE8_MEASURED : WORLD_PALETTE8;
    return WORLD_ANY;
}

}

// Resident waves per SIMD of a run: 6, or 4 at L = 2, whose interaction
// samplers spill at 80 VGPRs (1.5e8 histories of the impulse approximation:
// 47.5 ms with 6, 38.9 with 4)
uint32_t wavesFp32(uint32_t requested, int L)
{
    return requested == 0 ? (L == 2 ? 4u : 6u) : requested >= 6 ? 6u : 4u;
}

// bytes of LDS of a block: half a CU's 160 KiB less an allocation granule
constexpr uint32_t BLOCK_LDS = 80 * 1024 - 1280;
// Slots the staged tables have to leave a wave's pool. Code worlds of
// 192x160x120, 2e7 histories, ms at 48, 60, 72, 84, 96: 14 materials 3.28 3.32
// 3.02 3.04 3.63, 18 materials 3.68 3.29 3.30 3.27 3.78, 36 materials 4.17 4.03
// 4.04 4.06 4.09; L = 2, 18 materials 6.83 6.90 5.95 6.01 5.99, 30 materials
// 7.12 7.05 7.04 7.56 7.49.
constexpr uint32_t POOL_MIN = 72;

// what a run stages: the requested level, or by default the sampling tables
// (with the bounds of code worlds), less what leaves a wave's pool too few
// slots. The attenuation coefficients are staged on request only: they are
// read once an interaction, and the pool slots they would take are worth more.
LdsPlan planFp32(const dxmc_run_cfg& cfg, const Tables<float>& t, uint32_t W, uint32_t kind, bool pencil)
{
    const uint32_t level = cfg.lds_tables >= STAGE_NONE && cfg.lds_tables <= STAGE_ALL ? cfg.lds_tables : STAGE_SMALL;
    return planLds(t, level, cfg.low_energy_correction, kind == WORLD_CODES8, pencil, BLOCK_LDS, blockWaves(W), SLOT_BYTES,
        POOL_MIN);
}

bool usesCodesFp32(const dxmc_run_cfg& cfg, const Tables<float>& t, uint32_t voxelBytes, uint64_t voxels, bool pencil)
{
    const int L = cfg.low_energy_correction;
    return cfg.block_bounds != 0 || codesPay<float>(planFp32(cfg, t, wavesFp32(cfg.waves_per_simd, L), WORLD_CODES8, pencil), voxelBytes, voxels, L);
}

void launchFp32(dxmc_ctx* c, const dxmc_run_cfg& cfg, const World<float>& w, const Tables<float>& t, const Exposure<float>* exps,
    const uint64_t* expStart, uint32_t nExp, uint64_t hb, uint64_t he, const Tally& tally, Counters* ctr, unsigned long long* historyCounter, bool pencilBeam)
{
    const bool pencil = pencilBeam && w.index24;
    const int L = cfg.low_energy_correction;
    const uint64_t voxels = uint64_t(w.nx) * w.ny * w.nz;
    // the work counter is cleared by a kernel, not a memset, so the launch
    // sequence stays valid under stream capture
    auto* nx = historyCounter;
    hipLaunchKernelGGL(clearCounter, dim3(1), dim3(1), 0, c->stream, nx);
    World<float> world = w;
    Tables<float> tables = t;
    // the attenuation bounds pay where they also spare the record read
    // (worlds with codes); elsewhere the extra lookup costs more than the
    // evaluations it skips in diverged waves
    if ((cfg.flags & DXMC_RUN_EXACT_STEPS) || world.codeBytes == 0 || !usesCodesFp32(cfg, t, w.voxelBytes, voxels, pencil)) {
        world.codeBytes = 0;
        tables.lutSumBound = nullptr;
    }
    // the block code ranges spare most steps the code gather (CT spiral 180
    // ms against 277 without, CT-number world 34.6 against 46.8, DX 19.6
    // against 25.8); at L = 2, with 4 waves per SIMD, the longer chain of a
    // step whose draw falls in the block's band costs more than a code gather
    // from the Infinity Cache saves (401x333x151: 41.1 ms against 39.4), but
    // not more than one from HBM
    constexpr uint64_t INFINITY_CACHE_BYTES = uint64_t(256) << 20;
    const uint64_t codeArrayBytes = voxels * world.codeBytes;
    const bool blocksOn = world.codeBytes == 1 && world.blocks
        && (cfg.block_bounds == 1 || (cfg.block_bounds == 0 && !(L == 2 && codeArrayBytes <= INFINITY_CACHE_BYTES)));
    if (!blocksOn)
        world.blocks = nullptr;
    uint32_t kind = worldKind(world, tables);
    if (kind == WORLD_CODES8 && !world.blocks && L < 2)
        kind = WORLD_ANY;
    const uint32_t waves = wavesFp32(cfg.waves_per_simd, L);
    // launches with too few histories for full blocks on every CU get blocks
    // of fewer waves, spread over the CUs
    const uint64_t wavesNeeded = (he - hb + 63) / 64;
    const uint32_t wavesPerBlock = static_cast<uint32_t>(std::clamp<uint64_t>((wavesNeeded + c->numCU - 1) / c->numCU, 1, blockWaves(waves)));
    const LdsPlan plan = planFp32(cfg, tables, waves, kind, pencil);
    const uint32_t slots = plan.slots(wavesPerBlock);
    const uint32_t lds = plan.bytes + wavesPerBlock * slots * SLOT_BYTES;
    const uint32_t perCU = cfg.blocks_per_cu ? cfg.blocks_per_cu : 2u;
    // lanes without a photon before they are refilled (ms: CT spiral 8 185,
    // 12 180.5, 16 178.8, 20 181; DX 12 19.6, 16 19.3; impulse approximation
    // 12 40.9, 16 39.4, 20 38.3, 24 38.7)
    const uint32_t refill = cfg.regeneration_threshold ? std::min<uint32_t>(cfg.regeneration_threshold, 64u) : L == 2 ? 20u : 16u;
    // photons due before they interact, 48 or half the pool, 46 of its 93
    // slots on CT spiral (ms before the bounds were in LDS, with 48 and more
    // slots to half: 32 207, 40 202.4, 48 199.4, 56 198.7)
    const uint32_t interact = std::min<uint32_t>(cfg.interaction_threshold ? std::min<uint32_t>(cfg.interaction_threshold, 64u) : 48u, slots / 2);
    const uint64_t grid = std::clamp<uint64_t>((wavesNeeded + wavesPerBlock - 1) / wavesPerBlock, 1, static_cast<uint64_t>(c->numCU) * perCU);
    // histories a wave claims per atomic on the global counter
    const uint32_t pool = cfg.queue_depth ? std::clamp<uint32_t>(cfg.queue_depth, 64u, 1u << 16) : historiesPerClaim(he - hb, grid * wavesPerBlock);
    hipLaunchKernelGGL(kernelFor(L, waves, plan, kind), dim3(static_cast<uint32_t>(grid)), dim3(64 * wavesPerBlock), lds, c->stream,
        world, tables, exps, expStart, nExp, hb, he, cfg.seed, cfg.first_history, tally, ctr, nx, refill, interact, pool, slots, pencil);
}
}
