// FP64 photon transport: the plain method's histories on a persistent kernel.
//
// Same scheme as the FP32 kernel (transport_fp32.hip): one photon per lane in
// registers, a pool of further ones in LDS, and flights, interactions and
// sampling each run with most of a wave's lanes. Every value
// that decides a history (position, direction, energy, weight, attenuation,
// majorant) is computed in FP64 by the code the plain method uses
// (device/physics.hpp, compiled without FMA contraction), so histories round
// like the CPU oracle's.
//
// What a Woodcock step cannot do without is two PCG draws, one FP64 log and
// the move. The plain form also spends a log10, three pow and three divisions
// a step (about 850 of its 1000 vector instructions); here
//   - the LUT point and the majorant are kept per photon and renewed when the
//     energy changes;
//   - the acceptance u < (total * density) / majorant is settled from FP32
//     bounds: block and voxel density codes with the segment's attenuation
//     bounds where the world has them (as in the FP32 kernel), else or then
//     the attenuation evaluated in FP32 with a margin far above its error.
//     Only a draw inside the margin (about 1 in 10^4) evaluates the FP64
//     attenuation, so the decisions are those of the FP64 evaluation;
//   - voxel coordinates come from products with the reciprocal spacing; a
//     quotient within rounding of a whole number is divided as the plain
//     method does.
#include "device/persistent.hpp"
#include "internal.hpp"

using namespace dxmc_dev;

namespace {

constexpr double LOG2_10 = 3.321928094887362347870319429489390175864831393;

// Relative margin of the FP32 evaluation of an acceptance probability: float
// coefficients (|log2 mu| < 1000 rounds to 3e-5 at most, 1e-6 for ordinary
// attenuations), the exponent's product and sum, the hardware exp2 and four
// products are each below 1e-6 for ordinary tables.
constexpr float FILTER_MARGIN = 1e-4f;

// A slot of a wave's photon pool (the ring of the FP32 kernel): ten doubles
// (position, direction, energy, weight, log10 E, 1 / majorant) as pairs of
// words, PCG state, the history's offset in the launch, LUT segment |
// material << 20 | measurement flag << 28, and the history's steps so far. 25
// words, an odd stride (see the FP32 kernel).
constexpr uint32_t SLOT_DOUBLES = 10;
constexpr uint32_t SLOT_WORDS = 2 * SLOT_DOUBLES + 5;
constexpr uint32_t SLOT_BYTES = SLOT_WORDS * 4;
constexpr uint32_t FLIGHTS_PER_LOOP = 64; // most flights before the outer loop runs
constexpr uint32_t WAVES_PER_CU = 8; // 2 a SIMD
// Slots the staged tables have to leave a wave's pool. Code worlds of
// 192x160x120, 5e6 histories, ms at 48, 60, 72, 84, 96: 27 materials 3.38 3.42
// 3.68 3.33 3.32, 30 materials 3.62 3.00 3.04 2.91 2.95, 40 materials 3.30 3.32
// 3.32 3.23 3.11; L = 2, 24 materials 5.16 5.06 4.55 4.40 4.41, 30 materials
// 4.91 4.91 4.86 4.88 4.56, 36 materials 7.05 7.20 6.18 6.23 6.17.
constexpr uint32_t POOL_MIN = 96;

// voxel coordinate (uint32_t)((pos - lower) / spacing) of the plain method,
// clamped to the grid: from the product with the reciprocal, divided where
// that may truncate differently
__device__ inline uint3 voxelCoords64(const World<double>& w, const double* pos, const double* inv)
{
    double q[3];
    bool nearFace = false;
    for (int i = 0; i < 3; ++i) {
        q[i] = (pos[i] - w.extent[2 * i]) * inv[i];
        nearFace |= nearWhole(q[i]);
    }
    if (nearFace)
        for (int i = 0; i < 3; ++i)
            q[i] = (pos[i] - w.extent[2 * i]) / w.spacing[i];
    return make_uint3(min(static_cast<uint32_t>(q[0]), w.nx - 1), min(static_cast<uint32_t>(q[1]), w.ny - 1), min(static_cast<uint32_t>(q[2]), w.nz - 1));
}

// The kernel's only argument. The loops read it again on each pass through a
// pointer the compiler cannot follow (loopArgs): its 60-odd scalars then come
// by scalar loads where they are used, where kept in registers they were
// spilled to vector lanes and read back one by one in every flight.
struct Args64 {
    World<double> w;
    Tables<double> t;
    double inv[3]; // reciprocal spacing
    const float* coef32; // FP32 filter: attenuation coefficients and segment bounds
    const float2* sumBound;
    const Exposure<double>* exps;
    const uint64_t* expStart;
    uint64_t hBegin, hEnd, seed, firstHistory;
    Tally tally;
    Counters* ctr;
    unsigned long long* next;
    uint32_t nExp, refillThreshold, interactThreshold, poolSize, slots, exactSteps, pencil;
};

__device__ inline const Args64& loopArgs()
{
    auto p = (const __attribute__((address_space(4))) Args64*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const Args64*)p;
}

// K: world kind (WORLD_CODES8 with block codes, or WORLD_ANY: palette or
// 8-byte records). S: LDS staging level. BOUNDS_LDS: the bounds of a code world
// staged too. Two waves per SIMD (256 VGPRs): the
// FP64 samplers' temporaries spill with less. CT spiral 384x384x200, 4e7
// histories: 148 ms for the plain form (one thread a history); without pools
// 50.5 ms with 5 waves, 33.7 with 4, 28.4 with 3; with pools 31.6 with 4, 22.4
// with 3, 21.8 with 2 (186 vector instructions a history, vector issue 58 %
// busy). CTDI phantom, 2e7 histories: 19.9 ms plain, 8.7 without pools, 6.8.
template <int L, uint32_t S, uint32_t K, bool BOUNDS_LDS>
__global__ __launch_bounds__(64 * WAVES_PER_CU) __attribute__((amdgpu_waves_per_eu(2, 8))) void transportPersistent64(Args64 args)
{
    extern __shared__ __align__(16) unsigned char lds[];
    Tables<double> t = args.t;
    stageTables<double, S, L>(t, lds);
    // density intervals and attenuation bounds of code worlds
    const float2* sumBound = args.sumBound;
    const float2* bounds = nullptr;
    uint32_t poolAt = static_cast<uint32_t>(ldsBytes(args.t, S, L));
    if constexpr (BOUNDS_LDS) {
        unsigned char* c = lds + poolAt;
        sumBound = stageArray(args.sumBound, uint64_t(t.nMaterials) * t.lutNodes, c);
        float2* d = reinterpret_cast<float2*>(c);
        for (uint32_t i = threadIdx.x; i < 256; i += blockDim.x)
            d[i] = make_float2(args.w.bounds[i].lo, args.w.bounds[i].hi);
        bounds = d;
        poolAt += static_cast<uint32_t>(boundsBytes(args.t));
        __syncthreads();
    }
    Particle<double> p;
    Rng rng { 0, 1 };
    double majInv = 0;
    bool flying = false, due = false; // neither: the lane holds no photon
    const uint64_t span = args.hEnd - args.hBegin;
    uint64_t poolNext = 0, poolEnd = 0;
    uint32_t poolExp = 0;
    bool claimedAll = span == 0;
    uint32_t events = 0, steps = 0, historySteps = 0;
    uint32_t matMeas = 0; // material | measurement flag << 24 of the voxel reached
    // the photon's place in the LUT (x = log10 E), and the FP32 filter's
    // copies: log2 E above the segment's node, 1 / majorant
    LutPoint<double> lp { 0, 0.0 };
    float x32 = 0, maj32 = 0;
    const uint32_t lane = __lane_id();

    const ScoreCache cache(lds + poolAt);
    if (args.pencil) {
        poolAt += SCORE_CACHE_BYTES;
        cache.clear();
    }
    const uint32_t slots = args.slots;
    uint32_t* pool = reinterpret_cast<uint32_t*>(lds + poolAt + (threadIdx.x / 64) * (slots * SLOT_BYTES));
    uint32_t first = 0, ready = 0, pending = 0; // the ring's window (wave-uniform)
    auto slotAt = [&](uint32_t offset) {
        const uint32_t k = first + offset;
        return pool + (k >= slots ? k - slots : k) * SLOT_WORDS;
    };
    auto put = [](uint32_t* q, uint32_t f, double v) {
        q[2 * f] = static_cast<uint32_t>(__double2loint(v));
        q[2 * f + 1] = static_cast<uint32_t>(__double2hiint(v));
    };
    auto get = [](const uint32_t* q, uint32_t f) { return __hiloint2double(static_cast<int>(q[2 * f + 1]), static_cast<int>(q[2 * f])); };
    auto storeWords = [&](uint32_t* q, uint64_t launchFirst) {
        q[20] = static_cast<uint32_t>(rng.s);
        q[21] = static_cast<uint32_t>(rng.s >> 32);
        q[22] = static_cast<uint32_t>(rng.inc >> 1) - static_cast<uint32_t>(launchFirst);
        q[23] = lp.k | (matMeas & 0xffu) << 20 | (K != WORLD_CODES8 && matMeas >> 24 != 0 ? 1u << 28 : 0u);
        q[24] = historySteps;
    };
    auto store = [&](uint32_t* q, uint64_t launchFirst) {
        for (uint32_t i = 0; i < 3; ++i) {
            put(q, i, p.pos[i]);
            put(q, 3 + i, p.dir[i]);
        }
        put(q, 6, p.energy);
        put(q, 7, p.weight);
        put(q, 8, lp.x);
        put(q, 9, majInv);
        storeWords(q, launchFirst);
    };
    auto filter = [&]() { // the FP32 filter's copies
        x32 = static_cast<float>((lp.x - t.lutGrid[lp.k]) * LOG2_10);
        maj32 = static_cast<float>(majInv);
    };
    auto loadWords = [&](const uint32_t* v, uint64_t launchFirst) {
        rng.s = static_cast<uint64_t>(v[1]) << 32 | v[0];
        rng.inc = 2 * (launchFirst + v[2]) + 1;
        lp.k = v[3] & 0xfffffu;
        matMeas = (v[3] >> 20 & 0xffu) | (K != WORLD_CODES8 ? v[3] >> 28 << 24 : 0u);
        historySteps = v[4];
        filter();
    };
    auto load = [&](const uint32_t* q, uint64_t launchFirst) {
        for (uint32_t i = 0; i < 3; ++i) {
            p.pos[i] = get(q, i);
            p.dir[i] = get(q, 3 + i);
        }
        p.energy = get(q, 6);
        p.weight = get(q, 7);
        lp.x = get(q, 8);
        majInv = get(q, 9);
        loadWords(q + 20, launchFirst);
    };

    for (;;) {
        const uint64_t dueMask = __ballot(due);
        uint64_t flyMask = __ballot(flying);
        const uint32_t nDue = __popcll(dueMask);
        const uint32_t nFly = __popcll(flyMask);
        const uint32_t room = slots - ready - pending;
        const bool work = poolNext < poolEnd || !claimedAll;
        const bool canSample = work && room > POOL_RESERVE;
        // when interactions run, and how their photons come to the lanes: as
        // in the FP32 kernel
        const uint32_t waiting = nDue + pending;
        if (waiting != 0
            && (waiting >= args.interactThreshold || nDue > room || (!work && ready == 0 && waiting >= nFly)
                || (nFly == 0 && ready == 0 && !canSample))) {
            const Args64& a = loopArgs();
            const uint64_t launchFirst = a.firstHistory + a.hBegin;
            const uint64_t emptyMask = ~(dueMask | flyMask);
            const uint32_t back = min(64u - nDue - nFly, pending);
            const uint32_t front = min(nFly, pending - back);
            const bool taken = !due && !flying && rankBelow(emptyMask) < back;
            const bool exchanged = flying && rankBelow(flyMask) < front;
            if (taken || exchanged) {
                uint32_t* q = slotAt(taken ? ready + pending - 1 - rankBelow(emptyMask) : ready + rankBelow(flyMask));
                if (exchanged) { // field by field: few values live twice
                    auto swap = [&](uint32_t f, double& x) {
                        const double v = get(q, f);
                        put(q, f, x);
                        x = v;
                    };
                    for (uint32_t i = 0; i < 3; ++i) {
                        swap(i, p.pos[i]);
                        swap(3 + i, p.dir[i]);
                    }
                    swap(6, p.energy);
                    swap(7, p.weight);
                    swap(8, lp.x);
                    swap(9, majInv);
                    const uint32_t v[5] = { q[20], q[21], q[22], q[23], q[24] };
                    storeWords(q, launchFirst);
                    loadWords(v, launchFirst);
                } else {
                    steps += historySteps;
                    load(q, launchFirst);
                }
                due = true;
                flying = false;
            }
            pending -= back + front;
            ready += front;
            Deposits<double> deposits;
            uint64_t idx = 0;
            const bool wide = K != WORLD_CODES8 && a.w.index24 == 0;
            if (due) {
                const uint32_t mat = matMeas & 0xffu;
                idx = voxelIndexFast(a.w, voxelCoords64(a.w, p.pos, a.inv), !wide); // the voxel the flight ended in
                bool update = false;
                double att[3];
                attenuationAt(t, mat, lp, att);
                bool alive;
                if (K != WORLD_CODES8 && matMeas > 0xffffffu) { // forced event (measurement voxel)
                    const double prob = ((att[0] + att[1]) + att[2]) * a.w.density[idx] * majInv;
                    alive = computeInteractionsForced<double, L>(t, prob, att, p, mat, deposits, rng, update);
                } else {
                    alive = computeInteractions<double, L>(t, att, p, mat, deposits, rng, update);
                }
                if (alive && p.energy * p.weight < 5.0) { // Russian roulette
                    if (rng.uniform<double>() < 0.8)
                        alive = false;
                    else
                        p.weight *= 1.0 / (1.0 - 0.8);
                }
                if (alive && update) { // new energy: its LUT point and majorant
                    lp = lutPoint(t, p.energy);
                    majInv = majorantInverseAt(t, lp);
                    filter();
                }
                flying = alive && historySteps < MAX_STEPS;
                due = false;
            }
            events += deposits.n;
            bool scores = deposits.n > 0;
            if (a.pencil && scores)
                scores = !cache.add(static_cast<uint32_t>(idx), deposits.first);
            scoreWave(a.tally, scores, idx, deposits.first, wide);
            if (K != WORLD_CODES8 && __ballot(deposits.n > 1) != 0) // forced events with a Compton event
                scoreWave(a.tally, deposits.n > 1, idx, deposits.second, wide);
        } else if (nDue != 0) {
            // photons with an interaction due wait in the pool
            if (due) {
                store(slotAt(ready + pending + rankBelow(dueMask)), args.firstHistory + args.hBegin);
                historySteps = 0;
                due = false;
            }
            pending += nDue;
        }
        flyMask = __ballot(flying);
        const uint32_t nEmpty = 64u - __popcll(flyMask);
        if (work && ready < nEmpty && slots - ready - pending > POOL_RESERVE) {
            // sample with the whole wave: the next histories of the wave's
            // range, those that enter the world join the ready ones
            const Args64& a = loopArgs();
            const uint32_t want = min(64u, slots - ready - pending - POOL_RESERVE);
            uint32_t assigned = 0;
            bool sampled = false;
            Particle<double> np;
            Rng nr { 0, 1 };
            uint32_t nOffset = 0;
            while (assigned < want) {
                if (poolNext >= poolEnd) {
                    if (claimedAll)
                        break;
                    if (!claimHistories(a.next, a.poolSize, span, a.hBegin, lane, poolNext, poolEnd)) {
                        claimedAll = true;
                        break;
                    }
                    if (poolEnd == a.hEnd)
                        claimedAll = true;
                    poolExp = upperBound(a.expStart, a.nExp + 1, poolNext) - 1;
                }
                const uint64_t avail = poolEnd - poolNext;
                const uint32_t take = avail < want - assigned ? static_cast<uint32_t>(avail) : want - assigned;
                if (lane >= assigned && lane < assigned + take) {
                    const uint64_t h = poolNext + (lane - assigned);
                    uint32_t e = poolExp;
                    while (h >= a.expStart[e + 1])
                        ++e;
                    nr = Rng::forHistory(a.seed, a.firstHistory + h);
                    nOffset = static_cast<uint32_t>(h - a.hBegin);
                    sampleParticle(a.exps[e], t, nr, np);
                    sampled = transportToWorld(a.w, np);
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
                const LutPoint<double> np0 = lutPoint(t, np.energy);
                for (uint32_t i = 0; i < 3; ++i) {
                    put(q, i, np.pos[i]);
                    put(q, 3 + i, np.dir[i]);
                }
                put(q, 6, np.energy);
                put(q, 7, np.weight);
                put(q, 8, np0.x);
                put(q, 9, majorantInverseAt(t, np0));
                q[20] = static_cast<uint32_t>(nr.s);
                q[21] = static_cast<uint32_t>(nr.s >> 32);
                q[22] = nOffset;
                q[23] = np0.k;
                q[24] = 0;
            }
        }
        poolFence(); // slots written above, read below by other lanes
        // lanes without a photon take ready ones from the front of the window
        const uint32_t take = min(nEmpty, ready);
        if (take != 0) {
            const uint32_t r = rankBelow(~flyMask);
            if (!flying && r < take) {
                steps += historySteps;
                load(slotAt(r), args.firstHistory + args.hBegin);
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
        // Woodcock flights of the flying lanes until the outer loop is needed
        const uint32_t limit = more ? args.refillThreshold : 64u;
        const uint64_t faintMask = __ballot(p.energy * p.weight < 5.0);
        const bool nearCap = __ballot(flying && historySteps >= MAX_STEPS - FLIGHTS_PER_LOOP) != 0;
        for (uint32_t n = 0; n < FLIGHTS_PER_LOOP; ++n) {
            if (flying) {
                const Args64& a = loopArgs();
                const World<double>& w = a.w;
                const double u1 = rng.uniform<double>();
                const double step = -log(u1) * majInv * 10.0; // cm -> mm
                for (int i = 0; i < 3; ++i)
                    p.pos[i] += p.dir[i] * step;
                flying = insideFast(w, p.pos);
                if (flying) {
                    const uint3 vc = voxelCoords64(w, p.pos, a.inv);
                    const uint64_t idx = voxelIndexFast(w, vc, K == WORLD_CODES8 || w.index24 != 0);
                    Rng r2 = rng;
                    const uint32_t n2 = r2.next();
                    const double u2 = static_cast<double>(n2) * 2.32830643653869628906e-010;
                    const float f2 = static_cast<float>(n2) * 2.32830643653869628906e-010f;
                    // u2 against FP32 bounds of the acceptance probability;
                    // equality, infinities and NaN settle nothing
                    bool settled = false, real = false;
                    // total attenuation in FP32 times a density, with the margin
                    auto evaluate = [&](float density) {
                        const float* c = a.coef32 + (__umul24(matMeas, t.lutNodes) + lp.k) * 6u;
                        const float total = __builtin_amdgcn_exp2f(c[0] + c[1] * x32) + __builtin_amdgcn_exp2f(c[2] + c[3] * x32)
                            + __builtin_amdgcn_exp2f(c[4] + c[5] * x32);
                        const float prob = total * density * maj32;
                        settled = fabsf(f2 - prob) > prob * FILTER_MARGIN;
                        real = f2 < prob;
                    };
                    if constexpr (K == WORLD_CODES8) {
                        auto bracket = [&](float dLo, float dHi) {
                            const uint32_t row = __umul24(matMeas, t.lutNodes) + lp.k;
                            const float2 sb = BOUNDS_LDS ? sumBound[row] : loadAt(a.sumBound, row);
                            const float lo = sb.x * dLo * maj32, hi = sb.y * dHi * maj32;
                            settled = (f2 < lo) | (f2 > hi);
                            real = f2 < lo;
                        };
                        const uint32_t bc = loadAt(w.blocks, blockIndexFast(w, vc));
                        matMeas = __umul24(bc >> 8, w.codeMul) >> CODE_MUL_SHIFT;
                        if constexpr (BOUNDS_LDS)
                            bracket(bounds[bc & 0xffu].x, bounds[bc >> 8].y);
                        else
                            bracket(w.bounds[bc & 0xffu].lo, w.bounds[bc >> 8].hi);
                        settled &= bc != BLOCK_MIXED;
                        if (!settled) {
                            const uint32_t code = loadAt(static_cast<const uint8_t*>(w.codes), static_cast<uint32_t>(idx));
                            matMeas = __umul24(code, w.codeMul) >> CODE_MUL_SHIFT;
                            if constexpr (BOUNDS_LDS)
                                bracket(bounds[code].x, bounds[code].y);
                            else
                                bracket(w.bounds[code].lo, w.bounds[code].hi);
                            if (!settled)
                                evaluate(static_cast<float>(w.density[idx]));
                        }
                    } else {
                        float density;
                        readVoxelPacked(w, w.voxelBytes, idx, matMeas, density);
                        evaluate(density); // 24-bit row product: flag ignored
                    }
                    if (!settled | (a.exactSteps != 0)) {
                        double att[3];
                        attenuationAt(t, matMeas, lp, att);
                        real = u2 < ((att[0] + att[1]) + att[2]) * w.density[idx] * majInv;
                    }
                    // a forced event draws no decision (code worlds carry no flags)
                    const bool measured = K != WORLD_CODES8 && matMeas > 0xffffffu;
                    rng.s = measured ? rng.s : r2.s;
                    due = measured | real;
                    flying = !due;
                    if (flying & __builtin_amdgcn_inverse_ballot_w64(faintMask)) // Russian roulette
                        if (p.energy * p.weight < 5.0) {
                            if (rng.uniform<double>() < 0.8)
                                flying = false;
                            else
                                p.weight *= 1.0 / (1.0 - 0.8);
                        }
                    ++historySteps;
                    if (nearCap && historySteps >= MAX_STEPS) // an interaction due is still run
                        flying = false;
                }
            }
            const uint32_t flyNow = __popcll(__ballot(flying));
            if (flyNow == 0 || 64u - flyNow >= limit || (!more && __popcll(__ballot(due)) + pending >= flyNow))
                break;
        }
    }
    if (args.pencil)
        cache.flush(args.tally);
    if (args.ctr)
        dxmc_backend::accumulateCounters(args.ctr, steps + historySteps, events);
}

__global__ void clearCounter(unsigned long long* counter) { *counter = 0; }

using KernelFn = void (*)(Args64);

template <int L>
KernelFn variant(const LdsPlan& plan, uint32_t kind)
{
    if (kind != WORLD_CODES8)
        return plan.stage >= STAGE_SMALL ? transportPersistent64<L, STAGE_SMALL, WORLD_ANY, false> : transportPersistent64<L, STAGE_NONE, WORLD_ANY, false>;
    return plan.bounds ? transportPersistent64<L, STAGE_SMALL, WORLD_CODES8, true>
        : plan.stage >= STAGE_SMALL ? transportPersistent64<L, STAGE_SMALL, WORLD_CODES8, false>
                                    : transportPersistent64<L, STAGE_NONE, WORLD_CODES8, false>;
}

KernelFn kernelFor(int L, const LdsPlan& plan, uint32_t kind) { return L == 0 ? variant<0>(plan, kind) : L == 1 ? variant<1>(plan, kind) : variant<2>(plan, kind); }

}

namespace dxmc_backend {

namespace {

// (a block size that is no multiple of 64 is refused before a launch)
uint32_t blockWaves(const dxmc_run_cfg& cfg) { return cfg.block_size ? std::clamp(cfg.block_size / 64, 1u, WAVES_PER_CU) : WAVES_PER_CU; }

// what a run stages: a block's share of the CU's 160 KiB less an allocation
// granule
LdsPlan planFp64(const dxmc_run_cfg& cfg, const Tables<double>& t, bool codes, bool pencil)
{
    const uint32_t waves = blockWaves(cfg);
    return planLds(t, STAGE_SMALL, cfg.low_energy_correction, codes, pencil, 160 * 1024 / (WAVES_PER_CU / waves) - 1280, waves, SLOT_BYTES, POOL_MIN);
}

}

bool usesCodesFp64(const dxmc_run_cfg& cfg, const Tables<double>& t, uint32_t voxelBytes, uint64_t voxels, bool pencil)
{
    return cfg.block_bounds != 0 || codesPay<double>(planFp64(cfg, t, true, pencil), voxelBytes, voxels, cfg.low_energy_correction);
}

void launchFp64(dxmc_ctx* c, const dxmc_run_cfg& cfg, const World<double>& w, const Tables<double>& t, const Tables<float>& t32,
    const Exposure<double>* exps, const uint64_t* expStart, uint32_t nExp, uint64_t hb, uint64_t he, const Tally& tally, Counters* ctr,
    unsigned long long* historyCounter, bool pencilBeam)
{
    const bool pencil = pencilBeam && w.index24;
    // cleared by a kernel, not a memset, so the sequence stays valid under capture
    hipLaunchKernelGGL(clearCounter, dim3(1), dim3(1), 0, c->stream, historyCounter);
    const int L = cfg.low_energy_correction;
    const bool codes = w.index24 && w.codeBytes == 1 && w.blocks && t32.lutSumBound
        && usesCodesFp64(cfg, t, w.voxelBytes, uint64_t(w.nx) * w.ny * w.nz, pencil);
    const uint32_t kind = codes ? WORLD_CODES8 : WORLD_ANY;
    // one block of 8 waves a CU, so the tables are held once and the rest of
    // the LDS is the waves' pools; a block size asked for divides them.
    // Launches with too few histories get blocks of fewer waves.
    const uint64_t wavesNeeded = (he - hb + 63) / 64;
    const uint32_t fullBlock = blockWaves(cfg);
    const uint32_t perCU = cfg.blocks_per_cu ? cfg.blocks_per_cu : WAVES_PER_CU / fullBlock;
    const uint32_t wavesPerBlock = static_cast<uint32_t>(std::clamp<uint64_t>((wavesNeeded + c->numCU - 1) / c->numCU, 1, fullBlock));
    const LdsPlan plan = planFp64(cfg, t, codes, pencil);
    const uint32_t slots = plan.slots(wavesPerBlock);
    const uint32_t lds = plan.bytes + wavesPerBlock * slots * SLOT_BYTES;
    // thresholds on CT spiral, ms: interaction 48 22.3, 56 21.8, 64 21.9;
    // refill 10 22.2, 16 21.9, 20 21.9, 28 22.5
    const uint32_t refill = cfg.regeneration_threshold ? std::min<uint32_t>(cfg.regeneration_threshold, 64u) : 16u;
    const uint32_t interact = std::min<uint32_t>(cfg.interaction_threshold ? std::min<uint32_t>(cfg.interaction_threshold, 64u) : 56u, slots / 2);
    const uint64_t grid = std::clamp<uint64_t>((wavesNeeded + wavesPerBlock - 1) / wavesPerBlock, 1, static_cast<uint64_t>(c->numCU) * perCU);
    // histories a wave claims per atomic on the global counter
    const uint32_t pool = cfg.queue_depth ? std::clamp<uint32_t>(cfg.queue_depth, 64u, 1u << 16) : historiesPerClaim(he - hb, grid * wavesPerBlock);
    const Args64 args { w, t, { 1.0 / w.spacing[0], 1.0 / w.spacing[1], 1.0 / w.spacing[2] }, t32.lutCoef, t32.lutSumBound, exps, expStart, hb, he,
        cfg.seed, cfg.first_history, tally, ctr, historyCounter, nExp, refill, interact, pool, slots, (cfg.flags & DXMC_RUN_EXACT_STEPS) != 0, pencil };
    hipLaunchKernelGGL(kernelFor(L, plan, kind), dim3(static_cast<uint32_t>(grid)), dim3(64 * wavesPerBlock), lds, c->stream, args);
}
}
