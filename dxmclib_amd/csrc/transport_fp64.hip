// FP64 photon transport: the plain method's histories on a persistent kernel.
//
// Same scheme as the FP32 kernel (transport_fp32.hip): one photon per lane in
// registers, flights advanced together, interactions run when enough lanes
// are due, new photons sampled by whole waves into an LDS queue. Every value
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

// per-wave queue of sampled photons (SoA of 4-byte words): position,
// direction, energy, weight, log10 E and 1 / majorant as 11 pairs of words
// (low, high), PCG state (2), the history's offset in the launch and the LUT
// segment
constexpr uint32_t QUEUE_DOUBLES = 10;
constexpr uint32_t QUEUE_WORDS = 2 * QUEUE_DOUBLES + 4;
__host__ __device__ constexpr uint32_t queueBytes(uint32_t capacity) { return QUEUE_WORDS * capacity * 4; }

// voxel coordinate (uint32_t)((pos - lower) / spacing) of the plain method,
// clamped to the grid: the product q with the reciprocal differs from the
// rounded quotient by less than 2^-51 q, so they truncate alike unless q is
// that near a whole number
__device__ inline bool nearWhole(double q) { return fabs(q - rint(q)) <= fabs(q) * 0x1p-50; }

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
    uint32_t nExp, regenThreshold, interactThreshold, poolSize, queueCapacity, exactSteps;
};

__device__ inline const Args64& loopArgs()
{
    auto p = (const __attribute__((address_space(4))) Args64*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const Args64*)p;
}

// K: world kind (WORLD_CODES8 with block codes, or WORLD_ANY: palette or
// 8-byte records). S: LDS staging level. Three waves per SIMD (168 VGPRs):
// the FP64 samplers' temporaries spill, and fewer waves with fewer spills won
// (CT spiral 384x384x200, 4e7 histories: 148 ms for the plain form, one
// thread a history; here 50.5 ms with 5 waves, 33.7 with 4, 28.4 with 3,
// 30.1 with 2; CTDI phantom, 2e7 histories: 19.9 ms plain, 8.7 with 3).
template <int L, uint32_t S, uint32_t K>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 8))) void transportPersistent64(Args64 args)
{
    extern __shared__ __align__(16) unsigned char lds[];
    Tables<double> t = args.t;
    stageTables<double, S, L>(t, lds);
    Particle<double> p;
    Rng rng { 0, 1 };
    double majInv = 0;
    bool update = true;
    uint32_t phase = DEAD;
    const uint64_t span = args.hEnd - args.hBegin;
    uint64_t poolNext = 0, poolEnd = 0;
    uint32_t poolExp = 0;
    bool claimedAll = span == 0;
    uint32_t events = 0; // scoring events of the lane's interactions
    uint32_t steps = 0;
    uint32_t historySteps = 0;
    uint64_t idx = 0;
    uint32_t matMeas = 0; // material | measurement flag << 24 of the voxel reached
    // the photon's place in the LUT (x = log10 E), and the FP32 filter's
    // copies: log2 E above the segment's node, 1 / majorant
    LutPoint<double> lp { 0, 0.0 };
    float x32 = 0, maj32 = 0;
    const uint32_t lane = __lane_id();

    const uint32_t cap = args.queueCapacity;
    uint32_t* q = reinterpret_cast<uint32_t*>(lds + ldsBytes(args.t, S, L) + (threadIdx.x / 64) * queueBytes(cap));
    uint32_t queued = 0;

    for (;;) {
        const uint64_t dead = __ballot(phase == DEAD);
        const uint32_t nDead = __popcll(dead);
        const bool work = poolNext < poolEnd || !claimedAll;
        if (work && queued < nDead) {
            const Args64& a = loopArgs();
            // sample with the whole wave: the next histories of the wave's
            // pool, those that enter the world join the queue
            const uint32_t want = cap - queued;
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
            if (sampled) {
                const uint32_t slot = queued + rankBelow(entered);
                const LutPoint<double> np0 = lutPoint(t, np.energy);
                const double v[QUEUE_DOUBLES] = { np.pos[0], np.pos[1], np.pos[2], np.dir[0], np.dir[1], np.dir[2], np.energy, np.weight, np0.x,
                    majorantInverseAt(t, np0) };
                for (uint32_t f = 0; f < QUEUE_DOUBLES; ++f) {
                    q[2 * f * cap + slot] = static_cast<uint32_t>(__double2loint(v[f]));
                    q[(2 * f + 1) * cap + slot] = static_cast<uint32_t>(__double2hiint(v[f]));
                }
                q[(2 * QUEUE_DOUBLES) * cap + slot] = static_cast<uint32_t>(nr.s);
                q[(2 * QUEUE_DOUBLES + 1) * cap + slot] = static_cast<uint32_t>(nr.s >> 32);
                q[(2 * QUEUE_DOUBLES + 2) * cap + slot] = nOffset;
                q[(2 * QUEUE_DOUBLES + 3) * cap + slot] = np0.k;
            }
            queued += __popcll(entered);
        }
        // dead lanes take photons from the queue (last in, first out)
        if (nDead >= args.regenThreshold || (nDead > 0 && !work)) {
            const Args64& a = loopArgs();
            const uint32_t take = nDead < queued ? nDead : queued;
            if (phase == DEAD) {
                const uint32_t r = rankBelow(dead);
                if (r < take) {
                    const uint32_t slot = queued - 1 - r;
                    double v[QUEUE_DOUBLES];
                    for (uint32_t f = 0; f < QUEUE_DOUBLES; ++f)
                        v[f] = __hiloint2double(static_cast<int>(q[(2 * f + 1) * cap + slot]), static_cast<int>(q[2 * f * cap + slot]));
                    for (int i = 0; i < 3; ++i) {
                        p.pos[i] = v[i];
                        p.dir[i] = v[3 + i];
                    }
                    p.energy = v[6];
                    p.weight = v[7];
                    rng.s = static_cast<uint64_t>(q[(2 * QUEUE_DOUBLES + 1) * cap + slot]) << 32 | q[(2 * QUEUE_DOUBLES) * cap + slot];
                    rng.inc = 2 * (a.firstHistory + a.hBegin + q[(2 * QUEUE_DOUBLES + 2) * cap + slot]) + 1;
                    lp.k = q[(2 * QUEUE_DOUBLES + 3) * cap + slot];
                    lp.x = v[8];
                    majInv = v[9];
                    x32 = static_cast<float>((lp.x - t.lutGrid[lp.k]) * LOG2_10);
                    maj32 = static_cast<float>(majInv);
                    update = false;
                    steps += historySteps;
                    historySteps = 0;
                    phase = FLYING;
                }
            }
            queued -= take;
        }
        const uint64_t pend = __ballot(phase == PENDING);
        const uint64_t fly = __ballot(phase == FLYING);
        if ((pend | fly) == 0) {
            if (poolNext >= poolEnd && claimedAll && queued == 0)
                break;
            continue;
        }
        const uint32_t nPend = __popcll(pend);
        if (nPend != 0 && (nPend >= args.interactThreshold || fly == 0)) {
            Deposits<double> deposits;
            if (phase == PENDING) {
                const Args64& a = loopArgs();
                const uint32_t mat = matMeas & 0xffu;
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
                    x32 = static_cast<float>((lp.x - t.lutGrid[lp.k]) * LOG2_10);
                    maj32 = static_cast<float>(majInv);
                    update = false;
                }
                phase = alive && historySteps < MAX_STEPS ? FLYING : DEAD;
            }
            events += deposits.n;
            const bool wide = K != WORLD_CODES8 && args.w.index24 == 0;
            scoreWave(args.tally, deposits.n > 0, idx, deposits.first, wide);
            if (K != WORLD_CODES8 && __ballot(deposits.n > 1) != 0) // forced events with a Compton event
                scoreWave(args.tally, deposits.n > 1, idx, deposits.second, wide);
        } else {
            // Woodcock flights of the FLYING lanes until the outer loop is needed
            for (;;) {
                if (phase == FLYING) {
                    const Args64& a = loopArgs();
                    const World<double>& w = a.w;
                    const double u1 = rng.uniform<double>();
                    const double step = -log(u1) * majInv * 10.0; // cm -> mm
                    for (int i = 0; i < 3; ++i)
                        p.pos[i] += p.dir[i] * step;
                    const bool in = insideFast(w, p.pos);
                    const uint3 vc = voxelCoords64(w, p.pos, a.inv); // clamped: a valid voxel also outside
                    idx = voxelIndexFast(w, vc, K == WORLD_CODES8 || w.index24 != 0);
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
                        const uint32_t bc = loadAt(w.blocks, blockIndexFast(w, vc));
                        matMeas = __umul24(bc >> 8, w.codeMul) >> CODE_MUL_SHIFT;
                        {
                            const float bLo = w.bounds[bc & 0xffu].lo;
                            const float bHi = w.bounds[bc >> 8].hi;
                            const float2 sb = loadAt(a.sumBound, __umul24(matMeas, t.lutNodes) + lp.k);
                            const float lo = sb.x * bLo * maj32, hi = sb.y * bHi * maj32;
                            settled = (bc != BLOCK_MIXED) & ((f2 < lo) | (f2 > hi));
                            real = f2 < lo;
                        }
                        if (!settled) {
                            const uint32_t code = loadAt(static_cast<const uint8_t*>(w.codes), static_cast<uint32_t>(idx));
                            matMeas = __umul24(code, w.codeMul) >> CODE_MUL_SHIFT;
                            const uint2 b = *reinterpret_cast<const uint2*>(w.bounds + code);
                            const float2 sb = loadAt(a.sumBound, __umul24(matMeas, t.lutNodes) + lp.k);
                            const float lo = sb.x * __uint_as_float(b.x) * maj32, hi = sb.y * __uint_as_float(b.y) * maj32;
                            settled = (f2 < lo) | (f2 > hi);
                            real = f2 < lo;
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
                    const bool measured = matMeas > 0xffffffu; // (code worlds carry no flags)
                    rng.s = (in & !measured) ? r2.s : rng.s;
                    uint32_t now = in ? ((measured | real) ? PENDING : FLYING) : DEAD;
                    if (now == FLYING && p.energy * p.weight < 5.0) { // Russian roulette
                        if (rng.uniform<double>() < 0.8)
                            now = DEAD;
                        else
                            p.weight *= 1.0 / (1.0 - 0.8);
                    }
                    historySteps += in ? 1u : 0u;
                    phase = (now == FLYING && historySteps >= MAX_STEPS) ? DEAD : now;
                }
                const uint64_t flyNow = __ballot(phase == FLYING);
                const uint32_t nPendNow = __popcll(__ballot(phase == PENDING));
                const uint32_t nDeadNow = __popcll(__ballot(phase == DEAD));
                if (flyNow == 0 || nPendNow >= args.interactThreshold || nDeadNow >= args.regenThreshold || (work && nDeadNow > queued)
                    || (!work && nDeadNow > 0 && queued > 0))
                    break;
            }
        }
    }
    if (args.ctr)
        dxmc_backend::accumulateCounters(args.ctr, steps + historySteps, events);
}

__global__ void clearCounter(unsigned long long* counter) { *counter = 0; }

using KernelFn = void (*)(Args64);

template <int L, uint32_t S>
KernelFn variant(uint32_t kind)
{
    return kind == WORLD_CODES8 ? transportPersistent64<L, S, WORLD_CODES8> : transportPersistent64<L, S, WORLD_ANY>;
}

KernelFn kernelFor(int L, bool staged, uint32_t kind)
{
    if (staged)
        return L == 0 ? variant<0, STAGE_SMALL>(kind) : L == 1 ? variant<1, STAGE_SMALL>(kind) : variant<2, STAGE_SMALL>(kind);
    return L == 0 ? variant<0, STAGE_NONE>(kind) : L == 1 ? variant<1, STAGE_NONE>(kind) : variant<2, STAGE_NONE>(kind);
}

}

namespace dxmc_backend {

void launchFp64(dxmc_ctx* c, const dxmc_run_cfg& cfg, const World<double>& w, const Tables<double>& t, const Tables<float>& t32,
    const Exposure<double>* exps, const uint64_t* expStart, uint32_t nExp, uint64_t hb, uint64_t he, const Tally& tally, Counters* ctr,
    unsigned long long* historyCounter)
{
    // cleared by a kernel, not a memset, so the sequence stays valid under capture
    hipLaunchKernelGGL(clearCounter, dim3(1), dim3(1), 0, c->stream, historyCounter);
    const int L = cfg.low_energy_correction;
    const uint32_t kind = w.index24 && w.codeBytes == 1 && w.blocks && t32.lutSumBound ? WORLD_CODES8 : WORLD_ANY;
    // queue capacity and staging with the most resident blocks, the staged
    // tables and the larger queue first among equals (CT spiral with 7
    // materials: 25 KB of tables and 64 photons fit 3 blocks, which is what
    // the registers allow)
    const uint32_t block = cfg.block_size ? cfg.block_size : 256;
    constexpr uint32_t LDS_PER_BLOCK = 64 * 1024;
    uint32_t cap = 64, lds = 0, perCU = 0;
    bool staged = true;
    for (const bool st : { true, false })
        for (const uint32_t q : { 64u, 48u, 32u }) {
            const uint64_t bytes = uint64_t(ldsBytes(t, st ? STAGE_SMALL : STAGE_NONE, L)) + block / 64 * queueBytes(q);
            if (bytes > LDS_PER_BLOCK)
                continue;
            int blocks = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, reinterpret_cast<const void*>(kernelFor(L, st, kind)), static_cast<int>(block), bytes)
                != hipSuccess) {
                hipGetLastError();
                blocks = 1;
            }
            if (static_cast<uint32_t>(std::max(blocks, 1)) > perCU) {
                cap = q;
                lds = static_cast<uint32_t>(bytes);
                perCU = static_cast<uint32_t>(std::max(blocks, 1));
                staged = st;
            }
        }
    if (cfg.blocks_per_cu)
        perCU = cfg.blocks_per_cu;
    // thresholds on CT spiral, ms: interaction 12 50.1, 20 42.1, 28 38.8, 40
    // 38.7 (at 4 waves); 28 28.4, 36 28.6, 44 30.7 (at 3); regeneration 1
    // 45.5, 4 38.8, 8 37.7, 16 39.0 (at 4)
    const uint32_t regen = cfg.regeneration_threshold ? std::min<uint32_t>(cfg.regeneration_threshold, 64u) : 8u;
    const uint32_t interact = cfg.interaction_threshold ? std::min<uint32_t>(cfg.interaction_threshold, 64u) : 28u;
    uint64_t grid = static_cast<uint64_t>(c->numCU) * perCU;
    grid = std::max<uint64_t>(1, std::min<uint64_t>(grid, (he - hb + block - 1) / block));
    // histories a wave claims per atomic on the global counter
    const uint32_t pool = cfg.queue_depth ? std::clamp<uint32_t>(cfg.queue_depth, 64u, 1u << 16) : 512u;

    const Args64 args { w, t, { 1.0 / w.spacing[0], 1.0 / w.spacing[1], 1.0 / w.spacing[2] }, t32.lutCoef, t32.lutSumBound, exps, expStart, hb, he,
        cfg.seed, cfg.first_history, tally, ctr, historyCounter, nExp, regen, interact, pool, cap, (cfg.flags & DXMC_RUN_EXACT_STEPS) != 0 };
    hipLaunchKernelGGL(kernelFor(L, staged, kind), dim3(static_cast<uint32_t>(grid)), dim3(block), lds, c->stream, args);
}
}
