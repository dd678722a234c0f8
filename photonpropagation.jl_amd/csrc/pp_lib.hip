// pp_lib.hip - libphotonprop_hip.so: gfx950 photon propagation kernels and the
// C ABI declared in include/photonprop_hip.h.
//
// Kernel design (one photon per lane, photons grid-strided over the launch):
//   * targets (float4 x,y,z,r^2) and the spectrum's inverse-CDF knots are
//     staged in LDS once per workgroup; target reads are wave-uniform
//     broadcasts;
//   * every photon draws from its own Philox4x32-10 stream (counter =
//     (word, photon id, source)), so hits do not depend on the launch shape;
//   * one Philox block per step supplies all four uniforms of a step;
//   * hits are compacted per wave: ballot + mbcnt rank, one 64-bit atomic per
//     wave, coalesced SoA stores; slots past capacity are dropped and flagged.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <numeric>
#include <string>
#include <vector>

#include "pp_device.h"
#include "pp_grid_build.h"
#include "pp_hits.h"
#include "pp_search.h"
#include "pp_stage.h"

#include <rocprim/device/device_radix_sort.hpp>

using pp::f3;

// ---------------------------------------------------------------------------
// device data
// ---------------------------------------------------------------------------
namespace {

using pp::HitRecord;
using pp::kMaxPhotonsPerSource;
using pp::kPidBits;
constexpr int kMaxTargets = 65535;

struct HitCols {
    HitRecord* rec;
    uint64_t capacity;
};

struct Counters {
    unsigned long long n_hits;    // reserved slots (may exceed capacity)
    unsigned long long n_lost;    // photons of started work that an overflow left incomplete
    unsigned int err;             // 1 = overflow
    unsigned int pad;
    // work counts of the instrumented kernel (pp_config.count_work)
    unsigned long long steps, tests, cells, walks;
    unsigned long long next_chunk;  // work-stealing counter of the batch kernel
};

struct KParams {
    const pp_source* sources;  // device copy of the source list (one launch per source)
    pp::Medium med;
    uint32_t k0, k1, src_ix;
    int32_t n_steps;
    uint64_t n_photons;
    const float4* targets;
    int32_t n_targets;
    // uniform grid over the targets (GridSearch)
    pp::GridDesc grid;
    const float4* cells;
    const uint16_t* cell_items;
    int32_t spec_n;
    int32_t spec_map;
    float spec_mono;
    float spec_nf, spec_lastf;  // float(spec_n), float(spec_n - 1)
    const float* spec;
    HitCols hits;
    Counters* counters;
    uint32_t queue_off;  // LDS byte offset of the waves' walk queues (grid searches)
};

// ---------------------------------------------------------------------------
// photon emission   src/photon_prop_cuda.jl:158-276
// ---------------------------------------------------------------------------
struct PhotonInit {
    f3 pos, dir;
    float time, wl;
    pp::MediumValues mv;
};

// The launch constants that an emission reads.
struct EmitParams {
    pp::Medium med;
    int32_t spec_n, spec_map;
    float spec_mono, spec_nf, spec_lastf;
};

// Launch constants read again from the kernel's arguments (KParams, the first
// one) through scalar loads, opaque to the optimiser: as values of the whole
// kernel the constants of the emission and of the walk did not fit the scalar
// registers, and the compiler kept 90 of them in lanes of vector registers,
// from which it read them back one by one for every group of photons (about 70
// v_readlane a group) and every batch of walks (7-10). With this and without a
// move after the last segment a cascade of 1e8 photons takes 7.29 ms of kernel
// time instead of 7.67, 1e8 photons of a point source 4.8 instead of 5.3.
#if defined(__HIP_DEVICE_COMPILE__)
using ConstParams = const __attribute__((address_space(4))) KParams;
#else
using ConstParams = const KParams;
#endif

__device__ __forceinline__ ConstParams* kernel_params() {
#if defined(__HIP_DEVICE_COMPILE__)
    ConstParams* c = (ConstParams*)__builtin_amdgcn_kernarg_segment_ptr();
    __asm__ volatile("" : "+s"(c));
    return c;
#else
    return nullptr;
#endif
}

__device__ __forceinline__ EmitParams emit_params() {
    ConstParams* c = kernel_params();
    EmitParams e;
    e.med = c->med;
    e.spec_n = c->spec_n;
    e.spec_map = c->spec_map;
    e.spec_mono = c->spec_mono;
    e.spec_nf = c->spec_nf;
    e.spec_lastf = c->spec_lastf;
    return e;
}

// p + s d, each component one FMA (the same bits wherever it is inlined)
__device__ __forceinline__ f3 add_scaled(f3 p, float s, f3 d) {
    return pp::make3(fmaf(s, d.x, p.x), fmaf(s, d.y, p.y), fmaf(s, d.z, p.z));
}

// sample_cherenkov_direction[_no_smear|_custom_smear]  :80-111, :134-154
__device__ __forceinline__ f3 cherenkov_dir(const pp_source& src, const pp::MediumValues& mv,
                                            const pp::Stream& s, int smear) {
    const uint4 x = s.block(PP_CTR_INIT_EXTRA | 1u);
    f3 ph = pp::dir_from_cos_phi(mv.cos_c, mv.sin_c, pp::u01(x.x));
    if (smear == 1) {
        ph = pp::rot_from_ez(pp::cherenkov_track_dir(pp::u01(x.y), pp::u01(x.z)), ph);
    } else if (smear == 2) {
        const float gx = pp::gamma_sample(src.beta_a, 1.0f, s, PP_SUB_BETA_X);
        const float gy = pp::gamma_sample(src.beta_b, 1.0f, s, PP_SUB_BETA_Y);
        const float tc = (gx / (gx + gy)) * 2.0f - 1.0f;
        const float ts = pp::sqrt_hw((1.0f - tc) * (1.0f + tc));
        ph = pp::rot_from_ez(pp::dir_from_cos_phi(tc, ts, pp::u01(x.y)), ph);
    }
    const f3 axis = pp::make3(src.direction[0], src.direction[1], src.direction[2]);
    return pp::rot_from_ez(axis, ph);
}

__device__ __forceinline__ PhotonInit init_photon(const EmitParams& p, const pp_source& src,
                                                  const float* spec, const pp::Stream& s) {
    const uint4 r = s.block(PP_CTR_INIT);
    PhotonInit st;
    st.wl = pp::spectrum_sample(spec, p.spec_n, p.spec_nf, p.spec_lastf, p.spec_map, p.spec_mono,
                                pp::u01(r.x));
    st.mv = pp::medium_values(p.med, st.wl);
    st.pos = pp::make3(src.position[0], src.position[1], src.position[2]);
    st.time = src.time;
    const f3 axis = pp::make3(src.direction[0], src.direction[1], src.direction[2]);
    switch (src.kind) {
    case PP_SRC_POINTLIKE_ISOTROPIC:
        st.dir = pp::isotropic_dir(pp::u01(r.y), pp::u01(r.z));
        break;
    case PP_SRC_POINTLIKE_TIME_RANGE:
        st.dir = pp::isotropic_dir(pp::u01(r.y), pp::u01(r.z));
        st.time = src.time + pp::u01(r.w) * (src.time_end - src.time);
        break;
    case PP_SRC_AXICONE: {
        float theta = src.angle;
        if (src.beam_divergence > 0.0f)
            theta += pp::normal_sample(s, PP_SUB_NORMAL) * src.beam_divergence;
        float sn, cs;
        sincosf(theta, &sn, &cs);
        st.dir = pp::rot_from_ez(axis, pp::dir_from_cos_phi(cs, sn, pp::u01(r.y)));
        break;
    }
    case PP_SRC_COLLIMATED_ISOTROPIC: {
        const float ct = src.cut_angle_cos + pp::u01(r.z) * (1.0f - src.cut_angle_cos);
        st.dir = pp::dir_from_cos_phi(ct, pp::sqrt_hw((1.0f - ct) * (1.0f + ct)), pp::u01(r.y));
        break;
    }
    case PP_SRC_PENCIL:
        if (src.beam_divergence > 0.0f) {
            const float theta =
                pp::sqrt_hw(pp::u01(r.y) * (src.beam_divergence * src.beam_divergence));
            float sn, cs;
            sincosf(theta, &sn, &cs);
            st.dir = pp::rot_from_ez(axis, pp::dir_from_cos_phi(cs, sn, pp::u01(r.z)));
        } else {
            st.dir = axis;
        }
        break;
    case PP_SRC_EXTENDED_CHERENKOV:
    case PP_SRC_EXTENDED_CHERENKOV_NO_SMEAR:
    case PP_SRC_EXTENDED_CHERENKOV_CUSTOM_SMEAR: {
        const float lp =
            pp::gamma_sample(src.long_a, 1.0f / src.long_b, s, PP_SUB_LONG_GAMMA) * src.long_lrad;
        st.pos = add_scaled(st.pos, lp, axis);
        st.time = src.time + lp * (1.0f / pp::kCVacMNs);
        const int smear = src.kind == PP_SRC_EXTENDED_CHERENKOV ? 1
                          : src.kind == PP_SRC_EXTENDED_CHERENKOV_NO_SMEAR ? 0 : 2;
        st.dir = cherenkov_dir(src, st.mv, s, smear);
        break;
    }
    case PP_SRC_POINTLIKE_CHERENKOV:
        st.dir = cherenkov_dir(src, st.mv, s, 1);
        break;
    case PP_SRC_CHERENKOV_TRACK:
    default: {
        const float along = pp::u01(r.y) * src.length;
        st.pos = add_scaled(st.pos, along, axis);
        st.time = src.time + along * (1.0f / pp::kCVacMNs);
        st.dir = cherenkov_dir(src, st.mv, s, 1);
        break;
    }
    }
    return st;
}

// ---------------------------------------------------------------------------
// wave-compacted hit store
// ---------------------------------------------------------------------------
struct HitRec {
    f3 pos, dir, init_dir;
    float wl, time, dist;
    int32_t module_ix, n_steps;
    uint64_t pid;
};

// x of the wave's first lane, as a scalar (the builtin returns an int, which would
// extend its sign into the high word)
__device__ __forceinline__ uint64_t uniform64(uint64_t x) {
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(x >> 32)) << 32) |
           (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)x);
}

// Returns false if this lane's record did not fit (overflow).
__device__ __forceinline__ bool store_hits(bool has_hit, const HitRec& h, uint32_t src_ix,
                                           const HitCols& out, Counters* ctr) {
    const uint64_t mask = __ballot(has_hit);
    if (mask == 0) return true;
    const uint32_t lane = __lane_id();
    const uint32_t rank =
        __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
    const uint32_t leader = (uint32_t)__builtin_ctzll(mask);
    unsigned long long base = 0;
    if (lane == leader) base = atomicAdd(&ctr->n_hits, (unsigned long long)__popcll(mask));
    const uint32_t blo = __builtin_amdgcn_readlane((uint32_t)base, leader);
    const uint32_t bhi = __builtin_amdgcn_readlane((uint32_t)(base >> 32), leader);
    base = ((unsigned long long)bhi << 32) | blo;
    if (!has_hit) return true;
    const uint64_t i = base + rank;
    if (i >= out.capacity) return false;
    float4* r = reinterpret_cast<float4*>(out.rec + i);
    r[0] = make_float4(h.pos.x, h.pos.y, h.pos.z, h.dir.x);
    r[1] = make_float4(h.dir.y, h.dir.z, h.init_dir.x, h.init_dir.y);
    r[2] = make_float4(h.init_dir.z, h.wl, h.time, h.dist);
    const uint64_t id = h.pid | ((uint64_t)(uint32_t)h.module_ix << kPidBits);
    r[3] = make_float4(__uint_as_float((uint32_t)id), __uint_as_float((uint32_t)(id >> 32)),
                       __int_as_float(h.n_steps), __uint_as_float(src_ix));
    return true;
}

// ---------------------------------------------------------------------------
// propagation kernel: cuda_propagate_photons!   src/photon_prop_cuda.jl:429-549
// ---------------------------------------------------------------------------
using pp::lds_bytes;

// kSearchGridMem: the grid search with its cells in LDS and its targets read from
// memory (L2 and the vector cache), where their LDS copy would cost resident waves
// kSearchGridGlobal: all its tables read from memory, for target lists whose
// records and grid tables exceed the LDS
// kSearchBruteQueued, kSearchMixedQueued: the every-target scans over queued
// segments, those that come near the targets' box. The scans are bound by the
// VALU: a test is 30-40 instructions for 64 lanes, of which few need it (photons
// leave the targets' box after a step or two). 1e7 photons on 24 panels, discs
// and spheres: 3.07 ms of kernel in the plain scan, 0.86 queued with the hits
// held back (take_hits) and the planes filtered (PlaneFilter)
enum {
    kSearchBrute = 0,
    kSearchGrid = 1,
    kSearchMixed = 2,
    kSearchGridGlobal = 3,
    kSearchGridMem = 4,
    kSearchBruteQueued = 5,
    kSearchMixedQueued = 6,
    kSearchKinds = 7
};
template <int SEARCH>
constexpr bool kLdsCells = SEARCH == kSearchGrid || SEARCH == kSearchGridMem;
// two records per target
template <int SEARCH>
constexpr bool kMixedList = SEARCH == kSearchMixed || SEARCH == kSearchMixedQueued;
// the grid searches and the queued scans search in batches (transport_group);
// the plain every-target scans test each step at once (transport_photon): they
// serve small launches, more than 2^26 - 1 steps, lists that leave no LDS for the
// queues, and callers who ask for them
constexpr bool deferred_kind(int search) {
    return search != kSearchBrute && search != kSearchMixed;
}
template <int SEARCH>
constexpr bool kDeferredWalk = deferred_kind(SEARCH);
template <int SEARCH>
constexpr bool kQueuedScan = SEARCH == kSearchBruteQueued || SEARCH == kSearchMixedQueued;

// LDS tables of one workgroup: targets, grid cells and items, spectrum knots
struct Lds {
    const float4* tgt;
    const float4* cells;
    const uint16_t* items;
    float* spec;
};

template <int SEARCH>
__device__ __forceinline__ Lds stage_lds(const KParams& p) {
    extern __shared__ float4 lds[];
    Lds l;
    if constexpr (SEARCH == kSearchGridGlobal) {
        // only the spectrum is staged; the search reads the device tables
        l.tgt = p.targets;
        l.cells = p.cells;
        l.items = p.cell_items;
        l.spec = reinterpret_cast<float*>(lds);
        for (int i = threadIdx.x; i < p.spec_n; i += blockDim.x) l.spec[i] = p.spec[i];
        __syncthreads();
        return l;
    }
    // a mixed (sphere and planar) list has two records per target
    const int n_rec = SEARCH == kSearchGridMem ? 0
                      : kMixedList<SEARCH> ? 2 * p.n_targets : p.n_targets;
    float4* const tgt = lds;
    float4* const cells = lds + n_rec;
    uint16_t* const items =
        reinterpret_cast<uint16_t*>(cells + (kLdsCells<SEARCH> ? 2 * p.grid.n_cells : 0));
    l.tgt = SEARCH == kSearchGridMem ? p.targets : tgt;
    l.cells = cells;
    l.items = items;
    l.spec = reinterpret_cast<float*>(items + (kLdsCells<SEARCH> ? ((p.grid.n_items + 1) & ~1) : 0));
    for (int i = threadIdx.x; i < n_rec; i += blockDim.x) tgt[i] = p.targets[i];
    if (kLdsCells<SEARCH>) {
        for (int i = threadIdx.x; i < 2 * p.grid.n_cells; i += blockDim.x) cells[i] = p.cells[i];
        for (int i = threadIdx.x; i < p.grid.n_items; i += blockDim.x) items[i] = p.cell_items[i];
    }
    for (int i = threadIdx.x; i < p.spec_n; i += blockDim.x) l.spec[i] = p.spec[i];
    __syncthreads();
    return l;
}

// An every-target scan whose segments near the targets' box are scanned in batches
template <typename Scan>
struct QueuedScan {
    Scan scan;
    pp::GridDesc box;  // its corners ox..oz, ex..ez alone
    __device__ __forceinline__ pp::BoxSides sides(f3 p) const { return pp::box_sides(box, p); }
    template <bool COUNT>
    __device__ __forceinline__ int find(f3 pos, f3 dir, float step, float& dt, pp::Work& w) const {
        return scan.template find<COUNT>(pos, dir, step, dt, w);
    }
};

template <int SEARCH>
__device__ __forceinline__ auto make_search(const KParams& p, const Lds& l) {
    if constexpr (SEARCH == kSearchBrute) {
        return pp::BruteSearch{l.tgt, p.n_targets};
    } else if constexpr (SEARCH == kSearchMixed) {
        return pp::MixedSearch{l.tgt, p.n_targets};
    } else if constexpr (SEARCH == kSearchBruteQueued) {
        return QueuedScan<pp::BruteSearch>{{l.tgt, p.n_targets}, p.grid};
    } else if constexpr (SEARCH == kSearchMixedQueued) {
        return QueuedScan<pp::MixedSearch>{{l.tgt, p.n_targets}, p.grid};
    } else {
        return pp::GridSearch{l.tgt, l.cells, l.items, p.grid};
    }
}
template <int SEARCH>
using SearchT = decltype(make_search<SEARCH>(std::declval<const KParams&>(), std::declval<const Lds&>()));

// The search for a batch: a grid search with its grid, and what it reads from
// memory, read again (kernel_params); the scans hold nothing worth reading again.
template <int SEARCH>
__device__ __forceinline__ SearchT<SEARCH> reread(const SearchT<SEARCH>& s) {
    if constexpr (SEARCH == kSearchGrid) {
        return pp::GridSearch{s.tgt, s.cells, s.items, kernel_params()->grid};
    } else if constexpr (SEARCH == kSearchGridMem) {
        ConstParams* const p = kernel_params();
        return pp::GridSearch{p->targets, s.cells, s.items, p->grid};
    } else if constexpr (SEARCH == kSearchGridGlobal) {
        ConstParams* const p = kernel_params();
        return pp::GridSearch{p->targets, p->cells, p->cell_items, p->grid};
    } else {
        return s;
    }
}

// position, distance and time after moving d along dir
__device__ __forceinline__ void move_by(f3& pos, float& dist, float& time, f3 dir, float d,
                                        float inv_c) {
    pos = add_scaled(pos, d, dir);
    dist += d;
    time = fmaf(d, inv_c, time);
}

// One photon's life: emission, then up to n_steps steps of
// src/photon_prop_cuda.jl:486-539. Returns true on a hit; h holds the record.
template <bool COUNT, typename Search>
__device__ __forceinline__ bool transport_photon(const KParams& p, const pp_source& src,
                                                 uint32_t src_ix, uint64_t pid, const float* spec,
                                                 const Search& search, const pp::Phase& phase,
                                                 pp::Work& work, unsigned long long& n_steps_done,
                                                 HitRec& h) {
    pp::Stream s{p.k0, p.k1, (uint32_t)pid, (uint32_t)(pid >> 32), src_ix};
    const PhotonInit st = init_photon(emit_params(), src, spec, s);
    const pp::StepStream ss(s);
    f3 pos = st.pos, dir = st.dir;
    float time = st.time, dist = 0.0f;
    const float ln2_sca = st.mv.sca_len * pp::kLn2, inv_c = st.mv.inv_c_grp;
    bool hit = false;
    int32_t module_ix = 0, n_at = 0;
    for (int32_t step = 1; step <= p.n_steps; ++step) {
        const uint4 r = ss.block((uint32_t)step);
        const float step_size = pp::step_length(pp::u01_open0(r.x), ln2_sca);
        // first target in index order whose near root lies inside the step
        float dt = 0.0f;
        const int found = search.template find<COUNT>(pos, dir, step_size, dt, work);
        if (COUNT) ++n_steps_done;
        if (found >= 0) {
            move_by(pos, dist, time, dir, dt, inv_c);
            hit = true;
            module_ix = found + 1;
            n_at = step;
            break;
        }
        if (step == p.n_steps) break;  // nothing follows the last segment
        move_by(pos, dist, time, dir, step_size, inv_c);
        const float ct = pp::phase_cos_words(phase, r.y, r.z);
        dir = pp::update_direction(dir, ct, pp::u01(r.w));
    }
    h = HitRec{pos, dir, st.dir, st.wl, time, dist, module_ix, n_at, pid};
    return hit;
}

// ---------------------------------------------------------------------------
// Deferred walk of the grid searches and queued scans. A wave transports its 64 photons step
// by step as in transport_photon, but a step whose segment comes near the
// grid box (its end points' box meets it) does not walk the grid at once: the
// segment becomes a job in the wave's LDS queue, the photon moves on as if
// nothing were hit, and whenever 64 jobs are queued every lane of the wave
// walks one of them. The walks of a step run with 20-30% of the lanes in the
// one-photon schedule (the others are outside the grid or done); in a batch
// every lane walks. A job that hits records (step << 16 | target) in its
// photon's LDS slot with an atomic minimum; the earliest step wins, which is
// the step at which transport_photon stops (its later steps were never taken
// by the reference and their jobs only lose the minimum), so a photon need
// not stop at a hit it does not yet know of. A hit's record holds the photon
// id, module and step; replay_hits_kernel then emits the few photons with a
// hit again and replays their steps up to it (same random stream, same
// arithmetic) for the rest of the record, so no emission state
// stays live across the steps. The result is that of transport_photon bit
// for bit.
// ---------------------------------------------------------------------------
// Jobs per wave: a batch of up to 64 runs at the start of a step whenever 64
// or more are pending or the step's new jobs would not fit, so at most kQueue
// are pending after any step.
constexpr uint32_t kQueue = 96;
constexpr uint32_t kHitSlots = 16;  // hits a wave of a queued scan holds back
constexpr uint32_t kWaveQueueBytes = kQueue * 32 + 64 * 8;
constexpr uint32_t kScanQueueBytes = kWaveQueueBytes + kHitSlots * 16;
constexpr uint32_t wave_queue_bytes(int search) {
    return search == kSearchBruteQueued || search == kSearchMixedQueued ? kScanQueueBytes
                                                                        : kWaveQueueBytes;
}
constexpr int32_t kDeferredMaxSteps = (1 << 26) - 1;  // step index of a job: 26 bits

struct WaveQueue {
    char* base;  // one address: the parts lie at constant offsets
    // 2 per job: (position, step length), (direction, lane | step << 6)
    __device__ __forceinline__ float4* job() const { return reinterpret_cast<float4*>(base); }
    // per lane: earliest (step << 16 | target) hit, ~0 if none
    __device__ __forceinline__ unsigned long long* key() const {
        return reinterpret_cast<unsigned long long*>(base + kQueue * 32);
    }
    // queued scans: hits not yet stored, a record's last 16 bytes each
    __device__ __forceinline__ uint4* out() const {
        return reinterpret_cast<uint4*>(base + kQueue * 32 + 64 * 8);
    }
};

template <int SEARCH>
__device__ __forceinline__ WaveQueue wave_queue(const KParams& p) {
    extern __shared__ float4 lds[];
    return WaveQueue{reinterpret_cast<char*>(lds) + p.queue_off +
                     (threadIdx.x >> 6) * wave_queue_bytes(SEARCH)};
}

// Orders the wave's LDS accesses: the LDS executes one wave's accesses in
// issue order, so only the compiler must not move them across this point.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// `n` slots of the hit buffer for the wave, the first of them in `first`. Returns
// those that lie beyond its end.
__device__ __forceinline__ uint32_t reserve_hits(uint32_t n, uint64_t& first) {
    ConstParams* const p = kernel_params();
    unsigned long long got = 0;
    if (__lane_id() == 0) got = atomicAdd(&p->counters->n_hits, (unsigned long long)n);
    first = uniform64(got);
    const uint64_t cap = (uint64_t)p->hits.capacity;
    const uint32_t fit = first >= cap ? 0u : cap - first < n ? (uint32_t)(cap - first) : n;
    if (fit < n && __lane_id() == 0) atomicOr(&p->counters->err, 1u);
    return n - fit;
}

// Of a hit record only the last 16 bytes: replay_hits_kernel writes the rest.
__device__ __forceinline__ void store_hit(uint64_t i, uint4 v) {
    ConstParams* const p = kernel_params();
    if (i < (uint64_t)p->hits.capacity) reinterpret_cast<uint4*>(p->hits.rec + i)[3] = v;
}

// The wave's `n` hits in q.out to the hit buffer. Returns those that did not fit.
__device__ __forceinline__ uint32_t store_queued(const WaveQueue& q, uint32_t n) {
    if (n == 0) return 0;
    wave_sync();
    const uint32_t lane = __lane_id();
    uint64_t first;
    const uint32_t lost = reserve_hits(n, first);
    if (lane < n) store_hit(first + lane, q.out()[lane]);
    wave_sync();
    return lost;
}

// The hits of a group (key: per lane, ~0 if none): a grid search stores them, a
// queued scan (HOLD) adds them to the wave's `count` in q.out, which are stored
// kHitSlots at a time. One atomic on the hit count per group with a hit was what
// bounded lists that most groups hit (the device serves them at one per 12 ns:
// 1e7 photons on 24 panels, discs and spheres 1.90 ms, with the slots 0.93); in
// the grid searches, with a hit in one group of ten, the slots' LDS and registers
// cost more than they save (1e8-photon cascade 7.1 -> 8.0 ms).
// Returns the hits that did not fit the buffer.
template <bool HOLD>
__device__ __forceinline__ uint32_t take_hits(const WaveQueue& q, bool hit, unsigned long long key,
                                              uint64_t first_pid, uint32_t src_ix,
                                              uint32_t& count) {
    const uint64_t m = __ballot(hit);
    if (m == 0) return 0;
    const uint32_t lane = __lane_id();
    const uint32_t n = (uint32_t)__popcll(m);
    const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    const uint64_t id = (first_pid + lane) | ((uint64_t)((uint32_t)(key & 0xFFFFu) + 1u) << kPidBits);
    const uint4 v = make_uint4((uint32_t)id, (uint32_t)(id >> 32), (uint32_t)(key >> 16), src_ix);
    uint32_t lost = 0;
    if constexpr (!HOLD) {
        uint64_t first;
        lost = reserve_hits(n, first);
        if (hit) store_hit(first + rank, v);
        return lost;
    }
    for (uint32_t done = 0; done < n;) {
        const uint32_t take = kHitSlots - count < n - done ? kHitSlots - count : n - done;
        if (hit && rank - done < take) q.out()[count + rank - done] = v;
        count += take;
        done += take;
        if (count == kHitSlots) {
            lost += store_queued(q, count);
            count = 0;
        }
    }
    return lost;
}

// One photon per lane (active lanes), the whole wave together. Hits go to the
// wave's queue; returns those that did not fit the hit buffer (wave-uniform).
template <bool COUNT, int SEARCH>
__device__ __forceinline__ uint32_t transport_group(const KParams& p, const pp_source& src,
                                                    uint32_t src_ix, uint64_t pid, bool active,
                                                    const float* spec, const SearchT<SEARCH>& search,
                                                    const pp::Phase& phase, const WaveQueue& q,
                                                    uint32_t& n_queued, pp::Work& work,
                                                    unsigned long long& n_steps_done) {
    const uint32_t lane = __lane_id();
    pp::Stream s{p.k0, p.k1, (uint32_t)pid, (uint32_t)(pid >> 32), src_ix};
    const pp::StepStream ss(s);
    // the wave's photon ids are consecutive: pid = wave_first + lane
    const uint64_t wave_first = uniform64(pid - lane);
    f3 pos = pp::make3(0.0f, 0.0f, 0.0f), dir = pos;
    float ln2_sca = 0.0f;
    if (active) {
        // only what the steps need stays live; a hit emits the photon again
        const PhotonInit st = init_photon(emit_params(), src, spec, s);
        pos = st.pos;
        dir = st.dir;
        ln2_sca = st.mv.sca_len * pp::kLn2;
    }
    // no hit yet: all ones, materialised here (a 64-bit constant kept in a
    // register pair across the photon loop was spilled and reloaded per photon)
    uint32_t ones;
    __asm__ volatile("v_mov_b32 %0, -1" : "=v"(ones));
    *reinterpret_cast<uint2*>(q.key() + lane) = make_uint2(ones, ones);
    // the stepping lanes as a wave mask (scalar). A photon whose hit is known
    // keeps stepping in a grid search: its later steps cannot change the earliest
    // (step, target), and with ~1e-3 of the photons hit, stopping them would cost
    // a read of every lane's key after each batch (an LDS round trip) for
    // nothing. The queued scans, whose targets may fill the sky, read the keys
    // after a batch that hit.
    uint64_t going_m = __ballot(active);
    // of the moving lanes' positions: a queued scan keeps them from the step before
    // (six compares fewer a step); the walks leave a grid search no scalar registers
    // for them (12: spilled around every batch, 7.8 -> 8.8 ms for a 1e8-photon cascade)
    pp::BoxSides start{};
    if constexpr (kQueuedScan<SEARCH>) start = search.sides(pos);
    uint32_t head = 0, count = 0;  // wave-uniform ring of pending jobs
    // every lane walks one pending job (lanes >= n none)
    auto walk_jobs = [&](uint32_t n) {
        wave_sync();
        const auto grid = reread<SEARCH>(search);
        int found = -1;
        float dt = 0.0f;
        unsigned long long key = 0;
        uint32_t owner = 0;
        if (lane < n) {
            uint32_t slot = head + lane;
            if (slot >= kQueue) slot -= kQueue;
            const float4 a = q.job()[2 * slot], b = q.job()[2 * slot + 1];
            const uint32_t meta = __float_as_uint(b.w);
            owner = meta & 63u;
            if (COUNT) work.walks += 1;
            found = grid.template find<COUNT>(pp::make3(a.x, a.y, a.z), pp::make3(b.x, b.y, b.z),
                                                a.w, dt, work);
            if (found >= 0) {
                key = ((unsigned long long)(meta >> 6) << 16) | (uint32_t)found;
                atomicMin(q.key() + owner, key);
            }
        }
        if constexpr (kQueuedScan<SEARCH>) {
            if (__ballot(found >= 0)) {
                wave_sync();
                going_m &= ~__ballot(q.key()[lane] != ~0ull);
            }
        }
        head += n;
        if (head >= kQueue) head -= kQueue;
        count -= n;
    };
    // one loop for the steps and the final batches, so that the walk is
    // inlined once
    // The lane conditions below are these scalar masks, applied with
    // inverse ballots: no per-lane copy of a condition is kept or converted.
    int32_t step = 0;
    bool stepping = true;  // wave-uniform
    for (;;) {
        stepping = stepping && step < p.n_steps && going_m != 0;
        if (!stepping && count == 0) break;
        // r, step_size and next are set and read only while stepping (a
        // uniform branch); every lane computes them, the moving lanes
        // (move_m) use them (no register is set for the others)
        uint64_t move_m = 0, m = 0;
        uint4 r;
        float step_size;
        f3 next;
        if (stepping) {
            move_m = going_m;
            ++step;
            r = ss.block((uint32_t)step);
            step_size = pp::step_length(pp::u01_open0(r.x), ln2_sca);
            next = add_scaled(pos, step_size, dir);
            // a walk only for a segment near the grid; the walk clips it exactly
            const pp::BoxSides end = search.sides(next);
            if constexpr (!kQueuedScan<SEARCH>) start = search.sides(pos);
            m = pp::touch_mask(start, end) & move_m;
            if constexpr (kQueuedScan<SEARCH>) start = end;
        }
        const uint32_t n_new = (uint32_t)__popcll(m);
        if (!stepping || count >= 64 || count + n_new > kQueue) walk_jobs(count < 64 ? count : 64);
        if (__builtin_amdgcn_inverse_ballot_w64(m)) {
            const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                            __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
            uint32_t slot = head + count + rank;
            if (slot >= kQueue) slot -= kQueue;
            q.job()[2 * slot] = make_float4(pos.x, pos.y, pos.z, step_size);
            q.job()[2 * slot + 1] =
                make_float4(dir.x, dir.y, dir.z, __uint_as_float(lane | ((uint32_t)step << 6)));
        }
        count += n_new;
        // nothing follows the last segment
        if (step < p.n_steps && __builtin_amdgcn_inverse_ballot_w64(move_m)) {
            pos = next;
            const float ct = pp::phase_cos_words(phase, r.y, r.z);
            dir = pp::update_direction(dir, ct, pp::u01(r.w));
        }
    }
    wave_sync();
    const unsigned long long key = q.key()[lane];
    const bool hit = active && key != ~0ull;
    if (COUNT && active) n_steps_done += hit ? (unsigned long long)(key >> 16) : (unsigned long long)p.n_steps;
    // the record holds the photon id, module and step; replay_hits_kernel
    // completes it (emission again, steps 1..k-1, the target's test of step
    // k for the distance within it), so that neither
    // the emission's state nor a second inlined emission stays in this
    // kernel's registers. The photon id is recomputed from the wave's first
    // id (scalar) and the lane.
    uint64_t first = wave_first;
    __asm__ volatile("" : "+s"(first));
    return take_hits<kQueuedScan<SEARCH>>(q, hit, key, first, src_ix, n_queued);
}

// Propagation of one source: cuda_propagate_photons! (src/photon_prop_cuda.jl:
// 429-549) with photons grid-strided over the launch.
// COUNT: instrumented variant that also counts photon steps, sphere tests
// and grid-cell visits (roofline accounting); the results are identical.
// Minimum waves per SIMD the register allocation must allow (the VGPR budget
// is 512 / waves per lane): 7 for the grid searches, whose walks wait for LDS
// (1e8-photon cascade on 320 targets: 7.07 ms, at 6 7.29, at 8 8.15; the
// 256-source batch on 1000 targets: 25.7, at 6 25.9, at 8 29.8, at 5 36.9),
// 6 for the every-target scans.
template <int SEARCH>
constexpr int kWavesPerSimd = kDeferredWalk<SEARCH> ? 7 : 6;
#define PP_PROPAGATE_ATTRS \
    __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(kWavesPerSimd<SEARCH>)))

// *p read through the constant address space: a scalar load into SGPRs for
// a wave-uniform address (the tables the kernels read are not written
// during a launch)
template <typename T>
__device__ __forceinline__ T load_constant(const T* p) {
#if defined(__HIP_DEVICE_COMPILE__)
    return *(const __attribute__((address_space(4))) T*)p;
#else
    return *p;
#endif
}

// The source record at sp, read through the constant address space (scalar
// loads into SGPRs), and the source index, both opaque to the optimiser: a
// caller that reads them in every iteration of a photon loop gets what the
// emission derives from the source computed in that iteration, not hoisted
// out of the loop into registers that spill to scratch.
__device__ __forceinline__ pp_source source_record(const pp_source* sp, uint32_t& si) {
#if defined(__HIP_DEVICE_COMPILE__)
    using ConstSource = const __attribute__((address_space(4))) pp_source;
    ConstSource* c = (ConstSource*)sp;
    __asm__ volatile("" : "+s"(c), "+s"(si));
    return *c;
#else
    return *sp;
#endif
}

// What a wave carries from group to group.
struct WaveState {
    WaveQueue q{};
    uint32_t n_queued = 0;    // hits in q.out
    unsigned long long n_steps_done = 0;
    pp::Work work;
};

// n photons (wave-uniform) that were not completed, only after the hit buffer
// overflowed: the completed ones are the launch's photons less these (counting
// them took an atomic per lane or wave at the end of every launch, 18 us of the
// README example's 36).
__device__ __forceinline__ void add_lost(uint64_t n) {
    if (n && __lane_id() == 0)
        atomicAdd(&kernel_params()->counters->n_lost, (unsigned long long)n);
}

// Photons of the groups of 64 that start at first, first + stride, ... before end.
__device__ __forceinline__ uint64_t strided_photons(uint64_t first, uint64_t end, uint64_t stride) {
    if (first >= end) return 0;
    const uint64_t more = (end - 1 - first) / stride;  // groups after the first
    const uint64_t last = first + more * stride;
    return more * 64 + (end - last < 64 ? end - last : 64);
}

// 64 photons from base on (up to end), one per lane, the whole wave together,
// hits stored or queued. Returns the photons (wave-uniform) whose hits the full buffer
// did not take: they are lost, and the wave takes no more.
template <bool COUNT, int SEARCH>
__device__ __forceinline__ uint32_t propagate_group(const KParams& p, const pp_source& src,
                                                    uint32_t src_ix, uint64_t base, uint64_t end,
                                                    const float* spec, const SearchT<SEARCH>& search,
                                                    const pp::Phase& phase, WaveState& w) {
    const uint64_t pid = base + __lane_id();
    if constexpr (kDeferredWalk<SEARCH>) {
        return transport_group<COUNT, SEARCH>(p, src, src_ix, pid, pid < end, spec, search, phase, w.q,
                                              w.n_queued, w.work, w.n_steps_done);
    } else {
        bool stored = true;
        if (pid < end) {
            HitRec h;
            const bool hit = transport_photon<COUNT>(p, src, src_ix, pid, spec, search, phase,
                                                     w.work, w.n_steps_done, h);
            stored = store_hits(hit, h, src_ix, p.hits, p.counters);
            if (!stored) atomicOr(&p.counters->err, 1u);
        }
        return (uint32_t)__popcll(__ballot(!stored));
    }
}

// The wave's queued hits stored, and its counts added.
template <bool COUNT, int SEARCH>
__device__ __forceinline__ void finish_wave(const KParams& p, WaveState& w) {
    if constexpr (kDeferredWalk<SEARCH>) add_lost(store_queued(w.q, w.n_queued));
    if (COUNT) {
        atomicAdd(&p.counters->steps, w.n_steps_done);
        atomicAdd(&p.counters->tests, (unsigned long long)w.work.tests);
        atomicAdd(&p.counters->cells, (unsigned long long)w.work.cells);
        atomicAdd(&p.counters->walks, (unsigned long long)w.work.walks);
    }
}

template <int PHASE, int SEARCH, bool COUNT = false>
__global__ void PP_PROPAGATE_ATTRS propagate_kernel(KParams p) {
    const Lds l = stage_lds<SEARCH>(p);
    pp::Phase phase = p.med.phase;
    phase.kind = PHASE;
    const auto search = make_search<SEARCH>(p, l);
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    WaveState w;
    if constexpr (kDeferredWalk<SEARCH>) w.q = wave_queue<SEARCH>(p);
    // whole waves of photons, the loop condition uniform across the wave
    for (uint64_t base = (uint64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~63u);
         base < p.n_photons; base += stride) {
        uint32_t si = p.src_ix;
        const pp_source src = source_record(p.sources + p.src_ix, si);
        const uint32_t lost =
            propagate_group<COUNT, SEARCH>(p, src, si, base, p.n_photons, l.spec, search, phase, w);
        if (__builtin_expect(lost != 0, 0)) {
            // the call fails: the wave's later groups are given up in one sum (an
            // atomic for each held a launch of 1e9 photons for 190 ms)
            add_lost(lost + strided_photons(base + stride, p.n_photons, stride));
            break;
        }
    }
    finish_wave<COUNT, SEARCH>(p, w);
}

// Batch of sources in one persistent launch. Work items are chunks of
// `chunk` consecutive photons of one source (chunk_prefix[s] = first chunk
// of source s). Each wave starts with the item of its index and then takes the
// next one from a global counter (work stealing: waves that drew cheap photons
// simply take more chunks) or, in a small launch (dealt), every waves-th item
// after it, and exits past the last item, so every wave ends.
// Chunks from split_from on are handed out as `parts` pieces of `piece`
// photons each (the last piece of a chunk may be shorter), so that the waves
// end closer together. Photon ids and random streams are those of the
// one-launch-per-source kernel: the hits are identical.
struct BatchParams {
    const pp_source* sources;
    const uint64_t* n_photons;     // per source
    const uint64_t* chunk_prefix;  // n_sources + 1
    int32_t n_sources;
    uint32_t chunk;                // multiple of 64
    uint32_t parts, piece;         // pieces per split chunk; photons per piece, a multiple of 64
    uint64_t split_from;           // first split chunk (the number of chunks: none)
    uint64_t n_items;              // chunks and pieces
    bool dealt;                    // every item by wave index, none from the counter
};

// A batch kernel's arguments, for the second of them read again like the first
struct BatchKernelArgs {
    KParams p;
    BatchParams b;
};
__device__ __forceinline__ BatchParams batch_params() {
#if defined(__HIP_DEVICE_COMPILE__)
    return reinterpret_cast<const __attribute__((address_space(4))) BatchKernelArgs*>(kernel_params())->b;
#else
    return BatchParams{};
#endif
}

struct BatchItem {
    int source;
    uint64_t first, end;  // its photons
};

// Work item k of the batch (k wave-uniform).
__device__ __forceinline__ BatchItem batch_item(uint64_t k) {
    const BatchParams b = batch_params();
    // chunk c, photons [off, off + len) of it
    uint64_t c = k;
    uint32_t off = 0, len = b.chunk;
    if (k >= b.split_from) {
        const uint32_t j = (uint32_t)(k - b.split_from);
        c = b.split_from + j / b.parts;
        off = (j % b.parts) * b.piece;
        len = b.chunk - off < b.piece ? b.chunk - off : b.piece;
    }
    // source of this chunk: last s with chunk_prefix[s] <= c
    int lo = 0, hi = b.n_sources - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (load_constant(b.chunk_prefix + mid) <= c) lo = mid;
        else hi = mid - 1;
    }
    BatchItem it;
    it.source = lo;
    const uint64_t n_src = load_constant(b.n_photons + lo);
    const uint64_t first = (c - load_constant(b.chunk_prefix + lo)) * b.chunk + off;
    // the last chunk's pieces may lie beyond the source's photons
    it.end = first + len < n_src ? first + len : n_src;
    it.first = first < it.end ? first : it.end;
    return it;
}

template <int PHASE, int SEARCH, bool COUNT = false>
__global__ void PP_PROPAGATE_ATTRS propagate_batch_kernel(KParams p, BatchParams) {
    const Lds l = stage_lds<SEARCH>(p);
    pp::Phase phase = p.med.phase;
    phase.kind = PHASE;
    const auto search = make_search<SEARCH>(p, l);
    WaveState w;
    if constexpr (kDeferredWalk<SEARCH>) w.q = wave_queue<SEARCH>(p);
    const uint32_t waves = gridDim.x * (blockDim.x >> 6);
    // the first item by the wave's index
    uint64_t next = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    for (;;) {
        const uint64_t ck = uniform64(next);
        if (ck >= batch_params().n_items) break;
        const BatchItem it = batch_item(ck);
        uint32_t lost = 0;
        for (uint64_t base = it.first; base < it.end; base += 64) {
            // the source index and record, opaque to the optimiser in every
            // iteration: what the emission derives from them is computed here
            // (one scalar reload per 64 photons) instead of being hoisted out
            // of the loop into registers that then spill to scratch
            uint32_t si = (uint32_t)it.source;
            const pp_source src = source_record(batch_params().sources + it.source, si);
            lost = propagate_group<COUNT, SEARCH>(p, src, si, base, it.end, l.spec, search, phase, w);
            if (__builtin_expect(lost != 0, 0)) {
                lost += (uint32_t)(it.end - base > 64 ? it.end - base - 64 : 0);
                break;
            }
        }
        if (__builtin_expect(lost != 0, 0)) {
            // the call fails; take no more chunks, and give those dealt to this wave up
            const BatchParams b = batch_params();
            uint64_t left = lost;
            if (b.dealt)
                for (uint64_t k = ck + waves; k < b.n_items; k += waves) {
                    const BatchItem rest = batch_item(k);
                    left += rest.end - rest.first;
                }
            add_lost(left);
            break;
        }
        next = ck;
        if (!batch_params().dealt && __lane_id() == 0)
            next = atomicAdd(&kernel_params()->counters->next_chunk, 1ull);
        next += waves;
    }
    finish_wave<COUNT, SEARCH>(p, w);
}

// The counters to pinned host memory, where the host reads them once the stream
// is done (a copy of their own took 10 us of a call).
__device__ __forceinline__ void publish(const Counters* c, Counters* host) {
    const unsigned long long* a = reinterpret_cast<const unsigned long long*>(c);
    unsigned long long* b = reinterpret_cast<unsigned long long*>(host);
    if (threadIdx.x < sizeof(Counters) / 8) b[threadIdx.x] = a[threadIdx.x];
}

__global__ void publish_counters_kernel(const Counters* c, Counters* host) { publish(c, host); }

// Completion of the hit records of the deferred-walk kernels (transport_group):
// a record holds the photon id, module (target + 1), step k and source. One
// lane per record emits the photon again, replays steps 1..k-1 with
// transport_photon's arithmetic on the same random stream (contraction off:
// the same bits as the one-photon schedule), takes step k's distance to the
// target from the walk's own sphere test on the same operands, and writes
// position, directions, wavelength, time and distance.
// sources: the call's source list on the device.
__global__ void __launch_bounds__(256) replay_hits_kernel(KParams p, const pp_source* sources,
                                                          Counters* host, bool mixed) {
    if (blockIdx.x == 0) publish(p.counters, host);
    const pp::Phase phase = p.med.phase;
    const unsigned long long n_hits = p.counters->n_hits;
    const uint64_t n = n_hits < (unsigned long long)p.hits.capacity ? n_hits : p.hits.capacity;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        float4* r = reinterpret_cast<float4*>(p.hits.rec + i);
        const float4 r3 = r[3];
        const uint64_t id = (uint64_t)__float_as_uint(r3.x) | ((uint64_t)__float_as_uint(r3.y) << 32);
        const uint64_t pid = id & (kMaxPhotonsPerSource - 1);
        const int32_t target = (int32_t)((id >> kPidBits) & 0xFFFFu) - 1;
        const int32_t k = __float_as_int(r3.z);
        const uint32_t si = __float_as_uint(r3.w);
        const pp_source src = sources[si];
        const pp::Stream s{p.k0, p.k1, (uint32_t)pid, (uint32_t)(pid >> 32), si};
        const pp::StepStream ss(s);
        const PhotonInit st = init_photon(emit_params(), src, p.spec, s);
        const float ln2_sca = st.mv.sca_len * pp::kLn2, inv_c = st.mv.inv_c_grp;
        f3 rp = st.pos, rd = st.dir;
        float rt = st.time, rdist = 0.0f;
        for (int32_t j = 1; j < k; ++j) {
            const uint4 w = ss.block((uint32_t)j);
            const float step_size = pp::step_length(pp::u01_open0(w.x), ln2_sca);
            move_by(rp, rdist, rt, rd, step_size, inv_c);
            const float ct = pp::phase_cos_words(phase, w.y, w.z);
            rd = pp::update_direction(rd, ct, pp::u01(w.w));
        }
        // step k, cut at the target: the distance as the search finds it
        const uint4 w = ss.block((uint32_t)k);
        const float step_size = pp::step_length(pp::u01_open0(w.x), ln2_sca);
        float d = 0.0f;
        const float4 t = p.targets[mixed ? 2 * target : target];
        const float4 e = mixed ? p.targets[2 * target + 1] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const uint32_t kind = mixed ? __float_as_uint(e.x) : (uint32_t)PP_SHAPE_SPHERE;
        if (kind == PP_SHAPE_SPHERE)
            pp::sphere_hit(t, rp, rd, pp::dir_excess(rd), step_size, d);
        else
            pp::plane_hit(kind, t, e, rp, rd, step_size, d);
        move_by(rp, rdist, rt, rd, d, inv_c);
        r[0] = make_float4(rp.x, rp.y, rp.z, rd.x);
        r[1] = make_float4(rd.y, rd.z, st.dir.x, st.dir.y);
        r[2] = make_float4(st.dir.z, st.wl, rt, rdist);
    }
}

// Zeroes the counters in a captured graph (a kernel node, not a memset node).
__global__ void clear_counters_kernel(Counters* c) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *c = Counters{};
}

// ---------------------------------------------------------------------------
// step-function evaluation kernel (parity tests)
// ---------------------------------------------------------------------------
struct EvalParams {
    int fn;
    int in_stride, out_stride;
    int64_t n;
    const float* in;
    float* out;
    pp::Medium med;
    const float* spec;
    int spec_n, spec_map;
    float spec_mono;
    float spec_nf, spec_lastf;  // float(spec_n), float(spec_n - 1)
};

__device__ __forceinline__ uint32_t bits(float x) { return __float_as_uint(x); }
__device__ __forceinline__ float as_f(uint32_t x) { return __uint_as_float(x); }

__global__ void __launch_bounds__(256) eval_fn_kernel(EvalParams e) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= e.n) return;
    const float* x = e.in + i * e.in_stride;
    float* y = e.out + i * e.out_stride;
    switch (e.fn) {
    case PP_FN_ISOTROPIC_DIR: {
        f3 d = pp::isotropic_dir(x[0], x[1]);
        y[0] = d.x; y[1] = d.y; y[2] = d.z;
        break;
    }
    case PP_FN_ROT_FROM_EZ: {
        f3 d = pp::rot_from_ez(pp::make3(x[0], x[1], x[2]), pp::make3(x[3], x[4], x[5]));
        y[0] = d.x; y[1] = d.y; y[2] = d.z;
        break;
    }
    case PP_FN_HG_COS: {
        pp::Phase ph = pp::make_phase(PP_PHASE_HG, x[0], 1.0f, 1.0f);
        y[0] = pp::hg_cos(ph, x[1]);
        break;
    }
    case PP_FN_ES_COS: {
        pp::Phase ph = pp::make_phase(PP_PHASE_MIXED_HG_ES, 0.5f, x[0], 0.0f);
        y[0] = pp::es_cos(ph, x[1]);
        break;
    }
    case PP_FN_UPDATE_DIR: {
        f3 d = pp::update_direction(pp::make3(x[0], x[1], x[2]), x[3], x[4]);
        y[0] = d.x; y[1] = d.y; y[2] = d.z;
        break;
    }
    case PP_FN_SPHERE_ISEC: {
        float d;
        const pp::f3 dir = pp::make3(x[7], x[8], x[9]);
        const bool h = pp::sphere_hit(make_float4(x[0], x[1], x[2], x[3] * x[3]),
                                      pp::make3(x[4], x[5], x[6]), dir, pp::dir_excess(dir),
                                      x[10], d);
        y[0] = h ? 1.0f : 0.0f;
        y[1] = h ? d : 0.0f;
        break;
    }
    case PP_FN_STEP_LEN:
        y[0] = pp::step_length(x[0], x[1] * pp::kLn2);
        break;
    case PP_FN_CASCADIA: {
        pp::MediumValues mv = pp::medium_values(e.med, x[0]);
        y[0] = mv.sca_len;
        y[1] = 1.0f / mv.inv_c_grp;
        y[2] = 1.0f / mv.cos_c;
        break;
    }
    case PP_FN_TRACK_DIR: {
        f3 d = pp::cherenkov_track_dir(x[0], x[1]);
        y[0] = d.x; y[1] = d.y; y[2] = d.z;
        break;
    }
    case PP_FN_PHILOX: {
        // the step path's StepStream, Stream{k0, k1, c1, c2, c3}.block(c0), and
        // the plain ten rounds of the emission draws: all ones where they differ
        const pp::Stream s{bits(x[4]), bits(x[5]), bits(x[1]), bits(x[2]), bits(x[3])};
        uint4 r = pp::StepStream(s).block(bits(x[0]));
        const uint4 g = pp::philox(make_uint4(bits(x[0]), bits(x[1]), bits(x[2]), bits(x[3])),
                                   bits(x[4]), bits(x[5]));
        if (r.x != g.x || r.y != g.y || r.z != g.z || r.w != g.w) r = make_uint4(~0u, ~0u, ~0u, ~0u);
        y[0] = as_f(r.x); y[1] = as_f(r.y); y[2] = as_f(r.z); y[3] = as_f(r.w);
        break;
    }
    case PP_FN_GAMMA: {
        pp::Stream s{bits(x[2]), bits(x[3]), bits(x[4]), bits(x[5]), bits(x[6])};
        float xa = 0.0f;
        y[0] = pp::gamma_sample(x[0], x[1], s, PP_SUB_LONG_GAMMA, &xa);
        y[1] = xa;
        break;
    }
    case PP_FN_SPECTRUM:
        y[0] = pp::spectrum_sample(e.spec, e.spec_n, e.spec_nf, e.spec_lastf, e.spec_map,
                                   e.spec_mono, x[0]);
        break;
    case PP_FN_SL_COS: {
        pp::Phase ph = pp::make_phase(PP_PHASE_MIXED_HG_SL, x[0], 1.0f, 0.0f);
        y[0] = pp::sl_cos(ph, x[1]);
        break;
    }
    case PP_FN_MIXED_HGES: {
        // the sampler the kernels run for a MixedHGES medium, on the random
        // words whose u01 are x[3], x[4] (multiples of 2^-24 in [0, 1))
        pp::Phase ph = pp::make_phase(PP_PHASE_MIXED_HG_ES, x[0], x[1], x[2]);
        const uint32_t wc = (uint32_t)(x[3] * 0x1p24f) << 8, wu = (uint32_t)(x[4] * 0x1p24f) << 8;
        y[0] = pp::phase_cos_words(ph, wc, wu);
        // the words form must give the float form's bits: NaN where it does not
        if (__float_as_uint(y[0]) != __float_as_uint(pp::hg_es_cos(ph, pp::u01(wc), pp::u01(wu))))
            y[0] = __uint_as_float(0x7fc00000u);
        break;
    }
    case PP_FN_PLANE_ISEC: {
        float d;
        const uint32_t kind = bits(x[0]);
        const float4 t = make_float4(x[1], x[2], x[3], x[4] * x[4]);
        const float4 ext = make_float4(x[0], x[4] / 2.0f, x[5] / 2.0f, 0.0f);
        const bool h = pp::plane_hit(kind, t, ext, pp::make3(x[6], x[7], x[8]),
                                     pp::make3(x[9], x[10], x[11]), x[12], d);
        y[0] = h ? 1.0f : 0.0f;
        y[1] = h ? d : 0.0f;
        break;
    }
    default:
        break;
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
thread_local std::string g_err;

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

#define PP_HIP(expr)                                                                     \
    do {                                                                                 \
        hipError_t e_ = (expr);                                                          \
        if (e_ != hipSuccess)                                                            \
            return fail(PP_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

pp::Medium lower_medium(const pp_medium& m) {
    pp::Medium d{};
    d.kind = m.kind;
    d.phase = pp::make_phase(m.phase_kind, m.hg_g, m.es_b, m.hg_fraction);
    d.sca_len = m.sca_len;
    d.c_grp = m.group_velocity;
    d.inv_c_grp = 1.0f / m.group_velocity;
    d.n_phase = m.phase_refractive_index;
    d.sca_scale = (double)m.sca_scale;
    d.kop1 = (double)0.0017f;
    d.kop2 = (double)(float)(1.34 * (double)m.vol_conc_small);
    d.kop3 = (double)(float)(0.312 * (double)m.vol_conc_large);
    // Quan & Fry (1995) coefficients; linear pressure term 1.45e-5 / atm
    const double S = m.salinity, T = m.temperature, P = m.pressure;
    d.qf0 = (float)(1.31405 + (1.779e-4 - 1.05e-6 * T + 1.6e-8 * T * T) * S - 2.02e-6 * T * T +
                    1.45e-5 * P);
    d.qf1 = (float)(15.868 + 0.01155 * S - 0.00423 * T);
    d.qf2 = (float)(-4382.0);
    d.qf3 = (float)(1.1455e6);
    d.qg1 = 2.0f * d.qf1;
    d.qg2 = 3.0f * d.qf2;
    d.qg3 = 4.0f * d.qf3;
    if (m.kind == PP_MEDIUM_ICE) {
        d.ice_pref = (float)((double)m.sca_scale * (1.0 - (double)m.hg_g) / (double)m.ice_b_dust_400);
        d.ice_alpha = m.ice_alpha_sca_dust;
    }
    return d;
}

bool finite3(const float* v) {
    return std::isfinite(v[0]) && std::isfinite(v[1]) && std::isfinite(v[2]);
}

}  // namespace

// What the automatic block size and placement of a launch depend on.
struct OccKey {
    const void* fn = nullptr;
    size_t tables = 0, mem_tables = 0;  // LDS tables with and without the targets
    int block = 0;                      // the set block size
    bool operator==(const OccKey& o) const {
        return fn == o.fn && tables == o.tables && mem_tables == o.mem_tables && block == o.block;
    }
};

struct pp_ctx {
    int device = 0;
    int n_cu = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    pp_config cfg{};
    void* hit_mem = nullptr;
    HitCols hits{};
    Counters* d_counters = nullptr;  // at the front of d_batch
    // in h_batch, after the staged zeros: the last propagation's, written by its last kernel
    Counters* h_counters = nullptr;
    bool has_medium = false;
    pp_medium medium_in{};
    pp::Medium medium{};
    bool has_spectrum = false;
    float spec_mono = 0.0f;
    int spec_n = 0, spec_map = 0;
    float* d_spec = nullptr;
    std::vector<float> h_spec;  // the knots on the device
    int spec_cap = 0;
    int n_targets = -1;
    float4* d_targets = nullptr;
    int tgt_cap = 0;
    std::vector<float4> h_targets;  // x, y, z, r^2
    std::vector<float> h_radius;
    std::vector<pp_target> h_pods;  // the list as it was given (empty: none staged)
    bool planar = false;  // the list holds rectangles or discs: two records per target
    // uniform grid over the targets, rebuilt when targets or cell size change
    pp::GridDesc grid{};
    float grid_cell_built = -1.0f;  // requested cell size of the built grid
    bool grid_global = false;        // the built grid's tables exceed the LDS: read from memory
    float grid_cell_z_built = 0.0f;
    size_t grid_budget = 0;          // LDS bytes the built grid and a spectrum may take
    float4* d_cells = nullptr;
    uint16_t* d_cell_items = nullptr;
    size_t cell_cap = 0, item_cap = 0;
    int last_search = 0;
    int64_t n_hits = 0, n_ph_sim = 0;
    int64_t work_steps = 0, work_tests = 0, work_cells = 0, work_walks = 0;
    float last_ms = 0.0f;
    int32_t n_launch = 0;
    int block = 256;  // threads per block of the last launch (cfg.block_size, or chosen for 0)
    bool perm_valid = false;
    std::vector<int64_t> perm;
    // pinned host staging of hit records for pp_copy_hits
    HitRecord* h_rec = nullptr;
    int64_t h_rec_cap = 0;
    pp::PinnedPair pin;  // PMT ids and hit columns on their way to pageable host memory
    // device sort of the hits by (source, photon id): the records in that
    // order, keys, indices and the radix sort's scratch, in one allocation
    char* d_sort = nullptr;
    size_t d_sort_cap = 0;
    bool sorted_valid = false;  // d_sort holds the sorted records of the last propagation
    int32_t last_n_sources = 0;
    // one propagation's table: device copy and pinned host staging, laid out
    // counters (uploaded as zeros: one copy clears them and brings the sources) |
    // sources | photon counts | chunk prefix
    char* d_batch = nullptr;
    char* h_batch = nullptr;
    size_t batch_cap = 0;     // bytes of each
    bool table_busy = false;  // a copy of h_batch may still be under way
    // the last batch launch, for the photons that an overflow left untaken
    BatchParams last_batch{};
    uint64_t last_waves = 0, last_items = 0;
    // automatic block size and search kind of the last launch shape
    OccKey occ_key{};
    int occ_block = 0, occ_skind = 0;
    // PMT detection of the context's hits: targets as (x, y, z, radius), and
    // one device block holding the acceptance table | PMT ids
    float4* d_tgt_r = nullptr;
    char* d_pmt = nullptr;
    size_t pmt_cap = 0;
    // hipGraph of the batch mode PP_BATCH_GRAPH: counter clear -> propagation
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    hipGraphNode_t graph_prop = nullptr;
    const void* graph_fn = nullptr;
    const Counters* graph_counters = nullptr;
    unsigned graph_blocks = 0, graph_block = 0;
    size_t graph_lds = 0;
};

namespace {

// Make the context's device current and drop any error state left by an
// earlier, already reported call, so that launch checks see only their own.
int set_dev(pp_ctx* c) {
    PP_HIP(hipSetDevice(c->device));
    (void)hipGetLastError();
    return PP_OK;
}

constexpr int kMaxLdsBytes = 160 * 1024;
// records per pinned staging chunk of pp_copy_hits (64 MB)
constexpr int64_t kStageRecords = (int64_t)1 << 20;
constexpr size_t kGridLdsBudget = 64 * 1024;  // grid tables + targets + spectrum per block
// the largest table set that leaves room for the walk queues of 16 waves
constexpr size_t kGridLdsMax = kMaxLdsBytes - 16 * (size_t)kWaveQueueBytes;
constexpr size_t kGridGlobalBudget = (size_t)64 << 20;  // tables read from device memory

// (Re)build the target grid for the requested cell edge and upload it.
int build_grid(pp_ctx* c, float cell_req, float cell_z_req) {
    std::vector<float> xyz(3 * (size_t)c->n_targets);
    for (int i = 0; i < c->n_targets; ++i) {
        xyz[3 * i] = c->h_targets[i].x;
        xyz[3 * i + 1] = c->h_targets[i].y;
        xyz[3 * i + 2] = c->h_targets[i].z;
    }
    pp::GridTables t;
    // the occupancy-friendly budget first; for many targets (their records
    // alone may fill it) the whole LDS, at fewer workgroups per CU; beyond
    // that, tables in device memory that the search reads through the caches
    auto build = [&](size_t budget) {
        return pp::build_grid_tables(xyz.data(), c->h_radius.data(), c->n_targets, cell_req,
                                     cell_z_req, c->spec_n, budget, t);
    };
    size_t budget = kGridLdsBudget;
    if (!build(budget) && !build(budget = kGridLdsMax)) {
        if (!build(kGridGlobalBudget)) return fail(PP_ERR_INVALID, "grid: no cell size fits");
        budget = 0;
    }
    if (t.cells.size() > c->cell_cap) {
        if (c->d_cells) PP_HIP(hipFree(c->d_cells));
        c->d_cells = nullptr;
        PP_HIP(hipMalloc(&c->d_cells, t.cells.size() * sizeof(float4)));
        c->cell_cap = t.cells.size();
    }
    if (t.items.size() > c->item_cap) {
        if (c->d_cell_items) PP_HIP(hipFree(c->d_cell_items));
        c->d_cell_items = nullptr;
        PP_HIP(hipMalloc(&c->d_cell_items, t.items.size() * 2));
        c->item_cap = t.items.size();
    }
    // uploads are ordered on the context stream, where the kernels that read
    // them run (a blocking-stream copy from pageable memory may still be in
    // flight when it returns); the sync keeps the host tables alive until done
    PP_HIP(hipMemcpyAsync(c->d_cells, t.cells.data(), t.cells.size() * sizeof(float4),
                          hipMemcpyHostToDevice, c->stream));
    PP_HIP(hipMemcpyAsync(c->d_cell_items, t.items.data(), t.items.size() * 2,
                          hipMemcpyHostToDevice, c->stream));
    PP_HIP(hipStreamSynchronize(c->stream));
    c->grid = t.g;
    c->grid_global = budget == 0;
    c->grid_budget = budget;
    c->grid_cell_built = cell_req;
    c->grid_cell_z_built = cell_z_req;
    return PP_OK;
}

// A bound of the scattering length over the spectrum's wavelengths, or infinity.
double longest_scattering(const pp_ctx* c) {
    const pp::Medium& m = c->medium;
    if (m.kind == PP_MEDIUM_SIMPLE) return m.sca_len;
    const auto ends = std::minmax_element(c->h_spec.begin(), c->h_spec.end());
    const double wl[2] = {c->spec_n > 0 ? *ends.first : c->spec_mono,
                          c->spec_n > 0 ? *ends.second : c->spec_mono};
    double longest = 0.0;
    for (double l : wl) {  // monotonic in between
        if (m.kind == PP_MEDIUM_ICE) {
            longest = std::max(longest, m.ice_pref * std::pow(l / 400.0, (double)m.ice_alpha));
        } else {
            if (!(m.kop1 >= 0.0 && m.kop2 >= 0.0 && m.kop3 >= 0.0)) return INFINITY;
            const double x = l / 550.0;
            longest = std::max(longest, m.sca_scale / (m.kop1 * std::pow(x, -4.3) +
                                                       m.kop2 * std::pow(x, -1.7) +
                                                       m.kop3 * std::pow(x, -0.3)));
        }
    }
    return longest;
}

// The box that a segment meets if it hits a target, for the queued scans; false
// where there is no useful one. A direction that has drifted to |dir|^2 = 1 + e
// hits a sphere at a point within sqrt(r^2 + e d^2) of its centre (the reference's
// discriminant keeps the drift), d being at most the longest step: 24 ln 2
// scattering lengths for the smallest uniform number. e is taken as 1e-6 times the
// step and four. It grows by roundings of 2e-7 a step, and a turn about a direction
// of excess e can leave up to 2 e, so that its largest value over many photons lies
// well above the typical one: of 2e6 simulated ones, over 40 steps from unit
// directions or sources within 4e-7, 0.6 of the bound where up to 30% of the
// scattering is isotropic; where all of it is, 7 in 1e7 exceed it, by up to 1.5. Such
// a photon also has to take a step within a fifth of the longest (1 in 5e5) past the
// target's rim to be missed. Sources off by 2e-6 left up to 3 times the bound, so
// they take the plain scan. The margin is far above the rounding of the hit tests
// and of the segment's end.
bool scan_box(const pp_ctx* c, const pp_source* sources, int n_sources, int32_t n_steps,
              pp::GridDesc* g) {
    const double step = 16.64 * 1.01 * longest_scattering(c), e = 1e-6 * ((double)n_steps + 4.0);
    if (!(step < 1e6) || !(e < 1e-3)) return false;
    double size = 0.0, far = 0.0;
    for (int i = 0; i < n_sources; ++i) {
        const pp_source& x = sources[i];
        double d2 = 0.0;
        for (int a = 0; a < 3; ++a) {
            far = std::max(far, (double)std::fabs(x.position[a]));
            d2 += (double)x.direction[a] * x.direction[a];
        }
        if (x.kind != PP_SRC_POINTLIKE_ISOTROPIC && x.kind != PP_SRC_POINTLIKE_TIME_RANGE &&
            !(d2 - 1.0 <= 4e-7 && d2 - 1.0 >= -2e-6))
            return false;
    }
    double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (const pp_target& t : c->h_pods) {
        double r[3] = {0.5 * t.length[0], 0.5 * t.length[1], 0.0};
        if (t.shape_kind != PP_SHAPE_RECTANGLE) r[0] = r[1] = t.radius;
        if (t.shape_kind == PP_SHAPE_SPHERE)
            r[0] = r[1] = r[2] = std::sqrt((double)t.radius * t.radius + e * step * step);
        for (int a = 0; a < 3; ++a) {
            lo[a] = std::min(lo[a], t.position[a] - r[a]);
            hi[a] = std::max(hi[a], t.position[a] + r[a]);
            size = std::max(size, std::max(std::fabs(lo[a]), std::fabs(hi[a])));
        }
    }
    const double m = 0.02 + 1e-4 * size + 1e-5 * far + 1e-6 * step * n_steps;
    g->ox = (float)(lo[0] - m);
    g->oy = (float)(lo[1] - m);
    g->oz = (float)(lo[2] - m);
    g->ex = (float)(hi[0] + m);
    g->ey = (float)(hi[1] + m);
    g->ez = (float)(hi[2] + m);
    return true;
}

// Whether an automatic every-target scan queues its segments. The queues save tests
// and the hit's emission state; the replay of the hits adds 3-6 us to a launch.
// Plain and queued kernel time meet at about 1.5e6 photons x targets: one sphere
// 0.080 / 0.081 ms at 1e6 photons, 0.529 / 0.501 at 1e7; three spheres 0.096 /
// 0.087 at 1e6; eight 0.031 / 0.030 at 1e5; 24 panels, discs and spheres 0.090 /
// 0.049 at 1e5, 2.62 / 0.86 at 1e7.
bool queue_scan(const pp_ctx* c, uint64_t photons) {
    return c->n_targets > 0 && photons > (3u << 19) / (uint64_t)c->n_targets;
}

// Defaults and range checks of a pp_config.
int normalise_config(pp_config& c, const char* who) {
    const std::string w(who);
    // block_size 0: chosen per call from the LDS the launch needs (pp_propagate)
    if (c.block_size != 0 && (c.block_size < 64 || c.block_size > 1024 || c.block_size % 64))
        return fail(PP_ERR_INVALID, w + ": block_size must be 0 or a multiple of 64 in [64,1024]");
    if (c.waves_per_simd < 0 || c.waves_per_simd > 32)
        return fail(PP_ERR_INVALID, w + ": waves_per_simd must be in [0,32]");
    if (c.search < PP_SEARCH_AUTO || c.search > PP_SEARCH_GRID)
        return fail(PP_ERR_INVALID, w + ": unknown search");
    if (!(c.grid_cell >= 0.0f) || !std::isfinite(c.grid_cell))
        return fail(PP_ERR_INVALID, w + ": grid_cell must be finite and >= 0");
    if (!std::isfinite(c.grid_cell_z))
        return fail(PP_ERR_INVALID, w + ": grid_cell_z must be finite");
    if (c.batch_mode < PP_BATCH_AUTO || c.batch_mode > PP_BATCH_GRAPH)
        return fail(PP_ERR_INVALID, w + ": unknown batch_mode");
    if (c.chunk_photons < 0 || c.chunk_photons % 64 || c.chunk_photons > (1 << 24))
        return fail(PP_ERR_INVALID, w + ": chunk_photons must be a multiple of 64 in [0, 2^24]");
    if (c.deterministic_order < 0 || c.deterministic_order > 2)
        return fail(PP_ERR_INVALID, w + ": deterministic_order must be 0, 1 or 2");
    return PP_OK;
}

// Blocks that fill the device: occupancy limit or cfg.waves_per_simd.
int max_resident_blocks(pp_ctx* c, const void* fn, int block, size_t lds, int64_t& out) {
    int occ = 0;
    PP_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, fn, block, lds));
    // LDS is allocated in 512-byte units per workgroup, which the query leaves out
    if (lds > 0) occ = std::min<int>(occ, (int)((size_t)kMaxLdsBytes / ((lds + 511) & ~(size_t)511)));
    if (occ < 1) return fail(PP_ERR_INVALID, "pp_propagate: kernel does not fit one block per CU");
    out = (int64_t)occ * c->n_cu;
    if (c->cfg.waves_per_simd > 0)
        out = std::max<int64_t>(1, (int64_t)c->n_cu * 4 * c->cfg.waves_per_simd * 64 / block);
    return PP_OK;
}

// offset of the sources in the table, after the counters (in the pinned table: the
// staged zeros, then the counters that come back)
constexpr size_t kCounterBytes = 256, kTableSources = 2 * kCounterBytes;
static_assert(sizeof(Counters) <= kCounterBytes, "counters precede the sources");

// The context's table (device) and its pinned staging, grown to at least
// `bytes`, the staged counters zeroed. Waits for the stream where earlier work
// may still read them (a call that failed half way).
int ensure_batch_table(pp_ctx* c, size_t bytes) {
    if (c->table_busy) PP_HIP(hipStreamSynchronize(c->stream));
    c->table_busy = false;
    if (bytes > c->batch_cap) {
        if (c->d_batch) PP_HIP(hipFree(c->d_batch));
        if (c->h_batch) PP_HIP(hipHostFree(c->h_batch));
        c->d_batch = c->h_batch = nullptr;
        c->d_counters = c->h_counters = nullptr;
        c->batch_cap = 0;
        const size_t cap = std::max<size_t>(bytes, 64 * 1024);
        PP_HIP(hipMalloc((void**)&c->d_batch, cap));
        PP_HIP(hipHostMalloc((void**)&c->h_batch, cap, hipHostMallocDefault));
        c->batch_cap = cap;
        c->d_counters = (Counters*)c->d_batch;
        c->h_counters = (Counters*)(c->h_batch + kCounterBytes);
    }
    std::memset(c->h_batch, 0, kCounterBytes);
    return PP_OK;
}

// The staged table to the device
int upload_batch_table(pp_ctx* c, size_t bytes) {
    c->table_busy = true;
    PP_HIP(hipMemcpyAsync(c->d_batch, c->h_batch, bytes, hipMemcpyHostToDevice, c->stream));
    return PP_OK;
}

// Photons of the items that no wave took before every wave had met the overflow
// (taken from the counter: item waves + next_chunk on), a source at a time.
uint64_t photons_not_taken(const pp_ctx* c, const Counters& hc, const std::vector<uint64_t>& nph) {
    const BatchParams& b = c->last_batch;
    const uint64_t k = c->last_waves + hc.next_chunk;
    if (b.dealt || k >= c->last_items) return 0;
    // the first item not taken: chunk ch from its photon off on
    uint64_t ch = k, off = 0;
    if (k >= b.split_from) {
        ch = b.split_from + (k - b.split_from) / b.parts;
        off = (k - b.split_from) % b.parts * b.piece;
    }
    uint64_t n = 0, chunk0 = 0;  // first chunk of the source
    for (const uint64_t m : nph) {
        const uint64_t chunks = (m + b.chunk - 1) / b.chunk;
        const uint64_t first = ch < chunk0 ? 0 : (ch - chunk0) * b.chunk + off;
        if (first < m) n += m - first;
        chunk0 += chunks;
    }
    return n;
}

// The persistent kernel of a search kind and phase: the one whose occupancy
// chooses the automatic block size.
const void* batch_kernel_fn(int skind, int phase) {
    using BatchFn = void (*)(KParams, BatchParams);
#define PP_K(PH, S) propagate_batch_kernel<PH, S, false>
#define PP_K3(S) {PP_K(PP_PHASE_HG, S), PP_K(PP_PHASE_MIXED_HG_ES, S), PP_K(PP_PHASE_MIXED_HG_SL, S)}
    static const BatchFn kKernels[kSearchKinds][3] = {
        PP_K3(kSearchBrute), PP_K3(kSearchGrid), PP_K3(kSearchMixed), PP_K3(kSearchGridGlobal),
        PP_K3(kSearchGridMem), PP_K3(kSearchBruteQueued), PP_K3(kSearchMixedQueued)};
#undef PP_K3
#undef PP_K
    return (const void*)kKernels[skind][phase];
}

// One launch per source, as src/photon_prop_cuda.jl:925-944.
int launch_per_source(pp_ctx* c, KParams& kp, const pp_source* sources,
                      const std::vector<uint64_t>& nph, int skind, int phase, bool count, size_t lds) {
    using KernelFn = void (*)(KParams);
#define PP_K(PH, S, C) propagate_kernel<PH, S, C>
#define PP_K3(S, C) {PP_K(PP_PHASE_HG, S, C), PP_K(PP_PHASE_MIXED_HG_ES, S, C), PP_K(PP_PHASE_MIXED_HG_SL, S, C)}
    // [count][search kind][phase kind]
    static const KernelFn kKernels[2][kSearchKinds][3] = {
        {PP_K3(kSearchBrute, false), PP_K3(kSearchGrid, false), PP_K3(kSearchMixed, false),
         PP_K3(kSearchGridGlobal, false), PP_K3(kSearchGridMem, false),
         PP_K3(kSearchBruteQueued, false), PP_K3(kSearchMixedQueued, false)},
        {PP_K3(kSearchBrute, true), PP_K3(kSearchGrid, true), PP_K3(kSearchMixed, true),
         PP_K3(kSearchGridGlobal, true), PP_K3(kSearchGridMem, true),
         PP_K3(kSearchBruteQueued, true), PP_K3(kSearchMixedQueued, true)}};
#undef PP_K3
#undef PP_K
    const KernelFn kern = kKernels[count][skind][phase];
    const int block = c->block;
    int64_t max_blocks = 0;
    if (int rc = max_resident_blocks(c, (const void*)kern, block, lds, max_blocks)) return rc;
    // the source list on the device (the kernels read their source from it)
    const size_t bytes = kTableSources + nph.size() * sizeof(pp_source);
    if (int rc = ensure_batch_table(c, bytes)) return rc;
    if (!nph.empty()) std::memcpy(c->h_batch + kTableSources, sources, bytes - kTableSources);
    if (int rc = upload_batch_table(c, bytes)) return rc;
    kp.sources = (const pp_source*)(c->d_batch + kTableSources);
    kp.counters = c->d_counters;
    PP_HIP(hipEventRecord(c->ev0, c->stream));
    for (size_t i = 0; i < nph.size(); ++i) {
        if (nph[i] == 0) continue;
        kp.src_ix = (uint32_t)i;
        kp.n_photons = nph[i];
        const int64_t need = (int64_t)((nph[i] + block - 1) / block);
        const int blocks = (int)std::min<int64_t>(need, max_blocks);
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(block), lds, c->stream, kp);
        PP_HIP(hipGetLastError());
        ++c->n_launch;
    }
    return PP_OK;
}

// The whole source list in one persistent launch (propagate_batch_kernel);
// with use_graph, as a hipGraph of counter clear + propagation.
int launch_batch(pp_ctx* c, KParams& kp, const pp_source* sources,
                 const std::vector<uint64_t>& nph, int skind, int phase, bool count, size_t lds,
                 bool use_graph) {
    using BatchFn = void (*)(KParams, BatchParams);
#define PP_K(PH, S, C) propagate_batch_kernel<PH, S, C>
#define PP_K3(S, C) {PP_K(PP_PHASE_HG, S, C), PP_K(PP_PHASE_MIXED_HG_ES, S, C), PP_K(PP_PHASE_MIXED_HG_SL, S, C)}
    static const BatchFn kKernels[2][kSearchKinds][3] = {
        {PP_K3(kSearchBrute, false), PP_K3(kSearchGrid, false), PP_K3(kSearchMixed, false),
         PP_K3(kSearchGridGlobal, false), PP_K3(kSearchGridMem, false),
         PP_K3(kSearchBruteQueued, false), PP_K3(kSearchMixedQueued, false)},
        {PP_K3(kSearchBrute, true), PP_K3(kSearchGrid, true), PP_K3(kSearchMixed, true),
         PP_K3(kSearchGridGlobal, true), PP_K3(kSearchGridMem, true),
         PP_K3(kSearchBruteQueued, true), PP_K3(kSearchMixedQueued, true)}};
#undef PP_K3
#undef PP_K
    const BatchFn kern = kKernels[count][skind][phase];
    const int block = c->block;
    const size_t n = nph.size();
    uint64_t total_ph = 0;
    for (uint64_t v : nph) total_ph += v;
    if (total_ph == 0) {
        // nothing to run; the counters still have to read zero
        if (int rc = ensure_batch_table(c, kTableSources)) return rc;
        if (int rc = upload_batch_table(c, kTableSources)) return rc;
        kp.counters = c->d_counters;
        PP_HIP(hipEventRecord(c->ev0, c->stream));
        return PP_OK;
    }
    int64_t max_blocks = 0;
    if (int rc = max_resident_blocks(c, (const void*)kern, block, lds, max_blocks)) return rc;
    const int64_t waves = max_blocks * (block / 64);
    // Chunks of a small launch are dealt out: wave i takes items i, i + waves, ...
    // and no counter is touched (the device serves its atomics at about one per
    // 12 ns, so that 64-photon chunks from the counter cost more than their
    // photons, and the 256-photon chunks taken before left most waves idle).
    // One item per wave up to 256 photons, then 128-photon items. Large launches
    // take theirs from the counter, since waves progress at rates that differ by
    // a quarter (1e8-photon cascade: 7.6 ms taken, 9.7 ms dealt): about 32
    // chunks per resident wave, at least 384 photons. The line lies where the
    // two meet, at about 768 photons per wave (README point source, then
    // cascade: 3e6 photons 0.209 / 0.329 ms dealt, 0.261 / 0.358 taken; 1e7
    // photons 0.651 / 1.02 and 0.656 / 0.93).
    uint64_t chunk = (uint64_t)c->cfg.chunk_photons;
    const uint64_t per_wave = total_ph / (uint64_t)waves;
    const bool dealt = per_wave < 768;
    if (chunk == 0) {
        if (dealt)
            chunk = per_wave < 256 ? (per_wave / 64 + 1) * 64 : 128;
        else
            chunk = std::min<uint64_t>(std::max<uint64_t>(per_wave / 32 / 64 * 64, 384), 8192);
    }
    // table: counters | sources | photon counts | chunk prefix, each 256-byte aligned
    const size_t off_n = (kTableSources + n * sizeof(pp_source) + 255) & ~(size_t)255;
    const size_t off_p = off_n + ((n * 8 + 255) & ~(size_t)255);
    const size_t bytes = off_p + (n + 1) * 8;
    if (int rc = ensure_batch_table(c, bytes)) return rc;
    char* h = c->h_batch;
    std::memcpy(h + kTableSources, sources, n * sizeof(pp_source));
    uint64_t* hn = (uint64_t*)(h + off_n);
    uint64_t* hp = (uint64_t*)(h + off_p);
    hp[0] = 0;
    for (size_t i = 0; i < n; ++i) {
        hn[i] = nph[i];
        hp[i + 1] = hp[i] + (nph[i] + chunk - 1) / chunk;
    }
    const uint64_t n_chunks = hp[n];
    char* d = c->d_batch;
    kp.counters = c->d_counters;
    BatchParams bp{};
    bp.sources = (const pp_source*)(d + kTableSources);
    bp.n_photons = (const uint64_t*)(d + off_n);
    bp.chunk_prefix = (const uint64_t*)(d + off_p);
    bp.n_sources = (int32_t)n;
    bp.chunk = (uint32_t)chunk;
    // With several sources the chunks' costs differ (a track's photons are
    // not a cascade's), and the last two chunks per resident wave go out in
    // pieces of 256 photons (the 256-source batch: 27.45 -> 27.05 ms). One
    // source keeps whole chunks: its tail is even, and the pieces' extra
    // grabs on the one counter cost more than they save.
    bp.piece = (uint32_t)chunk;
    bp.parts = 1;
    bp.split_from = n_chunks;
    if (n > 1 && !dealt) {
        bp.piece = (uint32_t)std::min<uint64_t>(chunk, 256);
        bp.parts = (uint32_t)((chunk + bp.piece - 1) / bp.piece);
        const uint64_t tail = (uint64_t)waves * 2;
        bp.split_from = n_chunks > tail ? n_chunks - tail : 0;
    }
    const uint64_t n_items = bp.split_from + (n_chunks - bp.split_from) * bp.parts;
    const int64_t want = (int64_t)((n_items + block / 64 - 1) / (block / 64));
    const unsigned blocks = (unsigned)std::min<int64_t>(want, max_blocks);
    bp.n_items = n_items;
    bp.dealt = dealt;
    c->last_batch = bp;
    c->last_waves = (uint64_t)blocks * (block / 64);
    c->last_items = n_items;
    if (int rc = upload_batch_table(c, bytes)) return rc;
    if (!use_graph) {
        PP_HIP(hipEventRecord(c->ev0, c->stream));
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(block), lds, c->stream, kp, bp);
        PP_HIP(hipGetLastError());
        c->n_launch = 1;
        return PP_OK;
    }
    KParams kp_arg = kp;
    void* args[] = {&kp_arg, &bp};
    hipKernelNodeParams np{};
    np.func = (void*)kern;
    np.gridDim = dim3(blocks);
    np.blockDim = dim3(block);
    np.sharedMemBytes = (unsigned)lds;
    np.kernelParams = args;
    np.extra = nullptr;
    // (a table that has grown since moves the counters: the clear node's argument)
    const bool same_shape = c->graph_exec && c->graph_counters == c->d_counters && c->graph_fn == (const void*)kern &&
                            c->graph_blocks == blocks && c->graph_block == (unsigned)block &&
                            c->graph_lds == lds;
    bool updated = false;
    if (same_shape)
        updated = hipGraphExecKernelNodeSetParams(c->graph_exec, c->graph_prop, &np) == hipSuccess;
    if (!updated) {
        (void)hipGetLastError();
        if (c->graph_exec) PP_HIP(hipGraphExecDestroy(c->graph_exec));
        if (c->graph) PP_HIP(hipGraphDestroy(c->graph));
        c->graph_exec = nullptr;
        c->graph = nullptr;
        PP_HIP(hipGraphCreate(&c->graph, 0));
        // the counters are cleared by a kernel node, not a memset node
        Counters* ctr = c->d_counters;
        void* cargs[] = {&ctr};
        hipKernelNodeParams cp{};
        cp.func = (void*)clear_counters_kernel;
        cp.gridDim = dim3(1);
        cp.blockDim = dim3(64);
        cp.sharedMemBytes = 0;
        cp.kernelParams = cargs;
        cp.extra = nullptr;
        hipGraphNode_t clear = nullptr;
        PP_HIP(hipGraphAddKernelNode(&clear, c->graph, nullptr, 0, &cp));
        PP_HIP(hipGraphAddKernelNode(&c->graph_prop, c->graph, &clear, 1, &np));
        PP_HIP(hipGraphInstantiate(&c->graph_exec, c->graph, nullptr, nullptr, 0));
        c->graph_fn = (const void*)kern;
        c->graph_counters = c->d_counters;
        c->graph_blocks = blocks;
        c->graph_block = (unsigned)block;
        c->graph_lds = lds;
    }
    PP_HIP(hipEventRecord(c->ev0, c->stream));
    PP_HIP(hipGraphLaunch(c->graph_exec, c->stream));
    c->n_launch = 1;
    return PP_OK;
}

}  // namespace

extern "C" {

int pp_abi_version(void) { return PP_ABI_VERSION; }

const char* pp_last_error(void) { return g_err.c_str(); }

}  // extern "C"

// used by pp_mlp.hip, the surrogate half of the library
void pp_set_error_message(const char* msg) { g_err = msg; }

extern "C" {

int pp_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int pp_device_memory(int device, int64_t* total_bytes, int64_t* free_bytes) {
    int ndev = pp_device_count();
    if (device < 0 || device >= ndev) return fail(PP_ERR_INVALID, "pp_device_memory: no such device");
    PP_HIP(hipSetDevice(device));
    size_t fr = 0, tot = 0;
    PP_HIP(hipMemGetInfo(&fr, &tot));
    if (total_bytes) *total_bytes = (int64_t)tot;
    if (free_bytes) *free_bytes = (int64_t)fr;
    return PP_OK;
}

int pp_device_info(int device, char* arch, int arch_len, int32_t* n_cu) {
    int ndev = pp_device_count();
    if (device < 0 || device >= ndev) return fail(PP_ERR_INVALID, "pp_device_info: no such device");
    hipDeviceProp_t prop{};
    PP_HIP(hipGetDeviceProperties(&prop, device));
    if (arch && arch_len > 0) {
        std::string a(prop.gcnArchName);
        a = a.substr(0, a.find(':'));
        std::snprintf(arch, (size_t)arch_len, "%s", a.c_str());
    }
    if (n_cu) *n_cu = prop.multiProcessorCount;
    return PP_OK;
}

int64_t pp_hit_record_bytes(void) {
    return (int64_t)sizeof(HitRecord);
}

int pp_create(pp_ctx** out, int device, int64_t hit_capacity, const pp_config* cfg) {
    if (!out) return fail(PP_ERR_INVALID, "pp_create: out is NULL");
    *out = nullptr;
    if (hit_capacity <= 0) return fail(PP_ERR_INVALID, "pp_create: hit_capacity must be > 0");
    int ndev = pp_device_count();
    if (device < 0 || device >= ndev)
        return fail(PP_ERR_INVALID, "pp_create: no HIP device " + std::to_string(device) +
                                        " (" + std::to_string(ndev) + " visible)");
    pp_config c{};
    if (cfg) c = *cfg;
    if (int rc = normalise_config(c, "pp_create")) return rc;
    auto* ctx = new pp_ctx();
    ctx->device = device;
    ctx->cfg = c;
    auto cleanup = [&](int code) {
        pp_destroy(ctx);
        return code;
    };
    if (hipSetDevice(device) != hipSuccess) return cleanup(fail(PP_ERR_HIP, "hipSetDevice failed"));
    if (hipDeviceGetAttribute(&ctx->n_cu, hipDeviceAttributeMultiprocessorCount, device) !=
        hipSuccess)
        return cleanup(fail(PP_ERR_HIP, "hipDeviceGetAttribute failed"));
    if (hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&ctx->ev0) != hipSuccess || hipEventCreate(&ctx->ev1) != hipSuccess)
        return cleanup(fail(PP_ERR_HIP, "stream/event creation failed"));
    const size_t cap = (size_t)hit_capacity;
    const size_t bytes = cap * sizeof(HitRecord);
    if (hipMalloc(&ctx->hit_mem, bytes) != hipSuccess) {
        (void)hipGetLastError();
        return cleanup(fail(PP_ERR_NOMEM, "pp_create: cannot allocate " + std::to_string(bytes) +
                                              " bytes of hit buffer"));
    }
    ctx->hits.rec = (HitRecord*)ctx->hit_mem;
    ctx->hits.capacity = cap;
    *out = ctx;
    return PP_OK;
}

int pp_destroy(pp_ctx* ctx) {
    if (!ctx) return PP_OK;
    (void)hipSetDevice(ctx->device);
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    if (ctx->hit_mem) (void)hipFree(ctx->hit_mem);
    if (ctx->d_spec) (void)hipFree(ctx->d_spec);
    if (ctx->d_targets) (void)hipFree(ctx->d_targets);
    if (ctx->d_cells) (void)hipFree(ctx->d_cells);
    if (ctx->d_cell_items) (void)hipFree(ctx->d_cell_items);
    if (ctx->graph_exec) (void)hipGraphExecDestroy(ctx->graph_exec);
    if (ctx->graph) (void)hipGraphDestroy(ctx->graph);
    if (ctx->d_batch) (void)hipFree(ctx->d_batch);
    if (ctx->h_batch) (void)hipHostFree(ctx->h_batch);
    if (ctx->h_rec) (void)hipHostFree(ctx->h_rec);
    if (ctx->d_sort) (void)hipFree(ctx->d_sort);
    if (ctx->d_tgt_r) (void)hipFree(ctx->d_tgt_r);
    if (ctx->d_pmt) (void)hipFree(ctx->d_pmt);
    ctx->pin.release();
    if (ctx->ev0) (void)hipEventDestroy(ctx->ev0);
    if (ctx->ev1) (void)hipEventDestroy(ctx->ev1);
    if (ctx->stream) (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return PP_OK;
}

int pp_set_medium(pp_ctx* ctx, const pp_medium* m) {
    if (!ctx || !m) return fail(PP_ERR_INVALID, "pp_set_medium: NULL argument");
    if (m->kind != PP_MEDIUM_SIMPLE && m->kind != PP_MEDIUM_CASCADIA && m->kind != PP_MEDIUM_ICE)
        return fail(PP_ERR_INVALID, "pp_set_medium: unknown medium kind");
    if (m->phase_kind != PP_PHASE_HG && m->phase_kind != PP_PHASE_MIXED_HG_ES &&
        m->phase_kind != PP_PHASE_MIXED_HG_SL)
        return fail(PP_ERR_INVALID, "pp_set_medium: unknown phase function kind");
    if (m->phase_kind == PP_PHASE_MIXED_HG_SL && !(m->hg_fraction >= 0.0f && m->hg_fraction <= 1.0f))
        return fail(PP_ERR_INVALID, "pp_set_medium: hg_fraction in [0,1] required");
    if (m->kind == PP_MEDIUM_ICE &&
        !(m->ice_b_dust_400 > 0.0f && std::isfinite(m->ice_alpha_sca_dust) && m->sca_scale > 0.0f))
        return fail(PP_ERR_INVALID, "pp_set_medium: ICE needs b_dust_400 > 0, sca_scale > 0");
    if (!(m->hg_g > 0.0f && m->hg_g < 1.0f))
        return fail(PP_ERR_INVALID, "pp_set_medium: hg_g must be in (0,1)");
    if (m->phase_kind == PP_PHASE_MIXED_HG_ES &&
        !(m->es_b > 0.0f && m->hg_fraction >= 0.0f && m->hg_fraction <= 1.0f))
        return fail(PP_ERR_INVALID, "pp_set_medium: es_b > 0 and hg_fraction in [0,1] required");
    if (m->kind == PP_MEDIUM_SIMPLE &&
        !(m->sca_len > 0.0f && m->group_velocity > 0.0f && m->phase_refractive_index >= 1.0f))
        return fail(PP_ERR_INVALID, "pp_set_medium: SIMPLE needs sca_len>0, group_velocity>0, n>=1");
    if (m->kind == PP_MEDIUM_CASCADIA && !(m->sca_scale > 0.0f))
        return fail(PP_ERR_INVALID, "pp_set_medium: sca_scale must be > 0");
    ctx->medium_in = *m;
    ctx->medium = lower_medium(*m);
    ctx->has_medium = true;
    return PP_OK;
}

int pp_set_spectrum(pp_ctx* ctx, float mono_wl, const float* table, int n, int mapping) {
    if (!ctx) return fail(PP_ERR_INVALID, "pp_set_spectrum: NULL ctx");
    if (int rc = set_dev(ctx)) return rc;
    if (!table) {
        if (!(mono_wl > 0.0f) || !std::isfinite(mono_wl))
            return fail(PP_ERR_INVALID, "pp_set_spectrum: monochromatic wavelength must be > 0");
        ctx->spec_mono = mono_wl;
        ctx->spec_n = 0;
        ctx->has_spectrum = true;
        return PP_OK;
    }
    if (n < 2 || n > 8192) return fail(PP_ERR_INVALID, "pp_set_spectrum: n must be in [2, 8192]");
    if (mapping != PP_SPEC_KNOTS && mapping != PP_SPEC_TEXTURE)
        return fail(PP_ERR_INVALID, "pp_set_spectrum: unknown mapping");
    for (int i = 0; i < n; ++i)
        if (!std::isfinite(table[i]) || table[i] <= 0.0f)
            return fail(PP_ERR_INVALID, "pp_set_spectrum: knots must be finite and > 0");
    // the table that is staged already: the device copy stands
    if (ctx->h_spec.size() == (size_t)n &&
        std::memcmp(ctx->h_spec.data(), table, (size_t)n * sizeof(float)) == 0) {
        ctx->spec_n = n;
        ctx->spec_map = mapping;
        ctx->has_spectrum = true;
        return PP_OK;
    }
    ctx->h_spec.clear();
    if (n > ctx->spec_cap) {
        if (ctx->d_spec) PP_HIP(hipFree(ctx->d_spec));
        ctx->d_spec = nullptr;
        ctx->spec_cap = 0;
        PP_HIP(hipMalloc(&ctx->d_spec, (size_t)n * sizeof(float)));
        ctx->spec_cap = n;
    }
    PP_HIP(hipMemcpyAsync(ctx->d_spec, table, (size_t)n * sizeof(float), hipMemcpyHostToDevice,
                          ctx->stream));
    PP_HIP(hipStreamSynchronize(ctx->stream));
    ctx->h_spec.assign(table, table + n);
    ctx->spec_n = n;
    ctx->spec_map = mapping;
    ctx->has_spectrum = true;
    return PP_OK;
}

int pp_set_targets(pp_ctx* ctx, const pp_target* t, int n) {
    if (!ctx) return fail(PP_ERR_INVALID, "pp_set_targets: NULL ctx");
    if (n < 0 || (n > 0 && !t)) return fail(PP_ERR_INVALID, "pp_set_targets: bad target list");
    bool planar = false;
    for (int i = 0; i < n; ++i) {
        const pp_target& x = t[i];
        auto bad = [&](const char* what) {
            return fail(PP_ERR_INVALID, "pp_set_targets: target " + std::to_string(i) + what);
        };
        if (!finite3(x.position)) return bad(" has a non-finite position");
        if (x.shape_kind == PP_SHAPE_SPHERE || x.shape_kind == PP_SHAPE_DISC) {
            if (!(x.radius > 0.0f) || !std::isfinite(x.radius))
                return bad(" needs a finite radius > 0");
        } else if (x.shape_kind == PP_SHAPE_RECTANGLE) {
            if (!(x.length[0] > 0.0f) || !(x.length[1] > 0.0f) || !std::isfinite(x.length[0]) ||
                !std::isfinite(x.length[1]))
                return bad(" needs finite side lengths > 0");
        } else {
            return bad(" has an unknown shape_kind");
        }
        planar |= x.shape_kind != PP_SHAPE_SPHERE;
    }
    // records per target: (x, y, z, r^2), plus (kind bits, lx/2, ly/2, 0) in a
    // list with planar targets
    const int per = planar ? 2 : 1;
    // planar lists are scanned from LDS; sphere lists of any length up to
    // kMaxTargets are searched by the grid, from device memory if need be
    if (planar && (size_t)n * per * sizeof(float4) + 8192 * sizeof(float) > (size_t)kMaxLdsBytes)
        return fail(PP_ERR_INVALID, "pp_set_targets: too many planar targets for LDS staging");
    if (n > kMaxTargets) return fail(PP_ERR_INVALID, "pp_set_targets: more than 65535 targets");
    if (int rc = set_dev(ctx)) return rc;
    // the list that is staged already, value for value (a driver stages its
    // detector for every event): the device copies and the grid stand. (Upload
    // and grid of 16000 targets: 79 ms a call before, 5 ms for a new list now.)
    if (ctx->n_targets == n && ctx->h_pods.size() == (size_t)n &&
        (n == 0 || std::memcmp(ctx->h_pods.data(), t, (size_t)n * sizeof(pp_target)) == 0))
        return PP_OK;
    ctx->h_pods.clear();
    std::vector<float4> h((size_t)std::max(n * per, 1));
    for (int i = 0; i < n; ++i) {
        const pp_target& x = t[i];
        // r^2 and the half lengths are Float32 values, as target_shape.radius^2
        // and length_x/2 of the reference
        const float w = x.shape_kind == PP_SHAPE_RECTANGLE ? 0.0f : x.radius * x.radius;
        h[(size_t)i * per] = make_float4(x.position[0], x.position[1], x.position[2], w);
        if (planar) {
            uint32_t kind = (uint32_t)x.shape_kind;
            float kf;
            std::memcpy(&kf, &kind, 4);
            h[(size_t)i * per + 1] = x.shape_kind == PP_SHAPE_RECTANGLE
                                         ? make_float4(kf, x.length[0] / 2.0f, x.length[1] / 2.0f, 0.0f)
                                         : make_float4(kf, x.radius, x.radius, 0.0f);
        }
    }
    // (x, y, z, radius) per target for the PMT detection of hits
    std::vector<float4> hr((size_t)std::max(n, 1));
    for (int i = 0; i < n; ++i)
        hr[(size_t)i] = make_float4(t[i].position[0], t[i].position[1], t[i].position[2],
                                    t[i].radius);
    if (n * per > ctx->tgt_cap) {
        if (ctx->d_targets) PP_HIP(hipFree(ctx->d_targets));
        if (ctx->d_tgt_r) PP_HIP(hipFree(ctx->d_tgt_r));
        ctx->d_targets = ctx->d_tgt_r = nullptr;
        ctx->tgt_cap = 0;
        PP_HIP(hipMalloc(&ctx->d_targets, (size_t)n * per * sizeof(float4)));
        PP_HIP(hipMalloc(&ctx->d_tgt_r, (size_t)n * per * sizeof(float4)));
        ctx->tgt_cap = n * per;
    }
    if (n > 0) {
        PP_HIP(hipMemcpyAsync(ctx->d_targets, h.data(), (size_t)n * per * sizeof(float4),
                              hipMemcpyHostToDevice, ctx->stream));
        PP_HIP(hipMemcpyAsync(ctx->d_tgt_r, hr.data(), (size_t)n * sizeof(float4),
                              hipMemcpyHostToDevice, ctx->stream));
    }
    PP_HIP(hipStreamSynchronize(ctx->stream));
    ctx->n_targets = n;
    ctx->planar = planar;
    ctx->h_targets.resize((size_t)n);
    ctx->h_radius.resize((size_t)n);
    for (int i = 0; i < n; ++i) {
        ctx->h_targets[(size_t)i] = h[(size_t)i * per];
        ctx->h_radius[(size_t)i] = t[i].radius;
    }
    ctx->grid_cell_built = -1.0f;  // grid is rebuilt on the next propagation
    ctx->h_pods.assign(t, t + n);
    return PP_OK;
}

int pp_propagate(pp_ctx* ctx, const pp_source* sources, int n_sources, uint64_t seed,
                 int32_t n_steps, float photon_scaling, int64_t* n_hits_out,
                 int64_t* n_ph_sim_out) {
    if (!ctx) return fail(PP_ERR_INVALID, "pp_propagate: NULL ctx");
    if (n_sources < 0 || (n_sources > 0 && !sources))
        return fail(PP_ERR_INVALID, "pp_propagate: bad source list");
    if (!ctx->has_medium || !ctx->has_spectrum || ctx->n_targets < 0)
        return fail(PP_ERR_STATE, "pp_propagate: set medium, spectrum and targets first");
    if (ctx->n_targets > kMaxTargets)
        return fail(PP_ERR_INVALID, "pp_propagate: more than 65535 targets");
    if (n_steps < 0 || n_steps > PP_MAX_STEPS)
        return fail(PP_ERR_INVALID, "pp_propagate: n_steps out of range");
    if (!(photon_scaling >= 0.0f) || !std::isfinite(photon_scaling))
        return fail(PP_ERR_INVALID, "pp_propagate: photon_scaling must be finite and >= 0");
    for (int i = 0; i < n_sources; ++i) {
        const pp_source& s = sources[i];
        if (s.kind < 0 || s.kind >= PP_SRC_KIND_COUNT)
            return fail(PP_ERR_INVALID, "pp_propagate: source " + std::to_string(i) +
                                            " has an unknown kind");
        if (s.photons < 0)
            return fail(PP_ERR_INVALID, "pp_propagate: negative photon count");
        if (!finite3(s.position) || !finite3(s.direction))
            return fail(PP_ERR_INVALID, "pp_propagate: non-finite source position/direction");
        const bool cascade = s.kind == PP_SRC_EXTENDED_CHERENKOV ||
                             s.kind == PP_SRC_EXTENDED_CHERENKOV_NO_SMEAR ||
                             s.kind == PP_SRC_EXTENDED_CHERENKOV_CUSTOM_SMEAR;
        if (cascade && !(s.long_a > 0.0f && s.long_b > 0.0f && s.long_lrad > 0.0f))
            return fail(PP_ERR_INVALID, "pp_propagate: cascade needs long_a, long_b, lrad > 0");
        if (s.kind == PP_SRC_EXTENDED_CHERENKOV_CUSTOM_SMEAR &&
            !(s.beta_a > 0.0f && s.beta_b > 0.0f))
            return fail(PP_ERR_INVALID, "pp_propagate: custom smear needs beta_a, beta_b > 0");
    }
    if (int rc = set_dev(ctx)) return rc;

    // search: grid for more than a handful of targets unless asked otherwise
    int search = ctx->cfg.search;
    if (ctx->planar && search == PP_SEARCH_GRID)
        return fail(PP_ERR_INVALID,
                    "pp_propagate: the grid search takes spherical targets only (the list holds "
                    "rectangles or discs)");
    const bool automatic = search == PP_SEARCH_AUTO;
    if (automatic)
        search = ctx->n_targets > 8 && !ctx->planar ? PP_SEARCH_GRID : PP_SEARCH_BRUTE;
    if (ctx->n_targets == 0) search = PP_SEARCH_BRUTE;
    if (search == PP_SEARCH_GRID && n_steps > kDeferredMaxSteps) {
        if (!automatic)
            return fail(PP_ERR_INVALID, "pp_propagate: the grid search takes at most 2^26 - 1 steps");
        search = PP_SEARCH_BRUTE;
    }
    if (search == PP_SEARCH_GRID) {
        const float want = ctx->cfg.grid_cell, want_z = ctx->cfg.grid_cell_z;
        // a grid in the LDS stands as long as the spectrum fits beside it, one in memory
        // for any (built again for every other length, a call on 3000 targets between
        // two spectra took 602 us, on 7680 targets 1444; like this 225 and 300)
        const bool full = !ctx->grid_global &&
                          lds_bytes(ctx->n_targets, ctx->grid.n_cells, ctx->grid.n_items,
                                    ctx->spec_n, true) > ctx->grid_budget;
        if (ctx->grid_cell_built != want || ctx->grid_cell_z_built != want_z ||
            ctx->grid_cell_built < -0.5f || full) {
            if (int rc = build_grid(ctx, want, want_z)) {
                if (!automatic) return rc;
                search = PP_SEARCH_BRUTE;  // no grid fits: the every-target scan
            }
        }
    }
    // photon count of src/photon_prop_cuda.jl:456 (Float32 product)
    std::vector<uint64_t> nph((size_t)n_sources);
    uint64_t n_sim = 0;
    for (int i = 0; i < n_sources; ++i) {
        // the limit is checked on the float product, before it is converted
        const float prod = std::floor((float)sources[i].photons * photon_scaling);
        if (!(prod < (float)kMaxPhotonsPerSource))
            return fail(PP_ERR_INVALID, "pp_propagate: source " + std::to_string(i) +
                                            " has 2^40 or more photons after scaling");
        nph[(size_t)i] = prod > 0.0f ? (uint64_t)prod : 0;
        n_sim += nph[(size_t)i];
    }
    const bool grid = search == PP_SEARCH_GRID;
    const bool global = grid && ctx->grid_global;
    int skind = global ? kSearchGridGlobal
                : grid ? kSearchGrid : ctx->planar ? kSearchMixed : kSearchBrute;
    const int phase = ctx->medium.phase.kind;
    // LDS tables of a search: the global grid stages only the spectrum
    auto table_bytes = [&](int kind) {
        if (kind == kSearchGridGlobal) return std::max<size_t>((size_t)ctx->spec_n * 4, 16);
        const int n = kind == kSearchGridMem ? 0 : ctx->planar ? 2 * ctx->n_targets : ctx->n_targets;
        return lds_bytes(n, grid ? ctx->grid.n_cells : 0, grid ? ctx->grid.n_items : 0, ctx->spec_n,
                         grid);
    };
    // the walk queues of the waves that search in batches follow the tables
    auto with_queues = [&](int kind, int threads) {
        const size_t tables = table_bytes(kind);
        return deferred_kind(kind)
                   ? ((tables + 15) & ~(size_t)15) + (size_t)(threads / 64) * wave_queue_bytes(kind)
                   : tables;
    };
    pp::GridDesc box{};
    if (automatic && !grid && n_steps <= kDeferredMaxSteps && queue_scan(ctx, n_sim) &&
        scan_box(ctx, sources, n_sources, n_steps, &box)) {
        const int kind = ctx->planar ? kSearchMixedQueued : kSearchBruteQueued;
        if (with_queues(kind, ctx->cfg.block_size ? ctx->cfg.block_size : 256) <= (size_t)kMaxLdsBytes)
            skind = kind;
    }
    // block size: the set one or, for 0, the one of 256, 384, 512, 768 and 1024
    // threads with the most waves resident per CU: the runtime's occupancy
    // query (registers: 6 or 7 waves per SIMD) and the LDS a workgroup needs (the
    // tables once and, with a grid, a walk queue per wave) in 512-byte
    // allocation units, which the query does not apply (it reports three
    // workgroups of 54320 bytes, and they run as two); the smallest on a tie.
    // A grid search leaves its targets in memory where that makes room for more
    // waves: 1000 targets, 16 KB, leave 24 waves in 768-thread blocks (27.0 ms
    // for the 256-source batch) and 28 in 256-thread blocks without them (25.8
    // ms); 320 targets leave 28 either way, and are read from LDS (1e8-photon
    // cascade: 7.07 ms, from memory 7.27). With a set block size the placement
    // follows the same rule (another 256-source batch at a set 256: 17.0 ms, with
    // the targets held in LDS 20.4; automatic 17.0).
    int block = ctx->cfg.block_size;
    if (block == 0 || skind == kSearchGrid) {
        const OccKey key{batch_kernel_fn(skind, phase), table_bytes(skind),
                         table_bytes(kSearchGridMem), block};
        if (!(key == ctx->occ_key)) {
            int best_waves = 0;
            ctx->occ_block = block ? block : 64;  // the LDS check below reports what does not fit
            ctx->occ_skind = skind;
            for (int kind : {skind, (int)kSearchGridMem}) {
                if (kind != skind && (skind != kSearchGrid || best_waves == 0)) continue;
                const void* fn = batch_kernel_fn(kind, phase);
                for (int b : block ? std::vector<int>{block} : std::vector<int>{256, 384, 512, 768, 1024}) {
                    const size_t need = with_queues(kind, b);
                    if (need > (size_t)kMaxLdsBytes) continue;
                    int occ = 0;
                    PP_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, fn, b, need));
                    const size_t alloc = (need + 511) & ~(size_t)511;
                    occ = std::min<int>(occ, (int)((size_t)kMaxLdsBytes / alloc));
                    if (occ * (b / 64) > best_waves) {
                        best_waves = occ * (b / 64);
                        ctx->occ_block = b;
                        ctx->occ_skind = kind;
                    }
                }
            }
            ctx->occ_key = key;
        }
        block = ctx->occ_block;
        skind = ctx->occ_skind;
    }
    const size_t tables = table_bytes(skind);
    const uint32_t queue_off = (uint32_t)((tables + 15) & ~(size_t)15);
    const size_t lds = with_queues(skind, block);
    ctx->block = block;
    if (lds > (size_t)kMaxLdsBytes)
        return fail(PP_ERR_INVALID, "pp_propagate: targets, tables and walk queues exceed the LDS "
                                    "of a workgroup (a smaller block_size may fit)");
    const bool count = ctx->cfg.count_work != 0;
    ctx->last_search = search;
    KParams kp{};
    kp.med = ctx->medium;
    kp.k0 = (uint32_t)seed;
    kp.k1 = (uint32_t)(seed >> 32);
    kp.n_steps = n_steps;
    kp.queue_off = queue_off;
    kp.targets = ctx->d_targets;
    kp.n_targets = ctx->n_targets;
    if (grid) {
        kp.grid = ctx->grid;
        kp.cells = ctx->d_cells;
        kp.cell_items = ctx->d_cell_items;
    } else if (deferred_kind(skind)) {
        kp.grid = box;
    }
    kp.spec_n = ctx->spec_n;
    kp.spec_map = ctx->spec_map;
    kp.spec_mono = ctx->spec_mono;
    kp.spec_nf = (float)ctx->spec_n;
    kp.spec_lastf = (float)(ctx->spec_n - 1);
    kp.spec = ctx->d_spec;
    kp.hits = ctx->hits;
    ctx->n_launch = 0;
    ctx->last_items = 0;
    const int mode = ctx->cfg.batch_mode == PP_BATCH_AUTO ? PP_BATCH_PERSISTENT : ctx->cfg.batch_mode;
    if (mode == PP_BATCH_PER_SOURCE) {
        if (int rc = launch_per_source(ctx, kp, sources, nph, skind, phase, count, lds)) return rc;
    } else {
        if (int rc = launch_batch(ctx, kp, sources, nph, skind, phase, count, lds, mode == PP_BATCH_GRAPH))
            return rc;
    }
    // the kernels that search in batches leave their hit records to be completed
    if (deferred_kind(skind)) {
        hipLaunchKernelGGL(replay_hits_kernel, dim3((unsigned)(4 * ctx->n_cu)), dim3(256), 0,
                           ctx->stream, kp, (const pp_source*)(ctx->d_batch + kTableSources),
                           ctx->h_counters, ctx->planar);
    } else {
        hipLaunchKernelGGL(publish_counters_kernel, dim3(1), dim3(64), 0, ctx->stream, kp.counters,
                           ctx->h_counters);
    }
    PP_HIP(hipGetLastError());
    PP_HIP(hipEventRecord(ctx->ev1, ctx->stream));
    PP_HIP(hipStreamSynchronize(ctx->stream));
    ctx->table_busy = false;
    const Counters hc = *ctx->h_counters;
    PP_HIP(hipEventElapsedTime(&ctx->last_ms, ctx->ev0, ctx->ev1));
    ctx->n_hits = (int64_t)std::min<unsigned long long>(hc.n_hits, ctx->hits.capacity);
    ctx->n_ph_sim = (int64_t)(n_sim - hc.n_lost - (hc.err ? photons_not_taken(ctx, hc, nph) : 0));
    ctx->work_steps = (int64_t)hc.steps;
    ctx->work_tests = (int64_t)hc.tests;
    ctx->work_cells = (int64_t)hc.cells;
    ctx->work_walks = (int64_t)hc.walks;
    ctx->perm_valid = false;
    ctx->sorted_valid = false;
    ctx->last_n_sources = n_sources;
    if (n_hits_out) *n_hits_out = ctx->n_hits;
    if (n_ph_sim_out) *n_ph_sim_out = ctx->n_ph_sim;
    if (hc.err) return fail(PP_ERR_HIT_OVERFLOW, "hit buffer overflow (PhotonPropOOMException)");
    return PP_OK;
}

int pp_get_config(pp_ctx* ctx, pp_config* cfg) {
    if (!ctx || !cfg) return fail(PP_ERR_INVALID, "pp_get_config: NULL argument");
    *cfg = ctx->cfg;
    return PP_OK;
}

int pp_set_config(pp_ctx* ctx, const pp_config* cfg) {
    if (!ctx || !cfg) return fail(PP_ERR_INVALID, "pp_set_config: NULL argument");
    pp_config c = *cfg;
    if (int rc = normalise_config(c, "pp_set_config")) return rc;
    ctx->cfg = c;
    return PP_OK;
}

int pp_autotune(pp_ctx* ctx, const pp_source* sources, int n_sources, uint64_t seed,
                int32_t n_steps, float photon_scaling, int64_t sample_photons, pp_config* best,
                float* best_ms) {
    if (!ctx) return fail(PP_ERR_INVALID, "pp_autotune: NULL ctx");
    if (n_sources <= 0 || !sources) return fail(PP_ERR_INVALID, "pp_autotune: no sources");
    if (sample_photons <= 0) return fail(PP_ERR_INVALID, "pp_autotune: sample_photons must be > 0");
    if (!(photon_scaling > 0.0f) || !std::isfinite(photon_scaling))
        return fail(PP_ERR_INVALID, "pp_autotune: photon_scaling must be finite and > 0");
    double total = 0.0;
    for (int i = 0; i < n_sources; ++i) total += (double)sources[i].photons * photon_scaling;
    if (!(total > 0.0)) return fail(PP_ERR_INVALID, "pp_autotune: the sources hold no photons");
    const float scale = (float)std::min<double>(photon_scaling,
                                                photon_scaling * (double)sample_photons / total);
    const pp_config saved = ctx->cfg;
    pp_config cur = saved;
    if (cur.batch_mode == PP_BATCH_AUTO) cur.batch_mode = PP_BATCH_PERSISTENT;
    cur.count_work = 0;
    cur.waves_per_simd = 0;
    auto run = [&](const pp_config& c, float& ms) -> int {
        ctx->cfg = c;
        float t = INFINITY;
        for (int r = 0; r < 3; ++r) {
            int64_t nh = 0, ns = 0;
            const int rc = pp_propagate(ctx, sources, n_sources, seed, n_steps, scale, &nh, &ns);
            if (rc != PP_OK) return rc;
            if (r > 0) t = std::min(t, ctx->last_ms);
        }
        ms = t;
        return PP_OK;
    };
    float t_best = 0.0f;
    if (int rc = run(cur, t_best)) {
        ctx->cfg = saved;
        return rc;
    }
    // automatic grid edge of these targets, for the cell candidates
    const bool grid = ctx->last_search == PP_SEARCH_GRID;
    const float h_auto = grid ? ctx->grid.h : 0.0f;
    std::vector<float> cells = {0.0f};
    if (grid)
        for (float f : {0.6f, 0.8f, 0.9f, 1.1f, 1.25f}) cells.push_back(f * h_auto);
    const int blocks[] = {64, 128, 256, 384, 512, 768, 1024};
    const int chunks[] = {0, 64, 128, 256, 512, 1024};
    // cell shapes: cubic, columns, and cells twice as tall as wide (set when tried)
    float shapes[] = {0.0f, -1.0f, 0.0f};
    for (int pass = 0; pass < 2; ++pass) {
        for (int knob = 0; knob < 4; ++knob) {
            if (knob >= 2 && !grid) continue;
            const size_t n_cand = knob == 0 ? 7 : knob == 1 ? 6 : knob == 2 ? cells.size() : 3;
            if (knob == 3) shapes[2] = 2.0f * (cur.grid_cell > 0.0f ? cur.grid_cell : h_auto);
            for (size_t k = 0; k < n_cand; ++k) {
                pp_config c = cur;
                if (knob == 0) c.block_size = blocks[k];
                if (knob == 1) c.chunk_photons = chunks[k];
                if (knob == 2) c.grid_cell = cells[k];
                if (knob == 3) c.grid_cell_z = shapes[k];
                if (c.block_size == cur.block_size && c.chunk_photons == cur.chunk_photons &&
                    c.grid_cell == cur.grid_cell && c.grid_cell_z == cur.grid_cell_z)
                    continue;
                if (c.batch_mode == PP_BATCH_PER_SOURCE && knob == 1) continue;
                float t = 0.0f;
                const int rc = run(c, t);
                if (rc == PP_ERR_HIT_OVERFLOW || rc == PP_ERR_INVALID) continue;  // e.g. LDS budget
                if (rc != PP_OK) {
                    ctx->cfg = saved;
                    return rc;
                }
                if (t < t_best) {
                    t_best = t;
                    cur = c;
                }
            }
        }
    }
    cur.count_work = saved.count_work;
    cur.deterministic_order = saved.deterministic_order;
    ctx->cfg = cur;
    ctx->n_hits = 0;  // the tuning runs' hits are not results
    ctx->n_ph_sim = 0;
    ctx->perm_valid = false;
    ctx->sorted_valid = false;
    if (best) *best = cur;
    if (best_ms) *best_ms = t_best;
    return PP_OK;
}

int pp_last_timing(pp_ctx* ctx, float* kernel_ms, int32_t* n_launches) {
    if (!ctx) return fail(PP_ERR_INVALID, "pp_last_timing: NULL ctx");
    if (kernel_ms) *kernel_ms = ctx->last_ms;
    if (n_launches) *n_launches = ctx->n_launch;
    return PP_OK;
}

void* pp_stream(pp_ctx* ctx) { return ctx ? (void*)ctx->stream : nullptr; }

int pp_work_counts(pp_ctx* ctx, int64_t* steps, int64_t* sphere_tests, int64_t* cell_visits,
                   int64_t* grid_walks) {
    if (!ctx) return fail(PP_ERR_INVALID, "pp_work_counts: NULL ctx");
    if (!ctx->cfg.count_work)
        return fail(PP_ERR_STATE, "pp_work_counts: context created without count_work");
    if (steps) *steps = ctx->work_steps;
    if (sphere_tests) *sphere_tests = ctx->work_tests;
    if (cell_visits) *cell_visits = ctx->work_cells;
    if (grid_walks) *grid_walks = ctx->work_walks;
    return PP_OK;
}

int pp_search_info(pp_ctx* ctx, int32_t* search, float* cell, int32_t* dims, int32_t* n_items) {
    if (!ctx) return fail(PP_ERR_INVALID, "pp_search_info: NULL ctx");
    if (search) *search = ctx->last_search;
    const bool g = ctx->last_search == PP_SEARCH_GRID && ctx->grid_cell_built > -0.5f;
    if (cell) *cell = g ? ctx->grid.h : 0.0f;
    if (dims) {
        dims[0] = g ? ctx->grid.nx : 0;
        dims[1] = g ? ctx->grid.ny : 0;
        dims[2] = g ? ctx->grid.nz : 0;
    }
    if (n_items) *n_items = g ? ctx->grid.n_items : 0;
    return PP_OK;
}

// Sort key of hit k: the source index above the 40 photon-id bits, so that an
// ascending sort orders by source, then by photon id; the value is k.
__global__ void hit_keys_kernel(const HitRecord* __restrict__ rec, int64_t n,
                                uint64_t* __restrict__ key, uint32_t* __restrict__ idx) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    key[k] = ((uint64_t)(uint32_t)rec[k].source_ix << kPidBits) |
             (rec[k].id & (kMaxPhotonsPerSource - 1));
    idx[k] = (uint32_t)k;
}

// out[k] = rec[idx[k]], 64 bytes per lane as four 16-byte loads and stores.
__global__ void gather_hits_kernel(const HitRecord* __restrict__ rec,
                                   const uint32_t* __restrict__ idx, int64_t n,
                                   HitRecord* __restrict__ out) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const uint4* src = (const uint4*)(rec + idx[k]);
    uint4* dst = (uint4*)(out + k);
    const uint4 a = src[0], b = src[1], c = src[2], d = src[3];
    dst[0] = a;
    dst[1] = b;
    dst[2] = c;
    dst[3] = d;
}

// The order of up to kRankMost hits in one launch: the rank of a hit is the
// number of keys below its own (keys are unique), and its record goes straight to
// that place, in device memory and, where `host` is set, in pinned host memory
// too (the copy of a small hit table). 64 hits per workgroup, the keys in tiles
// of LDS, a quarter of each tile per wave. For a few thousand hits the radix sort
// is five launches of a few workgroups and the copy a sixth: 25-45 us of a call
// for the README example's 14 hits or a small shower's 1200; 2.5 and 13 us here. The
// compares grow with the square of the count, and at 4096 the two are near.
constexpr int kRankMost = 4096;

__global__ void __launch_bounds__(256) rank_hits_kernel(const HitRecord* __restrict__ rec, int n,
                                                        HitRecord* __restrict__ out,
                                                        HitRecord* __restrict__ host) {
    __shared__ uint64_t key[1024];
    __shared__ uint32_t part[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int k = blockIdx.x * 64 + lane;
    auto key_of = [&](int i) {
        return ((uint64_t)(uint32_t)rec[i].source_ix << kPidBits) |
               (rec[i].id & (kMaxPhotonsPerSource - 1));
    };
    const uint64_t own = k < n ? key_of(k) : 0;
    uint32_t below = 0;
    for (int t0 = 0; t0 < n; t0 += 1024) {
        for (int i = threadIdx.x; i < 1024; i += 256)
            key[i] = t0 + i < n ? key_of(t0 + i) : ~0ull;
        __syncthreads();
        const int most = n - t0 < 1024 ? n - t0 : 1024;
        const int i1 = min((w + 1) * 256, most);
#pragma unroll 8
        for (int i = w * 256; i < i1; ++i) below += key[i] < own ? 1u : 0u;
        __syncthreads();
    }
    part[w][lane] = below;
    __syncthreads();
    if (k >= n) return;
    const uint32_t rank = part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
    const uint4 v = reinterpret_cast<const uint4*>(rec + k)[w];  // a quarter of the record each
    reinterpret_cast<uint4*>(out + rank)[w] = v;
    if (host) reinterpret_cast<uint4*>(host + rank)[w] = v;
}

static size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

// The hits in (source, photon id) order, written by the device to the front
// of ctx->d_sort: a radix sort over 40 + bits(n_sources - 1) key bits carries
// the record indices (the sort is stable; a photon hits at most once, so keys
// are unique), then a gather writes the records in that order.  Sets
// *done = false and does nothing when the keys do not fit 64 bits, the
// indices 32 bits or the buffer device memory; the caller then sorts on the
// host. Up to kRankMost hits are ordered by rank_hits_kernel, to `host` too.
static int sort_hits_device(pp_ctx* ctx, bool* done, HitRecord* host = nullptr) {
    *done = false;
    const int64_t n = ctx->n_hits;
    const int32_t ns = ctx->last_n_sources;
    if (n <= 0 || n > INT32_MAX || ns <= 0 || ns > (1 << 24)) return PP_OK;
    auto grow = [&](size_t need) {
        if (need <= ctx->d_sort_cap) return true;
        if (ctx->d_sort) (void)hipFree(ctx->d_sort);
        ctx->d_sort = nullptr;
        ctx->d_sort_cap = 0;
        if (hipMalloc((void**)&ctx->d_sort, need) != hipSuccess) {
            (void)hipGetLastError();  // out of device memory: sort on the host
            ctx->d_sort = nullptr;
            return false;
        }
        ctx->d_sort_cap = need;
        return true;
    };
    if (n <= kRankMost) {
        if (!grow(align256((size_t)kRankMost * sizeof(HitRecord)))) return PP_OK;
        hipLaunchKernelGGL(rank_hits_kernel, dim3((unsigned)((n + 63) / 64)), dim3(256), 0,
                           ctx->stream, ctx->hits.rec, (int)n, (HitRecord*)ctx->d_sort, host);
        PP_HIP(hipGetLastError());
        *done = true;
        return PP_OK;
    }
    int end_bit = (int)kPidBits;
    for (uint32_t v = (uint32_t)(ns - 1); v; v >>= 1) ++end_bit;
    size_t temp = 0;
    PP_HIP(rocprim::radix_sort_pairs(nullptr, temp, (const uint64_t*)nullptr, (uint64_t*)nullptr,
                                     (const uint32_t*)nullptr, (uint32_t*)nullptr, (uint32_t)n, 0u,
                                     (unsigned)end_bit, ctx->stream));
    const size_t br = align256((size_t)n * sizeof(HitRecord));
    const size_t bk = align256((size_t)n * 8), bv = align256((size_t)n * 4);
    const size_t need = br + 2 * bk + 2 * bv + align256(temp);
    if (!grow(need)) return PP_OK;
    char* base = ctx->d_sort + br;
    uint64_t* k_in = (uint64_t*)base;
    uint64_t* k_out = (uint64_t*)(base + bk);
    uint32_t* v_in = (uint32_t*)(base + 2 * bk);
    uint32_t* v_out = (uint32_t*)(base + 2 * bk + bv);
    void* tmp = base + 2 * bk + 2 * bv;
    hit_keys_kernel<<<(unsigned)((n + 255) / 256), 256, 0, ctx->stream>>>(ctx->hits.rec, n, k_in, v_in);
    PP_HIP(hipGetLastError());
    PP_HIP(rocprim::radix_sort_pairs(tmp, temp, k_in, k_out, v_in, v_out, (uint32_t)n, 0u,
                                     (unsigned)end_bit, ctx->stream));
    gather_hits_kernel<<<(unsigned)((n + 255) / 256), 256, 0, ctx->stream>>>(
        ctx->hits.rec, v_out, n, (HitRecord*)ctx->d_sort);
    PP_HIP(hipGetLastError());
    *done = true;
    return PP_OK;
}

// The caller's columns of a hit table, and where each lies in a slice of
// its rows (kNoColumn: not asked for).
enum { kColPos, kColDir, kColInit, kColWl, kColTime, kColDist, kColModule, kColSteps, kColPid, kColSrc,
       kColumns };
constexpr int64_t kSliceRows = 16384;  // of tables of up to 8 such slices; longer ones: twice
constexpr uint32_t kNoColumn = ~0u;
struct ColumnSet {
    uint32_t off[kColumns];
    int32_t time_f64;
};

// Rows of hit records as columns, `out` being pinned host memory. Splitting the
// records up on the host cost 7 ns a row and could not run beside the copy of the
// next ones (383224 hits: 2.8-3.2 ms a call); the columns of a slice are written
// while the host moves those of the slice before, one memcpy a column (1.0 ms).
// Written to device memory and copied from there, the first four copies of a
// context were slow: first and fourth call on 15430 hits 0.28 and 0.12 ms (split up
// on the host: 0.24-0.28 and 0.17-0.19), on 65177 hits 0.63 and 0.25 (0.74-0.82 and
// 0.50-0.56); straight to host memory 0.12 and 0.11, 0.26 and 0.23. Pinned memory
// that is new to the process costs the host 0.35 ms a MB when it is first touched:
// a table of one slice takes one half, and the slices of a few are half as long
// (65177 hits in a process's first context: 1.1-2.5 ms of call, else 3.6-4.3). Beyond
// 131072 rows the longer ones save more (383224 hits: 0.97-1.03 and 1.06-1.08 ms).
__global__ void __launch_bounds__(256) hit_columns_kernel(const HitRecord* __restrict__ rec, int n,
                                                          char* __restrict__ out, ColumnSet cs) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= n) return;
    const float4* r = reinterpret_cast<const float4*>(rec + k);
    const float4 a = r[0], b = r[1], c = r[2], d = r[3];
    auto put3 = [&](int col, float x, float y, float z) {
        if (cs.off[col] == kNoColumn) return;
        float* o = reinterpret_cast<float*>(out + cs.off[col]) + 3 * k;
        o[0] = x;
        o[1] = y;
        o[2] = z;
    };
    auto put = [&](int col, auto v) {
        if (cs.off[col] != kNoColumn) reinterpret_cast<decltype(v)*>(out + cs.off[col])[k] = v;
    };
    const uint64_t id = (uint64_t)__float_as_uint(d.x) | ((uint64_t)__float_as_uint(d.y) << 32);
    put3(kColPos, a.x, a.y, a.z);
    put3(kColDir, a.w, b.x, b.y);
    put3(kColInit, b.z, b.w, c.x);
    put(kColWl, c.y);
    if (cs.time_f64) put(kColTime, (double)c.z);
    else put(kColTime, c.z);
    put(kColDist, c.w);
    put(kColModule, (int64_t)((id >> kPidBits) & 0xFFFF));
    put(kColSteps, __float_as_int(d.z));
    put(kColPid, id & (kMaxPhotonsPerSource - 1));
    put(kColSrc, __float_as_int(d.w));
}

// Rows [0, n) of the device records src to the caller's columns (NULL: not asked
// for), slice by slice. Sets *done = false and does nothing where the slices do
// not fit pinned memory.
static int copy_columns(pp_ctx* ctx, const HitRecord* src, int64_t n, void* const col[kColumns],
                        const uint32_t width[kColumns], int time_f64, bool* done) {
    *done = false;
    ColumnSet cs{};
    cs.time_f64 = time_f64;
    const int64_t rows = std::min<int64_t>(n, n <= 8 * kSliceRows ? kSliceRows : 2 * kSliceRows);
    size_t bytes = 0;
    for (int c = 0; c < kColumns; ++c) {
        cs.off[c] = col[c] ? (uint32_t)bytes : kNoColumn;
        if (col[c]) bytes += align256((size_t)rows * width[c]);
    }
    if (bytes == 0) {
        *done = true;
        return PP_OK;
    }
    const int64_t slices = (n + rows - 1) / rows;
    if (ctx->pin.ensure(bytes, slices > 1 ? 2 : 1) != hipSuccess) {
        (void)hipGetLastError();
        return PP_OK;
    }
    auto slice_rows = [&](int64_t k) { return std::min<int64_t>(rows, n - k * rows); };
    auto move = [&](int64_t k) -> int {
        if (k < slices) {
            const int64_t m = slice_rows(k);
            hipLaunchKernelGGL(hit_columns_kernel, dim3((unsigned)((m + 255) / 256)), dim3(256), 0,
                               ctx->stream, src + k * rows, (int)m, ctx->pin.at((int)(k & 1)), cs);
            PP_HIP(hipGetLastError());
            PP_HIP(hipEventRecord(ctx->pin.ev[k & 1], ctx->stream));
        }
        if (k > 0) {
            PP_HIP(hipEventSynchronize(ctx->pin.ev[(k - 1) & 1]));
            const char* in = ctx->pin.at((int)((k - 1) & 1));
            for (int c = 0; c < kColumns; ++c)
                if (col[c])
                    std::memcpy((char*)col[c] + (k - 1) * rows * width[c], in + cs.off[c],
                                (size_t)slice_rows(k - 1) * width[c]);
        }
        return PP_OK;
    };
    for (int64_t k = 0; k <= slices; ++k)
        if (int rc = move(k)) {
            (void)hipStreamSynchronize(ctx->stream);
            return rc;
        }
    *done = true;
    return PP_OK;
}

int pp_copy_hits(pp_ctx* ctx, int64_t first, int64_t n, float* pos3, float* dir3,
                 float* init_dir3, float* wavelength, void* time, int time_f64,
                 float* dist_travelled, int64_t* module_ix, int32_t* n_steps,
                 uint64_t* photon_id, int32_t* source_ix) {
    if (!ctx) return fail(PP_ERR_INVALID, "pp_copy_hits: NULL ctx");
    if (first < 0 || n < 0 || first > ctx->n_hits || n > ctx->n_hits - first)
        return fail(PP_ERR_INVALID, "pp_copy_hits: range outside [0, n_hits)");
    if (n == 0) return PP_OK;
    if (int rc = set_dev(ctx)) return rc;
    // deterministic_order: 0 = buffer order, 1 = sorted on the device (host
    // where the device cannot), 2 = sorted on the host (no device buffer)
    const bool ordered = ctx->cfg.deterministic_order != 0;
    auto ensure_staging = [&](int64_t records) -> int {
        if (records <= ctx->h_rec_cap) return PP_OK;
        if (ctx->h_rec) PP_HIP(hipHostFree(ctx->h_rec));
        ctx->h_rec = nullptr;
        ctx->h_rec_cap = 0;
        PP_HIP(hipHostMalloc((void**)&ctx->h_rec, (size_t)records * sizeof(HitRecord),
                             hipHostMallocDefault));
        ctx->h_rec_cap = records;
        return PP_OK;
    };
    bool staged = false;  // every ordered record is on its way to h_rec
    if (ordered && ctx->cfg.deterministic_order != 2 && !ctx->sorted_valid && !ctx->perm_valid) {
        bool done = false;
        const bool few = ctx->n_hits <= kRankMost;
        if (few)
            if (int rc = ensure_staging(kRankMost)) return rc;
        if (int rc = sort_hits_device(ctx, &done, few ? ctx->h_rec : nullptr)) return rc;
        ctx->sorted_valid = done;
        staged = few && done;
    }
    // the host sorts only where the device could not: it then reads every record
    const bool host_sort = ordered && (ctx->cfg.deterministic_order == 2 || !ctx->sorted_valid);
    // records to read: [lo, lo+cnt) of the device buffer src
    const HitRecord* src = ordered && !host_sort ? (const HitRecord*)ctx->d_sort : ctx->hits.rec;
    const int64_t lo = host_sort ? 0 : first, cnt = host_sort ? ctx->n_hits : n;
    if (!staged && !host_sort) {
        void* const col[kColumns] = {pos3, dir3, init_dir3, wavelength, time, dist_travelled,
                                     module_ix, n_steps, photon_id, source_ix};
        const uint32_t width[kColumns] = {12, 12, 12, 4, time_f64 ? 8u : 4u, 4, 8, 4, 8, 4};
        bool done = false;
        if (int rc = copy_columns(ctx, src + lo, cnt, col, width, time_f64, &done)) return rc;
        if (done) return PP_OK;
    }
    // otherwise records stream through a pinned staging buffer of at most
    // kStageRecords records (kept by the context); the host sort, which
    // needs random access to every record, collects them in pageable memory
    const int64_t stage = std::min<int64_t>(cnt, kStageRecords);
    if (!staged)
        if (int rc = ensure_staging(stage)) return rc;
    const uint64_t pid_mask = kMaxPhotonsPerSource - 1;
    auto scatter = [&](const HitRecord& r, int64_t k) {
        for (int c = 0; c < 3; ++c) {
            if (pos3) pos3[3 * k + c] = r.f[c];
            if (dir3) dir3[3 * k + c] = r.f[3 + c];
            if (init_dir3) init_dir3[3 * k + c] = r.f[6 + c];
        }
        if (wavelength) wavelength[k] = r.f[9];
        if (time) {
            if (time_f64)
                ((double*)time)[k] = r.f[10];
            else
                ((float*)time)[k] = r.f[10];
        }
        if (dist_travelled) dist_travelled[k] = r.f[11];
        if (module_ix) module_ix[k] = (int64_t)((r.id >> kPidBits) & 0xFFFF);
        if (n_steps) n_steps[k] = r.n_steps;
        if (photon_id) photon_id[k] = r.id & pid_mask;
        if (source_ix) source_ix[k] = r.source_ix;
    };
    if (staged) {
        PP_HIP(hipStreamSynchronize(ctx->stream));
        for (int64_t k = 0; k < n; ++k) scatter(ctx->h_rec[first + k], k);
        return PP_OK;
    }
    std::vector<HitRecord> all;
    if (host_sort) all.resize((size_t)cnt);
    for (int64_t off = 0; off < cnt; off += stage) {
        const int64_t m = std::min<int64_t>(stage, cnt - off);
        PP_HIP(hipMemcpyAsync(ctx->h_rec, src + lo + off, (size_t)m * sizeof(HitRecord),
                              hipMemcpyDeviceToHost, ctx->stream));
        PP_HIP(hipStreamSynchronize(ctx->stream));
        if (host_sort)
            std::memcpy(all.data() + off, ctx->h_rec, (size_t)m * sizeof(HitRecord));
        else
            for (int64_t k = 0; k < m; ++k) scatter(ctx->h_rec[k], off + k);
    }
    if (!host_sort) return PP_OK;
    if (!ctx->perm_valid) {
        // sort (source, photon id) keys beside their record index: one
        // contiguous array instead of indirect two-field compares
        struct Key {
            int32_t src;
            uint64_t pid;
            int64_t idx;
        };
        std::vector<Key> keys((size_t)ctx->n_hits);
        for (int64_t k = 0; k < ctx->n_hits; ++k)
            keys[(size_t)k] = {all[(size_t)k].source_ix, all[(size_t)k].id & pid_mask, k};
        std::sort(keys.begin(), keys.end(), [](const Key& a, const Key& b) {
            return a.src != b.src ? a.src < b.src : a.pid < b.pid;
        });
        ctx->perm.resize((size_t)ctx->n_hits);
        for (int64_t k = 0; k < ctx->n_hits; ++k) ctx->perm[(size_t)k] = keys[(size_t)k].idx;
        ctx->perm_valid = true;
    }
    for (int64_t k = 0; k < n; ++k) scatter(all[(size_t)ctx->perm[(size_t)(first + k)]], k);
    return PP_OK;
}

}  // extern "C"

int pp::ctx_hit_records(pp_ctx* ctx, const HitRecord** rec, int64_t* n, hipStream_t* stream,
                        int* device) {
    if (!ctx) return fail(PP_ERR_INVALID, "NULL ctx");
    if (int rc = set_dev(ctx)) return rc;
    *rec = ctx->hits.rec;
    *n = ctx->n_hits;
    *stream = ctx->stream;
    *device = ctx->device;
    return PP_OK;
}

extern "C" {

int pp_release_scratch(pp_ctx* ctx) {
    if (!ctx) return fail(PP_ERR_INVALID, "pp_release_scratch: NULL ctx");
    if (int rc = set_dev(ctx)) return rc;
    PP_HIP(hipStreamSynchronize(ctx->stream));
    if (ctx->d_sort) PP_HIP(hipFree(ctx->d_sort));
    if (ctx->h_rec) PP_HIP(hipHostFree(ctx->h_rec));
    if (ctx->d_pmt) PP_HIP(hipFree(ctx->d_pmt));
    ctx->d_sort = nullptr;
    ctx->d_sort_cap = 0;
    ctx->sorted_valid = false;
    ctx->h_rec = nullptr;
    ctx->h_rec_cap = 0;
    ctx->d_pmt = nullptr;
    ctx->pmt_cap = 0;
    ctx->pin.release();
    std::vector<int64_t>().swap(ctx->perm);
    ctx->perm_valid = false;
    return PP_OK;
}

int pp_pom_pmt_hits_ctx(pp_ctx* ctx, const pp_pom_model* m, const float* wl_grid,
                        const float* acc1, const float* acc2, uint64_t seed, int64_t first,
                        int64_t n, int32_t* pmt_id_out, int64_t* n_detected, float* kernel_ms) {
    if (!ctx) return fail(PP_ERR_INVALID, "pp_pom_pmt_hits_ctx: NULL ctx");
    if (n_detected) *n_detected = 0;
    if (kernel_ms) *kernel_ms = 0.0f;
    if (!m || m->n_wl < 2 || m->n_wl > 1024)
        return fail(PP_ERR_INVALID, "pp_pom_pmt_hits_ctx: model with n_wl in [2, 1024] required");
    if (first < 0 || n < 0 || first > ctx->n_hits || n > ctx->n_hits - first)
        return fail(PP_ERR_INVALID, "pp_pom_pmt_hits_ctx: range outside [0, n_hits)");
    if (ctx->planar)
        return fail(PP_ERR_INVALID,
                    "pp_pom_pmt_hits_ctx: the target list holds planar targets (POMs are spheres)");
    pp::PmtSetup st{};
    std::vector<float> tab(3 * (size_t)m->n_wl);
    if (int rc = pp::pmt_setup(m, wl_grid, acc1, acc2, seed, &st, tab.data())) return rc;
    if (n == 0) return PP_OK;
    if (!pmt_id_out) return fail(PP_ERR_INVALID, "pp_pom_pmt_hits_ctx: NULL output");
    if (int rc = set_dev(ctx)) return rc;
    // the records in the order pp_copy_hits returns them
    const bool ordered = ctx->cfg.deterministic_order != 0;
    if (ordered && ctx->cfg.deterministic_order != 2 && !ctx->sorted_valid && !ctx->perm_valid) {
        bool done = false;
        if (int rc = sort_hits_device(ctx, &done)) return rc;
        ctx->sorted_valid = done;
    }
    const bool host_sort = ordered && (ctx->cfg.deterministic_order == 2 || !ctx->sorted_valid);
    const HitRecord* src = ordered && !host_sort ? (const HitRecord*)ctx->d_sort : ctx->hits.rec;
    const int64_t lo = host_sort ? 0 : first, cnt = host_sort ? ctx->n_hits : n;
    // table | PMT ids, kept by the context and grown when needed
    const size_t off_out = align256(tab.size() * sizeof(float));
    const size_t need = off_out + (size_t)cnt * sizeof(int32_t);
    if (need > ctx->pmt_cap) {
        PP_HIP(hipStreamSynchronize(ctx->stream));
        if (ctx->d_pmt) PP_HIP(hipFree(ctx->d_pmt));
        ctx->d_pmt = nullptr;
        ctx->pmt_cap = 0;
        if (hipMalloc((void**)&ctx->d_pmt, need) != hipSuccess) {
            (void)hipGetLastError();
            return fail(PP_ERR_NOMEM, "pp_pom_pmt_hits_ctx: device allocation failed");
        }
        ctx->pmt_cap = need;
    }
    float* d_tab = (float*)ctx->d_pmt;
    auto* d_out = (int32_t*)(ctx->d_pmt + off_out);
    if (m->n_wl > pp::kArgKnots)
        PP_HIP(hipMemcpyAsync(d_tab, tab.data(), tab.size() * sizeof(float), hipMemcpyHostToDevice,
                              ctx->stream));
    PP_HIP(hipEventRecord(ctx->ev0, ctx->stream));
    if (int rc = pp::pmt_launch_records(st, tab.data(), d_tab, src + lo, cnt, ctx->d_tgt_r, d_out,
                                        ctx->stream, ctx->n_cu))
        return rc;
    PP_HIP(hipEventRecord(ctx->ev1, ctx->stream));
    std::vector<int32_t> all;
    int32_t* dst = pmt_id_out;
    if (host_sort) {
        all.resize((size_t)cnt);
        dst = all.data();
    }
    PP_HIP(ctx->pin.copy_out(ctx->stream, dst, d_out, (size_t)cnt * sizeof(int32_t)));
    if (kernel_ms) PP_HIP(hipEventElapsedTime(kernel_ms, ctx->ev0, ctx->ev1));
    if (host_sort) {
        if (!ctx->perm_valid) {
            // the same (source, photon id) order as pp_copy_hits's host sort
            std::vector<HitRecord> rec((size_t)ctx->n_hits);
            PP_HIP(hipMemcpyAsync(rec.data(), ctx->hits.rec, rec.size() * sizeof(HitRecord),
                                  hipMemcpyDeviceToHost, ctx->stream));
            PP_HIP(hipStreamSynchronize(ctx->stream));
            std::vector<int64_t> perm((size_t)ctx->n_hits);
            std::iota(perm.begin(), perm.end(), 0);
            const uint64_t mask = kMaxPhotonsPerSource - 1;
            std::sort(perm.begin(), perm.end(), [&](int64_t a, int64_t b) {
                const HitRecord &x = rec[(size_t)a], &y = rec[(size_t)b];
                return x.source_ix != y.source_ix ? x.source_ix < y.source_ix
                                                  : (x.id & mask) < (y.id & mask);
            });
            ctx->perm.swap(perm);
            ctx->perm_valid = true;
        }
        for (int64_t k = 0; k < n; ++k) pmt_id_out[k] = all[(size_t)ctx->perm[(size_t)(first + k)]];
    }
    if (n_detected) {
        int64_t c = 0;
        for (int64_t k = 0; k < n; ++k) c += pmt_id_out[k] != 0;
        *n_detected = c;
    }
    return PP_OK;
}

int pp_eval_fn(pp_ctx* ctx, int fn, const float* in, int in_stride, float* out, int out_stride,
               int64_t n) {
    static const int kIn[PP_FN_COUNT] = {2, 6, 2, 2, 5, 11, 2, 1, 2, 6, 7, 1, 2, 13, 5};
    static const int kOut[PP_FN_COUNT] = {3, 3, 1, 1, 3, 2, 1, 3, 3, 4, 2, 1, 1, 2, 1};
    if (!ctx) return fail(PP_ERR_INVALID, "pp_eval_fn: NULL ctx");
    if (fn < 0 || fn >= PP_FN_COUNT) return fail(PP_ERR_INVALID, "pp_eval_fn: unknown function");
    if (n < 0 || (n > 0 && (!in || !out)))
        return fail(PP_ERR_INVALID, "pp_eval_fn: bad buffers");
    if (in_stride < kIn[fn] || out_stride < kOut[fn])
        return fail(PP_ERR_INVALID, "pp_eval_fn: stride smaller than the function's arity");
    if (fn == PP_FN_CASCADIA && !ctx->has_medium)
        return fail(PP_ERR_STATE, "pp_eval_fn: set a medium first");
    if (fn == PP_FN_SPECTRUM && !ctx->has_spectrum)
        return fail(PP_ERR_STATE, "pp_eval_fn: set a spectrum first");
    if (n == 0) return PP_OK;
    if (int rc = set_dev(ctx)) return rc;
    float *d_in = nullptr, *d_out = nullptr;
    const size_t in_b = (size_t)n * in_stride * 4, out_b = (size_t)n * out_stride * 4;
    PP_HIP(hipMalloc(&d_in, in_b));
    if (hipMalloc(&d_out, out_b) != hipSuccess) {
        (void)hipFree(d_in);
        return fail(PP_ERR_NOMEM, "pp_eval_fn: output allocation");
    }
    int rc = PP_OK;
    do {
        // everything on the context stream, in order
        if (hipMemcpyAsync(d_in, in, in_b, hipMemcpyHostToDevice, ctx->stream) != hipSuccess) { rc = fail(PP_ERR_HIP, "copy in"); break; }
        if (hipMemsetAsync(d_out, 0, out_b, ctx->stream) != hipSuccess) { rc = fail(PP_ERR_HIP, "memset"); break; }
        EvalParams e{};
        e.fn = fn;
        e.in_stride = in_stride;
        e.out_stride = out_stride;
        e.n = n;
        e.in = d_in;
        e.out = d_out;
        e.med = ctx->medium;
        e.spec = ctx->d_spec;
        e.spec_n = ctx->spec_n;
        e.spec_map = ctx->spec_map;
        e.spec_mono = ctx->spec_mono;
        e.spec_nf = (float)ctx->spec_n;
        e.spec_lastf = (float)(ctx->spec_n - 1);
        const int64_t grid = (n + 255) / 256;
        hipLaunchKernelGGL(eval_fn_kernel, dim3((unsigned)grid), dim3(256), 0, ctx->stream, e);
        if (hipGetLastError() != hipSuccess) { rc = fail(PP_ERR_HIP, "eval launch"); break; }
        if (hipMemcpyAsync(out, d_out, out_b, hipMemcpyDeviceToHost, ctx->stream) != hipSuccess) { rc = fail(PP_ERR_HIP, "copy out"); break; }
        if (hipStreamSynchronize(ctx->stream) != hipSuccess) { rc = fail(PP_ERR_HIP, "eval sync"); break; }
    } while (0);
    (void)hipFree(d_in);
    (void)hipFree(d_out);
    return rc;
}

}  // extern "C"
