// kernels.hip -- gfx950 kernels of the electron Monte Carlo path.
//
// Work unit: a chunk of up to ~1k main electrons of one condition, owned by
// one wavefront, with its own newborn region and hole list.  One
// synchronization interval of every running condition is this sequence:
//   k_advance      persistent per field case: each wave takes chunks from a
//                  work queue and flies every electron of the chunk, and every
//                  electron ejected on the way, to t_sync.  Lanes take the
//                  next electron as soon as theirs is done (ballot-ranked
//                  queue), so a wave never waits for its slowest electron.
//                  Collisions are counted in LDS per wave and added to the
//                  condition's integer accumulators; attached electrons leave
//                  holes that the chunk's own newborns refill.
//   k_marks        exact uniform removal of R electrons, first half: Bernoulli
//                  marks drawn by geometric skips, counted per chunk.
//   k_apply_marks  second half: the R marks with the smallest random keys are
//                  removed.  (k_plan_marks finds the R-th smallest key of a
//                  large condition, k_plan_pairs the hole and newborn offsets
//                  of a condition of very many chunks, one block each.)
//   k_settle       surplus newborns fill holes; clones of uniformly chosen
//                  electrons fill the holes that remain (rejection, as the
//                  reference does at BoltzmannMC.C:1368-1371); FP64 moments of
//                  the N electrons at t_sync, per chunk (BoltzmannMC.C:1410-1482).
//   k_finish       per condition: fixed-order sums of the chunk records, the
//                  integer accumulators, the plan; resets the queues.
// Every floating-point reduction runs in a fixed order (wave butterflies, then
// chunks in index order), everything else is integer, so runs are bitwise
// reproducible whatever the order in which waves take chunks.
#include "kernels.h"
#include "device_physics.h"

namespace ekmc {

const char* kKernelNames[K_COUNT] = {"init", "advance", "marks", "apply_marks", "settle", "hist", "finish"};

// level 1 times the flight kernels only, level 2 every kernel
static inline bool timed(const KernelTimer* t, int k) { return t && (t->level >= 2 || (t->level == 1 && k == K_ADVANCE)); }
static inline void timer_start(KernelTimer* t, int k, hipStream_t st) {
    if (timed(t, k)) (void)hipEventRecord(t->start[k], st);
}
static inline void timer_stop(KernelTimer* t, int k, hipStream_t st) {
    if (timed(t, k)) { (void)hipEventRecord(t->stop[k], st); t->armed[k] = true; }
}

constexpr double kFix = 16777216.0;  // 2^24: fixed-point scale of energy sums [eV]
static inline unsigned grid_of(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }
constexpr int kWavesPerBlock = kBlock / kWave;
// Null-collision events a lane may run in one phase-A step of the flight
// kernel: a null event costs a flight and a null test, not a whole step of
// the wave's bookkeeping.  Measured per interval on the 64-condition scan,
// mixed form: 1 / 2 / 3 / 4 events, 0.981 / 0.963 / 0.989 / 1.062 ms (longer
// runs leave more lanes idle in the loop than they save); FP64 form, whose flights
// are the longer: 1 / 2 events, 1.419 / 1.434 ms, one condition of 3e7 electrons
// 2106 / 2122 us, four ECR conditions 76.3 / 77.7, one of 1e5 67.5 / 66.3.
template <typename V> constexpr int null_run() { return sizeof(V) == 8 ? 1 : 2; }

// LDS of one wave of the flight kernel: collision tallies [3P] (64-bit), the
// histogram grid of the chunk's condition [8] (FP64), the null-test envelope
// [2 kEnvBins] (V) and the EEDF counts of a histogram taken at load [histLds]
// (16-bit, two cells per word: a chunk holds at most 65535 main electrons).
// The record ring is a separate static array.
template <typename V> __host__ __device__ constexpr size_t flight_wave_lds(int P, int histLds) {
    return (size_t)3 * P * 8 + 8 * 8 + (size_t)2 * kEnvBins * sizeof(V) + (size_t)((histLds + 1) / 2) * 4;
}

// ------------------------------------------------------------ wave helpers
__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }
// number of set bits of `mask` below this lane
__device__ __forceinline__ int lane_rank(uint64_t mask) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, kWave));
    return v;
}
__device__ __forceinline__ uint32_t wave_sum_u(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
    return v;
}
__device__ __forceinline__ uint32_t wave_or(uint32_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v |= __shfl_xor(v, o, kWave);
    return v;
}
// exclusive prefix over the lanes of a wave
__device__ __forceinline__ int wave_exclusive_scan(int v) {
    int incl = v;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        int t = __shfl_up(incl, o, kWave);
        if (lane_id() >= o) incl += t;
    }
    return incl - v;
}
// Wait until this wave's LDS operations are done (all lanes), so that other
// lanes of the same wave see them.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
}

// ------------------------------------------------------------ records
template <typename V> __device__ __forceinline__ void rec_to_electron(const Rec<V>& q, Electron<V>& e) {
    e.x = q.a.x; e.y = q.a.y; e.z = q.a.z; e.t = q.a.t;
    e.vx = q.a.vx; e.vy = q.a.vy; e.vz = q.a.vz;
    e.eps = energy_of(q.a.vx, q.a.vy, q.a.vz);
    e.tfree = q.a.tfree;
    e.nue = draw_part(q).nue; e.stream = draw_part(q).stream; e.event = draw_part(q).event;
}
template <typename V> __device__ __forceinline__ Rec<V> rec_get(const DevState<V>& s, int64_t i) {
    Rec<V> q;
    q.a = s.ra[i];
    if constexpr (split_record<V>()) q.b = s.rb[i];
    return q;
}
template <typename V> __device__ __forceinline__ void rec_put(const DevState<V>& s, int64_t i, const Rec<V>& q) {
    s.ra[i] = q.a;
    if constexpr (split_record<V>()) s.rb[i] = q.b;
}
template <typename V> __device__ __forceinline__ void load_rec(const DevState<V>& s, int64_t i, Electron<V>& e) {
    rec_to_electron(rec_get(s, i), e);
}
template <typename V> __device__ __forceinline__ void store_rec(const DevState<V>& s, int64_t i, const Electron<V>& e) {
    Rec<V> q = {};
    q.a.x = e.x; q.a.y = e.y; q.a.z = e.z; q.a.t = e.t;
    q.a.vx = e.vx; q.a.vy = e.vy; q.a.vz = e.vz; q.a.tfree = e.tfree;
    draw_part(q).nue = e.nue; draw_part(q).event = e.event; draw_part(q).stream = e.stream;
    rec_put(s, i, q);
}
// A value of the lane that quad_perm CTRL names, within each four lanes.
template <int CTRL> __device__ __forceinline__ uint32_t quad_get(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xf, 0xf, true);
}
// Lanes 2k and 2k + 1 (XOR 1), or k and k + 2 of four (XOR 2), exchange: the lower
// keeps a and gets the upper's a in b, the upper keeps b and gets the lower's b in a.
template <int XOR> __device__ __forceinline__ void lane_swap(uint4& a, uint4& b, bool upper) {
    constexpr int ctrl = XOR == 1 ? 0xB1 : 0x4E;  // quad_perm 1,0,3,2 / 2,3,0,1
    uint32_t x[4] = {a.x, a.y, a.z, a.w}, y[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t xo = quad_get<ctrl>(x[k]), yo = quad_get<ctrl>(y[k]);
        x[k] = upper ? yo : x[k];
        y[k] = upper ? y[k] : xo;
    }
    a = make_uint4(x[0], x[1], x[2], x[3]);
    b = make_uint4(y[0], y[1], y[2], y[3]);
}
template <int J> __device__ __forceinline__ void store_quad(char* base, uint32_t slot, const uint4& v, int lane) {
    const uint32_t to = quad_get<J * 0x55>(slot);
    if (to != 0xffffffffu) *(uint4*)(base + ((size_t)to * 64 + (lane & 3) * 16)) = v;
}
// Store the records of the lanes with `put` (called by a whole wave).  A lane
// storing its own record writes 16 bytes to each of 64 places per instruction,
// four L2 writes per record; here the lanes of four exchange pieces first, so
// that each instruction writes whole 64-byte records, four lanes to a record.
// The exchange is about 50 instructions a step; it pays where the chip is full
// of waves and the L2 writes are what they wait for, so for the mixed form in
// launches with more chunks than waves.  Flight kernel per interval, own record
// against this: 64-condition scan 827 -> 784 us, one condition of 3e7 electrons
// 1324 -> 1234, 24 AC conditions of 2e5 635 -> 620; but one condition of 1e4
// 43.9 -> 46.6, eight of 1e5 (a wave per chunk) 137 -> 145, one of 1e8 with
// thermal targets (bound by the collision step) 14.1 -> 14.3 ms, and the FP64
// form, whose record has a second part of 32 bytes, 2341 -> 2450 for one of 3e7.
template <typename V>
__device__ __forceinline__ void store_recs(const DevState<V>& s, bool put, int64_t slot, const Electron<V>& e) {
    Rec<V> q = {};
    q.a.x = e.x; q.a.y = e.y; q.a.z = e.z; q.a.t = e.t;
    q.a.vx = e.vx; q.a.vy = e.vy; q.a.vz = e.vz; q.a.tfree = e.tfree;
    draw_part(q).nue = e.nue; draw_part(q).event = e.event; draw_part(q).stream = e.stream;
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t to = put ? (uint32_t)slot : 0xffffffffu;  // the pool has less than 2^32 - 16 slots
    static_assert(sizeof(q.a) == 64, "four pieces");
    uint4 p[4];
    __builtin_memcpy(p, &q.a, 64);
    lane_swap<1>(p[0], p[1], lane & 1);
    lane_swap<1>(p[2], p[3], lane & 1);
    lane_swap<2>(p[0], p[2], lane & 2);
    lane_swap<2>(p[1], p[3], lane & 2);
    char* base = (char*)s.ra;
    store_quad<0>(base, to, p[0], lane);
    store_quad<1>(base, to, p[1], lane);
    store_quad<2>(base, to, p[2], lane);
    store_quad<3>(base, to, p[3], lane);
}
template <typename V> __device__ __forceinline__ double rec_energy(const RecA<V>& q) {
    return (double)energy_of(q.vx, q.vy, q.vz);
}

// ------------------------------------------------------------ record ring
// The main records of a chunk stream through a per-wave ring in LDS of
// ring_segs<V>() segments of kRingSeg records, filled by direct-to-LDS loads
// issued up to ring_segs - 1 segments ahead of use: a lane taking the next
// main electron reads LDS, and the HBM latency of the record overlaps the
// flights of the wave.  Fill f of a chunk loads chunk-relative main records
// [f kRingSeg, (f + 1) kRingSeg) into segment f % ring_segs; piece k
// (16 bytes) of slot j of a segment is seg[k * kRingSeg + j].  Lane
// j < kRingSeg issues the loads of slot j (the LDS address a lane writes is
// the base plus 16 * lane), so every fill is rec_pieces vector memory
// instructions (lane 0 always has a record).  A wave's vector memory
// operations complete in issue order (vmcnt), so fill f has landed once at
// most rec_pieces * (fills issued after f) operations are outstanding: the
// first read of a segment waits for exactly that, not for the younger fills.
// A read completes inside its own instruction group, so a later fill of that
// segment cannot overtake it.
static_assert(kRingSeg == kWave / 2, "a segment's records once per half-wave");
template <typename V> __host__ __device__ constexpr int rec_pieces() { return (int)(sizeof(Rec<V>) / 16); }
template <typename V> __host__ __device__ constexpr int rec_pieces_a() { return (int)(sizeof(RecA<V>) / 16); }
static_assert(flight_ring_lds<float>() == (size_t)ring_segs<float>() * kWavesPerBlock * kRingSeg * sizeof(Rec<float>),
              "ring size");
typedef __attribute__((address_space(1))) void global_void;
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) uint4 lds_uint4;  // LDS pointers stay LDS pointers

template <typename V> __device__ __forceinline__ lds_uint4* ring_segment(lds_uint4* ring, int record) {
    return ring + ((record / kRingSeg) % ring_segs<V>()) * (rec_pieces<V>() * kRingSeg);
}
// Loads of main records [loaded, loaded + kRingSeg) of a chunk of `count`
// into their segment.  PAIR: each direct-to-LDS load of the wave writes 1 KB,
// the lower half-wave piece k of the 32 records and the upper half-wave piece
// k + 1 (mixed flight kernel 0.900 -> 0.883 ms per interval on the
// 64-condition scan, FP64 1.477 -> 1.466 ms); otherwise the lower half-wave
// loads one piece per instruction.  A fill always holds record `loaded`, so
// it issues exactly ring_loads<V, PAIR>() loads.
template <typename V, bool PAIR> __host__ __device__ constexpr int ring_loads() {
    return PAIR ? rec_pieces<V>() / 2 : rec_pieces<V>();
}
template <typename V, bool PAIR>
__device__ __forceinline__ void ring_fill(const DevState<V>& s, int64_t first, int count, int loaded, lds_uint4* ring) {
    const int lane = lane_id();
    lds_uint4* seg = ring_segment<V>(ring, loaded);
    if constexpr (PAIR) {
        static_assert(rec_pieces<V>() % 2 == 0, "pieces are loaded in pairs");
        const int half = lane / kRingSeg;  // lanes 32-63 load the odd pieces
        const int idx = loaded + (lane % kRingSeg);
        if (idx < count) {
            const char* srcA = (const char*)(s.ra + first + idx);
            const char* srcB = (const char*)(s.rb + first + idx);
#pragma unroll
            for (int k = 0; k < rec_pieces<V>(); k += 2) {
                const int piece = k + half;
                const char* src = piece < rec_pieces_a<V>() ? srcA + 16 * piece : srcB + 16 * (piece - rec_pieces_a<V>());
                __builtin_amdgcn_global_load_lds((global_void*)src, (lds_void*)(seg + k * kRingSeg), 16, 0, 0);
            }
        }
    } else {
        const int idx = loaded + lane;
        if (lane < kRingSeg && idx < count) {
            const char* srcA = (const char*)(s.ra + first + idx);
            const char* srcB = (const char*)(s.rb + first + idx);
#pragma unroll
            for (int k = 0; k < rec_pieces<V>(); ++k) {
                const char* src = k < rec_pieces_a<V>() ? srcA + 16 * k : srcB + 16 * (k - rec_pieces_a<V>());
                __builtin_amdgcn_global_load_lds((global_void*)src, (lds_void*)(seg + k * kRingSeg), 16, 0, 0);
            }
        }
    }
}
// s_waitcnt with vmcnt(N) (expcnt and lgkmcnt not waited for)
template <int N> __device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// Wait until a fill followed by `later` younger fills has landed (each fill
// is ring_loads<V, PAIR>() loads; completion is in order).
template <typename V, bool PAIR> __device__ __forceinline__ void ring_wait(int later) {
    constexpr int p = ring_loads<V, PAIR>();
    static_assert(ring_segs<V>() <= 4, "ring_wait covers at most 3 younger fills");
    if (later <= 0) wait_vmcnt<0>();
    else if (later == 1) wait_vmcnt<p>();
    else if (later == 2) wait_vmcnt<2 * p>();
    else wait_vmcnt<3 * p>();
}
// The pieces of one ring slot at LDS byte address `a`, read and waited for
// in one group.
__device__ __forceinline__ void ring_pieces(uint32_t a, uint4 (&p)[4]) {
    asm volatile(
        "ds_read_b128 %0, %4\n\t"
        "ds_read_b128 %1, %4 offset:512\n\t"
        "ds_read_b128 %2, %4 offset:1024\n\t"
        "ds_read_b128 %3, %4 offset:1536\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(p[0]), "=&v"(p[1]), "=&v"(p[2]), "=&v"(p[3])
        : "v"(a)
        : "memory");
}
__device__ __forceinline__ void ring_pieces(uint32_t a, uint4 (&p)[6]) {
    asm volatile(
        "ds_read_b128 %0, %6\n\t"
        "ds_read_b128 %1, %6 offset:512\n\t"
        "ds_read_b128 %2, %6 offset:1024\n\t"
        "ds_read_b128 %3, %6 offset:1536\n\t"
        "ds_read_b128 %4, %6 offset:2048\n\t"
        "ds_read_b128 %5, %6 offset:2560\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(p[0]), "=&v"(p[1]), "=&v"(p[2]), "=&v"(p[3]), "=&v"(p[4]), "=&v"(p[5])
        : "v"(a)
        : "memory");
}
static_assert(kRingSeg * 16 == 512, "ring piece stride");
// LDS atomic add without return, issued as is: the compiler would otherwise
// order it after the outstanding ring loads (it cannot tell the histogram
// from the ring), which would expose their HBM latency.
__device__ __forceinline__ void lds_add_u32(uint32_t* p, uint32_t v) {
    asm volatile("ds_add_u32 %0, %1" : : "v"((uint32_t)(size_t)(lds_void*)p), "v"(v) : "memory");
}
// Slot j of a ring segment.
template <typename V> __device__ __forceinline__ void ring_read(const lds_uint4* seg, int j, Electron<V>& e) {
    uint4 p[rec_pieces<V>()];
    ring_pieces((uint32_t)(size_t)(seg + j), p);
    Rec<V> q;
    __builtin_memcpy(&q, p, sizeof(q));
    rec_to_electron(q, e);
}

// -------------------------------------------- population-control totals
// A condition's totals: the waves of its chunks add to kPopCopies copies, by
// block index, so to different addresses on different XCDs (blocks go to the
// XCDs in turn).  Adds to one address from all of them take 8 ns each: with
// one copy, the 98,000 chunks of one condition of 1e8 electrons made k_marks
// 0.81 ms instead of 0.08 ms.
__device__ __forceinline__ CondPop& pop_mine(const DevWork& w, int c) {
    return w.pop[(size_t)(blockIdx.x % kPopCopies) * w.popStride + c];
}
__device__ __forceinline__ CondPop pop_total(const DevWork& w, int c) {
    CondPop t = {};
#pragma unroll
    for (int k = 0; k < kPopCopies; ++k) {
        const CondPop p = w.pop[(size_t)k * w.popStride + c];
        t.holes += p.holes; t.surplus += p.surplus; t.marks += p.marks; t.holesAfter += p.holesAfter;
    }
    return t;
}

// ------------------------------------------------------- block helpers
// Sum over a kBlock-thread block in a fixed order; result valid in thread 0.
__device__ double block_sum(double v, double* red) {
    v = wave_sum(v);
    int lane = lane_id(), wid = threadIdx.x / kWave;
    __syncthreads();
    if (lane == 0) red[wid] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < (int)(blockDim.x / kWave); ++i) r += red[i];
    __syncthreads();
    return r;
}
__device__ double block_max(double v, double* red) {
    v = wave_max(v);
    int lane = lane_id(), wid = threadIdx.x / kWave;
    __syncthreads();
    if (lane == 0) red[wid] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0)
        for (int i = 0; i < (int)(blockDim.x / kWave); ++i) r = fmax(r, red[i]);
    __syncthreads();
    return r;
}

// Exclusive scan of `in[0,n)` (int32) into `out` (int64) by one block of
// `blockDim.x` threads (a multiple of the wave, at most 64 waves); returns the
// total in every thread.  Tiles of 8 consecutive values per thread: a serial
// scan in each thread, a shuffle scan of the thread totals in each wave, a
// scan of the wave totals by the first wave, three barriers per tile (a
// one-value-per-thread Hillis-Steele tile took twenty; a condition of 1e8
// electrons has about 98,000 work units).  Integer sums: any order gives the
// same offsets.  `lds` holds at least 2 kWave + 1 values.
__device__ int64_t block_exclusive_scan(const int32_t* in, int64_t* out, int64_t n, int64_t* lds) {
    constexpr int E = 8;
    const int lane = lane_id(), wid = threadIdx.x / kWave, nw = blockDim.x / kWave;
    const int64_t tile = (int64_t)blockDim.x * E;
    int64_t running = 0;
    for (int64_t base = 0; base < n; base += tile) {
        const int64_t i0 = base + (int64_t)threadIdx.x * E;
        int64_t v[E], t = 0;
#pragma unroll
        for (int k = 0; k < E; ++k) {
            v[k] = i0 + k < n ? in[i0 + k] : 0;
            t += v[k];
        }
        int64_t incl = t;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int64_t u = __shfl_up(incl, o, kWave);
            if (lane >= o) incl += u;
        }
        if (lane == kWave - 1) lds[wid] = incl;
        __syncthreads();
        if (wid == 0) {
            const int64_t wt = lane < nw ? lds[lane] : 0;
            int64_t wi = wt;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const int64_t u = __shfl_up(wi, o, kWave);
                if (lane >= o) wi += u;
            }
            if (lane < nw) lds[kWave + lane] = wi - wt;
            if (lane == kWave - 1) lds[2 * kWave] = wi;
        }
        __syncthreads();
        int64_t pre = running + lds[kWave + wid] + incl - t;
#pragma unroll
        for (int k = 0; k < E; ++k) {
            if (i0 + k < n) out[i0 + k] = pre;
            pre += v[k];
        }
        running += lds[2 * kWave];
        __syncthreads();
    }
    return running;
}

// Index t of the range [off[t], off[t+1]) that contains i (largest t with
// off[t] <= i) over n exclusive offsets.
__device__ __forceinline__ int64_t owner_of(const int64_t* off, int64_t n, int64_t i) {
    int64_t lo = 0, hi = n - 1;
    while (lo < hi) {
        int64_t mid = (lo + hi + 1) >> 1;
        if (off[mid] <= i) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ double u53(uint64_t seed, uint64_t stream, uint32_t ev, uint32_t purpose, uint32_t call) {
    uint32_t w[4];
    philox_call(seed, stream, ev, purpose, call, w);
    uint64_t x = ((((uint64_t)w[0]) << 32) | w[1]) >> 11;
    return (double)x * (1.0 / 9007199254740992.0);
}

// ----------------------------------------------------------------- init
// Maxwellian at initialElecTempOverGasTemp * Tg (BoltzmannMC.C:491-516):
// three normals from four uniforms (0,1] of Philox calls 0 and 1 of stream i.
template <typename V>
__global__ __launch_bounds__(kBlock) void k_init(DevState<V> s, const CondParams* conds, int nCond,
                                                 int64_t totalMain, const int64_t* mainBase,
                                                 const double* thermalDev) {
    int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (g >= totalMain) return;
    int lo = 0, hi = nCond - 1;  // condition whose main range holds g
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (mainBase[mid] <= g) lo = mid; else hi = mid - 1;
    }
    const int c = lo;
    const CondParams& cp = conds[c];
    int64_t i = g - mainBase[c];
    int64_t slot = cp.base + i;
    uint32_t w[4], w2[4];
    philox_call(cp.seed, (uint64_t)i, 0, P_INIT, 0, w);
    philox_call(cp.seed, (uint64_t)i, 0, P_INIT, 1, w2);
    const double k = 1.0 / 9007199254740992.0;
    double r1 = ((double)(((((uint64_t)w[0]) << 32) | w[1]) >> 11) + 1.0) * k;
    double r2 = ((double)(((((uint64_t)w[2]) << 32) | w[3]) >> 11) + 1.0) * k;
    double r3 = ((double)(((((uint64_t)w2[0]) << 32) | w2[1]) >> 11) + 1.0) * k;
    double r4 = ((double)(((((uint64_t)w2[2]) << 32) | w2[3]) >> 11) + 1.0) * k;
    double aux1 = sqrt(-2.0 * log(r1)), aux2 = 2.0 * kPi * r2;
    double n0 = aux1 * cos(aux2), n1 = aux1 * sin(aux2), n2 = sqrt(-2.0 * log(r3)) * cos(2.0 * kPi * r4);
    double dev = thermalDev[c];
    Electron<V> e;
    e.x = 0; e.y = 0; e.z = 0; e.t = 0;
    e.vx = (V)(n0 * dev); e.vy = (V)(n1 * dev); e.vz = (V)(n2 * dev);
    e.eps = 0;
    e.tfree = (V)kNonDef;
    e.nue = (V)cp.trial;
    e.stream = (uint64_t)i;
    e.event = 0;
    store_rec(s, slot, e);
    s.alive[slot] = 1;
}

// ----------------------------------------------------- newborn refill
// After a chunk's electrons are at t_sync (or after removals): surviving
// newborns of the chunk's region, in region order, fill the chunk's holes in
// hole-list order; the rest move to the front of the region.  Wave-level, in
// groups of 64 newborns: every lane loads its record before any lane stores
// (each store waits on the group's loads), sources are cleared before
// destinations are set, and destinations never lie beyond the group.
template <typename V>
__device__ void wave_refill(const DevState<V>& s, uint32_t* holeList, const Chunk& ch, int& holes, int nNew,
                            int& remaining) {
    const int lane = lane_id();
    int used = 0;
    for (int b = 0; b < nNew; b += kWave) {
        const int j = b + lane;
        const bool al = j < nNew && s.alive[ch.region + j] != 0;
        const uint64_t am = __ballot(al);
        const int r = used + lane_rank(am);
        int64_t dst = -1;
        if (al) {
            if (r < holes) dst = holeList[ch.first + r];
            else if (r - holes != j) dst = ch.region + (r - holes);
        }
        if (dst >= 0) {
            const Rec<V> q = rec_get(s, ch.region + j);
            rec_put(s, dst, q);
            s.alive[ch.region + j] = 0;
        }
        __builtin_amdgcn_wave_barrier();
        if (dst >= 0) s.alive[dst] = 1;
        used += __popcll(am);
    }
    const int filled = used < holes ? used : holes;
    for (int b = filled; filled > 0 && b < holes; b += kWave) {  // remaining holes to the list front
        const int h = b + lane;
        uint32_t v = 0;
        if (h < holes) v = holeList[ch.first + h];
        __builtin_amdgcn_wave_barrier();
        if (h < holes) holeList[ch.first + h - filled] = v;
    }
    holes -= filled;
    remaining = used - filled;
}

// ------------------------------------------------------------- histograms
// One electron into the histograms of condition c (getTimeDependDistributions,
// BoltzmannMC.C:1551-1571; MathFunctions::histogramCount/histogram2DCount,
// MathFunctions.C:61-81,106-127): the EEDF into `lhist` (LDS, flushed later)
// or directly into HBM (phase row `row`, or -1), the EADF and EVDF into HBM
// when `cyl`.  The per-condition values are read once per chunk by the caller.
// Histogram modes of a flight launch, fixed per launch so that the paths a
// launch cannot take are not compiled into it: the EEDF in LDS and no
// cylindrically symmetric condition, the EEDF in LDS and EADF/EVDF in HBM,
// or everything in HBM.
enum HistMode { HIST_LDS = 0, HIST_LDS_CYL = 1, HIST_HBM = 2 };

template <typename V, int HIST>
__device__ __forceinline__ void hist_count(const DevHist& h, int c, const double* g, const Electron<V>& e,
                                           uint32_t* lhist, int row, bool cyl) {
    const double en = (double)e.eps;
    const int cell = (int)(en / g[0]);
    if (cell >= 0 && cell < h.nCells) {
        if (HIST != HIST_HBM) lds_add_u32(lhist + (cell >> 1), (cell & 1) ? 0x10000u : 1u);
        else {
            atomicAdd(&h.eedf[(size_t)c * h.nCells + cell], 1ull);
            if (row >= 0 && h.eedfPer) atomicAdd(&h.eedfPer[((size_t)c * h.nPhases + row) * h.nCells + cell], 1ull);
        }
    }
    if (HIST != HIST_LDS && cyl) {
        const double vx = e.vx, vy = e.vy, vz = e.vz;
        const double cosA = vz / sqrt(vx * vx + vy * vy + vz * vz);
        const int cy = (int)((cosA + 1.0) / g[1]);
        if (cell < h.nCells && cell >= 0 && cy < h.nCos && cy >= 0)
            atomicAdd(&h.eadf[((size_t)c * h.nCells + cell) * h.nCos + cy], 1ull);
        const int rx = (int)(sqrt(vx * vx + vy * vy) / g[2]);
        const int az = (int)((vz + g[4]) / g[3]);
        if (rx < h.nRad && rx >= 0 && az < h.nAx && az >= 0)
            atomicAdd(&h.evdf[((size_t)c * h.nRad + rx) * h.nAx + az], 1ull);
    }
}

// --------------------------------------------------------------- advance
// One chunk: every main electron and every newborn flies to t_sync (the
// passes of BoltzmannMC.C:630-681 for this set of electrons).
template <typename V, int FC, bool THERMAL, int HIST>
__device__ __forceinline__ void advance_chunk(const DevState<V>& s, const DevWork& w, const DevProcesses& pr,
                                              const V* tables, const DevHist& h, const CondParams* conds, int cid,
                                              unsigned long long* cnt, lds_uint4* ring, bool lines) {
    const int lane = lane_id();
    const int P = pr.P;
    long long* gainL = (long long*)(cnt + P);
    long long* lossL = gainL + P;
    const Chunk ch = w.chunks[cid];
    const int c = ch.cond;
    const CondParams cp = conds[c];
    const int64_t I = cp.I;
    const V* cumul = tables + cp.tableOffset;
    const V* interp = cumul + I * P;
    const V* nutot = interp + I * P;
    double* hg = (double*)(cnt + 3 * P);
    V* envHi = (V*)(hg + 8);
    V* envLo = envHi + kEnvBins;
    uint32_t* lhist = (uint32_t*)(envLo + kEnvBins);
    for (int i = lane; i < 3 * P; i += kWave) ((long long*)cnt)[i] = 0;
    for (int i = lane; i < 2 * kEnvBins; i += kWave) envHi[i] = nutot[I + i];
    // histograms of the sampled state (the state this interval starts from),
    // counted as main electrons are loaded (fill flag 2 of the condition);
    // the condition's grid is copied to LDS
    if (lane < 6) hg[lane] = h.grid[6 * (size_t)c + lane];
    const bool histOn = h.grid[6 * (size_t)c + 5] == 2.0;
    const bool histLds = HIST != HIST_HBM && histOn;
    const int histRow = histOn ? h.phaseRow[c] : -1;
    const bool histCyl = HIST != HIST_LDS && histOn && h.eadf && h.cyl[c] != 0;
    if (histLds)
        for (int i = lane; i < (h.nCells + 1) / 2; i += kWave) lhist[i] = 0;
    wave_lds_sync();

    // two record pieces per ring load, except with the cylindrical histograms
    // counted at load: six VGPRs more there (mixed 130 -> 136 in DC, but AC+B 164 -> 170,
    // past the 168 of three waves per SIMD), for no gain where they fit: flight
    // kernel per interval, pairs against single pieces, one condition of 1e5 electrons
    // in FP64 67.7 / 67.5 us, eight of 1e5 150.5 / 150.0, 24 AC conditions of 2e5
    // 664 / 664
    constexpr bool kPairFill = HIST != HIST_LDS_CYL;
    const int count = ch.count;
    int nextMain = 0, nq = 0, nextNew = 0, holes = 0;
    int loaded = 0;  // main records whose ring loads are issued
    int landed = 0;  // ring fills known to have landed
    constexpr bool kLines = !split_record<V>() && !THERMAL;
    constexpr int kAhead = (ring_segs<V>() - 1) * kRingSeg;
    for (; loaded < count && loaded <= nextMain + kAhead; loaded += kRingSeg)
        ring_fill<V, kPairFill>(s, ch.first, count, loaded, ring);
    Electron<V> e;
    bool have = false, isNew = false, parked = false;
    int64_t slot = 0;
    uint32_t c0[4] = {0, 0, 0, 0};  // call 0 of a parked electron's event
    uint32_t iter = 0, nNull = 0, nReal = 0, nEsc = 0, status = 0;
    double fieldGain = 0, maxE = 0;
    while (true) {
        // lanes without an electron take the next main electron, then newborns
        // (every main slot holds an alive electron after population control)
        const uint64_t need = __ballot(!have);
        if (need) {
            const int nNeed = __popcll(need);
            const int availMain = (loaded < count ? loaded : count) - nextMain;
            const int takeMain = availMain < nNeed ? availMain : nNeed;
            const int availNew = nq - nextNew;
            const int takeNew = (nNeed - takeMain) < availNew ? (nNeed - takeMain) : availNew;
            if (takeMain > 0) {
                // main records [nextMain, nextMain + takeMain): the youngest
                // fill they need, and the fills issued after it
                const int need = (nextMain + takeMain - 1) / kRingSeg;
                if (need >= landed) {
                    ring_wait<V, kPairFill>(loaded / kRingSeg - 1 - need);
                    landed = need + 1;
                }
            }
            if (!have) {
                const int r = lane_rank(need);
                if (r < takeMain) {
                    slot = ch.first + nextMain + r;
                    isNew = false;
                    have = true;
                } else if (r - takeMain < takeNew) {
                    slot = ch.region + nextNew + (r - takeMain);
                    isNew = true;
                    have = true;
                }
                if (have) {
                    if (isNew) {
                        load_rec(s, slot, e);
                    } else {
                        const int idx = (int)(slot - ch.first);
                        ring_read<V>(ring_segment<V>(ring, idx), idx % kRingSeg, e);
                    }
                    iter = 0;
                    if (histOn && !isNew) hist_count<V, HIST>(h, c, hg, e, lhist, histRow, histCyl);
                }
            }
            nextMain += takeMain;
            nextNew += takeNew;
        }
        const uint64_t live = __ballot(have);
        if (live == 0) break;
        // refill the ring segments this step's lanes emptied, two or more at a
        // time, before the flights: every wait for a table load also waits for
        // the ring fills issued before it (a wave's vector memory operations
        // complete in order), so fewer, larger and earlier fills leave fewer
        // steps waiting on HBM latency (flight kernel per interval on the
        // 64-condition scan, mixed / FP64: 3 and 2 segments filled one at a
        // time at the end of a step 0.964 / 1.613 ms, 4 segments two at a time
        // 0.936 / 1.526 ms, the same filled before the flights 0.920 ms mixed)
        if (loaded + kRingSeg <= nextMain + kAhead)
            for (; loaded < count && loaded <= nextMain + kAhead; loaded += kRingSeg)
                ring_fill<V, kPairFill>(s, ch.first, count, loaded, ring);

        bool done = false, dead = false, spawn = false;
        CollOut<V> o;
        o.pid = -1;
        // phase A: flight, and the null test of the cold branch; a lane whose
        // event is a null collision flies on in the same step, up to null_run<V>()
        // events (the draws are keyed by the event, so the run length changes
        // no trajectory).  A lane at t_sync is done without a step: step_a leaves it as
        // it is, but asked here the answer joins the mask of the lanes that fly and
        // is no branch of its own inside (flight kernel per interval, a branch in step_a
        // against this: 64-condition scan in mixed precision 913 -> 896 us, one
        // condition of 3e7 electrons 1269 -> 1247, in FP64 2133 -> 2112; 899, 1252
        // and 2109 without the question)
        bool fly = have && !parked && e.t != cp.tsync;
        done = have && !parked && !fly;
#pragma unroll
        for (int run = 0; run < null_run<V>(); ++run) {
            if (run > 0) {
                const bool idle = fly && e.t == cp.tsync;
                done = done || idle;
                fly = fly && !idle;
            }
            if (!fly) continue;
            double gain;
            bool escape;
            EventRng<V> rng(cp.seed, e.stream, e.event);
            const int st = step_a<V, FC, THERMAL>(cp, pr, nutot, envHi, envLo, e, rng, escape, gain);
            fieldGain += gain;
            const bool bad = st != STEP_DONE && (!isfinite(e.t) || !isfinite((double)e.eps));
            status |= bad ? (uint32_t)ST_NONFINITE : 0u;
            e.t = bad ? cp.tsync : e.t;
            nEsc += escape && !bad ? 1u : 0u;
            c0[0] = rng.w0[0]; c0[1] = rng.w0[1]; c0[2] = rng.w0[2]; c0[3] = rng.w0[3];
            done = st == STEP_DONE || bad;
            parked = st == STEP_REAL && !bad;
            fly = st == STEP_NULL && !bad;
            if (fly) {
                ++nNull;
                after_event(cp, e);
                if (++iter >= kMaxLoopPerSync) {
                    status |= ST_LOOP_CAP;
                    done = true;
                    fly = false;
                }
            }
        }
        // phase B: real collisions, once enough lanes wait for one (or all do)
        const uint64_t pk = __ballot(parked);
        if (pk && (__popcll(pk) >= pr.parkLanes || pk == (live & ~__ballot(done)))) {
            if (parked) {
                EventRng<V> rng(cp.seed, e.stream, e.event, c0);
                step_b<V, THERMAL>(cp, pr, cumul, interp, nutot + I + 2 * kEnvBins, e, rng, o);
                status |= o.flags;
                if (o.pid < 0) {
                    ++nNull;
                } else {
                    ++nReal;
                    atomicAdd(&cnt[o.pid], 1ull);
                    const long long fx = __double2ll_rn(o.dE * kFix);
                    if (o.dE >= 0) atomicAdd((unsigned long long*)&gainL[o.pid], (unsigned long long)fx);
                    else atomicAdd((unsigned long long*)&lossL[o.pid], (unsigned long long)fx);
                    const int type = pr.proc[o.pid].type;
                    if (type == 1) spawn = true;
                    else if (type == 2) { done = true; dead = true; }
                }
                after_event(cp, e);
                parked = false;
                if (++iter >= kMaxLoopPerSync) { status |= ST_LOOP_CAP; done = true; }
            }
        }
        // ejected electrons join the chunk's newborn queue, in lane order
        const uint64_t sp = __ballot(spawn);
        if (sp) {
            if (spawn) {
                const int idx = nq + lane_rank(sp);
                if (idx < ch.regionCap) {
                    Electron<V> n;
                    n.x = e.x; n.y = e.y; n.z = e.z; n.t = e.t;
                    n.vx = o.ejv[0]; n.vy = o.ejv[1]; n.vz = o.ejv[2]; n.eps = o.ejEps;
                    n.tfree = (V)kNonDef; n.nue = (V)cp.trial;
                    n.stream = child_stream(cp.seed, e.stream, e.event - 1);
                    n.event = 0;
                    store_rec(s, ch.region + idx, n);
                    s.alive[ch.region + idx] = 1;
                } else {
                    status |= ST_REGION_OVERFLOW;
                }
            }
            const int tot = nq + __popcll(sp);
            nq = tot < ch.regionCap ? tot : ch.regionCap;
        }
        // finished electrons: store, or leave a hole in the chunk's list
        const uint64_t dm = __ballot(done && dead && !isNew);
        if (kLines && lines) store_recs(s, done && !dead, slot, e);
        if (done) {
            if (dead) {
                s.alive[slot] = 0;
                if (!isNew) w.holeList[ch.first + holes + lane_rank(dm)] = (uint32_t)slot;
            } else {
                if (!(kLines && lines)) store_rec(s, slot, e);
                maxE = fmax(maxE, (double)e.eps);
            }
            have = false;
        }
        holes += __popcll(dm);
    }

    int remaining = 0;
    wave_refill<V>(s, w.holeList, ch, holes, nq, remaining);

    const double fg = wave_sum(fieldGain);
    const double mx = wave_max(maxE);
    const uint32_t nn = wave_sum_u(nNull), nr = wave_sum_u(nReal), ne = wave_sum_u(nEsc);
    const uint32_t stw = wave_or(status);
    if (lane == 0) {
        w.holesC[cid] = holes;
        w.surplusC[cid] = remaining;
        if (holes) atomicAdd(&pop_mine(w, c).holes, (uint32_t)holes);
        if (remaining) atomicAdd(&pop_mine(w, c).surplus, (uint32_t)remaining);
        double* t = w.tailC + (size_t)cid * CT_SIZE;
        t[CT_FIELD] = fg;
        t[CT_NULL] = (double)nn;
        t[CT_REAL] = (double)nr;
        t[CT_EVENTS] = (double)nn + (double)nr;
        t[CT_ESCAPE] = (double)ne;
        t[CT_MAXE] = mx;
        t[CT_GROWTH] = 0;
        t[CT_PAD] = 0;
        if (stw) atomicOr(&w.status[c], stw);
    }
    wave_lds_sync();
    for (int p = lane; p < P; p += kWave) {
        const unsigned long long n = cnt[p];
        if (n) {
            atomicAdd(&w.accCount[(size_t)c * P + p], n);
            const long long gq = gainL[p], lq = lossL[p];
            if (gq) atomicAdd((unsigned long long*)&w.accGain[(size_t)c * P + p], (unsigned long long)gq);
            if (lq) atomicAdd((unsigned long long*)&w.accLoss[(size_t)c * P + p], (unsigned long long)lq);
        }
    }
    if (histLds) {
        const int row = h.phaseRow[c];
        for (int i = lane; i < h.nCells; i += kWave) {
            const uint32_t n = (lhist[i >> 1] >> ((i & 1) * 16)) & 0xffffu;
            if (!n) continue;
            atomicAdd(&h.eedf[(size_t)c * h.nCells + i], (unsigned long long)n);
            if (row >= 0 && h.eedfPer)
                atomicAdd(&h.eedfPer[((size_t)c * h.nPhases + row) * h.nCells + i], (unsigned long long)n);
        }
    }
    wave_lds_sync();
}

// Waves per SIMD the flight kernel is compiled for.  FP64: two (172-210 VGPRs;
// its record rings leave the LDS room for two blocks per CU anyway).  Mixed form:
// the compiler's choice (130-168 VGPRs, three waves; two for AC+B off resonance with
// thermal targets and no cylindrical condition, at 173).  More waves do not make
// either faster: with a ring of 80 records and an FP32 envelope, so that the LDS
// held them, one condition of 3e7 electrons took 2416 us per interval with three
// FP64 waves against 2354 with two, and 1515 with four mixed waves against 1389
// with three.
template <typename V, int FC> constexpr int flight_waves_per_eu() { return sizeof(V) == 8 ? 2 : 1; }

// Flight kernel of one field case.  The work list has one part per XCD
// (kXcds contiguous parts of about equal work; blocks go to the XCDs in turn):
// chunks of one condition then run on one XCD, or on neighbouring ones, at about
// the same time, and its tables and cylindrical histograms stay in that XCD's
// L2.  Where the grid has a wave for every chunk a wave takes the chunk of its
// place; otherwise waves take chunks of their XCD's part through an atomic
// counter, then of the other parts, until the list is exhausted.  (Flight kernel per
// interval, one queue for all XCDs against this: 8 conditions of 1e5 with EADF
// and EVDF 146 -> 126 us, one condition of 9.5e5 in FP64 155 -> 148 us, 24 AC
// conditions of 2e5 557 -> 523 us; no difference for the 64-condition scan.)
template <typename V, int FC, bool THERMAL, int HIST>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(flight_waves_per_eu<V, FC>()))) void k_advance(DevState<V> s, DevWork w, const CondParams* conds, DevProcesses pr, const V* tables,
                                                    DevHist h, FlightList fl, uint32_t* queue) {
    extern __shared__ unsigned char smem[];
    constexpr int kRingWave = ring_segs<V>() * rec_pieces<V>() * kRingSeg;  // 16-byte pieces per wave
    __shared__ uint4 rings[kWavesPerBlock * kRingWave];
    const int wid = threadIdx.x / kWave;
    // the process records in LDS: a collision reads its process's constants
    // at LDS latency, outside the in-order queue of the ring loads
    uint4* procL = (uint4*)smem;
    for (int i = threadIdx.x; i < pr.P * (int)(sizeof(ProcRec) / 16); i += kBlock)
        procL[i] = ((const uint4*)pr.proc)[i];
    // The interval's parameters are read where the host wrote them, and written to
    // w.conds for the kernels that follow; k_finish writes the summaries to host
    // memory in turn.  A copy either way cost a launch and its gap: passes of one
    // condition of 1e4 electrons (64 intervals) 5.90 -> 5.47 ms, of 1e5 in FP64 7.99 ->
    // 7.52, of 9.5e5 (32) 6.40 -> 6.17; no difference for 1.6e7 electrons and more.
    static_assert(sizeof(CondParams) % 8 == 0, "whole words");
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < w.nCond * (int)(sizeof(CondParams) / 8); i += gridDim.x * kBlock)
        ((uint64_t*)(w.conds + w.cond0))[i] = ((const uint64_t*)(conds + w.cond0))[i];
    __syncthreads();
    DevProcesses prl = pr;
    prl.proc = (const ProcRec*)smem;
    unsigned long long* cnt =
        (unsigned long long*)(smem + (size_t)pr.P * sizeof(ProcRec) + (size_t)wid * flight_wave_lds<V>(pr.P, h.histLds));
    lds_uint4* ring = (lds_uint4*)(rings + wid * kRingWave);
    const int xcd = blockIdx.x % kXcds;
    int x = xcd;
    while (true) {  // one call of advance_chunk: two would be inlined twice (174 VGPRs)
        uint32_t item = (blockIdx.x / kXcds) * kWavesPerBlock + wid;
        if (!fl.oneShot && lane_id() == 0) item = atomicAdd(&queue[x * kQueueStride], 1u);
        item = (uint32_t)__builtin_amdgcn_readfirstlane((int)item) + (uint32_t)fl.part[x];
        if (item >= (uint32_t)fl.part[x + 1]) {
            x = x + 1 < kXcds ? x + 1 : 0;
            if (fl.oneShot || x == xcd) break;
            continue;
        }
        advance_chunk<V, FC, THERMAL, HIST>(s, w, prl, tables, h, conds, fl.list[item], cnt, ring, !fl.oneShot);
        if (fl.oneShot) break;
    }
}

// ------------------------------------------------------ population control
// Four kernels after the flights bring every condition back to N electrons
// and sample it: k_marks and k_apply_marks remove surplus electrons, k_settle
// moves and clones electrons into holes and samples, k_finish reduces.  What
// bounds them at ordinary sizes is latency: a kernel starts with cold L2s, so
// each load that depends on another costs about 0.7 us, and a kernel that
// does nothing about 2.5 us.  So what a planning kernel of one block per
// condition would compute is taken from totals the waves add up (the removals),
// or worked out again by every wave or block that needs it (offsets, removal
// threshold) while it has little else to do.  One kernel for everything with
// the last block of a condition planning was slower: handing values between
// blocks of one launch costs more than a launch (12 us against 7 us for the
// marks of one condition of 1e4 electrons).  Measured, all kernels after the
// flights, against ten launches with planning kernels between them: one
// condition of 1e4 electrons 55 -> 27 us, of 1e5 60 -> 36 us, the 64-condition
// scan 322 -> 277 us.

// The population of a condition after its flights: M alive, and the removals
// that bring it back to N.
__device__ __forceinline__ PopPlan plan_of(const CondPop& pop, const CondParams& cp) {
    const int64_t H = pop.holes, S = pop.surplus;
    PopPlan pl = {};
    pl.alive = cp.nMain - H + S;
    pl.remove = S > H ? S - H : 0;
    const double R = (double)pl.remove;
    pl.markProb = pl.remove > 0 ? fmin(1.0, (R + 8.0 * sqrt(R) + 20.0) / (double)pl.alive) : 0.0;
    return pl;
}

// Bernoulli(p) marks over a chunk's candidates [0, L): main slots
// [0, count) (holes are not alive and never count) and the surplus
// newborns [count, L).  Lane l draws geometric skips over its segment
// [l L / 64, (l+1) L / 64) with Philox keyed by (chunk, lane, interval).
struct MarkGen {
    uint64_t seed, key;
    uint32_t sync, call;
    double logq;
    bool all;
    int64_t pos, hi;
    uint32_t w[4];
    __device__ MarkGen(const CondParams& cp, const Chunk& ch, int lane, double p, int64_t L) {
        seed = cp.seed;
        key = ((uint64_t)(uint32_t)lane << 32) | (uint32_t)ch.local;
        sync = (uint32_t)cp.syncIndex;
        call = 0;
        all = !(p < 1.0);
        logq = all ? -1.0 : log1p(-p);
        pos = (int64_t)lane * L / kWave - 1;
        hi = (int64_t)(lane + 1) * L / kWave;
    }
    __device__ bool next() {
        if (all) return ++pos < hi;
        const bool h = (call & 1) != 0;
        if (!h) philox_call(seed, key, sync, P_POPCTL, call >> 1, w);
        ++call;
        const uint32_t hiw = h ? w[2] : w[0], low = h ? w[3] : w[1];
        const uint64_t x = ((((uint64_t)hiw) << 32) | low) >> 11;
        const double u = ((double)x + 1.0) * (1.0 / 9007199254740992.0);  // (0,1]
        const double skip = floor(log(u) / logq);
        if (!(skip < (double)(hi - pos - 1))) { pos = hi; return false; }
        pos += 1 + (int64_t)skip;
        return true;
    }
};

__device__ __forceinline__ bool mark_alive(const uint8_t* alive, const Chunk& ch, int64_t pos) {
    return pos >= ch.count || alive[ch.first + pos] != 0;
}

// A condition of at most kPlanDirect electrons has its removal threshold and
// its chunks' mark offsets worked out by every block of k_apply_marks: its
// few hundred marks cost a block less than the launch of k_plan_marks and the
// loads of its results.  Per interval, in the blocks against with k_plan_marks:
// one condition of 1e4 electrons 8.3 us against 6.1 + 6.9, one of 1e5 11.6
// against 6.4 + 6.5, eight of 1e5 at up to 500 Td (2 % newborns) 31 against
// 10.3 + 10.3.  It does not pay beside larger conditions, for which k_plan_marks is
// launched all the same: the 64-condition scan with half of its conditions planned in
// the blocks 67 + 18 against 30 + 17.
__host__ __device__ __forceinline__ bool plans_direct(const CondParams& cp) { return cp.nMain <= kPlanDirect; }

// The marks of each chunk of a condition with removals, counted per lane and
// added to the condition's total.
__global__ __launch_bounds__(kBlock) void k_marks(const uint8_t* alive, DevWork w) {
    const int lane = lane_id();
    const int cid = w.chunk0 + blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
    if (cid >= w.chunk0 + w.nChunks) return;
    const Chunk ch = w.chunks[cid];
    const int sur = w.surplusC[cid];
    const CondParams& cp = w.conds[ch.cond];
    if (!cp.active) return;
    const PopPlan pl = plan_of(pop_total(w, ch.cond), cp);
    if (pl.remove == 0) return;
    MarkGen g(cp, ch, lane, pl.markProb, (int64_t)ch.count + sur);
    uint32_t m = 0;
    while (g.next()) m += mark_alive(alive, ch, g.pos) ? 1u : 0u;
    w.laneMarks[(size_t)cid * kWave + lane] = (uint8_t)(m < 255u ? m : 255u);
    m = wave_sum_u(m);
    if (lane == 0) {
        w.markC[cid] = (int32_t)m;
        if (m && plans_direct(cp)) atomicAdd(&pop_mine(w, ch.cond).marks, m);
    }
}

// Key of the mark with condition-wide index j (uniform 32-bit word).
__device__ __forceinline__ uint32_t mark_key(const CondParams& cp, int64_t j) {
    uint32_t w[4];
    philox_call(cp.seed, (uint64_t)j, (uint32_t)cp.syncIndex, P_POPCTL,
                0x8000u | ((uint32_t)(cp.syncIndex >> 32) & 0x7fffu), w);
    return w[0];
}

constexpr int kTieCap = 1024;
constexpr int kNearCap = 2048;
struct PopLds {
    uint64_t near[kNearCap];  // (key, index) of the marks near the threshold
    uint32_t hist[256], ties[kTieCap];
    uint32_t sh[4];           // prefix, mask, need, tie count
    uint32_t below, nNear;
    int last;
};

// Key of the R-th smallest of K marks by a 4-pass, 8-bit radix select; ties
// on that key are ordered by index.  Sets the plan's threshold; false when it
// cannot.
__device__ bool radix_threshold(PopLds& L, const CondParams& cp, int64_t K, int64_t R, PopPlan& pl) {
    uint32_t* sh = L.sh;
    uint32_t* hist = L.hist;
    uint32_t* ties = L.ties;
    if (threadIdx.x == 0) { sh[0] = 0; sh[1] = 0; sh[2] = (uint32_t)R; sh[3] = 0; }
    __syncthreads();
    for (int pass = 0; pass < 4; ++pass) {
        const int shift = 24 - 8 * pass;
        for (int i = threadIdx.x; i < 256; i += blockDim.x) hist[i] = 0;
        __syncthreads();
        const uint32_t prefix = sh[0], mask = sh[1];
        for (int64_t j = threadIdx.x; j < K; j += blockDim.x) {
            const uint32_t k = mark_key(cp, j);
            if ((k & mask) == prefix) atomicAdd(&hist[(k >> shift) & 255u], 1u);
        }
        __syncthreads();
        if (threadIdx.x < kWave) {
            // the bucket holding the need-th smallest key: lane l scans
            // buckets [4l, 4l + 4) after an exclusive scan of the lane sums
            // (bucket 255 takes the rest, as a serial scan would)
            const int l = threadIdx.x;
            const uint32_t need = sh[2];
            uint32_t b[4], sum = 0;
            for (int q = 0; q < 4; ++q) { b[q] = hist[4 * l + q]; sum += b[q]; }
            uint32_t incl = sum;
            for (int o = 1; o < kWave; o <<= 1) {
                const uint32_t t = __shfl_up(incl, o, kWave);
                if (l >= o) incl += t;
            }
            uint32_t cum = incl - sum;
            int found = -1;
            uint32_t before = 0;
            for (int q = 0; q < 4; ++q) {
                const int bkt = 4 * l + q;
                if (found < 0 && (cum + b[q] >= need || bkt == 255)) { found = bkt; before = cum; }
                cum += b[q];
            }
            // the first lane with a bucket is the answer
            const uint64_t has = __ballot(found >= 0);
            const int first = __ffsll((long long)has) - 1;
            if (l == first) {
                sh[0] = prefix | ((uint32_t)found << shift);
                sh[1] = mask | (255u << shift);
                sh[2] = need - before;
            }
        }
        __syncthreads();
    }
    const uint32_t T = sh[0], need = sh[2];  // R-th smallest key; its rank among keys == T
    for (int64_t j = threadIdx.x; j < K; j += blockDim.x) {
        if (mark_key(cp, j) == T) {
            const uint32_t slot = atomicAdd(&sh[3], 1u);
            if (slot < kTieCap) ties[slot] = (uint32_t)j;
        }
    }
    __syncthreads();
    const uint32_t nt = sh[3];
    if (nt > kTieCap || need < 1 || need > nt) return false;
    // bitonic sort of the tied indices (padded to a power of two)
    int n2 = 1;
    while (n2 < (int)nt) n2 <<= 1;
    for (int i = threadIdx.x; i < n2; i += blockDim.x)
        if (i >= (int)nt) ties[i] = 0xffffffffu;
    __syncthreads();
    for (int k = 2; k <= n2; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = threadIdx.x; i < n2; i += blockDim.x) {
                int l = i ^ j;
                if (l > i) {
                    bool up = (i & k) == 0;
                    uint32_t a = ties[i], bb = ties[l];
                    if ((a > bb) == up) { ties[i] = bb; ties[l] = a; }
                }
            }
            __syncthreads();
        }
    }
    pl.thrKey = T;
    pl.thrIndex = ties[need - 1];
    return true;
}

// The removal threshold of a condition by one block: of the K marks, the R
// with the smallest (key, index) go, which is a uniform R-subset.  The keys
// are uniform 32-bit words, so the R-th smallest lies within a few standard
// deviations of 2^32 R / K: the marks below that window are counted and the few
// hundred inside it (the standard deviation of the count is sqrt(R (K - R) /
// K), K - R = 8 sqrt(R) + 20) ranked, in one pass over the keys.  A threshold
// outside the window (six standard deviations) takes the radix select, which
// needs five passes.  Every thread gets the plan's threshold, or the status.
__device__ void removal_threshold(const CondParams& cp, int64_t K, PopPlan& pl, PopLds& L) {
    const int64_t R = pl.remove;
    if (K < R || K > 0xffffffffLL) {
        pl.status |= ST_POPCTL;
        return;
    }
    __syncthreads();
    if (threadIdx.x == 0) { L.below = 0; L.nNear = 0; }
    __syncthreads();
    const double mid = 4294967296.0 * ((double)R / (double)K);
    const double half = 4294967296.0 / (double)K * (6.0 * sqrt((double)R * (double)(K - R) / (double)K) + 8.0);
    const uint32_t lo = (uint32_t)fmax(0.0, mid - half), hi = (uint32_t)fmin(4294967295.0, mid + half);
    uint32_t under = 0;
    for (int64_t j = threadIdx.x; j < K; j += blockDim.x) {
        const uint32_t k = mark_key(cp, j);
        if (k < lo) ++under;
        else if (k <= hi) {
            const uint32_t n = atomicAdd(&L.nNear, 1u);
            if (n < kNearCap) L.near[n] = ((uint64_t)k << 32) | (uint32_t)j;
        }
    }
    under = wave_sum_u(under);
    if (lane_id() == 0) atomicAdd(&L.below, under);
    __syncthreads();
    const int64_t need = R - (int64_t)L.below;  // rank of the threshold among the near marks
    const uint32_t nNear = L.nNear;
    if (need < 1 || need > (int64_t)nNear || nNear > kNearCap) {
        if (!radix_threshold(L, cp, K, R, pl)) pl.status |= ST_POPCTL;
        return;
    }
    for (uint32_t i = threadIdx.x; i < nNear; i += blockDim.x) {
        const uint64_t me = L.near[i];
        uint32_t rank = 1;
        for (uint32_t q = 0; q < nNear; ++q) rank += L.near[q] < me ? 1u : 0u;
        if (rank == (uint32_t)need) L.last = (int)i;
    }
    __syncthreads();
    const uint64_t thr = L.near[L.last];
    pl.thrKey = (uint32_t)(thr >> 32);
    pl.thrIndex = (int64_t)(uint32_t)thr;
}

// Mark offsets and removal threshold of the larger conditions, one block each.
// (512 threads: a block of 1024 found no place beside the other part's flights
// and waited for their tail; pass of the mixed 64-condition scan 16.25 -> 15.86 ms,
// of eight conditions of 1e5 7.00 -> 6.85; one condition 6.5 us either way.)
constexpr int kPlanBlock = 512;
__global__ __launch_bounds__(kPlanBlock) void k_plan_marks(DevWork w) {
    __shared__ int64_t lds[2 * kWave + 1];
    __shared__ PopLds L;
    const int c = w.cond0 + blockIdx.x;
    const CondParams cp = w.conds[c];
    if (!cp.active || plans_direct(cp)) return;
    PopPlan pl = plan_of(pop_total(w, c), cp);
    if (pl.remove == 0) return;
    const int64_t K = block_exclusive_scan(w.markC + cp.chunkBegin, w.markOff + cp.chunkBegin, cp.nChunks, lds);
    removal_threshold(cp, K, pl, L);
    if (threadIdx.x == 0) w.plans[c] = pl;
}

// Marks in chunk order, then lane order, then position order; a mark at or
// below the threshold is removed.  Removed main electrons become holes of the
// chunk, then the chunk refills them from its newborns.
template <typename V>
__device__ __forceinline__ void apply_marks(const DevState<V>& s, const DevWork& w, const Chunk& ch,
                                            const CondParams& cp, int cid, const PopPlan& pl, int sur, int holes,
                                            int mine, int64_t offset) {
    const int lane = lane_id();
    const int64_t L = (int64_t)ch.count + sur;
    if (__ballot(mine == 255)) {  // a count that did not fit its byte: count again
        mine = 0;
        MarkGen g(cp, ch, lane, pl.markProb, L);
        while (g.next()) mine += mark_alive(s.alive, ch, g.pos) ? 1 : 0;
    }
    int64_t gi = offset + wave_exclusive_scan(mine);
    double growth = 0;
    MarkGen g(cp, ch, lane, pl.markProb, L);
    int left = mine;  // marks of this lane not yet visited
    bool more = left > 0 && g.next();
    while (__ballot(more)) {
        bool kill = false, killMain = false;
        int64_t slot = 0;
        if (more && mark_alive(s.alive, ch, g.pos)) {
            const uint32_t k = mark_key(cp, gi);
            if (k < pl.thrKey || (k == pl.thrKey && gi <= pl.thrIndex)) {
                kill = true;
                killMain = g.pos < ch.count;
                slot = killMain ? ch.first + g.pos : ch.region + (g.pos - ch.count);
            }
            ++gi;
            --left;
        }
        const uint64_t km = __ballot(killMain);
        if (kill) {
            growth -= rec_energy(s.ra[slot]);
            s.alive[slot] = 0;
            if (killMain) w.holeList[ch.first + holes + lane_rank(km)] = (uint32_t)slot;
        }
        holes += __popcll(km);
        if (more) more = left > 0 && g.next();
    }
    int remaining = 0;
    wave_refill<V>(s, w.holeList, ch, holes, sur, remaining);
    const double gsum = wave_sum(growth);
    if (lane == 0) {
        w.holesC[cid] = holes;
        w.surplusC[cid] = remaining;
        if (holes) atomicAdd(&pop_mine(w, ch.cond).holesAfter, (uint32_t)holes);
        if (gsum != 0) w.tailC[(size_t)cid * CT_SIZE + CT_GROWTH] += gsum;
    }
}

template <typename V>
__global__ __launch_bounds__(kBlock) void k_apply_marks(DevState<V> s, DevWork w) {
    __shared__ PopLds L;
    __shared__ int conds[kWavesPerBlock];
    const int lane = lane_id(), wid = threadIdx.x / kWave;
    const int cid = w.chunk0 + blockIdx.x * kWavesPerBlock + wid;
    const bool in = cid < w.chunk0 + w.nChunks;
    Chunk ch = {};
    int c = -1, sur = 0, holes = 0, mine = 0;
    PopPlan pl = {};
    if (in) {
        ch = w.chunks[cid];
        sur = w.surplusC[cid];
        holes = w.holesC[cid];
        mine = w.laneMarks[(size_t)cid * kWave + lane];
        if (w.conds[ch.cond].active) {
            pl = plan_of(pop_total(w, ch.cond), w.conds[ch.cond]);
            if (pl.remove > 0) c = ch.cond;
        }
    }
    const bool direct = c >= 0 && plans_direct(w.conds[c]);
    if (lane == 0) conds[wid] = direct ? c : -1;
    __syncthreads();
    // thresholds of the block's conditions (one, but where a block ends one
    // condition and begins the next)
    for (int k = 0; k < kWavesPerBlock; ++k) {
        const int cc = conds[k];
        if (cc < 0 || (k > 0 && conds[k - 1] == cc)) continue;
        const CondPop pop = pop_total(w, cc);
        PopPlan q = plan_of(pop, w.conds[cc]);
        removal_threshold(w.conds[cc], pop.marks, q, L);
        if (c == cc) pl = q;
        __syncthreads();
    }
    if (c < 0) return;
    const CondParams& cp = w.conds[c];
    int64_t offset;
    if (direct) {
        uint32_t before = 0;
        for (int k = lane; k < ch.local; k += kWave) before += (uint32_t)w.markC[cp.chunkBegin + k];
        offset = wave_sum_u(before);
    } else {
        pl = w.plans[c];
        offset = w.markOff[cid];
    }
    if (pl.status & ST_POPCTL) {
        if (lane == 0) atomicOr(&w.status[c], (uint32_t)ST_POPCTL);
        return;
    }
    apply_marks<V>(s, w, ch, cp, cid, pl, sur, holes, mine, offset);
}

// Offsets of the holes and surplus newborns of the conditions with more than
// kPairsDirect chunks, one block each.  (k_settle finds the pairs of the
// others in the per-chunk counts.)
__global__ __launch_bounds__(1024) void k_plan_pairs(DevWork w) {
    __shared__ int64_t lds[2 * kWave + 1];
    const int c = w.cond0 + blockIdx.x;
    const CondParams cp = w.conds[c];
    if (!cp.active || cp.nChunks <= kPairsDirect) return;
    const CondPop pop = pop_total(w, c);
    if (pop.holes == 0 && pop.surplus == 0) return;
    block_exclusive_scan(w.holesC + cp.chunkBegin, w.holeOff + cp.chunkBegin, cp.nChunks, lds);
    block_exclusive_scan(w.surplusC + cp.chunkBegin, w.surOff + cp.chunkBegin, cp.nChunks, lds);
}

// Chunk and place within it of every lane's item i, over the per-chunk counts
// of a condition's n chunks (items are numbered in chunk order).  Tiles of 512
// counts, 8 per lane: a wave scan gives the lanes' offsets, a binary search
// over the lanes the lane, and its 8 counts the chunk.  Called by a whole wave;
// lanes without an item pass want = false.
__device__ __forceinline__ void wave_locate(const int32_t* counts, int n, int64_t i, bool want, int& chunk, int& place) {
    constexpr int E = 8;
    const int lane = lane_id();
    int64_t running = 0;
    chunk = 0;
    place = 0;
    for (int base = 0; base < n && __ballot(want); base += E * kWave) {
        int v[E], t = 0;
#pragma unroll
        for (int k = 0; k < E; ++k) {
            const int j = base + lane * E + k;
            v[k] = j < n ? counts[j] : 0;
            t += v[k];
        }
        const int first = wave_exclusive_scan(t);
        const int total = __shfl(first + t, kWave - 1, kWave);
        const bool here = want && i < running + total;
        int r = here ? (int)(i - running) : 0;
        int lo = 0;  // largest lane whose offset is at most r
#pragma unroll
        for (int step = kWave / 2; step > 0; step >>= 1)
            if (__shfl(first, lo + step, kWave) <= r) lo += step;
        r -= __shfl(first, lo, kWave);
        bool found = false;
#pragma unroll
        for (int k = 0; k < E; ++k) {
            const int m = __shfl(v[k], lo, kWave);
            if (here && !found) {
                if (r < m) { chunk = base + lo * E + k; place = r; found = true; }
                else r -= m;
            }
        }
        want = want && !here;
        running += total;
    }
}

// Item i of a condition's holes or surplus newborns: its chunk and place.
__device__ __forceinline__ void locate(const CondParams& cp, const int32_t* countC, const int64_t* offC, int64_t i,
                                       bool want, int& chunk, int& place) {
    if (cp.nChunks <= kPairsDirect) {
        wave_locate(countC + cp.chunkBegin, cp.nChunks, i, want, chunk, place);
    } else {
        const int64_t* off = offC + cp.chunkBegin;
        chunk = want ? (int)owner_of(off, cp.nChunks, i) : 0;
        place = want ? (int)(i - off[chunk]) : 0;
    }
}

// Index, over a condition's holes in chunk order, of the hole at main slot
// `slot` (the same in every lane).  Called by a whole wave.
__device__ int64_t hole_index(const DevWork& w, const CondParams& cp, int64_t slot) {
    // chunk sizes differ by at most one, the larger ones first
    const int64_t at = slot - cp.base, each = cp.nMain / cp.nChunks, more = cp.nMain % cp.nChunks;
    const int64_t big = more * (each + 1);
    const int j = (int)(at < big ? at / (each + 1) : more + (at - big) / each);
    const int lane = lane_id();
    const int64_t first = w.chunks[cp.chunkBegin + j].first;
    int place = 0;
    for (int k = lane; k < w.holesC[cp.chunkBegin + j]; k += kWave)
        if ((int64_t)w.holeList[first + k] == slot) place = k;
    uint32_t n = (uint32_t)place;  // one lane found it
    if (cp.nChunks <= kPairsDirect) {
        for (int k = lane; k < j; k += kWave) n += (uint32_t)w.holesC[cp.chunkBegin + k];
        return wave_sum_u(n);
    }
    return w.holeOff[cp.chunkBegin + j] + wave_sum_u(n);
}

// Sums over the wave of 26 values per lane, each in the order of a butterfly
// (wave_sum), transposed: a step halves the values a lane holds, so 32
// shuffles do what 26 butterflies need 156 for.  Lane l gets the sum of value
// wave_sums_field(l).
__device__ __forceinline__ int wave_sums_field(int lane) {
    return ((lane >> 5) & 1) * 16 + ((lane >> 4) & 1) * 8 + ((lane >> 3) & 1) * 4 + ((lane >> 2) & 1) * 2 + ((lane >> 1) & 1);
}
__device__ __forceinline__ double wave_sums(const double (&m)[kMomentRecord], int lane) {
    double a[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const double lo = m[k], hi = k + 16 < kMomentRecord - 1 ? m[k + 16] : 0.0;
        const bool up = lane & 32;
        a[k] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, 32, kWave);
    }
#pragma unroll
    for (int o = 16; o > 1; o >>= 1) {
        const bool up = lane & o;
#pragma unroll
        for (int k = 0; k < o / 2; ++k) {
            const double lo = a[k], hi = a[k + o / 2];
            a[k] = (up ? hi : lo) + __shfl_xor(up ? lo : hi, o, kWave);
        }
    }
    return a[0] + __shfl_xor(a[0], 1, kWave);
}

// ----------------------------------------------------------------- settle
// The last part of population control and the ensemble sums of one sampling
// instant, one wave per chunk.
//  - Pair i of a condition (the waves of its chunks stride over them): hole i
//    takes surplus newborn i while there are newborns; the remaining holes get
//    clones of uniformly drawn electrons (BoltzmannMC.C:1368-1371).
//  - FP64 sums (calculateMeanDataForSwarmParams, BoltzmannMC.C:1410-1482) of
//    the electrons the chunk holds and of those its wave put into holes: eps,
//    r, v, r r^T, r v^T, count, max eps.
// Both in one kernel, so that neither waits for the other: a slot filled here
// is flagged 2 or 3, by the interval's parity, and the wave that owns the slot
// neither reads its record nor changes its flag; flags of the interval before
// become 1.  (With a flag of 1 the flight kernel need store none for an
// electron that survives its interval: 23 us of it on the 64-condition scan.)
// On the 64-condition scan the record reads bound it (64 bytes of each
// electron at the card's copy rate); one condition of 1e4 electrons is bound by
// the chain of loads.
template <typename V>
__global__ __launch_bounds__(kBlock) void k_settle(DevState<V> s, DevWork w) {
    const int lane = lane_id();
    const int cid = w.chunk0 + blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
    if (cid >= w.chunk0 + w.nChunks) return;
    const Chunk me = w.chunks[cid];
    const CondParams& cp = w.conds[me.cond];
    if (!cp.active) return;
    const uint8_t filled = (uint8_t)(2 + (cp.syncIndex & 1));
    double m[kMomentRecord];
#pragma unroll
    for (int k = 0; k < kMomentRecord; ++k) m[k] = 0;
    auto add = [&](const RecA<V>& q) {
        const double r[3] = {q.x, q.y, q.z};
        const double v[3] = {(double)q.vx, (double)q.vy, (double)q.vz};
        const double e = rec_energy(q);
        m[0] += e;
        for (int a = 0; a < 3; ++a) { m[1 + a] += r[a]; m[4 + a] += v[a]; }
        for (int a = 0; a < 3; ++a)
            for (int bb = 0; bb < 3; ++bb) { m[7 + 3 * a + bb] += r[a] * r[bb]; m[16 + 3 * a + bb] += r[a] * v[bb]; }
        m[25] += 1;
        m[26] = fmax(m[26], e);
    };

    const CondPop pop = pop_total(w, me.cond);
    const bool removed = pop.surplus > pop.holes;  // then as many newborns as holes are left
    const int64_t H = removed ? pop.holesAfter : pop.holes, S = removed ? pop.holesAfter : pop.surplus;
    const int64_t stride = (int64_t)cp.nChunks * kWave;
    double growth = 0;
    uint32_t status = 0;
    for (int64_t i0 = (int64_t)me.local * kWave; i0 < H; i0 += stride) {
        const int64_t i = i0 + lane;
        const bool want = i < H, move = i < S;
        int hc, hp, sc, sp;
        locate(cp, w.holesC, w.holeOff, i, want, hc, hp);
        locate(cp, w.surplusC, w.surOff, i, move, sc, sp);
        int64_t src = -1;
        if (move) src = w.chunks[cp.chunkBegin + sc].region + sp;
        // uniform alive source by rejection over the main slots (BoltzmannMC.C:1368-1371);
        // draw k of hole i: counter {i, k >> 16, interval, clone | (k & 0xffff)},
        // so no two of the 2^20 draws share a counter (i < 2^32)
        bool seek = want && !move;
        for (uint32_t k = 0; k < (1u << 20) && __ballot(seek); ++k) {
            int64_t cand = 0;
            bool hole = false;
            if (seek) {
                const double u = u53(cp.seed, (uint64_t)(uint32_t)i | ((uint64_t)(k >> 16) << 32),
                                     (uint32_t)cp.syncIndex, P_CLONE, k & 0xffffu);
                cand = cp.base + (int64_t)fmin(floor(u * (double)cp.nMain), (double)(cp.nMain - 1));
                const uint8_t a = s.alive[cand];
                hole = a == 0 || a == filled;
                if (!hole) { src = cand; seek = false; }
            }
            // a hole is a source where a newborn takes it; its record is read
            // where the newborn is
            for (uint64_t hm = S > 0 ? __ballot(hole) : 0; hm; hm &= hm - 1) {
                const int l = __ffsll((unsigned long long)hm) - 1;
                const int64_t j = hole_index(w, cp, __shfl(cand, l, kWave));
                if (j >= S) continue;
                int nc, np;
                locate(cp, w.surplusC, w.surOff, j, lane == l, nc, np);
                if (lane == l) { src = w.chunks[cp.chunkBegin + nc].region + np; seek = false; }
            }
        }
        if (!want) continue;
        if (src < 0) { status |= ST_POPCTL; continue; }
        const int64_t dst = w.holeList[w.chunks[cp.chunkBegin + hc].first + hp];
        Rec<V> q = rec_get(s, src);
        if (move) {
            s.alive[src] = 0;
        } else {
            growth += rec_energy(q.a);
            uint32_t wds[4];
            philox_call(cp.seed ^ 0x5851F42D4C957F2Dull, draw_part(q).stream, (uint32_t)dst, P_CLONE,
                        (uint32_t)(cp.syncIndex & 0xffffu), wds);
            draw_part(q).stream = ((uint64_t)wds[1] << 32) | wds[0];
            draw_part(q).event = 0;
        }
        rec_put(s, dst, q);
        s.alive[dst] = filled;
        add(q.a);
    }

    // two records per lane in flight; each lane adds its records in slot order
    auto own = [&](const RecA<V>& q, uint8_t a, int64_t slot) {
        if (a == 0 || a == filled) return;  // a hole before the pairs
        add(q);
        if (a != 1) s.alive[slot] = 1;
    };
    int64_t k = lane;
    for (; k + kWave < me.count; k += 2 * kWave) {
        const RecA<V> q0 = s.ra[me.first + k], q1 = s.ra[me.first + k + kWave];
        const uint8_t a0 = s.alive[me.first + k], a1 = s.alive[me.first + k + kWave];
        own(q0, a0, me.first + k);
        own(q1, a1, me.first + k + kWave);
    }
    if (k < me.count) own(s.ra[me.first + k], s.alive[me.first + k], me.first + k);
    const double mx = wave_max(m[26]);
    m[26] = 0;
    const double sum = wave_sums(m, lane);
    const uint32_t st = wave_or(status);
    const double g = H > S ? wave_sum(growth) : 0.0;
    double* out = w.momC + (size_t)cid * kMomentRecord;
    const int f = wave_sums_field(lane);
    if ((lane & 1) == 0 && f < kMomentRecord - 1) out[f] = sum;
    if (lane == 1) out[kMomentRecord - 1] = mx;
    if (lane == 0) {
        if (st) atomicOr(&w.status[me.cond], st);
        if (g != 0) w.tailC[(size_t)cid * CT_SIZE + CT_GROWTH] += g;
    }
}

// Histograms of one sampling instant (getTimeDependDistributions,
// BoltzmannMC.C:1551-1571; MathFunctions::histogramCount/histogram2DCount,
// MathFunctions.C:61-81,106-127), added to integer accumulators.  One block
// per range of main slots of one condition; the EEDF is counted in LDS when
// it fits, else directly in HBM.
template <typename V>
__global__ __launch_bounds__(kBlock) void k_hist(DevState<V> s, const SlotRange* ranges, DevHist h, int ldsCells) {
    extern __shared__ unsigned char smem[];
    const SlotRange rg = ranges[blockIdx.x];
    const int c = rg.cond;
    const double* g = h.grid + 6 * (size_t)c;
    if (g[5] != 1.0) return;  // flag 2: counted by the flight kernel as it loads the state
    const bool useLds = ldsCells >= h.nCells;
    uint32_t* lhist = (uint32_t*)smem;
    if (useLds) {
        for (int i = threadIdx.x; i < h.nCells; i += kBlock) lhist[i] = 0;
        __syncthreads();
    }
    const double eStep = g[0], cStep = g[1], rStep = g[2], aStep = g[3], maxSpeed = g[4];
    const bool cyl = h.cyl[c] != 0 && h.eadf;
    const int row = h.phaseRow[c];
    for (int64_t k = threadIdx.x; k < rg.count; k += kBlock) {
        const RecA<V> q = s.ra[rg.first + k];
        const double e = rec_energy(q);
        const int cell = (int)(e / eStep);
        if (cell >= 0 && cell < h.nCells) {
            if (useLds) atomicAdd(&lhist[cell], 1u);
            else {
                atomicAdd(&h.eedf[(size_t)c * h.nCells + cell], 1ull);
                if (row >= 0 && h.eedfPer) atomicAdd(&h.eedfPer[((size_t)c * h.nPhases + row) * h.nCells + cell], 1ull);
            }
        }
        if (cyl) {
            const double vx = q.vx, vy = q.vy, vz = q.vz;
            const double cosA = vz / sqrt(vx * vx + vy * vy + vz * vz);
            const int cy = (int)((cosA + 1.0) / cStep);
            if (cell < h.nCells && cell >= 0 && cy < h.nCos && cy >= 0)
                atomicAdd(&h.eadf[((size_t)c * h.nCells + cell) * h.nCos + cy], 1ull);
            const int rx = (int)(sqrt(vx * vx + vy * vy) / rStep);
            const int az = (int)((vz + maxSpeed) / aStep);
            if (rx < h.nRad && rx >= 0 && az < h.nAx && az >= 0)
                atomicAdd(&h.evdf[((size_t)c * h.nRad + rx) * h.nAx + az], 1ull);
        }
        if (h.evdf3) {
            // cells of width 2 v_max / n3 from -v_max on each axis; floor, so
            // that a velocity below -v_max is not counted in the first cell
            const double inv = h.n3 / (2.0 * maxSpeed);
            const double fx = floor(((double)q.vx + maxSpeed) * inv), fy = floor(((double)q.vy + maxSpeed) * inv),
                         fz = floor(((double)q.vz + maxSpeed) * inv);
            if (fx >= 0 && fx < h.n3 && fy >= 0 && fy < h.n3 && fz >= 0 && fz < h.n3)
                atomicAdd(&h.evdf3[(((size_t)c * h.n3 + (size_t)fx) * h.n3 + (size_t)fy) * h.n3 + (size_t)fz], 1ull);
        }
    }
    if (!useLds) return;
    __syncthreads();
    for (int i = threadIdx.x; i < h.nCells; i += kBlock) {
        const uint32_t n = lhist[i];
        if (!n) continue;
        atomicAdd(&h.eedf[(size_t)c * h.nCells + i], (unsigned long long)n);
        if (row >= 0 && h.eedfPer)
            atomicAdd(&h.eedfPer[((size_t)c * h.nPhases + row) * h.nCells + i], (unsigned long long)n);
    }
}

// ----------------------------------------------------------------- finish
// summary[c] = [ event record (3P + 8) | moment sums (kMomentRecord) | status ]
// Chunk records are summed in a fixed order: thread (r, f) of a block adds
// field f of records r, r + kFinishRows, ... in order (neighbouring threads
// read neighbouring fields), then thread f adds the rows.  The integer
// accumulators are converted and cleared for the next interval, and block 0
// resets the flight-kernel work queues of the launch's part.
constexpr int kFinishFields = CT_SIZE + kMomentRecord;
constexpr int kFinishBlock = 1024;
constexpr int kFinishRows = kFinishBlock / (kFinishFields + 1);
// Sums (maxima for the two maximum fields) over the records [first, first + n)
// of a chunk-tail array and a moment array by one block; the result is valid
// in threads f < kFinishFields.  One thread per record with every field in
// registers and 35 wave reductions took 12.6 us for the 40 records of one
// condition of 1e4 electrons, this 5.2 us.
__device__ double finish_reduce(const double* tsrc, const double* msrc, size_t first, int n,
                                double (*red)[kFinishFields + 1]) {
    const int row = threadIdx.x / (kFinishFields + 1), f = threadIdx.x % (kFinishFields + 1);
    const bool isMax = f == CT_MAXE || f == kFinishFields - 1;
    if (row < kFinishRows && f < kFinishFields) {
        const double* src = f < CT_SIZE ? tsrc + first * CT_SIZE + f : msrc + first * kMomentRecord + (f - CT_SIZE);
        const int each = f < CT_SIZE ? CT_SIZE : kMomentRecord;
        double acc = 0;
#pragma unroll 8
        for (int k = row; k < n; k += kFinishRows) {
            const double v = src[(size_t)k * each];
            acc = isMax ? fmax(acc, v) : acc + v;
        }
        red[row][f] = acc;
    }
    __syncthreads();
    double tot = 0;
    if (threadIdx.x < kFinishFields) {
        const bool top = threadIdx.x == CT_MAXE || threadIdx.x == kFinishFields - 1;
        double part[4] = {0, 0, 0, 0};
#pragma unroll
        for (int r = 0; r < kFinishRows; ++r) {
            const double v = red[r][threadIdx.x];
            part[r & 3] = top ? fmax(part[r & 3], v) : part[r & 3] + v;
        }
        tot = top ? fmax(fmax(part[0], part[1]), fmax(part[2], part[3])) : (part[0] + part[1]) + (part[2] + part[3]);
    }
    return tot;
}

// First pass for conditions with many work units: group g's sums, in the
// record layout of the chunk tails and moments.
__global__ __launch_bounds__(kFinishBlock) void k_finish_group(DevWork w) {
    __shared__ double red[kFinishRows][kFinishFields + 1];
    const int g = w.group0 + blockIdx.x;
    if (!w.conds[w.groupCond[g]].active) return;
    const double tot = finish_reduce(w.tailC, w.momC, (size_t)w.groupFirst[g], w.groupCount[g], red);
    if (threadIdx.x < kFinishFields) {
        const int f = threadIdx.x;
        if (f < CT_SIZE) w.tailG[(size_t)g * CT_SIZE + f] = tot;
        else w.momG[(size_t)g * kMomentRecord + (f - CT_SIZE)] = tot;
    }
}

__global__ __launch_bounds__(kFinishBlock) void k_finish(DevWork w, int P) {
    __shared__ double red[kFinishRows][kFinishFields + 1];
    const int c = w.cond0 + blockIdx.x;
    if (blockIdx.x == 0)
        for (int k = threadIdx.x; k < kFlightClasses * kXcds; k += blockDim.x) w.queue[k * kQueueStride] = 0;
    const CondParams cp = w.conds[c];
    if (!cp.active) return;
    double* out = w.summary + (size_t)c * w.summarySize;
    const int R = w.recSize;
    // the work units themselves, or the sums of their reduction groups
    const double tot = w.nGroups ? finish_reduce(w.tailG, w.momG, (size_t)w.condGroup[c], w.condGroups[c], red)
                                 : finish_reduce(w.tailC, w.momC, (size_t)cp.chunkBegin, cp.nChunks, red);
    if (threadIdx.x < kFinishFields) {
        const int f = threadIdx.x;
        if (f < CT_SIZE) out[3 * P + f] = tot;
        else out[R + (f - CT_SIZE)] = tot;
    }
    for (int p = threadIdx.x; p < P; p += blockDim.x) {
        const size_t i = (size_t)c * P + p;
        out[p] = (double)w.accCount[i];
        out[P + p] = (double)w.accGain[i] / kFix;
        out[2 * P + p] = (double)w.accLoss[i] / kFix;
        w.accCount[i] = 0;
        w.accGain[i] = 0;
        w.accLoss[i] = 0;
    }
    if (threadIdx.x == 0) {
        out[R + kMomentRecord] = (double)w.status[c];
        for (int k = 0; k < kPopCopies; ++k) w.pop[(size_t)k * w.popStride + c] = CondPop{};
    }
}

// ----------------------------------------------------------------- tables
// Linear interpolation as gsl_interp_linear evaluates it: the interval is the
// last one with x[j] <= v (the last point belongs to the last interval), and
// y = y_j + (v - x_j)/dx*(y_{j+1} - y_j).
__device__ __forceinline__ double table_at(const double* x, const double* y, int n, double v) {
#pragma clang fp contract(off)
    int lo = 0, hi = n - 2;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (x[mid] <= v) lo = mid; else hi = mid - 1;
    }
    const double dx = x[lo + 1] - x[lo];
    return dx > 0.0 ? y[lo] + (v - x[lo]) / dx * (y[lo + 1] - y[lo]) : 0.0;
}

// Interpolated cross section x relative density of process p at `energy`
// (interpolateCrossSections, BoltzmannMC.C:571-609), FP64.
__device__ __forceinline__ double table_value(const DevTableSrc& a, int p, double energy) {
#pragma clang fp contract(off)
    const int b = a.srcBegin[p], n = a.srcEnd[p] - b;
    double value = 0;
    if (a.isSuper[p]) {
        // Klein-Rosseland: (g_i/g_f)(1 + E_th/u) sigma_if(u + E_th)
        if (energy > a.minE[p] && energy <= a.maxE[p]) {
            const double thr = a.thrPartner[p];
            value = a.statW[p] * (1.0 + thr / energy) * table_at(a.energy + b, a.sigma + b, n, energy + thr) *
                    a.relDens[p];
        }
    } else if (energy >= a.minE[p] && energy <= a.maxE[p]) {
        value = table_at(a.energy + b, a.sigma + b, n, energy) * a.relDens[p];
    }
    return value;
}

// Rows of a table block: every (row, process) value by its own thread into
// LDS, then each row's running sum in process order by one thread -- the
// arithmetic and order of the host FP64 build (BoltzmannMC.C:571-614).
// A block holds table_rows_per_block(P) rows.
inline __host__ __device__ int table_rows_per_block(int P) { return P >= kBlock ? 1 : kBlock / P; }
template <typename V>
__global__ __launch_bounds__(kBlock) void k_table_rows(DevTableSrc a, double N, double step, V* tables,
                                                       double* nutot64) {
#pragma clang fp contract(off)
    extern __shared__ double vals[];  // [rows * P]
    const int P = a.P, I = a.I;
    const int rows = table_rows_per_block(P);
    const int i0 = blockIdx.x * rows;
    V* cumul = tables;
    V* interp = tables + (size_t)I * P;
    V* nutot = interp + (size_t)I * P;
    V* gasSum = nutot + I + 2 * kEnvBins;
    for (int q = threadIdx.x; q < rows * P; q += kBlock) {
        const int i = i0 + q / P;
        if (i >= I) break;
        const double v = table_value(a, q % P, i * step);
        vals[q] = v;
        interp[(size_t)i0 * P + q] = (V)v;
    }
    __syncthreads();
    for (int r = threadIdx.x; r < rows; r += kBlock) {
        const int i = i0 + r;
        if (i >= I) break;
        double acc = 0;
        for (int p = 0; p < P; ++p) {
            acc += vals[r * P + p];
            cumul[(size_t)i * P + p] = (V)acc;
        }
        for (int g = 0; g < a.G; ++g) {
            const int L = a.gasFirst[g];
            const V below = L > 0 ? cumul[(size_t)i * P + L - 1] : (V)0;
            gasSum[(size_t)i * a.G + g] = cumul[(size_t)i * P + a.gasLast[g]] - below;
        }
        acc *= N * sqrt(i * step * 2.0 * kCharge / kMass);
        nutot[i] = (V)acc;
        nutot64[i] = acc;
    }
}

// Running maximum of the total collision frequency (BoltzmannMC.C:612-613):
// one block; each thread takes a contiguous segment.
__global__ __launch_bounds__(1024) void k_table_max(const double* nutot64, double* numax64, int I) {
    __shared__ double lds[1024];
    const int per = (I + 1023) / 1024;
    const int b = threadIdx.x * per, e = min(I, b + per);
    double m = 0;
    for (int i = b; i < e; ++i) m = fmax(m, nutot64[i]);
    lds[threadIdx.x] = m;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {  // inclusive max-scan of the segment maxima
        const double v = threadIdx.x >= o ? lds[threadIdx.x - o] : 0.0;
        __syncthreads();
        lds[threadIdx.x] = fmax(lds[threadIdx.x], v);
        __syncthreads();
    }
    double run = threadIdx.x > 0 ? lds[threadIdx.x - 1] : 0.0;
    for (int i = b; i < e; ++i) {
        run = fmax(nutot64[i], run);
        numax64[i] = run;
    }
}

// Null-test envelope: for bin b (rows b<<s .. (b+1)<<s, the last row being
// the partner of the bin's last interpolation), the largest and smallest
// total frequency, widened by a few ulp of V so that every interpolated value
// w1*a + w2*b of the bin's rows lies inside.
template <typename V> struct EnvMargin;
template <> struct EnvMargin<float> { static constexpr double up = 1.0 + 0x1p-20, down = 1.0 - 0x1p-20; };
template <> struct EnvMargin<double> { static constexpr double up = 1.0 + 0x1p-48, down = 1.0 - 0x1p-48; };

template <typename V>
__global__ __launch_bounds__(kEnvBins) void k_table_env(V* tables, int I, int P, int shift) {
    const V* nutot = tables + 2 * (size_t)I * P;
    V* envHi = tables + 2 * (size_t)I * P + I;
    V* envLo = envHi + kEnvBins;
    const int b = threadIdx.x;
    const int k0 = b << shift;
    if (k0 > I - 1) { envHi[b] = (V)0; envLo[b] = (V)0; return; }
    const int k1 = min(((b + 1) << shift), I - 1);
    V hi = nutot[k0], lo = nutot[k0];
    for (int k = k0 + 1; k <= k1; ++k) { hi = fmax(hi, nutot[k]); lo = fmin(lo, nutot[k]); }
    envHi[b] = (V)((double)hi * EnvMargin<V>::up);
    envLo[b] = (V)((double)lo * EnvMargin<V>::down);
}

template <typename V>
hipError_t launch_tables(const DevTableSrc& src, double N, double step, int envShift, V* tables, double* nutot64,
                         double* numax64, hipStream_t st) {
    const int rows = table_rows_per_block(src.P);
    hipLaunchKernelGGL(k_table_rows<V>, dim3((src.I + rows - 1) / rows), dim3(kBlock),
                       (size_t)rows * src.P * sizeof(double), st, src, N, step, tables, nutot64);
    hipLaunchKernelGGL(k_table_env<V>, dim3(1), dim3(kEnvBins), 0, st, tables, src.I, src.P, envShift);
    hipLaunchKernelGGL(k_table_max, dim3(1), dim3(1024), 0, st, nutot64, numax64, src.I);
    return hipGetLastError();
}

// ------------------------------------------------------- batch operators
template <typename V>
__global__ __launch_bounds__(kBlock) void k_op_accelerate(const CondParams* cond, int64_t n, const double* time,
                                                          const double* dt, double* pos, double* vel,
                                                          double* energy, double* gain) {
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const CondParams cp = *cond;
    Electron<V> e;
    e.x = pos[3 * i]; e.y = pos[3 * i + 1]; e.z = pos[3 * i + 2]; e.t = time[i];
    e.vx = (V)vel[3 * i]; e.vy = (V)vel[3 * i + 1]; e.vz = (V)vel[3 * i + 2];
    e.eps = energy_of(e.vx, e.vy, e.vz);
    double g = 0;
    flight<-1>(cp, e, dt[i], g);
    pos[3 * i] = e.x; pos[3 * i + 1] = e.y; pos[3 * i + 2] = e.z;
    vel[3 * i] = e.vx; vel[3 * i + 1] = e.vy; vel[3 * i + 2] = e.vz;
    energy[i] = e.eps;
    gain[i] = g;
}

template <typename V>
__global__ __launch_bounds__(kBlock) void k_op_collide(const CondParams* cond, DevProcesses pr, const V* tables,
                                                       int64_t n, double* vel, double* energy, const double* nue,
                                                       const double* variates, int32_t* pid, double* ejv,
                                                       double* eje, double* de) {
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const CondParams cp = *cond;
    const int64_t I = cp.I, P = pr.P;
    const V* cumul = tables + cp.tableOffset;
    const V* interp = cumul + I * P;
    const V* nutot = interp + I * P;
    Electron<V> e;
    e.x = e.y = e.z = e.t = 0;
    e.vx = (V)vel[3 * i]; e.vy = (V)vel[3 * i + 1]; e.vz = (V)vel[3 * i + 2];
    e.eps = (V)energy[i];
    e.nue = (V)nue[i];
    e.tfree = 0; e.stream = 0; e.event = 0;
    EventRng<V> rng(0, 0, 0, variates + (size_t)i * 11);
    CollOut<V> o;
    collide<V, true>(cp, pr, cumul, interp, nutot, e, rng, o);
    pid[i] = o.pid;
    vel[3 * i] = e.vx; vel[3 * i + 1] = e.vy; vel[3 * i + 2] = e.vz;
    energy[i] = e.eps;
    ejv[3 * i] = o.ejv[0]; ejv[3 * i + 1] = o.ejv[1]; ejv[3 * i + 2] = o.ejv[2];
    eje[i] = o.ejEps;
    de[i] = o.dE;
}

__global__ __launch_bounds__(kBlock) void k_op_philox(int64_t n, const uint32_t* ctr, const uint32_t* key, uint32_t* out) {
    int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    uint32_t c[4] = {ctr[4 * i], ctr[4 * i + 1], ctr[4 * i + 2], ctr[4 * i + 3]};
    philox10(c, key[2 * i], key[2 * i + 1]);
    for (int k = 0; k < 4; ++k) out[4 * i + k] = c[k];
}

// Whether kernels of two streams run at the same time: one waits for the other's
// word, for at most a millisecond or so (word[0] the signal, word[1] the answer).
constexpr int kBesidePolls = 1000;
__global__ void k_await(uint32_t* word) {
    for (int k = 0; k < kBesidePolls; ++k) {
        if (atomicAdd(&word[0], 0u) != 0) {
            word[1] = 1;
            return;
        }
        __builtin_amdgcn_s_sleep(16);
    }
}
__global__ void k_signal(uint32_t* word) { atomicExch(&word[0], 1u); }

// ------------------------------------------------------------- launchers
static inline unsigned chunk_grid(int nChunks) { return (unsigned)((nChunks + kWavesPerBlock - 1) / kWavesPerBlock); }
// Dynamic LDS of a flight-kernel block: the process records [P], then the
// per-wave areas.
template <typename V> static inline size_t flight_lds(int P, int histLds) {
    return (size_t)P * sizeof(ProcRec) + (size_t)kWavesPerBlock * flight_wave_lds<V>(P, histLds);
}

template <typename V>
hipError_t launch_init(const DevState<V>& s, const DevWork& w, int64_t totalMain, const int64_t* mainBase,
                       const double* thermalDev, KernelTimer* timer, hipStream_t st) {
    if (totalMain == 0) return hipSuccess;
    timer_start(timer, K_INIT, st);
    hipLaunchKernelGGL(k_init<V>, dim3(grid_of(totalMain)), dim3(kBlock), 0, st, s, w.conds, w.nCond, totalMain,
                       mainBase, thermalDev);
    timer_stop(timer, K_INIT, st);
    return hipGetLastError();
}

// Histogram mode of the flight launches of an engine: the EEDF in LDS when
// the engine counts it there, EADF/EVDF code only when a condition is
// cylindrically symmetric.
static inline int hist_mode(const DevHist& h) {
    if (h.histLds < h.nCells) return HIST_HBM;
    return h.eadf ? HIST_LDS_CYL : HIST_LDS;
}

template <typename V, int FC, bool TH>
static const void* flight_kernel(int hist) {
    if (hist == HIST_LDS) return (const void*)k_advance<V, FC, TH, HIST_LDS>;
    if (hist == HIST_LDS_CYL) return (const void*)k_advance<V, FC, TH, HIST_LDS_CYL>;
    return (const void*)k_advance<V, FC, TH, HIST_HBM>;
}

template <typename V, int FC, bool TH, int HIST>
static void launch_advance_hist(const DevState<V>& s, const DevWork& w, const CondParams* conds, const DevProcesses& pr, const V* tables,
                                const DevHist& h, const FlightLists& fl, hipStream_t st) {
    dim3 g(fl.grid[FC]), b(kBlock);
    const size_t lds = flight_lds<V>(pr.P, h.histLds);
    hipLaunchKernelGGL((k_advance<V, FC, TH, HIST>), g, b, lds, st, s, w, conds, pr, tables, h, fl.cls[FC],
                       w.queue + FC * kXcds * kQueueStride);
}

template <typename V, int FC, bool TH>
static void launch_advance_th(const DevState<V>& s, const DevWork& w, const CondParams* conds, const DevProcesses& pr, const V* tables,
                              const DevHist& h, const FlightLists& fl, hipStream_t st) {
    switch (hist_mode(h)) {
        case HIST_LDS: launch_advance_hist<V, FC, TH, HIST_LDS>(s, w, conds, pr, tables, h, fl, st); break;
        case HIST_LDS_CYL: launch_advance_hist<V, FC, TH, HIST_LDS_CYL>(s, w, conds, pr, tables, h, fl, st); break;
        default: launch_advance_hist<V, FC, TH, HIST_HBM>(s, w, conds, pr, tables, h, fl, st); break;
    }
}

template <typename V, int FC>
static void launch_advance_case(const DevState<V>& s, const DevWork& w, const CondParams* conds, const DevProcesses& pr, const V* tables,
                                const DevHist& h, const FlightLists& fl, hipStream_t st) {
    if (fl.grid[FC] == 0) return;
    if (pr.gasTempEffect == 0) launch_advance_th<V, FC, false>(s, w, conds, pr, tables, h, fl, st);
    else launch_advance_th<V, FC, true>(s, w, conds, pr, tables, h, fl, st);
}

template <typename V>
int flight_blocks_per_cu(int fc, bool thermal, int P, const DevHist& h) {
    const void* k = nullptr;
    const int hm = hist_mode(h);
    switch (fc) {
        case FIELD_DC: k = thermal ? flight_kernel<V, FIELD_DC, true>(hm) : flight_kernel<V, FIELD_DC, false>(hm); break;
        case FIELD_AC: k = thermal ? flight_kernel<V, FIELD_AC, true>(hm) : flight_kernel<V, FIELD_AC, false>(hm); break;
        case FIELD_DC_B:
            k = thermal ? flight_kernel<V, FIELD_DC_B, true>(hm) : flight_kernel<V, FIELD_DC_B, false>(hm);
            break;
        case FIELD_ECR:
            k = thermal ? flight_kernel<V, FIELD_ECR, true>(hm) : flight_kernel<V, FIELD_ECR, false>(hm);
            break;
        case FLIGHT_DC_ANY:
            k = thermal ? flight_kernel<V, FLIGHT_DC_ANY, true>(hm) : flight_kernel<V, FLIGHT_DC_ANY, false>(hm);
            break;
        default: k = thermal ? flight_kernel<V, FIELD_AC_B, true>(hm) : flight_kernel<V, FIELD_AC_B, false>(hm); break;
    }
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, kBlock, flight_lds<V>(P, h.histLds)) != hipSuccess || n < 1)
        n = 1;
    return n;
}

template <typename V>
hipError_t launch_flights(const DevState<V>& s, const DevWork& w, const CondParams* conds, const DevProcesses& pr, const V* tables,
                          const DevHist& h, const FlightLists& fl, KernelTimer* timer, hipStream_t st) {
    timer_start(timer, K_ADVANCE, st);
    launch_advance_case<V, FIELD_DC>(s, w, conds, pr, tables, h, fl, st);
    launch_advance_case<V, FIELD_AC>(s, w, conds, pr, tables, h, fl, st);
    launch_advance_case<V, FIELD_DC_B>(s, w, conds, pr, tables, h, fl, st);
    launch_advance_case<V, FIELD_ECR>(s, w, conds, pr, tables, h, fl, st);
    launch_advance_case<V, FIELD_AC_B>(s, w, conds, pr, tables, h, fl, st);
    launch_advance_case<V, FLIGHT_DC_ANY>(s, w, conds, pr, tables, h, fl, st);
    timer_stop(timer, K_ADVANCE, st);
    return hipGetLastError();
}

template <typename V>
hipError_t launch_popctl(const DevState<V>& s, const DevWork& w, KernelTimer* timer, hipStream_t st) {
    const dim3 g(chunk_grid(w.nChunks)), b(kBlock);
    timer_start(timer, K_MARKS, st);
    hipLaunchKernelGGL(k_marks, g, b, 0, st, s.alive, w);
    if (w.planMarks) hipLaunchKernelGGL(k_plan_marks, dim3(w.nCond), dim3(kPlanBlock), 0, st, w);
    timer_stop(timer, K_MARKS, st);
    timer_start(timer, K_APPLY, st);
    hipLaunchKernelGGL(k_apply_marks<V>, g, b, 0, st, s, w);
    if (w.planPairs) hipLaunchKernelGGL(k_plan_pairs, dim3(w.nCond), dim3(1024), 0, st, w);
    timer_stop(timer, K_APPLY, st);
    return hipGetLastError();
}

template <typename V>
hipError_t launch_settle(const DevState<V>& s, const DevWork& w, KernelTimer* timer, hipStream_t st) {
    timer_start(timer, K_SETTLE, st);
    hipLaunchKernelGGL(k_settle<V>, dim3(chunk_grid(w.nChunks)), dim3(kBlock), 0, st, s, w);
    timer_stop(timer, K_SETTLE, st);
    return hipGetLastError();
}

template <typename V>
hipError_t launch_hist(const DevState<V>& s, const DevHist& h, KernelTimer* timer, hipStream_t st) {
    if (h.nRanges == 0) return hipSuccess;
    const int ldsCells = h.nCells <= 8192 ? h.nCells : 0;
    const size_t lds = (size_t)ldsCells * 4;
    timer_start(timer, K_HIST, st);
    hipLaunchKernelGGL(k_hist<V>, dim3(h.nRanges), dim3(kBlock), lds, st, s, h.ranges, h, ldsCells);
    timer_stop(timer, K_HIST, st);
    return hipGetLastError();
}

hipError_t launch_finish(const DevWork& w, int P, KernelTimer* timer, hipStream_t st) {
    timer_start(timer, K_REDUCE, st);
    if (w.nGroups) hipLaunchKernelGGL(k_finish_group, dim3(w.nGroups), dim3(kFinishBlock), 0, st, w);
    hipLaunchKernelGGL(k_finish, dim3(w.nCond), dim3(kFinishBlock), 0, st, w, P);
    timer_stop(timer, K_REDUCE, st);
    return hipGetLastError();
}

template <typename V>
hipError_t launch_op_accelerate(const CondParams* cond, int64_t n, const double* time, const double* dt,
                                double* pos, double* vel, double* energy, double* gain, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_op_accelerate<V>, dim3(grid_of(n)), dim3(kBlock), 0, st, cond, n, time, dt, pos, vel,
                       energy, gain);
    return hipGetLastError();
}

template <typename V>
hipError_t launch_op_collide(const CondParams* cond, const DevProcesses& pr, const V* tables, int64_t n,
                             double* vel, double* energy, const double* nue, const double* variates,
                             int32_t* pid, double* ejv, double* eje, double* de, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_op_collide<V>, dim3(grid_of(n)), dim3(kBlock), 0, st, cond, pr, tables, n, vel, energy,
                       nue, variates, pid, ejv, eje, de);
    return hipGetLastError();
}

hipError_t run_beside(hipStream_t a, hipStream_t b, uint32_t* word, bool* beside) {
    uint32_t answer = 0;
    hipError_t e = hipSuccess;
    // the first turn only brings the streams into being on the device
    for (int turn = 0; turn < 2 && e == hipSuccess; ++turn) {
        e = hipMemsetAsync(word, 0, 2 * sizeof(uint32_t), a);
        if (e == hipSuccess) e = hipStreamSynchronize(a);
        if (e == hipSuccess && turn == 1) {
            hipLaunchKernelGGL(k_await, dim3(1), dim3(1), 0, a, word);
            e = hipGetLastError();
        }
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_signal, dim3(1), dim3(1), 0, b, word);
            e = hipGetLastError();
        }
        const hipError_t ea = hipStreamSynchronize(a), eb = hipStreamSynchronize(b);
        if (e == hipSuccess) e = ea != hipSuccess ? ea : eb;
    }
    if (e == hipSuccess) e = hipMemcpy(&answer, word + 1, sizeof(answer), hipMemcpyDeviceToHost);
    *beside = e == hipSuccess && answer != 0;
    return e;
}

hipError_t launch_op_philox(int64_t n, const uint32_t* ctr, const uint32_t* key, uint32_t* out, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_op_philox, dim3(grid_of(n)), dim3(kBlock), 0, st, n, ctr, key, out);
    return hipGetLastError();
}

#define EKMC_INSTANTIATE(V)                                                                                   \
    template hipError_t launch_init<V>(const DevState<V>&, const DevWork&, int64_t, const int64_t*,           \
                                       const double*, KernelTimer*, hipStream_t);                                           \
    template hipError_t launch_flights<V>(const DevState<V>&, const DevWork&, const CondParams*, const DevProcesses&, const V*,  \
                                          const DevHist&, const FlightLists&, KernelTimer*, hipStream_t);                   \
    template hipError_t launch_popctl<V>(const DevState<V>&, const DevWork&, KernelTimer*, hipStream_t);                    \
    template hipError_t launch_settle<V>(const DevState<V>&, const DevWork&, KernelTimer*, hipStream_t);                    \
    template hipError_t launch_hist<V>(const DevState<V>&, const DevHist&, KernelTimer*, hipStream_t);                     \
    template int flight_blocks_per_cu<V>(int, bool, int, const DevHist&);                                                \
    template hipError_t launch_tables<V>(const DevTableSrc&, double, double, int, V*, double*, double*,        \
                                         hipStream_t);                                                       \
    template hipError_t launch_op_accelerate<V>(const CondParams*, int64_t, const double*, const double*,     \
                                                double*, double*, double*, double*, hipStream_t);             \
    template hipError_t launch_op_collide<V>(const CondParams*, const DevProcesses&, const V*, int64_t,       \
                                             double*, double*, const double*, const double*, int32_t*,        \
                                             double*, double*, double*, hipStream_t);
EKMC_INSTANTIATE(double)
EKMC_INSTANTIATE(float)

}  // namespace ekmc
