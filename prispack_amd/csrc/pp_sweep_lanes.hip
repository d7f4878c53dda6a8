// pp_sweep_lanes.hip -- the chunked triangular sweeps (PP_TRSV_BLOCK): one
// workgroup runs both sweeps of a dependency-closed chunk of rows, the
// chunk's part of the vector in LDS.
//
// What bounds them is the chain of dependent rows (1012 per sweep for ICT(1e-3)
// on the 128^2 Poisson problem, about 16 rows wide): its length times what one
// link costs.  A link is a row's gathers from LDS, its products, its ordered
// subtractions (bit for bit the serial sweep's), the division and the LDS
// write, and the instructions around them, which one wavefront issues at one
// per four cycles or so.  So the rows are scheduled on the host into steps
// that one wavefront executes in lockstep without any barrier (LDS accesses
// of a wavefront stay in order); a row may be spread over several lanes, which
// gather and multiply its entries at once; every step's data comes in a
// ready-to-use layout, loaded kLaneAhead steps ahead; and divisions go by
// the pivots' reciprocals (five operations, same bits).  An apply of that
// factor takes 0.42 ms in FP64 (0.18 us a step); one workgroup barrier and
// one LDS round trip more per level, with data loaded one level ahead, took
// 2.0 ms (1.0 us a level).  Rows of several parts kept in consecutive steps,
// their sums carried in registers, took 0.45 ms (flags and selects a step).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <memory>
#include <queue>
#include <unordered_map>

#include "pp_internal.h"

namespace pp {

namespace {

constexpr int kAhead = kLaneAhead;  // steps whose data is in flight or in registers
constexpr int kLaneThreads = 256;
constexpr uint32_t kExtra = 1;      // LDS words past the chunk's rows: a zero
constexpr uint32_t kNeedUnit = 8;   // a strip's step waits for so many imports at a time
constexpr uint32_t kNoExport = 0xffffu;

// What a lane needs of one step: 16-byte pieces, piece k of the step's
// active lanes contiguous, so every load is one coalesced 16-byte load per lane.
//   values   S values of T
//   indices  16 bits each: the S dependencies' LDS words; the row's word; the
//            imports the step waits for (kNeedUnit each, strips only); the
//            step's rows - 1 and those of the step kAhead later (8 bits each);
//            the row's export number in its strip or kNoExport
//   pivot    the row's diagonal and its reciprocal rounded to FP64
template <class T, int S>
struct Step {
    static constexpr int kVal = S * (int)sizeof(T) / 16, kIdx = (2 * S + 8 + 15) / 16;
    static constexpr int kPieces = kVal + kIdx + 1;
    static constexpr int kRowWord = S / 2, kInfoWord = S / 2 + 1;  // 32-bit words of the indices
    int4 p[kPieces];
    __device__ static int word(const int4 &q, int w) { return w == 0 ? q.x : w == 1 ? q.y : w == 2 ? q.z : q.w; }
    __device__ T v(int j) const {
        if constexpr (sizeof(T) == 8) {
            const int4 &q = p[j >> 1];
            return __hiloint2double(word(q, 2 * (j & 1) + 1), word(q, 2 * (j & 1)));
        } else {
            return __int_as_float(word(p[j >> 2], j & 3));
        }
    }
    // 32-bit word w of the indices
    __device__ int ix(int w) const { return word(p[kVal + (w >> 2)], w & 3); }
    __device__ T d() const {
        if constexpr (sizeof(T) == 8) return __hiloint2double(p[kPieces - 1].y, p[kPieces - 1].x);
        else return __int_as_float(p[kPieces - 1].x);
    }
    __device__ double rcp() const { return __hiloint2double(p[kPieces - 1].w, p[kPieces - 1].z); }
};

// s / d, correctly rounded, by the reciprocal r = RN(1 / d): one Newton
// correction makes q faithful, and then q + (s - q d) r rounds to the
// quotient (P. Markstein, IBM J. Res. Dev. 34 (1990) 111-119): five dependent
// operations instead of the dozen of an IEEE division, which sit on every
// level's critical path.  Quotients outside [2^-500, 2^500] (zeros,
// infinities and NaNs among them) and pivots outside [2^-300, 2^300], whose r
// is NaN, take the division itself.
__device__ inline double quotient(double s, double d, double r) {
    double q = s * r;
    const bool plain = (((uint32_t)__double2hiint(q) >> 20) & 0x7ffu) - 523u <= 1000u;
    q = __builtin_fma(__builtin_fma(-q, d, s), r, q);
    q = __builtin_fma(__builtin_fma(-q, d, s), r, q);
    if (__builtin_expect(__any(!plain), 0)) {
        asm volatile("" : "+v"(d));  // keeps the division out of the common path
        if (!plain) q = s / d;
    }
    return q;
}
// FP32: the FP64 product s r is within 2^-52 of the quotient, and a quotient
// of two 24-bit numbers lies further than 2^-49 from every midpoint of two
// neighbouring normal FP32 numbers, so rounding it gives RN(s / d).
__device__ inline float quotient(float s, float d, double r) {
    float q = (float)((double)s * r);
    const bool plain = (((uint32_t)__float_as_int(q) >> 23) & 0xffu) - 7u <= 240u;  // 2^-120 <= |q| <= 2^120
    if (__builtin_expect(__any(!plain), 0)) {
        asm volatile("" : "+v"(d));
        if (!plain) q = s / d;
    }
    return q;
}
// the pivots quotient() takes by their reciprocal
template <class T>
double step_reciprocal(T d) {
    const double a = std::fabs((double)d), lim = sizeof(T) == 8 ? 0x1p300 : 0x1p100;
    return a <= lim && a >= 1.0 / lim ? 1.0 / (double)d : std::nan("");
}

template <int CTRL>
__device__ inline double dpp(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
template <int CTRL>
__device__ inline float dpp(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
constexpr int kRowShr = 0x110;  // DPP: lane i takes lane i - n of its 16

// Word h (0 low, 1 high) of a pair of 16-bit LDS words, as a byte offset.
template <class T, int H>
__device__ inline uint32_t lds_byte(int pair) {
    uint32_t o;
    const uint32_t sh = sizeof(T) == 8 ? 3 : 2;
    if constexpr (H == 0)
        asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0"
            : "=v"(o)
            : "v"(sh), "v"(pair));
    else
        asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1"
            : "=v"(o)
            : "v"(sh), "v"(pair));
    return o;
}
// The LDS word at a byte offset: the kernel has no static LDS, so its
// dynamic LDS starts at address 0 and an offset is an address (the generic
// pointer's base costs an addition per access).
template <class T>
using LdsWord = __attribute__((address_space(3))) T;
template <class T>
__device__ inline LdsWord<T> *lds_word(uint32_t byte) {
    return (LdsWord<T> *)byte;
}

// The next step's data; p moves past it.  Lanes past the active ones take
// the last one's, so every load is unconditional and the compiler knows how
// many are in flight: it waits for the oldest step's alone.
template <class T, int S>
__device__ inline void load_step(Step<T, S> &q, const char *&p, uint32_t active, uint32_t lane) {
    const uint32_t off = min(lane, active - 1) * 16, stride = active * 16;
#pragma unroll
    for (int k = 0; k < Step<T, S>::kPieces; ++k)
        q.p[k] = *reinterpret_cast<const int4 *>(p + (uint32_t)(off + k * stride));
    p += Step<T, S>::kPieces * stride;
    // steps stay in order: the oldest loads are the next needed
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// The LDS words of a step: its dependencies, then its row.
template <class T, int S>
struct StepAddr {
    uint32_t dep[S], row;
    __device__ void set(const Step<T, S> &q) {
#pragma unroll
        for (int j = 0; j < S; j += 2) {
            dep[j] = lds_byte<T, 0>(q.ix(j / 2));
            dep[j + 1] = lds_byte<T, 1>(q.ix(j / 2));
        }
        row = lds_byte<T, 0>(q.ix(Step<T, S>::kRowWord));
    }
};

// Carried from step to step.
template <class T, int S>
struct Carry {
    StepAddr<T, S> addr;  // of the next step
    uint32_t need;        // imports the next step waits for
    uint32_t active;      // lanes of the step kAhead - 1 past the next one
};

// One step, its data in q: G lanes a row, S entries a lane, in storage order
// along the row's lanes.  Every lane gathers and multiplies its entries at
// once; the subtractions follow one after another, the partial sum moving
// from lane to lane (DPP), so the row's operations are those of the serial
// sweep.  A row of more than G S entries is several such parts, each in a
// step of its own: the partial sum waits in the row's LDS word, and a part
// whose diagonal operation is not due holds the pivot 1 (s / 1 and s * 1 are
// s).  The gathers go out first: while they are on their way, the loads of
// the step kAhead - 1 later (into `past`, the last step's slot) are issued
// and the next step's addresses unpacked.  xchg.wait(need) returns once the
// step's imports are in LDS, xchg.put passes a finished row on.
template <class T, int W, int G, int S, int MODE, class Xchg>
__device__ inline void run_step(const Step<T, S> &q, const Step<T, S> &next, Step<T, S> &past, const char *&p,
                                Carry<T, S> &c, uint32_t lane, uint32_t tail_lane, Xchg &xchg) {
#pragma clang fp contract(off)
    xchg.wait(c.need);
    T x[S];
#pragma unroll
    for (int j = 0; j < S; ++j) x[j] = *lds_word<T>(c.addr.dep[j]);
    LdsWord<T> *mine = lds_word<T>(c.addr.row);
    T s = *mine;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    load_step<T, S>(past, p, c.active, lane);
    const uint32_t info = (uint32_t)__builtin_amdgcn_readfirstlane(q.ix(Step<T, S>::kInfoWord));
    c.active = ((info >> 8 & 0xffu) + 1) * G;
    c.addr.set(next);
    if constexpr (Xchg::kOn) c.need = (uint32_t)__builtin_amdgcn_readfirstlane(next.ix(Step<T, S>::kRowWord)) >> 16;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (MODE == HostSweep::PREDIVIDE) s = quotient(s, q.d(), q.rcp());
#pragma unroll
    for (int j = 0; j < S; ++j) x[j] = q.v(j) * x[j];
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int j = 0; j < S; ++j) s = s - x[j];
        if (g < G - 1) s = dpp<kRowShr + 1>(s);
    }
    if constexpr (MODE == HostSweep::DIVIDE) s = quotient(s, q.d(), q.rcp());
    else if constexpr (MODE == HostSweep::MULTIPLY) s = s * q.d();
    if (tail_lane < ((info & 0xffu) + 1) * G) {
        *mine = s;
        xchg.put((uint32_t)q.ix(Step<T, S>::kInfoWord) >> 16, s);
    }
    if constexpr (W > 1) __syncthreads();
}

struct NoExchange {
    static constexpr bool kOn = false;
    __device__ void wait(uint32_t) {}
    template <class T>
    __device__ void put(uint32_t, T) {}
};

// Copies n elements between global memory and LDS, eight loads of a thread
// in flight (one at a time, the 16,384 rows of a chunk cost 0.1 ms).
template <class T>
__device__ inline void copy_rows(T *dst, const T *src, uint32_t n) {
    constexpr int U = 8;
    for (uint32_t j = threadIdx.x; j < n; j += U * kLaneThreads) {
        T v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = src[min(j + u * kLaneThreads, n - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (j + u * kLaneThreads < n) dst[j + u * kLaneThreads] = v[u];
    }
}

// The first W wavefronts run the steps; the others help to copy the chunk's
// part of the vector in and out.
template <class T, int W, int G, int S, int MLO, int MUP>
__global__ __launch_bounds__(kLaneThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_sweep_lanes(
    const uint32_t *__restrict__ start, const LaneHead *__restrict__ head, const char *data, const T *x, T *y,
    const int *stop) {
    static_assert(W == 1 || W * 64 == kLaneThreads, "a barrier inside the steps needs the whole workgroup");
    extern __shared__ unsigned char lds_raw[];
    T *xs = reinterpret_cast<T *>(lds_raw);
    if (stop && *stop) return;
    const uint32_t c = blockIdx.x, r0 = start[c], nr = start[c + 1] - r0;
    const uint32_t lo = head[c].rounds_lo, up = head[c].rounds_up;
    copy_rows(xs, x + r0, nr);
    if (threadIdx.x == 0) xs[nr] = T(0);
    __syncthreads();
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wave < W) {
        const char *p = data + head[c].first;
        // a lane that finishes a row: its number; the others: none
        const uint32_t lane = threadIdx.x, tail_lane = (lane & (G - 1)) == G - 1 ? lane : 0xffffffffu;
        Step<T, S> q[kAhead];
#pragma unroll
        for (int a = 0; a < kAhead - 1; ++a) load_step<T, S>(q[a], p, head[c].active[a], lane);
        Carry<T, S> st;
        st.active = head[c].active[kAhead - 1];
        st.addr.set(q[0]);
        NoExchange xchg;
        for (uint32_t k = 0; k < lo; ++k) {
#pragma unroll
            for (int a = 0; a < kAhead; ++a)
                run_step<T, W, G, S, MLO>(q[a], q[(a + 1) % kAhead], q[(a + kAhead - 1) % kAhead], p, st, lane,
                                          tail_lane, xchg);
        }
        for (uint32_t k = 0; k < up; ++k) {
#pragma unroll
            for (int a = 0; a < kAhead; ++a)
                run_step<T, W, G, S, MUP>(q[a], q[(a + 1) % kAhead], q[(a + kAhead - 1) % kAhead], p, st, lane,
                                          tail_lane, xchg);
        }
    }
    __syncthreads();
    copy_rows(y + r0, xs, nr);
}

// ---------------------------------------------------------------------------
// Strips: the sweeps of a factor whose rows do not chunk (one connected part
// larger than LDS).  The rows are cut into contiguous strips, a workgroup and
// its LDS each; wavefront 0 runs the strip's steps.  A finished row that
// other strips read goes from its lane's register straight to the row's slot
// of an exchange buffer (agent-scope store); in the strips that read it, the
// other wavefronts poll the slots in the order the steps need them and put the
// values into LDS.  A slot holds a signalling NaN, which no sum is, until its
// value arrives, so a value is its own ready flag (a value passes between
// two compute units in about 0.6 us, 0.45 on one XCD).  The buffers belong to
// the context, whose stream keeps its applies apart (two contexts may apply
// one preconditioner at the same time): the forward sweep's is empty between
// applies, because the backward sweep empties the slots it used, and the
// backward sweep's is emptied by the forward sweep before it.
// A strip waits only for strips before it in its sweep's direction, whose
// workgroups are dispatched before its own, so the first unfinished strip
// always proceeds; a wait past the deadline (nothing new among the 256 imports
// a wavefront polls) sets C_SPIN, and every wavefront runs to its end (the rows
// become NaN).
// ---------------------------------------------------------------------------
constexpr int kImport = kLaneThreads / 64 - 1, kBatch = 4;
constexpr uint32_t kStripCtl = 32;  // bytes of LDS: per import wavefront the imports it has seen; the abort word
enum : uint32_t { CW_ABORT = 7 };

template <class T>
struct SlotBits;
template <>
struct SlotBits<double> {
    using U = unsigned long long;
    static constexpr U empty = 0x7FF4B5A5C3D2E1F0ull;
};
template <>
struct SlotBits<float> {
    using U = unsigned int;
    static constexpr U empty = 0x7FA5C3E1u;
};

struct StripHead {
    LaneHead lanes;                 // rounds_lo: all of the sweep's rounds
    uint32_t row = 0, rows = 0;
    uint32_t imp = 0, nimp = 0;     // imports: slots, by the step that first needs them
    uint32_t exp = 0;               // first slot of its exported rows
};

// control words in LDS (not through a generic pointer: a flat access would
// wait for every step in flight)
using CtlWord = volatile __attribute__((address_space(3))) uint32_t;

// Wavefront 0's side of the exchange.
template <class T>
struct Exchange {
    static constexpr bool kOn = true;
    CtlWord *cw;
    T *slots;       // the strip's own
    uint32_t have;  // imports known to be in LDS
    __device__ void wait(uint32_t need) {
        while (have < need * kNeedUnit) {
            uint32_t done = 0xffffffffu;
#pragma unroll
            for (int f = 0; f < kImport; ++f) done = min(done, cw[f]);
            if (cw[CW_ABORT]) done = 0xffffffffu;
            have = (uint32_t)__builtin_amdgcn_readfirstlane(done);
        }
        // the step's gathers are ordinary loads: they stay behind the polls
        asm volatile("" ::: "memory");
    }
    __device__ void put(uint32_t number, T s) {
        using U = typename SlotBits<T>::U;
        if (number != kNoExport)
            __hip_atomic_store(reinterpret_cast<U *>(slots) + number, __builtin_bit_cast(U, s), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
};

template <class T>
__global__ void k_slots_empty(uint32_t n, T *slots) {
    using U = typename SlotBits<T>::U;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        reinterpret_cast<U *>(slots)[i] = SlotBits<T>::empty;
}

// imp: the imports of all strips; slots: the sweep's exchange buffer; other:
// the other sweep's, emptied here.
template <class T, int G, int S, int MODE>
__global__ __launch_bounds__(kLaneThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) void k_sweep_strips(
    const StripHead *__restrict__ heads, const char *data, const uint32_t *__restrict__ imp, T *slots,
    uint32_t other_n, T *other, uint32_t ctl_off, const T *x, T *y, long long deadline, int *ctl, int *late,
    const int *stop) {
    using U = typename SlotBits<T>::U;
    constexpr U kEmpty = SlotBits<T>::empty;
    extern __shared__ unsigned char lds_raw[];
    T *xs = reinterpret_cast<T *>(lds_raw);
    CtlWord *cw = (CtlWord *)ctl_off;  // dynamic LDS starts at address 0
    if (stop && *stop) return;
    const StripHead &h = heads[blockIdx.x];
    const uint32_t nr = h.rows;
    copy_rows(xs, x + h.row, nr);
    if (threadIdx.x == 0) xs[nr] = T(0);
    if (threadIdx.x < kStripCtl / 4) cw[threadIdx.x] = threadIdx.x < kImport ? threadIdx.x * kBatch * 64 : 0;
    for (uint32_t i = blockIdx.x * kLaneThreads + threadIdx.x; i < other_n; i += gridDim.x * kLaneThreads)
        reinterpret_cast<U *>(other)[i] = kEmpty;
    __syncthreads();
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t rounds = h.lanes.rounds_lo;
    if (wave == 0) {
        const char *p = data + h.lanes.first;
        const uint32_t tail_lane = (lane & (G - 1)) == G - 1 ? lane : 0xffffffffu;
        Step<T, S> q[kAhead];
#pragma unroll
        for (int a = 0; a < kAhead - 1; ++a) load_step<T, S>(q[a], p, h.lanes.active[a], lane);
        Carry<T, S> st;
        st.active = h.lanes.active[kAhead - 1];
        st.addr.set(q[0]);
        st.need = (uint32_t)__builtin_amdgcn_readfirstlane(q[0].ix(S / 2)) >> 16;
        Exchange<T> xchg{cw, slots + h.exp, 0};
        for (uint32_t k = 0; k < rounds; ++k) {
#pragma unroll
            for (int a = 0; a < kAhead; ++a)
                run_step<T, 1, G, S, MODE>(q[a], q[(a + 1) % kAhead], q[(a + kAhead - 1) % kAhead], p, st, lane,
                                           tail_lane, xchg);
        }
    } else {
        // kBatch groups of 64 imports polled together, the wavefronts taking
        // turns; cw[f]: the imports below it are in LDS, as far as wavefront
        // f is concerned
        const uint32_t f = wave - 1;
        bool abort = false;
        const auto slot_of = [&](uint32_t i) { return imp[h.imp + min(i, h.nimp - 1)]; };
        uint32_t to[kBatch] = {};
        if (h.nimp) {
#pragma unroll
            for (int b = 0; b < kBatch; ++b) to[b] = slot_of((f * kBatch + b) * 64 + lane);
        }
        for (uint32_t i0 = f * kBatch * 64; i0 < h.nimp && !abort; i0 += kImport * kBatch * 64) {
            U *slot[kBatch];
            bool wait[kBatch];
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                wait[b] = i0 + b * 64 + lane < h.nimp;
                slot[b] = reinterpret_cast<U *>(slots) + to[b];
                to[b] = slot_of(i0 + (kImport * kBatch + b) * 64 + lane);  // the next batch's
            }
            WaitClock clock;
            bool got = false;
            for (uint32_t iter = 1;; ++iter) {
                U v[kBatch];
#pragma unroll
                for (int b = 0; b < kBatch; ++b)
                    v[b] = wait[b] ? __hip_atomic_load(slot[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : kEmpty;
                uint32_t seen = kBatch * 64;  // imports of the batch before the first one missing
#pragma unroll
                for (int b = kBatch - 1; b >= 0; --b) {
                    if (v[b] != kEmpty) {
                        xs[nr + 1 + i0 + b * 64 + lane] = __builtin_bit_cast(T, v[b]);
                        wait[b] = false;
                        got = true;
                    }
                    const unsigned long long m = __ballot(wait[b]);
                    if (m) seen = b * 64 + __builtin_ctzll(m);
                }
                asm volatile("" ::: "memory");
                // all of them: the next one to see is the next batch's first
                cw[f] = i0 + (seen < kBatch * 64 ? seen : kImport * kBatch * 64);
                if (seen == kBatch * 64) break;
                if (!WaitClock::due(iter, deadline)) continue;
                if (__any(got)) {  // another wait from here on
                    got = false;
                    clock = WaitClock();
                } else if (clock.expired(deadline) ||
                           __hip_atomic_load(&ctl[C_SPIN], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                    give_up(ctl, late);
                    cw[CW_ABORT] = 1;
                    abort = true;
                    break;
                }
            }
        }
        cw[f] = 0x7fffffffu;  // no import left: nothing to wait for here
    }
    __syncthreads();
    if (cw[CW_ABORT])
        for (uint32_t j = threadIdx.x; j < nr; j += kLaneThreads) xs[j] = __builtin_nanf("");
    __syncthreads();
    copy_rows(y + h.row, xs, nr);
}

// ---------------------------------------------------------------------------
// Host: which rows go into which step.
// ---------------------------------------------------------------------------

// A row's entries [a, b) of one step (a row of more entries than a step's G S
// is several parts, the remainder first, so that the last part, which the
// rows after it wait for, holds as many of the latest dependencies as it can).
struct Part {
    uint32_t row, a, b;
    bool first, last;
};
// The parts of one chunk or strip in the order of its steps.
struct LanePlan {
    struct Group {
        uint32_t first, count;  // parts[first, first + count) make a step
    };
    std::vector<Part> parts;
    std::vector<Group> steps;
};

// List scheduling of the rows [bound[0], bound.back()) of a sweep, all strips
// [bound[k], bound[k + 1]) together, a step of every strip at a time: a step
// takes up to `width` parts whose dependencies are visible, those with the
// longest chains behind them first; so the steps are about as few as the
// longest chain, or the parts over `width`, allows.  A row of another strip
// is visible kStripLag steps after its step (the exchange takes about
// 1.5 us), so the order in which a strip takes its rows is one in which it
// rarely waits.  span: the steps until the last strip ends.
constexpr uint32_t kStripLag = 10;
std::vector<LanePlan> plan_steps(const HostSweep &s, const std::vector<uint32_t> &bound, uint32_t width,
                                 uint32_t entries, uint32_t &span) {
    const uint32_t K = (uint32_t)bound.size() - 1, r0 = bound[0], n = bound[K] - r0;
    std::vector<LanePlan> P(K);
    span = 0;
    if (!n) return P;
    // parts, row after row; part[i] .. part[i + 1] are row r0 + i's
    std::vector<uint32_t> part(n + 1, 0), strip_of(n);
    for (uint32_t k = 0; k < K; ++k)
        std::fill(strip_of.begin() + (bound[k] - r0), strip_of.begin() + (bound[k + 1] - r0), k);
    for (uint32_t i = 0; i < n; ++i)
        part[i + 1] = part[i] + std::max(1u, (s.rp[r0 + i + 1] - s.rp[r0 + i] + entries - 1) / entries);
    const uint32_t np = part[n];
    std::vector<Part> parts(np);
    std::vector<uint32_t> wait(np), seen(np, 0), height(np), sp(n + 1, 0), sc(s.rp[r0 + n] - s.rp[r0]);
    for (uint32_t i = 0; i < n; ++i) {
        const uint32_t m = part[i + 1] - part[i], e1 = s.rp[r0 + i + 1];
        uint32_t a = s.rp[r0 + i], b = e1 - (m - 1) * entries;
        for (uint32_t u = part[i]; u < part[i + 1]; ++u, a = b, b += entries) {
            parts[u] = {r0 + i, a, b, u == part[i], u + 1 == part[i + 1]};
            wait[u] = b - a + (u == part[i] ? 0 : 1);
            for (uint32_t e = a; e < b; ++e) sp[s.ci[e] - r0 + 1]++;
        }
    }
    for (uint32_t i = 0; i < n; ++i) sp[i + 1] += sp[i];
    {
        std::vector<uint32_t> at(sp.begin(), sp.end() - 1);
        for (uint32_t u = 0; u < np; ++u)
            for (uint32_t e = parts[u].a; e < parts[u].b; ++e) sc[at[s.ci[e] - r0]++] = u;
    }
    auto strip = [&](uint32_t u) { return strip_of[parts[u].row - r0]; };
    // dependents of a row come after it (lower) or before it (upper)
    for (uint32_t k = 0; k < n; ++k) {
        const uint32_t i = s.lower ? n - 1 - k : k;
        uint32_t h = 0;
        for (uint32_t e = sp[i]; e < sp[i + 1]; ++e)
            h = std::max(h, height[sc[e]] + (strip(sc[e]) != strip_of[i] ? kStripLag : 0u));
        for (uint32_t u = part[i + 1]; u-- > part[i];) height[u] = ++h;
    }
    auto less = [&](uint32_t a, uint32_t b) { return height[a] != height[b] ? height[a] < height[b] : a > b; };
    std::vector<std::vector<uint32_t>> ready(K), due;  // due[t]: parts whose dependencies are visible at step t
    auto make_due = [&](uint32_t u, uint32_t t) {
        if (t >= due.size()) due.resize(t + 1 + t / 2);
        due[t].push_back(u);
    };
    for (uint32_t u = 0; u < np; ++u)
        if (!wait[u]) make_due(u, 0);
    uint32_t left = np;
    for (uint32_t t = 0; left; ++t) {
        if (t < due.size()) {
            std::vector<uint32_t> now;
            now.swap(due[t]);
            for (uint32_t u : now) {
                auto &q = ready[strip(u)];
                q.push_back(u);
                std::push_heap(q.begin(), q.end(), less);
            }
        }
        for (uint32_t k = 0; k < K; ++k) {
            auto &q = ready[k];
            if (q.empty()) continue;
            LanePlan &p = P[k];
            LanePlan::Group g{(uint32_t)p.parts.size(), 0};
            const auto visible = [&](uint32_t u, uint32_t at) {
                seen[u] = std::max(seen[u], at);
                if (--wait[u] == 0) make_due(u, seen[u]);
            };
            while (!q.empty() && g.count < width) {
                std::pop_heap(q.begin(), q.end(), less);
                const uint32_t u = q.back();
                q.pop_back();
                p.parts.push_back(parts[u]);
                ++g.count;
                if (!parts[u].last) {
                    visible(u + 1, t + 1);
                    continue;
                }
                const uint32_t i = parts[u].row - r0;
                for (uint32_t e = sp[i]; e < sp[i + 1]; ++e)
                    visible(sc[e], t + 1 + (strip(sc[e]) != k ? kStripLag : 0u));
            }
            left -= g.count;
            p.steps.push_back(g);
        }
        span = t + 1;
    }
    return P;
}

// A step to write: nullptr: idle (fills a sweep's last round).
struct StepRef {
    const HostSweep *sweep = nullptr;
    const LanePlan *plan = nullptr;
    LanePlan::Group group{0, 1};
    uint32_t need = 0;  // imports (kNeedUnit each) it waits for
};
inline uint32_t rows_of(const std::vector<StepRef> &v, size_t k) { return k < v.size() ? v[k].group.count : 1u; }

void append_steps(const HostSweep &s, const LanePlan &P, std::vector<StepRef> &out) {
    for (const auto &g : P.steps) out.push_back({&s, &P, g, 0});
    while (out.size() % kAhead) out.push_back({});
}

// One step at `out`, `rows` of it and `ahead` of the step kAhead later; its
// LDS holds the rows from r0 on at words 0 .. nr - 1 and a zero at nr.
// word(row): the LDS word of a dependency; number(row): its export number.
template <class T, int S, class Word, class Number>
void write_step(const StepRef &r, uint32_t r0, uint32_t nr, int G, uint32_t ahead, unsigned char *out,
                const Word &word, const Number &number) {
    using St = Step<T, S>;
    const uint32_t rows = r.group.count, lanes = rows * G;
    const size_t piece = (size_t)lanes * 16;
    for (uint32_t l = 0; l < lanes; ++l) {
        T v[S] = {}, d = T(1);
        uint16_t ix[St::kIdx * 8];
        std::fill(ix, ix + St::kIdx * 8, (uint16_t)nr);
        uint32_t exported = kNoExport;
        if (r.sweep) {
            const HostSweep &s = *r.sweep;
            const Part &q = r.plan->parts[r.group.first + l / G];
            const uint32_t a = q.a + (l % G) * S;
            for (int j = 0; j < S; ++j)
                if (a + j < q.b) {
                    v[j] = (T)s.val[a + j];
                    ix[j] = (uint16_t)word(s.ci[a + j]);
                }
            ix[S] = (uint16_t)(q.row - r0);
            if (s.mode == HostSweep::PREDIVIDE ? q.first : s.mode != HostSweep::UNIT && q.last) d = (T)s.diag[q.row];
            if (q.last) exported = number(q.row);
        }
        ix[S + 1] = (uint16_t)r.need;
        ix[S + 2] = (uint16_t)((rows - 1) | (ahead - 1) << 8);
        ix[S + 3] = (uint16_t)exported;
        const double rcp = step_reciprocal<T>(d);
        for (int q = 0; q < St::kVal; ++q) std::memcpy(out + q * piece + 16 * l, (unsigned char *)v + 16 * q, 16);
        for (int q = 0; q < St::kIdx; ++q)
            std::memcpy(out + (St::kVal + q) * piece + 16 * l, (unsigned char *)ix + 16 * q, 16);
        unsigned char *pv = out + (St::kPieces - 1) * piece + 16 * l;
        std::memset(pv, 0, 8);
        std::memcpy(pv, &d, sizeof(T));
        std::memcpy(pv + 8, &rcp, 8);
    }
}

// Byte offset and lane counts of every chunk's or strip's steps; returns the total.
template <class Head>
uint64_t place_steps(const std::vector<std::vector<StepRef>> &steps, int G, size_t lane_bytes, std::vector<Head> &head,
                     LaneHead &(*lanes)(Head &)) {
    uint64_t total = 0;
    for (size_t c = 0; c < steps.size(); ++c) {
        LaneHead &h = lanes(head[c]);
        h.first = total;
        for (int a = 0; a < kAhead; ++a) h.active[a] = rows_of(steps[c], a) * G;
        for (size_t k = 0; k < steps[c].size(); ++k) total += lane_bytes * G * rows_of(steps[c], k);
    }
    return total;
}

// pl, pu: every chunk's plans for W wavefronts, G lanes a row, S entries a lane
template <class T, int S>
void build_steps(const HostSweep &lo, const HostSweep &up, const ChunkSet &C, int W, int G,
                 const std::vector<LanePlan> &pl, const std::vector<LanePlan> &pu, LaneSweep<T> &L) {
    std::vector<LaneHead> head(C.nchunk);
    std::vector<std::vector<StepRef>> steps(C.nchunk);
    parallel_for(C.nchunk, 1, [&](size_t c0, size_t c1) {
        for (size_t c = c0; c < c1; ++c) {
            append_steps(lo, pl[c], steps[c]);
            head[c].rounds_lo = (uint32_t)steps[c].size() / kAhead;
            append_steps(up, pu[c], steps[c]);
            head[c].rounds_up = (uint32_t)steps[c].size() / kAhead - head[c].rounds_lo;
        }
    });
    constexpr size_t kLane = (size_t)Step<T, S>::kPieces * 16;
    const uint64_t total = place_steps<LaneHead>(steps, G, kLane, head, [](LaneHead &h) -> LaneHead & { return h; });
    // the loads past the last chunk's steps: kAhead steps of one row
    const uint64_t spare = kLane * G * kAhead;
    std::unique_ptr<unsigned char[]> host(new unsigned char[total + spare]);
    std::memset(host.get() + total, 0, spare);
    parallel_for(C.nchunk, 1, [&](size_t c0, size_t c1) {
        for (size_t c = c0; c < c1; ++c) {
            const uint32_t r0 = C.start[c], nr = C.start[c + 1] - r0;
            unsigned char *p = host.get() + head[c].first;
            for (size_t k = 0; k < steps[c].size(); ++k) {
                write_step<T, S>(steps[c][k], r0, nr, G, rows_of(steps[c], k + kAhead), p,
                                 [r0](uint32_t j) { return j - r0; }, [](uint32_t) { return kNoExport; });
                p += kLane * G * rows_of(steps[c], k);
            }
        }
    });
    L.data = dalloc<unsigned char>(total + spare);
    L.head = (LaneHead *)dalloc<unsigned char>(std::max<size_t>(1, head.size()) * sizeof(LaneHead));
    PP_HIP(hipMemcpy(L.data, host.get(), total + spare, hipMemcpyHostToDevice));
    PP_HIP(hipMemcpy(L.head, head.data(), head.size() * sizeof(LaneHead), hipMemcpyHostToDevice));
    L.waves = W;
    L.group = G;
    L.slots = S;
    L.mode_lo = lo.mode;
    L.mode_up = up.mode;
}

// LDS words of the largest strip: its rows, a zero, the rows it imports.
uint32_t strip_words(const HostSweep &s, const std::vector<uint32_t> &start) {
    std::vector<uint32_t> words(start.size() - 1);
    parallel_for(words.size(), 1, [&](size_t k0, size_t k1) {
        std::vector<uint32_t> seen(s.n, 0);  // the last strip of this thread that reads the row, + 1
        for (size_t k = k0; k < k1; ++k) {
            words[k] = start[k + 1] - start[k] + 1;
            for (uint32_t e = s.rp[start[k]]; e < s.rp[start[k + 1]]; ++e) {
                const uint32_t j = s.ci[e];
                if ((j < start[k] || j >= start[k + 1]) && seen[j] != k + 1) {
                    seen[j] = (uint32_t)k + 1;
                    ++words[k];
                }
            }
        }
    });
    return *std::max_element(words.begin(), words.end());
}

// One sweep's strips, on the host.
template <class T>
struct StripHost {
    std::vector<StripHead> head;
    std::vector<uint32_t> imp;
    std::unique_ptr<unsigned char[]> data;
    uint64_t bytes = 0;
    uint32_t nslots = 0, max_words = 0, span = 0;
};

template <class T, int S>
void build_strips_host(const HostSweep &s, const std::vector<uint32_t> &start, int G, StripHost<T> &D) {
    const uint32_t K = (uint32_t)start.size() - 1, n = s.n;
    std::vector<LanePlan> P = plan_steps(s, start, 64 / G, G * S, D.span);
    std::vector<StripHead> &head = D.head;
    head.resize(K);
    std::vector<std::vector<StepRef>> steps(K);
    std::vector<std::vector<uint32_t>> imports(K);  // rows, in the order their values are needed
    std::vector<std::unordered_map<uint32_t, uint32_t>> word(K);
    parallel_for(K, 1, [&](size_t k0, size_t k1) {
        for (size_t k = k0; k < k1; ++k) {
            const uint32_t r0 = start[k], r1 = start[k + 1], nr = r1 - r0;
            for (const auto &g : P[k].steps) {
                for (uint32_t u = g.first; u < g.first + g.count; ++u) {
                    const Part &q = P[k].parts[u];
                    for (uint32_t e = q.a; e < q.b; ++e) {
                        const uint32_t j = s.ci[e];
                        if (j >= r0 && j < r1) continue;
                        if (word[k].emplace(j, nr + 1 + (uint32_t)imports[k].size()).second) imports[k].push_back(j);
                    }
                }
                steps[k].push_back({&s, &P[k], g, ((uint32_t)imports[k].size() + kNeedUnit - 1) / kNeedUnit});
            }
            while (steps[k].size() % kAhead) steps[k].push_back({});
        }
    });
    // exchange slots: each strip's imported rows, numbered in the order its
    // steps finish them
    constexpr uint32_t kUnused = 0xffffffffu, kUsed = 0xfffffffeu;
    std::vector<uint32_t> slot(n, kUnused);
    for (uint32_t k = 0; k < K; ++k)
        for (uint32_t j : imports[k]) slot[j] = kUsed;
    for (uint32_t k = 0; k < K; ++k) {
        head[k].row = start[k];
        head[k].rows = start[k + 1] - start[k];
        head[k].exp = D.nslots;
        for (const Part &q : P[k].parts)
            if (q.last && slot[q.row] == kUsed) slot[q.row] = D.nslots++;
    }
    for (uint32_t k = 0; k < K; ++k) {
        head[k].imp = (uint32_t)D.imp.size();
        head[k].nimp = (uint32_t)imports[k].size();
        for (uint32_t j : imports[k]) D.imp.push_back(slot[j]);
        D.max_words = std::max(D.max_words, head[k].rows + 1 + head[k].nimp);
        head[k].lanes.rounds_lo = (uint32_t)steps[k].size() / kAhead;
    }
    constexpr size_t kLane = (size_t)Step<T, S>::kPieces * 16;
    const uint64_t total = place_steps<StripHead>(steps, G, kLane, head, [](StripHead &h) -> LaneHead & { return h.lanes; });
    const uint64_t spare = kLane * G * kAhead;
    D.bytes = total + spare;
    D.data.reset(new unsigned char[D.bytes]);
    std::memset(D.data.get() + total, 0, spare);
    parallel_for(K, 1, [&](size_t k0, size_t k1) {
        for (size_t k = k0; k < k1; ++k) {
            const uint32_t r0 = start[k], r1 = start[k + 1], exp0 = head[k].exp;
            const auto &w = word[k];
            unsigned char *p = D.data.get() + head[k].lanes.first;
            for (size_t q = 0; q < steps[k].size(); ++q) {
                write_step<T, S>(
                    steps[k][q], r0, r1 - r0, G, rows_of(steps[k], q + kAhead), p,
                    [&](uint32_t j) { return j >= r0 && j < r1 ? j - r0 : w.find(j)->second; },
                    [&](uint32_t j) { return slot[j] == kUnused ? kNoExport : slot[j] - exp0; });
                p += kLane * G * rows_of(steps[k], q);
            }
        }
    });
    if (!s.lower) std::reverse(head.begin(), head.end());  // workgroups in the sweep's direction
}

template <class T>
void upload_strips(const StripHost<T> &H, int mode, StripSide<T> &D) {
    auto up = [](const void *src, size_t bytes) {
        unsigned char *d = dalloc<unsigned char>(std::max<size_t>(16, bytes));
        if (bytes) PP_HIP(hipMemcpy(d, src, bytes, hipMemcpyHostToDevice));
        return d;
    };
    D.data = up(H.data.get(), H.bytes);
    D.head = up(H.head.data(), H.head.size() * sizeof(StripHead));
    D.imp = (uint32_t *)up(H.imp.data(), H.imp.size() * 4);
    D.nslots = H.nslots;
    D.max_words = H.max_words;
    D.mode = mode;
}

// slots: this sweep's exchange buffer; other, on: the other sweep's, to be emptied
template <class T>
void launch_strip_side(pp_ctx *ctx, const StripSweep<T> &L, const StripSide<T> &D, T *slots, uint32_t on, T *other,
                       const T *x, T *y) {
    const uint32_t ctl_off = (uint32_t)((L.max_words * sizeof(T) + 15) / 16 * 16);
    const size_t lds = ctl_off + kStripCtl;
    PP_CHECK(lds <= ctx->max_lds && D.data, PP_ERR_INVALID, "strip sweep: storage missing or strip exceeds LDS");
    bool launched = false;
#define PP_STRIP(G, S, MODE)                                                                                      \
    if (L.group == G && L.slots == S && D.mode == HostSweep::MODE) {                                              \
        launched = true;                                                                                          \
        if (lds > 65536)                                                                                          \
            PP_HIP(hipFuncSetAttribute((const void *)k_sweep_strips<T, G, S, HostSweep::MODE>,                    \
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                    \
        k_sweep_strips<T, G, S, HostSweep::MODE><<<L.nstrip, kLaneThreads, lds, ctx->stream>>>(                   \
            (const StripHead *)D.head, (const char *)D.data, D.imp, slots, on, other, ctl_off, x, y,             \
            ctx->spin_deadline, ctx->ctl, ctx->late_dev, ctx->stop_word);                                                      \
    }
#define PP_STRIPS(G, S)          \
    PP_STRIP(G, S, DIVIDE)       \
    PP_STRIP(G, S, UNIT)         \
    PP_STRIP(G, S, MULTIPLY)     \
    PP_STRIP(G, S, PREDIVIDE)
    PP_STRIPS(1, 8)
    PP_STRIPS(2, 8)
    PP_STRIPS(4, 8)
#undef PP_STRIPS
#undef PP_STRIP
    PP_CHECK(launched, PP_ERR_UNSUPPORTED, "strip sweep: no kernel of this step shape and diagonal mode");
    PP_HIP(hipGetLastError());
}

}  // namespace

template <class T>
void LaneSweep<T>::free_all() {
    dfree(head);
    dfree(data);
    head = nullptr;
    data = nullptr;
    waves = group = slots = 0;
}
template struct LaneSweep<double>;
template struct LaneSweep<float>;

uint32_t lane_sweep_max_rows(size_t lds) {
    return (uint32_t)std::min<size_t>(lds / sizeof(double) - kExtra, 65535 - kExtra);
}

// The shapes of a step, and what one took on MI355X (us, FP64: ICT(1e-3) and
// ICT(1e-2) of the 128^2 Poisson problem, ICT(3e-3) of 27^3, ILDLT of 16
// blocks; without divisions 0.03 less, FP32 5 to 10% less).  About half of a
// step is fixed work (loads, addresses: 40 instructions of about four cycles
// each), shared by the rows and entries it holds; one wavefront needs no
// barrier, four pay about 0.1 us for it and win where many rows are ready at
// a time.  So the shape that needs the fewest steps for its price wins:
//   128^2 ICT(1e-3), 1012 levels of 16 rows, 13 entries a row, apply in us:
//     {1,1,4} 500, {1,1,8} 514, {1,4,4} 415, {1,2,8} 459, {4,4,4} 602
//   128^2 ICT(1e-2), 509 levels of 32 rows, 4 entries: 138, 192, 387, 272, 304
//   27^3 ICT(3e-3), 312 levels of 63 rows, 12 entries: 257, 251, 450, 289, 211
// Levels of hundreds of rows take the whole workgroup, a lane a row, {4,1,4}
// (with one workgroup's 1024 threads a level and two barriers, in brackets):
//   IC(0) in colour order, 4 levels: 140^2 96 -> 48 us (49), 27^3 128 -> 63 (58)
//   ILUT(5, 0.1) in colour order, 27^3, 43 levels: 131 -> 59 (85)
//   27^3 ICT(0.1), 158 levels, 3 entries: 94 -> 55 (184); ICT(1e-2): 135 -> 111
struct LaneShape {
    int waves, group, slots;
    float us;
};
constexpr LaneShape kShapes[] = {{1, 1, 4, 0.125f}, {1, 1, 8, 0.18f}, {1, 4, 4, 0.18f},
                                 {1, 2, 8, 0.22f},  {1, 4, 8, 0.30f}, {4, 4, 4, 0.27f},
                                 {4, 1, 4, 0.21f}};

// The fewest steps a sweep's rows [r0, r1) can take: the longest chain of
// parts, the parts over the width.
uint32_t fewest_steps(const HostSweep &s, uint32_t r0, uint32_t r1, uint32_t width, uint32_t entries) {
    const uint32_t n = r1 - r0;
    std::vector<uint32_t> level(n, 0);
    uint64_t parts = 0;
    uint32_t chain = 0;
    for (uint32_t k = 0; k < n; ++k) {
        const uint32_t i = s.lower ? k : n - 1 - k, e0 = s.rp[r0 + i], e1 = s.rp[r0 + i + 1];
        const uint32_t m = std::max(1u, (e1 - e0 + entries - 1) / entries);
        uint32_t a = e0, b = e1 - (m - 1) * entries, l = 0;
        for (uint32_t q = 0; q < m; ++q, a = b, b += entries) {
            for (uint32_t e = a; e < b; ++e) l = std::max(l, level[s.ci[e] - r0]);
            ++l;
        }
        level[i] = l;
        chain = std::max(chain, l);
        parts += m;
    }
    return std::max<uint32_t>(chain, (uint32_t)((parts + width - 1) / width));
}

template <class T>
void build_lane_sweep(const HostSweep &lo, const HostSweep &up, const ChunkSet &C, LaneSweep<T> &L) {
    L.free_all();
    constexpr size_t K = sizeof(kShapes) / sizeof(kShapes[0]);
    // plans: the chunks' plans of the shape (lower, upper), else (NULL) only
    // the fewest steps they can take; chunks share the 256 compute units
    // (a small factor's plans take less time than starting threads for them)
    using Plans = std::vector<LanePlan>[2];
    const size_t grain = lo.rp[lo.n] + up.rp[up.n] < 1u << 16 ? 2 * C.nchunk : 1;
    const auto price = [&](const LaneShape &h, Plans *plans) {
        const HostSweep *sweep[2] = {&lo, &up};
        std::vector<uint32_t> steps(2 * C.nchunk, 0);
        if (plans)
            for (auto &p : *plans) p.resize(C.nchunk);
        parallel_for(2 * C.nchunk, grain, [&](size_t q0, size_t q1) {
            for (size_t q = q0; q < q1; ++q) {
                const uint32_t c = q / 2, width = 64 * h.waves / h.group, entries = h.group * h.slots;
                if (plans)
                    (*plans)[q % 2][c] =
                        std::move(plan_steps(*sweep[q % 2], {C.start[c], C.start[c + 1]}, width, entries, steps[q])[0]);
                else
                    steps[q] = fewest_steps(*sweep[q % 2], C.start[c], C.start[c + 1], width, entries);
            }
        });
        double longest = 0, total = 0;
        for (size_t q = 0; q < steps.size(); q += 2) {
            longest = std::max(longest, (double)steps[q] + steps[q + 1]);
            total += (double)steps[q] + steps[q + 1];
        }
        return std::max(longest, total / 256) * h.us;
    };
    // shapes by their least price; planned until none left can be cheaper
    std::vector<std::pair<double, size_t>> least(K);
    for (size_t k = 0; k < K; ++k) least[k] = {price(kShapes[k], nullptr), k};
    std::sort(least.begin(), least.end());
    size_t best = K;
    double best_us = 0;
    Plans plans;
    for (size_t q = 0; q < K && (best == K || least[q].first < best_us); ++q) {
        Plans p;
        const double us = price(kShapes[least[q].second], &p);
        if (best == K || us < best_us) {
            best = least[q].second;
            best_us = us;
            for (int k = 0; k < 2; ++k) plans[k].swap(p[k]);
        }
    }
    const LaneShape &h = kShapes[best];
    if (h.slots == 4) build_steps<T, 4>(lo, up, C, h.waves, h.group, plans[0], plans[1], L);
    else build_steps<T, 8>(lo, up, C, h.waves, h.group, plans[0], plans[1], L);
}
template void build_lane_sweep<double>(const HostSweep &, const HostSweep &, const ChunkSet &, LaneSweep<double> &);
template void build_lane_sweep<float>(const HostSweep &, const HostSweep &, const ChunkSet &, LaneSweep<float> &);

template <class T>
void launch_lane_sweep(pp_ctx *ctx, const ChunkSet &C, const LaneSweep<T> &L, const T *x, T *y) {
    const size_t lds = (size_t)(C.max_rows + kExtra) * sizeof(T);
    PP_CHECK(C.nchunk && L.data && lds <= ctx->max_lds, PP_ERR_INVALID,
             "chunked sweep: storage missing or chunk exceeds LDS");
    bool launched = false;
#define PP_LANES_M(W, G, S, MLO, MUP)                                                                          \
    if (L.mode_lo == HostSweep::MLO && L.mode_up == HostSweep::MUP) {                                          \
        launched = true;                                                                                       \
        if (lds > 65536)                                                                                       \
            PP_HIP(hipFuncSetAttribute(                                                                        \
                (const void *)k_sweep_lanes<T, W, G, S, HostSweep::MLO, HostSweep::MUP>,                       \
                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                                        \
        k_sweep_lanes<T, W, G, S, HostSweep::MLO, HostSweep::MUP><<<C.nchunk, kLaneThreads, lds, ctx->stream>>>( \
            C.dstart, L.head, (const char *)L.data, x, y, ctx->stop_word);                                     \
    }
#define PP_LANES(W, G, S)                           \
    if (L.waves == W && L.group == G && L.slots == S) { \
        PP_LANES_M(W, G, S, DIVIDE, DIVIDE)         \
        PP_LANES_M(W, G, S, UNIT, MULTIPLY)         \
        PP_LANES_M(W, G, S, UNIT, PREDIVIDE)        \
    }
    PP_LANES(1, 1, 4)
    PP_LANES(1, 1, 8)
    PP_LANES(1, 4, 4)
    PP_LANES(1, 2, 8)
    PP_LANES(1, 4, 8)
    PP_LANES(4, 4, 4)
    PP_LANES(4, 1, 4)
#undef PP_LANES
#undef PP_LANES_M
    PP_CHECK(launched, PP_ERR_UNSUPPORTED, "chunked sweep: no kernel of this step shape and diagonal modes");
    PP_HIP(hipGetLastError());
}
template void launch_lane_sweep<double>(pp_ctx *, const ChunkSet &, const LaneSweep<double> &, const double *,
                                        double *);
template void launch_lane_sweep<float>(pp_ctx *, const ChunkSet &, const LaneSweep<float> &, const float *, float *);

template <class T>
void StripSide<T>::free_all() {
    dfree(head);
    dfree(data);
    dfree(imp);
    head = data = nullptr;
    imp = nullptr;
    nslots = max_words = 0;
}
template <class T>
void StripSweep<T>::free_all() {
    lo.free_all();
    up.free_all();
    nstrip = max_words = 0;
}
template struct StripSweep<double>;
template struct StripSweep<float>;

// How many strips: more run more rows at a time, but the sweep passes through
// them one after another, a hop of about 10 steps each.  Rows over strips of
// about 14 sqrt(n) were within 5% of the best count everywhere it was
// measured (FP64 apply, us: ICT(1e-2) 64^3 32 strips 341, 20 378, 64 434;
// ILUT 50x43x31 16 strips 293, 8 416, 31 322; ICT(3e-3) 60x48x68 34 strips
// 608, 24 758, 68 717; ICT(1e-3) 400^2 16 strips 1861, 32 1958, 64 2116;
// ICT(1e-2) 100^3, where LDS asks for 100, 686, 128 731), unless LDS asks for
// more.  The lanes of a row by its mean entries, eight a lane (64^3, 7
// entries: one lane 347, two 520, four 904; 60x48x68, 12 entries: 692, 669,
// 1419; ILUT, 12 entries: 364, 280, 487).
template <class T>
bool build_strip_sweeps(pp_ctx *ctx, const HostSweep &lo, const HostSweep &up, StripSweep<T> &L) {
    L.free_all();
    const uint32_t n = lo.n;
    if (!n) return false;
    // the same cut in both precisions
    const uint32_t cap =
        std::min<uint32_t>((uint32_t)((ctx->max_lds - kStripCtl - 16) / sizeof(double)), 65535);
    std::vector<uint32_t> start;
    uint32_t K = std::max(2u, (uint32_t)(std::sqrt((double)n) / 14 + 0.5));
    K = std::min(n, std::max(K, n / cap + 1));
    for (;; K = std::min(n, K + K / 4 + 1)) {
        start.resize(K + 1);
        for (uint32_t k = 0; k <= K; ++k) start[k] = (uint32_t)((uint64_t)n * k / K);
        if (std::max(strip_words(lo, start), strip_words(up, start)) <= cap) break;
        if (K >= 1024 || K == n) return false;
    }
    const double mean = (double)std::max(lo.rp[n], up.rp[n]) / n;
    L.group = mean <= 8.5 ? 1 : mean <= 17 ? 2 : 4;
    L.slots = 8;
    StripHost<T> H[2];
    parallel_for(2, 1, [&](size_t a, size_t b) {
        for (size_t q = a; q < b; ++q) build_strips_host<T, 8>(q ? up : lo, start, L.group, H[q]);
    });
    upload_strips<T>(H[0], lo.mode, L.lo);
    upload_strips<T>(H[1], up.mode, L.up);
    L.nstrip = K;
    L.max_words = std::max(L.lo.max_words, L.up.max_words);
    strip_reserve(ctx, L);
    return true;
}
template bool build_strip_sweeps<double>(pp_ctx *, const HostSweep &, const HostSweep &, StripSweep<double> &);
template bool build_strip_sweeps<float>(pp_ctx *, const HostSweep &, const HostSweep &, StripSweep<float> &);

template <class T>
bool strip_reserve(pp_ctx *ctx, const StripSweep<T> &L) {
    pp_ctx::StripSlots *S = ctx->strip_slots[sizeof(T) == 4];
    const uint32_t want[2] = {L.lo.nslots, L.up.nslots};
    if (S[0].p && S[1].p && S[0].n >= want[0] && S[1].n >= want[1]) return true;
    if (ctx->arena) return false;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    PP_HIP(hipStreamIsCapturing(ctx->stream, &capturing));
    if (capturing != hipStreamCaptureStatusNone) return false;
    if (!ctx->strip_event) PP_HIP(hipEventCreateWithFlags(&ctx->strip_event, hipEventDisableTiming));
    for (int k = 0; k < 2; ++k) {
        if (S[k].p && S[k].n >= want[k]) continue;
        const uint32_t n = std::max({1024u, want[k], 2 * S[k].n});
        void *p = nullptr;  // not from the set-ups' block pool: it lives as long as the context
        if (hipMalloc(&p, (size_t)n * sizeof(T)) != hipSuccess) throw Error(PP_ERR_NOMEM, "strip exchange buffer");
        if (S[k].p) ctx->old_strip_slots.push_back(S[k].p);
        S[k] = {p, n};
        k_slots_empty<T><<<256, 256, 0, ctx->stream>>>(n, (T *)p);
        PP_HIP(hipGetLastError());
    }
    return true;
}
template bool strip_reserve<double>(pp_ctx *, const StripSweep<double> &);
template bool strip_reserve<float>(pp_ctx *, const StripSweep<float> &);

template <class T>
bool launch_strip_sweeps(pp_ctx *ctx, const StripSweep<T> &L, const T *x, T *y) {
    if (!strip_reserve(ctx, L)) return false;
    const pp_ctx::StripSlots *S = ctx->strip_slots[sizeof(T) == 4];
    T *lo = (T *)S[0].p, *up = (T *)S[1].p;
    ctx->strips_queued = true;
    launch_strip_side<T>(ctx, L, L.lo, lo, L.up.nslots, up, x, y);
    launch_strip_side<T>(ctx, L, L.up, up, L.lo.nslots, lo, y, y);
    return true;
}
template bool launch_strip_sweeps<double>(pp_ctx *, const StripSweep<double> &, const double *, double *);
template bool launch_strip_sweeps<float>(pp_ctx *, const StripSweep<float> &, const float *, float *);

}  // namespace pp
