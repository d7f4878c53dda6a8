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
// of a wavefront stay in order); a row is spread over several lanes, which
// gather and multiply its entries at once; every step's data comes in a
// ready-to-use layout, loaded kLaneAhead steps ahead; and divisions go by
// the pivots' reciprocals (five operations, same bits).  An apply of that
// factor takes 0.45 ms in FP64 (0.19 us a step); one workgroup barrier and
// one LDS round trip more per level, with data loaded one level ahead, took
// 2.0 ms (1.0 us a level).
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

// Flags of a step, the same in all its lanes: the first, the last of its rows' steps.
// From bit kNeedShift on: what a strip's step waits for (how many imports, in
// units of kNeedUnit, must be there before it).
enum : uint32_t { F_FIRST = 1, F_LAST = 2 };
constexpr int kNeedShift = 2;
constexpr uint32_t kNeedUnit = 8;

// What a lane needs of one step: 16-byte pieces, piece k of the step's
// `active` lanes contiguous, so every load is one coalesced 16-byte load per lane.
//   values   S values of T
//   indices  S 16-bit LDS words of the dependencies, then the row's word, the
//            flags, the step's active lanes, the active lanes kAhead steps later
//            and (S = 8) the row's 32-bit exchange slot or kNoSlot
//   pivot    the row's diagonal and its reciprocal rounded to FP64
constexpr uint32_t kNoSlot = 0xffffffffu;
template <class T, int S>
struct Step {
    static constexpr int kVal = S * (int)sizeof(T) / 16, kIdx = (2 * S + 8 + 15) / 16;
    static constexpr int kPieces = kVal + kIdx + 1;
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
constexpr int kRowShl = 0x100, kRowShr = 0x110;  // DPP: lane i takes lane i + n, i - n of its 16

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
        row = lds_byte<T, 0>(q.ix(S / 2));
    }
};

// Carried from step to step.
template <class T, int S>
struct Carry {
    StepAddr<T, S> addr;  // of the next step
    uint32_t flags;       // of the next step
    uint32_t active;      // lanes of the step kAhead - 1 past the next one
    T t;                  // the rows' sums after the last step
};

// Step k, its data in q: G lanes a row, S entries a lane, in storage order
// along the row's lanes.  Every lane gathers and multiplies its entries at
// once; the subtractions follow one after another, the partial sum moving
// from lane to lane (DPP), so the row's operations are those of the serial
// sweep.  The gathers go out first: while they are on their way, the loads
// of step k + kAhead - 1 (into `past`, step k - 1's slot) are issued and the
// next step's addresses unpacked.
// xchg.wait(need) returns once the step's imports are in LDS, xchg.put
// passes a finished row on.
template <class T, int W, int G, int S, int MODE, class Xchg>
__device__ inline void run_step(const Step<T, S> &q, const Step<T, S> &next, Step<T, S> &past, const char *&p,
                                Carry<T, S> &c, uint32_t lane, uint32_t tail_lane, Xchg &xchg) {
#pragma clang fp contract(off)
    const uint32_t flags = c.flags;
    xchg.wait(flags >> kNeedShift);
    T x[S];
#pragma unroll
    for (int j = 0; j < S; ++j) x[j] = *lds_word<T>(c.addr.dep[j]);
    LdsWord<T> *mine = lds_word<T>(c.addr.row);
    const T rhs = *mine;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    load_step<T, S>(past, p, c.active, lane);
    const uint32_t active = (uint32_t)__builtin_amdgcn_readfirstlane(q.ix(S / 2 + 1));
    c.addr.set(next);
    c.flags = (uint32_t)__builtin_amdgcn_readfirstlane(next.ix(S / 2)) >> 16;
    c.active = active >> 16;
    __builtin_amdgcn_sched_barrier(0);
    T s = rhs;
    if (flags & F_FIRST) {
        if constexpr (MODE == HostSweep::PREDIVIDE) s = quotient(s, q.d(), q.rcp());
    } else {
        if constexpr (G > 1) s = dpp<kRowShl + G - 1>(c.t);
        else s = c.t;
    }
#pragma unroll
    for (int j = 0; j < S; ++j) x[j] = q.v(j) * x[j];
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int j = 0; j < S; ++j) s = s - x[j];
        if (g < G - 1) s = dpp<kRowShr + 1>(s);
    }
    c.t = s;
    if (flags & F_LAST) {
        if constexpr (MODE == HostSweep::DIVIDE) s = quotient(s, q.d(), q.rcp());
        else if constexpr (MODE == HostSweep::MULTIPLY) s = s * q.d();
        if (tail_lane < (active & 0xffffu)) {
            *mine = s;
            xchg.put(q, s);
        }
        if constexpr (W > 1) __syncthreads();
    }
}

struct NoExchange {
    __device__ void wait(uint32_t) {}
    template <class Q, class T>
    __device__ void put(const Q &, T) {}
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
        st.t = 0;
        st.active = head[c].active[kAhead - 1];
        st.addr.set(q[0]);
        st.flags = (uint32_t)__builtin_amdgcn_readfirstlane(q[0].ix(S / 2)) >> 16;
        NoExchange no_xchg;
        for (uint32_t k = 0; k < lo; ++k) {
#pragma unroll
            for (int a = 0; a < kAhead; ++a)
                run_step<T, W, G, S, MLO>(q[a], q[(a + 1) % kAhead], q[(a + kAhead - 1) % kAhead], p, st, lane,
                                          tail_lane, no_xchg);
        }
        for (uint32_t k = 0; k < up; ++k) {
#pragma unroll
            for (int a = 0; a < kAhead; ++a)
                run_step<T, W, G, S, MUP>(q[a], q[(a + 1) % kAhead], q[(a + kAhead - 1) % kAhead], p, st, lane,
                                          tail_lane, no_xchg);
        }
    }
    __syncthreads();
    copy_rows(y + r0, xs, nr);
}

// Rows of one chunk in the order and grouping of its steps.
struct LanePlan {
    struct Group {
        uint32_t first, count, steps;  // rows[first, first + count), each taking `steps` steps
    };
    std::vector<uint32_t> rows;
    std::vector<Group> groups;
    uint32_t steps = 0;
};

// Groups the rows [r0, r1) of a sweep: a group holds at most `width` rows
// whose dependencies all lie in earlier groups, the rows with the longest
// chains behind them first (list scheduling), so the groups are about as few
// as the longest chain, or the rows over `width`, allows.  A row of more
// entries than one step takes runs over several steps; a group takes only
// rows of at most its first row's steps.
LanePlan plan_chunk(const HostSweep &s, uint32_t r0, uint32_t r1, uint32_t width, uint32_t entries) {
    const uint32_t n = r1 - r0;
    LanePlan P;
    std::vector<uint32_t> ns(n), wait(n), sp(n + 1, 0), sc, height(n, 0);
    for (uint32_t i = 0; i < n; ++i) {
        const uint32_t a = s.rp[r0 + i], b = s.rp[r0 + i + 1];
        ns[i] = std::max(1u, (b - a + entries - 1) / entries);
        wait[i] = b - a;
        for (uint32_t e = a; e < b; ++e) sp[s.ci[e] - r0 + 1]++;
    }
    for (uint32_t i = 0; i < n; ++i) sp[i + 1] += sp[i];
    sc.resize(sp[n]);
    {
        std::vector<uint32_t> at(sp.begin(), sp.end() - 1);
        for (uint32_t i = 0; i < n; ++i)
            for (uint32_t e = s.rp[r0 + i]; e < s.rp[r0 + i + 1]; ++e) sc[at[s.ci[e] - r0]++] = i;
    }
    // dependents of a row come after it (lower) or before it (upper)
    for (uint32_t k = 0; k < n; ++k) {
        const uint32_t i = s.lower ? n - 1 - k : k;
        uint32_t h = 0;
        for (uint32_t e = sp[i]; e < sp[i + 1]; ++e) h = std::max(h, height[sc[e]]);
        height[i] = h + ns[i];
    }
    auto less = [&](uint32_t a, uint32_t b) { return height[a] != height[b] ? height[a] < height[b] : a > b; };
    std::priority_queue<uint32_t, std::vector<uint32_t>, decltype(less)> ready(less);
    for (uint32_t i = 0; i < n; ++i)
        if (!wait[i]) ready.push(i);
    P.rows.reserve(n);
    std::vector<uint32_t> skipped;
    while (!ready.empty()) {
        LanePlan::Group g{(uint32_t)P.rows.size(), 0, ns[ready.top()]};
        skipped.clear();
        while (!ready.empty() && g.count < width) {
            const uint32_t i = ready.top();
            ready.pop();
            if (ns[i] > g.steps) {
                skipped.push_back(i);
                continue;
            }
            P.rows.push_back(i);
            ++g.count;
        }
        for (uint32_t i : skipped) ready.push(i);
        for (uint32_t k = g.first; k < g.first + g.count; ++k) {
            const uint32_t i = P.rows[k];
            for (uint32_t e = sp[i]; e < sp[i + 1]; ++e)
                if (--wait[sc[e]] == 0) ready.push(sc[e]);
        }
        P.groups.push_back(g);
        P.steps += g.steps;
    }
    return P;
}

// A chunk's steps: what each holds, before it is written out.
struct StepRef {
    const HostSweep *sweep;  // nullptr: idle (fills a sweep's last round)
    uint32_t row, count, part, parts;  // plan rows [row, row + count), step `part` of their `parts`
    const LanePlan *plan;
    uint32_t need;           // imports (kNeedUnit each) it waits for
};

void append_steps(const HostSweep &s, const LanePlan &P, std::vector<StepRef> &out) {
    for (const auto &g : P.groups)
        for (uint32_t k = 0; k < g.steps; ++k) out.push_back({&s, g.first, g.count, k, g.steps, &P, 0});
    while (out.size() % kAhead) out.push_back({nullptr, 0, 0, 0, 0, nullptr, 0});
}

// One step at `out` (zeroed), `active` lanes; ahead: the lanes kAhead steps later.
// word(row): the LDS word of a dependency; slot: the exchange slots of all
// rows (kNoSlot: none), or nullptr.
template <class T, int S, class Word>
void write_step(const StepRef &r, uint32_t r0, uint32_t nr, int G, uint32_t active, uint32_t ahead,
                unsigned char *out, const Word &word, const uint32_t *slot = nullptr) {
    using St = Step<T, S>;
    const size_t piece = (size_t)active * 16;
    for (uint32_t l = 0; l < active; ++l) {
        T v[S] = {}, d = T(1);
        uint16_t ix[St::kIdx * 8] = {};
        uint32_t flags = 0;
        if (r.sweep) {
            const HostSweep &s = *r.sweep;
            const uint32_t i = r.plan->rows[r.row + l / G];
            const uint32_t a = s.rp[r0 + i] + (r.part * G + l % G) * S, b = s.rp[r0 + i + 1];
            for (int j = 0; j < S; ++j) {
                const bool has = a + j < b;
                if (has) v[j] = (T)s.val[a + j];
                ix[j] = (uint16_t)(has ? word(s.ci[a + j]) : nr);  // word nr holds a zero
            }
            ix[S] = (uint16_t)i;
            if constexpr (S == 8) {
                const uint32_t to = slot ? slot[r0 + i] : kNoSlot;
                ix[S + 4] = (uint16_t)to;
                ix[S + 5] = (uint16_t)(to >> 16);
            }
            flags = (r.part == 0 ? F_FIRST : 0u) | (r.part + 1 == r.parts ? F_LAST : 0u);
            if (s.mode != HostSweep::UNIT) d = (T)s.diag[r0 + i];
        }
        ix[S + 1] = (uint16_t)(flags | r.need << kNeedShift);
        ix[S + 2] = (uint16_t)active;
        ix[S + 3] = (uint16_t)ahead;
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

template <class T, int S>
void build_steps(const HostSweep &lo, const HostSweep &up, const ChunkSet &C, int W, int G, LaneSweep<T> &L) {
    std::vector<LanePlan> pl(C.nchunk), pu(C.nchunk);
    std::vector<LaneHead> head(C.nchunk);
    std::vector<std::vector<StepRef>> steps(C.nchunk);
    auto lanes = [&](const std::vector<StepRef> &v, size_t k) {
        return k < v.size() && v[k].sweep ? v[k].count * (uint32_t)G : 1u;
    };
    parallel_for(C.nchunk, 1, [&](size_t c0, size_t c1) {
        for (size_t c = c0; c < c1; ++c) {
            pl[c] = plan_chunk(lo, C.start[c], C.start[c + 1], 64 * W / G, G * S);
            pu[c] = plan_chunk(up, C.start[c], C.start[c + 1], 64 * W / G, G * S);
            append_steps(lo, pl[c], steps[c]);
            head[c].rounds_lo = (uint32_t)steps[c].size() / kAhead;
            append_steps(up, pu[c], steps[c]);
            head[c].rounds_up = (uint32_t)steps[c].size() / kAhead - head[c].rounds_lo;
        }
    });
    constexpr size_t kLane = (size_t)Step<T, S>::kPieces * 16;
    uint64_t total = 0;
    for (uint32_t c = 0; c < C.nchunk; ++c) {
        head[c].first = total;
        for (int a = 0; a < kAhead; ++a) head[c].active[a] = lanes(steps[c], a);
        for (size_t k = 0; k < steps[c].size(); ++k) total += kLane * lanes(steps[c], k);
    }
    // the loads past the last chunk's steps: kAhead steps of one lane
    const uint64_t spare = kLane * kAhead;
    std::unique_ptr<unsigned char[]> host(new unsigned char[total + spare]);
    std::memset(host.get() + total, 0, spare);
    parallel_for(C.nchunk, 1, [&](size_t c0, size_t c1) {
        for (size_t c = c0; c < c1; ++c) {
            const uint32_t r0 = C.start[c], nr = C.start[c + 1] - r0;
            unsigned char *p = host.get() + head[c].first;
            for (size_t k = 0; k < steps[c].size(); ++k) {
                const uint32_t active = lanes(steps[c], k);
                write_step<T, S>(steps[c][k], r0, nr, G, active, lanes(steps[c], k + kAhead), p,
                                 [r0](uint32_t j) { return j - r0; });
                p += kLane * active;
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

// ---------------------------------------------------------------------------
// Strips: the sweeps of a factor whose rows do not chunk (one connected part
// larger than LDS).  The rows are cut into contiguous strips, a workgroup and
// its LDS each; wavefront 0 runs the strip's steps.  A finished row that
// other strips read goes from its lane's register straight to the row's slot
// of an exchange buffer (agent-scope store); in the strips that read it, the
// other wavefronts poll the slots in the order the steps need them and put the
// values into LDS.  A slot holds a signalling NaN, which no sum is, until its
// value arrives, so a value is its own ready flag (a value passes between
// two compute units in about 0.6 us, 0.45 on one XCD).  The slots of one
// sweep are emptied while the other runs.
// A strip waits only for strips before it in its sweep's direction, whose
// workgroups are dispatched before its own, so the first unfinished strip
// always proceeds; a wait past the deadline sets C_SPIN, and every wavefront
// runs to its end (the rows become NaN).
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
};

// control words in LDS (not through a generic pointer: a flat access would
// wait for every step in flight)
using CtlWord = volatile __attribute__((address_space(3))) uint32_t;

// Wavefront 0's side of the exchange.
template <class T>
struct Exchange {
    CtlWord *cw;
    T *slots;
    uint32_t have;  // imports known to be in LDS
    __device__ void wait(uint32_t need) {
        while (have < need * kNeedUnit) {
            uint32_t done = 0xffffffffu;
#pragma unroll
            for (int f = 0; f < kImport; ++f) done = min(done, cw[f]);
            if (cw[CW_ABORT]) done = 0xffffffffu;
            have = (uint32_t)__builtin_amdgcn_readfirstlane(done);
        }
    }
    template <class Q>
    __device__ void put(const Q &q, T s) {
        using U = typename SlotBits<T>::U;
        const uint32_t to = (uint32_t)q.ix(6);
        if (to != kNoSlot)
            __hip_atomic_store(reinterpret_cast<U *>(slots) + to, __builtin_bit_cast(U, s), __ATOMIC_RELAXED,
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
    uint32_t other_n, T *other, uint32_t ctl_off, const T *x, T *y, long long deadline, int *ctl, const int *stop) {
    static_assert(S == 8, "the steps carry exchange slots");
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
        st.t = 0;
        st.active = h.lanes.active[kAhead - 1];
        st.addr.set(q[0]);
        st.flags = (uint32_t)__builtin_amdgcn_readfirstlane(q[0].ix(S / 2)) >> 16;
        Exchange<T> xchg{cw, slots, 0};
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
        const long long t0 = wall_clock64();
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
                    }
                    const unsigned long long m = __ballot(wait[b]);
                    if (m) seen = b * 64 + __builtin_ctzll(m);
                }
                asm volatile("" ::: "memory");
                // all of them: the next one to see is the next batch's first
                cw[f] = i0 + (seen < kBatch * 64 ? seen : kImport * kBatch * 64);
                if (seen == kBatch * 64) break;
                if ((iter & 63) == 0 && (wall_clock64() - t0 > deadline ||
                                         __hip_atomic_load(&ctl[C_SPIN], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
                    atomicOr(&ctl[C_SPIN], 1);
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

// The strips' plans: list scheduling of all strips together, a step of every
// strip at a time, a row of another strip visible kStripLag steps after its
// step (the exchange takes about 1.5 us), so that the order in which a strip
// takes its rows is one in which it rarely waits.
constexpr uint32_t kStripLag = 10;
std::vector<LanePlan> plan_strips(const HostSweep &s, const std::vector<uint32_t> &start, uint32_t width,
                                  uint32_t entries) {
    const uint32_t n = s.n, K = (uint32_t)start.size() - 1;
    std::vector<LanePlan> P(K);
    std::vector<uint32_t> sp(n + 1, 0), sc(s.rp[n]), height(n, 0), ns(n), strip_of(n);
    std::vector<int32_t> wait(n);
    std::vector<uint32_t> at_time(n, 0);  // when the dependencies seen so far are visible
    for (uint32_t k = 0; k < K; ++k) std::fill(strip_of.begin() + start[k], strip_of.begin() + start[k + 1], k);
    for (uint32_t i = 0; i < n; ++i) {
        wait[i] = (int32_t)(s.rp[i + 1] - s.rp[i]);
        ns[i] = std::max(1u, ((uint32_t)wait[i] + entries - 1) / entries);
        for (uint32_t e = s.rp[i]; e < s.rp[i + 1]; ++e) sp[s.ci[e] + 1]++;
    }
    for (uint32_t i = 0; i < n; ++i) sp[i + 1] += sp[i];
    {
        std::vector<uint32_t> at(sp.begin(), sp.end() - 1);
        for (uint32_t i = 0; i < n; ++i)
            for (uint32_t e = s.rp[i]; e < s.rp[i + 1]; ++e) sc[at[s.ci[e]]++] = i;
    }
    for (uint32_t k = 0; k < n; ++k) {
        const uint32_t i = s.lower ? n - 1 - k : k;
        uint32_t h = 0;
        for (uint32_t e = sp[i]; e < sp[i + 1]; ++e)
            h = std::max(h, height[sc[e]] + (strip_of[sc[e]] != strip_of[i] ? kStripLag : 0u));
        height[i] = h + ns[i];
    }
    auto less = [&](uint32_t a, uint32_t b) { return height[a] != height[b] ? height[a] < height[b] : a > b; };
    std::vector<std::vector<uint32_t>> ready(K), due;  // due[t]: rows whose dependencies are visible at step t
    std::vector<uint32_t> busy(K, 0);
    auto make_due = [&](uint32_t i, uint32_t t) {
        if (t >= due.size()) due.resize(t + 1 + t / 2);
        due[t].push_back(i);
    };
    for (uint32_t i = 0; i < n; ++i)
        if (!wait[i]) make_due(i, 0);
    std::vector<uint32_t> skipped, group;
    uint32_t left = n;
    for (uint32_t t = 0; left; ++t) {
        if (t < due.size()) {
            std::vector<uint32_t> now;
            now.swap(due[t]);
            for (uint32_t i : now) {
                auto &q = ready[strip_of[i]];
                q.push_back(i);
                std::push_heap(q.begin(), q.end(), less);
            }
        }
        for (uint32_t k = 0; k < K; ++k) {
            auto &q = ready[k];
            if (busy[k] > t || q.empty()) continue;
            LanePlan &p = P[k];
            LanePlan::Group g{(uint32_t)p.rows.size(), 0, ns[q.front()]};
            skipped.clear();
            while (!q.empty() && g.count < width) {
                std::pop_heap(q.begin(), q.end(), less);
                const uint32_t i = q.back();
                q.pop_back();
                if (ns[i] > g.steps) {
                    skipped.push_back(i);
                    if (skipped.size() > 64) break;
                    continue;
                }
                p.rows.push_back(i - start[k]);
                ++g.count;
            }
            for (uint32_t i : skipped) {
                q.push_back(i);
                std::push_heap(q.begin(), q.end(), less);
            }
            busy[k] = t + g.steps;
            left -= g.count;
            for (uint32_t r = g.first; r < g.first + g.count; ++r) {
                const uint32_t i = p.rows[r] + start[k];
                for (uint32_t e = sp[i]; e < sp[i + 1]; ++e) {
                    const uint32_t j = sc[e], vis = t + g.steps + (strip_of[j] != k ? kStripLag : 0u);
                    at_time[j] = std::max(at_time[j], vis);
                    if (--wait[j] == 0) make_due(j, std::max(at_time[j], t + 1));
                }
            }
            p.groups.push_back(g);
            p.steps += g.steps;
        }
    }
    return P;
}


// LDS words of the largest strip: its rows, a zero, the rows it imports.
uint32_t strip_words(const HostSweep &s, const std::vector<uint32_t> &start) {
    std::vector<uint32_t> words(start.size() - 1);
    parallel_for(words.size(), 1, [&](size_t k0, size_t k1) {
        std::vector<uint32_t> remote;
        for (size_t k = k0; k < k1; ++k) {
            remote.clear();
            for (uint32_t e = s.rp[start[k]]; e < s.rp[start[k + 1]]; ++e)
                if (s.ci[e] < start[k] || s.ci[e] >= start[k + 1]) remote.push_back(s.ci[e]);
            std::sort(remote.begin(), remote.end());
            const size_t n = std::unique(remote.begin(), remote.end()) - remote.begin();
            words[k] = start[k + 1] - start[k] + 1 + (uint32_t)n;
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
    uint32_t nslots = 0, max_words = 0;
};

template <class T, int S>
void build_strips_host(const HostSweep &s, const std::vector<uint32_t> &start, int G, StripHost<T> &D) {
    const uint32_t K = (uint32_t)start.size() - 1, n = s.n;
    std::vector<LanePlan> P = plan_strips(s, start, 64 / G, G * S);
    std::vector<StripHead> &head = D.head;
    head.resize(K);
    std::vector<std::vector<StepRef>> steps(K);
    std::vector<std::vector<uint32_t>> imports(K);          // rows, in the order their values are needed
    std::vector<std::unordered_map<uint32_t, uint32_t>> word(K);
    parallel_for(K, 1, [&](size_t k0, size_t k1) {
        for (size_t k = k0; k < k1; ++k) {
            const uint32_t r0 = start[k], r1 = start[k + 1], nr = r1 - r0;
            for (const auto &g : P[k].groups) {
                for (uint32_t r = g.first; r < g.first + g.count; ++r) {
                    const uint32_t i = r0 + P[k].rows[r];
                    for (uint32_t e = s.rp[i]; e < s.rp[i + 1]; ++e) {
                        const uint32_t j = s.ci[e];
                        if (j >= r0 && j < r1) continue;
                        if (word[k].emplace(j, nr + 1 + (uint32_t)imports[k].size()).second) imports[k].push_back(j);
                    }
                }
                const uint32_t need = ((uint32_t)imports[k].size() + kNeedUnit - 1) / kNeedUnit;
                for (uint32_t q = 0; q < g.steps; ++q) steps[k].push_back({&s, g.first, g.count, q, g.steps, &P[k], need});
            }
            while (steps[k].size() % kAhead)
                steps[k].push_back({nullptr, 0, 0, 0, 0, nullptr, 0});
        }
    });
    // exchange slots: the imported rows, numbered strip by strip in the order
    // their steps finish them
    std::vector<uint32_t> slot(n, kNoSlot);
    std::vector<uint32_t> &imp = D.imp;
    uint32_t &nslots = D.nslots;
    for (uint32_t k = 0; k < K; ++k)
        for (uint32_t j : imports[k]) slot[j] = kNoSlot - 1;  // to be numbered
    for (uint32_t k = 0; k < K; ++k) {
        head[k].row = start[k];
        head[k].rows = start[k + 1] - start[k];
        for (uint32_t r : P[k].rows)
            if (slot[start[k] + r] != kNoSlot) slot[start[k] + r] = nslots++;
    }
    for (uint32_t k = 0; k < K; ++k) {
        head[k].imp = (uint32_t)imp.size();
        head[k].nimp = (uint32_t)imports[k].size();
        for (uint32_t j : imports[k]) imp.push_back(slot[j]);
        D.max_words = std::max(D.max_words, head[k].rows + 1 + head[k].nimp);
    }
    constexpr size_t kLane = (size_t)Step<T, S>::kPieces * 16;
    auto lanes = [&](const std::vector<StepRef> &v, size_t k) {
        return k < v.size() && v[k].sweep ? v[k].count * (uint32_t)G : 1u;
    };
    uint64_t total = 0;
    for (uint32_t k = 0; k < K; ++k) {
        LaneHead &h = head[k].lanes;
        h.first = total;
        h.rounds_lo = (uint32_t)steps[k].size() / kAhead;
        for (int a = 0; a < kAhead; ++a) h.active[a] = lanes(steps[k], a);
        for (size_t q = 0; q < steps[k].size(); ++q) total += kLane * lanes(steps[k], q);
    }
    const uint64_t spare = kLane * kAhead;
    D.bytes = total + spare;
    D.data.reset(new unsigned char[D.bytes]);
    std::memset(D.data.get() + total, 0, spare);
    parallel_for(K, 1, [&](size_t k0, size_t k1) {
        for (size_t k = k0; k < k1; ++k) {
            const uint32_t r0 = start[k], r1 = start[k + 1];
            const auto &w = word[k];
            unsigned char *p = D.data.get() + head[k].lanes.first;
            for (size_t q = 0; q < steps[k].size(); ++q) {
                const uint32_t active = lanes(steps[k], q);
                write_step<T, S>(steps[k][q], r0, r1 - r0, G, active, lanes(steps[k], q + kAhead), p, [&](uint32_t j) {
                    return j >= r0 && j < r1 ? j - r0 : w.find(j)->second;
                }, slot.data());
                p += kLane * active;
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
    D.slots = dalloc<T>(std::max(1u, H.nslots));
    D.max_words = H.max_words;
    D.mode = mode;
}

template <class T>
void launch_strip_side(pp_ctx *ctx, const StripSweep<T> &L, const StripSide<T> &D, const StripSide<T> &O, const T *x,
                       T *y) {
    const uint32_t ctl_off = (uint32_t)((L.max_words * sizeof(T) + 15) / 16 * 16);
    const size_t lds = ctl_off + kStripCtl;
    PP_CHECK(lds <= ctx->max_lds && D.data, PP_ERR_INVALID, "strip sweep: storage missing or strip exceeds LDS");
#define PP_STRIP(G, S, MODE)                                                                                      \
    if (L.group == G && L.slots == S && D.mode == HostSweep::MODE) {                                              \
        if (lds > 65536)                                                                                          \
            PP_HIP(hipFuncSetAttribute((const void *)k_sweep_strips<T, G, S, HostSweep::MODE>,                    \
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                    \
        k_sweep_strips<T, G, S, HostSweep::MODE><<<L.nstrip, kLaneThreads, lds, ctx->stream>>>(                   \
            (const StripHead *)D.head, (const char *)D.data, D.imp, D.slots, O.nslots, O.slots, \
            ctl_off, x, y, ctx->spin_deadline, ctx->ctl, ctx->stop_word);                                \
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

// The shapes of a step, and what one took on MI355X (us; single wave of
// 2.4 GHz; ICT(1e-3) and ICT(1e-2) of the 128^2 Poisson problem, ICT(3e-3) of
// 27^3, 4 to 13 entries a row; FP32 5 to 10% less).  One wavefront needs no
// barrier; four pay about 0.1 us for it, and win where levels are wide.  A
// lane's fixed work (loads, addresses, flags: about 50 instructions, which
// issue one in four cycles) is shared by the rows and entries a step holds,
// so the shape that needs the fewest steps for its price wins.
struct LaneShape {
    int waves, group, slots;
    float us;
};
constexpr LaneShape kShapes[] = {{1, 4, 4, 0.19f}, {1, 2, 8, 0.23f}, {1, 1, 8, 0.18f}, {4, 4, 4, 0.29f}, {4, 2, 4, 0.21f}};

template <class T>
void build_lane_sweep(const HostSweep &lo, const HostSweep &up, const ChunkSet &C, LaneSweep<T> &L) {
    L.free_all();
    // every shape's steps; chunks share the 256 compute units
    constexpr size_t K = sizeof(kShapes) / sizeof(kShapes[0]);
    std::vector<uint32_t> steps(K * C.nchunk);
    parallel_for(K * C.nchunk, 1, [&](size_t q0, size_t q1) {
        for (size_t q = q0; q < q1; ++q) {
            const LaneShape &h = kShapes[q % K];
            const uint32_t r0 = C.start[q / K], r1 = C.start[q / K + 1];
            steps[q] = plan_chunk(lo, r0, r1, 64 * h.waves / h.group, h.group * h.slots).steps +
                       plan_chunk(up, r0, r1, 64 * h.waves / h.group, h.group * h.slots).steps;
        }
    });
    size_t best = 0;
    double best_us = 0;
    for (size_t k = 0; k < K; ++k) {
        double longest = 0, total = 0;
        for (uint32_t c = 0; c < C.nchunk; ++c) {
            longest = std::max(longest, (double)steps[c * K + k]);
            total += steps[c * K + k];
        }
        const double us = std::max(longest, total / 256) * kShapes[k].us;
        if (k == 0 || us < best_us) {
            best = k;
            best_us = us;
        }
    }
    const LaneShape &h = kShapes[best];
    if (h.slots == 4) build_steps<T, 4>(lo, up, C, h.waves, h.group, L);
    else build_steps<T, 8>(lo, up, C, h.waves, h.group, L);
}
template void build_lane_sweep<double>(const HostSweep &, const HostSweep &, const ChunkSet &, LaneSweep<double> &);
template void build_lane_sweep<float>(const HostSweep &, const HostSweep &, const ChunkSet &, LaneSweep<float> &);

template <class T>
void launch_lane_sweep(pp_ctx *ctx, const ChunkSet &C, const LaneSweep<T> &L, const T *x, T *y) {
    const size_t lds = (size_t)(C.max_rows + kExtra) * sizeof(T);
    PP_CHECK(C.nchunk && L.data && lds <= ctx->max_lds, PP_ERR_INVALID,
             "chunked sweep: storage missing or chunk exceeds LDS");
#define PP_LANES_M(W, G, S, MLO, MUP)                                                                          \
    if (L.mode_lo == HostSweep::MLO && L.mode_up == HostSweep::MUP) {                                          \
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
    PP_LANES(1, 4, 4)
    PP_LANES(1, 2, 8)
    PP_LANES(1, 1, 8)
    PP_LANES(4, 4, 4)
    PP_LANES(4, 2, 4)
#undef PP_LANES
#undef PP_LANES_M
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
    dfree(slots);
    head = data = nullptr;
    imp = nullptr;
    slots = nullptr;
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
// entries: one lane 341, two 517; 60x48x68, 12 entries: 801, 608, four 1208).
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
    for (StripSide<T> *D : {&L.lo, &L.up}) {
        k_slots_empty<T><<<256, 256, 0, ctx->stream>>>(D->nslots, D->slots);
        PP_HIP(hipGetLastError());
    }
    return true;
}
template bool build_strip_sweeps<double>(pp_ctx *, const HostSweep &, const HostSweep &, StripSweep<double> &);
template bool build_strip_sweeps<float>(pp_ctx *, const HostSweep &, const HostSweep &, StripSweep<float> &);

template <class T>
void launch_strip_sweeps(pp_ctx *ctx, const StripSweep<T> &L, const T *x, T *y) {
    launch_strip_side(ctx, L, L.lo, L.up, x, y);
    launch_strip_side(ctx, L, L.up, L.lo, (const T *)y, y);
}
template void launch_strip_sweeps<double>(pp_ctx *, const StripSweep<double> &, const double *, double *);
template void launch_strip_sweeps<float>(pp_ctx *, const StripSweep<float> &, const float *, float *);

}  // namespace pp
