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
#include <cmath>
#include <cstring>
#include <memory>
#include <queue>

#include "pp_internal.h"

namespace pp {

namespace {

constexpr int kAhead = kLaneAhead;  // steps whose data is in flight or in registers
constexpr int kLaneThreads = 256;
constexpr uint32_t kExtra = 1;      // LDS words past the chunk's rows: a zero

// Flags of a step, the same in all its lanes: the first, the last of its rows' steps.
enum : uint32_t { F_FIRST = 1, F_LAST = 2 };

// What a lane needs of one step: 16-byte pieces, piece k of the step's
// `active` lanes contiguous, so every load is one coalesced 16-byte load per lane.
//   values   S values of T
//   indices  S 16-bit LDS words of the dependencies, then the row's word, the
//            flags, the step's active lanes, the active lanes kAhead steps later
//   pivot    the row's diagonal and its reciprocal rounded to FP64
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
template <class T, int W, int G, int S, int MODE>
__device__ inline void run_step(const Step<T, S> &q, const Step<T, S> &next, Step<T, S> &past, const char *&p,
                                Carry<T, S> &c, uint32_t lane, uint32_t tail_lane) {
#pragma clang fp contract(off)
    T x[S];
#pragma unroll
    for (int j = 0; j < S; ++j) x[j] = *lds_word<T>(c.addr.dep[j]);
    LdsWord<T> *mine = lds_word<T>(c.addr.row);
    const T rhs = *mine;
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    load_step<T, S>(past, p, c.active, lane);
    const uint32_t flags = (uint32_t)__builtin_amdgcn_readfirstlane(q.ix(S / 2)) >> 16;
    const uint32_t active = (uint32_t)__builtin_amdgcn_readfirstlane(q.ix(S / 2 + 1));
    c.addr.set(next);
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
        if (tail_lane < (active & 0xffffu)) *mine = s;
        if constexpr (W > 1) __syncthreads();
    }
}

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
        for (uint32_t k = 0; k < lo; ++k) {
#pragma unroll
            for (int a = 0; a < kAhead; ++a)
                run_step<T, W, G, S, MLO>(q[a], q[(a + 1) % kAhead], q[(a + kAhead - 1) % kAhead], p, st, lane,
                                          tail_lane);
        }
        for (uint32_t k = 0; k < up; ++k) {
#pragma unroll
            for (int a = 0; a < kAhead; ++a)
                run_step<T, W, G, S, MUP>(q[a], q[(a + 1) % kAhead], q[(a + kAhead - 1) % kAhead], p, st, lane,
                                          tail_lane);
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
};

void append_steps(const HostSweep &s, const LanePlan &P, std::vector<StepRef> &out) {
    for (const auto &g : P.groups)
        for (uint32_t k = 0; k < g.steps; ++k) out.push_back({&s, g.first, g.count, k, g.steps, &P});
    while (out.size() % kAhead) out.push_back({nullptr, 0, 0, 0, 0, nullptr});
}

// One step at `out` (zeroed), `active` lanes; ahead: the lanes kAhead steps later.
template <class T, int S>
void write_step(const StepRef &r, uint32_t r0, uint32_t nr, int G, uint32_t active, uint32_t ahead,
                unsigned char *out) {
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
                ix[j] = (uint16_t)(has ? s.ci[a + j] - r0 : nr);  // word nr holds a zero
            }
            ix[S] = (uint16_t)i;
            flags = (r.part == 0 ? F_FIRST : 0u) | (r.part + 1 == r.parts ? F_LAST : 0u);
            if (s.mode != HostSweep::UNIT) d = (T)s.diag[r0 + i];
        }
        ix[S + 1] = (uint16_t)flags;
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
                write_step<T, S>(steps[c][k], r0, nr, G, active, lanes(steps[c], k + kAhead), p);
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

}  // namespace pp
