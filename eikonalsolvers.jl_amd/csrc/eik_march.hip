// eik_march.hip -- forward traveltime engine: ordered node marching (gfx950).
//
// The heap FMM's answer is the fixed point of the local replay (eik_stencil.h), whatever the order
// in which nodes are replayed; the order only decides how often a node is replayed.  Here a node is
// replayed when no node that its stencil reads is pending with a lower expected value, so nearly
// every node is replayed once, after the nodes it depends on (1.01-1.04 replays per node measured on
// 600x400 and 201x201x101 models, against 17 for relaxing whole tiles until they settle).
//
// State per instance (a source's grid or its refined box): the traveltimes, the pop keys of cascade
// nodes, and per node a pending value P (+inf: idle), the value the node is expected to get, a
// float.  The pending nodes are listed.  One round:
//   select:  a listed node runs if its P lies within the band above the instance's lowest P and no
//            node within two along an axis is pending with a lower P (lower index on ties); the
//            others stay listed.  Two nodes that run in the same round are therefore never in each
//            other's stencil;
//   replay:  each running node is replayed from its neighbours' state, which no other node of the
//            round changes, and written if it changed;
//   wake:    a changed node makes every neighbour pending whose replay the change can alter: those
//            whose pop key is not below the smaller of the node's old and new keys (a change whose
//            keys both exceed a node's key leaves its replay as it is), and of the nodes two away
//            only those whose in-between node pops no later than they do.
// The node with an instance's lowest P always runs, so a round always makes progress; when nothing
// is pending every node's replay equals its value, and there is nothing to verify at the end.  No read of
// a value or key races a write: what a node's replay reads no other node of the round changes.  Pending
// values do race (a wake may lower one while its holder reads it) and a round has room for so many nodes,
// so the order depends on the schedule, and the result where the replay has more than one fixed point:
// exact ties, FP32's near-ties, the roughest media.  A march can circulate where the order means
// little; it then stops at its limit (march_ctl).
//
// Layout.  Values, pending values and slowness lie in bricks of 64 nodes (4x4x4, or 8x8 in 2D), so
// that a node's stencil and the nodes around it on the front share cache lines whatever the front's
// direction; node indices below are positions in this layout.  k_march_finish writes the values to
// the x-fastest grids that the rest of the library reads.  Depth bytes and pop keys, which only
// cascade nodes have, are kept in the x-fastest pools throughout.
//
// Marked nodes.  A value with the sign bit set is an init node (depth byte kInitDepth, never
// changes) or a cascade node (depth byte 1..kMaxCascade, pop key in the K and S pools); all other
// nodes' key is their value.  A wave none of whose lanes sees a mark reads values only.  At the end
// the marks of cascade nodes come off, and init nodes' depth bytes go back to 0.
#include <array>

#include "eik_internal.h"

namespace eik {

constexpr unsigned kIdle = 0x7f800000u;  // P of a node that is not pending: +inf

// A list entry: node, and either kOnce, once the entry is known to be its node's only one, with the stencil
// position that held it up when last looked at (kNoHint: none), or in a device round its waker's tag.
constexpr unsigned kNodeBits = 27, kNodeMask = (1u << kNodeBits) - 1u;
constexpr unsigned kHintShift = kNodeBits, kNoHint = 15u, kOnce = 0x80000000u;
constexpr unsigned kNoEntry = 0xffffffffu;  // (no march has kNodeMask nodes)

// x[i] of a uniform x, i < 2^kNodeBits.  In 3D with a 32-bit offset: one address register per access
// rather than two, which the FP64 replay would otherwise spill (201x201x101 x 16: 63.6 -> 59.9 ms, along
// with the view kept out of memory in hint_index).  In 2D nothing spills and the plain form is 4 % faster.
template <int ND, typename T>
__device__ __forceinline__ T& at(T* x, unsigned i) {
    static_assert(sizeof(T) <= 8, "offsets of 2^27 nodes fit 32 bits");
    if constexpr (ND == 3) return *(T*)((char*)x + i * (unsigned)sizeof(T));
    return x[i];
}

// ------------------------------------------------------------------ one node's replay
// A grid with its pools, per instance (wave-uniform).
template <int ND, typename T>
struct GridView {
    static constexpr int E = fwd_tile_edge(ND);  // brick edge
    T* tt;           // bricked
    const T* slow;   // bricked
    T* kk;           // x-fastest
    T* ss;
    uint8_t* dd;
    int n[3];
    unsigned bs[3];  // nodes from a brick to the next along an axis
    double rbx, rby; // 1 / bricks along x, y
    unsigned bx, by;

    __device__ __forceinline__ void coords(unsigned l, int* g) const {
        // floor(b / n) = floor((b + 0.5) * (1 / n)) exactly for b < 2^31: (b + 0.5) / n lies at
        // least 0.5 / n from an integer, far more than the rounding of the product
        const unsigned b = l >> 6;
        const unsigned row = (unsigned)(((double)b + 0.5) * rbx);
        const unsigned cx = b - row * bx;
        if (ND == 2) {
            g[0] = (int)(cx * 8u + (l & 7u));
            g[1] = (int)(row * 8u + ((l >> 3) & 7u));
            g[2] = 0;
        } else {
            const unsigned pl = (unsigned)(((double)row + 0.5) * rby);
            const unsigned cy = row - pl * by;
            g[0] = (int)(cx * 4u + (l & 3u));
            g[1] = (int)(cy * 4u + ((l >> 2) & 3u));
            g[2] = (int)(pl * 4u + ((l >> 4) & 3u));
        }
    }
    // index change of d steps (d = 1, 2) up or down axis ax from coordinate c
    __device__ __forceinline__ unsigned step(int ax, int c, int d, bool down) const {
        const int r = c & (E - 1);
        const unsigned s = ax == 0 ? 1u : (ax == 1 ? (unsigned)E : (unsigned)(E * E));
        const unsigned in = (unsigned)d * s, out = bs[ax] - (unsigned)(E - d) * s;
        const unsigned u = down ? (r >= d ? in : out) : (r + d < E ? in : out);
        return down ? 0u - u : u;
    }
    __device__ __forceinline__ int64_t linear(const int* g) const {
        return g[0] + (int64_t)n[0] * (g[1] + (ND == 3 ? (int64_t)n[1] * g[2] : 0));
    }
    __device__ __forceinline__ unsigned index(const int* g) const {
        const unsigned s = E == 8 ? 3u : 2u, m = E - 1;
        const unsigned b = ((unsigned)g[0] >> s) + bx * (((unsigned)g[1] >> s) + (ND == 3 ? by * ((unsigned)g[2] >> s) : 0u));
        const unsigned o = ((unsigned)g[0] & m) | ((unsigned)g[1] & m) << s | (ND == 3 ? ((unsigned)g[2] & m) << (2 * s) : 0u);
        return b * 64u + o;
    }
};

// the march's own pools (bricked; an instance's part starts at 64 * tile_base)
template <typename T>
struct MarchPools {
    T* tt;
    const T* slow;    // per model: InstDev::ms_off
    unsigned* p[3];   // pending values
    unsigned* own;    // list position of a node's newest entry (a workgroup per instance)
    unsigned* less;   // a listed node's pending value lowered by a later wake (device rounds)
    unsigned* lists;  // two lists per instance (list_start)
};

constexpr unsigned long long kOverflow = 2ull;  // counters[3]: a list was too short (1: not converged)
template <typename T>
__device__ __forceinline__ unsigned* inst_lists(const MarchPools<T>& M, const InstDev& I, int in, int blocks) {
    return M.lists + list_start(I.tile_base, in, blocks);
}

template <int ND, typename T>
__device__ __forceinline__ GridView<ND, T> grid_view(const InstDev& I, const TTPools& P, const MarchPools<T>& M) {
    GridView<ND, T> G;
    G.tt = M.tt + I.tile_base * 64;
    G.slow = M.slow + I.ms_off;
    G.kk = (T*)P.k + I.tt_off;
    G.ss = (T*)P.s + I.tt_off;
    G.dd = P.d + I.tt_off;
    G.n[0] = I.n[0];
    G.n[1] = I.n[1];
    G.n[2] = ND == 3 ? I.n[2] : 1;
    G.bx = (unsigned)I.t[0];
    G.by = (unsigned)I.t[1];
    G.bs[0] = 64u;
    G.bs[1] = 64u * G.bx;
    G.bs[2] = 64u * G.bx * G.by;
    G.rbx = I.rbx;
    G.rby = I.rby;
    return G;
}

// smallest key that a change with (smaller) key c can reach: c itself; in FP32, where keys within
// the tie margin pop as one batch, a node may hold a key up to the margin below its trigger's
__device__ __forceinline__ double reach_key(double c) { return c; }
__device__ __forceinline__ float reach_key(float c) { return c < EIK_INFF ? c - 2.f * kTieUlps * 1.1920929e-7f * fabsf(c) : c; }

// A change smaller than `settle` relative (value and key) wakes nothing; see march_run_t.
template <typename T>
__device__ __forceinline__ bool quiet_change(T v0, T k0, T v1, T k1, T settle) {
    if (!(settle > T(0)) || !(v0 < tinf<T>())) return false;
    return fabs(v1 - v0) <= settle * v0 && fabs(k1 - k0) <= settle * fabs(k0);
}

// The pending value of a woken node, as bits: never 0 (may_run steps it down by one), and never an
// idle node's, whatever the expected value (times beyond the float range: its largest number).
__device__ __forceinline__ unsigned pend_bits(float p) { return min(max(__float_as_uint(p), 1u), kIdle - 1u); }

// The same in a device round, with the stencil position k of the woken node as seen from the node that wakes
// it in the low bits (20 bits of mantissa are left for the order).  No two nodes of a round wake a node with
// the same k, so the minimum that the node ends up with names one of them.  Among equal values the later
// position goes first: the other way round 3D spheres need up to 18 % more rounds (50x90x90 x 5: 352 -> 416,
// 5.6 -> 6.4 ms).
constexpr unsigned kTagMask = 15u;
__device__ __forceinline__ unsigned wake_tag(int k) { return 14u - (unsigned)k; }
__device__ __forceinline__ unsigned pend_tagged(float p, int k) { return (pend_bits(p) & ~kTagMask) | wake_tag(k); }

// Replays node l (on: this lane has one) and writes it if it changed; returns whether it did.
// p: the round's pending values (only read here).  wake(k, w, q, idle, pq, p): if w, neighbour q (the
// k-th of 4 * ND, idle or pending with pq) becomes pending with value p; k = 0 .. 2 * ND - 1 are the adjacent nodes.
// Nodes two away are rarely woken (only by a change of a node that they were replayed with): unless
// some lane wakes one, wake is not called for them and *two stays false.  Every lane of the wave
// calls it.
template <int ND, typename T, bool SPH, bool MIX, bool NEAR, class Wake>
__device__ __forceinline__ bool relax_node(const InstDev& I, const GridView<ND, T>& G, const Metric<Arith<T, MIX>>& mcart,
                                           const unsigned* p, unsigned l, bool on, T settle, bool* two, Wake wake) {
    using A = Arith<T, MIX>;
    int g[3];
    G.coords(l, g);
    // all values of the stencil in one round trip; positions outside it fall back to the node itself
    T r1[2 * ND], r2[2 * ND];
    unsigned q1[2 * ND], q2[2 * ND], p1[2 * ND], ok1 = 0u, ok2 = 0u;
#pragma unroll
    for (int k = 0; k < 2 * ND; k++) {
        const int ax = k >> 1, sh = (k & 1) ? -1 : 1;
        const int c = g[ax] + sh;
        const bool in1 = c >= 0 && c < G.n[ax];
        // the adjacent node off every boundary plane: its far neighbour may be used
        bool in2 = c >= 1 && c <= G.n[ax] - 2;
#pragma unroll
        for (int d = 0; d < ND; d++)
            if (d != ax) in2 = in2 && g[d] >= 1 && g[d] <= G.n[d] - 2;
        ok1 |= (unsigned)in1 << k;
        ok2 |= (unsigned)in2 << k;
        q1[k] = in1 ? l + G.step(ax, g[ax], 1, k & 1) : l;
        q2[k] = in2 ? l + G.step(ax, g[ax], 2, k & 1) : l;
        r1[k] = at<ND>(G.tt, q1[k]);
        r2[k] = at<ND>(G.tt, q2[k]);
        p1[k] = at<ND>(p, q1[k]);
    }
    const T raw = at<ND>(G.tt, l);
    const T sl = at<ND>(G.slow, l);
    bool marked = signbit(raw);
    unsigned idle1 = 0u;  // adjacent nodes that are not pending
#pragma unroll
    for (int k = 0; k < 2 * ND; k++) {
        idle1 |= (unsigned)(p1[k] == kIdle) << k;
        if (!((ok1 >> k) & 1u)) r1[k] = tinf<T>();
        if (!((ok2 >> k) & 1u)) r2[k] = tinf<T>();
        marked = marked || signbit(r1[k]) || signbit(r2[k]);
    }
    Metric<A> mt;
    if constexpr (SPH) {
        node_spacing<A>(I, g, mt.dh);
        metric_coefs(mt, ND);
    } else {
        mt = mcart;
    }
    // What the wakes need of the loads is formed here: a use of a loaded value behind the stores below
    // would wait for those too (memory operations are counted in order).
    float step[ND];
#pragma unroll
    for (int ax = 0; ax < ND; ax++) {
        step[ax] = (float)mt.dh[ax] * (float)sl;
        asm volatile("" : "+v"(step[ax]));
    }
    asm volatile("" : "+v"(idle1));
    int code[3];
    Key<T> nk;
    T nv;
    const T v0 = fabs(raw);
    Key<T> k0{v0, -tinf<T>(), 0};
    unsigned f1 = 0u, f2 = 0u, m1 = 0u, m2 = 0u;  // init nodes; marked nodes
    T v1[2 * ND], v2[2 * ND];
    bool near64 = false;  // mixed precision near the source: the FP64 stencil
    if constexpr (MIX && NEAR) near64 = in_fp64_region(I, g);
    const bool fast = __ballot(on && (marked || near64)) == 0ull;
    const int64_t lin = G.linear(g);
    if (fast) {
        auto nokeys = [](int, bool) { return Key<T>{T(0), T(0), 0}; };  // never called: no cascade key
#pragma unroll
        for (int k = 0; k < 2 * ND; k++) {
            v1[k] = r1[k];
            v2[k] = r2[k];
        }
        nv = replay<ND, T, MIX>(v1, v2, nokeys, 0u, 0u, 0u, 0u, 0u, ok1, ok2, (A)sl, mt, code, &nk);
    } else {
        unsigned d1 = 0u, d2 = 0u, dcap = 0u;
        const int64_t ls[3] = {1, G.n[0], (int64_t)G.n[0] * G.n[1]};
#pragma unroll
        for (int k = 0; k < 2 * ND; k++) {
            const int ax = k >> 1, sh = (k & 1) ? -1 : 1;
            v1[k] = fabs(r1[k]);
            v2[k] = fabs(r2[k]);
            const bool s1 = signbit(r1[k]), s2 = signbit(r2[k]);
            const int e1 = s1 ? (int)G.dd[lin + sh * ls[ax]] : 0;
            const int e2 = s2 ? (int)G.dd[lin + 2 * sh * ls[ax]] : 0;
            m1 |= (unsigned)s1 << k;
            m2 |= (unsigned)s2 << k;
            f1 |= (unsigned)(e1 == kInitDepth) << k;
            f2 |= (unsigned)(e2 == kInitDepth) << k;
            d1 |= (unsigned)(s1 && e1 != kInitDepth) << k;
            d2 |= (unsigned)(s2 && e2 != kInitDepth) << k;
            dcap |= (unsigned)(s1 && e1 != kInitDepth && e1 >= kMaxCascade) << k;
        }
        if (signbit(raw)) {  // a listed node is never an init node
            k0.K = G.kk[lin];
            k0.S = G.ss[lin];
            k0.D = (int)G.dd[lin];
        }
        // pop key of slot k's neighbour, from memory (only the cascade path asks)
        auto keys = [&](int k, bool two) {
            const int64_t q = lin + ((k & 1) ? -1 : 1) * (two ? 2 : 1) * ls[k >> 1];
            if (((two ? d2 : d1) >> k) & 1u) return Key<T>{G.kk[q], G.ss[q], (int)G.dd[q]};
            return Key<T>{two ? v2[k] : v1[k], -tinf<T>(), 0};
        };
        nv = tinf<T>();
        if constexpr (MIX && NEAR) {
            if (near64) {
                Metric<double> m64;
                node_spacing<double>(I, g, m64.dh);
                metric_coefs(m64, ND);
                nv = replay<ND, T, false>(v1, v2, keys, d1, d2, dcap, f1, f2, ok1, ok2, (double)sl, m64, code, &nk);
            }
        }
        if (!near64) nv = replay<ND, T, MIX>(v1, v2, keys, d1, d2, dcap, f1, f2, ok1, ok2, (A)sl, mt, code, &nk);
    }
    const bool vchg = nv == nv && nv != v0 && !(nv >= tinf<T>() && v0 >= tinf<T>());
    const bool kchg = nv < tinf<T>() && !keq(nk, k0);
    const bool chg = on && (vchg || kchg);
    if (chg) {
        at<ND>(G.tt, l) = nk.D ? -nv : nv;
        if (nk.D != k0.D) G.dd[lin] = (uint8_t)nk.D;
        if (nk.D) {
            G.kk[lin] = nk.K;
            G.ss[lin] = nk.S;
        }
    }
    const bool loud = chg && !quiet_change<T>(v0, k0.K, nv, nk.K, settle);
    // the smaller of the old and new keys (an unreached node's key is +inf)
    const T ck = k0.K < nk.K ? k0.K : nk.K;
    const T c = reach_key(ck);
    const float cf = (float)ck;
    // adjacent nodes whose key the change reaches; of the nodes two away, which use this one only
    // through the node between, those whose key it reaches and whose node between pops no later (an
    // unreached one is pending already: the node between was reached)
    unsigned w1 = 0u, w2 = 0u;
#pragma unroll
    for (int k = 0; k < 2 * ND; k++) {
        const bool r = (v2[k] < tinf<T>()) & (v1[k] < tinf<T>());
        const bool far = (v2[k] >= c) & (reach_key(v1[k]) <= v2[k]);
        w1 |= (unsigned)(v1[k] >= c) << k;
        w2 |= (unsigned)(r & far) << k;
    }
    if (!fast) {  // a marked node's key is not its value: woken whatever it is, unless an init node
#pragma unroll
        for (int k = 0; k < 2 * ND; k++) {
            const bool r = (v2[k] < tinf<T>()) & (v1[k] < tinf<T>());
            const bool k1m = (m1 >> k) & 1u, k2m = (m2 >> k) & 1u;
            w1 |= (unsigned)k1m << k;
            w2 |= (unsigned)(r & (k2m | ((v2[k] >= c) & k1m))) << k;
        }
        w1 &= ~f1;
        w2 &= ~f2;
    }
    w1 = loud ? w1 & ok1 : 0u;
    w2 = loud ? w2 & ok2 : 0u;
#pragma unroll
    for (int k = 0; k < 2 * ND; k++)
        wake(k, (w1 >> k) & 1u, q1[k], (idle1 >> k) & 1u, p1[k], fmaxf(cf, fminf((float)v1[k], cf + step[k >> 1])));
    *two = __ballot(w2 != 0u) != 0ull;
    if (*two) {
        unsigned p2[2 * ND];
#pragma unroll
        for (int k = 0; k < 2 * ND; k++) p2[k] = at<ND>(p, ((w2 >> k) & 1u) ? q2[k] : l);
#pragma unroll
        for (int k = 0; k < 2 * ND; k++) wake(2 * ND + k, (w2 >> k) & 1u, q2[k], p2[k] == kIdle, p2[k], fmaxf(cf, (float)v2[k]));
    }
    return chg;
}

// The stencil position k (0 .. 4 * ND - 1) of a node: axis k >> 2, down if k & 1, two steps if k & 2.
// True if no node at one holds up node l, pending with value own; *hold: the position of the pending
// node that holds it up longest (the largest lower value), kNoHint if none.  One round trip.
template <int ND, typename T>
__device__ __forceinline__ bool may_run(const GridView<ND, T>& G, const unsigned* p, unsigned l, unsigned own, unsigned* hold) {
    int g[3];
    G.coords(l, g);
    unsigned v[4 * ND];
#pragma unroll
    for (int k = 0; k < 4 * ND; k++) {
        const int ax = k >> 2, d = (k & 2) ? 2 : 1;
        const bool in = (k & 1) ? g[ax] >= d : g[ax] + d < G.n[ax];
        v[k] = at<ND>(p, in ? l + G.step(ax, g[ax], d, k & 1) : l);
        // outside the grid nothing holds it up; a node further down also wins a tie
        v[k] = in ? v[k] - (unsigned)(k & 1) : kIdle;
    }
    unsigned best = 0u, at = kNoHint;
#pragma unroll
    for (int k = 0; k < 4 * ND; k++)
        if (v[k] < own && v[k] >= best) {
            best = v[k];
            at = (unsigned)k;
        }
    *hold = at;
    return at == kNoHint;
}

// Whether the node at stencil position k of l is still pending with a lower value than `own`.
template <int ND, typename T>
__device__ __forceinline__ unsigned hint_index(const GridView<ND, T>& G, unsigned l, unsigned k) {
    // positions inside the grid only (a hint names a pending node)
    const int ax = (int)(k >> 2), d = (k & 2u) ? 2 : 1;
    constexpr unsigned S = GridView<ND, T>::E == 8 ? 3u : 2u;
    const int c = (int)((l >> (S * (unsigned)ax)) & (unsigned)(GridView<ND, T>::E - 1));
    const unsigned s = 1u << (S * (unsigned)ax);
    // (not a choice between the three: the compiler would put the view in memory and choose an address)
    const unsigned b = (G.bs[0] & (0u - (ax == 0))) | (G.bs[1] & (0u - (ax == 1))) | (G.bs[2] & (0u - (ax == 2)));
    const unsigned in = (unsigned)d * s, out = b - (unsigned)(GridView<ND, T>::E - d) * s;
    if (k & 1u) return l - (c >= d ? in : out);
    return l + (c + d < GridView<ND, T>::E ? in : out);
}

// Position of this lane among the lanes of mask m.
__device__ __forceinline__ unsigned lane_rank(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}

// A workgroup barrier for LDS alone: waits for this wave's LDS accesses, not for its memory accesses.
// For phases that exchange nothing through memory.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Listing.  Several nodes of a round may wake the same idle node, and each lists it; the next selection drops
// all entries but one, without waiting for an atomic's return value.  In a workgroup each writes its list
// position into the node's `own` word, and the entry that the word names stands.  In a device round, whose
// blocks run on several XCDs, that would be a race on memory (after plain stores from two XCDs in one launch
// each went on reading its own in the next: both entries stood, and one was left listed for good when the
// node had run), so the entry carries its waker's tag, and the one stands whose tag the node's pending value
// carries (pend_tagged).

// The neighbours of the init nodes (values in the x-fastest pool) are pending with their smallest init
// neighbour's value: add(q, p, k) for each of them, k its position from that neighbour, by the threads of one block.  The init nodes'
// values go to the bricked pool first.
template <int ND, typename T, class Add>
__device__ __forceinline__ void seed_march(const InstDev& I, const GridView<ND, T>& G, const T* tt_lin, const SrcPt* seeds, int ns,
                                           Add add) {
    auto coords = [&](int64_t l, int* g) {
        g[0] = (int)(l % G.n[0]);
        g[1] = (int)((l / G.n[0]) % G.n[1]);
        g[2] = ND == 3 ? (int)(l / ((int64_t)G.n[0] * G.n[1])) : 0;
    };
    for (int i = threadIdx.x; i < ns; i += blockDim.x) {
        int g[3];
        coords(seeds[i].node, g);
        G.tt[G.index(g)] = tt_lin[seeds[i].node];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < ns * 2 * ND; i += blockDim.x) {
        const int64_t l = seeds[i / (2 * ND)].node;
        const int k = i % (2 * ND), ax = k >> 1, sh = (k & 1) ? -1 : 1;
        int g[3];
        coords(l, g);
        g[0] += ax == 0 ? sh : 0;
        g[1] += ax == 1 ? sh : 0;
        g[2] += ax == 2 ? sh : 0;
        if (g[0] < 0 || g[0] >= G.n[0] || g[1] < 0 || g[1] >= G.n[1] || g[2] < 0 || g[2] >= G.n[2]) continue;
        const unsigned q = G.index(g);
        if (!signbit(G.tt[q])) add(q, (float)fabs(tt_lin[l]), k);
    }
}

// ------------------------------------------------------------------ one workgroup per instance
// The whole march of an instance in one workgroup: the rounds are separated by workgroup barriers,
// so they cost no launches and need nothing of the rest of the device.
constexpr int kGroupList = 6144;  // pending nodes listed in LDS (of each of two lists); the rest in memory
constexpr int kGroupRun = 2048;   // nodes run per round (a further one waits for the next round)

template <int ND, typename T, bool SPH, bool MIX, bool NEAR, int BT>
__global__ void __launch_bounds__(BT) k_march_group(const InstDev* __restrict__ inst, TTPools pools, MarchPools<T> M,
                                                    const SrcPt* __restrict__ seeds, int cap, const int* __restrict__ nseed,
                                                    T settle, MarchCtl ctl, unsigned long long* __restrict__ counters) {
    using A = Arith<T, MIX>;
    __shared__ unsigned s_list[2][kGroupList];
    __shared__ unsigned s_run[kGroupRun];
    __shared__ unsigned s_cnt[3], s_min[3], s_nrun[2];
    const InstDev& I = inst[blockIdx.x];
    const GridView<ND, T> G = grid_view<ND, T>(I, pools, M);
    const unsigned nodes = 64u * (unsigned)(I.t[0] * I.t[1] * I.t[2]);
    const unsigned lcap = min(list_cap(nodes), ctl.list_limit);
    unsigned* const sp = inst_lists(M, I, blockIdx.x, 0);  // list k's entries beyond kGroupList: sp + k * lcap
    unsigned* const pend = M.p[0] + I.tile_base * 64;
    unsigned* const own = M.own + I.tile_base * 64;
    const int tid = threadIdx.x, lane = tid & 63;
    const float band = (float)I.mband;
    Metric<A> mcart;
#pragma unroll
    for (int ax = 0; ax < 3; ax++) mcart.dh[ax] = (A)I.h[0];
    metric_coefs(mcart, ND);
    auto put = [&](int k, unsigned at, unsigned e) {
        if (at < (unsigned)kGroupList) s_list[k][at] = e;
        else if (at - kGroupList < lcap) sp[(size_t)k * lcap + (at - kGroupList)] = e;
    };
    auto get = [&](int k, unsigned at) { return at < (unsigned)kGroupList ? s_list[k][at] : sp[(size_t)k * lcap + (at - kGroupList)]; };
    auto lower = [&](unsigned q, unsigned p) {
        (void)__hip_atomic_fetch_min(&at<ND>(pend, q), p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    if (tid < 3) {
        s_cnt[tid] = 0u;
        s_min[tid] = kIdle;
    }
    if (tid < 2) s_nrun[tid] = 0u;
    __syncthreads();
    seed_march<ND, T>(I, G, (const T*)pools.tt + I.tt_off, seeds + (int64_t)blockIdx.x * cap, nseed[blockIdx.x], [&](unsigned q, float pf, int) {
        const unsigned at = atomicAdd(&s_cnt[0], 1u), p = pend_bits(pf);
        lower(q, p);
        atomicMin(&s_min[0], p);
        own[q] = at;
        put(0, at, q);
    });
    __syncthreads();
    unsigned long long tot_upd = 0ull, tot_chg = 0ull;
    unsigned round = 0;
    int cur = 0, slot = 0;
    for (;; round++) {
        const unsigned cnt = s_cnt[slot];
        if (cnt == 0u || cnt > lcap || round >= ctl.max_rounds) break;
        const int nslot = slot == 2 ? 0 : slot + 1, rslot = nslot == 2 ? 0 : nslot + 1;
        const int par = (int)(round & 1u);
        const unsigned lim = __float_as_uint(__uint_as_float(s_min[slot]) + band);
        if (tid == 0) {  // last used two rounds ago
            s_cnt[rslot] = 0u;
            s_min[rslot] = kIdle;
        }
        // select
        unsigned lowest = kIdle;
        for (unsigned b = 0; b < cnt; b += BT) {
            const unsigned i = b + tid;
            bool have = i < cnt, run = false;
            unsigned l = 0u;
            unsigned p = kIdle, hold;
            if (have) {
                const unsigned e = get(cur, i);
                l = e & kNodeMask;
                const unsigned ow = at<ND>(own, l);
                p = at<ND>(pend, l);
                run = may_run<ND, T>(G, pend, l, p, &hold) && p <= lim;
                have = (e & kOnce) || ow == i;
                run = run && have;
            }
            const unsigned long long mr = __ballot(run);
            if (mr) {
                unsigned at = 0u;
                if (lane == 0) at = atomicAdd(&s_nrun[par], (unsigned)__popcll(mr));
                at = (unsigned)__builtin_amdgcn_readfirstlane((int)at) + lane_rank(mr);
                run = run && at < (unsigned)kGroupRun;
                if (run) s_run[at] = l;
            }
            const bool keep = have && !run;
            const unsigned long long mk = __ballot(keep);
            if (mk) {
                unsigned to = 0u;
                if (lane == 0) to = atomicAdd(&s_cnt[nslot], (unsigned)__popcll(mk));
                to = (unsigned)__builtin_amdgcn_readfirstlane((int)to) + lane_rank(mk);
                if (keep) {
                    put(cur ^ 1, to, l | kOnce);
                    lowest = min(lowest, p);
                }
            }
        }
        lds_barrier();  // the selection writes LDS (and list entries that the next round reads)
        // replay and wake
        const unsigned nrun = min(s_nrun[par], (unsigned)kGroupRun);
        if (tid == 0) s_nrun[par ^ 1] = 0u;
        for (unsigned b = (unsigned)(tid & ~63); b < nrun; b += BT) {
            const unsigned j = b + lane;
            const bool on = j < nrun;
            const unsigned l = s_run[on ? j : b];
            unsigned who[4 * ND] = {}, fresh = 0u;
            bool two;
            const bool chg = relax_node<ND, T, SPH, MIX, NEAR>(
                I, G, mcart, pend, l, on, settle, &two, [&](int k, bool w, unsigned q, bool idle, unsigned, float p) {
                    who[k] = q;
                    if (w) {
                        const unsigned pu = pend_bits(p);
                        lowest = min(lowest, pu);
                        lower(q, pu);
                    }
                    fresh |= (unsigned)(w & idle) << k;
                });
            if (on) at<ND>(pend, l) = kIdle;  // (no node of the round wakes it)
            unsigned total = 0u;
#pragma unroll
            for (int k = 0; k < 4 * ND; k++)
                if (k < 2 * ND || two) total += (unsigned)__popcll(__ballot((fresh >> k) & 1u));
            if (total) {
                unsigned base = 0u;
                if (lane == 0) base = atomicAdd(&s_cnt[nslot], total);
                base = (unsigned)__builtin_amdgcn_readfirstlane((int)base);
#pragma unroll
                for (int k = 0; k < 4 * ND; k++) {
                    if (k < 2 * ND || two) {
                        const unsigned long long m = __ballot((fresh >> k) & 1u);
                        const unsigned to = base + lane_rank(m);
                        if ((fresh >> k) & 1u) {
                            put(cur ^ 1, to, who[k]);
                            at<ND>(own, who[k]) = to;
                        }
                        base += (unsigned)__popcll(m);
                    }
                }
            }
            tot_upd += on;
            tot_chg += chg;
        }
        lowest = wave_min_u32(lowest);
        if (lane == 0 && lowest != kIdle) atomicMin(&s_min[nslot], lowest);
        __syncthreads();
        cur ^= 1;
        slot = nslot;
    }
    // statistics: one atomic per counter and wave
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        tot_upd += __shfl_xor(tot_upd, o);
        tot_chg += __shfl_xor(tot_chg, o);
    }
    if (lane == 0) {
        atomicAdd(&counters[0], tot_upd);
        atomicAdd(&counters[1], tot_chg);
    }
    if (tid == 0) {
        atomicMax(&counters[2], (unsigned long long)round);
        if (s_cnt[slot]) atomicOr(&counters[3], s_cnt[slot] > lcap ? kOverflow : 1ull);
    }
}

// ------------------------------------------------------------------ the whole device per round
// One launch per round over all instances: every block takes an equal, contiguous part of an
// instance's list, selects, and replays what it selected.  A launch orders its reads before the next
// launch's, so within one launch the round's pending values (buffer round % 3) and its list are only
// read; the next round's go to buffer (round + 1) % 3 and the other list:
//   a node that stays listed takes its value along, or a lower one that wakes have left in `less`
//   (its holder reads it while they lower it, and sees it in this round or the next);
//   a node that runs becomes idle in the next buffer and in the third (which nobody reads or writes
//   in this round), and in the present one a round later, when that is the third: by the block that
//   ran it, from the list `ran` it keeps;
//   an idle node that is woken gets its value in the next buffer, by an atomic minimum over the
//   nodes that wake it: it is idle in all three buffers.
// Atomics between the XCDs are slow (about 1e10 a second over the device, and loads issued after
// them wait for them), so there is one per newly listed node and wake, none per listed node.
// A block writes the next round's entries to its own segment of the list and their number and lowest
// value to its own words, so that nothing is reserved by an atomic whose return a wave would wait
// for (several microseconds); the next round's blocks share the segments out by a scan over their
// lengths.  blockIdx.x is the instance: consecutive blocks go to consecutive XCDs, so an instance's
// blocks share an XCD's L2 when there are a multiple of eight instances.
struct MarchSlots {
    unsigned* cnt;   // 2 x ninst x kMaxBlocks, by round parity: entries in each block's segment
    unsigned* low;   // the same: lowest pending value among them
    unsigned* ran;   // per block: count, then up to kRoundRun nodes
    unsigned* stat;  // per block: nodes replayed and changed
    unsigned limit;  // entries of a segment at most (MarchCtl::list_limit)
};
constexpr int kRoundThreads = 256;
constexpr int kRoundPer = 4;                                 // entries per thread and pass
constexpr int kRoundPass = kRoundThreads * kRoundPer;        // entries a block looks at together
constexpr int kRoundFresh = 3072;                            // newly listed nodes a pass collects in LDS

template <int ND, typename T>
__global__ void __launch_bounds__(256) k_march_seed(const InstDev* __restrict__ inst, int ninst, TTPools pools, MarchPools<T> M,
                                                    const SrcPt* __restrict__ seeds, int cap, const int* __restrict__ nseed,
                                                    MarchSlots S, int blocks, unsigned long long* __restrict__ counters) {
    __shared__ unsigned s_n, s_low;
    const int in = blockIdx.x;
    const InstDev& I = inst[in];
    const GridView<ND, T> G = grid_view<ND, T>(I, pools, M);
    const unsigned scap = min(seg_cap(64u * (unsigned)(I.t[0] * I.t[1] * I.t[2]), blocks), S.limit);
    unsigned* const list = inst_lists(M, I, in, blocks);
    unsigned* const pend = M.p[0] + I.tile_base * 64;
    if (threadIdx.x == 0) {
        s_n = 0u;
        s_low = kIdle;
    }
    for (int b = threadIdx.x; b < blocks; b += 256) {
        S.ran[(size_t)(in * blocks + b) * (kRoundRun + 1)] = 0u;
        S.stat[2 * (in * blocks + b)] = S.stat[2 * (in * blocks + b) + 1] = 0u;
    }
    __syncthreads();
    seed_march<ND, T>(I, G, (const T*)pools.tt + I.tt_off, seeds + (int64_t)in * cap, nseed[in], [&](unsigned q, float pf, int k) {
        const unsigned at = atomicAdd(&s_n, 1u), p = pend_tagged(pf, k);
        atomicMin(&pend[q], p);
        atomicMin(&s_low, p);
        if (at < scap) list[at] = q | wake_tag(k) << kHintShift;
    });
    __syncthreads();
    if (threadIdx.x == 0 && s_n > scap) atomicOr(&counters[3], kOverflow);
    if (threadIdx.x < kMaxBlocks) {  // all in the first block's segment
        S.cnt[in * kMaxBlocks + threadIdx.x] = threadIdx.x == 0 ? min(s_n, scap) : 0u;
        S.low[in * kMaxBlocks + threadIdx.x] = threadIdx.x == 0 ? s_low : kIdle;
    }
}

// inclusive sum over the lanes up to this one
__device__ __forceinline__ unsigned wave_scan(unsigned v) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned u = __shfl_up(v, o);
        v += lane >= o ? u : 0u;
    }
    return v;
}

template <int ND, typename T, bool SPH, bool MIX, bool NEAR>
__global__ void __launch_bounds__(kRoundThreads, 2)
    k_march_round(const InstDev* __restrict__ inst, int ninst, TTPools pools, MarchPools<T> M, MarchSlots S, int slot, int par,
                  T settle, unsigned long long* __restrict__ counters) {
    using A = Arith<T, MIX>;
    __shared__ unsigned s_run[kRoundRun], s_keep[kRoundPass], s_fresh[kRoundFresh], s_end[kRoundThreads / 64][kMaxBlocks];
    __shared__ unsigned s_nrun, s_nkeep, s_nfresh, s_low[kRoundThreads / 64], s_chg[kRoundThreads / 64];
    const int in = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nslot = slot == 2 ? 0 : slot + 1, rslot = nslot == 2 ? 0 : nslot + 1;
    const unsigned nblk = gridDim.y, blk = blockIdx.y;
    // the segments' lengths and lowest values, one per lane (every wave for itself)
    const size_t words = ((size_t)par * ninst + in) * kMaxBlocks, nwords = ((size_t)(par ^ 1) * ninst + in) * kMaxBlocks;
    const unsigned c0 = S.cnt[words + lane], low0 = S.low[words + lane];
    unsigned* const ran = S.ran + (size_t)(in * nblk + blk) * (kRoundRun + 1);
    const unsigned nran = ran[0];
    const InstDev& I = inst[in];
    const GridView<ND, T> G = grid_view<ND, T>(I, pools, M);
    const unsigned nodes = 64u * (unsigned)(I.t[0] * I.t[1] * I.t[2]);
    const unsigned* const p = M.p[slot] + I.tile_base * 64;
    unsigned* const pn = M.p[nslot] + I.tile_base * 64;
    unsigned* const pr = M.p[rslot] + I.tile_base * 64;
    unsigned* const less = M.less + I.tile_base * 64;
    const unsigned scap = min(seg_cap(nodes, nblk), S.limit), half = scap * nblk;  // a list: nblk segments
    const unsigned* const from = inst_lists(M, I, in, (int)nblk) + (par ? half : 0u);
    unsigned* const to = inst_lists(M, I, in, (int)nblk) + (par ? 0u : half) + (size_t)blk * scap;
    const unsigned end = wave_scan(c0), cnt = (unsigned)__builtin_amdgcn_readlane((int)end, 63);
    s_end[wave][lane] = end;
    // this block's part of the list, a multiple of a wave's entries
    const unsigned part = ((cnt + nblk - 1) / nblk + 63u) & ~63u;
    const unsigned lo = min(cnt, blk * part), hi = min(cnt, lo + part);
    // the nodes this block ran in the last round become idle in the buffer of that round
    const auto clear_ran = [&] {
        for (unsigned i = tid; i < nran; i += kRoundThreads) at<ND>(pr, ran[1 + i]) = kIdle;
    };
    if (lo >= hi) {
        clear_ran();
        if (tid == 0) {
            S.cnt[nwords + blk] = 0u;
            S.low[nwords + blk] = kIdle;
        }
        if (blk == 0 && lane >= (int)nblk && wave == 0) {  // words without a block
            S.cnt[nwords + lane] = 0u;
            S.low[nwords + lane] = kIdle;
        }
        if (nran) {
            __syncthreads();  // every thread has read the count
            if (tid == 0) ran[0] = 0u;
        }
        return;
    }
    const unsigned lim = __float_as_uint(__uint_as_float(wave_min_u32(low0)) + (float)I.mband);
    Metric<A> mcart;
#pragma unroll
    for (int ax = 0; ax < 3; ax++) mcart.dh[ax] = (A)I.h[0];
    metric_coefs(mcart, ND);
    if (tid == 0) s_nrun = 0u;
    // looking first only at the node that held an entry up before saves most reads, but costs a round
    // trip: not worth it for a wave or so
    const bool hints = part > kRoundThreads;
    unsigned lowest = kIdle, nchg = 0u, done = 0u, out = 0u;
    for (unsigned base = lo; base < hi; base += kRoundPass) {
        if (base != lo) lds_barrier();  // the pass before has read its counts
        if (tid == 0) {
            s_nkeep = 0u;
            s_nfresh = 0u;
        }
        lds_barrier();  // also: every thread has read the run list of the last round
        unsigned e[kRoundPer], pv[kRoundPer], pb[kRoundPer];
#pragma unroll
        for (int u = 0; u < kRoundPer; u++) {
            // entry i lies in the segment whose end is the first beyond i
            const unsigned i0 = base + u * kRoundThreads + (unsigned)(tid & ~63), i = i0 + lane;
            unsigned s = (unsigned)__popcll(__ballot(end <= i0));
            if (i < hi)
                while (s_end[wave][s] <= i) s++;
            e[u] = i < hi ? from[s * scap + (i - (s ? s_end[wave][s - 1] : 0u))] : kNoEntry;
        }
        if (base == lo) clear_ran();
        // own value, that of the node that held it up before, and a lowered one, in one round trip
        unsigned ls[kRoundPer];
#pragma unroll
        for (int u = 0; u < kRoundPer; u++) {
            const bool have = e[u] != kNoEntry;
            const unsigned l = have ? e[u] & kNodeMask : 0u, h = (e[u] & kOnce) ? (e[u] >> kHintShift) & 15u : kNoHint;
            pv[u] = at<ND>(p, l);
            pb[u] = at<ND>(p, hints && have && h != kNoHint ? hint_index<ND, T>(G, l, h) : l);
            ls[u] = at<ND>(less, l);
        }
        // the other stencil positions of the entries that are not held up still, in another
        unsigned hold[kRoundPer];
        bool run[kRoundPer];
#pragma unroll
        for (int u = 0; u < kRoundPer; u++) {
            const unsigned t = (e[u] >> kHintShift) & 15u, h = (e[u] & kOnce) ? t : kNoHint;
            if (e[u] != kNoEntry && !(e[u] & kOnce) && t != (pv[u] & kTagMask)) e[u] = kNoEntry;
            // still held up: lower, or as low and further down
            const bool held = hints && h != kNoHint && (pb[u] < pv[u] || ((h & 1u) && pb[u] == pv[u]));
            run[u] = e[u] != kNoEntry && pv[u] <= lim && !held;
            hold[u] = h;
        }
#pragma unroll
        for (int u = 0; u < kRoundPer; u++)
            if (__ballot(run[u]) != 0ull) {
                unsigned h;
                const bool ok = may_run<ND, T>(G, p, run[u] ? e[u] & kNodeMask : 0u, pv[u], &h);
                if (run[u]) hold[u] = h;
                run[u] = run[u] && ok;
            }
#pragma unroll
        for (int u = 0; u < kRoundPer; u++) {
            const unsigned l = e[u] & kNodeMask;
            const unsigned long long mr = __ballot(run[u]);
            if (mr) {
                unsigned b = 0u;
                if (lane == 0) b = atomicAdd(&s_nrun, (unsigned)__popcll(mr));
                b = (unsigned)__builtin_amdgcn_readfirstlane((int)b) + lane_rank(mr);
                if (run[u] && b >= (unsigned)kRoundRun) {
                    run[u] = false;
                    hold[u] = kNoHint;
                }
                if (run[u]) s_run[b] = l;
            }
            const bool keep = e[u] != kNoEntry && !run[u];
            const unsigned long long mk = __ballot(keep);
            if (mk) {
                unsigned b = 0u;
                if (lane == 0) b = atomicAdd(&s_nkeep, (unsigned)__popcll(mk));
                b = (unsigned)__builtin_amdgcn_readfirstlane((int)b) + lane_rank(mk);
                if (keep) {
                    const unsigned pk = min(pv[u], ls[u]);
                    s_keep[b] = l | hold[u] << kHintShift | kOnce;
                    at<ND>(pn, l) = pk;
                    lowest = min(lowest, pk);
                }
            }
        }
        lds_barrier();
        const unsigned nrun = min(s_nrun, (unsigned)kRoundRun), nkeep = s_nkeep;
        const auto list_fresh = [&](unsigned j, unsigned e) {
            if (j < scap) to[j] = e;
        };
        for (unsigned b = done + (unsigned)(tid & ~63); b < nrun; b += kRoundThreads) {
            const unsigned j = b + lane;
            const bool on = j < nrun;
            const unsigned l = s_run[on ? j : b];
            if (on) {
                at<ND>(pn, l) = kIdle;
                at<ND>(pr, l) = kIdle;
                at<ND>(less, l) = kIdle;
                ran[1 + j] = l;
            }
            unsigned who[4 * ND] = {}, fresh = 0u;
            bool two;
            const bool chg = relax_node<ND, T, SPH, MIX, NEAR>(
                I, G, mcart, p, l, on, settle, &two, [&](int k, bool w, unsigned q, bool idle, unsigned pq, float pf) {
                    who[k] = q | wake_tag(k) << kHintShift;
                    const unsigned pu = pend_tagged(pf, k);
                    if (w && pu < pq) {
                        lowest = min(lowest, pu);
                        atomicMin(idle ? &at<ND>(pn, q) : &at<ND>(less, q), pu);
                    }
                    fresh |= (unsigned)(w & idle) << k;
                });
            unsigned total = 0u;
#pragma unroll
            for (int k = 0; k < 4 * ND; k++)
                if (k < 2 * ND || two) total += (unsigned)__popcll(__ballot((fresh >> k) & 1u));
            // a pass that runs a thousand nodes can list more than LDS holds: the rest goes to its place at once
            if (total) {
                unsigned to_at = 0u;
                if (lane == 0) to_at = atomicAdd(&s_nfresh, total);
                to_at = (unsigned)__builtin_amdgcn_readfirstlane((int)to_at);
#pragma unroll
                for (int k = 0; k < 4 * ND; k++) {
                    if (k < 2 * ND || two) {
                        const unsigned long long m = __ballot((fresh >> k) & 1u);
                        const unsigned f = to_at + lane_rank(m);
                        if ((fresh >> k) & 1u) {
                            if (f < (unsigned)kRoundFresh) s_fresh[f] = who[k];
                            else list_fresh(out + nkeep + f, who[k]);
                        }
                        to_at += (unsigned)__popcll(m);
                    }
                }
            }
            nchg += (unsigned)__popcll(__ballot(chg));
        }
        lds_barrier();
        done = nrun;
        const unsigned nfresh = s_nfresh;
        if (tid == 0 && out + nkeep + nfresh > scap) atomicOr(&counters[3], kOverflow);
        for (unsigned i = tid; i < nkeep; i += kRoundThreads)
            if (out + i < scap) to[out + i] = s_keep[i];
        for (unsigned i = tid; i < min(nfresh, (unsigned)kRoundFresh); i += kRoundThreads) list_fresh(out + nkeep + i, s_fresh[i]);
        out = min(out + nkeep + nfresh, scap);
    }
    lowest = wave_min_u32(lowest);
    if (lane == 0) {
        s_low[wave] = lowest;
        s_chg[wave] = nchg;
    }
    lds_barrier();
    if (tid == 0) {
        unsigned lw = s_low[0], ch = s_chg[0];
        for (int w = 1; w < kRoundThreads / 64; w++) {
            lw = min(lw, s_low[w]);
            ch += s_chg[w];
        }
        S.cnt[nwords + blk] = out;
        S.low[nwords + blk] = lw;
        ran[0] = done;
        unsigned* const st = S.stat + 2 * (in * nblk + blk);
        st[0] += done;
        st[1] += ch;
    }
    if (blk == 0 && lane >= (int)nblk && wave == 0) {  // words without a block
        S.cnt[nwords + lane] = 0u;
        S.low[nwords + lane] = kIdle;
    }
}

// sums of the blocks' statistics
__global__ void __launch_bounds__(256) k_march_stats(const unsigned* __restrict__ stat, int n, unsigned long long* __restrict__ counters) {
    unsigned long long a = 0ull, c = 0ull;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        a += stat[2 * i];
        c += stat[2 * i + 1];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o);
        c += __shfl_xor(c, o);
    }
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&counters[0], a);
        atomicAdd(&counters[1], c);
    }
}

// The slowness grids in bricks: blockIdx.y is the instance that owns the grid.
template <int ND, typename T>
__global__ void __launch_bounds__(256) k_march_bricks(const InstDev* __restrict__ inst, const int* __restrict__ owner,
                                                      const T* __restrict__ slowpool, T* __restrict__ slow) {
    const InstDev& I = inst[owner[blockIdx.y]];
    const int E = fwd_tile_edge(ND);
    const int64_t n = (int64_t)I.t[0] * I.t[1] * I.t[2] * 64;
    const T* src = slowpool + I.s_off;
    T* dst = slow + I.ms_off;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int64_t b = i >> 6;
        const int o = (int)(i & 63);
        int g[3];
        g[0] = (int)(b % I.t[0]) * E + o % E;
        g[1] = (int)((b / I.t[0]) % I.t[1]) * E + (o / E) % E;
        g[2] = ND == 3 ? (int)(b / ((int64_t)I.t[0] * I.t[1])) * E + o / (E * E) : 0;
        const bool in = g[0] < I.n[0] && g[1] < I.n[1] && (ND == 2 || g[2] < I.n[2]);
        dst[i] = in ? src[g[0] + (int64_t)I.n[0] * (g[1] + (ND == 3 ? (int64_t)I.n[1] * g[2] : 0))] : T(0);
    }
}

// The values from the bricks to the x-fastest grids (blockIdx.y: instance); cascade nodes' marks come
// off their values, init nodes keep theirs and lose the depth byte.
template <int ND, typename T>
__global__ void __launch_bounds__(256) k_march_finish(const InstDev* __restrict__ inst, TTPools pools, MarchPools<T> M) {
    const InstDev& I = inst[blockIdx.y];
    const GridView<ND, T> G = grid_view<ND, T>(I, pools, M);
    T* tt = (T*)pools.tt + I.tt_off;
    const int64_t n = (int64_t)G.n[0] * G.n[1] * G.n[2];
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        int g[3];
        g[0] = (int)(i % G.n[0]);
        g[1] = (int)((i / G.n[0]) % G.n[1]);
        g[2] = ND == 3 ? (int)(i / ((int64_t)G.n[0] * G.n[1])) : 0;
        T v = G.tt[G.index(g)];
        if (signbit(v)) {
            if (G.dd[i] == kInitDepth) G.dd[i] = 0;
            else v = fabs(v);
        }
        tt[i] = v;
    }
}

// ================================================================= host side

static const char* const kMarchBuf[kMarchBufs] = {"march_tt", "march_slow", "march_pend", "march_own", "march_list", "march_cnt", "march_ran"};

// Which solver runs an instance set (EIK_MARCH overrides: kMarch*).  A workgroup per instance costs
// about the same for one instance as for one per CU, and grows with the instance's nodes; the
// whole-device rounds cost about 12 us each whatever they hold, until the device is full; the tile
// solver needs fewer, longer rounds, which wins where its sweeps are cheap and instances few and large.
// Milliseconds per call, tiles / workgroup / device, on a velocity that grows with depth (where two are
// given, the second on layers):
//   2D FP64   300x240 x 1   6.5 /  4.1 /  8.5    600x480 x 64   37.5 / 11.3 / 22.0
//             900x890 x 4     - / 33 / 41        1100x900 x 16     - / 46 / 55, - / 37 / 43
//             1200x960 x 4  52.8 / 38.7 / 34.1   1500x1400 x 24    - / 102 / 111, - / 87 / 83
//             1700x1360 x 32 189 / 114 / 128, 163 / 100 / 93       2400x1920 x 32 342 / 251 / 207
//             2400x1920 x 64   - / 264 / 288, - / 231 / 202        3000x2400 x 128  - / 516 / 631
//             2400x1920 x 4 175 / 206 / 98       600x600 sphere x 8 50.8 / 28.2 / 31.2 (mixed the same)
//   2D mixed  390x380 x 1   7.4 /  7.4, 7.0 / 6.1   570x560 x 1  11.7 / 13.4, 10.5 / 11.3
//             570x560 x 4  14.0 / 14.3, 12.9 / 11.4 650x650 x 4  17.3 / 18.3, 16.1 / 14.2
//             1060x1060 x 16 57 / 51 / 63, 62 / 45 / 48            1300x1300 x 16   73 / 82 / 85, 73 / 72 / 64
//   2D FP32   300x300 x 1   4.8 /  5.0, 4.9 / 4.5   390x380 x 1   6.2 /  7.4, 5.9 / 5.9
//             390x380 x 4   7.4 /  7.5, 7.5 / 6.2   450x450 x 4   8.8 /  9.8, 8.7 / 7.9
//             640x620 x 8  17.6 / 17.6, 17.0 / 16.1 1200x960 x 16 36.9 / 42.8 / 43.8
//   3D FP64   24^3 x 4      4.0 /  2.7 /  2.6    24^3 x 16       6.1 /  2.9 /  3.3   24^3 sphere x 1 1.5 / 1.2 / 1.7
//             48x48x28 x 16 9.7 /  5.4 /  4.6    48x48x28 x 64  15.7 /  6.2 /  6.8   64x64x38 x 64  23.3 / 11.9 / 10.8
//             100x100x60 x 1 11.3 / 32 / 6.7     200x200x120 x 4 74.6 / 1032 / 29.6 (mixed 54.2 / - / 28.9)
//             140x140x100 x 200 288 / - / 278 (mixed 282 / - / 282)
//   3D FP32   48x48x28 x 1  3.5 /  4.5 /  3.9    180x180x170 x 1 21.4 / - / 20.2     200x200x145 x 2 27.4 / - / 22.3
//             240x240x140 x 4 40.1 / - / 38.7    260x260x150 x 4 46.8 / - / 47.5     260x260x150 x 8 64.5 / - / 57.1
//             300x300x160 x 2 41.7 / - / 52.2    320x320x160 x 8 89 / - / 89         201x201x101 x 16 48.9 / - / 46
//   (FP32 on a model of sharp diagonal stripes, 2.0 and 3.5: 120x120x60 x 4 22.9 / - / 30.3, 220x220x120 x 4 49 /
//   - / 95: the size does not tell, and tiles take 1700 ms on noise where the march takes 30)
// FP32 spheres stay with the tiles: within FP32 resolution their many near-ties have several fixed points,
// and the march can circulate among them (600x600 x 8: 31 ms, the march 579).
// Unlike grids in one call (requests that share launches): the lines between the solvers hold for the largest
// grid, and as many of them as the call's nodes make.  Device rounds give every instance the same number of
// blocks, so the small ones' stand idle while the largest march on; beyond 1.5 M such bricks (nodes / 64) the
// tiles are faster.  Tiles / device, idle bricks in M: 100^3 x 16 with 60^3 x 16 92 / 46 (0.2), 140^3 x 2 with
// 80^3 x 10 and 60^3 x 25 111 / 81 (1.3), 120^3 x 10 with 90^3 x 100 210 / 200 (1.6), 112^3 x 31 with 73^3 x 51,
// 83^3 x 53 and 68^3 x 56 228 / 341 (2.5), 157^3 x 9 with 68^3 x 56 190 / 256 (3.1), 222 of 68^3 to 157^3 308 / 841 (11).
constexpr int64_t kIdleBricks = 1500000;
MarchSize march_size(int nd, int kind, int prec, int64_t ntiles, int64_t stiles, int64_t most, int ninst, int nowners) {
    const bool f32 = prec == EIK_PREC_FP32, sph = kind == EIK_GRID2D_SPHERE || kind == EIK_GRID3D_SPHERE;
    MarchSize z{ntiles, stiles, most, f32 ? sizeof(float) : sizeof(double), nullptr, nowners, kMarchNone};
    if (const char* e = getenv("EIK_MARCH")) {
        z.mode = std::max(0, std::min(2, atoi(e)));
        return z;
    }
    const int64_t nodes = most * 64, n = most > 0 ? (ntiles + most / 2) / most : 0;
    if (f32 && sph) return z;
    if (nd == 2 && f32)
        z.mode = nodes <= (n >= 8 ? 400000 : n >= 4 ? 150000 : 100000) ? kMarchGroup : kMarchNone;
    else if (nd == 2 && prec == EIK_PREC_MIXED && !sph)
        z.mode = nodes <= (n >= 16 ? 1200000 : n >= 4 ? 320000 : 210000) ? kMarchGroup : kMarchNone;
    else if (nd == 2)
        z.mode = nodes <= std::max<int64_t>(800000, 70000 * n) ? kMarchGroup : kMarchDevice;
    else if (f32 && nodes > (n >= 8 ? 10000000 : 6000000))
        z.mode = kMarchNone;
    else
        z.mode = nodes <= std::max<int64_t>(16000, 1500 * n) ? kMarchGroup : kMarchDevice;
    if (z.mode == kMarchDevice && round_blocks(ninst) < kMaxBlocks && most * ninst - ntiles > kIdleBricks) z.mode = kMarchNone;
    return z;
}

int64_t march_request_bytes(const std::vector<GridSet>& sets, const eik_params& P) {
    const eik_params e = effective_params(&P, sets[0].g->kind);
    const int nd = sets[0].g->ndim, kind = sets[0].g->kind;
    int64_t ntiles = 0, stiles = 0, most = 0, ninst = 0;
    for (const GridSet& q : sets) {
        InstDev I;
        make_inst(*q.g, I);
        set_tiles(I, nd);
        const int64_t t = (int64_t)I.t[0] * I.t[1] * I.t[2];
        ntiles += q.nsrc * t;
        stiles += t;
        most = std::max(most, t);
        ninst += q.nsrc;
    }
    if (ninst == 0 || ninst > 65535) return 0;
    const MarchSize z = march_size(nd, kind, e.precision, ntiles, stiles, most, (int)ninst, (int)sets.size());
    size_t a[kMarchBufs], f[kMarchBufs] = {};
    march_bytes(z.mode, ntiles, stiles, (int)ninst, z.esz, a);
    if (e.refinearoundsrc) {  // (a box at the model's border is smaller, and may fall on the other side of a line)
        int64_t tf = 1;
        for (int d = 0; d < nd; d++)
            tf *= ((2 * (int64_t)e.noderadius + 1) * e.downscalefactor + fwd_tile_edge(nd)) / fwd_tile_edge(nd);
        for (int mode : {kMarchGroup, kMarchDevice}) {
            size_t b[kMarchBufs];
            march_bytes(mode, ninst * tf, ninst * tf, (int)ninst, 8, b);
            for (int k = 0; k < kMarchBufs; k++) f[k] = std::max(f[k], b[k]);
        }
    }
    int64_t b = 0;
    for (int k = 0; k < kMarchBufs; k++) b += (int64_t)std::max(a[k], f[k]);
    return b + 65536;
}

bool march_reserve(eik_ctx* ctx, const MarchSize* sizes, int nsizes, int ninst) {
    if (ctx->tiles_only || ninst > 65535) return false;  // 65535: grid.y
    size_t need[kMarchBufs] = {};
    for (int i = 0; i < nsizes; i++) {
        if (sizes[i].mode != kMarchNone && sizes[i].most * 64 >= (int64_t)kNodeMask) return false;
        size_t n[kMarchBufs];
        march_bytes(sizes[i].mode, sizes[i].ntiles, sizes[i].stiles, ninst, sizes[i].esz, n);
        for (int k = 0; k < kMarchBufs; k++) need[k] = std::max(need[k], n[k]);
    }
    if (ctx->arena) {
        size_t sum = (size_t)ninst * 512 + 16384;
        for (size_t n : need) sum += n + 256;
        if (sum > ctx->arena->spare) return false;
    }
    if (ctx->march_limit >= 0) {
        int64_t sum = 0, grown = 0;
        for (int k = 0; k < kMarchBufs; k++) {
            sum += (int64_t)need[k];
            grown += (int64_t)std::max(need[k], ctx->buf(kMarchBuf[k]).cap);
        }
        if (sum > ctx->march_limit) return false;
        if (grown > ctx->march_limit) (void)march_release(ctx);
    }
    if (*std::max_element(need, need + kMarchBufs) == 0) return true;
    ctx->march_live = true;  // (no buffer of its own is released for another)
    for (int k = 0; k < kMarchBufs; k++)
        if (need[k] && ctx->buf(kMarchBuf[k]).ensure(need[k])) {
            ctx->march_live = false;
            (void)march_release(ctx);
            return false;
        }
    ctx->march_used = true;
    return true;
}

int64_t march_held(eik_ctx* ctx) {
    int64_t b = 0;
    for (const char* k : kMarchBuf) b += (int64_t)ctx->buf(k).cap;
    return b;
}

bool march_release(eik_ctx* ctx) {
    if (ctx->march_live || ctx->arena || march_held(ctx) == 0) return false;
    if (ctx->stream) (void)hipStreamSynchronize(ctx->stream);
    for (const char* b : kMarchBuf) ctx->buf(b).release();
    return true;
}

MarchScope::MarchScope(eik_ctx* ctx) : c(ctx) {
    c->march_used = march_held(c) > 0;
    if (c->peer) c->peer->march_used = march_held(c->peer) > 0;
}

MarchScope::~MarchScope() {
    const int64_t held = march_held(c) + (c->peer ? march_held(c->peer) : 0);
    size_t fr = 0;
    if (held < ((int64_t)1 << 30) || (!c->mem_total && hipMemGetInfo(&fr, &c->mem_total) != hipSuccess)) return;
    if (held <= (int64_t)(c->mem_total / 16)) return;
    (void)march_release(c);
    if (c->peer) (void)march_release(c->peer);
}

// The limit lies far above what a converging march needs (measured: up to 9 rounds per grid node along
// the axes together).  A march that has not ended by then circulates among near-ties, or in an order
// that means nothing (times that underflow a float), and the tile solver, which settles such cycles at
// rounding level, takes the call over.
MarchCtl march_ctl(const std::vector<InstDev>& coarse, const std::vector<InstDev>& fine) {
    int64_t len = 1;
    for (const std::vector<InstDev>* v : {&coarse, &fine})
        for (const InstDev& I : *v) len = std::max(len, (int64_t)I.n[0] + I.n[1] + I.n[2]);
    MarchCtl c{};
    const char* es = getenv("EIK_SETTLE_ROUND");  // test hook: settle from an earlier round (the tile solver's)
    c.max_rounds = (unsigned)(es ? std::max(0, atoi(es)) : std::min<int64_t>(2000 + 32 * len, 1 << 26));
    const char* el = getenv("EIK_LIST_LIMIT");  // test hook: lists of at most this many entries
    c.list_limit = el ? (unsigned)std::max(1, atoi(el)) : 0xffffffffu;
    return c;
}

// For the host: bit 0 if some instance has nodes listed (next round's slot), kOverflow if a list was too
// short.  After an overflow some pending nodes are in no list and hold up others for good, so the march
// has to end there.
__global__ void __launch_bounds__(256) k_march_left(const unsigned* __restrict__ cnt, int ninst,
                                                    const unsigned long long* __restrict__ counters, unsigned long long* __restrict__ left) {
    __shared__ unsigned s_any;
    if (threadIdx.x == 0) s_any = 0u;
    __syncthreads();
    unsigned any = 0u;
    for (int i = threadIdx.x; i < ninst; i += 256) any |= cnt[i];
    if (any) s_any = 1u;
    __syncthreads();
    if (threadIdx.x == 0) *left = s_any | (counters[3] & kOverflow);
}

template <typename T>
static T tinf_host() {
    return (T)INFINITY;
}

constexpr int kMarchBatch = 32;  // rounds enqueued between two looks at what is left

template <int ND, typename T, bool SPH, bool MIX, bool NEAR>
static int march_run_t(eik_ctx* ctx, const InstDev* d_inst, int ninst, const MarchSize& sz, const TTPools& P, const T* slowpool,
                       const MarchSeeds& sd, bool exact, FimStats* fs) {
    hipStream_t st = ctx->stream;
    const int64_t nb = sz.ntiles * 64;
    unsigned* pend = (unsigned*)ctx->buf("march_pend").p;  // march_reserve made the buffers
    MarchPools<T> M{(T*)ctx->buf("march_tt").p, (const T*)ctx->buf("march_slow").p, {pend, pend + nb, pend + 2 * nb},
                    (unsigned*)ctx->buf("march_own").p, (unsigned*)ctx->buf("march_own").p,  // (one or the other)
                    (unsigned*)ctx->buf("march_list").p};
    unsigned long long* d_c = (unsigned long long*)ctx->buf("march_cnt").p;
    unsigned long long* h = (unsigned long long*)ctx->h_small;
    const bool device = sz.mode == kMarchDevice;
    fill<T>(st, M.tt, nb, tinf_host<T>());
    fill<unsigned>(st, pend, (device ? 3 : 1) * nb, kIdle);
    if (device) fill<unsigned>(st, M.less, nb, kIdle);
    fill<unsigned>(st, d_c, 32, 0u);
    k_march_bricks<ND, T><<<dim3((unsigned)std::min<int64_t>(1024, (sz.most * 64 + 255) / 256), (unsigned)sz.nowners), 256, 0, st>>>(
        d_inst, sz.owners, slowpool, (T*)ctx->buf("march_slow").p);
    CK(hipGetLastError());
    MarchCtl ctl = sd.ctl;
    // changes below this relative size wake nothing (as in the tile solver; 0 in an exact solve)
    const T settle = MIX ? T(mix_settle()) : (sizeof(T) == 8 ? (!exact ? T(1e-12) : T(0)) : T(f32_settle()));
    const int blocks = round_blocks(ninst);
    // (march_ctl's limit, and rounds for the nodes that a round has no room for)
    if (ctl.max_rounds) ctl.max_rounds += (unsigned)(4 * sz.most * 64 / (device ? (int64_t)kRoundRun * blocks : (int64_t)kGroupRun));
    CK(hipEventRecord(ctx->kev[0], st));
    int64_t rounds = 0;
    if (!device) {
        constexpr int BT = 512;  // against 256: 600x400 x 256 21.2 -> 15.0 ms, 300x220 x 4 4.95 -> 4.67; 1024 is slower than both
        k_march_group<ND, T, SPH, MIX, NEAR, BT><<<(unsigned)ninst, BT, 0, st>>>(
            d_inst, P, M, sd.seeds, sd.cap, sd.nseed, settle, ctl, d_c);
        CK(hipGetLastError());
    } else {
        unsigned* words = (unsigned*)(d_c + 32);
        const size_t nw = (size_t)kMaxBlocks * ninst;
        const MarchSlots S{words, words + 2 * nw, (unsigned*)ctx->buf("march_ran").p, words + 4 * nw, ctl.list_limit};
        const dim3 gr((unsigned)ninst, (unsigned)blocks);
        k_march_seed<ND, T><<<(unsigned)ninst, 256, 0, st>>>(d_inst, ninst, P, M, sd.seeds, sd.cap, sd.nseed, S, blocks, d_c);
        CK(hipGetLastError());
        int par = 0;  // the list the next round reads
        // two batches are in flight: the host looks at what the one before left while the next runs
        for (int64_t batch = 0;; batch++) {
            for (int r = 0; r < kMarchBatch; r++, rounds++) {
                const int slot = (int)(rounds % 3);
                k_march_round<ND, T, SPH, MIX, NEAR><<<gr, kRoundThreads, 0, st>>>(d_inst, ninst, P, M, S, slot, par, settle, d_c);
                par ^= 1;
                CK(hipGetLastError());
            }
            const int k = (int)(batch & 1);
            k_march_left<<<1, 256, 0, st>>>(S.cnt + (size_t)par * nw, (int)nw, d_c, d_c + 4 + k);
            CK(hipMemcpyAsync(h + 16 + k, d_c + 4 + k, sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
            CK(hipEventRecord(ctx->kev[2 + k], st));
            if (batch > 0) {
                CK(hipEventSynchronize(ctx->kev[2 + (k ^ 1)]));
                if (h[16 + (k ^ 1)] & kOverflow) return kMarchAgain;
                if (h[16 + (k ^ 1)] == 0ull) break;
            }
            if (rounds >= ctl.max_rounds) return kMarchAgain;
        }
        k_march_stats<<<std::max(1, ninst * blocks / 2048), 256, 0, st>>>(S.stat, ninst * blocks, d_c);
        CK(hipGetLastError());
        rounds -= 2 * kMarchBatch;  // to within a batch: the last two found nothing
    }
    CK(hipEventRecord(ctx->kev[1], st));
    k_march_finish<ND, T><<<dim3((unsigned)std::min<int64_t>(1024, (sz.most * 64 + 255) / 256), (unsigned)ninst), 256, 0, st>>>(d_inst, P, M);
    CK(hipGetLastError());
    CK(hipMemcpyAsync(h, d_c, 8 * sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
    CK(hipStreamSynchronize(st));
    if (h[3]) return kMarchAgain;
    FimStats s{};
    float ms = 0.f;
    CK(hipEventElapsedTime(&ms, ctx->kev[0], ctx->kev[1]));
    s.kernel_ms = ms;
    if (ctx->tbase) {
        float a = 0.f, b = 0.f;
        CK(hipEventElapsedTime(&a, ctx->tbase, ctx->kev[0]));
        CK(hipEventElapsedTime(&b, ctx->tbase, ctx->kev[1]));
        ctx->kspans.push_back(KSpan{a, b, ctx->span_fine});
    }
    s.launches = 1;
    s.updates = (double)h[0];
    s.changed = (double)h[1];
    s.rounds = device ? rounds : (int64_t)h[2];
    s.activations = s.updates / 64.0;
    s.sweeps = s.activations;
    if (fs) *fs = s;
    return EIK_OK;
}

template <int ND, typename T, bool MIX>
static int march_run_k(eik_ctx* ctx, bool sph, bool near, const InstDev* d_inst, int ninst, const MarchSize& sz, const TTPools& P,
                       const void* slow, const MarchSeeds& sd, bool exact, FimStats* fs) {
    if constexpr (MIX) {
        if (near)
            return sph ? march_run_t<ND, T, true, true, true>(ctx, d_inst, ninst, sz, P, (const T*)slow, sd, exact, fs)
                       : march_run_t<ND, T, false, true, true>(ctx, d_inst, ninst, sz, P, (const T*)slow, sd, exact, fs);
    }
    return sph ? march_run_t<ND, T, true, MIX, false>(ctx, d_inst, ninst, sz, P, (const T*)slow, sd, exact, fs)
               : march_run_t<ND, T, false, MIX, false>(ctx, d_inst, ninst, sz, P, (const T*)slow, sd, exact, fs);
}

template <int ND>
static int march_run_nd(eik_ctx* ctx, int prec, bool sph, bool near, const InstDev* d_inst, int ninst, const MarchSize& sz,
                        const TTPools& P, const void* slow, const MarchSeeds& sd, bool exact, FimStats* fs) {
    if (prec == EIK_PREC_FP32)
        return march_run_k<ND, float, false>(ctx, sph, false, d_inst, ninst, sz, P, slow, sd, exact, fs);
    if (prec == EIK_PREC_MIXED)
        return march_run_k<ND, double, true>(ctx, sph, near, d_inst, ninst, sz, P, slow, sd, exact, fs);
    return march_run_k<ND, double, false>(ctx, sph, false, d_inst, ninst, sz, P, slow, sd, exact, fs);
}

int march_run(eik_ctx* ctx, int nd, int prec, int kind, const InstDev* d_inst, int ninst, const MarchSize& sz, const TTPools& pools,
              const void* slowpool, const MarchSeeds& sd, bool exact, bool near, FimStats* fs) {
    const bool sph = kind == EIK_GRID2D_SPHERE || kind == EIK_GRID3D_SPHERE;
    return nd == 2 ? march_run_nd<2>(ctx, prec, sph, near, d_inst, ninst, sz, pools, slowpool, sd, exact, fs)
                   : march_run_nd<3>(ctx, prec, sph, near, d_inst, ninst, sz, pools, slowpool, sd, exact, fs);
}

}  // namespace eik
