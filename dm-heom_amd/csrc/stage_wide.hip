// stage_wide.hip -- the HEOM RHS with the fused RK4 stage epilogue, and the thermal state
// search's iteration, for large systems, 8 < N <= 32 states (dm-heom/cl/heom/heom_ode.cl
// :24-451 plus rk_weighted_add.cl:19-106; thermal_state_search.cl:10-52), complex128 / FP64
// and complex64 / FP32.
//
// The state is matrix-major for these systems (heom_device.hpp: element e of ADO q at
// q * N * N + e), and one wavefront works on one ADO at a time:
//   * every access to the state, the stage operand and the outputs moves whole cache lines
//     of one matrix (lane = element);
//   * which neighbours an ADO has, and which matrices they are, is uniform over the
//     wavefront: it walks the edges that exist (seven of 48 on average in a 24-mode
//     hierarchy of depth 4), and for each the elements that its mode couples to (the rows
//     and columns of its bath's states, 47 of 576 at one state per bath) as lanes;
//   * the matrix goes to LDS once; the matrix cores take sigma H - H sigma from there as
//     16 x 16 x 4 products (rows and columns beyond N are padding), and the result replaces
//     the matrix in LDS, where the neighbour terms are added.
// The wavefronts of a workgroup share only H / hbar and the "same" constants in LDS, so there
// is a barrier only where the instance changes; the LDS accesses of one wavefront complete
// in order.
// An ADO of many edges in a launch of one ADO to a wavefront adds its terms with the elements in
// the lanes instead (add_by_element, up to 16 sites).
// Measured at 24 sites, 20,475 ADOs (ms per RK4 step; before: workgroups of 4 ADOs on element
// planes, every element's term list with a missing neighbour's zeros read as well): 1.008 ->
// 0.668 in complex128, 0.697 -> 0.449 in complex64; at 9 sites, 55 ADOs, 0.0250 -> 0.0207.  A
// complex128 step moves 3.2 GB between the L2 and the fabric at 4.7 TB/s (a large copy: 5.0), 2.3 GB
// of it the state's 12 passes and the rest neighbours that miss the L2; in complex64 it is 1.7 GB
// at 3.9 TB/s.  The two or three wavefronts of a SIMD wait 40% of their cycles for loads and LDS.
#include <algorithm>
#include <type_traits>

#include "heom_device.hpp"

namespace heom_hip {

namespace {

constexpr int kWideLdsAll = 163840;  // LDS of a CU
constexpr int kMaxWideStates = 32;
// at most 8 wavefronts per workgroup, so that a lane may hold up to 256 VGPRs
constexpr int kWideThreads = 512;
// wavefronts on a SIMD (so on a CU four times as many, with which the grid walks the
// hierarchy): as many as the registers of the kernel without spills allow (24 sites, 20,475
// ADOs, ms per RK4 step: complex128 1.42 at 3 against 0.84 at 2, with the spills of 168
// registers; complex64 0.57 at 4 against 0.54 at 3)
template <typename R, int SZ>
constexpr int kWideOccupancy = SZ <= 16                                 ? (sizeof(R) == sizeof(float) ? 5 : 4)
                               : sizeof(R) == sizeof(float) && SZ <= 24 ? 3
                                                                        : 2;
constexpr int kWideCus = 256;
// bytes of the places by mode that a workgroup keeps in LDS, at most
constexpr int kWideWhereBytes = 16384;
// modes whose neighbour loads are in flight together: more where a wavefront has one ADO at
// most (ONE: no registers for the next one's matrix, and the ADOs with an edge in every mode
// are the launch's critical path).  A mode costs its wavefront some 400 cycles of issue
// besides the loads, so more of them ahead only wait for one another (ms per RK4 step at 24
// sites, 20,475 ADOs: 0.682 with 2, 0.692 with 3, 0.728 with 4; at 9 sites, 715 ADOs, one
// each: 0.0304 with 3, 0.0337 with 4).
template <typename R, int SZ, bool ONE>
constexpr int kWideModesAhead = SZ > 24 && sizeof(R) == sizeof(double) ? (ONE ? 2 : 1) : (ONE ? 3 : 2);

// LDS of a workgroup of T wavefronts, in bytes: the constant matrix (H / hbar or C, complex or
// its real part), the places by mode (where they take at most kWideWhereBytes), the "same"
// constants (not beside 32 x 32 matrices in complex128), and a matrix per wavefront.  What lies
// where is known at compile time: a pointer into either memory would make every access wait
// for all loads under way.
template <typename R, int SZ>
constexpr bool kWideGamLds = sizeof(R) == sizeof(float) || SZ <= 24;
struct WideLds {
    int gam, where, mat, total;
};
__host__ __device__ constexpr int wide_round16(int b) { return (b + 15) / 16 * 16; }
__host__ __device__ constexpr WideLds wide_lds(int N, int cbytes, bool real, bool gam_lds, int T, int where_bytes)
{
    const int m = N * wide_pitch(N), h = wide_round16((real ? cbytes / 2 : cbytes) * m), g = gam_lds ? cbytes * m : 0;
    const int el = wide_round16(where_bytes);
    return {h, h + g, h + g + el, h + g + el + T * cbytes * m};
}
// bytes of the places by mode in LDS, 0 if they stay in global memory
constexpr int wide_where_bytes(int words) { return words * 4 <= kWideWhereBytes ? words * 4 : 0; }
// the most wavefronts that the LDS holds the matrices of: 8 but for 32 x 32 in complex128 with
// a complex constant matrix and many places, where it is 4
constexpr int wide_most_waves(int N, int cbytes, bool real, int words)
{
    const bool gam_lds = cbytes == sizeof(float2) ? kWideGamLds<float, kMaxWideStates>
                         : N <= 24                ? kWideGamLds<double, 24>
                                                  : kWideGamLds<double, kMaxWideStates>;
    int T = kWideThreads / 64;
    while (T > 1 && wide_lds(N, cbytes, real, gam_lds, T, wide_where_bytes(words)).total > kWideLdsAll)
        T /= 2;
    return T;
}

template <typename R>
using v4 = R __attribute__((ext_vector_type(4)));

// d += a b, 16 x 16 x 4: lane l holds a[l % 16][l / 16], b[l / 16][l % 16] and, in d, four
// elements of column l % 16 at the rows d_row(l, 0..3)
__device__ __forceinline__ v4<double> mfma(double a, double b, v4<double> c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4<float> mfma(float a, float b, v4<float> c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
template <typename R>
__device__ __forceinline__ int d_row(int lane, int v);
template <>
__device__ __forceinline__ int d_row<double>(int lane, int v)
{
    return (lane >> 4) + 4 * v;
}
template <>
__device__ __forceinline__ int d_row<float>(int lane, int v)
{
    return 4 * (lane >> 4) + v;
}

// what one lane wrote to LDS before is what another lane of the wavefront reads after: the
// hardware keeps a wavefront's LDS accesses in order, the compiler has to as well
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

template <typename R, int NB>
struct Product {
    v4<R> re[NB][NB], im[NB][NB];
    __device__ __forceinline__ void clear()
    {
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b)
                re[a][b] = im[a][b] = v4<R>{R(0), R(0), R(0), R(0)};
    }
};

// p += sigma M (LEFT = false) or M sigma, or with NEG minus that, M (real or complex) or its
// transpose in LDS.  k = 4 s + l / 16 at step s; zero in k beyond N; rows and columns of the
// result beyond N are not kept, so their operands may be anything inside the matrix.
template <bool LEFT, bool TRANS, bool NEG, typename R, int NB, int NP, typename TM>
__device__ __forceinline__ void multiply(Product<R, NB>& p, const c2<R>* sig, const TM* m, int N, int lane)
{
    constexpr bool REAL = sizeof(TM) == sizeof(R);
    const int g = lane >> 4;
    const c2<R>* xs[NB];
    const TM* ys[NB];
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        const int r = min(16 * t + (lane & 15), N - 1);
        xs[t] = sig + (LEFT ? g * NP + r : r * NP + g);
        ys[t] = m + (LEFT != TRANS ? r * NP + g : g * NP + r);
    }
    constexpr int XK = LEFT ? NP : 1, YK = LEFT != TRANS ? 1 : NP;  // strides in k
    auto step = [&](int k0, bool in) {
        c2<R> x[NB];
        TM y[NB];
#pragma unroll
        for (int t = 0; t < NB; ++t) {
            x[t] = xs[t][in ? k0 * XK : 0];
            y[t] = ys[t][in ? k0 * YK : 0];
            if (!in)
                x[t] = mk2<R>(R(0), R(0));
            if constexpr (REAL)
                y[t] = in ? (NEG ? -y[t] : y[t]) : R(0);
            else
                y[t] = in ? (NEG ? mk2<R>(-y[t].x, -y[t].y) : y[t]) : mk2<R>(R(0), R(0));
        }
        auto add = [&](v4<R>& c, R xv, R yv) { c = LEFT ? mfma(yv, xv, c) : mfma(xv, yv, c); };
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const c2<R> xv = LEFT ? x[b] : x[a];
                const TM yv = LEFT ? y[a] : y[b];
                if constexpr (REAL) {
                    add(p.re[a][b], xv.x, yv);
                    add(p.im[a][b], xv.y, yv);
                } else {
                    add(p.re[a][b], xv.x, yv.x);
                    add(p.re[a][b], -xv.y, yv.y);
                    add(p.im[a][b], xv.y, yv.x);
                    add(p.im[a][b], xv.x, yv.y);
                }
            }
    };
    int k0 = 0;
#pragma unroll 2
    for (; k0 + 4 <= N; k0 += 4)
        step(k0, true);
    if (k0 < N)
        step(k0, k0 + g < N);
}

// p += sigma H - H sigma, complex128: the two products one after the other
template <int NB, int NP, typename TM>
__device__ __forceinline__ void commutator(Product<double, NB>& p, const double2* sig, const TM* h, int N, int lane)
{
    multiply<false, false, false, double, NB, NP>(p, sig, h, N, lane);
    multiply<true, false, true, double, NB, NP>(p, sig, h, N, lane);
}

// The same for complex64, where the order of the sum shows in the sixth digit of small
// elements: the products interleave in the k steps of the matrix cores, lane group
// g = lane / 16 holding a factor of
//   real H:     -H_ik sigma_kj (g = 0, 2) and sigma_ik H_kj (g = 1, 3), two k to a step;
//   complex H:  sigma_ik H_kj as x.x, y.y and -H_ik sigma_kj as x.x, y.y (real part; the
//               imaginary part x.y, y.x of each), one k to a step,
// which sums every element in the order of k, as the scalar loop of the kernels for N <= 8
// does.  A lane needs one element of sigma and one of H per step and 16-block: it is the left
// operand of one product and the right operand of the other.
template <int NB, int NP>
__device__ __forceinline__ void commutator(Product<float, NB>& p, const float2* sig, const float* h, int N, int lane)
{
    const int g = lane >> 4;
    const bool odd = g & 1;
    const int xk = odd ? 1 : NP, hk = odd ? NP : 1;  // strides in k
    const float2* xs[NB];
    const float* ys[NB];
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        const int r = min(16 * t + (lane & 15), N - 1), k = g >> 1;
        xs[t] = sig + (odd ? r * NP + k : k * NP + r);
        ys[t] = h + (odd ? k * NP + r : r * NP + k);
    }
    auto step = [&](int k0, bool in) {
        float2 x[NB];
        float y[NB];
#pragma unroll
        for (int t = 0; t < NB; ++t) {
            x[t] = xs[t][in ? k0 * xk : 0];
            y[t] = ys[t][in ? k0 * hk : 0];
            if (!in)
                x[t] = make_float2(0.f, 0.f);
            y[t] = in ? (odd ? y[t] : -y[t]) : 0.f;
        }
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                p.re[a][b] = mfma(odd ? x[a].x : y[a], odd ? y[b] : x[b].x, p.re[a][b]);
                p.im[a][b] = mfma(odd ? x[a].y : y[a], odd ? y[b] : x[b].y, p.im[a][b]);
            }
    };
    int k0 = 0;
#pragma unroll 2
    for (; k0 + 2 <= N; k0 += 2)
        step(k0, true);
    if (k0 < N)
        step(k0, g < 2);
}
template <int NB, int NP>
__device__ __forceinline__ void commutator(Product<float, NB>& p, const float2* sig, const float2* h, int N, int lane)
{
    const int g = lane >> 4;
    const bool odd = g & 1, first = g < 2;  // first: sigma H
    const int xk = first ? 1 : NP, hk = first ? NP : 1;
    const float2 *xs[NB], *ys[NB];
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        const int r = min(16 * t + (lane & 15), N - 1);
        xs[t] = sig + (first ? r * NP : r);
        ys[t] = h + (first ? r : r * NP);
    }
#pragma unroll 2
    for (int k = 0; k < N; ++k) {
        float2 x[NB], y[NB];
#pragma unroll
        for (int t = 0; t < NB; ++t) {
            x[t] = xs[t][k * xk];
            y[t] = ys[t][k * hk];
        }
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                // left and right factors: re  (x.x, y.x), (-x.y, y.y) | (-y.x, x.x), (y.y, x.y)
                //                         im  (x.x, y.y), (x.y, y.x)  | (-y.x, x.y), (-y.y, x.x)
                const float ar = first ? (odd ? -x[a].y : x[a].x) : (odd ? y[a].y : -y[a].x);
                const float br = first ? (odd ? y[b].y : y[b].x) : (odd ? x[b].y : x[b].x);
                const float ai = first ? (odd ? x[a].y : x[a].x) : (odd ? -y[a].y : -y[a].x);
                const float bi = first ? (odd ? y[b].x : y[b].y) : (odd ? x[b].x : x[b].y);
                p.re[a][b] = mfma(ar, br, p.re[a][b]);
                p.im[a][b] = mfma(ai, bi, p.im[a][b]);
            }
    }
}

// value = fn(place, i, j, value) for the elements (i, j) of a product that lie in N x N;
// place = i * NP + j
template <typename R, int NB, int NP, typename Fn>
__device__ __forceinline__ void each_element(Product<R, NB>& p, int N, int lane, Fn&& fn)
{
    const int i0 = d_row<R>(lane, 0), j0 = lane & 15, at0 = i0 * NP + j0;
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int di = 16 * a + d_row<R>(0, v), dj = 16 * b;
                if (i0 + di < N && j0 + dj < N) {
                    const c2<R> r = fn(at0 + di * NP + dj, i0 + di, j0 + dj, mk2<R>(p.re[a][b][v], p.im[a][b][v]));
                    p.re[a][b][v] = r.x;
                    p.im[a][b][v] = r.y;
                }
            }
}

// the value of `tab` in lane `idx`, the same in every lane
__device__ __forceinline__ double uniform_lane(double tab, int idx)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(tab), idx),
                            __builtin_amdgcn_readlane(__double2loint(tab), idx));
}
__device__ __forceinline__ float uniform_lane(float tab, int idx)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tab), idx));
}

// one ADO's lanes of 64 modes' table entries
struct EdgeLanes {
    int2 v;
    __device__ __forceinline__ void load(const int2* nb, int64_t mp, int64_t q, int m, int W, int zero_slot)
    {
        v = m < W ? nb[(int64_t)m * mp + q] : make_int2((int32_t)((uint32_t)zero_slot << 6), zero_slot);
    }
};

// The neighbour terms of one ADO, summed into the matrix f in LDS: for every element in the
// order of the modes, plus before minus.  Its edges in modes m0 .. m0 + 63 are in the lanes of
// `ed`; the modes with an edge are walked with D of them in flight (a mode that couples to
// more than 64 elements makes several rounds, as many as its own list needs: with all modes as
// long as the longest, 24 sites with a bath each and one more for all of them, 3,276 ADOs, took
// 0.441 ms per RK4 step, 0.180 so).  Every round makes the same loads -- through a buffer
// resource that ends at once where the edge is missing, so that nothing is read and zeros come
// back -- and so the wait for one round's loads is not one for those behind it.  `where` is
// this class's, in LDS where it fits.
template <typename R, int D, bool LONG>
struct Neighbours {
    using C = c2<R>;
    using V = vec2_t<R>;
    const StageArgsT<R>& a;
    const WideTables<R>& wt;
    const TermT<R>* terms;
    const uint32_t* where;
    int64_t q;
    int nel, lane, m0 = 0, round = 0, todo;
    EdgeLanes ed;
    uint32_t spans;  // of the modes in the lanes (LONG: stride = 0)
    uint64_t has_p, has_m, left;
    V mc[D], xp[D], xm[D];
    R pc[D];
    int at[D], n[D];

    __device__ __forceinline__ Neighbours(const StageArgsT<R>& a_, const WideTables<R>& wt_, int cls,
                                          const uint32_t* where_, EdgeLanes entries, int64_t q_, int nel_, int lane_)
        : a(a_), wt(wt_), terms(wt_.terms + (int64_t)cls * wt_.words), where(where_), q(q_), nel(nel_),
          lane(lane_), ed(entries)
    {
        begin();
    }
    __device__ __forceinline__ void begin()
    {
        has_p = __ballot((int32_t)((uint32_t)ed.v.x >> 6) != a.zero_slot);
        has_m = __ballot(ed.v.y != a.zero_slot);
        left = has_p | has_m;
        todo = __popcll(left) * ((wt.stride + 63) / 64);
        if (LONG) {
            todo = __popcll(left);
            spans = m0 + lane < wt.W ? where[m0 + lane] : 0;
            uint64_t longer = left;
            for (int r = 1; longer != 0; ++r) {
                longer &= __ballot((int)(spans >> 16) > 64 * r);
                todo += __popcll(longer);
            }
        }
        round = 0;
    }
    __device__ __forceinline__ void start()
    {
#pragma unroll
        for (int u = 0; u < D; ++u)
            fetch(u);
    }
    __device__ __forceinline__ V element(int64_t slot, bool there, int pos) const
    {
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(a.yin + slot * nel), (short)0, there ? nel * (int)sizeof(C) : 0, 0x00020000);
        if constexpr (sizeof(C) == 16) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, pos * (int)sizeof(C), 0, 0);
            return V{__hiloint2double((int)v[1], (int)v[0]), __hiloint2double((int)v[3], (int)v[2])};
        } else {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, pos * (int)sizeof(C), 0, 0);
            return V{__int_as_float((int)v[0]), __int_as_float((int)v[1])};
        }
    }
    // requests the next mode (none left: loads that read nothing, or a term that is not used)
    __device__ __forceinline__ void fetch(int u)
    {
        const bool some = left != 0;
        const int m = some ? __builtin_ctzll(left) : 0;
        const int vx = __builtin_amdgcn_readlane(ed.v.x, m), vy = __builtin_amdgcn_readlane(ed.v.y, m);
        const int k = lane + 64 * round;
        int count = wt.stride, from = (m0 + m) * wt.stride;
        if (LONG) {
            const uint32_t span = (uint32_t)__builtin_amdgcn_readlane((int)spans, m);
            count = (int)(span >> 16);
            from = (int)(span & 0xffff);
        }
        const int i = from + (LONG ? max(min(k, count - 1), 0) : min(k, count - 1));
        const bool in = k < count;
        if (++round * 64 >= count) {
            round = 0;
            left &= left - 1;
        }
        const uint32_t pp = where[i];
        const bool p = (has_p >> m & 1) && some, mn = (has_m >> m & 1) && some;
        xp[u] = element(p ? (int64_t)((uint32_t)vx >> 6) : 0, p, (int)(pp & 0xffff));
        xm[u] = element(mn ? (int64_t)(uint32_t)vy : 0, mn, (int)(pp & 0xffff));
        mc[u] = V{terms[i].minus_c.x, terms[i].minus_c.y};
        pc[u] = terms[i].plus_c;
        at[u] = some && in ? (int)(pp >> 16) : 0xffff;
        n[u] = vx & 63;
    }
    template <bool SCALED>
    __device__ __forceinline__ void add(int u, R scale, R sq_lane, C* f)
    {
        const R sp = uniform_lane(sq_lane, n[u] + 1), sm = uniform_lane(sq_lane, n[u]);
        const R cp = SCALED ? scale * (pc[u] * sp) : pc[u] * sp, cm = SCALED ? scale * sm : sm;
        if (at[u] != 0xffff) {
            C s = f[at[u]];
            s.x = fma(-cp, xp[u].y, s.x);
            s.y = fma(cp, xp[u].x, s.y);
            f[at[u]] = cfma(mk2<R>(mc[u].x, mc[u].y), mk2<R>(cm * xm[u].x, cm * xm[u].y), s);
        }
        wave_sync();
    }
    template <bool SCALED>
    __device__ __forceinline__ void run(R scale, R sq_lane, C* f)
    {
        for (;;) {
            for (; todo > D; todo -= D)
#pragma unroll
                for (int u = 0; u < D; ++u) {
                    add<SCALED>(u, scale, sq_lane, f);
                    fetch(u);
                }
#pragma unroll
            for (int u = 0; u < D; ++u)
                if (u < todo)
                    add<SCALED>(u, scale, sq_lane, f);
            m0 += 64;
            if (m0 >= wt.W)
                break;
            ed.load(a.nb, a.mp, q, m0 + lane, wt.W, a.zero_slot);
            begin();
            start();
        }
    }
};

// The same sum with the elements in the lanes, each with its own list of NT terms in the order of
// the modes (`lists`, by position): for an ADO with edges in many modes, whose walk is a chain
// of an LDS pass a mode.  Two slots of two of a lane's NL elements are requested together.  The ADO's
// edges are all in the lanes of `ed` (W <= 64).
template <bool SCALED, typename R, int NL, typename Place>
__device__ __forceinline__ void add_by_element(const StageArgsT<R>& a, const TermT<R>* lists, int NT, int W, int2 ed,
                                               int nel, int lane, R scale, R sq_lane, Place&& place, c2<R>* f)
{
    using V = vec2_t<R>;
    constexpr int G = NL < 2 ? NL : 2, B = 2;
    const int n = ed.x & 63;
    const R sp_lane = __shfl(sq_lane, n + 1), sm_lane = __shfl(sq_lane, n);
#pragma unroll
    for (int k0 = 0; k0 < NL; k0 += G) {
        c2<R> s[G];
        const TermT<R>* te[G];
#pragma unroll
        for (int k = 0; k < G && k0 + k < NL; ++k) {
            te[k] = lists + min(lane + 64 * (k0 + k), nel - 1) * NT;
            s[k] = f[place(k0 + k)];
        }
        for (int t = 0; t < NT; t += B) {
            V mc[G][B], xp[G][B], xm[G][B];
            R pc[G][B];
            int mode[G][B];
#pragma unroll
            for (int k = 0; k < G && k0 + k < NL; ++k)
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    mode[k][b] = te[k][t + b].mode;
                    pc[k][b] = te[k][t + b].plus_c;
                    mc[k][b] = V{te[k][t + b].minus_c.x, te[k][t + b].minus_c.y};
                }
#pragma unroll
            for (int k = 0; k < G && k0 + k < NL; ++k)
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    const int m = mode[k][b], e = lane + 64 * (k0 + k);
                    const uint32_t plus = (uint32_t)__shfl(ed.x, m) >> 6, minus = (uint32_t)__shfl(ed.y, m);
                    const bool in = m < W && e < nel;  // W: a slot without a term
                    xp[k][b] = xm[k][b] = V{R(0), R(0)};
                    if (in && (int32_t)plus != a.zero_slot)
                        xp[k][b] = *reinterpret_cast<const V*>(a.yin + (int64_t)plus * nel + e);
                    if (in && (int32_t)minus != a.zero_slot)
                        xm[k][b] = *reinterpret_cast<const V*>(a.yin + (int64_t)minus * nel + e);
                }
#pragma unroll
            for (int k = 0; k < G && k0 + k < NL; ++k)
#pragma unroll
                for (int b = 0; b < B; ++b) {
                    const R sp = __shfl(sp_lane, mode[k][b]), sm = __shfl(sm_lane, mode[k][b]);
                    const R cp = SCALED ? scale * (pc[k][b] * sp) : pc[k][b] * sp, cm = SCALED ? scale * sm : sm;
                    s[k].x = fma(-cp, xp[k][b].y, s[k].x);
                    s[k].y = fma(cp, xp[k][b].x, s[k].y);
                    s[k] = cfma(mk2<R>(mc[k][b].x, mc[k][b].y), mk2<R>(cm * xm[k][b].x, cm * xm[k][b].y), s[k]);
                }
        }
#pragma unroll
        for (int k = 0; k < G && k0 + k < NL; ++k)
            if (lane + 64 * (k0 + k) < nel)
                f[place(k0 + k)] = s[k];
    }
    wave_sync();
}

// The sequence of groups of T consecutive ADOs (one per wavefront) of a workgroup: the tiles
// in tile_order are dealt to the XCDs in turn, a tile's groups to the XCD's workgroups in
// turn.  T divides the 64-ADO tile, so a group has one instance and one bath class.  The tiles
// with plus neighbours come first in the order: their ADOs have several times the edges of the
// others, and every workgroup gets its share of them.
struct Walk {
    const int32_t* order;
    int x, j, gx, per, T, nt;
    __device__ __forceinline__ Walk(const int32_t* order_, int ntiles, int T_)
        : order(order_), x((int)(blockIdx.x % kNumXcd)), j((int)(blockIdx.x / kNumXcd)),
          gx((int)(gridDim.x / kNumXcd)), per(kTile / T_), T(T_), nt(ntiles)
    {
    }
    // the first ADO of the XCD's jj-th group, or -1 past the end (IN_ORDER: of the tiles as
    // they lie, without a look at tile_order: where every workgroup has one group)
    template <bool IN_ORDER>
    __device__ __forceinline__ int64_t group(int jj) const
    {
        const int t = jj / per * kNumXcd + x;
        if (t >= nt)
            return -1;
        return (int64_t)(IN_ORDER ? t : __builtin_amdgcn_readfirstlane(order[t])) * kTile + jj % per * T;
    }
};

// Whether an ADO whose walk has `rounds` rounds adds its terms by element, NL elements to a lane
// with `slots` terms each: a round costs its wavefront 0.27 us, a slot about 1.5 rounds.  In a
// launch of one ADO to a wavefront the ADOs with an edge in every mode set its length (ms per
// RK4 step in complex128, walked and by element: 9 sites, 55 ADOs 0.0243 and 0.0207; with four
// modes per site, 703 ADOs 0.0540 and 0.0407; 16 sites, three modes each, 1,225 ADOs, 48 rounds
// for 32 slots 0.0796 and 0.0842).  Launches in which no ADO can reach it have kernels without
// that code, which their registers notice (16 sites in 4 baths, 210 ADOs: 0.0296 and 0.0284).
__host__ __device__ constexpr bool by_element(int rounds, int NL, int slots) { return 2 * rounds > 3 * NL * slots; }

// one matrix in registers, lane = element: NL elements per lane
template <typename R, int NL>
struct Lin {
    vec2_t<R> v[NL];
    __device__ __forceinline__ c2<R> operator[](int k) const { return mk2<R>(v[k].x, v[k].y); }
    __device__ __forceinline__ void load(const c2<R>* p, int nel, int lane)
    {
#pragma unroll
        for (int k = 0; k < NL; ++k)
            if (lane + 64 * k < nel)
                v[k] = *reinterpret_cast<const vec2_t<R>*>(p + lane + 64 * k);
    }
    __device__ __forceinline__ void load_nt(const c2<R>* p, int nel, int lane)
    {
#pragma unroll
        for (int k = 0; k < NL; ++k)
            if (lane + 64 * k < nel)
                v[k] = __builtin_nontemporal_load(reinterpret_cast<const vec2_t<R>*>(p + lane + 64 * k));
    }
};

// the workgroup's constants in LDS: M (H / hbar or C; its real part for TM = R), gam and the
// places by mode
template <typename R, typename TM, int SZ, bool WLDS>
__device__ __forceinline__ void load_constants(const c2<R>* __restrict__ m, const c2<R>* __restrict__ gam,
                                               const uint32_t* __restrict__ where, int words, int N, TM* ml,
                                               c2<R>* gl, uint32_t* el, bool first)
{
    const int NP = wide_pitch(N);
    const uint32_t ninv = (1u << 20) / (uint32_t)N + 1u;
    if (!first)
        __syncthreads();  // nobody uses the previous ones any more
    // the loads of up to four rounds before the first store
    constexpr int U = SZ <= 16 ? 1 : 4;
    constexpr bool GL = kWideGamLds<R, SZ>;
    const int n = N * N, step = (int)blockDim.x;
    for (int e0 = threadIdx.x; e0 < n; e0 += U * step) {
        vec2_t<R> mv[U], gv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = min(e0 + u * step, n - 1);
            mv[u] = vec2_t<R>{m[e].x, m[e].y};
            if (GL)
                gv[u] = vec2_t<R>{gam[e].x, gam[e].y};
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = min(e0 + u * step, n - 1);  // past the end: the last element again
            const int at = e + (NP - N) * (int)(((uint32_t)e * ninv) >> 20);
            if constexpr (sizeof(TM) == sizeof(R))
                ml[at] = mv[u].x;
            else
                ml[at] = mk2<R>(mv[u].x, mv[u].y);
            if (GL)
                gl[at] = mk2<R>(gv[u].x, gv[u].y);
        }
    }
    if (WLDS)
        for (int i0 = threadIdx.x; i0 < words; i0 += U * step) {
            uint32_t v[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                v[u] = where[min(i0 + u * step, words - 1)];
#pragma unroll
            for (int u = 0; u < U; ++u)
                el[min(i0 + u * step, words - 1)] = v[u];
        }
    __syncthreads();
}

// One RK4 stage (STAGE 1..4, or 0: the RHS alone) over the whole hierarchy.  N <= SZ.
template <typename R, int SZ, int STAGE, bool REALH, bool ONE, bool WLDS, bool LONG, bool BYEL>
__global__ __launch_bounds__(kWideThreads) __attribute__((amdgpu_waves_per_eu(kWideOccupancy<R, SZ>)))
void rk4_stage_wide(StageArgsT<R> a, WideTables<R> wt, const c2<R>* __restrict__ hs_all,
                    const c2<R>* __restrict__ gam_all, int N_, int T)
{
    using C = c2<R>;
    using TM = std::conditional_t<REALH, R, C>;
    constexpr int NB = (SZ + 15) / 16, NL = (SZ * SZ + 63) / 64, NP = wide_pitch(SZ);
    // complex128: the neighbour terms are added, times c1, to the value that already holds
    // the rest of the result; complex64: they are summed by themselves (stages 1 and 4),
    // since one rounding more or less shows there
    constexpr bool LINEAR = STAGE == 1 || STAGE == 4;
    constexpr bool APART = LINEAR && sizeof(R) == sizeof(float);
    // the next ADO's matrix goes to registers during the neighbour terms (36 at most; stage 2
    // needs its own values to the end and loads the next ones after that)
    constexpr bool EARLY = STAGE != 2 && NL * sizeof(C) <= 144;
    extern __shared__ __align__(16) unsigned char wide_mem[];
    // one round trip for the arguments that the first loads need, not one at each of them (9
    // sites, 715 ADOs: 0.0285 -> 0.0268 ms per RK4 step); not in the longer kernels, which
    // have no scalar registers to spare
    if (ONE)
        asm volatile("" ::"s"(a.yin), "s"(a.nb), "s"(a.mp), "s"(a.pfss), "s"(a.tile_inst), "s"(a.tile_class), "s"(wt.place),
                     "s"(wt.where), "s"(wt.terms), "s"(wt.W), "s"(wt.stride), "s"(wt.words), "s"(hs_all), "s"(gam_all), "s"(N_), "s"(T),
                     "s"(wt.slots), "s"(a.zero_slot), "s"(a.ntiles), "s"(a.y0), "s"(a.yout));
    const int nel = N_ * N_;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int words = wt.words;
    constexpr bool GL = kWideGamLds<R, SZ>;
    const WideLds L = wide_lds(N_, (int)sizeof(C), REALH, GL, T, WLDS ? words * 4 : 0);
    TM* hl = reinterpret_cast<TM*>(wide_mem);
    C* gl = reinterpret_cast<C*>(wide_mem + L.gam);
    uint32_t* el = reinterpret_cast<uint32_t*>(wide_mem + L.where);
    C* sig = reinterpret_cast<C*>(wide_mem + L.mat) + (int64_t)w * (N_ * NP);  // this wavefront's matrix
    int places[(NL + 1) / 2];  // of this lane's elements, two to a register
#pragma unroll
    for (int k = 0; k < NL; ++k) {
        const int at = wt.place[min((int)(threadIdx.x & 63) + 64 * k, nel - 1)];
        places[k / 2] = k & 1 ? places[k / 2] | at << 16 : at;
    }
    auto place = [&](int k) { return k & 1 ? (int)((uint32_t)places[k / 2] >> 16) : places[k / 2] & 0xffff; };
    const R sq_lane = sqrt((R)(threadIdx.x & 63));  // sqrt(n), n = 0..63, one value per lane

    const Walk walk(wt.tile_order, a.ntiles, T);
    int j = walk.j, inst = -1, cls = -1;
    const int lane_ = threadIdx.x & 63;
    int64_t q0 = walk.template group<ONE>(j);
    if (q0 < 0)
        return;  // the whole workgroup leaves together
    // a wavefront whose slot holds no ADO (the last tile's padding) goes through the motions
    // with the last ADO and stores nothing
    auto slot = [&](int64_t g) { return min(g + w, (int64_t)a.zero_slot - 1); };
    Lin<R, NL> own;
    EdgeLanes ed;
    own.load(a.yin + slot(q0) * nel, nel, lane_);
    ed.load(a.nb, a.mp, slot(q0), lane_, wt.W, a.zero_slot);
    for (;;) {
        const int it = a.tile_inst ? a.tile_inst[q0 / kTile] : 0;
        const int cl = tile_bath_class(a, (int)(q0 / kTile));
        const C* gam = gam_all + (int64_t)cl * nel;
        const uint32_t* where = wt.where + (int64_t)cl * words;
        if (it != inst || cl != cls)
            load_constants<R, TM, SZ, WLDS>(hs_all + (int64_t)it * nel, gam, where, words, N_, hl, gl, el, inst < 0);
        inst = it;
        cls = cl;
        j += walk.gx;
        const int64_t q = slot(q0), q0n = ONE ? -1 : walk.template group<ONE>(j);
        const bool live = q0 + w < a.zero_slot;
        auto ahead = [&](bool edges, bool matrix) {  // the next ADO's
            if (q0n >= 0) {
                if (edges)
                    ed.load(a.nb, a.mp, slot(q0n), lane_, wt.W, a.zero_slot);
                if (matrix)
                    own.load(a.yin + slot(q0n) * nel, nel, lane_);
            }
        };
        // the masks and addresses of the elements are formed where they are used: kept over
        // the loop they would not fit the registers
        int lane = lane_, N = N_;
        asm volatile("" : "+v"(lane), "+s"(N));
        const C S = a.pfss[q];
        Lin<R, NL> ep;
        auto operand = [&] {
            if (STAGE == 2 || STAGE == 3)
                ep.load_nt(a.y0 + q * nel, nel, lane);
            if (STAGE == 4)
                ep.load_nt(a.pbuf + q * nel, nel, lane);
        };
        {
#pragma unroll
            for (int k = 0; k < NL; ++k)
                if (lane + 64 * k < nel)
                    sig[place(k)] = own[k];
            wave_sync();
            // the first neighbours are under way during the commutator
            Neighbours<R, kWideModesAhead<R, SZ, ONE>, LONG> nbs(a, wt, cl, WLDS ? el : where, ed, q, nel, lane);
            nbs.start();
            __builtin_amdgcn_sched_barrier(0);

            Product<R, NB> cm;  // sigma H - H sigma (over hbar)
            cm.clear();
            commutator<NB, NP>(cm, sig, hl, N, lane);
            wave_sync();
            each_element<R, NB, NP>(cm, N, lane, [&](int at, int i, int jj, C c) {
                const C g = GL ? gl[at] : gam[i * N + jj];
                const C s = sig[at];
                const C fb = cfma(mk2<R>(S.x + g.x, S.y + g.y), s, mk2<R>(-c.y, c.x));
                // stages 1 and 4 take the element's own value linearly (s + c1 f, and
                // (ep + s) / 3 + c1 f): its part goes in here
                C r = fb;
                if (STAGE == 1)
                    r = mk2<R>(fma(a.c1, fb.x, s.x), fma(a.c1, fb.y, s.y));
                else if (STAGE == 4)
                    r = mk2<R>(fma(s.x, R(1) / R(3), a.c1 * fb.x), fma(s.y, R(1) / R(3), a.c1 * fb.y));
                sig[at] = APART ? mk2<R>(R(0), R(0)) : r;
                return r;
            });
            wave_sync();
            __builtin_amdgcn_sched_barrier(0);
            operand();  // the neighbour terms cover it
            if (BYEL && wt.W <= 64 && by_element(nbs.todo, NL, wt.slots))
                add_by_element<LINEAR && !APART, R, NL>(a, wt.lists + (int64_t)cl * nel * wt.slots, wt.slots, wt.W, ed.v,
                                                        nel, lane, a.c1, sq_lane, place, sig);
            else
                nbs.template run<LINEAR && !APART>(a.c1, sq_lane, sig);
            if (!ONE)
                ahead(true, EARLY);
            wave_sync();
            if (APART) {
                each_element<R, NB, NP>(cm, N, lane, [&](int at, int, int, C r) {
                    const C f = sig[at];
                    sig[at] = mk2<R>(fma(a.c1, f.x, r.x), fma(a.c1, f.y, r.y));
                    return r;
                });
                wave_sync();
            }
#pragma unroll
            for (int k = 0; k < NL; ++k) {
                const int e = lane + 64 * k;  // position
                if (e >= nel)
                    continue;
                const C f = sig[place(k)];
                C r0, r1 = mk2<R>(R(0), R(0));
                if (STAGE == 1) {
                    r0 = f;
                } else if (STAGE == 4) {
                    constexpr R third = R(1) / R(3);
                    r0 = mk2<R>(fma(ep[k].x, third, f.x), fma(ep[k].y, third, f.y));
                } else {
                    stage_values<STAGE, R>(a.c1, STAGE == 2 ? own[k] : mk2<R>(R(0), R(0)), f,
                                           STAGE == 2 || STAGE == 3 ? ep[k] : mk2<R>(R(0), R(0)), r0, r1);
                }
                if (live)
                    stage_store<STAGE, R>(a, q * nel + e, r0, r1);
            }
            wave_sync();
            if (!ONE && !EARLY)
                ahead(false, true);
        }
        if (ONE || q0n < 0)
            break;
        q0 = q0n;
    }
}

// One iteration of the thermal state search (tss.hip): y_u = C^T [ (C k_u C^T) / D_u ] C with
// k = f_TSS(y), the "same" and neighbour terms alone; the matrix stays in LDS through the four
// products (24 sites, 2,925 ADOs: 241 us an iteration as a stage launch and four passes, 54 us so).
template <int SZ, bool REALC, bool WLDS, bool LONG>
__global__ __launch_bounds__(kWideThreads) void tss_iteration_wide(StageArgsT<double> a, WideTables<double> wt,
                                                                   WideTss ts, const double2* __restrict__ gam_all,
                                                                   int N, int T)
{
    using C = double2;
    using TM = std::conditional_t<REALC, double, C>;
    constexpr int NB = (SZ + 15) / 16, NL = (SZ * SZ + 63) / 64, NP = wide_pitch(SZ);
    extern __shared__ __align__(16) unsigned char wide_mem[];
    const int nel = N * N;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int words = wt.words;
    constexpr bool GL = kWideGamLds<double, SZ>;
    const WideLds L = wide_lds(N, (int)sizeof(C), REALC, GL, T, WLDS ? words * 4 : 0);
    TM* cl = reinterpret_cast<TM*>(wide_mem);
    C* gl = reinterpret_cast<C*>(wide_mem + L.gam);
    uint32_t* el = reinterpret_cast<uint32_t*>(wide_mem + L.where);
    C* sig = reinterpret_cast<C*>(wide_mem + L.mat) + (int64_t)w * (N * NP);
    int places[(NL + 1) / 2];  // of this lane's elements, two to a register
#pragma unroll
    for (int k = 0; k < NL; ++k) {
        const int at = wt.place[min(lane + 64 * k, nel - 1)];
        places[k / 2] = k & 1 ? places[k / 2] | at << 16 : at;
    }
    auto place = [&](int k) { return k & 1 ? (int)((uint32_t)places[k / 2] >> 16) : places[k / 2] & 0xffff; };
    const double sq_lane = sqrt((double)lane);

    const Walk walk(wt.tile_order, a.ntiles, T);
    int inst = -1, cls = -1;
    for (int j = walk.j;; j += walk.gx) {
        const int64_t q0 = walk.group<false>(j), q = q0 + w;
        if (q0 < 0)
            break;
        const int it = a.tile_inst ? a.tile_inst[q0 / kTile] : 0;
        const int cc = tile_bath_class(a, (int)(q0 / kTile));
        const C* gam = gam_all + (int64_t)cc * nel;
        const uint32_t* where = wt.where + (int64_t)cc * words;
        if (it != inst || cc != cls)
            load_constants<double, TM, SZ, WLDS>(ts.c + (int64_t)it * nel, gam, where, words, N, cl, gl, el, inst < 0);
        inst = it;
        cls = cc;
        if (q >= a.zero_slot)
            continue;
        EdgeLanes ed;
        ed.load(a.nb, a.mp, q, lane, wt.W, a.zero_slot);
        const C S = a.pfss[q], em = ts.epsm[q];
#pragma unroll
        for (int k = 0; k < NL; ++k) {
            const int e = lane + 64 * k;
            if (e < nel) {
                const int at = place(k);
                const C g = GL ? gl[at] : gam[at / NP * N + at % NP], y = a.yin[q * nel + e];
                sig[at] = cfma(mk2<double>(S.x + g.x, S.y + g.y), y, mk2<double>(0.0, 0.0));
            }
        }
        wave_sync();
        Neighbours<double, kWideModesAhead<double, SZ, true>, LONG> nbs(a, wt, cc, WLDS ? el : where, ed, q, nel, lane);
        nbs.start();
        nbs.template run<false>(1.0, sq_lane, sig);
        wave_sync();
        const C* w_ij = ts.w + (int64_t)it * nel;
        auto put = [&](int at, int, int, C v) {
            sig[at] = v;
            return v;
        };
        Product<double, NB> p;
        p.clear();
        multiply<true, false, false, double, NB, NP>(p, sig, cl, N, lane);  // C k
        wave_sync();
        each_element<double, NB, NP>(p, N, lane, put);
        wave_sync();
        // the denominators' part of this lane's elements, all of them under way during the
        // product (one at a time they were a round trip each: 24 sites, 2,925 ADOs 57 -> 54 us
        // an iteration); 32 x 32 matrices spill with them (32 sites, depth 3: 157 us, 161 so)
        constexpr bool kDenAhead = SZ <= 24;
        vec2_t<double> wv[kDenAhead ? NB * NB * 4 : 1];
        if constexpr (kDenAhead) {
#pragma unroll
            for (int t = 0; t < NB * NB * 4; ++t) {
                const int i = min(16 * (t / (4 * NB)) + d_row<double>(lane, t % 4), N - 1);
                const int jj = min(16 * (t / 4 % NB) + (lane & 15), N - 1);
                wv[t] = *reinterpret_cast<const vec2_t<double>*>(w_ij + i * N + jj);
            }
        }
        p.clear();
        multiply<false, true, false, double, NB, NP>(p, sig, cl, N, lane);  // (C k) C^T
        wave_sync();
#pragma unroll
        for (int t = 0; t < NB * NB * 4; ++t) {
            const int ta = t / (4 * NB), tb = t / 4 % NB, i = 16 * ta + d_row<double>(lane, t % 4), jj = 16 * tb + (lane & 15);
            const C v = mk2<double>(p.re[ta][tb][t % 4], p.im[ta][tb][t % 4]);
            if (i < N && jj < N) {
                const C wij = kDenAhead ? mk2<double>(wv[kDenAhead ? t : 0].x, wv[kDenAhead ? t : 0].y) : w_ij[i * N + jj];
                const C d = mk2<double>(wij.x + em.x, wij.y + em.y);
                const double den = d.x * d.x + d.y * d.y;
                sig[i * NP + jj] = mk2<double>((v.x * d.x + v.y * d.y) / den, (v.y * d.x - v.x * d.y) / den);
            }
        }
        wave_sync();
        p.clear();
        multiply<true, true, false, double, NB, NP>(p, sig, cl, N, lane);  // C^T B
        wave_sync();
        each_element<double, NB, NP>(p, N, lane, put);
        wave_sync();
        p.clear();
        multiply<false, false, false, double, NB, NP>(p, sig, cl, N, lane);  // (C^T B) C
        wave_sync();
        each_element<double, NB, NP>(p, N, lane, put);
        wave_sync();
        const bool pad = ts.q2u[q] < 0;
#pragma unroll
        for (int k = 0; k < NL; ++k) {
            const int e = lane + 64 * k;
            if (e < nel)
                nt_store<double>(pad ? mk2<double>(0.0, 0.0) : sig[place(k)], a.yout + q * nel + e);
        }
        wave_sync();
    }
}

// How a launch is divided: T wavefronts per workgroup (`ados` where a caller chose), and a
// workgroup per group of T ADOs where all of them fit the card at once (`one`; the tiles are
// dealt to the XCDs whole, so the XCD with the most tiles sets the number), or as many as run
// at once.
struct WideShape {
    int T;
    bool one;
    unsigned wgs;
};
template <typename R, int SZ>
constexpr WideShape wide_shape(int N, bool real, int words, int ntiles, int ados)
{
    const auto shape = [&](int T) {
        const int64_t all = (int64_t)(ntiles + kNumXcd - 1) / kNumXcd * kNumXcd * (kTile / T);
        const int64_t most = (int64_t)kWideCus * 4 * kWideOccupancy<R, SZ> / T;
        return WideShape{T, all <= most, (unsigned)std::min(all, most)};
    };
    const int fit = wide_most_waves(N, (int)sizeof(c2<R>), real, words);
    if (ados > 0 && ados <= fit && kTile % ados == 0)
        return shape(ados);
    // 4, as many as a CU's SIMDs; 8 where the CU's LDS does not hold two such workgroups and
    // each wavefront has several ADOs to go through (32 sites, ms per RK4 step in complex128:
    // 6,545 ADOs 0.640 with 4, 0.582 with 8; 561 ADOs 0.101 and 0.133)
    const WideShape four = shape(std::min(fit, 4));
    const int lds = wide_lds(N, (int)sizeof(c2<R>), real, kWideGamLds<R, SZ>, 4, wide_where_bytes(words)).total;
    return !four.one && 2 * lds > kWideLdsAll && fit >= 8 ? shape(8) : four;
}

template <typename R, int SZ, bool REALH, bool ONE, bool WLDS, bool LONG, bool BYEL>
void launch_wl(int N, int stage, const StageArgsT<R>& a, const ElementArgsT<R>& el, const WideTables<R>& wt,
               WideShape sh, hipStream_t st)
{
    const int T = sh.T;
    const dim3 grid(sh.wgs), block(64 * T);
    const size_t lds =
        (size_t)wide_lds(N, (int)sizeof(c2<R>), REALH, kWideGamLds<R, SZ>, T, wide_where_bytes(wt.words)).total;
    switch (stage) {
    case 0: hipLaunchKernelGGL((rk4_stage_wide<R, SZ, 0, REALH, ONE, WLDS, LONG, BYEL>), grid, block, lds, st, a, wt, el.hs, el.gam, N, T); break;
    case 1: hipLaunchKernelGGL((rk4_stage_wide<R, SZ, 1, REALH, ONE, WLDS, LONG, BYEL>), grid, block, lds, st, a, wt, el.hs, el.gam, N, T); break;
    case 2: hipLaunchKernelGGL((rk4_stage_wide<R, SZ, 2, REALH, ONE, WLDS, LONG, BYEL>), grid, block, lds, st, a, wt, el.hs, el.gam, N, T); break;
    case 3: hipLaunchKernelGGL((rk4_stage_wide<R, SZ, 3, REALH, ONE, WLDS, LONG, BYEL>), grid, block, lds, st, a, wt, el.hs, el.gam, N, T); break;
    default: hipLaunchKernelGGL((rk4_stage_wide<R, SZ, 4, REALH, ONE, WLDS, LONG, BYEL>), grid, block, lds, st, a, wt, el.hs, el.gam, N, T); break;
    }
}

// lists of unequal rounds (WideTables: stride = 0) have kernels of their own: as a branch or
// selects in the others' they cost these 1 to 2%
template <typename R, int SZ, bool REALH, bool ONE, bool WLDS, bool BYEL>
void launch_wo(int N, int stage, const StageArgsT<R>& a, const ElementArgsT<R>& el, const WideTables<R>& wt,
               WideShape sh, hipStream_t st)
{
    if (wt.stride == 0)
        launch_wl<R, SZ, REALH, ONE, WLDS, true, BYEL>(N, stage, a, el, wt, sh, st);
    else
        launch_wl<R, SZ, REALH, ONE, WLDS, false, BYEL>(N, stage, a, el, wt, sh, st);
}

template <typename R, int SZ, bool REALH>
void launch_ws(int N, int stage, const StageArgsT<R>& a, const ElementArgsT<R>& el, const WideTables<R>& wt, int ados,
               hipStream_t st)
{
    const WideShape sh = wide_shape<R, SZ>(N, REALH, wt.words, a.ntiles, ados);
    if (wide_where_bytes(wt.words) == 0) {
        launch_wo<R, SZ, REALH, false, false, false>(N, stage, a, el, wt, sh, st);
    } else if (!sh.one) {
        launch_wo<R, SZ, REALH, false, true, false>(N, stage, a, el, wt, sh, st);
    } else if constexpr (SZ <= kWideListStates) {
        // two, three or four elements to a lane (12 sites, 1,820 ADOs in complex128: 0.0356 ms
        // per RK4 step with three, 0.0392 with four)
        const int NL = N <= 11 ? 2 : N <= 13 ? 3 : 4;
        if (wt.stride > 0 && (wt.W > 64 || !by_element(wt.W * ((wt.stride + 63) / 64), NL, wt.slots)))
            launch_wl<R, SZ, REALH, true, true, false, false>(N, stage, a, el, wt, sh, st);
        else if (NL == 2)
            launch_wo<R, 11, REALH, true, true, true>(N, stage, a, el, wt, sh, st);
        else if (NL == 3)
            launch_wo<R, 13, REALH, true, true, true>(N, stage, a, el, wt, sh, st);
        else
            launch_wo<R, SZ, REALH, true, true, true>(N, stage, a, el, wt, sh, st);
    } else {
        launch_wo<R, SZ, REALH, true, true, false>(N, stage, a, el, wt, sh, st);
    }
}

template <typename R, bool REALH>
void launch_w(int N, int stage, const StageArgsT<R>& a, const ElementArgsT<R>& el, const WideTables<R>& wt, int ados,
              hipStream_t st)
{
    if (N <= 16)
        launch_ws<R, 16, REALH>(N, stage, a, el, wt, ados, st);
    else if (N <= 24)
        launch_ws<R, 24, REALH>(N, stage, a, el, wt, ados, st);
    else
        launch_ws<R, 32, REALH>(N, stage, a, el, wt, ados, st);
}

template <int SZ, bool REALC>
void launch_tr(int N, const StageArgsT<double>& a, const double2* gam, const WideTables<double>& wt, const WideTss& ts,
               hipStream_t st)
{
    const WideShape sh = wide_shape<double, SZ>(N, REALC, wt.words, a.ntiles, 0);
    const int wb = wide_where_bytes(wt.words), T = sh.T;
    const size_t lds = (size_t)wide_lds(N, (int)sizeof(double2), REALC, kWideGamLds<double, SZ>, T, wb).total;
    const dim3 grid(sh.wgs), block(64 * T);
    if (wb && wt.stride == 0)
        hipLaunchKernelGGL((tss_iteration_wide<SZ, REALC, true, true>), grid, block, lds, st, a, wt, ts, gam, N, T);
    else if (wb)
        hipLaunchKernelGGL((tss_iteration_wide<SZ, REALC, true, false>), grid, block, lds, st, a, wt, ts, gam, N, T);
    else if (wt.stride == 0)
        hipLaunchKernelGGL((tss_iteration_wide<SZ, REALC, false, true>), grid, block, lds, st, a, wt, ts, gam, N, T);
    else
        hipLaunchKernelGGL((tss_iteration_wide<SZ, REALC, false, false>), grid, block, lds, st, a, wt, ts, gam, N, T);
}

template <int SZ>
void launch_ts(int N, bool real_c, const StageArgsT<double>& a, const double2* gam, const WideTables<double>& wt,
               const WideTss& ts, hipStream_t st)
{
    if (real_c)
        launch_tr<SZ, true>(N, a, gam, wt, ts, st);
    else
        launch_tr<SZ, false>(N, a, gam, wt, ts, st);
}

}  // namespace

// the limit on the modes of a handle: two matrices and a table entry per mode in 144 KB
bool wide_supported(int N, int complex_bytes, int W)
{
    return N > kMaxStates && N <= kMaxWideStates &&
           2 * (int64_t)N * (N + 1) * complex_bytes + (((int64_t)W + 2) & ~1) * 8 <= 147456;
}

int wide_max_ados(int N, int complex_bytes, bool real_h, int words)
{
    return wide_most_waves(N, complex_bytes, real_h, words);
}

void launch_stage_wide(int N, bool real_h, int stage, const StageArgsT<double>& a, const ElementArgsT<double>& el,
                       const WideTables<double>& wt, int ados, hipStream_t s)
{
    if (real_h)
        launch_w<double, true>(N, stage, a, el, wt, ados, s);
    else
        launch_w<double, false>(N, stage, a, el, wt, ados, s);
}

void launch_stage_wide(int N, bool real_h, int stage, const StageArgsT<float>& a, const ElementArgsT<float>& el,
                       const WideTables<float>& wt, int ados, hipStream_t s)
{
    if (real_h)
        launch_w<float, true>(N, stage, a, el, wt, ados, s);
    else
        launch_w<float, false>(N, stage, a, el, wt, ados, s);
}

void launch_tss_wide(int N, bool real_c, const StageArgsT<double>& a, const double2* gam, const WideTables<double>& wt,
                     const WideTss& ts, hipStream_t s)
{
    if (N <= 16)
        launch_ts<16>(N, real_c, a, gam, wt, ts, s);
    else if (N <= 24)
        launch_ts<24>(N, real_c, a, gam, wt, ts, s);
    else
        launch_ts<32>(N, real_c, a, gam, wt, ts, s);
}

}  // namespace heom_hip
