// tss.hip -- the thermal state search (heom_create_tss / heom_tss_step of include/heom_hip.h),
// after dm-heom/include/heom/thermal_state_search_solver.hpp:124-300 and
// dm-heom/cl/heom/thermal_state_search.cl:10-52.
//
// One iteration of the search maps the hierarchy y to
//   k   = f_TSS(y)                   the HEOM RHS with the commutator replaced by the
//                                    elementwise product with a pseudo-Hamiltonian that
//                                    holds eps in every element, and without the S_u term
//                                    (heom_ode.cl:116-121, 130-136), i.e. eps y + the rest
//   y_u = C^T [ (C k_u C^T) / D_u ] C    D_u(i, j) = i (E_i - E_j) / hbar + eps - S_u
// with C the transposed eigenvectors of H and E its eigenvalues; a fixed point solves
// L y = 0, the stationary (thermal) hierarchy.
//
// k needs no kernel of its own: eps y is the S_u y term of the ordinary RHS with S_u = eps
// for every ADO and H = 0, so a search handle is an ordinary handle built from such a
// descriptor, whose stage kernels (STAGE 0, one evaluation) compute f_TSS unchanged for
// heom_rhs.  An iteration is one kernel that leaves out the commutator of H = 0 and keeps k
// and the four products on the CU: here for N <= 8 (a tile of 64 ADOs in LDS), in
// stage_wide.hip for 8 < N <= 32 (a matrix per wavefront).  It reads the state and writes the
// next one into the work buffer; the two then exchange their places.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <functional>
#include <type_traits>
#include <vector>

#include "handle.hpp"
#include "heom_device.hpp"
#include "heom_hip.h"

using namespace heom_hip;
using namespace heom_rt;

namespace {

__device__ __forceinline__ double2 cdiv(double2 a, double2 d)  // a / d
{
    const double den = d.x * d.x + d.y * d.y;
    return make_double2((a.x * d.x + a.y * d.y) / den, (a.y * d.x - a.x * d.y) / den);
}

// One iteration's arguments: the state and the result (planes), the ordinary tables of a
// handle (neighbour table, pf_same_sum = eps, tile flags, instance and bath class), and
// epsm[q] = eps - S_u of the ADO in slot q (eps in unused slots, which are written as zero).
// The constants with wave-uniform indices (C, C^T, w[i*N+j] = (i/hbar)(E_i - E_j) per
// instance; gam and terms per class) are kernel arguments of their own, read with scalar
// loads.
struct TssArgs {
    const double2* __restrict__ y;
    double2* __restrict__ out;
    const int2* __restrict__ nb;
    const double2* __restrict__ pfss;
    const double2* __restrict__ epsm;
    const int32_t* __restrict__ q2u;        // < 0: padding or the zero slot, kept at zero
    const int32_t* __restrict__ tile_inst;  // instance of each tile (null: one instance)
    const int32_t* __restrict__ tile_plus;
    const int32_t* __restrict__ tile_class;  // bath class of each tile (null: one class)
    int64_t mp;
    int32_t ntiles, zero_slot, xcd_chunk;
};

// c * x (+ acc): C's entries are real for a real symmetric H (two multiplies per product
// instead of four, and half the scalar loads), complex otherwise
__device__ __forceinline__ double2 cmac(double c, double2 x, double2 acc)
{
    return make_double2(fma(c, x.x, acc.x), fma(c, x.y, acc.y));
}
__device__ __forceinline__ double2 cmac(double2 c, double2 x, double2 acc) { return cfma(c, x, acc); }

// One iteration for the 64 ADOs of a tile (lane = ADO), one wavefront per column, then per
// row, of the matrices.  Wavefront j evaluates column j of k = f_TSS(y) -- the "same" term
// and the neighbour terms, no commutator -- and, holding the column in registers, column j
// of C k.  The tile goes through LDS; wavefront i takes row i of C k, multiplies by C^T,
// divides by D and multiplies by C, all within the row; the tile goes through LDS once
// more (each wavefront overwrites the row that only it has read), and wavefront j stores
// column j of C^T (B C).  So k and the products between never leave the CU, and the four
// products cost two tile writes and two tile reads of LDS instead of a read of the whole
// tile per matrix row for each left product.
template <int N, int NT, typename TC, bool PLUS>
__device__ __forceinline__ void tss_tile(const TssArgs& a, const double2* __restrict__ gam,
                                         const Term* __restrict__ terms, const int32_t* __restrict__ modes,
                                         const TC* __restrict__ C, const TC* __restrict__ CT,
                                         const double2* __restrict__ Wd, int tile, double2* t)
{
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t mp = a.mp;
    const int64_t q = (int64_t)tile * kTile + lane;
    const double2 S = a.pfss[q];
    const double sq_lane = sqrt((double)lane);  // sqrt(n), n = 0..63, one value per lane
    // gathers as raw buffer loads, one resource per element plane whose range ends at the
    // zero slot: an edge to it returns zero without a memory request
    const int nrec = a.zero_slot * (int)sizeof(double2);
    auto gather = [&](__amdgpu_buffer_rsrc_t rsrc, uint32_t idx) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, idx * (uint32_t)sizeof(double2), 0, 0);
        return make_double2(__hiloint2double((int)v[1], (int)v[0]), __hiloint2double((int)v[3], (int)v[2]));
    };
    // offsets the compiler cannot see through keep the (scalar, cached) loads of the
    // uniform constants next to the row or column that uses them: hoisted together they
    // would need several times the scalar registers
    auto opaque = [](const auto* p) {
        int z;
        asm volatile("s_mov_b32 %0, 0" : "=s"(z));
        return p + z;
    };
    // the wavefront's constants are contiguous (column-major elements)
    gam += w * N;
    terms += w * N * NT;
    modes += w * N * NT;
    // The table entries of a batch of elements are requested together, and where the
    // registers allow (two workgroups of 8 wavefronts per CU: 128) an element's gathers and
    // own value go out before the previous element's are summed.
    constexpr bool AHEAD = NT * (PLUS ? 2 : 1) <= 4;
    constexpr int HB = NT <= 2 ? N : NT <= 4 ? (N + 1) / 2 : 1;
    double2 r[N];
#pragma unroll
    for (int i0 = 0; i0 < N; i0 += HB) {  // r = column w of k
        int2 nbv[HB][NT];
#pragma unroll
        for (int i = i0; i < i0 + HB && i < N; ++i)
#pragma unroll
            for (int k = 0; k < NT; ++k)
                nbv[i - i0][k] = a.nb[(int64_t)modes[i * NT + k] * mp + q];
        double2 xp[AHEAD ? 2 : 1][NT], xm[AHEAD ? 2 : 1][NT], own[AHEAD ? 2 : 1];
        auto load = [&](int i, int b) {
            const double2* plane = a.y + (int64_t)(i * N + w) * mp;
            const __amdgpu_buffer_rsrc_t rsrc =
                __builtin_amdgcn_make_buffer_rsrc((void*)plane, (short)0, nrec, 0x00020000);
            own[b] = plane[q];
#pragma unroll
            for (int k = 0; k < NT; ++k) {
                if constexpr (PLUS)
                    xp[b][k] = gather(rsrc, (uint32_t)nbv[i - i0][k].x >> 6);
                xm[b][k] = gather(rsrc, (uint32_t)nbv[i - i0][k].y);
            }
        };
        if (AHEAD)
            load(i0, 0);
#pragma unroll
        for (int i = i0; i < i0 + HB && i < N; ++i) {
            const int b = AHEAD ? (i - i0) & 1 : 0;
            __builtin_amdgcn_sched_barrier(0);
            if (!AHEAD)
                load(i, 0);
            else if (i + 1 < i0 + HB && i + 1 < N)
                load(i + 1, 1 - b);
            const Term* te = opaque(terms) + i * NT;
            const double2 g = opaque(gam)[i];
            double2 f = cfma(make_double2(S.x + g.x, S.y + g.y), own[b], make_double2(0.0, 0.0));
#pragma unroll
            for (int k = 0; k < NT; ++k) {
                const int v = nbv[i - i0][k].x & 63;
                if constexpr (PLUS) {
                    const double cp = te[k].plus_c * lane_value(sq_lane, v + 1);
                    f.x = fma(-cp, xp[b][k].y, f.x);
                    f.y = fma(cp, xp[b][k].x, f.y);
                }
                const double sm = lane_value(sq_lane, v);
                f = cfma(te[k].minus_c, make_double2(sm * xm[b][k].x, sm * xm[b][k].y), f);
            }
            // the sum is formed here, before the next element's gathers replace this one's
            asm volatile("" : "+v"(f.x), "+v"(f.y));
            r[i] = f;
        }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {  // column w of C k
        const TC* Ci = opaque(C) + i * N;
        double2 v = make_double2(0.0, 0.0);
#pragma unroll
        for (int m = 0; m < N; ++m)
            v = cmac(Ci[m], r[m], v);
        t[(i * N + w) * kTile + lane] = v;
    }
    const double2 em = a.epsm[q];
    const bool pad = a.q2u[q] < 0;
    __syncthreads();
    double2 s[N];
#pragma unroll
    for (int m = 0; m < N; ++m)
        r[m] = t[(w * N + m) * kTile + lane];
#pragma unroll
    for (int j = 0; j < N; ++j) {  // s = row w of (C k C^T) / D
        const TC* Cj = opaque(C) + j * N;
        double2 v = make_double2(0.0, 0.0);
#pragma unroll
        for (int m = 0; m < N; ++m)
            v = cmac(Cj[m], r[m], v);  // CT[m][j]
        const double2 wij = Wd[w * N + j];
        s[j] = cdiv(v, make_double2(wij.x + em.x, wij.y + em.y));
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {  // row w of B C
        const TC* CTj = opaque(CT) + j * N;
        double2 v = make_double2(0.0, 0.0);
#pragma unroll
        for (int m = 0; m < N; ++m)
            v = cmac(CTj[m], s[m], v);  // C[m][j]
        t[(w * N + j) * kTile + lane] = v;
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < N; ++m)
        r[m] = t[(m * N + w) * kTile + lane];
#pragma unroll
    for (int i = 0; i < N; ++i) {  // column w of C^T (B C)
        const TC* CTi = opaque(CT) + i * N;
        double2 v = make_double2(0.0, 0.0);
#pragma unroll
        for (int m = 0; m < N; ++m)
            v = cmac(CTi[m], r[m], v);
        nt_store<double>(pad ? make_double2(0.0, 0.0) : v, a.out + (int64_t)(i * N + w) * mp + q);
    }
}

template <int N, int NT, typename TC>
__global__ __launch_bounds__(64 * N) void tss_iteration(TssArgs a, const double2* __restrict__ gam,
                                                        const Term* __restrict__ terms,
                                                        const int32_t* __restrict__ modes, const TC* __restrict__ c,
                                                        const TC* __restrict__ ct, const double2* __restrict__ wd)
{
    __shared__ double2 t[N * N * kTile];
    const int tile = xcd_tile(blockIdx.x, a.ntiles, a.xcd_chunk);
    const int64_t off = a.tile_inst ? (int64_t)a.tile_inst[tile] * N * N : 0;
    const int cls = a.tile_class ? a.tile_class[tile] : 0;
    gam += cls * (N * N);
    terms += cls * (N * N * NT);
    modes += cls * (N * N * NT);
    if (a.tile_plus[tile] != 0)
        tss_tile<N, NT, TC, true>(a, gam, terms, modes, c + off, ct + off, wd + off, tile, t);
    else
        tss_tile<N, NT, TC, false>(a, gam, terms, modes, c + off, ct + off, wd + off, tile, t);
}

template <int N, int NT>
void launch_iteration_t(heom_handle* h, const TssArgs& a)
{
    const TssState& T = *h->tss;
    const dim3 grid(h->ntiles), block(64 * N);
    if (T.real_c)
        hipLaunchKernelGGL((tss_iteration<N, NT, double>), grid, block, 0, h->stream, a, T.gam, T.terms, T.modes, T.cr,
                           T.ctr, T.w);
    else
        hipLaunchKernelGGL((tss_iteration<N, NT, double2>), grid, block, 0, h->stream, a, T.gam, T.terms, T.modes,
                           T.c, T.ct, T.w);
}

template <int N>
void launch_iteration(heom_handle* h, const TssArgs& a)
{
    switch (h->term_slots) {
    case 2: launch_iteration_t<N, 2>(h, a); break;
    case 4: launch_iteration_t<N, 4>(h, a); break;
    default: launch_iteration_t<N, 8>(h, a); break;
    }
}

void check_tss(heom_handle* h)
{
    if (!h->tss)
        raise(HEOM_E_INVALID, "not a thermal-state-search handle (heom_create_tss)");
}

}  // namespace

namespace heom_rt {

void reject_tss(heom_handle* h, const char* what)
{
    if (h->tss)
        raise(HEOM_E_UNSUPPORTED, std::string(what) + " is not available on a thermal-state-search handle");
}

}  // namespace heom_rt

extern "C" {

int heom_create_tss_batch(const heom_desc* descs, int32_t count, const double* c, const double* eigenvalues,
                          const double* epsilon, heom_handle** out)
{
    if (!out) {
        g_error = "out is NULL";
        return HEOM_E_INVALID;
    }
    *out = nullptr;
    heom_handle* h = nullptr;
    const int rc = guard([&] {
        if (!descs || !c || !eigenvalues || !epsilon)
            raise(HEOM_E_INVALID, "descs, c, eigenvalues and epsilon must not be NULL");
        if (count < 1)
            raise(HEOM_E_INVALID, "count must be >= 1");
        const int N = descs[0].states;
        if (N < 1)
            raise(HEOM_E_INVALID, "states must be >= 1");
        if (N > 32)
            raise(HEOM_E_UNSUPPORTED, "more than 32 states");
        for (int k = 0; k < count; ++k) {
            if (descs[k].precision != HEOM_PRECISION_FP64)
                raise(HEOM_E_UNSUPPORTED, "the thermal state search runs in FP64 only");
            if (descs[k].states != N || descs[k].matrices < 1)
                raise(HEOM_E_INVALID, "every instance needs the same states and matrices >= 1");
            // read below for eps - S_u; the descriptor handed on carries replacements
            if (!descs[k].pf_same_sum)
                raise(HEOM_E_INVALID, "desc has a NULL array (pf_same_sum)");
        }
        const std::complex<double> eps(epsilon[0], epsilon[1]);
        if (!std::isfinite(eps.real()) || !std::isfinite(eps.imag()) || eps == 0.0)
            raise(HEOM_E_INVALID, "epsilon must be finite and non-zero");
        const int nel = N * N;
        for (int64_t e = 0; e < (int64_t)count * 2 * nel; ++e)
            if (!std::isfinite(c[e]))
                raise(HEOM_E_INVALID, "c must be finite");
        for (int64_t e = 0; e < (int64_t)count * 2 * N; ++e)
            if (!std::isfinite(eigenvalues[e]))
                raise(HEOM_E_INVALID, "eigenvalues must be finite");
        // the f_TSS operator: H = 0 and S_u = eps (thermal_state_search_solver.hpp:199-209,
        // the pseudo-Hamiltonian eps in every element through heom_ode.cl:116-121)
        std::vector<heom_desc> d(descs, descs + count);
        const std::vector<double> zero_h((size_t)(2 * nel), 0.0);
        std::vector<std::vector<double>> pss((size_t)count);
        for (int k = 0; k < count; ++k) {
            pss[(size_t)k].resize((size_t)(2 * d[(size_t)k].matrices));
            for (int64_t u = 0; u < d[(size_t)k].matrices; ++u) {
                pss[(size_t)k][(size_t)(2 * u)] = eps.real();
                pss[(size_t)k][(size_t)(2 * u + 1)] = eps.imag();
            }
            d[(size_t)k].hamiltonian = zero_h.data();
            d[(size_t)k].pf_same_sum = pss[(size_t)k].data();
        }
        h = new heom_handle();
        HostTables host;
        create_batch(h, d.data(), count, &host);
        auto T = std::make_unique<TssState>();
        std::vector<double2> cv((size_t)count * nel), ctv((size_t)count * nel), wv((size_t)count * nel);
        for (int k = 0; k < count; ++k) {
            const double* ck = c + (size_t)k * 2 * nel;
            const double* ek = eigenvalues + (size_t)k * 2 * N;
            double2* cvk = &cv[(size_t)k * nel];
            double2* ctk = &ctv[(size_t)k * nel];
            double2* wk = &wv[(size_t)k * nel];
            for (int i = 0; i < N; ++i)
                for (int j = 0; j < N; ++j) {
                    cvk[i * N + j] = make_double2(ck[2 * (i * N + j)], ck[2 * (i * N + j) + 1]);
                    ctk[i * N + j] = make_double2(ck[2 * (j * N + i)], ck[2 * (j * N + i) + 1]);
                    // (i / hbar)(E_i - E_j) as thermal_state_search.cl:45 forms it
                    const double der = ek[2 * i] - ek[2 * j];
                    const double dei = ek[2 * i + 1] - ek[2 * j + 1];
                    wk[i * N + j] = make_double2(-dei / kHbar, der / kHbar);
                }
        }
        // eps - S_u per slot, in the handle's ADO order (q2u holds batch-global uids)
        std::vector<double2> em((size_t)h->Mp, make_double2(eps.real(), eps.imag()));
        for (int64_t q = 0; q < h->Mp; ++q) {
            const int32_t u = host.q2u[(size_t)q];
            if (u < 0)
                continue;
            const int k = (int)(std::upper_bound(h->inst_u.begin(), h->inst_u.end(), (int64_t)u) - h->inst_u.begin()) - 1;
            const int64_t lu = u - h->inst_u[(size_t)k];
            em[(size_t)q] = make_double2(eps.real() - descs[k].pf_same_sum[2 * lu],
                                         eps.imag() - descs[k].pf_same_sum[2 * lu + 1]);
        }
        T->real_c = true;
        for (const double2& x : cv)
            T->real_c = T->real_c && x.y == 0.0;
        // one allocation and one copy for what the iteration's kernel reads
        std::vector<unsigned char> mem;
        std::vector<std::function<void()>> places;
        auto add = [&](auto& place, const auto& v) {
            const size_t at = (mem.size() + 15) / 16 * 16, bytes = v.size() * sizeof(v[0]);
            mem.resize(at + bytes);
            std::memcpy(mem.data() + at, v.data(), bytes);
            places.push_back([&place, at, t = T.get()] {
                place = reinterpret_cast<std::decay_t<decltype(place)>>(t->mem.p + at);
            });
        };
        add(T->w, wv);
        add(T->epsm, em);
        if (N > kMaxStates || !T->real_c)
            add(T->c, cv);
        if (N <= kMaxStates) {
            if (T->real_c) {
                std::vector<double> cr(cv.size()), ctr(cv.size());
                for (size_t e = 0; e < cv.size(); ++e) {
                    cr[e] = cv[e].x;
                    ctr[e] = ctv[e].x;
                }
                add(T->cr, cr);
                add(T->ctr, ctr);
            } else {
                add(T->ct, ctv);
            }
            // the element constants in column-major order (a wavefront of the iteration kernel
            // evaluates one column)
            const int NT = h->term_slots, classes = (int)h->classes.size();
            std::vector<double2> gam(host.gam.size());
            std::vector<Term> terms(host.terms.size());
            std::vector<int32_t> modes(terms.size());
            for (int cl = 0; cl < classes; ++cl)
                for (int i = 0; i < N; ++i)
                    for (int j = 0; j < N; ++j) {
                        const size_t from = (size_t)cl * nel + i * N + j, to = (size_t)cl * nel + j * N + i;
                        gam[to] = host.gam[from];
                        for (int k = 0; k < NT; ++k) {
                            terms[to * NT + k] = host.terms[from * NT + k];
                            modes[to * NT + k] = host.terms[from * NT + k].mode;
                        }
                    }
            add(T->gam, gam);
            add(T->terms, terms);
            add(T->modes, modes);
        }
        T->mem.alloc(mem.size());
        HIPC(hipMemcpyAsync(T->mem.p, mem.data(), mem.size(), hipMemcpyHostToDevice, h->stream));
        for (const auto& place : places)
            place();
        HIPC(hipStreamSynchronize(h->stream));
        h->tss = std::move(T);
    });
    if (rc != HEOM_OK) {
        delete h;
        return rc;
    }
    *out = h;
    return HEOM_OK;
}

int heom_create_tss(const heom_desc* desc, const double* c, const double* eigenvalues, const double* epsilon,
                    heom_handle** out)
{
    return heom_create_tss_batch(desc, 1, c, eigenvalues, epsilon, out);
}

int heom_tss_step(heom_handle* h, int64_t n)
{
    return guard([&] {
        need(h);
        check_tss(h);
        if (n < 0)
            raise(HEOM_E_INVALID, "n must be >= 0");
        const TssState& T = *h->tss;
        const int N = h->N;
        const int32_t* ti = h->count > 1 ? h->tile_inst.p : nullptr;
        for (int64_t s = 0; s < n; ++s) {
            if (N <= kMaxStates) {
                // y -> ya, then the two exchange their places
                const TssArgs a{h->y.as<double2>(), h->ya.as<double2>(), h->nb.p, h->pfss.p, T.epsm, h->q2u.p, ti,
                                h->tile_plus.p, h->uniform ? nullptr : h->tile_class.p, h->Mp, h->ntiles,
                                h->zero_slot, h->xcd_chunk};
                switch (N) {
                case 1: launch_iteration<1>(h, a); break;
                case 2: launch_iteration<2>(h, a); break;
                case 3: launch_iteration<3>(h, a); break;
                case 4: launch_iteration<4>(h, a); break;
                case 5: launch_iteration<5>(h, a); break;
                case 6: launch_iteration<6>(h, a); break;
                case 7: launch_iteration<7>(h, a); break;
                default: launch_iteration<8>(h, a); break;
                }
                HIPC(hipGetLastError());
                std::swap(h->y.p, h->ya.p);
                h->timing.rhs_launches += 1;
                continue;
            }
            const StageArgsT<double> a = stage_args64(h, h->y.p, h->y.p, h->pbuf.p, h->ya.p, 0.0, false);
            launch_tss_wide(N, T.real_c, a, h->gam.p, h->wide_tables<double>(),
                            WideTss{T.c, T.w, T.epsm, h->q2u.p}, h->stream);
            HIPC(hipGetLastError());
            std::swap(h->y.p, h->ya.p);
            h->timing.rhs_launches += 1;
        }
    });
}

}  // extern "C"
