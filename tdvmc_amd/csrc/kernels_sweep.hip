// Persistent Metropolis sweeps: every walker performs n_moves single-particle
// trial moves inside one launch (a sweep is N moves).
//
// Restates the move of src/TDVMC.cpp:858-916 (DoMetropolisStep: random
// particle, Gaussian displacement of width MC_STEP in every component, accept
// with probability min(1, |psi_new / psi_old|^2), restore on reject) with the
// incremental ratio of src/PhysicalSystems/BosonsBulk.cpp:553-657
// (CalculateWFChange: old and new pair terms of the moved particle, pairs
// beyond the cutoff contribute the last pair parameter), plus the k-space
// term (incremental rho_k update, one representative per +-k pair with the
// summed amplitude) and the one-body factor.
//
// Mapping: a walker is a group of LPW lanes (LPW = 16, 32 or 64) inside a
// wavefront; a 256-thread workgroup holds 256/LPW walkers.  The walker's
// coordinates live in LDS (structure of arrays) for the whole launch; lane g
// of the group handles partners i = g, g + LPW, ... and k-vectors
// k = g + m LPW (their rho_k stay in that lane's registers).  The change of
// ln|psi| is summed with DPP row steps whose result is bitwise identical in
// every lane of the group, so all lanes take the same accept decision without
// further communication.  Random numbers come from Philox4x32-10 (counter =
// trial, call epoch, walker): each lane draws the numbers of one future
// trial, and trial t of a batch reads them from lane t (v_readlane when the
// group is the whole wavefront).  The pair terms are branch-free.  In a
// periodic box the coordinates are held in box units (x / L): as 32-bit
// fractions of the box in the FP32 form (the wrapping integer difference is
// the minimum image), as d - rint(d) in FP64; the phase in revolutions is
// n . s, and the spline table runs out to the largest minimum-image distance
// with the outer-pair value past the cutoff.

#include "common.hpp"
#include "kernels.hpp"
#include "sweep_rules.hpp"

namespace tdvmc {

namespace {

constexpr int kThreads = kSweepThreads;

template <typename T>
struct Vec4 { T x, y, z, w; };
template <typename T>
struct alignas(2 * sizeof(T)) Vec2 { T x, y; };

template <int LPW, typename T>
__device__ __forceinline__ T bcast(T v, int src)
{
    if (LPW == 64) return readlane_f(v, src);
    return __shfl(v, src, LPW);
}
template <int LPW>
__device__ __forceinline__ int bcast_i(int v, int src)
{
    if (LPW == 64) return readlane_i(v, src);
    return __shfl(v, src, LPW);
}
template <int LPW>
__device__ __forceinline__ uint32_t bcast(uint32_t v, int src)
{
    return (uint32_t)bcast_i<LPW>((int)v, src);
}

// Metropolis decision 2 (sum over the group of d - us) >= lu, the same in
// every lane of each aligned group of LPW lanes.  Groups of at most 16 lanes
// sum within their row (every lane gets the same bits).  Wider groups add the
// row sums with row broadcasts: rows 1 and 3 receive r0 + r1 and r2 + r3
// (LPW = 32), row 3 then r0 + r1 + r2 + r3 (LPW = 64); the last lane of the
// group decides and a ballot hands its decision to the group.
constexpr int kDppRowBcast15 = 0x142;   // row r + 1 <- lane 15 of row r
constexpr int kDppRowBcast31 = 0x143;   // rows 2, 3 <- lane 31
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_rows(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xF, false));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_rows(double v)
{
    const int2 x = *reinterpret_cast<int2*>(&v);
    int2 y;
    y.x = __builtin_amdgcn_update_dpp(0, x.x, CTRL, ROWS, 0xF, false);
    y.y = __builtin_amdgcn_update_dpp(0, x.y, CTRL, ROWS, 0xF, false);
    return *reinterpret_cast<double*>(&y);
}
template <int LPW, typename T>
__device__ __forceinline__ bool group_accept(T d, T us, T lu)
{
    if constexpr (LPW <= 16) {
        return (T)2 * (group_sum<LPW>(d) - us) >= lu;
    } else {
        d = group_sum<16>(d);
        d += dpp_rows<kDppRowBcast15, 0xA>(d);
        if constexpr (LPW == 64) d += dpp_rows<kDppRowBcast31, 0x8>(d);
        const uint64_t m = __builtin_amdgcn_ballot_w64((T)2 * (d - us) >= lu);
        if constexpr (LPW == 64) return (m >> 63) & 1;
        return ((threadIdx.x & 63) < 32 ? (m >> 31) : (m >> 63)) & 1;
    }
}

// u(r) from the spline table.  Periodic box: the table extends over every
// possible minimum-image distance, entries past the cutoff hold the
// outer-pair value, so the lookup needs no clamp or select.  Open space:
// clamp to the last interval and select the outer value past the cutoff.
template <typename T, bool PER>
__device__ __forceinline__ T pair_u(T r, T rc, T hinv, int Ps, const Vec4<T>* spl, T u_out)
{
    const T x = r * hinv;
    if (PER) {
        const int j = (int)x;
        const T t = Prec<T>::fract_(x);
        const Vec4<T> cf = spl[j];
        return cf.x + t * (cf.y + t * (cf.z + t * cf.w));
    }
    int j = (int)x;
    j = j > Ps - 2 ? Ps - 2 : j;
    const T t = x - (T)j;
    const Vec4<T> cf = spl[j];
    const T u = cf.x + t * (cf.y + t * (cf.z + t * cf.w));
    return r <= rc ? u : u_out;
}

// u(r) on non-uniform knots (periodic box): cell c = min((int)(r cin), ncell-1)
// (rows past the P_s interval rows) gives the interval (j, or j + 1 past the cell's knot b) and its left knot;
// the piece is a cubic in s = (r - g) unitR (real length).  Row P_s - 1 of
// spl is the constant outer-pair value beyond rc.
template <typename T>
__device__ __forceinline__ T pair_u_nu(T r, T cin, int cmax, T unitR, int Ps, const Vec4<T>* spl)
{
    int c = (int)(r * cin);
    c = c < cmax ? c : cmax;
    const Vec4<T> e = spl[Ps + c];
    const bool right = r > e.x;
    const int j = (int)e.y + (right ? 1 : 0);
    const T s = (r - (right ? e.w : e.z)) * unitR;
    const Vec4<T> cf = spl[j];
    return cf.x + s * (cf.y + s * (cf.z + s * cf.w));
}

typedef const __attribute__((address_space(3))) unsigned char* LdsBytes;

// One workgroup's share of the sweep: walkers blk * WPB .. (blk + 1) * WPB - 1
// of the system described by (sy, tb, a).  TAB: FP64, k-space terms from the phase
// table (sweep_phase_table); FP32, spline rows in the wide table (sweep_wide).
template <typename T, int D, int LPW, int KPL, bool PER, bool NU = false, bool TAB = false>
__device__ __forceinline__ void sweep_body(const KSys& sy, const KTables<T>& tb, const SweepArgs& a, int64_t blk)
{
    using C = Coord<T, PER>;
    using S = typename C::S;
    using Inc = typename C::Inc;
    constexpr int WPB = kThreads / LPW;   // walkers per block
    const int N = sy.N, Ps = sy.P_s, K = sy.Kh;   // k-space: one representative per +-k pair
    const int NT = sweep_table_len(sy);
    const int tid = threadIdx.x;
    const int grp = tid / LPW, gl = tid % LPW;
    const int64_t w = blk * WPB + grp;

    extern __shared__ __align__(16) unsigned char smem[];
    Vec4<T>* spl = reinterpret_cast<Vec4<T>*>(smem);                       // NT x (A0..A3) of Re u
    constexpr bool WIDE = TAB && sizeof(T) == 4, PHASES = TAB && sizeof(T) == 8;
    S* posb = reinterpret_cast<S*>(spl + NT * (WIDE ? kWide : 1));                                                    // WPB x N x D (particle-major)
    S* pos = posb + (size_t)grp * N * D;
    const int km = sy.kmax, prow = 2 * km + 1;                             // PHASES: rows per axis
    Vec2<T>* ptab = reinterpret_cast<Vec2<T>*>(smem + sweep_base_lds<T>(sy, LPW)) +
                    (size_t)grp * sweep_phase_len(sy);                     // PHASES: [D][prow][2]

    const T u_out = (T)tb.uR[sy.outer_idx];
    // real length per coordinate-difference unit
    const double scale = PER ? sy.Linv : 1.0;
    const double unit_len = C::kUnit / scale;
    if constexpr (NU) {
        // P_s rows (the last one the outer constant), then the cells in
        // coordinate-difference units
        for (int i = tid; i < Ps; i += kThreads) {
            const T* q = tb.spl + 8 * i;
            spl[i] = Vec4<T>{q[0], q[1], q[2], q[3]};
        }
        for (int i = tid; i < sy.ncell; i += kThreads) {
            const double* e = tb.nucell + 4 * i;
            spl[Ps + i] = Vec4<T>{(T)(e[0] / unit_len), (T)e[1], (T)(e[2] / unit_len), (T)(e[3] / unit_len)};
        }
    }
    for (int e = NU ? NT : tid; e < NT * (WIDE ? kWide : 1); e += kThreads) {
        const int i = WIDE ? e / kWide : e;
        const T* q = tb.spl + 8 * i;
        if (i < Ps - 1)
            spl[e] = Vec4<T>{q[0], q[1], q[2], q[3]};
        else
            spl[e] = Vec4<T>{u_out, (T)0, (T)0, (T)0};
    }
    // lengths in box units when periodic (scale = 1/L), unscaled otherwise;
    // diff() and raw() return multiples of C::kUnit of that unit
    const bool active = w < a.W;
    double* Rw = a.R + (active ? w : 0) * (size_t)N * D;
    if (active) {
        for (int e = gl; e < N * D; e += LPW) pos[e] = C::load(Rw[e] * scale);
    }
    __syncthreads();
    if (!active) return;

    const T hinv = (T)(sy.hinv / scale * C::kUnit), rc = (T)(sy.rc * scale / C::kUnit);
    const T cin = (T)(sy.cinv * unit_len), unitR = (T)unit_len;
    // WIDE: LDS address of the lane's copy of a row, byte 1 the row (two, for the
    // old and the new distance).  Right only while the table starts at LDS address
    // 0, that is while the kernel has no static LDS (tests/test_kernel_registers_cpu.py
    // reads that from the built kernels); adding the start to each address instead
    // is two more instructions a pair
    uint32_t row_at[2];
    row_at[0] = row_at[1] = (uint32_t)(uintptr_t)(LdsBytes)smem + (tid & (kWide - 1)) * sizeof(Vec4<T>);
    auto uof = [&](T r, int q = 0) -> T {
        if constexpr (WIDE) {
            const T x = r * hinv;
            const T t = Prec<T>::fract_(x);
            asm("v_cvt_u32_f32_sdwa %0, %1 dst_sel:BYTE_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD" : "+v"(row_at[q]) : "v"(x));
            typedef float Row __attribute__((ext_vector_type(4)));   // 16-byte aligned: one LDS read
            const Row cf = *(const __attribute__((address_space(3))) Row*)(LdsBytes)(uintptr_t)row_at[q];
            return cf.x + t * (cf.y + t * (cf.z + t * cf.w));
        } else if constexpr (NU)
            return pair_u_nu<T>(r, cin, sy.ncell - 1, unitR, Ps, spl);
        else
            return pair_u<T, PER>(r, rc, hinv, Ps, spl, u_out);
    };
    const T step = (T)(sy.step * scale);
    // one-body factor on raw coordinates: -ob sum raw^2
    const T ob = sy.one_body ? (T)(tb.uR[0] / (scale * scale) * C::kUnit * C::kUnit) : (T)0;

    // this lane's k-vectors and amplitudes, and twice their rho_k (sR + i sI =
    // 2 rho_k: scaling by 2 is exact, and it saves a multiply per k and trial)
    constexpr int KP = KPL > 0 ? KPL : 1;
    T sR[KP], sI[KP], qa[KP];
    // PHASES: the lane's rows in the phase table; otherwise revolutions per raw
    // coordinate unit
    T qx[KP], qy[KP], qz[KP];
    int rx[KP], ry[KP], rz[KP];
    // periodic: kv L is the integer lattice vector n (rounded to remove the
    // storage error of n / L)
    auto lattice = [&](T v) { return PER ? rint((double)v / scale) : (double)v; };
    // all loads under way before the first is used: one by one behind a branch they
    // were 2 to 4 us of a small batch (4 systems, 101 terms, 256 walkers each: 61 us
    // against 63)
    T kv[KP][3], al[KP];
    if (KPL > 0) {
#pragma unroll
        for (int m = 0; m < KPL; m++) {
            const int k = min(gl + m * LPW, K - 1);
            if (K == 0) break;
#pragma unroll
            for (int c = 0; c < 3; c++) kv[m][c] = tb.kv[4 * k + c];
            al[m] = tb.alpha[2 * k];
        }
    }
#pragma unroll
    for (int m = 0; m < KPL; m++) {
        sR[m] = sI[m] = (T)0;
        const int k = gl + m * LPW;
        qx[m] = qy[m] = qz[m] = qa[m] = (T)0;   // lanes past K: zero amplitude, no effect
        rx[m] = ry[m] = rz[m] = 2 * km;
        if (k < K) {
            const T* q = kv[m];
            qa[m] = al[m];
            if constexpr (PHASES) {
                rx[m] = 2 * (km + (int)lattice(q[0]));
                ry[m] = 2 * (prow + km + (int)lattice(q[1]));
                if (D > 2) rz[m] = 2 * (2 * prow + km + (int)lattice(q[2]));
            } else {
                qx[m] = (T)(lattice(q[0]) * C::kUnit);
                qy[m] = (T)(lattice(q[1]) * C::kUnit);
                qz[m] = (T)(lattice(q[2]) * C::kUnit);
            }
        }
    }
    // PHASES: lane gl computes the factors e = gl + j LPW of (position, axis, m =
    // 1 .. kmax): the coordinate's axis, the power, whether the position's
    // displacement is added (as a 0 / 1 weight per axis), the rows of m and -m
    constexpr int NE = PHASES ? 64 / LPW : 1;
    T ew[NE][3], em[NE];
    int ea[NE], eq[NE], eplus[NE], eminus[NE];
    const int ne = 2 * D * km;
    if constexpr (PHASES) {
#pragma unroll
        for (int j = 0; j < NE; j++) {
            const int e = gl + j * LPW;
            const bool on = e < ne;
            const int q = on ? e / (D * km) : 0, f = on ? e - q * (D * km) : 0;
            ea[j] = km ? f / km : 0;
            eq[j] = q;
            const int m = on ? f - ea[j] * km + 1 : 0;   // 0: an idle lane, whose put is left out
            em[j] = (T)m;
            eplus[j] = 2 * (ea[j] * prow + km + m) + q;
            eminus[j] = 2 * (ea[j] * prow + km - m) + q;
#pragma unroll
            for (int c = 0; c < 3; c++) ew[j][c] = (q == 1 && ea[j] == c) ? (T)1 : (T)0;
        }
        for (int e = gl; e < 2 * D; e += LPW) ptab[2 * ((e >> 1) * prow + km) + (e & 1)] = Vec2<T>{(T)1, (T)0};
    }
    // factor e^{2 pi i m x} into both rows, |x| <= 3/2; the phase is reduced
    // before it is rounded
    auto put = [&](int j, T x) {
        const T t = em[j] * x;
        T sn, cs;
        Prec<T>::sincos_rev(__builtin_fma(em[j], x, -Prec<T>::rint_(t)), &sn, &cs);
        ptab[eplus[j]] = Vec2<T>{cs, sn};
        ptab[eminus[j]] = Vec2<T>{cs, -sn};
    };
    // e^{ik.r} of this lane's term m at position q
    auto take = [&](int m, int q, T* re, T* im) {
        Vec2<T> z = ptab[rx[m] + q];
        const Vec2<T> y = ptab[ry[m] + q];
        z = Vec2<T>{z.x * y.x - z.y * y.y, z.x * y.y + z.y * y.x};
        if (D > 2) {
            const Vec2<T> v = ptab[rz[m] + q];
            z = Vec2<T>{z.x * v.x - z.y * v.y, z.x * v.y + z.y * v.x};
        }
        *re = z.x;
        *im = z.y;
    };
    auto lds_order = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    if constexpr (PHASES) {
        // rho_k of the walker, two particles per pass
        for (int n = 0; n < N; n += 2) {
            lds_order();
#pragma unroll
            for (int j = 0; j < NE; j++)
                if (gl + j * LPW < ne) put(j, pos[min(n + eq[j], N - 1) * D + ea[j]]);
            lds_order();
            const T w1 = n + 1 < N ? (T)1 : (T)0;
#pragma unroll
            for (int m = 0; m < KPL; m++) {
                T c0, s0, c1, s1;
                take(m, 0, &c0, &s0);
                take(m, 1, &c1, &s1);
                sR[m] += c0 + w1 * c1;
                sI[m] += s0 + w1 * s1;
            }
        }
        lds_order();
    } else {
#pragma unroll
        for (int m = 0; m < KPL; m++) {
            if (gl + m * LPW >= K) continue;
            for (int n = 0; n < N; n++) {
                T ph = qx[m] * C::raw(pos[n * D]);
                if (D > 1) ph += qy[m] * C::raw(pos[n * D + 1]);
                if (D > 2) ph += qz[m] * C::raw(pos[n * D + 2]);
                T s, c;
                Prec<T>::sincos_small(ph, &s, &c);
                sR[m] += c;
                sI[m] += s;
            }
        }
    }
#pragma unroll
    for (int m = 0; m < KPL; m++) {
        sR[m] *= (T)2;
        sI[m] *= (T)2;
    }
    // u at distance 0: the moved particle meets itself in the partner loop
    const T u_zero = uof((T)0);

    const uint32_t k0 = (uint32_t)a.seed, k1 = (uint32_t)(a.seed >> 32);
    const uint32_t ep = a.epoch ? *a.epoch : 0u;
    const int64_t ntr = a.n_moves;
    unsigned long long nacc = 0;
    int seq = 0;   // sequential order: particle of trial base + gl

    for (int64_t base = 0; base < ntr; base += LPW) {
        // lane gl prepares trial base + gl: particle, displacement increments,
        // log u, and the self term u(|move|) - u(0) that the partner loop adds
        const uint32_t tr = (uint32_t)(base + gl);
        Philox4 x = philox4x32_10(tr, ep, (uint32_t)w, 0u, k0, k1);
        int pm;
        if (sy.move_order == 0) {
            pm = (int)__umulhi(x.v[0], (uint32_t)N);
        } else {
            pm = seq + gl;
            while (pm >= N) pm -= N;
            seq += LPW;
            while (seq >= N) seq -= N;
        }
        Inc dl[3];
        T logu, uself;
        {
            // Box-Muller on (v1, v2) -> two normals; D = 3 draws a second block
            T z[3];
            const float u1 = u01f(x.v[1]), u2 = u01f(x.v[2]);
            const float rr = sqrtf(-2.0f * __logf(u1));
            float sn, cs;
            Prec<float>::sincos_rev(u2, &sn, &cs);
            z[0] = (T)(rr * cs);
            z[1] = (T)(rr * sn);
            if (D == 3) {
                Philox4 y = philox4x32_10(tr, ep, (uint32_t)w, 1u, k0, k1);
                const float v1 = u01f(y.v[0]), v2 = u01f(y.v[1]);
                const float r2 = sqrtf(-2.0f * __logf(v1));
                float s2, c2;
                Prec<float>::sincos_rev(v2, &s2, &c2);
                z[2] = (T)(r2 * c2);
            } else {
                z[2] = (T)0;
            }
            logu = (T)__logf(u01f(x.v[3]));
            T s2 = Prec<T>::kR2Floor;
#pragma unroll
            for (int c = 0; c < D; c++) {
                dl[c] = C::inc(step * z[c]);
                const T dm = C::diff((S)0, C::add((S)0, dl[c]));
                s2 += dm * dm;
            }
            uself = uof(Prec<T>::sqrt_r2(s2)) - u_zero;
        }
        const int nb = (int)((ntr - base) < LPW ? (ntr - base) : LPW);
        for (int tt = 0; tt < nb; tt++) {
            const int p = bcast_i<LPW>(pm, tt);
            S* const pp = pos + __umul24((uint32_t)p, (uint32_t)D);   // the moved particle's slot
            S old[D], nw[D];
            Inc dz[D];
#pragma unroll
            for (int c = 0; c < D; c++) {
                old[c] = pp[c];
                dz[c] = bcast<LPW>(dl[c], tt);
                nw[c] = C::add(old[c], dz[c]);
            }
            if constexpr (PHASES) {
                // phase factors of the old and the new position (read after the
                // partner loop); a whole box added or taken off leaves them alone
#pragma unroll
                for (int j = 0; j < NE; j++) {
                    if (gl + j * LPW < ne) {
                        T x = pp[ea[j]];
#pragma unroll
                        for (int c = 0; c < D; c++) x = __builtin_fma(ew[j][c], dz[c], x);
                        put(j, x);
                    }
                }
                lds_order();
            }
            const T lu = bcast<LPW>(logu, tt);
            const T us = bcast<LPW>(uself, tt);
            T delta = (T)0;
            auto partner = [&](int i) {
                T ro2 = Prec<T>::kR2Floor, rn2 = Prec<T>::kR2Floor;
#pragma unroll
                for (int c = 0; c < D; c++) {
                    const S pi = pos[i * D + c];
                    const T dOld = C::diff(pi, old[c]), dNew = C::diff(pi, nw[c]);
                    ro2 += dOld * dOld;
                    rn2 += dNew * dNew;
                }
                const T uo = uof(Prec<T>::sqrt_r2(ro2));
                const T un = uof(Prec<T>::sqrt_r2(rn2), 1);
                delta += un - uo;
            };
            // rounds in which every lane of the group has a partner run under a
            // bound common to the group (loop control on scalar registers), the
            // last, partial round under the lane's own test; same partners, same
            // order as one loop over i = gl, gl + LPW, ... < N
            const int nfull = N / LPW;
#pragma unroll 1
            for (int m = 0; m < nfull; m++) partner(gl + m * LPW);
            if (gl + nfull * LPW < N) partner(gl + nfull * LPW);
            T oc[D], ncd[D];
#pragma unroll
            for (int c = 0; c < D; c++) {
                oc[c] = C::raw(old[c]);
                ncd[c] = C::raw(nw[c]);
            }
            T dR[KPL > 0 ? KPL : 1], dI[KPL > 0 ? KPL : 1];
#pragma unroll
            for (int m = 0; m < KPL; m++) {
                T so, co, sn, cn;
                if constexpr (PHASES) {
                    take(m, 0, &co, &so);
                    take(m, 1, &cn, &sn);
                } else {
                    // |phase| <= sum |n_a| / 2 revolutions: no range reduction needed
                    T po = qx[m] * oc[0], pn = qx[m] * ncd[0];
                    if (D > 1) {
                        po += qy[m] * oc[1];
                        pn += qy[m] * ncd[1];
                    }
                    if (D > 2) {
                        po += qz[m] * oc[2];
                        pn += qz[m] * ncd[2];
                    }
                    Prec<T>::sincos_small(po, &so, &co);
                    Prec<T>::sincos_small(pn, &sn, &cn);
                }
                dR[m] = cn - co;
                dI[m] = sn - so;
                // |rho + d|^2 - |rho|^2 = 2 Re(conj(rho) d) + |d|^2 = Re((2 rho + d) conj(d))
                delta += qa[m] * ((sR[m] + dR[m]) * dR[m] + (sI[m] + dI[m]) * dI[m]);
            }
            if (sy.one_body) {
                // a branch on the (uniform) flag, not a select: systems without
                // the one-body factor skip these instructions
                asm volatile("" ::: "memory");
                T ro2 = (T)0, rn2 = (T)0;
#pragma unroll
                for (int c = 0; c < D; c++) {
                    ro2 += oc[c] * oc[c];
                    rn2 += ncd[c] * ncd[c];
                }
                if (gl == 0) delta += -ob * (rn2 - ro2);
            }
            const bool accept = group_accept<LPW>(delta, us, lu);
            if (accept) {
                if (gl == 0) {
#pragma unroll
                    for (int c = 0; c < D; c++) pp[c] = nw[c];
                }
#pragma unroll
                for (int m = 0; m < KPL; m++) {
                    sR[m] += (T)2 * dR[m];
                    sI[m] += (T)2 * dI[m];
                }
                nacc++;
            }
            // the moved particle's LDS slot is read by every lane of the group next trial
            lds_order();
        }
    }

    for (int e = gl; e < N * D; e += LPW) Rw[e] = C::store(pos[e]) * (PER ? sy.L : 1.0);
    if (a.rho_out) {
        T* ro = static_cast<T*>(a.rho_out) + (size_t)w * K * 2;
#pragma unroll
        for (int m = 0; m < KPL; m++) {
            const int k = gl + m * LPW;
            if (k < K) {
                ro[2 * k] = (T)0.5 * sR[m];
                ro[2 * k + 1] = (T)0.5 * sI[m];
            }
        }
    }
    if (gl == 0 && a.acc) a.acc[w] += nacc;
}

// FP64: scheduled for 4 wavefronts per SIMD (3 with many k-space terms, whose
// sums and rows fill the registers): the LDS of the larger systems allows no
// more, and a scheduler that aims at 5 serialises the old and the new pair
// term to save the registers (N = 343: 7.6 against 7.5 ms).
constexpr int sweep_least_waves(bool fp64, int kpl) { return !fp64 ? 1 : (kpl > 2 ? 3 : 4); }
constexpr int sweep_most_waves(bool fp64) { return fp64 ? 4 : 8; }
template <typename T, int D, int LPW, int KPL, bool PER, bool NU, bool TAB>
__global__ __launch_bounds__(kThreads)
    __attribute__((amdgpu_waves_per_eu(sweep_least_waves(sizeof(T) == 8, KPL), sweep_most_waves(sizeof(T) == 8))))
    void sweep_kernel(KSys sy, KTables<T> tb, SweepArgs a)
{
    sweep_body<T, D, LPW, KPL, PER, NU, TAB>(sy, tb, a, blockIdx.x);
}

// Batch of independent systems in one launch: workgroup b belongs to system
// s with block_start[s] <= b < block_start[s + 1].
template <typename T, int D, int LPW, int KPL, bool PER>
__global__ __launch_bounds__(kThreads) void sweep_batch_kernel(SweepBatch<T> bt)
{
    int lo = 0, hi = bt.n;   // last s with block_start[s] <= blockIdx.x
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (bt.block_start[mid] <= (int64_t)blockIdx.x)
            lo = mid;
        else
            hi = mid;
    }
    const int64_t blk = (int64_t)blockIdx.x - bt.block_start[lo];
    if constexpr (sizeof(T) == 8 && KPL > 0 && D > 1) {
        if (sweep_phase_table<T>(bt.sys[lo], LPW)) {
            sweep_body<T, D, LPW, KPL, PER, false, true>(bt.sys[lo], bt.tab[lo], bt.args[lo], blk);
            return;
        }
    }
    sweep_body<T, D, LPW, KPL, PER>(bt.sys[lo], bt.tab[lo], bt.args[lo], blk);
}

}  // namespace

template <typename T, int D, int LPW, int KPL, bool PER>
static hipError_t launch_sweep_k(const KSys& sy, const KTables<T>& tb, const SweepArgs& a, hipStream_t st)
{
    size_t lds = sweep_lds_bytes<T>(sy, LPW);
    if (sy.nu && (!PER || !tb.nucell)) return hipErrorInvalidValue;
    auto kern = sy.nu ? sweep_kernel<T, D, LPW, KPL, PER, PER, false> : sweep_kernel<T, D, LPW, KPL, PER, false, false>;
    if constexpr (sizeof(T) == 8 && KPL > 1 && D > 1) {
        if (sweep_phase_table<T>(sy, LPW))
            kern = sy.nu ? sweep_kernel<T, D, LPW, KPL, PER, PER, true> : sweep_kernel<T, D, LPW, KPL, PER, false, true>;
    }
    if constexpr (sizeof(T) == 4 && PER) {
        if (sweep_wide<T>(sy, LPW)) {
            kern = sweep_kernel<T, D, LPW, KPL, PER, false, true>;
            lds = sweep_wide_lds<T>(sy, LPW);
        }
    }
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    const int wpb = kThreads / LPW;
    const int64_t blocks = (a.W + wpb - 1) / wpb;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kThreads), lds, st, sy, tb, a);
    return hipGetLastError();
}

template <typename T, int D, int LPW, bool PER>
static hipError_t launch_sweep_l(const KSys& sy, const KTables<T>& tb, const SweepArgs& a, hipStream_t st)
{
    const int kpl = (sy.Kh + LPW - 1) / LPW;
    if (kpl == 0) return launch_sweep_k<T, D, LPW, 0, PER>(sy, tb, a, st);
    if constexpr (!PER) {
        return hipErrorInvalidValue;   // k-space terms need the periodic box
    } else {
        // a term past the lane's last costs what a real one does (31 issue
        // slots of about 450 per trial in the FP32 form): every count has its
        // kernel (258 terms of a 2-D system with 512 k on 64 lanes, 5 instead of
        // 8: mixed sweep 35.2 -> 29.6 ms at 131072 walkers, N = 400), but 7,
        // which runs in the kernel of 8 with one empty term
        switch (kpl) {
        case 1: return launch_sweep_k<T, D, LPW, 1, PER>(sy, tb, a, st);
        case 2: return launch_sweep_k<T, D, LPW, 2, PER>(sy, tb, a, st);
        case 3: return launch_sweep_k<T, D, LPW, 3, PER>(sy, tb, a, st);
        case 4: return launch_sweep_k<T, D, LPW, 4, PER>(sy, tb, a, st);
        case 5: return launch_sweep_k<T, D, LPW, 5, PER>(sy, tb, a, st);
        case 6: return launch_sweep_k<T, D, LPW, 6, PER>(sy, tb, a, st);
        case 7:
        case 8: return launch_sweep_k<T, D, LPW, 8, PER>(sy, tb, a, st);
        }
        return hipErrorInvalidValue;
    }
}

template <typename T, int D>
static hipError_t launch_sweep_d(const KSys& sy, const KTables<T>& tb, const SweepArgs& a, hipStream_t st)
{
    const int lpw = a.lanes_per_walker > 0 ? a.lanes_per_walker : default_lanes<T>(sy, a.W);
    const bool per = sy.periodic != 0;
    switch (lpw) {
    case 16: return per ? launch_sweep_l<T, D, 16, true>(sy, tb, a, st) : launch_sweep_l<T, D, 16, false>(sy, tb, a, st);
    case 32: return per ? launch_sweep_l<T, D, 32, true>(sy, tb, a, st) : launch_sweep_l<T, D, 32, false>(sy, tb, a, st);
    case 64: return per ? launch_sweep_l<T, D, 64, true>(sy, tb, a, st) : launch_sweep_l<T, D, 64, false>(sy, tb, a, st);
    default: return hipErrorInvalidValue;
    }
}

// Batch without k-space terms, each system with its own lanes per walker
// (8, 16, 32 or 64, from its SweepArgs); a workgroup belongs to one system.
template <typename T, int D, bool PER>
__global__ __launch_bounds__(kThreads) void sweep_batch_lanes_kernel(SweepBatch<T> bt)
{
    int lo = 0, hi = bt.n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (bt.block_start[mid] <= (int64_t)blockIdx.x)
            lo = mid;
        else
            hi = mid;
    }
    const int64_t blk = (int64_t)blockIdx.x - bt.block_start[lo];
    switch (bt.args[lo].lanes_per_walker) {
    case 8: sweep_body<T, D, 8, 0, PER>(bt.sys[lo], bt.tab[lo], bt.args[lo], blk); break;
    case 16: sweep_body<T, D, 16, 0, PER>(bt.sys[lo], bt.tab[lo], bt.args[lo], blk); break;
    case 64: sweep_body<T, D, 64, 0, PER>(bt.sys[lo], bt.tab[lo], bt.args[lo], blk); break;
    default: sweep_body<T, D, 32, 0, PER>(bt.sys[lo], bt.tab[lo], bt.args[lo], blk); break;
    }
}

template <typename T, int D, bool PER>
static hipError_t launch_sweep_batch_lanes(const SweepBatch<T>& bt, int64_t blocks, size_t lds, hipStream_t st)
{
    auto kern = sweep_batch_lanes_kernel<T, D, PER>;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kThreads), lds, st, bt);
    return hipGetLastError();
}

template <typename T, int D, int LPW, int KPL, bool PER>
static hipError_t launch_sweep_batch_k(const SweepBatch<T>& bt, int64_t blocks, size_t lds, hipStream_t st)
{
    auto kern = sweep_batch_kernel<T, D, LPW, KPL, PER>;
    if (lds > 65536) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kThreads), lds, st, bt);
    return hipGetLastError();
}

template <typename T, int D, int LPW, bool PER>
static hipError_t launch_sweep_batch_l(const SweepBatch<T>& bt, int kh_max, int64_t blocks, size_t lds,
                                       hipStream_t st)
{
    const int kpl = (kh_max + LPW - 1) / LPW;
    if (kpl == 0) return launch_sweep_batch_k<T, D, LPW, 0, PER>(bt, blocks, lds, st);
    if constexpr (!PER) {
        return hipErrorInvalidValue;
    } else {
        if (kpl <= 2) return launch_sweep_batch_k<T, D, LPW, 2, PER>(bt, blocks, lds, st);
        if (kpl <= 4) return launch_sweep_batch_k<T, D, LPW, 4, PER>(bt, blocks, lds, st);
        if (kpl <= 8) return launch_sweep_batch_k<T, D, LPW, 8, PER>(bt, blocks, lds, st);
        return hipErrorInvalidValue;
    }
}

template <typename T>
hipError_t launch_sweep_batch(const SweepBatch<T>& bt, int D, bool periodic, int lanes, int kh_max, int64_t blocks,
                              size_t lds, hipStream_t st)
{
    if (blocks <= 0) return hipSuccess;
    if (lanes == 0) {
        // per-system lanes (no k-space terms)
        if (kh_max > 0) return hipErrorInvalidValue;
        switch (D) {
        case 1: return periodic ? launch_sweep_batch_lanes<T, 1, true>(bt, blocks, lds, st)
                                : launch_sweep_batch_lanes<T, 1, false>(bt, blocks, lds, st);
        case 2: return periodic ? launch_sweep_batch_lanes<T, 2, true>(bt, blocks, lds, st)
                                : launch_sweep_batch_lanes<T, 2, false>(bt, blocks, lds, st);
        case 3: return periodic ? launch_sweep_batch_lanes<T, 3, true>(bt, blocks, lds, st)
                                : launch_sweep_batch_lanes<T, 3, false>(bt, blocks, lds, st);
        default: return hipErrorInvalidValue;
        }
    }
#define TDVMC_SWEEP_BATCH_D(DD)                                                                              \
    switch (lanes) {                                                                                         \
    case 16: return periodic ? launch_sweep_batch_l<T, DD, 16, true>(bt, kh_max, blocks, lds, st)             \
                             : launch_sweep_batch_l<T, DD, 16, false>(bt, kh_max, blocks, lds, st);           \
    case 32: return periodic ? launch_sweep_batch_l<T, DD, 32, true>(bt, kh_max, blocks, lds, st)             \
                             : launch_sweep_batch_l<T, DD, 32, false>(bt, kh_max, blocks, lds, st);           \
    case 64: return periodic ? launch_sweep_batch_l<T, DD, 64, true>(bt, kh_max, blocks, lds, st)             \
                             : launch_sweep_batch_l<T, DD, 64, false>(bt, kh_max, blocks, lds, st);           \
    default: return hipErrorInvalidValue;                                                                    \
    }
    switch (D) {
    case 1: TDVMC_SWEEP_BATCH_D(1)
    case 2: TDVMC_SWEEP_BATCH_D(2)
    case 3: TDVMC_SWEEP_BATCH_D(3)
    default: return hipErrorInvalidValue;
    }
#undef TDVMC_SWEEP_BATCH_D
}

int sweep_walkers_per_block(int lanes) { return kThreads / lanes; }
int sweep_default_lanes(int N, int Kh) { return pick_lpw(N, Kh); }

template <typename T>
hipError_t launch_sweep(const KSys& sy, const KTables<T>& tb, const SweepArgs& a, hipStream_t st)
{
    if (a.W <= 0 || a.n_moves <= 0) return hipSuccess;
    switch (sy.D) {
    case 1: return launch_sweep_d<T, 1>(sy, tb, a, st);
    case 2: return launch_sweep_d<T, 2>(sy, tb, a, st);
    case 3: return launch_sweep_d<T, 3>(sy, tb, a, st);
    default: return hipErrorInvalidValue;
    }
}

template hipError_t launch_sweep_batch<float>(const SweepBatch<float>&, int, bool, int, int, int64_t, size_t,
                                              hipStream_t);
template hipError_t launch_sweep_batch<double>(const SweepBatch<double>&, int, bool, int, int, int64_t, size_t,
                                               hipStream_t);
template hipError_t launch_sweep<float>(const KSys&, const KTables<float>&, const SweepArgs&, hipStream_t);
template hipError_t launch_sweep<double>(const KSys&, const KTables<double>&, const SweepArgs&, hipStream_t);
template size_t sweep_lds_bytes<float>(const KSys&, int);
template size_t sweep_lds_bytes<double>(const KSys&, int);

}  // namespace tdvmc
