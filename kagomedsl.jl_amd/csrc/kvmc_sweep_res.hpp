// Sweep kernel of small clusters (gfx950): one wavefront per walker, W in LDS.
//
// Carlo.sweep! (src/MonteCarlo.jl:538-607) with the arithmetic of k_sweep,
// operation by operation, where both W of a walker are LDS-resident and no
// spin has more than 64 rows or labels: a row and a label per lane, no barrier.
// Bound by latency: a launch is a dozen dependent steps per accepted move, so
//   - what a walker needs is loaded at once at the start (W and the bond
//     tables as 16-byte vectors, several in flight), and stored so at the end;
//   - 64 draws are held in registers, one per lane, until they are passed;
//   - Z_mu changes by one bond per lane, for the accepted move only (k_sweep
//     walks the neighbours of every proposal);
//   - no vector register spills (k_sweep's instance for 12 terms spilled 89);
//     150 to 212 scalar ones do, into lanes of vector registers.
// us of sweep kernels per N sweeps, k_sweep and here: 777 walkers of 108 sites,
// FP64, 263 and 192; 4096 walkers of 48 sites, FP32, delay 12, 320 and 272 (96
// with the counters kept per walker).
#pragma once

#include "kvmc_kernels.hpp"

namespace kvmc {

// w += a * b of one element, as vmac does per element of its vectors.
__device__ __forceinline__ void emac(float& w, float a, float b) { w += a * b; }
__device__ __forceinline__ void emac(double& w, double a, double b) { w += a * b; }
template <typename R>
__device__ __forceinline__ void emac(cplx<R>& w, cplx<R> a, cplx<R> b) {
    w.re += a.re * b.re - a.im * b.im;
    w.im += a.im * b.re + a.re * b.im;
}

// W0[:, j] += sum_{q<c} A_q B_q[j], W in LDS: a row per lane, its A_q in
// registers, B_q[j] an LDS broadcast; four or eight columns in flight.
template <typename T, int DMAX>
__device__ __forceinline__ void flush_w1(T* W0, const T* sA, const T* sB, int ld, int nsa, int nmax, int ncols, int c) {
    const int lane = (int)threadIdx.x;
    if (lane >= ld) return;
    T a[DMAX];
#pragma unroll
    for (int q = 0; q < DMAX; ++q) a[q] = sA[(q < c ? q : 0) * nsa + lane];
    constexpr int U = DMAX <= 1 ? 8 : 4;
    for (int j0 = 0; j0 < ncols; j0 += U) {
        T v[U];
        int jc[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            jc[u] = j0 + u < ncols ? j0 + u : ncols - 1;
            v[u] = W0[jc[u] * ld + lane];
        }
#pragma unroll
        for (int q = 0; q < DMAX; ++q) {
            if (q < c) {
#pragma unroll
                for (int u = 0; u < U; ++u) emac(v[u], a[q], sB[q * nmax + jc[u]]);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (j0 + u < ncols) W0[(j0 + u) * ld + lane] = v[u];
    }
}

// Copies n 16-byte vectors with one wavefront, eight in flight.
__device__ __forceinline__ void copy_vec(f32x4* d, const f32x4* g, int n) {
    constexpr int U = 8;
    for (int t0 = (int)threadIdx.x; t0 < n; t0 += 64 * U) {
        f32x4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (t0 + 64 * u < n) v[u] = g[t0 + 64 * u];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (t0 + 64 * u < n) d[t0 + 64 * u] = v[u];
    }
}

inline size_t sweep_w1_lds(size_t es, int ns, int nup, int ndn, int delay, int nb) {
    const int nmax = nup > ndn ? nup : ndn;
    const size_t nsp = (size_t)(ns + 3) / 4 * 4;
    return w_stride(ns, nup, ndn) * es                                          // W (whole 16-byte vectors)
           + 2 * (size_t)delay * ((size_t)w_nsa(ns, nup, ndn) + (nmax + 3) / 4 * 4) * es   // pending terms
           + 4 * nsp * sizeof(int16_t) + bond_table_bytes(ns, nb);
}

// A row and a label per lane; with thousands of bonds the LDS can exceed that
// of k_sweep, which takes the handle then.
inline bool sweep_w1_fits(size_t es, int ns, int nup, int ndn, int delay, int nb) {
    const int nmax = nup > ndn ? nup : ndn;
    return w_nsa(ns, nup, ndn) <= 64 && nmax <= 64 && ns <= 128 && sweep_w1_lds(es, ns, nup, ndn, delay, nb) <= 160 * 1024;
}

template <typename T, int DMAX>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) k_sweep_w1(SweepArgs a) {
    extern __shared__ __align__(16) unsigned char lds[];
    const int w = a.walker0 + (int)blockIdx.x, lane = (int)threadIdx.x;
    const int ns = a.ns, nup = a.nup, ndn = a.ndn, nb = a.nb;
    const int nsp = round_up(ns, 4), nmx = round_up(a.nmax, 4);
    const int nsa = w_nsa(ns, nup, ndn), delay = a.delay;
    const int ldu = w_ld(ns, nup), ldd = w_ld(ns, ndn);
    const size_t wstride = w_stride(ns, nup, ndn);
    T* Wup = reinterpret_cast<T*>(lds);
    T* Wdn = Wup + w_off_dn(ns, nup);
    T* sAu = Wup + wstride;                               // [2][delay][nsa]
    T* sAd = sAu + delay * nsa;
    T* sBu = sAu + 2 * delay * nsa;                       // [2][delay][nmx]
    T* sBd = sBu + delay * nmx;
    uint32_t* s_bond = reinterpret_cast<uint32_t*>(sBu + 2 * delay * nmx);   // the bond tables
    uint16_t* s_noff = reinterpret_cast<uint16_t*>(s_bond + nb);
    uint16_t* s_nbr = s_noff + ns + 1;
    int16_t* s_kup = reinterpret_cast<int16_t*>(reinterpret_cast<unsigned char*>(s_bond) + bond_table_bytes(ns, nb));
    int16_t* s_kdn = s_kup + nsp;
    int16_t* s_slu = s_kdn + nsp;                         // site -> row of W_up (-1: occupied)
    int16_t* s_sld = s_slu + nsp;

    long long sweeps = a.sweeps[w];
    const long long stop = a.stop[w];
    int c = a.npend[w];
    int acc_since = a.acc_since[w];
    if (sweeps >= stop || *a.failed != 0x7fffffff) return;
    {
        // labels and rows first, so that their loads are under way with W's
        const int* ku = a.kup + (size_t)w * ns;
        const int* kd = a.kdn + (size_t)w * ns;
        const int* sg = a.slot + (size_t)w * 2 * ns;
        int v[2][4];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int t = lane + 64 * u;
            if (t < ns) { v[u][0] = ku[t]; v[u][1] = kd[t]; v[u][2] = sg[t]; v[u][3] = sg[ns + t]; }
        }
        copy_vec(reinterpret_cast<f32x4*>(s_bond), reinterpret_cast<const f32x4*>(a.table),
                 (int)(bond_table_bytes(ns, nb) / 16));
        copy_vec(reinterpret_cast<f32x4*>(Wup),
                 reinterpret_cast<const f32x4*>(reinterpret_cast<const T*>(a.W) + (size_t)w * wstride),
                 (int)(wstride * sizeof(T) / 16));
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int t = lane + 64 * u;
            if (t < ns) {
                s_kup[t] = (int16_t)v[u][0]; s_kdn[t] = (int16_t)v[u][1];
                s_slu[t] = (int16_t)v[u][2]; s_sld[t] = (int16_t)v[u][3];
            }
        }
    }
    constexpr int V = 16 / (int)sizeof(T), NVC = (DMAX + V - 1) / V;
    using VT = typename VecT<T, V>::type;
    if (c > 0) {
        // pending terms: planes over rows and labels in HBM (pend_at)
        const int dp = pend_ld(delay);
        const T* gA = reinterpret_cast<const T*>(a.A) + (size_t)w * 2 * nsa * dp;
        const T* gB = reinterpret_cast<const T*>(a.Bm) + (size_t)w * 2 * a.nmax * dp;
#pragma unroll
        for (int part = 0; part < 4; ++part) {
            const int n = part < 2 ? nsa : a.nmax, st = part < 2 ? nsa : nmx;
            const T* g = part < 2 ? gA + (size_t)part * nsa * dp : gB + (size_t)(part - 2) * a.nmax * dp;
            T* d = part == 0 ? sAu : part == 1 ? sAd : part == 2 ? sBu : sBd;
            if (lane < n) {
                VT v[NVC];
#pragma unroll
                for (int p = 0; p < NVC; ++p)
                    if (V * p < c) v[p] = reinterpret_cast<const VT*>(g)[p * n + lane];
#pragma unroll
                for (int p = 0; p < NVC; ++p) {
                    const T* e = reinterpret_cast<const T*>(&v[p]);
#pragma unroll
                    for (int u = 0; u < V; ++u)
                        if (V * p + u < c) d[(V * p + u) * st + lane] = e[u];
                }
            }
        }
    }
    wave_sync();
    int zmu = 0;
    for (int b0 = 0; b0 < nb; b0 += 64) {
        bool ap = false;
        if (b0 + lane < nb) {
            const uint32_t bp = s_bond[b0 + lane];
            const int i = (int)(bp & 0xffffu), j = (int)(bp >> 16);
            ap = (s_kup[i] != 0 && s_kdn[j] != 0) || (s_kup[j] != 0 && s_kdn[i] != 0);
        }
        zmu += __popcll(__ballot(ap));
    }
    const double zmax = (double)nb;
    unsigned long long n_moves = 0, n_acc = 0, n_flush = 0;
    const long long sweeps0 = sweeps;
    bool pause = false;
    long long dbase = sweeps - 64;   // the draws held are those of sweeps dbase .. dbase + 63
    unsigned dmod = (unsigned)((sweeps + (long long)a.nocc * 64 - 64) % a.nocc);   // dbase modulo nocc
    double r = 1.0;
    int i = 0, site = 0;             // the drawn bond's sites
    while (sweeps < stop && !pause) {
        if (sweeps >= dbase + 64) {
            dbase = sweeps;
            const long long sw = dbase + lane;
            int bidx = 0;
            r = 1.0;
            if (sw < stop) {
                if (a.tape_u) {
                    const long long tidx = (long long)w * a.tape_len + (sw - a.tape_base[w]);
                    r = a.tape_u[tidx];
                    bidx = a.tape_bond[tidx];
                } else {
                    sweep_draws(a.seed, (uint32_t)w, sw, nb, &r, &bidx);
                }
            }
            const uint32_t bp = s_bond[bidx];
            i = (int)(bp & 0xffffu);
            site = (int)(bp >> 16);
            dmod = (dmod + 64) % (unsigned)a.nocc;
        }
        const long long sw = dbase + lane;
        const bool live = sw >= sweeps && sw < stop;
        const double zr = (double)zmu / zmax;
        const int iu = s_kup[i], su = s_kup[site], id = s_kdn[i], sd = s_kdn[site];
        const bool pre = a.kernel_mode == KERNEL_REFERENCE && r > zr;
        const bool can1 = iu != 0 && sd != 0, can2 = su != 0 && id != 0;
        const bool mv = live && !pre && (can1 || can2);
        bool acc = false;
        // flag = 1: up moves i -> site, down moves site -> i; max() keeps a
        // walker with an inconsistent state (failed refresh) inside W
        const int lup = mv ? (can1 ? iu : su) - 1 : 0, ldn = mv ? (can1 ? sd : id) - 1 : 0;
        const int eu = max((int)s_slu[can1 ? site : i], 0), ed = max((int)s_sld[can1 ? i : site], 0);
        T wu = T(0), wd = T(0);
        if (mv) {
            wu = Wup[lup * ldu + eu];
            wd = Wdn[ldn * ldd + ed];
#pragma unroll 4
            for (int q = 0; q < c; ++q) {
                wu += sAu[q * nsa + eu] * sBu[q * nmx + lup];
                wd += sAd[q * nsa + ed] * sBd[q * nmx + ldn];
            }
            const double acc_prob = abs2d(wu * wd);
            if (a.kernel_mode == KERNEL_REFERENCE)
                acc = (acc_prob >= 1.0 && r < zr) || (acc_prob < 1.0 && r < zr * acc_prob);
            else
                acc = r < acc_prob;
        }
        const bool dref = a.policy == POLICY_REFERENCE && (dmod + lane) % (unsigned)a.nocc == 0;
        const unsigned long long tmask = __ballot(mv && (acc || dref));
        const int tl = __ffsll((long long)tmask) - 1;   // lane of the terminal sweep, -1: none
        const long long next = tmask ? dbase + tl + 1 : (dbase + 64 < stop ? dbase + 64 : stop);
        if (a.outcomes && live && sw < next)
            a.outcomes[(size_t)w * a.tape_len + (sw - a.tape_base[w])] =
                (signed char)(pre ? OUT_PRE_REJECT : !(can1 || can2) ? OUT_NO_MOVE : acc ? OUT_ACCEPT : OUT_REJECT);
        n_moves += __popcll(__ballot(mv && sw < next));
        sweeps = next;
        if (!tmask) continue;
        const bool t_ref = __builtin_amdgcn_readlane((int)dref, tl) != 0;
        if (__builtin_amdgcn_readlane((int)acc, tl)) {
            const int ti = __builtin_amdgcn_readlane(i, tl), tsite = __builtin_amdgcn_readlane(site, tl);
            const bool tcan1 = __builtin_amdgcn_readlane((int)can1, tl) != 0;
            const int tlup = __builtin_amdgcn_readlane(lup, tl), tldn = __builtin_amdgcn_readlane(ldn, tl);
            const int teu = __builtin_amdgcn_readlane(eu, tl), ted = __builtin_amdgcn_readlane(ed, tl);
            const T twu = lane_t(wu, tl), twd = lane_t(wd, tl);
            ++n_acc;
            ++acc_since;
            // both spins' terms (append_terms): column and row of W0 plus the pending ones
            T cu = lane < ldu ? Wup[tlup * ldu + lane] : T(0), cd = lane < ldd ? Wdn[tldn * ldd + lane] : T(0);
            T ru = lane < nup ? Wup[lane * ldu + teu] : T(0), rd = lane < ndn ? Wdn[lane * ldd + ted] : T(0);
            const int la = lane < nsa ? lane : 0, lb = lane < nmx ? lane : 0;
#pragma unroll 2
            for (int q = 0; q < c; ++q) {
                cu += sAu[q * nsa + la] * sBu[q * nmx + tlup];
                cd += sAd[q * nsa + la] * sBd[q * nmx + tldn];
                ru += sAu[q * nsa + teu] * sBu[q * nmx + lb];
                rd += sAd[q * nsa + ted] * sBd[q * nmx + lb];
            }
            const T au = T(-1) / twu, ad = T(-1) / twd;
            if (lane < ldu) sAu[c * nsa + lane] = cu + (lane == teu ? T(1) : T(0));
            if (lane < ldd) sAd[c * nsa + lane] = cd + (lane == ted ? T(1) : T(0));
            if (lane == tlup) ru -= T(1);
            if (lane == tldn) rd -= T(1);
            if (lane < nup) sBu[c * nmx + lane] = au * ru;
            if (lane < ndn) sBd[c * nmx + lane] = ad * rd;
            zmu += z_delta_wave(s_bond, s_noff, s_nbr, s_kup, s_kdn, ti, tsite, lane);
            if (lane == 0) {
                const int Ku = tcan1 ? tsite : ti, Kd = tcan1 ? ti : tsite;   // targets; the sources are Kd and Ku
                s_slu[Kd] = (int16_t)teu; s_slu[Ku] = -1;
                s_sld[Ku] = (int16_t)ted; s_sld[Kd] = -1;
                s_kup[Kd] = 0; s_kup[Ku] = (int16_t)(tlup + 1);
                s_kdn[Ku] = 0; s_kdn[Kd] = (int16_t)(tldn + 1);
            }
            wave_sync();
            ++c;
            if (c == delay) {
                flush_w1<T, DMAX>(Wup, sAu, sBu, ldu, nsa, nmx, nup, c);
                flush_w1<T, DMAX>(Wdn, sAd, sBd, ldd, nsa, nmx, ndn, c);
                c = 0;
                ++n_flush;
                wave_sync();
            }
            pause = a.policy == POLICY_REFERENCE ? t_ref : a.policy == POLICY_EVERY_K && acc_since >= a.refresh_k;
        } else {
            pause = true;   // rejected move on a reference-cadence refresh sweep
        }
    }
    wave_sync();
    {
        int* ku = a.kup + (size_t)w * ns;
        int* kd = a.kdn + (size_t)w * ns;
        int* sg = a.slot + (size_t)w * 2 * ns;
        for (int t = lane; t < ns; t += 64) {
            ku[t] = s_kup[t];
            kd[t] = s_kdn[t];
            sg[t] = s_slu[t];
            sg[ns + t] = s_sld[t];
        }
        if (n_flush) {
            // W itself changes in a flush only
            copy_vec(reinterpret_cast<f32x4*>(reinterpret_cast<T*>(a.W) + (size_t)w * wstride),
                     reinterpret_cast<const f32x4*>(Wup), (int)(wstride * sizeof(T) / 16));
        }
    }
    if (c > 0) {
        const int dp = pend_ld(delay);
        T* gA = reinterpret_cast<T*>(a.A) + (size_t)w * 2 * nsa * dp;
        T* gB = reinterpret_cast<T*>(a.Bm) + (size_t)w * 2 * a.nmax * dp;
        // written as 16-byte vectors (slots c.. of the last one get zeros;
        // readers use the first c)
#pragma unroll
        for (int part = 0; part < 4; ++part) {
            const int n = part == 0 ? ldu : part == 1 ? ldd : part == 2 ? nup : ndn;
            const int st = part < 2 ? nsa : nmx;
            T* g = part < 2 ? gA + (size_t)part * nsa * dp : gB + (size_t)(part - 2) * a.nmax * dp;
            const T* d = part == 0 ? sAu : part == 1 ? sAd : part == 2 ? sBu : sBd;
            if (lane < n) {
#pragma unroll
                for (int p = 0; p < NVC; ++p) {
                    if (V * p < c) {
                        VT v;
                        T* e = reinterpret_cast<T*>(&v);
#pragma unroll
                        for (int u = 0; u < V; ++u) e[u] = V * p + u < c ? d[(V * p + u) * st + lane] : T(0);
                        reinterpret_cast<VT*>(g)[p * (part < 2 ? nsa : a.nmax) + lane] = v;
                    }
                }
            }
        }
    }
    if (lane == 0) {
        a.sweeps[w] = sweeps;
        a.npend[w] = c;
        a.acc_since[w] = acc_since;
        a.zmu[w] = zmu;
        // AT_END: a walker that reached refresh_k accepts during this call
        // finishes its sweeps and is refreshed after the launch
        if (pause || (a.policy == POLICY_AT_END && acc_since >= a.refresh_k)) {
            const int s = atomicAdd(a.refresh_count, 1);
            a.refresh_list[s] = w;
            a.counters[(size_t)w * CNT_SLOTS + CNT_PAUSES] += 1ull;
        }
        a.counters[(size_t)w * CNT_SLOTS + CNT_MOVES] += n_moves;
        a.counters[(size_t)w * CNT_SLOTS + CNT_ACCEPTED] += n_acc;
        a.counters[(size_t)w * CNT_SLOTS + CNT_FLUSHES] += n_flush;
        a.counters[(size_t)w * CNT_SLOTS + CNT_SWEEPS] += (unsigned long long)(sweeps - sweeps0);
    }
}

template <typename T, int D>
hipError_t launch_w1_d(const SweepArgs& a, int nw, hipStream_t s) {
    const size_t lds = sweep_w1_lds(sizeof(T), a.ns, a.nup, a.ndn, a.delay, a.nb);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_sweep_w1<T, D>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_sweep_w1<T, D>), dim3(nw), dim3(64), lds, s, a);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_w1(const SweepArgs& a, int nw, hipStream_t s) {
    if (a.delay <= 1) return launch_w1_d<T, 1>(a, nw, s);
    if (a.delay <= 4) return launch_w1_d<T, 4>(a, nw, s);
    if (a.delay <= 8) return launch_w1_d<T, 8>(a, nw, s);
    if (a.delay <= 12) return launch_w1_d<T, 12>(a, nw, s);
    return launch_w1_d<T, kMaxDelay>(a, nw, s);
}

}  // namespace kvmc
