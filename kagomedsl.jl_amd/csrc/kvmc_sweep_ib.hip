// Sweep kernel with implicit pending rows (gfx950): FP32 W with delayed
// updates, and FP64 W, real and complex, streamed from HBM, when a column of W
// has at most 256 rows.
//
// Carlo.sweep! (src/MonteCarlo.jl:538-607) with delayed Sherman-Morrison
// updates (update_W!, :279-292).
//
// The delayed update of k_sweep keeps, per accepted move q, a column A_q and
// a row B_q = alpha_q (W_cur[K_q, :] - e_l), and building B_q reads the row
// K_q of W: N single elements at a stride of ld, one cache line each.  Here
// the rows are never read at an accept.  With g_r = W0[K_r, :] - e_{l_r} (W0:
// W in HBM since the last flush) every row term is a combination of the g_r,
// B_q = sum_{r<=q} T[q][r] g_r, so
//
//   W_cur = W0 + sum_r At_r g_r^T,    At_r = sum_{q>=r} A_q T[q][r],
//
// and an accept updates the columns At in LDS only:
//   A_c   = W_cur[:, l] + e_K          (column l of W0 plus the terms),
//   At_r += A_c * alpha At_r[K]        for r < c,
//   At_c  = alpha A_c,                 alpha = -1 / W_cur[K, l].
// The flush applies W0 += sum_r At_r g_r^T with one wavefront per column of
// W, 16-byte units of the column per lane, and g_r[j] = W0[K_r, j] -
// delta(j, l_r) is read from the column itself (through the wavefront's LDS
// slot), so the rows cost no traffic.
//
// One wavefront of the workgroup (the evaluator) draws, decides and publishes
// the next accepted move; all of them apply it.  Every wavefront evaluating
// the same window (as k_sweep does) made four wavefronts issue the same
// instructions and gathers on four SIMDs.
//   - 64 draws at a time, one per lane, kept until the walker has passed them.
//   - Which of them reach the ratio (pre-reject, antiparallel bond) is
//     decided for all 64 at once; the first 8 that do fill 8 slots.
//   - A slot takes 8 lanes, 4 per spin.  W_cur[K, l] = W0[K, l] + sum_r
//     At_r[K] (W0[K_r, l] - delta(l, l_r)) needs c + 1 elements of column l:
//     each lane of the quad gathers a quarter of them (one memory round trip),
//     and the sum runs through the quad in the order of the terms.
//   - The accepted slot's gathers and coefficients At_r[K] are what the accept
//     needs of the column's term rows, so they are published with the move and
//     an accept costs one load of the two columns and two barriers.
//
// Bound by HBM: the flushes' reads and writes of W, plus about 30 % more for
// the gathers, an accept's columns and the launch's ends.  Measured per N
// sweeps of 8192 walkers at 216 rows: FP32, delay 12, 5.12 -> 4.25 ms (17.4 GB
// counted, 4.1 TB/s; a plain copy reaches 4.8); FP64 with immediate updates
// asked for, 74.1 -> 7.0 ms (delay 12 inside).  4096 walkers at 96 rows, FP64:
// 2.56 -> 0.68 ms; 2048 at 96 rows, complex FP64: 4.37 -> 1.38 ms.
//
// Between launches the pending terms are kept in the layout of k_sweep
// (pend_at) with A = At and B = g, so the local energy, the flush kernel,
// get_w and the refresh drift check read them unchanged; the rows g are
// gathered once at launch exit.  The term rows and labels (K_r, l_r) are kept
// beside them for the next launch.
#include "kvmc_kernels.hpp"

namespace kvmc {

// Columns of W per wavefront and iteration of the flush (the next ones are in
// flight besides).  Two cost registers and LDS; measured for one and two, us
// of sweep kernel per N sweeps: float 216 rows 4283, 4632, 96 rows 642, 701;
// double 96 rows 842, 689, 216 rows at delay 12 7451, 7041, at delay 8 9003,
// 10040; complex double 96 rows 1624, 1376.
template <typename T>
__host__ __device__ inline int ib_unroll(int nsa, int delay) {
    if (sizeof(T) == 4) return 1;
    return nsa <= 128 || (sizeof(T) == 8 && delay > 8) ? 2 : 1;
}
constexpr int kIbSlots = 8;     // proposals evaluated at a time
enum : int { IB_DONE = 0, IB_ACCEPT = 1, IB_ACCEPT_PAUSE = 2, IB_PAUSE = 3 };

// The move that the evaluator publishes.
template <typename T>
struct IbMove {
    T alpha[2];                 // -1 / W_cur[K, l] per spin
    int type, pad;
    int e[2], l[2];             // row of the target site, label
};

template <typename T>
__host__ __device__ inline size_t sweep_ib_lds(int ns, int nsa, int nwave, int delay, int nb) {
    const size_t nsp = (size_t)(ns + 3) / 4 * 4;
    const size_t b = 4 * nsp * sizeof(int16_t)                       // kappa and slot maps
                     + 2 * (size_t)delay * nsa * sizeof(T)             // At columns
                     + (size_t)nwave * ib_unroll<T>(nsa, delay) * nsa * sizeof(T)     // flush staging
                     + 4 * (size_t)kMaxDelay * sizeof(T)               // an accept's column elements and coefficients
                     + sizeof(IbMove<T>)
                     + 16 * sizeof(double)                             // reductions
                     + 64 * (sizeof(double) + sizeof(int)) + kIbSlots * sizeof(int)   // draws, slots
                     + 4 * (size_t)kMaxDelay * sizeof(int)             // term rows and labels
                     + (size_t)nb * sizeof(uint32_t) + (size_t)(ns + 1 + 2 * nb) * sizeof(uint16_t);
    return (b + 15) / 16 * 16;
}

// Value of lane perm[i] of each quad (DPP quad_perm), for any W element.
template <int CTRL>
__device__ __forceinline__ int quad_i(int v) { return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false); }
template <int CTRL>
__device__ __forceinline__ float quad_t(float v) { return __int_as_float(quad_i<CTRL>(__float_as_int(v))); }
template <int CTRL>
__device__ __forceinline__ double quad_t(double v) {
    const long long b = __double_as_longlong(v);
    const uint32_t lo = (uint32_t)quad_i<CTRL>((int)(uint32_t)b);
    const uint32_t hi = (uint32_t)quad_i<CTRL>((int)(uint32_t)((unsigned long long)b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <int CTRL>
__device__ __forceinline__ cf64 quad_t(cf64 v) { return cf64(quad_t<CTRL>(v.re), quad_t<CTRL>(v.im)); }
constexpr int kQuadUp = 0x90;     // lanes 0 0 1 2: the lane below
constexpr int kQuadLast = 0xFF;   // lanes 3 3 3 3

__device__ __forceinline__ float xor4(float v) { return __shfl_xor(v, 4, 64); }
__device__ __forceinline__ double xor4(double v) { return __shfl_xor(v, 4, 64); }
__device__ __forceinline__ cf64 xor4(cf64 v) { return cf64(__shfl_xor(v.re, 4, 64), __shfl_xor(v.im, 4, 64)); }

__device__ __forceinline__ float ib_mac(float v, float a, float b) { return v + a * b; }
__device__ __forceinline__ double ib_mac(double v, double a, double b) { return v + a * b; }
__device__ __forceinline__ cf64 ib_mac(cf64 v, cf64 a, cf64 b) {
    return cf64(v.re + a.re * b.re - a.im * b.im, v.im + a.re * b.im + a.im * b.re);
}

// Waves per SIMD the instance is compiled for.
template <typename T, int DMAX, int M> struct IbWaves { static constexpr int value = DMAX * M <= 16 ? 3 : 2; };
template <int DMAX, int M> struct IbWaves<float, DMAX, M> { static constexpr int value = DMAX <= 12 ? 4 : 3; };
template <int DMAX, int M> struct IbWaves<cf64, DMAX, M> { static constexpr int value = 2; };

// W elements per 16-byte unit of a column.
template <typename T> struct UnitOf { static constexpr int value = 16 / (int)sizeof(T); };

// W0 += sum_{r<c} At_r g_r^T for one spin (ld rows, N columns).  Wavefront
// `wave` of `nwave` takes columns wave, wave + nwave, ...; lane i holds the
// 16-byte units i, i + 64, ... (M of them) of the column.  K and L (uniform)
// are the terms' rows and labels.  Each loaded column is also written to the
// wavefront's own LDS slot (UNR columns of nsa elements), and g_r[j] =
// W0[K_r, j] - delta(j, l_r) is read back as an LDS broadcast before the
// column is updated.  A wavefront reads only what it wrote, in order, so no
// barrier.  The next columns are loaded while the current ones are updated.
// EX: c == DMAX, no test per term: with the tests every term is a branch
// with its own LDS round trip (L=12, FP32, delay 12: 128 us per flush of both
// spins).  Lanes past the column load its first unit and store nothing.
template <typename T, int DMAX, int M, int UNR, bool EX>
__device__ __forceinline__ void flush_ib(T* __restrict__ W0, const T* __restrict__ sAt, const int* sK,
                                         const int* sL, int ld, int nsa, int N, int c, T* s_stage) {
    constexpr int V = UnitOf<T>::value;
    using VT = typename VecT<T, V>::type;
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int nwave = (int)blockDim.x >> 6;
    const int nu = ld / V;
    T* stg = s_stage + wave * UNR * nsa;
    VT at[DMAX][M];
    int K[DMAX], L[DMAX], uo[M];
#pragma unroll
    for (int m = 0; m < M; ++m) uo[m] = lane + 64 * m < nu ? V * (lane + 64 * m) : 0;
#pragma unroll
    for (int q = 0; q < DMAX; ++q) {
        const int qc = EX || q < c ? q : 0;
#pragma unroll
        for (int m = 0; m < M; ++m) at[q][m] = *reinterpret_cast<const VT*>(sAt + (size_t)qc * nsa + uo[m]);
        K[q] = __builtin_amdgcn_readfirstlane(sK[qc]);
        L[q] = __builtin_amdgcn_readfirstlane(sL[qc]);
    }
    VT nx[UNR][M];
    auto load = [&](int j0) {
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const T* __restrict__ col = W0 + (size_t)min(j0 + u * nwave, N - 1) * ld;
#pragma unroll
            for (int m = 0; m < M; ++m) nx[u][m] = *reinterpret_cast<const VT*>(col + uo[m]);
        }
    };
    if (wave < N) load(wave);
    for (int j0 = wave; j0 < N; j0 += UNR * nwave) {
        VT v[UNR][M], d[UNR][M];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
#pragma unroll
            for (int m = 0; m < M; ++m) {
                v[u][m] = nx[u][m];
                d[u][m] = VT(0);
                // lanes past the column write its first unit once more
                *reinterpret_cast<VT*>(stg + u * nsa + uo[m]) = v[u][m];
            }
        }
        if (j0 + UNR * nwave < N) load(j0 + UNR * nwave);
#pragma unroll
        for (int q = 0; q < DMAX; ++q) {
            if (EX || q < c) {
#pragma unroll
                for (int u = 0; u < UNR; ++u) {
                    const T g = stg[u * nsa + K[q]] - (j0 + u * nwave == L[q] ? T(1) : T(0));
#pragma unroll
                    for (int m = 0; m < M; ++m) vmac(d[u][m], at[q][m], g);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const int j = j0 + u * nwave;
#pragma unroll
            for (int m = 0; m < M; ++m)
                if (lane + 64 * m < nu && j < N)
                    *reinterpret_cast<VT*>(W0 + (size_t)j * ld + uo[m]) = v[u][m] + d[u][m];
        }
    }
}

// W0 += A (alpha g)^T, one term applied at once with the arithmetic of
// k_sweep's immediate update (columns A in sA, row K of W0, label L).
template <typename T, int M>
__device__ __forceinline__ void apply_ib(T* __restrict__ W0, const T* __restrict__ sA, int K, int L, T alpha,
                                         int ld, int nsa, int N, T* s_stage) {
    constexpr int V = UnitOf<T>::value;
    using VT = typename VecT<T, V>::type;
    const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6, nwave = (int)blockDim.x >> 6;
    const int nu = ld / V;
    T* stg = s_stage + wave * nsa;
    for (int j = wave; j < N; j += nwave) {
        VT v[M];
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int u = lane + 64 * m;
            if (u < nu) {
                v[m] = *reinterpret_cast<const VT*>(W0 + (size_t)j * ld + V * u);
                *reinterpret_cast<VT*>(stg + V * u) = v[m];
            }
        }
        wave_sync();
        T b = stg[K];
        if (j == L) b -= T(1);
        b = alpha * b;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int u = lane + 64 * m;
            if (u < nu) {
                vmac(v[m], *reinterpret_cast<const VT*>(sA + V * u), b);
                *reinterpret_cast<VT*>(W0 + (size_t)j * ld + V * u) = v[m];
            }
        }
    }
}

template <typename T, int DMAX, int M, int UNR, bool EX>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(IbWaves<T, DMAX, M>::value)))
k_sweep_ib(SweepArgs a) {
    extern __shared__ __align__(16) unsigned char lds[];
    constexpr int V = UnitOf<T>::value;
    using VT = typename VecT<T, V>::type;
    const int w = a.walker0 + (int)blockIdx.x;
    const int ns = a.ns, nup = a.nup, ndn = a.ndn, nb = a.nb, nmax = a.nmax;
    const int nsp = round_up(ns, 4);
    const int nsa = w_nsa(ns, nup, ndn);
    const int delay = a.delay;
    const int tid = (int)threadIdx.x, bd = (int)blockDim.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwave = bd >> 6;
    int16_t* s_kup = reinterpret_cast<int16_t*>(lds);
    int16_t* s_kdn = s_kup + nsp;
    int16_t* s_slu = s_kdn + nsp;                     // site -> row of W_up (-1: occupied)
    int16_t* s_sld = s_slu + nsp;
    T* s_At = reinterpret_cast<T*>(s_sld + nsp);      // [2][delay][nsa] (8 nsp bytes: 16-byte aligned)
    T* s_stage = s_At + 2 * delay * nsa;              // [nwave][UNR][nsa] flush staging
    T* s_g = s_stage + nwave * UNR * nsa;       // [2][kMaxDelay] g_q[l] of an accept
    T* s_tc = s_g + 2 * kMaxDelay;                    // [2][kMaxDelay] alpha At_q[K] of an accept
    IbMove<T>* s_mv = reinterpret_cast<IbMove<T>*>(s_tc + 2 * kMaxDelay);
    double* s_red = reinterpret_cast<double*>(s_mv + 1);
    double* s_du = s_red + 16;                        // [64] u of the draws held
    uint32_t* s_db = reinterpret_cast<uint32_t*>(s_du + 64);   // [64] their bonds' sites, packed
    int* s_sf = reinterpret_cast<int*>(s_db + 64);    // [kIbSlots] a slot's draw lane and flags
    int* s_K = s_sf + kIbSlots;                       // [2][kMaxDelay] term rows
    int* s_L = s_K + 2 * kMaxDelay;                   // [2][kMaxDelay] term labels
    uint32_t* s_bond = reinterpret_cast<uint32_t*>(s_L + 2 * kMaxDelay);
    uint16_t* s_noff = reinterpret_cast<uint16_t*>(s_bond + nb);
    uint16_t* s_nbr = s_noff + ns + 1;

    const size_t wstride = w_stride(ns, nup, ndn);
    const int ldu = w_ld(ns, nup), ldd = w_ld(ns, ndn);
    T* const Wup = reinterpret_cast<T*>(a.W) + (size_t)w * wstride;
    T* const Wdn = Wup + w_off_dn(ns, nup);
    const int* const slot_g = a.slot + (size_t)w * 2 * ns;
    const int dp = pend_ld(delay);
    T* sAu = s_At;
    T* sAd = s_At + delay * nsa;

    long long sweeps = a.sweeps[w];
    const long long stop = a.stop[w];
    if (sweeps >= stop || *a.failed != 0x7fffffff) return;
    int c = a.npend[w];
    const int c_in = c;
    int acc_since = a.acc_since[w];
    // FP64: a walker whose last refresh found a nearly singular tildeU (its W
    // is large, and an update cancels most of its digits) updates W at once:
    // pending terms would round differently there, and by more than elsewhere.
    const bool at_once = sizeof(T) > 4 && c == 0 && (a.stiff[2 * w] | a.stiff[2 * w + 1]) != 0;

    // The copies into LDS are unrolled so that several loads are in flight
    // before the first store waits on them.
#pragma unroll 2
    for (int t = tid; t < ns; t += bd) {
        s_kup[t] = (int16_t)a.kup[(size_t)w * ns + t];
        s_kdn[t] = (int16_t)a.kdn[(size_t)w * ns + t];
        s_slu[t] = (int16_t)slot_g[t];
        s_sld[t] = (int16_t)slot_g[ns + t];
    }
    constexpr int NVC = (DMAX + V - 1) / V;   // planes of terms (dp a multiple of 4 elements)
    if (c > 0) {
        const T* gA = reinterpret_cast<const T*>(a.A) + (size_t)w * 2 * nsa * dp;
        const int* pt = a.pterm + (size_t)w * 2 * kMaxDelay * 2;
#pragma unroll 2
        for (int t = tid; t < 2 * nsa; t += bd) {
            const int sp = t >= nsa ? 1 : 0;
            T* d = s_At + sp * delay * nsa + (t - sp * nsa);
            const VT* g = reinterpret_cast<const VT*>(gA + (size_t)sp * nsa * dp) + (t - sp * nsa);
            VT v[NVC];
#pragma unroll
            for (int p = 0; p < NVC; ++p)
                if (V * p < c) v[p] = g[p * nsa];
#pragma unroll
            for (int p = 0; p < NVC; ++p) {
                const T* e = reinterpret_cast<const T*>(&v[p]);
#pragma unroll
                for (int u = 0; u < V; ++u)
                    if (V * p + u < c) d[(V * p + u) * nsa] = e[u];
            }
        }
        for (int t = tid; t < 2 * c; t += bd) {
            const int sp = t / c, q = t % c;
            s_K[sp * kMaxDelay + q] = pt[(sp * kMaxDelay + q) * 2];
            s_L[sp * kMaxDelay + q] = pt[(sp * kMaxDelay + q) * 2 + 1];
        }
    }
#pragma unroll 4
    for (int b = tid; b < nb; b += bd) {
        const int2 bb = a.bonds[b];
        s_bond[b] = (uint32_t)bb.x | ((uint32_t)bb.y << 16);
    }
#pragma unroll 2
    for (int t = tid; t <= ns; t += bd) s_noff[t] = (uint16_t)a.nbr_off[t];
    const int nnbr = a.nbr_off[ns];
#pragma unroll 4
    for (int t = tid; t < nnbr; t += bd) s_nbr[t] = (uint16_t)a.nbr[t];
    __syncthreads();
    int zmu;
    {
        double part = 0.0;
        for (int b = tid; b < nb; b += bd) {
            const uint32_t bp = s_bond[b];
            const int i = (int)(bp & 0xffffu), j = (int)(bp >> 16);
            part += (s_kup[i] != 0 && s_kdn[j] != 0) || (s_kup[j] != 0 && s_kdn[i] != 0);
        }
        zmu = (int)block_sum_double(part, s_red);
    }
    const double zmax = (double)nb;
    const int nocc = a.nocc;
    const bool has_out = a.outcomes != nullptr;
    // kept by the evaluator alone: sweeps, zmu, n_moves and the draws; by
    // every wavefront: c, acc_since and the other counts
    unsigned long long n_moves = 0, n_acc = 0, n_flush = 0;
    const long long sweeps0 = sweeps;
    bool pause = false;
    // walkers that share a CU (blocks apart by 8, the XCDs, times a power of
    // two) let wavefronts on different SIMDs evaluate
    const int ev = (int)(((blockIdx.x >> 3) + (blockIdx.x >> 8)) % (unsigned)nwave);
    long long dbase = sweeps - 64;   // the draws held are those of sweeps dbase .. dbase + 63
    // dbase modulo nocc; the first window adds 64
    unsigned dmod = (unsigned)((sweeps + (long long)nocc * 64 - 64) % nocc);
    constexpr int DQ = (DMAX + 3) / 4;   // terms per lane of a quad
    const int quad = lane & 3, spin = (lane >> 2) & 1, slot = lane >> 3;

    for (;;) {
        if (wave == ev) {
            int type = IB_DONE;
            while (sweeps < stop) {
                if (sweeps >= dbase + 64) {
                    dbase = sweeps;
                    const long long sw = dbase + lane;
                    int bidx = 0;
                    double u = 1.0;
                    if (sw < stop) {
                        const auto k = late_args();
                        if (k->tape_u) {
                            const long long tidx = (size_t)w * k->tape_len + (sw - k->tape_base[w]);
                            u = k->tape_u[tidx];
                            bidx = k->tape_bond[tidx];
                        } else {
                            sweep_draws(k->seed, (uint32_t)w, sw, nb, &u, &bidx);
                        }
                    }
                    s_du[lane] = u;
                    s_db[lane] = s_bond[bidx];
                    dmod = (dmod + 64) % (unsigned)nocc;
                }
                const double zr = (double)zmu / zmax;
                const long long sw = dbase + lane;
                const bool live = sw >= sweeps && sw < stop;
                const double r = s_du[lane];
                const uint32_t db = s_db[lane];
                const int di = (int)(db & 0xffffu), dj = (int)(db >> 16);
                // a sweep on which the reference cadence refreshes
                const bool dref = a.policy == POLICY_REFERENCE && (dmod + lane) % (unsigned)nocc == 0;
                const bool pre = a.kernel_mode == KERNEL_REFERENCE && r > zr;
                const bool can1 = s_kup[di] != 0 && s_kdn[dj] != 0;
                const bool can2 = s_kup[dj] != 0 && s_kdn[di] != 0;
                const bool mv = live && !pre && (can1 || can2);
                const unsigned long long mvmask = __ballot(mv);
                const int nmv = __popcll(mvmask);
                long long next = dbase + 64 < stop ? dbase + 64 : stop;
                bool t_acc = false, t_term = false, t_ref = false;
                if (nmv) {
                    const int rank = __popcll(mvmask & ((1ull << lane) - 1ull));
                    if (mv && rank < kIbSlots) s_sf[rank] = lane | (can1 ? 256 : 0) | (dref ? 512 : 0);
                    wave_sync();
                    const int nslot = nmv < kIbSlots ? nmv : kIbSlots;
                    const bool in = slot < nslot;
                    const int sl = in ? slot : 0;
                    const int sf = s_sf[sl];
                    const double ru = s_du[sf & 63];
                    const int si = (int)s_db[sf & 63];
                    const int i = si & 0xffff, j = (int)((unsigned)si >> 16);
                    const bool one = (sf & 256) != 0;
                    // flag = 1: up moves i -> j, down moves j -> i.  The target
                    // is empty for the moving spin; max() keeps a walker with
                    // an inconsistent state (failed refresh) inside W.
                    const int src = (one == (spin == 0)) ? i : j, K = (one == (spin == 0)) ? j : i;
                    const int l = (spin ? (int)s_kdn[src] : (int)s_kup[src]) - 1;
                    const int e = max(spin ? (int)s_sld[K] : (int)s_slu[K], 0);
                    const T* col = spin ? Wdn + (size_t)l * ldd : Wup + (size_t)l * ldu;
                    const T* At = s_At + spin * delay * nsa + e;
                    // every gather is issued before any is used: term slots
                    // past c re-read row e, in bounds
                    T g[DQ], s[DQ];
#pragma unroll
                    for (int k = 0; k < DQ; ++k) {
                        const int q = quad * DQ + k;
                        g[k] = col[q < c ? s_K[spin * kMaxDelay + q] : e];
                    }
                    T v = col[e];
#pragma unroll
                    for (int k = 0; k < DQ; ++k) {
                        const int q = quad * DQ + k;
                        s[k] = q < c ? At[q * nsa] : T(0);
                        const bool own = q < c && s_L[spin * kMaxDelay + (q < c ? q : 0)] == l;
                        g[k] = g[k] - (own ? T(1) : T(0));
                    }
                    // the sum in the order of the terms, through the quad
#pragma unroll
                    for (int step = 0; step < 4; ++step) {
                        T t = v;
#pragma unroll
                        for (int k = 0; k < DQ; ++k) {
                            const T t1 = ib_mac(t, s[k], g[k]);
                            t = quad * DQ + k < c ? t1 : t;
                        }
                        if (step < 3) {
                            const T up = quad_t<kQuadUp>(t);
                            v = quad == step + 1 ? up : v;
                        } else {
                            v = quad_t<kQuadLast>(t);
                        }
                    }
                    const T x = xor4(v);
                    const double acc_prob = abs2d(spin ? x * v : v * x);
                    bool acc;
                    if (a.kernel_mode == KERNEL_REFERENCE)
                        acc = (acc_prob >= 1.0 && ru < zr) || (acc_prob < 1.0 && ru < zr * acc_prob);
                    else
                        acc = ru < acc_prob;
                    const bool term = acc || (sf & 512);
                    const unsigned long long tmask = __ballot(in && term && (lane & 7) == 0);
                    if (tmask) {
                        const int tl = __ffsll((long long)tmask) - 1;   // lane 0 of the terminal slot
                        n_moves += (tl >> 3) + 1;
                        const int tf = __builtin_amdgcn_readlane(sf, tl);
                        next = dbase + (tf & 255) + 1;
                        t_term = true;
                        t_ref = (tf & 512) != 0;
                        t_acc = __builtin_amdgcn_readlane((int)acc, tl) != 0;
                        if (t_acc) {
                            const int tsi = __builtin_amdgcn_readlane(si, tl);
                            const int ti = tsi & 0xffff, tj = (int)((unsigned)tsi >> 16);
                            const bool tone = (tf & 256) != 0;
                            if (slot == (tl >> 3)) {
                                const T al = T(-1) / v;
#pragma unroll
                                for (int k = 0; k < DQ; ++k) {
                                    const int q = quad * DQ + k;
                                    if (q < c) {
                                        s_g[spin * kMaxDelay + q] = g[k];
                                        s_tc[spin * kMaxDelay + q] = al * s[k];
                                    }
                                }
                                if (quad == 0) {
                                    s_mv->alpha[spin] = al;
                                    s_mv->e[spin] = e;
                                    s_mv->l[spin] = l;
                                    s_K[spin * kMaxDelay + c] = e;
                                    s_L[spin * kMaxDelay + c] = l;
                                }
                            }
                            zmu += z_delta_wave(s_bond, s_noff, s_nbr, s_kup, s_kdn, ti, tj, lane);
                            const int eu = __builtin_amdgcn_readlane(e, tl), ed = __builtin_amdgcn_readlane(e, tl + 4);
                            const int lu = __builtin_amdgcn_readlane(l, tl), ldl = __builtin_amdgcn_readlane(l, tl + 4);
                            if (lane == 0) {
                                const int Ku = tone ? tj : ti, Kd = tone ? ti : tj;   // targets; the sources are Kd and Ku
                                s_slu[Kd] = (int16_t)eu; s_slu[Ku] = -1;
                                s_sld[Ku] = (int16_t)ed; s_sld[Kd] = -1;
                                s_kup[Kd] = 0; s_kup[Ku] = (int16_t)(lu + 1);
                                s_kdn[Ku] = 0; s_kdn[Kd] = (int16_t)(ldl + 1);
                            }
                            wave_sync();
                        }
                    } else {
                        n_moves += nslot;
                        if (nmv > kIbSlots) next = dbase + __builtin_amdgcn_readfirstlane(s_sf[kIbSlots - 1] & 255) + 1;
                    }
                }
                if (has_out && live && sw < next)
                    late_args()->outcomes[(size_t)w * late_args()->tape_len + (sw - late_args()->tape_base[w])] =
                        (signed char)(pre ? OUT_PRE_REJECT : !(can1 || can2) ? OUT_NO_MOVE
                                      : (t_acc && sw + 1 == next) ? OUT_ACCEPT : OUT_REJECT);
                sweeps = next;
                if (t_term) {
                    bool due = true;   // a rejected move on a reference-cadence refresh sweep
                    if (t_acc)
                        due = a.policy == POLICY_REFERENCE ? t_ref
                            : a.policy == POLICY_EVERY_K ? acc_since + 1 >= a.refresh_k
                                                         : false;   // AT_END: listed at exit
                    type = t_acc ? (due ? IB_ACCEPT_PAUSE : IB_ACCEPT) : IB_PAUSE;
                    break;
                }
            }
            if (lane == 0) s_mv->type = type;
        }
        __syncthreads();
        const int type = __builtin_amdgcn_readfirstlane(s_mv->type);
        if (type == IB_DONE) break;
        if (type == IB_PAUSE) { pause = true; break; }
        {
            const int eu = __builtin_amdgcn_readfirstlane(s_mv->e[0]), ed = __builtin_amdgcn_readfirstlane(s_mv->e[1]);
            const int lu = __builtin_amdgcn_readfirstlane(s_mv->l[0]), ldl = __builtin_amdgcn_readfirstlane(s_mv->l[1]);
            // A_c = W_cur[:, l] + e_K, one row per thread and spin (blockDim.x
            // >= nsa); each thread updates only its own row of At
            // (opaque: the addresses of the DMAX rows are not kept across the loop)
            const int row = opaque_v(tid), st = opaque_s(nsa);
            const bool ru = row < ldu, rd = row < ldd;
            T Au = ru ? Wup[(size_t)lu * ldu + row] : T(0);
            T Ad = rd ? Wdn[(size_t)ldl * ldd + row] : T(0);
            const T au = s_mv->alpha[0], ad = s_mv->alpha[1];
            if (at_once) {
                // c == 0: the columns as they are, then one streaming pass each
                if (row < st) {
                    sAu[row] = ru ? Au + (row == eu ? T(1) : T(0)) : T(0);
                    sAd[row] = rd ? Ad + (row == ed ? T(1) : T(0)) : T(0);
                }
                __syncthreads();
                apply_ib<T, M>(Wup, sAu, eu, lu, au, ldu, nsa, nup, s_stage);
                apply_ib<T, M>(Wdn, sAd, ed, ldl, ad, ldd, nsa, ndn, s_stage);
            } else if (row < st) {
#pragma unroll 4
                for (int q = 0; q < c; ++q) {
                    Au = ib_mac(Au, sAu[q * st + row], s_g[q]);
                    Ad = ib_mac(Ad, sAd[q * st + row], s_g[kMaxDelay + q]);
                }
                Au += row == eu ? T(1) : T(0);
                Ad += row == ed ? T(1) : T(0);
#pragma unroll 4
                for (int q = 0; q < c; ++q) {
                    if (ru) sAu[q * st + row] = ib_mac(sAu[q * st + row], Au, s_tc[q]);
                    if (rd) sAd[q * st + row] = ib_mac(sAd[q * st + row], Ad, s_tc[kMaxDelay + q]);
                }
                sAu[c * st + row] = ru ? au * Au : T(0);
                sAd[c * st + row] = rd ? ad * Ad : T(0);
            }
        }
        ++n_acc;
        ++acc_since;
        c += at_once ? 0 : 1;
        n_flush += at_once ? 1 : 0;
        __syncthreads();
        if (c == delay) {
#pragma clang loop unroll(disable)
            for (int sp = 0; sp < 2; ++sp)
                flush_ib<T, DMAX, M, UNR, EX>(sp ? Wdn : Wup, s_At + sp * delay * nsa, s_K + sp * kMaxDelay,
                                     s_L + sp * kMaxDelay, sp ? ldd : ldu, nsa, sp ? ndn : nup, c, s_stage);
            c = 0;
            ++n_flush;
            __syncthreads();
        }
        if (type == IB_ACCEPT_PAUSE) { pause = true; break; }
    }
    __syncthreads();
    const auto k = late_args();
    if (n_acc) {
        int* const slot_o = k->slot + (size_t)w * 2 * ns;
        for (int t = tid; t < ns; t += bd) {
            k->kup[(size_t)w * ns + t] = s_kup[t];
            k->kdn[(size_t)w * ns + t] = s_kdn[t];
            slot_o[t] = s_slu[t];
            slot_o[ns + t] = s_sld[t];
        }
    }
    // the terms are kept also for a walker due a refresh: the refresh may
    // measure the drift of the carried W first, and a walker whose refresh
    // fails keeps a W consistent with its configuration.  Without an accepted
    // move they are in memory as they were, and without a flush so are the
    // rows of the terms that the launch began with (a call of one sweep, FP64,
    // 8192 walkers at 216 rows: 831 us with all of them gathered and written,
    // 336 now; at 96 rows 255 and 130).
    if (c > 0 && n_acc) {
        const int q0 = n_flush ? 0 : c_in / V * V;   // planes of rows before it are left
        T* gA = reinterpret_cast<T*>(k->A) + (size_t)w * 2 * nsa * dp;
        T* gB = reinterpret_cast<T*>(k->Bm) + (size_t)w * 2 * nmax * dp;
        int* pt = k->pterm + (size_t)w * 2 * kMaxDelay * 2;
        // written as 16-byte vectors (slots c.. of the last one get zeros;
        // readers use the first c); all of a label's gathers are issued
        // before the first is stored
        for (int t = tid; t < 2 * nsa; t += bd) {
            const int sp = t >= nsa ? 1 : 0;
            const T* d = s_At + sp * delay * nsa + (t - sp * nsa);
            VT* g = reinterpret_cast<VT*>(gA + (size_t)sp * nsa * dp) + (t - sp * nsa);
#pragma unroll
            for (int p = 0; p < NVC; ++p) {
                if (V * p < c) {
                    VT v;
                    T* e = reinterpret_cast<T*>(&v);
#pragma unroll
                    for (int u = 0; u < V; ++u) e[u] = V * p + u < c ? d[(V * p + u) * nsa] : T(0);
                    g[p * nsa] = v;
                }
            }
        }
        // the rows g_q = W0[K_q, :] - e_{l_q}, one label per thread
        for (int t = tid; t < 2 * nmax; t += bd) {
            const int sp = t >= nmax ? 1 : 0, l = t - sp * nmax;
            if (l >= (sp ? ndn : nup)) continue;
            const T* col = (sp ? Wdn : Wup) + (size_t)l * (sp ? ldd : ldu);
            __align__(16) T v[V * NVC];
#pragma unroll
            for (int q = 0; q < V * NVC; ++q)
                v[q] = q >= q0 && q < c ? col[s_K[sp * kMaxDelay + q]] - (l == s_L[sp * kMaxDelay + q] ? T(1) : T(0)) : T(0);
            VT* g = reinterpret_cast<VT*>(gB + (size_t)sp * nmax * dp) + l;
#pragma unroll
            for (int p = 0; p < NVC; ++p)
                if (V * p >= q0 && V * p < c) g[p * nmax] = *reinterpret_cast<const VT*>(&v[V * p]);
        }
        for (int t = tid; t < 2 * c; t += bd) {
            const int sp = t / c, q = t % c;
            pt[(sp * kMaxDelay + q) * 2] = s_K[sp * kMaxDelay + q];
            pt[(sp * kMaxDelay + q) * 2 + 1] = s_L[sp * kMaxDelay + q];
        }
    }
    if (wave == ev && lane == 0) {
        k->sweeps[w] = sweeps;
        k->npend[w] = c;
        k->acc_since[w] = acc_since;
        k->zmu[w] = zmu;
        if (pause || (k->policy == POLICY_AT_END && acc_since >= k->refresh_k)) {
            const int s = atomicAdd(k->refresh_count, 1);
            k->refresh_list[s] = w;
            k->counters[(size_t)w * CNT_SLOTS + CNT_PAUSES] += 1ull;
        }
        k->counters[(size_t)w * CNT_SLOTS + CNT_MOVES] += n_moves;
        k->counters[(size_t)w * CNT_SLOTS + CNT_ACCEPTED] += n_acc;
        k->counters[(size_t)w * CNT_SLOTS + CNT_FLUSHES] += n_flush;
        k->counters[(size_t)w * CNT_SLOTS + CNT_SWEEPS] += (unsigned long long)(sweeps - sweeps0);
    }
}

int sweep_ib_block(int ns, int nup, int ndn) {
    const int nsa = w_nsa(ns, nup, ndn);
    return nsa <= 64 ? 64 : nsa <= 128 ? 128 : nsa <= 192 ? 192 : 256;
}

static size_t ib_lds(int prec, int cplx, int ns, int nup, int ndn, int delay, int nb) {
    const int nsa = w_nsa(ns, nup, ndn), nwave = sweep_ib_block(ns, nup, ndn) / 64;
    if (prec == 1) return sweep_ib_lds<float>(ns, nsa, nwave, delay, nb);
    return cplx ? sweep_ib_lds<cf64>(ns, nsa, nwave, delay, nb) : sweep_ib_lds<double>(ns, nsa, nwave, delay, nb);
}

bool sweep_ib_supported(int prec, int cplx, int ns, int nup, int ndn, int delay, int nb) {
    const int ld = w_ld(ns, nup) > w_ld(ns, ndn) ? w_ld(ns, nup) : w_ld(ns, ndn);
    // complex: a lane holds the terms of 2 or 4 rows, 4 registers each, and
    // more than 8 of them would spill.  Such delays run on k_sweep: us of sweep
    // kernel per N sweeps there at 12 terms and here at 8, 1024 walkers at 96
    // rows 740 and 541, 512 at 150 rows 1384 and 1067.
    const int dmax = prec == 0 && cplx ? 8 : kMaxDelay;
    if (prec == 1 && cplx) return false;
    return delay > 1 && delay <= dmax && ld <= 256 && !sweep_resident(w_elem_bytes(prec, cplx), ns, nup, ndn) &&
           ib_lds(prec, cplx, ns, nup, ndn, delay, nb) <= 160 * 1024;
}

int sweep_ib_fp64_delay(int cplx, int ns, int nup, int ndn, int nb) {
    // Fewer flushes against LDS (walkers per CU) and the terms a measurement
    // reads.  us of sweep kernel per N sweeps at delays 8 and 12: 216 rows
    // 9003, 7041 (74090 with immediate updates), its local energies 182, 230;
    // 150 rows 1103, 1154; 96 rows 689, 664 (2563 immediate).  Complex: 4 is
    // slower everywhere (96 rows 1910 against 1376, 4371 immediate; 216 rows,
    // 512 walkers, 3306 against 2420, 11519 immediate; 150 rows 1065, 3216
    // immediate), also where 8 terms spill 10 registers (above 128 rows).
    const int d = !cplx && w_nsa(ns, nup, ndn) > 192 ? 12 : 8;
    return sweep_ib_supported(0, cplx, ns, nup, ndn, d, nb) ? d : 1;
}

template <typename T, int D, int M, int UNR, bool EX>
static hipError_t launch_ib_d(const SweepArgs& a, int nw, size_t lds, hipStream_t s) {
    const void* fn = reinterpret_cast<const void*>(&k_sweep_ib<T, D, M, UNR, EX>);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((k_sweep_ib<T, D, M, UNR, EX>), dim3(nw), dim3(sweep_ib_block(a.ns, a.nup, a.ndn)), lds, s, a);
    return hipGetLastError();
}

// Exact instances for delays 4, 8, 12 and 16 (complex: 4 and 8); any other
// delay runs the next larger of 8 and 16 with a test per term.
template <typename T, int M>
static hipError_t launch_ib_m(const SweepArgs& a, int nw, size_t lds, hipStream_t s) {
    constexpr int U8 = sizeof(T) > 4 && M * UnitOf<T>::value <= 2 ? 2 : 1;   // ib_unroll at delays <= 8
    constexpr int U16 = sizeof(T) == 8 ? 2 : 1;                                 // and above
    if (a.delay == 4) return launch_ib_d<T, 4, M, U8, true>(a, nw, lds, s);
    if (a.delay == 8) return launch_ib_d<T, 8, M, U8, true>(a, nw, lds, s);
    if (a.delay < 8) return launch_ib_d<T, 8, M, U8, false>(a, nw, lds, s);
    if constexpr (!is_cplx<T>::value) {
        if (a.delay == 12) return launch_ib_d<T, 12, M, U16, true>(a, nw, lds, s);
        if (a.delay == 16) return launch_ib_d<T, 16, M, U16, true>(a, nw, lds, s);
        return launch_ib_d<T, 16, M, U16, false>(a, nw, lds, s);
    }
    return hipErrorInvalidValue;   // sweep_ib_supported
}

template <typename T>
static hipError_t launch_ib(const SweepArgs& a, int nw, size_t lds, hipStream_t s) {
    constexpr int V = UnitOf<T>::value;     // rows per 16-byte unit: a lane's unit covers 64 V rows of a column
    if constexpr (sizeof(T) > 4) {
        if (w_nsa(a.ns, a.nup, a.ndn) <= 128) return launch_ib_m<T, 2 / V>(a, nw, lds, s);
    }
    return launch_ib_m<T, 4 / V>(a, nw, lds, s);
}

hipError_t launch_sweep_ib(int prec, int cplx, const SweepArgs& a, int nw, hipStream_t s) {
    const size_t lds = ib_lds(prec, cplx, a.ns, a.nup, a.ndn, a.delay, a.nb);
    if (prec == 1) return launch_ib<float>(a, nw, lds, s);
    return cplx ? launch_ib<cf64>(a, nw, lds, s) : launch_ib<double>(a, nw, lds, s);
}

}  // namespace kvmc
