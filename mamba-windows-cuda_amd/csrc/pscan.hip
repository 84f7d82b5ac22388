// Standalone first-order linear recurrence ("parallel_scan_fn") for gfx950.
//
// Semantics: parallel_scan_ref (pscan.py:153-171): over the middle axis of
// [nseq][L][ncols], H_0 = X_0 (A_0 unused), H_t = A_t*H_{t-1} + X_t, with fp32
// accumulation; and its adjoint (replacing PScan.backward, pscan.py:97-136,
// whose math is wrong for L >= 4): G_t = dH_t + A_{t+1}*G_{t+1}, dX = G,
// dA_t = G_t*H_{t-1} for t >= 1 and dA_0 = 0.
//
// Design: one pass over HBM (12 B/element forward, 20 B/element backward).
// A tile is TS consecutive steps x CW threads across; each thread owns one column
// (a pair of them in wide 16-bit scans) and RUN consecutive steps held in VGPRs. Thread runs are combined inside the
// tile through LDS; tiles along L are chained with a decoupled look-back:
// each tile publishes its aggregate map h -> a*h + b per column, then its
// inclusive prefix once known, as 64-bit (status << 32 | fp32 bits) words so
// a single relaxed agent-scope atomic carries both the flag and the value
// (no cache-wide release/acquire fences). Tiles are taken from an atomic
// ticket (see ticket_chains), so every predecessor of a waiting tile is
// already resident, and each spin is bounded so a lost update can never hang
// the device. A wait that runs out of spins sets the workspace's error word (read by mwc_pscan_status) and
// gives the tile a NaN prefix, so its outputs, and every later tile's, are NaN
// rather than a plausible wrong value.
//
// Range: the coefficient of a map over many steps is a product that leaves fp32 long before the states do (1.42^256
// overflows, 0.66^256 is 0), and inf * 0 is NaN. So such products carry an exponent of their own, from a thread's run
// to the look-back: states of 0, tiny ones and infinite ones pass through any number of finite coefficients as they do
// step by step. Where no product leaves fp32 the results are the same bit for bit; narrow calls take 0.1 to 0.7 us
// longer ((700, 300, 32) fp16 13.3 -> 14.0 us, (2048, 300, 32) 27.1 -> 27.8), a long one with exponents in every tile
// 1.5 us ((1, 30000, 16) fp16 14.6 -> 16.1); large calls and those over wide rows are unchanged.
#include <algorithm>

#include "common.h"
#include "launch.h"

namespace mwc {

namespace {

constexpr int kThreads = 256;
// Steps of a tile of cw thread columns. Narrow tiles are longer, for fewer look-backs: (3072, 1024, 16) fp16 71 and
// 134 us (forward, adjoint) against 80 and 139 with 128, (1, 30000, 16) 15 us against 19; 512 steps at 8 columns made
// (20000, 200, 8) fp16 56 us instead of 40.
constexpr int tile_steps(int cw) { return cw <= 16 ? 256 : 128; }
// Waves a SIMD that the kernels are compiled to fit. 80 VGPRs leave 6, which narrow forwards would exceed by two.
constexpr int scan_waves(int cw, bool rev) { return cw == 64 ? 3 : cw == 8 ? 8 : rev ? 5 : 6; }
constexpr uint32_t kStAgg = 1, kStInc = 2;
constexpr int kTicketStride = 16;  // words: a ticket has a cache line of its own
// Column blocks (chains of tiles along L) that share a ticket. One ticket for all tiles serves one in about 12 ns, which
// bound calls of many small tiles: (384, 1024, 16) fp32 45 -> 17 us, (1, 4096, 512) 13.8 -> 11.8. Long calls over wide
// rows share one by up to 64: with one each the blocks of a row drift apart and rows are no longer read whole,
// (4, 65536, 1024) fp32 673 us, and 635 with one a sequence, against 625.
int ticket_chains(int cw, int64_t ntiles) { return cw < 64 || ntiles <= 1024 ? 1 : 64; }

struct PscanGeom {
    int cw, vec, ncolblk, nltile;
    int gchains;      // column blocks of a ticket group
    int64_t ngroups;  // ticket groups
    int64_t nblocks;  // workgroups
    size_t flags_offset, bytes;
};

// Workspace: the error word's line, the tickets, the flags. vec: columns per thread.
PscanGeom geom(int64_t nseq, int64_t seqlen, int64_t ncols, int vec) {
    PscanGeom g;
    const int64_t lanes = ncols / vec;
    g.vec = vec;
    g.cw = lanes <= 8 ? 8 : lanes <= 16 ? 16 : lanes <= 32 ? 32 : 64;
    g.ncolblk = (int)((lanes + g.cw - 1) / g.cw);
    g.nltile = (int)((seqlen + tile_steps(g.cw) - 1) / tile_steps(g.cw));
    const bool one = g.nltile == 1;  // no tickets and no flags: the error word is all that such a scan uses
    const int64_t nchains = nseq * g.ncolblk, most = one ? 1 : ticket_chains(g.cw, nchains * g.nltile);
    g.ngroups = (nchains + most - 1) / most;
    g.gchains = (int)((nchains + g.ngroups - 1) / g.ngroups);
    g.ngroups = (nchains + g.gchains - 1) / g.gchains;
    g.nblocks = g.ngroups * g.gchains * g.nltile;
    g.flags_offset = (size_t)(1 + (one ? 0 : g.ngroups)) * kTicketStride * sizeof(unsigned);
    g.bytes = g.flags_offset + (one ? 0 : (size_t)nchains * g.nltile * g.cw * vec * 2 * sizeof(uint64_t));
    return g;
}

// Whether 16-bit scans run on pairs of columns, a row segment of 128 or 256 bytes a tile: (4, 65536, 1024) fp16 432 and
// 547 us (forward, adjoint) -> 344 and 526, (1024, 700, 64) 57 and 101 -> 54 and 100. Below 33 columns and with too few
// tiles to fill the chip single columns are faster: (384, 1024, 16) 15.5 us against 16.7, (3, 1000, 100) 9.0 against 9.4.
bool use_pairs(int64_t nseq, int64_t seqlen, int64_t ncols) {
    if (ncols % 2 != 0 || ncols <= 32) return false;
    const PscanGeom g = geom(nseq, seqlen, ncols, 2);
    return nseq * g.ncolblk * g.nltile >= 128;
}

__device__ __forceinline__ uint64_t pack(uint32_t st, float v) {
    return ((uint64_t)st << 32) | (uint64_t)__builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float unpack_v(uint64_t w) { return __builtin_bit_cast(float, (uint32_t)(w & 0xffffffffu)); }
// A tile's coefficient m * 2^e: e above the two status bits (at most 256 steps of |e| <= 149, so it fits 30 bits).
__device__ __forceinline__ uint64_t pack_coef(uint32_t st, float m, int e) { return pack(st | (uint32_t)e << 2, m); }
__device__ __forceinline__ int unpack_e(uint64_t w) { return (int)(uint32_t)(w >> 32) >> 2; }

// Whether a product is not safely inside fp32's normal range (NaN included)
__device__ __forceinline__ bool out_of_range(float m) {
    m = __builtin_fabsf(m);
    return !(m >= 0x1p-100f && m <= 0x1p100f);
}
// m * 2^e * h + b, rounded once where h * 2^e is a normal number
__device__ __forceinline__ float apply(float m, int e, float h, float b) {
    return __builtin_fmaf(m, __builtin_ldexpf(h, e), b);
}

__device__ __forceinline__ void publish(uint64_t* p, uint64_t w) {
    __hip_atomic_store(p, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Wait until *p carries a non-zero status; returns the word. If `limit` polls pass without one, the
// error word is set and an inclusive NaN is returned: the tile's prefix, and so its outputs, are NaN.
__device__ __forceinline__ uint64_t wait_word(const uint64_t* p, unsigned* err, unsigned limit) {
    for (unsigned it = 0; it < limit; ++it) {
        const uint64_t w = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((w >> 32) != 0) return w;
        __builtin_amdgcn_s_sleep(2);
    }
    atomicOr(err, 1u);
    return pack(kStInc, __builtin_nanf(""));
}

}  // namespace

__global__ void __launch_bounds__(256) pscan_clear_kernel(uint64_t* __restrict__ p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = 0;
}

// A thread's V values of one row as loaded: one value, or a pair of 16-bit ones in the register that its load fills.
template <typename T, int V> __device__ __forceinline__ raw_t<T> row_ld(const T* p) {
    if constexpr (V == 2)
        return *reinterpret_cast<const uint32_t*>(p);
    else
        return raw_ld(p);
}
template <typename T> __device__ __forceinline__ float row_val(raw_t<T> w, int v) {
    if constexpr (sizeof(T) == 4)
        return w;
    else
        return raw_f<T>(w >> (16 * v));
}
template <typename T, int V> __device__ __forceinline__ void row_st(T* p, const float (&x)[V]) {
    if constexpr (V == 2) {
        const T lo = static_cast<T>(x[0]), hi = static_cast<T>(x[1]);
        *reinterpret_cast<uint32_t*>(p) =
            (uint32_t)__builtin_bit_cast(uint16_t, lo) | (uint32_t)__builtin_bit_cast(uint16_t, hi) << 16;
    } else {
        st(p, x[0]);
    }
}

// REV = false: forward scan of X with coefficients A (A_0 ignored) into Out.
// REV = true : adjoint; X = dH, Out = dX, Hs = forward H, dAo = dA.
// A thread owns V adjacent columns (2: 16-bit pairs).
template <typename T, int CW, int V, bool REV>
__global__ void __launch_bounds__(kThreads, scan_waves(CW, REV))
pscan_kernel(const T* __restrict__ A, const T* __restrict__ X, const T* __restrict__ Hs, T* __restrict__ Out,
             T* __restrict__ dAo, uint64_t* __restrict__ flags, unsigned* __restrict__ tickets,
             unsigned* __restrict__ err, int L, int ncols, int ncolblk, int64_t nchains, int gchains,
             unsigned ngroups, unsigned spin_limit) {
    constexpr int R = kThreads / CW;     // thread rows per tile
    constexpr int TS = tile_steps(CW), RUN = TS / R;  // steps of a tile and of a thread
    __shared__ int s_tile, s_wide;
    __shared__ float s_a[R][V][CW], s_h[R][V][CW], s_p[V][CW];
    __shared__ int s_e[R][V][CW];  // exponents of s_a, read where s_wide: some run's coefficient leaves fp32

    // a ticket group's tiles: its column blocks, all at one step range before the next
    const unsigned group = blockIdx.x % ngroups;
    const int64_t chain0 = (int64_t)group * gchains;
    const int gw = (int)min((int64_t)gchains, nchains - chain0);
    const int nltile = (L + TS - 1) / TS;
    if (threadIdx.x == 0) {  // one tile along L: nothing waits, a group is one tile
        s_tile = nltile > 1 ? (int)atomicAdd(tickets + (size_t)group * kTicketStride, 1u) : 0;
        s_wide = 0;
    }
    if (nltile == 1 && blockIdx.x == 0 && threadIdx.x == 0) *err = 0;  // nor is the workspace cleared
    __syncthreads();
    const int lt = s_tile / gw;  // position of the tile along L (in scan order)
    if (lt >= nltile) return;    // a smaller last group has more blocks than tiles
    const int64_t chain = chain0 + s_tile % gw;
    const int64_t seq = chain / ncolblk;
    const int cb = (int)(chain % ncolblk);
    const int cl = threadIdx.x % CW, r = threadIdx.x / CW;
    const int col = (cb * CW + cl) * V;
    const bool cvalid = col < ncols;  // V divides ncols
    const int64_t base = seq * L * ncols + (cvalid ? col : ncols - V);
    const int p0 = lt * TS + r * RUN;

    // Position p -> step t (the adjoint runs from the end). Rows past the ends are read from the nearest row of the
    // sequence and set to 0 afterwards: 16-bit loads under a branch were converted, and so waited for, one by one there
    // ((4, 65536, 1024) fp16: 1140 us against 431, the adjoint 1491 against 573; fp32 adjoint 1178 against 1038).
    raw_t<T> wa[RUN], wx[RUN], wh[REV ? RUN : 1];
    auto row = [&](int t) { return base + (int64_t)max(0, min(t, L - 1)) * ncols; };
#pragma unroll
    for (int i = 0; i < RUN; ++i) {
        const int t = REV ? L - 1 - p0 - i : p0 + i;
        wa[i] = row_ld<T, V>(A + row(REV ? t + 1 : t));
        wx[i] = row_ld<T, V>(X + row(t));
        if constexpr (REV) wh[i] = row_ld<T, V>(Hs + row(t - 1));
    }
    // else this load is moved under the test of its row, behind all the others: (2048, 300, 32) fp16 28.3 us, not 27.8
    asm volatile("" : "+v"(wx[0]));
#pragma unroll
    for (int i = 0; i < RUN; ++i) {
        const bool has_a = p0 + i > 0 && p0 + i < L;  // A_0 (forward) and A_L (adjoint) do not enter
        wa[i] = has_a ? wa[i] : 0;
        wx[i] = p0 + i < L ? wx[i] : 0;
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {  // the run's map h -> ra*h + rh
        float ra = 1.f, rh = 0.f;
#pragma unroll
        for (int i = 0; i < RUN; ++i) {
            if constexpr (V == 2) asm volatile("" : "+v"(wa[i]), "+v"(wx[i]));  // see the second pass below
            const float a = row_val<T>(wa[i], v);
            rh = __builtin_fmaf(a, rh, row_val<T>(wx[i], v));
            ra *= a;
        }
        // Out of this range the product is formed again from mantissas and exponents (rare: one compare a run). The
        // first run's coefficient has no state to multiply, and that of a run past the end is not used.
        int re = 0;
        if (out_of_range(ra) && p0 > 0 && p0 + RUN <= L) {
            ra = 1.f;
#pragma unroll
            for (int i = 0; i < RUN; ++i) {
                const float p = ra * row_val<T>(wa[i], v);
                re += __builtin_amdgcn_frexp_expf(p);
                ra = __builtin_amdgcn_frexp_mantf(p);
            }
            s_wide = 1;
        }
        s_a[r][v][cl] = ra;
        s_e[r][v][cl] = re;
        s_h[r][v][cl] = rh;
    }
    __syncthreads();

    const bool wide = s_wide != 0;
    if (r < V) {  // thread row v joins the tiles' column v of each thread
        float ta = 1.f, th = 0.f;  // the tile's map ta * 2^te * h + th
        int te = 0;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            th = __builtin_fmaf(s_a[q][r][cl], th, s_h[q][r][cl]);
            ta *= s_a[q][r][cl];
        }
        if (wide || (lt > 0 && lt + 1 < nltile && out_of_range(ta))) {  // again with exponents: a product of R mantissas is above 2^-R
            ta = 1.f, th = 0.f;
#pragma unroll 2  // all at once the loads take 30 to 60 registers more, and the waves that they hold
            for (int q = 0; q < R; ++q) {
                const float qa = s_a[q][r][cl];
                const int qe = s_e[q][r][cl];
                th = apply(qa, qe, th, s_h[q][r][cl]);
                ta *= __builtin_amdgcn_frexp_mantf(qa);
                te += qe + __builtin_amdgcn_frexp_expf(qa);
            }
        }
        uint64_t* f = flags + ((chain * nltile + lt) * (CW * V) + r * CW + cl) * 2;
        float prefix = 0.f;  // state entering the tile (the scan starts from 0; t = 0 ignores A_0)
        if (lt == 0) {
            if (nltile > 1) publish(f, pack(kStInc, th));
        } else {
            publish(f + 1, pack_coef(kStAgg, ta, te));
            publish(f, pack(kStAgg, th));
            float acc_a = 1.f, acc_h = 0.f;  // map of the tiles between the predecessor and this one
            int acc_e = 0;
            uint64_t* pf = f - (int64_t)(CW * V) * 2;
            for (int j = lt - 1; j >= 0; --j, pf -= (int64_t)(CW * V) * 2) {
                const uint64_t w = wait_word(pf, err, spin_limit);
                if ((w >> 32) == kStInc) {
                    prefix = apply(acc_a, acc_e, unpack_v(w), acc_h);
                    break;
                }
                const uint64_t wa = wait_word(pf + 1, err, spin_limit);
                acc_h = apply(acc_a, acc_e, unpack_v(w), acc_h);
                acc_a *= unpack_v(wa);
                acc_e += unpack_e(wa) + __builtin_amdgcn_frexp_expf(acc_a);
                acc_a = __builtin_amdgcn_frexp_mantf(acc_a);
            }
            publish(f, pack(kStInc, apply(ta, te, prefix, th)));
        }
        s_p[r][cl] = prefix;
    }
    __syncthreads();

    // state entering this thread's run: rows 0..r-1 applied to the tile prefix
    float h[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        h[v] = s_p[v][cl];
        if (wide)
#pragma unroll 1
            for (int q = 0; q < r; ++q) h[v] = apply(s_a[q][v][cl], s_e[q][v][cl], h[v], s_h[q][v][cl]);
        else
            for (int q = 0; q < r; ++q) h[v] = __builtin_fmaf(s_a[q][v][cl], h[v], s_h[q][v][cl]);
    }
#pragma unroll
    for (int i = 0; i < RUN; ++i) {
        const int p = p0 + i;
        if constexpr (V == 2) asm volatile("" : "+v"(wa[i]), "+v"(wx[i]));  // convert again rather than keep both pairs
#pragma unroll
        for (int v = 0; v < V; ++v) h[v] = __builtin_fmaf(row_val<T>(wa[i], v), h[v], row_val<T>(wx[i], v));
        if (p < L && cvalid) {
            const int t = REV ? L - 1 - p : p;
            row_st<T, V>(Out + base + (int64_t)t * ncols, h);
            if constexpr (REV) {
                float da[V];
#pragma unroll
                for (int v = 0; v < V; ++v) da[v] = t > 0 ? h[v] * row_val<T>(wh[i], v) : 0.f;
                row_st<T, V>(dAo + base + (int64_t)t * ncols, da);
            }
        }
    }
}

size_t pscan_workspace_bytes(int64_t nseq, int64_t seqlen, int64_t ncols) {
    if (nseq <= 0 || seqlen <= 0 || ncols <= 0) return 0;
    size_t n = geom(nseq, seqlen, ncols, 1).bytes;
    if (use_pairs(nseq, seqlen, ncols)) n = std::max(n, geom(nseq, seqlen, ncols, 2).bytes);
    return n;
}

bool pscan_waits(int64_t nseq, int64_t seqlen, int64_t ncols) {
    return nseq > 0 && seqlen > 0 && ncols > 0 && geom(nseq, seqlen, ncols, 1).nltile > 1;  // the same for pairs
}

template <typename T, bool REV>
static hipError_t pscan_t(const void* A, const void* X, const void* Hs, void* Out, void* dAo, int64_t nseq,
                          int64_t seqlen, int64_t ncols, void* ws, unsigned spin_limit, hipStream_t st) {
    bool pairs = sizeof(T) == 2 && use_pairs(nseq, seqlen, ncols);
    for (const void* p : {A, X, Hs, (const void*)Out, (const void*)dAo}) pairs = pairs && (uintptr_t)p % 4 == 0;
    const PscanGeom g = geom(nseq, seqlen, ncols, pairs ? 2 : 1);
    if (g.nblocks > INT32_MAX) return hipErrorInvalidValue;
    unsigned* err = (unsigned*)ws;
    unsigned* tickets = err + kTicketStride;
    uint64_t* flags = (uint64_t*)((char*)ws + g.flags_offset);
    if (g.nltile > 1) {
        const int64_t nwords = (int64_t)g.bytes / 8;
        const int cgrid = (int)std::min<int64_t>((nwords + 255) / 256, 4096);
        hipLaunchKernelGGL(pscan_clear_kernel, dim3(cgrid), dim3(256), 0, st, (uint64_t*)ws, nwords);
    }
#define MWC_PSCAN(CWV, VV)                                                                                          \
    if (g.cw == CWV && g.vec == VV)                                                                                 \
        hipLaunchKernelGGL((pscan_kernel<T, CWV, VV, REV>), dim3((unsigned)g.nblocks), dim3(kThreads), 0, st,       \
                           (const T*)A, (const T*)X, (const T*)Hs, (T*)Out, (T*)dAo, flags, tickets, err,           \
                           (int)seqlen, (int)ncols, g.ncolblk, nseq * g.ncolblk, g.gchains,              \
                           (unsigned)g.ngroups, spin_limit);
    MWC_PSCAN(8, 1)
    MWC_PSCAN(16, 1)
    MWC_PSCAN(32, 1)
    MWC_PSCAN(64, 1)
    if constexpr (sizeof(T) == 2) {  // pairs: more than 32 columns
        MWC_PSCAN(32, 2)
        MWC_PSCAN(64, 2)
    }
#undef MWC_PSCAN
    return hipGetLastError();
}

hipError_t launch_pscan_fwd(int dt, const void* A, const void* X, void* H, int64_t nseq, int64_t seqlen,
                            int64_t ncols, void* ws, unsigned spin_limit, hipStream_t st) {
    MWC_DISPATCH_DTYPE(dt, TT,
                       return pscan_t<TT, false>(A, X, nullptr, H, nullptr, nseq, seqlen, ncols, ws, spin_limit, st));
}

hipError_t launch_pscan_bwd(int dt, const void* A, const void* H, const void* dH, void* dA, void* dX,
                            int64_t nseq, int64_t seqlen, int64_t ncols, void* ws, unsigned spin_limit,
                            hipStream_t st) {
    MWC_DISPATCH_DTYPE(dt, TT, return pscan_t<TT, true>(A, dH, H, dX, dA, nseq, seqlen, ncols, ws, spin_limit, st));
}

}  // namespace mwc
