// Standalone first-order linear recurrence ("parallel_scan_fn") for gfx950.
//
// Semantics: parallel_scan_ref (pscan.py:153-171): over the middle axis of
// [nseq][L][ncols], H_0 = X_0 (A_0 unused), H_t = A_t*H_{t-1} + X_t, with fp32
// accumulation; and its adjoint (replacing PScan.backward, pscan.py:97-136,
// whose math is wrong for L >= 4): G_t = dH_t + A_{t+1}*G_{t+1}, dX = G,
// dA_t = G_t*H_{t-1} for t >= 1 and dA_0 = 0.
//
// Two designs, chosen by use_chains: one wave per sequence (pscan_chain_kernel) for many narrow sequences, and the
// tiled look-back scan described here.
//
// Design: one pass over HBM (12 B/element forward, 20 B/element backward).
// A tile is TL consecutive steps x CW columns; each thread owns one column and
// RUN consecutive steps held in VGPRs. Thread runs are combined inside the
// tile through LDS; tiles along L are chained with a decoupled look-back:
// each tile publishes its aggregate map h -> a*h + b per column, then its
// inclusive prefix once known, as 64-bit (status << 32 | fp32 bits) words so
// a single relaxed agent-scope atomic carries both the flag and the value
// (no cache-wide release/acquire fences). Tiles are taken from an atomic
// ticket so every predecessor of a waiting tile is already resident, and each
// spin is bounded so a lost update can never hang the device. A wait that runs
// out of spins sets the workspace's error word (read by mwc_pscan_status) and
// gives the tile a NaN prefix, so its outputs, and every later tile's, are NaN
// rather than a plausible wrong value.
#include <algorithm>

#include "common.h"
#include "launch.h"

namespace mwc {

namespace {

constexpr int kThreads = 256;
constexpr int kTileSteps = 128;
constexpr uint32_t kStAgg = 1, kStInc = 2;

int pick_cw(int64_t ncols) { return ncols <= 16 ? 16 : (ncols <= 32 ? 32 : 64); }

struct PscanGeom {
    int cw, ncolblk, nltile;
    int64_t nchains, ntiles;
    size_t flag_bytes;
};

PscanGeom geom(int64_t nseq, int64_t seqlen, int64_t ncols) {
    PscanGeom g;
    g.cw = pick_cw(ncols);
    g.ncolblk = (int)((ncols + g.cw - 1) / g.cw);
    g.nltile = (int)((seqlen + kTileSteps - 1) / kTileSteps);
    g.nchains = nseq * g.ncolblk;
    g.ntiles = g.nchains * g.nltile;
    g.flag_bytes = (size_t)g.ntiles * g.cw * 2 * sizeof(uint64_t);
    return g;
}

__device__ __forceinline__ uint64_t pack(uint32_t st, float v) {
    return ((uint64_t)st << 32) | (uint64_t)__builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ float unpack_v(uint64_t w) { return __builtin_bit_cast(float, (uint32_t)(w & 0xffffffffu)); }

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

// REV = false: forward scan of X with coefficients A (A_0 ignored) into Out.
// REV = true : adjoint; X = dH, Out = dX, Hs = forward H, dAo = dA.
template <typename T, int CW, bool REV>
__global__ void __launch_bounds__(kThreads) pscan_kernel(const T* __restrict__ A, const T* __restrict__ X,
                                                         const T* __restrict__ Hs, T* __restrict__ Out,
                                                         T* __restrict__ dAo, uint64_t* __restrict__ flags,
                                                         unsigned* __restrict__ ticket, unsigned* __restrict__ err,
                                                         int L, int ncols, int ncolblk, int64_t nchains,
                                                         unsigned spin_limit) {
    constexpr int R = kThreads / CW;     // thread rows per tile
    constexpr int RUN = kTileSteps / R;  // steps per thread
    __shared__ int s_tile;
    __shared__ float s_a[R][CW], s_h[R][CW], s_p[CW];

    if (threadIdx.x == 0) s_tile = (int)atomicAdd(ticket, 1u);
    __syncthreads();
    const int64_t tile = s_tile;
    const int lt = (int)(tile / nchains);  // position of the tile along L (in scan order)
    const int64_t chain = tile % nchains;
    const int64_t seq = chain / ncolblk;
    const int cb = (int)(chain % ncolblk);
    const int cl = threadIdx.x % CW, r = threadIdx.x / CW;
    const int col = cb * CW + cl;
    const bool cvalid = col < ncols;
    const int64_t base = seq * L * ncols + (cvalid ? col : ncols - 1);
    const int p0 = lt * kTileSteps + r * RUN;

    // Position p -> step t (the adjoint runs from the end). Rows past the ends are read from the nearest row of the
    // sequence and set to 0 afterwards: 16-bit loads under a branch were converted, and so waited for, one by one there
    // ((4, 65536, 1024) fp16: 1140 us against 431, the adjoint 1491 against 573; fp32 adjoint 1178 against 1038).
    raw_t<T> wa[RUN], wx[RUN], wh[REV ? RUN : 1];
    auto row = [&](int t) { return base + (int64_t)max(0, min(t, L - 1)) * ncols; };
#pragma unroll
    for (int i = 0; i < RUN; ++i) {
        const int t = REV ? L - 1 - p0 - i : p0 + i;
        wa[i] = raw_ld(A + row(REV ? t + 1 : t));
        wx[i] = raw_ld(X + row(t));
        if constexpr (REV) wh[i] = raw_ld(Hs + row(t - 1));
    }
    float a[RUN], x[RUN];
#pragma unroll
    for (int i = 0; i < RUN; ++i) {
        const bool has_a = p0 + i > 0 && p0 + i < L;  // A_0 (forward) and A_L (adjoint) do not enter
        a[i] = has_a ? raw_f<T>(wa[i]) : 0.f;
        x[i] = p0 + i < L ? raw_f<T>(wx[i]) : 0.f;
    }
    // the run's map h -> ra*h + rh
    float ra = 1.f, rh = 0.f;
#pragma unroll
    for (int i = 0; i < RUN; ++i) {
        rh = __builtin_fmaf(a[i], rh, x[i]);
        ra *= a[i];
    }
    s_a[r][cl] = ra;
    s_h[r][cl] = rh;
    __syncthreads();

    if (r == 0) {
        float ta = 1.f, th = 0.f;  // the tile's map
#pragma unroll
        for (int q = 0; q < R; ++q) {
            th = __builtin_fmaf(s_a[q][cl], th, s_h[q][cl]);
            ta *= s_a[q][cl];
        }
        uint64_t* f = flags + ((chain * (int64_t)((L + kTileSteps - 1) / kTileSteps) + lt) * CW + cl) * 2;
        float prefix = 0.f;  // state entering the tile (the scan starts from 0; t = 0 ignores A_0)
        if (lt == 0) {
            publish(f, pack(kStInc, th));
        } else {
            publish(f + 1, pack(kStAgg, ta));
            publish(f, pack(kStAgg, th));
            float acc_a = 1.f, acc_h = 0.f;  // map of the tiles between the predecessor and this one
            uint64_t* pf = f - (int64_t)CW * 2;
            for (int j = lt - 1; j >= 0; --j, pf -= (int64_t)CW * 2) {
                const uint64_t w = wait_word(pf, err, spin_limit);
                if ((w >> 32) == kStInc) {
                    prefix = __builtin_fmaf(acc_a, unpack_v(w), acc_h);
                    break;
                }
                const uint64_t wa = wait_word(pf + 1, err, spin_limit);
                acc_h = __builtin_fmaf(acc_a, unpack_v(w), acc_h);
                acc_a *= unpack_v(wa);
            }
            publish(f, pack(kStInc, __builtin_fmaf(ta, prefix, th)));
        }
        s_p[cl] = prefix;
    }
    __syncthreads();

    // state entering this thread's run: rows 0..r-1 applied to the tile prefix
    float h = s_p[cl];
    for (int q = 0; q < r; ++q) h = __builtin_fmaf(s_a[q][cl], h, s_h[q][cl]);
#pragma unroll
    for (int i = 0; i < RUN; ++i) {
        const int p = p0 + i;
        h = __builtin_fmaf(a[i], h, x[i]);
        if (p < L && cvalid) {
            const int t = REV ? L - 1 - p : p;
            st(Out + base + (int64_t)t * ncols, h);
            if constexpr (REV) st(dAo + base + (int64_t)t * ncols, t > 0 ? h * raw_f<T>(wh[i]) : 0.f);
        }
    }
}

// One wave per sequence of up to CW columns, for calls with sequences enough to fill the chip without
// cutting L: the wave walks its sequence in tiles of (64/CW)*RUN steps with the state carried in a register, so
// there are no tickets, flags, look-back or workgroup barriers. A lane owns one column and RUN consecutive steps
// of a tile; the 64/CW runs of a column are joined by lane shuffles. The next tile's loads are in flight while a
// tile is scanned. Bound: HBM.
template <typename T, int CW, bool REV>
__global__ void __launch_bounds__(kThreads) pscan_chain_kernel(const T* __restrict__ A, const T* __restrict__ X,
                                                               const T* __restrict__ Hs, T* __restrict__ Out,
                                                               T* __restrict__ dAo, unsigned* __restrict__ err, int L,
                                                               int ncols, int64_t nseq) {
    constexpr int R = 64 / CW;  // runs per tile
    constexpr int RUN = sizeof(T) == 4 ? 8 : 16;  // steps per run: the same bytes in flight at 2 bytes an element
    constexpr int TS = R * RUN;
    if (blockIdx.x == 0 && threadIdx.x == 0) *err = 0;  // no wait that could give up
    const int64_t seq = (int64_t)blockIdx.x * (kThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (seq >= nseq) return;
    const int lane = threadIdx.x & 63;
    const int col = lane % CW, r = lane / CW;
    const int row_bytes = ncols * (int)sizeof(T);  // ncols <= 32: a tile's byte offsets are small
    const int64_t base = seq * L * ncols;
    const int ntile = (L + TS - 1) / TS;

    // Tile n covers positions p = n*TS .. n*TS + TS - 1 in scan order: step t = p, or L - 1 - p for the adjoint.
    // Rows are addressed from the tile's lowest step t0; offsets of positions at or past L (negative ones for the
    // adjoint), of columns past ncols and of the neighbours that do not exist lie outside the resources, which
    // return 0 for them and drop their stores.
    auto first_row = [&](int n) { return REV ? max(0, L - (n + 1) * TS) : n * TS; };
    auto lane_off = [&](int n, int i) {  // byte offset of the lane's step i from row first_row(n)
        const int row = REV ? (L - 1 - n * TS - (r * RUN + i)) - first_row(n) : r * RUN + i;
        return col < ncols ? (uint32_t)(row * row_bytes + col * (int)sizeof(T)) : kOob;
    };
    auto rsrc = [&](const T* p, int row) {  // rows [row, min(row + TS, L))
        return make_rsrc(p + base + (int64_t)row * ncols, (uint32_t)(max(0, min(TS, L - row)) * row_bytes));
    };
    raw_t<T> na[RUN], nx[RUN], nh[REV ? RUN : 1];
    auto issue = [&](int n) {
        const int t0 = first_row(n);
        // the adjoint's coefficient is A_{t+1} (none at t = L - 1) and its factor H_{t-1} (none at t = 0)
        const rsrc_t ra = rsrc(A, REV ? t0 + 1 : t0), rx = rsrc(X, t0);
        const int th = t0 > 0 ? t0 - 1 : 0;
        const rsrc_t rh = rsrc(REV ? Hs : X, th);
        const int dh = t0 > 0 ? 0 : row_bytes;
#pragma unroll
        for (int i = 0; i < RUN; ++i) {
            const uint32_t o = lane_off(n, i);
            na[i] = buf_raw<T>(ra, o);
            nx[i] = buf_raw<T>(rx, o);
            if constexpr (REV) nh[i] = buf_raw<T>(rh, o - dh);
        }
    };
    float h = 0.f;  // state entering the tile (the scan starts from 0)
    issue(0);
    for (int n = 0; n < ntile; ++n) {
        float a[RUN], x[RUN], g[RUN];
#pragma unroll
        for (int i = 0; i < RUN; ++i) {
            a[i] = raw_f<T>(na[i]);
            x[i] = raw_f<T>(nx[i]);
            if constexpr (REV) g[i] = raw_f<T>(nh[i]);
        }
        if (!REV && n == 0) a[0] = r == 0 ? 0.f : a[0];  // A_0 is not used, whatever it holds
        if (n + 1 < ntile) issue(n + 1);
        float ra = 1.f, rh = 0.f;  // the run's map h -> ra*h + rh
#pragma unroll
        for (int i = 0; i < RUN; ++i) {
            rh = __builtin_fmaf(a[i], rh, x[i]);
            ra *= a[i];
        }
        float s = h;  // state entering this lane's run; h becomes the one entering the next tile
#pragma unroll
        for (int q = 0; q < R; ++q) {
            if (q == r) s = h;
            h = __builtin_fmaf(__shfl(ra, q * CW + col), h, __shfl(rh, q * CW + col));
        }
#pragma unroll
        for (int i = 0; i < RUN; ++i) x[i] = s = __builtin_fmaf(a[i], s, x[i]);
        const int t0 = first_row(n);
        const rsrc_t ro = rsrc(Out, t0), rd = rsrc(REV ? dAo : Out, t0);
#pragma unroll
        for (int i = 0; i < RUN; ++i) {
            const uint32_t o = lane_off(n, i);
            buf_st<T>(ro, o, x[i]);
            if constexpr (REV) {
                float da = x[i] * g[i];
                if (t0 == 0) da = L - 1 - n * TS - (r * RUN + i) == 0 ? 0.f : da;  // dA_0 = 0, whatever x holds
                buf_st<T>(rd, o, da);
            }
        }
    }
}

// Whether the one-wave-per-sequence kernel runs, at *cw columns a wave, rather than the tiled look-back kernel.
// Forward and adjoint, against the look-back kernel: (768, 1024, 16) 45 and 83 us against 81 and 86 in fp32, 47 and
// 83 against 79 and 81 in fp16; at (384, 1024, 16) too few bytes are in flight and the look-back kernel is as fast.
// Sequences of up to 32 columns need more of them: (1024, 700, 32) fp16 64 and 120 us against 81 and 84, and
// (2048, 300, 32) 36 and 67 against 79 and 82. Rows of 64 columns, whose look-back tiles hold four times a 16-column
// one's bytes, stay there: (1024, 700, 64) fp16 87 and 107 us against 98 and 264 in waves of 64 columns.
bool use_chains(int64_t nseq, int64_t ncols, int* cw) {
    *cw = ncols <= 8 ? 8 : ncols <= 16 ? 16 : 32;
    return ncols <= 32 && nseq >= (*cw == 32 ? 2048 : 768);
}

size_t pscan_workspace_bytes(int64_t nseq, int64_t seqlen, int64_t ncols) {
    if (nseq <= 0 || seqlen <= 0 || ncols <= 0) return 0;
    const PscanGeom g = geom(nseq, seqlen, ncols);
    return ((g.flag_bytes + 255) & ~(size_t)255) + 256;  // flags, then ticket + error word
}

bool pscan_waits(int64_t nseq, int64_t seqlen, int64_t ncols) {
    int cw = 0;
    return nseq > 0 && seqlen > 0 && ncols > 0 && !use_chains(nseq, ncols, &cw);
}

size_t pscan_error_word_offset(int64_t nseq, int64_t seqlen, int64_t ncols) {
    const PscanGeom g = geom(nseq, seqlen, ncols);
    return ((g.flag_bytes + 255) & ~(size_t)255) + sizeof(unsigned);  // after the ticket
}

template <typename T, bool REV>
static hipError_t pscan_t(const void* A, const void* X, const void* Hs, void* Out, void* dAo, int64_t nseq,
                          int64_t seqlen, int64_t ncols, void* ws, unsigned spin_limit, hipStream_t st) {
    const PscanGeom g = geom(nseq, seqlen, ncols);
    uint64_t* flags = (uint64_t*)ws;
    const size_t fb = (g.flag_bytes + 255) & ~(size_t)255;
    unsigned* ticket = (unsigned*)((char*)ws + fb);
    unsigned* err = ticket + 1;
    const int64_t nwords = (int64_t)(fb + 256) / 8;
    if (g.ntiles > INT32_MAX) return hipErrorInvalidValue;
    int cw = 0;
    if (use_chains(nseq, ncols, &cw)) {
        const unsigned grid = (unsigned)((nseq + kThreads / 64 - 1) / (kThreads / 64));
#define MWC_CHAIN_CW(CWV)                                                                                         \
    if (cw == CWV)                                                                                                \
        hipLaunchKernelGGL((pscan_chain_kernel<T, CWV, REV>), dim3(grid), dim3(kThreads), 0, st, (const T*)A,       \
                           (const T*)X, (const T*)Hs, (T*)Out, (T*)dAo, err, (int)seqlen, (int)ncols, nseq);
        MWC_CHAIN_CW(8)
        MWC_CHAIN_CW(16)
        MWC_CHAIN_CW(32)
#undef MWC_CHAIN_CW
        return hipGetLastError();
    }
    const int cgrid = (int)std::min<int64_t>((nwords + 255) / 256, 4096);
    hipLaunchKernelGGL(pscan_clear_kernel, dim3(cgrid), dim3(256), 0, st, flags, nwords);
#define MWC_PSCAN_CW(CWV)                                                                                         \
    if (g.cw == CWV)                                                                                              \
        hipLaunchKernelGGL((pscan_kernel<T, CWV, REV>), dim3((unsigned)g.ntiles), dim3(kThreads), 0, st,          \
                           (const T*)A, (const T*)X, (const T*)Hs, (T*)Out, (T*)dAo, flags, ticket, err,           \
                           (int)seqlen, (int)ncols, g.ncolblk, g.nchains, spin_limit);
    MWC_PSCAN_CW(16)
    MWC_PSCAN_CW(32)
    MWC_PSCAN_CW(64)
#undef MWC_PSCAN_CW
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
