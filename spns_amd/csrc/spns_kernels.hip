// HIP kernels for the pseudospectral HIT step on MI355X (gfx950).
//
// Data layout in HBM (k3 contiguous everywhere):
//   state u_c, R_c      : FP64 compact retained box [i2][i1][i3], nk2 x nk1 x nk3,
//                          the reference's Fourier-dump order (src/HIT_LES_output.cpp:46-53)
//   X1 (after the y pass): T complex [y][i1][i3], My x nk1 x nk3 per field
//   X2 (after the x pass): T complex [y][x][i3],  My x Mx  x nk3 per field
// Passes of one step (DNS; LES adds six SGS fields to the forward passes):
//   inv_y  : u_c -> {F_c = FFT_y u_c, G_c = FFT_y(i k2 u_c)}          (strided, pruned in)
//   inv_x  : {F_c, G_c} -> {u_c, d_x u_c, d_y u_c}                   (strided, pruned in)
//   z pass : c2r of 12 fields (d_z from i k3), advective products,
//            Smagorinsky nu_t and tau, CFL max, skewness, r2c          (pencil, pruned in/out)
//   fwd_x, fwd_y : forward transforms back to the compact box         (strided, pruned out)
//   epilogue: normalise, R, rotation, forcing, AB2 / kappa, projection,
//            E(K) and enstrophy partials                              (elementwise, FP64)
//   finalize: fixed-order sums, CFL time step, time, iteration count
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdlib.h>

#include "spns_device.hpp"
#include "spns_internal.hpp"

#ifndef SPNS_PART
#define SPNS_PART 0
#endif

namespace spns {

// ---------------------------------------------------------------------------
// shell index K = round(|k|) computed exactly in integers (src/HIT_LES.cpp:1166)
// ---------------------------------------------------------------------------
__device__ __forceinline__ int shell_of(int k2)
{
    int m = (int)sqrt((double)k2);
    while (m * m > k2) m--;
    while ((m + 1) * (m + 1) <= k2) m++;
    return (k2 > m * m + m) ? m + 1 : m;
}

__device__ __forceinline__ int wrap_k(int i, int n)  // compact index -> wavenumber
{
    return (i <= n / 2) ? i : i - n;
}

// i k v, formed in the input precision (src/HIT_LES.cpp:37) and rounded to
// the transform type T.  The products are rounded before they enter a
// butterfly: with contraction off, the compiler cannot fuse them into the
// butterflies' additions in one loader and not in another, so every pass
// that forms a derivative on load (the strided inverse passes, and the next
// step's inverse y pass inside the fused forward y kernel) has the same
// rounding.
template <typename T, typename TIN>
__device__ __forceinline__ cx<T> times_ik(TIN kk, cx<TIN> v)
{
#pragma clang fp contract(off)
    const TIN re = -kk * v.y, im = kk * v.x;
    return cx<T>{(T)re, (T)im};
}

template <typename T, int L>
constexpr int strided_tb()
{
    // largest column tile with the FFT tile in <= 48 KB of LDS
    constexpr int bytes = (int)sizeof(cx<T>) * L;
    return (bytes * 16 <= 49152) ? 16 : (bytes * 8 <= 49152) ? 8 : (bytes * 4 <= 49152) ? 4 : (bytes * 2 <= 49152) ? 2 : 1;
}

// ---------------------------------------------------------------------------
// Strided batched pass: transforms along a row dimension of [A][rows][B]
// (B contiguous), TB consecutive columns per block.
// ---------------------------------------------------------------------------
template <typename TIN, typename TOUT, typename T, int L, int TB, int NT, int DIR>
__global__ __launch_bounds__(NT) void k_strided(StridedArgs a)
{
    __shared__ cx<T> lds[L * TB];
    if (a.skip && *a.skip) return;
    // Workgroups are dispatched round-robin over the 8 XCDs, each with its own
    // L2.  Remap the (padded, multiple-of-8) 1-D grid so every XCD owns a
    // contiguous run of tiles: neighbouring column tiles, which share cache
    // lines, then meet in the same L2.
    const int ntiles = (a.B + TB - 1) / TB;
    const int per = gridDim.x / 8;
    const int lin = (blockIdx.x % 8) * per + blockIdx.x / 8;
    const int64_t ai = lin / ntiles;
    if (ai >= a.A) return;
    const int b0 = (lin % ntiles) * TB;
    const cx<T>* tw = (const cx<T>*)a.tw;
    const int hin = a.nin / 2, hout = a.nout / 2;
    for (int jb = 0; jb < a.njobs; jb++) {
        const cx<TIN>* __restrict__ in = (const cx<TIN>*)a.job[jb].in + ai * a.in_a_stride;
        cx<TOUT>* __restrict__ out = (cx<TOUT>*)a.job[jb].out + ai * a.out_a_stride;
        const int deriv = a.job[jb].deriv;
        auto load = [&](int b, int p) -> cx<T> {
            const int bb = b0 + b;
            int i, k;
            if (a.nin == L) { i = p; k = (p <= L / 2) ? p : p - L; }
            else if (p <= hin) { i = p; k = p; }
            else if (p >= L - hin) { i = a.nin - (L - p); k = p - L; }
            else return cx<T>{(T)0, (T)0};
            if (bb >= a.B) return cx<T>{(T)0, (T)0};
            cx<TIN> v = in[(int64_t)i * a.in_row_stride + bb];
            if (deriv) return times_ik<T>((TIN)k, v);
            return cx<T>{(T)v.x, (T)v.y};
        };
        auto store = [&](int b, int p, cx<T> v) {
            const int bb = b0 + b;
            int i;
            if (a.nout == L || p <= hout) i = p;
            else if (p >= L - hout) i = a.nout - (L - p);
            else return;
            if (bb >= a.B) return;
            out[(int64_t)i * a.out_row_stride + bb] = cx<TOUT>{(TOUT)v.x, (TOUT)v.y};
        };
        Fft<T, L, TB, NT, TB, DIR>::run(lds, tw, load, store);
    }
}

// ---------------------------------------------------------------------------
// Strided batched pass with the next tile's input in flight (the default
// form of k_strided).  Persistent blocks walk work items (a, job, column
// tile); item order puts neighbouring column tiles of one row on the same
// XCD at the same time (they share cache lines).  Per item:
//   stage 0 reads the staged input tile [row][TB] (TIN) from LDS, with the
//   pruning and the i k derivative of k_strided; after its barrier the
//   block issues the asynchronous global->LDS copy (dma16) of the next
//   item's tile; the remaining stages run on fbuf; the last stage writes
//   fbuf; then each wave waits for its own copies and the block writes the
//   output tile from fbuf to global memory, so the wait never covers the
//   item's fresh stores.
// Requires the column tile rounded up to TB to stay inside the input
// buffers (StridedArgs::padded_ok, checked by the host).
// ---------------------------------------------------------------------------
template <int L, int DIR>
__host__ __device__ constexpr int sstage_rows()
{
    return DIR > 0 ? (2 * L) / 3 + 2 : L;  // pruned inverse input: N + 1 rows of M = 3N/2
}

template <int L, int TB>
__host__ __device__ constexpr int sstage_nt()
{
    int m = 0;
    for (int s = 0; s < Plan<L>::n; s++) {
        const int b = (L / Plan<L>::r(s)) * TB;
        m = b > m ? b : m;
    }
    m = (m + 63) / 64 * 64;
    return m > 1024 ? 1024 : (m < 64 ? 64 : m);
}

// NBM = 2: the transform holds 2 TB columns (the combined dual job below).
template <typename TIN, typename T, int L, int TB, int DIR, int NBM = 1>
__host__ __device__ constexpr size_t sstage_lds_bytes()
{
    return sizeof(cx<T>) * ((size_t)L * TB * NBM + fft_twiddle_span<L, sizeof(T) == 8 ? 1 : 2>()) +
           sizeof(cx<TIN>) * (size_t)sstage_rows<L, DIR>() * TB;
}

template <typename TIN, typename T, int L, int TB, int DIR, int NBM = 1>
__host__ __device__ constexpr bool sstage_fits()
{
    return sstage_lds_bytes<TIN, T, L, TB, DIR, NBM>() <= 160 * 1024 - 512 && (TB * sizeof(cx<TIN>)) % 16 == 0;
}

// STDP: inverse pass at the standard 3/2 padding (nin = 2 (L/3) + 1 stored
// rows) with L/R0 = 64 or 128 and one stage-0 butterfly per thread; the zone
// of each stage-0 input (stored low rows, stored high rows, zero padding) is
// then fixed at compile time.
// JSEL picks the jobs a launch takes: 0 all of them; 1 the dual jobs, each
// item as one transform of 2 TB columns (columns b < TB plain, b >= TB the
// i k transform of column b - TB, both formed from one staged tile), so the
// next item's copy is issued after the one shared stage 0 and stays in
// flight across both transforms; 2 the single jobs.
template <typename TIN, typename TOUT, typename T, int L, int TB, int NT, int DIR, bool STDP = false, int JSEL = 0>
__device__ __forceinline__ void sstage_body(const StridedArgs& a)
{
    constexpr int NB = JSEL == 1 ? 2 * TB : TB;  // columns of the transform (and LDS row pitch of fbuf)
    static_assert((TB & (TB - 1)) == 0, "column tile must be a power of two");
    constexpr int SROWS = sstage_rows<L, DIR>();
    constexpr int SPR = TB * (int)sizeof(cx<TIN>) / 16;  // 16-byte copy slots per staged row
    constexpr int EPS = 16 / (int)sizeof(cx<TIN>);        // input elements per slot
    constexpr int NW = NT / 64;
    constexpr int TWM = sizeof(T) == 8 ? 1 : 2;
    constexpr int TWN = fft_twiddle_span<L, TWM>();  // the table entries the transform reads
    __shared__ __align__(16) cx<T> fbuf[L * NB];
    __shared__ __align__(16) cx<TIN> stg[SROWS * TB];
    __shared__ __align__(16) cx<T> twl[TWN];
    if (a.skip && *a.skip) return;  // uniform: every thread reads the same flag
    const int t = threadIdx.x;
    const int hin = a.nin / 2, hout = a.nout / 2;
    const int ntiles = (a.B + TB - 1) / TB;
    // the launch's jobs as 4-bit job indices (at most 9 jobs)
    uint64_t jsel = 0;
    int nsel = 0;
    for (int j = 0; j < a.njobs; j++) {
        const bool d = a.job[j].out2 != nullptr;
        if (JSEL == 0 || (JSEL == 1) == d) {
            jsel |= (uint64_t)j << (4 * nsel);
            nsel++;
        }
    }
    const int64_t per_a = (int64_t)nsel * ntiles;
    const int64_t nitems = (int64_t)a.A * per_a;
    const int G = gridDim.x;  // a multiple of 8
    const int64_t lin = (int64_t)(blockIdx.x % 8) * (G / 8) + blockIdx.x / 8;

    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const uint32_t stg_base = lds_addr(stg);
    const int nslot = a.nin * SPR;
    auto issue = [&](int64_t it) {
        const int64_t ai = it / per_a;
        const int r = (int)(it - ai * per_a);
        const int js = r / ntiles, b0 = (r - js * ntiles) * TB;
        const int jb = (int)((jsel >> (4 * js)) & 15);
        const cx<TIN>* in = (const cx<TIN>*)a.job[jb].in + ai * a.in_a_stride + b0;
        for (int m = wave; m * 64 < nslot; m += NW) {
            const int s = m * 64 + lane;
            const int row = s / SPR, part = s - row * SPR;
            if (s < nslot) dma16(in + (int64_t)row * a.in_row_stride + part * EPS, stg_base + (uint32_t)m * 1024u);
        }
    };

    int64_t it = lin;
    if (it < nitems) issue(it);  // in flight while the twiddles are read
    for (int i = t; i < TWN; i += NT) twl[i] = ((const cx<T>*)a.tw)[i];
    dma_wait();
    lds_barrier();
    for (; it < nitems; it += G) {
        const int64_t ai = it / per_a;
        const int r = (int)(it - ai * per_a);
        const int js = r / ntiles, b0 = (r - js * ntiles) * TB;
        const int jb = (int)((jsel >> (4 * js)) & 15);
        const bool dual = JSEL == 1 || (JSEL == 0 && a.job[jb].out2 != nullptr);
        int deriv = dual ? 0 : a.job[jb].deriv;
        const int64_t nxt = it + G;
        auto load = [&](int b, int p) -> cx<T> {
            int i, k;
            if (a.nin == L) { i = p; k = (p <= L / 2) ? p : p - L; }
            else if (p <= hin) { i = p; k = p; }
            else if (p >= L - hin) { i = a.nin - (L - p); k = p - L; }
            else return cx<T>{(T)0, (T)0};
            const cx<TIN> v = stg[i * TB + (b & (TB - 1))];
            if (JSEL == 1 ? b >= TB : deriv) return times_ik<T>((TIN)k, v);
            return cx<T>{(T)v.x, (T)v.y};
        };
        auto load_std = [&](int b, int j, auto rc) -> cx<T> {
            constexpr int r = decltype(rc)::value;
            constexpr int LR0 = L / Plan<L>::r(0);
            constexpr int p0 = LR0 * r;
            constexpr int H = L / 3, NIN = 2 * H + 1;
            constexpr bool LO = p0 + LR0 - 1 <= H, HI = p0 >= L - H, ZERO = p0 > H && p0 + LR0 - 1 < L - H;
            if constexpr (ZERO) {
                return cx<T>{(T)0, (T)0};
            } else {
                const int p = p0 + j;
                bool lo = LO, hi = HI;
                if constexpr (!LO && !HI) {
                    lo = p <= H;
                    hi = p >= L - H;
                    if (!(lo || hi)) return cx<T>{(T)0, (T)0};
                }
                const int i = lo ? p : p - (L - NIN);
                const cx<TIN> v = stg[i * TB + (b & (TB - 1))];
                if (JSEL == 1 ? b >= TB : deriv) return times_ik<T>((TIN)(lo ? p : p - L), v);
                return cx<T>{(T)v.x, (T)v.y};
            }
        };
        auto store_lds = [&](int b, int p, cx<T> v) { fbuf[p * NB + b] = v; };
        auto prefetch = [&]() {
            if (nxt < nitems) issue(nxt);
        };
        // output tile from fbuf columns [0, TB) (and [TB, 2 TB) into dst2)
        auto write_tile = [&](void* dst, void* dst2) {
            cx<TOUT>* out = (cx<TOUT>*)dst + ai * a.out_a_stride + b0;
            cx<TOUT>* out2 = (JSEL == 1) ? (cx<TOUT>*)dst2 + ai * a.out_a_stride + b0 : out;
            for (int idx = t; idx < a.nout * NB; idx += NT) {
                const int i = idx / NB, bq = idx - i * NB, b = bq & (TB - 1);
                const int p = (a.nout == L || i <= hout) ? i : L - (a.nout - i);
                if (b0 + b < a.B) {
                    const cx<T> v = fbuf[p * NB + bq];
                    (bq >= TB ? out2 : out)[(int64_t)i * a.out_row_stride + b] = cx<TOUT>{(TOUT)v.x, (TOUT)v.y};
                }
            }
        };
        auto fft = [&](auto lead, auto& hook) {
            constexpr bool LEAD = decltype(lead)::value;
            if constexpr (STDP)
                FftS<T, L, NB, NT, NB, DIR, false, TWM>::template run<LEAD>(fbuf, twl, load_std, store_lds, hook, t);
            else
                FftS<T, L, NB, NT, NB, DIR, false, TWM>::template run<LEAD>(fbuf, twl, load, store_lds, hook, t);
        };
        if constexpr (JSEL == 1) {
            // both transforms of the dual job at once; the copy of the next
            // item's tile is in flight from the end of stage 0 on
            fft(std::false_type{}, prefetch);
        } else if (dual) {
            // plain transform first, from the staged tile; the tile stays
            // staged (no prefetch yet) for the i k transform below
            auto none = [] {};
            fft(std::false_type{}, none);
            lds_barrier();
            write_tile(a.job[jb].out, nullptr);
            deriv = 1;
            fft(std::true_type{}, prefetch);
        } else {
            fft(std::false_type{}, prefetch);
        }
        lds_barrier();
        dma_wait();  // the next item's tile (this wave's copies) has landed
        if constexpr (JSEL == 1) write_tile(a.job[jb].out, a.job[jb].out2);
        else write_tile(dual ? a.job[jb].out2 : a.job[jb].out, nullptr);
        lds_barrier();  // every wave's copies are in; fbuf is free again
    }
}

template <typename TIN, typename TOUT, typename T, int L, int TB, int NT, int DIR, bool STDP = false, int JSEL = 0>
__global__ __launch_bounds__(NT) void k_sstage(StridedArgs a)
{
    sstage_body<TIN, TOUT, T, L, TB, NT, DIR, STDP, JSEL>(a);
}

// ---------------------------------------------------------------------------
// In-place unpruned transforms of the FFT_package drop-in along y or x, whose
// rows have no pitch (FP32 rows start at odd multiples of 8 bytes).  Persistent
// blocks over column tiles; a thread holds the stage-0 inputs of its butterfly,
// loaded while the tile before is transformed, and the last stage stores to
// global memory itself, so a block needs LDS for the transform alone and several
// fit a CU.  A tile's outputs are its own columns, which no other tile reads, so
// in place is safe with the next tile's loads in flight.  Every twiddle factor is
// read from the table.  Bounded by HBM (one read and one write of the field).
// A whole r2c, this against tiles staged in LDS (one or two blocks a CU), which
// had taken a pass from 2.58 to 2.07 ms (768^3 FP64) and 353 to 132 us (384^3
// FP32): 768^3 FP64 5.54 -> 4.98 ms, 384^3 FP32 351 -> 275 us, 288x144x96 FP32
// 58 -> 47 us, 48^3 26.0 -> 21.6 us.
// ---------------------------------------------------------------------------
// Columns per tile: 128-byte row pieces as far as the threads (at most 1024) and
// the LDS go, which is L = 512.  FP32: 16 (there 668 us a 512^3 transform against 811
// with 8), FP64: 8 (192^3: 76 us against 121 with 16, whose blocks have 1024
// threads; 512^3 r2c 1340 us against 1587 with 4, 256x512x256 392 against 484, where
// the passes before these took 1547 and 455); beyond, the strided passes' tile.
template <typename T, int L>
__host__ __device__ constexpr int line_tb()
{
    return L > 512 ? strided_tb<T, L>() : sizeof(T) == 4 ? 16 : 8;
}

template <typename T, int L, int TB, int NT, int DIR>
__global__ __launch_bounds__(NT) void k_line(StridedArgs a)
{
    constexpr int R0 = Plan<L>::r(0), LR0 = L / R0;
    static_assert(LR0 * TB <= NT, "one stage-0 butterfly a thread");
    __shared__ __align__(16) cx<T> fbuf[L * TB];
    __shared__ __align__(16) cx<T> twl[L];
    const int t = threadIdx.x, b = t % TB, j = t / TB;
    const int ntiles = (a.B + TB - 1) / TB;
    const int64_t nitems = (int64_t)a.A * ntiles;
    const int G = gridDim.x;  // a multiple of 8
    cx<T>* data = (cx<T>*)a.job[0].in;
    cx<T> in[R0];
    // first element of an item's tile; its columns
    auto tile = [&](int64_t it, int& ncol) -> cx<T>* {
        const int64_t ai = it / ntiles;
        const int b0 = (int)(it - ai * ntiles) * TB;
        ncol = min(TB, a.B - b0);
        return data + ai * a.in_a_stride + b0;
    };
    auto fetch = [&](int64_t it) {
        int ncol;
        const cx<T>* src = tile(it, ncol) + b;
        if (j < LR0 && b < ncol) {
#pragma unroll
            for (int r = 0; r < R0; r++) in[r] = src[(int64_t)(j + r * LR0) * a.in_row_stride];
        }
    };
#pragma unroll
    for (int r = 0; r < R0; r++) in[r] = cx<T>{(T)0, (T)0};
    int64_t it = (int64_t)(blockIdx.x % 8) * (G / 8) + blockIdx.x / 8;
    if (it < nitems) fetch(it);
    for (int i = t; i < L; i += NT) twl[i] = ((const cx<T>*)a.tw)[i];
    for (; it < nitems; it += G) {
        int ncol;
        cx<T>* out = tile(it, ncol);
        auto load = [&](int, int, auto rc) -> cx<T> { return in[decltype(rc)::value]; };
        auto store = [&](int bb, int p, cx<T> v) {
            if (bb < ncol) out[(int64_t)p * a.out_row_stride + bb] = v;
        };
        auto next = [&]() {
            if (it + G < nitems) fetch(it + G);
        };
        FftS<T, L, TB, NT, TB, DIR, false, 0>::template run<false>(fbuf, twl, load, store, next, t);
    }
}

template <typename TIN, typename TOUT, typename T, int L, int TB, int NT, int DIR, bool STDP = false, int JSEL = 0>
__global__ __launch_bounds__(NT) void k_sstage_b(const StridedArgs* __restrict__ arr, const int* __restrict__ left)
{
    if (left[blockIdx.y] <= 0) return;
    sstage_body<TIN, TOUT, T, L, TB, NT, DIR, STDP, JSEL>(arr[blockIdx.y]);
}

// ---------------------------------------------------------------------------
// Block reductions
// ---------------------------------------------------------------------------
// Fixed-order sums and maxima: within a wave by DPP moves, then over the waves
// in order through LDS.  (A shuffle goes through LDS: six dependent ones cost
// about 1200 cycles, these about 100.)
// v of the lane DPP control CTRL names, 0 where there is none or its row is not
// in RMASK
template <int CTRL, int RMASK>
__device__ __forceinline__ double dpp_from(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, RMASK, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, RMASK, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ double lane_value(double v, int lane)  // lane: uniform
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Over the wave's 64 lanes (all active): prefixes within each row of 16 (row
// shifts by 1, 2, 4, 8), then row ends into the next rows (broadcasts of lanes
// 15 and 31); lane 63 holds the whole, which every lane returns.
__device__ __forceinline__ double wave_sum(double v)
{
    v = v + dpp_from<0x111, 0xf>(v);
    v = v + dpp_from<0x112, 0xf>(v);
    v = v + dpp_from<0x114, 0xf>(v);
    v = v + dpp_from<0x118, 0xf>(v);
    v = v + dpp_from<0x142, 0xa>(v);
    v = v + dpp_from<0x143, 0xc>(v);
    return lane_value(v, 63);
}

__device__ __forceinline__ double wave_max(double v)  // v >= 0
{
    v = fmax(v, dpp_from<0x111, 0xf>(v));
    v = fmax(v, dpp_from<0x112, 0xf>(v));
    v = fmax(v, dpp_from<0x114, 0xf>(v));
    v = fmax(v, dpp_from<0x118, 0xf>(v));
    v = fmax(v, dpp_from<0x142, 0xa>(v));
    v = fmax(v, dpp_from<0x143, 0xc>(v));
    return lane_value(v, 63);
}

// Sum over the block, in every thread; sh: NT / 64 doubles (free again on return).
template <int NT>
__device__ __forceinline__ double block_sum(double v, double* sh)
{
    constexpr int NW = NT / 64;
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    double r = sh[0];
#pragma unroll
    for (int w = 1; w < NW; w++) r = r + sh[w];
    __syncthreads();
    return r;
}

// NV block-wide values at once (the first NS are sums, the rest maxima of
// values >= 0), for the threads of wave 0; sh: NV NT / 64 doubles.
template <int NT, int NV, int NS>
__device__ __forceinline__ void block_reduce(double* v, double* sh)
{
    constexpr int NW = NT / 64;
#pragma unroll
    for (int i = 0; i < NV; i++) v[i] = i < NS ? wave_sum(v[i]) : wave_max(v[i]);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int i = 0; i < NV; i++) sh[NV * (threadIdx.x >> 6) + i] = v[i];
    }
    __syncthreads();
    if (threadIdx.x < 64) {  // lane i takes value i over the waves
        const int i = threadIdx.x < NV ? threadIdx.x : 0;
        double r = sh[i];
#pragma unroll
        for (int w = 1; w < NW; w++) {
            const double x = sh[NV * w + i];
            r = i < NS ? r + x : fmax(r, x);
        }
#pragma unroll
        for (int k = 0; k < NV; k++) v[k] = lane_value(r, k);
    }
}

// The z pass's block partials, [4] per block: sums s2, s3; the block's CFL
// velocity max(|u|/Ax, |v|/Ay, |w|/Az) (src/HIT_LES.cpp:393) and its sum form.
// k_finalize takes the maxima over the blocks.  (A device-wide atomicMax per
// block instead cost 50 of the 60 us of the 48^3 z pass: its 2304 blocks'
// 64-bit atomics on one address are served one after the other.)  One LDS
// exchange for all six values; sh: 6 NT / 64 doubles.
template <int NT>
__device__ __forceinline__ void z_partials(const ZArgs& a, double mu, double mv, double mw, double vsa, double s2, double s3, double* sh)
{
    double q[6] = {s2, s3, mu, mv, mw, vsa};
    block_reduce<NT, 6, 2>(q, sh);
    if (threadIdx.x == 0) {
        double* o = a.z_partial + 4 * (int64_t)blockIdx.x;
        o[0] = q[0];
        o[1] = q[1];
        o[2] = fmax(q[2] / a.Ax, fmax(q[3] / a.Ay, q[4] / a.Az));
        o[3] = q[5];
    }
}

// Row of pencil pen = y Mx + x in the physical export's [x][y][z] order.
__device__ __forceinline__ int64_t phys_row(const ZArgs& a, int64_t pen)
{
    const uint32_t y = (uint32_t)pen / (uint32_t)a.Mx;
    return (int64_t)((uint32_t)pen - y * (uint32_t)a.Mx) * a.My + y;
}

// ---------------------------------------------------------------------------
// z pass: one (y,x) pencil per block iteration.
// Six paired c2r transforms of length L hold the twelve physical fields
//   (u,v) (w,ux) (uy,uz) (vx,vy) (vz,wx) (wy,wz)
// in LDS as [z][pair]; products are formed in place, then the forward
// transforms of (cx,cy) (cz,-) [DNS] or (cx,cy) (cz,t11) (t21,t22) (t31,t32)
// (t33,-) [LES] are unpacked to half spectra and written over the inputs.
// MODE 0: full step; MODE 1: velocity only (u,v,w -> CFL, optional export).
// ---------------------------------------------------------------------------
template <typename T, int L, int NT, int MODE>
__global__ __launch_bounds__(NT) void k_zpass(ZArgs a)
{
    constexpr int LD = 6;
    __shared__ cx<T> lds[L * LD];
    __shared__ double red[6 * (NT / 64)];
    const cx<T>* tw = (const cx<T>*)a.tw;
    const int nk = a.nk3;
    const int t = threadIdx.x;
    T mu = (T)0, mv = (T)0, mw = (T)0;
    double vmax_sa = 0.0, s2 = 0.0, s3 = 0.0;
    const double iAx = a.Ax, iAy = a.Ay, iAz = a.Az;
    const bool sa = a.sa;

    // Source of each logical field f (0 u,1 v,2 w | 3 ux,4 uy,5 uz | 6 vx,7 vy,8 vz
    // | 9 wx,10 wy,11 wz): X2 slot and whether it is d_z (i k3 times a
    // velocity spectrum).  Resolved once per block so the loads below are
    // branch-free and use no per-lane kernel-argument indexing.
    __shared__ const cx<T>* srcp[12];
    __shared__ int sderiv[12];
    if (t < 12) {
        const int f = t;
        const cx<T>* p = nullptr;
        int dz = 0;
        if (f < 3) p = (const cx<T>*)a.f[f];
        else {
            const int c = (f - 3) / 3, d = (f - 3) % 3;
            if (d == 0) p = (const cx<T>*)a.f[3 + c];
            else if (d == 1) p = (const cx<T>*)a.f[6 + c];
            else { p = (const cx<T>*)a.f[c]; dz = 1; }
        }
        if (MODE == 1 && f >= 3) p = nullptr;  // velocity mode: pairs (u,v), (w,0)
        srcp[f] = p;
        sderiv[f] = dz;
    }
    __syncthreads();

    for (int64_t pen = blockIdx.x; pen < a.npencil; pen += gridDim.x) {
        const int64_t off = pen * a.pitch;
        // -------- inverse: build paired Hermitian spectra and transform.
        // Z[p] = A[p] + i B[p] for 0 <= p < nk, conj(A[L-p]) + i conj(B[L-p])
        // for L-p < nk; only Re of the p = 0 terms enters (as in a c2r).
        constexpr int NPI = (MODE == 0) ? 6 : 2;
        auto load_inv = [&](int b, int p) -> cx<T> {
            const bool lo = p < nk, hi = p > L - nk;
            if (!(lo || hi)) return cx<T>{(T)0, (T)0};
            const int k = lo ? p : L - p;
            const T kk = (T)k;
            const int fa = 2 * b, fb = 2 * b + 1;
            const cx<T>* pa = srcp[fa];
            const cx<T>* pb = srcp[fb];
            cx<T> A = pa[off + k];
            if (sderiv[fa]) A = cx<T>{-kk * A.y, kk * A.x};
            cx<T> B = cx<T>{(T)0, (T)0};
            if (pb) {
                B = pb[off + k];
                if (sderiv[fb]) B = cx<T>{-kk * B.y, kk * B.x};
            }
            const T s = lo ? (T)1 : (T)-1;
            const T ay = (p == 0) ? (T)0 : s * A.y;
            const T by = (p == 0) ? (T)0 : s * B.y;
            return cx<T>{A.x - by, ay + B.x};
        };
        auto store_lds = [&](int b, int p, cx<T> v) { lds[p * LD + b] = v; };
        Fft<T, L, NPI, NT, LD, +1>::run(lds, tw, load_inv, store_lds);
        __syncthreads();

        // -------- physical space
        for (int n = t; n < L; n += NT) {
            cx<T>* row = &lds[n * LD];
            const T u = row[0].x, v = row[0].y, w = row[1].x;
            mu = fmax(mu, fabs(u));
            mv = fmax(mv, fabs(v));
            mw = fmax(mw, fabs(w));
            if (sa) vmax_sa = fmax(vmax_sa, fabs((double)u) / iAx + fabs((double)v) / iAy + fabs((double)w) / iAz);  // src/HIT_LES.cpp:377
            if constexpr (MODE == 1) {
                s2 += (double)u * (double)u + (double)v * (double)v + (double)w * (double)w;  // src/HIT_LES.cpp:1236-1239
                if (a.phys[0]) {
                    const int64_t o = phys_row(a, pen) * L + n;
                    a.phys[0][o] = u;
                    a.phys[1][o] = v;
                    a.phys[2][o] = w;
                }
            } else {
                const T ux = row[1].y, uy = row[2].x, uz = row[2].y;
                const T vx = row[3].x, vy = row[3].y, vz = row[4].x;
                const T wx = row[4].y, wy = row[5].x, wz = row[5].y;
                s2 += (double)ux * (double)ux;
                s3 += (double)ux * (double)ux * (double)ux;
                // advective form (src/HIT_LES.cpp:118-120)
                const T cxv = u * ux + v * uy + w * uz;
                const T cyv = u * vx + v * vy + w * vz;
                const T czv = u * wx + v * wy + w * wz;
                if (a.les) {
                    // Smagorinsky (src/HIT_LES.cpp:130-154)
                    const T ct = (T)a.ct;
                    T ne = (T)2.0 * ux * ux;
                    ne += (T)2.0 * vy * vy;
                    ne += (T)2.0 * wz * wz;
                    ne += (uy + vx) * (uy + vx);
                    ne += (uz + wx) * (uz + wx);
                    ne += (vz + wy) * (vz + wy);
                    ne = ct * sqrt(ne);
                    const T t11 = (T)(-2.0) * ne * ux;
                    const T t21 = (T)(-1.0) * ne * (uy + vx);
                    const T t22 = (T)(-2.0) * ne * vy;
                    const T t31 = (T)(-1.0) * ne * (uz + wx);
                    const T t32 = (T)(-1.0) * ne * (vz + wy);
                    const T t33 = (T)(-2.0) * ne * wz;
                    row[0] = cx<T>{cxv, cyv};
                    row[1] = cx<T>{czv, t11};
                    row[2] = cx<T>{t21, t22};
                    row[3] = cx<T>{t31, t32};
                    row[4] = cx<T>{t33, (T)0};
                } else {
                    row[0] = cx<T>{cxv, cyv};
                    row[1] = cx<T>{czv, (T)0};
                }
            }
        }
        if constexpr (MODE == 0) {
            // -------- forward transforms of the products (in place in LDS)
            auto load_lds = [&](int b, int p) -> cx<T> { return lds[p * LD + b]; };
            if (a.les) Fft<T, L, 5, NT, LD, -1, true>::run(lds, tw, load_lds, store_lds);
            else Fft<T, L, 2, NT, LD, -1, true>::run(lds, tw, load_lds, store_lds);
            __syncthreads();
            // -------- unpack pairs to half spectra, keep k3 < nk
            const int npairs = a.les ? 5 : 2;
            const int nfields = a.les ? 9 : 3;
            for (int idx = t; idx < npairs * nk; idx += NT) {
                const int q = idx / nk, k = idx % nk;
                const cx<T> Z = lds[k * LD + q];
                const cx<T> Zc = lds[((L - k) % L) * LD + q];
                const T h = (T)0.5;
                const cx<T> A = cx<T>{h * (Z.x + Zc.x), h * (Z.y - Zc.y)};
                const cx<T> B = cx<T>{h * (Z.y + Zc.y), h * (Zc.x - Z.x)};
                const int fa = 2 * q, fb = 2 * q + 1;
                ((cx<T>*)a.f[fa])[off + k] = A;
                if (fb < nfields) ((cx<T>*)a.f[fb])[off + k] = B;
            }
        }
        __syncthreads();
    }
    z_partials<NT>(a, (double)mu, (double)mv, (double)mw, vmax_sa, s2, s3, red);
}


// ---------------------------------------------------------------------------
// Velocity-gradient invariants of g[3 i + j] = d u_i / d x_j, in the order
// QG QS RG RS V2 (src/tensor_algebra.cpp:250-303, calc_QO :356):
//   S = 0.5 G + 0.5 G^T, Omega = G - S, Q(T) = 0.5((tr T)^2 - tr(T T)),
//   R(T) = det T (calc_determinant's term order), V2 = 4(tr(S^2 Omega^2) - 2 QS QO),
//   QO = QG - QS.
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void mul3(const T a[9], const T b[9], T ab[9])
{
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            T s = (T)0;
#pragma unroll
            for (int k = 0; k < 3; k++) s += a[3 * i + k] * b[3 * k + j];
            ab[3 * i + j] = s;
        }
}

template <typename T>
__device__ __forceinline__ T second_inv(const T a[9])
{
    T a2[9];
    mul3(a, a, a2);
    const T tr = a[0] + a[4] + a[8], tr2 = a2[0] + a2[4] + a2[8];
    return (T)0.5 * (tr * tr - tr2);
}

template <typename T>
__device__ __forceinline__ T det3(const T t[9])
{
    T d = (T)0;
    d += t[0] * t[4] * t[8];
    d += t[1] * t[5] * t[6];
    d += t[2] * t[3] * t[7];
    d -= t[2] * t[4] * t[6];
    d -= t[1] * t[3] * t[8];
    d -= t[0] * t[5] * t[7];
    return d;
}

template <typename T>
__device__ __forceinline__ void grad_invariants(const T g[9], T out[5])
{
    T S[9], O[9], S2[9], O2[9], S2O2[9];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) S[3 * i + j] = (T)0.5 * g[3 * i + j] + (T)0.5 * g[3 * j + i];
#pragma unroll
    for (int i = 0; i < 9; i++) O[i] = g[i] - S[i];
    const T QG = second_inv(g), QS = second_inv(S);
    mul3(S, S, S2);
    mul3(O, O, O2);
    mul3(S2, O2, S2O2);
    out[0] = QG;
    out[1] = QS;
    out[2] = det3(g);
    out[3] = det3(S);
    out[4] = (T)4.0 * ((S2O2[0] + S2O2[4] + S2O2[8]) - (T)2.0 * QS * (QG - QS));
}

// ---------------------------------------------------------------------------
// z pass with the next pencil's inputs in flight: the velocity-only and
// invariants passes, and the step where the retained k3 count is not that of the
// 3/2 padding (else k_zreg or k_zfuse).
// Same arithmetic as k_zpass, restructured around HBM latency:
//   * the nine half-spectrum source fields of a pencil are staged into LDS
//     as [field][k] (pitch SP = pitch + pad) by asynchronous global->LDS
//     copies (dma16), issued for pencil n+1 as soon as pencil n's first
//     inverse stage has consumed the staging area, so the copy overlaps the
//     rest of pencil n's transforms and products;
//   * all barriers inside the loop are LDS-only (lds_barrier);
//   * twiddles are read from an LDS copy of the table (FftS);
//   * field pointers come from a small LDS table, so no per-lane indexing
//     of kernel arguments.
// Staging capacity is a compile-time maximum (zstage_spc); the launcher
// checks pitch + pad against it and the LDS total against the CU's 160 KB.
// ---------------------------------------------------------------------------
template <int L>
__host__ __device__ constexpr int zstage_spc()
{
    return (L / 3 + 1 + 15) / 16 * 16 + 2;
}

template <typename T>
__host__ __device__ constexpr int zstage_pad()
{
    return sizeof(T) == 8 ? 1 : 2;  // odd pitch (FP64) / even pitch for 16-byte pairs (FP32)
}

template <int MODE>
__host__ __device__ constexpr int zstage_ld()
{
    // LDS row pitch of the pair buffer, in complex elements: one more than the
    // pairs per point, so row-strided accesses (the physical-space loop, the
    // unpack) spread over all banks
    return MODE == 1 ? 3 : 7;
}

template <typename T, int L, int NT, int MODE, int LD = zstage_ld<MODE>()>
__host__ __device__ constexpr size_t zstage_lds_bytes()
{
    return sizeof(cx<T>) * ((size_t)L * LD + (size_t)(MODE == 1 ? 3 : 9) * zstage_spc<L>() + L) +
           sizeof(double) * 6 * (NT / 64) + 2 * 9 * sizeof(void*);
}

template <typename T, int L, int NT, int MODE, int LD = zstage_ld<MODE>()>
__host__ __device__ constexpr bool zstage_fits()
{
    return zstage_lds_bytes<T, L, NT, MODE, LD>() <= 160 * 1024 - 512;
}

// ZOPAQUE: route the thread index through opaque() once per pencil, so the
// compiler recomputes the transforms' per-thread LDS addresses instead of
// holding them in registers across the pencil loop.  In FP32 that takes the
// kernel from 184 to 64-80 VGPRs and two blocks per CU (9.2-9.9 ms against
// 13.7 ms at 512^3); in FP64 the LDS allows one block per CU anyway and the
// recomputation only costs time, so it is off there.
// NKC > 0: the retained k3 count is the compile-time constant NKC (the
// standard 3/2 padding, nk3 = L/3 + 1), so the pruning of the first inverse
// stage resolves at compile time and its zero inputs fold away.
template <typename T, int L, int NT, int MODE, int LD = zstage_ld<MODE>(), int MINW = 1, bool ZOPAQUE = (sizeof(T) == 4),
          int NKC = 0, int TWM = (sizeof(T) == 8 ? 1 : 2)>
__device__ __forceinline__ void zstage_body(const ZArgs& a)
{
    static_assert(LD >= (MODE == 1 ? 2 : 6), "pair buffer pitch too small");
    constexpr int NSRC = (MODE == 1) ? 3 : 9;
    constexpr int SPC = zstage_spc<L>();
    constexpr int NW = NT / 64;
    constexpr int EPS = 16 / (int)sizeof(cx<T>);  // elements per 16-byte copy slot
    __shared__ __align__(16) cx<T> fbuf[L * LD];
    __shared__ __align__(16) cx<T> stg[NSRC * SPC];
    __shared__ __align__(16) cx<T> twl[L];
    __shared__ double red[6 * (NT / 64)];
    __shared__ const cx<T>* srcp[9];
    __shared__ cx<T>* dstp[9];
    const int t = threadIdx.x;
    const int nk = a.nk3, pitch = a.pitch;
    const int SP = pitch + zstage_pad<T>();
    const int nslot = NSRC * SP / EPS;
    T mu = (T)0, mv = (T)0, mw = (T)0;
    double vmax_sa = 0.0, s2 = 0.0, s3 = 0.0;
    const double iAx = a.Ax, iAy = a.Ay, iAz = a.Az;
    const bool sa = a.sa;

    if (t < 9) {
        srcp[t] = (const cx<T>*)a.f[t];
        dstp[t] = (cx<T>*)a.f[t];
    }
    for (int i = t; i < L; i += NT) twl[i] = ((const cx<T>*)a.tw)[i];
    __syncthreads();

    // copy slot s (16 bytes) holds staging elements s*EPS .. s*EPS+EPS-1,
    // element e = field f * SP + k; slots with k >= pitch (the pad) are skipped
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const uint32_t stg_base = lds_addr(stg);
    auto issue = [&](int64_t pen) {
        const int64_t off = pen * (int64_t)pitch;
        for (int m = wave; m * 64 < nslot; m += NW) {
            const int s = m * 64 + lane;
            const int e = s * EPS;
            const int f = e / SP, k = e - f * SP;
            if (s < nslot && k < pitch) dma16(srcp[f] + off + k, stg_base + (uint32_t)m * 1024u);
        }
    };

    // pair b of the inverse: logical fields (2b, 2b+1) of
    //   u v w ux uy uz vx vy vz wx wy wz
    // from source fields (u v w | ux vx wx | uy vy wy); d_z = i k3 * (u v w)
    //   A: u w uy vx vz wy  -> 0 2 6 4 1 8   (d_z for vz)
    //   B: v ux uz vy wx wz -> 1 3 0 7 5 2   (d_z for uz, wz)
    constexpr uint32_t SRC_A = 0x814620u, SRC_B = 0x257031u, DZ_A = 0x10u, DZ_B = 0x24u;

    int64_t pen = blockIdx.x;
    if (pen < a.npencil) issue(pen);
    dma_wait();
    lds_barrier();
    for (; pen < a.npencil; pen += gridDim.x) {
        const int64_t off = pen * (int64_t)pitch;
        const int64_t nxt = pen + gridDim.x;
        constexpr int NPI = (MODE == 1) ? 2 : 6;
        const int tl = ZOPAQUE ? opaque(t) : t;
        auto load_inv = [&](int b, int p) -> cx<T> {
            const int nkv = NKC > 0 ? NKC : nk;
            const bool lo = p < nkv, hi = p > L - nkv;
            if (!(lo || hi)) return cx<T>{(T)0, (T)0};
            const int k = lo ? p : L - p;
            const T kk = (T)k;
            const int fa = (SRC_A >> (4 * b)) & 15, fb = (SRC_B >> (4 * b)) & 15;
            cx<T> A = stg[fa * SP + k];
            if ((DZ_A >> b) & 1) A = cx<T>{-kk * A.y, kk * A.x};
            cx<T> B = cx<T>{(T)0, (T)0};
            if (MODE != 1 || b == 0) {
                B = stg[fb * SP + k];
                if ((DZ_B >> b) & 1) B = cx<T>{-kk * B.y, kk * B.x};
            }
            const T s = lo ? (T)1 : (T)-1;
            const T ay = (p == 0) ? (T)0 : s * A.y;
            const T by = (p == 0) ? (T)0 : s * B.y;
            return cx<T>{A.x - by, ay + B.x};
        };
        auto store_lds = [&](int b, int p, cx<T> v) { fbuf[p * LD + b] = v; };
        auto prefetch = [&]() {
            if (nxt < a.npencil) issue(nxt);
        };
        auto none = [&]() {};
        FftS<T, L, NPI, NT, LD, +1, false, TWM, sizeof(T) == 4>::template run<false>(fbuf, twl, load_inv, store_lds, prefetch, tl);
        lds_barrier();

        // -------- physical space
        for (int n = t; n < L; n += NT) {
            cx<T>* row = &fbuf[n * LD];
            if constexpr (MODE == 2) {
                // velocity-gradient invariants QG QS RG RS V2 (src/HIT_LES.cpp:1297-1319)
                const T g[9] = {row[1].y, row[2].x, row[2].y, row[3].x, row[3].y, row[4].x, row[4].y, row[5].x, row[5].y};
                T q[5];
                grad_invariants(g, q);
                row[0] = cx<T>{q[0], q[1]};
                row[1] = cx<T>{q[2], q[3]};
                row[2] = cx<T>{q[4], (T)0};
                continue;
            }
            const T u = row[0].x, v = row[0].y, w = row[1].x;
            mu = fmax(mu, fabs(u));
            mv = fmax(mv, fabs(v));
            mw = fmax(mw, fabs(w));
            if (sa) vmax_sa = fmax(vmax_sa, fabs((double)u) / iAx + fabs((double)v) / iAy + fabs((double)w) / iAz);  // src/HIT_LES.cpp:377
            if constexpr (MODE == 1) {
                s2 += (double)u * (double)u + (double)v * (double)v + (double)w * (double)w;  // src/HIT_LES.cpp:1236-1239
                if (a.phys[0]) {
                    const int64_t o = phys_row(a, pen) * L + n;
                    a.phys[0][o] = u;
                    a.phys[1][o] = v;
                    a.phys[2][o] = w;
                }
            } else {
                const T ux = row[1].y, uy = row[2].x, uz = row[2].y;
                const T vx = row[3].x, vy = row[3].y, vz = row[4].x;
                const T wx = row[4].y, wy = row[5].x, wz = row[5].y;
                s2 += (double)ux * (double)ux;
                s3 += (double)ux * (double)ux * (double)ux;
                // advective form (src/HIT_LES.cpp:118-120)
                const T cxv = u * ux + v * uy + w * uz;
                const T cyv = u * vx + v * vy + w * vz;
                const T czv = u * wx + v * wy + w * wz;
                if (a.les) {
                    // Smagorinsky (src/HIT_LES.cpp:130-154)
                    const T ct = (T)a.ct;
                    T ne = (T)2.0 * ux * ux;
                    ne += (T)2.0 * vy * vy;
                    ne += (T)2.0 * wz * wz;
                    ne += (uy + vx) * (uy + vx);
                    ne += (uz + wx) * (uz + wx);
                    ne += (vz + wy) * (vz + wy);
                    ne = ct * sqrt(ne);
                    row[0] = cx<T>{cxv, cyv};
                    row[1] = cx<T>{czv, (T)(-2.0) * ne * ux};
                    row[2] = cx<T>{(T)(-1.0) * ne * (uy + vx), (T)(-2.0) * ne * vy};
                    row[3] = cx<T>{(T)(-1.0) * ne * (uz + wx), (T)(-1.0) * ne * (vz + wy)};
                    row[4] = cx<T>{(T)(-2.0) * ne * wz, (T)0};
                } else {
                    row[0] = cx<T>{cxv, cyv};
                    row[1] = cx<T>{czv, (T)0};
                }
            }
        }
        if constexpr (MODE == 2) {
            auto load_lds = [&](int b, int p) -> cx<T> { return fbuf[p * LD + b]; };
            FftS<T, L, 3, NT, LD, -1, true, TWM>::template run<true>(fbuf, twl, load_lds, store_lds, none, tl);
            lds_barrier();
            dma_wait();
            for (int idx = t; idx < 3 * nk; idx += NT) {
                const int q = idx / nk, k = idx - q * nk;
                const cx<T> Z = fbuf[k * LD + q];
                const cx<T> Zc = fbuf[((L - k) % L) * LD + q];
                const T h = (T)0.5;
                dstp[2 * q][off + k] = cx<T>{h * (Z.x + Zc.x), h * (Z.y - Zc.y)};
                if (q < 2) dstp[2 * q + 1][off + k] = cx<T>{h * (Z.y + Zc.y), h * (Zc.x - Z.x)};
            }
        } else if constexpr (MODE == 0) {
            auto load_lds = [&](int b, int p) -> cx<T> { return fbuf[p * LD + b]; };
            if (a.les) FftS<T, L, 5, NT, LD, -1, true, TWM>::template run<true>(fbuf, twl, load_lds, store_lds, none, tl);
            else FftS<T, L, 2, NT, LD, -1, true, TWM>::template run<true>(fbuf, twl, load_lds, store_lds, none, tl);
            lds_barrier();
            dma_wait();  // the next pencil's sources (this wave's copies) have landed
            const int npairs = a.les ? 5 : 2;
            const int nfields = a.les ? 9 : 3;
            for (int idx = t; idx < npairs * nk; idx += NT) {
                const int q = idx / nk, k = idx - q * nk;
                const cx<T> Z = fbuf[k * LD + q];
                const cx<T> Zc = fbuf[((L - k) % L) * LD + q];
                const T h = (T)0.5;
                const cx<T> A = cx<T>{h * (Z.x + Zc.x), h * (Z.y - Zc.y)};
                const cx<T> B = cx<T>{h * (Z.y + Zc.y), h * (Zc.x - Z.x)};
                dstp[2 * q][off + k] = A;
                if (2 * q + 1 < nfields) dstp[2 * q + 1][off + k] = B;
            }
        } else {
            dma_wait();
        }
        lds_barrier();  // every wave's copies are in; fbuf is free again
    }
    if constexpr (MODE == 2) return;  // a diagnostic pass: no CFL or skewness partials
    z_partials<NT>(a, (double)mu, (double)mv, (double)mw, vmax_sa, s2, s3, red);
}

template <typename T, int L, int NT, int MODE, int LD = zstage_ld<MODE>(), int MINW = 1, bool ZOPAQUE = (sizeof(T) == 4),
          int NKC = 0, int TWM = (sizeof(T) == 8 ? 1 : 2)>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(MINW))) void k_zstage(ZArgs a)
{
    zstage_body<T, L, NT, MODE, LD, MINW, ZOPAQUE, NKC, TWM>(a);
}

template <typename T, int L, int NT, int MODE, int LD = zstage_ld<MODE>(), int MINW = 1, bool ZOPAQUE = (sizeof(T) == 4),
          int NKC = 0, int TWM = (sizeof(T) == 8 ? 1 : 2)>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(MINW))) void k_zstage_b(const ZArgs* __restrict__ arr,
                                                                                           const int* __restrict__ left)
{
    if (left[blockIdx.y] <= 0) return;
    zstage_body<T, L, NT, MODE, LD, MINW, ZOPAQUE, NKC, TWM>(arr[blockIdx.y]);
}

// ---------------------------------------------------------------------------
// DNS z pass with the forward transforms of pencil n-1 folded into the
// inverse transforms of pencil n (DNS from 768 points, FP32 at 288 and 384 too;
// k_zreg elsewhere).
// One Stockham transform of 8 columns per pencil step:
//   columns 0-5: the six paired c2r inputs of pencil n (from the staging
//                area, as in k_zstage);
//   columns 6-7: the products (cx, cy) and (cz, 0) of pencil n-1, written
//                by the previous step's physical-space loop.
// All columns run as inverse transforms; the forward ones through
// conj(inverse(conj x)), so one set of twiddles and butterflies serves both
// and every stage keeps all threads busy (768 = 64 x 12: 512 then 768
// butterflies at 768 threads).  Per step: the transform (the staging copy
// of pencil n+1 is issued after its first stage), then the unpack of
// pencil n-1's half spectra, then pencil n's products into columns 6-7.
// The loop runs one step past the block's last pencil to finish it.
// LDS row pitch 9 (odd), twiddle table trimmed to the entries read.  In FP32
// stage 0 maps threads column-major (one column per wave, so the loader runs
// without divergence: 8.96 -> 8.67 ms at 512^3); in FP64 the column-major
// stage-0 writes conflict in LDS and cost more than that saves.
// ---------------------------------------------------------------------------
// Pair buffer layout: the swizzled 8-column form of FftS where its index
// algebra applies and the compile-time stage-0 loader runs (L/R0 = 64 or 128:
// 768 and 1536), else pitch 9.
template <typename T, int L>
__host__ __device__ constexpr bool zfuse_swz()
{
    return fft_swz_ok<L, (int)sizeof(cx<T>)>() && (L / Plan<L>::r(0) == 64 || L / Plan<L>::r(0) == 128);
}

template <typename T, int L, int NT, int NKC, int TWM = (sizeof(T) == 8 ? 1 : 2)>
__host__ __device__ constexpr size_t zfuse_lds_bytes()
{
    return sizeof(cx<T>) * ((size_t)L * (zfuse_swz<T, L>() ? 8 : 9) + (size_t)9 * zstage_spc<L>() + fft_twiddle_span<L, TWM>()) +
           3 * 9 * sizeof(void*);
}

template <typename T, int L, int NT, int NKC = 0, int TWM = (sizeof(T) == 8 ? 1 : 2), bool ZOPAQUE = (sizeof(T) == 4)>
__device__ __forceinline__ void zfuse_body(const ZArgs& a)
{
    constexpr bool SWZ = zfuse_swz<T, L>();
    constexpr int LD = SWZ ? 8 : 9, NB = 8;
    constexpr int SPC = zstage_spc<L>();
    constexpr int NW = NT / 64;
    constexpr int EPS = 16 / (int)sizeof(cx<T>);
    constexpr int TWN = fft_twiddle_span<L, TWM>();
    static_assert(L * LD * sizeof(cx<T>) >= 6 * (NT / 64) * sizeof(double), "reduction scratch aliases the pair buffer");
    __shared__ __align__(16) cx<T> fbuf[L * LD];
    __shared__ __align__(16) cx<T> stg[9 * SPC];
    __shared__ __align__(16) cx<T> twl[TWN];
    __shared__ const cx<T>* srcp[9];
    const int t = threadIdx.x;
    const int nk = a.nk3, pitch = a.pitch;
    const int SP = pitch + zstage_pad<T>();
    const int nslot = 9 * SP / EPS;
    T mu = (T)0, mv = (T)0, mw = (T)0;
    double vmax_sa = 0.0, s2 = 0.0, s3 = 0.0;
    const double iAx = a.Ax, iAy = a.Ay, iAz = a.Az;
    const bool sa = a.sa;
    // element (row, column) of the pair buffer
    auto fidx = [](int row, int col) -> int { return SWZ ? fft_swz<(int)sizeof(cx<T>)>(row, col) : row * LD + col; };

    if (t < 9) srcp[t] = (const cx<T>*)a.f[t];
    for (int i = t; i < TWN; i += NT) twl[i] = ((const cx<T>*)a.tw)[i];
    __syncthreads();

    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const uint32_t stg_base = lds_addr(stg);
    // Staging copies: slot m (16 bytes per lane) of wave m % NW.  Each lane's
    // source pointer (field f, k3 = k) is the same for every pencil up to the
    // pencil offset, so it is formed once here.
    constexpr int MAXM = (9 * (SPC + zstage_pad<T>()) / EPS + 64 * NW - 1) / (64 * NW);
    const cx<T>* gsrc[MAXM];
    bool gok[MAXM];
#pragma unroll
    for (int i = 0; i < MAXM; i++) {
        const int m = wave + i * NW;
        const int s = m * 64 + lane;
        const int e = s * EPS;
        const int f = e / SP, k = e - f * SP;
        gok[i] = s < nslot && k < pitch;
        gsrc[i] = srcp[gok[i] ? f : 0] + (gok[i] ? k : 0);
    }
    auto issue = [&](int64_t pen) {
        const int64_t off = pen * (int64_t)pitch;
#pragma unroll
        for (int i = 0; i < MAXM; i++) {
            const int m = wave + i * NW;
            if (m * 64 < nslot && gok[i]) dma16(gsrc[i] + off, stg_base + (uint32_t)m * 1024u);
        }
    };
    // inverse pair b (0..5): logical fields (2b, 2b+1) of u v w ux uy uz vx vy vz wx wy wz
    constexpr uint32_t SRC_A = 0x814620u, SRC_B = 0x257031u, DZ_A = 0x10u, DZ_B = 0x24u;
    // compile-time stage-0 loader: needs the compile-time k3 count, L/R0 = 64
    // or 128 and at most one stage-0 butterfly per thread
    constexpr int LR0 = L / Plan<L>::r(0);
    constexpr bool FAST = NKC > 0 && (LR0 == 64 || LR0 == 128) && NB * LR0 <= NT;
    constexpr bool S0COL = sizeof(T) == 4;  // column-major stage 0 in FP32 (its writes conflict in FP64)

    int64_t pen = blockIdx.x;
    if (pen < a.npencil) issue(pen);
    dma_wait();
    lds_barrier();
    int64_t prev = -1;  // pencil whose products sit in columns 6-7
    for (;; pen += gridDim.x) {
        const bool have = pen < a.npencil;
        const bool havep = prev >= 0;
        if (!have && !havep) break;
        const int tl = ZOPAQUE ? opaque(t) : t;
        const int64_t nxt = pen + gridDim.x;
        auto load = [&](int b, int p) -> cx<T> {
            if (b >= 6) {
                if (!havep) return cx<T>{(T)0, (T)0};
                const cx<T> v = fbuf[fidx(p, b)];
                return cx<T>{v.x, -v.y};  // forward = conj(inverse(conj x))
            }
            if (!have) return cx<T>{(T)0, (T)0};
            const int nkv = NKC > 0 ? NKC : nk;
            const bool lo = p < nkv, hi = p > L - nkv;
            if (!(lo || hi)) return cx<T>{(T)0, (T)0};
            const int k = lo ? p : L - p;
            const T kk = (T)k;
            const int fa = (SRC_A >> (4 * b)) & 15, fb = (SRC_B >> (4 * b)) & 15;
            cx<T> A = stg[fa * SP + k];
            if ((DZ_A >> b) & 1) A = cx<T>{-kk * A.y, kk * A.x};
            cx<T> B = stg[fb * SP + k];
            if ((DZ_B >> b) & 1) B = cx<T>{-kk * B.y, kk * B.x};
            const T s = lo ? (T)1 : (T)-1;
            const T ay = (p == 0) ? (T)0 : s * A.y;
            const T by = (p == 0) ? (T)0 : s * B.y;
            return cx<T>{A.x - by, ay + B.x};
        };
        // Fast loader.  With L/R0 = LR0 (64 or 128) and one stage-0 butterfly
        // per thread, input p = LR0 r + j with j < LR0, so the zone of p
        // (direct k3 = p, mirrored k3 = L - p, or zero padding) is fixed for
        // each r at compile time.  The thread's column is the wave index over
        // LR0 / 64 (a scalar) when stage 0 is column-major, else t mod 8.  Columns pair each velocity component
        // with its own z derivative, (f, i k f) -> (1 - k) f direct and
        // (1 + k) conj f mirrored (one read, no derivative product), then
        // (fx, fy) of u, v, w.
        const int col = S0COL ? wave / (LR0 / 64) : (tl & (NB - 1));
        const cx<T>* pa = stg + col * SP;        // f (columns 0-2) or fx (3-5)
        const cx<T>* pb = stg + (col + 3) * SP;  // fy (columns 3-5)
        auto load_fast = [&](int, int j, auto rc) -> cx<T> {
            constexpr int r = decltype(rc)::value;
            constexpr int p0 = LR0 * r;
            if (col >= 6) {
                if (!havep) return cx<T>{(T)0, (T)0};
                const cx<T> v = fbuf[fidx(p0 + j, col)];
                return cx<T>{v.x, -v.y};  // forward = conj(inverse(conj x))
            }
            if (!have) return cx<T>{(T)0, (T)0};
            constexpr bool LO = p0 + LR0 - 1 < NKC, HI = p0 > L - NKC, ZERO = p0 >= NKC && p0 + LR0 - 1 <= L - NKC;
            if constexpr (ZERO) {
                return cx<T>{(T)0, (T)0};
            } else {
                const int p = p0 + j;
                bool lo = LO, hi = HI;
                if constexpr (!LO && !HI) {
                    lo = p < NKC;
                    hi = p > L - NKC;
                    if (!(lo || hi)) return cx<T>{(T)0, (T)0};
                }
                const int k = lo ? p : L - p;
                const cx<T> A = pa[k];
                T ay = lo ? A.y : -A.y;
                if constexpr (r == 0) {
                    if (j == 0) ay = (T)0;  // the k3 = 0 imaginary part is dropped, as by a c2r
                }
                if (col < 3) {
                    const T sc = lo ? (T)1 - (T)k : (T)1 + (T)k;
                    return cx<T>{sc * A.x, sc * ay};
                }
                const cx<T> B = pb[k];
                T by = lo ? B.y : -B.y;
                if constexpr (r == 0) {
                    if (j == 0) by = (T)0;
                }
                return cx<T>{A.x - by, ay + B.x};
            }
        };
        auto store = [&](int b, int p, cx<T> v) { fbuf[p * LD + b] = (b >= 6) ? cx<T>{v.x, -v.y} : v; };
        auto store_swz = [&](int b, int, int li, cx<T> v) { fbuf[li] = (b >= 6) ? cx<T>{v.x, -v.y} : v; };
        auto prefetch = [&]() {
            if (have && nxt < a.npencil) issue(nxt);
        };
        if constexpr (SWZ) {
            static_assert(FAST, "the swizzled layout is only built with the compile-time loader");
            FftS<T, L, NB, NT, LD, +1, true, TWM, S0COL, true>::template run<false>(fbuf, twl, load_fast, store_swz, prefetch, tl);
        } else if constexpr (FAST) {
            FftS<T, L, NB, NT, LD, +1, true, TWM, S0COL>::template run<false>(fbuf, twl, load_fast, store, prefetch, tl);
        } else {
            FftS<T, L, NB, NT, LD, +1, true, TWM, S0COL>::template run<false>(fbuf, twl, load, store, prefetch, tl);
        }
        lds_barrier();
        dma_wait();  // pencil n+1's sources (this wave's copies) have landed
        if (havep) {
            // -------- unpack pencil n-1: (cx, cy) and (cz, -) half spectra
            const int64_t offp = prev * (int64_t)pitch;
            const int nkv = NKC > 0 ? NKC : nk;
            cx<T>* const d0 = (cx<T>*)a.f[0] + offp;
            cx<T>* const d1 = (cx<T>*)a.f[1] + offp;
            cx<T>* const d2 = (cx<T>*)a.f[2] + offp;
            for (int idx = t; idx < 2 * nkv; idx += NT) {
                const int q = idx >= nkv ? 1 : 0, k = idx - q * nkv;
                const cx<T> Z = fbuf[fidx(k, 6 + q)];
                const cx<T> Zc = fbuf[fidx(k == 0 ? 0 : L - k, 6 + q)];
                const T h = (T)0.5;
                (q ? d2 : d0)[k] = cx<T>{h * (Z.x + Zc.x), h * (Z.y - Zc.y)};
                if (q == 0) d1[k] = cx<T>{h * (Z.y + Zc.y), h * (Zc.x - Z.x)};
            }
            lds_barrier();
        }
        if (have) {
            // -------- physical space of pencil n: products into columns 6-7
            for (int n = t; n < L; n += NT) {
                // the row's 8 elements: 8n + c, XORed with the row's swizzle
                const int rb = SWZ ? 8 * n : n * LD, rh = SWZ ? fft_swz<(int)sizeof(cx<T>)>(n, 0) ^ (8 * n) : 0;
                auto row = [&](int c) -> cx<T>& { return fbuf[SWZ ? ((rb + c) ^ rh) : rb + c]; };
                T u, v, w, ux, uy, uz, vx, vy, vz, wx, wy, wz;
                if constexpr (FAST) {
                    u = row(0).x, uz = row(0).y, v = row(1).x, vz = row(1).y, w = row(2).x, wz = row(2).y;
                    ux = row(3).x, uy = row(3).y, vx = row(4).x, vy = row(4).y, wx = row(5).x, wy = row(5).y;
                } else {
                    u = row(0).x, v = row(0).y, w = row(1).x;
                    ux = row(1).y, uy = row(2).x, uz = row(2).y;
                    vx = row(3).x, vy = row(3).y, vz = row(4).x;
                    wx = row(4).y, wy = row(5).x, wz = row(5).y;
                }
                mu = fmax(mu, fabs(u));
                mv = fmax(mv, fabs(v));
                mw = fmax(mw, fabs(w));
                if (sa) vmax_sa = fmax(vmax_sa, fabs((double)u) / iAx + fabs((double)v) / iAy + fabs((double)w) / iAz);  // src/HIT_LES.cpp:377
                s2 += (double)ux * (double)ux;
                s3 += (double)ux * (double)ux * (double)ux;
                // advective form (src/HIT_LES.cpp:118-120)
                row(6) = cx<T>{u * ux + v * uy + w * uz, u * vx + v * vy + w * vz};
                row(7) = cx<T>{u * wx + v * wy + w * wz, (T)0};
            }
            lds_barrier();
        }
        prev = have ? pen : -1;
    }
    z_partials<NT>(a, (double)mu, (double)mv, (double)mw, vmax_sa, s2, s3, (double*)fbuf);
}

template <typename T, int L, int NT, int NKC = 0, int TWM = (sizeof(T) == 8 ? 1 : 2), bool ZOPAQUE = (sizeof(T) == 4)>
__global__ __launch_bounds__(NT) void k_zfuse(ZArgs a)
{
    zfuse_body<T, L, NT, NKC, TWM, ZOPAQUE>(a);
}

template <typename T, int L, int NT, int NKC = 0, int TWM = (sizeof(T) == 8 ? 1 : 2), bool ZOPAQUE = (sizeof(T) == 4)>
__global__ __launch_bounds__(NT) void k_zfuse_b(const ZArgs* __restrict__ arr, const int* __restrict__ left)
{
    if (left[blockIdx.y] <= 0) return;
    zfuse_body<T, L, NT, NKC, TWM, ZOPAQUE>(arr[blockIdx.y]);
}

// ---------------------------------------------------------------------------
// z pass with the next pencils' inputs held in registers (the default at the
// standard 3/2 padding for every LES and for DNS below L = 768).
// A block takes PP pencils at a time.  Each thread holds its share of their
// spectra (pair column b, k3 = k), loaded one group ahead, and spreads it into
// the pair buffer as Z[k] and Z[L - k]; nothing is staged in LDS, and what the
// pairing costs is paid once per (k, column) instead of once per transform
// input.  The buffer's columns are c PP + pp (pair c of pencil pp), so each
// point's products stay in that point's own columns.
//   LES: 6 PP inverse columns, products in place, 5 PP forward columns.
//   DNS: one transform of 8 PP columns; the last 2 PP are the products of the
//   previous group, run forward as conj(inverse(conj x)) (as k_zfuse does).
// What bounds it: LDS and the latency between barriers in FP64 (so the room the
// staging area took goes to more blocks per CU), vector-ALU issue in FP32 at
// short lengths (so PP is taken to fill whole waves with butterflies).
// z pass, one run: 256^3 LES 2.93 -> 2.34 ms FP64, 1.43 -> 1.18 FP32; 192^3 DNS
// FP64 1.01 -> 0.66; 128^3 DNS FP64 243 -> 181 us; 16 x 64^3 DNS FP32 359 -> 261 us.
// Long LES pencils (192 x 192 of them; from 768 on 1024 threads spill in FP64, 20 to
// 177 registers): 768 FP64 1.40 -> 1.27 ms, FP32 0.73 -> 0.65; 1152 9.5 -> 3.0, 1.38 ->
// 1.11; 1536 13.7 -> 4.8, 1.78 -> 1.45 (FP64 there against the unstaged k_zpass).
// ---------------------------------------------------------------------------
// Pair (A, B) at k3 = k: Z[k] (lo) and Z[L - k] (hi) of A + i B; dza / dzb: the
// field is d_z of the one read.  Only the real part of k3 = 0 enters (as in a
// c2r).  Products are rounded before the sums, as in every loader of these pairs.
template <typename T>
__device__ __forceinline__ void z_pair(cx<T> A, cx<T> B, int k, bool dza, bool dzb, cx<T>& lo, cx<T>& hi)
{
#pragma clang fp contract(off)
    const T kk = (T)k;
    if (dza) A = cx<T>{-kk * A.y, kk * A.x};
    if (dzb) B = cx<T>{-kk * B.y, kk * B.x};
    if (k == 0) A.y = B.y = (T)0;
    lo = cx<T>{A.x - B.y, A.y + B.x};
    hi = cx<T>{A.x + B.y, B.x - A.y};
}

// (f, d_z f) = (1 - k) f and (1 + k) conj f
template <typename T>
__device__ __forceinline__ void z_pair_dz(cx<T> A, int k, cx<T>& lo, cx<T>& hi)
{
#pragma clang fp contract(off)
    const T a = (T)1 - (T)k, b = (T)1 + (T)k;
    if (k == 0) A.y = (T)0;
    lo = cx<T>{a * A.x, a * A.y};
    hi = cx<T>{b * A.x, b * -A.y};
}

// Pencils per block: two at the short DNS lengths, so that butterflies fill whole
// waves (96^3 points, FP32: a run 84 us a step against 87 with one, 16 of them 654
// against 670; four: 89 and 720), but one in FP64 where two hold too many registers:
// 126 VGPRs at 96 and 144 (16 x 64^3: 1.23 ms a step against 1.47, 64^3 alone 116 us
// against 125), and 33 spilt at 36 (z pass of 96x96x24 33.7 us against 37.7, 24^3
// 11.1 against 11.4).
template <typename T, int L, bool LES>
__host__ __device__ constexpr int zreg_pp()
{
    if (LES) return 1;
    if (sizeof(T) == 8) return L <= 72 && L != 36 ? 2 : 1;
    return L <= 144 ? 2 : 1;
}

// Threads: one butterfly each in every stage after the first (whose radix is
// small where it has more), and one point each (an LES holds the products of a
// thread's points in registers: two of them cost 208 us against 134 at 144, FP64).
template <int L, int NB>
__host__ __device__ constexpr int zreg_nt(int points)
{
    int m = points > 64 ? points : 64;
    for (int s = 1; s < Plan<L>::n; s++) {
        const int b = (L / Plan<L>::r(s)) * NB;
        m = b > m ? b : m;
    }
    if (Plan<L>::r(0) > 4 && (L / Plan<L>::r(0)) * NB > m) m = (L / Plan<L>::r(0)) * NB;
    m = (m + 63) / 64 * 64;
    return m > 1024 ? 1024 : m;
}

// DNS pairs each velocity component with its own d_z where k_zfuse's
// compile-time loader did (L / R0 = 64 or 128), else the logical fields in order.
template <int L, bool LES>
__host__ __device__ constexpr bool zreg_dzpair()
{
    return !LES && (L / Plan<L>::r(0) == 64 || L / Plan<L>::r(0) == 128);
}

template <typename T, int L, bool LES>
struct ZReg {
    static constexpr int PP = zreg_pp<T, L, LES>();
    static constexpr int NI = 6 * PP, NF = (LES ? 5 : 2) * PP;
    static constexpr int NB = LES ? NI : NI + NF;
    static constexpr int NT = zreg_nt<L, NB>(LES ? PP * L : 0);
    // row pitch: LES columns are packed (consecutive butterflies then read
    // consecutive elements), the products repacked to their five columns; the
    // DNS's eight would put a column's rows on the same banks
    static constexpr int LD = LES ? NB : NB + 1;
    static constexpr int LDF = LES ? NF : LD;
    static constexpr int NKC = L / 3 + 1;
    static constexpr int TWM = sizeof(T) == 8 ? 1 : 2;
    static constexpr size_t lds = sizeof(cx<T>) * ((size_t)L * LD + fft_twiddle_span<L, TWM>()) + 9 * sizeof(void*);
    static constexpr bool fits = L % 3 == 0 && lds <= 160 * 1024 - 512;
    static constexpr int waves = (int)((160 * 1024) / lds) * (NT / 64) / 4;  // per SIMD, by LDS
    static constexpr int W = waves < 1 ? 1 : waves > 4 ? 4 : waves;
};

// k_zreg for DNS: below L = 768, where k_zfuse has its swizzled layout, and not
// for FP32 at 288 and 384, where k_zfuse's three blocks per CU keep the vector
// ALU busier (0.373 against 0.405 ms at 192^3, 0.779 against 0.858 at 256^3).
template <typename T, int L>
constexpr bool zreg_dns()
{
    return L < 768 && !(sizeof(T) == 4 && (L == 288 || L == 384)) && ZReg<T, L, false>::fits;
}

template <typename T, int L, bool LES>
__device__ __forceinline__ void zreg_body(const ZArgs& a)
{
    using Z = ZReg<T, L, LES>;
    constexpr int PP = Z::PP, NI = Z::NI, NF = Z::NF, NB = Z::NB, NT = Z::NT, LD = Z::LD, LDF = Z::LDF, NKC = Z::NKC, TWM = Z::TWM;
    constexpr int NITEM = NI * NKC, NIT = (NITEM + NT - 1) / NT;
    constexpr int TWN = fft_twiddle_span<L, TWM>();
    constexpr bool DZP = zreg_dzpair<L, LES>();
    // What a thread keeps across the loop instead of recomputing it per group: in
    // a DNS its items' indices and source pointers, in an FP64 LES the pointers.
    // (FP32 LES at 384: 1.39 ms with the pointers kept, 1.19 without: 64 VGPRs.)
    constexpr bool HOIST = !LES || sizeof(T) == 8, HOISTI = !LES;
    static_assert(sizeof(cx<T>) * L * LD >= 6 * (NT / 64) * sizeof(double), "reduction scratch aliases the pair buffer");
    __shared__ __align__(16) cx<T> fbuf[L * LD];
    __shared__ __align__(16) cx<T> twl[TWN];
    __shared__ cx<T>* fld[9];
    const int t = threadIdx.x;
    const int pitch = a.pitch;
    T mu = (T)0, mv = (T)0, mw = (T)0;
    double vmax_sa = 0.0, s2 = 0.0, s3 = 0.0;
    const double iAx = a.Ax, iAy = a.Ay, iAz = a.Az;
    const bool sa = a.sa;
    if (t < 9) fld[t] = (cx<T>*)a.f[t];
    __syncthreads();

    // logical pairs in order: see k_zstage; with DZP pair c < 3 is (f_c, d_z f_c),
    // c >= 3 (d_x, d_y) of component c - 3
    constexpr uint32_t SRC_A = DZP ? 0x543210u : 0x814620u, SRC_B = DZP ? 0x876000u : 0x257031u;
    constexpr uint32_t DZ_A = DZP ? 0u : 0x10u, DZ_B = DZP ? 0u : 0x24u;
    // this thread's items: column, k3 and where the two spectra lie (global
    // loads: a pointer read from LDS would make them flat ones, which the
    // LDS-only barriers wait for)
    typedef const __attribute__((address_space(1))) cx<T>* gptr;
    const int64_t step = (int64_t)gridDim.x * PP * pitch;  // a group's pencils to the next group's
    cx<T> A[NIT], B[NIT];
    auto item = [&](int i, int tl, int& col, int& c, int& k) -> bool {
        const int idx = tl + i * NT;
        col = idx / NKC;
        k = idx - col * NKC;
        c = col / PP;
        return (i + 1) * NT <= NITEM || idx < NITEM;
    };
    // source pointer of an item's two spectra in the group at pen0
    auto src = [&](uint32_t tab, int col, int c, int k, int64_t pen0) -> gptr {
        return (gptr)fld[(tab >> (4 * c)) & 15] + (pen0 + (col - c * PP)) * pitch + k;
    };
    gptr ga[HOIST ? NIT : 1], gb[HOIST ? NIT : 1];
#pragma unroll
    for (int i = 0; i < NIT; i++) {
        A[i] = B[i] = cx<T>{(T)0, (T)0};
        if constexpr (HOIST) {
            int col, c, k;
            if (!item(i, t, col, c, k)) col = c = k = 0;
            ga[i] = src(SRC_A, col, c, k, (int64_t)blockIdx.x * PP);
            gb[i] = src(SRC_B, col, c, k, (int64_t)blockIdx.x * PP);
        }
    }
    // loads the group at pen0 (with HOIST the one the pointers are at, and
    // moves them on to the next)
    auto fetch = [&](int64_t pen0, int tl) {
#pragma unroll
        for (int i = 0; i < NIT; i++) {
            int col, c, k;
            if (item(i, tl, col, c, k)) {
                const gptr pa = HOIST ? ga[HOIST ? i : 0] : src(SRC_A, col, c, k, pen0);
                A[i].x = pa->x, A[i].y = pa->y;
                if (!DZP || c >= 3) {
                    const gptr pb = HOIST ? gb[HOIST ? i : 0] : src(SRC_B, col, c, k, pen0);
                    B[i].x = pb->x, B[i].y = pb->y;
                }
            }
            if constexpr (HOIST) {
                ga[i] += step;
                gb[i] += step;
            }
        }
    };
    auto spread = [&](int tl) {
#pragma unroll
        for (int i = 0; i < NIT; i++) {
            int col, c, k;
            if (item(i, tl, col, c, k)) {
                cx<T> lo, hi;
                if (DZP && c < 3) z_pair_dz(A[i], k, lo, hi);
                else z_pair(A[i], B[i], k, (DZ_A >> c) & 1, (DZ_B >> c) & 1, lo, hi);
                fbuf[k * LD + col] = lo;
                if (k > 0) fbuf[(L - k) * LD + col] = hi;
            }
        }
        if constexpr (!LES) {
            // the zero padding (an LES's loader skips it)
            constexpr int GAP = L - 2 * NKC + 1;
            for (int idx = tl; idx < GAP * NI; idx += NT) {
                const int r = idx / NI;
                fbuf[(NKC + r) * LD + (idx - r * NI)] = cx<T>{(T)0, (T)0};
            }
        }
    };

    const int64_t G = (int64_t)gridDim.x * PP;
    int64_t pen = (int64_t)blockIdx.x * PP;
    if (pen < a.npencil) fetch(pen, t);
    for (int i = t; i < TWN; i += NT) twl[i] = ((const cx<T>*)a.tw)[i];
    if constexpr (!LES) {
        for (int idx = t; idx < L * NF; idx += NT) {  // no products yet
            const int r = idx / NF;
            fbuf[r * LD + NI + (idx - r * NF)] = cx<T>{(T)0, (T)0};
        }
    }
    int64_t prev = -1;  // DNS: group whose products sit in columns NI ..
    for (;; pen += G) {
        const bool have = pen < a.npencil, havep = prev >= 0;
        if (!have && (LES || !havep)) break;
        const int tl = opaque(t);
        const int ti = HOISTI ? t : tl;
        if (have) {
            spread(ti);
            if (pen + G < a.npencil) fetch(pen + G, ti);
        }
        lds_barrier();
        auto load = [&](int b, int j, auto rc) -> cx<T> {
            constexpr int LR0 = L / Plan<L>::r(0), p0 = LR0 * decltype(rc)::value;
            constexpr bool IN = !LES || p0 + LR0 - 1 < NKC || p0 > L - NKC;
            constexpr bool ZERO = LES && p0 >= NKC && p0 + LR0 - 1 <= L - NKC;
            const int p = p0 + j;
            if constexpr (ZERO) return cx<T>{(T)0, (T)0};
            const cx<T> v = fbuf[p * LD + b];
            const bool in = IN || p < NKC || p > L - NKC;
            return cx<T>{in ? v.x : (T)0, in ? v.y : (T)0};
        };
        auto store = [&](int b, int p, cx<T> v) { fbuf[p * LD + b] = v; };
        auto none = [] {};
        FftS<T, L, NB, NT, LD, +1, true, TWM>::template run<false>(fbuf, twl, load, store, none, tl);
        lds_barrier();
        // -------- half spectra of the products of group gp, in columns C0 ..
        // (DNS: those columns hold the conjugates, forward = conj(inverse(conj x)))
        auto unpack = [&](int64_t gp, auto c0) {
            constexpr int C0 = decltype(c0)::value;
            constexpr T sg = LES ? (T)1 : (T)-1;
            for (int idx = ti; idx < NF * NKC; idx += NT) {
                const int col = idx / NKC, k = idx - col * NKC;
                const int q = col / PP;
                cx<T> Zk = fbuf[k * LDF + C0 + col], Zc = fbuf[(k == 0 ? 0 : L - k) * LDF + C0 + col];
                Zk.y *= sg;
                Zc.y *= sg;
                const T h = (T)0.5;
                const int64_t o = (gp + (col - q * PP)) * pitch + k;
                typedef __attribute__((address_space(1))) cx<T>* gout;
                const gout d0 = (gout)fld[2 * q] + o;
                d0->x = h * (Zk.x + Zc.x);
                d0->y = h * (Zk.y - Zc.y);
                if (2 * q + 1 < (LES ? 9 : 3)) {
                    const gout d1 = (gout)fld[2 * q + 1] + o;
                    d1->x = h * (Zk.y + Zc.y);
                    d1->y = h * (Zc.x - Zk.x);
                }
            }
        };
        if constexpr (!LES) {
            if (havep) {
                unpack(prev, std::integral_constant<int, NI>{});
                lds_barrier();
            }
        }
        if (have) {
            // -------- physical space
            constexpr int NITP = (PP * L + NT - 1) / NT;
            cx<T> out[LES ? NITP : 1][5];  // LES: the products, until every wave has read its points
#pragma unroll
            for (int i = 0; i < NITP; i++) {
                const int idx = tl + i * NT, n = idx / PP;
                if (PP * L % NT != 0 && idx >= PP * L) continue;
                cx<T>* row = &fbuf[n * LD + (idx - n * PP)];
                T u, v, w, ux, uy, uz, vx, vy, vz, wx, wy, wz;
                if constexpr (DZP) {
                    u = row[0].x, uz = row[0].y, v = row[PP].x, vz = row[PP].y, w = row[2 * PP].x, wz = row[2 * PP].y;
                    ux = row[3 * PP].x, uy = row[3 * PP].y, vx = row[4 * PP].x, vy = row[4 * PP].y;
                    wx = row[5 * PP].x, wy = row[5 * PP].y;
                } else {
                    u = row[0].x, v = row[0].y, w = row[PP].x;
                    ux = row[PP].y, uy = row[2 * PP].x, uz = row[2 * PP].y;
                    vx = row[3 * PP].x, vy = row[3 * PP].y, vz = row[4 * PP].x;
                    wx = row[4 * PP].y, wy = row[5 * PP].x, wz = row[5 * PP].y;
                }
                mu = fmax(mu, fabs(u));
                mv = fmax(mv, fabs(v));
                mw = fmax(mw, fabs(w));
                if (sa) vmax_sa = fmax(vmax_sa, fabs((double)u) / iAx + fabs((double)v) / iAy + fabs((double)w) / iAz);  // src/HIT_LES.cpp:377
                s2 += (double)ux * (double)ux;
                s3 += (double)ux * (double)ux * (double)ux;
                // advective form (src/HIT_LES.cpp:118-120)
                const T cxv = u * ux + v * uy + w * uz;
                const T cyv = u * vx + v * vy + w * vz;
                const T czv = u * wx + v * wy + w * wz;
                if constexpr (LES) {
                    // Smagorinsky (src/HIT_LES.cpp:130-154)
                    const T ct = (T)a.ct;
                    T ne = (T)2.0 * ux * ux;
                    ne += (T)2.0 * vy * vy;
                    ne += (T)2.0 * wz * wz;
                    ne += (uy + vx) * (uy + vx);
                    ne += (uz + wx) * (uz + wx);
                    ne += (vz + wy) * (vz + wy);
                    ne = ct * sqrt(ne);
                    out[i][0] = cx<T>{cxv, cyv};
                    out[i][1] = cx<T>{czv, (T)(-2.0) * ne * ux};
                    out[i][2] = cx<T>{(T)(-1.0) * ne * (uy + vx), (T)(-2.0) * ne * vy};
                    out[i][3] = cx<T>{(T)(-1.0) * ne * (uz + wx), (T)(-1.0) * ne * (vz + wy)};
                    out[i][4] = cx<T>{(T)(-2.0) * ne * wz, (T)0};
                } else {
                    row[6 * PP] = cx<T>{cxv, -cyv};
                    row[7 * PP] = cx<T>{czv, (T)0};
                }
            }
            if constexpr (LES) {
                if constexpr (LDF != LD) lds_barrier();
#pragma unroll
                for (int i = 0; i < NITP; i++) {
                    const int idx = tl + i * NT, n = idx / PP;
                    if (PP * L % NT != 0 && idx >= PP * L) continue;
#pragma unroll
                    for (int q = 0; q < 5; q++) fbuf[n * LDF + q * PP + (idx - n * PP)] = out[i][q];
                }
                auto load_f = [&](int b, int p) -> cx<T> { return fbuf[p * LDF + b]; };
                auto store_f = [&](int b, int p, cx<T> v) { fbuf[p * LDF + b] = v; };
                FftS<T, L, NF, NT, LDF, -1, true, TWM>::template run<true>(fbuf, twl, load_f, store_f, none, tl);
                lds_barrier();
                unpack(pen, std::integral_constant<int, 0>{});
            }
        }
        lds_barrier();
        prev = have ? pen : -1;
    }
    z_partials<NT>(a, (double)mu, (double)mv, (double)mw, vmax_sa, s2, s3, (double*)fbuf);
}

template <typename T, int L, bool LES>
__global__ __launch_bounds__((ZReg<T, L, LES>::NT)) __attribute__((amdgpu_waves_per_eu(ZReg<T, L, LES>::W))) void k_zreg(ZArgs a)
{
    zreg_body<T, L, LES>(a);
}

template <typename T, int L, bool LES>
__global__ __launch_bounds__((ZReg<T, L, LES>::NT)) __attribute__((amdgpu_waves_per_eu(ZReg<T, L, LES>::W))) void k_zreg_b(
    const ZArgs* __restrict__ arr, const int* __restrict__ left)
{
    if (left[blockIdx.y] <= 0) return;
    zreg_body<T, L, LES>(arr[blockIdx.y]);
}

// ---------------------------------------------------------------------------
// z pass, one wave per pencil (DNS and velocity-only modes, L = 64*E).
// Lane t owns the physical points z = t + 64 m; the twelve fields arrive pair
// by pair from WaveFft and the products u.grad(u) accumulate in registers in
// the reference's operand order ((u g1 + v g2) + w g3, src/HIT_LES.cpp:119).
// The forward transforms read their first stage straight from those
// registers; only the final unpack goes through the wave's LDS column.
// ---------------------------------------------------------------------------
template <typename T, int L>
__device__ __forceinline__ void wave_inv_pair(cx<T>* lds, const cx<T>* tw, const cx<T>* pa, int da, const cx<T>* pb, int db,
                                              int64_t off, int nk, T* outA, T* outB)
{
    auto load = [&](int p, int slot) -> cx<T> {
        (void)slot;
        const bool lo = p < nk, hi = p > L - nk;
        if (!(lo || hi)) return cx<T>{(T)0, (T)0};
        const int k = lo ? p : L - p;
        const T kk = (T)k;
        cx<T> A = pa[off + k];
        if (da) A = cx<T>{-kk * A.y, kk * A.x};
        cx<T> B = cx<T>{(T)0, (T)0};
        if (pb) {
            B = pb[off + k];
            if (db) B = cx<T>{-kk * B.y, kk * B.x};
        }
        const T sg = lo ? (T)1 : (T)-1;
        const T ay = (p == 0) ? (T)0 : sg * A.y;
        const T by = (p == 0) ? (T)0 : sg * B.y;
        return cx<T>{A.x - by, ay + B.x};
    };
    auto store = [&](int p, cx<T> v, int slot) {
        (void)p;
        outA[slot] = v.x;
        outB[slot] = v.y;
    };
    WaveFft<T, L, +1>::run(lds, tw, load, store);
}

template <typename T, int L>
__device__ __forceinline__ void wave_fwd_pair(cx<T>* lds, const cx<T>* tw, const T* inA, const T* inB, cx<T>* qa, cx<T>* qb,
                                              int64_t off, int nk)
{
    auto load = [&](int p, int slot) -> cx<T> {
        (void)p;
        return cx<T>{inA[slot], inB ? inB[slot] : (T)0};
    };
    auto store = [&](int p, cx<T> v, int slot) {
        (void)slot;
        lds[p] = v;
    };
    WaveFft<T, L, -1>::run(lds, tw, load, store);
    wave_sync();
    const int t = threadIdx.x & 63;
    for (int k = t; k < nk; k += 64) {
        const cx<T> Z = lds[k], Zc = lds[(L - k) % L];
        const T h = (T)0.5;
        qa[off + k] = cx<T>{h * (Z.x + Zc.x), h * (Z.y - Zc.y)};
        if (qb) qb[off + k] = cx<T>{h * (Z.y + Zc.y), h * (Zc.x - Z.x)};
    }
}

template <typename T, int L, int MODE>
__global__ __launch_bounds__(256) void k_zwave(ZArgs a)
{
    constexpr int E = L / 64, WPB = 4;
    __shared__ cx<T> ldsw[WPB][L];
    __shared__ double red[6 * 4];
    const int w = threadIdx.x >> 6, t = threadIdx.x & 63;
    cx<T>* lds = ldsw[w];
    const cx<T>* tw = (const cx<T>*)a.tw;
    const int nk = a.nk3;
    const cx<T>* F[9];
#pragma unroll
    for (int f = 0; f < 9; f++) F[f] = (const cx<T>*)a.f[f];
    // max over points of max(|u|/Ax, |v|/Ay, |w|/Az) equals the max of the
    // per-component maxima divided once (correctly rounded division by a
    // positive constant is monotonic); the sum form needs every point.
    T mu = (T)0, mv = (T)0, mw = (T)0;
    double vmax_sa = 0.0, s2 = 0.0, s3 = 0.0;
    const double iAx = a.Ax, iAy = a.Ay, iAz = a.Az;
    const bool sa = a.sa;

    for (int64_t pen = (int64_t)blockIdx.x * WPB + w; pen < a.npencil; pen += (int64_t)gridDim.x * WPB) {
        const int64_t off = pen * a.pitch;
        T U[E], V[E], W[E];
        wave_inv_pair<T, L>(lds, tw, F[0], 0, F[1], 0, off, nk, U, V);  // (u, v)
        if constexpr (MODE == 1) {
            T Z0[E];
            wave_inv_pair<T, L>(lds, tw, F[2], 0, nullptr, 0, off, nk, W, Z0);  // (w, -)
        }
        if constexpr (MODE == 1) {
#pragma unroll
            for (int m = 0; m < E; m++) {
                mu = fmax(mu, fabs(U[m]));
                mv = fmax(mv, fabs(V[m]));
                mw = fmax(mw, fabs(W[m]));
                s2 += (double)U[m] * (double)U[m] + (double)V[m] * (double)V[m] + (double)W[m] * (double)W[m];  // src/HIT_LES.cpp:1236-1239
            }
            if (sa) {
                for (int m = 0; m < E; m++)
                    vmax_sa = fmax(vmax_sa, fabs((double)U[m]) / iAx + fabs((double)V[m]) / iAy + fabs((double)W[m]) / iAz);
            }
            if (a.phys[0]) {
                const int64_t r = phys_row(a, pen) * L;
#pragma unroll
                for (int m = 0; m < E; m++) {
                    const int64_t o = r + t + 64 * m;
                    a.phys[0][o] = U[m];
                    a.phys[1][o] = V[m];
                    a.phys[2][o] = W[m];
                }
            }
        } else {
            T CX[E], CY[E], CZ[E], G1[E], G2[E];
            wave_inv_pair<T, L>(lds, tw, F[2], 0, F[3], 0, off, nk, W, G1);  // (w, ux)
            if (sa) {
                for (int m = 0; m < E; m++)
                    vmax_sa = fmax(vmax_sa, fabs((double)U[m]) / iAx + fabs((double)V[m]) / iAy + fabs((double)W[m]) / iAz);
            }
#pragma unroll
            for (int m = 0; m < E; m++) {
                mu = fmax(mu, fabs(U[m]));
                mv = fmax(mv, fabs(V[m]));
                mw = fmax(mw, fabs(W[m]));
                const double g = (double)G1[m];
                s2 += g * g;
                s3 += g * g * g;
                CX[m] = U[m] * G1[m];
            }
            wave_inv_pair<T, L>(lds, tw, F[6], 0, F[0], 1, off, nk, G1, G2);  // (uy, uz)
#pragma unroll
            for (int m = 0; m < E; m++) CX[m] = CX[m] + V[m] * G1[m] + W[m] * G2[m];
            wave_inv_pair<T, L>(lds, tw, F[4], 0, F[7], 0, off, nk, G1, G2);  // (vx, vy)
#pragma unroll
            for (int m = 0; m < E; m++) CY[m] = U[m] * G1[m] + V[m] * G2[m];
            wave_inv_pair<T, L>(lds, tw, F[1], 1, F[5], 0, off, nk, G1, G2);  // (vz, wx)
#pragma unroll
            for (int m = 0; m < E; m++) {
                CY[m] = CY[m] + W[m] * G1[m];
                CZ[m] = U[m] * G2[m];
            }
            wave_inv_pair<T, L>(lds, tw, F[8], 0, F[2], 1, off, nk, G1, G2);  // (wy, wz)
#pragma unroll
            for (int m = 0; m < E; m++) CZ[m] = CZ[m] + V[m] * G1[m] + W[m] * G2[m];
            wave_fwd_pair<T, L>(lds, tw, CX, CY, (cx<T>*)a.f[0], (cx<T>*)a.f[1], off, nk);
            wave_fwd_pair<T, L>(lds, tw, CZ, (const T*)nullptr, (cx<T>*)a.f[2], (cx<T>*)nullptr, off, nk);
        }
    }
    z_partials<256>(a, (double)mu, (double)mv, (double)mw, vmax_sa, s2, s3, red);
}

// ---------------------------------------------------------------------------
// Plain z transforms for the FFT_package drop-in (reference layouts):
//   c2r: complex [y][x][nk] -> real [x][y][2nk] padded (src/util.h:75-80)
//   r2c: real [x][y][2nk] -> complex [y][x][nk]
// Two pencils are paired into one complex transform, NB pairs at a time.
// Bounded by HBM (one read and one write of the field); every global access
// runs along z, and the exchanges through LDS ([row][NB + 1]: an odd pitch, so
// accesses along z spread over the banks) keep it so on both sides.  One pair
// per 64-thread block, as before, left 56 of 64 lanes idle at L = 48 and wrote
// the c2r's results 8 bytes at a time: 768^3 FP64 c2r 1.99 -> 1.63 ms, r2c 1.62 ->
// 1.55 ms (4.7 TB/s), 384^3 FP32 122 -> 100 us.  Loads that wait for each other
// in a loop cost more than either: 4.1 ms for the r2c.
// ---------------------------------------------------------------------------
// Pairs per block: 8 at most, fewer where the exchange buffer would leave room
// for less than three blocks per CU (two are the least: FP64 at 1152 and 1536 has
// two blocks and one).
template <typename T, int L>
__host__ __device__ constexpr int zline_nb()
{
    constexpr size_t el = sizeof(cx<T>) * L;
    return L <= 144 ? 8 : el * 5 <= 40960 ? 4 : 2;
}

template <typename T, int L, int NB, int NT, int DIR>
__global__ __launch_bounds__(NT) void k_zline(ZPlainArgs a)
{
    constexpr int LD = NB + 1, nk = L / 2 + 1;
    constexpr int NIT = (NB * nk + NT - 1) / NT;
    __shared__ __align__(16) cx<T> fbuf[L * LD];
    __shared__ __align__(16) cx<T> twl[L];
    const int t = threadIdx.x;
    const uint32_t Mx = a.Mx, My = a.My, np = Mx * My;
    // pencil p = y Mx + x: offset of its real row
    auto real_row = [&](uint32_t p) -> int64_t {
        const uint32_t y = p / Mx;
        return ((int64_t)(p - y * Mx) * My + y) * (2 * nk);
    };
    auto store_lds = [&](int b, int p, cx<T> v) { fbuf[p * LD + b] = v; };
    auto none = [] {};
    bool first = true;
    for (uint32_t q0 = blockIdx.x * NB; 2 * q0 < np; q0 += gridDim.x * NB) {  // first pair of the group
        if constexpr (DIR > 0) {
            const cx<T>* __restrict__ in = (const cx<T>*)a.in;
            T* __restrict__ out = (T*)a.out;
            // every load of the group is in flight before the first is used
            cx<T> A[NIT], B[NIT];
#pragma unroll
            for (int i = 0; i < NIT; i++) {
                const int idx = t + i * NT, b = idx / nk, k = idx - b * nk;
                const uint32_t p0 = 2 * (q0 + b);
                const bool ok = idx < NB * nk;
                A[i] = ok && p0 < np ? in[(int64_t)p0 * nk + k] : cx<T>{(T)0, (T)0};
                B[i] = ok && p0 + 1 < np ? in[(int64_t)(p0 + 1) * nk + k] : cx<T>{(T)0, (T)0};
            }
            if (first)
                for (int i = t; i < L; i += NT) twl[i] = ((const cx<T>*)a.tw)[i];
            lds_barrier();  // the previous group's reads are done
#pragma unroll
            for (int i = 0; i < NIT; i++) {
                const int idx = t + i * NT, b = idx / nk, k = idx - b * nk;
                if (idx < NB * nk) {
                    if (k == 0 || 2 * k == L) {
                        fbuf[k * LD + b] = cx<T>{A[i].x, B[i].x};  // only the real part of the end terms enters
                    } else {
                        fbuf[k * LD + b] = cx<T>{A[i].x - B[i].y, A[i].y + B[i].x};
                        fbuf[(L - k) * LD + b] = cx<T>{A[i].x + B[i].y, B[i].x - A[i].y};
                    }
                }
            }
            auto load_lds = [&](int b, int p) -> cx<T> { return fbuf[p * LD + b]; };
            FftS<T, L, NB, NT, LD, +1, true, 0>::template run<true>(fbuf, twl, load_lds, store_lds, none, t);
            lds_barrier();
            for (int idx = t; idx < NB * L; idx += NT) {
                const int b = idx / L, n = idx - b * L;
                const uint32_t p0 = 2 * (q0 + b);
                const cx<T> v = fbuf[n * LD + b];
                if (p0 < np) out[real_row(p0) + n] = v.x;
                if (p0 + 1 < np) out[real_row(p0 + 1) + n] = v.y;
            }
        } else {
            const T* __restrict__ in = (const T*)a.in;
            cx<T>* __restrict__ out = (cx<T>*)a.out;
            // stage 0 reads its inputs itself, consecutive threads along z
            auto load = [&](int b, int p) -> cx<T> {
                const uint32_t p0 = 2 * (q0 + b);
                cx<T> v = cx<T>{(T)0, (T)0};
                if (p0 < np) v.x = in[real_row(p0) + p];
                if (p0 + 1 < np) v.y = in[real_row(p0 + 1) + p];
                return v;
            };
            if (first)
                for (int i = t; i < L; i += NT) twl[i] = ((const cx<T>*)a.tw)[i];
            // SYNC0: a barrier between stage 0's reads and its writes, which
            // the previous group's unpack must have left
            FftS<T, L, NB, NT, LD, -1, true, 0, true>::template run<false>(fbuf, twl, load, store_lds, none, t);
            lds_barrier();
            for (int idx = t; idx < NB * nk; idx += NT) {
                const int b = idx / nk, k = idx - b * nk;
                const uint32_t p0 = 2 * (q0 + b);
                if (p0 >= np) continue;
                const cx<T> Z = fbuf[k * LD + b], Zc = fbuf[(k == 0 ? 0 : L - k) * LD + b];
                const T h = (T)0.5;
                out[(int64_t)p0 * nk + k] = cx<T>{h * (Z.x + Zc.x), h * (Z.y - Zc.y)};
                if (p0 + 1 < np) out[(int64_t)(p0 + 1) * nk + k] = cx<T>{h * (Z.y + Zc.y), h * (Zc.x - Z.x)};
            }
        }
        first = false;
    }
}

// ---------------------------------------------------------------------------
// Spectral epilogue over the compact box (FP64 state).
// src/HIT_LES.cpp:205-242 (R), :243-278 (constant power), :295-339 (AB2 /
// kappa), :346-359 (projection); reductions :991-1003, :1137-1214.
// ---------------------------------------------------------------------------
// Step epilogue of one retained mode m = (k1, k2, k3) (src/HIT_LES.cpp:196-363):
// R1 from the normalised convective term C (and, LES, the SGS stress S:
// 11 21 22 31 32 33), viscosity, rotation, constant-power forcing; AB2 or the
// kappa scheme; projection; the state and history written back; then the
// shell-energy and enstrophy contributions of the new state.  With step
// false only the reductions of the current state.
struct EpiScalars {
    double dt, nu, alpha, kap, k05;
    bool first;
};

static __device__ __forceinline__ EpiScalars epi_scalars(const EpiArgs& a)
{
    EpiScalars q;
    q.dt = a.scal->dt;
    q.nu = a.scal->nu;
    q.alpha = a.scal->alpha;
    q.kap = a.scal->kappa;
    q.k05 = 1.0 / (q.kap + 0.5);
    q.first = a.scal->iter == 0;
    return q;
}

// RT: the storage type of the R history (the transform type of the form:
// the FP32-split form keeps R in FP32, whose convective part already carries
// the FP32 transforms' rounding; R is combined in FP64 either way).
// epi_core takes the mode's state U and history R0 already loaded.
template <typename RT>
static __device__ __forceinline__ void epi_core(const EpiArgs& a, const EpiScalars& q, int64_t m, int k1, int k2, int k3,
                                         bool step, cx<double>* U, const cx<double>* R0, const cx<double>* C, const cx<double>* S,
                                         double* myh, double& om, double& ed, cx<double>* Nout)
{
    const int ik2 = k1 * k1 + k2 * k2 + k3 * k3;
    const double rad2 = (double)ik2;
    const int K = shell_of(ik2);
    cx<double> R1[3];
    if (step) {
        const double dt = q.dt, kap = q.kap, k05 = q.k05, alpha = q.alpha;
        const double ct = q.nu * rad2;
        const bool mean = !(rad2 > 0.0);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            R1[c].x = -(mean ? 0.0 : C[c].x) - ct * U[c].x;
            R1[c].y = -(mean ? 0.0 : C[c].y) - ct * U[c].y;
        }
        if (S) {
            // S: 11, 21, 22, 31, 32, 33 (src/HIT_LES.cpp:179-191)
            const double K1 = k1, K2 = k2, K3 = k3;
            const double dxr = -K1 * S[0].y - K2 * S[1].y - K3 * S[3].y;
            const double dxi = K1 * S[0].x + K2 * S[1].x + K3 * S[3].x;
            const double dyr = -K1 * S[1].y - K2 * S[2].y - K3 * S[4].y;
            const double dyi = K1 * S[1].x + K2 * S[2].x + K3 * S[4].x;
            const double dzr = -K1 * S[3].y - K2 * S[4].y - K3 * S[5].y;
            const double dzi = K1 * S[3].x + K2 * S[4].x + K3 * S[5].x;
            R1[0].x -= dxr; R1[0].y -= dxi;
            R1[1].x -= dyr; R1[1].y -= dyi;
            R1[2].x -= dzr; R1[2].y -= dzi;
        }
        if (a.rot) {
            const double ox = a.ox, oy = a.oy, oz = a.oz;
            R1[0].x += 2 * (oz * U[1].x - oy * U[2].x); R1[0].y += 2 * (oz * U[1].y - oy * U[2].y);
            R1[1].x += 2 * (ox * U[2].x - oz * U[0].x); R1[1].y += 2 * (ox * U[2].y - oz * U[0].y);
            R1[2].x += 2 * (oy * U[0].x - ox * U[1].x); R1[2].y += 2 * (oy * U[0].y - ox * U[1].y);
        }
        if (a.force_on) {
            if (a.kfmin <= K && K <= a.kfmax) {
#pragma unroll
                for (int c = 0; c < 3; c++) { R1[c].x += alpha * U[c].x; R1[c].y += alpha * U[c].y; }
            } else if (K == 0) {
#pragma unroll
                for (int c = 0; c < 3; c++) R1[c] = cx<double>{0.0, 0.0};
            }
        }
        cx<double> N[3];
        if (a.sa) {
            // self-adaptive kappa scheme; the oldest level at the first
            // step is the current field
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const cx<double> Up = a.ukprev[c][m];  // read unconditionally: a select of
                const cx<double> Ua = q.first ? U[c] : Up;  // pointers would push U to scratch
                a.ukprev[c][m] = U[c];
                N[c].x = k05 * (2.0 * kap * U[c].x + dt * ((1.0 + kap) * R1[c].x - kap * R0[c].x) - (kap - 0.5) * Ua.x);
                N[c].y = k05 * (2.0 * kap * U[c].y + dt * ((1.0 + kap) * R1[c].y - kap * R0[c].y) - (kap - 0.5) * Ua.y);
            }
        } else {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                if (a.keepprev) a.ukprev[c][m] = U[c];  // the start-of-step state
                N[c].x = U[c].x + dt * (1.5 * R1[c].x - 0.5 * R0[c].x);
                N[c].y = U[c].y + dt * (1.5 * R1[c].y - 0.5 * R0[c].y);
            }
        }
        {
            const double K1 = k1, K2 = k2, K3 = k3;
            const double ir2 = (rad2 > 0) ? 1.0 / rad2 : 0.0;
            const double axr = (K1 * N[0].x + K2 * N[1].x + K3 * N[2].x) * ir2;
            const double axi = (K1 * N[0].y + K2 * N[1].y + K3 * N[2].y) * ir2;
            N[0].x -= axr * K1; N[1].x -= axr * K2; N[2].x -= axr * K3;
            N[0].y -= axi * K1; N[1].y -= axi * K2; N[2].y -= axi * K3;
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            a.uk[c][m] = N[c];
            ((cx<RT>*)a.R[c])[m] = cx<RT>{(RT)R1[c].x, (RT)R1[c].y};
            U[c] = N[c];
            if (Nout) Nout[c] = N[c];
        }
    }
    // reductions on the (new) state
    const double ke = 0.5 * (U[0].x * U[0].x + U[0].y * U[0].y + U[1].x * U[1].x + U[1].y * U[1].y +
                             U[2].x * U[2].x + U[2].y * U[2].y);
    const bool conj = (k3 != 0) && !((a.Mz % 2 == 0) && (k3 == a.Mz / 2));
    atomicAdd(&myh[K], conj ? 2 * ke : ke);
    const double en = 2 * rad2 * ke;
    om += conj ? 2 * en : en;
    ed += conj ? 2 * ke : ke;
}

template <typename RT>
static __device__ __forceinline__ void epi_load(const EpiArgs& a, int64_t m, bool step, cx<double>* U, cx<double>* R0)
{
#pragma unroll
    for (int c = 0; c < 3; c++) U[c] = a.uk[c][m];
    if (step) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            const cx<RT> r = ((const cx<RT>*)a.R[c])[m];
            R0[c] = cx<double>{(double)r.x, (double)r.y};
        }
    }
}

template <typename RT>
static __device__ __forceinline__ void epi_mode(const EpiArgs& a, const EpiScalars& q, int64_t m, int k1, int k2, int k3,
                                         bool step, const cx<double>* C, const cx<double>* S, double* myh, double& om,
                                         double& ed, cx<double>* Nout = nullptr)
{
    cx<double> U[3], R0[3];
    epi_load<RT>(a, m, step, U, R0);
    epi_core<RT>(a, q, m, k1, k2, k3, step, U, R0, C, S, myh, om, ed, Nout);
}

// Per-wave shell histograms [NW][nbins] summed in wave order into the
// block's partial, and the block's enstrophy partial.
template <int NT>
__device__ __forceinline__ void epi_flush(const EpiArgs& a, const double* hist, double om, double* red)
{
    constexpr int NW = NT / 64;
    const int nb = a.nbins;
    __syncthreads();
    for (int K = threadIdx.x; K < nb; K += NT) {
        double s = 0.0;
        for (int w = 0; w < NW; w++) s += hist[w * nb + K];
        a.hist_partial[(int64_t)blockIdx.x * nb + K] = s;
    }
    om = block_sum<NT>(om, red);
    if (threadIdx.x == 0) a.om_partial[blockIdx.x] = om;
}

template <typename T, int NT>
__device__ __forceinline__ void epilogue_body(const EpiArgs& a)
{
    constexpr int NW = NT / 64;
    extern __shared__ double hist[];  // NW * nbins
    __shared__ double red[NW];
    const int nb = a.nbins;
    for (int i = threadIdx.x; i < NW * nb; i += NT) hist[i] = 0.0;
    __syncthreads();
    double* myh = hist + (threadIdx.x / 64) * nb;
    const EpiScalars q = epi_scalars(a);
    double om = 0.0, ed = 0.0;
    const int nk1 = a.nk1, nk2 = a.nk2, nk3 = a.nk3, nk3p = a.nk3p;
    const double inv_nf = 1.0 / a.nf;
    const bool step = a.mode == EPI_STEP;
    auto mode = [&](int row, int i3) {
        const int i2 = row / nk1, i1 = row - i2 * nk1;
        const int64_t m = (int64_t)row * nk3p + i3;
        const int k1 = wrap_k(i1, nk1), k2 = wrap_k(i2, nk2), k3 = i3;
        if (a.notcubic && ((k1 % a.Lx) || (k2 % a.Ly) || (k3 % a.Lz))) return;  // src/HIT_LES.cpp:867-871
        cx<double> C[3], S[6];
        if (step) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const cx<T> cv = ((const cx<T>*)a.conv[c])[m];
                C[c] = cx<double>{(double)cv.x * inv_nf, (double)cv.y * inv_nf};  // Fourier_Normalization
            }
            if (a.les) {
#pragma unroll
                for (int s = 0; s < 6; s++) {
                    const cx<T> v = ((const cx<T>*)a.conv[3 + s])[m];
                    S[s] = cx<double>{(double)v.x * inv_nf, (double)v.y * inv_nf};
                }
            }
        }
        epi_mode<T>(a, q, m, k1, k2, k3, step, C, (step && a.les) ? S : nullptr, myh, om, ed);
    };
    // The first nfull = 64 floor(nk3 / 64) modes of each (i2, i1) row: one
    // wave per row, lanes along i3 (no per-mode index division, coalesced
    // row reads).  The rest of every row (nk3 mod 64 modes: 1 at the
    // 2^n-cubed grids, where a wave per row would run its last pass with one
    // lane) are spread over all threads of the grid, row-major.
    const int lane = threadIdx.x & 63;
    const int nrow = nk1 * nk2;
    const int nfull = nk3 & ~63, rem = nk3 - nfull;
    if (nfull > 0) {
        for (int row = blockIdx.x * NW + (int)(threadIdx.x >> 6); row < nrow; row += gridDim.x * NW)
            for (int i3 = lane; i3 < nfull; i3 += 64) mode(row, i3);
    }
    if (rem > 0) {
        // row = floor(f / rem) through FP64: (f + 1/2) / rem is never within
        // 1/(2 rem) of an integer, far above the product's rounding error
        const double inv_rem = 1.0 / rem;
        const int64_t ntail = (int64_t)nrow * rem;
        for (int64_t f = (int64_t)blockIdx.x * NT + threadIdx.x; f < ntail; f += (int64_t)gridDim.x * NT) {
            const int row = (int)(((double)f + 0.5) * inv_rem);
            mode(row, nfull + (int)(f - (int64_t)row * rem));
        }
    }
    epi_flush<NT>(a, hist, om, red);
    if (a.ed_partial) {
        // the direct sum of E (HIT::Check_PhysFour_Energy's EkFour, src/HIT_LES.cpp:1218-1230)
        ed = block_sum<NT>(ed, red);
        if (threadIdx.x == 0) a.ed_partial[blockIdx.x] = ed;
    }
}

template <typename T, int NT>
__global__ __launch_bounds__(NT) void k_epilogue(EpiArgs a)
{
    epilogue_body<T, NT>(a);
}

template <typename T, int NT>
__global__ __launch_bounds__(NT) void k_epilogue_b(const EpiArgs* __restrict__ arr, const int* __restrict__ left)
{
    if (left[blockIdx.y] <= 0) return;
    epilogue_body<T, NT>(arr[blockIdx.y]);
}

// ---------------------------------------------------------------------------
// Forward y pass of the three DNS convective fields fused with the step
// epilogue.  A persistent block walks items (k1 index, tile of TB k3
// columns); per item the three components run one after the other through
// the staged strided transform (input tile copied asynchronously, the next
// component's copy issued after stage 0), components 0 and 1 keep their
// retained outputs in registers, and after component 2 every retained mode
// of the item goes through epi_mode.  The convective spectra never reach
// HBM.  Shell histograms are per wave, as in k_epilogue.
// ---------------------------------------------------------------------------
// INV: after the epilogue of an item, the next step's inverse y pass of the
// item's new state (the same (k1, k3 tile) columns): component 0 goes into the
// staging tile (FP64, [2 (L/3) + 1][TB]) as the epilogue computes each mode;
// components 1 and 2 are staged back from the state this block has just
// written (through the cache hierarchy), each copy issued during the previous
// component's transforms (holding them in registers would spill in FP32).
// Each component is transformed twice, plain and i k2, into u_c and d/dy u_c
// (X1 slots c and 3 + c), with the same arithmetic as the strided inverse
// pass at the next step; the kernel sets *x1v, which lets that pass skip.  The item's X1 columns are the ones its
// forward transforms read, so the writes touch nothing another item still
// needs.  The staging tile grows to the FP64 state tile (at 512^3 FP32 the
// LDS is then 160,584 bytes with the 12 waves' histograms).
// Staging tile of k_yepi (elements of cx<T>): the forward pass's input
// tile, or with INV also a staged FP64 state tile [2 (L/3) + 1][TB].
template <typename T, int L, int TB, bool INV>
__host__ __device__ constexpr int yepi_stg_elems()
{
    constexpr size_t a = (size_t)L * TB, b = INV ? ((size_t)(2 * (L / 3) + 1) * TB * sizeof(cx<double>) + sizeof(cx<T>) - 1) / sizeof(cx<T>) : 0;
    return (int)(a > b ? a : b);
}

template <typename T, int L, int TB, int NT, bool INV = false>
__device__ __forceinline__ void yepi_body(const StridedArgs& a, const EpiArgs& e, const StridedArgs& ia, int* x1v)
{
    constexpr int SPR = TB * (int)sizeof(cx<T>) / 16;  // 16-byte copy slots per staged row
    constexpr int EPS = 16 / (int)sizeof(cx<T>);
    constexpr int NW = NT / 64;
    constexpr int TWM = sizeof(T) == 8 ? 1 : 2;
    constexpr int TWN = fft_twiddle_span<L, TWM>();
    constexpr int NOUTMAX = 2 * (L / 3) + 1;  // the launcher checks nout against it
    constexpr int Q = (NOUTMAX * TB + NT - 1) / NT;
    constexpr int STGN = yepi_stg_elems<T, L, TB, INV>();
    static_assert(L * TB * sizeof(cx<T>) >= (NT / 64) * sizeof(double), "reduction scratch aliases fbuf");
    __shared__ __align__(16) cx<T> fbuf[L * TB];
    __shared__ __align__(16) cx<T> stg[STGN];
    __shared__ __align__(16) cx<T> twl[TWN];
    extern __shared__ double hist[];  // [NW][nbins]
    const int t = threadIdx.x;
    const int nb = e.nbins;
    if (INV && blockIdx.x == 0 && t == 0) *x1v = 1;  // read by the next step's inverse y pass only
    for (int i = t; i < NW * nb; i += NT) hist[i] = 0.0;
    for (int i = t; i < TWN; i += NT) twl[i] = ((const cx<T>*)a.tw)[i];
    __syncthreads();
    double* myh = hist + (t >> 6) * nb;
    const EpiScalars q = epi_scalars(e);
    double om = 0.0, ed_unused = 0.0;
    const double inv_nf = 1.0 / e.nf;
    const int nout = a.nout, hout = nout / 2;
    const int ntiles = (a.B + TB - 1) / TB;
    const int64_t nitems = (int64_t)a.A * ntiles;
    const int G = gridDim.x;  // a multiple of 8
    const int64_t lin = (int64_t)(blockIdx.x % 8) * (G / 8) + blockIdx.x / 8;

    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const uint32_t stg_base = lds_addr(stg);
    const int nslot = a.nin * SPR;
    auto issue = [&](int64_t it, int c) {
        const int64_t ai = it / ntiles;
        const int b0 = (int)(it - ai * ntiles) * TB;
        const cx<T>* in = (const cx<T>*)a.job[c].in + ai * a.in_a_stride + b0;
        for (int m = wave; m * 64 < nslot; m += NW) {
            const int s = m * 64 + lane;
            const int row = s / SPR, part = s - row * SPR;
            if (s < nslot) dma16(in + (int64_t)row * a.in_row_stride + part * EPS, stg_base + (uint32_t)m * 1024u);
        }
    };
    auto load = [&](int b, int p) -> cx<T> { return stg[p * TB + b]; };
    auto store_lds = [&](int b, int p, cx<T> v) { fbuf[p * TB + b] = v; };
    // INV: the FP64 state tile [nin][TB] of the component being transformed
    cx<double>* stgw = (cx<double>*)stg;
    auto issue_inv = [&](int64_t it, int c) {
        const int64_t ai = it / ntiles;
        const int b0 = (int)(it - ai * ntiles) * TB;
        const cx<double>* in = (const cx<double>*)ia.job[c].in + ai * ia.in_a_stride + b0;
        const int ns = ia.nin * TB;
        for (int m = wave; m * 64 < ns; m += NW) {
            const int s = m * 64 + lane;
            const int row = s / TB, col = s - row * TB;
            if (s < ns) dma16(in + (int64_t)row * ia.in_row_stride + col, stg_base + (uint32_t)m * 1024u);
        }
    };

    int64_t it = lin;
    if (it < nitems) issue(it, 0);
    dma_wait();
    lds_barrier();
    for (; it < nitems; it += G) {
        const int64_t ai = it / ntiles;
        const int b0 = (int)(it - ai * ntiles) * TB;
        const int i1 = (int)ai;
        const int k1 = wrap_k(i1, e.nk1);
        cx<T> keep[2][Q];
        auto comp = [&](auto cc) {
            constexpr int c = decltype(cc)::value;
            auto prefetch = [&]() {
                if (c < 2) issue(it, c + 1);
                else if (!INV && it + G < nitems) issue(it + G, 0);  // INV: the state parts come first
            };
            FftS<T, L, TB, NT, TB, -1, false, TWM>::template run<false>(fbuf, twl, load, store_lds, prefetch, t);
            lds_barrier();
            dma_wait();  // the next component's tile (this wave's copies) has landed
#pragma unroll
            for (int qq = 0; qq < Q; qq++) {
                const int idx = t + qq * NT;
                if (idx < nout * TB) {
                    const int i = idx / TB, b = idx - i * TB;
                    const int p = (i <= hout) ? i : L - (nout - i);
                    if constexpr (c < 2) {
                        keep[c][qq] = fbuf[p * TB + b];
                    } else {
                        const int k2 = wrap_k(i, e.nk2), k3 = b0 + b;
                        if (k3 < a.B && !(e.notcubic && ((k1 % e.Lx) || (k2 % e.Ly) || (k3 % e.Lz)))) {  // src/HIT_LES.cpp:867-871
                            const cx<T> v2 = fbuf[p * TB + b];
                            const cx<double> C[3] = {
                                cx<double>{(double)keep[0][qq].x * inv_nf, (double)keep[0][qq].y * inv_nf},
                                cx<double>{(double)keep[1][qq].x * inv_nf, (double)keep[1][qq].y * inv_nf},
                                cx<double>{(double)v2.x * inv_nf, (double)v2.y * inv_nf}};  // Fourier_Normalization
                            const int64_t m = ((int64_t)i * e.nk1 + i1) * e.nk3p + k3;
                            if constexpr (INV) {
                                cx<double> nn[3];
                                epi_mode<T>(e, q, m, k1, k2, k3, true, C, nullptr, myh, om, ed_unused, nn);
                                stgw[i * TB + b] = nn[0];
                            } else {
                                epi_mode<T>(e, q, m, k1, k2, k3, true, C, nullptr, myh, om, ed_unused);
                            }
                        } else if constexpr (INV) {
                            stgw[i * TB + b] = cx<double>{0.0, 0.0};  // padding columns: transformed, never written out
                        }
                    }
                }
            }
            lds_barrier();  // every wave's copies are in; fbuf is free again
        };
        static_for<3>(comp);
        if constexpr (INV) {
            // -------- the next step's inverse y pass of this item's new state
            // (component 0 is in the staging tile, published by the barrier
            // that ended the epilogue; the copies of components 1 and 2 read
            // the epilogue's stores, so every wave's stores complete first)
            dma_wait();
            lds_barrier();
            const int ihin = ia.nin / 2;
            // a runtime loop over the components, with the thread index through
            // an opaque copy: per-thread addresses are recomputed per component
            // rather than held across the item (register pressure)
            for (int c = 0; c < 3; c++) {
                const int tl = opaque(t);
                auto next = [&]() {
                    if (c < 2) issue_inv(it, c + 1);
                    else if (it + G < nitems) issue(it + G, 0);
                };
                auto none = [] {};
                int deriv = 0;  // 0 for the plain transform, 1 for the i k2 one
                // the inverse pass's loader (its input precision is FP64: i k u
                // formed in FP64, then rounded to T)
                auto load_inv = [&](int b, int p) -> cx<T> {
                    int i, k;
                    if (p <= ihin) { i = p; k = p; }
                    else if (p >= L - ihin) { i = ia.nin - (L - p); k = p - L; }
                    else return cx<T>{(T)0, (T)0};
                    const cx<double> v = stgw[i * TB + b];
                    if (deriv) return times_ik<T>((double)k, v);
                    return cx<T>{(T)v.x, (T)v.y};
                };
                auto write_inv = [&](void* dst) {
                    cx<T>* o = (cx<T>*)dst + ai * ia.out_a_stride + b0;
                    for (int idx = tl; idx < L * TB; idx += NT) {
                        const int i = idx / TB, b = idx - i * TB;
                        if (b0 + b < ia.B) o[(int64_t)i * ia.out_row_stride + b] = fbuf[i * TB + b];
                    }
                };
                FftS<T, L, TB, NT, TB, +1, false, TWM>::template run<false>(fbuf, twl, load_inv, store_lds, none, tl);
                lds_barrier();
                write_inv(ia.job[c].out);
                deriv = 1;
                FftS<T, L, TB, NT, TB, +1, false, TWM>::template run<true>(fbuf, twl, load_inv, store_lds, next, tl);
                lds_barrier();
                dma_wait();  // the next component's (or item's) tile has landed
                write_inv(ia.job[c].out2);
                lds_barrier();
            }
        }
    }
    epi_flush<NT>(e, hist, om, (double*)fbuf);
}

// ---------------------------------------------------------------------------
// The same at the short lengths, with an item's fields side by side: one
// forward transform of all 3 (LES: 9) TB columns, the epilogue, and with INV one
// inverse transform of the 6 TB columns (u_c, then d/dy u_c).  Also the LES form.
// What bounds these sizes is the chain of transforms and barriers a block runs
// through, not bytes: nine transforms one after the other at 48 points, two here.
// The transform
// buffer is the copy's target and the inverse's input, so nothing else is staged
// and several blocks fit a CU, which hides the copies.
// fwd_y + epilogue + next inv_y, a step: 32^3 DNS FP32 21.3 -> 5.8 us; in three
// kernels before: 96x64x64 LES FP32 41 -> 25 us, 16 of them 616 -> 400.
// ---------------------------------------------------------------------------
template <typename T, int L, bool LES>
struct YComb {
    static constexpr int NF = LES ? 9 : 3;
    static constexpr size_t bytes(int tb) { return sizeof(cx<T>) * L * (size_t)(NF > 6 ? NF : 6) * tb; }
    // 4 columns at the shortest lengths: 147 against 170 us a step for 16 x 32^3
    static constexpr int TB = L <= 48 || bytes(8) > 112 * 1024 ? 4 : 8;
    // one butterfly a thread in every stage as far as 1024 threads go (LES from 128
    // on: two to five).  State and history are the separate kernels' bit for bit at
    // every length; two a thread where one would do had changed FP32 bits.
    static constexpr int NT = sstage_nt<L, (NF > 6 ? NF : 6) * TB>();
    // state and history read before the forward transform: at the shortest
    // lengths (beyond, the registers cost more than the latency)
    static constexpr bool PRE = L <= 72;
    static constexpr int TWM = sizeof(T) == 8 ? 1 : 2;
    static constexpr size_t lds = bytes(TB) + sizeof(cx<T>) * fft_twiddle_span<L, TWM>();
    // DNS: from 96 points on the batched runs are faster with k_yepi's smaller
    // blocks (16 x 64^3 FP32: 691 against 838 us a step; one run 97 against 84).
    // LES, which has no other fused form: to 144 points, FP64 to 192 (128^3 870 ->
    // 808 us; FP32 there 612 -> 606, but a batch of 16 7.80 -> 8.17 ms).  Several LES
    // forms spill (1024 threads hold 128 VGPRs: 38 at 72 FP64, 19 at 128 FP32, up to
    // 16 at 96, 144 and 192), and each is still faster than the separate kernels, a
    // step: 48x48x64 at 72 FP64 89 against 104 us, 128x84x64 at 128 FP32 215 against
    // 263, 8 x 96^3 at 144 FP32 1.55 against 1.77 ms, 8 x 128^3 FP64 6.10 against 6.53.
    static constexpr bool use = L <= (!LES ? 72 : sizeof(T) == 8 ? 192 : 144) && lds <= 144 * 1024;
};

template <typename T, int L, bool LES, bool INV>
__device__ __forceinline__ void ycomb_body(const StridedArgs& a, const EpiArgs& e, const StridedArgs& ia, int* x1v)
{
    using Y = YComb<T, L, LES>;
    constexpr int TB = Y::TB, NT = Y::NT, NF = Y::NF, NW = NT / 64, TWM = Y::TWM;
    constexpr int NBF = NF * TB, NBI = 6 * TB;
    constexpr int TWN = fft_twiddle_span<L, TWM>();
    constexpr int EPS = 16 / (int)sizeof(cx<T>), SPF = TB / EPS, SPR = NF * SPF;  // 16-byte copy slots per field and per row
    constexpr int NOUTMAX = 2 * (L / 3) + 1;
    constexpr int Q = (NOUTMAX * TB + NT - 1) / NT;
    __shared__ __align__(16) cx<T> fbuf[L * (NBF > NBI ? NBF : NBI)];
    __shared__ __align__(16) cx<T> twl[TWN];
    __shared__ const cx<T>* src[NF];
    extern __shared__ double hist[];  // [NW][nbins]
    static_assert(sizeof(fbuf) >= NW * sizeof(double), "reduction scratch aliases fbuf");
    const int t = threadIdx.x, nb = e.nbins;
    if (INV && blockIdx.x == 0 && t == 0) *x1v = 1;  // read by the next step's inverse y pass only
    if (t < NF) src[t] = (const cx<T>*)a.job[t].in;
    for (int i = t; i < NW * nb; i += NT) hist[i] = 0.0;
    for (int i = t; i < TWN; i += NT) twl[i] = ((const cx<T>*)a.tw)[i];
    __syncthreads();
    double* myh = hist + (t >> 6) * nb;
    const EpiScalars q = epi_scalars(e);
    double om = 0.0, ed_unused = 0.0;
    const double inv_nf = 1.0 / e.nf;
    const int nout = a.nout, hout = nout / 2;
    const int ntiles = (a.B + TB - 1) / TB;
    const int nitems = a.A * ntiles, G = gridDim.x;  // G a multiple of 8
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    const uint32_t base = lds_addr(fbuf);
    auto none = [] {};
    for (int it = (blockIdx.x % 8) * (G / 8) + blockIdx.x / 8; it < nitems; it += G) {
        const int i1 = it / ntiles, b0 = (it - i1 * ntiles) * TB;
        const int k1 = wrap_k(i1, e.nk1);
        const int64_t off = (int64_t)i1 * a.in_a_stride + b0;
        for (int m = wave; m * 64 < L * SPR; m += NW) {
            const int s = m * 64 + lane;
            const int row = s / SPR, r = s - row * SPR, f = r / SPF;
            if (s < L * SPR) dma16(src[f] + off + (int64_t)row * a.in_row_stride + (r - f * SPF) * EPS, base + (uint32_t)m * 1024u);
        }
        // this thread's modes: i = k2 index, b = column
        cx<double> U[Q][3], R0[Q][3];
        bool ok[Q];
#pragma unroll
        for (int qq = 0; qq < Q; qq++) {
            const int idx = t + qq * NT, i = idx / TB, b = idx - i * TB;
            const int k2 = wrap_k(i, e.nk2), k3 = b0 + b;
            ok[qq] = idx < nout * TB && k3 < a.B && !(e.notcubic && ((k1 % e.Lx) || (k2 % e.Ly) || (k3 % e.Lz)));  // src/HIT_LES.cpp:867-871
            if (Y::PRE && ok[qq]) epi_load<T>(e, ((int64_t)i * e.nk1 + i1) * e.nk3p + k3, true, U[qq], R0[qq]);
        }
        dma_wait();
        lds_barrier();
        auto load_f = [&](int b, int p) -> cx<T> { return fbuf[p * NBF + b]; };
        auto store_f = [&](int b, int p, cx<T> v) { fbuf[p * NBF + b] = v; };
        FftS<T, L, NBF, NT, NBF, -1, true, TWM>::template run<false>(fbuf, twl, load_f, store_f, none, t);
        lds_barrier();
        cx<double> nn[Q][3];
#pragma unroll
        for (int qq = 0; qq < Q; qq++) {
            const int idx = t + qq * NT, i = idx / TB, b = idx - i * TB;
            if (ok[qq]) {
                const int p = (i <= hout) ? i : L - (nout - i);
                const int k2 = wrap_k(i, e.nk2), k3 = b0 + b;
                cx<double> CS[NF];  // convective term, then SGS stress 11 21 22 31 32 33 (Fourier_Normalization)
#pragma unroll
                for (int f = 0; f < NF; f++) {
                    const cx<T> v = fbuf[p * NBF + f * TB + b];
                    CS[f] = cx<double>{(double)v.x * inv_nf, (double)v.y * inv_nf};
                }
                if (!Y::PRE) epi_load<T>(e, ((int64_t)i * e.nk1 + i1) * e.nk3p + k3, true, U[qq], R0[qq]);
                epi_core<T>(e, q, ((int64_t)i * e.nk1 + i1) * e.nk3p + k3, k1, k2, k3, true, U[qq], R0[qq], CS, LES ? CS + (LES ? 3 : 0) : nullptr,
                            myh, om, ed_unused, nn[qq]);
            }
        }
        lds_barrier();  // every wave has read its transforms
        if constexpr (INV) {
            const int hin = ia.nin / 2;
#pragma unroll
            for (int qq = 0; qq < Q; qq++) {
                const int idx = t + qq * NT, i = idx / TB, b = idx - i * TB;
                if (ok[qq]) {
                    const int k2 = wrap_k(i, e.nk2), p = (i <= hin) ? i : L - (ia.nin - i);
#pragma unroll
                    for (int c = 0; c < 3; c++) {
                        fbuf[p * NBI + c * TB + b] = cx<T>{(T)nn[qq][c].x, (T)nn[qq][c].y};
                        fbuf[p * NBI + (3 + c) * TB + b] = times_ik<T>((double)k2, nn[qq][c]);
                    }
                }
            }
            lds_barrier();
            auto load_i = [&](int b, int p) -> cx<T> {
                const cx<T> v = fbuf[p * NBI + b];
                const bool in = p <= hin || p >= L - hin;  // else zero padding
                return cx<T>{in ? v.x : (T)0, in ? v.y : (T)0};
            };
            auto store_i = [&](int b, int p, cx<T> v) { fbuf[p * NBI + b] = v; };
            FftS<T, L, NBI, NT, NBI, +1, true, TWM>::template run<false>(fbuf, twl, load_i, store_i, none, t);
            lds_barrier();
#pragma unroll
            for (int c = 0; c < 6; c++) {
                cx<T>* o = (cx<T>*)(c < 3 ? ia.job[c % 3].out : ia.job[c % 3].out2) + (int64_t)i1 * ia.out_a_stride + b0;
                for (int idx = t; idx < L * TB; idx += NT) {
                    const int i = idx / TB, b = idx - i * TB;
                    if (b0 + b < ia.B) o[(int64_t)i * ia.out_row_stride + b] = fbuf[i * NBI + c * TB + b];
                }
            }
            lds_barrier();
        }
    }
    epi_flush<NT>(e, hist, om, (double*)fbuf);
}

template <typename T, int L, bool LES, bool INV>
__global__ __launch_bounds__((YComb<T, L, LES>::NT)) void k_ycomb(StridedArgs a, EpiArgs e, StridedArgs ia, int* x1v)
{
    ycomb_body<T, L, LES, INV>(a, e, ia, x1v);
}

template <typename T, int L, bool LES, bool INV>
__global__ __launch_bounds__((YComb<T, L, LES>::NT)) void k_ycomb_b(const StridedArgs* __restrict__ arr, const EpiArgs* __restrict__ earr,
                                                                    const StridedArgs* __restrict__ iarr, const int* __restrict__ left)
{
    if (left[blockIdx.y] <= 0) return;
    if constexpr (INV) {
        const StridedArgs& ia = iarr[blockIdx.y];
        ycomb_body<T, L, LES, true>(arr[blockIdx.y], earr[blockIdx.y], ia, ia.setflag);
    } else {
        ycomb_body<T, L, LES, false>(arr[blockIdx.y], earr[blockIdx.y], arr[blockIdx.y], nullptr);
    }
}

template <typename T, int L, int TB, int NT>
__global__ __launch_bounds__(NT) void k_yepi(StridedArgs a, EpiArgs e)
{
    yepi_body<T, L, TB, NT>(a, e, a, nullptr);
}

template <typename T, int L, int TB, int NT>
__global__ __launch_bounds__(NT) void k_yepi_inv(StridedArgs a, EpiArgs e, StridedArgs ia, int* x1v)
{
    yepi_body<T, L, TB, NT, true>(a, e, ia, x1v);
}

// batched k_yepi_inv: slot = blockIdx.y; each slot's flag is its inverse
// pass struct's setflag
template <typename T, int L, int TB, int NT>
__global__ __launch_bounds__(NT) void k_yepi_inv_b(const StridedArgs* __restrict__ arr, const EpiArgs* __restrict__ earr,
                                                   const StridedArgs* __restrict__ iarr, const int* __restrict__ left)
{
    if (left[blockIdx.y] <= 0) return;
    const StridedArgs& ia = iarr[blockIdx.y];
    yepi_body<T, L, TB, NT, true>(arr[blockIdx.y], earr[blockIdx.y], ia, ia.setflag);
}

template <typename T, int L, int TB, int NT>
__global__ __launch_bounds__(NT) void k_yepi_b(const StridedArgs* __restrict__ arr, const EpiArgs* __restrict__ earr,
                                               const int* __restrict__ left)
{
    if (left[blockIdx.y] <= 0) return;
    yepi_body<T, L, TB, NT>(arr[blockIdx.y], earr[blockIdx.y], arr[blockIdx.y], nullptr);
}

// ---------------------------------------------------------------------------
// Self-adaptive time step helpers (src/HIT_LES.h:249-269, src/HIT_LES.cpp:1049-1078)
// ---------------------------------------------------------------------------
static __device__ double FuL(double x, double x0, double x1, double f0, double f1) { return f0 + (x - x0) * (f1 - f0) / (x1 - x0); }
static __device__ double FuQ(double x, double x0, double x1) { return (x - x0) * (x - x1); }
static __device__ double FuG(double x, double a, double b, double c, double x0, double x1, double f0, double f1)
{
    return (a * x * x + b * x + c) * FuQ(x, x0, x1) + FuL(x, x0, x1, f0, f1);
}

// ---------------------------------------------------------------------------
// Finalize: fixed-order sums of the partials; time step (src/HIT_LES.cpp:365-403)
// With FIN_REDUCE the grid has one block per 64 shells: block x sums its
// shells' block partials (wave w takes rows w, w + 16, ...), and the block that
// arrives last does the rest.  What bounds it is latency: of the partials'
// reads, which other XCDs wrote (so a shell's rows are read sixteen at a time
// and every read that depends on nothing is issued first), and of the exchanges
// between the waves (one for all block sums; the shells go from block to block
// through one wave's fence and reads).  One block that summed part after part
// took 60 us at 512^3 DNS (256 x 445 partials), 51 at 256^3 LES (1024 x 223) and
// 10.4 at 32^3; this 9, 17 and 5.8.
// Returns whether this block was the last one of its context's launch.
// ---------------------------------------------------------------------------
template <int NT>
__device__ __forceinline__ bool finalize_body(const FinArgs& a)
{
    constexpr int NW = NT / 64, U = 16, UZ = 3;
    __shared__ double q[NW][64];
    __shared__ double red[NW * 6];
    __shared__ int last;
    DevScalars* s = a.scal;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const bool zsum = a.flags & (FIN_SKEW | FIN_EPHYS | FIN_MAXVEL);
    const int K = blockIdx.x * 64 + lane;
    const double nu = s->nu;
    double om = 0.0, ed = 0.0, s2 = 0.0, s3 = 0.0, mx = 0.0, mxs = 0.0;
    double z[UZ][4];
#pragma unroll
    for (int u = 0; u < UZ; u++)
#pragma unroll
        for (int i = 0; i < 4; i++) z[u][i] = (zsum && t + u * NT < a.nblk_z) ? a.z_partial[4 * (t + u * NT) + i] : 0.0;
    if ((a.flags & FIN_REDUCE) && t < a.nblk_epi) om = a.om_partial[t];
    if ((a.flags & FIN_EFOUR) && t < a.nblk_epi) ed = a.ed_partial[t];
    double e = 0.0, ef = 0.0;  // wave 0: its lanes' shells
    if (a.flags & FIN_REDUCE) {
        double acc = 0.0;
        for (int b = w; b < a.nblk_epi; b += U * NW) {
            double h[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                h[u] = (K < a.nbins && b + u * NW < a.nblk_epi) ? a.hist_partial[(int64_t)(b + u * NW) * a.nbins + K] : 0.0;
#pragma unroll
            for (int d = U / 2; d > 0; d >>= 1)
#pragma unroll
                for (int u = 0; u < d; u++) h[u] += h[u + d];
            acc += h[0];
        }
        q[w][lane] = acc;
        __syncthreads();
        if (w == 0) {
            if (K < a.nbins) {
                e = q[0][lane];
#pragma unroll
                for (int i = 1; i < NW; i++) e += q[i][lane];
                a.ek[K] = e;
            }
            if (gridDim.x > 1) {
                // this block's shells (all written by this wave) before its
                // count; the last block leaves the counter at 0
                __threadfence();
                if (lane == 0) {
                    last = atomicAdd(a.ticket, 1) == (int)gridDim.x - 1;
                    if (last) atomicExch(a.ticket, 0);
                }
                __threadfence();
            }
        }
        if (gridDim.x > 1) {
            __syncthreads();
            if (!last) return false;
            if (w == 0) {
                e = 0.0;
                for (int k = lane; k < a.nbins; k += 64) {
                    const double v = a.ek[k];
                    e += v;
                    if (k >= a.kfmin && k <= a.kfmax) ef += v;
                }
            }
        } else if (w == 0 && K >= a.kfmin && K <= a.kfmax) {
            ef = e;
        }
        for (int b = t + NT; b < a.nblk_epi; b += NT) om += a.om_partial[b];
    }
    if (a.flags & FIN_EFOUR)
        for (int b = t + NT; b < a.nblk_epi; b += NT) ed += a.ed_partial[b];
#pragma unroll
    for (int u = 0; u < UZ; u++) { s2 += z[u][0]; s3 += z[u][1]; mx = fmax(mx, z[u][2]); mxs = fmax(mxs, z[u][3]); }
    if (zsum)
        for (int b = t + UZ * NT; b < a.nblk_z; b += NT) {
            s2 += a.z_partial[4 * b];
            s3 += a.z_partial[4 * b + 1];
            mx = fmax(mx, a.z_partial[4 * b + 2]);
            mxs = fmax(mxs, a.z_partial[4 * b + 3]);
        }
    if (w == 0) {
        e = wave_sum(e);
        ef = wave_sum(ef);
    }
    double v[6] = {om, ed, s2, s3, mx, mxs};
    block_reduce<NT, 6, 4>(v, red);
    if (t == 0) {
        if (a.flags & FIN_REDUCE) {
            s->ek = e;
            s->om = v[0];
            s->relambda = e / nu * sqrt(20.0 / 3.0 / v[0]);
            // constant-power coefficient for the next step (src/HIT_LES.cpp:251-256)
            s->alpha = (ef > 1e-30) ? a.force_eps / (2.0 * ef) : 0.0;
        }
        if (a.flags & FIN_SKEW) { s->skew2 = v[2]; s->skew3 = v[3]; }
        if (a.flags & FIN_EFOUR) s->ek_four = v[1];
        if (a.flags & FIN_EPHYS) s->ek_phys = v[2];
        if (a.flags & FIN_MAXVEL) { s->maxvel = v[4]; s->maxvel_sa = v[5]; }
        if (a.flags & FIN_DT) {
            if (a.sa) {
                const double MaxVel = s->maxvel_sa, Ah = a.Ah;
                const double phi0 = atan(MaxVel * Ah * Ah / (0.35 * nu * 12.0));
                double Topt, Kopt;
                const double PI = 3.141592653589793238462643;
                if (phi0 >= 0.0 && phi0 < a.phi[0]) Topt = FuG(phi0, 0.0, a.c[0], a.c[1], 0.0, a.phi[0], 4.0 / 3.0, a.t1);
                else Topt = FuG(phi0, a.c[2], a.c[3], a.c[4], a.phi[0], PI / 2.0, a.t1, 1.0);
                if (phi0 >= 0.0 && phi0 <= a.phi[0]) Kopt = 1.0;
                else if (phi0 > a.phi[0] && phi0 <= a.phi[1]) Kopt = FuG(phi0, a.c[5], a.c[6], a.c[7], a.phi[0], a.phi[1], 1.0, a.kk[0]);
                else if (phi0 > a.phi[1] && phi0 <= a.phi[2]) Kopt = FuG(phi0, a.c[8], a.c[9], a.c[10], a.phi[1], a.phi[2], a.kk[0], a.kk[1]);
                else Kopt = FuG(phi0, a.c[11], a.c[12], a.c[13], a.phi[2], PI / 2.0, a.kk[1], 0.0);
                double At = Topt / sqrt((MaxVel * MaxVel) / (0.35 * 0.35) + (144.0 * nu * nu / (Ah * Ah * Ah * Ah)));
                s->kappa = Kopt;
                s->dt = a.C_At * At;
            } else {
                const double ax2 = a.Ax * a.Ax, ay2 = a.Ay * a.Ay, az2 = a.Az * a.Az;
                const double C_visc = 0.2 * fmin(ax2, fmin(ay2, az2)) / nu;
                const double C_conv = 0.35 / s->maxvel;
                double At = fmin(C_visc, C_conv);
                s->dt = a.C_At * At;
                if (a.fixed_dt > 0.0) s->dt = a.fixed_dt;
            }
        }
        if (a.flags & FIN_ADVANCE) {
            s->time = s->time + s->dt;
            s->iter = s->iter + 1;
        }
    }
    return true;
}

template <int NT>
__global__ __launch_bounds__(NT) void k_finalize(FinArgs a)
{
    finalize_body<NT>(a);
}

// Batched form: the slot's step ends here, so its steps-left counter drops
// by one: by the slot's last block, after every wave of its blocks has read it
// at entry.
template <int NT>
__global__ __launch_bounds__(NT) void k_finalize_b(const FinArgs* __restrict__ arr, int* __restrict__ left)
{
    if (left[blockIdx.y] <= 0) return;
    const bool last = finalize_body<NT>(arr[blockIdx.y]);
    __syncthreads();
    if (last && threadIdx.x == 0) left[blockIdx.y] -= 1;
}

// Streaming copy (the measured practical HBM ceiling beside the data-sheet
// peak): each thread moves U 16-byte vectors per iteration, all loads
// issued before the stores, non-temporal so the copy does not keep lines in
// the caches; XCD-interleaved block order is irrelevant for a linear sweep.
typedef float vf4 __attribute__((ext_vector_type(4)));
template <int U>
__global__ __launch_bounds__(256) void k_stream_copy(const vf4* __restrict__ in, vf4* __restrict__ out, int64_t n)
{
    const int64_t stride = (int64_t)gridDim.x * 256 * U;
    for (int64_t base = (int64_t)blockIdx.x * 256 * U + threadIdx.x; base < n; base += stride) {
        vf4 v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t i = base + (int64_t)u * 256;
            if (i < n) v[u] = __builtin_nontemporal_load(in + i);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int64_t i = base + (int64_t)u * 256;
            if (i < n) __builtin_nontemporal_store(v[u], out + i);
        }
    }
}

// The state between the pitched fields and the host's compact box.  Rows of
// nk3 modes leave the pitch here, on the device, so that what crosses the host
// link is one contiguous copy: a strided copy to pageable memory moved row by
// row (6.7 us each: 350 ms for a 128^3 state of 52 MB, and 460 ms inwards).
// Bounded by HBM: one read and one write of the state, 0.03 ms there.  A launch
// takes one piece of the box; its contiguous side is device or pinned memory.

// Element i of the launch: its field, row and k3.
static __device__ __forceinline__ void pack_element(const PackArgs& a, uint32_t i, uint32_t& c, uint32_t& r, uint32_t& k3)
{
    const uint32_t per = a.nrow * a.nk3;  // < 2^31 (the launcher's check)
    const uint64_t e = (uint64_t)a.first + i;
    c = e >= 2ull * per ? 2 : e >= per ? 1 : 0;
    const uint32_t q = (uint32_t)(e - (uint64_t)c * per);
    r = q / a.nk3;
    k3 = q - r * a.nk3;
    r += a.row0;
}

template <typename TS>
__global__ __launch_bounds__(256) void k_pack(PackArgs a)
{
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < a.n; i += gridDim.x * 256u) {
        uint32_t c, r, k3;
        pack_element(a, i, c, r, k3);
        const cx<TS>* in = (const cx<TS>*)(c == 0 ? a.padded[0] : c == 1 ? a.padded[1] : a.padded[2]);
        const cx<TS> v = in[(int64_t)r * a.nk3p + k3];
        a.compact[i] = cx<double>{(double)v.x, (double)v.y};
    }
}

static __global__ __launch_bounds__(256) void k_unpack(PackArgs a)
{
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < a.n; i += gridDim.x * 256u) {
        uint32_t c, r, k3;
        pack_element(a, i, c, r, k3);
        cx<double> v = a.compact[i];
        if (a.notcubic) {  // src/HIT_LES.cpp:867-871
            const int row = (int)r, i2 = row / a.nk1;
            const int k1 = wrap_k(row - i2 * a.nk1, a.nk1), k2 = wrap_k(i2, a.nk2);
            if ((k1 % a.Lx) || (k2 % a.Ly) || ((int)k3 % a.Lz)) v = cx<double>{0.0, 0.0};
        }
        cx<double>* out = (cx<double>*)(c == 0 ? a.padded[0] : c == 1 ? a.padded[1] : a.padded[2]);
        out[(int64_t)r * a.nk3p + k3] = v;
    }
}

// Steps-left counters of a batch for its next chunk, from the kernel's
// arguments (so the host may reuse its copy right after the launch).
static __global__ void k_set_left(int* left, SlotSteps s, int nslots)
{
    if ((int)threadIdx.x < nslots) left[threadIdx.x] = s.n[threadIdx.x];
}

// Spectrum imposition (src/HIT_LES.cpp:410-444): FT[K] from E(K), then scale.
static __global__ void k_forcing_ft(const double* ek, const double* forced, double* ft, int last_eff)
{
    for (int K = threadIdx.x; K <= last_eff; K += blockDim.x)
        ft[K] = ((ek[K] > 0.0) ? sqrt(forced[K] / ek[K]) : 0.0);
}

static __global__ void k_scale_shells(ShellArgs a)
{
    const int nk1 = a.nk1, nk2 = a.nk2, nk3 = a.nk3, nk3p = a.nk3p;
    for (int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; m < a.nmodes; m += (int64_t)gridDim.x * blockDim.x) {
        const int i3 = (int)(m % nk3p);
        if (i3 >= nk3) continue;  // pitch padding
        const int64_t r12 = m / nk3p;
        const int i1 = (int)(r12 % nk1), i2 = (int)(r12 / nk1);
        const int k1 = wrap_k(i1, nk1), k2 = wrap_k(i2, nk2), k3 = i3;
        if (a.notcubic && ((k1 % a.Lx) || (k2 % a.Ly) || (k3 % a.Lz))) continue;
        const int K = shell_of(k1 * k1 + k2 * k2 + k3 * k3);
        for (int c = 0; c < 3; c++) {
            cx<double> v = a.uk[c][m];
            if (K <= a.last_eff) { v.x *= a.ft[K]; v.y *= a.ft[K]; }
            else if (a.nullify) v = cx<double>{0.0, 0.0};
            a.uk[c][m] = v;
        }
    }
}

// Complex conjugate correction of the k3 = 0 plane (src/HIT_LES.cpp:446-476)
static __global__ void k_ccc(ShellArgs a)
{
    const int nk1 = a.nk1, nk2 = a.nk2;
    const int n = nk1 * nk2;
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) {
        const int i1 = q % nk1, i2 = q / nk1;
        const int k1 = wrap_k(i1, nk1), k2 = wrap_k(i2, nk2);
        if (k1 < 0 || (k1 == 0 && k2 < 0)) {
            const int j1 = (-k1 >= 0) ? -k1 : nk1 - k1;
            const int j2 = (-k2 >= 0) ? -k2 : nk2 - k2;
            const int64_t m = ((int64_t)i2 * nk1 + i1) * a.nk3p;
            const int64_t mc = ((int64_t)j2 * nk1 + j1) * a.nk3p;
            for (int c = 0; c < 3; c++) {
                cx<double> v = a.uk[c][mc];
                a.uk[c][m] = cx<double>{v.x, -v.y};
            }
        }
    }
}

// Normalisation of a reference-layout complex field on the retained set
// (src/FFTW_package.cpp:33-42).
template <typename T>
__global__ void k_normalize(NormArgs a)
{
    const int nk = a.Mz / 2 + 1;
    const int64_t n = (int64_t)a.My * a.Mx * nk;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
        const int k3 = (int)(q % nk);
        const int64_t r = q / nk;
        const int ax = (int)(r % a.Mx), by = (int)(r / a.Mx);
        const int k1 = (ax <= a.Mx / 2) ? ax : ax - a.Mx, k2 = (by <= a.My / 2) ? by : by - a.My;
        bool rel = (abs(k1) <= a.Nx2 && abs(k2) <= a.Ny2 && k3 <= a.Nz2);
        if (a.notcubic && ((k1 % a.Lx) || (k2 % a.Ly) || (k3 % a.Lz))) rel = false;
        if (a.all || rel) {
            cx<T>* p = (cx<T>*)a.data;
            p[q].x = p[q].x / (T)a.nf;
            p[q].y = p[q].y / (T)a.nf;
        }
    }
}

// ---------------------------------------------------------------------------
// Launch tables
// ---------------------------------------------------------------------------
template <int L>
constexpr int zpass_nt()
{
    return L >= 768 ? 512 : (L >= 288 ? 256 : (L >= 144 ? 128 : 64));
}

// One launch of the staged kernel over the jobs JSEL selects (njsel of them).
template <typename TIN, typename TOUT, typename T, int L, int TB, int DIR, int JSEL>
static hipError_t launch_sstage(const StridedArgs& b, int A, int njsel, hipStream_t st, const BatchLaunch* bl)
{
    constexpr int NB = JSEL == 1 ? 2 * TB : TB;
    constexpr int NT = sstage_nt<L, NB>();
    constexpr int LR0 = L / Plan<L>::r(0);
    constexpr bool STDP_OK = DIR > 0 && (LR0 == 64 || LR0 == 128) && NB * LR0 <= NT;
    const bool stdp = STDP_OK && b.nin == 2 * (L / 3) + 1;
    static const int occ = [] {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_sstage<TIN, TOUT, T, L, TB, NT, DIR, false, JSEL>, NT, 0) !=
            hipSuccess)
            n = 1;
        return n > 0 ? n : 1;
    }();
    int dev = 0, ncu = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    const int64_t items = (int64_t)A * njsel * ((b.B + TB - 1) / TB);
    int64_t g = (int64_t)ncu * occ;
    if (items < g) g = items;
    g = (g + 7) / 8 * 8;
    if (bl) {
        // batched: each slot's struct (with A set) is in bl->args
        if constexpr (batch_length(L)) {
            const dim3 grid((unsigned)g, (unsigned)bl->nslots);
            const StridedArgs* arr = (const StridedArgs*)bl->args;
            if constexpr (STDP_OK) {
                if (stdp) {
                    hipLaunchKernelGGL((k_sstage_b<TIN, TOUT, T, L, TB, NT, DIR, true, JSEL>), grid, dim3(NT), 0, st, arr, bl->left);
                    return hipGetLastError();
                }
            }
            hipLaunchKernelGGL((k_sstage_b<TIN, TOUT, T, L, TB, NT, DIR, false, JSEL>), grid, dim3(NT), 0, st, arr, bl->left);
            return hipGetLastError();
        }
        return hipErrorNotSupported;
    }
    if constexpr (STDP_OK) {
        if (stdp) {
            hipLaunchKernelGGL((k_sstage<TIN, TOUT, T, L, TB, NT, DIR, true, JSEL>), dim3((unsigned)g), dim3(NT), 0, st, b);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((k_sstage<TIN, TOUT, T, L, TB, NT, DIR, false, JSEL>), dim3((unsigned)g), dim3(NT), 0, st, b);
    return hipGetLastError();
}

// The combined dual-job kernel (JSEL 1) for the inverse passes at L >= 512,
// unless SPNS_DUALC=0; the single jobs of the same pass then take a second
// launch.  At 512^3 it took FP64 inv_x from 8.00 to 7.59 ms and inv_y from
// 3.81 to 3.60 ms.  In FP32 it took inv_x from 4.01 to 3.76 ms, but with the
// pitch-9 z pass the z pass that follows ran 0.3 ms longer at the same cycle
// count (rocprofv3 GRBM_GUI_ACTIVE: a lower engine clock after the faster
// memory-bound kernel) and the step gained nothing; with the swizzled z pass
// the FP32 inv_x goes from 3.98 to 3.72 ms and the step to 16.76 ms on one
// box (16.81-17.03 ms without, on others), so both forms use it.
template <typename TIN, typename T, int L, int TB, int DIR>
constexpr bool dualc_applies()
{
    return DIR > 0 && L >= 512 && sstage_fits<TIN, T, L, TB, DIR, 2>();
}

static bool dualc_enabled()
{
    static const bool on = [] {
        const char* s = getenv("SPNS_DUALC");
        return !(s && s[0] == '0');
    }();
    return on;
}

template <typename TIN, typename TOUT, typename T, int L, int DIR>
static hipError_t launch_strided_L(const StridedArgs& a, int A, hipStream_t st, const BatchLaunch* bl)
{
    constexpr int TB = strided_tb<T, L>();
    StridedArgs b = a;
    b.A = A;
    if constexpr (sstage_fits<TIN, T, L, TB, DIR>()) {
        if (a.padded_ok && a.nin <= sstage_rows<L, DIR>()) {
            if constexpr (dualc_applies<TIN, T, L, TB, DIR>()) {
                int nd = 0;
                for (int j = 0; j < a.njobs; j++) nd += a.job[j].out2 != nullptr;
                if (nd > 0 && dualc_enabled()) {
                    hipError_t e = launch_sstage<TIN, TOUT, T, L, TB, DIR, 1>(b, A, nd, st, bl);
                    if (e == hipSuccess && nd < a.njobs) e = launch_sstage<TIN, TOUT, T, L, TB, DIR, 2>(b, A, a.njobs - nd, st, bl);
                    return e;
                }
            }
            return launch_sstage<TIN, TOUT, T, L, TB, DIR, 0>(b, A, a.njobs, st, bl);
        }
    }
    if (bl) return hipErrorNotSupported;  // no batched form of the direct-load kernel
    // the direct-load kernel takes single jobs: a dual job becomes two
    int n = 0;
    for (int j = 0; j < a.njobs; j++) {
        if (a.job[j].out2) {
            if (n + 2 > 9) return hipErrorInvalidValue;
            b.job[n++] = StridedJob{a.job[j].in, a.job[j].out, 0, 0, nullptr};
            b.job[n++] = StridedJob{a.job[j].in, a.job[j].out2, 1, 0, nullptr};
        } else {
            if (n + 1 > 9) return hipErrorInvalidValue;
            b.job[n++] = a.job[j];
        }
    }
    b.njobs = n;
    constexpr int NT = 256;
    const int64_t blocks = (int64_t)((a.B + TB - 1) / TB) * A;
    dim3 grid((unsigned)((blocks + 7) / 8 * 8), 1, 1);
    hipLaunchKernelGGL((k_strided<TIN, TOUT, T, L, TB, NT, DIR>), grid, dim3(NT), 0, st, b);
    return hipGetLastError();
}

#define SPNS_FOR_EACH_L(X) \
    X(16) X(24) X(32) X(36) X(48) X(64) X(72) X(96) X(128) X(144) X(192) X(256) X(288) X(384) X(512) X(576) X(768) X(1024) X(1152) X(1536)

#if SPNS_PART == 0 || SPNS_PART == 4
int strided_tile(int L, int prec)
{
#define X(LL) \
    if (L == LL) return prec == PREC_FP64 ? strided_tb<double, LL>() : strided_tb<float, LL>();
    SPNS_FOR_EACH_L(X)
#undef X
    return 0;
}

bool supported_length(int L)
{
#define X(LL) \
    if (L == LL) return true;
    SPNS_FOR_EACH_L(X)
#undef X
    return false;
}

#endif

template <typename TIN, typename TOUT, typename T, int DIR>
static hipError_t launch_strided_T(int L, const StridedArgs& a, int A, hipStream_t st, const BatchLaunch* bl)
{
#define X(LL) \
    if (L == LL) return launch_strided_L<TIN, TOUT, T, LL, DIR>(a, A, st, bl);
    SPNS_FOR_EACH_L(X)
#undef X
    return hipErrorInvalidValue;
}

#if SPNS_PART == 0 || SPNS_PART == 1
hipError_t launch_strided_fp64(int L, int dir, const StridedArgs& a, int A, hipStream_t st, const BatchLaunch* bl)
{
    return dir > 0 ? launch_strided_T<double, double, double, +1>(L, a, A, st, bl)
                   : launch_strided_T<double, double, double, -1>(L, a, A, st, bl);
}
#endif

#if SPNS_PART == 0 || SPNS_PART == 2
hipError_t launch_strided_fp32(int L, int in_fp64, int dir, const StridedArgs& a, int A, hipStream_t st, const BatchLaunch* bl)
{
    if (in_fp64) {
        return dir > 0 ? launch_strided_T<double, float, float, +1>(L, a, A, st, bl)
                       : launch_strided_T<double, float, float, -1>(L, a, A, st, bl);
    }
    return dir > 0 ? launch_strided_T<float, float, float, +1>(L, a, A, st, bl)
                   : launch_strided_T<float, float, float, -1>(L, a, A, st, bl);
}
#endif

#if SPNS_PART == 0 || SPNS_PART == 4
hipError_t launch_strided(int L, int prec, int in_fp64, int out_fp64, int dir, const StridedArgs& a, int A, hipStream_t st,
                          const BatchLaunch* bl)
{
    (void)out_fp64;
    if (prec == PREC_FP64) return launch_strided_fp64(L, dir, a, A, st, bl);
    return launch_strided_fp32(L, in_fp64, dir, a, A, st, bl);
}
#endif

template <class K>
static int blocks_per_cu(K kernel, int nt)
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, nt, 0) != hipSuccess) return -1;
    return nb > 0 ? nb : 1;
}

#if SPNS_PART == 0 || SPNS_PART == 6
template <typename T, int L, bool LES>
static hipError_t launch_zreg_L(const ZArgs& a, int grid, hipStream_t st, const BatchLaunch* bl)
{
    using Z = ZReg<T, L, LES>;
    if constexpr (LES ? Z::fits : zreg_dns<T, L>()) {
        if (a.nk3 != Z::NKC || a.npencil % Z::PP || grid < 1) return hipErrorInvalidValue;
        if (bl) {
            if constexpr (batch_length(L)) {
                hipLaunchKernelGGL((k_zreg_b<T, L, LES>), dim3((unsigned)grid, (unsigned)bl->nslots), dim3(Z::NT), 0, st,
                                   (const ZArgs*)bl->args, bl->left);
                return hipGetLastError();
            }
            return hipErrorNotSupported;
        }
        hipLaunchKernelGGL((k_zreg<T, L, LES>), dim3(grid), dim3(Z::NT), 0, st, a);
        return hipGetLastError();
    }
    return hipErrorNotSupported;
}

hipError_t launch_zreg(int L, int prec, const ZArgs& a, int grid, hipStream_t st, const BatchLaunch* bl)
{
#define X(LL)                                                                                                          \
    if (L == LL) {                                                                                                     \
        if (prec == PREC_FP64)                                                                                         \
            return a.les ? launch_zreg_L<double, LL, true>(a, grid, st, bl) : launch_zreg_L<double, LL, false>(a, grid, st, bl); \
        return a.les ? launch_zreg_L<float, LL, true>(a, grid, st, bl) : launch_zreg_L<float, LL, false>(a, grid, st, bl); \
    }
    SPNS_FOR_EACH_L(X)
#undef X
    return hipErrorInvalidValue;
}

template <typename T, int L, bool LES>
static int zreg_blocks_L()
{
    using Z = ZReg<T, L, LES>;
    if constexpr (LES ? Z::fits : zreg_dns<T, L>()) return blocks_per_cu(k_zreg<T, L, LES>, Z::NT);
    return -1;
}

int zreg_blocks(int L, int prec, bool les)
{
#define X(LL)                                                                                          \
    if (L == LL) {                                                                                     \
        if (prec == PREC_FP64) return les ? zreg_blocks_L<double, LL, true>() : zreg_blocks_L<double, LL, false>(); \
        return les ? zreg_blocks_L<float, LL, true>() : zreg_blocks_L<float, LL, false>();             \
    }
    SPNS_FOR_EACH_L(X)
#undef X
    return -1;
}
#endif

#if SPNS_PART == 0 || SPNS_PART == 7
// Grid of k_ycomb: both forms (with and without the inverse pass) take the
// smaller of their occupancies, so that the shell partials are the same.
template <typename T, int L, bool LES>
static int ycomb_grid_L(int nbins, int nout, int A, int B, int max_grid)
{
    using Y = YComb<T, L, LES>;
    if (nout > 2 * (L / 3) + 1) return 0;
    const size_t shm = sizeof(double) * (Y::NT / 64) * (size_t)nbins;
    if (Y::lds + shm + 256 > 160 * 1024 - 512) return 0;
    int n0 = 0, n1 = 0, dev = 0, ncu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n0, k_ycomb<T, L, LES, false>, Y::NT, shm) != hipSuccess || n0 < 1) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n1, k_ycomb<T, L, LES, true>, Y::NT, shm) != hipSuccess || n1 < 1) return 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    int64_t g = (int64_t)ncu * (n0 < n1 ? n0 : n1);
    const int64_t items = (int64_t)A * ((B + Y::TB - 1) / Y::TB);
    if (items < g) g = items;
    g = (g + 7) / 8 * 8;
    return (int)(g > max_grid ? max_grid / 8 * 8 : g);
}

template <typename T, int L, bool LES>
static hipError_t launch_ycomb_L(const StridedArgs& a, const EpiArgs& e, int grid, hipStream_t st, const BatchLaunch* bl, const StridedArgs* ia,
                                 int* x1v)
{
    using Y = YComb<T, L, LES>;
    const size_t shm = sizeof(double) * (Y::NT / 64) * (size_t)e.nbins;
    if (bl) {
        if constexpr (batch_length(L)) {
            const dim3 g(grid, bl->nslots);
            if (ia)
                hipLaunchKernelGGL((k_ycomb_b<T, L, LES, true>), g, dim3(Y::NT), shm, st, (const StridedArgs*)bl->args, (const EpiArgs*)bl->args2,
                                   (const StridedArgs*)bl->args3, bl->left);
            else
                hipLaunchKernelGGL((k_ycomb_b<T, L, LES, false>), g, dim3(Y::NT), shm, st, (const StridedArgs*)bl->args, (const EpiArgs*)bl->args2,
                                   (const StridedArgs*)bl->args3, bl->left);
            return hipGetLastError();
        }
        return hipErrorNotSupported;
    }
    if (ia) hipLaunchKernelGGL((k_ycomb<T, L, LES, true>), dim3(grid), dim3(Y::NT), shm, st, a, e, *ia, x1v);
    else hipLaunchKernelGGL((k_ycomb<T, L, LES, false>), dim3(grid), dim3(Y::NT), shm, st, a, e, a, nullptr);
    return hipGetLastError();
}

// the length's k_ycomb, where it is used (ycomb_use): f(L, T, LES) below
#define SPNS_YCOMB_CALL(FN, ...)                                                                              \
    if constexpr (YComb<T, LL_, true>::use) {                                                                 \
        if (les) return FN<T, LL_, true>(__VA_ARGS__);                                                        \
    }                                                                                                         \
    if constexpr (YComb<T, LL_, false>::use) {                                                                \
        if (!les) return FN<T, LL_, false>(__VA_ARGS__);                                                      \
    }

template <typename T, int LL_>
static int ycomb_grid_any(bool les, int nbins, int nout, int A, int B, int max_grid)
{
    SPNS_YCOMB_CALL(ycomb_grid_L, nbins, nout, A, B, max_grid)
    return 0;
}

template <typename T, int LL_>
static hipError_t launch_ycomb_any(bool les, const StridedArgs& a, const EpiArgs& e, int grid, hipStream_t st, const BatchLaunch* bl,
                                   const StridedArgs* ia, int* x1v)
{
    SPNS_YCOMB_CALL(launch_ycomb_L, a, e, grid, st, bl, ia, x1v)
    return hipErrorNotSupported;
}
#undef SPNS_YCOMB_CALL

int ycomb_grid(int L, int prec, bool les, int nbins, int nout, int A, int B, int max_grid)
{
#define X(LL)                                                                                              \
    if (L == LL)                                                                                           \
        return prec == PREC_FP64 ? ycomb_grid_any<double, LL>(les, nbins, nout, A, B, max_grid)            \
                                 : ycomb_grid_any<float, LL>(les, nbins, nout, A, B, max_grid);
    SPNS_FOR_EACH_L(X)
#undef X
    return 0;
}

hipError_t launch_ycomb(int L, int prec, const StridedArgs& a, const EpiArgs& e, int grid, hipStream_t st, const BatchLaunch* bl,
                        const StridedArgs* ia, int* x1v)
{
#define X(LL)                                                                                              \
    if (L == LL)                                                                                           \
        return prec == PREC_FP64 ? launch_ycomb_any<double, LL>(e.les, a, e, grid, st, bl, ia, x1v)        \
                                 : launch_ycomb_any<float, LL>(e.les, a, e, grid, st, bl, ia, x1v);
    SPNS_FOR_EACH_L(X)
#undef X
    return hipErrorInvalidValue;
}
#endif

#if SPNS_PART == 0 || SPNS_PART == 3
// Compile-time retained k3 count of the standard 3/2 padding (M = 3N/2,
// nk3 = N/2 + 1 = M/3 + 1), 0 where M is not a multiple of 3.
template <int L>
constexpr int zstage_nkc()
{
    return (L % 3 == 0) ? L / 3 + 1 : 0;
}

// Threads of the staged z pass.  FP32 at L = 768: 12 waves (measured 9.5 ms
// against 9.9 ms with 8 waves at 512^3); otherwise as the block kernel.
template <typename T, int L>
constexpr int zstage_nt()
{
    return (sizeof(T) == 4 && L == 768) ? 768 : zpass_nt<L>();
}

template <typename T, int L, int MODE>
static bool zstage_ok(const ZArgs& a)
{
    constexpr int NT = zstage_nt<T, L>();
    if constexpr (!zstage_fits<T, L, NT, MODE>()) return false;
    return a.pitch + zstage_pad<T>() <= zstage_spc<L>() && a.nk3 <= a.pitch;
}

// z-pass kernel variants and the choice among them
enum { ZV_BLOCK, ZV_WAVE, ZV_STAGE, ZV_STAGE_NKC, ZV_FUSE_NKC, ZV_REG };

template <typename T, int L>
constexpr int zfuse_nt()
{
    return sstage_nt<L, 8>();
}

template <typename T, int L>
constexpr bool zfuse_fits()
{
    return !zreg_dns<T, L>() && zstage_nkc<L>() > 0 && zfuse_lds_bytes<T, L, zfuse_nt<T, L>(), zstage_nkc<L>()>() <= 160 * 1024 - 512;
}

template <typename T, int L, int MODE>
static int zpass_pick(const ZArgs& a)
{
    if constexpr (MODE != 2 && has_wave_plan<L>::value) {
        if ((!a.les || MODE == 1) && a.kernel == ZK_WAVE) return ZV_WAVE;
    }
    if (a.kernel == ZK_STAGED || a.kernel == ZK_STAGED_NOFUSE) {
        const bool pitch_ok = a.pitch + zstage_pad<T>() <= zstage_spc<L>() && a.nk3 <= a.pitch;
        const bool nkc = zstage_nkc<L>() > 0 && a.nk3 == zstage_nkc<L>();
        if constexpr (MODE == 0 && L % 3 == 0) {
            if (a.kernel == ZK_STAGED && nkc && (a.les ? ZReg<T, L, true>::fits && a.npencil % ZReg<T, L, true>::PP == 0
                                                       : zreg_dns<T, L>() && a.npencil % ZReg<T, L, false>::PP == 0))
                return ZV_REG;
        }
        if constexpr (MODE == 0 && zfuse_fits<T, L>()) {
            if (a.kernel == ZK_STAGED && !a.les && pitch_ok && nkc) return ZV_FUSE_NKC;
        }
        if constexpr (zstage_fits<T, L, zstage_nt<T, L>(), MODE>()) {
            if (pitch_ok) return nkc ? ZV_STAGE_NKC : ZV_STAGE;
        }
    }
    return ZV_BLOCK;
}

template <typename T, int L, int MODE>
static hipError_t launch_zpass_L(const ZArgs& a, int grid, hipStream_t st, const BatchLaunch* bl)
{
    constexpr int NTS = zstage_nt<T, L>();
    constexpr int NKC = zstage_nkc<L>();
    if (bl) {
        // batched step (MODE 0) over the slots' structs in bl->args
        if constexpr (MODE == 0 && batch_length(L)) {
            const dim3 g((unsigned)grid, (unsigned)bl->nslots);
            const ZArgs* arr = (const ZArgs*)bl->args;
            switch (zpass_pick<T, L, MODE>(a)) {
            case ZV_REG:
                return launch_zreg(L, sizeof(T) == 8 ? PREC_FP64 : PREC_FP32, a, grid, st, bl);
            case ZV_FUSE_NKC:
                if constexpr (zfuse_fits<T, L>()) {
                    constexpr int NTF = zfuse_nt<T, L>();
                    hipLaunchKernelGGL((k_zfuse_b<T, L, NTF, NKC>), g, dim3(NTF), 0, st, arr, bl->left);
                    return hipGetLastError();
                }
                break;
            case ZV_STAGE_NKC:
                if constexpr (NKC > 0 && zstage_fits<T, L, NTS, MODE>()) {
                    hipLaunchKernelGGL((k_zstage_b<T, L, NTS, MODE, zstage_ld<MODE>(), 1, sizeof(T) == 4, NKC>), g, dim3(NTS), 0, st,
                                       arr, bl->left);
                    return hipGetLastError();
                }
                break;
            case ZV_STAGE:
                if constexpr (zstage_fits<T, L, NTS, MODE>()) {
                    hipLaunchKernelGGL((k_zstage_b<T, L, NTS, MODE>), g, dim3(NTS), 0, st, arr, bl->left);
                    return hipGetLastError();
                }
                break;
            default:
                break;
            }
        }
        return hipErrorNotSupported;
    }
    switch (zpass_pick<T, L, MODE>(a)) {
    case ZV_WAVE:
        if constexpr (has_wave_plan<L>::value) {
            hipLaunchKernelGGL((k_zwave<T, L, MODE>), dim3(grid), dim3(256), 0, st, a);
            return hipGetLastError();
        }
        break;
    case ZV_REG:
        return launch_zreg(L, sizeof(T) == 8 ? PREC_FP64 : PREC_FP32, a, grid, st, nullptr);
    case ZV_FUSE_NKC:
        if constexpr (MODE == 0 && zfuse_fits<T, L>()) {
            constexpr int NTF = zfuse_nt<T, L>();
            hipLaunchKernelGGL((k_zfuse<T, L, NTF, NKC>), dim3(grid), dim3(NTF), 0, st, a);
            return hipGetLastError();
        }
        break;
    case ZV_STAGE_NKC:
        if constexpr (NKC > 0 && zstage_fits<T, L, NTS, MODE>()) {
            hipLaunchKernelGGL((k_zstage<T, L, NTS, MODE, zstage_ld<MODE>(), 1, sizeof(T) == 4, NKC>), dim3(grid), dim3(NTS),
                               0, st, a);
            return hipGetLastError();
        }
        break;
    case ZV_STAGE:
        if constexpr (zstage_fits<T, L, NTS, MODE>()) {
            hipLaunchKernelGGL((k_zstage<T, L, NTS, MODE>), dim3(grid), dim3(NTS), 0, st, a);
            return hipGetLastError();
        }
        break;
    default:
        break;
    }
    if constexpr (MODE == 2) {
        return hipErrorNotSupported;  // the invariants pass exists only in the staged kernel
    } else {
        constexpr int NT = zpass_nt<L>();
        hipLaunchKernelGGL((k_zpass<T, L, NT, MODE>), dim3(grid), dim3(NT), 0, st, a);
        return hipGetLastError();
    }
}

// Grid of the z pass: the staged kernels run persistent blocks (as many as
// fit on the device at once, counted for the full step's kernel), the others
// one block per pencil up to 65536.
template <typename T, int L>
static int zpass_grid_L(const ZArgs& a, int64_t npen)
{
    constexpr int NTS = zstage_nt<T, L>();
    constexpr int NKC = zstage_nkc<L>();
    int nb = 0;
    int64_t items = npen;
    int min_groups = 1;
    switch (zpass_pick<T, L, 0>(a)) {
    case ZV_REG:
        nb = zreg_blocks(L, sizeof(T) == 8 ? PREC_FP64 : PREC_FP32, a.les);
        items = npen / (a.les ? zreg_pp<T, L, true>() : zreg_pp<T, L, false>());
        // a DNS block runs one step more than it has groups (its last products),
        // so at least two groups each, as long as every CU keeps two blocks
        // (16 x 32^3: 125 -> 114 us a step; one run the same)
        if (!a.les) min_groups = 2;
        break;
    case ZV_FUSE_NKC:
        if constexpr (zfuse_fits<T, L>()) nb = blocks_per_cu(k_zfuse<T, L, zfuse_nt<T, L>(), NKC>, zfuse_nt<T, L>());
        break;
    case ZV_STAGE_NKC:
        if constexpr (NKC > 0 && zstage_fits<T, L, NTS, 0>())
            nb = blocks_per_cu(k_zstage<T, L, NTS, 0, zstage_ld<0>(), 1, sizeof(T) == 4, NKC>, NTS);
        break;
    case ZV_STAGE:
        if constexpr (zstage_fits<T, L, NTS, 0>()) nb = blocks_per_cu(k_zstage<T, L, NTS, 0>, NTS);
        break;
    default:
        return (int)(npen < 65536 ? npen : 65536);
    }
    if (nb <= 0) return -1;
    int dev = 0, ncu = 0;
    if (hipGetDevice(&dev) != hipSuccess) return -1;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return -1;
    int64_t g = (int64_t)ncu * nb;
    if (items < g) g = items;
    const int64_t fewer = (items + min_groups - 1) / min_groups;
    if (fewer < g && fewer >= 2 * ncu) g = fewer;
    return (int)g;
}

int zpass_grid(int L, int prec, const ZArgs& a, int64_t npen)
{
#define X(LL)                                                                                          \
    if (L == LL) return prec == PREC_FP64 ? zpass_grid_L<double, LL>(a, npen) : zpass_grid_L<float, LL>(a, npen);
    SPNS_FOR_EACH_L(X)
#undef X
    return -1;
}

// Kernel a z pass with these arguments runs (ZK_*; the staged forms report
// ZK_STAGED): falls back to ZK_BLOCK where the staged kernels' LDS does not fit.
template <typename T, int L>
static int zpass_kernel_L(const ZArgs& a)
{
    switch (zpass_pick<T, L, 0>(a)) {
    case ZV_WAVE: return ZK_WAVE;
    case ZV_BLOCK: return ZK_BLOCK;
    default: return ZK_STAGED;
    }
}

int zpass_kernel(int L, int prec, const ZArgs& a)
{
#define X(LL)                                                                                        \
    if (L == LL) return prec == PREC_FP64 ? zpass_kernel_L<double, LL>(a) : zpass_kernel_L<float, LL>(a);
    SPNS_FOR_EACH_L(X)
#undef X
    return -1;
}

hipError_t launch_zpass(int L, int prec, int mode, const ZArgs& a, int grid, hipStream_t st, const BatchLaunch* bl)
{
#define X(LL)                                                                                  \
    if (L == LL) {                                                                             \
        if (prec == PREC_FP64)                                                                 \
            return mode == 0   ? launch_zpass_L<double, LL, 0>(a, grid, st, bl)                \
                   : mode == 1 ? launch_zpass_L<double, LL, 1>(a, grid, st, bl)                \
                               : launch_zpass_L<double, LL, 2>(a, grid, st, bl);               \
        return mode == 0   ? launch_zpass_L<float, LL, 0>(a, grid, st, bl)                     \
               : mode == 1 ? launch_zpass_L<float, LL, 1>(a, grid, st, bl)                     \
                           : launch_zpass_L<float, LL, 2>(a, grid, st, bl);                    \
    }
    SPNS_FOR_EACH_L(X)
#undef X
    return hipErrorInvalidValue;
}

#endif

#if SPNS_PART == 0 || SPNS_PART == 5
// Persistent grid of a kernel: as many blocks as fit the device, at most items,
// rounded up to the 8 XCDs; -1 on an error.
template <class Kern>
static int resident_grid(Kern kern, int nt, int64_t items)
{
    int nb = 0, dev = 0, ncu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, nt, 0) != hipSuccess || nb < 1) nb = 1;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return -1;
    int64_t g = (int64_t)ncu * nb;
    if (items < g) g = items;
    return (int)((g + 7) / 8 * 8);
}

// The launches' grids, which ask the runtime for the device and the occupancy:
// host time that a plan pays once (spns_fft keeps them).
template <typename T, int L, int DIR>
static int zline_grid_L(int64_t np)
{
    constexpr int NB = zline_nb<T, L>(), NT = sstage_nt<L, NB>();
    if (np >= ((int64_t)1 << 30)) return -1;  // 32-bit pencil index
    return resident_grid(k_zline<T, L, NB, NT, DIR>, NT, ((np + 1) / 2 + NB - 1) / NB);
}

template <typename T, int L, int DIR>
static int line_grid_L(int64_t A, int64_t B)
{
    constexpr int TB = line_tb<T, L>(), NT = sstage_nt<L, TB>();
    return resident_grid(k_line<T, L, TB, NT, DIR>, NT, A * ((B + TB - 1) / TB));
}

template <typename T, int L, int DIR>
static hipError_t launch_zline_L(const ZPlainArgs& a, int grid, hipStream_t st)
{
    constexpr int NB = zline_nb<T, L>(), NT = sstage_nt<L, NB>();
    if (grid < 1 || (int64_t)a.Mx * a.My >= ((int64_t)1 << 30)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_zline<T, L, NB, NT, DIR>), dim3(grid), dim3(NT), 0, st, a);
    return hipGetLastError();
}

template <typename T, int L, int DIR>
static hipError_t launch_line_L(const StridedArgs& a, int grid, hipStream_t st)
{
    constexpr int TB = line_tb<T, L>(), NT = sstage_nt<L, TB>();
    static_assert(sizeof(cx<T>) * ((size_t)L * TB + L) <= 160 * 1024 - 512, "tile and table fit the LDS");
    if (a.njobs != 1 || a.nin != L || a.nout != L || a.job[0].out2 || a.job[0].deriv || a.job[0].in != a.job[0].out) return hipErrorInvalidValue;
    if (grid < 8 || grid % 8) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_line<T, L, TB, NT, DIR>), dim3(grid), dim3(NT), 0, st, a);
    return hipGetLastError();
}

#define X(LL)                                                                                              \
    case LL:                                                                                               \
        if (prec == PREC_FP64) return dir > 0 ? zline_grid_L<double, LL, +1>(np) : zline_grid_L<double, LL, -1>(np); \
        return dir > 0 ? zline_grid_L<float, LL, +1>(np) : zline_grid_L<float, LL, -1>(np);
int zline_grid(int L, int prec, int dir, int64_t np)
{
    switch (L) { SPNS_FOR_EACH_L(X) }
    return -1;
}
#undef X
#define X(LL)                                                                                              \
    case LL:                                                                                               \
        if (prec == PREC_FP64) return dir > 0 ? line_grid_L<double, LL, +1>(A, B) : line_grid_L<double, LL, -1>(A, B); \
        return dir > 0 ? line_grid_L<float, LL, +1>(A, B) : line_grid_L<float, LL, -1>(A, B);
int line_grid(int L, int prec, int dir, int64_t A, int64_t B)
{
    switch (L) { SPNS_FOR_EACH_L(X) }
    return -1;
}
#undef X
#define X(LL)                                                                                              \
    case LL:                                                                                               \
        if (prec == PREC_FP64) return dir > 0 ? launch_zline_L<double, LL, +1>(a, grid, st) : launch_zline_L<double, LL, -1>(a, grid, st); \
        return dir > 0 ? launch_zline_L<float, LL, +1>(a, grid, st) : launch_zline_L<float, LL, -1>(a, grid, st);
hipError_t launch_zplain(int L, int prec, int dir, const ZPlainArgs& a, int grid, hipStream_t st)
{
    switch (L) { SPNS_FOR_EACH_L(X) }
    return hipErrorInvalidValue;
}
#undef X
#define X(LL)                                                                                              \
    case LL:                                                                                               \
        if (prec == PREC_FP64) return dir > 0 ? launch_line_L<double, LL, +1>(a, grid, st) : launch_line_L<double, LL, -1>(a, grid, st); \
        return dir > 0 ? launch_line_L<float, LL, +1>(a, grid, st) : launch_line_L<float, LL, -1>(a, grid, st);
hipError_t launch_line(int L, int prec, int dir, const StridedArgs& a, int grid, hipStream_t st)
{
    switch (L) { SPNS_FOR_EACH_L(X) }
    return hipErrorInvalidValue;
}
#undef X

#endif

#if SPNS_PART == 0 || SPNS_PART == 4

// ---------------------------------------------------------------------------
// Shell spectra of the five velocity-gradient invariants (src/HIT_LES.cpp:
// 1297-1319 with the integrands |I_k|^2 of :1006-1025 and the shell sums of
// Integrate_Field :1137-1214): one wave per block walks (i2, i1) rows of the
// compact box, lanes along i3; per-block LDS histograms [5][nbins] (fixed
// order within the wave), then a fixed-order sum over the blocks.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(64) void k_inv_spectra(InvSpecArgs a)
{
    // One wave per block, rows (k1, k2) grid-strided.  Along a row the shell
    // K = round(|k|) never decreases with k3, so each 64-mode chunk splits
    // into runs of equal K: the first lane of a run sums it in order and adds
    // it to the block's bins.  Runs of one chunk hit distinct bins and the
    // chunks follow in program order, so the sums are deterministic (no
    // atomics); k_inv_sum adds the block partials in block order.
    extern __shared__ double hs[];  // [5][nbins] bins, [5][64] values, [64] shells
    const int nb = a.nbins, lane = threadIdx.x;
    double* vals = hs + 5 * nb;
    int* kb = (int*)(vals + 5 * 64);
    for (int i = lane; i < 5 * nb; i += 64) hs[i] = 0.0;
    __syncthreads();
    const int nrow = a.nk1 * a.nk2;
    for (int row = blockIdx.x; row < nrow; row += gridDim.x) {
        const int i2 = row / a.nk1, i1 = row - i2 * a.nk1;
        const int k1 = wrap_k(i1, a.nk1), k2 = wrap_k(i2, a.nk2);
        for (int base = 0; base < a.nk3; base += 64) {
            const int i3 = base + lane;
            int K = -1;
            if (i3 < a.nk3) {
                const int k3 = i3;
                K = shell_of(k1 * k1 + k2 * k2 + k3 * k3);
                const bool skip = a.notcubic && ((k1 % a.Lx) || (k2 % a.Ly) || (k3 % a.Lz));  // src/HIT_LES.cpp:867-871
                const bool conj = (k3 != 0) && !((a.Mz % 2 == 0) && (k3 == a.Mz / 2));       // src/HIT_LES.cpp:880
                const double w = skip ? 0.0 : (conj ? 2.0 : 1.0) * a.inv_nf2;
                const int64_t m = (int64_t)row * a.nk3p + i3;
#pragma unroll
                for (int f = 0; f < 5; f++) {
                    const cx<T> c = ((const cx<T>*)a.f[f])[m];
                    vals[f * 64 + lane] = w * ((double)c.x * (double)c.x + (double)c.y * (double)c.y);
                }
            }
            kb[lane] = K;
            __syncthreads();
            if (K >= 0 && (lane == 0 || kb[lane - 1] != K)) {
                int e = lane + 1;
                while (e < 64 && kb[e] == K) e++;
#pragma unroll
                for (int f = 0; f < 5; f++) {
                    double sum = 0.0;
                    for (int j = lane; j < e; j++) sum += vals[f * 64 + j];
                    hs[f * nb + K] += sum;
                }
            }
            __syncthreads();
        }
    }
    for (int i = lane; i < 5 * nb; i += 64) a.partial[(int64_t)blockIdx.x * 5 * nb + i] = hs[i];
}

static __global__ void k_inv_sum(const double* partial, int nblk, int n, double* out)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        double s = 0.0;
        for (int b = 0; b < nblk; b++) s += partial[(int64_t)b * n + i];
        out[i] = s;
    }
}

hipError_t launch_inv_spectra(int prec, const InvSpecArgs& a, int grid, double* out, hipStream_t st)
{
    const size_t shm = sizeof(double) * (5 * (size_t)a.nbins + 5 * 64) + sizeof(int) * 64;
    if (prec == PREC_FP64) hipLaunchKernelGGL((k_inv_spectra<double>), dim3(grid), dim3(64), shm, st, a);
    else hipLaunchKernelGGL((k_inv_spectra<float>), dim3(grid), dim3(64), shm, st, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int n = 5 * a.nbins;
    hipLaunchKernelGGL(k_inv_sum, dim3((n + 255) / 256), dim3(256), 0, st, a.partial, grid, n, out);
    return hipGetLastError();
}

// Fused forward y pass + step epilogue (DNS): grid for A x tiles items with
// nbins shell bins, or 0 where the kernel does not apply (staging or LDS
// does not fit, or more retained rows than the 3/2 padding leaves).
// Block size of k_yepi: that of the staged strided pass, except
//   * for the longest transforms, where half of it leaves LDS for the
//     per-wave shell histograms;
//   * where that block has 1024 threads (L = 192 and 384 with 16-column
//     tiles): 16 waves leave 128 VGPRs a thread, and the fused kernel
//     spills there; 8 waves leave 256.
// The transforms then take up to two butterflies per thread.
template <int L, int TB>
__host__ __device__ constexpr int yepi_nt()
{
    return (L > 1152 || sstage_nt<L, TB>() >= 1024) ? sstage_nt<L, TB>() / 2 : sstage_nt<L, TB>();
}

// LDS check and occupancy of k_yepi (INV false) or k_yepi_inv (true)
template <typename T, int L, int TB, int NT, bool INV, class K>
static int yepi_blocks_per_cu(K kern, int nbins, int max_spill)
{
    const size_t shm = sizeof(double) * (NT / 64) * (size_t)nbins;
    const size_t lds = sizeof(cx<T>) * ((size_t)L * TB + yepi_stg_elems<T, L, TB, INV>() +
                                        fft_twiddle_span<L, sizeof(T) == 8 ? 1 : 2>());
    if (lds + shm > 160 * 1024 - 512) return 0;
    hipFuncAttributes fa;
    if (hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(kern)) != hipSuccess || (int)fa.localSizeBytes > max_spill) return 0;
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, NT, shm) != hipSuccess || n < 1) return 0;
    return n;
}

template <typename T, int L>
static int yepi_grid_L(int nbins, int nout, int A, int B, int max_grid, bool inv, bool les)
{
    if (les ? YComb<T, L, true>::use : YComb<T, L, false>::use)
        return ycomb_grid(L, sizeof(T) == 8 ? PREC_FP64 : PREC_FP32, les, nbins, nout, A, B, max_grid);
    if (les) return 0;
    constexpr int TB = strided_tb<T, L>();
    if constexpr (YComb<T, L, false>::use || TB <= 0 || (TB * sizeof(cx<T>)) % 16 != 0) {
        return 0;
    } else {
        if (nout > 2 * (L / 3) + 1) return 0;
        const int64_t items = (int64_t)A * ((B + TB - 1) / TB);
        constexpr int NT = yepi_nt<L, TB>();
        // a variant that spills registers (the 1024-thread tiles) is slower
        // than the two separate kernels; k_yepi_inv may keep a few
        // loop-invariant values in scratch (FP32 at L = 768: 20 bytes, three
        // reloads per item outside the transforms)
        const int n = inv ? yepi_blocks_per_cu<T, L, TB, NT, true>(k_yepi_inv<T, L, TB, NT>, nbins, 32)
                          : yepi_blocks_per_cu<T, L, TB, NT, false>(k_yepi<T, L, TB, NT>, nbins, 0);
        if (n < 1) return 0;
        int dev = 0, ncu = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        int64_t g = (int64_t)ncu * n;
        if (items < g) g = items;
        g = (g + 7) / 8 * 8;
        if (g > max_grid) g = max_grid / 8 * 8;
        return (int)g;
    }
}

int yepi_grid(int L, int prec, int nbins, int nout, int A, int B, int max_grid, bool inv, bool les)
{
#define X(LL)                                                                                   \
    if (L == LL)                                                                                \
        return prec == PREC_FP64 ? yepi_grid_L<double, LL>(nbins, nout, A, B, max_grid, inv, les) \
                                 : yepi_grid_L<float, LL>(nbins, nout, A, B, max_grid, inv, les);
    SPNS_FOR_EACH_L(X)
#undef X
    return 0;
}

template <typename T, int L>
static hipError_t launch_yepi_L(const StridedArgs& a, int A, const EpiArgs& e, int grid, hipStream_t st, const BatchLaunch* bl,
                                const StridedArgs* ia, int* x1v)
{
    constexpr int TB = strided_tb<T, L>();
    if constexpr (TB <= 0 || (TB * sizeof(cx<T>)) % 16 != 0) {
        return hipErrorNotSupported;
    } else {
        StridedArgs b = a;
        b.A = A;
        if (!a.padded_ok || a.nin != L || a.njobs != (e.les ? 9 : 3) || a.nout > 2 * (L / 3) + 1 || grid < 8 || grid % 8)
            return hipErrorInvalidValue;
        if (e.les ? YComb<T, L, true>::use : YComb<T, L, false>::use) {
            StridedArgs ib{};
            if (ia) {
                // the inverse pass's items must be the forward pass's
                bool ok = (bl ? bl->args3 && ia->setflag : x1v != nullptr) && ia->padded_ok && ia->njobs == 3 && ia->nout == L &&
                          ia->nin == a.nout && ia->B == a.B;
                for (int j = 0; ok && j < 3; j++) ok = ia->job[j].in && ia->job[j].out && ia->job[j].out2;
                if (!ok) return hipErrorInvalidValue;
                ib = *ia;
                ib.A = A;
            }
            return launch_ycomb(L, sizeof(T) == 8 ? PREC_FP64 : PREC_FP32, b, e, grid, st, bl, ia ? &ib : nullptr, x1v);
        }
        if (e.les) return hipErrorNotSupported;
        if constexpr (!YComb<T, L, false>::use) {
            if (bl) {
                constexpr int NT = yepi_nt<L, TB>();
                const size_t shm = sizeof(double) * (NT / 64) * (size_t)e.nbins;
                if constexpr (batch_length(L)) {
                    if (ia) {
                        // with the next step's inverse y pass: ia is a slot's struct (all
                        // slots share the shape class), the slots' structs are in args3
                        bool ok = bl->args3 && ia->setflag && ia->padded_ok && ia->njobs == 3 && ia->nout == L && ia->nin == a.nout &&
                                  ia->B == a.B;
                        for (int j = 0; ok && j < 3; j++) ok = ia->job[j].in && ia->job[j].out && ia->job[j].out2;
                        if (!ok) return hipErrorInvalidValue;
                        hipLaunchKernelGGL((k_yepi_inv_b<T, L, TB, NT>), dim3(grid, bl->nslots), dim3(NT), shm, st,
                                           (const StridedArgs*)bl->args, (const EpiArgs*)bl->args2, (const StridedArgs*)bl->args3, bl->left);
                        return hipGetLastError();
                    }
                    hipLaunchKernelGGL((k_yepi_b<T, L, TB, NT>), dim3(grid, bl->nslots), dim3(NT), shm, st, (const StridedArgs*)bl->args,
                                       (const EpiArgs*)bl->args2, bl->left);
                    return hipGetLastError();
                }
                return hipErrorNotSupported;
            }
            if (ia) {
                // the inverse pass's items must be the forward pass's: same
                // outer extent and column tiles, all rows of the transform out
                bool ok = x1v && ia->padded_ok && ia->njobs == 3 && ia->nout == L && ia->nin == a.nout && ia->B == a.B;
                for (int j = 0; ok && j < 3; j++) ok = ia->job[j].in && ia->job[j].out && ia->job[j].out2;
                if (!ok) return hipErrorInvalidValue;
                StridedArgs ib = *ia;
                ib.A = A;
                constexpr int NT = yepi_nt<L, TB>();
                const size_t shm = sizeof(double) * (NT / 64) * (size_t)e.nbins;
                hipLaunchKernelGGL((k_yepi_inv<T, L, TB, NT>), dim3(grid), dim3(NT), shm, st, b, e, ib, x1v);
                return hipGetLastError();
            }
            constexpr int NT = yepi_nt<L, TB>();
            const size_t shm = sizeof(double) * (NT / 64) * (size_t)e.nbins;
            hipLaunchKernelGGL((k_yepi<T, L, TB, NT>), dim3(grid), dim3(NT), shm, st, b, e);
            return hipGetLastError();
        }
        return hipErrorNotSupported;
    }
}

hipError_t launch_yepi(int L, int prec, const StridedArgs& a, int A, const EpiArgs& e, int grid, hipStream_t st, const BatchLaunch* bl,
                       const StridedArgs* ia, int* x1v)
{
#define X(LL)                                                                                        \
    if (L == LL)                                                                                     \
        return prec == PREC_FP64 ? launch_yepi_L<double, LL>(a, A, e, grid, st, bl, ia, x1v) \
                                 : launch_yepi_L<float, LL>(a, A, e, grid, st, bl, ia, x1v);
    SPNS_FOR_EACH_L(X)
#undef X
    return hipErrorInvalidValue;
}

// Sets an int flag in device memory (stream-ordered, no memset node).
static __global__ void k_set_int(int* p, int v)
{
    *p = v;
}

hipError_t launch_set_int(int* p, int v, hipStream_t st)
{
    hipLaunchKernelGGL(k_set_int, dim3(1), dim3(1), 0, st, p, v);
    return hipGetLastError();
}

hipError_t launch_epilogue(int prec, const EpiArgs& a, int grid, hipStream_t st, const BatchLaunch* bl)
{
    constexpr int NT = 256;
    const size_t shm = sizeof(double) * (NT / 64) * a.nbins;
    if (bl) {
        const EpiArgs* arr = (const EpiArgs*)bl->args;
        if (prec == PREC_FP64) hipLaunchKernelGGL((k_epilogue_b<double, NT>), dim3(grid, bl->nslots), dim3(NT), shm, st, arr, bl->left);
        else hipLaunchKernelGGL((k_epilogue_b<float, NT>), dim3(grid, bl->nslots), dim3(NT), shm, st, arr, bl->left);
        return hipGetLastError();
    }
    if (prec == PREC_FP64) hipLaunchKernelGGL((k_epilogue<double, NT>), dim3(grid), dim3(NT), shm, st, a);
    else hipLaunchKernelGGL((k_epilogue<float, NT>), dim3(grid), dim3(NT), shm, st, a);
    return hipGetLastError();
}

hipError_t launch_finalize(const FinArgs& a, hipStream_t st, const BatchLaunch* bl)
{
    const unsigned g = (a.flags & FIN_REDUCE) ? (unsigned)((a.nbins + 63) / 64) : 1u;
    if (bl) {
        hipLaunchKernelGGL((k_finalize_b<1024>), dim3(g, bl->nslots), dim3(1024), 0, st, (const FinArgs*)bl->args, bl->left);
        return hipGetLastError();
    }
    hipLaunchKernelGGL((k_finalize<1024>), dim3(g), dim3(1024), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_stream_copy(const void* in, void* out, int64_t bytes, int blocks, hipStream_t st)
{
    if (bytes % 16 || blocks < 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_stream_copy<4>), dim3(blocks), dim3(256), 0, st, (const vf4*)in, (vf4*)out, bytes / 16);
    return hipGetLastError();
}

// grid of the pack kernels: 0 if the elements exceed the box or a field their 32-bit index
static unsigned pack_grid(const PackArgs& a)
{
    const int64_t per = (int64_t)a.nrow * a.nk3;
    if (per >= ((int64_t)1 << 31) || a.n < 1 || a.n >= (1u << 31) || a.first < 0 || a.first + a.n > 3 * per) return 0;
    const uint32_t g = (a.n + 255) / 256;
    return g < 8192 ? g : 8192;
}

hipError_t launch_pack(const PackArgs& a, bool from_fp32, hipStream_t st)
{
    const unsigned g = pack_grid(a);
    if (!g) return hipErrorInvalidValue;
    if (from_fp32) hipLaunchKernelGGL((k_pack<float>), dim3(g), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_pack<double>), dim3(g), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_unpack(const PackArgs& a, hipStream_t st)
{
    const unsigned g = pack_grid(a);
    if (!g) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_unpack, dim3(g), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_set_left(int* left, const SlotSteps& s, int nslots, hipStream_t st)
{
    if (nslots < 1 || nslots > kMaxBatchSlots) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_set_left, dim3(1), dim3(kMaxBatchSlots), 0, st, left, s, nslots);
    return hipGetLastError();
}

hipError_t launch_forcing(const double* ek, const double* forced, double* ft, int last_eff, const ShellArgs& a, hipStream_t st)
{
    hipLaunchKernelGGL(k_forcing_ft, dim3(1), dim3(256), 0, st, ek, forced, ft, last_eff);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    int grid = (int)((a.nmodes + 255) / 256);
    if (grid > 4096) grid = 4096;
    if (grid < 1) grid = 1;
    hipLaunchKernelGGL(k_scale_shells, dim3(grid), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_ccc(const ShellArgs& a, hipStream_t st)
{
    int n = a.nk1 * a.nk2;
    int grid = (n + 255) / 256;
    hipLaunchKernelGGL(k_ccc, dim3(grid), dim3(256), 0, st, a);
    return hipGetLastError();
}


// ---------------------------------------------------------------------------
// Synthetic initial field: random-phase, solenoidal, E(k) ~ k^4 exp(-2(k/k0)^2)
// (unscaled).  Counter-based: each mode's value depends only on
// (seed, k1, k2, k3), so the field is the same for any launch shape.  The
// k3 = 0 plane is made Hermitian by taking the mirror of the canonical half.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t splitmix(uint64_t x)
{
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}
__device__ __forceinline__ double unif(uint64_t seed, int k1, int k2, int k3, int d)
{
    uint64_t key = splitmix(seed) ^ splitmix(((uint64_t)(uint32_t)(k1 + 65536) << 40) ^
                                             ((uint64_t)(uint32_t)(k2 + 65536) << 20) ^ (uint64_t)(uint32_t)k3 ^
                                             ((uint64_t)d << 58));
    return ((double)(splitmix(key) >> 11) + 0.5) * (1.0 / 9007199254740992.0);
}

static __global__ void k_init_random(RandArgs a)
{
    const int nk1 = a.nk1, nk2 = a.nk2, nk3 = a.nk3, nk3p = a.nk3p;
    const double PI = 3.141592653589793238462643;
    for (int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; m < a.nmodes; m += (int64_t)gridDim.x * blockDim.x) {
        const int i3 = (int)(m % nk3p);
        if (i3 >= nk3) continue;  // pitch padding
        const int64_t r12 = m / nk3p;
        const int i1 = (int)(r12 % nk1), i2 = (int)(r12 / nk1);
        int k1 = wrap_k(i1, nk1), k2 = wrap_k(i2, nk2);
        const int k3 = i3;
        bool masked = a.notcubic && ((k1 % a.Lx) || (k2 % a.Ly) || (k3 % a.Lz));
        const bool canon = k3 > 0 || k1 > 0 || (k1 == 0 && k2 > 0);
        const bool mirror = (k3 == 0) && !canon && !(k1 == 0 && k2 == 0);
        cx<double> out[3] = {{0.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}};
        if (!masked && (canon || mirror)) {
            if (mirror) { k1 = -k1; k2 = -k2; }
            const double K1 = k1, K2 = k2, K3 = k3;
            const double r2 = K1 * K1 + K2 * K2 + K3 * K3;
            double gr[3], gi[3];
            for (int c = 0; c < 3; c++) {
                const double u1 = unif(a.seed, k1, k2, k3, 2 * c), u2 = unif(a.seed, k1, k2, k3, 2 * c + 1);
                const double rr = sqrt(-2.0 * log(u1));
                gr[c] = rr * cos(2 * PI * u2);
                gi[c] = rr * sin(2 * PI * u2);
            }
            const double dr = (K1 * gr[0] + K2 * gr[1] + K3 * gr[2]) / r2;
            const double di = (K1 * gi[0] + K2 * gi[1] + K3 * gi[2]) / r2;
            const double kk[3] = {K1, K2, K3};
            double nrm = 0.0;
            for (int c = 0; c < 3; c++) {
                gr[c] -= dr * kk[c];
                gi[c] -= di * kk[c];
                nrm += gr[c] * gr[c] + gi[c] * gi[c];
            }
            if (nrm > 0.0) {
                const double km = sqrt(r2);
                const double Ek = km * km * km * km * exp(-2.0 * (km / a.k0) * (km / a.k0));
                const double amp = sqrt(Ek / (4.0 * PI * r2) / nrm);
                for (int c = 0; c < 3; c++) out[c] = cx<double>{gr[c] * amp, (mirror ? -1.0 : 1.0) * gi[c] * amp};
            }
        }
        for (int c = 0; c < 3; c++) a.uk[c][m] = out[c];
    }
}

static __global__ void k_scale_state(ShellArgs a, double sc)
{
    for (int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; m < a.nmodes; m += (int64_t)gridDim.x * blockDim.x)
        for (int c = 0; c < 3; c++) {
            cx<double> v = a.uk[c][m];
            a.uk[c][m] = cx<double>{v.x * sc, v.y * sc};
        }
}

hipError_t launch_init_random(const RandArgs& a, hipStream_t st)
{
    int grid = (int)((a.nmodes + 255) / 256);
    if (grid > 16384) grid = 16384;
    hipLaunchKernelGGL(k_init_random, dim3(grid), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_scale_state(const ShellArgs& a, double sc, hipStream_t st)
{
    int grid = (int)((a.nmodes + 255) / 256);
    if (grid > 16384) grid = 16384;
    hipLaunchKernelGGL(k_scale_state, dim3(grid), dim3(256), 0, st, a, sc);
    return hipGetLastError();
}

hipError_t launch_normalize(int prec, const NormArgs& a, hipStream_t st)
{
    const int64_t n = (int64_t)a.My * a.Mx * (a.Mz / 2 + 1);
    int grid = (int)((n + 255) / 256);
    if (grid > 8192) grid = 8192;
    if (prec == PREC_FP64) hipLaunchKernelGGL((k_normalize<double>), dim3(grid), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((k_normalize<float>), dim3(grid), dim3(256), 0, st, a);
    return hipGetLastError();
}

#endif
}  // namespace spns
