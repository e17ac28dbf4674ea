// kernels_march.h -- the temporally blocked steps: several plain steps of a
// lattice in one launch, bit-identical to single steps (they run the node
// functions of kernels_impl.h).
#pragma once
#include "kernels_impl.h"

namespace tclbx {

// ------------------------------------------------------ 2D: marching waves ---
// The stored form of population i, rounded as the single step rounds its
// store; with stochastic rounding direction 2j takes word j of the node's
// stream and 2j + 1 word j << 16 (w advances after each odd direction).
template <class S, class L, bool DEV>
__device__ __forceinline__ typename S::T tb_stored(typename S::R v, int i, uint32_t& w) {
    using R = typename S::R;
    if constexpr (S::stochastic) {
        const uint32_t r = (i & 1) ? w << 16 : w;
        const typename S::T out = DEV ? S::unraw_sr(v, r) : S::put_sr(v, (R)L::w(i), r);
        if (i & 1) w = xorshift32(w);
        return out;
    } else {
        return DEV ? S::unraw(v) : S::put(v, (R)L::w(i));
    }
}

// Stores past the L2 (NT) where one round of blocks is the whole launch: the
// launch then does not end with the L2's write-back (1024x128 in FP64, a launch
// of 4 steps: 3.39 us per step against 3.58); plain stores where there is more
// to overlap it with, whose partial lines at a tile's edge the L2 joins
// (4096x2048 on tiles, 4 steps: 128 us against 152), and in batches.
template <bool NT, class T> __device__ __forceinline__ void tb_store(T v, gptr<T> p) {
    if constexpr (NT) __builtin_nontemporal_store(v, p);
    else *p = v;
}

// the value of the lane one to the left (x - 1) or to the right (x + 1) of
// this one, by a data-parallel-primitive move over the wavefront; the first
// (last) lane gets 0
template <int CTRL> __device__ __forceinline__ int dpp_mov(int v) {
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}
template <int CTRL> __device__ __forceinline__ float dpp_mov(float v) {
    return __builtin_bit_cast(float, dpp_mov<CTRL>(__builtin_bit_cast(int, v)));
}
template <int CTRL> __device__ __forceinline__ double dpp_mov(double v) {
    typedef int int2v __attribute__((ext_vector_type(2)));
    int2v b = __builtin_bit_cast(int2v, v);
    b[0] = dpp_mov<CTRL>(b[0]);
    b[1] = dpp_mov<CTRL>(b[1]);
    return __builtin_bit_cast(double, b);
}
constexpr int DPP_WAVE_SHL1 = 0x130, DPP_WAVE_SHR1 = 0x138;
template <class R> __device__ __forceinline__ R from_left(R v) { return dpp_mov<DPP_WAVE_SHR1>(v); }
template <class R> __device__ __forceinline__ R from_right(R v) { return dpp_mov<DPP_WAVE_SHL1>(v); }

// The columns of a node's zone row that the node reads, in registers, loaded
// only where they are needed and waited for there: a load left in flight
// past the branch would make every wave wait, which would also drain the
// next row's loads.
struct ZoneCols {
    double c[5];
    __device__ __forceinline__ double operator[](int i) const { return c[i]; }
};

// one node of the march: Run() on the pulled populations f
template <int MODEL, int ST>
__device__ __forceinline__ void march_node2d(const StepArgs& a, typename Store<ST>::R* f, unsigned nt, double gx0,
                                             double gy0) {
    using L = Lat<MODEL>;
    using S = Store<ST>;
    using R = typename S::R;
    constexpr bool DEV = S::shifted;
    int zone = (int)(nt >> L::ZSHIFT);
    if (zone >= a.nzones) zone = 0;
    const double* zr = a.zone + (size_t)zone * a.zcols;
    double* g = nullptr;
    ZoneCols z{};
    if constexpr (is_d2q9m<MODEL>) {
        // VelocityX, VelocityY, Pressure of the Zou-He nodes
        if ((nt & 0xFu) != 0) {
            z.c[0] = zr[0]; z.c[1] = zr[1]; z.c[2] = zr[2];
            asm volatile("" : "+v"(z.c[0]), "+v"(z.c[1]), "+v"(z.c[2]));
        }
        if constexpr (DEV) d2q9m_node_dev<false, MODEL == MODEL_D2Q9_DRAG, false>(f, nt, a.par, z, g, nullptr, 0);
        else d2q9m_node<R, false, MODEL == MODEL_D2Q9_DRAG, false>(f, nt, a.par, z, g, nullptr, 0);
    } else {
        // Velocity_x of the Zou-He nodes; the gravitation, of zone 0 for
        // nearly every node
        z.c[3] = gx0; z.c[4] = gy0;
        if (zone != 0 || (nt & 0x7u) != 0) {
            z.c[1] = zr[1]; z.c[3] = zr[3]; z.c[4] = zr[4];
            asm volatile("" : "+v"(z.c[1]), "+v"(z.c[3]), "+v"(z.c[4]));
        }
        if constexpr (DEV) d2q9_node_dev<MODEL == MODEL_D2Q9_SRT_DRAG, false>(f, nt, (R)a.par[0], (R)a.par[1], z, g);
        else d2q9_node<R, MODEL == MODEL_D2Q9_SRT_DRAG, false>(f, nt, (R)a.par[0], (R)a.par[1], z, g);
    }
}

// K plain steps of the nodes of one wave's strip.  The strip is 64 columns
// wide, lane = column, of which the middle 64 - 2(K-1) are written; the wave
// marches along y over the rows y0 - (K-1) .. y0 + rows - 1 + (K-1).  Each
// iteration takes one row through the K steps: step 1 of the row pulls from
// the current snapshot; step s of the row s - 1 behind it pulls what step
// s - 1 left in this wave's registers: its e_y = -1 populations of the row
// just computed, its e_y = 0 ones of the row before and its e_y = +1 ones of
// the row before that, so 9 values per step stay in registers from one
// iteration to the next.  Neighbours in x are the neighbouring lanes, read by
// DPP moves; no value passes through LDS or waits at a barrier.  After step s
// the columns at least s - 1 from the strip's edge hold exact values, and the
// row of step s is first exact in iteration 2(s - 1).
template <int MODEL, int ST, int K>
__device__ __forceinline__ void march2d(const StepArgs& a, int strip, int y0, int rows) {
    using L = Lat<MODEL>;
    using S = Store<ST>;
    using T = typename S::T;
    using R = typename S::R;
    constexpr int Q = 9, W = 64 - 2 * (K - 1);
    constexpr bool DEV = S::shifted;
    const int lane = threadIdx.x & 63;
    const int nx = a.nx, ny = a.ny;
    const int ux = strip * W - (K - 1) + lane;
    int x = ux % nx;
    if (x < 0) x += nx;
    const int xm = x == 0 ? nx - 1 : x - 1, xp = x == nx - 1 ? 0 : x + 1;
    const bool writes = lane >= K - 1 && lane < 64 - (K - 1) && ux < nx;
    const size_t pbytes = (size_t)a.pitch * sizeof(T);
    const char* fin = (const char*)a.fin;
    char* fout = (char*)a.fout;
    double gx0 = 0, gy0 = 0;
    if constexpr (!is_d2q9m<MODEL>) { gx0 = a.zone[3]; gy0 = a.zone[4]; }

    // the row step 1 reads this iteration and its neighbours, wrapped
    int y = (y0 - (K - 1)) % ny;
    if (y < 0) y += ny;
    int yrow[K];            // rows (wrapped) of the steps 1..K
    unsigned ntp[K];        // their NodeTypes
    R Z[K][3], P1[K][3], P2[K][3];   // inputs of step s + 1 from step s
#pragma unroll
    for (int s = 0; s < K; s++) {
        yrow[s] = 0; ntp[s] = 0;
#pragma unroll
        for (int j = 0; j < 3; j++) Z[s][j] = P1[s][j] = P2[s][j] = R(0);
    }
    T v[Q];
    unsigned nt_next;
    auto fetch = [&](int yy) {
        const int ym = yy == 0 ? ny - 1 : yy - 1, yp = yy == ny - 1 ? 0 : yy + 1;
        nt_next = *(gptr<const uint16_t>)(a.flags + ((unsigned)x + (unsigned)nx * (unsigned)yy));
#pragma unroll
        for (int i = 0; i < Q; i++) {
            const int sx = L::ex(i) > 0 ? xm : (L::ex(i) < 0 ? xp : x);
            const int sy = L::ey(i) > 0 ? ym : (L::ey(i) < 0 ? yp : yy);
            const unsigned src = (unsigned)sx + (unsigned)nx * (unsigned)sy;
            v[i] = *(gptr<const T>)(fin + (size_t)i * pbytes + src * (unsigned)sizeof(T));
        }
    };
    fetch(y);
    const int iters = rows + 2 * (K - 1);
    for (int it = 0; it < iters; it++) {
        R f[Q];
#pragma unroll
        for (int i = 0; i < Q; i++) f[i] = DEV ? S::raw(v[i]) : S::get(v[i], (R)L::w(i));
#pragma unroll
        for (int s = K - 1; s > 0; s--) { yrow[s] = yrow[s - 1]; ntp[s] = ntp[s - 1]; }
        yrow[0] = y;
        ntp[0] = nt_next;
        y = y == ny - 1 ? 0 : y + 1;
        // the next row's loads run under this row's K steps
        if (it + 1 < iters) fetch(y);
#pragma unroll
        for (int s = 1; s <= K; s++) {
            if (it < 2 * (s - 1)) break;   // not yet a row with exact inputs
            march_node2d<MODEL, ST>(a, f, ntp[s - 1], gx0, gy0);
            const unsigned n = (unsigned)x + (unsigned)nx * (unsigned)yrow[s - 1];
            uint32_t w = 0;
            if constexpr (S::stochastic) w = sr_word0(n, sr_key(a.sr_step + (unsigned)(s - 1), a.sr_seed));
            if (s == K) {
                if (writes) {
#pragma unroll
                    for (int i = 0; i < Q; i++)
                        *(gptr<T>)(fout + (size_t)i * pbytes + n * (unsigned)sizeof(T)) = tb_stored<S, L, DEV>(f[i], i, w);
                }
            } else {
                R h[Q];
#pragma unroll
                for (int i = 0; i < Q; i++) {
                    const T t = tb_stored<S, L, DEV>(f[i], i, w);
                    h[i] = DEV ? S::raw(t) : S::get(t, (R)L::w(i));
                }
                // the pulls of the next step, one row behind
                f[0] = Z[s][0]; f[1] = Z[s][1]; f[3] = Z[s][2];
                f[2] = P2[s][0]; f[5] = P2[s][1]; f[6] = P2[s][2];
                f[4] = h[4]; f[7] = from_right(h[7]); f[8] = from_left(h[8]);
                Z[s][0] = h[0]; Z[s][1] = from_left(h[1]); Z[s][2] = from_right(h[3]);
#pragma unroll
                for (int j = 0; j < 3; j++) P2[s][j] = P1[s][j];
                P1[s][0] = h[2]; P1[s][1] = from_left(h[5]); P1[s][2] = from_right(h[6]);
            }
        }
    }
}

// strips of a lattice of nx columns at K steps per launch
__host__ __device__ constexpr int march2d_strips(int nx, int K) { return (nx + 64 - 2 * (K - 1) - 1) / (64 - 2 * (K - 1)); }

// One wave per work item: strip item % nstrips, rows [seg * a.tb_rows, + a.tb_rows)
// with seg = item / nstrips
template <int MODEL, int ST, int K>
__device__ __forceinline__ void march2d_item(const StepArgs& a, int item) {
    const int nstrips = march2d_strips(a.nx, K), seg = item / nstrips, y0 = seg * a.tb_rows;
    march2d<MODEL, ST, K>(a, item - seg * nstrips, y0, min(a.tb_rows, a.ny - y0));
}
template <int MODEL, int ST, int K>
__global__ void __launch_bounds__(256) k_march2d(StepArgs a, int items) {
    const int item = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (item < items) march2d_item<MODEL, ST, K>(a, item);
}

// ------------------------------------------------------- 2D: LDS tiles ---
// Up to K = a.tb_k plain steps of a lattice too small for enough marching
// waves.  A block steps the a.tb_tx x a.tb_ty tile whose middle (tb_tx -
// 2(K-1)) x (tb_ty - 2(K-1)) nodes it writes, one node per thread (the threads
// past the tile compute values nobody reads).  Step 1
// pulls from the current snapshot; every later step pulls from the LDS tile
// the step before filled, all pulls read before any node writes its own
// populations (a barrier between), so one LDS copy serves every step.  After
// step s the nodes at least s - 1 from the tile's edge hold exact values.
// LDS: plane i of the tile at i * blockDim.x; the pulls of edge nodes fall
// into the plane before or after (past the last plane: tb_tx + 1 values of
// padding), which only nodes not exact anyway read.
// The last step is written out behind the loop: inside it the addresses of
// its stores were held in 18 registers across the steps, which cost the f16s
// tile of d2q9 MRT its second block per CU.
template <int MODEL, int ST, bool NT>
__device__ __forceinline__ void tile2d(const StepArgs& a, int tile, int steps) {
    using L = Lat<MODEL>;
    using S = Store<ST>;
    using T = typename S::T;
    using R = typename S::R;
    constexpr int Q = 9;
    constexpr bool DEV = S::shifted;
    static_assert(tb_model<MODEL> && L::Q == 9, "2D models");
    extern __shared__ double tile2d_lds[];
    const int TX = a.tb_tx, TY = a.tb_ty;
    const int nx = a.nx, ny = a.ny;
    const int h = a.tb_k - 1, tiles_x = (nx + TX - 2 * h - 1) / (TX - 2 * h);
    const int by = tile / tiles_x, bx = tile - by * tiles_x;
    const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
    // this thread's tile node: unwrapped coordinates (ux, uy), lattice node (x, y)
    const int ux = bx * (TX - 2 * h) - h + tx, uy = by * (TY - 2 * h) - h + ty;
    int x = ux % nx, y = uy % ny;
    if (x < 0) x += nx;
    if (y < 0) y += ny;
    const unsigned n = (unsigned)x + (unsigned)nx * (unsigned)y;
    const unsigned nt = *(gptr<const uint16_t>)(a.flags + n);
    const size_t pbytes = (size_t)a.pitch * sizeof(T);
    T v[Q];
    {
        const int xm = x == 0 ? nx - 1 : x - 1, xp = x == nx - 1 ? 0 : x + 1;
        const int ym = y == 0 ? ny - 1 : y - 1, yp = y == ny - 1 ? 0 : y + 1;
        const char* fin = (const char*)a.fin;
#pragma unroll
        for (int i = 0; i < Q; i++) {
            const int sx = L::ex(i) > 0 ? xm : (L::ex(i) < 0 ? xp : x);
            const int sy = L::ey(i) > 0 ? ym : (L::ey(i) < 0 ? yp : y);
            const unsigned src = (unsigned)sx + (unsigned)nx * (unsigned)sy;
            v[i] = *(gptr<const T>)(fin + (size_t)i * pbytes + src * (unsigned)sizeof(T));
        }
    }
    double gx0 = 0, gy0 = 0;
    if constexpr (!is_d2q9m<MODEL>) { gx0 = a.zone[3]; gy0 = a.zone[4]; }
    const int plane = blockDim.x;
    T* const own = (T*)tile2d_lds + threadIdx.x;
    R f[Q];
    // one step on the pulled values v; returns the node's first random word:
    // stochastic rounding draws the words of this node at the iteration step
    // s computes, as the single step of that iteration does
    const auto step = [&](int s) -> uint32_t {
#pragma unroll
        for (int i = 0; i < Q; i++) f[i] = DEV ? S::raw(v[i]) : S::get(v[i], (R)L::w(i));
        march_node2d<MODEL, ST>(a, f, nt, gx0, gy0);
        if constexpr (S::stochastic) return sr_word0(n, sr_key(a.sr_step + (unsigned)(s - 1), a.sr_seed));
        return 0;
    };
    for (int s = 1; s < steps; s++) {
        uint32_t w = step(s);
#pragma unroll
        for (int i = 0; i < Q; i++) own[i * plane] = tb_stored<S, L, DEV>(f[i], i, w);
        __syncthreads();
        // (direction 0, the first plane, is not shifted: no pull falls before it)
#pragma unroll
        for (int i = 0; i < Q; i++) v[i] = own[i * plane - L::ex(i) - L::ey(i) * TX];
        __syncthreads();
    }
    uint32_t w = step(steps);
    // each lattice node is the middle node of exactly one tile
    if (tx >= h && tx < TX - h && ty >= h && ty < TY - h && ux < nx && uy < ny) {
        char* fout = (char*)a.fout;
#pragma unroll
        for (int i = 0; i < Q; i++)
            tb_store<NT>(tb_stored<S, L, DEV>(f[i], i, w), (gptr<T>)(fout + (size_t)i * pbytes + n * (unsigned)sizeof(T)));
    }
}

template <int MODEL, int ST, bool NT>
__global__ void __launch_bounds__(1024) k_tile2d(StepArgs a) {
    tile2d<MODEL, ST, NT>(a, blockIdx.x, a.tb_k);
}

// LDS of a block of `threads` threads whose tiles are at most tx wide
template <int ST> constexpr size_t tile2d_lds_bytes(int threads, int tx) {
    return ((size_t)9 * threads + tx + 1) * sizeof(typename Store<ST>::T);
}

template <int MODEL, int ST>
hipError_t tile2d_ms(const StepArgs& a, hipStream_t s) {
    const int threads = (a.tb_tx * a.tb_ty + 63) / 64 * 64, tiles = blocked2d_items(a);
    if (a.nz != 1 || a.tb_k < 2 || tiles < 1 || threads > 1024) return hipErrorInvalidValue;
    const size_t lds = tile2d_lds_bytes<ST>(threads, a.tb_tx);
    if (a.tb_nt) hipLaunchKernelGGL((k_tile2d<MODEL, ST, true>), dim3(tiles), dim3(threads), lds, s, a);
    else hipLaunchKernelGGL((k_tile2d<MODEL, ST, false>), dim3(tiles), dim3(threads), lds, s, a);
    return hipGetLastError();
}

template <int MODEL, int ST, int K>
hipError_t march2d_k(const StepArgs& a, hipStream_t s) {
    const int items = blocked2d_items(a);
    hipLaunchKernelGGL((k_march2d<MODEL, ST, K>), dim3((items + 3) / 4), dim3(256), 0, s, a, items);
    return hipGetLastError();
}

template <int MODEL, int ST>
hipError_t blocked2d_ms(const StepArgs& a, hipStream_t s) {
    if (a.tb_rows == 0) return tile2d_ms<MODEL, ST>(a, s);
    if (a.nz != 1 || a.tb_rows < 1) return hipErrorInvalidValue;
    static_assert(MARCH2D_MAX_K == 5, "one case per number of steps");
    switch (a.tb_k) {
    case 2: return march2d_k<MODEL, ST, 2>(a, s);
    case 3: return march2d_k<MODEL, ST, 3>(a, s);
    case 4: return march2d_k<MODEL, ST, 4>(a, s);
    case 5: return march2d_k<MODEL, ST, 5>(a, s);
    }
    return hipErrorInvalidValue;
}

// ------------------------------------------------------------- batches ---
// `steps` plain steps of every lattice of a batch in one launch: one item
// {case, tile or strip of the case} per block (LDS tiles) or wave (marching
// waves, steps = K).  The phase word as in k_batch_step; its step index is
// that of the first step.
template <int ST>
__device__ __forceinline__ StepArgs batch_case_args(const BatchCase* cases, int c, int phase) {
    StepArgs a = cases[c].args;
    if ((phase ^ cases[c].parity) & 1) {
        const void* tmp = a.fin;
        a.fin = a.fout;
        a.fout = (void*)tmp;
    }
    if constexpr (Store<ST>::stochastic) {
        a.sr_step = cases[c].sr_iter + ((unsigned)phase >> 2);
        a.sr_seed = cases[c].sr_seed;
    }
    return a;
}

template <int MODEL, int ST>
__global__ void __launch_bounds__(1024) k_batch_tile2d(const BatchCase* __restrict__ cases,
                                                       const int2* __restrict__ items, int phase, int steps) {
    const int2 it = items[blockIdx.x];
    const StepArgs a = batch_case_args<ST>(cases, it.x, phase);
    tile2d<MODEL, ST, false>(a, it.y, steps);
}

template <int MODEL, int ST, int K>
__global__ void __launch_bounds__(256) k_batch_march2d(const BatchCase* __restrict__ cases,
                                                       const int2* __restrict__ items, int nitems, int phase) {
    const int i = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6));
    if (i >= nitems) return;
    const int2 it = items[i];
    const StepArgs a = batch_case_args<ST>(cases, it.x, phase);
    march2d_item<MODEL, ST, K>(a, it.y);
}

template <int MODEL, int ST>
hipError_t blocked_batch2d_ms(const BatchCase* cases, const int2* items, int nitems, int phase, int steps,
                              const BlockedBatch& b, hipStream_t s) {
    if (nitems <= 0) return hipSuccess;
    if (steps < 2 || steps > b.k || (b.rows > 0 && steps != b.k)) return hipErrorInvalidValue;
    const dim3 waves((nitems + 3) / 4), blk(256);
    if (b.rows == 0) {
        hipLaunchKernelGGL((k_batch_tile2d<MODEL, ST>), dim3(nitems), dim3(b.threads),
                           tile2d_lds_bytes<ST>(b.threads, TILE2D_MAX_TX), s, cases, items, phase, steps);
        return hipGetLastError();
    }
    switch (b.k) {
    case 2: hipLaunchKernelGGL((k_batch_march2d<MODEL, ST, 2>), waves, blk, 0, s, cases, items, nitems, phase); break;
    case 3: hipLaunchKernelGGL((k_batch_march2d<MODEL, ST, 3>), waves, blk, 0, s, cases, items, nitems, phase); break;
    case 4: hipLaunchKernelGGL((k_batch_march2d<MODEL, ST, 4>), waves, blk, 0, s, cases, items, nitems, phase); break;
    case 5: hipLaunchKernelGGL((k_batch_march2d<MODEL, ST, 5>), waves, blk, 0, s, cases, items, nitems, phase); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int MODEL>
hipError_t blocked_batch2d_m(int st, const BatchCase* cases, const int2* items, int nitems, int phase, int steps,
                             const BlockedBatch& b, hipStream_t s) {
    switch (st) {
#if TCLBX_HAS_F64
    case ST_F64: return blocked_batch2d_ms<MODEL, ST_F64>(cases, items, nitems, phase, steps, b, s);
#endif
#if TCLBX_HAS_FLOAT
    case ST_F32: return blocked_batch2d_ms<MODEL, ST_F32>(cases, items, nitems, phase, steps, b, s);
    case ST_F32S: return blocked_batch2d_ms<MODEL, ST_F32S>(cases, items, nitems, phase, steps, b, s);
    case ST_F16S: return blocked_batch2d_ms<MODEL, ST_F16S>(cases, items, nitems, phase, steps, b, s);
    case ST_BF16S: return blocked_batch2d_ms<MODEL, ST_BF16S>(cases, items, nitems, phase, steps, b, s);
    case ST_F16S_SR: return blocked_batch2d_ms<MODEL, ST_F16S_SR>(cases, items, nitems, phase, steps, b, s);
    case ST_BF16S_SR: return blocked_batch2d_ms<MODEL, ST_BF16S_SR>(cases, items, nitems, phase, steps, b, s);
#endif
    }
    return hipErrorInvalidValue;
}

}  // namespace tclbx
