// kernels.hip -- host side of the node kernels (kernels_impl.h): the
// non-template kernels (density access, the Globals reduction, the copy),
// and the launch entry points of kernels.h, which hand each model to the
// compile unit of its family (kernels_<family>.hip).
#include "kernels_impl.h"

#include <algorithm>
#include <cmath>
#include <vector>

namespace tclbx {

// the compile unit of a family that holds the kernels of this storage format
#define TCLBX_PICK(name, storage) ((storage) == ST_F64 ? name##_f64 : name##_f32)

int kernel_nglobals(int model) {
    switch (model) {
    case MODEL_D2Q9_SRT: return Lat<MODEL_D2Q9_SRT>::G;
    case MODEL_D2Q9_SRT_DRAG: return Lat<MODEL_D2Q9_SRT_DRAG>::G;
    case MODEL_D3Q19: return Lat<MODEL_D3Q19>::G;
    case MODEL_D3Q19_LID: return Lat<MODEL_D3Q19_LID>::G;
    case MODEL_D2Q9: return Lat<MODEL_D2Q9>::G;
    case MODEL_D2Q9_DRAG: return Lat<MODEL_D2Q9_DRAG>::G;
    case MODEL_D3Q27: return Lat<MODEL_D3Q27>::G;
    case MODEL_D3Q27_CUMULANT: return Lat<MODEL_D3Q27_CUMULANT>::G;
    case MODEL_D3Q27_CUMULANT_SMAG: return Lat<MODEL_D3Q27_CUMULANT_SMAG>::G;
    case MODEL_D3Q27_CUMULANT_IB: return Lat<MODEL_D3Q27_CUMULANT_IB>::G;
    case MODEL_D3Q27_CUMULANT_IB_SMAG: return Lat<MODEL_D3Q27_CUMULANT_IB_SMAG>::G;
    case MODEL_D3Q27_CUMULANT_AVG: return Lat<MODEL_D3Q27_CUMULANT_AVG>::G;
    case MODEL_D3Q27_CUMULANT_AVG_IB: return Lat<MODEL_D3Q27_CUMULANT_AVG_IB>::G;
    case MODEL_D3Q27_CUMULANT_AVG_SMAG: return Lat<MODEL_D3Q27_CUMULANT_AVG_SMAG>::G;
    case MODEL_D3Q27_CUMULANT_AVG_IB_SMAG: return Lat<MODEL_D3Q27_CUMULANT_AVG_IB_SMAG>::G;
    case MODEL_D2Q9_AUTOSYM: return Lat<MODEL_D2Q9_AUTOSYM>::G;
    case MODEL_D2Q9_AUTOSYM2: return Lat<MODEL_D2Q9_AUTOSYM2>::G;
    case MODEL_D2Q9_BC: return Lat<MODEL_D2Q9_BC>::G;
    case MODEL_D2Q9_BC_AUTOSYM: return Lat<MODEL_D2Q9_BC_AUTOSYM>::G;
    case MODEL_D2Q9_BC_AUTOSYM2: return Lat<MODEL_D2Q9_BC_AUTOSYM2>::G;
    }
    return 0;
}

template <int ST>
__global__ void k_get_density(const void* buf, long long pitch, long long n, int q, double w, double* out) {
    using S = Store<ST>;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = (double)S::get(((const typename S::T*)buf)[q * pitch + i], (typename S::R)w);
}

template <int ST>
__global__ void k_set_density(void* buf, long long pitch, long long n, int q, double w, const double* in) {
    using S = Store<ST>;
    using R = typename S::R;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    ((typename S::T*)buf)[q * pitch + i] = S::put((R)in[i], (R)w);
}

// deterministic second pass: block (Global gi, lattice c) sums slots
// [first_c, first_c + count_c) of that Global's partials contiguously, TwoSum
// pairs throughout, and adds the result to out[c*nglob + gi] (cleared before
// a Globals step, accumulated over steps with ITER_GLOBS).  The order depends
// only on the lattice's own tiles, so a lattice gets the same Globals alone
// and in a batch.
__global__ void __launch_bounds__(256) k_reduce_globals(const double* gpart, int nslots, int nglob,
                                                        int sum_globals, const int* first, const int* count,
                                                        double* out) {
    const int gi = blockIdx.x;
    const int c = blockIdx.y;
    const bool is_sum = gi < sum_globals;
    const int n0 = first ? first[c] : 0;
    const int nb = count ? count[c] : nslots;
    const double* p = gpart + ((size_t)gi * nslots + n0) * 2;
    double v = 0.0, cc = 0.0;
    for (int b = threadIdx.x; b < nb; b += blockDim.x) {
        if (is_sum) dd_add(v, cc, p[2 * b], p[2 * b + 1]);
        else v = fmax(v, p[2 * b]);
    }
    __shared__ double lds[4][2];
    if (is_sum) wave_sum_dd(v, cc);
    else v = wave_max(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) { lds[wave][0] = v; lds[wave][1] = cc; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = lds[0][0], rc = lds[0][1];
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) {
            if (is_sum) dd_add(r, rc, lds[w][0], lds[w][1]);
            else r = fmax(r, lds[w][0]);
        }
        double* o = out + (size_t)c * nglob + gi;
        *o = is_sum ? *o + (r + rc) : fmax(*o, r);
    }
}

// plain device copy, one 16-byte vector per thread (the fastest of the copy
// shapes measured on MI355X): the bandwidth ceiling the node kernel is
// compared with, and a kernel of known traffic for calibrating the HBM byte
// counters
__global__ void __launch_bounds__(256) k_copy(const uint4* __restrict__ src, uint4* __restrict__ dst, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

hipError_t launch_copy(const void* src, void* dst, size_t bytes, hipStream_t s) {
    const size_t n = bytes / sizeof(uint4);
    const size_t blocks = (n + 255) / 256;
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_copy, dim3((unsigned)blocks), dim3(256), 0, s, (const uint4*)src, (uint4*)dst, n);
    return hipGetLastError();
}

namespace {
double weight(int model, int q) {
    if (model == MODEL_D3Q27) return Lat<MODEL_D3Q27>::w(q);
    if ((model >= MODEL_D3Q27_CUMULANT_IB && model <= MODEL_D3Q27_CUMULANT_AVG_IB_SMAG) ||
        model == MODEL_D3Q27_CUMULANT || model == MODEL_D3Q27_CUMULANT_SMAG)
        return Lat<MODEL_D3Q27_CUMULANT>::w(q);
    return (model == MODEL_D3Q19 || model == MODEL_D3Q19_LID) ? Lat<MODEL_D3Q19>::w(q) : Lat<MODEL_D2Q9_SRT>::w(q);
}
}  // namespace

// What a 2D lattice takes: single steps, marching waves or LDS tiles, whichever
// has the least estimated time per step.  The coefficients (us; MB of
// populations moved) are fitted to the times of 46 lattices, from 64x64 to
// 4096x2048 and among them 4x262144, 57x20000 and 1000000x4, with single steps,
// waves of k = 3 to 5 and tiles of k = 3 to 5 and 256 to 1024 nodes: within 6
// to 15% (rms) of each, then moved a little so that the choices come closest to
// the best of all: 1.2% behind on average (lines by size alone: 17%, up to 4.2
// times).  us per step
// of single steps, waves and tiles where sizes alone mislead: f32s 256x256 3.6,
// 4.7 and, with k = 3 and 5, 2.5 and 1.8; 1500x1000 21.6, 8.1, 13.4; f16s
// 4x262144, where a strip or tile wastes most of its columns, 10, 56, 18; f64
// 8x131072 33, 66, 18; with stochastic rounding, whose random streams a blocked
// step draws in its halo too, f16s 2000x1500 22, 24, 22 (without 22, 16, 19).
// (k = 4 tiles are left out: the better of 3 and 5 is at most 10% behind.)
struct StepCost2d {
    double single, single_mb;                            // a step
    double tile, tile_mb, tile_rounds;                   // a launch of tiles, a round of blocks,
    double tile_stage, tile_wave, tile_block;            // a round's step, of a SIMD's waves, of a block's
    double march, march_mb, march_hbm, march_row, march_wave;   // waves: a row's step, of a SIMD's waves
};
static const StepCost2d& step_cost2d(int model, int storage, bool sr) {
    static const StepCost2d costs[2][4] = {
        // d2q9_SRT(_drag): f64, f32 and f32s, 16 bit, 16 bit with stochastic rounding
        {{2.60, 0.183, 3.50, 0.117, 0, 1.09, 0.123, 0, 6.64, 0.0399, 0.0444, 0.303, 0.190},
         {2.40, 0.157, 4.15, 0.191, 0, 0.0874, 0.0346, 0.124, 5.24, 0.0735, 0.0478, 0.195, 0.0254},
         {3.32, 0.221, 4.35, 0.227, 0, 0.220, 0.0924, 0.0744, 5.92, 0.0342, 0.0410, 0.228, 0.0851},
         {2.98, 0.267, 4.49, 0.306, 0, 0.192, 0.133, 0, 8.57, 0.0342, 0.0562, 0.241, 0.152}},
        // d2q9(_drag), the same
        {{3.09, 0.182, 1.91, 0.133, 0, 0.897, 0.156, 0.203, 7.54, 0.0261, 0.0499, 0.372, 0.244},
         {2.83, 0.193, 3.41, 0.222, 0, 0.268, 0.0458, 0.128, 6.73, 0.0341, 0.0516, 0.268, 0.0793},
         {2.73, 0.192, 3.40, 0.284, 0, 0.217, 0.090, 0.116, 6.85, 0.0395, 0.0418, 0.196, 0.106},
         {3.04, 0.220, 4.34, 0.207, 0, 0.206, 0.184, 0, 6.76, 0.0608, 0.0222, 0.288, 0.241}}};
    const int f = storage == ST_F64 ? 0 : storage == ST_F32 || storage == ST_F32S ? 1 : sr ? 3 : 2;
    return costs[model == MODEL_D2Q9 || model == MODEL_D2Q9_DRAG][f];
}
static double mb2d(double nodes, int storage) { return nodes * 9 * storage_bytes(storage) / 1e6; }

static int strips2d(int nx, int k) { return (nx + 64 - 2 * (k - 1) - 1) / (64 - 2 * (k - 1)); }

// Marching waves for n lattices of `nodes` nodes in all, and their us per
// step.  With k = 0 the number of steps by size: f64 4096x2048 k 3 104, 4 98, 5
// 95 us per step; 2048x1024 k 3 30.6, 4 27.7, 5 30.5; f32s 4096x2048 60, 50, 44;
// f16s 44.6, 46.7, 50.5 (its conversions make a step dearer than the bytes it
// saves).  Rows for about 3,000 waves, between what pays for the extra rows
// and what evens out the last round (f64 8-12 to 24, float 8 to 12 measured).
static BlockedBatch march_split(const StepCost2d& c, const int2* sizes, int n, long long nodes, int storage, int k,
                                Blocking* cases, double& us) {
    const bool f64 = storage == ST_F64, half = storage == ST_F16S || storage == ST_BF16S;
    BlockedBatch b;
    b.k = k ? k : f64 ? (nodes >= 1ll << 22 ? 5 : 4) : half ? 3 : 5;
    long long rows = 0;
    for (int i = 0; i < n; i++) rows += (long long)strips2d(sizes[i].x, b.k) * sizes[i].y;
    b.rows = (int)std::min<long long>(f64 ? 24 : 12, std::max<long long>(f64 ? 6 : 8, (rows + 3071) / 3072));
    b.threads = 256;
    double wave_rows = 0;   // rows that the waves walk, and the longest walk
    int longest = 0;
    for (int i = 0; i < n; i++) {
        cases[i] = Blocking();
        cases[i].k = b.k;
        cases[i].rows = std::min(b.rows, sizes[i].y);
        const int walk = cases[i].rows + 2 * (b.k - 1);
        wave_rows += (double)strips2d(sizes[i].x, b.k) * ((sizes[i].y + cases[i].rows - 1) / cases[i].rows) * walk;
        longest = std::max(longest, walk);
    }
    const double mb = mb2d(64 * wave_rows + (double)nodes, storage);
    const bool hbm = mb2d(2.0 * (double)nodes, storage) > 200;   // past the Infinity Cache
    us = (c.march + (c.march_mb + (hbm ? c.march_hbm : 0)) * mb) / b.k + c.march_row * longest +
         c.march_wave * wave_rows / 1024;
    return b;
}

// The tiles of the least estimated time per step, among ks steps per launch:
// a round of blocks takes k stages, in each of which a SIMD steps its waves
// one after the other.
static BlockedBatch tile_split(const StepCost2d& c, const int2* sizes, int n, long long nodes, int storage,
                               const std::vector<int>& ks, Blocking* cases, double& us) {
    const int capacity = storage == ST_F64 ? 6 : 8;   // waves per SIMD
    std::vector<Blocking> trial(n);
    BlockedBatch best;
    us = 1e300;
    for (int k : ks)
        for (int threads : {256, 512, 1024}) {
            long long tiles = 0;
            for (int i = 0; i < n && tiles >= 0; i++) {
                long long fewest = 0;
                // the widest of the shapes with the fewest tiles: its rows
                // are longer runs of memory (1024x128 in FP64: 256 tiles
                // of 40x25 3.1 us per step, of 24x42 3.6)
                for (int tx : {TILE2D_MAX_TX, 56, 48, 44, 40, 36, 32, 28, 24, 20, 16}) {
                    const int ty = threads / tx, wx = tx - 2 * (k - 1), wy = ty - 2 * (k - 1);
                    if (wx < 1 || wy < 1) continue;
                    const long long t = (long long)((sizes[i].x + wx - 1) / wx) * ((sizes[i].y + wy - 1) / wy);
                    if (fewest == 0 || t < fewest) {
                        fewest = t;
                        trial[i].k = k; trial[i].rows = 0; trial[i].tx = tx; trial[i].ty = ty;
                    }
                }
                tiles = fewest ? tiles + fewest : -1;
            }
            if (tiles < 0) continue;   // no tile of this many nodes has a middle
            const int waves = threads / 256, fit = std::max(1, capacity / waves);   // blocks a CU holds
            const long long per_cu = (tiles + 255) / 256;
            double rounds = (double)tiles / (256.0 * fit);
            rounds = rounds < 4 ? std::ceil(rounds) : rounds + 0.5;
            const double t = (c.tile + c.tile_mb * mb2d((double)tiles * threads + (double)nodes, storage) +
                              c.tile_rounds * rounds) / k + c.tile_block * waves +
                             rounds * (c.tile_stage + c.tile_wave * waves * std::min<long long>(fit, per_cu));
            if (t < us) {
                us = t;
                best.k = k; best.rows = 0; best.threads = threads;
                for (int i = 0; i < n; i++) {
                    cases[i] = trial[i];
                    cases[i].nt = per_cu <= fit;
                }
            }
        }
    return best;
}

Blocking blocking2d(int model, int nx, int ny, int storage, bool sr, int k) {
    const StepCost2d& c = step_cost2d(model, storage, sr);
    const int2 size = make_int2(nx, ny);
    const long long nodes = (long long)nx * ny;
    Blocking tile, march;
    double tile_us, march_us = 1e300;
    tile_split(c, &size, 1, nodes, storage, k ? std::vector<int>{k} : std::vector<int>{3, 5}, &tile, tile_us);
    if (k <= MARCH2D_MAX_K) march_split(c, &size, 1, nodes, storage, k, &march, march_us);
    const double single_us = c.single + c.single_mb * mb2d(2.0 * (double)nodes, storage);
    if (k == 0 && single_us < std::min(tile_us, march_us)) return Blocking();
    return march_us < tile_us ? march : tile;
}

// A batch marches by whole launches of k steps and takes the rest as single
// steps, which short calls pay for (Globals every 10 steps), so it marches only
// where that gains most; its tiles' coefficients are those of single rounds of
// 128x32 and 1024x128 (f64: 16x16 tiles, one wave per SIMD, 0.84 us a stage,
// 32x16 1.33, 32x32 2.25; f32s 0.55, 1.06, 1.37; f16s 0.83, -, 2.1).
BlockedBatch blocking2d_batch(const int2* sizes, int n, int storage, int k, Blocking* cases) {
    StepCost2d c = {};
    c.tile_rounds = 2.8;
    c.tile_stage = 0.4;
    c.tile_wave = storage == ST_F64 ? 0.47 : storage == ST_F32 || storage == ST_F32S ? 0.22 : 0.26;
    long long nodes = 0;
    for (int i = 0; i < n; i++) nodes += (long long)sizes[i].x * sizes[i].y;
    double us;
    if (k <= MARCH2D_MAX_K && nodes >= (storage == ST_F64 ? 1ll << 20 : 1ll << 22))
        return march_split(c, sizes, n, nodes, storage, k, cases, us);
    return tile_split(c, sizes, n, nodes, storage, k ? std::vector<int>{k} : std::vector<int>{3, 4, 5}, cases, us);
}

// The march's time is rounds of blocks (one per CU: the tile fills its LDS) x
// (layers + 3 iterations) x the time of an iteration, which depends on the
// tile and little on the lattice (us, below and above 4M nodes): d3q19 f64
// 34x15 8.5, 8.9, f32s 66x15 7.1, 7.8, 34x30 7.2, 8.6; FP64 34x10 d3q27 7.5,
// cumulant 8.8.  So the layers are those of the fewest iterations in all, and
// the march is taken where they beat the single step's rate (MLUPS, below and
// above 8M nodes: d3q19 17.3k, 18.1k and 34k, 37.2k, d3q27 12.8k, cumulant
// 12.5k).  us per step, single / march: d3q19 f64 256^3 924 / 784, 192x176x160
// 309 / 245, 61x48x57 13.6 / 24 (single stays); f32s 256^3 450 / 352,
// 192x176x160 156 / 114, 157x131x97 72 / 47; d3q27 f64 256x128x128 326 / 251;
// cumulant f64 336 / 295.  The 16-bit formats and the 27-velocity float steps
// are bound by their instructions and gain nothing (d3q19 f16s 256^3 253 /
// 257, d3q27 f32s 256x128x128 170 / 172).
Blocking blocking3d(int model, int nx, int ny, int nz, int storage) {
    struct Tile { int tx, ty; double us, us_large; };
    const Tile f64[1] = {{34, 15, 8.5, 8.9}}, f32[2] = {{66, 15, 7.1, 7.8}, {34, 30, 7.2, 8.6}};
    const Tile q27[1] = {{34, 10, 7.5, 7.5}}, cum[1] = {{34, 10, 8.8, 8.8}};
    const double nodes = (double)nx * ny * nz;
    const Tile* tiles = nullptr;
    int ntiles = 1;
    double mlups = 0;
    if (model == MODEL_D3Q19 || model == MODEL_D3Q19_LID) {
        if (storage == ST_F64) { tiles = f64; mlups = nodes < 8e6 ? 17300 : 18100; }
        if (storage == ST_F32 || storage == ST_F32S) { tiles = f32; ntiles = 2; mlups = nodes < 8e6 ? 34000 : 37200; }
    } else if (storage == ST_F64 && model == MODEL_D3Q27) {
        tiles = q27; mlups = 12800;
    } else if (storage == ST_F64 && (model == MODEL_D3Q27_CUMULANT || model == MODEL_D3Q27_CUMULANT_SMAG)) {
        tiles = cum; mlups = 12500;
    }
    Blocking best;
    if (!tiles) return best;
    double best_us = 2 * 0.97 * nodes / mlups;   // two single steps
    for (int t = 0; t < ntiles; t++) {
        const int wx = tiles[t].tx - 2, wy = tiles[t].ty - 2;
        const long long columns = (long long)((nx + wx - 1) / wx) * ((ny + wy - 1) / wy);
        for (int segs = 1; segs <= nz; segs++) {
            const int rows = (nz + segs - 1) / segs;
            const long long blocks = columns * ((nz + rows - 1) / rows);
            if (blocks > 256 * 64 && segs > 1) break;
            const double us = (double)((blocks + 255) / 256) * (rows + 3) * (nodes < 4e6 ? tiles[t].us : tiles[t].us_large);
            if (us < best_us) {
                best_us = us;
                best.k = 2; best.rows = rows; best.tx = tiles[t].tx; best.ty = tiles[t].ty;
            }
        }
    }
    return best;
}

int blocked2d_items(const StepArgs& a) {
    if (a.tb_rows > 0) return strips2d(a.nx, a.tb_k) * ((a.ny + a.tb_rows - 1) / a.tb_rows);
    const int wx = a.tb_tx - 2 * (a.tb_k - 1), wy = a.tb_ty - 2 * (a.tb_k - 1);
    if (wx < 1 || wy < 1) return 0;
    return ((a.nx + wx - 1) / wx) * ((a.ny + wy - 1) / wy);
}

bool blocked2d_model(int model) {
    return model == MODEL_D2Q9_SRT || model == MODEL_D2Q9_SRT_DRAG || model == MODEL_D2Q9 || model == MODEL_D2Q9_DRAG;
}

hipError_t launch_blocked_batch(int model, int storage, const BatchCase* cases, const int2* items, int nitems,
                                int phase, int steps, const BlockedBatch& b, hipStream_t s) {
    const hipError_t e = TCLBX_PICK(blocked_batch_2d, storage)(model, storage, cases, items, nitems, phase, steps, b, s);
    return e == hipErrorNotFound ? hipErrorInvalidValue : e;
}

int step_blocks(const StepArgs& a, bool globals, int block) {
    const int rpb = globals ? a.rpb : a.rpt;
    if (a.flat & (globals ? 2 : 1)) {
        const long long chunks = ((long long)a.nx * a.ny * a.nz + block - 1) / block;
        return (int)((chunks + rpb - 1) / rpb);
    }
    const int rows = a.ny * a.nz;
    return a.bpr * ((rows + rpb - 1) / rpb);
}

hipError_t launch_step(int model, int storage, bool globals, const StepArgs& a, int block, hipStream_t s) {
    if (hipError_t e = TCLBX_PICK(step_2d, storage)(model, storage, globals, a, block, s); e != hipErrorNotFound) return e;
    if (hipError_t e = TCLBX_PICK(step_d3q19, storage)(model, storage, globals, a, block, s); e != hipErrorNotFound) return e;
    if (hipError_t e = TCLBX_PICK(step_d3q27, storage)(model, storage, globals, a, block, s); e != hipErrorNotFound) return e;
    if (hipError_t e = TCLBX_PICK(step_cum, storage)(model, storage, globals, a, block, s); e != hipErrorNotFound) return e;
    if (hipError_t e = TCLBX_PICK(step_cumavg, storage)(model, storage, globals, a, block, s); e != hipErrorNotFound) return e;
    return hipErrorInvalidValue;
}

hipError_t launch_init(int model, int storage, const StepArgs& a, int block, hipStream_t s) {
    if (hipError_t e = TCLBX_PICK(init_2d, storage)(model, storage, a, block, s); e != hipErrorNotFound) return e;
    if (hipError_t e = TCLBX_PICK(init_d3q19, storage)(model, storage, a, block, s); e != hipErrorNotFound) return e;
    if (hipError_t e = TCLBX_PICK(init_d3q27, storage)(model, storage, a, block, s); e != hipErrorNotFound) return e;
    if (hipError_t e = TCLBX_PICK(init_cum, storage)(model, storage, a, block, s); e != hipErrorNotFound) return e;
    if (hipError_t e = TCLBX_PICK(init_cumavg, storage)(model, storage, a, block, s); e != hipErrorNotFound) return e;
    return hipErrorInvalidValue;
}

hipError_t launch_reduce_globals(const double* gpart, int nblocks, int nglob, int sum_globals, double* out,
                                 hipStream_t s) {
    hipLaunchKernelGGL(k_reduce_globals, dim3(nglob, 1), dim3(256), 0, s, gpart, nblocks, nglob, sum_globals,
                       (const int*)nullptr, (const int*)nullptr, out);
    return hipGetLastError();
}

hipError_t launch_reduce_globals_cases(const double* gpart, int nslots, int nglob, int sum_globals, int ncases,
                                       const int* first, const int* count, double* out, hipStream_t s) {
    if (ncases <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_reduce_globals, dim3(nglob, ncases), dim3(256), 0, s, gpart, nslots, nglob, sum_globals,
                       first, count, out);
    return hipGetLastError();
}

hipError_t launch_batch_step(int model, int storage, bool globals, const BatchCase* cases, const int2* tiles,
                             int ntiles, int phase, double* gpart, int grid, int block, hipStream_t s) {
    if (hipError_t e = TCLBX_PICK(batch_2d, storage)(model, storage, globals, cases, tiles, ntiles, phase, gpart, grid, block, s);
        e != hipErrorNotFound)
        return e;
    if (hipError_t e = TCLBX_PICK(batch_d3q19, storage)(model, storage, globals, cases, tiles, ntiles, phase, gpart, grid, block, s);
        e != hipErrorNotFound)
        return e;
    if (hipError_t e = TCLBX_PICK(batch_d3q27, storage)(model, storage, globals, cases, tiles, ntiles, phase, gpart, grid, block, s);
        e != hipErrorNotFound)
        return e;
    if (hipError_t e = TCLBX_PICK(batch_cum, storage)(model, storage, globals, cases, tiles, ntiles, phase, gpart, grid, block, s);
        e != hipErrorNotFound)
        return e;
    if (hipError_t e = TCLBX_PICK(batch_cumavg, storage)(model, storage, globals, cases, tiles, ntiles, phase, gpart, grid, block, s);
        e != hipErrorNotFound)
        return e;
    return hipErrorInvalidValue;
}

hipError_t launch_quantity(int model, int storage, int q, const StepArgs& a, int x0, int y0, int z0, int rx,
                           int ry, int rz, double scale, double* out, hipStream_t s) {
    if (hipError_t e = TCLBX_PICK(quantity_2d, storage)(model, storage, q, a, x0, y0, z0, rx, ry, rz, scale, out, s);
        e != hipErrorNotFound)
        return e;
    if (hipError_t e = TCLBX_PICK(quantity_d3q19, storage)(model, storage, q, a, x0, y0, z0, rx, ry, rz, scale, out, s);
        e != hipErrorNotFound)
        return e;
    if (hipError_t e = TCLBX_PICK(quantity_d3q27, storage)(model, storage, q, a, x0, y0, z0, rx, ry, rz, scale, out, s);
        e != hipErrorNotFound)
        return e;
    if (hipError_t e = TCLBX_PICK(quantity_cum, storage)(model, storage, q, a, x0, y0, z0, rx, ry, rz, scale, out, s);
        e != hipErrorNotFound)
        return e;
    if (hipError_t e = TCLBX_PICK(quantity_cumavg, storage)(model, storage, q, a, x0, y0, z0, rx, ry, rz, scale, out, s);
        e != hipErrorNotFound)
        return e;
    return hipErrorInvalidValue;
}

hipError_t launch_get_density(int model, int storage, const void* buf, long long pitch, long long n, int q,
                              double* out, hipStream_t s) {
    const dim3 grid((unsigned)((n + 255) / 256)), blk(256);
    const double w = weight(model, q);
    switch (storage) {
    case ST_F64: hipLaunchKernelGGL(k_get_density<ST_F64>, grid, blk, 0, s, buf, pitch, n, q, w, out); break;
    case ST_F32: hipLaunchKernelGGL(k_get_density<ST_F32>, grid, blk, 0, s, buf, pitch, n, q, w, out); break;
    case ST_F32S: hipLaunchKernelGGL(k_get_density<ST_F32S>, grid, blk, 0, s, buf, pitch, n, q, w, out); break;
    case ST_F16S: hipLaunchKernelGGL(k_get_density<ST_F16S>, grid, blk, 0, s, buf, pitch, n, q, w, out); break;
    case ST_BF16S: hipLaunchKernelGGL(k_get_density<ST_BF16S>, grid, blk, 0, s, buf, pitch, n, q, w, out); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_set_density(int model, int storage, void* buf, long long pitch, long long n, int q,
                              const double* in, hipStream_t s) {
    const dim3 grid((unsigned)((n + 255) / 256)), blk(256);
    const double w = weight(model, q);
    switch (storage) {
    case ST_F64: hipLaunchKernelGGL(k_set_density<ST_F64>, grid, blk, 0, s, buf, pitch, n, q, w, in); break;
    case ST_F32: hipLaunchKernelGGL(k_set_density<ST_F32>, grid, blk, 0, s, buf, pitch, n, q, w, in); break;
    case ST_F32S: hipLaunchKernelGGL(k_set_density<ST_F32S>, grid, blk, 0, s, buf, pitch, n, q, w, in); break;
    case ST_F16S: hipLaunchKernelGGL(k_set_density<ST_F16S>, grid, blk, 0, s, buf, pitch, n, q, w, in); break;
    case ST_BF16S: hipLaunchKernelGGL(k_set_density<ST_BF16S>, grid, blk, 0, s, buf, pitch, n, q, w, in); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace tclbx
