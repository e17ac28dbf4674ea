// kernels_march3d.h -- two plain steps of a 3D lattice in one launch,
// bit-identical to single steps (they run the node functions of
// kernels_impl.h).
#pragma once
#include "kernels_impl.h"

namespace tclbx {

// one node: Run() on the pulled populations f, no Globals
template <int MODEL, int ST>
__device__ __forceinline__ void plain_node3d(const StepArgs& a, typename Store<ST>::R* f, unsigned nt) {
    using L = Lat<MODEL>;
    using S = Store<ST>;
    using R = typename S::R;
    double* g = nullptr;
    if constexpr (is_d3q19<MODEL>) {
        // (the zone row and the node's place are read by Globals steps only)
        if constexpr (S::shifted)
            d3q19_node_dev<R, false, MODEL == MODEL_D3Q19_LID>(f, nt, a.par, nullptr, g, nullptr, 0, 0, 0, 0, 0, 0, a.fpar);
        else
            d3q19_node<R, false, MODEL == MODEL_D3Q19_LID>(f, nt, a.par, nullptr, g, nullptr, 0, 0, 0, 0, 0, 0, a.fpar);
    } else {
        int zone = (int)(nt >> L::ZSHIFT);
        if (zone >= a.nzones) zone = 0;
        const double* zr = a.zone + (size_t)zone * a.zcols;
        if constexpr (MODEL == MODEL_D3Q27) d3q27_node<R, false>(f, nt, a.par, zr, g);
        else cum_node<R, false, is_cum_smag<MODEL>>(f, nt, a.par, zr, g);
    }
}

// place of direction i among the directions of its e_z
template <class L> __host__ __device__ constexpr int ez_rank(int i) {
    int r = 0;
    for (int j = 0; j < i; j++) r += L::ez(j) == L::ez(i);
    return r;
}
template <class L> __host__ __device__ constexpr int ez_count(int ez) {
    int r = 0;
    for (int j = 0; j < L::Q; j++) r += L::ez(j) == ez;
    return r;
}
// values per column that the march keeps in LDS
template <class L> constexpr int march3d_slots = ez_count<L>(-1) + 2 * ez_count<L>(0) + 3 * ez_count<L>(1);

// f stored: populations of a node rounded as the single step rounds its
// stores, put(i, value) for each
template <class S, class L, bool DEV, class PUT>
__device__ __forceinline__ void store_node(const typename S::R* f, PUT put) {
    static_assert(!S::stochastic, "the formats that march are not rounded stochastically");
#pragma unroll
    for (int i = 0; i < L::Q; i++) put(i, DEV ? S::unraw(f[i]) : S::put(f[i], (typename S::R)L::w(i)));
}

// Two plain steps of a column of tiles.  Block b owns a TX x TY tile of
// columns, one per thread, of which it writes the middle (TX - 2) x (TY - 2),
// and marches along z over the layers z0 .. z0 + layers - 1.  Each iteration
// takes one layer z: its pulls from the current snapshot are issued; while
// they are in flight layer z - 2 is stepped a second time, pulling from what
// the tile holds in LDS (the e_z = -1 populations of layer z - 1, the e_z = 0
// ones of layer z - 2 and the e_z = +1 ones of layer z - 3); then layer z is
// stepped once and left in LDS.  LDS holds one, two and three layers of the
// three kinds.  A node is read from memory once and written once for two
// steps; the tile's edge and one layer at each end are stepped by two blocks.
// The two barriers stand around the LDS writes alone, so waves drift over
// their arithmetic.
template <int MODEL, int ST, int TX, int TY>
__global__ void __launch_bounds__(TX * TY) k_march3d(StepArgs a, int tiles_x, int tiles_xy, int blocks) {
    using L = Lat<MODEL>;
    using S = Store<ST>;
    using T = typename S::T;
    using R = typename S::R;
    constexpr int Q = L::Q, NT = TX * TY, NM = ez_count<L>(-1), NZ = ez_count<L>(0), NP = ez_count<L>(1);
    constexpr bool DEV = is_d3q19<MODEL> && S::shifted;
    __shared__ T lds[march3d_slots<L> * NT + 2 * (TX + 1)];
    T* const own = lds + TX + 1 + threadIdx.x;
    const int b = xcd_tile(blockIdx.x, blocks);
    const int seg = b / tiles_xy, txy = b - seg * tiles_xy;
    const int by = txy / tiles_x, bx = txy - by * tiles_x;
    const int tx = threadIdx.x % TX, ty = threadIdx.x / TX;
    const int nx = a.nx, ny = a.ny, nz = a.nz;
    const int z0 = seg * a.tb_rows, layers = min(a.tb_rows, nz - z0);
    const int ux = bx * (TX - 2) - 1 + tx, uy = by * (TY - 2) - 1 + ty;
    int x = ux % nx, y = uy % ny;
    if (x < 0) x += nx;
    if (y < 0) y += ny;
    const bool writes = tx >= 1 && tx < TX - 1 && ty >= 1 && ty < TY - 1 && ux < nx && uy < ny;
    const size_t pbytes = (size_t)a.pitch * sizeof(T);
    const unsigned layer = (unsigned)nx * (unsigned)ny;
    // byte offsets, within a layer, of the pulls from y - 1, y, y + 1 (rows)
    // and x - 1, x, x + 1 (columns)
    unsigned off[3][3];
    {
        const int xs[3] = {x == 0 ? nx - 1 : x - 1, x, x == nx - 1 ? 0 : x + 1};
        const int ys[3] = {y == 0 ? ny - 1 : y - 1, y, y == ny - 1 ? 0 : y + 1};
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
            for (int i = 0; i < 3; i++) off[j][i] = ((unsigned)xs[i] + (unsigned)nx * (unsigned)ys[j]) * (unsigned)sizeof(T);
    }
    T v[Q];
    unsigned nt_next;
    // the pulls of layer z: a scalar base and one of the 32-bit offsets each
    const auto fetch = [&](int z) {
        const int zm = z == 0 ? nz - 1 : z - 1, zp = z == nz - 1 ? 0 : z + 1;
        const char* plane = (const char*)a.fin;
        asm volatile("" : "+s"(plane));
        const size_t at[3] = {(size_t)zm * layer * sizeof(T), (size_t)z * layer * sizeof(T), (size_t)zp * layer * sizeof(T)};
        nt_next = *(gptr<const uint16_t>)((const char*)(a.flags + (size_t)z * layer) + off[1][1] / (unsigned)(sizeof(T) / 2));
#pragma unroll
        for (int i = 0; i < Q; i++) {
            v[i] = *(gptr<const T>)(plane + at[1 - L::ez(i)] + off[1 - L::ey(i)][1 - L::ex(i)]);
            plane += pbytes;
            asm volatile("" : "+s"(plane));
        }
    };
    unsigned nt0 = 0, nt1 = 0, nt2 = 0;  // NodeTypes of layers z, z - 1 and z - 2
    int z = z0 == 0 ? nz - 1 : z0 - 1, z1 = 0, z2 = 0;
    int zc = 0;                      // the e_z = 0 layer of z - 2, where z goes
    int p0 = 0, p1 = 1, p2 = 2;      // the e_z = +1 layers of z - 3 (where z goes), z - 2 and z - 1
    fetch(z);
    for (int it = 0; it < layers + 3; it++) {
        // opaque to the optimiser, which would otherwise keep a 64-bit address
        // per direction in registers across the loop and add to each by
        // vector instructions
#pragma unroll
        for (int j = 0; j < 3; j++)
#pragma unroll
            for (int i = 0; i < 3; i++) asm volatile("" : "+v"(off[j][i]));
        R f[Q], fn[Q];
#pragma unroll
        for (int i = 0; i < Q; i++) fn[i] = DEV ? S::raw(v[i]) : S::get(v[i], (R)L::w(i));
        nt0 = nt_next;
        const int znext = z == nz - 1 ? 0 : z + 1;
        if (it + 1 < layers + 2) fetch(znext);
        if (it >= 3) {
            T u[Q];
#pragma unroll
            for (int i = 0; i < Q; i++) {
                const T* src = own - L::ex(i) - L::ey(i) * TX;
                if (L::ez(i) < 0) u[i] = src[ez_rank<L>(i) * NT];
                else if (L::ez(i) == 0) u[i] = src[(NM + zc * NZ + ez_rank<L>(i)) * NT];
                else u[i] = src[(NM + 2 * NZ + p0 * NP + ez_rank<L>(i)) * NT];
            }
#pragma unroll
            for (int i = 0; i < Q; i++) f[i] = DEV ? S::raw(u[i]) : S::get(u[i], (R)L::w(i));
            plain_node3d<MODEL, ST>(a, f, nt2);
            if (writes) {
                char* plane = (char*)a.fout + (size_t)z2 * layer * sizeof(T);
                asm volatile("" : "+s"(plane));
                store_node<S, L, DEV>(f, [&](int, T out) {
                    *(gptr<T>)(plane + off[1][1]) = out;
                    plane += pbytes;
                    asm volatile("" : "+s"(plane));
                });
            }
        }
        if (it < layers + 2) {
            plain_node3d<MODEL, ST>(a, fn, nt0);
            __syncthreads();
            store_node<S, L, DEV>(fn, [&](int i, T out) {
                if (L::ez(i) < 0) own[ez_rank<L>(i) * NT] = out;
                else if (L::ez(i) == 0) own[(NM + zc * NZ + ez_rank<L>(i)) * NT] = out;
                else own[(NM + 2 * NZ + p0 * NP + ez_rank<L>(i)) * NT] = out;
            });
            __syncthreads();
        }
        nt2 = nt1; nt1 = nt0;
        z2 = z1; z1 = z;
        z = znext;
        zc = 1 - zc;
        const int t = p0; p0 = p1; p1 = p2; p2 = t;
    }
}

template <int MODEL, int ST, int TX, int TY>
hipError_t march3d_ms(const StepArgs& a, hipStream_t s) {
    if (a.tb_rows < 1) return hipErrorInvalidValue;
    const int bx = (a.nx + TX - 3) / (TX - 2), by = (a.ny + TY - 3) / (TY - 2), bz = (a.nz + a.tb_rows - 1) / a.tb_rows;
    hipLaunchKernelGGL((k_march3d<MODEL, ST, TX, TY>), dim3(bx * by * bz), dim3(TX * TY), 0, s, a, bx, bx * by, bx * by * bz);
    return hipGetLastError();
}

// the tiles that blocking3d may ask for; their written columns, TX - 2, are
// whole 128-byte lines of a row that starts on one: with a middle of 30 or 62
// columns, whose rows end inside a line, the stores alone ran at 1.6 TB/s
// (256^3 f32s, 450 us per single step: 64x16 tiles 494 us, 66x15 352)
template <int MODEL, int ST>
hipError_t blocked3d_ms(const StepArgs& a, hipStream_t s) {
    if constexpr (Lat<MODEL>::Q == 27) {
        if (a.tb_tx == 34 && a.tb_ty == 10) return march3d_ms<MODEL, ST, 34, 10>(a, s);
    } else if constexpr (ST == ST_F64) {
        if (a.tb_tx == 34 && a.tb_ty == 15) return march3d_ms<MODEL, ST, 34, 15>(a, s);
    } else {
        if (a.tb_tx == 66 && a.tb_ty == 15) return march3d_ms<MODEL, ST, 66, 15>(a, s);
        if (a.tb_tx == 34 && a.tb_ty == 30) return march3d_ms<MODEL, ST, 34, 30>(a, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace tclbx
