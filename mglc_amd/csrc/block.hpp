// block.hpp -- a few steps of the isothermal D3Q19 update on small boxes, one
// block of cells per workgroup.  Internal to libmglc_lbm.so.
//
// A small box does not fill the chip: a one-step launch there costs its launch
// and one chain of load, collision and store, whatever the box.  Here a
// workgroup loads its cells and a rim of `steps - 1` cells around them (one
// cell per thread), makes the first step, and exchanges populations through
// LDS for the further ones; after each step one layer of the rim has served.
// The arithmetic on the rim is repeated by the neighbours, on units that would
// idle.  Every cell goes through the operations of the one-step kernel, so the
// result is the same bit for bit.
#pragma once
#include "step.hpp"

namespace lbm {

struct BlockTiles {
    int steps;             // steps per launch
    int t[3];              // cells written along x, y, z
    int h[3];              // rim on each side (0 along an axis one block spans)
    int w[3];              // cells held: t + 2 h
    int n[3];              // blocks along each axis
};

struct BlockArgs : StepArgs {
    double* lid_out;       // lid density after the last step (lid_rho: before the first)
    void* halo[2];         // loopback: the halo written by the first, third, ... and the second, fourth, ... step
    BlockTiles b;
};

template <class S, int COLL, bool MACRO, int NT, class MakePost>
__device__ __forceinline__ void cavity_block(const BlockArgs& a, const BlockTiles& b, int wg,
                                             typename S::T (&buf)[Q][NT], MakePost&& make_post) {
    using T = typename S::T;
    using R = typename S::Real;
    const T* __restrict__ src = static_cast<const T*>(a.src);
    T* __restrict__ dst = static_cast<T*>(a.dst);
    const int bx = wg % b.n[0], by = (wg / b.n[0]) % b.n[1], bz = wg / (b.n[0] * b.n[1]);
    const int tid = threadIdx.x;
    const int wh = b.w[0] * b.w[1], cells = wh * b.w[2];
    const int cell = min(tid, cells - 1);  // threads past the block repeat its last cell
    const int lz = cell / wh, ly = (cell - lz * wh) / b.w[0], lx = cell - lz * wh - ly * b.w[0];
    const int i = bx * b.t[0] - b.h[0] + lx, j = by * b.t[1] - b.h[1] + ly, k = bz * b.t[2] - b.h[2] + lz;
    const bool own = tid < cells && lx >= b.h[0] && lx < b.h[0] + b.t[0] && ly >= b.h[1] && ly < b.h[1] + b.t[1] &&
                     lz >= b.h[2] && lz < b.h[2] + b.t[2] && i < a.nx && j < a.ny && k < a.nz;
    // a thread outside the domain repeats the nearest cell's work; nobody reads it
    const int ci = min(max(i, 0), a.nx - 1), cj = min(max(j, 0), a.ny - 1), ck = min(max(k, 0), a.nz - 1);
    const bool top = ck == a.nz - 1;
    const int lid_idx = ci + a.nx * cj;
    const long long c = ci + (long long)a.px * (cj + (long long)a.ny * ck);
    double rho_top = top ? a.lid_rho[lid_idx] : 0.0;

    auto from_wall = [&](auto A) {  // the pull of population al leaves the domain
        constexpr int al = decltype(A)::value;
        bool out = false;
        if constexpr (EX[al] != 0) out = out || (unsigned)(ci - EX[al]) >= (unsigned)a.nx;
        if constexpr (EY[al] != 0) out = out || (unsigned)(cj - EY[al]) >= (unsigned)a.ny;
        if constexpr (EZ[al] != 0) out = out || (unsigned)(ck - EZ[al]) >= (unsigned)a.nz;
        return out;
    };
    R f[Q];
    T held[Q];
    const T* s = src + c;
    sfor<Q>([&](auto A) {
        constexpr int al = decltype(A)::value;
        const long long off = (long long)EX[al] + (long long)EY[al] * a.px + (long long)EZ[al] * a.pxy;
        held[al] = s[from_wall(A) ? (long long)OPP[al] * a.ps : (long long)al * a.ps - off];
    });
    sfor<Q>([&](auto A) { f[decltype(A)::value] = S::val(held[decltype(A)::value]); });
    for (int step = 1;; ++step) {
        if (top) {
            f[13] = lid_bounce<S, COLL>(f[13], rho_top, a.u_lid, a.scale, true);
            f[14] = lid_bounce<S, COLL>(f[14], rho_top, a.u_lid, a.scale, false);
        }
        const Moments<R> m = moments<S, COLL>(f, a.inv_scale);
        if (top) rho_top = density_f64<S>(m.sum, a.inv_scale);
        const bool last = step == b.steps;
        if constexpr (MACRO) {
            if (last && own) {
                const long long mc = i + (long long)a.nx * (j + (long long)a.ny * k);
                a.rho[mc] = density_f64<S>(m.sum, a.inv_scale);
                a.u[mc] = double(m.u);
                a.v[mc] = double(m.v);
                a.w[mc] = double(m.w);
            }
        }
        collide<S, COLL>(f, m, a);
        const unsigned h = cell_random<S>(c, a.seed + (unsigned)(step - 1));
        sfor<Q>([&](auto A) {
            constexpr int al = decltype(A)::value;
            held[al] = S::cvt(f[al], store_random<S, al>(h));
        });
        if (own) {
            const auto post = make_post(i, j, k, step);
            if (post.active()) post.store(held);
        }
        if (last) break;
        if (step > 1) __syncthreads();  // the last step's pulls are read
        sfor<Q>([&](auto A) { buf[decltype(A)::value][tid] = held[decltype(A)::value]; });
        __syncthreads();
        sfor<Q>([&](auto A) {
            constexpr int al = decltype(A)::value;
            // (past the rim's edge: any column, for a cell whose use is over)
            const int nb = min(max(tid - EX[al] - EY[al] * b.w[0] - EZ[al] * wh, 0), NT - 1);
            f[al] = from_wall(A) ? S::val(held[OPP[al]]) : S::val(buf[al][nb]);
        });
    }
    if (own) {
        if (top) a.lid_out[lid_idx] = rho_top;
        sfor<Q>([&](auto A) { dst[(long long)decltype(A)::value * a.ps + c] = held[decltype(A)::value]; });
    }
}

// The blocks for a box on a device of `cus` CUs; false: another kernel is
// faster.
bool block_plan(int nx, int ny, int nz, int storage, int cus, BlockTiles* out);

}  // namespace lbm

// Launch b.steps steps of the block kernel (walls only) for `a` on `stream`.
int lbm_launch_block(const lbm::BlockArgs& a, int storage, int collision, bool macro, bool loop, hipStream_t stream);
