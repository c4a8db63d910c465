// pair.hip -- launches of the two-step kernel (pair.hpp) for one cavity.
#include <hip/hip_runtime.h>

#include "context.hpp"
#include "pair.hpp"

using namespace lbm;

namespace {

// Threads of a block (= cells of a plane with its rim), and the waves per SIMD
// its registers must allow: two planes of 19 populations fill the LDS of a CU in
// FP64 and FP32 (one block per CU; in FP32 two blocks of 512, with their larger
// share of rim, took 8 % more time at 256^3).
template <class S>
struct PairShape;
template <>
struct PairShape<StoreF64> {
    static constexpr int NT = 512, WAVES = 2;
};
template <>
struct PairShape<StoreF32> {
    static constexpr int NT = 1024, WAVES = 4;
};

template <class S, int COLL, bool MACRO, bool LOOP>
__global__ __launch_bounds__(PairShape<S>::NT, PairShape<S>::WAVES) void k_cavity_pair(const PairArgs a) {
    __shared__ typename S::T buf[2][Q][PairShape<S>::NT];
    const int wg = xcd_order(blockIdx.x, gridDim.x);
    cavity_pair<S, COLL, MACRO, PairShape<S>::NT>(a, a.t, wg, buf, [&](int i, int j, int k, bool mid) {
        if constexpr (LOOP) return LoopbackHalo<S>{a, mid ? a.halo_mid : a.halo_out, i, j, k};
        else return NoPost{};
    });
}

using PairFn = void (*)(const PairArgs);

template <class S>
struct PairTable {
    // step[collision][macro][loop]
    static constexpr PairFn step[2][2][2] = {
        {{k_cavity_pair<S, COLL_MRT, false, false>, k_cavity_pair<S, COLL_MRT, false, true>},
         {k_cavity_pair<S, COLL_MRT, true, false>, k_cavity_pair<S, COLL_MRT, true, true>}},
        {{k_cavity_pair<S, COLL_BGK, false, false>, k_cavity_pair<S, COLL_BGK, false, true>},
         {k_cavity_pair<S, COLL_BGK, true, false>, k_cavity_pair<S, COLL_BGK, true, true>}}};
};

}  // namespace

namespace lbm {

bool pair_plan(int nx, int ny, int nz, int storage, int cus, PairTiles* out) {
    switch (storage) {
    case LBM_STORE_F64: return pair_plan(nx, ny, nz, PairShape<StoreF64>::NT, Q, 8, cus, out);
    case LBM_STORE_F32: return pair_plan(nx, ny, nz, PairShape<StoreF32>::NT, Q, 4, cus, out);
    }
    return false;  // FP16: see below
}

// The tiles, and whether two steps go faster this way.
//
// Time goes by turns (planes) of the busiest CU: with one block per CU a launch
// takes ceil(blocks / CUs) rounds of cz + 2 turns.  A turn takes at least 4.3 us
// (65^3 and 96^3, which lie in the memory-side cache).  On large boxes it is
// bound by memory (256^3 FP64: 622 us a step without the arithmetic and LDS, 627
// with them) and goes as the bytes it moves, a row of the tile and its rim
// costing 128 bytes more per population than it holds (the lines at its ends):
// FP64 32 x 13 tiles 7.3 us, 64 x 5 5.7; FP32 64 x 13 6.9, 32 x 26 8.0, i.e.
// 0.77 ns per such byte with every CU busy, less where fewer are (6.5 us for FP64
// 32 x 13 with 240 of 256), 0.5 ns in the cache.  Rows that are not whole 64-byte
// groups cost 1.1 to 1.4 times that outside the cache.  A one-step launch takes
// 5 us and 5.2 TB/s of its traffic.
// FP16 keeps the one-step kernel: it is bound by VALU issue, of which the rim
// takes a third more (276 against 238 us a step at 256^3).
bool pair_plan(int nx, int ny, int nz, int nt, int pops, int elem, int cus, PairTiles* out) {
    const double bytes = elem, share = pops / 19.0;
    const bool cached = double(nx) * ny * nz * 2 * pops * bytes < 200e6;
    const long long plane = ((long long)nx + 15) / 16 * 16 * ny;
    if (plane * (long long)bytes >= PLANE_RANGE) return false;  // the lanes' offsets
    double best = 1e30;
    auto consider = [&](int tx) {
        PairTiles t{};
        t.tx = tx;
        t.ntx = (nx + tx - 1) / tx;
        t.hx = t.ntx > 1;
        t.w = tx + 2 * t.hx;
        if (t.w > nt) return;
        const int rows = nt / t.w;
        if (rows >= ny) {
            t.ty = ny;
        } else if (rows >= 3) {
            t.nty = (ny + rows - 3) / (rows - 2);
            t.ty = (ny + t.nty - 1) / t.nty;  // even tiles
        } else {
            return;
        }
        t.nty = (ny + t.ty - 1) / t.ty;
        t.hy = t.nty > 1;
        t.h = t.ty + 2 * t.hy;
        for (int ncz = 1; ncz <= nz; ++ncz) {
            t.cz = (nz + ncz - 1) / ncz;
            t.ncz = (nz + t.cz - 1) / t.cz;
            const long long blocks = (long long)t.ntx * t.nty * t.ncz;
            if (blocks > (1 << 24)) break;
            const long long rounds = (blocks + cus - 1) / cus;
            const double busy = double(blocks) / double(rounds * cus);
            const double moved = t.h * (t.w * bytes + 128.0) + t.tx * t.ty * bytes;
            double turn = (cached ? 5.0e-4 : 7.7e-4) * share * moved * (0.5 + 0.5 * busy);
            if (!cached && t.tx % 16 != 0 && t.ntx > 1) turn *= 1.2;
            if (turn < 4.3) turn = 4.3;
            const double time = (double(rounds) * (t.cz + 2) * turn + 4.0) / 2;
            if (time < best) {
                best = time;
                *out = t;
            }
        }
    };
    for (int tx = 32; tx < nx && tx <= 128; tx += 32) consider(tx);
    for (int n = 1; n <= 4; ++n) consider((nx + n - 1) / n);
    const double one = double(nx) * ny * nz * 2 * pops * bytes / 5.2e6 + 5.0;
    // (a margin for what the model misses: 0.85 on small boxes, where FP32 with
    // temperature at 51^3 took 10.9 us in pairs, 8.8 one by one)
    return best < (one < 12.0 ? 0.85 : 0.95) * one;
}

}  // namespace lbm

int lbm_launch_pair(const PairArgs& a, int storage, int collision, bool macro, bool loop, hipStream_t stream) {
    const int coll = collision == LBM_BGK ? COLL_BGK : COLL_MRT;
    PairFn fn;
    int threads;
    if (storage == LBM_STORE_F32) {
        fn = PairTable<StoreF32>::step[coll][macro][loop];
        threads = PairShape<StoreF32>::NT;
    } else {
        fn = PairTable<StoreF64>::step[coll][macro][loop];
        threads = PairShape<StoreF64>::NT;
    }
    const dim3 grid((unsigned)(a.t.ntx * a.t.nty * a.t.ncz));
    hipLaunchKernelGGL(fn, grid, dim3(threads), 0, stream, a);
    return lbm_check_launch();
}
