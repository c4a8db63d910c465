// pair.hip -- launches of the two-step kernel (pair.hpp) for one cavity.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <functional>
#include <utility>

#include "context.hpp"
#include "pair.hpp"

using namespace lbm;

namespace {

template <class S, int COLL, bool MACRO, bool LOOP>
__global__ __launch_bounds__(PairShape<S>::NT, PairShape<S>::WAVES) void k_cavity_pair(const PairArgs a) {
    __shared__ typename S::T buf[2][Q][PairShape<S>::NT];
    const int wg = xcd_order(blockIdx.x, gridDim.x);
    cavity_pair<S, COLL, MACRO, PairShape<S>::NT>(a, a.t, wg, buf, [&](auto edge, int i, int j, int k, bool mid) {
        if constexpr (LOOP) return LoopbackHalo<S, !decltype(edge)::value>{a, mid ? a.halo_mid : a.halo_out, i, j, k};
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

// What a turn takes at least, and how its bytes count in the cache (see below).
constexpr PairCost COST_F64{4.3, 1.0, 0.25}, COST_F32{5.5, 1.2, 0.2};
constexpr PairCost COST_F64_LOOP{5.8, 1.2, 0.5}, COST_F32_LOOP{7.2, 1.5, 0.3};  // with the looped-back halo's stores

}  // namespace

namespace lbm {

bool pair_plan(int nx, int ny, int nz, int storage, bool loop, int cus, PairTiles* out) {
    switch (storage) {
    case LBM_STORE_F64: return pair_plan(nx, ny, nz, PairShape<StoreF64>::NT, Q, 8, loop ? COST_F64_LOOP : COST_F64, cus, out);
    case LBM_STORE_F32: return pair_plan(nx, ny, nz, PairShape<StoreF32>::NT, Q, 4, loop ? COST_F32_LOOP : COST_F32, cus, out);
    }
    return false;  // FP16: see below
}

// The tiles, and whether two steps go faster this way.
//
// Time goes by turns (planes) of the busiest CU: with one block per CU a launch
// takes ceil(blocks / CUs) rounds of cz + 2 turns.  A turn takes at least 4.3 us
// in FP64, 5.5 in FP32 (twice the cells), 5.8 and 7.2 with the looped-back halo,
// 5.1 and 5.8 with temperature (medians over 2000 random boxes of 16 to 256 cells a
// side).  Against one step per launch in transforms, which the pair form replaced:
// of 1064 random boxes of 12 to 256 cells planned in pairs or blocks 2 ran below
// 0.97 of its speed (0.94), half at 1.4 and more.  On large boxes a turn is bound
// by memory (256^3 FP64: 622 us a step without the arithmetic and LDS, 627 with
// them) and goes as the bytes it moves, a row of the tile and its rim costing 128
// bytes more per population than it holds (the lines at its ends):
// FP64 32 x 13 tiles 7.3 us, 64 x 5 5.7; FP32 64 x 13 6.9, 32 x 26 8.0, i.e.
// 0.77 ns per such byte with every CU busy, less where fewer are (6.5 us for FP64
// 32 x 13 with 240 of 256), 0.5 ns in the cache.  Rows that are not whole 64-byte
// groups cost 1.1 to 1.4 times that outside the cache.  A one-step launch takes
// 5 us and 5.2 TB/s of its traffic.
// FP16 keeps the one-step kernel: half the bytes, but the rim adds a third to its
// VALU issue, which alone takes 205 us of 241 a step at 256^3 (481 instructions a
// wave; with the collision in pair form, which issues a fifth less, two steps per
// launch took 276 us a step against 238).
namespace {

// Tiles of width tx for an nx x ny plane; false where nt threads cannot hold them.
bool tiles_of_width(int nx, int ny, int nt, int tx, PairTiles* out) {
    PairTiles t{};
    t.tx = tx;
    t.ntx = (nx + tx - 1) / tx;
    t.hx = t.ntx > 1;
    t.w = tx + 2 * t.hx;
    if (t.w > nt) return false;
    const int rows = nt / t.w;
    if (rows >= ny) {
        t.ty = ny;
    } else if (rows >= 3) {
        t.nty = (ny + rows - 3) / (rows - 2);
        t.ty = (ny + t.nty - 1) / t.nty;  // even tiles
    } else {
        return false;
    }
    t.nty = (ny + t.ty - 1) / t.ty;
    t.hy = t.nty > 1;
    t.h = t.ty + 2 * t.hy;
    *out = t;
    return true;
}

template <class F>
void for_widths(int nx, F&& f) {
    for (int tx = 32; tx < nx && tx <= 128; tx += 32) f(tx);
    for (int n = 1; n <= 4; ++n) f((nx + n - 1) / n);
}

// us of a turn (see above); busy: the share of the CUs at work.
double turn_us(const PairTiles& t, double bytes, int pops, PairCost cost, bool cached, double busy) {
    const double moved = t.h * (t.w * bytes + 128.0) + t.tx * t.ty * bytes;
    double turn = (cached ? 5.0e-4 * cost.cached : 7.7e-4) * (pops / 19.0) * moved * (0.5 + 0.5 * busy);
    if (!cached && t.tx % 16 != 0 && t.ntx > 1) turn *= 1.2;
    return std::max(turn, cost.least);
}

// us of a launch of blocks of given times and counts, one block per CU.
double launch_us(std::vector<std::pair<double, long long>> runs, int cus) {
    std::sort(runs.rbegin(), runs.rend());
    std::vector<double> free(cus, 0.0);  // a heap: when each CU is free, the first in front
    double end = 0;
    long long steps = 0;
    for (const auto& r : runs)
        for (long long n = 0; n < r.second; ++n) {
            if (++steps > 16LL * cus) {  // long launches: the mean, and the last blocks
                double rest = r.first * double(r.second - n);
                for (const auto* q = &r + 1; q != runs.data() + runs.size(); ++q) rest += q->first * double(q->second);
                return end + rest / cus;
            }
            std::pop_heap(free.begin(), free.end(), std::greater<double>());
            free.back() += r.first;
            end = std::max(end, free.back());
            std::push_heap(free.begin(), free.end(), std::greater<double>());
        }
    return end;
}

double one_step_us(double cells, double bytes, int pops) { return cells * 2 * pops * bytes / 5.2e6 + 5.0; }
bool in_cache(double cells, double bytes, int pops) { return cells * 2 * pops * bytes < 200e6; }

}  // namespace

bool pair_plan(int nx, int ny, int nz, int nt, int pops, int elem, PairCost cost, int cus, PairTiles* out) {
    const double bytes = elem, cells = double(nx) * ny * nz;
    const bool cached = in_cache(cells, bytes, pops);
    if (((long long)nx + 15) / 16 * 16 * ny * elem >= (long long)PLANE_RANGE) return false;  // the lanes' offsets
    if ((long long)((nx + 63) / 64) * ny * nz <= (long long)cost.held * cus) return false;
    double best = 1e30;
    for_widths(nx, [&](int tx) {
        PairTiles t;
        if (!tiles_of_width(nx, ny, nt, tx, &t)) return;
        for (int ncz = 1; ncz <= nz; ++ncz) {
            t.cz = (nz + ncz - 1) / ncz;
            t.ncz = (nz + t.cz - 1) / t.cz;
            const long long blocks = (long long)t.ntx * t.nty * t.ncz;
            if (blocks > (1 << 24)) break;
            const long long rounds = (blocks + cus - 1) / cus;
            const double turn = turn_us(t, bytes, pops, cost, cached, double(blocks) / double(rounds * cus));
            const double time = (double(rounds) * (t.cz + 2) * turn + 4.0) / 2;
            if (time < best) {
                best = time;
                *out = t;
            }
        }
    });
    // One step per launch: a row's last wave is part empty, which counts where the
    // lattices lie in the cache.  Fitted to 340 random boxes there: per lane, rows a
    // quarter full took 0.5 (FP64) and 0.36 (FP32) of what full ones take, half full
    // ones 0.62 and 0.64.  (As 0.7 of a cell per lane, full or not, boxes of 13 to 32
    // cells along x went in pairs at 0.83 to 0.97 of the one-step kernel's speed.)
    const double idle = double((nx + 63) / 64 * 64 - nx) * ny * nz;
    const double one = one_step_us(cached ? cells + cost.lanes * idle : cells, bytes, pops);
    // (margins for what the model misses)
    return best < (one < 16.0 ? 0.9 : 0.95) * one;
}

bool pair_batch_plan(const std::vector<PairBox>& boxes, int storage, int cus, std::vector<PairTiles>* tiles,
                     std::vector<PairBlock>* blocks) {
    if (storage == LBM_STORE_F16) return false;
    const bool f64 = storage == LBM_STORE_F64;
    const int nt = f64 ? PairShape<StoreF64>::NT : PairShape<StoreF32>::NT;
    const double bytes = f64 ? 8.0 : 4.0;
    double cells = 0;
    for (const PairBox& b : boxes) {
        if (((long long)b.nx + 15) / 16 * 16 * b.ny * (f64 ? 8 : 4) >= (long long)PLANE_RANGE) return false;
        cells += double(b.nx) * b.ny * b.nz;
    }
    const bool cached = in_cache(cells, bytes, Q);
    // each box's tiles in the plane: those whose turns take least together
    std::vector<PairTiles> cand(boxes.size());
    std::vector<double> turn(boxes.size());
    for (size_t m = 0; m < boxes.size(); ++m) {
        double least = 1e30;
        for_widths(boxes[m].nx, [&](int tx) {
            PairTiles t;
            if (!tiles_of_width(boxes[m].nx, boxes[m].ny, nt, tx, &t)) return;
            const double us = turn_us(t, bytes, Q, f64 ? COST_F64 : COST_F32, cached, 1.0);
            if (us * t.ntx * t.nty < least) {
                least = us * t.ntx * t.nty;
                turn[m] = us;
                cand[m] = t;
            }
        });
        if (least > 1e29) return false;
    }
    // Chunks of about one time for all boxes: long ones repeat fewer planes, short
    // ones leave less of the chip idle at the end.  A launch is played through: its
    // blocks go to the CUs in order, the longest first.
    double best = 1e30;
    long long last = 0;
    std::vector<std::pair<double, long long>> runs(boxes.size());  // a block's time, how many
    for (double limit = 1000.0; limit > 10.0; limit *= 0.97) {
        double total = 0;
        long long count = 0;
        for (size_t m = 0; m < boxes.size(); ++m) {
            PairTiles& t = cand[m];
            const int nz = boxes[m].nz;
            const int most = std::min(nz, std::max(1, (int)(limit / turn[m]) - 2));  // planes of a chunk
            t.ncz = (nz + most - 1) / most;
            t.cz = (nz + t.ncz - 1) / t.ncz;
            t.ncz = (nz + t.cz - 1) / t.cz;
            runs[m] = {(t.cz + 2) * turn[m], (long long)t.ntx * t.nty * t.ncz};
            total += runs[m].first * double(runs[m].second);
            count += runs[m].second;
        }
        if (count == last) continue;  // the same chunks as before
        last = count;
        if ((total / cus + 4.0) / 2 >= best) break;
        const double time = (launch_us(runs, cus) + 4.0) / 2;
        if (time < best) {
            best = time;
            *tiles = cand;
        }
    }
    if (best >= 0.95 * one_step_us(cells, bytes, Q)) return false;
    blocks->clear();
    for (size_t m = 0; m < boxes.size(); ++m) {
        const PairTiles& t = (*tiles)[m];
        for (int z = 0; z < t.ncz; ++z)
            for (int y = 0; y < t.nty; ++y)
                for (int x = 0; x < t.ntx; ++x)
                    blocks->push_back({(int)m, x * t.tx - t.hx, y * t.ty - t.hy, z * t.cz});
    }
    // the longest first
    std::stable_sort(blocks->begin(), blocks->end(), [&](const PairBlock& a, const PairBlock& b) {
        return ((*tiles)[a.box].cz + 2) * turn[a.box] > ((*tiles)[b.box].cz + 2) * turn[b.box];
    });
    return true;
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
