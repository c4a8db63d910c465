// block.hip -- launches of the block kernel (block.hpp) for one cavity.
#include <hip/hip_runtime.h>

#include "block.hpp"
#include "context.hpp"

using namespace lbm;

namespace {

constexpr int NT = 512;  // threads of a workgroup (= cells it holds)

template <class S, int COLL, bool MACRO, bool LOOP>
__global__ __launch_bounds__(NT) void k_cavity_block(const BlockArgs a) {
    __shared__ typename S::T buf[Q][NT];
    cavity_block<S, COLL, MACRO, NT>(a, a.b, blockIdx.x, buf, [&](int i, int j, int k, int step) {
        if constexpr (LOOP) return LoopbackHalo<S>{a, a.halo[(step + 1) & 1], i, j, k};
        else return NoPost{};
    });
}

using BlockFn = void (*)(const BlockArgs);

template <class S>
struct BlockTable {
    // step[collision][macro][loop]
    static constexpr BlockFn step[2][2][2] = {
        {{k_cavity_block<S, COLL_MRT, false, false>, k_cavity_block<S, COLL_MRT, false, true>},
         {k_cavity_block<S, COLL_MRT, true, false>, k_cavity_block<S, COLL_MRT, true, true>}},
        {{k_cavity_block<S, COLL_BGK, false, false>, k_cavity_block<S, COLL_BGK, false, true>},
         {k_cavity_block<S, COLL_BGK, true, false>, k_cavity_block<S, COLL_BGK, true, true>}}};
};

}  // namespace

namespace lbm {

// The blocks: as many steps per launch as still leave no CU more than one
// workgroup (three, else two), in as few workgroups as hold the box.  Measured on
// MI355X, us per step, one-step launches against blocks of 6 x 3 x 3 with three
// steps at 17^3 (108 workgroups) and of 6 x 5 x 7 with two at 33^3 (210): FP64 5.0 /
// 2.9 and 6.8 / 5.1, FP32 4.0 / 2.5 and 5.2 / 4.7, FP16 5.7 / 3.0 and 6.5 / 5.2.
// Four steps at 17^3 (729 workgroups of 2^3) 6.0, two at 51^3 (729 of 6^3) FP64
// 12.6 against 13.7, FP32 9.8 against 7.7: past one workgroup a CU the repeated
// rim costs what it saves.  Two steps only where the one-step kernel's waves, 64
// cells of a row each, are a third empty or more: 128 x 16 x 16 took 4.9 us in
// blocks, 4.6 without; in FP32 two fifths or more: at 0.6 to 0.65 full, eight
// random boxes took 0.96 to 1.22 of the blocks' time (83 x 15 x 25: 4.7 and 4.9 us).
bool block_plan(int nx, int ny, int nz, int storage, int cus, BlockTiles* out) {
    const int n[3] = {nx, ny, nz};
    // (a box this large cannot be covered; it also bounds the search)
    if ((long long)nx * ny * nz > (long long)cus * NT) return false;
    for (int steps = 3; steps >= 2; --steps) {
        if (steps == 2 && nx > (storage == LBM_STORE_F32 ? 0.6 : 2.0 / 3.0) * 64 * ((nx + 63) / 64)) return false;
        long long best = cus + 1;
        // parts along each axis; a part is the written cells of a workgroup
        for (int nbz = 1; nbz <= nz && nbz <= cus; ++nbz)
            for (int nby = 1; nby <= ny && nby * nbz <= cus; ++nby)
                for (int nbx = 1; nbx <= nx && nbx * nby * nbz <= cus; ++nbx) {
                    const int nb[3] = {nbx, nby, nbz};
                    BlockTiles b{};
                    b.steps = steps;
                    long long cells = 1, count = 1;
                    for (int d = 0; d < 3; ++d) {
                        b.t[d] = (n[d] + nb[d] - 1) / nb[d];
                        b.n[d] = (n[d] + b.t[d] - 1) / b.t[d];
                        b.h[d] = b.n[d] > 1 ? steps - 1 : 0;
                        b.w[d] = b.t[d] + 2 * b.h[d];
                        cells *= b.w[d];
                        count *= b.n[d];
                    }
                    // (rows of fewer than 8 cells load too little per line: 3 x 3 x 6 took
                    // 3.2 us at 17^3, 4 x 4 x 3 3.0)
                    if (cells <= NT && count < best && (b.w[0] >= 8 || b.n[0] == 1)) {
                        best = count;
                        *out = b;
                    }
                }
        if (best <= cus) return true;
    }
    return false;
}

}  // namespace lbm

int lbm_launch_block(const BlockArgs& a, int storage, int collision, bool macro, bool loop, hipStream_t stream) {
    const int coll = collision == LBM_BGK ? COLL_BGK : COLL_MRT;
    BlockFn fn;
    switch (storage) {
    case LBM_STORE_F32: fn = BlockTable<StoreF32>::step[coll][macro][loop]; break;
    case LBM_STORE_F16: fn = BlockTable<StoreF16>::step[coll][macro][loop]; break;
    default: fn = BlockTable<StoreF64>::step[coll][macro][loop];
    }
    hipLaunchKernelGGL(fn, dim3((unsigned)(a.b.n[0] * a.b.n[1] * a.b.n[2])), dim3(NT), 0, stream, a);
    return lbm_check_launch();
}
