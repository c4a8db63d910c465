// pair.hpp -- two steps of the isothermal D3Q19 update in one pass over the
// lattice.  Internal to libmglc_lbm.so.
//
// The one-step kernel is bound by its memory traffic: 19 populations read and
// written per cell and step.  Here a block keeps the first step's result on
// the chip: it owns a column of tx x ty cells, walks it along z, and per plane
//   1. computes step 1 on the plane's (tx + 2) x (ty + 2) cells (one per
//      thread, pulled from memory as the one-step kernel does) and leaves the
//      19 stored populations in LDS;
//   2. computes step 2 on the plane below, whose pulls now lie in LDS, and
//      writes it to memory.
// Memory sees one read (and the rim once more) and one write per two steps.
// Step 1 on the rim is computed by both neighbours: (tx + 2)(ty + 2)/(tx ty)
// of its arithmetic.  Every cell goes through the operations of the one-step
// kernel, so the result is the same bit for bit.
//
// LDS holds two planes (the one just written and the one below); what step 2
// pulls from the plane below that (e_z = +1, five values) is read one turn
// earlier into registers.  The next plane's 19 loads are issued before step 2
// of the current one and are in flight behind it and the barriers, which
// order LDS accesses only.
#pragma once
#include <vector>

#include "step.hpp"

namespace lbm {

struct PairTiles {
    int w, h;        // threads along x and y: the tile and its rim
    int tx, ty;      // cells written
    int hx, hy;      // rim width (0 along an axis one tile spans)
    int ntx, nty;    // tiles along x and y
    int cz, ncz;     // planes of a chunk, chunks along z
};

struct PairArgs : StepArgs {
    double* lid_out;   // lid density after the second step (lid_rho: before the first)
    void* halo_mid;    // loopback: the halo the first step writes (halo_out: the second)
    PairTiles t;
};

// Orders LDS accesses over the block; global loads and stores stay in flight.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A plane of a population as a buffer: a scalar base and a 32-bit byte offset
// per lane.  An offset of NOWHERE is out of the buffer's range, so the store is
// dropped by the address unit: the stores need no branch around them, and
// without one the compiler knows how many follow the next plane's loads and
// waits for the loads alone, not for the stores behind them too.
constexpr unsigned PLANE_RANGE = 0x80000000u, NOWHERE = 0xffffffffu;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_of(const void* base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, PLANE_RANGE, 0x00020000);
}

template <class T>
__device__ __forceinline__ T plane_load(__amdgpu_buffer_rsrc_t r, unsigned bytes) {
    if constexpr (sizeof(T) == 8) {
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, bytes, 0, 0));
    } else if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, bytes, 0, 0));
    } else {
        return __builtin_bit_cast(T, (unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r, bytes, 0, 0));
    }
}

template <class T>
__device__ __forceinline__ void plane_store(T v, __amdgpu_buffer_rsrc_t r, unsigned bytes) {
    typedef unsigned uint2_t __attribute__((ext_vector_type(2)));
    if constexpr (sizeof(T) == 8)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2_t, v), r, bytes, 0, 0);
    else if constexpr (sizeof(T) == 4)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, bytes, 0, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), r, bytes, 0, 0);
}

// Block b of n as a position in the tile order such that the blocks one XCD
// receives (every eighth) are neighbours: the rims they share are read through
// one L2.
__device__ __forceinline__ int xcd_order(int b, int n) {
    const int q = n >> 3, r = n & 7, x = b & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

constexpr int up_slot(int al) { return al == 5 ? 0 : (al < 15 ? al - 10 : al - 12); }
static_assert(up_slot(5) == 0 && up_slot(11) == 1 && up_slot(12) == 2 && up_slot(15) == 3 && up_slot(16) == 4,
              "the five velocities with e_z = +1");

// make_post(edge, i, j, k, mid): the hook that sees a cell's stored populations, after the first
// (mid) or the second step.
// EDGE: some cell of the block, rim included, lies on an x or y wall.
template <class S, int COLL, bool MACRO, bool EDGE, int NT, class MakePost>
__device__ __forceinline__ void cavity_pair(const PairArgs& a, const PairTiles& t, int x0, int y0, int zs,
                                            typename S::T (&buf)[2][Q][NT], MakePost&& make_post) {
    using T = typename S::T;
    using R = typename S::Real;
    const T* __restrict__ src = static_cast<const T*>(a.src);
    T* __restrict__ dst = static_cast<T*>(a.dst);
    const int tid = threadIdx.x;
    const int cell = min(tid, t.w * t.h - 1);  // threads past the tile repeat its last cell
    const int lx = cell % t.w, ly = cell / t.w;
    const int i = x0 + lx, j = y0 + ly;
    const bool own = tid < t.w * t.h && lx >= t.hx && lx < t.hx + t.tx && ly >= t.hy && ly < t.hy + t.ty &&
                     i < a.nx && j < a.ny;
    // a thread outside the domain repeats the nearest cell's work; nobody reads
    // its LDS column
    const int ci = min(max(i, 0), a.nx - 1), cj = min(max(j, 0), a.ny - 1);
    const int ze = min(zs + t.cz, a.nz);
    const int lid_idx = ci + a.nx * cj;
    const int cxy = ci + a.px * cj;
    const int nbw = t.w;
    // the LDS column step 2 pulls around (a thread that writes nothing: its own
    // on an edge, where every pull is tested, else any column inside the tile)
    const int col = own || EDGE ? tid : nbw + 1;
    double rho_top = a.lid_rho[lid_idx];  // the top layer's rho before step 1, then after it

    // hides from the compiler that a value is the same in every turn: it would
    // keep addresses made from it in registers
    auto fresh = [](int v) {
        asm volatile("" : "+v"(v));
        return v;
    };
    T in[Q];  // the plane to compute next, as stored
    auto load = [&](int k) {
        const T* s = src + (long long)a.pxy * k;
        const int cl = fresh(cxy);
        sfor<Q>([&](auto A) {
            constexpr int al = decltype(A)::value;
            constexpr int ex = EX[al], ey = EY[al], ez = EZ[al];
            const bool zok = ez == 0 || (ez > 0 ? k > 0 : k < a.nz - 1);
            const long long from = (long long)al * a.ps - (ex + (long long)ey * a.px + (long long)ez * a.pxy);
            const long long bounced = (long long)OPP[al] * a.ps;
            if constexpr (EDGE && (ex != 0 || ey != 0)) {
                bool ok = zok;
                if constexpr (ex != 0) ok = ok && (unsigned)(ci - ex) < (unsigned)a.nx;
                if constexpr (ey != 0) ok = ok && (unsigned)(cj - ey) < (unsigned)a.ny;
                in[al] = s[cl + (ok ? from : bounced)];
            } else {
                in[al] = plane_load<T>(plane_of(s + (zok ? from : bounced)), (unsigned)cl * (unsigned)sizeof(T));
            }
        });
    };
    // the lid's momentum on the two populations that come down along x
    auto lid = [&](R(&f)[Q], double rho) {
        f[13] = lid_bounce<S, COLL>(f[13], rho, a.u_lid, a.scale, true);
        f[14] = lid_bounce<S, COLL>(f[14], rho, a.u_lid, a.scale, false);
    };
    // step 1 on plane p, from `in` into LDS
    auto produce = [&](int p) {
        R f[Q];
        sfor<Q>([&](auto A) {
            constexpr int al = decltype(A)::value;
            f[al] = S::val(in[al]);
        });
        const bool top = p == a.nz - 1;
        if (top) lid(f, rho_top);
        const Moments<R> m = moments<S, COLL>(f, a.inv_scale);
        if (top) rho_top = density_f64<S>(m.sum, a.inv_scale);
        collide<S, COLL>(f, m, a);
        const unsigned h = cell_random<S>(cxy + (long long)a.pxy * p, a.seed);
        T out[Q];
        sfor<Q>([&](auto A) {
            constexpr int al = decltype(A)::value;
            out[al] = S::cvt(f[al], store_random<S, al>(h));
            buf[p & 1][al][tid] = out[al];
        });
        const auto post = make_post(std::bool_constant<EDGE>{}, fresh(i), fresh(j), p, true);
        if (post.active() && own && p >= zs && p < ze) post.store(out);
    };
    // Step 2's pull of population al at plane k: from the neighbour's column in
    // the plane the velocity comes from, or bounced from the cell's own.
    auto pull = [&](auto A, int k, int c) {
        constexpr int al = decltype(A)::value;
        constexpr int ex = EX[al], ey = EY[al], ez = EZ[al];
        const bool zok = ez == 0 || (ez > 0 ? k > 0 : k < a.nz - 1);
        const int plane = ez == 0 ? (k & 1) : ((k + 1) & 1);
        const int from = (plane * Q + al) * NT - (ex + ey * nbw), bounced = ((k & 1) * Q + OPP[al]) * NT;
        const T* b = &buf[0][0][0];
        if constexpr (EDGE && (ex != 0 || ey != 0)) {
            bool ok = zok && own;
            if constexpr (ex != 0) ok = ok && (unsigned)(i - ex) < (unsigned)a.nx;
            if constexpr (ey != 0) ok = ok && (unsigned)(j - ey) < (unsigned)a.ny;
            return S::val(b[c + (ok ? from : bounced)]);
        } else {
            return S::val(b[c + (zok ? from : bounced)]);
        }
    };
    // The pulls along e_z = +1 come out of plane k - 1, whose buffer plane k + 1
    // takes: they are made a turn early.
    R up[5];
    auto take_up = [&](int k) {
        const int c = fresh(col);
        sfor<Q>([&](auto A) {
            constexpr int al = decltype(A)::value;
            if constexpr (EZ[al] > 0) up[up_slot(al)] = pull(A, k, c);
        });
    };
    // step 2 on plane k
    auto finish = [&](int k) {
        R f[Q];
        const bool top = k == a.nz - 1;
        const int c = fresh(col);
        sfor<Q>([&](auto A) {
            constexpr int al = decltype(A)::value;
            if constexpr (EZ[al] > 0) f[al] = up[up_slot(al)];
            else f[al] = pull(A, k, c);
        });
        if (top) lid(f, rho_top);
        const Moments<R> m = moments<S, COLL>(f, a.inv_scale);
        if (top && own) a.lid_out[lid_idx] = density_f64<S>(m.sum, a.inv_scale);
        if constexpr (MACRO) {
            if (own) {
                const long long mc = i + (long long)a.nx * (j + (long long)a.ny * k);
                a.rho[mc] = density_f64<S>(m.sum, a.inv_scale);
                a.u[mc] = double(m.u);
                a.v[mc] = double(m.v);
                a.w[mc] = double(m.w);
            }
        }
        collide<S, COLL>(f, m, a);
        const unsigned h = cell_random<S>(cxy + (long long)a.pxy * k, a.seed + 1u);
        const unsigned where = own ? (unsigned)fresh(cxy) * (unsigned)sizeof(T) : NOWHERE;
        T out[Q];
        T* d = dst + (long long)a.pxy * k;
        sfor<Q>([&](auto A) {
            constexpr int al = decltype(A)::value;
            out[al] = S::cvt(f[al], store_random<S, al>(h));
            plane_store(out[al], plane_of(d + (long long)al * a.ps), where);
        });
        const auto post = make_post(std::bool_constant<EDGE>{}, fresh(i), fresh(j), k, false);
        if (post.active() && own) post.store(out);
    };

    const int p0 = max(zs - 1, 0), p1 = min(ze, a.nz - 1);
    load(p0);
    int p = p0;
    do {  // (at least once, which the compiler has to see: see NOWHERE)
        produce(p);
        load(min(p + 1, p1));
        lds_barrier();
        if (p == zs) take_up(p);
        // as many stores as step 2 makes, all dropped (see NOWHERE)
        sfor<Q>([&](auto A) { plane_store(T(0), plane_of(dst + (long long)decltype(A)::value * a.ps), NOWHERE); });
        lds_barrier();
    } while (++p <= zs);
    for (; p <= p1; ++p) {
        produce(p);
        load(min(p + 1, p1));  // (the last plane once more: the count of loads in flight stays known)
        lds_barrier();
        finish(p - 1);
        take_up(p);
        lds_barrier();
    }
    if (ze == a.nz) finish(a.nz - 1);  // the top chunk's last plane needs none above it
}

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

template <class S, int COLL, bool MACRO, int NT, class MakePost>
__device__ __forceinline__ void cavity_pair_at(const PairArgs& a, const PairTiles& t, int x0, int y0, int zs,
                                               typename S::T (&buf)[2][Q][NT], MakePost&& make_post) {
    if (x0 >= 1 && x0 + t.w <= a.nx - 1 && y0 >= 1 && y0 + t.h <= a.ny - 1)
        cavity_pair<S, COLL, MACRO, false, NT>(a, t, x0, y0, zs, buf, make_post);
    else
        cavity_pair<S, COLL, MACRO, true, NT>(a, t, x0, y0, zs, buf, make_post);
}

template <class S, int COLL, bool MACRO, int NT, class MakePost>
__device__ __forceinline__ void cavity_pair(const PairArgs& a, const PairTiles& t, int wg,
                                            typename S::T (&buf)[2][Q][NT], MakePost&& make_post) {
    const int bx = wg % t.ntx, by = (wg / t.ntx) % t.nty, bz = wg / (t.ntx * t.nty);
    const int x0 = bx * t.tx - t.hx, y0 = by * t.ty - t.hy;
    cavity_pair_at<S, COLL, MACRO, NT>(a, t, x0, y0, bz * t.cz, buf, make_post);
}

// The tiles of the two-step kernel for a box on a device of `cus` CUs; false:
// the one-step kernel is faster.
bool pair_plan(int nx, int ny, int nz, int storage, bool loop, int cus, PairTiles* out);

// The same for a two-step kernel with blocks of nt threads that moves `pops`
// values of `elem` bytes per cell and step each way.
struct PairCost {
    double least;   // us of a turn at least
    double cached;  // times what a turn's bytes take where the lattices lie in the cache
    double lanes;   // what an idle lane of a row's last wave costs the one-step kernel there, as a share of a cell
    int held = 0;   // boxes whose one-step waves, up to this many per CU, all run at once keep that kernel
};
bool pair_plan(int nx, int ny, int nz, int nt, int pops, int elem, PairCost cost, int cus, PairTiles* out);

// Many boxes in one launch: each box's tiles and the flat list of blocks; false:
// the one-step kernel is faster.
struct PairBox {
    int nx, ny, nz;
};
struct PairBlock {
    int box, x0, y0, zs;  // the block's first cell with its rim, and its first plane
};
bool pair_batch_plan(const std::vector<PairBox>& boxes, int storage, int cus, std::vector<PairTiles>* tiles,
                     std::vector<PairBlock>* blocks);

}  // namespace lbm

// Launch the two-step kernel (walls only) for `a` on `stream`.
int lbm_launch_pair(const lbm::PairArgs& a, int storage, int collision, bool macro, bool loop, hipStream_t stream);
