// Two collide-and-stream steps in one pass over memory.
//
// The single-step kernels (kernels.h) read and write every population once per
// step and run at the rate the memory sustains for that (5.1-5.8 TB/s on
// lattices beyond the last-level cache), so the only way to a faster step is
// fewer bytes. fused_two_steps takes the state after an even step (slot opp(i)
// of x holds f*_i(x), the post-collision populations) from one array to the
// state two steps later in a second array: an odd step (gather f_i from x - c_i,
// collide) whose outputs stay on the chip, and the following even step
// (collide in place) on what streamed in from the neighbours.
//
// A workgroup takes a tile of rows x cols cells of the (y, z) plane, one thread
// per cell, and marches along x. The tile's rim (one cell all around) takes the
// first step only: its outputs are what the inner cells need from outside. The
// first step's outputs of one plane x = k go to LDS (19 values per thread, in
// the storage type, as they would have been rounded in memory); the second step
// of plane k - 1 takes the populations with c_x = 0 from that plane's LDS
// content, those with c_x = -1 from plane k's, and those with c_x = +1 from
// plane k - 2's, which waited in registers. Two barriers per plane: one before
// plane k's outputs replace plane k - 1's (by then read), one after.
//
// The arithmetic is the single-step kernels' (collide_bulk on the same values
// in the same order), so the populations are bit-identical to theirs.
//
// Bytes per cell and two steps: 19 values read, plus the rim's share (half of the
// rim misses L2: FP64 256^3 reads 1.24 times its populations), and 19 written (the
// single steps move twice as much). FP64 256^3 runs at 4.7 TB/s of those bytes, FP32
// 5.0: with one workgroup per CU the loads of a plane wait for the plane before.
// 16-bit storage is bound by instructions (57 % of the time in vector ones).
#pragma once

#include "kernels.h"

namespace plbamd {

// Threads of a workgroup: one workgroup per CU takes all its registers. `arith` is
// the size of the arithmetic type. The larger the tile, the smaller the share of its
// rim: two workgroups of 512 threads per CU instead of one of 1024 cost FP32 256^3
// 348 us a step instead of 303, 200^3 185 instead of 148 (FP16 122 instead of 107);
// FP64 has registers for 512 threads only (768 spill: 652 instead of 612).
constexpr int fused_threads(size_t arith) { return arith == 8 ? 512 : 1024; }

// Per-cell word of lattices with edges or tags: bit i (1-18) set where f_i comes
// back from the cell's own f*_opp(i) (a non-periodic edge or a link wall at
// x - c_i), and from bit kFusedKind on what the cell does.
constexpr int kFusedKind = 24;
enum FusedKind : uint32_t { FK_BULK = 0, FK_BOUNCE_BACK = 1, FK_NO_DYNAMICS = 2, FK_SOLID = 3, FK_SPECIAL = 4 };

struct FusedArgs {
    const void* src;          // populations after an even step (swapped layout)
    void* dst;                // the same after two more steps
    uint64_t slot;
    int nx, ny, nz;
    int px, py, pz;
    int rows, cols;           // tile with its rim: rows * cols <= fused_threads
    int tilesY, tilesZ;
    int len;                  // planes along x per workgroup
    double omega;
    double force[3];
    const void* alpha;        // Brinkman porosity per cell, in the arithmetic type, or null
    const uint32_t* info;     // INFO: the per-cell words
    const uint32_t* index;    // INFO: record of every special cell
    const void* outputs;      // INFO: first-step outputs of the special cells, [19][nSpecial], storage type
    uint32_t nSpecial;
};

// One population of a plane (bytes from base): buffer accesses, whose address is
// a scalar base and one 32-bit lane offset. (Flat accesses kept a 64-bit
// address per direction in vector registers: 147 instead of 109 for FP64.)
template<typename S>
__device__ __forceinline__ typename Store<S>::R plane_load(const S* base, uint32_t bytes, uint32_t offset) {
    const auto d = __builtin_amdgcn_make_buffer_rsrc(const_cast<S*>(base), 0, bytes, 0x00027000);
    typename Store<S>::R r;
    if constexpr (sizeof(S) == 8) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(d, offset, 0, 0);
        __builtin_memcpy(&r, &v, 8);
    } else if constexpr (sizeof(S) == 4) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b32(d, offset, 0, 0);
        __builtin_memcpy(&r, &v, 4);
    } else {
        const auto v = __builtin_amdgcn_raw_buffer_load_b16(d, offset, 0, 0);
        __builtin_memcpy(&r, &v, 2);
    }
    return r;
}
template<typename S>
__device__ __forceinline__ void plane_store(S* base, uint32_t bytes, uint32_t offset, typename Store<S>::R r) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    const auto d = __builtin_amdgcn_make_buffer_rsrc(base, 0, bytes, 0x00027000);
    if constexpr (sizeof(S) == 8) {
        u32x2 v;
        __builtin_memcpy(&v, &r, 8);
        __builtin_amdgcn_raw_buffer_store_b64(v, d, offset, 0, 0);
    } else if constexpr (sizeof(S) == 4) {
        uint32_t v;
        __builtin_memcpy(&v, &r, 4);
        __builtin_amdgcn_raw_buffer_store_b32(v, d, offset, 0, 0);
    } else {
        __builtin_amdgcn_raw_buffer_store_b16(r, d, offset, 0, 0);
    }
}

// The collision of a cell by its kind (solid and special cells: nothing here).
template<typename S, int DYN, bool FORCED>
__device__ __forceinline__ void fused_collide(const FusedArgs& a, uint64_t cell, uint32_t kind,
                                              typename Store<S>::T f[19]) {
    using T = typename Store<S>::T;
    if (kind == FK_BULK) {
        const T F[3] = {(T)a.force[0], (T)a.force[1], (T)a.force[2]};
        T rhoBar, drag[3];
        const T alpha = (FORCED && a.alpha) ? reinterpret_cast<const T*>(a.alpha)[cell] : (T)0;
        (void)collide_bulk<T, DYN, FORCED, sizeof(S) == 2>(f, (T)a.omega, F, alpha, rhoBar, drag);
    } else if (kind == FK_BOUNCE_BACK) {
#pragma unroll
        for (int i = 1; i <= 9; ++i) { T t = f[i]; f[i] = f[i + 9]; f[i + 9] = t; }
    }
}

// INFO: the lattice has non-periodic edges or cells that are not background
// dynamics. The special cells (planes, momentum-exchange nodes) take their first
// step in a launch before this one (special_step with `pre`), which leaves their
// outputs in a.outputs; their second step's inputs are written to dst in natural
// layout for the even special_step that follows.
//
// The scheduling barriers keep the LDS reads of plane k - 1 and the gather of
// plane k + 1 where they are written: moved up, they would be live through a
// collision.
template<typename S, int DYN, bool INFO, bool FORCED>
__global__ void __launch_bounds__(fused_threads(sizeof(typename Store<S>::T)))
    __attribute__((amdgpu_waves_per_eu(fused_threads(sizeof(typename Store<S>::T)) / 256))) fused_two_steps(FusedArgs a) {
    using T = typename Store<S>::T;
    constexpr int kThreads = fused_threads(sizeof(T));
    using R = typename Store<S>::R;
    extern __shared__ __align__(16) unsigned char ldsRaw[];
    R* lds = reinterpret_cast<R*>(ldsRaw);     // [19][kThreads]
    const uint32_t wg = xcd_item(blockIdx.x, gridDim.x);
    const uint32_t tiles = (uint32_t)a.tilesY * a.tilesZ;
    const uint32_t chunk = wg / tiles, tile = wg % tiles;
    const int y0 = (int)(tile / (uint32_t)a.tilesZ) * (a.rows - 2), z0 = (int)(tile % (uint32_t)a.tilesZ) * (a.cols - 2);
    const int xa = (int)chunk * a.len, xb = min(a.nx, xa + a.len);
    const int t = (int)threadIdx.x;
    const int r = t / a.cols, c = t - r * a.cols;
    int y = y0 + r - 1, z = z0 + c - 1;
    const bool inner = r >= 1 && r <= a.rows - 2 && c >= 1 && c <= a.cols - 2 && y < a.ny && z < a.nz;
    bool act = r < a.rows && y <= a.ny && z <= a.nz;
    if (y < 0) { act = act && a.py; y += a.ny; }
    if (y == a.ny) { act = act && a.py; y = 0; }
    if (z < 0) { act = act && a.pz; z += a.nz; }
    if (z == a.nz) { act = act && a.pz; z = 0; }
    if (!act) { y = 0; z = 0; }
    const uint64_t plane = (uint64_t)a.ny * a.nz;
    const uint32_t planeBytes = (uint32_t)plane * (uint32_t)sizeof(S);
    uint32_t off[3][3];
    {
        // neighbours beyond a non-periodic edge are replaced by the cell itself:
        // their values are not used (the edge bits of the cell's word)
        int ym = y, yp = y, zm = z, zp = z;
        if (!shift(y, -1, a.ny, a.py, ym)) ym = y;
        if (!shift(y, 1, a.ny, a.py, yp)) yp = y;
        if (!shift(z, -1, a.nz, a.pz, zm)) zm = z;
        if (!shift(z, 1, a.nz, a.pz, zp)) zp = z;
        const int ys[3] = {ym, y, yp}, zs[3] = {zm, z, zp};
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int q = 0; q < 3; ++q) off[p][q] = ((uint32_t)ys[p] * a.nz + zs[q]) * (uint32_t)sizeof(S);
    }
    const uint32_t own = off[1][1];
    const uint32_t ownCell = own / (uint32_t)sizeof(S);
    const S* src = reinterpret_cast<const S*>(a.src);
    S* dst = reinterpret_cast<S*>(a.dst);

    auto infoOf = [&](const uint32_t* words, int k) -> uint32_t {
        int xk = 0;
        if (!INFO || !act || !shift(k, 0, a.nx, a.px, xk)) return 0u;
        return words[(uint64_t)xk * plane + ownCell];
    };
    // first-step inputs of plane k (raw); special cells: their first-step outputs
    R next[19];
    auto gather = [&](int k, uint32_t word, uint32_t rec) {
        int xk = 0;
        if (!(act && shift(k, 0, a.nx, a.px, xk))) return;
        int xm = xk, xp = xk;
        if (!shift(xk, -1, a.nx, a.px, xm)) xm = xk;
        if (!shift(xk, 1, a.nx, a.px, xp)) xp = xk;
        const int xs[3] = {xm, xk, xp};
        const bool special = INFO && (word >> kFusedKind) == FK_SPECIAL;
        if (!INFO || __ballot(special || (word & 0x7ffffu)) == 0) {
#pragma unroll
            for (int i = 0; i < 19; ++i)
                next[i] = plane_load<S>(src + (uint64_t)opp(i) * a.slot + (uint64_t)xs[1 - cx(i)] * plane, planeBytes,
                                        off[1 - cy(i)][1 - cz(i)]);
        } else {
            // a wavefront with reflections: one load per direction all the same, from
            // an offset chosen per lane (slots i and opp(i) are nine slots apart). The
            // lane's offsets are opaque here, so that no sum of them is kept in a
            // register across planes.
            uint32_t o[3][3];
#pragma unroll
            for (int p = 0; p < 3; ++p)
#pragma unroll
                for (int q = 0; q < 3; ++q) { o[p][q] = off[p][q]; asm("" : "+v"(o[p][q])); }
#pragma unroll
            for (int i = 0; i < 19; ++i) {
                const int xs_i = xs[1 - cx(i)], lowX = min(xs_i, xk);
                const S* base = src + (uint64_t)(i < opp(i) ? i : opp(i)) * a.slot + (uint64_t)lowX * plane;
                const uint32_t there = (uint32_t)(((i < opp(i) ? 9 : 0) * a.slot + (uint64_t)(xs_i - lowX) * plane) * sizeof(S));
                const uint32_t back = (uint32_t)(((i > opp(i) ? 9 : 0) * a.slot + (uint64_t)(xk - lowX) * plane) * sizeof(S));
                const uint32_t lane = ((word >> i) & 1u) ? o[1][1] + back : o[1 - cy(i)][1 - cz(i)] + there;
                next[i] = plane_load<S>(base, 0xffffffffu, lane);
            }
            if (special) {
                const R* g = reinterpret_cast<const R*>(a.outputs) + rec;
#pragma unroll
                for (int i = 0; i < 19; ++i) next[i] = g[(uint64_t)i * a.nSpecial];
            }
        }
    };
    R p2[19], refl[19];   // c_x = +1 from plane k - 2; INFO: plane k - 1's own f*_opp(i), c_x(i) = -1
#pragma unroll
    for (int i = 0; i < 19; ++i) { p2[i] = R(); refl[i] = R(); }
    const bool specials = INFO && a.nSpecial != 0;
    uint32_t wordPrev = 0, word = infoOf(a.info, xa - 1), wordNext = infoOf(a.info, xa);
    uint32_t recNext = specials ? infoOf(a.index, xa) : 0u;
    gather(xa - 1, word, specials ? infoOf(a.index, xa - 1) : 0u);
    for (int k = xa - 1; k <= xb; ++k) {
        int xk = 0;
        const bool planeOk = act && shift(k, 0, a.nx, a.px, xk);
        const uint32_t kind = word >> kFusedKind;
        T g[19];
#pragma unroll
        for (int i = 0; i < 19; ++i) g[i] = Store<S>::from_raw(next[i]);
        // plane k + 1 goes out before plane k is collided: its loads are in flight
        // through both collisions and the barriers (issued after the barriers: FP64
        // 128^3 83 us a step, now 77; 256^3 632, now 612)
        __builtin_amdgcn_sched_barrier(0);
        if (k < xb) gather(k + 1, wordNext, recNext);
        __builtin_amdgcn_sched_barrier(0);
        if (planeOk) fused_collide<S, DYN, FORCED>(a, (uint64_t)xk * plane + ownCell, kind, g);
        __builtin_amdgcn_sched_barrier(0);
        // what plane k - 1 (in LDS) sends to its own cells and to plane k
        auto arriving = [&](int i) -> R { return lds[i * kThreads + (t - cy(i) * a.cols - cz(i))]; };
        R p1[19], hold[19];
        if (inner && k >= xa) {
            if (!INFO || __ballot(wordPrev & 0x7ffffu) == 0) {
#pragma unroll
                for (int i = 0; i < 19; ++i) {
                    if (cx(i) > 0) {
                        hold[i] = p2[i];
                        p1[i] = arriving(i);
                    } else if (cx(i) == 0) {
                        hold[i] = arriving(i);
                    }
                }
            } else {
                int here = t;
                asm("" : "+v"(here));
#pragma unroll
                for (int i = 0; i < 19; ++i) {
                    const bool back = (wordPrev >> i) & 1u;
                    if (cx(i) > 0) {
                        const R v = lds[opp(i) * kThreads + here];
                        hold[i] = back ? v : p2[i];
                        p1[i] = lds[i * kThreads + (here - cy(i) * a.cols - cz(i))];
                    } else if (cx(i) == 0) {
                        hold[i] = lds[here + (back ? opp(i) * kThreads
                                                   : i * kThreads - cy(i) * a.cols - cz(i))];
                    } else {
                        refl[i] = lds[opp(i) * kThreads + here];
                    }
                }
            }
        }
        __syncthreads();   // plane k - 1 is read
        if (planeOk) {
#pragma unroll
            for (int i = 0; i < 19; ++i) lds[i * kThreads + t] = Store<S>::to_raw(g[i]);
        }
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t wordAhead = (k + 2 <= xb) ? infoOf(a.info, k + 2) : 0u;
        const uint32_t recAhead = (specials && k + 2 <= xb) ? infoOf(a.index, k + 2) : 0u;
        __builtin_amdgcn_sched_barrier(0);
        if (inner && k >= xa) {
            if (k > xa) {
                // second step of plane k - 1
                const uint64_t base = (uint64_t)(k - 1) * plane;
                const uint32_t kindPrev = wordPrev >> kFusedKind;
                T f[19];
#pragma unroll
                for (int i = 0; i < 19; ++i) {
                    R v;
                    if (cx(i) < 0) {
                        v = arriving(i);
                        if constexpr (INFO) { if ((wordPrev >> i) & 1u) v = refl[i]; }
                    } else {
                        v = hold[i];
                    }
                    f[i] = Store<S>::from_raw(v);
                }
                fused_collide<S, DYN, FORCED>(a, base + ownCell, kindPrev, f);
                if (!INFO || kindPrev <= FK_NO_DYNAMICS) {
#pragma unroll
                    for (int i = 0; i < 19; ++i)
                        plane_store<S>(dst + (uint64_t)opp(i) * a.slot + base, planeBytes, own, Store<S>::to_raw(f[i]));
                } else if (kindPrev == FK_SPECIAL) {
                    // natural layout: the even special_step completes and collides them
#pragma unroll
                    for (int i = 0; i < 19; ++i)
                        plane_store<S>(dst + (uint64_t)i * a.slot + base, planeBytes, own, Store<S>::to_raw(f[i]));
                }
            }
#pragma unroll
            for (int i = 0; i < 19; ++i) if (cx(i) > 0) p2[i] = p1[i];
        }
        wordPrev = word;
        word = wordNext;
        wordNext = wordAhead;
        recNext = recAhead;
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The per-cell words of a lattice from its tags, link masks and edges; then the
// special cells' kinds and record numbers.
static __global__ void __launch_bounds__(256) fused_info(BlockGeom g, const uint8_t* tags, const uint32_t* walls,
                                                         uint32_t* info) {
    const uint64_t cell = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    const uint64_t cells = (uint64_t)g.nx * g.ny * g.nz;
    if (cell >= cells) return;
    const uint32_t plane = (uint32_t)g.ny * (uint32_t)g.nz, cc = (uint32_t)cell;
    const int x = (int)(cc / plane), rem = (int)(cc % plane);
    const int y = rem / g.nz, z = rem % g.nz;
    const uint8_t tag = tags ? tags[cell] : (uint8_t)BT_BULK;
    const uint32_t wall = walls ? walls[cell] : 0u;
    uint32_t m = 0;
#pragma unroll
    for (int i = 1; i < 19; ++i) {
        int sx, sy, sz;
        const bool in = shift(x, -cx(i), g.nx, g.px, sx) && shift(y, -cy(i), g.ny, g.py, sy) && shift(z, -cz(i), g.nz, g.pz, sz);
        if (!in || ((wall >> opp(i)) & 1u)) m |= 1u << i;
    }
    const uint32_t kind = tag == BT_BOUNCE_BACK ? FK_BOUNCE_BACK
                          : tag == BT_NO_DYNAMICS ? FK_NO_DYNAMICS : tag == BT_SKIP ? FK_SOLID : FK_BULK;
    info[cell] = m | (kind << kFusedKind);
}

// Link-wall solids keep their values: copied to the second array once per call.
template<typename S>
__global__ void __launch_bounds__(256) fused_solids(const uint32_t* info, uint64_t cells, uint64_t slot, const void* src,
                                                    void* dst) {
    using R = typename Store<S>::R;
    const uint64_t cell = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (cell >= cells || (info[cell] >> kFusedKind) != FK_SOLID) return;
    const R* s = reinterpret_cast<const R*>(src) + cell;
    R* d = reinterpret_cast<R*>(dst) + cell;
#pragma unroll
    for (int i = 0; i < 19; ++i) d[(uint64_t)i * slot] = s[(uint64_t)i * slot];
}

static __global__ void __launch_bounds__(256) fused_info_special(const SpecialCell* cells, uint32_t count, uint32_t* info,
                                                                 uint32_t* index) {
    const uint32_t k = blockIdx.x * 256u + threadIdx.x;
    if (k >= count) return;
    const uint32_t cell = cells[k].cell;
    info[cell] = (info[cell] & 0x7ffffu) | ((uint32_t)FK_SPECIAL << kFusedKind);
    index[cell] = k;
}

}  // namespace plbamd
