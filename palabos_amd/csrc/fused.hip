// palabos_amd: the launches of two fused steps (fused.h) of one storage type and
// one dynamics, compiled once per (PLBAMD_S, PLBAMD_DYN).
#include "engine.h"
#include "fused.h"

#if !defined(PLBAMD_S) || !defined(PLBAMD_DYN)
#error "compile with -DPLBAMD_S=<storage type> -DPLBAMD_DYN=<0 BGK | 1 RBGK>"
#endif

namespace plbamd {

// FP64 and FP32 tiles take 76 KB of LDS, above the default limit per workgroup.
template<typename K>
static int allowLds(K kernel, size_t bytes) {
    if (bytes > 65536)
        PLBAMD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)bytes));
    return PLBAMD_OK;
}

template<typename S, int DYN>
int launchFused(Lattice& L, FusedOp op) {
    const BlockGeom& g = L.geom[0];
    const bool forced = L.dAlpha || L.desc.force[0] != 0 || L.desc.force[1] != 0 || L.desc.force[2] != 0;
    constexpr int threads = fused_threads(sizeof(typename Store<S>::T));
    const size_t lds = 19 * (size_t)threads * sizeof(typename Store<S>::R);
    if (op == FUSED_PREPARE) {
        PLBAMD_TRY(allowLds(fused_two_steps<S, DYN, false, false>, lds));
        PLBAMD_TRY(allowLds(fused_two_steps<S, DYN, false, true>, lds));
        PLBAMD_TRY(allowLds(fused_two_steps<S, DYN, true, false>, lds));
        PLBAMD_TRY(allowLds(fused_two_steps<S, DYN, true, true>, lds));
        if (L.dInfo) {
            const dim3 grid = itemsGrid((uint64_t)g.nx * g.ny * g.nz);
            hipLaunchKernelGGL(fused_info, grid, dim3(256), 0, L.stream, g, L.dTags, L.dWalls, L.dInfo);
            if (L.nSpecial)
                hipLaunchKernelGGL(fused_info_special, itemsGrid(L.nSpecial), dim3(256), 0, L.stream, L.dSpecial,
                                   L.nSpecial, L.dInfo, L.dIndex);
            PLBAMD_HIP(hipGetLastError());
        }
        return PLBAMD_OK;
    }
    if (op == FUSED_BEGIN) {
        if (L.anySolid)
            hipLaunchKernelGGL((fused_solids<S>), itemsGrid(L.cells), dim3(256), 0, L.stream, L.dInfo, L.cells, g.slot,
                               L.arena, L.spare);
        PLBAMD_HIP(hipGetLastError());
        return PLBAMD_OK;
    }
    SpecialArgs s{};
    if (L.nSpecial) {
        s.arena = L.arena; s.blocks = L.dGeom; s.nBlocks = (int)L.geom.size(); s.omega = L.desc.omega;
        for (int c = 0; c < 3; ++c) s.force[c] = L.desc.force[c];
        s.alpha = L.dAlpha;
        s.cells = L.dSpecial; s.count = L.nSpecial; s.values = L.dValues;
        s.pre = L.dPre;
        const dim3 sg((L.nSpecial + kSpecialThreads - 1) / kSpecialThreads);
        if (forced) hipLaunchKernelGGL((special_step<S, DYN, true, false, true>), sg, dim3(kSpecialThreads), 0, L.stream, s);
        else hipLaunchKernelGGL((special_step<S, DYN, true, false, false>), sg, dim3(kSpecialThreads), 0, L.stream, s);
    }
    FusedArgs a{};
    a.src = L.arena;
    a.dst = L.spare;
    a.slot = g.slot;
    a.nx = g.nx; a.ny = g.ny; a.nz = g.nz;
    a.px = g.px; a.py = g.py; a.pz = g.pz;
    a.rows = L.fused.rows; a.cols = L.fused.cols;
    a.tilesY = L.fused.tilesY; a.tilesZ = L.fused.tilesZ;
    a.len = L.fused.len;
    a.omega = L.desc.omega;
    for (int c = 0; c < 3; ++c) a.force[c] = L.desc.force[c];
    a.alpha = L.dAlpha;
    a.info = L.dInfo;
    a.index = L.dIndex;
    a.outputs = L.dPre;
    a.nSpecial = L.nSpecial;
    const dim3 grid((unsigned)(a.tilesY * a.tilesZ * ((g.nx + a.len - 1) / a.len))), block(threads);
    if (L.dInfo) {
        if (forced) hipLaunchKernelGGL((fused_two_steps<S, DYN, true, true>), grid, block, lds, L.stream, a);
        else hipLaunchKernelGGL((fused_two_steps<S, DYN, true, false>), grid, block, lds, L.stream, a);
    } else {
        if (forced) hipLaunchKernelGGL((fused_two_steps<S, DYN, false, true>), grid, block, lds, L.stream, a);
        else hipLaunchKernelGGL((fused_two_steps<S, DYN, false, false>), grid, block, lds, L.stream, a);
    }
    if (L.nSpecial) {
        s.arena = L.spare;
        s.pre = nullptr;
        const dim3 sg((L.nSpecial + kSpecialThreads - 1) / kSpecialThreads);
        if (forced) hipLaunchKernelGGL((special_step<S, DYN, false, false, true>), sg, dim3(kSpecialThreads), 0, L.stream, s);
        else hipLaunchKernelGGL((special_step<S, DYN, false, false, false>), sg, dim3(kSpecialThreads), 0, L.stream, s);
    }
    PLBAMD_HIP(hipGetLastError());
    std::swap(L.arena, L.spare);
    return PLBAMD_OK;
}

template int launchFused<PLBAMD_S, PLBAMD_DYN>(Lattice&, FusedOp);

}  // namespace plbamd
