// palabos_amd: the operations of one storage type (PLBAMD_S) other than the
// step: envelope exchange, host transfers, checkpoint files, equilibrium
// initialisation and moments.
#include "engine.h"
#include "external.h"
#include "hostio.h"

#if !defined(PLBAMD_S)
#error "compile with -DPLBAMD_S=<storage type>"
#endif

namespace plbamd {

template<typename S>
int exchange(Lattice& L) {
    if (!L.multi || L.nSegs == 0) return PLBAMD_OK;
    hipLaunchKernelGGL((exchange_envelopes<S>), dim3(L.nTasks), dim3(256), 0, L.stream, L.arena, L.dGeom, L.dSegs,
                       L.dTasks);
    PLBAMD_HIP(hipGetLastError());
    return PLBAMD_OK;
}


// Populations of box b between the lattice and a device buffer of boxCells(b)
// * 19 elements of type elem, C order; launches only (no host copy, no wait).
template<typename S>
hipError_t transferDevice(Lattice& L, const plbamd_box& b, int elem, void* staging, bool up, hipStream_t stream) {
    hipError_t err = hipSuccess;
    for (size_t bi = 0; bi < L.geom.size() && err == hipSuccess; ++bi) {
        BoxArgs a;
        if (!boxArgs(L, bi, b, a)) continue;
        const dim3 grid = gridFor((uint64_t)a.ilx * a.ily * a.ilz), block(256);
        if (up) {
            if (elem == PLBAMD_F64) hipLaunchKernelGGL((upload_box<S, double>), grid, block, 0, stream, L.arena, a, (const double*)staging);
            else if (elem == PLBAMD_F32) hipLaunchKernelGGL((upload_box<S, float>), grid, block, 0, stream, L.arena, a, (const float*)staging);
            else hipLaunchKernelGGL((upload_box_raw<S>), grid, block, 0, stream, L.arena, a, (const uint16_t*)staging);
        } else {
            if (elem == PLBAMD_F64) hipLaunchKernelGGL((download_box<S, double>), grid, block, 0, stream, L.arena, a, (double*)staging);
            else if (elem == PLBAMD_F32) hipLaunchKernelGGL((download_box<S, float>), grid, block, 0, stream, L.arena, a, (float*)staging);
            else hipLaunchKernelGGL((download_box_raw<S>), grid, block, 0, stream, L.arena, a, (uint16_t*)staging);
            err = hipGetLastError();
            if (err == hipSuccess && L.anyWrapped && L.nSpecial) {
                const dim3 g2 = gridFor(L.nSpecial);
                if (elem == PLBAMD_F64)
                    hipLaunchKernelGGL((complete_download<S, double>), g2, block, 0, stream, L.arena, a, L.dValues, (double*)staging, 0);
                else if (elem == PLBAMD_F32)
                    hipLaunchKernelGGL((complete_download<S, float>), g2, block, 0, stream, L.arena, a, L.dValues, (float*)staging, 0);
                else
                    hipLaunchKernelGGL((complete_download<S, float>), g2, block, 0, stream, L.arena, a, L.dValues, (float*)staging, 1);
            }
        }
        if (err == hipSuccess) err = hipGetLastError();
    }
    return err;
}

template<typename S>
int transfer(Lattice& L, const plbamd_box& b, int elem, void* data, size_t bytes, bool up) {
    const uint64_t n = boxCells(b);
    const size_t hostElem = (elem == PLBAMD_F64) ? 8 : (elem == PLBAMD_F32 ? 4 : 2);
    if (bytes != n * 19 * hostElem) return fail(PLBAMD_EINVAL, "transfer: byte count does not match the box");
    if ((elem == PLBAMD_F16 || elem == PLBAMD_BF16) && elem != L.desc.storage)
        return fail(PLBAMD_EINVAL, "transfer: 16-bit host data must match the storage type");
    if (up && L.multi && (L.time & 1))
        return fail(PLBAMD_ESTATE, "upload: a multi-block lattice accepts populations after an even number of steps");
    PLBAMD_TRY(rebuild(L));
    PLBAMD_HIP(hipStreamSynchronize(L.stream));
    const HostPart part{static_cast<char*>(data), 19 * hostElem};
    PLBAMD_TRY(hostTransfer(L, b, &part, 1, up, [&](const plbamd_box& k, void* const* staged, hipStream_t stream) {
        return transferDevice<S>(L, k, elem, staged[0], up, stream);
    }));
    if (up && L.multi) {
        PLBAMD_TRY(exchange<S>(L));
        PLBAMD_HIP(hipStreamSynchronize(L.stream));
    }
    return PLBAMD_OK;
}

// ---------------------------------------------------------------------------
// Palabos checkpoint files (saveBinaryBlock / loadBinaryBlock,
// io/serializerIO_3D.cpp:37-66): the cells are serialized and base64-coded on
// the device; the host writes or reads the text.

template<typename S, typename T>
int checkpointTyped(Lattice& L, const char* path, int elem, bool force, bool enforceUint, bool save) {
    const plbamd_box whole{0, L.desc.nx - 1, 0, L.desc.ny - 1, 0, L.desc.nz - 1};
    const uint64_t cells = boxCells(whole);
    const int recLen = force ? 22 : 19;
    const uint64_t dataBytes = cells * recLen * sizeof(T);
    const uint64_t nChars = (dataBytes + 2) / 3 * 4;
    if (enforceUint && dataBytes > 0xffffffffull)
        return fail(PLBAMD_EINVAL, "binary block: the data does not fit a 32-bit size header (enforce_uint)");
    if (dataBytes / kB64Bytes + 1 > (uint64_t)INT32_MAX * 256)
        return fail(PLBAMD_EINVAL, "binary block: lattice too large for one conversion launch");
    PLBAMD_TRY(rebuild(L));
    DeviceBuffers buf;
    T* pops = static_cast<T*>(buf.get(cells * 19 * sizeof(T)));
    T* rec = force ? static_cast<T*>(buf.get(dataBytes)) : pops;
    char* text = static_cast<char*>(buf.get((nChars + 63) / 64 * 64));
    int* bad = static_cast<int*>(buf.get(2 * sizeof(int)));
    if (!pops || !rec || !text || !bad) return fail(PLBAMD_ENOMEM, "binary block: cannot allocate device buffers");
    const T fx = (T)L.desc.force[0], fy = (T)L.desc.force[1], fz = (T)L.desc.force[2];
    if (save) {
        // cells in no block are zeros, as the reference's forward ordering writes them
        PLBAMD_HIP(hipMemsetAsync(pops, 0, cells * 19 * sizeof(T), L.stream));
        PLBAMD_HIP(transferDevice<S>(L, whole, elem, pops, false, L.stream));
        if (force) hipLaunchKernelGGL((append_force<T>), itemsGrid(cells), dim3(256), 0, L.stream, pops, rec, cells, fx, fy, fz);
        hipLaunchKernelGGL(base64_encode, itemsGrid(dataBytes / kB64Bytes + 1), dim3(256), 0, L.stream,
                           reinterpret_cast<const uint8_t*>(rec), dataBytes, text);
        PLBAMD_HIP(hipGetLastError());
        std::vector<char> host(nChars);
        PLBAMD_HIP(hipMemcpyAsync(host.data(), text, nChars, hipMemcpyDeviceToHost, L.stream));
        PLBAMD_HIP(hipStreamSynchronize(L.stream));
        uint8_t header[8];
        const uint64_t size64 = dataBytes;
        std::memcpy(header, &size64, 8);   // little-endian host
        const std::string head = base64Host(header, enforceUint ? 4 : 8);
        FILE* fp = std::fopen(path, "wb");
        if (!fp) return fail(PLBAMD_EINVAL, std::string("save_binary_block: cannot open ") + path);
        const bool ok = std::fwrite(head.data(), 1, head.size(), fp) == head.size() &&
                        std::fwrite(host.data(), 1, host.size(), fp) == host.size();
        if (std::fclose(fp) != 0 || !ok) return fail(PLBAMD_EINVAL, std::string("save_binary_block: cannot write ") + path);
        return PLBAMD_OK;
    }
    if (L.multi && (L.time & 1))
        return fail(PLBAMD_ESTATE, "load_binary_block: a multi-block lattice accepts populations after an even number of steps");
    std::string file;
    {
        FILE* fp = std::fopen(path, "rb");
        if (!fp) return fail(PLBAMD_EINVAL, std::string("load_binary_block: cannot open ") + path);
        if (std::fseek(fp, 0, SEEK_END) == 0) {
            const long size = std::ftell(fp);
            if (size > 0) file.reserve((size_t)size);
            std::rewind(fp);
        }
        char chunk[1 << 16];
        size_t got;
        while ((got = std::fread(chunk, 1, sizeof(chunk), fp)) > 0) file.append(chunk, got);
        std::fclose(fp);
    }
    // the reference reads with operator>>, which skips white space (every
    // white-space character is at most ' '; every base64 character above it)
    // (the least character, 16 at a time: a search that stops at the first one ran at a
    // byte a cycle or less, whichever way its loop was aligned)
    unsigned char least = 255;
    for (size_t k = 0; k < file.size(); ++k) least = std::min(least, (unsigned char)file[k]);
    if (least <= ' ')
        file.erase(std::remove_if(file.begin(), file.end(), [](char c) { return std::isspace((unsigned char)c) != 0; }),
                   file.end());
    const size_t headChars = enforceUint ? 8 : 12;
    if (file.size() < headChars) return fail(PLBAMD_EINVAL, "load_binary_block: file shorter than its size header");
    uint8_t header[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (!unbase64Host(file.data(), enforceUint ? 4 : 8, header))
        return fail(PLBAMD_EINVAL, "load_binary_block: the size header is not base64");
    uint64_t size64 = 0;
    std::memcpy(&size64, header, 8);
    if (size64 != dataBytes)
        return fail(PLBAMD_EINVAL, "load_binary_block: the file holds " + std::to_string(size64) +
                                       " bytes of cells, this lattice takes " + std::to_string(dataBytes));
    if (file.size() - headChars < nChars) return fail(PLBAMD_EINVAL, "load_binary_block: the file is truncated");
    PLBAMD_HIP(hipMemsetAsync(bad, 0, 2 * sizeof(int), L.stream));
    PLBAMD_HIP(hipMemcpyAsync(text, file.data() + headChars, nChars, hipMemcpyHostToDevice, L.stream));
    hipLaunchKernelGGL(base64_decode, itemsGrid(dataBytes / kB64Bytes + 1), dim3(256), 0, L.stream, text, dataBytes,
                       reinterpret_cast<uint8_t*>(rec), bad);
    if (force) hipLaunchKernelGGL((split_force<T>), itemsGrid(cells), dim3(256), 0, L.stream, rec, pops, cells, fx, fy, fz, bad + 1);
    PLBAMD_HIP(hipGetLastError());
    int flags[2] = {0, 0};
    PLBAMD_HIP(hipMemcpyAsync(flags, bad, sizeof(flags), hipMemcpyDeviceToHost, L.stream));
    PLBAMD_HIP(hipStreamSynchronize(L.stream));
    if (flags[0]) return fail(PLBAMD_EINVAL, "load_binary_block: the cell data is not base64");
    if (flags[1]) return fail(PLBAMD_EINVAL, "load_binary_block: the force externals differ from the lattice's force");
    PLBAMD_HIP(transferDevice<S>(L, whole, elem, pops, true, L.stream));
    PLBAMD_TRY(exchange<S>(L));
    PLBAMD_HIP(hipStreamSynchronize(L.stream));
    return PLBAMD_OK;
}

template<typename S>
int checkpoint(Lattice& L, const char* path, int elem, bool force, bool enforceUint, bool save) {
    if (elem == PLBAMD_F64) return checkpointTyped<S, double>(L, path, elem, force, enforceUint, save);
    return checkpointTyped<S, float>(L, path, elem, force, enforceUint, save);
}

template<typename S>
int equilibrium(Lattice& L, const plbamd_box& b, const double* rho, const double* u) {
    if (L.multi && (L.time & 1))
        return fail(PLBAMD_ESTATE, "initialize_at_equilibrium: a multi-block lattice accepts populations after an even number of steps");
    PLBAMD_TRY(rebuild(L));
    PLBAMD_HIP(hipStreamSynchronize(L.stream));
    const HostPart parts[2] = {{reinterpret_cast<char*>(const_cast<double*>(rho)), 8},
                               {reinterpret_cast<char*>(const_cast<double*>(u)), 24}};
    PLBAMD_TRY(hostTransfer(L, b, parts, 2, true, [&](const plbamd_box& k, void* const* staged, hipStream_t stream) {
        for (size_t bi = 0; bi < L.geom.size(); ++bi) {
            BoxArgs a;
            if (!boxArgs(L, bi, k, a)) continue;
            hipLaunchKernelGGL((equilibrium_box<S>), gridFor((uint64_t)a.ilx * a.ily * a.ilz), dim3(256), 0, stream,
                               L.arena, a, (const double*)staged[0], (const double*)staged[1]);
        }
        return hipGetLastError();
    }));
    if (L.multi) {
        PLBAMD_TRY(exchange<S>(L));
        PLBAMD_HIP(hipStreamSynchronize(L.stream));
    }
    return PLBAMD_OK;
}

template<typename S>
int moments(Lattice& L, const plbamd_box& b, double* rho, double* u, double* sums, double* fields,
            const MomentsScratch* scratch) {
    if (scratch) {
        if (rho || u || fields) return fail(PLBAMD_EINVAL, "moments: a fixed scratch takes the sums only");
        if (L.dirty)
            return fail(PLBAMD_ESTATE, "reduce_moments_noalloc: the lattice's tags, planes or porosity changed since "
                                       "its last step; run a step or plbamd_reduce_moments first");
    } else {
        PLBAMD_TRY(rebuild(L));
    }
    const bool planes = L.nSpecial > 0 && L.dValues != nullptr;
    MomentsArgs m{};
    m.tags = L.dTags;
    m.values = L.dValues;
    for (int c = 0; c < 3; ++c) m.force[c] = L.desc.force[c];
    m.forced = L.desc.force[0] != 0 || L.desc.force[1] != 0 || L.desc.force[2] != 0;
    for (int k = 0; k < 3; ++k) m.solidRho[k] = L.solidRho[k];
    if (!sums) {
        // per-cell values only, straight into the host's chunks
        PLBAMD_HIP(hipStreamSynchronize(L.stream));
        const HostPart parts[3] = {{reinterpret_cast<char*>(rho), 8}, {reinterpret_cast<char*>(u), 24},
                                   {reinterpret_cast<char*>(fields), 56}};
        return hostTransfer(L, b, parts, 3, false, [&](const plbamd_box& k, void* const* staged, hipStream_t stream) {
            MomentsArgs mk = m;
            mk.fields = (double*)staged[2];
            for (size_t bi = 0; bi < L.geom.size(); ++bi) {
                BoxArgs a;
                if (!boxArgs(L, bi, k, a)) continue;
                const dim3 grid = gridFor((uint64_t)a.ilx * a.ily * a.ilz);
                if (a.parity)
                    hipLaunchKernelGGL((moments_box<S, 1>), grid, dim3(256), 0, stream, L.arena, a, mk, (double*)staged[0],
                                       (double*)staged[1], (double*)nullptr);
                else
                    hipLaunchKernelGGL((moments_box<S, 0>), grid, dim3(256), 0, stream, L.arena, a, mk, (double*)staged[0],
                                       (double*)staged[1], (double*)nullptr);
                if (planes)
                    hipLaunchKernelGGL((moments_planes<S>), gridFor(L.nSpecial), dim3(256), 0, stream, L.arena, a, mk,
                                       (double*)staged[0], (double*)staged[1], (double*)nullptr);
            }
            return hipGetLastError();
        });
    }
    uint64_t nRecords = 0;
    for (size_t bi = 0; bi < L.geom.size(); ++bi) {
        BoxArgs a;
        if (!boxArgs(L, bi, b, a)) continue;
        nRecords += gridFor((uint64_t)a.ilx * a.ily * a.ilz).x;
        if (planes) nRecords += gridFor(L.nSpecial).x;
    }
    // records reduced in two levels when there are many: kMomentsLevel1 workgroups, then one
    const uint32_t level1 = nRecords > 4096 ? kMomentsLevel1 : 0u;
    double* d = nullptr;
    double *dPart, *dLevel1;
    if (scratch) {
        if (nRecords > scratch->maxRecords)
            return fail(PLBAMD_EINVAL, "reduce_moments_noalloc: the box needs " + std::to_string(nRecords) +
                                           " partial records, the fixed scratch holds " +
                                           std::to_string(scratch->maxRecords));
        dPart = scratch->base;
        dLevel1 = dPart + 8 * scratch->maxRecords;
    } else {
        PLBAMD_HIP(deviceAlloc((void**)&d, (nRecords * 8 + 8 * level1 + 8) * sizeof(double)));
        dPart = d;
        dLevel1 = dPart + nRecords * 8;
    }
    double* const none = nullptr;
    double* dSum = dLevel1 + 8 * (scratch ? kMomentsLevel1 : level1);
    hipError_t err = hipSuccess;
    uint64_t rec = 0;
    for (size_t bi = 0; bi < L.geom.size(); ++bi) {
        BoxArgs a;
        if (!boxArgs(L, bi, b, a)) continue;
        const dim3 grid = gridFor((uint64_t)a.ilx * a.ily * a.ilz);
        if (a.parity)
            hipLaunchKernelGGL((moments_box<S, 1>), grid, dim3(256), 0, L.stream, L.arena, a, m, none, none, dPart + rec * 8);
        else
            hipLaunchKernelGGL((moments_box<S, 0>), grid, dim3(256), 0, L.stream, L.arena, a, m, none, none, dPart + rec * 8);
        rec += grid.x;
        err = hipGetLastError();
        if (err != hipSuccess) break;
        if (planes) {
            const dim3 pg = gridFor(L.nSpecial);
            hipLaunchKernelGGL((moments_planes<S>), pg, dim3(256), 0, L.stream, L.arena, a, m, none, none, dPart + rec * 8);
            rec += pg.x;
            err = hipGetLastError();
            if (err != hipSuccess) break;
        }
    }
    if (err == hipSuccess) {
        if (level1) {
            hipLaunchKernelGGL(sum_records, dim3(level1), dim3(256), 0, L.stream, dPart, (uint32_t)nRecords, dLevel1);
            hipLaunchKernelGGL(sum_records, dim3(1), dim3(256), 0, L.stream, dLevel1, level1, dSum);
        } else {
            hipLaunchKernelGGL(sum_records, dim3(1), dim3(256), 0, L.stream, dPart, (uint32_t)nRecords, dSum);
        }
        err = hipGetLastError();
    }
    double host[8];
    if (err == hipSuccess) err = hipMemcpyAsync(host, dSum, sizeof(host), hipMemcpyDeviceToHost, L.stream);
    if (err == hipSuccess) err = hipStreamSynchronize(L.stream);
    if (d) hipFree(d);
    if (err != hipSuccess) return fail(PLBAMD_EHIP, std::string("moments: ") + hipGetErrorString(err));
    sums[0] = host[0];  // sum of rhoBar
    sums[1] = host[1];  // sum of |u|^2
    sums[2] = host[3];  // sum of u
    sums[3] = host[4];
    sums[4] = host[5];
    return PLBAMD_OK;
}


template<typename S>
int launchProcessors(Lattice& L, int parity) {
    if (!L.dProc) return PLBAMD_OK;
    ProcArgs a{};
    a.arena = L.arena;
    a.blocks = L.dGeom;
    a.values = L.dValues;
    a.cells = L.dProc;
    a.parity = parity;
    a.omega = L.desc.omega;
    for (int ph = 0; ph < 4; ++ph) {
        a.begin = L.procPhase[ph];
        a.end = L.procPhase[ph + 1];
        if (a.end == a.begin) continue;
        hipLaunchKernelGGL((boundary_processors<S>), dim3((a.end - a.begin + kProcRecords - 1) / kProcRecords),
                           dim3(256), 0, L.stream, a);
        PLBAMD_HIP(hipGetLastError());
    }
    return PLBAMD_OK;
}

// The external-moment field of a single-block lattice: op 0 fills it on box b
// from the populations (BoxRhoBarJfunctional3D), 1 copies its values on b to the
// host, 2 sets them from the host. Allocated on first use, [4][allocCells].
template<typename S>
int externalField(Lattice& L, const plbamd_box& b, double* rhoBar, double* j, int op) {
    using T = typename Store<S>::T;
    PLBAMD_TRY(rebuild(L));
    if (!L.dExtField) {
        PLBAMD_HIP(deviceAlloc(&L.dExtField, 4 * L.allocCells * sizeof(T)));
        PLBAMD_HIP(hipMemsetAsync(L.dExtField, 0, 4 * L.allocCells * sizeof(T), L.stream));
    }
    T* field = static_cast<T*>(L.dExtField);
    BoxArgs a;
    if (!boxArgs(L, 0, b, a)) return fail(PLBAMD_EINVAL, "rhobar_j: box outside the lattice");
    const dim3 grid = gridFor((uint64_t)a.ilx * a.ily * a.ilz);
    if (op == 0) {
        if (a.parity)
            hipLaunchKernelGGL((rhobar_j_box<S, 1>), grid, dim3(256), 0, L.stream, L.arena, a, L.dTags,
                               L.solidRho[0], field, L.allocCells);
        else
            hipLaunchKernelGGL((rhobar_j_box<S, 0>), grid, dim3(256), 0, L.stream, L.arena, a, L.dTags,
                               L.solidRho[0], field, L.allocCells);
        PLBAMD_HIP(hipGetLastError());
        PLBAMD_HIP(hipStreamSynchronize(L.stream));
        return PLBAMD_OK;
    }
    PLBAMD_HIP(hipStreamSynchronize(L.stream));
    const HostPart parts[2] = {{reinterpret_cast<char*>(rhoBar), 8}, {reinterpret_cast<char*>(j), 24}};
    return hostTransfer(L, b, parts, 2, op == 2, [&](const plbamd_box& k, void* const* staged, hipStream_t stream) {
        BoxArgs c;
        (void)boxArgs(L, 0, k, c);
        const dim3 g = gridFor((uint64_t)c.ilx * c.ily * c.ilz);
        if (op == 1)
            hipLaunchKernelGGL((field_get<T>), g, dim3(256), 0, stream, c, (const T*)field, L.allocCells,
                               (double*)staged[0], (double*)staged[1]);
        else
            hipLaunchKernelGGL((field_set<T>), g, dim3(256), 0, stream, c, field, L.allocCells,
                               (const double*)staged[0], (const double*)staged[1]);
        return hipGetLastError();
    });
}

// nsteps ExternalRhoJcollideAndStream3D steps with the field as it is.
template<typename S>
int externalSteps(Lattice& L, int nsteps) {
    using T = typename Store<S>::T;
    PLBAMD_TRY(rebuild(L));
    if (!L.dExtField) return fail(PLBAMD_ESTATE, "external_collide_and_stream: no rhoBar / j field (compute or set it first)");
    const BlockGeom& g = L.geom[0];
    const dim3 grid = itemsGrid((uint64_t)g.nx * g.ny * g.nz);
    const T* field = static_cast<const T*>(L.dExtField);
    const bool rbgk = L.desc.dynamics == PLBAMD_RBGK;
    for (int s = 0; s < nsteps; ++s) {
        const bool odd = (L.time & 1) != 0;
        if (rbgk) {
            if (odd) hipLaunchKernelGGL((external_step<S, 1, true>), grid, dim3(256), 0, L.stream, L.arena, g, L.dTags, field, L.desc.omega);
            else hipLaunchKernelGGL((external_step<S, 1, false>), grid, dim3(256), 0, L.stream, L.arena, g, L.dTags, field, L.desc.omega);
        } else {
            if (odd) hipLaunchKernelGGL((external_step<S, 0, true>), grid, dim3(256), 0, L.stream, L.arena, g, L.dTags, field, L.desc.omega);
            else hipLaunchKernelGGL((external_step<S, 0, false>), grid, dim3(256), 0, L.stream, L.arena, g, L.dTags, field, L.desc.omega);
        }
        PLBAMD_HIP(hipGetLastError());
        ++L.time;
    }
    L.statsValid = false;
    PLBAMD_HIP(hipStreamSynchronize(L.stream));
    return PLBAMD_OK;
}

template int externalField<PLBAMD_S>(Lattice&, const plbamd_box&, double*, double*, int);
template int externalSteps<PLBAMD_S>(Lattice&, int);
template int launchProcessors<PLBAMD_S>(Lattice&, int);
template int exchange<PLBAMD_S>(Lattice&);
template hipError_t transferDevice<PLBAMD_S>(Lattice&, const plbamd_box&, int, void*, bool, hipStream_t);
template int transfer<PLBAMD_S>(Lattice&, const plbamd_box&, int, void*, size_t, bool);
template int checkpoint<PLBAMD_S>(Lattice&, const char*, int, bool, bool, bool);
template int equilibrium<PLBAMD_S>(Lattice&, const plbamd_box&, const double*, const double*);
template int moments<PLBAMD_S>(Lattice&, const plbamd_box&, double*, double*, double*, double*,
                                const MomentsScratch*);

}  // namespace plbamd
