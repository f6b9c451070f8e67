// Device launcher and registry descriptor for the mixed-batch kernel (multi.hpp).
#pragma once

namespace fx {

template <typename T, int PRESET, bool G17 = true>
long multi_grid(long ntasks)
{
    static const int per = resident_per_cu(k_multi<T, PRESET, G17>, MultiCfg<T, PRESET>::NT);
    return persistent_grid(per, 8, ntasks);
}
template <typename T, int PRESET>
long multi_launch_grid(long ntasks, bool g17)
{
    if constexpr (kMultiSmall<PRESET>)
        if (!g17) return multi_grid<T, PRESET, false>(ntasks);
    return multi_grid<T, PRESET>(ntasks);
}

template <typename T, int PRESET>
hipError_t launch_multi(const void* args, const int2* tasks, int ntasks, const void* bank,
                        unsigned* work, hipStream_t stream)
{
    using M = MultiCfg<T, PRESET>;
    if (ntasks <= 0) return hipSuccess;
    const MultiArgs<T>& a = *(const MultiArgs<T>*)args;
    const bool g17 = !kMultiSmall<PRESET> || multi_has17(a);
    const long grid = multi_launch_grid<T, PRESET>(ntasks, g17);
    auto* k = k_multi<T, PRESET>;
    if constexpr (kMultiSmall<PRESET>)
        if (!g17) k = k_multi<T, PRESET, false>;
    hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(M::NT), 0, stream, a, tasks, ntasks,
                       (const Bank<T>*)bank, claim_counter(work, grid, ntasks));
    return hipGetLastError();
}

template <typename T, int PRESET>
hipError_t launch_multi_dev(const void* d, const void* bank, unsigned* work, int grid,
                            hipStream_t stream)
{
    using M = MultiCfg<T, PRESET>;
    hipLaunchKernelGGL((k_multi_dev<T, PRESET>), dim3((unsigned)grid), dim3(M::NT), 0, stream,
                       (MultiDescriptor<T>*)d, (const Bank<T>*)bank, work);
    return hipGetLastError();
}

template <typename T, int PRESET>
int multi_dev_grid()
{
    using M = MultiCfg<T, PRESET>;
    static const int per = resident_per_cu(k_multi_dev<T, PRESET>, M::NT);
    return (int)persistent_grid(per, 8, 1L << 30);
}

template <typename T, int PRESET>
MultiDesc multi_desc(const char* name, int order = 0)
{
    using M = MultiCfg<T, PRESET>;
    return MultiDesc{prec_of<T>(), PRESET, M::NT,
                     {M::vpw(0), M::vpw(1), M::vpw(2), M::vpw(3), M::vpw(4)},
                     sizeof(cx<T>) * (size_t)M::LDS, name, &launch_multi<T, PRESET>,
                     &launch_multi_dev<T, PRESET>, &multi_dev_grid<T, PRESET>, 0,
                     &multi_launch_grid<T, PRESET>, order};
}

}  // namespace fx
