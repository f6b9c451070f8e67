// Balanced 17^3 kernels (f17.hpp): complex128 at two workgroups per CU, complex64 at four,
// both directions; and the plane-per-workgroup kernels for small batches (plane17.hpp).
#include "f17.hpp"
#include "plane17.hpp"

namespace fx {

#define FX_B(T, TAG, S, DIR, P) \
    r.push_back(f17_desc<F17Cfg<T, S, P>>("bal_17x17x17_" TAG "_" DIR "_v1t256p" #P "_fold"))

void register_f17(std::vector<KernelDesc>& r)
{
    FX_B(double, "c128", -1, "fwd", 2);
    FX_B(double, "c128", +1, "bwd", 2);
    FX_B(double, "c128", -1, "fwd", 1);
    FX_B(double, "c128", +1, "bwd", 1);
    FX_B(float, "c64", -1, "fwd", 4);
    FX_B(float, "c64", +1, "bwd", 4);
    FX_B(float, "c64", -1, "fwd", 2);
    FX_B(float, "c64", +1, "bwd", 2);
    r.push_back(plane17_desc<Plane17Cfg<double, -1>>("plane_17x17x17_c128_fwd_v1t320"));
    r.push_back(plane17_desc<Plane17Cfg<double, +1>>("plane_17x17x17_c128_bwd_v1t320"));
    r.push_back(plane17_desc<Plane17Cfg<float, -1>>("plane_17x17x17_c64_fwd_v1t320"));
    r.push_back(plane17_desc<Plane17Cfg<float, +1>>("plane_17x17x17_c64_bwd_v1t320"));
}

}  // namespace fx
