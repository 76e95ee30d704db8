// Dilation / erosion forward for gfx950: the entry of every storage type, over the kernel instances of
// morpho_fwd.hpp (one source per operation and storage type, so that they compile in parallel).
#include "morpho_fwd.hpp"

namespace mca
{

#define MCA_DECLARE_FWD(ST)                                                                 \
    extern template hipError_t forward_op<ST, DILATION>(int, FwdParams<ST>, hipStream_t); \
    extern template hipError_t forward_op<ST, EROSION>(int, FwdParams<ST>, hipStream_t);
MCA_DECLARE_FWD(float)
MCA_DECLARE_FWD(double)
MCA_DECLARE_FWD(_Float16)
MCA_DECLARE_FWD(__bf16)

template <typename ST>
hipError_t morpho_forward(int op, int merge, bool replicate, compute_t<ST> fill, const ST* x, const ST* w, ST* out, void* indices,
                          const Geom& g, hipStream_t stream)
{
    if ((int64_t)g.B * g.Cout * g.plane() == 0) return hipSuccess;
    if (g.Cin == 0 && merge != MERGE_IDENTITY)
    {
        const int64_t n = (int64_t)g.B * g.Cout * g.plane();
        hipError_t err = fill_async<ST>(out, n, empty_merge_value<ST>(merge), stream);
        if (err == hipSuccess && indices && packed_winners(merge)) err = fill_async<int32_t>(static_cast<int32_t*>(indices), n, 0, stream);
        return err;
    }
    FwdParams<ST> p{};
    p.x = x;
    p.w = w;
    p.out = out;
    p.idx = indices;
    p.g = g;
    p.replicate = replicate ? 1 : 0;
    p.fill = fill;
    p.average = 0;
    return op == DILATION ? forward_op<ST, DILATION>(merge, p, stream) : forward_op<ST, EROSION>(merge, p, stream);
}

#define MCA_INSTANTIATE_ENTRY(ST)                                                                                                      \
    template hipError_t morpho_forward<ST>(int, int, bool, compute_t<ST>, const ST*, const ST*, ST*, void*, const Geom&, hipStream_t); \
    template size_t morpho_forward_lds<ST>(const Geom&);
MCA_INSTANTIATE_ENTRY(float)
MCA_INSTANTIATE_ENTRY(double)
MCA_INSTANTIATE_ENTRY(_Float16)
MCA_INSTANTIATE_ENTRY(__bf16)

}  // namespace mca
