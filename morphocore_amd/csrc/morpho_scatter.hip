// Backward of dilation / erosion by scattering into LDS, for gfx950: a workgroup owns a tile of
// grad_input and reads every output pixel whose winning tap can lie in it (the tile and a halo of the
// element's size), adding those that do to a double copy of the tile in LDS. Each grad_input pixel is
// then written once: no zero fill, no global atomics, no rounding pass, and outputs near a tile's edge
// are read by the two to four workgroups that may own their tap. An LDS double add takes ~9 cycles per
// wave, ~3 times that with the bank conflicts of scattered taps (a global double atomic ~35 ps per add
// over the whole chip), and its cost does not grow with the element, unlike a gather's comparison per
// tap of the window.
//   packed_tile_kernel  MAX / MIN: all the input channels of a tile (in groups of at most 64), from the
//                       packed winners; grad_input only (morpho_bwd_packed_kernel sums grad_weight).
//   ident_tile_kernel   IDENTITY: one channel of a tile, from the taps; grad_input and the tile's share of
//                       grad_weight. Float64 3x3 / 5x5 stays with the gathers, whose sums are in tap
//                       order (n float32 terms add exactly in double, in any order, while their
//                       magnitudes span at most 2^(29 - log2 n)).
// Measured (us, before -> after): max / min bfloat16 3x3 at (16, 64 -> 64, 57, 57), fill + scatter + round
// 145 -> 33 (grad_weight 13, tiles 20); float32 11x11 at (2, 64 -> 64, 256, 256), two scatters of 171 and
// 362 -> 123 each; identity float32 5x5 at (8, 32, 179, 250), tiled gather 72 -> 35; at (32, 128, 112, 112)
// with both reductions, row-band gather 3x3 158 -> 134, 5x5 339 -> 133 (bfloat16 168 -> 132, 338 -> 132).
#include <algorithm>

#include "launch.hpp"

namespace mca
{

// ------------------------------------------------------------------------------------------------
// MAX / MIN
// ------------------------------------------------------------------------------------------------

template <typename ST>
struct PackedTileParams
{
    const int32_t* __restrict__ idx;
    const ST* __restrict__ gout;
    ST* __restrict__ gin;
    Geom g;
    PackedTiles t;
    unsigned kw_magic;  // ceil(2^32 / KW): __umulhi(k, kw_magic) = k / KW for k < 2^16
};

// Division of n < 2^16 by d through the high half of a product with ceil(2^32 / d) (exact there; d == 1
// has no such 32-bit factor).
static unsigned div_magic(int d) { return d == 1 ? 0u : (unsigned)(((uint64_t(1) << 32) + d - 1) / d); }
__device__ __forceinline__ int div_by(int n, unsigned magic) { return magic ? (int)__umulhi((unsigned)n, magic) : n; }

template <typename T, typename ST, int THREADS>
__global__ __launch_bounds__(THREADS) void packed_tile_kernel(const PackedTileParams<ST> p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    Acc* acc = reinterpret_cast<Acc*>(smem_raw);
    const Geom& g = p.g;
    const PackedTiles& t = p.t;
    int work = xcd_work_index(blockIdx.x, gridDim.x);
    const int cgi = work % t.ncg;  // the groups of a tile share its winners in L2
    work /= t.ncg;
    const int tx = work % t.ntx;
    work /= t.ntx;
    const int ty = work % t.nty;
    const int b = work / t.nty;
    const int c0 = cgi * t.cg, nc = min(t.cg, g.Cin - c0);
    const int x0 = tx * t.tw, y0 = ty * t.th;
    const int cols = min(t.tw, g.W - x0), rows = min(t.th, g.H - y0);
    const int px = t.tw * t.th;
    for (int j = threadIdx.x; j < nc * px; j += THREADS) acc[j] = Acc(0);
    __syncthreads();

    // Output pixels (h, w) whose tap (kh, kw) reads (h + KH/2 - kh, w + KW/2 - kw) in the tile.
    const int ph = g.pad_h(), pw = g.pad_w();
    const int h_lo = max(y0 - ph, 0), h_hi = min(y0 + rows - ph + g.KH - 1, g.H);
    const int w_lo = max(x0 - pw, 0), w_hi = min(x0 + cols - pw + g.KW - 1, g.W);
    const int rcols = w_hi - w_lo, n = (h_hi - h_lo) * rcols;
    // Regions smaller than the workgroup are shared by several threads a pixel, each with every
    // `slices`-th output channel.
    const int slices = max(1, min(THREADS / max(n, 1), g.Cout));
    const int64_t plane = g.plane();
    const int32_t* __restrict__ idx = p.idx + (int64_t)b * g.Cout * plane;
    const ST* __restrict__ gout = p.gout + (int64_t)b * g.Cout * plane;
    for (int i = threadIdx.x; i < n * slices; i += THREADS)
    {
        const int s = i / n, pix = i - s * n;
        const int r = pix / rcols;
        const int h = h_lo + r, w = w_lo + pix - r * rcols;
        const int64_t at = (int64_t)h * g.W + w;
        const int dy = h + ph - y0, dx = w + pw - x0;
        constexpr int U = 4;  // output channels whose loads are in flight together
        for (int o = s; o < g.Cout; o += U * slices)
        {
            int pk[U];
            T gv[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                const int64_t q = (int64_t)min(o + u * slices, g.Cout - 1) * plane + at;
                pk[u] = idx[q];
                gv[u] = (T)gout[q];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                const int c = (int)((unsigned)pk[u] >> 16) - c0, k = pk[u] & 0xffff;
                const int kh = div_by(k, p.kw_magic);
                const int iy = dy - kh, ix = dx - (k - kh * g.KW);
                if ((unsigned)c < (unsigned)nc && (unsigned)iy < (unsigned)rows && (unsigned)ix < (unsigned)cols && o + u * slices < g.Cout)
                    lds_add(&acc[c * px + iy * t.tw + ix], (Acc)gv[u]);
            }
        }
    }
    __syncthreads();
    const int tile = rows * cols;
    for (int j = threadIdx.x; j < nc * tile; j += THREADS)
    {
        const int c = j / tile, pix = j - c * tile;
        const int r = pix / cols, col = pix - r * cols;
        p.gin[((int64_t)b * g.Cin + c0 + c) * plane + (int64_t)(y0 + r) * g.W + x0 + col] = (ST)(T)acc[c * px + r * t.tw + col];
    }
}

// Tiles about 32 columns wide (a 128-byte row of winners) and as many rows as the LDS budget holds of
// cg channels: 64 KiB (two workgroups of 512 threads per CU), 128 KiB (one of 1024) where that would
// leave fewer than 256 pixels, so that the halo stays small. Halved while fewer than 512 workgroups
// would run.
PackedTiles packed_tiles(const Geom& g)
{
    PackedTiles t{};
    if (g.Cin < 1 || g.H < 1 || g.W < 1 || g.taps() > 0xffff) return t;
    t.ncg = (g.Cin + 63) / 64;
    t.cg = (g.Cin + t.ncg - 1) / t.ncg;
    int64_t budget = 64 * 1024;
    t.threads = 512;
    if (budget / (int64_t)sizeof(Acc) / t.cg < 256)
    {
        budget = 128 * 1024;
        t.threads = 1024;
    }
    int px = (int)std::min<int64_t>(budget / (int64_t)sizeof(Acc) / t.cg, 4096);
    for (;; px /= 2)
    {
        const int want_w = px >= 1024 ? 64 : 32;
        t.ntx = (g.W + want_w - 1) / want_w;
        t.tw = (g.W + t.ntx - 1) / t.ntx;
        t.th = std::max(1, std::min(px / t.tw, g.H));
        t.nty = (g.H + t.th - 1) / t.th;
        t.th = (g.H + t.nty - 1) / t.nty;
        t.blocks = (int64_t)g.B * t.nty * t.ntx * t.ncg;
        if (t.blocks >= 512 || px <= 128) break;
    }
    t.lds = (size_t)t.cg * t.tw * t.th * sizeof(Acc);
    // What the halo and the channel groups multiply the reads by: up to 16 times is less than the
    // global atomics cost; elements far larger than a tile keep those.
    const int64_t region = (int64_t)std::min(t.th + g.KH - 1, g.H) * std::min(t.tw + g.KW - 1, g.W);
    t.ok = region * t.ncg <= 16 * (int64_t)t.th * t.tw && region < 65536 && t.lds <= device_lds_limit() && t.blocks <= 0x7fffffff;
    return t;
}

template <typename T, typename ST>
hipError_t packed_tile_backward(const int32_t* idx, const ST* grad_out, ST* grad_in, const Geom& g, hipStream_t stream)
{
    PackedTileParams<ST> p{};
    p.idx = idx;
    p.gout = grad_out;
    p.gin = grad_in;
    p.g = g;
    p.t = packed_tiles(g);
    p.kw_magic = div_magic(g.KW);
    if (!p.t.ok) return hipErrorInvalidValue;
    const auto kernel = p.t.threads == 512 ? packed_tile_kernel<T, ST, 512> : packed_tile_kernel<T, ST, 1024>;
    kernel<<<(unsigned)p.t.blocks, p.t.threads, p.t.lds, stream>>>(p);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// IDENTITY
// ------------------------------------------------------------------------------------------------

template <typename T, typename ST>
struct IdentTileParams
{
    const void* __restrict__ taps;
    const ST* __restrict__ gout;
    ST* __restrict__ gin;
    T* __restrict__ part;  // [B * tiles][C][K]
    Geom g;
    IdentTiles t;
    unsigned kw_magic;
};

template <int OP, typename T, typename ST, typename AT, int THREADS>
__global__ __launch_bounds__(THREADS) void ident_tile_kernel(const IdentTileParams<T, ST> p)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const Geom& g = p.g;
    const IdentTiles& t = p.t;
    const int K = g.KH * g.KW;
    Acc* acc = reinterpret_cast<Acc*>(smem_raw);
    Acc* bins = acc + t.tw * t.th;
    int work = xcd_work_index(blockIdx.x, gridDim.x);
    const int tile = work % (t.ntx * t.nty);  // a channel's tiles share their halo in L2
    work /= t.ntx * t.nty;
    const int c = work % g.Cin;
    const int b = work / g.Cin;
    const int ty = tile / t.ntx, tx = tile - ty * t.ntx;
    const int x0 = tx * t.tw, y0 = ty * t.th;
    const int cols = min(t.tw, g.W - x0), rows = min(t.th, g.H - y0);
    const int ncopy = 1 << t.ncopy_log2;
    for (int j = threadIdx.x; j < t.tw * t.th + K * ncopy; j += THREADS) acc[j] = Acc(0);
    const int ph = g.pad_h(), pw = g.pad_w();
    const int h_lo = max(y0 - ph, 0), h_hi = min(y0 + rows - ph + g.KH - 1, g.H);
    const int w_lo = max(x0 - pw, 0), w_hi = min(x0 + cols - pw + g.KW - 1, g.W);
    const int rcols = w_hi - w_lo, n = (h_hi - h_lo) * rcols;
    const unsigned rmagic = rcols == 1 ? 0u : (unsigned)(((uint64_t(1) << 32) + rcols - 1) / rcols);
    const int64_t base = ((int64_t)b * g.Cin + c) * g.plane();
    const ST* __restrict__ gout = p.gout + base;
    const AT* __restrict__ taps = static_cast<const AT*>(p.taps) + base;
    Acc* bl = bins + (threadIdx.x & (ncopy - 1));
    __syncthreads();

    constexpr int U = 8;  // pixels whose loads are in flight together
    for (int i0 = threadIdx.x; i0 < n; i0 += U * THREADS)
    {
        int at[U], k[U], dy[U], dx[U];
        T gv[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            const int i = min(i0 + u * THREADS, n - 1);
            const int r = div_by(i, rmagic);
            const int h = h_lo + r, w = w_lo + i - r * rcols;
            at[u] = h * g.W + w;
            dy[u] = h - y0;
            dx[u] = w - x0;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            gv[u] = (T)gout[at[u]];
            k[u] = (int)taps[at[u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            if (i0 + u * THREADS >= n) break;
            const int kh = div_by(k[u], p.kw_magic);
            const int iy = dy[u] + ph - kh, ix = dx[u] + pw - (k[u] - kh * g.KW);
            const Acc v = (Acc)gv[u];
            if ((unsigned)iy < (unsigned)rows && (unsigned)ix < (unsigned)cols) lds_add(&acc[iy * t.tw + ix], v);
            // grad_weight: each output pixel belongs to the tile that holds its own position.
            if ((unsigned)dy[u] < (unsigned)rows && (unsigned)dx[u] < (unsigned)cols)
                lds_add(&bl[k[u] << t.ncopy_log2], OP == DILATION ? v : -v);
        }
    }
    __syncthreads();
    const unsigned cmagic = cols == 1 ? 0u : (unsigned)(((uint64_t(1) << 32) + cols - 1) / cols);
    ST* __restrict__ gin = p.gin + base + (int64_t)y0 * g.W + x0;
    for (int j = threadIdx.x; j < rows * cols; j += THREADS)
    {
        const int r = div_by(j, cmagic), col = j - r * cols;
        gin[r * g.W + col] = (ST)(T)acc[r * t.tw + col];
    }
    T* __restrict__ part = p.part + (((int64_t)b * t.ntx * t.nty + tile) * g.Cin + c) * K;
    for (int j = threadIdx.x; j < K; j += THREADS)
    {
        Acc s = Acc(0);
        for (int q = 0; q < ncopy; ++q) s += bins[(j << t.ncopy_log2) + ((q + j) & (ncopy - 1))];
        part[j] = (T)s;
    }
}

// Tiles of up to 4096 pixels (32 KiB) and 256 columns, balanced over the plane; halved in height while
// fewer than 1024 workgroups would run and the halo rows stay fewer than the tile's, but, from 256
// workgroups (one per CU) on, not past 32 partial slots: with up to 512 the backward was 2% slower (60 random
// shapes, from 0.73 to 1.46 times the time).
IdentTiles ident_tiles(const Geom& g)
{
    IdentTiles t{};
    if (g.Cin < 1 || g.H < 1 || g.W < 1 || g.taps() > 0xffff || g.plane() > 0x7fffffff) return t;
    t.ntx = (g.W + 255) / 256;
    t.tw = (g.W + t.ntx - 1) / t.ntx;
    for (int th = std::max(1, std::min(4096 / t.tw, g.H));; th /= 2)
    {
        t.nty = (g.H + th - 1) / th;
        t.th = (g.H + t.nty - 1) / t.nty;
        const int64_t blocks = (int64_t)g.B * g.Cin * t.nty * t.ntx;
        const bool few_slots = blocks < 256 || (int64_t)g.B * t.ntx * ((g.H + th / 2 - 1) / std::max(th / 2, 1)) <= REDUCE_GROUP;
        if (blocks >= 1024 || th / 2 < std::max(g.KH - 1, 4) || !few_slots) break;
    }
    // Copies of every grad_weight bin, one per lane of a half wave while they take at most 16 KiB.
    for (t.ncopy_log2 = 5; t.ncopy_log2 > 0 && ((size_t)g.taps() << t.ncopy_log2) * sizeof(Acc) > 16 * 1024; --t.ncopy_log2) {}
    t.lds = ((size_t)t.tw * t.th + ((size_t)g.taps() << t.ncopy_log2)) * sizeof(Acc);
    const int64_t region = (int64_t)std::min(t.th + g.KH - 1, g.H) * std::min(t.tw + g.KW - 1, g.W);
    t.ok = t.lds <= LDS_LIMIT && region < 65536 && region <= 8 * (int64_t)t.tw * t.th &&
           (int64_t)g.B * g.Cin * t.nty * t.ntx <= 0x7fffffff;
    return t;
}

// Pixels up to which one wave takes a tile: backward of 3x3 at (2114, 10 -> 10, 3, 8) 24 us, 62 by four waves.
constexpr int IDENT_WAVE_TILE = 256;

template <typename T, typename ST>
hipError_t ident_tile_backward(int op, const IdentTiles& tiles, const void* taps, const ST* grad_out, ST* grad_in, T* part, const Geom& g,
                               hipStream_t stream)
{
    IdentTileParams<T, ST> p{};
    p.taps = taps;
    p.gout = grad_out;
    p.gin = grad_in;
    p.part = part;
    p.g = g;
    p.t = tiles;
    p.kw_magic = div_magic(g.KW);
    const int64_t blocks = (int64_t)g.B * g.Cin * tiles.nty * tiles.ntx;
    if (!tiles.ok || blocks > 0x7fffffff) return hipErrorInvalidValue;
    const bool wide = pair_tap_bytes(g) == 2;
    // Tiles of a few hundred pixels (small planes) by one wave each: four waves would mostly wait for one another.
    const bool small = tiles.tw * tiles.th <= IDENT_WAVE_TILE;
    auto launch = [&](auto kernel, int threads) { kernel<<<(unsigned)blocks, threads, p.t.lds, stream>>>(p); };
    auto sized = [&](auto one, auto four) { small ? launch(one, WAVE) : launch(four, BLOCK); };
    if (op == DILATION)
        wide ? sized(ident_tile_kernel<DILATION, T, ST, uint16_t, WAVE>, ident_tile_kernel<DILATION, T, ST, uint16_t, BLOCK>)
             : sized(ident_tile_kernel<DILATION, T, ST, uint8_t, WAVE>, ident_tile_kernel<DILATION, T, ST, uint8_t, BLOCK>);
    else
        wide ? sized(ident_tile_kernel<EROSION, T, ST, uint16_t, WAVE>, ident_tile_kernel<EROSION, T, ST, uint16_t, BLOCK>)
             : sized(ident_tile_kernel<EROSION, T, ST, uint8_t, WAVE>, ident_tile_kernel<EROSION, T, ST, uint8_t, BLOCK>);
    return hipGetLastError();
}

template hipError_t packed_tile_backward<float, float>(const int32_t*, const float*, float*, const Geom&, hipStream_t);
template hipError_t packed_tile_backward<double, double>(const int32_t*, const double*, double*, const Geom&, hipStream_t);
template hipError_t packed_tile_backward<float, _Float16>(const int32_t*, const _Float16*, _Float16*, const Geom&, hipStream_t);
template hipError_t packed_tile_backward<float, __bf16>(const int32_t*, const __bf16*, __bf16*, const Geom&, hipStream_t);
template hipError_t ident_tile_backward<float, float>(int, const IdentTiles&, const void*, const float*, float*, float*, const Geom&, hipStream_t);
template hipError_t ident_tile_backward<double, double>(int, const IdentTiles&, const void*, const double*, double*, double*, const Geom&, hipStream_t);
template hipError_t ident_tile_backward<float, _Float16>(int, const IdentTiles&, const void*, const _Float16*, _Float16*, float*, const Geom&, hipStream_t);
template hipError_t ident_tile_backward<float, __bf16>(int, const IdentTiles&, const void*, const __bf16*, __bf16*, float*, const Geom&, hipStream_t);

}  // namespace mca
