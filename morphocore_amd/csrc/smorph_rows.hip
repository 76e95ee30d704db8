// Smorph forward for launches with few workgroups (small planes, few output channels) and for narrow planes,
// gfx950: square 3x3 to 11x11 elements, float32 and float64. The other forwards give a workgroup four rows of
// a 64-column tile and walk the input channels one after the other, since a sum over channels is rounded
// in channel order; a small problem then runs one wave per SIMD or less, each waiting on its own chain of
// exponentials. Here the four waves of a workgroup take four input channels of the same 64 pixels, each
// staging its own channel's tile, and exchange W and 1 / S through LDS, which every wave merges in channel
// order: four times the workgroups for the same work and the same roundings. The 64 pixels are rows of up
// to 64 columns, or two or more shorter rows where the plane is narrow, whose lanes the other forwards leave
// idle. Bound by the exponentials' latency at these sizes.
// Measured (us, before -> after): float64 5x5 at (2, 8 -> 8, 64, 60) 60 -> 24; float32, saving statistics, 11x11 at
// (1, 51 -> 51, 32, 28) 432 -> 266 and 7x7 at (4, 56 -> 6, 48, 34) 219 -> 110.
#include <algorithm>

#include "smorph_common.hpp"

namespace mca
{

template <typename T>
struct RowsParams
{
    SmorphFwdParams<T> f;
    int tw, rpw;  // columns and rows of a wave's pixels (tw * rpw <= 64)
    int ntx, nty;
    unsigned tw_magic, cols_magic;  // ceil(2^32 / tw), ceil(2^32 / (tw + KS - 1))
};

template <typename T, int MK, int KS, bool SAVE>
__global__ __launch_bounds__(BLOCK) void smorph_fwd_rows(const RowsParams<T> q)
{
#pragma clang fp contract(off)  // fused only where the reference fuses (written as fma)
    // A wave's tile has (rpw + KS - 1) rows of (tw + KS - 1) columns: most for one row of 64.
    constexpr int ELEMS = KS * (WAVE + KS - 1), NS = (ELEMS + WAVE - 1) / WAVE;
    __shared__ T tiles[NWAVES][NS * WAVE];
    // The wave's element, read at the same address by every lane (scalar loads share the LDS reads' wait
    // counter, and a scalar operand halves an instruction's rate).
    constexpr int K = KS * KS, NW = (K + WAVE - 1) / WAVE;
    __shared__ __align__(16) T wts[NWAVES][NW * WAVE];
    __shared__ T xw[NWAVES][WAVE], xi[NWAVES][WAVE];
    const SmorphFwdParams<T>& p = q.f;
    const Geom& g = p.g;
    const int lane = threadIdx.x & (WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    int work = xcd_work_index(blockIdx.x, gridDim.x);
    const int o = work % g.Cout;
    work /= g.Cout;
    const int tx = work % q.ntx;
    work /= q.ntx;
    const int ty = work % q.nty;
    const int b = work / q.nty;
    const int h0 = ty * q.rpw, w0 = tx * q.tw;
    constexpr int P = KS / 2;
    const int y0 = h0 + P - (KS - 1), x0 = w0 + P - (KS - 1);
    const int cols = q.tw + KS - 1, rows = q.rpw + KS - 1, nelem = rows * cols;
    const bool inside = y0 >= 0 && x0 >= 0 && y0 + rows <= g.H && x0 + cols <= g.W;
    // This lane's pixel (lanes past the last row compute the first one's and store nothing).
    const int lr = (int)__umulhi((unsigned)lane, q.tw_magic), lc = lane - lr * q.tw;
    const int row = lr < q.rpw ? lr : 0;
    const int h = h0 + row, wc = w0 + lc;
    const bool in = lr < q.rpw && h < g.H && wc < g.W;
    const int64_t plane = g.plane();
    const int64_t pix = (int64_t)h * g.W + wc;

    // Staging plan: the clamped in-image offset of each element this lane stages, and whether 0 replaces it.
    int off[NS];
    unsigned outside = 0;
#pragma unroll
    for (int j = 0; j < NS; ++j)
    {
        const int idx = min(lane + j * WAVE, nelem - 1);
        const int ly = (int)__umulhi((unsigned)idx, q.cols_magic), lx = idx - ly * cols;
        const int y = y0 + ly, x = x0 + lx;
        off[j] = clampi(y, 0, g.H - 1) * g.W + clampi(x, 0, g.W - 1);
        if (y < 0 || y >= g.H || x < 0 || x >= g.W) outside |= 1u << j;
    }
    T pre[NS], wpre[NW], apre;
    auto load = [&](int i) {
        i = min(i, g.Cin - 1);
        const T* __restrict__ xp = p.x + ((int64_t)b * g.Cin + i) * plane;
#pragma unroll
        for (int j = 0; j < NS; ++j) pre[j] = xp[off[j]];
        const T* __restrict__ wg = p.w + ((int64_t)o * g.Cin + i) * K;
#pragma unroll
        for (int j = 0; j < NW; ++j) wpre[j] = wg[min(lane + j * WAVE, K - 1)];
        apre = p.alpha[o * g.Cin + i];
    };
    T* tile = tiles[wave];
    const T* tbase = tile + (row + KS - 1) * cols + lc + KS - 1;
    T m = MK == MK_MAX ? lowest_of<T>() : (MK == MK_MIN ? max_of<T>() : T(0));
    load(wave);
    for (int i0 = 0; i0 < g.Cin; i0 += NWAVES)
    {
        // The wave's own tile: its reads of the previous channel are done (the barrier below).
#pragma unroll
        for (int j = 0; j < NS; ++j) tile[lane + j * WAVE] = (outside >> j) & 1 ? T(0) : pre[j];
#pragma unroll
        for (int j = 0; j < NW; ++j) wts[wave][lane + j * WAVE] = wpre[j];
        const T a = apre;
        load(i0 + NWAVES + wave);  // in flight while this channel computes
        const int i = min(i0 + wave, g.Cin - 1);  // (a wave past the last channel repeats it, unused)
        const int pair = o * g.Cin + i;
        const T* wp = wts[wave];
        T ref[1], S[1], Wsum[1];
        // The wave's lanes read what its other lanes staged: in order for the compiler too (no instruction waits).
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (inside)
            smorph_pair_stats<T, 1, KS, false>(tbase, cols, nullptr, wp, a, g, h + P, wc + P, ref, S, Wsum);
        else
            smorph_pair_stats<T, 1, KS, true>(tbase, cols, nullptr, wp, a, g, h + P, wc + P, ref, S, Wsum);
        const T inv = T(1) / S[0];
        if (in && i0 + wave < g.Cin)
        {
            const int64_t at = ((int64_t)b * g.Cout * g.Cin + pair) * plane + pix;
            if constexpr (SAVE)
            {
                p.pstats[at] = (float)ref[0];
                p.pstats[p.nstat + at] = (float)inv;
                p.pstats[2 * p.nstat + at] = (float)(Wsum[0] * inv);
            }
            if constexpr (MK == MK_SMOOTH && !SAVE) p.pout[at] = Wsum[0] * inv;
        }
        if constexpr (MK != MK_SMOOTH)
        {
            xw[wave][lane] = Wsum[0];
            xi[wave][lane] = inv;
            __syncthreads();
            const int n = min(NWAVES, g.Cin - i0);
            for (int v = 0; v < n; ++v)
            {
                const T wv = xw[v][lane], iv = xi[v][lane];
                if constexpr (MK == MK_SUM)
                {
                    m = fma(wv, iv, m);
                }
                else
                {
                    const T c = wv * iv;
                    if constexpr (MK == MK_MAX)
                        m = m < c ? c : m;
                    else
                        m = c < m ? c : m;
                }
            }
        }
        __syncthreads();
    }
    if constexpr (MK == MK_SMOOTH) return;  // merged by smorph_soft_merge_kernel
    if (wave != 0 || !in) return;
    if constexpr (MK == MK_SUM)
    {
        if (p.average) m = m / (T)g.Cin;
    }
    p.out[((int64_t)b * g.Cout + o) * plane + pix] = m;
}

// Columns and rows of a wave's pixels (from 16 to 64 columns): the shape that takes the fewest waves, the
// widest on a tie.
struct RowsTile
{
    int tw, rpw, ntx, nty;
};

static RowsTile rows_tile(const Geom& g)
{
    RowsTile t{};
    for (int ntx = std::max(1, (g.W + TILE_W - 1) / TILE_W); ntx <= std::max(1, (g.W + 15) / 16); ++ntx)
    {
        const int tw = std::max((g.W + ntx - 1) / ntx, 16), rpw = WAVE / tw;
        const int nty = (g.H + rpw - 1) / rpw;
        if (t.tw > 0 && (int64_t)ntx * nty >= (int64_t)t.ntx * t.nty) continue;
        t = {tw, rpw, ntx, nty};
    }
    return t;
}

// This kernel's work in waves (64 pixels of every input channel; a count of channels that is no multiple of
// four leaves waves idle) against that of the others. Us here | there, at waves here / there:
// float32 of the static sizes runs about 1.6 times as long per wave once the chip is full. 5x5: 15 | 20 at
// 1024 / 1024, 30 | 36 at 1280 / 1280, 24 | 20 at 2048 / 2048, 231 | 310 at 7168 / 14336, 86 | 89 at
// 4864 / 7168; 11x11: 52 | 66, 141 | 135, 96 | 72, 1183 | 1268 and 419 | 362. Two input channels: 8 | 7 and 25 | 19
// at 1280 / 640.
// The unrolled generic kernels (float64, float32 9x9) are as fast per wave: float64 7x7 46 | 75 at
// 1024 / 1024, 439 | 438 at 6144 / 6144, 582 | 563 at 8192 / 8192, 913 | 1043 at 14336 / 16384; with channels to
// spare 26 | 30 at 1365 / 1024, 46 | 49 at 1638 / 1024, 26 | 21 at 1920 / 960, 65 | 51 at 4096 / 3072.
template <typename T>
bool smorph_rows_supported(int mk, const Geom& g)
{
    if (mk == MK_IDENT || g.Cin < 2 || g.KH != g.KW || g.KH < 3 || g.KH > 11 || g.KH % 2 == 0 || g.plane() > 0x7fffffff) return false;
    const RowsTile t = rows_tile(g);
    const int64_t planes = (int64_t)g.B * g.Cout;
    const int64_t here = planes * t.ntx * t.nty * ((g.Cin + NWAVES - 1) / NWAVES * NWAVES) / g.Cin;
    const int64_t there = planes * ((g.W + TILE_W - 1) / TILE_W) * ((g.H + NWAVES - 1) / NWAVES) * NWAVES;
    if (smorph_static_supported<T>(g)) return g.Cin >= NWAVES && (here <= 1280 || 2 * here <= there);
    return here <= 1664 || (here <= 6144 && here <= there) || 10 * here <= 9 * there;
}

template <typename T, int MK, int KS>
static hipError_t rows_launch(const RowsParams<T>& q, unsigned blocks, hipStream_t stream)
{
    if constexpr (sizeof(T) == 4)
        if (q.f.pstats)
        {
            smorph_fwd_rows<T, MK, KS, true><<<blocks, BLOCK, 0, stream>>>(q);
            return hipGetLastError();
        }
    smorph_fwd_rows<T, MK, KS, false><<<blocks, BLOCK, 0, stream>>>(q);
    return hipGetLastError();
}

template <typename T, int MK>
static hipError_t rows_size(const RowsParams<T>& q, unsigned blocks, hipStream_t stream)
{
    switch (q.f.g.KH)
    {
        case 3: return rows_launch<T, MK, 3>(q, blocks, stream);
        case 5: return rows_launch<T, MK, 5>(q, blocks, stream);
        case 7: return rows_launch<T, MK, 7>(q, blocks, stream);
        case 9: return rows_launch<T, MK, 9>(q, blocks, stream);
        default: return rows_launch<T, MK, 11>(q, blocks, stream);
    }
}

template <typename T>
hipError_t launch_smorph_fwd_rows(int mk, const SmorphFwdParams<T>& p, hipStream_t stream)
{
    RowsParams<T> q{};
    q.f = p;
    const Geom& g = p.g;
    const RowsTile t = rows_tile(g);
    q.tw = t.tw;
    q.rpw = t.rpw;
    q.ntx = t.ntx;
    q.nty = t.nty;
    const int cols = q.tw + g.KW - 1;
    q.tw_magic = (unsigned)(((uint64_t(1) << 32) + q.tw - 1) / q.tw);
    q.cols_magic = (unsigned)(((uint64_t(1) << 32) + cols - 1) / cols);
    const unsigned blocks = (unsigned)((int64_t)g.B * q.nty * q.ntx * g.Cout);
    switch (mk)
    {
        case MK_SUM: return rows_size<T, MK_SUM>(q, blocks, stream);
        case MK_MAX: return rows_size<T, MK_MAX>(q, blocks, stream);
        case MK_MIN: return rows_size<T, MK_MIN>(q, blocks, stream);
        case MK_SMOOTH: return rows_size<T, MK_SMOOTH>(q, blocks, stream);
        default: return hipErrorInvalidValue;
    }
}

template bool smorph_rows_supported<float>(int, const Geom&);
template bool smorph_rows_supported<double>(int, const Geom&);
template hipError_t launch_smorph_fwd_rows<float>(int, const SmorphFwdParams<float>&, hipStream_t);
template hipError_t launch_smorph_fwd_rows<double>(int, const SmorphFwdParams<double>&, hipStream_t);

}  // namespace mca
