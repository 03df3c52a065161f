// tall_kernels.hip -- transforms of 648 to 4096 points along a strided dimension (the columns of an
// image or of a spectrum) over interleaved arrays, one pass over memory.
//
// The tile kernel of fast_core.h keeps at most 17 values a thread and 512 threads a workgroup, so
// from 641 points on its column tiles get narrower than 64 bytes, and most lengths took the two
// passes of a split instead.  Here a workgroup has up to 1024 threads of up to 128 registers and a
// tile of 64 bytes of neighbouring columns (32 bytes beyond 2400 points, where 160 KB of LDS end).
// Values go straight from global memory to registers and back; LDS serves the exchanges between
// the radix passes.  What bounds it is memory: neighbouring tiles complete one another's 128-byte
// lines in the L2 of one XCD (tile_decode's ranges).  Up to 1200 points two workgroups share a compute
// unit, so that one loads while the other computes, for 129 of 149 kernels; the other 20 have more
// than 512 threads of more registers than that leaves them, and lose when they are held to those
// (1190 points x 20000 columns 137 us, held to 80 registers 194 us, the passes before 161 us).
// Single precision, arrays that stay in the last-level cache: 960 points x 15000 columns 105 -> 55 us
// (4.2 TB/s), among other calls 119 -> 77 us; 1080 x 15000 120 -> 68; 2048 x 60000 976 -> 617.  Double,
// 960 x 25000: 418 -> 219 us; 2400 x 25000 1073 -> 604.  Whole 128-byte tiles (16 columns, one workgroup
// a compute unit) were slower on arrays in that cache: 960 x 15000 62 us.  Lines are read and written
// once (1 to 4 % more than needed) with 64-byte runs; with 32-byte runs 26 % more are written, and
// 4096 x 4096 x 8 takes 0.735 ms, a plain copy of its shape 0.737 ms.
#include "fast_core.h"
#include "tall_registry.h"
#include "gpu_rt.h"
#include "lds_limit.h"
#include <hip/hip_runtime.h>
#include <algorithm>
#include <mutex>
#include <vector>

#ifndef TALL_SLICE
#error "compile with -DTALL_SLICE=<n>"
#endif

namespace
{

// schedule of a column kernel: the members of FastCfg (fast_core.h) that its helpers use, with the
// threads per transform given and no limit of 17 values a thread
template <int N_, int R0_, int R1_, int R2_, int R3_, int TPT_, int SHIFT_>
struct TallCfg
{
    static constexpr int N   = N_;
    static constexpr int NP  = (R0_ > 1) + (R1_ > 1) + (R2_ > 1) + (R3_ > 1);
    static constexpr int TPT = TPT_;
    static constexpr int max2(int a, int b)
    {
        return a > b ? a : b;
    }
    static constexpr int radix(int p)
    {
        return p == 0 ? R0_ : p == 1 ? R1_ : p == 2 ? R2_ : R3_;
    }
    static constexpr int S(int p)
    {
        return (N_ / radix(p) + TPT - 1) / TPT;
    }
    static constexpr bool exact(int p)
    {
        return (N_ / radix(p)) % TPT == 0;
    }
    static constexpr int elems(int p)
    {
        return p < NP ? S(p) * radix(p) : 0;
    }
    static constexpr int EPT = max2(max2(elems(0), elems(1)), max2(elems(2), elems(3)));
    static constexpr int cum(int p)
    {
        return p == 0 ? 1 : p == 1 ? R0_ : p == 2 ? R0_ * R1_ : R0_ * R1_ * R2_;
    }
    static constexpr int twoff(int p)
    {
        return p <= 1 ? 0 : twoff(p - 1) + cum(p - 1) * (radix(p - 1) - 1);
    }
    static constexpr int PADSHIFT = SHIFT_;
    static constexpr int PITCH    = N_ + ((N_ - 1) >> PADSHIFT); // LDS positions of a column
    static_assert(N_ == R0_ * R1_ * R2_ * R3_, "radices must multiply to N");
    // (data and twiddles of a thread: 20 values in single and 11 in double precision fit 128 registers, 12
    // in double may take a few of them to scratch memory, see gen_tall_schedules.py)
    template <typename T>
    static constexpr bool fits = EPT * sizeof(T) <= 96;
};

// Where element j of column w lives in LDS: the columns lie beside each other, as in memory, one
// position of padding every 2^PADSHIFT elements.
template <typename Cfg, int W>
struct TallAddr
{
    static FFT_DEV uint32_t at(uint32_t w, uint32_t j)
    {
        const uint32_t pos = Cfg::PADSHIFT < 31 ? j + (j >> Cfg::PADSHIFT) : j;
        return pos * (uint32_t)W + w;
    }
};

template <typename Cfg, int W>
constexpr int tall_threads()
{
    return (Cfg::TPT * W + 63) / 64 * 64;
}

// four waves a SIMD: one workgroup of 1024 threads a compute unit, or two of 512
template <typename T, typename Cfg, int W>
__global__ __launch_bounds__((tall_threads<Cfg, W>()), 4) void tall_kernel(const fftk_params p)
{
    typedef typename cplx_of<T>::type C;
    extern __shared__ double2         tall_smem[];
    C*                                tall_lds = reinterpret_cast<C*>(tall_smem);
    static_assert(Cfg::template fits<T>, "values of a thread");
    constexpr int            N = Cfg::N, TPT = Cfg::TPT, LAST = Cfg::NP - 1;
    constexpr int            R0 = Cfg::radix(0), S0 = Cfg::S(0), RL = Cfg::radix(LAST), SL = Cfg::S(LAST);
    TileCtx<T>               c;
    tile_decode<T>(p, blockIdx.x, c);
    const uint32_t w      = threadIdx.x % (uint32_t)W;
    const uint32_t tt     = threadIdx.x / (uint32_t)W;
    const bool     active = tt < (uint32_t)TPT;
    const bool     ok     = active && c.tile0 + w < p.tile_cnt;
    const bool     inv    = p.dir > 0;
    const C*       src    = reinterpret_cast<const C*>(static_cast<const T*>(p.in0) + c.ibase);
    C*             dst    = reinterpret_cast<C*>(static_cast<T*>(p.out0) + c.obase);
    C              r[Cfg::EPT];
    if(ok)
    {
        const uint32_t lane = tt * p.t_is_c + w;
#pragma unroll
        for(int s = 0; s < S0; ++s)
#pragma unroll
            for(int k = 0; k < R0; ++k)
                if(fk_live<Cfg, 0>(tt, s))
                {
                    C v           = (src + (uint64_t)(s * TPT + k * (N / R0)) * p.t_is_c)[lane];
                    r[s * R0 + k] = inv ? c_swap(v) : v;
                }
    }
    fk_passes_tw<T, Cfg, TallAddr<Cfg, W>>(p.tw, tall_lds, w, tt, active, r, false);
    if(ok)
    {
        const T        sc   = (p.flags & FFTK_F_SCALE) ? (T)p.scale : (T)1;
        const uint32_t lane = tt * p.t_os_c + w;
#pragma unroll
        for(int s = 0; s < SL; ++s)
#pragma unroll
            for(int k = 0; k < RL; ++k)
                if(fk_live<Cfg, LAST>(tt, s))
                {
                    C v = inv ? c_swap(r[s * RL + k]) : r[s * RL + k];
                    v.x *= sc;
                    v.y *= sc;
                    (dst + (uint64_t)(s * TPT + k * (N / RL)) * p.t_os_c)[lane] = v;
                }
    }
}

template <typename T, typename Cfg, int W>
int tall_launch(const fftk_params* p, void* stream)
{
    constexpr size_t   lds = (size_t)Cfg::PITCH * W * 2 * sizeof(T);
    static_assert(lds <= 160 * 1024, "the tile fits the LDS of a compute unit");
    static FftLdsLimit limit;
    if(int rc = limit.allow(tall_kernel<T, Cfg, W>))
        return rc;
    hipLaunchKernelGGL((tall_kernel<T, Cfg, W>), dim3(p->grid), dim3(tall_threads<Cfg, W>()), lds, (hipStream_t)stream,
                       *p);
    return (int)hipGetLastError();
}

// the table entry of one kernel, or an empty one (n = 0) in the translation units that do not
// instantiate it
template <int SLICE, typename T, typename Cfg, int R0, int R1, int R2, int R3, int W>
constexpr TallEntry tall_entry()
{
    if constexpr(SLICE == TALL_SLICE)
        return TallEntry{(uint32_t)Cfg::N,
                         sizeof(T) == 8 ? 1 : 0,
                         {(uint32_t)R0, (uint32_t)R1, (uint32_t)R2, (uint32_t)R3},
                         (uint32_t)Cfg::TPT,
                         (uint32_t)W,
                         (uint32_t)tall_threads<Cfg, W>(),
                         (uint32_t)Cfg::PITCH,
                         &tall_launch<T, Cfg, W>};
    else
        return TallEntry{0, 0, {1, 1, 1, 1}, 0, 0, 0, 0, nullptr};
}

#define TALL_SCHED(SLICE, T, N, A, B, C, D, TPT, W, SHIFT) \
    tall_entry<SLICE, T, TallCfg<N, A, B, C, D, TPT, SHIFT>, A, B, C, D, W>(),
const TallEntry g_slice[] = {
#include "tall_schedules.h"
};

} // namespace

#define TALL_SLICE_FN2(I) fftrt_tall_slice_##I
#define TALL_SLICE_FN(I) TALL_SLICE_FN2(I)

extern "C" const TallEntry* TALL_SLICE_FN(TALL_SLICE)(int* count)
{
    *count = (int)(sizeof(g_slice) / sizeof(g_slice[0]));
    return g_slice;
}

#if TALL_SLICE == 0
extern "C" const TallEntry* fftrt_tall_slice_1(int*);
extern "C" const TallEntry* fftrt_tall_slice_2(int*);
extern "C" const TallEntry* fftrt_tall_slice_3(int*);

namespace
{

// all entries, sorted by (precision, n)
const std::vector<const TallEntry*>& tall_index()
{
    static std::vector<const TallEntry*> index;
    static std::once_flag                once;
    std::call_once(once, []() {
        for(auto f : {&fftrt_tall_slice_0, &fftrt_tall_slice_1, &fftrt_tall_slice_2, &fftrt_tall_slice_3})
        {
            int              cnt = 0;
            const TallEntry* e   = f(&cnt);
            for(int i = 0; i < cnt; ++i)
                if(e[i].n != 0)
                    index.push_back(e + i);
        }
        std::sort(index.begin(), index.end(), [](const TallEntry* a, const TallEntry* b) {
            return a->precision != b->precision ? a->precision < b->precision : a->n < b->n;
        });
    });
    return index;
}

const TallEntry* find_tall(int precision, uint32_t n)
{
    const auto& index = tall_index();
    auto        it    = std::lower_bound(index.begin(), index.end(), n, [&](const TallEntry* e, uint32_t v) {
        return e->precision != precision ? e->precision < precision : e->n < v;
    });
    return it != index.end() && (*it)->precision == precision && (*it)->n == n ? *it : nullptr;
}

} // namespace

extern "C" int fftrt_tall_info(int precision, uint32_t n, uint32_t* radix, uint32_t* nf, uint32_t* tpt, uint32_t* width,
                               uint32_t* threads, uint32_t* pitch)
{
    const TallEntry* e = find_tall(precision, n);
    if(!e)
        return 0;
    uint32_t cnt = 0;
    for(uint32_t i = 0; i < 4; ++i)
        if(e->radix[i] > 1)
            radix[cnt++] = e->radix[i];
    *nf      = cnt;
    *tpt     = e->tpt;
    *width   = e->width;
    *threads = e->threads;
    *pitch   = e->pitch;
    return 1;
}

extern "C" int fftrt_launch_tall(const struct fftk_params* p, int precision, void* stream)
{
    const TallEntry* e = find_tall(precision, p->n);
    if(!e || p->T != e->tpt || p->nthreads != e->threads || p->W != e->width || p->pitch != e->pitch || p->grid == 0
       || p->w_inner)
        return (int)hipErrorInvalidValue;
    return e->launch(p, stream);
}
#endif
