// conv_inst.hip -- instantiations of the sphere-form kernels.  Compiled once
// per CONV_PART (build.py), so that the many compiled line lengths build in
// parallel.
#include <hip/hip_runtime.h>

#include "conv_launch.hpp"

#ifndef CONV_PART
#error "CONV_PART: 0 maps and products, 1 / 2 planes, 3 / 4 boxes, 5 / 6 x lines (FP64 / FP32), 7 / 8 spinor planes, 9 / 10 square planes"
#endif

#define CV_LAUNCH(K, GRID, NT, LDS, ...)                                                          \
    do                                                                                            \
    {                                                                                             \
        auto fn = K;                                                                              \
        if ((LDS) > 48 * 1024)                                                                    \
            HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(fn),                        \
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)(LDS))); \
        hipLaunchKernelGGL(fn, GRID, dim3(NT), LDS, st, __VA_ARGS__);                             \
        HIP_TRY(hipGetLastError());                                                               \
    } while (0)

#if CONV_PART == 0

int conv_maps_launch(int nsides, int npw_max, hipStream_t st, const SphSide* sides, int Nx, int Ny,
                     int Nz, int words, int nzk_max, int nst_max, int* err)
{
    CV_LAUNCH(k_sph_mask, dim3((unsigned)cdiv(npw_max, 256), (unsigned)nsides), 256, 0, sides, Nx,
              Ny, Nz, words, err);
    CV_LAUNCH(k_sph_scan, dim3((unsigned)nsides), 1024, 0, sides, Ny, Nz, words, nzk_max, nst_max,
              err);
    return LELPH_OK;
}

template <typename T>
int conv_gather_launch(dim3 grid, hipStream_t st, const SphSide* sides, int64_t nsets,
                       int nspinor, int Ny, int Nz, int words, int per)
{
    CV_LAUNCH(k_sph_gather<T>, grid, 256, 0, sides, nsets, nspinor, Ny, Nz, words, per);
    return LELPH_OK;
}
template int conv_gather_launch<double>(dim3, hipStream_t, const SphSide*, int64_t, int, int, int,
                                        int, int);
template int conv_gather_launch<float>(dim3, hipStream_t, const SphSide*, int64_t, int, int, int,
                                       int, int);

template <typename T>
int sph_gemm_launch(int nsplit, int npairs, hipStream_t st, const ConvPair* pairs,
                    const SphSide* sides, int nm, int nspin, int nb, int nspinor, double scale,
                    z64* out)
{
    const dim3 grid((unsigned)sph_gemm_tiles(nm, nb), (unsigned)nsplit,
                    (unsigned)(npairs * nspin));
    switch (sph_gemm_shape(nb))
    {
    case 0:
        CV_LAUNCH((k_sph_gemm<T, 1, 1, 4, 1>), grid, 256, 0, pairs, sides, nm, nspin, nb, nspinor,
                  nsplit, npairs, scale, out);
        break;
    case 1:
        CV_LAUNCH((k_sph_gemm<T, 1, 2, 4, 1>), grid, 256, 0, pairs, sides, nm, nspin, nb, nspinor,
                  nsplit, npairs, scale, out);
        break;
    case 2:
        CV_LAUNCH((k_sph_gemm<T, 1, 3, 4, 1>), grid, 256, 0, pairs, sides, nm, nspin, nb, nspinor,
                  nsplit, npairs, scale, out);
        break;
    default:
        CV_LAUNCH((k_sph_gemm<T, 2, 2, 2, 2>), grid, 256, 0, pairs, sides, nm, nspin, nb, nspinor,
                  nsplit, npairs, scale, out);
    }
    return LELPH_OK;
}
template int sph_gemm_launch<double>(int, int, hipStream_t, const ConvPair*, const SphSide*, int,
                                     int, int, int, double, z64*);
template int sph_gemm_launch<float>(int, int, hipStream_t, const ConvPair*, const SphSide*, int,
                                    int, int, int, double, z64*);

#else

#if CONV_PART % 2 == 1
typedef double PT;
#else
typedef float PT;
#endif

#if CONV_PART >= 9
template <typename T>
int conv_square_launch(size_t lds, int64_t grid, hipStream_t st, const ConvPair* pairs,
                       const SphSide* sides, const ConvArgs& a, const z64* W)
{
    const dim3 gr((unsigned)grid);
    switch (a.Ny)
    {
#define SQ_CASE(N, A, B)                                                                          \
    case N:                                                                                       \
        CV_LAUNCH((k_conv_square<T, A, B, rx_square_waves<T>(N)>), gr,                            \
                  64 * rx_square_waves<T>(N), lds, pairs, sides, a, W);                           \
        return LELPH_OK;
        RX_SQUARES(SQ_CASE)
#undef SQ_CASE
        default: return LELPH_ERR_UNSUPPORTED;
    }
}
template int conv_square_launch<PT>(size_t, int64_t, hipStream_t, const ConvPair*, const SphSide*,
                                    const ConvArgs&, const z64*);

#elif CONV_PART == 1 || CONV_PART == 2 || CONV_PART == 7 || CONV_PART == 8
#define CV_TWO (CONV_PART >= 7)
template <typename T, bool TWO>
int conv_plane_t(const PlaneShape& sh, int64_t grid, hipStream_t st, const ConvPair* pairs,
                 const SphSide* sides, const ConvArgs& a, const PlaneArgs& pa, const z64* Wy,
                 const z64* Wz)
{
    const dim3 gr((unsigned)grid);
    if (sh.cls == 0)
        CV_LAUNCH((k_conv_plane<T, TWO, 0>), gr, sh.nt, sh.lds.bytes, pairs, sides, a, pa, Wy,
                  Wz);
    else
        CV_LAUNCH((k_conv_plane<T, TWO, 1>), gr, sh.nt, sh.lds.bytes, pairs, sides, a, pa, Wy,
                  Wz);
    return LELPH_OK;
}
template int conv_plane_t<PT, CV_TWO>(const PlaneShape&, int64_t, hipStream_t, const ConvPair*,
                                      const SphSide*, const ConvArgs&, const PlaneArgs&,
                                      const z64*, const z64*);
#if CONV_PART <= 2
extern template int conv_plane_t<PT, true>(const PlaneShape&, int64_t, hipStream_t,
                                           const ConvPair*, const SphSide*, const ConvArgs&,
                                           const PlaneArgs&, const z64*, const z64*);
template <typename T>
int conv_plane_launch(bool two, const PlaneShape& sh, int64_t grid, hipStream_t st,
                      const ConvPair* pairs, const SphSide* sides, const ConvArgs& a,
                      const PlaneArgs& pa, const z64* Wy, const z64* Wz)
{
    return two ? conv_plane_t<T, true>(sh, grid, st, pairs, sides, a, pa, Wy, Wz)
               : conv_plane_t<T, false>(sh, grid, st, pairs, sides, a, pa, Wy, Wz);
}
template int conv_plane_launch<PT>(bool, const PlaneShape&, int64_t, hipStream_t, const ConvPair*,
                                   const SphSide*, const ConvArgs&, const PlaneArgs&,
                                   const z64*, const z64*);
#endif

#elif CONV_PART == 3 || CONV_PART == 4
template <typename T>
int conv_box_plane_launch(const PlaneShape& sh, int64_t grid, hipStream_t st, const SphSide* sides,
                          const BoxArgs& a, const PlaneArgs& pa, const z64* Wy,
                          const z64* Wz)
{
    const dim3 gr((unsigned)grid);
    if (sh.cls == 0 && sh.nt == 512)
        CV_LAUNCH((k_box_plane<T, 0, 512>), gr, 512, sh.lds.bytes, sides, a, pa, Wy, Wz);
    else if (sh.cls == 0)
        CV_LAUNCH((k_box_plane<T, 0, 256>), gr, 256, sh.lds.bytes, sides, a, pa, Wy, Wz);
    else
        CV_LAUNCH((k_box_plane<T, 1, 256>), gr, 256, sh.lds.bytes, sides, a, pa, Wy, Wz);
    return LELPH_OK;
}
template int conv_box_plane_launch<PT>(const PlaneShape&, int64_t, hipStream_t, const SphSide*,
                                       const BoxArgs&, const PlaneArgs&, const z64*,
                                       const z64*);

#else
template <typename T>
int conv_x_launch(int cls, size_t lds, dim3 grid, hipStream_t st, const ConvPair* pairs,
                  const SphSide* sides, const ConvArgs& a, const z64* W)
{
    if (cls == 0)
        CV_LAUNCH((k_conv_x<T, 0>), grid, X_THREADS, lds, pairs, sides, a, W);
    else
        CV_LAUNCH((k_conv_x<T, 1>), grid, X_THREADS, lds, pairs, sides, a, W);
    return LELPH_OK;
}
template <typename T>
int conv_box_x_launch(int cls, size_t lds, dim3 grid, hipStream_t st, const SphSide* sides,
                      const BoxArgs& a, const z64* W)
{
    if (cls == 0)
        CV_LAUNCH((k_box_x<T, 0>), grid, X_THREADS, lds, sides, a, W);
    else
        CV_LAUNCH((k_box_x<T, 1>), grid, X_THREADS, lds, sides, a, W);
    return LELPH_OK;
}
template int conv_x_launch<PT>(int, size_t, dim3, hipStream_t, const ConvPair*, const SphSide*,
                               const ConvArgs&, const z64*);
template int conv_box_x_launch<PT>(int, size_t, dim3, hipStream_t, const SphSide*, const BoxArgs&,
                                   const z64*);
#endif
#endif
