// conv_launch.hpp -- launches of the sphere-form kernels (conv.hpp), whose
// instantiations are spread over several objects (conv_inst.hip).
#pragma once

#include "conv.hpp"

// a plane block: class of its line lengths (rx_class), threads (a multiple of
// 64 up to plane_threads in k_conv_plane, 256 or 512 in k_box_plane) and LDS
struct PlaneShape
{
    int cls, nt;
    PlaneLds lds;
};

template <typename T>
int conv_plane_launch(bool two, const PlaneShape& sh, int64_t grid, hipStream_t st,
                      const ConvPair* pairs, const SphSide* sides, const ConvArgs& a,
                      const PlaneArgs& pa, const z64* Wy, const z64* Wz);
// square planes (rx_square) of one component; lds: exchange rows and plane
template <typename T>
int conv_square_launch(size_t lds, int64_t grid, hipStream_t st, const ConvPair* pairs,
                       const SphSide* sides, const ConvArgs& a, const z64* W);
template <typename T>
int conv_box_plane_launch(const PlaneShape& sh, int64_t grid, hipStream_t st, const SphSide* sides,
                          const BoxArgs& a, const PlaneArgs& pa, const z64* Wy,
                          const z64* Wz);
template <typename T>
int conv_x_launch(int cls, size_t lds, dim3 grid, hipStream_t st, const ConvPair* pairs,
                  const SphSide* sides, const ConvArgs& a, const z64* W);
template <typename T>
int conv_box_x_launch(int cls, size_t lds, dim3 grid, hipStream_t st, const SphSide* sides,
                      const BoxArgs& a, const z64* W);
template <typename T>
int conv_gather_launch(dim3 grid, hipStream_t st, const SphSide* sides, int64_t nsets,
                       int nspinor, int Ny, int Nz, int words, int per);
int conv_maps_launch(int nsides, int npw_max, hipStream_t st, const SphSide* sides, int Nx, int Ny,
                     int Nz, int words, int nzk_max, int nst_max, int* err);

// column tiles of k_sph_gemm: 64 x 16, 64 x 32, 64 x 48, 64 x 64
static inline int sph_gemm_shape(int nb) { return nb <= 16 ? 0 : nb <= 32 ? 1 : nb <= 48 ? 2 : 3; }
static inline int64_t sph_gemm_tiles(int nm, int nb)
{
    static const int cols[4] = {16, 32, 48, 64};
    return cdiv((int64_t)nm * nb, 64) * cdiv(nb, cols[sph_gemm_shape(nb)]);
}
template <typename T>
int sph_gemm_launch(int nsplit, int npairs, hipStream_t st, const ConvPair* pairs,
                    const SphSide* sides, int nm, int nspin, int nb, int nspinor, double scale,
                    z64* out);
