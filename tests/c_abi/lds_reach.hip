// The LDS bytes that a wave exchange of the sphere form's plane kernels reads
// (csrc/conv.hpp:ln_exchange), lane by lane, against what the launches ask for.
// Host code only; prints the number of cases and of those that fall short.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "conv_launch.hpp"

template <typename T>
static size_t furthest(int R1, int R2, int NW)
{
    // elements of 8 bytes: one part of an FP64 number, a whole FP32 one
    size_t most = 0;
    const size_t wave = (size_t)(NW - 1) * ln_space(R2) * ln_row_bytes<T>(R1, R2);
    for (int lane = 0; lane < 64; ++lane)
    {
        const int rd = lane / R1, k1 = lane % R1, r = lane / R2, j = lane % R2;
        for (int i = 0; i < R2; ++i)
            most = std::max(most, wave + 8 * (size_t)(rd * ln_row(R1, R2) + k1 + i * (R1 | 1) + 1));
        for (int k = 0; k < R1; ++k)
            most = std::max(most, wave + 8 * (size_t)(r * ln_row(R1, R2) + j * (R1 | 1) + k + 1));
    }
    return most;
}

static int cases = 0, short_of = 0;
static void check(size_t have, size_t need)
{
    ++cases;
    if (have < need) ++short_of;
}

template <typename T>
static void all()
{
    static const int len[][3] = {
#define ROW(N, A, B) {N, A, B},
        RX_LENGTHS(ROW)
#undef ROW
    };
    static const int nzks[] = {1, 2, 3, 5, 8, 12};
    for (const auto& z : len)
        for (const auto& y : len)
            for (int nw = 4; nw <= 12; ++nw)
                for (int nzk : nzks)
                    check(plane_lds<T>(y[1], y[2], z[1], z[2], nzk, 64 * nw).bytes,
                          furthest<T>(z[1], z[2], nw));
#define SQUARE(N, A, B)                                                                           \
    for (int nzk = 1; nzk <= N; ++nzk)                                                            \
        check(square_lds<T>(A, B, rx_square_waves<T>(N), nzk),                                    \
              furthest<T>(A, B, rx_square_waves<T>(N)));
    RX_SQUARES(SQUARE)
#undef SQUARE
}

int main()
{
    all<double>();
    all<float>();
    std::printf("%d %d\n", cases, short_of);
    return 0;
}
