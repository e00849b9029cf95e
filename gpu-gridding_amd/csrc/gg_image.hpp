// gg_image.hpp -- grid -> image: the 2-D FFT of the grid that follows
// gridding (README:24-26).  For an even grid size G, c = G/2,
//   image[y][x] = Re( sum_{v,u} grid[v][u]
//                     * exp(+2 pi i ((u - c)(x - c) + (v - c)(y - c)) / G) ) * scale
//               = Re( (-1)^(x+y) * BACKWARD_DFT[ (-1)^(u+v) grid ][y][x] ) * scale
// (the constant phase exp(2 pi i c^2 / G) squares to 1 over the two axes).
// The signs (-1)^(x+y) are a shift of the input by c along both axes, and the
// real part is the transform of the input's Hermitian part, which a
// complex-to-real transform takes from its half u <= c alone.  So:
//   k_image_pre    work[v][u] = (-1)^(u+v) * scale / 2 *
//                      (grid[v + c][u + c] + conj(grid[c - v][c - u])),
//                  indices mod G, u = 0 .. c  (one pass, HBM-bound: every cell
//                  is read once, half as much is written)
//   hipFFT         unnormalised backward C2R / Z2D, into the image
// against a full complex transform between a sign pass and a real-part pass
// this moves half the bytes (8192^2 FP32: 1.19 -> 0.72 ms, its error against 64 bits the same).
#pragma once

#include "gg_device.hpp"

namespace gg {

template <typename T>
__global__ __launch_bounds__(256)
void k_image_pre(const typename V2<T>::t* __restrict__ grid, typename V2<T>::t* __restrict__ work,
        unsigned G, T half_scale)
{
    const unsigned c = G / 2;
    for (unsigned v = blockIdx.y; v < G; v += gridDim.y)
    {
        const typename V2<T>::t* a = grid + (size_t)(v < c ? v + c : v - c) * G;
        const typename V2<T>::t* b = grid + (size_t)(v <= c ? c - v : c + G - v) * G;
        typename V2<T>::t* w = work + (size_t)v * (c + 1);
        for (unsigned u = blockIdx.x * 256u + threadIdx.x; u <= c; u += gridDim.x * 256u)
        {
            const typename V2<T>::t p = a[u < c ? u + c : 0u], q = b[c - u];
            const T s = ((u + v) & 1u) ? -half_scale : half_scale;
            w[u] = {s * (p.x + q.x), s * (p.y - q.y)};
        }
    }
}

// image = src * scale (one pass; in place where they are the same): where the
// transform cannot write the image itself, or the scale could push values out
// of range before the transform.
template <typename T>
__global__ __launch_bounds__(256)
void k_image_scale(const T* src, T* image, unsigned long long n, T scale)
{
    for (unsigned long long i = blockIdx.x * (unsigned long long)blockDim.x + threadIdx.x; i < n;
            i += (unsigned long long)gridDim.x * blockDim.x)
        image[i] = src[i] * scale;
}

} // namespace gg
