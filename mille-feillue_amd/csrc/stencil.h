// Stencil planes: the compute layout of matrices whose rows all draw their
// entries from one short list of offsets column - row (grids with a 5-, 7- or
// 27-point operator and the like), and the product over it that the resident
// solvers run.
//
// The slab layout reads headers and indices before it can gather, and its
// quads of entries pad a 7-point row to 8.  Here the matrix has one ascending
// offset table, held in scalar registers, and its values stand in planes
// of one row after the other, so a wave reads contiguous blocks and nothing is
// read but values: row r's entry at table position j sits at position j,
// positions it lacks hold value 0.  Loads of one row do not depend on each
// other, and the loop keeps two rows, or four quads, in flight.  Entries keep their order
// and zeros add nothing to a sum that starts at +0, so the sums are bit
// for bit those of the slabs.
//
// Measured on the solvers, slabs -> planes, us per iteration: 128^3 Poisson CG
// FP64 32.6 -> 27.3 (134 -> 117 MB of values, 3 of 16 rows per thread in LDS;
// bound by the Infinity Cache, 7.2 TB/s), E4M3 17.6 -> 13.3 (values in LDS);
// 151 x 149 x 147 E4M3, whose vectors the slab kernels stream, 63.8 -> 25.8;
// 39^3 27-point BiCGSTAB FP64 23.1 -> 21.2; 30 x 31 Laplacian, one workgroup,
// 3.24 -> 2.97.
//
// A plane set holds one class c (0 FP64, 1 FP32, 2 FP16, 3 E4M3; layouts of
// rounded tiles have a few tiles of one or two entries that a narrower class
// happens to hold: those entries stand in a short list, PlaneExc, sorted by
// row, and follow the planes' entries of their row, as the slabs sum them), with rows
// of exactly SW = 5 or 7 entries (5- and 7-point stencils) or, SW = 0, of quads
// of 4 (any table of up to STENCIL_MAX offsets, padded to a multiple of 4):
//   FP64  pairs of entries (16 B a row) one after the other, then, when the
//         row has an odd entry, one plane of it (8 B a row)
//   FP32  quads (16 B a row), then the last two (8 B) and the last one (4 B)
//   FP16  8 B a quad; SW: one plane of 8 entries (16 B)
//   E4M3  4 B a quad; SW: one plane of 8 entries (8 B)
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mf_device.h"

namespace mf {

struct Planes {
    const uint8_t *val;
    unsigned stride;  // rows of a plane
    int L;            // offsets of the table
};
// The offset table of a matrix on the device (tiles.hip: find_stencil).
struct StencilTable {
    unsigned long long key;  // longest row, see k_longest_row
    int L, bad;              // offsets; no stencil matrix
    int off[STENCIL_MAX];
};
// The offsets of the table, ascending, zeros from L up to a multiple of 4: read
// with scalar loads (constant address space).
using OffPtr = const __attribute__((address_space(4))) int *;
__device__ __forceinline__ OffPtr off_ptr(const int *p) { return (OffPtr)(uintptr_t)p; }

// An entry of a plane set's matrix that another class than the planes' stores
// (its position there holds 0): value as that class rounds it.
struct PlaneExc {
    int row, off;
    float val;
    int cls;
};
constexpr int EXC_LDS = 64;  // of a chunk, kept in LDS

// Specialised row width of a table of L offsets (0: quads).
__host__ __device__ constexpr int plane_sw(int L) { return L == 5 || L == 7 ? L : 0; }
// Entries of a row with their padding, and bytes of a row over all planes.
__host__ __device__ constexpr int plane_entries(int cls, int L)
{
    return plane_sw(L) ? (cls >= 2 ? 8 : L) : (L + 3) / 4 * 4;
}
__host__ __device__ constexpr int plane_row_bytes(int cls, int L) { return plane_entries(cls, L) * cls_width(cls); }

// Byte position of entry j of row r in a plane set of stride rows.
__host__ __device__ inline size_t plane_pos(int cls, int L, size_t stride, size_t r, int j)
{
    const size_t w = (size_t)cls_width(cls);
    const int sw = plane_sw(L);
    if (cls >= 2) {
        const size_t per = sw ? 8 : 4;  // entries of a plane
        return (j / per) * per * w * stride + (r * per + j % per) * w;
    }
    const int n = plane_entries(cls, L);  // exact for SW, a multiple of 4 otherwise
    if (cls == 0) {
        if (j < (n & ~1)) return (size_t)(j / 2) * 16 * stride + (r * 2 + j % 2) * 8;
        return (size_t)(n / 2) * 16 * stride + r * 8;
    }
    size_t base = 0;
    int j0 = 0;
    for (int step = 4; step >= 1; step >>= 1)
        while (n - j0 >= step) {
            if (j < j0 + step) return base + (r * step + (j - j0)) * 4;
            base += (size_t)step * 4 * stride;
            j0 += step;
        }
    return base;
}

// NE consecutive entries of one row's plane set (NE = SW: the whole row; else
// one quad), base at their first plane, planes of mul rows.
template <int CLS, int SW> struct PlaneVals {
    static constexpr int NE = SW ? SW : 4;
    static constexpr int NW = CLS == 0 ? NE : CLS == 1 ? NE : CLS == 2 ? (SW ? 4 : 2) : (SW ? 2 : 1);
    using W = typename std::conditional<CLS == 0, double, typename std::conditional<CLS == 1, float, uint32_t>::type>::type;
    W w[NW];
    __device__ __forceinline__ void load(const uint8_t *base, size_t mul, uint32_t r)
    {
        if constexpr (CLS == 0) {
#pragma unroll
            for (int p = 0; p < NE / 2; p++) {
                const double2 d = *reinterpret_cast<const double2 *>(base + (size_t)p * 16 * mul + r * 16u);
                w[2 * p] = d.x;
                w[2 * p + 1] = d.y;
            }
            if constexpr (NE & 1) w[NE - 1] = *reinterpret_cast<const double *>(base + (size_t)(NE / 2) * 16 * mul + r * 8u);
        } else if constexpr (CLS == 1) {
            const float4 d = *reinterpret_cast<const float4 *>(base + r * 16u);
            w[0] = d.x;
            w[1] = d.y;
            w[2] = d.z;
            w[3] = d.w;
            if constexpr (NE >= 6) {
                const float2 e = *reinterpret_cast<const float2 *>(base + 16 * mul + r * 8u);
                w[4] = e.x;
                w[5] = e.y;
            }
            if constexpr (NE & 1)
                w[NE - 1] = *reinterpret_cast<const float *>(base + (size_t)(NE - 1) * 4 * mul + r * 4u);
        } else if constexpr (NW == 4) {
            const uint4 d = *reinterpret_cast<const uint4 *>(base + r * 16u);
            w[0] = d.x;
            w[1] = d.y;
            w[2] = d.z;
            w[3] = d.w;
        } else if constexpr (NW == 2) {
            const uint2 d = *reinterpret_cast<const uint2 *>(base + r * 8u);
            w[0] = d.x;
            w[1] = d.y;
        } else {
            w[0] = *reinterpret_cast<const uint32_t *>(base + r * 4u);
        }
    }
    template <int E> __device__ __forceinline__ auto get() const
    {
        if constexpr (CLS <= 1) return w[E];
        else if constexpr (CLS == 2) return f16_to_f32((uint16_t)((w[E / 2] >> (16 * (E & 1))) & 0xffffu));
        else return __builtin_amdgcn_cvt_f32_fp8((int)w[E / 4], E % 4);
    }
};

// FP64-accumulated product of NV vectors for one row (true-residual passes);
// n rows, gathers clamped into them (entries out of range have value 0).
template <int CLS, int SW, int NV>
__device__ __forceinline__ void plane_row_f64(const Planes &P, OffPtr off, uint32_t row, int n,
                                              const double *const (&g)[NV], double (&acc)[NV])
{
    constexpr int NE = SW ? SW : 4;
    const int nq = SW ? 1 : (P.L + 3) >> 2;
    for (int q = 0; q < nq; q++) {
        PlaneVals<CLS, SW> v;
        v.load(P.val + (size_t)q * 4 * cls_width(CLS) * P.stride, P.stride, row);
        static_for<NE>([&](auto e) {
            const double a = (double)v.template get<e>();
            const int c = min(max((int)row + off[q * 4 + e], 0), n - 1);
#pragma unroll
            for (int k = 0; k < NV; k++) acc[k] = __builtin_fma(a, g[k][c], acc[k]);
        });
    }
}

}  // namespace mf
