// The product over stencil planes (stencil.h) as the resident solvers of
// persistent.h run it; included there after SolveArgs.
#pragma once

namespace mf {

constexpr int LDS_BYTES = 160 * 1024;

// The stencil product of a resident kernel (persistent.h): CLS the values'
// class; A64: low-precision values summed in FP64 against the FP64 vector.
template <int CLS, int SW, bool A64> struct Stencil {
    // r in registers: LDS then holds more of the matrix
    static constexpr bool r_regs = true;
    static constexpr bool lds_tags = false;
    // VECS: vectors of RPT x TPB doubles the kernel keeps in LDS; VREGS:
    // registers it holds per row
    template <int TPB, int RPT, int VECS, int VREGS> struct Op {
        using Acc = typename std::conditional<CLS == 0 || A64, double, float>::type;
        static constexpr int NE = SW ? SW : 4;
        // LDS left for values beside the vectors, the gathered-vector copy of
        // one-workgroup solves and the reduction scratch
        static constexpr int VB = (LDS_BYTES - VECS * RPT * TPB * 8 - (RPT <= 4 ? 12 * 2048 : 0) - 1024 -
                                  EXC_LDS * (int)sizeof(PlaneExc)) / 16 * 16;
        // rows (quads where SW = 0) in flight: two rows of 5 or 7 entries (three
        // and four measure 0 to 4 % slower: 128^3 Poisson CG FP64 25.8 us per
        // iteration with two, 26.8 and 26.9 with three and four; 151 x 149 x 147
        // E4M3 24.9, 25.5, 25.5; eight 28.3), four quads, or what the registers
        // beside the vectors hold
        static constexpr int STEP_REGS = PlaneVals<CLS, SW>::NW * (CLS == 0 ? 2 : 1) + NE * (int)sizeof(Acc) / 4;
        static constexpr int FIT = (190 - VREGS * RPT) / STEP_REGS;
        static constexpr int DMAX = SW == 0 ? 4 : RPT < 2 ? RPT : 2;
        static constexpr int D = FIT < 1 ? 1 : FIT < DMAX ? FIT : DMAX;
        struct Shared {
            alignas(16) uint8_t val[VB];
            PlaneExc exc[EXC_LDS];
        };
        struct Buf {
            PlaneVals<CLS, SW> v;
            Acc x[NE];
        };
        const Shared &sh;
        const uint8_t *s_val;
        int row0, row1;  // rows of the chunk
        int slots;       // row slots in use: row0 + i TPB + tid, i < slots
        int nlds;        // the first nlds of them have their values in LDS
        bool edge;       // a gather may leave the vector
        // products alternate the direction in which they walk the streamed
        // rows: the next one starts with the values that the L2 still holds
        mutable bool down = false;
        // the chunk's listed entries
        const PlaneExc *exc = nullptr;
        int nexc = 0;

        // Copies each thread's own rows; a __syncthreads must follow for the
        // listed entries.
        __device__ Op(const SolveArgs &A, Shared &s, int r0, int r1) : sh(s), s_val(s.val), row0(r0), row1(r1)
        {
            const int rb = plane_row_bytes(CLS, A.pl.L), tid = threadIdx.x;
            slots = (row1 - row0 + TPB - 1) / TPB;
            nlds = min(slots, VB / (rb * TPB));
            const OffPtr off = off_ptr(A.off);
            edge = row0 + min(off[0], 0) < 0 || row1 - 1 + max(off[A.pl.L - 1], 0) >= A.nrows;
            const int nq = SW ? 1 : (A.pl.L + 3) >> 2;
            if (A.nexc) {
                auto first = [&](int r) {  // first entry of row r or later
                    int lo = 0, hi = A.nexc;
                    while (lo < hi) {
                        const int mid = (lo + hi) >> 1;
                        if (A.exc[mid].row < r) lo = mid + 1;
                        else hi = mid;
                    }
                    return lo;
                };
                const int e0 = first(row0);
                nexc = first(row1) - e0;
                exc = A.exc + e0;
                if (tid < min(nexc, EXC_LDS)) s.exc[tid] = exc[tid];
            }
            for (int i = 0; i < nlds; i++) {
                const uint32_t r = (uint32_t)min(row0 + i * TPB + tid, row1 - 1);
                for (int q = 0; q < nq; q++) {
                    PlaneVals<CLS, SW> v;
                    v.load(A.pl.val + (size_t)q * 4 * cls_width(CLS) * A.pl.stride, A.pl.stride, r);
                    put(s.val + (size_t)i * rb * TPB + (size_t)q * 4 * cls_width(CLS) * TPB, v, tid);
                }
            }
        }
        __device__ PlaneExc listed(int e) const
        {
            if (e < EXC_LDS) return sh.exc[e];
            return exc[e];
        }
        // Adds the listed entries to a product that body stored at dst[i TPB +
        // tid] as it came (the sums are Acc values, so they go on exactly where
        // they stopped).  Beside the product's loop, which has no registers to
        // spare for it; BiCGSTAB alone, CG folds its products into s.
        __device__ void add_listed(double *dst, const double *g64, const float *g32) const
        {
            for (int e = 0; e < nexc; e++) {
                const PlaneExc x = listed(e);
                const int at = x.row - row0;
                if (at % TPB != (int)threadIdx.x) continue;
                Acc xg;
                if constexpr (sizeof(Acc) == 8) xg = g64[x.row + x.off];
                else xg = g32[x.row + x.off];
                dst[at] = (double)fma_t((Acc)x.val, xg, (Acc)dst[at]);
            }
        }
        __device__ static void put(uint8_t *base, const PlaneVals<CLS, SW> &v, int t)
        {
            if constexpr (CLS == 0) {
#pragma unroll
                for (int p = 0; p < NE / 2; p++)
                    reinterpret_cast<double2 *>(base + p * 16 * TPB)[t] = make_double2(v.w[2 * p], v.w[2 * p + 1]);
                if constexpr (NE & 1) reinterpret_cast<double *>(base + NE / 2 * 16 * TPB)[t] = v.w[NE - 1];
            } else if constexpr (CLS == 1) {
                reinterpret_cast<float4 *>(base)[t] = make_float4(v.w[0], v.w[1], v.w[2], v.w[3]);
                if constexpr (NE >= 6) reinterpret_cast<float2 *>(base + 16 * TPB)[t] = make_float2(v.w[4], v.w[5]);
                if constexpr (NE & 1) reinterpret_cast<float *>(base + (NE - 1) * 4 * TPB)[t] = v.w[NE - 1];
            } else if constexpr (PlaneVals<CLS, SW>::NW == 4) {
                reinterpret_cast<uint4 *>(base)[t] = make_uint4(v.w[0], v.w[1], v.w[2], v.w[3]);
            } else if constexpr (PlaneVals<CLS, SW>::NW == 2) {
                reinterpret_cast<uint2 *>(base)[t] = make_uint2(v.w[0], v.w[1]);
            } else {
                reinterpret_cast<uint32_t *>(base)[t] = v.w[0];
            }
        }

        // y of the thread's rows, handed to body(i, y) in some order of i (0
        // for the lanes beyond the chunk's last row).
        template <bool, int, int, typename F>
        __device__ __forceinline__ void product(const SolveArgs &A, int rbase, const double *g64, const float *g32,
                                                F &&body) const
        {
            if constexpr (sizeof(Acc) == 8) run(A, rbase, g64, body);
            else run(A, rbase, g32, body);
        }
        template <typename F>
        __device__ __forceinline__ void run(const SolveArgs &A, int rbase, const Acc *g, F &&body) const
        {
            down = !down;
            if (edge) {
                if (nlds > 0) loop<true, true>(A, rbase, g, 0, nlds, 1, body);
                if (nlds < slots) loop<true, false>(A, rbase, g, down ? slots - 1 : nlds, slots - nlds, down ? -1 : 1, body);
            } else {
                if (nlds > 0) loop<false, true>(A, rbase, g, 0, nlds, 1, body);
                if (nlds < slots) loop<false, false>(A, rbase, g, down ? slots - 1 : nlds, slots - nlds, down ? -1 : 1, body);
            }
        }
        // n row slots from i0 on by dir, D steps (a row, or a quad of one) in flight:
        // step t + D is fetched behind step t's sums.  The last fetches repeat
        // the last step, so that the count of loads in flight is fixed.
        template <bool EDGE, bool LDSV, typename F>
        __device__ __forceinline__ void loop(const SolveArgs &A, int rbase, const Acc *g, int i0, int n, int dir,
                                             F &&body) const
        {
            const Planes &P = A.pl;
            const OffPtr off = off_ptr(A.off);
            const int tid = threadIdx.x, nq = SW ? 1 : (P.L + 3) >> 2;
            const int rb = plane_row_bytes(CLS, P.L);
            const int T = n * nq, NG = (T + D - 1) / D, last = i0 + (n - 1) * dir;
            Buf buf[D];
            int fi = i0, fq = 0;  // next step to fetch
            auto fetch = [&](Buf &b) {
                const int r = min(rbase + fi * TPB, row1 - 1);
                if constexpr (LDSV)
                    b.v.load(s_val + (size_t)fi * rb * TPB + (size_t)fq * 4 * cls_width(CLS) * TPB, TPB, tid);
                else
                    b.v.load(P.val + (size_t)fq * 4 * cls_width(CLS) * P.stride, P.stride, (uint32_t)r);
                static_for<NE>([&](auto e) {
                    const int o = off[SW ? (int)e : fq * 4 + e];
                    if constexpr (EDGE)
                        b.x[e] = ld_elem(g, (uint32_t)min(max(r + o, 0), A.nrows - 1));
                    else
                        b.x[e] = ld_elem(g, (uint32_t)(r + o));
                });
                if (fq + 1 < nq) fq++;
                else if (fi != last) {
                    fi += dir;
                    fq = 0;
                }
            };
            int ci = i0, cq = 0;  // step to sum
            Acc acc = 0;
            auto sum = [&](const Buf &b) {
                static_for<NE>([&](auto e) { acc = fma_t((Acc)b.v.template get<e>(), b.x[e], acc); });
                if (SW || ++cq == nq) {
                    body(ci, rbase + ci * TPB < row1 ? (double)acc : 0.0);
                    ci += dir;
                    cq = 0;
                    acc = 0;
                }
            };
#pragma unroll
            for (int d = 0; d < D; d++) fetch(buf[d]);
#pragma unroll 1
            for (int k = 0; k + 1 < NG; k++) {
#pragma unroll
                for (int d = 0; d < D; d++) {
                    sum(buf[d]);
                    __builtin_amdgcn_sched_barrier(0);
                    fetch(buf[d]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            const int left = T - (NG - 1) * D;
#pragma unroll
            for (int d = 0; d < D; d++)
                if (d < left) sum(buf[d]);
        }

        // FP64-accumulated product of row slot i (the true-residual passes)
        template <bool, int NV>
        __device__ __forceinline__ void pass_row(const SolveArgs &A, int i, size_t row, const double *const (&g)[NV],
                                                 double (&acc)[NV]) const
        {
            if (A.use64) plane_row_f64<0, SW, NV>(A.pl64, off_ptr(A.off), (uint32_t)row, A.nrows, g, acc);
            else {
                plane_row_f64<CLS, SW, NV>(A.pl, off_ptr(A.off), (uint32_t)row, A.nrows, g, acc);
                for (int e = 0; e < nexc; e++) {
                    const PlaneExc x = listed(e);
                    if (x.row == (int)row)
#pragma unroll
                        for (int k = 0; k < NV; k++)
                            acc[k] = __builtin_fma((double)x.val, g[k][x.row + x.off], acc[k]);
                }
            }
        }
    };
};

}  // namespace mf
