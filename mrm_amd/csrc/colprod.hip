// colprod.hip - the column transforms and the k-space product of the split path in one
// kernel: forward y-FFT of the 3 n_lay source columns of one kx, the product of
// demag.f90:117-121 and the inverse y-FFT, with the Engine member that launches it.
// FP64 form only (Engine::choose_split).
#include "engine.h"
#include "device_common.h"

// One workgroup per column as laid out (RowSplit: kx, or (kx, r) of a split transform), its
// 3 NL columns of L values in LDS throughout.  The product takes a thread per value of ky
// with the NL layers' spectra and field sums in registers and reads each of the 2 NL - 1
// offset blocks of the tensor once, in k_prod_offsets' order.  Bound by the tensor's and the
// spectra's memory traffic, which as three kernels (k_colT, k_prod_offsets, k_colT) includes
// the spectra four times more.
template <typename T, int E, int NL>
__global__ void __launch_bounds__(512) k_colp(DemagOps<T> one, const DemagOps<T>* __restrict__ tab, int L, int vnx,
                                              FFTPlan py, const C2<T>* __restrict__ twy)
{
    const C2<T>* __restrict__ S1 = tab ? tab[blockIdx.z].S1 : one.S1;
    C2<T>* __restrict__ S2 = tab ? tab[blockIdx.z].S2 : one.S2;
    const C2<T>* __restrict__ Tspec = tab ? tab[blockIdx.z].Tspec : one.Tspec;
    const int kx = xcd_remap(blockIdx.x, gridDim.x);
    if (kx >= vnx) return;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    constexpr int NC = 3 * NL;
    T* re = reinterpret_cast<T*>(smem_raw);
    T* im = re + LPN(NC * L);
    staged_load<8, T>(
        NC * L,
        [&](int idx) {
            const int col = idx / L, y = idx - col * L;
            return S1[((size_t)col * vnx + kx) * L + y];
        },
        [&](int idx, C2<T> v) { re[LP(idx)] = v.x; im[LP(idx)] = v.y; });
    __syncthreads();
    lds_fft<T, E, false, true>(re, im, NC, py, twy);
    const C2<T>* Tk = Tspec + (size_t)kx * (2 * NL - 1) * 6 * L;
    for (int ky = threadIdx.x; ky < L; ky += blockDim.x) {
        C2<T> m[NL][3], h[NL][3];
#pragma unroll
        for (int k = 0; k < NL; k++)
#pragma unroll
            for (int b = 0; b < 3; b++) {
                const int i = LP((3 * k + b) * L + ky);
                m[k][b] = {re[i], im[i]};
                h[k][b] = {0, 0};
            }
#pragma unroll
        for (int d = NL - 1; d >= -(NL - 1); d--) {
            const C2<T>* t = Tk + (size_t)(d + NL - 1) * 6 * L + ky;   // slots xx yy zz xy xz yz
            C2<T> tv[6];
#pragma unroll
            for (int sl = 0; sl < 6; sl++) tv[sl] = ld_s<true>(t + (size_t)sl * L);
#pragma unroll
            for (int ko = 0; ko < NL; ko++) {
                const int ks = ko - d;
                if (ks < 0 || ks >= NL) continue;
                const C2<T> mx = m[ks][0], my = m[ks][1], mz = m[ks][2];
                C2<T> a;
                a = cmul(tv[0], mx); h[ko][0].x += a.x; h[ko][0].y += a.y;
                a = cmul(tv[3], my); h[ko][0].x += a.x; h[ko][0].y += a.y;
                a = cmul(tv[4], mz); h[ko][0].x += a.x; h[ko][0].y += a.y;
                a = cmul(tv[3], mx); h[ko][1].x += a.x; h[ko][1].y += a.y;
                a = cmul(tv[1], my); h[ko][1].x += a.x; h[ko][1].y += a.y;
                a = cmul(tv[5], mz); h[ko][1].x += a.x; h[ko][1].y += a.y;
                a = cmul(tv[4], mx); h[ko][2].x += a.x; h[ko][2].y += a.y;
                a = cmul(tv[5], my); h[ko][2].x += a.x; h[ko][2].y += a.y;
                a = cmul(tv[2], mz); h[ko][2].x += a.x; h[ko][2].y += a.y;
            }
        }
        // each value of ky is one thread's: written over its own spectra
#pragma unroll
        for (int k = 0; k < NL; k++)
#pragma unroll
            for (int b = 0; b < 3; b++) {
                const int i = LP((3 * k + b) * L + ky);
                re[i] = h[k][b].x;
                im[i] = h[k][b].y;
            }
    }
    __syncthreads();
    lds_fft<T, E, true, true>(re, im, NC, py, twy);
    for (int idx = threadIdx.x; idx < NC * L; idx += blockDim.x) {
        const int col = idx / L, y = idx - col * L;
        S2[((size_t)col * vnx + kx) * L + y] = C2<T>{re[LP(idx)], im[LP(idx)]};
    }
}

// the kernel's dynamic LDS at most (choose_split): with 512 threads 14 elements a thread, with
// 256 for up to 56 KB as well
#define MRMG_COLP_LDS (112 * 1024)
#define MRMG_COLP_E 16

#define COLP_FN(NL) ((const void*)k_colp<double, MRMG_COLP_E, NL>)
#define COLP_NL(M) M(1) M(2) M(3) M(4)

// dynamic LDS above 64 KiB must be requested: the most that any context's kernel takes, so that
// one context's request is not another's limit
template <>
int Engine<double>::lds_attr_colp()
{
#define COLP_ATTR(NL) HIPCHK(hipFuncSetAttribute(COLP_FN(NL), hipFuncAttributeMaxDynamicSharedMemorySize, MRMG_COLP_LDS));
    COLP_NL(COLP_ATTR)
#undef COLP_ATTR
    return MRMG_OK;
}

template <>
int Engine<double>::launch_colp()
{
    const DemagOps<double> o = ops();
    const int z = btab ? bn : 1, L = vL(), vx = vnx(), th = colp_threads, e = pick_e(3 * c->nl, pcol, th);
    if (e < 0 || e > MRMG_COLP_E || lds_colp > MRMG_COLP_LDS || nslot != 6 || !one_fit)
        return set_err(MRMG_ERR_STATE, "the one-kernel column path does not fit");
    const dim3 g((unsigned)((vx + 7) / 8 * 8), 1, (unsigned)z);
#define COLP_LAUNCH(NL)                                                                                                 \
    case NL:                                                                                                            \
        hipLaunchKernelGGL((k_colp<double, MRMG_COLP_E, NL>), g, dim3(th), lds_colp, c->stream, o, btab, L, vx, pcol,   \
                           twy.p);                                                                                      \
        break;
    switch (c->nl) {
        COLP_NL(COLP_LAUNCH)
    default:
        return set_err(MRMG_ERR_STATE, "the one-kernel column path is not built for %d layers", c->nl);
    }
#undef COLP_LAUNCH
    HIPCHK(hipGetLastError());
    return MRMG_OK;
}
