// rowsplit.hip - the row FFT kernels of a split column transform (RowSplit in kernels.h):
// they take the column transform's first radix-R step after the row r2c and its last one
// before the row c2r, with the Engine member that launches them.  FP64 form only
// (Engine::choose_split).
#include "engine.h"
#include "device_common.h"

#define MRMG_UF 4   // cells of a run per iteration, as in demag.hip

// The runs of a split row workgroup (RowSplit): its rows i = j Rm + q are the layer's rows
// y0 + j + q L, whose runs are numbered through; run t of row i is run base[i] + t of the
// row-by-row list, pref[i] <= t < pref[i + 1].
#define MRMG_SPLIT_ROWS 16
struct SplitRuns {
    int base[MRMG_SPLIT_ROWS], pref[MRMG_SPLIT_ROWS + 1];   // in LDS
    // by the workgroup's first 16 lanes; the caller synchronises
    template <typename T>
    __device__ __forceinline__ void init(const RowRuns& R, int k, int ny, int y0, const RowSplit<T>& rs)
    {
        const int i = (int)threadIdx.x;
        if (i >= MRMG_SPLIT_ROWS) return;
        const int j = i / rs.Rm, q = i - j * rs.Rm;
        int a = 0, n = 0;
        if (j < rs.Y && y0 + j < rs.L) {
            const int* ro = R.row_off + k * ny + y0 + j + q * rs.L;
            a = ro[0];
            n = ro[1] - a;
        }
        int p = n;   // the runs up to and with row i
#pragma unroll
        for (int o = 1; o < MRMG_SPLIT_ROWS; o *= 2) {
            const int v = __shfl_up(p, o, MRMG_SPLIT_ROWS);
            if (i >= o) p += v;
        }
        base[i] = a - (p - n);
        pref[i] = p - n;
        if (i == MRMG_SPLIT_ROWS - 1) pref[MRMG_SPLIT_ROWS] = p;
    }
    __device__ __forceinline__ int runs() const { return pref[MRMG_SPLIT_ROWS]; }
    // the row of run t, from a row at or before it (a thread's runs come in increasing t)
    __device__ __forceinline__ int row_of(int t, int row) const
    {
        while (t >= pref[row + 1]) row++;
        return row;
    }
};

// runs_to_lds (demag.hip) for a split row workgroup of one component: row i of SplitRuns at row pair i/2
template <typename T, int RU>
__device__ __forceinline__ void split_runs_to_lds(const RowRuns& R, const SplitRuns& S, const T* __restrict__ Mg, int np,
                                                  int nx, T* re, T* im)
{
    const int nt = (int)blockDim.x, tid = (int)threadIdx.x, n = S.runs();
    int geo[RU], row[RU], last = 0;
    T v[RU];
    auto fetch = [&](int tb) {
        int g[RU];
#pragma unroll
        for (int u = 0; u < RU; u++) {
            const int t = tb + u * nt;
            if (t < n) {
                last = row[u] = S.row_of(t, last);
                const int q = S.base[row[u]] + t;
                geo[u] = R.geo[q];
                g[u] = R.grain[q];
            }
        }
#pragma unroll
        for (int u = 0; u < RU; u++)
            if (tb + u * nt < n) v[u] = Mg[g[u]];
    };
    fetch(tid);
    const int tot = 2 * LPN(np * nx), per = 16 / (int)sizeof(T), n16 = tot / per;
    uint4* z = reinterpret_cast<uint4*>(re);   // 16-byte aligned: the start of the workgroup's LDS
    for (int i = tid; i < n16; i += nt) z[i] = uint4{0u, 0u, 0u, 0u};
    for (int i = n16 * per + tid; i < tot; i += nt) re[i] = (T)0;
    __syncthreads();
    for (int tb = tid; tb < n; tb += RU * nt) {
        if (tb != tid) fetch(tb);
#pragma unroll
        for (int u = 0; u < RU; u++) {
            if (tb + u * nt >= n) break;
            const int i0 = geo[u] & 0xffff, len = geo[u] >> 16;
            T* dst = (row[u] & 1) ? im : re;
            const int b = (row[u] >> 1) * nx + i0;
            for (int t = 0; t < len; t += MRMG_UF)
#pragma unroll
                for (int j = 0; j < MRMG_UF; j++) dst[LP(b + min(t + j, len - 1))] = v[u];
        }
    }
}

// lds_to_runs for a split row workgroup
template <typename T>
__device__ __forceinline__ void split_lds_to_runs(const RowRuns& R, const SplitRuns& S, double* __restrict__ Hr, int nx,
                                                  const T* re, const T* im)
{
    constexpr int RU = 4;
    const int nt = (int)blockDim.x, n = S.runs();
    int last = 0;
    for (int tb = (int)threadIdx.x; tb < n; tb += RU * nt) {
        int geo[RU], row[RU], to[RU];
#pragma unroll
        for (int u = 0; u < RU; u++)
            if (tb + u * nt < n) {
                last = row[u] = S.row_of(tb + u * nt, last);
                const int q = S.base[row[u]] + tb + u * nt;
                geo[u] = R.geo[q];
                to[u] = R.perm ? R.perm[q] : q;
            }
#pragma unroll
        for (int u = 0; u < RU; u++) {
            if (tb + u * nt >= n) break;
            const int i0 = geo[u] & 0xffff, len = geo[u] >> 16;
            const T* src = (row[u] & 1) ? im : re;
            const int b = (row[u] >> 1) * nx + i0;
            double s = 0.0;
            for (int t = 0; t < len; t += MRMG_UF) {
                T a[MRMG_UF];
#pragma unroll
                for (int j = 0; j < MRMG_UF; j++) a[j] = src[LP(b + min(t + j, len - 1))];
#pragma unroll
                for (int j = 0; j < MRMG_UF; j++) s += (double)(t + j < len ? a[j] : (T)0);
            }
            Hr[to[u]] = s;
        }
    }
}

// The two rows of pair p at kx from their packed transform.
template <typename T>
__device__ __forceinline__ void unpack_pair(const T* re, const T* im, int p, int nx, int kx, C2<T>& a, C2<T>& b)
{
    const int kn = kx == 0 ? 0 : nx - kx;
    const T zr = re[LP(p * nx + kx)], zi = im[LP(p * nx + kx)], nr = re[LP(p * nx + kn)], ni = im[LP(p * nx + kn)];
    a = {(zr + nr) * (T)0.5, (zi - ni) * (T)0.5};
    b = {(zi + ni) * (T)0.5, (nr - zr) * (T)0.5};
}

// The radix-R step of the column transforms over the rows in LDS, and the store: one item
// per (kx, j), consecutive items consecutive y'.  S: the plane's R nxh columns.
template <typename T, int R, int RM>
__device__ __forceinline__ void split_store(const T* re, const T* im, int nx, int nxh, int y0, const RowSplit<T>& rs,
                                            C2<T>* __restrict__ S)
{
    const int ly = __builtin_ctz(rs.Y);
    for (int idx = threadIdx.x; idx < nxh << ly; idx += blockDim.x) {
        const int kx = idx >> ly, j = idx & (rs.Y - 1), y = y0 + j;
        if (y >= rs.L) continue;
        C2<T> v[R];
        if constexpr (RM == 1) {
            C2<T> a, b;
            unpack_pair(re, im, j >> 1, nx, kx, a, b);
            v[0] = (j & 1) ? b : a;
        } else {
#pragma unroll
            for (int q = 0; q < RM; q += 2) unpack_pair(re, im, (j * RM + q) >> 1, nx, kx, v[q], v[q + 1]);
        }
#pragma unroll
        for (int q = RM; q < R; q++) v[q] = {0, 0};
        Dft<T, R, false>::run(v);
#pragma unroll
        for (int r = 0; r < R; r++)
            S[((size_t)r * nxh + kx) * rs.L + y] = r ? cmul(v[r], rs.tw[y * R + r]) : v[r];
    }
}

// The inverse: the radix-R step back to the rows, packed in pairs for the row c2r.
template <typename T, int R, int RM>
__device__ __forceinline__ void split_load(T* re, T* im, int nx, int nxh, int y0, const RowSplit<T>& rs,
                                           const C2<T>* __restrict__ S)
{
    const int ly = __builtin_ctz(rs.Y);
    constexpr int U = R >= 8 ? 1 : 2;   // items whose R loads are in flight together
    const int total = nxh << ly, nt = (int)blockDim.x;
    for (int ib = threadIdx.x; ib < total; ib += U * nt) {
        C2<T> v[U][R];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int idx = min(ib + u * nt, total - 1), kx = idx >> ly, y = min(y0 + (idx & (rs.Y - 1)), rs.L - 1);
#pragma unroll
            for (int r = 0; r < R; r++) v[u][r] = S[((size_t)r * nxh + kx) * rs.L + y];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int idx = ib + u * nt;
            if (idx >= total) break;
            const int kx = idx >> ly, j = idx & (rs.Y - 1), y = min(y0 + j, rs.L - 1);
#pragma unroll
            for (int r = 1; r < R; r++) {
                C2<T> w = rs.tw[y * R + r];
                w.y = -w.y;
                v[u][r] = cmul(v[u][r], w);
            }
            Dft<T, R, true>::run(v[u]);
            const bool edge = kx == 0 || 2 * kx == nx;
            if constexpr (RM == 1) {
                // rows j and j + 1 of a pair are two items: each adds its part of z = A + iB
                C2<T> a = v[u][0];
                if (edge) a.y = 0;
                C2<T> b;
                b.x = __shfl_xor(a.x, 1);
                b.y = __shfl_xor(a.y, 1);
                if (j & 1) continue;
                const int p = j >> 1;
                re[LP(p * nx + kx)] = a.x - b.y;
                im[LP(p * nx + kx)] = a.y + b.x;
                if (kx > 0 && nx - kx != kx) {
                    re[LP(p * nx + nx - kx)] = a.x + b.y;
                    im[LP(p * nx + nx - kx)] = b.x - a.y;
                }
            } else {
#pragma unroll
                for (int q = 0; q < RM; q += 2) {
                    C2<T> a = v[u][q], b = v[u][q + 1];
                    if (edge) { a.y = 0; b.y = 0; }
                    const int p = (j * RM + q) >> 1;
                    re[LP(p * nx + kx)] = a.x - b.y;
                    im[LP(p * nx + kx)] = a.y + b.x;
                    if (kx > 0 && nx - kx != kx) {
                        re[LP(p * nx + nx - kx)] = a.x + b.y;
                        im[LP(p * nx + nx - kx)] = b.x - a.y;
                    }
                }
            }
        }
    }
}

// Row r2c of the rows of rs.Y values of y' of one (component, layer), and the radix-R step of
// the column transforms, as k_rowT_fwd otherwise.  tab: one launch over a batch of contexts,
// blockIdx.z the member, or null for the context's own operands (one).  A kernel of its own:
// as a branch of k_rowT_fwd its registers cost the other kernel occupancy (2048x2048x8 FP64:
// 528 us against 430).
template <typename T, int E>
__global__ void __launch_bounds__(256) k_rowS_fwd(DemagOps<T> one, const DemagOps<T>* __restrict__ tab, int nx, int ny,
                                                  int sy, int nl, int nxh, int TY, FFTPlan px,
                                                  const C2<T>* __restrict__ tw, RowSplit<T> rs)
{
    const DemagOps<T> o = tab ? tab[blockIdx.z] : one;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ SplitRuns sr;
    const int B = TY / 2, nyb = (rs.L + rs.Y - 1) / rs.Y;
    T* re = reinterpret_cast<T*>(smem_raw);
    T* im = re + LPN(B * nx);
    const int L = xcd_remap(blockIdx.x, gridDim.x);
    if (L >= nyb * 3 * nl) return;
    const int y0 = (L % nyb) * rs.Y, kc = L / nyb, k = kc / 3, c = kc - 3 * k;   // kc = k*3 + c
    sr.init(o.R, k, ny, y0, rs);
    __syncthreads();
    split_runs_to_lds<T, 4>(o.R, sr, o.Mg + (size_t)c * o.G, B, nx, re, im);
    __syncthreads();
    lds_fft<T, E, false, true>(re, im, B, px, tw);
    C2<T>* dst = o.S1 + (size_t)kc * nxh * sy;
    if (rs.Rm == rs.R) {
        if (rs.R == 8) split_store<T, 8, 8>(re, im, nx, nxh, y0, rs, dst);
        else if (rs.R == 4) split_store<T, 4, 4>(re, im, nx, nxh, y0, rs, dst);
        else split_store<T, 2, 2>(re, im, nx, nxh, y0, rs, dst);
    } else {
        if (rs.R == 8) split_store<T, 8, 4>(re, im, nx, nxh, y0, rs, dst);
        else if (rs.R == 4) split_store<T, 4, 2>(re, im, nx, nxh, y0, rs, dst);
        else split_store<T, 2, 1>(re, im, nx, nxh, y0, rs, dst);
    }
}

// The inverse of k_rowS_fwd with the run sums of k_rowT_inv.  CELLS: the cell field into
// Hcell (mx: the media row length) instead.
template <typename T, int E, bool CELLS>
__global__ void __launch_bounds__(256) k_rowS_inv(DemagOps<T> one, const DemagOps<T>* __restrict__ tab, int nx, int ny,
                                                  int sy, int mx, int nl, int nxh, int TY, FFTPlan px,
                                                  const C2<T>* __restrict__ tw, RowSplit<T> rs)
{
    const DemagOps<T> o = tab ? tab[blockIdx.z] : one;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ SplitRuns sr;
    const int B = TY / 2, nyb = (rs.L + rs.Y - 1) / rs.Y;
    T* re = reinterpret_cast<T*>(smem_raw);
    T* im = re + LPN(B * nx);
    const int L = xcd_remap(blockIdx.x, gridDim.x);
    if (L >= nyb * 3 * nl) return;
    const int y0 = (L % nyb) * rs.Y, kc = L / nyb, k = kc / 3, c = kc - 3 * k;
    const C2<T>* src = o.S2 + (size_t)kc * nxh * sy;
    if (!CELLS) sr.init(o.R, k, ny, y0, rs);   // synchronised with the spectra
    if (rs.Rm == rs.R) {
        if (rs.R == 8) split_load<T, 8, 8>(re, im, nx, nxh, y0, rs, src);
        else if (rs.R == 4) split_load<T, 4, 4>(re, im, nx, nxh, y0, rs, src);
        else split_load<T, 2, 2>(re, im, nx, nxh, y0, rs, src);
    } else {
        if (rs.R == 8) split_load<T, 8, 4>(re, im, nx, nxh, y0, rs, src);
        else if (rs.R == 4) split_load<T, 4, 2>(re, im, nx, nxh, y0, rs, src);
        else split_load<T, 2, 1>(re, im, nx, nxh, y0, rs, src);
    }
    __syncthreads();
    lds_fft<T, E, true, true>(re, im, B, px, tw);
    if (!CELLS) {
        split_lds_to_runs<T>(o.R, sr, o.Hr + (size_t)c * o.R.nruns, nx, re, im);
        return;
    }
    T* hc = o.Hcell + ((size_t)c * nl + k) * (size_t)mx * ny;
    for (int idx = threadIdx.x; idx < rs.Rm * rs.Y * mx; idx += blockDim.x) {
        const int i = idx / mx, x = idx - i * mx, j = i / rs.Rm, q = i - j * rs.Rm;
        if (y0 + j < rs.L) hc[(size_t)(y0 + j + q * rs.L) * mx + x] = ((i & 1) ? im : re)[LP((i >> 1) * nx + x)];
    }
}

template <int E>
static int rowS(bool inv, bool cells, dim3 g, dim3 b, size_t lds, hipStream_t s, const DemagOps<double>& o,
                const DemagOps<double>* tab, const mrmg_ctx* c, int TY, const FFTPlan& px, const C2<double>* tw,
                const RowSplit<double>& rs)
{
    if (!inv)
        hipLaunchKernelGGL((k_rowS_fwd<double, E>), g, b, lds, s, o, tab, c->fx, c->ny, c->fy, c->nl, c->nxh, TY, px, tw,
                           rs);
    else if (cells)
        hipLaunchKernelGGL((k_rowS_inv<double, E, true>), g, b, lds, s, o, tab, c->fx, c->ny, c->fy, c->nx, c->nl,
                           c->nxh, TY, px, tw, rs);
    else
        hipLaunchKernelGGL((k_rowS_inv<double, E, false>), g, b, lds, s, o, tab, c->fx, c->ny, c->fy, c->nx, c->nl,
                           c->nxh, TY, px, tw, rs);
    HIPCHK(hipGetLastError());
    return MRMG_OK;
}

// as lds_attr_colp; SplitRuns takes 132 bytes of the 160 KB
template <int E>
static int rowS_attr()
{
    const hipFuncAttribute a = hipFuncAttributeMaxDynamicSharedMemorySize;
    const int lds = 160 * 1024 - 256;
    HIPCHK(hipFuncSetAttribute((const void*)k_rowS_fwd<double, E>, a, lds));
    HIPCHK(hipFuncSetAttribute((const void*)k_rowS_inv<double, E, false>, a, lds));
    HIPCHK(hipFuncSetAttribute((const void*)k_rowS_inv<double, E, true>, a, lds));
    return MRMG_OK;
}

template <>
int Engine<double>::lds_attr_rowS()
{
    RCHK(rowS_attr<4>()); RCHK(rowS_attr<8>()); RCHK(rowS_attr<16>()); RCHK(rowS_attr<32>()); RCHK(rowS_attr<64>());
    return MRMG_OK;
}

template <>
int Engine<double>::launch_rowS(bool inv, dim3 g, dim3 b)
{
    const DemagOps<double> o = ops();
#define ROWS(E) rowS<E>(inv, cells_out, g, b, lds_rowT, c->stream, o, btab, c, TYr_eff(), prow, twx.p, row_split())
    if (maxb_rowT <= 4) return ROWS(4);
    if (maxb_rowT <= 8) return ROWS(8);
    if (maxb_rowT <= 16) return ROWS(16);
    if (maxb_rowT <= 32) return ROWS(32);
    return ROWS(64);
#undef ROWS
}
