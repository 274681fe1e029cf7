// ops.hip -- device-resident operator applies: staging, pair-kernel dispatch,
// epilogues (AvT, SL diagonal, mass, alpha/beta) and the incident waves.
#include <algorithm>
#include <atomic>
#include <numeric>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <utility>

#include "ops.hpp"
#include "stage.hpp"

namespace baemm {

// --------------------------------------------------------------- helpers

static inline int next_pow2(int x)
{
    int p = 1;
    while (p < x) p <<= 1;
    return p;
}

// Padded chunk width of the plain kernels (instantiated 4..64).
int wcsp_plain(int wcs) { return std::max(4, next_pow2(wcs)); }
// Padded chunk width of the MFMA kernel (16, 32 or 64: 2*WCSP real columns
// must fill 32-column MFMA blocks).
int wcsp_mixed(int wcs) { return std::max(16, next_pow2(wcs)); }

// --------------------------------------------------------------- staging

// b = Av B row by row (av_elem).
template <int BT>
__global__ void av_gather_kernel(const int4* __restrict__ tris, const float* __restrict__ area, int nt,
                                 int64_t total, const void* __restrict__ Bv, int64_t ldB, int wcs, int WCSP,
                                 int ldb, float2* __restrict__ b)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    b[idx] = av_elem<BT>(tris, area, nt, Bv, ldB, wcs, WCSP, ldb, idx);
}

// b[r][q*WCSP+kk] = (conj?) G[r][q*wcs+kk] for r < nrows, zero padding.
template <int BT>
__global__ void stage_rows_kernel(int nrows, int64_t total, const void* __restrict__ Gv, int64_t ldG, int wcs,
                                  int WCSP, int ldb, int conj, float2* __restrict__ b)
{
    using T = typename Elem<BT>::type;
    const T* G = static_cast<const T*>(Gv);
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const int r = (int)(idx / ldb);
    const int pc = (int)(idx % ldb);
    const int q = pc / WCSP, kk = pc % WCSP;
    float2 out = make_float2(0.f, 0.f);
    if (r < nrows && kk < wcs) {
        const double2 v = to_d2(G[(int64_t)r * ldG + q * wcs + kk]);
        out = make_float2((float)v.x, (float)(conj ? -v.y : v.y));
    }
    b[idx] = out;
}

// Per-column max of |re|, |im| (positive floats order like their bit patterns).
// Block: 4 row lanes x 64 columns; blocks stride over rows; one atomicMax per
// column and block.  colmax must be zero on entry.
__global__ __launch_bounds__(256) void colmax_kernel(const float2* __restrict__ b, int nrows, int ldb,
                                                     unsigned* __restrict__ colmax)
{
    __shared__ float sm[4][64];
    const int c = threadIdx.x & 63, rl = threadIdx.x >> 6;
    for (int c0 = 0; c0 < ldb; c0 += 64) {
        float m = 0.0f;
        if (c0 + c < ldb)
            for (int r = blockIdx.x * 4 + rl; r < nrows; r += gridDim.x * 4) {
                const float2 v = b[(int64_t)r * ldb + c0 + c];
                m = fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y)));
            }
        sm[rl][c] = m;
        __syncthreads();
        if (rl == 0 && c0 + c < ldb) {
            m = fmaxf(fmaxf(sm[0][c], sm[1][c]), fmaxf(sm[2][c], sm[3][c]));
            atomicMax(&colmax[c0 + c], __float_as_uint(m));
        }
        __syncthreads();
    }
}

// b = Av B (av_elem) and the maxima of |re|, |im| over each column of b
// (positive floats order like their bit patterns).  Threads stride over the
// elements by the grid's thread count, a multiple of ldb, so each thread stays
// in one column: its running maximum, then per block in LDS (ldb entries of
// dynamic shared memory), then one atomicMax per column and block.  colmax
// must be zero on entry.
// Largest grid of av_gather_max_kernel (more blocks: the separate gather and
// colmax_kernel).
constexpr int64_t kGatherMaxBlocks = 512;

template <int BT>
__global__ __launch_bounds__(256) void av_gather_max_kernel(const int4* __restrict__ tris,
                                                            const float* __restrict__ area, int nt, int64_t total,
                                                            const void* __restrict__ Bv, int64_t ldB, int wcs,
                                                            int WCSP, int ldb, float2* __restrict__ b,
                                                            unsigned* __restrict__ colmax)
{
    extern __shared__ unsigned s_max[];
    for (int c = threadIdx.x; c < ldb; c += blockDim.x) s_max[c] = 0u;
    __syncthreads();
    const int64_t first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float m = 0.0f;
    for (int64_t idx = first; idx < total; idx += (int64_t)gridDim.x * blockDim.x) {
        const float2 v = av_elem<BT>(tris, area, nt, Bv, ldB, wcs, WCSP, ldb, idx);
        b[idx] = v;
        m = fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y)));
    }
    if (m > 0.0f) atomicMax(&s_max[(int)(first % ldb)], __float_as_uint(m));
    __syncthreads();
    for (int c = threadIdx.x; c < ldb; c += blockDim.x)
        if (s_max[c]) atomicMax(&colmax[c], s_max[c]);
}

// B-operand of the MFMA kernel (split_elem) with the column scales
// s_pc = col_scale(colmax[pc]), powers of two that put max |s b| in [2^13, 2^14);
// the first ncols threads also write unscale[pc] = 1 / s_pc (ncols < the element
// count).  The A scales of the chunks come off in the FP64 factors of the
// epilogues: their product with s_pc can leave the FP32 range.
__global__ void split_kernel(const float2* __restrict__ b, int ldb, int nst, int WCSP, int K,
                             const unsigned* __restrict__ colmax, int ncols, float* __restrict__ unscale, uint4* __restrict__ bop)
{
    const int NCB = 2 * WCSP / 32;
    const int64_t total = (int64_t)K * nst * NCB * 64;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    if (idx < ncols) {
        const int pc = (int)idx;
        unscale[pc] = 1.0f / col_scale(colmax[pc]);
    }
    split_elem(b, ldb, nst, WCSP, idx, [&](int pc) { return col_scale(colmax[pc]); }, bop);
}

// out[j] = s * nrm[j] for j < n: source normals carrying the common scale of
// the non-adjoint MFMA kernel values (out NULL: none); zero[j] = 0 for j < nzero.
__global__ void scale_nrm_kernel(const float4* __restrict__ nrm, int n, float s, float4* __restrict__ out,
                                 unsigned* __restrict__ zero, int nzero)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < nzero) zero[j] = 0u;
    if (j >= n || !out) return;
    const float4 v = nrm[j];
    out[j] = make_float4(s * v.x, s * v.y, s * v.z, v.w);
}

// B-operand of the FP32 MFMA kernel: for (chunk, step, col-block) and lane,
// the 8 FP32 values of MFMAs m = 0..7 (two 16-byte parts), in the order of the
// FP16 operand of split_kernel: rows (source 4 (lane / 32) + m / 2, re | im) of
// [[br, bi], [-bi, br]], unscaled.
__global__ void stage_f32_kernel(const float2* __restrict__ b, int ldb, int nst, int WCSP, int K,
                                 uint4* __restrict__ bop)
{
    const int NCB = 2 * WCSP / 32;
    const int64_t total = (int64_t)K * nst * NCB * 64;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= total) return;
    const int lane = (int)(idx % 64);
    int64_t rest = idx / 64;
    const int cb = (int)(rest % NCB);
    rest /= NCB;
    const int st = (int)(rest % nst);
    const int q = (int)(rest / nst);
    const int g = lane >> 5;
    const int c = cb * 32 + (lane & 31);
    const bool imcol = c >= WCSP;
    const int kk = imcol ? c - WCSP : c;
    const int pc = q * WCSP + kk;
    float e[8];
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
        const int j = 8 * st + 4 * g + jj;
        const float2 v = b[(int64_t)j * ldb + pc];
        e[2 * jj] = imcol ? v.y : v.x;
        e[2 * jj + 1] = imcol ? v.x : -v.y;
    }
    const int64_t base = ((((int64_t)q * nst + st) * NCB + cb) * 2) * 64 + lane;
    bop[base] = make_uint4(__float_as_uint(e[0]), __float_as_uint(e[1]), __float_as_uint(e[2]), __float_as_uint(e[3]));
    bop[base + 64] = make_uint4(__float_as_uint(e[4]), __float_as_uint(e[5]), __float_as_uint(e[6]), __float_as_uint(e[7]));
}

// out = (the largest float, 0), the starts of a minimum and a maximum as bits.
__global__ void range_init_kernel(unsigned* __restrict__ out)
{
    if (threadIdx.x < 2) out[threadIdx.x] = threadIdx.x ? 0u : 0x7f7fffffu;
}

// Minimum (out[0]) and maximum (out[1], not SELF) squared distance between the
// targets x_i (i < ntgt) and the centroids y_j (j < nt); they set the A scale of the
// split-FP16 MFMA path.  SELF: the targets are the centroids, distinct ones, and
// each pair is taken once, blocks with their sources all before their targets return.
// One target per thread, the centroids of segment blockIdx.y (seg_len of them, a
// multiple of 256); the results (non-negative floats) are reduced as bits.  Bound by
// vector-ALU issue: 20,480 centroids 130 us with every pair twice, 91 with
// each once (81,920: 1.81 and 1.16 ms).
template <bool SELF>
__global__ __launch_bounds__(256) void rmin_kernel(const float4* __restrict__ tgt, int ntgt,
                                                   const float4* __restrict__ mid, int nt, int seg_len,
                                                   unsigned* __restrict__ out)
{
    __shared__ float4 s[256];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const float4 x = tgt[min(i, ntgt - 1)];
    float m = 3.0e38f, M = 0.0f;
    const int j0 = blockIdx.y * seg_len, j1 = min(nt, j0 + seg_len), tile = blockIdx.x * 256;
    if (SELF && j1 <= tile) return;
    for (int jb = SELF ? max(j0, tile) : j0; jb < j1; jb += 256) {
        __syncthreads();
        if (jb + threadIdx.x < j1) s[threadIdx.x] = mid[jb + threadIdx.x];
        __syncthreads();
        const int jn = min(256, j1 - jb);
        // (the target itself is in its own tile's block only)
        const int own = SELF && jb == tile ? (int)threadIdx.x : -1;
        for (int jj = 0; jj < jn; ++jj) {
            const float4 y = s[jj];
            const float d0 = y.x - x.x, d1 = y.y - x.y, d2 = y.z - x.z;
            const float r2 = fmaf(d0, d0, fmaf(d1, d1, d2 * d2));
            if (jj != own) m = fminf(m, r2);
            if (!SELF) M = fmaxf(M, r2);
        }
    }
    if (i >= ntgt) {   // a repeated last target, whose own centroid was not left out
        m = 3.0e38f;
        M = 0.0f;
    }
    for (int off = 32; off > 0; off >>= 1) {
        m = fminf(m, __shfl_xor(m, off));
        M = fmaxf(M, __shfl_xor(M, off));
    }
    // one value per block, and an atomic only where it may count (one per wave
    // on the two words took 0.33 ms at 20,480 triangles)
    __shared__ float sm[4], sM[4];
    if ((threadIdx.x & 63) == 0) {
        sm[threadIdx.x >> 6] = m;
        sM[threadIdx.x >> 6] = M;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        m = fminf(fminf(sm[0], sm[1]), fminf(sm[2], sm[3]));
        M = fmaxf(fmaxf(sM[0], sM[1]), fmaxf(sM[2], sM[3]));
        const volatile unsigned* cur = out;
        if (__float_as_uint(m) < cur[0]) atomicMin(&out[0], __float_as_uint(m));
        if (!SELF && __float_as_uint(M) > cur[1]) atomicMax(&out[1], __float_as_uint(M));
    }
}

// --------------------------------------------------------------- epilogues

// The boundary epilogue, one vertex per lpv lanes (epi_vertex).
template <int BT, int CT, bool TSUM>
__global__ __launch_bounds__(256) void bdr_epilogue_kernel(EpiArgs a, int lpv)
{
    const int lane = threadIdx.x & (lpv - 1);
    const int v = blockIdx.x * (256 / lpv) + threadIdx.x / lpv;
    if (v >= a.nv) return;
    epi_vertex<BT, CT, TSUM>(a, v, lane, lpv);
}

// Factors per wave-number chunk the MFMA near-field partials are multiplied by.
struct ChunkRot {
    double r[64], i[64];
};

// Work-groups of the segment sums: SW threads to an element, kSegElems<SW>
// elements to a work-group (one wave's up to SW = 16, then a quarter of it).
template <int SW>
constexpr int kSegElems = SW == 1 ? 256 : (SW > 16 ? 16 : 64);
template <int SW>
constexpr int kSegThreads = SW == 1 ? 256 : SW * kSegElems<SW>;

// Sum over the segments s (FP64) of the partials pp[s * stride] and pp[s * stride
// + im], shared by the SW threads of an element: thread w sums s = w, w + SW,
// ..., eight loads issued before the first is added, and the first adds the
// others' sums in order (true there).  More threads where there are many
// segments and few elements, whose sums are otherwise one long chain of loads on
// few CUs: a far field of 256 directions, 32 columns and 600 segments 45 us
// with one, 9.5 with 16; the triangles of a 1,280-triangle mesh, 16 columns and 20
// segments 5.1 us, 3.8 with four; a far field of 81 directions, two columns and 320
// segments 23 us with 16, 9.9 with 64.
template <int SW>
__device__ __forceinline__ bool segment_sum(const float* __restrict__ pp, int64_t stride, int im, int S, double& pr,
                                            double& pi)
{
    constexpr int EL = kSegElems<SW>;
    const int w = SW > 1 ? (int)(threadIdx.x / EL) : 0;
    pr = pi = 0.0;
    for (int s0 = w; s0 < S; s0 += EPI_SEG * SW) {
        float xr[EPI_SEG], xi[EPI_SEG];
#pragma unroll
        for (int j = 0; j < EPI_SEG; ++j) {
            const int64_t o = (int64_t)min(s0 + j * SW, S - 1) * stride;
            xr[j] = pp[o];
            xi[j] = pp[o + im];
        }
#pragma unroll
        for (int j = 0; j < EPI_SEG; ++j)
            if (s0 + j * SW < S) {
                pr += (double)xr[j];
                pi += (double)xi[j];
            }
    }
    if constexpr (SW > 1) {
        // the threads of a wave that share an element, then the waves
        for (int d = EL; d < 64; d *= 2) {
            pr += __shfl_xor(pr, d);
            pi += __shfl_xor(pi, d);
        }
        constexpr int NW = SW * EL / 64;
        __shared__ double2 sm[NW][EL];
        const int l = threadIdx.x & (EL - 1);
        if ((threadIdx.x & 63) < EL) sm[threadIdx.x >> 6][l] = make_double2(pr, pi);
        __syncthreads();
        if (w > 0) return false;
#pragma unroll
        for (int u = 1; u < NW; ++u) {
            pr += sm[u][l].x;
            pi += sm[u][l].y;
        }
    }
    return true;
}
// The element of a thread of a segment_sum<SW> launch.
template <int SW>
__device__ __forceinline__ int64_t segment_element()
{
    return (int64_t)blockIdx.x * kSegElems<SW> + threadIdx.x % kSegElems<SW>;
}
// Threads per element: about eight segments to a thread while the launch has
// fewer than 4,096 waves.
static int segment_threads(int64_t elements, int S)
{
    int sw = 1;
    while (sw < 64 && S > 8 * sw && elements * sw * 4 <= 64 * 4096) sw *= 4;
    return sw;
}
// Calls go with segment_threads(elements, S) as a compile-time constant.
template <class F>
static void with_segment_threads(int64_t elements, int S, const F& go)
{
    switch (segment_threads(elements, S)) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 16: go(std::integral_constant<int, 16>{}); break;
    default: go(std::integral_constant<int, 64>{}); break;
    }
}

// F[i][k] = alpha * rot_q * unscale_k * sum_s part_s[i][k] + beta * F[i][k]
// (far field, potential; unscale null and rot = 1 for the FP32 kernels).
template <int CT, int SW>
__global__ __launch_bounds__(kSegThreads<SW>) void rows_epilogue_kernel(
    int nrows, int W, int wcs, int WCSP, int S, int64_t seg_stride, int ldp, const float* __restrict__ part, double ar,
    double ai, double br, double bi, void* Cv, int64_t ldC, const float* __restrict__ unscale, ChunkRot rot)
{
    using TC = typename Elem<CT>::type;
    const int64_t idx = segment_element<SW>();
    const bool in = idx < (int64_t)nrows * W;
    if (SW == 1 && !in) return;
    const int r = in ? (int)(idx / W) : 0, k = in ? (int)(idx % W) : 0;
    const int q = k / wcs, kk = k % wcs;
    double pr, pi;
    if (!segment_sum<SW>(part + (int64_t)r * ldp + q * 2 * WCSP + kk, seg_stride, WCSP, S, pr, pi) || !in) return;
    if (unscale) {
        const double us = (double)unscale[q * WCSP + kk];
        pr *= us;
        pi *= us;
    }
    {
        const double rr = rot.r[q], ri = rot.i[q];
        const double tr = pr * rr - pi * ri;
        pi = pr * ri + pi * rr;
        pr = tr;
    }
    TC* C = static_cast<TC*>(Cv);
    TC& dst = C[(int64_t)r * ldC + k];
    double outr = ar * pr - ai * pi, outi = ar * pi + ai * pr;
    if (br != 0.0 || bi != 0.0) {
        const double2 c = to_d2(dst);
        outr += br * c.x - bi * c.y;
        outi += br * c.y + bi * c.x;
    }
    from_d2(dst, make_double2(outr, outi));
}

// Incident-wave values per triangle written as a single "segment" partial
// (IncidentWaveKernel_Plane.hpp:190-233, IncidentWaveKernel_Radial.hpp:5-57):
//   plane : (c1 + c2 i kappa (d.n)) exp(i kappa d.x)
//   radial: (c1 + c2 (-(n.delta)/R^2 + i kappa (n.delta)/R)) exp(i kappa R) / (4 pi R)
struct IncArgs {
    int nt, W, wcs, WCSP, ldp, radial;
    const float4* mid;
    const float4* nrm;
    float* part;
    float dirs[64][3];
    float kap[64], c1r[64], c1i[64], c2r[64], c2i[64];
};

__global__ void incident_kernel(IncArgs a)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)a.nt * a.W) return;
    const int t = (int)(idx / a.W), k = (int)(idx % a.W);
    const int q = k / a.wcs, j = k % a.wcs;
    const float4 x = a.mid[t], n = a.nrm[t];
    const double dx = a.dirs[j][0], dy = a.dirs[j][1], dz = a.dirs[j][2];
    const double kap = a.kap[q];
    double ur, ui;
    if (!a.radial) {
        const double ph = kap * (x.x * dx + x.y * dy + x.z * dz);
        const double dn = kap * (n.x * dx + n.y * dy + n.z * dz);
        const double fr = a.c1r[q] - a.c2i[q] * dn, fi = a.c1i[q] + a.c2r[q] * dn;
        const double cs = cos(ph), sn = sin(ph);
        ur = fr * cs - fi * sn;
        ui = fr * sn + fi * cs;
    } else {
        const double e0 = x.x - dx, e1 = x.y - dy, e2 = x.z - dz;
        const double R = sqrt(e0 * e0 + e1 * e1 + e2 * e2);
        const double nd = n.x * e0 + n.y * e1 + n.z * e2;
        const double A = 1.0 / (4.0 * M_PI * R);
        const double Br = -nd / (R * R), Bi = kap * nd / R;
        const double fr = A * (a.c1r[q] + a.c2r[q] * Br - a.c2i[q] * Bi);
        const double fi = A * (a.c1i[q] + a.c2r[q] * Bi + a.c2i[q] * Br);
        const double cs = cos(kap * R), sn = sin(kap * R);
        ur = fr * cs - fi * sn;
        ui = fr * sn + fi * cs;
    }
    float* out = a.part + (int64_t)t * a.ldp + q * 2 * a.WCSP + j;
    out[0] = (float)ur;
    out[a.WCSP] = (float)ui;
}

// --------------------------------------------------------------- dispatch

static void p0_record(Handle& h, const float2* b, int ldb, int WCSP, const EpiArgs* ea);

CoefPack make_pack(const Params& p, int q0, int kg, const float* scale_per_chunk, const cdouble* rot)
{
    CoefPack cp{};
    for (int g = 0; g < kg; ++g) {
        const float s = scale_per_chunk ? scale_per_chunk[q0 + g] : 1.0f;
        cp.c[g] = chunk_coefs(p, q0 + g, 1, s, rot)[0];
    }
    return cp;
}

#define PLAIN_CASES(OP, ADJ)                                                                             \
    if (WCSP == 4 && KG == 1) return &pair_plain_kernel<OP, 4, 1, ADJ>;                               \
    if (WCSP == 4 && KG == 2) return &pair_plain_kernel<OP, 4, 2, ADJ>;                               \
    if (WCSP == 8 && KG == 1) return &pair_plain_kernel<OP, 8, 1, ADJ>;                               \
    if (WCSP == 8 && KG == 2) return &pair_plain_kernel<OP, 8, 2, ADJ>;                               \
    if (WCSP == 16 && KG == 1) return &pair_plain_kernel<OP, 16, 1, ADJ>;                             \
    if (WCSP == 16 && KG == 2) return &pair_plain_kernel<OP, 16, 2, ADJ>;                             \
    if (WCSP == 32 && KG == 1) return &pair_plain_kernel<OP, 32, 1, ADJ>;                             \
    if (WCSP == 32 && KG == 2) return &pair_plain_kernel<OP, 32, 2, ADJ>;                             \
    if (WCSP == 64 && KG == 1) return &pair_plain_kernel<OP, 64, 1, ADJ>;

using PlainFn = void (*)(const float4*, const float4*, int, const float4*, const float4*, int, const float2*, int,
                         CoefPack, float*, int64_t, int, int, int, int, const int*);

static PlainFn plain_fn(int op, bool adj, int WCSP, int KG)
{
    if (op == OP_BDR && adj) { PLAIN_CASES(OP_BDR, true) }
    if (op == OP_BDR && !adj) { PLAIN_CASES(OP_BDR, false) }
    if (op == OP_NEAR) { PLAIN_CASES(OP_NEAR, false) }
    if (op == OP_FAR) { PLAIN_CASES(OP_FAR, false) }
    if (op == OP_HERG) { PLAIN_CASES(OP_HERG, false) }
    throw ArgError{"internal: no plain kernel instance"};
}

using MixedFn = void (*)(const float4*, int, int, const float4*, const float4*, int, const uint4*, int, CoefPack,
                         float*, int64_t, int, int, StepRange, const int*);

static MixedFn mixed_ws_fn(bool adj, int WCSP, int KG, bool f32, bool tn = false)
{
#define MIXWS(W_, K_)                                                                                    \
    if (WCSP == W_ && KG == K_) {                                                                        \
        if (tn) return f32 ? &bdr_mixed_ws_kernel<W_, K_, false, true, true> : &bdr_mixed_ws_kernel<W_, K_, false, false, true>; \
        if (f32) return adj ? &bdr_mixed_ws_kernel<W_, K_, true, true> : &bdr_mixed_ws_kernel<W_, K_, false, true>; \
        return adj ? &bdr_mixed_ws_kernel<W_, K_, true> : &bdr_mixed_ws_kernel<W_, K_, false>;           \
    }
    MIXWS(16, 1)
    MIXWS(16, 2)
    MIXWS(32, 1)
    MIXWS(32, 2)
    MIXWS(64, 1)
#undef MIXWS
    throw ArgError{"internal: no wave-specialised mixed kernel instance"};
}

// Coefficient form of chunk c for the single-wave kernel (its mixed_vals_q):
// 1 Re c1 = 0, 2 Im c1 = 0, else 0.
static int coef_form(const ChunkCoef& c) { return c.c1r == 0.0f ? 1 : (c.c1i == 0.0f ? 2 : 0); }

// The single-wave kernel for KG chunks with coefficients cp (NULL: the
// general form).  Without the adjoint term, one or two chunks take their own
// coefficient forms, four chunks a form they share; else the general form.
static MixedFn mixed_fn(bool adj, int WCSP, int KG, const CoefPack* cp = nullptr, bool tn = false)
{
    if (tn) {
        // the target-normal form: the general coefficient form, or every chunk
        // without Re c1 (the Dirichlet-to-Neumann rows (1/2, -i kappa, 0, 1))
        bool re0 = cp != nullptr;
        for (int q = 0; cp && q < KG; ++q) re0 = re0 && coef_form(cp->c[q]) == 1;
#define MIXTN(W_, K_, F_)                                                                      \
    if (WCSP == W_ && KG == K_)                                                                \
        return re0 ? &bdr_mixed_kernel<W_, K_, false, F_, true> : &bdr_mixed_kernel<W_, K_, false, 0, true>;
        MIXTN(16, 1, 1)
        MIXTN(16, 2, 4)
        MIXTN(16, 4, 40)
        MIXTN(32, 1, 1)
        MIXTN(32, 2, 4)
        MIXTN(64, 1, 1)
#undef MIXTN
        throw ArgError{"internal: no mixed kernel instance"};
    }
    int forms = 0;
    if (cp && !adj) {
        if (KG <= 2) {
            for (int q = KG - 1; q >= 0; --q) forms = 3 * forms + coef_form(cp->c[q]);
        } else {
            const int f = coef_form(cp->c[0]);
            bool same = true;
            for (int q = 1; q < KG; ++q) same = same && coef_form(cp->c[q]) == f;
            forms = same ? f * 40 : 0;   // 40 = 1 + 3 + 9 + 27: form f in every digit
        }
    }
#define MIXF1(W_)                                                     \
    if (WCSP == W_ && KG == 1) {                                      \
        if (adj) return &bdr_mixed_kernel<W_, 1, true>;               \
        if (forms == 1) return &bdr_mixed_kernel<W_, 1, false, 1>;    \
        if (forms == 2) return &bdr_mixed_kernel<W_, 1, false, 2>;    \
        return &bdr_mixed_kernel<W_, 1, false, 0>;                    \
    }
#define MIXF2(W_)                                                     \
    if (WCSP == W_ && KG == 2) {                                      \
        if (adj) return &bdr_mixed_kernel<W_, 2, true>;               \
        switch (forms) {                                              \
            case 1: return &bdr_mixed_kernel<W_, 2, false, 1>;        \
            case 2: return &bdr_mixed_kernel<W_, 2, false, 2>;        \
            case 3: return &bdr_mixed_kernel<W_, 2, false, 3>;        \
            case 4: return &bdr_mixed_kernel<W_, 2, false, 4>;        \
            case 5: return &bdr_mixed_kernel<W_, 2, false, 5>;        \
            case 6: return &bdr_mixed_kernel<W_, 2, false, 6>;        \
            case 7: return &bdr_mixed_kernel<W_, 2, false, 7>;        \
            case 8: return &bdr_mixed_kernel<W_, 2, false, 8>;        \
            default: return &bdr_mixed_kernel<W_, 2, false, 0>;       \
        }                                                             \
    }
    MIXF1(16)
    MIXF2(16)
    MIXF1(32)
    MIXF2(32)
    MIXF1(64)
#undef MIXF1
#undef MIXF2
    if (WCSP == 16 && KG == 4) {
        if (adj) return &bdr_mixed_kernel<16, 4, true>;
        if (forms == 40) return &bdr_mixed_kernel<16, 4, false, 40>;
        if (forms == 80) return &bdr_mixed_kernel<16, 4, false, 80>;
        return &bdr_mixed_kernel<16, 4, false, 0>;
    }
    throw ArgError{"internal: no mixed kernel instance"};
}

static int pick_kg(int WCSP, int remaining, bool mixed)
{
    const int maxkg = std::max(1, kMaxCols / WCSP);
    const int lim = mixed ? 4 : 2;
    int kg = 1;
    while (kg * 2 <= std::min({maxkg, remaining, lim})) kg *= 2;
    return kg;
}

// Number of source segments: enough work-groups to fill 256 CUs several times,
// and at most kMaxSegSources sources per segment, which bounds the length of
// each FP32 accumulation (the segment partials are summed in FP64).
constexpr int kMaxSegSources = 32768;
static int min_segments(int64_t nsrc) { return (int)((nsrc + kMaxSegSources - 1) / kMaxSegSources); }
static int choose_segments(const Handle& h, int tiles, int max_seg, int64_t nsrc, int target = 2048)
{
    const int min_seg = min_segments(nsrc);
    const int want = h.segments > 0 ? h.segments : (target + tiles - 1) / tiles;
    return std::max(1, std::min(std::max(want, min_seg), max_seg));
}

// CUs of the current device.
static int cu_count()
{
    static std::atomic<int> cache[64];   // per device (the query takes about 1 us)
    int dev = 0, cus = 256;
    BAEMM_HIP(hipGetDevice(&dev));
    if (dev >= 0 && dev < 64 && (cus = cache[dev].load(std::memory_order_relaxed)) > 0) return cus;
    BAEMM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    cus = std::max(1, cus);
    if (dev >= 0 && dev < 64) cache[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

// Work-groups of kernel fn (bs threads each) resident on the current device at
// once: the occupancy per CU times the CU count, cached per device and kernel.
static int resident_blocks(const void* fn, int bs)
{
    static std::mutex mtx;
    static std::map<std::pair<int, const void*>, int> cache;
    int dev = 0;
    BAEMM_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mtx);
    auto it = cache.find({dev, fn});
    if (it != cache.end()) return it->second;
    int per_cu = 0, cus = 0;
    BAEMM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, bs, 0));
    BAEMM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int r = std::max(1, per_cu * cus);
    cache[{dev, fn}] = r;
    return r;
}

// Automatic segment count of a launch of tiles x S work-groups whose segments
// split nst source units (8-source steps or 64-source blocks): among the
// counts from S0 to 2 S0 (within max_seg), the one whose grid fills the last
// round of resident work-groups best (a part-empty last round costs a whole
// round of kernel time); the first count that fills it to 99.5 %, else the
// fullest (the smallest on ties).  Returns the count to split nst by.
static int balance_segments(int tiles, int nst, int S0, int max_seg, int resident)
{
    int best = S0;
    double best_fill = -1.0;
    for (int c = S0; c <= std::min(2 * S0, std::max(S0, max_seg)); ++c) {
        const int steps = (nst + c - 1) / c;
        const int S = (nst + steps - 1) / steps;
        const double rounds = (double)tiles * S / resident;
        const double fill = rounds / std::ceil(rounds);
        if (fill >= 0.995) return c;
        if (fill > best_fill + 1e-9) {
            best_fill = fill;
            best = c;
        }
    }
    return best;
}

// Sources per segment of a plain pair launch of kernel fn on `tiles`
// target tiles.  Multiples of the 64 staged at a time; launches of fewer than
// 512 work-groups (two waves a SIMD) at that size take multiples of 16, as
// their blocks are bound by the latency of the staged reads: 2,806 triangles, two
// wave numbers of five columns, all operators 39.4 us with 64 sources (484
// work-groups), 35.5 with 32; 320 triangles, four columns 11.6, 5.2 with 16.  (A far
// field of 600 work-groups gains nothing: 54 us either way.)  But not more
// work-groups than are resident together (768 of 64 columns: far field of 6,936
// triangles, 1,000 directions 120 us with 436, 149 with 872, 110 with 584), and with
// 192 columns in all only below 256, as their partial sums cost more than that gives
// (64 wave numbers of one column, 2,772 triangles 714 us, 785 with 32 sources; 640
// triangles 524, 240 with 16).
// coarse: multiples of 64 always.
static int plain_seg_len(const Handle& h, int tiles, int64_t nsrc, int64_t nsrc_pad, const void* fn,
                         bool coarse = false)
{
    const int nsb = (int)(nsrc_pad / kSrcBlock);
    int unit = kSrcBlock, S;
    const bool wide = h.prm.K * wcsp_plain((int)h.prm.wcs) >= 192;
    if (h.segments == 0 && !coarse && tiles * nsb < (wide ? 256 : 512)) {
        unit = 16;
        const int res = resident_blocks(fn, kTile);
        S = res < 1024 ? std::max(1, res / tiles) : (1024 + tiles - 1) / tiles;
        S = std::min(S, (int)(nsrc_pad / unit));
    } else {
        S = choose_segments(h, tiles, nsb, nsrc);
        if (h.segments == 0) S = balance_segments(tiles, nsb, S, nsb, resident_blocks(fn, kTile));
    }
    return (int)(((nsrc_pad + S - 1) / S + unit - 1) / unit) * unit;
}

// Automatic segment count of an MFMA pair launch on grids of up to about four
// rounds (32,768 targets): the count of at least min_seg whose modelled time is least.  A CU runs
// ceil(blocks / CUs) blocks, up to four at a time; relative to four waves a
// SIMD, a step costs kShare[k - 1] with k blocks left on the CU (measured on
// the 32-column kernels: one wave a SIMD is latency bound, from two on the
// vector ALU is), and a block costs ovh steps for its start and its partial
// sums, which the epilogue reads again (about 2.5 per column block).  Against
// the fullest last round of resident blocks (the rule for larger grids), two
// wave numbers of 32 columns: 20,480 triangles 32 -> 16 segments, 0.970 ->
// 0.905 ms (32 segments: 0.918); 5,120 triangles 52 -> 24 segments, 0.111 -> 0.100 ms.
// (Other widths use the same shares: 8 columns, 9,922 triangles 126 us with the 32
// segments it takes, 136 with the 13 that it took without a lower bound.)
static int mfma_segments(int tiles, int nst, int col_blocks, bool ws, int min_seg, int cus)
{
    static const double kShareSingle[4] = {0.87, 0.60, 0.55, 0.53}, kShareWs[4] = {0.80, 0.75, 0.75, 0.75};
    const double* kShare = ws ? kShareWs : kShareSingle;
    const double ovh = col_blocks == 1 ? 1.0 : 2.5 * col_blocks - 1.5;
    int best = std::max(1, min_seg);
    double least = 1e300;
    for (int c = std::max(1, min_seg); c <= std::max({min_seg, 1, std::min(nst / 8, 64)}); ++c) {
        const int steps = (nst + c - 1) / c, S = (nst + steps - 1) / steps;
        const int n = (int)(((int64_t)tiles * S + cus - 1) / cus);
        const double t = ((n - n % 4) * kShare[3] + (n % 4 ? n % 4 * kShare[n % 4 - 1] : 0.0)) * (steps + ovh);
        if (t < 0.999 * least) {
            least = t;
            best = S;
        }
    }
    return best;
}

// Which MFMA kernel a mixed plan runs on `tiles` target tiles: the
// wave-specialised one for the FP32 contraction, when selected, and (automatic
// selection) with the adjoint double layer in more than 16 columns on small meshes,
// where the single-wave kernel has one wave a SIMD; else the single-wave kernel, also
// with the adjoint double layer, where it is built for 3 waves per SIMD.  All
// operators, wave-specialised against single-wave, us: one wave number of 64 columns 640
// triangles 29.2 / 30.9, 2,772 53.9 / 53.5, 4,000 74.5 / 75.1, 5,400 112 / 111, 8,066 193 /
// 188; two of 24 columns 30.4 / 32.0, 59.3 / 59.3, 82.8 / 83.6, 128 / 126, 223 / 219; two of 16
// columns 26.0 / 26.6, 49.8 / 50.4, 68.1 / 67.9, 103 / 100, 173 / 169; four of 16, which the
// single-wave kernel takes in one launch, 39 / 35, 79 / 68, 117 / 101, 188 / 159, 334 / 282.
static bool mixed_uses_ws(const Handle& h, const BdrPlan& pl, int tiles)
{
    return pl.f32 || h.mixed_kernel == 1 || (h.mixed_kernel == 2 && pl.adj && tiles <= 40 && pl.WCSP > 16);
}

// Whether the vertex epilogue reads per-triangle values formed
// beforehand (tri_epilogue_kernel): with four or more segments, where re-reading
// every segment's partials for each of a triangle's three vertices costs more
// than one extra pass.
static bool use_tsum(const BdrPlan& pl) { return pl.kernel_on && pl.S >= 4; }

// Runs a plain pair kernel over all chunk groups: part has ntgt_pad rows.
static void run_plain(Handle& h, int op, bool adj, int WCSP, const float4* tx, const float4* tn, int ntgt,
                      int ntgt_pad, const float4* sy, const float4* sn, int nsrc, int nsrc_pad, const float2* b,
                      int ldb, float* part, int64_t seg_stride, int ldp, int S, int seg_len, hipStream_t s)
{
    const Params& p = h.prm;
    Timed tm(h, s);
    for (int q0 = 0; q0 < p.K;) {
        const int kg = pick_kg(WCSP, (int)p.K - q0, false);
        const CoefPack cp = make_pack(p, q0, kg, nullptr);
        PlainFn fn = plain_fn(op, adj, WCSP, kg);
        dim3 grid(ntgt_pad / kTile, S);
        hipLaunchKernelGGL(fn, grid, dim3(kTile), 0, s, tx, tn, ntgt, sy, sn, nsrc, b, ldb, cp, part, seg_stride, ldp,
                           q0, seg_len, nsrc_pad, op == OP_BDR ? h.step_skip : nullptr);
        BAEMM_HIP(hipGetLastError());
        q0 += kg;
    }
    tm.done();
}

// Distances of evaluation points to the triangles' centroids: rmin is a positive
// lower bound, rmax an upper bound (rmin = 0: not known).
struct DistRange {
    float rmin, rmax;
};

// For points well outside the mesh's bounding sphere, bounds from their distances to
// its centre.  The kernels see points and centroids rounded to FP32, each coordinate
// by up to 2^-24 of itself: of the sphere's centre here, the rest is within the
// 0.999 and 1.001.
static DistRange outside_range(const Handle& h, const double* pts, int64_t P)
{
    double lo2 = 1e300, hi2 = 0.0;
    const double c0 = h.centre[0], c1 = h.centre[1], c2 = h.centre[2];
    for (int64_t i = 0; i < P; ++i) {
        const double x = pts[3 * i] - c0, y = pts[3 * i + 1] - c1, z = pts[3 * i + 2] - c2;
        const double r2 = x * x + y * y + z * z;
        lo2 = r2 < lo2 ? r2 : lo2;
        hi2 = r2 > hi2 ? r2 : hi2;
    }
    const double slack = 0.001 * h.radius + std::ldexp(std::fabs(c0) + std::fabs(c1) + std::fabs(c2), -23);
    const double gap = 0.999 * std::sqrt(lo2) - h.radius - slack, far = 1.001 * std::sqrt(hi2) + h.radius + slack;
    if (!(gap >= 0.1 * h.radius && gap < 1e18)) return {0.0f, 0.0f};
    return {(float)gap, (float)far};
}

// Smallest and (not self) largest distance between the targets and the centroids,
// reduced in the two device words buf (synchronises s).
static DistRange distance_range(Handle& h, const float4* tgt, int ntgt, bool self, unsigned* buf, hipStream_t s)
{
    hipLaunchKernelGGL(range_init_kernel, dim3(1), dim3(64), 0, s, buf);
    // about 2,048 work-groups of 256 targets: 8 per CU hide the LDS latency (one
    // per 256 targets, 320 at 81,920 triangles, took 2.73 ms)
    const int tiles = (ntgt + 255) / 256, nb = ((int)h.nt + 255) / 256;
    const int S = std::max(1, std::min(nb, (2048 + tiles - 1) / tiles));
    const int seg_len = (nb + S - 1) / S * 256;
    hipLaunchKernelGGL(self ? &rmin_kernel<true> : &rmin_kernel<false>,
                       dim3(tiles, ((int)h.nt + seg_len - 1) / seg_len), dim3(256), 0, s, tgt, ntgt, h.d_mid, (int)h.nt,
                       seg_len, buf);
    BAEMM_HIP(hipGetLastError());
    unsigned out[2] = {0, 0};
    BAEMM_HIP(hipMemcpyAsync(out, buf, sizeof(out), hipMemcpyDeviceToHost, s));
    BAEMM_HIP(hipStreamSynchronize(s));
    float r2[2];
    memcpy(r2, out, sizeof(out));
    return {std::sqrt(std::max(r2[0], 1e-30f)), std::sqrt(std::max(r2[1], 1e-30f))};
}

bool find_rmin(Handle& h, hipStream_t s)
{
    if (h.rmin >= 0.0f) return true;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    BAEMM_HIP(hipStreamIsCapturing(s, &cs));
    if (cs != hipStreamCaptureStatusNone) return false;
    h.rmin = distance_range(h, h.d_mid, (int)h.nt, true, h.ws_misc.as<unsigned>(), h.stream).rmin;
    return true;
}

// The power-of-two factors sA that bring the kernel values of the split-FP16
// MFMA kernels into the range of FP16: per chunk (general form), or one for
// all chunks (non-adjoint form, values divided by rot = c2, with tn c3).  A
// bound of |A| over distances >= rmin, times sA, lies in [2^14, 2^15).
// typ: the scaled size A has over the mesh's extent, the smallest over the
// chunks.  The split's relative error is at most 2^-23 (in the mean 2^-24.5) for
// values down to 2^-2; below, its absolute error is at most 2^-25 (the FP16
// subnormals of the low part).
struct MfmaScales {
    float sA[64];
    double typ;
};
static MfmaScales mfma_scales(const Params& p, bool adj, bool tn, double rmin, double extent)
{
    MfmaScales m{};
    const int cn = tn ? 3 : 2;
    double amax[64], atyp[64], all = 0.0;
    for (int q = 0; q < p.K; ++q) {
        const double kap = std::fabs((double)p.kappa[q]);
        double c1 = std::abs(std::complex<double>(p.c[4 * q + 1])), cd = 1.0;
        if (adj)
            cd = std::abs(std::complex<double>(p.c[4 * q + 2])) + std::abs(std::complex<double>(p.c[4 * q + 3]));
        else
            c1 /= std::abs(std::complex<double>(p.c[4 * q + cn]));
        amax[q] = c1 / rmin + cd * (1.0 + kap * rmin) / (rmin * rmin);
        atyp[q] = (c1 + 0.5 * cd * std::max(kap, 1.0 / extent)) / extent;
        all = std::max(all, amax[q]);
    }
    m.typ = 1e300;
    for (int q = 0; q < p.K; ++q) {
        int e = 0;
        std::frexp(std::max(adj ? amax[q] : all, 1e-30), &e);
        m.sA[q] = (float)std::ldexp(1.0, 15 - e);
        m.typ = std::min(m.typ, atyp[q] * m.sA[q]);
    }
    return m;
}

template <int BT, int CT>
static void launch_bdr_epilogue(EpiArgs& ea, hipStream_t s)
{
    const int lpv = epi_lanes(ea.W);
    const int vpb = 256 / lpv;
    const dim3 grid((ea.nv + vpb - 1) / vpb);
    if (ea.kernel_on && ea.tsum)
        hipLaunchKernelGGL((bdr_epilogue_kernel<BT, CT, true>), grid, dim3(256), 0, s, ea, lpv);
    else
        hipLaunchKernelGGL((bdr_epilogue_kernel<BT, CT, false>), grid, dim3(256), 0, s, ea, lpv);
}

static void bdr_epilogue(Handle& h, EpiArgs& ea, int Btype, int Ctype, hipStream_t s)
{
    if (Btype == kC128 && Ctype == kC128) launch_bdr_epilogue<kC128, kC128>(ea, s);
    else if (Btype == kC128 && Ctype == kC64) launch_bdr_epilogue<kC128, kC64>(ea, s);
    else if (Btype == kC64 && Ctype == kC128) launch_bdr_epilogue<kC64, kC128>(ea, s);
    else launch_bdr_epilogue<kC64, kC64>(ea, s);
    BAEMM_HIP(hipGetLastError());
}

static EpiArgs base_epi(Handle& h, const ApplyArgs& a, int WCSP)
{
    const Params& p = h.prm;
    if (p.K > 64) throw ArgError{"at most 64 wave-number chunks are supported"};
    EpiArgs ea{};
    ea.nv = (int)h.nv;
    ea.W = (int)p.W;
    ea.wcs = (int)p.wcs;
    ea.WCSP = WCSP;
    ea.K = (int)p.K;
    ea.ar = a.alpha.real();
    ea.ai = a.alpha.imag();
    ea.br = a.beta.real();
    ea.bi = a.beta.imag();
    ea.vt_ptr = h.d_vt_ptr;
    ea.vt_idx = h.d_vt_idx;
    ea.area = h.d_area;
    ea.sdiag = h.d_sdiag;
    ea.M_ptr = h.d_M_ptr;
    ea.M_idx = h.d_M_idx;
    ea.M_val = h.d_M_val;
    ea.B = a.B;
    ea.ldB = a.ldB;
    ea.C = a.C;
    ea.ldC = a.ldC;
    for (int q = 0; q < p.K; ++q) {
        ea.rotr[q] = 1.0f;
        ea.roti[q] = 0.0f;
        ea.c0r[q] = p.c[4 * q].real();
        ea.c0i[q] = p.c[4 * q].imag();
        ea.c1r[q] = p.c[4 * q + 1].real();
        ea.c1i[q] = p.c[4 * q + 1].imag();
        ea.kap[q] = p.kappa[q];
    }
    return ea;
}

static void launch_av(Handle& h, const void* B, int64_t ldB, int Btype, int WCSP, float2* b, int ldb,
                      hipStream_t s)
{
    const int64_t total = h.nt_pad * (int64_t)ldb;
    const dim3 grid((unsigned)((total + 255) / 256));
    if (Btype == kC128)
        hipLaunchKernelGGL(av_gather_kernel<kC128>, grid, dim3(256), 0, s, h.d_tris, h.d_area, (int)h.nt, total, B,
                           ldB, (int)h.prm.wcs, WCSP, ldb, b);
    else
        hipLaunchKernelGGL(av_gather_kernel<kC64>, grid, dim3(256), 0, s, h.d_tris, h.d_area, (int)h.nt, total, B,
                           ldB, (int)h.prm.wcs, WCSP, ldb, b);
    BAEMM_HIP(hipGetLastError());
}

// Operands of the MFMA pair kernels for the staged sources pl.b: the B operand
// (hi/lo split with per-column scales, or FP32), the chunk factors pl.rot and
// scales pl.sA folded into the coefficients, the source normals pl.nrm the
// kernel reads, and pl.unscale (per column, null for FP32 MFMA).  rmin: lower
// bound of the target-centroid distances (mixed precision only).
static void stage_mfma(Handle& h, BdrPlan& pl, float rmin, hipStream_t s, const void* B, int64_t ldB, int Btype)
{
    const Params& p = h.prm;
    if (pl.f32) {
        if (pl.defer) throw ArgError{"internal: deferred staging of the FP32 MFMA operand"};
        launch_av(h, B, ldB, Btype, pl.WCSP, pl.b, pl.ldb, s);
        // FP32 MFMA: no FP16 range to fit, no scales; the non-adjoint form still
        // divides each chunk by c2 (the epilogue multiplies it back)
        pl.sA.assign(p.K, 1.0f);
        pl.rot.assign(p.K, cdouble(1.0, 0.0));
        if (!pl.adj)
            for (int q = 0; q < p.K; ++q) pl.rot[q] = p.cd[4 * q + (pl.tn ? 3 : 2)];
        pl.back = pl.rot;
        const int NCB = 2 * pl.WCSP / 32;
        const int64_t nbop = (int64_t)p.K * pl.nst * NCB * 64;
        uint4* bop = static_cast<uint4*>(pl.ws.take(h.ws_bop, sizeof(uint4) * nbop * 2));
        hipLaunchKernelGGL(stage_f32_kernel, dim3((unsigned)((nbop + 255) / 256)), dim3(256), 0, s, pl.b, pl.ldb,
                           pl.nst, pl.WCSP, (int)p.K, bop);
        BAEMM_HIP(hipGetLastError());
        pl.bop = bop;
        pl.unscale = nullptr;
        return;
    }
    // scales: A per chunk from a bound at the minimum target-centroid
    // distance rmin, b per column from its maximum.
    pl.sA.assign(p.K, 1.0f);
    pl.rot.assign(p.K, cdouble(1.0, 0.0));
    const MfmaScales ms = mfma_scales(p, pl.adj, pl.tn, rmin, std::max(h.extent, 1e-30));
    for (int q = 0; q < p.K; ++q) pl.sA[q] = ms.sA[q];
    float nrm_sig = 0.0f;      // the common scale of the source normals (non-adjoint form)
    float4* nrm_out = nullptr;  // the scaled normals (non-adjoint form)
    if (!pl.adj) {
        // Every chunk has c2 != 0: the kernel values are taken as A' = s A / c2
        // with one scale s for all chunks, carried by the source normals
        // (Q' = c1/c2 s / r - s (z.n)/r^3 + i kappa s (z.n)/r^2); the epilogue
        // multiplies c2 / s back.
        // (with pl.tn: c3 in place of c2, the target normals in place of the
        // source normals)
        for (int q = 0; q < p.K; ++q) pl.rot[q] = p.cd[4 * q + (pl.tn ? 3 : 2)];
        nrm_sig = ms.sA[0];
        float4* nrm = static_cast<float4*>(pl.ws.take(h.ws_nrm, sizeof(float4) * h.nt_pad));
        if (pl.defer) {
            pl.sd.nrm_in = h.d_nrm;
            pl.sd.nrm_out = nrm;
            pl.sd.nrm_s = nrm_sig;
        }
        nrm_out = nrm;
        pl.nrm = nrm;
    }
    pl.back = pl.rot;
    for (int q = 0; q < p.K; ++q) pl.back[q] /= (double)pl.sA[q];
    const int ncols = pl.ldb;
    unsigned* colmax = static_cast<unsigned*>(pl.ws.take(h.ws_scale, sizeof(float) * 3 * ncols));
    float* scale = reinterpret_cast<float*>(colmax + ncols);
    float* unscale = scale + ncols;
    const int NCB = 2 * pl.WCSP / 32;
    const int64_t nbop = (int64_t)p.K * pl.nst * NCB * 64;
    uint4* bop = static_cast<uint4*>(pl.ws.take(h.ws_bop, sizeof(uint4) * nbop * 2));
    pl.bop = bop;
    pl.unscale = unscale;
    if (pl.defer) {
        StageDesc& d = pl.sd;
        d.split = 1;
        d.K = (int)p.K;
        d.nst = pl.nst;
        d.colmax = colmax;
        d.scale = scale;
        d.unscale = unscale;
        d.bop = bop;
        return;
    }
    // the scaled source normals (non-adjoint form) with the column maxima
    // cleared; the Av gather and the column maxima (one launch for small
    // meshes, where the launches are the cost; two above, where the blocks'
    // atomics on the few maxima of the one launch cost more); the split operand
    // with the column scales and their inverses
    const int nn = pl.adj ? 0 : (int)h.nt_pad;
    hipLaunchKernelGGL(scale_nrm_kernel, dim3((unsigned)((std::max(nn, ncols) + 255) / 256)), dim3(256), 0, s,
                       h.d_nrm, nn, nrm_sig, nrm_out, colmax, ncols);
    const int64_t total = h.nt_pad * (int64_t)pl.ldb;
    if ((total + 255) / 256 <= kGatherMaxBlocks) {
        // a multiple of ldb / gcd(ldb, 256) blocks: the grid's thread count is
        // a multiple of ldb
        const int64_t unit = pl.ldb / std::gcd(pl.ldb, 256);
        const dim3 grid((unsigned)(((total + 255) / 256 + unit - 1) / unit * unit));
        const size_t lds = sizeof(unsigned) * (size_t)pl.ldb;
        if (Btype == kC128)
            hipLaunchKernelGGL(av_gather_max_kernel<kC128>, grid, dim3(256), lds, s, h.d_tris, h.d_area, (int)h.nt,
                               total, B, ldB, (int)p.wcs, pl.WCSP, pl.ldb, pl.b, colmax);
        else
            hipLaunchKernelGGL(av_gather_max_kernel<kC64>, grid, dim3(256), lds, s, h.d_tris, h.d_area, (int)h.nt,
                               total, B, ldB, (int)p.wcs, pl.WCSP, pl.ldb, pl.b, colmax);
    } else {
        launch_av(h, B, ldB, Btype, pl.WCSP, pl.b, pl.ldb, s);
        hipLaunchKernelGGL(colmax_kernel, dim3(256), dim3(256), 0, s, pl.b, (int)h.nt, pl.ldb, colmax);
    }
    hipLaunchKernelGGL(split_kernel, dim3((unsigned)((nbop + 255) / 256)), dim3(256), 0, s, pl.b, pl.ldb, pl.nst,
                       pl.WCSP, (int)p.K, colmax, ncols, unscale, bop);
    BAEMM_HIP(hipGetLastError());
}

// Source segments of the MFMA pair launches of a plan on `tiles` target tiles.
//
// least (split products, up to 256 tiles): the segments that keep the error
// against 64 bits no larger than the vector-ALU kernel's.  The rounding of an
// accumulation of kSubStepsSmall steps shows where the other errors, which grow
// with the mesh, are small: of 5,104 triangles the vector ALU has
// 1.102e-7, 16 steps 1.096e-7, 24 steps 1.107e-7, 48 steps 1.133e-7; of 9,922 1.524e-7, 32
// steps 1.515e-7, 48 steps 1.526e-7, 100 steps 1.561e-7; of 30,960 2.741e-7, 100 steps
// 2.711e-7.  So at least 32 segments, of at least 8 steps.  MIXED has no more to keep
// than the fill rule's (30,960 triangles, 2 x 32 columns 1.98 ms and 2.736e-7; with 39
// segments 2.04 ms and 2.717e-7).
// points (the potential): away from the surface every source weighs about the
// same and the rounding of an accumulation shows in full (2 x 32 columns, 20,416
// triangles, 2,500 points: 16 steps 2.53e-7, 24 steps 2.70e-7, 48 steps 3.15e-7), so
// the accumulations are as short as the fill rule's, and for FP32 as the vector
// ALU's on these points.
static void plan_mfma_segments(Handle& h, BdrPlan& pl, int tiles, int64_t points = 0)
{
    const Params& p = h.prm;
    const bool ws = mixed_uses_ws(h, pl, tiles);
    const int kg = std::min(pick_kg(pl.WCSP, (int)p.K, true), ws ? 2 : 4);
    const int res = ws ? resident_blocks((const void*)mixed_ws_fn(pl.adj, pl.WCSP, kg, pl.f32, pl.tn), 512)
                       : resident_blocks((const void*)mixed_fn(pl.adj, pl.WCSP, kg, nullptr, pl.tn), 256);
    const int fill = choose_segments(h, tiles, pl.nst / 8, h.nt);
    int S0 = fill;
    if (h.segments == 0 && !pl.lean) {
        // The single-wave kernel runs 2-3 % faster with about four times the
        // work-groups (finer last rounds): up to 16 segments where the rule of
        // choose_segments gives fewer.
        int full = fill;
        if (!ws && full < 16) full = std::max(full, std::min({16, (8192 + tiles - 1) / tiles, pl.nst / 8}));
        full = balance_segments(tiles, pl.nst, full, pl.nst / 8, res);
        if (points && h.precision == BAEMM_PRECISION_FP32) {
            const int WCSP = wcsp_plain((int)p.wcs);
            const int len = plain_seg_len(h, (int)((points + kTile - 1) / kTile), h.nt, h.nt_pad,
                                          (const void*)plain_fn(OP_NEAR, false, WCSP, pick_kg(WCSP, (int)p.K, false)),
                                          true);
            full = std::min(std::max(full, (int)((h.nt_pad + len - 1) / len)), std::max(1, pl.nst / 8));
        }
        if (!pl.f32 && tiles <= 256) {
            // FP32: no more steps than one accumulation may have (run_mfma would split
            // the launch: 12,696 triangles, three wave numbers of one column 10 segments
            // of two launches 493 us, 20 of one 450)
            int least = std::max(min_segments(h.nt), (pl.nst + kSubStepsSmall - 1) / kSubStepsSmall);
            least = std::max(least, points ? full : std::min(32, pl.nst / 8));
            if (h.precision == BAEMM_PRECISION_MIXED) least = std::min(least, full);
            S0 = mfma_segments(tiles, pl.nst, kg * 2 * pl.WCSP / 32, ws, least, cu_count());
        } else {
            S0 = full;
        }
    }
    pl.steps = (pl.nst + S0 - 1) / S0;
    pl.S = (pl.nst + pl.steps - 1) / pl.steps;
    pl.rounds = (double)tiles * fill / res;
}

// The kernels of a plan:
//  - kSplit: kernel values and sources as FP16 hi + lo on the matrix cores.  An
//    operand keeps 23 bits where FP32 has 24; the accumulations are short enough
//    (plan_mfma_segments) that the error against 64 bits is no larger all the same:
//    81,920 triangles, two wave numbers of 32 columns 5.15e-7, vector ALU 5.28e-7;
//    means over three seeds of 120 applies of 400 to 32,000 triangles 0.84 to 1.003 of
//    it, of 90 potentials 0.74 to 1.000.  That holds while the kernel values over the
//    mesh keep their bits next to the largest one, at the least distance of two
//    centroids: with typ >= 0.5 values of the typical size keep their 23 bits and
//    smaller ones an absolute 2^-25 (mfma_scales).
//  - kF32: FP32 products on the matrix cores where typ is smaller: meshes with a
//    few triangles much closer together than the others (for any distances; the
//    vector-ALU kernel takes 1.6 times as long at 81,920 triangles).
//  - kPlain: the vector-ALU kernel, for FP32 and MIXED (whose error it does not
//    reach) on small meshes: the matrix cores pad to 16 columns and need two
//    staging launches more.  Times in us, vector ALU against split, by the
//    columns of a launch: one wave number of 16 columns 160 triangles 17.6 / 22.9,
//    960 23.8 / 23.7; 32 columns 160 triangles 21.0 / 24.2; two of 32, 37 / 26.6;
//    8 columns 2,806 triangles 33 / 38, 5,120 66 / 59; 4 columns 5,120 triangles
//    49 / 59, 10,000 141 / 135, 20,480 458 / 411 (two wave numbers: 10,000 214 /
//    218, 20,480 733 / 655; with the adjoint double layer 10,000 154 / 168).
enum class PairPath { kPlain, kSplit, kF32 };
// Whether the sizes ask for the matrix cores at all (FP32 and MIXED).
// With the adjoint double layer beside others (adj) FP32 stays on the vector ALU in up
// to three wave numbers of four columns: 34,000 triangles, one 1,338 / 1,392 us, three
// 3,490 / 3,574, 41,000 1,815 / 1,980, 4,760 / 5,170, 82,000 7,671 / 7,657, 19,626 / 19,461.
// MIXED has lines of its own where it has several wave numbers: the single-wave kernel
// takes four to a launch, the vector ALU two.  Vector ALU against split: 16 columns
// 180 triangles four wave numbers 35 / 29, seven 57 / 51; 8 columns 2,090 triangles two 40 /
// 44, 2,772 two 47 / 46, three 68 / 63, 640 four 33 / 33, 1,472 50 / 49, 2,090 60 / 54,
// eight 180 triangles 44 / 42, 1,472 84 / 68; 4 columns 2,772 triangles four 61 / 61, 3,952
// 85 / 86, 5,400 140 / 128, all operators 5,400 158 / 157, 6,936 227 / 222.  Rows with the
// adjoint double layer and no double layer (tn) take the adjoint kernel on the vector
// ALU and a form as fast as the double layer's on the matrix cores: 4 columns, 5,400
// triangles two wave numbers 85 / 85, 6,936 117 / 111, 9,922 207 / 185, 2,100 four 54 / 55, eight
// 91 / 90, 2,772 64 / 61, 115 / 104.
static bool mfma_sizes(int precision, int64_t K, int64_t wcs, int64_t nt, bool adj, bool tn)
{
    if (K > 64) return precision != BAEMM_PRECISION_FP32;   // (refused later)
    const int WCSP = wcsp_plain((int)wcs);
    const int cols = WCSP * (K > 1 ? 2 : 1);   // of a plain launch (its pick_kg)
    const bool mixed = precision == BAEMM_PRECISION_MIXED;
    const double n = (double)nt;
    double least;
    if (WCSP > 8) {
        least = cols >= 64 || (mixed && K >= 4) ? 0.0 : (cols == 32 ? 320.0 : 900.0);
    } else if (WCSP == 8) {
        least = 4096.0;
        if (mixed && K > 1) least = K >= 8 ? 0.0 : (K >= 4 ? 1024.0 : 2560.0);
    } else if (mixed && K >= 4) {
        least = adj ? 6144.0 : (tn ? 2048.0 : 4096.0);
    } else if (adj) {
        least = mixed || K >= 4 ? 32768.0 : 100000.0;
    } else {
        least = cols > 4 ? (mixed && tn ? 5120.0 : 12288.0) : 8192.0;
    }
    return n >= least;
}
// The same for the potential at P points, by its pairs times columns: the matrix
// cores need the operand of all sources, and mostly a pass over the distances
// and its synchronisation first.  Times in us, vector ALU against matrix cores,
// one wave number: 5,120 triangles 2,560 points 16 columns 140 / 156, 10,240
// points 344 / 313; 20,480 triangles 32 columns 640 points 295 / 302, 1,280 points 355 /
// 330; 8 columns 5,120 points 290 / 282; three of 8 columns, 12,972
// triangles, 3,000 points 361 / 375, 8,000 points 714 / 627; 4 columns, 52,000 triangles, 20,000
// points 1,104 / 1,061; two of 4 columns, 12,972 triangles, 20,000 points 579 / 621, 52,000 triangles,
// 3,000 points 411 / 458, 20,000 points 1,843 / 1,782; three, 12,972 triangles, 20,000 points
// 988 / 1,052, 26,000 1,685 / 1,678;
// two of 32 columns 320 points 487 / 448 (1,280 triangles, 2,560 points 304 / 274),
// of 16 320 points 276 / 290, 1,280 points 356 / 340.
static bool mfma_points(const Handle& h, int64_t P)
{
    const Params& p = h.prm;
    if (p.K > 64) return h.precision != BAEMM_PRECISION_FP32;   // (refused later)
    const int WCSP = wcsp_plain((int)p.wcs);
    const int cols = WCSP * (p.K > 1 ? 2 : 1);   // of a plain launch
    const double least = WCSP <= 4 ? 4.8e9 : (cols >= 64 ? 1.5e8 : (WCSP == 8 && p.K > 1 ? 1.5e9 : 8e8));
    return (double)P * (double)h.nt * (double)(p.K * WCSP) >= least;
}
// Whether a plan may leave the matrix cores for its sizes: FP32, and MIXED with
// the automatic kernel and segments (a kernel or segments chosen by the caller
// are those of the MFMA kernels).
static bool may_be_plain(const Handle& h)
{
    return h.precision == BAEMM_PRECISION_FP32 ||
           (h.precision == BAEMM_PRECISION_MIXED && h.mixed_kernel == 2 && h.segments == 0);
}
// FP32_MFMA on small meshes: the FP32 operand takes one staging launch less
// (1,440 triangles, 32 columns 34.8 against 38.7 us; 2,560 triangles 50.4 / 48.9)
static bool f32_sizes(const Handle& h) { return h.precision == BAEMM_PRECISION_FP32_MFMA && h.nt < 2048; }
// The MFMA kernels of the precision; distances from rmin to extent.
static PairPath mfma_path(const Handle& h, bool adj, bool tn, double rmin, double extent)
{
    if (h.precision == BAEMM_PRECISION_MIXED) return PairPath::kSplit;
    if (mfma_scales(h.prm, adj, tn, rmin, extent).typ >= 0.5) return PairPath::kSplit;
    if (h.precision == BAEMM_PRECISION_FP32) {
        if (wcsp_plain((int)h.prm.wcs) <= 8) return PairPath::kPlain;
        // c1 / c2 (non-adjoint form, without the scales of the split) times a source has
        // to stay in the FP32 range
        const Params& p = h.prm;
        for (int q = 0; q < p.K && !adj; ++q)
            if (std::abs(p.cd[4 * q + 1]) > 1e12 * std::abs(p.cd[4 * q + (tn ? 3 : 2)])) return PairPath::kPlain;
    }
    return PairPath::kF32;
}

void bdr_setup(Handle& h, BdrPlan& pl, hipStream_t s)
{
    const Params& p = h.prm;
    if (!p.loaded) throw ArgError{"operators not loaded"};
    pl.planned = true;
    pl.kernel_on = p.kernel_on();
    pl.mass_on = p.mass_on();
    // The MFMA kernels' non-adjoint form divides each chunk by its c2; chunks
    // without a double layer take the general (adjoint) form, unless every
    // chunk has the adjoint double layer and no double layer: the MFMA
    // kernels then take the non-adjoint form divided by c3, on the target
    // normals (the adjoint double layer has the double layer's values with the
    // target normal in place of the source normal).
    bool adj = p.any(3), tn = p.K > 0;
    for (int q = 0; q < p.K; ++q) {
        if (p.c[4 * q + 2] == cfloat(0.0f, 0.0f)) adj = true;
        tn = tn && p.c[4 * q + 2] == cfloat(0.0f, 0.0f) && p.c[4 * q + 3] != cfloat(0.0f, 0.0f);
    }
    if (tn) adj = false;
    pl.mixed = pl.kernel_on;
    if (pl.kernel_on) {
        const bool plain = pl.plain_only || (!pl.mfma_only && may_be_plain(h) && !mfma_sizes(h.precision, p.K, p.wcs, h.nt, adj, tn)) ||
                           (h.precision != BAEMM_PRECISION_MIXED && p.K > 64);
        // (without the least distance, in a capture before any other apply: kernels that
        // do not need it)
        PairPath path = PairPath::kPlain;
        if (!plain) {
            if (pl.f32_only || f32_sizes(h)) path = PairPath::kF32;
            else if (find_rmin(h, s)) path = mfma_path(h, adj, tn, h.rmin, h.extent);
            else path = h.precision == BAEMM_PRECISION_FP32 ? PairPath::kPlain : PairPath::kF32;
        }
        pl.mixed = path != PairPath::kPlain;
        pl.f32 = path == PairPath::kF32;
    }
    pl.WCSP = pl.mixed ? wcsp_mixed((int)p.wcs) : wcsp_plain((int)p.wcs);
    pl.ldb = (int)p.K * pl.WCSP;
    pl.ldp = 2 * pl.ldb;
    pl.adj = pl.mixed ? adj : p.any(3);
    pl.tn = pl.mixed && tn;
    if (!pl.kernel_on) return;
    if (!pl.mixed) {
        const int tiles = (int)(h.nt_pad / kTile);
        const void* fn = (const void*)plain_fn(OP_BDR, pl.adj, pl.WCSP, pick_kg(pl.WCSP, (int)p.K, false));
        const int res = resident_blocks(fn, kTile);
        pl.seg_len = plain_seg_len(h, tiles, h.nt, h.nt_pad, fn, pl.lean);
        pl.S = (int)((h.nt_pad + pl.seg_len - 1) / pl.seg_len);
        // (rounds of segments of at least 64 sources)
        pl.rounds = (double)tiles * std::min<int64_t>(pl.S, h.nt_pad / kSrcBlock) / res;
        return;
    }
    pl.nst = (int)(h.nt_pad / 8);
    plan_mfma_segments(h, pl, (int)(h.nt_pad / kMixTile));
}

// Per triangle t and column k of chunk q: the sum over the segments s (FP64) of
// part_s[t][q][k], real and imaginary parts, turned
// into the triangle's value (epi_tri_value) at tsum[t * ldb + q * WCSP + k % wcs]:
// the values the vertex epilogue forms, once per triangle instead of once per
// incident vertex.
template <int SW>
__global__ __launch_bounds__(kSegThreads<SW>) void tri_epilogue_kernel(EpiArgs a, int nt,
                                                                      double2* __restrict__ tsum)
{
    const int64_t idx = segment_element<SW>();
    const bool in = idx < (int64_t)nt * a.W;
    if (SW == 1 && !in) return;
    const int t = in ? (int)(idx / a.W) : 0, k = in ? (int)(idx % a.W) : 0;
    const int q = k / a.wcs, kk = k % a.wcs;
    const int pc = q * a.WCSP + kk;
    double pr, pi;
    if (!segment_sum<SW>(a.part + (int64_t)t * a.ldp + q * 2 * a.WCSP + kk, a.seg_stride, a.WCSP, a.S, pr, pi) || !in)
        return;
    double qr, qi;
    epi_tri_value(a, t, q, pc, pr, pi, qr, qi);
    tsum[(int64_t)t * a.ldb + pc] = make_double2(qr, qi);
}

size_t bdr_workspace_bytes(const Handle& h, const BdrPlan& pl)
{
    if (!pl.kernel_on) return 0;
    const auto al = [](size_t n) { return (n + 255) & ~(size_t)255; };
    const Params& p = h.prm;
    size_t n = al(sizeof(float2) * h.nt_pad * pl.ldb);                       // staged sources b
    if (pl.mixed) {
        const int NCB = 2 * pl.WCSP / 32;
        n += al(sizeof(uint4) * 2 * (size_t)p.K * pl.nst * NCB * 64);       // MFMA B operand
        if (!pl.f32) {
            if (!pl.adj) n += al(sizeof(float4) * h.nt_pad);                // scaled source normals
            n += al(sizeof(float) * 3 * pl.ldb);                             // column maxima and scales
        }
    }
    n += al(sizeof(float) * (size_t)pl.S * h.nt_pad * pl.ldp);              // segment partials
    if (use_tsum(pl)) n += al(sizeof(double2) * h.nt_pad * pl.ldb);         // their sums per triangle
    return n;
}

// Most segments of a plain pair launch (plain_seg_len) and of an MFMA one
// (plan_mfma_segments on the boundary operators) with automatic segments.
static int64_t most_plain_segments(int64_t tiles, int64_t nsrc_pad)
{
    const int64_t nsb = nsrc_pad / kSrcBlock;
    if (tiles * nsb < 512) return std::min((1024 + tiles - 1) / tiles, nsrc_pad / 16);
    const int64_t S = std::min(std::max((2048 + tiles - 1) / tiles, (int64_t)min_segments(nsrc_pad)), nsb);
    return std::min(2 * S, nsb);
}
static int64_t most_mfma_segments(int64_t tiles, int64_t nst)
{
    const int64_t eighth = std::max<int64_t>(1, nst / 8);
    int64_t S = std::min(std::max((2048 + tiles - 1) / tiles, (int64_t)min_segments(8 * nst)), eighth);
    S = std::min(2 * std::max(S, std::min<int64_t>(16, eighth)), eighth);
    if (tiles <= 256) S = std::max({S, (nst + kSubStepsSmall - 1) / kSubStepsSmall, std::min<int64_t>(64, eighth)});
    return S;
}

size_t pair_workspace_bound(int64_t nt, int64_t m, int64_t K, int64_t wcs, int precision)
{
    const int64_t nt_pad = (nt + kTile - 1) / kTile * kTile, m_pad = (m + kTile - 1) / kTile * kTile;
    int64_t padded = 4;
    while (padded < wcs) padded *= 2;
    const int64_t nst = nt_pad / 8, ldb = K * padded, ldm = K * std::max<int64_t>(padded, 16);
    // the boundary operators: the kernels that the sizes can lead to, and the batched
    // apply, which is on the matrix cores at any size
    const bool mfma = precision == BAEMM_PRECISION_FP32_MFMA || mfma_sizes(precision, K, std::min<int64_t>(wcs, 64), nt, false, true);
    const int64_t Sm = mfma ? most_mfma_segments(nt_pad / kMixTile, nst) : (nst + kSubStepsSmall - 1) / kSubStepsSmall;
    const bool plain = precision != BAEMM_PRECISION_FP32_MFMA && (!mfma || padded <= 8);
    const int64_t Sp = plain ? most_plain_segments(nt_pad / kTile, nt_pad) : 0;
    // far field: m targets; Herglotz wave: m sources
    const int64_t Sf = most_plain_segments(m_pad / kTile, nt_pad), Sh = most_plain_segments(nt_pad / kTile, m_pad);
    const int64_t part = std::max({Sm * nt_pad * ldm, Sp * nt_pad * ldb, Sf * m_pad * ldb, Sh * nt_pad * ldb});
    size_t n = sizeof(float) * 2 * (size_t)part;
    n += sizeof(float2) * (size_t)(nt_pad * ldm + m_pad * ldb);         // staged sources, of the Herglotz wave
    n += sizeof(uint4) * 2 * (size_t)(nst * (2 * ldm / 32) * 64);       // MFMA B operand
    n += sizeof(double2) * (size_t)(nt_pad * ldm);                      // values per triangle
    n += sizeof(float4) * (size_t)nt_pad + sizeof(float) * 3 * (size_t)ldm;   // scaled normals, column scales
    return n;
}

void bdr_begin(Handle& h, const ApplyArgs& a, BdrPlan& pl, hipStream_t s)
{
    const Params& p = h.prm;
    if (!pl.planned) bdr_setup(h, pl, s);
    if (!pl.kernel_on && !pl.mass_on) return;   // the reference leaves C_out untouched
    pl.nrm = h.d_nrm;
    EpiArgs& ea = pl.ea;
    ea = base_epi(h, a, pl.WCSP);
    ea.mass_on = pl.mass_on;
    ea.kernel_on = pl.kernel_on;
    ea.diag_on = pl.kernel_on && h.use_diagonal && p.any(1);
    if (!pl.kernel_on) return;
    pl.b = static_cast<float2*>(pl.ws.take(h.ws_b32, sizeof(float2) * h.nt_pad * pl.ldb));
    if (pl.defer) {
        StageDesc& d = pl.sd;
        d.tris = h.d_tris;
        d.area = h.d_area;
        d.nt = (int)h.nt;
        d.nt_pad = (int)h.nt_pad;
        d.B = a.B;
        d.ldB = a.ldB;
        d.wcs = (int)p.wcs;
        d.WCSP = pl.WCSP;
        d.ldb = pl.ldb;
        d.b = pl.b;
    } else if (!pl.mixed) {
        launch_av(h, a.B, a.ldB, a.Btype, pl.WCSP, pl.b, pl.ldb, s);
    }
    ea.b = pl.b;
    ea.ldp = pl.ldp;
    ea.ldb = pl.ldb;
    ea.unscale = nullptr;
    if (!pl.mixed) return;
    // (not deferred: the Av gather too)
    stage_mfma(h, pl, h.rmin, s, a.B, a.ldB, a.Btype);
    ea.unscale = pl.unscale;
    for (int q = 0; q < p.K; ++q) {
        ea.rotr[q] = pl.back[q].real();
        ea.roti[q] = pl.back[q].imag();
    }
}

float* bdr_reserve_part(Handle& h, BdrPlan& pl, int S)
{
    const int64_t seg_stride = h.nt_pad * (int64_t)pl.ldp;
    float* part = static_cast<float*>(pl.ws.take(h.ws_part, sizeof(float) * seg_stride * S));
    pl.ea.S = S;
    pl.ea.seg_stride = seg_stride;
    pl.ea.part = part;
    return part;
}

// The MFMA pair launches of a plan over all chunk groups: targets tgt[0 ..
// ntgt) in `tiles` tiles of 128 (self: the centroids).  A segment longer
// than the longest accumulation (kSubSteps, kSubStepsSmall) is taken in several
// launches, of which the later ones add to the partial sums.
static void run_mfma(Handle& h, const BdrPlan& pl, const float4* tgt, int ntgt, bool self, int tiles, float* part,
                     int64_t seg_stride, hipStream_t s)
{
    const Params& p = h.prm;
    // the FP32 MFMA contraction exists in the wave-specialised kernel only
    const bool ws = mixed_uses_ws(h, pl, tiles);
    const int longest = h.precision == BAEMM_PRECISION_MIXED ? pl.steps : (tiles <= 256 ? kSubStepsSmall : kSubSteps);
    const int subs = (pl.steps + longest - 1) / longest;
    // an even number of steps, two to a stage of the single-wave kernel
    const int len = subs > 1 ? ((pl.steps + subs - 1) / subs + 1) & ~1 : pl.steps;
    Timed tm(h, s);
    for (int q0 = 0; q0 < p.K;) {
        int kg = pick_kg(pl.WCSP, (int)p.K - q0, true);
        if (ws) kg = std::min(kg, 2);
        const CoefPack cp = make_pack(p, q0, kg, pl.sA.data(), pl.rot.data());
        const MixedFn fn = ws ? mixed_ws_fn(pl.adj, pl.WCSP, kg, pl.f32, pl.tn)
                              : mixed_fn(pl.adj, pl.WCSP, kg, &cp, pl.tn);
        for (int off = 0; off < pl.steps; off += len)
            hipLaunchKernelGGL(fn, dim3(tiles, pl.S), dim3(ws ? 512 : 256), 0, s, tgt, ntgt, self ? 1 : 0, h.d_mid,
                               pl.nrm, (int)h.nt, pl.bop, pl.nst, cp, part, seg_stride, pl.ldp, q0,
                               StepRange{pl.steps, off, len}, self ? h.step_skip : nullptr);
        BAEMM_HIP(hipGetLastError());
        q0 += kg;
    }
    tm.done();
}

void bdr_pairs(Handle& h, BdrPlan& pl, hipStream_t s)
{
    if (!pl.kernel_on) return;
    float* part = bdr_reserve_part(h, pl, pl.S);
    if (!pl.mixed) {
        run_plain(h, OP_BDR, pl.adj, pl.WCSP, h.d_mid, h.d_nrm, (int)h.nt, (int)h.nt_pad, h.d_mid, h.d_nrm,
                  (int)h.nt, (int)h.nt_pad, pl.b, pl.ldb, part, pl.ea.seg_stride, pl.ldp, pl.S, pl.seg_len, s);
        return;
    }
    run_mfma(h, pl, h.d_mid, (int)h.nt_pad, true, (int)(h.nt_pad / kMixTile), part, pl.ea.seg_stride, s);
}

void bdr_end(Handle& h, const ApplyArgs& a, BdrPlan& pl, hipStream_t s)
{
    if (!pl.kernel_on && !pl.mass_on) return;
    EpiArgs& ea = pl.ea;
    ea.tsum = nullptr;
    if (use_tsum(pl)) {
        // each triangle's value once, then the vertex gather reads them (three
        // vertices per triangle) instead of every segment's partials
        const int nt = (int)h.nt;
        double2* ts = static_cast<double2*>(pl.ws.take(h.ws_tsum, sizeof(double2) * h.nt_pad * pl.ldb));
        const int64_t total = (int64_t)nt * ea.W;
        with_segment_threads(total, ea.S, [&](auto sw) {
            constexpr int SW = decltype(sw)::value;
            hipLaunchKernelGGL(tri_epilogue_kernel<SW>, dim3((unsigned)((total + kSegElems<SW> - 1) / kSegElems<SW>)),
                               dim3(kSegThreads<SW>), 0, s, ea, nt, ts);
        });
        BAEMM_HIP(hipGetLastError());
        ea.tsum = ts;
    }
    bdr_epilogue(h, ea, a.Btype, a.Ctype, s);
}

void apply_boundary_dev(Handle& h, const ApplyArgs& a, hipStream_t s, char* scratch, size_t scratch_bytes)
{
    BdrPlan pl;
    bdr_setup(h, pl, s);
    if (scratch) {
        // the first plan that fits: the automatic one; the kernels of the precision's own
        // arithmetic (the vector ALU for FP32, which pads to fewer columns) and the
        // automatic ones with few segments
        size_t need = bdr_workspace_bytes(h, pl), least = need;
        for (int k = 0; k < 2 && need > scratch_bytes; ++k) {
            const bool own = (h.precision == BAEMM_PRECISION_FP32) == (k == 0);
            pl = BdrPlan{};
            pl.lean = true;
            pl.plain_only = own && h.precision == BAEMM_PRECISION_FP32;
            pl.mfma_only = own && h.precision == BAEMM_PRECISION_MIXED;
            pl.f32_only = own && h.precision == BAEMM_PRECISION_FP32_MFMA;
            bdr_setup(h, pl, s);
            need = bdr_workspace_bytes(h, pl);
            least = std::min(least, need);
        }
        if (need > scratch_bytes)
            throw ArgError{"the apply needs " + std::to_string(least) + " bytes of workspace; the fixed scratch "
                           "array holds " + std::to_string(scratch_bytes)};
        pl.ws = WsSource{scratch, scratch_bytes, 0};
    }
    bdr_begin(h, a, pl, s);
    bdr_pairs(h, pl, s);
    bdr_end(h, a, pl, s);
    // the fixed scratch array is shared by every handle of the device: its
    // contents are no P0 buffer of this handle
    if (scratch) p0_invalidate(h);
    else if (pl.kernel_on) p0_record(h, pl.b, pl.ldb, pl.WCSP, &pl.ea);
}

static void rows_epilogue(int nrows, const Params& p, int WCSP, int S, int64_t seg_stride, int ldp, const float* part,
                          const ApplyArgs& a, hipStream_t s, const float* unscale = nullptr,
                          const std::vector<cdouble>* rotv = nullptr)
{
    ChunkRot rot;
    for (int q = 0; q < 64; ++q) {
        const cdouble f = (rotv && q < (int)rotv->size()) ? (*rotv)[q] : cdouble(1.0, 0.0);
        rot.r[q] = f.real();
        rot.i[q] = f.imag();
    }
    const int64_t total = (int64_t)nrows * p.W;
    with_segment_threads(total, S, [&](auto sw) {
        constexpr int SW = decltype(sw)::value;
        const auto fn = a.Ctype == kC128 ? &rows_epilogue_kernel<kC128, SW> : &rows_epilogue_kernel<kC64, SW>;
        hipLaunchKernelGGL(fn, dim3((unsigned)((total + kSegElems<SW> - 1) / kSegElems<SW>)), dim3(kSegThreads<SW>), 0, s,
                           nrows, (int)p.W, (int)p.wcs, WCSP, S, seg_stride, ldp, part, a.alpha.real(), a.alpha.imag(),
                           a.beta.real(), a.beta.imag(), a.C, a.ldC, unscale, rot);
    });
    BAEMM_HIP(hipGetLastError());
}

// Far field / potential share the structure "targets x triangles", b = Av B.
static void apply_rows_op(Handle& h, int op, const ApplyArgs& a, const float4* tx, int ntgt, int ntgt_pad,
                          hipStream_t s)
{
    const Params& p = h.prm;
    if (!p.loaded) throw ArgError{"parameters not loaded"};
    if (!(p.any(1) || p.any(2))) return;   // ApplyFarFieldOperators.hpp:83
    if (p.K > 64) throw ArgError{"at most 64 wave-number chunks are supported"};
    const int WCSP = wcsp_plain((int)p.wcs);
    const int ldb = (int)p.K * WCSP, ldp = 2 * ldb;
    h.ws_b32.reserve(sizeof(float2) * h.nt_pad * ldb);
    float2* b = h.ws_b32.as<float2>();
    launch_av(h, a.B, a.ldB, a.Btype, WCSP, b, ldb, s);
    const int tiles = ntgt_pad / kTile;
    const int seg_len = plain_seg_len(h, tiles, h.nt, h.nt_pad,
                                      (const void*)plain_fn(op, false, WCSP, pick_kg(WCSP, (int)p.K, false)));
    const int S = (int)((h.nt_pad + seg_len - 1) / seg_len);
    const int64_t seg_stride = (int64_t)ntgt_pad * ldp;
    h.ws_part.reserve(sizeof(float) * seg_stride * S);
    run_plain(h, op, false, WCSP, tx, nullptr, ntgt, ntgt_pad, h.d_mid, h.d_nrm, (int)h.nt, (int)h.nt_pad, b, ldb,
              h.ws_part.as<float>(), seg_stride, ldp, S, seg_len, s);
    rows_epilogue(ntgt, p, WCSP, S, seg_stride, ldp, h.ws_part.as<float>(), a, s);
    p0_record(h, b, ldb, WCSP, nullptr);
}

void apply_far_dev(Handle& h, const ApplyArgs& a, hipStream_t s)
{
    if (h.m < 1) throw ArgError{"no measurement directions"};
    apply_rows_op(h, OP_FAR, a, h.d_meas, (int)h.m, (int)h.m_pad, s);
}

// Potential at P points with the MFMA kernels: the boundary kernels with the
// points as targets and no pair left out (NearFieldOperatorKernel.cl uses the
// same single/double-layer kernel values), then the row epilogue with the
// scales and chunk factors.  Returns false where the FP32 precision takes the
// vector-ALU kernel instead.
static bool apply_near_mfma(Handle& h, const ApplyArgs& a, const float4* d_pts, const double* pts, int P,
                            hipStream_t s)
{
    const Params& p = h.prm;
    BdrPlan pl;
    pl.kernel_on = pl.mixed = true;
    // no adjoint double layer for points: the general form only for chunks without c2
    pl.adj = false;
    for (int q = 0; q < p.K; ++q)
        if (p.c[4 * q + 2] == cfloat(0.0f, 0.0f)) pl.adj = true;
    if (may_be_plain(h) && !mfma_points(h, P)) {
        // MIXED leaves the matrix cores only for segments of up to 32 sources, whose
        // error is smaller; with 64 the vector ALU's is the larger one (5,400
        // triangles, 10,001 points 2.99e-7 against 2.79e-7)
        if (h.precision == BAEMM_PRECISION_FP32) return false;
        const int WCSP = wcsp_plain((int)p.wcs);
        if (plain_seg_len(h, (P + kTile - 1) / kTile, h.nt, h.nt_pad,
                          (const void*)plain_fn(OP_NEAR, false, WCSP, pick_kg(WCSP, (int)p.K, false))) <= 32)
            return false;
    }
    // FP32_MFMA with few pairs: the FP32 matrix instructions, with fewer launches and no
    // distances (one wave number of 8 columns: 3,266 triangles, 400 points 71 us against
    // 101 split, 5,400 triangles, 2,500 points 113 / 139, 20,416 triangles, 2,500 points
    // 220 / 225; two of 32: 9,922 triangles, 400 points 266 / 286, 2,500 points 494 / 467; of 16:
    // 6,936 triangles, 3,000 points 265 / 285, 12,972 triangles, 3,000 points 366 / 357)
    DistRange dr{0.0f, 0.0f};
    PairPath path = PairPath::kF32;
    if (!f32_sizes(h) &&
        (h.precision != BAEMM_PRECISION_FP32_MFMA || (double)P * (double)h.nt * (double)p.K >= 6e7)) {
        // (the host's loop takes 5 us at 10,000 points; the pass over all pairs and its
        // synchronisation 60 us at 20,001 points and 20,480 triangles)
        dr = outside_range(h, pts, P);
        if (!(dr.rmin > 0.0f))
            dr = distance_range(h, d_pts, P, false, static_cast<unsigned*>(pl.ws.take(h.ws_misc, 256)), s);
        path = mfma_path(h, pl.adj, false, dr.rmin, dr.rmax);
    }
    if (path == PairPath::kPlain) return false;
    pl.f32 = path == PairPath::kF32;
    pl.WCSP = wcsp_mixed((int)p.wcs);
    pl.ldb = (int)p.K * pl.WCSP;
    pl.ldp = 2 * pl.ldb;
    pl.nrm = h.d_nrm;
    pl.nst = (int)(h.nt_pad / 8);
    pl.b = static_cast<float2*>(pl.ws.take(h.ws_b32, sizeof(float2) * h.nt_pad * pl.ldb));
    stage_mfma(h, pl, dr.rmin, s, a.B, a.ldB, a.Btype);
    const int P_pad = (P + kMixTile - 1) / kMixTile * kMixTile;
    const int tiles = P_pad / kMixTile;
    plan_mfma_segments(h, pl, tiles, P);
    const int S = pl.S;
    const int64_t seg_stride = (int64_t)P_pad * pl.ldp;
    h.ws_part.reserve(sizeof(float) * seg_stride * S);
    float* part = h.ws_part.as<float>();
    run_mfma(h, pl, d_pts, P, false, tiles, part, seg_stride, s);
    rows_epilogue(P, p, pl.WCSP, S, seg_stride, pl.ldp, part, a, s, pl.unscale, &pl.back);
    p0_record(h, pl.b, pl.ldb, pl.WCSP, nullptr);
    return true;
}

void apply_near_dev(Handle& h, const ApplyArgs& a, const float4* d_pts, const double* pts, int64_t P, hipStream_t s)
{
    const Params& p = h.prm;
    if (p.loaded && (p.any(1) || p.any(2)) && p.K <= 64 && P > 0 && apply_near_mfma(h, a, d_pts, pts, (int)P, s)) return;
    const int P_pad = (int)(((P + kTile - 1) / kTile) * kTile);
    apply_rows_op(h, OP_NEAR, a, d_pts, (int)P, P_pad, s);
}

void herglotz_dev(Handle& h, const ApplyArgs& a, hipStream_t s)
{
    p0_invalidate(h);   // rewrites the workspaces; no P0 buffer of the reference kind
    const Params& p = h.prm;
    if (!p.loaded) throw ArgError{"parameters not loaded"};
    if (!(p.any(1) || p.any(2))) return;   // CreateHerglotzWave.hpp:200
    if (h.m < 1) throw ArgError{"no measurement directions"};
    if (p.K > 64) throw ArgError{"at most 64 wave-number chunks are supported"};
    const int WCSP = wcsp_plain((int)p.wcs);
    const int ldb = (int)p.K * WCSP, ldp = 2 * ldb;
    // g (m x W) -> conj(g) staged with m_pad rows (HerglotzWaveKernel.cl:143-144)
    h.ws_g.reserve(sizeof(float2) * h.m_pad * ldb);
    float2* gb = h.ws_g.as<float2>();
    const int64_t total = h.m_pad * (int64_t)ldb;
    const dim3 grid((unsigned)((total + 255) / 256));
    if (a.Btype == kC128)
        hipLaunchKernelGGL(stage_rows_kernel<kC128>, grid, dim3(256), 0, s, (int)h.m, total, a.B, a.ldB, (int)p.wcs,
                           WCSP, ldb, 1, gb);
    else
        hipLaunchKernelGGL(stage_rows_kernel<kC64>, grid, dim3(256), 0, s, (int)h.m, total, a.B, a.ldB, (int)p.wcs,
                           WCSP, ldb, 1, gb);
    BAEMM_HIP(hipGetLastError());
    const int tiles = (int)(h.nt_pad / kTile);
    const int seg_len = plain_seg_len(h, tiles, h.m, h.m_pad,
                                      (const void*)plain_fn(OP_HERG, false, WCSP, pick_kg(WCSP, (int)p.K, false)));
    const int S = (int)((h.m_pad + seg_len - 1) / seg_len);
    const int64_t seg_stride = h.nt_pad * (int64_t)ldp;
    h.ws_part.reserve(sizeof(float) * seg_stride * S);
    run_plain(h, OP_HERG, false, WCSP, h.d_mid, h.d_nrm, (int)h.nt, (int)h.nt_pad, h.d_meas, nullptr, (int)h.m,
              (int)h.m_pad, gb, ldb, h.ws_part.as<float>(), seg_stride, ldp, S, seg_len, s);
    EpiArgs ea = base_epi(h, a, WCSP);
    ea.kernel_on = 1;
    ea.diag_on = 0;
    ea.mass_on = 0;
    ea.S = S;
    ea.seg_stride = seg_stride;
    ea.ldp = ldp;
    ea.ldb = ldb;
    ea.part = h.ws_part.as<float>();
    ea.b = gb;
    ea.unscale = nullptr;
    bdr_epilogue(h, ea, kC64, a.Ctype, s);
}

void incident_dev(Handle& h, const ApplyArgs& a, const double* dirs, int64_t inc_count, int wave_type,
                  hipStream_t s)
{
    p0_invalidate(h);   // rewrites the workspaces; no P0 buffer of the reference kind
    const Params& p = h.prm;
    if (!p.loaded) throw ArgError{"parameters not loaded"};
    if (!(p.any(1) || p.any(2))) return;   // CreateIncidentWave.hpp:95
    if (!dirs) throw ArgError{"incident directions must not be NULL"};
    if (inc_count < p.wcs) throw ArgError{"inc_count must be >= wave_chunk_size"};
    if (p.wcs > 64 || p.K > 64) throw ArgError{"at most 64 directions and 64 chunks are supported"};
    if (wave_type != BAEMM_WAVE_PLANE && wave_type != BAEMM_WAVE_RADIAL) throw ArgError{"unknown wave type"};
    const int WCSP = (int)p.wcs;
    const int ldp = 2 * (int)p.K * WCSP;
    h.ws_part.reserve(sizeof(float) * h.nt_pad * ldp);
    IncArgs ia{};
    ia.nt = (int)h.nt;
    ia.W = (int)p.W;
    ia.wcs = (int)p.wcs;
    ia.WCSP = WCSP;
    ia.ldp = ldp;
    ia.radial = (wave_type == BAEMM_WAVE_RADIAL);
    ia.mid = h.d_mid;
    ia.nrm = h.d_nrm;
    ia.part = h.ws_part.as<float>();
    for (int j = 0; j < p.wcs; ++j)
        for (int d = 0; d < 3; ++d) ia.dirs[j][d] = (float)dirs[3 * j + d];
    for (int q = 0; q < p.K; ++q) {
        ia.kap[q] = p.kappa[q];
        ia.c1r[q] = p.c[4 * q + 1].real();
        ia.c1i[q] = p.c[4 * q + 1].imag();
        ia.c2r[q] = p.c[4 * q + 2].real();
        ia.c2i[q] = p.c[4 * q + 2].imag();
    }
    const int64_t total = h.nt * p.W;
    hipLaunchKernelGGL(incident_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, ia);
    BAEMM_HIP(hipGetLastError());
    EpiArgs ea = base_epi(h, a, WCSP);
    ea.kernel_on = 1;
    ea.diag_on = 0;
    ea.mass_on = 0;
    ea.S = 1;
    ea.seg_stride = 0;
    ea.ldp = ldp;
    ea.ldb = 0;
    ea.part = h.ws_part.as<float>();
    ea.b = nullptr;
    ea.unscale = nullptr;
    bdr_epilogue(h, ea, kC64, a.Ctype, s);
}


// --------------------------------------------------------------- P0 buffers

// The reference's P0 buffers (InputOutput.hpp) from the device data of the
// last apply, as complex float, simplex_count x W: which = 0: B, the staged
// sources b[t][k]; which = 1: C, the triangle values before AvT,
// rot_q * unscale_k * sum_s part_s[t][k] + D_t b[t][k] (the inner term of
// bdr_epilogue_kernel, summed in the same order in FP64).
__global__ void p0_kernel(P0Source src, int which, int nt, const float* __restrict__ sdiag,
                          float2* __restrict__ out)
{
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)nt * src.W) return;
    const int t = (int)(idx / src.W), k = (int)(idx % src.W);
    const int q = k / src.wcs, kk = k % src.wcs;
    const int pc = q * src.WCSP + kk;
    const float2 bv = src.bptr[(int64_t)t * src.ldb + pc];
    if (which == 0) {
        out[idx] = bv;
        return;
    }
    double pr = 0.0, pi = 0.0;
    const float* pp = src.part + (int64_t)t * src.ldp + q * 2 * src.WCSP + kk;
    for (int sg = 0; sg < src.S; ++sg) {
        pr += (double)pp[(int64_t)sg * src.seg_stride];
        pi += (double)pp[(int64_t)sg * src.seg_stride + src.WCSP];
    }
    const double us = src.unscale ? (double)src.unscale[pc] : 1.0;
    double qr = pr * us, qi = pi * us;
    const double rr = src.rotr[q], ri = src.roti[q];
    const double tr = qr * rr - qi * ri;
    qi = qr * ri + qi * rr;
    qr = tr;
    if (src.diag) {
        const double fr = (double)src.c1r[q] * sdiag[t] - (double)src.c1i[q] * src.kap[q];
        const double fi = (double)src.c1i[q] * sdiag[t] + (double)src.c1r[q] * src.kap[q];
        qr += fr * bv.x - fi * bv.y;
        qi += fr * bv.y + fi * bv.x;
    }
    out[idx] = make_float2((float)qr, (float)qi);
}

// Records the device data of an apply as the source of the P0 buffers: b
// (B) and, for a boundary-operator apply (ea != null), the partials behind C.
static void p0_record(Handle& h, const float2* b, int ldb, int WCSP, const EpiArgs* ea)
{
    const Params& p = h.prm;
    P0Source& src = h.p0.src;
    src.b = b != nullptr;
    src.bptr = b;
    src.ldb = ldb;
    src.WCSP = WCSP;
    src.wcs = (int)p.wcs;
    src.K = (int)p.K;
    src.W = (int)p.W;
    h.p0.host_current[0] = false;
    h.p0.host_current[1] = false;
    src.c = ea != nullptr && ea->kernel_on;
    if (!src.c) return;
    src.part = ea->part;
    src.S = ea->S;
    src.ldp = ea->ldp;
    src.seg_stride = ea->seg_stride;
    src.unscale = ea->unscale;
    src.diag = ea->diag_on != 0;
    for (int q = 0; q < p.K; ++q) {
        src.rotr[q] = ea->rotr[q];
        src.roti[q] = ea->roti[q];
        src.c1r[q] = ea->c1r[q];
        src.c1i[q] = ea->c1i[q];
        src.kap[q] = ea->kap[q];
    }
}

void p0_invalidate(Handle& h)
{
    h.p0.src.b = h.p0.src.c = false;
    h.p0.host_current[0] = h.p0.host_current[1] = false;
}

bool p0_sync(Handle& h, int which, hipStream_t s)
{
    P0State& st = h.p0;
    if (st.host_current[which]) return true;
    const P0Source& src = st.src;
    if (!(which == 0 ? src.b : src.c)) return false;
    const int64_t n = h.nt * (int64_t)src.W;
    h.ws_p0.reserve(sizeof(float2) * std::max<int64_t>(n, 1));
    hipLaunchKernelGGL(p0_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, src, which, (int)h.nt, h.d_sdiag,
                       h.ws_p0.as<float2>());
    BAEMM_HIP(hipGetLastError());
    st.host[which].resize((size_t)n);
    BAEMM_HIP(hipMemcpyAsync(st.host[which].data(), h.ws_p0.ptr, sizeof(float2) * n, hipMemcpyDeviceToHost, s));
    BAEMM_HIP(hipStreamSynchronize(s));
    st.W[which] = src.W;
    st.host_current[which] = true;
    return true;
}

// --------------------------------------------------------------- diagnostics

__global__ void hw_sincos_kernel(const float* __restrict__ rev, int64_t n, float* __restrict__ s,
                                 float* __restrict__ c)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    s[i] = hw_sin_rev(rev[i]);
    c[i] = hw_cos_rev(rev[i]);
}

void hw_sincos_dev(const float* rev, int64_t n, float* sin_out, float* cos_out, hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(hw_sincos_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, rev, n, sin_out,
                       cos_out);
    BAEMM_HIP(hipGetLastError());
}

}  // namespace baemm
