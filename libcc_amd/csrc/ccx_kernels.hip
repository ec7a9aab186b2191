// Closed-shell (T) triples correction on gfx950: device kernels and their thin C ABI.
//
// Formulation (closed form of what src/triples-ijk/ijk_tuple.f90:56-84 builds with 12
// DGEMMs and trant3 steps):
//
//   W_ijk(a,b,c) = sum over the 6 simultaneous permutations s of the pairs (i,a),(j,b),(k,c)
//                  of  sum_K AX[x](alpha,beta,K) * BX[y,z](gamma,K)
//   AX[x](alpha,beta,K) = VVVO(K,beta,alpha,x)      K <  nu
//                       = T2(alpha,beta,K-nu,x)     nu <= K < nu+no
//   BX[y,z](gamma,K)    = T2(gamma,K,y,z)           K <  nu
//                       = -VM(K-nu,gamma,z,y)       nu <= K < nu+no
//
// with (x,alpha),(y,beta),(z,gamma) the permuted pairs.  Particle (VVVO*T2, K=nu) and
// hole (T2*VM, K=no) contractions are one GEMM over K = nu+no.
//
// Work item = (occupied tuple, virtual block orbit).  The virtual cube is cut into
// 16^3 blocks; a work item owns the blocks (A<=B<=C) and accumulates, for the
// orderings P of its occupied tuple, w_P(a,b,c) = W_P(a,b,c) over (a,b,c) in A x B x C.
// Because W_{pi.P}(pi.e) = W_P(e) (pi permuting tuple positions and virtual positions
// alike), the six w_P hold W_ijk at the six positional permutations of (a,b,c), in the
// SAME register slot, so the energy needs no transposition of W:
//   sum_s f(s.e) = Q(w) / D,  Q = 6 sum w_P^2 + 2 E^2 + 2 O^2 - 8 E O,
//   E = w over even orderings, O = w over odd orderings,
// f being the summand of t1wt3_ijk's E[T] loop (src/triples-ijk/t1wt3.f90:143-159).
// Degenerate tuples (i,j,j)/(i,i,j) have three distinct orderings; blocks with equal
// edges (A=B, B=C, A=B=C) get the missing orderings by an in-block transpose, so no
// ordering is computed twice.  The index permutations (trant3,
// src/common/common_cc.f90:62-333) become the choice of operand slab and orientation.
//
// FP64 MFMA v_mfma_f64_16x16x4_f64: lane l supplies A[l%16][l/16] and B[l/16][l%16]
// and holds D[l/16 + 4v][l%16], v = 0..3 (checked on the device).

#include "ccx_item.h"
extern "C" {
#include "ccx_dev.h"
}
#include <stdlib.h>
#include <string.h>


// ---------------------------------------------------------------------------------
// packing kernels (once per problem)
// ---------------------------------------------------------------------------------
// Layouts VVVO comes in; (K, b, a, x) is the element VVVO(K,b,a,x), 0-based.
enum VvvoLayout {
    V_FULL = 0,     // (nu, nu, nu, no)
    V_PACKED = 1,   // distributed (nutr, nu no): column a + nu x holds the lower-packed symmetric (K,b)
                    // block, row p (p+1)/2 + q for q <= p, as DDCC_T_GETVE / CPYTSQ expand it
                    // (src/triples-ijk/common_functions.f:43-60,106-125)
    V_VE = 2        // VE_x(K,a,b), the cube the reference's per-tuple routines take
};

template <int LAYOUT>
__device__ __forceinline__ double vvvo_at(const double *__restrict__ v, int nu, int x, int a, int b, int K)
{
    if constexpr (LAYOUT == V_FULL) {
        return v[K + (long long)nu * (b + (long long)nu * (a + (long long)nu * x))];
    } else if constexpr (LAYOUT == V_PACKED) {
        const int hi = K > b ? K : b, lo = K > b ? b : K;
        return v[(long long)hi * (hi + 1) / 2 + lo + ((long long)nu * (nu + 1) / 2) * (a + (long long)nu * x)];
    } else {
        return v[K + (long long)nu * (a + (long long)nu * (b + (long long)nu * x))];
    }
}

// Both orientations of the AX slab from VVVO and T2, for nx occupied indices from those the pointers
// stand at.  Bound by HBM: VVVO and T2 read once, the two slabs written once.  A work group takes
// PK_K K of one 16 x 16 panel through LDS, because no thread order is good for both ends: VVVO runs
// along K (packed, above the diagonal: along b), T2 along a, and the slabs' fragments are
// [outer/2][K/4][lane: K%4, inner][outer%2].  At no=8, nu=120 the two slabs took 144 us as two
// kernels with an index chain of 64-bit divisions per element and strided reads, and the packed
// layout first went through an unpacked copy.
constexpr int PK_K = 16;

template <int LAYOUT>
__global__ void __launch_bounds__(256) pack_ax_kernel(const double *__restrict__ vvvo, const double *__restrict__ t2,
                                                      double *__restrict__ axr, double *__restrict__ axc, int no,
                                                      int nu, int nb, int kp, int nkc)
{
    constexpr int STR = 273, STR_A = 17;
    __shared__ double tile[PK_K * STR];   // [K][a][b], padded for reads along a and writes along K
    const int tid = threadIdx.x;
    unsigned int u = blockIdx.x;
    const int kc = u % nkc; u /= nkc;
    const int Q = u % nb; u /= nb;
    const int P = u % nb;
    const int x = u / nb;
    const int K0 = kc * PK_K;
    if (K0 < nu) {
        const bool along_b = LAYOUT == V_PACKED && K0 + PK_K - 1 > Q * TB;
        for (int i = tid; i < PK_K * 256; i += 256) {
            const int k = along_b ? (i >> 4) & 15 : i & 15, row = along_b ? (i >> 8) * 16 + (i & 15) : i >> 4;
            const int a = P * TB + (row >> 4), b = Q * TB + (row & 15), K = K0 + k;
            if (K < nu) tile[k * STR + (row >> 4) * STR_A + (row & 15)] = a < nu && b < nu ? vvvo_at<LAYOUT>(vvvo, nu, x, a, b, K) : 0.0;
        }
    }
    if (K0 + PK_K > nu)
        for (int i = tid; i < PK_K * 256; i += 256) {
            const int k = i >> 8, row = (i & 15) * 16 + ((i >> 4) & 15);
            const int a = P * TB + (row >> 4), b = Q * TB + (row & 15), K = K0 + k;
            if (K >= nu)
                tile[k * STR + (row >> 4) * STR_A + (row & 15)] = a < nu && b < nu && K < nu + no
                    ? t2[a + (long long)nu * (b + (long long)nu * ((K - nu) + (long long)no * x))] : 0.0;
        }
    __syncthreads();
    const long long panel = (((long long)x * nb + P) * nb + Q) * (256LL * kp);
    for (int i = tid; i < PK_K * 128; i += 256) {
        const int lane = i & 63, kb = (i >> 6) & 3, pr = i >> 8;      // outer pair pr
        if (K0 / 4 + kb >= kp / 4) continue;
        const double *r = tile + (kb * 4 + (lane >> 4)) * STR;
        const int in = lane & 15;
        const long long o = panel + ((long long)pr * (kp / 4) + K0 / 4 + kb) * 128 + lane * 2;
        *reinterpret_cast<double2 *>(axr + o) = make_double2(r[2 * pr * STR_A + in], r[(2 * pr + 1) * STR_A + in]);
        *reinterpret_cast<double2 *>(axc + o) = make_double2(r[in * STR_A + 2 * pr], r[in * STR_A + 2 * pr + 1]);
    }
}

// BX[y,z](g,K) = T2(g,K,y,z) for K < nu, -VM(K-nu,g,z,y) after, [y][z][g block][K][16]
__device__ __forceinline__ void pack_bx(const double *__restrict__ t2, const double *__restrict__ vm,
                                        double *__restrict__ bx, int no, int nu, int nb, int kp, int wg, int nwg)
{
    const long long total = (long long)no * no * nb * kp * 16;
    for (long long idx = wg * 256LL + threadIdx.x; idx < total; idx += nwg * 256LL) {
        const int gl = (int)(idx & 15);
        const long long r = idx >> 4, pg = r / kp;
        const int K = (int)(r - pg * kp), yz = (int)(pg / nb), g = (int)(pg - (long long)yz * nb) * TB + gl;
        const int y = yz / no, z = yz % no;
        double v = 0.0;
        if (g < nu) {
            if (K < nu) v = t2[g + (long long)nu * (K + (long long)nu * (y + (long long)no * z))];
            else if (K < nu + no) v = -vm[(K - nu) + (long long)no * (g + (long long)nu * (z + (long long)no * y))];
        }
        bx[idx] = v;
    }
}

// out[q][r][x][y] = VOE(x,y,q,r), zero past nu, by 16 x 16 tiles through LDS (VOE runs along x, out along y)
__device__ __forceinline__ void pack_voe(const double *__restrict__ voe, double *__restrict__ out, int no, int nu,
                                         int nup, int wg, int nwg)
{
    __shared__ double tile[16 * 17];
    const int nb = nup / TB, i = threadIdx.x & 15, j = threadIdx.x >> 4;
    const long long ntile = (long long)no * no * nb * nb;
    for (long long u = wg; u < ntile; u += nwg) {
        const int Y = (int)(u % nb), X = (int)(u / nb % nb);
        const long long qr = u / nb / nb;               // q no + r
        const int q = (int)(qr / no), r = (int)(qr % no);
        const int x = X * TB + i, y = Y * TB + j;
        tile[i * 17 + j] = x < nu && y < nu ? voe[x + (long long)nu * (y + (long long)nu * (q + (long long)no * r))] : 0.0;
        __syncthreads();
        out[(qr * nup + X * TB + j) * nup + Y * TB + i] = tile[j * 17 + i];
        __syncthreads();
    }
}

// The rest of a problem in one launch: BX, the padded VOE, and the small arrays (eps_virtual padded
// with finite values, since padded elements carry W = 0; eps_occupied and T1 copied).
struct RestArgs {
    const double *t2, *vm, *voe, *eh, *ep, *t1;
    double *bx, *voep, *ehp, *epp, *t1p;   // the last three may be null
    int no, nu, nup, kp, gbx, gvoe;
};
__global__ void __launch_bounds__(256) pack_rest_kernel(RestArgs a)
{
    const int wg = blockIdx.x;
    if (wg < a.gbx) pack_bx(a.t2, a.vm, a.bx, a.no, a.nu, a.nup / TB, a.kp, wg, a.gbx);
    else if (wg < a.gbx + a.gvoe) pack_voe(a.voe, a.voep, a.no, a.nu, a.nup, wg - a.gbx, a.gvoe);
    else {
        if (a.epp) for (int i = threadIdx.x; i < a.nup; i += 256) a.epp[i] = i < a.nu ? a.ep[i] : 1.0e3;
        if (a.ehp) for (int i = threadIdx.x; i < a.no; i += 256) a.ehp[i] = a.eh[i];
        if (a.t1p) for (int i = threadIdx.x; i < a.no * a.nu; i += 256) a.t1p[i] = a.t1[i];
    }
}

// The pairs of one tuple (at most six) in one launch: BX[y,z](g,K) = T2(g,K,y,z) for K < nu, then
// -VM(K-nu,g,z,y), as [g block][kp][16], and the padded VOE block of each pair that has one.
// t2 = T2(:,:,y,z) (nu^2), vm = VM(:,:,z,y) (no nu), voe = VOE(:,:,y,z).  Work groups 0 .. npb-1 of
// a pair build BX, the others VOE; as two launches a pair these were 12 of the call's 30.
struct PairArgs {
    ccx_pair_pack p[6];
    int no, nu, nup, kp, npb, npv;
};
__global__ void __launch_bounds__(256) pack_pairs_kernel(PairArgs a)
{
    const int per = a.npb + a.npv, wg = blockIdx.x % per;
    const ccx_pair_pack &p = a.p[blockIdx.x / per];
    if (wg >= a.npb) {
        if (p.voe) pack_voe(p.voe, p.voep, 1, a.nu, a.nup, wg - a.npb, a.npv);
        return;
    }
    const long long total = (long long)(a.nup / TB) * a.kp * 16;
    for (long long idx = wg * 256LL + threadIdx.x; idx < total; idx += a.npb * 256LL) {
        const int gl = (int)(idx & 15), gk = (int)(idx >> 4), gb = gk / a.kp, K = gk - gb * a.kp, g = gb * TB + gl;
        double v = 0.0;
        if (g < a.nu) {
            if (K < a.nu) v = p.t2[g + (long long)a.nu * K];
            else if (K < a.nu + a.no) v = -p.vm[(K - a.nu) + (long long)a.no * g];
        }
        p.bx[idx] = v;
    }
}

// ---------------------------------------------------------------------------------
// split forms: fixed-point digit slices of the FP64 operand slabs
// ---------------------------------------------------------------------------------

// max |x| over a slab (non-negative doubles order like their bit patterns).  One atomic per work
// group, and few work groups: with one per wave of 65536 groups the atomics, which all go to one
// address, took 4.6 ms at no=16, nu=181 (a pass over the slab takes 0.2 ms).
__global__ void __launch_bounds__(256) absmax_kernel(const double *__restrict__ x, long long n,
                                                     unsigned long long *__restrict__ out)
{
    __shared__ double part[4];
    double m = 0.0;
    const long long step = (long long)gridDim.x * blockDim.x;
    long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    for (; i + 3 * step < n; i += 4 * step) {   // four loads in flight
        const double a = fabs(x[i]), b = fabs(x[i + step]), c = fabs(x[i + 2 * step]), d = fabs(x[i + 3 * step]);
        m = fmax(fmax(m, fmax(a, b)), fmax(c, d));
    }
    for (; i < n; i += step) m = fmax(m, fabs(x[i]));
    for (int off = 32; off >= 1; off >>= 1) m = fmax(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0)
        atomicMax(out, (unsigned long long)__double_as_longlong(fmax(fmax(part[0], part[1]), fmax(part[2], part[3]))));
}

// OCP e4m3 byte of an integer |d| <= 16 (every such integer has at most 4 significant bits)
__device__ __forceinline__ unsigned char e4m3_of_int(int d)
{
    if (d == 0) return 0;
    const unsigned char sgn = d < 0 ? 0x80 : 0;
    const int m = d < 0 ? -d : d;
    const int p = 31 - __builtin_clz(m);          // 2^p <= m < 2^(p+1)
    const int frac = ((m << 3) >> p) & 7;         // the three bits after the leading one
    return sgn | (unsigned char)((p + 7) << 3) | (unsigned char)frac;
}

// Slices of a slab in the fragment order of the form's MFMA (see run_phase_split).  One thread
// per group of EL elements of one row (AX: row = the panel's outer index; BX: no outer index),
// inner index lane & 15.  Output: [panel][outer][kb][slice][16-byte unit f][lane][16 B].  The MFMA
// sums over every K of a block, so any placement of K inside a block that A and B share gives
// the same products:
//   bf16 (EL 8): the group is lane's fragment, K = 32 kb + 8 (lane >> 4) + e;
//   fp8 (EL 32): the group is scale block b = lane >> 4 of the 128-K block (K = 128 kb + 32 b + q,
//     q < 32), which v_mfma_scale_f32_16x16x128_f8f6f4 reads as bytes 16 (b >> 1) + (q & 15) of
//     lanes 16 (2 (b & 1) + (q >> 4)) + row and scales with the word of lane 16 b + row (the
//     layout measured on the device); the group's exponent word goes to [panel][outer][kb][lane].
// Source: the FP64 slab, AX [panel][outer/2][K/4][lane 64][2] or BX [panel][K][16 gamma].
// inv_scale = 1 / sigma of the slab.
template <int FK, int BX>
__global__ void pack_split_kernel(const double *__restrict__ src, unsigned char *__restrict__ dst,
                                  int *__restrict__ dexp, long long npanel, int kp, int kps, double inv_scale)
{
    typedef SplitCfg<FK> CF;
    constexpr int NS = CF::NS, F16 = CF::F16, KB = CF::KB;
    constexpr int EL = CF::FMT == 0 ? 8 : 32, EB = CF::FMT == 0 ? 2 : 1;
    const int nkb = kps / KB;
    const long long ngroups = npanel * (BX ? 1 : 16) * nkb * 64;
    for (long long gi = blockIdx.x * (long long)blockDim.x + threadIdx.x; gi < ngroups;
         gi += (long long)gridDim.x * blockDim.x) {
        const int lane = (int)(gi & 63);
        const long long rr = gi >> 6;      // (panel, outer, kb) or (panel, kb)
        const int kb = (int)(rr % nkb);
        const long long po = rr / nkb;     // panel * 16 + outer, or panel
        const int inner = lane & 15;
        double v[EL];
        double m = 0.0;
#pragma unroll
        for (int e = 0; e < EL; ++e) {
            const int K = kb * KB + (lane >> 4) * EL + e;
            double x = 0.0;
            if (K < kp) {
                if (BX) {
                    x = src[po * (16LL * kp) + (long long)K * 16 + inner];
                } else {
                    const int outer = (int)(po % 16);
                    const long long panel = po / 16;
                    x = src[panel * (256LL * kp) + (((long long)(outer >> 1) * (kp / 4) + K / 4) * 64 + (K & 3) * 16 + inner) * 2 +
                            (outer & 1)];
                }
            }
            v[e] = x * inv_scale;          // |v| <= 1
            m = fmax(m, fabs(v[e]));
        }
        int gexp = 0;                      // FP8 form: group exponent, |v| <= 2^gexp
        if constexpr (CF::MX) {
            if (m > 0.0) frexp(m, &gexp);
            if (gexp < -100) gexp = -100;  // a group this small is carried as zero digits
        }
#pragma unroll
        for (int e = 0; e < EL; ++e) {
            int f = (e * EB) / 16, byte = (e * EB) % 16, ol = lane;
            if constexpr (CF::MX) {   // element q = e of scale block b = lane >> 4
                const int b = lane >> 4;
                ol = 16 * (2 * (b & 1) + (e >> 4)) + inner;
                f = b >> 1;
                byte = e & 15;
            }
            double t = v[e];
            if constexpr (CF::MX) t = ldexp(t, -gexp);
#pragma unroll
            for (int sl = 0; sl < NS; ++sl) {
                const long long o = (((rr * NS + sl) * F16 + f) * 64 + ol) * 16 + byte;
                if constexpr (FK == 2) {          // per element: bf16 rounding of what is left
                    const __bf16 h = (__bf16)(float)t;
                    t -= (double)(float)h;
                    *reinterpret_cast<__bf16 *>(dst + o) = h;
                } else if constexpr (FK == 4) {   // fixed point: digits base 2^8
                    t *= 256.0;
                    const double d = rint(t);
                    t -= d;
                    *reinterpret_cast<__bf16 *>(dst + o) = (__bf16)(float)ldexp(d, -8 * (sl + 1));   // exact
                } else {                          // digits base 2^4 as e4m3 integers
                    t *= 16.0;
                    const double d = rint(t);
                    t -= d;
                    dst[o] = gexp > -100 ? e4m3_of_int((int)d) : 0;
                }
            }
        }
        if constexpr (CF::MX) {
            // byte s: biased E8M0 exponent of slice s, 2^(gexp - 4(s+1))
            unsigned int w = 0;
#pragma unroll
            for (int sl = 0; sl < NS; ++sl) w |= (unsigned int)(127 + gexp - 4 * (sl + 1)) << (8 * sl);
            dexp[rr * 64 + lane] = (int)w;
        }
    }
}

// ---------------------------------------------------------------------------------
// persistent (tuple, block-orbit) kernel, FP64 MFMA
// ---------------------------------------------------------------------------------
namespace {

// Energy, v1 partials and the optional W store of one item from its six w (layout L).  One copy for
// every mode: the modes differ in the sweeps only (dispatch in triples_kernel), and the FP64 kernel
// is 80 KB of code instead of 324 KB.  Bound by the FP64 VALU and, before the reductions went to DPP
// and row swaps, by their LDS shuffles.  Of 475 kcycles per item at no=24, nu=216 the point loop took
// 15.8 and now takes 10.4 (two multiply-adds per v1 term instead of five operations), the
// reductions 15.9 and now 7.5; the kernel went from 1137 to 1109 ms there, from 4.79 to 4.49 ms
// at no=8, nu=120, where an item's sweeps are half as long (energy calls repeated on loaded slabs; 4.57 when
// a load comes before each), and FP32 from 783 to 753 ms (650 since its BX goes straight into LDS).
template <class T, int FK>
__device__ __forceinline__ void item_epilogue(const TriplesArgs &g, double *lds, double (*red)[112], const ItemCtx &it,
                                              const typename Mfma<T>::acc_t (&acc)[6][BPW],
                                              const f4 (&acc1)[FK == 4 ? 6 : 1][BPW], long long item, int tkind,
                                              int mult, bool swap_bc, int wave, int lane, int tid)
{
    const int A = it.blk[0], B = it.blk[1], C = it.blk[2];
    // ---- stage the 36 VOE sub-blocks: [ordered tuple-position pair][ordered block pair]
    for (int idx = tid; idx < 36 * 16 * 4; idx += NTHR) {
        const int quad = idx & 3, row = (idx >> 2) & 15, sb = idx >> 6;
        const int qr = sb / 6, bpair = sb % 6;
        const int y = qr >> 1, z = (qr & 1) ? (y == 2 ? 1 : 2) : (y == 0 ? 1 : 0);
        const int ry = bpair >> 1, rz = (bpair & 1) ? (ry == 2 ? 1 : 2) : (ry == 0 ? 1 : 0);
        const double *src = g.voe + (((long long)pick3(it.tpos, y) * g.no + pick3(it.tpos, z)) * g.nup
                                     + pick3(it.blk, ry) * TB + row) * g.nup + pick3(it.blk, rz) * TB + quad * 4;
        double *d = lds + sb * VBLK + row * VSTR + quad * 4;
        d[0] = src[0]; d[1] = src[1]; d[2] = src[2]; d[3] = src[3];
    }
    __syncthreads();

    // ---- epilogue: energy, v1 partials, optional W store
    const double dijk = g.eh[it.tpos[0]] + g.eh[it.tpos[1]] + g.eh[it.tpos[2]];
    const double wgt = (tkind == 1 ? 1.0 : 0.5) / (double)mult;
    double esum = 0.0;
    double va[4][3], vb[BPW][3], vc[3];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int p = 0; p < 3; ++p) va[i][p] = 0.0;
#pragma unroll
    for (int i = 0; i < BPW; ++i)
#pragma unroll
        for (int p = 0; p < 3; ++p) vb[i][p] = 0.0;
    vc[0] = vc[1] = vc[2] = 0.0;
    const int cl = lane & 15;
    const int cg = C * TB + cl;
#pragma unroll
    for (int bb = 0; bb < BPW; ++bb) {
        const int bl = wave * BPW + bb;
        const int bg = B * TB + bl;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int al = Mfma<T>::row(lane, v);
            const int ag = A * TB + al;
            if (ag >= g.nu || bg >= g.nu || cg >= g.nu) continue;
            double w[6];
#pragma unroll
            for (int p = 0; p < 6; ++p) {
                if constexpr (FK == 4) w[p] = ((double)acc[p][bb][v] + (double)acc1[p][bb][v]) * g.wscale;
                else if constexpr (FK >= 2) w[p] = (double)acc[p][bb][v] * g.wscale;
                else w[p] = (double)acc[p][bb][v];
            }
            const double inv = 1.0 / (dijk - g.ep[ag] - g.ep[bg] - g.ep[cg]);
            const double ev = w[0] + w[3] + w[4], od = w[1] + w[2] + w[5];
            const double sq = w[0] * w[0] + w[1] * w[1] + w[2] * w[2] + w[3] * w[3] + w[4] * w[4] + w[5] * w[5];
            esum += (6.0 * sq + 2.0 * ev * ev + 2.0 * od * od - 8.0 * ev * od) * inv;
            double d[3][3];
            even_odd_differences(w, inv, d);
            const int el[3] = {al, bl, cl};
            static_for<6>([&](auto S) __attribute__((always_inline)) {
                constexpr int s = decltype(S)::value;
                constexpr int r0 = PERM[s][0], r1 = PERM[s][1], r2 = PERM[s][2];
                constexpr int bpair = pair_index(r1, r2);
                static_for<6>([&](auto PP) __attribute__((always_inline)) {
                    constexpr int p = decltype(PP)::value;
                    constexpr int qr = pair_index(PERM[p][1], PERM[p][2]);
                    const double z = z_term<s, p>(d);
                    const double vv = lds[(qr * 6 + bpair) * VBLK + el[r1] * VSTR + el[r2]];
                    if constexpr (r0 == 0) va[v][PERM[p][0]] = fma(z, vv, va[v][PERM[p][0]]);
                    else if constexpr (r0 == 1) vb[bb][PERM[p][0]] = fma(z, vv, vb[bb][PERM[p][0]]);
                    else vc[PERM[p][0]] = fma(z, vv, vc[PERM[p][0]]);
                });
            });
            if (g.wout != nullptr) {
                const int xg[3] = {ag, bg, cg};
                static_for<6>([&](auto S) __attribute__((always_inline)) {
                    constexpr int s = decltype(S)::value;
                    constexpr int q0 = wsrc_comp(0, s, 0);
                    g.wout[xg[PERM[s][0]] + (long long)g.nu * (xg[PERM[s][1]] + (long long)g.nu * xg[PERM[s][2]])] = w[q0];
                });
            }
        }
    }

    // ---- deterministic reductions
    double *rw = red[wave];
#pragma unroll
    for (int v = 0; v < 4; ++v)          // role a: rows (lane>>4)+4v
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const double s = group16_sum(va[v][p]);
            if ((lane & 15) == 0) rw[Mfma<T>::row(lane, v) * 3 + p] = s;
        }
#pragma unroll
    for (int bb = 0; bb < BPW; ++bb)     // role b: rows wave*BPW+bb
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const double s = wave_sum(vb[bb][p]);
            if (lane == 0) rw[48 + bb * 3 + p] = s;
        }
#pragma unroll
    for (int p = 0; p < 3; ++p) {        // role c: rows lane&15
        const double s = add_xor32(add_xor16(vc[p]));
        if (lane < 16) rw[54 + lane * 3 + p] = s;
    }
    {
        const double s = wave_sum(esum);
        if (lane == 0) rw[102] = s;
    }
    __syncthreads();
    double *vp = g.v1_part + item * 144;
    const int slot_b = swap_bc ? 96 : 48, slot_c = swap_bc ? 48 : 96;   // table role order
    if (tid < 48) {
        double s = 0.0;
#pragma unroll
        for (int w2 = 0; w2 < NWAVE; ++w2) s += red[w2][tid];
        vp[tid] = s * wgt;
    } else if (tid < 96) {
        const int r = tid - 48, row = r / 3, p = r % 3;
        vp[slot_b + r] = red[row / BPW][48 + (row % BPW) * 3 + p] * wgt;
    } else if (tid < 144) {
        const int r = tid - 96;
        double s = 0.0;
#pragma unroll
        for (int w2 = 0; w2 < NWAVE; ++w2) s += red[w2][54 + r];
        vp[slot_c + r] = s * wgt;
    } else if (tid == 144) {
        double s = 0.0;
#pragma unroll
        for (int w2 = 0; w2 < NWAVE; ++w2) s += red[w2][102];
        g.e_part[item] = s * wgt;
    }
    __syncthreads();
}

}  // namespace

template <class T, int FK>
__global__ void __launch_bounds__(NTHR, 1) triples_kernel(TriplesArgs g)
{
    extern __shared__ double lds[];
    __shared__ double red[NWAVE][112];
    __shared__ long long next_item;
    // BX buffers of the FP32 and the split sweeps (run_phase_split).  The FP8 form's, 99 KB, do not fit beside the
    // transposition cubes and share their array.
    constexpr bool OWN_BX = FK == 2 || FK == 4;
    constexpr int BXU = FK >= 2 ? split_bx_units<FK >= 2 ? FK : 2>() : F32_BXU;
    __shared__ i32x4 bx0[OWN_BX || FK == 1 ? BXU : 1], bx1[OWN_BX || FK == 1 ? BXU : 1], bx2[FK == 1 ? BXU : 1];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    for (;;) {
        // The lane number is made new for every item: the LDS addresses that follow from it are then
        // computed where they are used, not kept through the sweeps (that is, in scratch).
        int lane = tid & 63;
        asm volatile("" : "+v"(lane));
        // Work order: block triple major (default), so the tuples of one block triple run
        // together and the operand panels they share stay in the last-level cache (34% less
        // L2 miss traffic than tuple major at no=24, nu=216); tuple major on request.
        if (tid == 0) {
            const unsigned int p = atomicAdd(g.counter, 1u);
            long long it = -1;
            if (p < g.nitems) it = g.block_major ? (long long)p : (long long)(p % g.nblk) * g.ntup + p / g.nblk;
            next_item = it;
        }
        __syncthreads();
        const long long pos = next_item;   // = q * ntup + t
        __syncthreads();
        if (pos < 0) break;
        const int q = __builtin_amdgcn_readfirstlane((int)(pos / g.ntup));
        const int t = __builtin_amdgcn_readfirstlane((int)(pos % g.ntup));
        const long long item = (long long)t * g.nblk + q;   // storage index
        int tkind, mult;
        ItemCtx it = make_item_ctx(g.tuples, g.blocks, t, q, tkind, mult);
        const bool swap_bc = ragged_block_to_b(g, it, mult);
        typename Mfma<T>::acc_t acc[6][BPW];
        f4 acc1[FK == 4 ? 6 : 1][BPW];   // two-accumulator split form: the levels above 0
        auto sweeps = [&](auto M) __attribute__((always_inline)) {
            constexpr int MODE = decltype(M)::value;
            if constexpr (OWN_BX) item_w_split<MODE, FK>(g, lds, it, acc, acc1, wave, lane, bx0, bx1);
            else if constexpr (FK >= 2)
                item_w_split<MODE, FK>(g, lds, it, acc, acc1, wave, lane, reinterpret_cast<i32x4 *>(lds),
                                       reinterpret_cast<i32x4 *>(lds) + BXU);
            else if constexpr (FK == 1)
                item_w_f32v<MODE>(g, lds, it, acc, wave, lane, reinterpret_cast<f4 *>(bx0), reinterpret_cast<f4 *>(bx1),
                                  reinterpret_cast<f4 *>(bx2));
            else item_w<MODE, T>(g, lds, it, acc, wave, lane);
        };
        if constexpr (pair_modes(FK)) {
            dispatch_mode(tkind, mult, it, sweeps);
        } else {
            if (tkind == 2) sweeps(std::integral_constant<int, M_IJJ>{});
            else if (tkind == 3) sweeps(std::integral_constant<int, M_IIJ>{});
            else if (mult == 1) sweeps(std::integral_constant<int, M_FULL>{});
            else if (mult == 6) sweeps(std::integral_constant<int, M_AAA>{});
            else if (it.blk[0] == it.blk[1]) sweeps(std::integral_constant<int, M_AAC>{});
            else sweeps(std::integral_constant<int, M_ACC>{});
        }
        item_epilogue<T, FK>(g, lds, red, it, acc, acc1, item, tkind, mult, swap_bc, wave, lane, tid);
    }
}

// ---------------------------------------------------------------------------------
// finalize: deterministic reductions
// ---------------------------------------------------------------------------------
// Index of the block orbit (A <= B <= C) in the table's order (A outermost, then B, then C).
__device__ __forceinline__ int orbit_index(int A, int B, int C, int nb)
{
    auto t2 = [](int n) { return n * (n + 1) / 2; };
    auto t3 = [](int n) { return n * (n + 1) * (n + 2) / 6; };
    return t3(nb) - t3(nb - A) + t2(nb - A) - t2(nb - B) + (C - B);
}

constexpr int RV_GRP = 5;             // groups of 48 lanes (virtual index of the block, tuple position)
constexpr int RE_CHUNKS = 256;        // most work groups of the energy sum

// Work groups 0 .. ntup nb - 1: v1t[t][a][p] for the 16 indices a of block ab, the sum over the orbits
// holding ab in some role.  Those are the orbits {ab, X, Y} of the pairs X <= Y, so the work group
// walks the pairs, RV_GRP at a time (with one lane per (t,a,p) walking all orbits, a few thousand
// lanes took serial chains of nblk loads: 111 us at no=4, nu=167 for 5 MB of partials, now 10).
// Work groups after them: the compensated sum of one chunk of the energy partials, left in the
// chunk's first element.  Every order is fixed.
__global__ void __launch_bounds__(256) reduce_partials_kernel(const double *__restrict__ v1_part, double *e_part,
                                                              double *__restrict__ v1t, int ntup, int nblk, int nu,
                                                              int nb, long long nitems, long long chunk)
{
    __shared__ double sh[256];
    const int tid = threadIdx.x;
    const long long wg = blockIdx.x;
    if (wg < (long long)ntup * nb) {
        const long long t = wg / nb;
        const int ab = (int)(wg % nb), grp = tid / 48, e = tid % 48;
        double s = 0.0;
        if (grp < RV_GRP) {
            const double *vt = v1_part + t * nblk * 144 + e;
            int X = 0, Y = grp;
            for (;;) {
                while (X < nb && Y >= nb) { ++X; Y += X - nb; }   // row X of the pair list holds Y = X .. nb-1
                if (X >= nb) break;
                const int lo = ab < X ? ab : X, hi = ab > Y ? ab : Y, mid = ab + X + Y - lo - hi;
                const double *vp = vt + (long long)orbit_index(lo, mid, hi, nb) * 144;
                if (lo == ab) s += vp[0];
                if (mid == ab) s += vp[48];
                if (hi == ab) s += vp[96];
                Y += RV_GRP;
            }
        }
        sh[tid] = s;
        __syncthreads();
        const int a = ab * TB + e / 3;
        if (tid < 48 && a < nu) {
            double r = sh[tid];
#pragma unroll
            for (int q = 1; q < RV_GRP; ++q) r += sh[q * 48 + tid];
            v1t[(t * nu + a) * 3 + e % 3] = r;
        }
    } else {
        const long long beg = (wg - (long long)ntup * nb) * chunk;
        const long long end = beg + chunk < nitems ? beg + chunk : nitems;
        double s = 0.0, c = 0.0;
        for (long long i = beg + tid; i < end; i += 256) {
            const double y = e_part[i], tt = s + y;
            c += (fabs(s) >= fabs(y)) ? ((s - tt) + y) : ((y - tt) + s);
            s = tt;
        }
        sh[tid] = s + c;
        __syncthreads();
        for (int w = 128; w >= 1; w >>= 1) {
            if (tid < w) sh[tid] += sh[tid + w];
            __syncthreads();
        }
        if (tid == 0) e_part[beg] = sh[0];
    }
}

// v1(a,o) (column-major nu x no) = sum over tuples and positions p with tuple[p] == o: work group per
// o and 64 indices a, four groups of lanes over the tuples, whose table entries pass through LDS.
__global__ void __launch_bounds__(256) reduce_v1_kernel(const double *__restrict__ v1t, const int *__restrict__ tuples,
                                                        double *__restrict__ v1, int ntup, int nu, int no)
{
    __shared__ int4 tab[256];
    __shared__ double sh[256];
    const int tid = threadIdx.x, grp = tid >> 6;
    const int na = (nu + 63) / 64, o = blockIdx.x / na, a = (blockIdx.x % na) * 64 + (tid & 63);
    double s = 0.0;
    for (int t0 = 0; t0 < ntup; t0 += 256) {
        const int n = ntup - t0 < 256 ? ntup - t0 : 256;
        if (tid < n) tab[tid] = reinterpret_cast<const int4 *>(tuples)[t0 + tid];
        __syncthreads();
        if (a < nu)
            for (int t = grp; t < n; t += 4) {
                const int4 tp = tab[t];
                const double *r = v1t + ((long long)(t0 + t) * nu + a) * 3;
                if (tp.x == o) s += r[0];
                if (tp.y == o) s += r[1];
                if (tp.z == o) s += r[2];
            }
        __syncthreads();
    }
    sh[tid] = s;
    __syncthreads();
    if (grp == 0 && a < nu) v1[a + (long long)nu * o] = (sh[tid] + sh[tid + 64]) + (sh[tid + 128] + sh[tid + 192]);
}

// out[0] = etd = sum of the chunk sums e_part[0], e_part[chunk], ...; out[1] = ets = 2 sum T1(o,a) v1(a,o)
// (both compensated, fixed order)
__global__ void __launch_bounds__(1024) finalize_energy_kernel(const double *__restrict__ e_part, int nchunk,
                                                               long long chunk, const double *__restrict__ t1,
                                                               const double *__restrict__ v1, int no, int nu,
                                                               double *__restrict__ out)
{
    __shared__ double sh[2][1024];
    const int tid = threadIdx.x;
    double s2 = 0.0, c2 = 0.0;
    for (int i = tid; i < no * nu; i += 1024) {
        const int a = i % nu, o = i / nu;
        const double y = t1[o + no * a] * v1[i];
        const double tt = s2 + y;
        c2 += (fabs(s2) >= fabs(y)) ? ((s2 - tt) + y) : ((y - tt) + s2);
        s2 = tt;
    }
    sh[0][tid] = tid < nchunk ? e_part[tid * chunk] : 0.0;
    sh[1][tid] = s2 + c2;
    __syncthreads();
    for (int w = 512; w >= 1; w >>= 1) {
        if (tid < w) {
            sh[0][tid] += sh[0][tid + w];
            sh[1][tid] += sh[1][tid + w];
        }
        __syncthreads();
    }
    if (tid == 0) {
        out[0] = sh[0][0];
        out[1] = 2.0 * sh[1][0];
    }
}

// E[T] and v1 of one tuple from a given W_ijk cube (nu^3, column-major), the computation of
// t1wt3_ijk (src/triples-ijk/t1wt3.f90:53-102) as a full sum over (b,c) per work group a:
//   x3[a]      = sum_{b,c, not a=b=c} W(abc) (8W(abc) - 4(W(acb)+W(cba)+W(bac)) + 2(W(bca)+W(cab))) / D
//   v1p[a][0]  = sum_{b,c} (Z_ijk(abc) VOE_jk(bc) + Z_ikj(abc) VOE_kj(bc)) / D     (row i)
//   v1p[a][1]  = sum_{b,c} (Z_jik(abc) VOE_ik(bc) + Z_kij(abc) VOE_ki(bc)) / D     (row j)
//   v1p[a][2]  = sum_{b,c} (Z_jki(abc) VOE_ij(bc) + Z_kji(abc) VOE_ji(bc)) / D     (row k)
// with Z_P the antisymmetric combination 2(W_P(abc)-W_P(bac)) - W_P(acb) + W_P(bca) of the
// cube read in ordering P.  voe6 = VOE(:,:,x,y) for xy = ij, ji, ik, ki, jk, kj.  Fixed-order
// tree reduction per work group: deterministic.
__global__ void __launch_bounds__(256) t1wt3_kernel(const double *__restrict__ w, const double *__restrict__ voe6,
                                                    double dijk, const double *__restrict__ ep, int nu,
                                                    double *__restrict__ x3, double *__restrict__ v1p)
{
    __shared__ double sh[4][256];
    const int a = blockIdx.x, tid = threadIdx.x;
    const long long n2 = (long long)nu * nu;
    auto W = [&](int x, int y, int z) { return w[x + (long long)nu * (y + (long long)nu * z)]; };
    double e = 0.0, ri = 0.0, rj = 0.0, rk = 0.0;
    for (long long bc = tid; bc < n2; bc += 256) {
        const int b = (int)(bc % nu), c = (int)(bc / nu);
        if (a == b && b == c) continue;
        const double inv = 1.0 / (dijk - ep[a] - ep[b] - ep[c]);
        const double abc = W(a, b, c), acb = W(a, c, b), bac = W(b, a, c);
        const double bca = W(b, c, a), cab = W(c, a, b), cba = W(c, b, a);
        e += abc * (8.0 * abc - 4.0 * (acb + cba + bac) + 2.0 * (bca + cab)) * inv;
        const double z1 = 2.0 * (abc - bac) - acb + bca;   // ijk
        const double z2 = 2.0 * (acb - bca) - abc + bac;   // ikj
        const double z3 = 2.0 * (bac - abc) - cab + cba;   // jik
        const double z4 = 2.0 * (bca - acb) - cba + cab;   // jki
        const double z5 = 2.0 * (cab - cba) - bac + abc;   // kij
        const double z6 = 2.0 * (cba - cab) - bca + acb;   // kji
        const long long o = b + (long long)nu * c;
        ri += (z1 * voe6[4 * n2 + o] + z2 * voe6[5 * n2 + o]) * inv;
        rj += (z3 * voe6[2 * n2 + o] + z5 * voe6[3 * n2 + o]) * inv;
        rk += (z4 * voe6[0 * n2 + o] + z6 * voe6[1 * n2 + o]) * inv;
    }
    sh[0][tid] = e; sh[1][tid] = ri; sh[2][tid] = rj; sh[3][tid] = rk;
    __syncthreads();
    for (int s2 = 128; s2 >= 1; s2 >>= 1) {
        if (tid < s2)
            for (int q = 0; q < 4; ++q) sh[q][tid] += sh[q][tid + s2];
        __syncthreads();
    }
    if (tid == 0) {
        x3[a] = sh[0][0];
        v1p[3 * a] = sh[1][0]; v1p[3 * a + 1] = sh[2][0]; v1p[3 * a + 2] = sh[3][0];
    }
}

__global__ void zero_counter_kernel(unsigned int *c) { *c = 0u; }

// flag |= 1 when any of the doubles of the arrays is NaN or infinite (one atomic per wave at most),
// all arrays in one launch
struct ScanArgs {
    const double *p[7];
    long long n[7];
    int narr;
};
__global__ void __launch_bounds__(256) nonfinite_kernel(ScanArgs a, unsigned int *__restrict__ flag)
{
    int bad = 0;
    const long long step = (long long)gridDim.x * blockDim.x, first = blockIdx.x * (long long)blockDim.x + threadIdx.x;
    for (int q = 0; q < a.narr; ++q) {
        const double *__restrict__ p = a.p[q];
        const long long n = a.n[q];
        long long i = first;
        for (; i + 3 * step < n; i += 4 * step) {   // four loads in flight
            const double x0 = p[i], x1 = p[i + step], x2 = p[i + 2 * step], x3 = p[i + 3 * step];
            bad |= !isfinite(x0) | !isfinite(x1) | !isfinite(x2) | !isfinite(x3);
        }
        for (; i < n; i += step) bad |= !isfinite(p[i]);
    }
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(flag, 1u);
}

// FP32 slabs from the FP64 ones in the FP32 sweep's fragment order: AX [panel][outer][K block
// of 16][lane][4], BX [panel][K block][lane][4]; lane l holds inner index l & 15, element j
// is at K = 16 kb + 4 j + (l >> 4).  BX = 1: the source is the BX slab [panel][K][16 gamma].
template <int BX>
__global__ void pack_f32v_kernel(const double *__restrict__ src, float *__restrict__ dst, long long npanel, int kp,
                                 int kpf)
{
    const int nkb = kpf / 16;
    const long long total = npanel * (BX ? 16LL : 256LL) * kpf;
    for (long long idx = blockIdx.x * (long long)blockDim.x + threadIdx.x; idx < total;
         idx += (long long)gridDim.x * blockDim.x) {
        const int j = (int)(idx & 3), lane = (int)((idx >> 2) & 63);
        const long long rr = idx >> 8;     // (panel, outer, kb) or (panel, kb)
        const int kb = (int)(rr % nkb);
        const long long po = rr / nkb;
        const int K = kb * 16 + j * 4 + (lane >> 4), inner = lane & 15;
        double v = 0.0;
        if (K < kp) {
            if (BX) {
                v = src[po * (16LL * kp) + (long long)K * 16 + inner];
            } else {
                const int outer = (int)(po % 16);
                const long long panel = po / 16;
                v = src[panel * (256LL * kp) + (((long long)(outer >> 1) * (kp / 4) + K / 4) * 64 + (K & 3) * 16 + inner) * 2 +
                        (outer & 1)];
            }
        }
        dst[idx] = (float)v;
    }
}

// grid-stride launches: enough work groups to fill the GPU, at most 65536
static int grid_for(long long total)
{
    long long g = (total + 255) / 256;
    if (g > 65536) g = 65536;
    if (g < 1) g = 1;
    return (int)g;
}

template <int FK>
static void launch_pack_split(const double *axr, const double *axc, const double *bx, void *const *sl, int no, int nb,
                              int kp, int kps, const double *sc, hipStream_t s)
{
    constexpr int EL = SplitCfg<FK>::FMT == 0 ? 8 : 32;
    const long long ax_g = (long long)no * nb * nb * 256 * kps / EL, bx_g = (long long)no * no * nb * 16 * kps / EL;
    pack_split_kernel<FK, 0><<<grid_for(ax_g), 256, 0, s>>>(axr, (unsigned char *)sl[0], (int *)sl[3],
                                                            (long long)no * nb * nb, kp, kps, 1.0 / sc[0]);
    pack_split_kernel<FK, 0><<<grid_for(ax_g), 256, 0, s>>>(axc, (unsigned char *)sl[1], (int *)sl[4],
                                                            (long long)no * nb * nb, kp, kps, 1.0 / sc[0]);
    pack_split_kernel<FK, 1><<<grid_for(bx_g), 256, 0, s>>>(bx, (unsigned char *)sl[2], (int *)sl[5],
                                                            (long long)no * no * nb, kp, kps, 1.0 / sc[1]);
}

// ---------------------------------------------------------------------------------
// thin C ABI used by the C host layer
// ---------------------------------------------------------------------------------
extern "C" {

int ccx_hip_device_count(int *n) { return hipGetDeviceCount(n) == hipSuccess ? 0 : 1; }

int ccx_hip_malloc(void **p, size_t bytes)
{
    *p = nullptr;
    if (bytes == 0) return 0;
    if (hipMalloc(p, bytes) == hipSuccess) return 0;
    *p = nullptr;
    (void)hipGetLastError();   // reported here: the check of a later launch must not find it
    return 1;
}

int ccx_hip_mem_info(size_t *free_bytes, size_t *total_bytes)
{
    return hipMemGetInfo(free_bytes, total_bytes) == hipSuccess ? 0 : 1;
}

int ccx_hip_free(void *p) { return (p == nullptr || hipFree(p) == hipSuccess) ? 0 : 1; }

int ccx_hip_memcpy_h2d(void *dst, const void *src, size_t bytes, void *stream)
{
    if (bytes == 0) return 0;
    if (hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, (hipStream_t)stream) != hipSuccess) return 1;
    return hipStreamSynchronize((hipStream_t)stream) == hipSuccess ? 0 : 1;
}

int ccx_hip_memcpy_d2h(void *dst, const void *src, size_t bytes, void *stream)
{
    if (bytes == 0) return 0;
    if (hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, (hipStream_t)stream) != hipSuccess) return 1;
    return hipStreamSynchronize((hipStream_t)stream) == hipSuccess ? 0 : 1;
}

int ccx_hip_memcpy_d2d(void *dst, const void *src, size_t bytes, void *stream)
{
    if (bytes == 0) return 0;
    return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, (hipStream_t)stream) == hipSuccess ? 0 : 1;
}

int ccx_hip_memcpy_h2d_queue(void *dst, const void *src, size_t bytes, void *stream)
{
    if (bytes == 0) return 0;
    return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, (hipStream_t)stream) == hipSuccess ? 0 : 1;
}

int ccx_hip_host_malloc(void **p, size_t bytes)
{
    *p = nullptr;
    if (hipHostMalloc(p, bytes, hipHostMallocDefault) == hipSuccess) return 0;
    *p = nullptr;
    (void)hipGetLastError();
    return 1;
}

int ccx_hip_host_free(void *p) { return (p == nullptr || hipHostFree(p) == hipSuccess) ? 0 : 1; }

int ccx_hip_sync(void *stream) { return hipStreamSynchronize((hipStream_t)stream) == hipSuccess ? 0 : 1; }

int ccx_hip_cu_count(int *n)
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 1;
    return hipDeviceGetAttribute(n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess ? 0 : 1;
}


// AX in both orientations from VVVO (layout V_FULL, V_PACKED or V_VE) and T2 of nx occupied indices
static int launch_pack_ax(int layout, const double *vvvo, const double *t2, double *axr, double *axc, int no, int nu,
                          int nup, int kp, int nx, hipStream_t s)
{
    const int nb = nup / TB, nkc = (kp + PK_K - 1) / PK_K;
    const long long grid = (long long)nx * nb * nb * nkc;
    if (grid > 0x7fffffffLL) return 3;
    if (layout == V_FULL) pack_ax_kernel<V_FULL><<<(unsigned)grid, 256, 0, s>>>(vvvo, t2, axr, axc, no, nu, nb, kp, nkc);
    else if (layout == V_PACKED) pack_ax_kernel<V_PACKED><<<(unsigned)grid, 256, 0, s>>>(vvvo, t2, axr, axc, no, nu, nb, kp, nkc);
    else pack_ax_kernel<V_VE><<<(unsigned)grid, 256, 0, s>>>(vvvo, t2, axr, axc, no, nu, nb, kp, nkc);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// The operand slabs, the padded VOE and (where their destinations are given) the small arrays of a
// problem, from the reference-layout arrays; vvvo_layout 0 or 1 as in ccx_load_device.
int ccx_hip_pack(int vvvo_layout, const double *vvvo, const double *t2, const double *vm, const double *voe,
                 const double *eh, const double *ep, const double *t1, double *axr, double *axc, double *bx,
                 double *voep, double *ehp, double *epp, double *t1p, int no, int nu, int nup, int kp, void *stream)
{
    hipStream_t s = (hipStream_t)stream;
    const int nb = nup / TB;
    const int rc = launch_pack_ax(vvvo_layout, vvvo, t2, axr, axc, no, nu, nup, kp, no, s);
    if (rc != 0) return rc;
    const long long ntile = (long long)no * no * nb * nb;
    RestArgs a = {t2, vm, voe, eh, ep, t1, bx, voep, ehp, epp, t1p, no, nu, nup, kp,
                  grid_for((long long)no * no * nb * kp * 16), (int)(ntile < 65536 ? ntile : 65536)};
    pack_rest_kernel<<<a.gbx + a.gvoe + 1, 256, 0, s>>>(a);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// The FP64 panels of one occupied index (both AX orientations) from its cube (layout 0: VE_x(d,p,q) =
// VVVO(d,q,p,x); 1: the packed columns of x) and t2_x = T2(:,:,:,x) (nu^2 no); axr_x / axc_x point at
// that index's panels.
int ccx_hip_pack_ax_one(int layout, const double *cube, const double *t2_x, double *axr_x, double *axc_x, int no,
                        int nu, int nup, int kp, void *stream)
{
    return launch_pack_ax(layout == 1 ? V_PACKED : V_VE, cube, t2_x, axr_x, axc_x, no, nu, nup, kp, 1, (hipStream_t)stream);
}

// BX panels and padded VOE blocks of n <= 6 ordered pairs (PairArgs)
int ccx_hip_pack_pairs(const struct ccx_pair_pack *p, int n, int no, int nu, int nup, int kp, void *stream)
{
    if (n < 1 || n > 6) return 3;
    const int nb = nup / TB;
    PairArgs a;
    for (int q = 0; q < n; ++q) a.p[q] = p[q];
    a.no = no; a.nu = nu; a.nup = nup; a.kp = kp;
    a.npb = grid_for((long long)nb * kp * 16);
    a.npv = p[0].voe ? (nb * nb < 65536 ? nb * nb : 65536) : 0;
    pack_pairs_kernel<<<n * (a.npb + a.npv), 256, 0, (hipStream_t)stream>>>(a);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// K padding of a form's slabs: FP32 48; split forms two K blocks of their MFMA (64 for bf16,
// 256 for fp8 e4m3); FP64 4
int ccx_hip_form_kpad(int form) { return form == 1 ? 48 : form == 3 ? 256 : form >= 2 ? 64 : 4; }

// form 0: FP64 slabs; 1: FP32 slabs in the FP32 sweep's order (K padded to kps, a multiple of
// 48); 2-4: split slices (split[] = axr_s, axc_s, bx_s and, for form 3, the exponent words
// axr_e, axc_e, bx_e; K padded to kps, W scaled by wscale)
int ccx_hip_triples(int form, const void *axr, const void *axc, const void *bx, const double *voep,
                    const double *eh, const double *ep, const int *tuples, const int *blocks, double *e_part,
                    double *v1_part, double *wout, unsigned int *counter, int no, int nu, int nup, int kp,
                    int ntup, int nblk, int grid, const void *const *split, int kps, double wscale, void *stream)
{
    static bool attr_set[5] = {false, false, false, false, false};
    const size_t lds_bytes = sizeof(double) * LDS_DOUBLES;
    if (form < 0 || form > 4) return 3;
    if (form >= 2 && (split == nullptr || kps % ccx_hip_form_kpad(form) != 0)) return 3;
    if (form == 1 && kps % 48 != 0) return 3;   // FP32 slabs: K padded to 48 (kps)
    const void *fns[5] = {(const void *)triples_kernel<double, 0>, (const void *)triples_kernel<float, 1>,
                          (const void *)triples_kernel<float, 2>, (const void *)triples_kernel<float, 3>,
                          (const void *)triples_kernel<float, 4>};
    if (!attr_set[form]) {
        if (hipFuncSetAttribute(fns[form], hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes) != hipSuccess)
            return 2;
        attr_set[form] = true;
    }
    const bool sp = form >= 2;
    TriplesArgs g;
    g.axr = axr; g.axc = axc; g.bx = bx; g.voe = voep; g.eh = eh; g.ep = ep; g.tuples = tuples;
    g.blocks = blocks; g.e_part = e_part; g.v1_part = v1_part; g.wout = wout; g.counter = counter;
    g.no = no; g.nu = nu; g.nup = nup; g.nb = nup / TB; g.kp = kp; g.ntup = ntup; g.nblk = nblk;
    g.nitems = (long long)ntup * nblk;
    g.axr_s = sp ? split[0] : nullptr;
    g.axc_s = sp ? split[1] : nullptr;
    g.bx_s = sp ? split[2] : nullptr;
    g.axr_e = form == 3 ? (const int *)split[3] : nullptr;
    g.axc_e = form == 3 ? (const int *)split[4] : nullptr;
    g.bx_e = form == 3 ? (const int *)split[5] : nullptr;
    g.kps = kps;
    g.wscale = sp ? wscale : 1.0;
    {
        const char *env = getenv("CCX_ITEM_ORDER");
        g.block_major = (env && env[0] == 't') ? 0 : 1;
    }
    if (g.nitems == 0) return 0;
    if (grid <= 0) grid = 256;
    if (grid > g.nitems) grid = (int)g.nitems;
    hipStream_t s = (hipStream_t)stream;
    zero_counter_kernel<<<1, 1, 0, s>>>(counter);
    switch (form) {
    case 0: triples_kernel<double, 0><<<grid, NTHR, lds_bytes, s>>>(g); break;
    case 1: triples_kernel<float, 1><<<grid, NTHR, lds_bytes, s>>>(g); break;
    case 2: triples_kernel<float, 2><<<grid, NTHR, lds_bytes, s>>>(g); break;
    case 3: triples_kernel<float, 3><<<grid, NTHR, lds_bytes, s>>>(g); break;
    default: triples_kernel<float, 4><<<grid, NTHR, lds_bytes, s>>>(g); break;
    }
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// Bytes per slab element of a split form's slices (BF16 x 3: 6, FP8 x 4: 4, BF16 x 4: 8); the FP8
// form adds one exponent word per 32 elements.
int ccx_hip_split_elem_bytes(int form) { return form == 2 ? 6 : form == 3 ? 4 : form == 4 ? 8 : 0; }

// Split slabs from the FP64 ones: power-of-two scales sigma_A >= max|AX|, sigma_B >= max|BX| (the
// fixed-point grid of the BF16 x 4 slabs; for every form they keep FP64 inputs of any range inside
// FP32's), then the slices of AX / sigma_A (both orientations) and BX / sigma_B; sl[] = axr_s, axc_s,
// bx_s, axr_e, axc_e, bx_e; *wscale = sigma_A sigma_B.
int ccx_hip_pack_split(int form, const double *axr, const double *axc, const double *bx, void *const *sl,
                       unsigned long long *dmax, int no, int nb, int kp, int kps, double *wscale, void *stream)
{
    if (form < 2 || form > 4 || kps % ccx_hip_form_kpad(form) != 0) return 3;
    hipStream_t s = (hipStream_t)stream;
    const long long n_ax = (long long)no * nb * nb * 256 * kp, n_bx = (long long)no * no * nb * 16 * kp;
    zero_counter_kernel<<<1, 1, 0, s>>>(reinterpret_cast<unsigned int *>(dmax));
    zero_counter_kernel<<<1, 1, 0, s>>>(reinterpret_cast<unsigned int *>(dmax) + 1);
    zero_counter_kernel<<<1, 1, 0, s>>>(reinterpret_cast<unsigned int *>(dmax) + 2);
    zero_counter_kernel<<<1, 1, 0, s>>>(reinterpret_cast<unsigned int *>(dmax) + 3);
    const int g_ax = grid_for(n_ax), g_bx = grid_for(n_bx);
    absmax_kernel<<<g_ax < 2048 ? g_ax : 2048, 256, 0, s>>>(axr, n_ax, dmax);
    absmax_kernel<<<g_bx < 2048 ? g_bx : 2048, 256, 0, s>>>(bx, n_bx, dmax + 1);
    unsigned long long h[2];
    if (hipMemcpyAsync(h, dmax, sizeof(h), hipMemcpyDeviceToHost, s) != hipSuccess || hipStreamSynchronize(s) != hipSuccess)
        return 1;
    double sc[2];
    for (int q = 0; q < 2; ++q) {
        double m;
        memcpy(&m, &h[q], sizeof(m));
        int e = 0;
        if (m > 0.0) frexp(m, &e);   // m < 2^e
        sc[q] = m > 0.0 ? ldexp(1.0, e) : 1.0;
    }
    if (form == 2) launch_pack_split<2>(axr, axc, bx, sl, no, nb, kp, kps, sc, s);
    else if (form == 3) launch_pack_split<3>(axr, axc, bx, sl, no, nb, kp, kps, sc, s);
    else launch_pack_split<4>(axr, axc, bx, sl, no, nb, kp, kps, sc, s);
    *wscale = sc[0] * sc[1];
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// Sums the work items' partials (the energy partials are overwritten): out = {etd, ets}, v1(nu,no).
int ccx_hip_finalize(double *e_part, const double *v1_part, const int *tuples, const double *t1, double *v1t,
                     double *v1, double *out, int no, int nu, int ntup, int nblk, void *stream)
{
    hipStream_t s = (hipStream_t)stream;
    const int nb = (nu + TB - 1) / TB;
    const long long nitems = (long long)ntup * nblk;
    long long chunk = (nitems + RE_CHUNKS - 1) / RE_CHUNKS;
    if (chunk < 1024) chunk = 1024;
    const int nchunk = (int)((nitems + chunk - 1) / chunk);
    if (ntup > 0) {
        reduce_partials_kernel<<<(unsigned)((long long)ntup * nb + nchunk), 256, 0, s>>>(v1_part, e_part, v1t, ntup, nblk,
                                                                                         nu, nb, nitems, chunk);
        reduce_v1_kernel<<<no * ((nu + 63) / 64), 256, 0, s>>>(v1t, tuples, v1, ntup, nu, no);
    } else {
        if (hipMemsetAsync(v1, 0, sizeof(double) * nu * no, s) != hipSuccess) return 1;
    }
    finalize_energy_kernel<<<1, 1024, 0, s>>>(e_part, nchunk, chunk, t1, v1, no, nu, out);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ccx_hip_t1wt3(const double *w, const double *voe6, double dijk, const double *ep, int nu, double *x3,
                  double *v1p, void *stream)
{
    if (nu < 1) return 0;
    t1wt3_kernel<<<nu, 256, 0, (hipStream_t)stream>>>(w, voe6, dijk, ep, nu, x3, v1p);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ccx_hip_lds_bytes(void) { return (int)(sizeof(double) * LDS_DOUBLES); }

int ccx_hip_pack_f32v(const double *axr, const double *axc, const double *bx, float *axr32, float *axc32,
                      float *bx32, int no, int nb, int kp, int kpf, void *stream)
{
    if (kpf % 48 != 0) return 3;
    hipStream_t s = (hipStream_t)stream;
    const long long nax = (long long)no * nb * nb * 256 * kpf, nbx = (long long)no * no * nb * 16 * kpf;
    pack_f32v_kernel<0><<<grid_for(nax), 256, 0, s>>>(axr, axr32, (long long)no * nb * nb, kp, kpf);
    pack_f32v_kernel<0><<<grid_for(nax), 256, 0, s>>>(axc, axc32, (long long)no * nb * nb, kp, kpf);
    pack_f32v_kernel<1><<<grid_for(nbx), 256, 0, s>>>(bx, bx32, (long long)no * no * nb, kp, kpf);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ccx_hip_zero_flag(unsigned int *d_flag, void *stream)
{
    zero_counter_kernel<<<1, 1, 0, (hipStream_t)stream>>>(d_flag);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// *nonfinite = 1 when any element of the arrays p[0..narr) (n[q] doubles each, at most 7 arrays) is NaN
// or infinite.  *d_flag is zero before the call; it is left non-zero when *nonfinite is.
int ccx_hip_nonfinite(const double *const *p, const size_t *n, int narr, unsigned int *d_flag, int *nonfinite,
                      void *stream)
{
    hipStream_t s = (hipStream_t)stream;
    if (narr > 7) return 3;
    ScanArgs a;
    long long most = 1;
    a.narr = narr;
    for (int q = 0; q < narr; ++q) {
        a.p[q] = p[q];
        a.n[q] = (long long)n[q];
        if (a.n[q] > most) most = a.n[q];
    }
    const int grid = grid_for((most + 3) / 4);
    nonfinite_kernel<<<grid < 4096 ? grid : 4096, 256, 0, s>>>(a, d_flag);
    unsigned int h = 0;
    if (hipGetLastError() != hipSuccess || hipMemcpyAsync(&h, d_flag, sizeof(h), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
        return 1;
    *nonfinite = h != 0;
    return 0;
}

int ccx_hip_event_create(void **ev)
{
    hipEvent_t e;
    if (hipEventCreate(&e) != hipSuccess) return 1;
    *ev = (void *)e;
    return 0;
}

int ccx_hip_event_destroy(void *ev) { return hipEventDestroy((hipEvent_t)ev) == hipSuccess ? 0 : 1; }

int ccx_hip_event_record(void *ev, void *stream)
{
    return hipEventRecord((hipEvent_t)ev, (hipStream_t)stream) == hipSuccess ? 0 : 1;
}

int ccx_hip_event_ms(void *start, void *stop, float *ms)
{
    if (hipEventSynchronize((hipEvent_t)stop) != hipSuccess) return 1;
    return hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop) == hipSuccess ? 0 : 1;
}

}  // extern "C"
