// Virtual-triple view of the (T) intermediate: for a fixed virtual triple (a,b,c) the
// occupied cube V3(i,j,k) = W_ijk(a,b,c), the quantity the triples-abc prototype
// abc_tuple_formv3 assembles from 12 GEMMs of shape no^2 x nu x no and no x no^2 x no
// (src/triples-abc/abc_tuple.f90:1-81), and E[T] re-summed over virtual triples.
//
// W comes from the closed form on the FP64 operand slabs the context already holds
// (AX[x](a,b,K) = VVVO(K,b,a,x) for K < nu, T2(a,b,K-nu,x) after; BX[y,z](c,K) = T2(c,K,y,z),
// then -VM(K-nu,c,z,y)):
//   W_ijk(a,b,c) = sum over the 6 simultaneous permutations s of the pairs (i,a),(j,b),(k,c)
//                  of sum_K AX[i'](a',b',K) BX[j',k'](c',K).
// This path is a cross-check and a surface for virtual-triple callers, not the hot path.  One
// triple alone, and lists of them where there is no room for copies of the slabs or nothing to win
// from them: FP64 FMA on cached slab reads (w_abc_kernel).
// The sum over all triples: each term s is the GEMM
//   G_s[x][(y,z)] = sum_K AX[x](v_s0, v_s1, K) BX[y,z](v_s2, K),   no x no^2 x (nu+no),
// on the FP64 matrix cores, from copies of the slabs with x and (y,z) innermost (w_abc_mfma_kernel).

#include <hip/hip_runtime.h>

namespace {

constexpr int ABC_TB = 16;        // virtual block edge of the slab layouts
constexpr int ABC_THR = 256;
constexpr long long ABC_LANES = 24576;   // elements from which a lane each is the faster (ccx_hip_w_abc)
__device__ constexpr int ABC_PERM[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};

// V3 of triple t = (abc[4t], abc[4t+1], abc[4t+2]) into w[t * no^3 ...], column-major
// (i fastest).  V3(i,i,i) is set to 0, as zerot3 does at the end of abc_tuple_formv3
// (src/triples-abc/abc_tuple.f90:77); E[T] does not depend on those elements.
// LPE lanes per element along K.  64 where the elements alone do not fill the chip: a single triple has
// only no^3 of them, and with one lane each its time was the 6 (nu + no) dependent slab reads of
// a lane (142 us at no=6, nu=64).  One for long lists: neighbouring lanes then read neighbouring x at
// one K, where a wave along K fetches a line per lane and element.
template <int LPE>
__global__ void __launch_bounds__(ABC_THR) w_abc_kernel(const double *__restrict__ axr, const double *__restrict__ bx,
                                                        const int *__restrict__ trip, int ntrip, int no, int nu,
                                                        int nb, int kp, double *__restrict__ w)
{
    const int lane = threadIdx.x % LPE;
    const int no3 = no * no * no;
    const long long total = (long long)ntrip * no3, step = (long long)gridDim.x * (ABC_THR / LPE);
    const int kn = nu + no;
    for (long long id = blockIdx.x * (long long)(ABC_THR / LPE) + threadIdx.x / LPE; id < total; id += step) {
        const int t = (int)(id / no3), e = (int)(id % no3);
        const int v[3] = {trip[4 * t], trip[4 * t + 1], trip[4 * t + 2]};
        const int o[3] = {e % no, (e / no) % no, e / (no * no)};
        double acc = 0.0;
        if (!(o[0] == o[1] && o[1] == o[2])) {
#pragma unroll
            for (int s = 0; s < 6; ++s) {
                const int p0 = ABC_PERM[s][0], p1 = ABC_PERM[s][1], p2 = ABC_PERM[s][2];
                const int x = o[p0], y = o[p1], z = o[p2];
                const int av = v[p0], bv = v[p1], cv = v[p2];
                // row layout of AX (axr): panel (x, a-block, b-block), then
                // [alpha/2][K/4][lane = (K%4)*16 + beta][alpha%2]
                const int al = av % ABC_TB, be = bv % ABC_TB;
                const double *ap = axr + (((long long)x * nb + av / ABC_TB) * nb + bv / ABC_TB) * (256LL * kp)
                                   + (long long)(al >> 1) * (kp / 4) * 128 + be * 2 + (al & 1);
                // BX: [y][z][c-block][K][gamma]
                const double *bp = bx + (((long long)y * no + z) * nb + cv / ABC_TB) * ((long long)kp * 16) + cv % ABC_TB;
                double sum = 0.0;
                for (int K = lane; K < kn; K += LPE) sum = fma(ap[(K >> 2) * 128 + (K & 3) * 32], bp[(long long)K * 16], sum);
                acc += sum;
            }
#pragma unroll
            for (int d = LPE / 2; d >= 1; d >>= 1) acc += __shfl_xor(acc, d, 64);
        }
        if (lane == 0) w[id] = acc;
    }
}

typedef double d4 __attribute__((ext_vector_type(4)));

// Copies of the slabs in the operand order of v_mfma_f64_16x16x4_f64 with the occupied indices as the
// tile axis, zero past no and no^2:
//   axt [a][b][x tile][K/4][lane]   x = 16 tile + (lane & 15),        K = 4 (K/4) + (lane >> 4)
//   bxt [c][pair tile][K/4][lane]   y no + z = 16 tile + (lane & 15)
// Source element order: neighbouring threads read neighbouring slab elements.
__global__ void abc_pack_a_kernel(const double *__restrict__ axr, double *__restrict__ axt, int no, int nu, int nb,
                                  int kp, int mt)
{
    const long long per_panel = 256LL * kp, total = (long long)mt * 16 * nb * nb * per_panel;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total; i += (long long)gridDim.x * blockDim.x) {
        const int r = (int)(i % per_panel);
        const long long pnl = i / per_panel;
        const int lane = (r >> 1) & 63, rr = r >> 7, kb = rr % (kp / 4);
        const int q = (int)(pnl % nb), pb = (int)(pnl / nb % nb), x = (int)(pnl / ((long long)nb * nb));
        const int a = pb * ABC_TB + (rr / (kp / 4)) * 2 + (r & 1), b = q * ABC_TB + (lane & 15);
        if (a >= nu || b >= nu) continue;
        axt[((((long long)a * nu + b) * mt + (x >> 4)) * (kp / 4) + kb) * 64 + (lane >> 4) * 16 + (x & 15)] =
            x < no ? axr[i] : 0.0;
    }
}

__global__ void abc_pack_b_kernel(const double *__restrict__ bx, double *__restrict__ bxt, int no, int nu, int nb,
                                  int kp, int nt)
{
    const long long per_pair = (long long)nb * kp * 16, total = (long long)nt * 16 * per_pair;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total; i += (long long)gridDim.x * blockDim.x) {
        const int r = (int)(i % per_pair);
        const int n = (int)(i / per_pair), gl = r & 15, K = (r >> 4) % kp, c = (r >> 4) / kp * ABC_TB + gl;
        if (c >= nu) continue;
        bxt[(((long long)c * nt + (n >> 4)) * (kp / 4) + (K >> 2)) * 64 + (K & 3) * 16 + (n & 15)] =
            n < no * no ? bx[i] : 0.0;
    }
}

// The cubes of w_abc_kernel for a list of triples, WPT waves per triple (one while a triple has at
// most four pair tiles, so that a small no does not leave waves idle), NC pair tiles per wave and
// sweep.  The six terms are added into the triple's cube in order by the waves that own it, with a
// fence between terms; each element is touched once per term, so the sum is deterministic.  Bound by
// the matrix cores' padding (no of 16 rows, no^2 of 16 nt columns) and the operand loads, 1 + NC
// fragments per NC MFMAs.
template <int WPT, int NC>
__global__ void __launch_bounds__(ABC_THR) w_abc_mfma_kernel(const double *__restrict__ axt,
                                                             const double *__restrict__ bxt,
                                                             const int *__restrict__ trip, int ntrip, int no, int nu,
                                                             int kp, int mt, int nt, double *__restrict__ w)
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int t = WPT == 1 ? (int)blockIdx.x * (ABC_THR / 64) + wave : (int)blockIdx.x;
    if (t >= ntrip) return;   // WPT 1: no barrier below; otherwise the whole work group
    const int sub = WPT == 1 ? 0 : wave;
    const int v[3] = {__builtin_amdgcn_readfirstlane(trip[4 * t]), __builtin_amdgcn_readfirstlane(trip[4 * t + 1]),
                      __builtin_amdgcn_readfirstlane(trip[4 * t + 2])};
    const long long tile = (long long)kp * 16;
    const int nk = kp / 4, no2 = no * no;
    double *wt = w + (long long)t * no2 * no;
#pragma unroll 1
    for (int s = 0; s < 6; ++s) {
        const int p0 = ABC_PERM[s][0], p1 = ABC_PERM[s][1], p2 = ABC_PERM[s][2];
        const int va = p0 == 0 ? v[0] : p0 == 1 ? v[1] : v[2];
        const int vb = p1 == 0 ? v[0] : p1 == 1 ? v[1] : v[2];
        const int vc = p2 == 0 ? v[0] : p2 == 1 ? v[1] : v[2];
        // cube strides of x, y and z
        const int sx = p0 == 0 ? 1 : p0 == 1 ? no : no2, sy = p1 == 0 ? 1 : p1 == 1 ? no : no2,
                  sz = p2 == 0 ? 1 : p2 == 1 ? no : no2;
        const double *ab = axt + ((long long)va * nu + vb) * mt * tile + lane;
        const double *bb = bxt + (long long)vc * nt * tile + lane;
        for (int m = 0; m < mt; ++m)
            for (int n0 = sub * NC; n0 < nt; n0 += WPT * NC) {
                const double *pa = ab + m * tile;
                const double *pb[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) pb[c] = bb + (n0 + c < nt ? n0 + c : nt - 1) * tile;
                d4 acc[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) acc[c] = d4{0, 0, 0, 0};
                // four K steps per round: their loads are issued together (the compiler does not
                // unroll a loop with MFMAs of itself)
                int k = 0;
                for (; k + 4 <= nk; k += 4) {
                    double a[4], b[4][NC];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        a[j] = pa[(k + j) * 64];
#pragma unroll
                        for (int c = 0; c < NC; ++c) b[j][c] = pb[c][(k + j) * 64];
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int c = 0; c < NC; ++c) acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[j], b[j][c], acc[c], 0, 0, 0);
                }
                for (; k < nk; ++k) {
                    const double a = pa[k * 64];
#pragma unroll
                    for (int c = 0; c < NC; ++c) acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, pb[c][k * 64], acc[c], 0, 0, 0);
                }
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    const int n = (n0 + c) * 16 + (lane & 15), y = n / no, z = n % no;
                    if (n0 + c >= nt || n >= no2) continue;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int x = m * 16 + (lane >> 4) + 4 * r;   // accumulator row of the FP64 MFMA
                        if (x >= no) continue;
                        double *o = wt + x * sx + y * sy + z * sz;
                        if (s == 5 && x == y && y == z) *o = 0.0;
                        else if (s == 0) *o = acc[c][r];
                        else *o += acc[c][r];
                    }
                }
            }
        __threadfence_block();
        if constexpr (WPT > 1) __syncthreads();
    }
}

// X_abc = sum_ijk V(ijk) [8 V(ijk) - 4 (V(ikj) + V(kji) + V(jik)) + 2 (V(kij) + V(jki))] / D
// with D = e_i + e_j + e_k - e_a - e_b - e_c, times the triple's weight (1 for a > b > c,
// 1/2 for a > b = c and a = b > c).  It is the ijk-driven t1wt3_ijk / T3SQUA sum
// (src/triples-ijk/t1wt3.f90:53-69, src/triples-ijk/t3squa_acc.f:18-56) with the roles of
// the occupied and the virtual indices exchanged through the pair-permutation symmetry of W.
// Fixed-order reduction: each lane sums its elements in order, then a tree over the group.
__global__ void __launch_bounds__(ABC_THR) x_abc_kernel(const double *__restrict__ w, const int *__restrict__ trip,
                                                        int ntrip, int no, const double *__restrict__ eh,
                                                        const double *__restrict__ ep, double *__restrict__ x)
{
    __shared__ double part[ABC_THR];
    const int t = blockIdx.x;
    if (t >= ntrip) return;
    const double eabc = ep[trip[4 * t]] + ep[trip[4 * t + 1]] + ep[trip[4 * t + 2]];
    const double wt = trip[4 * t + 3] == 1 ? 1.0 : 0.5;
    const int no3 = no * no * no;
    const double *V = w + (long long)t * no3;
    double s = 0.0;
    for (int e = threadIdx.x; e < no3; e += ABC_THR) {
        const int i = e % no, j = (e / no) % no, k = e / (no * no);
        auto at = [&](int p, int q, int r) { return V[p + no * (q + no * r)]; };
        const double vijk = V[e];
        const double br = 8.0 * vijk - 4.0 * (at(i, k, j) + at(k, j, i) + at(j, i, k)) + 2.0 * (at(k, i, j) + at(j, k, i));
        s += vijk * br / (eh[i] + eh[j] + eh[k] - eabc);
    }
    part[threadIdx.x] = s;
    __syncthreads();
    for (int h = ABC_THR / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) part[threadIdx.x] += part[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) x[t] = part[0] * wt;
}

// Tiles of 16 occupied indices and of 16 ordered occupied pairs
int abc_mt(int no) { return (no + 15) / 16; }
int abc_nt(int no) { return (no * no + 15) / 16; }

template <int WPT>
void launch_w_abc(int nc, int grid, const double *axt, const double *bxt, const int *trip, int ntrip, int no,
                         int nu, int kp, double *w, hipStream_t s)
{
    const int mt = abc_mt(no), nt = abc_nt(no);
    switch (nc) {
    case 1: w_abc_mfma_kernel<WPT, 1><<<grid, ABC_THR, 0, s>>>(axt, bxt, trip, ntrip, no, nu, kp, mt, nt, w); break;
    case 2: w_abc_mfma_kernel<WPT, 2><<<grid, ABC_THR, 0, s>>>(axt, bxt, trip, ntrip, no, nu, kp, mt, nt, w); break;
    case 3: w_abc_mfma_kernel<WPT, 3><<<grid, ABC_THR, 0, s>>>(axt, bxt, trip, ntrip, no, nu, kp, mt, nt, w); break;
    default: w_abc_mfma_kernel<WPT, 4><<<grid, ABC_THR, 0, s>>>(axt, bxt, trip, ntrip, no, nu, kp, mt, nt, w); break;
    }
}

}  // namespace

extern "C" {

int ccx_hip_w_abc(const void *axr, const void *bx, const int *trip, int ntrip, int no, int nu, int nb, int kp,
                  double *w, void *stream)
{
    if (ntrip <= 0) return 0;
    if (kp % 4 != 0 || kp < nu + no) return 3;
    // A lane per element once those lanes fill the chip: 16384 elements (no=16, nu=40) took 61 us with a lane
    // and 48 us with a wave each, 27648 (no=3, nu=120) 112 and 150 us, 16.8 M (no=16) 13.5 and 51.9 ms.
    const long long total = (long long)ntrip * no * no * no;
    const int lpe = total >= ABC_LANES ? 1 : 64;
    const long long groups = (total * lpe + ABC_THR - 1) / ABC_THR;
    const int grid = (int)(groups < 65536 ? groups : 65536);
    const double *a = (const double *)axr, *b = (const double *)bx;
    if (lpe == 1) w_abc_kernel<1><<<grid, ABC_THR, 0, (hipStream_t)stream>>>(a, b, trip, ntrip, no, nu, nb, kp, w);
    else w_abc_kernel<64><<<grid, ABC_THR, 0, (hipStream_t)stream>>>(a, b, trip, ntrip, no, nu, nb, kp, w);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// sizes (in doubles) of the packed copies that ccx_hip_abc_pack fills
size_t ccx_hip_abc_a_doubles(int no, int nu, int kp) { return (size_t)nu * nu * abc_mt(no) * 16 * kp; }
size_t ccx_hip_abc_b_doubles(int no, int nu, int kp) { return (size_t)nu * abc_nt(no) * 16 * kp; }

int ccx_hip_abc_pack(const void *axr, const void *bx, double *axt, double *bxt, int no, int nu, int nb, int kp,
                     void *stream)
{
    if (kp % 4 != 0 || kp < nu + no) return 3;
    hipStream_t s = (hipStream_t)stream;
    const long long na = (long long)abc_mt(no) * 16 * nb * nb * 256 * kp, n2 = (long long)abc_nt(no) * 16 * nb * kp * 16;
    const long long ga = (na + 255) / 256, g2 = (n2 + 255) / 256;
    abc_pack_a_kernel<<<(int)(ga < 65536 ? ga : 65536), 256, 0, s>>>((const double *)axr, axt, no, nu, nb, kp, abc_mt(no));
    abc_pack_b_kernel<<<(int)(g2 < 65536 ? g2 : 65536), 256, 0, s>>>((const double *)bx, bxt, no, nu, nb, kp, abc_nt(no));
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

// ccx_hip_w_abc from the packed copies, for lists of triples.  Up to four pair tiles (no <= 8) a
// wave takes a whole triple; above, the four waves of a work group share one, with the tile count
// per wave that leaves the fewest tile slots empty.
int ccx_hip_w_abc_packed(const double *axt, const double *bxt, const int *trip, int ntrip, int no, int nu, int kp,
                         double *w, void *stream)
{
    if (ntrip <= 0) return 0;
    const int nt = abc_nt(no), waves = ABC_THR / 64;
    hipStream_t s = (hipStream_t)stream;
    if (nt <= 4) {
        launch_w_abc<1>(nt, (ntrip + waves - 1) / waves, axt, bxt, trip, ntrip, no, nu, kp, w, s);
    } else {
        int best = 4, slots = 1 << 30;
        for (int nc = 4; nc >= 1; --nc) {
            const int used = (nt + waves * nc - 1) / (waves * nc) * waves * nc;
            if (used < slots) { slots = used; best = nc; }
        }
        launch_w_abc<ABC_THR / 64>(best, ntrip, axt, bxt, trip, ntrip, no, nu, kp, w, s);
    }
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

int ccx_hip_x_abc(const double *w, const int *trip, int ntrip, int no, const double *eh, const double *ep,
                  double *x, void *stream)
{
    if (ntrip <= 0) return 0;
    x_abc_kernel<<<ntrip, ABC_THR, 0, (hipStream_t)stream>>>(w, trip, ntrip, no, eh, ep, x);
    return hipGetLastError() == hipSuccess ? 0 : 1;
}

}  // extern "C"
