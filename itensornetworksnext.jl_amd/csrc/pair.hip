// pair.hip -- BP messages of a vertex from two pair environments, on FP64 (or FP32) MFMA.
//
// The ports of a vertex are split into two pairs; with n = (i, j) running over the two bond
// indices of a pair, the site tensor of each physical slice is an n0 x n1 matrix A_s.  With
// M0 = m_0 (x) m_1 and M1 = m_2 (x) m_3 (Kronecker products of the incoming messages, n x n),
//   R1[n1, n1'] = sum_s sum_n0' (M0^T A_s)[n0', n1] conj(A_s)[n0', n1']
//   R0[n0, n0'] = sum_s sum_n1' (A_s M1)[n0, n1'] conj(A_s)[n0', n1']
// are the vertex's environments of the two pairs, and the message out of a port is its pair's
// environment with the partner port's message absorbed,
//   out_0[a, a'] = sum_bb' R0[(a b), (a' b')] m_1[b, b'],
// normalised by its sum (src/beliefpropagation/beliefpropagation.jl:242-257).
//
// Why this split: everything but the last step is a chain of matrix products, which runs on
// 16x16x4 MFMA without moving a result.  Lane l of an MFMA result holds column l % 16 of four
// rows, which is the B operand of a product that contracts those rows; so E = M^T X goes
// straight into R^T += conj(A)^T E from registers, and the only LDS traffic is the operands'.
// Sides that are no multiple of 16 are padded with zeros in LDS only (the site tensors are
// read unpadded).  Per vertex of degree 4 the two products take 8 d D^6 FLOP against 24 d D^5
// for single mode products and opens: more FLOP above D = 3, but 4 barriers and no strided
// pass per product.
//
// Work split: wave (h, J, g) takes the 16 columns J of the other pair, contracts pair h with
// them for every slice of its share g, and holds the 16-column block of the environment (at
// most four 16x16 tiles) in registers.  The slices are staged in LDS `chunk` at a time.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "pair.h"

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

template <int TY>
struct PairTy;
template <>
struct PairTy<PAIR_F64> {
    using E = double;
    using V = v4d;
    static constexpr bool CX = false;
    static __device__ __forceinline__ V mma(E a, E b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // row of the 16x16 result in register r of lane block lk
    static __device__ __forceinline__ int row(int lk, int r) { return lk + 4 * r; }
};
template <>
struct PairTy<PAIR_C128> : PairTy<PAIR_F64> {
    static constexpr bool CX = true;
};
template <>
struct PairTy<PAIR_F32> {
    using E = float;
    using V = v4f;
    static constexpr bool CX = false;
    static __device__ __forceinline__ V mma(E a, E b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
};

__host__ __device__ inline int pair_pad(int n) { return (n + 15) & ~15; }

// LDS elements per plane (complex: two planes): staged slices, Kronecker messages or
// environments (they share the space), incoming messages.
__host__ __device__ inline int pair_slice_elems(int n0, int n1) {
    // an odd row pitch: both the rows and the columns of a slice are read 16 at a time
    return pair_pad(n0) * (pair_pad(n1) + 1);
}

// floor(i / n) for 0 <= i < 2^22, 1 <= n
__device__ __forceinline__ int fdiv(int i, float rn) { return (int)(((float)i + 0.5f) * rn); }

// NT: tiles of the largest pair side this instance handles.
template <int TY, int NT>
__global__ __launch_bounds__(64 * PAIR_MAXWAVES) void k_pair(
    const PairRec *__restrict__ recs, const int *__restrict__ items,
    const typename PairTy<TY>::E *__restrict__ sites, const typename PairTy<TY>::E *mold,
    typename PairTy<TY>::E *mnew, NetCtl ctl, double *__restrict__ res_fid,
    double *__restrict__ res_abs, SweepFold fold, int chunk, int split, int slice_elems,
    int env_elems, double *__restrict__ zv) {
    using P = PairTy<TY>;
    using E = typename P::E;
    using V = typename P::V;
    constexpr bool CX = P::CX;
    constexpr int PL = CX ? 2 : 1;  // planes; global elements are interleaved (re, im)
    extern __shared__ __align__(16) char smem[];
    __shared__ double fold_m[PAIR_MAXWAVES];
    E *Al = reinterpret_cast<E *>(smem);                  // [plane][chunk][slice_elems]
    E *Ml = Al + (size_t)PL * chunk * slice_elems;        // [plane][env_elems]
    E *ml = Ml + (size_t)PL * env_elems;                  // [position][plane][64]
    const int plA = chunk * slice_elems;

    const int item = blockIdx.x;
    const int ri = items ? items[item] >> 2 : item;
    // positions to update; the vertex scalar comes from position 0's unnormalised message
    const int mask = zv ? 1 : items ? 1 << (items[item] & 3) : 15;
    const PairRec &rec = recs[ri];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nthr = blockDim.x;
    const int W = nthr >> 6;
    const int net = rec.net;

    if (vx_fold_begin(ctl, fold, net, item)) {
        for (int p = 0; p < 4; ++p) {
            const int q = rec.slot[p];
            if (q < 0 || !((mask >> p) & 1)) continue;
            const int len = rec.dim[p] * rec.dim[p] * PL;
            const long long o = rec.out[p] * PL;
            for (int i = tid; i < len; i += nthr) mnew[o + i] = mold[o + i];
            if (tid == 0) {
                res_fid[q] = 0.0;
                res_abs[q] = 0.0;
            }
        }
        return;
    }

    const int n0 = rec.n[0], n1 = rec.n[1], d = rec.d;
    const int N0 = pair_pad(n0), N1 = pair_pad(n1), P1 = N1 + 1;
    const int SL = N0 * P1;
    const bool need[2] = {(mask & 12) != 0 && rec.slot[2] >= 0, (mask & 3) != 0};  // half h

    // ---- incoming messages (one position per wave) and the first slices, zero-padded; every
    // load of a batch is issued before the first LDS store waits for it
    const E *A = sites + rec.site * PL;
    const float rP = 1.0f / (float)P1, rN = 1.0f / (float)N0;
    constexpr int B = CX ? 4 : 8;
    auto stage = [&](int s0, int cnt) {
        const int total = cnt * SL;
        for (int i0 = tid; i0 < total; i0 += B * nthr) {
            E v[B], vi[CX ? B : 1];
#pragma unroll
            for (int k = 0; k < B; ++k) {
                const int i = i0 + k * nthr;
                const int row = fdiv(i, rP), c = i - row * P1;
                const int s = fdiv(row, rN), r = row - s * N0;
                const bool in = i < total && r < n0 && c < n1;
                const long long g = in ? ((long long)(s0 + s) * n0 + r) * n1 + c : 0;
                if constexpr (CX) {
                    const double2 z = reinterpret_cast<const double2 *>(A)[g];
                    v[k] = in ? z.x : E(0);
                    vi[k] = in ? z.y : E(0);
                } else {
                    const E z = A[g];
                    v[k] = in ? z : E(0);
                }
            }
#pragma unroll
            for (int k = 0; k < B; ++k) {
                const int i = i0 + k * nthr;
                if (i < total) {
                    Al[i] = v[k];
                    if constexpr (CX) Al[plA + i] = vi[k];
                }
            }
        }
    };
    for (int p = w; p < 4; p += W) {
        const int DD = rec.dim[p] * rec.dim[p];
        if (lane >= DD) continue;
        const bool have = rec.slot[p] >= 0;
        if constexpr (CX) {
            ml[(p * 2) * 64 + lane] = have ? mold[(rec.in[p] + lane) * 2] : E(1);
            ml[(p * 2 + 1) * 64 + lane] = have ? mold[(rec.in[p] + lane) * 2 + 1] : E(0);
        } else {
            ml[p * 64 + lane] = have ? mold[rec.in[p] + lane] : E(1);
        }
    }
    stage(0, min(chunk, d));
    __syncthreads();
    // ---- Kronecker products M_h[(a b)][(a' b')] = m_a[a][a'] m_b[b][b'], zero-padded
    for (int h = 0; h < 2; ++h) {
        const int n = h ? n1 : n0, N = h ? N1 : N0, Db = rec.dim[2 * h + 1], Da = rec.dim[2 * h];
        E *M = Ml + (h ? N0 * N0 : 0);
        const E *ma = ml + (2 * h) * PL * 64, *mb = ml + (2 * h + 1) * PL * 64;
        const int rows = nthr / N;  // rows of M per pass
        const int col = tid % N, r0 = tid / N;
        if (r0 >= rows) continue;
        const float rb = 1.0f / (float)Db;
        const int a2 = fdiv(col, rb), b2 = col - a2 * Db;
        for (int k = r0; k < N; k += rows) {
            const int a = fdiv(k, rb), b = k - a * Db;
            const bool in = k < n && col < n;
            if constexpr (CX) {
                E re = E(0), im = E(0);
                if (in) {
                    const E xr = ma[a * Da + a2], xi = ma[64 + a * Da + a2];
                    const E yr = mb[b * Db + b2], yi = mb[64 + b * Db + b2];
                    re = xr * yr - xi * yi;
                    im = xr * yi + xi * yr;
                }
                M[k * N + col] = re;
                M[env_elems + k * N + col] = im;
            } else {
                M[k * N + col] = in ? ma[a * Da + a2] * mb[b * Db + b2] : E(0);
            }
        }
    }
    __syncthreads();

    // ---- environments: this wave's (half, columns, slice share)
    const int lk = lane >> 4, li = lane & 15;
    const int t0 = N0 >> 4, t1 = N1 >> 4;
    const int per = NT * split;          // waves per half
    const int h = w / per, J = (w % per) / split, sg = w % split;
    const int nI = h ? t1 : t0, nJ = h ? t0 : t1;  // tiles of the contracted / the other pair
    const int nh = h ? n1 : n0;
    const bool work = h < 2 && need[h & 1] && J < nJ;
    V R[NT], Ri[CX ? NT : 1];
#pragma unroll
    for (int j = 0; j < NT; ++j) R[j] = V{0, 0, 0, 0};
    if constexpr (CX) {
#pragma unroll
        for (int j = 0; j < NT; ++j) Ri[j] = V{0, 0, 0, 0};
    }
    const int sk = h ? 1 : P1, sj = h ? P1 : 1;  // strides of the contracted / the other index
    const E *M = Ml + (h ? N0 * N0 : 0);
    const int Nh = h ? N1 : N0;
    for (int s0 = 0; s0 < d; s0 += chunk) {
        if (s0) {
            __syncthreads();
            stage(s0, min(chunk, d - s0));
            __syncthreads();
        }
        if (!work) continue;
        const int cnt = min(chunk, d - s0);
        for (int s = sg; s < cnt; s += split) {
            const E *As = Al + s * SL + li * sj;
            E X[4 * NT], Xi[CX ? 4 * NT : 1];
#pragma unroll
            for (int t = 0; t < 4 * NT; ++t)
                if (4 * t < nh) {
                    const int o = (4 * t + lk) * sk + 16 * J * sj;
                    X[t] = As[o];
                    if constexpr (CX) Xi[t] = As[plA + o];
                }
#pragma unroll
            for (int I = 0; I < NT; ++I) {
                if (I >= nI) break;
                V C = V{0, 0, 0, 0}, Ci = V{0, 0, 0, 0};
#pragma unroll
                for (int t = 0; t < 4 * NT; ++t)
                    if (4 * t < nh) {
                        const int o = (4 * t + lk) * Nh + 16 * I + li;
                        if constexpr (CX) {
                            const E mr = M[o], mi = M[env_elems + o];
                            C = P::mma(mr, X[t], C);
                            C = P::mma(-mi, Xi[t], C);
                            Ci = P::mma(mr, Xi[t], Ci);
                            Ci = P::mma(mi, X[t], Ci);
                        } else {
                            C = P::mma(M[o], X[t], C);
                        }
                    }
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    if (j >= nJ) break;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int o = (16 * I + P::row(lk, r)) * sk + 16 * j * sj;
                        const E a = As[o];
                        if constexpr (CX) {
                            const E ai = As[plA + o];
                            R[j] = P::mma(a, C[r], R[j]);
                            R[j] = P::mma(ai, Ci[r], R[j]);
                            Ri[j] = P::mma(a, Ci[r], Ri[j]);
                            Ri[j] = P::mma(-ai, C[r], Ri[j]);
                        } else {
                            R[j] = P::mma(a, C[r], R[j]);
                        }
                    }
                }
            }
        }
    }
    __syncthreads();  // every wave has read M: its space takes the environments
    // R^T of the other pair: [share][pair][n'][n]
    const int No = h ? N0 : N1;
    const int eshare = N0 * N0 + N1 * N1;
    if (work) {
        E *Ro = Ml + sg * eshare + (h ? 0 : N0 * N0);
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            if (j >= nJ) break;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int o = (16 * j + P::row(lk, r)) * No + 16 * J + li;
                Ro[o] = R[j][r];
                if constexpr (CX) Ro[env_elems + o] = Ri[j][r];
            }
        }
    }
    __syncthreads();

    // ---- messages: wave w takes positions w, w + W, ...
    double fm = 0.0;
    const bool fcrit = fold.acc && fold.rp->crit != 0;
    for (int p = w; p < 4; p += W) {
        const int q = rec.slot[p];
        if (q < 0 || !((mask >> p) & 1)) continue;
        const int o = p >> 1, D = rec.dim[p], Dp = rec.dim[p ^ 1], DD = D * D;
        const int sa = (p & 1) ? 1 : Dp, sb = (p & 1) ? D : 1;
        const int N = o ? N1 : N0;
        const E *mp = ml + (p ^ 1) * PL * 64;
        const E *Ro = Ml + (o ? N0 * N0 : 0);
        int G = 1;
        while (2 * G * DD <= 64) G *= 2;  // lanes per entry, lane = g * DD + entry
        const int g = lane / DD, e = lane - g * DD, a = e / D, a2 = e - a * D;
        E x = E(0), xi = E(0);
        if (g < G) {
            // lane g takes rows b = g, g + G, ... of the partner message; the eight columns
            // are read at once (clamped, the absent ones dropped)
            for (int b = g; b < Dp; b += G) {
                E v[8], m[8], vi[CX ? 8 : 1], mi[CX ? 8 : 1];
#pragma unroll
                for (int b2 = 0; b2 < 8; ++b2) {
                    const int bc = min(b2, Dp - 1);
                    const int at = (a2 * sa + bc * sb) * N + a * sa + b * sb;
                    v[b2] = Ro[at];
                    m[b2] = mp[b * Dp + bc];
                    if (split > 1) v[b2] += Ro[eshare + at];
                    if constexpr (CX) {
                        vi[b2] = Ro[env_elems + at];
                        mi[b2] = mp[64 + b * Dp + bc];
                        if (split > 1) vi[b2] += Ro[env_elems + eshare + at];
                    }
                }
#pragma unroll
                for (int b2 = 0; b2 < 8; ++b2) {
                    if (b2 >= Dp) break;
                    if constexpr (CX) {
                        x += v[b2] * m[b2] - vi[b2] * mi[b2];
                        xi += v[b2] * mi[b2] + vi[b2] * m[b2];
                    } else {
                        x += v[b2] * m[b2];
                    }
                }
            }
        }
        for (int k = G >> 1; k > 0; k >>= 1) {
            x += __shfl_down(x, k * DD, 64);
            if constexpr (CX) xi += __shfl_down(xi, k * DD, 64);
        }
        const bool real = lane < DD;
        if (zv) {
            if constexpr (CX) {
                const E mr = ml[lane & 63], mi = ml[64 + (lane & 63)];
                const double zr = wave_sum_v(real ? x * mr - xi * mi : 0.0);
                const double zi = wave_sum_v(real ? x * mi + xi * mr : 0.0);
                if (lane == 0) {
                    zv[2 * rec.vertex] = zr;
                    zv[2 * rec.vertex + 1] = zi;
                }
            } else {
                const double z = wave_sum_v(real ? (double)x * (double)ml[lane] : 0.0);
                if (lane == 0) zv[rec.vertex] = z;
            }
            continue;
        }
        const long long mo = rec.out[p] + lane;
        double fid, mx;
        if constexpr (CX) {
            const double sr = wave_sum_v(real ? x : 0.0), si = wave_sum_v(real ? xi : 0.0);
            double yr = x, yi = xi;
            if (sr != 0.0 || si != 0.0) {  // x / S, scaled against overflow of |S|^2
                const double sc = fmax(fabs(sr), fabs(si));
                const double br = sr / sc, bi = si / sc, den = (br * br + bi * bi) * sc;
                yr = (x * br + xi * bi) / den;
                yi = (xi * br - x * bi) / den;
            }
            const double xr = real ? mold[2 * mo] : 0.0, xo = real ? mold[2 * mo + 1] : 0.0;
            if (!real) yr = yi = 0.0;
            if (real) {
                mnew[2 * mo] = yr;
                mnew[2 * mo + 1] = yi;
            }
            const double dr = wave_sum_v(xr * yr + xo * yi), di = wave_sum_v(xr * yi - xo * yr);
            const double nn = wave_sum_v(yr * yr + yi * yi), oo = wave_sum_v(xr * xr + xo * xo);
            mx = wave_max_v(sqrt((yr - xr) * (yr - xr) + (yi - xo) * (yi - xo)));
            fid = 1.0 - (dr * dr + di * di) / (nn * oo);
        } else {
            const double S = wave_sum_v(real ? (double)x : 0.0);
            const E y = real ? (E)(S != 0.0 ? (double)x / S : (double)x) : E(0);
            const double xo = real ? (double)mold[mo] : 0.0, yn = (double)y;
            if (real) mnew[mo] = y;
            const double dn = wave_sum_v(yn * xo), nn = wave_sum_v(yn * yn),
                         oo = wave_sum_v(xo * xo);
            mx = wave_max_v(fabs(yn - xo));
            const double c = dn / sqrt(nn * oo);
            fid = 1.0 - c * c;
        }
        if (lane == 0) {
            res_fid[q] = fid;
            res_abs[q] = mx;
            fm = fold_max(fm, fcrit ? mx : fid);
        }
    }
    if (fold.acc) {
        if (lane == 0) fold_m[w] = fm;
        __syncthreads();
        if (tid == 0) {
            double m = 0.0;
            for (int k = 0; k < W; ++k) m = fold_max(m, fold_m[k]);
            atomicMax(fold.acc + (long long)net * FOLD_SLOTS + (item % FOLD_SLOTS),
                      (unsigned long long)__double_as_longlong(m));
        }
    }
}

// ------------------------------------------------------------------ host

static constexpr size_t PAIR_LDS_MAX = 160 * 1024 - 256;  // 256: the static fold buffer

void pair_release(PairPlan *p) {
    if (p->d_recs) (void)hipFree(p->d_recs);
    if (p->d_lead) (void)hipFree(p->d_lead);
    *p = PairPlan();
}

template <int TY>
static const void *pair_fn(int nt) {
    switch (nt) {
        case 1: return (const void *)k_pair<TY, 1>;
        case 2: return (const void *)k_pair<TY, 2>;
    }
    if constexpr (TY == PAIR_C128) return nullptr;
    else return nt == 3 ? (const void *)k_pair<TY, 3> : (const void *)k_pair<TY, 4>;
}

int pair_plan_build(PairPlan *p, int dtype, int plain, int nv, int nnet, const int *port_off,
                    const int *port_edge, const int *edge_dim, const int *phys_dim,
                    const int *port_rev, const int *vnet, const long long *site_off,
                    const long long *msg_off) {
    pair_release(p);
    if (plain) return 4;
    p->dtype = dtype;
    p->rec_of.assign(nv, -1);
    // complex tensors take two planes: bond dimensions up to 5 (25-wide pairs)
    const int side = dtype == PAIR_C128 ? 32 : PAIR_SIDE;
    int maxn = 1, maxd = 1;
    std::vector<int> lead(nnet, -1);
    for (int u = 0; u < nv; ++u) {
        const int base = port_off[u], k = port_off[u + 1] - base;
        int dm[4] = {1, 1, 1, 1}, at[4] = {-1, -1, -1, -1};
        bool ok = k >= 1 && k <= 4;
        for (int j = 0; j < k && ok; ++j) {
            const int pos = k == 2 ? 2 * j : j;
            dm[pos] = edge_dim[port_edge[base + j]];
            at[pos] = base + j;
            if (dm[pos] > PAIR_MAXD) ok = false;
        }
        if (ok && (dm[0] * dm[1] > side || dm[2] * dm[3] > side)) ok = false;
        if (!ok) {
            for (int q = base; q < base + k; ++q) p->rest.push_back(q);
            continue;
        }
        PairRec r{};
        r.site = site_off[u];
        for (int t = 0; t < 4; ++t) {
            r.dim[t] = dm[t];
            r.slot[t] = at[t];
            r.in[t] = at[t] >= 0 ? msg_off[port_rev[at[t]]] : 0;
            r.out[t] = at[t] >= 0 ? msg_off[at[t]] : 0;
        }
        r.d = phys_dim[u];
        r.net = vnet[u];
        r.n[0] = dm[0] * dm[1];
        r.n[1] = dm[2] * dm[3];
        r.vertex = u;
        maxn = std::max(maxn, std::max(r.n[0], r.n[1]));
        maxd = std::max(maxd, r.d);
        p->rec_of[u] = (int)p->recs.size();
        if (lead[r.net] < 0) lead[r.net] = (int)p->recs.size();
        p->recs.push_back(r);
    }
    if (p->recs.empty()) return 4;
    p->covers = p->rest.empty();
    p->all = (int)p->recs.size() == nv;
    for (int n = 0; n < nnet; ++n) p->covers = p->covers && lead[n] >= 0;
    p->nt = (maxn + 15) / 16;
    // one tile column per half leaves two waves: share the slices between two more
    p->split = p->nt <= 2 && maxd >= 2 ? 2 : 1;
    p->waves = 2 * p->nt * p->split;
    const size_t esz = dtype == PAIR_F32 ? 4 : dtype == PAIR_C128 ? 16 : 8;
    int slice = 0, env = 0;
    for (const PairRec &r : p->recs) {
        const int N0 = pair_pad(r.n[0]), N1 = pair_pad(r.n[1]);
        slice = std::max(slice, pair_slice_elems(r.n[0], r.n[1]));
        env = std::max(env, p->split * (N0 * N0 + N1 * N1));
    }
    const size_t fixed = esz * ((size_t)env + 4 * 64);
    // as many slices at a time as fit the LDS
    int chunk = maxd;
    while (chunk > 1 && fixed + esz * (size_t)chunk * slice > PAIR_LDS_MAX) --chunk;
    p->chunk = chunk;
    p->slice_elems = slice;
    p->env_elems = env;
    p->lds_bytes = fixed + esz * (size_t)chunk * slice;
    if (p->lds_bytes > PAIR_LDS_MAX) { pair_release(p); return 4; }
    if (hipMalloc((void **)&p->d_recs, sizeof(PairRec) * p->recs.size()) != hipSuccess ||
        hipMalloc((void **)&p->d_lead, sizeof(int) * nnet) != hipSuccess ||
        hipMemcpy(p->d_recs, p->recs.data(), sizeof(PairRec) * p->recs.size(),
                  hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->d_lead, lead.data(), sizeof(int) * nnet, hipMemcpyHostToDevice) !=
            hipSuccess) {
        pair_release(p);
        return 5;
    }
    const void *fn = dtype == PAIR_F64 ? pair_fn<PAIR_F64>(p->nt)
                     : dtype == PAIR_C128 ? pair_fn<PAIR_C128>(p->nt) : pair_fn<PAIR_F32>(p->nt);
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)PAIR_LDS_MAX) != hipSuccess) {
        pair_release(p);
        return 2;
    }
    return 0;
}

double pair_mfma_per_slice(const PairPlan *p) {
    double n = 0.0, slices = 0.0;
    for (const PairRec &r : p->recs) {
        for (int h = 0; h < 2; ++h) {  // per column tile: E, then the environment
            const int tI = (r.n[h] + 15) / 16, tJ = (r.n[1 - h] + 15) / 16, kt = (r.n[h] + 3) / 4;
            n += (double)r.d * tJ * (tI * kt + 4 * tI * tJ);
        }
        slices += r.d;
    }
    return slices > 0.0 ? n / slices : 0.0;
}

template <int TY>
static int pair_go(const PairPlan *p, hipStream_t st, const void *sites, const void *src,
                   void *dst, const NetCtl &ctl, double *rf, double *ra, const SweepFold &fold,
                   const int *items, int n, double *zv) {
    using E = typename PairTy<TY>::E;
    const int blocks = items ? n : (int)p->recs.size();
    if (blocks == 0) return 0;
#define PAIR_GO(NT)                                                                               \
    hipLaunchKernelGGL((k_pair<TY, NT>), dim3(blocks), dim3(64 * p->waves), p->lds_bytes, st,      \
                       p->d_recs, items, (const E *)sites, (const E *)src, (E *)dst, ctl, rf, ra, \
                       fold, p->chunk, p->split, p->slice_elems, p->env_elems, zv)
    switch (p->nt) {
        case 1: PAIR_GO(1); break;
        case 2: PAIR_GO(2); break;
        case 3: if constexpr (TY != PAIR_C128) PAIR_GO(3); break;
        default: if constexpr (TY != PAIR_C128) PAIR_GO(4); break;
    }
#undef PAIR_GO
    return hipGetLastError() == hipSuccess ? 0 : 2;
}

static int pair_any(const PairPlan *p, hipStream_t st, const void *sites, const void *src,
                    void *dst, const NetCtl &ctl, double *rf, double *ra, const SweepFold &fold,
                    const int *items, int n, double *zv) {
    if (p->dtype == PAIR_F64)
        return pair_go<PAIR_F64>(p, st, sites, src, dst, ctl, rf, ra, fold, items, n, zv);
    if (p->dtype == PAIR_C128)
        return pair_go<PAIR_C128>(p, st, sites, src, dst, ctl, rf, ra, fold, items, n, zv);
    return pair_go<PAIR_F32>(p, st, sites, src, dst, ctl, rf, ra, fold, items, n, zv);
}

int pair_sweep(const PairPlan *p, hipStream_t st, const void *sites, const void *src, void *dst,
               const NetCtl &ctl, double *res_fid, double *res_abs, const SweepFold &fold,
               const int *items, int n) {
    return pair_any(p, st, sites, src, dst, ctl, res_fid, res_abs, fold, items, n, nullptr);
}

int pair_scalars(const PairPlan *p, hipStream_t st, const void *sites, const void *msgs,
                 double *zv) {
    NetCtl off{};
    return pair_any(p, st, sites, msgs, nullptr, off, nullptr, nullptr, SweepFold{}, nullptr, 0,
                    zv);
}
