// pair.hip -- BP messages of a vertex from two pair environments, on FP64 MFMA.
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
    static constexpr int ROW = 4;  // register r holds rows 4 r .. 4 r + 3
};
template <>
struct PairTy<PAIR_C128> : PairTy<PAIR_F64> {
    static constexpr bool CX = true;
};

// waves of the largest workgroup with NT tile columns
constexpr int pair_waves(int NT) { return NT == 3 ? 12 : 8; }

__host__ __device__ inline int pair_pad(int n) { return (n + 15) & ~15; }

// LDS elements per plane (complex: two planes): staged slices, Kronecker messages or
// environments (they share the space), incoming messages.
__host__ __device__ inline int pair_slice_elems(int n0, int n1) {
    // an odd row pitch: both the rows and the columns of a slice are read 16 at a time
    return pair_pad(n0) * (pair_pad(n1) + 1);
}

// environments have an odd row pitch too: a message is opened over rows, columns or both
__host__ __device__ inline int pair_env_elems(int N0, int N1) {
    return N0 * (N0 + 1) + N1 * (N1 + 1);
}

// floor(i / n) for 0 <= i < 2^22, 1 <= n
__device__ __forceinline__ int fdiv(int i, float rn) { return (int)(((float)i + 0.5f) * rn); }

// One workgroup's work on one vertex, from LDS; NT: tiles of the largest pair side this
// instance handles.  Every member is inlined into the kernels below.
template <int TY, int NT>
struct PairCore {
    using P = PairTy<TY>;
    using E = typename P::E;
    using V = typename P::V;
    static constexpr bool CX = P::CX;
    static constexpr int PL = CX ? 2 : 1;  // planes; global elements are interleaved (re, im)

    E *Al, *Ml, *ml;  // [plane][chunk][slice], [plane][env_elems], [position][plane][64]
    const PairRec &rec;
    int tid, lane, w, nthr, W;
    int plA, env_elems, split;
    int n0, n1, d, N0, N1, P1, SL;

    __device__ __forceinline__ PairCore(char *smem, const PairRec &r, int chunk, int split_,
                                        int slice_elems, int env_elems_)
        : rec(r), env_elems(env_elems_), split(split_) {
        Al = reinterpret_cast<E *>(smem);
        Ml = Al + (size_t)PL * chunk * slice_elems;
        ml = Ml + (size_t)PL * env_elems;
        plA = chunk * slice_elems;
        tid = threadIdx.x;
        lane = tid & 63;
        w = __builtin_amdgcn_readfirstlane(tid >> 6);  // scalar: what depends on it is, too
        nthr = blockDim.x;
        W = nthr >> 6;
        n0 = rec.n[0];
        n1 = rec.n[1];
        d = rec.d;
        N0 = pair_pad(n0);
        N1 = pair_pad(n1);
        P1 = N1 + 1;
        SL = N0 * P1;
    }

    // ---- slices [s0, s0 + cnt) into LDS, zero-padded; every load of a batch is issued before
    // the first LDS store waits for it
    __device__ __forceinline__ void stage(const E *A, int s0, int cnt) {
        const float rP = 1.0f / (float)P1, rN = 1.0f / (float)N0;
        constexpr int B = CX ? 4 : 8;
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
    }

    // ---- Kronecker products M_h[(a b)][(a' b')] = m_a[a][a'] m_b[b][b'], zero-padded
    __device__ __forceinline__ void kron(int h) {
        const int n = h ? n1 : n0, N = h ? N1 : N0, Db = rec.dim[2 * h + 1], Da = rec.dim[2 * h];
        E *M = Ml + (h ? N0 * N0 : 0);
        const E *ma = ml + (2 * h) * PL * 64, *mb = ml + (2 * h + 1) * PL * 64;
        const int rows = nthr / N;  // rows of M per pass
        const int col = tid % N, r0 = tid / N;
        if (r0 >= rows) return;
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

    // ---- environments: this wave's (half, columns, slice share)
    int h, J, sg, nI, nJ;
    bool work;

    // need: halves whose environment is wanted
    __device__ __forceinline__ void env_begin(bool need0, bool need1, V (&R)[NT],
                                              V (&Ri)[CX ? NT : 1]) {
        const int t0 = N0 >> 4, t1 = N1 >> 4;
        const int per = NT * split;  // waves per half
        h = w / per;
        J = (w % per) / split;
        sg = w % split;
        nI = h ? t1 : t0;  // tiles of the contracted / the other pair
        nJ = h ? t0 : t1;
        work = h < 2 && ((h & 1) ? need1 : need0) && J < nJ;
#pragma unroll
        for (int j = 0; j < NT; ++j) R[j] = V{0, 0, 0, 0};
        if constexpr (CX) {
#pragma unroll
            for (int j = 0; j < NT; ++j) Ri[j] = V{0, 0, 0, 0};
        }
    }

    // the staged slices [0, cnt); m(I, t, re, im) gives this lane's entry of the Kronecker
    // message, row 4 t + lane / 16 and column 16 I + lane % 16
    template <typename Operand>
    __device__ __forceinline__ void env_add(int cnt, V (&R)[NT], V (&Ri)[CX ? NT : 1],
                                            const Operand &m) {
        if (!work) return;
        const int lk = lane >> 4, li = lane & 15;
        const int nh = h ? n1 : n0;
        const int sk = h ? 1 : P1, sj = h ? P1 : 1;  // strides of the contracted / other index
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
                        E mr, mi;
                        m(I, t, mr, mi);
                        if constexpr (CX) {
                            C = P::mma(mr, X[t], C);
                            C = P::mma(-mi, Xi[t], C);
                            Ci = P::mma(mr, Xi[t], Ci);
                            Ci = P::mma(mi, X[t], Ci);
                        } else {
                            C = P::mma(mr, X[t], C);
                        }
                    }
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    if (j >= nJ) break;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if (16 * I + P::ROW * r >= nh) break;  // padding
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

    // the Kronecker message in LDS
    __device__ __forceinline__ auto staged() const {
        const E *M = Ml + (h ? N0 * N0 : 0) + (lane >> 4) * (h ? N1 : N0) + (lane & 15);
        const int Nh = h ? N1 : N0, im = env_elems;
        return [M, Nh, im](int I, int t, E &mr, E &mi) {
            const int o = 4 * t * Nh + 16 * I;
            mr = M[o];
            if constexpr (CX) mi = M[im + o];
        };
    }

    // R^T of the other pair into the space of the Kronecker messages: [share][pair][n'][n]
    __device__ __forceinline__ void env_store(const V (&R)[NT], const V (&Ri)[CX ? NT : 1]) {
        if (!work) return;
        const int lk = lane >> 4, li = lane & 15;
        const int No = (h ? N0 : N1) + 1;
        E *Ro = Ml + sg * pair_env_elems(N0, N1) + (h ? 0 : N0 * (N0 + 1));
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

    // ---- unnormalised message out of position p (one wave): entry `lane` of lanes below D^2.
    // What a lane reads depends on the vertex only.
    struct OpenAt {
        int v, m, b;  // first environment entry, partner entry, partner row (of lanes in use)
    };
    __device__ __forceinline__ int open_groups(int p) const {
        const int DD = rec.dim[p] * rec.dim[p], Dp = rec.dim[p ^ 1];
        int G = 1;
        while (2 * G * DD <= 64 && G < Dp) G *= 2;  // lanes per entry, lane = g * DD + entry
        return G;
    }
    __device__ __forceinline__ OpenAt open_at(int p) const {
        const int D = rec.dim[p], Dp = rec.dim[p ^ 1], DD = D * D;
        const int sa = (p & 1) ? 1 : Dp, sb = (p & 1) ? D : 1;
        const int N = ((p >> 1) ? N1 : N0) + 1;
        const int g = fdiv(lane, 1.0f / (float)DD), e = lane - g * DD;
        const int a = fdiv(e, 1.0f / (float)D), a2 = e - a * D;
        OpenAt o;
        o.v = ((p >> 1) ? N0 * (N0 + 1) : 0) + a2 * sa * N + a * sa + g * sb;
        o.m = (p ^ 1) * PL * 64 + g * Dp;
        o.b = g < open_groups(p) ? g : Dp;
        return o;
    }
    struct Entry {
        E re, im;
    };
    __device__ __forceinline__ Entry open(int p, const OpenAt at) const {
        const int D = rec.dim[p], Dp = rec.dim[p ^ 1], DD = D * D, G = open_groups(p);
        const int sb = (p & 1) ? D : 1;
        const int N = ((p >> 1) ? N1 : N0) + 1;
        const E *mp = ml + at.m, *Ro = Ml + at.v;
        // the other share of the slices (without one, the same entry read again and dropped: a
        // branch here would wait for every load by itself)
        constexpr bool SHARES = NT < 4;
        const bool two = split > 1;
        const int eshare = two ? pair_env_elems(N0, N1) : 0;
        E x = E(0), xi = E(0);
        // lane g takes rows b = g, g + G, ... of the partner message; the eight columns are
        // read at once (clamped, the absent ones dropped)
        for (int b = at.b; b < Dp; b += G, mp += G * Dp, Ro += G * sb) {
            E v[8], m[8], u[8], vi[CX ? 8 : 1], mi[CX ? 8 : 1], ui[CX ? 8 : 1];
#pragma unroll
            for (int b2 = 0; b2 < 8; ++b2) {
                const int bc = min(b2, Dp - 1), o = bc * sb * N;
                v[b2] = Ro[o];
                m[b2] = mp[bc];
                if constexpr (SHARES) u[b2] = Ro[eshare + o];
                if constexpr (CX) {
                    vi[b2] = Ro[env_elems + o];
                    mi[b2] = mp[64 + bc];
                    ui[b2] = Ro[env_elems + eshare + o];
                }
            }
#pragma unroll
            for (int b2 = 0; b2 < 8; ++b2) {
                if constexpr (SHARES) v[b2] = two ? v[b2] + u[b2] : v[b2];
                if constexpr (CX) vi[b2] = two ? vi[b2] + ui[b2] : vi[b2];
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
        for (int k = G >> 1; k > 0; k >>= 1) {
            x += __shfl_down(x, k * DD, 64);
            if constexpr (CX) xi += __shfl_down(xi, k * DD, 64);
        }
        return {x, xi};
    }

    // the message's residuals against its previous values xo (+ i xoi), zero on lanes that
    // hold no entry
    __device__ __forceinline__ static void residual(E y, E yi, E xo, E xoi, double &fid,
                                                    double &mx) {
        if constexpr (CX) {
            const double dr = wave_sum_v(xo * y + xoi * yi), di = wave_sum_v(xo * yi - xoi * y);
            const double nn = wave_sum_v(y * y + yi * yi), oo = wave_sum_v(xo * xo + xoi * xoi);
            mx = wave_max_v(sqrt((y - xo) * (y - xo) + (yi - xoi) * (yi - xoi)));
            fid = 1.0 - (dr * dr + di * di) / (nn * oo);
        } else {
            const double dn = wave_sum_v(y * xo), nn = wave_sum_v(y * y),
                         oo = wave_sum_v(xo * xo);
            mx = wave_max_v(fabs(y - xo));
            const double c = dn / sqrt(nn * oo);
            fid = 1.0 - c * c;
        }
    }

    // the message divided by its sum, zero on lanes that hold no entry
    __device__ __forceinline__ static Entry normalise(bool real, const Entry v) {
        const E x = v.re, xi = v.im;
        if constexpr (CX) {
            const double sr = wave_sum_v(real ? x : 0.0), si = wave_sum_v(real ? xi : 0.0);
            double yr = x, yi = xi;
            if (sr != 0.0 || si != 0.0) {  // x / S, scaled against overflow of |S|^2
                const double sc = fmax(fabs(sr), fabs(si));
                const double br = sr / sc, bi = si / sc, den = (br * br + bi * bi) * sc;
                yr = (x * br + xi * bi) / den;
                yi = (xi * br - x * bi) / den;
            }
            return {real ? yr : 0.0, real ? yi : 0.0};
        } else {
            const double S = wave_sum_v(real ? x : 0.0);
            return {real ? (S != 0.0 ? x / S : x) : 0.0, 0.0};
        }
    }
};

template <int TY, int NT>
__global__ __launch_bounds__(64 * pair_waves(NT)) void k_pair(
    const PairRec *__restrict__ recs, const int *__restrict__ items,
    const typename PairTy<TY>::E *__restrict__ sites, const typename PairTy<TY>::E *mold,
    typename PairTy<TY>::E *mnew, NetCtl ctl, double *__restrict__ res_fid,
    double *__restrict__ res_abs, SweepFold fold, int chunk, int split, int slice_elems,
    int env_elems, double *__restrict__ zv) {
    using Core = PairCore<TY, NT>;
    using E = typename PairTy<TY>::E;
    constexpr bool CX = Core::CX;
    constexpr int PL = Core::PL;
    extern __shared__ __align__(16) char smem[];
    __shared__ double fold_m[pair_waves(NT)];

    const int item = blockIdx.x;
    const int ri = items ? items[item] >> 2 : item;
    // positions to update; the vertex scalar comes from position 0's unnormalised message
    const int mask = zv ? 1 : items ? 1 << (items[item] & 3) : 15;
    const PairRec &rec = recs[ri];
    Core K(smem, rec, chunk, split, slice_elems, env_elems);
    const int tid = K.tid, lane = K.lane, w = K.w, nthr = K.nthr, W = K.W;
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

    // ---- incoming messages (one position per wave) and the first slices
    const E *A = sites + rec.site * PL;
    E *ml = K.ml;
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
    K.stage(A, 0, min(chunk, K.d));
    __syncthreads();
    for (int h = 0; h < 2; ++h) K.kron(h);
    __syncthreads();

    typename Core::V R[NT], Ri[CX ? NT : 1];
    K.env_begin((mask & 12) != 0 && rec.slot[2] >= 0, (mask & 3) != 0, R, Ri);
    for (int s0 = 0; s0 < K.d; s0 += chunk) {
        if (s0) {
            __syncthreads();
            K.stage(A, s0, min(chunk, K.d - s0));
            __syncthreads();
        }
        K.env_add(min(chunk, K.d - s0), R, Ri, K.staged());
    }
    __syncthreads();  // every wave has read M: its space takes the environments
    K.env_store(R, Ri);
    __syncthreads();

    // ---- messages: wave w takes positions w, w + W, ...
    double fm = 0.0;
    const bool fcrit = fold.acc && fold.rp->crit != 0;
    for (int p = w; p < 4; p += W) {
        const int q = rec.slot[p];
        if (q < 0 || !((mask >> p) & 1)) continue;
        typename Core::Entry v = K.open(p, K.open_at(p));
        const bool real = lane < rec.dim[p] * rec.dim[p];
        if (zv) {
            if constexpr (CX) {
                const E mr = ml[lane & 63], mi = ml[64 + (lane & 63)];
                const double zr = wave_sum_v(real ? v.re * mr - v.im * mi : 0.0);
                const double zi = wave_sum_v(real ? v.re * mi + v.im * mr : 0.0);
                if (lane == 0) {
                    zv[2 * rec.vertex] = zr;
                    zv[2 * rec.vertex + 1] = zi;
                }
            } else {
                const double z = wave_sum_v(real ? v.re * ml[lane] : 0.0);
                if (lane == 0) zv[rec.vertex] = z;
            }
            continue;
        }
        const long long mo = rec.out[p] + lane;
        v = Core::normalise(real, v);
        E xo = E(0), xoi = E(0);
        if (real) {
            xo = mold[PL * mo];
            mnew[PL * mo] = v.re;
            if constexpr (CX) {
                xoi = mold[PL * mo + 1];
                mnew[PL * mo + 1] = v.im;
            }
        }
        double fid, mx;
        Core::residual(v.re, v.im, xo, xoi, fid, mx);
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

// ------------------------------------------------------------------ many sweeps a launch

// A whole run of one network whose vertices are all resident at once: workgroup i keeps vertex
// i's slices in LDS for up to PAIR_RUN_SWEEPS sweeps, and the messages go from workgroup to
// workgroup through a ring of PAIR_RING versions in device memory, version s holding the
// messages after sweep s of the launch.
//
// Why: the sweeps of small networks are launch latency and cold loads (8.9 us a sweep of a 4x4
// lattice at D = 2, of which the products are a fraction of a microsecond), and a sequential
// sweep of L x L vertices is about 4 L launches.  Here a sweep costs one trip of a message
// through memory and the products, and the sweeps of a sequential schedule overlap.
//
// Waiting: an entry not yet written holds PAIR_POISON, a signalling NaN that no arithmetic
// produces, so a reader polls the entries it needs and no flag or fence orders them.  The
// writer of version s poisons version s + 2 beside it, and waits for its own earlier stores
// before it stores version s + 1; a reader looks at version s + 2 only after version s + 1.
// A schedule is a list of steps per vertex: the positions it updates together and, per
// incoming message, whether it reads this sweep's version or the last one's.  The unfinished
// step that comes first in the schedule has its inputs, so some step can always run as long as
// every workgroup is resident.
//
// Bounded run-ahead: a workgroup starts sweep s when all have finished sweep s - 4 and the
// stopping rule says that sweep s - 5 was not the last, so the versions in use, s - 5 to
// s + 2, are distinct entries of the ring; all workgroups leave at the same sweep.  A sequential
// sweep is long: it waits for all to have finished sweep s - 2 and reads that one's residual
// then (the sweeps after the last one are work for nothing: 10x10 D = 4, eight sweeps, 1136 us
// a call with the longer look back).
//
// Every poll ends after the caller's limit (0.25 s by default), when the network turns out not to be resident as a
// whole (another process on the device, say): the run's state is then marked PAIR_RUN_BAILED
// and the caller runs it again launch by launch from the untouched source messages.  The next
// 1, 2, 4, .. runs of the plan go launch by launch too, so what was there for a moment costs one
// wait, and what stays costs a wait in ever more runs.
static constexpr int PAIR_RING = 8;
static constexpr unsigned long long PAIR_POISON = 0x7FF4DEADBEEF0001ull;
static constexpr unsigned long long PAIR_QUIET = 1ull << 51;
#define PAIR_CTRL_LINES 8  // counters of a sweep, on separate cache lines

struct alignas(64) PairCtrl {
    unsigned long long acc;  // largest residual, as bits of a value >= 0 or NaN
    unsigned int cnt;        // workgroups that have finished the sweep
};

struct PairRunArgs {
    unsigned long long *ring;  // [PAIR_RING][nm]
    long long nm;              // doubles of one version
    double *dst;               // the messages after the last sweep
    PairCtrl *ctrl;            // [sweep][PAIR_CTRL_LINES]
    double *res;               // [PAIR_RING][2][nports]
    double *res_fid, *res_abs;
    int *done, *iter, *at;     // state of the network
    double *delta;
    double tol;
    int crit, sweeps, first, last;  // sweeps of this launch and before it; whether it ends the run
    int nports, nrec;
    int split, slice_elems, env_elems, chunk;
    int every, maxiter;
    long long ticks;  // wait limit, in ticks of the 100 MHz clock
    int looks;        // the clock is read when a wait's count of looks & looks is 0
};

__global__ void k_pair_run_init(const unsigned long long *__restrict__ src, PairRunArgs a) {
    const long long n = (long long)gridDim.x * blockDim.x;
    const long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    for (long long i = i0; i < a.nm; i += n) {
        const unsigned long long v = src[i];
        a.ring[i] = v == PAIR_POISON ? v | PAIR_QUIET : v;
        for (int k = 1; k < PAIR_RING; ++k) a.ring[k * a.nm + i] = PAIR_POISON;
    }
    for (long long i = i0; i < (long long)a.sweeps * PAIR_CTRL_LINES; i += n) {
        a.ctrl[i].acc = 0ull;
        a.ctrl[i].cnt = 0u;
    }
    if (i0 == 0 && a.first == 0) {
        *a.done = 0;
        *a.iter = 0;
        *a.at = -1;
        *a.delta = INFINITY;
    }
}

template <typename T>
__device__ __forceinline__ T pair_get(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// earlier stores and atomics of this wave have reached the coherence point of the device
__device__ __forceinline__ void pair_settle() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0);
    asm volatile("" ::: "memory");
}

// One look at a wait that has not ended; false once it must be given up.
__device__ __forceinline__ bool pair_wait(const PairRunArgs &a, long long t0, int &n) {
    __builtin_amdgcn_s_sleep(1);
    if ((++n & a.looks) != 0) return true;
    return wall_clock64() - t0 < a.ticks && !(pair_get(a.done) & PAIR_RUN_BAILED);
}

// All workgroups have finished sweep t (1-based); one wave, v: its counters as last seen.
__device__ __forceinline__ bool pair_finished(const PairRunArgs &a, int t, int lane,
                                              unsigned int v) {
    const PairCtrl *c = a.ctrl + (long long)(t - 1) * PAIR_CTRL_LINES;
    long long t0 = 0;
    for (int n = 0;;) {
        v += __shfl_xor(v, 1, 64);
        v += __shfl_xor(v, 2, 64);
        v += __shfl_xor(v, 4, 64);
        if ((int)__builtin_amdgcn_readfirstlane((int)v) == a.nrec) return true;
        if (t0 == 0) t0 = wall_clock64();
        if (!pair_wait(a, t0, n)) return false;
        v = lane < PAIR_CTRL_LINES ? pair_get(&c[lane].cnt) : 0u;
    }
}

// The largest residual of a finished sweep (one wave).
__device__ __forceinline__ double pair_delta(const PairRunArgs &a, int t, int lane) {
    const PairCtrl *c = a.ctrl + (long long)(t - 1) * PAIR_CTRL_LINES;
    const unsigned long long v = lane < PAIR_CTRL_LINES ? pair_get(&c[lane].acc) : 0ull;
    return wave_max_v(__longlong_as_double((long long)v));
}

// steps: [record][4], positions | incoming versions << 4 (bit set: this sweep's), 0: none
// Pairs of up to 16 form the entries of the Kronecker messages from the messages as the products
// read them, which saves the pass that stages them and two of its barriers (the LDS offsets stay
// in registers); larger ones stage them.  Pairs of up to 32 in FP64: four waves a SIMD, two
// workgroups on a CU.
template <int TY, int NT>
__global__ __launch_bounds__(64 * pair_waves(NT), TY == PAIR_F64 && NT == 2 ? 4 : 1) void k_pair_run(
    const PairRec *__restrict__ recs, const int4 *__restrict__ step_list,
    const double *__restrict__ sites, PairRunArgs a) {
    using Core = PairCore<TY, NT>;
    constexpr bool CX = Core::CX, DIRECT = NT == 1;
    constexpr int PL = Core::PL;
    constexpr int MB = 4 * PL * 64;  // one set of incoming messages
    extern __shared__ __align__(16) char smem[];
    __shared__ double fold_m[pair_waves(NT)];
    __shared__ int verdict;  // 0: go on, 1: the sweep of the look-back was the last, 2: give up
    __shared__ int stop_at;

    const int ri = blockIdx.x;
    const PairRec &rec = recs[ri];
    Core K(smem, rec, a.chunk, a.split, a.slice_elems, a.env_elems);
    const int tid = K.tid, lane = K.lane, w = K.w, W = K.W;
    // ml: the incoming messages, two sets taken in turn by the sweeps of a Jacobi run; own: the
    // outgoing ones
    double *const ml0 = K.ml, *zero = ml0 + MB;  // the zeros belong to their set
    constexpr int SET = MB + 128;
    double *own = ml0 + 2 * SET;
    const int4 steps = step_list[ri];
    const bool turns = a.every > 0;  // Jacobi: one step a sweep, which reads every message anew
    const int lag = turns ? 4 : 2, back = turns ? 5 : 2;

    if (tid == 0) verdict = 0;
    if (tid < 128) zero[tid] = zero[SET + tid] = 0.0;
    for (int p = w; p < 4; p += W) {
        const bool have = rec.slot[p] >= 0, real = have && lane < rec.dim[p] * rec.dim[p];
        for (int b = 0; b < 2; ++b) {
            ml0[b * SET + p * PL * 64 + lane] = 1.0;
            if constexpr (CX) ml0[b * SET + (p * 2 + 1) * 64 + lane] = 0.0;
        }
        own[p * PL * 64 + lane] =
            real ? __longlong_as_double((long long)a.ring[(rec.out[p] + lane) * PL]) : 0.0;
        if constexpr (CX)
            own[(p * 2 + 1) * 64 + lane] =
                real ? __longlong_as_double((long long)a.ring[(rec.out[p] + lane) * 2 + 1]) : 0.0;
    }
    K.stage(sites + rec.site * PL, 0, K.d);
    // offsets of the factors of this lane's Kronecker entries: first | second << 16
    unsigned int at[DIRECT ? 4 * NT * NT : 1];
    if constexpr (DIRECT) {
        typename Core::V R[NT], Ri[CX ? NT : 1];
        K.env_begin(true, true, R, Ri);  // this wave's half
        const int h = K.h & 1, n = h ? K.n1 : K.n0, Da = rec.dim[2 * h], Db = rec.dim[2 * h + 1];
#pragma unroll
        for (int I = 0; I < NT; ++I)
#pragma unroll
            for (int t = 0; t < 4 * NT; ++t) {
                const int k = 4 * t + (lane >> 4), c = 16 * I + (lane & 15);
                const int ia = (k / Db) * Da + c / Db, ib = (k % Db) * Db + c % Db;
                const int z = (int)(zero - ml0);
                at[I * 4 * NT + t] = k < n && c < n
                                         ? (unsigned)(2 * h * PL * 64 + ia) |
                                               (unsigned)((2 * h + 1) * PL * 64 + ib) << 16
                                         : (unsigned)z | (unsigned)z << 16;
            }
    }
    __syncthreads();

    typename Core::OpenAt where[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) where[i] = K.open_at(min(w + i * W, 3));
    int loaded[2] = {-1, -1};  // version of the incoming message in LDS, per position of the wave
    int stop = 0, s = 1;
    bool leave = false;
    // the maximum of sweep s goes out (thread 0), and in a Jacobi run sweep s - 1 is counted: a
    // maximum is stored a sweep before its count, and this wave has settled in between
    // (position 0 is always there and is updated once a sweep)
    auto report = [&](int s) {
        PairCtrl *c = a.ctrl + (long long)(s - 1) * PAIR_CTRL_LINES + ri % PAIR_CTRL_LINES;
        double m = 0.0;
        for (int k = 0; k < W; ++k) m = fold_max(m, fold_m[k]);
        if (turns && s > 1)
            __hip_atomic_fetch_add(&c[-PAIR_CTRL_LINES].cnt, 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_fetch_max(&c->acc, (unsigned long long)__double_as_longlong(m),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    for (; s <= a.sweeps; ++s) {
        double fm = 0.0;
        double *ml = ml0 + (turns ? (s & 1) * SET : 0);
        K.ml = ml;
        for (int k = 0; k < 4; ++k) {
            const int step = k == 0 ? steps.x : k == 1 ? steps.y : k == 2 ? steps.z : steps.w;
            if (step == 0) break;
            const int mask = step & 15;
            const bool need0 = (mask & 12) != 0 && rec.slot[2] >= 0, need1 = (mask & 3) != 0;
            // addresses are formed anew for every step: kept across the loop, they spill
            if constexpr (!DIRECT) asm volatile("" : "+v"(K.lane), "+v"(K.tid));
            // ---- once a sweep, the last wave: has the run ended, may this sweep's versions be
            // written.  Its loads go ahead of the first poll's, its waits come after.
            bool look = k == 0 && w == W - 1 && s > lag;
            unsigned long long acc = 0ull;
            unsigned int cnt = 0u;
            if (look && lane < PAIR_CTRL_LINES) {
                const PairCtrl *c = a.ctrl + (long long)(s - lag - 1) * PAIR_CTRL_LINES + lane;
                cnt = pair_get(&c->cnt);
                if (turns && s > back) acc = pair_get(&c[-PAIR_CTRL_LINES].acc);
            }
            auto look_back = [&]() {
                look = false;
                if (turns && s > back && a.tol >= 0.0 &&
                    wave_max_v(__longlong_as_double((long long)acc)) < a.tol)
                    verdict = 1;
                else if (!pair_finished(a, s - lag, lane, cnt))
                    verdict = 2;
                else if (!turns && a.tol >= 0.0 && pair_delta(a, s - back, lane) < a.tol)
                    verdict = 1;
            };
            // ---- the messages this step reads, polled until they are there; a run that has
            // ended writes no more of them
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int p = w + i * W;
                if (p >= 4) break;
                const int ver = s - 1 + ((step >> (4 + p)) & 1);
                if (rec.slot[p] < 0 || (mask & ~(1 << p)) == 0 || loaded[i] == ver) continue;
                const unsigned long long *in =
                    a.ring + (ver % PAIR_RING) * a.nm + (rec.in[p] + lane) * PL;
                const bool real = lane < rec.dim[p] * rec.dim[p];
                unsigned long long v = 0ull, vi = 0ull;
                auto get = [&]() {
                    if (!real) return;
                    v = pair_get(in);
                    if constexpr (CX) vi = pair_get(in + 1);
                };
                get();
                if (look) look_back();
                if (!__all(v != PAIR_POISON && vi != PAIR_POISON)) {
                    const long long t0 = wall_clock64();
                    for (int n = 0;;) {
                        get();
                        if (__all(v != PAIR_POISON && vi != PAIR_POISON)) break;
                        if (*(volatile int *)&verdict) break;
                        if (!pair_wait(a, t0, n)) {
                            verdict = 2;
                            break;
                        }
                    }
                }
                if (real) {
                    ml[p * PL * 64 + lane] = __longlong_as_double((long long)v);
                    if constexpr (CX)
                        ml[(p * 2 + 1) * 64 + lane] = __longlong_as_double((long long)vi);
                }
                loaded[i] = ver;
            }
            if (look) look_back();
            __syncthreads();
            if (verdict) {  // read here only: the last wave may already look back from sweep s + 1
                leave = true;
                break;
            }
            if (turns && s > 1 && tid == 0) report(s - 1);
            typename Core::V R[NT], Ri[CX ? NT : 1];
            K.env_begin(need0, need1, R, Ri);
            if constexpr (DIRECT) {
                K.env_add(K.d, R, Ri, [&](int I, int t, double &mr, double &mi) {
                    const unsigned int o = at[I * 4 * NT + t];
                    const double *x = ml + (o & 0xffffu), *y = ml + (o >> 16);
                    if constexpr (CX) {
                        const double xr = x[0], xi = x[64], yr = y[0], yi = y[64];
                        mr = xr * yr - xi * yi;
                        mi = xr * yi + xi * yr;
                    } else {
                        mr = x[0] * y[0];
                    }
                });
            } else {
                if (need0) K.kron(0);
                if (need1) K.kron(1);
                __syncthreads();
                K.env_add(K.d, R, Ri, K.staged());
                __syncthreads();
            }
            K.env_store(R, Ri);
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int p = w + i * W;
                if (p >= 4) break;
                const int q = rec.slot[p];
                if (q < 0 || !((mask >> p) & 1)) continue;
                const bool real = lane < rec.dim[p] * rec.dim[p];
                const typename Core::Entry y = Core::normalise(real, K.open(p, where[i]));
                const long long o = (rec.out[p] + lane) * PL;
                pair_settle();  // the poison of version s, stored a sweep ago
                if (real) {
                    unsigned long long *out = a.ring + (s % PAIR_RING) * a.nm + o;
                    unsigned long long *ahead = a.ring + ((s + 2) % PAIR_RING) * a.nm + o;
                    auto put = [&](unsigned long long *to, double z) {
                        unsigned long long v = (unsigned long long)__double_as_longlong(z);
                        if (v == PAIR_POISON) v |= PAIR_QUIET;
                        __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    };
                    put(out, y.re);
                    if constexpr (CX) put(out + 1, y.im);
                    __hip_atomic_store(ahead, PAIR_POISON, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                    if constexpr (CX)
                        __hip_atomic_store(ahead + 1, PAIR_POISON, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                }
                double *mine = own + p * PL * 64 + lane;
                double xo = mine[0], xoi = 0.0, fid, mx;
                mine[0] = y.re;
                if constexpr (CX) {
                    xoi = mine[64];
                    mine[64] = y.im;
                }
                Core::residual(y.re, y.im, xo, xoi, fid, mx);
                if (lane == 0) {
                    double *r = a.res + (long long)(s % PAIR_RING) * 2 * a.nports + q;
                    r[0] = fid;
                    r[a.nports] = mx;
                    fm = fold_max(fm, a.crit ? mx : fid);
                }
            }
            if (lane == 0) fold_m[w] = fm;
            // ml is free again; a Jacobi run goes on in its other set, and to the environments
            // only past the next barrier
            if (!turns) __syncthreads();
        }
        if (leave) break;
        if (!turns && tid == 0) {
            report(s);
            pair_settle();
            __hip_atomic_fetch_add(&a.ctrl[(long long)(s - 1) * PAIR_CTRL_LINES +
                                           ri % PAIR_CTRL_LINES].cnt,
                                   1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __syncthreads();
    if (turns && !verdict && tid == 0) report(a.sweeps);
    const bool lead = ri == 0;
    if (w == 0) {
        bool bail = verdict == 2;
        double m = 0.0;
        if (!bail && verdict == 1) {
            stop = s - back;
            m = pair_delta(a, stop, lane);
        } else if (!bail) {
            if (turns && lane == 0) {
                pair_settle();
                __hip_atomic_fetch_add(&a.ctrl[(long long)(a.sweeps - 1) * PAIR_CTRL_LINES +
                                               ri % PAIR_CTRL_LINES].cnt,
                                       1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            // the sweeps the loop has not looked at (sweep t is finished before sweep t + 1)
            if (lead || a.tol >= 0.0) {
                bail = !pair_finished(a, a.sweeps, lane, 0u);
                for (int t = max(1, a.sweeps - back + 1); t <= a.sweeps && !bail && !stop; ++t) {
                    m = pair_delta(a, t, lane);
                    if (a.tol >= 0.0 && m < a.tol) stop = t;
                }
            }
        }
        if (lane == 0) {
            stop_at = bail ? -1 : stop ? stop : a.sweeps;
            if (bail) {
                atomicOr(a.done, PAIR_RUN_BAILED);
            } else if (lead) {
                *a.delta = m;
                *a.iter = a.first + stop_at;
                if (stop) *a.at = a.first + stop;
                if (stop || a.last) atomicOr(a.done, 1);
            }
        }
    }
    __syncthreads();
    const int t = stop_at;
    if (t < 0) return;
    // a Jacobi run launch by launch checks every 16 sweeps, and the sweeps in between that it
    // skips have residual 0
    const bool cleared = a.every > 0 && (a.first + t) % a.every != 0 && a.first + t < a.maxiter;
    for (int p = w; p < 4; p += W) {  // the wave that stored them
        const int q = rec.slot[p];
        if (q < 0) continue;
        const long long o = (rec.out[p] + lane) * PL;
        if (lane < rec.dim[p] * rec.dim[p]) {
            const unsigned long long *out = a.ring + (t % PAIR_RING) * a.nm + o;
            a.dst[o] = __longlong_as_double((long long)pair_get(out));
            if constexpr (CX) a.dst[o + 1] = __longlong_as_double((long long)pair_get(out + 1));
        }
        if (lane == 0) {
            const double *r = a.res + (long long)(t % PAIR_RING) * 2 * a.nports + q;
            a.res_fid[q] = cleared ? 0.0 : r[0];
            a.res_abs[q] = cleared ? 0.0 : r[a.nports];
        }
    }
}

// ------------------------------------------------------------------ host

static constexpr size_t PAIR_LDS_MAX = 160 * 1024 - 256;  // 256: the static fold buffer

void pair_release(PairPlan *p) {
    if (p->d_recs) (void)hipFree(p->d_recs);
    if (p->d_lead) (void)hipFree(p->d_lead);
    if (p->d_run) (void)hipFree(p->d_run);
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
    const size_t esz = dtype == PAIR_C128 ? 16 : 8;
    // Few tile columns leave few waves: share the slices between two more each.  Three columns
    // a half are six waves, which four SIMDs take in two turns; twelve are even, but take the
    // LDS of two workgroups, so only where the vertices are at most one to a CU (us a sweep of
    // a run at 16x16 D = 6: 18.4 against 14.9).
    p->split = maxd >= 2 && (p->nt <= 2 || (p->nt == 3 && p->recs.size() <= 256)) ? 2 : 1;
    p->waves = 2 * p->nt * p->split;
    int slice = 0, env = 0;
    for (const PairRec &r : p->recs) {
        const int N0 = pair_pad(r.n[0]), N1 = pair_pad(r.n[1]);
        slice = std::max(slice, pair_slice_elems(r.n[0], r.n[1]));
        env = std::max(env, p->split * pair_env_elems(N0, N1));
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
    const void *fn = dtype == PAIR_F64 ? pair_fn<PAIR_F64>(p->nt) : pair_fn<PAIR_C128>(p->nt);
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
    return pair_go<PAIR_C128>(p, st, sites, src, dst, ctl, rf, ra, fold, items, n, zv);
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

// ------------------------------------------------------------------ runs

template <int TY>
static const void *pair_run_fn(int nt) {
    switch (nt) {
        case 1: return (const void *)k_pair_run<TY, 1>;
        case 2: return (const void *)k_pair_run<TY, 2>;
    }
    if constexpr (TY == PAIR_C128) return nullptr;
    else return nt == 3 ? (const void *)k_pair_run<TY, 3> : (const void *)k_pair_run<TY, 4>;
}

static const void *pair_run_any(const PairPlan *p) {
    return p->dtype == PAIR_F64 ? pair_run_fn<PAIR_F64>(p->nt) : pair_run_fn<PAIR_C128>(p->nt);
}

static size_t pair_run_lds(const PairPlan *p) {
    // a second set of messages, the outgoing ones, and the zeros of each set
    return p->lds_bytes + sizeof(double) * (2 * 4 * 64 * (p->dtype == PAIR_C128 ? 2 : 1) + 2 * 128);
}

bool pair_run_ready(PairPlan *p, int nnet, long long nmsg, int nports) {
    if (p->run_state != 0) return p->run_state > 0;
    p->run_state = -1;
    const void *fn = pair_run_any(p);
    const size_t lds = pair_run_lds(p);
    int maxd = 0;
    for (const PairRec &r : p->recs) maxd = std::max(maxd, r.d);
    if (!fn || nnet != 1 || !p->covers || maxd > p->chunk || lds > PAIR_LDS_MAX) return false;
    int dev = 0, cus = 0, per = 0;
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)PAIR_LDS_MAX) !=
            hipSuccess ||
        hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, 64 * p->waves, lds) != hipSuccess)
        return false;
    if ((long long)p->recs.size() > (long long)per * cus) return false;
    std::vector<int> steps(4 * p->recs.size(), 0);
    for (size_t i = 0; i < p->recs.size(); ++i)
        for (int t = 0; t < 4; ++t)
            if (p->recs[i].slot[t] >= 0) steps[4 * i] |= 1 << t;
    const size_t pl = p->dtype == PAIR_C128 ? 2 : 1, sb = sizeof(int) * steps.size();
    p->run_nm = (long long)pl * nmsg;
    p->run_nports = nports;
    // one allocation: ring, residuals, counters, schedules
    const size_t ring = sizeof(double) * PAIR_RING * (size_t)p->run_nm;
    const size_t res = sizeof(double) * 2 * PAIR_RING * (size_t)nports;
    const size_t ctrl = sizeof(PairCtrl) * PAIR_CTRL_LINES * PAIR_RUN_SWEEPS;
    const size_t at_ctrl = (ring + res + 63) / 64 * 64;
    char *base = nullptr;
    if (hipMalloc((void **)&base, at_ctrl + ctrl + 2 * sb) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    p->d_run = base;
    p->d_ring = base;
    p->d_ring_res = (double *)(base + ring);
    p->d_ctrl = base + at_ctrl;
    p->d_steps[0] = (int *)(base + at_ctrl + ctrl);
    p->d_steps[1] = (int *)(base + at_ctrl + ctrl + sb);
    if (hipMemcpy(p->d_steps[0], steps.data(), sb, hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    p->run_state = 1;
    return true;
}

bool pair_run_paused(PairPlan *p) {
    if (p->run_pause == 0) return false;
    --p->run_pause;
    return true;
}

void pair_run_ended(PairPlan *p, bool gave_up) {
    p->run_next = gave_up ? std::min(2 * std::max(p->run_next, 1), 1 << 20) : 0;
    p->run_pause = p->run_next / 2;
}

int pair_run_steps(PairPlan *p, hipStream_t st, const std::vector<int> &steps) {
    if (steps.size() != 4 * p->recs.size()) return 1;
    return hipMemcpyAsync(p->d_steps[1], steps.data(), sizeof(int) * steps.size(),
                          hipMemcpyHostToDevice, st) == hipSuccess ? 0 : 2;
}

int pair_run(const PairPlan *p, hipStream_t st, bool sequential, const void *sites,
             const void *src, void *dst, int *done, int *iter, int *at, double *delta,
             double *res_fid, double *res_abs, const RunParams &rp, int first, int sweeps,
             int wait_us) {
    if (p->run_state <= 0 || sweeps < 1 || sweeps > PAIR_RUN_SWEEPS) return 1;
    PairRunArgs a{};
    a.ring = (unsigned long long *)p->d_ring;
    a.nm = p->run_nm;
    a.dst = (double *)dst;
    a.ctrl = (PairCtrl *)p->d_ctrl;
    a.res = p->d_ring_res;
    a.res_fid = res_fid;
    a.res_abs = res_abs;
    a.done = done;
    a.iter = iter;
    a.at = at;
    a.delta = delta;
    a.tol = rp.tol;
    a.crit = rp.crit;
    a.sweeps = sweeps;
    a.first = first;
    a.last = first + sweeps >= rp.maxiter;
    a.nports = p->run_nports;
    a.nrec = (int)p->recs.size();
    a.split = p->split;
    a.slice_elems = p->slice_elems;
    a.env_elems = p->env_elems;
    a.chunk = p->chunk;
    a.every = sequential ? 0 : RUN_CHUNK;
    a.maxiter = rp.maxiter;
    a.ticks = 100ll * wait_us;
    a.looks = wait_us < 1000 ? 0 : 15;  // a look takes about 0.7 us
    const long long n = std::max(a.nm, (long long)sweeps * PAIR_CTRL_LINES);
    hipLaunchKernelGGL(k_pair_run_init, dim3((unsigned)std::min<long long>((n + 255) / 256, 1024)),
                       dim3(256), 0, st, (const unsigned long long *)src, a);
    const int4 *steps = (const int4 *)p->d_steps[sequential ? 1 : 0];
    const double *s64 = (const double *)sites;
    void *args[] = {(void *)&p->d_recs, &steps, &s64, &a};
    if (hipGetLastError() != hipSuccess) return 2;
    return hipLaunchKernel(pair_run_any(p), dim3(a.nrec), dim3(64 * p->waves), args,
                           pair_run_lds(p), st) == hipSuccess ? 0 : 2;
}
