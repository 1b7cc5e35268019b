// Adjoint (reverse-mode) chain of chi2 for the profile path on the real, even
// spectrum.  galario has no gradient; this differentiates its arithmetic:
//
//   V  = sgn(Z) A e^{i theta},  A = sum_k b_k |y_k|,  Z = sum_k b_k y_k
//        (y_k the four real corners, b_k the bilinear weights), theta =
//        2 pi (u dRA + v dDec) (the rotated form urot dRArot + vrot dDecrot
//        is the same number in exact arithmetic, so d theta/dPA = 0)
//   chi2 = sum w |V - O|^2,  G = dchi2/dV = 2 w (V - O)
//   dchi2/dA     = sgn(Z) Re(conj(G) e^{i theta})
//   dchi2/dtheta = Im(G) Re(V) - Re(G) Im(V)
//   dchi2/dy_k   = dchi2/dA b_k sgn(y_k)          (the phase of a real Z is
//                                                  locally constant)
//   PA moves the sampling point: dq/durot = s/duv, dt/dvrot = v_origin s/duv,
//   durot/dPA = -vrot, dvrot/dPA = urot.
//
// The corner gradients are scattered with FP64 atomics into Hh, the adjoint
// of the half spectrum H (both mirror rows of a frequency land on the same
// element, which is the adjoint of reading H at |r - N/2|).  The two passes
// are then transposed: each is sum_k c[k] cos(2 pi k m / N) over an even
// sequence, so its adjoint is the same even-real transform of the weighted
// even extension (weight 1/2 on interior input frequencies) times the
// multiplicity of each output index (1 at 0 and N/2, 2 elsewhere).  The row
// adjoint ends in the sweep adjoint: every pixel feeds I[iR] with weight
// sr (1 - alpha) and I[iR+1] with sr alpha, and inc through dr/dinc =
// (x/cos inc)^2 tan(inc) / r; the central pixel is linear in I[0..iIN+1].
#pragma once

#include <climits>

#include "gl_kernels.hpp"

namespace gl {

__device__ __forceinline__ void atomic_add_f64(double* p, double v) { unsafeAtomicAdd(p, v); }

// ---------------------------------------------------------------------------
// sample + its adjoint: chi2 and (PA, dRA, dDec) partials per workgroup,
// corner gradients scattered into Hh.
//
// Global FP64 atomics on gfx950 are resolved beyond the per-XCD L2, one request per 64-byte line and wave
// instruction, at 17 G requests/s, and atomics on one address serialise: with log-uniform
// baselines ~10% of all points fall in the few cells around the origin.  Each workgroup
// therefore first accumulates its corner gradients in LDS:
//   * in a window over the bounding box of its cells when that holds at most WIN cells (points are
//     stored in a locality order, so where they are dense it does), flushed with one atomic per
//     non-zero cell;
//   * otherwise in a table of the 64-byte lines of Hh that its points touch (open addressing in the
//     same LDS), flushed with one request per line.  256 sparse points touch 200 to 500 lines with their
//     1.9 lines each, so the table takes a third to a half off the requests: on 64 sets of parameters
//     and datasets of 5e5 / 1.5e6 / 3e6 points at nxy = 4096 the kernel takes 0.79 / 1.6 / 2.6 ms, against
//     0.95 / 2.1 / 3.6 ms with every corner of a sparse point sent to memory.
// Cells with column < GHOT and folded row < GHOT do not go to Hh but to one of GREP replicas of that
// tile (by workgroup index), which the adjoint column pass folds into Hh.
//
// What bounds it: those requests and, where the points are dense, vector instruction issue (about
// 260 instructions per 64 points with GPT 2, 417 with 1; 650 before).  A thread takes GPT points: the bounding box, the
// window's clearing and flush and the wave reductions are paid once per GPT points.
// ---------------------------------------------------------------------------
constexpr int GHOT = 16;          // hot tile: columns [0, GHOT) x folded rows [0, GHOT)
constexpr int GREP = 32;          // replicas of the hot tile in global memory
constexpr int GWIN = 3072;        // LDS window capacity (cells): 6 workgroups per CU
                                  // (the single call's; the batched form's autotuner also tries 2048 and 4096)
constexpr int GHOT_ELEMS = GREP * GHOT * GHOT;
template <typename T>
struct GradArgs {
    double* Hh;          // adjoint of H, same layout (h_index, ldH), zero on entry
    double* hot;         // GREP x GHOT x GHOT replicas [rep][col][row], zero on entry
    double* partials;    // 4 streams of partials per block of 256 points: chi2, dPA, ddRA, ddDec
    int ldp;             // stride between the streams (>= number of blocks)
    int nblk;            // blocks of 256 points
    int direct;          // sparse points: 1 straight to Hh, 0 through the line table
};

__device__ __forceinline__ void lds_add_f64(double* p, double v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ double xor_sign(double x, double s) {   // x with its sign flipped where s is negative
    return __hiloint2double(__double2hiint(x) ^ (__double2hiint(s) & int(0x80000000u)), __double2loint(x));
}

// The same at a byte offset below 2^32 from a uniform base (Hh holds less than 2^30 bytes).
__device__ __forceinline__ void atomic_add_at(double* base, unsigned bytes, double v) {
    atomic_add_f64(reinterpret_cast<double*>(reinterpret_cast<char*>(base) + size_t(bytes)), v);
}

// Slot of a line in a table of NLINE keys (0xFFFFFFFF: free), entered if it is not there; -1 when eight
// probes find no place.  Several lanes may look for the same or for colliding lines at once.
template <int NLINE>
__device__ __forceinline__ int line_slot(unsigned* keys, unsigned line) {
    unsigned h = __umulhi(line * 2654435769u, unsigned(NLINE));
    int slot = -1;
#pragma unroll 1
    for (int probe = 0; probe < 8 && slot < 0; ++probe) {
        const unsigned was = atomicCAS(&keys[h], 0xFFFFFFFFu, line);
        if (was == 0xFFFFFFFFu || was == line) slot = int(h);
        h = h + 1 < unsigned(NLINE) ? h + 1 : 0u;
    }
    return slot;
}

// One point's reverse mode (all in double).
struct GradPoint {
    int iu, d;           // cell (SymPoint); iu = -1: nothing to add
    double g[4];         // gradients of corners (iu, |d|), (iu, |d + 1|), (iu + 1, |d|), (iu + 1, |d + 1|)
};

// x times the sign of y (0 for y = 0)
__device__ __forceinline__ double times_sign(double x, double y) {
    const int one = (__double2hiint(y) & int(0x80000000u)) | 0x3FF00000;
    return x * __hiloint2double(y == 0.0 ? 0 : one, 0);
}

// Storage T (H and the dataset streams of `a`), arithmetic P with the scalars of `sc` (P = T, sc = a:
// galario's arithmetic in that precision; T = float, P = double: the FP32-bulk form with FP64
// per-point arithmetic).  The reverse mode runs in double either way.  WIN: LDS window capacity
// (cells); a larger window keeps more workgroups off the direct atomics, a smaller one leaves room
// for more workgroups per CU.  blk: workgroup, covering blocks GPT blk .. GPT blk + GPT - 1 of 256 points.
template <typename T, typename P, int WIN, int GPT>
__device__ __forceinline__ void sample_grad_sym_body(const SampleArgs<T>& a, const SampleArgs<P>& sc,
                                                     const GradArgs<T>& g, int blk) {
    static_assert(WIN % 512 == 0, "whole rounds of the workgroup over the window and the line table");
    __shared__ __align__(16) double win[WIN];
    constexpr int NLINE = WIN / 8;           // lines of the sparse points' table
    constexpr unsigned EMPTY = 0xFFFFFFFFu;
    __shared__ unsigned keys[NLINE];
    __shared__ double red[3 + GPT][16];      // per wave and row of 16 lanes
    __shared__ unsigned box[32];             // likewise: packed minima, lo and hi in turn
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    double c2[GPT], gpa = 0.0, gra = 0.0, gde = 0.0;
    GradPoint pt[GPT];
    bool oob_any = false;
    unsigned blo = 0xFFFFFFFFu, bhi = 0xFFFFFFFFu;   // packed (column pair, row) minima, and of 0xFFFF - maxima
    // (lanes beyond the data take the last point and count nothing)
    const int base = blk * (256 * GPT);
    P u0[GPT], v0[GPT], ore[GPT], oim[GPT], w[GPT];
    bool valid[GPT];
#pragma unroll
    for (int k = 0; k < GPT; ++k) {
        valid[k] = base + k * 256 + tid < a.nd;
        const unsigned i = unsigned(min(k * 256 + tid, a.nd - 1 - base)) * unsigned(sizeof(T));
        u0[k] = P(h_at(a.u + base, i));
        v0[k] = P(h_at(a.v + base, i));
        ore[k] = P(h_at(a.re + base, i));
        oim[k] = P(h_at(a.im + base, i));
        w[k] = P(h_at(a.w + base, i));
    }
    SymPoint<P> p[GPT];
    SymValues<P> y[GPT];
#pragma unroll
    for (int k = 0; k < GPT; ++k) {
        p[k] = sym_position(sc, u0[k], v0[k]);
        y[k] = sym_values<P>(a.H, a.ldH, p[k].iu, p[k].d);
    }
#pragma unroll
    for (int k = 0; k < GPT; ++k) {
        const bool oob = !p[k].in | beyond_extent(sc.ext2, u0[k], v0[k]);
        const bool live = valid[k] & !oob;
        oob_any |= valid[k] & oob;
        P cth = P(1), sth = P(0);
        if (std::is_same<P, double>::value || sc.phase) phase_factor(sc, p[k].urot, p[k].vrot, &sth, &cth);
        const P V0 = sym_amplitude(y[k], p[k].q, p[k].t);
        const P Vre = V0 * cth, Vim = V0 * sth;
        const P dre = Vre - ore[k], dim = Vim - oim[k];
        // a point outside the grid makes every sum NaN, a lane beyond the data adds nothing
        const double none = valid[k] ? double(NAN) : 0.0;
        const double term = chi2_term(weight_factor(w[k]), dre, dim);
        c2[k] = live ? term : none;
        // reverse mode in double
        const double w2 = 2.0 * double(w[k]);
        const double Gre = w2 * double(dre), Gim = w2 * double(dim);
        const double gA = xor_sign(ffma(Gre, double(cth), Gim * double(sth)), double(V0));
        const double gt = ffma(Gim, double(Vre), -(Gre * double(Vim)));
        const double gth = live ? gt : none;
        const double q = double(p[k].q), t = double(p[k].t);
        const double y0 = double(y[k].y0), y1 = double(y[k].y1), y2 = double(y[k].y2), y3 = double(y[k].y3);
        const double e10 = fabs(y3) - fabs(y0), e01 = fabs(y1) - fabs(y0), e11 = (fabs(y2) - fabs(y3)) - e01;
        // A's slopes in the grid position, turned into the slope in PA (the position in cells is
        // (urot, vrot) / duv, both negated for a folded point)
        const double dq = ffma(t, e11, e10), dt = ffma(q, e11, e01);
        const double gp = gA * ffma(dt, double(p[k].urot), -(dq * double(p[k].vrot)));
        const double gps = xor_sign(gp, double(p[k].urot));
        gpa += live ? gps : none;
        gra = ffma(gth, double(u0[k]), gra);
        gde = ffma(gth, double(v0[k]), gde);
        // corners: the bilinear weights times gA, with the corner's sign (0 for a corner that is 0)
        const double gq = gA * q, g0 = gA - gq;
        const double k3 = gq * t, k2 = gq - k3, k1 = g0 * t, k0 = g0 - k1;
        pt[k].iu = live ? p[k].iu : -1;
        pt[k].d = p[k].d;
        pt[k].g[0] = times_sign(k0, y0);
        pt[k].g[1] = times_sign(k1, y1);
        pt[k].g[2] = times_sign(k2, y3);
        pt[k].g[3] = times_sign(k3, y2);
        const int m0 = row_lo(p[k].d), m1 = row_hi(p[k].d);
        const unsigned lo = unsigned(p[k].iu >> 1) | (unsigned(min(m0, m1)) << 16);
        const unsigned hi = ~(unsigned((p[k].iu + 1) >> 1) | (unsigned(max(m0, m1)) << 16));
        blo = pk_min_u16(blo, live ? lo : 0xFFFFFFFFu);
        bhi = pk_min_u16(bhi, live ? hi : 0xFFFFFFFFu);
    }
    if (oob_any && a.flag) raise_flag(a.flag);
    // bounding box of the workgroup's cells, columns in pairs (the window follows h_index)
    const unsigned bx = row_pk_min2(blo, bhi, lane);
    if ((lane & 15) < 2) box[8 * wv + 2 * (lane >> 4) + (lane & 1)] = bx;
    __syncthreads();
    // the minima over the rows of all waves, as scalars: what follows from them takes no vector instructions
    unsigned kb = box[lane & 31];
    kb = pk_min_u16(kb, unsigned(dpp_i32<DPP_XOR2>(int(kb))));
    kb = pk_min_u16(kb, unsigned(dpp_i32<DPP_ROW_ROR4>(int(kb))));
    kb = pk_min_u16(kb, unsigned(dpp_i32<DPP_ROW_ROR8>(int(kb))));
    const unsigned l0 = unsigned(__builtin_amdgcn_readlane(int(kb), 0)), l1 = unsigned(__builtin_amdgcn_readlane(int(kb), 16));
    const unsigned h0 = unsigned(__builtin_amdgcn_readlane(int(kb), 1)), h1 = unsigned(__builtin_amdgcn_readlane(int(kb), 17));
    const int pmin = int(min(l0 & 0xFFFFu, l1 & 0xFFFFu)), mmin = int(min(l0 >> 16, l1 >> 16));
    const int pmax = 0xFFFF - int(min(h0 & 0xFFFFu, h1 & 0xFFFFu)), mmax = 0xFFFF - int(min(h0 >> 16, h1 >> 16));
    const bool any = pmin <= pmax;                   // (no live point: 0xFFFF and 0)
    const int wp = pmax - pmin + 1, w2 = 2 * (mmax - mmin + 1);
    const bool use_win = any && wp * w2 <= WIN;      // (wp <= 2^12 + 1, w2 <= 2^14 + 2: no overflow)
    const int nwin = use_win ? wp * w2 : 0;          // even
    const int nclear = use_win ? nwin : GPT == 1 && g.direct ? GHOT * GHOT : WIN;
    for (int j = 2 * tid; j < nclear; j += 512)
        *reinterpret_cast<cpx<double>*>(&win[j]) = cpx<double>{0.0, 0.0};
    double* rep = g.hot + size_t(blk % GREP) * (GHOT * GHOT);
    __syncthreads();
    if (use_win) {
        // LDS additions.  Neighbouring lanes (points in locality order) often lie in the same
        // cell: lanes l and l ^ 1, then l and l ^ 2, of one cell add their four corner values into the
        // lower lane first (DPP moves), which halves to quarters the same-address LDS atomics where
        // the points are dense.  key: the cell, -1: nothing to add (iu = -1).
        const int c0 = -(pmin * w2 + 2 * mmin);
#pragma unroll
        for (int k = 0; k < GPT; ++k) {
            int key = pt[k].iu < 0 ? -1 : pt[k].iu * 32768 + (pt[k].d + 8192);
            double x0 = pt[k].g[0], x1 = pt[k].g[1], x2 = pt[k].g[2], x3 = pt[k].g[3];
            // (a lane with nothing to add may hold a NaN, which a factor of 0 would pass on)
            if (__ballot(key < 0) != 0) {
                x0 = key < 0 ? 0.0 : x0;
                x1 = key < 0 ? 0.0 : x1;
                x2 = key < 0 ? 0.0 : x2;
                x3 = key < 0 ? 0.0 : x3;
            }
            {
                const bool same = key == dpp_i32<DPP_XOR1>(key);
                const double f = same ? 1.0 : 0.0;
                x0 = ffma(dpp_f64<DPP_XOR1>(x0), f, x0);
                x1 = ffma(dpp_f64<DPP_XOR1>(x1), f, x1);
                x2 = ffma(dpp_f64<DPP_XOR1>(x2), f, x2);
                x3 = ffma(dpp_f64<DPP_XOR1>(x3), f, x3);
                key = same && (lane & 1) ? -1 : key;
            }
            {
                const bool same = key == dpp_i32<DPP_XOR2>(key);
                const double f = same ? 1.0 : 0.0;
                x0 = ffma(dpp_f64<DPP_XOR2>(x0), f, x0);
                x1 = ffma(dpp_f64<DPP_XOR2>(x1), f, x1);
                x2 = ffma(dpp_f64<DPP_XOR2>(x2), f, x2);
                x3 = ffma(dpp_f64<DPP_XOR2>(x3), f, x3);
                key = same && (lane & 2) ? -1 : key;
            }
            if (key >= 0) {
                const int iu = pt[k].iu, d = pt[k].d;
                const int o0 = c0 + __mul24(iu >> 1, w2) + (iu & 1) + 2 * row_lo(d);
                const int o2 = o0 + (iu & 1 ? w2 - 1 : 1);
                const int dm = d >= 0 ? 2 : -2;
                lds_add_f64(&win[o0], x0);
                lds_add_f64(&win[o0 + dm], x1);
                lds_add_f64(&win[o2], x2);
                lds_add_f64(&win[o2 + dm], x3);
            }
        }
    } else if (GPT == 1 && g.direct) {
        // Sparse points of a small call: straight to Hh, a point's four corners by a lane quad (they lie in one
        // 32-byte run when the lower column is even, h_index): in round r, lane l carries corner l & 3 of point
        // (l >> 2) + 16 r of its wave.  Cells of the hot tile are summed in LDS first.
        const int corner = lane & 3;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int src = (lane >> 2) + 16 * r;
            const int iu = __shfl(pt[0].iu, src, 64), d = __shfl(pt[0].d, src, 64);
            const double x0 = __shfl(pt[0].g[0], src, 64), x1 = __shfl(pt[0].g[1], src, 64);
            const double x2 = __shfl(pt[0].g[2], src, 64), x3 = __shfl(pt[0].g[3], src, 64);
            const double xl = corner & 1 ? x1 : x0, xh = corner & 1 ? x3 : x2;
            const double x = corner & 2 ? xh : xl;
            const int col = iu + (corner >> 1), m = corner & 1 ? row_hi(d) : row_lo(d);
            if (iu >= 0 && x != 0.0) {
                if (col < GHOT && m < GHOT) lds_add_f64(&win[col * GHOT + m], x);
                else atomic_add_f64(g.Hh + h_index(col, m, a.ldH), x);
            }
        }
        __syncthreads();
        static_assert(GHOT * GHOT == 256, "one cell per thread");
        if (win[tid] != 0.0) atomic_add_f64(rep + tid, win[tid]);
    } else {
        // Sparse points: a table of 64-byte lines of Hh (2 columns x 4 rows, h_index), open addressing,
        // built and flushed for one block of 256 points at a time.
        for (int k = 0; k < GPT; ++k) {
            GradPoint p = pt[0];          // (shadows the positions, which are done with)
#pragma unroll
            for (int j = 1; j < GPT; ++j)
                if (j == k) p = pt[j];
            for (int j = tid; j < NLINE; j += 256) keys[j] = EMPTY;
            __syncthreads();
            if (p.iu >= 0) {
                const int m0 = row_lo(p.d), m1 = row_hi(p.d);
                const unsigned ld4 = unsigned(a.ldH) >> 2;
                const unsigned p0 = unsigned(p.iu >> 1) * ld4, p1 = unsigned((p.iu + 1) >> 1) * ld4;
                const unsigned r0 = unsigned(m0 >> 2), r1 = unsigned(m1 >> 2);
                const int e0 = 2 * (m0 & 3), e1 = 2 * (m1 & 3), o0 = p.iu & 1, o1 = o0 ^ 1;
                const int s00 = line_slot<NLINE>(keys, p0 + r0);
                const int s01 = r1 == r0 ? s00 : line_slot<NLINE>(keys, p0 + r1);
                int s10 = s00, s11 = s01;
                if (p1 != p0) {
                    s10 = line_slot<NLINE>(keys, p1 + r0);
                    s11 = r1 == r0 ? s10 : line_slot<NLINE>(keys, p1 + r1);
                }
                const auto add = [&](int slot, int e, int col, int m, double x) {
                    if (slot >= 0) lds_add_f64(&win[8 * slot + e], x);
                    else if (col < GHOT && m < GHOT) atomic_add_f64(rep + col * GHOT + m, x);
                    else atomic_add_f64(g.Hh + h_index(col, m, a.ldH), x);
                };
                add(s00, e0 + o0, p.iu, m0, p.g[0]);
                add(s01, e1 + o0, p.iu, m1, p.g[1]);
                add(s10, e0 + o1, p.iu + 1, m0, p.g[2]);
                add(s11, e1 + o1, p.iu + 1, m1, p.g[3]);
            }
            __syncthreads();
            // eight lanes per line: element e of line `key` is Hh[8 key + e] (a line with a non-zero element has
            // a key); FB rounds' LDS reads together, more than which cost registers (4: 7.5 against 7.07 ms)
            const unsigned ld4 = unsigned(a.ldH) >> 2;
            constexpr int FB = 2;
            static_assert(8 * NLINE % (256 * FB) == 0, "whole rounds");
#pragma unroll 1
            for (int j0 = tid; j0 < 8 * NLINE; j0 += 256 * FB) {
                unsigned key[FB];
                double x[FB];
#pragma unroll
                for (int h = 0; h < FB; ++h) {
                    key[h] = keys[(j0 >> 3) + 32 * h];
                    x[h] = win[j0 + 256 * h];
                }
#pragma unroll
                for (int h = 0; h < FB; ++h) {
                    if (k + 1 < GPT) win[j0 + 256 * h] = 0.0;
                    if (x[h] != 0.0) {
                        const unsigned e = unsigned(tid) & 7u;
                        if (key[h] < unsigned(GHOT / 2) * ld4) {
                            const unsigned cp = key[h] / ld4, r = key[h] - cp * ld4;
                            if (r < unsigned(GHOT / 4)) {
                                atomic_add_f64(rep + (2 * cp + (e & 1)) * GHOT + 4 * r + (e >> 1), x[h]);
                                continue;
                            }
                        }
                        atomic_add_at(g.Hh, (8u * key[h] + e) * 8u, x[h]);
                    }
                }
            }
            __syncthreads();
        }
    }
    if (use_win) {
        __syncthreads();
        // window cell j = cp * w2 + 2 mm + (column & 1) is Hh offset ((pmin + cp) ldH + mmin) * 2 + j - cp * w2
        // (consecutive j, consecutive addresses); cp from a float reciprocal (exact after one
        // correction, j < 2^24)
        const float inv_w2 = 1.0f / float(w2);
        for (int j = tid; j < nwin; j += 256) {
            const double x = win[j];
            if (x != 0.0) {
                int c = int(float(j) * inv_w2);
                c += (c + 1) * w2 <= j;
                c -= c * w2 > j;
                const int o = j - c * w2, cp = pmin + c, m = mmin + (o >> 1);
                if (cp < GHOT / 2 && m < GHOT) atomic_add_f64(rep + (2 * cp + (o & 1)) * GHOT + m, x);
                else atomic_add_at(g.Hh, unsigned(2 * (cp * a.ldH + mmin) + o) * 8u, x);
            }
        }
    }
    // partials of chi2 per block of 256 points (the forward kernels' order, so the gradient call's chi2
    // equals the forward call's bit for bit), of dPA, ddRA, ddDec per workgroup (the scale factors
    // 1 / duv and 2 pi applied to the sums), stored with the first block
    const int row = 4 * wv + (lane >> 4);
    const double sums[4] = {c2[0], gpa, gra, gde};
    const double sum = joint_row_sums<4>(sums, lane);
    if ((lane & 15) < 4) red[lane & 3][row] = sum;
#pragma unroll
    for (int k = 1; k < GPT; ++k) {
        const double y = row_sum(c2[k]);
        if ((lane & 15) == 0) red[3 + k][row] = y;
    }
    __syncthreads();
    if (tid < 4 * GPT) {
        const int st = tid & 3, k = tid >> 2, b = blk * GPT + k;
        const double* r = red[st == 0 && k > 0 ? 3 + k : st];
        double ws[4];                          // the waves' sums in wave_sum's order
#pragma unroll
        for (int w = 0; w < 4; ++w) ws[w] = (r[4 * w] + r[4 * w + 1]) + (r[4 * w + 2] + r[4 * w + 3]);
        double x = (ws[0] + ws[1]) + (ws[2] + ws[3]);
        if (st == 1) {
            if constexpr (std::is_same<P, double>::value) x *= sc.inv_duv;
            else x /= double(sc.duv);
        } else if (st > 1) {
            x *= 6.283185307179586476925286766559;
        }
        if (st != 0 && k != 0) x = 0.0;
        if (b < g.nblk) g.partials[size_t(st) * g.ldp + b] = x;
    }
}

// Points per thread.  One call (1e6 points at nxy = 4096): 1, since its 3907 workgroups take two and a half
// rounds of the chip and 1954 longer ones end with a half-empty round (77.2 against 80.2 us per gradient call);
// the batched form: 2 (7.07 against 7.45 ms with 1 and 9.3 ms with 4, whose 180 VGPRs leave two waves per
// SIMD, on 64 sets x 5e6 points).
constexpr int GPT_SINGLE = 1, GPT_BATCH = 2;
// Batched launches of at most this many one-point workgroups take one point per thread too.
constexpr size_t GRAD_FEW_WORKGROUPS = 8192;
// Launches of at most this many workgroups add their sparse points straight to Hh: all of them are resident at once, so
// the launch takes one workgroup's latency, to which the line table's building and flush add 2 to 4 us, while the
// atomics' rate does not bind yet.  The kernel, direct against table: nxy = 4096, 8000 points 4.9 / 8.4 us, 64000 7.1 / 8.4,
// 128000 11.1 / 10.2, 256000 14.4 / 13.0; nxy = 1024, 8000 4.4 / 9.4, 128000 6.2 / 9.4.  The gradient call at 131000
// points: nxy = 1024 32.3 / 34.6 us, 2048 37.0 / 38.9, 4096 56.1 / 55.2, 8192 128.1 / 130.3.  (At 4096 the two meet at
// 90000 points, 350 workgroups, and the table would save 0.9 us of the call at 512; a lower line would cost the other
// sizes 2 us.)
constexpr int GRAD_DIRECT_BLOCKS = 512;
template <typename T>
__global__ __launch_bounds__(256) void k_sample_grad_sym(SampleArgs<T> a, GradArgs<T> g) {
    sample_grad_sym_body<T, T, GWIN, GPT_SINGLE>(a, a, g, blockIdx.x);
}

// Destinations of the 4 partial streams (chi2, dPA, ddRA, ddDec).
struct Dst4 {
    double* d[4];
};

// ---------------------------------------------------------------------------
// adjoint of the column pass: Hh (two columns per workgroup) -> Th[m][l],
// m = 0..Rs'; Hh is set back to zero after it is read.
// ---------------------------------------------------------------------------
template <typename T>
struct AdjColArgs {
    double* Hh;
    double* hot;         // GREP replicas of the hot tile, added to Hh columns < GHOT, rows < GHOT
    int ldH;
    int N, Rs;           // Rs': outputs m = 0..Rs'
    const cpx<T>* tw;
    T* Th;               // row-major [Rs'+1][ldTh]
    int ldTh;
    const double* part;  // optional: 4 streams of np partials (stride np), each summed into dst by one of
    int np;              // 8 extra workgroups after the nfft FFT workgroups
    Dst4 dst;
    int nfft;
    double rc2;          // > 0: Hh is zero beyond the store radius sqrt(rc2) (stored_rows)
    const cpx<T>* tw512; // W_512^e table (k_adjcol_sub)
};

// Deterministic sum *dst = sum_i p[i] of n partials in the order of
// k_sum_partials (1024 virtual threads, thread t summing p[t], p[t + 1024],
// ...; the 16 virtual waves' sums added in order), so chi2 equals the forward
// call's bit for bit; run by one workgroup of NT threads, NT a multiple of 64:
// real wave w plays virtual waves w, w + NT/64, ... (below 16), lane for lane.
template <int NT>
__device__ __forceinline__ void sum_partials_in_block(const double* __restrict__ p, int n, double* dst,
                                                      double* red16) {
    static_assert(NT % 64 == 0 && NT <= 1024, "whole waves");
    constexpr int NW = NT / 64;
    constexpr int V = (16 + NW - 1) / NW;     // virtual waves per real wave (the last ones may be beyond 16)
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    double acc[V];
#pragma unroll
    for (int q = 0; q < V; ++q) {
        const int vw = wv + q * NW;
        acc[q] = vw < 16 ? sum_stride1024(p, vw * 64 + lane, n, 0.0) : 0.0;
    }
#pragma unroll
    for (int q = 0; q < V; ++q) {
        const int vw = wv + q * NW;
        const double x = wave_sum(acc[q]);
        if (vw < 16 && lane == 0) red16[vw] = x;
    }
    __syncthreads();
    if (t == 0) {
        double s = 0.0;
        for (int w = 0; w < 16; ++w) s += red16[w];
        if (dst) *dst = s;
    }
}

__device__ __forceinline__ double mult(int m, int N) { return (m == 0 || m == N / 2) ? 1.0 : 2.0; }
__device__ __forceinline__ double ext_weight(int k, int N) { return (k == 0 || k == N / 2) ? 1.0 : 0.5; }

// Sums of the hot tile's replicas over columns la, la + 1 (hs[0], hs[1]), rows 0..GHOT-1, by the first
// NT' = 2^k <= NT threads of a workgroup; each replica element is read by one thread, all its loads in flight
// together, and set back to zero.  (32 reads one after the other per element made the eight
// workgroups of the hot columns the last to finish: nxy = 512, 5003 points: 6.1 against 4.3 us for the pass.)
// The caller's barrier orders hs before its use.
template <int NT>
__device__ __forceinline__ void fold_hot(double* hot, int la, double (*hs)[GHOT]) {
    constexpr int TP = NT >= 1024 ? 32 : NT >= 512 ? 16 : NT >= 256 ? 8 : NT >= 128 ? 4 : 2;   // threads per element
    constexpr int PER = GREP / TP;
    const int tid = threadIdx.x;
    if (tid >= 2 * GHOT * TP) return;          // (whole waves)
    const int part = tid % TP, el = tid / TP, c = el / GHOT, p = el % GHOT;
    double x[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) x[j] = hot[((part * PER + j) * GHOT + la + c) * GHOT + p];
    double sum = 0.0;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        sum += x[j];
        hot[((part * PER + j) * GHOT + la + c) * GHOT + p] = 0.0;
    }
#pragma unroll
    for (int d = 1; d < TP; d *= 2) sum += __shfl_xor(sum, d, 64);
    if (part == 0) hs[c][p] = sum;
}

// PARTIALS: workgroups blk >= nfft sum the sample kernel's partial streams
// (the batched form sums them in its own reduction kernel).
template <typename T, int LOG2N, bool PARTIALS = true, bool SPLIT = true>
__device__ __forceinline__ void adjcol_sym_body(const AdjColArgs<T>& a, int blk, int nblk) {
    using S = FftShape<LOG2N>;
    using F = BlockFft<T, LOG2N, false, SPLIT>;
    constexpr int N = S::N, NT = S::NT, E = S::E;
    constexpr int C = N / 2 + 1;
    constexpr int NPAIR = (C + 1) / 2;
    __shared__ T lds[F::LDS_REALS];
    if (PARTIALS && blk >= a.nfft) {        // extra workgroups: the partial sums of the sample kernel
        const int j = blk - a.nfft;
        __shared__ double red16[16];
        if (a.part && j < 4) sum_partials_in_block<NT>(a.part + size_t(j) * a.np, a.np, a.dst.d[j], red16);
        return;
    }
    const int pair = xcd_column(blk, a.nfft);
    if (pair >= NPAIR) return;
    const int la = 2 * pair, lb = la + 1;
    const bool has_b = lb < C;
    const int tid = threadIdx.x;
    cpx<double>* hab = reinterpret_cast<cpx<double>*>(a.Hh + h_index(la, 0, a.ldH));   // columns la, lb (h_index)
    const bool hot_cols = la < GHOT;   // GHOT is even: lb < GHOT too
    // rows the sample kernel can have touched (column lb: no more); beyond them Hh, and the
    // replicas of the hot tile, hold zeros
    const int kc = stored_rows(a.rc2, la, N);
    if (kc < 0) return;                // (the adjoint row pass reads no frequency of these columns)
    __shared__ double hs[2][GHOT];
    if (hot_cols) {
        fold_hot<NT>(a.hot, la, hs);
        __syncthreads();
    }
    unsigned touched = 0;              // bit r: row tid + r NT holds a value, in this lane or its quad
    cpx<T> v[E];
    F::run(v, lds, tid, N / 2, a.tw, [&](int k) -> cpx<T> {
        const int p = k <= N / 2 ? k : N - k;
        const double wk = ext_weight(k, N);
        const cpx<double> x = p <= kc ? hab[p] : cpx<double>{0.0, 0.0};
        if (k <= N / 2) touched |= unsigned((x.re != 0.0) | (x.im != 0.0)) << (k / NT);
        double xa = x.re, xb = has_b ? x.im : 0.0;
        if (hot_cols && p < GHOT) {
            xa += hs[0][p];
            xb += hs[1][p];
        }
        return cpx<T>{T(wk * xa), T(wk * xb)};
    }, a.Rs < NT);        // outputs m <= Rs' only
    // all reads of Hh are done (the FFT synchronised after its first pass): clear it for the next call, by 64-byte
    // lines (four lanes) that hold a value (64 sets x 5e6 points: 6.99 -> 6.93 ms; the residue form, whose
    // workgroups all clear at once, gains nothing from it)
    touched |= unsigned(dpp_i32<DPP_XOR1>(int(touched)));
    touched |= unsigned(dpp_i32<DPP_XOR2>(int(touched)));
#pragma unroll
    for (int r = 0; r <= E / 2; ++r)                          // (slot lb of the last pair: padding)
        if ((touched >> r & 1u) && tid + r * NT <= kc) hab[tid + r * NT] = cpx<double>{0.0, 0.0};
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int m = tid + r * NT;
        if (r * NT <= a.Rs && m <= a.Rs) {
            const T cm = T(mult(m, N));
            T* o = a.Th + size_t(m) * a.ldTh + la;
            o[0] = cm * v[r].re;
            if (has_b) o[1] = cm * v[r].im;
        }
    }
}

template <typename T, int LOG2N>
__global__ __launch_bounds__(FftShape<LOG2N>::NT) void k_adjcol_sym(AdjColArgs<T> a) {
    adjcol_sym_body<T, LOG2N>(a, blockIdx.x, gridDim.x);
}

// Few workgroups: as k_colpass_sym_few.
template <typename T, int LOG2N>
__global__ __launch_bounds__(FftShape<LOG2N>::NT) void k_adjcol_sym_few(AdjColArgs<T> a) {
    adjcol_sym_body<T, LOG2N, true, false>(a, blockIdx.x, gridDim.x);
}

// Residue form of the adjoint column pass (N >= 1024, profile within 255 pixels: Rs' <= 256; the single
// call's: a shorter path per workgroup and 84 instead of 166 VGPRs, so all of one call's workgroups are
// resident at once, +2-3% on the gradient call; the batched form, bound by throughput, keeps the full
// transform).  Its
// outputs are rows m = 0..Rs' of the N-point transform of the even extension z[k] = w_k x[fold(k)]
// of a column pair of Hh.  With Y_k0 the 512-point transform of z[k0 + P K] (P = N / 512),
//   Z[m] = sum over k0 = 0..P/2 of  W_N^(m k0) Y_k0[m]  +  W_N^(-m k0) Y_k0[512 - m],
// the second term for k0 other than 0 and P/2: it is residue P - k0, whose sequence is residue k0's
// reversed (z is even).  One wave per residue k0: its 512-point transform (ResidueFft at k0 = 0) leaves
// Y[lane + 64 s] in v[s], and Y[512 - m] of m = lane + 64 s sits in lane 64 - lane, slot 7 - s (lane 0:
// its own slot 8 - s).  The column pair is staged in LDS, real parts then imaginary parts, for the
// waves' strided gathers (row p at p + p/8: rows P apart fall in different banks) and cleared as soon
// as it is read; the waves' terms are summed in LDS in residue order.
template <typename T, int LOG2N>
__device__ __forceinline__ void adjcol_sub_body(const AdjColArgs<T>& a, int blk) {
    using CS = ResidueShape<LOG2N>;
    using F = ResidueFft<T>;
    constexpr int N = CS::N, P = CS::P, NT = CS::NT, NK = CS::NK;
    constexpr int C = N / 2 + 1, NPAIR = (C + 1) / 2;
    constexpr int PER = (C + NT - 1) / NT;              // staged rows per thread
    constexpr int MOUT = 260;                           // output rows 0..Rs' (<= 256) per residue
    constexpr size_t STG_BYTES = size_t(N / 2 + N / 16 + 1) * sizeof(double);
    constexpr size_t EXCH_BYTES = size_t(NK) * F::LDS_REALS * sizeof(T);
    constexpr size_t SUM_BYTES = size_t(NK) * MOUT * sizeof(cpx<T>);
    constexpr size_t BYTES = STG_BYTES + EXCH_BYTES > SUM_BYTES ? STG_BYTES + EXCH_BYTES : SUM_BYTES;
    __shared__ __align__(16) unsigned char smem[BYTES];
    double* stg = reinterpret_cast<double*>(smem);
    T* exch = reinterpret_cast<T*>(smem + STG_BYTES);
    cpx<T>* sums = reinterpret_cast<cpx<T>*>(smem);
    const int tid = threadIdx.x;
    if (blk >= a.nfft) {               // extra workgroups: the partial sums of the sample kernel
        const int j = blk - a.nfft;
        __shared__ double red16[16];
        if (a.part && j < 4) sum_partials_in_block<NT>(a.part + size_t(j) * a.np, a.np, a.dst.d[j], red16);
        return;
    }
    const int pair = xcd_column(blk, a.nfft);
    if (pair >= NPAIR) return;
    const int la = 2 * pair, lb = la + 1;
    const bool has_b = lb < C;
    const int lane = tid & 63;
    const int k0 = __builtin_amdgcn_readfirstlane(tid >> 6);
    cpx<double>* hab = reinterpret_cast<cpx<double>*>(a.Hh + h_index(la, 0, a.ldH));   // columns la, lb
    const bool hot_cols = la < GHOT;   // GHOT is even: lb < GHOT too
    const int kc = stored_rows(a.rc2, la, N);
    if (kc < 0) return;                // (the adjoint row pass reads no frequency of these columns)
    // rows 0..kc of the pair (+ the hot tile's replicas), each read by one thread and then cleared
    __shared__ double hs[2][GHOT];
    if (hot_cols) {
        fold_hot<NT>(a.hot, la, hs);
        __syncthreads();
    }
    cpx<double> xs[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int p = tid + q * NT;
        xs[q] = cpx<double>{0.0, 0.0};
        if (p <= kc) {
            xs[q] = hab[p];
            if (hot_cols && p < GHOT) {
                xs[q].re += hs[0][p];
                xs[q].im += hs[1][p];
            }
            hab[p] = cpx<double>{0.0, 0.0};
        }
        if (p < C) stg[p + (p >> 3)] = xs[q].re;
    }
    __syncthreads();
    cpx<T> v[8];
    int sp[8];
    double wk[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const int k = k0 + P * (lane + 64 * r);
        const int p = k <= N / 2 ? k : N - k;
        sp[r] = p + (p >> 3);
        wk[r] = ext_weight(k, N);
        v[r].re = T(wk[r] * stg[sp[r]]);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int p = tid + q * NT;
        if (p < C) stg[p + (p >> 3)] = has_b ? xs[q].im : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r].im = T(wk[r] * stg[sp[r]]);
    F::run(v, exch + k0 * F::LDS_REALS, lane, a.tw, a.tw512, P, 0);
    // this residue's terms of rows m = lane + 64 s
    const bool mirror = k0 != 0 && 2 * k0 != P;
    const int src = (64 - lane) & 63;
    cpx<T> c[5];
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        const int m = lane + 64 * s;
        const cpx<T> w = a.tw[(m * k0) & (N - 1)];
        c[s] = cmul(v[s], w);
        if (mirror) {
            const T yr = __shfl(v[7 - s].re, src, 64), yi = __shfl(v[7 - s].im, src, 64);
            const cpx<T> ym = lane == 0 ? v[(8 - s) & 7] : cpx<T>{yr, yi};
            c[s] = cadd(c[s], cmul(ym, cconj(w)));
        }
    }
    __syncthreads();                   // every wave is done with the staged pair and its exchange region
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        const int m = lane + 64 * s;
        if (m <= a.Rs) sums[k0 * MOUT + m] = c[s];
    }
    __syncthreads();
    for (int m = tid; m <= a.Rs; m += NT) {
        cpx<T> acc = sums[m];
#pragma unroll
        for (int k = 1; k < NK; ++k) acc = cadd(acc, sums[k * MOUT + m]);
        const T cm = T(mult(m, N));
        T* o = a.Th + size_t(m) * a.ldTh + la;
        o[0] = cm * acc.re;
        if (has_b) o[1] = cm * acc.im;
    }
}

template <typename T, int LOG2N>
__global__ __launch_bounds__(ResidueShape<LOG2N>::NT) void k_adjcol_sub(AdjColArgs<T> a) {
    adjcol_sub_body<T, LOG2N>(a, blockIdx.x);
}

// ---------------------------------------------------------------------------
// adjoint of the row pass (two rows per workgroup) fused with the sweep
// adjoint: Th rows -> pixel gradients -> dchi2/dI (atomics) and dchi2/dinc.
// ---------------------------------------------------------------------------
template <typename T>
struct AdjRowArgs {
    SweepPrm<T> sw;
    const T* Th;
    int ldTh;
    int N, Rs, nrows;    // pixels j = 0..Rs', rows m = 0..nrows-1
    const cpx<T>* tw;
    double tan_inc;
    double* gI;          // nr, zeroed by the forward row pass
    double* ginc;        // 1, zeroed by the forward row pass
    const cpx<T>* tw512; // W_512^e table (k_adjrow_sub)
    int ncol;            // frequencies 0..ncol-1 of Th were written; beyond them it is zero
};

// dchi2/d(pixel value) = gz: accumulate into dI (workgroup-local copy in LDS)
// and return the inc term.
template <typename T>
__device__ __forceinline__ double sweep_pixel_adjoint(int xi, int yi, double gz, const SweepPrm<T>& p, double tan_inc,
                                                      double* gI) {
    if (gz == 0.0) return 0.0;
    const T x = T(xi) * p.dxy;
    const T y = T(yi) * p.dxy;
    T r;
    double xs2;
    if constexpr (std::is_same<T, double>::value) {
        const double xs = x / p.cos_inc;
        xs2 = xs * xs;
        r = sqrt(xs * xs + y * y);
    } else {
        const double xs = double(x / p.cos_inc);
        xs2 = xs * xs;
        r = float(sqrt(xs * xs + double(y) * double(y)));
    }
    T fi = floor((r - p.Rmin) / p.dR);
    fi = fi > T(0) ? fi : T(0);
    if (!(fi <= T(p.nr - 2))) return 0.0;
    const int iR = int(fi);
    const double alpha = (double(r) - double(iR) * double(p.dR) - double(p.Rmin)) / double(p.dR);
    const double sr = double(p.sr_to_px);
    lds_add_f64(gI + iR, gz * sr * (1.0 - alpha));
    lds_add_f64(gI + iR + 1, gz * sr * alpha);
    if (r == T(0)) return 0.0;
    const double dvdr = sr * (double(p.I[iR + 1]) - double(p.I[iR])) / double(p.dR);
    return gz * dvdr * xs2 * tan_inc / double(r);
}

// Bins i = t, t + nt, ... of the central pixel's adjoint (all threads t < nt
// of a workgroup together cover bins 0..iIN+1).
template <typename T>
__device__ __forceinline__ void central_adjoint(double gz, const SweepPrm<T>& p, double* gI, int t, int nt) {
    const int iIN = p.iIN;
    const double Rmin = p.Rmin, dR = p.dR, h = double(p.dxy) / 2.0;
    const double area = h * h - Rmin * Rmin;
    const double sc = gz * double(p.sr_to_px) / area;
    const double RiIN = Rmin + iIN * dR;
    const double delta = h - RiIN, beta = delta / dR;
    for (int i = t; i <= iIN + 1; i += nt) {
        if (i == 0) lds_add_f64(gI + 0, sc * dR * Rmin);
        if (i >= 1 && i < iIN) lds_add_f64(gI + i, sc * 2.0 * dR * (Rmin + i * dR));
        if (i == iIN) lds_add_f64(gI + iIN, sc * (dR * RiIN + delta * (RiIN + h * (1.0 - beta))));
        if (i == iIN + 1) lds_add_f64(gI + iIN + 1, sc * delta * h * beta);
    }
}

constexpr int ADJROW_LDS_NR = 2048;   // profile bins accumulated in LDS by the adjoint row pass

// SPLIT: as in rowpass_sym_body (the batched form uses the half-LDS exchange).
template <typename T, int LOG2N, bool SPLIT = false>
__device__ __forceinline__ void adjrow_sym_body(const AdjRowArgs<T>& a, int blk) {
    using S = FftShape<LOG2N>;
    using F = BlockFft<T, LOG2N, false, SPLIT>;
    constexpr int N = S::N, NT = S::NT, E = S::E;
    __shared__ T lds[F::LDS_REALS];
    __shared__ double red[16];
    __shared__ double gIl[ADJROW_LDS_NR];    // this workgroup's share of dchi2/dI (nr <= ADJROW_LDS_NR)
    const int tid = threadIdx.x;
    for (int k = tid; k < a.sw.nr; k += NT) gIl[k] = 0.0;   // ordered before use by the FFT's barriers
    const int ma = 2 * blk, mb = ma + 1;
    const bool hb = mb < a.nrows;
    const T* ra = a.Th + size_t(ma) * a.ldTh;
    const T* rb = ra + a.ldTh;
    cpx<T> v[E];
    F::run(v, lds, tid, N / 2, a.tw, [&](int k) -> cpx<T> {
        const int l = k <= N / 2 ? k : N - k;
        if (l >= a.ncol) return cpx<T>{T(0), T(0)};
        const T wk = T(ext_weight(k, N));
        return cpx<T>{wk * ra[l], hb ? wk * rb[l] : T(0)};
    }, a.Rs < NT);        // pixels j <= Rs' only
    __shared__ double gcen;
    double ginc = 0.0;
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int j = tid + r * NT;
        if (r * NT <= a.Rs && j <= a.Rs) {
            const double cj = mult(j, N);
            const double gza = cj * double(v[r].re), gzb = cj * double(v[r].im);
            if (ma == 0 && j == 0) gcen = gza;      // the central pixel: spread over the workgroup below
            else ginc += sweep_pixel_adjoint(j, ma, gza, a.sw, a.tan_inc, gIl);
            if (hb) ginc += sweep_pixel_adjoint(j, mb, gzb, a.sw, a.tan_inc, gIl);
        }
    }
    if (ma == 0) {                                 // (uniform per workgroup)
        __syncthreads();
        central_adjoint(gcen, a.sw, gIl, tid, NT);
    }
    const double b = block_sum_any(ginc, red);    // (its barrier also orders the LDS sums before the flush)
    if (tid == 0 && b != 0.0) atomic_add_f64(a.ginc, b);
    for (int k = tid; k < a.sw.nr; k += NT) {      // consecutive bins: coalesced atomics
        const double x = gIl[k];
        if (x != 0.0) atomic_add_f64(a.gI + k, x);
    }
}

template <typename T, int LOG2N>
__global__ __launch_bounds__(FftShape<LOG2N>::NT) void k_adjrow_sym(AdjRowArgs<T> a) {
    adjrow_sym_body<T, LOG2N>(a, blockIdx.x);
}

// Residue form of the adjoint row pass (N >= 1024, Rs' <= 256).  Its outputs are the pixels
// j = 0..Rs' of the N-point transform of the weighted even extension of two Th rows (real and
// imaginary parts), so it is the residue adjoint column transform over rows instead of column pairs:
// the rows are staged in LDS (real, then imaginary parts), one wave per residue class k0 = 0..P/2 of
// the input frequencies takes the 512-point transform of its decimated sequence, and the waves'
// terms W_N^(j k0) Y_k0[j] (with the mirror term of residue P - k0) are summed in LDS in residue
// order.  The pixel adjoints, the central pixel and the dI flush are those of adjrow_sym_body.  Its
// 5 waves per workgroup (N = 4096) run their transforms without workgroup barriers, which shortens
// the single workgroup path that the pass's ~100 workgroups take.
template <typename T, int LOG2N>
__device__ __forceinline__ void adjrow_sub_body(const AdjRowArgs<T>& a, int blk) {
    using CS = ResidueShape<LOG2N>;
    using F = ResidueFft<T>;
    constexpr int N = CS::N, P = CS::P, NT = CS::NT, NK = CS::NK;
    constexpr int C = N / 2 + 1;
    constexpr int PER = (C + NT - 1) / NT;              // staged frequencies per thread
    constexpr int MOUT = 260;                           // pixels 0..Rs' (<= 256) per residue
    constexpr size_t STG_BYTES = size_t(N / 2 + N / 16 + 1) * sizeof(T);
    constexpr size_t EXCH_BYTES = size_t(NK) * F::LDS_REALS * sizeof(T);
    constexpr size_t SUM_BYTES = size_t(NK) * MOUT * sizeof(cpx<T>);
    constexpr size_t BYTES = STG_BYTES + EXCH_BYTES > SUM_BYTES ? STG_BYTES + EXCH_BYTES : SUM_BYTES;
    __shared__ __align__(16) unsigned char smem[BYTES];
    __shared__ double gIl[ADJROW_LDS_NR];    // this workgroup's share of dchi2/dI (nr <= ADJROW_LDS_NR)
    __shared__ double red[16];
    __shared__ double gcen;
    T* stg = reinterpret_cast<T*>(smem);
    T* exch = reinterpret_cast<T*>(smem + STG_BYTES);
    cpx<T>* sums = reinterpret_cast<cpx<T>*>(smem);
    const int tid = threadIdx.x, lane = tid & 63;
    const int k0 = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int k = tid; k < a.sw.nr; k += NT) gIl[k] = 0.0;   // ordered before use by the barriers below
    const int ma = 2 * blk, mb = ma + 1;
    const bool hb = mb < a.nrows;
    const T* ra = a.Th + size_t(ma) * a.ldTh;
    const T* rb = ra + a.ldTh;
    // row ma staged (frequency p at p + p/8: the waves' stride-P gathers spread over the banks), row mb
    // held in registers until the first gather is done
    T xb[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int p = tid + q * NT;
        xb[q] = (hb && p < a.ncol) ? rb[p] : T(0);
        if (p < C) stg[p + (p >> 3)] = p < a.ncol ? ra[p] : T(0);
    }
    __syncthreads();
    cpx<T> v[8];
    int sp[8];
    T wk[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
        const int k = k0 + P * (lane + 64 * r);
        const int p = k <= N / 2 ? k : N - k;
        sp[r] = p + (p >> 3);
        wk[r] = T(ext_weight(k, N));
        v[r].re = wk[r] * stg[sp[r]];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int p = tid + q * NT;
        if (p < C) stg[p + (p >> 3)] = xb[q];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 8; ++r) v[r].im = wk[r] * stg[sp[r]];
    F::run(v, exch + k0 * F::LDS_REALS, lane, a.tw, a.tw512, P, 0);
    // this residue's terms of pixels j = lane + 64 s
    const bool mirror = k0 != 0 && 2 * k0 != P;
    const int src = (64 - lane) & 63;
    cpx<T> c[5];
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        const int j = lane + 64 * s;
        const cpx<T> w = a.tw[(j * k0) & (N - 1)];
        c[s] = cmul(v[s], w);
        if (mirror) {
            const T yr = __shfl(v[7 - s].re, src, 64), yi = __shfl(v[7 - s].im, src, 64);
            const cpx<T> ym = lane == 0 ? v[(8 - s) & 7] : cpx<T>{yr, yi};
            c[s] = cadd(c[s], cmul(ym, cconj(w)));
        }
    }
    __syncthreads();                   // every wave is done with the staged rows and its exchange region
#pragma unroll
    for (int s = 0; s < 5; ++s) {
        const int j = lane + 64 * s;
        if (j <= a.Rs) sums[k0 * MOUT + j] = c[s];
    }
    __syncthreads();
    double ginc = 0.0;
    for (int j = tid; j <= a.Rs; j += NT) {
        cpx<T> acc = sums[j];
#pragma unroll
        for (int k = 1; k < NK; ++k) acc = cadd(acc, sums[k * MOUT + j]);
        const double cj = mult(j, N);
        const double gza = cj * double(acc.re), gzb = cj * double(acc.im);
        if (ma == 0 && j == 0) gcen = gza;      // the central pixel: spread over the workgroup below
        else ginc += sweep_pixel_adjoint(j, ma, gza, a.sw, a.tan_inc, gIl);
        if (hb) ginc += sweep_pixel_adjoint(j, mb, gzb, a.sw, a.tan_inc, gIl);
    }
    if (ma == 0) {                                 // (uniform per workgroup)
        __syncthreads();
        central_adjoint(gcen, a.sw, gIl, tid, NT);
    }
    const double b = block_sum_any(ginc, red);    // (its barrier also orders the LDS sums before the flush)
    if (tid == 0 && b != 0.0) atomic_add_f64(a.ginc, b);
    for (int k = tid; k < a.sw.nr; k += NT) {      // consecutive bins: coalesced atomics
        const double x = gIl[k];
        if (x != 0.0) atomic_add_f64(a.gI + k, x);
    }
}

template <typename T, int LOG2N>
__global__ __launch_bounds__(ResidueShape<LOG2N>::NT) void k_adjrow_sub(AdjRowArgs<T> a) {
    adjrow_sub_body<T, LOG2N>(a, blockIdx.x);
}

}  // namespace gl
