// Marching P-SV step: two time steps of a grid's interior in one launch,
// reading the fields of step n from one buffer set and writing those of step
// n+2 to the other, so that a cell update moves 20 bytes of FP32 fields and
// its share of the material instead of the two passes' 80.
//
// A workgroup owns a strip of W - 32 columns of one shot and marches down a
// segment of its rows; it computes W columns, since a step moves information
// 8 columns (the velocities of x read stresses of x-4..x+4, and those read
// the old velocities).  Iteration s computes, from the rows loaded so far,
//   the first step's stresses of row s and velocities of row s-4,
//   the second step's stresses of row s-8 and velocities of row s-12,
// so an iteration loads one row of every array and stores one of each field.
// z-derivatives come from registers: every field is a ring of 8 rows whose
// slot is the row modulo 8, and the loop body is unrolled 8 times, so that no
// row is ever moved.  x-derivatives come from LDS: the eight rows an iteration
// differentiates along x were complete when it began; six are written at its
// start (two buffers in turn), the two Txx rows come from 8-row LDS rings
// that also hold them for their own column, so one barrier per row orders all.
// A thread holds two adjacent columns: 8-byte loads, stores and LDS accesses,
// two independent chains, and 4 LDS reads for the 14 neighbours of two cells.
// The fields are loaded two rows ahead, the material one.
//
// The loop without sources, receivers or segment ends has no branch: with
// one, the compiler moves the loads ahead behind it and waits for each row
// (121 against 163 Gcell/s on 4096 x 2048 x 8 in FP32).  Lanes that own
// nothing, and rows outside the segment, store beyond the buffer's range,
// which drops them.  Items with a source tap or a recorded receiver run the
// same rows with the checks (a source, or a line of receivers, at mid-depth:
// 0 to 9% more a step in FP32, 11 to 23% in 16 bits; a receiver in every row of
// one column 2 to 20% and 24 to 43%).
//
// Measured, 8 shots of 4096 x 2048, FP32: 701-725 us for the two steps of the
// 4000 x 1984 interior (176-181 Gcell/s; 3.08 GB from and to the HBM, 4.2 TB/s;
// 206 M wavefront instructions of the vector units, 46% of their issue slots)
// where the two passes take 1680; FP16 591-617 us (1.91 GB, 3.2 TB/s, 254 M,
// 68%).  One column per thread and three workgroups per CU: 781 us.
// Non-temporal field loads and stores keep the material in the L2: 757 -> 701
// us in FP32; FP16, half the bytes, is not faster with them (617 / 629).  The
// register files are full: 256 VGPRs, two wavefronts per SIMD; nothing spills
// to memory but, in 16 bits, the checked body that gathers maxima (40).
//
// The arithmetic of a cell is that of the two-pass kernels' interior path
// (psv_stress_interior, psv_velocity_interior), and values that the passes
// store and read back are rounded through the storage type: bitwise equal.
// It covers the rectangle that keeps 12 cells of plain arithmetic on every
// side; the frame around it runs the two passes (see launch_march_t).
#pragma once
#include "fd_fused.hpp"

namespace fd23 {

constexpr int NC = 2;            // columns of a thread
constexpr int MH = 16;           // halo columns on each side, two steps of 8
constexpr int kMarchReach = 12;  // cells around the rectangle that run plain arithmetic
constexpr int kMarchTail = 24;   // iterations of a segment beyond its rows

struct MarchWork {
    int x0, x1, z0, z1;     // the rectangle, in cells
    int W;                  // columns of a strip with its halo, 256 or 512
    int nstrip, nseg, H;    // H rows per segment
    int nwork;              // work item = (segment, strip, shot), shot fastest
};

// a value as the passes would read it back after storing it
template <class S> __device__ __forceinline__ float through(float v, float inv, float s) {
    if constexpr (Store<S>::scaled) {
        S b[1];
        Store<S>::st(b, 0, v, inv);
        return Store<S>::ld(b, 0, s);
    }
    return v;
}

// two adjacent stored elements as loaded, 8 or 4 bytes; taken apart (and
// scaled) where they are used, so that a load in flight stays in flight
template <class S> struct Raw2 {
    using T = float __attribute__((ext_vector_type(2)));
};
template <> struct Raw2<__half> {
    using T = unsigned;
};
template <> struct Raw2<__hip_bfloat16> {
    using T = unsigned;
};
template <class S, class R> __device__ __forceinline__ void unpack2(R v, float s, float (&o)[NC]) {
    if constexpr (sizeof(S) == 4) {
        o[0] = v.x;
        o[1] = v.y;
    } else {
        S b[2];
        b[0] = __builtin_bit_cast(S, (unsigned short)(v & 0xffffu));
        b[1] = __builtin_bit_cast(S, (unsigned short)(v >> 16));
        o[0] = Store<S>::ld(b, 0, s);
        o[1] = Store<S>::ld(b, 1, s);
    }
}
// at a uniform base and a lane's byte offset; NT: read once, not to be kept
// in the caches
template <class S, bool NT = false>
__device__ __forceinline__ typename Raw2<S>::T load2(const void *base, unsigned vo) {
    const auto *p = (const typename Raw2<S>::T *)((const char *)base + (size_t)vo);
    return NT && sizeof(S) == 4 ? __builtin_nontemporal_load(p) : *p;
}
// through a buffer resource, at byte offsets vo (lane) + so (uniform)
template <class S>
__device__ __forceinline__ void store2(BufRsrc r, unsigned vo, unsigned so, const float (&v)[NC], float inv) {
    if constexpr (sizeof(S) == 4) {
        using U2 = decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0));
        U2 q;
        q[0] = __builtin_bit_cast(unsigned, v[0]);
        q[1] = __builtin_bit_cast(unsigned, v[1]);
        __builtin_amdgcn_raw_buffer_store_b64(q, r, vo, so, 2); // non-temporal
    } else {
        S b[2];
        Store<S>::st(b, 0, v[0], inv);
        Store<S>::st(b, 1, v[1], inv);
        const unsigned q = (unsigned)__builtin_bit_cast(unsigned short, b[0]) |
                           (unsigned)__builtin_bit_cast(unsigned short, b[1]) << 16;
        __builtin_amdgcn_raw_buffer_store_b32(q, r, vo, so, 0);
    }
}

// a list read at a uniform index, through the scalar cache: a vector load
// there would wait for the rows loaded ahead
template <class T> __device__ __forceinline__ const __attribute__((address_space(4))) T *uniform(const T *p) {
    return (const __attribute__((address_space(4))) T *)p;
}
__device__ __forceinline__ RecF uniform_rec(const RecF *p, int e) {
    const auto *r = uniform(p) + e;
    return RecF{r->row, r->lane, r->comp, r->out, r->next, r->nextrow};
}
// receivers of a row that are not worth two barriers and a vector load (a
// borehole's one per row: SH, 2 shots of 2000 x 1000 40 us a step, 46 with)
constexpr int kFewRecs = 4;

// a work item, and what happens in it: source taps [t0, t1) of rows
// trow0..trow1, active in the first (onA) or second step (onB); receivers
// from list entry r on, the next row recorded in either step
struct MarchItem {
    int shot, strip, xs, za, zb;
    int t0, t1, trow0, trow1, r, r1, nextA, nextB, ts;
    double svA, svB;
    bool onA, onB;
};
template <int MW> struct MarchLds {
    float rows[2][6][MW + 2 * HALO]; // rows an iteration differentiates along x
    float ring[2][8][MW + 2 * HALO]; // Txx of the first and the second step, slot (row - s0) & 7
    float park[2][MW];               // U and W of a recorded row
};

// the item's rows.  CHECK: with sources and receivers; TRACK: gathering the
// maxima of the second step's values for a scale check.  sa: the scales of
// the set that is read; scl: current scales [0, kNextScale) and next ones
// after them, in which fields are written.
template <class S, int MW, bool CHECK, bool TRACK>
__device__ __forceinline__ void march_item(const PsvFields<S> &fa, const PsvFields<S> &fb, const PsvMat5<float> &m,
                                           const Grid &g, const MarchWork &w, const FusedEvents &ev,
                                           const float *__restrict__ sa, const float *__restrict__ scl,
                                           unsigned *__restrict__ amax, const MarchItem &q, MarchLds<MW> &l) {
    using C = float;
    using ST = Store<S>;
    constexpr int MT = MW / NC, LW = MW + 2 * HALO;
    const int lc = (int)threadIdx.x * NC; // the thread's first column in the strip
    const int nz = g.nz, px = g.px;
    const int xs = q.xs, za = q.za, zb = q.zb;
    const int col = min(xs - MH + lc, w.x1 + MH - NC);
    const bool own = lc >= MH && lc < MW - MH && xs - MH + lc < w.x1;

    const long org = (long)q.shot * g.sstride;
    // loads: the loop's row offsets are folded into the bases, so that one lane
    // offset (row s) serves the fields, one the first step's material and one
    // the second's
    const S *bU = fa.U + org + 3L * px, *bW = fa.W + org + 4L * px, *bXX = fa.Txx + org, *bZZ = fa.Tzz + org,
            *bXZ = fa.Txz + org;
    const BufRsrc oU = buf_rsrc(fb.U + org), oW = buf_rsrc(fb.W + org), oXX = buf_rsrc(fb.Txx + org),
                  oZZ = buf_rsrc(fb.Tzz + org), oXZ = buf_rsrc(fb.Txz + org);
    const C *rBU = m.BU - 4L * px, *rBW = m.BW - 4L * px, *rMU = m.MU, *rMUA = m.MUA, *rLAM = m.LAM;
    const unsigned vc = (unsigned)col * sizeof(S), vm = (unsigned)col * sizeof(C);
    const unsigned vst = own ? vc : 0x80000000u; // beyond the buffer's range: dropped
    const unsigned pxb = (unsigned)px * sizeof(S), pxm = (unsigned)px * sizeof(C);

    float rd[5] = {1.f, 1.f, 1.f, 1.f, 1.f}, nx_[5] = {1.f, 1.f, 1.f, 1.f, 1.f}, wi[5] = {1.f, 1.f, 1.f, 1.f, 1.f};
    if (ST::scaled) {
#pragma unroll
        for (int i = 0; i < 5; i++) {
            rd[i] = sa[i];
            nx_[i] = scl[kNextScale + i];
            wi[i] = inv_pow2(nx_[i]);
        }
    }
    float mx[5] = {0.f, 0.f, 0.f, 0.f, 0.f};

    auto inject = [&](int row, double sv, C (&a)[NC], C (&b)[NC], C (&c)[NC]) {
        for (int e = q.t0; e < q.t1; e++) {
            const auto *t = uniform(ev.taps) + e;
            if (t->row != row) continue;
            const TapF tp{t->row, t->lane, t->field, t->mode, t->m, t->q};
#pragma unroll
            for (int i = 0; i < NC; i++) {
                // selects: with a branch per field the compiler takes the address
                // of the one that is changed, and all three live in scratch memory,
                // whose reloads wait for the rows ahead (2 shots of 3000 x 1800
                // with a source at mid-depth 143 us a step, 113 so, 106 without)
                const bool mine = tp.lane == lc + i;
                a[i] = mine && tp.field == 2 ? apply_tap(a[i], tp, sv) : a[i];
                b[i] = mine && tp.field == 3 ? apply_tap(b[i], tp, sv) : b[i];
                c[i] = mine && tp.field == 4 ? apply_tap(c[i], tp, sv) : c[i];
            }
        }
    };
    auto record = [&](int step, int &r, const C (&u)[NC], const C (&ww)[NC]) -> int {
        const int e0 = r;
        RecF rc = uniform_rec(ev.recs, e0);
        const int e1 = rc.next, row = rc.nextrow;
        r = e1;
        C *seis = (C *)ev.seis + (long)(step / ev.itrecord) * ev.frame_size;
        if (e1 - e0 <= kFewRecs) { // straight from the registers of the columns' threads
            for (int e = e0;;) {
#pragma unroll
                for (int i = 0; i < NC; i++)
                    if (rc.lane == lc + i) seis[rc.out] = rc.comp == 0 ? u[i] : ww[i];
                if (++e >= e1) return row;
                rc = uniform_rec(ev.recs, e);
            }
        }
#pragma unroll
        for (int i = 0; i < NC; i++) {
            l.park[0][lc + i] = u[i];
            l.park[1][lc + i] = ww[i];
        }
        __syncthreads();
        for (int e = e0 + (int)threadIdx.x; e < e1; e += MT) {
            const RecF rc = ev.recs[e];
            seis[rc.out] = l.park[rc.comp == 0 ? 0 : 1][rc.lane];
        }
        __syncthreads();
        return row;
    };

    int rA = q.r, rB = q.r, nextA = q.nextA, nextB = q.nextB;
    using RS = typename Raw2<S>::T;
    using RC = typename Raw2<C>::T;
    struct Row {
        RS u, w, xx, zz, xz;
    };
    struct Mat {
        RC lam, mu, mua, bu, bw, lam2, mu2, mua2, bu2, bw2;
    };
    // rows past the last one needed (the loop runs in eights, loads two rows
    // ahead) read the last row again
    auto load = [&](int s) __attribute__((always_inline)) {
        const unsigned vo = vc + (unsigned)min(s, nz - 5) * pxb;
        return Row{load2<S, true>(bU, vo), load2<S, true>(bW, vo), load2<S, true>(bXX, vo), load2<S, true>(bZZ, vo),
                   load2<S, true>(bXZ, vo)};
    };
    auto loadm = [&](int s) __attribute__((always_inline)) {
        const unsigned vo = vm + (unsigned)min(s, nz - 5) * pxm, v8 = vm + (unsigned)min(max(s - 8, 4), nz - 5) * pxm;
        return Mat{load2<C>(rLAM, vo), load2<C>(rMU, vo), load2<C>(rMUA, vo), load2<C>(rBU, vo), load2<C>(rBW, vo),
                   load2<C>(rLAM, v8), load2<C>(rMU, v8), load2<C>(rMUA, v8), load2<C>(rBU, v8), load2<C>(rBW, v8)};
    };
    auto mat = [](RC v, int i) __attribute__((always_inline)) { return i == 0 ? v.x : v.y; };

    const C c0 = C(1225. / 1024.), c1 = C(245. / 3072.), c2 = C(49. / 5120.), c3 = C(5. / 7168.);
    const int s0 = za - kMarchReach;
    const int o = lc + HALO;
    // the thread's columns of an LDS row, always as one 8-byte value (an access
    // of another type to the same place could be moved across it)
    auto put = [&](C *row, const C (&v)[NC]) __attribute__((always_inline)) {
        *(float2 *)(row + o) = make_float2(v[0], v[1]);
    };
    auto take = [&](const C *row, C (&v)[NC]) __attribute__((always_inline)) {
        const float2 p = *(const float2 *)(row + o);
        v[0] = p.x, v[1] = p.y;
    };
    C u0[8][NC], w0[8][NC], zz1[8][NC], xz1[8][NC], u1[8][NC], w1[8][NC], zz2[8][NC], xz2[8][NC];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int d = i - 4;
        const C none[NC] = {C(0), C(0)};
        put(l.ring[0][i], none);
        put(l.ring[1][i], none);
#pragma unroll
        for (int k = 0; k < NC; k++) {
            zz1[i][k] = xz1[i][k] = u1[i][k] = w1[i][k] = zz2[i][k] = xz2[i][k] = C(0);
            u0[3][k] = C(0);
        }
        if (i < 7) unpack2<S>(load2<S>(fa.U + org, vc + (unsigned)(s0 + d) * pxb), rd[0], u0[d & 7]);
        unpack2<S>(load2<S>(fa.W + org, vc + (unsigned)(s0 + d) * pxb), rd[1], w0[d & 7]);
    }
    // x-derivatives from an LDS row around the thread's columns
    auto xdiff = [&](const C *row, const C (&v)[NC], bool ahead, C (&d)[NC]) __attribute__((always_inline)) {
        const float2 p0 = *(const float2 *)(row + o - 4), p1 = *(const float2 *)(row + o - 2),
                     p2 = *(const float2 *)(row + o + 2), p3 = *(const float2 *)(row + o + 4);
        const C f[10] = {p0.x, p0.y, p1.x, p1.y, v[0], v[1], p2.x, p2.y, p3.x, p3.y};
#pragma unroll
        for (int i = 0; i < NC; i++)
            d[i] = ahead ? dp8(f[i + 1], f[i + 2], f[i + 3], f[i + 4], f[i + 5], f[i + 6], f[i + 7], f[i + 8], c0, c1,
                               c2, c3)
                         : dm8(f[i], f[i + 1], f[i + 2], f[i + 3], f[i + 4], f[i + 5], f[i + 6], f[i + 7], c0, c1, c2,
                               c3);
    };
    // z-derivatives from a ring whose lowest row is in slot j
#define RING8(f, j, i)                                                                                        \
    f[(j)&7][i], f[((j) + 1) & 7][i], f[((j) + 2) & 7][i], f[((j) + 3) & 7][i], f[((j) + 4) & 7][i],              \
        f[((j) + 5) & 7][i], f[((j) + 6) & 7][i], f[((j) + 7) & 7][i]

    Mat cm = loadm(s0);
    Row cur = load(s0), n1 = load(s0 + 1);
    const int nit = (zb - za + kMarchTail + 7) & ~7;
#pragma unroll 1
    for (int sb = s0; sb < s0 + nit; sb += 8) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int s = sb + j;
            const Mat nm = loadm(s + 1);
            const Row n2 = load(s + 2);
            const int j4 = (j + 4) & 7;
            C(*row)[LW] = l.rows[j & 1];
            put(row[0], u0[j]);
            put(row[1], w0[j]);
            put(row[2], xz1[j4]);
            put(row[3], u1[j]);
            put(row[4], w1[j]);
            put(row[5], xz2[j4]);
            C wv[NC], xa[NC], xb[NC], wn[NC], a[NC], b[NC], c[NC];
            take(l.ring[0][j4], xa);
            take(l.ring[1][j4], xb);
            unpack2<S>(cur.u, rd[0], u0[(j + 3) & 7]);
            unpack2<S>(cur.w, rd[1], wn);
            unpack2<S>(cur.xx, rd[2], a);
            unpack2<S>(cur.zz, rd[3], b);
            unpack2<S>(cur.xz, rd[4], c);
#pragma unroll
            for (int i = 0; i < NC; i++) {
                wv[i] = w0[j4][i]; // W of row s-4
                w0[j4][i] = wn[i];
            }
            __syncthreads();
            C ux[NC], wx[NC], dxx[NC], dxz[NC];
            C u[NC], ww[NC], wv2[NC], a2[NC], b2[NC], cc2[NC];
            // ---- first step: stresses of row s
            xdiff(row[0], u0[j], false, ux);
            xdiff(row[1], w0[j], true, wx);
#pragma unroll
            for (int i = 0; i < NC; i++) {
                const C uz = dm8(RING8(u0, j + 4, i), c0, c1, c2, c3), wz = dp8(RING8(w0, j + 5, i), c0, c1, c2, c3);
                psv_stress_interior(ux[i], uz, wx[i], wz, mat(cm.lam, i), mat(cm.mu, i), mat(cm.mua, i), a[i], b[i], c[i]);
            }
            if (CHECK && q.onA && s >= q.trow0 && s <= q.trow1) inject(s, q.svA, a, b, c);
            // ---- first step: velocities of row s-4
            xdiff(l.ring[0][j4], xa, true, dxx);
            xdiff(row[2], xz1[j4], false, dxz);
            take(l.ring[0][j], a2); // row s-8 of the first step's stresses goes to the second
#pragma unroll
            for (int i = 0; i < NC; i++) {
                a[i] = through<S>(a[i], wi[2], nx_[2]);
                b[i] = through<S>(b[i], wi[3], nx_[3]);
                c[i] = through<S>(c[i], wi[4], nx_[4]);
                const C dzz = dm8(RING8(zz1, j, i), c0, c1, c2, c3);
                b2[i] = zz1[j][i], cc2[i] = xz1[j][i];
                zz1[j][i] = b[i];
                xz1[j][i] = c[i];
                const C dzx = dp8(RING8(xz1, j + 1, i), c0, c1, c2, c3);
                u[i] = u0[j4][i], ww[i] = wv[i];
                psv_velocity_interior(dxx[i], dzz, dxz[i], dzx, mat(cm.bu, i), mat(cm.bw, i), u[i], ww[i]);
            }
            put(l.ring[0][j], a);
            if (CHECK && s - 4 == nextA) nextA = record(q.ts, rA, u, ww);
#pragma unroll
            for (int i = 0; i < NC; i++) {
                u[i] = through<S>(u[i], wi[0], nx_[0]);
                ww[i] = through<S>(ww[i], wi[1], nx_[1]);
                wv2[i] = w1[j4][i]; // first step's W of row s-12
                w1[j4][i] = ww[i];
            }
            // ---- second step: stresses of row s-8
            xdiff(row[3], u1[j], false, ux);
            xdiff(row[4], w1[j], true, wx);
#pragma unroll
            for (int i = 0; i < NC; i++) {
                const C uz = dm8(RING8(u1, j + 4, i), c0, c1, c2, c3), wz = dp8(RING8(w1, j + 5, i), c0, c1, c2, c3);
                psv_stress_interior(ux[i], uz, wx[i], wz, mat(cm.lam2, i), mat(cm.mu2, i), mat(cm.mua2, i), a2[i], b2[i], cc2[i]);
            }
            const int rs = s - 8;
            if (CHECK && q.onB && rs >= q.trow0 && rs <= q.trow1) inject(rs, q.svB, a2, b2, cc2);
            {
                const bool in = rs >= za && rs < zb;
                const unsigned so = in ? (unsigned)rs * pxb : 0u, vo = in ? vst : 0x80000000u;
                store2<S>(oXX, vo, so, a2, wi[2]);
                store2<S>(oZZ, vo, so, b2, wi[3]);
                store2<S>(oXZ, vo, so, cc2, wi[4]);
                if (TRACK) {
#pragma unroll
                    for (int i = 0; i < NC; i++) {
                        mx[2] = fmaxf(mx[2], in && own ? fabsf(a2[i]) : 0.f);
                        mx[3] = fmaxf(mx[3], in && own ? fabsf(b2[i]) : 0.f);
                        mx[4] = fmaxf(mx[4], in && own ? fabsf(cc2[i]) : 0.f);
                    }
                }
            }
            // ---- second step: velocities of row s-12
            xdiff(l.ring[1][j4], xb, true, dxx);
            xdiff(row[5], xz2[j4], false, dxz);
            C u2[NC], ww2[NC];
#pragma unroll
            for (int i = 0; i < NC; i++) {
                a2[i] = through<S>(a2[i], wi[2], nx_[2]);
                b2[i] = through<S>(b2[i], wi[3], nx_[3]);
                cc2[i] = through<S>(cc2[i], wi[4], nx_[4]);
                const C dzz = dm8(RING8(zz2, j, i), c0, c1, c2, c3);
                zz2[j][i] = b2[i];
                xz2[j][i] = cc2[i];
                const C dzx = dp8(RING8(xz2, j + 1, i), c0, c1, c2, c3);
                u2[i] = u1[j4][i], ww2[i] = wv2[i];
                u1[j4][i] = u[i];
                psv_velocity_interior(dxx[i], dzz, dxz[i], dzx, mat(cm.bu2, i), mat(cm.bw2, i), u2[i], ww2[i]);
            }
            put(l.ring[1][j], a2);
            const int rv = s - 12;
            {
                const bool in = rv >= za && rv < zb;
                const unsigned so = in ? (unsigned)rv * pxb : 0u, vo = in ? vst : 0x80000000u;
                store2<S>(oU, vo, so, u2, wi[0]);
                store2<S>(oW, vo, so, ww2, wi[1]);
                if (TRACK) {
#pragma unroll
                    for (int i = 0; i < NC; i++) {
                        mx[0] = fmaxf(mx[0], in && own ? fabsf(u2[i]) : 0.f);
                        mx[1] = fmaxf(mx[1], in && own ? fabsf(ww2[i]) : 0.f);
                    }
                }
            }
            if (CHECK && rv == nextB) nextB = record(q.ts + 1, rB, u2, ww2);
            cur = n1;
            n1 = n2;
            cm = nm;
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#undef RING8
    if (TRACK) {
        amax_update(amax, SC_U, mx[0]);
        amax_update(amax, SC_W, mx[1]);
        amax_update(amax, SC_TXX, mx[2]);
        amax_update(amax, SC_TZZ, mx[3]);
        amax_update(amax, SC_TXZ, mx[4]);
    }
}

// work item L; whether a source or receiver is in it
template <int MW>
__device__ __forceinline__ bool march_find(const Grid &g, const MarchWork &w, const FusedEvents &ev, int L, MarchItem &q) {
    const int rest = L / g.nshots, seg = rest / w.nstrip;
    q.shot = L % g.nshots;
    q.strip = rest % w.nstrip;
    q.xs = w.x0 + q.strip * (MW - 2 * MH);
    q.za = w.z0 + seg * w.H;
    q.zb = min(q.za + w.H, w.z1);
    // sources and receivers of both steps
    q.t0 = q.t1 = q.trow0 = q.r = q.r1 = q.ts = 0;
    q.trow1 = q.nextA = q.nextB = kNoRow;
    q.svA = q.svB = 0.0;
    q.onA = q.onB = false;
    if (ev.clock) {
        const int it = ev.clock[0] + ev.k;
        const SrcInfo si = ev.src[q.shot];
        q.t0 = ev.tap_start[q.strip * g.nshots + q.shot];
        q.t1 = ev.tap_start[q.strip * g.nshots + q.shot + 1];
        if (q.t1 > q.t0) {
            q.onA = src_sample(si, ev.stf, it, q.svA);
            q.onB = src_sample(si, ev.stf, it + 1, q.svB);
            q.trow0 = q.trow1 = uniform(ev.taps)[q.t0].row;
            for (int e = q.t0 + 1; e < q.t1; e++) {
                const int row = uniform(ev.taps)[e].row;
                q.trow0 = min(q.trow0, row);
                q.trow1 = max(q.trow1, row);
            }
        }
        const int rkey = (seg * w.nstrip + q.strip) * g.nshots + q.shot;
        q.r = ev.rec_start[rkey];
        q.r1 = ev.rec_start[rkey + 1];
        q.ts = it - si.t0;
        auto recorded = [&](int t) { return t >= 0 && t % ev.itrecord == 0 && t / ev.itrecord < ev.max_frames; };
        if (q.r < q.r1) {
            const int row = uniform(ev.recs)[q.r].row;
            q.nextA = recorded(q.ts) ? row : kNoRow;
            q.nextB = recorded(q.ts + 1) ? row : kNoRow;
        }
    }
    const bool taps = (q.onA || q.onB) && q.trow1 >= q.za - kMarchReach && q.trow0 < q.zb + kMarchReach;
    return taps || q.nextA != kNoRow || q.nextB != kNoRow;
}

template <class S, int MW>
__global__ __launch_bounds__(MW / NC, 2) void k_psv_march(PsvFields<S> fa, PsvFields<S> fb, PsvMat5<float> m, Grid g,
                                                          MarchWork w, FusedEvents ev, const float *__restrict__ sa,
                                                          const float *__restrict__ scl,
                                                          unsigned *__restrict__ amax) {
    __shared__ MarchLds<MW> l;
    const int qd = gridDim.x >> 3; // grid padded to a multiple of 8
    const int L = (int)(blockIdx.x & 7) * qd + (int)(blockIdx.x >> 3);
    if (L >= w.nwork) return;
    MarchItem q;
    const bool checked = march_find<MW>(g, w, ev, L, q);
    // amax is null on steps that no scale check follows, three launches
    // of four: they run the bodies without the maxima, whose checked
    // one spills 40 registers in 16 bits (FP16, 4 shots of 3000 x 1800 with
    // sources at mid-depth 246 us a step, 198 so)
    const bool track = Store<S>::scaled && amax;
    if (checked && track)
        march_item<S, MW, true, Store<S>::scaled>(fa, fb, m, g, w, ev, sa, scl, amax, q, l);
    else if (checked)
        march_item<S, MW, true, false>(fa, fb, m, g, w, ev, sa, scl, amax, q, l);
    else if (track)
        march_item<S, MW, false, Store<S>::scaled>(fa, fb, m, g, w, ev, sa, scl, amax, q, l);
    else
        march_item<S, MW, false, false>(fa, fb, m, g, w, ev, sa, scl, amax, q, l);
}

// fd23_march.hip
template <class S>
void march_launch(hipStream_t stream, const PsvFields<S> &fa, const PsvFields<S> &fb, const PsvMat5<float> &m,
                  const Grid &g, const MarchWork &w, const FusedEvents &ev, const float *sa, const float *scl,
                  unsigned *amax);

// SH (fd_sh_march.hpp), FP32
void sh_march_launch(hipStream_t stream, const ShFields<float> &fa, const ShFields<float> &fb, const ShMat3<float> &m,
                     const Grid &g, const MarchWork &w, const FusedEvents &ev);

} // namespace fd23
