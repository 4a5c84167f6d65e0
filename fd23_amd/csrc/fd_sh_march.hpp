// Marching SH step, FP32: two time steps of a grid's interior in one launch,
// from one buffer set to the other, in the manner of the P-SV one
// (fd_march.hpp): a cell update moves 12 bytes of fields instead of the two
// passes' 36.  Iteration s computes, from the rows loaded so far,
//   the first step's Tx, Tz of row s and V of row s-4,
//   the second step's Tx, Tz of row s-8 and V of row s-12.
// V and Tz of both steps are register rings of 8 rows (z-derivatives); V rows
// are written to LDS when an iteration differentiates them along x, Tx lives
// in 8-row LDS rings.  The second step's material is the first one's of eight
// iterations ago, a third register ring: loaded again, half of the loads went
// to the material (6 shots of 2048 x 1024 77 us a step instead of 68).  The
// arithmetic is the two passes' interior path: bitwise equal.
//
// Measured, us a step with the frame's passes (two passes on the whole grid):
// 6 shots of 2048 x 1024 68 (82), 4 shots of 4096 x 2048 133 (265).  The
// registers (204) leave two wavefronts per SIMD; three, with segments a third
// shorter, take 81 and 149: the 24 rows that a segment recomputes weigh more.
// Of the 68 us the frame's four launches take 25.
#pragma once
#include "fd_march.hpp"

namespace fd23 {

template <int MW> struct ShMarchLds {
    float rows[2][2][MW + 2 * HALO]; // V of the first and the second step's row
    float ring[2][8][MW + 2 * HALO]; // Tx of the first and the second step, slot (row - s0) & 7
    float park[MW];                  // V of a recorded row
};

// CHECK: with sources and receivers
template <int MW, bool CHECK>
__device__ __forceinline__ void sh_march_item(const ShFields<float> &fa, const ShFields<float> &fb,
                                              const ShMat3<float> &m, const Grid &g, const MarchWork &w,
                                              const FusedEvents &ev, const MarchItem &q, ShMarchLds<MW> &l) {
    using C = float;
    using R2 = typename Raw2<C>::T;
    constexpr int MT = MW / NC, LW = MW + 2 * HALO;
    const int lc = (int)threadIdx.x * NC; // the thread's first column in the strip
    const int nz = g.nz, px = g.px;
    const int xs = q.xs, za = q.za, zb = q.zb;
    const int col = min(xs - MH + lc, w.x1 + MH - NC);
    const bool own = lc >= MH && lc < MW - MH && xs - MH + lc < w.x1;

    const long org = (long)q.shot * g.sstride;
    // the loop's row offsets are folded into the bases
    const C *bV = fa.V + org + 3L * px, *bX = fa.Tx + org, *bZ = fa.Tz + org;
    const BufRsrc oV = buf_rsrc(fb.V + org), oX = buf_rsrc(fb.Tx + org), oZ = buf_rsrc(fb.Tz + org);
    const C *rBV = m.BV - 4L * px, *rMX = m.MUX, *rMZ = m.MUZ;
    const unsigned vc = (unsigned)col * sizeof(C), pxb = (unsigned)px * sizeof(C);
    const unsigned vst = own ? vc : 0x80000000u; // beyond the buffer's range: dropped

    auto inject = [&](int row, double sv, int field, C (&a)[NC]) {
        for (int e = q.t0; e < q.t1; e++) {
            const auto *t = uniform(ev.taps) + e;
            if (t->row != row || t->field != field) continue;
            const TapF tp{t->row, t->lane, t->field, t->mode, t->m, t->q};
#pragma unroll
            for (int i = 0; i < NC; i++)
                if (tp.lane == lc + i) a[i] = apply_tap(a[i], tp, sv);
        }
    };
    auto record = [&](int step, int &r, const C (&v)[NC]) -> int {
        const int e0 = r;
        RecF rc = uniform_rec(ev.recs, e0);
        const int e1 = rc.next, row = rc.nextrow;
        r = e1;
        C *seis = (C *)ev.seis + (long)(step / ev.itrecord) * ev.frame_size;
        if (e1 - e0 <= kFewRecs) {
            for (int e = e0;;) {
#pragma unroll
                for (int i = 0; i < NC; i++)
                    if (rc.lane == lc + i) seis[rc.out] = v[i];
                if (++e >= e1) return row;
                rc = uniform_rec(ev.recs, e);
            }
        }
#pragma unroll
        for (int i = 0; i < NC; i++) l.park[lc + i] = v[i];
        __syncthreads();
        for (int e = e0 + (int)threadIdx.x; e < e1; e += MT) {
            const RecF rc = ev.recs[e];
            seis[rc.out] = l.park[rc.lane];
        }
        __syncthreads();
        return row;
    };

    int rA = q.r, rB = q.r, nextA = q.nextA, nextB = q.nextB;
    struct Row {
        R2 v, x, z;
    };
    struct Mat {
        R2 mx, mz, bv;
    };
    auto load = [&](int s) __attribute__((always_inline)) {
        const unsigned vo = vc + (unsigned)min(s, nz - 5) * pxb;
        return Row{load2<C, true>(bV, vo), load2<C, true>(bX, vo), load2<C, true>(bZ, vo)};
    };
    auto loadm = [&](int s) __attribute__((always_inline)) {
        const unsigned vo = vc + (unsigned)min(s, nz - 5) * pxb;
        return Mat{load2<C>(rMX, vo), load2<C>(rMZ, vo), load2<C>(rBV, vo)};
    };
    auto at = [](R2 v, int i) __attribute__((always_inline)) { return i == 0 ? v.x : v.y; };

    const C c0 = C(1225. / 1024.), c1 = C(245. / 3072.), c2 = C(49. / 5120.), c3 = C(5. / 7168.);
    const int s0 = za - kMarchReach;
    const int o = lc + HALO;
    auto put = [&](C *row, const C (&v)[NC]) __attribute__((always_inline)) {
        *(float2 *)(row + o) = make_float2(v[0], v[1]);
    };
    auto take = [&](const C *row, C (&v)[NC]) __attribute__((always_inline)) {
        const float2 p = *(const float2 *)(row + o);
        v[0] = p.x, v[1] = p.y;
    };
    C v0[8][NC], z1[8][NC], v1[8][NC], z2[8][NC];
    Mat ring[8]; // material of the second step: that of the first, eight iterations ago
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int d = i - 4;
        const C none[NC] = {C(0), C(0)};
        put(l.ring[0][i], none);
        put(l.ring[1][i], none);
        ring[i] = Mat{R2{0.f, 0.f}, R2{0.f, 0.f}, R2{0.f, 0.f}};
#pragma unroll
        for (int k = 0; k < NC; k++) {
            z1[i][k] = v1[i][k] = z2[i][k] = C(0);
            v0[3][k] = C(0);
        }
        if (i < 7) {
            const R2 r = load2<C>(fa.V + org, vc + (unsigned)(s0 + d) * pxb);
            v0[d & 7][0] = r.x, v0[d & 7][1] = r.y;
        }
    }
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
            const Mat om = ring[j];
            ring[j] = cm;
            C(*row)[LW] = l.rows[j & 1];
            put(row[0], v0[j]);
            put(row[1], v1[j]);
            C xa[NC], xb[NC], a[NC], b[NC], a2[NC], b2[NC], d[NC], u[NC], u2[NC];
            take(l.ring[0][j4], xa);
            take(l.ring[1][j4], xb);
#pragma unroll
            for (int i = 0; i < NC; i++) {
                v0[(j + 3) & 7][i] = at(cur.v, i);
                a[i] = at(cur.x, i);
                b[i] = at(cur.z, i);
            }
            __syncthreads();
            // ---- first step: Tx, Tz of row s
            xdiff(row[0], v0[j], true, d);
#pragma unroll
            for (int i = 0; i < NC; i++) {
                a[i] = mad(at(cm.mx, i), d[i], a[i]);
                b[i] = mad(at(cm.mz, i), dm8(RING8(v0, j + 4, i), c0, c1, c2, c3), b[i]);
            }
            if (CHECK && q.onA && s >= q.trow0 && s <= q.trow1) {
                inject(s, q.svA, 1, a);
                inject(s, q.svA, 2, b);
            }
            // ---- first step: V of row s-4
            xdiff(l.ring[0][j4], xa, false, d);
            take(l.ring[0][j], a2); // row s-8 of the first step's Tx, Tz goes to the second
#pragma unroll
            for (int i = 0; i < NC; i++) {
                b2[i] = z1[j][i];
                z1[j][i] = b[i];
                u[i] = v0[j4][i];
            }
            if (CHECK && q.onA && s - 4 >= q.trow0 && s - 4 <= q.trow1) inject(s - 4, q.svA, 0, u);
#pragma unroll
            for (int i = 0; i < NC; i++) {
                u[i] = mad(at(cm.bv, i), d[i], u[i]);
                u[i] = mad(at(cm.bv, i), dp8(RING8(z1, j + 1, i), c0, c1, c2, c3), u[i]);
            }
            put(l.ring[0][j], a);
            if (CHECK && s - 4 == nextA) nextA = record(q.ts, rA, u);
            // ---- second step: Tx, Tz of row s-8
            const int rs = s - 8;
            xdiff(row[1], v1[j], true, d);
#pragma unroll
            for (int i = 0; i < NC; i++) {
                a2[i] = mad(at(om.mx, i), d[i], a2[i]);
                b2[i] = mad(at(om.mz, i), dm8(RING8(v1, j + 4, i), c0, c1, c2, c3), b2[i]);
            }
            if (CHECK && q.onB && rs >= q.trow0 && rs <= q.trow1) {
                inject(rs, q.svB, 1, a2);
                inject(rs, q.svB, 2, b2);
            }
            {
                const bool in = rs >= za && rs < zb;
                const unsigned so = in ? (unsigned)rs * pxb : 0u, vo = in ? vst : 0x80000000u;
                store2<C>(oX, vo, so, a2, 1.f);
                store2<C>(oZ, vo, so, b2, 1.f);
            }
            // ---- second step: V of row s-12
            const int rv = s - 12;
            xdiff(l.ring[1][j4], xb, false, d);
#pragma unroll
            for (int i = 0; i < NC; i++) {
                z2[j][i] = b2[i];
                u2[i] = v1[j4][i];
                v1[j4][i] = u[i];
            }
            if (CHECK && q.onB && rv >= q.trow0 && rv <= q.trow1) inject(rv, q.svB, 0, u2);
#pragma unroll
            for (int i = 0; i < NC; i++) {
                u2[i] = mad(at(om.bv, i), d[i], u2[i]);
                u2[i] = mad(at(om.bv, i), dp8(RING8(z2, j + 1, i), c0, c1, c2, c3), u2[i]);
            }
            put(l.ring[1][j], a2);
            {
                const bool in = rv >= za && rv < zb;
                const unsigned so = in ? (unsigned)rv * pxb : 0u, vo = in ? vst : 0x80000000u;
                store2<C>(oV, vo, so, u2, 1.f);
            }
            if (CHECK && rv == nextB) nextB = record(q.ts + 1, rB, u2);
            cur = n1;
            n1 = n2;
            cm = nm;
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#undef RING8
}

template <int MW>
__global__ __launch_bounds__(MW / NC, 2) void k_sh_march(ShFields<float> fa, ShFields<float> fb, ShMat3<float> m,
                                                         Grid g, MarchWork w, FusedEvents ev) {
    __shared__ ShMarchLds<MW> l;
    const int qd = gridDim.x >> 3; // grid padded to a multiple of 8
    const int L = (int)(blockIdx.x & 7) * qd + (int)(blockIdx.x >> 3);
    if (L >= w.nwork) return;
    MarchItem q;
    if (march_find<MW>(g, w, ev, L, q)) sh_march_item<MW, true>(fa, fb, m, g, w, ev, q, l);
    else sh_march_item<MW, false>(fa, fb, m, g, w, ev, q, l);
}

} // namespace fd23
