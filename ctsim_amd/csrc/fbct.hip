// 2D fan-beam projector family for gfx950: distance-driven and separable-footprint
// forward projection (geom/fbct_os/fbct_proj.c fbct_proj_dd :155-291, fbct_proj_tf
// :294-466), their matched backprojections (geom/fbct_os/fbct_back.c fbct_back_dd
// :82-225, fbct_back_tf :227-399) and the pixel-driven FBP backprojection
// (fbct_back_pd :3-80).  2D footprints are not capped (the 3D code caps at 16 cells).
//
// Layouts as in MATLAB: image [nx ny] (x fastest), sinogram [nu nviews].
// Batched forms take a table of independent slices, each with its own geometry,
// and walk a flat work list of (slice, view, tile) or (slice, pixel block) items,
// so slices of uneven size share one launch.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "internal.h"

namespace ctsim {

constexpr int kW2 = 64;
// image lines whose strip holds at least this many pixels on average take a batch each in
// the forward projection (fewer: several lines share a batch)
constexpr int kLineBatch = 12;

enum Foot2 { F2_DD = 0, F2_TF = 1 };

// ---------------------------------------------------------------------------------
// forward, line walk (FP32): one wavefront per (view, 64 detector cells); lanes own cells.
// Along an image line (a row where |Y| >= |X| for the ray from the source, else a column)
// the pixels' footprints meet edge to edge on the detector: the pixel spans the projections
// of its two minor edges, and edge j is shared by pixels j - 1 and j.  So a cell inverts the
// line once, to the pixel ja that holds its first boundary, and sums
//     q_{K-1} + sum_{0 < k < K} c_k (q_{k-1} - q_k),   q = amp * pixel of ja + k,
// where c_k is the part of the cell before edge ja + k (0 at k = 0 and 1 at k = K, which K
// guarantees): sum_k (c_{k+1} - c_k) q_k telescoped, the same products of overlap, amplitude
// and pixel as the pixel-by-pixel footprints.  The edge is measured from the cell's own
// boundary, u_edge - u_cell = sdd/du a dx (j - xi) / d (a: the ray's major direction cosine,
// xi: where the boundary crosses the line, in pixel edges), so nothing cancels.  On an arc
// the same difference is sdd/du atan z with z = (t - k d) / (d + k t) of the order of one
// cell, where z - z^3 / 3 is exact in FP32.  An SF edge is soft: its two corners (the line's
// two sides) bound a ramp, and c_k is one minus the ramp's integral over the cell; with
// |X| dy <= |Y| dx the left pair of a pixel's corners lies before its right pair, as in the
// sorted trapezoid.
// amp = dx / max(|cos|, |sin|) / 10 = dx hypot(X, Y) / max(|X|, |Y|) / 10 with (X, Y) the
// pixel relative to the source.
//
// EACH: fan_lines_each, for tiles that meet a value that is not finite.
//
// Each wave stages kFanWords words of amp * pixel at a time (16 lines of 100 pixels, or 8 of
// 196) in LDS, zero outside the image: amp is formed once per pixel, and image columns are
// read 8 or 16 neighbours at a time instead of one word per image row.  Tiles whose rays
// straddle |X| = |Y| take both walks, each with the other walk's pixels at zero.
// fan_walk_ok (host) says which geometries the walk covers; the rest take the candidate form.
//
// Issue-bound: 47 vector instructions per (line, 64 cells) all told, against some 230 per 64
// pixels of the candidate form below with its LDS min / max.  256^2, 360 views, 512 bins, DD:
// 239 -> 86 us (the pair's few waves wait for issue 41% of their cycles and on counters 31%); 64
// uneven FP16 slices: 18.4 -> 6.1 ms (51% and 13%).  The distance of the pair from 64-bit results
// went from 3.3e-6 to 2.4e-6 (no subtraction of large detector coordinates).
// ---------------------------------------------------------------------------------
constexpr int kFanWaves = 6;     // waves per SIMD the line-walk kernels are compiled for
constexpr int kFanWords = 1600;  // staged words per wave: six 4-wave blocks fit a CU's LDS

struct FanLane {          // one walk, per lane (cell) unless noted
    float rho, cst;       // xi(line) = maj * rho + cst: the cell's first boundary in minor edge units
    float G;              // sdd/du * |major direction| * minor pitch
    float kk;             // slope of that boundary (arc)
    float dconst, cmaj, dd;  // uniform: d of edge j of a line = maj * cmaj + dconst + j * dd
    float tconst, tmaj, dt;  // uniform: t likewise (arc)
    float h, hd;          // SF: the corners sit at xi +- h with denominators +- hd
    float smin, smaj;     // uniform: minor / major coordinate of the source, negated
};

// the staged lines m0 .. m0 + nl - 1 (pitch P words, first word pixel jb) walked by every lane
template <int FOOT, bool ARC, int K>
__device__ __forceinline__ float fan_lines(const FanLane& L, const float* buf, int P, int jb, int m0, int nl, float wmaj,
                                           float dmaj, float inv3) {
    float acc = 0.f;
    const float ah = FOOT == F2_TF ? fabsf(L.h) : 0.f;
    const float dden = ARC ? fmaf(L.kk, L.dt, L.dd) : L.dd;
    const float gh = FOOT == F2_TF ? L.G * L.h : 0.f;
    // the chunk's first line, and what one line adds to xi and to d (d + k t on an arc)
    const float maj = (float(m0) + wmaj) * dmaj;
    const float xi0 = fmaf(maj, L.rho, L.cst), dxi = L.rho * dmaj;
    float den0 = fmaf(maj, L.cmaj, L.dconst), dl = L.cmaj * dmaj;
    if constexpr (ARC) {
        den0 = fmaf(L.kk, fmaf(maj, L.tmaj, L.tconst), den0);
        dl = fmaf(L.kk, L.tmaj * dmaj, dl);
    }
    const float fjb = float(jb), top = float(P - K);
#pragma unroll 2
    for (int i = 0; i < nl; ++i) {
        const float fi = float(i);
        const float xi = fmaf(fi, dxi, xi0);
        const float jf = floorf(xi - ah);
        const float fr = jf - xi;
        const float* pq = buf + (i * P + (int)__builtin_amdgcn_fmed3f(jf - fjb, 0.f, top));
        const float den = fmaf(jf, dden, fmaf(fi, dl, den0));
        float s = pq[K - 1];
#pragma unroll
        for (int k = 1; k < K; ++k) {
            const float dk = fmaf(float(k), dden, den), num = fmaf(fr, L.G, float(k) * L.G);
            float c;
            auto edge = [&](float nu_, float de_) {
                float f = nu_ * frcp(de_);
                if constexpr (ARC) f = fmaf(f * f, -inv3 * f, f);  // sdd/du atan(f du/sdd)
                return f;
            };
            if constexpr (FOOT == F2_DD) {
                c = clamp01(edge(num, dk));
            } else {
                const float e0 = edge(num - gh, dk + L.hd), e1 = edge(num + gh, dk - L.hd);
                const float ea = fminf(e0, e1), eb = fmaxf(e0, e1);
                // 1 - integral over [0, 1] of the ramp from ea to eb
                const float i2 = 0.5f * frcp(fmaxf(eb - ea, 1.0e-20f));
                const float z1 = __builtin_amdgcn_fmed3f(1.f, ea, eb) - ea, z0 = __builtin_amdgcn_fmed3f(0.f, ea, eb) - ea;
                c = 1.f - ((z1 - z0) * (z1 + z0) * i2 + fmaxf(1.f - eb, 0.f) - fmaxf(-eb, 0.f));
            }
            s = fmaf(c, pq[k - 1] - pq[k], s);
        }
        acc += s;
    }
    return acc;
}

// the same lines pixel by pixel, without those that the cell does not overlap: the telescoped sum
// takes a value that is not finite to the cells beside it (0 Inf, Inf - Inf).  K = 4 covers every
// tile.
template <int FOOT, bool ARC>
__device__ __forceinline__ float fan_lines_each(const FanLane& L, const float* buf, int P, int jb, int m0, int nl, float wmaj,
                                                float dmaj, float inv3) {
    constexpr int K = 4;
    float acc = 0.f;
    const float ah = FOOT == F2_TF ? fabsf(L.h) : 0.f;
    const float dden = ARC ? fmaf(L.kk, L.dt, L.dd) : L.dd;
    const float gh = FOOT == F2_TF ? L.G * L.h : 0.f;
#pragma unroll 1
    for (int i = 0; i < nl; ++i) {
        const float maj = (float(m0 + i) + wmaj) * dmaj;
        const float xi = fmaf(maj, L.rho, L.cst);
        const float jf = floorf(xi - ah);
        const float* pq = buf + (i * P + (int)__builtin_amdgcn_fmed3f(jf - float(jb), 0.f, float(P - K)));
        float den = fmaf(jf, dden, fmaf(maj, L.cmaj, L.dconst));
        if constexpr (ARC) den = fmaf(L.kk, fmaf(maj, L.tmaj, L.tconst), den);
        float c0 = 0.f, a0 = 0.f;  // part of the cell before the pixel's first edge, and that edge's start
#pragma unroll 1
        for (int k = 1; k <= K; ++k) {
            const float dk = fmaf(float(k), dden, den), num = ((jf - xi) + float(k)) * L.G;
            auto edge = [&](float nu_, float de_) {
                float f = nu_ * frcp(de_);
                if constexpr (ARC) f = fmaf(f * f, -inv3 * f, f);
                return f;
            };
            float c, a, b;
            if constexpr (FOOT == F2_DD) {
                a = b = edge(num, dk);
                c = clamp01(a);
            } else {
                const float e0 = edge(num - gh, dk + L.hd), e1 = edge(num + gh, dk - L.hd);
                a = fminf(e0, e1);
                b = fmaxf(e0, e1);
                const float i2 = 0.5f * frcp(fmaxf(b - a, 1.0e-20f));
                const float z1 = __builtin_amdgcn_fmed3f(1.f, a, b) - a, z0 = __builtin_amdgcn_fmed3f(0.f, a, b) - a;
                c = 1.f - ((z1 - z0) * (z1 + z0) * i2 + fmaxf(1.f - b, 0.f) - fmaxf(-b, 0.f));
            }
            if (k == K) c = b = 1.f;
            if (a0 < 1.f && b > 0.f) acc = fmaf(c - c0, pq[k - 1], acc);
            c0 = c;
            a0 = a;
        }
    }
    return acc;
}

// the walks of one tile over share `share` of `nshares` of the lines
template <class Tin, int FOOT, bool ARC, bool EACH>
__device__ __forceinline__ float fan_tile(const Geom<float>& g, const View<float>& v, int ut, const Tin* __restrict__ img,
                                          int exhaustive, int share, int nshares, float* buf) {
    const int lane = lane_id();
    const float pm = fmaxf(g.dx, g.dy);
    const float inv3 = ARC ? uni(1.f / (g.sdd_du * g.sdd_du * 3.f)) : 0.f;
    const int iu_a = ut * kW2;
    const float kA = uni(u_to_slope(g, float(iu_a) - 0.5f)), kB = uni(u_to_slope(g, float(iu_a + kW2) - 0.5f));
    // direction of the tile's outer rays: X = s + k c, Y = c - k s
    const float XA = fmaf(kA, v.c, v.s), XB = fmaf(kB, v.c, v.s), YA = fmaf(-kA, v.s, v.c), YB = fmaf(-kB, v.s, v.c);
    const float fx = FOOT == F2_DD ? 1.f : g.dy, fy = FOOT == F2_DD ? 1.f : g.dx;
    // a pixel on a ray may lie a pixel beside it
    const float reach = 0.5f * (float(g.nx) * g.dx + float(g.ny) * g.dy) + fabsf(g.wx + 0.5f * float(g.nx - 1)) * g.dx +
                        fabsf(g.wy + 0.5f * float(g.ny - 1)) * g.dy;
    const float m = 1.f + 4.f * pm * frcp(fmaxf(g.sad - reach, 2.f * pm));
    const bool row = uni((int)(fabsf(XA) * fx <= fabsf(YA) * fy * m || fabsf(XB) * fx <= fabsf(YB) * fy * m)) != 0;
    const bool col = uni((int)(fabsf(YA) * fy <= fabsf(XA) * fx * m || fabsf(YB) * fy <= fabsf(XB) * fx * m)) != 0;
    const bool gen = (row && col) || (FOOT == F2_TF && g.dx != g.dy);
    float acc = 0.f;
#pragma unroll 1
    for (int w = row ? 0 : 1; w < (col ? 2 : 1); ++w) {
        const bool rm = w == 0;
        const int nmin = rm ? g.nx : g.ny, nmaj = rm ? g.ny : g.nx;
        const float dmin = rm ? g.dx : g.dy, dmaj = rm ? g.dy : g.dx;
        const float wmin = rm ? g.wx : g.wy, wmaj = rm ? g.wy : g.wx;
        FanLane L;
        const float cmin = rm ? v.s : v.c, tmin = rm ? v.c : -v.s;
        L.cmaj = rm ? v.c : v.s;
        L.tmaj = rm ? -v.s : v.c;
        L.smin = uni(g.sad * cmin);
        L.smaj = uni(g.sad * L.cmaj);
        // u grows along the minor axis: the first boundary is the cell's lower edge, else its upper
        const bool up = uni((int)(rm ? YA > 0.f : XA < 0.f)) != 0;
        L.kk = u_to_slope(g, float(iu_a + lane) + (up ? -0.5f : 0.5f));
        {
            const float X = fmaf(L.kk, v.c, v.s), Y = fmaf(-L.kk, v.s, v.c);
            const float a = rm ? Y : X, b = rm ? X : Y;
            const float ia = 1.f / (a * dmin);
            L.rho = b * ia;
            L.cst = (rm ? L.kk : -L.kk) * g.sad * ia + (0.5f - wmin);
            L.G = g.sdd_du * fabsf(a) * dmin;
        }
        L.dd = uni(dmin * cmin);
        L.dconst = uni(fmaf(wmin - 0.5f, L.dd, g.sad));
        L.dt = uni(dmin * tmin);
        L.tconst = uni((wmin - 0.5f) * L.dt);
        L.h = 0.5f * dmaj * L.rho;
        L.hd = 0.5f * dmaj * (ARC ? fmaf(L.kk, L.tmaj, L.cmaj) : L.cmaj);
        // the tile's first and last boundaries; the pixels a cell can meet, at the tile's ends and
        // the first and last line (the width is monotone along the tile and linear along the lines)
        const float rho0 = rdl(L.rho, 0), rho1 = rdl(L.rho, kW2 - 1), cst0 = rdl(L.cst, 0), cst1 = rdl(L.cst, kW2 - 1);
        const float y0 = wmaj * dmaj, y1 = (float(nmaj - 1) + wmaj) * dmaj;
        const float hm = FOOT == F2_TF ? uni(fmaxf(fabsf(rdl(L.h, 0)), fabsf(rdl(L.h, kW2 - 1)))) : 0.f;
        auto width = [&](int l0, int l1, float y) {
            return fabsf(fmaf(y, rdl(L.rho, l1) - rdl(L.rho, l0), rdl(L.cst, l1) - rdl(L.cst, l0)));
        };
        const float wpx = fmaf(fmaxf(fmaxf(width(0, 1, y0), width(0, 1, y1)),
                                     fmaxf(width(kW2 - 2, kW2 - 1, y0), width(kW2 - 2, kW2 - 1, y1))),
                               1.05f, 2.f * hm + 0.01f);
        const int K = uni(EACH ? 4 : wpx <= 1.f ? 2 : wpx <= 2.f ? 3 : 4);
        // staged width of one line, its drift from line to line, and the lines per chunk
        const float span = fmaxf(width(0, kW2 - 1, y0), width(0, kW2 - 1, y1)) + 2.f * hm + float(K + 4);
        const float drift = fmaxf(fabsf(rho0), fabsf(rho1)) * dmaj;
        const int lg = uni(span + 16.f * drift <= 100.f ? 4 : 3);  // log2 of the lines per chunk
        const int NL = 1 << lg, P = lg == 4 ? 100 : 196;           // pitches are 4 mod 64: no bank conflicts
        const int rounds = uni(min((int)span, P - 1) / kW2 + 1);   // 64-pixel loads per line
        const int mb = nmaj * share / nshares, me = nmaj * (share + 1) / nshares;
        for (int m0 = mb; m0 < me; m0 += NL) {
            const int nl = min(NL, me - m0);
            // minor range that the chunk's lines can read
            const float ya = (float(m0) + wmaj) * dmaj, yb = (float(m0 + nl - 1) + wmaj) * dmaj;
            const float x00 = fmaf(ya, rho0, cst0), x01 = fmaf(ya, rho1, cst1);
            const float x10 = fmaf(yb, rho0, cst0), x11 = fmaf(yb, rho1, cst1);
            const float xlo = fminf(fminf(x00, x01), fminf(x10, x11)) - hm;
            const float xhi = fmaxf(fmaxf(x00, x01), fmaxf(x10, x11)) + hm;
            if (!exhaustive && (xhi < -float(K) || xlo > float(nmin))) continue;  // beside the image
            // (clamped so that chunks far outside the image convert to integers)
            const int jb = uni((int)floorf(__builtin_amdgcn_fmed3f(xlo, -1.0e6f, 1.0e6f)) - 1);
            // hypot(X, Y) / max(|X|, |Y|) * pixel at minor coordinate mn of the line at major
            // coordinate mj from the source (rmj = 1 / mj)
            auto weighed = [&](auto gen_k, float mn, float pix, float mj, float rmj) -> float {
                if constexpr (decltype(gen_k)::value) {
                    const float am = fabsf(mn), aj = fabsf(mj);
                    // (DD: the x edges where |Y| > |X|, as the reference's cos > sin; SF: the
                    // walk whose edges' corners keep their order)
                    const float l = FOOT == F2_DD ? aj : aj * dmin, r = FOOT == F2_DD ? am : am * dmaj;
                    pix = (rm ? l > r : l >= r) ? pix : 0.f;
                    return pix * (fsqrt(fmaf(mn, mn, mj * mj)) * frcp(fmaxf(am, aj)));
                } else {
                    const float q = mn * rmj;
                    return pix * fsqrt(fmaf(q, q, 1.f));
                }
            };
            // minor and major coordinate of pixel 0 from the source.  Both walks form a pixel's
            // coordinates with the same operations, so that on the diagonal exactly one keeps it
            const float cmn = uni(fmaf(wmin, dmin, L.smin)), cmj = uni(fmaf(wmaj, dmaj, L.smaj));
            // pixels outside the image read zero through the resources' ranges (a line's, or the
            // image's where a column index runs along the lines of a chunk)
            auto fill = [&](auto gen_k) {
                if (rm) {
                    // lane i: first pixel and major coordinate of line m0 + i; then four lines of
                    // 64 pixels at a time (lines past the chunk read and store zeros)
                    const float yl = (float(m0 + lane) + wmaj) * dmaj;
                    const float xs = fminf(fmaf(yl, rho0, cst0), fmaf(yl, rho1, cst1)) - hm;
                    const int first = max(jb, (int)floorf(__builtin_amdgcn_fmed3f(xs, -1.0e6f, 1.0e6f)) - 1);
                    const float mjl = fmaf(float(m0 + lane), dmaj, cmj), rmjl = frcp(mjl);
                    for (int c = 0; c < rounds; ++c) {
                        const Tin* line = img + (size_t)m0 * g.nx;
                        const int lc = c * kW2 + lane;
                        int row = -jb * 4;  // bytes from pixel 0's word to the line's first word
                        for (int i0 = 0; i0 < nl; i0 += 4) {
                            Tin pv[4];
                            int jj[4];
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                jj[e] = rdl_i(first, i0 + e) + lc;
                                pv[e] = buf_ld<Tin>(buf_rsrc(line, i0 + e < nl ? g.nx * (int)sizeof(Tin) : 0),
                                                    jj[e] * (int)sizeof(Tin));
                                line += g.nx;
                            }
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const float w = weighed(gen_k, fmaf(float(jj[e]), dmin, cmn), to_f(pv[e]), rdl(mjl, i0 + e),
                                                        rdl(rmjl, i0 + e));
                                // pixels past the pitch fall on its last word, which no cell reads
                                *(float*)((char*)buf + (row + min(jj[e] * 4, (jb + P - 1) * 4))) = w;
                                row += P * 4;
                            }
                        }
                    }
                } else {
                    // NL neighbouring image columns of 64 / NL rows per load, four loads at a time
                    const int i = lane & (NL - 1), dr = kW2 >> lg;
                    const float mj = fmaf(float(m0 + i), dmaj, cmj), rmj = frcp(mj);
                    const int jn = uni(min(P, (int)fminf(xhi - xlo, 1.0e6f) + K + 4));
                    const auto rs = buf_rsrc(img, g.nx * g.ny * (int)sizeof(Tin));
                    const int step = dr * g.nx * (int)sizeof(Tin);
                    int r = lane >> lg;
                    int off = ((jb + r) * g.nx + (m0 + i)) * (int)sizeof(Tin);
                    float* dst = buf + i * P;
                    for (int r0 = 0; r0 < jn; r0 += 4 * dr) {
                        Tin pv[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) pv[e] = buf_ld<Tin>(rs, off + e * step);
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            dst[min(r + e * dr, P - 1)] = weighed(gen_k, fmaf(float(jb + r + e * dr), dmin, cmn), to_f(pv[e]), mj, rmj);
                        r += 4 * dr;
                        off += 4 * step;
                    }
                }
            };
            if (gen) fill(std::true_type{});
            else fill(std::false_type{});
            __builtin_amdgcn_wave_barrier();
            if constexpr (EACH) acc += fan_lines_each<FOOT, ARC>(L, buf, P, jb, m0, nl, wmaj, dmaj, inv3);
            else if (K == 2) acc += fan_lines<FOOT, ARC, 2>(L, buf, P, jb, m0, nl, wmaj, dmaj, inv3);
            else if (K == 3) acc += fan_lines<FOOT, ARC, 3>(L, buf, P, jb, m0, nl, wmaj, dmaj, inv3);
            else acc += fan_lines<FOOT, ARC, 4>(L, buf, P, jb, m0, nl, wmaj, dmaj, inv3);
            __builtin_amdgcn_wave_barrier();
        }
    }
    return acc * (g.dx * 0.1f);
}

// ---------------------------------------------------------------------------------
// forward, candidate form (FP64, and geometries outside the line walk): candidate
// pixels of the strip are evaluated 64 at a time (one per lane) into LDS entries, and
// every tile cell notes the first and the last entry whose footprint covers it (LDS
// min / max, order-free).  Each lane then walks the entries of its own cell range in
// candidate order, so a cell adds the same products in the same order as a walk over
// all candidates would, and a pixel costs the few lanes it covers, not the whole wave.
// ---------------------------------------------------------------------------------
// share `share` of `nshares` of the strip (its rows or columns along the major axis):
// returns this lane's cell sum.  Called by whole 256-thread blocks (four waves).
template <class Tin, class T, int FOOT>
__device__ __forceinline__ T fbct_proj_acc(const Geom<T>& g, const View<T>& v, int ut, const Tin* __restrict__ img,
                                           int exhaustive, int share, int nshares) {
    __shared__ T ep[4][FOOT == F2_DD ? 2 : 4][kW2];  // footprint parameters of the entries
    __shared__ T eval_[4][kW2];                        // amp * pixel value
    __shared__ int ecell[4][kW2];                      // ilo | ihi << 16 (empty: ilo 1 > ihi 0)
    __shared__ int cfirst[4][kW2], clast[4][kW2];      // per tile cell: first and last entry
    const int wv = (int)(threadIdx.x / kW2);
    const int lane = lane_id();
    const int iu_a = ut * kW2;
    const int iu_b = min(iu_a + kW2, g.nu) - 1;
    const int iu = iu_a + lane;
    const bool row_major = fabs_t(v.c) >= fabs_t(v.s);
    const int nmajor = row_major ? g.ny : g.nx;
    const int m_begin = nmajor * share / nshares, m_end = nmajor * (share + 1) / nshares;
    const T kL = u_to_slope(g, T(iu_a) - T(0.5));
    const T kR = u_to_slope(g, T(iu_b) + T(0.5));
    T acc = T(0);
    for (int m0 = m_begin; m0 < m_end; m0 += kW2) {
        const int m = m0 + lane;
        int lo = 0, hi = -1;
        if (m < m_end) {
            if (!strip_range(g, v, row_major, m, kL, kR, exhaustive != 0, lo, hi)) hi = lo - 1;
        }
        const int cnt = hi - lo + 1 > 0 ? hi - lo + 1 : 0;
        const int incl = wave_incl_scan(cnt);
        const int excl = incl - cnt;
        const int total = rdl_i(incl, kW2 - 1);
        // one batch of 64 candidates: entries in LDS, the covering range of every tile cell,
        // then each lane's walk over that range
        auto batch = [&](int major, int minor, bool ok) {
            const int ix = row_major ? minor : major;
            const int iy = row_major ? major : minor;
            int ilo = 0, ihi = -1;
            T p0 = T(0), p1 = T(0), p2 = T(0), p3 = T(0), val = T(0);
            // the pixel is loaded before its footprint is known (every candidate lies inside
            // the image), so that the load's latency overlaps the footprint arithmetic
            T pix = T(0);
            if (ok) pix = ld<T>(img + (size_t)iy * g.nx + ix);
            if (ok) {
                const T xc = (T(ix) + g.wx) * g.dx, yc = (T(iy) + g.wy) * g.dy;
                const Column<T> cg = column_geom(xc, yc, v, g.sad, g.dx);
                T clo, chi;
                if (FOOT == F2_DD) {
                    T umin, umax;
                    dd_bounds(cg, v, g, umin, umax);
                    ok = clamp_cells(umin, umax, g.nu, 0, clo, chi, ilo, ihi);
                    p0 = clo;
                    p1 = chi;
                } else {
                    T tau[4];
                    sf_taus(cg, v, g, tau);
                    ok = clamp_cells(tau[0], tau[3], g.nu, 0, clo, chi, ilo, ihi);
                    p0 = tau[0]; p1 = tau[1]; p2 = tau[2]; p3 = tau[3];
                }
                ok = ok && ihi >= iu_a && ilo <= iu_b;
                if (ok) val = cg.amp * pix;
            }
            ecell[wv][lane] = ok ? (ilo | (ihi << 16)) : 1;
            ep[wv][0][lane] = p0;
            ep[wv][1][lane] = p1;
            if constexpr (FOOT == F2_TF) {
                ep[wv][2][lane] = p2;
                ep[wv][3][lane] = p3;
            }
            eval_[wv][lane] = val;
            cfirst[wv][lane] = kW2;
            clast[wv][lane] = -1;
            __builtin_amdgcn_wave_barrier();
            if (ok) {
                const int c1 = min(ihi, iu_b) - iu_a;
                for (int c = max(ilo, iu_a) - iu_a; c <= c1; ++c) {
                    atomicMin(&cfirst[wv][c], lane);
                    atomicMax(&clast[wv][c], lane);
                }
            }
            __builtin_amdgcn_wave_barrier();
            const int jl = clast[wv][lane];
            for (int e = cfirst[wv][lane]; e <= jl; ++e) {
                const int cl = ecell[wv][e];
                const int cilo = cl & 0xffff, cihi = cl >> 16;
                if (iu >= cilo && iu <= cihi) {
                    const T cp0 = ep[wv][0][e], cp1 = ep[wv][1][e];
                    T w;
                    if constexpr (FOOT == F2_DD) {
                        w = dd_weight(iu, cp0, cp1, cilo, cihi);
                    } else {
                        w = sf_weight(iu, cp0, cp1, ep[wv][2][e], ep[wv][3][e]);
                    }
                    acc += w * eval_[wv][e];
                }
            }
            __builtin_amdgcn_wave_barrier();
        };
        const unsigned long long nonempty = __ballot(cnt > 0);
        const int nlines = __popcll(nonempty);
        if (total >= kLineBatch * nlines) {
            // wide strips: one image line per batch.  The pixels of a line project in order,
            // so the ones covering a cell are consecutive entries and each lane's walk is as
            // long as its cell's coverage, where a batch spanning several lines walks the
            // entries of every line in between
            unsigned long long left = nonempty;
            while (left) {
                const int j = __ffsll((long long)left) - 1;
                left &= left - 1;
                const int lo_j = rdl_i(lo, j), cnt_j = rdl_i(cnt, j);
                for (int k0 = 0; k0 < cnt_j; k0 += kW2) batch(m0 + j, lo_j + k0 + lane, k0 + lane < cnt_j);
            }
        } else {
            // narrow strips: consecutive candidates of several lines share a batch
            for (int k0 = 0; k0 < total; k0 += kW2) {
                const int k = k0 + lane;
                int j = 0;
#pragma unroll
                for (int step = 32; step >= 1; step >>= 1) {
                    const int e = __shfl(excl, j + step, 64);
                    if (e <= k) j += step;
                }
                const int lo_j = __shfl(lo, j, 64);
                const int ex_j = __shfl(excl, j, 64);
                batch(m0 + j, lo_j + (k - ex_j), k < total);
            }
        }
    }
    return acc;
}

template <class T, int S>
__device__ __forceinline__ T combine_shares(T (*part)[kW2], int wv, int lane) {
    const int w0 = wv - wv % S;
    if (S == 1) return part[w0][lane];
    if (S == 2) return part[w0][lane] + part[w0 + 1][lane];
    return (part[w0][lane] + part[w0 + 1][lane]) + (part[w0 + 2][lane] + part[w0 + 3][lane]);
}

// S waves share a (view, tile) item, each walking 1/S of the strip's lines; the partial
// sums are added in a fixed order.  S = 4 when the items alone would leave the chip
// with few waves.
// FORM 0: candidates; 1: line walk, flat detector; 2: line walk, arc
template <class Tin, class T, int FOOT, int FORM>
__device__ __forceinline__ T fbct_proj_item(const Geom<T>& g, const View<T>& v, int ut, const Tin* __restrict__ img,
                                            int exhaustive, int share, int nshares) {
    if constexpr (FORM == 0) {
        return fbct_proj_acc<Tin, T, FOOT>(g, v, ut, img, exhaustive, share, nshares);
    } else {
        __shared__ __align__(16) float buf[4][kFanWords];
        float* const b = buf[threadIdx.x / kW2];
        const float acc = fan_tile<Tin, FOOT, FORM == 2, false>(g, v, ut, img, exhaustive, share, nshares, b);
        // a value that is not finite stays with the cells that it weighs on: the sums of those that
        // came out not finite again, pixel by pixel.  (In the arc kernels whose waves share a tile
        // the second copy of the walk costs one to three spilled registers, 0 to 9% for images of
        // up to 64^2 pixels.)
        if (__builtin_expect(!__any(!__builtin_isfinite(acc)), 1)) return acc;
        const float each = fan_tile<Tin, FOOT, FORM == 2, true>(g, v, ut, img, exhaustive, share, nshares, b);
        return __builtin_isfinite(acc) ? acc : each;
    }
}

template <class Tin, class Tout, class T, int FOOT, int S, int FORM>
__global__ __launch_bounds__(256, FORM ? kFanWaves : 1) void fbct_proj_kernel(Geom<T> g, const View<T>* __restrict__ views, int vstride,
                                                        int nviews, const Tin* __restrict__ img,
                                                        Tout* __restrict__ proj, int exhaustive) {
    __shared__ T part[4][kW2];
    const int nut = (g.nu + kW2 - 1) / kW2;
    const int wv = (int)(threadIdx.x / kW2), lane = lane_id();
    const int wid = blockIdx.x * (4 / S) + wv / S;
    const bool valid = wid < nviews * nut;
    // longest work first: every view's tile of the central ray, then the tiles beside it
    const int ut = valid ? tile_by_rank(wid / nviews, min(max((int)floor(-g.wu / T(kW2)), 0), nut - 1), nut) : 0;
    const int b = valid ? wid % nviews : 0;
    T acc = T(0);
    if (valid) {
        // the view in registers (a wave-uniform index: scalar loads, once per item), so that
        // the walk's LDS atomics and barriers do not make the compiler reload it every batch
        const View<T> vw = views[(size_t)uni(b) * vstride];
        // (the tile in a scalar register is for the line walk: it cost the candidate form 1 to 3%,
        // SF of 512^2 at 0.5 mm on 1024 bins of 0.8 mm, 984 views, 2410 against 2447 us)
        acc = fbct_proj_item<Tin, T, FOOT, FORM>(g, vw, FORM ? uni(ut) : ut, img, exhaustive, wv % S, S);
    }
    if (S > 1) {
        part[wv][lane] = acc;
        __syncthreads();
        if (wv % S) return;
        acc = combine_shares<T, S>(part, wv, lane);
    }
    const int iu = ut * kW2 + lane;
    if (valid && iu < g.nu) proj[(size_t)b * g.nu + iu] = cvt_store<Tout>(acc);
}

// ---------------------------------------------------------------------------------
// matched backprojection (DD / SF) and pixel-driven backprojection: lanes own 64
// consecutive pixels of a row; the 4 waves of a block split the views into four
// contiguous ranges and their partial sums are added in a fixed order.
// ---------------------------------------------------------------------------------
// One view's matched backprojection of pixel (xc, yc), FP32: amp * sum_i w_i row_i.  The
// first three footprint cells are loaded at once through the row's resource (cells past the
// detector read zero), wider footprints loop over the rest.
//   amp = dx hypot(X, Y) / max(|X|, |Y|) / 10, (X, Y) the pixel relative to the source: the
//     ray's cosines are |Y| and |X| over hypot(X, Y), so no normalised direction is formed;
//   DD: cell k of [lo, hi] weighs min(hi, k + 1) - max(lo, k);
//   SF: cell k weighs C(k + 1) - C(k), C the trapezoid's running integral, the difference of
//     its two ramps' integrals; two reciprocals per pixel where the per-cell form takes two
//     per cell.
// Bound by instruction issue where there are waves enough: 98 -> 56 (DD) vector instructions per
// 64 pixel-views, with the views through scalar loads.  64 uneven FP16 slices: 7.5 -> 4.3 ms;
// 256^2, 360 views, DD: 75 -> 43 us (16 waves per CU, which wait on counters 42% of their cycles).
// The cells are returned as loaded: the caller evaluates a second view's footprint before it
// uses them.
// EACH: only cells that the footprint reaches are read.  Without it (DD) those after its end weigh
// exactly nothing, which keeps them out of the sum unless they are not finite; SF weights there
// are differences of rounded integrals, and beside the detector they grow with the distance.
// (Reading each in DD too: 41.3 -> 43.1 us above, 327 -> 355 us for 512^2 from 984 views; SF pays
// 86.2 -> 87.2 and 743 -> 765.)
template <class Tin>
struct BackView {
    Tin p0, p1, p2;
    float w0, w1, w2, rest;  // weights times amp; the sum of the cells past the third
};
struct BackEdges {
    float lo, hi;          // the footprint's ends, on the detector or not
    float t0, t1, t2, t3;  // SF: the trapezoid's corners
    float amp;
};
template <int KIND>
__device__ __forceinline__ BackEdges fbct_back_edges(const Geom<float>& g, const View<float>& v, float xc, float yc) {
    const float t = xc * v.c - yc * v.s, d = fmaf(yc, v.c, fmaf(xc, v.s, g.sad));
    const float X = fabsf(fmaf(g.sad, v.s, xc)), Y = fabsf(fmaf(g.sad, v.c, yc));
    BackEdges e;
    e.amp = fsqrt(fmaf(X, X, Y * Y)) * frcp(fmaxf(X, Y)) * (g.dx * 0.1f);
    const float half = 0.5f - g.wu;
    auto det = [&](float num, float den) {
        const float q = num * frcp(den);
        return fmaf(g.sdd_du, g.dettype == 1 ? q : atanf(q), half);
    };
    e.t0 = e.t1 = e.t2 = e.t3 = 0.f;
    if constexpr (KIND == 0) {
        const bool xdom = Y > X;
        // (through uni, so that the choice is made between registers and not between addresses)
        const float a = xdom ? uni(v.dxc2) : uni(v.dys2), b = xdom ? uni(v.dxs2) : uni(v.ndyc2);
        const float u0 = det(t + a, d + b), u1 = det(t - a, d - b);
        e.lo = fminf(u0, u1);
        e.hi = fmaxf(u0, u1);
    } else {
        const float ax = v.dxc2 + v.dys2, bx = v.dxs2 + v.ndyc2, ay = v.dxc2 - v.dys2, by = v.dxs2 - v.ndyc2;
        e.t0 = det(t + ax, d + bx);
        e.t1 = det(t - ay, d - by);
        e.t2 = det(t + ay, d + by);
        e.t3 = det(t - ax, d - bx);
        cswap(e.t0, e.t1);
        cswap(e.t2, e.t3);
        cswap(e.t0, e.t2);
        cswap(e.t1, e.t3);
        cswap(e.t1, e.t2);
        e.lo = e.t0;
        e.hi = e.t3;
    }
    return e;
}

template <class Tin, int KIND, bool EACH>
__device__ __forceinline__ BackView<Tin> fbct_back_view(const Geom<float>& g, const BackEdges& ed, const Tin* __restrict__ row) {
    const float lo = ed.lo, hi = ed.hi, t0 = ed.t0, t1 = ed.t1, t2 = ed.t2, t3 = ed.t3, amp = ed.amp;
    const float fn = float(g.nu);
    const float cl = __builtin_amdgcn_fmed3f(lo, 0.f, fn), ch = __builtin_amdgcn_fmed3f(hi, 0.f, fn);
    const int ilo = (int)cl;  // cl >= 0: truncation is floor
    const float f = __builtin_amdgcn_fractf(cl), fi = cl - f, h = ch - fi;
    const auto rs = buf_rsrc(row, g.nu * (int)sizeof(Tin));
    const int off = ilo * (int)sizeof(Tin);
    BackView<Tin> r;
    // where x < 0, an offset past the row (loads give zero there)
    auto reach = [&](float x) { return EACH ? off | (__float_as_int(x) & (int)0x80000000u) : off; };
    r.p0 = buf_ld<Tin>(rs, reach(hi));
    r.p1 = buf_ld<Tin>(rs, reach(h - 1.f) + (int)sizeof(Tin));
    r.p2 = buf_ld<Tin>(rs, reach(h - 2.f) + 2 * (int)sizeof(Tin));
    float s = 0.f;
    if constexpr (KIND == 0) {
        r.w0 = (fminf(h, 1.f) - f) * amp;
        r.w1 = clamp01(h - 1.f) * amp;
        r.w2 = clamp01(h - 2.f) * amp;
        if (h > 3.f)
            for (int k = 3; float(k) < h; ++k) s += fminf(h - float(k), 1.f) * to_f(buf_ld<Tin>(rs, off + k * (int)sizeof(Tin)));
    } else {
        const float ia = 0.5f * frcp(fmaxf(t1 - t0, 1.0e-20f)), ib = 0.5f * frcp(fmaxf(t3 - t2, 1.0e-20f));
        // integral of the trapezoid up to cell edge fi + k
        auto cum = [&](float k) {
            const float e = fi + k;
            const float a = __builtin_amdgcn_fmed3f(e, t0, t1) - t0, b = __builtin_amdgcn_fmed3f(e, t2, t3) - t2;
            return fmaf(a * a, ia, fmaxf(e - t1, 0.f)) - fmaf(b * b, ib, fmaxf(e - t3, 0.f));
        };
        float c0 = cum(0.f);  // zero unless the footprint starts before the detector
        const float c1 = cum(1.f), c2 = cum(2.f);
        float c3 = cum(3.f);
        r.w0 = (c1 - c0) * amp;
        r.w1 = (c2 - c1) * amp;
        r.w2 = (c3 - c2) * amp;
        if (h > 3.f)
            for (int k = 3; float(k) < h; ++k) {
                c0 = c3;
                c3 = cum(float(k + 1));
                s += (c3 - c0) * to_f(buf_ld<Tin>(rs, off + k * (int)sizeof(Tin)));
            }
    }
    r.rest = amp * s;
    return r;
}

// a view of the table at a wave-uniform index through scalar loads (the pointer of a batch's
// slice comes from memory, which alone would make them flat vector loads with their latency in
// every view)
__device__ __forceinline__ View<float> load_view(const View<float>* p) {
    const auto* q = (const __attribute__((address_space(4))) float*)(const void*)p;
    return View<float>{q[0], q[1], q[2], q[3], q[4], q[5], q[6], q[7]};
}

// KIND 0 dd, 1 tf, 2 pd; SKIP: leave a pair of views at its footprints where no pixel of the wave
// lies before the detector (fan_back_skips says when)
template <class Tin, class T, int KIND, bool SKIP>
__device__ __forceinline__ T fbct_back_pixel(const Geom<T>& g, const View<T>* __restrict__ views, int vstride, int b0,
                                             int b1, int ix, int iy, const Tin* __restrict__ proj) {
    T img = T(0);
    if (ix >= g.nx) return img;
    const T xc = (T(ix) + g.wx) * g.dx, yc = (T(iy) + g.wy) * g.dy;
    if constexpr (KIND != 2 && sizeof(T) == 4) {
        auto sum = [&](auto each_k) {
            constexpr bool E = decltype(each_k)::value;
            float acc = 0.f;
            auto view = [&](int b) { return load_view(views + (size_t)b * vstride); };
            auto edges = [&](const View<float>& v) { return fbct_back_edges<KIND>(g, v, xc, yc); };
            auto cells = [&](int b, const BackEdges& e) { return fbct_back_view<Tin, KIND, E>(g, e, proj + (size_t)b * g.nu); };
            auto add = [&](const BackView<Tin>& r) {
                acc += fmaf(r.w2, to_f(r.p2), fmaf(r.w1, to_f(r.p1), fmaf(r.w0, to_f(r.p0), r.rest)));
            };
            int b = b0;
            for (; b + 1 < b1; b += 2) {
                const View<float> v0 = view(b), v1 = view(b + 1);  // (both before either is used)
                BackView<Tin> r0, r1;
                if constexpr (SKIP) {
                    const BackEdges e0 = edges(v0), e1 = edges(v1);
                    if (!__any(!(fmaxf(e0.hi, e1.hi) < 0.f) && !(fminf(e0.lo, e1.lo) > float(g.nu)))) continue;
                    r0 = cells(b, e0);
                    r1 = cells(b + 1, e1);
                } else {
                    r0 = cells(b, edges(v0));
                    r1 = cells(b + 1, edges(v1));
                }
                add(r0);
                add(r1);
            }
            if (b < b1) add(cells(b, edges(view(b))));
            return acc;
        };
        if constexpr (KIND == 1 || SKIP) return sum(std::true_type{});
        img = sum(std::false_type{});
        // a value that is not finite stays with the pixels whose footprints reach it: their sums
        // again, without the cells beside them
        if (__any(!__builtin_isfinite(img))) {
            const float each = sum(std::true_type{});
            img = __builtin_isfinite(img) ? img : each;
        }
        return img;
    }
    for (int b = b0; b < b1; ++b) {
        const View<T> v = views[(size_t)b * vstride];
        const Tin* row = proj + (size_t)b * g.nu;
        if (KIND == 2) {
            const T xr = xc * v.c - yc * v.s;
            const T yr = xc * v.s + yc * v.c;
            T u, w2s;
            if (g.dettype == 1) {
                const T w2 = g.sdd / (g.sad + yr);
                w2s = w2 * w2;
                u = xr * w2 / g.du - g.wu;
            } else {
                const T roff = g.ou * g.sad / g.sdd;
                u = atan((xr - roff) / (g.sad + yr)) * g.sdd / g.du - g.wu;
                w2s = g.sdd * g.sdd / ((g.sad + yr) * (g.sad + yr) + (xr - roff) * (xr - roff));
            }
            if (!((double)u >= 1e-6 && (double)u <= (double)(g.nu - 1) - 1e-6)) continue;  // also skips NaN
            const int iu = (int)floor(u);
            const T wl = u - T(iu);
            img += w2s * ((T(1) - wl) * ld<T>(row + iu) + wl * ld<T>(row + iu + 1));
            continue;
        }
        const Column<T> cg = column_geom(xc, yc, v, g.sad, g.dx);
        T clo, chi, p0, p1, p2 = T(0), p3 = T(0);
        int ilo, ihi;
        bool ok;
        if (KIND == 0) {
            T umin, umax;
            dd_bounds(cg, v, g, umin, umax);
            ok = clamp_cells(umin, umax, g.nu, 0, clo, chi, ilo, ihi);
            p0 = clo;
            p1 = chi;
        } else {
            T tau[4];
            sf_taus(cg, v, g, tau);
            ok = clamp_cells(tau[0], tau[3], g.nu, 0, clo, chi, ilo, ihi);
            p0 = tau[0]; p1 = tau[1]; p2 = tau[2]; p3 = tau[3];
        }
        if (!ok) continue;
        T s = T(0);
        for (int iu = ilo; iu <= ihi; ++iu) {
            const T w = KIND == 0 ? dd_weight(iu, p0, p1, ilo, ihi) : sf_weight(iu, p0, p1, p2, p3);
            s += w * ld<T>(row + iu);
        }
        img += cg.amp * s;
    }
    return img;
}

template <class Tin, class Tout, class T, int KIND, bool SKIP>
__global__ __launch_bounds__(256) void fbct_back_kernel(Geom<T> g, const View<T>* __restrict__ views, int vstride,
                                                        int nviews, const Tin* __restrict__ proj,
                                                        Tout* __restrict__ img, T scale) {
    __shared__ T part[3][kW2];
    const int nxb = (g.nx + kW2 - 1) / kW2;
    const int iy = blockIdx.x / nxb;
    const int ix = (blockIdx.x % nxb) * kW2 + lane_id();
    const int w = uni((int)(threadIdx.x / kW2));  // wave-uniform, so that the views come through scalar loads
    const int per = (nviews + 3) / 4;
    const int b0 = min(w * per, nviews), b1 = min(b0 + per, nviews);
    const T s = fbct_back_pixel<Tin, T, KIND, SKIP>(g, views, vstride, b0, b1, ix, iy, proj);
    if (w > 0) part[w - 1][lane_id()] = s;
    __syncthreads();
    if (w == 0 && ix < g.nx) {
        const T tot = (s + part[0][lane_id()]) + (part[1][lane_id()] + part[2][lane_id()]);
        img[(size_t)iy * g.nx + ix] = cvt_store<Tout>(scale * tot);
    }
}

// ---------------------------------------------------------------------------------
// Batched uneven slices in one launch.  items are (slice, view, u-tile) for the
// forward and (slice, row, 64-pixel block) for the back pass; a wave finds its slice
// by binary search over the slices' first item.  One launch covers the whole batch.
// ---------------------------------------------------------------------------------
template <class T>
__device__ __forceinline__ int find_slice(const Slice2<T>* __restrict__ sl, int nslices, int item) {
    int lo = 0, hi = nslices - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sl[mid].item0 <= item) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Schedules: the forward pass splits each (slice, view, tile) item's strip over S waves
// of a block (S = 1, 2, 4; the shares are added in a fixed order); the back pass splits
// each (slice, row, 64-pixel) item's views over VS waves (VS = 1, 2, 4).  A block is
// always 4 waves and holds 4/S (4/VS) items.
template <class Tin, class Tout, class T, int FOOT, int S, int FORM>
__global__ __launch_bounds__(256, FORM ? kFanWaves : 1) void fbct_proj_batch_kernel(const Slice2<T>* __restrict__ sl, int nslices,
                                                              int nitems, const Tin* __restrict__ img,
                                                              Tout* __restrict__ proj) {
    __shared__ T part[4][kW2];
    // blocks in dispatch order (consecutive blocks on different XCDs): a slice's items, longest
    // first, spread over the chip (a contiguous range of the list per XCD, which would keep a
    // slice's 0.5 MB image in one L2, measured 18% slower: it leaves the XCDs unevenly loaded)
    const int bid = blockIdx.x;
    const int wv = (int)(threadIdx.x / kW2), lane = lane_id();
    const int item = bid * (4 / S) + wv / S;
    const bool valid = item < nitems;
    T acc = T(0);
    int si = 0, ut = 0, b = 0;
    if (valid) {
        // the item's slice geometry and view in registers (wave-uniform indices: scalar loads,
        // once per item), so that the walk's LDS atomics and barriers do not make the
        // compiler reload them from the slice table every batch
        si = uni(find_slice(sl, nslices, item));
        const Slice2<T>& s = sl[si];
        const Geom<T> g = s.g;
        const int local = item - s.item0;
        const int nut = (g.nu + kW2 - 1) / kW2;
        // within the slice, longest work first (the tiles around the central ray's)
        ut = uni(tile_by_rank(local / s.nviews, min(max((int)floor(-g.wu / T(kW2)), 0), nut - 1), nut));
        b = uni(local % s.nviews);
        const View<T> vw = s.views[b];
        acc = fbct_proj_item<Tin, T, FOOT, FORM>(g, vw, ut, img + s.img_off, 0, wv % S, S);
    }
    if (S > 1) {
        part[wv][lane] = acc;
        __syncthreads();
        if (wv % S) return;
        acc = combine_shares<T, S>(part, wv, lane);
    }
    if (!valid) return;
    const Slice2<T>& s = sl[si];
    const int iu = ut * kW2 + lane;
    if (iu < s.g.nu) proj[s.sino_off + (size_t)b * s.g.nu + iu] = cvt_store<Tout>(acc);
}

template <class Tin, class Tout, class T, int KIND, int VS, bool SKIP>
__global__ __launch_bounds__(256) void fbct_back_batch_kernel(const Slice2<T>* __restrict__ sl, int nslices,
                                                              int nitems, const Tin* __restrict__ proj,
                                                              Tout* __restrict__ img) {
    __shared__ T part[4][kW2];
    // blocks in dispatch order, as in the forward (a contiguous range per XCD measured 19%
    // slower here too)
    const int bid = blockIdx.x;
    const int wv = (int)(threadIdx.x / kW2), lane = lane_id();
    const int item = bid * (4 / VS) + wv / VS;
    const bool valid = item < nitems;
    T v = T(0);
    int si = 0, ix = 0, iy = 0;
    if (valid) {
        // the item's slice geometry in registers (a wave-uniform index: scalar loads, once
        // per item) rather than read from the slice table inside the view loop
        si = uni(find_slice(sl, nslices, item));
        const Slice2<T>& s = sl[si];
        const Geom<T> g = s.g;
        const View<T>* views = s.views;
        const int nviews = uni(s.nviews);
        const int local = item - s.item0;
        const int nxb = (g.nx + kW2 - 1) / kW2;
        iy = local / nxb;
        ix = (local % nxb) * kW2 + lane;
        const int share = uni(wv % VS);
        const int per = (nviews + VS - 1) / VS;
        const int b0 = min(share * per, nviews), b1 = min(b0 + per, nviews);
        v = fbct_back_pixel<Tin, T, KIND, SKIP>(g, views, 1, b0, b1, ix, iy, proj + s.sino_off);
    }
    if (VS > 1) {
        part[wv][lane] = v;
        __syncthreads();
        if (wv % VS) return;
        v = combine_shares<T, VS>(part, wv, lane);
    }
    if (!valid) return;
    const Slice2<T>& s = sl[si];
    if (ix < s.g.nx) img[s.img_off + (size_t)iy * s.g.nx + ix] = cvt_store<Tout>(v);
}

}  // namespace ctsim

// ===================================================================================
// host launchers
// ===================================================================================
namespace ctsim {

// Whether the line walk covers every tile of a geometry: the source beyond the image for
// every ray's walk, cells of at most three pixels along a line (soft edges included) and a
// tile's line within the staged pitch.  phi bounds the angle between a ray and the walk's
// major axis: the split at |X| = |Y| (SF: |X| dy = |Y| dx), the tile that straddles it and
// the pixel beside the ray.
bool fan_walk_ok(const Geom<float>& g, int kind) {
    if (!(g.dx > 0.f && g.dy > 0.f && g.du > 0.f && g.sdd > 0.f && g.sdd_du > 50.f)) return false;
    if ((double)g.nx * g.ny > 1.0e8) return false;  // image offsets in 32 bits, chunks outside it included
    const double dx = g.dx, dy = g.dy, pm = std::max(dx, dy), da = (double)g.du / g.sdd;
    const double ex = 0.5 * g.nx * dx + std::fabs(g.wx + 0.5 * (g.nx - 1)) * dx + pm;
    const double ey = 0.5 * g.ny * dy + std::fabs(g.wy + 0.5 * (g.ny - 1)) * dy + pm;
    const double R = ex + ey, sad = g.sad;
    if (!(sad > R + 4.0 * pm)) return false;
    const int cells = (g.nu + kW2 - 1) / kW2 * kW2;
    const double um = std::max(std::fabs(g.wu - 0.5), std::fabs(g.wu + cells + 0.5)) * da;
    const double gam = g.dettype == 1 ? std::atan(um) : um;
    const double slack = kW2 * da + 4.0 * pm / (sad - R);
    for (int w = 0; w < 2; ++w) {
        const double dmin = w == 0 ? dx : dy, dmaj = w == 0 ? dy : dx;
        const double phi = (kind == F2_DD ? 0.78539816339744831 : std::atan2(dmin, dmaj)) + slack;
        if (!(phi + gam < 1.4)) return false;
        if (!(sad * std::cos(phi + gam) > (w == 0 ? ey : ex) + 4.0 * pm)) return false;
        const double wpx = (sad + R) / std::cos(phi) * da / dmin, h = kind == F2_DD ? 0.0 : std::tan(phi) * dmaj / dmin;
        if (!(1.05 * wpx + h + 0.01 <= 3.0)) return false;
        if (!(kW2 * wpx + h + 8.0 + 8.0 * std::tan(phi) * dmaj / dmin <= 196.0)) return false;
    }
    return true;
}

// Whether the 2D matched backprojection leaves a pair of views at its footprints where no pixel of
// a wave lies before the detector.  The test holds the pair's loads back until both footprints are
// there, which costs up to 10% where most pixels are seen (256^2 DD from 512 bins 41 -> 43 us, 64^2
// from 64 bins 9.6 -> 10.5), so it is for images of at least 256^2 pixels whose shadow reaches three
// times as far as the detector.  Without it / with it, and the form that left each such pixel before
// its cells: 700^2 on 64 bins, 100 views, SF 153 / 76 us (84), DD 61 / 45 (61); 512^2 at 0.5 mm on
// 200 bins of 0.8 mm, 400 views, SF 314 / 256 us (308), DD 122 / 117 (169).
bool fan_back_skips(const Geom<float>& g) {
    const double hx = std::max(std::fabs((double)g.wx), std::fabs((double)g.wx + g.nx - 1)) * std::fabs((double)g.dx);
    const double hy = std::max(std::fabs((double)g.wy), std::fabs((double)g.wy + g.ny - 1)) * std::fabs((double)g.dy);
    const double det = std::max(std::fabs((double)g.wu), std::fabs((double)g.wu + g.nu - 1)) * g.sad;
    return (double)g.nx * g.ny >= 65536.0 && std::sqrt(hx * hx + hy * hy) * g.sdd_du >= 3.0 * det;
}

template <class Tin, class Tout, class T, int FOOT, int S>
static void proj2_form(unsigned blocks, hipStream_t st, const Geom<T>& g, const View<T>* views, int vstride, int nviews,
                       const void* img, void* proj, int exhaustive) {
#define CT_P2(F)                                                                                                        \
    hipLaunchKernelGGL((fbct_proj_kernel<Tin, Tout, T, FOOT, S, F>), dim3(blocks), dim3(256), 0, st, g, views, vstride, \
                       nviews, (const Tin*)img, (Tout*)proj, exhaustive)
    if constexpr (sizeof(T) == 4) {
        if (fan_walk_ok(g, FOOT)) {
            if (g.dettype == 1) CT_P2(1);
            else CT_P2(2);
            return;
        }
    }
    CT_P2(0);
#undef CT_P2
}

template <class Tin, class Tout, class T>
static hipError_t proj2(const Geom<T>& g, const View<T>* views, int vstride, int nviews, const void* img, void* proj,
                        int kind, int exhaustive, hipStream_t st) {
    const long long nut = (g.nu + kW2 - 1) / kW2;
    const long long items = (long long)nviews * nut;
    if (items == 0) return hipSuccess;
    const bool few = items < kFewItems2D;
    const unsigned blocks = few ? (unsigned)items : (unsigned)((items + 3) / 4);
#define CT_P2S(F)                                                                                             \
    do {                                                                                                      \
        if (few) proj2_form<Tin, Tout, T, F, 4>(blocks, st, g, views, vstride, nviews, img, proj, exhaustive); \
        else proj2_form<Tin, Tout, T, F, 1>(blocks, st, g, views, vstride, nviews, img, proj, exhaustive);    \
    } while (0)
    if (kind == F2_DD) CT_P2S(F2_DD);
    else CT_P2S(F2_TF);
#undef CT_P2S
    return hipGetLastError();
}

template <class Tin, class Tout, class T>
static hipError_t back2(const Geom<T>& g, const View<T>* views, int vstride, int nviews, const void* proj, void* img,
                        int kind, T scale, hipStream_t st) {
    const unsigned blocks = (unsigned)(((g.nx + kW2 - 1) / kW2) * g.ny);
    if (blocks == 0) return hipSuccess;
#define CT_B2(K, SKIP)                                                                                          \
    hipLaunchKernelGGL((fbct_back_kernel<Tin, Tout, T, K, SKIP>), dim3(blocks), dim3(256), 0, st, g, views, vstride, \
                       nviews, (const Tin*)proj, (Tout*)img, scale)
    if constexpr (sizeof(T) == 4) {
        if (kind != 2 && fan_back_skips(g)) {
            if (kind == 0) CT_B2(0, true);
            else CT_B2(1, true);
            return hipGetLastError();
        }
    }
    if (kind == 0) CT_B2(0, false);
    else if (kind == 1) CT_B2(1, false);
    else CT_B2(2, false);
#undef CT_B2
    return hipGetLastError();
}

#define CT_DISPATCH_IN(dt, MACRO)                   \
    switch (dt) {                                   \
        case DT_F32: MACRO(float);                  \
        case DT_F16: MACRO(__half);                 \
        case DT_BF16: MACRO(__hip_bfloat16);        \
        default: return hipErrorInvalidValue;       \
    }

template <>
hipError_t fbct_proj_launch<float>(const Geom<float>& g, const View<float>* views, int vstride, int nviews,
                                   const void* img, int img_dt, void* proj, int proj_dt, int kind, int exhaustive,
                                   hipStream_t st) {
#define OUT_F32(TI) return proj2<TI, float, float>(g, views, vstride, nviews, img, proj, kind, exhaustive, st)
#define OUT_F16(TI) return proj2<TI, __half, float>(g, views, vstride, nviews, img, proj, kind, exhaustive, st)
#define OUT_BF16(TI) return proj2<TI, __hip_bfloat16, float>(g, views, vstride, nviews, img, proj, kind, exhaustive, st)
    switch (proj_dt) {
        case DT_F32: CT_DISPATCH_IN(img_dt, OUT_F32);
        case DT_F16: CT_DISPATCH_IN(img_dt, OUT_F16);
        case DT_BF16: CT_DISPATCH_IN(img_dt, OUT_BF16);
        default: return hipErrorInvalidValue;
    }
#undef OUT_F32
#undef OUT_F16
#undef OUT_BF16
}

template <>
hipError_t fbct_proj_launch<double>(const Geom<double>& g, const View<double>* views, int vstride, int nviews,
                                    const void* img, int img_dt, void* proj, int proj_dt, int kind, int exhaustive,
                                    hipStream_t st) {
    if (img_dt != DT_F64 || proj_dt != DT_F64) return hipErrorInvalidValue;
    return proj2<double, double, double>(g, views, vstride, nviews, img, proj, kind, exhaustive, st);
}

template <>
hipError_t fbct_back_launch<float>(const Geom<float>& g, const View<float>* views, int vstride, int nviews,
                                   const void* proj, int proj_dt, void* img, int img_dt, int kind, float scale,
                                   hipStream_t st) {
    if (img_dt != DT_F32) return hipErrorInvalidValue;
#define B2(TI) return back2<TI, float, float>(g, views, vstride, nviews, proj, img, kind, scale, st)
    CT_DISPATCH_IN(proj_dt, B2);
#undef B2
}

template <>
hipError_t fbct_back_launch<double>(const Geom<double>& g, const View<double>* views, int vstride, int nviews,
                                    const void* proj, int proj_dt, void* img, int img_dt, int kind, double scale,
                                    hipStream_t st) {
    if (img_dt != DT_F64 || proj_dt != DT_F64) return hipErrorInvalidValue;
    return back2<double, double, double>(g, views, vstride, nviews, proj, img, kind, scale, st);
}

size_t slice2_size(bool dbl) { return dbl ? sizeof(Slice2<double>) : sizeof(Slice2<float>); }

template <class Tin, class Tout, class T, int FOOT, int S>
static void proj2b_s(const void* sl, int nslices, int nitems, const void* img, void* proj, int form, hipStream_t st) {
    const unsigned blocks = (unsigned)(((long long)nitems * S + 3) / 4);
#define CT_P2B(F)                                                                                        \
    hipLaunchKernelGGL((fbct_proj_batch_kernel<Tin, Tout, T, FOOT, S, F>), dim3(blocks), dim3(256), 0, st, \
                       (const Slice2<T>*)sl, nslices, nitems, (const Tin*)img, (Tout*)proj)
    if constexpr (sizeof(T) == 4) {
        if (form == 1) { CT_P2B(1); return; }
        if (form == 2) { CT_P2B(2); return; }
    }
    CT_P2B(0);
#undef CT_P2B
}

template <class Tin, class Tout, class T>
static hipError_t proj2b(const void* sl, int nslices, int nitems, const void* img, void* proj, int kind, int split,
                         int form, hipStream_t st) {
    if (nitems == 0) return hipSuccess;
    if (split != 1 && split != 2 && split != 4) return hipErrorInvalidValue;
#define CT_P2B(F, S) proj2b_s<Tin, Tout, T, F, S>(sl, nslices, nitems, img, proj, form, st)
    if (kind == F2_DD) {
        if (split == 1) CT_P2B(F2_DD, 1); else if (split == 2) CT_P2B(F2_DD, 2); else CT_P2B(F2_DD, 4);
    } else {
        if (split == 1) CT_P2B(F2_TF, 1); else if (split == 2) CT_P2B(F2_TF, 2); else CT_P2B(F2_TF, 4);
    }
#undef CT_P2B
    return hipGetLastError();
}

template <class Tin, class Tout, class T, int KIND, int VS>
static void back2b_s(const void* sl, int nslices, int nitems, const void* proj, void* img, int skip, hipStream_t st) {
    const unsigned blocks = (unsigned)(((long long)nitems * VS + 3) / 4);
#define CT_B2B(SKIP)                                                                                            \
    hipLaunchKernelGGL((fbct_back_batch_kernel<Tin, Tout, T, KIND, VS, SKIP>), dim3(blocks), dim3(256), 0, st, \
                       (const Slice2<T>*)sl, nslices, nitems, (const Tin*)proj, (Tout*)img)
    if constexpr (sizeof(T) == 4 && KIND != 2)
        if (skip) { CT_B2B(true); return; }
    CT_B2B(false);
#undef CT_B2B
}

template <class Tin, class Tout, class T>
static hipError_t back2b(const void* sl, int nslices, int nitems, const void* proj, void* img, int kind, int split,
                         int skip, hipStream_t st) {
    if (nitems == 0) return hipSuccess;
    if (split != 1 && split != 2 && split != 4) return hipErrorInvalidValue;
#define CT_B2B(K)                                                                               \
    do {                                                                                        \
        if (split == 1) back2b_s<Tin, Tout, T, K, 1>(sl, nslices, nitems, proj, img, skip, st); \
        else if (split == 2) back2b_s<Tin, Tout, T, K, 2>(sl, nslices, nitems, proj, img, skip, st); \
        else back2b_s<Tin, Tout, T, K, 4>(sl, nslices, nitems, proj, img, skip, st);            \
    } while (0)
    if (kind == 0) CT_B2B(0);
    else if (kind == 1) CT_B2B(1);
    else CT_B2B(2);
#undef CT_B2B
    return hipGetLastError();
}

template <>
hipError_t fbct_proj_batch_launch<float>(const void* sl, int nslices, int nitems, const void* img, int img_dt,
                                         void* proj, int proj_dt, int kind, int split, int form, hipStream_t st) {
#define OUT_F32(TI) return proj2b<TI, float, float>(sl, nslices, nitems, img, proj, kind, split, form, st)
#define OUT_F16(TI) return proj2b<TI, __half, float>(sl, nslices, nitems, img, proj, kind, split, form, st)
#define OUT_BF16(TI) return proj2b<TI, __hip_bfloat16, float>(sl, nslices, nitems, img, proj, kind, split, form, st)
    switch (proj_dt) {
        case DT_F32: CT_DISPATCH_IN(img_dt, OUT_F32);
        case DT_F16: CT_DISPATCH_IN(img_dt, OUT_F16);
        case DT_BF16: CT_DISPATCH_IN(img_dt, OUT_BF16);
        default: return hipErrorInvalidValue;
    }
#undef OUT_F32
#undef OUT_F16
#undef OUT_BF16
}

template <>
hipError_t fbct_proj_batch_launch<double>(const void* sl, int nslices, int nitems, const void* img, int img_dt,
                                          void* proj, int proj_dt, int kind, int split, int form, hipStream_t st) {
    if (img_dt != DT_F64 || proj_dt != DT_F64) return hipErrorInvalidValue;
    return proj2b<double, double, double>(sl, nslices, nitems, img, proj, kind, split, form, st);
}

template <>
hipError_t fbct_back_batch_launch<float>(const void* sl, int nslices, int nitems, const void* proj, int proj_dt,
                                         void* img, int img_dt, int kind, int split, int skip, hipStream_t st) {
#define OUT_F32(TI) return back2b<TI, float, float>(sl, nslices, nitems, proj, img, kind, split, skip, st)
#define OUT_F16(TI) return back2b<TI, __half, float>(sl, nslices, nitems, proj, img, kind, split, skip, st)
    switch (img_dt) {
        case DT_F32: CT_DISPATCH_IN(proj_dt, OUT_F32);
        case DT_F16: CT_DISPATCH_IN(proj_dt, OUT_F16);
        default: return hipErrorInvalidValue;
    }
#undef OUT_F32
#undef OUT_F16
}

template <>
hipError_t fbct_back_batch_launch<double>(const void* sl, int nslices, int nitems, const void* proj, int proj_dt,
                                          void* img, int img_dt, int kind, int split, int skip, hipStream_t st) {
    if (img_dt != DT_F64 || proj_dt != DT_F64) return hipErrorInvalidValue;
    return back2b<double, double, double>(sl, nslices, nitems, proj, img, kind, split, skip, st);
}

}  // namespace ctsim
