// Two time steps of a tile held on chip.
//
// A block of 8 waves loads a region of the state once, advances it two steps in registers and LDS,
// and stores the points whose halo was complete.  A lane is a column and a thread holds P
// consecutive rows of it (velocities, strains, C-PML memory variables in registers), so a wave's row
// of 64 columns needs no other wave for its x neighbours and a thread's inner rows none for their z
// neighbours: four LDS planes, holding the velocities while stresses are formed and the stresses
// while velocities are, carry the rest.  A step consumes three rows and columns of the region on
// each side, so a region of 64 x 8 P points stores 52 x (8 P - 12): 52 x 36 for P = 6 (FP32 tiles
// away from the border) and 52 x 12 for P = 3 (twice the blocks; and the tiles at C-PML strips and
// the border, whose twelve memory variables per point stay in registers from load to store).
//
// What bounds it.  Every load of a tile is issued at the start, so a launch pays one memory latency
// where a block marching down its rows pays one per row step (about 2 us each, 4 with C-PML records):
// two steps of a 161^2 grid take 13 us instead of 119, 401^2 14 instead of 122, 701 x 523 FP64 36
// instead of 127 (two single-step launches).  Large grids are bound by instruction issue: 4001^2
// takes 274 us per launch at 52 x 36 against 298 for the marching kernel, four waves per SIMD
// (128 VGPRs, 61 KB of LDS, two blocks per CU).
//
// The arithmetic is the single-step kernel's expression by expression, so results equal it bit for
// bit; state buffers alternate as the marching two-step kernel's.
#include <cstdint>
#include <type_traits>

#include "step_common.h"

namespace poe2d {

// LDS planes: the velocities of the region while stresses are formed, the stresses while velocities
// are.
enum { PL_VX = 0, PL_VY = 1, PL_WX = 2, PL_WY = 3, PL_SXX = 0, PL_SYY = 1, PL_SXY = 2, PL_P = 3, NPLANES = 4 };

constexpr int kTileThreads = 512, kTileWaves = kTileThreads / 64;
constexpr int kTilePad = 4;  // plane entries before and after the region, read by the outer lanes only

// One region: 64 columns (one per lane) x kTileWaves * P rows (P consecutive rows per thread, in
// registers).  nst steps from step n.
template <class T, int P, bool AVG, bool PAL, bool EDGE>
__device__ __forceinline__ void tile_region(const StepArgs<T> &A, const TileItem it, const long long n, const int nst,
                                            T *const pl, const int plane, const Vec4<T> *lpal)
{
    constexpr uint32_t VB = sizeof(Vec4<T>);
    constexpr int RH = kTileWaves * P;
    typedef __attribute__((address_space(1))) nvec4<T> GN;
    typedef __attribute__((address_space(1))) T GT;
    typedef __attribute__((address_space(1))) const T GCT;
    typedef __attribute__((address_space(4))) const T KT;
    const int lane = threadIdx.x & 63;
    const int r0 = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) * P;  // first region row of this wave
    const int nx = A.nx, nz = A.nz, pitch = A.pitch;
    const int c = it.x0 - kTileHalo + lane;
    const int z0 = it.z0 - kTileHalo + r0;  // grid row of this thread's row 0
    const int in = (int)((((n - A.pair0) >> 1) + A.pcur) & 1);
    const T rdx = A.rdx, rdz = A.rdz, dt = A.dt;

    gchar *const gb = (gchar *)A.grp;
    const long long gsb = A.group_stride * (long long)VB;
    const int cc = min(max(c, -kPadCols), nx + 1);
    const uint32_t rowb = (uint32_t)pitch * VB;
    const int last_row = nz + kPadRows;
    auto prow = [&](int z) -> uint32_t { return (uint32_t)(min(z, last_row) + kPadRows); };
    auto off = [&](int z) -> uint32_t { return (uint32_t)(cc + kPadCols) * VB + prow(z) * rowb; };
    auto ld = [&](const gchar *g, int z) -> Vec4<T> {
        const nvec4<T> v = *(const GN *)(g + off(z));
        return Vec4<T>{v.x, v.y, v.z, v.w};
    };
    const gchar *const Vo = gb + group_v(in) * gsb;
    const gchar *const So = gb + group_s(in) * gsb;
    Vec4<T> V[P], S[P];
#pragma unroll
    for (int i = 0; i < P; ++i) V[i] = ld(Vo, z0 + i);
#pragma unroll
    for (int i = 0; i < P; ++i) S[i] = ld(So, z0 + i);

    // material: palette entries of rows 0 .. P, or the coefficient groups (read where used)
    int id[P + 1];
    const gchar *const MSg = (const gchar *)A.mat + G_MS * gsb;
    const gchar *const MVg = (const gchar *)A.mat + G_MV * gsb;
    if constexpr (PAL) {
        gcuchar *const mid = (gcuchar *)A.mid;
#pragma unroll
        for (int i = 0; i <= P; ++i) id[i] = mid[(uint32_t)(cc + kPadCols) + prow(z0 + i) * (uint32_t)pitch];
    }

    // C-PML: memory variables of this thread's points and the profiles of its column and rows
    const bool inx = c >= 0 && c <= nx;
    const int sx = (EDGE && inx) ? ((gcint *)A.xmap)[c] : -1;
    T qx[EDGE ? P : 1][NPSI_X], qz[EDGE ? P : 1][NPSI_Z];
    T ax = 0, bx = 1, rkx = 1, axh = 0, bxh = 1, rkxh = 1;
    GT *const psi = (GT *)A.psi;
    auto px = [&](int b, int z) -> GT * { return psi + ((long long)b * A.pxn + (long long)z * A.wxs + sx) * NPSI_X; };
    auto pz = [&](int b, int s) -> GT * {
        return psi + 2LL * NPSI_X * A.pxn + ((long long)b * A.pzn + (long long)s * pitch + c) * NPSI_Z;
    };
    if constexpr (EDGE) {
        const GCT *const tab = (const GCT *)A.tab;
        if (sx >= 0) {
            ax = tab[TB_AX * A.tn + c], bx = tab[TB_BX * A.tn + c], rkx = tab[TB_RKX * A.tn + c];
            axh = tab[TB_AXH * A.tn + c], bxh = tab[TB_BXH * A.tn + c], rkxh = tab[TB_RKXH * A.tn + c];
        }
        typedef T pair __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(1))) const pair GP;
#pragma unroll
        for (int i = 0; i < P; ++i) {
#pragma unroll
            for (int q = 0; q < NPSI_X; ++q) qx[i][q] = qz[i][q] = T(0);
            const int z = z0 + i;
            if (sx >= 0 && z >= 0 && z <= nz) {
                const GP *const r = (const GP *)px(in, z);
#pragma unroll
                for (int q = 0; q < NPSI_X / 2; ++q) {
                    const pair v = r[q];
                    qx[i][2 * q] = v.x, qx[i][2 * q + 1] = v.y;
                }
            }
            const int s = zstrip(A, z);
            if (s >= 0 && inx) {
                const GP *const r = (const GP *)pz(in, s);
#pragma unroll
                for (int q = 0; q < NPSI_Z / 2; ++q) {
                    const pair v = r[q];
                    qz[i][2 * q] = v.x, qz[i][2 * q + 1] = v.y;
                }
            }
        }
    }
    const KT *const ktab = (const KT *)A.tab;

    const bool xr1 = !EDGE || (c >= 1 && c < nx);      // stress1
    const bool xr2 = !EDGE || (c >= 2 && c < nx);      // stress2
    const bool xr3 = !EDGE || (c >= 1 && c < nx - 1);  // stress3
    const bool xr4 = !EDGE || (c >= 2 && c < nx);      // vx
    const bool xr5 = !EDGE || (c >= 1 && c < nx - 1);  // vz
    const bool src_p = A.src_kind == POE2D_SRC_PRESSURE_DGAUSS && c == A.src_x;
    const bool src_f = A.src_kind == POE2D_SRC_FORCE_Y_RICKER && c == A.src_x;

    T *const own = pl + kTilePad + r0 * 64 + lane;  // this thread's row 0 of plane 0
    // row i (which may be another wave's) of plane k; rows off the region read its nearest row,
    // into values no stored point depends on
    auto at = [&](int k, int i) -> T { return own[k * plane + (min(max(r0 + i, 0), RH - 1) - r0) * 64]; };
    typedef int nint4 __attribute__((ext_vector_type(4)));
    const __attribute__((address_space(1))) nint4 *const rec = (const __attribute__((address_space(1))) nint4 *)A.rec_points;

#pragma unroll
    for (int i = 0; i < P; ++i) {
        own[PL_VX * plane + i * 64] = V[i].x;
        own[PL_VY * plane + i * 64] = V[i].y;
        own[PL_WX * plane + i * 64] = V[i].z;
        own[PL_WY * plane + i * 64] = V[i].w;
    }
    __syncthreads();

    for (int k = 0; k < nst; ++k) {
        const int nk = (int)n + k;
        T srcv = T(0);
        {
            const long long q = nk - A.src_n0;
            if (A.src_series && q >= 0 && q < A.src_len) srcv = ((const KT *)A.src_series)[q];
        }
        const bool rec_on = it.rec_hi > it.rec_lo && nk % A.rec_dec == 0 && nk / A.rec_dec < A.rec_nsamp;
        GT *const trace = (GT *)A.traces + (rec_on ? (long long)(nk / A.rec_dec) * A.rec_ncomp * A.rec_n : 0);
        auto entry = [&](const nint4 e) -> int { return kTilePad + (e.y - it.z0 + kTileHalo) * 64 + e.x - it.x0 + kTileHalo; };
        if (rec_on)
            for (int e = it.rec_lo + (int)threadIdx.x; e < it.rec_hi; e += kTileThreads) {
                const nint4 en = rec[e];
                int q = 0;
                if (A.rec_mask & POE2D_VX) trace[(long long)(q++) * A.rec_n + en.z] = pl[PL_VX * plane + entry(en)];
                if (A.rec_mask & POE2D_VY) trace[(long long)q * A.rec_n + en.z] = pl[PL_VY * plane + entry(en)];
            }

        // ---- stresses
        T sxx[P], syy[P], p[P];
        {
            T vy[P + 3], wy[P + 3], vx[P + 3];  // rows -2 .. P (vy, wy), -1 .. P + 1 (vx)
            vy[0] = at(PL_VY, -2), vy[1] = at(PL_VY, -1), vy[P + 2] = at(PL_VY, P);
            wy[0] = at(PL_WY, -2), wy[1] = at(PL_WY, -1), wy[P + 2] = at(PL_WY, P);
            vx[0] = at(PL_VX, -1), vx[P + 1] = at(PL_VX, P), vx[P + 2] = at(PL_VX, P + 1);
#pragma unroll
            for (int i = 0; i < P; ++i) vy[i + 2] = V[i].y, wy[i + 2] = V[i].w, vx[i + 1] = V[i].x;
#pragma unroll
            for (int i = 0; i < P; ++i) {
                sxx[i] = syy[i] = p[i] = T(0);
                const int z = z0 + i;
                if (r0 + i < 3 * k + 1 || r0 + i > RH - 2 - 3 * k) continue;
                const T *const x0 = own + PL_VX * plane + i * 64, *const x1 = own + PL_WX * plane + i * 64;
                const T *const x2 = own + PL_VY * plane + i * 64;
                const int szs = EDGE ? zstrip(A, z) : -1;
                const bool u1 = xr1 && (!EDGE || (z >= 2 && z < nz - 1)), u2 = xr2 && (!EDGE || (z >= 1 && z < nz - 1));
                Vec4<T> ms;
                T mu_nxt;
                if constexpr (PAL) {
                    ms = lpal[PAL_MS * kMaxPalette + id[i]];
                    mu_nxt = lpal[PAL_MS * kMaxPalette + id[i + 1]].w;
                } else {
                    ms = ld(MSg, z);
                    mu_nxt = ld(MSg, z + 1).w;
                }
                T az = 0, bz = 1, rkz = 1, azh = 0, bzh = 1;
                if (szs >= 0) {
                    az = ktab[TB_AZ * A.tn + z], bz = ktab[TB_BZ * A.tn + z], rkz = ktab[TB_RKZ * A.tn + z];
                    azh = ktab[TB_AZH * A.tn + z], bzh = ktab[TB_BZH * A.tn + z];
                }
                if (u1) {
                    T dvx = d4(x0[1], vx[i + 1], x0[2], x0[-1], rdx);
                    T dwx = d4(x1[1], V[i].z, x1[2], x1[-1], rdx);
                    T dvz = d4(vy[i + 2], vy[i + 1], vy[i + 3], vy[i], rdz);
                    T dwz = d4(wy[i + 2], wy[i + 1], wy[i + 3], wy[i], rdz);
                    if constexpr (EDGE) {
                        if (sx >= 0) {
                            dvx = cpml_held(dvx, qx[i][PX_DVX], axh, bxh, rkxh);
                            dwx = cpml_held(dwx, qx[i][PX_DWX], axh, bxh, rkxh);
                        }
                        if (szs >= 0) {
                            dvz = cpml_held(dvz, qz[i][PZ_DVZ], az, bz, rkz);
                            dwz = cpml_held(dwz, qz[i][PZ_DWZ], az, bz, rkz);
                        }
                    }
                    S[i].x = S[i].x + dt * dvx;
                    S[i].y = S[i].y + dt * dvz;
                    S[i].z = (S[i].z - dwx * dt) - dwz * dt;
                    p[i] = pore_pressure(S[i].x, S[i].y, S[i].z, ms.x, ms.y);
                    if (src_p && z == A.src_z) p[i] += srcv;
                    if (xr3) {
                        const T lc = ms.z, al = ms.x;
                        const T l2m = lc + T(2) * ms.w;
                        sxx[i] = l2m * S[i].x + lc * S[i].y - al * p[i];
                        syy[i] = lc * S[i].x + l2m * S[i].y - al * p[i];
                    }
                }
                if (u2) {
                    T ddx = d4(V[i].y, x2[-1], x2[1], x2[-2], rdx);
                    T ddz = d4(vx[i + 2], vx[i + 1], vx[i + 3], vx[i], rdz);
                    if constexpr (EDGE) {
                        if (sx >= 0) ddx = cpml_held(ddx, qx[i][PX_DVY], ax, bx, rkx);
                        // half-grid memory coefficients, full-grid K_z divisor (reference :224-226)
                        if (szs >= 0) ddz = cpml_held(ddz, qz[i][PZ_DVX], azh, bzh, rkz);
                    }
                    const T mu_xy = AVG ? harmonic_mu(ms.w, mu_nxt) : mu_nxt;
                    S[i].w = S[i].w + mu_xy * (ddx + ddz) * dt;
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < P; ++i) {
            own[PL_SXX * plane + i * 64] = sxx[i];
            own[PL_SYY * plane + i * 64] = syy[i];
            own[PL_SXY * plane + i * 64] = S[i].w;
            own[PL_P * plane + i * 64] = p[i];
        }
        __syncthreads();
        if (rec_on && (A.rec_mask & POE2D_P))
            for (int e = it.rec_lo + (int)threadIdx.x; e < it.rec_hi; e += kTileThreads) {
                const nint4 en = rec[e];
                trace[(long long)(A.rec_ncomp - 1) * A.rec_n + en.z] = pl[PL_P * plane + entry(en)];
            }

        // ---- velocities
        {
            T sy[P + 3], pp[P + 3], sh[P + 3];  // rows -1 .. P + 1 (syy, p), -2 .. P (sxy)
            sy[0] = at(PL_SYY, -1), sy[P + 1] = at(PL_SYY, P), sy[P + 2] = at(PL_SYY, P + 1);
            pp[0] = at(PL_P, -1), pp[P + 1] = at(PL_P, P), pp[P + 2] = at(PL_P, P + 1);
            sh[0] = at(PL_SXY, -2), sh[1] = at(PL_SXY, -1), sh[P + 2] = at(PL_SXY, P);
#pragma unroll
            for (int i = 0; i < P; ++i) sy[i + 1] = syy[i], pp[i + 1] = p[i], sh[i + 2] = S[i].w;
#pragma unroll
            for (int i = 0; i < P; ++i) {
                const int z = z0 + i;
                if (r0 + i < 3 * k + 3 || r0 + i > RH - 4 - 3 * k) continue;
                const T *const x0 = own + PL_SXX * plane + i * 64, *const x1 = own + PL_P * plane + i * 64;
                const T *const x2 = own + PL_SXY * plane + i * 64;
                const int szj = EDGE ? zstrip(A, z) : -1;
                const bool u4 = xr4 && (!EDGE || (z >= 2 && z < nz)), u5 = xr5 && (!EDGE || (z >= 1 && z < nz - 1));
                Vec4<T> mv, mv1, cn, cn1;
                if constexpr (PAL) {
                    mv = lpal[PAL_MV * kMaxPalette + id[i]];
                    mv1 = lpal[PAL_MV * kMaxPalette + id[i + 1]];
                    if constexpr (sizeof(T) == 4) {
                        cn = lpal[PAL_CN * kMaxPalette + id[i]];
                        cn1 = lpal[PAL_CN * kMaxPalette + id[i + 1]];
                    }
                } else {
                    mv = ld(MVg, z);
                    mv1 = ld(MVg, z + 1);
                }
                T az = 0, bz = 1, rkz = 1, azh = 0, bzh = 1, rkzh = 1;
                if (szj >= 0) {
                    az = ktab[TB_AZ * A.tn + z], bz = ktab[TB_BZ * A.tn + z], rkz = ktab[TB_RKZ * A.tn + z];
                    azh = ktab[TB_AZH * A.tn + z], bzh = ktab[TB_BZH * A.tn + z], rkzh = ktab[TB_RKZH * A.tn + z];
                }
                if (u4) {
                    T e1 = d4(sxx[i], x0[-1], x0[1], x0[-2], rdx);
                    T e2 = d4(p[i], x1[-1], x1[1], x1[-2], rdx);
                    T e3 = d4(sh[i + 2], sh[i + 1], sh[i + 3], sh[i], rdz);
                    if constexpr (EDGE) {
                        if (sx >= 0) {
                            e1 = cpml_held(e1, qx[i][PX_DSXX], ax, bx, rkx);
                            e2 = cpml_held(e2, qx[i][PX_DPX], ax, bx, rkx);
                        }
                        if (szj >= 0) e3 = cpml_held(e3, qz[i][PZ_DSXY], az, bz, rkz);
                    }
                    if constexpr (PAL && sizeof(T) == 4)
                        biot_velocity_cn(V[i].x, V[i].z, e1 + e3, e2, mv.x, mv.y, mv.z, cn);
                    else
                        biot_velocity(V[i].x, V[i].z, e1 + e3, e2, mv.x, mv.y, mv.z, mv.w, A.inv_dt);
                }
                if (u5) {
                    T e1 = d4(x2[1], S[i].w, x2[2], x2[-1], rdx);
                    T e2 = d4(sy[i + 2], sy[i + 1], sy[i + 3], sy[i], rdz);
                    T e3 = d4(pp[i + 2], pp[i + 1], pp[i + 3], pp[i], rdz);
                    if constexpr (EDGE) {
                        if (sx >= 0) e1 = cpml_held(e1, qx[i][PX_DSXY], axh, bxh, rkxh);
                        if (szj >= 0) {
                            e2 = cpml_held(e2, qz[i][PZ_DSYY], azh, bzh, rkzh);
                            e3 = cpml_held(e3, qz[i][PZ_DPZ], azh, bzh, rkzh);
                        }
                    }
                    T div = e1 + e2;
                    if (src_f && z == A.src_z) div += srcv;
                    if constexpr (AVG) {
                        const Vec4<T> mvy = mean_rows(mv, mv1);
                        biot_velocity(V[i].y, V[i].w, div, e3, mvy.x, mvy.y, mvy.z, mvy.w, A.inv_dt);
                    } else if constexpr (PAL && sizeof(T) == 4) {
                        biot_velocity_cn(V[i].y, V[i].w, div, e3, mv1.x, mv1.y, mv1.z, cn1);
                    } else {
                        biot_velocity(V[i].y, V[i].w, div, e3, mv1.x, mv1.y, mv1.z, mv1.w, A.inv_dt);
                    }
                }
            }
        }
        if (k + 1 < nst) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < P; ++i) {
                own[PL_VX * plane + i * 64] = V[i].x;
                own[PL_VY * plane + i * 64] = V[i].y;
                own[PL_WX * plane + i * 64] = V[i].z;
                own[PL_WY * plane + i * 64] = V[i].w;
            }
            __syncthreads();
        }
    }

    // ---- the owned points
    if (lane < kTileHalo || lane >= 64 - kTileHalo || c > nx) return;
    gchar *const Vn = gb + group_v(in ^ 1) * gsb;
    gchar *const Sn = gb + group_s(in ^ 1) * gsb;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int z = z0 + i;
        if (r0 + i < kTileHalo || z >= it.z1) continue;
        *(GN *)(Vn + off(z)) = nvec4<T>{V[i].x, V[i].y, V[i].z, V[i].w};
        *(GN *)(Sn + off(z)) = nvec4<T>{S[i].x, S[i].y, S[i].z, S[i].w};
        if constexpr (EDGE) {
            typedef T pair __attribute__((ext_vector_type(2)));
            typedef __attribute__((address_space(1))) pair GP;
            if (sx >= 0) {
                GP *const r = (GP *)px(in ^ 1, z);
#pragma unroll
                for (int q = 0; q < NPSI_X / 2; ++q) r[q] = pair{qx[i][2 * q], qx[i][2 * q + 1]};
            }
            const int s = zstrip(A, z);
            if (s >= 0) {
                GP *const r = (GP *)pz(in ^ 1, s);
#pragma unroll
                for (int q = 0; q < NPSI_Z / 2; ++q) r[q] = pair{qz[i][2 * q], qz[i][2 * q + 1]};
            }
        }
    }
}

template <class T, bool AVG, bool PAL>
__global__ void __launch_bounds__(kTileThreads, sizeof(T) == 4 ? 4 : 2)
    tile_steps(const StepArgs<T> *__restrict__ models, const TileItem *__restrict__ work, int nwork, int per_xcd,
               const long long *__restrict__ base, int k, int nst)
{
    constexpr int PMAX = sizeof(T) == 4 ? 6 : 3;
    constexpr int plane = kTileWaves * PMAX * 64 + 2 * kTilePad;
    __shared__ T pl[NPLANES * plane];
    __shared__ Vec4<T> lpal[PAL ? PAL_SECTIONS * kMaxPalette : 1];
    const int wi = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (wi >= nwork) return;
    const TileItem it = work[wi];
    if (it.model < 0) return;
    const StepArgs<T> A = models[it.model];
    const long long n = *(const kcll *)base + k;
    if constexpr (PAL) {
        typedef __attribute__((address_space(1))) nvec4<T> GN;
        const GN *const pal = (const GN *)A.pal;
        constexpr int sections = sizeof(T) == 4 ? PAL_SECTIONS : 2;
        for (int i = threadIdx.x; i < sections * A.npal; i += kTileThreads) {
            const int s = i / A.npal, e = s * kMaxPalette + i % A.npal;
            const nvec4<T> v = pal[e];
            lpal[e] = Vec4<T>{v.x, v.y, v.z, v.w};
        }
    }
    if (it.kind == TILE_EDGE) tile_region<T, 3, AVG, PAL, true>(A, it, n, nst, pl, plane, lpal);
    else if (it.kind == TILE_SHORT) tile_region<T, 3, AVG, PAL, false>(A, it, n, nst, pl, plane, lpal);
    else if constexpr (sizeof(T) == 4) tile_region<T, 6, AVG, PAL, false>(A, it, n, nst, pl, plane, lpal);
}

template <class T>
hipError_t launch_tiles(const StepArgs<T> *models, const TileItem *work, int nwork, int per_xcd, bool palette, bool avg,
                        const long long *base, int k, int nst, hipStream_t stream)
{
    if (nwork < 1 || per_xcd < 1 || 8LL * per_xcd < nwork || nst < 1 || nst > 2) return hipErrorInvalidValue;
    const dim3 grid(8 * per_xcd);
    if (palette) {
        if (avg) tile_steps<T, true, true><<<grid, kTileThreads, 0, stream>>>(models, work, nwork, per_xcd, base, k, nst);
        else tile_steps<T, false, true><<<grid, kTileThreads, 0, stream>>>(models, work, nwork, per_xcd, base, k, nst);
    } else {
        if (avg) tile_steps<T, true, false><<<grid, kTileThreads, 0, stream>>>(models, work, nwork, per_xcd, base, k, nst);
        else tile_steps<T, false, false><<<grid, kTileThreads, 0, stream>>>(models, work, nwork, per_xcd, base, k, nst);
    }
    return hipGetLastError();
}

template hipError_t launch_tiles<float>(const StepArgs<float> *, const TileItem *, int, int, bool, bool, const long long *, int,
                                        int, hipStream_t);
template hipError_t launch_tiles<double>(const StepArgs<double> *, const TileItem *, int, int, bool, bool, const long long *,
                                         int, int, hipStream_t);

}  // namespace poe2d
