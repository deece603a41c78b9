// Two or three time steps of a tile held on chip.
//
// A block of 8 waves loads a region of the state once, advances it two or three steps, and stores the points
// whose halo was complete.  A lane is a column and a thread holds P consecutive rows of it
// (velocities, strains, C-PML memory variables in registers), so x neighbours are the neighbouring
// lanes' registers (wave shifts, folded into the differences where the instruction allows) and z
// neighbours the thread's own; only the two or three rows at a wave's ends go through LDS, its
// velocities before the stresses and its stresses before the velocities, one barrier each.  A step
// consumes three rows and columns of the region on each side, so a region of 64 x 8 P points stores
// 52 x (8 P - 12) of two steps: 52 x 36 for P = 6 (FP32 tiles away from the border), 52 x 20 for P = 4
// (tiles at the C-PML strips or the border of one axis, whose six memory variables per point stay in
// registers from load to store) and 52 x 12 for P = 3 (corners, with twelve; or twice the blocks).  Lower
// tiles load and compute only the rows they need.
//
// What bounds it.  Every load of a tile is issued at the start, so a launch pays one memory latency
// where a block marching down its rows pays one per row step (about 2 us each, 4 with C-PML records):
// two steps of a 161^2 grid take 11 us instead of 119, 401^2 12 instead of 122, 701 x 523 FP64 28
// instead of 127 (two single-step launches).  Large grids are bound by HBM: 4001^2 takes 231 us per
// launch against 298 for the marching kernel, 1.14 GB (1.06 compulsory) at 4.95 TB/s (128 VGPRs, four
// waves per SIMD, two blocks per CU).  Mid-sized ones by their edges' wider halo: with P = 3 and both
// axes' code along every edge, 401^2 took 6.1 us a step instead of 5.0 (three steps per launch), 801^2
// 12.0 instead of 8.8, 1201^2 16.7 instead of 15.1, 64 models of 401^2 127 instead of 103.
//
// The arithmetic is the single-step kernel's expression by expression, so results equal it bit for
// bit; state buffers alternate as the marching two-step kernel's.
#include <cstdint>
#include <type_traits>

#include "step_common.h"

namespace poe2d {

constexpr int kTileThreads = 512, kTileWaves = kTileThreads / 64;

// Rows a wave publishes to its neighbours, before the stresses (its velocities) and before the
// velocities (its stresses): of each field the rows a z difference of the wave below or above reads.
enum { BV_VY_L2, BV_VY_L1, BV_VY_F1, BV_WY_L2, BV_WY_L1, BV_WY_F1, BV_VX_L1, BV_VX_F1, BV_VX_F2, NBOUNDARY };
enum { BS_SXY_L2, BS_SXY_L1, BS_SXY_F1, BS_SYY_L1, BS_SYY_F1, BS_SYY_F2, BS_P_L1, BS_P_F1, BS_P_F2 };

constexpr int NXTAB = TB_RKXH - TB_AX + 1;  // C-PML profiles of a column

// The value of the lane one column to the right (zero past the last lane) / to the left.
__device__ __forceinline__ int dpp_right(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x130, 0xf, 0xf, true); }
__device__ __forceinline__ int dpp_left(int x) { return __builtin_amdgcn_update_dpp(0, x, 0x138, 0xf, 0xf, true); }
__device__ __forceinline__ float right(float x) { return __builtin_bit_cast(float, dpp_right(__builtin_bit_cast(int, x))); }
__device__ __forceinline__ float left(float x) { return __builtin_bit_cast(float, dpp_left(__builtin_bit_cast(int, x))); }
__device__ __forceinline__ double right(double x)
{
    const int2 v = __builtin_bit_cast(int2, x);
    return __builtin_bit_cast(double, int2{dpp_right(v.x), dpp_right(v.y)});
}
__device__ __forceinline__ double left(double x)
{
    const int2 v = __builtin_bit_cast(int2, x);
    return __builtin_bit_cast(double, int2{dpp_left(v.x), dpp_left(v.y)});
}
// Staggered x difference between a column and the one to its right / left.
template <class T>
__device__ __forceinline__ T ddx_fwd(T f, T rh)
{
    const T f1 = right(f);
    return d4(f1, f, right(f1), left(f), rh);
}
template <class T>
__device__ __forceinline__ T ddx_bwd(T f, T rh)
{
    const T f0 = left(f);
    return d4(f, f0, right(f), left(f0), rh);
}

// One region: 64 columns (one per lane) x kTileWaves * P rows (P consecutive rows per thread, in
// registers).  nst steps from step n.  EDGE: the region reaches x strips or the outer columns (EDGE_X),
// z strips or the outer rows (EDGE_Z).
enum { EDGE_X = 1, EDGE_Z = 2 };
template <class T, int P, bool AVG, bool PAL, int EDGE, bool ROOM>
__device__ __forceinline__ void tile_region(const __attribute__((address_space(4))) StepArgs<T> &A, const TileItem it, const long long n, const int in, const int halo, const int nst, const bool stream,
                                            T (*const bv)[kTileWaves][64], T (*const bs)[kTileWaves][64],
                                            T (*const xtab)[64], const Vec4<T> *lpal)
{
    constexpr uint32_t VB = sizeof(Vec4<T>);
    constexpr bool EX = EDGE & EDGE_X, EZ = EDGE & EDGE_Z;
    const int rows = min(it.z1 - it.z0 + 2 * halo, kTileWaves * P);  // the region's rows (the last waves' may be past it)
    typedef __attribute__((address_space(1))) nvec4<T> GN;
    typedef __attribute__((address_space(1))) T GT;
    typedef __attribute__((address_space(1))) const T GCT;
    typedef __attribute__((address_space(4))) const T KT;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wb = max(w - 1, 0), wa = min(w + 1, kTileWaves - 1);  // (the region's outer waves read values nothing stored depends on)
    const int r0 = w * P;  // first region row of this wave
    const int nx = A.nx, nz = A.nz, pitch = A.pitch;
    const int c = it.x0 - halo + lane;
    const int z0 = it.z0 - halo + r0;  // grid row of this thread's row 0
    const T rdx = A.rdx, rdz = A.rdz, dt = A.dt;
    const int ztop = A.ztop, zbot = A.zbot;
    auto strip = [&](int z) -> int { return z < 0 ? -1 : z < ztop ? z : z < zbot ? -1 : z <= nz ? ztop + (z - zbot) : -1; };

    gchar *const gb = (gchar *)A.grp;
    const long long gsb = A.group_stride * (long long)VB;
    const int cc = min(max(c, -kPadCols), nx + 1);
    const uint32_t rowb = (uint32_t)pitch * VB;
    const int last_row = min(nz + kPadRows, it.z0 - halo + rows - 1);
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
    constexpr bool PACK = EDGE;  // entries of four rows in one register
    int id[PACK ? P / 4 + 1 : P + 1];
    auto entry = [&](int i) -> int {
        if constexpr (PACK) return (id[i / 4] >> (8 * (i % 4))) & 255;
        else return id[i];
    };
    const gchar *const MSg = (const gchar *)A.mat + G_MS * gsb;
    const gchar *const MVg = (const gchar *)A.mat + G_MV * gsb;
    if constexpr (PAL) {
        gcuchar *const mid = (gcuchar *)A.mid;
        if constexpr (PACK)
            for (int &q : id) q = 0;
#pragma unroll
        for (int i = 0; i <= P; ++i) {
            const int e = mid[(uint32_t)(cc + kPadCols) + prow(z0 + i) * (uint32_t)pitch];
            if constexpr (PACK) id[i / 4] |= e << (8 * (i % 4));
            else id[i] = e;
        }
    }

    // C-PML: memory variables of this thread's points and the profiles of its column and rows
    // (a column's profiles in registers; in LDS, a few per cent slower on launches of one tile per CU,
    // where FP32 blocks share a CU: there they would spill)
    constexpr bool XLDS = EX && sizeof(T) == 4 && !ROOM;
    const bool inx = c >= 0 && c <= nx;
    const int sx = (EX && inx) ? ((gcint *)A.xmap)[c] : -1;
    T qx[EX ? P : 1][NPSI_X], qz[EZ ? P : 1][NPSI_Z];
    GT *const psi = (GT *)A.psi;
    auto px = [&](int b, int z) -> GT * { return psi + ((long long)b * A.pxn + (long long)z * A.wxs + sx) * NPSI_X; };
    auto pz = [&](int b, int s) -> GT * {
        return psi + 2LL * NPSI_X * A.pxn + ((long long)b * A.pzn + (long long)s * pitch + c) * NPSI_Z;
    };
    if constexpr (EDGE) {
        if (XLDS && w < NXTAB && inx) xtab[w][lane] = ((const GCT *)A.tab)[(TB_AX + w) * A.tn + c];
        typedef T pair __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(1))) const pair GP;
#pragma unroll
        for (int i = 0; i < P; ++i) {
#pragma unroll
            for (int q = 0; q < NPSI_X; ++q) {
                if constexpr (EX) qx[i][q] = T(0);
                if constexpr (EZ) qz[i][q] = T(0);
            }
            const int z = z0 + i;
            if constexpr (EX)
                if (sx >= 0 && z >= 0 && z <= min(nz, last_row)) {
                    const GP *const r = (const GP *)px(in, z);
#pragma unroll
                    for (int q = 0; q < NPSI_X / 2; ++q) {
                        const pair v = r[q];
                        qx[i][2 * q] = v.x, qx[i][2 * q + 1] = v.y;
                    }
                }
            if constexpr (EZ) {
                const int s = strip(z);
                if (s >= 0 && inx && z <= last_row) {
                    const GP *const r = (const GP *)pz(in, s);
#pragma unroll
                    for (int q = 0; q < NPSI_Z / 2; ++q) {
                        const pair v = r[q];
                        qz[i][2 * q] = v.x, qz[i][2 * q + 1] = v.y;
                    }
                }
            }
        }
    }
    const KT *const ktab = (const KT *)A.tab;
    T xr[EX && !XLDS ? NXTAB : 1];
    if constexpr (EX && !XLDS)
#pragma unroll
        for (int k = 0; k < NXTAB; ++k) xr[k] = inx ? ((const GCT *)A.tab)[(TB_AX + k) * A.tn + c] : T(0);
    auto xt = [&](int k) -> T { return XLDS ? xtab[k - TB_AX][lane] : xr[EX && !XLDS ? k - TB_AX : 0]; };

    const bool xr1 = !EX || (c >= 1 && c < nx);      // stress1
    const bool xr2 = !EX || (c >= 2 && c < nx);      // stress2
    const bool xr3 = !EX || (c >= 1 && c < nx - 1);  // stress3
    const bool xr4 = !EX || (c >= 2 && c < nx);      // vx
    const bool xr5 = !EX || (c >= 1 && c < nx - 1);  // vz
    const bool src_p = A.src_kind == POE2D_SRC_PRESSURE_DGAUSS && c == A.src_x;
    const bool src_f = A.src_kind == POE2D_SRC_FORCE_Y_RICKER && c == A.src_x;

    typedef int nint2 __attribute__((ext_vector_type(2)));
    const __attribute__((address_space(1))) nint2 *const rec = (const __attribute__((address_space(1))) nint2 *)A.rec_entries;
    kcint *const rec_ptr = (kcint *)A.rec_tile_ptr + it.rec;

    // without a palette: coefficients of this thread's rows and the one below, from the groups, read
    // once and held for every step where the registers allow (no memory variables, FP32, no means of
    // rows), else requested a barrier ahead of each use
    constexpr bool HOLD = !PAL && sizeof(T) == 4 && (ROOM || (!EDGE && !AVG));
    Vec4<T> mg[PAL ? 1 : P + 1], mh[HOLD ? P + 1 : 1];
    auto groups = [&](const gchar *g, Vec4<T> *m) {
#pragma unroll
        for (int i = 0; i <= P; ++i) m[i] = ld(g, z0 + i);
    };
    if constexpr (HOLD) groups(MSg, mg), groups(MVg, mh);
    auto publish = [&]() {
        bv[BV_VY_L2][w][lane] = V[P - 2].y, bv[BV_VY_L1][w][lane] = V[P - 1].y, bv[BV_VY_F1][w][lane] = V[0].y;
        bv[BV_WY_L2][w][lane] = V[P - 2].w, bv[BV_WY_L1][w][lane] = V[P - 1].w, bv[BV_WY_F1][w][lane] = V[0].w;
        bv[BV_VX_L1][w][lane] = V[P - 1].x, bv[BV_VX_F1][w][lane] = V[0].x, bv[BV_VX_F2][w][lane] = V[1].x;
    };
    if constexpr (!PAL && !HOLD) groups(MSg, mg);
    publish();
    __syncthreads();

    for (int k = 0; k < nst; ++k) {
        const int nk = (int)n + k;
        T srcv = T(0);
        {
            const long long q = nk - A.src_n0;
            if (A.src_series && q >= 0 && q < A.src_len) srcv = ((const KT *)A.src_series)[q];
        }
        const bool rec_on = it.rec >= 0 && nk % A.rec_dec == 0 && nk / A.rec_dec < A.rec_nsamp;
        GT *const trace = (GT *)A.traces + (rec_on ? (long long)(nk / A.rec_dec) * A.rec_ncomp * A.rec_n : 0);
        // component q of row i's receivers, one per lane, from the lane that holds their column
        auto record = [&](int i, int q, T value) {
            if (r0 + i < halo || z0 + i >= it.z1) return;
            const int lo = rec_ptr[z0 + i - it.z0], hi = rec_ptr[z0 + i - it.z0 + 1];
            for (int e = lo; e < hi; e += 64) {
                const nint2 en = rec[min(e + lane, hi - 1)];
                const T v = __shfl(value, en.x - it.x0 + halo);
                if (e + lane < hi) trace[(long long)q * A.rec_n + en.y] = v;
            }
        };
        if (rec_on) {
            int q = 0;
            if (A.rec_mask & POE2D_VX) {
#pragma unroll
                for (int i = 0; i < P; ++i) record(i, q, V[i].x);
                ++q;
            }
            if (A.rec_mask & POE2D_VY)
#pragma unroll
                for (int i = 0; i < P; ++i) record(i, q, V[i].y);
        }

        // ---- stresses
        T sxx[P], syy[P], p[P];
        {
            T vy[P + 3], wy[P + 3], vx[P + 3];  // rows -2 .. P (vy, wy), -1 .. P + 1 (vx)
            vy[0] = bv[BV_VY_L2][wb][lane], vy[1] = bv[BV_VY_L1][wb][lane], vy[P + 2] = bv[BV_VY_F1][wa][lane];
            wy[0] = bv[BV_WY_L2][wb][lane], wy[1] = bv[BV_WY_L1][wb][lane], wy[P + 2] = bv[BV_WY_F1][wa][lane];
            vx[0] = bv[BV_VX_L1][wb][lane], vx[P + 1] = bv[BV_VX_F1][wa][lane], vx[P + 2] = bv[BV_VX_F2][wa][lane];
#pragma unroll
            for (int i = 0; i < P; ++i) vy[i + 2] = V[i].y, wy[i + 2] = V[i].w, vx[i + 1] = V[i].x;
#pragma unroll
            for (int i = 0; i < P; ++i) {
                sxx[i] = syy[i] = p[i] = T(0);
                const int z = z0 + i;
                if (r0 + i < 3 * k + 1 || r0 + i > rows - 2 - 3 * k) continue;
                const int szs = EZ ? strip(z) : -1;
                const bool u1 = xr1 && (!EZ || (z >= 2 && z < nz - 1)), u2 = xr2 && (!EZ || (z >= 1 && z < nz - 1));
                Vec4<T> ms;
                T mu_nxt;
                if constexpr (PAL) {
                    ms = lpal[PAL_MS * kMaxPalette + entry(i)];
                    mu_nxt = lpal[PAL_MS * kMaxPalette + entry(i + 1)].w;
                } else {
                    ms = mg[i];
                    mu_nxt = mg[i + 1].w;
                }
                T az = 0, bz = 1, rkz = 1, azh = 0, bzh = 1;
                if (szs >= 0) {
                    az = ktab[TB_AZ * A.tn + z], bz = ktab[TB_BZ * A.tn + z], rkz = ktab[TB_RKZ * A.tn + z];
                    azh = ktab[TB_AZH * A.tn + z], bzh = ktab[TB_BZH * A.tn + z];
                }
                // (x differences read other lanes' registers: every lane takes part, updated or not)
                T dvx = ddx_fwd(V[i].x, rdx), dwx = ddx_fwd(V[i].z, rdx), ddx = ddx_bwd(V[i].y, rdx);
                if (u1) {
                    T dvz = d4(vy[i + 2], vy[i + 1], vy[i + 3], vy[i], rdz);
                    T dwz = d4(wy[i + 2], wy[i + 1], wy[i + 3], wy[i], rdz);
                    if constexpr (EX)
                        if (sx >= 0) {
                            dvx = cpml_held(dvx, qx[i][PX_DVX], xt(TB_AXH), xt(TB_BXH), xt(TB_RKXH));
                            dwx = cpml_held(dwx, qx[i][PX_DWX], xt(TB_AXH), xt(TB_BXH), xt(TB_RKXH));
                        }
                    if constexpr (EZ)
                        if (szs >= 0) {
                            dvz = cpml_held(dvz, qz[i][PZ_DVZ], az, bz, rkz);
                            dwz = cpml_held(dwz, qz[i][PZ_DWZ], az, bz, rkz);
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
                    T ddz = d4(vx[i + 2], vx[i + 1], vx[i + 3], vx[i], rdz);
                    if constexpr (EX)
                        if (sx >= 0) ddx = cpml_held(ddx, qx[i][PX_DVY], xt(TB_AX), xt(TB_BX), xt(TB_RKX));
                    // half-grid memory coefficients, full-grid K_z divisor (reference :224-226)
                    if constexpr (EZ)
                        if (szs >= 0) ddz = cpml_held(ddz, qz[i][PZ_DVX], azh, bzh, rkz);
                    const T mu_xy = AVG ? harmonic_mu(ms.w, mu_nxt) : mu_nxt;
                    S[i].w = S[i].w + mu_xy * (ddx + ddz) * dt;
                }
            }
        }
        if constexpr (!PAL && !HOLD) groups(MVg, mg);
        bs[BS_SXY_L2][w][lane] = S[P - 2].w, bs[BS_SXY_L1][w][lane] = S[P - 1].w, bs[BS_SXY_F1][w][lane] = S[0].w;
        bs[BS_SYY_L1][w][lane] = syy[P - 1], bs[BS_SYY_F1][w][lane] = syy[0], bs[BS_SYY_F2][w][lane] = syy[1];
        bs[BS_P_L1][w][lane] = p[P - 1], bs[BS_P_F1][w][lane] = p[0], bs[BS_P_F2][w][lane] = p[1];
        __syncthreads();
        if (rec_on && (A.rec_mask & POE2D_P))
#pragma unroll
            for (int i = 0; i < P; ++i) record(i, A.rec_ncomp - 1, p[i]);

        // ---- velocities
        {
            T sy[P + 3], pp[P + 3], sh[P + 3];  // rows -1 .. P + 1 (syy, p), -2 .. P (sxy)
            sy[0] = bs[BS_SYY_L1][wb][lane], sy[P + 1] = bs[BS_SYY_F1][wa][lane], sy[P + 2] = bs[BS_SYY_F2][wa][lane];
            pp[0] = bs[BS_P_L1][wb][lane], pp[P + 1] = bs[BS_P_F1][wa][lane], pp[P + 2] = bs[BS_P_F2][wa][lane];
            sh[0] = bs[BS_SXY_L2][wb][lane], sh[1] = bs[BS_SXY_L1][wb][lane], sh[P + 2] = bs[BS_SXY_F1][wa][lane];
#pragma unroll
            for (int i = 0; i < P; ++i) sy[i + 1] = syy[i], pp[i + 1] = p[i], sh[i + 2] = S[i].w;
#pragma unroll
            for (int i = 0; i < P; ++i) {
                const int z = z0 + i;
                if (r0 + i < 3 * k + 3 || r0 + i > rows - 4 - 3 * k) continue;
                const int szj = EZ ? strip(z) : -1;
                const bool u4 = xr4 && (!EZ || (z >= 2 && z < nz)), u5 = xr5 && (!EZ || (z >= 1 && z < nz - 1));
                Vec4<T> mv, mv1, cn, cn1;
                if constexpr (PAL) {
                    mv = lpal[PAL_MV * kMaxPalette + entry(i)];
                    mv1 = lpal[PAL_MV * kMaxPalette + entry(i + 1)];
                    if constexpr (sizeof(T) == 4) {
                        cn = lpal[PAL_CN * kMaxPalette + entry(i)];
                        cn1 = lpal[PAL_CN * kMaxPalette + entry(i + 1)];
                    }
                } else {
                    mv = HOLD ? mh[i] : mg[i];
                    mv1 = HOLD ? mh[i + 1] : mg[i + 1];
                }
                T az = 0, bz = 1, rkz = 1, azh = 0, bzh = 1, rkzh = 1;
                if (szj >= 0) {
                    az = ktab[TB_AZ * A.tn + z], bz = ktab[TB_BZ * A.tn + z], rkz = ktab[TB_RKZ * A.tn + z];
                    azh = ktab[TB_AZH * A.tn + z], bzh = ktab[TB_BZH * A.tn + z], rkzh = ktab[TB_RKZH * A.tn + z];
                }
                T dsx = ddx_bwd(sxx[i], rdx), dpx = ddx_bwd(p[i], rdx), dhx = ddx_fwd(S[i].w, rdx);
                if (u4) {
                    T e1 = dsx;
                    T e2 = dpx;
                    T e3 = d4(sh[i + 2], sh[i + 1], sh[i + 3], sh[i], rdz);
                    if constexpr (EX)
                        if (sx >= 0) {
                            e1 = cpml_held(e1, qx[i][PX_DSXX], xt(TB_AX), xt(TB_BX), xt(TB_RKX));
                            e2 = cpml_held(e2, qx[i][PX_DPX], xt(TB_AX), xt(TB_BX), xt(TB_RKX));
                        }
                    if constexpr (EZ)
                        if (szj >= 0) e3 = cpml_held(e3, qz[i][PZ_DSXY], az, bz, rkz);
                    if constexpr (PAL && sizeof(T) == 4)
                        biot_velocity_cn(V[i].x, V[i].z, e1 + e3, e2, mv.x, mv.y, mv.z, cn);
                    else
                        biot_velocity(V[i].x, V[i].z, e1 + e3, e2, mv.x, mv.y, mv.z, mv.w, A.inv_dt);
                }
                if (u5) {
                    T e1 = dhx;
                    T e2 = d4(sy[i + 2], sy[i + 1], sy[i + 3], sy[i], rdz);
                    T e3 = d4(pp[i + 2], pp[i + 1], pp[i + 3], pp[i], rdz);
                    if constexpr (EX)
                        if (sx >= 0) e1 = cpml_held(e1, qx[i][PX_DSXY], xt(TB_AXH), xt(TB_BXH), xt(TB_RKXH));
                    if constexpr (EZ)
                        if (szj >= 0) {
                            e2 = cpml_held(e2, qz[i][PZ_DSYY], azh, bzh, rkzh);
                            e3 = cpml_held(e3, qz[i][PZ_DPZ], azh, bzh, rkzh);
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
            if constexpr (!PAL && !HOLD) groups(MSg, mg);
            publish();  // (every wave has read the velocities before: the stresses' barrier is past)
            __syncthreads();
        }
    }

    // ---- the owned points
    if (lane < halo || lane >= 64 - halo || c > nx) return;
    gchar *const Vn = gb + group_v(in ^ 1) * gsb;
    gchar *const Sn = gb + group_s(in ^ 1) * gsb;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int z = z0 + i;
        if (r0 + i < halo || z >= it.z1) continue;
        const nvec4<T> v = {V[i].x, V[i].y, V[i].z, V[i].w}, t = {S[i].x, S[i].y, S[i].z, S[i].w};
        if (stream) {
            asm volatile("" ::: "memory");  // (or the two branches' stores merge into ordinary ones)
            __builtin_nontemporal_store(v, (GN *)(Vn + off(z)));
            __builtin_nontemporal_store(t, (GN *)(Sn + off(z)));
            asm volatile("" ::: "memory");
        } else {
            *(GN *)(Vn + off(z)) = v;
            *(GN *)(Sn + off(z)) = t;
        }
        if constexpr (EDGE) {
            typedef T pair __attribute__((ext_vector_type(2)));
            typedef __attribute__((address_space(1))) pair GP;
            if constexpr (EX)
                if (sx >= 0) {
                    GP *const r = (GP *)px(in ^ 1, z);
#pragma unroll
                    for (int q = 0; q < NPSI_X / 2; ++q) r[q] = pair{qx[i][2 * q], qx[i][2 * q + 1]};
                }
            if constexpr (EZ) {
                const int s = strip(z);
                if (s >= 0) {
                    GP *const r = (GP *)pz(in ^ 1, s);
#pragma unroll
                    for (int q = 0; q < NPSI_Z / 2; ++q) r[q] = pair{qz[i][2 * q], qz[i][2 * q + 1]};
                }
            }
        }
    }
}

// ROOM: launches of at most one block per CU, which may then use twice the registers.  FP64 blocks
// always do.
template <class T, bool AVG, bool PAL, bool ROOM>
__global__ void __launch_bounds__(kTileThreads, sizeof(T) == 4 && !ROOM ? 4 : 2)
    tile_steps(const StepArgs<T> *__restrict__ models, const TileItem *__restrict__ work, int nwork, int per_xcd,
               long long n, int flip, int steps, int nst, int stream)
{
    __shared__ T bv[NBOUNDARY][kTileWaves][64], bs[NBOUNDARY][kTileWaves][64];
    __shared__ T xtab[NXTAB][64];
    __shared__ Vec4<T> lpal[PAL ? PAL_SECTIONS * kMaxPalette : 1];
    const int wi = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (wi >= nwork) return;
    const TileItem it = work[wi];
    if (it.model < 0) return;
    // (fields are read where used: held from the start, a hundred of them would spill)
    const __attribute__((address_space(4))) StepArgs<T> &A =
        *((const __attribute__((address_space(4))) StepArgs<T> *)models + it.model);
    const int in = (flip + A.pcur) & 1, halo = 3 * steps;
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
    auto region = [&](auto p, auto edge) {
        tile_region<T, decltype(p)::value, AVG, PAL, decltype(edge)::value, ROOM>(A, it, n, in, halo, nst, stream, bv, bs, xtab, lpal);
    };
    using std::integral_constant;
    constexpr integral_constant<int, tile_edge_p(PAL)> edge_p{};
    if (it.kind == TILE_EDGE) region(integral_constant<int, 3>{}, integral_constant<int, EDGE_X | EDGE_Z>{});
    else if (it.kind == TILE_EDGE_X) region(edge_p, integral_constant<int, EDGE_X>{});
    else if (it.kind == TILE_EDGE_Z) region(edge_p, integral_constant<int, EDGE_Z>{});
    else if (it.kind == TILE_SHORT) region(integral_constant<int, 3>{}, integral_constant<int, 0>{});
    else region(integral_constant<int, tile_tall_p(sizeof(T) == 4, PAL)>{}, integral_constant<int, 0>{});
}

template <class T>
hipError_t launch_tiles(const StepArgs<T> *models, const TileItem *work, int nwork, int per_xcd, bool palette, bool avg,
                        long long n, int flip, int steps, int nst, bool stream_out, hipStream_t stream)
{
    if (nwork < 1 || per_xcd < 1 || 8LL * per_xcd < nwork || steps < 2 || steps > kTileStepsMax || nst < 1 || nst > steps)
        return hipErrorInvalidValue;
    auto launch_as = [&](auto av, auto pal) {
        constexpr bool AVG = decltype(av)::value, PAL = decltype(pal)::value;
        const dim3 grid(8 * per_xcd);
        if (sizeof(T) == 8 || nwork <= kTileCus)
            tile_steps<T, AVG, PAL, true>
                <<<grid, kTileThreads, 0, stream>>>(models, work, nwork, per_xcd, n, flip, steps, nst, stream_out);
        else if constexpr (sizeof(T) == 4)
            tile_steps<T, AVG, PAL, false>
                <<<grid, kTileThreads, 0, stream>>>(models, work, nwork, per_xcd, n, flip, steps, nst, stream_out);
    };
    using Yes = std::true_type;
    using No = std::false_type;
    if (palette) avg ? launch_as(Yes{}, Yes{}) : launch_as(No{}, Yes{});
    else avg ? launch_as(Yes{}, No{}) : launch_as(No{}, No{});
    return hipGetLastError();
}

template hipError_t launch_tiles<float>(const StepArgs<float> *, const TileItem *, int, int, bool, bool, long long, int, int,
                                        int, bool, hipStream_t);
template hipError_t launch_tiles<double>(const StepArgs<double> *, const TileItem *, int, int, bool, bool, long long, int, int,
                                         int, bool, hipStream_t);

}  // namespace poe2d
