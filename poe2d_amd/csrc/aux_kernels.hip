// Small kernels around the time step: the receiver gather of the two-pass schedule, derived-field
// recompute and component extraction for snapshots, and the stability reduction.
#include "aux_kernels.h"

#include <algorithm>

namespace poe2d {

namespace {

template <class T>
__device__ T pressure_at(const StepArgs<T> &A, const Vec4<T> *S, const Vec4<T> *MS, int x, int z, long long o)
{
    if (!(x >= 1 && x < A.nx && z >= 2 && z < A.nz - 1)) return T(0);
    const Vec4<T> s = S[o], m = MS[o];
    T p = pore_pressure(s.x, s.y, s.z, m.x, m.y);
    if (A.src_kind == POE2D_SRC_PRESSURE_DGAUSS && x == A.src_x && z == A.src_z) p += A.src_val;
    return p;
}

template <class T>
__global__ void gather_kernel(StepArgs<T> A, int vbuf, int sbuf, Receivers R, T *out)
{
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= R.n) return;
    const int x = R.ix[r], z = R.iz[r];
    const long long o = (long long)z * A.pitch + x;
    const Vec4<T> v = state_group(A, group_v(vbuf))[o];
    int c = 0;
    if (R.mask & POE2D_VX) out[(size_t)(c++) * R.n + r] = v.x;
    if (R.mask & POE2D_VY) out[(size_t)(c++) * R.n + r] = v.y;
    if (R.mask & POE2D_P) out[(size_t)c * R.n + r] = pressure_at(A, state_group(A, group_s(sbuf)), mat_group(A, G_MS), x, z, o);
}

template <class T>
__global__ void derived_kernel(StepArgs<T> A, int buf, int what, T *out)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int z = blockIdx.y;
    if (x > A.nx || z > A.nz) return;
    const long long o = (long long)z * A.pitch + x;
    const Vec4<T> *S = state_group(A, group_s(buf));
    const Vec4<T> *MS = mat_group(A, G_MS);
    const T p = pressure_at(A, S, MS, x, z, o);
    T v = p;
    if (what != 0) {
        v = 0;
        if (x >= 1 && x < A.nx - 1 && z >= 2 && z < A.nz - 1) {
            const Vec4<T> s = S[o], m = MS[o];
            const T l2m = m.z + T(2) * m.w;
            v = what == 1 ? l2m * s.x + m.z * s.y - m.x * p : m.z * s.x + l2m * s.y - m.x * p;
        }
    }
    out[(size_t)z * (A.nx + 1) + x] = v;
}

template <class T>
__global__ void extract_kernel(StepArgs<T> A, int g, int comp, T *out)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int z = blockIdx.y;
    if (x > A.nx || z > A.nz) return;
    const Vec4<T> v = state_group(A, g)[(long long)z * A.pitch + x];
    out[(size_t)z * (A.nx + 1) + x] = comp == 0 ? v.x : comp == 1 ? v.y : comp == 2 ? v.z : v.w;
}

template <class T>
__global__ void insert_kernel(StepArgs<T> A, int g, int comp, const T *in)
{
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int z = blockIdx.y;
    if (x > A.nx || z > A.nz) return;
    Vec4<T> &v = state_group(A, g)[(long long)z * A.pitch + x];
    const T a = in[(size_t)z * (A.nx + 1) + x];
    if (comp == 0) v.x = a;
    else if (comp == 1) v.y = a;
    else if (comp == 2) v.z = a;
    else v.w = a;
}

// Largest |vx|, |vy| of points i = first, first + step, ... < npts (a block's 256 threads), non-finite
// as +inf.
template <class T>
__device__ float block_absmax(const Vec4<T> *V, long long npts, long long first, long long step)
{
    __shared__ float red[256];
    float m = 0.f;
    for (long long i = first; i < npts; i += step) {
        const Vec4<T> v = V[i];  // rows 0..nz, pad columns included (zero)
        float a = fabsf((float)v.x), b = fabsf((float)v.y);
        if (!(a <= 3.0e38f)) a = INFINITY;
        if (!(b <= 3.0e38f)) b = INFINITY;
        m = fmaxf(m, fmaxf(a, b));
    }
    red[threadIdx.x] = m;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    return red[0];
}

template <class T>
__global__ void __launch_bounds__(256) absmax_blocks(StepArgs<T> A, int buf, float *partial)
{
    const float m = block_absmax(state_group(A, group_v(buf)), (long long)(A.nz + 1) * A.pitch,
                                 blockIdx.x * 256LL + threadIdx.x, gridDim.x * 256LL);
    if (threadIdx.x == 0) partial[blockIdx.x] = m;
}

// Of several members (blockIdx.x, the grid's axis without a limit of 65 535): checked one after the other,
// 64 members of 1201 x 1201 points cost 128 launches and 64 read-backs after a batch run.
template <class T>
__global__ void __launch_bounds__(256) absmax_members(const FieldRange *ranges, float *partial)
{
    const FieldRange r = ranges[blockIdx.x];
    const float m = block_absmax((const Vec4<T> *)r.v, r.n, blockIdx.y * 256LL + threadIdx.x, gridDim.y * 256LL);
    if (threadIdx.x == 0) partial[(size_t)blockIdx.x * gridDim.y + blockIdx.y] = m;
}

// 16-byte stores over the aligned middle of each range, single words at its ends.
__global__ void __launch_bounds__(256) clear_kernel(ClearRanges r)
{
    const size_t first = blockIdx.x * 256ull + threadIdx.x, step = gridDim.x * 256ull;
    for (int k = 0; k < kClearRanges; ++k) {
        if (!r.words[k]) continue;
        unsigned *const p = (unsigned *)r.p[k];
        const size_t head = min((size_t)(4 - ((size_t)p / 4) % 4) % 4, r.words[k]), mid = (r.words[k] - head) / 4;
        uint4 *const q = (uint4 *)(p + head);
        for (size_t i = first; i < mid; i += step) q[i] = make_uint4(0, 0, 0, 0);
        const size_t tail = head + 4 * mid;
        if (first < head) p[first] = 0;
        if (first < r.words[k] - tail) p[tail + first] = 0;
    }
}

// 32 x 32 tiles through LDS, a row of 32 values per half wave on either side.
template <class T>
__global__ void __launch_bounds__(256) transpose_kernel(const T *in, size_t ld, int rows, int cols, T *out)
{
    __shared__ T tile[32][33];
    const int c0 = blockIdx.x * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int r0 = blockIdx.y * 32; r0 < rows; r0 += gridDim.y * 32) {
        for (int y = ty; y < 32; y += 8)
            if (r0 + y < rows && c0 + tx < cols) tile[y][tx] = in[(size_t)(r0 + y) * ld + c0 + tx];
        __syncthreads();
        for (int y = ty; y < 32; y += 8)
            if (c0 + y < cols && r0 + tx < rows) out[(size_t)(c0 + y) * rows + r0 + tx] = tile[tx][y];
        __syncthreads();
    }
}

// out[b] = largest of in[b * n .. b * n + n).
__global__ void __launch_bounds__(256) absmax_final(const float *in, int n, float *out)
{
    __shared__ float red[256];
    float m = 0.f;
    in += (size_t)blockIdx.x * n;
    for (int i = threadIdx.x; i < n; i += blockDim.x) m = fmaxf(m, in[i]);
    red[threadIdx.x] = m;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

}  // namespace

template <class T>
void launch_gather(const StepArgs<T> &A, int vbuf, int sbuf, const Receivers &R, T *out, hipStream_t stream)
{
    gather_kernel<T><<<(R.n + 255) / 256, 256, 0, stream>>>(A, vbuf, sbuf, R, out);
}

template <class T>
void launch_derived(const StepArgs<T> &A, int buf, int what, T *out, hipStream_t stream)
{
    derived_kernel<T><<<dim3((A.nx + 1 + 255) / 256, A.nz + 1), 256, 0, stream>>>(A, buf, what, out);
}

template <class T>
void launch_extract(const StepArgs<T> &A, int g, int comp, T *out, hipStream_t stream)
{
    extract_kernel<T><<<dim3((A.nx + 1 + 255) / 256, A.nz + 1), 256, 0, stream>>>(A, g, comp, out);
}

template <class T>
void launch_insert(const StepArgs<T> &A, int g, int comp, const T *in, hipStream_t stream)
{
    insert_kernel<T><<<dim3((A.nx + 1 + 255) / 256, A.nz + 1), 256, 0, stream>>>(A, g, comp, in);
}

template <class T>
void launch_absmax(const StepArgs<T> &A, int buf, float *partials, int nblocks, float *result, hipStream_t stream)
{
    absmax_blocks<T><<<nblocks, 256, 0, stream>>>(A, buf, partials);
    absmax_final<<<1, 256, 0, stream>>>(partials, nblocks, result);
}

template <class T>
void launch_absmax_members(const FieldRange *ranges, int n, float *partials, int nblocks, float *result, hipStream_t stream)
{
    absmax_members<T><<<dim3(n, nblocks), 256, 0, stream>>>(ranges, partials);
    absmax_final<<<n, 256, 0, stream>>>(partials, nblocks, result);
}

void launch_clear(const ClearRanges &r, hipStream_t stream)
{
    size_t words = 0;
    for (size_t w : r.words) words = std::max(words, w);
    const int blocks = (int)std::min<size_t>(std::max<size_t>((words + 4095) / 4096, 1), 2048);
    clear_kernel<<<blocks, 256, 0, stream>>>(r);
}

template <class T>
void launch_transpose(const T *in, size_t ld, int rows, int cols, T *out, hipStream_t stream)
{
    const dim3 grid((cols + 31) / 32, std::min((rows + 31) / 32, 4096));
    transpose_kernel<T><<<grid, 256, 0, stream>>>(in, ld, rows, cols, out);
}

__global__ void __launch_bounds__(256) cn_palette_kernel(Vec4<float> *pal, int npal, float inv_dt)
{
    const int e = (int)threadIdx.x;
    if (e >= npal) return;
    const Vec4<float> mv = pal[PAL_MV * kMaxPalette + e];
    float co, c1, c2;
    cn_coeffs(mv.x, mv.y, mv.z, mv.w, inv_dt, co, c1, c2);
    const float rhofb = mv.y * mv.w;
    pal[PAL_CN * kMaxPalette + e] = Vec4<float>{c2, __builtin_amdgcn_rcpf(c1), rhofb, __builtin_amdgcn_rcpf(co)};
}

void launch_cn_palette(Vec4<float> *pal, int npal, float inv_dt, hipStream_t stream)
{
    static_assert(kMaxPalette <= 256, "one thread per palette entry");
    cn_palette_kernel<<<1, 256, 0, stream>>>(pal, npal, inv_dt);
}

#define POE2D_AUX_INSTANTIATE(T)                                                                      \
    template void launch_gather<T>(const StepArgs<T> &, int, int, const Receivers &, T *, hipStream_t); \
    template void launch_derived<T>(const StepArgs<T> &, int, int, T *, hipStream_t);                 \
    template void launch_extract<T>(const StepArgs<T> &, int, int, T *, hipStream_t);                 \
    template void launch_insert<T>(const StepArgs<T> &, int, int, const T *, hipStream_t);            \
    template void launch_absmax<T>(const StepArgs<T> &, int, float *, int, float *, hipStream_t);         \
    template void launch_absmax_members<T>(const FieldRange *, int, float *, int, float *, hipStream_t); \
    template void launch_transpose<T>(const T *, size_t, int, int, T *, hipStream_t);
POE2D_AUX_INSTANTIATE(float)
POE2D_AUX_INSTANTIATE(double)
#undef POE2D_AUX_INSTANTIATE

}  // namespace poe2d
