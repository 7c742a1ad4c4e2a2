// Strided copy of bit patterns between two views of the same shape and type.  Either side may be pinned host
// memory, which the kernels read and write over PCIe directly: host access to a tensor is one launch that moves
// the data and changes its layout at once, instead of a transfer and a pass of the host over every element.
#include "common.hpp"

namespace {

// Same layout on both sides, 16 bytes per lane.
__global__ void __launch_bounds__(256) copy_flat(uint4 *__restrict__ dst, const uint4 *__restrict__ src, int64_t nvec)
{
    for(int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < nvec; i += (int64_t)gridDim.x * 256)
        dst[i] = src[i];
}

// Channels-first <-> channels-last.  A block moves a tile of `ct` channels x `pt` pixels through LDS: the side
// that is channels-first is accessed along the pixels, the other along the channels (the whole tile is one run
// of memory when it holds all channels), so that neighbouring lanes are neighbours in memory on both sides.
constexpr int TILE_MAX = 5184;

template <typename T, bool TO_LAST>
__global__ void __launch_bounds__(256)
    copy_transpose(T *__restrict__ dst, const T *__restrict__ src, int C, int HW, int64_t npitch, int64_t pitch, int ct,
                   int pt, int tiles_c, int tiles_p)
{
    __shared__ T tile[TILE_MAX];
    const int lp = ct | 1; // odd: pixels of one channel fall into different banks
    const int b = blockIdx.x, tp = b % tiles_p, tc = (b / tiles_p) % tiles_c, n = b / (tiles_p * tiles_c);
    const int c0 = tc * ct, p0 = tp * pt;
    const int cn = C - c0 < ct ? C - c0 : ct, pn = HW - p0 < pt ? HW - p0 : pt;
    const int64_t first = (int64_t)n * npitch + (int64_t)c0 * HW + p0, last = ((int64_t)n * HW + p0) * pitch + c0;
    if(TO_LAST) {
        for(int e = threadIdx.x; e < cn * pn; e += 256) {
            const int c = e / pn, p = e - c * pn;
            tile[p * lp + c] = src[first + (int64_t)c * HW + p];
        }
    } else {
        for(int e = threadIdx.x; e < cn * pn; e += 256) {
            const int p = e / cn, c = e - p * cn;
            tile[p * lp + c] = src[last + (int64_t)p * pitch + c];
        }
    }
    __syncthreads();
    if(TO_LAST) {
        for(int e = threadIdx.x; e < cn * pn; e += 256) {
            const int p = e / cn, c = e - p * cn;
            dst[last + (int64_t)p * pitch + c] = tile[p * lp + c];
        }
    } else {
        for(int e = threadIdx.x; e < cn * pn; e += 256) {
            const int c = e / pn, p = e - c * pn;
            dst[first + (int64_t)c * HW + p] = tile[p * lp + c];
        }
    }
}

template <typename T> __global__ void __launch_bounds__(256) copy_strided(DView dst, DView src, int64_t total)
{
    for(int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        int64_t r = i, so = 0, d = 0;
#pragma unroll
        for(int j = 3; j >= 0; j--) {
            const int64_t q = r / dst.d[j], c = r - q * dst.d[j];
            so += c * src.s[j];
            d += c * dst.s[j];
            r = q;
        }
        ((T *)dst.ptr)[d] = ((const T *)src.ptr)[so];
    }
}

template <typename T> int run(const SagaTensorView *src, const SagaTensorView *dst, hipStream_t st)
{
    const int64_t total = view_elements(src);
    CLInfo sl, dl;
    CFInfo sf, df;
    const bool src_first = as_channels_first(src, &sf), dst_first = as_channels_first(dst, &df);
    const bool src_last = as_channels_last(src, &sl), dst_last = as_channels_last(dst, &dl);
    const int64_t CHW = (int64_t)src->dims[1] * src->dims[2] * src->dims[3];
    const bool dense = (src_first && dst_first && sf.npitch == CHW && df.npitch == CHW) ||
                       (src_last && dst_last && sl.pitch == sl.C && dl.pitch == dl.C);
    if(dense && aligned16(src->ptr) && aligned16(dst->ptr) && total * sizeof(T) % 16 == 0) {
        const int64_t nvec = total * sizeof(T) / 16;
        copy_flat<<<grid_for(nvec, 256), 256, 0, st>>>((uint4 *)dst->ptr, (const uint4 *)src->ptr, nvec);
        return 0;
    }
    if(((src_first && dst_last) || (src_last && dst_first)) && !dense && CHW / src->dims[1] < (1ll << 30)) {
        const int C = src->dims[1], HW = (int)(CHW / C);
        const int ct = C < 64 ? C : 64;
        int pt = 4096 / ct & ~63; // at least one wavefront of pixels
        pt = pt > 1024 ? 1024 : pt;
        const int tiles_c = (C + ct - 1) / ct, tiles_p = (HW + pt - 1) / pt;
        const int64_t blocks = (int64_t)src->dims[0] * tiles_c * tiles_p;
        if(blocks < (1ll << 31)) {
            if(src_first && dst_last)
                copy_transpose<T, true><<<(unsigned)blocks, 256, 0, st>>>((T *)dst->ptr, (const T *)src->ptr, C, HW, sf.npitch,
                                                                          dl.pitch, ct, pt, tiles_c, tiles_p);
            else
                copy_transpose<T, false><<<(unsigned)blocks, 256, 0, st>>>((T *)dst->ptr, (const T *)src->ptr, C, HW,
                                                                           df.npitch, sl.pitch, ct, pt, tiles_c, tiles_p);
            return 0;
        }
    }
    copy_strided<T><<<grid_for(total, 256), 256, 0, st>>>(dview(dst), dview(src), total);
    return 0;
}

} // namespace

extern "C" int saga_hip_copy(const SagaTensorView *src, const SagaTensorView *dst, saga_stream_t stream)
{
    if(!valid_view(src) || !valid_view(dst))
        return SAGA_HIP_EINVAL;
    if(!same_dims(src, dst) || src->dtype != dst->dtype)
        return SAGA_HIP_ESHAPE;
    hipStream_t st = as_stream(stream);
    switch(dtype_size(src->dtype)) {
    case 1: run<uint8_t>(src, dst, st); break;
    case 2: run<uint16_t>(src, dst, st); break;
    case 4: run<uint32_t>(src, dst, st); break;
    default: run<uint64_t>(src, dst, st); break;
    }
    SAGA_CHECK_LAUNCH();
    return 0;
}
