// iks.hip -- batched identity key switching and small element-wise kernels.
//
// IdentityKeySwitch (thirdparty/TFHEpp/src/keyswitch.cpp:12-48):
//   b'   = b                         (same torus width)
//        = (b + 2^(W-33)) >> (W-32)  (64-bit domain -> 32-bit target)
//   for i < dn, j < t:  a_ij = ((a_i + 2^(W-1-t*basebit)) >> (W-(j+1)basebit)) & mask
//                       if a_ij != 0: res -= ksk[i][j][a_ij - 1]
// The reference runs this on the host CPU before every bootstrap
// (src/cuHEDB/gatebootstrap_gpu.cuh:42,59,...).  Here a batch is one launch
// of k_iks_rows (kinds 10 and 20, basebit 10), which reads every selected key
// row whole from the reference's own layout [dn][t][2^basebit - 1][tn + 1],
// one workgroup per ciphertext, or the matrix product of iks21.hip (kind 21,
// basebit 3).
#include "launch.hpp"
#include "params.hpp"

namespace fhe {

namespace {

// Whole-row form for large bases (kinds 10 and 20: basebit 10, 1023
// candidate rows per digit position, so ciphertexts rarely share a row): one
// workgroup per ciphertext, wave w takes every fourth digit position and
// reads each selected row whole (tn + 1 words as NCH = ceil((tn + 1) / 64)
// coalesced loads, one per lane and 64 columns), two rows at a time, so the
// memory system sees 2.5 KB contiguous requests with 2 NCH loads in flight
// per wave; the four waves' partial sums meet in LDS.  The loop body has no
// branch: a zero digit reads a valid row and discards it, and lanes past the
// last column read up to 63 words beyond the row (the device key carries
// kKskPadWords spare words) into sums that are never written.
template <class TD, int DN, int T, int BB, int NCH>
__global__ __launch_bounds__(256) void k_iks_rows(const TD *__restrict__ in,
                                                  const uint32_t *__restrict__ ksk,
                                                  uint32_t *__restrict__ out, int tn, int B)
{
    constexpr int W = int(sizeof(TD) * 8);
    constexpr int NDIG = DN * T;
    static_assert(NDIG % 64 == 0, "digit positions are split in multiples of 8 pairs");
    constexpr uint32_t mask = (1u << BB) - 1;
    constexpr size_t nd = (size_t(1) << BB) - 1;
    __shared__ uint16_t dig[NDIG];
    __shared__ uint32_t part[4][NCH * 64];
    const int b = blockIdx.x;
    if (b >= B) return;
    // split gridDim.y ways over the digit positions: this workgroup takes
    // [e0, e0 + per) and adds its sum into the zero-filled output
    const int nsplit = gridDim.y, per = NDIG / nsplit, e0 = blockIdx.y * per;
    const TD *c = in + size_t(b) * (DN + 1);
    const TD prec = TD(1) << (W - (1 + BB * T));
    for (int e = e0 + threadIdx.x; e < e0 + per; e += blockDim.x) {
        const int i = e / T, j = e % T;
        dig[e] = uint16_t(((c[i] + prec) >> (W - (j + 1) * BB)) & mask);
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const size_t row = size_t(tn) + 1;
    uint32_t acc[NCH];
#pragma unroll
    for (int j = 0; j < NCH; j++) acc[j] = 0;
    for (int e = e0 + wave; e < e0 + per; e += 8) {
        const uint32_t d0 = __builtin_amdgcn_readfirstlane(uint32_t(dig[e]));
        const uint32_t d1 = __builtin_amdgcn_readfirstlane(uint32_t(dig[e + 4]));
        const uint32_t keep0 = d0 ? 0xffffffffu : 0u, keep1 = d1 ? 0xffffffffu : 0u;
        const uint32_t *k0 = ksk + (size_t(e) * nd + (d0 ? d0 - 1 : 0)) * row + lane;
        const uint32_t *k1 = ksk + (size_t(e + 4) * nd + (d1 ? d1 - 1 : 0)) * row + lane;
        uint32_t v0[NCH], v1[NCH];
#pragma unroll
        for (int j = 0; j < NCH; j++) v0[j] = k0[64 * j];
#pragma unroll
        for (int j = 0; j < NCH; j++) v1[j] = k1[64 * j];
#pragma unroll
        for (int j = 0; j < NCH; j++) acc[j] -= (v0[j] & keep0) + (v1[j] & keep1);
    }
#pragma unroll
    for (int j = 0; j < NCH; j++) part[wave][lane + 64 * j] = acc[j];
    __syncthreads();
    uint32_t body;
    if constexpr (W == 32)
        body = uint32_t(c[DN]);
    else
        body = uint32_t((c[DN] + (TD(1) << (W - 33))) >> (W - 32));
    uint32_t *o = out + size_t(b) * row;
    if (nsplit == 1) {
        for (int k = threadIdx.x; k < int(row); k += blockDim.x)
            o[k] = (k == tn ? body : 0u) + part[0][k] + part[1][k] + part[2][k] + part[3][k];
    } else {
        // integer sums mod 2^32: the order of the workgroups' additions does
        // not change the result
        for (int k = threadIdx.x; k < int(row); k += blockDim.x)
            atomicAdd(o + k, (k == tn && blockIdx.y == 0 ? body : 0u) + part[0][k] + part[1][k] +
                                 part[2][k] + part[3][k]);
    }
}

__global__ void k_fill_zero32(uint32_t *p, size_t n)
{
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// launch k_iks_rows with NCH = ceil((tn + 1) / 64), tn <= kMaxN0, split
// ways over the digit positions (1, 2, 4 or 8; a split output is zeroed by a
// kernel first, so the launch stays capturable)
template <class TD, int DN, int T, int BB, int NCH = 1>
void launch_iks_rows(const TD *in, const uint32_t *ksk, uint32_t *out, int tn, int B, int split,
                     hipStream_t s)
{
    if constexpr (NCH < (kMaxN0 + 1 + 63) / 64) {
        if ((tn + 1 + 63) / 64 > NCH)
            return launch_iks_rows<TD, DN, T, BB, NCH + 1>(in, ksk, out, tn, B, split, s);
    }
    if (split > 1) {
        const size_t n = size_t(B) * (tn + 1);
        hipLaunchKernelGGL(k_fill_zero32, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, out, n);
    }
    hipLaunchKernelGGL((k_iks_rows<TD, DN, T, BB, NCH>), dim3(B, split), dim3(256), 0, s, in, ksk,
                       out, tn, B);
}

__global__ void k_tlwe1_lincomb(const uint32_t *__restrict__ a, const uint32_t *__restrict__ b,
                                int sa, int sb, uint32_t offset, uint32_t *__restrict__ out,
                                int B)
{
    const size_t gid = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    constexpr int W = Lvl1::N + 1;
    if (gid >= size_t(B) * W) return;
    uint32_t v = uint32_t(sa) * a[gid] + uint32_t(sb) * b[gid];
    if (gid % W == Lvl1::N) v += offset;
    out[gid] = v;
}

__global__ void k_tlwe1_add_body(uint32_t *__restrict__ tlwe, uint32_t add, int B)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < B) tlwe[size_t(b) * (Lvl1::N + 1) + Lvl1::N] += add;
}

__global__ void k_tv1_const(uint32_t *tv, uint32_t u)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < Lvl1::N) tv[i] = u;
}

// gpolygen (src/HEDB/comparison/tfhepp_utils.h:113-120): 2^scale * (i >> 6)
__global__ void k_tv1_ide(uint32_t *tv, uint32_t scale_bits)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < Lvl1::N) tv[i] = (1u << scale_bits) * uint32_t(i >> 6);
}

// out = in with `add` added to the body word (W words per TLWE)
template <class T>
__global__ void k_tlwe_copy_add_body(const T *__restrict__ in, T *__restrict__ out, int W, T add,
                                     int B)
{
    const size_t gid = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gid >= size_t(B) * W) return;
    T v = in[gid];
    if (gid % W == size_t(W - 1)) v += add;
    out[gid] = v;
}

// out = sa*a + sb*b (+ add on the body word); W words per TLWE.  b == nullptr
// drops the second term; b_bcast makes every record use b's first TLWE.
template <class T>
__global__ void k_tlwe_lincomb(const T *__restrict__ a, const T *__restrict__ b, int sa, int sb,
                               T add, T *__restrict__ out, int W, int b_bcast, int B)
{
    const size_t gid = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gid >= size_t(B) * W) return;
    const int e = int(gid % W);
    T v = T(sa) * a[gid];
    if (b) v += T(sb) * b[b_bcast ? size_t(e) : gid];
    if (e == W - 1) v += add;
    out[gid] = v;
}

// out = in << shift on every word (HomMSB's digit shift, msb_gpu.cuh:15-18)
template <class T>
__global__ void k_tlwe_shl(const T *__restrict__ in, T *__restrict__ out, int shift, size_t n)
{
    const size_t gid = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gid < n) out[gid] = in[gid] << shift;
}

template <class T>
__global__ void k_tlwe_add_body(T *__restrict__ tlwe, int W, T add, int B)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < B) tlwe[size_t(b) * W + W - 1] += add;
}

template <class T>
__global__ void k_tv_const(T *tv, T u, int N)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) tv[i] = u;
}

// gpolygen with padding 6: 2^scale * (i >> 6)
template <class T>
__global__ void k_tv_ide(T *tv, uint32_t scale_bits, int N)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) tv[i] = (T(1) << scale_bits) * T(i >> 6);
}

}  // namespace

template <class T>
hipError_t launch_tlwe_copy_add_body(const T *in, T *out, int W, T add, int B, hipStream_t s)
{
    if (B <= 0) return hipSuccess;
    const size_t n = size_t(B) * W;
    hipLaunchKernelGGL(k_tlwe_copy_add_body<T>, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s,
                       in, out, W, add, B);
    return hipGetLastError();
}
template hipError_t launch_tlwe_copy_add_body<uint32_t>(const uint32_t *, uint32_t *, int, uint32_t,
                                                        int, hipStream_t);
template hipError_t launch_tlwe_copy_add_body<uint64_t>(const uint64_t *, uint64_t *, int, uint64_t,
                                                        int, hipStream_t);

template <class T>
hipError_t launch_tlwe_lincomb(const T *a, const T *b, int sa, int sb, T add, T *out, int W,
                               bool b_bcast, int B, hipStream_t s)
{
    if (B <= 0) return hipSuccess;
    const size_t n = size_t(B) * W;
    hipLaunchKernelGGL(k_tlwe_lincomb<T>, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, a, b,
                       sa, sb, add, out, W, int(b_bcast), B);
    return hipGetLastError();
}
template hipError_t launch_tlwe_lincomb<uint32_t>(const uint32_t *, const uint32_t *, int, int,
                                                  uint32_t, uint32_t *, int, bool, int, hipStream_t);
template hipError_t launch_tlwe_lincomb<uint64_t>(const uint64_t *, const uint64_t *, int, int,
                                                  uint64_t, uint64_t *, int, bool, int, hipStream_t);

template <class T>
hipError_t launch_tlwe_shl(const T *in, T *out, int W, int shift, int B, hipStream_t s)
{
    if (B <= 0) return hipSuccess;
    const size_t n = size_t(B) * W;
    hipLaunchKernelGGL(k_tlwe_shl<T>, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, in, out,
                       shift, n);
    return hipGetLastError();
}
template hipError_t launch_tlwe_shl<uint32_t>(const uint32_t *, uint32_t *, int, int, int,
                                              hipStream_t);
template hipError_t launch_tlwe_shl<uint64_t>(const uint64_t *, uint64_t *, int, int, int,
                                              hipStream_t);

template <class T>
hipError_t launch_tlwe_add_body(T *tlwe, int W, T add, int B, hipStream_t s)
{
    if (B <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_tlwe_add_body<T>, dim3(unsigned((B + 255) / 256)), dim3(256), 0, s, tlwe,
                       W, add, B);
    return hipGetLastError();
}
template hipError_t launch_tlwe_add_body<uint32_t>(uint32_t *, int, uint32_t, int, hipStream_t);
template hipError_t launch_tlwe_add_body<uint64_t>(uint64_t *, int, uint64_t, int, hipStream_t);

template <class T>
hipError_t launch_tv_const(T *tv, T u, int N, hipStream_t s)
{
    hipLaunchKernelGGL(k_tv_const<T>, dim3(unsigned((N + 255) / 256)), dim3(256), 0, s, tv, u, N);
    return hipGetLastError();
}
template hipError_t launch_tv_const<uint32_t>(uint32_t *, uint32_t, int, hipStream_t);
template hipError_t launch_tv_const<uint64_t>(uint64_t *, uint64_t, int, hipStream_t);

template <class T>
hipError_t launch_tv_ide(T *tv, uint32_t scale_bits, int N, hipStream_t s)
{
    hipLaunchKernelGGL(k_tv_ide<T>, dim3(unsigned((N + 255) / 256)), dim3(256), 0, s, tv,
                       scale_bits, N);
    return hipGetLastError();
}
template hipError_t launch_tv_ide<uint32_t>(uint32_t *, uint32_t, int, hipStream_t);
template hipError_t launch_tv_ide<uint64_t>(uint64_t *, uint32_t, int, hipStream_t);

hipError_t launch_iks(int kind, const void *in, const uint32_t *ksk, uint32_t *out, int tn, int B,
                      hipStream_t s, int tile)
{
    if (B <= 0) return hipSuccess;
    switch (kind) {
    case 10:
    case 20: {
        // `tile` = workgroups per ciphertext over the digit positions
        const int split = tile == 2 || tile == 4 || tile == 8 ? tile : 1;
        if (kind == 10)
            launch_iks_rows<uint32_t, Lvl1::N, KS10::t, KS10::basebit>(
                static_cast<const uint32_t *>(in), ksk, out, tn, B, split, s);
        else
            launch_iks_rows<uint64_t, Lvl2::N, KS20::t, KS20::basebit>(
                static_cast<const uint64_t *>(in), ksk, out, tn, B, split, s);
        break;
    }
    case 21:
        return launch_iks21(static_cast<const uint64_t *>(in), ksk, out, B, tile, s);
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_tlwe1_lincomb(const uint32_t *a, const uint32_t *b, int sa, int sb,
                                uint32_t offset, uint32_t *out, int B, hipStream_t s)
{
    if (B <= 0) return hipSuccess;
    const size_t n = size_t(B) * (Lvl1::N + 1);
    hipLaunchKernelGGL(k_tlwe1_lincomb, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, a, b, sa,
                       sb, offset, out, B);
    return hipGetLastError();
}

hipError_t launch_tlwe1_add_body(uint32_t *tlwe, uint32_t add, int B, hipStream_t s)
{
    if (B <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_tlwe1_add_body, dim3(unsigned((B + 255) / 256)), dim3(256), 0, s, tlwe,
                       add, B);
    return hipGetLastError();
}

hipError_t launch_tv1_const(uint32_t *tv, uint32_t u, hipStream_t s)
{
    hipLaunchKernelGGL(k_tv1_const, dim3(Lvl1::N / 256), dim3(256), 0, s, tv, u);
    return hipGetLastError();
}

hipError_t launch_tv1_ide(uint32_t *tv, uint32_t scale_bits, hipStream_t s)
{
    hipLaunchKernelGGL(k_tv1_ide, dim3(Lvl1::N / 256), dim3(256), 0, s, tv, scale_bits);
    return hipGetLastError();
}

}  // namespace fhe
