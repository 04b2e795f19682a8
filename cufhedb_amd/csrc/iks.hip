// iks.hip -- batched identity key switching and small element-wise kernels.
//
// IdentityKeySwitch (thirdparty/TFHEpp/src/keyswitch.cpp:12-48):
//   b'   = b                         (same torus width)
//        = (b + 2^(W-33)) >> (W-32)  (64-bit domain -> 32-bit target)
//   for i < dn, j < t:  a_ij = ((a_i + 2^(W-1-t*basebit)) >> (W-(j+1)basebit)) & mask
//                       if a_ij != 0: res -= ksk[i][j][a_ij - 1]
// The reference runs this on the host CPU before every bootstrap
// (src/cuHEDB/gatebootstrap_gpu.cuh:42,59,...).  Here a batch is one launch
// from the reference's own key layout [dn][t][2^basebit - 1][tn + 1] for kinds
// 10 and 20 (basebit 10), where k_iks_rows reads every selected row whole, one
// workgroup per ciphertext, and k_iks_gather, for large batches, stages the
// rows of a position in LDS for 4096 ciphertexts; kind 21 (basebit 3) is the
// matrix product of iks21.hip.
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

// Gather form of the same switch for batches that select every key row
// several times: a workgroup of 1024 threads takes four ciphertexts per thread
// (1024 apart) on a slice of 16 output columns and a range of digit positions.
// A position's 1023 rows on the slice (64 KB, behind a zero row for digit 0)
// are staged in LDS, two buffers, the next position's words in flight in
// registers, and every lane adds the row that its digit selects: the key is
// read once per 4096 ciphertexts instead of once per ciphertext.  A row's four
// 16-byte chunks are rotated by its number (chunk k at k ^ (r >> 2)) so that
// the lanes' random rows meet all the banks.
//
// Bound by the key's way into the compute units: 64 KB a position in 64-byte
// pieces of 2692-byte rows, 4.0 TB/s over the chip (without it 8192
// ciphertexts take 2.3 of their 3.8 ms).  One MI355X, n0 = 672, against a
// workgroup per ciphertext: kind 10 2.0 against 2.5 ms at 3000 ciphertexts,
// 3.8 against 6.7 at 8192, 6.5 against 13.5 at 16384; kind 20 3.8 against 5.3,
// 7.3 against 14.3, 14.0 against 28.7.  Not kept: two ciphertexts per thread
// (4.6 at 8192), one word per load (4.2), each lane adding its own columns to
// the output (a line per lane: 9.1).
constexpr int kGatherCols = 16, kGatherPer = 4;
// from these batches on (kind 10 / 20): one round of the key costs the gather
// form 1.4-1.6 / 2.8-3.2 ms whatever the batch, k_iks_rows 0.82 / 1.75 us a
// ciphertext (2200: 1.86 against 1.82 ms, 2400: 1.92 against 1.99; kind 20,
// 1500: 3.27 against 2.64, 2048: 3.44 against 3.59)
constexpr int kGatherFrom10 = 2400, kGatherFrom20 = 2048;

template <class TD, int DN, int T, int BB>
__global__ __launch_bounds__(1024) void k_iks_gather(const TD *__restrict__ in,
                                                     const uint32_t *__restrict__ ksk,
                                                     uint32_t *__restrict__ out, int tn, int B,
                                                     int slices, int tiles, int per)
{
    constexpr int W = int(sizeof(TD) * 8);
    constexpr uint32_t mask = (1u << BB) - 1;
    constexpr int kRowsLds = 1 << BB;               // candidate rows, row 0 zero
    constexpr int kWords = 16 / int(sizeof(TD));    // mask words loaded at a time
    constexpr int kStep = kWords * T;               // positions between loads
    static_assert(kRowsLds == 1024 && T == 2, "one 16-byte chunk in four per thread and row");
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    __shared__ __align__(16) u32x4 buf[2][kRowsLds * 4];
    const int tid = threadIdx.x;
    // workgroups go to the eight XCDs in turn: an XCD's take the tiles and
    // slices of the same positions, which share the key rows' cache lines
    const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
    const int tile = loc % tiles, c0 = loc / tiles % slices * kGatherCols;
    const int split = xcd + 8 * (loc / tiles / slices);
    const int e0 = split * per, e1 = min(e0 + per, DN * T);
    if (e0 >= e1) return;
    const size_t row = size_t(tn) + 1;

    // chunk c of LDS row r: threads take rows tid / 4 + 256 k
    const int c = tid & 3;
    u32x4 v[4];
    const uint32_t row4 = uint32_t(row) * 4u;
    const uint32_t voff = uint32_t(tid >> 2) * row4 + 16u * c;  // of LDS row tid / 4 + 1
    auto fetch = [&](int e) {
        const char *base = reinterpret_cast<const char *>(ksk + size_t(e) * mask * row + c0);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            // key row tid / 4 + 256 k - 1; its place before the first is not stored
            const uint32_t o = k ? voff + (256u * k - 1u) * row4 : voff >= row4 ? voff - row4 : voff;
            __builtin_memcpy(&v[k], base + o, 16);
        }
    };
    auto store = [&](int b) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int r = (tid >> 2) + 256 * k;
            if (r) buf[b][4 * r + (c ^ ((r >> 2) & 3))] = v[k];
        }
    };
    if (tid < 8) buf[tid >> 2][tid & 3] = u32x4{0, 0, 0, 0};

    // the next kWords mask words of this thread's ciphertexts (the digits are
    // in the upper halves of 64-bit ones)
    const int b0 = tile * 1024 * kGatherPer + tid;
    u32x4 raw[kGatherPer];
    uint32_t acc[kGatherPer][kGatherCols];
#pragma unroll
    for (int n = 0; n < kGatherPer; n++)
#pragma unroll
        for (int k = 0; k < kGatherCols; k++) acc[n][k] = 0;

    fetch(e0);
    for (int e = e0; e < e1; e += kStep) {
#pragma unroll
        for (int n = 0; n < kGatherPer; n++)
            __builtin_memcpy(&raw[n], in + size_t(min(b0 + 1024 * n, B - 1)) * (DN + 1) + e / T, 16);
#pragma unroll 1
        for (int w = 0; w < kWords; w++) {
#pragma unroll
            for (int u = 0; u < T; u++) {
                const int p = e + T * w + u;
                store(u);
                if (p + 1 < e1) fetch(p + 1);
                __syncthreads();
                const char *rows = reinterpret_cast<const char *>(buf[u]);
#pragma unroll
                for (int n = 0; n < kGatherPer; n++) {
                    // a wave's 64 ciphertexts are neighbours: none of them
                    // left, nothing to add
                    if (__builtin_amdgcn_readfirstlane(b0 + 1024 * n) >= B) break;
                    const uint32_t x = raw[n][W == 32 ? 0 : 1] + (1u << (31 - BB * T));
                    const uint32_t d = x >> (32 - (u + 1) * BB) & mask;
                    const uint32_t at = d << 6 | (d << 2 & 0x30u);
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const u32x4 y = *reinterpret_cast<const u32x4 *>(rows + (at ^ uint32_t(16 * k)));
#pragma unroll
                        for (int q = 0; q < 4; q++) acc[n][4 * k + q] += y[q];
                    }
                    // one ciphertext's reads at a time, for their registers
#pragma unroll
                    for (int k = 0; k < kGatherCols; k++) asm volatile("" : "+v"(acc[n][k]));
                }
            }
#pragma unroll
            for (int n = 0; n < kGatherPer; n++)
                raw[n] = W == 32 ? __builtin_shufflevector(raw[n], raw[n], 1, 2, 3, 3)
                                 : __builtin_shufflevector(raw[n], raw[n], 2, 3, 3, 3);
        }
    }
    // 1024 ciphertexts at a time through LDS, so that the additions go out as
    // 16 adjacent words
    constexpr int kPad = kGatherCols + 1;
    uint32_t *flat = reinterpret_cast<uint32_t *>(buf);
    const int col = c0 + (tid & (kGatherCols - 1));
#pragma unroll
    for (int n = 0; n < kGatherPer; n++) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kGatherCols; q++) flat[tid * kPad + q] = acc[n][q];
        __syncthreads();
        const int first = tile * 1024 * kGatherPer + 1024 * n;
        for (int r = tid / kGatherCols; r < 1024 && first + r < B; r += 1024 / kGatherCols) {
            const size_t b = size_t(first + r);
            uint32_t x = 0u - flat[r * kPad + col - c0];
            if (split == 0 && col == tn) {
                const TD y = in[b * (DN + 1) + DN];
                x += W == 32 ? uint32_t(y) : uint32_t((y + (TD(1) << (W - 33))) >> (W - 32));
            }
            if (col <= tn) atomicAdd(out + b * row + col, x);
        }
    }
}

template <class TD, int DN, int T, int BB>
void launch_iks_gather(const TD *in, const uint32_t *ksk, uint32_t *out, int tn, int B, hipStream_t s)
{
    const int slices = (tn + 1 + kGatherCols - 1) / kGatherCols;
    const int tiles = (B + 1024 * kGatherPer - 1) / (1024 * kGatherPer);
    constexpr int kStep = 16 / int(sizeof(TD)) * T;
    auto range = [](int k) { return (DN * T / kStep + k - 1) / k * kStep; };
    // splits of the positions, eight at a time (one an XCD), so that the
    // workgroups fill the 256 compute units (one each), against about three
    // positions' worth of start and end per workgroup
    int split = 8;
    long best = 0;
    for (int k = 8; k <= 64; k += 8) {
        const long cost = (long(slices) * tiles * k + 255) / 256 * (range(k) + 3);
        if (k == 8 || cost < best) best = cost, split = k;
    }
    const size_t n = size_t(B) * (tn + 1);
    hipLaunchKernelGGL(k_fill_zero32, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, out, n);
    hipLaunchKernelGGL((k_iks_gather<TD, DN, T, BB>), dim3(unsigned(slices * tiles * split)),
                       dim3(1024), 0, s, in, ksk, out, tn, B, slices, tiles, range(split));
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
        // `tile` = workgroups per ciphertext over the digit positions; with 8
        // of them the gather form takes over where it is faster
        const int split = tile == 2 || tile == 4 || tile == 8 ? tile : 1;
        const bool gather = split == 8 && B >= (kind == 10 ? kGatherFrom10 : kGatherFrom20);
        const auto *x1 = static_cast<const uint32_t *>(in);
        const auto *x2 = static_cast<const uint64_t *>(in);
        if (kind == 10 && gather)
            launch_iks_gather<uint32_t, Lvl1::N, KS10::t, KS10::basebit>(x1, ksk, out, tn, B, s);
        else if (kind == 10)
            launch_iks_rows<uint32_t, Lvl1::N, KS10::t, KS10::basebit>(x1, ksk, out, tn, B, split, s);
        else if (gather)
            launch_iks_gather<uint64_t, Lvl2::N, KS20::t, KS20::basebit>(x2, ksk, out, tn, B, s);
        else
            launch_iks_rows<uint64_t, Lvl2::N, KS20::t, KS20::basebit>(x2, ksk, out, tn, B, split, s);
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
