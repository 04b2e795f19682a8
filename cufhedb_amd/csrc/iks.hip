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
// 10 and 20 (basebit 10), rows at whole 128-byte lines (ksk_row_words), where
// k_iks_rows reads every selected row whole, one workgroup per ciphertext, and
// k_iks_gather, for large batches, stages the rows of a position in LDS for
// 4096 ciphertexts; kind 21 (basebit 3) is the matrix product of iks21.hip.
#include "launch.hpp"
#include "params.hpp"

namespace fhe {

namespace {

// workgroups per ciphertext that a few ciphertexts take, at most
constexpr int kMaxSplit = 64;

// Whole-row form for large bases (kinds 10 and 20: basebit 10, 1023
// candidate rows per digit position, so ciphertexts rarely share a row): one
// workgroup per ciphertext, wave w takes every fourth digit position and
// reads each selected row whole (tn + 1 words as NCH = ceil((tn + 1) / 64)
// coalesced loads, one per lane and 64 columns), two rows at a time, so the
// memory system sees 2.5 KB contiguous requests with 2 NCH loads in flight
// per wave; the four waves' partial sums meet in LDS.  The loop body has no
// branch: a zero digit reads a valid row and discards it, and lanes past the
// last column read up to 63 words beyond the row (the device key carries
// kKskPadWords spare words) into sums that are never written.  (Rows at whole
// lines: 1.63 ms for 2000 ciphertexts of kind 10, 1.66 when packed.)
template <class TD, int DN, int T, int BB, int NCH>
__global__ __launch_bounds__(256) void k_iks_rows(const TD *__restrict__ in,
                                                  const uint32_t *__restrict__ ksk,
                                                  uint32_t *__restrict__ out, int tn, int B)
{
    constexpr int W = int(sizeof(TD) * 8);
    constexpr int NDIG = DN * T;
    static_assert(NDIG % (8 * kMaxSplit) == 0,
                  "every workgroup's range is whole steps of 8 positions at any split");
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
    const size_t row = size_t(tn) + 1, stride = size_t(ksk_row_words(tn));
    uint32_t acc[NCH];
#pragma unroll
    for (int j = 0; j < NCH; j++) acc[j] = 0;
    for (int e = e0 + wave; e < e0 + per; e += 8) {
        const uint32_t d0 = __builtin_amdgcn_readfirstlane(uint32_t(dig[e]));
        const uint32_t d1 = __builtin_amdgcn_readfirstlane(uint32_t(dig[e + 4]));
        const uint32_t keep0 = d0 ? 0xffffffffu : 0u, keep1 = d1 ? 0xffffffffu : 0u;
        const uint32_t *k0 = ksk + (size_t(e) * nd + (d0 ? d0 - 1 : 0)) * stride + lane;
        const uint32_t *k1 = ksk + (size_t(e + 4) * nd + (d1 ? d1 - 1 : 0)) * stride + lane;
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
// ways over the digit positions (a power of two up to kMaxSplit; a split
// output is zeroed by a kernel first, so the launch stays capturable)
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

// A few ciphertexts leave their workgroups waiting for one pair of rows after
// the other, so they are split further, up to 512 workgroups (one MI355X,
// n0 = 672, kind 10, split 8 / 16 / 32 / 64, us: 1 ciphertext 19.0 / 12.1 /
// 8.2 / 6.6, 8 24.6 / 15.4 / 11.2 / 11.5, 32 35.3 / 34.5 / 36.0 / 36.4, 64
// 64.7 / 66.1 / 66.7 / 68.6; kind 20, 1 36.7 / 20.5 / 12.4 / 8.9, 16 57.0 /
// 36.5 / 35.6 / 36.6; split 128 is slower again from two ciphertexts on)
constexpr int kSplitWorkgroups = 512;

// Gather form of the same switch for batches that select every key row
// several times: a workgroup of 1024 threads takes 4096 ciphertexts on a slice
// of 16 output columns and a range of digit positions.  A position's 1023 rows
// on the slice (64 KB, behind a zero row for digit 0) are staged in LDS, two
// buffers, the next position's words in flight in registers; a quad of lanes
// holds the slice's sums of 16 ciphertexts, four columns a lane, and adds the
// rows that their digits select: the key is read once per 4096 ciphertexts
// instead of once per ciphertext.  A quad's read is a row's 64 bytes, so the
// four quads that LDS serves in a cycle meet in its four bank groups; with a
// whole row per lane 16 lanes met in 16.  The digits come as byte offsets
// through LDS, each formed by one thread of the workgroup.
//
// Bound by the key's way into the compute units: 64 KB a position in 64-byte
// pieces of rows, one line each (without it 8192 ciphertexts take 2.0 of their
// 3.0 ms; rows packed without regard to lines, 2692 bytes apart: 3.4).  One
// MI355X, n0 = 672, against a row per lane on packed rows: kind 10 1.7 against
// 1.9 ms at 2400 ciphertexts, 2.1 against 2.5 at 4096, 3.0 against 3.8 at
// 8192, 5.0 against 6.6 at 16384; kind 20 3.0 against 3.5 at 2048, 5.9 against
// 7.4 at 8192.  Not kept: mask words loaded two at a time for their registers
// (the words' lines are read again: 3.2 at 8192), slices stored one after the
// other (2.7 at 8192, but 64-byte pieces double k_iks_rows' time).
constexpr int kGatherCols = 16, kGatherPer = 16;  // columns a workgroup, ciphertexts a quad
constexpr int kGatherTile = 256 * kGatherPer;     // ciphertexts a workgroup

// How the gather form splits a batch of B on tn + 1 output columns.
struct GatherShape {
    int slices, tiles, split, per;  // split: ranges of `per` digit positions
    long rounds, cost;              // of workgroups, one a unit; in positions
};

template <class TD, int DN, int T>
GatherShape gather_shape(int tn, int B)
{
    GatherShape g{};
    g.slices = (tn + 1 + kGatherCols - 1) / kGatherCols;
    g.tiles = (B + kGatherTile - 1) / kGatherTile;
    constexpr int kStep = 16 / int(sizeof(TD)) * T;
    // splits of the positions, eight at a time (one an XCD), so that the
    // workgroups fill the 256 compute units (one each), against about three
    // positions' worth of start and end per workgroup
    for (int k = 8; k <= 64; k += 8) {
        const int per = (DN * T / kStep + k - 1) / k * kStep;
        const long rounds = (long(g.slices) * g.tiles * k + 255) / 256;
        const long cost = rounds * (per + 3);
        if (k == 8 || cost < g.cost) g.split = k, g.per = per, g.rounds = rounds, g.cost = cost;
    }
    return g;
}

// Whether B ciphertexts are worth the gather form: a position of one of its
// rounds costs 3.7 to 5.2 us whatever the batch, k_iks_rows 0.56 ns per
// 1000 ciphertexts, positions and words of a row, so the line lies where
// k_iks_rows would read as many words as it can in the gather form's time.
// Staging a position is slowest when one round holds all workgroups (they all
// wait for the same positions), and slower when the rows' distance is an even
// number of lines, more so a multiple of four (they meet in fewer of the
// memory's channels).  Measured at 30 widths from 31 to 1025 columns, both
// kinds, 1400 to 2600 ciphertexts; lines by this rule against the crossing (kind
// 10 / 20): n0 = 255 2299 / 2273 against 2189 / 2331, 511 2273 / 2260 against
// 2007 / 2151, 636 2020 / 1974 against 1959 / 1941, 672 2030 / 1943 against
// 1982 / 1747, 1000 1952 / 1941 against 1699 / 1809; at no width of 400 and up is
// the choice more than 2 % slower than k_iks_rows (one line for all widths, 2000 /
// 1700: 31 % at n0 = 255, 12 % at 636).  From 2350 ciphertexts on the gather
// form is the faster one at every width.
constexpr int kGatherFrom = 2350;

template <class TD, int DN, int T>
bool gather_pays(int tn, int B)
{
    if (B >= kGatherFrom) return true;
    const GatherShape g = gather_shape<TD, DN, T>(tn, B);
    const int stride = ksk_row_words(tn), lines = stride / 32;
    const long unit = g.rounds == 1 ? 9200 : lines % 4 == 0 ? 7900 : lines % 2 == 0 ? 7600 : 6600;
    return long(B) * stride * (DN * T) >= unit * 1000 * g.cost;
}

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
    struct alignas(16) Lds {
        u32x4 row[2][kRowsLds * 4];
        uint16_t at[2][256][kGatherPer];  // byte offset of the row that a ciphertext selects
    };
    __shared__ Lds lds;
    const int tid = threadIdx.x;
    // workgroups go to the eight XCDs in turn: an XCD's take the tiles and
    // slices of the same positions, which share the key rows' cache lines
    const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
    const int tile = loc % tiles, c0 = loc / tiles % slices * kGatherCols;
    const int split = xcd + 8 * (loc / tiles / slices);
    const int e0 = split * per, e1 = min(e0 + per, DN * T);
    if (e0 >= e1) return;
    const size_t row = size_t(tn) + 1;
    const uint32_t stride = uint32_t(ksk_row_words(tn));

    // chunk c of LDS row r: threads take rows tid / 4 + 256 k
    const int c = tid & 3;
    u32x4 v[4];
    const uint32_t row4 = stride * 4u;
    const uint32_t voff = uint32_t(tid >> 2) * row4 + 16u * c;  // of LDS row tid / 4 + 1
    auto fetch = [&](int e) {
        const char *base = reinterpret_cast<const char *>(ksk + size_t(e) * mask * stride + c0);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            // key row tid / 4 + 256 k - 1; its place before the first is not stored
            const uint32_t o = k ? voff + (256u * k - 1u) * row4 : voff >= row4 ? voff - row4 : voff;
            v[k] = *reinterpret_cast<const u32x4 *>(base + o);
        }
    };
    auto store = [&](int b) {
#pragma unroll
        for (int k = 0; k < 4; k++)
            if (k || tid >= 4) lds.row[b][tid + 1024 * k] = v[k];
    };
    if (tid < 8) lds.row[tid >> 2][tid & 3] = u32x4{0, 0, 0, 0};

    // ciphertext of quad g = tid / 4 and sum n: b0 + 256 n + g.  This thread
    // provides the digits of quad `dg`, sums 4 dn to 4 dn + 3: raw holds their
    // next kWords mask words (the digits are in the upper halves of 64-bit ones)
    const int b0 = tile * kGatherTile, g = tid >> 2, dg = tid & 255, dn = tid >> 8;
    u32x4 raw[kGatherPer / 4];
    uint32_t acc[kGatherPer][4];
#pragma unroll
    for (int n = 0; n < kGatherPer; n++)
#pragma unroll
        for (int k = 0; k < 4; k++) acc[n][k] = 0;

    auto load_words = [&](int e) {
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const size_t b = size_t(min(b0 + 256 * (4 * dn + m) + dg, B - 1));
            __builtin_memcpy(&raw[m], in + b * (DN + 1) + e / T, 16);
        }
    };

    fetch(e0);
    load_words(e0);
    for (int e = e0; e < e1; e += kStep) {
#pragma unroll 1
        for (int w = 0; w < kWords; w++) {
#pragma unroll
            for (int u = 0; u < T; u++) {
                const int p = e + T * w + u;
                store(u);
                uint32_t x[4];
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const uint32_t d = (raw[m][W == 32 ? 0 : 1] + (1u << (31 - BB * T))) >> (32 - (u + 1) * BB);
                    x[m] = (d & mask) << 6;
                }
                *reinterpret_cast<uint64_t *>(&lds.at[u][dg][4 * dn]) =
                    uint64_t(x[2] | x[3] << 16) << 32 | (x[0] | x[1] << 16);
                if (u == T - 1) {
#pragma unroll
                    for (int m = 0; m < 4; m++)
                        raw[m] = W == 32 ? __builtin_shufflevector(raw[m], raw[m], 1, 2, 3, 3)
                                         : __builtin_shufflevector(raw[m], raw[m], 2, 3, 3, 3);
                    if (w == kWords - 1 && p + 1 < e1) load_words(p + 1);
                }
                if (p + 1 < e1) fetch(p + 1);
                __syncthreads();
                const char *rows = reinterpret_cast<const char *>(lds.row[u]) + 16 * c;
                const u32x4 *at = reinterpret_cast<const u32x4 *>(lds.at[u][g]);
#pragma unroll
                for (int h = 0; h < kGatherPer / 8; h++) {
                    const u32x4 o = at[h];
#pragma unroll
                    for (int j = 0; j < 8; j++) {
                        const int n = 8 * h + j;
                        const uint32_t a = j & 1 ? o[j >> 1] >> 16 : o[j >> 1] & 0xffffu;
                        const u32x4 y = *reinterpret_cast<const u32x4 *>(rows + a);
#pragma unroll
                        for (int q = 0; q < 4; q++) acc[n][q] += y[q];
                        // four rows' reads at a time, for their registers
                        if (j & 4 ? j == 7 : j == 3)
#pragma unroll
                            for (int k = n - 3; k <= n; k++)
#pragma unroll
                                for (int q = 0; q < 4; q++) asm volatile("" : "+v"(acc[k][q]));
                    }
                }
            }
        }
    }
    // 1024 ciphertexts at a time through LDS, so that the additions go out as
    // 16 adjacent words
    constexpr int kPad = kGatherCols + 1;
    uint32_t *flat = reinterpret_cast<uint32_t *>(lds.row);
    const int col = c0 + (tid & (kGatherCols - 1));
#pragma unroll
    for (int n = 0; n < kGatherPer; n += 4) {
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 4; m++)
#pragma unroll
            for (int q = 0; q < 4; q++) flat[(256 * m + g) * kPad + 4 * c + q] = acc[n + m][q];
        __syncthreads();
        const int first = b0 + 256 * n;
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

// rows first .. first + count - 1, packed in src, to their places in the key;
// the words between them are zeroed
__global__ __launch_bounds__(256) void k_ksk_spread(const uint32_t *__restrict__ src,
                                                    uint32_t *__restrict__ key, int row, int stride,
                                                    size_t count)
{
    const size_t gid = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (gid >= count * stride) return;
    const size_t r = gid / stride;
    const int k = int(gid % stride);
    key[gid] = k < row ? src[r * row + k] : 0u;
}

template <class TD, int DN, int T, int BB>
void launch_iks_gather(const TD *in, const uint32_t *ksk, uint32_t *out, int tn, int B, hipStream_t s)
{
    const GatherShape g = gather_shape<TD, DN, T>(tn, B);
    const size_t n = size_t(B) * (tn + 1);
    hipLaunchKernelGGL(k_fill_zero32, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, out, n);
    hipLaunchKernelGGL((k_iks_gather<TD, DN, T, BB>), dim3(unsigned(g.slices * g.tiles * g.split)),
                       dim3(1024), 0, s, in, ksk, out, tn, B, g.slices, g.tiles, g.per);
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

hipError_t launch_ksk_spread(uint32_t *key, int tn, size_t rows, uint32_t *tmp, size_t tmp_rows,
                             hipStream_t s)
{
    const size_t row = size_t(tn) + 1, stride = size_t(ksk_row_words(tn));
    // the packed rows start rows * (stride - row) words into the buffer, so a
    // row's place ends before the next packed row starts: in ascending order,
    // a part at a time through tmp, no row is overwritten before it is read
    const uint32_t *packed = key + rows * (stride - row);
    for (size_t r = 0; r < rows; r += tmp_rows) {
        const size_t n = rows - r < tmp_rows ? rows - r : tmp_rows;
        const hipError_t e = hipMemcpyAsync(tmp, packed + r * row, n * row * sizeof(uint32_t),
                                            hipMemcpyDeviceToDevice, s);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_ksk_spread, dim3(unsigned((n * stride + 255) / 256)), dim3(256), 0, s,
                           tmp, key + r * stride, int(row), int(stride), n);
    }
    return hipGetLastError();
}

hipError_t launch_iks(int kind, const void *in, const uint32_t *ksk, uint32_t *out, int tn, int B,
                      hipStream_t s, int tile)
{
    if (B <= 0) return hipSuccess;
    switch (kind) {
    case 10:
    case 20: {
        // `tile` = workgroups per ciphertext over the digit positions; 8 of
        // them become more for a few ciphertexts, and the gather form takes
        // over from 8 where it is faster
        int split = tile == 2 || tile == 4 || tile == 8 ? tile : 1;
        const bool gather = split == 8 && (kind == 10 ? gather_pays<uint32_t, Lvl1::N, KS10::t>(tn, B)
                                                      : gather_pays<uint64_t, Lvl2::N, KS20::t>(tn, B));
        if (split == 8)
            while (split < kMaxSplit && 2 * split * B <= kSplitWorkgroups) split *= 2;
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
