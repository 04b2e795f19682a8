// iks21.hip -- lvl2 -> lvl1 identity key switching on the integer matrix cores.
//
// IdentityKeySwitch<lvl21param> (thirdparty/TFHEpp/src/keyswitch.cpp:12-48):
// every mask word gives ten 3-bit digits, and digit d != 0 of position (i, j)
// subtracts key row [i][j][d - 1], so the switch is
//   out[b] = (0, body) - sum over positions of f_ij(d), f_ij(0) = 0,
// a product of a one-hot matrix (ciphertexts x 8 slots per position) with the
// key.  The key's 32-bit words are split into four signed bytes (their sum
// with weights 2^8l is the word mod 2^32), which makes it an int8 product with
// exact 32-bit sums: a position selects at most two of the bytes, |sum| <=
// 2 * 20480 * 128 < 2^31.
//
// v_smfmac_i32_32x32x64_i8 multiplies a 2:4-sparse left operand at twice the
// dense rate, and one-hot digits are sparse: a position's eight slots are two
// groups of four.  With t = d mod 4 the lower group always selects slot t,
// f(t), and the upper one, when bit 2 of d is set, slot t of f(4 + t) - f(t);
// the second element of each group is zero.
//
// One 32x32x64 step covers eight positions: lanes 0-31 and 32-63 hold four
// (p = 0..3) each for their row (ciphertext).  Registers 0 and 1 are their
// lower groups (two a register, constant ones), registers 2 and 3 their upper
// groups (bit 2 of each digit); the index word repeats its half of four
// nibbles t.  Four mask words are a stage of five steps: lane half h takes
// words A = 4s + 2h, B = A + 1,
//   step 0: A digits 3-p   1: A digits 7-p   2: A 8, A 9, B 8, B 9 (from p = 3)
//   step 3: B digits 3-p   4: B digits 7-p.
// Key layout (one block of 40 KB per stage and 32 output columns):
//   [column block 32][stage 512][step 5][byte 4][h 2][lane 64][16 bytes],
// byte 4 p + t of (h, lane = n + 32 g) being slot t of the lower (g = 0) or
// upper (g = 1) group of position p of lane half h, column n.  The body
// column follows as [position][8] words.
#include <algorithm>

#include "common.hpp"
#include "launch.hpp"
#include "params.hpp"

namespace fhe {

namespace {

constexpr int kDn = Lvl2::N, kTn = Lvl1::N, kT = KS21::t, kNd = (1 << KS21::basebit) - 1;
constexpr int kBlocks = kTn / 32;             // column blocks
constexpr int kStages = kDn / 4;              // four mask words each
constexpr int kSteps = 5;                     // 32x32x64 steps per stage
constexpr int kStageBytes = kSteps * 4 * 2048;
constexpr size_t kMainBytes = size_t(kBlocks) * kStages * kStageBytes;
static_assert(kT == 10 && KS21::basebit == 3 && kTn % 32 == 0 && kDn % 4 == 0, "shape");

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));

// digit position (mask word of the stage 0..3, digit) of lane half h, step c,
// register p
__host__ __device__ constexpr int pos_word(int h, int c, int p)
{
    return 2 * h + (c < 2 ? 0 : c > 2 ? 1 : p < 2);
}
__host__ __device__ constexpr int pos_digit(int c, int p)
{
    return c == 0 || c == 3 ? 3 - p : c == 1 || c == 4 ? 7 - p : 9 - (p & 1);
}

// the reference layout [dn][t][7][tn + 1] -> the layout above
__global__ __launch_bounds__(256) void k_ksk21_layout(const uint32_t *__restrict__ ksk,
                                                      uint8_t *__restrict__ dst)
{
    // one thread: (block, stage, step, h, lane), 16 bytes of each byte plane
    const size_t e = size_t(blockIdx.x) * 256 + threadIdx.x;
    const int lane = int(e & 63), h = int(e >> 6) & 1;
    size_t r = e >> 7;
    const int c = int(r % kSteps);
    r /= kSteps;
    const int s = int(r % kStages), blk = int(r / kStages);
    const int col = blk * 32 + (lane & 31);
    uint32_t w[16];
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const size_t pos = size_t(4 * s + pos_word(h, c, p)) * kT + pos_digit(c, p);
        const uint32_t *f = ksk + pos * kNd * (kTn + 1) + col;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const uint32_t lower = t ? f[size_t(t - 1) * (kTn + 1)] : 0u;
            w[4 * p + t] = lane < 32 ? lower : f[size_t(3 + t) * (kTn + 1)] - lower;
        }
    }
    // signed bytes: (w + 0x80808080) ^ 0x80808080
#pragma unroll
    for (int j = 0; j < 16; j++) w[j] = (w[j] + 0x80808080u) ^ 0x80808080u;
    uint8_t *o = dst + ((size_t(blk) * kStages + s) * kSteps + c) * (4 * 2048) + h * 1024 + lane * 16;
#pragma unroll
    for (int l = 0; l < 4; l++) {
        uint32_t q[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            q[j] = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) q[j] |= ((w[4 * j + k] >> (8 * l)) & 0xffu) << (8 * k);
        }
        *reinterpret_cast<uint4 *>(o + l * 2048) = uint4{q[0], q[1], q[2], q[3]};
    }
}

__global__ __launch_bounds__(256) void k_ksk21_body(const uint32_t *__restrict__ ksk,
                                                    uint32_t *__restrict__ dst)
{
    const int e = blockIdx.x * 256 + threadIdx.x;  // position * 8 + digit
    const int d = e & 7;
    dst[e] = d ? ksk[(size_t(e >> 3) * kNd + d - 1) * (kTn + 1) + kTn] : 0u;
}

// NW waves, MT x 32 ciphertexts each, on 32 output columns and a range of
// stages.  All waves read the same key block: a stage's 40 KB are staged in
// LDS (two buffers) from registers that hold the next stage's words.
// The mask words' high halves pass through LDS too, 16 words of every row at
// a time (a 128-byte line, four stages), a quarter of the rows a stage: read
// by the lanes that use them they would cost the L1 a line per row and stage.
//
// What bounds it: up to 256 ciphertexts the key's 671 MB (0.14-0.15 ms, 4.7
// TB/s); from 512 on the matrix cores together with the waves' other
// instructions (16384 ciphertexts: 5.0 ms, 4.4 POPS of the 8.8 that the
// instruction alone reaches; 3.4-4.0 with operands that toggle less, so the
// clock gives way too).  One MI355X, against one ciphertext per lane with the
// rows summed from LDS (a column per lane below 512): 100 ciphertexts 1.86 ->
// 0.15 ms, 1024 2.7 -> 0.35, 4096 4.8 -> 1.25, 16384 15.3 -> 5.0.  Not kept:
// each lane reading its own mask words (6.2 ms), four waves of 4 x 32 (5.2
// against 4.1 at the same point), operands read ahead one by one with the
// stores in mid-stage (5.1 against 4.1).
template <int NW, int MT>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW / 4, NW / 4)))
void k_iks21(const uint64_t *__restrict__ in, const uint8_t *__restrict__ key,
             uint32_t *__restrict__ out, int B, int per, int add)
{
    constexpr int kThreads = 64 * NW, kRows = 32 * MT * NW;
    constexpr int kLoads = kStageBytes / 16 / kThreads;   // 16-byte words of a stage per thread
    constexpr int kPieces = 2 * kRows / kThreads;         // 16-byte pieces of a row quarter
    constexpr int kRowWords = 18;                         // 16 words, padded off the banks
    static_assert(kStageBytes / 16 % kThreads == 0 && 2 * kRows % kThreads == 0, "shape");
    __shared__ __align__(16) v4i buf[2][kStageBytes / 16];
    __shared__ __align__(16) uint32_t inw[2][kRows * kRowWords];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroups go to the eight XCDs in turn: each XCD takes four column
    // blocks, so the workgroups that read a key block share its L2
    const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
    const int blk = xcd * (kBlocks / 8) + loc % (kBlocks / 8);
    const int t0 = loc / (kBlocks / 8) * kRows;           // the workgroup's first ciphertext
    const int s0 = blockIdx.y * per;
    const v4i *src = reinterpret_cast<const v4i *>(key + (size_t(blk) * kStages + s0) * kStageBytes) + tid;

    v4i kv[kLoads];
    auto fetch = [&](int s) {
        const v4i *p = src + size_t(s) * (kStageBytes / 16);
#pragma unroll
        for (int k = 0; k < kLoads; k++) kv[k] = p[kThreads * k];
    };
    auto store = [&](int b) {
#pragma unroll
        for (int k = 0; k < kLoads; k++) buf[b][tid + kThreads * k] = kv[k];
    };
    // quarter q of the rows: mask words 16 g .. + 15 (of the range), two words
    // a piece, eight pieces a row
    v4i piece[kPieces];
    auto fetch_in = [&](int g, int q) {
#pragma unroll
        for (int k = 0; k < kPieces; k++) {
            const int e = tid + kThreads * k, r = t0 + q * (kRows / 4) + (e >> 3);
            __builtin_memcpy(&piece[k], in + size_t(min(r, B - 1)) * (kDn + 1) + 4 * s0 + 16 * g + 2 * (e & 7),
                             16);
        }
    };
    auto store_in = [&](int b, int q) {
#pragma unroll
        for (int k = 0; k < kPieces; k++) {
            const int e = tid + kThreads * k;
            // not before here: taken apart where they are loaded, the words
            // would be waited for there
            asm volatile("" : "+v"(piece[k]));
            *reinterpret_cast<uint2 *>(&inw[b][(q * (kRows / 4) + (e >> 3)) * kRowWords + 2 * (e & 7)]) =
                uint2{uint32_t(piece[k][1]), uint32_t(piece[k][3])};
        }
    };
    v16i acc[MT][4];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int l = 0; l < 4; l++)
#pragma unroll
            for (int k = 0; k < 16; k++) acc[m][l][k] = 0;

    fetch(0);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        fetch_in(0, q);
        store_in(0, q);
    }
    const int groups = per / 4;
    for (int g = 0; g < groups; g++) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int s = 4 * g + u;
            // this stage's key words into the buffer that every wave left
            // before the last barrier, and the next group's rows (the quarter
            // loaded in the last stage)
            store(u & 1);
            if (s + 1 < per) fetch(s + 1);
            if (u > 0 && g + 1 < groups) store_in((g + 1) & 1, u - 1);
            if (u == 0 && g > 0) store_in(g & 1, 3);
            if (g + 1 < groups) fetch_in(g + 1, u);
            __syncthreads();
            uint32_t xa[MT], xb[MT];
#pragma unroll
            for (int m = 0; m < MT; m++) {
                const uint2 x = *reinterpret_cast<const uint2 *>(
                    &inw[g & 1][((wave * MT + m) * 32 + (lane & 31)) * kRowWords + 4 * u + 2 * half]);
                xa[m] = x.x + 2u;  // rounded: + 2^33 on the 64-bit word
                xb[m] = x.y + 2u;
            }
            const v4i *kb = buf[u & 1] + lane;
#pragma unroll
            for (int c = 0; c < kSteps; c++) {
                v8i kf[4];
#pragma unroll
                for (int l = 0; l < 4; l++)
                    kf[l] = __builtin_shufflevector(kb[(c * 4 + l) * 128], kb[(c * 4 + l) * 128 + 64], 0, 1, 2,
                                                    3, 4, 5, 6, 7);
#pragma unroll
                for (int m = 0; m < MT; m++) {
                    // the step's four digits of this lane, digit p from bit 3 p
                    const uint32_t y = c == 0 ? xa[m] >> 20
                                     : c == 1 ? (xa[m] >> 8) & 0xfffu
                                     : c == 3 ? xb[m] >> 20
                                     : c == 4 ? (xb[m] >> 8) & 0xfffu
                                              : ((xa[m] << 4) & 0xfc0u) | ((xb[m] >> 2) & 0x3fu);
                    // bits 2 of digits 0 and 1, of 2 and 3, sixteen apart
                    const uint32_t r = y | y << 13;
                    const v4i a{0x10001, 0x10001, int((r >> 2) & 0x10001u), int((r >> 8) & 0x10001u)};
                    // their low two bits from 3 p to 4 p: digits 2 and 3 up by
                    // two (fields times four), then 1 and 3 up by one (twice)
                    uint32_t z = y & 03333u;
                    z += (z & 03300u) * 3u;
                    z += z & 0x1818u;
                    const int idx = int(z | z << 16);
#pragma unroll
                    for (int l = 0; l < 4; l++)
                        acc[m][l] = __builtin_amdgcn_smfmac_i32_32x32x64_i8(a, kf[l], acc[m][l], idx, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const int b = t0 + (wave * MT + m) * 32 + 8 * (k >> 2) + 4 * half + (k & 3);
            const uint32_t sum = uint32_t(acc[m][0][k]) + (uint32_t(acc[m][1][k]) << 8) +
                                 (uint32_t(acc[m][2][k]) << 16) + (uint32_t(acc[m][3][k]) << 24);
            uint32_t *o = out + size_t(b) * (kTn + 1) + blk * 32 + (lane & 31);
            if (b < B) {
                if (add)
                    atomicAdd(o, 0u - sum);
                else
                    *o = 0u - sum;
            }
        }
}

// the rounded bodies; zero: also clear the mask words, which k_iks21 then
// adds to
__global__ __launch_bounds__(256) void k_iks21_init(const uint64_t *__restrict__ in,
                                                    uint32_t *__restrict__ out, int B, int zero)
{
    const size_t e = size_t(blockIdx.x) * 256 + threadIdx.x;
    const size_t b = zero ? e / (kTn + 1) : e;
    if (b >= size_t(B)) return;
    const int k = zero ? int(e % (kTn + 1)) : kTn;
    uint32_t w = 0;
    if (k == kTn) w = uint32_t((in[b * (kDn + 1) + kDn] + (1ull << 31)) >> 32);
    out[b * (kTn + 1) + k] = w;
}

// body column: one ciphertext per lane over kBodyWords mask words, the
// column's key words in LDS (a position's eight candidates are eight adjacent
// banks, so a wave's reads do not conflict)
constexpr int kBodyWords = 64;
__global__ __launch_bounds__(256) void k_iks21_bodies(const uint64_t *__restrict__ in,
                                                      const uint32_t *__restrict__ body,
                                                      uint32_t *__restrict__ out, int B)
{
    __shared__ uint32_t tab[kBodyWords * kT * 8];
    const int i0 = blockIdx.y * kBodyWords;
    for (int e = threadIdx.x; e < kBodyWords * kT * 8; e += 256) tab[e] = body[size_t(i0) * kT * 8 + e];
    __syncthreads();
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= B) return;
    const uint32_t *x = reinterpret_cast<const uint32_t *>(in + size_t(b) * (kDn + 1) + i0) + 1;
    uint32_t sum = 0;
#pragma unroll 4
    for (int i = 0; i < kBodyWords; i++) {
        const uint32_t w = x[2 * i] + 2u;
#pragma unroll
        for (int j = 0; j < kT; j++) sum += tab[(i * kT + j) * 8 + ((w >> (29 - 3 * j)) & 7u)];
    }
    atomicAdd(out + size_t(b) * (kTn + 1) + kTn, 0u - sum);
}

template <int NW, int MT>
void launch_main(const uint64_t *in, const uint8_t *key, uint32_t *out, int B, int split, hipStream_t s)
{
    constexpr int rows = 32 * MT * NW;
    const int tiles = (B + rows - 1) / rows;
    hipLaunchKernelGGL((k_iks21<NW, MT>), dim3(unsigned(kBlocks * tiles), unsigned(split)),
                       dim3(64 * NW), 0, s, in, key, out, B, kStages / split, int(split > 1));
}

}  // namespace

size_t ksk21_bytes() { return kMainBytes + size_t(kDn) * kT * 8 * 4; }

hipError_t launch_ksk21_layout(const uint32_t *ksk, uint32_t *dst, hipStream_t s)
{
    const size_t n = size_t(kBlocks) * kStages * kSteps * 128;
    auto *bytes = reinterpret_cast<uint8_t *>(dst);
    hipLaunchKernelGGL(k_ksk21_layout, dim3(unsigned(n / 256)), dim3(256), 0, s, ksk, bytes);
    hipLaunchKernelGGL(k_ksk21_body, dim3(kDn * kT * 8 / 256), dim3(256), 0, s, ksk,
                       reinterpret_cast<uint32_t *>(bytes + kMainBytes));
    return hipGetLastError();
}

hipError_t launch_iks21(const uint64_t *in, const uint32_t *key, uint32_t *out, int B, int tile,
                        hipStream_t s)
{
    const auto *bytes = reinterpret_cast<const uint8_t *>(key);
    const int rows = tile == 64 ? 512 : tile == 32 ? 256 : 128;
    const int tiles = (B + rows - 1) / rows;
    // split the stages so that the workgroups fill the compute units (one
    // each), weighing the rounds against about six stages' worth of start and
    // end per workgroup
    int split = 1;
    long best = 0;
    for (int k = 1; k <= 32; k *= 2) {
        const long rounds = (long(kBlocks) * tiles * k + 255) / 256;
        const long cost = rounds * (kStages / k + 6);
        if (k == 1 || cost < best) best = cost, split = k;
    }
    const size_t n = split > 1 ? size_t(B) * (kTn + 1) : size_t(B);
    hipLaunchKernelGGL(k_iks21_init, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, in, out, B,
                       int(split > 1));
    if (rows == 512)
        launch_main<8, 2>(in, bytes, out, B, split, s);
    else if (rows == 256)
        launch_main<8, 1>(in, bytes, out, B, split, s);
    else
        launch_main<4, 1>(in, bytes, out, B, split, s);
    hipLaunchKernelGGL(k_iks21_bodies, dim3(unsigned((B + 255) / 256), kDn / kBodyWords), dim3(256), 0,
                       s, in, reinterpret_cast<const uint32_t *>(bytes + kMainBytes), out, B);
    return hipGetLastError();
}

}  // namespace fhe
