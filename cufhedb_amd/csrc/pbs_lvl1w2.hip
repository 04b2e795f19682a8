// pbs_lvl1w2.hip -- lvl1 blind rotation with two waves per polynomial and the
// digit rows side by side, for batches too small to fill the GPU with one
// wave per ciphertext; and with the rows in turn, for larger ones
// (k_blind_rotate1w2_pair).
//
// Same computation as k_blind_rotate1 (pbs_lvl1.hip; TFHEpp BlindRotate,
// gatebootstrapping.hpp:15-43, CMUX detwfa.cpp:21-30, external product
// trgsw.cpp:78-103), with a whole compute unit on one ciphertext: each
// polynomial is split over two waves (256 of the 512 complex points each, 4
// per lane), the six digit rows of a CMUX step are transformed at once by
// twelve waves, and four more carry the two accumulator columns back.  The
// transform (512 = 4 x 128) exchanges once between its two waves:
//   step A (registers): u_k[n0] = w^(n0 (4k+1)) sum_p c_p z[n0 + 128 p] i^(pk),
//           c_p = exp(i pi p / 8), n0 = lane + 64 wave < 128, k < 4;
//   exchange: wave v takes u_k for k = 2v, 2v+1 (all 128 n0);
//   step C: per sequence, radix 2 over n0 = L + 64 h, twiddle W128^(L m1),
//           then the 64-point DFT over the lanes (lanes64_fwd).
// Time domain: wave w, lane L, register p holds z[L + 64 w + 128 p],
// z_n = a_n + i a_(n+512).  Frequency domain: wave w, lane l, register q
// holds Z[f1w(w, l, q)].  The key is the one-wave kernel's device key with
// each (i, row, col) slice permuted into this order (same FD values).
#include "fft64.hpp"
#include "launch.hpp"
#include "params.hpp"

namespace fhe {

namespace {

constexpr int N1 = Lvl1::N;
constexpr int kPolyW = 512;  // complex points per polynomial
constexpr uint32_t kDecOffW = decomp_total_offset<uint32_t, 32, Lvl1::l, Lvl1::Bgbit>();
constexpr uint32_t kDigitFlipW = (1u << 31) | (1u << 25) | (1u << 19);

// natural frequency of (wave, lane, register) in the output layout
__host__ __device__ constexpr int f1w(int w, int l, int q)
{
    return 4 * (((l >> 4) & 1) + 2 * (((l >> 2) & 3) + 4 * (l & 3) + 16 * q)) + 2 * w + (l >> 5);
}

struct TwW {
    cd beta, rho;  // w^n0, w^(4 n0), n0 = lane + 64 wave, w = exp(i pi / 1024)
    cd t128;       // W128^lane
    cd t64, t16;   // lanes64 twiddles
};

__device__ __forceinline__ TwW make_tww(int lane, int wave)
{
    TwW t;
    const int n0 = lane + 64 * wave;
    t.beta = unit_root(double(n0), 1024.0);
    t.rho = unit_root(double(n0), 256.0);
    t.t128 = unit_root(double(lane), 64.0);
    t.t64 = unit_root(double(lane & 15), 32.0);
    t.t16 = unit_root(double(lane & 3), 8.0);
    return t;
}

// exp(i pi p / 8), p = 1..3
__device__ __forceinline__ cd c8w(int p)
{
    constexpr double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173;
    return p == 1 ? cd{c1, s1} : p == 2 ? cd{kR2, kR2} : cd{s1, c1};
}

// The exchanges of the transforms.  A wave keeps the words of its own two
// sequences and trades the others with the other half, two words a lane each
// way: put_* before the caller's barrier, get_* behind it on the tile that the
// other half wrote.  Forward (seqs), from the four sequences' words at the
// wave's n0 to its sequence s at n0 of half h in register 2 s + h; inverse
// (parts), back.  The empty asm keeps the two branches apart: merged, a load
// becomes one into a selected register and v moves to scratch.  (Whole
// exchanges through LDS: 2.39 against 2.35 ms at one ciphertext, 4.9 against
// 4.75 at 300.)
__device__ __forceinline__ void put_seqs(const cd v[4], cd *tile, int lane, int half)
{
    if (half == 0) {
        asm volatile("; half 0: in");
        tile[lane] = v[2];
        tile[64 + lane] = v[3];
        asm volatile("; half 0: out");
    } else {
        asm volatile("; half 1: in");
        tile[lane] = v[0];
        tile[64 + lane] = v[1];
        asm volatile("; half 1: out");
    }
}

__device__ __forceinline__ void get_seqs(cd v[4], const cd *tile, int lane, int half)
{
    if (half == 0) {
        asm volatile("; half 0: in");
        v[2] = v[1];
        v[1] = tile[lane];
        v[3] = tile[64 + lane];
        asm volatile("; half 0: out");
    } else {
        asm volatile("; half 1: in");
        v[1] = v[2];
        v[0] = tile[lane];
        v[2] = tile[64 + lane];
        asm volatile("; half 1: out");
    }
}

__device__ __forceinline__ void put_parts(const cd v[4], cd *tile, int lane, int half)
{
    if (half == 0) {
        asm volatile("; half 0: in");
        tile[lane] = v[1];
        tile[64 + lane] = v[3];
        asm volatile("; half 0: out");
    } else {
        asm volatile("; half 1: in");
        tile[lane] = v[0];
        tile[64 + lane] = v[2];
        asm volatile("; half 1: out");
    }
}

__device__ __forceinline__ void get_parts(cd v[4], const cd *tile, int lane, int half)
{
    if (half == 0) {
        asm volatile("; half 0: in");
        v[1] = v[2];
        v[2] = tile[lane];
        v[3] = tile[64 + lane];
        asm volatile("; half 0: out");
    } else {
        asm volatile("; half 1: in");
        v[2] = v[1];
        v[0] = tile[lane];
        v[1] = tile[64 + lane];
        asm volatile("; half 1: out");
    }
}

// The forward transform of one wave's half, in two parts around the exchange
// between the two halves: after part A the caller puts the other half's words
// into its tile (put_seqs), part C goes on behind the barrier in the half's own
// tile, which no other wave touches until the next exchange.
__device__ __forceinline__ void fft512w_fwd_a(cd v[4], const TwW &tw)
{
    v[1] = cmul(v[1], c8w(1));
    v[2] = cmul(v[2], c8w(2));
    v[3] = cmul(v[3], c8w(3));
    dft4<1>(v[0], v[1], v[2], v[3]);
    {
        cd g = tw.beta;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            v[k] = cmul(v[k], g);
            if (k < 3) g = cmul(g, tw.rho);
        }
    }
}

__device__ __forceinline__ void fft512w_fwd_c(cd v[4], cd *tile, int lane, int half, const TwW &tw)
{
    get_seqs(v, tile, lane, half);
    wave_lds_sync();
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const cd a = v[2 * s], b = v[2 * s + 1];
        v[2 * s] = cadd(a, b);
        v[2 * s + 1] = cmul(csub(a, b), tw.t128);
    }
    lanes64_fwd<true, true>(v, tile, lane, tw.t64, tw.t16);
}

// The inverse (unnormalised: returns 512 z), frequency layout in, time layout
// out, in two parts around the exchange: part A ends with the other half's
// words in the wave's own tile, part C reads the other half's tile.
__device__ __forceinline__ void fft512w_inv_a(cd v[4], cd *tile, int lane, int half, const TwW &tw)
{
    lanes64_inv<true, true>(v, tile, lane, tw.t64, tw.t16);
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const cd a = v[2 * s], b = cmulc(v[2 * s + 1], tw.t128);
        v[2 * s] = cadd(a, b);
        v[2 * s + 1] = csub(a, b);
    }
    put_parts(v, tile, lane, half);
}

__device__ __forceinline__ void fft512w_inv_c(cd v[4], const cd *theirs, int lane, int half,
                                              const TwW &tw)
{
    get_parts(v, theirs, lane, half);
    {
        cd g = tw.beta;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            v[k] = cmulc(v[k], g);
            if (k < 3) g = cmul(g, tw.rho);
        }
    }
    dft4<-1>(v[0], v[1], v[2], v[3]);
    v[1] = cmulc(v[1], c8w(1));
    v[2] = cmulc(v[2], c8w(2));
    v[3] = cmulc(v[3], c8w(3));
}

constexpr int kRowWaves = 2 * Lvl1::rows;     // two halves per digit row
constexpr int kColWaves = 4;                  // two halves per accumulator column
constexpr int kWaves = kRowWaves + kColWaves; // 16: also (column, half, register) of the products
static_assert(kWaves == 2 * 2 * 4, "one product wave per column, half and register");

// LDS of one blind rotation (108 KB of the CU's 160).  ext holds a column
// followed by its negation and the column again, so that coefficient n of
// X^a acc is word ((n - a) mod 2N) + k with the wrap's sign in the data and
// the lane's eight words at immediate offsets from one base.
struct alignas(16) Br1wLds {
    cd row[kRowWaves][kLaneTile];  // row waves' tiles, then their row's spectrum
    cd col[kColWaves][kLaneTile];  // product sums, then the column waves' tiles
    uint32_t ext[2][3 * N1];
    uint32_t step[kMaxN0 + 1];
    int rank[kWaves];
};
static_assert(64 * kWaves >= kMaxN0, "one thread per step");

// One workgroup of 16 waves per ciphertext, one workgroup per compute unit.
// A CMUX step, with a barrier after each phase:
//   1. row waves (12: digit row r, half h) rotate and decompose their own
//      256 points of the row and run the transform up to its exchange;
//   2. they finish it and leave the row's spectrum in their tile;
//   3. all 16 waves form the products: wave (column, half, register) sums
//      the six rows in row order for its 64 points, with the key words
//      loaded one step ahead;
//   4. column waves (4: column, half) run the inverse up to its exchange;
//   5. they finish it and add it to their words of the accumulator (kept in
//      registers), writing the three copies the rotation reads.
// Every value is computed by the same operations in the same order whatever
// the batch size.
//
// Bound by the LDS writes of the row waves (74-80 bytes a clock) and by the
// chain through the five barriers, about 7,500 cycles a step (8,100 with whole
// exchanges and lane bits 2-3 through LDS: 1,420 / 3,030 / 750 / 1,870 / 1,050
// by phase); it is for
// batches that leave the chip idle.  One MI355X, n0 = 672, up to 256
// ciphertexts: 2.2 ms against 4.5-4.6 with the rows one after the other
// on two waves.  Not kept: all lane exchanges as DPP selects (no LDS traffic,
// but about 8 cycles an instruction: phase 2 3,950), the first exchange
// through LDS instead of register swaps (3,970), loading the key words right
// after the products (96 KB through the 64-byte L1 port: phase 3 1,930).
__global__ __launch_bounds__(64 * kWaves) void k_blind_rotate1w2(
    const uint32_t *__restrict__ in, int n0, const cd *__restrict__ bk,
    const uint32_t *__restrict__ tv, int tv_stride, uint32_t *__restrict__ out, int sample_extract,
    int B)
{
    __shared__ Br1wLds lds;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ct = blockIdx.x;
    if (ct >= B) return;
    const uint32_t *c0 = in + size_t(ct) * (n0 + 1);
    const uint32_t *tvp = tv + size_t(ct) * tv_stride;
    const int half = wave & 1;
    const TwW tw = make_tww(lane, half);
    const int nb = lane + 64 * half;
    const bool is_row = wave < kRowWaves;
    // row waves: the row's column and digit.  The digit's sign flip is an
    // addition into its field's top bit (its carry leaves the field upwards):
    // digit = signed field of (X^a acc - acc) + kd.
    const int rcol = (wave >> 1) / Lvl1::l, rdig = (wave >> 1) % Lvl1::l;
    const int sh = 32 - Lvl1::Bgbit * (rdig + 1);
    const uint32_t kd = kDecOffW + (1u << (sh + Lvl1::Bgbit - 1));
    // column waves: their column and the words lane + 64 half + 128 p (+ 512)
    const int col = (wave - kRowWaves) >> 1;
    uint32_t own[8];
    auto put = [&](int k) {
        uint32_t *e = lds.ext[col] + nb + 128 * (k >> 1) + 512 * (k & 1);
        e[0] = own[k];
        e[N1] = 0u - own[k];
        e[2 * N1] = own[k];
    };

    // acc = (0, X^bbar tv), bbar = 2N - (b >> 21)   (no rounding)
    if (!is_row) {
        const uint32_t bbar = 2u * N1 - (c0[n0] >> (32 - 1 - Lvl1::nbit));
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int n = nb + 128 * (k >> 1) + 512 * (k & 1);
            const uint32_t idx = (uint32_t(n) - bbar) & (2u * N1 - 1);
            const uint32_t v = tvp[idx & (N1 - 1)];
            own[k] = col == 0 ? 0u : (idx & N1) ? 0u - v : v;
            put(k);
        }
    }

    // the steps with a rotation to do (a-bar = 0 is skipped), in order, as
    // i << 12 | a-bar: thread i ranks its step among the nonzero ones
    constexpr uint32_t kRound = 1u << (32 - 2 - Lvl1::nbit);
    {
        const uint32_t abar = tid < n0 ? (c0[tid] + kRound) >> (32 - 1 - Lvl1::nbit) : 0u;
        const uint64_t some = __ballot(abar != 0);
        if (lane == 0) lds.rank[wave] = __popcll(some);
        __syncthreads();
        int at = 0, all = 0;
        for (int w = 0; w < kWaves; w++) {
            if (w == wave) at = all;
            all += lds.rank[w];
        }
        if (abar) lds.step[at + __popcll(some & ((1ull << lane) - 1))] = uint32_t(tid) << 12 | abar;
        if (tid == 0) lds.step[all] = 0;
    }
    // product wave: column, and slot (half, register) of 64 points
    const int pcol = wave >> 3, slot = wave & 7;
    cd key[Lvl1::rows];
    auto load_key = [&](uint32_t step) {
        const cd *k = bk + (size_t(step >> 12) * Lvl1::rows * 2 + pcol) * kPolyW + slot * 64 + lane;
#pragma unroll
        for (int r = 0; r < Lvl1::rows; r++) key[r] = k[r * 2 * kPolyW];
    };
    __syncthreads();
    uint32_t step = __builtin_amdgcn_readfirstlane(lds.step[0]);
    if (step) load_key(step);

    for (int k = 1; step; k++) {
        const uint32_t ahead = lds.step[k];
        cd v[4];
        if (is_row) {
            const uint32_t *rot = lds.ext[rcol] + ((uint32_t(nb) - step) & (2u * N1 - 1));
            const uint32_t *neg = lds.ext[rcol] + N1 + nb;
            double x[8];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int o = 128 * (k >> 1) + 512 * (k & 1);
                x[k] = double(int32_t(__builtin_amdgcn_sbfe(int32_t(rot[o] + neg[o] + kd), sh, Lvl1::Bgbit)));
            }
#pragma unroll
            for (int p = 0; p < 4; p++) v[p] = cd{x[2 * p], x[2 * p + 1]};
            fft512w_fwd_a(v, tw);
            put_seqs(v, lds.row[wave ^ 1], lane, half);
        }
        __syncthreads();
        if (is_row) {
            fft512w_fwd_c(v, lds.row[wave], lane, half, tw);
#pragma unroll
            for (int q = 0; q < 4; q++) lds.row[wave][q * 64 + lane] = v[q];
        }
        __syncthreads();
        {
            cd fd{0.0, 0.0};
#pragma unroll
            for (int r = 0; r < Lvl1::rows; r++)
                cmac(fd, lds.row[2 * r + (slot >> 2)][(slot & 3) * 64 + lane], key[r]);
            lds.col[2 * pcol + (slot >> 2)][(slot & 3) * 64 + lane] = fd;
        }
        __syncthreads();
        if (!is_row) {
            cd *tile = lds.col[wave - kRowWaves];
#pragma unroll
            for (int q = 0; q < 4; q++) v[q] = tile[q * 64 + lane];
            wave_lds_sync();
            fft512w_inv_a(v, tile, lane, half, tw);
        }
        // the next step's key words, in flight until its products
        step = __builtin_amdgcn_readfirstlane(ahead);
        if (step) load_key(step);
        __syncthreads();
        if (!is_row) {
            fft512w_inv_c(v, lds.col[(wave - kRowWaves) ^ 1], lane, half, tw);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                own[k] += trunc_torus32(k & 1 ? v[k >> 1].y : v[k >> 1].x);
                put(k);
            }
        }
        __syncthreads();
    }

    if (sample_extract) {
        // SampleExtractIndex 0: out[0] = acc0[0], out[n] = -acc0[N - n], out[N] = acc1[0]
        uint32_t *o = out + size_t(ct) * (N1 + 1);
        o[tid] = tid == 0 ? lds.ext[0][0] : lds.ext[0][2 * N1 - tid];
        if (tid == 0) o[N1] = lds.ext[1][0];
    } else {
        uint32_t *o = out + size_t(ct) * 2 * N1;
        o[tid] = lds.ext[0][tid];
        o[N1 + tid] = lds.ext[1][tid];
    }
}

// gadget digits (trgsw.cpp:21-39) of (X^a acc - acc) at coefficient n, a in
// [0, 2N), as one signed field extract of the word prepared with the offset and
// the flipped top bit of every 6-bit field
__device__ __forceinline__ uint32_t prep_rot(const uint32_t *poly, uint32_t a, int n)
{
    const uint32_t idx = (uint32_t(n) - a) & (2u * N1 - 1);
    uint32_t v = poly[idx & (N1 - 1)];
    if (idx & N1) v = 0u - v;
    return (v - poly[n] + kDecOffW) ^ kDigitFlipW;
}
__device__ __forceinline__ double digit_w(uint32_t u, int d)
{
    const int sh = 32 - Lvl1::Bgbit * (d + 1);
    return double(int32_t(__builtin_amdgcn_sbfe(int32_t(u), sh, Lvl1::Bgbit)));
}

// Two waves and 18 KB of LDS per ciphertext, the digit rows one after the
// other: six ciphertexts fit a compute unit, so batches of more than two rounds
// of k_blind_rotate1w2's one per unit are faster here (one MI355X, n0 = 672, ms
// against k_blind_rotate1w2: 513 to 768 ciphertexts 6.4-6.5 / 6.7, 1024 6.9 /
// 8.9, 4096 25.6 / 35.5, 8192 52.5 / 70.9; up to 256 4.4-4.5 / 2.2, 512 6.5 /
// 4.5).  The same operations per value in the same order, hence the same words.
// Three waves per SIMD (166 VGPRs, no spills), bound by the dependence of each
// transform's passes on each other and two barriers a row.  The lane exchanges
// as register swaps and DPP moves against all through LDS: 25.6 / 27.5 at 4096,
// 6.9 / 7.2 at 1024, 6.5 / 6.3 at 600.
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(3, 3))) void k_blind_rotate1w2_pair(
    const uint32_t *__restrict__ in, int n0, const cd *__restrict__ bk,
    const uint32_t *__restrict__ tv, int tv_stride, uint32_t *__restrict__ out, int sample_extract,
    int B)
{
    __shared__ uint32_t acc[2][N1];
    __shared__ cd tiles[2][kLaneTile];
    const int tid = threadIdx.x, lane = tid & 63;
    const int half = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ct = blockIdx.x;
    if (ct >= B) return;
    const uint32_t *c0 = in + size_t(ct) * (n0 + 1);
    const uint32_t *tvp = tv + size_t(ct) * tv_stride;
    const TwW tw = make_tww(lane, half);
    const int nb = lane + 64 * half;
    cd *own = tiles[half], *theirs = tiles[half ^ 1];

    // acc = (0, X^bbar tv), bbar = 2N - (b >> 21)   (no rounding)
    {
        const uint32_t bbar = 2u * N1 - (c0[n0] >> (32 - 1 - Lvl1::nbit));
#pragma unroll
        for (int k = 0; k < N1 / 128; k++) {
            const int n = tid + 128 * k;
            const uint32_t idx = (uint32_t(n) - bbar) & (2u * N1 - 1);
            const uint32_t v = tvp[idx & (N1 - 1)];
            acc[0][n] = 0;
            acc[1][n] = (idx & N1) ? 0u - v : v;
        }
    }
    __syncthreads();

    constexpr uint32_t kRound = 1u << (32 - 2 - Lvl1::nbit);
    for (int i = 0; i < n0; i++) {
        const uint32_t abar = (c0[i] + kRound) >> (32 - 1 - Lvl1::nbit);
        if (abar == 0) continue;
        const cd *bki = bk + size_t(i) * (Lvl1::rows * 2 * kPolyW) + half * 256 + lane;
        cd fd[2][4];
#pragma unroll
        for (int q = 0; q < 4; q++) fd[0][q] = fd[1][q] = cd{0.0, 0.0};
#pragma unroll 1
        for (int c = 0; c < 2; c++) {
            uint32_t u[8];
#pragma unroll
            for (int k = 0; k < 8; k++) u[k] = prep_rot(acc[c], abar, nb + 128 * (k >> 1) + 512 * (k & 1));
#pragma unroll 1
            for (int d = 0; d < Lvl1::l; d++) {
                // key words requested before the transform
                const cd *k0 = bki + (c * Lvl1::l + d) * 2 * kPolyW;
                cd b0[4], b1[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    b0[q] = k0[q * 64];
                    b1[q] = k0[kPolyW + q * 64];
                }
                cd v[4];
#pragma unroll
                for (int p = 0; p < 4; p++) v[p] = cd{digit_w(u[2 * p], d), digit_w(u[2 * p + 1], d)};
                fft512w_fwd_a(v, tw);
                __syncthreads();  // the other wave has left its tile
                put_seqs(v, theirs, lane, half);
                __syncthreads();
                fft512w_fwd_c(v, own, lane, half, tw);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    cmac(fd[0][q], v[q], b0[q]);
                    cmac(fd[1][q], v[q], b1[q]);
                }
            }
        }
        // both waves' rotation reads of acc are complete (the transforms
        // synchronised them); each wave updates only its own coefficients
#pragma unroll
        for (int c = 0; c < 2; c++) {
            fft512w_inv_a(fd[c], own, lane, half, tw);
            __syncthreads();
            fft512w_inv_c(fd[c], theirs, lane, half, tw);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const cd z = fd[c][k >> 1];
                acc[c][nb + 128 * (k >> 1) + 512 * (k & 1)] += trunc_torus32(k & 1 ? z.y : z.x);
            }
            // the exchange words are read, and after column 1 the accumulator
            // is whole
            __syncthreads();
        }
    }

    if (sample_extract) {
        // SampleExtractIndex 0: out[0] = acc0[0], out[n] = -acc0[N - n], out[N] = acc1[0]
        uint32_t *o = out + size_t(ct) * (N1 + 1);
        for (int n = tid; n < N1; n += 128) o[n] = n == 0 ? acc[0][0] : 0u - acc[0][N1 - n];
        if (tid == 0) o[N1] = acc[1][0];
    } else {
        uint32_t *o = out + size_t(ct) * 2 * N1;
        for (int n = tid; n < N1; n += 128) {
            o[n] = acc[0][n];
            o[N1 + n] = acc[1][n];
        }
    }
}

// one-wave device key -> the order of both kernels: slice element (w, q, l) holds
// frequency f = f1w(w, l, q), which the one-wave layout keeps at register
// f >> 6 of lane ((f & 7) << 3) | ((f >> 3) & 7)
__global__ __launch_bounds__(256) void k_bk1_to_w2(const cd *__restrict__ src, cd *__restrict__ dst,
                                                  size_t nslices)
{
    const size_t e = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (e >= nslices * kPolyW) return;
    const size_t slice = e / kPolyW;
    const int k = int(e % kPolyW);
    const int w = k >> 8, q = (k >> 6) & 3, l = k & 63;
    const int f = f1w(w, l, q);
    const int s = ((f & 7) << 3) | ((f >> 3) & 7);
    dst[e] = src[slice * kPolyW + (f >> 6) * 64 + s];
}

}  // namespace

hipError_t launch_bk1_to_w2(const cd *bk1, cd *bk_w2, int n0, hipStream_t s)
{
    const size_t nslices = size_t(n0) * Lvl1::rows * 2;
    const size_t n = nslices * kPolyW;
    hipLaunchKernelGGL(k_bk1_to_w2, dim3(unsigned((n + 255) / 256)), dim3(256), 0, s, bk1, bk_w2,
                       nslices);
    return hipGetLastError();
}

// k_blind_rotate1w2 up to two ciphertexts per compute unit, one after the other
// (its third round makes it the slower one, figures at k_blind_rotate1w2_pair);
// reached above kPbs1TwoWaveBelow only where a tuned table asks for two waves
constexpr int kRoundsW2 = 2 * 256;

hipError_t launch_blind_rotate1w2(const uint32_t *in, int n0, const cd *bk, const uint32_t *tv,
                                  int tv_stride, uint32_t *out, bool sample_extract, int B,
                                  hipStream_t s, bool shared)
{
    if (B <= 0) return hipSuccess;
    if (shared || B > kRoundsW2)
        hipLaunchKernelGGL(k_blind_rotate1w2_pair, dim3(B), dim3(128), 0, s, in, n0, bk, tv,
                           tv_stride, out, int(sample_extract), B);
    else
        hipLaunchKernelGGL(k_blind_rotate1w2, dim3(B), dim3(64 * kWaves), 0, s, in, n0, bk, tv,
                           tv_stride, out, int(sample_extract), B);
    return hipGetLastError();
}

}  // namespace fhe
