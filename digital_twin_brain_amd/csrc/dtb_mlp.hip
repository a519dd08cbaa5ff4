// dtb_mlp.hip -- kernels of the learned surrogate: a bf16 MFMA GEMM with
// FP32 accumulation and fused bias + activation, and the small elementwise
// kernels of MLP training (ReLU backward, bias gradient, MSE gradient, Adam).
//
// GEMM form "NT": C[M,N] = act(A[M,K] * B[N,K]^T + bias[N]); both operands are
// K-contiguous row-major bf16, so a forward layer is (X, W^T) and the two
// backward products use transposed copies made by dtb_mlp_transpose_bf16.
// A workgroup of four wavefronts computes a tile of C with
// v_mfma_f32_32x32x16_bf16 over K in steps of 16.
//
// MFMA operand layout (32x32x16 bf16): lane l holds 8 consecutive K values
// k = 8*(l/32) .. +7 of row (l % 32) for A and of column (l % 32) for B; the
// 16 accumulator registers hold C[8*(r/4) + 4*(l/32) + r%4][l % 32].
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "dtb_internal.hpp"

namespace dtb {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ inline uint16_t f2bf(float f)
{
    // round to nearest even
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40); // NaN stays NaN
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// two at a time with v_cvt_pk_bf16_f32: the same rounding (and quieting) as f2bf
__device__ inline uint32_t f2bf_pk(float lo, float hi)
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 h = {(__bf16)lo, (__bf16)hi};
    uint32_t u;
    __builtin_memcpy(&u, &h, 4);
    return u;
}

__device__ inline float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// act: 0 identity, 1 ReLU

// Products of one chain over K (gemm_one_chain): LDS-staged tiles filled by
// direct global-to-LDS loads.  A workgroup of four wavefronts (2 x 2), one on
// each SIMD of its CU, computes a (64 TM) x (64 TN) tile of C, each wavefront
// TM x TN sub-tiles of 32x32.  The bound is the matrix pipe, and next to it
// the LDS ports: with 128x128 per wavefront (TM = TN = 4) a 16-wide K step
// reads 8 KB of fragments for 16 MFMAs, half the port rate (64x128 per
// wavefront, as eight wavefronts had it, saturated the ports, and the copies
// through registers came on top).
// K advances 64 at a time.  A and B slices go through a ring of five LDS
// slots (two and a half slices: all 160 KB with TM = TN = 4), and the loop is
// pipelined so that neither a fragment read, nor the barrier, nor the latency
// of a slice leaves the matrix pipe idle:
//   K step s of a slice multiplies fragments read during step s - 1;
//   at the last step of slice t the wavefronts meet (slice t + 1 has landed,
//   nobody reads slice t any more) and read slice t + 1's first fragments;
//   from there to the next meeting they request, spread over the MFMAs, B of
//   slice t + 2 into A(t)'s slot, then A of slice t + 3 into B(t)'s.  (All at
//   once the requests queue up: 64 of 16 cycles each at the load unit of the
//   CU.)  B has most of a slice's time to arrive, A most of two.
// A slot row is 64 bf16 = 8 chunks of 16 bytes; the load unit writes 64
// lanes' chunks back to back, so the lanes permute what they fetch: chunk c
// of row r sits at position c ^ (r / 2 % 8), and the 16 rows that a quarter of
// a fragment read touches fall on distinct banks without padding.
// M and N are multiples of 32, K of 16: rows past the edge are clamped (and
// not stored), a last slice shorter than 64 fetches clamped chunks that no
// step multiplies.  Workgroups are dealt to tiles XCD by XCD (workgroup w
// runs on XCD w mod 8): each XCD takes a contiguous run of tiles, ordered in
// bands of GM tile rows, column by column, so that the tiles it has in flight
// form a near-square block and share their slices in its L2.
// 8192^3: 1110 -> 830 us a call (1.32 PFLOP/s; matrix pipe busy 74% of the cycles, no
// LDS bank conflicts); 960 x 960 x 6144: 112 -> 39 us; 992 x 4160 x 3008 (no
// multiples of 128): 181 -> 44 us.
__device__ __forceinline__ void lds_dma16(const uint16_t* src, uint32_t lds_byte)
{
    // the wavefront's 64 chunks of 16 bytes, to consecutive LDS addresses from lds_byte (M0);
    // counted by vmcnt, for which the caller waits
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_byte), "v"(src)
                 : "memory", "m0");
}

// N of this wavefront's loads may still be under way, its LDS reads are done; then all wavefronts meet
template <int N>
__device__ __forceinline__ void lds_dma_meet()
{
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// RANGES: each wavefront's sums are those of four consecutive ranges of K added
// in order, as gemm_nt_splitk_kernel adds them, instead of one chain.
template <int T, int GM, bool RANGES>
__global__ __launch_bounds__(256, T == 4 ? 1 : T == 2 ? 2 : 4) void gemm_nt_tile_kernel(
    int32_t M, int32_t N, int32_t K, const uint16_t* __restrict__ A, int64_t lda, const uint16_t* __restrict__ B,
    int64_t ldb, const float* __restrict__ bias, int32_t act, float* __restrict__ C, int64_t ldc,
    uint16_t* __restrict__ Cb, int64_t ldcb)
{
    constexpr int TM = T, TN = T;
    constexpr int kSlot = 64 * T * 64; // elements: 64 T rows of A or B
    extern __shared__ __align__(128) uint16_t lds[]; // [5][kSlot]
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int wm = wid >> 1, wn = wid & 1;
    // this workgroup's tile
    const int tm = (M + 64 * TM - 1) / (64 * TM), tn = (N + 64 * TN - 1) / (64 * TN);
    const int tiles = tm * tn;
    const int per = (tiles + 7) / 8;
    const int tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= per || tile >= tiles) return; // workgroup-uniform
    const int band = tile / (GM * tn);
    const int rows = min(GM, tm - band * GM);
    const int in = tile - band * GM * tn;
    const int m_blk = (band * GM + in % rows) * (64 * TM), n_blk = in / rows * (64 * TN);
    // what this wavefront fetches of a slice: 2 TM groups of 8 rows of A, 2 TN of B
    constexpr int kFetch = 2 * (TM + TN);
    // columns of this lane's chunk in the slice, in even and odd groups of 8 rows
    const int ch[2] = {((lane & 7) ^ (lane >> 4)) * 8, ((lane & 7) ^ (4 + (lane >> 4))) * 8};
    const uint16_t* src[kFetch];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)lds;
#pragma unroll
    for (int u = 0; u < kFetch; ++u) {
        if (u < 2 * TM) src[u] = A + (int64_t)min(m_blk + (wid * 2 * TM + u) * 8 + (lane >> 3), M - 1) * lda;
        else src[u] = B + (int64_t)min(n_blk + (wid * 2 * TN + u - 2 * TM) * 8 + (lane >> 3), N - 1) * ldb;
    }
    auto fetch = [&](int u, int kt, int slot) { // group u of K slice kt to a slot of the ring
        const int row0 = (wid * 2 * T + u % (2 * T)) * 8;
        lds_dma16(src[u] + min(kt * 64 + ch[u & 1], K - 8), lds0 + (uint32_t)(slot * kSlot + row0 * 64) * 2u);
    };
    const int r = lane & 31, kh = lane >> 5;
    int oa[4], ob[4]; // element offset of this lane's fragments in a slot, by K step
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int slot = ((2 * s + kh) ^ ((r >> 1) & 7)) * 8;
        oa[s] = (wm * 32 * TM + r) * 64 + slot;
        ob[s] = (wn * 32 * TN + r) * 64 + slot;
    }
    bf16x8 fr[2][TM + TN];
    int sa = 0, sb = 1; // the slots of the current slice: 2 t mod 5 and 2 t + 1 mod 5
    auto next = [](int slot) { return slot < 3 ? slot + 2 : slot - 3; };
    auto read = [&](int f, int x, int a, int b, int s) { // fragment x of K step s of the slice in slots a, b
        fr[f][x] = *reinterpret_cast<const bf16x8*>(x < TM ? lds + a * kSlot + oa[s] + x * 32 * 64
                                                           : lds + b * kSlot + ob[s] + (x - TM) * 32 * 64);
    };
    f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int x = 0; x < 16; ++x) acc[i][j][x] = 0.0f;
    const int nk = (K + 63) / 64;
    constexpr int kHalf = kFetch / 2;        // this wavefront's loads of one operand's slice
    constexpr int kFirst = (3 * kHalf + 3) / 4; // of them, those of B requested right after a meeting
#pragma unroll
    for (int u = 0; u < kFetch; ++u) fetch(u, 0, u / kHalf);
    if (nk > 1) {
#pragma unroll
        for (int u = 0; u < kHalf + kFirst; ++u) fetch(u, 1, 2 + u / kHalf);
        lds_dma_meet<kHalf + kFirst>(); // slice 0 has landed
    } else {
        lds_dma_meet<0>();
    }
#pragma unroll
    for (int x = 0; x < TM + TN; ++x) read(0, x, 0, 1, 0);
    // one K step's MFMAs from fr[f]; after the i-th, side(i) issues what overlaps it
    auto multiply = [&](int f, auto&& side) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[f][i], fr[f][TM + j], acc[i][j], 0, 0, 0);
                side(i * TN + j);
                __builtin_amdgcn_sched_barrier(0);
            }
    };
    constexpr int kProd = TM * TN;
    // RANGES: the sum of the finished ranges, and the K steps left in the current one
    f32x16 tot[RANGES ? TM : 1][RANGES ? TN : 1];
    const int range_steps = RANGES ? (K / 16 + 3) / 4 : 0;
    int range = 0, to_fold = range_steps;
    auto step_done = [&]() {
        if constexpr (RANGES) {
            if (--to_fold == 0) {
                to_fold = range_steps;
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int x = 0; x < 16; ++x) {
                            tot[i][j][x] = range == 0 ? acc[i][j][x] : tot[i][j][x] + acc[i][j][x];
                            acc[i][j][x] = 0.0f;
                        }
                ++range;
            }
        }
    };
    // a slice that one other (more: several others) follows
    auto slice = [&](int kt, auto more_) {
        constexpr bool more = decltype(more_)::value;
        constexpr int kRest = kFetch - kFirst; // requests in steps 0 to 2
        const int na = next(sa), nb = next(sb);
#pragma unroll
        for (int s = 0; s < 3; ++s) {
            multiply(s & 1, [&](int i) {
                // the next step's fragments, two after each MFMA while they last
#pragma unroll
                for (int x = 0; x < TM + TN; ++x)
                    if (x / 2 == i || (i == kProd - 1 && x / 2 > i)) read((s + 1) & 1, x, sa, sb, s + 1);
#pragma unroll
                for (int y = 0; y < kRest; ++y)
                    if (y * 3 * kProd / kRest == s * kProd + i) {
                        if (y < kHalf - kFirst) fetch(kHalf + kFirst + y, kt + 1, nb);
                        else if (more) fetch(y - (kHalf - kFirst), kt + 2, next(na));
                    }
            });
            step_done();
        }
        // slice kt + 1 has landed (A of slice kt + 2 may be under way), and
        // this wavefront's last fragments of slice kt are in registers
        lds_dma_meet<more ? kHalf : 0>();
        multiply(1, [&](int i) {
#pragma unroll
            for (int x = 0; x < TM + TN; ++x)
                if (x / 2 == i || (i == kProd - 1 && x / 2 > i)) read(0, x, na, nb, 0);
#pragma unroll
            for (int u = 0; u < kFirst; ++u)
                if (more && u * kProd / kFirst == i) fetch(kHalf + u, kt + 2, sa);
        });
        step_done();
        sa = na;
        sb = nb;
    };
    int kt = 0;
    for (; kt + 2 < nk; ++kt) slice(kt, std::true_type{});
    if (kt + 1 < nk) slice(kt++, std::false_type{});
    // the last slice, of one to four steps
    for (int s = 0; 64 * kt + 16 * s < K; ++s) {
        const int slot = ((2 * s + kh) ^ ((r >> 1) & 7)) * 8 + r * 64;
#pragma unroll
        for (int x = 0; x < TM + TN; ++x)
            fr[0][x] = *reinterpret_cast<const bf16x8*>(x < TM ? lds + sa * kSlot + slot + (wm * TM + x) * 32 * 64
                                                               : lds + sb * kSlot + slot + (wn * TN + x - TM) * 32 * 64);
        multiply(0, [](int) {});
        step_done();
    }
    if constexpr (RANGES) {
        // a range that K's steps do not fill, or the empty ones after it (adding zeros as they would)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int x = 0; x < 16; ++x)
                    acc[i][j][x] = range == 0 ? acc[i][j][x] : range < 4 ? tot[i][j][x] + acc[i][j][x] : tot[i][j][x];
    }
    const int m0 = m_blk + wm * 32 * TM, n0 = n_blk + wn * 32 * TN;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        if (n0 + 32 * j >= N) continue;
        const int col = n0 + 32 * j + r;
        const float bv = bias ? bias[col] : 0.0f;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            if (m0 + 32 * i >= M) continue;
            // one running pointer an output (addresses kept for all stores would spill)
            const int64_t row = m0 + 32 * i + 4 * kh;
            float* c = C + row * ldc + col;
            uint16_t* cb = Cb + row * ldcb + col;
#pragma unroll
            for (int x = 0; x < 16; ++x) {
                float v = acc[i][j][x] + bv;
                if (act == 1) v = v > 0.0f ? v : 0.0f;
                if (C) *c = v;
                if (Cb) *cb = f2bf(v);
                c += (x & 3) == 3 ? 5 * ldc : ldc; // rows 0..3, 8..11, 16..19, 24..27
                cb += (x & 3) == 3 ? 5 * ldcb : ldcb;
                asm volatile("" : "+v"(c), "+v"(cb));
            }
        }
    }
}

// Small products (too few 64x64 tiles to fill the chip): a workgroup computes
// one 32x32 tile of C and its four wavefronts split K in four consecutive
// ranges; wavefronts 1-3 hand their partial sums to wavefront 0 through LDS,
// which adds them in wavefront order (a fixed order: results do not depend on
// timing).  Each wavefront's serial chain of K steps is a quarter as long.
__global__ __launch_bounds__(256) void gemm_nt_splitk_kernel(int32_t M, int32_t N, int32_t K,
                                                             const uint16_t* __restrict__ A, int64_t lda,
                                                             const uint16_t* __restrict__ B, int64_t ldb,
                                                             const float* __restrict__ bias, int32_t act,
                                                             float* __restrict__ C, int64_t ldc,
                                                             uint16_t* __restrict__ Cb, int64_t ldcb)
{
    __shared__ float red[3][16][64];
    const int wid = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int m0 = blockIdx.y * 32;
    const int n0 = blockIdx.x * 32;
    const int r = lane & 31;
    const int kh = (lane >> 5) * 8;
    const int steps = K / 16;
    const int per = (steps + 3) / 4;
    const int kb = min(wid * per, steps) * 16;
    const int ke = min((wid + 1) * per, steps) * 16;
    const uint16_t* pa = A + (int64_t)(m0 + r) * lda + kh;
    const uint16_t* pb = B + (int64_t)(n0 + r) * ldb + kh;
    f32x16 acc;
#pragma unroll
    for (int x = 0; x < 16; ++x) acc[x] = 0.0f;
    for (int k0 = kb; k0 < ke; k0 += 16) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(pa + k0);
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(pb + k0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    }
    if (wid > 0) {
#pragma unroll
        for (int x = 0; x < 16; ++x) red[wid - 1][x][lane] = acc[x];
    }
    __syncthreads();
    if (wid != 0) return;
#pragma unroll
    for (int w = 0; w < 3; ++w)
#pragma unroll
        for (int x = 0; x < 16; ++x) acc[x] += red[w][x][lane];
    const int col = n0 + r;
    const float bv = bias ? bias[col] : 0.0f;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
        const int row = m0 + 8 * (x >> 2) + 4 * (lane >> 5) + (x & 3);
        float v = acc[x] + bv;
        if (act == 1) v = v > 0.0f ? v : 0.0f;
        if (C) C[(int64_t)row * ldc + col] = v;
        if (Cb) Cb[(int64_t)row * ldcb + col] = f2bf(v);
    }
}

// dZ = dY * relu'(Z)  (Z > 0), written in FP32 and bf16
__global__ void relu_backward_kernel(int64_t n, const float* __restrict__ dY, const float* __restrict__ Z,
                                     float* __restrict__ dZ, uint16_t* __restrict__ dZb)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float v = Z[i] > 0.0f ? dY[i] : 0.0f;
    if (dZ) dZ[i] = v;
    if (dZb) dZb[i] = f2bf(v);
}

// db[j] = sum_i dZ[i][j], added in row order (a bias one rounding away from
// another one's changes which way a GRU's states round, and so every gradient
// after the next update).  One thread walking a column waits for its loads, 465
// us for 2,048 rows; here a workgroup stages kBiasRows rows x 64 columns in
// LDS at a time, all 1024 threads' loads of the next rows in flight while the
// first wavefront adds the staged ones (a lane per column).  The adds, a
// dependent chain, are then what is left: 21 us for 2,048 x 1,056.
constexpr int kBiasCols = 64, kBiasRows = 256, kBiasThreads = 1024;
constexpr int kBiasLoads = kBiasRows * kBiasCols / kBiasThreads;

__device__ __forceinline__ void column_sums(int64_t M, int32_t N, const float* __restrict__ src, int64_t ld, int j0,
                                            float* lds, float* __restrict__ dst, float* __restrict__ dst2)
{
    const int c = threadIdx.x % kBiasCols, r0 = threadIdx.x / kBiasCols;
    const int j = j0 + c;
    float v[kBiasLoads];
    auto load = [&](int64_t i0) {
#pragma unroll
        for (int u = 0; u < kBiasLoads; ++u) {
            const int64_t i = i0 + r0 + u * (kBiasThreads / kBiasCols);
            v[u] = i < M && j < N ? src[i * ld + j] : 0.0f;
        }
    };
    float s = 0.0f;
    load(0);
    for (int64_t i0 = 0; i0 < M; i0 += kBiasRows) {
#pragma unroll
        for (int u = 0; u < kBiasLoads; ++u) lds[(r0 + u * (kBiasThreads / kBiasCols)) * kBiasCols + c] = v[u];
        __syncthreads();
        if (i0 + kBiasRows < M) load(i0 + kBiasRows);
        if (threadIdx.x < kBiasCols) {
            const int n = (int)(M - i0 < kBiasRows ? M - i0 : kBiasRows);
            // the next 16 rows are read while the 16 before are added
            float x[2][16];
            auto read = [&](float (&d)[16], int i) {
#pragma unroll
                for (int u = 0; u < 16; ++u) d[u] = lds[(i + u) * kBiasCols + c];
            };
            read(x[0], 0);
#pragma unroll
            for (int q = 0; q < kBiasRows / 16; ++q) {
                if (q + 1 < kBiasRows / 16) read(x[(q + 1) & 1], 16 * (q + 1));
                if (16 * q + 16 <= n) { // uniform
#pragma unroll
                    for (int u = 0; u < 16; ++u) s += x[q & 1][u];
                } else {
#pragma unroll
                    for (int u = 0; u < 16; ++u)
                        if (16 * q + u < n) s += x[q & 1][u];
                }
            }
        }
        __syncthreads();
    }
    if (threadIdx.x < kBiasCols && j < N) {
        dst[j] = s;
        if (dst2) dst2[j] = s;
    }
}

__global__ __launch_bounds__(kBiasThreads) void bias_grad_kernel(int32_t M, int32_t N, const float* __restrict__ dZ,
                                                                 float* __restrict__ db)
{
    __shared__ float lds[kBiasRows * kBiasCols];
    column_sums(M, N, dZ, N, blockIdx.x * kBiasCols, lds, db, nullptr);
}

// grad = scale * (out - target) masked; loss partial sums in lsum[blockIdx]
__global__ void mse_grad_kernel(int64_t n, const float* __restrict__ out, const float* __restrict__ target,
                                const float* __restrict__ mask, float scale, float* __restrict__ grad,
                                uint16_t* __restrict__ gradb, float* __restrict__ lsum)
{
    __shared__ float red[256];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float e = 0.0f;
    if (i < n) {
        const float mk = mask ? mask[i] : 1.0f;
        const float d = (out[i] - target[i]) * mk;
        e = d * d;
        const float g = scale * d;
        if (grad) grad[i] = g;
        if (gradb) gradb[i] = f2bf(g);
    }
    red[threadIdx.x] = e;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0 && lsum) lsum[blockIdx.x] = red[0];
}

// Adam (Kingma & Ba, 2015) on FP32 master weights, refreshing the bf16 copy
__device__ __forceinline__ float adam_update(float w, float gi, float& m, float& v, float lr, float b1, float b2,
                                             float eps, float c1, float c2)
{
    const float mi = b1 * m + (1.0f - b1) * gi;
    const float vi = b2 * v + (1.0f - b2) * gi * gi;
    m = mi;
    v = vi;
    return w - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

__global__ void adam_kernel(int64_t n, float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                            float* __restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2,
                            uint16_t* __restrict__ wb)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float mi = m[i], vi = v[i];
    const float wi = adam_update(w[i], g[i], mi, vi, lr, b1, b2, eps, c1, c2);
    m[i] = mi;
    v[i] = vi;
    w[i] = wi;
    if (wb) wb[i] = f2bf(wi);
}

__global__ void transpose_bf16_kernel(int32_t M, int32_t N, const uint16_t* __restrict__ in, uint16_t* __restrict__ out)
{
    __shared__ uint16_t tile[32][33];
    const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5; // 256 threads: 32 x 8
    for (int y = ty; y < 32; y += 8) {
        const int r = by + y, c = bx + tx;
        if (r < M && c < N) tile[y][tx] = in[(int64_t)r * N + c];
    }
    __syncthreads();
    for (int y = ty; y < 32; y += 8) {
        const int r = bx + y, c = by + tx; // out is [N][M]
        if (r < N && c < M) out[(int64_t)r * M + c] = tile[tx][y];
    }
}

__global__ void f32_to_bf16_kernel(int64_t n, const float* __restrict__ in, uint16_t* __restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = f2bf(in[i]);
}

// out[r][c] = in[r][c] * scale[c] + shift[c] for c < cin, 0 for cin <= c < cout
__global__ void affine_kernel(int32_t rows, int32_t cin, int32_t cout, const float* __restrict__ in, int64_t ldi,
                              const float* __restrict__ scale, const float* __restrict__ shift,
                              float* __restrict__ out, uint16_t* __restrict__ outb, int64_t ldo)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)rows * cout) return;
    const int32_t r = (int32_t)(i / cout), c = (int32_t)(i % cout);
    float v = 0.0f;
    if (c < cin) v = in[(int64_t)r * ldi + c] * (scale ? scale[c] : 1.0f) + (shift ? shift[c] : 0.0f);
    if (out) out[(int64_t)r * ldo + c] = v;
    if (outb) outb[(int64_t)r * ldo + c] = f2bf(v);
}

// ------------------------------------------------ whole-network MLP kernels
// A surrogate's layers are small (512 x 512 weights, at most 2,048 rows a
// batch), so a product per launch leaves the device idle between launches:
// a training step was 43 launches, a 23,040-row prediction 72.  Rows never
// mix inside the forward pass or in the chain of activation gradients, so one
// workgroup takes 32 rows through every layer, with the activations in LDS:
//   mlp_chain_kernel<false, RT>  normalise, all layers, denormalise (RT x 32 rows)
//   mlp_chain_kernel<true, 1>  normalise, all layers, loss, and the gradients of
//                            every layer's output down to the first; writes the
//                            transposed bf16 operands of the weight gradients
//                            and each 32-row tile's column sums of the gradients
//   mlp_dw_kernel            the weight gradients of all layers (contraction
//                            over the batch) and the bias gradients
//   adam_multi_kernel        Adam on every parameter, with the bf16 copy and
//                            its transpose
// Bound of the chain: each workgroup reads every weight once from its XCD's L2.
// A CU takes about 110 B/ns that way (one workgroup or 256 streaming at once),
// 4.7 us for the 512 KB of a 512 x 512 layer, against 1.7 us of matrix work for
// 32 rows; with the rounding to bf16 and the stores a layer takes 5.5 us.
// Measured (18 -> 512 x 3 -> 6): a training step of 2,048 rows 210 -> 67 us
// (chain 45, weight gradients 14, Adam 6.7), 23,040 predicted rows 465 -> 47 us.
//
// Every bf16 operand that these kernels read from memory is kept in fragment
// order: for each 32 rows and 16 columns of a matrix [N][K] the 1 KB that one
// v_mfma_f32_32x32x16_bf16 takes, lane by lane (frag_at).  A wavefront's load
// is then 8 whole cache lines; from row-major weights it touched 32 lines for
// 32 bytes each, and the first form of the chain took 91 us instead of 53 for a
// 2,048-row batch and 130 instead of 74 for a 23,040-row prediction
// (18 -> 512 x 3 -> 6).
//
// Each product is summed as dtb_mlp_gemm_bf16_nt sums it -- one chain over K
// where the batch's product has at least 256 64x64 tiles, else four
// consecutive ranges of K added in order -- so results equal the
// layer-by-layer launches bit for bit.
constexpr int kMlpMaxLayers = 8;
constexpr int kMlpRows = 32;    // rows of a chain workgroup
constexpr int kMlpWaves = 8;    // two 32-column tiles each of a 512-wide layer
constexpr int kMlpThreads = 64 * kMlpWaves;

// one chain over K (else four ranges), by the tile count of the whole product
__host__ __device__ inline bool gemm_one_chain(int32_t M, int32_t N)
{
    return (int64_t)((N + 63) / 64) * ((M + 63) / 64) >= 256;
}

// where element (n, k) of a matrix [N][K] in fragment order is
__host__ __device__ inline int64_t frag_at(int64_t K, int64_t n, int64_t k)
{
    return (n / 32 * (K / 16) + k / 16) * 512 + (k % 16 / 8 * 32 + n % 32) * 8 + k % 8;
}

// All bf16 arrays in fragment order.
struct MlpLayerDev {
    int32_t in, out;       // padded widths (multiples of 32)
    const uint16_t* w;     // weights [out][in]
    const uint16_t* wt;    // weights [in][out] (training)
    const float* bias;     // [out]
    uint16_t* hT;          // input of the layer [in][B] (training)
    uint16_t* gT;          // gradient of the layer's output [out][B] (training)
    float* dbp;            // [B / 32][out] column sums of that gradient per row tile (training)
};

struct MlpChainArgs {
    int32_t rows, layers, cin, cout, max_batch, bufw;
    const float* X;
    int64_t ldx;
    const float *xs, *xh;  // input scale and shift
    const float *ys, *yh;  // prediction: output scale and shift; training: target scale and shift
    float* out;            // prediction [rows][cout]; training: raw network output [B][last width]
    int64_t ldo;
    const float* Y;        // targets [rows][cout] (training)
    int64_t ldy;
    const float* mask;     // [rows][cout] or NULL (training)
    int64_t ldm;
    float scale;
    float* lsum;
    MlpLayerDev l[kMlpMaxLayers];
};

// tot[i][j] = A[32 i ..][K] W[tile + j][K]^T over steps s0 .. s1 of 16 of this
// wavefront; A in LDS, W (fragment order, `steps` steps a tile) streamed from
// L2: blocks of four steps (4 KB a tile), two blocks ahead of their use (one
// where a block feeds two row tiles), in register buffers taken in turn.  Loads
// past the end repeat the last block, so that no load sits behind a branch.
// per > 0: the running sum is folded into tot after every `per` steps, which
// splits K into consecutive ranges (FOLD 1: per is a multiple of the block, 2:
// any).
// SWAP: the operands change places, so a lane holds 16 columns of one row of
// the result (mfma_row gives the column) instead of 16 rows of one column.
template <int RT, int TN, int FOLD, bool SWAP>
__device__ __forceinline__ void chain_gemm(const uint16_t* sA, int lda, const uint16_t* __restrict__ W, int steps,
                                           int tile, int s0, int s1, int per, f32x16 (&tot)[RT][TN])
{
    const int lane = threadIdx.x & 63;
    const uint16_t* pa = sA + (lane & 31) * lda + (lane >> 5) * 8;
    const uint16_t* pb[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) pb[j] = W + (int64_t)(tile + j) * steps * 512 + lane * 8;
    f32x16 acc[RT][TN];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int x = 0; x < 16; ++x) {
                acc[i][j][x] = 0.0f;
                if (FOLD) tot[i][j][x] = -0.0f; // the additive identity: the first fold leaves its sum as it is
            }
    int left = per; // steps until the next fold
    auto fold = [&]() {
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int x = 0; x < 16; ++x) {
                    tot[i][j][x] += acc[i][j][x];
                    acc[i][j][x] = 0.0f;
                }
        left = per;
    };
    auto step = [&](int s, const bf16x8 (&b)[TN]) {
        if (FOLD == 2 && left == 0) fold();
        --left;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
            const bf16x8 av = *reinterpret_cast<const bf16x8*>(pa + 32 * i * lda + 16 * s);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = SWAP ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[j], av, acc[i][j], 0, 0, 0)
                                 : __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, b[j], acc[i][j], 0, 0, 0);
        }
    };
    const int nb = (s1 - s0) >> 2; // whole blocks
    if (nb > 0) {
        constexpr int D = RT == 1 ? 3 : 2; // register buffers
        bf16x8 buf[D][4][TN];
        auto load = [&](bf16x8 (&d)[4][TN], int blk) {
            const int s = s0 + 4 * min(blk, nb - 1);
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int j = 0; j < TN; ++j) d[u][j] = *reinterpret_cast<const bf16x8*>(pb[j] + (s + u) * 512);
        };
#pragma unroll
        for (int q = 0; q + 1 < D; ++q) load(buf[q], q);
        for (int blk = 0; blk < nb; blk += D) {
#pragma unroll
            for (int q = 0; q < D; ++q) {
                if (blk + q >= nb) break; // uniform
                load(buf[(q + D - 1) % D], blk + q + D - 1);
                if (FOLD == 1 && left <= 0) fold();
#pragma unroll
                for (int u = 0; u < 4; ++u) step(s0 + 4 * (blk + q) + u, buf[q][u]);
            }
        }
    }
    for (int s = s0 + 4 * nb; s < s1; ++s) {
        bf16x8 b[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = *reinterpret_cast<const bf16x8*>(pb[j] + s * 512);
        if (FOLD == 1 && left <= 0) fold();
        step(s, b);
    }
    if (FOLD) fold();
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
            if (!FOLD) tot[i][j] = acc[i][j];
}

// A split K takes the row tiles one after the other (its second accumulator
// would not leave registers for two), reading the weights again.
template <int RT, int TN, bool SWAP, typename F>
__device__ __forceinline__ void chain_tiles(const uint16_t* sA, int lda, const uint16_t* __restrict__ W, int steps,
                                            int tile, int per, F epi)
{
    if (per == 0) {
        f32x16 acc[RT][TN];
        chain_gemm<RT, TN, 0, SWAP>(sA, lda, W, steps, tile, 0, steps, 0, acc);
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) epi(i, tile + j, acc[i][j]);
        return;
    }
    for (int i = 0; i < RT; ++i) {
        f32x16 acc[1][TN];
        if (per % 4 == 0) chain_gemm<1, TN, 1, SWAP>(sA + 32 * i * lda, lda, W, steps, tile, 0, steps, per, acc);
        else chain_gemm<1, TN, 2, SWAP>(sA + 32 * i * lda, lda, W, steps, tile, 0, steps, per, acc);
#pragma unroll
        for (int j = 0; j < TN; ++j) epi(i, tile + j, acc[0][j]);
    }
}

// The product A[32 RT][K] W[N][K]^T of a workgroup: epi(row tile, tile, acc)
// for every 32-column tile, called by the wavefront that holds it: the
// neighbouring tiles 2 wid and 2 wid + 1 (which share their reads of A), then
// 16 further.  A single tile with split K spreads the four ranges over four
// wavefronts for each row tile (`red`: RT x 3 x 16 x 64 floats of LDS).
template <int RT, bool SWAP, typename F>
__device__ __forceinline__ void chain_layer(const uint16_t* sA, int lda, const uint16_t* __restrict__ W, int N, int K,
                                            bool one_chain, float* red, F epi)
{
    static_assert(RT <= kMlpWaves / 4, "one wavefront per row tile and range");
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int steps = K / 16;
    const int per = one_chain ? 0 : (steps + 3) / 4;
    if (N == 32 && !one_chain) {
        f32x16 acc[1][1];
#pragma unroll
        for (int x = 0; x < 16; ++x) acc[0][0][x] = 0.0f;
        const int rt = wid >> 2, q = wid & 3; // row tile, range
        if (rt < RT) {
            const int sb = min(q * per, steps), se = min((q + 1) * per, steps);
            if (sb < se) chain_gemm<1, 1, 0, SWAP>(sA + 32 * rt * lda, lda, W, steps, 0, sb, se, 0, acc);
            if (q > 0) {
#pragma unroll
                for (int x = 0; x < 16; ++x) red[((rt * 3 + q - 1) * 16 + x) * 64 + lane] = acc[0][0][x];
            }
        }
        __syncthreads();
        if (rt < RT && q == 0) {
#pragma unroll
            for (int w = 0; w < 3; ++w)
#pragma unroll
                for (int x = 0; x < 16; ++x) acc[0][0][x] += red[((rt * 3 + w) * 16 + x) * 64 + lane];
        }
        __syncthreads(); // red may be where epi writes
        if (rt < RT && q == 0) epi(rt, 0, acc[0][0]);
        return;
    }
    const int tiles = N / 32;
    for (int tile = 2 * wid; tile < tiles; tile += 2 * kMlpWaves) {
        if (tile + 1 < tiles) chain_tiles<RT, 2, SWAP>(sA, lda, W, steps, tile, per, epi);
        else chain_tiles<RT, 1, SWAP>(sA, lda, W, steps, tile, per, epi);
    }
}

// the 16 rows of a 32x32 tile that a lane's accumulator holds
__device__ inline int mfma_row(int x, int lane) { return 8 * (x >> 2) + 4 * (lane >> 5) + (x & 3); }

// a tile's values rounded to bf16 in row pairs (h), and into LDS [32][ld] at column c
__device__ inline void put_tile(const float (&v)[16], uint32_t (&h)[8], uint16_t* dst, int ld, int c, int lane)
{
#pragma unroll
    for (int x = 0; x < 8; ++x) h[x] = f2bf_pk(v[2 * x], v[2 * x + 1]);
    uint16_t* p = dst + 4 * (lane >> 5) * ld + c;
#pragma unroll
    for (int x = 0; x < 16; ++x) p[mfma_row(x, 0) * ld] = (uint16_t)(h[x >> 1] >> (16 * (x & 1)));
}

// store them (rows row0 .. row0 + 31 of column c) into [..][B] in fragment
// order, four rows (8 bytes) at a time: 2 KB of a tile contiguous
__device__ inline void store_transposed(uint16_t* __restrict__ T, int64_t B, int c, int row0, int lane,
                                        const uint32_t (&h)[8])
{
    uint16_t* p = T + frag_at(B, c, row0) + 4 * (lane >> 5);
#pragma unroll
    for (int q = 0; q < 4; ++q)
        *reinterpret_cast<uint2*>(p + (q >> 1) * 512 + (q & 1) * 256) = make_uint2(h[2 * q], h[2 * q + 1]);
}

template <bool TRAIN, int RT>
__global__ __launch_bounds__(kMlpThreads) void mlp_chain_kernel(MlpChainArgs a)
{
    constexpr int kRows = 32 * RT;
    extern __shared__ __align__(16) uint16_t smem[];
    const int t = threadIdx.x, lane = t & 63;
    // the last rows first: they may be a short batch whose products are split,
    // which takes longer
    const int row0 = (TRAIN ? blockIdx.x : gridDim.x - 1 - blockIdx.x) * kRows;
    // batch of max_batch rows this tile belongs to: its padded size decides how products are summed
    const int c0 = row0 / a.max_batch * a.max_batch;
    const int B = (min(a.max_batch, a.rows - c0) + 31) / 32 * 32;
    uint16_t* cur = smem;                       // activations or gradients [32 RT][bufw]
    uint16_t* nxt = smem + kRows * a.bufw;
    uint16_t* smask = smem + 2 * kRows * a.bufw; // [hidden tiles][64]: which of a lane's 16 outputs were > 0
    const int ld = a.bufw;
    const int I = a.l[0].in;
    for (int x = t; x < kRows * I; x += kMlpThreads) {
        const int r = x / I, c = x % I;
        float v = 0.0f;
        if (c < a.cin && row0 + r < a.rows)
            v = a.X[(int64_t)(row0 + r) * a.ldx + c] * (a.xs ? a.xs[c] : 1.0f) + (a.xh ? a.xh[c] : 0.0f);
        cur[r * ld + c] = f2bf(v);
    }
    __syncthreads();
    if (TRAIN) {
        for (int x = t; x < I * 8; x += kMlpThreads) { // eight groups of four rows per column
            const int c = x >> 3, q = (x & 7) * 4;
            *reinterpret_cast<ushort4*>(a.l[0].hT + frag_at(B, c, row0 + q)) =
                make_ushort4(cur[q * ld + c], cur[(q + 1) * ld + c], cur[(q + 2) * ld + c], cur[(q + 3) * ld + c]);
        }
    }
    int mbase = 0; // hidden tiles of the layers before
    for (int l = 0; l + 1 < a.layers; ++l) {
        const MlpLayerDev& L = a.l[l];
        uint16_t* hT = TRAIN ? a.l[l + 1].hT : nullptr;
        chain_layer<RT, !TRAIN>(
            cur, ld, L.w, L.out, L.in, gemm_one_chain(B, L.out), reinterpret_cast<float*>(nxt),
            [&](int rt, int tile, const f32x16& acc) {
                if (!TRAIN) { // a lane holds four runs of four columns of one row: 8-byte stores
                    const int c = tile * 32 + 4 * (lane >> 5);
                    uint16_t* p = nxt + (32 * rt + (lane & 31)) * ld + c;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float4 bv = *reinterpret_cast<const float4*>(L.bias + c + 8 * q);
                        float v[4] = {acc[4 * q] + bv.x, acc[4 * q + 1] + bv.y, acc[4 * q + 2] + bv.z,
                                      acc[4 * q + 3] + bv.w};
#pragma unroll
                        for (int x = 0; x < 4; ++x) v[x] = v[x] > 0.0f ? v[x] : 0.0f;
                        *reinterpret_cast<uint2*>(p + 8 * q) = make_uint2(f2bf_pk(v[0], v[1]), f2bf_pk(v[2], v[3]));
                    }
                    return;
                }
                const int c = tile * 32 + (lane & 31);
                const float bv = L.bias[c];
                float v[16];
                uint32_t m = 0;
#pragma unroll
                for (int x = 0; x < 16; ++x) {
                    v[x] = acc[x] + bv;
                    v[x] = v[x] > 0.0f ? v[x] : 0.0f;
                    if (v[x] > 0.0f) m |= 1u << x;
                }
                uint32_t h[8];
                put_tile(v, h, nxt, ld, c, lane);
                smask[(mbase + tile) * 64 + lane] = (uint16_t)m;
                store_transposed(hT, B, c, row0, lane, h);
            });
        __syncthreads();
        mbase += L.out / 32;
        uint16_t* sw = cur;
        cur = nxt;
        nxt = sw;
    }
    const MlpLayerDev& LL = a.l[a.layers - 1];
    if (!TRAIN) {
        chain_layer<RT, true>(cur, ld, LL.w, LL.out, LL.in, gemm_one_chain(B, LL.out), reinterpret_cast<float*>(nxt),
                              [&](int rt, int tile, const f32x16& acc) {
                                  const int row = row0 + 32 * rt + (lane & 31);
                                  if (row >= a.rows) return;
#pragma unroll
                                  for (int x = 0; x < 16; ++x) {
                                      const int c = tile * 32 + mfma_row(x, lane);
                                      if (c >= a.cout) continue;
                                      const float sc = a.ys ? a.ys[c] : 1.0f, sh = a.yh ? a.yh[c] : 0.0f;
                                      a.out[(int64_t)row * a.ldo + c] = (acc[x] + LL.bias[c]) * sc + sh;
                                  }
                              });
        return;
    }
    static_assert(!TRAIN || RT == 1, "the training kernel takes 32 rows");
    // output and its gradient
    const int no = LL.out;
    auto residual = [&](int row, int c, float o) { // mask * (out - target)
        float tgt = 0.0f, mk = 0.0f;
        if (c < a.cout && row < a.rows) {
            tgt = a.Y[(int64_t)row * a.ldy + c] * (a.ys ? a.ys[c] : 1.0f) + (a.yh ? a.yh[c] : 0.0f);
            mk = a.mask ? a.mask[(int64_t)row * a.ldm + c] : 1.0f;
        }
        return (o - tgt) * mk;
    };
    chain_layer<RT, false>(cur, ld, LL.w, no, LL.in, gemm_one_chain(B, no), reinterpret_cast<float*>(nxt),
                           [&](int, int tile, const f32x16& acc) {
                               const int c = tile * 32 + (lane & 31);
                               const float bv = LL.bias[c];
                               float g[16];
                               float colsum = 0.0f;
#pragma unroll
                               for (int x = 0; x < 16; ++x) {
                                   const int row = row0 + mfma_row(x, lane);
                                   const float o = acc[x] + bv;
                                   a.out[(int64_t)row * a.ldo + c] = o;
                                   g[x] = a.scale * residual(row, c, o);
                                   colsum += g[x];
                               }
                               uint32_t h[8];
                               put_tile(g, h, nxt, ld, c, lane);
                               store_transposed(LL.gT, B, c, row0, lane, h);
                               colsum += __shfl_xor(colsum, 32);
                               if (lane < 32) LL.dbp[(int64_t)blockIdx.x * no + c] = colsum;
                           });
    __syncthreads();
    // loss: squared errors in runs of 256 consecutive elements of [B][width]
    for (int k = t >> 6; k < no / 8; k += kMlpWaves) {
        float e = 0.0f;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int x = k * 256 + u * 64 + lane, row = row0 + x / no, c = x % no;
            const float d = residual(row, c, a.out[(int64_t)row * a.ldo + c]);
            e += d * d;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) e += __shfl_xor(e, off);
        if (lane == 0) a.lsum[(int64_t)blockIdx.x * (no / 8) + k] = e;
    }
    {
        uint16_t* sw = cur;
        cur = nxt;
        nxt = sw;
    }
    // the gradient of each hidden output, masked by its sign
    for (int l = a.layers - 1; l > 0; --l) {
        const MlpLayerDev& L = a.l[l];
        const MlpLayerDev& P = a.l[l - 1];
        mbase -= L.in / 32;
        chain_layer<RT, false>(cur, ld, L.wt, L.in, L.out, gemm_one_chain(B, L.in), reinterpret_cast<float*>(nxt),
                    [&](int rt, int tile, const f32x16& acc) {
                        const int c = tile * 32 + (lane & 31);
                        const uint32_t m = smask[(mbase + tile) * 64 + lane];
                        float g[16];
                        float colsum = 0.0f;
#pragma unroll
                        for (int x = 0; x < 16; ++x) {
                            g[x] = m >> x & 1u ? acc[x] + 0.0f : 0.0f;
                            colsum += g[x];
                        }
                        uint32_t h[8];
                        put_tile(g, h, nxt, ld, c, lane);
                        store_transposed(P.gT, B, c, row0, lane, h);
                        colsum += __shfl_xor(colsum, 32);
                        if (lane < 32) P.dbp[(int64_t)blockIdx.x * L.in + c] = colsum;
                    });
        __syncthreads();
        uint16_t* sw = cur;
        cur = nxt;
        nxt = sw;
    }
}

// Weight and bias gradients of every layer.  Workgroups [first[l], first[l+1])
// take layer l: a 64x64 tile of dW = G^T H each (both operands [width][B] in
// fragment order, K = B), K split in four ranges over the wavefronts and added in
// order (or walked as one chain by each wavefront for its own quarter of the
// tile, where dtb_mlp_gemm_bf16_nt would); the workgroups of the first tile
// column also add the row tiles' column sums into db.
struct MlpDwArgs {
    int32_t layers, B;     // B: rows (K of the products)
    int32_t first[kMlpMaxLayers + 1];
    int32_t in[kMlpMaxLayers], out[kMlpMaxLayers];
    int64_t ldh[kMlpMaxLayers], ldg[kMlpMaxLayers]; // columns of the arrays that hT and gT are part of
    int32_t parts[kMlpMaxLayers]; // partial column sums (rows of dbp)
    const uint16_t* hT[kMlpMaxLayers];
    const uint16_t* gT[kMlpMaxLayers];
    const float* dbp[kMlpMaxLayers];
    float* dW[kMlpMaxLayers];
    float* db[kMlpMaxLayers];
};

// Column sums of FP32 arrays [rows][ld] in row order, workgroups
// [first[i], first[i + 1]) for array i, 64 columns each.
struct ColsumArgs {
    int32_t n;
    int64_t rows;
    int32_t first[kMlpMaxLayers + 1];
    int32_t cols[kMlpMaxLayers];
    int64_t ld[kMlpMaxLayers];
    const float* src[kMlpMaxLayers];
    float* dst[kMlpMaxLayers];
    float* dst2[kMlpMaxLayers]; // a second copy, or NULL
};

__global__ __launch_bounds__(kBiasThreads) void colsum_kernel(ColsumArgs a)
{
    __shared__ float lds[kBiasRows * kBiasCols];
    int i = 0;
    while (i + 1 < a.n && (int)blockIdx.x >= a.first[i + 1]) ++i;
    column_sums(a.rows, a.cols[i], a.src[i], a.ld[i], (blockIdx.x - a.first[i]) * kBiasCols, lds, a.dst[i], a.dst2[i]);
}

__global__ __launch_bounds__(256) void mlp_dw_kernel(MlpDwArgs a)
{
    __shared__ float red[2][64][64]; // two wavefronts' partial tiles at a time: [register][lane]
    __shared__ float dred[4][64];
    int l = 0;
    while (l + 1 < a.layers && (int)blockIdx.x >= a.first[l + 1]) ++l;
    const int M = a.out[l], N = a.in[l], B = a.B;
    const int tn = (N + 63) / 64;
    const int tile = blockIdx.x - a.first[l];
    const int m0 = tile / tn * 64, n0 = tile % tn * 64;
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r = lane & 31;
    const bool one = gemm_one_chain(M, N);
    const int per = (B / 16 + 3) / 4 * 16;
    const int kb = one ? 0 : min(wid * per, B), ke = one ? B : min((wid + 1) * per, B);
    const uint16_t *pa[2], *pb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) { // a sub-tile past the edge repeats the last one and is not stored
        pa[i] = a.gT[l] + min(m0 + 32 * i, M - 32) * a.ldg[l] + lane * 8;
        pb[i] = a.hT[l] + min(n0 + 32 * i, N - 32) * a.ldh[l] + lane * 8;
    }
    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int x = 0; x < 16; ++x) acc[i][j][x] = 0.0f;
    if (one) {
        // wavefront (wid / 2, wid % 2) walks all of K for one 32x32 sub-tile
        const uint16_t* qa = pa[wid >> 1];
        const uint16_t* qb = pb[wid & 1];
#pragma unroll 4
        for (int k = 0; k < B; k += 16)
            acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                *reinterpret_cast<const bf16x8*>(qa + (int64_t)k * 32),
                *reinterpret_cast<const bf16x8*>(qb + (int64_t)k * 32), acc[0][0], 0, 0, 0);
        const int ms = m0 + 32 * (wid >> 1), ns = n0 + 32 * (wid & 1);
        if (ms < M && ns < N) {
#pragma unroll
            for (int x = 0; x < 16; ++x)
                a.dW[l][(int64_t)(ms + mfma_row(x, lane)) * N + ns + r] = acc[0][0][x] + 0.0f;
        }
    } else {
        bf16x8 ca[4][2], cb[4][2], xa[4][2], xb[4][2];
        auto load = [&](bf16x8 (&da)[4][2], bf16x8 (&db)[4][2], int k) {
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (k + 16 * u < ke) {
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        da[u][i] = *reinterpret_cast<const bf16x8*>(pa[i] + (int64_t)(k + 16 * u) * 32);
                        db[u][i] = *reinterpret_cast<const bf16x8*>(pb[i] + (int64_t)(k + 16 * u) * 32);
                    }
                }
        };
        load(ca, cb, kb);
        for (int k = kb; k < ke; k += 64) {
            if (k + 64 < ke) load(xa, xb, k + 64);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (k + 16 * u >= ke) break; // uniform
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ca[u][i], cb[u][j], acc[i][j], 0, 0, 0);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    ca[u][i] = xa[u][i];
                    cb[u][i] = xb[u][i];
                }
        }
        // wavefronts 1 and 2, then 3, hand their tiles to wavefront 0, which adds them in order
        if (wid == 1 || wid == 2) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int x = 0; x < 16; ++x) red[wid - 1][q * 16 + x][lane] = acc[q >> 1][q & 1][x];
        }
        __syncthreads();
        if (wid == 0) {
#pragma unroll
            for (int w = 0; w < 2; ++w)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int x = 0; x < 16; ++x) acc[q >> 1][q & 1][x] += red[w][q * 16 + x][lane];
        }
        __syncthreads();
        if (wid == 3) {
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int x = 0; x < 16; ++x) red[0][q * 16 + x][lane] = acc[q >> 1][q & 1][x];
        }
        __syncthreads();
        if (wid == 0) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int ms = m0 + 32 * (q >> 1), ns = n0 + 32 * (q & 1);
                if (ms >= M || ns >= N) continue;
#pragma unroll
                for (int x = 0; x < 16; ++x)
                    a.dW[l][(int64_t)(ms + mfma_row(x, lane)) * N + ns + r] =
                        acc[q >> 1][q & 1][x] + red[0][q * 16 + x][lane] + 0.0f;
            }
        }
    }
    if (tile % tn == 0 && a.db[l]) {
        const int c = m0 + lane;
        float s = 0.0f;
        if (c < M) {
#pragma unroll 8
            for (int k = wid; k < a.parts[l]; k += 4) s += a.dbp[l][(int64_t)k * M + c];
        }
        dred[wid][lane] = s;
        __syncthreads();
        if (wid == 0 && c < M) a.db[l][c] = (dred[0][lane] + dred[1][lane]) + (dred[2][lane] + dred[3][lane]);
    }
}

// Adam (UPDATE) on a list of parameter tensors [rows][cols] in one launch:
// 32x32 tiles, tile q of tensor i for first[i] <= q < first[i + 1].  The bf16
// copies are written with the update, through LDS: row-major (wb), transposed
// (wt), and in fragment order (wf, and wtf of the transpose; rows and cols
// multiples of 32), a tile of which is 2 KB contiguous.
constexpr int kAdamMax = 2 * kMlpMaxLayers;
struct AdamMultiArgs {
    int32_t n;
    int32_t first[kAdamMax + 1];
    int32_t rows[kAdamMax], cols[kAdamMax];
    float* w[kAdamMax];
    const float* g[kAdamMax];
    float* m[kAdamMax];
    float* v[kAdamMax];
    uint16_t* wb[kAdamMax];
    uint16_t* wt[kAdamMax];
    uint16_t* wf[kAdamMax];
    uint16_t* wtf[kAdamMax];
    float lr, b1, b2, eps, c1, c2;
};

template <bool UPDATE>
__global__ __launch_bounds__(256) void adam_multi_kernel(AdamMultiArgs a)
{
    __shared__ uint16_t tb[32][34];
    int i = 0;
    while (i + 1 < a.n && (int)blockIdx.x >= a.first[i + 1]) ++i;
    const int R = a.rows[i], C = a.cols[i], tc = (C + 31) / 32;
    const int tile = blockIdx.x - a.first[i];
    const int r0 = tile / tc * 32, c0 = tile % tc * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    float w[4], g[4], m[4], v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = r0 + ty + 8 * u, c = c0 + tx;
        if (r >= R || c >= C) continue;
        const int64_t x = (int64_t)r * C + c;
        w[u] = a.w[i][x];
        if (UPDATE) {
            g[u] = a.g[i][x];
            m[u] = a.m[i][x];
            v[u] = a.v[i][x];
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int r = r0 + ty + 8 * u, c = c0 + tx;
        if (r >= R || c >= C) continue;
        const int64_t x = (int64_t)r * C + c;
        if (UPDATE) {
            w[u] = adam_update(w[u], g[u], m[u], v[u], a.lr, a.b1, a.b2, a.eps, a.c1, a.c2);
            a.w[i][x] = w[u];
            a.m[i][x] = m[u];
            a.v[i][x] = v[u];
        }
        const uint16_t h = f2bf(w[u]);
        if (a.wb[i]) a.wb[i][x] = h;
        tb[ty + 8 * u][tx] = h;
    }
    if (!a.wt[i] && !a.wf[i] && !a.wtf[i]) return; // workgroup-uniform
    __syncthreads();
    if (a.wt[i]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int c = c0 + ty + 8 * u, r = r0 + tx; // [cols][rows]
            if (r < R && c < C) a.wt[i][(int64_t)c * R + r] = tb[tx][ty + 8 * u];
        }
    }
    // fragment order: thread -> four consecutive k of one row, 8 bytes
    const int x = threadIdx.x * 4;
    const int k = x / 512 * 16 + x % 512 / 256 * 8 + x % 8, n = x % 256 / 8;
    if (a.wf[i])
        *reinterpret_cast<ushort4*>(a.wf[i] + frag_at(C, r0, c0) + x) =
            make_ushort4(tb[n][k], tb[n][k + 1], tb[n][k + 2], tb[n][k + 3]);
    if (a.wtf[i])
        *reinterpret_cast<ushort4*>(a.wtf[i] + frag_at(R, c0, r0) + x) =
            make_ushort4(tb[k][n], tb[k + 1][n], tb[k + 2][n], tb[k + 3][n]);
}

__device__ inline float sigm(float x) { return 1.0f / (1.0f + __expf(-x)); }

// GRU cell (gate order r, z, n as torch.nn.GRU):
//   r = s(gi_r + gh_r), z = s(gi_z + gh_z), n = tanh(gi_n + r * gh_n), h' = (1 - z) n + z h
// gi = x W_ih^T + b_ih and gh = h W_hh^T + b_hh come from the GEMM, [B][3H] each.
__global__ void gru_forward_kernel(int32_t B, int32_t H, const float* __restrict__ gi, const float* __restrict__ gh,
                                   const float* __restrict__ h, float* __restrict__ hn, uint16_t* __restrict__ hnb)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)B * H) return;
    const int64_t b = i / H, j = i % H;
    const float* a = gi + b * 3 * H;
    const float* c = gh + b * 3 * H;
    const float r = sigm(a[j] + c[j]);
    const float z = sigm(a[H + j] + c[H + j]);
    const float n = tanhf(a[2 * H + j] + r * c[2 * H + j]);
    const float v = fmaf(1.0f - z, n, z * h[i]); // the sequence kernel's rounding too
    hn[i] = v;
    if (hnb) hnb[i] = f2bf(v);
}

// Backward of one GRU step with the gates recomputed from gi, gh, h.
// dh = dh_a + dh_b + dh_c (readout gradient, direct and GEMM parts of the
// next step's recurrent gradient; dh_b/dh_c may be NULL).  Writes
// dgi = [dr', dz', dn'] and dgh = [dr', dz', dn' * r] (FP32 and bf16) and the
// direct recurrent part dh_z = dh * z.
__global__ void gru_backward_kernel(int32_t B, int32_t H, const float* __restrict__ gi, const float* __restrict__ gh,
                                    const float* __restrict__ h, const float* __restrict__ dh_a,
                                    const float* __restrict__ dh_b, const float* __restrict__ dh_c,
                                    float* __restrict__ dgi, uint16_t* __restrict__ dgib, float* __restrict__ dgh,
                                    uint16_t* __restrict__ dghb, float* __restrict__ dh_z)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)B * H) return;
    const int64_t b = i / H, j = i % H;
    const int64_t o = b * 3 * H;
    const float r = sigm(gi[o + j] + gh[o + j]);
    const float z = sigm(gi[o + H + j] + gh[o + H + j]);
    const float ghn = gh[o + 2 * H + j];
    const float n = tanhf(gi[o + 2 * H + j] + r * ghn);
    float d = dh_a[i];
    if (dh_b) d += dh_b[i];
    if (dh_c) d += dh_c[i];
    const float dn = d * (1.0f - z) * (1.0f - n * n);
    const float dz = d * (h[i] - n) * z * (1.0f - z);
    const float dr = dn * ghn * r * (1.0f - r);
    dh_z[i] = d * z;
    dgi[o + j] = dr;
    dgi[o + H + j] = dz;
    dgi[o + 2 * H + j] = dn;
    dgh[o + j] = dr;
    dgh[o + H + j] = dz;
    dgh[o + 2 * H + j] = dn * r;
    if (dgib) {
        dgib[o + j] = f2bf(dr);
        dgib[o + H + j] = f2bf(dz);
        dgib[o + 2 * H + j] = f2bf(dn);
    }
    if (dghb) {
        dghb[o + j] = f2bf(dr);
        dghb[o + H + j] = f2bf(dz);
        dghb[o + 2 * H + j] = f2bf(dn * r);
    }
}

// ------------------------------------------------------ whole-sequence GRU
// A GRU step is a 64 x 768 x 256 product and 16,384 gates, so a launch per
// product and gate kernel left the device idle between them: 32 steps forward
// and backward were 128 launches, about 10 us each.  Batch rows never mix in
// the recurrence, so a workgroup takes kGruRows rows through all steps of the
// sequence, and keeps the recurrent weights on its CU: wavefront w holds the
// 16-row tiles w, w + 16, ... of W_hh (forward, 3H x H) or of its transpose
// (backward, H x 3H) as operands of v_mfma_f32_16x16x32_bf16, in registers and
// the rest in LDS (GruWeights).  Four rows a workgroup fill a quarter of an instruction's 16
// columns; more workgroups share the gates' arithmetic, which costs more than
// the products.  A step: products -> LDS -> barrier -> gates (a thread owns its
// rows' hidden units and keeps their h or gradient) -> LDS -> barrier; the
// step's inputs are loaded one step ahead.
// The products are summed as dtb_mlp_gemm_bf16_nt splits them (four
// consecutive ranges of K, added in order; a 16x16x32 instruction adds 32
// terms as two 32x32x16 ones do), so results equal the launch-per-step path.
// 32 steps x 64 rows x H = 256: 73 us forward and 112 us backward, against
// about 320 us each; the training step 2007 -> 251 us.
constexpr int kGruRows = 4;
constexpr int kGruFwdWaves = 8, kGruFwdHeld = 34;  // wavefronts and operands that each holds in registers
constexpr int kGruBwdWaves = 16, kGruBwdHeld = 16;
typedef float f32x4v __attribute__((ext_vector_type(4)));

// The recurrent weights of one of NW wavefronts: TW tiles of KS instructions'
// operands, the first HELD in registers and the others in LDS, 112 to 128 KB
// of it at H = 256.  Forward, eight wavefronts that hold 34 of their 48
// operands leave least to LDS (32 steps of 64 rows: 73 us, 109 with sixteen);
// backward the loaded gates need the registers too, and sixteen wavefronts that
// hold 16 of 24 do not spill (111 us, 189 with eight).
template <int TW, int KS, int NW, int HELD>
struct GruWeights {
    static constexpr int N = TW * KS;
    static constexpr int kReg = N < HELD ? N : HELD;
    static constexpr int kLds = (N - kReg) * NW * 64 * 16; // bytes of a workgroup
    bf16x8 r[kReg];
    const bf16x8* l;

    // rows of W: tile wid + NW i, [16 tiles][K]; past the last tile the last one again
    __device__ __forceinline__ void load(const uint16_t* __restrict__ W, int tiles, int wid, int lane, uint16_t* lds)
    {
        bf16x8* p = reinterpret_cast<bf16x8*>(lds) + (size_t)wid * (N - kReg) * 64 + lane;
        l = p;
#pragma unroll
        for (int i = 0; i < TW; ++i) {
            const int tile = min(wid + NW * i, tiles - 1);
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const bf16x8 v = *reinterpret_cast<const bf16x8*>(W + (int64_t)(tile * 16 + (lane & 15)) * (32 * KS) +
                                                                  32 * s + (lane >> 4) * 8);
                if (i * KS + s < kReg) r[i * KS + s] = v;
                else p[(i * KS + s - kReg) * 64] = v; // read back by this lane alone
            }
        }
    }
    __device__ __forceinline__ bf16x8 get(int f) const { return f < kReg ? r[f < kReg ? f : 0] : l[(f - kReg) * 64]; }
};

// KS = K / 32.  tot = sum over K in four consecutive ranges of `per` steps of
// 16: tile i of the weights by h, the other operand in LDS.
template <int KS, typename Weights>
__device__ __forceinline__ f32x4v gru_product(const Weights& W, int i, const uint16_t* h, bool upper)
{
    constexpr int per = (2 * KS + 3) / 4;
    f32x4v acc = {0.0f, 0.0f, 0.0f, 0.0f}, tot = {-0.0f, -0.0f, -0.0f, -0.0f};
    const bf16x8 zero = {};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(h + 32 * s);
        const bf16x8 a = W.get(i * KS + s);
        if (s > 0 && (2 * s) % per == 0) {
            tot += acc;
            acc = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
        }
        if ((2 * s + 1) % per == 0) { // a range ends inside this instruction's 32 columns: its halves apart
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(upper ? zero : a, b, acc, 0, 0, 0);
            tot += acc;
            acc = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(upper ? a : zero, b, acc, 0, 0, 0);
        } else {
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
        }
    }
    return tot + acc;
}

// G = H / 32.  gi [T][B][3H]; h0 [rows][H] or NULL (zeros; rows past h0_rows
// start at zero); writes gh [T][B][3H], hs [T + 1][B][H] and its bf16 copy.
template <int G>
__global__ __launch_bounds__(64 * kGruFwdWaves) void gru_seq_forward_kernel(int32_t T, int32_t B, const float* __restrict__ gi,
                                                                     const uint16_t* __restrict__ W,
                                                                     const float* __restrict__ bhh,
                                                                     const float* __restrict__ h0, int32_t h0_rows,
                                                                     float* __restrict__ gh, float* __restrict__ hs,
                                                                     uint16_t* __restrict__ hb)
{
    constexpr int kGruWaves = kGruFwdWaves, kGruThreads = 64 * kGruWaves;
    constexpr int H = 32 * G, NT = 3 * H / 16, TW = (NT + kGruWaves - 1) / kGruWaves;
    constexpr int EP = (kGruRows * H + kGruThreads - 1) / kGruThreads;
    constexpr int LH = H + 8, LG = 3 * H + 4;
    __shared__ __align__(16) uint16_t sh[kGruRows * LH];
    __shared__ __align__(16) float sg[kGruRows * LG];
    const int t = threadIdx.x, lane = t & 63;
    const int wid = __builtin_amdgcn_readfirstlane(t >> 6);
    const int row0 = blockIdx.x * kGruRows;
    extern __shared__ __align__(16) uint16_t sw[];
    GruWeights<TW, G, kGruWaves, kGruFwdHeld> w;
    w.load(W, NT, wid, lane, sw);
    // this thread's elements (row, unit j): x = t + threads u
    float h[EP], b3[EP][3], g[EP][3];
    uint32_t at[EP], at3[EP]; // element of a step's [B][H] and [B][3H]
    auto own = [&](int u) { return (kGruRows * H) % kGruThreads == 0 || t + kGruThreads * u < kGruRows * H; };
#pragma unroll
    for (int u = 0; u < EP; ++u) {
        const int x = t + kGruThreads * u, r = x / H, j = x % H;
        const int rr = own(u) ? r : 0, jj = own(u) ? j : 0;
        at[u] = (uint32_t)(row0 + rr) * H + jj;
        at3[u] = (uint32_t)(row0 + rr) * 3 * H + jj;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            b3[u][q] = bhh[q * H + jj];
            g[u][q] = gi[at3[u] + q * H];
        }
        h[u] = h0 && row0 + rr < h0_rows ? h0[at[u]] : 0.0f;
        if (own(u)) {
            const uint16_t hv = (uint16_t)f2bf_pk(h[u], 0.0f);
            hs[at[u]] = h[u];
            hb[at[u]] = hv;
            sh[r * LH + j] = hv;
        }
    }
    __syncthreads();
    for (int32_t k = 0; k < T; ++k) {
        const int64_t step = (int64_t)k * B;
        float gn[EP][3]; // the next step's input projections
        const float* gk = gi + (k + 1 < T ? step + B : step) * 3 * H;
        float* ghk = gh + step * 3 * H;
        float* hsk = hs + (step + B) * H;
        uint16_t* hbk = hb + (step + B) * H;
#pragma unroll
        for (int u = 0; u < EP; ++u)
#pragma unroll
            for (int q = 0; q < 3; ++q) gn[u][q] = gk[at3[u] + q * H];
        const uint16_t* ph = sh + (lane & (kGruRows - 1)) * LH + (lane >> 4) * 8;
#pragma unroll
        for (int i = 0; i < TW; ++i) {
            const int tile = wid + kGruWaves * i;
            if (tile >= NT) break; // uniform
            const f32x4v p = gru_product<G>(w, i, ph, lane >= 32);
            if ((lane & 15) < kGruRows)
                *reinterpret_cast<f32x4v*>(sg + (lane & 15) * LG + tile * 16 + 4 * (lane >> 4)) = p;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < EP; ++u) {
            if (!own(u)) continue;
            const int x = t + kGruThreads * u, r = x / H, j = x % H;
            const float c0 = sg[r * LG + j] + b3[u][0], c1 = sg[r * LG + H + j] + b3[u][1],
                        c2 = sg[r * LG + 2 * H + j] + b3[u][2];
            ghk[at3[u]] = c0;
            ghk[at3[u] + H] = c1;
            ghk[at3[u] + 2 * H] = c2;
            const float rr = sigm(g[u][0] + c0);
            const float z = sigm(g[u][1] + c1);
            const float n = tanhf(g[u][2] + rr * c2);
            h[u] = fmaf(1.0f - z, n, z * h[u]);
            const uint16_t hv = (uint16_t)f2bf_pk(h[u], 0.0f);
            hsk[at[u]] = h[u];
            hbk[at[u]] = hv;
            sh[r * LH + j] = hv;
#pragma unroll
            for (int q = 0; q < 3; ++q) g[u][q] = gn[u][q];
        }
        __syncthreads();
    }
}

// Backward through the sequence.  dho [T][B][H] gradients from the readout;
// writes dgi and dgh in bf16 [T][B][3H], and in FP32 dg [T][B][4H] = dr, dz, dn
// (of gi) and dn r (of gh), whose sums are the bias gradients.
template <int G>
__global__ __launch_bounds__(64 * kGruBwdWaves) void gru_seq_backward_kernel(int32_t T, int32_t B,
                                                                      const float* __restrict__ gi,
                                                                      const float* __restrict__ gh,
                                                                      const float* __restrict__ hs,
                                                                      const float* __restrict__ dho,
                                                                      const uint16_t* __restrict__ WT,
                                                                      uint16_t* __restrict__ dgib,
                                                                      uint16_t* __restrict__ dghb,
                                                                      float* __restrict__ dg)
{
    constexpr int kGruWaves = kGruBwdWaves, kGruThreads = 64 * kGruWaves;
    constexpr int H = 32 * G, NT = H / 16, TW = (NT + kGruWaves - 1) / kGruWaves, KS = 3 * G;
    constexpr int EP = (kGruRows * H + kGruThreads - 1) / kGruThreads;
    constexpr int LG = 3 * H + 8, LD = H + 4;
    __shared__ __align__(16) uint16_t sg[kGruRows * LG]; // dgh of the step, bf16
    __shared__ __align__(16) float sd[kGruRows * LD];    // its product with W_hh
    const int t = threadIdx.x, lane = t & 63;
    const int wid = __builtin_amdgcn_readfirstlane(t >> 6);
    const int row0 = blockIdx.x * kGruRows;
    extern __shared__ __align__(16) uint16_t sw[];
    GruWeights<TW, KS, kGruWaves, kGruBwdHeld> w;
    w.load(WT, NT, wid, lane, sw);
    struct In {
        float gi[3], gh[3], h, dho;
    };
    uint32_t at[EP], at3[EP]; // element of a step's [B][H] and [B][3H]
    auto own = [&](int u) { return (kGruRows * H) % kGruThreads == 0 || t + kGruThreads * u < kGruRows * H; };
    float dhz[EP];
    In cur[EP];
    auto load = [&](In& v, int u, int64_t k) {
        const float* gik = gi + k * B * 3 * H;
        const float* ghk = gh + k * B * 3 * H;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            v.gi[q] = gik[at3[u] + q * H];
            v.gh[q] = ghk[at3[u] + q * H];
        }
        v.h = (hs + k * B * H)[at[u]];
        v.dho = (dho + k * B * H)[at[u]];
    };
#pragma unroll
    for (int u = 0; u < EP; ++u) {
        const int x = t + kGruThreads * u;
        const int r = own(u) ? x / H : 0, j = own(u) ? x % H : 0;
        at[u] = (uint32_t)(row0 + r) * H + j;
        at3[u] = (uint32_t)(row0 + r) * 3 * H + j;
        dhz[u] = 0.0f;
        load(cur[u], u, T - 1);
    }
    for (int32_t k = T - 1; k >= 0; --k) {
        In next[EP];
#pragma unroll
        for (int u = 0; u < EP; ++u) load(next[u], u, k > 0 ? k - 1 : 0);
#pragma unroll
        for (int u = 0; u < EP; ++u) {
            if (!own(u)) continue;
            const int x = t + kGruThreads * u, r = x / H, j = x % H;
            const In& v = cur[u];
            const float rr = sigm(v.gi[0] + v.gh[0]);
            const float z = sigm(v.gi[1] + v.gh[1]);
            const float n = tanhf(v.gi[2] + rr * v.gh[2]);
            float d = v.dho;
            if (k < T - 1) {
                d += dhz[u];
                d += sd[r * LD + j] + 0.0f;
            }
            const float dn = d * (1.0f - z) * (1.0f - n * n);
            const float dz = d * (v.h - n) * z * (1.0f - z);
            const float dr = dn * v.gh[2] * rr * (1.0f - rr);
            const float dnr = dn * rr;
            dhz[u] = d * z;
            const uint32_t a = f2bf_pk(dr, dz), c = f2bf_pk(dn, dnr);
            uint16_t* gib = dgib + (int64_t)k * B * 3 * H;
            uint16_t* ghb = dghb + (int64_t)k * B * 3 * H;
            gib[at3[u]] = (uint16_t)a;
            gib[at3[u] + H] = (uint16_t)(a >> 16);
            gib[at3[u] + 2 * H] = (uint16_t)c;
            ghb[at3[u]] = (uint16_t)a;
            ghb[at3[u] + H] = (uint16_t)(a >> 16);
            ghb[at3[u] + 2 * H] = (uint16_t)(c >> 16);
            uint16_t* p = sg + r * LG + j;
            p[0] = (uint16_t)a;
            p[H] = (uint16_t)(a >> 16);
            p[2 * H] = (uint16_t)(c >> 16);
            float* g4 = dg + (int64_t)k * B * 4 * H + at3[u] + (at3[u] - j) / 3; // row * 4H + j
            g4[0] = dr;
            g4[H] = dz;
            g4[2 * H] = dn;
            g4[3 * H] = dnr;
        }
        __syncthreads();
        if (k == 0) break; // uniform: nothing before the first step
        const uint16_t* ph = sg + (lane & (kGruRows - 1)) * LG + (lane >> 4) * 8;
#pragma unroll
        for (int i = 0; i < TW; ++i) {
            const int tile = wid + kGruWaves * i;
            if (tile >= NT) break; // uniform
            const f32x4v p = gru_product<KS>(w, i, ph, lane >= 32);
            if ((lane & 15) < kGruRows)
                *reinterpret_cast<f32x4v*>(sd + (lane & 15) * LD + tile * 16 + 4 * (lane >> 4)) = p;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < EP; ++u) cur[u] = next[u];
    }
}

// Row-major bf16 [K][N] (row stride ld) into the fragment order of [N][K]:
// tile q of matrix i for first[i] <= q < first[i + 1], 32 rows x 32 columns.
struct PackArgs {
    int32_t n;
    int32_t first[kMlpMaxLayers * 2 + 1];
    int32_t K[kMlpMaxLayers * 2], N[kMlpMaxLayers * 2];
    const uint16_t* in[kMlpMaxLayers * 2];
    int64_t ld[kMlpMaxLayers * 2];
    uint16_t* out[kMlpMaxLayers * 2];
};

__global__ __launch_bounds__(256) void pack_transposed_kernel(PackArgs a)
{
    __shared__ uint16_t tb[32][34]; // [k][n]
    int i = 0;
    while (i + 1 < a.n && (int)blockIdx.x >= a.first[i + 1]) ++i;
    const int tn = a.N[i] / 32, tile = blockIdx.x - a.first[i];
    const int k0 = tile / tn * 32, n0 = tile % tn * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
#pragma unroll
    for (int u = 0; u < 4; ++u) tb[ty + 8 * u][tx] = a.in[i][(int64_t)(k0 + ty + 8 * u) * a.ld[i] + n0 + tx];
    __syncthreads();
    const int x = threadIdx.x * 4;
    const int k = x / 512 * 16 + x % 512 / 256 * 8 + x % 8, n = x % 256 / 8;
    *reinterpret_cast<ushort4*>(a.out[i] + frag_at(a.K[i], n0, k0) + x) =
        make_ushort4(tb[k][n], tb[k + 1][n], tb[k + 2][n], tb[k + 3][n]);
}

// Gradient and loss of a sequence's outputs [T][B][O]: targets and mask
// [T][rows][n_out] (masked out past rows and n_out), the arithmetic of
// affine_kernel and mse_grad_kernel.
__global__ __launch_bounds__(256) void seq_loss_kernel(int64_t n, int32_t B, int32_t O, int32_t rows, int32_t n_out,
                                                       const float* __restrict__ out, const float* __restrict__ Y,
                                                       const float* __restrict__ ys, const float* __restrict__ yh,
                                                       const float* __restrict__ mask, float scale,
                                                       float* __restrict__ grad, uint16_t* __restrict__ gradb,
                                                       float* __restrict__ lsum)
{
    __shared__ float red[256];
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    float e = 0.0f;
    if (i < n) {
        const int32_t c = (int32_t)(i % O);
        const int64_t tb = i / O;
        const int32_t b = (int32_t)(tb % B);
        float tgt = 0.0f, mk = 0.0f;
        if (c < n_out) tgt = yh[c]; // a padded row's target is the shift of a zero
        if (c < n_out && b < rows) {
            const int64_t x = (tb / B * rows + b) * n_out + c;
            tgt = Y[x] * ys[c] + yh[c];
            mk = mask ? mask[x] : 1.0f;
        }
        const float d = (out[i] - tgt) * mk;
        e = d * d;
        const float g = scale * d;
        grad[i] = g;
        gradb[i] = f2bf(g);
    }
    red[threadIdx.x] = e;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) lsum[blockIdx.x] = red[0];
}

template <int G>
using GruFwdWeights = GruWeights<(6 * G + kGruFwdWaves - 1) / kGruFwdWaves, G, kGruFwdWaves, kGruFwdHeld>;
template <int G>
using GruBwdWeights = GruWeights<(2 * G + kGruBwdWaves - 1) / kGruBwdWaves, 3 * G, kGruBwdWaves, kGruBwdHeld>;

// Which kernel takes a product: the tile of gemm_nt_tile_kernel in units of 64
// (-1: 64x64 tiles, K in four ranges), or 0 for the split-K kernel.
// Rules from both sides' times, us (K = 2048 unless given):
//   128 or more 64x64 tiles: split-K's 32x32 tiles read each operand row twice
//     as often, in 32-byte pieces (768^2 K = 768: 13.5 split, 7.1 tiles; 96 x
//     6144 K = 3008: 38.3, 21.1); up to 64 its workgroups are the only ones
//     that fill the CUs (512^2 K = 512: 4.7, 6.0), and so they are up to 256
//     32x32 tiles, a round of one a CU, where a 64x64 tile is half padding (32 x
//     8192 K = 4096: 22.0, 29.0; 32 x 12000, 375 tiles: 36.9, 30.1);
//   128x128 tiles once every CU gets one (2048^2: 64x64 29.4, 128x128 23.8;
//     1536^2 K = 1536, 144 tiles: 15.5, 17.0);
//   256x256 tiles, one a CU and 1.75 times the time of a round of 128x128
//     tiles, two a CU, where that many fewer rounds do (best of several back
//     to back, 8192^3: 808 against
//     1033; 5024 x 1632 K = 2000: 51 against 59; 6144^3, 2.25 rounds: 426
//     against 416);
//   a short K is bound by the stores of C, which several workgroups a CU
//     overlap and one does not: 64x64 tiles up to K = 256, or 192 past 2,304
//     tiles of 256 (8192^2, tiles of 64, 128 and 256: K = 64 48, 52, 62; 128 53,
//     57, 67; 256 77, 73, 82; 384 101, 88, 95.  8192 x 12288: 128 84, 114, 106;
//     256 113, 137, 125; 384 144, 185, 149.  4096^2 K = 256: 22.0, 22.3, 23.5.
//     16384^2: 128 278, 281, 309; 256 397, 373, 362).
static int gemm_tile(int32_t M, int32_t N, int32_t K)
{
    auto tiles = [&](int32_t t) { return (int64_t)((M + t - 1) / t) * ((N + t - 1) / t); };
    if (!gemm_one_chain(M, N)) return tiles(64) >= 128 && tiles(32) > 256 ? -1 : 0;
    if (tiles(128) < 256 || K <= 192 || (K <= 256 && tiles(256) <= 2304)) return 1;
    const int64_t r4 = (tiles(256) + 255) / 256, r2 = (tiles(128) + 511) / 512;
    return 7 * r4 <= 4 * r2 ? 4 : 2;
}

template <int T, bool RANGES>
static int launch_gemm_tile(int32_t M, int32_t N, int32_t K, const void* A, int64_t lda, const void* B, int64_t ldb,
                            const float* bias, int32_t act, float* C, int64_t ldc, void* Cb, int64_t ldcb, void* stream)
{
    constexpr int GM = T == 4 ? 4 : 8; // about the square root of the tiles an XCD's 32 CUs hold
    constexpr int lds = 5 * 64 * T * 64 * (int)sizeof(uint16_t);
    const int64_t tiles = (int64_t)((M + 64 * T - 1) / (64 * T)) * ((N + 64 * T - 1) / (64 * T));
    DTB_TRY_HIP(hipFuncSetAttribute((const void*)gemm_nt_tile_kernel<T, GM, RANGES>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, lds));
    hipLaunchKernelGGL((gemm_nt_tile_kernel<T, GM, RANGES>), dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(256), lds,
                       (hipStream_t)stream, M, N, K, (const uint16_t*)A, lda, (const uint16_t*)B, ldb, bias, act, C, ldc,
                       (uint16_t*)Cb, ldcb);
    return DTB_OK;
}

static inline dim3 g1(int64_t n) { return dim3((unsigned)((n + 255) / 256)); }

} // namespace dtb

using namespace dtb;

extern "C" {

int dtb_mlp_gemm_bf16_nt(int32_t M, int32_t N, int32_t K, const void* A, int64_t lda, const void* B, int64_t ldb,
                         const float* bias, int32_t act, float* C, int64_t ldc, void* Cb, int64_t ldcb, void* stream)
{
    DTB_REQUIRE(M > 0 && N > 0 && K > 0, "M, N, K must be positive");
    DTB_REQUIRE(M % 32 == 0 && N % 32 == 0 && K % 16 == 0, "M and N must be multiples of 32 and K of 16");
    DTB_REQUIRE(A && B && (C || Cb), "A, B and an output are required");
    DTB_REQUIRE(lda >= K && ldb >= K && lda % 8 == 0 && ldb % 8 == 0, "lda, ldb must be >= K and multiples of 8");
    DTB_REQUIRE(act == 0 || act == 1, "act must be 0 (identity) or 1 (ReLU)");
    DTB_REQUIRE((reinterpret_cast<uintptr_t>(A) & 15) == 0 && (reinterpret_cast<uintptr_t>(B) & 15) == 0,
                "A and B must be 16-byte aligned");
    switch (gemm_tile(M, N, K)) {
    case 4: DTB_TRY((launch_gemm_tile<4, false>(M, N, K, A, lda, B, ldb, bias, act, C, ldc, Cb, ldcb, stream))); break;
    case 2: DTB_TRY((launch_gemm_tile<2, false>(M, N, K, A, lda, B, ldb, bias, act, C, ldc, Cb, ldcb, stream))); break;
    case 1: DTB_TRY((launch_gemm_tile<1, false>(M, N, K, A, lda, B, ldb, bias, act, C, ldc, Cb, ldcb, stream))); break;
    case -1: DTB_TRY((launch_gemm_tile<1, true>(M, N, K, A, lda, B, ldb, bias, act, C, ldc, Cb, ldcb, stream))); break;
    default: {
        dim3 grid((unsigned)(N / 32), (unsigned)(M / 32));
        hipLaunchKernelGGL(gemm_nt_splitk_kernel, grid, dim3(256), 0, (hipStream_t)stream, M, N, K,
                           (const uint16_t*)A, lda, (const uint16_t*)B, ldb, bias, act, C, ldc, (uint16_t*)Cb, ldcb);
    }
    }
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_relu_backward(int64_t n, const float* dY, const float* Z, float* dZ, void* dZb, void* stream)
{
    DTB_REQUIRE(n >= 0 && dY && Z && (dZ || dZb), "bad arguments");
    if (n == 0) return DTB_OK;
    hipLaunchKernelGGL(relu_backward_kernel, g1(n), dim3(256), 0, (hipStream_t)stream, n, dY, Z, dZ, (uint16_t*)dZb);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_bias_grad(int32_t M, int32_t N, const float* dZ, float* db, void* stream)
{
    DTB_REQUIRE(M > 0 && N > 0 && dZ && db, "bad arguments");
    hipLaunchKernelGGL(bias_grad_kernel, dim3((unsigned)((N + kBiasCols - 1) / kBiasCols)), dim3(kBiasThreads),
                       0, (hipStream_t)stream, M, N, dZ, db);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_mse_grad(int64_t n, const float* out, const float* target, const float* mask, float scale, float* grad,
                     void* gradb, float* lsum, void* stream)
{
    DTB_REQUIRE(n > 0 && out && target, "bad arguments");
    hipLaunchKernelGGL(mse_grad_kernel, g1(n), dim3(256), 0, (hipStream_t)stream, n, out, target, mask, scale, grad,
                       (uint16_t*)gradb, lsum);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_adam(int64_t n, float* w, const float* g, float* m, float* v, float lr, float b1, float b2, float eps,
                 int32_t t, void* wb, void* stream)
{
    DTB_REQUIRE(n > 0 && w && g && m && v && t >= 1, "bad arguments");
    const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
    hipLaunchKernelGGL(adam_kernel, g1(n), dim3(256), 0, (hipStream_t)stream, n, w, g, m, v, lr, b1, b2, eps, c1, c2,
                       (uint16_t*)wb);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_transpose_bf16(int32_t M, int32_t N, const void* in, void* out, void* stream)
{
    DTB_REQUIRE(M > 0 && N > 0 && in && out, "bad arguments");
    dim3 grid((unsigned)((N + 31) / 32), (unsigned)((M + 31) / 32));
    hipLaunchKernelGGL(transpose_bf16_kernel, grid, dim3(256), 0, (hipStream_t)stream, M, N, (const uint16_t*)in,
                       (uint16_t*)out);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_f32_to_bf16(int64_t n, const float* in, void* out, void* stream)
{
    DTB_REQUIRE(n >= 0 && in && out, "bad arguments");
    if (n == 0) return DTB_OK;
    hipLaunchKernelGGL(f32_to_bf16_kernel, g1(n), dim3(256), 0, (hipStream_t)stream, n, in, (uint16_t*)out);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_affine(int32_t rows, int32_t cin, int32_t cout, const float* in, int64_t ldi, const float* scale,
                   const float* shift, float* out, void* outb, int64_t ldo, void* stream)
{
    DTB_REQUIRE(rows >= 0 && cin >= 0 && cout >= cin && in && (out || outb), "bad arguments");
    DTB_REQUIRE(ldi >= cin && ldo >= cout, "ldi must be >= cin and ldo >= cout");
    if ((int64_t)rows * cout == 0) return DTB_OK;
    hipLaunchKernelGGL(affine_kernel, g1((int64_t)rows * cout), dim3(256), 0, (hipStream_t)stream, rows, cin, cout,
                       in, ldi, scale, shift, out, (uint16_t*)outb, ldo);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

// LDS of the chain kernel: two activation buffers of 32 rows (wide enough for
// the widest layer and for the exchange of a split product; the row stride
// keeps the 32 rows of a fragment on distinct banks), then in training the sign
// masks of the hidden outputs.
static int chain_layout(int32_t n_layers, const dtb_mlp_layer* L, bool train, int32_t* bufw, size_t* lds)
{
    DTB_REQUIRE(n_layers >= 1 && L != nullptr, "at least one layer is required");
    int64_t wide = 192, hidden = 0;
    for (int32_t l = 0; l < n_layers; ++l) {
        DTB_REQUIRE(L[l].n_in > 0 && L[l].n_out > 0 && L[l].n_in % 32 == 0 && L[l].n_out % 32 == 0,
                    "layer %d: widths must be positive multiples of 32", l);
        DTB_REQUIRE(L[l].n_in < (1 << 24) && L[l].n_out < (1 << 24), "layer %d: widths must be below 2^24", l);
        DTB_REQUIRE(l == 0 || L[l].n_in == L[l - 1].n_out, "layer %d does not take the width of the layer before", l);
        wide = std::max(wide, std::max(L[l].n_in, L[l].n_out));
        if (l + 1 < n_layers) hidden += L[l].n_out / 32;
    }
    wide = (wide + 63) / 64 * 64 + 8;
    const int64_t need = 2 * kMlpRows * wide * 2 + (train ? hidden * 128 : 0);
    if (n_layers > kMlpMaxLayers || need > 160 * 1024) {
        set_error("the chain kernel holds at most %d layers and 160 KB of activations", kMlpMaxLayers);
        return DTB_UNSUPPORTED;
    }
    *bufw = (int32_t)wide;
    *lds = (size_t)need;
    return DTB_OK;
}

static int chain_fill(MlpChainArgs& a, int32_t n_layers, const dtb_mlp_layer* L, bool train)
{
    for (int32_t l = 0; l < n_layers; ++l) {
        DTB_REQUIRE(L[l].w && L[l].bias &&
                        ((reinterpret_cast<uintptr_t>(L[l].w) | reinterpret_cast<uintptr_t>(L[l].bias)) & 15) == 0,
                    "layer %d: bf16 weights and bias (16-byte aligned) are required", l);
        DTB_REQUIRE(!train || (L[l].wt && L[l].dw && L[l].db && L[l].ht && L[l].gt && L[l].dbp &&
                               ((reinterpret_cast<uintptr_t>(L[l].wt) | reinterpret_cast<uintptr_t>(L[l].ht) |
                                 reinterpret_cast<uintptr_t>(L[l].gt)) & 15) == 0),
                    "layer %d: training needs the transposed weights, gradients and scratch (16-byte aligned)", l);
        a.l[l] = MlpLayerDev{(int32_t)L[l].n_in, (int32_t)L[l].n_out, (const uint16_t*)L[l].w, (const uint16_t*)L[l].wt,
                             L[l].bias, (uint16_t*)L[l].ht, (uint16_t*)L[l].gt, L[l].dbp};
    }
    a.layers = n_layers;
    return DTB_OK;
}

int dtb_mlp_chain_fits(int32_t n_layers, const dtb_mlp_layer* layers, int32_t train)
{
    int32_t bufw;
    size_t lds;
    return chain_layout(n_layers, layers, train != 0, &bufw, &lds);
}

int dtb_mlp_predict(int32_t n_layers, const dtb_mlp_layer* layers, int32_t rows, int32_t batch, const float* X,
                    int64_t ldx, int32_t cin, const float* x_scale, const float* x_shift, const float* y_scale,
                    const float* y_shift, int32_t cout, float* out, int64_t ldo, void* stream)
{
    MlpChainArgs a{};
    size_t lds = 0;
    DTB_TRY(chain_layout(n_layers, layers, false, &a.bufw, &lds));
    DTB_TRY(chain_fill(a, n_layers, layers, false));
    DTB_REQUIRE(rows >= 0 && rows < 0x7fffffe0 && batch > 0 && batch % 32 == 0, "batch must be a positive multiple of 32");
    DTB_REQUIRE(cin >= 0 && cin <= layers[0].n_in && cout >= 0 && cout <= layers[n_layers - 1].n_out,
                "cin and cout must be within the widths");
    if (rows == 0 || cout == 0) return DTB_OK;
    DTB_REQUIRE((X || cin == 0) && out && ldx >= cin && ldo >= cout, "X, out and their strides are required");
    a.rows = rows; a.max_batch = batch; a.cin = cin; a.cout = cout;
    a.X = X; a.ldx = ldx; a.xs = x_scale; a.xh = x_shift; a.ys = y_scale; a.yh = y_shift; a.out = out; a.ldo = ldo;
    // 64 rows a workgroup, which halve the weights read per row, once 32-row
    // ones would not all be resident (the second buffer must still fit, and a
    // batch boundary must not fall inside a workgroup's rows)
    const bool wide = rows > 32 * 256 && batch % 64 == 0 && 2 * lds <= 160 * 1024;
    if (wide) {
        DTB_TRY_HIP(hipFuncSetAttribute((const void*)mlp_chain_kernel<false, 2>,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        hipLaunchKernelGGL((mlp_chain_kernel<false, 2>), dim3((unsigned)((rows + 63) / 64)), dim3(kMlpThreads), 2 * lds,
                           (hipStream_t)stream, a);
    } else {
        DTB_TRY_HIP(hipFuncSetAttribute((const void*)mlp_chain_kernel<false, 1>,
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        hipLaunchKernelGGL((mlp_chain_kernel<false, 1>), dim3((unsigned)((rows + 31) / 32)), dim3(kMlpThreads), lds,
                           (hipStream_t)stream, a);
    }
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_train_gradients(int32_t n_layers, const dtb_mlp_layer* layers, int32_t rows, const float* X, int64_t ldx,
                            int32_t cin, const float* x_scale, const float* x_shift, const float* Y, int64_t ldy,
                            int32_t cout, const float* y_scale, const float* y_shift, const float* mask, int64_t ldm,
                            float scale, float* out, float* lsum, void* stream)
{
    MlpChainArgs a{};
    size_t lds = 0;
    DTB_TRY(chain_layout(n_layers, layers, true, &a.bufw, &lds));
    DTB_TRY(chain_fill(a, n_layers, layers, true));
    DTB_REQUIRE(rows > 0 && rows < (1 << 26), "rows must be in 1 .. 2^26");
    DTB_REQUIRE(cin >= 0 && cin <= layers[0].n_in && cout >= 0 && cout <= layers[n_layers - 1].n_out,
                "cin and cout must be within the widths");
    DTB_REQUIRE((X || cin == 0) && (Y || cout == 0) && out && lsum && ldx >= cin && ldy >= cout &&
                    (!mask || ldm >= cout),
                "X, Y, out, lsum and their strides are required");
    const int32_t B = (rows + 31) / 32 * 32;
    a.rows = rows; a.max_batch = B; a.cin = cin; a.cout = cout;
    a.X = X; a.ldx = ldx; a.xs = x_scale; a.xh = x_shift; a.ys = y_scale; a.yh = y_shift;
    a.out = out; a.ldo = layers[n_layers - 1].n_out;
    a.Y = Y; a.ldy = ldy; a.mask = mask; a.ldm = ldm; a.scale = scale; a.lsum = lsum;
    DTB_TRY_HIP(hipFuncSetAttribute((const void*)mlp_chain_kernel<true, 1>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    160 * 1024));
    hipLaunchKernelGGL((mlp_chain_kernel<true, 1>), dim3((unsigned)(B / 32)), dim3(kMlpThreads), lds, (hipStream_t)stream, a);
    DTB_TRY_HIP(hipGetLastError());
    MlpDwArgs d{};
    d.layers = n_layers;
    d.B = B;
    for (int32_t l = 0; l < n_layers; ++l) {
        d.in[l] = a.l[l].in; d.out[l] = a.l[l].out;
        d.ldh[l] = d.ldg[l] = B; d.parts[l] = B / 32;
        d.hT[l] = a.l[l].hT; d.gT[l] = a.l[l].gT; d.dbp[l] = a.l[l].dbp;
        d.dW[l] = layers[l].dw; d.db[l] = layers[l].db;
        d.first[l + 1] = d.first[l] + (a.l[l].out + 63) / 64 * ((a.l[l].in + 63) / 64);
    }
    hipLaunchKernelGGL(mlp_dw_kernel, dim3((unsigned)d.first[n_layers]), dim3(256), 0, (hipStream_t)stream, d);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

static int adam_multi(int32_t n, const dtb_adam_param* p, bool update, float lr, float b1, float b2, float eps,
                      int32_t t, void* stream)
{
    DTB_REQUIRE(n >= 0 && (n == 0 || p) && t >= 1, "bad arguments");
    for (int32_t i = 0; i < n; ++i) {
        DTB_REQUIRE(p[i].rows > 0 && p[i].cols > 0 && p[i].rows < (1 << 24) && p[i].cols < (1 << 24) && p[i].w &&
                        (!update || (p[i].g && p[i].m && p[i].v)),
                    "parameter %d: bad arguments", i);
        DTB_REQUIRE((!p[i].wf && !p[i].wtf) ||
                        (p[i].rows % 32 == 0 && p[i].cols % 32 == 0 &&
                         ((reinterpret_cast<uintptr_t>(p[i].wf) | reinterpret_cast<uintptr_t>(p[i].wtf)) & 15) == 0),
                    "parameter %d: fragment order needs multiples of 32 and 16-byte alignment", i);
    }
    const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
    for (int32_t i0 = 0; i0 < n; i0 += kAdamMax) {
        AdamMultiArgs a{};
        a.n = std::min(kAdamMax, n - i0);
        int64_t tiles = 0;
        for (int32_t i = 0; i < a.n; ++i) {
            const dtb_adam_param& q = p[i0 + i];
            a.rows[i] = (int32_t)q.rows; a.cols[i] = (int32_t)q.cols;
            a.w[i] = q.w; a.g[i] = q.g; a.m[i] = q.m; a.v[i] = q.v;
            a.wb[i] = (uint16_t*)q.wb; a.wt[i] = (uint16_t*)q.wt;
            a.wf[i] = (uint16_t*)q.wf; a.wtf[i] = (uint16_t*)q.wtf;
            tiles += (q.rows + 31) / 32 * ((q.cols + 31) / 32);
            DTB_REQUIRE(tiles < (1ll << 31), "too many parameters for one launch");
            a.first[i + 1] = (int32_t)tiles;
        }
        a.lr = lr; a.b1 = b1; a.b2 = b2; a.eps = eps; a.c1 = c1; a.c2 = c2;
        if (update)
            hipLaunchKernelGGL(adam_multi_kernel<true>, dim3((unsigned)tiles), dim3(256), 0, (hipStream_t)stream, a);
        else
            hipLaunchKernelGGL(adam_multi_kernel<false>, dim3((unsigned)tiles), dim3(256), 0, (hipStream_t)stream, a);
    }
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_adam_multi(int32_t n, const dtb_adam_param* params, float lr, float b1, float b2, float eps, int32_t t,
                       void* stream)
{
    return adam_multi(n, params, true, lr, b1, b2, eps, t, stream);
}

int dtb_mlp_refresh_bf16(int32_t n, const dtb_adam_param* params, void* stream)
{
    return adam_multi(n, params, false, 0.0f, 0.0f, 0.0f, 0.0f, 1, stream);
}

int dtb_gru_forward(int32_t B, int32_t H, const float* gi, const float* gh, const float* h, float* hn, void* hnb,
                    void* stream)
{
    DTB_REQUIRE(B > 0 && H > 0 && gi && gh && h && hn, "bad arguments");
    hipLaunchKernelGGL(gru_forward_kernel, g1((int64_t)B * H), dim3(256), 0, (hipStream_t)stream, B, H, gi, gh, h, hn,
                       (uint16_t*)hnb);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_gru_backward(int32_t B, int32_t H, const float* gi, const float* gh, const float* h, const float* dh_a,
                     const float* dh_b, const float* dh_c, float* dgi, void* dgib, float* dgh, void* dghb, float* dh_z,
                     void* stream)
{
    DTB_REQUIRE(B > 0 && H > 0 && gi && gh && h && dh_a && dgi && dgh && dh_z, "bad arguments");
    hipLaunchKernelGGL(gru_backward_kernel, g1((int64_t)B * H), dim3(256), 0, (hipStream_t)stream, B, H, gi, gh, h,
                       dh_a, dh_b, dh_c, dgi, (uint16_t*)dgib, dgh, (uint16_t*)dghb, dh_z);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}


int dtb_gru_sequence_fits(int32_t B, int32_t H)
{
    // the products must be ones that dtb_mlp_gemm_bf16_nt splits over K
    if (B > 0 && B % 32 == 0 && H > 0 && H % 32 == 0 && H <= 256 && !gemm_one_chain(B, 3 * H) && !gemm_one_chain(B, H))
        return DTB_OK;
    set_error("the sequence kernels take B and H multiples of 32, H <= 256 and products of fewer than 256 tiles");
    return DTB_UNSUPPORTED;
}

static int gru_lds(const void* kernel, int bytes)
{
    if (bytes > 0) DTB_TRY_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
    return DTB_OK;
}

int dtb_gru_sequence_forward(int32_t T, int32_t B, int32_t H, const float* gi, const void* w_hh, const float* b_hh,
                             const float* h0, int32_t h0_rows, float* gh, float* hs, void* hb, void* stream)
{
    DTB_TRY(dtb_gru_sequence_fits(B, H));
    DTB_REQUIRE(T > 0 && gi && w_hh && b_hh && gh && hs && hb && (!h0 || (h0_rows >= 0 && h0_rows <= B)), "bad arguments");
    DTB_REQUIRE((reinterpret_cast<uintptr_t>(w_hh) & 15) == 0, "W_hh must be 16-byte aligned");
    const dim3 g((unsigned)(B / kGruRows)), b(64 * kGruFwdWaves);
    const uint16_t* w = (const uint16_t*)w_hh;
    switch (H / 32) {
#define DTB_GRU_CASE(G)                                                                                              \
    case G:                                                                                                          \
        DTB_TRY(gru_lds((const void*)gru_seq_forward_kernel<G>, GruFwdWeights<G>::kLds));                \
        hipLaunchKernelGGL(gru_seq_forward_kernel<G>, g, b, (GruFwdWeights<G>::kLds),                   \
                           (hipStream_t)stream, T, B, gi, w, b_hh, h0, h0_rows, gh, hs, (uint16_t*)hb);               \
        break;
        DTB_GRU_CASE(1) DTB_GRU_CASE(2) DTB_GRU_CASE(3) DTB_GRU_CASE(4) DTB_GRU_CASE(5) DTB_GRU_CASE(6) DTB_GRU_CASE(7)
        DTB_GRU_CASE(8)
#undef DTB_GRU_CASE
    }
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_gru_sequence_backward(int32_t T, int32_t B, int32_t H, const float* gi, const float* gh, const float* hs,
                              const float* dho, const void* w_hh_t, void* dgib, void* dghb, float* dg, void* stream)
{
    DTB_TRY(dtb_gru_sequence_fits(B, H));
    DTB_REQUIRE(T > 0 && gi && gh && hs && dho && w_hh_t && dgib && dghb && dg, "bad arguments");
    DTB_REQUIRE((reinterpret_cast<uintptr_t>(w_hh_t) & 15) == 0, "the transpose of W_hh must be 16-byte aligned");
    const dim3 g((unsigned)(B / kGruRows)), b(64 * kGruBwdWaves);
    const uint16_t* w = (const uint16_t*)w_hh_t;
    switch (H / 32) {
#define DTB_GRU_CASE(G)                                                                                              \
    case G:                                                                                                          \
        DTB_TRY(gru_lds((const void*)gru_seq_backward_kernel<G>, GruBwdWeights<G>::kLds));           \
        hipLaunchKernelGGL(gru_seq_backward_kernel<G>, g, b, (GruBwdWeights<G>::kLds),               \
                           (hipStream_t)stream, T, B, gi, gh, hs, dho, w, (uint16_t*)dgib, (uint16_t*)dghb, dg);      \
        break;
        DTB_GRU_CASE(1) DTB_GRU_CASE(2) DTB_GRU_CASE(3) DTB_GRU_CASE(4) DTB_GRU_CASE(5) DTB_GRU_CASE(6) DTB_GRU_CASE(7)
        DTB_GRU_CASE(8)
#undef DTB_GRU_CASE
    }
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_sequence_loss(int32_t T, int32_t B, int32_t O, int32_t rows, int32_t n_out, const float* out,
                          const float* Y, const float* y_scale, const float* y_shift, const float* mask, float scale,
                          float* grad, void* gradb, float* lsum, void* stream)
{
    DTB_REQUIRE(T > 0 && B > 0 && O > 0 && rows >= 0 && rows <= B && n_out >= 0 && n_out <= O && out &&
                    (Y || rows == 0 || n_out == 0) && y_scale && y_shift && grad && gradb && lsum,
                "bad arguments");
    const int64_t n = (int64_t)T * B * O;
    hipLaunchKernelGGL(seq_loss_kernel, g1(n), dim3(256), 0, (hipStream_t)stream, n, B, O, rows, n_out, out, Y, y_scale,
                       y_shift, mask, scale, grad, (uint16_t*)gradb, lsum);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_pack_transposed(int32_t n, const dtb_pack_item* p, void* stream)
{
    DTB_REQUIRE(n >= 0 && n <= 2 * kMlpMaxLayers && (n == 0 || p), "at most %d matrices", 2 * kMlpMaxLayers);
    PackArgs a{};
    a.n = n;
    int64_t tiles = 0;
    for (int32_t i = 0; i < n; ++i) {
        DTB_REQUIRE(p[i].rows > 0 && p[i].cols > 0 && p[i].rows % 32 == 0 && p[i].cols % 32 == 0 &&
                        p[i].rows < (1ll << 30) && p[i].cols < (1 << 24) && p[i].ld >= p[i].cols && p[i].in &&
                        p[i].out && (reinterpret_cast<uintptr_t>(p[i].out) & 15) == 0,
                    "matrix %d: bad arguments", i);
        a.K[i] = (int32_t)p[i].rows; a.N[i] = (int32_t)p[i].cols; a.ld[i] = p[i].ld;
        a.in[i] = (const uint16_t*)p[i].in; a.out[i] = (uint16_t*)p[i].out;
        tiles += p[i].rows / 32 * (p[i].cols / 32);
        DTB_REQUIRE(tiles < (1ll << 31), "too many tiles for one launch");
        a.first[i + 1] = (int32_t)tiles;
    }
    if (tiles == 0) return DTB_OK;
    hipLaunchKernelGGL(pack_transposed_kernel, dim3((unsigned)tiles), dim3(256), 0, (hipStream_t)stream, a);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_column_sums(int32_t n, const dtb_colsum_item* p, int64_t rows, void* stream)
{
    DTB_REQUIRE(n >= 1 && n <= kMlpMaxLayers && p && rows >= 0, "1 to %d arrays", kMlpMaxLayers);
    ColsumArgs a{};
    a.n = n;
    a.rows = rows;
    int64_t wgs = 0;
    for (int32_t i = 0; i < n; ++i) {
        DTB_REQUIRE(p[i].cols > 0 && p[i].cols < (1 << 30) && p[i].ld >= p[i].cols && (p[i].src || rows == 0) && p[i].dst,
                    "array %d: bad arguments", i);
        a.cols[i] = (int32_t)p[i].cols; a.ld[i] = p[i].ld; a.src[i] = p[i].src;
        a.dst[i] = p[i].dst; a.dst2[i] = p[i].dst2;
        wgs += (p[i].cols + kBiasCols - 1) / kBiasCols;
        DTB_REQUIRE(wgs < (1ll << 31), "too many columns for one launch");
        a.first[i + 1] = (int32_t)wgs;
    }
    hipLaunchKernelGGL(colsum_kernel, dim3((unsigned)wgs), dim3(kBiasThreads), 0, (hipStream_t)stream, a);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_mlp_weight_gradients(int32_t n, const dtb_dw_item* p, int32_t rows, void* stream)
{
    DTB_REQUIRE(n >= 1 && n <= kMlpMaxLayers && p && rows > 0 && rows % 32 == 0, "1 to %d products over a multiple of 32 rows",
                kMlpMaxLayers);
    MlpDwArgs d{};
    d.layers = n;
    d.B = rows;
    int64_t tiles = 0;
    for (int32_t l = 0; l < n; ++l) {
        DTB_REQUIRE(p[l].n_in > 0 && p[l].n_out > 0 && p[l].n_in % 32 == 0 && p[l].n_out % 32 == 0 &&
                        p[l].n_in < (1 << 24) && p[l].n_out < (1 << 24) && p[l].h && p[l].g && p[l].dw &&
                        p[l].ldh >= rows && p[l].ldg >= rows && p[l].ldh % 32 == 0 && p[l].ldg % 32 == 0 &&
                        ((reinterpret_cast<uintptr_t>(p[l].h) | reinterpret_cast<uintptr_t>(p[l].g)) & 15) == 0 &&
                        (!p[l].db || (p[l].dbp && p[l].parts >= 0)),
                    "product %d: bad arguments", l);
        d.in[l] = (int32_t)p[l].n_in; d.out[l] = (int32_t)p[l].n_out;
        d.ldh[l] = p[l].ldh; d.ldg[l] = p[l].ldg; d.parts[l] = (int32_t)p[l].parts;
        d.hT[l] = (const uint16_t*)p[l].h; d.gT[l] = (const uint16_t*)p[l].g; d.dbp[l] = p[l].dbp;
        d.dW[l] = p[l].dw; d.db[l] = p[l].db;
        tiles += (p[l].n_out + 63) / 64 * ((p[l].n_in + 63) / 64);
        DTB_REQUIRE(tiles < (1ll << 31), "too many tiles for one launch");
        d.first[l + 1] = (int32_t)tiles;
    }
    hipLaunchKernelGGL(mlp_dw_kernel, dim3((unsigned)tiles), dim3(256), 0, (hipStream_t)stream, d);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

} // extern "C"
