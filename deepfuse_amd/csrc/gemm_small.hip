// gemm_small.hip -- the fp8 NT GEMM on 16x16 or 32x32 tiles whose waves
// share the reduction: C[M, N] = A[M, K] . B[N, K]^T * sa * sb + bias.
//
// For outputs too small for the persistent kernel's 256-row tiles: few rows (a
// decode batch), or a few hundred rows and columns.  There a 256x128 tile
// leaves most CUs without work, and one tile's chain -- first operand step,
// K steps behind one barrier each, epilogue -- is the launch's time.  What
// bounds such a call is latency, then the rate at which a CU takes in operand
// bytes.
//
// So a block owns a 16*MT x 16*NT tile, and its W waves take the 128-byte K
// steps in turn, each wave the whole tile of its steps: no wave waits for
// another before the end, and up to W*U steps of operands are on their way at
// once (K = 768 is six steps: all of it).  The waves' partial tiles meet in
// LDS and are added in wave order, so the result does not depend on timing.
// No second launch adds K slices up.  Measured, against the persistent
// kernel's tiles (us a call; bf16 output):
//       8 x 1600, K = 1600    3.3  against 16.4    8 x 6400, K = 1600   4.8  against 17.3
//       8 x 1600, K = 6400    6.1  against 20.6   64 x 3072, K = 768    3.5  against  7.3
//     512 x 768,  K = 768     4.3  against  7.7  512 x 768,  K = 3072   7.5  against 22.6
//    1000 x 771,  K = 1037    8.6  against 14.5  768 x 768,  K = 8192  20.6  against 30.8
//
// Operand path: each load instruction takes 8 rows x 128 bytes, whole cache
// lines, into registers; a wave-private LDS slab turns them into MFMA
// fragments (16 rows, 32 bytes per lane).  Loading the fragments straight from
// memory needs no LDS but puts 16 rows into every 16 lanes, and the CU then
// took in about 14 bytes a cycle.
// Rows past M or N and K chunks past K lie outside the buffer ranges and read
// as zero.
//
// Replaces fully_connected_forward_kernel, fc_backward_input and
// fc_backward_weights (dnn/layers/fully_connected_layer.cu:14-89) at these
// sizes.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "df_common.hpp"
#include "gemm_common.hpp"

namespace dfk {

template <int FA, int FB, int MT, int NT, int W, int U>
__global__ __launch_bounds__(64 * W) void gemm_small_kernel(
    const uint8_t* __restrict__ A, int lda, const uint8_t* __restrict__ B, int ldb, int M, int N, int K,
    const float* __restrict__ sa, const float* __restrict__ sb, int bias_dtype, const void* __restrict__ bias,
    int c_dtype, void* __restrict__ C, int ldc, int vec_out) {
    constexpr int ROWS = 16 * MT, COLS = 16 * NT;
    constexpr int NL = 2 * (MT + NT);              // loads of 8 rows x 128 bytes per step
    constexpr int SLAB = NL * 1024;                // a wave's step: A rows, then B rows
    constexpr int RSTR = COLS + 4;                 // row of a partial tile (floats)
    constexpr int RED = ROWS * RSTR * 4;
    constexpr uint32_t kOOB = 0x80000000u;
    // slabs during the reduction over K, partial tiles after it
    __shared__ __attribute__((aligned(1024))) uint8_t lds[W * (SLAB > RED ? SLAB : RED)];
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tiles_n = (N + COLS - 1) / COLS;
    const int m0 = (int)(blockIdx.x / tiles_n) * ROWS, n0 = (int)(blockIdx.x % tiles_n) * COLS;
    const __amdgpu_buffer_rsrc_t rA = __builtin_amdgcn_make_buffer_rsrc((void*)A, (short)0, M * lda, 0x00020000);
    const __amdgpu_buffer_rsrc_t rB = __builtin_amdgcn_make_buffer_rsrc((void*)B, (short)0, N * ldb, 0x00020000);
    const int nk = (K + 127) >> 7;

    // loads: lane l takes 16-byte chunk l%8 of row l/8 of each 8-row group
    const int lr = lane >> 3, lc = (lane & 7) * 16;
    const uint32_t oa = (uint32_t)(m0 + lr) * (uint32_t)lda + (uint32_t)lc;
    const uint32_t ob = (uint32_t)(n0 + lr) * (uint32_t)ldb + (uint32_t)lc;
    u32x4 buf[U][NL];
    auto load = [&](u32x4* b, int s) {
        const int k = s * 128;  // past the last step: every chunk out of range
        const bool in = k + lc < K;
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i)
            b[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                rA, in ? oa + (uint32_t)(8 * i) * (uint32_t)lda + (uint32_t)k : kOOB, 0, 0));
#pragma unroll
        for (int i = 0; i < 2 * NT; ++i)
            b[2 * MT + i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                rB, in ? ob + (uint32_t)(8 * i) * (uint32_t)ldb + (uint32_t)k : kOOB, 0, 0));
    };
    // slab: rows of 128 bytes, 16-byte chunk c of row r in slot c ^ (r/2 % 8):
    // the 16 rows of a fragment read spread over all banks
    uint8_t* const slab = lds + w * SLAB;
    const int wr_even = lr * 128 + (((lane & 7) ^ (lr >> 1)) << 4);
    const int wr_odd = wr_even ^ 64;  // rows 8..15 of a 16-row fragment: r/2 % 8 is 4 more
    const int fr = lane & 15, fq = (lane >> 4) * 2, fs = (fr >> 1) & 7;
    const int rd0 = fr * 128 + ((fq ^ fs) << 4), rd1 = fr * 128 + (((fq + 1) ^ fs) << 4);

    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

    // The lanes of a wave hand chunks to each other through the slab.  Its LDS
    // operations execute in order, so no instruction is needed, but the compiler
    // must not move one lane's reads above its writes, nor the next step's writes
    // above the reads.  A fragment's reads follow its own two writes: with one
    // meeting after all of a step's writes 64 x 1600, K = 6400 took 8.2 us against
    // 7.85, 768 x 768, K = 8192 21.3 against 20.4.
    auto lanes_meet = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    };
    // fragment t (16 rows) of a step in registers, through its part of the slab
    auto frag = [&](const u32x4* b, int t) -> v8i {
        *reinterpret_cast<u32x4*>(slab + t * 2048 + wr_even) = b[2 * t];
        *reinterpret_cast<u32x4*>(slab + t * 2048 + 1024 + wr_odd) = b[2 * t + 1];
        lanes_meet();
        const u32x4 lo = *reinterpret_cast<const u32x4*>(slab + t * 2048 + rd0);
        const u32x4 hi = *reinterpret_cast<const u32x4*>(slab + t * 2048 + rd1);
        v8i f;
        f[0] = (int)lo.x; f[1] = (int)lo.y; f[2] = (int)lo.z; f[3] = (int)lo.w;
        f[4] = (int)hi.x; f[5] = (int)hi.y; f[6] = (int)hi.z; f[7] = (int)hi.w;
        return f;
    };
    // one step: MT x NT products
    auto step = [&](const u32x4* b) {
        lanes_meet();  // the step before has read the slab
        v8i fb[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j) fb[j] = frag(b, MT + j);
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const v8i fa = frag(b, i);
#pragma unroll
            for (int j = 0; j < NT; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[j], fa, acc[i][j], FB, FA, 0, 0, 0, 0);
        }
    };
#pragma unroll
    for (int u = 0; u < U; ++u) load(buf[u], w + u * W);
    for (int s = w; s < nk; s += W * U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s + u * W < nk) step(buf[u]);
            load(buf[u], s + (u + U) * W);
        }
    }
    // B in the first operand slot: the accumulator is C^T, lane l holds row
    // l%16 and columns 4*(l/16) .. +4.  Every wave is done with its slab
    // before partial tiles go over them.
    __syncthreads();
    float* const red = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
            *reinterpret_cast<v4f*>(red + (w * ROWS + 16 * i + fr) * RSTR + 16 * j + 4 * (lane >> 4)) = acc[i][j];
    __syncthreads();
    const float sab = sa[0] * sb[0];
    for (int e = threadIdx.x; e < ROWS * COLS / 4; e += 64 * W) {
        const int r = e / (COLS / 4), c = (e % (COLS / 4)) * 4, row = m0 + r, col = n0 + c;
        if (row >= M || col >= N) continue;
        v4f t = *reinterpret_cast<const v4f*>(red + r * RSTR + c);
#pragma unroll
        for (int v = 1; v < W; ++v) t += *reinterpret_cast<const v4f*>(red + (v * ROWS + r) * RSTR + c);
        float o[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            float b = 0.0f;
            if (bias && col + x < N) {
                if (bias_dtype == DF_DTYPE_FLOAT32) b = bias_ld(static_cast<const float*>(bias), col + x);
                else if (bias_dtype == DF_DTYPE_HALF) b = bias_ld(static_cast<const f16_t*>(bias), col + x);
                else b = bias_ld(static_cast<const uint16_t*>(bias), col + x);
            }
            o[x] = t[x] * sab + b;
        }
        auto put = [&](auto* p) {
            using T = typename std::remove_reference<decltype(*p)>::type;
            if (vec_out && col + 3 < N) {
                store4(p, o);
            } else {
#pragma unroll
                for (int x = 0; x < 4; ++x)
                    if (col + x < N) p[x] = OutCvt<T>::cvt(o[x]);
            }
        };
        const int64_t at = (int64_t)row * ldc + col;
        if (c_dtype == DF_DTYPE_FLOAT32) put(static_cast<float*>(C) + at);
        else if (c_dtype == DF_DTYPE_HALF) put(static_cast<f16_t*>(C) + at);
        else put(static_cast<uint16_t*>(C) + at);
    }
}

// The best tiling of one GEMM and its modelled time.  Measured (MI355X, bf16
// output, 50 calls in a graph over 8 weight copies): a launch takes a latency
// part -- 2.5 us plus the chain of a wave's K steps -- and, per block and CU, a
// fixed part (partial tiles, output) plus the K steps' operand bytes:
//   16x16 tiles, 4 waves: 2.5 + 0.06 nk + (blocks / CUs) * (0.75 + 0.031 nk) us
//   32x32 tiles:          2.6 + 0.11 nk + (blocks / CUs) * (0.75 + 0.080 nk) us
// within 10-15% from 8 to 2048 rows, K = 512 to 6400.  Longer reductions stream
// operand panels that no L2 holds, and 16x16 tiles, which take in twice the bytes
// of 32x32 ones, then cost more a step: 0.045 nk (102 x 1808, K = 12112: 31.8 us on
// 16x16 tiles, 19.6 on 32x32, 28.3 on the persistent kernel's).  16x32, 32x64 and 64x64
// tiles were measured too and were nowhere faster by more than 5%: their
// blocks are too few where the latency counts, and where bytes count the
// persistent kernel is ahead.  32x32 tiles run eight waves instead of four
// where the blocks do not fill the CUs anyway and a wave of four would have
// more than one round of steps.  Eight / four waves, us: 128 x 1600, K = 6400
// (200 blocks, 50 steps) 10.3 / 11.1; 96 x 1600, K = 6400 8.7 / 9.7; 128 x 1600,
// K = 1600 (13 steps) 5.40 / 5.46; near a full chip at 24 steps four are a
// little ahead (512 x 512, K = 3072, 256 blocks: 5.43 / 5.26), and past it
// clearly (512 x 768, K = 3072, 384 blocks: 8.6 / 7.2).
SmallPlan small_plan(int M, int N, int K, int cus) {
    const double nk = (K + 127) / 128;
    const double b16 = (double)((M + 15) / 16) * ((N + 15) / 16), b32 = (double)((M + 31) / 32) * ((N + 31) / 32);
    const double t16 = 2.5 + 0.06 * nk + b16 / cus * (0.75 + (nk > 50 ? 0.045 : 0.031) * nk);
    const double t32 = 2.6 + 0.11 * nk + b32 / cus * (0.75 + 0.080 * nk);
    if (t16 < t32) return SmallPlan{1, 1, 4, t16 / kStepUs};
    return SmallPlan{2, 2, b32 <= cus && nk > 8 ? 8 : 4, t32 / kStepUs};
}

template <int FA, int FB>
static void launch_formats(const SmallPlan& p, int bias_dtype, int c_dtype, const GemmArgs& g) {
    const int esz = c_dtype == DF_DTYPE_FLOAT32 ? 4 : 2;
    const int vec_out = ((int64_t)g.ldc * esz) % 16 == 0 && aligned16(g.C);
    const int grid = ((g.N + 16 * p.nt - 1) / (16 * p.nt)) * ((g.M + 16 * p.mt - 1) / (16 * p.mt));
#define DF_SMALL(MT, NT, W, U)                                                                                       \
    if (p.mt == MT && p.nt == NT && p.waves == W) {                                                                  \
        gemm_small_kernel<FA, FB, MT, NT, W, U><<<grid, 64 * W, 0, g.st>>>(                                          \
            g.A, g.lda, g.B, g.ldb, g.M, g.N, g.K, g.sa, g.sb, bias_dtype, g.bias, c_dtype, g.C, g.ldc, vec_out);    \
        return;                                                                                                      \
    }
    DF_SMALL(1, 1, 4, 4)
    DF_SMALL(2, 2, 4, 2)
    DF_SMALL(2, 2, 8, 2)
#undef DF_SMALL
}

void launch_small(const SmallPlan& p, int fmt_a, int fmt_b, int bias_dtype, int c_dtype, const GemmArgs& g) {
    if (fmt_a == E4M3 && fmt_b == E4M3) launch_formats<E4M3, E4M3>(p, bias_dtype, c_dtype, g);
    else if (fmt_a == E5M2 && fmt_b == E4M3) launch_formats<E5M2, E4M3>(p, bias_dtype, c_dtype, g);
    else if (fmt_a == E4M3 && fmt_b == E5M2) launch_formats<E4M3, E5M2>(p, bias_dtype, c_dtype, g);
    else launch_formats<E5M2, E5M2>(p, bias_dtype, c_dtype, g);
}

}  // namespace dfk
