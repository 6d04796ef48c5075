// 32-bit matrix product on the matrix cores: out[m, n] (+)= sum_k a[m, k] * w[n, k] + bias[n] with both operands, every product and
// every sum in 32 bits (v_mfma_f32_16x16x4_f32: fused multiply-adds, no reduced mode).
//
// The order of a sum depends on K alone, never on the number of rows or on the kernel that takes them, so a row gives the same bits in
// any batch: runs of SEG columns are one chain of matrix instructions from zero, the runs of a group of GROUP columns are added in
// ascending order, and so are the groups (from zero, or from the old value of an accumulated output). A matrix instruction takes
// columns k, k + 4, k + 8 and k + 12 of 16 (a lane's operands of four instructions are then 16 consecutive bytes of a row). Short chains
// are also nearer to the exact sum than the one long chain of the plain kernel (gemm_generic.hip), which stays for what this path does
// not take: K or a row stride that is no multiple of 4, unaligned bases, 16-bit operands or results.
//
// gemm_f32_rows_kernel (up to 64 rows): the weights are read once and straight from memory into operand registers, a wave one run of
// SEG columns for 32 (or 16) rows of W, all of its 16 KB asked for before the first product; the eight waves of a block are the runs of
// a group, whose sums meet in LDS. Bound by the weights' stream where there are many of them (3,584 x 18,944 at one row: 50 us, 5.4 TB/s;
// the plain kernel 282), by launch and one trip to memory where there are few (896 x 4,864 at 8 rows: 15 us a call, the plain kernel's 28
// blocks 74).
//
// gemm_f32_tile_kernel (more rows): tiles of 128 x 128 (eight waves) or 64 x 64 (four), operands through two LDS stages of 32 columns (64 for the small tile,
// whose products of 32 columns take less time than a load), the
// next stage on its way in registers. A matrix instruction keeps its SIMD busy for 32 cycles and needs two fragments of 256 bytes, so
// neither LDS nor the caches bound it but the matrix cores (157 TFLOP/s; the plain kernel's multiply-adds peak at 79). 2,048 rows of
// 9,728 x 896: 105 TFLOP/s (339 us, plain 614); 700 rows 88 (139 us, plain 240; 456 tiles are 1.8 a CU); 700 rows of 896 x 4,864: 73
// (83 us with the sum of the groups, plain 353). Tiles of 64 x 64, and groups of K dealt over blockIdx.z, where the larger tiles would
// leave CUs without a block.
#include "common.h"
#include "gemm_internal.h"

typedef float floatx4 __attribute__((ext_vector_type(4)));

#define SEG 128
#define GROUP 1024
#define N_XCD 8
#define GROUP_M 8

// Where a sum goes: the output itself (F32_SET, F32_ACC) or a plane of partial sums per group.
#define F32_SET 0
#define F32_ACC 1
#define F32_PLANE 2

__device__ __forceinline__ float4 load4(const float* p, bool ok) {
    return ok ? *reinterpret_cast<const float4*>(p) : make_float4(0.f, 0.f, 0.f, 0.f);
}
__device__ __forceinline__ float part(const float4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// MT: tiles of 16 rows of a; NT: tiles of 16 rows of w that a block takes. One block per (column tiles, group of K).
template <int MT, int NT, int MODE>
__global__ __launch_bounds__(512) void gemm_f32_rows_kernel(const float* __restrict__ a, int lda, const float* __restrict__ w, int ldw,
                                                            const float* __restrict__ bias, float* __restrict__ out, int ldo, int M, int N,
                                                            int K) {
    constexpr int STEPS = SEG / 16, WAVES = GROUP / SEG, TILE = MT * NT * 256;
    __shared__ __attribute__((aligned(16))) float sums[WAVES][TILE];
    const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
    const int n0 = blockIdx.x * NT * 16, g0 = blockIdx.y * GROUP;
    const int k0 = g0 + wave * SEG + (lane >> 4) * 4;
    if (g0 + wave * SEG < K) {
        float4 wf[NT][STEPS];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int n = n0 + t * 16 + (lane & 15);
            const float* src = w + (size_t)(n < N ? n : N - 1) * ldw + k0;
#pragma unroll
            for (int s = 0; s < STEPS; s++) wf[t][s] = load4(src + s * 16, k0 + s * 16 < K);
        }
        floatx4 acc[MT][NT];
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int t = 0; t < NT; t++) acc[i][t] = floatx4{0.f, 0.f, 0.f, 0.f};
        // the rows' own values, two tiles of rows at a time (registers), all steps of them under way together
#pragma unroll
        for (int i0 = 0; i0 < MT; i0 += 2) {
            constexpr int PAIR = MT > 1 ? 2 : 1;
            float4 af[PAIR][STEPS];
#pragma unroll
            for (int i = 0; i < PAIR; i++) {
                const int m = (i0 + i) * 16 + (lane & 15);
                const float* src = a + (size_t)(m < M ? m : 0) * lda + k0;
#pragma unroll
                for (int s = 0; s < STEPS; s++) af[i][s] = load4(src + s * 16, m < M && k0 + s * 16 < K);
            }
#pragma unroll
            for (int s = 0; s < STEPS; s++)
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int i = 0; i < PAIR; i++)
#pragma unroll
                        for (int t = 0; t < NT; t++)
                            acc[i0 + i][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(part(af[i][s], e), part(wf[t][s], e), acc[i0 + i][t], 0, 0, 0);
        }
        // element r of a lane: row 4 (lane / 16) + r, column lane % 16 of its tile
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) sums[wave][((i * 16 + (lane >> 4) * 4 + r) * NT + t) * 16 + (lane & 15)] = acc[i][t][r];
    }
    __syncthreads();
    const int left = (K - g0 + SEG - 1) / SEG, runs = left < WAVES ? left : WAVES;
    for (int e = threadIdx.x; e < TILE; e += 512) {
        const int m = e / (NT * 16), n = n0 + e % (NT * 16);
        if (m >= M || n >= N) continue;
        float g = 0.f;
        for (int s = 0; s < runs; s++) g += sums[s][e];
        if (MODE == F32_PLANE) {
            out[((size_t)blockIdx.y * M + m) * N + n] = g;
        } else {
            float* dst = out + (size_t)m * ldo + n;
            float v = (MODE == F32_ACC ? *dst : 0.f) + g;
            if (bias) v += bias[n];
            *dst = v;
        }
    }
}

// BM x BN outputs by WM x WN waves. blockIdx.z: which groups of K (all of them: `groups` of one block; or, F32_PLANE,
// one each). A block that takes several groups adds them up in the output itself: it owns those outputs.
template <int BM, int BN, int WM, int WN, int BK, int MODE>
__global__ __launch_bounds__(WM * WN * WAVE) void gemm_f32_tile_kernel(const float* __restrict__ a, int lda, const float* __restrict__ w, int ldw,
                                                            const float* __restrict__ bias, float* __restrict__ out, int ldo, int M, int N,
                                                            int K, int tiles_m, int tiles_n) {
    constexpr int STRIDE = BK + 4;                            // 16 bytes of padding: sixteen rows' 16-byte reads hit different banks
    constexpr int FM = BM / WM / 16, FN = BN / WN / 16;       // tiles of 16 x 16 of a wave
    constexpr int LROWS = WM * WN * WAVE / (BK / 4);          // rows that the block's threads load at a time, 16 bytes each
    constexpr int A_LD = BM / LROWS, W_LD = BN / LROWS;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE, wm = wave / WN, wn = wave % WN;
    // blocks are dealt round-robin to the XCDs: undone, so that an XCD works on neighbouring tiles; eight rows of tiles at a time
    const int n_tiles = tiles_m * tiles_n;
    int pid = blockIdx.x;
    {
        const int per = n_tiles / N_XCD, rem = n_tiles % N_XCD, x = pid % N_XCD, q = pid / N_XCD;
        pid = x * per + (x < rem ? x : rem) + q;
    }
    const int in_group = GROUP_M * tiles_n, first_m = pid / in_group * GROUP_M;
    const int gsize = tiles_m - first_m < GROUP_M ? tiles_m - first_m : GROUP_M;
    const int m0 = (first_m + (pid % in_group) % gsize) * BM, n0 = (pid % in_group) / gsize * BN;
    const int kbeg = MODE == F32_PLANE ? blockIdx.z * GROUP : 0;
    const int kend = MODE == F32_PLANE && kbeg + GROUP < K ? kbeg + GROUP : K;

    const int lr = tid / (BK / 4), lk = (tid % (BK / 4)) * 4;               // this thread's row (of LROWS) and columns of a stage
    const float* ap[A_LD];
    const float* wp[W_LD];
#pragma unroll
    for (int i = 0; i < A_LD; i++) {
        const int m = m0 + i * LROWS + lr;
        ap[i] = a + (size_t)(m < M ? m : M - 1) * lda + lk;    // rows past the edge repeat the last one
    }
#pragma unroll
    for (int i = 0; i < W_LD; i++) {
        const int n = n0 + i * LROWS + lr;
        wp[i] = w + (size_t)(n < N ? n : N - 1) * ldw + lk;
    }
    float4 ra[A_LD], rw[W_LD];
    auto fetch = [&](int k) {
        const bool ok = k + lk < kend;
#pragma unroll
        for (int i = 0; i < A_LD; i++) ra[i] = load4(ap[i] + k, ok);
#pragma unroll
        for (int i = 0; i < W_LD; i++) rw[i] = load4(wp[i] + k, ok);
    };
    auto put = [&](int stage) {
        float* sa = lds + stage * (BM + BN) * STRIDE + lr * STRIDE + lk;
#pragma unroll
        for (int i = 0; i < A_LD; i++) *reinterpret_cast<float4*>(sa + i * LROWS * STRIDE) = ra[i];
#pragma unroll
        for (int i = 0; i < W_LD; i++) *reinterpret_cast<float4*>(sa + (BM + i * LROWS) * STRIDE) = rw[i];
    };
    floatx4 acc[FM][FN], sum[FM][FN];
    auto clear = [&](floatx4 (&v)[FM][FN]) {
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) v[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    };
    clear(acc);
    clear(sum);
    // a group's sum leaves: into its plane, or onto what the groups before it left in the output
    auto leave = [&](bool first, bool last) {
#pragma unroll
        for (int i = 0; i < FM; i++) {
#pragma unroll
            for (int j = 0; j < FN; j++) {
                const int n = n0 + (wn * FN + j) * 16 + (lane & 15);
                if (n >= N) continue;
                const float b = MODE != F32_PLANE && last && bias ? bias[n] : 0.f;
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int m = m0 + (wm * FM + i) * 16 + (lane >> 4) * 4 + r;
                    if (m >= M) continue;
                    if (MODE == F32_PLANE) {
                        out[((size_t)blockIdx.z * M + m) * N + n] = sum[i][j][r];
                    } else {
                        float* dst = out + (size_t)m * ldo + n;
                        float v = (MODE == F32_ACC || !first ? *dst : 0.f) + sum[i][j][r];
                        if (last && bias) v += b;
                        *dst = v;
                    }
                }
            }
        }
    };

    fetch(kbeg);
    put(0);
    if (kbeg + BK < kend) fetch(kbeg + BK);
    __syncthreads();
    int stage = 0;
    for (int k = kbeg; k < kend; k += BK, stage ^= 1) {
        const float* sa = lds + stage * (BM + BN) * STRIDE + (wm * FM * 16 + (lane & 15)) * STRIDE + (lane >> 4) * 4;
        const float* sw = lds + stage * (BM + BN) * STRIDE + (BM + wn * FN * 16 + (lane & 15)) * STRIDE + (lane >> 4) * 4;
#pragma unroll
        for (int s = 0; s < BK; s += 16) {
            float4 fa[FM], fw[FN];
#pragma unroll
            for (int i = 0; i < FM; i++) fa[i] = *reinterpret_cast<const float4*>(sa + i * 16 * STRIDE + s);
#pragma unroll
            for (int j = 0; j < FN; j++) fw[j] = *reinterpret_cast<const float4*>(sw + j * 16 * STRIDE + s);
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int i = 0; i < FM; i++)
#pragma unroll
                    for (int j = 0; j < FN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(part(fa[i], e), part(fw[j], e), acc[i][j], 0, 0, 0);
        }
        if (k + BK < kend) put(stage ^ 1);                    // (the stage before was left at the barrier)
        if (k + 2 * BK < kend) fetch(k + 2 * BK);
        const int done = k + BK;
        if (done % SEG == 0 || done >= kend) {                // the end of a run
#pragma unroll
            for (int i = 0; i < FM; i++)
#pragma unroll
                for (int j = 0; j < FN; j++) sum[i][j] += acc[i][j];
            clear(acc);
        }
        if (MODE != F32_PLANE && done % GROUP == 0 && done < kend) {
            leave(done == GROUP, false);
            clear(sum);
        }
        __syncthreads();
    }
    leave(K <= GROUP, true);
}

bool gemm_f32_supports(const GemmArgs& g) {
    return g.a_dtype == HFA_F32 && g.w_dtype == HFA_F32 && g.out_dtype == HFA_F32 && g.K % 4 == 0 && g.lda % 4 == 0 && g.ldw % 4 == 0 &&
           ((uintptr_t)g.a & 15) == 0 && ((uintptr_t)g.w & 15) == 0;
}

template <int MT, int NT>
static void launch_rows(const GemmArgs& g, int mode, float* out, int groups) {
    const dim3 grid((g.N + NT * 16 - 1) / (NT * 16), groups);
    const float *a = (const float*)g.a, *w = (const float*)g.w;
    if (mode == F32_PLANE)
        gemm_f32_rows_kernel<MT, NT, F32_PLANE><<<grid, 512, 0, g.stream>>>(a, g.lda, w, g.ldw, g.bias, out, g.ldo, g.M, g.N, g.K);
    else if (mode == F32_ACC)
        gemm_f32_rows_kernel<MT, NT, F32_ACC><<<grid, 512, 0, g.stream>>>(a, g.lda, w, g.ldw, g.bias, out, g.ldo, g.M, g.N, g.K);
    else
        gemm_f32_rows_kernel<MT, NT, F32_SET><<<grid, 512, 0, g.stream>>>(a, g.lda, w, g.ldw, g.bias, out, g.ldo, g.M, g.N, g.K);
}

template <int BM, int BN, int WM, int WN, int BK>
static void launch_tiles(const GemmArgs& g, int mode, float* out, int groups) {
    const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
    const size_t smem = 2 * (BM + BN) * (BK + 4) * sizeof(float);
    const float *a = (const float*)g.a, *w = (const float*)g.w;
    const dim3 grid((unsigned)(tiles_m * tiles_n), 1, mode == F32_PLANE ? groups : 1);
    if (mode == F32_PLANE)
        gemm_f32_tile_kernel<BM, BN, WM, WN, BK, F32_PLANE><<<grid, WM * WN * WAVE, smem, g.stream>>>(a, g.lda, w, g.ldw, g.bias, out, g.ldo, g.M, g.N, g.K, tiles_m, tiles_n);
    else if (mode == F32_ACC)
        gemm_f32_tile_kernel<BM, BN, WM, WN, BK, F32_ACC><<<grid, WM * WN * WAVE, smem, g.stream>>>(a, g.lda, w, g.ldw, g.bias, out, g.ldo, g.M, g.N, g.K, tiles_m, tiles_n);
    else
        gemm_f32_tile_kernel<BM, BN, WM, WN, BK, F32_SET><<<grid, WM * WN * WAVE, smem, g.stream>>>(a, g.lda, w, g.ldw, g.bias, out, g.ldo, g.M, g.N, g.K, tiles_m, tiles_n);
}

template <int BM, int BN, int WM, int WN, int BK>
static int reserve_lds() {
    const int smem = 2 * (BM + BN) * (BK + 4) * (int)sizeof(float);
    const void* kernels[3] = {(const void*)gemm_f32_tile_kernel<BM, BN, WM, WN, BK, F32_SET>, (const void*)gemm_f32_tile_kernel<BM, BN, WM, WN, BK, F32_ACC>,
                              (const void*)gemm_f32_tile_kernel<BM, BN, WM, WN, BK, F32_PLANE>};
    for (const void* k : kernels) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
        if (e != hipSuccess) {
            hfa_set_error("gemm_f32: cannot reserve %d bytes of LDS: %s", smem, hipGetErrorString(e));
            return 2;
        }
    }
    return 0;
}

int gemm_f32_launch(const GemmArgs& g, void* workspace, size_t workspace_bytes, int defer, int* pending_splits) {
    static const int reserved = reserve_lds<128, 128, 2, 4, 32>() | reserve_lds<64, 64, 2, 2, 64>();
    if (reserved) return 2;
    const int groups = (g.K + GROUP - 1) / GROUP;
    const bool planes_fit = workspace != nullptr && groups > 1 && groups <= 65535 && (size_t)groups * g.M * g.N * sizeof(float) <= workspace_bytes;
    int mode = g.accumulate ? F32_ACC : F32_SET;
    float* out = (float*)g.out;
    const long tiles64 = (long)((g.M + 63) / 64) * ((g.N + 63) / 64), tiles128 = (long)((g.M + 127) / 128) * ((g.N + 127) / 128);
    if (g.M <= 64 && (groups == 1 || planes_fit)) {
        if (groups > 1) {
            mode = F32_PLANE;
            out = (float*)workspace;
        }
        // two tiles of columns a block (the rows' values are fetched half as often) where that still gives every CU a block
        const bool wide = (long)((g.N + 31) / 32) * groups >= 256;
        if (g.M <= 16) wide ? launch_rows<1, 2>(g, mode, out, groups) : launch_rows<1, 1>(g, mode, out, groups);
        else if (g.M <= 32) wide ? launch_rows<2, 2>(g, mode, out, groups) : launch_rows<2, 1>(g, mode, out, groups);
        else wide ? launch_rows<4, 2>(g, mode, out, groups) : launch_rows<4, 1>(g, mode, out, groups);
    } else {
        HFA_REQUIRE(tiles64 <= 0x7fffffffL, "gemm: an output of %d x %d is beyond the grid", g.M, g.N);
        // 512 blocks of 64 x 64 are two a CU; fewer, and the groups of K become blocks of their own
        if (tiles128 < 256 && tiles64 < 512 && planes_fit) {
            mode = F32_PLANE;
            out = (float*)workspace;
        }
        if (tiles128 >= 256) launch_tiles<128, 128, 2, 4, 32>(g, mode, out, groups);
        else launch_tiles<64, 64, 2, 2, 64>(g, mode, out, groups);
    }
    HFA_LAUNCH_CHECK("gemm_f32");
    if (mode != F32_PLANE) return 0;
    if (defer && pending_splits) {
        *pending_splits = groups;
        return 0;
    }
    return gemm_finish_launch((const float*)workspace, groups, g.bias, g.out, gemm_mode_of(g), g.ldo, g.M, g.N, g.stream);
}
