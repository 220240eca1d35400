// Router and combine around the expert path (the reference runs them as precompiled Triton kernels `topk` and
// `combine`, glm-flash-rs src/moe.rs:89-100,171-181, whose source is not in its repository). Two gates (route.hpp):
// the benchmark's softmax (top-k by logit, ties: lower id, weights renormalised over the k picks) and GLM's
// sigmoid + bias selection with scaled renormalised weights; the shared expert is appended as the last slot with
// weight 1; combine = the slot-ordered weighted sum.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "route.hpp"

namespace gfr {

__global__ void __launch_bounds__(64) route_kernel(const float* __restrict__ logits, int E, int topk, int shared_id,
                                                   int* __restrict__ picks, float* __restrict__ weights, RouteGate g) {
    const int r = blockIdx.x, slots = topk + 1;
    route_token(logits + (size_t)r * E, E, topk, shared_id, picks + (size_t)r * slots, weights + (size_t)r * slots,
                g);
}

// out[r][n] = sum over slots s (in order) of weights[r][s] * (y[r * slots + s][n] for the EXL3 slots s < exl3_slots,
// shared[r * shared_stride + n] for the others when the caller gives the shared expert's output, else nothing) --
// the reference's combine(y, shared, weights, out), moe.rs:171-181. Four columns a thread (16-byte loads and
// stores); the slots in groups of 8, each group's rows in flight at once and added in slot order (a group's 8
// registers, not one per possible slot, keep the kernel at a few dozen VGPRs and many resident waves). D a multiple
// of 4.
__global__ void __launch_bounds__(256) combine_kernel(const float* __restrict__ y, const float* __restrict__ weights,
                                                      int slots, int exl3_slots, int D,
                                                      const float* __restrict__ shared, int shared_stride,
                                                      float* __restrict__ out) {
    typedef float f4v __attribute__((ext_vector_type(4)));
    constexpr int G = 8;
    const int r = blockIdx.y, n = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (n >= D) return;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s0 = 0; s0 < slots; s0 += G) {
        f4v v[G];
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const int s = s0 + j;
            if (s < slots) {
                if (s < exl3_slots)
                    v[j] = __builtin_nontemporal_load(reinterpret_cast<const f4v*>(y + ((size_t)r * slots + s) * D + n));
                else
                    v[j] = shared ? *reinterpret_cast<const f4v*>(shared + (size_t)r * shared_stride + n)
                                  : (f4v){0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const int s = s0 + j;
            if (s < slots && (s < exl3_slots || shared)) {
                const float w = weights[r * slots + s];
                acc.x += w * v[j].x;
                acc.y += w * v[j].y;
                acc.z += w * v[j].z;
                acc.w += w * v[j].w;
            }
        }
    }
    *reinterpret_cast<float4*>(out + (size_t)r * D + n) = acc;
}

// Router logits (the reference's router_part + router_sum, moe.rs:77-87; Triton, source absent): logits[r][e] =
// sum over k of x[r][k] * W[e][k], bf16 inputs, fp32 products and sums in a fixed order (v_dot2_f32_bf16 pairs in
// k order within a lane, then the 64 lanes in a fixed tree). Program (8 experts, up to RTMAX rows); wave w owns
// experts 8 b + w and 8 b + w + 4 and holds their weight chunks in registers while the program's rows stream past
// them (hidden sizes above 4096 reload the chunks a pass of 4096 a row).
typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
constexpr int ROUTER_RTMAX = 8;   // rows a program (the weight chunks are loaded once for them)
__global__ void __launch_bounds__(256) router_logits_kernel(const uint16_t* __restrict__ x, int x_stride,
                                                            const uint16_t* __restrict__ W, int D, int E, int rows,
                                                            int RT, float* __restrict__ logits) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    constexpr int CH = 8;                            // 16-byte chunks a lane a pass (4096 values a pass)
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int r0 = blockIdx.y * RT, r1 = r0 + RT < rows ? r0 + RT : rows;
    const int ex[2] = {(int)blockIdx.x * 8 + wave, (int)blockIdx.x * 8 + wave + 4};
    u32x4 w[2][CH];                                  // lane l: 8 weights at k = k0 + (c * 64 + l) * 8
    auto load_w = [&](int k0) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const int e = ex[q] < E ? ex[q] : E - 1;
                const int k = k0 + (c * 64 + lane) * 8;
                w[q][c] = k < D ? *reinterpret_cast<const u32x4*>(W + (size_t)e * D + k) : (u32x4){0, 0, 0, 0};
            }
    };
    const bool one_pass = D <= CH * 512;
    if (one_pass) load_w(0);
    for (int r = r0; r < r1; ++r) {
        float acc[2] = {0.f, 0.f};
        for (int k0 = 0; k0 < D; k0 += CH * 512) {
            if (!one_pass) load_w(k0);
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const int k = k0 + (c * 64 + lane) * 8;
                const u32x4 xv = k < D ? *reinterpret_cast<const u32x4*>(x + (size_t)r * x_stride + k) : (u32x4){0, 0, 0, 0};
                const uint32_t xs[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const uint32_t ws[4] = {w[q][c].x, w[q][c].y, w[q][c].z, w[q][c].w};
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[q] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf2_t, ws[j]),
                                                                __builtin_bit_cast(bf2_t, xs[j]), acc[q], false);
                }
            }
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            float v = acc[q];
            v += lane_xor_f<1>(v);
            v += lane_xor_f<2>(v);
            v += lane_xor_f<4>(v);
            v += lane_xor_f<8>(v);
            v += lane_xor_f<16>(v);
            v += lane_xor_f<32>(v);
            if (lane == 0 && ex[q] < E) logits[(size_t)r * E + ex[q]] = v;
        }
    }
}

// The same product on the matrix core, for windows of many rows: v_mfma_f32_16x16x32_bf16 with 16 experts as A and 16
// rows as B, fragments loaded straight from memory (a 64-k chunk a round: lane (row or expert l % 16, q = l / 16) holds
// k = 16 q .. 16 q + 15, 32 bytes; both operands take the chunk's k in that order, so each row's 128 bytes are one full
// line). A workgroup owns RB x EB tiles over the whole K: its 8 waves take contiguous eighths of the chunks, in chains
// of four MFMAs added in fp32, and the waves' sums meet in LDS in wave order in fp64 (error against fp64 7.7e-8 at
// hidden 4096, 8.3e-8 for the lanes' dot products; chains of 16 with an fp32 sum 1.4e-7). Bound by the operand reads from
// L2 (a row is read by E / (16 EB) workgroups, an expert by rows / (16 RB)), so the tiles are as large as the registers
// allow (RB x EB = 4 x 5: two sums of 80 and 72 of loads) and one round of workgroups covers the window. Measured against
// router_logits_kernel (us): 4096 rows, hidden 4096, 288 experts 202 -> 38; 8192 rows, hidden 5120, 160 experts 599 ->
// 48; 700 rows 60 -> 15. Error against fp64 at hidden 1024, 2048, 5120, 16384 and 65536: 6.5, 7.0, 7.9, 10.1 and 16.1e-8,
// 6.8, 7.4, 8.7, 12.3 and 24.6e-8 for the dot products.
//
// Which form a window runs: a wave of this kernel waits for a round of loads every 1024 k (hidden / 1024 rounds of about
// 2.5 us), while the dot products take one pass of 4096 k and grow with their programs (8 experts x 8 rows, four waves).
// Measured (us, dot products / matrix core):
//   one program a CU (rows x experts = 16384: 64 experts, 256 rows): hidden 1024 7.1 / 4.9, 1792 7.2 / 6.9, 2048 7.3 / 7.5,
//     3072 8.1 / 10.2, 4096 8.6 / 12.8, 5120 18.2 / 16.0, 6144 18.2 / 18.0, 8192 22.1 / 23.1, 16384 40.2 / 43.7
//   1.25 a CU (160 experts, 128 rows): 2048 8.5 / 7.6, 2560 8.9 / 9.1, 3072 9.3 / 10.2, 4096 9.9 / 12.8
//   two a CU (64 experts, 512 rows): 2048 8.5 / 7.5, 2560 9.0 / 9.1, 3072 9.5 / 10.2, 4096 11.2 / 12.7
//   2.5 a CU (160 experts, 256 rows): 4096 12.7 / 12.8; above that, and below 1792 at any count, the matrix core wins
// Above one program a CU the dot products win only at hidden sizes that are multiples of 512 (4088, 96 experts, 256 rows
// 10.0 / 8.8): there the 16 rows of a fragment lie a multiple of 1 KB apart, so that its loads likely meet in few of the
// L2's channels.
constexpr int ROUTER_MFMA_ROWS = 128;
static bool router_on_mfma(int rows, int E, int D) {
    if (rows < ROUTER_MFMA_ROWS) return false;
    const int64_t products = (int64_t)rows * E;
    if (products <= 16384) return D <= 1792 || (D > 4096 && D < 6144);
    return products > 32768 || D < 2560 || D > 4096 || D % 512;
}
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef float f4_t __attribute__((ext_vector_type(4)));
constexpr int ROUTER_WAVES = 8;
template <int RB, int EB>
__global__ void __launch_bounds__(64 * ROUTER_WAVES) router_mfma_kernel(const uint16_t* __restrict__ x, int x_stride,
                                                                        const uint16_t* __restrict__ W, int D, int E,
                                                                        int rows, float* __restrict__ logits) {
    constexpr int GT = RB * EB < 8 ? RB * EB : 8;          // tiles of a reduction round
    __shared__ f4_t part[ROUTER_WAVES][GT][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, a = lane & 15, q = lane >> 4;
    const int e0 = blockIdx.x * 16 * EB, r0 = blockIdx.y * 16 * RB;
    const int nc = (D + 63) / 64, c0 = wave * nc / ROUTER_WAVES, c1 = (wave + 1) * nc / ROUTER_WAVES;
    // rows and experts past the end repeat the last one (their results are not stored)
    const uint16_t *wp[EB], *xp[RB];
#pragma unroll
    for (int i = 0; i < EB; ++i) wp[i] = W + (size_t)min(e0 + 16 * i + a, E - 1) * D + 16 * q;
#pragma unroll
    for (int i = 0; i < RB; ++i) xp[i] = x + (size_t)min(r0 + 16 * i + a, rows - 1) * x_stride + 16 * q;
    f4_t sum[EB][RB];
#pragma unroll
    for (int i = 0; i < EB; ++i)
#pragma unroll
        for (int j = 0; j < RB; ++j) sum[i][j] = (f4_t){0.f, 0.f, 0.f, 0.f};
    for (int c = c0; c < c1; c += 2) {
        f4_t acc[EB][RB];
#pragma unroll
        for (int i = 0; i < EB; ++i)
#pragma unroll
            for (int j = 0; j < RB; ++j) acc[i][j] = (f4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int k = (c + u) * 64;
            auto load = [&](const uint16_t* p, bf8_t (&v)[2]) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    uint4 t = make_uint4(0u, 0u, 0u, 0u);
                    if (c + u < c1 && k + 16 * q + 8 * h < D) t = *reinterpret_cast<const uint4*>(p + k + 8 * h);
                    v[h] = __builtin_bit_cast(bf8_t, t);
                }
            };
            bf8_t wv[EB][2], xv[RB][2];
#pragma unroll
            for (int i = 0; i < EB; ++i) load(wp[i], wv[i]);
#pragma unroll
            for (int j = 0; j < RB; ++j) load(xp[j], xv[j]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < RB; ++j)
#pragma unroll
                    for (int i = 0; i < EB; ++i)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[i][h], xv[j][h], acc[i][j], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < EB; ++i)
#pragma unroll
            for (int j = 0; j < RB; ++j) sum[i][j] += acc[i][j];
    }
    // D holds experts 4 q .. 4 q + 3 of the tile for row a: the waves' sums in order, GT tiles a round
#pragma unroll
    for (int g = 0; g < RB * EB; g += GT) {
        if (g) __syncthreads();
#pragma unroll
        for (int t = 0; t < GT; ++t)
            if (g + t < RB * EB) part[wave][t][lane] = sum[(g + t) / RB][(g + t) % RB];
        __syncthreads();
        if (wave < GT && g + wave < RB * EB) {
            double d[4] = {0., 0., 0., 0.};
#pragma unroll
            for (int w = 0; w < ROUTER_WAVES; ++w) {
                const f4_t p = part[w][wave][lane];
#pragma unroll
                for (int j = 0; j < 4; ++j) d[j] += (double)p[j];
            }
            const f4_t v = {(float)d[0], (float)d[1], (float)d[2], (float)d[3]};
            const int e = e0 + (g + wave) / RB * 16 + 4 * q, r = r0 + (g + wave) % RB * 16 + a;
            if (r < rows) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (e + j < E) logits[(size_t)r * E + e + j] = v[j];
            }
        }
    }
}

}  // namespace gfr

#include "launch.hpp"

namespace gfr {

hipError_t launch_route(hipStream_t s, const float* logits, int rows, int E, int topk, int shared_id, int* picks,
                        float* weights, const float* bias, float scale) {
    route_kernel<<<rows, 64, 0, s>>>(logits, E, topk, shared_id, picks, weights, RouteGate{bias, scale});
    return hipGetLastError();
}

hipError_t launch_combine(hipStream_t s, const float* y, const float* weights, int rows, int slots, int exl3_slots,
                          int D, const float* shared, int shared_stride, float* out) {
    combine_kernel<<<dim3((D / 4 + 255) / 256, rows), 256, 0, s>>>(y, weights, slots, exl3_slots, D, shared,
                                                                   shared_stride, out);
    return hipGetLastError();
}

int router_logits_max_hidden() { return 1 << 16; }

hipError_t launch_router_logits(hipStream_t s, const uint16_t* x, int x_stride, const uint16_t* W, int D, int E,
                                int rows, float* logits) {
    if (router_on_mfma(rows, E, D)) {
        // the tile with the lowest estimate: rounds of one workgroup a CU, each as long as its operand reads (rows and
        // experts of a tile) plus a fixed part
        const auto wgs = [&](int rb, int eb) { return (rows + 16 * rb - 1) / (16 * rb) * ((E + 16 * eb - 1) / (16 * eb)); };
        const int tiles[5][2] = {{4, 5}, {4, 4}, {2, 4}, {2, 2}, {1, 2}};
        int best = 0, cost = 0;
        for (int t = 0; t < 5; ++t) {
            const int c = (wgs(tiles[t][0], tiles[t][1]) + 255) / 256 * (tiles[t][0] + tiles[t][1] + 4);
            if (t == 0 || c < cost) best = t, cost = c;
        }
        const auto go = [&](auto rb, auto eb) {
            constexpr int RB = decltype(rb)::value, EB = decltype(eb)::value;
            router_mfma_kernel<RB, EB><<<dim3((E + 16 * EB - 1) / (16 * EB), (rows + 16 * RB - 1) / (16 * RB)),
                                         64 * ROUTER_WAVES, 0, s>>>(x, x_stride, W, D, E, rows, logits);
            return hipGetLastError();
        };
        using std::integral_constant;
        switch (best) {
            case 0: return go(integral_constant<int, 4>{}, integral_constant<int, 5>{});
            case 1: return go(integral_constant<int, 4>{}, integral_constant<int, 4>{});
            case 2: return go(integral_constant<int, 2>{}, integral_constant<int, 4>{});
            case 3: return go(integral_constant<int, 2>{}, integral_constant<int, 2>{});
            default: return go(integral_constant<int, 1>{}, integral_constant<int, 2>{});
        }
    }
    const int RT = rows >= 64 ? ROUTER_RTMAX : rows >= 8 ? 4 : 1;
    router_logits_kernel<<<dim3((E + 7) / 8, (rows + RT - 1) / RT), 256, 0, s>>>(x, x_stride, W, D, E, rows, RT,
                                                                                  logits);
    return hipGetLastError();
}

}  // namespace gfr
