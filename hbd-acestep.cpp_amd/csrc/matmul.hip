// ggml_mul_mat(w, x) with Q8_0 weights and F32 activations, the way ggml-cpu
// computes it: each row of x is quantized to Q8_0 (the x86 from_float:
// id = 127 / amax, round to nearest even, saturate), and each output is
// sum over blocks b of (d_w[b] * d_x[b]) * sum_i q_w[i] q_x[i] -- an exact int32
// dot per block, scaled in fp32 (ggml_vec_dot_q8_0_q8_0).
// Reference call sites: qwen3_linear (qwen3-enc.h:86-88) for the Q/K/V, O,
// gate/up and down projections, dit_ggml_linear (dit-graph.h:36-49), and the
// LM head over the Q8_0 token table (qwen3-lm.h:755).
//
// Weights are repacked once, at load, into the "R64" layout (lossless: the same
// 34 bytes per block): rows in groups of 64 (the last group zero-padded), and per
// (group g, block b) the 32 quants of the 64 rows as two 1 KB halves -- half j,
// lane l holds bytes [16 j, 16 j + 16) of row 64 g + l's block -- followed, after
// all quants, by the scales d[g][b][l] (fp16). A wave with lane = row then reads
// every quant byte with fully coalesced 16-byte loads.
//
// Matrix-vector kernel (up to 8 rows of x, the batched decode shapes): one wave
// per (row group, key split); lanes are weight rows, the quantized x is uniform
// across the wave and read through the scalar cache; sdot4 per 4 quants. Up to
// 8 key splits of a row group share a workgroup and are added in LDS in wave
// order; with more, each workgroup writes its partial sums and a small kernel
// adds them in workgroup order, so the result does not depend on scheduling. One row
// of x can run as one launch instead of the quantization, the product and that sum.
//
// Matrix kernels (more than 8 rows): int8 MFMAs for the block dots, the scales applied
// to every block. 128 x 128 outputs per workgroup with operands from global memory and,
// on idle grids, key splits through memory; or 64 x 64 with the keys split over four wave
// groups of the workgroup and operands through LDS. rules.h says which call takes which.
#include "common.h"
#include "launch.h"
#include "rules.h"

namespace mi {

__global__ void __launch_bounds__(256) k_q8_0_repack(const char * src, int64_t nb1, uint32_t n, uint32_t nbk,
                                                     uint32_t ng, char * dst) {
    const uint64_t i     = (uint64_t) blockIdx.x * 256u + threadIdx.x;  // ((g * nbk + b) * 64 + l)
    const uint64_t total = (uint64_t) ng * nbk * 64;
    if (i >= total) {
        return;
    }
    const uint32_t l   = (uint32_t) (i % 64);
    const uint64_t gb  = i / 64;
    const uint32_t b   = (uint32_t) (gb % nbk);
    const uint32_t row = (uint32_t) (gb / nbk) * 64 + l;
    uint32_t       q[8] = { 0, 0, 0, 0, 0, 0, 0, 0 };
    uint16_t       d    = 0;
    if (row < n) {
        const uint16_t * p = (const uint16_t *) (src + (int64_t) row * nb1 + (int64_t) b * 34);
        d                  = p[0];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            q[k] = (uint32_t) p[1 + 2 * k] | ((uint32_t) p[2 + 2 * k] << 16);
        }
    }
    char * qd = dst + gb * 2048 + 16 * l;
    *(uint4 *) qd          = make_uint4(q[0], q[1], q[2], q[3]);
    *(uint4 *) (qd + 1024) = make_uint4(q[4], q[5], q[6], q[7]);
    *(uint16_t *) (dst + (uint64_t) ng * nbk * 2048 + i * 2) = d;
}

// d = amax / 127, the IEEE quotient (q0 = amax * (1/127) corrected by one fma)
__device__ __forceinline__ float mm_div127(float amax) {
    constexpr float C  = 1.0f / 127.0f;
    const float     q0 = amax * C;
    const float     r  = __builtin_fmaf(-q0, 127.0f, amax);
    return __builtin_fmaf(r, C, q0);
}

// x rows -> Q8_0 (x86 rounding), block-major: quants xq[b][m][32] and widened
// scales xd[b][m] at a row stride mp >= m (the matrix-vector kernel reads all
// rows of a block in one 32 * m + 4 * m byte run with a few wide scalar loads;
// the matrix kernel reads 32-row tiles); 8 lanes per 32-element block, and the
// blocks of a wave are one block of 8 consecutive rows: each row's 128 input
// bytes are a whole line, and the wave's quants one contiguous 256-byte run.
#ifndef MI_QX_U
#define MI_QX_U 4  // blocks per 8-lane group, a grid stride apart, all loads issued first
#endif
__global__ void __launch_bounds__(256) k_mmv_quant_x(const MmvArgs a) {
    constexpr int  U     = MI_QX_U;
    const uint32_t gid   = blockIdx.x * 256u + threadIdx.x;
    const uint32_t grp   = gid / 8, sub = gid % 8;
    const uint32_t total = a.m * a.nbk;
    const uint32_t ngrp  = gridDim.x * 32u;  // 8-lane groups in the grid
    auto           ld4   = [&](const char * p, float (&v)[4]) {
        if (a.xvec) {
            const float4 q = *(const float4 *) p;
            v[0]           = q.x;
            v[1]           = q.y;
            v[2]           = q.z;
            v[3]           = q.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = ((const float *) p)[e];
            }
        }
    };
    // the U blocks' inputs (g and u for the SwiGLU prologue), all in flight at once
    float f[U][4], h[U][4];
#pragma unroll
    for (int k = 0; k < U; ++k) {
        const uint32_t blk = grp + (uint32_t) k * ngrp;
        if (blk < total) {  // uniform over the 8 lanes of a block
            const uint32_t b = blk / a.m, m = blk - b * a.m;
            if (a.glu) {
                const int64_t off = (int64_t) m * a.gu1 + (int64_t) (b * 32 + sub * 4) * 4;
                ld4(a.g + off, f[k]);
                ld4(a.u + off, h[k]);
            } else {
                ld4(a.x + (int64_t) m * a.x1 + (int64_t) (b * 32 + sub * 4) * 4, f[k]);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
        const uint32_t blk = grp + (uint32_t) k * ngrp;
        if (blk >= total) {
            break;  // whole groups of 8 lanes; later blocks are further out
        }
        const uint32_t b = blk / a.m, m = blk - b * a.m;
        float          x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            x[e] = a.glu ? silu_f(f[k][e]) * h[k][e] : f[k][e];  // x = silu(g) * u, as mi_swiglu computes it
        }
        float amax = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
        amax       = group_max<8>(amax);
        const float d  = mm_div127(amax);
        const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
        uint32_t    w  = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float q = __builtin_amdgcn_fmed3f(__builtin_rintf(x[e] * id), -128.0f, 127.0f);
            w |= ((uint32_t) (int32_t) q & 0xffu) << (8 * e);
        }
        *(uint32_t *) (a.xq + ((int64_t) b * a.mp + m) * 32 + sub * 4) = w;
        if (sub == 0) {
            a.xd[(int64_t) b * a.mp + m] = (float) __builtin_bit_cast(_Float16, f32_to_f16_bits(d));
        }
    }
}

// RMSNorm*w and the quantization of x in one kernel (the norm -> product
// prologue), one workgroup per row: the scale from the double sum of the float
// squares and x' = (x * scale) * w, the arithmetic of mi_rms_norm on F32 rows
// (only the order of the double additions differs, which leaves the float mean
// unchanged short of a double rounding tie); then x' is quantized as
// k_mmv_quant_x does, 8 lanes per 32-element block. With an addend (a.ab), x is
// the residual sum a.x + a.ab, written to a.sum in the first pass (the
// arithmetic of mi_add_rms_norm) and formed again from the two inputs in the
// second. With a gate (a.gate) the addend is scaled first, x + ab * gate (the
// arithmetic of mi_add_rms_norm's gated form); with a modulate (a.msc, a.msh)
// the normalized rows become (x' * (msc + 1)) + msh, each step rounded as
// mi_rms_norm_modulate rounds it.
__global__ void __launch_bounds__(256) k_mmv_quant_x_norm(const MmvArgs a) {
    __shared__ double red[4];
    __shared__ float  scl;
    const uint32_t m   = blockIdx.x;
    const int      tid = threadIdx.x;
    const char *   xr  = a.x + (int64_t) m * a.x1;
    auto           ld4 = [&](const char * p, float (&v)[4]) {
        if (a.xvec) {
            const float4 q = *(const float4 *) p;
            v[0]           = q.x;
            v[1]           = q.y;
            v[2]           = q.z;
            v[3]           = q.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = ((const float *) p)[e];
            }
        }
    };
    const char * br = a.ab ? a.ab + (int64_t) m * a.ab1 : nullptr;
    // x (or the residual sum) at element i: 4 floats
    auto xv = [&](uint32_t i, float (&v)[4]) {
        ld4(xr + (size_t) i * 4, v);
        if (br) {
            float b4[4];
            ld4(br + (size_t) i * 4, b4);
            if (a.gate) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    b4[e] = b4[e] * a.gate[i + e];
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = v[e] + b4[e];
            }
        }
    };
    double ss = 0.0;
    for (uint32_t i = 4u * (uint32_t) tid; i < a.k; i += 1024u) {
        float v[4];
        xv(i, v);
        if (a.sum) {
            float * sp = (float *) (a.sum + (int64_t) m * a.sum1) + i;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sp[e] = v[e];
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            ss += (double) (v[e] * v[e]);
        }
    }
    ss = group_sum<64>(ss);
    if ((tid & 63) == 0) {
        red[tid >> 6] = ss;
    }
    __syncthreads();
    if (tid == 0) {
        scl = rms_scale(red[0] + red[1] + red[2] + red[3], (int) a.k, a.eps);
    }
    __syncthreads();
    const float    scale = scl;
    const uint32_t sub   = (uint32_t) tid & 7u;
    for (uint32_t b = (uint32_t) tid >> 3; b < a.nbk; b += 32u) {  // the 8 lanes of a block share b
        const uint32_t i0 = b * 32u + sub * 4u;
        float          f[4];
        xv(i0, f);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = f[e] * scale;
            f[e]          = v * a.nw[i0 + e];
        }
        if (a.msc) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f[e] = f[e] * (a.msc[i0 + e] + 1.0f);
                f[e] = f[e] + a.msh[i0 + e];
            }
        }
        float amax = fmaxf(fmaxf(fabsf(f[0]), fabsf(f[1])), fmaxf(fabsf(f[2]), fabsf(f[3])));
        amax       = group_max<8>(amax);
        const float d  = mm_div127(amax);
        const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
        uint32_t    w  = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float q = __builtin_amdgcn_fmed3f(__builtin_rintf(f[e] * id), -128.0f, 127.0f);
            w |= ((uint32_t) (int32_t) q & 0xffu) << (8 * e);
        }
        *(uint32_t *) (a.xq + ((int64_t) b * a.mp + m) * 32 + sub * 4) = w;
        if (sub == 0) {
            a.xd[(int64_t) b * a.mp + m] = (float) __builtin_bit_cast(_Float16, f32_to_f16_bits(d));
        }
    }
}

// The same prologue for longer x (prefill): a workgroup per 8 consecutive rows.
// Lane (row r0 + l / 8, part l % 8) of wave w holds 4 elements of each of its
// row's blocks w, w + 4, ... in registers, all loaded at once: their float
// squares summed in double, over the row's 8 lanes and over the 4 waves (LDS),
// give the row's scale; the same registers are then scaled, multiplied by w,
// quantized and stored, so that each store instruction writes the 8 rows'
// quants of one block as one 256-byte run of the block-major layout (one
// workgroup per row wrote 32-byte pieces 32 * mp bytes apart). With an addend
// the residual sum is formed once and written in the first pass (ADD: a.ab is
// given, so that the plain prologue holds no registers for it); the gate and
// the modulate as in k_mmv_quant_x_norm. Rows of x are at most 4 * NBW blocks.
template <int NBW, bool ADD>
__global__ void __launch_bounds__(256) k_mmv_quant_x_norm8(const MmvArgs a) {
    __shared__ double red[4][8];
    __shared__ float  scl[8];
    const int      tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const uint32_t row = blockIdx.x * 8u + (uint32_t) (lane >> 3), sub = (uint32_t) lane & 7u;
    const bool     rv  = row < a.m;  // uniform over a row's 8 lanes
    const uint32_t rc  = rv ? row : a.m - 1;
    const char *   xr  = a.x + (int64_t) rc * a.x1;
    const char *   br  = ADD ? a.ab + (int64_t) rc * a.ab1 : nullptr;
    auto           ld4 = [&](const char * p, float (&v)[4]) {
        if (a.xvec) {
            const float4 q = *(const float4 *) p;
            v[0]           = q.x;
            v[1]           = q.y;
            v[2]           = q.z;
            v[3]           = q.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = ((const float *) p)[e];
            }
        }
    };
    // every load unconditional (blocks past the row clamped to its last one), so
    // all are in flight before the first is used
    float v[NBW][4], u[ADD ? NBW : 1][4];
#pragma unroll
    for (int j = 0; j < NBW; ++j) {
        const uint32_t b  = (uint32_t) wv + 4u * (uint32_t) j;
        const uint32_t bc = b < a.nbk ? b : a.nbk - 1;
        ld4(xr + (size_t) (bc * 32u + sub * 4u) * 4, v[j]);
        if constexpr (ADD) {
            ld4(br + (size_t) (bc * 32u + sub * 4u) * 4, u[j]);
        }
    }
    double ss = 0.0;
#pragma unroll
    for (int j = 0; j < NBW; ++j) {
        const uint32_t b = (uint32_t) wv + 4u * (uint32_t) j;
        if (b < a.nbk && rv) {
            if constexpr (ADD) {
                if (a.gate) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        u[j][e] = u[j][e] * a.gate[b * 32u + sub * 4u + e];
                    }
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    v[j][e] = v[j][e] + u[j][e];
                }
                if (a.sum) {
                    *(float4 *) ((float *) (a.sum + (int64_t) row * a.sum1) + b * 32u + sub * 4u) =
                        make_float4(v[j][0], v[j][1], v[j][2], v[j][3]);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                ss += (double) (v[j][e] * v[j][e]);
            }
        }
    }
    ss = group_sum<8>(ss);
    if (sub == 0) {
        red[wv][lane >> 3] = ss;
    }
    __syncthreads();
    if (tid < 8) {
        scl[tid] = rms_scale(red[0][tid] + red[1][tid] + red[2][tid] + red[3][tid], (int) a.k, a.eps);
    }
    __syncthreads();
    const float scale = scl[lane >> 3];
#pragma unroll
    for (int j = 0; j < NBW; ++j) {
        const uint32_t b = (uint32_t) wv + 4u * (uint32_t) j;
        if (b >= a.nbk) {
            break;  // uniform over the wave
        }
        const uint32_t i0 = b * 32u + sub * 4u;
        float          f[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            f[e] = (v[j][e] * scale) * a.nw[i0 + e];
        }
        if (a.msc) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f[e] = f[e] * (a.msc[i0 + e] + 1.0f);
                f[e] = f[e] + a.msh[i0 + e];
            }
        }
        float amax = fmaxf(fmaxf(fabsf(f[0]), fabsf(f[1])), fmaxf(fabsf(f[2]), fabsf(f[3])));
        amax       = group_max<8>(amax);
        const float d  = mm_div127(amax);
        const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
        uint32_t    wq = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float q = __builtin_amdgcn_fmed3f(__builtin_rintf(f[e] * id), -128.0f, 127.0f);
            wq |= ((uint32_t) (int32_t) q & 0xffu) << (8 * e);
        }
        if (rv) {
            *(uint32_t *) (a.xq + ((int64_t) b * a.mp + row) * 32 + sub * 4) = wq;
            if (sub == 0) {
                a.xd[(int64_t) b * a.mp + row] = (float) __builtin_bit_cast(_Float16, f32_to_f16_bits(d));
            }
        }
    }
}

#ifndef MI_MMV_UNROLL
#define MI_MMV_UNROLL 4  // blocks whose weight loads are issued together
#endif

// y element (m, n) as stored: the product, or ggml_add(product, res) then, with
// rclamp, ggml_clamp -- the residual add fused after the product (one rounding,
// as the separate add; the add is commutative, so the operand order is ggml's)
__device__ __forceinline__ float mm_epilogue(const MmvArgs & a, uint32_t m, uint32_t n, float v) {
    if (a.res != nullptr) {
        if (a.rgate) {
            v = v * a.rgate[n];  // ggml_add(res, ggml_mul(product, gate)): the product rounded first
        }
        v = v + *(const float *) (a.res + (int64_t) m * a.res1 + (int64_t) n * 4);
        if (a.rclamp) {
            v = clamp_ggml(v, a.rlo, a.rhi);
        }
    }
    return v;
}

// The epilogue split in two for an output group: the residual values loaded
// first (all of a group's loads in flight together; callers clamp m and n into
// the output), then added (with the clamp) as mm_epilogue adds them.
__device__ __forceinline__ float mm_res(const MmvArgs & a, uint32_t m, uint32_t n) {
    return *(const float *) (a.res + (int64_t) m * a.res1 + (int64_t) n * 4);
}
__device__ __forceinline__ float mm_add_res(const MmvArgs & a, float v, float r, uint32_t n) {
    if (a.rgate) {
        v = v * a.rgate[n];
    }
    v = v + r;
    return a.rclamp ? clamp_ggml(v, a.rlo, a.rhi) : v;
}

template <int M>
__global__ void __launch_bounds__(512) k_mmv_q8_0(const MmvArgs a) {
    extern __shared__ float red[];  // [wave][m][lane], W * M * 64 floats when W > 1
    const uint32_t g = blockIdx.x, s1 = blockIdx.y;
    const int      tid = threadIdx.x, l = tid & 63;
    const int      w   = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: x loads stay scalar
    const int      W   = (int) a.wpg;
    const uint32_t s   = s1 * (uint32_t) W + (uint32_t) w;  // this wave's key split
    const uint32_t b0  = s * a.bps < a.nbk ? s * a.bps : a.nbk;
    const uint32_t b1  = b0 + a.bps < a.nbk ? b0 + a.bps : a.nbk;
    const char *   wq  = a.w + (uint64_t) g * a.nbk * 2048 + 16 * l;
    const char *   wd  = a.w + a.qbytes + (uint64_t) g * a.nbk * 128 + 2 * l;
    const char * __restrict__ xq  = a.xq;
    const float * __restrict__ xd = a.xd;
    float acc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        acc[m] = 0.0f;
    }
    constexpr int U = MI_MMV_UNROLL;
    auto block = [&](const uint4 & w0, const uint4 & w1, uint16_t dh, uint32_t b) {
        const uint32_t wv[8] = { w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w };
        const float    dw    = (float) __builtin_bit_cast(_Float16, dh);
        const uint32_t * xb  = (const uint32_t *) (xq + (size_t) b * (M * 32));
        const float *    xdb = xd + (size_t) b * M;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            int isum = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                isum = __builtin_amdgcn_sdot4((int) wv[k], (int) xb[8 * m + k], isum, false);
            }
            acc[m] = __builtin_fmaf((float) isum, dw * xdb[m], acc[m]);
        }
    };
    // two register sets of U blocks: the loads of one are in flight while the
    // other's dot products run
    uint4    a0[U], a1[U], c0[U], c1[U];
    uint16_t ad[U], cd[U];
    auto load = [&](uint4 (&w0)[U], uint4 (&w1)[U], uint16_t (&dh)[U], uint32_t bb) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            w0[u] = ld16(wq + (size_t) (bb + u) * 2048);
            w1[u] = ld16(wq + (size_t) (bb + u) * 2048 + 1024);
            dh[u] = *(const uint16_t *) (wd + (size_t) (bb + u) * 128);
        }
    };
    auto run = [&](const uint4 (&w0)[U], const uint4 (&w1)[U], const uint16_t (&dh)[U], uint32_t bb) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            block(w0[u], w1[u], dh[u], bb + u);
        }
    };
    uint32_t b = b0;
    if (b + U <= b1) {
        load(a0, a1, ad, b);
    }
    while (b + U <= b1) {
        const bool nc = b + 2 * U <= b1;
        if (nc) {
            load(c0, c1, cd, b + U);
        }
        run(a0, a1, ad, b);
        b += U;
        if (!nc) {
            break;
        }
        const bool na = b + 2 * U <= b1;
        if (na) {
            load(a0, a1, ad, b + U);
        }
        run(c0, c1, cd, b);
        b += U;
        if (!na) {
            break;
        }
    }
    for (; b < b1; ++b) {
        block(ld16(wq + (size_t) b * 2048), ld16(wq + (size_t) b * 2048 + 1024),
              *(const uint16_t *) (wd + (size_t) b * 128), b);
    }
    const uint32_t row = g * 64 + l;
    auto store_y = [&](int m, float v) {
        if (row < a.n) {
            *(float *) (a.y + (int64_t) m * a.y1 + (int64_t) row * 4) = mm_epilogue(a, (uint32_t) m, row, v);
        }
    };
    if (W == 1 && a.splits == 1) {
        if (a.res != nullptr) {
            const uint32_t rc = row < a.n ? row : a.n - 1;
            float          r[M];
#pragma unroll
            for (int m = 0; m < M; ++m) {
                r[m] = mm_res(a, (uint32_t) m, rc);
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                if (row < a.n) {
                    *(float *) (a.y + (int64_t) m * a.y1 + (int64_t) row * 4) = mm_add_res(a, acc[m], r[m], row);
                }
            }
            return;
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            store_y(m, acc[m]);
        }
        return;
    }
    // the workgroup's splits, added in wave order; wave w then owns rows m = w, w + W, ...
#pragma unroll
    for (int m = 0; m < M; ++m) {
        red[(w * M + m) * 64 + l] = acc[m];
    }
    __syncthreads();
    for (int m = w; m < M; m += W) {
        float v = 0.0f;
        for (int w2 = 0; w2 < W; ++w2) {
            v += red[(w2 * M + m) * 64 + l];
        }
        if (a.splits == 1) {
            store_y(m, v);
        } else {
            a.part[((size_t) s1 * M + m) * a.npad + row] = v;
        }
    }
}

// Matrix-vector product of one row of x in one launch: the x prologue (the plain
// quantization, SwiGLU, or [residual add ->] RMSNorm [-> modulate]), the product and
// the sum of its key splits. At these sizes (one token: 1-25 MB of weights,
// 4-12 KB of x) a product as prologue, product and split sum is bound by its
// three launches, each about 3 us with its gap and mostly idle; so every workgroup
// quantizes all of x itself, from the caches, into LDS, while its first weight blocks
// are in flight, and holds all key splits of a 64-row group, added in LDS in the order
// in which k_mmv_q8_0 and k_mmv_reduce add them: the same bits as the three launches. A
// wave's share is its splits times a.bps blocks: up to 8, or 9 (3 sets, the last of one
// block) with 3 splits of 3 blocks at 171 to 255 row groups. The row's RMS sum is formed
// the same way in every workgroup (the first one writes the residual sum).
__global__ void __launch_bounds__(512) k_mmv1_q8_0(const MmvArgs a) {
    constexpr int W = 8;  // waves = key splits
    // x quants [nbk][32], read 16 bytes at a time, scales [nbk], the splits' sums [W * splits][64]
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ double rs[W];  // (the first 4 waves sum the squares, in k_mmv_quant_x_norm's order)
    __shared__ float  scl;
    const uint32_t g = blockIdx.x;
    const int      tid = threadIdx.x, l = tid & 63;
    const int      w = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int  T = 64 * W;
    // the wave's key splits: a.splits in a row of a.bps blocks each
    const uint32_t bw = a.splits * a.bps;
    const uint32_t b0 = (uint32_t) w * bw < a.nbk ? (uint32_t) w * bw : a.nbk;
    const uint32_t b1 = b0 + bw < a.nbk ? b0 + bw : a.nbk;
    const char *   wq = a.w + (uint64_t) g * a.nbk * 2048 + 16 * l;
    const char *   wd = a.w + a.qbytes + (uint64_t) g * a.nbk * 128 + 2 * l;
    constexpr int  U  = MI_MMV_UNROLL;
    uint4          a0[U], a1[U], c0[U], c1[U];
    uint16_t       ad[U], cd[U];
    // a set of U blocks; blocks past the wave's range are clamped to its last one (not used)
    auto load = [&](uint4 (&w0)[U], uint4 (&w1)[U], uint16_t (&dh)[U], uint32_t bb) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t b = bb + u < b1 ? bb + u : b1 - 1;
            w0[u]            = ld16(wq + (size_t) b * 2048);
            w1[u]            = ld16(wq + (size_t) b * 2048 + 1024);
            dh[u]            = *(const uint16_t *) (wd + (size_t) b * 128);
        }
    };
    if (b0 < b1) {
        load(a0, a1, ad, b0);
    }
    char *  xq = lds;
    float * xd = (float *) (lds + (size_t) a.nbk * 32);
    auto    ld4 = [&](const char * p, float (&v)[4]) {
        if (a.xvec) {
            const float4 q = *(const float4 *) p;
            v[0]           = q.x;
            v[1]           = q.y;
            v[2]           = q.z;
            v[3]           = q.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = ((const float *) p)[e];
            }
        }
    };
    // x at element i: 4 floats (with the residual sum or the SwiGLU formed)
    auto xv = [&](uint32_t i, float (&v)[4]) {
        if (a.glu) {
            float h[4];
            ld4(a.g + (int64_t) i * 4, v);
            ld4(a.u + (int64_t) i * 4, h);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = silu_f(v[e]) * h[e];
            }
            return;
        }
        ld4(a.x + (int64_t) i * 4, v);
        if (a.ab) {
            float b4[4];
            ld4(a.ab + (int64_t) i * 4, b4);
            if (a.gate) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    b4[e] = b4[e] * a.gate[i + e];
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[e] = v[e] + b4[e];
            }
        }
    };
    float scale = 1.0f;
    if (a.nw) {
        double ss = 0.0;
        for (uint32_t i = tid < 256 ? 4u * (uint32_t) tid : a.k; i < a.k; i += 1024u) {
            float v[4];
            xv(i, v);
            if (a.sum && g == 0) {
                float * sp = (float *) a.sum + i;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    sp[e] = v[e];
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                ss += (double) (v[e] * v[e]);
            }
        }
        ss = group_sum<64>(ss);
        if (l == 0) {
            rs[w] = ss;
        }
        __syncthreads();
        if (tid == 0) {
            scl = rms_scale(rs[0] + rs[1] + rs[2] + rs[3], (int) a.k, a.eps);
        }
        __syncthreads();
        scale = scl;
    }
    const uint32_t sub = (uint32_t) tid & 7u;
    for (uint32_t b = (uint32_t) tid >> 3; b < a.nbk; b += (uint32_t) T / 8) {  // the 8 lanes of a block share b
        const uint32_t i0 = b * 32u + sub * 4u;
        float          f[4];
        xv(i0, f);
        if (a.nw) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = f[e] * scale;
                f[e]          = v * a.nw[i0 + e];
            }
            if (a.msc) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    f[e] = f[e] * (a.msc[i0 + e] + 1.0f);
                    f[e] = f[e] + a.msh[i0 + e];
                }
            }
        }
        float amax = fmaxf(fmaxf(fabsf(f[0]), fabsf(f[1])), fmaxf(fabsf(f[2]), fabsf(f[3])));
        amax       = group_max<8>(amax);
        const float d  = mm_div127(amax);
        const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
        uint32_t    qv = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float q = __builtin_amdgcn_fmed3f(__builtin_rintf(f[e] * id), -128.0f, 127.0f);
            qv |= ((uint32_t) (int32_t) q & 0xffu) << (8 * e);
        }
        *(uint32_t *) (xq + (size_t) b * 32 + sub * 4) = qv;
        if (sub == 0) {
            xd[b] = (float) __builtin_bit_cast(_Float16, f32_to_f16_bits(d));
        }
    }
    __syncthreads();
    float    acc  = 0.0f;
    float *  red  = xd + a.nbk;  // [split][lane]
    uint32_t vs   = (uint32_t) w * a.splits, left = a.bps;  // the split, its blocks left
    for (uint32_t q = 0; q < a.splits; ++q) {
        red[(vs + q) * 64 + l] = 0.0f;
    }
    // a set's dots, straight-line: the LDS reads of all its blocks are in flight together
    // (a block past the range reads the last one, its dot is dropped by a select)
    auto run = [&](const uint4 (&w0)[U], const uint4 (&w1)[U], const uint16_t (&dh)[U], uint32_t bb) {
        uint4 x0[U], x1[U];
        float xs[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t b  = bb + u < b1 ? bb + u : b1 - 1;
            const uint4 *  xb = (const uint4 *) (xq + (size_t) b * 32);
            x0[u]             = xb[0];
            x1[u]             = xb[1];
            xs[u]             = xd[b];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t wv[8] = { w0[u].x, w0[u].y, w0[u].z, w0[u].w, w1[u].x, w1[u].y, w1[u].z, w1[u].w };
            const uint32_t xw[8] = { x0[u].x, x0[u].y, x0[u].z, x0[u].w, x1[u].x, x1[u].y, x1[u].z, x1[u].w };
            int            isum  = 0;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                isum = __builtin_amdgcn_sdot4((int) wv[q], (int) xw[q], isum, false);
            }
            const float dw = (float) __builtin_bit_cast(_Float16, dh[u]);
            const float v  = __builtin_fmaf((float) isum, dw * xs[u], acc);
            acc            = bb + u < b1 ? v : acc;
            if (--left == 0 || bb + u + 1 == b1) {  // uniform: the split's last block
                if (bb + u < b1) {
                    red[vs * 64 + l] = acc;
                }
                acc  = 0.0f;
                left = a.bps;
                ++vs;
            }
        }
    };
    // two register sets of U blocks: one's loads are in flight while the other's dots run
    for (uint32_t b = b0; b < b1; b += 2 * U) {
        if (b + U < b1) {
            load(c0, c1, cd, b + U);
        }
        run(a0, a1, ad, b);
        if (b + 2 * U < b1) {
            load(a0, a1, ad, b + 2 * U);
        }
        if (b + U < b1) {
            run(c0, c1, cd, b + U);
        }
    }
    const uint32_t row = g * 64 + l;
    __syncthreads();
    // the splits of a workgroup of k_mmv_q8_0 in wave order, a wave each, and then those
    // sums in k_mmv_reduce's order
    for (uint32_t s1 = (uint32_t) w; s1 < a.splits; s1 += (uint32_t) W) {
        float p = 0.0f;
#pragma unroll
        for (uint32_t w2 = 0; w2 < (uint32_t) W; ++w2) {
            p += w2 < a.wpg ? red[(s1 * a.wpg + w2) * 64 + l] : 0.0f;
        }
        red[s1 * a.wpg * 64 + l] = p;  // (this wave's own lane read it)
    }
    __syncthreads();
    if (w == 0 && row < a.n) {
        float v = 0.0f;
        for (uint32_t s1 = 0; s1 < a.splits; ++s1) {
            v += red[s1 * a.wpg * 64 + l];
        }
        *(float *) (a.y + (int64_t) row * 4) = mm_epilogue(a, 0, row, v);
    }
}

// y[m][row] = sum over the workgroups' partials, in workgroup order (splits > 1)
template <int M>
__global__ void __launch_bounds__(256) k_mmv_reduce(const MmvArgs a) {
    const uint32_t gid = blockIdx.x * 256u + threadIdx.x;
    if (gid >= M * a.npad) {
        return;
    }
    const uint32_t m = gid / a.npad, row = gid - m * a.npad;
    if (row >= a.n) {
        return;
    }
    const float * pp = a.part + (size_t) m * a.npad + row;
    const size_t  st = (size_t) M * a.npad;
    float         v  = 0.0f;
    uint32_t      s2 = 0;
    for (; s2 + 8 <= a.splits; s2 += 8) {
        float t[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            t[j] = pp[(s2 + j) * st];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            v += t[j];
        }
    }
    for (; s2 < a.splits; ++s2) {
        v += pp[s2 * st];
    }
    *(float *) (a.y + (int64_t) m * a.y1 + (int64_t) row * 4) = mm_epilogue(a, m, row, v);
}


// Matrix kernel (more than 8 rows of x: prefill, the DiT): a workgroup of 4
// waves owns 128 rows of x x 128 weight rows; each wave a 64 x 64 tile as 2 x 2
// v_mfma_i32_32x32x32_i8 tiles (D rows = rows of x, columns = weight rows, so a
// lane stores consecutive outputs). Per 32-element block: one MFMA per tile
// gives the exact int32 block dots, and acc = fma(float(isum), d_w * d_x, acc)
// scales them in block order -- the arithmetic of the matrix-vector kernel
// (the d_w * d_x products come from an f32 outer-product MFMA, exactly).
// Operands come straight from global memory in MFMA lane order: x from the
// block-major quantized rows (lane l: row l % 32, bytes 16 (l / 32) of the
// block), weights from the R64 layout (a 32-row half of a group is two 512-byte
// runs), so no LDS staging is needed; one block ahead is in flight.
#ifndef MI_MMQ_PRIO
#define MI_MMQ_PRIO 1  // > 0: the wave's issue priority while it issues a block's MFMAs
#endif
#ifndef MI_MMQ_WG_PER_CU
#define MI_MMQ_WG_PER_CU 2  // resident workgroups of the matrix kernel per CU (2 waves per SIMD)
#endif
#ifndef MI_MMQ_MAX_KSPLIT
#define MI_MMQ_MAX_KSPLIT 4  // key splits of the matrix kernel at most
#endif
#ifndef MI_MMQ_MIN_BPS
#define MI_MMQ_MIN_BPS 32  // blocks of 32 keys per split at least
#endif
typedef int mm_i32x4 __attribute__((ext_vector_type(4)));
typedef int mm_i32x16 __attribute__((ext_vector_type(16)));
typedef float mm_f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 mm_f16x8 __attribute__((ext_vector_type(8)));
typedef float mm_f32x32 __attribute__((ext_vector_type(32)));

__global__ void __launch_bounds__(256) k_mmq_q8_0(const MmvArgs a) {
    const int      tid = threadIdx.x, l = tid & 63, wv = tid >> 6;
    const int      hh  = l >> 5, c = l & 31;
    const uint32_t m0  = blockIdx.y * 128 + (wv >> 1) * 64;  // rows of x (padded to 128)
    const uint32_t n0  = blockIdx.x * 128 + (wv & 1) * 64;   // weight rows
    const uint32_t g   = n0 / 64;                             // R64 row group
    if (g >= a.ng) {
        return;  // whole wave
    }
    const char *   wq = a.w + (uint64_t) g * a.nbk * 2048 + (size_t) hh * 1024 + 16 * c;
    const char *   wd = a.w + a.qbytes + (uint64_t) g * a.nbk * 128 + 2 * c;
    const char *   xq = a.xq + (size_t) (m0 + c) * 32 + hh * 16;
    const float *  xd = a.xd + m0;
    const uint64_t xqs = (uint64_t) a.mp * 32;  // per block
    float          acc[2][2][16];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[i][j][e] = 0.0f;
            }
        }
    }
    struct Blk {
        uint4    x[2], w[2];
        uint16_t dw[2];
        float    dx[2];
    };
    auto load = [&](Blk & k, uint32_t b) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {  // x tile i: rows m0 + 32 i + c
            k.x[i]  = *(const uint4 *) (xq + b * xqs + (size_t) i * 32 * 32);
            k.dx[i] = xd[(size_t) b * a.mp + 32 * i + c];
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {  // weight tile j: rows n0 + 32 j + c
            k.w[j]  = *(const uint4 *) (wq + (size_t) b * 2048 + 512 * j);  // cached: every row tile of x reads it
            k.dw[j] = *(const uint16_t *) (wd + (size_t) b * 128 + 64 * j);
        }
    };
    // the block's scales d_x[m] d_w[n] as a 32 x 32 outer product on the matrix
    // core, in the D layout of the int32 dots, so each output costs one
    // conversion and one fma. Both scales are fp16 values (d_x was rounded to
    // fp16 when x was quantized), so an fp16 MFMA with k-slot 0 carrying them and
    // the other 15 slots zero forms every product exactly, at half the matrix-core
    // time of an fp32 outer product.
    auto run = [&](const Blk & k) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const mm_i32x4 av = { (int) k.x[i].x, (int) k.x[i].y, (int) k.x[i].z, (int) k.x[i].w };
            mm_f16x8       sx = {};
            sx[0]             = hh == 0 ? (_Float16) k.dx[i] : (_Float16) 0.0f;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const mm_i32x4  bv = { (int) k.w[j].x, (int) k.w[j].y, (int) k.w[j].z, (int) k.w[j].w };
                if constexpr (MI_MMQ_PRIO > 0) {
                    __builtin_amdgcn_s_setprio(MI_MMQ_PRIO);
                }
                const mm_i32x16 d  = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, bv, mm_i32x16{}, 0, 0, 0);
                mm_f16x8        sw = {};
                sw[0]              = hh == 0 ? __builtin_bit_cast(_Float16, k.dw[j]) : (_Float16) 0.0f;
                const mm_f32x16 sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(sx, sw, mm_f32x16{}, 0, 0, 0);
                if constexpr (MI_MMQ_PRIO > 0) {
                    __builtin_amdgcn_s_setprio(0);
                }
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    acc[i][j][e] = __builtin_fmaf((float) d[e], sc[e], acc[i][j][e]);
                }
            }
        }
    };
    // this workgroup's blocks: split blockIdx.z of the key range
    const uint32_t bb = blockIdx.z * a.bps;
    const uint32_t be = bb + a.bps < a.nbk ? bb + a.bps : a.nbk;
    Blk            k0, k1;
    uint32_t       b = bb;
    if (b < be) {
        load(k0, b);
    }
    while (b < be) {
        const bool n1 = b + 1 < be;
        if (n1) {
            load(k1, b + 1);
        }
        run(k0);
        ++b;
        if (!n1) {
            break;
        }
        const bool n0b = b + 1 < be;
        if (n0b) {
            load(k0, b + 1);
        }
        run(k1);
        ++b;
        if (!n0b) {
            break;
        }
    }
    if (a.splits > 1) {
        // the split's sums to the workspace [split][mp][npad] (every row and
        // column of the tile lies inside the padded extent); k_mmq_reduce adds
        // the splits in order and applies the epilogue
        float * pp = a.part + (size_t) blockIdx.z * a.mp * a.npad;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        pp[(size_t) (m0 + 32 * i + 8 * q + 4 * hh + e) * a.npad + n0 + 32 * j + c] = acc[i][j][4 * q + e];
                    }
                }
            }
        }
        return;
    }
    // D lane l: column n0 + 32 j + c, rows m0 + 32 i + 8 q + 4 hh + e; with a
    // residual, the 16 values of an (i, j) tile are loaded before any is added
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uint32_t n = n0 + 32 * j + c;
        if (n >= a.n) {
            continue;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float r[16];
            if (a.res != nullptr) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t m = m0 + 32 * i + 8 * q + 4 * hh + e;
                        r[4 * q + e]     = mm_res(a, m < a.m ? m : a.m - 1, n);
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t m = m0 + 32 * i + 8 * q + 4 * hh + e;
                    if (m < a.m) {
                        const float v = acc[i][j][4 * q + e];
                        *(float *) (a.y + (int64_t) m * a.y1 + (int64_t) n * 4) =
                            a.res != nullptr ? mm_add_res(a, v, r[4 * q + e], n) : v;
                    }
                }
            }
        }
    }
}

// Matrix kernel for grids that the 128 x 128 tiles leave idle (short x: short
// prompts and clips, a few rows more than the matrix-vector kernel takes): a
// workgroup owns 64 rows of x x 64 weight rows, and its 8 waves are 2 positions (32
// rows of x x 64 weight rows each) x 4 key groups: every stage of 4 blocks gives each
// key group one, and the groups' sums are added in group order in LDS, so the keys
// are split over 4 waves without partials in memory or a second launch. What bounds
// it is the latency of one wave's chain of blocks (LDS reads, 3 MFMAs, 32 subtractions
// and 32 fmas), so the split is over keys and the operands are fetched ahead:
// global_load_lds copies them into LDS 3 stages (12 blocks) before use, in MFMA lane
// order, so that the reads are linear and conflict-free; 124 VGPRs without a spill keep
// 4 waves per SIMD (2 workgroups per CU). The block's scales are two f32 outer products by one
// v_mfma_f32_32x32x1_2b (K = 1: a lane holds one d_x and one d_w, no zero slots to
// build). Measured against the 128 x 128 kernel (x quantization and split sum
// included, us, 2048 -> 2048 / 2048 -> 12288): 9 rows 27.5 ->
// 13.2 / 30.2 -> 16.7, 128 rows 28.4 -> 14.5 / 35.2 -> 23.4, 375 rows 32.7 -> 17.8 /
// 54.8 -> 49.3, 1537 rows of 2048 -> 2048 45.9 -> 42.9. On large grids it loses
// (12288 x 1024 rows: 110 against 89): twice the operand traffic per output.

// 16 bytes per lane from base + off straight into LDS at dst + 16 * lane (dst uniform; the
// instruction takes it from m0, which the compiler sets, a wait state before)
__device__ __forceinline__ void mmq_dma(uint32_t dst, const char * base, uint32_t off) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "{m0}"(dst), "v"(off), "s"(base) : "memory");
}
__device__ __forceinline__ void mmq_dma_v(uint32_t dst, const char * p) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "{m0}"(dst), "v"(p) : "memory");
}

__global__ void __launch_bounds__(512, 4) k_mmq64_q8_0(const MmvArgs a) {
    // 32-row tiles per wave (of x, of w), wave positions, key groups, blocks per stage, stages
    constexpr int WM = 1, WN = 2, NM = 2, NN = 1, KG = 4, KB = 4, D = 4;
    static_assert(WN % 2 == 0 && KB % KG == 0, "the scales of two weight tiles come from one MFMA");
    constexpr int XT = WM * NM, WT = WN * NN, NP = NM * NN, NW = NP * KG;  // 32-row tiles, wave positions, waves
    constexpr int QI    = KB * (XT + WT);                                   // 1 KB loads of a stage's quants
    constexpr int XS    = KB * XT * 8, WS = KB * WT * 4;                    // 16-byte chunks of its scales of x, of w
    constexpr int SCI   = (XS + WS + 63) / 64;                              // 1 KB loads of those
    constexpr int STAGE = QI * 1024 + (XS + WS) * 16;
    constexpr int RED   = NW * WM * WN * 4096;                              // the key groups' sums
    static_assert(QI % NW == 0 && SCI <= NW, "every wave issues QI / NW loads, the first SCI waves one more");
    __shared__ __attribute__((aligned(1024))) char lds[D * STAGE > RED ? D * STAGE : RED];
    const int      tid = threadIdx.x, l = tid & 63;
    const int      wv  = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int      hh  = l >> 5, c = l & 31;
    // Workgroups go to the XCDs in turn: each XCD takes one run of tiles, in
    // groups of 8 row tiles, so that the tiles resident on it share x and w in its L2.
    const uint32_t tn = (a.n + 32 * WT - 1) / (32 * WT), tm = (a.m + 32 * XT - 1) / (32 * XT);
    const uint32_t per = tn * tm, total = per * a.splits;
    uint32_t       t   = blockIdx.x;
    {
        const uint32_t x8 = t % 8, q = total / 8, r = total % 8;
        t = x8 * q + (x8 < r ? x8 : r) + t / 8;
    }
    const uint32_t z = t / per;
    t -= z * per;
    const uint32_t gm = t / (8 * tn), gh = tm - 8 * gm < 8 ? tm - 8 * gm : 8;
    t -= gm * 8 * tn;
    const uint32_t nt = t / gh, mt = 8 * gm + (t - nt * gh);
    const uint32_t mw = mt * 32 * XT, nw = nt * 32 * WT;  // the workgroup's first rows of x and of w
    // this workgroup's blocks: split z of the key range
    const uint32_t bb = z * a.bps;
    const uint32_t be = bb + a.bps < a.nbk ? bb + a.bps : a.nbk;

    const uint32_t lds0  = (uint32_t) (uintptr_t) (__attribute__((address_space(3))) char *) lds;
    const uint64_t xqs   = (uint64_t) a.mp * 32;  // quants of x per block
    const uint32_t xoff  = (uint32_t) (c * 32 + hh * 16), woff = (uint32_t) (hh * 1024 + c * 16);
    // A stage's loads: every 1 KB tile lands in LDS in MFMA lane order (lane l: row
    // l % 32, bytes 16 (l / 32) of the block), so the reads are linear; blocks past
    // the split's end and row groups past the weight are clamped (never used / stored).
    auto issue = [&](uint32_t b, uint32_t buf) {
        const uint32_t base = lds0 + buf * STAGE;
#pragma unroll
        for (int i = 0; i < QI / NW; ++i) {
            const int      o = wv + NW * i, kb = o / (XT + WT), r = o % (XT + WT);
            const uint32_t bk = b + kb < a.nbk ? b + kb : a.nbk - 1;
            if (r < XT) {
                mmq_dma(base + (uint32_t) o * 1024, a.xq + bk * xqs + (uint64_t) (mw + 32 * r) * 32, xoff);
            } else {
                const uint32_t g0 = nw / 64 + (r - XT) / 2, g = g0 < a.ng ? g0 : a.ng - 1;
                mmq_dma(base + (uint32_t) o * 1024, a.w + ((uint64_t) g * a.nbk + bk) * 2048 + 512 * ((r - XT) & 1), woff);
            }
        }
        if (wv < SCI) {
            const uint32_t q = (uint32_t) (wv * 64 + l);  // 16-byte chunk: x scales [kb][32 XT] f32, then w's [kb][32 WT] fp16
            const char *   p = nullptr;
            if (q < XS) {
                const uint32_t kb = q / (8 * XT), o = q % (8 * XT);
                const uint32_t bk = b + kb < a.nbk ? b + kb : a.nbk - 1;
                p = (const char *) a.xd + ((uint64_t) bk * a.mp + mw) * 4 + o * 16;
            } else if (q < XS + WS) {
                const uint32_t qw = q - XS, kb = qw / (4 * WT), o = qw % (4 * WT);
                const uint32_t bk = b + kb < a.nbk ? b + kb : a.nbk - 1;
                const uint32_t g0 = nw / 64 + o / 8, g = g0 < a.ng ? g0 : a.ng - 1;
                p = a.w + a.qbytes + ((uint64_t) g * a.nbk + bk) * 128 + (o % 8) * 16;
            }
            if (p) {
                mmq_dma_v(base + (uint32_t) (QI + wv) * 1024, p);
            }
        }
    };
#pragma unroll
    for (int s = 0; s < D - 1; ++s) {
        if (bb + s * KB < be) {
            issue(bb + s * KB, s);
        }
    }
    float acc[WM][WN][16];
#pragma unroll
    for (int i = 0; i < WM; ++i) {
#pragma unroll
        for (int j = 0; j < WN; ++j) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[i][j][e] = 0.0f;
            }
        }
    }
    // The int32 dot comes out as the bits of the float MAGIC + dot (the MFMA adds to
    // the bits of MAGIC = 1.5 * 2^23, whose ulp is 1; |dot| <= 32 * 128 * 128 < 2^22),
    // so one subtraction gives float(dot), exactly: with several waves on a SIMD
    // v_sub_f32 issues at twice the rate of v_cvt_f32_i32 (32 of them: 30 against 54 ns).
    constexpr float MAGIC = 12582912.0f;
    mm_i32x16       mg;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        mg[e] = __builtin_bit_cast(int, MAGIC);
    }
    const int kg = wv / NP, wp = wv % NP;            // the wave's key group and position
    const int wm = wp / NN * WM, wn = wp % NN * WN;  // its first tiles
    // its operands' offsets in a stage (the blocks' own are immediates)
    const uint32_t xq0 = (uint32_t) (kg * (XT + WT) + wm) * 1024, wq0 = (uint32_t) (kg * (XT + WT) + XT + wn) * 1024;
    const uint32_t xs0 = (uint32_t) (QI * 1024 + (kg * XT + wm) * 128);
    const uint32_t ws0 = (uint32_t) (QI * 1024 + XS * 16 + (kg * WT + wn) * 64);
    auto block = [&](const char * st, int kb) {
        mm_i32x4 xf[WM], wf[WN];
        float    sx[WM], sw[WN / 2];
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            xf[i] = *(const mm_i32x4 *) (st + xq0 + l * 16 + (kb * (XT + WT) + i) * 1024);
            sx[i] = *(const float *) (st + xs0 + c * 4 + (kb * XT + i) * 128);
        }
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            wf[j] = *(const mm_i32x4 *) (st + wq0 + l * 16 + (kb * (XT + WT) + j) * 1024);
        }
#pragma unroll
        for (int j = 0; j < WN / 2; ++j) {
            sw[j] = (float) *(const _Float16 *) (st + ws0 + l * 2 + (kb * WT + 2 * j) * 64);
        }
#pragma unroll
        for (int i = 0; i < WM; ++i) {
#pragma unroll
            for (int j = 0; j < WN; j += 2) {
                // the scales d_x[m] d_w[n] of tiles j and j + 1: two 32 x 32 outer products (exact)
                __builtin_amdgcn_s_setprio(1);
                const mm_f32x32 sv = __builtin_amdgcn_mfma_f32_32x32x1f32(sx[i], sw[j / 2], mm_f32x32{}, 0, 0, 0);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    __builtin_amdgcn_s_setprio(1);
                    const mm_i32x16 d = __builtin_amdgcn_mfma_i32_32x32x32_i8(xf[i], wf[j + h], mg, 0, 0, 0);
                    __builtin_amdgcn_s_setprio(0);
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int bits   = d[e];  // (a copy: a bit cast of the vector element itself takes element 0)
                        acc[i][j + h][e] =
                            __builtin_fmaf(__builtin_bit_cast(float, bits) - MAGIC, sv[16 * h + e], acc[i][j + h][e]);
                    }
                }
            }
        }
    };
    uint32_t buf = 0, b = bb;
    // a stage has landed when its turn comes (each wave waits for its own loads, later
    // stages' stay in flight), and every wave is done reading the buffer the next loads go to
    auto next = [&]() {
        if (b + (D - 2) * KB < be) {
            if (wv < SCI) {
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((D - 2) * (QI / NW + 1)) : "memory");
            } else {
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((D - 2) * (QI / NW)) : "memory");
            }
        } else {
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        if (b + (D - 1) * KB < be) {
            issue(b + (D - 1) * KB, buf == 0 ? D - 1 : buf - 1);
        }
    };
    for (; b + KB <= be; b += KB) {
        next();
#pragma unroll
        for (int kb = 0; kb < KB; kb += KG) {
            block(lds + buf * STAGE, kb);
        }
        buf = buf + 1 == D ? 0 : buf + 1;
    }
    if (b < be) {  // the last, partial stage: nothing is left to issue
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        for (int kb = 0; b + kb + kg < be; kb += KG) {
            block(lds + buf * STAGE, kb);
        }
    }
    // Half a tile's outputs per call: D lane l holds column n0 + 32 j + c, rows m0 + 32 i
    // + 8 q + 4 hh + e (value 4 q + e); v: values e0 .. e0 + 7 of tile (i, j). Row
    // pointers are uniform (scalar), the lane's part of the address is one offset.
    const uint32_t m0 = mw + 32 * wm, n0 = nw + 32 * wn;
    const bool     in  = m0 + 32 * WM <= a.m && n0 + 32 * WN <= a.n;  // uniform: no bounds to check
    int            el  = l;  // (opaque: nothing of the epilogue's addresses is held over the loop)
    asm volatile("" : "+v"(el));
    const int      eh = el >> 5, ec = el & 31;
    const int64_t  ylo = 4 * eh * a.y1 + 4 * ec, rlo = 4 * eh * a.res1 + 4 * ec;
    auto store = [&](int i, int j, int e0, float (&v)[8]) {
        const uint32_t mt0 = m0 + 32 * i + 2 * e0, nt0 = n0 + 32 * j, n = nt0 + ec;
        if (a.splits > 1) {
            // the split's sums to the workspace [split][mp][npad] (the rows of the tile lie
            // inside the padded extent, row groups past the weight are skipped);
            // k_mmq_reduce adds the splits in order and applies the epilogue
            if (nt0 < a.npad) {
                float *        pp = a.part + ((size_t) z * a.mp + mt0) * a.npad + nt0;
                const uint32_t lo = (uint32_t) (4 * eh) * a.npad + ec;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    (pp + (size_t) (8 * (e / 4) + e % 4) * a.npad)[lo] = v[e];
                }
            }
            return;
        }
        if (!in && n >= a.n) {
            return;
        }
        if (a.res != nullptr) {  // the residual values are loaded before any is added
            const char * rt = a.res + (int64_t) mt0 * a.res1 + (int64_t) nt0 * 4;
            float        r[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t m = mt0 + 8 * (e / 4) + 4 * eh + e % 4;
                r[e] = in ? *(const float *) (rt + (int64_t) (8 * (e / 4) + e % 4) * a.res1 + rlo)
                          : mm_res(a, m < a.m ? m : a.m - 1, n);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] = mm_add_res(a, v[e], r[e], n);
            }
        }
        char * yt = a.y + (int64_t) mt0 * a.y1 + (int64_t) nt0 * 4;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (in || mt0 + 8 * (e / 4) + 4 * eh + e % 4 < a.m) {
                *(float *) (yt + (int64_t) (8 * (e / 4) + e % 4) * a.y1 + ylo) = v[e];
            }
        }
    };
    // the key groups' sums added in group order, through LDS ([wave][value][lane]);
    // each group then stores its share of the position's half tiles
    float * red = (float *) lds;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave is done with the stages
#pragma unroll
    for (int i = 0; i < WM; ++i) {
#pragma unroll
        for (int j = 0; j < WN; ++j) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                red[(wv * WM * WN + i * WN + j) * 1024 + e * 64 + el] = acc[i][j][e];
            }
        }
    }
    __syncthreads();
    for (int h = kg; h < 2 * WM * WN; h += KG) {
        const int t2 = h / 2, e0 = h % 2 * 8;
        float     v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            v[e] = 0.0f;
        }
#pragma unroll
        for (int g = 0; g < KG; ++g) {
            const float * rg = red + ((g * NP + wp) * WM * WN + t2) * 1024 + e0 * 64 + el;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] = g == 0 ? rg[e * 64] : v[e] + rg[e * 64];
            }
        }
        store(t2 / WN, t2 % WN, e0, v);
    }
}

// The matrix kernel's key splits added in split order, then the epilogue
// (residual, clamp): one thread per output, consecutive threads along a row.
__global__ void __launch_bounds__(256) k_mmq_reduce(const MmvArgs a) {
    const uint64_t gid = (uint64_t) blockIdx.x * 256u + threadIdx.x;
    const uint32_t m   = (uint32_t) (gid / a.n);
    const uint32_t n   = (uint32_t) (gid - (uint64_t) m * a.n);
    if (m >= a.m) {
        return;
    }
    const float *  pp  = a.part + (size_t) m * a.npad + n;
    const size_t   st  = (size_t) a.mp * a.npad;
    float          v[MI_MMQ_MAX_KSPLIT];
#pragma unroll
    for (int s2 = 0; s2 < MI_MMQ_MAX_KSPLIT; ++s2) {
        v[s2] = pp[(size_t) (s2 < (int) a.splits ? s2 : 0) * st];  // all loads before any add
    }
    float t = v[0];
#pragma unroll
    for (int s2 = 1; s2 < MI_MMQ_MAX_KSPLIT; ++s2) {
        if (s2 < (int) a.splits) {
            t += v[s2];
        }
    }
    *(float *) (a.y + (int64_t) m * a.y1 + (int64_t) n * 4) = mm_epilogue(a, m, n, t);
}

#ifndef MI_MMQ64_LONG_BPS
#define MI_MMQ64_LONG_BPS 96  // blocks per split from which the 64 x 64 tiles split a half-filled grid
#endif
#ifndef MI_MMV_NORED_MIN
#define MI_MMV_NORED_MIN 8  // waves per CU from which key splits stop at one workgroup per row group (0: never)
#endif
#ifndef MI_MMV_WAVES_PER_CU
#define MI_MMV_WAVES_PER_CU 16  // waves to spread one product over, per CU
#endif

// key splits: enough waves to keep the loads of the whole chip in flight; up to
// 8 splits of a row group share a workgroup (reduced in LDS), the rest go
// through the workspace
void mul_mat_q8_0_plan(MmvArgs & a, int cus) {
    a.ng     = (a.n + 63) / 64;
    a.npad   = a.ng * 64;
    a.qbytes = (uint64_t) a.ng * a.nbk * 2048;
    a.mp     = a.m <= 8 ? a.m : (a.m + 127) / 128 * 128;
    if (a.m > 8) {
        // the matrix kernels: key splits (workspace partials, added by
        // k_mmq_reduce) only when its 128 x 128 tiles leave resident workgroup
        // slots empty -- the narrow products (n = H) at prefill sizes
        a.wpg             = 1;
        const uint64_t tl = (uint64_t) ((a.n + 127) / 128) * (a.mp / 128);
        const uint64_t sl = (uint64_t) (cus > 0 ? cus : 256) * MI_MMQ_WG_PER_CU;
        uint64_t       ks = tl < sl ? sl / tl : 1;
        ks                = ks > MI_MMQ_MAX_KSPLIT ? MI_MMQ_MAX_KSPLIT : ks;
        ks                = ks > a.nbk / MI_MMQ_MIN_BPS ? a.nbk / MI_MMQ_MIN_BPS : ks;
        ks                = ks < 1 ? 1 : ks;
        // With the 64 x 64 tiles (keys split in the workgroup) workspace partials on top only
        // where the grid is under a quarter of the slots (9 x 2048 x 2048: 13.2 with, 16.0 us
        // without; 375 rows: 21.5 and 17.8), or under half with long key ranges (257 x 2048 x
        // 6144: 29 and 37 us); never more splits than the 128 x 128 tiles take, so the
        // workspace stays as it was.
        const uint64_t t64 = (uint64_t) ((a.n + 63) / 64) * ((a.m + 63) / 64);
        a.tile             = mmq_small_tiles(t64, sl, ks, a.nbk) ? 64 : 128;
        if (a.tile == 64) {
            const uint64_t k64 = 4 * t64 <= sl ? ks : 2 * t64 <= sl ? a.nbk / MI_MMQ64_LONG_BPS : 1;
            const uint64_t fit = t64 <= sl ? sl / t64 : 1;
            ks                 = ks < k64 ? ks : k64;
            ks                 = ks < fit ? ks : fit;
            ks                 = ks < 1 ? 1 : ks;
        }
        a.bps             = a.nbk == 0 ? 1 : (uint32_t) ((a.nbk + ks - 1) / ks);
        a.splits          = a.nbk == 0 ? 1 : (a.nbk + a.bps - 1) / a.bps;
        return;
    }
    const uint32_t want = (uint32_t) (cus > 0 ? cus : 256) * MI_MMV_WAVES_PER_CU;
    uint32_t       s    = a.ng == 0 || a.ng >= want ? 1 : (want + a.ng - 1) / a.ng;
    // when one workgroup per row group (its splits added in LDS) still gives the
    // grid enough waves, stop there: no partials, no second launch to add them
    if (MI_MMV_NORED_MIN > 0 && s > 8 && (uint64_t) a.ng * 8 >= (uint64_t) (cus > 0 ? cus : 256) * MI_MMV_NORED_MIN) {
        s = 8;
    }
    if (s > a.nbk) {
        s = a.nbk;
    }
    if (s < 1) {
        s = 1;
    }
    a.wpg    = s < 8 ? s : 8;
    a.splits = (s + a.wpg - 1) / a.wpg;                       // workgroups per row group
    a.bps    = a.nbk == 0 ? 1 : (a.nbk + a.splits * a.wpg - 1) / (a.splits * a.wpg);
    a.one    = a.m == 1 && a.nbk > 0 && mmv_one_launch(a.nbk, a.ng);
}

static size_t al256(size_t v) {
    return (v + 255) & ~(size_t) 255;
}

size_t mul_mat_q8_0_workspace(const MmvArgs & a) {
    size_t b = al256((size_t) a.mp * a.k) + al256((size_t) a.mp * a.nbk * 4);
    if (a.splits > 1) {  // partials: [splits][m][npad], or [splits][mp][npad] for the matrix kernel
        b += al256((size_t) a.splits * (a.m > 8 ? a.mp : a.m) * a.npad * 4);
    }
    return b;
}

void mul_mat_q8_0_bind(MmvArgs & a, char * ws) {
    a.xq  = ws;
    a.xd  = (float *) (ws + al256((size_t) a.mp * a.k));
    char * p = (char *) a.xd + al256((size_t) a.mp * a.nbk * 4);
    a.part = a.splits > 1 ? (float *) p : nullptr;
}

int launch_q8_0_repack(const char * src, int64_t nb1, uint32_t k, uint32_t n, char * dst, hipStream_t s) {
    const uint32_t nbk   = k / 32, ng = (n + 63) / 64;
    const uint64_t total = (uint64_t) ng * nbk * 64;
    if (total == 0) {
        return MI_OK;
    }
    MI_LAUNCH(k_q8_0_repack, dim3((uint32_t) ((total + 255) / 256)), dim3(256), 0, s, src, nb1, n, nbk, ng,
                       dst);
    return MI_OK;
}

#ifndef MI_QXN8_MIN_ROWS
#define MI_QXN8_MIN_ROWS 4096  // rows of x from which the norm prologue takes 8 rows per workgroup
#endif
template <bool ADD>
static void launch_quant_x_norm8(const MmvArgs & a, hipStream_t s) {
    const dim3 grid((a.m + 7) / 8);
    if (a.nbk <= 4 * 8) {
        MI_LAUNCH((k_mmv_quant_x_norm8<8, ADD>), grid, dim3(256), 0, s, a);
    } else if (a.nbk <= 4 * 16) {
        MI_LAUNCH((k_mmv_quant_x_norm8<16, ADD>), grid, dim3(256), 0, s, a);
    } else if (a.nbk <= 4 * 24) {
        MI_LAUNCH((k_mmv_quant_x_norm8<24, ADD>), grid, dim3(256), 0, s, a);
    } else {
        MI_LAUNCH((k_mmv_quant_x_norm8<32, ADD>), grid, dim3(256), 0, s, a);
    }
}

// Whether a workgroup of the one-launch kernel would write what another still reads: y, or
// the residual sum (the entry point refuses it over its addends only), sharing memory with
// an operand that every workgroup reads, or with each other. Then the prologue keeps its
// own launch, whose one workgroup has read the operands in its order before y is written.
static bool mmv1_overlaps(const MmvArgs & a) {
    const uintptr_t kb = (uintptr_t) a.k * 4;
    auto over = [&](const void * p, uintptr_t bytes, const void * q) {  // q: k floats
        return p != nullptr && q != nullptr && (uintptr_t) q < (uintptr_t) p + bytes && (uintptr_t) p < (uintptr_t) q + kb;
    };
    for (const void * q : { (const void *) a.x, (const void *) a.ab, (const void *) a.g, (const void *) a.u,
                            (const void *) a.nw, (const void *) a.gate, (const void *) a.msc, (const void *) a.msh }) {
        if (over(a.y, (uintptr_t) a.n * 4, q) || over(a.sum, kb, q)) {
            return true;
        }
    }
    return over(a.y, (uintptr_t) a.n * 4, a.sum);
}

int launch_mul_mat_q8_0(const MmvArgs & a, hipStream_t s) {
    if (a.n == 0 || a.m == 0) {
        return MI_OK;
    }
    if (a.one && !mmv1_overlaps(a)) {
        MI_LAUNCH(k_mmv1_q8_0, dim3(a.ng), dim3(512), (size_t) a.nbk * 36 + (size_t) a.splits * 8 * 256, s, a);
        return MI_OK;
    }
    if (a.nw && a.m >= (uint32_t) MI_QXN8_MIN_ROWS && a.nbk <= 4 * 32) {
        // long x: 8 rows per workgroup, x held in registers (4 * NBW blocks per row at most)
        if (a.ab) {
            launch_quant_x_norm8<true>(a, s);
        } else {
            launch_quant_x_norm8<false>(a, s);
        }
    } else if (a.nw) {
        MI_LAUNCH(k_mmv_quant_x_norm, dim3(a.m), dim3(256), 0, s, a);
    } else {
        const uint64_t threads = ((uint64_t) a.m * a.nbk + MI_QX_U - 1) / MI_QX_U * 8;
        MI_LAUNCH(k_mmv_quant_x, dim3((uint32_t) ((threads + 255) / 256)), dim3(256), 0, s, a);
    }
    if (a.m > 8) {
        if (a.tile == 64) {
            MI_LAUNCH(k_mmq64_q8_0, dim3((a.n + 63) / 64 * ((a.m + 63) / 64) * a.splits), dim3(512), 0, s, a);
        } else {
            MI_LAUNCH(k_mmq_q8_0, dim3((a.n + 127) / 128, a.mp / 128, a.splits), dim3(256), 0, s, a);
        }
        if (a.splits > 1) {
            const uint64_t outs = (uint64_t) a.m * a.n;
            MI_LAUNCH(k_mmq_reduce, dim3((uint32_t) ((outs + 255) / 256)), dim3(256), 0, s, a);
        }
        return MI_OK;
    }
    const dim3   grid(a.ng, a.splits), blk(64 * a.wpg);
    const size_t lds = a.wpg > 1 ? (size_t) a.wpg * a.m * 64 * 4 : 0;
    switch (a.m) {
        case 1: MI_LAUNCH(k_mmv_q8_0<1>, grid, blk, lds, s, a); break;
        case 2: MI_LAUNCH(k_mmv_q8_0<2>, grid, blk, lds, s, a); break;
        case 3: MI_LAUNCH(k_mmv_q8_0<3>, grid, blk, lds, s, a); break;
        case 4: MI_LAUNCH(k_mmv_q8_0<4>, grid, blk, lds, s, a); break;
        case 5: MI_LAUNCH(k_mmv_q8_0<5>, grid, blk, lds, s, a); break;
        case 6: MI_LAUNCH(k_mmv_q8_0<6>, grid, blk, lds, s, a); break;
        case 7: MI_LAUNCH(k_mmv_q8_0<7>, grid, blk, lds, s, a); break;
        case 8: MI_LAUNCH(k_mmv_q8_0<8>, grid, blk, lds, s, a); break;
        default: return MI_ERR_UNSUPPORTED;
    }
    if (a.splits > 1) {
        const dim3 rg((a.m * a.npad + 255) / 256);
        switch (a.m) {
            case 1: MI_LAUNCH(k_mmv_reduce<1>, rg, dim3(256), 0, s, a); break;
            case 2: MI_LAUNCH(k_mmv_reduce<2>, rg, dim3(256), 0, s, a); break;
            case 3: MI_LAUNCH(k_mmv_reduce<3>, rg, dim3(256), 0, s, a); break;
            case 4: MI_LAUNCH(k_mmv_reduce<4>, rg, dim3(256), 0, s, a); break;
            case 5: MI_LAUNCH(k_mmv_reduce<5>, rg, dim3(256), 0, s, a); break;
            case 6: MI_LAUNCH(k_mmv_reduce<6>, rg, dim3(256), 0, s, a); break;
            case 7: MI_LAUNCH(k_mmv_reduce<7>, rg, dim3(256), 0, s, a); break;
            default: MI_LAUNCH(k_mmv_reduce<8>, rg, dim3(256), 0, s, a); break;
        }
    }
    return MI_OK;
}

}  // namespace mi
