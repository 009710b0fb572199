// Noisy-device array read for reads whose input digits do not fit the registers of a wave
// beside its conductance terms: 64-row reads with six to eight input slices (the default
// Config's one-bit slices on 64x64 arrays) and 128-row reads.  Linear converters, programming
// noise and stuck-at faults.
//
// The model, the two fp16 terms and the converter are noisy_mfma.hip's.  What differs is
// where the operands live: a workgroup of up to four waves reads the same 32 vectors through
// 32 columns per wave, and the digits of those vectors (every input slice of one read) are
// built once per read in LDS in MFMA operand order, [slice][16-row step][64 lanes] of 16 bytes,
// so each ds_read_b128 is conflict-free.  A wave keeps one weight slice's terms in registers
// and walks the input slices over them: 2*KS MFMAs, KS LDS reads and three VALU instructions
// per output and pair of slices.
//
// Each term is two fp16, 22 bits of the FP32 conductance's 24.  Terms carry a power of two, plan.k1[w] = S_w * V*Mw/unit, chosen on the host as large as the
// fp16 range allows: small conductances keep their low term out of fp16's subnormals, and the
// converter takes the scale for nothing (its rounding constant and its limit are scaled by the
// same power, which is exact).  The low terms are accumulated first,
// so that only KS additions round at the full current's magnitude.
//
// Bound: MFMA.  2048^3 under the default Config (64 pairs, two terms: 2.2e12 fp16 operations)
// takes 1.74-1.84 ms, 1.25 PFLOP/s, what an 8192^3 bf16 library product reaches on the same card;
// the general FP32 kernel took 130.9 ms.  128-row reads of the same size: 1.64-1.72 ms
// (127 ms before).  Two column blocks per wave, which halve the LDS reads, measured the same
// there (1.80-1.82 ms) and worse on smaller products (1000x1500x700: 0.30 against 0.26 ms),
// and so did unrolling the slice loop by two or four.
#include <cfloat>

#include "mf_noisy.h"

namespace mf {

template <int KS>
__global__ __launch_bounds__(256, 2) void k_noisy_block(const NoisyPlan plan,
                                                        const NoisyArgs args) {
    constexpr int P = 16 * KS;
    extern __shared__ __align__(16) uint4 digits[];   // [A][KS][64 lanes]
    const int A = plan.n_in, W = plan.n_w;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int waves = blockDim.x >> 6;
    const int lrow = lane & 31, lhalf = lane >> 5;

    u32 vtile, ctile;
    xcd_tile(blockIdx.x + blockIdx.y * gridDim.x, gridDim.x, gridDim.y, vtile, ctile);
    const i64 c0 = (i64(ctile) * waves + wave) * 32;   // chunk-relative first column
    const i64 v0 = i64(vtile) * 32;
    const int G = int(args.G);
    const i64 kp = args.kp;
    const i64 vrows = (args.n - v0) < 32 ? (args.n - v0) : 32;
    const __amdgpu_buffer_rsrc_t qbuf = noisy_buffer(args.q + v0 * kp, vrows * kp);
    const int q_off = lrow * int(kp) + lhalf * 8;
    const bool live = c0 < args.blocks * 32;   // the last workgroup may hold waves past these
    const i64 col_tile = args.c_begin + c0;
    const i64 n_out = v0 + lrow;
    const i64 w_stride = args.CB * i64(G) * NOISY_TERMS * KS * 64;
    const uint4 *frag_base = args.gs + (c0 / 32) * i64(G) * NOISY_TERMS * KS * 64 + lane;

    float acc0[16], acc1[16];   // levels 0 and 1 of the cascade over reads
#pragma unroll
    for (int r = 0; r < 16; ++r) { acc0[r] = 0.0f; acc1[r] = 0.0f; }

    const int g0 = int(args.g_begin + i64(blockIdx.z) * args.g_step);
    const int g1 = int((g0 + args.g_step) < args.g_end ? (g0 + args.g_step) : args.g_end);
    // Wave w builds the digits of the 16-row steps w, w + waves, ..; their codes are loaded a
    // read ahead.
    uint2 qw[KS];
    auto fetch = [&](int g) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            if (ks % waves == wave)
                qw[ks] = make_uint2(
                    __builtin_amdgcn_raw_buffer_load_b32(qbuf, q_off + g * P + ks * 16, 0, 0),
                    __builtin_amdgcn_raw_buffer_load_b32(qbuf, q_off + g * P + ks * 16 + 4, 0, 0));
    };
    if (g0 < g1) fetch(g0);

    for (int g = g0; g < g1; ++g) {
        __syncthreads();   // every wave is done with the previous read's digits
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            if (ks % waves == wave)
                for (int a = 0; a < A; ++a)
                    digits[(a * KS + ks) * 64 + lane] = __builtin_bit_cast(
                        uint4, digits_f16(qw[ks], plan.in_shift[a], plan.in_mask4[a]));
        __syncthreads();
        if (g + 1 < g1) fetch(g + 1);
        if (!live) continue;

        u32 Ti[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) Ti[r] = plan.bias;
        for (int w = 0; w < W; ++w) {
            v8h F[NOISY_TERMS][KS];
            const uint4 *frag = frag_base + i64(g) * NOISY_TERMS * KS * 64 + w * w_stride;
#pragma unroll
            for (int term = 0; term < NOISY_TERMS; ++term)
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    F[term][ks] = __builtin_bit_cast(v8h, frag[(term * KS + ks) * 64]);
            const float magic = plan.magic[w], top = plan.top_magic[w];
            for (int a = 0; a < A; ++a) {
                v8h B[KS];
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
                    B[ks] = __builtin_bit_cast(v8h, digits[(a * KS + ks) * 64 + lane]);
                v16f I = {};
#pragma unroll
                for (int term = NOISY_TERMS - 1; term >= 0; --term)
#pragma unroll
                    for (int ks = 0; ks < KS; ++ks)
                        I = __builtin_amdgcn_mfma_f32_32x32x16_f16(F[term][ks], B[ks], I, 0, 0, 0);
                // Sign-extended here so the compiler sees a 24-bit operand (v_mad_i32_i24).
                const u32 f24 = u32(int(plan.f24[a][w] << 8) >> 8);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float y = __builtin_amdgcn_fmed3f(I[r] + magic, magic, top);
                    const int low = int(__float_as_uint(y) << 8) >> 8;
                    Ti[r] += u32(low) * f24;
                }
            }
        }

        if (args.totals) {
            if (n_out < args.n) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const i64 c = col_tile + (r >> 2) * 8 + lhalf * 4 + (r & 3);
                    if (c < args.ncols)
                        args.out[(n_out * G + g) * args.ldo + c] = float(int(Ti[r]));
                }
            }
            continue;
        }

        // Scale restore (float(T) * xs) * ws and torch's cascade over reads.
        const float xs = n_out < args.n ? args.xscale[n_out * G + g] : 0.0f;
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
            const i64 c = col_tile + qd * 8 + lhalf * 4;
            v4fn ws = {0.0f, 0.0f, 0.0f, 0.0f};
            if (c + 3 < args.ncols) {
                ws = *reinterpret_cast<const v4fn *>(args.wscale + i64(g) * args.ldws + c);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (c + e < args.ncols) ws[e] = args.wscale[i64(g) * args.ldws + c + e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float v = float(int(Ti[qd * 4 + e])) * xs;
                v = v * ws[e];
                acc0[qd * 4 + e] = acc0[qd * 4 + e] + v;
            }
        }
        const int count = g + 1;
        if ((count & 15) == 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc1[r] = acc1[r] + acc0[r];
                acc0[r] = 0.0f;
            }
            if ((count & 255) == 0) {
                // Level 2 of the cascade lives in `out` (more than 255 reads).
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const i64 c = col_tile + (r >> 2) * 8 + lhalf * 4 + (r & 3);
                    if (n_out < args.n && c < args.ncols) {
                        float *dst = args.out + n_out * args.ldo + c;
                        *dst = count == 256 ? acc1[r] : *dst + acc1[r];
                    }
                    acc1[r] = 0.0f;
                }
            }
        }
    }
    if (args.totals || !live || n_out >= args.n) return;

    bool finite = true;
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
        const i64 c = col_tile + qd * 8 + lhalf * 4;
        float *dst = args.out + n_out * args.ldo + c;
        v4fn v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float s = acc0[qd * 4 + e] + acc1[qd * 4 + e];
            if (g1 >= 256 && c + e < args.ncols) s = s + dst[e];
            v[e] = s;
            finite = finite && (c + e >= args.ncols || fabsf(s) <= FLT_MAX);
        }
        if (c + 3 < args.ncols) {
            *reinterpret_cast<v4fn *>(dst) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < args.ncols) dst[e] = v[e];
        }
    }
    if (!finite && args.status) atomicOr(args.status, u32(MF_STATUS_OUTPUT));
}

template __global__ void k_noisy_block<4>(const NoisyPlan, const NoisyArgs);
template __global__ void k_noisy_block<8>(const NoisyPlan, const NoisyArgs);

}  // namespace mf
