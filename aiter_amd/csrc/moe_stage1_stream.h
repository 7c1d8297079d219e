// MoE stage 1 (gate / up projection, activation, MXFP4 output quant) for decode
// batches: few rows per expert, so the launch is a stream of the touched
// experts' weights (257 experts, 7168 x 2 * 256, 64 tokens: 420 MB, 65 us at
// 6.5 TB/s; the flat tile kernel takes 86 us, this one 66).  The flat kernel
// keeps one K stage per workgroup ahead and meets at a barrier per stage; here
// each wave has 8 KB of weights in flight and none to wait for.
#pragma once
#include <algorithm>

#include "gemm_flat.h"

namespace aiter_amd {

struct S1Ops {
    i32x4_t b[4][2];   // gate 16-column halves 0, 1, up halves 0, 1; k-step
    i32x4_t a[2];      // k-step
    int sg, su, sa;    // scale dwords: byte 2 * k-step + 16-row half
};

// An item is the 16-row half C of a unit of 32 sorted rows (one scale group, one
// expert) by 32 gate and the same 32 up columns: a whole MXFP4 output block.
// NWK waves of the workgroup share its K; each streams its weights straight to
// registers, one 256-element window ahead, with no barrier until its sums are
// added through LDS in wave order.
template <int NWK, int C>
AA_DEV void stage1_stream_body(const GemmParams& p, const MoeParams& mq, int units, int block,
                               f32x4_t (*part)[4][64]) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kpart = wave % NWK;
    const int cols = mq.inter / 32;
    const int item = block * (8 / NWK) + wave / NWK;
    const int u = item / cols, cg = item % cols;
    const int pos0 = 32 * u;

    const bool in = u < units && pos0 + (lane & 31) < mq.sorted_len;
    const int id = in ? mq.sorted_ids[pos0 + (lane & 31)] : mq.token_num;
    const float wgt = (in && mq.sorted_w) ? mq.sorted_w[pos0 + (lane & 31)] : 1.0f;
    const int e = __builtin_amdgcn_readfirstlane(u < units ? mq.sorted_eids[pos0 / mq.sort_bs] : -1);
    const bool live = e >= 0 && e < mq.n_experts;
    auto valid = [&](int x) { return (x & 0xffffff) < mq.token_num && (int)((unsigned)x >> 24) < mq.topk; };
    const uint32_t rows = (live ? (uint32_t)__ballot(valid(id)) : 0) >> (16 * C) & 0xffffu;
    const int rid = __shfl(id, 16 * C + (lane & 15));
    const float w = __shfl(wgt, 16 * C + (lane & 15));

    const int nkp = p.K / 256;
    const int per = (nkp + NWK - 1) / NWK;
    const int k0 = kpart * per, k1 = min(k0 + per, nkp);
    const __amdgpu_buffer_rsrc_t a_rsrc = make_rsrc(p.A, mq.a_rows * p.lda);
    const uint8_t* we = p.B + (int64_t)max(e, 0) * mq.b_expert_bytes;
    const uint8_t* se = p.Bs + (int64_t)max(e, 0) * mq.bs_expert_bytes;
    const uint8_t* bp[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) bp[t] = we + (int64_t)((t >> 1) * mq.inter + 32 * cg + 16 * (t & 1)) * p.ldb;
    const uint8_t* sg = se + (int64_t)cg * 32 * p.sb_stride;
    const uint8_t* su = se + (int64_t)(mq.inter / 32 + cg) * 32 * p.sb_stride;
    const uint8_t* sa = p.As + (int64_t)u * 32 * p.sa_stride;

    f32x4_t acc[4] = {};
    if (rows) {
        const int a_off = valid(rid) ? (rid & 0xffffff) * (int)p.lda + (lane >> 4) * 16 : (int)(mq.a_rows * p.lda);
        auto load = [&](int kp, S1Ops& o) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int s = 0; s < 2; ++s)
                    o.b[t][s] = load_once<i32x4_t>(bp[t] + kp * 2048 + s * 1024 + lane * 16);
            o.sg = load_once<int>(sg + kp * 256 + lane * 4);
            o.su = load_once<int>(su + kp * 256 + lane * 4);
            o.sa = *reinterpret_cast<const int*>(sa + kp * 256 + lane * 4);
#pragma unroll
            for (int s = 0; s < 2; ++s)
                o.a[s] = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, a_off + s * 64, kp * 128, 0);
        };
        auto mma = [&](const S1Ops& o) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    acc[t] = mma_step<kFp4, kFp4>(&o.b[t][s], &o.a[s], acc[t], t < 2 ? o.sg : o.su, 2 * s + (t & 1),
                                                  o.sa, 2 * s + C);
        };
        if (k0 < k1) {
            S1Ops o0, o1;
            load(k0, o0);
            int k = k0;
            for (; k + 2 < k1; k += 2) {
                load(k + 1, o1);
                mma(o0);
                load(k + 2, o0);
                mma(o1);
            }
            if (k + 1 < k1) {
                load(k + 1, o1);
                mma(o0);
                mma(o1);
            } else {
                mma(o0);
            }
        }
    }
    if constexpr (NWK > 1) {
        if (rows && kpart)
#pragma unroll
            for (int t = 0; t < 4; ++t) part[wave][t][lane] = acc[t];
        __syncthreads();
        if (kpart) return;
        if (rows)
#pragma unroll
            for (int q = 1; q < NWK; ++q)
#pragma unroll
                for (int t = 0; t < 4; ++t) acc[t] += part[wave + q][t][lane];
    }
    // lane: row lane % 16 of the half, columns 16 j + 4 (lane / 16) + r
    const int pos = pos0 + 16 * C + (lane & 15);
    if (!live || pos >= mq.sorted_len) return;
    uint32_t raw[2][2];
    float amax = 1e-10f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = moe_act(acc[j][r] * w, mq.act) * (acc[2 + j][r] * w);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            raw[j][h] = pack_bf16x2(v[2 * h], v[2 * h + 1]);
            amax = __builtin_fmaxf(amax, __builtin_fabsf(bf16_bits_to_f32(raw[j][h] & 0xffffu)));
            amax = __builtin_fmaxf(amax, __builtin_fabsf(bf16_bits_to_f32(raw[j][h] >> 16)));
        }
    }
    amax = __builtin_fmaxf(amax, __shfl_xor(amax, 16));
    amax = __builtin_fmaxf(amax, __shfl_xor(amax, 32));
    uint32_t byte = mx::e8m0_byte<mx::kRoundUp>(amax, 1.0f / 6.0f, 0.25f, 0u, 2u);
    uint32_t code[2] = {0, 0};
    const bool ok = valid(rid);
    if (!ok || (mq.q_w && mq.q_w[pos] == 0.0f)) {
        byte = 0;
    } else if (byte != 0u && byte != 255u) {
        const float ds = __builtin_bit_cast(float, byte << 23);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            code[j] = mx::cvt_fp4_pair<uint16_t>(code[j], raw[j][0], 0.f, 0.f, ds, 0);
            code[j] = mx::cvt_fp4_pair<uint16_t>(code[j], raw[j][1], 0.f, 0.f, ds, 1);
        }
    } else {
        const float inv = mx::inv_scale_from_byte(byte);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                code[j] |= mx::f32_to_e2m1(bf16_bits_to_f32(raw[j][r >> 1] >> (16 * (r & 1)) & 0xffffu) * inv)
                           << (4 * r);
    }
    if (ok) {
        uint8_t* row = mq.q_out + ((int64_t)(rid & 0xffffff) * mq.topk + (int)((unsigned)rid >> 24)) * mq.q_stride +
                       cg * 16 + 2 * (lane >> 4);
#pragma unroll
        for (int j = 0; j < 2; ++j) *reinterpret_cast<uint16_t*>(row + 8 * j) = (uint16_t)code[j];
    }
    if (lane < 16) mq.q_scale[mx::scale_shuffle_idx(mq.q_scale_n_pad, pos, cg)] = (uint8_t)byte;
}

// Waves per item: the most (up to 8) whose items fit `waves`, 8 per CU: where some
// CUs have two workgroups those end last (257 experts, 7168 x 2 * 256: 32 tokens
// 57.3 us with 1 wave per item, 70.0 with 2, 63.4 with 4).  The items are those of
// the units that hold rows, which only the sort knows: routing may be uneven (64
// tokens on 18 experts 19.9 us; 91 with the waves that even routing would
// leave, 30 by the flat kernel).
template <int C>
AA_DEV void stage1_stream_part(const GemmParams& p, const MoeParams& mq, int waves, int units,
                               f32x4_t (*part)[4][64]) {
    const int items = units * (mq.inter / 32), block = blockIdx.x;
    if (items * 8 <= waves) stage1_stream_body<8, C>(p, mq, units, block, part);
    else if (items * 4 <= waves) stage1_stream_body<4, C>(p, mq, units, block, part);
    else if (items * 2 <= waves) stage1_stream_body<2, C>(p, mq, units, block, part);
    else stage1_stream_body<1, C>(p, mq, units, block, part);
}

// blockIdx.y 0: first halves; 1: second halves likewise, or 1 to 8: second halves
// with 8 waves per item
__global__ __launch_bounds__(512, 4) void moe_stage1_stream_kernel(GemmParams p, MoeParams mq, int waves) {
    __shared__ f32x4_t part[8][4][64];
    const int units = __builtin_amdgcn_readfirstlane(min((mq.num_valid[0] + 31) / 32, (mq.sorted_len + 31) / 32));
    if (blockIdx.y == 0) stage1_stream_part<0>(p, mq, waves, units, part);
    else if (gridDim.y == 2) stage1_stream_part<1>(p, mq, waves, units, part);
    else stage1_stream_body<8, 1>(p, mq, units, (blockIdx.y - 1) * gridDim.x + blockIdx.x, part);
}

// `units`: the most that can hold rows.  The grid has room for one wave of each of
// their items, or for all the waves that the CUs take one workgroup of.
inline void launch_stage1_stream(const GemmParams& p, const MoeParams& mq, int64_t units, int64_t entries, int cus,
                                 hipStream_t st) {
    const int64_t items = units * (mq.inter / 32);
    const int64_t wgs = std::max((items + 7) / 8, std::min<int64_t>(items, cus));
    // Up to 16 entries fill no second half of a unit, up to 16 tokens hardly any.
    // Above, a few experts with more rows than that are usual, and one workgroup
    // that walks such a half's whole K beside a first half on its CU ends last (64
    // tokens, one expert with 17 rows: 95 us, with 8 waves per item 68).
    const dim3 grid((unsigned)wgs, entries <= 16 ? 1 : mq.token_num <= 16 ? 2 : 9);
    moe_stage1_stream_kernel<<<grid, 512, 0, st>>>(p, mq, 8 * (int)std::min<int64_t>(wgs, cus));
}

}  // namespace aiter_amd
