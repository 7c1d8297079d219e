// MoE stage 2 (down projection) with the sum over a token's slots in the same
// launch, for decode batches (up to 128 tokens), short K (K = inter_dim of 256
// or 512) and MXFP4 A.
//
// Bound: the touched experts' weights, read once (257 experts, 7168 x 256, 100
// tokens: 243 MB, 37 us at 6.5 TB/s); with one row per routed pair and a sum
// the same call also writes and reads 26 MB and starts twice (53 + 4.5 us, here
// 45), and below 128 rows packed-bf16 atomics went to memory one dword at a
// time (8 tokens 22 us, here 14).  f32 adds into one shared LDS copy were the
// limit of an earlier form (about 169 clocks per wave instruction); a wave's
// own copy takes a 16-byte read, four adds and a write (30 clocks).
#pragma once
#include <utility>

#include "gemm_flat.h"

namespace aiter_amd {

constexpr int kS2ReduceTokens = 128;

template <int KW, int CB>
struct S2Ops {
    i32x4_t b[CB][2 * KW];  // 16-column block, k-step
    i32x4_t a[2][2 * KW];   // 16-row half, k-step
    int sb[KW], sa[KW];     // scale dwords: byte 2 * (k-step & 1) + half
    uint32_t mask;          // rows of the unit that name a token (0: nothing loaded)
    int id;                 // entry of row lane % 32
    float w;
};

// A workgroup owns C = 16 CB output columns (CB = 1: half BH of a 32-row scale
// group); its waves deal out the units of 32 sorted rows (one scale group, one
// expert each), keep the loads of D units in flight, and add each row's product
// into the wave's own f32 copy of the [tokens, C] result in LDS.  At the end
// the copies are added in wave order and every token's row is stored once: no
// atomics, no cleared output, no second launch.
template <int KW, int CB, int BH, int NW, int D>
AA_DEV void stage2_reduce_body(const GemmParams& p, const MoeParams& mq, float* sums) {
    constexpr int C = 16 * CB, PC = C / 4;   // columns, 16-byte pieces of a row
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.x * C;
    const int nt = mq.token_num;
    float* own = sums + wave * nt * C;
    for (int i = lane; i < nt * PC; i += 64) reinterpret_cast<f32x4_t*>(own)[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // a row's pieces are rotated by token against bank conflicts
    auto turn = [](int tl) { return CB == 2 ? tl & 7 : (tl >> 1) & 3; };

    const int units = min((mq.num_valid[0] + 31) / 32, (mq.sorted_len + 31) / 32);
    const __amdgpu_buffer_rsrc_t a_rsrc = make_rsrc(p.A, mq.a_rows * p.lda);
    const int a_out = (int)(mq.a_rows * p.lda);   // reads zeros

    struct Entry {
        int id, e;
        float w;
    };
    auto load_entry = [&](int u) {
        const int pos = 32 * u + (lane & 31);
        const bool in = u < units && pos < mq.sorted_len;
        Entry t;
        t.id = in ? mq.sorted_ids[pos] : nt;
        t.w = (in && mq.sorted_w) ? mq.sorted_w[pos] : 1.0f;
        t.e = u < units ? mq.sorted_eids[32 * u / mq.sort_bs] : -1;
        return t;
    };
    auto valid = [&](int id) { return (id & 0xffffff) < nt && (int)((unsigned)id >> 24) < mq.topk; };
    auto load_ops = [&](int u, const Entry& t, S2Ops<KW, CB>& o) {
        o.id = t.id;
        o.w = t.w;
        const int e = __builtin_amdgcn_readfirstlane(t.e);
        o.mask = (e < 0 || e >= mq.n_experts) ? 0 : (uint32_t)__ballot(valid(t.id));
        if (o.mask == 0) return;
        const uint8_t* b = p.B + (int64_t)e * mq.b_expert_bytes + (int64_t)n0 * p.ldb;
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int s = 0; s < 2 * KW; ++s)
                o.b[j][s] = load_once<i32x4_t>(b + j * 16 * p.ldb + s * 1024 + lane * 16);
        const uint8_t* bs = p.Bs + (int64_t)e * mq.bs_expert_bytes + (int64_t)(n0 / 32) * 32 * p.sb_stride;
        const uint8_t* as = p.As + (int64_t)u * 32 * p.sa_stride;
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            o.sb[k] = load_once<int>(bs + k * 256 + lane * 4);
            o.sa[k] = *reinterpret_cast<const int*>(as + k * 256 + lane * 4);
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if ((o.mask >> (16 * c) & 0xffffu) == 0) continue;
            const int rid = __shfl(t.id, 16 * c + (lane & 15));
            const int row = (rid & 0xffffff) * mq.topk + (int)((unsigned)rid >> 24);
            const int off = valid(rid) ? row * (int)p.lda + (lane >> 4) * 16 : a_out;
#pragma unroll
            for (int s = 0; s < 2 * KW; ++s)
                o.a[c][s] = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, off + s * 64, 0, 0);
        }
    };
    auto add_unit = [&](const S2Ops<KW, CB>& o) {
        if (o.mask == 0) return;
        // a token with two slots on one expert may have two rows in one half: their
        // adds would meet in one read-modify-write, so such a unit goes row by
        // row (rotations by 1..8 inside each 16 lanes compare every pair)
        const int tok = valid(o.id) ? o.id & 0xffffff : -1 - lane;
        bool same = false;
        [&]<int... R>(std::integer_sequence<int, R...>) {
            ((same |= __builtin_amdgcn_update_dpp(0, tok, 0x121 + R, 0xf, 0xf, false) == tok), ...);
        }(std::make_integer_sequence<int, 8>{});
        const bool twice = __ballot(same) != 0;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            if ((o.mask >> (16 * c) & 0xffffu) == 0) continue;
            f32x4_t acc[CB] = {};
#pragma unroll
            for (int s = 0; s < 2 * KW; ++s)
#pragma unroll
                for (int j = 0; j < CB; ++j)
                    acc[j] = mma_step<kFp4, kFp4>(&o.b[j][s], &o.a[c][s], acc[j], o.sb[s / 2], 2 * (s & 1) + BH + j,
                                                  o.sa[s / 2], 2 * (s & 1) + c);
            // lane: row lane % 16 of the half, columns 16 j + 4 (lane / 16) + 0..3
            const int rid = __shfl(o.id, 16 * c + (lane & 15));
            const float w = __shfl(o.w, 16 * c + (lane & 15));
            const int tl = rid & 0xffffff;
            f32x4_t* row = reinterpret_cast<f32x4_t*>(own + tl * C);
            const int q = (lane >> 4) ^ turn(tl);
            if (!twice) {
                if (valid(rid))
#pragma unroll
                    for (int j = 0; j < CB; ++j) row[q ^ (4 * j)] += acc[j] * w;
            } else {
                for (int r = 0; r < 16; ++r)
                    if ((lane & 15) == r && valid(rid)) {
#pragma unroll
                        for (int j = 0; j < CB; ++j) row[q ^ (4 * j)] += acc[j] * w;
                        asm volatile("" ::: "memory");
                    }
            }
        }
    };

    S2Ops<KW, CB> o[D];
    Entry t[D];
#pragma unroll
    for (int d = 0; d < D; ++d) t[d] = load_entry(wave + d * NW);
#pragma unroll
    for (int d = 0; d < D; ++d) load_ops(wave + d * NW, t[d], o[d]);
    Entry next = load_entry(wave + D * NW);
    for (int u = wave; u < units; u += D * NW) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            add_unit(o[d]);
            load_ops(u + (d + D) * NW, next, o[d]);
            next = load_entry(u + (d + D + 1) * NW);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nt * (PC / 2); i += 64 * NW) {
        const int tl = i / (PC / 2), q = i % (PC / 2) * 2;
        f32x4_t v[2] = {};
#pragma unroll
        for (int k = 0; k < NW; ++k) {
            const f32x4_t* src = reinterpret_cast<const f32x4_t*>(sums + (k * nt + tl) * C);
            v[0] += src[q ^ turn(tl)];
            v[1] += src[(q + 1) ^ turn(tl)];
        }
        i32x4_t r;
        r[0] = (int)pack_bf16x2(v[0][0], v[0][1]);
        r[1] = (int)pack_bf16x2(v[0][2], v[0][3]);
        r[2] = (int)pack_bf16x2(v[1][0], v[1][1]);
        r[3] = (int)pack_bf16x2(v[1][2], v[1][3]);
        *reinterpret_cast<i32x4_t*>(mq.out + (int64_t)tl * mq.out_stride + n0 + 4 * q) = r;
    }
}

template <int KW, int CB, int NW, int D, int T, int MINW>
__global__ __launch_bounds__(64 * NW, MINW) void moe_stage2_reduce_kernel(GemmParams p, MoeParams mq) {
    __shared__ __attribute__((aligned(16))) float sums[NW * T * 16 * CB];
    if constexpr (CB == 1)
        if (blockIdx.x & 1) return stage2_reduce_body<KW, 1, 1, NW, D>(p, mq, sums);
    stage2_reduce_body<KW, CB, 0, NW, D>(p, mq, sums);
}

// 32 columns per workgroup where that leaves three quarters of the CUs with
// one, else 16; 16 waves while their copies of the result fit the LDS, then 8
// (K = 512 needs the registers of 8 waves)
inline void launch_stage2_reduce(const GemmParams& p, const MoeParams& mq, int cus, hipStream_t st) {
    const bool wide = p.N / 32 * 4 >= cus * 3;
    const dim3 grid((unsigned)(p.N / (wide ? 32 : 16)));
    if (p.K == 512) {
        if (wide) moe_stage2_reduce_kernel<2, 2, 8, 2, 128, 2><<<grid, 512, 0, st>>>(p, mq);
        else moe_stage2_reduce_kernel<2, 1, 8, 3, 128, 2><<<grid, 512, 0, st>>>(p, mq);
    } else if (!wide) {
        moe_stage2_reduce_kernel<1, 1, 16, 3, 128, 4><<<grid, 1024, 0, st>>>(p, mq);
    } else if (mq.token_num <= 64) {
        moe_stage2_reduce_kernel<1, 2, 16, 2, 64, 4><<<grid, 1024, 0, st>>>(p, mq);
    } else {
        moe_stage2_reduce_kernel<1, 2, 8, 4, 128, 2><<<grid, 512, 0, st>>>(p, mq);
    }
}

}  // namespace aiter_amd
