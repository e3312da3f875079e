// decode_stream.hip — paged decode attention for fp16 queries over fp16 caches
// at head_dim 64, 80, 96, 112 or 128 with groups of up to 32 query heads, and
// over FP8 caches at head_dim 128 with groups of up to 8, both products on the
// matrix cores (gfx950); and all in fp32 at head_dim 64, groups of up to 32 (of up to
// four where stream_f32_pays says so).
// Semantics as in decode.hip (the reference's src/attention/
// paged_attention.cu:13-82).
//
// A wave streams the K and V rows of its tokens through LDS, 32 tokens a step,
// with direct global->LDS loads (global_load_lds_dwordx4, 1 KiB per wave
// instruction) into a ring that is the wave's own: no barrier, no registers
// held by loads in flight, and a load waits only for its own stage
// (s_waitcnt vmcnt counted in asm).  A step then costs, whatever the group:
//   S^T = K Q^T   v_mfma_f32_16x16x32_f16 (and one 16x16x16 when head_dim is
//                 an odd multiple of 16): A = K rows from LDS, B = Q in
//                 registers (columns = the group's heads, 16 per tile);
//   softmax       lane-local on the S^T layout (lane l: head l % 16, keys
//                 4 (l / 16) + e of each 16-key half);
//   O^T += V^T P^T  A = V^T by ds_read_b64_tr_b16 from the row-major tile,
//                 B = P^T straight from the S^T registers, so the weights
//                 never leave the lane and the accumulators are head_dim / 4
//                 registers per 16 heads.
// FP8: codes become fp16 exactly (v_cvt_scalef32_pk_f16_fp8, scale 1) as they
// are read from LDS, V^T by ds_read_b64_tr_b8; the token's K scale multiplies
// the logit, its V scale the weight.
// fp32: v_mfma_f32_16x16x4_f32 for both products, its k slots chosen so that a
// lane's 16 bytes of a row feed four of them and the weights stay in place;
// weights and sums in fp32.
// Before: the VALU kernels of head_dim 64 and the generic shapes spent ~300
// instructions per 16 tokens and held 4 KiB of loads per wave, waited for in
// turn; head_dim 128's kernel ran P V on the VALU (packed dot products, 16 G
// of them and as many accumulators per 16 tokens), which left FP8 groups of 7
// one chunk in flight at two waves per SIMD: 178 us where it now takes 125.
#include <atomic>
#include <type_traits>

#include "common.hpp"
#include "decode_common.hpp"
#include "launch.hpp"

namespace vkv {
namespace dec {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr int kStep = 32;            // tokens per step (the k of the P V products)

// LDS tile of a step's K (or V) rows: row-major, unpadded (a direct load
// writes lane L's 16 bytes at 16 L).  Where a row is a power of two of 16-byte
// chunks, chunk c of row r sits at slot c ^ key(r): the operand reads take one
// chunk column of 16 rows, which would otherwise meet in the same banks.
// (Rows of 160, 192 or 224 bytes are spread by their own stride.)
template <int D, int KVT>
struct Tile {
    static constexpr bool FP8 = KVT == kFp8;
    static constexpr bool F32 = KVT == kF32;
    static constexpr int ROW = D * KvTraits<KVT>::bytes;
    static constexpr int CH = ROW / 16;
    static constexpr int NI = kStep * CH / 64;  // direct loads per tile
    static constexpr int BYTES = kStep * ROW;
    static constexpr int STAGE = 2 * BYTES + (FP8 ? 8 * kStep : 0);  // K, V, then the K and V scales
    static constexpr int LOADS = 2 * NI + (FP8 ? 1 : 0);             // wave loads per stage
    static constexpr bool SWZ = (CH & (CH - 1)) == 0;
    static constexpr int KS = D / 32;       // 32-dim MFMA steps of K Q^T
    static constexpr bool HALF = D % 32 != 0;  // and a 16-dim one
    static constexpr int DT = D / 16;       // dim tiles of O^T
    static_assert(D % 16 == 0 && kStep * CH % 64 == 0, "whole loads");
    static_assert(!FP8 || (SWZ && KS % 2 == 0), "FP8 operands are pairs of 8 codes of one chunk");
    static_assert(!F32 || D == 64, "the fp32 dim tiles hold dims 4 m + t, m < 16");
    __device__ static __forceinline__ int slot(int row, int chunk) {
        return SWZ ? chunk ^ (row / (16 / (SWZ ? CH : 16)) % CH) : chunk;
    }
    __device__ static __forceinline__ int off(int row, int chunk) { return row * ROW + slot(row, chunk) * 16; }
    // first of the 8 dims that lane group grp holds for MFMA i of K Q^T
    __device__ static __forceinline__ int dim(int i, int grp) {
        return FP8 ? 16 * (grp * (KS / 2) + i / 2) + 8 * (i % 2) : 32 * i + 8 * grp;
    }
};

__device__ __forceinline__ uint32_t lds_addr(const char* p) {
    typedef const __attribute__((address_space(3))) char* lds_cptr;
    return uint32_t(size_t((lds_cptr)p));
}
// One 16-byte direct load per lane to LDS bytes lds + 16 lane (s_nop 0: the
// wait state between the M0 write and the load that reads it).
// Rows of whole 128-byte lines stream past the caches (nt); other rows share
// lines with the neighbouring heads, whose waves read them soon after.
template <bool NT>
__device__ __forceinline__ void dma16(const char* g, const uint32_t lds) {
    const uint32_t l = __builtin_amdgcn_readfirstlane(lds);
    if constexpr (NT)
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" : : "v"(g), "s"(l) : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(g), "s"(l) : "memory", "m0");
}
// One 4-byte direct load per lane to LDS bytes lds + 4 lane.
__device__ __forceinline__ void dma4(const float* g, const uint32_t lds) {
    const uint32_t l = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(g), "s"(l) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_loads() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
// This wave's LDS operations have completed (before a load overwrites what they read).
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory"); }

__device__ __forceinline__ u32x2 tr_read(const char* lds) {
    typedef __fp16 fp16x4_t __attribute__((__vector_size__(4 * sizeof(__fp16))));
    typedef __attribute__((address_space(3))) fp16x4_t* lds_ptr;
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4f16((lds_ptr)(lds)));
}

// ds_read_b64_tr_b8: within each 16-lane group, lane i receives byte i % 8 of
// the 8-byte chunks addressed by lanes i / 8 + 2 e, e = 0..7 (checked on the
// device).
__device__ __forceinline__ u32x2 tr_read8(const char* lds) {
    typedef int i32x2 __attribute__((ext_vector_type(2)));
    typedef __attribute__((address_space(3))) i32x2* lds_ptr;
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_ptr)(lds)));
}
// Eight e4m3fn codes as their exact fp16 values, in order.
__device__ __forceinline__ half8_t codes8(const uint32_t lo, const uint32_t hi) {
    return __builtin_bit_cast(half8_t, u32x4{fp8x2_to_half2<false>(lo), fp8x2_to_half2<true>(lo),
                                             fp8x2_to_half2<false>(hi), fp8x2_to_half2<true>(hi)});
}

// Attention state of one wave: CT tiles of 16 heads.
template <int D, int CT, int KVT>
struct State {
    using T = Tile<D, KVT>;
    half8_t q[CT][T::F32 ? 1 : T::KS];
    half4_t qh[CT];
    float4_t qf[CT][T::F32 ? D / 16 : 1];
    float m[CT];              // running max of head 16 ct + l % 16, raw logits
    float4_t l[CT];           // weight sums (every element the same; FP8, fp32: element 0, this lane's keys)
    float4_t o[CT][T::DT];    // O^T: lane l holds dims 16 t + 4 (l / 16) + e of head l % 16
                              // (fp32: dims 16 (l / 16) + 4 e + t)
    // Four consecutive dims of head 16 c + l % 16, from dim() on.
    __device__ __forceinline__ float4_t out4(const int c, const int i) const {
        if constexpr (T::F32) return float4_t{o[c][0][i], o[c][1][i], o[c][2][i], o[c][3][i]};
        else return o[c][i];
    }
    __device__ static __forceinline__ int dim(const int i, const int grp) {
        return T::F32 ? 16 * grp + 4 * i : 16 * i + 4 * grp;
    }
};

// Queries need only their element's alignment (any row stride): loads that say
// so (the compiler takes whole-vector loads where the target allows them).
__device__ __forceinline__ u32x4 load_q16(const char* p) {
    typedef u32x4 any_u32x4 __attribute__((aligned(2)));
    return *reinterpret_cast<const any_u32x4*>(p);
}
__device__ __forceinline__ u32x2 load_q8(const char* p) {
    typedef u32x2 any_u32x2 __attribute__((aligned(2)));
    return *reinterpret_cast<const any_u32x2*>(p);
}

// Q as the B operand and an empty state.  Columns past the group read head 0
// and are zeroed; a negative scale is moved into Q (exact sign flip).
template <int D, int CT, int KVT>
__device__ __forceinline__ void init_state(const DecodeArgs& a, State<D, CT, KVT>& st, const int s, const int kvh,
                                           const int G, const int lane) {
    using T = Tile<D, KVT>;
    const int col = lane & 15, grp = lane >> 4;
    const uint32_t flip = a.scale_log2 < 0.0f ? (T::F32 ? 0x80000000u : 0x80008000u) : 0u;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        const int h = 16 * c + col;
        const uint32_t keep = h < G ? 0xFFFFFFFFu : 0u;
        const char* qrow = static_cast<const char*>(a.q) +
                           (query_row(a, s) * a.q_stride + int64_t(kvh * G + (h < G ? h : 0)) * D) * (T::F32 ? 4 : 2);
#pragma unroll
        for (int i = 0; i < (T::F32 ? D / 16 : 0); ++i) {
            u32x4 w = load_q16(qrow + (16 * i + 4 * grp) * 4);
            w = (w ^ u32x4{flip, flip, flip, flip}) & u32x4{keep, keep, keep, keep};
            st.qf[c][i] = __builtin_bit_cast(float4_t, w);
        }
#pragma unroll
        for (int i = 0; i < (T::F32 ? 0 : T::KS); ++i) {
            u32x4 w = load_q16(qrow + T::dim(i, grp) * 2);
            w = (w ^ u32x4{flip, flip, flip, flip}) & u32x4{keep, keep, keep, keep};
            st.q[c][i] = __builtin_bit_cast(half8_t, w);
        }
        if constexpr (T::HALF && !T::F32) {
            u32x2 w = load_q8(qrow + (32 * T::KS + 4 * grp) * 2);
            w = (w ^ u32x2{flip, flip}) & u32x2{keep, keep};
            st.qh[c] = __builtin_bit_cast(half4_t, w);
        }
        st.m[c] = -INFINITY;
        st.l[c] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < T::DT; ++t) st.o[c][t] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
}

// Attends tokens [t0, t0 + n) (n >= 1) of row s at kv head kvh.  ring: NST
// stages of a K and a V tile, this wave's own.  my_block: block ids of
// [win, win + 64) in the row's table, one per lane (0 where out of the pool).
template <int D, int CT, int KVT, int NST>
__device__ __forceinline__ void stream_tokens(const DecodeArgs& a, State<D, CT, KVT>& st, char* ring, const int s,
                                              const int32_t* table, const int ctx, const int kvh, const int t0,
                                              const int n, int win, int my_block, const int lane) {
    using T = Tile<D, KVT>;
    constexpr bool FP8 = T::FP8;
    constexpr int kStage = T::STAGE;
    const int col = lane & 15, grp = lane >> 4;
    const uint32_t slot_stride = uint32_t(a.num_kv_heads) * T::ROW;
    const uint32_t ring_lds = lds_addr(ring);
    const float sc = a.scale_log2 < 0.0f ? -a.scale_log2 : a.scale_log2;
    const int steps = (n + kStep - 1) / kStep;
    // The fused append: the row's last position reads the new token's rows
    // when the append targets that position's slot.
    const bool fused = a.fkey && t0 + n == ctx;
    const int64_t fslot = fused ? int64_t(a.fslots[s]) : -1;

    auto issue = [&](const int step, const int stage) __attribute__((always_inline)) {
        const int last = min(step * kStep + kStep, n) - 1;
        if (block_div(a, t0 + last) - win >= kWave) {  // (wave-uniform)
            win = block_div(a, t0 + step * kStep);
            my_block = 0;
            if (win + lane < a.max_blocks_per_seq) {
                my_block = table[win + lane];
                if (a.num_blocks > 0 && unsigned(my_block) >= unsigned(a.num_blocks)) my_block = 0;
            }
        }
        const bool has_new = fused && step == steps - 1;
        const uint32_t dst = ring_lds + uint32_t(stage * kStage);
#pragma unroll
        for (int i = 0; i < T::NI; ++i) {
            const int row = (i * 64 + lane) / T::CH;
            const uint32_t chunk = uint32_t(T::slot(row, (i * 64 + lane) % T::CH)) * 16;  // (slot is its own inverse)
            // tokens past the end read the last one again (masked below)
            const int tok = t0 + min(step * kStep + row, n - 1);
            const int blk = block_div(a, tok);
            const int64_t slot = int64_t(__shfl(my_block, blk - win, kWave)) * a.block_size + (tok - blk * a.block_size);
            const uint64_t off = uint64_t(slot) * slot_stride + (uint32_t(kvh * T::ROW) + chunk);
            const char* kp = a.kc + off;
            const char* vp = a.vc + off;
            if (has_new && tok == ctx - 1 && slot == fslot) {
                kp = a.fkey + s * a.fkey_stride + kvh * T::ROW + chunk;
                vp = a.fval + s * a.fval_stride + kvh * T::ROW + chunk;
            }
            dma16<T::ROW % 128 == 0>(kp, dst + i * 1024);
            dma16<T::ROW % 128 == 0>(vp, dst + T::BYTES + i * 1024);
        }
        if constexpr (FP8) {
            // lanes 0-31 the K scales of the step's tokens, 32-63 the V scales
            const int tok = t0 + min(step * kStep + (lane & 31), n - 1);
            const int blk = block_div(a, tok);
            const int64_t slot = int64_t(__shfl(my_block, blk - win, kWave)) * a.block_size + (tok - blk * a.block_size);
            dma4((lane < 32 ? a.ks : a.vs) + (slot * a.num_kv_heads + kvh), dst + 2 * T::BYTES);
        }
    };

    const half8_t ones = {1.0f16, 1.0f16, 1.0f16, 1.0f16, 1.0f16, 1.0f16, 1.0f16, 1.0f16};
    auto compute = [&](const int step, const int stage) __attribute__((always_inline)) {
        char* kb = ring + stage * kStage;
        char* vb = kb + T::BYTES;
        const bool tail = step * kStep + kStep > n;
        if (!FP8 && tail) {  // (a code of a clamped row times a zero weight is zero)
            // rows past the end: V zero whatever the slots hold (their weight is 0)
#pragma unroll
            for (int i = 0; i < T::NI; ++i)
                if (step * kStep + (i * 64 + lane) / T::CH >= n) store16(vb + i * 1024 + lane * 16, u32x4{0u, 0u, 0u, 0u});
            wave_lds_sync();
        }
        float4_t sv[CT][2];
        [[maybe_unused]] float4_t half_sv[CT][2];
#pragma unroll
        for (int c = 0; c < CT; ++c) sv[c][0] = sv[c][1] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            if constexpr (T::F32) {
                // v_mfma_f32_16x16x4_f32: lane (col, grp) holds one k slot, dim
                // 16 i + 4 grp + e of product (i, e).  Each product's 4 dims a
                // sum of their own, added in pairs, as the VALU kernel's lanes
                // of 4 dims were: one chain over the 64 dims (and one over all
                // tokens below) doubled its error against 64 bits, chains of
                // 16 still added a tenth to it at contexts of 1 to 300.
                float4_t part[CT][D / 16];
#pragma unroll
                for (int i = 0; i < D / 16; ++i) {
                    const float4_t k = __builtin_bit_cast(float4_t, load16(kb + T::off(16 * hh + col, 4 * i + grp)));
                    float4_t four[CT][4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
#pragma unroll
                        for (int c = 0; c < CT; ++c)
                            four[c][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[e], st.qf[c][i][e],
                                                                              float4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                    for (int c = 0; c < CT; ++c) part[c][i] = (four[c][0] + four[c][1]) + (four[c][2] + four[c][3]);
                }
#pragma unroll
                for (int c = 0; c < CT; ++c) sv[c][hh] = (part[c][0] + part[c][1]) + (part[c][2] + part[c][3]);
            } else if constexpr (FP8) {
#pragma unroll
                for (int j = 0; j < T::KS / 2; ++j) {
                    const u32x4 w = load16(kb + T::off(16 * hh + col, grp * (T::KS / 2) + j));
#pragma unroll
                    for (int c = 0; c < CT; ++c) {
                        sv[c][hh] = __builtin_amdgcn_mfma_f32_16x16x32_f16(codes8(w[0], w[1]), st.q[c][2 * j], sv[c][hh], 0, 0, 0);
                        sv[c][hh] = __builtin_amdgcn_mfma_f32_16x16x32_f16(codes8(w[2], w[3]), st.q[c][2 * j + 1], sv[c][hh], 0, 0, 0);
                    }
                }
            } else {
#pragma unroll
                for (int i = 0; i < T::KS; ++i) {
                    const half8_t k = __builtin_bit_cast(half8_t, load16(kb + T::off(16 * hh + col, 4 * i + grp)));
#pragma unroll
                    for (int c = 0; c < CT; ++c)
                        sv[c][hh] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k, st.q[c][i], sv[c][hh], 0, 0, 0);
                }
            }
            if constexpr (T::HALF && !T::F32) {
                // A product of its own, added on the VALU: accumulated onto the
                // 16x16x32 result right behind it (no wait state between the
                // two shapes in the compiler's code), head_dim 112 gave wrong
                // scores.
                const half4_t k = __builtin_bit_cast(
                    half4_t, *reinterpret_cast<const u32x2*>(kb + (16 * hh + col) * T::ROW + 64 * T::KS + 8 * grp));
#pragma unroll
                for (int c = 0; c < CT; ++c) {
                    const float4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
                    half_sv[c][hh] = __builtin_amdgcn_mfma_f32_16x16x16f16(k, st.qh[c], zero, 0, 0, 0);
                }
            }
        }
        if constexpr (T::HALF) {
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) sv[c][hh] += half_sv[c][hh];
        }
        // FP8: the token's K scale times the logit, its V scale times the weight
        // (lane: keys 16 hh + 4 grp + e)
        [[maybe_unused]] float4_t vsc[2];
        if constexpr (FP8) {
            const float* scales = reinterpret_cast<const float*>(kb + 2 * T::BYTES);
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                const float4_t ksc = *reinterpret_cast<const float4_t*>(scales + 16 * hh + 4 * grp);
                vsc[hh] = *reinterpret_cast<const float4_t*>(scales + kStep + 16 * hh + 4 * grp);
#pragma unroll
                for (int c = 0; c < CT; ++c) sv[c][hh] *= ksc;
            }
        }
        half8_t p[CT];
        [[maybe_unused]] float pf[CT][8];
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = sv[c][e >> 2][e & 3];
            if (tail) {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (step * kStep + 16 * (e >> 2) + 4 * grp + (e & 3) >= n) x[e] = -INFINITY;
            }
            const float mx = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
            // The running max follows every score that passes it, so that weights
            // are at most 1 (letting it lag by 2^8 is no faster here, and its
            // weights round more: error against 64 bits 2.9e-4 for 2.7e-4).
            if (__builtin_amdgcn_ballot_w64(mx > st.m[c])) {
                const float mn = fmaxf(st.m[c], xor_max<32>(xor_max<16>(mx)));
                const float alpha = mn > st.m[c] ? __builtin_amdgcn_exp2f((st.m[c] - mn) * sc) : 1.0f;
                st.m[c] = mn;
                st.l[c] *= alpha;
#pragma unroll
                for (int t = 0; t < T::DT; ++t) st.o[c][t] *= alpha;
            }
            const float msc = st.m[c] == -INFINITY ? 0.0f : st.m[c] * sc;
            if constexpr (T::F32) {
#pragma unroll
                for (int e = 0; e < 8; ++e) pf[c][e] = __builtin_amdgcn_exp2f(fmaf(x[e], sc, -msc));
                st.l[c][0] += ((pf[c][0] + pf[c][1]) + (pf[c][2] + pf[c][3])) + ((pf[c][4] + pf[c][5]) + (pf[c][6] + pf[c][7]));
            } else if constexpr (FP8) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float w = __builtin_amdgcn_exp2f(fmaf(x[e], sc, -msc));
                    st.l[c][0] += w;
                    p[c][e] = static_cast<_Float16>(w * vsc[e >> 2][e & 3]);
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) p[c][e] = static_cast<_Float16>(__builtin_amdgcn_exp2f(fmaf(x[e], sc, -msc)));
                // sums of the rounded weights, on the matrix pipe
                st.l[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, p[c], st.l[c], 0, 0, 0);
            }
        }
        // V^T operand, weight slots (grp, e) = key 4 grp + e, (grp, 4 + e) = key
        // 16 + 4 grp + e.  fp16: within each 16-lane group, lane i receives
        // element i % 4 of the 8-byte chunks addressed by lanes i / 4 + 4 e, so
        // lane (col, grp) addresses key 4 grp + col / 4 (+ 16), dims 16 t + 4
        // (col % 4).  FP8 (tr_read8): the key of slot col / 2, dims 16 t + 8 (col % 2).
        if constexpr (T::F32) {
            // product (hh, e): the k slot of lane (col, grp) is key 16 hh + 4 grp
            // + e, whose weight it holds; dims 4 col + t of that key's row.  Each
            // product's 4 keys a sum of their own, added in pairs.
            float4_t half[CT][2][T::DT];
#pragma unroll
            for (int hh = 0; hh < 2; ++hh) {
                float4_t four[CT][4][T::DT];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float4_t v = __builtin_bit_cast(float4_t, load16(vb + T::off(16 * hh + 4 * grp + e, col)));
#pragma unroll
                    for (int t = 0; t < T::DT; ++t)
#pragma unroll
                        for (int c = 0; c < CT; ++c)
                            four[c][e][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t], pf[c][4 * hh + e],
                                                                                 float4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                }
#pragma unroll
                for (int c = 0; c < CT; ++c)
#pragma unroll
                    for (int t = 0; t < T::DT; ++t)
                        half[c][hh][t] = (four[c][0][t] + four[c][1][t]) + (four[c][2][t] + four[c][3][t]);
            }
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int t = 0; t < T::DT; ++t) st.o[c][t] += half[c][0][t] + half[c][1][t];
            return;
        }
        const int vrow = FP8 ? (col < 8 ? 4 * grp + (col >> 1) : 12 + 4 * grp + (col >> 1)) : 4 * grp + (col >> 2);
#pragma unroll
        for (int t = 0; t < T::DT; ++t) {
            half8_t v;
            if constexpr (FP8) {
                const u32x2 w = tr_read8(vb + T::off(vrow, t) + 8 * (col & 1));
                v = codes8(w[0], w[1]);
            } else {
                const int chunk = 2 * t + ((col & 3) >> 1);
                const u32x2 lo = tr_read(vb + T::off(vrow, chunk) + 8 * (col & 1));
                const u32x2 hi = tr_read(vb + T::off(16 + vrow, chunk) + 8 * (col & 1));
                v = __builtin_bit_cast(half8_t, u32x4{lo[0], lo[1], hi[0], hi[1]});
            }
#pragma unroll
            for (int c = 0; c < CT; ++c) st.o[c][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, p[c], st.o[c][t], 0, 0, 0);
        }
    };

    if constexpr (NST == 1) {
        for (int step = 0; step < steps; ++step) {
            wait_lds();
            issue(step, 0);
            wait_loads<0>();
            compute(step, 0);
        }
    } else {
        static_assert(NST == 2, "one or two stages");
        wait_lds();
        issue(0, 0);
        for (int step = 0; step < steps; ++step) {
            if (step + 1 < steps) {
                wait_lds();  // (the stage's reads, two steps ago in program order, are done)
                issue(step + 1, (step + 1) & 1);
                wait_loads<T::LOADS>();
            } else {
                wait_loads<0>();
            }
            compute(step, step & 1);
        }
    }
    if constexpr (FP8 || T::F32) {
#pragma unroll
        for (int c = 0; c < CT; ++c) st.l[c][0] = xor_add<32>(xor_add<16>(st.l[c][0]));
    }
}

__device__ __forceinline__ int load_block(const DecodeArgs& a, const int32_t* table, const int i) {
    int id = 0;
    if (i < a.max_blocks_per_seq) {
        id = table[i];
        if (a.num_blocks > 0 && unsigned(id) >= unsigned(a.num_blocks)) id = 0;
    }
    return id;
}

// ---------------------------------------------------------------------------
// A workgroup of W waves per (row, kv head): each wave attends a contiguous
// share of the context and the shares are merged in LDS, so the call is one
// launch with no workspace.
template <int D, int CT, int KVT, int W, int NST>
__global__ __launch_bounds__(64 * W) void decode_rows_kernel(const DecodeArgs a) {
    using T = Tile<D, KVT>;
    using IO = typename std::conditional<T::F32, float, _Float16>::type;
    constexpr int kRing = (NST * T::STAGE + 1023) / 1024 * 1024;
    constexpr int kMergeBytes = W * 16 * CT * (D + 2) * 4;
    __shared__ __attribute__((aligned(1024))) char lds[W * kRing > kMergeBytes ? W * kRing : kMergeBytes];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // Rows that are not whole 128-byte lines share lines with the neighbouring
    // heads (four heads are whole lines): four adjacent heads go to one XCD
    // (workgroups are dealt to the 8 XCDs in turn), next to each other there.
    int pair = int(blockIdx.x);
    if (T::ROW % 128 != 0 && pair < int(gridDim.x) / 32 * 32)
        pair = pair / 32 * 32 + (pair % 8) * 4 + pair % 32 / 8;
    const int s = pair / a.num_kv_heads;
    const int kvh = pair - s * a.num_kv_heads;
    const int G = a.num_heads / a.num_kv_heads;
    const int seq = a.row_seq ? a.row_seq[s] : s;
    const int32_t* table = a.bt + int64_t(seq) * a.max_blocks_per_seq;
    if (a.qsl && a.qsl[s + 1] - a.qsl[s] != 1) return;  // (a prefill sequence of a mixed call)
    // requested together with the context length: Q, and the block ids while
    // the table fits one id per lane
    const bool whole = a.max_blocks_per_seq <= kWave;
    int ids = whole ? load_block(a, table, lane) : 0;
    State<D, CT, KVT> st;
    init_state(a, st, s, kvh, G, lane);
    const int ctx = row_context(a, s);
    const int per = ((ctx + W - 1) / W + kStep - 1) / kStep * kStep;
    const int t0 = wave * per;
    const int n = min(ctx - t0, per);
    if (n > 0) {
        int win = 0;
        if (!whole) {
            win = block_div(a, t0);
            ids = load_block(a, table, win + lane);
        }
        stream_tokens<D, CT, KVT, NST>(a, st, lds + wave * kRing, s, table, ctx, kvh, t0, n, win, ids, lane);
    }
    // ---------------- merge
    const float sc = a.scale_log2 < 0.0f ? -a.scale_log2 : a.scale_log2;
    const int col = lane & 15, grp = lane >> 4;
    float* mo = reinterpret_cast<float*>(lds);      // [W][16 CT][D]
    float* mml = mo + W * 16 * CT * D;              // [W][16 CT][2]
    __syncthreads();
    if (n > 0) {
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const int h = 16 * c + col;
            if (h >= G) continue;
            float* row = mo + (wave * 16 * CT + h) * D;
#pragma unroll
            for (int t = 0; t < T::DT; ++t) *reinterpret_cast<float4_t*>(row + st.dim(t, grp)) = st.out4(c, t);
            if (grp == 0) {
                mml[(wave * 16 * CT + h) * 2] = st.m[c] * sc;
                mml[(wave * 16 * CT + h) * 2 + 1] = st.l[c][0];
            }
        }
    } else if (lane < 16 * CT) {
        mml[(wave * 16 * CT + lane) * 2] = -INFINITY;  // (no share: weight 0 below)
        mml[(wave * 16 * CT + lane) * 2 + 1] = 0.0f;
    }
    __syncthreads();
    IO* out = static_cast<IO*>(a.out) + (query_row(a, s) * a.num_heads + kvh * G) * D;
    const int shares = ctx > 0 ? (ctx + per - 1) / per : 0;
    for (int i = threadIdx.x; i < G * (D / 2); i += 64 * W) {
        const int h = i / (D / 2), d = (i - h * (D / 2)) * 2;
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < W; ++w) mx = fmaxf(mx, mml[(w * 16 * CT + h) * 2]);
        float l = 0.0f, x0 = 0.0f, x1 = 0.0f;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            if (w < shares) {
                const float f = __builtin_amdgcn_exp2f(mml[(w * 16 * CT + h) * 2] - mx);
                const float* row = mo + (w * 16 * CT + h) * D + d;
                l = fmaf(f, mml[(w * 16 * CT + h) * 2 + 1], l);
                x0 = fmaf(f, row[0], x0);
                x1 = fmaf(f, row[1], x1);
            }
        }
        float r0 = shares > 0 ? x0 / l : 0.0f, r1 = shares > 0 ? x1 / l : 0.0f;
        IO* o = out + h * D + d;
        if (a.accumulate) {
            r0 += static_cast<float>(o[0]);
            r1 += static_cast<float>(o[1]);
        }
        o[0] = static_cast<IO>(r0);
        o[1] = static_cast<IO>(r1);
    }
    // Fused append: this workgroup alone reads the new token's slot at this kv
    // head, and has.
    if (a.fkey) {
        const int64_t slot = a.fslots[s];
        if (slot >= 0 && slot < a.fnum_slots && threadIdx.x < 2 * T::CH) {
            const bool v = threadIdx.x >= T::CH;
            const int64_t c = int64_t(kvh) * T::ROW + (threadIdx.x - (v ? T::CH : 0)) * 16;
            const char* src = v ? a.fval + s * a.fval_stride + c : a.fkey + s * a.fkey_stride + c;
            char* dst = const_cast<char*>(v ? a.vc : a.kc) + slot * a.num_kv_heads * T::ROW + c;
            store16(dst, load16(src));
        }
    }
}

// ---------------------------------------------------------------------------
// Split-K in equal slices.  The rows' contexts are laid end to end in steps of
// 32 tokens and cut into slices of the same number of steps (a slice may end
// in the middle of a row and begin another), one (slice, kv head) per resident
// wave, kv heads fastest: every wave streams the same amount, whatever the
// context lengths, where partitions of a fixed size leave some waves a second
// one (256 rows of head_dim 64, contexts up to 4 096: 66 to 78 us over sizes
// 128 to 512, 57 at the best of them).  A row's partials are its slices in
// order; row_parts holds the first one and their number for the merge kernel.
// Slices are at least so long that no row has more than max_parts of them, and the
// call no more than max_slices.
constexpr int kMinSliceSteps = 2;
// Building with -DVKV_STREAM_ROWS=1 (2) runs every launch as one workgroup per
// (row, kv head) (in equal slices): an A/B switch.
#ifndef VKV_STREAM_ROWS
#define VKV_STREAM_ROWS 0
#endif

template <int D, int CT, int KVT, int NST>
__global__ __launch_bounds__(256) void decode_stream_kernel(const DecodeArgs a) {
    using T = Tile<D, KVT>;
    constexpr int kRing = NST * T::STAGE;
    __shared__ __attribute__((aligned(1024))) char lds[kWavesPerBlock * kRing];
    __shared__ int wave_total[kWavesPerBlock], wave_longest[kWavesPerBlock];
    extern __shared__ int prefix[];  // [num_rows + 1] exclusive prefix of the rows' steps
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int G = a.num_heads / a.num_kv_heads;
    const int nrows = a.num_rows;
    // Prefix scan: each thread sums a contiguous tile of rows, the tile sums
    // are scanned across the workgroup, then each thread writes its entries.
    auto steps_of = [&](int r) {
        const int ctx = row_context(a, r);
        return ctx > 0 ? (ctx + kStep - 1) / kStep : 0;
    };
    {
        const int per = (nrows + kBlockThreads - 1) / kBlockThreads;
        const int r0 = int(threadIdx.x) * per;
        int local = 0, longest = 0;
        for (int i = 0; i < per; ++i) {
            const int x = r0 + i < nrows ? steps_of(r0 + i) : 0;
            local += x;
            longest = x > longest ? x : longest;
        }
        const int incl = wave_incl_scan(local);
        for (int o = 32; o > 0; o >>= 1) longest = max(longest, __shfl_xor(longest, o, kWave));
        if (lane == kWave - 1) {
            wave_total[wave] = incl;
            wave_longest[wave] = longest;
        }
        __syncthreads();
        int run = incl - local;
        for (int w = 0; w < wave; ++w) run += wave_total[w];
        for (int i = 0; i < per; ++i) {
            if (r0 + i < nrows) {
                prefix[r0 + i] = run;
                run += steps_of(r0 + i);
            }
        }
        if (threadIdx.x == kBlockThreads - 1) prefix[nrows] = run;
        __syncthreads();
    }
    const int total = __builtin_amdgcn_readfirstlane(prefix[nrows]);
    int longest = 0;
    for (int w = 0; w < kWavesPerBlock; ++w) longest = max(longest, wave_longest[w]);
    // Steps per slice: an equal share of every resident wave (a size the
    // caller asked for instead, a.P), within max_parts partials per row and
    // max_slices slices.
    const int waves = int(gridDim.x) * kWavesPerBlock;
    const int share = waves / a.num_kv_heads > 0 ? waves / a.num_kv_heads : 1;
    int R = a.num_cands > 1 ? max((total + share - 1) / share, kMinSliceSteps) : a.P / kStep;
    R = max(R, (longest + a.max_parts - 2) / (a.max_parts - 1));
    R = max(R, (total + a.max_slices - 1) / a.max_slices);
    R = __builtin_amdgcn_readfirstlane(max(R, 1));
    if (blockIdx.x == 0) {
        for (int r = int(threadIdx.x); r < nrows; r += kBlockThreads) {
            const int b = prefix[r], e = prefix[r + 1];
            a.row_parts[r] = int2{b / R + r, e > b ? (e - 1) / R - b / R + 1 : 0};
        }
    }
    const int items = (total + R - 1) / R * a.num_kv_heads;
    const float sc = a.scale_log2 < 0.0f ? -a.scale_log2 : a.scale_log2;
    const int col = lane & 15, grp = lane >> 4;
    for (int it = int(blockIdx.x) * kWavesPerBlock + wave; it < items; it += waves) {
        const int slice = it / a.num_kv_heads;
        const int kvh = it - slice * a.num_kv_heads;
        const int end = min((slice + 1) * R, total);
        int at = slice * R;
        int lo = 0, hi = nrows - 1;  // row = last r with prefix[r] <= at
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (prefix[mid] <= at) lo = mid;
            else hi = mid - 1;
        }
        for (int s = lo; at < end; ++s) {
            const int b = prefix[s], e = min(prefix[s + 1], end);
            if (e <= at) continue;  // (a row without keys)
            const int seq = a.row_seq ? a.row_seq[s] : s;
            const int32_t* table = a.bt + int64_t(seq) * a.max_blocks_per_seq;
            const int ctx = row_context(a, s);
            const int t0 = (at - b) * kStep;
            const int n = min(ctx - t0, (e - at) * kStep);
            const int win = block_div(a, t0);
            const int ids = load_block(a, table, win + lane);
            State<D, CT, KVT> st;
            init_state(a, st, s, kvh, G, lane);
            stream_tokens<D, CT, KVT, NST>(a, st, lds + wave * kRing, s, table, ctx, kvh, t0, n, win, ids, lane);
            const int64_t slot = int64_t(kvh) * a.part_slots + slice + s;
#pragma unroll
            for (int c = 0; c < CT; ++c) {
                const int h = 16 * c + col;
                if (h >= G) continue;
                float* row = a.part_o + (slot * G + h) * D;
#pragma unroll
                for (int t = 0; t < T::DT; ++t) *reinterpret_cast<float4_t*>(row + st.dim(t, grp)) = st.out4(c, t);
                if (grp == 0) {
                    a.part_ml[(slot * G + h) * 2] = st.m[c] * sc;
                    a.part_ml[(slot * G + h) * 2 + 1] = st.l[c][0];
                }
            }
            at = e;
        }
    }
}

// Split-K in partitions of a fixed size (decode.hip's items and size choice).
template <int D, int CT, int KVT, int NST>
__global__ __launch_bounds__(256) void decode_parts_kernel(const DecodeArgs a) {
    using T = Tile<D, KVT>;
    constexpr int kRing = (NST * T::STAGE + 1023) / 1024 * 1024;
    __shared__ __attribute__((aligned(1024))) char lds[kWavesPerBlock * kRing];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int G = a.num_heads / a.num_kv_heads;
    run_partitions<false, true>(a, a.num_kv_heads, [&](const int P, const int s, const int part, const int kvh)
                                                __attribute__((always_inline)) {
        const int seq = a.row_seq ? a.row_seq[s] : s;
        const int32_t* table = a.bt + int64_t(seq) * a.max_blocks_per_seq;
        const int ctx = row_context(a, s);
        const int t0 = part * P;
        if (t0 >= ctx) return;
        const int n = min(ctx - t0, P);
        const int win = block_div(a, t0);
        const int ids = load_block(a, table, win + lane);
        State<D, CT, KVT> st;
        init_state(a, st, s, kvh, G, lane);
        stream_tokens<D, CT, KVT, NST>(a, st, lds + wave * kRing, s, table, ctx, kvh, t0, n, win, ids, lane);
        const float sc = a.scale_log2 < 0.0f ? -a.scale_log2 : a.scale_log2;
        const int col = lane & 15, grp = lane >> 4;
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const int h = 16 * c + col;
            if (h >= G) continue;
            const int64_t item = ((int64_t(s) * a.num_kv_heads + kvh) * a.max_parts + part) * G + h;
            float* row = a.part_o + item * D;
#pragma unroll
            for (int t = 0; t < T::DT; ++t) *reinterpret_cast<float4_t*>(row + st.dim(t, grp)) = st.out4(c, t);
            if (grp == 0) {
                a.part_ml[item * 2] = st.m[c] * sc;
                a.part_ml[item * 2 + 1] = st.l[c][0];
            }
        }
    });
}

// One workgroup per resident slot (occupancy queried once per variant).
template <int D, int CT, int KVT, int NST>
void launch_split(DecodeArgs& a, size_t lds, hipStream_t st) {
    static std::atomic<int> cached{0};
    auto kernel = decode_stream_kernel<D, CT, KVT, NST>;
    int per_cu = cached.load(std::memory_order_relaxed);
    if (per_cu <= 0) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kBlockThreads, 0) != hipSuccess || per_cu <= 0) per_cu = 1;
        cached.store(per_cu, std::memory_order_relaxed);
    }
    const int by_lds = kLdsPerCu / int(lds + 1024 + kWavesPerBlock * NST * Tile<D, KVT>::STAGE);
    if (by_lds < per_cu) per_cu = by_lds > 0 ? by_lds : 1;
    hipLaunchKernelGGL(kernel, dim3(device_cu_count() * per_cu), dim3(kBlockThreads), lds, st, a);
}

// Eight waves per row while every (row, kv head) has a CU, else four, so that
// two workgroups share a CU; two stages per wave where a stage is 8 KiB.  Many
// pairs of short tables: two waves or one, of one stage.  LDS bounds what a CU
// holds, and a wave of a row that has no step for it (contexts shorter than 32
// tokens a wave) holds its ring for nothing; with four pairs to a CU the others
// cover a wave's loads.  Measured over contexts U[1, max] (us per appending step,
// FP8 per decode; four waves / two / one):
//   head_dim 64,   512 pairs: max 64: 8.4 / 7.4 / 7.3   128: 7.5 / 7.9 / 9.7    256: 10.1 / 10.6 / 14.7
//                 1280 pairs:     64: 13.7 / 8.0 / 7.9  128: 15.2 / 9.5 / 10.8  384: 21.0 / 18.0 / 21.3
//                 8192 pairs:     64: 66.6 / 24.2 / 21.0  128: 73.7 / 32.7 / 30.5  512: 121 / 102 / 107
//   head_dim 112, 2048 pairs:     64: 20.7 / 14.1 / 10.3  128: 25.0 / 18.4 / 16.2  256: 32.0 / 25.8 / 28.4
//   head_dim 128, 1280 pairs:     64: 17.5 / 13.6 / 11.2  256: 26.2 / 24.1 / 25.1  512: 40.4 / 42.1 / 43.4
//                 8192 pairs:     64: 83.8 / 54.3 / 41.5  128: 96.4 / 73.3 / 63.8  512: 221 / 201 / 206
//   FP8,          1280 pairs:     64: 14.6 / 8.8 / 9.5  256: 20.2 / 16.4 / 20.7  1 024: 44.5 / 51.3 / 61.7
//                 8192 pairs:     64: 69.5 / 33.7 / 27.1  128: 77.0 / 44.7 / 39.5  512: 143 / 127 / 130
//     (every row of 512 tokens, 2048 pairs: 61.5 / 65.3; head_dim 128: 95.1 / 100.7)
//   fp32, group 7, 2048 pairs:    64: 33.6 / 23.1 / 18.3  128: 35.8 / 32.2 / 28.7  256: 52.1 / 50.8 / 49.7
template <int D, int CT, int KVT>
void launch_row_groups(DecodeArgs& a, hipStream_t st) {
    constexpr int NST = Tile<D, KVT>::STAGE <= 8192 + 256 ? 2 : 1;
    const int64_t pairs = int64_t(a.num_rows) * a.num_kv_heads, cus = device_cu_count();
    const dim3 grid{unsigned(pairs)};
    if constexpr (CT == 1) {
        if (pairs >= 4 * cus && a.max_ctx <= (pairs >= 8 * cus ? 132 : 66)) {
            hipLaunchKernelGGL((decode_rows_kernel<D, CT, KVT, 1, 1>), grid, dim3(64), 0, st, a);
            return;
        }
        if (pairs >= 4 * cus && a.max_ctx <= (pairs >= 16 * cus ? 528 : 396)) {
            hipLaunchKernelGGL((decode_rows_kernel<D, CT, KVT, 2, 1>), grid, dim3(128), 0, st, a);
            return;
        }
    }
    if (pairs <= cus)
        hipLaunchKernelGGL((decode_rows_kernel<D, CT, KVT, 8, NST == 2 && KVT == kFp8 ? 1 : NST>), grid, dim3(512), 0, st, a);
    else
        hipLaunchKernelGGL((decode_rows_kernel<D, CT, KVT, 4, NST>), grid, dim3(256), 0, st, a);
}

template <int D, int CT, int KVT>
void launch_shape(DecodeArgs& a, bool rows, size_t lds, hipStream_t st) {
    if (rows) {
        launch_row_groups<D, CT, KVT>(a, st);
        return;
    }
    // (calls over thousands of rows leave LDS for one stage only)
    if constexpr (D > 80) {
        if (lds <= (16 << 10)) {
            launch_split<D, CT, KVT, 2>(a, lds, st);
            return;
        }
    }
    launch_split<D, CT, KVT, D == 64 && KVT == kF16 ? 2 : 1>(a, lds, st);
}

template <int D, int KVT = kF16>
void launch_dim(DecodeArgs& a, int G, bool rows, size_t lds, hipStream_t st) {
    if (G <= 16) launch_shape<D, 1, KVT>(a, rows, lds, st);
    else launch_shape<D, 2, KVT>(a, rows, lds, st);
}

}  // namespace

// One workgroup per (row, kv head) saves the merge launch and the scan of the
// rows, but the longest row's workgroup streams alone at the end, at about 54
// bytes per ns.  Measured both ways over contexts U[1, max_ctx] (us per
// appending step, FP8 per decode; workgroup per row, of four waves beyond 256 pairs,
// against equal slices):
//   head_dim 64,   64 pairs: max 1 024: 9.3 / 13.4   2 048: 14.4 / 14.3   4 096: 26.5 / 20.9
//                 512 pairs:     1 024: 17.8 / 24.7   2 048: 32.3 / 34.7   4 096: 62.5 / 55.4
//                2048 pairs:     1 024: 52.9 / 65.3   2 048: 95 / 108      4 096: 185 / 191
//   head_dim 128,  64 pairs:       512: 11.3 / 14.7   1 024: 16.2 / 15.9   2 048: 28.9 / 20.2
//     (group 16)  256 pairs:     1 024: 19.1 / 27.1   2 048: 35.3 / 38.9   4 096: 63.9 / 60.4
//                1024 pairs:     1 024: 58.5 / 68.8   2 048: 109 / 115     4 096: 207 / 207
//   head_dim 80,   64 pairs:       512: 7.1 / 10.7    1 024: 9.4 / 11.3    2 048: 19.1 / 16.5
//                1024 pairs:       512: 19.4 / 23.2   1 024: 32.8 / 33.2   2 048: 73.6 / 63.6
//                2048 pairs:       256: 21.7 / 25.8     512: 34.7 / 37.4   1 024: 85.1 / 75.6
//   fp32, group 7, 64 pairs:       512: 13.4 / 18.6   1 024: 22.5 / 19.1   2 048: 40.3 / 20.6
//     head_dim 64 512 pairs:       512: 26.7 / 31.1   1 024: 47.8 / 41.5   2 048: 86.5 / 63.1
// Against partitions (matrix_split; head_dim 128, group 4): 32 pairs, 1 024: 14.4 /
// 14.3; 256 pairs, 1 024: 17.9 / 22.7; 2 048: 32.8 / 34.4; 1 024 pairs, 1 024: 54.0 /
// 79.9; 2 048: 114 / 109.  FP8: 32 pairs, 1 024: 11.3 / 13.1; 2 048: 19.4 / 16.5; 256
// pairs, 2 048: 24.1 / 28.0; 1 024 pairs, 1 024: 37.7 / 63.7; 2 048: 77.3 / 67.2.
bool stream_decode_rows(int num_rows, int num_kv_heads, int half_dims, int max_ctx, bool matrix_split, int f32_group) {
#if VKV_STREAM_ROWS
    return VKV_STREAM_ROWS == 1;
#endif
    const int64_t pairs = int64_t(num_rows) * num_kv_heads, cus = device_cu_count();
    if (f32_group > 16) return max_ctx <= 264;
    if (f32_group > 0) return max_ctx <= (pairs < cus ? 528 : pairs < 4 * cus ? 1056 : 264);
    if (matrix_split && half_dims == 64) return max_ctx <= (2 * pairs >= cus && pairs <= cus ? 2112 : 1056);
    if (half_dims % 64 != 0) return max_ctx <= (pairs < 2 * cus ? 1056 : pairs < 8 * cus ? 528 : 264);
    const int64_t row_bytes = int64_t(max_ctx) * half_dims * 4;
    return max_ctx <= 2112 && (row_bytes <= 528 << 10 || (pairs >= cus && !matrix_split));
}

int stream_split_waves(int head_dim, bool f32) {
    // (256 CUs: asking for the device takes 0.1 us of a small call's 6.  Stages as
    // launch_shape takes them; two stages at the wider heads: fewer)
    const int stage = 2 * kStep * head_dim * (f32 ? 4 : 2) * (head_dim == 64 && !f32 ? 2 : 1);
    return 256 * (kLdsPerCu / (1024 + kWavesPerBlock * stage)) * kWavesPerBlock;
}

// Contexts U[1, max_ctx], us per appending step (VALU kernel / workgroup per row, of
// four waves beyond 256 pairs / equal slices):
//   group 1,   64 pairs: 256 tokens: 10 / 11 / 18     1 024: 13 / 22 / 20   4 096: 23 / 73 / 33
//            1 024 pairs: 64: 15 / 18 / 19    512: 44 / 45 / 40   1 024: 75 / 77 / 61   4 096: 190 / 296 / 206
//   group 4,  256 pairs:  512: 20 / 16 / 23   1 024: 27 / 25 / 29   2 048: 48 / 44 / 42   4 096: 73 / 80 / 65
//   group 5,   64 pairs:  512: 16 / 14 / 19   1 024: 18 / 23 / 20   2 048: 26 / 41 / 22   4 096: 38 / 74 / 33
// (Blocks of no power of two alike: 8/8 heads, 24-token blocks, 256 rows of 1 to 64
// tokens: 18.8 us on the generic kernel, 32.1 streamed by four waves.)
bool stream_f32_pays(int num_rows, int num_kv_heads, int group, int max_ctx) {
    if (group > 4) return true;
    const int64_t pairs = int64_t(num_rows) * num_kv_heads, cus = device_cu_count();
    if (pairs < cus) return max_ctx <= (group > 2 ? 264 : 132);
    if (pairs < 4 * cus) return max_ctx <= (group > 2 ? 528 : 264) || (group == 4 && pairs < 2 * cus && max_ctx > 1056);
    return max_ctx > 264 && max_ctx <= (group > 1 ? 2112 : pairs < 8 * cus ? 1056 : 0);
}

template <int KVT, int NST>
static void launch_parts(DecodeArgs& a, int64_t max_items, size_t lds, hipStream_t st) {
    static std::atomic<int> cached{0};
    auto kernel = decode_parts_kernel<128, 1, KVT, NST>;
    const int cus = device_cu_count();
    int per_cu = cached.load(std::memory_order_relaxed);
    if (per_cu <= 0) {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kBlockThreads, 0) != hipSuccess || per_cu <= 0) per_cu = 1;
        cached.store(per_cu, std::memory_order_relaxed);
    }
    const int by_lds = kLdsPerCu / int(lds + 2048 + kWavesPerBlock * ((NST * Tile<128, KVT>::STAGE + 1023) / 1024 * 1024));
    if (by_lds < per_cu) per_cu = by_lds > 0 ? by_lds : 1;
    const int64_t groups = (max_items + kWavesPerBlock - 1) / kWavesPerBlock, wgs = int64_t(cus) * per_cu;
    const int gx = int(groups < wgs ? (groups > 0 ? groups : 1) : wgs);
    a.static_parts = 0;
    a.wave_slots = gx * kWavesPerBlock;
    a.level_waves = (gx < cus ? gx : cus) * kWavesPerBlock;
    // (beyond two rounds of full-size partitions the default stands: 256 long-tailed
    // rows, FP8: 311 us at 768 tokens, 335 at the least cost)
    if (a.P >= 768) a.keep_above = 2 * a.wave_slots;
    hipLaunchKernelGGL(kernel, dim3(gx), dim3(kBlockThreads), lds, st, a);
}

// Rows of FP8 caches are half the bytes, as head_dim 64 in fp16.  One stage per
// wave leaves room for two workgroups per CU in fp16 (two stages: one) and is
// the faster for small FP8 groups; larger ones compute longer per step and keep
// a second one in flight (us, one stage / two: 64 sequences of C2's lengths,
// group 4, fp16 105.4 / 110.8; 256 long-tailed ones, group 4, FP8 312.4 / 317.0;
// 120 of 1 024 to 8 192, group 7, FP8 132.2 / 125.3).
bool launch_decode_matrix(DecodeArgs& a, bool fp8, int64_t max_items, size_t lds, hipStream_t st) {
    if (fp8 && stream_decode_rows(a.num_rows, a.num_kv_heads, 64, a.max_ctx, true, 0)) {
        launch_row_groups<128, 1, kFp8>(a, st);
        return true;
    }
    if (!fp8) launch_parts<kF16, 1>(a, max_items, lds, st);
    else if (a.num_heads / a.num_kv_heads <= 4) launch_parts<kFp8, 1>(a, max_items, lds, st);
    else launch_parts<kFp8, 2>(a, max_items, lds, st);
    return false;
}

int launch_decode_stream(DecodeArgs& a, bool f32, bool rows, size_t lds, hipStream_t st) {
    const int G = a.num_heads / a.num_kv_heads;
    if (f32) {
        if (a.head_dim != 64) return VKV_ERR_UNSUPPORTED;
        launch_dim<64, kF32>(a, G, rows, lds, st);
        return 0;
    }
    switch (a.head_dim) {
        case 64: launch_dim<64>(a, G, rows, lds, st); return 0;
        case 80: launch_dim<80>(a, G, rows, lds, st); return 0;
        case 96: launch_dim<96>(a, G, rows, lds, st); return 0;
        case 112: launch_dim<112>(a, G, rows, lds, st); return 0;
        case 128: launch_dim<128>(a, G, rows, lds, st); return 0;
        default: return VKV_ERR_UNSUPPORTED;
    }
}

}  // namespace dec
}  // namespace vkv
