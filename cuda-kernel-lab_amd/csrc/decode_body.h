// decode_body.h -- paged decode attention on CDNA4 fp16 MFMA: the segment runner shared by the
// decode kernels (decode.hip: plan/run, uniform split, device ranges, the fused cascade step).
//
// A wave handles one kv head and all G query heads that share it, 32 keys (two pages) at a time:
//
//   S^T = K Q^T      v_mfma_f32_16x16x32_f16, A = 16 keys x 32 dims, B = 32 dims x 16 columns
//   O^T += V^T P^T   A = 16 dims x 32 keys, B = 32 keys x 16 columns
//
// A decode batch has only G <= 8 rows per kv head, so half of the 16 columns would idle. They hold
// the weights' low halves instead: columns 0-7 are the heads with p rounded to fp16, columns 8-15
// the same heads with (p - fp16(p)) * 2^11 rounded to fp16, and the output is the first plus 2^-11
// times the second. The PV product then sees every weight to 22 bits (an error of 2^-23 of the
// weight on average, fp32's own rounding is 2^-25), at no extra MFMA; scores and sums are fp32.
//
// Staging: a wave moves its own pages with 16-byte direct global->LDS loads into its own 16 KB slots
// (K and V of two pages), so the loop has no workgroup barrier. Per block the wave waits for its
// slot, reads all operands of the block into registers (K rows with ds_read_b128, V with the
// transposing ds_read_b64_tr_b16), issues the next loads into the slot, and computes. One slot keeps
// 16 KB per wave, 64 KB per CU, in flight, which covers the loaded latency of long streams; two slots
// (G <= 4) start short sequences sooner: one sequence of 4096 tokens 9.43 -> 8.93 us, 128 of 16-512
// at G = 1 96.2 -> 94.6 us, 32768 tokens 27.6 -> 26.8 us; 64 x 1024 41.9 -> 42.1 us.
//
// Bound: HBM (64 ragged sequences of 256-4096 tokens, 548 MB: 85 us at G = 4 and 87 us at G = 8 for
// the decode launch, where one contiguous read of as many bytes takes 82 us). The vector-unit body
// before it took 768 instructions per 32 keys at G = 4 and about twice that at G = 8, where the
// arithmetic and not the memory set the pace: 95 and 151 us.
#pragma once

#include "prefix_body.h"

namespace pdattn {
namespace {

// HP kv heads per 4-wave workgroup, WPH waves each (HP > 1: page-range plans, whose HP
// neighbouring workgroups read the same pages for neighbouring heads).
template <int G_, int HP_>
struct DecCfg {
    static constexpr int G = G_;              // query heads per kv head
    static constexpr int HP = HP_;
    static constexpr int NW = 4;
    static constexpr int NT = NW * 64;
    static constexpr int WPH = NW / HP_;
};

constexpr int kDecPageBytes = kPage * kHeadDim * 2;      // one page of one head, K or V
constexpr int kDecSlotBytes = 4 * kDecPageBytes;         // K of two pages, then V of two pages
constexpr int kDecQBytes = 4 * kHeadDim * 2;             // q rows of up to 4 heads
constexpr float kLoScale = 2048.f;                       // scale of the weights' low halves
constexpr float kDecLn2 = 0.69314718055994531f;

// LDS layouts: kLayWide holds two blocks per wave (one at G = 8); kLayOne one block and leaves room for
// the device-range kernel's own arrays; kLayStep (the fused cascade step, so that a CU holds the
// workgroup beside a prefix workgroup, 80 KB each) one block, a shorter page list, one flush buffer,
// and at G = 8 the flush in two passes.
enum { kLayWide, kLayOne, kLayStep };
template <class C, int LAY>
struct DecShared {
    static constexpr int PGMAX = LAY == kLayStep ? kStepRangeMax : kRangeMax;
    static constexpr int HG = LAY == kLayStep && C::G > 4 ? 4 : C::G;   // heads per flush pass
    // 32-key blocks in LDS per wave. Two: the slots also carry the block's q rows (see run_segments).
    static constexpr int NS = LAY == kLayWide && C::G <= 4 ? 2 : 1;
    static constexpr int NB = LAY == kLayStep || NS > 1 ? 1 : 2;         // flush buffers
    static constexpr int SLOT = kDecSlotBytes + (NS > 1 ? kDecQBytes : 0);
    alignas(256) uint8_t slot[C::NW][NS][SLOT];
    alignas(16) float o[NB][C::NW][HG][kHeadDim + 4];
    float m[NB][C::NW][C::G];
    float l[NB][C::NW][C::G];
    int pg[PGMAX];                       // the workgroup's page ids
    int sd[C::HP][kBalDescInts];         // descriptor block(s): header, then segments
};

// x / d for x < 2^32 without a division, m = floor((2^32 - 1) / d): the high product is the quotient or
// one less.
__device__ __forceinline__ uint32_t dec_div(uint32_t x, uint32_t d, uint32_t m) {
    const uint32_t t = (uint32_t)(((uint64_t)x * m) >> 32);
    return t + ((t + 1) * (uint64_t)d <= x ? 1u : 0u);
}
// nnz g / ngroups (g <= ngroups) of a page-range plan
__device__ __forceinline__ uint32_t dec_range(const BalArgs& a, uint32_t g) {
    if (a.ngroups < 65536) return a.range_q * g + dec_div(a.range_r * g, (uint32_t)a.ngroups, a.range_m);
    return (uint32_t)((uint64_t)a.nnz * g / (uint32_t)a.ngroups);
}

// The segment fields of a descriptor block (8 ints each) through a window of 8 segments in one
// register: field f of segment si is a lane read, and LDS is read once per 8 segments.
struct SegWin {
    const int* seg;
    int v, base;
    __device__ __forceinline__ void init(const int* s) {
        seg = s;
        base = 0;
        v = s[threadIdx.x & 63];
    }
    __device__ __forceinline__ int get(int si, int f) {
        if ((si >> 3) != base) {
            base = si >> 3;
            v = seg[64 * base + (threadIdx.x & 63)];
        }
        return __builtin_amdgcn_readlane(v, 8 * (si & 7) + f);
    }
};
static_assert(kSegInts == 8 && kBalDescInts == 8 + 3 * 64, "three windows of 8 segments");

// One wave's running state: column c of the accumulators is head c % 8 (its fp16 weights for
// c < 8, their low halves for c >= 8). m is the same in the four lanes of a column; l is the sum
// over the lane's own keys.
struct DecState {
    float m, l;
    pf32x4 acc[8];
};
__device__ __forceinline__ void dec_reset(DecState& st) {
    st.m = -INFINITY;
    st.l = 0.f;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) st.acc[dt] = pf32x4{0.f, 0.f, 0.f, 0.f};
}

// The operands of one 32-key block: K rows of page t, 8 dims per lane and k-step, and V^T (16 dims
// x 32 keys) per dim tile, element e < 4 of lane (lg, l16) being key 4 lg + e of the first page,
// e >= 4 key 4 lg + e - 4 of the second.
struct DecBlock {
    pf16x8 k[2][4];
    pf16x8 v[8];
};

// 16 bytes per lane from a wave-uniform base plus a 32-bit lane offset into LDS: lane i's bytes land
// at lds + 16 i (M0 holds the LDS address; one wait state between the M0 write and the load).
// Non-temporal: K and V bytes are read once. The compiler does not count these loads; the waits
// are explicit.
__device__ __forceinline__ void dec_dma(const uint8_t* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt"
                 :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
// the same with the default cache policy (q rows, read by every block of a sequence)
__device__ __forceinline__ void dec_dma_q(const _Float16* base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}
// All of this wave's loads but the newest n (0, 9 or 17) are done.
__device__ __forceinline__ void dec_wait_loads(int n) {
    __builtin_amdgcn_sched_barrier(0);
    if (n >= 17)
        asm volatile("s_waitcnt vmcnt(17)" ::: "memory");
    else if (n >= 9)
        asm volatile("s_waitcnt vmcnt(9)" ::: "memory");
    else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// All of this wave's loads are done. (The builtin, not inline asm: the compiler then knows that the q
// rows it loaded are there, and puts no wait for them between the next block's loads and the MFMAs,
// which would wait for those loads.)
__device__ __forceinline__ void dec_wait_loads() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void dec_wait_lds() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// LDS writes done, then the workgroup barrier; page loads stay in flight across it (a
// __syncthreads() fence would wait for them).
__device__ __forceinline__ void dec_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// lane l ^ 8 within each 16-lane row (row_ror:8)
__device__ __forceinline__ float dec_ror8(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xF, 0xF, true));
}

// Reads a block from the wave's slot (LDS byte address). K: row l16 of page t, chunk (4 ks + lg) at
// position (4 ks + lg) ^ l16. V: transposing reads as in prefix_chunk: lane reads 4 dims of key
// 4 lg + l16 / 4 of page h, chunk 2 dt + ((l16 & 3) >> 1) at position chunk ^ ((key & 7) << 1), and
// receives dim 16 dt + l16 of keys 4 lg .. + 3.
__device__ __forceinline__ void dec_read_block(DecBlock& b, uint8_t* slot, int l16, int lg) {
    typedef __attribute__((address_space(3))) uint8_t lds_u8;
    lds_u8* const s = (lds_u8*)slot;
    const uint32_t kl = (uint32_t)(l16 * 256 + ((((l16 >> 2) << 2) | (lg ^ (l16 & 3))) << 4));
    const int key = 4 * lg + (l16 >> 2);
    const uint32_t vl = (uint32_t)(2 * kDecPageBytes + key * 256 + ((((key & 7) << 1) | ((l16 & 3) >> 1)) << 4) +
                                   8 * (l16 & 1));
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
            b.k[t][ks] = __builtin_bit_cast(pf16x8, *(const __attribute__((address_space(3))) pu32x4*)(
                                                        s + ((kl ^ (uint32_t)(ks << 6)) + kDecPageBytes * t)));
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
        pf16x4 half[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
            half[h] = __builtin_bit_cast(pf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4f16(
                (__attribute__((address_space(3))) lds_f16x4*)(s + ((vl ^ (uint32_t)(dt << 5)) + kDecPageBytes * h))));
        b.v[dt] = pf16x8{half[0][0], half[0][1], half[0][2], half[0][3],
                         half[1][0], half[1][1], half[1][2], half[1][3]};
    }
}

// The q rows of a slot as B operands: head r = (l16 & 7) % G, chunk 4 ks + lg at position chunk ^ 4 r of
// its row (the rows then lie in different LDS banks).
template <int G>
__device__ __forceinline__ void dec_read_q(pf16x8 (&q)[4], uint8_t* qs, int l16, int lg) {
    typedef __attribute__((address_space(3))) uint8_t lds_u8;
    const int r = (l16 & 7) % G;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
        q[ks] = __builtin_bit_cast(pf16x8, *(const __attribute__((address_space(3))) pu32x4*)(
                                               (lds_u8*)qs + r * 256 + ((((ks ^ r) << 2) | lg) << 4)));
}

// One 32-key block: scores, online softmax (base 2, on scores scaled by scale2), PV product. tok0 /
// tok1: (wave-uniform) token index of the two pages' first slots; keys outside [tb, te) are masked
// (a padding page: tok1 >= te). A masked key weighs 0 and, since 0 * NaN is not 0, its V elements
// are zeroed as well: slots the cache never filled may hold any bits. Its K row only feeds its own
// score, which is replaced.
// lo_a, lo_b: (1, 0) in columns 0-7, (2^11, -2^11) in columns 8-15: fma(fp16(p), lo_b, p lo_a) is p
// or its scaled rounding error, both exact.
__device__ __forceinline__ void dec_block(DecState& st, DecBlock& b, const pf16x8 (&q)[4], int tok0, int tok1,
                                          int tb, int te, float scale2, float lo_a, float lo_b, int lg) {
    float x[8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        // (two chains of two: fewer roundings in a row than one of four, and half its latency)
        pf32x4 c[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
            c[i] = mfma16x16x32(b.k[t][2 * i + 1], q[2 * i + 1],
                                mfma16x16x32(b.k[t][2 * i], q[2 * i], pf32x4{0.f, 0.f, 0.f, 0.f}));
#pragma unroll
        for (int j = 0; j < 4; ++j) x[4 * t + j] = (c[0][j] + c[1][j]) * scale2;
    }
    if (tok0 < tb || tok0 + kPage > te || tok1 + kPage > te) {   // wave-uniform: an edge block
        uint32_t keep[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int tok = (e < 4 ? tok0 : tok1) + 4 * lg + (e & 3);
            if (tok >= tb && tok < te) keep[e / 2] |= e & 1 ? 0xFFFF0000u : 0x0000FFFFu;
            else x[e] = -INFINITY;
        }
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) {
            pu32x4 w = __builtin_bit_cast(pu32x4, b.v[dt]);
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] &= keep[i];
            b.v[dt] = __builtin_bit_cast(pf16x8, w);
        }
    }
    float mx = x[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) mx = fmaxf(mx, x[e]);
    const float mn = fmaxf(st.m, col4_reduce<true>(mx));
    if (__builtin_amdgcn_ballot_w64(mn > st.m)) {
        const float al = mn > st.m ? __builtin_amdgcn_exp2f(st.m - mn) : 1.f;
        st.l *= al;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) st.acc[dt] *= al;
        st.m = mn;
    }
    const float ms = st.m == -INFINITY ? 0.f : st.m;
    pf16x8 pb;
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float p = __builtin_amdgcn_exp2f(x[e] - ms);
        sum += p;
        const _Float16 hi = (_Float16)p;
        pb[e] = (_Float16)fmaf((float)hi, lo_b, p * lo_a);
    }
    st.l += sum;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) st.acc[dt] = mfma16x16x32(b.v[dt], pb, st.acc[dt]);
}

// End of a segment: the waves of a kv head hand their states (maximum, sum, output) to LDS, and
// each thread forms four outputs of one query head as a weighted sum over those waves, in wave
// order. Writes the G rows as the final fp16 out / lse (slot < 0) or as partial slot `slot`
// (normalized o, lse). Every thread of the workgroup calls it. With two flush buffers the one
// barrier suffices: a buffer is written again two flushes later, after the barrier of the next.
template <class C, int LAY, class ArgP>
__device__ __forceinline__ void dec_flush(DecShared<C, LAY>& S, DecState& st, int par, ArgP a,
                                          size_t row0, int slot) {
    typedef DecShared<C, LAY> Sh;
    constexpr int G = C::G, HG = Sh::HG, WPH = C::WPH;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int l16 = lane & 15, lg = lane >> 4, w0 = wave / WPH * WPH;
    const int ltid = tid - w0 * 64;
    const float L = col4_reduce<false>(st.l);
    // High plus scaled low halves (in columns 0-7).
    float o[8][4], top = 0.f, ks = 1.f / kLoScale;
    asm("" : "+v"(ks));   // (in a register: the exchange then folds into the multiply-add)
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float hi = st.acc[dt][j];
            o[dt][j] = fmaf(dec_ror8(hi), ks, hi);
            top = fmaxf(top, fabsf(hi));
        }
    // An infinite V makes the high half infinite and the low half NaN (0 * inf, inf - inf): the high
    // half is then the answer.
    if (__builtin_amdgcn_ballot_w64(top == INFINITY)) {
#pragma unroll
        for (int dt = 0; dt < 8; ++dt)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (fabsf(st.acc[dt][j]) == INFINITY) o[dt][j] = st.acc[dt][j];
    }
    const int bf = Sh::NB == 2 ? par : 0;
    if (lg == 0 && l16 < G) {
        S.m[bf][wave][l16] = st.m;
        S.l[bf][wave][l16] = L;
    }
#pragma unroll
    for (int hp = 0; hp < G / HG; ++hp) {
        if (l16 >= hp * HG && l16 < (hp + 1) * HG) {
#pragma unroll
            for (int dt = 0; dt < 8; ++dt)
                *reinterpret_cast<float4*>(&S.o[bf][wave][l16 - hp * HG][16 * dt + 4 * lg]) =
                    make_float4(o[dt][0], o[dt][1], o[dt][2], o[dt][3]);
        }
        dec_barrier();
#pragma unroll
        for (int idx = ltid; idx < HG * 32; idx += WPH * 64) {
            const int hh = idx / 32, h = hp * HG + hh, d0 = 4 * (idx % 32);
            float mw[WPH], M = -INFINITY;
#pragma unroll
            for (int w = 0; w < WPH; ++w) {
                mw[w] = S.m[bf][w0 + w][h];
                M = fmaxf(M, mw[w]);
            }
            float Ls = 0.f;
            float4 O = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int w = 0; w < WPH; ++w) {
                const float al = mw[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mw[w] - M);
                const float4 ov = *reinterpret_cast<const float4*>(&S.o[bf][w0 + w][hh][d0]);
                Ls = fmaf(al, S.l[bf][w0 + w][h], Ls);
                O.x = fmaf(al, ov.x, O.x);
                O.y = fmaf(al, ov.y, O.y);
                O.z = fmaf(al, ov.z, O.z);
                O.w = fmaf(al, ov.w, O.w);
            }
            const float ri = Ls > 0.f ? 1.f / Ls : 0.f;
            const float lse = Ls > 0.f ? (M + __builtin_amdgcn_logf(Ls)) * kDecLn2 : -INFINITY;
            O.x *= ri;
            O.y *= ri;
            O.z *= ri;
            O.w *= ri;
            if (slot < 0) {
                const pf16x4 hv = {(_Float16)O.x, (_Float16)O.y, (_Float16)O.z, (_Float16)O.w};
                *reinterpret_cast<pf16x4*>(a->out + (row0 + h) * kHeadDim + d0) = hv;
                if (d0 == 0) a->lse[row0 + h] = lse;
            } else {
                const int ps = a->part_stride;
                const size_t e = ps > 0 ? (row0 + h) * (size_t)ps + slot : (size_t)slot * G + h;
                *reinterpret_cast<float4*>(a->part_o + e * kHeadDim + d0) = O;
                if (d0 == 0) a->part_lse[e] = lse;
            }
        }
        if (Sh::NB == 1 || hp + 1 < G / HG) dec_barrier();
    }
}

}  // namespace
}  // namespace pdattn
