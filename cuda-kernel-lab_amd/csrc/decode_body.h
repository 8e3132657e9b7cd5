// decode_body.h -- paged decode attention on CDNA4 fp16 MFMA: the segment runner shared by the
// decode kernels (decode.hip: plan/run, uniform split, device ranges, the fused cascade step).
//
// A wave handles one kv head and all G query heads that share it, 32 keys (two pages) at a time:
//
//   S^T = K Q^T      v_mfma_f32_16x16x32_f16, A = 16 keys x 32 dims, B = 32 dims x 16 columns
//   O^T += V^T P^T   A = 16 dims x 32 keys, B = 32 keys x 16 columns
//
// The weights p (fp32, at most 1) enter the PV product whole, as three fp16 parts of p * 2^15:
//   hi = fp16(p 2^15),  mid = fp16((p 2^15 - hi) 2^11),  lo = fp16((p 2^15 - hi) 2^11 - mid)
// and the output is (hi V + 2^-11 (mid V + lo V)) 2^-15. A decode batch has only G <= 8 rows per kv head,
// so half of the 16 columns would idle: columns 0-7 (head c % 8 % G) hold hi and columns 8-15 mid; lo
// goes through a second MFMA into the latter. hi and mid take 11 bits each and lo the rest: the sum is p
// exactly, all 24 bits, for p >= 2^-27 of the running maximum's weight 1; below that it is within 2^-51
// (fp16's smallest value, 2^-24, at lo's scale), which no fp16 output can show. Scores, sums and
// accumulators are fp32. Error of the fp32 partials against 64 bits with fp32 weights on the vector unit
// / with hi and mid alone, rounded scaled scores / this: 4096 keys 3.4e-7 / 2.7e-7 / 2.6e-7, q eight
// times larger 6.1e-7 / 5.8e-7 / 5.2e-7, 8192 keys at G = 8 4.5e-7 / 3.4e-7 / 3.4e-7, q eight times larger
// 6.5e-7 / 6.7e-7 / 5.9e-7.
//
// Staging: a wave moves its own pages with 16-byte direct global->LDS loads into its own 16 KB slots
// (K and V of two pages), so the loop has no workgroup barrier. Per block the wave waits for its
// slot, reads all operands of the block into registers (K rows with ds_read_b128, V with the
// transposing ds_read_b64_tr_b16), issues the next loads into the slot, the score MFMAs between them, and
// computes. One slot keeps 16 KB per wave, 64 KB per CU, in flight, which covers the loaded latency of
// long streams; two slots (plans at G <= 4) start short sequences sooner: one sequence of 4096 tokens 9.43
// -> 8.93 us, 32768 26.8 -> 26.2, 128 of 16-512 at G = 1 95.2 -> 94.5; 64 x 1024 41.9 -> 42.4. Which batches
// run with one, and the uniform split's rule: launch_rules.h.
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
constexpr float kWScale = 32768.f;                       // scale of the weights in the PV product
constexpr float kLoScale = 2048.f;                       // and, on top, of their lower parts
constexpr float kDecLn2 = 0.69314718055994531f;

// LDS layouts: kLayWide holds two blocks per wave (one at G = 8); kLayOne one block (where that is faster,
// and the device-range kernel, whose own arrays it leaves room for); kLayStep (the fused cascade step, so that a CU holds the
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

// One wave's running state: the accumulators (times 2^15) of the columns above. m, the largest unscaled
// score, is the same in the four lanes of a column; l is the sum over the lane's own keys.
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

// q of a negative sm_scale (wave-uniform) with its signs turned: exact, and the scale is positive from there.
__device__ __forceinline__ void dec_sign_q(pf16x8 (&q)[4], float scale) {
    if (__builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, scale)) >= 0) return;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) q[ks] = __builtin_bit_cast(pf16x8, __builtin_bit_cast(pu32x4, q[ks]) ^ 0x80008000u);
}

// The constants of the weights' parts, per lane, and in vector registers (the compiler sees no
// constants, so that each step is one mixed-precision multiply-add): with hi = fp16(h p + t),
// u = b hi + (a p + k): w1 = fp16(u), truncated, and w2 = fp16(n w1 + u) are mid and lo in columns 8-15, where
// u = (p 2^15 - hi) 2^11 is exact, and hi and 0 in columns 0-7.
// An infinite V makes columns 0-7 infinite whatever its key's weight, as neither MFMA multiplies it by 0
// there: hi is rounded from p 2^15 + 1.25 2^-25, so that it is never 0, and w2's 0 is replaced by 2^-24.
// mid takes both differences back (k the second; exact but for that 2^-24, 2^-39 of the largest weight,
// where p >= 2^-15). (Half of hi in either MFMA does that too, but rounds the accumulators twice: 4096
// keys 4.2e-7 against 2.6e-7.)
struct DecWeights {
    float h, t, a, k, b, n;
    uint32_t w2;
};
__device__ __forceinline__ DecWeights dec_weights(int l16) {
    const bool low = (l16 & 8) != 0;
    DecWeights w = {kWScale, 1.25f * 0x1p-25f, low ? kWScale * kLoScale : 0.f, low ? -0x1p-24f * kLoScale : 0.f,
                    low ? -kLoScale : 1.f, -1.f, low ? 0u : 0x00010001u};
    asm("" : "+v"(w.h), "+v"(w.t), "+v"(w.a), "+v"(w.k), "+v"(w.b), "+v"(w.n), "+v"(w.w2));
    return w;
}

// The scores of a block, eight MFMAs: step n < 8 of them. Two chains of two per 16 keys: fewer roundings in
// a row than one of four, and half its latency.
__device__ __forceinline__ void dec_score(pf32x4 (&c)[2][2], const DecBlock& b, const pf16x8 (&q)[4], int n) {
    const int k = n >> 2, t = (n >> 1) & 1, i = n & 1;
    c[t][i] = mfma16x16x32(b.k[t][2 * i + k], q[2 * i + k], k ? c[t][i] : pf32x4{0.f, 0.f, 0.f, 0.f});
}

// A 32-key block from its scores c: online softmax (base 2), PV product. scale2: |sm_scale| log2(e), not 0
// (of a negative scale q carries the sign). tok0 / tok1: (wave-uniform) token index of the two pages' first
// slots; keys outside [tb, te) are masked (a padding page: tok1 >= te). A masked key weighs 0 and, since
// 0 * NaN is not 0, its V elements are zeroed as well: slots the cache never filled may hold any bits. Its
// K row only feeds its own score, which is replaced.
// The running maximum is an unscaled score, and a key's exponent is (score - m) scale2: never above 0,
// and as accurate for large scores as for small ones (with the scaled scores rounded first, q eight
// times N(0, 1): error of the output against 64 bits 6.7e-7 at 8192 keys, G = 8).
// A short segment is a block or two per wave, so what only edge blocks and first blocks do counts: a
// segment's first block (first) has nothing to rescale, and an absent second page is masked without
// looking at its keys. With the scores between the next loads and the flush's own loads in one trip, GPU
// time: one sequence of 2048 tokens 7.27 -> 6.98 us, 8 of 94-988 11.9 -> 11.35, 16 of 64-512 at G = 1 and 32
// kv heads 19.6 -> 19.2.
__device__ __forceinline__ void dec_block(DecState& st, DecBlock& b, const pf32x4 (&c)[2][2], int tok0, int tok1,
                                          int tb, int te, float scale2, const DecWeights& wc, int lg, bool first) {
    float x[8];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) x[4 * t + j] = c[t][0][j] + c[t][1][j];
    if (tok0 < tb || tok0 + kPage > te || tok1 + kPage > te) {   // wave-uniform: an edge block
        if (tok0 >= tb && tok0 + kPage <= te && tok1 >= te) {   // a whole page and none
#pragma unroll
            for (int e = 4; e < 8; ++e) x[e] = -INFINITY;
#pragma unroll
            for (int dt = 0; dt < 8; ++dt) {
                pu32x4 w = __builtin_bit_cast(pu32x4, b.v[dt]);
                w[2] = w[3] = 0u;
                b.v[dt] = __builtin_bit_cast(pf16x8, w);
            }
        } else {
            uint32_t keep[4] = {0u, 0u, 0u, 0u};
            const uint32_t n = (uint32_t)(te - tb);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint32_t k = (uint32_t)((e < 4 ? tok0 : tok1) - tb + 4 * lg + (e & 3));
                if (k < n) keep[e / 2] |= e & 1 ? 0xFFFF0000u : 0x0000FFFFu;
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
    }
    float mx = x[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) mx = fmaxf(mx, x[e]);
    const float mn = fmaxf(st.m, col4_reduce<true>(mx));
    if (first) {   // (wave-uniform)
        st.m = mn;
    } else if (__builtin_amdgcn_ballot_w64(mn > st.m)) {
        const float al = mn > st.m ? __builtin_amdgcn_exp2f((st.m - mn) * scale2) : 1.f;
        st.l *= al;
#pragma unroll
        for (int dt = 0; dt < 8; ++dt) st.acc[dt] *= al;
        st.m = mn;
    }
    const float ms = st.m == -INFINITY ? 0.f : st.m;
    pf16x8 w1, w2;
    float sum = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        float u[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float p = __builtin_amdgcn_exp2f((x[e + i] - ms) * scale2);
            sum += p;
            u[i] = fmaf((float)(_Float16)fmaf(p, wc.h, wc.t), wc.b, fmaf(p, wc.a, wc.k));
        }
        const auto w = __builtin_amdgcn_cvt_pkrtz(u[0], u[1]);   // (truncating: w2 takes what is left either way)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            w1[e + i] = (_Float16)w[i];
            w2[e + i] = (_Float16)fmaf((float)w[i], wc.n, u[i]);
        }
    }
    st.l += sum;
    pu32x4 w2b = __builtin_bit_cast(pu32x4, w2);
#pragma unroll
    for (int i = 0; i < 4; ++i) w2b[i] |= wc.w2;
    w2 = __builtin_bit_cast(pf16x8, w2b);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) st.acc[dt] = mfma16x16x32(b.v[dt], w1, st.acc[dt]);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) st.acc[dt] = mfma16x16x32(b.v[dt], w2, st.acc[dt]);
}

// End of a segment: the waves of a kv head hand their states (maximum, sum, output) to LDS, and
// each thread forms four outputs of one query head as a weighted sum over those waves, in wave
// order. Writes the G rows as the final fp16 out / lse (slot < 0) or as partial slot `slot`
// (normalized o, lse). Every thread of the workgroup calls it. With two flush buffers the one
// barrier suffices: a buffer is written again two flushes later, after the barrier of the next.
template <class C, int LAY, class ArgP>
__device__ __forceinline__ void dec_flush(DecShared<C, LAY>& S, DecState& st, int par, ArgP a,
                                          size_t row0, int slot, float scale2) {
    typedef DecShared<C, LAY> Sh;
    constexpr int G = C::G, HG = Sh::HG, WPH = C::WPH;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int l16 = lane & 15, lg = lane >> 4, w0 = wave / WPH * WPH;
    const int ltid = tid - w0 * 64;
    // where the rows go (read from the kernel arguments here, in the time of the arithmetic before the barrier)
    void* const dst = slot < 0 ? (void*)a->out : (void*)a->part_o;
    float* const dst_lse = slot < 0 ? a->lse : a->part_lse;
    const int ps = a->part_stride;
    const float L = col4_reduce<false>(st.l);
    // The parts together, still times 2^15 (in columns 0-7).
    float o[8][4], top = 0.f, ks = 1.f / kLoScale;
    asm("" : "+v"(ks));
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float hi = st.acc[dt][j];
            o[dt][j] = fmaf(dec_ror8(hi), ks, hi);
            top = fmaxf(top, fabsf(hi));
        }
    // An infinite V makes columns 0-7 infinite and columns 8-15 NaN or infinite of either sign (mid and lo
    // may be 0 or negative): the first are then the answer.
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
        for (int i = 0; i < (HG * 32 + WPH * 64 - 1) / (WPH * 64); ++i) {
            const int idx = ltid + i * WPH * 64;
            if ((i + 1) * WPH * 64 > HG * 32 && idx >= HG * 32) break;
            const int hh = idx >> 5, h = hp * HG + hh, d0 = 4 * (idx & 31);
            float mw[WPH], lw[WPH], M = -INFINITY;
            float4 ov[WPH];
#pragma unroll
            for (int w = 0; w < WPH; ++w) {
                mw[w] = S.m[bf][w0 + w][h];
                lw[w] = S.l[bf][w0 + w][h];
                ov[w] = *reinterpret_cast<const float4*>(&S.o[bf][w0 + w][hh][d0]);
            }
#pragma unroll
            for (int w = 0; w < WPH; ++w) M = fmaxf(M, mw[w]);
            float Ls = 0.f;
            float4 O = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int w = 0; w < WPH; ++w) {
                const float al = mw[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((mw[w] - M) * scale2);
                Ls = fmaf(al, lw[w], Ls);
                O.x = fmaf(al, ov[w].x, O.x);
                O.y = fmaf(al, ov[w].y, O.y);
                O.z = fmaf(al, ov[w].z, O.z);
                O.w = fmaf(al, ov[w].w, O.w);
            }
            const float ri = Ls > 0.f ? (1.f / kWScale) / Ls : 0.f;
            const float lse = Ls > 0.f ? fmaf(M, scale2, __builtin_amdgcn_logf(Ls)) * kDecLn2 : -INFINITY;
            O.x *= ri;
            O.y *= ri;
            O.z *= ri;
            O.w *= ri;
            const size_t e = slot < 0 ? row0 + h : ps > 0 ? (row0 + h) * (size_t)ps + slot : (size_t)slot * G + h;
            if (slot < 0) {
                const pf16x4 hv = {(_Float16)O.x, (_Float16)O.y, (_Float16)O.z, (_Float16)O.w};
                *reinterpret_cast<pf16x4*>(static_cast<_Float16*>(dst) + e * kHeadDim + d0) = hv;
            } else {
                *reinterpret_cast<float4*>(static_cast<float*>(dst) + e * kHeadDim + d0) = O;
            }
            if (d0 == 0) dst_lse[e] = lse;
        }
        if (Sh::NB == 1 || hp + 1 < G / HG) dec_barrier();
    }
}

}  // namespace
}  // namespace pdattn
