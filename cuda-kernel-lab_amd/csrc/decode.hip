// decode.hip -- paged split-KV GQA decode attention for gfx950 (CDNA4, wave64).
//
// What it computes (qilem/cuda-kernel-lab, 01_decode_attention.cu:76-255): for each sequence b,
// kv head kvh and each of the G query heads h sharing it, over a range of keys,
//   s_j = sm_scale * q_h . k_j,   o = sum_j softmax(s)_j v_j,   lse = ln sum_j exp(s_j)
// as a normalized partial (o, lse), then a log-sum-exp merge of the partials.
//
// How it maps to CDNA4:
//  * The segment runner (decode_body.h, run_segments below): 4-wave workgroups, one per CU, each wave
//    on one kv head and all its query heads, 32 keys at a time on fp16 MFMA, its pages staged by the
//    wave itself with direct global->LDS loads. A workgroup walks a list of segments (pieces of
//    sequences) for one kv head, or for two neighbouring heads of the same pages. The plan/run path
//    (decode_balanced_kernel) reads the list from a host-built plan; the reference-shaped uniform
//    split (decode_uniform_kernel) and the device-range drop-in (decode_ranges_kernel) build it in
//    the kernel from the device page table; the fused cascade step runs it beside the prefix pass.
//  * A uniform chunk too long for the runner's LDS page list runs on decode_partial_kernel, one
//    workgroup per (sequence, kv head, chunk), on the vector unit:
//    - K and V rows go straight from HBM into VGPRs with 16-byte non-temporal loads: a 256-byte row
//      (128 fp16) is read by 16 lanes, so one wave-wide load instruction reads 4 rows of one page, each
//      as whole 128-byte lines; a two-page ring, one page in flight;
//    - each lane takes the fp16 dot product of its slice of q_h and k_j with v_dot2_f32_f16, and the
//      16 lanes of a row sum with DPP row ops, which leaves the score in every lane of the row;
//    - every lane keeps its own online-softmax state over the keys it holds; the four states of a
//      wave are merged once at the end, and the waves of the workgroup through LDS.
//    Lane (r = lane / 16, c = lane % 16) holds rows 4 i + r of each page and dims 8 c .. 8 c + 7.
//  * Softmax runs in base 2 on log2(e)-prescaled scores with v_exp_f32 / v_log_f32
//    (exp(x) = 2^(x log2 e)); the running output is rescaled only when some max grows (a
//    wave-uniform branch), which after the first pages is rare.
#include <math.h>

#include <algorithm>
#include <cstdlib>

#include "launch_rules.h"
#include "pdattn_internal.h"
#include "timeline.h"

PD_TIMELINE_TABLE(decode)

#include "decode_body.h"

namespace pdattn {
namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.69314718055994531f;

// Compile-time shape of a decode kernel instance.
template <int G_, int NW_, int NBUF_>
struct Cfg {
    static constexpr int G = G_;                   // query heads per kv head
    static constexpr int LPR = 16;                 // lanes per 256-byte K/V row
    static constexpr int NW = NW_;                 // waves per workgroup
    static constexpr int NBUF = NBUF_;             // pages held in VGPRs per wave (NBUF-1 in flight)
    static constexpr int NT = NW * 64;
    static constexpr int RPI = 64 / LPR;           // rows per wave-wide load
    static constexpr int PPL = 16 / LPR;           // 16-byte pieces per lane per row
    static constexpr int RG = kPage / RPI;         // rows of each page held by one lane
    static constexpr int DPL = PPL * 8;            // head dims held by one lane
};

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}

// Sums over the 16 lanes (a DPP row) that share one K/V row of N independent values, one
// DPP step at a time across all of them.
template <int N>
__device__ __forceinline__ void row_sum_all(float* v) {
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] += dpp<0xB1>(v[j]);
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] += dpp<0x4E>(v[j]);
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] += dpp<0x141>(v[j]);
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] += dpp<0x140>(v[j]);
}

// Combine of the four row groups of a wave (lanes 16 apart hold the same head dims), leaving the result
// in every lane: v_permlane16_swap / v_permlane32_swap pair whole 16-lane rows, all in the VALU. After
// swap(a, b) the two results hold, in every lane, the values of both rows of its pair (rows
// r and r^1 for the 16-lane swap, r and r^2 for the 32-lane swap), always in the same order, so
// r0 + r1 is bitwise the same in all lanes. The second operand is passed through an empty asm
// statement: given the same SSA value twice, the compiler treats the two results as equal and
// drops the second one. The statement is not volatile, so the many independent reductions of a
// merge can still be interleaved by the scheduler.
__device__ __forceinline__ unsigned opaque_copy(unsigned v) {
    asm("" : "+v"(v));
    return v;
}
template <bool ROWS32>
__device__ __forceinline__ void row_pair(float v, float& a, float& b) {
    const unsigned x = __builtin_bit_cast(unsigned, v);
    unsigned r0, r1;
    if constexpr (ROWS32) {
        const auto r = __builtin_amdgcn_permlane32_swap(x, opaque_copy(x), false, false);
        r0 = r[0]; r1 = r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(x, opaque_copy(x), false, false);
        r0 = r[0]; r1 = r[1];
    }
    a = __builtin_bit_cast(float, r0);
    b = __builtin_bit_cast(float, r1);
}

// Reinterprets one 32-bit word as two fp16. The word is taken by value: bit-casting an
// ext-vector element expression in place was observed to read element 0 for every index.
__device__ __forceinline__ f16x2 as_h2(uint32_t w) { return __builtin_bit_cast(f16x2, w); }

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }

__device__ __forceinline__ float xgroup_sum(float v) {
    float a, b;
    row_pair<false>(v, a, b);
    row_pair<true>(a + b, a, b);
    return a + b;
}
__device__ __forceinline__ float xgroup_max(float v) {
    float a, b;
    row_pair<false>(v, a, b);
    row_pair<true>(fmaxf(a, b), a, b);
    return fmaxf(a, b);
}

template <class C>
struct WaveState {
    float m[C::G];                // running max, log2 units
    float l[C::G];                // running sum of 2^(x - m)
    float o[C::G][C::DPL];        // running unnormalized output slice
};

template <class C>
struct PageRegs {
    u32x4 k[C::RG][C::PPL];
    u32x4 v[C::RG][C::PPL];
};

template <int G, int NW>
struct Smem {
    float m[NW][G];
    float l[NW][G];
    float o[NW][G][kHeadDim];
    float fo[G][kHeadDim];    // combined, normalized output of the workgroup
    float flse[G];            // combined lse (natural log)
};

// A page of one kv head seen through a buffer resource: base = cache + page * page_bytes +
// kvh * 256, num_records = the bytes from there to the end of the page, so every lane's offset is
// in range. A padding slot of the ring uses num_records = 0: its loads return zeros without a
// memory access, while the ring still issues the same loads in every slot (exact wait counts).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t page_rsrc(const uint8_t* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), (short)0, (int)bytes, 0x00020000);
}

template <class C>
__device__ __forceinline__ void load_page_rsrc(PageRegs<C>& pr, __amdgpu_buffer_rsrc_t rk,
                                               __amdgpu_buffer_rsrc_t rv, uint32_t lbase, uint32_t rstride) {
#pragma unroll
    for (int i = 0; i < C::RG; ++i)
#pragma unroll
        for (int kk = 0; kk < C::PPL; ++kk) {
            const int off = (int)(lbase + i * rstride + kk * (C::LPR * 16));
            // aux = 2: non-temporal (K/V bytes are read once)
            pr.k[i][kk] = __builtin_amdgcn_raw_buffer_load_b128(rk, off, 0, 2);
            pr.v[i][kk] = __builtin_amdgcn_raw_buffer_load_b128(rv, off, 0, 2);
        }
}

// One page: scores, online-softmax update, PV accumulation. tok0 is the (wave-uniform) token
// index of the page's first slot, and this lane's row of row group i is slot r + i * RPI; keys
// outside [tb, te) are masked. A masked key gets weight 0, and on a page that holds masked keys
// (the first or last page of a range) their V rows are zeroed as well, so that slots the cache
// never filled (NaN or Inf bit patterns in unused slots of a last page) cannot reach the output
// through 0 * v.
template <class C>
__device__ __forceinline__ void page_step(WaveState<C>& st, PageRegs<C>& pr,
                                          const f16x2 (&qv)[C::G][C::PPL][4], int tok0, int r,
                                          int tb, int te, float scale2) {
    using g = C;
    constexpr int G = C::G;
    const int tok_r = tok0 + r;
    if (tok0 < tb || tok0 + kPage > te) {   // wave-uniform: an edge page
#pragma unroll
        for (int i = 0; i < g::RG; ++i) {
            const int tok = tok_r + i * g::RPI;
            if (tok < tb || tok >= te) {
#pragma unroll
                for (int kk = 0; kk < g::PPL; ++kk) pr.v[i][kk] = u32x4{0u, 0u, 0u, 0u};
            }
        }
    }
    // Scores: the lane's partial dot products of every (row, head) first, then each DPP step of
    // the row sums across all of them, so that every dependent DPP add has RG * G - 1 independent
    // instructions in front of it instead of a hazard stall (s_nop).
    float x[g::RG][G];
#pragma unroll
    for (int i = 0; i < g::RG; ++i)
#pragma unroll
        for (int h = 0; h < G; ++h) {
            float acc = 0.f;
#pragma unroll
            for (int kk = 0; kk < g::PPL; ++kk)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc = __builtin_amdgcn_fdot2(qv[h][kk][e],
                                                 as_h2(pr.k[i][kk][e]), acc,
                                                 false);
            x[i][h] = acc;
        }
    row_sum_all<g::RG * G>(&x[0][0]);
#pragma unroll
    for (int i = 0; i < g::RG; ++i) {
        const int tok = tok_r + i * g::RPI;
        const bool ok = tok >= tb && tok < te;
#pragma unroll
        for (int h = 0; h < G; ++h) x[i][h] = ok ? x[i][h] * scale2 : -INFINITY;
    }
    float mn[G];
    bool grow = false;
#pragma unroll
    for (int h = 0; h < G; ++h) {
        float mt = x[0][h];
#pragma unroll
        for (int i = 1; i < g::RG; ++i) mt = fmaxf(mt, x[i][h]);
        mn[h] = fmaxf(st.m[h], mt);
        grow |= mn[h] > st.m[h];
    }
    if (__builtin_amdgcn_ballot_w64(grow)) {
#pragma unroll
        for (int h = 0; h < G; ++h) {
            const float a = (mn[h] > st.m[h]) ? fast_exp2(st.m[h] - mn[h]) : 1.f;
            st.l[h] *= a;
#pragma unroll
            for (int d = 0; d < g::DPL; ++d) st.o[h][d] *= a;
            st.m[h] = mn[h];
        }
    }
#pragma unroll
    for (int h = 0; h < G; ++h) {
        const float ms = (st.m[h] == -INFINITY) ? 0.f : st.m[h];
#pragma unroll
        for (int i = 0; i < g::RG; ++i) {
            const float p = fast_exp2(x[i][h] - ms);
            st.l[h] += p;
#pragma unroll
            for (int kk = 0; kk < g::PPL; ++kk)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const f16x2 vv = as_h2(pr.v[i][kk][e]);
                    float* od = &st.o[h][kk * 8 + 2 * e];
                    od[0] = fmaf((float)vv[0], p, od[0]);
                    od[1] = fmaf((float)vv[1], p, od[1]);
                }
        }
    }
}

// Attention of the G query heads of (b, kvh) over keys [t0, t1) of one sequence. pages[i] is the
// physical page holding tokens [tok_base + 16 i, tok_base + 16 i + 16) (global memory or LDS).
// Leaves the normalized output in sm.fo and the lse in sm.flse (all threads of the workgroup
// must call it; it ends with a barrier).
template <class C>
__device__ __forceinline__ void process_range(Smem<C::G, C::NW>& sm, const _Float16* qrow, const uint8_t* kbase,
                              const uint8_t* vbase, const int32_t* pages, int tok_base, int t0, int t1,
                              int Hkv, int kvh, float scale2) {
    using g = C;
    constexpr int G = C::G, NW = C::NW, NBUF = C::NBUF;
    // the wave index is made wave-uniform explicitly: the page counts and buffer resources derived
    // from it must live in scalar registers (a non-uniform resource turns each load into a loop)
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = lane / g::LPR, c = lane % g::LPR;

    f16x2 qv[G][g::PPL][4];
#pragma unroll
    for (int h = 0; h < G; ++h)
#pragma unroll
        for (int kk = 0; kk < g::PPL; ++kk) {
            const u32x4 raw =
                *reinterpret_cast<const u32x4*>(qrow + h * kHeadDim + (kk * g::LPR + c) * 8);
#pragma unroll
            for (int e = 0; e < 4; ++e) qv[h][kk][e] = as_h2(raw[e]);
        }

    WaveState<C> st;
#pragma unroll
    for (int h = 0; h < G; ++h) {
        st.m[h] = -INFINITY;
        st.l[h] = 0.f;
#pragma unroll
        for (int d = 0; d < g::DPL; ++d) st.o[h][d] = 0.f;
    }

    if (t1 > t0) {
        const int pfirst = (t0 - tok_base) / kPage, plast = (t1 - 1 - tok_base) / kPage;
        const int npg = plast - pfirst + 1;
        const int nmine = npg > wave ? (npg - wave + NW - 1) / NW : 0;
        const uint32_t page_bytes = (uint32_t)(kPage * Hkv * 256);
        const uint32_t lbase = (uint32_t)(r * Hkv * 256 + c * 16);
        const uint32_t rstride = (uint32_t)(g::RPI * Hkv * 256);
        // slot j of the window: page j of it through a buffer resource over the rest of the page
        // (from this kv head's row), or, past the end, a zero-length resource whose loads return
        // zeros without a memory access, so every iteration issues the same loads (exact waits)
        // and no page is read twice
        auto issue = [&](PageRegs<C>& b, int pidv, int j, int cnt) {
            const uint8_t* kb = kbase;
            const uint8_t* vb = vbase;
            uint32_t nrec = 0;
            if (j < cnt) {
                const size_t off = (size_t)(uint32_t)__builtin_amdgcn_readlane(pidv, j) * page_bytes +
                                   (size_t)kvh * 256;
                kb += off;
                vb += off;
                nrec = page_bytes - (uint32_t)kvh * 256;
            }
            load_page_rsrc<C>(b, page_rsrc(kb, nrec), page_rsrc(vb, nrec), lbase, rstride);
        };
        for (int base = 0; base < nmine; base += 64) {
            const int cnt = min(64, nmine - base);
            // lane j holds the physical page of this wave's (base + j)-th page
            const int pidv = lane < cnt ? pages[pfirst + wave + NW * (base + lane)] : 0;
            // ring of NBUF pages in VGPRs: page i lives in buf[i % NBUF]; NBUF-1 are in flight
            // while one is computed
            PageRegs<C> buf[NBUF];
#pragma unroll
            for (int u = 0; u < NBUF - 1; ++u) issue(buf[u], pidv, u, cnt);
            for (int it = 0; it < cnt; it += NBUF) {
#pragma unroll
                for (int u = 0; u < NBUF; ++u) {
                    if (it + u >= cnt) break;
                    issue(buf[(u + NBUF - 1) % NBUF], pidv, it + u + NBUF - 1, cnt);
                    page_step<C>(st, buf[u], qv, tok_base + (pfirst + wave + NW * (base + it + u)) * kPage, r,
                                 t0, t1, scale2);
                }
            }
        }
    }

    // merge the four row-group states of this wave (lanes 16 apart hold the same dims)
#pragma unroll
    for (int h = 0; h < G; ++h) {
        const float M = xgroup_max(st.m[h]);
        const float a = (st.m[h] == -INFINITY) ? 0.f : fast_exp2(st.m[h] - M);
        st.l[h] = xgroup_sum(st.l[h] * a);
#pragma unroll
        for (int d = 0; d < g::DPL; ++d) st.o[h][d] = xgroup_sum(st.o[h][d] * a);
        st.m[h] = M;
    }
    if (lane < g::LPR) {
#pragma unroll
        for (int h = 0; h < G; ++h)
#pragma unroll
            for (int kk = 0; kk < g::PPL; ++kk)
#pragma unroll
                for (int e = 0; e < 8; ++e) sm.o[wave][h][(kk * g::LPR + c) * 8 + e] = st.o[h][kk * 8 + e];
        if (lane == 0) {
#pragma unroll
            for (int h = 0; h < G; ++h) {
                sm.m[wave][h] = st.m[h];
                sm.l[wave][h] = st.l[h];
            }
        }
    }
    __syncthreads();
    for (int idx = tid; idx < G * kHeadDim; idx += NW * 64) {
        const int h = idx / kHeadDim, d = idx % kHeadDim;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < NW; ++w) M = fmaxf(M, sm.m[w][h]);
        float L = 0.f, O = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const float a = (sm.m[w][h] == -INFINITY) ? 0.f : fast_exp2(sm.m[w][h] - M);
            L += a * sm.l[w][h];
            O += a * sm.o[w][h][d];
        }
        sm.fo[h][d] = L > 0.f ? O / L : 0.f;
        if (d == 0) sm.flse[h] = L > 0.f ? (M + fast_log2(L)) * kLn2 : -INFINITY;
    }
    __syncthreads();
}


// Kernel arguments of the balanced kernel read in place from the kernarg segment. The pointer is
// laundered through an empty asm statement at every use, so the compiler reloads those fields
// (scalar loads, cached) where they are needed instead of holding them in SGPRs across the page
// loop, where they would spill. The kernarg-segment intrinsic is only valid in the kernel body
// itself (in a called function it evaluates to null), so kargs() is called only from the kernel
// and the pointer is passed down to the (force-inlined) helpers.
typedef const __attribute__((address_space(4))) BalArgs* KArgPtr;
__device__ __forceinline__ KArgPtr kargs() {
    KArgPtr p = (KArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

// ---- merging partial states ----------------------------------------------------------------
// Log-sum-exp merge of one row (128 dims) from partial states in a fixed order (merge_states,
// 01_decode_attention.cu:238-255), by one workgroup of kMergeThreads = 4 waves (or four of one wave,
// merge_d0 below), with no LDS and no barrier. The sources are two lists, A then B (a pair's partial slots, then a cascade row's prefix
// partials): source k of a list has its lse at lse[k * stride] and its output row at
// o[k * stride * 128]. Wave w covers dims [32 w, 32 w + 32): lane 8 q + r holds the 4 dims
// 32 w + 4 q .. of sources r, r + 8, r + 16, ... of the two lists as one. 8 U sources (U chosen at the
// launch) are loaded before any is waited for (one round trip), each lane folds its sources in order (A's,
// then B's), and the 8 source lanes of a quad are then combined by three DPP exchanges (lane
// distances 1, 2, then the other quad of the 8-lane half row): a fixed order, so the result is
// deterministic. keepA(k), evaluated after the loads, drops source k of A (a slot the decode launch
// did not write). The state is left in every lane: merged output acc / ws, lse m + ln ws.
constexpr int kMergeThreads = 256;
struct MState {
    float m, ws;
    float4 acc;
};
struct MSrc {
    const float* lse;
    const float* o;
    size_t stride;
    int n;
};

template <int CTRL>
__device__ __forceinline__ void mstate_fold_dpp(MState& s) {
    const float m2 = dpp<CTRL>(s.m), w2 = dpp<CTRL>(s.ws);
    const float x2 = dpp<CTRL>(s.acc.x), y2 = dpp<CTRL>(s.acc.y);
    const float z2 = dpp<CTRL>(s.acc.z), u2 = dpp<CTRL>(s.acc.w);
    const float M = fmaxf(s.m, m2);
    const float s1 = (s.m == -INFINITY) ? 0.f : fast_exp2((s.m - M) * kLog2e);
    const float s2 = (m2 == -INFINITY) ? 0.f : fast_exp2((m2 - M) * kLog2e);
    s.ws = s.ws * s1 + w2 * s2;
    s.acc.x = s.acc.x * s1 + x2 * s2;
    s.acc.y = s.acc.y * s1 + y2 * s2;
    s.acc.z = s.acc.z * s1 + z2 * s2;
    s.acc.w = s.acc.w * s1 + u2 * s2;
    s.m = M;
}

// The first of this lane's 4 dims. A row is one workgroup of 4 waves (32 dims each), or (WIDE) four
// workgroups of one wave, blockIdx % 4 being the wave's place: few rows with many sources each then
// spread over four times as many CUs.
template <bool WIDE>
__device__ __forceinline__ int merge_d0() {
    const int w = WIDE ? (int)(blockIdx.x & 3) : (int)(threadIdx.x >> 6);
    return 32 * w + 4 * (int)((threadIdx.x & 63) >> 3);
}
template <bool WIDE>
__device__ __forceinline__ int merge_row() { return WIDE ? (int)(blockIdx.x >> 2) : (int)blockIdx.x; }

// The sources of a row are list A then list B, as one list of A.n + B.n: source k is A's k-th
// for k < A.n, else B's (k - A.n)-th. Lane r of each 8-lane group takes sources k0 + r + 8 u
// (u < U), loaded unconditionally: a lane past the last source reloads the last one, and
// the list a source comes from is a per-lane select of its address, so every lane issues the same
// loads and no load waits for another (conditional loads would make the compiler copy the
// results, and wait for them, where the branches join). 8 U sources per round trip.
template <int U>
__device__ __forceinline__ void merge_load(const MSrc& A, const MSrc& B, int k0, int d0, float (&l)[U],
                                           float4 (&o)[U]) {
    const int r = threadIdx.x & 7, n = A.n + B.n;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int k = min(k0 + r + 8 * u, n - 1);
        const bool inA = k < A.n;
        const size_t ia = (size_t)k * A.stride, ib = (size_t)(k - A.n) * B.stride;
        l[u] = *(inA ? A.lse + ia : B.lse + ib);
        o[u] = *reinterpret_cast<const float4*>((inA ? A.o + ia * kHeadDim : B.o + ib * kHeadDim) + d0);
    }
}
// Folds this lane's loaded sources into s in order, branch-free (a dropped or empty source weighs 0
// and its values are replaced, not multiplied, so unused slots may hold anything): with every
// loaded value used unconditionally, the compiler keeps all the loads ahead of the first wait.
// For a kept source this is the online log-sum-exp rule: the running state (m, ws, acc) is rescaled
// by exp(m - max(m, l)) (exactly 1 when l <= m) and the source (lse l, normalized output o) added
// with weight exp(l - max(m, l)); an empty source (l = -inf) weighs 0. keepA(k) drops sources of
// list A (B's are all kept).
template <int U, class KeepA>
__device__ __forceinline__ void merge_fold(MState& s, const MSrc& A, const MSrc& B, int k0,
                                           const float (&l)[U], const float4 (&o)[U], KeepA keepA) {
    const int r = threadIdx.x & 7, n = A.n + B.n;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int k = k0 + r + 8 * u;
        const bool ok = k < n && (k >= A.n || keepA(k)) && l[u] != -INFINITY;
        const float lv = ok ? l[u] : -INFINITY;
        const float4 ov = ok ? o[u] : make_float4(0.f, 0.f, 0.f, 0.f);
        const float mn = fmaxf(s.m, lv);
        const float sc = (s.m == -INFINITY) ? 0.f : fast_exp2((s.m - mn) * kLog2e);
        const float w = ok ? fast_exp2((lv - mn) * kLog2e) : 0.f;
        s.ws = fmaf(s.ws, sc, w);
        s.acc.x = fmaf(w, ov.x, s.acc.x * sc);
        s.acc.y = fmaf(w, ov.y, s.acc.y * sc);
        s.acc.z = fmaf(w, ov.z, s.acc.z * sc);
        s.acc.w = fmaf(w, ov.w, s.acc.w * sc);
        s.m = mn;
    }
}

template <int U, class KeepA>
__device__ __forceinline__ MState merge_lanes(const MSrc& A, const MSrc& B, int d0, KeepA keepA) {
    constexpr int SPT = 8 * U;   // sources per round trip
    MState s{-INFINITY, 0.f, make_float4(0.f, 0.f, 0.f, 0.f)};
    const int n = A.n + B.n;
    if (n > 0) {
        float l[U];
        float4 o[U];
        merge_load<U>(A, B, 0, d0, l, o);
        __builtin_amdgcn_sched_barrier(0);   // every load above is issued before anything waits
        merge_fold<U>(s, A, B, 0, l, o, keepA);
        for (int k0 = SPT; k0 < n; k0 += SPT) {
            merge_load<U>(A, B, k0, d0, l, o);
            merge_fold<U>(s, A, B, k0, l, o, keepA);
        }
    }
    mstate_fold_dpp<0xB1>(s);    // quad_perm [1,0,3,2]
    mstate_fold_dpp<0x4E>(s);    // quad_perm [2,3,0,1]
    mstate_fold_dpp<0x141>(s);   // row_half_mirror: the other quad of the 8-lane half row
    return s;
}

// Writes a merged row: lane 0 of each 8-lane group its 4 fp16 outputs, the first of them the lse.
// A row whose every source is empty gets out = 0, lse = -inf.
__device__ __forceinline__ void merge_store(const MState& s, int d0, _Float16* out_row, float* lse_out) {
    if ((threadIdx.x & 7) != 0) return;
    const float inv = s.ws > 0.f ? 1.f / s.ws : 0.f;
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    const h4 hv = {(_Float16)(s.acc.x * inv), (_Float16)(s.acc.y * inv), (_Float16)(s.acc.z * inv),
                   (_Float16)(s.acc.w * inv)};
    *reinterpret_cast<h4*>(out_row + d0) = hv;
    if (d0 == 0) *lse_out = s.ws > 0.f ? s.m + fast_log2(s.ws) * kLn2 : -INFINITY;
}

// ---- uniform chunks: the reference's decode_partial launch shape -------------------------
template <class C>
__global__ __launch_bounds__(C::NT) void decode_partial_kernel(PartialArgs a) {
    constexpr int G = C::G;
    __shared__ Smem<G, C::NW> sm;
    const int chunk = blockIdx.x;
    const int b = blockIdx.y / a.Hkv, kvh = blockIdx.y % a.Hkv;
    const int pb = a.kv_indptr[b];
    const int np = a.kv_indptr[b + 1] - pb;
    const int len = np > 0 ? (np - 1) * kPage + min(kPage, max(1, a.kv_last[b])) : 0;
    const int kbeg = a.kv_start + chunk * a.chunk_tokens;
    const int kend = min(len, kbeg + a.chunk_tokens);
    process_range<C>(sm, a.q + ((size_t)b * a.Hq + kvh * G) * kHeadDim, a.k, a.v,
                     a.kv_indices + pb, 0, kbeg, kend, a.Hkv, kvh, a.scale_log2);
    if (a.out != nullptr) {
        // the only chunk: its normalized state is the result (the merge's weight would be 1)
        const size_t row0 = (size_t)b * a.Hq + kvh * G;
        for (int idx = threadIdx.x; idx < G * kHeadDim; idx += C::NT) {
            const int h = idx / kHeadDim, d = idx % kHeadDim;
            a.out[(row0 + h) * kHeadDim + d] = (_Float16)sm.fo[h][d];
            if (d == 0) a.lse[row0 + h] = sm.flse[h];
        }
        return;
    }
    for (int idx = threadIdx.x; idx < G * kHeadDim; idx += C::NT) {
        const int h = idx / kHeadDim, d = idx % kHeadDim;
        const size_t slot = ((size_t)b * a.Hq + kvh * G + h) * a.part_stride + a.chunk_base + chunk;
        a.part_o[slot * kHeadDim + d] = sm.fo[h][d];
        if (d == 0) a.part_lse[slot] = sm.flse[h];
    }
}

// ---- log-sum-exp merge: the reference's merge_states launch shape -------------------------
// One workgroup per row, `num_chunks` consecutive partial slots.
template <int U, bool WIDE>
__global__ __launch_bounds__(kMergeThreads) void merge_states_kernel(const float* __restrict__ part_o,
                                                                      const float* __restrict__ part_lse,
                                                                      _Float16* __restrict__ out,
                                                                      float* __restrict__ lse_out,
                                                                      int num_chunks) {
    const size_t row = merge_row<WIDE>();
    const int d0 = merge_d0<WIDE>();
    const MSrc A{part_lse + row * num_chunks, part_o + row * num_chunks * kHeadDim, 1, num_chunks};
    const MSrc B{part_lse, part_o, 1, 0};
    const MState st = merge_lanes<U>(A, B, d0, [](int) { return true; });
    merge_store(st, d0, out + row * kHeadDim, lse_out + row);
}

// ---- balanced launch -------------------------------------------------------------------------
// Merge of the pairs listed by the planner: one workgroup per row (entry, head). Sources: the
// pair's partial slots in order, then the row's extra partials (cascade prefix chunks). A list
// whose header does not carry the launch's tag, or an entry outside the batch or the workspace's
// slots, is someone else's bytes: the row is left alone.
// RECT (slots laid out by entry, cmax > 0): the list header, the entry and every partial are loaded
// in one round trip (the header and entry as vector loads through a zero lane offset the compiler
// cannot see through, so that they count against the same counter as the partials and nothing is
// waited for before all are issued). Otherwise the partials follow the entry.
template <bool RECT, int U, bool WIDE>
__global__ __launch_bounds__(kMergeThreads) void merge_split_kernel(MergeArgs a) {
    const int G = a.G, er = merge_row<WIDE>(), e = er / G, h = er - e * G, d0 = merge_d0<WIDE>();
    int z = 0;
    asm volatile("v_mov_b32 %0, 0" : "=v"(z));
    // header {tag, n_entries, cmax, 0} and entry {b, kvh, slot0, nc}
    const int4 hd = *reinterpret_cast<const int4*>(a.list + z);
    const int4 en = *reinterpret_cast<const int4*>(a.list + 4 + 4 * (size_t)e + z);
    const int n_extra = a.n_extra;
    MState st;
    if constexpr (RECT) {
        const int cmax = a.cmax;
        const size_t sl0 = (size_t)e * cmax * G + h;   // slot e * cmax, head h
        const size_t row = (size_t)e * G + h;          // with extra partials entry e is pair e
        const MSrc A{a.part_lse + sl0, a.part_o + sl0 * kHeadDim, (size_t)G, cmax};
        const MSrc B{a.extra_lse + row * n_extra, a.extra_o + row * n_extra * kHeadDim, 1, n_extra};
        st = merge_lanes<U>(A, B, d0, [&](int k) { return k < en.w; });
        if (en.w > cmax || (n_extra > 0 && (int64_t)en.x * a.Hkv + en.y != (int64_t)e)) return;
    } else {
        if (hd.x != a.tag || en.z < 0 || en.w < 0 || (int64_t)en.z + en.w > a.n_slots) return;
        if (en.x < 0 || en.x >= a.B || en.y < 0 || en.y >= a.Hkv) return;
        const size_t sl0 = (size_t)en.z * G + h;
        const size_t row = ((size_t)en.x * a.Hkv + en.y) * G + h;
        const MSrc A{a.part_lse + sl0, a.part_o + sl0 * kHeadDim, (size_t)G, en.w};
        const MSrc B{a.extra_lse + row * n_extra, a.extra_o + row * n_extra * kHeadDim, 1, n_extra};
        st = merge_lanes<U>(A, B, d0, [](int) { return true; });
    }
    if (hd.x != a.tag || en.x < 0 || en.x >= a.B || en.y < 0 || en.y >= a.Hkv) return;
    const size_t orow = ((size_t)en.x * a.Hkv + en.y) * G + h;
    merge_store(st, d0, a.out + orow * kHeadDim, a.lse + orow);
}

// The page list of the segments staged in S.sd, where it is not one range of kv_indices: item i of
// the list is found in the segment whose range [qa, qa + npg) holds it (LDS reads only: a search
// loop with loads in flight would wait for them at every iteration), then all ids are loaded in one
// round trip. Ends with a barrier.
template <class C, int LAY>
__device__ __forceinline__ void stage_pages(const BalArgs& a, DecShared<C, LAY>& S, int nseg) {
    constexpr int NT = C::NT, PMAX = DecShared<C, LAY>::PGMAX / NT;
    const int tid = threadIdx.x;
    const int* seg = S.sd[0] + 8;
    const int npages = __builtin_amdgcn_readfirstlane(seg[(nseg - 1) * kSegInts + 2] + seg[(nseg - 1) * kSegInts + 3]);
    const int32_t* kvi = a.kv_indices;
    int src[PMAX];
#pragma unroll
    for (int k = 0; k < PMAX; ++k) {
        const int i = tid + k * NT;
        src[k] = -1;
        if (i < npages) {
            int si = 0;
            while (si + 1 < nseg && seg[(si + 1) * kSegInts + 2] <= i) ++si;
            src[k] = seg[si * kSegInts + 6] + (i - seg[si * kSegInts + 2]);
        }
    }
    // (unconditional within the list, so one round trip; none at all for a workgroup whose items
    // hold no page, whose kv_indices may be empty)
    if (npages > 0) {
        int pv[PMAX];
#pragma unroll
        for (int k = 0; k < PMAX; ++k) pv[k] = kvi[max(src[k], 0)];
#pragma unroll
        for (int k = 0; k < PMAX; ++k)
            if (tid + k * NT < npages) S.pg[tid + k * NT] = pv[k];
    }
    __syncthreads();
}

// The segments staged in S.sd (nseg of them, one block per kv head) with their page ids in S.pg:
// every wave streams its pages of all segments, two pages at a time, flushing each segment at its
// end. A kv head's WPH waves take every WPH-th page of a segment each. The next block's loads, the
// next segment's first block included, are in flight while a block is computed or a segment
// flushed. All threads of the workgroup call it. qpre: the q rows are already in qn.
template <class C, int LAY>
__device__ __forceinline__ void run_segments(const BalArgs& a, DecShared<C, LAY>& S, int nseg,
                                             pf16x8 (&qn)[4], bool qpre = false) {
    typedef DecShared<C, LAY> Sh;
    constexpr int G = C::G, WPH = C::WPH, NS = Sh::NS;
    int* pg = S.pg;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hh = wave / WPH, lw = wave % WPH;
    const int l16 = lane & 15, lg = lane >> 4;
    // this head's segments: one window for the segment being computed, one for the loads' cursor
    SegWin cur, nxt;
    cur.init(S.sd[hh] + 8);
    auto wcount = [&](int npg) { return npg > lw ? (npg - lw + WPH - 1) / WPH : 0; };
    // this lane's q pieces of segment si: head (l16 & 7) % G, dims 32 ks + 8 lg ..
    auto qload = [&](int si) {
        const _Float16* qp = a.q + ((size_t)cur.get(si, 0) * a.Hq + (size_t)cur.get(si, 1) * G + (l16 & 7) % G) * kHeadDim;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) qn[ks] = *reinterpret_cast<const pf16x8*>(qp + 32 * ks + 8 * lg);
    };
    if (NS == 1 && !qpre) qload(0);

    // The cursor of the loads: blocks in stream order. advance() leaves the next block's page ids,
    // head and page count (0 at the end) in scalar registers, read from LDS while the block before
    // is computed, so that issue() follows the operand reads at once.
    const uint32_t page_bytes = (uint32_t)(kPage * a.Hkv * 256);
    nxt = cur;
    int ps = 0, pslot = 0, pcnt = wcount(nxt.get(0, 3));
    int have = 0, pid0 = 0, pid1 = 0, pkvh = 0, pb = 0;
    auto advance = [&]() {
        while (ps < nseg && pslot >= pcnt) {
            ++ps;
            pslot = 0;
            pcnt = ps < nseg ? wcount(nxt.get(ps, 3)) : 0;
        }
        have = ps < nseg ? min(2, pcnt - pslot) : 0;
        if (have > 0) {
            const int qa = nxt.get(ps, 2) + lw + WPH * pslot;
            const int pv = pg[(lane & 1) && have > 1 ? qa + WPH : qa];
            pid0 = __builtin_amdgcn_readlane(pv, 0);
            pid1 = __builtin_amdgcn_readlane(pv, 1);
            pkvh = nxt.get(ps, 1);
            pb = nxt.get(ps, 0);
            pslot += 2;
        }
    };
    // Row n = 4 i + lane / 16 of a page, LDS position p = lane % 16 of it: chunk p ^ n of K, p ^ ((n & 7)
    // << 1) of V (the swizzles that dec_read_block reads).
    uint32_t koff[4], voff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = 4 * i + lg;
        koff[i] = (uint32_t)(n * a.Hkv * 256 + ((l16 ^ n) << 4));
        voff[i] = (uint32_t)(n * a.Hkv * 256 + ((l16 ^ ((n & 7) << 1)) << 4));
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)S.slot[wave][0];
    // (NS = 2) this lane's 16 bytes of a block's q rows, LDS position lane of them: row r = (lane / 16) % G
    const uint32_t qoff = (uint32_t)((lg % G) * 256 + (((l16 >> 2 ^ (lg % G)) << 2 | (l16 & 3)) << 4));
    int sl = 0, nfl = 0;   // the slot of the next block, computed and loaded; loads of the newest block
    const uint8_t* const kc = a.k;
    const uint8_t* const vc = a.v;
    // Issues the next block's loads, with step n of `other` (n < 8: the scores of the block just read)
    // between them: a load takes the issue of 16 cycles, and so does an MFMA.
    auto issue = [&](auto other) {
        nfl = 0;
        if (have <= 0) {
#pragma unroll
            for (int i = 0; i < 8; ++i) other(i);
            return;
        }
        nfl = 8 * have + 1;
        const uint32_t lds = lds0 + (uint32_t)(sl * Sh::SLOT);
        if constexpr (NS > 1)
            dec_dma_q(a.q + ((size_t)pb * a.Hq + (size_t)pkvh * G) * kHeadDim, qoff, lds + kDecSlotBytes);
        {
            const size_t off = (size_t)(uint32_t)pid0 * page_bytes + (size_t)pkvh * 256;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (i < 4) dec_dma(kc + off, koff[i], lds + 1024 * i);
                else dec_dma(vc + off, voff[i - 4], lds + 2 * kDecPageBytes + 1024 * (i - 4));
                other(i);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (have > 1) {
            const size_t off = (size_t)(uint32_t)pid1 * page_bytes + (size_t)pkvh * 256;
#pragma unroll
            for (int i = 0; i < 4; ++i) dec_dma(kc + off, koff[i], lds + kDecPageBytes + 1024 * i);
#pragma unroll
            for (int i = 0; i < 4; ++i) dec_dma(vc + off, voff[i], lds + 3 * kDecPageBytes + 1024 * i);
        }
    };
    auto nothing = [](int) {};

    PD_STAMP(2);
    advance();
    issue(nothing);
    advance();
    if constexpr (NS > 1) {
        sl = 1;
        issue(nothing);
        advance();
        sl = 0;
    }
    const DecWeights wc = dec_weights(l16);
    // (a scale of 0 would make a masked key's -inf a NaN: every exponent is then 0 all the same)
    float scale = a.scale_log2 == 0.f ? 0x1p-126f : a.scale_log2;
    asm("" : "+v"(scale));
    const float scale2 = fabsf(scale);
    DecState st;
    int par = 0;
    for (int si = 0; si < nseg; ++si) {
        const int npg = cur.get(si, 3), t0 = cur.get(si, 4), t1 = cur.get(si, 5);
        const int b_ = cur.get(si, 0), kvh = cur.get(si, 1), ps_ = cur.get(si, 7);
        const int tbase = t0 & ~(kPage - 1);   // first token of the segment's first page
        pf16x8 q[4];
        if constexpr (NS == 1) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) q[ks] = qn[ks];
            dec_sign_q(q, scale);
            if (si + 1 < nseg && !qpre) qload(si + 1);   // (a one-sequence plan has one segment's rows)
        }
        dec_reset(st);
        const int cnt = wcount(npg);
        for (int blk = 0; blk < cnt; blk += 2) {
            DecBlock b;
            if constexpr (NS > 1) {
                dec_wait_loads(nfl);
                dec_read_q<G>(q, S.slot[wave][sl] + kDecSlotBytes, l16, lg);
            } else {
                dec_wait_loads();
            }
            dec_read_block(b, S.slot[wave][sl], l16, lg);
            dec_wait_lds();
            if (NS > 1) dec_sign_q(q, scale);
            pf32x4 c[2][2];
            issue([&](int n) { dec_score(c, b, q, n); });
            advance();
            if (NS > 1) sl ^= 1;
            const int tok0 = tbase + (lw + WPH * blk) * kPage;
            dec_block(st, b, c, tok0, blk + 1 < cnt ? tok0 + WPH * kPage : t1, t0, t1, scale2, wc, lg, blk == 0);
            if (si == 0 && blk == 0) PD_STAMP(3);
        }
        if (si < 12) PD_STAMP(4 + 2 * si);
        dec_flush<C, LAY>(S, st, par, kargs(), (size_t)b_ * a.Hq + (size_t)kvh * G, ps_, scale2);
        par ^= 1;
        if (si < 12) PD_STAMP(5 + 2 * si);
    }
    PD_STAMP(31);
}

// The body of one balanced-decode workgroup: workgroups HP w .. HP w + HP - 1 of the plan (HP > 1:
// neighbouring kv heads of one page range). The kernel's argument block must start with the
// BalArgs `a`, which kargs() reads.
template <class C, bool UNI = false, int LAY = kLayWide, bool RANGES = false>
__device__ __forceinline__ void balanced_body(const BalArgs& a, DecShared<C, LAY>& S, int x,
                                              const UniArgs* u = nullptr) {
    static_assert(!(UNI && RANGES), "the uniform split builds its own descriptors");
    static_assert(C::HP == 1 || RANGES || UNI, "several heads share a page list");
    constexpr int G = C::G, NT = C::NT, HP = C::HP, PMAX = DecShared<C, LAY>::PGMAX / NT;
    int* pg = S.pg;
    int* sd = S.sd[0];
    const int tid = threadIdx.x, w = x * HP;
    // Segment fields are staged in LDS (sd: a header of 8 ints, then the segments) and read back
    // wave-uniform by run_segments.
    int* seg = sd + 8;
    // timestamps (timeline build only): 0 start, 1 descriptors (and page ids) staged, 2 the first
    // loads issued next, 3 the first block computed, 4 + 2 s / 5 + 2 s segment s streamed / flushed
    // (s < 12), 31 done; thread 0 of the workgroup
    PD_STAMP(0);
    pf16x8 qn[4];
    bool qpre = false;   // q rows loaded in round trip 1 (a one-sequence page-range plan)
    int nseg;
    if constexpr (!UNI) {
        // A page-range plan (RANGES: ngroups > 0) gives workgroup w = g * Hkv + kvh the pages
        // [lo, hi) of the page table (relative to kv_indptr[0]), lo = nnz g / ngroups: its page list
        // is known from the kernel arguments, so the page ids are loaded together with the
        // descriptor block(s), in round trip 1.
        uint32_t g = 0, lo = 0, npr = 0;
        if constexpr (RANGES) {
            g = div_by((uint32_t)w, (uint32_t)a.Hkv, a.rc.hkv_m);
            lo = range_start(a.rc, a.nnz, a.ngroups, g);
            npr = min(range_start(a.rc, a.nnz, a.ngroups, g + 1) - lo, (uint32_t)DecShared<C, LAY>::PGMAX);
            qpre = DecShared<C, LAY>::NS == 1 && a.qrow_b >= 0;
        }
        const int dst = a.desc_stride;   // <= kBalDescInts <= NT
        const int32_t* desc = a.desc + (size_t)w * dst;
        const int32_t* kvi = a.kv_indices + lo;
        int dv[HP], pv[PMAX];
#pragma unroll
        for (int h = 0; h < HP; ++h) dv[h] = desc[h * dst + min(tid, dst - 1)];
        if constexpr (RANGES) {
            // (NG <= nnz: every range holds a page)
            pv[0] = kvi[min((uint32_t)tid, npr - 1)];
            // a one-sequence plan: the q rows of (qrow_b, this wave's kv head) in the same trip
            // (every segment uses them)
            if (qpre) {
                const int lane = tid & 63, hh = __builtin_amdgcn_readfirstlane(tid >> 6) / C::WPH;
                const _Float16* qp = a.q + ((size_t)a.qrow_b * a.Hq + (size_t)(w - g * a.Hkv + hh) * G +
                                            (lane & 7) % G) * kHeadDim + 8 * (lane >> 4);
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) qn[ks] = *reinterpret_cast<const pf16x8*>(qp + 32 * ks);
            }
            if (npr > NT) {   // (wave-uniform)
#pragma unroll
                for (int k = 1; k < PMAX; ++k) pv[k] = kvi[min((uint32_t)(tid + k * NT), npr - 1)];
#pragma unroll
                for (int k = 1; k < PMAX; ++k) pg[tid + k * NT] = pv[k];
            }
            pg[tid] = pv[0];
        }
#pragma unroll
        for (int h = 0; h < HP; ++h)
            if (tid < dst) S.sd[h][tid] = dv[h];
        __syncthreads();
        PD_STAMP(1);
        nseg = __builtin_amdgcn_readfirstlane(sd[0]);
        // (uniform: every thread leaves) no segment, or not this plan's descriptor block(s): the
        // workspace was written over since the upload, and nothing here is to be trusted
        if (nseg <= 0 || nseg > kSegMax) return;
#pragma unroll
        for (int h = 0; h < HP; ++h)
            if (__builtin_amdgcn_readfirstlane(S.sd[h][0]) != nseg ||
                __builtin_amdgcn_readfirstlane(S.sd[h][1]) != a.tag)
                return;
    } else {
        // items x, x + W, ... (W workgroups): thread t builds the descriptors of the t-th, one per
        // head (the decode_partial rule, 01_decode_attention.cu:88-97: keys [kv_start + chunk *
        // chunk_tokens, + chunk_tokens) clipped to the sequence; an empty range writes 0 / -inf). t0
        // is the first key of the range, which need not start a page: keys are numbered from its
        // page's first token.
        nseg = min(u->per_wg, (u->n_items - x + a.W - 1) / a.W);
        if (nseg <= 0) return;   // uniform: the host sizes the grid so that every workgroup has items
        if (tid < nseg) {
            const int item = x + tid * a.W, groups = a.Hkv / HP;
            const int pair = item / u->num_chunks, chunk = item - pair * u->num_chunks;
            const int b = pair / groups, kvh = (pair - b * groups) * HP;
            const int pb = u->kv_indptr[b], np = u->kv_indptr[b + 1] - pb;
            // (a last-page length outside [1, 16] is clamped: no key past the sequence's pages)
            const int len = np > 0 ? (np - 1) * kPage + min(kPage, max(1, u->kv_last[b])) : 0;
            const int kbeg = u->kv_start + chunk * u->chunk_tokens;
            const int kend = max(kbeg, min(len, kbeg + u->chunk_tokens));
            const int pf = kbeg / kPage;
#pragma unroll
            for (int h = 0; h < HP; ++h) {
                int* sg = S.sd[h] + 8 + tid * kSegInts;
                sg[0] = b;
                sg[1] = kvh + h;
                sg[3] = kend > kbeg ? (kend - 1) / kPage - pf + 1 : 0;
                sg[4] = kbeg;
                sg[5] = kend;
                sg[6] = pb + pf;
                sg[7] = a.out != nullptr ? -1 : u->chunk_base + chunk;
            }
        }
        __syncthreads();
        // page-list offsets: exclusive prefix sum of the page counts
        if (tid < nseg) {
            int qa = 0;
            for (int j = 0; j < tid; ++j) qa += seg[j * kSegInts + 3];
#pragma unroll
            for (int h = 0; h < HP; ++h) S.sd[h][8 + tid * kSegInts + 2] = qa;
        }
        __syncthreads();
        PD_STAMP(1);
    }

    if constexpr (!RANGES) stage_pages<C, LAY>(a, S, nseg);
    run_segments<C, LAY>(a, S, nseg, qn, qpre);
}

// ---- page ranges found on the device (the drop-in decode_attention without a host plan) -----
template <class C>
struct DevShared {
    DecShared<C, kLayOne> b;
    int ip[kDevMaxB + 1];      // kv_indptr
    int piece[kDevMaxB];       // the sequences with a piece in the range, in order
    int pb[kDevMaxB];          // of those: attended pages before the sequence, its attended pages,
    int cnt[kDevMaxB];         // its length (indexed by sequence; written where they are needed)
    int len[kDevMaxB];
    int wx[2 * C::NW];         // per-wave piece counts and clip flags of the common-case guess
    int sc[C::NW];             // block-scan scratch
    int keep[4];               // the range, the end of the keys and the workgroup, for later batches
};

// Exclusive prefix sum of v over the workgroup's threads, in thread order, and the total. All
// threads call it (it holds two barriers).
template <int NW>
__device__ __forceinline__ int block_exscan(int v, int* sc, int& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) sc[wave] = x;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const int t = sc[i];
        base += i < wave ? t : 0;
        tot += t;
    }
    __syncthreads();
    total = tot;
    return base + x - v;
}

// Workgroup w = g * Hkv + kvh: range g of the attended pages, kv head kvh. Thread t handles
// sequences 4 t .. 4 t + 3 (B <= kDevMaxB). One round trip loads kv_indptr and the last-page
// lengths. In the common case (keys from 0, no sequence cut short by the span) the attended pages
// of sequence b are all its pages, their prefix sums are kv_indptr[b] - kv_indptr[0], and a range's
// page ids are contiguous in kv_indices: that case is assumed at once, its page ids are loaded
// while one barrier settles whether it holds, and its pieces run as a host page-range plan's do.
// Otherwise two block scans give the prefix sums of the attended pages and the index of each
// sequence piece in the range, and the pieces run in batches of at most kSegMax segments (a range of
// many short sequences), each batch like a host plan's workgroup (run_segments).
template <class C>
__device__ __forceinline__ void dev_body(const DevArgs& da, DevShared<C>& D, int wg) {
    constexpr int G = C::G, HP = C::HP, NW = C::NW, NT = C::NT, SEGS = kSegMax;
    constexpr int PMAX = kRangeMax / NT;
    static_assert(4 * NT >= kDevMaxB + 1, "four sequences per thread");
    const BalArgs& a = da.d;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, B = a.B, Hkv = a.Hkv;
    // (w: the slots' workgroup index of the first of this workgroup's HP kv heads)
    const int w = wg * HP, g = w / Hkv;
    const int64_t NG = a.ngroups;
    PD_STAMP(0);
    // (unconditional loads at clamped indices, B >= 1: a conditional load per element would be
    // waited for before the next is issued)
    int ipv[4], lnv[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int b = 4 * tid + k;
        ipv[k] = da.kv_indptr[min(b, B)];
        lnv[k] = da.kv_last[min(b, B - 1)];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (4 * tid + k <= B) D.ip[4 * tid + k] = ipv[k];
    __syncthreads();
    PD_STAMP(1);
    // (32-bit arithmetic from here on: page positions are int32, and a sequence's keys fit an int;
    // wave64 integer work costs four cycles an instruction, and 64-bit work twice that)
    const int ks = da.kv_start;   // >= 0
    const int ke = (int)min((int64_t)ks + da.span, (int64_t)INT_MAX);
    // The common-case guess (uniform: every thread takes the same branches on it). Its page ids
    // [ip0 + lo, ip0 + hi) lie in [ip0, kv_indptr[B]), entries of the page table whatever the
    // outcome; a range of more than kRangeMax pages (the guess being wrong) loads only the first.
    // They are loaded first, while the rest is worked out.
    const int ip0 = __builtin_amdgcn_readfirstlane(D.ip[0]);
    const int ipB = __builtin_amdgcn_readfirstlane(D.ip[B]);
    const bool guess = ks == 0 && ip0 >= 0 && ipB >= ip0;
    int N = guess ? ipB - ip0 : 0;
    int lo = (int)((int64_t)N * g / NG), hi = (int)((int64_t)N * (g + 1) / NG);
    // (branch-free loads at indices clamped into the range, or of kv_indptr[0] with no range to
    // load: the waits for the loads before them then count exactly, and none waits for these)
    int pv[PMAX];
    {
        const bool ok = guess && hi > lo;
        const int32_t* kvi = ok ? kargs()->kv_indices + ip0 + lo : da.kv_indptr;
        const int last = ok ? hi - lo - 1 : 0;
#pragma unroll
        for (int k = 0; k < PMAX; ++k) pv[k] = kvi[min(tid + k * NT, last)];
    }
    // attended pages of each sequence: keys [ks, min(len, ks + span)), from page ks / 16 (a
    // last-page length outside [1, 16] is clamped, as in the uniform split)
    const int ipn = D.ip[min(4 * tid + 4, B)];
    int cnt[4], lenv[4], pb[4], sum = 0, clipped = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int b = 4 * tid + k;
        const int np = b < B ? (k < 3 ? ipv[k + 1] : ipn) - ipv[k] : 0;
        const int len = np > 0 ? (np - 1) * kPage + min(kPage, max(1, lnv[k])) : 0;
        const int kend = min(len, ke);
        const int c = kend > ks ? (int)((uint32_t)(kend - 1) / kPage) - ks / kPage + 1 : 0;
        clipped |= c != np;
        cnt[k] = c;
        lenv[k] = len;
        pb[k] = b <= B ? ipv[k] - ip0 : N;
        sum += c;
    }
    // one barrier: the guess's per-wave piece counts and clip flags. Piece k of each thread is one
    // bit of a ballot, so the wave's exclusive prefix is four masked popcounts.
    int fl[4], nf = 0, x = 0, wn = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        fl[k] = cnt[k] > 0 && pb[k] < hi && pb[k] + cnt[k] > lo;
        nf += fl[k];
        const uint64_t m = __builtin_amdgcn_ballot_w64(fl[k] != 0);
        x += __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
        wn += __builtin_popcountll(m);
    }
    const bool wclip = __builtin_amdgcn_ballot_w64(clipped != 0) != 0;
    if (lane == 0) {
        D.wx[wave] = wn;
        D.wx[NW + wave] = wclip;
    }
    __syncthreads();
    PD_STAMP(28);
    int f0 = x, ntot = 0, anyclip = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const int t = D.wx[i];
        f0 += i < wave ? t : 0;
        ntot += t;
        anyclip |= D.wx[NW + i];
    }
    const bool fast = guess && !anyclip;
    if (!fast) {
        // prefix sums of the attended pages, then the pieces of the range
        int run = block_exscan<NW>(sum, D.sc, N);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            pb[k] = run;
            run += cnt[k];
        }
        lo = (int)((int64_t)N * g / NG);
        hi = (int)((int64_t)N * (g + 1) / NG);
        nf = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            fl[k] = cnt[k] > 0 && pb[k] < hi && pb[k] + cnt[k] > lo;
            nf += fl[k];
        }
        f0 = block_exscan<NW>(nf, D.sc, ntot);
    }
    if (wg == 0) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (4 * tid + k <= B) da.prefix[4 * tid + k] = pb[k];
    }
    if (lo == hi) {
        // an empty range (fewer pages than ranges): its slots are read as empty by the merge
        if (tid < 2 * HP * G) a.part_lse[(size_t)2 * w * G + tid] = -INFINITY;
        return;
    }
    // The piece of sequence b (attended pages [p, p + c), length len) as segment si of a batch whose
    // page list starts at attended page bs0.
    auto describe = [&](int si, int b, int p, int c, int len, int bs0, int lo, int hi, int ks, int ke, int w) {
        const int s0 = max(p, lo), s1 = min(p + c, hi), kvh = w % a.Hkv;
        const int pa0 = ks / kPage + (s0 - p), pa1 = ks / kPage + (s1 - p);
#pragma unroll
        for (int h = 0; h < HP; ++h) {
            int* sg = D.b.sd[h] + 8 + si * kSegInts;
            sg[0] = b;
            sg[1] = kvh + h;
            sg[2] = s0 - bs0;
            sg[3] = s1 - s0;
            sg[4] = max(ks, pa0 * kPage);
            sg[5] = min(min(len, ke), pa1 * kPage);
            sg[6] = D.ip[b] + pa0;
            sg[7] = (s0 == p && s1 == p + c) ? -1 : (s0 == lo && p < lo) ? 2 * (w + h) : 2 * (w + h) + 1;
        }
    };
    // Batches of at most SEGS segments. The common case is one batch, whose page list is the range's
    // pages, already loaded. The first batch is described from the registers above, the others from
    // LDS, so that none of that state stays live through the page loops.
    const bool one = fast && ntot <= SEGS;
    int nseg = min(SEGS, ntot);
    {
        int fi = f0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (!fl[k]) continue;
            const int b = 4 * tid + k, si = fi++;
            if (si < SEGS) describe(si, b, pb[k], cnt[k], lenv[k], lo, lo, hi, ks, ke, w);
            if (ntot > SEGS) {
                D.piece[si] = b;
                D.pb[b] = pb[k];
                D.cnt[b] = cnt[k];
                D.len[b] = lenv[k];
            }
        }
    }
    if (one) {
#pragma unroll
        for (int k = 0; k < PMAX; ++k)
            if (tid + k * NT < hi - lo) D.b.pg[tid + k * NT] = pv[k];
    }
    if (tid == 0) {
        D.keep[0] = lo;
        D.keep[1] = hi;
        D.keep[2] = ke;
        D.keep[3] = w;
    }
    __syncthreads();
    PD_STAMP(30);
    pf16x8 qn[4];
    for (int sb = 0;;) {
        if (!one) stage_pages<C, kLayOne>(a, D.b, nseg);
        run_segments<C, kLayOne>(a, D.b, nseg, qn);
        sb += SEGS;
        if (sb >= ntot) break;
        nseg = min(SEGS, ntot - sb);
        const int bs0 = D.pb[D.piece[sb]];   // (a later batch starts with a whole sequence or its start)
        __syncthreads();
        if (tid < nseg) {
            const int b = D.piece[sb + tid];
            describe(tid, b, D.pb[b], D.cnt[b], D.len[b], bs0, D.keep[0], D.keep[1], da.kv_start, D.keep[2],
                     D.keep[3]);
        }
        __syncthreads();
    }
}

// Merge of the sequences split over ranges: one workgroup per row (b, q head); the prefix sums
// written by the decode launch say which ranges hold sequence b's pages. A row of a sequence
// with no attended key gets 0 / -inf; a sequence within one range was written by its workgroup.
template <int U, bool WIDE>
__global__ __launch_bounds__(kMergeThreads) void merge_ranges_kernel(DevMergeArgs a) {
    const int row = merge_row<WIDE>(), d0 = merge_d0<WIDE>(), b = row / a.Hq, hq = row - b * a.Hq;
    const int kvh = hq / a.G, hh = hq - kvh * a.G;
    const int64_t pb = a.prefix[b], pe = a.prefix[b + 1], N = a.prefix[a.B];
    MSrc A{a.part_lse, a.part_o, 1, 0}, Bs = A;   // (no source: the fold leaves the empty state, out 0, lse -inf)
    if (pe > pb) {
        const int64_t NG = a.ngroups;
        const int64_t g0 = ((pb + 1) * NG - 1) / N, g1 = (pe * NG - 1) / N;
        if (g0 == g1) return;
        const size_t i0 = ((size_t)(g0 * a.Hkv + kvh) * 2 + 1) * a.G + hh;       // slot 2 w + 1 of g0
        const size_t i1 = ((size_t)((g0 + 1) * a.Hkv + kvh) * 2) * a.G + hh;     // slot 2 w of g0 + 1
        A = MSrc{a.part_lse + i0, a.part_o + i0 * kHeadDim, 1, 1};
        Bs = MSrc{a.part_lse + i1, a.part_o + i1 * kHeadDim, (size_t)2 * a.Hkv * a.G, (int)(g1 - g0)};
    }
    const MState st = merge_lanes<U>(A, Bs, d0, [](int) { return true; });
    merge_store(st, d0, a.out + (size_t)row * kHeadDim, a.lse + row);
}

// One kv head per workgroup (C::HP = 1), or HP neighbouring heads of a page-range plan: workgroup x
// runs the plan's workgroups HP x .. HP x + HP - 1.
template <class C, bool RANGES, int LAY = kLayWide>
__global__ __launch_bounds__(C::NT, 1) void decode_balanced_kernel(BalArgs a) {
    __shared__ DecShared<C, LAY> S;
    balanced_body<C, false, LAY, RANGES>(a, S, blockIdx.x);
}

// The reference-shaped uniform split on the balanced body (items of equal key ranges, descriptors
// built in the kernel from the device page table).
template <class C, int LAY>
__global__ __launch_bounds__(C::NT, 1) void decode_uniform_kernel(UniArgs u) {
    __shared__ DecShared<C, LAY> S;
    balanced_body<C, true, LAY>(u.d, S, blockIdx.x, &u);
}

// The drop-in decode_attention over page ranges found on the device.
template <class C>
__global__ __launch_bounds__(C::NT, 1) void decode_ranges_kernel(DevArgs d) {
    __shared__ DevShared<C> S;
    dev_body<C>(d, S, blockIdx.x);
}

// The fused cascade step: blocks [0, n_dec) are the suffix decode's workgroups, the rest the
// prefix pass's (item x, kv head) workgroups. Both roles are 4-wave workgroups of at most 256 VGPRs
// and half the LDS, so a CU holds one of each: the dispatcher places the first n_dec blocks
// one per CU, and the prefix blocks fill the second slots, so every CU streams suffix pages
// while its matrix core works on the prefix. Partials of both go to the workspace and are merged
// by the next launch.
template <class C, bool RANGES>
__global__ __launch_bounds__(C::NT, 2) void cascade_step_kernel(StepArgs s) {
    static_assert(C::NT == kPrefixThreads, "both roles use the same workgroup shape");
    typedef DecShared<C, kLayStep> Dec;
    constexpr size_t SB = sizeof(Dec) > sizeof(PSmem) ? sizeof(Dec) : sizeof(PSmem);
    static_assert(2 * SB <= 160 * 1024, "a CU's LDS holds two of these workgroups");
    __shared__ __align__(256) unsigned char raw[SB];
    const int i = blockIdx.x;
    if (i < s.n_dec) {
        balanced_body<C, false, kLayStep, RANGES>(s.d, *reinterpret_cast<Dec*>(raw), i);
    } else {
        const int j = i - s.n_dec, n_items = s.p.num_chunks;
        prefix_workgroup(s.p, *reinterpret_cast<PSmem*>(raw), j % n_items, 0, j / n_items);
    }
}

int occupancy_of(const void* fn, int threads) {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, threads, 0) != hipSuccess) return 1;
    return n > 0 ? n : 1;
}

// Kernel shapes per group size G.
// One-chunk-per-workgroup kernel (the uniform split's fallback for chunks past the LDS page list):
// 16 lanes per 256-byte row, 4 waves, a two-page ring. Against 8 lanes per row and 8 waves, measured
// cold when it ran every uniform split: 64x1K 57.0 vs 64.3 us, 1x32K 39.9 vs 39.8 us, 8x8K 57.2 vs 57.8 us.
template <int G>
using PartialCfg = Cfg<G, 4, 2>;
// MFMA body (plan/run, the uniform split, device ranges and the cascade's suffix): one kv head per
// 4-wave workgroup, or two neighbouring heads of a page range, two waves each.
template <int G>
using BalCfg = DecCfg<G, 1>;
template <int G>
using PairCfg = DecCfg<G, 2>;

template <class C>
void launch_p(const PartialArgs& a, hipStream_t s) {
    decode_partial_kernel<C><<<dim3(a.num_chunks, a.B * a.Hkv), C::NT, 0, s>>>(a);
}
template <class C>
void launch_b(const BalArgs& a, hipStream_t s) {
    if (a.ngroups > 0) decode_balanced_kernel<C, true><<<a.W, C::NT, 0, s>>>(a);
    else decode_balanced_kernel<C, false><<<a.W, C::NT, 0, s>>>(a);
}
template <class C>
void launch_pair(const BalArgs& a, hipStream_t s) {
    if constexpr (DecShared<C, kLayWide>::NS > 1)
        if (plan_one_slot(a.B, a.nnz, a.ngroups, C::G)) {
            decode_balanced_kernel<C, true, kLayOne><<<a.W / C::HP, C::NT, 0, s>>>(a);
            return;
        }
    decode_balanced_kernel<C, true><<<a.W / C::HP, C::NT, 0, s>>>(a);
}
template <class C>
void launch_u(const UniArgs& a, bool two_slots, hipStream_t s) {
    if constexpr (DecShared<C, kLayWide>::NS > 1)
        if (!two_slots) {
            decode_uniform_kernel<C, kLayOne><<<a.d.W, C::NT, 0, s>>>(a);
            return;
        }
    decode_uniform_kernel<C, kLayWide><<<a.d.W, C::NT, 0, s>>>(a);
}
template <class C>
void launch_step(const StepArgs& a, hipStream_t s) {
    if constexpr (C::HP == 1)
        if (a.d.ngroups <= 0) {
            cascade_step_kernel<C, false><<<a.n_dec + a.n_pre, C::NT, 0, s>>>(a);
            return;
        }
    cascade_step_kernel<C, true><<<a.n_dec + a.n_pre, C::NT, 0, s>>>(a);
}
template <class C>
void launch_r(const DevArgs& a, hipStream_t s) {
    decode_ranges_kernel<C><<<a.d.W, C::NT, 0, s>>>(a);
}
template <class C>
int occ_step() { return occupancy_of(reinterpret_cast<const void*>(&cascade_step_kernel<C, true>), C::NT); }
template <class C>
int occ_p() { return occupancy_of(reinterpret_cast<const void*>(&decode_partial_kernel<C>), C::NT); }
template <class C>
int occ_b() { return occupancy_of(reinterpret_cast<const void*>(&decode_balanced_kernel<C, true>), C::NT); }

#define PD_DISPATCH(CFG, G, FN, ...)                         \
    do {                                                     \
        if ((G) == 1) FN<CFG<1>>(__VA_ARGS__);               \
        else if ((G) == 2) FN<CFG<2>>(__VA_ARGS__);          \
        else if ((G) == 4) FN<CFG<4>>(__VA_ARGS__);          \
        else FN<CFG<8>>(__VA_ARGS__);                        \
    } while (0)

#define PD_DISPATCH_RET(CFG, G, FN)                          \
    do {                                                     \
        if ((G) == 1) return FN<CFG<1>>();                   \
        if ((G) == 2) return FN<CFG<2>>();                   \
        if ((G) == 4) return FN<CFG<4>>();                   \
        return FN<CFG<8>>();                                 \
    } while (0)

}  // namespace

hipError_t launch_decode_partial(const PartialArgs& a, int G, hipStream_t s) {
    if (G != 1 && G != 2 && G != 4 && G != 8) return hipErrorInvalidValue;
    PD_DISPATCH(PartialCfg, G, launch_p, a, s);
    return hipGetLastError();
}

// The merge kernels: `n` sources per row (the most, or about as many) choose how many a lane loads in
// one round trip, so that short lists load nothing twice and long ones take one trip, and up to 64 rows
// (one or two sequences) run on four times as many CUs. Against 32 per trip in 4-wave workgroups always: 1
// x 32768 tokens (32 rows of 64 sources) 26.8 -> 25.9 us, 64 ragged sequences at G = 8 (2944 rows of 2
// or 3 sources) 93.8 -> 92.0.
template <class F>
hipError_t launch_merge(int n, int64_t rows, F launch) {
    const bool wide = rows <= 64;
    const dim3 grid((unsigned)(wide ? 4 * rows : rows)), block(wide ? 64 : kMergeThreads);
    auto go = [&](auto u) {
        if (wide) launch(u, std::true_type{}, grid, block);
        else launch(u, std::false_type{}, grid, block);
    };
    if (n <= 8) go(std::integral_constant<int, 1>{});
    else if (n <= 16) go(std::integral_constant<int, 2>{});
    else if (n <= 24) go(std::integral_constant<int, 3>{});
    else if (n <= 32) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, 8>{});
    return hipGetLastError();
}

hipError_t launch_merge_states(const float* part_o, const float* part_lse, _Float16* out,
                               float* lse, int rows, int num_chunks, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    return launch_merge(num_chunks, rows, [&](auto u, auto wide, dim3 grid, dim3 block) {
        merge_states_kernel<decltype(u)::value, decltype(wide)::value><<<grid, block, 0, s>>>(part_o, part_lse, out,
                                                                                              lse, num_chunks);
    });
}

hipError_t launch_decode_balanced(const BalArgs& a, int G, hipStream_t s) {
    if (G != 1 && G != 2 && G != 4 && G != 8) return hipErrorInvalidValue;
    PD_DISPATCH(BalCfg, G, launch_b, a, s);
    return hipGetLastError();
}

hipError_t launch_decode_pair(const BalArgs& a, int G, hipStream_t s) {
    if (G != 1 && G != 2 && G != 4 && G != 8) return hipErrorInvalidValue;
    if (a.ngroups <= 0 || a.Hkv % 2 != 0 || a.W % 2 != 0 || a.W <= 0) return hipErrorInvalidValue;
    PD_DISPATCH(PairCfg, G, launch_pair, a, s);
    return hipGetLastError();
}

hipError_t launch_decode_uniform(const UniArgs& a, int G, int hp, hipStream_t s) {
    if (G != 1 && G != 2 && G != 4 && G != 8) return hipErrorInvalidValue;
    if (hp != 1 && (hp != 2 || a.d.Hkv % 2 != 0)) return hipErrorInvalidValue;
    if (a.d.W <= 0) return hipSuccess;
    const bool two = uniform_two_slots(a.per_wg, ((int64_t)a.chunk_tokens + kPage - 1) / kPage + 1);
    if (hp == 2) PD_DISPATCH(PairCfg, G, launch_u, a, two, s);
    else PD_DISPATCH(BalCfg, G, launch_u, a, two, s);
    return hipGetLastError();
}

hipError_t launch_cascade_step(const StepArgs& a, int G, int hp, hipStream_t s) {
    if (G != 1 && G != 2 && G != 4 && G != 8) return hipErrorInvalidValue;
    if (hp != 1 && (hp != 2 || a.d.Hkv % 2 != 0 || a.d.ngroups <= 0)) return hipErrorInvalidValue;
    if (a.n_dec + a.n_pre <= 0) return hipSuccess;
    if (hp == 2) PD_DISPATCH(PairCfg, G, launch_step, a, s);
    else PD_DISPATCH(BalCfg, G, launch_step, a, s);
    return hipGetLastError();
}

int occupancy_cascade_step(int G) { PD_DISPATCH_RET(BalCfg, G, occ_step); }

hipError_t launch_merge_split(const MergeArgs& a, int n_entries, hipStream_t s) {
    if (n_entries <= 0) return hipSuccess;
    if (a.cmax > 0)
        return launch_merge(a.cmax + a.n_extra, (int64_t)n_entries * a.G, [&](auto u, auto wide, dim3 grid, dim3 block) {
            merge_split_kernel<true, decltype(u)::value, decltype(wide)::value><<<grid, block, 0, s>>>(a);
        });
    merge_split_kernel<false, 4, false><<<n_entries * a.G, kMergeThreads, 0, s>>>(a);
    return hipGetLastError();
}

hipError_t launch_decode_ranges(const DevArgs& a, int G, int hp, hipStream_t s) {
    if (G != 1 && G != 2 && G != 4 && G != 8) return hipErrorInvalidValue;
    if (hp != 1 && (hp != 2 || a.d.Hkv % 2 != 0)) return hipErrorInvalidValue;
    if (a.d.W <= 0) return hipSuccess;
    if (hp == 2) PD_DISPATCH(PairCfg, G, launch_r, a, s);
    else PD_DISPATCH(BalCfg, G, launch_r, a, s);
    return hipGetLastError();
}

hipError_t launch_merge_ranges(const DevMergeArgs& a, hipStream_t s) {
    if (a.B <= 0) return hipSuccess;
    return launch_merge(merge_ranges_sources(a.ngroups, a.B), (int64_t)a.B * a.Hq, [&](auto u, auto wide, dim3 grid, dim3 block) {
        merge_ranges_kernel<decltype(u)::value, decltype(wide)::value><<<grid, block, 0, s>>>(a);
    });
}

int occupancy_decode_partial(int G) { PD_DISPATCH_RET(PartialCfg, G, occ_p); }
int occupancy_decode_balanced(int G) { PD_DISPATCH_RET(BalCfg, G, occ_b); }

}  // namespace pdattn
