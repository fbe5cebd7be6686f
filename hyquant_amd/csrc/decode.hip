// Fused four-segment hybrid decode attention for gfx950 (MI355X).
//
// Math (fused_d_stage_decode, src/ops/decode_d_stage.py:916-1005, split-K
// kernels :481-782): for each query head, one online softmax (log2 domain,
// scale sm_scale*log2e) over [int4 prefix | top-k | staging | window].  On the
// int4 prefix the per-token K scale is factored out of the dot product,
// s = (q . k_code) * s_k, and P is rounded to bf16 after multiplying by the
// per-token V scale, P' = bf16(p * s_v), before P' . v_code (F8).
//
// One launch per step.  A workgroup of 4 wavefronts owns one piece of one KV
// head (all G query heads of the GQA group ride along as MFMA columns); the
// grid is (KV heads, pieces per head).  A head's keys are laid end to end as
// schedule units, int4 groups of 32 tokens and then bf16 units of 8 tokens
// of each segment, and the host cuts them into `nwg` pieces, each inside one
// segment and of about equal bytes within it (make_plan); the cut points
// travel in the kernel arguments.  With many KV heads the pieces are sized
// so that the grid is about 1.25 rounds of the resident workgroup slots.  In
// a piece:
//   its int4 tokens are walked in 32-token groups (wavefront w takes groups
//     w, w+4, ...) through a three-deep register ring, so two groups' loads
//     are in flight while one is computed;
//   the tokens of each bf16 segment it reaches are walked in 16-token tiles
//     (wavefront w takes tiles w, w+4, ...) through a two-deep register ring.
// Every load goes through a buffer descriptor whose range is the piece's part
// of the segment (past the end reads zeros), so the rings' loads are
// unconditional and their wait counts exact; the loop position travels in the
// scalar offset.
//
// The four wavefronts' (m, l, acc) are merged in LDS and the workgroup writes
// one partial with device-scope stores (write-through to the device coherence
// point), waits for them, and counts itself in on its head's arrival counter.
// The workgroup that arrives last merges the head's partials (one wavefront
// per query head; see merge_head_waves) and resets the counter to zero, so the
// counters are zero again when the launch ends.  No fence is needed: the
// partials never sit dirty in a per-XCD L2, and the merge reads them with
// device-scope loads.
//
// Per wavefront, lane l = 16*kb + c (c = l & 15, kb = l >> 4):
//   PV  O^T[channel][g] = V^T . P'^T with v_mfma_f32_16x16x32_bf16:
//       A = 16 channels x 32 token slots, B = P'^T.  Slot e of lane-row kb
//       is token 4e + kb of the 32-token group, so V load e of the wavefront
//       reads four consecutive packed rows 4e..4e+3 (whole 128-byte lines).
//   QK  S^T[token][g] = K_tile . Q^T with v_mfma_f32_16x16x32_{f16,bf16}:
//       A = 16 tokens x 32 channels, B = Q^T (lane = head c).  Row i of tile
//       t is token 16t + 4(i & 3) + (i >> 2), so output lane (g = c, kb),
//       which holds rows 4kb..4kb+3, holds tokens 16t + 4i + kb: exactly the
//       P' slots 4t + i of its lane-row.  No cross-lane shuffle of P.
//   Channel 8*j+nb of V sits in row j of PV MFMA nb (lane j loads the dword /
//   16 bytes holding channels 8j..8j+7).  bf16 tiles use the K=16 form
//   (v_mfma_f32_16x16x16_bf16) whose slot e of lane-row kb is token 4kb+e.
//   Lane i of a quad loads the K and V scales of token 16t + 4i + kb of a
//   tile and quad-broadcast DPP moves hand every lane all four.
//   Loads whose instructions cover whole 128-byte lines are non-temporal:
//   the quantised prefix's packed rows and the bf16 tiles' V rows.  This
//   raised a loads-only copy of the prefix schedule from 75% to 82% of HBM
//   peak, the kernel at B=16, 32K from 66% to 81% and the bf16-only
//   comparator from 72% to 80%.  Loads that read a line in pieces from
//   several instructions (the scales, the bf16 tiles' K rows) were slower
//   non-temporal and keep the default policy.
// int4 -> MFMA operand conversion is done in registers without any lookup:
//   K: u = nibble ^ 8 placed in the mantissa of an fp16 subnormal (value
//      u * 2^-24, one shift and one bitop3 per pair of codes); Q is fed as
//      fp16, pre-scaled by a power of two so every bf16 query value is
//      exact, every product is exact in fp32, and the QK accumulators start
//      at -2^-24 * 8 * sum(q) so that they end at 2^-24 * q . code.
//   V: nibble ^ 8 -> bf16(128 + u); the constant 136 is removed after the
//      product with a ninth MFMA against an all-ones operand, which yields
//      sum_t P'[g][t] rounded exactly as the main product.
#include "hyq_common.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <mutex>
#include <string>

namespace hyq {
namespace {

constexpr int D = 128;
constexpr int WAVES = 4;                 // wavefronts per workgroup
constexpr int THREADS = 64 * WAVES;
constexpr int GROUP = 32;                // int4 tokens per wavefront iteration
constexpr int TILE = 16;                 // bf16 tokens per wavefront iteration
constexpr int BUNIT = 8;                 // bf16 tokens per schedule unit (an int4 unit is a GROUP)
constexpr float LOG2E = 1.44269504f;     // src/ops/decode_d_stage.py:17
constexpr float RESCALE_SLACK = 8.0f;    // lazy max update threshold (log2 units)
constexpr float M_INIT = -1.0e30f;
constexpr int MAX_PARTIALS = 1024;       // nwg * G bound
constexpr int MAX_NWG = 256;             // chunks per head (merge weight table)
constexpr int CNT_PAD = 32;              // arrival counters 128 bytes apart
constexpr int CNT_CAP = 16384;           // counter slots at the head of every workspace (bh_kv bound)

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// Kernel arguments.  The first PRO_DWORDS dwords are everything the
// prologue needs before its first loads; decode_kernel reads them, with its
// piece's two entries of bnd, in one batch of scalar loads (kernel_args), so
// their layout is fixed: pointers on 8-byte boundaries, the rest 32-bit (row
// and head strides fit 31 bits, checked on the host).
struct DecArgs {
    const uint16_t* q;     // dwords 0-1
    const uint8_t* kp;     // 2-3
    const uint8_t* vp;     // 4-5
    const uint16_t* ks;    // 6-7
    const uint16_t* vs;    // 8-9
    const uint16_t* sk[3]; // 10-15
    const uint16_t* sv[3]; // 16-21
    const int32_t* len_q;  // 22-23  optional per-head valid prefix tokens
    const int32_t* len_s0; // 24-25  optional per-head valid tokens of segment 0
    int32_t q_stride;      // 26
    int32_t kp_bh, vp_bh, ks_bh, vs_bh;   // 27-30
    int32_t sk_bh[3];      // 31-33
    int32_t sv_bh[3];      // 34-36
    int32_t n_quant;       // 37
    int32_t sn[3];         // 38-40
    int32_t G;             // 41
    int32_t nqg;           // 42     int4 schedule units (GROUP tokens) per head
    int32_t segu[2];       // 43-44  bf16 schedule units (BUNIT tokens) of segments 0 and 1
    float qk_scale;        // 45     sm_scale * log2(e)
    int32_t io;            // 46     HYQ_DT_* flags: fp16 q / fp16 segments / fp16 out
    int32_t pad0;          // 47
    // used once the stream is done (loaded with the prologue block, waited
    // for after the stream)
    uint16_t* out;         // 48-49
    float* part;           // 50-51  [bh_kv][nwg][G][D] partial numerators
    float* ml;             // 52-53  [bh_kv][nwg][G][2] = (m, l)
    uint32_t* cnt;         // 54-55  arrival counter of head h at cnt[h * CNT_PAD]
    int32_t out_stride;    // 56
    int32_t nwg;           // 57     pieces (workgroups) per head
    int32_t mj;            // 58     merge batch: partial columns per merging thread and load batch
    int32_t bh_kv;         // 59
    int32_t bnd[MAX_NWG + 1];  // piece p: schedule units [bnd[p], bnd[p+1]) of its head
};
constexpr int PRO_DWORDS = 48;
static_assert(offsetof(DecArgs, pad0) == 4 * (PRO_DWORDS - 1), "prologue block layout");
static_assert(offsetof(DecArgs, bh_kv) == 4 * 59, "epilogue block layout");

typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x8 __attribute__((ext_vector_type(8)));

// The prologue block of the kernel arguments and this piece's bounds
// (bnd[wg], bnd[wg + 1]) in one batch of scalar loads with one wait: left to
// the compiler, they came in two batches (two round trips) before the first
// vector load.  The epilogue block's loads are issued right after, into
// registers of their own, and waited for by epilogue_args once the stream is
// done (the compiler does not see these loads: its own lgkmcnt waits only
// over-wait for them).
struct KArgs {
    u32x16 a, b, c;
    u32x2 bnd;
    u32x8 e0;              // dwords 48-55
    u32x4 e1;              // dwords 56-59
};
__device__ __forceinline__ KArgs kernel_args(int wg) {
    const char* const base = (const char*)__builtin_amdgcn_kernarg_segment_ptr();
    const char* const bp = base + offsetof(DecArgs, bnd) + 4 * wg;
    KArgs k;
    asm volatile(
        "s_load_dwordx16 %0, %4, 0x0\n\t"
        "s_load_dwordx16 %1, %4, 0x40\n\t"
        "s_load_dwordx16 %2, %4, 0x80\n\t"
        "s_load_dwordx2 %3, %5, 0x0\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&s"(k.a), "=&s"(k.b), "=&s"(k.c), "=&s"(k.bnd)
        : "s"(base), "s"(bp)
        : "memory");
    asm volatile(
        "s_load_dwordx8 %0, %2, 0xc0\n\t"
        "s_load_dwordx4 %1, %2, 0xe0"
        : "=&s"(k.e0), "=&s"(k.e1)
        : "s"(base));
    return k;
}
__device__ __forceinline__ void epilogue_args(KArgs& k) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(k.e0), "+s"(k.e1)::"memory");
}
// dword i of the prologue block
__device__ __forceinline__ uint32_t kdw(const KArgs& k, int i) {
    return i < 16 ? k.a[i] : i < 32 ? k.b[i - 16] : k.c[i - 32];
}
template <typename T>
__device__ __forceinline__ T* kptr(const KArgs& k, int i) {
    return reinterpret_cast<T*>(static_cast<uintptr_t>(kdw(k, i)) | (static_cast<uintptr_t>(kdw(k, i + 1)) << 32));
}
template <typename T>
__device__ __forceinline__ T* eptr(const KArgs& k, int i) {
    return reinterpret_cast<T*>(static_cast<uintptr_t>(k.e0[i]) | (static_cast<uintptr_t>(k.e0[i + 1]) << 32));
}

// ---------------------------------------------------------------------------
// Phase trace (built only with -DHYQ_PHASE_TRACE, into a separate library:
// `python -m hyquant_amd.build --trace`).  Every wavefront reads
// s_memrealtime (a 100 MHz clock common to every XCD) at the phase points
// below, keeps the stamps in SGPRs and stores them once at its end, into a
// ring of the last TRACE_SLOTS launches (one record per wavefront).  The
// workgroup that finishes a launch last advances the ring.
// ---------------------------------------------------------------------------
#ifdef HYQ_PHASE_TRACE
constexpr int TRACE_SLOTS = 32;
constexpr int TRACE_MAX_WG = 4096;
constexpr int TRACE_PH = 14;
//  0 entry                       7 arrival counter returned
//  1 kernel arguments loaded
//  2 Q arrived                   8 merge: (m, l) arrived       (merging
//  3 first K/V group arrived     9 merge: partials summed       wavefronts of
//  4 own stream done            10 merge: output acked          G <= 4 heads;
//  5 all four wavefronts in LDS 11 merge: entered               else 0)
//  6 partial stored, acknowledged 12 merge: loads issued
//                               13 launch index (not a time)
__device__ uint64_t g_trace[TRACE_SLOTS][TRACE_MAX_WG * 4][TRACE_PH];
__device__ uint32_t g_trace_launch;
__device__ uint32_t g_trace_done;
// One workgroup has ended (called by one of its threads): the launch's last
// advances the ring.
__device__ __forceinline__ void trace_end() {
    const uint32_t total = gridDim.x * gridDim.y;
    if (__hip_atomic_fetch_add(&g_trace_done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == total - 1) {
        __hip_atomic_store(&g_trace_done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_fetch_add(&g_trace_launch, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}
#define HYQ_STAMP(i) (ph[i] = __builtin_amdgcn_s_memrealtime())
#define TRACE_PARAM , uint64_t (&ph)[TRACE_PH]
#define TRACE_ARG , ph
#else
#define HYQ_STAMP(i) ((void)0)
#define TRACE_PARAM
#define TRACE_ARG
#endif

struct WaveState {
    float m;               // running reference max of column g (same in the 4 lanes of g)
    float l;               // this lane's partial softmax denominator
    f32x4 acc[8];          // O^T tiles: acc[nb][i] = O[g][32*kb + 8*i + nb]
    f32x4 ones;            // sum of P' per column (int4 V offset correction)
};

__device__ __forceinline__ f32x4 mfma_f16(const f16x8& a, const f16x8& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_bf16(const bf16x8& a, const bf16x8& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_bf16_k16(const bf16x4& a, const bf16x4& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) {
    return __builtin_amdgcn_perm(hi, lo, sel);
}


// NB: operand vectors are always assembled from scalars with a brace list;
// element-wise stores into an ext_vector inside unrolled loops were
// miscompiled (every element received element 0).

// nibble pair (s, s+16) of x, offset to u = code + 8 and tagged with a magic
// exponent: ((x >> s) & 0x000f000f) ^ (0x00080008 | magic).
__device__ __forceinline__ uint32_t nib2(uint32_t x, int s, uint32_t magic_xor) {
    return ((x >> s) & 0x000f000fu) ^ magic_xor;
}

// v_exp_f32: 2^x without the denormal range fix-up of exp2f (results below
// 2^-126 flush to zero, which is harmless for softmax weights).
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Cross-lane max / sum over the 4 lanes {c, c+16, c+32, c+48} of a column,
// with the gfx950 row-swap instructions: v_permlane16_swap leaves lane l
// holding {v[l], v[l^16]} in its two results and v_permlane32_swap
// {v[l], v[l^32]}, so two VALU swaps replace two LDS-routed shuffles.
__device__ __forceinline__ float xor16_pair_max(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xor32_pair_max(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float col_max(float v) { return xor32_pair_max(xor16_pair_max(v)); }

// q.to(bf16) of an fp16 query (mask all ones) or the bf16 query unchanged
// (mask zero), without a branch: a branch here made the compiler wait for the
// Q loads at its join, before the first K/V loads were issued, which put the
// whole Q round trip in front of the K/V stream.  Called after those loads;
// the empty asm statements keep the compiler from hoisting the conversion
// (and so the wait for Q) above them.
__device__ __forceinline__ void q_to_bf16(u32x4 (&q)[4], uint32_t mask) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t w[4] = {q[i][0], q[i][1], q[i][2], q[i][3]};
        asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]));
        q[i] = u32x4{(f16x2_to_bf16x2(w[0]) & mask) | (w[0] & ~mask), (f16x2_to_bf16x2(w[1]) & mask) | (w[1] & ~mask),
                     (f16x2_to_bf16x2(w[2]) & mask) | (w[2] & ~mask), (f16x2_to_bf16x2(w[3]) & mask) | (w[3] & ~mask)};
    }
}

// One int32 through the scalar cache (a wave-uniform address written before
// the launch): a vector load there would be waited for with vmcnt(0), which
// also waits for the Q loads already in flight.
__device__ __forceinline__ int sload_i32(const int32_t* p) {
    int v;
    asm volatile("s_load_dword %0, %1, 0x0\n\ts_waitcnt lgkmcnt(0)" : "=s"(v) : "s"(p) : "memory");
    return v;
}
__device__ __forceinline__ float col_sum(float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// token slot e of lane-row kb within a 32-token group
__device__ __forceinline__ constexpr int slot_token(int kb, int e) { return 4 * e + kb; }
// token of row i of a 16-token QK tile (relative to the tile)
__device__ __forceinline__ constexpr int krow_token(int i) { return 4 * (i & 3) + (i >> 2); }

// Online-softmax update with this lane's N log2-domain scores; on return s
// holds p = exp2(s - m) relative to the (possibly raised) running max.
template <int N>
__device__ __forceinline__ void softmax_step(WaveState& st, float (&s)[N], bool has_ones) {
    // this lane's max (plain v_max3 steps), tested against the running max
    // on its own: st.m is the same on the four lanes of a column, so some
    // lane passes exactly when the column max does, and the column max (two
    // row swaps) is formed only when the running max moves
    float mx = s[0];
    int e = 1;
#pragma unroll
    for (; e + 1 < N; e += 2) mx = vmax3(mx, s[e], s[e + 1]);
    if (e < N) mx = vmax2(mx, s[e]);
    if (__builtin_amdgcn_ballot_w64(mx > st.m + RESCALE_SLACK)) {   // rare after the first group
        mx = col_max(mx);
        const float mnew = fmaxf(st.m, mx);
        const float alpha = fast_exp2(st.m - mnew);
        st.l *= alpha;
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) st.acc[nb] *= alpha;
        if (has_ones) st.ones *= alpha;
        st.m = mnew;
    }
    float lsum = 0.f;
#pragma unroll
    for (int e = 0; e < N; ++e) {
        s[e] = fast_exp2(s[e] - st.m);
        lsum += s[e];
    }
    st.l += lsum;
}

// ---------------------------------------------------------------------------
// int4 prefix
// ---------------------------------------------------------------------------
// Every load goes through a buffer descriptor whose range is the chunk, so a
// token past the chunk end reads zeros without touching memory: the loads of
// the ring are unconditional, which keeps the compiler's wait counts exact
// (a load under a branch makes every later wait a full drain).
typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr int RSRC_W3 = 0x00020000;      // raw buffer, 32-bit data format

__device__ __forceinline__ Rsrc make_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, RSRC_W3);
}
// voff: per-lane byte offset (constant across a loop), soff: wave-uniform
// byte offset (the loop position, kept in an SGPR); POL: cache policy bits
// (NT: non-temporal, for data read once)
constexpr int NT = 2;
template <int POL = 0>
__device__ __forceinline__ u32x4 bld128(Rsrc r, uint32_t voff, uint32_t soff = 0) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, POL));
}
template <int POL = 0>
__device__ __forceinline__ uint32_t bld32(Rsrc r, uint32_t voff, uint32_t soff = 0) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, POL);
}
template <int POL = 0>
__device__ __forceinline__ u32x2 bld64(Rsrc r, uint32_t voff, uint32_t soff = 0) {
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, POL));
}
template <int POL = 0>
__device__ __forceinline__ uint32_t bld16(Rsrc r, uint32_t voff, uint32_t soff = 0) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, POL);
}

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_mov(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), CTRL, 0xf, 0xf, false));
}

// Quantised prefix with KB-bit K codes and VB-bit V codes (2, 4 or 8; packed
// rows of 16*bits bytes, src/ops/decode_d_stage.py:104-133).  Per lane:
//   k[t][*]  tile t: token 16t + krow_token(c), channels 32kb..32kb+31 (KB dwords)
//   v[e][*]  slot e: token slot_token(kb, e) = 4e + kb, channels 8c..8c+7 (VB
//            bytes; 2-byte loads are zero-extended)
//   sk, sv   tile t: fp16 scale bits of token 16t + 4(c & 3) + kb
template <int KB, int VB>
struct QRaw {
    uint32_t k[2][KB];
    uint32_t v[8][VB == 8 ? 2 : 1];
    uint32_t sk[2], sv[2];
};

constexpr int prow(int bits) { return 16 * bits; }   // packed bytes per token (D = 128)
constexpr int BROW = D;                   // bf16 row stride in elements

struct QCtx {
    Rsrc k, v, ks, vs;     // this chunk's packed K / V rows and scales
    uint32_t klane;        // lane offset of tile 0: krow_token(c) * prow(KB) + 4 KB kb
    uint32_t vlane;        // lane offset of slot 0: kb * prow(VB) + VB c
    uint32_t slane;        // lane offset of the scale of tile 0: (4 (c & 3) + kb) * 2
};

// t0 is wave-uniform: it only enters the scalar offsets
template <int KB, int VB>
__device__ __forceinline__ void qload(QRaw<KB, VB>& r, const QCtx& x, int t0) {
    const uint32_t sok = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(t0) * prow(KB));
    const uint32_t sov = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(t0) * prow(VB));
    const uint32_t ss = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(t0) * 2);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const uint32_t ko = x.klane + t * 16 * prow(KB);
        if constexpr (KB == 2) {
            const u32x2 w = bld64<NT>(x.k, ko, sok);
            r.k[t][0] = w[0]; r.k[t][1] = w[1];
        } else {
#pragma unroll
            for (int h = 0; h < KB / 4; ++h) {
                const u32x4 w = bld128<NT>(x.k, ko + 16 * h, sok);
                r.k[t][4 * h] = w[0]; r.k[t][4 * h + 1] = w[1]; r.k[t][4 * h + 2] = w[2]; r.k[t][4 * h + 3] = w[3];
            }
        }
    }
    // scales (in the order qcompute uses them: after the K tiles, before the
    // V rows): a 128-byte line of them is read by several instructions, so
    // they keep the default cache policy
    r.sk[0] = bld16(x.ks, x.slane, ss);
    r.sk[1] = bld16(x.ks, x.slane + 32, ss);
    r.sv[0] = bld16(x.vs, x.slane, ss);
    r.sv[1] = bld16(x.vs, x.slane + 32, ss);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const uint32_t vo = x.vlane + slot_token(0, e) * prow(VB);
        if constexpr (VB == 2) {
            r.v[e][0] = bld16<NT>(x.v, vo, sov);
        } else if constexpr (VB == 4) {
            r.v[e][0] = bld32<NT>(x.v, vo, sov);
        } else {
            const u32x2 w = bld64<NT>(x.v, vo, sov);
            r.v[e][0] = w[0]; r.v[e][1] = w[1];
        }
    }
}

// QK A operand of MFMA m (channels 32kb + 8m + [0..7]) in slot order
// [c0,c4,c1,c5,c2,c6,c3,c7], the order of the Q operands, as fp16
// subnormals whose bits are the offset-binary code u = code + 2^(KB-1):
// the value is u * 2^-24 exactly, so every product with the fp16 query is
// exact in fp32 and the MFMA yields 2^-24 (q . code + 2^(KB-1) sum(q)).  The
// second term is the same for every token of a query column: the QK
// accumulators start at minus that bias (kbias, one MFMA product per piece),
// which leaves 2^-24 q . code.
//   4 bits: (nibble ^ 8) pairs (s, s + 16) of one dword
//   8 bits: byte j of the two dwords paired by one perm, ^ 0x80
//   2 bits: the two bytes of the 16-bit half spread to the two fp16 halves by
//           one perm, crumbs ^ 2
template <int KB>
__device__ __forceinline__ f16x8 k_operand(const uint32_t (&k)[KB], int m) {
    if constexpr (KB == 4) {
        const uint32_t x = k[m];
        const u32x4 o = {nib2(x, 0, 0x00080008u), nib2(x, 4, 0x00080008u), nib2(x, 8, 0x00080008u),
                         nib2(x, 12, 0x00080008u)};
        return __builtin_bit_cast(f16x8, o);
    } else if constexpr (KB == 8) {
        const uint32_t lo = k[2 * m], hi = k[2 * m + 1];
        const u32x4 o = {perm(hi, lo, 0x0c040c00u) ^ 0x00800080u, perm(hi, lo, 0x0c050c01u) ^ 0x00800080u,
                         perm(hi, lo, 0x0c060c02u) ^ 0x00800080u, perm(hi, lo, 0x0c070c03u) ^ 0x00800080u};
        return __builtin_bit_cast(f16x8, o);
    } else {
        const uint32_t w = k[m >> 1];
        const uint32_t y = (m & 1) ? perm(w, w, 0x0c030c02u) : perm(w, w, 0x0c010c00u);
        const u32x4 o = {((y >> 0) & 0x00030003u) ^ 0x00020002u, ((y >> 2) & 0x00030003u) ^ 0x00020002u,
                         ((y >> 4) & 0x00030003u) ^ 0x00020002u, ((y >> 6) & 0x00030003u) ^ 0x00020002u};
        return __builtin_bit_cast(f16x8, o);
    }
}

// Minus the K operand's offset term of each query column, -2^-24 2^(KB-1)
// sum_d q_d, as the MFMA forms it: the product of an all-offset K tile (every
// slot the subnormal 2^(KB-1) * 2^-24) with the Q operands.  Lane (c, kb)
// gets column c in all four entries.
template <int KB>
__device__ __forceinline__ f32x4 k_bias(const f16x8 (&qop)[4]) {
    constexpr uint32_t half = 1u << (KB - 1);
    const u32x4 w = {half | half << 16, half | half << 16, half | half << 16, half | half << 16};
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < 4; ++m) acc = mfma_f16(__builtin_bit_cast(f16x8, w), qop[m], acc);
    return -acc;
}

// The constant the PV operands add to every V code (removed at the end with
// the all-ones product): bf16(128 + u) operands, u = code + 8 (4 bits),
// code + 2 (2 bits); 8-bit codes are split into their nibbles,
// bf16(128 + lo) + bf16(16 (128 + (hi ^ 8))) = code + 2304.
template <int VB>
constexpr float v_offset() { return VB == 4 ? 136.0f : VB == 2 ? 130.0f : 2304.0f; }

// x of lane i of this lane's quad (a DPP quad broadcast, which the compiler
// folds into the VOP2 instruction that consumes it)
template <int I>
__device__ __forceinline__ float quad_bcast(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), I * 0x55, 0xf, 0xf, true));
}

template <int KB, int VB>
__device__ __forceinline__ void qcompute(WaveState& st, const QRaw<KB, VB>& r, const f16x8 (&qop)[4],
                                         const f32x4& kbias, int nv, int lane, float qk) {
    const int kb = lane >> 4;
    // each lane converts the scales of its own token of each tile (lane i of
    // a quad holds token 16t + 4i + kb, the token of score slot 4t + i); the
    // scores and P' take them with quad broadcasts
    const float skq[2] = {f16_bits_to_f32(static_cast<uint16_t>(r.sk[0])) * qk,
                          f16_bits_to_f32(static_cast<uint16_t>(r.sk[1])) * qk};
    const float svo[2] = {f16_bits_to_f32(static_cast<uint16_t>(r.sv[0])),
                          f16_bits_to_f32(static_cast<uint16_t>(r.sv[1]))};
    // QK: S^T tile = K_tile . Q^T (exact fp16 codes x fp16 q)
    float s[8];
#pragma unroll
    for (int tile = 0; tile < 2; ++tile) {
        f32x4 acc = kbias;
#pragma unroll
        for (int m = 0; m < 4; ++m) acc = mfma_f16(k_operand<KB>(r.k[tile], m), qop[m], acc);
        s[4 * tile + 0] = acc[0] * quad_bcast<0>(skq[tile]);
        s[4 * tile + 1] = acc[1] * quad_bcast<1>(skq[tile]);
        s[4 * tile + 2] = acc[2] * quad_bcast<2>(skq[tile]);
        s[4 * tile + 3] = acc[3] * quad_bcast<3>(skq[tile]);
    }
    if (nv < GROUP) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (slot_token(kb, e) >= nv) s[e] = -INFINITY;
    }
    softmax_step<8>(st, s, true);
    // P' = bf16(p * s_v): B operand of the PV MFMAs (slot e = token slot_token(kb, e))
    const u32x4 pw = {pack_bf16x2(s[0] * quad_bcast<0>(svo[0]), s[1] * quad_bcast<1>(svo[0])),
                      pack_bf16x2(s[2] * quad_bcast<2>(svo[0]), s[3] * quad_bcast<3>(svo[0])),
                      pack_bf16x2(s[4] * quad_bcast<0>(svo[1]), s[5] * quad_bcast<1>(svo[1])),
                      pack_bf16x2(s[6] * quad_bcast<2>(svo[1]), s[7] * quad_bcast<3>(svo[1]))};
    const bf16x8 pop = __builtin_bit_cast(bf16x8, pw);
    // V^T operands (A of PV MFMA nb: channel 8c + nb of the 8 token slots),
    // token pairs (2pr, 2pr + 1) merged into one dword per operand register
    if constexpr (VB == 4) {
        // bf16(128 + u) = code + 136
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int pr = 0; pr < 4; ++pr) {
            lo[pr] = perm(r.v[2 * pr + 1][0], r.v[2 * pr][0], 0x05040100u);  // nibbles 0-3 of both tokens
            hi[pr] = perm(r.v[2 * pr + 1][0], r.v[2 * pr][0], 0x07060302u);  // nibbles 4-7
        }
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) {
            const uint32_t* src = nb < 4 ? lo : hi;
            const int sh = 4 * (nb & 3);
            const u32x4 w = {nib2(src[0], sh, 0x43084308u), nib2(src[1], sh, 0x43084308u),
                             nib2(src[2], sh, 0x43084308u), nib2(src[3], sh, 0x43084308u)};
            st.acc[nb] = mfma_bf16(__builtin_bit_cast(bf16x8, w), pop, st.acc[nb]);
        }
    } else if constexpr (VB == 2) {
        // bf16(128 + (crumb ^ 2)) = code + 130
        uint32_t x[4];
#pragma unroll
        for (int pr = 0; pr < 4; ++pr) x[pr] = perm(r.v[2 * pr + 1][0], r.v[2 * pr][0], 0x05040100u);
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) {
            const int sh = 2 * nb;
            const u32x4 w = {((x[0] >> sh) & 0x00030003u) ^ 0x43024302u, ((x[1] >> sh) & 0x00030003u) ^ 0x43024302u,
                             ((x[2] >> sh) & 0x00030003u) ^ 0x43024302u, ((x[3] >> sh) & 0x00030003u) ^ 0x43024302u};
            st.acc[nb] = mfma_bf16(__builtin_bit_cast(bf16x8, w), pop, st.acc[nb]);
        }
    } else {
        // code = 16 hi + lo (hi signed, lo unsigned): two products per channel
        // into one accumulator, bf16(128 + lo) and bf16(16 (128 + (hi ^ 8)))
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) {
            const int dw = nb >> 2;
            const uint32_t sel = 0x0c040c00u + 0x00010001u * (nb & 3);
            uint32_t x[4];
#pragma unroll
            for (int pr = 0; pr < 4; ++pr) x[pr] = perm(r.v[2 * pr + 1][dw], r.v[2 * pr][dw], sel);
            const u32x4 wl = {(x[0] & 0x000f000fu) | 0x43004300u, (x[1] & 0x000f000fu) | 0x43004300u,
                              (x[2] & 0x000f000fu) | 0x43004300u, (x[3] & 0x000f000fu) | 0x43004300u};
            const u32x4 wh = {nib2(x[0], 4, 0x45084508u), nib2(x[1], 4, 0x45084508u),
                              nib2(x[2], 4, 0x45084508u), nib2(x[3], 4, 0x45084508u)};
            st.acc[nb] = mfma_bf16(__builtin_bit_cast(bf16x8, wl), pop, st.acc[nb]);
            st.acc[nb] = mfma_bf16(__builtin_bit_cast(bf16x8, wh), pop, st.acc[nb]);
        }
    }
    const u32x4 onesw = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
    st.ones = mfma_bf16(__builtin_bit_cast(bf16x8, onesw), pop, st.ones);
}

// ---------------------------------------------------------------------------
// bf16 segments: 16-token tiles
// ---------------------------------------------------------------------------
struct Bf16Raw {
    u32x4 k[4];            // token c, channels 32kb..32kb+31
    u32x4 v[4];            // slot e: token 4kb+e, channels 8c..8c+7
};

__device__ __forceinline__ void f16_to_bf16(Bf16Raw& r) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            r.k[i][j] = f16x2_to_bf16x2(r.k[i][j]);
            r.v[i][j] = f16x2_to_bf16x2(r.v[i][j]);
        }
}

// rk / rv cover this chunk's rows; tokens past the chunk read zeros
__device__ __forceinline__ void bf16_load(Bf16Raw& r, Rsrc rk, Rsrc rv, int t0, int lane) {
    const int c = lane & 15, kb = lane >> 4;
    const uint32_t so = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(t0) * (BROW * 2));
    const uint32_t ko = static_cast<uint32_t>(c) * (BROW * 2) + 64 * kb;
    const uint32_t vo = static_cast<uint32_t>(4 * kb) * (BROW * 2) + 16 * c;
#pragma unroll
    for (int i = 0; i < 4; ++i) r.k[i] = bld128(rk, ko + 16 * i, so);
#pragma unroll
    for (int e = 0; e < 4; ++e) r.v[e] = bld128<NT>(rv, vo + e * (BROW * 2), so);
}

__device__ __forceinline__ void bf16_compute(WaveState& st, const Bf16Raw& r, const bf16x8 (&qop)[4], int nv,
                                             int lane, float qk) {
    const int kb = lane >> 4;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = mfma_bf16(__builtin_bit_cast(bf16x8, r.k[i]), qop[i], acc);
    float s[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = (4 * kb + i < nv) ? acc[i] * qk : -INFINITY;
    softmax_step<4>(st, s, false);
    const u32x2 pw = {pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
    const bf16x4 pop = __builtin_bit_cast(bf16x4, pw);
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) {
        const uint32_t sel = (nb & 1) ? 0x07060302u : 0x05040100u;
        const int dw = nb >> 1;
        const u32x2 w = {perm(r.v[1][dw], r.v[0][dw], sel), perm(r.v[3][dw], r.v[2][dw], sel)};
        st.acc[nb] = mfma_bf16_k16(__builtin_bit_cast(bf16x4, w), pop, st.acc[nb]);
    }
}

// ---------------------------------------------------------------------------
// merge of a head's partials by its last workgroup
// ---------------------------------------------------------------------------
__device__ __forceinline__ u32x2 ld2_dev(Rsrc r, uint32_t off) {
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 16));    // sc1: device scope
}
__device__ __forceinline__ f32x4 ld4_dev(Rsrc r, uint32_t off) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 16));
}

template <int CTRL>
__device__ __forceinline__ float dppf(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
// full-wavefront max / sum: DPP within each row of 16 (quad swaps, half-row
// and row mirrors), then the gfx950 row swaps across rows
__device__ __forceinline__ float wave_max64(float v) {
    v = fmaxf(v, dppf<0xb1>(v));
    v = fmaxf(v, dppf<0x4e>(v));
    v = fmaxf(v, dppf<0x141>(v));
    v = fmaxf(v, dppf<0x140>(v));
    return col_max(v);
}
__device__ __forceinline__ float wave_sum64(float v) {
    v += dppf<0xb1>(v);
    v += dppf<0x4e>(v);
    v += dppf<0x141>(v);
    v += dppf<0x140>(v);
    return col_sum(v);
}

// The merge of a head's partials, by all THREADS threads of its last
// workgroup.  The partials of query head g are rows of D floats, so the head
// has NC = 32 G float4 columns.  For G <= 8 thread t owns column t % NC of
// the partials s, s + TPC, ... (s = t / NC, TPC = THREADS / NC threads per
// column); for G > 8 it owns columns t and t + THREADS of every partial.  A
// thread's items alternate between two accumulators: item e goes to acc[e & 1]
// (its two columns for G > 8, the even and odd partials of its column
// otherwise).
//   1. every (m, l) pair of the head is loaded (two float4 per thread), then
//      the thread's first MJ items, all before any wait: the weights are
//      built while the partial loads are in flight;
//   2. (m, l) go to LDS; wavefront w takes query heads w, w + 4, ...: lane p
//      holds partial p (p + 64, ...), the wavefront max / sum give M_g and
//      den_g = sum_p exp2(m_p - M_g) l_p, and the weight exp2(m_p - M_g)
//      replaces m_p in LDS;
//   3. each thread sums weight * partial over its items in order (further
//      batches of MJ loads when it owns more), the TPC threads of a column
//      add their sums in subset order through LDS, and the column is divided
//      by den_g and stored.
// Items past a thread's share load from an offset outside the buffer range
// (zeros) and take their weight from an LDS slot holding zero, so the loops
// have no branches.  The summation order depends on nothing but (G, nwg):
// every call gives the same result.
struct MergeArgs {
    int G, nwg;
    int64_t first;         // slot of the head's first partial
    const float* part;
    const float* ml;
    uint16_t* out;
    int64_t out_stride;
    int out16;             // store fp16 instead of bf16
};

constexpr int ML_LDS = 2 * MAX_PARTIALS;               // (m, l) per partial; the weights overwrite m
constexpr int ZERO_SLOT = ML_LDS + 16;                  // holds 0.0f (weight of an empty item)
constexpr int COMB_LDS = ML_LDS + 32;                   // one float4 per thread (column sums)
constexpr int MERGE_LDS = COMB_LDS + 4 * THREADS;
constexpr uint32_t OUT_OF_RANGE = 0xfffffff0u;          // a buffer offset past every range: reads zero

// Column q (channels 4q..4q+3) of query head g: acc / den rounded once to
// the output dtype (out.to(q.dtype) of the fp32 result), 0 when den == 0.
__device__ __forceinline__ void store_out(const MergeArgs& a, int head, int g, int q, const f32x4& acc, float den) {
    float r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = den > 0.f ? acc[i] / den : 0.f;
    const u32x2 o = a.out16 ? u32x2{static_cast<uint32_t>(f32_to_f16_bits(r[0])) |
                                        (static_cast<uint32_t>(f32_to_f16_bits(r[1])) << 16),
                                    static_cast<uint32_t>(f32_to_f16_bits(r[2])) |
                                        (static_cast<uint32_t>(f32_to_f16_bits(r[3])) << 16)}
                            : u32x2{static_cast<uint32_t>(f32_to_bf16_rne(r[0])) |
                                        (static_cast<uint32_t>(f32_to_bf16_rne(r[1])) << 16),
                                    static_cast<uint32_t>(f32_to_bf16_rne(r[2])) |
                                        (static_cast<uint32_t>(f32_to_bf16_rne(r[3])) << 16)};
    *reinterpret_cast<u32x2*>(a.out + static_cast<int64_t>(head * a.G + g) * a.out_stride + 4 * q) = o;
}

// G <= 4: one wavefront per query head g, no workgroup barrier.  Lane
// (h, q) = (lane >> 5, lane & 31) sums channels 4q..4q+3 of g over the
// partials 2j + h; lane p holds (m, l) of partial p (p + 64, ...).  The (m, l)
// loads go first, then the first MJ partial loads (MJ >= half the partials
// when the host can pick it), so the weights are built while the partials
// are in flight; they reach the lanes through a per-wavefront LDS table
// (same-address reads broadcast), whose entries past nwg hold zero, and a
// row swap adds the two halves.
template <int MJ>
__device__ __forceinline__ void merge_head_waves(const MergeArgs& a, int head, float* lds TRACE_PARAM) {
    const int G = a.G, P = a.nwg;
    const int lane = threadIdx.x & 63;
    const int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (g >= G) return;
    HYQ_STAMP(11);
    const int h = lane >> 5, q = lane & 31;
    const int npair = P * G;
    const Rsrc rp = make_rsrc(a.part + a.first * G * D, static_cast<uint32_t>(npair) * D * 4);
    const Rsrc rm = make_rsrc(a.ml + a.first * G * 2, static_cast<uint32_t>(npair) * 8);
    float* wt = lds + g * MAX_NWG;
    // (m, l) of partials lane, lane + 64, ... (past nwg: out of range, zeros);
    // the host's choice of MJ covers every partial in one batch when nwg <=
    // 48, so only the blocks of 64 that 2 MJ partials reach are loaded (a load
    // past the range still takes the CU's address path, which bounds the merge)
    constexpr int NML = MJ < 24 ? (2 * MJ + 63) / 64 : MAX_NWG / 64;
    u32x2 mlr[NML];
#pragma unroll
    for (int k = 0; k < NML; ++k) mlr[k] = ld2_dev(rm, static_cast<uint32_t>(((lane + 64 * k) * G + g) * 8));
    const uint32_t pbase = static_cast<uint32_t>(((h * G + g) * D + 4 * q) * 4);
    const uint32_t pstep = static_cast<uint32_t>(2 * G * D * 4);
    f32x4 px[MJ];
#pragma unroll
    for (int j = 0; j < MJ; ++j) px[j] = ld4_dev(rp, pbase + j * pstep);
    HYQ_STAMP(12);
    float M = M_INIT;
#pragma unroll
    for (int k = 0; k < NML; ++k)
        if (lane + 64 * k < P) M = fmaxf(M, __uint_as_float(mlr[k][0]));
    M = wave_max64(M);
    HYQ_STAMP(8);
    float den = 0.f;
#pragma unroll
    for (int k = 0; k < NML; ++k) {
        const bool ok = lane + 64 * k < P;
        const float w = ok ? fast_exp2(__uint_as_float(mlr[k][0]) - M) : 0.f;
        den += ok ? w * __uint_as_float(mlr[k][1]) : 0.f;
        wt[lane + 64 * k] = w;
    }
#pragma unroll
    for (int k = NML; k < MAX_NWG / 64; ++k) wt[lane + 64 * k] = 0.f;
    den = wave_sum64(den);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    static_assert(2 * MJ <= MAX_NWG, "a batch lies inside the weight table");
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc += wt[2 * j + h] * px[j];
    const int npr = (P + 1) / 2;                          // partial pairs
    for (int j0 = MJ; j0 < npr; j0 += MJ) {              // more than MJ pairs: one round trip per batch
#pragma unroll
        for (int j = 0; j < MJ; ++j) px[j] = ld4_dev(rp, pbase + (j0 + j) * pstep);
#pragma unroll
        for (int j = 0; j < MJ; ++j)
            if (2 * (j0 + j) + h < P) acc += wt[2 * (j0 + j) + h] * px[j];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i]), __float_as_uint(acc[i]), false, false);
        acc[i] = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    HYQ_STAMP(9);
    if (h == 0) store_out(a, head, g, q, acc, den);
#ifdef HYQ_PHASE_TRACE
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    HYQ_STAMP(10);
#endif
}

// MJ: items loaded per thread per batch (even; the host picks the smallest
// instance that covers a thread's items, merge_batch)
template <int MJ>
__device__ __forceinline__ void merge_head_cols(const MergeArgs& a, int head, float* lds) {
    static_assert(MJ % 2 == 0, "items come in (even, odd) pairs");
    const int G = a.G, P = a.nwg;
    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int npair = P * G;
    const Rsrc rp = make_rsrc(a.part + a.first * G * D, static_cast<uint32_t>(npair) * D * 4);
    const Rsrc rm = make_rsrc(a.ml + a.first * G * 2, static_cast<uint32_t>(npair) * 8);
    const int NC = G * (D / 4);
    const bool two = NC > THREADS;                       // G > 8
    const int TPC = two ? 1 : THREADS / NC;
    const int s = two ? 0 : t / NC;                      // partial subset (s >= TPC: idle thread)
    const int col0 = two ? t : t - s * NC;
    // item e = 2k + b: partial pb[b] + pstep * k, column col[b]
    const int pstep = two ? 1 : 2 * TPC;
    int pb[2], vb[2], wb[2];
    bool ok[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        pb[b] = two ? 0 : s + TPC * b;
        const int col = two ? col0 + THREADS * b : col0;
        ok[b] = col < NC && s < TPC;
        vb[b] = (pb[b] * G * D + 4 * col) * 4;           // byte offset in the head's partials
        wb[b] = (pb[b] * G + (col >> 5)) * 2;            // LDS index of the weight
    }
    const int vstep = pstep * G * D * 4, wstep = pstep * G * 2;
    auto voff = [&](int e) -> uint32_t {
        const int b = e & 1, k = e >> 1;
        return ok[b] && pb[b] + pstep * k < P ? static_cast<uint32_t>(vb[b] + k * vstep) : OUT_OF_RANGE;
    };
    auto widx = [&](int e) -> int {
        const int b = e & 1, k = e >> 1;
        return ok[b] && pb[b] + pstep * k < P ? wb[b] + k * wstep : ZERO_SLOT;
    };
    // 1. (m, l) table, then the first batch of items
    static_assert(2 * MAX_PARTIALS <= 2 * 4 * THREADS, "two float4 (m, l) loads per thread cover the table");
    f32x4 mlv[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) mlv[k] = ld4_dev(rm, static_cast<uint32_t>((t + THREADS * k) * 16));
    f32x4 px[MJ];
#pragma unroll
    for (int j = 0; j < MJ; ++j) px[j] = ld4_dev(rp, voff(j));
    // 2. weights
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int u = t + THREADS * k;                   // float4 unit: pairs 2u, 2u + 1
        if (4 * u < 2 * npair) *reinterpret_cast<f32x4*>(lds + 4 * u) = mlv[k];
    }
    if (t == 0) lds[ZERO_SLOT] = 0.f;
    __syncthreads();
    // one 16-lane row per query head (heads 4 w .. 4 w + 3 on wavefront w,
    // then 16 more per pass), lane j of the row taking partials j, j + 16, ...:
    // every head's max and denominator at once, by 16-lane DPP reductions
    const int seg = lane >> 4, jl = lane & 15;
    for (int g0 = 4 * wave; g0 < G; g0 += 4 * WAVES) {
        const int g = g0 + seg;
        const bool gv = g < G;
        float M = M_INIT;
        if (gv)
            for (int p = jl; p < P; p += 16) M = fmaxf(M, lds[(p * G + g) * 2]);
        M = max16_dpp(M);
        float den = 0.f;
        if (gv)
            for (int p = jl; p < P; p += 16) {
                const float w = fast_exp2(lds[(p * G + g) * 2] - M);
                den += w * lds[(p * G + g) * 2 + 1];
                lds[(p * G + g) * 2] = w;
            }
        den = sum16_dpp(den);
        if (gv && jl == 0) lds[ML_LDS + g] = den;
    }
    __syncthreads();
    // 3. weighted sums in item order
    f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[j & 1] += lds[widx(j)] * px[j];
    const int nitems = s < TPC ? (two ? 2 * P : (P - s + TPC - 1) / TPC) : 0;
    for (int j0 = MJ; j0 < nitems; j0 += MJ) {           // a thread with more than MJ items
#pragma unroll
        for (int j = 0; j < MJ; ++j) px[j] = ld4_dev(rp, voff(j0 + j));
#pragma unroll
        for (int j = 0; j < MJ; ++j) acc[j & 1] += lds[widx(j0 + j)] * px[j];
    }
    if (!two) acc[0] += acc[1];
    f32x4* comb = reinterpret_cast<f32x4*>(lds + COMB_LDS);
    if (TPC > 1) {
        if (s >= 1 && s < TPC) comb[t] = acc[0];
        __syncthreads();
        if (s == 0)
            for (int k = 1; k < TPC; ++k) acc[0] += comb[t + k * NC];
    }
    if (s == 0) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int col = col0 + THREADS * b;
            if ((b == 0 || two) && col < NC) {
                store_out(a, head, col >> 5, col & 31, acc[b], lds[ML_LDS + (col >> 5)]);
            }
        }
    }
}

// Largest number of items one merging thread loads (the host's choice of
// the MJ instance).
constexpr int merge_items(int G, int nwg) {
    return 32 * G > THREADS ? 2 * nwg : (nwg + THREADS / (32 * G) - 1) / (THREADS / (32 * G));
}

// The merge instance: for G <= 4 merge_head_waves with the smallest batch
// covering a lane's partial pairs (else batches of 24); for G > 4
// merge_head_cols (100 + batch) with the smallest batch covering a thread's
// items (else batches of 24).
__host__ __device__ inline int merge_batch(int G, int nwg) {
    if (G <= WAVES) {
        const int pairs = (nwg + 1) / 2;
        return pairs <= 24 ? (pairs + 3) / 4 * 4 : 24;
    }
    const int items = merge_items(G, nwg);
    return items <= 8 ? 108 : items <= 16 ? 116 : 124;
}

// ---------------------------------------------------------------------------
// ragged lengths: the pieces planned on the device
// ---------------------------------------------------------------------------
// With per-head lengths only the device knows how much there is to read.  The
// padded plan, cut by the longest head, leaves short heads' pieces empty and
// the long ones' as large as a full batch's.  So every workgroup of a large
// ragged launch reads all lengths.  Where they fill RAGGED_FILL of the padded
// bytes or more, it takes its piece of the padded plan; else it forms piece
// sizes from the bytes that are there, numbers the pieces (int4 pieces of all
// heads, then bf16 pieces) by a prefix sum and takes the piece of its own
// number; workgroups past the last piece leave.  Piece size, with `cus` and
// `slots` as in make_plan: 4/5 of a piece per CU below 48 MB, 5/4 per resident
// slot above (of at least 96 KiB), at least 16 KiB, and large enough for the
// merge tables and, with G > 4, for the merge to load a head's partials in one
// or two batches.  The grid covers any lengths (ragged_grid).
//
// Both plans over 570 calls of up to 256 heads (32/8, 64/8 and 32/2 heads;
// K4V4, K4V2 and K8V8; batches 2-32, longest 2.5K-30K tokens; evenly spread,
// log-spread, one long among short, nearly equal lengths), device / padded:
//   - reading the lengths and planning costs 0.7-1.1 us of a launch whatever it
//     then takes: 4-5% of calls of 60-130 MB of padded bytes that keep the
//     padded plan, 2-4% from 130 MB on, 1% from 240 MB on, 5-15% of a 7-14 us
//     call;
//   - filled to less than 60% the device's pieces are the faster ones from 90
//     MB on: 0.66-0.86 times the padded plan's time (mean 0.77) at less than a
//     quarter, 0.82 to 40%, 0.94 to 50%, 0.99 to 60% at 90-130 MB, where the
//     two lines lie; 0.55, 0.68, 0.78 and 0.89 from 240 MB on (16 sequences
//     of 600 to 32000 tokens 63.3 -> 37.8 us; 16 on two key heads, 154 MB,
//     29.8 -> 22; 4 at G = 8, 154 MB, 27.2 -> 20);
//   - at 60-80% and above they gain nothing (0.86-1.12 times), hence the fill;
//   - at 20-60 MB the coarser pieces and the cost outweigh the balance (1.07
//     and 1.0 times on average, to 1.27).
// More than four heads per lane would take registers from every ragged launch
// (sixteen: 10-25% slower), so more than 256 heads keep the padded plan.
constexpr int RAGGED_HEADS = 256;        // four per lane
constexpr float RAGGED_FILL = 0.6f;
constexpr int64_t RAGGED_BYTES = 100000000;

// pieces a ragged launch can have: total / target, and one rounded up per
// head and segment
__host__ __device__ inline int ragged_grid(int bh, int cus, int slots) {
    const int a = cus * 4 / 5, b = slots * 5 / 4;
    return (a > b ? a : b) + 1 + 2 * bh;
}

struct RaggedPiece {
    int head, piece, pieces;   // head -1: no piece of this number
    int first;                 // slot of the head's first partial
    int u0, u1, nqg, nb;       // schedule units: the piece's, and the head's int4 and bf16 units
    int nq, ns;                // the head's valid prefix and bf16 tokens
};

// inclusive prefix sum over the wavefront (rows of 16, then across rows)
__device__ __forceinline__ uint32_t wave_scan64(uint32_t v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
    return v;
}

// Every wavefront for itself: no barrier, no LDS.  Lane l holds heads 4l ..
// 4l + 3; all its loads are issued before any is waited for (heads past bh
// read zero).  `p` comes in as the padded plan's piece.
template <int KB, int VB>
__device__ __forceinline__ void ragged_piece(RaggedPiece& p, int bh, int G, int nquant, int sn0, const int32_t* len_q,
                                             const int32_t* len_s0, int cus, int slots) {
    constexpr int CQ = GROUP * (16 * KB + 16 * VB + 4), CB = BUNIT * 4 * D;   // bytes per unit
    const int lane = threadIdx.x & 63;
    int lq[4], ls[4];
    {
        const uint32_t bytes = static_cast<uint32_t>(bh) * 4;
        const Rsrc rq = make_rsrc(len_q, len_q ? bytes : 0u), rs = make_rsrc(len_s0, len_s0 ? bytes : 0u);
        uint32_t a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[i] = bld32(rq, 16 * lane + 4 * i);
            b[i] = bld32(rs, 16 * lane + 4 * i);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool in = 4 * lane + i < bh;
            lq[i] = len_q ? min(nquant, max(0, static_cast<int>(a[i]))) : in ? nquant : 0;
            ls[i] = len_s0 ? min(sn0, max(0, static_cast<int>(b[i]))) : in ? sn0 : 0;
        }
    }
    uint32_t nq[4], nb[4];
    float sum = 0.f, mx = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        nq[i] = static_cast<uint32_t>(lq[i] + GROUP - 1) / GROUP;
        nb[i] = static_cast<uint32_t>(ls[i] + BUNIT - 1) / BUNIT;
        const float bytes = static_cast<float>(nq[i]) * CQ + static_cast<float>(nb[i]) * CB;
        sum += bytes;
        mx = fmaxf(mx, bytes);
    }
    const float total = wave_sum64(sum);
    // the valid tokens of head h
    auto tokens = [&](int h) {
        const int i = h & 3, l = h >> 2;
        p.nq = __builtin_amdgcn_readlane(i == 0 ? lq[0] : i == 1 ? lq[1] : i == 2 ? lq[2] : lq[3], l);
        p.ns = __builtin_amdgcn_readlane(i == 0 ? ls[0] : i == 1 ? ls[1] : i == 2 ? ls[2] : ls[3], l);
    };
    const float padded = (static_cast<float>(p.nqg) * CQ + static_cast<float>(p.nb) * CB) * static_cast<float>(bh);
    if (__builtin_amdgcn_readfirstlane(total >= RAGGED_FILL * padded)) {
        if (p.piece >= p.pieces) p.head = -1;
        else tokens(p.head);
        return;
    }
    mx = wave_max64(mx);
    float target = total < 48e6f ? total / static_cast<float>(cus * 4 / 5)
                                 : fmaxf(98304.f, total / static_cast<float>(slots * 5 / 4));
    const int most = G > WAVES ? 24 : MAX_PARTIALS / 16;   // pieces per head (below the tables' limits)
    target = fmaxf(fmaxf(target, 16384.f), mx / static_cast<float>(most - 3));
    const uint32_t uq = static_cast<uint32_t>(target / CQ) + 1, ub = static_cast<uint32_t>(target / CB) + 1;
    uint32_t pc[4], mine = 0;                         // pieces: int4 in the low half, bf16 in the high
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t pq = (nq[i] + uq - 1) / uq;
        uint32_t pb = (nb[i] + ub - 1) / ub;
        if (pq + pb == 0) pb = 1;                     // an empty head still writes its (zero) output
        pc[i] = 4 * lane + i < bh ? pq | pb << 16 : 0u;
        mine += pc[i];
    }
    const uint32_t incl = wave_scan64(mine);
    const int totq = static_cast<int>(__builtin_amdgcn_readlane(incl, 63) & 0xffffu);
    const int id = blockIdx.y * bh + blockIdx.x;
    uint32_t base = incl - mine;
    int o[8] = {};
    bool found = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int bq = static_cast<int>(base & 0xffffu), bb = static_cast<int>(base >> 16);
        const int pq = static_cast<int>(pc[i] & 0xffffu), pb = static_cast<int>(pc[i] >> 16);
        const int iq = id - bq, ib = id - totq - bb;
        const bool q = iq >= 0 && iq < pq, b = ib >= 0 && ib < pb;
        if (q || b) {                                 // one lane at most
            const int n0 = static_cast<int>(nq[i]), n1 = static_cast<int>(nb[i]);
            found = true;
            o[0] = 4 * lane + i;
            o[1] = q ? iq : pq + ib;
            o[2] = pq + pb;
            o[3] = bq + bb;
            // (units times pieces stay below 2^27: 2^21 units, 64 pieces)
            o[4] = q ? n0 * iq / pq : n0 + n1 * ib / pb;
            o[5] = q ? n0 * (iq + 1) / pq : n0 + n1 * (ib + 1) / pb;
            o[6] = n0;
            o[7] = n1;
        }
        base += pc[i];
    }
    const uint64_t who = __builtin_amdgcn_ballot_w64(found);
    if (who == 0) {
        p.head = -1;
        return;
    }
    const int l = __builtin_ctzll(who);
    p.head = __builtin_amdgcn_readlane(o[0], l);
    p.piece = __builtin_amdgcn_readlane(o[1], l);
    p.pieces = __builtin_amdgcn_readlane(o[2], l);
    p.first = __builtin_amdgcn_readlane(o[3], l);
    p.u0 = __builtin_amdgcn_readlane(o[4], l);
    p.u1 = __builtin_amdgcn_readlane(o[5], l);
    p.nqg = __builtin_amdgcn_readlane(o[6], l);
    p.nb = __builtin_amdgcn_readlane(o[7], l);
    tokens(p.head);
}

// ---------------------------------------------------------------------------
// the kernel
// ---------------------------------------------------------------------------
// RAGGED: the pieces of ragged_piece.  Segments 1 and 2 are empty; the head
// strides of their K hold the device's CUs and resident workgroups.
template <int KB, int VB, bool RAGGED>
__global__ __launch_bounds__(THREADS, 2) void decode_kernel(DecArgs a) {
#ifdef HYQ_PHASE_TRACE
    uint64_t ph[TRACE_PH] = {};
    HYQ_STAMP(0);
    const uint32_t launch = __hip_atomic_load(&g_trace_launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#endif
    int head = blockIdx.x;
    int wg = blockIdx.y;                             // piece of the head
    KArgs K = kernel_args(RAGGED ? min(wg, MAX_NWG - 1) : wg);
    int u0 = static_cast<int>(K.bnd[0]), u1 = static_cast<int>(K.bnd[1]);         // its schedule units
    const uint16_t* const qp = kptr<const uint16_t>(K, 0);
    const uint8_t* const kp = kptr<const uint8_t>(K, 2);
    const uint8_t* const vp = kptr<const uint8_t>(K, 4);
    const uint16_t* const ksp = kptr<const uint16_t>(K, 6);
    const uint16_t* const vsp = kptr<const uint16_t>(K, 8);
    const uint16_t* const sk0 = kptr<const uint16_t>(K, 10);
    const uint16_t* const sk1 = kptr<const uint16_t>(K, 12);
    const uint16_t* const sk2 = kptr<const uint16_t>(K, 14);
    const uint16_t* const sv0 = kptr<const uint16_t>(K, 16);
    const uint16_t* const sv1 = kptr<const uint16_t>(K, 18);
    const uint16_t* const sv2 = kptr<const uint16_t>(K, 20);
    const int32_t* const len_q = kptr<const int32_t>(K, 22);
    const int32_t* const len_s0 = kptr<const int32_t>(K, 24);
    const int32_t q_stride = static_cast<int32_t>(kdw(K, 26));
    // head strides fit 32 bits (the host checks); products are formed in 64
    const int32_t kp_bh = static_cast<int32_t>(kdw(K, 27)), vp_bh = static_cast<int32_t>(kdw(K, 28));
    const int32_t ks_bh = static_cast<int32_t>(kdw(K, 29)), vs_bh = static_cast<int32_t>(kdw(K, 30));
    const int32_t skb0 = static_cast<int32_t>(kdw(K, 31)), skb1 = static_cast<int32_t>(kdw(K, 32));
    const int32_t skb2 = static_cast<int32_t>(kdw(K, 33)), svb0 = static_cast<int32_t>(kdw(K, 34));
    const int32_t svb1 = static_cast<int32_t>(kdw(K, 35)), svb2 = static_cast<int32_t>(kdw(K, 36));
    int nquant = static_cast<int>(kdw(K, 37));
    int sn0 = static_cast<int>(kdw(K, 38));
    const int sn1 = static_cast<int>(kdw(K, 39)), sn2 = static_cast<int>(kdw(K, 40));
    const int G = static_cast<int>(kdw(K, 41));
    int nqg = static_cast<int>(kdw(K, 42));
    int su0 = static_cast<int>(kdw(K, 43));
    const int su1 = static_cast<int>(kdw(K, 44));
    const float qk_scale = __uint_as_float(kdw(K, 45));
    const int io = static_cast<int>(kdw(K, 46));
    HYQ_STAMP(1);
    int pieces = 0, first = 0;                     // RAGGED: the head's pieces and first slot
    if constexpr (RAGGED) {
        epilogue_args(K);                          // (before anything can move the registers of those loads)
        const int nwg = static_cast<int>(K.e1[1]);
        RaggedPiece r{head, wg, nwg, head * nwg, u0, u1, nqg, su0, 0, 0};
        ragged_piece<KB, VB>(r, static_cast<int>(K.e1[3]), G, nquant, sn0, len_q, len_s0, skb1, skb2);
        if (r.head < 0) {
#ifdef HYQ_PHASE_TRACE
            if (threadIdx.x == 0) trace_end();
#endif
            return;
        }
        head = r.head;
        wg = r.piece;
        pieces = r.pieces;
        first = r.first;
        u0 = r.u0;
        u1 = r.u1;
        nqg = r.nqg;
        nquant = r.nq;
        sn0 = r.ns;
        su0 = r.nb;
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int c = lane & 15, kb = lane >> 4;

    extern __shared__ float s_acc[];               // [WAVES][G][D+1]; later the merge weights
    __shared__ float s_m[WAVES][16];
    __shared__ float s_l[WAVES][16];
    __shared__ int s_last;

    WaveState st;
    st.m = M_INIT;
    st.l = 0.f;
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) st.acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    st.ones = f32x4{0.f, 0.f, 0.f, 0.f};

    // Q row of head c (zero for padding columns c >= G): channels 32kb..32kb+31
    u32x4 qraw[4];
    {
        const Rsrc rq = make_rsrc(qp + static_cast<int64_t>(head) * G * q_stride,
                                  static_cast<uint32_t>(G * q_stride * 2));
        const uint32_t qo = static_cast<uint32_t>(c * q_stride * 2 + 64 * kb);
#pragma unroll
        for (int i = 0; i < 4; ++i) qraw[i] = bld128(rq, qo + 16 * i);
    }
    // an fp16 query is rounded to bf16 (as the reference's Q loads) once the
    // first K/V loads are in flight
    uint32_t q16 = (io & HYQ_DT_Q_FP16) ? ~0u : 0u;
    asm volatile("" : "+s"(q16));

    if (u0 < nqg) {
        // ---------------- int4 part: groups wave, wave+WAVES, ... ----------------
        const int lo = u0 * GROUP;
        int nq = nquant;
        if (!RAGGED && len_q != nullptr) nq = min(nq, max(0, sload_i32(len_q + head)));
        const int ntok = max(0, min((min(u1, nqg) - u0) * GROUP, nq - lo));   // 0: past a ragged head's end
        QCtx x;
        x.k = make_rsrc(kp + static_cast<int64_t>(head) * kp_bh + static_cast<int64_t>(lo) * prow(KB),
                        static_cast<uint32_t>(ntok) * prow(KB));
        x.v = make_rsrc(vp + static_cast<int64_t>(head) * vp_bh + static_cast<int64_t>(lo) * prow(VB),
                        static_cast<uint32_t>(ntok) * prow(VB));
        x.ks = make_rsrc(ksp + static_cast<int64_t>(head) * ks_bh + lo, static_cast<uint32_t>(ntok) * 2);
        x.vs = make_rsrc(vsp + static_cast<int64_t>(head) * vs_bh + lo, static_cast<uint32_t>(ntok) * 2);
        x.klane = static_cast<uint32_t>(krow_token(c) * prow(KB) + 4 * KB * kb);
        x.vlane = static_cast<uint32_t>(kb * prow(VB) + VB * c);
        x.slane = static_cast<uint32_t>((4 * (c & 3) + kb) * 2);
        // groups wave, wave+WAVES, ... of the piece through a three-deep
        // register ring: two groups' loads in flight while one is computed
        constexpr int STRIDE = WAVES * GROUP;
        const int ngrp = (ntok + GROUP - 1) / GROUP;
        const int nmine = ngrp > wave ? (ngrp - wave + WAVES - 1) / WAVES : 0;
        const int t0 = wave * GROUP;
        QRaw<KB, VB> b0, b1, b2;
        // in issue order (the scheduler would otherwise group the three
        // groups' loads by kind, which puts the first group's last load near
        // the end and its wait near a full drain)
        qload(b0, x, t0);
        __builtin_amdgcn_sched_barrier(0);
        qload(b1, x, t0 + STRIDE);
        __builtin_amdgcn_sched_barrier(0);
        qload(b2, x, t0 + 2 * STRIDE);
        __builtin_amdgcn_sched_barrier(0);
        q_to_bf16(qraw, q16);
        HYQ_STAMP(2);
#ifdef HYQ_PHASE_TRACE
        asm volatile("" ::"v"(b0.sv[1]));   // the last load of the first group
        HYQ_STAMP(3);
#endif

        // Q -> fp16 in int4 slot order, pre-scaled by 2^-ex so |q| < 2^15
        float qf[32];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t ww[4] = {qraw[i][0], qraw[i][1], qraw[i][2], qraw[i][3]};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                qf[8 * i + 2 * j] = __uint_as_float(ww[j] << 16);
                qf[8 * i + 2 * j + 1] = __uint_as_float(ww[j] & 0xffff0000u);
            }
        }
        float amax = 0.f;
#pragma unroll
        for (int i = 0; i < 32; ++i) amax = fmaxf(amax, fabsf(qf[i]));
        amax = col_max(amax);
        const int ex = amax >= 16384.f ? ilogbf(amax) - 13 : 0;
        const float qscale = ldexpf(1.0f, -ex);
        f16x8 qop[4];
#pragma unroll
        for (int sidx = 0; sidx < 4; ++sidx) {
            const float* f = qf + 8 * sidx;
            const f16x8 v = {static_cast<_Float16>(f[0] * qscale), static_cast<_Float16>(f[4] * qscale),
                             static_cast<_Float16>(f[1] * qscale), static_cast<_Float16>(f[5] * qscale),
                             static_cast<_Float16>(f[2] * qscale), static_cast<_Float16>(f[6] * qscale),
                             static_cast<_Float16>(f[3] * qscale), static_cast<_Float16>(f[7] * qscale)};
            qop[sidx] = v;
        }
        // the K operands are u * 2^-24 (k_operand): 2^24 goes into the score scale
        const float qk = qk_scale * ldexpf(1.0f, ex + 24);
        const f32x4 kbias = k_bias<KB>(qop);
        // First round peeled (its three groups' loads were all issued before
        // the wait for Q; straight-line code keeps the compiler's waits exact),
        // then the ring: each round issues a group's loads before computing
        // the oldest, two groups in flight while one is computed.
        do {
            qcompute(st, b0, qop, kbias, ntok - t0, lane, qk);
            if (nmine <= 1) break;
            qload(b0, x, t0 + 3 * STRIDE);
            qcompute(st, b1, qop, kbias, ntok - t0 - STRIDE, lane, qk);
            if (nmine <= 2) break;
            qload(b1, x, t0 + 4 * STRIDE);
            qcompute(st, b2, qop, kbias, ntok - t0 - 2 * STRIDE, lane, qk);
            for (int i = 3; i < nmine; i += 3) {
                const int t = t0 + i * STRIDE;
                qload(b2, x, t + 2 * STRIDE);
                __builtin_amdgcn_sched_barrier(0);
                qcompute(st, b0, qop, kbias, ntok - t, lane, qk);
                if (i + 1 >= nmine) break;
                qload(b0, x, t + 3 * STRIDE);
                __builtin_amdgcn_sched_barrier(0);
                qcompute(st, b1, qop, kbias, ntok - t - STRIDE, lane, qk);
                if (i + 2 >= nmine) break;
                qload(b1, x, t + 4 * STRIDE);
                __builtin_amdgcn_sched_barrier(0);
                qcompute(st, b2, qop, kbias, ntok - t - 2 * STRIDE, lane, qk);
            }
        } while (false);
        // remove the offset of the V operands: acc -= offset * sum_t P'
        const float corr = v_offset<VB>() * st.ones[0];
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) st.acc[nb] -= corr;
    } else {
        // ------------- bf16 parts: tiles wave, wave+WAVES, ... of each segment -------------
        // (a piece never holds both int4 and bf16 tokens: make_plan cuts at
        // the segment boundaries, so the Q copies of one part are dead
        // during the other's loop)
        // fp16 segments (an fp16 model's cache) are rounded to bf16 after
        // their loads, as the reference's .to(tl.bfloat16) of each tile
        const bool seg16 = io & HYQ_DT_SEG_FP16;
        // segment bounds in units: [nqg, b1), [b1, b2), [b2, end of head)
        const int b1 = nqg + su0, b2 = b1 + su1;
        for (int seg = 0; seg < 3; ++seg) {
            const int sb = seg == 0 ? nqg : seg == 1 ? b1 : b2;
            const int ua = max(u0, sb), ub = min(u1, seg == 0 ? b1 : seg == 1 ? b2 : u1);
            if (ua >= ub) continue;
            const int lo = (ua - sb) * BUNIT;
            int seg_len = seg == 0 ? sn0 : seg == 1 ? sn1 : sn2;
            if (!RAGGED && seg == 0 && len_s0 != nullptr) seg_len = min(seg_len, max(0, sload_i32(len_s0 + head)));
            const int n = max(0, min((ub - ua) * BUNIT, seg_len - lo));     // 0: past a ragged head's end
            const uint16_t* const skp = seg == 0 ? sk0 : seg == 1 ? sk1 : sk2;
            const uint16_t* const svp = seg == 0 ? sv0 : seg == 1 ? sv1 : sv2;
            const int32_t skb = seg == 0 ? skb0 : seg == 1 ? skb1 : skb2;
            const int32_t svb = seg == 0 ? svb0 : seg == 1 ? svb1 : svb2;
            const uint16_t* kbase = skp + static_cast<int64_t>(head) * skb + static_cast<int64_t>(lo) * BROW;
            const uint16_t* vbase = svp + static_cast<int64_t>(head) * svb + static_cast<int64_t>(lo) * BROW;
            const uint32_t nbytes = static_cast<uint32_t>(n) * (BROW * 2);
            const Rsrc rk = make_rsrc(kbase, nbytes), rv = make_rsrc(vbase, nbytes);
            // tiles wave, wave+WAVES, ... through a two-deep register ring
            constexpr int TSTRIDE = WAVES * TILE;
            const int ntile = (n + TILE - 1) / TILE;
            const int nmine = ntile > wave ? (ntile - wave + WAVES - 1) / WAVES : 0;
            const int t0 = wave * TILE;
            Bf16Raw r0, r1;
            bf16_load(r0, rk, rv, t0, lane);
            bf16_load(r1, rk, rv, t0 + TSTRIDE, lane);
            u32x4 qs[4] = {qraw[0], qraw[1], qraw[2], qraw[3]};
            q_to_bf16(qs, q16);
#ifdef HYQ_PHASE_TRACE
            if (ph[2] == 0) {
                HYQ_STAMP(2);
                asm volatile("" ::"v"(r0.v[3][3]));   // the last load of the first tile
                HYQ_STAMP(3);
            }
#endif
            const bf16x8 qb[4] = {__builtin_bit_cast(bf16x8, qs[0]), __builtin_bit_cast(bf16x8, qs[1]),
                                  __builtin_bit_cast(bf16x8, qs[2]), __builtin_bit_cast(bf16x8, qs[3])};
            // the ring: the tile two ahead is loaded into the slot just computed
            for (int i = 0; i < nmine; i += 2) {
                const int t = t0 + i * TSTRIDE;
                if (seg16) f16_to_bf16(r0);
                bf16_compute(st, r0, qb, n - t, lane, qk_scale);
                if (i + 1 >= nmine) break;
                bf16_load(r0, rk, rv, t + 2 * TSTRIDE, lane);
                if (seg16) f16_to_bf16(r1);
                bf16_compute(st, r1, qb, n - t - TSTRIDE, lane, qk_scale);
                if (i + 2 >= nmine) break;
                bf16_load(r1, rk, rv, t + 3 * TSTRIDE, lane);
            }
        }
    }

    // ---- wave -> LDS ----------------------------------------------------------
    HYQ_STAMP(4);
    epilogue_args(K);
    const int nwg = RAGGED ? pieces : static_cast<int>(K.e1[1]);
    const int mj = RAGGED ? merge_batch(G, nwg) : static_cast<int>(K.e1[2]);
    const MergeArgs ma{G, nwg, RAGGED ? static_cast<int64_t>(first) : static_cast<int64_t>(head) * nwg,
                       eptr<const float>(K, 2), eptr<const float>(K, 4), eptr<uint16_t>(K, 0),
                       static_cast<int64_t>(static_cast<int32_t>(K.e1[0])), io & HYQ_DT_OUT_FP16};
    uint32_t* const cnt = eptr<uint32_t>(K, 6);
    // The rings' last loads (past the piece's end: zeros, no memory access)
    // are drained here, with a wait the compiler sees, so that it has no
    // stale loads to wait for among the stores below.
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
    st.l = col_sum(st.l);
    if (kb == 0) {
        s_m[wave][c] = st.m;
        s_l[wave][c] = st.l;
    }
    if (c < G) {
        float* row = s_acc + (wave * G + c) * (D + 1);
#pragma unroll
        for (int nb = 0; nb < 8; ++nb)
#pragma unroll
            for (int i = 0; i < 4; ++i) row[32 * kb + 8 * i + nb] = st.acc[nb][i];
    }
    __syncthreads();
    HYQ_STAMP(5);

    // ---- workgroup merge -> partial acc[G][D] and (m, l)[G] ----------------------
    const int64_t slot = ma.first + wg;
    {
        const Rsrc rpart = make_rsrc(ma.part + slot * G * D, static_cast<uint32_t>(G * D * 4));
        for (int o = threadIdx.x; o < G * (D / 4); o += THREADS) {
            const int g = o / (D / 4), ch = 4 * (o % (D / 4));
            float M = s_m[0][g];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) M = fmaxf(M, s_m[w][g]);
            f32x4 accv = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                const float wt = fast_exp2(s_m[w][g] - M);
                const float* row = s_acc + (w * G + g) * (D + 1) + ch;
                accv += wt * f32x4{row[0], row[1], row[2], row[3]};
            }
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, accv), rpart, o * 16, 0, 16);   // sc1
        }
    }
    if (threadIdx.x < G) {
        const int g = threadIdx.x;
        float M = s_m[0][g];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) M = fmaxf(M, s_m[w][g]);
        float lv = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) lv += fast_exp2(s_m[w][g] - M) * s_l[w][g];
        float* const mlw = const_cast<float*>(ma.ml);
        __hip_atomic_store(mlw + (slot * G + g) * 2, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(mlw + (slot * G + g) * 2 + 1, lv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // every store of this workgroup acknowledged before its arrival is counted
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    HYQ_STAMP(6);
    if (threadIdx.x == 0) {
        const uint32_t old = __hip_atomic_fetch_add(cnt + head * CNT_PAD, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = (old == static_cast<uint32_t>(ma.nwg - 1));
    }
    __syncthreads();
    HYQ_STAMP(7);
    if (s_last) {
        if (threadIdx.x == 0) __hip_atomic_store(cnt + head * CNT_PAD, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        switch (mj) {      // G <= 4: merge_head_waves, pairs per lane; G > 4: merge_head_cols, items per thread
            case 4: merge_head_waves<4>(ma, head, s_acc TRACE_ARG); break;
            case 8: merge_head_waves<8>(ma, head, s_acc TRACE_ARG); break;
            case 12: merge_head_waves<12>(ma, head, s_acc TRACE_ARG); break;
            case 16: merge_head_waves<16>(ma, head, s_acc TRACE_ARG); break;
            case 20: merge_head_waves<20>(ma, head, s_acc TRACE_ARG); break;
            case 24: merge_head_waves<24>(ma, head, s_acc TRACE_ARG); break;
            case 108: merge_head_cols<8>(ma, head, s_acc); break;
            case 116: merge_head_cols<16>(ma, head, s_acc); break;
            default: merge_head_cols<24>(ma, head, s_acc); break;
        }
    }
#ifdef HYQ_PHASE_TRACE
    const uint32_t lwg = blockIdx.y * gridDim.x + blockIdx.x;
    if (lane == 0 && lwg < TRACE_MAX_WG) {
        ph[13] = launch;
        uint64_t* dst = g_trace[launch % TRACE_SLOTS][lwg * 4 + wave];
        for (int i = 0; i < TRACE_PH; ++i) dst[i] = ph[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) trace_end();
#endif
}

// ---------------------------------------------------------------------------
// legacy-format decode
// ---------------------------------------------------------------------------
// The legacy decode format of src/ops/d_stage_cache.py (fused_decode_
// attention_k4v4 :504-591, splitk_decode_attention_k4v4 :825-951 and its MMA
// variant :1247-1366 with K_BITS / V_BITS of 4 or 2, :977-1092): a prefix of
// offset-encoded codes (int4: channel 2j in the high nibble of byte j, value
// u - 8; int2: channel 4j + i in bits 7-2i..6-2i of byte j, value u - 1.5)
// with one fp16 scale per (group of tokens, channel), then the top-k,
// staging and window bf16 rows.
//
// The scales are folded out of the products, so that the codes go to the
// matrix cores as they are:
//   scores  q . (code * s_k) = (q * s_k) . code: once per scale group each
//     lane multiplies its 32 query channels by the group's scales in fp32 and
//     rounds them once to fp16, scaled by a power of two that puts the
//     column's largest product in [2^14, 2^15) (rounding error 2^-12 of a
//     channel's product, against 2^-9 for K rounded to bf16); the codes are
//     exact fp16 subnormals, as in k_operand;
//   P.V     sum_t P_t (code_t * s_v) = s_v * sum_t P_t code_t: the group's
//     sum is formed on its own accumulators (bf16(128 + u) operands and the
//     all-ones product that removes the offset, as in qcompute) and joins the
//     running one with one fp32 multiply-add per channel at the group's end.
// A tile's conversion then costs what the per-token format's does, where
// dequantising every element to bf16 cost about 2.9 VALU instructions an
// element and kept the VALU busy 59-67% of the time.  128 KV heads at 30011
// tokens (618 MB with the bf16 rows): K4V4 161 -> 101 us (6.1 TB/s, near the
// 6.8 TB/s of a read-only stream), K4V2 172 -> 91, K2V4 159 -> 94, K2V2 169 ->
// 90 us; 60 heads at G = 16, 5838 tokens 43 -> 21 us.  Two workgroups per CU
// (214-233 VGPRs, no spill; BLK = 1 at three per CU spills in its loop).  Error against float64, K4V4: 3.2e-3 -> 2.0e-3 of
// the output's norm.
//
// Prefix units are chunks of 32 tokens that never cross a scale group (a
// group that is not a multiple of 32 ends in a short chunk).  A wavefront
// walks blocks of BLK chunks of one scale group (legacy_blk): BLK = 4 shares
// one folding of the scales among a 128-token group's chunks; BLK = 1 folds
// them for every chunk.  Pieces, partials, arrival and merge are
// decode_kernel's.
//
// Kernel arguments.  The numbered dwords are read in one batch of scalar
// loads (legacy_args), so their layout is fixed, as DecArgs' is; qk_scale and
// mj stand in the lines of the arguments read later, which that batch brings
// into the scalar cache.
struct LegArgs {
    const uint16_t* q;             // dwords 0-1
    const uint8_t* kc;             // 2-3    prefix codes [bh][n][16 * bits] (byte strides)
    const uint8_t* vc;             // 4-5
    const uint16_t* ks;            // 6-7    prefix scales [bh][groups][D] (element head strides)
    const uint16_t* vs;            // 8-9
    int64_t kc_bh, vc_bh, ks_bh, vs_bh;   // 10-17
    uint64_t cdiv;                 // 18-19  2^40 / cpg, rounded up
    int32_t q_stride;              // 20
    uint32_t kc_n, vc_n;           // 21-22  bytes between code rows
    uint32_t ks_row, vs_row;       // 23-24  bytes between scale rows
    uint32_t ks_bytes, vs_bytes;   // 25-26  bytes of a head's scale rows (the descriptors' ranges)
    int32_t n_leg, group;          // 27-28
    int32_t cpg;                   // 29     chunks per scale group
    int32_t nqg;                   // 30     prefix schedule units (blocks) per head
    int32_t G;                     // 31
    int32_t segu[2];               // 32-33  bf16 schedule units (BUNIT tokens) of segments 0 and 1
    int32_t sn[3];                 // 34-36
    int32_t nwg;                   // 37
    const uint16_t* sk[3];         // top-k, staging, window rows [bh][n][D]
    int32_t pad0[4];
    float qk_scale;                // 48     sm_scale * log2(e)
    int32_t pad1;
    const uint16_t* sv[3];
    int64_t sk_bh[3], sv_bh[3];
    int32_t mj;                    // 68
    int32_t pad2;
    float* part;
    float* ml;
    uint32_t* cnt;
    uint16_t* out;
    int64_t out_stride;
    int32_t bnd[MAX_NWG + 1];      // piece p: schedule units [bnd[p], bnd[p + 1]) of its head
};
static_assert(offsetof(LegArgs, cdiv) == 4 * 18 && offsetof(LegArgs, nqg) == 4 * 30 && offsetof(LegArgs, nwg) == 4 * 37 &&
                  offsetof(LegArgs, qk_scale) == 4 * 48 && offsetof(LegArgs, mj) == 4 * 68 &&
                  offsetof(LegArgs, bnd) == 4 * 80, "argument block layout");

// The numbered arguments and the piece's bounds in one batch with one wait.
// Left to the compiler they came in five round trips one after the other (q,
// the bounds, the groups, the strides, the pointers), with two divisions
// between them, which show in a short cache's call of 7-10 us.
struct LegK {
    u32x16 a, b;
    u32x8 c;
    u32x2 bnd;
    uint32_t qk_scale, mj;
    __device__ __forceinline__ uint32_t d(int i) const { return i < 16 ? a[i] : i < 32 ? b[i - 16] : c[i - 32]; }
    __device__ __forceinline__ int i(int n) const { return static_cast<int>(d(n)); }
    __device__ __forceinline__ uint64_t q(int n) const { return d(n) | static_cast<uint64_t>(d(n + 1)) << 32; }
    template <typename T>
    __device__ __forceinline__ const T* p(int n) const { return reinterpret_cast<const T*>(static_cast<uintptr_t>(q(n))); }
};
__device__ __forceinline__ LegK legacy_args(int wg) {
    const char* const base = (const char*)__builtin_amdgcn_kernarg_segment_ptr();
    const char* const bp = base + offsetof(LegArgs, bnd) + 4 * wg;
    LegK k;
    asm volatile(
        "s_load_dwordx16 %0, %6, 0x0\n\t"
        "s_load_dwordx16 %1, %6, 0x40\n\t"
        "s_load_dwordx8 %2, %6, 0x80\n\t"
        "s_load_dwordx2 %3, %7, 0x0\n\t"
        "s_load_dword %4, %6, 0xc0\n\t"
        "s_load_dword %5, %6, 0x110\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&s"(k.a), "=&s"(k.b), "=&s"(k.c), "=&s"(k.bnd), "=&s"(k.qk_scale), "=&s"(k.mj)
        : "s"(base), "s"(bp)
        : "memory");
    return k;
}

// one 32-token chunk, in QRaw's layout (the scales are per group)
template <int KB, int VB>
struct LegRaw {
    uint32_t k[2][KB];
    uint32_t v[8];                 // VB bytes, zero-extended
};

// Chunk starting t tokens into its piece; the rows' strides (bytes) are
// uniform, so every load's position goes in its scalar offset.  Codes are
// read once: non-temporal.
template <int KB, int VB>
__device__ __forceinline__ void legacy_fetch(LegRaw<KB, VB>& r, Rsrc rk, Rsrc rv, uint32_t klane, uint32_t vlane,
                                             uint32_t t, uint32_t kc_n, uint32_t vc_n) {
    const uint32_t sk = __builtin_amdgcn_readfirstlane(t * kc_n);
    const uint32_t sv = __builtin_amdgcn_readfirstlane(t * vc_n);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if constexpr (KB == 4) {
            const u32x4 w = bld128<NT>(rk, klane, sk + 16 * i * kc_n);
            r.k[i][0] = w[0]; r.k[i][1] = w[1]; r.k[i][2] = w[2]; r.k[i][3] = w[3];
        } else {
            const u32x2 w = bld64<NT>(rk, klane, sk + 16 * i * kc_n);
            r.k[i][0] = w[0]; r.k[i][1] = w[1];
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
        r.v[e] = VB == 4 ? bld32<NT>(rv, vlane, sv + 4 * e * vc_n) : bld16<NT>(rv, vlane, sv + 4 * e * vc_n);
}

// A scale group's row, this lane's channels 32kb .. 32kb + 31 (8 fp16 per
// vector); every block of the group reads it: default policy.
__device__ __forceinline__ void legacy_scales(u32x4 (&s)[4], Rsrc r, int g, uint32_t row_bytes, int lane) {
    const uint32_t so = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(g) * row_bytes);
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] = bld128(r, static_cast<uint32_t>(64 * (lane >> 4) + 16 * i), so);
}

// The QK A operand of MFMA m (channels 32kb + 8m + [0..7]) as fp16 subnormals
// of value u * 2^-24 (int4) or 2u * 2^-24 (int2), in the channel order of
// leg_slot.
template <int KB>
__device__ __forceinline__ f16x8 legacy_k_operand(const uint32_t (&k)[KB], int m) {
    if constexpr (KB == 4) {
        const uint32_t x = k[m];
        const u32x4 o = {x & 0x000f000fu, (x >> 4) & 0x000f000fu, (x >> 8) & 0x000f000fu, (x >> 12) & 0x000f000fu};
        return __builtin_bit_cast(f16x8, o);
    } else {
        const uint32_t w = k[m >> 1];
        const uint32_t y = (m & 1) ? perm(w, w, 0x0c030c02u) : perm(w, w, 0x0c010c00u);
        const u32x4 o = {(y << 1) & 0x00060006u, (y >> 1) & 0x00060006u, (y >> 3) & 0x00060006u, (y >> 5) & 0x00060006u};
        return __builtin_bit_cast(f16x8, o);
    }
}
// channel (of 8) in fp16 half h of operand dword d: the pairs of
// legacy_k_operand's shifts
template <int KB>
__device__ __forceinline__ constexpr int leg_slot(int d, int h) {
    return KB == 4 ? (d ^ 1) + 4 * h : 3 - d + 4 * h;
}
// the code value is (u - 8) (int4) or (2u - 3) / 2 (int2); the operand's
// constant and the power of two that undoes 2^-24 (and the half)
template <int KB>
constexpr uint32_t leg_k_offset() { return KB == 4 ? 8u : 3u; }
template <int KB>
constexpr int leg_k_exp() { return KB == 4 ? 24 : 23; }
template <int VB>
constexpr float leg_v_offset() { return VB == 4 ? 136.0f : 129.5f; }

// x times the fp16 in the low or high half of sw (converted exactly)
__device__ __forceinline__ float mul_half(float x, uint32_t sw, int hi) {
    return x * f16_bits_to_f32(static_cast<uint16_t>(hi ? sw >> 16 : sw));
}

// The query column times a scale group's K scales: fp16 operands qop (scaled
// by 2^-e), the accumulators' start kbias and the score factor qk.  qn: the
// query's bf16 channels scaled by 2^-qex (legacy_norm_q).
template <int KB>
__device__ __forceinline__ void legacy_q_operand(f16x8 (&qop)[4], f32x4& kbias, float& qk, const u32x4 (&qn)[4],
                                                 const u32x4 (&ks)[4], float qk_scale, int qex) {
    float x[32];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x[8 * i + 2 * j] = mul_half(__uint_as_float(qn[i][j] << 16), ks[i][j], 0);
            x[8 * i + 2 * j + 1] = mul_half(__uint_as_float(qn[i][j] & 0xffff0000u), ks[i][j], 1);
        }
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) amax = fmaxf(amax, fabsf(x[i]));
    amax = col_max(amax);
    // 2^-e with e = exponent(amax) - 14; |qn| < 2 and |s| < 2^16, and a column
    // of zeros (or below 2^-113) keeps e = -127
    const int eb = max(static_cast<int>(__float_as_uint(amax) >> 23), 14);
    const float f = __uint_as_float(static_cast<uint32_t>(268 - eb) << 23);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const float* y = x + 8 * m;
        const f16x8 v = {
            static_cast<_Float16>(y[leg_slot<KB>(0, 0)] * f), static_cast<_Float16>(y[leg_slot<KB>(0, 1)] * f),
            static_cast<_Float16>(y[leg_slot<KB>(1, 0)] * f), static_cast<_Float16>(y[leg_slot<KB>(1, 1)] * f),
            static_cast<_Float16>(y[leg_slot<KB>(2, 0)] * f), static_cast<_Float16>(y[leg_slot<KB>(2, 1)] * f),
            static_cast<_Float16>(y[leg_slot<KB>(3, 0)] * f), static_cast<_Float16>(y[leg_slot<KB>(3, 1)] * f)};
        qop[m] = v;
    }
    qk = ldexpf(qk_scale, qex + leg_k_exp<KB>() + eb - 141);
    constexpr uint32_t o = leg_k_offset<KB>() * 0x00010001u;
    const u32x4 w = {o, o, o, o};
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < 4; ++m) acc = mfma_f16(__builtin_bit_cast(f16x8, w), qop[m], acc);
    kbias = -acc;
}

// The query column scaled in place by 2^-qex, so that its largest channel
// lies in [1, 2); returns qex (the same on the column's four lanes).
__device__ __forceinline__ int legacy_norm_q(u32x4 (&q)[4]) {
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            amax = fmaxf(amax, fmaxf(fabsf(__uint_as_float(q[i][j] << 16)), fabsf(__uint_as_float(q[i][j] & 0xffff0000u))));
    amax = col_max(amax);
    const int qex = max(static_cast<int>(__float_as_uint(amax) >> 23), 1) - 127;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            w[j] = pack_bf16x2(ldexpf(__uint_as_float(q[i][j] << 16), -qex),
                               ldexpf(__uint_as_float(q[i][j] & 0xffff0000u), -qex));
        q[i] = u32x4{w[0], w[1], w[2], w[3]};
    }
    return qex;
}

// One chunk: scores, online softmax (the running sums tot rescaled with the
// group's), P.V onto the group's accumulators st.acc / st.ones.
template <int KB, int VB>
__device__ __forceinline__ void legacy_compute(WaveState& st, f32x4 (&tot)[8], const LegRaw<KB, VB>& r,
                                               const f16x8 (&qop)[4], const f32x4& kbias, float qk, int nv, int lane) {
    const int kb = lane >> 4;
    float s[8];
#pragma unroll
    for (int tile = 0; tile < 2; ++tile) {
        f32x4 acc = kbias;
#pragma unroll
        for (int m = 0; m < 4; ++m) acc = mfma_f16(legacy_k_operand<KB>(r.k[tile], m), qop[m], acc);
#pragma unroll
        for (int i = 0; i < 4; ++i) s[4 * tile + i] = acc[i] * qk;
    }
    if (nv < GROUP) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (slot_token(kb, e) >= nv) s[e] = -INFINITY;
    }
    const float m0 = st.m;
    softmax_step<8>(st, s, true);
    if (__builtin_amdgcn_ballot_w64(st.m != m0)) {
        const float alpha = fast_exp2(m0 - st.m);
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) tot[nb] *= alpha;
    }
    const u32x4 pw = {pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3]), pack_bf16x2(s[4], s[5]),
                      pack_bf16x2(s[6], s[7])};
    const bf16x8 pop = __builtin_bit_cast(bf16x8, pw);
    uint32_t lo[4], hi[4];
#pragma unroll
    for (int pr = 0; pr < 4; ++pr) {
        lo[pr] = perm(r.v[2 * pr + 1], r.v[2 * pr], 0x05040100u);
        hi[pr] = VB == 4 ? perm(r.v[2 * pr + 1], r.v[2 * pr], 0x07060302u) : 0u;
    }
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) {
        // field nb of a row's dword is channel nb ^ 1 (nibbles) or nb ^ 3 (crumbs)
        u32x4 w;
        if constexpr (VB == 4) {
            const uint32_t* src = nb < 4 ? lo : hi;
            const int sh = 4 * (nb & 3);
            w = u32x4{nib2(src[0], sh, 0x43004300u), nib2(src[1], sh, 0x43004300u), nib2(src[2], sh, 0x43004300u),
                      nib2(src[3], sh, 0x43004300u)};
        } else {
            const int sh = 2 * nb;
            w = u32x4{((lo[0] >> sh) & 0x00030003u) | 0x43004300u, ((lo[1] >> sh) & 0x00030003u) | 0x43004300u,
                      ((lo[2] >> sh) & 0x00030003u) | 0x43004300u, ((lo[3] >> sh) & 0x00030003u) | 0x43004300u};
        }
        const int ch = VB == 4 ? nb ^ 1 : nb ^ 3;
        st.acc[ch] = mfma_bf16(__builtin_bit_cast(bf16x8, w), pop, st.acc[ch]);
    }
    const u32x4 onesw = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
    st.ones = mfma_bf16(__builtin_bit_cast(bf16x8, onesw), pop, st.ones);
}

// The scale group's end: tot += s_v * (acc - offset * sum P), accumulators
// cleared.  acc[nb][i] is channel 32kb + 8i + nb: element nb of vector i.
template <int VB>
__device__ __forceinline__ void legacy_flush(WaveState& st, f32x4 (&tot)[8], const u32x4 (&vs)[4]) {
    const float corr = leg_v_offset<VB>() * st.ones[0];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) {
            const float sc = f16_bits_to_f32(static_cast<uint16_t>((nb & 1) ? vs[i][nb >> 1] >> 16 : vs[i][nb >> 1]));
            tot[nb][i] = __builtin_fmaf(st.acc[nb][i] - corr, sc, tot[nb][i]);
        }
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) st.acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    st.ones = f32x4{0.f, 0.f, 0.f, 0.f};
}

template <int KB, int VB, int BLK>
__global__ __launch_bounds__(THREADS, 2) void legacy_decode_kernel(LegArgs a) {
#ifdef HYQ_PHASE_TRACE
    uint64_t ph[TRACE_PH] = {};    // (the merge stamps; not stored by this kernel)
#endif
    const int head = blockIdx.x;
    const int wg = blockIdx.y;
    const LegK K = legacy_args(wg);
    const int G = K.i(31);
    const int64_t h64 = head;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int c = lane & 15, kb = lane >> 4;

    extern __shared__ float s_acc[];               // [WAVES][G][D+1]; later the merge weights
    __shared__ float s_m[WAVES][16];
    __shared__ float s_l[WAVES][16];
    __shared__ u32x4 s_q[4][64];                   // the query column of each lane, scaled (prefix pieces)
    __shared__ int s_last;

    WaveState st;
    st.m = M_INIT;
    st.l = 0.f;
#pragma unroll
    for (int nb = 0; nb < 8; ++nb) st.acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    st.ones = f32x4{0.f, 0.f, 0.f, 0.f};

    // Q row of head c (zero for c >= G): channels 32kb..32kb+31
    u32x4 qs[4];
    {
        const int q_stride = K.i(20);
        const Rsrc rq = make_rsrc(K.p<uint16_t>(0) + h64 * G * q_stride, static_cast<uint32_t>(G * q_stride * 2));
        const uint32_t qo = static_cast<uint32_t>(c * q_stride * 2 + 64 * kb);
#pragma unroll
        for (int i = 0; i < 4; ++i) qs[i] = bld128(rq, qo + 16 * i);
    }

    const int u0 = static_cast<int>(K.bnd[0]), u1 = static_cast<int>(K.bnd[1]);   // this piece's schedule units
    const int nqg = K.i(30);
    if (u0 < nqg) {
        // chunk x of the head: group x / cpg, tokens [x / cpg * group + 32 (x % cpg), ...).
        // The quotient by multiplication: exact while x * cpg <= 2^40 (x is at
        // most 2^20 chunks and the loads past them, cpg at most 2^19)
        const int cpg = K.i(29), group = K.i(28), n_leg = K.i(27);
        const float qk_scale = __uint_as_float(K.qk_scale);
        const uint64_t cdiv = K.q(18);
        auto chunk_group = [&](int x) { return static_cast<int>(static_cast<uint32_t>(x) * cdiv >> 40); };
        auto chunk_token = [&](int x) {
            const int g = chunk_group(x);
            return g * group + (x - g * cpg) * GROUP;
        };
        const int x0 = u0 * BLK, x1 = min(u1, nqg) * BLK;
        const int lo = chunk_token(x0);
        const int n = min(n_leg, chunk_token(x1)) - lo;        // the piece's tokens
        const uint32_t kc_n = K.d(21), vc_n = K.d(22), ks_row = K.d(23), vs_row = K.d(24);
        const int64_t lo64 = lo;
        const Rsrc rk = make_rsrc(K.p<uint8_t>(2) + h64 * static_cast<int64_t>(K.q(10)) + lo64 * kc_n,
                                  static_cast<uint32_t>(n) * kc_n);
        const Rsrc rv = make_rsrc(K.p<uint8_t>(4) + h64 * static_cast<int64_t>(K.q(12)) + lo64 * vc_n,
                                  static_cast<uint32_t>(n) * vc_n);
        const Rsrc rks = make_rsrc(K.p<uint16_t>(6) + h64 * static_cast<int64_t>(K.q(14)), K.d(25));
        const Rsrc rvs = make_rsrc(K.p<uint16_t>(8) + h64 * static_cast<int64_t>(K.q(16)), K.d(26));
        const uint32_t klane = static_cast<uint32_t>(krow_token(c)) * kc_n + 4 * KB * kb;
        const uint32_t vlane = static_cast<uint32_t>(kb) * vc_n + VB * c;
        const int nblk = (x1 - x0) / BLK;
        // first token (from lo) and scale group of block b of the piece
        auto block_at = [&](int b, int& g) {
            const int x = x0 + b * BLK;
            g = __builtin_amdgcn_readfirstlane(chunk_group(x));
            return __builtin_amdgcn_readfirstlane(g * group + (x - g * cpg) * GROUP - lo);
        };
        // tokens of the group (and the prefix) from chunk start t on
        auto valid = [&](int t, int g) { return min((g + 1) * group, n_leg) - lo - t; };
        f32x4 tot[8];
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) tot[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (BLK == 4) {
            // a block's four chunks in four register slots
            LegRaw<KB, VB> r[BLK];
            u32x4 ksc[4], vsc[4];
            int g = 0, gn = 0;
            int t = block_at(wave, g), tn = 0;
            legacy_scales(ksc, rks, g, ks_row, lane);
#pragma unroll
            for (int j = 0; j < BLK; ++j) {
                legacy_fetch(r[j], rk, rv, klane, vlane, static_cast<uint32_t>(t + GROUP * j), kc_n, vc_n);
                __builtin_amdgcn_sched_barrier(0);
            }
            // the query waits in LDS between the groups (its 16 registers do
            // not fit beside the four slots)
            const int qex = legacy_norm_q(qs);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (i == wave) s_q[i][lane] = qs[i];
            __syncthreads();
            for (int b = wave; b < nblk; b += WAVES) {
                tn = block_at(b + WAVES, gn);          // past the piece: its loads read zeros
                f16x8 qop[4];
                f32x4 kbias;
                float qk;
                {
                    const u32x4 qn[4] = {s_q[0][lane], s_q[1][lane], s_q[2][lane], s_q[3][lane]};
                    legacy_q_operand<KB>(qop, kbias, qk, qn, ksc, qk_scale, qex);
                }
                legacy_scales(vsc, rvs, g, vs_row, lane);
#pragma unroll
                for (int j = 0; j < BLK; ++j) {
                    legacy_compute<KB, VB>(st, tot, r[j], qop, kbias, qk, valid(t + GROUP * j, g), lane);
                    legacy_fetch(r[j], rk, rv, klane, vlane, static_cast<uint32_t>(tn + GROUP * j), kc_n, vc_n);
                    if (j == BLK / 2) legacy_scales(ksc, rks, gn, ks_row, lane);
                    __builtin_amdgcn_sched_barrier(0);
                }
                legacy_flush<VB>(st, tot, vsc);
                t = tn;
                g = gn;
            }
        } else {
            // single chunks, each with its scale rows, in two slots
            struct Slot {
                LegRaw<KB, VB> r;
                u32x4 ks[4], vs[4];
                int t, g;
            } x[2];
            auto fetch = [&](Slot& y, int b) {
                y.t = block_at(b, y.g);                // past the piece: its loads read zeros
                legacy_scales(y.ks, rks, y.g, ks_row, lane);
                legacy_fetch(y.r, rk, rv, klane, vlane, static_cast<uint32_t>(y.t), kc_n, vc_n);
                legacy_scales(y.vs, rvs, y.g, vs_row, lane);
                __builtin_amdgcn_sched_barrier(0);
            };
            fetch(x[0], wave);
            fetch(x[1], wave + WAVES);
            const int qex = legacy_norm_q(qs);
            auto compute = [&](const Slot& y) {
                f16x8 qop[4];
                f32x4 kbias;
                float qk;
                legacy_q_operand<KB>(qop, kbias, qk, qs, y.ks, qk_scale, qex);
                legacy_compute<KB, VB>(st, tot, y.r, qop, kbias, qk, valid(y.t, y.g), lane);
                legacy_flush<VB>(st, tot, y.vs);
            };
            for (int b = wave; b < nblk; b += 2 * WAVES) {
                compute(x[0]);
                if (b + WAVES >= nblk) break;
                fetch(x[0], b + 2 * WAVES);
                compute(x[1]);
                if (b + 2 * WAVES >= nblk) break;
                fetch(x[1], b + 3 * WAVES);
            }
        }
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) st.acc[nb] = tot[nb];
    } else {
        const bf16x8 qb[4] = {__builtin_bit_cast(bf16x8, qs[0]), __builtin_bit_cast(bf16x8, qs[1]),
                              __builtin_bit_cast(bf16x8, qs[2]), __builtin_bit_cast(bf16x8, qs[3])};
        constexpr int TSTRIDE = WAVES * TILE;
        const int t0 = wave * TILE;
        const float qk_scale = __uint_as_float(K.qk_scale);
        const int b1 = nqg + K.i(32), b2 = b1 + K.i(33);
        const int sg = u0 < b1 ? 0 : u0 < b2 ? 1 : 2;            // a piece lies inside one segment
        const int lo = (u0 - (sg == 0 ? nqg : sg == 1 ? b1 : b2)) * BUNIT;
        const int n = min((u1 - u0) * BUNIT, (sg == 0 ? K.i(34) : sg == 1 ? K.i(35) : K.i(36)) - lo);
        const int ntile = (n + TILE - 1) / TILE;
        const int nmine = ntile > wave ? (ntile - wave + WAVES - 1) / WAVES : 0;
        const uint16_t* kbase = a.sk[sg] + h64 * a.sk_bh[sg] + static_cast<int64_t>(lo) * BROW;
        const uint16_t* vbase = a.sv[sg] + h64 * a.sv_bh[sg] + static_cast<int64_t>(lo) * BROW;
        const uint32_t nbytes = static_cast<uint32_t>(n) * (BROW * 2);
        const Rsrc rk = make_rsrc(kbase, nbytes), rv = make_rsrc(vbase, nbytes);
        Bf16Raw r0, r1;
        bf16_load(r0, rk, rv, t0, lane);
        bf16_load(r1, rk, rv, t0 + TSTRIDE, lane);
        for (int i = 0; i < nmine; i += 2) {
            const int t = t0 + i * TSTRIDE;
            bf16_compute(st, r0, qb, n - t, lane, qk_scale);
            if (i + 1 >= nmine) break;
            bf16_load(r0, rk, rv, t + 2 * TSTRIDE, lane);
            bf16_compute(st, r1, qb, n - t - TSTRIDE, lane, qk_scale);
            if (i + 2 >= nmine) break;
            bf16_load(r1, rk, rv, t + 3 * TSTRIDE, lane);
        }
    }

    // ---- wave -> LDS -> this piece's partial, then decode_kernel's arrival protocol ----
    const int nwg = K.i(37), mj = static_cast<int>(K.mj);
    const MergeArgs ma{G, nwg, h64 * nwg, a.part, a.ml, a.out, a.out_stride, 0};
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): the rings' last (empty) loads
    st.l = col_sum(st.l);
    if (kb == 0) {
        s_m[wave][c] = st.m;
        s_l[wave][c] = st.l;
    }
    if (c < G) {
        float* row = s_acc + (wave * G + c) * (D + 1);
#pragma unroll
        for (int nb = 0; nb < 8; ++nb)
#pragma unroll
            for (int i = 0; i < 4; ++i) row[32 * kb + 8 * i + nb] = st.acc[nb][i];
    }
    __syncthreads();
    const int64_t slot = static_cast<int64_t>(head) * ma.nwg + wg;
    {
        const Rsrc rpart = make_rsrc(ma.part + slot * G * D, static_cast<uint32_t>(G * D * 4));
        for (int o = threadIdx.x; o < G * (D / 4); o += THREADS) {
            const int g = o / (D / 4), ch = 4 * (o % (D / 4));
            float M = s_m[0][g];
#pragma unroll
            for (int w = 1; w < WAVES; ++w) M = fmaxf(M, s_m[w][g]);
            f32x4 accv = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < WAVES; ++w) {
                const float wt = fast_exp2(s_m[w][g] - M);
                const float* row = s_acc + (w * G + g) * (D + 1) + ch;
                accv += wt * f32x4{row[0], row[1], row[2], row[3]};
            }
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, accv), rpart, o * 16, 0, 16);   // sc1
        }
    }
    if (threadIdx.x < G) {
        const int g = threadIdx.x;
        float M = s_m[0][g];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) M = fmaxf(M, s_m[w][g]);
        float lv = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) lv += fast_exp2(s_m[w][g] - M) * s_l[w][g];
        __hip_atomic_store(a.ml + (slot * G + g) * 2, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(a.ml + (slot * G + g) * 2 + 1, lv, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // every store of this workgroup acknowledged before its arrival is counted
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t old = __hip_atomic_fetch_add(a.cnt + head * CNT_PAD, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = (old == static_cast<uint32_t>(ma.nwg - 1));
    }
    __syncthreads();
    if (s_last) {
        if (threadIdx.x == 0) __hip_atomic_store(a.cnt + head * CNT_PAD, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        switch (mj) {
            case 4: merge_head_waves<4>(ma, head, s_acc TRACE_ARG); break;
            case 8: merge_head_waves<8>(ma, head, s_acc TRACE_ARG); break;
            case 12: merge_head_waves<12>(ma, head, s_acc TRACE_ARG); break;
            case 16: merge_head_waves<16>(ma, head, s_acc TRACE_ARG); break;
            case 20: merge_head_waves<20>(ma, head, s_acc TRACE_ARG); break;
            case 24: merge_head_waves<24>(ma, head, s_acc TRACE_ARG); break;
            case 108: merge_head_cols<8>(ma, head, s_acc); break;
            case 116: merge_head_cols<16>(ma, head, s_acc); break;
            default: merge_head_cols<24>(ma, head, s_acc); break;
        }
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------

struct Slots {
    int slots, cus;        // workgroups resident at once, compute units (0: unknown)
};

struct Plan {
    int nwg;               // pieces per head
    int rows;              // workgroups per head that a ragged launch may have (0: none)
    bool ragged;           // planned on the device
    int cus, slots;        // of the device (rows > 0)
    int nqg, segu[3];      // schedule units: prefix units, bf16 units per segment
    int bnd[MAX_NWG + 1];  // piece p covers units [bnd[p], bnd[p+1])
};

// The prefix as schedule units: int4 groups of GROUP tokens, or the legacy
// format's blocks.
struct PrefixUnits {
    int64_t units;
    int tokens;            // per unit (full ones)
    int64_t bytes;         // per unit
    int64_t span;          // per unit, from its first row of K or V (the wider) to the next unit's
    int64_t conv;          // what converting a unit's codes costs, in bytes that a workgroup could read meanwhile
    bool legacy;
};
PrefixUnits group_units(int64_t n_quant, int kb, int vb) {
    return {(n_quant + GROUP - 1) / GROUP, GROUP, static_cast<int64_t>(GROUP) * (16 * kb + 16 * vb + 4),
            static_cast<int64_t>(GROUP) * 16 * std::max(kb, vb), kb + vb <= 8 ? 4750 : 9250, false};
}

// Bytes from a piece's first row to its end, in K or in V: its descriptors and
// the offsets into it are 32 bits wide, and the register slots are loaded up
// to 12 blocks past the end (4 MB covers 640 rows of the widest stride, 4096).
constexpr int64_t PIECE_SPAN = (int64_t{1} << 32) - (4 << 20);

size_t round256(size_t x) { return (x + 255) / 256 * 256; }

// Cut a head into pieces, each inside one segment (a piece spanning segments
// would walk their rings one after the other; decode_kernel relies on no
// piece holding both int4 and bf16 units), the int4 pieces first so that the
// short segment pieces fill the end of the grid.
//   requested > 0: pieces of about that many int4 tokens' bytes.
//   few KV heads (bh_kv < 32, a step of a few microseconds, bound by the
//     per-piece round trips), G <= 4: every segment cut into pieces of
//     equal bytes, total / (0.8 CUs) (measured best at B=1 from 2K to 32K
//     prefixes), at most 48 per head.
//   up to 64 KV heads and a launch of less than 48 MB (G <= 4, fewer than 32
//     heads in the legacy format only) or 80 MB (G > 4; any size with fewer
//     than 20 heads, or with G > 8 and codes of more than 8 bits a pair), 7-25
//     us that mix one piece's latency and the merge: the piece count with the
//     least modelled time (cheapest_pieces).  Swept over 515 shapes (32/8,
//     64/8 and 32/2 heads, batches 1-32, 1K-30K tokens, K4V4, K4V2 and K8V8;
//     graph replay over 700 MB of copies) and every count: 0.2% above each
//     shape's best on average, 4% at the worst, and up to 3% above
//     power-of-two pieces (fewer than 32 heads) and 1.25 rounds of at least 96
//     KiB, which are 11% above it on average.  6 x 2 heads, G = 16, 3600
//     tokens 15.3 (power-of-two pieces) -> 11.0 us; 5 x 8 heads, G = 4, 5151
//     tokens of K4V2 11.9 (1.25 rounds; 13.4 in pieces of equal bytes) ->
//     11.5; legacy 2-bit codes, 3 x 8 heads, 5151 tokens 17.4 (equal bytes) ->
//     12.2, 4 x 3600 16.1 -> 10.9.
//   G > 8, 20 to 64 KV heads, 60 MB or more and codes of at most 8 bits a
//     pair: 12 pieces, the most that the merge loads in one batch (48 heads,
//     16384 tokens 33.4 (1.25 rounds) -> 30.0 us, 13001 tokens with 2-bit V
//     25.9 -> 24.2; 32 heads, 30000 tokens 35.9 -> 35.2; 64 heads within 1%
//     of 1.25 rounds).  8-bit codes take longer per piece and lose by the
//     second round (32 heads, 30000 tokens 62.5 us in 1.25 rounds, 73.2 in 12
//     pieces, 54.2 in the model's ten).
//   else: pieces of about total / (1.25 * slots) bytes, `slots`
//     being the workgroups the device holds at once: the first round fills
//     every slot and the remaining quarter, with the short segment pieces,
//     evens out the workgroups that ran slow.  Pieces stay >= 96 KiB: below
//     that the per-piece round trips cost more than the balance gains.  From
//     a 384 KiB target the bf16 segments (the top-k rows above all, which
//     run in the last round) are cut at half the target: B=16, 32K went
//     from 100.9 to 98.2 us and B=8, 32K from 54.4 to 52.7 us (same box),
//     while with smaller targets the extra partials cost more than the
//     shorter round gains (GLM-4-9B shape, 248 KiB: 37.4 -> 40.1 us).
// Each segment gets its bytes / target pieces (rounded, at least one); the
// target grows until the pieces fit the merge tables.

// A head's segments as pieces: starting from the fewest (one each, or as many
// as PIECE_SPAN takes), every further piece goes to the segment whose pieces
// are the largest.
struct Pieces {
    const int64_t *su, *sc;             // units, bytes per unit
    int ks[4] = {0, 0, 0, 0};
    uint32_t per[4] = {0, 0, 0, 0};     // units and bytes of the segment's largest piece
    int64_t size[4] = {0, 0, 0, 0};
    int total = 0;
    void cut(int s) {                   // (a segment has at most 2^21 units)
        per[s] = (static_cast<uint32_t>(su[s]) + static_cast<uint32_t>(ks[s]) - 1) / static_cast<uint32_t>(ks[s]);
        size[s] = per[s] * sc[s];
    }
    Pieces(const int64_t (&u)[4], const int64_t (&c)[4], const int (&least)[4]) : su(u), sc(c) {
        for (int s = 0; s < 4; ++s)
            if (su[s] > 0) {
                ks[s] = least[s];
                cut(s);
                total += ks[s];
            }
    }
    int largest() const {
        int w = 0;
        for (int s = 1; s < 4; ++s)
            if (size[s] > size[w]) w = s;
        return w;
    }
    bool split() {                      // false: the largest piece is one unit
        const int w = largest();
        if (ks[w] >= su[w]) return false;
        ++ks[w];
        ++total;
        cut(w);
        return true;
    }
};

// Partials a merging thread loads for k pieces, rounded up to its batch.
int merge_loads(int G, int k) {
    const int items = G <= WAVES ? (k + 1) / 2 : merge_items(G, k);
    const int step = G <= WAVES ? 4 : 8;
    return items <= 24 ? (items + step - 1) / step * step : (items + 23) / 24 * 24;
}

// The piece count (at most kmax, and 15/16 of the resident slots: a full
// device starts its last workgroups late) with the least modelled time, in us.
// The grid runs piece by piece and fills every CU once, then a second time, so
// workgroup j shares its CU with workgroup j + cus: what both have to do at
// 32 KB/us and 0.2 us for the sharing, what the larger has left at 36.5 KB/us;
// plus 0.053 (G <= 4, a wavefront's merge) or 0.175 (a workgroup's) per
// partial loaded.  A unit of codes counts for more than its bytes (conv).
// Fitted to the sweep above.
Pieces cheapest_pieces(const Pieces& fewest, int64_t conv, int bh_kv, int G, int kmax, int64_t slots, int64_t cus) {
    Pieces p = fewest, best = p;
    const int most = std::min<int64_t>(kmax, std::max<int64_t>(p.total, slots * 15 / 16 / bh_kv));
    double least = 1e30;
    for (;;) {
        // more pieces load no fewer partials: once these alone cost the least
        // found, no further count can be cheaper (the loop is host time of
        // every call: 0.1-0.3 us this way, 1.4 to the last count)
        const double merge = (G <= WAVES ? 0.053 : 0.175) * merge_loads(G, p.total);
        if (merge >= least) break;
        double w[4];                    // modelled bytes of a segment's largest piece
        for (int s = 0; s < 4; ++s) w[s] = static_cast<double>(p.size[s]);
        w[0] += static_cast<double>(p.per[0] * conv);
        double stream = std::max(std::max(w[0], w[1]), std::max(w[2], w[3])) * (1.0 / 36.5e3);
        if (static_cast<int64_t>(p.total) * bh_kv > cus) {
            int64_t end[4];             // workgroups up to the segment's last
            for (int s = 0; s < 4; ++s) end[s] = (s > 0 ? end[s - 1] : 0) + static_cast<int64_t>(p.ks[s]) * bh_kv;
            int x = 0, y = 0;           // the segments of workgroups j and j + cus
            for (int64_t j = 0; j < std::min(cus, end[3] - cus);) {
                while (end[x] <= j) ++x;
                while (end[y] <= j + cus) ++y;
                stream = std::max(stream, std::min(w[x], w[y]) * (2.0 / 32e3) + std::fabs(w[x] - w[y]) * (1.0 / 36.5e3) + 0.2);
                j = std::min(end[x], end[y] - cus);
            }
        }
        const double cost = stream + merge;
        if (cost < least) {
            least = cost;
            for (int s = 0; s < 4; ++s) best.ks[s] = p.ks[s];
            best.total = p.total;
        }
        if (p.total >= most || !p.split()) break;
    }
    return best;
}

Plan make_plan(const PrefixUnits& pre, const int64_t seg_n[3], int bh_kv, int G, int requested, Slots sl_) {
    const int slots = sl_.slots;
    Plan p{};
    p.nqg = static_cast<int>(pre.units);
    for (int s = 0; s < 3; ++s) p.segu[s] = static_cast<int>((seg_n[s] + BUNIT - 1) / BUNIT);
    const int64_t cq = pre.bytes;                                               // bytes of a prefix unit
    const int64_t cb = static_cast<int64_t>(BUNIT) * 4 * D;                     // bytes of a bf16 unit (K and V)
    const int64_t su[4] = {p.nqg, p.segu[0], p.segu[1], p.segu[2]};             // units per segment
    const int64_t sc[4] = {cq, cb, cb, cb};
    int64_t head_bytes = 0;
    int least[4], fewest = 0;          // pieces that PIECE_SPAN takes
    for (int s = 0; s < 4; ++s) {
        head_bytes += su[s] * sc[s];
        const int64_t most = std::max<int64_t>(1, PIECE_SPAN / (s == 0 ? pre.span : cb / 2));   // units per piece
        least[s] = static_cast<int>((su[s] + most - 1) / most);
        fewest += least[s];
    }
    p.nwg = 0;
    if (fewest == 0) return p;
    // (2^24 rows of stride 4096 and three segments of 2^24 rows: 39 pieces at most)
    const int kmax = std::max(fewest, std::min(MAX_NWG, MAX_PARTIALS / G));
    int ks[4];
    int bdiv = 1;                      // the bf16 segments' pieces: target / bdiv bytes
    auto counts_for = [&](int64_t target) {
        int total = 0;
        for (int s = 0; s < 4; ++s) {
            const int64_t tg = s == 0 ? target : std::max<int64_t>(1, target / bdiv);
            ks[s] = su[s] > 0 ? static_cast<int>(std::min<int64_t>(
                                    su[s], std::max<int64_t>(least[s], (su[s] * sc[s] + tg / 2) / tg)))
                              : 0;
            total += ks[s];
        }
        return total;
    };
    int total;
    int64_t target;
    const bool wide = cq > static_cast<int64_t>(pre.tokens) * (16 * 8 + 4);   // codes of more than 8 bits a pair
    const bool large = G > 8 && bh_kv >= 20 && head_bytes * bh_kv >= 60000000;
    const bool twelve = large && !wide;
    const bool small = head_bytes * bh_kv < (G <= WAVES ? 48000000 : 80000000);
    if (requested > 0) {
        target = std::max<int64_t>(1, (requested + pre.tokens - 1) / pre.tokens) * cq;
        total = counts_for(target);
    } else if (bh_kv < 32 && G <= WAVES && !(pre.legacy && small)) {
        // few heads, G <= 4: pieces of equal bytes, about 0.8 per CU (a
        // workgroup per CU streams faster than two sharing one, and the
        // merge grows with the piece count), at least 8 KiB and at most 48
        // per head
        const int64_t cus = sl_.cus > 0 ? sl_.cus : 256;
        target = std::max<int64_t>(8 << 10, head_bytes * bh_kv * 5 / (4 * cus));
        target = std::max<int64_t>(target, (head_bytes + 47) / 48);
        total = counts_for(target);
    } else if (bh_kv <= 64 && (small || large || bh_kv < 20)) {
        Pieces best(su, sc, least);
        if (twelve) {
            while (best.total < std::min(kmax, 12) && best.split()) {}
        } else {
            best = cheapest_pieces(best, pre.conv, bh_kv, G, kmax, slots > 0 ? slots : 512,
                                   sl_.cus > 0 ? sl_.cus : 256);
        }
        for (int s = 0; s < 4; ++s) ks[s] = best.ks[s];
        total = best.total;
        target = (head_bytes + total - 1) / total;
    } else {
        const int64_t sl = slots > 0 ? slots : 512;
        target = std::max<int64_t>(96 << 10, head_bytes * bh_kv * 4 / (5 * sl));
        bdiv = target >= (384 << 10) ? 2 : 1;
        total = counts_for(target);
    }
    while (total > kmax) {
        target += target / 8 + 1;
        total = counts_for(target);
    }
    int64_t base = 0;
    for (int s = 0; s < 4; ++s) {
        for (int i = 0; i < ks[s]; ++i) p.bnd[p.nwg++] = static_cast<int>(base + su[s] * i / ks[s]);
        base += su[s];
    }
    p.bnd[p.nwg] = static_cast<int>(base);
    return p;
}

size_t lds_bytes(int G) {
    return std::max(static_cast<size_t>(WAVES) * G * (D + 1), static_cast<size_t>(MERGE_LDS)) * sizeof(float);
}

// Workgroups of a decode kernel the device holds at once (and the device's
// CU count), cached per device and GQA width (the LDS size).
Slots slots_of(const void* kernel, std::atomic<int> (&cache)[64][17][2], int G) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64 || G < 1 || G > 16) return {0, 0};
    const int known = cache[dev][G][0].load(std::memory_order_relaxed);
    if (known > 0) return {known, cache[dev][G][1].load(std::memory_order_relaxed)};
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, THREADS, lds_bytes(G)) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return {0, 0};
    cache[dev][G][1].store(cus, std::memory_order_relaxed);
    cache[dev][G][0].store(per_cu * cus, std::memory_order_relaxed);
    return {per_cu * cus, cus};
}

template <int KB, int VB>
Slots resident_slots_of(int G) {
    static std::atomic<int> cache[64][17][2];
    return slots_of(reinterpret_cast<const void*>(&decode_kernel<KB, VB, false>), cache, G);
}

Slots resident_slots(int kb, int vb, int G) {
    switch (10 * kb + vb) {
        case 44: return resident_slots_of<4, 4>(G);
        case 42: return resident_slots_of<4, 2>(G);
        case 48: return resident_slots_of<4, 8>(G);
        case 24: return resident_slots_of<2, 4>(G);
        case 22: return resident_slots_of<2, 2>(G);
        case 28: return resident_slots_of<2, 8>(G);
        case 84: return resident_slots_of<8, 4>(G);
        case 82: return resident_slots_of<8, 2>(G);
        default: return resident_slots_of<8, 8>(G);
    }
}

// Large calls with ragged lengths are planned on the device (ragged_piece);
// the others by the padded lengths, like a full batch.  The workspace of a
// ragged call is sized for the device's pieces either way.
Plan plan_for(const hyq_decode_params* p, bool ragged = true) {
    const int kb = p->n_quant > 0 ? p->k_bits : 4, vb = p->n_quant > 0 ? p->v_bits : 4;
    const Slots sl = resident_slots(kb, vb, p->kv_repeat);
    const PrefixUnits pre = group_units(p->n_quant, kb, vb);
    Plan pl = make_plan(pre, p->seg_n, p->bh_kv, p->kv_repeat, p->split_tokens, sl);
    const bool lens = (p->n_quant > 0 && p->seq_lens_quant) || (p->seg_n[0] > 0 && p->seq_lens_seg0);
    if (ragged && lens && p->bh_kv <= RAGGED_HEADS && p->seg_n[1] == 0 && p->seg_n[2] == 0 && p->split_tokens <= 0 &&
        sl.slots > 0) {
        const int64_t head_bytes = pre.units * pre.bytes + static_cast<int64_t>(pl.segu[0]) * BUNIT * 4 * D;
        pl.rows = std::max(pl.nwg, (ragged_grid(p->bh_kv, sl.cus, sl.slots) + p->bh_kv - 1) / p->bh_kv);
        pl.ragged = p->bh_kv * head_bytes >= RAGGED_BYTES;
        pl.cus = sl.cus;
        pl.slots = sl.slots;
    }
    return pl;
}

// workspace: [arrival counters: CNT_CAP slots, 128 B apart][(m, l) table][partials].
// The counter area has the same size and place for every call, so the data of
// one call never lands on the counters of another call of a different shape.
struct Layout {
    size_t cnt, ml, part, total;
};
Layout layout(const Plan& pl, int bh_kv, int G) {
    const size_t slots = static_cast<size_t>(bh_kv) * std::max({pl.nwg, pl.rows, 1}) * G;
    Layout L;
    L.cnt = 0;
    L.ml = static_cast<size_t>(CNT_CAP) * CNT_PAD * sizeof(uint32_t);
    L.part = L.ml + round256(slots * 2 * sizeof(float));
    L.total = L.part + round256(slots * D * sizeof(float));
    return L;
}

bool fits31(int64_t x) { return x >= 0 && x <= 0x7fffffffLL; }

int validate(const hyq_decode_params* p) {
    if (!p) return fail(HYQ_EINVAL, "null params");
    if (p->head_dim != D) return fail(HYQ_ENOTSUP, "head_dim must be 128, got " + std::to_string(p->head_dim));
    auto okbits = [](int b) { return b == 2 || b == 4 || b == 8; };
    if (!okbits(p->k_bits) || !okbits(p->v_bits))
        return fail(HYQ_EINVAL, "k_bits and v_bits must be 2, 4 or 8 (k_bits=" + std::to_string(p->k_bits) +
                                    ", v_bits=" + std::to_string(p->v_bits) + ")");
    if (p->kv_repeat < 1 || p->kv_repeat > 16)
        return fail(HYQ_ENOTSUP, "kv_repeat must be in [1, 16], got " + std::to_string(p->kv_repeat));
    if (p->bh_kv < 0) return fail(HYQ_EINVAL, "bh_kv < 0");
    if (p->bh_kv > CNT_CAP) return fail(HYQ_ENOTSUP, "bh_kv (batch * kv heads) above " + std::to_string(CNT_CAP));
    if (p->n_quant < 0 || p->n_quant > (1 << 24)) return fail(HYQ_EINVAL, "bad n_quant");
    if (p->dtype_flags & ~(HYQ_DT_Q_FP16 | HYQ_DT_SEG_FP16 | HYQ_DT_OUT_FP16))
        return fail(HYQ_EINVAL, "unknown dtype_flags bits " + std::to_string(p->dtype_flags));
    if (p->bh_kv == 0) return HYQ_OK;
    if (!p->q || !p->out) return fail(HYQ_EINVAL, "null q/out");
    if (!aligned(p->q, 16) || p->q_stride % 8 || p->q_stride < D)
        return fail(HYQ_EINVAL, "q must be 16-byte aligned with row stride % 8 == 0 and >= head_dim");
    if (static_cast<int64_t>(p->kv_repeat) * p->q_stride * 2 > 0x7fffffffLL) return fail(HYQ_ENOTSUP, "q row stride too large");
    if (!aligned(p->out, 8) || p->out_stride % 4 || p->out_stride < D)
        return fail(HYQ_EINVAL, "out must be 8-byte aligned with row stride % 4 == 0 and >= head_dim");
    if (!fits31(p->out_stride)) return fail(HYQ_ENOTSUP, "out row stride must lie in [0, 2^31)");
    if (p->n_quant > 0) {
        if (!p->k_packed || !p->v_packed || !p->k_scale || !p->v_scale) return fail(HYQ_EINVAL, "null prefix tensor");
        if (p->kp_stride_n != prow(p->k_bits) || p->vp_stride_n != prow(p->v_bits))
            return fail(HYQ_EINVAL, "packed K/V rows must be contiguous (token stride 16 * bits bytes)");
        const int ka = p->k_bits == 2 ? 8 : 16, va = p->v_bits;      // load sizes in bytes
        if (!aligned(p->k_packed, ka) || p->kp_stride_bh % ka)
            return fail(HYQ_EINVAL, "k_packed must be " + std::to_string(ka) + "-byte aligned, head stride included");
        if (!aligned(p->v_packed, va) || p->vp_stride_bh % va)
            return fail(HYQ_EINVAL, "v_packed must be " + std::to_string(va) + "-byte aligned, head stride included");
        if (!aligned(p->k_scale, 2) || !aligned(p->v_scale, 2))
            return fail(HYQ_EINVAL, "scales must be 2-byte aligned");
        if (!fits31(p->kp_stride_bh) || !fits31(p->vp_stride_bh) || !fits31(p->ks_stride_bh) || !fits31(p->vs_stride_bh))
            return fail(HYQ_ENOTSUP, "prefix head strides must lie in [0, 2^31)");
    }
    for (int s = 0; s < 3; ++s) {
        if (p->seg_n[s] < 0 || p->seg_n[s] > (1 << 23)) return fail(HYQ_EINVAL, "bad segment length");
        if (p->seg_n[s] == 0) continue;
        if (!p->seg_k[s] || !p->seg_v[s]) return fail(HYQ_EINVAL, "null bf16 segment");
        if (p->seg_k_stride_n[s] != BROW || p->seg_v_stride_n[s] != BROW)
            return fail(HYQ_EINVAL, "bf16 segment rows must be contiguous (token stride = head_dim)");
        if (!aligned(p->seg_k[s], 16) || !aligned(p->seg_v[s], 16) || p->seg_k_stride_bh[s] % 8 ||
            p->seg_v_stride_bh[s] % 8)
            return fail(HYQ_EINVAL, "bf16 segments must be 16-byte aligned with head strides % 8 == 0");
        if (!fits31(p->seg_k_stride_bh[s]) || !fits31(p->seg_v_stride_bh[s]))
            return fail(HYQ_ENOTSUP, "bf16 segment head strides must lie in [0, 2^31)");
    }
    return HYQ_OK;
}

// ---- legacy-format decode: plan and checks ----
// Scale-group length as the kernel walks it: a group that covers the whole
// prefix is cut to the prefix (rounded up to chunks).
int legacy_group(const hyq_legacy_params* p) {
    const int64_t whole = (p->n + GROUP - 1) / GROUP * GROUP;
    return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(p->group, whole)));
}
// Chunks per block: four, which share one folding of the scales, when the
// group's chunk count is a multiple of four (128-token groups) and one
// workgroup per CU gets a block for each of its wavefronts; else single
// chunks, which spread a short cache over more wavefronts.  Kernel time with
// the best piece count of each, single chunks / blocks: 8 KV heads at 1100
// tokens 6.7 / 8.3 us, at 7300 8.8 / 9.1, at 10000 9.9 / 9.5, at 30000 16.8 /
// 14.7; 32 heads at 1100 8.1 / 8.8, at 3600 11.1 / 10.6, at 7300 15.7 / 13.8.
int legacy_blk(const hyq_legacy_params* p, int cus) {
    const int64_t cpg = (legacy_group(p) + GROUP - 1) / GROUP;
    return cpg % 4 == 0 && p->n / (4 * GROUP) * p->bh_kv >= WAVES * (cus > 0 ? cus : 256) ? 4 : 1;
}

template <int KB, int VB, int BLK>
Slots legacy_slots_of(int G) {
    static std::atomic<int> cache[64][17][2];
    return slots_of(reinterpret_cast<const void*>(&legacy_decode_kernel<KB, VB, BLK>), cache, G);
}
Slots legacy_slots(int kb, int vb, int blk, int G) {
    switch (100 * kb + 10 * vb + blk) {
        case 444: return legacy_slots_of<4, 4, 4>(G);
        case 424: return legacy_slots_of<4, 2, 4>(G);
        case 244: return legacy_slots_of<2, 4, 4>(G);
        case 224: return legacy_slots_of<2, 2, 4>(G);
        case 441: return legacy_slots_of<4, 4, 1>(G);
        case 421: return legacy_slots_of<4, 2, 1>(G);
        case 241: return legacy_slots_of<2, 4, 1>(G);
        default: return legacy_slots_of<2, 2, 1>(G);
    }
}

Plan legacy_plan(const hyq_legacy_params* p) {
    PrefixUnits pre{0, GROUP, 1, 1, 0, true};
    int blk = 4;
    if (p->n > 0) {
        const int group = legacy_group(p);
        blk = legacy_blk(p, legacy_slots(p->k_bits, p->v_bits, 4, p->kv_repeat).cus);
        const int64_t cpg = (group + GROUP - 1) / GROUP, full = p->n / group, rest = p->n - full * group;
        pre.units = full * (cpg / blk) + ((rest + GROUP - 1) / GROUP + blk - 1) / blk;
        pre.tokens = blk * GROUP;
        pre.bytes = static_cast<int64_t>(pre.tokens) * (16 * p->k_bits + 16 * p->v_bits) + 4 * D;
        pre.span = std::min<int64_t>(pre.tokens, group) * std::max(p->kc_stride_n, p->vc_stride_n);
        pre.conv = blk == 4 ? 44000 : 20500;
    }
    return make_plan(pre, p->seg_n, p->bh_kv, p->kv_repeat, 0, legacy_slots(p->k_bits, p->v_bits, blk, p->kv_repeat));
}

int validate_legacy(const hyq_legacy_params* p) {
    const char* w = "hyq_decode_legacy: ";
    if (!p) return fail(HYQ_EINVAL, std::string(w) + "null params");
    if (p->head_dim != D) return fail(HYQ_ENOTSUP, std::string(w) + "head_dim must be 128");
    if ((p->k_bits != 2 && p->k_bits != 4) || (p->v_bits != 2 && p->v_bits != 4))
        return fail(HYQ_ENOTSUP, std::string(w) + "k_bits and v_bits must be 2 or 4");
    if (p->kv_repeat < 1 || p->kv_repeat > 16) return fail(HYQ_ENOTSUP, std::string(w) + "kv_repeat must be in [1, 16]");
    if (p->bh_kv < 0 || p->bh_kv > CNT_CAP) return fail(HYQ_ENOTSUP, std::string(w) + "bh_kv out of range");
    if (p->bh_kv == 0) return HYQ_OK;
    constexpr int64_t NMAX = int64_t{1} << 24;
    if (p->n < 0 || p->n > NMAX) return fail(HYQ_ENOTSUP, std::string(w) + "prefix length out of [0, 2^24]");
    int64_t total = p->n;
    for (int s = 0; s < 3; ++s) {
        if (p->seg_n[s] < 0 || p->seg_n[s] > NMAX) return fail(HYQ_ENOTSUP, std::string(w) + "segment length out of [0, 2^24]");
        total += p->seg_n[s];
        if (p->seg_n[s] == 0) continue;
        if (!p->seg_k[s] || !p->seg_v[s]) return fail(HYQ_EINVAL, std::string(w) + "null segment");
        if (!aligned(p->seg_k[s], 16) || !aligned(p->seg_v[s], 16) || p->seg_k_stride_bh[s] % 8 ||
            p->seg_v_stride_bh[s] % 8 || p->seg_k_stride_bh[s] < 0 || p->seg_v_stride_bh[s] < 0)
            return fail(HYQ_EINVAL, std::string(w) + "segments must be 16-byte aligned (head strides % 8 == 0)");
    }
    if (total == 0) return fail(HYQ_EINVAL, std::string(w) + "decode with zero key tokens");
    if (!p->q || !p->out) return fail(HYQ_EINVAL, std::string(w) + "null q or out");
    if (!aligned(p->q, 16) || p->q_stride % 8 || p->q_stride < D || p->q_stride > NMAX)
        return fail(HYQ_EINVAL, std::string(w) + "q rows must be 16-byte aligned, stride in [128, 2^24]");
    if (!aligned(p->out, 8) || p->out_stride % 4 || p->out_stride < D)
        return fail(HYQ_EINVAL, std::string(w) + "out rows must be 8-byte aligned");
    if (p->n > 0) {
        if (p->group <= 0 || p->group % 16) return fail(HYQ_EINVAL, std::string(w) + "group must be a positive multiple of 16");
        if (!p->k_codes || !p->v_codes || !p->k_scale || !p->v_scale) return fail(HYQ_EINVAL, std::string(w) + "null prefix");
        // a K row is read as one 4*k_bits-byte load per lane, a V row as
        // v_bits-byte loads: rows aligned to those sizes, at least 16*bits bytes
        const int ka = 4 * p->k_bits, va = p->v_bits, krow = 16 * p->k_bits, vrow = 16 * p->v_bits;
        if (!aligned(p->k_codes, ka) || p->kc_stride_n % ka || p->kc_stride_bh % ka || p->kc_stride_n < krow ||
            p->kc_stride_n > 4096 || p->kc_stride_bh < 0)
            return fail(HYQ_EINVAL, std::string(w) + "k_codes rows must be " + std::to_string(ka) +
                                        "-byte aligned, row stride in [" + std::to_string(krow) + ", 4096]");
        if (!aligned(p->v_codes, va) || p->vc_stride_n % va || p->vc_stride_bh % va || p->vc_stride_n < vrow ||
            p->vc_stride_n > 4096 || p->vc_stride_bh < 0)
            return fail(HYQ_EINVAL, std::string(w) + "v_codes rows must be " + std::to_string(va) +
                                        "-byte aligned, row stride in [" + std::to_string(vrow) + ", 4096]");
        if (!aligned(p->k_scale, 16) || !aligned(p->v_scale, 16) || p->ks_stride_g % 8 || p->vs_stride_g % 8 ||
            p->ks_stride_bh % 8 || p->vs_stride_bh % 8 || p->ks_stride_g < D || p->vs_stride_g < D ||
            p->ks_stride_bh < 0 || p->vs_stride_bh < 0)
            return fail(HYQ_EINVAL, std::string(w) + "scale rows must be 16-byte aligned (strides % 8 == 0)");
        const int64_t rows = (p->n + p->group - 1) / p->group;
        if (rows * std::max(p->ks_stride_g, p->vs_stride_g) * 2 > 0xffffffffLL)
            return fail(HYQ_ENOTSUP, std::string(w) + "a head's scale rows span 4 GiB or more");
    }
    return HYQ_OK;
}

int launch_legacy(const hyq_legacy_params* p, const Plan& pl, const Layout& L, void* workspace, void* stream) {
    LegArgs a{};
    a.q = p->q; a.q_stride = static_cast<int32_t>(p->q_stride);
    a.kc = p->k_codes; a.vc = p->v_codes;
    a.kc_bh = p->kc_stride_bh; a.vc_bh = p->vc_stride_bh;
    a.kc_n = static_cast<uint32_t>(p->kc_stride_n); a.vc_n = static_cast<uint32_t>(p->vc_stride_n);
    a.ks = p->k_scale; a.vs = p->v_scale;
    a.ks_bh = p->ks_stride_bh; a.vs_bh = p->vs_stride_bh;
    a.group = p->n > 0 ? legacy_group(p) : GROUP;
    const int64_t rows = (p->n + a.group - 1) / a.group;
    a.ks_row = static_cast<uint32_t>(p->ks_stride_g * 2); a.vs_row = static_cast<uint32_t>(p->vs_stride_g * 2);
    a.ks_bytes = static_cast<uint32_t>(rows * p->ks_stride_g * 2);
    a.vs_bytes = static_cast<uint32_t>(rows * p->vs_stride_g * 2);
    a.n_leg = static_cast<int>(p->n);
    a.cpg = (a.group + GROUP - 1) / GROUP;
    a.cdiv = ((uint64_t{1} << 40) + a.cpg - 1) / a.cpg;
    a.nqg = pl.nqg;
    a.segu[0] = pl.segu[0]; a.segu[1] = pl.segu[1];
    for (int s = 0; s < 3; ++s) {
        a.sk[s] = p->seg_k[s]; a.sv[s] = p->seg_v[s];
        a.sk_bh[s] = p->seg_k_stride_bh[s]; a.sv_bh[s] = p->seg_v_stride_bh[s];
        a.sn[s] = static_cast<int>(p->seg_n[s]);
    }
    a.G = p->kv_repeat;
    a.qk_scale = p->sm_scale * LOG2E;
    char* ws = static_cast<char*>(workspace);
    a.cnt = reinterpret_cast<uint32_t*>(ws + L.cnt);
    a.ml = reinterpret_cast<float*>(ws + L.ml);
    a.part = reinterpret_cast<float*>(ws + L.part);
    a.out = p->out; a.out_stride = p->out_stride;
    a.nwg = pl.nwg;
    a.mj = merge_batch(a.G, pl.nwg);
    for (int i = 0; i <= pl.nwg; ++i) a.bnd[i] = pl.bnd[i];
    hipStream_t st = static_cast<hipStream_t>(stream);
    const dim3 grid(static_cast<unsigned>(p->bh_kv), static_cast<unsigned>(pl.nwg));
    const size_t lds = lds_bytes(a.G);
    switch (100 * p->k_bits + 10 * p->v_bits + legacy_blk(p, legacy_slots(p->k_bits, p->v_bits, 4, a.G).cus)) {
        case 444: legacy_decode_kernel<4, 4, 4><<<grid, dim3(THREADS), lds, st>>>(a); break;
        case 424: legacy_decode_kernel<4, 2, 4><<<grid, dim3(THREADS), lds, st>>>(a); break;
        case 244: legacy_decode_kernel<2, 4, 4><<<grid, dim3(THREADS), lds, st>>>(a); break;
        case 224: legacy_decode_kernel<2, 2, 4><<<grid, dim3(THREADS), lds, st>>>(a); break;
        case 441: legacy_decode_kernel<4, 4, 1><<<grid, dim3(THREADS), lds, st>>>(a); break;
        case 421: legacy_decode_kernel<4, 2, 1><<<grid, dim3(THREADS), lds, st>>>(a); break;
        case 241: legacy_decode_kernel<2, 4, 1><<<grid, dim3(THREADS), lds, st>>>(a); break;
        default: legacy_decode_kernel<2, 2, 1><<<grid, dim3(THREADS), lds, st>>>(a); break;
    }
    return check_launch("hyq_decode_legacy");
}

}  // namespace
}  // namespace hyq

using namespace hyq;

extern "C" size_t hyq_decode_workspace_size(const hyq_decode_params* p) {
    if (validate(p) != HYQ_OK) return 0;
    const Plan pl = plan_for(p);
    return layout(pl, p->bh_kv, p->kv_repeat).total;
}

namespace hyq {
namespace {

// The launch of hyq_decode_hybrid once the workspace is settled (p validated,
// the plan checked against the merge tables, the workspace L.total bytes,
// 256-byte aligned, its counter area zero).
int launch_decode(const hyq_decode_params* p, const Plan& pl, const Layout& L, void* workspace, void* stream) {
    DecArgs a{};
    a.q = p->q; a.q_stride = static_cast<int32_t>(p->q_stride);
    a.out = p->out; a.out_stride = static_cast<int32_t>(p->out_stride);
    a.io = p->dtype_flags;
    a.kp = reinterpret_cast<const uint8_t*>(p->k_packed); a.kp_bh = static_cast<int32_t>(p->kp_stride_bh);
    a.vp = reinterpret_cast<const uint8_t*>(p->v_packed); a.vp_bh = static_cast<int32_t>(p->vp_stride_bh);
    a.ks = p->k_scale; a.ks_bh = static_cast<int32_t>(p->ks_stride_bh);
    a.vs = p->v_scale; a.vs_bh = static_cast<int32_t>(p->vs_stride_bh);
    a.n_quant = static_cast<int32_t>(p->n_quant);
    for (int s = 0; s < 3; ++s) {
        a.sk[s] = p->seg_k[s]; a.sv[s] = p->seg_v[s];
        a.sk_bh[s] = static_cast<int32_t>(p->seg_k_stride_bh[s]);
        a.sv_bh[s] = static_cast<int32_t>(p->seg_v_stride_bh[s]);
        a.sn[s] = static_cast<int32_t>(p->seg_n[s]);
    }
    a.segu[0] = pl.segu[0]; a.segu[1] = pl.segu[1];
    a.G = p->kv_repeat;
    a.bh_kv = p->bh_kv;
    a.qk_scale = p->sm_scale * LOG2E;
    a.nqg = pl.nqg; a.nwg = pl.nwg;
    a.mj = merge_batch(p->kv_repeat, pl.nwg);
    for (int i = 0; i <= pl.nwg; ++i) a.bnd[i] = pl.bnd[i];
    if (pl.ragged) {
        a.sk_bh[1] = pl.cus;
        a.sk_bh[2] = pl.slots;
    }
    char* ws = static_cast<char*>(workspace);
    a.cnt = reinterpret_cast<uint32_t*>(ws + L.cnt);
    a.ml = reinterpret_cast<float*>(ws + L.ml);
    a.part = reinterpret_cast<float*>(ws + L.part);
    a.len_q = p->n_quant > 0 ? p->seq_lens_quant : nullptr;
    a.len_s0 = p->seg_n[0] > 0 ? p->seq_lens_seg0 : nullptr;
    hipStream_t s = static_cast<hipStream_t>(stream);
    // x: KV head, y: piece; workgroups dispatch x-fastest, so piece 0 of
    // every head goes first
    const dim3 grid(static_cast<unsigned>(p->bh_kv), static_cast<unsigned>(pl.ragged ? pl.rows : pl.nwg)), block(THREADS);
    const size_t lds = lds_bytes(p->kv_repeat);
    const int bits = p->n_quant > 0 ? 10 * p->k_bits + p->v_bits : 44;   // no prefix: any instance
    auto launch = [&](auto k, auto v) {
        constexpr int KB = decltype(k)::value, VB = decltype(v)::value;
        if (pl.ragged) decode_kernel<KB, VB, true><<<grid, block, lds, s>>>(a);
        else decode_kernel<KB, VB, false><<<grid, block, lds, s>>>(a);
    };
    constexpr std::integral_constant<int, 2> b2;
    constexpr std::integral_constant<int, 4> b4;
    constexpr std::integral_constant<int, 8> b8;
    switch (bits) {
        case 44: launch(b4, b4); break;
        case 42: launch(b4, b2); break;
        case 48: launch(b4, b8); break;
        case 24: launch(b2, b4); break;
        case 22: launch(b2, b2); break;
        case 28: launch(b2, b8); break;
        case 84: launch(b8, b4); break;
        case 82: launch(b8, b2); break;
        default: launch(b8, b8); break;
    }
    return check_launch("hyq_decode_hybrid");
}

// validation, plan and layout shared by both decode entry points
int prepare(const hyq_decode_params* p, Plan& pl, Layout& L) {
    int rc = validate(p);
    if (rc != HYQ_OK) return rc;
    if (p->bh_kv == 0) return HYQ_OK;
    pl = plan_for(p);
    if (pl.nwg == 0) return fail(HYQ_EINVAL, "decode with zero key tokens");
    if (static_cast<int64_t>(pl.nwg) * p->kv_repeat > MAX_PARTIALS || pl.nwg > MAX_NWG)
        return fail(HYQ_ENOTSUP, "too many pieces per head for the merge tables");
    L = layout(pl, p->bh_kv, p->kv_repeat);
    return HYQ_OK;
}

// A ragged call whose workspace is too small for the device's plan, but sized
// for the padded lengths, runs by those.
void fit_plan(const hyq_decode_params* p, size_t bytes, Plan& pl, Layout& L) {
    if (bytes >= L.total || pl.rows == 0) return;
    const Plan padded = plan_for(p, false);
    const Layout PL = layout(padded, p->bh_kv, p->kv_repeat);
    if (PL.total > bytes) return;
    pl = padded;
    L = PL;
}

// ---------------------------------------------------------------------------
// allocation-free variant: the workspace is a file-scope device array
// ---------------------------------------------------------------------------
constexpr size_t SCRATCH_BYTES = 16u << 20;     // counters (2 MiB) + (m, l) table and partials
static __device__ __align__(256) uint8_t scratch[SCRATCH_BYTES];

__global__ void clear_words_kernel(uint32_t* __restrict__ p, int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// This device's address of `scratch`, looked up once per device with that
// device current; the first lookup also clears the counter area on `stream`
// (a fill kernel, so that a captured first call records no memset node).
// Every completed decode launch leaves the counters at zero again.
int scratch_for_current_device(hipStream_t stream, void** out) {
    static std::mutex mu;
    static void* ptrs[64] = {nullptr};
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
        return fail(HYQ_EDEVICE, "hyq_decode_hybrid_noalloc: no current HIP device");
    std::lock_guard<std::mutex> lock(mu);
    if (ptrs[dev] == nullptr) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || ptr == nullptr)
            return fail(HYQ_EDEVICE, std::string("hyq_decode_hybrid_noalloc: hipGetSymbolAddress failed: ") +
                                         hipGetErrorString(e));
        const int64_t words = static_cast<int64_t>(CNT_CAP) * CNT_PAD;
        clear_words_kernel<<<dim3(static_cast<unsigned>((words + 255) / 256)), dim3(256), 0, stream>>>(
            static_cast<uint32_t*>(ptr), words);
        if (int rc = check_launch("hyq_decode_hybrid_noalloc (clear)")) return rc;
        ptrs[dev] = ptr;
    }
    *out = ptrs[dev];
    return HYQ_OK;
}

}  // namespace
}  // namespace hyq

extern "C" int hyq_decode_hybrid(const hyq_decode_params* p, void* workspace, size_t ws_bytes, void* stream) {
    Plan pl{};
    Layout L{};
    int rc = prepare(p, pl, L);
    if (rc != HYQ_OK || p->bh_kv == 0) return rc;
    fit_plan(p, ws_bytes, pl, L);
    if (!workspace || ws_bytes < L.total || !aligned(workspace, 256))
        return fail(HYQ_ENOSPC, "decode workspace too small or misaligned: need " + std::to_string(L.total) + " bytes");
    return launch_decode(p, pl, L, workspace, stream);
}

extern "C" int hyq_decode_hybrid_noalloc(const hyq_decode_params* p, void* stream) {
    Plan pl{};
    Layout L{};
    int rc = prepare(p, pl, L);
    if (rc != HYQ_OK || p->bh_kv == 0) return rc;
    fit_plan(p, SCRATCH_BYTES, pl, L);
    if (L.total > SCRATCH_BYTES)
        return fail(HYQ_ENOSPC, "hyq_decode_hybrid_noalloc: the call needs " + std::to_string(L.total) +
                                    " bytes of workspace, above the " + std::to_string(SCRATCH_BYTES) +
                                    "-byte scratch; use hyq_decode_hybrid");
    void* ws = nullptr;
    rc = scratch_for_current_device(static_cast<hipStream_t>(stream), &ws);
    if (rc != HYQ_OK) return rc;
    return launch_decode(p, pl, L, ws, stream);
}

#ifdef HYQ_PHASE_TRACE
// Copies the trace ring (TRACE_SLOTS x 4 TRACE_MAX_WG x TRACE_PH uint64) and
// the number of launches recorded to the host; trace build only.
extern "C" int hyq_phase_trace_read(uint64_t* dst, size_t bytes, uint32_t* launches) {
    const size_t need = sizeof(uint64_t) * TRACE_SLOTS * TRACE_MAX_WG * 4 * TRACE_PH;
    if (bytes < need) return fail(HYQ_ENOSPC, "phase trace buffer too small");
    if (hipDeviceSynchronize() != hipSuccess ||
        hipMemcpyFromSymbol(dst, HIP_SYMBOL(g_trace), need) != hipSuccess ||
        hipMemcpyFromSymbol(launches, HIP_SYMBOL(g_trace_launch), sizeof(uint32_t)) != hipSuccess)
        return fail(HYQ_EDEVICE, "phase trace copy failed");
    return HYQ_OK;
}
extern "C" int hyq_phase_trace_geometry(int32_t* slots, int32_t* max_wg, int32_t* phases) {
    *slots = TRACE_SLOTS; *max_wg = TRACE_MAX_WG * 4; *phases = TRACE_PH;
    return HYQ_OK;
}
#endif

extern "C" size_t hyq_decode_bf16_workspace_size(int32_t bh_kv, int32_t kv_repeat, int64_t n, int32_t d) {
    if (bh_kv < 0 || kv_repeat < 1 || kv_repeat > 16 || d != D || n < 0) return 0;
    const int64_t seg_n[3] = {n, 0, 0};
    const Plan pl = make_plan(group_units(0, 4, 4), seg_n, bh_kv, kv_repeat, 0, resident_slots(4, 4, kv_repeat));
    return layout(pl, bh_kv, kv_repeat).total;
}

extern "C" int hyq_decode_bf16(const uint16_t* q, int64_t q_stride, uint16_t* out, int64_t out_stride,
                               const uint16_t* k, int64_t k_stride_bh, int64_t k_stride_n,
                               const uint16_t* v, int64_t v_stride_bh, int64_t v_stride_n,
                               int64_t n, int32_t bh_kv, int32_t kv_repeat, int32_t d, float sm_scale,
                               void* workspace, size_t workspace_bytes, void* stream) {
    hyq_decode_params p{};
    p.q = q; p.q_stride = q_stride; p.out = out; p.out_stride = out_stride;
    p.seg_k[0] = k; p.seg_k_stride_bh[0] = k_stride_bh; p.seg_k_stride_n[0] = k_stride_n;
    p.seg_v[0] = v; p.seg_v_stride_bh[0] = v_stride_bh; p.seg_v_stride_n[0] = v_stride_n;
    p.seg_n[0] = n;
    p.bh_kv = bh_kv; p.kv_repeat = kv_repeat; p.head_dim = d; p.k_bits = 4; p.v_bits = 4;
    p.sm_scale = sm_scale;
    return hyq_decode_hybrid(&p, workspace, workspace_bytes, stream);
}

extern "C" size_t hyq_decode_legacy_workspace_size(const hyq_legacy_params* p) {
    if (validate_legacy(p) != HYQ_OK || p->bh_kv == 0) return 0;
    return layout(legacy_plan(p), p->bh_kv, p->kv_repeat).total;
}

extern "C" int hyq_decode_legacy(const hyq_legacy_params* p, void* workspace, size_t ws_bytes, void* stream) {
    int rc = validate_legacy(p);
    if (rc != HYQ_OK || p->bh_kv == 0) return rc;
    const Plan pl = legacy_plan(p);
    const Layout L = layout(pl, p->bh_kv, p->kv_repeat);
    if (!workspace || ws_bytes < L.total || !aligned(workspace, 256))
        return fail(HYQ_ENOSPC, "hyq_decode_legacy: workspace too small or misaligned: need " + std::to_string(L.total) + " bytes");
    return launch_legacy(p, pl, L, workspace, stream);
}
