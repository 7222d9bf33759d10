// Reference-order GEMV: bit-identical to the reference's golden for every ggml type.
//
// Contract (tools/q4k_ref.py:67-92, RTL order src/glm_matmul_q4k.v:261-270): for each
// output (m, n) the weight row is dequantised exactly and
//     acc = f32(acc + f32(x[m][k] * w[n][k]))     for k = 0 .. K-1, in order,
// then y = bf16_RNE(acc).  The library is compiled with -ffp-contract=off, so the multiply and
// the add are two separately rounded ops.
//
// What bounds it: the K dependent adds of one output.  They cannot be split or reordered, and a
// dependent v_add_f32 takes 8.3 cycles on this part (measured), 21 us for K = 6144 at 2.4 GHz.
// A workgroup has chain waves, whose lanes own one output (m, row) each and add its products in
// k order, and four producer waves that dequantise for them: a producer lane takes a run (16
// consecutive weights of one row) and writes to LDS, four consecutive k per 16-B slot, neighbouring
// rows in neighbouring slots.  What it writes depends on what is scarce:
//   * One or two activation rows: the products x * w, so that the chain is a read and four adds per
//     four k (the reads hide behind the adds' latency).
//   * More: the weights, with the stage's activations as fp32 beside them, and the chain multiplies,
//     so that the producers convert and write each weight once.
// Stages of KS values of k go through a ring of three LDS buffers with one workgroup barrier per
// stage: in interval t the producers write stage t and the chains add stage t - 2, reading ahead
// into stage t - 1, which is complete already.
// Measured (Q4_K, 6144 x 6144), one wave per 64 rows doing everything -> here: M = 1 / 2 / 4 / 8
// 79 / 111 / 166 / 167 -> 23 / 26 / 39 / 39 us; the other types within a few us of these.  At many rows the chain
// is not what binds, and that one wave is the faster one (k_gemv_ref_wave, ref_wave_wins).
// Any K (the last stage may be partial), any 2-byte aligned pointers (unaligned 16-B loads).
#include "common.hpp"
#include "launch.hpp"

namespace aipu {

namespace {

constexpr int kRows = 64;      // rows per workgroup of the fp32-weight kernel (one wave)
constexpr int kMC = 8;         // activation rows per pass (blockIdx.y walks the rest)
constexpr int kStageW = 256;   // weights per stage of the fp32-weight kernel

// ---------------------------------------------------------------- runs of 16 weights
// 16 bytes at any 2-byte aligned address (global memory takes unaligned 16-B loads).
typedef uint32_t u32x4_u2 __attribute__((ext_vector_type(4), aligned(2)));
__device__ __forceinline__ uint4 load16_u2(const void* p) {
    const u32x4_u2 v = *(const u32x4_u2*)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ uint32_t word_of(const uint4& v, int i) {
    return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w;
}

// Byte B of v as fp32 in one instruction (plain C selects a bit-field extract, then the
// conversion of byte 0).  VALU only, no hazard beyond what the hardware interlocks.
template <int B>
__device__ __forceinline__ float cvt_ubyte(uint32_t v) {
    float r;
    if constexpr (B == 0) asm("v_cvt_f32_ubyte0 %0, %1" : "=v"(r) : "v"(v));
    else if constexpr (B == 1) asm("v_cvt_f32_ubyte1 %0, %1" : "=v"(r) : "v"(v));
    else if constexpr (B == 2) asm("v_cvt_f32_ubyte2 %0, %1" : "=v"(r) : "v"(v));
    else asm("v_cvt_f32_ubyte3 %0, %1" : "=v"(r) : "v"(v));
    return r;
}

// Run r of a row: weights 16 r .. 16 r + 15.  load() fetches its bytes, prepare() its scales,
// four() dequantises weights 4 i .. 4 i + 3 exactly as the reference does.
template <int TYPE>
struct Run;

// Q4_K (tools/q4k_ref.py:45-60): half (r & 1) of sub-block j = r / 2 of super-block r / 16, the
// low (j even) or high nibbles of one 16-B piece.  D = d * sc and D * q are exact in fp32
// (11 + 6 + 4 bits), so f32(f32(D * q) - Mn) is one fused multiply-add; the nibbles enter it as
// fp16 subnormals (q * 2^-24 low, 16 q * 2^-24 high), which the scale undoes exactly.
template <>
struct Run<T_Q4_K> {
    uint4 h, q;
    __device__ __forceinline__ void load(const uint8_t* row, int r) {
        const uint8_t* b = row + (int64_t)(r >> 4) * 144;
        h = load16_u2(b);
        q = load16_u2(b + 16 + 32 * ((r & 15) >> 2) + 16 * (r & 1));
    }
    struct Scale {
        float s, n;      // scaled D, -Mn
        uint32_t mask;   // of two nibbles
    };
    __device__ __forceinline__ Scale prepare(int r) const {
        const int j = (r & 15) >> 1, sh = 8 * (j & 3);
        const uint32_t a0 = h.y >> sh, a1 = h.z >> sh, a2 = h.w >> sh;
        const uint32_t hi = 0u - (uint32_t)(j >> 2);   // all ones for sub-blocks 4 .. 7
        const uint32_t sc = (a0 & 63u & ~hi) | (((a2 & 15u) | ((a0 >> 2) & 0x30u)) & hi);
        const uint32_t mn = (a1 & 63u & ~hi) | ((((a2 >> 4) & 15u) | ((a1 >> 2) & 0x30u)) & hi);
        Scale s;
        s.s = f16_to_f32(h.x & 0xFFFFu) * cvt_ubyte<0>(sc) * ((j & 1) ? 0x1p20f : 0x1p24f);
        s.n = -(f16_to_f32(h.x >> 16) * cvt_ubyte<0>(mn));
        s.mask = (j & 1) ? 0x00F000F0u : 0x000F000Fu;
        return s;
    }
    __device__ __forceinline__ void four(const Scale& s, int i, float (&w)[4]) const {
        typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
        const uint32_t x = word_of(q, i);
        const h2_t a = __builtin_bit_cast(h2_t, x & s.mask), b = __builtin_bit_cast(h2_t, (x >> 8) & s.mask);
        w[0] = __builtin_fmaf((float)a[0], s.s, s.n);
        w[1] = __builtin_fmaf((float)b[0], s.s, s.n);
        w[2] = __builtin_fmaf((float)a[1], s.s, s.n);
        w[3] = __builtin_fmaf((float)b[1], s.s, s.n);
    }
};

// Q6_K (tools/q4k_ref.py:105-124): one scale per run.
template <>
struct Run<T_Q6_K> {
    uint4 ql, qh;
    uint32_t sc, d;
    __device__ __forceinline__ void load(const uint8_t* row, int r) {
        const uint8_t* b = row + (int64_t)(r >> 4) * 210;
        const int hf = (r & 15) >> 3, t = (r >> 1) & 3, o = 16 * (r & 1);
        ql = load16_u2(b + 64 * hf + 32 * (t & 1) + o);
        qh = load16_u2(b + 128 + 32 * hf + o);
        sc = b[192 + (r & 15)];
        d = *(const uint16_t*)(b + 208);
    }
    struct Scale {
        float ds;
        int sl, sh;   // shifts of the nibble and of the two high bits
    };
    __device__ __forceinline__ Scale prepare(int r) const {
        const int t = (r >> 1) & 3;
        return Scale{f16_to_f32(d) * (float)(int8_t)(uint8_t)sc, 4 * (t >> 1), 2 * t};
    }
    __device__ __forceinline__ void four(const Scale& s, int i, float (&w)[4]) const {
        const uint32_t code = ((word_of(ql, i) >> s.sl) & 0x0F0F0F0Fu) | (((word_of(qh, i) >> s.sh) & 0x03030303u) << 4);
        w[0] = s.ds * (cvt_ubyte<0>(code) - 32.0f);
        w[1] = s.ds * (cvt_ubyte<1>(code) - 32.0f);
        w[2] = s.ds * (cvt_ubyte<2>(code) - 32.0f);
        w[3] = s.ds * (cvt_ubyte<3>(code) - 32.0f);
    }
};

// Q8_0: half (r & 1) of block r / 2 (fp16 d, 32 signed bytes; tools/q4k_ref.py:126-129).
template <>
struct Run<T_Q8_0> {
    uint4 q;
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t* row, int r) {
        const uint8_t* b = row + (int64_t)(r >> 1) * 34;
        d = *(const uint16_t*)b;
        q = load16_u2(b + 2 + 16 * (r & 1));
    }
    struct Scale {
        float d;
    };
    __device__ __forceinline__ Scale prepare(int) const { return Scale{f16_to_f32(d)}; }
    __device__ __forceinline__ void four(const Scale& s, int i, float (&w)[4]) const {
        const uint32_t x = word_of(q, i);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = s.d * (float)(int8_t)(uint8_t)(x >> (8 * e));
    }
};

template <int TYPE>
struct RunHalf {   // F16 / BF16
    uint4 v[2];
    __device__ __forceinline__ void load(const uint8_t* row, int r) {
        v[0] = load16_u2(row + (int64_t)r * 32);
        v[1] = load16_u2(row + (int64_t)r * 32 + 16);
    }
    struct Scale {};
    __device__ __forceinline__ Scale prepare(int) const { return Scale{}; }
    __device__ __forceinline__ void four(const Scale&, int i, float (&w)[4]) const {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t hw = (word_of(v[i >> 1], 2 * (i & 1) + (e >> 1)) >> (16 * (e & 1))) & 0xFFFFu;
            w[e] = TYPE == T_F16 ? f16_to_f32(hw) : bf16_to_f32(hw);
        }
    }
};
template <>
struct Run<T_F16> : RunHalf<T_F16> {};
template <>
struct Run<T_BF16> : RunHalf<T_BF16> {};

// ---------------------------------------------------------------- one workgroup
// RM: row capacity of a workgroup, MC: activation rows.  RM = 32 while that leaves every CU at
// most one workgroup (a half-empty chain wave costs nothing there), RM = 64 beyond, where the
// workgroups of a CU share its VALU (N = 16384, K = 6144: 37 us; one row's chain alone 24 us).
template <int MC, int RM>
struct RefCfg {
    static constexpr bool kMul = MC > 2;              // the chains multiply; else the producers do
    static constexpr int NBUF = 3;
    static constexpr int G = kMul ? 1 : MC;           // activation rows a producer lane multiplies with
    static constexpr int RW = RM / 4;                 // rows per producer wave
    static constexpr int RPS = 64 / RW;               // runs per stage
    static constexpr int KS = 16 * RPS;
    static constexpr int L = kMul ? RM : MC * RM;     // 16-B slots per four k
    static constexpr int kXBytes = kMul ? MC * KS * 4 : 0;
    static constexpr int kStageBytes = KS / 4 * L * 16 + kXBytes;
    static constexpr int kChains = MC * RM <= 64 ? 1 : MC * RM / 64;
    static constexpr int kThreads = 64 * (4 + kChains);
    static constexpr int kLds = NBUF * kStageBytes;
    static_assert(MC * KS <= 1024 && kLds <= 96 * 1024, "a stage must split over the producer lanes");
};

// A workgroup barrier that waits for this wave's LDS writes and nothing else: global loads for
// later stages stay in flight.
__device__ __forceinline__ void stage_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int TYPE, int G, bool MUL>
struct Held {   // one stage's operands of a producer lane
    Run<TYPE> w;
    uint4 x[G][2];   // !MUL: the run's activations
    uint2 xs;        // MUL: four activations to stage
};

typedef uint32_t u32x2_u2 __attribute__((ext_vector_type(2), aligned(2)));

// Rows [row0, row0 + R) of W [N][K] against activation rows X [mcnt][K]; y[m * ys + row].
// R <= RM, a multiple of 8; rows at or past N and activation rows at or past mcnt repeat the
// last one and are not stored.
template <int TYPE, int MC, int RM>
__device__ __forceinline__ void ref_rows(const uint8_t* __restrict__ W, int64_t N, int64_t K,
                                         const uint16_t* __restrict__ X, int mcnt, uint16_t* __restrict__ Y,
                                         float* __restrict__ Yf, int64_t ys, int64_t row0, int R, uint8_t* lds) {
    typedef RefCfg<MC, RM> C;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int S = (int)((K + C::KS - 1) / C::KS);
    constexpr int LA = C::NBUF - 1;                       // stages between the producers and the chains
    constexpr int kWBytes = C::kStageBytes - C::kXBytes;   // the stage's activations follow its slots

    if (wave >= C::kChains) {   // producer: rows RW * pw .. of the workgroup
        const int pw = wave - C::kChains;
        const int un = lane / C::RW;   // run of the stage
        const int row = pw * C::RW + lane % C::RW;
        const int64_t n = row0 + row < N ? row0 + row : N - 1;
        const uint8_t* wr = W + n * row_bytes(TYPE, K);
        const uint16_t* xr[C::G];
#pragma unroll
        for (int g = 0; g < C::G; ++g) xr[g] = X + (int64_t)(g < mcnt ? g : mcnt - 1) * K;
        // MUL: the four activations of the stage this lane stages: row xm, k xk .. xk + 3
        const int xi = pw * 64 + lane, xm = xi / (C::KS / 4), xk = 4 * (xi % (C::KS / 4));
        const uint16_t* xsr = X + (int64_t)(xm < mcnt ? xm : mcnt - 1) * K;
        const bool stager = C::kMul && xm < MC;
        const bool busy = pw * C::RW < R;   // wave-uniform: a wave past the last row only stages
        const int nr = (int)(K / 16);       // whole runs
        // stage t's operands; runs past the last whole one repeat it (their products are not
        // read, or come from the partial path below)
        // (16 r fits 32 bits: with one or two activation rows K < 2^31, see kMaxProductK)
        auto fetch = [&](Held<TYPE, C::G, C::kMul>& b, int t) {
            int r = t * C::RPS + un;
            r = r < nr ? r : nr - 1;
            b.w.load(wr, r);
            if constexpr (C::kMul) {
                const int64_t k = (int64_t)t * C::KS + xk;
                const u32x2_u2 v = *(const u32x2_u2*)(xsr + (k + 4 <= K ? k : K - 4));
                b.xs = make_uint2(v.x, v.y);
            } else {
#pragma unroll
                for (int g = 0; g < C::G; ++g) {
                    b.x[g][0] = load16_u2(xr[g] + 16 * r);
                    b.x[g][1] = load16_u2(xr[g] + 16 * r + 8);
                }
            }
        };
        auto slot = [&](int buf, int k4, int g) { return lds + buf * C::kStageBytes + (k4 * C::L + g * RM + row) * 16; };
        auto xslot = [&](int buf) { return (float*)(lds + buf * C::kStageBytes + kWBytes) + xm * C::KS + xk; };
        // this lane's run of stage t: its products, or its weights and the activations
        auto emit = [&](const Held<TYPE, C::G, C::kMul>& b, int t, int buf) {
            if (C::kMul && stager)
                *(float4*)xslot(buf) = make_float4(bf16_to_f32(b.xs.x & 0xFFFFu), __uint_as_float(b.xs.x & 0xFFFF0000u),
                                                   bf16_to_f32(b.xs.y & 0xFFFFu), __uint_as_float(b.xs.y & 0xFFFF0000u));
            if (!busy) return;
            const auto sc = b.w.prepare(t * C::RPS + un);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float w[4];
                b.w.four(sc, i, w);
                if constexpr (C::kMul) {
                    *(float4*)slot(buf, 4 * un + i, 0) = make_float4(w[0], w[1], w[2], w[3]);
                } else {
#pragma unroll
                    for (int g = 0; g < C::G; ++g) {
                        const uint4& xv = b.x[g][i >> 1];
                        const uint32_t x0 = word_of(xv, 2 * (i & 1)), x1 = word_of(xv, 2 * (i & 1) + 1);
                        float4 p;
                        p.x = bf16_to_f32(x0 & 0xFFFFu) * w[0];
                        p.y = __uint_as_float(x0 & 0xFFFF0000u) * w[1];
                        p.z = bf16_to_f32(x1 & 0xFFFFu) * w[2];
                        p.w = __uint_as_float(x1 & 0xFFFF0000u) * w[3];
                        *(float4*)slot(buf, 4 * un + i, g) = p;
                    }
                }
            }
        };
        // the last stage of a K that is not a multiple of 16 (F16 / BF16, any K): the last run and
        // the activations that go with it, one element at a time
        auto emit_partial = [&](int buf) {
            if constexpr (TYPE == T_F16 || TYPE == T_BF16) {
                const int kt = (int)(K % 16);
                if (kt == 0) return;
                const int64_t k0 = 16 * (int64_t)nr;
                if constexpr (C::kMul) {
                    const int64_t k = (int64_t)(S - 1) * C::KS + xk;
                    if (stager && k < K && (k + 4 > K || nr == 0))
                        for (int e = 0; e < 4; ++e) xslot(buf)[e] = k + e < K ? bf16_to_f32(xsr[k + e]) : 0.0f;
                }
                if ((S - 1) * C::RPS + un == nr) {
                    for (int k = 0; k < kt; ++k) {
                        const uint32_t hw = *(const uint16_t*)(wr + 2 * (k0 + k));
                        const float w = TYPE == T_F16 ? f16_to_f32(hw) : bf16_to_f32(hw);
#pragma unroll
                        for (int g = 0; g < C::G; ++g)
                            ((float*)slot(buf, 4 * un + (k >> 2), g))[k & 3] = C::kMul ? w : bf16_to_f32(xr[g][k0 + k]) * w;
                    }
                }
            }
        };
        if (nr) {
            // NBUF stages of loads in flight, so that every buffer index is a constant; the loop has
            // no branch between a load and its use, so each wait is for the oldest stage's loads only
            Held<TYPE, C::G, C::kMul> held[C::NBUF];
#pragma unroll
            for (int j = 0; j < C::NBUF; ++j) fetch(held[j], j);
            int t = 0;
            for (; t + C::NBUF < S; t += C::NBUF) {
#pragma unroll
                for (int j = 0; j < C::NBUF; ++j) {
                    emit(held[j], t + j, j);
                    fetch(held[j], t + j + C::NBUF);
                    stage_barrier();
                }
            }
#pragma unroll
            for (int j = 0; j < C::NBUF; ++j) {
                if (t + j < S) {
                    emit(held[j], t + j, j);
                    if (t + j == S - 1) emit_partial(j);
                    stage_barrier();
                }
            }
        } else {
            emit_partial(0);
            stage_barrier();
        }
#pragma unroll
        for (int t = 0; t < LA; ++t) stage_barrier();
        return;
    }

    // chain: lane = (activation row, row)
    __builtin_amdgcn_s_setprio(3);
    const int li = wave * 64 + lane;
    const int m = li / RM, row = li % RM;
    const bool live = row < R && m < mcnt && row0 + row < N;
    // The chain issues a group of GR reads at once and waits once per group: a wait before every
    // read's four adds cost 1.5 cycles per k (M = 1: 32 -> 25.5 us at 6144 x 6144).
    constexpr int GR = 4, D = 2 * GR, kReads = C::kMul ? 2 : 1;
    constexpr int NK4 = C::KS / 4;
    static_assert(NK4 % D == 0, "the read ring must start every stage at q[0]");
    const uint8_t* const base = lds + (C::kMul ? row : li) * 16;
    const uint8_t* const xbase = lds + kWBytes + m * (C::KS * 4);
    float acc = 0.0f;
#pragma unroll
    for (int t = 0; t < LA; ++t) stage_barrier();
    float4 q[D], xq[D];
    // reads j .. j + GR - 1 of the stage at offset oc, which runs on into the stage at offset on
    auto read_group = [&](int j0, int oc, int on) {
#pragma unroll
        for (int e = 0; e < GR; ++e) {
            const int j = j0 + e;
            q[j % D] = *(const float4*)(base + (j < NK4 ? oc + j * C::L * 16 : on + (j - NK4) * C::L * 16));
            if (C::kMul) xq[j % D] = *(const float4*)(xbase + (j < NK4 ? oc + j * 16 : on + (j - NK4) * 16));
        }
    };
    if (live) read_group(0, 0, 0);
    int cur = 0;
    for (int s = 0; s < S; ++s) {
        const int nxt = cur + 1 == C::NBUF ? 0 : cur + 1;
        const int oc = cur * C::kStageBytes, on = nxt * C::kStageBytes;
        if (live) {   // lanes without an output read nothing; every wave meets every barrier
            if (s < S - 1 || K % C::KS == 0) {
#pragma unroll
                for (int i = 0; i < NK4; ++i) {
                    if (i % GR == 0) {   // the group after next, then one wait for all of this group
                        read_group(i + D - GR, oc, on);
                        __builtin_amdgcn_s_waitcnt(0xC07F | (kReads * (D - GR)) << 8);   // lgkmcnt
                    }
                    float4 v = q[i % D];
                    if constexpr (C::kMul) {
                        const float4 x = xq[i % D];
                        v.x = x.x * v.x;
                        v.y = x.y * v.y;
                        v.z = x.z * v.z;
                        v.w = x.w * v.w;
                    }
                    acc = acc + v.x;
                    acc = acc + v.y;
                    acc = acc + v.z;
                    acc = acc + v.w;
                    __builtin_amdgcn_sched_barrier(0);   // the chain's order of issue is the plan
                }
            } else {   // the partial last stage
                const int kn = (int)(K - (int64_t)s * C::KS);
                for (int k = 0; k < kn; ++k) {
                    float p = ((const float*)(base + oc + (k >> 2) * C::L * 16))[k & 3];
                    if constexpr (C::kMul) p = ((const float*)(xbase + oc))[k] * p;
                    acc = acc + p;
                }
            }
        }
        asm volatile("s_barrier" ::: "memory");
        cur = nxt;
    }
    if (live) {
        Y[(int64_t)m * ys + row0 + row] = (uint16_t)bf16_rne(acc);
        if (Yf) Yf[(int64_t)m * ys + row0 + row] = acc;
    }
}

// ---------------------------------------------------------------- one wave per 64 rows
// At many rows the chain is not what binds: workgroups of ref_rows share a CU's VALU and LDS, and a
// product costs there a second conversion of the activations and 4 bytes written and read.  Here one
// wave owns 64 rows and does everything: lane = row, a unit of the row's weights in registers, loaded
// one unit ahead, the activations as fp32 in LDS, converted once for the 64 rows.  About five VALU
// operations per weight and one more pair per further activation row; slower alone (6144 x 6144:
// 79 us against 23) and faster once it fills the chip.  A unit is 256 weights (Q4_K: 9 16-B pieces;
// Q6_K: the 53 dwords that span a 210-B block, which starts 4-B aligned or 2 bytes past) or 64 (Q8_0:
// 17 dwords; F16 / BF16: 8 16-B pieces).
constexpr int kWaveChunk = 256;   // activations staged at a time

// A unit: load() fetches it, each() calls f(c, weight) for its weights 4 c .. 4 c + 3 in order, weight(e)
// dequantising weight 4 c + e exactly as the reference does.
template <int TYPE>
struct Unit;

template <>
struct Unit<T_Q4_K> {
    static constexpr int kW = 256, kBytes = 144;
    uint4 r[9];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t wr, uint32_t o) {
#pragma unroll
        for (int i = 0; i < 9; ++i) r[i] = buf_load16(wr, o + 16u * (uint32_t)i);
    }
    template <class F>
    __device__ __forceinline__ void each(uint32_t, F f) const {
        const float d = f16_to_f32(r[0].x & 0xFFFFu), dm = f16_to_f32(r[0].x >> 16);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            uint32_t sc, mn;
            q4k_scale_min(j, r[0].y, r[0].z, r[0].w, sc, mn);
            const float D = d * (float)sc, Mn = dm * (float)mn;
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const uint32_t x = word_of(r[1 + 2 * (j >> 1) + (c >> 2)], c & 3);
                const uint32_t v = ((j & 1) ? x >> 4 : x) & 0x0F0F0F0Fu;
                const float q[4] = {cvt_ubyte<0>(v), cvt_ubyte<1>(v), cvt_ubyte<2>(v), cvt_ubyte<3>(v)};
                f(8 * j + c, [&](int e) { return __builtin_fmaf(D, q[e], -Mn); });   // D * q is exact
            }
        }
    }
};

template <>
struct Unit<T_Q6_K> {
    static constexpr int kW = 256, kBytes = 210;
    uint32_t r[53];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t wr, uint32_t o) {   // o: the dword the block starts in
#pragma unroll
        for (int i = 0; i < 53; ++i) r[i] = buf_load4(wr, o + 4u * (uint32_t)i);
    }
    template <class F>
    __device__ __forceinline__ void each(uint32_t par, F f) const {   // the block starts par (0 or 2) bytes into r[0]
        const auto dw = [&](int o) { return __builtin_amdgcn_alignbyte(r[(o >> 2) + 1], r[o >> 2], par); };
        const float d = f16_to_f32(par ? r[52] >> 16 : r[52] & 0xFFFFu);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                __builtin_amdgcn_sched_barrier(0);   // one run of 32 weights at a time (registers)
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    const uint32_t ql = dw(64 * h + 32 * (t & 1) + 4 * c), qh = dw(128 + 32 * h + 4 * c);
                    const uint32_t code = ((t < 2 ? ql : ql >> 4) & 0x0F0F0F0Fu) | (((qh >> (2 * t)) & 0x03030303u) << 4);
                    const int si = 8 * h + 2 * t + (c >> 2);
                    const float ds = d * (float)(int8_t)(uint8_t)(dw(192 + (si & ~3)) >> (8 * (si & 3)));
                    const float q[4] = {cvt_ubyte<0>(code), cvt_ubyte<1>(code), cvt_ubyte<2>(code), cvt_ubyte<3>(code)};
                    f(32 * h + 8 * t + c, [&](int e) { return ds * (q[e] - 32.0f); });
                }
            }
    }
};

template <>
struct Unit<T_Q8_0> {
    static constexpr int kW = 64, kBytes = 68;
    uint32_t r[17];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t wr, uint32_t o) {
#pragma unroll
        for (int i = 0; i < 17; ++i) r[i] = buf_load4(wr, o + 4u * (uint32_t)i);
    }
    template <class F>
    __device__ __forceinline__ void each(uint32_t, F f) const {
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const float d = f16_to_f32(c < 8 ? r[0] & 0xFFFFu : r[8] >> 16);
            f(c, [&](int e) {
                const int b = (c < 8 ? 2 : 4) + 4 * c + e;   // byte of the unit: 2 of each block's d lie before it
                return d * (float)(int8_t)(uint8_t)(r[b >> 2] >> (8 * (b & 3)));
            });
        }
    }
};

template <int TYPE>
struct UnitHalf {   // F16 / BF16
    static constexpr int kW = 64, kBytes = 128;
    uint4 r[8];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t wr, uint32_t o) {
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = buf_load16(wr, o + 16u * (uint32_t)i);
    }
    template <class F>
    __device__ __forceinline__ void each(uint32_t, F f) const {
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            f(c, [&](int e) {
                const uint32_t h = word_of(r[c >> 1], 2 * (c & 1) + (e >> 1)) >> (16 * (e & 1)) & 0xFFFFu;
                return TYPE == T_F16 ? f16_to_f32(h) : bf16_to_f32(h);
            });
        }
    }
};
template <>
struct Unit<T_F16> : UnitHalf<T_F16> {};
template <>
struct Unit<T_BF16> : UnitHalf<T_BF16> {};

// Rows [row0, row0 + 64) of W [N][K] against activation rows X [mcnt][K], K a multiple of 64;
// y[m * ys + row].  s_x: [2][MC][kWaveChunk].
template <int TYPE, int MC>
__device__ __forceinline__ void ref_wave(const uint8_t* __restrict__ W, int64_t N, int64_t K,
                                         const uint16_t* __restrict__ X, int mcnt, uint16_t* __restrict__ Y,
                                         float* __restrict__ Yf, int64_t ys, int64_t row0, float* s_x) {
    typedef Unit<TYPE> U;
    constexpr int kPer = kWaveChunk / U::kW;   // units per chunk
    const int lane = threadIdx.x;
    const int nu = (int)(K / U::kW), nch = (nu + kPer - 1) / kPer;
    const uint32_t rb = (uint32_t)row_bytes(TYPE, K);
    const int nrows = (int)(N - row0 < 64 ? N - row0 : 64);
    const __amdgpu_buffer_rsrc_t wr = buf_rsrc(W + row0 * (int64_t)rb, (uint32_t)nrows * rb);   // rows past N read zeros
    const uint32_t wrow = (uint32_t)lane * rb;
    const auto load = [&](U& u, int i) {   // Q6_K: the dwords that span the block (the last may reach past the row)
        const uint32_t o = (uint32_t)U::kBytes * (uint32_t)i;
        u.load(wr, wrow + (TYPE == T_Q6_K ? o & ~3u : o));
    };
    // a chunk's activations: four per lane and row, past K the last ones (not used)
    uint2 xv[MC];
    const uint16_t* xr[MC];
#pragma unroll
    for (int m = 0; m < MC; ++m) xr[m] = X + (int64_t)(m < mcnt ? m : mcnt - 1) * K;
    const auto fetch = [&](int c) {
        int64_t k = (int64_t)c * kWaveChunk + 4 * lane;
        k = k + 4 <= K ? k : K - 4;
#pragma unroll
        for (int m = 0; m < MC; ++m) xv[m] = *(const uint2*)(xr[m] + k);
    };
    const auto stage = [&](int buf) {
#pragma unroll
        for (int m = 0; m < MC; ++m)
            *(float4*)(s_x + (buf * MC + m) * kWaveChunk + 4 * lane) =
                make_float4(bf16_to_f32(xv[m].x & 0xFFFFu), __uint_as_float(xv[m].x & 0xFFFF0000u),
                            bf16_to_f32(xv[m].y & 0xFFFFu), __uint_as_float(xv[m].y & 0xFFFF0000u));
    };
    float acc[MC];
#pragma unroll
    for (int m = 0; m < MC; ++m) acc[m] = 0.0f;
    U cur, nxt;
    fetch(0);
    load(nxt, 0);
    stage(0);
    fetch(1);
    int i = 0;
    for (int c = 0; c < nch; ++c) {
        // the next chunk (past K: repeated values) goes to the other buffer before this one is used: no wait
        // between chunks, and no barrier for one wave, whose LDS accesses are in order; a branch around
        // the last chunk's staging cost up to 6 %
        stage((c + 1) & 1);
        fetch(c + 2);
        __builtin_amdgcn_wave_barrier();
        const float* xb = s_x + (c & 1) * (MC * kWaveChunk);
        const int n = kPer == 1 ? 1 : nu - i < kPer ? nu - i : kPer;
        for (int u = 0; u < n; ++u, ++i) {
            cur = nxt;
            if (i + 1 < nu) load(nxt, i + 1);
            const float* xu = xb + u * U::kW;
            cur.each(((uint32_t)U::kBytes * (uint32_t)i) & 3u, [&](int q, auto weight) {
                constexpr bool kFirst = TYPE == T_Q8_0 && MC == 2;   // weights before the reads: 42 -> 38 us (16384 x 2048)
                float wf[4];
                if (kFirst)
#pragma unroll
                    for (int e = 0; e < 4; ++e) wf[e] = weight(e);
                float4 x[MC];
#pragma unroll
                for (int m = 0; m < MC; ++m) x[m] = *(const float4*)(xu + m * kWaveChunk + 4 * q);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float w = kFirst ? wf[e] : weight(e);
#pragma unroll
                    for (int m = 0; m < MC; ++m) {
                        const float p = (e == 0 ? x[m].x : e == 1 ? x[m].y : e == 2 ? x[m].z : x[m].w) * w;
                        acc[m] = acc[m] + p;
                    }
                }
            });
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (lane < nrows)
        for (int m = 0; m < mcnt; ++m) {
            Y[(int64_t)m * ys + row0 + lane] = (uint16_t)bf16_rne(acc[m]);
            if (Yf) Yf[(int64_t)m * ys + row0 + lane] = acc[m];
        }
}

// Slot gathering (MoE): blockIdx.z = slot z reads weight matrix sel[z] of the `_exps`
// stack at W + sel[z]*wstride when z < topk, else W_alt (the shared expert); activations
// and outputs are offset by z*x_zstride / z*y_zstride.  Slots nslots .. 2 nslots - 1 are the same
// slots of a second stack W2 / W2_alt with outputs Y2 (gate and up in one launch: one after the
// other they leave half the chip idle).  Plain GEMV: sel == nullptr, z = 0.
struct RefGather {
    const int32_t* sel;
    int topk;
    int nslots;
    const uint8_t* W2;
    const uint8_t* W2_alt;
    uint16_t* Y2;
    int64_t E;
    int64_t wstride;
    const uint8_t* W_alt;
    int64_t x_zstride;
    int64_t y_zstride;
};

// The slot's pointers.  A macro: through a function's references the kernels lose their __restrict__
// (6144 x 6144 Q4_K, M = 4: 38.6 -> 39.7 us; 2048 x 6144: 39.7 -> 42.9).
#define AIPU_REF_GATHER(ga, W, X, Y, Yf)                     \
    if (ga.sel) {                                            \
        int z = blockIdx.z;                                  \
        const uint8_t* alt = ga.W_alt;                       \
        if (z >= ga.nslots) {                                \
            z -= ga.nslots;                                  \
            W = ga.W2;                                       \
            alt = ga.W2_alt;                                 \
            Y = ga.Y2;                                       \
        }                                                    \
        if (z < ga.topk) {                                   \
            int e = ga.sel[z];                               \
            e = e < 0 ? 0 : (e >= ga.E ? (int)ga.E - 1 : e); \
            W += (int64_t)e * ga.wstride;                    \
        } else {                                             \
            W = alt;                                         \
        }                                                    \
        X += (int64_t)z * ga.x_zstride;                      \
        Y += (int64_t)z * ga.y_zstride;                      \
        if (Yf) Yf += (int64_t)z * ga.y_zstride;             \
    }

template <int TYPE, int MC, int RM>
__global__ __launch_bounds__((RefCfg<MC, RM>::kThreads)) void k_gemv_ref(const uint8_t* __restrict__ W, int64_t N, int64_t K,
                                                                         const uint16_t* __restrict__ X, int64_t M,
                                                                         uint16_t* __restrict__ Y, float* __restrict__ Yf,
                                                                         int64_t ys, int R, RefGather ga) {
    extern __shared__ __align__(16) uint8_t s_ref[];
    AIPU_REF_GATHER(ga, W, X, Y, Yf)
    const int64_t m0 = (int64_t)blockIdx.y * MC;
    const int mcnt = (int)((M - m0) < MC ? (M - m0) : MC);
    ref_rows<TYPE, MC, RM>(W, N, K, X + m0 * K, mcnt, Y + m0 * ys, Yf ? Yf + m0 * ys : nullptr, ys,
                           (int64_t)blockIdx.x * R, R, s_ref);
}

template <int TYPE, int MC>
__global__ __launch_bounds__(64) void k_gemv_ref_wave(const uint8_t* __restrict__ W, int64_t N, int64_t K,
                                                      const uint16_t* __restrict__ X, int64_t M, uint16_t* __restrict__ Y,
                                                      float* __restrict__ Yf, int64_t ys, RefGather ga) {
    __shared__ __align__(16) float s_x[2 * MC * kWaveChunk];
    AIPU_REF_GATHER(ga, W, X, Y, Yf)
    const int64_t m0 = (int64_t)blockIdx.y * MC;
    const int mcnt = (int)((M - m0) < MC ? (M - m0) : MC);
    ref_wave<TYPE, MC>(W, N, K, X + m0 * K, mcnt, Y + m0 * ys, Yf ? Yf + m0 * ys : nullptr, ys, (int64_t)blockIdx.x * 64, s_x);
}

// A tile sequence of mixed types in one launch: workgroup g belongs to the last tile whose wg0 is
// at most g.  The tiles' launches one after the other would each take a whole chain (24 tiles of
// 256 rows, K = 6144, M = 1: 1.82 ms as 24 launches of the earlier kernel, one launch 35 us).
struct RefTile {
    const uint8_t* w;
    int64_t row0, nrows;
    int32_t type, wg0;
};
struct RefTiles {
    RefTile t[AIPU_MAX_TILES];
    int n;
};

template <int MC, int RM>
__global__ __launch_bounds__((RefCfg<MC, RM>::kThreads)) void k_gemv_ref_tiles(RefTiles a, int64_t K,
                                                                               const uint16_t* __restrict__ X, int64_t M,
                                                                               uint16_t* __restrict__ Y,
                                                                               float* __restrict__ Yf, int64_t ys, int R) {
    extern __shared__ __align__(16) uint8_t s_ref[];
    const int g = blockIdx.x;
    int t = 0;
    while (t + 1 < a.n && a.t[t + 1].wg0 <= g) ++t;
    const RefTile T = a.t[t];
    const int64_t m0 = (int64_t)blockIdx.y * MC, r0 = (int64_t)(g - T.wg0) * R;
    const int mcnt = (int)((M - m0) < MC ? (M - m0) : MC);
    X += m0 * K;
    Y += m0 * ys + T.row0;
    if (Yf) Yf += m0 * ys + T.row0;
    switch (T.type) {
        case T_Q4_K: ref_rows<T_Q4_K, MC, RM>(T.w, T.nrows, K, X, mcnt, Y, Yf, ys, r0, R, s_ref); break;
        case T_Q6_K: ref_rows<T_Q6_K, MC, RM>(T.w, T.nrows, K, X, mcnt, Y, Yf, ys, r0, R, s_ref); break;
        case T_Q8_0: ref_rows<T_Q8_0, MC, RM>(T.w, T.nrows, K, X, mcnt, Y, Yf, ys, r0, R, s_ref); break;
        case T_F16: ref_rows<T_F16, MC, RM>(T.w, T.nrows, K, X, mcnt, Y, Yf, ys, r0, R, s_ref); break;
        default: ref_rows<T_BF16, MC, RM>(T.w, T.nrows, K, X, mcnt, Y, Yf, ys, r0, R, s_ref); break;
    }
}

// Reference order on already-dequantised fp32 weights (matmul_q4k_col on a wdeq column).
__global__ __launch_bounds__(kRows) void k_gemv_ref_f32(const float* __restrict__ W, int64_t N, int64_t K,
                                                        const float* __restrict__ X, int64_t M,
                                                        uint16_t* __restrict__ Y, float* __restrict__ Yf) {
    __shared__ float xs[kMC][kStageW];
    const int lane = threadIdx.x;
    const int64_t n = (int64_t)blockIdx.x * kRows + lane;
    const int64_t m0 = (int64_t)blockIdx.y * kMC;
    const int mcnt = (int)((M - m0) < kMC ? (M - m0) : kMC);
    float acc[kMC];
#pragma unroll
    for (int i = 0; i < kMC; ++i) acc[i] = 0.0f;
    for (int64_t k0 = 0; k0 < K; k0 += kStageW) {
        const int kn = (int)((K - k0) < kStageW ? (K - k0) : kStageW);
        __syncthreads();
        for (int idx = lane; idx < kMC * kStageW; idx += kRows) {
            const int mm = idx / kStageW, k = idx - mm * kStageW;
            xs[mm][k] = (mm < mcnt && k < kn) ? X[(m0 + mm) * K + k0 + k] : 0.0f;
        }
        __syncthreads();
        if (n < N) {
            for (int k = 0; k < kn; ++k) {
                const float w = W[n * K + k0 + k];
                for (int mm = 0; mm < kMC; ++mm) {
                    if (mm < mcnt) {
                        const float p = xs[mm][k] * w;
                        acc[mm] = acc[mm] + p;
                    }
                }
            }
        }
    }
    if (n < N) {
        for (int mm = 0; mm < mcnt; ++mm) {
            Y[(m0 + mm) * N + n] = (uint16_t)bf16_rne(acc[mm]);
            if (Yf) Yf[(m0 + mm) * N + n] = acc[mm];
        }
    }
}

// Rows per workgroup: a multiple of 8 that spreads `rows` over the CUs, at most `cap`.
int ref_rows_per_wg(int64_t rows, int cap) {
    const int64_t per = 8 * (int64_t)device_cu_count();
    const int64_t r = 8 * ((rows + per - 1) / per);
    return (int)(r < cap ? r : cap);
}

// One launch covers at most 2^26 rows and kMaxPasses passes of MC activation rows (a grid's threads
// along x fit 32 bits).
constexpr int64_t kMaxRows = 1LL << 26, kMaxPasses = 65535;

// Longer rows run the kernel of three and more activation rows, whose offsets into them are 64-bit (with
// 64-bit offsets the kernel of one row took 23.4 us at 6144 x 6144, 22.5 without); a run's index is 32-bit.
constexpr int64_t kMaxProductK = (1LL << 31) - 1, kMaxRefK = (1LL << 35) - 1;

// Calls fn(n0, n, m0, m) for pieces of at most kMaxRows rows and kMaxPasses passes.
template <class F>
hipError_t for_pieces(int64_t N, int64_t M, int mc, F fn) {
    for (int64_t m0 = 0; m0 < M; m0 += kMaxPasses * mc) {
        const int64_t m = M - m0 < kMaxPasses * mc ? M - m0 : kMaxPasses * mc;
        for (int64_t n0 = 0; n0 < N; n0 += kMaxRows) {   // slots (nslots > 1): N is an expert's row count
            fn(n0, N - n0 < kMaxRows ? N - n0 : kMaxRows, m0, m);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

RefGather gather_from(RefGather g, int64_t n0, int64_t rb) {
    if (g.W_alt) g.W_alt += n0 * rb;
    if (g.W2) g.W2 += n0 * rb;
    if (g.W2_alt) g.W2_alt += n0 * rb;
    if (g.Y2) g.Y2 += n0;
    return g;
}

struct RefCall {
    const uint8_t* W;
    int64_t N, K;
    const uint16_t* x;
    int64_t M;
    uint16_t* y;
    float* y_f32;
    int64_t ys;
    int nslots;
    RefGather ga;
    hipStream_t st;
};

template <int TYPE, int MC, int RM>
hipError_t run_ref(const RefCall& c) {
    typedef RefCfg<MC, RM> C;
    const int R = ref_rows_per_wg(c.N * c.nslots * ((c.M + MC - 1) / MC), RM);
    const int64_t rb = row_bytes(TYPE, c.K);
    return for_pieces(c.N, c.M, MC, [&](int64_t n0, int64_t n, int64_t m0, int64_t m) {
        const dim3 grid((unsigned)((n + R - 1) / R), (unsigned)((m + MC - 1) / MC), (unsigned)c.nslots);
        hipLaunchKernelGGL((k_gemv_ref<TYPE, MC, RM>), grid, dim3(C::kThreads), C::kLds, c.st, c.W + n0 * rb, n, c.K,
                           c.x + m0 * c.K, m, c.y + m0 * c.ys + n0, c.y_f32 ? c.y_f32 + m0 * c.ys + n0 : nullptr, c.ys, R,
                           gather_from(c.ga, n0, rb));
    });
}

template <int TYPE, int MC>
hipError_t run_ref_wave(const RefCall& c) {
    // 16-bit rows at two activation rows: four waves per CU where more would thrash the rows' lines (200000 x
    // 6144: 661 -> 570 us; 72000 x 6144, whose waves all fit, 198 -> 273)
    const bool few = (TYPE == T_F16 || TYPE == T_BF16) && MC == 2 && c.K >= 2048 &&
                     c.N * c.nslots * ((c.M + MC - 1) / MC) >= 440 * (int64_t)device_cu_count();
    const int pad = few ? 40 * 1024 - 2 * MC * kWaveChunk * 4 : 0;
    const int64_t rb = row_bytes(TYPE, c.K);
    return for_pieces(c.N, c.M, MC, [&](int64_t n0, int64_t n, int64_t m0, int64_t m) {
        const dim3 grid((unsigned)((n + 63) / 64), (unsigned)((m + MC - 1) / MC), (unsigned)c.nslots);
        hipLaunchKernelGGL((k_gemv_ref_wave<TYPE, MC>), grid, dim3(64), pad, c.st, c.W + n0 * rb, n, c.K, c.x + m0 * c.K, m,
                           c.y + m0 * c.ys + n0, c.y_f32 ? c.y_f32 + m0 * c.ys + n0 : nullptr, c.ys,
                           gather_from(c.ga, n0, rb));
    });
}

// Whether the one-wave kernel takes these pointers and this K (whole units, its loads' alignment).
bool ref_wave_takes(int type, const RefCall& c) {
    const uintptr_t wa = type == T_Q8_0 || type == T_Q6_K ? 4 : 16;
    const auto al = [](const void* p, uintptr_t a) { return ((uintptr_t)p & (a - 1)) == 0; };
    return c.K % (type == T_Q6_K ? 512 : type == T_Q4_K ? 256 : 64) == 0 && c.K <= (1 << 20) && al(c.x, 8) && al(c.W, wa) &&
           al(c.ga.W_alt, wa) && al(c.ga.W2, wa) && al(c.ga.W2_alt, wa) && c.ga.x_zstride % 4 == 0 &&
           c.ga.wstride % (int64_t)wa == 0;
}

// Whether the one-wave kernel is the faster one for `rows` rows (of all slots, times the passes of
// activation rows).  ref_rows takes a time that grows with the rows once every CU has a workgroup, in
// steps of 32 rows per CU; the one-wave kernel takes the same time up to 64 rows per SIMD.  The lines
// cross at these rows per CU, earlier where K is short and ref_rows' stages are few.  Q4_K, K = 6144,
// ref_rows > one wave: M = 1, 32768 / 65536 / 154880 rows 61 > 74 / 114 > 74 / 282 > 175 us; M = 2, 24576 /
// 32768 / 65536 rows 89 > 100 / 116 > 99 / 227 > 102 us; M = 4, 49152 / 65536 rows 155 > 172 / 204 > 171 us;
// M = 8, 65536 / 98304 rows 267 > 300 / 412 > 327 us.  Q8_0 and the 16-bit types, whose rows the one-wave
// kernel reads 68 or 128 bytes at a time, stay on ref_rows at M = 1 and M = 8 (Q8_0: 131072 rows 344 and
// 415 us at M = 1, 154880 rows 643 and 735 us at M = 8), but for a short K, and 16 bits
// from 130 rows per CU to 256 or 400 at M = 1 and K <= 2048 (200000 x 1024: 72 and 97 us).
bool ref_wave_wins(int type, int64_t rows, int64_t M, int64_t K) {
    const int per = (int)(rows / device_cu_count() < 1 << 20 ? rows / device_cu_count() : 1 << 20);
    const int i = M >= 5 ? 3 : M >= 3 ? 2 : (int)M - 1;
    if (type == T_Q4_K) {
        const int at[4] = {K <= 256 ? 104 : 130, K <= 512 ? 64 : 97, K <= 256 ? 130 : K <= 512 ? 156 : 194,
                           K <= 256 ? 208 : K <= 512 ? 256 : 288};
        return per >= at[i];
    }
    if (type == T_Q6_K) {
        const int at[4] = {66, K <= 512 ? 56 : 66, K <= 512 ? 130 : 192, K <= 512 ? 224 : 300};
        return per >= at[i];
    }
    if (i == 0) return K <= 256 ? per >= 120 : type != T_Q8_0 && K <= 2048 && per >= 130 && per < (K <= 1024 ? 400 : 256);
    if (i == 1) return per >= (K <= 512 ? 64 : type != T_Q8_0 && K >= 4096 ? 130 : 97);
    if (i == 2) return per >= (K <= 512 ? 130 : K > 8192 ? 256 : 194);
    return K <= 256 ? per >= 300 : K <= 512 && per >= 380;
}

template <int TYPE>
hipError_t run_ref_type(const RefCall& c) {
    const int64_t M = c.M, mc = M >= 5 ? 8 : M >= 3 ? 4 : M;
    if (ref_wave_takes(TYPE, c) && ref_wave_wins(TYPE, c.N * c.nslots * ((M + mc - 1) / mc), M, c.K)) {
        if (M >= 5) return run_ref_wave<TYPE, 8>(c);
        if (M >= 3) return run_ref_wave<TYPE, 4>(c);
        return M == 2 ? run_ref_wave<TYPE, 2>(c) : run_ref_wave<TYPE, 1>(c);
    }
    if (M >= 5) return run_ref<TYPE, 8, 32>(c);
    if (M >= 3 || c.K > kMaxProductK) return run_ref<TYPE, 4, 32>(c);
    if (M == 2) return run_ref<TYPE, 2, 32>(c);
    if (c.N * c.nslots <= 32 * (int64_t)device_cu_count()) return run_ref<TYPE, 1, 32>(c);
    return run_ref<TYPE, 1, 64>(c);
}

hipError_t run_ref_any(int type, const RefCall& c) {
    if (c.K > kMaxRefK) return hipErrorInvalidValue;
    switch (type) {
        case T_Q4_K: return run_ref_type<T_Q4_K>(c);
        case T_Q6_K: return run_ref_type<T_Q6_K>(c);
        case T_Q8_0: return run_ref_type<T_Q8_0>(c);
        case T_F16: return run_ref_type<T_F16>(c);
        case T_BF16: return run_ref_type<T_BF16>(c);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_gemv_ref_gather(int type, const void* w, int64_t N, int64_t K, const uint16_t* x, int64_t M,
                                  uint16_t* y, float* y_f32, int nslots, const int32_t* sel, int topk, int64_t E,
                                  int64_t wstride, const void* w_alt, int64_t x_zstride, int64_t y_zstride,
                                  hipStream_t st, const void* w2, const void* w2_alt, uint16_t* y2) {
    const RefGather ga{sel, topk, nslots, (const uint8_t*)w2, (const uint8_t*)w2_alt, y2, E, wstride,
                       (const uint8_t*)w_alt, x_zstride, y_zstride};
    return run_ref_any(type, RefCall{(const uint8_t*)w, N, K, x, M, y, y_f32, N, w2 ? 2 * nslots : nslots, ga, st});
}

hipError_t launch_gemv_ref(int type, const void* w, int64_t N, int64_t K, const uint16_t* x, int64_t M,
                           uint16_t* y, float* y_f32, hipStream_t st) {
    return launch_gemv_ref_gather(type, w, N, K, x, M, y, y_f32, 1, nullptr, 0, 0, 0, nullptr, 0, 0, st);
}

hipError_t launch_gemv_ref_tiles(const aipu_tile_desc* tiles, int n_tiles, int64_t K, const uint16_t* x, int64_t M,
                                 uint16_t* y, float* y_f32, int64_t ys, hipStream_t st) {
    if (n_tiles < 1 || n_tiles > AIPU_MAX_TILES || M < 1 || K > kMaxRefK) return hipErrorInvalidValue;
    // tiles of so many rows that the one-wave kernel is faster run by themselves, the others in one launch
    aipu_tile_desc rest[AIPU_MAX_TILES];
    int n_rest = 0;
    for (int i = 0; i < n_tiles; ++i) {
        const aipu_tile_desc& d = tiles[i];
        const RefCall c{(const uint8_t*)d.w, d.nrows, K, x, M, y + d.row0, y_f32 ? y_f32 + d.row0 : nullptr, ys, 1, RefGather{}, st};
        const int64_t mc = M >= 5 ? 8 : M >= 3 ? 4 : M;
        if (!ref_wave_takes(d.ggml_type, c) || !ref_wave_wins(d.ggml_type, d.nrows * ((M + mc - 1) / mc), M, K)) {
            rest[n_rest++] = d;
            continue;
        }
        const hipError_t e = run_ref_any(d.ggml_type, c);
        if (e != hipSuccess) return e;
    }
    if (n_rest == 0) return hipSuccess;
    tiles = rest;
    n_tiles = n_rest;
    int64_t rows = 0;
    for (int i = 0; i < n_tiles; ++i) rows += tiles[i].nrows;
    const auto run = [&](auto cfg, auto kernel, int mc, int rm) {
        typedef decltype(cfg) C;
        // a launch's threads must fit 32 bits: pieces of at most kMaxRows rows, flushed before they exceed it
        constexpr int64_t kMaxWgs = 0xFFFFFFFFLL / C::kThreads;
        const int R = ref_rows_per_wg(rows * ((M + mc - 1) / mc), rm);
        RefTiles a{};
        int64_t nwg = 0;
        const auto flush = [&] {
            for (int64_t m0 = 0; m0 < M && a.n; m0 += kMaxPasses * mc) {
                const int64_t m = M - m0 < kMaxPasses * mc ? M - m0 : kMaxPasses * mc;
                hipLaunchKernelGGL(kernel, dim3((unsigned)nwg, (unsigned)((m + mc - 1) / mc)), dim3(C::kThreads), C::kLds, st,
                                   a, K, x + m0 * K, m, y + m0 * ys, y_f32 ? y_f32 + m0 * ys : nullptr, ys, R);
                const hipError_t e = hipGetLastError();
                if (e != hipSuccess) return e;
            }
            a.n = 0;
            nwg = 0;
            return hipSuccess;
        };
        for (int i = 0; i < n_tiles; ++i) {
            const aipu_tile_desc& d = tiles[i];
            for (int64_t r0 = 0; r0 < d.nrows; r0 += kMaxRows) {
                const int64_t n = d.nrows - r0 < kMaxRows ? d.nrows - r0 : kMaxRows, wgs = (n + R - 1) / R;
                if (a.n == AIPU_MAX_TILES || nwg + wgs > kMaxWgs) {
                    const hipError_t e = flush();
                    if (e != hipSuccess) return e;
                }
                a.t[a.n++] = RefTile{(const uint8_t*)d.w + r0 * row_bytes(d.ggml_type, K), d.row0 + r0, n, d.ggml_type,
                                     (int32_t)nwg};
                nwg += wgs;
            }
        }
        return flush();
    };
    if (M >= 5) return run(RefCfg<8, 32>{}, k_gemv_ref_tiles<8, 32>, 8, 32);
    if (M >= 3 || K > kMaxProductK) return run(RefCfg<4, 32>{}, k_gemv_ref_tiles<4, 32>, 4, 32);
    if (M == 2) return run(RefCfg<2, 32>{}, k_gemv_ref_tiles<2, 32>, 2, 32);
    if (rows <= 32 * (int64_t)device_cu_count()) return run(RefCfg<1, 32>{}, k_gemv_ref_tiles<1, 32>, 1, 32);
    return run(RefCfg<1, 64>{}, k_gemv_ref_tiles<1, 64>, 1, 64);
}

hipError_t launch_gemv_ref_f32(const float* w, int64_t N, int64_t K, const float* x, int64_t M, uint16_t* y,
                               float* y_f32, hipStream_t st) {
    const dim3 grid((unsigned)((N + kRows - 1) / kRows), (unsigned)((M + kMC - 1) / kMC));
    hipLaunchKernelGGL(k_gemv_ref_f32, grid, dim3(kRows), 0, st, w, N, K, x, M, y, y_f32);
    return hipGetLastError();
}

}  // namespace aipu
