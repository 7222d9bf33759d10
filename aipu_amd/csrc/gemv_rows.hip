// Multi-row Q4_K GEMV for long or unevenly divided K (tolerance mode, M = 2 .. 8 activation rows, one
// weight pass), in the one-row order of mfma_gemv.hpp: every row is bit-identical to its one-row launch.
//
// It serves 8 .. 64 blocks where the persistent multi-row kernels and the register-resident small-batch
// kernels (which hold a wave's whole part of K) have no plan and a one-row kernel forms the same order: up
// to K = 8192 the block counts that do not split into at most eight parts of three (2816, 4352, 5632) and
// every K beyond 6144; beyond 8192 those that k_gemv1 splits into at most eight parts of eight (8960, 9216,
// 10240, 10752, 12288, .., 16384).  Any other K beyond 8192 runs a launch per row, or the streaming kernel.
//
// A workgroup owns a 16-row tile, wave w the w-th part of its blocks.  A wave walks its part block by
// block with kNS blocks in flight: a block's weights arrive in one of its kNS LDS slots by
// direct-to-LDS copies and its activations in registers.  Per block the wave moves the weights into
// registers, reuses the slot for block b + kNS, stages the activations of all rows as MFMA operands
// in its own LDS region (nothing is shared, so there is no barrier in the loop), builds the codes
// once, and runs rows 0-3 and rows 4-7 as two sets of eight MFMAs against them.  The block terms go
// to LDS and the whole workgroup sums them in the fixed order at the end.
//
// What bounds it is a wave's serial path through a block (LDS round trips, the MFMA chains, the
// codes' VALU) with two to four waves per SIMD, not the memory: four blocks in flight per wave
// instead of two were slower (fewer waves fit), and so were groups of three blocks.  Measured, one
// launch per row -> here, Q4_K 6144 x 12288: M = 2 / 4 / 8 25.8 / 46.9 / 91.9 -> 15.9 / 19.2 / 25.4 us;
// 6144 x 8192, M = 2 / 4 18 / 35 -> 12 / 14.7 us; 5000 x 2816, M = 4 / 8 (two rows at a time on the
// one-row kernel) 10.7 / 21.1 -> 8.1 / 13.5 us.  Where the kernels that hold a wave's whole part have
// a plan they are faster (6144 x 6144, M = 4: 8.5 against 12.9 us).
#include "common.hpp"
#include "launch.hpp"
#include "mfma_gemv.hpp"

namespace aipu {

using namespace mg;

namespace {

constexpr int kRowMaxW = 8;                   // waves per workgroup
constexpr int64_t kMaxN = 1LL << 26;          // rows of a launch: a grid's threads along x fit 32 bits
static_assert(kMaxN / kTR * kRowMaxW * 64 <= 0xFFFFFFFFLL, "grid too large");
constexpr int kNS = 2;                        // blocks in flight per wave
constexpr int kSlot = 3 * 1024;               // 16 rows x 144 B in whole 1 KB copies
// one activation row's operands of a block, [8 MFMAs][4 K-groups] 16 B, then its eight sub-block
// sums in fp32; 64 B past the operands put the rows' operand reads on different banks
constexpr int kActRow = 512 + 64;

template <int MR>
constexpr int term_stride() { return MR * kTR + 2; }   // floats per block; + 2: pairs on different banks

// A lane's bytes of a block from its LDS slot, read and waited for inside one asm statement: the
// compiler would order LDS loads it can see behind every direct-to-LDS copy in flight.
__device__ __forceinline__ Raw slot_read(uint32_t hdr, uint32_t qs) {
    u32x4_t h, q0, q1;
    asm volatile(
        "ds_read_b128 %0, %3\n\t"
        "ds_read_b128 %1, %4\n\t"
        "ds_read_b128 %2, %4 offset:16\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(h), "=&v"(q0), "=&v"(q1)
        : "v"(hdr), "v"(qs)
        : "memory");
    Raw r;
    r.h = make_uint4(h.x, h.y, h.z, h.w);
    r.q0 = make_uint4(q0.x, q0.y, q0.z, q0.w);
    r.q1 = make_uint4(q1.x, q1.y, q1.z, q1.w);
    return r;
}

// a_reads, and the sub-block sums (lo, hi) of RS activation rows at sa + m * kActRow, in one asm
// statement that waits for all of them (plain loads of the sums would wait for the copies, too).
template <int RS>
__device__ __forceinline__ void ops_read(u32x4_t (&A)[8], float2 (&as)[RS], uint32_t aa, uint32_t sa, uint64_t mask) {
    static_assert(RS == 2 || RS == 4, "two or four rows per set");
    uint64_t saved;
    if constexpr (RS == 4)
        asm volatile(
            "ds_read_b64 %8, %14\n\t"
            "ds_read_b64 %9, %14 offset:%c16\n\t"
            "ds_read_b64 %10, %14 offset:%c17\n\t"
            "ds_read_b64 %11, %14 offset:%c18\n\t"
            "s_mov_b64 %12, exec\n\t"
            "s_and_b64 exec, exec, %15\n\t"
            "ds_read_b128 %0, %13\n\t"
            "ds_read_b128 %1, %13 offset:64\n\t"
            "ds_read_b128 %2, %13 offset:128\n\t"
            "ds_read_b128 %3, %13 offset:192\n\t"
            "ds_read_b128 %4, %13 offset:256\n\t"
            "ds_read_b128 %5, %13 offset:320\n\t"
            "ds_read_b128 %6, %13 offset:384\n\t"
            "ds_read_b128 %7, %13 offset:448\n\t"
            "s_mov_b64 exec, %12\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "+v"(A[0]), "+v"(A[1]), "+v"(A[2]), "+v"(A[3]), "+v"(A[4]), "+v"(A[5]), "+v"(A[6]), "+v"(A[7]),
              "=&v"(as[0]), "=&v"(as[1]), "=&v"(as[2]), "=&v"(as[3]), "=&s"(saved)
            : "v"(aa), "v"(sa), "s"(mask), "i"(kActRow), "i"(2 * kActRow), "i"(3 * kActRow)
            : "memory", "scc");   // s_and_b64 writes SCC
    else
        asm volatile(
            "ds_read_b64 %8, %12\n\t"
            "ds_read_b64 %9, %12 offset:%c14\n\t"
            "s_mov_b64 %10, exec\n\t"
            "s_and_b64 exec, exec, %13\n\t"
            "ds_read_b128 %0, %11\n\t"
            "ds_read_b128 %1, %11 offset:64\n\t"
            "ds_read_b128 %2, %11 offset:128\n\t"
            "ds_read_b128 %3, %11 offset:192\n\t"
            "ds_read_b128 %4, %11 offset:256\n\t"
            "ds_read_b128 %5, %11 offset:320\n\t"
            "ds_read_b128 %6, %11 offset:384\n\t"
            "ds_read_b128 %7, %11 offset:448\n\t"
            "s_mov_b64 exec, %10\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "+v"(A[0]), "+v"(A[1]), "+v"(A[2]), "+v"(A[3]), "+v"(A[4]), "+v"(A[5]), "+v"(A[6]), "+v"(A[7]),
              "=&v"(as[0]), "=&v"(as[1]), "=&s"(saved)
            : "v"(aa), "v"(sa), "s"(mask), "i"(kActRow)
            : "memory", "scc");
}

template <int MR>
__global__ __launch_bounds__(kRowMaxW * 64) __attribute__((amdgpu_waves_per_eu(MR == 2 ? 4 : MR == 4 ? 3 : 2))) void k_gemvr(const uint8_t* __restrict__ W, int64_t N, int nsb,
                                                         const uint16_t* __restrict__ X, int M, uint16_t* __restrict__ Y,
                                                         float* __restrict__ Yf, int64_t ys) {
    constexpr int SETS = MR > 4 ? 2 : 1;      // MFMA sets of up to four rows
    constexpr int RS = MR > 4 ? 4 : MR;       // rows per set
    // the slots are an LDS object of their own: reads of the staged activations are then not ordered
    // behind the direct-to-LDS copies in flight
    __shared__ __align__(16) uint8_t s_slots[kRowMaxW * kNS * kSlot];
    extern __shared__ __align__(16) uint8_t s_rows[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), nw = (int)(blockDim.x >> 6);
    uint8_t* wA = s_rows + w * (MR * kActRow);
    float* terms = (float*)(s_rows + nw * (MR * kActRow));   // [block][row][16]
    uint8_t* wW = s_slots + w * (kNS * kSlot);
    const int kb0 = w * nsb / nw, kb1 = (w + 1) * nsb / nw;
    const uint32_t rb = (uint32_t)nsb * 144u;
    const int64_t r0 = (int64_t)blockIdx.x * kTR;
    const int nvalid = (int)(N - r0 < kTR ? N - r0 : kTR);
    const int K = nsb * QK_K;

    const __amdgpu_buffer_rsrc_t wr = buf_rsrc(W + r0 * (int64_t)rb, (uint32_t)nvalid * rb);
    const __amdgpu_buffer_rsrc_t xr = buf_rsrc(X, (uint32_t)M * (uint32_t)K * 2u);
    // piece j of a slot: 16-B piece j % 9 of weight row j / 9
    uint32_t off[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int j = 64 * i + lane, r = j / 9, p = j - r * 9;
        off[i] = r < kTR ? (uint32_t)r * rb + 16u * (uint32_t)p : kOOB;
    }
    // activations of a block: lane = (row parity, piece), register i = rows 2i, 2i + 1
    uint4 xv[kNS][MR / 2];
    const int xm = lane >> 5, xp = lane & 31;
    auto issue = [&](int b, int slot) {   // past the part, and rows past M: zeros, no memory access
        const bool in = b < kb1;
#pragma unroll
        for (int i = 0; i < MR / 2; ++i) {
            const int m = 2 * i + xm;
            xv[slot][i] = buf_load16(xr, in && m < M ? 2u * ((uint32_t)m * (uint32_t)K + (uint32_t)b * QK_K) + 16u * (uint32_t)xp
                                                     : kOOB);
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
            lds_dma16(wr, wW + slot * kSlot + 1024 * i, in && off[i] != kOOB ? off[i] + 144u * (uint32_t)b : kOOB);
    };
#pragma unroll
    for (int j = 0; j < kNS; ++j) issue(kb0 + j, j);
    const int n = lane & 15, g = lane >> 4;
    const HdrSel hs = hdr_sel(g);
    const CodeK ck = code_k();
    const uint64_t dmask = diag_mask(RS);
    const uint32_t aLane = lds_addr(wA) + (uint32_t)((n - 4 * g) & 3) * (uint32_t)kActRow + 16u * (uint32_t)g;
    const uint32_t hLane = lds_addr(wW) + 144u * (uint32_t)n, qLane = hLane + 16u + 32u * (uint32_t)g;
    const uint32_t sLane = lds_addr(wA) + 512u + 8u * (uint32_t)g;
    u32x4_t A[8];   // off-diagonal lanes stay zero
#pragma unroll
    for (int t = 0; t < 8; ++t) A[t] = u32x4_t{0u, 0u, 0u, 0u};

    auto block = [&](int b, int slot) {
        // this block's copies: the later blocks' are three operations each (their activation loads,
        // issued before their copies, are not counted on: the compiler may move or drop those)
        __builtin_amdgcn_s_waitcnt(wait_vm(3 * (kNS - 1)));
        const Raw R = slot_read(hLane + (uint32_t)(slot * kSlot), qLane + (uint32_t)(slot * kSlot));
        // stage the activations (k_gemvs' operand order and sums)
        {
            const int gg = xp >> 3, t = xp & 7;
            const uint32_t ones = 0x3F803F80u;
#pragma unroll
            for (int i = 0; i < MR / 2; ++i) {
                uint8_t* rA = wA + (2 * i + xm) * kActRow;
                const uint4 x = xv[slot][i];
                float sm = 0.f;
                sm = dot2(x.x, ones, sm);
                sm = dot2(x.y, ones, sm);
                sm = dot2(x.z, ones, sm);
                sm = dot2(x.w, ones, sm);
                sm += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sm), 0xB1, 0xF, 0xF, false));
                sm += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(sm), 0x4E, 0xF, 0xF, false));
                *(u32x4_t*)(rA + 16 * (t * 4 + gg)) = act_perm(x);
                if ((xp & 3) == 0) *(float*)(rA + 512 + 4 * (gg * 2 + ((xp >> 2) & 1))) = sm;
            }
        }
        issue(b + kNS, slot);
        const uint32_t qd[8] = {R.q0.x, R.q0.y, R.q0.z, R.q0.w, R.q1.x, R.q1.y, R.q1.z, R.q1.w};
        u32x4_t lo[4], hi[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            lo[t] = codes_lo(qd[2 * t], qd[2 * t + 1], ck);
            hi[t] = codes_hi(qd[2 * t], qd[2 * t + 1], ck);
        }
        const Hdr H = hdr_decode(R.h, hs);
#pragma unroll
        for (int s = 0; s < SETS; ++s) {
            float2 as[RS];
            ops_read<RS>(A, as, aLane + (uint32_t)(4 * s * kActRow), sLane + (uint32_t)(4 * s * kActRow), dmask);
            f32x4_t dlo = {0.f, 0.f, 0.f, 0.f}, dhi = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int m = 0; m < RS; ++m) {
                dlo[m] = -kCodeBiasF * as[m].x;
                dhi[m] = -kCodeBiasF * as[m].y;
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                dlo = mfma(A[t], lo[t], dlo);
                dhi = mfma(A[4 + t], hi[t], dhi);
            }
            float t[RS];
#pragma unroll
            for (int m = 0; m < RS; ++m) t[m] = block_term(H, dlo[m], dhi[m], as[m].x, as[m].y);
            float* te = terms + b * term_stride<MR>() + (4 * s + g) * kTR + n;
            if constexpr (RS == 4) {
                *te = block_sum4(t[0], t[1], t[2], t[3]);   // lane 16g + n: row 4s + g
            } else {
                const float v = block_sum2(t[0], t[1]);     // lane 16g + n: row g & 1
                if (g < 2) *te = v;
            }
        }
    };
    // whole turns of the slots without a branch between a load and its use (the compiler's waits for
    // the activations stay at their own block), then the rest
    int b = kb0;
    for (; b + kNS <= kb1; b += kNS) {
#pragma unroll
        for (int j = 0; j < kNS; ++j) block(b + j, j);
    }
#pragma unroll
    for (int j = 0; j + 1 < kNS; ++j)
        if (b + j < kb1) block(b + j, j);
    __builtin_amdgcn_s_waitcnt(kWaitVm0);   // the copies past the part, into this workgroup's LDS
    __syncthreads();
    // eight lanes per output; the trip count is the workgroup's, so every lane takes part
    const int per = (int)(blockDim.x >> 3);
    for (int o0 = 0; o0 < kTR * MR; o0 += per) {
        const int o = o0 + (tid >> 3), r = (o / kTR) % MR, c = o % kTR;
        const float v = canon_sum8(nsb, lane & 7, [&](int b) { return terms[b * term_stride<MR>() + r * kTR + c]; });
        if (o < kTR * MR && r < M && c < nvalid && (lane & 7) == 0) {
            Y[(int64_t)r * ys + r0 + c] = (uint16_t)bf16_rne(v);
            if (Yf) Yf[(int64_t)r * ys + r0 + c] = v;
        }
    }
}

template <int MR>
int64_t rows_lds(int nsb, int w) {
    return (int64_t)w * (MR * kActRow) + (int64_t)nsb * term_stride<MR>() * 4;   // dynamic
}

constexpr int kMinBlocks = kRowMaxW, kMaxBlocks = 64;
static_assert(kRowMaxW * 8 * kActRow + kMaxBlocks * term_stride<8>() * 4 <= 160 * 1024 - kRowMaxW * kNS * kSlot, "LDS");

// Waves per workgroup: the most that leave two workgroups on a CU, unless that is under four; else eight.
template <int MR>
int rows_waves(int nsb) {
    for (int w = kRowMaxW; w >= 4; --w)
        if (rows_lds<MR>(nsb, w) <= 80 * 1024 - kRowMaxW * kNS * kSlot) return w;
    return kRowMaxW;
}

template <int MR>
hipError_t run_rows_any(const uint8_t* W, int64_t N, int nsb, const uint16_t* x, int M, uint16_t* y, float* yf, int64_t ys,
                        hipStream_t st) {
    const int w = rows_waves<MR>(nsb);
    hipLaunchKernelGGL(k_gemvr<MR>, dim3((unsigned)((N + kTR - 1) / kTR)), dim3(64 * w), (size_t)rows_lds<MR>(nsb, w), st, W, N,
                       nsb, x, M, y, yf, ys);
    return hipGetLastError();
}

}  // namespace

bool gemv_rows_supported(int64_t N, int64_t K, int M) {
    return M >= 2 && M <= 8 && N >= 1 && N <= kMaxN && K % QK_K == 0 && K >= kMinBlocks * QK_K && K <= kMaxBlocks * QK_K;
}

hipError_t launch_gemv_rows(const uint8_t* W, int64_t N, int64_t K, const uint16_t* x, int M, uint16_t* y, float* yf,
                            int64_t ys, hipStream_t st) {
    if (!gemv_rows_supported(N, K, M)) return hipErrorInvalidValue;
    const int nsb = (int)(K / QK_K);
    if (M <= 2) return run_rows_any<2>(W, N, nsb, x, M, y, yf, ys, st);
    if (M <= 4) return run_rows_any<4>(W, N, nsb, x, M, y, yf, ys, st);
    return run_rows_any<8>(W, N, nsb, x, M, y, yf, ys, st);
}

}  // namespace aipu
