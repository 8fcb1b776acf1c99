// Batched TL1 contraction over M tokens on int8 MFMA (multi-token prefill).
//
// The reference prefills one token at a time: prefill_token
// (src/runtime/TenzoEngine.cpp:1809-1819) runs compute_from_lut (:129-146)
// once per token and projection. Here the M tokens of a prompt share one
// pass over the weights: acc[m][n] = sum_k W[n][k] * codes[m][k] is an
// integer GEMM on v_mfma_i32_32x32x32_i8 whose int32 results are exact, so
// every output equals the per-token GEMV's bit for bit.
//
// Operands (no extra weight copy: the decode GEMV layout is read as is):
//   W  the TL1 device layout of tl1.hip: per row block b (64 rows) and
//      super-chunk s (64 columns), row r's 16 bytes hold dword q = columns
//      64s+16q+c as u = w+1 at bit 8*(c%4)+2*(c/4). (dword >> 2j) & 0x03030303
//      are the bytes of columns 16q+4j .. 16q+4j+3 in order.
//   codes  int8 [M][Kp] (Kp = 64*ceil(K/64), zero padded), with
//      q[m] = {inv_scale, sum of codes} from the activation quantizer.
// Since u = w + 1, sum_k w_k a_k = sum_k u_k a_k - sum_k a_k: the epilogue
// subtracts the code sum of the token, as the GEMV does. Every output is one
// workgroup's, so there is no cross-workgroup reduction and no scratch.
//
// v_mfma_i32_32x32x32_i8 is used rather than 16x16x64: at one wave per SIMD
// it issues one per 34 cycles (4.6 POP/s over the chip) where 16x16x64
// issues one per 32 cycles for half the work.
#include "common.h"
#include "tl1.h"

namespace tz {
namespace {

typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i16v __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;
constexpr int kRawBuffer = 0x00020000;  // buffer resource word 3: raw buffer, gfx9 family
constexpr uint32_t kField = 0x03030303u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, kRawBuffer);
}
// 16 bytes per lane from a buffer straight into LDS (no registers): lane l's
// bytes land at dst + 16 l. Offsets past the resource's byte count read zeros.
__device__ __forceinline__ void to_lds16(__amdgpu_buffer_rsrc_t r, void* dst, uint32_t off) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)dst, 16, off, 0, 0, 0);
}
// The same load issued from assembly. Around the builtin the compiler cannot tell the
// ring's slots apart and may wait for every outstanding load (vmcnt 0) before each LDS
// read, which stops the ring; here only the waits written out are made. r: the buffer
// resource's four words; lds: the LDS byte address (uniform). The instruction has no
// output registers. M0 needs one wait state before it, and a scalar register that a vector
// instruction has written five: the compiler counts neither inside an asm. The resource's
// words are written by scalar instructions (five wait states before each load make 256 tokens of
// 3840 x 6912 13% slower), and M0, which cannot be declared as written (it is reserved), is used
// for nothing else: test_assembly_hazards.py checks both in the compiled code.
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u4v buf_words(const void* base, uint32_t bytes) {
    const uint64_t a = (uint64_t)base;
    return u4v{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xffffu)),
               (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), (uint32_t)kRawBuffer};
}
__device__ __forceinline__ void to_lds16_asm(u4v r, uint32_t lds, uint32_t off) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                 :
                 : "s"(lds), "v"(off), "s"(r)
                 : "memory");
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
}
// s_barrier without the workgroup fence of __syncthreads(), whose release half
// waits for every outstanding vector memory operation (vmcnt 0), which would
// drain the ring's loads at each chunk. The memory clobber keeps LDS accesses
// on their side of it; LDS-DMA completion is waited for explicitly (wait_vm).
__device__ __forceinline__ void block_barrier() { asm volatile("s_barrier" ::: "memory"); }
// Keeps the memory operations before it ahead of the instructions after it:
// the compiler memory clobber stops IR passes from sinking the loads to their
// first use, the scheduling barrier stops the machine scheduler.
__device__ __forceinline__ void issue_point() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
template <int N> __device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

template <int N> __device__ __forceinline__ void wait_vm_asm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// y = resid + float(acc - code_sum) * (inv_scale * row scale) for rows
// row .. row+3 of token m (compute_from_lut :118-126 and the residual adds of
// forward_layer_raw :1590 / :1628), one fp32 multiply and one fp32 add each.
__device__ __forceinline__ void finalize4(i4v v, const tenzo_hip_actq_t a, int m, int64_t row,
                                          int64_t N, const RowScales& rs, float* __restrict__ y,
                                          const float* __restrict__ resid,
                                          int32_t* __restrict__ acc_out) {
    int j = 0;
    while (j < rs.n - 1 && row >= rs.end[j]) ++j;  // segment ends are multiples of 64
    const float sc = __fmul_rn(a.inv_scale, rs.scale[j]);
    const int64_t o = (int64_t)m * N + row;
    const int d0 = v[0] - a.code_sum, d1 = v[1] - a.code_sum, d2 = v[2] - a.code_sum,
              d3 = v[3] - a.code_sum;
    float4 out = make_float4((float)d0 * sc, (float)d1 * sc, (float)d2 * sc, (float)d3 * sc);
    if (resid) {
        const float4 r = *reinterpret_cast<const float4*>(resid + o);
        out.x = __fadd_rn(r.x, out.x);
        out.y = __fadd_rn(r.y, out.y);
        out.z = __fadd_rn(r.z, out.z);
        out.w = __fadd_rn(r.w, out.w);
    }
    *reinterpret_cast<float4*>(y + o) = out;
    if (acc_out) *reinterpret_cast<int4*>(acc_out + o) = make_int4(d0, d1, d2, d3);
}

}  // namespace

// One workgroup = 4 waves = RW row waves x KW = 4 / RW K groups; it owns
// 64*RW rows (row blocks RW*bt .. RW*bt+RW-1) and BM = 32*CT tokens. K group
// kg takes the contiguous chunk run [kg*T, (kg+1)*T) (T = ceil(KS/KW); chunks
// past its end read zero weights). Each 64-column chunk is two 32-deep MFMA
// steps, h = 0, 1, and a wave's 64 rows are two 32-row tiles.
//
// v_mfma_i32_32x32x32_i8 operands (lane l = 32g + i):
//   A (weights): row i of the tile, k = 16g .. 16g+15 of the step: for step
//      h that is dword 2h + g of the row's 16-byte record, unpacked.
//   B (codes):   token i of the 32-token tile, the same columns: 16 bytes at
//      codes[m][64s + 16(2h + g)].
//   C:           token i, rows 8(j/4) + 4g + j%4 for registers j = 0..15.
// Per chunk and K group an LDS ring slot holds
//   codes:   2*CT fragments of 1 KiB (tile u, step h at (2u + h) KiB; lane l's
//            16 bytes at 16 l),
//   weights: RW row blocks of 1 KiB (lane l = the 16-byte record of row l),
// filled by direct-to-LDS loads issued kRing - 2 chunks ahead. Each wave loads
// its own row block's weights and 2*CT / RW of the group's code fragments.
// One block barrier per chunk both publishes the chunk and frees the slot the
// next loads overwrite. K groups then add their int32 tiles through LDS.
template <int RW, int KW, int CT>
__global__ void __launch_bounds__(64 * RW * KW)
tl1_mfma_kernel(const uint8_t* __restrict__ w, const int8_t* __restrict__ codes,
                const tenzo_hip_actq_t* __restrict__ aq, int M, int64_t N, int KS, int mtiles,
                RowScales rs, float* __restrict__ y, const float* __restrict__ resid,
                int32_t* __restrict__ acc_out) {
    constexpr int CH = 1;  // chunks per step (2 measured no faster)
    constexpr int BM = 32 * CT;
    constexpr int kFrags = 2 * CT;  // code fragments per chunk and K group
    static_assert(kFrags % RW == 0, "each row wave loads the same number of fragments");
    constexpr int kChunkBytes = (kFrags + RW) * 1024;  // one chunk of one K group
    constexpr int kGroupBytes = CH * kChunkBytes;       // one step of one K group
    constexpr int kSlotBytes = KW * kGroupBytes;
    constexpr int kLoads = CH * (1 + kFrags / RW);  // direct-to-LDS loads per wave and step
    // LDS ring of about 64 KiB, at least 4 slots: kRing - 2 steps in flight
    // ahead of the one being read (deeper rings measured no faster: the
    // per-wave issue rate, not the latency, bounds the stream)
    constexpr int kRingFit = 65536 / kSlotBytes;
    constexpr int kRing = kRingFit < 4 ? 4 : (kRingFit > 8 ? 8 : kRingFit);
    static_assert((kRing - 1) * kLoads <= 63, "vmcnt counts at most 63 loads");
    constexpr int kRingBytes = kRing * kSlotBytes;
    constexpr int kRedBytes = KW > 1 ? RW * 2 * CT * 4096 : 0;
    __shared__ __attribute__((aligned(16)))
    char lds[kRingBytes > kRedBytes ? kRingBytes : kRedBytes];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rw = wave % RW, kg = wave / RW;
    const int G = gridDim.x, id = blockIdx.x;
    // consecutive tile ids (same row blocks: the same weights) on one XCD
    const int tid = (G & 7) == 0 ? (id & 7) * (G >> 3) + (id >> 3) : id;
    const int bt = tid / mtiles, mt = tid - bt * mtiles;
    const int b = bt * RW + rw;
    const int m0 = mt * BM;
    const int Kp = KS * 64;
    const int run = (KS + KW - 1) / KW;
    const int cb = min(KS, kg * run), ce = min(KS, cb + run);
    const int T = (run + CH - 1) / CH;  // steps

    // weights of this wave's row block, chunks [0, ce) readable
    const __amdgpu_buffer_rsrc_t rw_res = buf(w + (size_t)b * KS * 1024, (uint32_t)ce * 1024u);
    const __amdgpu_buffer_rsrc_t rc_res =
        buf(codes + (size_t)m0 * Kp, (uint32_t)min(BM, M - m0) * (uint32_t)Kp);
    const uint32_t woff = (uint32_t)lane * 16u;
    const uint32_t coff = (uint32_t)((lane & 31) * Kp + (lane >> 5) * 16);

    // step i of this K group (chunks cb + CH*i + e) into ring slot i % kRing
    auto issue = [&](int i) {
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            char* slot = lds + (i % kRing) * kSlotBytes + kg * kGroupBytes + e * kChunkBytes;
            const int c = cb + CH * i + e;
            // past the group's run: an offset past both resources (reads zeros)
            const uint32_t cw = c < ce ? (uint32_t)c * 1024u + woff : 0x80000000u;
            to_lds16(rw_res, slot + kFrags * 1024 + rw * 1024, cw);
#pragma unroll
            for (int j = 0; j < kFrags / RW; ++j) {
                const int q = rw + RW * j, u = q >> 1, h = q & 1;
                const uint32_t cc = c < ce ? (uint32_t)c * 64u + (uint32_t)(u * 32 * Kp + h * 32) + coff
                                           : 0x80000000u;
                to_lds16(rc_res, slot + q * 1024, cc);
            }
        }
    };

    // Fragments of one step in registers: packed weight dwords (chunk e, row
    // tile t, MFMA step h) and the code fragments (chunk e, tile u, step h).
    struct Frag {
        uint32_t wd[CH][2][2];
        i4v B[CH][CT][2];
    };
    auto read = [&](int i, Frag& f) {
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            const char* slot = lds + (i % kRing) * kSlotBytes + kg * kGroupBytes + e * kChunkBytes;
#pragma unroll
            for (int u = 0; u < CT; ++u)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    f.B[e][u][h] =
                        *reinterpret_cast<const i4v*>(slot + (2 * u + h) * 1024 + lane * 16);
            const uint32_t* wrow = reinterpret_cast<const uint32_t*>(
                slot + kFrags * 1024 + rw * 1024 + (lane & 31) * 16 + (lane >> 5) * 4);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                f.wd[e][t][0] = wrow[t * 128];
                f.wd[e][t][1] = wrow[t * 128 + 2];
            }
        }
    };
    i16v acc[2][CT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < CT; ++u) acc[t][u] = i16v{};
    // The weight fields of the step's chunks x 2 row tiles x 2 MFMA steps,
    // then the MFMAs.
    auto unpack = [&](const Frag& f, i4v (&A)[CH][2][2]) {
#pragma unroll
        for (int e = 0; e < CH; ++e)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t wd = f.wd[e][t][h];
                    A[e][t][h] = i4v{(int)(wd & kField), (int)((wd >> 2) & kField),
                                     (int)((wd >> 4) & kField), (int)((wd >> 6) & kField)};
                }
    };
    auto mma = [&](const Frag& f, const i4v (&A)[CH][2][2]) {
#pragma unroll
        for (int e = 0; e < CH; ++e)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int u = 0; u < CT; ++u)
                        acc[t][u] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[e][t][h], f.B[e][u][h],
                                                                          acc[t][u], 0, 0, 0);
    };

    // Step j computes from registers while step j+1's fragments are read from
    // LDS and step j+kRing-1 is loaded into the slot of step j-1 (read at step
    // j-2, so free once every wave has passed this step's barrier). Step j's
    // weight fields are unpacked before step j+1's reads go out, so waiting for
    // its fragments does not wait for those reads. Steps run in pairs over two
    // register sets; an odd count ends on a zero step.
#pragma unroll
    for (int i = 0; i < kRing - 1; ++i) issue(i);
    wait_vm<(kRing - 2) * kLoads>();
    block_barrier();
    Frag f0, f1;
    i4v A[CH][2][2];
    read(0, f0);
    for (int j = 0; j < T; j += 2) {
        wait_vm<(kRing - 3) * kLoads>();  // step j+1 landed (this wave's loads)
        block_barrier();                   // and everyone's
        issue(j + kRing - 1);
        unpack(f0, A);
        issue_point();
        read(j + 1, f1);
        issue_point();  // the reads go out before the MFMAs
        mma(f0, A);
        __builtin_amdgcn_sched_barrier(0);  // the MFMAs stay ahead of the next barrier
        wait_vm<(kRing - 3) * kLoads>();
        block_barrier();
        issue(j + kRing);
        unpack(f1, A);
        issue_point();
        read(j + 2, f0);
        issue_point();
        mma(f1, A);
        __builtin_amdgcn_sched_barrier(0);
    }

    // the loads issued past the end (zeros) still write the ring: let them land
    // before the ring is reused or the workgroup's LDS is released
    wait_vm<0>();
    // K groups 1 .. KW-1 hand their tiles to group 0 one at a time through
    // one LDS buffer (RW * 2 * CT tiles of 4 KiB, over the ring)
    if (KW > 1) {
        i16v* red = reinterpret_cast<i16v*>(lds);
        for (int g = 1; g < KW; ++g) {
            __syncthreads();  // the ring (g = 1) or the buffer (g > 1) is free
            if (kg == g) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int u = 0; u < CT; ++u) red[((rw * 2 + t) * CT + u) * 64 + lane] = acc[t][u];
            }
            __syncthreads();
            if (kg == 0) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int u = 0; u < CT; ++u) acc[t][u] += red[((rw * 2 + t) * CT + u) * 64 + lane];
            }
        }
        if (kg > 0) return;
    }

    // C lane layout: token 32u + lane % 32, rows 32t + 8q + 4(lane / 32) + 0..3
    // in registers 4q .. 4q+3
#pragma unroll
    for (int u = 0; u < CT; ++u) {
        const int m = m0 + 32 * u + (lane & 31);
        if (m >= M) continue;
        const tenzo_hip_actq_t a = aq[m];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                finalize4(i4v{acc[t][u][4 * q], acc[t][u][4 * q + 1], acc[t][u][4 * q + 2],
                              acc[t][u][4 * q + 3]},
                          a, m, (int64_t)b * 64 + 32 * t + 8 * q + 4 * (lane >> 5), N, rs, y,
                          resid, acc_out);
    }
}

// The contraction for wide outputs. One workgroup = WR x WT x KW waves; a wave owns
// 32*RT rows x 32*CT tokens, the workgroup BN = 32*RT*WR rows x BM = 32*CT*WT
// tokens, and its KW K groups take turns of 128 columns (two super-chunks); their
// int32 tiles meet in LDS at the end. A step is one turn of every group. Its ring
// slot holds for each group
//   weights: BN/64 row blocks x 2 super-chunks of 1 KiB, as in memory (row r's
//            16-byte record at 16 r);
//   codes:   BM rows of 128 bytes; the 16-byte piece p (columns 16p .. 16p+15 of
//            the turn) of row r lies at place p ^ (r / 2 % 8) of its row.
// Both are filled by direct-to-LDS loads of 1 KiB, issued S - 1 steps ahead. A code
// load covers 8 whole 128-byte lines (lane l: row l / 8), so each line is looked up
// once; with the permuted places the 16 lanes of a fragment read that LDS serves
// together (16 rows, one piece) touch its 64 banks once each.
//
// MFMA operands (lane l = 32g + i), step h of super-chunk c:
//   A: row i of the tile, dword 2g + h of its record, unpacked;
//   B: token i, piece 4c + 2g + h.
// The codes are the MFMA's first operand, so that a register of the result holds one
// token's 32 consecutive rows in 32 lanes: every store is of whole 128-byte lines
// (1500 x 13824 outputs at K = 64: 18.6 us; with lanes along the tokens, 32 bytes of 32
// lines to a store, 21.2).
// Each super-chunk's fragments are read from LDS while the
// one before it is multiplied, and the next loads go out between the MFMAs.
template <int WR, int WT, int KW, int RT, int CT, int S, bool GLU>
__global__ void __launch_bounds__(64 * WR * WT * KW, 2)
tl1_mfma_wide_kernel(const uint8_t* __restrict__ w, const int8_t* __restrict__ codes,
                     const tenzo_hip_actq_t* __restrict__ aq, int M, int64_t N, int KS,
                     int mtiles, RowScales rs, float* __restrict__ y,
                     const float* __restrict__ resid, int32_t* __restrict__ acc_out) {
    constexpr int W = WR * WT * KW;
    constexpr int BN = 32 * RT * WR, BM = 32 * CT * WT;
    static_assert(BN % 64 == 0, "whole row blocks");
    constexpr int RB = BN / 64;
    static_assert(!GLU || (RT == 2 && RB % 2 == 0), "a gate tile and its up tile per wave");
    constexpr int kWLoads = 2 * RB, kGroup = kWLoads + BM / 8;  // loads of 1 KiB per group
    constexpr int kLoads = KW * kGroup;                         // and per step
    constexpr int kSlot = kLoads * 1024;
    constexpr int kFew = kLoads / W, kMore = kLoads % W;  // wave < kMore: one load more
    static_assert(S >= 3 && (S - 1) * (kFew + 1) <= 63, "vmcnt counts at most 63 loads");
    constexpr int kRed = (KW - 1) * WR * WT * RT * CT * 4096;
    constexpr int kRing = S * kSlot;
    __shared__ __attribute__((aligned(16))) char ring[kRing > kRed ? kRing : kRed];
    __shared__ __attribute__((aligned(16))) uint2 qs[BM];  // the tokens' {inv_scale, code sum}

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wave % WR, wt = wave / WR % WT, kg = wave / (WR * WT);
    const int G = gridDim.x, id = blockIdx.x;
    // consecutive tile ids (same row blocks: the same weights) on one XCD
    const int tid = (G & 7) == 0 ? (id & 7) * (G >> 3) + (id >> 3) : id;
    const int bt = tid / mtiles, mt = tid - bt * mtiles;
    const int nb = (int)(N >> 6);
    const int b0 = GLU ? 0 : bt * RB, m0 = mt * BM;
    const int Kp = KS * 64;
    for (int m = threadIdx.x; m < BM; m += 64 * W)
        qs[m] = m0 + m < M ? reinterpret_cast<const uint2*>(aq)[m0 + m] : make_uint2(0, 0);

    const uint32_t bstride = (uint32_t)KS * 1024u;
    // GLU: slot block r is gate block bt RB/2 + r, or its up block (RB/2 further on)
    const u4v rw_res = buf_words(w + (size_t)b0 * bstride,
                                 (uint32_t)(GLU ? nb : min(RB, nb - b0)) * bstride);
    auto block = [&](int r) {
        if (!GLU) return r;
        return bt * (RB / 2) + (r < RB / 2 ? r : (nb >> 1) + r - RB / 2);
    };
    const u4v rc_res = buf_words(codes + (size_t)m0 * Kp, (uint32_t)min(BM, M - m0) * (uint32_t)Kp);

    // This wave's loads of a step: their resource, byte offset (advanced from step to
    // step) and place in the slot. Steps past the end read other bytes of the
    // resources, or zeros past them, into places nobody reads.
    constexpr int X = kFew + (kMore ? 1 : 0);
    uint32_t off[X];
#pragma unroll
    for (int x = 0; x < X; ++x) {
        const int l = (wave + W * x) % kGroup, k = (wave + W * x) / kGroup;
        const int row = 8 * (l - kWLoads) + (lane >> 3);
        off[x] = l < kWLoads ? (uint32_t)block(l >> 1) * bstride +
                                   (uint32_t)(2 * k + (l & 1)) * 1024u + (uint32_t)lane * 16u
                             : (uint32_t)(row * Kp + 128 * k +
                                          (((lane & 7) ^ (row >> 1 & 7)) * 16));
    }
    auto load = [&](uint32_t slot, int x) {
        const int l = wave + W * x;
        if (x == kFew && wave >= kMore) return;
        const bool isw = l % kGroup < kWLoads;
        to_lds16_asm(isw ? rw_res : rc_res, slot + (uint32_t)l * 1024u, off[x]);
        off[x] += isw ? 2048u * KW : 128u * KW;
    };
    auto landed = [&]() {  // all but the last S - 3 steps' loads of this wave are in LDS
        if (kMore && wave < kMore) wait_vm_asm<(S - 3) * (kFew + 1)>();
        else wait_vm_asm<(S - 3) * kFew>();
    };

    i16v acc[RT][CT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int u = 0; u < CT; ++u) acc[t][u] = i16v{};

    const int i = lane & 31, g = lane >> 5;
    // the wave's row tile t as a tile of the slot: half tile % 2 of row block tile / 2
    auto tile = [&](int t) { return GLU ? t * WR + wr : wr * RT + t; };
    const uint32_t arow = (uint32_t)(kg * kGroup * 1024 + i * 16 + g * 8);
    const uint32_t brow = (uint32_t)((kg * kGroup + kWLoads) * 1024 + (wt * CT * 32 + i) * 128);
    const uint32_t bswz = (uint32_t)(((2 * g) ^ (i >> 1 & 7)) * 16);
    struct Frag {
        uint2 a[RT];
        i4v b[CT][2];
    };
    auto read = [&](const char* slot, int c, Frag& f) {  // super-chunk c of the turn
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const int rt = tile(t);
            f.a[t] = *reinterpret_cast<const uint2*>(slot + (rt >> 1) * 2048 + c * 1024 +
                                                     (rt & 1) * 512 + arow);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int u = 0; u < CT; ++u)
                f.b[u][h] = *reinterpret_cast<const i4v*>(slot + brow + u * 4096 +
                                                          (bswz ^ (uint32_t)((4 * c + h) * 16)));
    };
    // The super-chunk's MFMAs; the loads of a later step, if any, go out between them.
    auto mma = [&](const Frag& f, uint32_t slot, bool loads) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                const uint32_t wd = h ? f.a[t].y : f.a[t].x;
                const i4v a = i4v{(int)(wd & kField), (int)((wd >> 2) & kField),
                                  (int)((wd >> 4) & kField), (int)((wd >> 6) & kField)};
#pragma unroll
                for (int u = 0; u < CT; ++u)
                    acc[t][u] = __builtin_amdgcn_mfma_i32_32x32x32_i8(f.b[u][h], a, acc[t][u], 0, 0,
                                                                      0);
                if (loads) {
                    constexpr int kGroups = 2 * RT;
                    const int k = h * RT + t;
#pragma unroll
                    for (int x = 0; x < X; ++x)
                        if (x * kGroups / X == k) load(slot, x);
                }
            }
    };

    const uint32_t ring0 = lds_addr(ring);
    uint32_t in = ring0;  // slot of the next step to load
#pragma unroll
    for (int j = 0; j < S - 1; ++j) {
#pragma unroll
        for (int x = 0; x < X; ++x) load(in, x);
        in += kSlot;
    }
    const char* cur = ring;
    const char* nxt = ring + kSlot;
    Frag f0, f1;
    if (kMore && wave < kMore) wait_vm_asm<(S - 2) * (kFew + 1)>();
    else wait_vm_asm<(S - 2) * kFew>();
    block_barrier();
    read(cur, 0, f0);
    for (int s = 0; s < KS; s += 2 * KW) {  // super-chunk s + 2 kg is this group's next
        landed();  // the next step's loads, and everyone's; everyone has read the step before
        __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4));  // lgkmcnt(0)
        block_barrier();
        read(cur, 1, f1);
        issue_point();
        if (KW == 1 || s + 2 * kg < KS) mma(f0, in, true);
        issue_point();
        in = in == ring0 + (S - 1) * kSlot ? ring0 : in + kSlot;
        read(nxt, 0, f0);
        issue_point();
        if (s + 2 * kg + 1 < KS) mma(f1, 0, false);
        cur = nxt;
        nxt = nxt == ring + (S - 1) * kSlot ? ring : nxt + kSlot;
        __builtin_amdgcn_sched_barrier(0);  // the step's MFMAs stay ahead of the next barrier
    }
    wait_vm_asm<0>();  // the loads past the end still write the ring

    if (KW > 1) {  // groups 1 .. hand their tiles to group 0 through LDS, over the ring
        i16v* red = reinterpret_cast<i16v*>(ring);
        const int wv = wave % (WR * WT);
        __syncthreads();
        if (kg > 0) {
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int u = 0; u < CT; ++u)
                    red[((((kg - 1) * WR * WT + wv) * RT + t) * CT + u) * 64 + lane] = acc[t][u];
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int k = 0; k < KW - 1; ++k)
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int u = 0; u < CT; ++u)
                    acc[t][u] += red[(((k * WR * WT + wv) * RT + t) * CT + u) * 64 + lane];
    }

    // Lane (g, i) holds row 32 t + i of tokens 32 u + 8 q + 4 g + e in register 4 q + e.
    // Buffer stores: the rows of tokens past M lie past the resource and are dropped.
    const uint32_t ldy = (uint32_t)(GLU ? N / 2 : N) * 4u, ybytes = (uint32_t)min(BM, M - m0) * ldy;
    const int64_t y0 = (int64_t)m0 * (GLU ? N / 2 : N);
    const __amdgpu_buffer_rsrc_t ry = buf(y + y0, ybytes);
    const __amdgpu_buffer_rsrc_t rr = buf(resid ? resid + y0 : y, resid ? ybytes : 0);
    const __amdgpu_buffer_rsrc_t ra = buf(acc_out ? acc_out + y0 : (int32_t*)y, acc_out ? ybytes : 0);
    if (GLU) {  // act = max(0, gate)^2 * up (:1616-1620) of the two tiles' rows
        const int64_t row0 = (int64_t)bt * (BN / 2) + wr * 32;
        if (row0 >= N / 2) return;
#pragma unroll
        for (int u = 0; u < CT; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int ml = (wt * CT + u) * 32 + 8 * q + 4 * g;
                const uint4 a01 = *reinterpret_cast<const uint4*>(qs + ml);
                const uint4 a23 = *reinterpret_cast<const uint4*>(qs + ml + 2);
                const float inv[4] = {__uint_as_float(a01.x), __uint_as_float(a01.z),
                                      __uint_as_float(a23.x), __uint_as_float(a23.z)};
                const uint32_t cs[4] = {a01.y, a01.w, a23.y, a23.w};
                const uint32_t o = (uint32_t)ml * ldy + ((uint32_t)row0 + i) * 4u;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float gate = (float)(acc[0][u][4 * q + e] - (int)cs[e]) *
                                       __fmul_rn(inv[e], rs.scale[0]);
                    const float up = (float)(acc[RT - 1][u][4 * q + e] - (int)cs[e]) *
                                     __fmul_rn(inv[e], rs.scale[1]);
                    const float r = fmaxf(0.0f, gate);
                    __builtin_amdgcn_raw_buffer_store_b32(
                        __float_as_uint(__fmul_rn(__fmul_rn(r, r), up)), ry, o + e * ldy, 0, 0);
                }
            }
        return;
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const int64_t row0 = (int64_t)b0 * 64 + (wr * RT + t) * 32;
        if (row0 >= N) break;
        int sj = 0;
        while (sj < rs.n - 1 && row0 >= rs.end[sj]) ++sj;  // segment ends are multiples of 64
        const float wsc = rs.scale[sj];
#pragma unroll
        for (int u = 0; u < CT; ++u)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int ml = (wt * CT + u) * 32 + 8 * q + 4 * g;
                const uint4 a01 = *reinterpret_cast<const uint4*>(qs + ml);
                const uint4 a23 = *reinterpret_cast<const uint4*>(qs + ml + 2);
                const uint32_t inv[4] = {a01.x, a01.z, a23.x, a23.z};
                const uint32_t cs[4] = {a01.y, a01.w, a23.y, a23.w};
                const uint32_t o = (uint32_t)ml * ldy + ((uint32_t)row0 + i) * 4u;
                float r[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                if (resid)
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        r[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rr, o + e * ldy, 0, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int d = acc[t][u][4 * q + e] - (int)cs[e];
                    float out = (float)d * __fmul_rn(__uint_as_float(inv[e]), wsc);
                    if (resid) out = __fadd_rn(r[e], out);
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(out), ry, o + e * ldy, 0, 0);
                    if (acc_out) __builtin_amdgcn_raw_buffer_store_b32(d, ra, o + e * ldy, 0, 0);
                }
            }
    }
}

// Shapes of tl1_mfma_wide_kernel, by how many workgroups of each there would be for the
// 256 CUs. Small tiles with several K groups while one round of them covers the
// outputs, larger ones (fewer operand bytes and unpacked weights per product) as soon
// as they fill the chip. us at M x N x K (64x32 / 128x32 / 128x64 / 256x128 rows x tokens):
//   64 x 3840 x 2560     5.6   6.1   9.7  17.5   (120 workgroups of 64x32)
//   128 x 2560 x 6912    8.5  10.6  20.0  38.2   (160)
//   256 x 2560 x 6912   16.0  11.3  20.2  38.3   (320; 160 of 128x32)
//   512 x 2560 x 6912   23.6  17.6  22.2  38.9   (320 of 128x32)
//   1024 x 2560 x 6912  51.3  33.6  28.0  40.0   (640 of 128x32; 80 of 256x128)
//   1500 x 3840 x 2560  56.1  31.5  22.1  22.4   (180 of 256x128)
//   512 x 13824 x 2560  64.1  31.9  25.8  22.3   (216)
//   2048 x 13824 x 2560  250   123  94.5  71.1
// (tl1_mfma_kernel before it: 7.7, 12.1, 15.7, 23.1, 39.2, 26.4, 27.3 and 98.2.)
enum WideShape { kWide64x32, kWide128x32, kWide128x64, kWide256x128 };
WideShape wide_plan(int64_t M, int64_t N) {
    const int64_t nb = N / 64, m32 = ceil_div(M, 32);
    if (nb * m32 <= 256) return kWide64x32;
    if (ceil_div(nb, 2) * m32 <= 512) return kWide128x32;
    if (ceil_div(nb, 4) * ceil_div(M, 128) < 160) return kWide128x64;
    return kWide256x128;
}

template <int WR, int WT, int KW, int RT, int CT, int S, bool GLU>
int launch_wide(const int8_t* codes, const tenzo_hip_actq_t* q, const void* w_packed,
                const RowScales& rs, int64_t M, int64_t N, int64_t KS, float* y,
                const float* resid, int32_t* acc_out, hipStream_t st) {
    const int64_t mtiles = ceil_div(M, 32 * CT * WT);
    const int64_t grid = ceil_div(N, 32 * RT * WR) * mtiles;
    hipLaunchKernelGGL((tl1_mfma_wide_kernel<WR, WT, KW, RT, CT, S, GLU>), dim3((unsigned)grid),
                       dim3(64 * WR * WT * KW), 0, st, (const uint8_t*)w_packed, codes, q, (int)M,
                       N, (int)KS, (int)mtiles, rs, y, resid, acc_out);
    return launch_status("tl1_mfma_wide_kernel");
}

int launch_tl1_mfma(const int8_t* codes, const tenzo_hip_actq_t* q, const void* w_packed,
                    const RowScales& rs, int64_t M, int64_t N, int64_t K, float* y,
                    const float* resid, int32_t* acc_out, hipStream_t st, int tile) {
    const int64_t nb = N / 64, KS = ceil_div(K, 64);
    if (M * KS * 64 > (int64_t)INT32_MAX || K > (1 << 20) || nb * ceil_div(M, 32) > INT32_MAX) {
        set_error("tl1_mfma: unsupported shape (M=%lld N=%lld K=%lld tile=%d)", (long long)M,
                  (long long)N, (long long)K, tile);
        return TENZO_ERROR_INVALID_ARGUMENT;
    }
    // (its 32-bit offsets reach 128 rows of outputs)
    if (tile == 0 && N <= (1 << 22)) {
        switch (wide_plan(M, N)) {
            case kWide64x32:
                return launch_wide<2, 1, 4, 1, 1, 4, false>(codes, q, w_packed, rs, M, N, KS, y,
                                                            resid, acc_out, st);
            case kWide128x32:
                return launch_wide<4, 1, 2, 1, 1, 4, false>(codes, q, w_packed, rs, M, N, KS, y,
                                                            resid, acc_out, st);
            case kWide128x64:
                return launch_wide<2, 2, 1, 2, 1, 4, false>(codes, q, w_packed, rs, M, N, KS, y,
                                                            resid, acc_out, st);
            default:
                return launch_wide<4, 2, 1, 2, 2, 3, false>(codes, q, w_packed, rs, M, N, KS, y,
                                                            resid, acc_out, st);
        }
    }
    int KW = 4, RW = 1, CT = 1;  // (64 rows x 32 tokens)
    if (tile > 0) {              // forced shape of tl1_mfma_kernel: 100 * KW + 10 * RW + CT
        KW = tile / 100;
        RW = tile / 10 % 10;
        CT = tile % 10;
    }
    const int64_t mtiles = ceil_div(M, 32 * CT);
    const int64_t grid = (nb / (RW > 0 ? RW : 1)) * mtiles;
    if (RW <= 0 || nb % RW || grid > INT32_MAX) {
        set_error("tl1_mfma: unsupported shape (M=%lld N=%lld K=%lld tile=%d)", (long long)M,
                  (long long)N, (long long)K, tile);
        return TENZO_ERROR_INVALID_ARGUMENT;
    }

#define TL1_MFMA_CASE(KG, R, C)                                                               \
    if (KW == KG && RW == R && CT == C) {                                                     \
        hipLaunchKernelGGL((tl1_mfma_kernel<R, KG, C>), dim3((unsigned)grid),                 \
                           dim3(64 * R * KG), 0, st, (const uint8_t*)w_packed, codes, q,      \
                           (int)M, N, (int)KS, (int)mtiles, rs, y, resid, acc_out);           \
        return launch_status("tl1_mfma_kernel");                                              \
    }
    TL1_MFMA_CASE(1, 4, 2) TL1_MFMA_CASE(2, 4, 2) TL1_MFMA_CASE(4, 4, 2)
    TL1_MFMA_CASE(2, 2, 2) TL1_MFMA_CASE(4, 2, 2) TL1_MFMA_CASE(2, 2, 1) TL1_MFMA_CASE(4, 2, 1)
    TL1_MFMA_CASE(4, 1, 2) TL1_MFMA_CASE(4, 1, 1) TL1_MFMA_CASE(8, 1, 1)
#undef TL1_MFMA_CASE
    set_error("tl1_mfma: no kernel for tile KW=%d RW=%d CT=%d", KW, RW, CT);
    return TENZO_ERROR_INVALID_ARGUMENT;
}

bool tl1_mfma_glu_fits(int64_t M, int64_t F, int64_t K) {
    const int64_t KS = ceil_div(K, 64);
    // (32-bit offsets over the whole weight matrix and over 128 rows of outputs)
    return F % 64 == 0 && 2 * F <= (1 << 22) && M * KS * 64 <= (int64_t)INT32_MAX &&
           K <= (1 << 20) && F / 32 * KS * 1024 < (int64_t)UINT32_MAX;
}

int launch_tl1_mfma_glu(const int8_t* codes, const tenzo_hip_actq_t* q, const void* w_packed,
                        float gate_scale, float up_scale, int64_t M, int64_t F, int64_t K,
                        float* act, hipStream_t st) {
    const int64_t N = 2 * F, nb = N / 64, KS = ceil_div(K, 64);
    RowScales rs{};
    rs.n = 2;
    rs.end[0] = F;
    rs.end[1] = INT64_MAX;
    rs.scale[0] = gate_scale;
    rs.scale[1] = up_scale;
    // Shapes as for the plain product, two row tiles to a wave (one of each matrix).
    // us at 13824 x 2560 (128x32 / 128x64 with two K groups / 128x64 / 256x128): 20 tokens
    // 6.5 8.0 8.9 16.3; 128 tokens 9.3 8.8 9.5 16.5; 256 17.3 16.0 13.1 18.2; 512 29.2
    // 30.9 23.8 20.8; 2048 113 121 84.8 65.6 (the plain product: 71.1 and a row twice as
    // long for the quantizer to read).
    if (ceil_div(nb, 2) * ceil_div(M, 32) <= 256)
        return launch_wide<2, 1, 2, 2, 1, 4, true>(codes, q, w_packed, rs, M, N, KS, act, nullptr,
                                                   nullptr, st);
    if (ceil_div(nb, 2) * ceil_div(M, 64) <= 256)
        return launch_wide<2, 2, 2, 2, 1, 4, true>(codes, q, w_packed, rs, M, N, KS, act, nullptr,
                                                   nullptr, st);
    if (ceil_div(nb, 4) * ceil_div(M, 128) < 160)
        return launch_wide<2, 2, 1, 2, 1, 4, true>(codes, q, w_packed, rs, M, N, KS, act, nullptr,
                                                   nullptr, st);
    return launch_wide<4, 2, 1, 2, 2, 3, true>(codes, q, w_packed, rs, M, N, KS, act, nullptr,
                                               nullptr, st);
}

}  // namespace tz

using namespace tz;

extern "C" {

TENZO_HIP_API int tenzo_hip_bitlinear_tl1_batch(const int8_t* codes, const tenzo_hip_actq_t* q,
                                                const void* w_packed, float w_scale, int64_t M,
                                                int64_t N, int64_t K, float* y,
                                                int32_t* acc_out, int tile, void* stream) {
    TZ_CHECK(codes && q && w_packed && y, "bitlinear_tl1_batch: null pointer");
    TZ_CHECK(M > 0 && N > 0 && N % 64 == 0 && K > 0 && tile >= 0,
             "bitlinear_tl1_batch: need M > 0, N %% 64 == 0, K > 0 (M=%lld N=%lld K=%lld)",
             (long long)M, (long long)N, (long long)K);
    RowScales rs = RowScales::single(w_scale);
    return launch_tl1_mfma(codes, q, w_packed, rs, M, N, K, y, nullptr, acc_out,
                           (hipStream_t)stream, tile);
}

}  // extern "C"
