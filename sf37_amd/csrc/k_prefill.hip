// k_prefill.hip - routed experts for many tokens per expert (prefill) on
// the gfx950 matrix cores.
//
// Same results as the grouped dot-product kernels of k_moe.hip, bit for bit:
// the integer group sums I_g = sum (q - zp) * qs are formed exactly by the
// matrix cores, and the float epilogue is the canonical chain of the Q8_K path
//   blk = fma(s3,I3, fma(s2,I2, fma(s1,I1, fma(s0,I0,0))));  acc = fma(d_b, blk, acc)
// (sf37_cuda.cu:4226-4274 sums the same integers; this build fixes the order).
//
// Exactness.  The operands are 6-bit floats (v_mfma_f32_32x32x64_f8f6f4), one
// MFMA instruction spanning one 64-group.  A 3- or 2-bit weight code in the
// low bits of an E2M3 field is that code times 1/8 (E2M3 is linear up to
// 15/8), so dequantising is a mask per dword.  An activation code |qs| <= 128
// is split as qs = 16 h + l with the sign of qs on both: l (0..15) is linear
// in E2M3 (l/8), h (0..8) is exact in E3M2 as 2h.  The two MFMAs of a group
// add 2h * q/8 and l/8 * q/8, together q * qs / 64, and a third one (fp16,
// K = 8) starts the accumulator at -zp * gsum / 64, gsum = sum qs cut into
// two exact fp16 parts.  Every partial sum is a multiple of 1/64 below
// 2^18, exact in fp32 in any order, so D = I_g / 64, and fma(64 s_g, D, blk)
// rounds the same value as fma(s_g, I_g, blk).
//
// Why 6 bits: measured per SIMD (four waves, ns), a 64-group of a 32 x 32
// tile takes 65 as four fp16 32x32x16 MFMAs and 51 as these three, and the
// time of the VALU operations adds to it (about 1 ns each, hardly any
// overlap), so what counts is the sum: the fp16 operands took 1.5 VALU
// operations per weight code to dequantise, these 0.3-0.4.  Gate/up and down
// at 4096 tokens: 1153 + 626 us with fp16 operands, 885 + 495 now; 187 tokens
// (groups of ~5 pairs) 491 + 220 -> 336 + 142 us.  What bounds them: at 4096
// tokens about half of the time is MFMA and VALU issue, the rest waits for
// loads: a weight load touches all 32 rows of its lanes, so the address units
// are ~70 % busy (no weight loads: 700 us; weights through LDS tiles by
// direct loads, whole runs of a row at a time: 1020 us, the words' LDS reads
// cost more than that saves).
//
// Layouts.  Activations are re-quantised to Q8_K (sf37_cuda.cu:4168-4205,
// bit-exact) and written per (row, 256-block) as 384 bytes of 6-bit fields
// (24 16-byte pieces in the order the LDS reads want, below), the four
// groups' -gsum/64 as fp16 pairs and the scale d.  A workgroup owns (tile of
// <= 64 pairs of one expert, row tile); it stages the tile's blocks in LDS by
// direct global->LDS loads (two buffers, one block ahead), each wave loads
// its own weight rows into registers one block ahead, dequantises a block at
// once (24 registers) and runs the MFMAs over the tile's 32-pair blocks.
#include <type_traits>

#include "sf37_blocks.h"
#include "sf37_dispatch.h"
#include "sf37_launch.h"

namespace {

typedef _Float16 h4v __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr uint32_t PF_T = 64;           // pairs per tile
constexpr uint32_t PF_NW = 4;           // waves per workgroup, 32 weight columns each
constexpr uint32_t PF_GU_R = 16u * PF_NW;   // F rows per workgroup (16 gate + 16 up columns per wave)
constexpr uint32_t PF_DN_R = 32u * PF_NW;   // output rows per workgroup
// One (row, 256-block) of activations: 24 pieces of 16 bytes.  Group g, lane
// half kh (codes 32 kh .. 32 kh + 31 of the group) has 12 dwords: the E3M2
// fields of h (6 dwords), then the E2M3 fields of l; its piece j (0..2) is
// c = 3 g + j, stored as piece 8 (c / 4) + 2 (c % 4) + kh.  In LDS, piece
// 8 k + s of tile slot t is at k * PF_CHUNK + 128 t + 16 (s ^ (t % 8)): eight
// lanes reading one piece of eight slots touch all banks, and a 64-lane
// direct load fills eight slots' 128 contiguous bytes.
constexpr uint32_t PF_BLK = 384;
// ... and a record: the four groups' -gsum/64 as fp16 pairs, d, padding.
constexpr uint32_t PF_REC = 32;
constexpr uint32_t PF_CHUNK = PF_T * 128u;
constexpr uint32_t PF_ACT_BUF = 3u * PF_CHUNK;
static_assert(PF_BLK == SF37_QK * 12u / 8u && PF_BLK == 3u * 128u, "256 codes of 12 bits, three chunks");

// Extents of the LDS direct loads.  A global_load_lds writes its 64 lanes'
// bytes at M0 + 16 * lane (dwordx4) or M0 + 4 * lane (dword) whatever the
// source address, so every M0 a kernel forms must leave a whole 64-lane span
// inside the buffer it targets.
constexpr uint32_t DMA16_SPAN = 64u * 16u;
constexpr uint32_t DMA4_SPAN = 64u * 4u;
// pf_expert codes: M0 = buffer + k * PF_CHUNK + r8 * 1024, chunk k <= 2, slot
// octet r8 <= PF_T / 8 - 1
static_assert(DMA16_SPAN == 8u * 128u && 2u * PF_CHUNK + (PF_T / 8u - 1u) * DMA16_SPAN + DMA16_SPAN <= PF_ACT_BUF,
              "pf_expert code loads stay in their buffer");
static_assert(PF_T / 8u == 2u * PF_NW, "each wave loads two slot octets (one per 32-pair block)");
static_assert(PF_T * 16u == DMA16_SPAN && PF_T * 4u == DMA4_SPAN,
              "pf_expert group-sum and scale loads fill exactly one buffer row each");

// ---------------------------------------------------------------------------
// 6-bit fields.  A half-group's 32 fields are two 96-bit strings of 16: Q3,
// the even codes (field i = code 2 i) and the odd ones (code 2 i + 1), so a
// string is the lane's 96 payload bits (shifted by 3 for the odd codes) under
// one mask; Q2, the codes of payload dword 0 and of dword 1, each dword
// masked three ways: a 2-bit code keeps its bit in the dword, and codes 0, 3,
// 6 .. 15 are fields of the string's first dword, 2, 5 .. 14 of the second,
// 1, 4 .. 13 of the third.
// ---------------------------------------------------------------------------
// mask of dword k of a string whose fields hold `bits`-bit codes
__host__ __device__ constexpr uint32_t pf_mask(uint32_t k, uint32_t bits) {
    uint32_t m = 0;
    for (uint32_t i = 0; i < 32u; i++)
        if ((32u * k + i) % 6u < bits) m |= 1u << i;
    return m;
}
static_assert((pf_mask(0, 2) | pf_mask(1, 2) | pf_mask(2, 2)) == 0xffffffffu &&
                  (pf_mask(0, 2) & pf_mask(1, 2)) == 0 && (pf_mask(0, 2) & pf_mask(2, 2)) == 0,
              "the three masks split a dword of 2-bit codes");

// lanes exchanged within quads: xor 1 and xor 2
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_quad(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
constexpr int QUAD_XOR1 = 0xB1, QUAD_XOR2 = 0x4E;

// ---------------------------------------------------------------------------
// Activation kernel: Q8_K of one (row, 256-block) per wave, the codes as
// 6-bit fields, -gsum/64 of the four groups and d.
// ---------------------------------------------------------------------------
// A wave's units u0, u0 + stride, ..; row: PF_BLK bytes of LDS of its own.
template <bool Q3>
__device__ __forceinline__ void pf_act_units(uint32_t *__restrict__ codes, uint32_t *__restrict__ rec,
                                             const float *__restrict__ x, uint32_t units, uint32_t u0,
                                             uint32_t stride, uint8_t *row) {
    const uint32_t lane = threadIdx.x & 63u;
    // the lane's half-group (48 bytes), its quad in it, its place in the quad
    const uint32_t hb = (lane >> 3) * 48u, quad = (lane >> 2) & 1u, qj = lane & 3u;
    // piece `lane` (lanes < 24) of the output from the half-group order
    const uint32_t pc = 4u * (lane >> 3) + ((lane & 7u) >> 1);
    const uint32_t piece = (2u * (pc / 3u) + (lane & 1u)) * 48u + 16u * (pc % 3u);
    for (uint32_t u = u0; u < units; u += stride) {
        const float4 xv = *(const float4 *)(x + (uint64_t)u * SF37_QK + 4u * lane);
        const float v[4] = {xv.x, xv.y, xv.z, xv.w};
        int8_t q[4];
        int gsum;
        const float d = q8k_codes4(v, q, gsum);
        // magnitudes and signs, a byte per code; h = magnitude / 16, l the rest
        uint32_t m = 0, sg = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int a = q[k];
            m |= (uint32_t)(a < 0 ? -a : a) << (8 * k);
            sg |= (a < 0 ? 0x20u : 0u) << (8 * k);
        }
        const uint32_t hm = (m >> 4) & 0x0f0f0f0fu, h8 = hm & 0x08080808u;
        // E3M2 of 2 h: 0, 16, 20, 22, 24, 25, 26, 27 by table, 28 for h = 8
        // (for which the byte select reads the sign of 0x10: zero)
        uint32_t eh = vperm(0x1B1A1918u, 0x16141000u, hm);
        eh |= (h8 >> 1) | h8 | (h8 << 1) | sg;
        const uint32_t el = (m & 0x0f0f0f0fu) | sg;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the previous unit's reads are done
        if constexpr (Q3) {
#pragma unroll
            for (uint32_t k = 0; k < 4u; k++) {   // even h, odd h, even l, odd l
                const uint32_t e = k < 2u ? eh : el;
                const uint32_t two = (k & 1u) ? ((e >> 8) & 0x3fu) | ((e >> 18) & 0xfc0u)
                                              : (e & 0x3fu) | ((e >> 10) & 0xfc0u);
                uint32_t w = two << (12u * (lane & 1u));
                w |= dpp_quad<QUAD_XOR1>(w);                       // 24 bits of the lane pair
                const uint32_t t = dpp_quad<QUAD_XOR2>(w);         // the other pair's
                if (qj == 0u) {                                    // 48 bits of the quad
                    uint16_t *o = (uint16_t *)(row + hb + 12u * k + 6u * quad);
                    const uint32_t lo = w | (t << 24);
                    o[0] = (uint16_t)lo;
                    o[1] = (uint16_t)(lo >> 16);
                    o[2] = (uint16_t)(t >> 8);
                }
            }
        } else {
#pragma unroll
            for (uint32_t k = 0; k < 2u; k++) {   // h, l
                const uint32_t e = k ? el : eh;
                // the lane's codes 4 qj .. 4 qj + 3 by the dword of the string
                // they go to: X0 has codes 0 and 3, X1 code 1, X2 code 2
                const uint32_t x0 = (e & 0x3fu) | ((e >> 18) & 0xfc0u), x1 = ((e >> 8) & 0x3fu) << 2,
                               x2 = ((e >> 16) & 0x3fu) << 4;
                const uint32_t r0 = qj == 1u ? x2 : qj == 2u ? x1 : x0;
                const uint32_t r1 = qj == 1u ? x1 : qj == 2u ? x0 : x2;
                const uint32_t r2 = qj == 1u ? x0 : qj == 2u ? x2 : x1;
                uint32_t d0 = r0 << (8u * qj), d1 = r1 << (8u * qj), d2 = r2 << (8u * qj);
                // fields of codes 15 and 14 that run into the next dword
                d1 |= qj == 3u ? x0 >> 8 : 0u;
                d2 |= qj == 3u ? x2 >> 8 : 0u;
                d0 |= dpp_quad<QUAD_XOR1>(d0);
                d1 |= dpp_quad<QUAD_XOR1>(d1);
                d2 |= dpp_quad<QUAD_XOR1>(d2);
                d0 |= dpp_quad<QUAD_XOR2>(d0);
                d1 |= dpp_quad<QUAD_XOR2>(d1);
                d2 |= dpp_quad<QUAD_XOR2>(d2);
                if (qj < 3u) *(uint32_t *)(row + hb + 24u * k + 12u * quad + 4u * qj) = qj == 0u ? d0 : qj == 1u ? d1 : d2;
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // this unit's fields are in LDS
        __builtin_amdgcn_wave_barrier();
        if (lane < 24u) *(uint4 *)((uint8_t *)codes + (uint64_t)u * PF_BLK + 16u * lane) = *(const uint4 *)(row + piece);
        if ((lane & 15u) == 0u) {
            const _Float16 hi = (_Float16)((float)(gsum >> 4) * -0.25f), lo = (_Float16)((float)(gsum & 15) * -0.015625f);
            rec[(uint64_t)u * (PF_REC / 4u) + (lane >> 4)] = (uint32_t)__builtin_bit_cast(unsigned short, hi) |
                                                             (uint32_t)__builtin_bit_cast(unsigned short, lo) << 16;
        }
        if (lane == 0u) rec[(uint64_t)u * (PF_REC / 4u) + 4u] = __builtin_bit_cast(uint32_t, d);
    }
}

// Each wave owns its LDS row and walks the (row, block) units wave by wave
// over the grid; nothing is shared between waves.
template <bool Q3>
__global__ void __launch_bounds__(256) pf_act_kernel(uint32_t *__restrict__ codes, uint32_t *__restrict__ rec,
                                                     const float *__restrict__ x, uint32_t nblk, uint32_t n_rows) {
    __shared__ __align__(16) uint8_t st[4][PF_BLK];
    const uint32_t wv = threadIdx.x >> 6;
    pf_act_units<Q3>(codes, rec, x, nblk * n_rows, blockIdx.x * 4u + wv, gridDim.x * 4u, st[wv]);
}

// What the gate/up launch of a small batch needs, in one launch: workgroup 0
// sorts the pairs by expert and lists the tiles, the others write the rows'
// operands.  Each of the three is latency-bound, about 5 us with its launch.
// Measured per layer, three launches / one: 21 tokens 265 / 258 us, 64 tokens
// 155 / 150, 187 tokens 530 / 523.  At 512 tokens (4096 pairs) 370 / 375: the
// 1024-thread workgroups then wait for whole CUs that the shared expert's
// GEMM holds on its stream, which the 256-thread ones of pf_act_kernel do
// not, so the line is at PF_START_PAIRS pairs.
constexpr uint32_t PF_START_PAIRS = 2048;
static_assert(PF_START_PAIRS <= DISP_ONE_PAIRS, "one workgroup sorts them");
__global__ void __launch_bounds__(1024) pf_start_kernel(uint32_t *__restrict__ codes, uint32_t *__restrict__ rec,
                                                        const float *__restrict__ x, uint32_t units,
                                                        uint32_t *__restrict__ group_info,
                                                        uint32_t *__restrict__ sorted, uint32_t *__restrict__ counts,
                                                        uint32_t *__restrict__ offsets, uint32_t *__restrict__ tiles,
                                                        const int32_t *__restrict__ selected, uint32_t n_pairs,
                                                        uint32_t n_expert) {
    __shared__ __align__(16) uint8_t st[16][PF_BLK];
    if (blockIdx.x == 0u) {
        dispatch_pairs<PF_T>(group_info, sorted, counts, offsets, tiles, selected, n_pairs, n_expert);
        return;
    }
    const uint32_t wv = threadIdx.x >> 6;
    pf_act_units<true>(codes, rec, x, units, (blockIdx.x - 1u) * 16u + wv, (gridDim.x - 1u) * 16u, st[wv]);
}

// ---------------------------------------------------------------------------
// Tile list: every group split into tiles of <= PF_T pairs.
// tiles[0] = count; tile t at uint4 index 1 + t = {expert, first pair, count, 0}.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(1024) pf_tiles_kernel(uint32_t *__restrict__ tiles,
                                                        const uint32_t *__restrict__ ginfo,
                                                        uint32_t max_groups) {
    __shared__ uint32_t wsum[16];
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63u;
    const uint32_t ng = ginfo[0];
    uint32_t base = 0;
    for (uint32_t g0 = 0; g0 < ng; g0 += 1024u) {
        const uint32_t g = g0 + tid;
        uint32_t nt = 0, p0 = 0, cnt = 0;
        if (g < ng) {
            p0 = ginfo[1 + g];
            cnt = ginfo[2 + g] - p0;
            nt = (cnt + PF_T - 1u) / PF_T;
        }
        uint32_t sc = nt;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t a = __shfl_up(sc, o, 64);
            if (lane >= (uint32_t)o) sc += a;
        }
        if (lane == 63u) wsum[wave] = sc;
        __syncthreads();
        uint32_t before = base, all = 0;
        for (uint32_t w = 0; w < 16u; w++) {
            if (w < wave) before += wsum[w];
            all += wsum[w];
        }
        const uint32_t first = before + sc - nt;
        if (g < ng) {
            const uint32_t e = ginfo[2 + max_groups + g];
            for (uint32_t k = 0; k < nt; k++) {
                const uint32_t c = cnt - k * PF_T < PF_T ? cnt - k * PF_T : PF_T;
                ((uint4 *)tiles)[1 + first + k] = make_uint4(e, p0 + k * PF_T, c, 0u);
            }
        }
        base += all;
        __syncthreads();
    }
    if (tid == 0) tiles[0] = base;
}

// ---------------------------------------------------------------------------
// LDS direct loads (global -> LDS, no registers).  Issued through inline asm
// so the compiler does not wait for them before unrelated LDS reads; the
// kernel waits with s_waitcnt vmcnt(0) + barrier before reading the buffer.
// Lane i of a dwordx4 load writes LDS bytes [m0 + 16 i, m0 + 16 i + 16);
// one wait state separates the M0 write from the load.  m0 cannot be named
// as a clobber (the compiler reserves it and drops such a clobber), so these
// sequences rely on no compiler-generated code of these kernels reading m0:
// in the gfx950 assembly of this file every m0 access is one of these
// s_mov_b32 writes (no movrel, gpr-index or sendmsg use).
// ---------------------------------------------------------------------------
// sbase must be wave-uniform; it is moved to SGPRs with readfirstlane.
__device__ __forceinline__ uint64_t sgpr_ptr(const void *p) {
    const uint64_t v = (uint64_t)(uintptr_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ void lds_dma16(uint32_t lds, uint32_t voff, const void *sbase) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds)),
                 "v"(voff), "s"(sgpr_ptr(sbase))
                 : "memory");
}
__device__ __forceinline__ void lds_dma4(uint32_t lds, uint32_t voff, const void *sbase) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds)),
                 "v"(voff), "s"(sgpr_ptr(sbase))
                 : "memory");
}
__device__ __forceinline__ void wait_vm0() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ uint32_t lds_addr(const void *p) { return (uint32_t)(uintptr_t)p; }

// Direct loads of a block's records, a slot per lane: wave 0 the group sums,
// wave 1 the scales.  One asm statement with the branches inside, so that the
// code around it stays one block for the compiler (which otherwise moves the
// fmas before a branch behind it).
__device__ __forceinline__ void pf_rec_load(uint32_t wave, uint32_t gs_lds, uint32_t d_lds, uint32_t voff,
                                            const uint8_t *rec) {
    asm volatile("s_cmp_lg_u32 %0, 0\n\t"
                 "s_cbranch_scc1 .Lpfg%=\n\t"
                 "s_mov_b32 m0, %1\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dwordx4 %3, %4\n"
                 ".Lpfg%=:\n\t"
                 "s_cmp_lg_u32 %0, 1\n\t"
                 "s_cbranch_scc1 .Lpfd%=\n\t"
                 "s_mov_b32 m0, %2\n\t"
                 "s_nop 0\n\t"
                 "global_load_lds_dword %3, %5\n"
                 ".Lpfd%=:" ::"s"(__builtin_amdgcn_readfirstlane(wave)),
                 "s"(__builtin_amdgcn_readfirstlane(gs_lds)), "s"(__builtin_amdgcn_readfirstlane(d_lds)), "v"(voff),
                 "s"(sgpr_ptr(rec)), "s"(sgpr_ptr(rec + 16))
                 : "memory", "scc");
}

struct pf_params {
    float *mid, *gate_out, *up_out, *down_pair;
    const uint8_t *w0, *w1;        // gate / up (Q3) or down (Q2)
    const uint8_t *act;            // [rows][nblk][PF_BLK] fields
    const uint8_t *rec;            // [rows][nblk][PF_REC]
    const uint32_t *tiles;
    const uint32_t *sorted;
    const float *weights;
    uint32_t topk, nblk, out_rows, n_rt;
    float clamp;
    const uint8_t *s0, *s1;        // the same of expert sh_id, which has tensors of its own
    uint32_t sh_id;
    float sh_clamp;
};

// Weight bytes of one lane for one Q3 block: the header dwords (scales, zero
// points) and per group the aligned dwords that hold the half's 12 bytes:
// three of each when the block starts on a dword, four in an odd block, which
// starts two bytes in.
// (Vector types, so that the loop carries each load's result as the register
// tuple it was loaded into: as single words they are copied at the end of an
// iteration, which waits for them there.)
typedef uint32_t u32x4a __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x3a __attribute__((ext_vector_type(3), aligned(4)));
template <bool ODD> struct q3_raw {
    typedef typename std::conditional<ODD, u32x4a, u32x3a>::type vec;
    vec h, w[4];
};

// hp: the header's first dword (odd blocks: two bytes before the block); pp:
// the dword at which group 0's payload starts
template <bool ODD>
__device__ __forceinline__ void q3_load(q3_raw<ODD> &r, const uint8_t *hp, const uint8_t *pp) {
    typedef typename q3_raw<ODD>::vec vec;
    r.h = *(const vec *)hp;
#pragma unroll
    for (int g = 0; g < 4; g++) r.w[g] = *(const vec *)(pp + 24 * g);
}

// After a wait for them, mark a block's weight words as just defined: the
// compiler then knows no load is pending on them and places no s_waitcnt
// vmcnt of its own inside the compute (which would also wait for the loads
// and LDS direct loads issued since).
template <bool ODD>
__device__ __forceinline__ void raw_ready(q3_raw<ODD> &r) {
    asm volatile("" : "+v"(r.h), "+v"(r.w[0]), "+v"(r.w[1]), "+v"(r.w[2]), "+v"(r.w[3]));
}

struct q2_raw {
    uint32_t h[3];
    uint32_t w[4][2];
};
// What a lane loads of a Q2 block (21 dwords): dwords 8 kh .. 8 kh + 10,
// contiguous (three loads instead of eleven); pf_words then trades what each
// half needs from the other with v_permlane32_swap (lanes l and l + 32 hold
// the same row).
struct q2_half {
    u32x4a a, b;
    u32x3a c;
};
__device__ __forceinline__ void raw_ready(q2_half &r) { asm volatile("" : "+v"(r.a), "+v"(r.b), "+v"(r.c)); }
__device__ __forceinline__ void q2_load_half(q2_half &r, const uint8_t *bp, uint32_t kh) {
    const uint32_t *q = (const uint32_t *)bp + 8u * kh;
    r.a = *(const u32x4a *)q;
    r.b = *(const u32x4a *)(q + 4);
    r.c = *(const u32x3a *)(q + 8);
}
// q2_raw of both halves: the header dwords 0..2 and group g's dwords
// 3 + 4 g + 2 kh, +1.  permlane32_swap(A, B) gives [A of lanes 0-31, B of
// lanes 0-31] and [A of lanes 32-63, B of lanes 32-63]; with A, B = loaded
// dwords (3, 5), (4, 6), (7, 9), (8, 10) the first is a word of group 0 or 1
// for both halves, the second the same word of group 2 or 3 (8 dwords on);
// a swap of dword j with itself hands both halves header dword j.
__device__ __forceinline__ q2_raw pf_words(const q2_half &h) {
    const uint32_t w[11] = {h.a[0], h.a[1], h.a[2], h.a[3], h.b[0], h.b[1], h.b[2], h.b[3], h.c[0], h.c[1], h.c[2]};
    q2_raw r;
#pragma unroll
    for (int j = 0; j < 3; j++) r.h[j] = __builtin_amdgcn_permlane32_swap(w[j], w[j], false, false)[0];
#pragma unroll
    for (int g = 0; g < 2; g++) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const auto v = __builtin_amdgcn_permlane32_swap(w[3 + 4 * g + i], w[5 + 4 * g + i], false, false);
            r.w[g][i] = v[0];
            r.w[g + 2][i] = v[1];
        }
    }
    return r;
}
// f16 scale of group g, zero point of group g from the header bits at SH.
template <int SH, typename H>
__device__ __forceinline__ float hdr_scale(const H &h, int g) {
    const int a = SH + 16 * g;
    return sf37_f16(h[a >> 5] >> (a & 31));
}
template <int SH>
__device__ __forceinline__ uint32_t hdr_zp(const uint32_t *h, int g) {
    const int a = SH + 64 + 8 * g;
    return (h[a >> 5] >> (a & 31)) & 0xffu;
}

// A block's weight words into r.
template <bool Q3, bool ODD> using pf_raw_t = typename std::conditional<Q3, q3_raw<ODD>, q2_half>::type;
template <bool Q3, bool ODD>
__device__ __forceinline__ void pf_wload(pf_raw_t<Q3, ODD> &r, const uint8_t *wrow, uint32_t bn, uint32_t kh) {
    if constexpr (Q3) {
        const uint8_t *hp = wrow + (uint64_t)SF37_Q3_BYTES * bn - (ODD ? 2 : 0);
        q3_load<ODD>(r, hp, hp + 12u + 12u * kh);
    } else {
        q2_load_half(r, wrow + (uint64_t)SF37_Q2_BYTES * bn, kh);
    }
}

// All of the wave's vector-memory operations done but the newest block of
// weight words (the loads pf_wload makes: five, or three for Q2).
template <bool Q3>
__device__ __forceinline__ void wait_vm_keep_weights() {
    if constexpr (Q3) asm volatile("s_waitcnt vmcnt(5)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(3)" ::: "memory");
}

// A block's weights as MFMA operands: 4 groups x 32 columns x 64 codes.
struct pf_b {
    uint32_t w[4][6];   // E2M3 fields, code / 8
    uint32_t z[4];      // zp as an fp16 pair (lane half 0; zero in half 1)
    float s[4];         // 64 x the group's scale
};

// zt: fp16 high bytes of 0..7 for the zero points (zero in lane half 1, whose
// share of the fp16 MFMA's K is unused)
template <bool Q3, int SH, typename RAW>
__device__ __forceinline__ void pf_dequant(pf_b &o, const RAW &r, const uint32_t zt[2]) {
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const auto w = r.w[g];
        if constexpr (Q3) {
            constexpr uint32_t m0 = pf_mask(0, 3), m1 = pf_mask(1, 3), m2 = pf_mask(2, 3);
            if constexpr (SH == 0) {
                o.w[g][0] = w[0] & m0;
                o.w[g][1] = w[1] & m1;
                o.w[g][2] = w[2] & m2;
                o.w[g][5] = (w[2] >> 3) & m2;
            } else {
                o.w[g][0] = align_bits(w[1], w[0], SH) & m0;
                o.w[g][1] = align_bits(w[2], w[1], SH) & m1;
                o.w[g][2] = align_bits(w[3], w[2], SH) & m2;
                o.w[g][5] = align_bits(w[3], w[2], SH + 3) & m2;
            }
            o.w[g][3] = align_bits(w[1], w[0], SH + 3) & m0;
            o.w[g][4] = align_bits(w[2], w[1], SH + 3) & m1;
        } else {
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (uint32_t k = 0; k < 3u; k++) o.w[g][3 * j + k] = w[j] & pf_mask(k, 2);
        }
    }
    const uint32_t zps = (SH ? align_bits(r.h[SH ? 3 : 2], r.h[2], SH) : r.h[2]) & (Q3 ? 0x07070707u : 0x03030303u);
    const uint32_t zh = vperm(zt[1], zt[0], zps);
#pragma unroll
    for (uint32_t g = 0; g < 4u; g++) {
        o.z[g] = vperm(zh, zh, g << 8 | g << 24 | 0x000c000cu);
        o.s[g] = 64.0f * hdr_scale<SH>(r.h, (int)g);
    }
}

typedef int v8i __attribute__((ext_vector_type(8)));
constexpr int FMT_E2M3 = 2, FMT_E3M2 = 3;
// D += A (format FA) x B (E2M3) over one 64-group; only the first six dwords
// of each operand are read, and zero scale operands select the unscaled form
template <int FA>
__device__ __forceinline__ f16v pf_mfma6(const uint32_t *a, const uint32_t *b, f16v c) {
    const v8i A = {(int)a[0], (int)a[1], (int)a[2], (int)a[3], (int)a[4], (int)a[5], 0, 0};
    const v8i B = {(int)b[0], (int)b[1], (int)b[2], (int)b[3], (int)b[4], (int)b[5], 0, 0};
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A, B, c, FA, FMT_E2M3, 0, 0, 0, 0);
}

// One 256-block of the tile.  Chain c = (pair block i, group g): three MFMAs
// from zero; stage c issues its LDS reads and MFMAs and the epilogue
// blk = fma(s_g, D, blk) of chain c - 1; stages are fenced so the compiler
// interleaves within a stage only.  After a pair block's group 3,
// acc = fma(d, blk, acc).
template <int NTB>
__device__ __forceinline__ void pf_block(const pf_b &b, const uint8_t *act_lds, const uint8_t *gs_lds,
                                         const float *d_lds, const uint32_t aofs[4], uint32_t kh, uint32_t col,
                                         f16v *acc) {
    constexpr int NC = 4 * NTB;
    f16v D[2], blk;
    uint4 G;
    auto finish = [&](int c) {
        const int i = c >> 2, g = c & 3;
#pragma unroll
        for (int r = 0; r < 16; r++) blk[r] = __builtin_fmaf(b.s[g], D[c & 1][r], g == 0 ? 0.0f : blk[r]);
        if (g == 3) {
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                const float4 d = *(const float4 *)(d_lds + 32 * i + 8 * jj + 4u * kh);
                acc[i][4 * jj] = __builtin_fmaf(d.x, blk[4 * jj], acc[i][4 * jj]);
                acc[i][4 * jj + 1] = __builtin_fmaf(d.y, blk[4 * jj + 1], acc[i][4 * jj + 1]);
                acc[i][4 * jj + 2] = __builtin_fmaf(d.z, blk[4 * jj + 2], acc[i][4 * jj + 2]);
                acc[i][4 * jj + 3] = __builtin_fmaf(d.w, blk[4 * jj + 3], acc[i][4 * jj + 3]);
            }
        }
    };
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int i = c >> 2, g = c & 3;
        __builtin_amdgcn_sched_barrier(0);
        uint32_t A[12];   // the operands of h and l, six dwords each
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const int q = 3 * g + j;
            const uint4 v = *(const uint4 *)(act_lds + aofs[q & 3] + (q >> 2) * PF_CHUNK + i * 32u * 128u);
            A[4 * j] = v.x; A[4 * j + 1] = v.y; A[4 * j + 2] = v.z; A[4 * j + 3] = v.w;
        }
        if (g == 0) G = *(const uint4 *)(gs_lds + 16u * (32u * i + col));
        // -zp * gsum: two groups' sums are one operand, the other group's
        // zero point is zero
        typedef uint32_t u2 __attribute__((ext_vector_type(2)));
        const u2 ga = g < 2 ? u2{G.x, G.y} : u2{G.z, G.w};
        const u2 zb = (g & 1) ? u2{0u, b.z[g]} : u2{b.z[g], 0u};
        f16v d = {0.0f};
        d = __builtin_amdgcn_mfma_f32_32x32x8f16(__builtin_bit_cast(h4v, ga), __builtin_bit_cast(h4v, zb), d, 0, 0, 0);
        d = pf_mfma6<FMT_E3M2>(A, b.w[g], d);
        D[c & 1] = pf_mfma6<FMT_E2M3>(A + 6, b.w[g], d);
        if (c > 0) finish(c - 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    finish(NC - 1);
}

// The tile's outputs.  D layout: lane holds column col, tokens
// 8*(r/4) + 4*kh + r%4.  Gate/up: mid = ((g*sig(g))*u)*w per pair; down:
// the per-pair rows.
template <bool Q3, int NTB>
__device__ __forceinline__ void pf_epilogue(const pf_params &p, float clamp, const f16v *acc, const uint32_t *s_pair,
                                            const float *s_w, const uint64_t *s_tab, uint32_t kh, uint32_t col,
                                            uint32_t wcol, uint32_t cnt) {
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)NTB; i++) {
        if constexpr (Q3) {
            // lanes col and col ^ 16 hold the gate and up rows of one mid row:
            // after swapping values the gate lane forms the SwiGLU of tokens
            // r2 = k and the up lane of r2 = k + 8, so every lane takes half
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float va = acc[i][k], vb = acc[i][k + 8];
                const float oa = __shfl_xor(va, 16, 64), ob = __shfl_xor(vb, 16, 64);
                const bool up_lane = col >= 16u;
                const int r2 = up_lane ? k + 8 : k;
                const float g = up_lane ? ob : va, u = up_lane ? vb : oa;
                const uint32_t tl = 32u * i + 8u * ((uint32_t)r2 >> 2) + 4u * kh + ((uint32_t)r2 & 3u);
                if (tl < cnt) {
                    const uint64_t at = (uint64_t)s_pair[tl] * p.out_rows + wcol;
                    p.mid[at] = sf37_swiglu_mid_t(g, u, s_w[tl], clamp, s_tab);
                    if (p.gate_out) p.gate_out[at] = g;
                    if (p.up_out) p.up_out[at] = u;
                }
            }
        } else {
#pragma unroll
            for (int r2 = 0; r2 < 16; r2++) {
                const uint32_t tl = 32u * i + 8u * (r2 >> 2) + 4u * kh + (r2 & 3);
                if (tl < cnt) p.down_pair[(uint64_t)s_pair[tl] * p.out_rows + wcol] = acc[i][r2];
            }
        }
    }
}

// Gate/up (Q3 = true): row tile = 64 F rows, wave w has gate rows
// rt*64 + 16w + c and up rows (c < 16: gate, else up) as its 32 columns;
// epilogue mid = ((g*sig(g))*u)*w per pair.  Down (Q3 = false): row tile =
// 128 output rows, 32 per wave; epilogue down_pair[pair][row].  One item
// (tile, row tile) per workgroup: tiles interleaved over the XCDs, a tile's
// row tiles consecutive on one.
//
// Pipeline: at the top of a block its weight words (registers) and its
// activations (LDS) have landed; the words are dequantised at once, then the
// next block's activations go into the other buffer and the words of the
// block after next into the same registers while this block's chains run.
// The activations are issued first, so that waiting for them leaves the
// newest weight words in flight.
template <bool Q3, int NTB, typename ISSUE>
__device__ __forceinline__ void pf_loop(const uint8_t *wrow, uint32_t nblk, ISSUE &&issue_act,
                                        const uint8_t (*s_act)[PF_ACT_BUF], const uint8_t (*s_gs)[16u * PF_T],
                                        const float (*s_d)[PF_T], uint32_t kh, uint32_t col,
                                        pf_raw_t<Q3, false> &even, pf_raw_t<Q3, true> &oddr,
                                        f16v *acc) {
#pragma unroll
    for (int i = 0; i < NTB; i++)
#pragma unroll
        for (int r2 = 0; r2 < 16; r2++) acc[i][r2] = 0.0f;
    uint32_t aofs[4];
#pragma unroll
    for (uint32_t m = 0; m < 4u; m++) aofs[m] = 128u * col + 16u * ((2u * m) ^ kh ^ (col & 7u));
    const uint32_t zt[2] = {kh ? 0u : 0x42403C00u, kh ? 0u : 0x47464544u};
    constexpr std::integral_constant<bool, false> no{};
    constexpr std::integral_constant<bool, true> yes{};
    // next: block b + 1 exists; next2: b + 2 too
    auto step = [&](uint32_t b, auto &raw, auto odd, auto next, auto next2) {
        constexpr int P = decltype(odd)::value ? 1 : 0;
        if constexpr (decltype(next)::value) wait_vm_keep_weights<Q3>();
        else wait_vm0();
        raw_ready(raw);
        __syncthreads();
        pf_b w;
        if constexpr (Q3) pf_dequant<true, P ? 16 : 0>(w, raw, zt);
        else pf_dequant<false, 0>(w, pf_words(raw), zt);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (decltype(next)::value) issue_act(b + 1u, NTB);
        if constexpr (decltype(next2)::value) pf_wload<Q3, P>(raw, wrow, b + 2u, kh);
        pf_block<NTB>(w, s_act[P], s_gs[P], s_d[P], aofs, kh, col, acc);
    };
    uint32_t b = 0;
#pragma clang loop unroll(disable)
    for (; b + 3u < nblk; b += 2u) {
        step(b, even, no, yes, yes);
        step(b + 1u, oddr, yes, yes, yes);
    }
    if (b + 2u == nblk) {
        step(b, even, no, yes, no);
        step(b + 1u, oddr, yes, no, no);
    } else {
        if (b + 3u == nblk) {
            step(b, even, no, yes, yes);
            step(b + 1u, oddr, yes, yes, no);
            b += 2u;
        }
        step(b, even, no, no, no);
    }
}

template <bool Q3>
__global__ void __launch_bounds__(PF_NW * 64, 2) pf_expert_kernel(pf_params p) {
    __shared__ __align__(16) uint8_t s_act[2][PF_ACT_BUF];
    __shared__ __align__(16) uint8_t s_gs[2][16u * PF_T];   // [slot][group]
    __shared__ __align__(16) float s_d[2][PF_T];
    __shared__ uint32_t s_pair[PF_T];
    __shared__ float s_w[PF_T];
    __shared__ uint64_t s_tab[Q3 ? 32 : 1];    // the exp table of the SwiGLU epilogue
    const uint32_t idx = blockIdx.x, xcd = idx & 7u, item = idx >> 3;
    const uint32_t t = xcd + 8u * (item / p.n_rt), rt = item % p.n_rt;
    if (t >= p.tiles[0]) return;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, kh = lane >> 5, col = lane & 31u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t nblk = p.nblk;
    const uint4 ti = ((const uint4 *)p.tiles)[1 + t];
    const bool sh = ti.x == p.sh_id;
    const uint32_t e = sh ? 0u : ti.x, p0 = ti.y, cnt = ti.z;
    const uint8_t *w0 = sh ? p.s0 : p.w0, *w1 = sh ? p.s1 : p.w1;
    // this lane's weight row; block 0's words start loading, block 1's after
    // the first activations
    const uint32_t wcol = Q3 ? rt * PF_GU_R + 16u * wave + (col & 15u) : rt * PF_DN_R + 32u * wave + col;
    const uint8_t *wrow = (Q3 && col >= 16u ? w1 : w0) +
                          ((uint64_t)e * p.out_rows + wcol) * ((uint64_t)nblk * (Q3 ? SF37_Q3_BYTES : SF37_Q2_BYTES));
    pf_raw_t<Q3, false> even;
    pf_raw_t<Q3, true> oddr;
    pf_wload<Q3, false>(even, wrow, 0, kh);
    // pair of tile slot sl (pad slots repeat the last pair) and its activation row
    auto slot_pair = [&](uint32_t sl) { return p.sorted[p0 + (sl < cnt ? sl : cnt - 1u)]; };
    auto slot_row = [&](uint32_t pr) { return (Q3 ? pr / p.topk : pr) * nblk; };
    const uint32_t mine = slot_pair(lane);
    if (tid < PF_T) {
        s_pair[tid] = mine;
        if (Q3) s_w[tid] = p.weights[mine];
    }
    if (Q3) sf37_stage_exp_tab(s_tab);          // read after the block loop's barriers
    // activation loads: wave w copies slot octets w and w + 4 (one per
    // 32-pair block): lane l reads piece (l % 8) ^ (l / 8) of a chunk of slot
    // l / 8; wave 0 also the group sums, wave 1 the scales, a lane per slot
    uint32_t voff[2];
#pragma unroll
    for (uint32_t k = 0; k < 2u; k++)
        voff[k] = slot_row(slot_pair(8u * (wave + 4u * k) + (lane >> 3))) * PF_BLK + 16u * ((lane & 7u) ^ (lane >> 3));
    const uint32_t srow = slot_row(mine);
    const uint32_t act_l = lds_addr(&s_act[0][0]), gs_l = lds_addr(&s_gs[0][0]), d_l = lds_addr(&s_d[0][0]);
    auto issue_act = [&](uint32_t b, uint32_t ntb) {
        const uint32_t bf = b & 1u;
#pragma unroll
        for (uint32_t k = 0; k < 2u; k++)
            if (k < ntb)
#pragma unroll
                for (uint32_t c = 0; c < 3u; c++)
                    lds_dma16(act_l + bf * PF_ACT_BUF + c * PF_CHUNK + (wave + 4u * k) * DMA16_SPAN, voff[k],
                              p.act + (uint64_t)b * PF_BLK + c * 128u);
        pf_rec_load(wave, gs_l + bf * DMA16_SPAN, d_l + bf * DMA4_SPAN, srow * PF_REC, p.rec + b * PF_REC);
    };
    f16v acc[2];
    if (cnt <= 32u) {
        issue_act(0, 1);
        if (nblk > 1u) pf_wload<Q3, true>(oddr, wrow, 1u, kh);
        pf_loop<Q3, 1>(wrow, nblk, issue_act, s_act, s_gs, s_d, kh, col, even, oddr, acc);
        pf_epilogue<Q3, 1>(p, sh ? p.sh_clamp : p.clamp, acc, s_pair, s_w, s_tab, kh, col, wcol, cnt);
    } else {
        issue_act(0, 2);
        if (nblk > 1u) pf_wload<Q3, true>(oddr, wrow, 1u, kh);
        pf_loop<Q3, 2>(wrow, nblk, issue_act, s_act, s_gs, s_d, kh, col, even, oddr, acc);
        pf_epilogue<Q3, 2>(p, sh ? p.sh_clamp : p.clamp, acc, s_pair, s_w, s_tab, kh, col, wcol, cnt);
    }
}

// ---------------------------------------------------------------------------
// Shared expert (Q8_0, every token) on the int8 matrix cores.
//
// Canonical order of sf37_ops.c:92-108: acc = acc + ((float)isum_b * ws_b) * xs_b
// per 32-block in block order.  One v_mfma_i32_32x32x32_i8 per (32-block,
// 32-token block) forms isum_b exactly from the Q8_0 weight codes, read in
// place from the tensor (no repacked copy), and the Q8_0 activation codes.
// Its accumulator starts at the bits of SH_MAGIC = 1.5 * 2^23, so the int32
// result read as a float is F = SH_MAGIC + isum_b exactly (|isum_b| <=
// 32 * 127 * 128 < 2^22), and fma(F, ws_b, -SH_MAGIC * ws_b) is the exact
// isum_b * ws_b (the second term is exact: 2 * 11 significant bits) rounded
// once, the CPU's (float)isum * w_scale.  The epilogue is then the CPU's
// three float operations per output and block.
//
// Layouts.  Activations: Q8_0 codes of each token in natural order (int8,
// nb * 32 bytes per token) and a float scale per (token, block), bit-exact
// with sf37_ops.c:57-90.  A workgroup stages a chunk of SH_CB blocks of its
// 64 tokens in LDS: token row r holds 2 * SH_CB 16-byte pieces (block jj,
// half kh = piece 2 jj + kh), piece q stored at slot q ^ (r & 7), so the
// 8 rows a read of 8 lanes touches land on distinct banks.  MFMA operands:
// lane (row or column l % 32, half kh = l / 32) holds the 16 codes
// 16 kh .. 16 kh + 15 of a block, for activations and weights alike.
// ---------------------------------------------------------------------------
constexpr uint32_t SH_T = 64;                  // tokens per tile
constexpr uint32_t SH_CB = 4;                  // Q8_0 blocks per K chunk
constexpr uint32_t SH_RS = SH_CB * 32u;        // LDS bytes per token row of a chunk (int8 codes)
constexpr uint32_t SH_BUF = SH_T * SH_RS;      // one chunk buffer
constexpr float SH_MAGIC = 12582912.0f;        // 1.5 * 2^23
constexpr int32_t SH_MAGIC_BITS = 0x4B400000;
// sh_gemm direct loads (dwordx4): load L of a chunk fills token rows
// 8 L .. 8 L + 7 (1 KiB, contiguous), L < SH_T / 8, two per wave (4 waves);
// activation scales (dword): row `wave` of SH_T floats.
static_assert(SH_RS == 128u && DMA16_SPAN == 8u * SH_RS && SH_T / 8u == 2u * 4u,
              "sh_gemm code loads: 8 rows each, two per wave, inside the buffer");
static_assert(7u * DMA16_SPAN + DMA16_SPAN <= SH_BUF, "sh_gemm code loads stay in their buffer");
static_assert(SH_T * 4u == DMA4_SPAN && 4u <= SH_CB, "sh_gemm scale rows stay in their buffer");

// Q8_0 activations (arithmetic of q8_0_quantize_kernel, k_q8_0.hip): eight
// lanes per 32-block, four consecutive values per lane, whose codes are one
// dword store; the scale as a float.
__global__ void __launch_bounds__(256) sh_act_kernel(int8_t *__restrict__ a8, float *__restrict__ xs,
                                                     const float *__restrict__ x, uint32_t nb, uint64_t n_tok) {
    const uint64_t gid = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    const uint64_t blk = gid >> 3;
    const uint32_t j = (uint32_t)gid & 7u;
    const bool live = blk < nb * n_tok;
    const uint64_t u = live ? blk : 0u;
    const float4 v = *(const float4 *)(x + u * 32u + 4u * j);
    float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 8));
    uint32_t q = 0;
    float d = 0.0f;
    if (amax != 0.0f) {
        d = amax / 127.0f;
        const float iscale = 1.0f / d;
        const float vv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int c = (int)fminf(fmaxf(__builtin_rintf(iscale * vv[k]), -128.0f), 127.0f);
            q |= ((uint32_t)c & 0xffu) << (8 * k);
        }
    }
    if (!live) return;
    *(uint32_t *)(a8 + u * 32u + 4u * j) = q;
    if (j == 0u) xs[u] = d;
}

struct sh_params {
    float *out0, *out1;            // gate/up: mid (SwiGLU) [tok][rows]; else the products with w0 and w1 [tok][rows]
    const uint8_t *w0, *w1;        // Q8_0 gate, up (or one or two matrices) [rows][nb blocks]
    const int8_t *act;             // [tok][nb * 32]
    const float *xs;               // [tok][nb]
    uint32_t n_tok, nb, rows, n_ct, n_tt;
    float clamp;
};

// The lane's weight words of one K chunk: per block its 16 codes (half kh)
// from the dwords around them (block jj of a chunk starts at byte 34 jj of
// the chunk, so even blocks' codes sit 2 bytes into a dword and odd blocks'
// on a dword boundary), and the dword holding the f16 scale.
struct sh_raw {
    uint32_t c[18];                // 5 + 4 + 5 + 4 code dwords
    uint32_t s[4];
};

// What a lane loads of a K chunk: its half of the row's 136 bytes, dwords
// 17 kh .. 17 kh + 16, contiguous (five loads instead of one per block
// piece; lanes l and l + 32 hold the same row).
struct sh_half {
    uint32_t w[17];
};

__device__ __forceinline__ void sh_ready(sh_half &h) {
    asm volatile("" : "+v"(h.w[0]), "+v"(h.w[1]), "+v"(h.w[2]), "+v"(h.w[3]), "+v"(h.w[4]), "+v"(h.w[5]),
                 "+v"(h.w[6]), "+v"(h.w[7]), "+v"(h.w[8]));
    asm volatile("" : "+v"(h.w[9]), "+v"(h.w[10]), "+v"(h.w[11]), "+v"(h.w[12]), "+v"(h.w[13]), "+v"(h.w[14]),
                 "+v"(h.w[15]), "+v"(h.w[16]));
}

// dword offsets (within the chunk) of block jj's first code dword for half
// kh = 0, and of the dword holding its scale; the scale is that dword's high
// half for odd jj
__host__ __device__ constexpr uint32_t sh_code_dw(uint32_t jj) { return (34u * jj + 2u) / 4u; }
__host__ __device__ constexpr uint32_t sh_scale_dw(uint32_t jj) { return (34u * jj) / 4u; }
// first of block jj's code dwords in sh_raw::c (5 for even blocks, 4 for odd)
__host__ __device__ constexpr uint32_t sh_code_reg(uint32_t jj) { return (9u * jj + 1u) / 2u; }
static_assert(sh_code_dw(0) == 0 && sh_code_dw(1) == 9 && sh_code_dw(2) == 17 && sh_code_dw(3) == 26 &&
                  sh_scale_dw(1) == 8 && sh_scale_dw(3) == 25 && SH_CB == 4,
              "chunk word offsets");
static_assert(sh_code_reg(1) == 5 && sh_code_reg(2) == 9 && sh_code_reg(3) == 14 && sh_code_reg(4) == 18,
              "code dword slots");
static_assert(2u * 17u * 4u == SH_CB * SF37_Q8_0_BYTES, "the two halves cover the chunk exactly");

__device__ __forceinline__ void sh_load(sh_half &h, const uint8_t *wrow, uint32_t c, uint32_t kh) {
    const uint32_t *q = (const uint32_t *)(wrow + (uint64_t)c * (SH_CB * SF37_Q8_0_BYTES)) + 17u * kh;
#pragma unroll
    for (uint32_t i = 0; i < 17u; i++) h.w[i] = q[i];
}

// The chunk's words in the MFMA layout: half kh needs, per block, the code
// dwords sh_code_dw(jj) + 4 kh .. (+4 or +5) and the scale dwords 0, 8, 17,
// 25.  permlane32_swap(A, B) gives [A of lanes 0-31, B of lanes 0-31] and
// [A of lanes 32-63, B of lanes 32-63]: with A = dword i and B = dword
// 4 + i of each half, the first is block 0's dword i of both halves (dword i
// for kh = 0, dword 4 + i for kh = 1), the second block 2's (17 + i, 21 + i);
// blocks 1 and 3 likewise from dwords 9 + i and 13 + i; a swap of a dword
// with itself hands both halves the scale dwords 0 and 17 (8 and 25).
__device__ __forceinline__ void sh_swap(sh_raw &r, const sh_half &h) {
#pragma unroll
    for (uint32_t i = 0; i < 5u; i++) {
        const auto v = __builtin_amdgcn_permlane32_swap(h.w[i], h.w[4u + i], false, false);
        r.c[sh_code_reg(0) + i] = v[0];
        r.c[sh_code_reg(2) + i] = v[1];
    }
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) {
        const auto v = __builtin_amdgcn_permlane32_swap(h.w[9u + i], h.w[13u + i], false, false);
        r.c[sh_code_reg(1) + i] = v[0];
        r.c[sh_code_reg(3) + i] = v[1];
    }
    const auto s0 = __builtin_amdgcn_permlane32_swap(h.w[0], h.w[0], false, false);
    const auto s1 = __builtin_amdgcn_permlane32_swap(h.w[8], h.w[8], false, false);
    r.s[0] = s0[0];
    r.s[2] = s0[1];
    r.s[1] = s1[0];
    r.s[3] = s1[1];
}

typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x16 __attribute__((ext_vector_type(16)));

// One K chunk (SH_CB Q8_0 blocks) for TBW token blocks from token block tb0.
template <int TBW>
__device__ __forceinline__ void sh_chunk(const sh_raw &r, const uint8_t *act_lds, const float *xs_lds,
                                         uint32_t kh, uint32_t col, uint32_t tb0, float (*acc)[16]) {
    const uint8_t *a_row = act_lds + (32u * tb0 + col) * SH_RS;   // token row col of token block tb0
    const uint32_t sw = col & 7u;                      // the row's slot swizzle (32 i + col has the same)
    const float *x_lane = xs_lds + 32u * tb0 + 4u * kh;
    const i32x16 magic = (i32x16)SH_MAGIC_BITS;
#pragma unroll
    for (uint32_t jj = 0; jj < SH_CB; jj++) {
        const uint32_t o = sh_code_reg(jj);
        i32x4 b;
#pragma unroll
        for (int i = 0; i < 4; i++)
            b[i] = (int)((jj & 1u) ? r.c[o + i] : align_bytes(r.c[o + i + 1], r.c[o + i], 2u));
        const float ws = sf37_f16((jj & 1u) ? r.s[jj] >> 16 : r.s[jj]);
        const float nws = -SH_MAGIC * ws;
        const uint32_t slot = ((2u * jj + kh) ^ sw) * 16u;
        // the MFMAs of every token block first, so the epilogue of one block
        // runs while the matrix cores still work on the next
        i32x16 D[TBW];
#pragma unroll
        for (uint32_t i = 0; i < TBW; i++) {
            const i32x4 a = *(const i32x4 *)(a_row + i * 32u * SH_RS + slot);
            D[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, magic, 0, 0, 0);
        }
#pragma unroll
        for (uint32_t i = 0; i < TBW; i++) {
            // the whole result reinterpreted at once (a bit_cast of one
            // vector element would name the vector's storage, i.e. element 0)
            const f16v F = __builtin_bit_cast(f16v, D[i]);
#pragma unroll
            for (int jq = 0; jq < 4; jq++) {
                const float4 xv = *(const float4 *)(x_lane + jj * SH_T + 32u * i + 8u * jq);
                const float xa[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float p = __builtin_fmaf(F[4 * jq + q], ws, nws);
                    const float t = p * xa[q];
                    acc[i][4 * jq + q] = acc[i][4 * jq + q] + t;
                }
            }
        }
    }
}

// The same chunk with its LDS reads (activation operands and scales) all
// issued first and its MFMAs next, then the epilogues in block order (same
// arithmetic, same order per output).  For grids of at most two workgroups
// per CU, where about one wave per SIMD leaves the LDS and MFMA latencies
// unhidden: they are then paid once per chunk instead of once per read, at
// ~225 VGPRs.
template <int TBW>
__device__ __forceinline__ void sh_chunk_batched(const sh_raw &r, const uint8_t *act_lds, const float *xs_lds,
                                                 uint32_t kh, uint32_t col, uint32_t tb0, float (*acc)[16]) {
    const uint8_t *a_row = act_lds + (32u * tb0 + col) * SH_RS;
    const uint32_t sw = col & 7u;
    const float *x_lane = xs_lds + 32u * tb0 + 4u * kh;
    const i32x16 magic = (i32x16)SH_MAGIC_BITS;
    i32x4 a[SH_CB][TBW];
    float4 xv[SH_CB][TBW][4];
#pragma unroll
    for (uint32_t jj = 0; jj < SH_CB; jj++) {
        const uint32_t slot = ((2u * jj + kh) ^ sw) * 16u;
#pragma unroll
        for (uint32_t i = 0; i < TBW; i++) {
            a[jj][i] = *(const i32x4 *)(a_row + i * 32u * SH_RS + slot);
#pragma unroll
            for (int jq = 0; jq < 4; jq++) xv[jj][i][jq] = *(const float4 *)(x_lane + jj * SH_T + 32u * i + 8u * jq);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    i32x16 D[SH_CB][TBW];
    float ws[SH_CB], nws[SH_CB];
#pragma unroll
    for (uint32_t jj = 0; jj < SH_CB; jj++) {
        const uint32_t o = sh_code_reg(jj);
        i32x4 b;
#pragma unroll
        for (int i = 0; i < 4; i++)
            b[i] = (int)((jj & 1u) ? r.c[o + i] : align_bytes(r.c[o + i + 1], r.c[o + i], 2u));
        ws[jj] = sf37_f16((jj & 1u) ? r.s[jj] >> 16 : r.s[jj]);
        nws[jj] = -SH_MAGIC * ws[jj];
#pragma unroll
        for (uint32_t i = 0; i < TBW; i++) D[jj][i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[jj][i], b, magic, 0, 0, 0);
    }
#pragma unroll
    for (uint32_t jj = 0; jj < SH_CB; jj++) {
#pragma unroll
        for (uint32_t i = 0; i < TBW; i++) {
            const f16v F = __builtin_bit_cast(f16v, D[jj][i]);
#pragma unroll
            for (int jq = 0; jq < 4; jq++) {
                const float xa[4] = {xv[jj][i][jq].x, xv[jj][i][jq].y, xv[jj][i][jq].z, xv[jj][i][jq].w};
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const float p = __builtin_fmaf(F[4 * jq + q], ws[jj], nws[jj]);
                    const float t = p * xa[q];
                    acc[i][4 * jq + q] = acc[i][4 * jq + q] + t;
                }
            }
        }
    }
}

// GU: gate/up, 16 gate + 16 up rows per wave, epilogue mid = (g*sig(g))*u
// (shared clamp).  Otherwise plain products: 32 output rows per wave, written
// directly (the last column tile may be partial: its missing columns repeat
// the last row and are not stored); column tiles n_ct .. 2 n_ct - 1 are the
// second matrix's.  TBW = 2: a wave takes both 32-token blocks of the tile, the
// workgroup 128 weight columns; TBW = 1 (batches whose TBW = 2 grid would
// leave CUs idle): waves 2 c and 2 c + 1 take token block 0 and 1 of the
// same 32 columns, the workgroup 64 columns.  BAT (TBW = 1 only): the chunk
// body with its reads batched (sh_chunk_batched).
template <bool GU, int TBW, bool BAT = false>
__global__ void __launch_bounds__(256, 2) sh_gemm_kernel(sh_params p) {
    static_assert(!BAT || TBW == 1, "the batched chunk body is the narrow form's");
    __shared__ __align__(16) uint8_t s_act[2][SH_BUF];
    __shared__ __align__(16) float s_xs[2][SH_CB * SH_T];
    __shared__ uint64_t s_tab[GU ? 32 : 1];    // the exp table of the SwiGLU epilogue
    static_assert(TBW == 1 || TBW == 2, "token blocks per wave");
    if (GU) sf37_stage_exp_tab(s_tab);          // read after the chunk loop's barriers
    const uint32_t tt = blockIdx.x % p.n_tt, cti = blockIdx.x / p.n_tt;
    const uint32_t mat = !GU && cti >= p.n_ct ? 1u : 0u, ct = cti - mat * p.n_ct;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, kh = lane >> 5, col = lane & 31u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t tb0 = TBW == 2 ? 0u : (wave & 1u), cg = TBW == 2 ? wave : wave >> 1;
    constexpr uint32_t COLS = 64u * TBW;               // weight columns per workgroup
    const uint32_t t0 = tt * SH_T;
    const uint32_t nb = p.nb, nchunk = nb / SH_CB;
    // this lane's weight row
    const uint32_t wcol = GU ? ct * (COLS / 2u) + 16u * cg + (col & 15u) : ct * COLS + 32u * cg + col;
    const bool second = GU ? col >= 16u : mat != 0u;
    const uint32_t wr = GU || wcol < p.rows ? wcol : p.rows - 1u;
    const uint8_t *wrow = (second ? p.w1 : p.w0) + (uint64_t)wr * nb * SF37_Q8_0_BYTES;
    float *out = GU || !mat ? p.out0 : p.out1;
    // DMA: load L = 2 wave + k fills rows 8 L .. 8 L + 7; lane l writes row
    // 8 L + l / 8, slot l % 8, which holds piece (l % 8) ^ (l / 8) of it
    uint32_t voff[2];
#pragma unroll
    for (uint32_t k = 0; k < 2u; k++) {
        const uint32_t r = 8u * (2u * wave + k) + (lane >> 3);
        const uint32_t tr = t0 + r < p.n_tok ? t0 + r : p.n_tok - 1u;
        voff[k] = tr * nb * 32u + 16u * ((lane & 7u) ^ (lane >> 3));
    }
    const uint32_t tl = t0 + lane;
    const uint32_t tok_dma = tl < p.n_tok ? tl : p.n_tok - 1u;
    const uint32_t act_l = lds_addr(&s_act[0][0]), xs_l = lds_addr(&s_xs[0][0]);
    auto issue = [&](uint32_t c) {
        const uint32_t bf = c & 1u;
#pragma unroll
        for (uint32_t k = 0; k < 2u; k++)
            lds_dma16(act_l + bf * SH_BUF + (2u * wave + k) * DMA16_SPAN, voff[k],
                      (const uint8_t *)p.act + (uint64_t)c * (SH_CB * 32u));
        lds_dma4(xs_l + bf * (SH_CB * SH_T * 4u) + wave * SH_T * 4u, tok_dma * nb * 4u,
                 (const uint8_t *)p.xs + ((uint64_t)c * SH_CB + wave) * 4u);
    };
    float acc[TBW][16];
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)TBW; i++)
#pragma unroll
        for (int r2 = 0; r2 < 16; r2++) acc[i][r2] = 0.0f;
    sh_half ha, hb;
    issue(0);
    sh_load(ha, wrow, 0, kh);
    const uint32_t last = nchunk - 1u;
    for (uint32_t c = 0; c < nchunk; c += 2u) {
        const uint32_t c1 = c + 1u < nchunk ? c + 1u : last, c2 = c + 2u < nchunk ? c + 2u : last;
        wait_vm0();
        sh_ready(ha);
        __syncthreads();
        issue(c1);
        {
            sh_raw r;
            sh_swap(r, ha);
            sh_load(hb, wrow, c1, kh);
            if constexpr (BAT) sh_chunk_batched<TBW>(r, s_act[c & 1u], s_xs[c & 1u], kh, col, tb0, acc);
            else sh_chunk<TBW>(r, s_act[c & 1u], s_xs[c & 1u], kh, col, tb0, acc);
        }
        if (c + 1u < nchunk) {
            wait_vm0();
            sh_ready(hb);
            __syncthreads();
            issue(c2);
            sh_raw r;
            sh_swap(r, hb);
            sh_load(ha, wrow, c2, kh);
            if constexpr (BAT) sh_chunk_batched<TBW>(r, s_act[(c + 1u) & 1u], s_xs[(c + 1u) & 1u], kh, col, tb0, acc);
            else sh_chunk<TBW>(r, s_act[(c + 1u) & 1u], s_xs[(c + 1u) & 1u], kh, col, tb0, acc);
        }
    }
    wait_vm0();
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)TBW; i++) {
        if constexpr (GU) {
            // lanes col and col ^ 16 hold the gate and up rows of one mid row:
            // the gate lane forms the SwiGLU of tokens r2 = k, the up lane of
            // r2 = k + 8
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const float va = acc[i][k], vb = acc[i][k + 8];
                const float oa = __shfl_xor(va, 16, 64), ob = __shfl_xor(vb, 16, 64);
                const bool up_lane = col >= 16u;
                const uint32_t r2 = up_lane ? (uint32_t)k + 8u : (uint32_t)k;
                const float g = up_lane ? ob : va, u = up_lane ? vb : oa;
                const uint32_t t = t0 + 32u * (tb0 + i) + 8u * (r2 >> 2) + 4u * kh + (r2 & 3u);
                if (t < p.n_tok) out[(uint64_t)t * p.rows + wcol] = sf37_swiglu_mid_t(g, u, 1.0f, p.clamp, s_tab);
            }
        } else {
#pragma unroll
            for (int r2 = 0; r2 < 16; r2++) {
                const uint32_t t = t0 + 32u * (tb0 + i) + 8u * (r2 >> 2) + 4u * kh + (r2 & 3);
                if (t < p.n_tok && wcol < p.rows) out[(uint64_t)t * p.rows + wcol] = acc[i][r2];
            }
        }
    }
}

uint32_t pf_grid(uint32_t max_tiles, uint32_t n_rt) { return 8u * ((max_tiles + 7u) / 8u) * n_rt; }

}  // namespace

extern "C" uint32_t sf37k_pf_max_tiles(uint32_t n_pairs, uint32_t max_groups) {
    return (n_pairs + PF_T - 1u) / PF_T + max_groups;
}

extern "C" int sf37k_pf_supported(uint32_t in_dim, uint32_t mid_dim, uint32_t out_dim) {
    return in_dim % SF37_QK == 0 && mid_dim % SF37_QK == 0 && mid_dim % PF_GU_R == 0 &&
           out_dim % PF_DN_R == 0 && in_dim > 0 && mid_dim > 0;
}

// Activation operand buffer of n_rows rows: the fields, then the records.
extern "C" uint64_t sf37k_pf_act_bytes(uint32_t dim, uint64_t n_rows) {
    return (uint64_t)(dim / SF37_QK) * n_rows * (PF_BLK + PF_REC);
}
static uint8_t *pf_act_rec(const void *act, uint32_t nblk, uint64_t n_rows) {
    return (uint8_t *)act + nblk * n_rows * PF_BLK;
}

extern "C" int sf37k_pf_act(int q3, void *act, const float *x, uint32_t dim, uint32_t n_rows, sf37_stream_t s) {
    const uint32_t nblk = dim / SF37_QK;
    const uint64_t units = (uint64_t)nblk * n_rows;
    if (units == 0) return 0;
    if (units > 0xffffffffu) return (int)hipErrorInvalidValue;
    uint32_t *codes = (uint32_t *)act, *rec = (uint32_t *)pf_act_rec(act, nblk, n_rows);
    // four units per workgroup pass; at most 2048 workgroups, each wave then
    // walks several units
    const uint64_t wgs = (units + 3u) / 4u;
    const dim3 grid((unsigned)(wgs < 2048u ? wgs : 2048u));
    if (q3)
        hipLaunchKernelGGL(pf_act_kernel<true>, grid, dim3(256), 0, (hipStream_t)s, codes, rec, x, nblk, n_rows);
    else
        hipLaunchKernelGGL(pf_act_kernel<false>, grid, dim3(256), 0, (hipStream_t)s, codes, rec, x, nblk, n_rows);
    return (int)hipGetLastError();
}

extern "C" int sf37k_pf_start_supported(uint32_t n_pairs, uint32_t n_expert) {
    return n_pairs > 0 && n_pairs <= PF_START_PAIRS && n_expert > 0 && n_expert <= DISP_MAX_E;
}

extern "C" int sf37k_pf_start(void *act, const float *x, uint32_t dim, uint32_t n_rows, uint32_t *group_info,
                              uint32_t *sorted_pairs, uint32_t *counts, uint32_t *offsets, uint32_t *tiles,
                              const int32_t *selected, uint32_t n_pairs, uint32_t n_expert, sf37_stream_t s) {
    const uint32_t nblk = dim / SF37_QK;
    const uint64_t units = (uint64_t)nblk * n_rows;
    if (units > 0xffffffffu || !sf37k_pf_start_supported(n_pairs, n_expert)) return (int)hipErrorInvalidValue;
    // sixteen units per workgroup pass; at most two workgroups per CU of them
    const uint64_t wgs = (units + 15u) / 16u;
    hipLaunchKernelGGL(pf_start_kernel, dim3(1u + (unsigned)(wgs < 512u ? wgs : 512u)), dim3(1024), 0, (hipStream_t)s,
                       (uint32_t *)act, (uint32_t *)pf_act_rec(act, nblk, n_rows), x, (uint32_t)units, group_info,
                       sorted_pairs, counts, offsets, tiles, selected, n_pairs, n_expert);
    return (int)hipGetLastError();
}

extern "C" int sf37k_pf_tiles(uint32_t *tiles, const uint32_t *group_info, uint32_t max_groups,
                              sf37_stream_t s) {
    hipLaunchKernelGGL(pf_tiles_kernel, dim3(1), dim3(1024), 0, (hipStream_t)s, tiles, group_info, max_groups);
    return (int)hipGetLastError();
}

static void pf_act_params(pf_params &p, const void *act, uint32_t dim, uint64_t n_rows) {
    p.nblk = dim / SF37_QK;
    p.act = (const uint8_t *)act;
    p.rec = pf_act_rec(act, p.nblk, n_rows);
}

extern "C" int sf37k_pf_gate_up(float *mid, float *gate_out, float *up_out, const uint8_t *gate_w,
                                const uint8_t *up_w, const void *act, const uint32_t *tiles,
                                const uint32_t *sorted_pairs, const float *weights, uint32_t max_tiles,
                                uint32_t n_tok, uint32_t topk, uint32_t in_dim, uint32_t mid_dim, float clamp,
                                const sf37_pf_shared *sh, sf37_stream_t s) {
    pf_params p = {};
    p.s0 = sh ? sh->gate : NULL;
    p.s1 = sh ? sh->up : NULL;
    p.sh_id = sh ? sh->id : 0xffffffffu;
    p.sh_clamp = sh ? sh->clamp : 0.0f;
    p.mid = mid;
    p.gate_out = gate_out;
    p.up_out = up_out;
    p.w0 = gate_w;
    p.w1 = up_w;
    pf_act_params(p, act, in_dim, n_tok);
    p.tiles = tiles;
    p.sorted = sorted_pairs;
    p.weights = weights;
    p.topk = topk;
    p.out_rows = mid_dim;
    p.n_rt = mid_dim / PF_GU_R;
    p.clamp = clamp;
    hipLaunchKernelGGL(pf_expert_kernel<true>, dim3(pf_grid(max_tiles, p.n_rt)), dim3(PF_NW * 64), 0, (hipStream_t)s, p);
    return (int)hipGetLastError();
}

extern "C" int sf37k_pf_down(float *down_pair, const uint8_t *down_w, const void *act, const uint32_t *tiles,
                             const uint32_t *sorted_pairs, uint32_t max_tiles, uint32_t n_pairs, uint32_t mid_dim,
                             uint32_t out_dim, const sf37_pf_shared *sh, sf37_stream_t s) {
    pf_params p = {};
    p.s0 = sh ? sh->down : NULL;
    p.sh_id = sh ? sh->id : 0xffffffffu;
    p.down_pair = down_pair;
    p.w0 = down_w;
    pf_act_params(p, act, mid_dim, n_pairs);
    p.tiles = tiles;
    p.sorted = sorted_pairs;
    p.out_rows = out_dim;
    p.n_rt = out_dim / PF_DN_R;
    hipLaunchKernelGGL(pf_expert_kernel<false>, dim3(pf_grid(max_tiles, p.n_rt)), dim3(PF_NW * 64), 0, (hipStream_t)s, p);
    return (int)hipGetLastError();
}

// The 64-column shared GEMM when the 128-column grid (n_ct x n_tt
// workgroups) is under two workgroups per CU (measured crossover: at 2048
// tokens the 128-column gate/up grid of 640 workgroups takes 128 us, the
// 64-column one 157 us; at 512 tokens 64 columns win, 73 against 75 us).
static uint32_t sh_cus() {
    static int cus = 0;
    if (!cus) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            cus = 256;
    }
    return (uint32_t)cus;
}
static bool sh_narrow(uint32_t n_ct, uint32_t n_tt) { return (uint64_t)n_ct * n_tt < 2ull * sh_cus(); }
// The narrow form's batched chunk body when its grid (n_ct x n_tt, 64
// columns) is one round at two workgroups per CU (measured, gate/up + down:
// 256 tokens 57 + 21 -> 46 + 16 us, 512 tokens 73 + 27 -> 70 + 24 us; at
// 1024 tokens, 1.25 rounds, 97 -> 100 us, so that grid keeps the other body).
static bool sh_batched(uint32_t n_ct, uint32_t n_tt) { return (uint64_t)n_ct * n_tt <= 2ull * sh_cus(); }

extern "C" int sf37k_sh_supported(uint32_t in_dim, uint32_t mid_dim, uint32_t out_dim) {
    return in_dim % (32u * SH_CB * 2u) == 0 && mid_dim % (32u * SH_CB * 2u) == 0 && mid_dim % 64u == 0 &&
           out_dim % 128u == 0 && in_dim > 0 && mid_dim > 0;
}

extern "C" int sf37k_sh_act(void *a8, float *xs, const float *x, uint32_t dim, uint32_t n_tok, sf37_stream_t s) {
    const uint64_t n = (uint64_t)(dim / 32u) * n_tok;
    if (n == 0) return 0;
    hipLaunchKernelGGL(sh_act_kernel, dim3((unsigned)((n + 31u) / 32u)), dim3(256), 0, (hipStream_t)s,
                       (int8_t *)a8, xs, x, dim / 32u, (uint64_t)n_tok);
    return (int)hipGetLastError();
}

extern "C" int sf37k_sh_gate_up(float *mid, const uint8_t *gate_w, const uint8_t *up_w, const void *a8,
                                const float *xs, uint32_t n_tok, uint32_t in_dim, uint32_t mid_dim, float clamp,
                                sf37_stream_t s) {
    sh_params p = {};
    p.out0 = mid;
    p.w0 = gate_w;
    p.w1 = up_w;
    p.act = (const int8_t *)a8;
    p.xs = xs;
    p.n_tok = n_tok;
    p.nb = in_dim / 32u;
    p.rows = mid_dim;
    p.n_tt = (n_tok + SH_T - 1u) / SH_T;
    p.clamp = clamp;
    if (sh_narrow(mid_dim / 64u, p.n_tt)) {
        p.n_ct = mid_dim / 32u;
        if (sh_batched(p.n_ct, p.n_tt))
            hipLaunchKernelGGL((sh_gemm_kernel<true, 1, true>), dim3(p.n_ct * p.n_tt), dim3(256), 0, (hipStream_t)s, p);
        else
            hipLaunchKernelGGL((sh_gemm_kernel<true, 1>), dim3(p.n_ct * p.n_tt), dim3(256), 0, (hipStream_t)s, p);
    } else {
        p.n_ct = mid_dim / 64u;
        hipLaunchKernelGGL((sh_gemm_kernel<true, 2>), dim3(p.n_ct * p.n_tt), dim3(256), 0, (hipStream_t)s, p);
    }
    return (int)hipGetLastError();
}

extern "C" int sf37k_sh_matmul_supported(uint64_t in_dim, uint64_t out_dim, uint64_t n_tok) {
    return in_dim > 0 && in_dim % (32u * SH_CB * 2u) == 0 && out_dim > 0 && out_dim < (1u << 24) && n_tok > 0 &&
           n_tok * in_dim < (1ull << 32) && (out_dim + 63u) / 64u * 2u * ((n_tok + SH_T - 1u) / SH_T) < (1ull << 31);
}

extern "C" int sf37k_sh_matmul(float *out0, float *out1, const uint8_t *w0, const uint8_t *w1, const void *a8,
                               const float *xs, uint32_t n_tok, uint32_t in_dim, uint32_t out_dim, sf37_stream_t s) {
    sh_params p = {};
    p.out0 = out0;
    p.out1 = out1;
    p.w0 = w0;
    p.w1 = w1;
    p.act = (const int8_t *)a8;
    p.xs = xs;
    p.n_tok = n_tok;
    p.nb = in_dim / 32u;
    p.rows = out_dim;
    p.n_tt = (n_tok + SH_T - 1u) / SH_T;
    const uint32_t mats = out1 ? 2u : 1u;
    if (sh_narrow(mats * ((out_dim + 127u) / 128u), p.n_tt)) {
        p.n_ct = (out_dim + 63u) / 64u;
        const dim3 grid(mats * p.n_ct * p.n_tt);
        if (sh_batched(mats * p.n_ct, p.n_tt))
            hipLaunchKernelGGL((sh_gemm_kernel<false, 1, true>), grid, dim3(256), 0, (hipStream_t)s, p);
        else
            hipLaunchKernelGGL((sh_gemm_kernel<false, 1>), grid, dim3(256), 0, (hipStream_t)s, p);
    } else {
        p.n_ct = (out_dim + 127u) / 128u;
        hipLaunchKernelGGL((sh_gemm_kernel<false, 2>), dim3(mats * p.n_ct * p.n_tt), dim3(256), 0, (hipStream_t)s, p);
    }
    return (int)hipGetLastError();
}

extern "C" int sf37k_sh_down(float *out, const uint8_t *down_w, const void *a8, const float *xs, uint32_t n_tok,
                             uint32_t mid_dim, uint32_t out_dim, sf37_stream_t s) {
    return sf37k_sh_matmul(out, NULL, down_w, NULL, a8, xs, n_tok, mid_dim, out_dim, s);
}
