// sf37_dispatch.h - pairs grouped by expert in one 1024-thread workgroup.
#pragma once

#include "sf37_blocks.h"

namespace {

constexpr uint32_t DISP_WAVES = 16;
constexpr uint32_t DISP_MAX_E = 512;
constexpr uint32_t DISP_ONE_PAIRS = 8192;   // larger batches: many workgroups (k_moe.hip)
constexpr uint32_t DISP_UNROLL = 8;     // 64-pair chunks whose expert ids are loaded together

__device__ __forceinline__ uint32_t clamp_expert(int32_t e, uint32_t n) {
    return (e < 0 || (uint32_t)e >= n) ? 0u : (uint32_t)e;   // sf37_cuda.cu:4428-4429
}

// ---------------------------------------------------------------------------
// Dispatch: stable counting sort of pairs by expert in one workgroup.  With
// TILE, also the matrix-core kernels' tile list: every group split into tiles
// of <= TILE pairs; tiles[0] = count; tile t at uint4 index 1 + t = {expert,
// first pair, count, 0}.
// ---------------------------------------------------------------------------
template <uint32_t TILE>
__device__ __forceinline__ void dispatch_pairs(uint32_t *__restrict__ group_info, uint32_t *__restrict__ sorted,
                                               uint32_t *__restrict__ counts, uint32_t *__restrict__ offsets,
                                               uint32_t *__restrict__ tiles, const int32_t *__restrict__ selected,
                                               uint32_t n_pairs, uint32_t n_expert) {
    __shared__ uint32_t cnt[DISP_WAVES][DISP_MAX_E];
    __shared__ uint32_t off[DISP_MAX_E];
    __shared__ uint32_t gidx[DISP_MAX_E];
    __shared__ uint32_t wsum[3][DISP_WAVES];
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63u;
    for (uint32_t i = tid; i < DISP_WAVES * DISP_MAX_E; i += 1024u) (&cnt[0][0])[i] = 0u;
    __syncthreads();
    uint32_t span = (n_pairs + DISP_WAVES - 1) / DISP_WAVES;
    span = (span + 63u) & ~63u;
    const uint32_t beg = wave * span;
    const uint32_t end = beg + span < n_pairs ? beg + span : n_pairs;
    // DISP_UNROLL loads in flight per lane before their counts are added
    for (uint32_t p0 = beg + lane; p0 < end; p0 += 64u * DISP_UNROLL) {
        uint32_t ev[DISP_UNROLL];
#pragma unroll
        for (uint32_t u = 0; u < DISP_UNROLL; u++) {
            const uint32_t p = p0 + 64u * u;
            ev[u] = p < end ? clamp_expert(selected[p], n_expert) : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < DISP_UNROLL; u++)
            if (p0 + 64u * u < end) atomicAdd(&cnt[wave][ev[u]], 1u);
    }
    __syncthreads();
    // per expert: totals and exclusive offsets of each wave's share
    uint32_t tot = 0u, nz = 0u, nt = 0u;
    if (tid < n_expert) {
        for (uint32_t w = 0; w < DISP_WAVES; w++) {
            const uint32_t c = cnt[w][tid];
            cnt[w][tid] = tot;
            tot += c;
        }
        nz = tot ? 1u : 0u;
        if constexpr (TILE != 0u) nt = (tot + TILE - 1u) / TILE;
    }
    // block-wide exclusive scans of tot, nz and nt (tid < 1024 covers E <= 512)
    uint32_t st = tot, sn = nz, sk = nt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t a = __shfl_up(st, o, 64), b = __shfl_up(sn, o, 64), c = TILE ? __shfl_up(sk, o, 64) : 0u;
        if (lane >= (uint32_t)o) {
            st += a;
            sn += b;
            sk += c;
        }
    }
    if (lane == 63u) {
        wsum[0][wave] = st;
        wsum[1][wave] = sn;
        wsum[2][wave] = sk;
    }
    __syncthreads();
    uint32_t bt = 0u, bn = 0u, bk = 0u, all_n = 0u, all_k = 0u;
    for (uint32_t w = 0; w < DISP_WAVES; w++) {
        if (w < wave) {
            bt += wsum[0][w];
            bn += wsum[1][w];
            bk += wsum[2][w];
        }
        all_n += wsum[1][w];
        all_k += wsum[2][w];
    }
    if (tid < n_expert) {
        const uint32_t ex = bt + st - tot, gx = bn + sn - nz;
        off[tid] = ex;
        gidx[tid] = gx;
        counts[tid] = tot;
        offsets[tid] = ex;
        if (nz) {
            group_info[1u + gx] = ex;
            group_info[2u + n_expert + gx] = tid;
        }
        if constexpr (TILE != 0u)
            for (uint32_t k = 0; k < nt; k++)
                ((uint4 *)tiles)[1u + bk + sk - nt + k] =
                    make_uint4(tid, ex + k * TILE, tot - k * TILE < TILE ? tot - k * TILE : TILE, 0u);
    }
    if (tid == 0) {
        offsets[n_expert] = n_pairs;
        group_info[0] = all_n;
        group_info[1u + all_n] = n_pairs;
        if constexpr (TILE != 0u) tiles[0] = all_k;
    }
    __syncthreads();
    // ordered scatter: each wave walks its own range in pair order
    uint32_t nbits = 1;
    while ((1u << nbits) < n_expert) nbits++;
    // chunks of 64 pairs in order; the experts of DISP_UNROLL chunks are
    // loaded before the first of them is ranked
    for (uint32_t base0 = beg; base0 < end; base0 += 64u * DISP_UNROLL) {
        uint32_t ev[DISP_UNROLL];
#pragma unroll
        for (uint32_t u = 0; u < DISP_UNROLL; u++) {
            const uint32_t p = base0 + 64u * u + lane;
            ev[u] = p < end ? clamp_expert(selected[p], n_expert) : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < DISP_UNROLL; u++) {
            const uint32_t base = base0 + 64u * u;
            if (base >= end) break;                       // wave-uniform
            const uint32_t p = base + lane;
            const bool act = p < end;
            const uint32_t e = ev[u];
            uint64_t peers = __ballot(act);
            for (uint32_t b = 0; b < nbits; b++) {
                const uint64_t m = __ballot(act && ((e >> b) & 1u));
                peers &= ((e >> b) & 1u) ? m : ~m;
            }
            if (act) {
                const uint64_t lt = lane ? (~0ull >> (64u - lane)) : 0ull;
                const uint32_t rank = (uint32_t)__popcll(peers & lt);
                sorted[off[e] + cnt[wave][e] + rank] = p;
                if ((peers & lt) == 0ull) cnt[wave][e] += (uint32_t)__popcll(peers);
            }
        }
    }
}

}  // namespace
