// ppl_dedisp_u8group.h -- u8 dedispersion over sums of four channels.
//
// u8 sums are exact integers, so they may be taken in any order.  Four
// neighbouring channels c .. c+3 are summed once for many trials: with d the
// delay of channel c, trial dm needs
//   in[c][t + d] + sum_i in[c+i][t + d + r_i],  r_i = delay(c+i) - d,
// and in a tile of 48 trials each r_i takes two neighbouring values (the
// fraction of a sample by which d was cut off decides which).  So a pass
// builds the eight combinations as rows of 16-bit sums and every trial adds
// one value per sample from its row instead of four.  Where an r_i takes a
// third value in a tile, the trials that the first pass leaves out get another
// pass (LOFAR-size beam: 1.08 passes a group; 8704 channels x 517 trials: 1.00).
//
// A row is held in dwords: Q[x] = P[x] + 65536 P[x + 512], so a trial's 1024
// samples are 512 consecutive dwords at any offset: 64 lanes read 64
// consecutive ones, without alignment cases, and one 32-bit add sums two
// samples.  The 16-bit halves are widened to 32 bits every 64 passes (64 x
// 1020 < 65536).
//
// A workgroup is twelve waves of four trials and four waves that build rows
// two passes ahead of the sums (three buffers, so that a summing wave can have
// reads of the next pass in flight at the barrier, one a pass); input rows and
// pass records come by LDS DMA before that.
// Measured on the LOFAR-size beam (3968 channels x 2048 trials x 52640 samples):
// 25.4 ms with the one-word kernel, 14.3 with the ring kernel, 7.2 here; the
// building waves bound it (6.6 ms without the sums, 5.7 without the building).
// 8704 channels x 517 trials x 31584 samples: 12.1 -> 3.3 ms.
#pragma once

#include "ppl_dedisp_jobs.h"

namespace ppl {

constexpr int kU8gSum = 12, kU8gBuild = 4;            // summing and building waves
constexpr int kU8gND = 4;                             // trials a summing wave
constexpr int kU8gTD = kU8gSum * kU8gND;              // trials a tile
constexpr int kU8gTT = 1024;                          // samples a tile
constexpr int kU8gHalf = kU8gTT / 2;                  // distance of the samples of a dword
constexpr int kU8gRow = 256 * kU8gBuild;              // dwords of a row (a building wave makes 256)
constexpr int kU8gSpan = kU8gRow - kU8gHalf;          // delay spread a row holds
constexpr int kU8gRows = 8;                           // combinations
constexpr int kU8gRaw = 2048;                         // staged bytes of an input row
constexpr int kU8gZero = kU8gRows * kU8gRow;          // place of the row of zeros (trials not in the pass)
constexpr int kU8gBufDw = kU8gZero + kU8gHalf;        // dwords of a row buffer
constexpr int kU8gRec = 32;                           // dwords of a pass record
constexpr int kU8gNone = 0x7ffffff0;                  // a row past every input (inputs end below 2^31 bytes)
// A raw row holds 15 bytes of misalignment, the row's samples and the next
// four; the reads of one past the last dword stay inside it too.
static_assert(15 + kU8gRow + kU8gHalf + 4 + 8 <= kU8gRaw, "raw row");

// Passes a tile may have.  A pass takes as long as the one-word kernel takes
// for 1.1 channels and the ring kernel for 2 (LOFAR-size beam: 7.2 ms at 1.08
// passes a group, 25.4 and 14.3).
inline int u8g_capacity(int nChan) { return (nChan + 3) / 4 * 13 / 4 + 4; }
// Table: passes per tile (padded to 64 ints), then the records.
inline size_t u8g_table_bytes(int nTiles, int nChan)
{
    return ((size_t)(nTiles + 63) / 64 * 64 + (size_t)nTiles * u8g_capacity(nChan) * kU8gRec) * 4;
}

// Builds the passes of every (tile, group of four channels), a wave each.
// Record: dwords 0..3 the first sample of the four channels' rows in the input
// (past every input: no such channel, its row is staged as zeros), dword 4 the spread of the tile's delays in channel c,
// dwords 8..31 the trials' places in the rows, 16 bits each.  The order of a
// tile's records does not matter.  count[tile] may pass the capacity: the
// plan then does not use the table.
__global__ __launch_bounds__(256) void u8g_table_kernel(const int32_t* __restrict__ delayT, int nChan, int nsamp,
                                                        int tdms, int tdmsPad, int nTiles, int capacity,
                                                        int32_t* __restrict__ tab)
{
    const int nGroups = (nChan + 3) / 4;
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= nTiles * nGroups) return;
    const int tile = i / nGroups, c = 4 * (i % nGroups), lane = threadIdx.x & 63;
    const int dm = min(tile * kU8gTD + min(lane, kU8gTD - 1), tdms - 1);
    int d[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) d[k] = delayT[(size_t)min(c + k, nChan - 1) * tdmsPad + dm];
    const int d0 = __builtin_amdgcn_readfirstlane(d[0]);  // the tile's smallest
    const int span = __builtin_amdgcn_readlane(d[0], kU8gTD - 1) - d0;
    int r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) r[k] = c + k < nChan ? d[k] - d[0] : 0;
    int32_t* records = tab + (nTiles + 63) / 64 * 64 + (size_t)tile * capacity * kU8gRec;
    uint64_t left = (1ull << kU8gTD) - 1;
    while (left) {
        // the pass takes the first trial left: per channel its r or one less,
        // whichever is the smaller the trials left have
        const int first = __builtin_ctzll(left);
        int base[4], row = 0;
        bool in = (left >> lane) & 1;
        base[0] = 0;
#pragma unroll
        for (int k = 1; k < 4; ++k) {
            const int rf = __builtin_amdgcn_readlane(r[k], first);
            base[k] = __ballot(((left >> lane) & 1) && r[k] == rf - 1) ? rf - 1 : rf;
            const int b = r[k] - base[k];
            in = in && (b == 0 || b == 1);
            row |= (b & 1) << (k - 1);
        }
        left &= ~__ballot(in);
        int slot = 0;
        if (lane == 0) slot = atomicAdd(&tab[tile], 1);
        slot = __builtin_amdgcn_readfirstlane(slot);
        if (slot >= capacity) return;
        int32_t* rec = records + (size_t)slot * kU8gRec;
        if (lane < 4) {
            const int bl = lane == 0 ? 0 : lane == 1 ? base[1] : lane == 2 ? base[2] : base[3];
            rec[lane] = c + lane < nChan ? (c + lane) * nsamp + d0 + bl : kU8gNone;
        } else if (lane < 8) {
            rec[lane] = lane == 4 ? span : 0;
        }
        if (lane < kU8gTD)
            reinterpret_cast<uint16_t*>(rec + 8)[lane] = (uint16_t)(in ? row * kU8gRow + d[0] - d0 : kU8gZero);
    }
}

// LDS DMA of 16 bytes a lane through a descriptor, from byte `at` of it (per
// lane) to lds + 16 * lane; row: and the 1 KB after (the instruction's offset
// counts on both sides).  M0 is saved and restored; the wait state after its
// write is written out.
typedef uint32_t u8g_rsrc __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void u8g_dma(u8g_rsrc rsrc, uint32_t at, uint32_t lds)
{
    uint32_t saved;
    asm volatile("s_mov_b32 %0, m0\n\t"
                 "s_mov_b32 m0, %3\n\t"
                 "s_nop 0\n\t"
                 "buffer_load_dwordx4 %1, %2, 0 offen lds\n\t"
                 "s_nop 0\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(saved)
                 : "v"(at), "s"(rsrc), "s"(lds)
                 : "memory");
}
__device__ __forceinline__ void u8g_dma_row(u8g_rsrc rsrc, uint32_t at, uint32_t lds)
{
    uint32_t saved;
    asm volatile("s_mov_b32 %0, m0\n\t"
                 "s_mov_b32 m0, %3\n\t"
                 "s_nop 0\n\t"
                 "buffer_load_dwordx4 %1, %2, 0 offen lds\n\t"
                 "buffer_load_dwordx4 %1, %2, 0 offen offset:1024 lds\n\t"
                 "s_nop 0\n\t"
                 "s_mov_b32 m0, %0"
                 : "=&s"(saved)
                 : "v"(at), "s"(rsrc), "s"(lds)
                 : "memory");
}
__device__ __forceinline__ u8g_rsrc u8g_descriptor(const void* base, uint32_t bytes)
{
    const uint64_t b = (uint64_t)(uintptr_t)base;
    u8g_rsrc r;
    r.x = __builtin_amdgcn_readfirstlane((uint32_t)b);
    r.y = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
    r.z = __builtin_amdgcn_readfirstlane(bytes);
    r.w = 0x00020000u;
    return r;
}

// DMA targets first: an LDS DMA's address is kept below 64 KB.
struct U8gShared {
    unsigned char raw[4][4][kU8gRaw];
    int32_t rec[16][kU8gRec];
    uint32_t rows[3][kU8gBufDw];
};

__global__ __launch_bounds__(64 * (kU8gSum + kU8gBuild)) void dedisperse_u8_group_kernel(const DDBatch B)
{
    __shared__ __align__(16) U8gShared S;
    int local;
    const DDJob& J = find_job(B, local);
    // every XCD gets one run of consecutive tiles (see the window kernel)
    const int per = (J.nTiles + kXcds - 1) / kXcds;
    const int g = (local % kXcds) * per + local / kXcds;
    if (g >= J.nTiles) return;
    const int dmTile = g % J.nDMTiles, t0 = (g / J.nDMTiles) * kU8gTT;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nOut = J.nOut;
    const int n = J.delayT[dmTile];

    for (int i = threadIdx.x; i < kU8gHalf; i += 64 * (kU8gSum + kU8gBuild))
        S.rows[0][kU8gZero + i] = S.rows[1][kU8gZero + i] = S.rows[2][kU8gZero + i] = 0u;

    if (wave >= kU8gSum) {
        const int q = wave - kU8gSum;  // stages input row q, builds dwords 256 q .. of every row
        const uint32_t laneBytes = 16 * lane;
        const u8g_rsrc input = u8g_descriptor(J.in, (uint32_t)J.nChan * (uint32_t)J.nsamp);
        const u8g_rsrc records = u8g_descriptor(
            J.delayT + (J.nDMTiles + 63) / 64 * 64 + (size_t)dmTile * J.CB * kU8gRec, n * kU8gRec * 4);
        const uint32_t rawLds = lds_addr(S.raw[0][q]), recLds = lds_addr(S.rec[0]);
        // the record of pass p (past the last one zeros): eight lanes of the
        // first building wave
        auto fetch = [&](int p) {
            if (q == 0 && lane < 8) u8g_dma(records, laneBytes + p * (kU8gRec * 4), recLds + (p & 15) * (kU8gRec * 4));
        };
        // input row q of pass p, from the 16 bytes holding its first sample on
        // (t0 is a multiple of 16), into its buffer: two DMA instructions
        auto stage = [&](int p, int at) {
            u8g_dma_row(input, laneBytes + (((uint32_t)at + (uint32_t)t0) & ~15u), rawLds + (p & 3) * (4 * kU8gRaw));
        };
        // the DMA of all but the newest two periods have landed, and this
        // wave's LDS writes; then the barrier
        auto period_end = [&]() {
            if (q == 0) wait_vmcnt<6>();
            else wait_vmcnt<4>();
            lds_barrier();
        };
        // the first samples and the spread of a pass's rows; read a pass ahead,
        // like the start of the row to be staged
        int start[4], spread, ahead;
        int4 nextStart;
        int nextSpread, nextAhead;
        auto look = [&](int p) {
            nextStart = *reinterpret_cast<const int4*>(S.rec[p & 15]);
            nextSpread = S.rec[p & 15][4];
            nextAhead = S.rec[(p + 3) & 15][q];
        };
        auto seen = [&]() {
            start[0] = __builtin_amdgcn_readfirstlane(nextStart.x);
            start[1] = __builtin_amdgcn_readfirstlane(nextStart.y);
            start[2] = __builtin_amdgcn_readfirstlane(nextStart.z);
            start[3] = __builtin_amdgcn_readfirstlane(nextStart.w);
            spread = __builtin_amdgcn_readfirstlane(nextSpread);
            ahead = __builtin_amdgcn_readfirstlane(nextAhead);
        };
        // the rows of pass p: lane's dwords x .. x+3, x = 256 q + 4 lane
        auto build = [&](int p, uint32_t* buf, auto&& meanwhile) {
            const bool past = 256 * q >= kU8gHalf + spread;  // past every trial's samples
            uint32_t lo[2][4], hi[2][4];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int ch = 0; ch < 4; ++ch) {
                    const uint32_t* w = reinterpret_cast<const uint32_t*>(
                        &S.raw[p & 3][ch][256 * q + 4 * lane + (start[ch] & 12) + h * kU8gHalf]);
                    lo[h][ch] = w[0];
                    hi[h][ch] = w[1];
                }
            meanwhile();
            if (past) return;
            // the four channels' bytes at x (h = 0) and x + 512 (h = 1), in
            // 16-bit halves: e[k] holds samples x + k and x + k + 2 of the row
            uint32_t sum[2][kU8gRows][2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                uint32_t e[4][3];
#pragma unroll
                for (int ch = 0; ch < 4; ++ch) {
                    // bytes s+k and s+k+2 of the eight, s the misalignment
                    const uint32_t sel = 0x0c020c00u + 0x00010001u * (start[ch] & 3);
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        e[ch][k] = __builtin_amdgcn_perm(hi[h][ch], lo[h][ch], sel + k * 0x00010001u);
                }
#pragma unroll
                for (int v = 0; v < kU8gRows; ++v)
#pragma unroll
                    for (int o = 0; o < 2; ++o)
                        sum[h][v][o] = (e[0][o] + e[1][o + (v & 1)]) + e[2][o + (v >> 1 & 1)] + e[3][o + (v >> 2)];
            }
            uint32_t* out = buf + 256 * q + 4 * lane;
#pragma unroll
            for (int v = 0; v < kU8gRows; ++v) {
                // sum[h][v][0] is samples x, x+2, sum[h][v][1] x+1, x+3
                uint4 w;
                w.x = __builtin_amdgcn_perm(sum[1][v][0], sum[0][v][0], 0x05040100u);
                w.y = __builtin_amdgcn_perm(sum[1][v][1], sum[0][v][1], 0x05040100u);
                w.z = __builtin_amdgcn_perm(sum[1][v][0], sum[0][v][0], 0x07060302u);
                w.w = __builtin_amdgcn_perm(sum[1][v][1], sum[0][v][1], 0x07060302u);
                *reinterpret_cast<uint4*>(out + v * kU8gRow) = w;
            }
        };
        // a building wave is alone on its SIMD with three summing ones, which
        // wait for it: it goes first
        __builtin_amdgcn_s_setprio(3);
        for (int p = 0; p < 9; ++p) fetch(p);
        wait_vmcnt<0>();
        lds_barrier();  // records 0 .. 8
        for (int p = 0; p < 4; ++p) stage(p, __builtin_amdgcn_readfirstlane(S.rec[p][q]));
        wait_vmcnt<4>();
        lds_barrier();  // passes 0 and 1 staged
        look(0);
        seen();
        build(0, S.rows[0], [&]() { look(1); });
        seen();
        wait_vmcnt<2>();
        lds_barrier();  // pass 0's rows, pass 2 staged
        build(1, S.rows[1], [&]() {
            look(2);
            stage(4, ahead);
        });
        seen();
        wait_vmcnt<2>();
        lds_barrier();  // pass 1's rows, pass 3 staged
        uint32_t *to = S.rows[2], *then = S.rows[0], *last = S.rows[1];
        for (int p = 0; p < n; ++p) {
            build(p + 2, to, [&]() {
                look(p + 3);
                stage(p + 5, ahead);
                fetch(p + 9);
            });
            seen();
            period_end();  // pass p summed, pass p+2's rows, pass p+3 staged
            uint32_t* const was = to;
            to = then, then = last, last = was;
        }
        wait_vmcnt<0>();  // no LDS DMA may land after the workgroup has ended
        return;
    }

    uint32_t acc[kU8gND][8];
    int32_t lo[kU8gND][8], hi[kU8gND][8];
#pragma unroll
    for (int j = 0; j < kU8gND; ++j)
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[j][k] = 0u, lo[j][k] = hi[j][k] = 0;
    auto widen = [&]() {
#pragma unroll
        for (int j = 0; j < kU8gND; ++j)
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                lo[j][k] += (int32_t)(acc[j][k] & 0xffffu);
                hi[j][k] += (int32_t)(acc[j][k] >> 16);
                acc[j][k] = 0u;
            }
    };
    lds_barrier();  // records 0 .. 8
    // this wave's four places of the pass being summed and the next, and the
    // dwords of the first trial: read a pass ahead, as its rows are done then,
    // so that reads are in flight at the barrier too
    auto places = [&](int p) { return *reinterpret_cast<const uint2*>(&S.rec[p & 15][8 + 2 * wave]); };
    uint2 at = places(0), next = places(1);
    uint32_t a[8], b[8];
    auto read = [&](uint32_t (&v)[8], const uint32_t* rows, uint32_t place) {
        const uint32_t* s = rows + place;
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = s[64 * k];
    };
    auto add = [&](const uint32_t (&v)[8], int j) {
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[j][k] += v[k];
    };
    lds_barrier();
    lds_barrier();
    lds_barrier();
    const uint32_t *cur = S.rows[0] + lane, *then = S.rows[1] + lane, *last = S.rows[2] + lane;
    read(a, cur, at.x & 0xffffu);
    for (int p = 0; p < n; ++p) {
        const uint2 after = places(p + 2);
        read(b, cur, at.x >> 16);
        add(a, 0);
        read(a, cur, at.y & 0xffffu);
        add(b, 1);
        read(b, cur, at.y >> 16);
        add(a, 2);
        read(a, then, next.x & 0xffffu);
        add(b, 3);
        // the sums so far are made before the barrier, so the reads of this
        // pass's rows have landed when the builders overwrite them; those of
        // the next pass may stay in flight
#pragma unroll
        for (int j = 0; j < kU8gND; ++j)
            asm volatile("" : "+v"(acc[j][0]), "+v"(acc[j][1]), "+v"(acc[j][2]), "+v"(acc[j][3]), "+v"(acc[j][4]),
                              "+v"(acc[j][5]), "+v"(acc[j][6]), "+v"(acc[j][7]));
        if ((p & 63) == 63) widen();
        bare_barrier();
        at = next, next = after;
        const uint32_t* const was = cur;
        cur = then, then = last, last = was;
    }
    widen();
    int32_t* __restrict__ out = static_cast<int32_t*>(J.out);
#pragma unroll
    for (int j = 0; j < kU8gND; ++j) {
        const int dm = dmTile * kU8gTD + wave * kU8gND + j;
        if (dm >= J.tdms) break;
        int32_t* o = out + (size_t)dm * nOut + t0 + lane;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int t = t0 + lane + 64 * k;
            if (t < nOut) o[64 * k] = lo[j][k];
            if (t + kU8gHalf < nOut) o[64 * k + kU8gHalf] = hi[j][k];
        }
    }
}

}  // namespace ppl
