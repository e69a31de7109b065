// ppl_dedisp_window.h -- FP32 and FP16 dedispersion from a register window.
//
// What bounds these sums is one ordered FP32 add per (trial, channel, sample):
// packed adds are not used, so a CU does 64 a clock, and a kernel that reads 4
// bytes of LDS per add (114 to 228 B/clk/CU) is bound by LDS before it is by
// the adds.  Neighbouring trials read almost the same samples of a channel (on
// a LOFAR-size beam their delays differ by 0 to 6.3 samples), so here a lane
// owns R consecutive samples of four neighbouring trials: it reads the window
// those four need once into registers and each trial adds its own R samples
// from there.  At R = 20 that is at most 44 words for 80 adds instead of 80,
// and the row needs one staged copy, not four shifted ones.
//
// Which registers a trial adds depends on its delay, so on run-time values,
// while register numbers are part of the instructions.  The adds of trial j
// at window offset s are therefore code of their own (blocks of R adds), and a
// channel is four indirect jumps: a table holds, per channel and group of four
// trials, the four block addresses, the LDS address of the window and how much
// of it to read.  The channel loop is assembly for that reason; everything it
// loads is waited for inside it.
//
// The row goes straight to LDS in 16-byte pieces (its first sample rounded
// down to a whole piece; the rest of the alignment is in the window offsets),
// through a buffer descriptor that ends where the tile's last sample does, so
// nothing past the input is read.  R samples are an odd number of pieces, so
// 16-byte LDS reads at a lane stride of R samples touch every bank once per 16
// lanes with the row stored as it comes from memory.  Where the delays of four
// trials spread over more than the window holds, a trial reads a window of its
// own; the table says which.
//
// FP16 rows stay FP16 in LDS and in the window (two samples a register): an
// add is v_fma_mix_f32 of one half with 1.0, rounded once like the half's
// value plus the sum.
// Measured (start of the path to here, same card): LOFAR-size beam, 3968
// channels x 2048 trials x 52640 samples: FP32 18.6 -> 12.6 ms (34 T adds/s;
// the adds alone take 10.9 ms at one per clock and lane), FP16 35.6 -> 13.6;
// 8704 channels x 517 trials x 31584 samples, FP16: 16.0 -> 7.2; 496 x 512 x
// 17248 at 95 samples of delay a trial, FP32: 0.79 -> 0.36; 128 x 128 x 3360:
// 0.062 -> 0.035.  On the way at the LOFAR size: a barrier and a table entry
// per channel 14.6, two channels a barrier 13.6, half the scalar instructions
// (62 a channel and wave, as long to issue as 62 adds) 13.1, table entries
// loaded behind the adds 12.5.
#pragma once

#include "ppl_dedisp_jobs.h"

namespace ppl {

constexpr int kWinWaves = 8;                // waves a workgroup
constexpr int kWinND = 4;                   // trials a wave
constexpr int kWinTD = kWinWaves * kWinND;  // trials a tile
constexpr int kWinPad = 24;                 // entries past the last channel (the loop loads ahead)
constexpr int kWinEntry = 16 * kWinWaves;   // table bytes per tile and channel

// An instantiation: E samples in 16 bytes (4: FP32, 8: FP16), R samples a
// lane, window reads of up to Q pieces.  4 R sums, 4 Q window registers and
// three addresses stay below 128 registers, two workgroups a CU.
template <int E_, int R_, int Q_>
struct WinShape {
    static constexpr int E = E_, R = R_, Q = Q_;
    static constexpr int TT = 64 * R;                     // samples a tile
    static constexpr int offs = E * Q - R + 1;            // window offsets 0 .. offs-1
    static constexpr int blk = (E == 4 ? 4 : 8) * R + 4;  // bytes of a block: R adds and a jump
    static constexpr int alone = (R + 2 * (E - 1)) / E;   // reads of one trial's window
    static_assert(R % E == 0 && (R / E) % 2 == 1, "an odd number of pieces a lane");
    static_assert(4 * R + 4 * Q + 3 <= 128 && alone <= Q && Q < 15 && offs >= E, "window registers");
    static_assert(4 * offs * blk < 65536, "block addresses are 16-bit offsets");
};
using WinF32 = WinShape<4, 20, 11>;
using WinF32Short = WinShape<4, 12, 11>;
using WinF32Small = WinShape<4, 4, 11>;
using WinF16 = WinShape<8, 24, 7>;
using WinF16Small = WinShape<8, 8, 7>;

// How rows are staged.  Split: every wave loads `n` pieces a lane of every
// row, eight, four or two stages (64 KB), rounds of two channels (one at n =
// 4) between barriers.  Whole: each wave loads a row of its own, n pieces a
// lane, rounds of eight channels, two rounds of stages (32 or 64 KB).  Whole
// rows take a barrier and a round trip to memory per eight channels, not two,
// which is what short tiles spend their time on; they hold less.
enum WinStaging { kWinSplit1, kWinSplit2, kWinSplit4, kWinWhole2, kWinWhole4, kWinStagings };
constexpr bool win_whole(int g) { return g >= kWinWhole2; }
constexpr int win_loads(int g) { return g == kWinSplit1 ? 1 : g == kWinSplit2 || g == kWinWhole2 ? 2 : 4; }
constexpr int win_stage_bytes(int g) { return 1024 * win_loads(g) * (win_whole(g) ? 1 : kWinWaves); }
constexpr int win_ring_bytes(int g) { return g == kWinWhole2 ? 32768 : 65536; }

// The staging for delay spreads up to `span` within a tile of TT samples, or
// -1 where no stage holds the tile's samples.
inline int win_staging(int E, int TT, int span)
{
    for (int g : {kWinWhole2, kWinWhole4, kWinSplit1, kWinSplit2, kWinSplit4})
        if (16 / E * (TT + span + 2 * E) <= win_stage_bytes(g)) return g;
    return -1;
}

inline size_t win_table_bytes(int nDMTiles, int nChan) { return (size_t)nDMTiles * (nChan + kWinPad) * kWinEntry; }

// The table of a plan, from its device delays [nChan][tdmsPad] (rows padded
// with the last trial).  Per tile, channel and wave, with o_j the wave's trial
// delays less the tile's first delay rounded down to a whole piece:
//   word 0, low half: LDS byte of the wave's window in its stage (o_0 rounded
//     down), or 1 where the four trials read windows of their own; high half:
//     bytes to stage for a whole tile of samples;
//   words 1, 2: per trial the block address, or o_j;
//   word 3, whole rows: the row's first staged sample in the input; split
//     rows: bytes from the previous channel's row to this one.
template <class S>
__global__ void win_table_kernel(const int32_t* __restrict__ delayT, int nChan, int nsamp, int tdmsPad, int nDMTiles,
                                 int whole, int4* __restrict__ tab)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t n = (size_t)nDMTiles * (nChan + kWinPad) * kWinWaves;
    if (i >= n) return;
    constexpr int ES = 16 / S::E;
    const int w = (int)(i % kWinWaves);
    const size_t tc = i / kWinWaves;
    const int row = (int)(tc % (nChan + kWinPad)), c = min(row, nChan - 1);
    const int32_t* d = delayT + (size_t)c * tdmsPad + (tc / (nChan + kWinPad)) * kWinTD;
    const int first = d[0] & ~(S::E - 1);
    const int last = d[kWinTD - 1] - first;
    int o[kWinND];
    for (int j = 0; j < kWinND; ++j) o[j] = d[w * kWinND + j] - first;
    const int win = o[0] & ~(S::E - 1);
    int f[kWinND], low;
    if (o[kWinND - 1] - win < S::offs) {
        low = ES * win;
        for (int j = 0; j < kWinND; ++j) f[j] = (j * S::offs + o[j] - win) * S::blk;
    } else {
        low = 1;
        for (int j = 0; j < kWinND; ++j) f[j] = o[j];
    }
    const uint32_t bytes = (uint32_t)((last + S::TT + S::E - 1) / S::E * 16);
    uint32_t at = (uint32_t)c * (uint32_t)nsamp + first;
    if (!whole) {
        if (row >= nChan) at = 0;  // the last row again
        else if (row == 0) at = ES * first;
        else at = ES * (uint32_t)(nsamp + first - (d[-tdmsPad] & ~(S::E - 1)));
    }
    tab[i] = make_int4((int)((uint32_t)low | bytes << 16), (int)((uint32_t)f[0] | (uint32_t)f[1] << 16),
                       (int)((uint32_t)f[2] | (uint32_t)f[3] << 16), (int)at);
}

// The channel loop.  Scalar instructions are kept few: a SIMD issues one of
// them, like one add, every four clocks, and short tiles are bound by them.
// Registers, with W = 4R and T = W + 4Q: v0 .. v(W-1) the sums (trial j,
// sample r in v[Rj + r]), vW .. v(T-1) the window, vT an address.  s[40:43]
// and s[44:47] the table entries of even and odd channels, s[48:51] and
// s[80:83] those of the channels being staged, s[64:65] the table, s57 the
// place in it; s37 and s55 the LDS stages read and staged; s[60:63] the buffer
// descriptor of the row staged; s[66:67] to s[72:73] the four blocks, s[74:75]
// the end of the channel: block j jumps to s[68 + 2j].  s[76:77] the first
// label, s[38:39] the first block, s[84:85] and s[86:87] the ends of even and
// odd channels.
//
// Staging a channel: the descriptor starts at the row's first sample and ends
// at the tile's last.
#define PPL_WIN_PIECE(MORE)                                      \
    "s_add_u32 m0, s55, %[dmalds]\n\t"                           \
    "s_nop 0\n\t"                                                \
    "buffer_load_dwordx4 %[dma], s[60:63], 0 offen lds\n\t" MORE \
    "s_add_u32 s55, s55, %[dmastep]\n\t"                         \
    "s_and_b32 s55, s55, %[ring]-1\n\t"
#define PPL_WIN_STAGE(BYTES, ROW, MORE)  \
    "s_lshr_b32 s62, " BYTES ", 16\n\t"  \
    "s_sub_u32 s62, s62, %[cut]\n\t"     \
    "s_add_u32 s60, s60, " ROW "\n\t"    \
    "s_addc_u32 s61, s61, 0\n\t"         \
    PPL_WIN_PIECE(MORE)
#define PPL_WIN_STAGE_WHOLE(MORE)        \
    "s_lshr_b32 s62, s48, 16\n\t"        \
    "s_sub_u32 s62, s62, %[cut]\n\t"     \
    "s_lshl_b32 s52, s51, %[shift]\n\t"  \
    "s_lshr_b32 s53, s51, 32-%[shift]\n\t" \
    "s_add_u32 s60, %[inlo], s52\n\t"    \
    "s_addc_u32 s61, %[inhi], s53\n\t"   \
    PPL_WIN_PIECE(MORE)
// One more piece a lane, AT bytes on in the row and STEP from the last in LDS.
#define PPL_WIN_MORE(AT, STEP)                   \
    "v_add_u32_e32 v[ppl_T], " AT ", %[dma]\n\t" \
    "s_add_u32 m0, m0, " STEP "\n\t"             \
    "s_nop 0\n\t"                                \
    "buffer_load_dwordx4 v[ppl_T], s[60:63], 0 offen lds\n\t"
// The entries of the next channels to be staged, AT bytes past the current one's.
#define PPL_WIN_LOAD_A(AT) "s_load_dwordx4 s[48:51], s[64:65], s57 offset:" AT "\n\t"
#define PPL_WIN_LOAD_B(AT) "s_load_dwordx4 s[80:83], s[64:65], s57 offset:" AT "\n\t"
#define PPL_WIN_LANDED "s_waitcnt lgkmcnt(0)\n\t"
// A round begins: this wave's part of its rows has landed (VM loads of later
// ones may be in flight), then everyone's has, and everyone is done with the
// stages the next rows go to.
#define PPL_WIN_ROUND(VM)                      \
    "s_waitcnt vmcnt(" VM ") lgkmcnt(0)\n\t" \
    "s_barrier\n\t"
// Label addresses are sums with the first label's: an offset is added as an
// unsigned number, so it must not be negative.
#define PPL_WIN_GOTO(LO, HI, LABEL)                       \
    "s_add_u32 " LO ", s76, " LABEL "_%=-.Lfirst_%=\n\t" \
    "s_addc_u32 " HI ", s77, 0\n\t"
// Trial J with a window of its own: FIELD puts its offset into s56, THEN runs
// before the adds.
#define PPL_WIN_ALONE(FIELD, J, NEXT, THEN)            \
    FIELD                                              \
    "s_lshr_b32 s52, s56, 4-%[shift]\n\t"              \
    "s_lshl_b32 s52, s52, 4\n\t"                       \
    "s_add_u32 s52, s52, s37\n\t"                      \
    "v_add_u32_e32 v[ppl_T], s52, %[lane]\n\t"         \
    "s_and_b32 s56, s56, %[E]-1\n\t"                   \
    "s_mul_i32 s56, s56, %[blk]\n\t"                   \
    "s_add_u32 s56, s56, " J "*%[offs]*%[blk]\n\t"     \
    "s_add_u32 s66, s38, s56\n\t"                      \
    "s_addc_u32 s67, s39, 0\n\t"                       \
    ".set ppl_i, 0\n\t"                                \
    ".rept %[alone]\n\t"                               \
    "ds_read_b128 v[ppl_W+4*ppl_i:ppl_W+4*ppl_i+3], v[ppl_T] offset:16*ppl_i\n\t" \
    ".set ppl_i, ppl_i+1\n\t"                          \
    ".endr\n\t"                                        \
    NEXT                                               \
    "s_waitcnt lgkmcnt(0)\n\t" THEN                    \
    "s_setpc_b64 s[66:67]\n"
// The sums of a channel from the stage at s37: C0, C1, C2 its entry, in the
// registers E, END its end.  A table entry takes a round trip to L2, so none
// is waited for with the window's reads: once those are in, the entry of the
// channel after next goes to E, and LOADS issues others, behind the adds.  The
// loop ends after the last channel.  K makes the labels' names.
#define PPL_WIN_CHANNEL(K, C0, C1, C2, E, END, LOADS)                             \
    "s_bitcmp1_b32 " C0 ", 0\n\t"                                                 \
    "s_cbranch_scc1 .Lalone" K "_%=\n\t"                                          \
    "s_and_b32 s56, " C0 ", 0xffff\n\t"                                           \
    "s_add_u32 s56, s56, s37\n\t"                                                 \
    "v_add_u32_e32 v[ppl_T], s56, %[lane]\n\t"                                    \
    ".set ppl_i, 0\n\t"                                                           \
    ".rept %[Q]\n\t"                                                              \
    "ds_read_b128 v[ppl_W+4*ppl_i:ppl_W+4*ppl_i+3], v[ppl_T] offset:16*ppl_i\n\t" \
    ".set ppl_i, ppl_i+1\n\t"                                                     \
    ".endr\n\t"                                                                   \
    "s_and_b32 s66, " C1 ", 0xffff\n\t"                                           \
    "s_lshr_b32 s68, " C1 ", 16\n\t"                                              \
    "s_and_b32 s70, " C2 ", 0xffff\n\t"                                           \
    "s_lshr_b32 s72, " C2 ", 16\n\t"                                              \
    "s_add_u32 s66, s66, s38\n\t"                                                 \
    "s_addc_u32 s67, s39, 0\n\t"                                                  \
    "s_add_u32 s68, s68, s38\n\t"                                                 \
    "s_addc_u32 s69, s39, 0\n\t"                                                  \
    "s_add_u32 s70, s70, s38\n\t"                                                 \
    "s_addc_u32 s71, s39, 0\n\t"                                                  \
    "s_add_u32 s72, s72, s38\n\t"                                                 \
    "s_addc_u32 s73, s39, 0\n\t"                                                  \
    "s_mov_b64 s[74:75], " END "\n\t"                                             \
    "s_waitcnt lgkmcnt(0)\n\t"                                                    \
    "s_load_dwordx4 " E ", s[64:65], s57 offset:256\n\t" LOADS                    \
    "s_setpc_b64 s[66:67]\n"                                                      \
    ".Lalone" K "_%=:\n\t"                                                        \
    PPL_WIN_ALONE("s_and_b32 s56, " C1 ", 0xffff\n\t", "0", PPL_WIN_GOTO("s68", "s69", ".Lalone_1_" K), "") \
    ".Lalone_1_" K "_%=:\n\t"                                                     \
    PPL_WIN_ALONE("s_lshr_b32 s56, " C1 ", 16\n\t", "1", PPL_WIN_GOTO("s70", "s71", ".Lalone_2_" K), "") \
    ".Lalone_2_" K "_%=:\n\t"                                                     \
    PPL_WIN_ALONE("s_and_b32 s56, " C2 ", 0xffff\n\t", "2", PPL_WIN_GOTO("s72", "s73", ".Lalone_3_" K), "") \
    ".Lalone_3_" K "_%=:\n\t"                                                     \
    PPL_WIN_ALONE("s_lshr_b32 s56, " C2 ", 16\n\t", "3", "s_mov_b64 s[74:75], " END "\n\t",  \
                  "s_load_dwordx4 " E ", s[64:65], s57 offset:256\n\t" LOADS)             \
    ".Lend" K "_%=:\n\t"                                                          \
    "s_add_u32 s57, s57, 128\n\t"                                                 \
    "s_add_u32 s37, s37, %[stage]\n\t"                                            \
    "s_and_b32 s37, s37, %[ring]-1\n\t"                                           \
    "s_sub_u32 s36, s36, 1\n\t"                                                   \
    "s_cbranch_scc1 .Ldone_%=\n\t"
#define PPL_WIN_EVEN(LOADS) PPL_WIN_CHANNEL("0", "s40", "s41", "s42", "s[40:43]", "s[84:85]", LOADS)
#define PPL_WIN_ODD(LOADS) PPL_WIN_CHANNEL("1", "s44", "s45", "s46", "s[44:47]", "s[86:87]", LOADS)

// The adds: sample ppl_s + ppl_r of the window onto sum R ppl_j + ppl_r.
#define PPL_WIN_ADD32 \
    "v_add_f32_e32 v[%[R]*ppl_j+ppl_r], v[ppl_W+ppl_s+ppl_r], v[%[R]*ppl_j+ppl_r]\n\t"
#define PPL_WIN_ADD16                                                                                  \
    ".if (ppl_s+ppl_r)&1\n\t"                                                                          \
    "v_fma_mix_f32 v[%[R]*ppl_j+ppl_r], v[ppl_W+(ppl_s+ppl_r)/2], 1.0, v[%[R]*ppl_j+ppl_r] op_sel:[1,0,0] " \
    "op_sel_hi:[1,0,0]\n\t"                                                                            \
    ".else\n\t"                                                                                        \
    "v_fma_mix_f32 v[%[R]*ppl_j+ppl_r], v[ppl_W+(ppl_s+ppl_r)/2], 1.0, v[%[R]*ppl_j+ppl_r] op_sel:[0,0,0] " \
    "op_sel_hi:[1,0,0]\n\t"                                                                            \
    ".endif\n\t"

// ADD: the instruction of an add; PROLOGUE: the staging of the first channels;
// ROUND: a round of the loop.
#define PPL_WIN_LOOP(ADD, PROLOGUE, ROUND)                                        \
    asm volatile(                                                                 \
        ".set ppl_W, 4*%[R]\n\t"                                                  \
        ".set ppl_T, 4*%[R]+4*%[Q]\n\t"                                           \
        "s_mov_b32 s79, m0\n\t"                                                   \
        "s_getpc_b64 s[76:77]\n"                                                  \
        ".Lfirst_%=:\n\t"                                                         \
        PPL_WIN_GOTO("s38", "s39", ".Lblk")                                       \
        PPL_WIN_GOTO("s84", "s85", ".Lend0")                                      \
        PPL_WIN_GOTO("s86", "s87", ".Lend1")                                      \
        "s_sub_u32 s36, %[n], 1\n\t"                                              \
        "s_mov_b32 s37, 0\n\t"                                                    \
        "s_mov_b32 s55, 0\n\t"                                                    \
        "s_mov_b32 s57, 0\n\t"                                                    \
        "s_mov_b32 s60, %[inlo]\n\t"                                              \
        "s_mov_b32 s61, %[inhi]\n\t"                                              \
        "s_mov_b32 s63, 0x00020000\n\t"                                           \
        "s_mov_b64 s[64:65], %[tab]\n\t"                                          \
        ".set ppl_i, 0\n\t"                                                       \
        ".rept 4*%[R]\n\t"                                                        \
        "v_mov_b32_e32 v[ppl_i], 0\n\t"                                           \
        ".set ppl_i, ppl_i+1\n\t"                                                 \
        ".endr\n\t"                                                               \
        PROLOGUE                                                                  \
        "s_load_dwordx4 s[40:43], s[64:65], 0\n\t"                                \
        "s_load_dwordx4 s[44:47], s[64:65], 128\n"                                \
        ".Lloop_%=:\n\t"                                                          \
        ROUND                                                                     \
        "s_branch .Lloop_%=\n"                                                    \
        ".Lblk_%=:\n\t"                                                           \
        ".set ppl_j, 0\n\t"                                                       \
        ".rept 4\n\t"                                                             \
        ".set ppl_s, 0\n\t"                                                       \
        ".rept %[offs]\n\t"                                                       \
        ".set ppl_r, 0\n\t"                                                       \
        ".rept %[R]\n\t"                                                          \
        ADD                                                                       \
        ".set ppl_r, ppl_r+1\n\t"                                                 \
        ".endr\n\t"                                                               \
        "s_setpc_b64 s[68+2*ppl_j:69+2*ppl_j]\n\t"                                \
        ".set ppl_s, ppl_s+1\n\t"                                                 \
        ".endr\n\t"                                                               \
        ".set ppl_j, ppl_j+1\n\t"                                                 \
        ".endr\n"                                                                 \
        ".Ldone_%=:\n\t"                                                          \
        /* no LDS DMA may land after the workgroup has ended */                   \
        "s_waitcnt vmcnt(0) lgkmcnt(0)\n\t"                                       \
        "s_mov_b32 m0, s79\n\t"                                                   \
        "s_nop 0"                                                                 \
        : "=&{v[0:15]}"(a0), "=&{v[16:31]}"(a1), "=&{v[32:47]}"(a2), "=&{v[48:63]}"(a3),                \
          "=&{v[64:79]}"(a4), "=&{v[80:95]}"(a5)                                                        \
        : [lane] "v"(laneLds), [dma] "v"(dmaByte), [tab] "s"(tab), [inlo] "s"(inLo), [inhi] "s"(inHi),  \
          [n] "s"(nChan), [cut] "s"(cut), [dmalds] "s"(dmaLds), [R] "n"(S::R), [Q] "n"(S::Q),           \
          [E] "n"(S::E), [shift] "n"(S::E == 4 ? 2 : 1), [offs] "n"(S::offs), [blk] "n"(S::blk),        \
          [alone] "n"(S::alone), [stage] "n"(STAGE), [ring] "n"(RING),                                  \
          [dmastep] "n"(win_whole(G) ? kWinWaves * STAGE : STAGE), [ahead] "s"(128 * wave)              \
        : "memory", "scc", PPL_WIN_CLOBBERS)

// The sums are outputs; what the other shapes leave free of these is not worth
// a list of its own.
#define PPL_WIN_CLOBBERS                                                                                \
    "v96", "v97", "v98", "v99", "v100", "v101", "v102", "v103", "v104", "v105", "v106", "v107", "v108", \
    "v109", "v110", "v111", "v112", "v113", "v114", "v115", "v116", "v117", "v118", "v119", "v120",     \
    "v121", "v122", "v123", "v124", "s36", "s37", "s38", "s39", "s40", "s41", "s42", "s43", "s44",      \
    "s45", "s46", "s47", "s48", "s49", "s50", "s51", "s52", "s53", "s55", "s56", "s57", "s60", "s61",   \
    "s62", "s63", "s64", "s65", "s66", "s67", "s68", "s69", "s70", "s71", "s72", "s73", "s74", "s75",   \
    "s76", "s77", "s79", "s80", "s81", "s82", "s83", "s84", "s85", "s86", "s87", "s88"

template <class S, int G>
__global__ __launch_bounds__(64 * kWinWaves) __attribute__((amdgpu_waves_per_eu(4, 4))) void
dedisperse_window_kernel(const DDBatch B)
{
    constexpr int STAGE = win_stage_bytes(G), RING = win_ring_bytes(G);
    // a window is read whole, so past its stage by up to Q pieces
    __shared__ __align__(16) unsigned char ring[RING + 16 * S::Q];
    int local;
    const DDJob& J = find_job(B, local);
    // every XCD gets one run of consecutive tiles, DM tiles of a time tile
    // following one another, so that their overlapping rows share its L2
    const int per = (J.nTiles + kXcds - 1) / kXcds;
    const int g = (local % kXcds) * per + local / kXcds;
    if (g >= J.nTiles) return;
    const int dmTile = g % J.nDMTiles, t0 = (g / J.nDMTiles) * S::TT;
    const int lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nOut = J.nOut, nChan = J.nChan;

    const uint64_t in = (uint64_t)(uintptr_t)J.in + (uint64_t)(16 / S::E) * t0;
    const uint32_t inLo = (uint32_t)in, inHi = (uint32_t)(in >> 32);
    const char* tab = reinterpret_cast<const char*>(J.delayT) +
                      (size_t)dmTile * (nChan + kWinPad) * kWinEntry + 16 * wave;
    // a shorter last tile stages less (nOut is a multiple of E)
    const uint32_t cut = 16 / S::E * (S::TT - min(S::TT, nOut - t0));
    const uint32_t laneLds = lds_addr(ring) + 16 / S::E * S::R * lane;
    const uint32_t dmaLds = lds_addr(ring) + wave * (win_whole(G) ? STAGE : 1024);
    const uint32_t dmaByte = 16 * lane + (win_whole(G) ? 0 : 1024 * wave);

    // The sums' registers are outputs in sixteens; a shape with fewer sums
    // hands back window registers in the rest.
    typedef float vec16 __attribute__((ext_vector_type(16)));
    vec16 a0, a1, a2, a3, a4, a5;
#define PPL_WIN_PAIR(MORE) PPL_WIN_STAGE("s48", "s51", MORE) PPL_WIN_STAGE("s80", "s83", MORE)
#define PPL_WIN_PIECES4(STEP1, STEP2, STEP3, STEP) \
    PPL_WIN_MORE(STEP1, STEP) PPL_WIN_MORE(STEP2, STEP) PPL_WIN_MORE(STEP3, STEP)
#define PPL_WIN_ONE PPL_WIN_STAGE("s48", "s51", PPL_WIN_PIECES4("8192", "16384", "24576", "8192"))
    // whole rows: this wave's row of the round after next, s88 bytes on
#define PPL_WIN_LOAD_ROW "s_load_dwordx4 s[48:51], s[64:65], s88\n\ts_add_u32 s88, s88, 1024\n\t"
#define PPL_WIN_WHOLE(ADD, MORE)                                                                              \
    PPL_WIN_LOOP(ADD,                                                                                         \
                 "s_mov_b32 s88, %[ahead]\n\t" PPL_WIN_LOAD_ROW PPL_WIN_LANDED PPL_WIN_STAGE_WHOLE(MORE)      \
                     PPL_WIN_LOAD_ROW,                                                                        \
                 PPL_WIN_ROUND("0") PPL_WIN_STAGE_WHOLE(MORE) PPL_WIN_LOAD_ROW                                \
                 "\n.Lpair_%=:\n\t" PPL_WIN_EVEN("") PPL_WIN_ODD("")                                                  \
                 "s_and_b32 s56, s37, %[dmastep]-1\n\t"                                                       \
                 "s_cbranch_scc1 .Lpair_%=\n\t")
#define PPL_WIN_RUN(ADD)                                                                                      \
    if constexpr (G == kWinSplit1) {                                                                          \
        PPL_WIN_LOOP(ADD,                                                                                     \
                     PPL_WIN_LOAD_A("0") PPL_WIN_LOAD_B("128") PPL_WIN_LANDED PPL_WIN_PAIR("")                \
                     PPL_WIN_LOAD_A("256") PPL_WIN_LOAD_B("384") PPL_WIN_LANDED PPL_WIN_PAIR("")              \
                     PPL_WIN_LOAD_A("512") PPL_WIN_LOAD_B("640") PPL_WIN_LANDED PPL_WIN_PAIR("")              \
                     PPL_WIN_LOAD_A("768") PPL_WIN_LOAD_B("896"),                                             \
                     PPL_WIN_ROUND("4") PPL_WIN_PAIR("") PPL_WIN_EVEN("")                                     \
                     PPL_WIN_ODD(PPL_WIN_LOAD_A("896") PPL_WIN_LOAD_B("1024")));                              \
    } else if constexpr (G == kWinSplit2) {                                                                   \
        PPL_WIN_LOOP(ADD,                                                                                     \
                     PPL_WIN_LOAD_A("0") PPL_WIN_LOAD_B("128") PPL_WIN_LANDED                                 \
                     PPL_WIN_PAIR(PPL_WIN_MORE("8192", "8192")) PPL_WIN_LOAD_A("256") PPL_WIN_LOAD_B("384"),  \
                     PPL_WIN_ROUND("0") PPL_WIN_PAIR(PPL_WIN_MORE("8192", "8192"))                            \
                     PPL_WIN_EVEN("") PPL_WIN_ODD(PPL_WIN_LOAD_A("384") PPL_WIN_LOAD_B("512")));              \
    } else if constexpr (G == kWinSplit4) {                                                                   \
        PPL_WIN_LOOP(ADD, PPL_WIN_LOAD_A("0") PPL_WIN_LANDED PPL_WIN_ONE PPL_WIN_LOAD_A("128"),               \
                     PPL_WIN_ROUND("0") PPL_WIN_ONE PPL_WIN_EVEN(PPL_WIN_LOAD_A("256"))                       \
                     PPL_WIN_ROUND("0") PPL_WIN_ONE PPL_WIN_ODD(PPL_WIN_LOAD_A("256")));                      \
    } else if constexpr (G == kWinWhole2) {                                                                   \
        PPL_WIN_WHOLE(ADD, PPL_WIN_MORE("1024", "1024"));                                                     \
    } else {                                                                                                  \
        PPL_WIN_WHOLE(ADD, PPL_WIN_PIECES4("1024", "2048", "3072", "1024"));                                  \
    }
    if constexpr (S::E == 4) {
        PPL_WIN_RUN(PPL_WIN_ADD32)
    } else {
        PPL_WIN_RUN(PPL_WIN_ADD16)
    }

    float acc[96];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        acc[i] = a0[i];
        acc[16 + i] = a1[i];
        acc[32 + i] = a2[i];
        acc[48 + i] = a3[i];
        acc[64 + i] = a4[i];
        acc[80 + i] = a5[i];
    }
    float* __restrict__ out = static_cast<float*>(J.out);
    const int t = t0 + S::R * lane;
    const bool vec = (nOut & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
#pragma unroll
    for (int j = 0; j < kWinND; ++j) {
        const int dm = dmTile * kWinTD + (int)wave * kWinND + j;
        if (dm >= J.tdms) break;
        float* o = out + (size_t)dm * nOut + t;
        if (vec) {  // rows end on a multiple of four samples
#pragma unroll
            for (int q = 0; q < S::R; q += 4)
                if (t + q < nOut)
                    *reinterpret_cast<float4*>(o + q) = make_float4(acc[S::R * j + q], acc[S::R * j + q + 1],
                                                                    acc[S::R * j + q + 2], acc[S::R * j + q + 3]);
        } else {
#pragma unroll
            for (int k = 0; k < S::R; ++k)
                if (t + k < nOut) o[k] = acc[S::R * j + k];
        }
    }
}

}  // namespace ppl
