// fa2_kernels.h -- kernel argument blocks and launch entry points shared by
// the C ABI layer (fa2_capi.hip) and the kernel translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fa2 {

// All strides are in elements.  Kernel-side invariants established by the
// host (fa2_capi.hip): D == 64, base pointers 16-byte aligned, (b,h,s)
// strides multiples of 8, scale2 > 0 and finite.
struct FwdArgs {
    const _Float16 *q, *k, *v;
    _Float16 *o;
    float *lse;
    int64_t qsb, qsh, qss, ksb, ksh, kss, vsb, vsh, vss, osb, osh, oss, lsb, lsh;
    int B, H, S;         // S: query rows (q, o, lse)
    int Sk;              // key / value rows
    int coff;            // causal: key j visible to query i iff j <= i + coff
    // Split forward (launch_fwd_split): nsplit slices of split_keys keys (a
    // multiple of 64); partials [nsplit, B*H, S] x (64 fp32 O) and x (max, sum).
    int nsplit;
    int split_keys;
    float *part_o;
    float *part_ml;
    float scale2;        // |softmax_scale| * log2(e), at least FLT_MIN
    int negate;          // softmax_scale < 0: the Q operand is negated
    uint32_t seed;       // dropout hash seed
    uint32_t drop_thr;   // keep iff (hash >> 8) >= drop_thr
    float inv_keep;      // 1 / (1 - p)
    // Dropout keep bits (dmask_word layout) written for the backward, or null.
    uint32_t *drop_mask;
    // Workgroup order (query_block_order): heads per group, 0 = plain order.
    int hgroup;
    int qbase;           // first query of query block 0 (query_block_base)
    int bhp;             // head numbers of the grid (grid_heads)
    int wg0;             // decode: number of the launch's first workgroup
};

struct BwdArgs {
    const _Float16 *q, *k, *v, *o, *dout;
    const float *lse;
    _Float16 *dq, *dk, *dv;
    float *delta;        // [B*H, S] fp32 workspace: delta = rowsum(dO * O)
    float *lse2;         // [B*H, S] fp32 workspace: LSE * log2(e), right after delta
    // Per 32-query block of each (b,h) (blocks of 256 bytes, S rounded up to
    // 32): the block's 32 values of -LSE*log2(e)/scale2, then its 32 values of
    // -delta, fp32 -- the per-row terms the dK/dV pass starts its S and dP
    // accumulators from.
    float *rowterm;
    int64_t qsb, qsh, qss, ksb, ksh, kss, vsb, vsh, vss;
    int64_t osb, osh, oss, dosb, dosh, doss;
    int64_t dqsb, dqsh, dqss, dksb, dksh, dkss, dvsb, dvsh, dvss;
    int64_t lsb, lsh;
    int B, H, S;
    float scale;         // signed softmax scale (multiplies dQ and dK)
    float scale2;        // |softmax_scale| * log2(e), at least FLT_MIN
    int negate;          // softmax_scale < 0: the K operand of S is negated
    uint32_t seed;
    uint32_t drop_thr;
    float inv_keep;
    // Dropout keep bits the forward wrote (dmask_word layout), or null: the
    // passes then evaluate the hash themselves.
    const uint32_t *drop_mask;
    // dK/dV pass: one workgroup runs key blocks j and nkb - 1 - j (causal).
    bool dkv_pair;
    // dQ pass workgroup order (query_block_order): heads per group, 0 = plain.
    int hgroup;
    int qbase;           // dQ pass: first query of query block 0 (query_block_base)
    int bhp;             // head numbers of the grid (grid_heads)
};

struct RopeArgs {
    const _Float16 *q, *k;
    _Float16 *qo, *ko;
    const float *cs, *sn;
    int64_t qsb, qsh, qss, ksb, ksh, kss, oqb, oqh, oqs, okb, okh, oks;
    int64_t cs0, sn0;
    int B, H, S;
    // Every row pointer (q, k, qo, ko, cos, sin bases and strides) 16-byte
    // aligned: the vector kernel; otherwise the 4-byte one.
    bool vec16;
};

// First query of a head's query block 0 in the forward and the dQ pass
// (blocks of `qwg` queries, `wgs` workgroups in all, `slots` of them resident).
// Under the causal mask the blocks are moved down by whole 64-query groups until
// the last one ends within 64 queries of S: a partial block is then block 0,
// which reaches the fewest keys, where with blocks counted from query 0 it is
// the last, whose few queries run the head's whole key range.  Waves whose
// queries lie below 0 (block 0 only; all of a wave's or none, waves hold 32 or
// 64) compute and store nothing.  Whole groups keep every wave on the tile
// grid: ending the last block exactly at S gave each two-block dQ wave one more
// masked tile (4-5% slower at S = 1500 and 1985).  Measured against blocks
// counted from 0 (H = 12, about 24k rows): forward 72.2 -> 67.6 us at
// S = 1030, dQ pass 100.5 -> 92.3 us there and, with keep words, 87.2 -> 75.4
// at S = 632; equal where the last block is nearly full (505, 760, 1500, 1985).
// A grid that is resident at once keeps the blocks at 0: there the longest
// workgroup sets the time, and one with fewer active waves is shorter (forward
// of 64 heads at S = 700 13.5 us, moved 14.2).
inline int query_block_base(bool causal, int S, int qwg, int64_t wgs, int64_t slots) {
    return causal && wgs > slots ? -(((S + qwg - 1) / qwg * qwg - S) & ~63) : 0;
}

// Numbers a grid gives its heads: B*H rounded up to a multiple of 8, so that
// every workgroup of a head lands on one XCD and shares its tiles in that L2;
// the workgroups of the numbers past the last head leave at once.  Measured
// against B*H itself (H = 12): B=49 S=484 forward 50.1 -> 43.5 us (its heads can
// then go in groups, fwd_groups); forward and backward of B=13 S=1100
// without the causal mask 289 -> 276, B=11 S=2800 680 -> 668.  From 128 heads
// on: with fewer, the XCDs with one head more set the time (108 heads at
// S = 1500: dQ pass 67 -> 71 us); with 129, 17 heads on one XCD and 16 on the
// others, the shared tiles outweigh it (S = 1050 forward 33.0 -> 29.6, backward
// 100.3 -> 97.3; S = 2050 99.0 -> 86.6, 285 -> 278).  Not from 2^20 heads on:
// the rounding gains nothing there and could reach the launch limit of 2^32
// threads, which 2^24 - 1 heads of one block keep below.
inline int grid_heads(int64_t bh) { return (int)(bh >= 128 && bh < (1 << 20) ? (bh + 7) & ~(int64_t)7 : bh); }

// Whether the forward (`nq` query blocks a head) and the dQ pass (`wgs`
// workgroups in all, `slots` of them resident) take an XCD's heads in groups
// (query_block_order), where their lengths make groups pay.  Groups need whole
// XCDs of heads, and with one block a head they are the plain order at the price
// of another division (B=125 H=12 S=19 forward 8.81 us, 8.52 plain).  Rounded
// head numbers (grid_heads) leave a last group of any size, whose heaviest blocks
// come late in the grid, and under the causal mask that can cost more than the
// shared tiles save: in the dQ pass while the grid is resident at once (H = 12,
// B=11 S=512 21.7 us in groups, 17.8 plain; 188 heads 23.7, 21.5; B=17 24.1,
// 25.2), in the forward of five blocks and more up to 432 heads (B=11 S=1024
// 37.0 us in groups, 30.7 plain; B=25 S=640 32.9, 30.0; B=37 S=1024 87.8, 89.5).
// With up to four blocks neither is the faster throughout (S = 512: B=31 26.4,
// 27.3; B=33 30.1, 28.5).
inline bool fwd_groups(int64_t bh, bool causal, int nq) {
    return nq > 1 && grid_heads(bh) % 8 == 0 && (bh % 8 == 0 || !causal || nq <= 4 || bh > 432);
}
inline bool dq_groups(int64_t bh, bool causal, int64_t wgs, int64_t slots) {
    return wgs > grid_heads(bh) && grid_heads(bh) % 8 == 0 && (bh % 8 == 0 || !causal || wgs > slots);
}

// Whether a [B, H, keys, 64] view (strides in elements, not negative) holds
// that many elements: false for one expanded over batches, heads or keys
// (stride 0) and for overlapping rows.
inline bool view_is_dense(int B, int H, int64_t keys, int64_t sb, int64_t sh, int64_t ss) {
    if ((B > 1 && sb == 0) || (H > 1 && sh == 0) || (keys > 1 && ss == 0)) return false;
    return (B - 1) * sb + (H - 1) * sh + (keys - 1) * ss + 64 >= (int64_t)B * H * keys * 64;
}

// RoPE reads q and k by nontemporal loads when they take more than 88 MiB
// together: each row is read once, in whole 128-byte lines, and leaves the caches
// to the outputs, which attention reads next.  Smaller ones are still in the
// Infinity Cache from what made them, and plain loads find them there.  H = 12,
// S = 2048, plain -> nontemporal: the kernel on the same tensors again and again
// B=4 (24 MiB) 8.8 -> 10.1 us, B=14 (84 MiB) 26.2 -> 29.2, B=16 S=4096 (192 MiB)
// 70.7 -> 59.5; a copy that makes qkv, the rope and the attention forward
// together B=4 60.6 -> 60.9, B=14 181.5 -> 182.0, B=16 (96 MiB) 211.5 -> 206.1,
// B=16 S=4096 630 -> 626; attention backward, rope and a reader B=14 410.7 ->
// 412.3, B=16 S=4096 1554 -> 1543.
inline bool rope_streams(const RopeArgs &a) {
    return (int64_t)a.B * a.H * a.S * 64 * 2 * (int64_t)sizeof(_Float16) > (int64_t)88 << 20 &&
           view_is_dense(a.B, a.H, a.S, a.qsb, a.qsh, a.qss) && view_is_dense(a.B, a.H, a.S, a.ksb, a.ksh, a.kss);
}

// Decode reads K and V by nontemporal loads when they take more than 80 MiB, a
// third of the 256 MB Infinity Cache: 70 -> 58.7 us at 403 MB (B*H = 96,
// Sk = 16384; 6.9 TB/s), 19.8 -> 18.9 us at 101 MB.  Smaller caches can stay
// there from one call to the next and plain loads are then as fast or faster
// (74 MB, called again and again: 14.2 us against 14.7; 12.6 MB in one slice 14.1
// against 20.1).  A cache whose heads or batches share their rows is read many
// times and keeps plain loads: B=64 H=16 Sk=4096 expanded over the heads 80 us
// against 125, B=8 H=12 Sk=16384 over the batches 29 against 46.
inline bool decode_streams(const FwdArgs &a, bool causal) {
    constexpr int64_t BYTES = 80 << 20;
    int64_t keys = a.Sk;
    if (causal && (int64_t)a.coff + 1 < keys) keys = a.coff + 1 > 0 ? a.coff + 1 : 0;   // the keys read
    return (int64_t)a.B * a.H * keys * 64 * 2 * (int64_t)sizeof(_Float16) > BYTES &&
           view_is_dense(a.B, a.H, keys, a.ksb, a.ksh, a.kss) && view_is_dense(a.B, a.H, keys, a.vsb, a.vsh, a.vss);
}

// Waves of a decode workgroup: eight, or four for slices of at most 256 keys,
// which give each of four waves one 64-key block (and the same sums).  Four are
// 5-30% slower on longer slices where a head has one workgroup, sixteen equal
// there and slower with many heads; eight, half of them idle, take the slots of
// workgroups that have not started (B*H = 768: 64 keys 5.5 us against 3.8, 200
// keys 8.0 against 7.2).
inline int decode_waves(const FwdArgs &a) { return a.split_keys <= 256 ? 4 : 8; }

// Compute units of the current device (cached per device; 256 on MI355X).
// Launchers use it to size grids against the slots of two workgroups per CU.
int device_cus();

// Launchers; each returns the hipError_t of its launch.
hipError_t launch_fwd(const FwdArgs &a, bool causal, bool dropout, hipStream_t st);
// The forward over a.nsplit key slices (partials into a.part_o / a.part_ml), then their merge.
hipError_t launch_fwd_split(const FwdArgs &a, bool causal, bool dropout, hipStream_t st);
// One query (S = 1), no dropout: the VALU decode kernel over a.nsplit slices
// (a.part_o null when nsplit = 1), then the merge when nsplit > 1.
hipError_t launch_fwd_decode(const FwdArgs &a, bool causal, hipStream_t st);
hipError_t launch_bwd_delta(const BwdArgs &a, hipStream_t st);
hipError_t launch_bwd_dq(const BwdArgs &a, bool causal, bool dropout, hipStream_t st);
hipError_t launch_bwd_dkv(const BwdArgs &a, bool causal, bool dropout, hipStream_t st);
hipError_t launch_rope(const RopeArgs &a, bool backward, hipStream_t st);

}  // namespace fa2
