// Form of a decode call within the one-launch limit, by its shape (host code, no HIP).
#pragma once

#include <algorithm>
#include <cstdint>

namespace femto {

// The one-launch kernel's query heads per wave and waves per workgroup, and
// whether the split workers and their merge launch are faster where the call
// brings a workspace.
struct DecodeRoute {
    int nrep_tile, waves;
    bool split;
};

// A one-launch call takes whole sequences: it ends with its longest sequence
// and with the CU that got the most workgroups, but needs no merge launch
// (~4 us).  Its plain form has all of the plan's query heads in a wave and four
// waves, or one head and eight waves up to one (sequence, head) pair per CU.
// The host knows the longest context only, so another form is taken only where
// it was at most 2 % slower than the plain one for equal lengths and for lengths
// spread over a factor of eight alike, over 2,400 shapes (1-4096 sequences,
// 32-1024 keys, eleven head shapes, f32 and bf16; us per call, equal lengths where
// not said, plain form first):
//  * 16-bit types, at most one workgroup per CU: the fewest query heads per
//    wave (two at least) that keep the call there.  16 sequences of 1024 keys
//    on 32/8 heads 22.4 -> 17.4 (two heads, eight waves; split 20.3), 8 on 64/8
//    heads 32.2 -> 15.2.  A KV head's pages are read by at most four
//    workgroups: with six, 21 sequences on 24/2 heads took 27.1, not 23.1;
//  * ... and eight waves, so a wave walks half the pages.  At the plan's own
//    heads only while a quarter of the CUs stays free (18 sequences on 16/8
//    heads 19.5 -> 17.7; 32: 384 keys 11.4, 11.8 with eight waves), and with
//    four heads above 768 keys only (32 on 32/8 heads: 21.2 and 21.9 at 768);
//  * eight heads per wave need over 256 registers, one wave per SIMD.  Four
//    read the pages twice, by two workgroups, and are faster on short contexts:
//    64 sequences of 128 keys on 64/8 heads 20.1 -> 16.1; up to 512 keys where
//    eight heads would need a second round of workgroups too and the two
//    workgroups are launched close to each other, i.e. from four KV heads up
//    (64 of 512 keys on 64/8 heads, spread: 38.1 -> 34.9; 512 on 8/1: 41.1, 47.9);
//  * ... and in many rounds (64/8 heads from 65 sequences) split, from four KV
//    heads up: 100 of 1024 keys 129.6 -> 105.5, spread 74.6 -> 60.5; 200 of 32 keys
//    44.6 -> 27.8.  On 8/1 heads spread lengths lose (800 of 384 keys: 32.9 with
//    four heads, 39.0 with eight, 39.0 split; 1000 of 257 keys 37 -> 42);
//  * f32 (twice the bytes and registers per page), four heads per wave: split in
//    many rounds too, 100 of 128 keys on 64/8 heads 63.3 -> 38.8.  With two heads
//    or one it is as often behind (2048 sequences of one head: 42.7 and 51.7;
//    spread 22.3 and 34.9);
//  * f32, few sequences: most CUs would idle beside workgroups of 64 KB a round,
//    so near the limit the split workers win: 8 of 900 keys on 16/8 heads
//    21.6 -> 17.9, spread 19.8 -> 16.1; 1 of 900 on 32/8 heads 21.7 -> 16.1.  (They
//    cross between 576 and 770 keys.)  Not where the one-launch call fills
//    more than half the CUs or its heads share pages in the L2: 128 workgroups
//    on 16/16 heads 24.5 and 26.1, 8 on 8/1 heads spread 12.9 and 16.9.
inline DecodeRoute decode_route(int num_seqs, int n_heads, int n_kv_heads, int plan_nrep, int max_kv_len, bool f32,
                                int cus) {
    const int64_t pairs = (int64_t)num_seqs * n_heads;
    const int n_rep = n_heads / n_kv_heads;
    if (f32) {
        if (pairs <= cus) {
            const bool few = pairs <= cus / 2 && pairs / plan_nrep <= cus / 4 && n_rep <= 4 && (n_rep < 4 || num_seqs <= 4);
            return {1, 8, few && max_kv_len > 896};
        }
        return {plan_nrep, 4, plan_nrep == 4 && n_kv_heads >= 4 && pairs / 4 > 6 * cus};
    }
    if (pairs <= cus) return {1, 8, false};
    const int most = std::min(plan_nrep, 4);
    int r = std::min(most, 2);
    while (r < most && (pairs / r > cus || n_rep / r > 4)) r *= 2;
    const int64_t groups = pairs / r;
    if (groups <= cus) {
        const bool eight = r == 4 ? max_kv_len > 768 : r < plan_nrep || 4 * groups <= 3 * cus;
        return {r, eight ? 8 : 4, false};
    }
    if (plan_nrep < 8) return {r, 4, false};
    const bool near = n_kv_heads >= 4, rounds = groups > 4 * cus;
    const bool four = groups <= 12 * cus && max_kv_len <= (near && !rounds && pairs / 8 > cus ? 512 : 128);
    return {four ? 4 : 8, 4, near && rounds && (max_kv_len > 256 || groups > 12 * cus)};
}

}  // namespace femto
