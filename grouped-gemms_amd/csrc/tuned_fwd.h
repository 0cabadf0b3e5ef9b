// Tuned forward launch configurations, one per swept shape, consulted by
// pick_fwd (grouped_gemm.hip) before its built-in rule.  Written by
// `python grouped-gemms_amd/tune_driver.py --emit-header` from the sweep's
// best.json; regenerate rather than edit.  An entry applies to calls with
// the same E, N, K and weight format and M within a factor of two of the
// swept M, on every operand layout (the tile order can change the bits of a
// call whose last round is split).  Fields: E, M, N, K, b_fmt (0 e4m3, 4
// e2m1), block_m, block_n, group_m, xcd swizzle, split (1: the last round may
// be split along K when the workspace allows it, 0: whole tiles only).
// sweep: 36 shapes (e4m3, 8 offset draws), 18 with a gain of at least 1% on
// every draw; of those the 7 that the 128-element main loop still gains from
// (whole drop-in calls after a cache flush, entry against built-in rule; the
// other 11, most of them XCD swizzle 1, had come to cost up to 6%: (1, 16640,
// 8192, 2048) 275.8 us, 259.8 by the rule)
static const TunedFwd kTunedFwd[] = {
    {1, 16640, 2048, 8192, 0, 256, 256, 4, 1, 1},   // 239.3 us, built-in rule 240.8
    {1, 16640, 5120, 5120, 0, 256, 256, 4, 1, 1},   // 380.0 us, built-in rule 391.0
    {1, 16640, 5120, 8192, 0, 256, 256, 4, 1, 1},   // 558.7 us, built-in rule 575.1
    {1, 16640, 8192, 5120, 0, 256, 256, 4, 8, 1},   // 565.5 us, built-in rule 575.8
    {2, 16640, 2048, 8192, 0, 256, 256, 4, 1, 1},   // 264.8 us, built-in rule 271.2
    {2, 16640, 5120, 5120, 0, 256, 256, 4, 1, 1},   // 391.0 us, built-in rule 400.4
    {4, 16640, 8192, 8192, 0, 256, 256, 1, 1, 1},   // 872.5 us, built-in rule 893.6
    {0, 0, 0, 0, 0, 0, 0, 0, 0, 0},   // end
};
