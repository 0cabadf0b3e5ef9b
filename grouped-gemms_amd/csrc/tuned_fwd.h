// Tuned forward launch configurations, one per swept shape, consulted by
// pick_fwd (grouped_gemm.hip) before its built-in rule.  Proposed by
// `python grouped-gemms_amd/tune_driver.py --emit-header` from a sweep's
// best.json; an entry stays while whole calls, entry and built-in rule in turn,
// gain at least 1% by it.  An entry applies to calls with
// the same E, N, K and weight format and M within a factor of two of the
// swept M, on every operand layout (the tile order can change the bits of a
// call whose last round is split).  Fields: E, M, N, K, b_fmt (0 e4m3, 4
// e2m1), block_m, block_n, group_m, xcd swizzle, split (1: the last round may
// be split along K when the workspace allows it, 0: whole tiles only).
// sweep: 36 shapes (e4m3, 8 offset draws), 18 entries on the kernels of its
// time; with the present ones two are left.  Of the others the largest gains
// are (1, 16640, 5120, 5120) 0.9% and (1, 16640, 5120, 8192) 0.5%; (4, 16640,
// 8192, 8192) loses 1.6% on inputs that change from call to call, 3.4% on the
// same ones.
static const TunedFwd kTunedFwd[] = {
    {1, 16640, 2048, 8192, 0, 256, 256, 4, 1, 1},   // 215.4 us, built-in rule 218.9
    {2, 16640, 2048, 8192, 0, 256, 256, 4, 1, 1},   // 221.5 us, built-in rule 223.9
    {0, 0, 0, 0, 0, 0, 0, 0, 0, 0},   // end
};
