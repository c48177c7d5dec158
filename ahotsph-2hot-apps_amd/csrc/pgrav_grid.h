// The batched launches' shapes.  No HIP dependency: host tests compile the same rules.
#pragma once

#define NXCD 8      // MI355X accelerator complex dies (one L2 each)

namespace pgrav {

// Waves that share one group's lists, as a power of two.  A group's lists are a
// serial chain of LDS tiles and scalar record loads: a wave alone on its SIMD runs
// at its latency (1 us per order-4 cell), and a launch of a few groups per wave slot
// ends in a tail of long lists.  Four waves cost nothing where there are many groups;
// eight and sixteen pay while the groups are few.  us per evaluation by 1, 2, 4, 8, 16
// waves a group (order 4, theta 0.6 unless stated; in brackets: passes of two plans in
// turn on two streams, where the tails overlap), every cell in pairs and before the
// persistent launch's counters had a line each, which took sixteen waves to 33 us in the
// first row and 122 in the second:
//   111 groups (Plummer 4,099)            985   486   241   124    65
//   1,469 (Plummer 65,536, order 2)      1049   525   280   178   143
//   4,100 (lattice 64^3, images)         2054  1332  1176  1150  1139 [1713 .. 1051 1061 1073]
//   4,110 (clustered 262,144, FP64)      2217  1735  1367  1281  1348 [1572 .. 1166 1173 1267]
//   16,457 (clustered 1 M, tolerance)    2012  1613  1333  1246  1300 [1399 .. 1165 1151 1229]
//   25,034 (clustered 1 M)               3247  2895  2591  2527  2678 [2605 .. 2401 2421 2585]
//   32,795 (lattice 128^3, Ewald)        5562  5167  4956  5130  5121 [4928 .. 4779 5027 5037]
//   263,505 (clustered 16.8 M), ms       42.4  42.0  41.2  41.6  44.0 [40.5 .. 40.3 41.9 45.2]
constexpr int split_log2(int ngroups, int wave_slots) {
    // (a launch holds fewer than 2^32 lanes, and its workgroups are rounded up to NXCD)
    if (ngroups > (1 << 24) - NXCD)
        return ngroups > (1 << 25) - NXCD ? 0 : 1;
    if (ngroups < wave_slots / 2)
        return 4;
    return ngroups < 4 * wave_slots ? 3 : 2;
}

// The same for the Ewald kernels, whose waves take 6 KB (FP64 12 KB) of LDS: 24 (12) a CU in
// any split, and a workgroup's leave their places to nobody until its last is done.  us per
// evaluation by 1, 2, 4, 8 waves a group, passes of three plans in turn on three streams /
// one plan alone; in brackets one wave a group, square roots and divides, every cell in pairs:
//   4,098 (lattice 64^3)     1555/1466  1437/1338  1390/1228  1413/1221  [1537/2013]
//   7,878 (68^3)             2522/3051  2471/2674  2455/2424  2573/2420  [2559/2993]
//   8,435 (73^3)             2650/3118  2638/2742  2676/2564  2742/2589  [2713/3249]
//   11,065 (80^3)            2731/3173  2767/2816  2764/2651  2874/2696  [2785/3224]
//   14,045 (88^3)            4552/5660  4637/4889  4628/4585  4752/4653  [4531/5645]
//   16,384 (96^3)            3312/3588  3288/3307  3387/3220  4100/3351  [3458/3964]
//   32,767 (112^3)           3741/4244  3816/3939  3933/3973  5247/4507  [5013/5603]
//   FP64 4,098               2799/3459  2804/2892  2838/2755             [2862/3486]
//   FP64 11,065              6488/7126  6664/6674  6853/6584             [6389/7392]
//   FP64 16,384              8631/8576  8983/8457  9278/8484             [8836/9382]
//   FP64 32,767            11984/11151 12369/11281 12253/11009          [12861/13406]
constexpr int split_log2_ewald(int ngroups, int wave_slots, bool fp64) {
    if (ngroups < wave_slots * 3 / 4)
        return 3;
    if (fp64 || ngroups > (1 << 25) - NXCD)
        return 0;
    return ngroups < wave_slots * 5 / 4 ? 2 : 1;
}

// Workgroups of a persistent launch, `waves` waves each: as many as asked for, but no more
// than there are groups, or (negative) those of -blocks waves; a multiple of NXCD, because
// every XCD needs workgroups to drain its slice.  (Counted in waves, a grid of 256 was 32
// workgroups of 8 waves on 32 CUs: FP64 on 5,630 groups 8.0 ms, where 256 workgroups of one
// wave, on a CU each, had taken 6.8.)
constexpr int persistent_grid(int blocks, int ngroups, int waves) {
    const int grid = blocks < 0 ? (waves - 1 - blocks) / waves : blocks < ngroups ? blocks : ngroups;
    return (grid - 1) / NXCD * NXCD + NXCD;
}

}  // namespace pgrav
