// Which routed products take tiles of 128 rows and which of 64: chosen by the grouping, which counts the tiles, for each class of K.
#pragma once

// The classes of K that choose alike: the wide form's (128 rows; K 2,048 and more), long and short, and the four-wave form's.
__host__ __device__ inline int tile_k_class(int K) { return K >= 2560 ? 0 : K >= 2048 ? 1 : K >= 1536 ? 2 : 3; }

// Bit c: products of K class c take tiles of 128 rows; n_pairs rows in n128 tiles of 128 or n64 of 64, of `experts` experts that have rows.
//
// Tiles of 128 where they hold at most 1.6 times the rows, but not where many experts, or of short K any, have 130 to 190 rows each, two
// tiles of 128 or three of 64 (256 experts, 170 rows each, gate_up, 128- against 64-row tiles: 3,072 features of 3,072 values 1,690 and 1,583 us,
// 1,024 of 2,048 447 and 388, 2,048 of 1,536 613 and 554; but 64 experts, 160 rows, 2,816 of 2,048 270 and 347, 32 experts 4,096 of 4,096 296
// and 347; short: 128 experts, 2,048 of 768 185 and 169, 64 experts 1,024 of 1,024 56 and 50).
// Where they hold more, by the form.  Wide: an expert's weights stream from memory, and a first tile costs about 3.6 (64 rows) and 3.8 (128) of
// what a further one of 64 costs 1.25 and of 128 2.5, up to some 130 rows an expert (256 experts, 3,072 of 3,072: 70 rows 979 and 1,133, 128
// rows unevenly 1,318 and 1,380, but 140 rows 1,536 and 1,491; 128 experts, 3,072 of 4,096: 65 rows 671 and 711, 140 rows 1,011 and 973), and not
// for many experts of short K (256 experts, 1,024 of 2,048: 60 rows 289 and 264, 70 rows 292 and 279; 384 experts, 2,048 of 2,048: 60
// rows 776 and 723).  Four waves: only where 64-row tiles would be 1.6 times as many (256 experts, 3,072 of 1,536: 70 rows 557 and 609, 80
// rows unevenly, 1.4 times, 628 and 616; 2,048 of 1,536: 70 rows 377 and 399, 60 rows 367 and 358, 140 rows 569 and 525; 64 experts, 1,024
// of 1,024: 100 rows unevenly 53 and 45), or 1.5 times up to 80 rows an expert of K 1,536 and more (256 experts, 3,072 of 1,536: 65 rows 547
// and 583; but 1,536 of 768, 128 experts: 122 and 114).
__host__ __device__ inline int tile_choice(long n_pairs, long n128, long n64, long experts) {
    const bool ratio = 100 * n128 <= 61 * n64, weighed = 200 * n128 <= 84 * experts + 100 * n64;
    if (80 * n128 <= n_pairs) return ratio || weighed ? 15 : experts > 128 ? 0 : 7;
    const bool wide = ratio || (weighed && n_pairs <= 132 * experts), four = 10 * n64 >= 16 * n128;
    return (wide ? 1 : 0) | (wide && experts <= 128 ? 2 : 0) | (four || (2 * n64 >= 3 * n128 && n_pairs <= 80 * experts) ? 4 : 0) | (four ? 8 : 0);
}

// Which routed products take tiles by tickets, of those whose caller brings a counter: `strips` strips of weights of K values, n_pairs rows of n_groups
// experts (on the host, which does not know how many of them have rows).  Where an expert has few rows a workgroup that stays on its CU gains by what
// it does not wait for.  Where it has several tiles, one a workgroup finds its weights nearer: launched in order the row tiles of a strip go to one
// XCD if the strips are a multiple of 8, and the more so the longer they are.  Tickets and a workgroup a tile, us: 12 strips of 3,072
// values, 256 experts of 64 rows 839 and 865, of 130 1,260 and 1,287, 55 experts of 200 364 and 395, but 256 of 300 2,333 and 2,079; 8 strips of
// 2,048, 256 of 100 543 and 577, of 170 767 and 821, of 300 1,130 and 1,003.  8 and 16 strips of 3,072, 256 of 130 912 and 890, 1,724 and
// 1,662, 55 of 300 367 and 331, 688 and 588; of 4,096 1,180 and 1,134, 2,253 and 2,106, 468 and 412, 896 and 730; 12 strips of 3,584 and
// 4,096, 256 of 64 1,054 and 1,069, 1,336 and 1,387, but 55 of 300 612 and 567, 691 and 641.
// K from 1,024 on: there the other 128-row form has four waves a tile (wide_routed); 12 strips of 1,536, 256 of 100 575 and 612.
#define TILE_TICKETS_MIN_K 1024
inline int tile_takes_tickets(int K, int strips, long n_pairs, long n_groups) {
    return K >= TILE_TICKETS_MIN_K && K <= 3072 && (K < 2560 || strips % 8 != 0) && n_pairs <= 200 * n_groups;
}

// The choice for a step whose products bring a counter.  By tickets a tile of 128 costs what it has rows for, in halves, and its lookup and first loads
// are covered, so that it is the better one up to some 130 rows an expert, and for K of 1,536 on to 200 (256 experts, tiles of 128 and of 64, us:
// 3,072 features of 3,072 values, 16 rows an expert 756 and 762, 45 808 and 854, 64 839 and 1,028, 130 1,260 and 1,404, but 170 1,555 and
// 1,561; of 1,536 values 45 503 and 518, 130 709 and 776, 170 861 and 886; 2,048 features of 2,048 values 45 497 and 501, 64 510 and 564, 170
// 767 and 758).  Beyond that, and for shorter K, as above.  Bits 4 to 7: where the choice above is another one, for the products of the step
// that take no tickets.
__host__ __device__ inline int tile_choice_tickets(long n_pairs, long n128, long n64, long experts) {
    const int without = tile_choice(n_pairs, n128, n64, experts), with = without | (n_pairs <= 132 * experts ? 7 : n_pairs <= 200 * experts ? 4 : 0);
    return with | (with ^ without) << 4;
}
