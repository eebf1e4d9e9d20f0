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

// The choice where the products' workgroups take tiles by tickets.  A tile of 128 then costs what it has rows for, in halves, and its
// lookup and first loads are covered, so that it is the better one up to some 130 rows an expert, and for K of 1,536 on to 200 (256
// experts, tiles of 128 and of 64, us: 3,072 features of 3,072 values, 16 rows an expert 756 and 762, 45 817 and 855, 60 853 and 970, 130
// 1,345 and 1,420, but 170 1,654 and 1,592; of 1,536 values 32 rows 486 and 488, 52 504 and 540, 130 761 and 797, 170 923 and 907; 2,048 features
// of 2,048 values 20 rows 447 and 467, 60 497 and 532).  Beyond that, and for shorter K, as above.
__host__ __device__ inline int tile_choice_tickets(long n_pairs, long n128, long n64, long experts) {
    return tile_choice(n_pairs, n128, n64, experts) | (n_pairs <= 132 * experts ? 7 : n_pairs <= 200 * experts ? 4 : 0);
}
