// How a frame's launches are cut, by the lanes of a chunk and the linedefs of its map.  Host code without any of the library's types, so
// that tests can ask each rule where it changes its answer and render on both sides.
#ifndef GD_RULES_H
#define GD_RULES_H

#define SETUP_THREADS 256     // linedefs of a work-group that shares a lane's
// wall_setup_kernel: a work-group takes a whole lane where there are lanes enough for the chip, and where a lane's linedefs would be two
// work-groups at most anyway.  Stages up to the strips' order in us, dealt out / whole lanes: 120 linedefs, 16 lanes 48 / 37, 512 lanes
// 57 / 51; 320, 16 lanes 51 / 45, 512 lanes 67 / 58; 701, 16 lanes 49 / 55, 640 lanes 75 / 76; 1400, 256 lanes 64 / 73, 768 lanes 99 / 97, 1024 lanes
// 115 / 114; 2000, 256 lanes 68 / 104, 768 lanes 106 / 114, 1024 lanes 126 / 123; 4000, 256 lanes 79 / 116, 768 lanes 152 / 159, 1024 lanes
// 188 / 179, 4096 lanes 708 / 509.
inline bool setup_whole_lanes(int lanes, int linedefs) { return lanes >= 800 || linedefs <= 2 * SETUP_THREADS; }

// wall_select_kernel: how many of the longest strips have their columns' lists shared out, and over how many lanes a column.  More strips and more lanes
// shorten the longest strips' time, which is all that a small batch's lasts, and add to what all of them take together, which a large one's does.
// Since a lane alone keeps its column's nearest entries at hand, few strips are left to which sharing matters: none in large batches of all but the largest maps.
// Stage times in us of strips:lanes a column, on one draw of each map and two sets of poses: the rule's choice and the fastest two of the others (none, 128, 256,
// 512 or 768 strips of 8 or 16 lanes, up to 160 lanes of 32; + on two streams, see select_together).  Runs differ by 1 to 3 us, by 5 from 2048 lanes on.
//   lanes  240 linedefs                    320                             500
//      96  128:8 46, 256:8 51, 128:32 52   128:8 57, 128:16 59, 128:32 59  256:32 60, 128:32 57, 128:16 57
//     160  128:8 47, 256:8 51, 768:8 55    128:8 56, 128:32 57, 256:8 57   256:16 62, 128:16 60, 128:32 61
//     256  128:8 49, 256:8 49, 512:8 54    128:8 57, 256:8 56, 512:8 58    256:16 62, 512:8 61, 256:8 62
//     512  128:8 57, 256:8 58, 128:16 60   256:8 65, 256:16 65, 128:8 65   256:8 73, 256:16 73, 512:16 80
//     704  128:8 62, 256:8 62, 128:16 63   256:8 72, 256:16 75, 128:8 75   256:8 79, 256:16 80, 128:8 87
//    1024  128:8 69, 256:8 69, 128:16 73   256:8 80, 256:16 84, 128:8 86   256:8 89, 256:16 92, 128:8 93
//    1536  128:8 78, 128:16 79, 256:8 84   256:8 97, 128:8 91, 128:16 94   256:8 106, 128:8 105, 256:16 106
//    2048  0 94, 128:16 94, 128:8 97       128:8 112, 128:16 107, 0 111    128:8 118, 128:16 118, 256:16 125
//    2560  0 103, 128:16 109, 128:8 114    0 114, 128:16 123, 128:8 131    0 138, 128:16 131, 128:8 139
//    3072  0 105, 128:16 125, 128:8 132    0 123, 128:16 142, 128:16+ 150  0 144, 128:16 151, 128:16+ 159
//    4096  0 138, 128:16 158, 128:16+ 164  0 157, 128:16 181, 128:16+ 186  0 168, 128:16 194, 128:16+ 195
//   lanes  701, bricks                        1000, bricks                       1400
//      96  256:32 59, 128:32 63, 128:16 65    256:32 62, 256:16 75, 128:16 77    256:32 56, 256:16 60, 128:16 74
//     160  256:16 63, 512:16 65, 256:32 65    256:16 75, 256:32 75, 512:16 76    512:16 62, 256:32 63, 768:16 63
//     256  512:16 74, 256:16 80, 768:16 83    512:16 81, 768:16 87, 256:16 95    512:16 69, 768:16 76, 512:8 85
//     512  512:16 90, 256:8 92, 256:16 93     512:16 108, 512:8 118, 768:16 120  512:16 104, 768:16 95, 768:8 100
//     704  512:16 103, 256:8 110, 256:16 113  512:16 125, 768:16 135, 512:8 139  512:16 112, 768:16 112, 512:8 115
//    1024  256:8 135, 512:16 126, 128:8 132   256:8 155, 512:16 150, 256:16 160  512:16 127, 768:16 133, 512:8 139
//    1536  256:8 145, 128:8 146, 128:16 150   256:8 174, 128:8 175, 128:16 180   256:8 165, 512:8 151, 512:16 160
//    2048  128:8 152, 256:8 157, 128:16 158   128:8 190, 256:8 185, 256:16 190   256:8 167, 128:8 169, 512:8 174
//    2560  128:16 174, 128:8 170, 0 179       128:16 217, 128:8 208, 256:16 210  256:8 194, 128:8 193, 128:16 201
//    3072  0 189, 128:16 188, 128:8 197       0 245, 128:16 228, 128:8 238       256:8+ 221, 128:8 202, 128:16 207
//    4096  0 208, 128:16+ 235, 128:16 236     0 266, 128:16+ 273, 256:16+ 283    256:8+ 258, 128:16 244, 128:16+ 255
//   lanes  2000                                 2800                                 4000
//      96  256:32 63, 256:16 79, 128:32 84      256:32 76, 256:16 88, 128:16 108     256:32 90, 256:16 108, 128:16 143
//     160  512:16 82, 256:16 82, 256:32 82      512:16 96, 768:16 97, 512:32 98      512:16 132, 512:32 119, 768:16 133
//     256  512:16 83, 768:16 91, 256:16 107     768:16 102, 512:16 102, 256:16 135   768:16 137, 512:16 135, 256:16 168
//     512  512:16 125, 768:16 125, 512:8 129    768:16 133, 512:16 146, 512:8 165    768:16 175, 768:8 196, 512:16 197
//     704  512:16 149, 768:16 146, 512:8 151    768:16 158, 768:8 177, 512:8 179     768:16 196, 768:8 220, 512:8 222
//    1024  512:16 176, 256:8 178, 768:16 179    768:16 198, 512:16 206, 512:8 216    768:16 256, 512:8 272, 768:8 278
//    1536  256:8 212, 256:16 220, 512:8 224     768:16 266, 512:8 261, 512:16 262    768:16 337, 512:8 339, 512:16 360
//    2048  256:8 254, 512:8 251, 768:8+ 254     512:8 299, 768:8+ 292, 768:16+ 292   512:8 472, 256:8 483, 768:8 485
//    2560  256:8 268, 128:8 266, 512:16+ 270    256:8 340, 768:8+ 336, 768:16+ 336   512:8 449, 768:8+ 449, 768:16+ 449
//    3072  512:16+ 290, 128:8 293, 512:8+ 297   768:16+ 356, 768:8+ 369, 128:8 370   768:16+ 490, 768:8+ 490, 512:16+ 526
//    4096  512:16+ 355, 128:16 357, 256:8+ 363  768:16+ 431, 256:8+ 440, 512:8+ 445  768:16+ 566, 768:8+ 588, 512:8+ 592
// The lines lie where the choices change places over four draws of eighteen maps, 160 to 4000 linedefs, in grids and in bricks: over these the choice takes 0.9 %
// longer than the fastest in the mean, 17 % at worst (16 lanes on 160 linedefs; with the lines that the selection's kernels had before a linedef's record lay in
// registers 2.5 and 22 %).  Maps alike in their linedefs differ by as much in where their lines would be.
inline int select_strips(int lanes, int linedefs) {
    if (linedefs <= 128 || (linedefs < 280 && lanes > 1536) || (linedefs < 512 && lanes > 2304) || (linedefs < 1024 && lanes > 2688)) return 0;
    if (linedefs < 400) return linedefs >= 280 && lanes > 288 && lanes <= 1600 ? 256 : 128;
    if (linedefs < 1024) return lanes > 1792 ? 128 : (linedefs >= 660 && lanes > 192 && lanes <= 736 ? 512 : 256);
    if (lanes <= 112) return 256;
    if (linedefs < 2300) return lanes <= 1408 || (lanes > 2688 && linedefs >= 1700) ? 512 : 256;
    if (lanes <= 192) return 512;
    return lanes <= 1600 || lanes > 2688 ? 768 : (linedefs < 3000 && lanes > 2304 ? 256 : 512);
}
inline int select_lanes(int lanes, int linedefs) {
    if (linedefs < 400) return 8;
    if (lanes <= (linedefs < 2300 ? 112 : 144)) return 32;
    if (linedefs < 512) return lanes <= 384 ? 16 : 8;
    if (linedefs < 1024) return (lanes <= (linedefs < 660 ? 600 : 736)) || lanes > 2304 ? 16 : 8;
    if (linedefs < 2300) return lanes <= 1408 || (lanes > 2688 && linedefs >= 1700) ? 16 : 8;
    return lanes <= 1600 || lanes > 2688 ? 16 : 8;
}

// wall_select_kernel: the longest strips and the others in one launch?  A launch on the side stream and back costs 20 us of the stage.  In larger batches
// the others' wavefronts are so many that they hold the longest strips' up, which the side stream's start a little later do not.  Stage times in us, one
// launch / two, of the same strips and lanes up to 1536 lanes, then of the fastest that either has:
//   lanes     701, bricks    1400         2000         2800         4000
//     768      123 / 147    128 / 152    158 / 187    188 / 212    220 / 250
//    1536      154 / 182    165 / 187    223 / 248    276 / 301    349 / 361
//    2048      152 / 178    167 / 182    251 / 254    299 / 292    472 / 491
//    2560      170 / 191    193 / 203    266 / 270    340 / 336    449 / 449
//    3072      188 / 207    202 / 218    293 / 290    370 / 356    528 / 490
//    4096      236 / 235    244 / 255    357 / 355    458 / 431    628 / 566
// (Maps of fewer than 1024 linedefs have none among the longest from 2689 lanes on.)
inline bool select_together(int lanes) { return lanes <= 2688; }

// wall_geometry_kernel: wavefronts a lane for its linedefs (a power of two).  us with 4 / 8 / 16 of them: 16 lanes 13.6 / 10.7 / 8.3, 512 lanes
// 63 / 48 / 46, 1024 lanes 48 / 41 / 42, 4096 lanes 263 / 242 / 247.
inline int geometry_parts(int lanes) { return lanes >= 1024 ? 8 : 16; }

// wall_raster_kernel: wavefronts a strip.  One draws, pass after pass, the rows that any of its columns draws.  A small batch, which lasts as
// long as its longest strips, shares a strip out over eight wavefronts, a larger one over four, over two.  The wavefront's columns then have
// eight, four or two lanes each: these prepare as many passes at once and share every run of rows out, so that both the chain of waits and
// the vector instructions of a column shrink with them (when the spare lanes stood idle, eight wavefronts never paid).  What a strip more
// wavefronts costs is room on the SIMDs.  Stage times in us (wall_geometry_kernel among them) for 1 / 2 / 4 / 8 wavefronts a strip:
//   lanes           320 linedefs              701, bricks                 2000                      4000
//     256           / 103 / 93                / 231 / 199               / 142 / 130               / 225 / 219
//     336           / 104 / 99                / 242 / 202               / 162 / 155               / 255 / 244
//     384           / 105 / 111               / 243 / 207               / 163 / 160               / 260 / 258
//     512       143 / 111 / 142           283 / 251 / 229           208 / 177 / 189           309 / 271 / 289
//     704       150 / 139 / 194           293 / 261 / 280           220 / 191 / 257           345 / 316 / 370
//     768       152 / 151 / 213           293 / 265 / 306           223 / 204 / 277           353 / 324 / 394
//    1024       170 / 193                 308 / 290                 246 / 264                 409 / 400
//    1536  263 / 243 / 280           455 / 364 / 417           399 / 338 / 385           569 / 494 / 563
//    2048  336 / 317                 493 / 462                 462 / 438                 647 / 630
//    3072  482 / 467                 692 / 683                 647 / 635                 888 / 887
//    4096  636 / 619                 904 / 902                 842 / 831                1162 /1169
// Between 704 and 1024 lanes four and two change places at 600 lanes (200 linedefs) to 1024 (4000), between 336 and 512 eight and four at 336 (200) to 512
// (701 bricks); from 3328 lanes on one is as good as two on the 1400-linedef map and 1 % better on the 4000-linedef map, the headline's.  (Before a
// work-group staged its tables with all of its lanes one was the better from 2400 lanes on: 2 / 1 took 761 / 735 us on the 4000-linedef map, 716 / 731 now.)
// With one lane a column nothing is shared.  (A prepared pass's flags and rows kept in registers of their own there, not packed into words,
// issue 1.5 % fewer instructions and take as long.)
inline int raster_parts(int lanes) { return lanes <= 336 ? 8 : (lanes <= 704 ? 4 : (lanes <= 3328 ? 2 : 1)); }

// The smallest batches, whose strips leave most of the chip idle even so: sixteen wavefronts a strip, of four columns (as many as decide on a shared
// group of rows together) with sixteen lanes each.  A frame in us, sixteen / eight (32 billboards, two sets of poses):
//   lanes        320             800             1400            2000            4000          701, bricks
//      1     123 / 124       127 / 130       186 / 190       153 / 157       209 / 213       202 / 214
//     16     238 / 240       243 / 249       237 / 241       266 / 266       366 / 373       307 / 325
//     64     264 / 267       276 / 287       302 / 301       335 / 343       525 / 544       386 / 408
//     96     281 / 285       318 / 326       330 / 327       365 / 374       548 / 563       407 / 430
//    128     289 / 292       330 / 334       364 / 349       389 / 403       573 / 586       414 / 438
//    192     338 / 312       366 / 357       434 / 413       419 / 422       652 / 661       443 / 471
//    256     389 / 333       419 / 378       509 / 450       481 / 444       662 / 649       495 / 518
inline bool raster_sixteen(int lanes) { return lanes <= 96; }

// flat_gap_kernel: wavefronts a half of a column.  The fewer the lanes, the fewer such halves and the longer the kernel lasts as its slowest one; the
// more, the longer a large work-group waits for room beside the shading.  A frame in us with 2 / 4 / 8 / 16 wavefronts (32 billboards, two
// sets of poses; in brackets with a column's halves one after the other, 16 wavefronts up to 1536 lanes, 8 beyond):
//   lanes        320 linedefs                    2000                            4000                          1400, 13 plane levels
//    256   484 / 464 / 451 / 445 (464)   570 / 542 / 524 / 514 (542)     801 / 757 / 739 / 723 (746)      500 / 479 / 476 / 486 (495)
//    512   570 / 562 / 554 / 555 (560)   713 / 692 / 670 / 682 (682)    1142 /1103 /1089 /1076 (1098)     690 / 670 / 689 / 716 (728)
//    768   707 / 700 / 700 / 701 (705)   861 / 844 / 834 / 857 (842)    1370 /1340 /1316 /1351 (1322)     904 / 888 / 942 / 959 (968)
//   1024   802 / 798 / 798 / 803 (815)  1025 /1004 /1010 /1026 (1031)   1532 /1520 /1491 /1531 (1512)    1049 /1061 /1125 /1144 (1172)
//   2048  1260 /1260 /1266 /1285 (1278) 1624 /1632 /1639 /1696 (1659)   2347 /2338 /2346 /2404 (2371)    1721 /1737 /1833 /1888 (1870)
//   4096  2188 /2199 /2201 /2241 (2248) 2864 /2881 /2939 /2955 (2965)   3851 /3856 /3922 /3985 (3870)    3001 /2995 /3166 /3264 (3205)
// Since the kernels behind it are shorter, a frame with 64 billboards with 4 / 8 / 16:
//   lanes       320               800              1400             2000                4000
//    400   432 / 431 / 427   466 / 470 / 469   526 / 548 / 577   560 / 545 / 544    823 / 799 / 786
//    512   490 / 501 / 499   547 / 559 / 544   609 / 624 / 641   630 / 646 / 635    892 / 880 / 860
//    640   573 / 581 / 581   616 / 625 / 609   717 / 746 / 755   714 / 725 / 713    985 / 978 / 968
//    768   660 / 662 / 661   729 / 732 / 724   824 / 873 / 887   821 / 830 / 819   1156 /1148 /1154
//   1024   765 / 765 / 758                     958 /1020 /1041   977 / 974 / 971   1340 /1310 /1341
//   2048  1248 /1258 /1240                    1648 /1765 /1815  1606 /1610 /1640   2157 /2159 /2240
// Asked of the lanes alone: what halves have while eight wavefronts or more of each still find room.
inline int gap_waves(int lanes) { return lanes <= 384 ? 16 : 8; }
inline int gap_waves(int lanes, int linedefs) {
    if (linedefs >= 3000) return lanes <= 704 ? 16 : (lanes <= 1152 ? 8 : 4);
    return lanes <= 448 ? gap_waves(lanes) : 4;
}

// sprite_pixels_kernel: work-groups that share the rows of a block of columns.  From 512 lanes on one takes them all: fewer listings, but the
// last work-groups last longer.  Quarters and whole columns cost the same at 230 (4000 linedefs, 128 billboards) to 1100 lanes (320 linedefs,
// 32 billboards); the line lies between.  us, quarters / whole columns, two sets of poses each: 320 linedefs, 32 billboards, 256 lanes 66 / 97,
// 512 lanes 101 / 122, 1024 lanes 170 / 174; with 128 105 / 139, 174 / 179, 336 / 296; 2000 linedefs with 128 128 / 117, 170 / 144, 256 / 212; 4000
// with 32 81 / 90, 125 / 125, 185 / 172; with 128 186 / 172, 218 / 192, 299 / 250; 4096 lanes of it 840 / 700.
#define SPRITE_ROW_PARTS 4
inline int sprite_row_parts(int lanes) { return lanes >= 512 ? 1 : SPRITE_ROW_PARTS; }

// A frame that goes to the side stream and back pays some 20 us for it.  Without billboards only the shading goes there: batches of up to 112
// lanes do without.  With them it is their painting too, and which side gains is up to the cameras: where the flat pass has little to
// do, staying saves the 20 us up to some 10 lanes, elsewhere going saves as much from 2 lanes on; 4 lies between.
// A frame in us with the side stream / without it:
//   billboards, lanes   120 linedefs     320           701, bricks      800            2000           4000
//         0     96       283 / 280     376 / 374      415 / 413      358 / 354      431 / 429      550 / 547
//         0    112       292 / 292     376 / 376      416 / 415      352 / 351      435 / 433      565 / 563
//         0    128       296 / 297     390 / 390      440 / 441      354 / 355      446 / 446      602 / 602
//         0    160       309 / 312     401 / 415      433 / 449      435 / 449      463 / 466      645 / 646
//        24      1       165 /  94     186 / 166      290 / 268      159 / 138      184 / 167      280 / 256
//        24      2       176 / 189     202 / 181      354 / 337      198 / 219      207 / 202      289 / 268
//        24      4       216 / 239     202 / 183      364 / 343      214 / 235      232 / 229      289 / 268
//        24      8       215 / 239     205 / 187      366 / 377      220 / 242      237 / 234      289 / 269
//        24     16       251 / 281     225 / 223      368 / 391      283 / 306      256 / 256      373 / 384
//        24     32       259 / 293     266 / 297      382 / 413      330 / 357      372 / 397      496 / 508
//        96      4       215 / 258     214 / 198      365 / 351      216 / 230      237 / 239      294 / 274
//        96     16       251 / 293     232 / 234      376 / 408      283 / 315      274 / 277      374 / 403
inline bool side_stream_pays(int lanes, bool billboards) { return lanes > 112 || (billboards && lanes >= 4); }

// observe_kernel: few frames by half blocks of rows, a work-group each, or by blocks?  Up to 85 frames blocks leave compute units without any.  us,
// halves / blocks, plain pooling of 208 rows and a stack with flashes: 1 frame 4.6 / 5.4, 5.1 / 6.5; 16 frames 4.7 / 6.2, 5.0 / 6.4; 42 frames 4.8 / 6.2,
// 5.7 / 7.3; 64 frames 6.2 / 6.4, 6.9 / 7.5; 85 frames 6.5 / 6.5, 7.1 / 7.6; 128 frames 8.5 / 8.5, 9.9 / 9.6; 256 frames 15.6 / 11.0, 18.2 / 12.4.
inline bool observe_few(int frames) { return frames <= 85; }

// observe_kernel: work-groups, which share the frames' blocks of rows (three a frame).  Four of them are what a compute unit holds, and each pays once
// for its copies of the palette.  4096 frames with 512 / 768 / 1024 / 2048 / 12288 work-groups: 115 / 105 / 105 / 110 / 118 us.
inline int observe_groups(int blocks) { return blocks < 1024 ? blocks : 1024; }

#endif
