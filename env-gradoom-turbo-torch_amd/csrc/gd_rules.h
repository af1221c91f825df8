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
// Stage times in us of strips:lanes a column, two sets of poses; "before" is what the line of up to 1024 strips took that lists read from memory asked for.
//   lanes    240 linedefs                      320                              500                                        701, bricks
//     96   0 68, 128:8 52, 256:16 74         84, 59, 72                       91, 128:16 55, 256:32 60                   152, 256:8 98, 256:16 78, 256:32 70
//    256   80, 57, 68 (before 70)            86, 62, 66 (73)                  94, 256:8 65, 256:16 62 (68)               154, 103, 92, 512:16 94 (106)
//    384   82, 60, 69 (85)                   90, 63, 68 (87)                  98, 72, 71, 384:16 70 (83)                 161, 104, 102, 384:16 96 (116)
//    704   93, 73, 256:8 78 (113)            97, 81, 83 (112)                 111, 83, 89, 128:8 89 (112)                170, 119, 125, 128:8 125 (158)
//   1024   98, 81, 84 (122)                  104, 87, 89 (124)                118, 94, 102, 128:8 95 (123)               178, 131, 138, 128:8 138 (185)
//   1536   108, 97, 105 (127)                115, 99, 107 (130)               124, 109, 118, 128:8 112 (139)             191, 145, 156, 128:8 155 (206)
//   2048   116, 122, 130 (117)               124, 122, 132 (151)              134, 134, 138, 128:8 124 (151)             206, 178, 189, 128:8 170 (232)
//   4096   184, 216, 227 (184)               191, 224, 235 (191)              195, 240, 236 (195)                        263, 322, 314 (264)
//   lanes    1000 linedefs                          2000                                             4000
//     96                                          256:8 117, 256:16 85, 256:32 76 (81)             256:8 188, 256:16 132, 256:32 109 (115)
//    160                                          512:16 93, 256:32 96 (96)                        512:16 139, 256:32 146 (152)
//    256   256:8 95, 256:16 86 (98)               512:8 128, 512:16 95 (112)                       512:8 196, 512:16 144 (152)
//    384   98, 102 (116)                          129, 113, 768:16 122 (133)                       199, 175, 768:16 160 (175)
//    704   125, 134 (158)                         161, 151, 160 (182)                              240, 252, 222 (257)
//   1024   143, 153 (181)                         200, 187, 196, 256:8 188 (223)                   290, 303, 275 (307)
//   1536   158, 170 (209)                         233, 242, 258, 256:8 231 (260)                   383, 409, 373 (364)
//   2048   192, 196, 128:8 180 (237)              269, 295, 316, 256:8 259 (284)                   439, 473, 469 (452)
//   4096   0 276, 256:8 339, 256:16 323 (338)     0 436, 256:8 421, 256:16 403 (424)               0 842, 512:8 657, 512:16 670 (672)
// 160 linedefs: 1280 lanes 0 67, 128:8 63, 1792 lanes 74, 79.  330, bricks: 2560 lanes 0 120, 128:8 116, 3072 lanes 130, 136.  700: 184, 166 and 192, 196.
// 1400: 3072 lanes 0 237, 256:8 226, 4096 lanes 269, 291; 256 lanes 512:16 77, 512 lanes 512:8 105.  2800: 320 lanes 512:16 124, 900 lanes 206, 1792 lanes 256:8 294.
inline int select_strips(int lanes, int linedefs) {
    if (linedefs <= 128 || (linedefs < 280 && lanes > 1536) || (linedefs < 1024 && lanes > 2816) || (linedefs < 1700 && lanes > 3072)) return 0;
    if (linedefs < 400) return 128;
    if (linedefs < 1024) return lanes <= 1792 ? 256 : 128;
    if (linedefs < 3000) return lanes <= 1152 ? 512 : 256;
    return lanes <= 1792 ? 768 : 512;
}
inline int select_lanes(int lanes, int linedefs) {
    const int w = linedefs < 4096 ? linedefs : 4096;      // no map of more was timed
    if (w < 400) return 8;
    if (lanes <= 96 + w / 128) return 32;
    if (w < 1024) return lanes <= 384 ? 16 : 8;
    if (w < 3000) return lanes <= 1152 || lanes >= 3584 ? 16 : 8;
    return lanes <= 1792 ? 16 : 8;
}

// wall_select_kernel: the longest strips and the others in one launch?  A launch on the side stream and back costs 20 us of the stage.  In larger batches
// the others' wavefronts are so many that they hold the longest strips' up, which the side stream's start a little later do not.  Stage times in us, one
// launch / two, of the strips and lanes above:
//   lanes     320 linedefs    701, bricks    1400         2000         2800         4000
//    768       82 / 109       124 / 151                 156 / 184                 231 / 260
//   1536       99 / 128       145 / 179                 231 / 243                 373 / 385
//   2048      122 / 145       170 / 206                 259 / 270                 439 / 479
//   2560                                   204 / 241                 350 / 381    490 / 526
//   3072                                   227 / 256                 395 / 406    577 / 571
//   4096                                                407 / 403                 684 / 657
inline bool select_together(int lanes) { return lanes <= 3072; }

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
