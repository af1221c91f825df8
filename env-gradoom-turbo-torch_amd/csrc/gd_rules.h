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

// wall_select_kernel's launch for the longest strips: how many of them, and how many lanes a column has there.  More strips and more lanes
// shorten the longest strips' time, which is all that a small batch's lasts, and add to what all of them take together, which a
// large one's does.  Where the lists are short (they follow the map's linedefs) there is little to shorten: fewer strips in large batches, and none
// where the lanes are as many as twelve times the linedefs beyond a hundred, in the largest batches of up to 900 linedefs, or on the
// smallest maps.  Stage times in us of no such launch / 768 strips (1024 from 1024 linedefs on) of 8 / of 16 lanes
// (of 32), in brackets what it took with the lists in LDS and 8 columns of one lane a wavefront:
//   lanes       120              320                        800                         2000                          4000
//      16    46 / 55 / 76     97 / 53 / 64 (61; [60])    168 / 74 / 62 (52)         339 / 120 / 89 (68; [151])     361 / 119 / 90 (69; [156])
//     128    55 / 60 / 77     133 / 69 / 81 ([83])       181 / 83 / 71              436 / 153 / 113 (104; [203])   1003 / 236 / 172 (145; [430])
//     256    59 / 73          137 / 84 / 96 ([102])      212 / 106 / 99             447 / 164 / 132 ([214])        999 / 247 / 197 ([420])
//     512    63 / 81          140 / 107 / 119 ([111])    220 / 126 / 128            453 / 172 / 178 ([267])        1003 / 275 / 257 ([463])
//    1024    69               149 / 146 ([138])          241 / 174 / 174            520 / 265 / 264 ([336])        1060 / 408 / 413 ([563])
//    2048    80               166 / 180 ([171])          277 / 234 / 235            549 / 371 / 370 ([411])        1120 / 652 / 647 ([727])
//    4096    130              230 / 288 ([279])          328 / 363                  667 / 604 / 576 ([600])        1249 / 945 / 887 ([966])
// (the last two rows with 768 and with 512 strips.)  None / 256 / 512 / 768 strips of 8 lanes on maps below 1024 linedefs, in brackets as above:
//   lanes         200 linedefs            240                   320                330, bricks               500                701, bricks               1000
//     256    93/ 72/ 64/ 67 ( 67)   91/ 72/ 66/ 66 ( 72)  136/ 97/ 82/ 83 (104)  154/109/ 89/ 92 (105)  159/107/ 85/ 87 (116)  294/160/127/129 (166)
//     512    97/ 84/ 80/ 85 ( 79)   95/ 92/ 83/ 80 ( 81)  138/121/109/105 (111)  176/131/120/112 (127)  198/131/123/115 (127)  303/188/176/151 (190)
//     768   101/ 97/ 91/ 96 ( 90)   98/ 99/ 90/ 92 ( 89)  145/134/127/127 (128)  182/142/144/135 (145)  200/160/144/146 (148)  321/240/204/195 (210)  351/219/194/183 (215)
//    1024   105/102/ 98/106 ( 97)  102/106/101/103 (100)  147/138/142/141 (138)  190/150/151/152 (150)  204/165/160/158 (160)  325/265/227/215 (231)  360/249/231/205 (235)
//    1280   107/107/110/111 (108)  104/109/112/110 (110)  151/147/151/151 (146)  200/160/162/159 (162)  211/177/174/171 (173)  340/273/243/234 (250)  369/267/240/218 (248)
//    1536   109/116/113/120 (113)  108/118/115/115 (115)  157/155/159/163 (157)  203/169/172/169 (171)  216/181/187/188 (186)  350/297/269/255 (280)  381/281/252/244 (263)
//    2048   116/122/128/139 (124)  114/128/124/131 (125)  165/166/177/191 (170)  214/190/188/198 (184)  239/198/209/223 (206)  363/310/298/303 (312)  386/298/282/290 (296)
//    2560   120/137/145/157 (137)  120/142/138/148 (132)  179/192/204/218 (194)  224/199/209/222 (200)  249/224/238/252 (228)  379/330/335/353 (344)  402/334/321/340 (326)
//    3072   127/153/162/173 (153)  137/148/154/164 (146)  188/219/232/246 (220)  231/225/238/251 (225)  260/255/268/285 (259)  395/369/385/402 (372)  424/356/366/382 (358)
//    4096   150/189/197/209 (189)  148/184/190/200 (182)  227/276/289/306 (279)  252/289/301/314 (288)  284/326/342/359 (332)  425/466/483/500 (472)  475/449/465/482 (458)
// Over these and thirteen more maps of 60 to 800 linedefs, 16 to 4096 lanes, the rule's choice takes 1.2 % more in the mean than the best of the
// four, 16 % at most.  Against the brackets' it is 7 % faster in the geometric mean; it is more than 5 % slower on maps of up to 240 linedefs
// (by 4 to 12 us, mostly at 48 to 384 lanes) and at two places on 280.
inline int select_strips(int lanes, int linedefs) {
    if (linedefs <= 128 || lanes >= 12 * (linedefs - 100) || (lanes >= 3584 && linedefs < 900)) return 0;
    if (linedefs < 512) return lanes < 832 ? 768 : (lanes < 1152 ? 512 : 256);
    if (linedefs < 1024) return lanes < 2304 ? 768 : (lanes < 2816 ? 512 : 256);
    return lanes < 1792 ? 1024 : (lanes < 3584 ? 768 : 512);
}
inline int select_lanes(int lanes, int linedefs) {
    const int w = linedefs < 4096 ? linedefs : 4096;      // no map of more was timed
    if (w < 512) return 8;
    if (lanes <= 64 + w / 24) return 32;
    return lanes <= 128 + w / 8 || (lanes >= 1536 && w >= 1024) ? 16 : 8;
}

// wall_select_kernel: the longest strips and the others in one launch?  A launch on the side stream and back costs 8 us and more.  In larger batches
// the others' wavefronts are so many that they hold the longest strips' up, which the side stream's start a little later do not.  A frame in
// us, one launch / two (32 billboards, two sets of poses):
//   lanes        320             800             1400            2000            4000          701, bricks
//    256     335 / 342       382 / 390       454 / 463       449 / 457       653 / 661       520 / 527
//    384     420 / 423       464 / 474       575 / 582       547 / 554       780 / 787       586 / 587
//    512     496 / 498       552 / 562       629 / 645       639 / 643       880 / 912       669 / 670
//    640     570 / 572       617 / 627       747 / 761       716 / 720       978 / 994       724 / 726
//    768     642 / 643       709 / 715       857 / 873       814 / 812      1130 /1136       838 / 839
//   1024     737 / 742       817 / 805       956 / 952       973 / 962      1345 /1342       952 / 935
inline bool select_together(int lanes) { return lanes <= 704; }

// wall_geometry_kernel: wavefronts a lane for its linedefs (a power of two).  us with 4 / 8 / 16 of them: 16 lanes 13.6 / 10.7 / 8.3, 512 lanes
// 63 / 48 / 46, 1024 lanes 48 / 41 / 42, 4096 lanes 263 / 242 / 247.
inline int geometry_parts(int lanes) { return lanes >= 1024 ? 8 : 16; }

// wall_raster_kernel: wavefronts a strip.  One draws, pass after pass, the rows that any of its columns draws.  A small batch, which lasts as
// long as its longest strips, shares a strip out over eight wavefronts, a larger one over four, over two.  The wavefront's columns then have
// eight, four or two lanes each: these prepare as many passes at once and share every run of rows out, so that both the chain of waits and
// the vector instructions of a column shrink with them (when the spare lanes stood idle, eight wavefronts never paid).  What a strip more
// wavefronts costs is room on the SIMDs.  Stage times in us (wall_geometry_kernel among them) for 1 / 2 / 4 / 8 wavefronts a
// strip, in brackets with idle lanes and the lines of then (four up to 560 lanes, two up to 1344):
//   lanes           320 linedefs                     2000                             4000                             701, bricks
//      16         / 90 / 72 / 65 (106)            / 136 / 110 / 97 (155)           / 184 / 149 / 139 (196)          / 263 / 218 / 188 (285)
//     256        / 142 / 119 / 113 (155)         / 198 / 161 / 145 (212)          / 328 / 259 / 229 (327)          / 291 / 238 / 208 (310)
//     384        / 148 / 121 / 136 (174)         / 206 / 175 / 170 (229)          / 349 / 276 / 274 (345)          / 298 / 247 / 219 (322)
//     512        / 156 / 126 / 175 (202)         / 219 / 189 / 222 (250)          / 425 / 401 / 367 (480)          / 313 / 256 / 249 (318)
//     640        / 165 / 156 / 222 (202)         / 233 / 204 / 279 (277)          / 432 / 416 / 394 (498)          / 346 / 273 / 309 (408)
//     768     235 / 173 / 187 / 270 (214)     328 / 239 / 236 / 333 (282)      527 / 445 / 422 / 457 (513)      430 / 345 / 283 / 371 (415)
//    1024     253 / 204 / 233 / 351 (249)     385 / 270 / 303 / 437 (330)      555 / 466 / 445 / 598 (539)      449 / 354 / 334 / 487 (431)
//    1536     294 / 287 / 342 (298)           438 / 383 / 440 (448)            597 / 528 / 630 (619)            479 / 392 / 490 (501)
//    2048     365 / 357 / 450 (364)           492 / 478 / 583 (487)            701 / 674 / 835 (695)            524 / 509 / 643 (536)
//    2560     439 / 425 (440)                 596 / 589 (583)                  831 / 845 (820)                  639 / 625 (649)
//    3072     519 / 542 (514)                 700 / 722 (683)                  930 / 969 (918)                  751 / 744 (753)
// With one lane a column nothing is shared, and the stage takes up to 1.7 % longer than before columns could share: on one card at 4096 lanes 679 -> 684,
// 886 -> 901, 1229 -> 1238 and 971 -> 974 us.  (A prepared pass's flags and rows kept in registers of their own there, not packed into words,
// issue 1.5 % fewer instructions and take as long: 686, 905, 1239, 975.)
inline int raster_parts(int lanes) { return lanes <= 336 ? 8 : (lanes <= 704 ? 4 : (lanes <= 2400 ? 2 : 1)); }

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
