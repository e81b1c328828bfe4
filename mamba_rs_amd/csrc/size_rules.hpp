// Rules on sizes alone that choose a route, in plain C++ (tests compile them without a GPU).
#pragma once
#include <algorithm>
#include <cstdint>

namespace mrs {

// An operand that a kernel reads in pieces of sixteen bytes: it is there (a null pointer lies on such a piece as well) and begins on one.
inline bool in_pieces(const void *p) { return p && reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// conv1d + SiLU and x_proj of a prefill as one launch (conv_xproj.hip).  Columns of x_proj in tiles of 16: from three (33 columns, the fewest of d_state 16) to
// twelve, which leave room for four pieces of 64 channels in LDS, the fewest that keep requests ahead of their use.
constexpr int kConvPiece = 64, kConvMinTiles = 3, kConvMaxTiles = 12, kConvMaxSlices = 16;
inline int conv_xproj_col_tiles(int xd) { return (xd + 15) / 16; }
inline bool conv_xproj_columns_ok(int xd) { return xd % 4 == 0 && conv_xproj_col_tiles(xd) >= kConvMinTiles && conv_xproj_col_tiles(xd) <= kConvMaxTiles; }

// 0: two launches; 1: a workgroup has all channels of its steps; two or more: the channels in so many slices as well, for about one workgroup per compute unit, whose
// products a second launch sums.  In tiles of 32 steps.  Up to half a round of tiles the slices are ahead, as a workgroup that walks all channels takes its time however few
// there are; models of less than 1024 channels have little to share out.  Nine and eleven column tiles cost what ten and twelve do (a wave has half of
// them) and need most of a round.  Four layers of a bf16 prefill, two launches / slices / all channels, us:
//   d_model 256   32 tiles 231 / 227 / 224    64 275 / 273 / 261    128 338 / 315 / 307    200 415 / - / 393
//           448   32 301 / 297 / 300          64 348 / 346 / 342    128 498 / 481 / 474    200 655 / - / 624
//           512   32 263 / 266 / 274          64 328 / 326 / 331    128 474 / 459 / 456    200 590 / - / 564
//           640   24 273 / 276 / 289          64 413 / 395 / 401    128 559 / 542 / 541    200 700 / - / 665
//           768   32 318 / 312 / 332          64 436 / 414 / 430    128 602 / 585 / 581    200 792 / - / 766
//          1024   24 351 / 337 / 370          64 565 / 522 / 545    128 781 / 741 / 752    144 809 / - / 781
//          1280   24 396 / 380 / 432          64 658 / 628 / 670    128 900 / 874 / 895    144 1043 / - / 1037
//          1536   24 453 / 437 / 508          64 759 / 711 / 767    128 1105 / 1068 / 1100 144 1185 / - / 1170
//          1792   24 513 / 495 / 606          64 826 / 782 / 867    128 1217 / 1182 / 1224 144 1379 / - / 1375  200 1928 / - / 1864
//          2048   24 559 / 543 / 684          64 923 / 869 / 965    128 1493 / 1359 / 1404 144 1697 / - / 1624
//          2304   24 678 / 630 / 794          64 1079 / 1028 / 1160 128 1724 / 1684 / 1758 168 2057 / - / 2078  200 2340 / - / 2287
//          2560   24 725 / 688 / 856          64 1162 / 1119 / 1262 128 1941 / 1823 / 1909 144 2176 / - / 2113
inline int conv_xproj_form(int batch, int T, int di, int xd) {
    const int64_t tiles = (int64_t)batch * ((T + 31) / 32);
    const int columns = conv_xproj_col_tiles(xd);
    if (tiles > 128) return columns > 8 && columns % 2 && tiles < 192 ? 0 : 1;
    if (di < 1024) return tiles >= 64 ? 1 : 0;
    if (tiles < 24 || tiles * di < 40 * 1024) return 0;
    // (the shares fit in as many bytes as u has, and a slice has two pieces)
    const int slices = (int)std::min<int64_t>(std::min(std::min(di / (2 * xd), di / kConvPiece / 2), kConvMaxSlices), 256 / tiles);
    return slices >= 2 ? slices : 0;
}
// Steps of a workgroup with all channels: 32 as long as those are about one round over the compute units, else 64, which read x_proj's rows half as
// often (as above, 64 / 32: d_model 768, 8 x 1000 814 / 783, 6 x 2000 1052 / 1069, 8 x 2048 1276 / 1287; 1536, 8 x 1000 1702 / 1683, 8 x 2048 2953 / 3003; 2560, 8000 rows
// 3266 / 3221, 4 x 4096 5887 / 6038).
inline int conv_xproj_rows(int batch, int T) { return (int64_t)batch * ((T + 31) / 32) <= 320 ? 32 : 64; }

// Slices of K for the out_proj of a prefill of few rows (gemm_mid.hip), whose products the next kernel sums (it reads the result anyway).  A compute unit takes in some 60 bytes a
// nanosecond whatever it has asked for, so 24 tiles of 64 x 64 over K 1536 take 10 us with nine tenths of the chip idle.  As many slices as make a workgroup for every unit, or two where
// their walk stays long, four at most.  Us a layer of a bf16 prefill, one / two / three / four slices (six and eight: four's or behind):
//   d_model 768   64 rows 54.1 / 51.5 / 50.5 / 50.1    256 63.8 / 60.8 / 60.0 / 59.3    512 71.8 / 68.7 / 69.8 / 69.2    1024 83.9 / 85.6 / 87.2 / 87.4
//           1024  64 rows 65.5 / 61.9 / 60.7 / 60.0    256 71.2 / 66.9 / 65.5 / 65.4    512 79.6 / 75.9 / 77.1 / 77.1    777 92.0 / 91.5 / 93.0 / 94.3
//           2560  64 rows 129 / 128 / 125 / 124        128 154 / 141 / 139 / 141        256 172 / 170 / 164 / 167 (one: the vendor kernel)
//   Mamba-3 768   256 rows 80.5 / 77.8 / 77.0 / 76.7   512 84.9 / 82.0 / 82.8 / 82.5
constexpr int kMidTile = 64, kMidStepK = 64, kMaxMidSlices = 4;
inline int mid_gemm_slices(int64_t M, int N, int K) {
    const int64_t tiles = (M + kMidTile - 1) / kMidTile * ((N + kMidTile - 1) / kMidTile), steps = K / kMidStepK;
    const int64_t want = std::min<int64_t>(std::min(std::max(256 / tiles, std::min(512 / tiles, steps / 24)), steps / 3), kMaxMidSlices);
    if (want < 2 || K % kMidStepK != 0) return 1;
    const int64_t per = (steps + want - 1) / want;
    return (int)((steps + per - 1) / per);
}
// Floats that they take at most in a product of up to `rows` rows, which has slices by its own rows (0: none ever)
inline int64_t mid_gemm_parts_floats(int64_t rows, int N, int K) {
    const int64_t across = (N + kMidTile - 1) / kMidTile;
    int64_t most = 0;
    for (int64_t down = 1; down * across <= 256 && (down - 1) * kMidTile < rows; down++) {   // (a slice for every two units or fewer: past 256 tiles there are none)
        const int64_t M = std::min(down * kMidTile, rows);
        if (const int n = mid_gemm_slices(M, N, K); n > 1) most = std::max(most, n * M * N);
    }
    return most;
}

// Rows up to which a decode step's projections are the own kernels'.  Weights of up to ten million elements of in_proj (d_model 1536): as many as those kernels take; past that its
// tiles of 16 x 16 read too much over again.  Us a step, bf16, library / own:
//   12 layers of d_model 1024   48 rows 512 / 289, 64 540 / 329, 96 649 / 445, 128 682 / 511         1280   48 593 / 389, 64 675 / 485, 96 681 / 587, 128 821 / 697
//                   1536        65 rows 668 / 551, 96 735 / 628, 128 840 / 716    six of 1792        65 rows 411 / 399, 96 447 / 464, 128 485 / 554    2560   65 551 / 595, 128 716 / 821
//   Mamba-3, eight of 512       65 rows 288 / 212, 128 463 / 316    768   65 388 / 293, 128 496 / 420    1024   65 467 / 370, 128 623 / 540    1536   65 589 / 530, 128 841 / 811
inline bool own_chain_to_the_last_row(int64_t d_model, int64_t d_inner) { return d_model * 2 * d_inner <= 10 * 1000 * 1000; }

// The same for f32 models (16 x 16 tiles on the matrix cores' f32 instructions; one to four rows row by row where the width allows).  Wide rows of many are the library's again, those of
// Mamba-3 sooner: its launches per layer are fewer.  Us a step of four layers, library / own:
//   Mamba-1 d_model 192   1 row 101 / 65, 8 rows 106 / 81, 128 rows 112 / 101    256   8 rows 107 / 74, 128 rows 125 / 109    768   5 rows 202 / 97, 64 rows 211 / 175, 128 rows 260 / 250
//           1024   8 rows 247 / 144, 64 rows 269 / 229, 96 rows 285 / 309        1536  8 rows 361 / 200, 48 rows 425 / 373     2560  8 rows 1600 / 383, 48 rows 1639 / 835
//   Mamba-3 192   1 row 75 / 59, 128 rows 91 / 94    256   8 rows 87 / 72, 128 rows 103 / 103    512   8 rows 106 / 88, 48 rows 134 / 126, 64 rows 139 / 142
//           768   8 rows 164 / 102, 48 rows 196 / 168, 96 rows 245 / 249    1024   48 rows 242 / 219, 64 rows 248 / 252    2560   8 rows 1457 / 312, 48 rows 1572 / 757
inline int own_f32_chain_rows(int64_t d_model, int64_t d_inner, bool mamba3) {
    const int64_t n = d_model * 2 * d_inner;
    if (mamba3) return n <= 300 * 1000 ? 96 : 48;
    return n <= 2400 * 1000 ? 128 : n <= 4200 * 1000 ? 64 : 48;
}

// f32 models in a prefill, whose products are the library's: whether it is handed the transposed weights, which are there for the decode's own chain.  Its kernels for either order are ahead
// or behind by size, without a line to be drawn: from the transposed ones the prefill takes, of what it takes from the others, at d_model 1024 118 % with 256 rows, 110 % with 512, 91 % with
// 768 and 82 % with 2048, at 512 109 % with 128 rows, at 1280 119 % with 2048, at 2048 107 % with 32 rows and 77 % with 768; at 2560 60 to 66 % with up to 384 rows, 81 to 104 % past them.
// So models of that width alone, and as before those of one to four rows whose steps go row by row.
inline bool f32_prefill_transposed(int64_t d_model, int64_t d_inner, bool row_by_row) { return row_by_row || d_model * 2 * d_inner > 20 * 1000 * 1000; }

// Whether what a decode step touches (`bytes`: weights, states, the head's table) is more than the chip's last cache holds, 256 MB.  What is read once a step and not kept from one
// step to the next is then better read past it: cached, it drives out what could have stayed, and changed states have to be written back to make room.
// The head's table, cached / past, us a step, vocabulary 50280: 130m shape 1 row (259 MB) 205.1 / 202.1, 16 rows 292.7 / 277.7, 64 rows 357 / 351; 20 of its layers 1 row (229 MB)
// 168.7 / 174.2, 16 rows (266 MB) 241.7 / 235.2; 16 of them 16 rows (228 MB) 189.2 / 194.5, 64 rows (323 MB) 243.1 / 234.8; 12 of them 64 rows (262 MB) 184.4 / 182.9.
// The states, which are read and written once a step, cached / past (a launch per product; the weights then stay where they fit): 130m shape 72 rows 609 / 565, 128 rows 788 / 758; 24 layers
// of 1024 48 rows 591 / 568, 64 rows 659 / 623; 2.8b shape, 8 layers, 16 rows 323 / 316, 64 rows 578 / 565; Mamba-3, 24 layers of 768, 12 rows 390 / 361, 32 rows 494 / 427, 128 rows 1019
// / 930.  (In the resident step of several rows, which asks for them a phase ahead: 64 rows 344 / 357.)
inline bool step_outgrows_cache(int64_t bytes) { return bytes > (int64_t)240 << 20; }

// Layers whose weights (`layer_bytes` each) come through that cache in a decode step: all of them where the states and they fit, else as many as leave room for the states, and the
// others are read past it.  Walked from first to last at every step, more than it holds would leave nothing of it.  Us a step, bf16, 24 layers of which so many come through it:
//   d_model 1024 (13.1 MB a layer)   1 row 24 286, 20 278, 16 267, 12 271, 0 281     4 rows 316, 312, 295, 298, 301    13 rows 337, 332, 327, 320, 328   32 rows 371, 369, 364, 361, 362
//           768 (7.5)                32 rows 305, 301, 301, 305, 308     64 rows 351, 351, 349, 347, 351 (8 345)     16 rows, which fit 277, 281, 278, 279, 283
inline int layers_in_cache(int layers, int64_t layer_bytes, int64_t state_bytes) {
    if (!step_outgrows_cache(layers * layer_bytes + state_bytes)) return layers;
    return (int)std::min<int64_t>(layers, std::max<int64_t>(0, ((int64_t)220 << 20) - state_bytes) / std::max<int64_t>(layer_bytes, 1));
}

// Rows of a Mamba-3 head's state that a thread of the step kernel has (m3_engine.hip, the times there): four from 192 heads on, at d_state 64, where the workgroup is then still whole waves
// (its sums go over 64 lanes; headdim a multiple of 16) with a thread for every state and every pair to rotate.
inline int m3_step_rows(int64_t batch, int nheads, int headdim, int d_state, int n_rope) {
    const int threads = headdim * (d_state / 4) / 4;
    return batch * nheads >= 192 && d_state == 64 && threads % 64 == 0 && threads >= std::max(d_state, n_rope) ? 4 : 1;
}

// Decode of a launch per product (wide models, and one to four rows of f32 ones): in_proj's weights, two thirds of a layer's, are read past that cache where a step (`bytes` of weights and states) outgrows it, so that
// out_proj's and the states may stay and nothing has to be written back for what is read once.  Us a step, bf16, cached / past: d_model 2560, 8 layers 4 rows 322 / 294, 16 358 / 322,
// 32 438 / 426, 64 577 / 573; 24 layers 4 rows 833 / 808, 16 938 / 877; 2048, 12 layers 4 rows 354 / 331, 16 392 / 370, 48 557 / 563 (there states are most of it); 24 of 1024, the states past it, 48 rows 568 / 543, 64 rows 623 / 634.  Some of the
// layers' through the cache, as layers_in_cache: behind it everywhere (2560, 16 rows, two of eight 341).  out_proj's past it as well: no difference, and where the step kernel asks for
// its lines ahead that request past it costs 40.  f32, one row, 24 layers, with the head's table past it as well: all cached 383, in_proj's past 341, all past 362 (768); 510, 458, 468 (1024).
inline bool streams_in_proj(int64_t bytes, int rows) { return rows <= 48 && step_outgrows_cache(bytes); }

// Decode of wide models: whether the step kernel asks for the lines of out_proj (`bytes` of them) on the dies that will read them (m1_step.hip).  They have to stay in the dies' L2, eight
// of 4 MB, until the launch behind: more than that is read twice, and then many rows' worth of work must cover it.  Eight layers, bf16, us a step, without / with:
// 25 MB (d_model 2560) 4 rows 284 / 285, 8 304 / 297, 16 330 / 320, 40 454 / 433; 30 MB (2816) 314 / 317, 333 / 328, 367 / 356, 586 / 586; 36 MB (3072) 329 / 338, 351 / 351,
// 390 / 382, 522 / 521; 42 MB (3328) 379 / 398, 410 / 428, 465 / 468; 49 MB (3584) 405 / 429, 444 / 457, 499 / 504.  (Asking for the part that would fit: behind both everywhere.)
inline bool asks_out_proj_ahead(int64_t bytes, int rows) { return bytes <= (int64_t)(rows < 8 ? 28 : 40) << 20; }

}  // namespace mrs
