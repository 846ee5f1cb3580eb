// How the transforms of 2-D plans share their work out over threads (input_transform.hip, output_transform.hip).  Host code without HIP.
#pragma once

namespace wc {

// Channels a thread of the input transform, of `vec` at most: fewer until every CU has a workgroup of its own (65536 threads over tiles, rows of Cp
// channels and pieces).  fp32 on tile 2, stacked, where a thread's channels are 16 bytes and the pieces write columns of one row, gains up to half as many threads only:
// us, all four channels | line at 65536 | 32768, 5x5 stride 2, 243 tiles of 16 channels 4.02 | 3.60 | 3.60, 464 of 120 6.31 | 6.66 | 6.31, 425 of 88 5.38 | 5.99 | 5.38,
// 500 of 152 7.21 with any.  Over 539 launches of 16 to 380 channels the time against all channels a thread, mean and worst: stacked, fp32 on tile 2 0.980 and 1.11 | 0.978 and
// 1.00; at 65536 fp16 on tile 2 0.903 and 1.00, fp32 on tile 4 0.928 and 1.00, fp16 and bf16 on tile 4 0.964 and 0.960 and 1.03 (0.966, 0.956 and 1.00 at 32768).
// Not stacked, against the fastest number of channels for each: 16-bit types 1.009 and 1.08 on tile 2, 1.004 and 1.06 on tile 4, fp32 1.009 and 1.10, 1.045 and 1.16.
inline int input_channels(int vec, long long tiles, int Cp, int n_pieces, bool stacked, bool f32, int m) {
  const long long enough = stacked && f32 && m == 2 ? 32768 : 65536;
  while (vec > 1 && tiles * (Cp / vec) * n_pieces < enough) vec /= 2;
  return vec;
}

// Whether every piece gets threads of its own, of `threads` over tiles and channels: large launches keep one thread for all pieces of a tile, which reads each
// window from cache once per piece.  Stacked plans: 2.2 times as fast apart at N=8, 24 channels, 56x56, 7x7, in the loop 7 to 30 % the faster further up.  Others, over
// 240 launches of 30 to 530 thousand threads, apart against the loop: nine pieces 0.62 to 1.07, 0.83 in the mean of 16-bit types on tile 4 and 0.93 of fp32 on
// tile 2; four of fp32 0.90 in the mean on tile 4, 0.98 on tile 2; four of 16-bit types 0.69 at 70 thousand and 1.00 to 1.12 from 290 thousand on on tile 4,
// 0.71 at 30 and 1.05 to 1.13 from 185 thousand on on tile 2.  us, fp16 5x5, loop | apart: tile 2, N=13 48 channels, 78x78 26.4 | 25.3, N=9 160, 73x73 35.4 | 39.6; tile 4, N=51 136, 25x25
// 28.0 | 24.0, N=9 336, 68x68 46.9 | 52.5.
inline bool pieces_apart(long long threads, int n_pieces, bool stacked, bool f32, int m) {
  const int thousands = stacked || f32 || n_pieces > 4 ? 512 : m == 2 ? 160 : 288;
  return threads < thousands * 1024ll;
}

// Whether a thread of the output transform takes one channel instead of `vec`, so that more CUs have a workgroup: up to 65536 threads over tiles and groups
// of vec channels, where a thread gathers several pieces or in fp32 on tile 4, else up to half as many.  Of 588 launches of 16 to 380 output channels, time against vec
// channels a thread, mean and worst, line at 65536 | 32768: one piece, fp16 on tile 4 0.968 and 1.043 | 0.966 and 1.00, on tile 2 0.983 and 1.035 |
// 0.982 and 1.013, fp32 on tile 2 1.003 and 1.057 | 1.001 and 1.024, on tile 4 0.89 and 1.00 | 0.90 and 1.00; several 0.82 to 0.91 and 1.00 (fp32 on tile 2 once 1.05) | 0.84 to
// 0.92 and 1.00.  us, vec channels | one: fp16 6x6 N=4 136, 54x54 5.01 | 5.27, fp32 4x4 N=3 216, 34x34 3.86 | 4.32; F(4,3) fp32 N=8 352, 9x9 5.02 | 4.24, N=8 64, 60x60 5.83 | 5.44.
inline bool output_one_channel(long long tiles, int K, int vec, int n_pieces, bool f32, int m) {
  return tiles * (K / vec) < (n_pieces > 1 || (f32 && m == 4) ? 65536 : 32768);
}

}  // namespace wc
