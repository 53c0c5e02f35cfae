/*
 * soi_fft_lengths.h -- transform lengths of the register FFT passes and their schedules:
 * X(L, threads per sequence, radices in stage order).
 *
 * F * 2^a for the odd parts F = 1, 3, 5, 9, 15, 25: any M_hat = 2^a 3^b 5^c whose odd part is a
 * product of two of these splits into two of the lengths.  Up to 200 points two stages, above
 * that three.  The first radix is a power of two where there is one (the LDS swizzle then spreads
 * the first exchange over all banks), and the threads per sequence keep every stage at least
 * about two thirds busy with at most 20 values per thread.
 */
#define SOI_FFT_SHORT(X) \
  X(48, 8, 8, 6) X(50, 5, 10, 5) X(60, 10, 10, 6) X(64, 8, 8, 8) X(72, 9, 8, 9) X(80, 10, 8, 10) \
  X(96, 12, 8, 12) X(100, 10, 10, 10) X(120, 8, 8, 15) X(128, 8, 16, 8) X(144, 16, 16, 9) \
  X(160, 16, 16, 10) X(192, 16, 16, 12) X(200, 10, 20, 10) X(240, 40, 8, 6, 5) \
  X(256, 32, 8, 8, 4) X(288, 48, 8, 6, 6) X(320, 40, 8, 8, 5) X(384, 48, 8, 8, 6) \
  X(400, 50, 8, 10, 5) X(480, 60, 8, 6, 10) X(512, 32, 8, 8, 8) X(576, 72, 8, 8, 9) \
  X(640, 64, 8, 8, 10)
#define SOI_FFT_LONG(X) \
  X(768, 96, 8, 8, 12) X(800, 100, 8, 10, 10) X(960, 64, 16, 15, 4) X(1024, 64, 16, 8, 8) \
  X(1152, 72, 16, 8, 9) X(1280, 80, 16, 8, 10) X(1536, 96, 16, 16, 6) X(1600, 100, 16, 10, 10) \
  X(1920, 128, 16, 15, 8) X(2048, 128, 16, 16, 8)
/* rows of these are four (complex128) or eight (complex64) to a block, half of the others': as many
 * of 144 or more threads each do not fit one */
#define SOI_FFT_LONGEST(X) X(2304, 144, 16, 16, 9) X(2560, 160, 16, 16, 10)
/* one segment per block, one pass (two exchanges) */
#define SOI_FFT_ONE(X) \
  X(960, 64, 16, 15, 4) X(1024, 128, 8, 16, 8) X(1152, 128, 16, 9, 8) X(1280, 128, 10, 16, 8) \
  X(1200, 80, 16, 15, 5) X(1350, 90, 18, 15, 5) X(1440, 160, 16, 9, 10) X(1500, 150, 10, 15, 10) \
  X(1536, 192, 8, 16, 12) X(1600, 160, 16, 10, 10) X(1728, 144, 12, 12, 12) X(1800, 120, 8, 15, 15) \
  X(1920, 192, 16, 12, 10) X(2000, 200, 10, 20, 10) X(2048, 256, 8, 16, 16) \
  X(2160, 120, 18, 20, 6) X(2250, 150, 15, 15, 10) X(2304, 256, 16, 16, 9) X(2400, 240, 16, 15, 10) \
  X(2560, 256, 16, 16, 10) X(2700, 225, 12, 15, 15) X(2880, 180, 16, 18, 10) \
  X(3000, 200, 15, 20, 10) X(3072, 256, 16, 16, 12) X(3200, 200, 16, 20, 10) \
  X(3456, 288, 16, 18, 12) X(3600, 240, 16, 15, 15) X(3840, 256, 16, 16, 15) \
  X(4000, 200, 20, 20, 10) X(4096, 256, 16, 16, 16) X(4320, 288, 16, 18, 15) \
  X(4500, 300, 20, 15, 15) X(4608, 288, 16, 18, 16) X(4800, 320, 16, 20, 15) \
  X(5120, 320, 16, 20, 16)
