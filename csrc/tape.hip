// tape.hip — a decode step's launches again, from a list of them.
//
// A step is the same launches each time, its state on the device.  As a graph
// it runs without gaps inside, but 8 us pass between one graph's last kernel
// and the next one's first, and a first pass pays for the capture.  Called again
// from here a launch takes the host 3 us; it makes them while earlier ones run
// (kernels take 4 to 80) and waits for none.  us a step, a graph each -> launch
// by launch, and what the first two steps of a pass take, ms:
//   6 launches, 4096 wide MXFP4, 2 layers           97.8 ->   94.3   0.77 -> 0.40
//   21, 9B e4m3, 2 layers, 16 rows                 211.2 ->  204.5   1.20 -> 0.88
//   18, 8B e4m3, 8 layers                          457.7 ->  454.0   1.68 -> 1.08
//   66, 8B e4m3, 32 layers                        1734.2 -> 1730.5   4.87 -> 3.73
//   83, 1B bf16, 16 layers, 16 rows                901.5 ->  895.1   3.61 -> 2.85
//   143, 7B bf16, 28 layers, 6 rows               3024.6 -> 3018.4   8.12 -> 6.32
//   381, 9B e4m3, 42 layers, 16 rows              3601.1 -> 3597.2  12.44 -> 11.97
//   64, layer list, 4 rows                         391.2 ->  387.4   2.23 -> 1.69
//   45, layer list, one row                        372.5 ->  374.7   2.03 -> 1.32
//   34, 1B bf16, 16 layers, one row                557.9 ->  562.0   2.00 -> 1.30
// So all are made from here.  The last two lose 0.6% of a step and are behind
// once a pass has made some 300 and 170 of them; the others gain at any depth.
// The device depends on the host's thread for it, which is in C for all steps
// of a call.  Graphs of several steps are no faster and take 0.2 to 0.7 ms more
// to capture.
#include "common.h"

// A launcher with its arguments.  Numbers and pointers go in eight bytes
// each, in their order; floats apart.  That is how the x86-64 System V
// convention passes them, whatever the order of both among each other, while
// no more than eight are floats: six of the one kind and eight of the other in
// registers, the rest of the first on the stack; a function looks at as many
// as it has.  The last number is the stream.
#define TAPE_INTS 32
#define TAPE_FLOATS 8
struct TapeCall {
  void* fn;
  long n;
  long i[TAPE_INTS];
  float f[TAPE_FLOATS];
};

#if !defined(__x86_64__)
#error "arguments are passed as the x86-64 System V convention has it"
#endif

typedef hipError_t (*TapeFn)(
    long, long, long, long, long, long, long, long, long, long, long, long,
    long, long, long, long, long, long, long, long, long, long, long, long,
    long, long, long, long, long, long, long, long, float, float, float, float,
    float, float, float, float);

// n calls, `times` times over; at: the call that failed
extern "C" hipError_t tape_run(const TapeCall* calls, int n, int times,
                               hipStream_t stream, int* at) {
  for (int t = 0; t < times; t++)
    for (int k = 0; k < n; k++) {
      TapeCall c = calls[k];
      *at = k;
      if (c.n < 1 || c.n > TAPE_INTS) return hipErrorInvalidValue;
      c.i[c.n - 1] = (long)stream;
      const long* i = c.i;
      const float* f = c.f;
      const hipError_t e = ((TapeFn)c.fn)(
          i[0], i[1], i[2], i[3], i[4], i[5], i[6], i[7], i[8], i[9], i[10],
          i[11], i[12], i[13], i[14], i[15], i[16], i[17], i[18], i[19], i[20],
          i[21], i[22], i[23], i[24], i[25], i[26], i[27], i[28], i[29], i[30],
          i[31], f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]);
      if (e != hipSuccess) return e;
    }
  return hipSuccess;
}
