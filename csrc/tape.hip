// tape.hip — a decode step's launches again, from a list of them.
//
// A step is the same launches each time, its state on the device.  As a graph
// it runs without gaps inside, but 8 us pass between one graph's last kernel
// and the next one's first, and a first pass paid 1 to 2 ms for the capture.
// Called again from here a launch takes the host 3 us, less than its kernel
// runs (4 to 80), and the stream never runs dry.  us a step, a graph each ->
// launch by launch (graphs of four steps):
//   6 launches, 4096 wide MXFP4, 2 layers        99.3 ->  96.8 ( 95.9)
//   14 launches, experts                        128.1 -> 126.4 (124.7)
//   64 launches, layer list, 4 rows             391.4 -> 387.0 (387.8)
//   34 launches, 2048 wide bf16, 16 layers      558.6 -> 564 to 566 (564.1)
// Four steps a graph are half a percent less, and 0.2 to 0.5 ms of a first
// pass more.
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
