/* librecflex_mlp.so: the MLP of RecomModel on the GPU (fp32, matrix cores).  Functions return 0 or a
 * hipError_t.  Nothing is allocated and nothing synchronised: the caller owns every buffer, and calls
 * with buffers of their own may overlap on different streams. */
#ifndef RECFLEX_MLP_H_
#define RECFLEX_MLP_H_

#include <stdint.h>

#define RECFLEX_MLP_MAX_LAYERS 8            /* hidden layers */
#define RECFLEX_MLP_MAX_SPLITS 32
#define RECFLEX_MLP_TAIL_MAX_UNITS 128      /* of the last hidden layer */
#define RECFLEX_MLP_TAIL_MAX_INPUTS 1024    /* of the last hidden layer */

#ifdef __cplusplus
extern "C" {
#endif

/* x [batch, units[0]] -> Linear, ReLU (layers times, units[1] .. units[layers]) -> Linear to one unit,
 * sigmoid -> out [batch].  weights[l] is [units[l + 1], units[l]] (the last one [1, units[layers]]),
 * row-major.  layers >= 2; units[0 .. layers - 1] are multiples of 4; x, weights[0 .. layers - 1],
 * hidden[0 .. layers - 2] and workspace lie on 16-byte boundaries.
 * hidden[l] [batch, units[l + 1]] receives the output of layer l after its ReLU; the last two may be
 * null. */
typedef struct recflex_mlp_args {
  const float *x;
  float *out;
  float *workspace;                          /* recflex_mlp_workspace_floats */
  void *stream;
  int32_t batch, layers;
  int32_t units[RECFLEX_MLP_MAX_LAYERS + 1];
  const float *weights[RECFLEX_MLP_MAX_LAYERS + 1], *biases[RECFLEX_MLP_MAX_LAYERS + 1];
  float *hidden[RECFLEX_MLP_MAX_LAYERS];
} recflex_mlp_args;

int recflex_mlp_workspace_floats(const recflex_mlp_args *args, int64_t *floats);
int recflex_mlp_forward(const recflex_mlp_args *args);

#ifdef __cplusplus
}
#endif

#endif /* RECFLEX_MLP_H_ */
