/* The forward pass of a batch inside a sweep (cnn_path.c), queued and not waited for: its loss is added to the totals of
 * fitre_hip_totals_begin.  sameWeights: weights and batch size are those of the batch before, and its copies of the weights in
 * scratch are still there. */
#ifndef FITRE_SWEEP_H
#define FITRE_SWEEP_H

#include "fitre_cnn.h"

void fitre_forward_batch(CNN_MODEL *model, DEVICE_DATASET *data, SCRATCH_AREA *scratch, real *z, real *probs, real *errors, int n, EVAL_TYPE mode,
                         int sameWeights);

#endif
