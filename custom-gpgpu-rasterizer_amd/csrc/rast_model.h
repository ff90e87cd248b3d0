// rast_model.h -- learned bin-capacity model, internal interface used by the
// frame orchestration in rast_api.hip (implementation: rast_mlp.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "rast.h"
#include "rast_internal.h"

// Makes m (or none: null) the renderer's model; a frame queued with another one
// is waited for.
int rast_model_attach(rast_renderer *r, rast_binmodel *m);
// A renderer without queued work is being destroyed: its model and the models
// created on it forget it (those live on, on a stream of their own).
void rast_model_renderer_gone(rast_renderer *r);
// Hidden width of a model (16, 32 or 64) and its device parameters.
int rast_model_hidden(const rast_binmodel *m);
const float *rast_model_params(const rast_binmodel *m);
