// pagani_ext.h -- library-internal entry points shared between the driver
// and the precompiled Genz evaluation (genz_eval.hip).
#pragma once

#include "pagani.h"

#ifdef __cplusplus
extern "C" {
#endif

// Launch the evaluation of a Genz descriptor on args->stream.
int pagani_genz_eval_launch(const pagani_genz* f, int precision, const pagani_eval_args* args);

#ifdef __cplusplus
}

namespace pagani {
namespace internal {
// The same; own_list: a caller's flat list, which no loop's launches go on from.
int genz_eval(const pagani_genz* g, int precision, const pagani_eval_args* a, bool own_list);
}  // namespace internal
}  // namespace pagani

#endif
