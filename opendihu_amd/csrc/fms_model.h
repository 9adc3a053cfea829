// The cell model a library is compiled for: its header and type are selected at
// compile time (FMS_MODEL_HEADER / FMS_MODEL_TYPE).
#pragma once

#ifndef FMS_MODEL_HEADER
#define FMS_MODEL_HEADER "model_hh.h"
#define FMS_MODEL_TYPE fms::ModelHH
#endif
#include FMS_MODEL_HEADER

using Model = FMS_MODEL_TYPE;
