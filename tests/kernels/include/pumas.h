/*
 * Stands in for the reference's include/pumas.h where that is not installed,
 * so that the C caller is built and run all the same: the shared types as
 * pumas_gpu.h declares them, and the simulation context in the reference's
 * public layout (include/pumas.h:636-672). The layout checks of the C caller
 * are against the reference's own types only when it is built with them.
 */
#ifndef TESTS_PUMAS_H
#define TESTS_PUMAS_H

#include "pumas_gpu.h"

struct pumas_context {
        void * medium; /* callbacks, recorder and user data */
        void * random;
        void * recorder;
        void * user_data;
        struct pumas_context_mode mode;
        enum pumas_event event;
        struct pumas_context_limit limit;
        double accuracy;
};

#endif
