// cgstate.hpp -- device state of a conjugate gradient solve.
#pragma once

namespace svfsi {

struct CgState {
    double err, errO, alpha, eps;
    int done, suc, itr, mItr;
    unsigned int counter;
    int abort;   // a matrix-resident kernel gave up waiting (persist.hpp); done is set too
    double e[2]; // |R|^2 of the current and the next iteration, by iteration parity
};

} // namespace svfsi
