// jy_epi.h — what a product's epilogue does with each sum y of its output.
#pragma once

#include <stdexcept>
#include <string>

namespace jy {

// STORE out = y, BIAS out = y + aux, RESID out += y; SWIGLU, ROPE and ARGMAX only where a launch
// names them
enum Epi { EPI_STORE = 0, EPI_BIAS = 1, EPI_RESID = 2, EPI_SWIGLU = 3, EPI_ROPE = 4, EPI_ARGMAX = 5 };

// for launches of the first three alone: another one is an error of the call, not a plain store
inline Epi plain_epi(Epi e) {
    if (e != EPI_STORE && e != EPI_BIAS && e != EPI_RESID)
        throw std::invalid_argument("epilogue " + std::to_string((int)e) + " is not one of this product's");
    return e;
}

}  // namespace jy
