// The device-side error word: one bit per cause, so that causes raised together
// and the code that a call returns for them can be told apart.
#pragma once

#include "../../include/evd4sc.h"

namespace evd {

enum : unsigned {
  kErrTimeout = 1u << 0,     // a bounded wait expired
  kErrNonfinite = 1u << 1,   // the input held NaN or Inf
  kErrNoconverge = 1u << 2,  // a secular equation's root did not converge
  kErrRange = 1u << 3,       // a 16-bit operand out of range
};

// status (EVD_E_*) of a nonzero error word: of several causes the one that the
// others may follow from
inline int device_error_code(unsigned word) {
  if (word & kErrTimeout) return EVD_E_TIMEOUT;
  if (word & kErrNonfinite) return EVD_E_NONFINITE;
  if (word & kErrNoconverge) return EVD_E_NOCONVERGE;
  if (word & kErrRange) return EVD_E_RANGE;
  return EVD_E_HIP;  // no cause of this library: the word was overwritten
}

inline const char *device_error_text(unsigned word) {
  switch (device_error_code(word)) {
    case EVD_E_TIMEOUT: return "a bounded wait expired";
    case EVD_E_NONFINITE: return "the input held NaN or Inf";
    case EVD_E_NOCONVERGE: return "a secular equation did not converge";
    case EVD_E_RANGE: return "a mixed-precision operand left the 16-bit range";
    default: return "unknown cause";
  }
}

}  // namespace evd
