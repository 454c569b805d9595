// The method tableaux (rks_tableau.h) for the host.
#include "rks_tableau.h"

int rks_build_tableau(int method, rks_tableau* out) {
  if (method < RKS_M_ETD35 || method > RKS_M_IF4) return 1;
  *out = rks_tab::make(method);
  return 0;
}
