// Chip-resident time loop, FDORDER 2.
#define DN_F 1
#include "dn_resident_inst.inc"
