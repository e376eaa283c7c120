// Chip-resident time loop, FDORDER 6.
#define DN_F 3
#include "dn_resident_inst.inc"
