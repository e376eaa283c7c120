// Chip-resident time loop, FDORDER 4.
#define DN_F 2
#include "dn_resident_inst.inc"
