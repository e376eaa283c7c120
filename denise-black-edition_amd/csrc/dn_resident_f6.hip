// Chip-resident time loop, FDORDER 12.
#define DN_F 6
#include "dn_resident_inst.inc"
