// Chip-resident time loop, FDORDER 4, acoustic, VTI, TTI and SH.
#define DN_F 2
#define DN_GROUP 1
#include "dn_resident_inst.inc"
